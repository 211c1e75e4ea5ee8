"""The matrix products in inline asm of the row tiles past 256 rows (gemm_pp.hip, pp_mfma): the compiler does not know that their
results come late, so any copy of one that it puts close behind a product would read too early.  Read off the built code."""
import glob
import os
import re
import shutil
import subprocess

import pytest

import distributed_llms_amd

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
# Wait states between a product's issue and an access to its result that the hardware does not hold back: 19 for the longest
# products (16 passes; CDNA3 instruction set guide, "Software Dependencies"), these have 4.
WAITS = 20


def _regs(operand):
    """Vector registers of one operand: v7, v[4:7] (accumulation registers are not theirs)."""
    m = re.fullmatch(r"v(\d+)|v\[(\d+):(\d+)\]", operand)
    if not m:
        return set()
    return {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


def _parse(listing):
    """[(address, mnemonic, operands, branch target or None)] of one kernel's llvm-objdump lines."""
    out = []
    for line in listing:
        m = re.match(r"\s+(\w+)\s*(.*?)\s*// ([0-9A-F]+):(?:.*<\S+\+0x([0-9a-f]+)>)?", line)
        if m:
            ops = [o.strip().split(" ")[0] for o in re.split(r",\s*(?![^\[]*\])", m[2])] if m[2] else []
            out.append((int(m[3], 16), m[1], ops, int(m[4], 16) if m[4] else None))
    return out


def early_accesses(listing):
    """(products into vector registers, accesses to such a product's result that come before its wait states are over), along every
    path from the product on."""
    code = _parse(listing)
    if not code:
        return 0, []
    at = {a - code[0][0]: i for i, (a, *_) in enumerate(code)}
    bad, products = [], 0
    for i, (_, op, ops, _) in enumerate(code):
        if not op.startswith("v_mfma") or not _regs(ops[0]):
            continue
        products += 1
        dest, todo, seen = _regs(ops[0]), [(i + 1, 0)], {}
        while todo:
            j, states = todo.pop()
            if j >= len(code) or states >= WAITS or seen.get(j, WAITS + 1) <= states:
                continue
            seen[j] = states
            _, o, operands, target = code[j]
            if o.startswith("v_mfma"):                          # (its own sum may take the result up: the hardware waits)
                touched = set().union(*(_regs(x) for x in operands[1:3]))
                if _regs(operands[0]) & dest and _regs(operands[0]) != dest:
                    touched |= _regs(operands[0])
            else:
                touched = set().union(*(_regs(x) for x in operands)) if operands else set()
            if touched & dest:
                bad.append((i, code[i], j, code[j]))
                continue
            states += 1 + (int(operands[0]) if o == "s_nop" else 0)
            if target is not None and o.startswith(("s_branch", "s_cbranch")):
                todo.append((at[target], states))
            if not o.startswith(("s_branch", "s_endpgm", "s_setpc")):
                todo.append((j + 1, states))
    return products, bad


def _kernels(name, tmp_path):
    """{kernel: listing} of the built library's kernels whose mangled name matches."""
    so = glob.glob(os.path.join(os.path.dirname(distributed_llms_amd.__file__), "_C_kernels*.so"))[0]
    shutil.copy(so, tmp_path / "k.so")
    run = lambda *a: subprocess.run(a, cwd=tmp_path, check=True, capture_output=True, text=True).stdout
    run(f"{LLVM}/llvm-objdump", "--offloading", "k.so")
    out = {}
    for f in sorted(glob.glob(str(tmp_path / "*gfx950"))):
        if os.path.getsize(f) == 0 or not re.search(name, run(f"{LLVM}/llvm-readelf", "-sW", f)):
            continue
        kernel = None
        for line in run(f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", f).splitlines():
            m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if m:
                kernel = m[1] if re.search(name, m[1]) else None
                if kernel:
                    out[kernel] = []
            elif kernel:
                out[kernel].append(line)
    return out


@pytest.mark.skipif(not os.path.exists(f"{LLVM}/llvm-objdump"), reason="no llvm-objdump")
def test_no_result_of_an_asm_product_is_touched_early(tmp_path):
    if not glob.glob(os.path.join(os.path.dirname(distributed_llms_amd.__file__), "_C_kernels*.so")):
        pytest.skip("nothing built")
    tall = r"gemm_pf_kernelILi\d+ELi0ELb0ELi(9|10)E|gemm_pp_kernelILi256ELi\d+ELi(162|674)E"
    kernels = _kernels(tall, tmp_path)
    assert len(kernels) >= 12
    for kernel, listing in kernels.items():
        products, bad = early_accesses(listing)
        assert products >= 16, kernel                            # two K halves of eight columns past the eighth row
        assert not bad, (kernel, bad[:3])


def _lines(*code):
    return [f"\t{c.split(' // ')[0]} // {i * 4:012X}:{' <k+0x' + c.split(' // ')[1] + '>' if ' // ' in c else ''}" for i, c in enumerate(code)]


def test_the_check_sees_early_accesses():
    mfma = "v_mfma_f32_16x16x32_bf16 v[8:11], v[0:3], v[4:7], v[8:11]"
    assert early_accesses(_lines(mfma, "s_nop 15", "s_nop 15", "v_mov_b32_e32 v20, v9")) == (1, [])
    assert early_accesses(_lines(mfma, mfma, "v_mov_b32_e32 v20, v12")) == (2, [])
    for late in ("v_mov_b32_e32 v20, v9", "v_accvgpr_write_b32 a3, v8", "v_mov_b32_e32 v11, 0", "global_store_dwordx4 v30, v[8:11], s[2:3]",
                 "v_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[4:7], a[0:3]", "v_mfma_f32_16x16x32_bf16 v[10:13], v[0:3], v[4:7], v[10:13]"):
        assert len(early_accesses(_lines(mfma, "s_nop 3", late))[1]) == 1, late
    loop = _lines("v_mov_b32_e32 v20, v9", "s_nop 15", mfma, "s_cbranch_scc1 65532 // 0", "s_endpgm")
    assert len(early_accesses(loop)[1]) == 1
