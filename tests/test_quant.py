"""FP8 W8A8 quantization on the CPU (ops/quant.py reference path; SURVEY §2.8 quantization row).

The reference only documents quantization (bitsandbytes int8/int4 + absmax fallback,
``plan.md:109-112,438-456``); there is no reference output to pin against, so parity is
unpinned and these tests check the scheme's own invariants."""
import pytest
import torch

from distributed_llms_amd import ops
from distributed_llms_amd.config import EngineConfig
from distributed_llms_amd.engine.llm_engine import LLMEngine, build_stage
from distributed_llms_amd.engine.sequence import SamplingParams
from distributed_llms_amd.ops import quant


def test_weight_quantization_is_per_channel_absmax():
    w = torch.randn(64, 96)
    w[3] *= 100                                   # one loud channel does not crush the others
    fw = quant.quantize_weight(w)
    assert fw.q.dtype == torch.float8_e4m3fn and fw.scale.shape == (64,)
    torch.testing.assert_close(fw.scale, w.abs().amax(1) / 448.0)
    assert fw.q.float().abs().amax(1).eq(448.0).all()        # every row uses the full range
    rel = (fw.dequantize() - w).norm(dim=1) / w.norm(dim=1)
    assert rel.max() < 0.04
    assert fw.nbytes() == 64 * 96 + 64 * 4


def test_zero_rows_quantize_to_zero_with_unit_scale():
    x = torch.zeros(3, 16)
    x[1] = torch.linspace(-2, 2, 16)
    q, s = quant.quantize_rows_ref(x)
    assert s[0] == 1 and s[2] == 1 and q[0].float().abs().sum() == 0
    assert q[1].float().abs().max() == 448.0


@pytest.mark.parametrize("swiglu", [False, True])
def test_linear_dispatches_fp8_weights(swiglu):
    torch.manual_seed(0)
    x, w = torch.randn(5, 64), torch.randn(32, 64) * 0.1
    fw = quant.quantize_weight(w)
    y = ops.linear_swiglu(x, fw) if swiglu else ops.linear(x, fw)
    ref = x @ w.t()
    if swiglu:
        g, u = ref.chunk(2, -1)
        ref = torch.nn.functional.silu(g) * u
    assert ((y - ref).norm() / ref.norm()) < 0.08
    with pytest.raises(ValueError):
        ops.linear(x, fw, bias=torch.zeros(32))


def test_stage_quantize_converts_projections_and_experts():
    ecfg = EngineConfig(model="tiny-mixtral", dtype="float32", device="cpu", quant="fp8")
    s = build_stage(ecfg)
    lw = s.layers[0]
    assert isinstance(lw["wqkv"], quant.Fp8Weight) and isinstance(lw["wo"], quant.Fp8Weight)
    assert isinstance(lw["experts_gate_up"], quant.Fp8Experts) and isinstance(lw["experts_down"], quant.Fp8Experts)
    skip = set(quant.QUANT_KEYS) | set(quant.EXPERT_KEYS)
    assert all(isinstance(t, torch.Tensor) for k, t in lw.items() if k not in skip)     # router, norms
    with pytest.raises(ValueError):
        EngineConfig(model="tiny-llama", quant="int3").validate()


def test_fp8_moe_tracks_the_bf16_moe():
    from distributed_llms_amd.ops import moe
    torch.manual_seed(1)
    t, h, i, e = 12, 64, 96, 4
    x = torch.randn(t, h)
    wr, gu, dn = torch.randn(e, h), torch.randn(e, 2 * i, h) * 0.1, torch.randn(e, h, i) * 0.1
    ref = moe.forward(x, wr, gu, dn, 2)
    out = moe.forward(x, wr, quant.quantize_experts(gu), quant.quantize_experts(dn), 2)
    assert ((out - ref).norm() / ref.norm()) < 0.08
    with pytest.raises(TypeError):
        moe.forward(x, wr, quant.quantize_experts(gu), dn, 2)


def test_cpu_engine_runs_fp8():
    base = EngineConfig(model="tiny-llama", dtype="float32", device="cpu", max_batch=4, max_seq_len=64,
                        num_kv_blocks=64, use_graphs=False)
    prompts = [[1, 2, 3, 4], [5, 6, 7]]
    sp = SamplingParams(max_new_tokens=6, ignore_eos=True)
    ref = LLMEngine(base).generate(prompts, sp)
    e8 = LLMEngine(base.apply_overrides(quant="fp8"))
    out = e8.generate(prompts, sp)
    assert [len(o) for o in out] == [6, 6]
    assert [o[0] for o in out] == [o[0] for o in ref]       # first greedy tokens agree
    assert e8.stage.weight_bytes() < LLMEngine(base).stage.weight_bytes() / 2


def test_fp8_prompt_plan_splits_no_further():
    """Past 256 rows: a product that the decode rule leaves whole stays whole and no other gets more slices (the slabs hold
    16 bits), the slabs fit the workspace, and one full round of 256-row tiles is left as it is."""
    from distributed_llms_amd.ops import gemm, quant
    for m in (257, 300, 449, 640, 1025, 2048, 2817, 5000, 70000):
        for n in (128, 1024, 4096, 6144, 28672):
            for k in (128, 640, 4096, 14336):
                for swiglu in (False, True):
                    s, bm = quant.fp8_plan(m, n, k, swiglu)
                    assert 1 <= s <= min(8, gemm.wide_splits(m, n, k // 2, swiglu))
                    assert bm in (64, 128, 192, 256) and (s == 1 or s * m * n <= gemm._WS_FLOATS)
    assert quant.fp8_plan(2048, 4096, 4096) == (1, 256) and quant.fp8_plan(2816, 4096, 4096) == (1, 192)


@pytest.mark.parametrize("m", [1, 8, 64, 100, 128, 300, 700])
def test_reserved_cus_leave_small_splits_alone(m):
    """Products whose K (not the number of CUs) sets the slices are split alike with CUs reserved for communication: the
    stages of a pipeline sum in the order of a single engine."""
    from distributed_llms_amd.ops import gemm, quant
    from distributed_llms_amd.parallel.rccl_transport import comm_cus
    shapes = [(256, 256), (512, 512), (1024, 1024), (512, 1024), (1024, 2048)]
    plans = lambda: [(gemm.wide_splits(m, n, k), quant.fp8_plan(m, n, k), quant.fp8_plan(m, n, k, True)) for n, k in shapes]
    alone = plans()
    gemm.reserve_cus_for_comm(comm_cus())
    try:
        assert plans() == alone
    finally:
        gemm.release_cus_for_comm()


@pytest.mark.parametrize("m", [1, 16, 64, 65, 128])
def test_fp8_decode_plan_keeps_slices_of_8_k_tiles(m):
    """A slice's sum is handed on in 16 bits, so no slice is shorter than 8 K-tiles, and where the reserved CUs leave room for
    as many slices as K gives, a pipeline's stages split as one engine does."""
    from distributed_llms_amd.ops import gemm, quant
    shapes = [(1024, 4096), (2048, 2048), (4096, 4096), (8192, 2048), (8192, 2560), (1280, 8192), (4096, 14336)]
    alone = [quant.fp8_plan(m, n, k) for n, k in shapes]
    assert all(s == 1 or k // 128 >= 8 * s for (n, k), (s, _) in zip(shapes, alone)), alone
    gemm.reserve_cus_for_comm(16)
    try:
        for (n, k), p in zip(shapes, alone):
            room = 240 // (n // 128 * -(-m // gemm.wide_row_tile(m, n, k // 2))) >= min(k // 1024, 16)
            assert not room or quant.fp8_plan(m, n, k) == p, (n, k, p)
    finally:
        gemm.release_cus_for_comm()


def test_fp8_prompt_plan_splits_alike_beside_communication():
    """Past 256 rows a product that the decode rule splits alike with and without CUs reserved for communication gets the same
    number of slices on both sides (the row tile may differ: it changes no bit)."""
    from distributed_llms_amd.ops import gemm, quant
    cases = [(m, n, k, sw) for m in (257, 300, 384, 513, 700, 1000, 2048, 4096) for n in (256, 512, 1024, 2560, 4096)
             for k in (512, 2048, 4096, 7680, 14336) for sw in (False, True)]
    plans = lambda: [(gemm.wide_splits(m, n, k // 2, sw), quant.fp8_plan(m, n, k, sw)) for m, n, k, sw in cases]
    alone = plans()
    gemm.reserve_cus_for_comm(16)
    try:
        beside = plans()
    finally:
        gemm.release_cus_for_comm()
    alike = [(c, a, b) for c, (x, a), (y, b) in zip(cases, alone, beside) if x == y]
    assert len(alike) > len(cases) // 2
    assert all(a[0] == b[0] and b[1] in (64, 128, 192, 256) for _, a, b in alike), [v for v in alike if v[1][0] != v[2][0]][:5]


def test_pf8_plan_takes_what_the_kernel_takes():
    """A row tile that gemm_pf8 is built for, only for sizes that it takes; small products stay on the plan's tiles."""
    from distributed_llms_amd.ops import quant
    for m in (257, 449, 1000, 2560, 8192, 100000):
        for n in (128, 256, 384, 4096, 28672):
            for k in (128, 256, 384, 512, 640, 4096, 14336):
                for bm in (64, 128, 192, 256):
                    rows = quant._pf8_plan(m, n, k, bm)
                    assert rows in (0, 160, 192, 224, 256)
                    assert not rows or (n % 256 == 0 and k % 256 == 0 and k >= 512 and m * k < 1 << 32 and m * n * 2 < 1 << 31)
    assert quant._pf8_plan(300, 512, 512, 64) == 0 and quant._pf8_plan(2560, 4096, 14336, 192) == 160
    assert quant._pf8_plan(8192, 28672, 4096, 256) == 256 and quant._pf8_plan(70000, 28672, 4096, 256) == 0


def test_fp8_weights_read_by_several_row_tiles_are_cached():
    """Nontemporal weights only where one row tile reads them (or the deep ring of 64-row tiles goes with it); short slices and
    small matrices keep the default policy."""
    from distributed_llms_amd.ops import quant
    policy = lambda m, n, k: quant.fp8_variant(m, n, k, *quant.fp8_plan(m, n, k)) & 7
    assert [policy(m, 4096, 14336) for m in (1, 64, 128)] == [1, 1, 1]
    assert [policy(m, 4096, 14336) for m in (129, 256, 300, 640, 1024)] == [4] * 5
    assert [policy(m, 8192, 28672) for m in (64, 200, 300)] == [1, 4, 4]
    assert quant.fp8_variant(300, 2048, 8192, 3, 64) & 7 == 1 and policy(300, 2048, 8192) == 4
    assert policy(1, 6144, 4096) == 1 and policy(100, 6144, 4096) == 4 and policy(64, 1024, 8192) == 4
    assert policy(64, 28672, 4096) == 1 and quant.fp8_variant(4096, 28672, 4096, 1, 256) == 4 | 64 | 256 << 8
    assert quant.fp8_variant(2100, 4096, 4096, 1, 192) == 4 | 64 | 192 << 8 and quant.fp8_variant(2100, 4096, 4096, 1, 0) == 4


def test_fp8_prompt_plan_splits_where_the_consumer_sums():
    """A split whose slabs the norm or the append sums costs no launch: narrow products of a few hundred rows are split rather than
    run as one round of short tiles; a GLU, which pays for the sum, sooner stays whole."""
    from distributed_llms_amd.ops import quant
    assert [quant.fp8_plan(m, 4096, 4096) for m in (300, 384, 500, 640)] == [(3, 192), (3, 192), (2, 128), (2, 192)]
    assert [quant.fp8_plan(m, 6144, 4096) for m in (257, 300, 384)] == [(2, 192)] * 3
    assert quant.fp8_plan(448, 8192, 8192) == (2, 256) and quant.fp8_plan(300, 2048, 8192) == (5, 128)
    assert quant.fp8_plan(900, 4096, 4096) == (1, 128) and quant.fp8_plan(448, 4096, 4096, True) == (1, 64)
