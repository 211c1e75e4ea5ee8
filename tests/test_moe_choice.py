"""A mixture whose choice of experts is given (ops.moe.forward's ``choice``)."""
import pytest
import torch

from distributed_llms_amd import _ext, knobs
from distributed_llms_amd.ops import moe, quant
from distributed_llms_amd.ops import reference as ref


def _case(t, top, h=128, i=128, device="cpu", dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(t + top)
    r = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(dtype).to(device)     # noqa: E731
    ids = torch.stack([torch.randperm(8, generator=g)[:top] for _ in range(t)]).to(torch.int32).to(device)
    return r(t, h), r(8, h, scale=0.1), r(8, 2 * i, h, scale=0.05), r(8, h, i, scale=0.05), torch.rand(t, top, generator=g).to(device), ids


@pytest.mark.parametrize("t,top", [(1, 1), (3, 2), (40, 2)])
def test_taken_on_the_cpu(t, top):
    x, wr, gu, dn, tw, ids = _case(t, top)
    want = ref.moe_mlp(x, gu, dn, tw, ids)
    assert torch.equal(moe.forward(x, wr, gu, dn, top, choice=(tw, ids)), want)
    assert not torch.equal(moe.forward(x, wr, gu, dn, top), want)
    half = moe.forward(x, wr, gu[4:], dn[4:], top, 4, choice=(tw, ids))
    assert torch.equal(half, ref.moe_mlp(x, gu[4:], dn[4:], tw, ids - 4))
    q = quant.quantize_experts(gu), quant.quantize_experts(dn)
    assert torch.equal(moe.forward(x, wr, *q, top, choice=(tw, ids)), quant.moe_mlp_ref(x, *q, tw, ids))


def test_forms_refused():
    x, wr, gu, dn, tw, ids = _case(3, 2)
    for choice in ((tw[:2], ids), (tw, ids.long()), (tw.bfloat16(), ids), (tw[:, :1], ids[:, :1]), (tw.T.contiguous().T, ids)):
        with pytest.raises(ValueError, match="choice"):
            moe.forward(x, wr, gu, dn, 2, choice=choice)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("t", [1, 40])
def test_other_activations_refused(cuda, dtype, t):
    """The launches behind a choice are bf16 ones; nothing is launched for other activations."""
    x, wr, gu, dn, tw, ids = _case(t, 2, device="cuda", dtype=dtype)
    with pytest.raises(ValueError, match="bf16"):
        moe.forward(x, wr, gu, dn, 2, choice=(tw, ids))


@pytest.mark.parametrize("call", ["combine", "combine_norm"])
def test_combine_needs_slots_or_choices(call):
    """Neither slots nor choices, or choices of more pairs than a wave has lanes: an error in front of the launch."""
    k = _ext.kernels()
    for inv, ids, t in ((0, 0, 4), (0, 64, 33)):
        with pytest.raises(RuntimeError, match="pairs"):
            if call == "combine":
                k.moe_combine(64, 64, 64, inv, t, 64, 2, 0, ids)
            else:
                k.moe_combine_norm(64, 64, 64, 64, inv, ids, 64, t, 64, 2, 1e-5, 0)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("given", [False, True])
def test_no_tokens(device, given):
    x, wr, gu, dn, tw, ids = _case(1, 2, device=device)
    for defer in (False, True):
        out = moe.forward(x[:0], wr, gu, dn, 2, choice=(tw[:0], ids[:0]) if given else None, defer=defer)
        assert out.shape == (0, 128) and out.dtype == x.dtype


@pytest.mark.gpu
@pytest.mark.parametrize("t,top", [(1, 2), (3, 2), (8, 1)])
def test_either_kernel_can_be_forced(cuda, t, top, monkeypatch):
    """Which kernel serves the experts' products of few pairs: by the line, by the line alone, and by knobs that put it behind or in front of them."""
    x, wr, gu, dn, tw, ids = _case(t, top, h=128, i=16384, device="cuda")

    class Spy:
        def __init__(self, k, calls):
            self.k, self.calls = k, calls

        def __getattr__(self, name):
            f = getattr(self.k, name)
            if name.startswith("moe_") and name.endswith("_gemm"):
                return lambda *a: self.calls.append(name) or f(*a)
            return f

    k, calls = _ext.kernels(), []
    monkeypatch.setattr(_ext, "kernels", lambda: Spy(k, calls))
    want = None
    for kn, first in (({}, "moe_wide_gemm"), ({"moe_wide_fill": False}, "moe_wide_gemm" if t * top >= 8 else "moe_grouped_gemm"),
                      ({"moe_wide_fill": False, "moe_wide_min_pairs": 1000}, "moe_grouped_gemm"), ({"moe_wide_min_pairs": 0}, "moe_grouped_gemm"),
                      ({"moe_wide_min_pairs": 1}, "moe_wide_gemm")):
        calls.clear()
        with knobs.override(**kn):
            out = moe.forward(x, wr, gu, dn, top, choice=(tw, ids)).float()
        assert calls[0] == first and len(calls) == 2
        want = out if want is None else want
        assert (out - want).norm() <= 2 * 2.0 ** -8 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("t,top,h", [(1, 1, 8320), (1, 2, 4224), (2, 1, 8192)])
def test_wide_down_projections_of_few_pairs(cuda, t, top, h):
    """One or two pairs whose tiles of 32 columns are more than a round of the CUs keep the launches behind a slot list."""
    x, wr, gu, dn, tw, ids = _case(t, top, h=h, i=1024, device="cuda")
    if t == 2:
        ids[:, 0] = torch.tensor([5, 2], dtype=torch.int32)
    out = moe.forward(x, wr, gu, dn, top, choice=(tw, ids))
    pairs, moe.PICK_PAIRS = moe.PICK_PAIRS, 0
    try:
        assert torch.equal(out, moe.forward(x, wr, gu, dn, top, choice=(tw, ids)))
    finally:
        moe.PICK_PAIRS = pairs
