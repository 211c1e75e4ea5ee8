"""One row's products with the norm in front of them (csrc/kernels/gemm_one.hip): the bits of the launches they replace."""
import pytest
import torch

from distributed_llms_amd import _ext, knobs, ops
from distributed_llms_amd.ops import gemm


def _slabs(count, k, seed):
    """``count`` slabs of a row as a product of one row leaves them, in a workspace of their own."""
    g = torch.Generator("cuda").manual_seed(seed)
    ws = torch.randn(count * k, generator=g, device="cuda").half().view(torch.float32)
    return gemm.SplitKPartial(ws, count, 1, k, (1, k), torch.bfloat16, ws.device)


def _apart(h, residual, norm_w, w, glu):
    with knobs.override(one=False, stream=False):
        if h is None:
            x, r = ops.rms_norm(residual, norm_w, 1e-5), residual
        else:
            x, r = ops.fused_add_rms_norm(h, residual.clone(), norm_w, 1e-5)
        y = ops.linear_swiglu(x, w) if glu else ops.linear(x, w, defer=True)
        return (y.materialize() if isinstance(y, gemm.SplitKPartial) else y), r


# widths at and between the edges of the row's pieces (2048 in one of 256 lanes x 8, 4096, 8192), slices of few and of many K-tiles and a
# shorter last one, small weights (default cache policy), GLUs from the first size that is taken
@pytest.mark.gpu
@pytest.mark.parametrize("n,k,glu", [(256, 1024, False), (6144, 4096, False), (3072, 2112, False), (640, 2048, False), (10240, 8192, False),
                                     (1280, 6400, False), (128, 8192, False), (21888, 1088, True), (28672, 4096, True), (22016, 576, True),
                                     (32768, 6208, True)])
@pytest.mark.parametrize("added", ["nothing", "a row", 2, 5, 8])
def test_norm_linear_bits(cuda, n, k, glu, added):
    torch.manual_seed(n + k)
    r = lambda *s: torch.randn(*s, device="cuda").bfloat16()
    w, norm_w, residual = (r(n, k) * k ** -0.5).bfloat16(), r(k), r(1, k)
    h = {"nothing": None, "a row": r(1, k)}[added] if isinstance(added, str) else _slabs(added, k, n)
    before = residual.clone()
    one = ops.norm_linear(h, residual, norm_w, 1e-5, w, swiglu=glu)
    assert one is not None and torch.equal(residual, before)
    y = one[0].materialize() if isinstance(one[0], gemm.SplitKPartial) else one[0]
    assert isinstance(one[0], gemm.SplitKPartial) != glu
    want, stream = _apart(h, residual, norm_w, w, glu)
    assert torch.equal(one[1], stream)
    assert torch.equal(y, want) and bool(torch.isfinite(y).all())


# whole products and slices, also of rows with values that are not finite
@pytest.mark.gpu
@pytest.mark.parametrize("n,k,glu", [(128, 64, False), (256, 192, False), (32768, 320, False), (128256, 1024, False), (4096, 4096, False),
                                     (4096, 14336, False), (8192, 8192, False), (256, 1600, False), (28672, 4096, True)])
@pytest.mark.parametrize("value", [0.0, float("inf"), float("nan")])
def test_row_bits(cuda, n, k, glu, value):
    torch.manual_seed(n + k)
    x, w = torch.randn(1, k, device="cuda").bfloat16(), (torch.randn(n, k, device="cuda") * k ** -0.5).bfloat16()
    x[0, k // 3] = value
    go = lambda: (lambda y: y.materialize() if isinstance(y, gemm.SplitKPartial) else y)(gemm.linear_wide(x, w, swiglu=glu, defer=not glu))
    y = go()
    with knobs.override(one=False):
        want = go()
    assert torch.equal(y.view(torch.int16), want.view(torch.int16)) if value == 0.0 else torch.equal(y.nan_to_num(7.0), want.nan_to_num(7.0))


@pytest.mark.gpu
def test_slabs_that_are_read_are_not_written(cuda):
    """A product's slabs lie in the workspace that the next product's are written to: the other half of it then."""
    torch.manual_seed(1)
    r = lambda *s: torch.randn(*s, device="cuda").bfloat16()
    k, n = 4096, 6144
    w1, w2, norm_w, x, residual = (r(k, k) / 64).bfloat16(), (r(n, k) / 64).bfloat16(), r(k), r(1, k), r(1, k)
    h = ops.linear(x, w1, defer=True)
    assert isinstance(h, gemm.SplitKPartial)
    dense = h.materialize()
    y, stream = ops.norm_linear(h, residual, norm_w, 1e-5, w2)
    assert torch.equal(h.materialize(), dense) and y.ws.data_ptr() != h.ws.data_ptr()
    want, s2 = ops.norm_linear(dense, residual, norm_w, 1e-5, w2)
    assert torch.equal(stream, s2) and torch.equal(y.materialize(), want.materialize())


def test_refused():
    """What keeps launches of its own: more rows than one, other types, no K split in front of slabs, small GLUs."""
    r = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)
    assert ops.norm_linear(None, r(1, 4096), r(4096), 1e-5, r(6144, 4096)) is None       # (not on the GPU)
    assert not gemm.one_fits(6144, 4100, 5) and not gemm.one_fits(6145, 4096, 5)
    assert not gemm.one_fits(4096, 8256, 1) and gemm.one_fits(4096, 8256, 2)
    assert gemm.one_fits(21888, 4096, 1, swiglu=True) and not gemm.one_fits(21760, 4096, 1, swiglu=True)
    assert not gemm.one_fits(32768, 4096, 2, swiglu=True)
    with knobs.override(one=False):
        assert not gemm.one_fits(6144, 4096, 5)


@pytest.mark.gpu
def test_launcher_refuses(cuda):
    k = _ext.kernels()
    x = torch.zeros(1, 16384, device="cuda").bfloat16()
    p, s = x.data_ptr(), torch.cuda.current_stream().cuda_stream
    for n, kk, splits, mode, part, nslabs, w, out in ((130, 512, 1, 0, 0, 0, 0, p), (128, 500, 1, 0, 0, 0, 0, p), (128, 8256, 1, 0, 0, 0, 0, p),
                                                       (128, 512, 2, 0, 0, 0, 0, p), (128, 512, 1, 1, p, 9, p, p), (128, 512, 1, 0, 0, 0, p, p),
                                                       (128, 512, 1, 1, p, 2, p, p)):
        with pytest.raises(RuntimeError):
            k.gemm_one(out, 0, p, n, kk, splits, mode, 0, p, p, part, nslabs, w, p, 1e-5, s)
