"""Products of 65 to 512 rows in waves that multiply and waves that stage (csrc/kernels/gemm_duo.hip): gemm_wide's bits."""
import pytest
import torch
import torch.nn.functional as F

from distributed_llms_amd import _ext, knobs, ops
from distributed_llms_amd.ops import gemm


def _xw(m, n, k, seed=0):
    g = torch.Generator("cuda").manual_seed(seed + m * 7 + n + k)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    return r(m, k).bfloat16(), (r(n, k) * k ** -0.5).bfloat16()


# rows at the edges of the row tiles, one and more of them; slices of one K-tile to more than the ring holds and than a long slice's line (24), a
# shorter last one, slices in front of which the ring is not even full
@pytest.mark.gpu
@pytest.mark.parametrize("bm,m", [(128, 1), (128, 65), (128, 128), (128, 129), (128, 256), (192, 129), (192, 192), (192, 193), (192, 384), (256, 193),
                                  (256, 255), (256, 256), (256, 257), (256, 512)])
@pytest.mark.parametrize("n,k,s", [(128, 128, 2), (256, 320, 2), (384, 1088, 4), (256, 3200, 2), (128, 8192, 5)])
def test_slabs_bits(cuda, bm, m, n, k, s):
    x, w = _xw(m, n, k)
    ws = gemm._workspace(x.device)
    st = torch.cuda.current_stream().cuda_stream
    se = _ext.kernels().gemm_wide(0, x.data_ptr(), w.data_ptr(), ws.data_ptr(), ws.numel(), m, n, k, s, 2, 1 | bm << 8, st)
    used = ws.view(torch.float16)[:se * m * n]
    want = used.clone()
    used.fill_(float("nan"))
    room = ws.view(torch.float16)[se * m * n:se * m * n + 4096]
    room.fill_(3.0)
    part = gemm._duo(x, w, m, n, k, s, bm, False, True)
    assert part.splits == se and torch.equal(used, want) and bool((room == 3.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("bm,m", [(128, 65), (128, 128), (192, 129), (192, 192), (256, 193), (256, 255), (256, 256)])
@pytest.mark.parametrize("n,k", [(256, 64), (512, 192), (384, 1024), (28672, 4096), (24576, 320)])
def test_swiglu_bits(cuda, bm, m, n, k):
    x, w = _xw(m, n, k)
    st = torch.cuda.current_stream().cuda_stream
    want = torch.empty(m, n // 2, device="cuda", dtype=torch.bfloat16)
    _ext.kernels().gemm_wide(want.data_ptr(), x.data_ptr(), w.data_ptr(), 0, 0, m, n, k, 1, 1, 33 | bm << 8, st)
    y = gemm._duo(x, w, m, n, k, 1, bm, True, False)
    assert torch.equal(y, want)
    z = x.double() @ w.double().T
    ref = F.silu(z[:, :n // 2]) * z[:, n // 2:]
    assert (y.double() - ref).norm() <= 2.0 ** -8 * ref.norm()                  # (one rounding to bf16 and f32 sums)


# one row tile's edges in each of the three; K-tiles fewer than the ring holds and more than gemm_wide's rotation needs
@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 65, 128, 129, 192, 193, 255, 256])
@pytest.mark.parametrize("n,k", [(256, 64), (512, 192), (384, 1088), (24576, 4096)])
def test_swiglu_bits_of_gemm_pp(cuda, m, n, k):
    """In gemm_pp's place: its sums from K's start, its gate and up rounded to bf16 in front of the SiLU."""
    x, w = _xw(m, n, k)
    want = torch.empty(m, n // 2, device="cuda", dtype=torch.bfloat16)
    _ext.kernels().gemm_pp(want.data_ptr(), x.data_ptr(), w.data_ptr(), 0, 0, m, n, k, 1, 1, gemm.PP_GATE_UP_VARIANT,
                           torch.cuda.current_stream().cuda_stream)
    assert torch.equal(gemm._duo(x, w, m, n, k, 1, 128 if m <= 128 else 192 if m <= 192 else 256, True, False, like_pp=True), want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,glu", [(96, 28672, 4096, True), (160, 28672, 4096, True), (200, 28672, 4096, True), (256, 28672, 4096, True),
                                       (65, 8192, 28672, False), (128, 10240, 8192, False), (160, 4096, 4096, False), (256, 4096, 4096, False), (320, 4096, 4096, False), (512, 4096, 4096, False),
                                       (200, 6144, 4096, False), (256, 4096, 14336, False), (384, 4096, 14336, False)])
def test_reached_by_the_products(cuda, m, n, k, glu, monkeypatch):
    """The calls that are meant to take this kernel take it, and give what the kernel gives that they would take (gemm_wide; a SwiGLU of 200
    rows and more gemm_pp)."""
    x, w = _xw(m, n, k)
    calls, duo = [], gemm._duo
    monkeypatch.setattr(gemm, "_duo", lambda *a: calls.append(1) or duo(*a))
    go = (lambda: ops.linear_swiglu(x, w)) if glu else (lambda: ops.linear(x, w))
    y = go()
    assert calls
    with knobs.override(duo=False):
        assert torch.equal(y, go())


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [gemm.PP_GATE_UP_VARIANT, 64 | 2, 64])
def test_a_caller_that_asks_for_gemm_pp_gets_it(cuda, variant, monkeypatch):
    x, w = _xw(256, 28672, 4096)
    monkeypatch.setattr(gemm, "_duo", lambda *a: pytest.fail("gemm_duo"))
    y = gemm.linear_pp(x, w, splits=1, swiglu=True, variant=variant)
    z = x.double() @ w.double().T
    want = F.silu(z[:, :14336]) * z[:, 14336:]
    assert (y.double() - want).norm() <= 3 * 2.0 ** -9 * want.norm()            # (gate, up and the result rounded to bf16)


@pytest.mark.gpu
def test_replays_into_the_norm(cuda):
    """Slabs that are stored past the L2, and the launch that sums them, in a graph replayed between eager work."""
    m, n, k = 256, 4096, 4096
    x, w = _xw(m, n, k)
    res, nw = torch.randn(m, n, device="cuda").bfloat16(), torch.randn(n, device="cuda").bfloat16()
    call = lambda: ops.fused_add_rms_norm(ops.linear(x, w, defer=True), res.clone(), nw, 1e-5)[0]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = call()
    torch.cuda.current_stream().wait_stream(side)
    for i in range(4):
        x.copy_(_xw(m, n, k, seed=i)[0])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, call())


@pytest.mark.gpu
def test_launcher_refuses(cuda):
    x = torch.zeros(1 << 20, device="cuda").bfloat16()
    p, s = x.data_ptr(), torch.cuda.current_stream().cuda_stream
    for m, n, k, splits, glu, bm, c, ws, room in ((128, 130, 512, 2, False, 128, 0, p, 1 << 19), (128, 128, 500, 2, False, 128, 0, p, 1 << 19),
                                                  (128, 128, 512, 1, False, 128, 0, p, 1 << 19), (128, 128, 512, 2, True, 128, p, 0, 0),
                                                  (128, 128, 512, 2, False, 64, 0, p, 1 << 19), (128, 128, 512, 2, False, 128, 0, p, 100),
                                                  (128, 128, 512, 1, True, 128, 0, 0, 0)):
        with pytest.raises(RuntimeError):
            _ext.kernels().gemm_duo(c, p, p, ws, room, m, n, k, splits, glu, bm, s)


def test_rule():
    f = gemm.duo_fits
    assert f(128, 28672, 4096, 1, 128, True) and f(256, 28672, 4096, 1, 256, True) and not f(64, 28672, 4096, 1, 64, True)
    assert not f(256, 16384, 4096, 1, 256, True) and not f(300, 28672, 4096, 1, 192, True)
    assert f(256, 4096, 14336, 8, 256) and f(129, 4096, 4096, 4, 128) and not f(128, 4096, 14336, 8, 128)
    assert f(128, 8192, 28672, 4, 128) and f(65, 8192, 8192, 4, 128) and not f(64, 8192, 28672, 4, 128) and not f(96, 6144, 4096, 5, 128)
    assert not f(256, 2048, 2048, 4, 256) and not f(256, 65536, 4096, 1, 256)
    with knobs.override(duo=False):
        assert not f(256, 4096, 14336, 8, 256)
    # past 256 rows: the slices that gemm_wide takes, on the row tile that makes one round of them
    for m, n, k, tile in ((320, 4096, 4096, 192), (400, 4096, 4096, 128), (512, 4096, 4096, 128), (300, 3072, 2048, 192), (512, 3072, 3072, 192),
                          (300, 2560, 2560, 128), (512, 2560, 2560, 0), (512, 2048, 2048, 128), (400, 4096, 14336, 256), (256, 4096, 4096, 128)):
        s, bm = gemm.wide_splits(m, n, k), gemm.wide_row_tile(m, n, k)
        assert gemm.duo_row_tile(m, n, k, s, bm) == tile
