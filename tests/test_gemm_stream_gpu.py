"""The weight-streaming decode GEMM (csrc/kernels/gemm_stream.hip) against float64, and the rule that picks it."""
import pytest
import torch
import torch.nn.functional as F

from distributed_llms_amd import knobs
from distributed_llms_amd.ops import gemm


def _close(y, ref, terms, k):
    """``ref``: float64 result, ``terms``: the sum of the magnitudes of its products.  An f32 sum of k products in any
    order is within k 2^-24 of that; the bf16 result rounds by 2^-9."""
    tol = k * 2.0 ** -24 * terms + 2.0 ** -8 * ref.abs() + 1e-30
    return bool(((y.double() - ref).abs() <= tol).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(1, 64), (40, 64), (50, 192), (1024, 1024), (3088, 2560), (4097, 576), (4128, 128)])
@pytest.mark.parametrize("bias", [False, True])
def test_stream_linear(cuda, m, n, k, bias):
    """One 16-row weight tile per workgroup and two (N > 4096), fewer K-tiles than waves, ragged last tiles of N."""
    x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn(n, k, device="cuda") * 0.05).bfloat16()
    b = torch.randn(n, device="cuda").bfloat16() if bias else None
    guard = torch.full((m * n + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
    y = gemm.linear_stream(x, w, b)
    ref = F.linear(x.double(), w.double(), None if b is None else b.double())
    mag = x.double().abs() @ w.double().abs().t() + (0 if b is None else b.double().abs())
    assert _close(y, ref, mag, k + 1)
    # nothing outside y: the same launch into a window of a larger buffer
    from distributed_llms_amd import _ext
    _ext.kernels().gemm_stream(guard.data_ptr(), x.data_ptr(), w.data_ptr(), 0 if b is None else b.data_ptr(), m, n, k, 0, 1,
                               0.0, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(guard[:m * n].view(m, n), y) and bool((guard[m * n:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 16, 31, 64])
@pytest.mark.parametrize("half,k", [(24, 64), (1536, 1024), (4112, 640)])
@pytest.mark.parametrize("glu", ["silu", "clipped", "gelu"])
@pytest.mark.parametrize("bias", [False, True])
def test_stream_glu(cuda, m, half, k, glu, bias):
    x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn(2 * half, k, device="cuda") * k ** -0.5).bfloat16()
    b = torch.randn(2 * half, device="cuda").bfloat16() if bias else None
    y = gemm.linear_stream(x, w, b, glu, 0.7)
    z = F.linear(x.double(), w.double(), None if b is None else b.double())
    mag = (x.double().abs() @ w.double().abs().t() + (0 if b is None else b.double().abs())) * (k + 1) * 2.0 ** -24
    g, u = z[:, :half], z[:, half:]
    if glu == "silu":
        ref = F.silu(g) * u
    elif glu == "clipped":
        g, u = g.clamp(max=0.7), u.clamp(-0.7, 0.7)
        ref = g * torch.sigmoid(1.702 * g) * (u + 1)
    else:
        ref = F.gelu(g, approximate="tanh") * u
    # |d act / d gate| <= 1.2, act <= |gate|, |u| (+ 1 where clipped): the sums' errors through the product; the hardware
    # exponential and reciprocal are within 2^-20 of exact; the result rounds to bf16
    up = u.abs() + (1 if glu == "clipped" else 0)
    tol = 1.2 * mag[:, :half] * up + (g.abs() + 1e-3) * mag[:, half:] + (2.0 ** -8 + 2.0 ** -18) * ref.abs() + 2.0 ** -22
    assert bool(((y.double() - ref).abs() <= tol).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(2048, 128), (2049, 192), (4096, 128), (4100, 64), (6143, 192), (6145, 128), (10240, 2048),
                                 (12289, 64), (8, 2048)])
def test_stream_rows_per_workgroup(cuda, m, n, k):
    """8, 16, 24 and 32 weight rows per workgroup in one and several rounds, x in one and two groups of 8 rows, last
    workgroups that hold one row; and the same as a GLU where n has halves."""
    x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn(n, k, device="cuda") * 0.05).bfloat16()
    y = gemm.linear_stream(x, w)
    ref, mag = F.linear(x.double(), w.double()), x.double().abs() @ w.double().abs().t()
    assert _close(y, ref, mag, k)
    if n % 2 == 0:
        h = n // 2
        g, u = ref[:, :h], ref[:, h:]
        y = gemm.linear_stream(x, w, None, "silu")
        # as test_stream_glu: the sums' errors through the product, the activation's 2^-20, the bf16 result
        e = mag * k * 2.0 ** -24
        tol = 1.2 * e[:, :h] * u.abs() + (g.abs() + 1e-3) * e[:, h:] + (2.0 ** -8 + 2.0 ** -18) * (F.silu(g) * u).abs() + 2.0 ** -22
        assert bool(((y.double() - F.silu(g) * u).abs() <= tol).all())


@pytest.mark.gpu
@pytest.mark.parametrize("half,k,m", [(1024, 128, 1), (1024, 128, 16), (4096, 64, 16), (5120, 64, 3), (7681, 64, 16), (10240, 64, 16),
                                      (3072, 2048, 1), (8192, 2048, 16)])
def test_stream_glu_rows_per_workgroup(cuda, half, k, m):
    """Every GLU cut (8, 8, 16, 24, 32, 24, 12 and 16 columns), with biases."""
    x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn(2 * half, k, device="cuda") * k ** -0.5).bfloat16()
    b = torch.randn(2 * half, device="cuda").bfloat16()
    z = F.linear(x.double(), w.double(), b.double())
    e = (x.double().abs() @ w.double().abs().t() + b.double().abs()) * (k + 1) * 2.0 ** -24
    g, u = z[:, :half], z[:, half:]
    ref = F.silu(g) * u
    tol = 1.2 * e[:, :half] * u.abs() + (g.abs() + 1e-3) * e[:, half:] + (2.0 ** -8 + 2.0 ** -18) * ref.abs() + 2.0 ** -22
    assert bool(((gemm.linear_stream(x, w, b, "silu").double() - ref).abs() <= tol).all())


@pytest.mark.gpu
@pytest.mark.parametrize("glu", ["clipped", "gelu"])
def test_stream_glu_keeps_the_gate_kernels_arithmetic(cuda, glu):
    """Products of one term each are exact in f32, so the epilogue's result is the f32 gate kernel's, rounded once: bit for
    bit, over gates where the hardware exponential and reciprocal are several f32 ulps off (a million elements)."""
    from distributed_llms_amd.ops import seqmix as sm
    m, k, half = 64, 1024, 16384
    x = torch.linspace(-9, 3, m * k, device="cuda")[torch.randperm(m * k, device="cuda")].view(m, k).bfloat16()
    w = torch.zeros(2 * half, k, device="cuda", dtype=torch.bfloat16)
    rows = torch.arange(2 * half, device="cuda")
    w[rows, torch.randint(0, k, (2 * half,), device="cuda")] = (torch.rand(2 * half, device="cuda") * 2 + 0.5).bfloat16()
    gu = F.linear(x.double(), w.double()).float()
    want = sm.clipped_glu(gu, None, 7.0) if glu == "clipped" else sm.gelu_glu(gu)
    assert torch.equal(gemm.linear_stream(x, w, None, glu, 7.0), want.bfloat16())


@pytest.fixture
def counted(monkeypatch):
    """The calls that reach the kernel's entry point."""
    calls, real = [], gemm._stream
    monkeypatch.setattr(gemm, "_stream", lambda *a, **kw: (calls.append(a), real(*a, **kw))[1])
    return calls


@pytest.mark.gpu
def test_stream_is_reached_and_matches_the_wide_route(cuda, counted):
    """ops.linear / linear_swiglu at decode sizes take the kernel by default; knobs.stream off gives the former route."""
    from distributed_llms_amd import ops
    x = torch.randn(9, 1024, device="cuda").bfloat16()
    w = (torch.randn(2048, 1024, device="cuda") * 0.03).bfloat16()
    for f in (lambda: ops.linear(x, w), lambda: ops.linear_swiglu(x, w), lambda: ops.linear(x[:, None], w)):
        a = f()
        assert len(counted) == 1
        with knobs.override(stream=False):
            b = f()
        assert len(counted) == 1
        counted.clear()
        assert a.shape == b.shape
        torch.testing.assert_close(a.float(), b.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,reached", [(16, 2560, True), (17, 2560, False), (16, 4096, False), (64, 512, True), (65, 512, False)])
def test_stream_in_front_of_a_close(cuda, counted, m, n, reached):
    """linear_into_norm on both sides of its cutover: the finished product, or the slabs of a split grid."""
    from distributed_llms_amd import ops
    k = 1024 if n == 512 else 2560
    x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn(n, k, device="cuda") * 0.03).bfloat16()
    y = ops.linear_into_norm(x, w)
    assert len(counted) == reached and isinstance(y, torch.Tensor) >= reached
    y = y if isinstance(y, torch.Tensor) else y.materialize()
    torch.testing.assert_close(y.float(), x.float() @ w.float().t(), atol=2e-2, rtol=2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("m,reached", [(1, True), (64, True), (65, False)])
@pytest.mark.parametrize("biased", [False, True])
def test_stream_under_the_clipped_glu(cuda, counted, m, reached, biased):
    from distributed_llms_amd.ops import seqmix as sm
    x, w = torch.randn(m, 1024, device="cuda").bfloat16(), (torch.randn(3072, 1024, device="cuda") * 0.03).bfloat16()
    b = torch.randn(3072, device="cuda").bfloat16() if biased else None
    y = sm.linear_clipped_glu(x, w, b, 0.7)
    assert len(counted) == reached
    gu = x.float() @ w.float().t() + (0 if b is None else b.float())
    torch.testing.assert_close(y.float(), sm.clipped_glu(gu, None, 0.7), atol=2e-2, rtol=2e-2)


def test_stream_rule():
    assert gemm.stream_fits(1, 1024, 1024) and gemm.stream_fits(64, 5120, 2560) and not gemm.stream_fits(65, 1024, 1024)
    assert not gemm.stream_fits(8, 1024, 1000) and not gemm.stream_fits(8, 128256, 4096)
    assert gemm.stream_fits(32, 6144, 4096) and not gemm.stream_fits(33, 6144, 4096)
    assert gemm.stream_fits(16, 2560, 2560, defer=True) and not gemm.stream_fits(17, 2560, 2560, defer=True)
    assert not gemm.stream_fits(1, 4096, 4096, defer=True)             # the 8B projections stay on the wide kernel
    assert not gemm.stream_fits(1, 28672, 4096, "silu") and gemm.stream_fits(64, 15360, 2560, "gelu")
    assert not gemm.stream_fits(8, 1024, 448)
    # long K and many rows, few columns: staging x once per workgroup costs more than the saved launch
    assert gemm.stream_fits(16, 2048, 8192) and not gemm.stream_fits(17, 2048, 8192) and not gemm.stream_fits(16, 1024, 14336)
    assert gemm.stream_fits(32, 1024, 4096) and not gemm.stream_fits(33, 1024, 4096) and gemm.stream_fits(33, 1024, 4096, bias=True)
    assert not gemm.stream_fits(33, 500, 8192) and gemm.stream_fits(64, 500, 4096)
    assert not gemm.stream_fits(16, 1024, 8192, defer=True) and not gemm.stream_fits(17, 512, 4096, defer=True)
    assert gemm.stream_fits(16, 32000, 1024) and not gemm.stream_fits(17, 32000, 1024) and not gemm.stream_fits(16, 8192, 4096)
    assert gemm.stream_fits(16, 5120, 4096) and not gemm.stream_fits(32, 5120, 4096)
    # GLU: past 16 rows a round of workgroups that leaves CUs idle (up to 16 they are cut evenly), K past 4096
    assert gemm.stream_fits(32, 16384, 4096, "gelu") and not gemm.stream_fits(17, 22016, 4096, "gelu")
    assert not gemm.stream_fits(17, 10240, 4096, "silu") and not gemm.stream_fits(1, 4096, 8192, "clipped")
    x, w = torch.zeros(4, 512, dtype=torch.bfloat16), torch.zeros(256, 512, dtype=torch.bfloat16)
    assert gemm.use_stream(4, 256, 512, x, w)
    assert not gemm.use_stream(4, 256, 512, x.float(), w) and not gemm.use_stream(4, 256, 512, x, w.t().contiguous().t())
    assert not gemm.use_stream(4, 256, 512, x, torch.zeros(256 * 512 + 1, dtype=torch.bfloat16)[1:].view(256, 512))
    with knobs.override(stream=False):
        assert not gemm.use_stream(4, 256, 512, x, w)


def test_stream_rule_up_to_16_rows():
    """The line where a workgroup's rows follow the CU's share: further out than past 16 rows, on both sides of it."""
    assert gemm.stream_fits(16, 6144, 4096) and gemm.stream_fits(8, 10240, 8192) and not gemm.stream_fits(9, 10240, 8192)
    assert gemm.stream_fits(16, 5120, 5120) and not gemm.stream_fits(8, 4096, 8192)
    assert not gemm.stream_fits(16, 2560, 7680, defer=True)
    assert gemm.stream_fits(16, 16384, 4096, "silu") and not gemm.stream_fits(17, 16384, 4096, "silu")
    assert gemm.stream_fits(16, 14336, 5120, "silu") and not gemm.stream_fits(1, 27648, 5120, "silu")


def test_stream_rule_of_glus_up_to_16_rows_follows_the_cut():
    """A GLU's workgroups of up to 16 rows are cut evenly, so no size is left out for a round of 16 or 32 columns that they do not
    have; with 4 KiB strides and two groups of x the line lies at two rounds of 24 rows."""
    for m in (1, 8, 16):
        assert all(gemm.stream_fits(m, n, k, "silu") for n, k in ((10240, 4096), (22016, 4096), (17408, 2560), (11008, 5120), (24576, 2048)))
    assert not gemm.stream_fits(17, 10240, 4096, "silu") and not gemm.stream_fits(32, 22016, 4096, "clipped")
    assert gemm.stream_fits(8, 27648, 2048, "silu") and not gemm.stream_fits(9, 27648, 2048, "silu")
    assert gemm.stream_fits(16, 27648, 2560, "silu")
