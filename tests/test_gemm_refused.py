"""Calls in front of the weight-streaming GEMM that it must not get: the entry points refuse them or take another route.
The kernel entry points are stubbed, so that nothing is launched: the calls run on the CPU."""
import pytest
import torch

import torch.nn.functional as F

from distributed_llms_amd import _ext
from distributed_llms_amd.ops import gemm
from distributed_llms_amd.ops import seqmix as sm


class _Launches:
    """Stands in for the kernel module: counts what would have been launched."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *a: self.calls.append((name, a))


@pytest.fixture
def launches(monkeypatch):
    k = _Launches()
    monkeypatch.setattr(_ext, "kernels", lambda: k)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: type("S", (), {"cuda_stream": 0}))
    return k.calls


def _bf(*shape):
    return torch.zeros(*shape, dtype=torch.bfloat16)


GLU = {"linear": gemm.linear, "into_norm": gemm.linear_into_norm, "swiglu": gemm.linear_swiglu, "gelu": gemm.linear_gelu_glu,
       "clipped": lambda x, w: gemm.linear_clipped_glu(x, w, 7.0)}


@pytest.mark.parametrize("name", list(GLU))
@pytest.mark.parametrize("w", [(512, 512), (512, 2048), (512, 1024, 1)])
def test_operands_that_do_not_match_are_refused(launches, name, w):
    with pytest.raises(ValueError):
        GLU[name](_bf(4, 1024), _bf(*w))
    assert not launches
    GLU[name](_bf(4, 1024), _bf(512, 1024))                    # the same call with a weight that fits
    assert [n for n, _ in launches] == ["gemm_stream"]


@pytest.mark.parametrize("name", list(GLU))
def test_operands_on_two_devices_are_refused(launches, name):
    with pytest.raises(ValueError):
        GLU[name](_bf(4, 1024), torch.empty(512, 1024, dtype=torch.bfloat16, device="meta"))
    assert not launches


def test_bias_of_another_shape_goes_to_the_general_route(launches):
    """A bias that is not one element per output: added by its broadcast, or refused, as F.linear has it."""
    x, w = torch.randn(4, 1024).bfloat16(), torch.randn(512, 1024).bfloat16()
    for b in (torch.randn(1), torch.randn(4, 512), torch.randn(4, 1), torch.randn(1, 512)):
        assert torch.equal(gemm.linear(x, w, b.bfloat16()), F.linear(x, w, b.bfloat16()))
    for n in (0, 511, 513):
        with pytest.raises(RuntimeError):
            gemm.linear(x, w, _bf(n))
    with pytest.raises(RuntimeError):
        gemm.linear(x, w, torch.empty(512, dtype=torch.bfloat16, device="meta")).sum().item()
    assert not launches
    gemm.linear(x, w, _bf(512))
    assert [n for n, _ in launches] == ["gemm_stream"]


@pytest.mark.parametrize("bias", [_bf(1), _bf(511), _bf(1, 512), torch.zeros(512),
                                  torch.empty(512, dtype=torch.bfloat16, device="meta")])
def test_glu_bias_that_does_not_fit_is_refused(launches, bias):
    assert gemm.linear_clipped_glu(_bf(4, 1024), _bf(512, 1024), 7.0, bias) is None
    with pytest.raises(ValueError):
        sm.linear_clipped_glu(_bf(4, 1024), _bf(512, 1024), bias, 7.0)
    assert not launches


def test_recorded_calls_keep_their_derivatives(launches):
    """What F.linear differentiates or maps over is not taken from it: autograd, forward mode, vmap (N = 500 or a bias: the
    shapes of no other kernel)."""
    from torch.autograd import forward_ad
    x, w, b = torch.randn(4, 1024).bfloat16(), torch.randn(500, 1024).bfloat16(), torch.randn(500).bfloat16()
    for which in range(3):
        t = [x, w, b]
        t[which] = t[which].clone().requires_grad_()
        gemm.linear(*t).sum().backward()
        want = [x, w, b]
        want[which] = want[which].clone().requires_grad_()
        F.linear(*want).sum().backward()
        assert torch.equal(t[which].grad, want[which].grad)
    with forward_ad.dual_level():
        y = gemm.linear(forward_ad.make_dual(x, torch.ones_like(x)), w, b)
        assert torch.equal(forward_ad.unpack_dual(y).tangent, F.linear(torch.ones_like(x), w))
    assert torch.equal(torch.vmap(lambda v: gemm.linear(v, w, b))(x), torch.vmap(lambda v: F.linear(v, w, b))(x))
    assert not launches
    with torch.no_grad():
        gemm.linear(x.clone().requires_grad_(), w, b)
    assert [n for n, _ in launches] == ["gemm_stream"]


def test_traced_calls_keep_the_product(launches):
    """A traced graph holds the product, not the memory that a launch left behind while it was traced; a dispatch mode
    and a tensor subclass see the call."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode
    x, w, b = torch.randn(4, 1024).bfloat16(), torch.randn(500, 1024).bfloat16(), torch.randn(500).bfloat16()
    x2 = torch.randn(4, 1024).bfloat16()
    want = F.linear(x2, w, b)
    assert torch.equal(torch.jit.trace(lambda v: gemm.linear(v, w, b), x, check_trace=False)(x2), want)
    assert torch.equal(make_fx(lambda v: gemm.linear(v, w, b))(x)(x2), want)
    with FakeTensorMode() as mode:
        fake = [mode.from_tensor(t) for t in (x, w, b)]
    assert gemm.linear(*fake).shape == (4, 500)                 # (outside the mode: the tensors carry it)
    with FlopCounterMode(display=False) as flops:
        gemm.linear(x, w, b)
    assert flops.get_total_flops() == 2 * 4 * 500 * 1024
    assert not launches


def test_swiglu_of_an_odd_width_stays_refused(launches):
    """The SiLU GLU takes intermediate sizes in multiples of 8, at every number of rows."""
    for n in (1000, 1002):
        assert gemm.linear_swiglu(_bf(4, 1024), _bf(n, 1024)) is None and not launches
    gemm.linear_swiglu(_bf(4, 1024), _bf(1008, 1024))
    assert [n for n, _ in launches] == ["gemm_stream"]


def test_fp8_weight_in_front_of_a_norm():
    """linear_into_norm takes what linear(defer=True) takes: an fp8 weight too (latent_attention's output projection)."""
    from distributed_llms_amd import ops
    from distributed_llms_amd.ops import quant
    x, w = torch.randn(4, 256).bfloat16(), quant.quantize_weight(torch.randn(128, 256).bfloat16())
    assert torch.equal(ops.linear_into_norm(x, w), ops.linear(x, w, defer=True))
