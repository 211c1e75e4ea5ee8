"""Calls in front of the weight-streaming GEMM that it must not get: the entry points refuse them or take another route.
The kernel entry points are stubbed, so that nothing is launched: the calls run on the CPU."""
import pytest
import torch

from distributed_llms_amd import _ext, ops
from distributed_llms_amd.ops import gemm


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
