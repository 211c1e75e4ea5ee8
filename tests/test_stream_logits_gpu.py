"""Soft-capped float32 logits in the weight-streaming product's launch: the bits of the product and the cap in two launches."""
import pytest
import torch

from distributed_llms_amd import ops
from distributed_llms_amd.ops import gemm
from distributed_llms_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [0.0, 30.0])
@pytest.mark.parametrize("m,n,k", [(1, 32000, 1024), (8, 4096, 2560), (5, 1030, 192), (16, 513, 64), (16, 30000, 64), (17, 2048, 1024),
                                   (32, 9000, 512), (64, 1000, 256), (64, 8192, 1024)])
def test_stream_logits_bit_exact(cuda, m, n, k, cap):
    """Every number of weight rows per workgroup and of row groups, columns that are no multiple of four."""
    g = torch.Generator().manual_seed(n)
    x, w = (torch.randn(m, k, generator=g) * 3).bfloat16().to(cuda), torch.randn(n, k, generator=g).bfloat16().to(cuda)
    want = sm.softcap_f32(gemm.linear_stream(x, w), cap)
    assert torch.equal(gemm.stream_logits(x, w, cap), want)
    got = sm.logits_f32(x, w, cap)
    assert torch.equal(got, sm.softcap_f32(ops.linear(x, w), cap)) and got.dtype == torch.float32


def test_logits_of_other_products(cuda):
    """Rows, types and slices that the weight-streaming product does not take."""
    for dtype, m, k in ((torch.float32, 4, 256), (torch.bfloat16, 65, 256), (torch.bfloat16, 4, 100)):
        x, w = torch.randn(m, k, device=cuda).to(dtype), torch.randn(512, k, device=cuda).to(dtype)
        assert torch.equal(sm.logits_f32(x, w, 5.0), sm.softcap_f32(ops.linear(x, w), 5.0))
