"""The first sublayer's norm in the embedding's launch, the last one in the last close's: the bits of the two launches, at the edges
of the row's pieces."""
import pytest
import torch

from distributed_llms_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("layer", [False, True])
@pytest.mark.parametrize("width", [8, 1000, 1024, 1028, 2048, 2056, 3072, 3080, 4096, 8192, 8200])
@pytest.mark.parametrize("tokens", [1, 5])
def test_embedding_first_norm_bit_exact(cuda, dtype, layer, width, tokens):
    g = torch.Generator().manual_seed(width)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype).to(cuda)
    table, w, b = r(37, width), r(width), r(width) if layer else None
    ids = torch.tensor([0, 36, 7, -3, 99][:tokens], dtype=torch.int32, device=cuda)        # (out of range: the nearest row)
    x, y = sm.embedding_first_norm(ids, table, w, 1e-6, dtype, 3.5, b)
    want = sm.embedding_f32(ids, table, 3.5)
    norm = sm.layer_norm_f32(want, w, b, 1e-6, dtype) if layer else sm.rms_norm_f32(want, w, 1e-6, dtype)
    assert torch.equal(x, want) and torch.equal(y, norm)


@pytest.mark.parametrize("dtype,parts", [(torch.bfloat16, 0), (torch.bfloat16, 3), (torch.float32, 0)])
@pytest.mark.parametrize("width", [8, 1000, 1024, 1028, 1032, 2048, 2056, 2560, 3072, 3080, 4096, 4104, 8192, 8200])
def test_last_norm_in_the_close_bit_exact(cuda, dtype, parts, width):
    """The norm behind the last sublayer in its close's launch: the stream and the normed rows of two launches, of finished
    products and of slabs."""
    from distributed_llms_amd.ops.gemm import SplitKPartial
    g = torch.Generator().manual_seed(width)
    rows = 5
    r = lambda *s: torch.randn(*s, generator=g).to(dtype).to(cuda)
    x, o, bias, wp, wn = torch.randn(rows, width, generator=g).to(cuda), r(rows, width), r(width), r(width) * 0.2, r(width) * 0.2
    if parts:
        o = SplitKPartial((torch.randn(parts, rows, width, generator=g) / 64).half().to(cuda), parts, rows, width, (rows, width), dtype, x.device)
    a, h = sm.post_norm_add(x.clone(), o, wp, 1e-6, 0.75, bias=bias, w_next=wn, final=True)
    want, _ = sm.post_norm_add(x.clone(), o, wp, 1e-6, 0.75, bias=bias)
    assert torch.equal(a, want) and torch.equal(h, sm.rms_norm_f32(want, wn, 1e-6, dtype))
