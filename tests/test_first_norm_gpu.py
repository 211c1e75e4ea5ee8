"""The embedding and the first sublayer's norm in one launch: the bits of the two launches, at the edges of its row pieces."""
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
