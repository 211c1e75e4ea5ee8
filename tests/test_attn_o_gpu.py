"""Decode attention and the o-projection in one launch (csrc/kernels/attention.hip, attn_o_kernel) against the two launches."""
import pytest
import torch

from distributed_llms_amd import knobs, ops
from distributed_llms_amd.ops import gemm
from distributed_llms_amd.ops import reference as ref

D, BS = 128, 32


def _case(lens, hq, hkv, n, parts, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    b, width = len(lens), (hq + 2 * hkv) * D
    blocks = [-(-x // BS) for x in lens]
    order = (torch.randperm(sum(blocks), generator=torch.Generator().manual_seed(seed)) + 1).tolist()
    table = torch.zeros(b, max(max(blocks), 1) + 1, dtype=torch.int32)
    for i, c in enumerate(blocks):
        table[i, :c] = torch.tensor(order[sum(blocks[:i]):sum(blocks[:i]) + c], dtype=torch.int32)
    slots = [int(table[i, (x - 1) // BS]) * BS + (x - 1) % BS if x else 0 for i, x in enumerate(lens)]
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    kc, vc = r(sum(blocks) + 1, hkv, BS, D).bfloat16(), r(sum(blocks) + 1, hkv, D, BS).bfloat16()
    if parts:
        ws = (r(parts * b * width) / 64 * parts ** -0.5).half()
        qkv = gemm.SplitKPartial(torch.cat([ws, ws.new_zeros(8)]).view(torch.float32), parts, b, width, (b, width), torch.bfloat16, ws.device)
    else:
        qkv = r(b, width).bfloat16()
    wo = (r(n, hq * D) * (hq * D) ** -0.5).bfloat16()
    cs = ref.rope_cos_sin(D, 1024, 5e5, None, device="cuda")
    return qkv, i32([max(x - 1, 0) for x in lens]), cs, kc, vc, i32(slots), table.cuda(), i32(lens), wo


# contexts at the edges of blocks, of splits and of the bucket, none at all, two sequences of different lengths; eight, four and two kv heads,
# one round of workgroups and three quarters of one; the projection's input whole and in every number of slabs that has a build of its own and one that has not
@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[1], [31], [32], [33], [64], [65], [129], [255], [256], [257], [511], [512], [1, 256], [200, 33], [64, 0], [97, 96]])
@pytest.mark.parametrize("hq,hkv,n,parts", [(32, 8, 4096, 5), (32, 8, 3072, 0), (16, 4, 8192, 4), (8, 2, 12288, 8), (32, 8, 4096, 3)])
def test_attention_and_projection(cuda, lens, hq, hkv, n, parts):
    qkv, pos, cs, kc, vc, slots, table, sl, wo = _case(lens, hq, hkv, n, parts, sum(lens) + hq)
    k1, v1 = kc.clone(), vc.clone()
    got = ops.paged_attention_decode_o(qkv, pos, cs, k1, v1, slots, table, sl, hq, hkv, D, D ** -0.5, wo, max_ctx=max(lens))
    assert got is not None and got.splits == hkv
    y = got.materialize()
    a = ops.paged_attention_decode_rope(qkv, pos, cs, kc, vc, slots, table, sl, hq, hkv, D, D ** -0.5, max_ctx=max(lens))
    assert torch.equal(k1, kc) and torch.equal(v1, vc)
    want = a.view(len(lens), -1).double() @ wo.double().T
    mag = a.view(len(lens), -1).double().abs() @ wo.double().abs().T
    # the attention's own rounding to bf16 (other splits of the keys: a last bit of each of hq * 128 values, as if of one sign), slabs of
    # 11 bits and at least 2^-18, and the bf16 result
    assert bool(((y.double() - want).abs() <= (2.0 ** -8 + 2.0 ** -11 + 2.0 ** -18) * mag + 2.0 ** -8 * want.abs() + hkv * 2.0 ** -18).all())
    assert ((y.double() - want).norm() <= 6e-3 * want.norm()) or not any(lens)


@pytest.mark.gpu
@pytest.mark.parametrize("ctx", [37, 64, 200])
def test_equal_bits_where_the_splits_are(cuda, ctx):
    """One sequence of up to 256 keys of which no split is cut otherwise than in the launch of its own."""
    qkv, pos, cs, kc, vc, slots, table, sl, wo = _case([ctx], 32, 8, 4096, 5, ctx)
    table = torch.cat([table, table.new_zeros(1, 8 - table.shape[1])], 1)                 # 256 keys: splits of 64
    got = ops.paged_attention_decode_o(qkv, pos, cs, kc.clone(), vc.clone(), slots, table, sl, 32, 8, D, D ** -0.5, wo, max_ctx=256)
    a = ops.paged_attention_decode_rope(qkv, pos, cs, kc, vc, slots, table, sl, 32, 8, D, D ** -0.5, max_ctx=256)
    assert torch.equal(got.materialize(), ops.linear(a.view(1, -1), wo, defer=True).materialize())


# every number of splits that has a build of its own and those between, with empty ones (short sequences in a wide table) and none of a
# sequence's at all; one to sixteen sequences, also where the attention joins its splits itself
@pytest.mark.gpu
@pytest.mark.parametrize("lens,width", [([600], 0), ([1000, 30], 0), ([513], 32), ([200, 90, 1], 0), ([33, 64, 0, 250], 8), ([90, 80, 70, 60, 50, 40], 0),
                                        ([250] * 8, 8), ([40, 33] * 4, 8), ([300, 10, 20, 500], 16), ([100] * 16, 4), ([900, 900], 32)])
@pytest.mark.parametrize("hq,hkv,n,parts", [(32, 8, 4096, 5), (16, 4, 6144, 0)])
def test_joined_in_the_projection(cuda, lens, width, hq, hkv, n, parts):
    qkv, pos, cs, kc, vc, slots, table, sl, wo = _case(lens, hq, hkv, n, parts, sum(lens) + len(lens))
    table = torch.cat([table, table.new_zeros(len(lens), max(0, width - table.shape[1]))], 1)
    ctx = max(max(lens), 32 * width)
    k1, v1 = kc.clone(), vc.clone()
    got = ops.paged_attention_decode_o(qkv, pos, cs, k1, v1, slots, table, sl, hq, hkv, D, D ** -0.5, wo, max_ctx=ctx)
    dense = lambda t: t.materialize() if isinstance(t, gemm.SplitKPartial) else t
    got = dense(got)
    a = ops.paged_attention_decode_rope(qkv, pos, cs, kc, vc, slots, table, sl, hq, hkv, D, D ** -0.5, max_ctx=ctx)
    splits = ops.decode_split_plan(len(lens), hkv, ctx, BS, table.shape[1])[0]
    assert (got is not None) == (1 < splits <= 16 and len(lens) * splits <= 32), splits
    if got is None:
        return
    assert torch.equal(k1, kc) and torch.equal(v1, vc)
    assert torch.equal(got, dense(ops.linear(a.view(len(lens), -1), wo, defer=True)))


@pytest.mark.gpu
def test_replays(cuda):
    """A captured step, replayed with other lengths and keys between eager work, against the eager call."""
    qkv, pos, cs, kc, vc, slots, table, sl, wo = _case([150, 60], 32, 8, 4096, 5, 3)
    call = lambda: ops.paged_attention_decode_o(qkv, pos, cs, kc, vc, slots, table, sl, 32, 8, D, D ** -0.5, wo, max_ctx=192).materialize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = call()
    torch.cuda.current_stream().wait_stream(side)
    for lens in ([150, 60], [33, 1], [149, 59]):
        sl.copy_(torch.tensor(lens, dtype=torch.int32))
        kc.mul_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, call())


def test_rule():
    """One or two sequences of up to 512 keys together, heads of 128 in groups of up to four, one round of workgroups."""
    f = ops.attn_o_splits
    assert f(1, 37, 32, 8, 128, 4096) == 4 and f(1, 256, 32, 8, 128, 4096) == 4 and f(1, 257, 32, 8, 128, 4096) == 2
    assert f(2, 256, 32, 8, 128, 4096) == 2
    assert not f(1, 513, 32, 8, 128, 4096) and not f(2, 257, 32, 8, 128, 4096) and not f(3, 10, 32, 8, 128, 4096)
    # only where the projection's own plan has a slice per kv head: every slice's sum passes through a 16-bit slab
    for hq, hkv, n in ((24, 8, 3072), (16, 16, 2048), (8, 8, 4096), (20, 20, 1536), (32, 32, 1024), (16, 8, 4096), (20, 10, 2560)):
        assert gemm.wide_splits(1, n, hq * 128) != hkv and not f(1, 37, hq, hkv, 128, n)
    for hq, hkv, n in ((32, 8, 4096), (16, 4, 8192), (8, 2, 12288), (20, 5, 6144), (64, 16, 2048)):
        assert gemm.wide_splits(1, n, hq * 128) == gemm.wide_splits(16, n, hq * 128) == hkv and f(1, 37, hq, hkv, 128, n)
    assert not f(1, 10, 64, 8, 128, 8192) and not f(1, 10, 32, 8, 64, 4096) and not f(1, 10, 32, 32, 128, 4096) and not f(1, 10, 32, 8, 128, 2048)
    gemm.reserve_cus_for_comm(4)
    try:
        assert not f(1, 37, 32, 8, 128, 4096)
    finally:
        gemm.release_cus_for_comm()
    with knobs.override(attn_o=False):
        assert not f(1, 37, 32, 8, 128, 4096)
    with knobs.override(one=False):
        assert f(1, 37, 32, 8, 128, 4096)
