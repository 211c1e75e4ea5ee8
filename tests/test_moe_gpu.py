"""Mixtral MoE on the GPU (route + grouped expert GEMMs + combine) vs the fp32 PyTorch reference."""
import pytest
import torch
import torch.nn.functional as F

from distributed_llms_amd import ops
from distributed_llms_amd.ops import moe
from distributed_llms_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


def _bf(*s, scale=1.0):
    return (torch.randn(*s, device="cuda") * scale).to(torch.bfloat16)


@pytest.mark.parametrize("t", [1, 7, 64, 200, 300])
@pytest.mark.parametrize("e,k,h,i", [(8, 2, 512, 384), (4, 2, 256, 256), (8, 1, 256, 128)])
def test_moe_forward(cuda, t, e, k, h, i):
    x = _bf(t, h)
    wr = _bf(e, h, scale=0.1)
    wgu = _bf(e, 2 * i, h, scale=0.05)
    wd = _bf(e, h, i, scale=0.05)
    out = ops.moe_forward(x, wr, wgu, wd, k)
    # reference with the same bf16 router logits the GPU path routes on
    logits = ref.linear(x, wr).float()
    tw, tid = ref.moe_route(logits, k)
    expect = ref.moe_mlp(x.float(), wgu.float(), wd.float(), tw, tid)
    torch.testing.assert_close(out.float(), expect, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("t", [40, 100, 150])
def test_moe_skewed_routing_multi_chunk(cuda, t):
    """All tokens routed to the same two experts: far more rows per expert than the row tile the
    expected count selected (t*k/e -> 16/32/64-row tiles) exercises the row-chunk loop."""
    e, k, h, i = 8, 2, 256, 256
    x = _bf(t, h)
    wr = torch.zeros(e, h, device="cuda", dtype=torch.bfloat16)
    wr[3] = 0.05
    wr[5] = 0.04
    x = x.abs()                                   # positive rows -> experts 3 and 5 always win
    wgu, wd = _bf(e, 2 * i, h, scale=0.05), _bf(e, h, i, scale=0.05)
    out = moe.forward(x, wr, wgu, wd, k)
    tw, tid = ref.moe_route(ref.linear(x, wr).float(), k)
    assert set(tid.unique().tolist()) == {3, 5}
    expect = ref.moe_mlp(x.float(), wgu.float(), wd.float(), tw, tid)
    torch.testing.assert_close(out.float(), expect, atol=3e-2, rtol=3e-2)


def test_moe_graph_capturable(cuda):
    t, e, k, h, i = 32, 8, 2, 256, 256
    x, wr = _bf(t, h), _bf(e, h, scale=0.1)
    wgu, wd = _bf(e, 2 * i, h, scale=0.05), _bf(e, h, i, scale=0.05)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        moe.forward(x, wr, wgu, wd, k)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = moe.forward(x, wr, wgu, wd, k)
    for _ in range(2):
        x.copy_(_bf(t, h))
        g.replay()
        torch.cuda.synchronize()
        tw, tid = ref.moe_route(ref.linear(x, wr).float(), k)
        torch.testing.assert_close(out.float(), ref.moe_mlp(x.float(), wgu.float(), wd.float(), tw, tid),
                                   atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("t", [1, 7, 40, 64, 150, 256])
@pytest.mark.parametrize("skew", [False, True])
def test_moe_wide_grouped_kernel(cuda, monkeypatch, t, skew):
    """The MFMA-tiled grouped expert GEMM (gemm_wide.hip moe_wide_gemm) forced for every token
    count: 64-row tiles, 128-row chunks, multi-chunk experts (skewed routing) and empty experts."""
    from distributed_llms_amd import knobs
    monkeypatch.setattr(knobs.K, "moe_wide_min_pairs", 1)
    e, k, h, i = 8, 2, 512, 384
    x = _bf(t, h)
    if skew:
        x = x.abs()
        wr = torch.zeros(e, h, device="cuda", dtype=torch.bfloat16)
        wr[2] = 0.05
        wr[6] = 0.04
    else:
        wr = _bf(e, h, scale=0.1)
    wgu, wd = _bf(e, 2 * i, h, scale=0.05), _bf(e, h, i, scale=0.05)
    out = moe.forward(x, wr, wgu, wd, k)
    tw, tid = ref.moe_route(ref.linear(x, wr).float(), k)
    expect = ref.moe_mlp(x.float(), wgu.float(), wd.float(), tw, tid)
    torch.testing.assert_close(out.float(), expect, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("t,h,i", [(64, 128, 128), (150, 512, 384), (256, 1024, 2048), (40, 4096, 256)])
def test_moe_wide_deep_ring_bit_exact(cuda, monkeypatch, t, h, i):
    """The deep LDS ring of the grouped expert GEMM (6 / 5 slots) against the 3-slot ring: same
    K-tile order, so bit-identical outputs; K from 2 K-tiles (shorter than the ring) to 64."""
    from distributed_llms_amd import knobs
    monkeypatch.setattr(knobs.K, "moe_wide_min_pairs", 1)
    e, k = 8, 2
    x, wr = _bf(t, h), _bf(e, h, scale=0.1)
    wgu, wd = _bf(e, 2 * i, h, scale=0.05), _bf(e, h, i, scale=0.05)
    monkeypatch.setattr(knobs.K, "moe_deep_ring", True)
    deep = moe.forward(x, wr, wgu, wd, k)
    monkeypatch.setattr(knobs.K, "moe_deep_ring", False)
    shallow = moe.forward(x, wr, wgu, wd, k)
    assert torch.equal(deep, shallow)
    tw, tid = ref.moe_route(ref.linear(x, wr).float(), k)
    # the bf16 SwiGLU intermediate rounds at K = 4096: tolerance scaled to the output magnitude
    expect = ref.moe_mlp(x.float(), wgu.float(), wd.float(), tw, tid)
    torch.testing.assert_close(deep.float(), expect, atol=2e-2 * expect.abs().max().item(), rtol=3e-2)


@pytest.mark.parametrize("t", [1, 5, 64, 256])
@pytest.mark.parametrize("e", [8, 16])
def test_fused_router_matches_library_path(cuda, monkeypatch, t, e):
    """Fused router GEMV + top-k + scatter vs library router GEMM + route kernel: same experts and
    weights (logits rounded to bf16 in both), a consistent expert-sorted slot layout."""
    from distributed_llms_amd import _ext
    k_, h = 2, 4096
    x, wr = _bf(t, h), _bf(e, h, scale=0.05)
    kern = _ext.kernels()
    st = torch.cuda.current_stream().cuda_stream
    outs = []
    for fused in (True, False):
        tw = torch.empty(t, k_, dtype=torch.float32, device="cuda")
        tid = torch.empty(t, k_, dtype=torch.int32, device="cuda")
        cnt = torch.empty(e, dtype=torch.int32, device="cuda")
        off = torch.empty(e + 1, dtype=torch.int32, device="cuda")
        srt = torch.empty(t * k_, dtype=torch.int32, device="cuda")
        inv = torch.empty(t * k_, dtype=torch.int32, device="cuda")
        if fused:
            kern.moe_router_route(x.data_ptr(), wr.data_ptr(), t, h, e, k_, tw.data_ptr(), tid.data_ptr(),
                                  cnt.data_ptr(), off.data_ptr(), srt.data_ptr(), inv.data_ptr(), st)
        else:
            logits = ops.linear(x, wr)
            kern.moe_route(logits.data_ptr(), t, e, k_, tw.data_ptr(), tid.data_ptr(), cnt.data_ptr(),
                           off.data_ptr(), srt.data_ptr(), inv.data_ptr(), st)
        outs.append((tw, tid, cnt, off, srt, inv))
    (tw1, tid1, c1, o1, s1, i1), (tw2, tid2, c2, o2, s2, i2) = outs
    agree = (tid1 == tid2).all(dim=1)
    assert agree.float().mean() > 0.98                       # near-tie flips from accumulation order only
    # weights: one bf16 ulp of a logit (different accumulation order) moves a softmax weight ~1 %
    torch.testing.assert_close(tw1[agree], tw2[agree], atol=3e-2, rtol=3e-2)
    tok = torch.arange(t, device="cuda").repeat_interleave(k_)
    assert torch.equal(s1[i1.long()], tok.to(torch.int32))    # inv and sorted lists are consistent
    assert int(o1[-1]) == t * k_ and torch.equal(torch.diff(o1), c1)


@pytest.mark.parametrize("t,e,k,h,i,skew", [(4096, 8, 2, 1024, 2048, True), (4096, 8, 2, 1024, 2048, False),
                                            (777, 8, 2, 512, 384, True), (300, 4, 1, 256, 128, False),
                                            (4096, 8, 2, 4096, 14336, True)])
def test_moe_prefill_grouped_gemm(cuda, t, e, k, h, i, skew):
    """Prefill-sized T runs the device-side grouped GEMM (gemm_pp_moe: every expert's row tiles in
    one launch per projection, counts read on the device): skewed routing (two experts take most
    rows, the others few or none -> row tiles of many sizes, empty experts, tiles that end inside
    a segment) vs the fp32 reference on the same routing."""
    torch.manual_seed(t + h)
    x = _bf(t, h)
    if skew:
        x = x.abs() * 0.5
        wr = _bf(e, h, scale=0.002)
        wr[1] += 0.03
        wr[6] += 0.02
    else:
        wr = _bf(e, h, scale=0.1)
    wgu, wd = _bf(e, 2 * i, h, scale=0.03), _bf(e, h, i, scale=0.03)
    out = moe.forward(x, wr, wgu, wd, k)
    tw, tid = ref.moe_route(ref.linear(x, wr).float(), k)
    expect = ref.moe_mlp(x.float(), wgu.float(), wd.float(), tw, tid)
    tol = 2e-2 * expect.abs().max().item()
    torch.testing.assert_close(out.float(), expect, atol=tol, rtol=3e-2)


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [512, 2560])
@pytest.mark.parametrize("counts", [[0, 1, 128, 0, 129, 300, 384, 385], [3], [128] * 8, [0, 0, 100, 0, 90, 256, 512],
                                    [0] * 62 + [1, 2, 3, 0, 100] + [0] * 80 + [64] + [0] * 60 + [5]])
def test_moe_grouped_gemm_cuts_short_tiles(cuda, mode, n, counts):
    """Row tiles of up to 128 rows, alone and beside longer ones, in two workgroups where they leave half of the CUs idle (2560
    columns: 8 experts do not): the bits of a launch that is padded past one workgroup per CU with segments of their own."""
    from distributed_llms_amd import _ext
    k, tokens, pad = 256, 500, 256 * 9                 # the padding's tiles: 9 x 2 columns x 16 experts > 256
    w = _bf(len(counts), n, k, scale=0.1)
    glu = mode in (1, 3)

    def run(c, w, n_pad):
        c = torch.tensor(c, dtype=torch.int32, device="cuda")
        slots = int(c.sum())
        gather = torch.arange(slots, device="cuda", dtype=torch.int32).remainder_(tokens)
        y = torch.full((slots + 4, n // 2 if glu else n), 7.0, dtype=torch.bfloat16, device="cuda")
        off = torch.cumsum(c, 0).to(torch.int32) - c
        _ext.kernels().gemm_pp_moe(y.data_ptr(), x.data_ptr(), gather.data_ptr(), w.data_ptr(), c.data_ptr(), off.data_ptr(),
                                   len(c), n, k, tokens, slots, mode, torch.cuda.current_stream().cuda_stream, 0.7)
        assert bool((y[slots:] == 7.0).all())
        return y[:slots - n_pad]

    x = _bf(tokens, k)
    more = torch.cat([w, w[:1].expand(16, n, k)]).contiguous()
    assert torch.equal(run(counts, w, 0), run(counts + [pad] * 16, more, 16 * pad))


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("counts", [[257, 288, 289, 0, 512, 513, 576, 577, 256], [864, 865, 1, 769, 128],
                                    [1152, 1153, 1025, 1024], [0] * 70 + [300] + [0] * 70 + [545]])
def test_moe_grouped_gemm_tall_tiles(cuda, mode, counts):
    """Segments on either side of 1 to 4 row tiles of 288 rows: past one workgroup per CU (the padding's segments, which are on
    tiles of 256) the bits of the launch without padding, whose tiles have 256 rows."""
    from distributed_llms_amd import _ext
    k, n, tokens, pad = 320, 512, 500, 256 * 9         # the padding's tiles: 9 x 2 columns x 16 experts > 256
    x, w = _bf(tokens, k), _bf(len(counts), n, k, scale=0.1)
    more = torch.cat([w, w[:1].expand(16, n, k)]).contiguous()

    def run(c, w, n_pad):
        c = torch.tensor(c, dtype=torch.int32, device="cuda")
        slots = int(c.sum())
        gather = torch.arange(slots, device="cuda", dtype=torch.int32).remainder_(tokens)
        y = torch.full((slots + 4, n // 2 if mode in (1, 3) else n), 7.0, dtype=torch.bfloat16, device="cuda")
        off = torch.cumsum(c, 0).to(torch.int32) - c
        _ext.kernels().gemm_pp_moe(y.data_ptr(), x.data_ptr(), gather.data_ptr(), w.data_ptr(), c.data_ptr(), off.data_ptr(),
                                   len(c), n, k, tokens, slots, mode, torch.cuda.current_stream().cuda_stream, 0.7)
        assert bool((y[slots:] == 7.0).all())
        return y[:slots - n_pad]

    assert 2 * sum(-(-c // 256) for c in counts) <= 256
    assert torch.equal(run(counts, w, 0), run(counts + [pad] * 16, more, 16 * pad))


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
def test_moe_grouped_gemm_last_tiles(cuda, mode):
    """Segments whose last row tile holds 1 .. 256 rows, on either side of the 128- and 192-row tiles, with empty experts
    between, gathered and not: against each segment's own f32 product, nothing written past the segments."""
    from distributed_llms_amd import _ext
    counts = [1, 128, 0, 129, 192, 193, 255, 256, 257, 384, 0, 385, 448, 449, 513]
    e, k, n = len(counts), 192, 512
    slots, tokens = sum(counts), 700
    x = _bf(tokens, k)
    w = _bf(e, n, k, scale=0.1)
    gather = torch.randint(0, tokens, (slots,), device="cuda", dtype=torch.int32)
    c = torch.tensor(counts, dtype=torch.int32, device="cuda")
    off = torch.cumsum(c, 0).to(torch.int32) - c
    glu = mode in (1, 3)
    y = torch.full((slots + 8, n // 2 if glu else n), 7.0, dtype=torch.bfloat16, device="cuda")
    _ext.kernels().gemm_pp_moe(y.data_ptr(), x.data_ptr(), gather.data_ptr(), w.data_ptr(), c.data_ptr(), off.data_ptr(), e, n, k,
                               tokens, slots, mode, torch.cuda.current_stream().cuda_stream, 0.7)
    assert bool((y[slots:] == 7.0).all())
    at = 0
    for i, m in enumerate(counts):
        z = x[gather[at:at + m].long()].float() @ w[i].float().t()
        if mode == 2:
            z = z.clamp(min=0) ** 2
        elif glu:                       # gate and up are rounded to bf16 before the activation
            g, u = z[:, :n // 2].bfloat16().float(), z[:, n // 2:].bfloat16().float()
            if mode == 1:
                z = F.silu(g) * u
            else:
                g, u = g.clamp(max=0.7), u.clamp(-0.7, 0.7)
                z = g * torch.sigmoid(1.702 * g) * (u + 1)
        # bf16 result (and, under a GLU, a gate or up that rounds the other way: as much again, twice)
        torch.testing.assert_close(y[at:at + m].float(), z, atol=2e-2, rtol=2e-2)
        at += m


def test_moe_prefill_has_no_host_sync(cuda):
    """The prefill MoE path captures into a HIP graph (a host sync -- reading the expert counts on
    the host -- would fail the capture) and replays correctly for new inputs."""
    t, e, k, h, i = 2048, 8, 2, 512, 512
    x, wr = _bf(t, h), _bf(e, h, scale=0.1)
    wgu, wd = _bf(e, 2 * i, h, scale=0.05), _bf(e, h, i, scale=0.05)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        moe.forward(x, wr, wgu, wd, k)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = moe.forward(x, wr, wgu, wd, k)
    x.copy_(_bf(t, h))
    g.replay()
    torch.cuda.synchronize()
    tw, tid = ref.moe_route(ref.linear(x, wr).float(), k)
    expect = ref.moe_mlp(x.float(), wgu.float(), wd.float(), tw, tid)
    torch.testing.assert_close(out.float(), expect, atol=2e-2 * expect.abs().max().item(), rtol=3e-2)


def test_moe_fp8_prefill_grouped_no_host_sync(cuda):
    """W8A8 experts at prefill-sized T: one grouped fp8 launch per projection (no expert loop, no
    counts read on the host -- graph-capturable), against the fp8 reference numerics."""
    from distributed_llms_amd.ops import quant
    t, e, k, h, i = 1024, 8, 2, 512, 512
    torch.manual_seed(3)
    x, wr = _bf(t, h), _bf(e, h, scale=0.1)
    wgu, wd = quant.quantize_experts(_bf(e, 2 * i, h, scale=0.05)), quant.quantize_experts(_bf(e, h, i, scale=0.05))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        moe.forward(x, wr, wgu, wd, k)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = moe.forward(x, wr, wgu, wd, k)
    g.replay()
    torch.cuda.synchronize()
    tw, tid = ref.moe_route(ref.linear(x, wr).float(), k)
    expect = quant.moe_mlp_ref(x, wgu, wd, tw, tid)
    torch.testing.assert_close(out.float(), expect.float(), atol=3e-2 * expect.abs().max().item(), rtol=5e-2)


@pytest.mark.parametrize("t", [1, 2, 7, 64, 129, 200])
@pytest.mark.parametrize("n,k,s", [(4096, 4096, 8), (4096, 4096, 4), (2048, 2048, 4), (2048, 4096, 8)])
@pytest.mark.parametrize("top", [1, 2, 8])
def test_norm_and_choice_in_one_launch(cuda, t, n, k, s, top):
    """The add + norm of a split product's slabs with the choice of experts behind it: the bits of the two launches."""
    from distributed_llms_amd import _ext
    from distributed_llms_amd.ops import gemm
    x, w, wr = _bf(t, k), _bf(n, k, scale=k ** -0.5), _bf(8, n, scale=n ** -0.5)
    res, nw = _bf(t, n), _bf(n)
    r0, r1 = res.clone(), res.clone()
    part = gemm.linear_wide(x, w, splits=s, defer=True)
    assert part.splits == s
    y0, _ = ops.fused_add_rms_norm(part, r0, nw, 1e-5)
    got = moe.norm_route(part, r1, nw, 1e-5, wr, top)
    assert got is not None
    y1, _, (tw, ids) = got
    tw0, ids0 = torch.empty_like(tw), torch.empty_like(ids)
    i32 = lambda c: torch.empty(c, dtype=torch.int32, device="cuda")     # noqa: E731
    c0, o0, s0, v0, c1, o1, s1, v1 = (i32(m) for m in (8, 9, t * top, t * top) * 2)
    st = torch.cuda.current_stream().cuda_stream
    _ext.kernels().moe_router_route(y0.data_ptr(), wr.data_ptr(), t, n, 8, top, tw0.data_ptr(), ids0.data_ptr(), c0.data_ptr(), o0.data_ptr(),
                                    s0.data_ptr(), v0.data_ptr(), st)
    _ext.kernels().moe_scatter(ids.data_ptr(), t, 8, top, c1.data_ptr(), o1.data_ptr(), s1.data_ptr(), v1.data_ptr(), st)
    for a, b in ((y0, y1), (r0, r1), (ids0, ids), (tw0, tw), (c0, c1), (o0, o1)):
        assert torch.equal(a, b)
    assert torch.equal(s1[v1.long()], torch.arange(t * top, device="cuda", dtype=torch.int32) // top)
    want = (y0.double() @ wr.double().T).bfloat16().double().softmax(-1).topk(top, -1).values
    assert (tw.double() - want / want.sum(-1, keepdim=True)).abs().max() <= 2.0 ** -6       # (logits of up to 4 with an ulp of 2^-6)


@pytest.mark.parametrize("t", [1, 3, 64, 300])
@pytest.mark.parametrize("h", [8, 2048, 2056, 4096, 8200, 16384])
@pytest.mark.parametrize("top", [1, 2, 3, 8])
def test_combine_and_norm_in_one_launch(cuda, t, h, top):
    """The weighted sum of the experts' rows in the launch of the add + norm behind it: the bits of the two."""
    ys, inv = _bf(t * top, h), torch.randperm(t * top, device="cuda").to(torch.int32)
    tw = torch.rand(t, top, device="cuda")
    res, nw, like = _bf(t + 1, h), _bf(h), torch.empty(t, h, device="cuda", dtype=torch.bfloat16)
    c = moe.Combine(ys, tw, inv, top, like)
    r0, r1 = res.clone(), res.clone()
    y0, _ = ops.fused_add_rms_norm(c.materialize(), r0[:t], nw, 1e-5)
    y1, _ = ops.fused_add_rms_norm(c, r1[:t], nw, 1e-5)
    assert torch.equal(y0, y1) and torch.equal(r0, r1)


def test_norm_and_choice_refuse(cuda):
    """Other slabs, widths and experts keep their launches."""
    from distributed_llms_amd.ops import gemm
    nw, res = _bf(4096), _bf(2, 4096)
    part = gemm.linear_wide(_bf(2, 4096), _bf(4096, 4096), splits=2, defer=True)
    assert moe.norm_route(part, res, nw, 1e-5, _bf(8, 4096), 2) is None
    part = gemm.linear_wide(_bf(2, 4096), _bf(4096, 4096), splits=8, defer=True)
    assert moe.norm_route(part, res, nw, 1e-5, _bf(16, 4096), 2) is None
    assert moe.norm_route(part.materialize(), res, nw, 1e-5, _bf(8, 4096), 2) is None
    assert moe.norm_route(part, res, nw, 1e-5, _bf(8, 4096).T.contiguous().T, 2) is None


@pytest.mark.parametrize("t,top", [(1, 1), (1, 2), (3, 2), (4, 2), (7, 8), (8, 8), (21, 3), (32, 2), (64, 1)])
@pytest.mark.parametrize("skew", [False, True])
@pytest.mark.parametrize("first,local", [(0, 8), (2, 4)])
def test_experts_find_few_rows_themselves(cuda, t, top, skew, first, local):
    """Up to 64 pairs of a choice that is there: the bits of the launches behind counts and slot lists (all experts, or a range of them)."""
    h, i = 256, 256
    x, gu, dn = _bf(t, h), _bf(8, 2 * i, h, scale=0.05), _bf(8, h, i, scale=0.05)
    wr = _bf(8, h, scale=0.1)
    ids = torch.stack([torch.randperm(8, device="cuda")[:top] for _ in range(t)]).to(torch.int32)
    if skew:
        ids[:] = torch.arange(8, device="cuda", dtype=torch.int32).flip(0)[:top]
    tw = torch.rand(t, top, device="cuda")
    gu, dn = gu[first:first + local].contiguous(), dn[first:first + local].contiguous()
    res, nw = _bf(t, h), _bf(h)
    out = moe.forward(x, wr, gu, dn, top, first, choice=(tw, ids))
    part = moe.forward(x, wr, gu, dn, top, first, choice=(tw, ids), defer=True)
    assert part.inv is None
    pairs, moe.PICK_PAIRS = moe.PICK_PAIRS, 0
    try:
        want = moe.forward(x, wr, gu, dn, top, first, choice=(tw, ids))
    finally:
        moe.PICK_PAIRS = pairs
    if t * top > 2:
        assert torch.equal(out, want)
    r0, r1 = res.clone(), res.clone()
    assert torch.equal(ops.fused_add_rms_norm(part, r0, nw, 1e-5)[0], ops.fused_add_rms_norm(out, r1, nw, 1e-5)[0]) and torch.equal(r0, r1)
    local_ids = ids - first
    mine = (local_ids >= 0) & (local_ids < local)
    ref_out = ref.moe_mlp(x.float(), gu.float(), dn.float(), tw * mine, local_ids.clamp(0, local - 1))
    torch.testing.assert_close(out.float(), ref_out, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("t,top", [(1, 1), (1, 2), (2, 2), (3, 2)])
def test_few_pairs_of_large_experts(cuda, t, top):
    """Fewer pairs than the tiled kernel's line, on it where its workgroups fill the CUs; the down projection of one or two in narrow tiles. """
    h, i = 256, 16384
    x, gu, dn = _bf(t, h), _bf(8, 2 * i, h, scale=h ** -0.5), _bf(8, h, i, scale=i ** -0.5)
    ids = torch.stack([torch.randperm(8, device="cuda")[:top] for _ in range(t)]).to(torch.int32)
    tw = torch.rand(t, top, device="cuda")
    out = moe.forward(x, _bf(8, h), gu, dn, top, choice=(tw, ids))
    want = torch.zeros(t, h, device="cuda", dtype=torch.float64)
    for a in range(t):
        for j in range(top):
            z = gu[ids[a, j].item()].double() @ x[a].double()
            want[a] += tw[a, j].double() * (dn[ids[a, j].item()].double() @ (F.silu(z[:i]) * z[i:]))
    # 2^-9 for each of the activation, the expert's row and the result, rounded to bf16
    assert (out.double() - want).norm() <= 3 * 2.0 ** -9 * want.norm()
