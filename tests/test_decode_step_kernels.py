"""One-launch decode steps of the layer-list models against the same steps done by the general kernels' CPU reference."""
import numpy as np
import pytest
import torch

from distributed_llms_amd import ops
from distributed_llms_amd.ops import gemm
from distributed_llms_amd.ops import reference as ref
from distributed_llms_amd.ops import seqmix as sm

gpu = pytest.mark.gpu


def _sb(pos, slots, device):
    n = len(pos)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=device)
    return sm.SeqBatch(i32(list(range(n + 1))), i32(pos), i32(list(range(n))), i32(slots), n, n, 1)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("nb,bw,taps", [(1, 8, 1), (3, 40, 2), (4, 256, 4), (2, 264, 8), (10, 256, 4), (1, 512, 3)])
@pytest.mark.parametrize("seqs", [1, 5, 40, 141])
def test_rglru_step(cuda, dtype, nb, bw, taps, seqs):
    """One and two sequences per workgroup (an odd last one), blocks narrower and wider than 64 outputs and 256 rows,
    sequences at positions 0, 1, 2 and later (parts of the tail do not exist yet), slots out of order."""
    g = torch.Generator().manual_seed(seqs + bw)
    c = nb * bw
    r = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(dtype)
    yx, cw, cb, xb, yb = r(seqs, 2 * c), r(taps, c, scale=0.5), r(c, scale=0.1), r(c, scale=0.1), r(c, scale=0.1)
    ra, ri = r(nb, bw, bw, scale=bw ** -0.5), r(nb, bw, bw, scale=bw ** -0.5)
    rab, rib, lam = r(nb, bw, scale=0.3), r(nb, bw, scale=0.3), r(c)
    slots = (torch.randperm(seqs + 3, generator=g)[:seqs]).tolist()
    pos = [[0, 1, 2, 3, 57][i % 5] for i in range(seqs)]
    conv, state = r(seqs + 3, taps - 1, c), torch.randn(seqs + 3, c, generator=g)
    conv_d, state_d = conv.cuda(), state.cuda()
    d = lambda t: t.cuda()
    conv_2, state_2 = conv_d.clone(), state_d.clone()            # a second launch finds the counters as the first did
    again = sm.rglru_step(d(yx), d(cw), d(cb), d(xb), conv_2, d(yb), d(ra), d(rab), d(ri), d(rib), d(lam), state_2,
                          _sb(pos, slots, "cuda"))
    out = sm.rglru_step(d(yx), d(cw), d(cb), d(xb), conv_d, d(yb), d(ra), d(rab), d(ri), d(rib), d(lam), state_d,
                        _sb(pos, slots, "cuda"))
    ref = sm.rglru_step(yx, cw, cb, xb, conv, yb, ra, rab, ri, rib, lam, state, _sb(pos, slots, "cpu"))
    assert torch.equal(conv_d, conv_2) and torch.equal(state_d, state_2) and torch.equal(out, again)
    assert torch.equal(conv_d.cpu(), conv)                       # the tail is moved, not computed
    # float32 sums of bw products in another order: the gates' arguments within bw 2^-24 of their terms (|u| |w| sum to
    # a few units), times decay_scale softplus(lam) <= 30 through the exponential; sqrt(1 - a^2) steepens that near a = 1
    np.testing.assert_allclose(state_d.cpu().numpy(), state.numpy(), atol=2e-4, rtol=2e-4)
    tol = dict(atol=4e-4, rtol=4e-4) if dtype == torch.float32 else dict(atol=2e-3, rtol=2.0 ** -7)
    np.testing.assert_allclose(out.float().cpu().numpy(), ref.float().numpy(), **tol)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps,dim,vdim", [(2, 32, 48), (3, 128, 128), (4, 10, 6), (5, 16, 16)])
def test_attention_input_moves_the_tail(cuda, dtype, taps, dim, vdim):
    """One token per sequence: q, caches and the convolution's new tail as the general form leaves them (taps 5: past the
    one-launch form)."""
    g = torch.Generator().manual_seed(taps)
    heads, kvh, bs, pos = 6, 2, 16, [0, 1, 2, 3, 40]
    c, n = heads * dim + kvh * (dim + vdim), 5
    r = lambda *s: torch.randn(*s, generator=g).to(dtype)
    qkv, cw, conv, qn, kn = r(n, c), r(taps, c), r(9, taps - 1, c), r(dim), r(dim)
    freqs, slot_map = torch.rand(dim // 4, generator=g), torch.tensor([3, 17, 40, 5, 66], dtype=torch.int32)
    got = []
    for dev in ("cpu", "cuda"):
        kc, vc = torch.zeros(5, kvh, bs, dim, dtype=dtype, device=dev), torch.zeros(5, kvh, vdim, bs, dtype=dtype, device=dev)
        st = conv.to(dev, copy=True)
        q = sm.attn_prep(qkv.to(dev), cw.to(dev), st, qn.to(dev), kn.to(dev), freqs.to(dev), 1.1, 1e-6, kc, vc, slot_map.to(dev),
                         _sb(pos, [4, 2, 8, 1, 6], dev), heads, kvh, dim, vdim)
        got.append([t.float().cpu() for t in (q, kc, vc)] + [st.cpu()])
    tol = dict(atol=1e-4, rtol=1e-4) if dtype == torch.float32 else dict(atol=1e-2, rtol=2.0 ** -7)
    for a, b in zip(*[x[:3] for x in got]):
        torch.testing.assert_close(b, a, **tol)
    assert torch.equal(got[0][3], got[1][3])


@gpu
@pytest.mark.parametrize("warm", [True, False])
def test_rglru_step_graph_outlives_its_counters_successor(cuda, warm):
    """A graph captured with few sequences still has its arrival counters after a larger batch on the same stream needed
    more of them, whatever was allocated since; so has one captured on a stream that had none yet."""
    nb, bw, taps, c = 10, 8, 4, 80
    r = lambda *s: torch.randn(*s, device=cuda).bfloat16()
    ops_ = [r(taps, c), r(c), r(c)], [r(c), r(nb, bw, bw), r(nb, bw), r(nb, bw, bw), r(nb, bw), r(c)]
    state0, conv0, yx = torch.randn(301, c, device=cuda), r(301, taps - 1, c), r(300, 2 * c)
    run = lambda n, conv, state, sb: sm.rglru_step(yx[:n], *ops_[0], conv, *ops_[1], state, sb)
    few, many = _sb([5, 9, 7], [1, 2, 3], cuda), _sb([5] * 300, list(range(1, 301)), cuda)
    conv, state = conv0.clone(), state0.clone()
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        if warm:
            want = run(3, conv, state, few), conv.clone(), state.clone()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = run(3, conv, state, few)
        run(300, conv0.clone(), state0.clone(), many)            # 300 x 10 counters: more than the first buffer holds
        s.synchronize()
        if not warm:
            want = run(3, conv, state, few), conv.clone(), state.clone()
        taken = [torch.full((1 << 16,), 7, dtype=torch.int32, device=cuda) for _ in range(8)]
        for _ in range(3):
            conv.copy_(conv0)
            state.copy_(state0)
            g.replay()
            s.synchronize()
            for a, b in zip((out, conv, state), want):
                assert torch.equal(a, b)
    del taken


@gpu
@pytest.mark.parametrize("bw", [64, 200])
def test_rglru_step_counts_by_slot(cuda, bw):
    """Two graphs captured on one stream, of other slots of one pool, replayed side by side on two others, next to eager
    launches on the stream of their capture: each slot's count is its own.  Rows that share the scratch slot (padding) and
    odd last rows of a pair leave every count zero."""
    nb, taps, c, slots = 3, 4, 3 * bw, 120
    r = lambda *s: torch.randn(*s, device=cuda).bfloat16()
    par = [r(taps, c), r(c), r(c)], [r(c), r(nb, bw, bw) * 0.1, r(nb, bw), r(nb, bw, bw) * 0.1, r(nb, bw), r(c)]
    yx, conv0, state0 = r(41, 2 * c), r(slots, taps - 1, c), torch.randn(slots, c, device=cuda)
    arrived = sm.step_counters(slots, nb, cuda)
    parts = [list(range(1, 38)) + [0] * 4, list(range(40, 81)), [100, 101, 0, 0, 0]]
    sbs = [_sb([7] * len(p), p, cuda) for p in parts]

    def run(i, conv, state, counts):
        return sm.rglru_step(yx[:len(parts[i])], *par[0], conv, *par[1], state, sbs[i], arrived=counts)
    want_c, want_s, want = conv0.clone(), state0.clone(), []
    for i in range(3):
        want.append(run(i, want_c, want_s, None))
    conv, state = conv0.clone(), state0.clone()
    torch.cuda.synchronize()
    s, a, b = (torch.cuda.Stream() for _ in range(3))
    graphs, outs = [], []
    for i in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            outs.append(run(i, conv, state, arrived))
        graphs.append(g)
    for _ in range(4):
        conv.copy_(conv0)
        state.copy_(state0)
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            graphs[0].replay()
        with torch.cuda.stream(b):
            graphs[1].replay()
        with torch.cuda.stream(s):
            eager = run(2, conv, state, arrived)
        torch.cuda.synchronize()
        live = [37, 41, 2]
        for got, ref, n in zip(outs + [eager], want, live):
            assert torch.equal(got[:n], ref[:n])
        assert torch.equal(conv[1:], want_c[1:]) and torch.equal(state[1:], want_s[1:])
        assert not arrived.any()


def test_rglru_step_keeps_no_process_wide_state():
    """What the step counts in belongs to the caller's state pool: nothing is kept by stream or device."""
    assert not [k for k, v in vars(sm).items() if isinstance(v, (dict, list, set)) and not k.startswith("__")]


@gpu
@pytest.mark.parametrize("width", [1, 2047, 2056, 256 * 65535 + 3])
def test_embedding_f32_of_any_width(cuda, width):
    """Vector and scalar pieces, a partial last workgroup, and a row of more pieces than a grid has workgroups."""
    table = torch.arange(2 * width, device=cuda).view(2, width).remainder(251).bfloat16()
    ids = torch.tensor([1, 0, 5, -1], dtype=torch.int32, device=cuda)
    out = sm.embedding_f32(ids, table, 3.0)
    assert torch.equal(out, table[[1, 0, 1, 0]].float() * 3.0)


@gpu
@pytest.mark.parametrize("rows", [1, 7, 300])
@pytest.mark.parametrize("width", [4, 250, 1024, 2560, 4100, 16384, 16392])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["next", "bias", "two", "plain"])
def test_post_norm_add_rows(cuda, rows, width, dtype, form):
    """The register-resident close of a sublayer at partial last pieces, odd widths and past its largest row."""
    if rows == 300 and width > 4100:
        return
    g = torch.Generator().manual_seed(width)
    r = lambda *s: torch.randn(*s, generator=g)
    x, o, o2, b, wp, wn = r(rows, width), r(rows, width).to(dtype), r(rows, width).to(dtype), r(width).to(dtype), r(width).to(dtype), r(width).to(dtype)
    kw = {"next": dict(w_next=wn), "bias": dict(bias=b, w_next=wn), "two": dict(o2=o2, scales=(0.9, 0.7), one_plus=False, w_next=wn),
          "plain": dict(plain_next=True)}[form]
    d = lambda v: v.cuda() if isinstance(v, torch.Tensor) else v
    xr, hr = sm.post_norm_add(x.clone(), o, wp, 1e-6, 0.8, **kw)
    xg, hg = sm.post_norm_add(x.cuda(), o.cuda(), wp.cuda(), 1e-6, 0.8, **{k: d(v) for k, v in kw.items()})
    torch.testing.assert_close(xg.cpu(), xr, atol=2e-5, rtol=2e-5)
    tol = dict(atol=5e-5, rtol=5e-5) if dtype == torch.float32 else dict(atol=1e-3, rtol=2.0 ** -7)
    torch.testing.assert_close(hg.float().cpu(), hr.float(), **tol)


@gpu
def test_post_norm_add_refuses_other_types(cuda):
    x, o, w = torch.zeros(3, 64, device=cuda), torch.zeros(3, 64, device=cuda).half(), torch.zeros(64, device=cuda).half()
    with pytest.raises(TypeError):
        sm.post_norm_add(x, o, w, 1e-6, 1.0)


@gpu
@pytest.mark.parametrize("tokens,width,k", [(1, 256, 1024), (16, 2560, 7680), (40, 4096, 2048)])
def test_post_norm_add_sums_split_products(cuda, tokens, width, k):
    """On a split-K product that is not reduced yet, against the same on the reduced one: the slabs are summed in the same
    order and rounded to bf16 before the norm, so both see the same numbers."""
    a = torch.randn(tokens, k, device="cuda").bfloat16()
    w = (torch.randn(width, k, device="cuda") * k ** -0.5).bfloat16()
    wp, wn, b = (torch.randn(width, device="cuda").bfloat16() for _ in range(3))
    part = gemm.linear_wide(a, w, defer=True)
    assert isinstance(part, gemm.SplitKPartial)
    whole = part.materialize()
    x0 = torch.randn(tokens, width, device="cuda")
    got = sm.post_norm_add(x0.clone(), part, wp, 1e-5, 0.7, bias=b, w_next=wn)
    want = sm.post_norm_add(x0.clone(), whole, wp, 1e-5, 0.7, bias=b, w_next=wn)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@gpu
@pytest.mark.parametrize("n,slabs", [(4096, 5), (6144, 5), (8192, 3), (8192, 5), (8192, 8), (16384, 2), (16384, 3), (16384, 5), (16384, 7)])
def test_add_rms_norm_sums_slabs_inside_its_rows(cuda, n, slabs):
    """Every split of a row's vectors into chunks of loads: the sum of the slabs as the plain reduction makes it, and nothing
    written past the rows (5 slabs of 8192 were taken in chunks of three vectors of four)."""
    g = torch.Generator("cuda").manual_seed(n + slabs)
    ws = torch.randn(slabs * 2 * n, generator=g, device="cuda").half().view(torch.float32)
    part = gemm.SplitKPartial(ws, slabs, 2, n, (2, n), torch.bfloat16, ws.device)
    room = torch.randn(4, n, generator=g, device="cuda").bfloat16()
    w, before = torch.randn(n, generator=g, device="cuda").bfloat16(), room.clone()
    want, r = ops.fused_add_rms_norm(part.materialize(), room[:2].clone(), w, 1e-5)
    y, res = ops.fused_add_rms_norm(part, room[:2], w, 1e-5)
    assert torch.equal(y, want) and torch.equal(res, r) and torch.equal(room[2:], before[2:])


@gpu
@pytest.mark.parametrize("lens,width,splits", [
    ([1, 33, 64], 2, 1),                   # one chunk, and the new key alone in its chunk
    ([65, 64, 1], 4, 2), ([97, 200, 250], 8, 4), ([449, 1], 16, 8), ([1000], 32, 16), ([1025, 3], 33, 17),
    ([2048], 5120, 1), ([2400, 2049], 5120, 1)])   # splits of 2560 keys: past the 64 chunks of one pass over block ids
@pytest.mark.parametrize("d,slabs", [(128, 0), (128, 4), (128, 7), (64, 0)])
def test_decode_attention_rounds_and_passes(cuda, lens, width, splits, d, slabs):
    """Decode attention at the edges of its split rounds, chunk pairs and block id passes, against float32."""
    torch.manual_seed(5)
    b, hq, hkv, used = len(lens), 4, 1, sum(-(-n // 32) for n in lens)
    k = torch.randn(used, hkv, 32, d).bfloat16().cuda()
    v = torch.randn(used, hkv, d, 32).bfloat16().cuda()
    assert ops.decode_split_plan(b, hkv, max(lens), 32, width)[0] == splits
    bt = torch.zeros(b, width, dtype=torch.int32)
    at = 0
    for i, n in enumerate(lens):
        nb = -(-n // 32)
        bt[i, :nb] = torch.arange(at, at + nb)
        at += nb
    slots = torch.tensor([int(bt[i, (n - 1) // 32]) * 32 + (n - 1) % 32 for i, n in enumerate(lens)], dtype=torch.int32)
    bt, slots = bt.cuda(), slots.cuda()
    sl = torch.tensor(lens, dtype=torch.int32).cuda()
    n = (hq + 2 * hkv) * d
    qkv = torch.randn(b, n).bfloat16().cuda()
    arg = qkv
    if slabs:                               # whole numbers of 2^-6: exact in a slab's 16 bits and in any order of the sum
        parts = torch.randint(-64, 65, (slabs, b, n)).float() / 64
        qkv = parts.sum(0).bfloat16().cuda()
        arg = gemm.SplitKPartial((parts / 64).half().cuda(), slabs, b, n, (b, n), torch.bfloat16, qkv.device)
    cs = ref.rope_cos_sin(d, 4096, 500000.0, device="cuda")
    kf, vf = k.float(), v.float()
    q2 = ref.rope_cache_append(qkv.float(), sl - 1, cs, kf, vf, slots, hq, hkv, d)
    expect = ref.paged_attention_decode(q2.bfloat16().float(), kf.bfloat16().float(), vf, bt, sl, d ** -0.5)
    torch.cuda.synchronize()
    out = ops.paged_attention_decode_rope(arg, sl - 1, cs, k, v, slots, bt, sl, hq, hkv, d, d ** -0.5, max_ctx=max(lens))
    # probabilities and the result are rounded to bf16 (2^-9 each, of at most max |v|); as much again for a rotated
    # element that rounds the other way
    assert (out.float() - expect).abs().max() <= 2.0 ** -7 * vf.abs().max()
    assert torch.equal(v.float(), vf)


@gpu
@pytest.mark.parametrize("fused", [False, True])
def test_decode_attention_without_block_ids(cuda, fused):
    """A block table of no columns (every context empty): zeros, and nothing is read through it."""
    b, hq, hkv, d = 3, 4, 2, 128
    k, v = torch.randn(2, hkv, 32, d).bfloat16().cuda(), torch.randn(2, hkv, d, 32).bfloat16().cuda()
    bt, none = torch.zeros(b, 0, dtype=torch.int32, device=cuda), torch.zeros(b, dtype=torch.int32, device=cuda)
    if fused:
        qkv, cs = torch.randn(b, (hq + 2 * hkv) * d).bfloat16().cuda(), ref.rope_cos_sin(d, 64, 10000.0, device=cuda)
        torch.cuda.synchronize()
        out = ops.paged_attention_decode_rope(qkv, none, cs, k, v, none, bt, none, hq, hkv, d, d ** -0.5)
    else:
        out = ops.paged_attention_decode(torch.randn(b, hq, d).bfloat16().cuda(), k, v, bt, none, d ** -0.5)
    assert torch.equal(out, torch.zeros_like(out))


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [4097, 8191, 8193, 8200, 12288, 12292, 16383])
def test_norm_rows_past_4096(cuda, width, dtype):
    """The closes of a sublayer and the layer norm on rows whose stream and weights come in rounds: partial last pieces of
    the 12- and 16-piece forms, and odd widths."""
    g = torch.Generator().manual_seed(width)
    r = lambda *s: torch.randn(*s, generator=g)
    x, o, b, wp, bp, wn, bn = (r(3, width), r(3, width).to(dtype)) + tuple(r(width).to(dtype) for _ in range(5))
    c = lambda *t: [v.cuda() for v in t]
    tol = dict(atol=5e-5, rtol=5e-5) if dtype == torch.float32 else dict(atol=1e-3, rtol=2.0 ** -7)
    co, cb, cwp, cbp, cwn, cbn = c(o, b, wp, bp, wn, bn)
    for gpu_, cpu in ((sm.post_norm_add(x.cuda(), co, cwp, 1e-6, 0.8, bias=cb, w_next=cwn),
                       sm.post_norm_add(x.clone(), o, wp, 1e-6, 0.8, bias=b, w_next=wn)),
                      (sm.post_layer_norm_add(x.cuda(), co, cwp, cbp, 1e-6, bias=cb, w_next=cwn, b_next=cbn),
                       sm.post_layer_norm_add(x.clone(), o, wp, bp, 1e-6, bias=b, w_next=wn, b_next=bn))):
        torch.testing.assert_close(gpu_[0].cpu(), cpu[0], atol=5e-5, rtol=5e-5)
        torch.testing.assert_close(gpu_[1].float().cpu(), cpu[1].float(), **tol)
    torch.testing.assert_close(sm.layer_norm_f32(x.cuda(), cwp, cbp, 1e-6, dtype).float().cpu(),
                               sm.layer_norm_f32(x, wp, bp, 1e-6, dtype).float(), **tol)


@gpu
@pytest.mark.parametrize("n", [8192, 16384])
def test_wide_closes_sum_split_products(cuda, n):
    x, w = torch.randn(3, 1024, device=cuda).bfloat16(), (torch.randn(n, 1024, device=cuda) * 0.03).bfloat16()
    s, v = torch.randn(3, n, device=cuda), [torch.randn(n, device=cuda).bfloat16() for _ in range(4)]
    for close in (lambda t, o: sm.post_norm_add(t, o, v[0], 1e-6, 0.8, w_next=v[1]),
                  lambda t, o: sm.post_layer_norm_add(t, o, v[0], v[1], 1e-6, w_next=v[2], b_next=v[3])):
        part = gemm.linear_wide(x, w, splits=2, defer=True)
        assert isinstance(part, gemm.SplitKPartial)
        got = close(s.clone(), part)
        want = close(s.clone(), gemm.linear_wide(x, w, splits=2))
        torch.testing.assert_close(got[0], want[0], atol=1e-5, rtol=1e-5)
        torch.testing.assert_close(got[1].float(), want[1].float(), atol=1e-3, rtol=2.0 ** -7)


@gpu
@pytest.mark.parametrize("rows,heads", [(1, 3), (18, 16)])
@pytest.mark.parametrize("n_in,n_out", [(7, 32), (16, 32), (24, 128), (50, 128), (61, 512), (64, 512), (96, 384), (130, 512), (256, 64)])
def test_latent_products_by_rows_in_flight(cuda, rows, heads, n_in, n_out):
    """One, two, four and 16 weight rows in flight per thread, whole and partial rounds; grids of up to 256 workgroups and
    more (the 16-row form is the small grids')."""
    from distributed_llms_amd.ops import latent as lat
    q, uk = torch.randn(rows, heads * n_in, device=cuda).bfloat16(), torch.randn(heads, n_in, n_out, device=cuda).bfloat16()
    spec = lat.LatentSpec(heads=heads, dim=n_in, vdim=n_out, rank=n_out, q_rank=0, scale=1.0)
    pos = torch.arange(rows, dtype=torch.int32, device=cuda)
    q3 = q.view(rows, heads, n_in).double().transpose(0, 1)
    want, mag = (torch.matmul(a, b).transpose(0, 1) for a, b in ((q3, uk.double()), (q3.abs(), uk.double().abs())))
    for got in (lat.latent_queries(q, uk, spec, None, pos), lat.latent_values(q.view(rows, heads, n_in), uk).view(rows, heads, n_out)):
        assert ((got.double() - want).abs() <= n_in * 2.0 ** -24 * mag + 2.0 ** -8 * want.abs()).all()


@gpu
@pytest.mark.parametrize("d,dv", [(8, 8), (32, 32), (40, 24), (64, 64), (72, 96), (96, 96), (104, 128), (136, 128), (192, 128),
                                  (168, 136), (192, 192), (200, 192), (256, 256)])
@pytest.mark.parametrize("biased", [False, True])
def test_window_decode_head_sizes(cuda, d, dv, biased):
    """Every head size that has a kernel of its own, at its edges: contexts within a tile, past one and past a wave's share."""
    lens, h, g, bs, size = [1, 31, 33, 100, 700], 6, 2, 16, 300
    nb = (max(lens) + bs - 1) // bs
    b = len(lens)
    kc, vc = torch.randn(b * nb + 1, g, bs, d, device=cuda).bfloat16(), torch.randn(b * nb + 1, g, dv, bs, device=cuda).bfloat16()
    bt = (torch.randperm(b * nb, device=cuda) + 1).int().view(b, nb)
    q, bias = torch.randn(b, h, d, device=cuda).bfloat16(), torch.randn(h, 50, device=cuda) if biased else None
    out = sm.window_attention(q, kc, vc, bt, _sb([n - 1 for n in lens], list(range(b)), cuda), size, d ** -0.5, bias=bias)
    for i, n in enumerate(lens):
        at = torch.arange(max(0, n - size), n, device=cuda)
        blk = bt[i].long()[at // bs]
        k = kc[blk, :, at % bs].double().repeat_interleave(h // g, 1)                # [keys, h, d]
        v = vc[blk, :, :, at % bs].double().repeat_interleave(h // g, 1)
        s = (q[i].double() * k).sum(-1) * d ** -0.5
        if biased:
            s = s + bias.double()[:, (n - 1 - at).clamp_max(49)].t()
        want = (torch.softmax(s, 0)[..., None] * v).sum(0)
        # scores: d exact products, 2^-24 of their magnitudes (below 2^-15 in all); weights kept to 17 bits; the result in 8
        assert ((out[i].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * v.abs().max()).all()


@gpu
@pytest.mark.parametrize("sunk,gated", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("h,g,d,dv", [(3, 3, 64, 40), (6, 2, 128, 128), (34, 2, 72, 96), (16, 1, 256, 192)])
def test_window_decode_sinks_and_gates(cuda, h, g, d, dv, sunk, gated):
    """The end of a row: sinks and gates apart and together, 1 to 16 heads a workgroup and a group in two of them (17), channels that
    are no multiple of 16, waves without a tile, keys whole and (long contexts of few rows) in runs."""
    lens, bs = [1, 40, 129, 900], 32
    b, nb = len(lens), -(-max(lens) // 32)
    kc, vc = torch.randn(b * nb + 1, g, bs, d, device=cuda).bfloat16(), torch.randn(b * nb + 1, g, dv, bs, device=cuda).bfloat16()
    bt = (torch.randperm(b * nb, device=cuda) + 1).int().view(b, nb)
    q = torch.randn(b, h, d, device=cuda).bfloat16()
    sinks = torch.randn(h, device=cuda) if sunk else None
    gate = torch.randn(b, h + 3, device=cuda).bfloat16() if gated else None
    sb = _sb([n - 1 for n in lens], list(range(b)), cuda)
    for max_ctx in (None, max(lens)):
        out = sm.window_attention(q, kc, vc, bt, sb, 1 << 30, d ** -0.5, sinks=sinks, gate=gate, gate_col=2 if gated else 0, max_ctx=max_ctx)
        for i, n in enumerate(lens):
            at = torch.arange(n, device=cuda)
            blk = bt[i].long()[at // bs]
            k = kc[blk, :, at % bs].double().repeat_interleave(h // g, 1)
            v = vc[blk, :, :, at % bs].double().repeat_interleave(h // g, 1)
            s = (q[i].double() * k).sum(-1) * d ** -0.5
            w = torch.softmax(torch.cat([s, sinks.double()[None]]) if sunk else s, 0)[:n]
            want = (w[..., None] * v).sum(0)
            if gated:
                want = want * torch.sigmoid(gate[i, 2:2 + h].double())[:, None]
            # as above: scores within 2^-15, weights to 17 bits, the result in 8
            assert ((out[i].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * v.abs().max()).all()


@gpu
@pytest.mark.parametrize("b,hq,hkv,d,ctx", [(2, 4, 1, 128, 128), (3, 16, 1, 128, 100), (5, 2, 2, 64, 250), (64, 16, 4, 128, 129),
                                            (70, 32, 4, 64, 200), (16, 32, 2, 64, 256), (1, 1, 1, 64, 65)])
@pytest.mark.parametrize("fused", [False, True])
def test_decode_attention_joins_splits_in_a_workgroup(cuda, b, hq, hkv, d, ctx, fused):
    """2 to 4 splits summed in one workgroup: groups of 1 to 16 heads, sequences that leave the last splits (or all but the
    first) empty, an even and an uneven share of workgroups per CU; against float32."""
    torch.manual_seed(b + ctx)
    lens = [max(1, ctx - 37 * (i % 7)) if i else ctx for i in range(b)]
    width = 1 << (-(-ctx // 32) - 1).bit_length()
    splits, split_len = ops.decode_split_plan(b, hkv, ctx, 32, width)
    surplus = splits * -(-b * hkv // 256) - -(-splits * b * hkv // 256)
    assert 2 <= splits <= 4 and surplus * split_len * d < 14000           # the launcher's rule
    used = sum(-(-n // 32) for n in lens)
    k = torch.randn(used, hkv, 32, d).bfloat16().cuda()
    v = torch.randn(used, hkv, d, 32).bfloat16().cuda()
    bt, at = torch.zeros(b, width, dtype=torch.int32), 0
    for i, n in enumerate(lens):
        bt[i, :-(-n // 32)] = torch.arange(at, at + -(-n // 32))
        at += -(-n // 32)
    slots = torch.tensor([int(bt[i, (n - 1) // 32]) * 32 + (n - 1) % 32 for i, n in enumerate(lens)], dtype=torch.int32).cuda()
    bt, sl = bt.cuda(), torch.tensor(lens, dtype=torch.int32).cuda()
    kf, vf = k.float(), v.float()
    if fused:
        qkv = torch.randn(b, (hq + 2 * hkv) * d).bfloat16().cuda()
        cs = ref.rope_cos_sin(d, 4096, 500000.0, device="cuda")
        q = ref.rope_cache_append(qkv.float(), sl - 1, cs, kf, vf, slots, hq, hkv, d).bfloat16()
        out = ops.paged_attention_decode_rope(qkv, sl - 1, cs, k, v, slots, bt, sl, hq, hkv, d, d ** -0.5, max_ctx=ctx)
    else:
        q = torch.randn(b, hq, d).bfloat16().cuda()
        out = ops.paged_attention_decode(q, k, v, bt, sl, d ** -0.5, max_ctx=ctx)
    expect = ref.paged_attention_decode(q.float(), kf.bfloat16().float(), vf, bt, sl, d ** -0.5)
    # as above: bf16 probabilities and result, and as much again for a rotated element that rounds the other way
    assert (out.float() - expect).abs().max() <= 2.0 ** -7 * vf.abs().max()


@gpu
@pytest.mark.parametrize("b,hq,hkv,d,ctx,rest,splits,joined", [
    (64, 16, 8, 128, 120, 120, 2, True), (3, 32, 32, 64, 300, 250, 5, True), (3, 32, 32, 64, 384, 1, 6, True),
    (16, 16, 8, 64, 448, 447, 7, True), (32, 8, 8, 64, 512, 65, 8, True), (32, 32, 8, 128, 300, 60, 3, True),
    (32, 32, 8, 128, 1000, 60, 4, False), (64, 16, 8, 128, 700, 33, 2, False)])
@pytest.mark.parametrize("fused", [False, True])
def test_decode_attention_join_follows_the_longest_sequence(cuda, b, hq, hkv, d, ctx, rest, splits, joined, fused):
    """One sequence of ``ctx`` keys among ``rest``: 2 to 8 splits as the waves of a workgroup, which leaves the partials'
    workspace alone, and apart where the waves of one long sequence would wait for each other on a CU; against float32."""
    from distributed_llms_amd import knobs
    torch.manual_seed(b + ctx)
    lens = [ctx] + [rest] * (b - 1)
    used, width = sum(-(-n // 32) for n in lens), 1 << (-(-ctx // 32) - 1).bit_length()
    k, v = torch.randn(used, hkv, 32, d).bfloat16().cuda(), torch.randn(used, hkv, d, 32).bfloat16().cuda()
    bt, at = torch.zeros(b, width, dtype=torch.int32), 0
    for i, n in enumerate(lens):
        bt[i, :-(-n // 32)] = torch.arange(at, at + -(-n // 32))
        at += -(-n // 32)
    slots = torch.tensor([int(bt[i, (n - 1) // 32]) * 32 + (n - 1) % 32 for i, n in enumerate(lens)], dtype=torch.int32).cuda()
    bt, sl = bt.cuda(), torch.tensor(lens, dtype=torch.int32).cuda()
    kf, vf = k.float(), v.float()
    ws = (torch.full((b * hq * splits * d,), 7.0, device="cuda"), torch.full((b * hq * splits * 2,), 7.0, device="cuda"))
    with knobs.override(attn_target_waves=2048 if splits == 8 else knobs.K.attn_target_waves):
        assert ops.decode_split_plan(b, hkv, ctx, 32, width)[0] == splits
        if fused:
            qkv = torch.randn(b, (hq + 2 * hkv) * d).bfloat16().cuda()
            cs = ref.rope_cos_sin(d, 4096, 500000.0, device="cuda")
            q = ref.rope_cache_append(qkv.float(), sl - 1, cs, kf, vf, slots, hq, hkv, d).bfloat16()
            out = ops.paged_attention_decode_rope(qkv, sl - 1, cs, k, v, slots, bt, sl, hq, hkv, d, d ** -0.5, max_ctx=ctx,
                                                  workspace=ws)
        else:
            q = torch.randn(b, hq, d).bfloat16().cuda()
            out = ops.paged_attention_decode(q, k, v, bt, sl, d ** -0.5, max_ctx=ctx, workspace=ws)
    assert all(bool((t == 7.0).all()) for t in ws) == joined
    expect = ref.paged_attention_decode(q.float(), kf.bfloat16().float(), vf, bt, sl, d ** -0.5)
    # as above: bf16 probabilities and result, and as much again for a rotated element that rounds the other way
    assert (out.float() - expect).abs().max() <= 2.0 ** -7 * vf.abs().max()
