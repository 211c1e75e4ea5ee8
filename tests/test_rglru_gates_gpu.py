"""The gates of the recurrence over many tokens on the bf16 matrix cores, against 64-bit sums."""
import pytest
import torch

from distributed_llms_amd import _ext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,bw", [(1, 8), (2, 40), (1, 100), (1, 15), (4, 128), (3, 264), (2, 512)])
@pytest.mark.parametrize("tokens", [65, 128, 129, 300])
@pytest.mark.parametrize("size", [1e-3, 1.0, 30.0])
def test_gates_keep_all_bits_of_the_input(cuda, nb, bw, tokens, size):
    """Partial tiles of tokens, outputs and K chunks; the three bf16 pieces of an input carry all of its 24 bits."""
    g = torch.Generator().manual_seed(bw + tokens)
    r = lambda *s, scale=1.0: torch.randn(*s, generator=g) * scale
    u = r(tokens, nb, bw, scale=size)
    ra, ri = r(nb, bw, bw, scale=bw ** -0.5).bfloat16(), r(nb, bw, bw, scale=bw ** -0.5).bfloat16()
    rb, ib, lam = r(nb, bw, scale=0.3).bfloat16(), r(nb, bw, scale=0.3).bfloat16(), r(nb, bw).bfloat16()
    a, y = (torch.full((tokens, nb * bw), float("nan"), device=cuda) for _ in range(2))
    d = [x.to(cuda).contiguous() for x in (u, ra, rb, ri, ib, lam)]
    torch.cuda.synchronize()
    _ext.kernels().sm_rglru_gates(a.data_ptr(), y.data_ptr(), *(x.data_ptr() for x in d), tokens, nb, bw, 8.0, 0,
                                  torch.cuda.current_stream().cuda_stream)
    mul = lambda w: torch.matmul(u.double().transpose(0, 1), w.double()).transpose(0, 1)
    # the sums: exact products, bw float32 additions of at most the row's absolute sum each, 2^-24 apart
    bound = lambda w: torch.matmul(u.double().abs().transpose(0, 1), w.double().abs()).transpose(0, 1) * (3 * bw + 8) * 2.0 ** -24
    zr, zi = mul(ra) + rb.double(), mul(ri) + ib.double()
    sp = torch.nn.functional.softplus(lam.double())
    at = lambda z: torch.exp(-8.0 * torch.sigmoid(z) * sp)
    want = at(zr)
    # a falls by at most 2 sp = 8 sp / 4 per unit of its sum; as much as 1e-5 of the exponent for the float32 functions
    slack = want * (2 * sp * bound(ra) + 1e-5 * (1 + 8 * sp)) + 1e-12
    assert ((a.cpu().double().view(tokens, nb, bw) - want).abs() <= slack).all()
    x = u.double()
    mult = lambda v: torch.sqrt((1 - v * v).clamp_min(0))
    lo, hi = mult((want + slack).clamp_max(1)), mult((want - slack).clamp_min(0))
    gate, dg = torch.sigmoid(zi), bound(ri) / 4 + 1e-6
    err = (y.cpu().double().view(tokens, nb, bw) - mult(want) * gate * x).abs()
    assert (err <= ((hi - lo) * gate + dg + 1e-6) * x.abs() + 1e-12).all()


@pytest.mark.parametrize("nb,bw,tokens", [(8, 48, 4096), (8, 48, 4097), (8, 128, 4096), (8, 128, 4097), (8, 132, 4097), (3, 44, 200),
                                          (2, 257, 130)])
def test_gates_on_both_sides_of_the_rule(cuda, nb, bw, tokens):
    """Narrow blocks, many workgroups of blocks up to 128, widths that are no multiple of 4: an output per lane; else four."""
    test_gates_keep_all_bits_of_the_input(cuda, nb, bw, tokens, 1.0)


def _gates(cuda, u, ra, rb, ri, ib, lam):
    tokens, nb, bw = u.shape
    a, y = (torch.full((tokens, nb * bw), float("nan"), device=cuda) for _ in range(2))
    d = [x.to(cuda).contiguous() for x in (u, ra, rb, ri, ib, lam)]
    torch.cuda.synchronize()
    _ext.kernels().sm_rglru_gates(a.data_ptr(), y.data_ptr(), *(x.data_ptr() for x in d), tokens, nb, bw, 8.0, 0,
                                  torch.cuda.current_stream().cuda_stream)
    return a.cpu().view(tokens, nb, bw), y.cpu().view(tokens, nb, bw)


def test_gates_of_the_largest_inputs(cuda):
    """Finite inputs above the largest bf16 number stay finite (infinity times a zero weight is no number); infinite and
    NaN inputs reach the sums of their own token alone."""
    tokens, nb, bw = 70, 2, 64
    top = torch.finfo(torch.float32).max
    u = torch.zeros(tokens, nb, bw)
    u[0, 0, 3], u[1, 1, 5], u[2, 0, 0], u[3, 0, 0] = top, -top, float("inf"), float("nan")
    w = torch.zeros(nb, bw, bw)
    w[0, 3, 7] = 2.0 ** -120                                   # the one weight that meets a large input: 256 and -256
    w[1, 5, 9] = 2.0 ** -120
    zero = torch.zeros(nb, bw).bfloat16()
    a, _ = _gates(cuda, u, w.bfloat16(), zero, w.bfloat16(), zero, zero)
    want = torch.exp(-8.0 * torch.sigmoid(torch.matmul(u.double().transpose(0, 1), w.double()).transpose(0, 1)) *
                     torch.tensor(2.0).double().log())
    ok = torch.ones(tokens, dtype=torch.bool)
    ok[2:4] = False
    torch.testing.assert_close(a[ok].double(), want[ok], rtol=1e-5, atol=1e-12)
    assert a[2:4, 0].isnan().all() and (a[2:4, 1] == a[4, 1]).all()


@pytest.mark.parametrize("nb,bw", [(3, 128), (2, 256), (1, 512)])
def test_gates_see_the_last_bits_of_the_input(cuda, nb, bw):
    """One product per sum (a permutation for the weights), so that nothing but the input's own bits and the float32 functions
    round: the third piece shows in every block and every K chunk.  z = -3 .. -6: the gates are open to a change of z."""
    tokens = 130
    g = torch.Generator().manual_seed(bw)
    u = -(3.0 + 3.0 * torch.rand(tokens, nb, bw, generator=g))
    perm = torch.stack([torch.randperm(bw, generator=g) for _ in range(nb)])          # output o reads input perm[o]
    w = torch.zeros(nb, bw, bw)
    w[torch.arange(nb)[:, None], perm, torch.arange(bw)] = 1.0
    zero, lam = torch.zeros(nb, bw).bfloat16(), torch.full((nb, bw), 3.0).bfloat16()
    a, _ = _gates(cuda, u, w.bfloat16(), zero, w.bfloat16(), zero, lam)
    at = perm.expand(tokens, nb, bw)

    def gate(v):
        z = torch.gather(v.double(), 2, at)
        return z, 8.0 * torch.sigmoid(z) * torch.nn.functional.softplus(lam.double())
    z, e = gate(u)
    want = torch.exp(-e)
    # the exponent: the three pieces' sum (2^-23 of z at most, which moves it by as much of e |z|), expf, two additions, a
    # division, softplus and two products at 2^-23 or less each: 12 x 2^-24 of it; the last expf 2^-22
    tol = want * (e * z.abs() * 2.0 ** -23 + e * 12 * 2.0 ** -24 + 2.0 ** -22)
    assert ((a.double() - want).abs() <= tol).all()
    h = u.bfloat16()
    two = h.double() + (u - h.float()).bfloat16().double()                            # an input of two pieces would be seen
    seen = (torch.exp(-gate(two)[1]) - want).abs() > tol
    chunk = torch.nn.functional.one_hot(at // 64, bw // 64).bool()
    assert ((seen[..., None] & chunk).sum(0).sum(1) > 0.5 * chunk.sum(0).sum(1)).all()


@pytest.mark.parametrize("nb,bw,tokens", [(10, 256, 300), (4, 256, 168), (2, 132, 1001), (3, 48, 65), (1, 700, 130), (8, 128, 4096)])
def test_gates_have_the_same_bits_on_either_kernel(cuda, nb, bw, tokens):
    """Four outputs per lane, and an output per lane (which an input off its 16 bytes takes): the same products in the same order,
    and the same functions of them, over gates that are nearly shut, half open and nearly open."""
    g = torch.Generator().manual_seed(bw)
    r = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(cuda)
    u = r(tokens * nb * bw, scale=8.0)
    off = torch.empty(u.numel() + 1, device=cuda)[1:].copy_(u)
    assert u.data_ptr() % 16 == 0 and off.data_ptr() % 16 == 4
    w = [r(nb, bw, bw, scale=bw ** -0.5).bfloat16() for _ in range(2)]
    b = [r(nb, bw).bfloat16() for _ in range(3)]
    out = []
    for x in (u, off):
        a, y = (torch.full((tokens, nb * bw), float("nan"), device=cuda) for _ in range(2))
        _ext.kernels().sm_rglru_gates(a.data_ptr(), y.data_ptr(), x.data_ptr(), w[0].data_ptr(), b[0].data_ptr(), w[1].data_ptr(),
                                      b[1].data_ptr(), b[2].data_ptr(), tokens, nb, bw, 8.0, 0, torch.cuda.current_stream().cuda_stream)
        out.append((a, y))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert not out[0][0].isnan().any() and not out[0][1].isnan().any()
