"""The close of a sublayer in the launch of the product that reads it (csrc/kernels/gemm_close.hip), and the rule for it."""
import pytest
import torch
import torch.nn.functional as F

from distributed_llms_amd import knobs, ops
from distributed_llms_amd.ops import gemm
from distributed_llms_amd.ops import seqmix as sm


def _norm(v, w, b, eps):
    """RMS norm (no ``b``) around 1 + w, layer norm with one, in float64."""
    if b is None:
        return v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + eps) * (1.0 + w)
    c = v - v.mean(-1, keepdim=True)
    return c * torch.rsqrt(c.pow(2).mean(-1, keepdim=True) + eps) * w + b


def _args(kind, k, o_bias, seed, device):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().to(device)
    x, o = torch.randn(1, k, generator=g).to(device), r(1, k)
    kw = dict(w_post=r(k) * 0.2, w_next=r(k) * 0.2, eps=1e-5, bias=r(k) if o_bias else None)
    if kind == "rms":
        kw["mult"] = 0.75
    else:
        kw.update(b_post=r(k), b_next=r(k))
    return x, o, kw


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["rms", "layer"])
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("n,k", [(8, 512), (1536, 576), (2048, 1024), (6142, 1024), (6146, 1024), (3072, 1088), (5120, 2560), (15360, 2560), (4600, 3072)])
def test_close_product(cuda, kind, glu, n, k):
    """Widths at and between the edges of the row's pieces, few weight rows and many, ragged last workgroups, fewer workgroups
    than CUs and more, a clipped GLU with a bias and without; the new stream and the product."""
    x, o, kw = _args(kind, k, n % 4 == 0, n + k, "cuda")
    w = (torch.randn(n, k, device="cuda") * k ** -0.5).bfloat16()
    b = torch.randn(n, device="cuda").bfloat16() if glu and kind == "rms" and n != 6142 else None
    act = "" if not glu else "clipped" if kind == "rms" else "gelu"
    old = x.clone()
    r = gemm.close_product(kind, x, o, w, b, act, 0.7, kw["w_post"], kw["w_next"], kw["eps"], kw.get("mult", 1.0), 1.0 if kind == "rms" else 0.0,
                           kw["bias"], kw.get("b_post"), kw.get("b_next"))
    if (n, k, glu) == (15360, 2560, False):                                    # (more weights than this kernel is asked to take plain)
        assert r is None
        return
    xo, y = r
    assert torch.equal(x, old)
    d = lambda t: None if t is None else t.double()
    v = o.double() + (0 if kw["bias"] is None else kw["bias"].double())
    s = x.double() + kw.get("mult", 1.0) * _norm(v, d(kw["w_post"]), d(kw.get("b_post")), kw["eps"])
    # f32 sums of k squares and a handful of roundings, each within 2^-23
    assert bool(((xo.double() - s).abs() <= (k * 2.0 ** -24 + 2.0 ** -20) * (1.0 + s.abs())).all())
    h = _norm(xo.double(), d(kw["w_next"]), d(kw.get("b_next")), kw["eps"])
    z, mag = F.linear(h, w.double(), d(b)), h.abs() @ w.double().abs().t()
    # h rounds to bf16 (2^-9 each, and the norm's own 2^-20), the product sums k of them in f32
    e = (2.0 ** -9 + 2.0 ** -18 + k * 2.0 ** -24) * mag + (0 if b is None else 2.0 ** -20 * b.double().abs())
    if not glu:
        assert bool(((y.double() - z).abs() <= e + 2.0 ** -8 * z.abs()).all())
        return
    half = n // 2
    g, u = z[:, :half], z[:, half:]
    if act == "clipped":
        gc, uc = g.clamp(max=0.7), u.clamp(-0.7, 0.7)
        ref, up = gc * torch.sigmoid(1.702 * gc) * (uc + 1), uc.abs() + 1
    else:
        ref, up = F.gelu(g, approximate="tanh") * u, u.abs()
    # |d act / d gate| <= 1.2 |up|, act <= |gate| |up|: both sums' errors through the product; the result rounds to bf16
    tol = 1.2 * e[:, :half] * (up + e[:, half:]) + (g.abs() + 1e-3) * e[:, half:] + (2.0 ** -8 + 2.0 ** -18) * ref.abs() + 2.0 ** -22
    assert bool(((y.double() - ref).abs() <= tol).all())


# weight rows of a workgroup / 8 -> sizes of the plain product (with 8 waves, with 4) and of the GLU
PLAIN = [(8, 512), (1528, 576), (2560, 2560), (2056, 1024), (2560, 1280), (6152, 2048), (4104, 1024), (4610, 2112), (8200, 1024), (8200, 1536),
         (6152, 1024), (6152, 2560), (3072, 3072)]
GLUS = [(3072, 1024), (4096, 2048), (4096, 2560), (6146, 1024), (4104, 2560), (7680, 1280), (8192, 1024), (6152, 2560), (8200, 1088), (8206, 2560),
        (12296, 1024), (15360, 2560), (12296, 3072)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["rms", "layer"])
@pytest.mark.parametrize("n,k,glu", [(*s, False) for s in PLAIN] + [(*s, True) for s in GLUS])
def test_close_product_has_the_bits_of_two_launches(cuda, kind, n, k, glu):
    """Every split of the weight rows, both numbers of waves of a plain product, rows of one and of three pieces per lane, weights on
    either side of the cache policy's line: the stream and the product of the close's own launch and the product's."""
    x, o, kw = _args(kind, k, n % 16 == 0, n + k, "cuda")
    g = torch.Generator("cuda").manual_seed(n)
    w = (torch.randn(n, k, device="cuda", generator=g) * k ** -0.5).bfloat16()
    b = torch.randn(n, device="cuda", generator=g).bfloat16() if glu and kind == "rms" else None
    act = "" if not glu else "clipped" if kind == "rms" else "gelu"
    r = gemm.close_product(kind, x, o, w, b, act, 0.7, kw["w_post"], kw["w_next"], kw["eps"], kw.get("mult", 1.0), 1.0 if kind == "rms" else 0.0,
                           kw["bias"], kw.get("b_post"), kw.get("b_next"))
    assert r is not None
    f = sm.post_norm_add if kind == "rms" else sm.post_layer_norm_add
    xr, h = f(x.clone(), o, **kw)
    y = ops.linear(h, w) if not glu else sm.linear_clipped_glu(h, w, b, 0.7) if kind == "rms" else sm.linear_gelu_glu(h, w)
    assert torch.equal(r[0], xr) and torch.equal(r[1], y)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["rms", "layer"])
def test_close_refused(cuda, kind):
    """What the launch does not take goes to the close's own: several rows, widths past its registers, K no multiple of 64,
    float32, a view off its alignment, the switch."""
    def product(x, o, kw, n=2048, w=None):
        w = (torch.randn(n, x.shape[1], device="cuda") * 0.05).to(o.dtype) if w is None else w
        return gemm.close_product(kind, x, o, w, None, "", 0.0, kw["w_post"], kw["w_next"], kw["eps"], 1.0, 1.0, kw["bias"],
                                  kw.get("b_post"), kw.get("b_next"))
    x, o, kw = _args(kind, 1024, True, 1, "cuda")
    assert product(x, o, kw) is not None
    assert product(x.repeat(2, 1), o.repeat(2, 1), kw) is None
    assert product(x, o.float(), kw) is None
    pad = torch.zeros(1025, device="cuda")
    assert product(pad[1:].view(1, -1), o, kw) is None
    off = torch.zeros(1025, dtype=torch.bfloat16, device="cuda")[1:]
    assert product(x, o, {**kw, "w_next": off}) is None
    for k in (3136, 600):
        assert product(*_args(kind, k, False, 2, "cuda")) is None
    knobs.K.stream = False
    try:
        assert product(x, o, kw) is None
    finally:
        knobs.K.stream = True


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("kind", ["rms", "layer"])
@pytest.mark.parametrize("rows", [1, 3])
@pytest.mark.parametrize("last", [False, True])
def test_close_object(device, kind, rows, last, request):
    """Close gives the stream and the product that the calls of their own give, whichever way it takes (one rounding of h and
    one of the product apart at most)."""
    if device == "cuda":
        request.getfixturevalue("cuda")
    k, n = 1024, 256
    x, o, kw = _args(kind, k, True, 3, device)
    x, o = x.repeat(rows, 1), o.repeat(rows, 1)
    if last:
        kw.update(w_next=None, **({"b_next": None} if kind == "layer" else {}))
    w = (torch.randn(n, k, generator=torch.Generator().manual_seed(4)) * k ** -0.5).bfloat16().to(device)
    c = sm.Close(kind, x.clone(), o, **kw)
    f = sm.post_norm_add if kind == "rms" else sm.post_layer_norm_add
    rx, rh = f(x.clone(), o, **kw)
    if last:
        assert c.input() is None and torch.equal(c.x, rx)
        return
    y, ref = c.linear(w), ops.linear(rh, w)
    assert (c.x - rx).norm() <= 2.0 ** -18 * rx.norm()
    assert (y.double() - ref.double()).norm() <= 2.0 ** -7 * ref.double().norm()
    made = sm.Close.made(x, rh)
    assert made.input() is rh and torch.equal(made.linear(w), ref) and made.x is x


def test_no_load_of_a_close_can_move_in_front_of_its_barrier():
    """The barrier builtin orders nothing for the compiler: behind each one that ordinary LDS loads follow stands a clobber."""
    import os
    import re
    import distributed_llms_amd
    path = os.path.join(os.path.dirname(distributed_llms_amd.__file__), "csrc", "kernels", "gemm_stream.h")
    with open(path) as f:
        code = re.sub(r"//[^\n]*", "", f.read())
    behind = [code[m.end():].split(";")[0].strip() for m in re.finditer(r"^\s*__builtin_amdgcn_s_barrier\(\);", code, re.M)]
    assert len(behind) == 2 and all(b == 'asm volatile("" ::: "memory")' for b in behind)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("kind", ["rms", "layer"])
def test_close_is_read_by_one_product(monkeypatch, device, kind, request):
    """Behind a product that made the row in its launch there is no input to read: an error, not a product of nothing.  With
    the input asked for first any number of products read it."""
    if device == "cuda":
        request.getfixturevalue("cuda")
    x, o, kw = _args(kind, 1024, True, 5, device)
    w = (torch.randn(256, 1024, generator=torch.Generator().manual_seed(6)) / 32).bfloat16().to(device)
    if device == "cpu":
        monkeypatch.setattr(gemm, "close_product", lambda kind, x, o, w, *a, **k: (x + 1, o @ w.t()))
    c = sm.Close(kind, x.clone(), o, **kw)
    c.linear(w)
    for again in (c.input, lambda: c.linear(w)):
        with pytest.raises(RuntimeError, match="input"):
            again()
    c = sm.Close(kind, x.clone(), o, **kw)
    h = c.input()
    y = c.linear(w)
    assert c.input() is h and torch.equal(y, ops.linear(h, w)) and torch.equal(c.linear(w), y)


@pytest.mark.gpu
@pytest.mark.parametrize("more", [{"one_plus": False}, {"o2": True, "scales": (0.5, 2.0)}, {"plain_next": True}, {"final": True}])
def test_close_takes_every_argument_of_its_function(cuda, more):
    """Plain norm weights in either launch; what only the function makes is left to it."""
    x, o, kw = _args("rms", 1024, True, 7, "cuda")
    w = (torch.randn(256, 1024, generator=torch.Generator().manual_seed(8)) / 32).bfloat16().cuda()
    kw.update({k: o.flip(1).contiguous() if k == "o2" else v for k, v in more.items()})
    xr, h = sm.post_norm_add(x.clone(), o, **kw)
    c = sm.Close("rms", x.clone(), o, **kw)
    assert torch.equal(c.linear(w), ops.linear(h, w)) and torch.equal(c.x, xr)
