"""FP8 (OCP e4m3) W8A8 decode GEMMs -- the quantization capability the reference only documents
(``plan.md:109-112,438-456``, ``snippets.md:684-833`` sketch bitsandbytes int8/int4
with an absmax fallback; the reference code never quantizes anything).

MI355X-native form: CDNA4's block-scaled MFMA (``v_mfma_scale_f32_16x16x128_f8f6f4``) runs e4m3 at
twice the bf16 rate, and an e4m3 weight is half the bytes, so the decode projections -- which sit on
the bf16 ridge at batch 256 -- get both halves of their bound cut:

* weights: per-output-channel absmax scales, quantized once at load (:func:`quantize_weight`);
* activations: per-token absmax scales, quantized on the fly by ``quant_fp8_rows``
  (csrc/kernels/quant.hip);
* GEMM: ``gemm_wide_fp8`` (csrc/kernels/gemm_wide.hip) -- the wide kernel's LDS-DMA pipeline with
  fp8 K-tiles of 128, scales applied in the epilogue (also before SwiGLU and before split-K slabs,
  so the bf16 path's deferred reductions are reused unchanged); the larger prompt products on ``gemm_pf8``
  (csrc/kernels/gemm_pf8.hip), persistent workgroups on 256-column tiles with the same bits.

Mixtral experts take the same scheme through the grouped kernel (``moe_wide_gemm_fp8``: fp8 token
rows gathered by the expert-sorted slot list, per-(expert, channel) weight scales).

Opt-in (``EngineConfig.quant = "fp8"``, ``bench.py --quant fp8``): the LM head, embeddings, norms,
router, attention and the KV cache stay bf16.  CPU tensors take the PyTorch reference below (same
quantization, f32 math), which is also the numerics oracle of the GPU tests.
"""
from __future__ import annotations

import functools
from typing import Tuple

import torch

from .. import _ext, knobs
from .stream import current_stream

FP8 = torch.float8_e4m3fn
FP8_MAX = 448.0
QUANT_KEYS = ("wqkv", "wo", "w_gate_up", "w_down")
EXPERT_KEYS = ("experts_gate_up", "experts_down")


class Fp8Weight:
    """An [N, K] weight as e4m3 values ``q`` and per-row (output channel) f32 ``scale``:
    w ~= q * scale[:, None]."""

    __slots__ = ("q", "scale")

    def __init__(self, q: torch.Tensor, scale: torch.Tensor):
        if q.dtype != FP8 or q.dim() != 2 or scale.shape != (q.shape[0],) or scale.dtype != torch.float32:
            raise ValueError("Fp8Weight: q [N, K] float8_e4m3fn and scale [N] float32")
        self.q, self.scale = q.contiguous(), scale.contiguous()

    @property
    def shape(self):
        return self.q.shape

    @property
    def device(self):
        return self.q.device

    @property
    def dtype(self):
        return FP8

    def numel(self) -> int:
        return self.q.numel()

    def nbytes(self) -> int:
        return self.q.numel() + 4 * self.scale.numel()

    def dequantize(self, dtype=torch.float32) -> torch.Tensor:
        return (self.q.float() * self.scale[:, None]).to(dtype)

    def __repr__(self):
        return f"Fp8Weight(shape={tuple(self.q.shape)}, device={self.q.device})"


class Fp8Experts:
    """A stack of expert weights [E, N, K] as e4m3 ``q`` with per-(expert, channel) f32 ``scale``
    [E, N]; ``experts[j]`` is expert j's :class:`Fp8Weight`."""

    __slots__ = ("q", "scale")

    def __init__(self, q: torch.Tensor, scale: torch.Tensor):
        if q.dtype != FP8 or q.dim() != 3 or scale.shape != q.shape[:2] or scale.dtype != torch.float32:
            raise ValueError("Fp8Experts: q [E, N, K] float8_e4m3fn and scale [E, N] float32")
        self.q, self.scale = q.contiguous(), scale.contiguous()

    @property
    def shape(self):
        return self.q.shape

    @property
    def device(self):
        return self.q.device

    @property
    def dtype(self):
        return FP8

    def is_contiguous(self) -> bool:
        return True

    def numel(self) -> int:
        return self.q.numel()

    def nbytes(self) -> int:
        return self.q.numel() + 4 * self.scale.numel()

    def __getitem__(self, j: int) -> Fp8Weight:
        return Fp8Weight(self.q[j], self.scale[j])

    def __repr__(self):
        return f"Fp8Experts(shape={tuple(self.q.shape)}, device={self.q.device})"


class Fp8Act:
    """A per-token quantized activation [..., K]: e4m3 ``q`` [M, K], f32 ``scale`` [M].  Produced by
    the norm kernels when the next GEMM takes fp8 (``ops.rms_norm(..., quant=True)``), consumed by
    :func:`linear_fp8` without a separate quantization launch."""

    __slots__ = ("q", "scale", "shape", "dtype")

    def __init__(self, q, scale, shape, dtype):
        self.q, self.scale, self.shape, self.dtype = q, scale, tuple(shape), dtype

    @property
    def device(self):
        return self.q.device

    @property
    def is_cuda(self):
        return self.q.is_cuda

    def dequantize(self) -> torch.Tensor:
        return (self.q.float() * self.scale[:, None]).to(self.dtype).reshape(self.shape)


def _absmax_scale(amax: torch.Tensor) -> torch.Tensor:
    # a tensor divisor: torch divides a GPU tensor by a Python scalar as a multiply by its
    # (inexact) reciprocal; the kernel, and the CPU, divide correctly rounded
    return torch.where(amax > 0, amax / torch.full_like(amax, FP8_MAX), torch.ones_like(amax))


def quantize_weight(w: torch.Tensor) -> Fp8Weight:
    """Per-output-channel absmax quantization of an [N, K] weight (any float dtype, any device)."""
    wf = w.float()
    s = _absmax_scale(wf.abs().amax(dim=1))
    q = (wf / s[:, None]).clamp(-FP8_MAX, FP8_MAX).to(FP8)
    return Fp8Weight(q, s)


def quantize_experts(w: torch.Tensor) -> Fp8Experts:
    """Per-(expert, output channel) absmax quantization of an [E, N, K] expert stack."""
    wf = w.float()
    s = _absmax_scale(wf.abs().amax(dim=2))
    q = (wf / s[..., None]).clamp(-FP8_MAX, FP8_MAX).to(FP8)
    return Fp8Experts(q, s)


def quantize_rows_ref(x: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Per-row (per-token) absmax quantization, PyTorch reference: (q [M, K] e4m3, scale [M] f32)."""
    xf = x.reshape(-1, x.shape[-1]).float()
    s = _absmax_scale(xf.abs().amax(dim=1))
    return (xf / s[:, None]).clamp(-FP8_MAX, FP8_MAX).to(FP8), s


def quantize_rows(x: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Per-token quantization of a bf16 activation [..., K] -> (q [M, K] e4m3, scale [M] f32); the
    HIP kernel on the GPU (bit-identical to :func:`quantize_rows_ref`)."""
    if not x.is_cuda:
        return quantize_rows_ref(x)
    if x.dtype != torch.bfloat16 or not x.is_contiguous():
        raise ValueError("quantize_rows: bf16 contiguous activations")
    k = x.shape[-1]
    m = x.numel() // k
    if k % 8:
        raise ValueError("quantize_rows: K % 8")
    q = torch.empty(m, k, dtype=FP8, device=x.device)
    s = torch.empty(m, dtype=torch.float32, device=x.device)
    _ext.kernels().quant_fp8_rows(q.data_ptr(), s.data_ptr(), x.data_ptr(), m, k,
                                  current_stream())
    return q, s


def linear_ref(x, w: Fp8Weight, swiglu: bool = False) -> torch.Tensor:
    """The W8A8 product in f32 from the quantized operands (CPU path and GPU-test oracle);
    ``x``: a float tensor (quantized here) or an :class:`Fp8Act`."""
    q, s = (x.q, x.scale) if isinstance(x, Fp8Act) else quantize_rows_ref(x)
    y = (q.float() * s[:, None]) @ w.dequantize(torch.float32).t().to(q.device)
    if swiglu:
        g, u = y.chunk(2, dim=-1)
        y = torch.nn.functional.silu(g) * u
    return y.to(x.dtype).reshape(*x.shape[:-1], y.shape[-1])


# 128 < M <= 256 split-K grids (qkv / o / down): two 128-row tiles with at most half the K slices
# instead of one 256-row tile -- a third fewer staged bytes per workgroup per K-tile (the loop is
# bound by its LDS-DMA staging).  bench/fp8_bench.py --sweep at M = 256 (us, default 1-tile plan ->
# this): o_8b 21.4 -> 18.0, qkv_8b 20.3 -> 19.1 (2 slices; 3 slices: 26.0), down_8b 29.3 = 29.3
# (knobs.fp8_bm128)
# prefill-sized M (no K split): grouped row-tile order (gemm_wide_fp8 variant bit 64) from this M:
# at M = 32768 qkv 1018 -> 889 us, o 660 -> 599, gate|up 4509 -> 3924, down 2083 -> 1873 (1.8-2.0
# PFLOP/s); at M = 2048 it is 1-6 % slower (knobs.fp8_group_m).  Those are 256-row tiles; shorter ones gain from half as
# many rows: 4096 x 14336 in 192 rows, M = 3072 / 6144, 194 / 397 -> 179 / 363, 128 rows at M = 3072 221 -> 213


# Past 256 rows the workgroups of a grid run in rounds of one per CU, so what a launch takes is the number of rounds times
# what a workgroup of that row tile takes: a K-tile of 128, us, and the workgroup's start and epilogue (measured, one
# round, K = 2048 ... 14336).  Shorter tiles do less per byte staged.  Two 64-row workgroups share a CU: a further round adds
# less than the first.  A K split adds its slabs: written and read by the consumer, which sums them on its way (the norm behind
# o and down, the K / V append behind qkv: 0.3 us more than reading the finished product), or, for a GLU, by a launch of their
# own; us, and us per million slab elements.  Charged with a launch of its own throughout, a plain product went unsplit where that
# is slower: split as formerly / unsplit / now, 4096 x 4096 at 384 / 640 rows with the norm 25.2 / 28.5 / 25.2 and 33.2 / 34.4 / 30.3,
# 6144 x 4096 at 384 29.7 / 34.5 / 29.7 and with the append 31.1 / 35.5 / 31.1.  196 sizes (14 weights 512 x 4096 ... 8192 x 28672, 257 to
# 2800 rows) are within 0.1 % of the best grid in the mean, their norm included, 140 GLUs within 0.4 %, and none is 3 % slower than under
# the former plan (the decode kernels' K split, 192 / 256-row tiles).  Former -> this, norm included, us: 4096 x 14336 at M =
# 640 / 1232 89.5 / 130 -> 66.3 / 108; 4096 x 4096 at 500 / 768 31.1 / 44.4 -> 25.9 / 35.4; 6144 x 4096 at 448 / 768 43.7 / 46.5 -> 34.2 /
# 42.7; 1024 x 4096 at 300 / 1232 19.0 / 30.0 -> 14.9 / 26.0; 2048 x 8192 at 300 / 900 26.2 / 46.5 -> 23.8 / 38.5; where 256 rows
# fill their rounds (28672 x 4096 at 2432, 302 against 328 in 192 rows; 6144 x 4096 at 2048, 64 against 67 in 128) nothing changes.
_ROUND_US = {64: (0.435, 3.2), 128: (0.505, 5.0), 192: (0.66, 5.5), 256: (0.745, 6.6)}
_ROUND_64 = 0.36
_SLAB_US = {False: (0.3, 0.2), True: (3.0, 0.32)}      # GLU


@functools.lru_cache(maxsize=1024)        # a pass asks for the same few products in every layer, 7 to 29 us each
def _prompt_plan(m: int, n: int, k: int, most: int, cus: int, swiglu: bool) -> Tuple[int, int]:
    """(K slices, row tile) of the cheapest grid past 256 rows.  ``most``: the slabs hold 16 bits, so a product is split no
    further than the decode rule would split it, and one that this leaves whole stays whole.  The slices, which set how the
    result rounds, are those of the whole chip (and of no one consumer: a stage that ends behind the product has another);
    ``cus`` -- what communication leaves of it -- moves the row tile alone, which changes no bit: a pipeline's stages round as
    one engine does."""
    from . import gemm

    def us(s, bm, cus):
        tile_us, fixed = _ROUND_US[bm]
        rounds, kt = -(-(n // 128) * -(-m // bm) * s // cus), -(-(k // 128) // s)
        t = (tile_us + _ROUND_64 * (rounds - 1)) * kt + fixed if bm == 64 else rounds * (tile_us * kt + fixed)
        slab, per = _SLAB_US[swiglu]
        return t + (slab + per * s * m * n * 1e-6 if s > 1 else 0.0)

    best, plan = float("inf"), (1, 256)
    for bm in (256, 192, 128, 64):
        for s in range(1, min(most, 8, max(1, k // 128 // 4)) + 1):
            if s > 1 and (s * m * n > gemm._WS_FLOATS or (n // 128) * -(-m // bm) * s > 256):
                break
            if us(s, bm, 256) < best:
                best, plan = us(s, bm, 256), (s, bm)
    return plan if cus == 256 else (plan[0], min((256, 192, 128, 64), key=lambda bm: us(plan[0], bm, cus)))


# gemm_pf8 (256-column tiles, persistent) against that: us per K-tile of 128 and round, per K-tile of a full chip's tiles (the clock
# falls as the matrix cores fill), per round (epilogue, first K-tiles) and once.  Fitted over 17 weights (512 x 2048 ... 57344 x 8192)
# at 257 ... 4096 rows, 289 sizes, to 4 % where the tile is a likely one; gemm_wide_fp8 takes 1.11 times its model in the mean there.
# Of the 199 that the plan leaves whole none is slower than it was, and together they take 0.73 of the time (29.6 -> 21.6 ms; the better
# kernel and tile at each: 21.5).  us at 2560 rows:
# 28672 x 4096 with its SwiGLU 315 -> 221 (2.7 PFLOP/s; at 8192 rows 956 -> 629, 3.1), 4096 x 14336 169 -> 103, 6144 x 4096 68 -> 48,
# 4096 x 4096 54 -> 35; 28672 x 4096 at 300 rows 52 -> 35.  A product that the plan splits takes gemm_pf8 a fifth to a half longer.
_PF8_US = {160: (0.572, 0.28, 3.6, 3.7), 192: (0.643, 0.321, 4.75, 2.8), 224: (0.64, 0.474, 4.9, 3.65), 256: (0.77, 0.484, 6.0, 2.85)}


@functools.lru_cache(maxsize=1024)
def _pf8_plan(m: int, n: int, k: int, bm: int) -> int:
    """gemm_pf8's row tile for a product past 256 rows that :func:`fp8_plan` leaves whole, on row tiles of ``bm``; 0 where that is
    cheaper (a small product: half as many columns per tile leave fewer CUs idle).  No bit hangs on it."""
    if n % 256 or k % 256 or k < 512 or m * k >= 1 << 32 or n * k >= 1 << 32 or m * n * 2 >= 1 << 31:
        return 0
    kt, rounds = k // 128, -(-(n // 128) * -(-m // bm) // 256)
    tile_us, fixed = _ROUND_US[bm]
    best = 1.04 * ((tile_us + _ROUND_64 * (rounds - 1)) * kt + fixed if bm == 64 else rounds * (tile_us * kt + fixed)) + 1.5
    plan = 0
    for rows, (a, b, e, f) in _PF8_US.items():
        tiles = n // 256 * -(-m // rows)
        us = kt * (a * -(-tiles // 256) + b * tiles / 256) + e * -(-tiles // 256) + f
        if us < best:
            best, plan = us, rows
    return plan


def fp8_plan(m: int, n: int, k: int, swiglu: bool = False) -> Tuple[int, int]:
    """(K slices, row-tile override or 0) of gemm_wide_fp8 for this shape.  Past 256 rows the cheapest
    grid (:func:`_prompt_plan`) of the CUs that communication leaves.  Default: the bf16 kernel's rule on the 128-K tiles (a K-tile
    of fp8 holds the bytes of a 64-K bf16 tile).  Twice the slices of half the K are 1 to 1.5 us of 9 to 10 faster up to 64
    rows (4096 x 4096 in 8 instead of 4), but a slice's sum is handed on in 16 bits: with 8 the error of the slabs' sum against 64
    bits was 3.2e-4 instead of 2.6e-4 for results around 0.01."""
    from . import gemm
    s = gemm.wide_splits(m, n, k // 2, swiglu)
    if m > 256:
        return _prompt_plan(m, n, k, s, 256 - gemm._comm_cus, swiglu)
    if knobs.K.fp8_bm128 and not swiglu and s > 1 and 128 < m <= 256:
        tiles = (n // 128) * 2
        return max(1, min(256 // tiles, (k // 128) // 4, 16)), 128
    return s, 0


def fp8_splits(m: int, n: int, k: int, swiglu: bool = False) -> int:
    return fp8_plan(m, n, k, swiglu)[0]


def fp8_variant(m: int, n: int, k: int, splits: int, bm: int) -> int:
    """gemm_wide_fp8's variant: cache policy of the weights (4: the default one, 1: nontemporal), tile order (64: grouped) and
    row-tile override.  Nontemporal where a weight byte is read once: up to 256 rows without a K split, and with one where a
    single row tile covers M, the slices are long (8 K-tiles; past 64 rows 12) and the Infinity Cache does not keep the matrix
    from step to step.  With the norm that sums the slabs behind it, default -> nontemporal, us: 6144 x 4096 (8 K-tiles) 11.7 /
    13.9 -> 10.9 / 13.5 at M = 1 / 64, 8192 x 28672 (56) 48.8 / 52.1 / 60.6 -> 43.5 / 48.0 / 58.0 at M = 1 / 64 / 128; but read by
    several row tiles 4096 x 14336 at M = 200 / 300 34.7 / 41.0 -> 36.2 / 42.8, 5120 x 25600 66.7 / 77.2 -> 69.5 / 81.6 (from 384
    rows on within 2 % either way) -- unless those are of 64 rows with the deep ring that goes with it (2048 x 8192 at 300 in 3
    slices and five row tiles, 25.4 -> 24.3)."""
    order = 64 if 0 < knobs.K.fp8_group_m <= (2 * m if 0 < bm < 256 else m) else 0
    if splits == 1:
        return (1 if m <= 256 else 4 | order) | (bm << 8)
    from . import gemm
    rows, kt = bm or gemm.wide_bm(m), -(-(k // 128) // splits)
    nt = n * k >= 12 << 20 and (kt >= (8 if m <= 64 else 12) if m <= rows else rows == 64 and kt >= 14)
    return (1 if nt else 4) | (bm << 8)


def linear_fp8(x: torch.Tensor, w: Fp8Weight, swiglu: bool = False, defer: bool = False, splits: int = 0):
    """y = x w^T (``swiglu``: silu(x Wg^T) * (x Wu^T), w = [Wg; Wu]) with W8A8 e4m3 operands.
    ``defer``: may return a :class:`~distributed_llms_amd.ops.gemm.SplitKPartial` (no SwiGLU)."""
    if not x.is_cuda:
        return linear_ref(x, w, swiglu)
    from . import gemm
    pre = isinstance(x, Fp8Act)
    k = x.shape[-1]
    n, kw = w.shape
    if kw != k:
        raise ValueError(f"linear_fp8: x[..., {k}] vs w {tuple(w.shape)}")
    if n % 128 or k % 128:
        raise ValueError("linear_fp8: N % 128 and K % 128")
    if x.dtype != torch.bfloat16:
        raise TypeError("linear_fp8: bf16 activations")
    if pre:
        xq, xs = x.q, x.scale
        m = xq.shape[0]
    else:
        x = x.contiguous()
        m = x.numel() // k
        xq, xs = quantize_rows(x)
    s, bm = fp8_plan(m, n, k, swiglu)
    if splits:
        s, bm = splits, 0
    ws = gemm._workspace(x.device)
    if s > 1 and s * m * n > ws.numel():
        s = max(1, ws.numel() // (m * n))
    variant = fp8_variant(m, n, k, s, bm)
    stream = current_stream()
    kern = _ext.kernels()
    if defer and not swiglu and s > 1:
        se = kern.gemm_wide_fp8(0, xq.data_ptr(), xs.data_ptr(), w.q.data_ptr(), w.scale.data_ptr(), ws.data_ptr(),
                                ws.numel(), m, n, k, s, 2, variant, stream)
        return gemm.SplitKPartial(ws, se, m, n, (*x.shape[:-1], n), x.dtype, x.device)
    y = torch.empty(*x.shape[:-1], n // 2 if swiglu else n, dtype=x.dtype, device=x.device)
    # (beside reserved CUs a persistent workgroup could wait for its CU with a whole share of the tiles)
    rows = 0
    if m > 256 and s == 1 and bm and not gemm._comm_cus and (xq.data_ptr() | w.q.data_ptr()) % 16 == 0:
        rows = _pf8_plan(m, n, k, bm)
    if rows:
        kern.gemm_pf8(y.data_ptr(), xq.data_ptr(), xs.data_ptr(), w.q.data_ptr(), w.scale.data_ptr(), m, n, k,
                      1 if swiglu else 0, rows, stream)
        return y
    kern.gemm_wide_fp8(y.data_ptr(), xq.data_ptr(), xs.data_ptr(), w.q.data_ptr(), w.scale.data_ptr(), ws.data_ptr(),
                       ws.numel(), m, n, k, s, 1 if swiglu else 0, variant, stream)
    return y


def moe_mlp_ref(x: torch.Tensor, w_gate_up: Fp8Experts, w_down: Fp8Experts, topk_w: torch.Tensor,
                topk_ids: torch.Tensor) -> torch.Tensor:
    """Mixtral expert MLPs with W8A8 experts (reference): per-token e4m3 inputs, per-row e4m3
    SwiGLU outputs, f32 products -- the numerics of the grouped fp8 kernels."""
    t, h = x.shape
    out = torch.zeros(t, h, dtype=torch.float32, device=x.device)
    for e in range(w_gate_up.shape[0]):
        tok, slot = (topk_ids == e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        y = linear_ref(linear_ref(x[tok], w_gate_up[e], swiglu=True), w_down[e])
        out.index_add_(0, tok, y.float() * topk_w[tok, slot].unsqueeze(1).float())
    return out.to(x.dtype)


def quantize_layers(layers, keys=QUANT_KEYS, expert_keys=EXPERT_KEYS) -> int:
    """Replace the dense projections (and MoE expert stacks) of every layer dict by
    :class:`Fp8Weight` / :class:`Fp8Experts` (in place); returns how many were converted.  The
    router, norms and biases stay as they are."""
    def ok(t, dims):
        # the GPU kernels tile N and K by 128 (CPU reference: any shape)
        return isinstance(t, torch.Tensor) and t.dim() == dims and (
            not t.is_cuda or (t.shape[-2] % 128 == 0 and t.shape[-1] % 128 == 0))
    n = 0
    for lw in layers:
        for name in keys:
            if ok(lw.get(name), 2):
                lw[name] = quantize_weight(lw[name])
                n += 1
        for name in expert_keys:
            if ok(lw.get(name), 3):
                lw[name] = quantize_experts(lw[name])
                n += 1
    return n
