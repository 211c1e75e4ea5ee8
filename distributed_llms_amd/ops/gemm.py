"""Dense GEMM dispatch for y = x @ w^T (w is [N, K], nn.Linear layout).

Up to 64 rows, a small weight goes to the weight-streaming kernel (gemm_stream.hip, :func:`use_stream`): no K split,
bias and GLU in its epilogue.  Other decode-sized M go to hand-written gfx950 kernels, per projection role (cutovers measured in
the engine on Llama-3-8B, profiles/wide_gemm.md; each one is a field of :mod:`..knobs`):

* wide-M kernel (gemm_wide.hip: 64/128/192/256-row x 128 tiles, 3-stage LDS-DMA pipeline,
  split-K over workgroups) for every decode M:
  - gate|up (SwiGLU fused into the epilogue): M <= knobs.wide_gate_up_max_m (256);
  - down (K >= 8192 and K > N; split-K partials deferred into the next norm):
    M <= knobs.wide_down_max_m (512);
  - the other projections (qkv, o, LM head): M <= knobs.wide_proj_max_m (256); the o-projection
    (N K <= knobs.wide_small_bm_maxw) on 128-row tiles with half the K slices (knobs.wide_small_bm);
  with the 256 x 256 tile (gemm_sq.hip) taking unsplit grids at 225 <= M <= 256 (70B gate|up);
* the decode LM head at 225 <= M <= 256: gemm_pp.hip schedule 2 with nontemporal weights
  (knobs.pp_head_min_m);
* the decode SwiGLU gate|up at 200 <= M <= 256 on gemm_pp unsplit with nontemporal weights, on the
  column tile (128, else 256) that makes one round of CUs / 2 .. CUs tiles (8B: 224 x 128, 70B:
  224 x 256; knobs.pp_gate_up_min_m), and the long-K down projection (K >= knobs.pp_down_min_k,
  70B) at 225 <= M <= 256 on split gemm_pp 128-column tiles (profiles/round6_gate_up_pp.md);
* prefill (M >= knobs.pp_swiglu_min_m / pp_proj_min_m, above the decode ranges): the 4-wave
  schedule-2 kernel in its persistent form (gemm_pf in gemm_pp.hip, knobs.pp_persistent; 256 x 256 tiles, or row tiles of
  160 to 320 where they need fewer or cheaper rounds of the chip, :func:`_pf_tile`) -- gate|up with the GLU (and a clipped
  one's bias) in its epilogue, qkv / o / down plain (profiles/round4_gemm_counters.md);
* what none of them takes (a bias or N not a multiple of 128 past 64 rows, K not a multiple of 64, fp32 on CPU,
  operands >= 4 GiB): torch's F.linear.

The role is inferred from the shape: "down" = K >= 8192 and K > N, so the square / widening
K = 8192 projections of 70B-class models (qkv 8192 -> 10240, o 8192 -> 8192) stay "proj".
"""
from __future__ import annotations

import functools
import operator
from typing import Optional

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from .. import _ext
from .. import knobs
from .stream import current_stream


def is_down_proj(n: int, k: int) -> bool:
    """The MLP down projection's shape: long, narrowing K (8B: 14336 -> 4096, 70B: 28672 -> 8192).
    A K = 8192 qkv or o projection of a 70B-class model (N >= K) is not one."""
    return k >= 8192 and k > n


def _cus(device) -> int:
    if torch.device(device).type != "cuda":
        return 256                     # MI355X (dispatch unit tests on CPU)
    idx = device.index or 0
    n = _CUS.get(idx)
    if n is None:
        n = _CUS[idx] = torch.cuda.get_device_properties(idx).multi_processor_count
    return n


_CUS = {}


def _sizes(x: torch.Tensor, w: torch.Tensor, name: str):
    """(rows, N, K) of ``x w^T``; raises where the kernels, which see pointers and these numbers alone, would read past
    ``w`` or another device's memory."""
    k = x.size(-1)
    if w.dim() != 2 or w.size(1) != k:
        raise ValueError(f"{name}: x[..., {k}] vs w {tuple(w.shape)}")
    if w.device != x.device:
        raise ValueError(f"{name}: x on {x.device}, w on {w.device}")
    return x.numel() // k, w.size(0), k


def pf_fills(m: int, n: int, device) -> bool:
    """gemm_pf (one 256 x 256 tile per CU per round, no split-K) only where its grid fills the chip:
    at least one tile per CU and rounds that are mostly full (knobs.pf_min_eff), or many rounds.
    Below that the split-K gemm_pp grid wins at every measured M from 320 to 2048 -- gemm_pf's
    single-round grids run one tile's whole K loop: 74-78 us for the 8B o-projection at any
    M <= 2048, the down projection 250-283 us vs 55-174 us split (profiles/round5_medium_m_gemm.md)."""
    cus = _cus(device)
    tiles = (-(-m // 256)) * (n // 256)
    if tiles < cus:
        return False
    rounds = -(-tiles // cus)
    return rounds >= 4 or tiles / (rounds * cus) >= knobs.K.pf_min_eff


# Relative time of a round of gemm_pf's workgroups, by row tile.  A shorter tile does less per byte staged and per LDS read, so
# it pays only where it saves most of a round: 152 unsplit sizes (7 pairs of N 2560 .. 57344 and K 2560 .. 28672, M 264 ..
# 8192), each with every row tile, are within 0.3 % of the best tile in the mean under this rule, 5-6 % faster than 256 rows.
# us, 256 / 224 / 192 / 160 rows: 2560 x 2560, M = 7021 (280 / 320 / 370 / 440 tiles) 108 / 99 / 95 / 84; 4096 x 4096, 6210
# (400 / 448 / 528 / 624) 183 / 165 / 204 / 187; 6144 x 4096, 3072 (288 / 336 / 384 / 480) 172 / 153 / 146 / 136; 4096 x 14336,
# 5120 (320 / 368 / 432 / 512) 584 / 554 / 522 / 493; gate|up 28672 x 4096, 384 (224 / 224 / 224 / 336) 97 / 87 / 83 / 140.
# 128 rows (1.0 us a K-tile against 1.02 for 160) never win where there is no K split.
_PF_ROUND = {256: 1.0, 224: 0.93, 192: 0.84, 160: 0.76}
# ... and of the longer ones, which take a round away now and then: 63 unsplit sizes (7 pairs of N 4096 .. 28672 and K 2560 .. 14336,
# M 1232 .. 16384), each with every row tile, are 1.7 % from the best tile in the mean without them and 0.2 % with them.  us,
# 320 / 288 rows against the best of the others: 4096 x 14336, M = 4608 (240 / 256 tiles, 464 of 160 rows) 402 / 379, 468; 4096 x 4096,
# 4608 116 / 105, 127; 28672 x 4096, 1232 (448 / 560, 672 of 224) 226 / 280, 243, 7021 (2464 / 2800, 3584) 1164 / 1178, 1196; 6144 x 4096,
# 3000 (240 / 264, 456 of 160) 119 / 180, 129; 15360 x 2560, 1232 78 / 119, 87; 28672 x 4096, 16384 (no round less) 2678 / 2645, 2607.
_PF_ROUND_TALL = {288: 1.12, 320: 1.245}


def pf_row_tile(m: int, n: int, device, cus: int = 0) -> int:
    """Row tile with the shortest walk (over ``cus`` CUs, else the whole chip): rounds times the time of a round.  A single round
    of 256 rows is gemm_pp's (its epilogue through LDS is 5-7 % faster where no next tile hides the stores), which 224 rows
    do not beat."""
    cus = cus or _cus(device)
    best, at = 256, None
    for bm, c in _PF_ROUND.items():
        rounds = -(-(-(-m // bm) * (n // 256)) // cus)
        t = rounds * (_PF_ROUND[224] if bm == 256 and rounds == 1 else c)
        if at is None or t < at - 1e-6:
            best, at = bm, t
    return best


def _pf_tall(bm: int, m: int, n: int, out: int, device) -> int:
    """gemm_pf's row tile where :func:`_pf_plan` gives ``bm``: that, or 288 or 320 rows where their walk is cheaper.  No bit hangs
    on it; beside reserved CUs, with the dynamic tile queue (256 rows) and for outputs with nontemporal stores (a build of 256
    rows) the plan's stays."""
    if _comm_cus or pf_dynamic() or (out != n and m * out * 2 > 256 << 20):
        return bm
    cus = _cus(device)
    rounds = lambda b: -(-(-(-m // b) * (n // 256)) // cus)
    at = rounds(bm) * _PF_ROUND[bm]
    for b, c in _PF_ROUND_TALL.items():
        t = rounds(b) * c
        if t < at - 1e-6:
            bm, at = b, t
    return bm


def _pf_plan(m: int, n: int, k: int, out: int, device) -> int:
    """gemm_pf's row tile for an [m, k] x [n, k]^T product that no decode kernel takes (``out``: output columns), or 0 where
    gemm_pp serves.  Below 256 rows only where gemm_pp would not split K either -- the sums' order stays the same -- and
    nothing asks for nontemporal stores.  Beside reserved CUs (or with the dynamic tile queue, whose tiles have 256 rows) a
    plain product, which gemm_pp rounds alike, is left to that.  A GLU does not change kernels there -- gemm_pp's takes a gate
    and an up rounded to bf16, gemm_pf's the f32 sums -- so that a pipeline's stages round as one engine does: its row
    tile, which changes no bit, is the one for the CUs that are left.  us beside 16 reserved CUs, gemm_pp -> this: 28672 x
    4096 at 300 / 640 / 1232 rows 96 / 165 / 259 -> 67 / 122 / 236, 15360 x
    2560 at 640 / 1232 / 2300 57 / 109 / 171 -> 44 / 82 / 142."""
    if not knobs.K.pp_persistent or m * out * 2 >= 1 << 31:
        return 0
    if pp_splits(m, n, k) == 1 and (out == n or m * out * 2 <= 256 << 20):
        bm = pf_row_tile(m, n, device)
        if bm != 256:
            if not pf_dynamic() and not _comm_cus:
                return bm
            if out != n:
                return pf_row_tile(m, n, device, _pf_wgs(_cus(device)))
    return 256 if pf_fills(m, n, device) else 0


def _pf_tile(m: int, n: int, k: int, out: int, device) -> int:
    """Row tile of the prompt products: :func:`_pf_plan`'s kernel, with the longer tile where :func:`_pf_tall` finds its walk cheaper."""
    bm = _pf_plan(m, n, k, out, device)
    return _pf_tall(bm, m, n, out, device) if bm else 0


def _pf_wgs(cus: int) -> int:
    """Workgroups of gemm_pf's static walk: one per CU that is left (in eights: as many on every XCD).  One that has to wait
    for a CU would be waited for with its whole share of the tiles."""
    return max(8, (cus - _comm_cus) // 8 * 8)


@functools.lru_cache(maxsize=64)
def _roles(names: str) -> frozenset:
    return frozenset(t for t in names.split(",") if t and t != "none")


def _use_wide(m: int, n: int, k: int, x: torch.Tensor, w: torch.Tensor, swiglu: bool = False) -> bool:
    kn = knobs.K
    roles = _roles(kn.wide)
    if not roles or m < 1 or n % 128 or k % 64:
        return False
    if not (x.dtype == w.dtype == torch.bfloat16 and x.is_contiguous() and w.is_contiguous()):
        return False
    down = is_down_proj(n, k) and not swiglu
    if "all" in roles:
        return m <= 512 or (down and m <= kn.wide_down_max_m)
    if "auto" in roles:
        if swiglu:
            return m <= kn.wide_gate_up_max_m
        if down:
            return m <= kn.wide_down_max_m
        return m <= (kn.wide_o_max_m if n <= k else kn.wide_proj_max_m)
    if swiglu:
        return "gate_up" in roles and m <= 512
    return ("down" in roles) if is_down_proj(n, k) else ("proj" in roles and m <= 512)


# Where gemm_stream serves M <= 64 rows.  A launch and the slab sum that it saves are worth 2-4 us; what it pays is x, staged
# once per workgroup (so long K and many rows lose), and a last round of workgroups that leaves CUs idle.  Both sides as a
# caller gets them (reduction, gate kernel or closing norm included), cold weights, us, this kernel / the former route:
#  * plain, N a multiple of 128 (gemm_wide and its slab sum), M = 1 / 16 / 32 / 64: 1024 x 1024 2.8 / 3.0 / 3.4 / 4.2, 6.8 / 7.3 /
#    7.5 / 7.5; 4096 x 4096 8.3 / 8.7 / 10.4 / 13.6, 10.6 / 10.8 / 11.8 / 12.8; 2560 x 7680 10.5 / 13.3 / 16.8 / 22.8, 14.2 / 15.2 /
#    15.5 / 16.3; 1024 x 14336, 16 rows, 19.3, 16.9; 8192 x 4096 16.2 / 15.9 / 16.4, 15.6 / 15.6 / 16.0; 32000 x 1024 11.9 / 12.2 /
#    14.6, 12.6 / 12.6 / 12.8; 5120 x 4096 (160 workgroups), 32 rows, 14.6, 13.6;
#  * a bias or another N (F.linear), M = 17 / 33: 4096 x 4096 9-11, 17-24; 500 x 8192 12.3 / 16.5, 11.5 / 11.6; 6144 x 4096, 32
#    rows, 15.6, 14.8;
#  * in front of a close that sums the slabs itself, close included, M = 1 / 16 / 32 / 64: 2560 x 2560 7.6 / 9.1 / 10.6 / 13.3,
#    10.5 / 11.1 / 11.5 / 12.6; 512 x 4096 7.1 / 8.4 / 10.2 / 13.0, 8.6 / 9.1 / 9.2 / 9.5; 1024 x 8192, 16 rows, 13.2, 10.7;
#  * GLU, M = 1 / 32 / 64: 15360 x 2560 15.8 / 16.9 / 20.4, 18.4 / 19.3 / 20.9; 16384 x 4096 30.2 / 29.7 / 32.0, 34.4 / 33.6 / 34.3;
#    22016 x 4096 39.8 / 44.0 / 51.3, 34.1 / 35.0 / 39.2; 10240 x 4096 (160 workgroups) 22.0 / 22.6 / 25.7, 18.6 / 19.2 / 20.6;
#    28672 x 4096 41.8 / 45.0 / 53.4, 41.0 / 39.8 / 42.5; 4096 x 8192 17.8 / 24.0 / 28.7, 16.2 / 18.2 / 19.3.
# Up to 16 rows the workgroups are cut by what a CU stages (gemm_stream.hip, stream_rows), which took the line further out, us,
# M = 1 / 8 / 16:
#  * plain: 6144 x 4096 11.0 / 10.5 / 10.6, 13.3 / 13.2 / 13.5; 5120 x 5120 11.6 /
#    11.4 / 12.6, 13.4 / 14.0 / 14.4; 10240 x 8192 28.6 / 29.8 / 32.3, 32.4 / 32.7 / 31.6; 4096 x 8192 16.4 / 16.3, 16.0 / 15.6;
#  * in front of a close the line stays: 2560 x 7680 at 16 rows in a decode step 12.8 + 4.6 (close), 9.4 + 5.1;
#  * GLU: 16384 x 4096 24.7 / 23.6 / 25.8, 32.6 / 32.7 / 33.0; 14336 x 5120 25.8 / 24.8 / 26.0, 30.4 / 29.9 / 30.6; 28672 x 4096
#    38.6 / 37.3 / 42.1, 38.1 / 36.6 / 36.8; also where a round of the 16- or 32-column workgroups of more rows would leave CUs
#    idle: 10240 x 4096 16.9 / 16.9 / 17.5, 18.6 / 19.1 / 19.3; 22016 x 4096 30.9 / 31.1 / 31.9, 31.9 / 32.6 / 32.9; 17408 x 2560
#    17.2 / 17.7 / 19.4, 25.0 / 26.0 / 26.7.  With 4 KiB strides a third round of 24-row workgroups is too much for two groups
#    of x: 27648 x 2048 21.3 / 21.2 / 23.5, 21.0 / 21.1 / 21.1.
STREAM_MAX_M = 64


def _stream_fill(cols: int) -> float:
    """Share of the CUs that a round of gemm_stream's workgroups for ``cols`` output columns keeps busy past 16 rows (its
    launcher's rule there: tiles of 16 columns, of 32 once there are more than 256)."""
    tiles = -(-cols // 16)
    tiles = -(-cols // 32) if tiles > 256 else tiles
    return tiles / (256 * -(-tiles // 256))


def stream_fits(m: int, n: int, k: int, glu: str = "", defer: bool = False, bias: bool = False) -> bool:
    """Does gemm_stream serve an [m, k] x [n, k]^T product?  ``glu``: "" (plain), "silu", "clipped" or "gelu"."""
    if not 1 <= m <= STREAM_MAX_M or k % 64 or k < 512:
        return False                                 # K < 512: fewer K-tiles than waves, and no split to save either
    mi = n * k / (1 << 20)
    if glu and m <= 16:
        return k <= 5120 and mi <= 96 and (m <= 8 or n <= 24576 or k % 2048 != 0)
    if glu:
        if k > (4096 if m <= 32 else 2560) or (mi > (20 if m <= 32 else 12) and _stream_fill(n // 2) < 0.75):
            return False
        return mi <= (64 if m <= 32 and glu != "silu" else 40)
    if n > 65536:
        return False                                 # an LM head fills the chip unsplit on the wide kernel
    if defer and n % 128 == 0:
        return (mi <= 8 and k <= 4096) if m <= 16 else (mi <= 2 and k <= 2048)
    if m <= 16:
        return k <= 8192 and mi <= (32 if k <= 2560 else 80 if m <= 8 and n > 4096 else 28 if n > 4096 else 24)
    if m <= 32:
        return mi <= 24 and k <= 4096 and (mi <= 16 or _stream_fill(n) >= 0.75)
    if bias or n % 128:
        return mi <= 16 and k <= 4096
    return mi <= 12.5 and k <= 2560


_modes, _tracing, _transforms = (torch._C._len_torch_dispatch_stack, torch._C._get_tracing_state,
                                 torch._C._functorch.peek_interpreter_stack)
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _recorded(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor]) -> bool:
    """Is the call differentiated, transformed or traced (autograd, forward mode, vmap; torch.jit.trace, torch.compile,
    make_fx and other dispatch modes; tensor subclasses)?  The kernels leave no trace of it.  (Questions to the process
    first: an eager pass asks this for every product, and per tensor they cost three times as much.)"""
    if _modes() or _tracing() is not None or _transforms() is not None or forward_ad._current_level >= 0 \
            or torch.compiler.is_compiling():
        return True
    if type(x) not in _PLAIN or type(w) not in _PLAIN or (bias is not None and type(bias) not in _PLAIN):
        return True
    return torch.is_grad_enabled() and (x.requires_grad or w.requires_grad or (bias is not None and bias.requires_grad))


def use_stream(m: int, n: int, k: int, x: torch.Tensor, w: torch.Tensor, bias=None, glu: str = "", defer: bool = False) -> bool:
    return (knobs.K.stream and stream_fits(m, n, k, glu, defer, bias is not None) and x.dtype == w.dtype == torch.bfloat16
            # (a plain product without a bias, N a multiple of 128, and every GLU has kernels on either route)
            and not (not glu and (bias is not None or n % 128) and _recorded(x, w, bias))
            and x.is_contiguous() and w.is_contiguous() and x.data_ptr() % 16 == 0
            and w.data_ptr() % 16 == 0
            and (bias is None or (bias.dtype == torch.bfloat16 and bias.dim() == 1 and bias.size(0) == n
                                  and bias.is_contiguous() and bias.device == x.device)))


def linear_into_norm(x: torch.Tensor, w: torch.Tensor):
    """``x w^T`` for a consumer that sums split-K slabs itself (post_norm_add, post_layer_norm_add): the finished product
    where the weight-streaming kernel is faster than the split grid alone, else possibly a :class:`SplitKPartial`.  One row of
    a width that :func:`close_product` takes is finished wherever that kernel serves a plain product, also where the close then
    has a launch of its own (a latent layer's, the last one, one behind a product that is not fused).  us, with slabs / finished
    / finished and the close in the next product: 2560 x 7680 and 5120 x 2560 behind it 20.1 / 18.7 / 17.7, 2560 x 4096 17.7 /
    15.9 / 15.0, 2048 x 8192 and 4096 x 2048 18.5 / 16.3 / 16.0, 1536 x 6144 and 3072 x 1536 14.0 / 12.8 / 12.2, 1024 x 8192 and
    2048 x 1024 12.8 / 12.2 / 11.1, 3072 x 3072 and 4608 x 3072 18.1 / 15.3 / 14.5, 3072 x 8192 and 9216 x 3072 28.5 / 27.5 / 26.2."""
    m, n, k = _sizes(x, w, "linear_into_norm")
    if m <= STREAM_MAX_M and use_stream(m, n, k, x, w, defer=m > 1 or n > CLOSE_MAX_WIDTH):
        return _stream(m, n, k, x, w)
    return _linear(m, n, k, x, w, None, True)


CLOSE_MAX_WIDTH = 3072             # (csrc/kernels/gemm_close.hip: one row in the registers of four waves, and what more would cost)


def close_product(kind: str, x: torch.Tensor, o: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], glu: str,
                  limit: float, w_post, w_next, eps: float, mult: float = 1.0, offset: float = 0.0, o_bias=None, b_post=None,
                  b_next=None):
    """(x', y): the close of a sublayer (``kind`` "rms": post_norm_add, "layer": post_layer_norm_add) on a stream ``x`` [1, K]
    and the product of its output with ``w`` [N, K] (``glu``: "" (plain), "clipped" behind RMS norms or "gelu" behind layer
    norms) in one launch; None where a call of its own makes it: other numbers of rows (gemm_close.hip), widths, types or
    layouts, products that another kernel than the weight-streaming one serves."""
    n, k = w.shape if w.dim() == 2 else (0, 0)
    if not (knobs.K.stream and x.is_cuda and k <= CLOSE_MAX_WIDTH and x.shape == o.shape == (1, k) and x.dtype == torch.float32
            and w.dtype == torch.bfloat16 and glu in ("", "clipped" if kind == "rms" else "gelu") and (not glu or n % 2 == 0)
            and stream_fits(1, n, k, glu, False, bias is not None)):
        return None
    vecs = [t for t in (o, w_post, w_next, o_bias, b_post, b_next) if t is not None]
    if any(t.dtype != torch.bfloat16 or t.numel() != k or not t.is_contiguous() or t.device != x.device or t.data_ptr() % 8
           for t in vecs) or not (x.is_contiguous() and x.data_ptr() % 16 == 0 and w.is_contiguous() and w.device == x.device
                                  and w.data_ptr() % 16 == 0):
        return None
    if bias is not None and not (bias.dtype == torch.bfloat16 and bias.dim() == 1 and bias.size(0) == n and bias.is_contiguous()
                                 and bias.device == x.device):
        return None
    y = torch.empty(1, n // 2 if glu else n, dtype=torch.bfloat16, device=x.device)
    xo = torch.empty_like(x)
    p = lambda t: 0 if t is None else t.data_ptr()
    _ext.kernels().gemm_close(y.data_ptr(), w.data_ptr(), p(bias), n, k, _STREAM_GLU[glu], 1 if n * k * 2 >= WIDE_NT_MIN_BYTES else 0,
                              float(limit), 1 if kind == "rms" else 2, x.data_ptr(), o.data_ptr(), p(o_bias), w_post.data_ptr(),
                              p(b_post), w_next.data_ptr(), p(b_next), xo.data_ptr(), float(eps), float(mult), float(offset),
                              current_stream())
    return xo, y


_STREAM_GLU = {"": 0, "silu": 1, "clipped": 2, "gelu": 3}


def linear_stream(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None, glu: str = "",
                  limit: float = 0.0) -> torch.Tensor:
    """y = x w^T (+ bias), or its GLU with w = [Wg; Wu], for up to 64 rows (csrc/kernels/gemm_stream.hip)."""
    return _stream(*_sizes(x, w, "linear_stream"), x, w, bias, glu, limit)


def _stream(m: int, n: int, k: int, x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None, glu: str = "",
            limit: float = 0.0) -> torch.Tensor:
    """:func:`linear_stream` of operands whose sizes the caller has compared."""
    y = torch.empty(*x.shape[:-1], n // 2 if glu else n, dtype=x.dtype, device=x.device)
    _ext.kernels().gemm_stream(y.data_ptr(), x.data_ptr(), w.data_ptr(), 0 if bias is None else bias.data_ptr(), m, n, k,
                               _STREAM_GLU[glu], 1 if n * k * 2 >= WIDE_NT_MIN_BYTES else 0, float(limit),
                               current_stream())
    return y


def stream_logits(x: torch.Tensor, w: torch.Tensor, cap: float) -> torch.Tensor:
    """float32 cap tanh(z / cap) of z = x w^T rounded to bf16 (cap <= 0: z) of sizes that :func:`use_stream` takes."""
    (m, k), n = x.shape, w.shape[0]
    y = torch.empty(m, n, dtype=torch.float32, device=x.device)
    _ext.kernels().gemm_stream(y.data_ptr(), x.data_ptr(), w.data_ptr(), 0, m, n, k, 4, 1 if n * k * 2 >= WIDE_NT_MIN_BYTES else 0,
                               float(cap), current_stream())
    return y


class SplitKPartial:
    """Split-K partial sums of ``x @ w.T`` still in the per-stream workspace (not reduced).  Each K
    slice accumulates in f32; the slabs hold it as f16 x 2^-6 by default (csrc/kernels/common.h
    ``DLLM_PART_TYPE``: half the bytes of f32 slabs, 3 significand bits more than the bf16 result).

    Returned by ``linear(..., defer=True)`` when the split-K tiled kernel ran, so the NEXT op can
    fuse the reduction (``ops.fused_add_rms_norm`` -> splitk_add_rms_norm); anything else calls
    :meth:`materialize`.  Valid only until the next tiled GEMM on the same stream reuses the
    workspace -- consume it immediately."""

    __slots__ = ("ws", "splits", "m", "n", "shape", "dtype", "device")

    def __init__(self, ws, splits, m, n, shape, dtype, device):
        self.ws, self.splits, self.m, self.n = ws, splits, m, n
        self.shape, self.dtype, self.device = shape, dtype, device

    def materialize(self) -> torch.Tensor:
        y = torch.empty(self.shape, dtype=self.dtype, device=self.device)
        _ext.kernels().splitk_reduce(y.data_ptr(), self.ws.data_ptr(), 0, self.splits, self.m, self.n,
                                     current_stream())
        return y


def linear(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None, defer: bool = False):
    """y = x w^T (+bias).  ``defer``: may return a :class:`SplitKPartial` (see there)."""
    return _linear(*_sizes(x, w, "linear"), x, w, bias, defer)


def _linear(m: int, n: int, k: int, x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], defer: bool):
    """:func:`linear` of operands whose sizes the caller has compared."""
    kn = knobs.K
    if m <= STREAM_MAX_M and not (defer and n % 128 == 0) and use_stream(m, n, k, x, w, bias):
        return _stream(m, n, k, x, w, bias)
    # decode LM head on gemm_pp with nontemporal weights (236 vs 268 us for gemm_sq at M = 256) --
    # unless comm kernels may hold CUs: beside a 4-workgroup, 20 KiB-LDS receive spinning in
    # another process it took 284 us, gemm_sq 268 either way (bench/debug/lm_head_bench.py,
    # profiles/round5_raw/r5ae_head.txt) -- the pipeline's last stage holds the head
    if bias is None and n > 65536 and 0 < kn.pp_head_min_m <= m <= 256 \
            and (not _comm_cus or kn.head_beside_comm == "pp") and _use_pp(m, n, k, x, w, 1):
        return linear_pp(x, w, splits=1, variant=PP_HEAD_VARIANT)           # decode LM head
    if bias is None and 0 < kn.pp_down_min_k <= k and 225 <= m <= 256 and is_down_proj(n, k) and not _comm_cus \
            and n % 128 == 0 and _use_pp(m, n, k, x, w, 1):
        # long-K decode down projection (70B: K = 28672) on gemm_pp's 128-column tile, K slices filling
        # the CUs, weights nontemporal: 126 vs 135 us for gemm_wide (bench/debug/medium_m_sweep.py)
        s = max(1, min(16, _cus(x.device) // (n // 128)))
        return linear_pp(x, w, splits=s, defer=defer, variant=64 | 2 | 1)
    if bias is None and _use_wide(m, n, k, x, w):
        return linear_wide(x, w, defer=defer)
    if bias is None and _use_pp(m, n, k, x, w, knobs.K.pp_proj_min_m):
        bm = _pf_tile(m, n, k, n, x.device)
        if bm:
            return linear_pf(x, w, bm=bm)
        # medium M (mixed prefill + decode steps, short prompts): split-K tiles fill the CUs
        return linear_pp(x, w, variant=PP_PREFILL_VARIANT, defer=defer)
    return F.linear(x, w, bias)


PP_PREFILL_VARIANT = 64 | 4        # gemm_pp: schedule 2, grouped row-tile order, 256-column tile
PP_GATE_UP_VARIANT = 64 | 2 | 1    # gemm_pp: schedule 2, nontemporal weights, 128-column tile
PP_HEAD_VARIANT = 64 | 2           # gemm_pp: schedule 2, nontemporal weights (read once per step)


def _use_pp(m: int, n: int, k: int, x: torch.Tensor, w: torch.Tensor, min_m: int) -> bool:
    """Prefill-sized GEMM on gemm_pp (knobs.pp_swiglu_min_m / pp_proj_min_m)."""
    return (0 < min_m <= m and n % 256 == 0 and k % 64 == 0 and x.dtype == w.dtype == torch.bfloat16
            and x.is_contiguous() and w.is_contiguous() and m * k * 2 < (1 << 32) and n * k * 2 < (1 << 32))


_ws = {}
_WS_FLOATS = 32 << 20          # 128 MiB of split-K partials per (device, stream)


def _workspace(device: torch.device) -> torch.Tensor:
    key = (device.index or 0, current_stream())
    t = _ws.get(key)
    if t is None:
        t = _ws[key] = torch.empty(_WS_FLOATS, dtype=torch.float32, device=device)
    return t


def slab_space(device: torch.device, read: Optional[SplitKPartial]) -> torch.Tensor:
    """Where a launch that reads ``read`` may leave its own slabs (of up to half the workspace): the start of the workspace, or its
    second half where ``read`` lies at the start."""
    ws = _workspace(device)
    return ws[ws.numel() // 2:] if read is not None and read.ws.data_ptr() == ws.data_ptr() else ws


def wide_bm(m: int) -> int:
    """Row tile of gemm_wide for M rows (mirrors wide_bm in csrc/kernels/gemm_wide.hip)."""
    if m <= 64:
        return 64
    if m <= 128:
        return 128
    if m <= 192:
        return 192
    if m <= 256:
        return 256
    return 192 if m <= 384 else 256


def wide_row_tile(m: int, n: int, k: int, swiglu: bool = False) -> int:
    """Row tile gemm_wide uses for this shape (knobs.wide_small_bm for small split grids, else
    wide_bm): e.g. 128 runs an M = 256 o-projection as 2 row tiles x 4 K slices instead of 1 x 8."""
    kn = knobs.K
    if kn.wide_small_bm and not swiglu and n * k <= kn.wide_small_bm_maxw and kn.wide_small_bm < wide_bm(m):
        return kn.wide_small_bm
    return wide_bm(m)


# CUs a co-resident communication kernel may hold (set by the RCCL transport of a pipeline stage:
# a p2p receive spins on its CUs for as long as its peer has not sent).  gemm_wide's split-K grids
# are sized to leave them free: its workgroups (144 KiB of LDS) cannot share a CU with a kernel
# holding LDS, so a 256-workgroup grid beside 4 such CUs runs a second round for 4 workgroups --
# the down projection took 1.58x its solo time beside a 4-CU receive, the 224 / 240-workgroup
# grids 1.00x (scripts/hwq_probe.py gemms, profiles/round5_comm_queues.md)
_comm_cus = 0
_comm_users = 0


def pf_dynamic() -> bool:
    """gemm_pf's dynamic tile queue: knobs.pf_dynamic "on" / "off" / "auto" (on while comm kernels
    may hold CUs)."""
    v = str(knobs.K.pf_dynamic).strip().lower()
    if v == "auto":
        return _comm_cus > 0
    return v in ("1", "true", "on", "yes")


def reserve_cus_for_comm(n: int) -> None:
    """A transport with spinning comm kernels starts: size gemm_wide grids around ``n`` CUs."""
    global _comm_cus, _comm_users
    _comm_users += 1
    _comm_cus = max(_comm_cus, int(n))


def release_cus_for_comm() -> None:
    global _comm_cus, _comm_users
    _comm_users = max(0, _comm_users - 1)
    if not _comm_users:
        _comm_cus = 0


def wide_splits(m: int, n: int, k: int, swiglu: bool = False, target_wgs: int = 0) -> int:
    """K slices for gemm_wide: about one workgroup per CU, >= 8 K-tiles (512) per slice (with CUs
    reserved for communication: at most one workgroup per remaining CU).  Shorter slices are faster up to 128 rows (2560 x
    2560 in 8 instead of 5, close included, M = 8 / 128, 11.0 / 15.1 -> 9.7 / 14.1 us), but every slice's sum passes through a
    16-bit slab: for results around 0.01, whose slabs lose bits to the small end of f16, the error of the slabs' sum against
    64 bits grew from 2.7e-4 to 3.2e-4 (4 -> 8 slices 2.6e-4 to 3.2e-4)."""
    tiles = (n // 128) * (-(-m // wide_row_tile(m, n, k, swiglu)))
    target = target_wgs or knobs.K.wide_target_wgs
    if _comm_cus:
        s = max(1, (target - _comm_cus) // tiles)
    else:
        s = max(1, round(target / tiles))
    return max(1, min(s, (k // 64) // 8, 16))


WIDE_NT_MIN_BYTES = 12 << 20


def wide_variant(m: int, n: int, k: int, splits: int, bm: int) -> int:
    """gemm_wide's variant for these sizes, number of K slices and row tile: knobs.wide_variant on unsplit grids; on split
    ones knobs.wide_variant_split (weights nontemporal, each byte is read from memory once per step) or the default cache
    policy (1).  Nontemporal weights make the product 2-14 % faster, but from about 64 rows on the launch that sums the slabs
    loses more than that, unless a slice is long.  With its consumer (add + RMS norm), default -> nontemporal, us, M = 16 / 64 /
    128 / 256: 4096 x 4096 12.1 / 13.0 / 15.5 / 19.8 -> 11.3 / 13.2 / 16.2 / 20.1; 6144 x 4096 15.6 / 16.7 / 19.3 / 26.6 -> 14.8 /
    16.8 / 20.0 / 26.9; 4096 x 14336 (28 K-tiles a slice) 25.3 / 26.9 / 31.1 / 41.6 -> 23.4 / 25.9 / 30.5 / 41.5.  Below
    WIDE_NT_MIN_BYTES a small model's weights stay in the 256 MiB Infinity Cache from step to step (1024 x 1024 5.0 -> 5.9 us
    with nt), and on 192-row tiles it is slower throughout (8B down at M = 192: 32.0 -> 34.0 us)."""
    if splits == 1:
        return knobs.K.wide_variant
    if n * k * 2 < WIDE_NT_MIN_BYTES or bm == 192 or (m > 64 and k // 64 < 24 * splits):
        return 1
    return knobs.K.wide_variant_split


def linear_wide(x: torch.Tensor, w: torch.Tensor, splits: int = 0, swiglu: bool = False, defer: bool = False,
                variant: int = -1):
    """Wide-M decode GEMM (csrc/kernels/gemm_wide.hip): 256 x 128 x 64 tiles, 3-deep LDS-DMA pipeline,
    optional split-K and fused SwiGLU epilogue (``w`` = [Wg; Wu]).  ``defer``: may return a
    :class:`SplitKPartial` (no SwiGLU)."""
    k = x.shape[-1]
    n = w.shape[0]
    m = x.numel() // k
    own = splits == 0 and variant < 0
    sq, s, tall, v = _wide_plan(m, n, k, swiglu, splits, variant, _comm_cus, _WIDE_KNOBS(knobs.K))
    if sq:
        return linear_sq(x, w, swiglu=swiglu, defer=defer)
    if not (x.dtype == w.dtype == torch.bfloat16 and x.is_contiguous() and w.is_contiguous()):
        raise ValueError("linear_wide: bf16 contiguous operands")
    if n % 128 or k % 64:
        raise ValueError("linear_wide: N % 128 and K % 64")
    xp, wp = x.data_ptr(), w.data_ptr()
    if m == 1 and own and (s == 1 or (defer and not swiglu)) and one_fits(n, k, s, swiglu) and not (xp | wp) % 16:
        return _one(x, w, s, swiglu, x.shape[:-1], x=x)
    if tall and not (xp | wp) % 16:
        return _duo(x, w, m, n, k, s, tall, swiglu, defer)
    ws = _workspace(x.device)
    stream = current_stream()
    if defer and not swiglu and s > 1:
        se = _ext.kernels().gemm_wide(0, xp, wp, ws.data_ptr(), _WS_FLOATS, m, n, k, s, 2, v, stream)
        return SplitKPartial(ws, se, m, n, (*x.shape[:-1], n), x.dtype, x.device)
    y = torch.empty(*x.shape[:-1], n // 2 if swiglu else n, dtype=x.dtype, device=x.device)
    _ext.kernels().gemm_wide(y.data_ptr(), xp, wp, ws.data_ptr(), _WS_FLOATS, m, n, k, s, 1 if swiglu else 0, v, stream)
    return y


_WIDE_KNOBS = operator.attrgetter("sq", "sq_min_m", "sq_split", "wide_target_wgs", "wide_small_bm", "wide_small_bm_maxw", "wide_variant",
                                  "wide_variant_split", "duo")


@functools.lru_cache(maxsize=1024)         # a pass asks for the same few products in every layer, 6 us each
def _wide_plan(m: int, n: int, k: int, swiglu: bool, splits: int, variant: int, comm_cus: int, kn: tuple):
    """linear_wide's (does gemm_sq take it, K slices, gemm_duo's row tile or 0, variant word) for sizes, a caller's own slices and
    variant, the CUs reserved for communication and what is read of the knobs."""
    own = splits == 0 and variant < 0
    if own and use_sq(m, n, k, swiglu):
        return True, 0, 0, 0
    if n % 128 or k % 64:
        return False, 0, 0, 0
    s = splits or wide_splits(m, n, k, swiglu)
    if s > 1 and s * m * n > _WS_FLOATS and not (m == 1 and own):
        s = max(1, _WS_FLOATS // (m * n))
    bm = wide_row_tile(m, n, k, swiglu)
    v = variant if variant >= 0 else wide_variant(m, n, k, s, bm)
    return False, s, duo_row_tile(m, n, k, s, bm, swiglu) if own else 0, v | bm << 8 if bm != wide_bm(m) else v


def duo_fits(m: int, n: int, k: int, s: int, bm: int, swiglu: bool = False) -> bool:
    """Does gemm_duo serve an [m, k] x [n, k]^T product in ``s`` K slices on row tiles of ``bm`` (gemm_wide's plan, whose bits it has)?  GLUs from 65
    rows on, slabs from 129, or 65 where a slice is 32 K-tiles and more (us with the norm behind them, gemm_wide / this at 65 and 128 rows: 8192 x 28672
    in slices of 112 93.1 / 87.9 and 103.7 / 100.6, 10240 x 8192 of 43 40.7 / 40.2 and 46.2 / 44.5, 8192 x 8192 of 32 39.4 / 39.7 and 42.4 / 42.2,
    4096 x 14336 of 28 29.1 / 28.0 and 33.0 / 32.8, 6144 x 4096 of 13 17.5 / 18.1 and 19.9 / 21.0, 2560 x 7680 of 10 22.8 / 24.1 at 128), where
    the workgroups keep three quarters of the CUs busy: its four waves take twice as long over a K-tile as gemm_wide's eight where
    nothing else bounds them.  us, gemm_wide / this at 256 rows: 2048 x 2048 (64 workgroups) 12.0 / 14.1, 2560 x 2560 (100) 13.8 / 15.6,
    4096 x 2048 (128) 15.0 / 15.5, 8192 x 8192 (256) 45.4 / 43.6."""
    rows = 64 < m <= 256 and s == 1 if swiglu else (128 < m <= 512 or 64 < m <= 128 and k >= 2048 * s) and s > 1
    return (knobs.K.duo and rows and bm in (128, 192, 256) and n % 128 == 0 and k % 64 == 0 and n // 128 * s * -(-m // bm) >= 192
            and m * k * 2 < 1 << 32 and n * k * 2 < 1 << 32)


def duo_row_tile(m: int, n: int, k: int, s: int, bm: int, swiglu: bool = False) -> int:
    """gemm_duo's row tile for a product that gemm_wide would run in ``s`` K slices on row tiles of ``bm``, or 0.  Past 256 rows ``bm`` itself or the
    next taller one whose tiles are one round of the CUs; the slices stay, and with them every bit.  us with the sum and norm
    behind them, gemm_wide on ``bm`` / this, 300 and 512 rows: 4096 x 4096 31.9 / 23.6 (192-row tiles in 3 slices), 28.5 / 27.4 (128, 2); 3072 x 2048 19.4 /
    14.1, 22.6 / 16.5 (192); 3072 x 3072 23.3 / 17.0, 29.8 / 20.4 (192); 2048 x 4096 14.8 / 14.1, 18.1 / 16.6; 2048 x 2048 11.9 / 11.3, 14.6 / 12.7 (192
    and 256 workgroups of 128).  Four row tiles of 128 that leave CUs idle stay there: 2560 x 2560 (240) at 400 / 512 15.8 / 17.5, here 16.4 / 18.8."""
    def ok(t):
        wgs = n // 128 * s * -(-m // t)
        return duo_fits(m, n, k, s, t, swiglu) and not (t == 128 and m > 384 and wgs < 256)

    fits = [t for t in (128, 192, 256) if t >= bm and (t == bm or m > 256) and ok(t)]
    one = [t for t in fits if n // 128 * s * -(-m // t) <= 256]
    return (one or fits or [0])[0]


def _duo(x: torch.Tensor, w: torch.Tensor, m: int, n: int, k: int, s: int, bm: int, swiglu: bool, defer: bool,
         like_pp: bool = False):
    """gemm_duo's launch: the SwiGLU (gemm_wide's bits, ``like_pp``: gemm_pp's), or the slabs' :class:`SplitKPartial` (summed without
    ``defer``)."""
    ws = _workspace(x.device)
    y = torch.empty(*x.shape[:-1], n // 2, dtype=x.dtype, device=x.device) if swiglu else None
    se = _ext.kernels().gemm_duo(y.data_ptr() if swiglu else 0, x.data_ptr(), w.data_ptr(), ws.data_ptr(), ws.numel(), m, n, k, s,
                                 swiglu, bm, current_stream(), like_pp)
    if swiglu:
        return y
    part = SplitKPartial(ws, se, m, n, (*x.shape[:-1], n), x.dtype, x.device)
    return part if defer else part.materialize()


ONE_MAX_WIDTH = 8192               # (csrc/kernels/gemm_one.hip: a row, or its slice, in the registers of four waves)
ONE_MAX_SLABS = 8


def one_fits(n: int, k: int, s: int, swiglu: bool = False) -> bool:
    """Does gemm_one serve one row's [1, k] x [n, k]^T product in ``s`` K slices?  It has gemm_wide's bits and is as fast or faster
    wherever that would run (figures there).  GLUs unsplit: below 171 column tiles the weight-streaming kernel's shorter ones keep more
    CUs busy, us with the add + norm in front, apart / in one launch: 22016 x 4096 (172 tiles) 33.5 / 30.0, 16384 x 3072 (128) 20.6 /
    22.0, 13824 x 2560 (108) 17.1 / 19.1-21.6, 8192 x 2048 (64) 9.6 / 12.6."""
    return (knobs.K.one and n % 128 == 0 and k % 64 == 0 and n * k * 2 < 1 << 32 and -(-(k // 64) // s) * 64 <= ONE_MAX_WIDTH
            and (not swiglu or (s == 1 and n // 128 >= 171)))


def _one(like: torch.Tensor, w: torch.Tensor, s: int, swiglu: bool, lead, x=None, residual=None, part=None, norm_w=None,
         res_out=None, eps: float = 0.0):
    """gemm_one's launch: the finished product of one row, or its :class:`SplitKPartial` (``s`` > 1)."""
    n, k = w.shape
    p = lambda t: 0 if t is None else t.data_ptr()
    nt = 1 if n * k * 2 >= WIDE_NT_MIN_BYTES else 0
    args = (p(x), p(residual), 0 if part is None else part.ws.data_ptr(), 0 if part is None else part.splits, p(norm_w), p(res_out),
            float(eps), current_stream())
    if s > 1:
        ws = slab_space(like.device, part)
        se = _ext.kernels().gemm_one(0, ws.data_ptr(), w.data_ptr(), n, k, s, 2, nt, *args)
        return SplitKPartial(ws, se, 1, n, (*lead, n), like.dtype, like.device)
    y = torch.empty(*lead, n // 2 if swiglu else n, dtype=like.dtype, device=like.device)
    _ext.kernels().gemm_one(y.data_ptr(), 0, w.data_ptr(), n, k, 1, 1 if swiglu else 0, nt, *args)
    return y


def norm_linear(h, residual: torch.Tensor, norm_w: torch.Tensor, eps: float, w: torch.Tensor, swiglu: bool = False):
    """(y, r): r = ``residual`` + ``h`` (None: ``residual``; a :class:`SplitKPartial`: its sum), y = rms_norm(r) * ``norm_w`` times
    w^T (a :class:`SplitKPartial`) or its SwiGLU, in one launch -- one row of a weight that gemm_wide or gemm_one would serve behind a
    norm of its own, with the bits of the two; else None.  ``residual`` is left as it is."""
    k = residual.shape[-1]
    if not (residual.is_cuda and residual.numel() == k and w.dim() == 2 and w.size(1) == k and norm_w.numel() == k
            and k <= ONE_MAX_WIDTH and residual.dtype == w.dtype == norm_w.dtype == torch.bfloat16):
        return None
    n = w.size(0)
    if not _use_wide(1, n, k, residual, w, swiglu):
        return None
    s = wide_splits(1, n, k, swiglu)
    if not one_fits(n, k, s, swiglu) or (s == 1 and not swiglu):
        return None
    part = h if isinstance(h, SplitKPartial) else None
    if part is not None:
        if part.splits > ONE_MAX_SLABS or part.m != 1 or part.n != k or part.device != residual.device:
            return None
    elif h is not None and not (h.shape == residual.shape and h.dtype == residual.dtype and h.is_contiguous() and h.device == residual.device):
        return None
    if w.device != residual.device or norm_w.device != residual.device or not norm_w.is_contiguous() \
            or any(t.data_ptr() % 16 for t in (residual, norm_w, w)) or (part is None and h is not None and h.data_ptr() % 16):
        return None
    res_out = residual if h is None else torch.empty_like(residual)
    y = _one(residual, w, s, swiglu, residual.shape[:-1], None if part is not None else h, residual, part, norm_w,
             None if h is None else res_out, eps)
    return y, res_out


def pp_splits(m: int, n: int, k: int, bn: int = 256, target_wgs: int = 256) -> int:
    """K slices for gemm_pp: about one workgroup per CU (tiles x slices <= target), >= 3 K-tiles
    (192) per slice."""
    tiles = (n // bn) * (-(-m // 256))
    return max(1, min(target_wgs // max(1, tiles), (k // 64) // 3, 32))


def linear_pp(x: torch.Tensor, w: torch.Tensor, splits: int = 0, swiglu: bool = False, defer: bool = False,
              variant: int = 0, duo: bool = False):
    """Ping-pong 256-row-tile GEMM (csrc/kernels/gemm_pp.hip).  ``variant``: bit 0 = 128-column tile
    (else 256), bit 1 = weights nontemporal, bit 2 = grouped row-tile order (large M).  Split-K
    partials are reduced by splitk_reduce(_swiglu), or returned as a :class:`SplitKPartial` with
    ``defer`` (no SwiGLU).  ``duo``: an unsplit SwiGLU on 128-column tiles, weights nontemporal, on gemm_duo where that serves it
    (:func:`duo_fits`), with the same bits."""
    k = x.shape[-1]
    n = w.shape[0]
    m = x.numel() // k
    if not (x.dtype == w.dtype == torch.bfloat16 and x.is_contiguous() and w.is_contiguous()):
        raise ValueError("linear_pp: bf16 contiguous operands")
    bn = 128 if variant & 1 else 256
    if n % bn or k % 64:
        raise ValueError(f"linear_pp: N % {bn} and K % 64")
    s = splits or pp_splits(m, n, k, bn)
    ws = _workspace(x.device)
    if s > 1 and s * m * n > ws.numel():
        s = max(1, ws.numel() // (m * n))
    if duo and swiglu and variant == PP_GATE_UP_VARIANT and s == 1 and duo_fits(m, n, k, s, wide_bm(m), True) and x.data_ptr() % 16 == 0 \
            and w.data_ptr() % 16 == 0:
        return _duo(x, w, m, n, k, s, wide_bm(m), True, False, True)
    stream = current_stream()
    if defer and not swiglu and s > 1:
        se = _ext.kernels().gemm_pp(0, x.data_ptr(), w.data_ptr(), ws.data_ptr(), ws.numel(), m, n, k, s, 2, variant,
                                    stream)
        return SplitKPartial(ws, se, m, n, (*x.shape[:-1], n), x.dtype, x.device)
    y = torch.empty(*x.shape[:-1], n // 2 if swiglu else n, dtype=x.dtype, device=x.device)
    _ext.kernels().gemm_pp(y.data_ptr(), x.data_ptr(), w.data_ptr(), ws.data_ptr(), ws.numel(), m, n, k, s,
                           1 if swiglu else 0, variant, stream)
    return y


def linear_pf(x: torch.Tensor, w: torch.Tensor, swiglu: bool = False, variant: int = 0,
              limit: Optional[float] = None, gelu: bool = False, bm: int = 256,
              bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Persistent prefill GEMM (gemm_pf in csrc/kernels/gemm_pp.hip): schedule 2's ``bm`` x 256 tiles,
    one workgroup per CU walking its tiles with the LDS-DMA pipeline running across tile
    boundaries; optional fused SwiGLU (``w`` = [Wg; Wu], y [M, N / 2]) or -- ``limit`` -- clipped GLU (of the products plus
    ``bias`` [gate | up], where given) or -- ``gelu`` -- gelu_tanh GLU.  ``variant`` 8: nontemporal
    output stores (the default for SwiGLU outputs > 256 MiB).  256-row tiles come from per-XCD device queues while
    knobs.pf_dynamic says so (bit 16 of the launcher's variant); others (``bm``, pf_row_tile) are walked statically, by the CUs
    that communication leaves."""
    k = x.shape[-1]
    n = w.shape[0]
    m = x.numel() // k
    if not (x.dtype == w.dtype == torch.bfloat16 and x.is_contiguous() and w.is_contiguous()):
        raise ValueError("linear_pf: bf16 contiguous operands")
    if n % 256 or k % 64:
        raise ValueError("linear_pf: N % 256 and K % 64")
    glu = swiglu or gelu or limit is not None
    y = torch.empty(*x.shape[:-1], n // 2 if glu else n, dtype=x.dtype, device=x.device)
    dyn = pf_dynamic() and k >= 128 and bm == 256
    if torch.cuda.is_current_stream_capturing():
        # inside a graph: the static tile walk.  A tile queue is per stream and self-resetting, but
        # a replay may run on another stream beside eager launches that use the same queue
        dyn = False
    if dyn:
        variant |= 16                  # per-XCD dynamic tile queues (gemm_pp.hip, DYN)
    _ext.kernels().gemm_pf(y.data_ptr(), x.data_ptr(), w.data_ptr(), m, n, k,
                           4 if gelu else 3 if limit is not None else (1 if swiglu else 0), variant, current_stream(),
                           0.0 if limit is None else float(limit), bm, 0 if bias is None else bias.data_ptr(),
                           _pf_wgs(_cus(x.device)) if _comm_cus and bm != 256 else 0)
    return y


# 256 x 256-tile decode GEMM (gemm_sq.hip) for 128 < M <= 256: a third fewer staged bytes per FLOP
# than the wide kernel's 256 x 128 tile.  Measured (profiles/wide_gemm.md, "256 x 256 tile"): it
# wins only where the grid needs no K split -- the LM head (1.05x) and the 70B MLP gate|up (1.07x);
# split grids (8B qkv / o / gate|up / down) lose 6-20 % to the extra slab traffic.  knobs.sq: roles
# (gate_up, down, proj, head, all) or none; knobs.sq_split also admits split grids; knobs.sq_min_m
# (225: at M = 192 it loses 1-6 %).


def sq_role(n: int, k: int, swiglu: bool) -> str:
    if swiglu:
        return "gate_up"
    if is_down_proj(n, k):
        return "down"
    return "head" if n > 65536 else "proj"


def use_sq(m: int, n: int, k: int, swiglu: bool = False) -> bool:
    kn = knobs.K
    roles = _roles(kn.sq)
    if not roles or not (kn.sq_min_m <= m <= 256) or n % 256 or k % 64:
        return False
    if not kn.sq_split and sq_splits(m, n, k) > 1:
        return False
    return "all" in roles or sq_role(n, k, swiglu) in roles


def sq_splits(m: int, n: int, k: int, target_wgs: int = 256) -> int:
    """K slices for gemm_sq: as many as keep (N / 256) x slices within one workgroup per CU, at
    least 4 K-tiles (256) per slice."""
    tiles = (n // 256) * (-(-m // 256))
    return max(1, min(target_wgs // max(1, tiles), (k // 64) // 4, 16))


def linear_sq(x: torch.Tensor, w: torch.Tensor, splits: int = 0, swiglu: bool = False, defer: bool = False,
              variant: int = -1):
    """256 x 256-tile decode GEMM (csrc/kernels/gemm_sq.hip); split-K partials reduced by
    splitk_reduce(_swiglu), or returned as a :class:`SplitKPartial` with ``defer`` (no SwiGLU)."""
    k = x.shape[-1]
    n = w.shape[0]
    m = x.numel() // k
    if not (x.dtype == w.dtype == torch.bfloat16 and x.is_contiguous() and w.is_contiguous()):
        raise ValueError("linear_sq: bf16 contiguous operands")
    if n % 256 or k % 64:
        raise ValueError("linear_sq: N % 256 and K % 64")
    s = splits or sq_splits(m, n, k)
    ws = _workspace(x.device)
    if s > 1 and s * m * n > ws.numel():
        s = max(1, ws.numel() // (m * n))
    stream = current_stream()
    v = knobs.K.sq_variant if variant < 0 else variant
    if defer and not swiglu and s > 1:
        se = _ext.kernels().gemm_sq(0, x.data_ptr(), w.data_ptr(), ws.data_ptr(), ws.numel(), m, n, k, s, 2, v,
                                    stream)
        return SplitKPartial(ws, se, m, n, (*x.shape[:-1], n), x.dtype, x.device)
    y = torch.empty(*x.shape[:-1], n // 2 if swiglu else n, dtype=x.dtype, device=x.device)
    _ext.kernels().gemm_sq(y.data_ptr(), x.data_ptr(), w.data_ptr(), ws.data_ptr(), ws.numel(), m, n, k, s,
                           1 if swiglu else 0, v, stream)
    return y


def _glu_bias(bias: torch.Tensor, n: int, x: torch.Tensor) -> bool:
    """A bias that gemm_pf's epilogue reads: [gate | up] in bfloat16 on x's device, four columns per load."""
    return (bias.dtype == torch.bfloat16 and bias.dim() == 1 and bias.size(0) == n and bias.is_contiguous()
            and bias.device == x.device and bias.data_ptr() % 8 == 0)


def _linear_glu(x: torch.Tensor, w_gate_up: torch.Tensor, limit: Optional[float],
                bias: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """A GLU of x Wg^T and x Wu^T, W = [Wg; Wu], with the activation in the weight-streaming GEMM's epilogue (up to 64
    rows), in the persistent GEMM's (prompts; the forms that take a ``bias`` [gate | up]) or in the split-K
    reduction (decode): clipped (``limit``) or gelu_tanh (None); None if the shape takes none of them.  The prompt form of a
    bias, 700 / 3000 / 6376 / 12000 rows x 15360 x 2560: 65 / 211 / 434 / 810 us with the gate kernel behind the product,
    53 / 185 / 363 / 680 in its epilogue."""
    m, n, k = _sizes(x, w_gate_up, "linear_glu")
    glu = "gelu" if limit is None else "clipped"
    if m <= STREAM_MAX_M and n % 2 == 0 and use_stream(m, n, k, x, w_gate_up, bias, glu):
        return _stream(m, n, k, x, w_gate_up, bias, glu, 0.0 if limit is None else limit)
    if x.dtype != torch.bfloat16 or n % 256 or (bias is not None and not _glu_bias(bias, n, x)):
        return None
    if not _use_wide(m, n, k, x, w_gate_up) and _use_pp(m, n, k, x, w_gate_up, knobs.K.pp_swiglu_min_m):
        bm = _pf_tile(m, n, k, n // 2, x.device)
        if bm and not (bias is not None and (limit is None or _recorded(x, w_gate_up, bias))):
            return linear_pf(x, w_gate_up, limit=limit, gelu=limit is None, bm=bm, bias=bias)
    if bias is not None:
        return None
    y = linear(x, w_gate_up, defer=True)
    if isinstance(y, SplitKPartial):
        out = torch.empty(*x.shape[:-1], n // 2, dtype=x.dtype, device=x.device)
        st = current_stream()
        if limit is None:
            _ext.kernels().splitk_reduce_gelu(out.data_ptr(), y.ws.data_ptr(), y.splits, y.m, y.n, st)
        else:
            _ext.kernels().splitk_reduce_clipped(out.data_ptr(), y.ws.data_ptr(), y.splits, y.m, y.n, float(limit), st)
        return out
    from .seqmix import clipped_glu, gelu_glu
    return gelu_glu(y) if limit is None else clipped_glu(y, None, limit)


def linear_clipped_glu(x: torch.Tensor, w_gate_up: torch.Tensor, limit: float,
                       bias: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """g sigmoid(1.702 g) (u + 1), g = min(x Wg^T, limit), u = clamp(x Wu^T, -limit, limit) (``bias`` [gate | up] added
    to the products), fused (:func:`_linear_glu`)."""
    return _linear_glu(x, w_gate_up, float(limit), bias)


def linear_gelu_glu(x: torch.Tensor, w_gate_up: torch.Tensor) -> Optional[torch.Tensor]:
    """gelu_tanh(x Wg^T) * (x Wu^T), fused (:func:`_linear_glu`)."""
    return _linear_glu(x, w_gate_up, None)


def linear_swiglu(x: torch.Tensor, w_gate_up: torch.Tensor) -> Optional[torch.Tensor]:
    """silu(x Wg^T) * (x Wu^T) with W = [Wg; Wu] in one launch; None if the shape is not eligible."""
    m, n, k = _sizes(x, w_gate_up, "linear_swiglu")
    kn = knobs.K
    if m <= STREAM_MAX_M and n % 16 == 0 and use_stream(m, n, k, x, w_gate_up, glu="silu"):      # (the SiLU kernels' multiples of 8, at any m)
        return _stream(m, n, k, x, w_gate_up, glu="silu")
    if 0 < kn.pp_gate_up_min_m <= m <= 256 and not _comm_cus and _use_pp(m, n, k, x, w_gate_up, 1):
        # decode gate|up on gemm_pp, unsplit, weights nontemporal, on the column tile that gives one
        # round of CUs / 2 .. CUs tiles: 8B (224 x 128 columns) 62.1 vs 64.1 us for gemm_wide (60.6 on gemm_duo with its bits, which
        # takes these), 70B (224 x 256 columns) 204 vs 259 us for gemm_sq (bench/debug/medium_m_sweep.py --pp)
        cus = _cus(x.device)
        if n % 128 == 0 and cus // 2 <= n // 128 <= cus:
            return linear_pp(x, w_gate_up, splits=1, swiglu=True, variant=PP_GATE_UP_VARIANT, duo=True)
        if n % 256 == 0 and cus // 2 <= n // 256 <= cus:
            return linear_pp(x, w_gate_up, splits=1, swiglu=True, variant=PP_GATE_UP_VARIANT & ~1)
    if _use_wide(m, n, k, x, w_gate_up, swiglu=True):
        return linear_wide(x, w_gate_up, swiglu=True)
    if _use_pp(m, n, k, x, w_gate_up, knobs.K.pp_swiglu_min_m):
        bm = _pf_tile(m, n, k, n // 2, x.device)
        if bm:
            return linear_pf(x, w_gate_up, swiglu=True, bm=bm)
        return linear_pp(x, w_gate_up, swiglu=True, variant=PP_PREFILL_VARIANT)
    return None
