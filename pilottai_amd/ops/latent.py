"""Dispatch of the fp32-residual, latent-attention, grouped-projection and gated-linear-attention kernels (modules _latent and
_latent_linear).

Device tensors run the HIP kernels of csrc/ops/{residual_norm, latent_cache, latent_attention,
grouped_gemm, linear_attention, poly_norm}.hip and raise when the module is missing; CPU tensors run the fp32 references of
ops/reference.py. Every function takes its constants as arguments and works in bf16 or fp32.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import reference as ref
from .kernels import _on_gpu, require_family, require_grouped, require_latent

SCAN_CHUNK = 64  # tokens of a scan item of recurrent layers
SCAN_MIN = 8     # longer portions are scanned in chunks
LATENT_TILES = (1, 2, 3, 4, 6, 8, 12, 16)  # latent widths (in 32s) with MFMA kernels (latent_attention.hip)
ROT_TILES = (1, 2)


def pad_to(n: int, m: int) -> int:
    return (n + m - 1) // m * m


def latent_pad(R: int) -> int:
    """Cached width of an R-wide latent: the smallest width with an MFMA kernel, else whole 32s."""
    need = (R + 31) // 32
    return 32 * next((n for n in LATENT_TILES if n >= need), need)


# ---- fp32 residual stream -------------------------------------------------------------------
def residual_norm(resid: torch.Tensor, eps: float, *, y: Optional[torch.Tensor] = None, partials: int = 1,
                  y_scale: float = 1.0, w_post: Optional[torch.Tensor] = None, emb: Optional[torch.Tensor] = None,
                  ids: Optional[torch.Tensor] = None, emb_add: bool = False, w_next: Optional[torch.Tensor] = None,
                  out: Optional[torch.Tensor] = None, rows: Optional[torch.Tensor] = None, post_groups: int = 1,
                  next_groups: int = 1, mix: Optional[torch.Tensor] = None, hist: Optional[torch.Tensor] = None,
                  live: Optional[torch.Tensor] = None):
    """resid (fp32 [T, D], in place) += norm(y_scale * sum of a token's `partials` rows of y) * w_post
    (w_post None: without the norm), then += emb[ids] (emb_add) or = emb[ids]; out = norm(resid) * w_next (w_next
    None: resid as it is). The norms are of `post_groups` and `next_groups` equal parts of a row. Depth average, with
    mix [n + 1]: resid joins hist (fp32 [n, T, D]) as its last entry, and becomes mix[0] emb[ids] + sum_j mix[j]
    hist[j - 1]. Returns out. `rows`: out row i is row rows[i]'s, and resid and hist keep their values. `live`
    (ints by row, without `rows`): rows from the first one below 0 on are padding and may be left as they were."""
    if _on_gpu(resid):
        require_latent().residual_norm(resid, y, int(partials), float(y_scale), w_post, emb, ids, bool(emb_add),
                                       w_next, out, rows, float(eps), int(post_groups), int(next_groups), mix, hist, live)
        return out
    return ref.residual_norm(resid, eps, y, partials, y_scale, w_post, emb, ids, emb_add, w_next, out, rows, post_groups,
                             next_groups, mix, hist)


# ---- latent cache and attention ---------------------------------------------------------------
def latent_cache(x, nq: int, R: int, r: int, w_q, w_c, cq, pages, Rp: int, positions, slots, cos_sin, eps: float):
    """x [T, nq | R | r ...] -> cq = norm of the first nq columns, and the token's cache row: norm of the
    next R, and the rotated last r (csrc/ops/latent_cache.hip). nq 0: no cq; r 0: no rotated part."""
    if _on_gpu(x):
        require_latent().latent_cache(x, int(nq), int(R), int(r), w_q, w_c, cq, pages, int(Rp), positions, slots,
                                      cos_sin, float(eps))
    else:
        ref.latent_cache(x, nq, R, r, w_q, w_c, cq, pages, Rp, positions, slots, cos_sin, eps)


def latent_attention(out, part_o, part_ml, q, pages, items, n_items, q_start, q_len, ctx_len, block_table,
                     scale: float, window: int, dec_tokens: int, tile_tokens: int, num_seqs: Optional[int] = None,
                     simple: bool = False, expand: Optional["Expanded"] = None, heads: Optional[tuple] = None):
    """Attention of absorbed queries q [T, H, D] over latent pages -> out [T, H, Rp]; `window` 0: none.
    dec_tokens / tile_tokens: the scheduler's items hold at most dec_tokens tokens (split over keys) or
    tile_tokens (csrc/ops/latent_attention.hip). `simple`: the any-size kernel. `expand`: requests of its plan are left out
    here, and their outputs in the heads' own dimensions go to its `out`. `heads` = (W_uv packed by pack_groups, y): y = every head's
    product with W_uv, as head_gemm(out, Rp, W_uv, y, vp) behind this; `out` then holds anything (merge_heads: which sizes)."""
    if expand and expand.window != window:
        raise ValueError(f"a plan for a window of {expand.window} with one of {window}")
    if _on_gpu(q):
        require_latent().latent_attention(out, part_o, part_ml, q, pages, items, n_items, q_start, q_len,
                                          ctx_len, block_table, int(dec_tokens), int(tile_tokens), int(window),
                                          float(scale), bool(simple), expand.plan if expand else [],
                                          expand.tensors() if expand else [], *(expand.sizes if expand else (0, 0)),
                                          *(heads or (None, None)))
    else:
        ref.latent_attention(out, q, pages, q_start, q_len, ctx_len, block_table, scale, window,
                             len(q_len) if num_seqs is None else num_seqs)
        if heads:
            head_gemm(out.view(out.shape[0], -1), out.shape[2], heads[0], heads[1], heads[0].shape[1] * 16 if heads[0].dim() == 5 else heads[0].shape[1])
    return out


# Tokens of a step up to which the heads' products go with the merge. A step of bozupel-base, us apart and so: a decoding row 756, 730, 16 1,805,
# 1,768, 128 after 1,000 tokens 2,455, 2,432, 180 2,720, 2,690, 256 after 2,048 2,572, 2,552; one prompt of 60 tokens 2,055, 2,044, of 120 2,205, 2,195,
# four of 40 2,345, 2,331
MERGE_HEADS_T = 192


def merge_heads(T: int, rank: int, rot: int, vdim: int, dtype) -> bool:
    """Whether latent_attention's `heads` is the faster form for T tokens, and has these (padded) sizes."""
    return T <= MERGE_HEADS_T and dtype == torch.bfloat16 and rank <= 512 and \
        latent_pad(rank) == rank and rot <= 64 and vdim <= 128 and vdim % 16 == 0


# Prompt portions with the keys expanded per head (csrc/ops/latent_expand.h): sizes that have the form, and the most heads (an
# item's heads are units of as many workgroups, 256 of which the launch is sure to have)
EXPAND_SIZES, EXPAND_HEADS = dict(dim=128, vdim=128, rot=64, rank=512), 256
EXPAND_COLS, EXPAND_REQS = 128, 64


def expand_pays(T: int, slots: int) -> bool:
    """Whether a step of T rows has the plan and the launch a layer that the form takes, in an engine of `slots` requests.
    By what a captured step knows, so that its outputs depend on its tokens alone; the plan refuses on the device what does
    not pay (expand_plan_kernel), and then costs 1 to 2 %. From twice as many rows as slots on, at most half of them decode.
    A step of 8 layers of 16 heads, us, without the plan and with it: 256 slots, one prompt of 512 tokens 2,935, 2,655, of
    2,000 4,941, 4,282, 4 of 400 beside 30 decode rows 3,973, 3,796, one of 500 after 700 beside 200 3,623, 3,411; below, 4 of 60
    beside 30 2,521, 2,559, 64 decode rows alone 2,256, 2,285; 16 slots, one of 260 2,574, 2,484."""
    return T >= max(256, 2 * slots)


class ExpandPlan:
    """Which requests of a step of T rows have their keys expanded, decided on the device: [counts, base, form, attention
    items, expansion tiles], and the room for it. `form` [T] is 1 for their rows, `skip` [T] for those and the rows of no request."""

    def __init__(self, meta, T: int, heads: int, window: int):
        dev, S, self.window = meta.q_len.device, meta.q_len.numel(), window
        # as many keys as rows, and the cached ones of a long context
        self.blocks = (T + max(T, 4096)) // 16
        self.slots = max(8, 768 // heads)
        new = lambda *s: torch.empty(*s, dtype=torch.int32, device=dev)  # noqa: E731
        self.form, self.skip = new(T), new(T)
        self.lists = [new(2), new(S), self.form, new(T // EXPAND_COLS + EXPAND_REQS + self.slots, 4),
                      new(self.blocks // 4 + EXPAND_REQS, 4)]
        require_latent().latent_plan(self.lists, meta.q_start, meta.q_len, meta.ctx_len, int(T), int(heads), int(window),
                                     int(self.blocks), int(self.slots), self.skip)


class Expanded:
    """Keys and values of the plan's requests, from their pages, with wk and wv = pack_groups([H, 128, 512]), the heads' rows of
    W_uk and of W_uv; q [T, H (128 + 64)] and out [T, >= H 128] are what latent_attention reads and writes for them."""

    def __init__(self, plan: ExpandPlan, pages, wk, wv, block_table, q, cos_sin, out):
        H, dev = wk.shape[0], pages.device
        new = lambda dt, *s: torch.empty(*s, dtype=dt, device=dev)  # noqa: E731
        self.plan, self.form, self.skip, self.q, self.cos_sin, self.out = plan.lists, plan.form, plan.skip, q, cos_sin, out
        self.sizes, self.window = (plan.blocks, plan.slots), plan.window
        self.kx, self.kr = new(torch.bfloat16, plan.blocks, H, 32, 16, 8), new(torch.bfloat16, plan.blocks, 8, 16, 8)
        self.part_o = new(torch.float32, plan.slots, H, EXPAND_COLS, 128)
        self.part_ml = new(torch.float32, plan.slots, H, EXPAND_COLS, 2)
        require_latent().latent_expand(self.plan, plan.blocks, self.kx, self.kr, pages, wk, wv, block_table)

    def tensors(self):
        return [self.kx, self.kr, self.q, self.cos_sin, self.out, self.part_o, self.part_ml]


# ---- grouped projections ----------------------------------------------------------------------
def pack_groups(w: torch.Tensor, dtype) -> torch.Tensor:
    """[G, N, K] (N % 16 == 0, K % 32 == 0) -> the layout grouped_gemm.hip reads: MFMA fragments in bf16
    ([G, N/16, K/32, 64, 8]), row-major in fp32."""
    G, N, K = w.shape
    w = w.to(dtype)
    if dtype == torch.float32:
        return w.contiguous()
    return w.reshape(G, N // 16, 16, K // 32, 4, 8).permute(0, 1, 3, 4, 2, 5).reshape(G, N // 16, K // 32, 64, 8) \
        .contiguous()


def unpack_groups(wp: torch.Tensor) -> torch.Tensor:
    if wp.dim() == 3:
        return wp
    G, A, S = wp.shape[:3]
    return wp.view(G, A, S, 4, 16, 8).permute(0, 1, 4, 2, 3, 5).reshape(G, A * 16, S * 32)


def interleave_gate_up(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """[G, F, K] x 2 (F % 16 == 0) -> [G, 2F, K], 16 gate rows before the 16 up rows of the same outputs."""
    G, F, K = gate.shape
    return torch.stack([gate.reshape(G, F // 16, 16, K), up.reshape(G, F // 16, 16, K)], 2).reshape(G, 2 * F, K)


def head_gemm(x, x_step: int, w, out, out_step: int, rot: Optional[tuple] = None, gate: Optional[torch.Tensor] = None,
              skip: Optional[torch.Tensor] = None):
    """out[:, g * out_step : + N] = x[:, g * x_step : + K] @ w[g].T for every group g, times sigmoid(gate) (columns as
    out's) if given. rot = (positions, cos_sin, skip, r, rp): beside them, out[:, g * out_step + N : + rp] = x[:, g *
    x_step + skip : + r] rotated by the row's position and padded with zeros. Rows whose entry of `skip` (int32 [T]) is not 0
    stay as they are (on the GPU, bf16)."""
    if _on_gpu(x):
        pos, cs, at, r, rp = rot or (None, None, 0, 0, 0)
        require_grouped().head_gemm(x, int(x_step), w, out, int(out_step), pos, cs, int(at), int(r), int(rp), gate, skip)
    else:
        ref.head_gemm(x, x_step, unpack_groups(w), out, out_step, rot, gate)
    return out


def table_gemm(x, w, out, table, ids, col: int, glu: tuple):
    """out[:, :N] = the gated unit (limit, alpha, bias[, cubic]) of x @ w.T and table[ids, col : col + N]."""
    lim, alpha, bias, cubic = (tuple(glu) + (0.0,))[:4]
    if _on_gpu(x):
        require_grouped().table_gemm(x, w, out, table, ids, int(col), float(lim), float(alpha), float(bias), float(cubic))
    else:
        ref.table_gemm(x, unpack_groups(w)[0], out, table, ids, col, lim, alpha, bias, cubic)
    return out


def table_route(tables, desc, desc_host, ids, slots, T: int, tm: int, order, tiles, n_tiles):
    """Sort every layer's (token, choice) pairs by expert, from the layers' token tables, in one launch
    (grouped_gemm.hip table_route_kernel)."""
    if _on_gpu(ids):
        require_family("latent").table_route(tables, desc, desc_host, ids, slots, int(T), int(tm), order, tiles, n_tiles)
    else:
        ref.table_route(tables, desc_host, ids, slots, T, tm, order, tiles, n_tiles)


def expert_gemm(x, w, out, tiles, n_tiles, order, rows: int, *, x_div: int, out_order: bool, tm: int,
                glu: Optional[tuple] = None, relu2: bool = False, row_w: Optional[torch.Tensor] = None,
                live: Optional[torch.Tensor] = None, always: int = 0):
    """Rows sorted by expert: out row = x row @ w[expert].T; glu = (limit, alpha, bias[, cubic]): the gated
    pair of interleave_gate_up weights, min(g, limit) sigmoid(alpha (g + cubic g^3)) (clamp(u) + bias); relu2: the
    square of what is positive. x row = order[p] // x_div (0: p), out row = order[p] if out_order. row_w (with glu
    and x_div): x's row is multiplied by row_w[order[p]]. live (ints by position): tiles of 256 rows that begin at a
    position below 0 may be left out. always: the last groups, so many, hold every row (where their tiles are taken from matters to
    the time alone)."""
    lim, alpha, bias, cubic = (tuple(glu) + (0.0,))[:4] if glu else (0.0, 0.0, 0.0, 0.0)
    if _on_gpu(x):
        require_grouped().expert_gemm(x, w, out, tiles, n_tiles, order, int(rows), int(x_div), bool(out_order), int(tm),
                                      1 if glu is not None else 2 if relu2 else 0, float(lim), float(alpha), float(bias), float(cubic),
                                      row_w, live, int(always))
    else:
        ref.expert_gemm(x, unpack_groups(w), out, tiles, n_tiles, order, x_div, out_order, glu, relu2, row_w)
    return out


# ---- gated linear attention -------------------------------------------------------------------
def linear_attention(x, y, state, a2, bias, q_start, q_len, ctx_len, state_slot, scan_items, n_scan, cols, q_scale: float,
                     inv_tau: float, scan_min: int = SCAN_MIN, num_seqs: Optional[int] = None):
    """The recurrence S <- diag(e^g) S + k v^T, y = S^T q q_scale over the step's portions, from and to the sequences'
    state slots, with g = logsigmoid(a2 a + bias) inv_tau for every key channel (csrc/ops/linear_attention.hip). cols:
    columns of x where q, k, v and the low-rank inputs a start. state fp32 [slots, H, V, N], a2 [H N, rank]."""
    H, V, N = state.shape[1:]
    if not _on_gpu(x):
        ref.linear_attention(x, y, state, a2, bias, q_start, q_len, ctx_len, state_slot, cols, q_scale, inv_tau,
                             len(q_len) if num_seqs is None else num_seqs)
        return y
    T = x.shape[0]
    seqs = min(T, q_len.numel())
    items = 0 if T <= scan_min else min(scan_items.shape[0], T // SCAN_CHUNK + min(seqs, T // (scan_min + 1)) + 1)
    chunked = items if x.dtype == torch.bfloat16 else 0
    new = lambda dt, *s: torch.empty(*s, dtype=dt, device=x.device)  # noqa: E731
    rows = T if chunked else 0
    qd, kd, sc = (new(x.dtype, 2, rows, H, n) for n in (N, N, SCAN_CHUNK))
    require_family("latent_linear").linear_attention(
        x, y, state, new(torch.float32, chunked, H, V, N), qd, kd, sc, new(torch.float32, chunked, H, N), a2, bias, q_start, q_len,
        ctx_len, state_slot, scan_items, n_scan, int(chunked), int(seqs), [int(c) for c in cols], float(q_scale), float(inv_tau),
        int(scan_min))
    return y


# ---- activations ------------------------------------------------------------------------------
def poly_norm(z, n: int, act, eps: float):
    """z[:, :n] = a z / rms(z) + b z^2 / rms(z^2) + c z^3 / rms(z^3) + e with act = (a, b, c, e), in place; z's other
    columns are cleared (csrc/ops/poly_norm.hip)."""
    if _on_gpu(z):
        require_family("latent_linear").poly_norm(z, int(n), act, float(eps))
    else:
        ref.poly_norm(z, n, act, eps)
    return z
