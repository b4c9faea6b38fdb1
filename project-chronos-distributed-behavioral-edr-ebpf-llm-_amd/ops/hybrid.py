"""Ops of the hybrid decoders (recurrent matrix-memory layers, linear-state recurrences, latent and windowed
attention, mixtures of experts, layer and RMS norms on a float32 residual stream): gfx950 HIP kernels on the GPU
(csrc/hybrid/*.hip), the PyTorch references of :mod:`.hybrid_ref` on the CPU.

As everywhere in :mod:`chronos.ops` a GPU tensor never falls back silently: it goes to ``torch.ops.chronos.hy_*`` or
raises.  ``CHRONOS_HYBRID_REF=1`` is a bring-up switch that runs the PyTorch references on GPU tensors (it syncs with
the host and cannot be captured into a graph).

Activations are bfloat16 or float32 (one build serves both: the kernels are instantiated for the two); the residual
stream, norms, recurrent state, gates, router and attention scores are float32 in either mode.
"""
from __future__ import annotations

import os
import sys

import torch

from . import gemm as _gemm, hybrid_ref as ref
from .hybrid_ref import ACT_GELU, ACT_GLU, ACT_RELU2  # noqa: F401

_pkg = sys.modules[__package__]
_REF_ON_GPU = os.environ.get("CHRONOS_HYBRID_REF", "0") not in ("", "0")


def _gpu(t: torch.Tensor) -> bool:
    return t.is_cuda and not _REF_ON_GPU


_lib_loaded = False


def load() -> None:
    """Load (building in-tree if stale) the hybrid kernel library; raises on failure."""
    global _lib_loaded
    if not _lib_loaded:
        from ..native import hybrid_lib

        hybrid_lib()
        _lib_loaded = True


def _k():
    if not _lib_loaded:
        load()
    return torch.ops.chronos


def _f32(act_dtype) -> bool:
    return act_dtype == torch.float32


class JoinedRows:
    """scale_add_rms_norm(y, x, w, ..) for the product behind it: a launch less where every workgroup of that product makes the rows itself.
    ``stream()`` is the float32 residual behind the join, ``rows()`` its rows in the activation dtype; both join first, in x, if no product has."""

    def __init__(self, y, x, w, alpha: float, eps: float):
        self.y, self.x, self.w, self.alpha, self.eps, self.done = y, x, w, alpha, eps, False
        self.h = torch.empty(x.shape, dtype=torch.bfloat16, device=x.device)

    @staticmethod
    def serves(y, x) -> bool:
        return _gpu(x) and type(y) is torch.Tensor and type(x) is torch.Tensor and x.dim() == 2 and _gemm.join_rows_ok(*x.shape) and \
            y.is_contiguous() and x.is_contiguous() and (y.dtype == torch.float32 if y.dim() == 3 else y.dtype == torch.bfloat16 and y.shape == x.shape) and \
            not (torch.is_grad_enabled() and (y.requires_grad or x.requires_grad))

    def rows(self):
        if not self.done:
            self.h = scale_add_rms_norm(self.y, self.x, self.w, self.alpha, self.eps, torch.bfloat16)
            self.done = True
        return self.h

    def stream(self):
        self.rows()
        return self.x

    def product(self, w, kind: int, n0: int = 0, nf: int = 0, bias=None, limit: float = 0.0, slope: float = 0.0, shift: float = 0.0):
        """(product, its float32 rows) as _gemm.join_config's kinds, or None."""
        cfg = 0 if self.done else _gemm.join_config(self.h, w, kind, n0)
        if not cfg:
            return None
        out, few, self.x = _gemm._k().gemm_join(self.y, self.x, self.w, self.alpha, self.eps, self.h, w, cfg, 3 if kind == 2 else 0, n0, nf, bias, limit, slope, shift)
        self.done = True
        return out, few


def matmul(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None = None) -> torch.Tensor:
    """x @ w.T (+ bias): the framework's routed projection GEMMs for bfloat16, the library's float32 GEMM otherwise.
    A biased projection is one library GEMM whose epilogue adds the bias (in the activation dtype, like w) to the
    float accumulator before the rounding."""
    if type(x) is JoinedRows:
        y = x.product(w, 1) if bias is None else None
        if y is not None:
            return y[0]
        x = x.rows()
    if bias is not None:
        return torch.addmm(bias, x, w.t())
    if x.dtype == torch.bfloat16:
        return _pkg.linear(x, w)
    return torch.matmul(x, w.t())


def matmul_f32(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w.T as float32: the product's sums themselves where the framework's kernels take it, else the rounded product's values."""
    if _gpu(x) and x.dtype == torch.bfloat16:
        y = _gemm.product_f32(x, w)
        if y is not None:
            return y
    return matmul(x, w).float()


def matmul_slices(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w.T for add_layer_norm or scale_add_rms_norm, which also take a product of few rows as the float32 slices [S, T, n] of its split and
    sum and round them themselves, a launch less."""
    if _gpu(x) and x.dtype == torch.bfloat16:
        y = _gemm.product_slices(x, w)
        if y is not None:
            return y
    return matmul(x, w)


def matmul_parts(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """matmul_slices for any number of rows."""
    if _gpu(x) and x.dtype == torch.bfloat16 and x.shape[0] > 64:
        y = _gemm.product_parts(x, w)
        return matmul(x, w) if y is None else y
    return matmul_slices(x, w)


def embed_rows(ids, table, act_dtype, scale: float = 1.0, emit: bool = True):
    """(float32 residual rows times ``scale``, the same rows in the activation dtype or None when ``emit`` is off)."""
    if _gpu(table):
        if emit and not _f32(act_dtype):
            return _k().hy_embed_both(ids, table, scale)
        x = _k().hy_embed(ids, table, scale)
        return x, (x if emit else None)
    return ref.embed_rows(ids, table, act_dtype, scale, emit)


def embed_start(ids, table, act_dtype, scale: float, emit: bool, pos, q_start):
    """embed_rows and, behind them, pos at every sequence's first token (int32 [B]; sequences without tokens: at the next one's, or the last)."""
    if _gpu(table) and ids.numel() and pos.numel() == ids.numel() and all(t.dtype == torch.int32 and t.is_contiguous() for t in (pos, q_start)):
        both = emit and not _f32(act_dtype)
        x, h, pos0 = _k().hy_embed_start(ids, table, scale, both, pos, q_start)
        return x, (h if both else x if emit else None), pos0
    pos0 = pos.index_select(0, q_start[:-1].long().clamp(max=max(0, pos.numel() - 1)))
    return (*embed_rows(ids, table, act_dtype, scale, emit), pos0)


def layer_norm(x, w, eps: float, act_dtype, rows=None):
    """``rows`` (int64): of these rows of x only."""
    if _gpu(x):
        return _k().hy_layer_norm(x, w, eps, _f32(act_dtype), rows)
    return ref.layer_norm(x if rows is None else x.index_select(0, rows), w, eps, act_dtype)


def add_layer_norm(y, x, w, eps: float, act_dtype):
    """x (float32 residual, in place) <- x + layer_norm(y) * w; returns the updated rows in the activation dtype
    (x itself when that is float32).  y: rows, or on the GPU a product's slices (matmul_slices)."""
    if _gpu(x):
        h = _k().hy_add_layer_norm(y, x, w, eps, _f32(act_dtype))
        return x if _f32(act_dtype) else h
    return ref.add_layer_norm(y, x, w, eps, act_dtype)


def rowdot(h, w, bias=None):
    if type(h) is JoinedRows:
        h = h.rows()
    if _gpu(h):
        return _k().hy_rowdot(h, w, bias)
    return ref.rowdot(h, w, bias)


def matmul_rowdot(h, w, w_few, bias=None, joined=None):
    """(h @ w.T, rowdot(h, w_few, bias)); ``joined`` (whole, n0, nf): both matrices' rows one behind the other, which few rows of h take in
    one launch."""
    if type(h) is JoinedRows:
        y = h.product(joined[0], 0, joined[1], joined[2], bias) if joined is not None else None
        if y is not None:
            return y
        h = h.rows()
    if joined is not None and _gpu(h) and h.dtype == torch.bfloat16:
        y = _gemm.product_rows(h, *joined, bias)
        if y is not None:
            return y
    return matmul(h, w), rowdot(h, w_few, bias)


def act_inplace(x, kind: int):
    if _gpu(x):
        _k().hy_act(x, kind)
        return x
    return ref.act_inplace(x, kind)


def matmul_act(x, w, kind: int):
    """act_inplace(x @ w.T, kind), in the product's epilogue where that is faster (the activation then reads the unrounded product)."""
    if _gpu(x) and x.dtype == torch.bfloat16 and kind in (ACT_RELU2, ACT_GELU):
        y = _gemm.product_act(x, w, 4 if kind == ACT_RELU2 else 5)
        if y is not None:
            return y
    return act_inplace(matmul(x, w), kind)


def matmul_glu(x, w, limit: float, slope: float, shift: float, act_dtype):
    """glu(x @ w.T, ...), w = [gate; up], in the product's epilogue where that is faster (the unit then reads the unrounded product)."""
    if type(x) is JoinedRows:
        y = x.product(w, 2, 0, 0, None, limit, slope, shift) if act_dtype == torch.bfloat16 else None
        if y is not None:
            return y[0]
        x = x.rows()
    if _gpu(x) and x.dtype == torch.bfloat16 and act_dtype == torch.bfloat16:
        y = _gemm.product_act(x, w, 3, limit, slope, shift)
        if y is not None:
            return y
    return glu(matmul(x, w), limit, slope, shift, act_dtype)


def mlstm_scan(proj, gate_pre, q_start, pos0, slots, S, n, m, H: int, D: int, Dv: int, cap: float, max_q: int = 0):
    """``max_q``: the most tokens any sequence brings in this step (picks the kernel, any value gives the same
    results up to rounding; 0 = unknown)."""
    if _gpu(proj):
        return _k().hy_mlstm_scan(proj, gate_pre, q_start, pos0, slots, S, n, m, H, D, Dv, cap, max_q)
    return ref.mlstm_scan(proj, gate_pre, q_start, pos0, slots, S, n, m, H, D, Dv, cap)


def mlstm_out(o, proj, g_off: int, norm_w, eps: float, act_dtype):
    if _gpu(o):
        return _k().hy_mlstm_out(o, proj, g_off, norm_w, eps, _f32(act_dtype))
    return ref.mlstm_out(o, proj, g_off, norm_w, eps, act_dtype)


def latent_prep(q, dkv, pos, tok_seq, block_table, w_norm, eps: float, cos_sin, dims: int, rank: int, cache, qa=None,
                interleaved: bool = False, lat=None, kr=None) -> None:
    """``lat`` [T, rank] and ``kr`` [T, R]: also get the cached rows' two parts.  ``qa``: where the rotated query columns go (its last R columns per head; default: in place); ``interleaved``:
    neighbouring columns form the rotated pairs.  q and dkv may be column ranges of one wider projection; dkv None: the
    cache is another layer's and only the queries are rotated."""
    if _gpu(q):
        _k().hy_latent_prep(q, dkv, pos, tok_seq, block_table, w_norm, eps, cos_sin if dims else None, dims, rank, cache,
                            qa, interleaved, lat, kr)
    else:
        ref.latent_prep(q, dkv, pos, tok_seq, block_table, w_norm, eps, cos_sin, dims, rank, cache, qa, interleaved)
        if lat is not None:
            rows = cache[block_table[tok_seq.long(), (pos // cache.shape[1]).long()].long(), (pos % cache.shape[1]).long()]
            lat.copy_(rows[:, :rank])
            kr.copy_(rows[:, rank:])


def head_matmul(a, w, out=None, gate_src=None, g_off: int = -1):
    """Per-head products a[t, h] @ w[h].T (a [T, H, K], w [H, N, K]) into ``out`` [T, H, N] (a view with wider rows is
    fine), optionally times sigmoid of H N gate columns."""
    if _gpu(a):
        if out is None:
            out = torch.empty(a.shape[0], a.shape[1], w.shape[1], device=a.device, dtype=a.dtype)
        _k().hy_head_matmul(a, w, out, gate_src, g_off)
        return out
    return ref.head_matmul(a, w, out, gate_src, g_off)


def latent_attention(qa, cache, block_table, q_start, pos, gate, scale: float, rank: int, act_dtype, max_q: int,
                     window: int = 0, two_term: bool = False, sink=None):
    """``max_q``: the most tokens any sequence brings in this step (sizes the launch grid).  ``window`` > 0: a query
    sees only the last ``window`` positions.  ``two_term``: the matrix-core kernel feeds every softmax weight as a sum
    of two bfloat16 terms (float32 weights to about 2^-17).  ``sink`` f32 [H]: joins the softmax denominator."""
    if _gpu(qa):
        return _k().hy_latent_attention(qa, cache, block_table, q_start, pos, gate, scale, rank, max_q, window, two_term, sink)
    return ref.latent_attention(qa, cache, block_table, q_start, pos, gate, scale, rank, act_dtype, window, sink)


def latent_expanded_ok(D: int, R: int, Dv: int) -> bool:
    return _k().hy_latent_expanded_ok(D, R, Dv)


def latent_expanded(q, kv, kr, q_start, gate, gate_src, g_off: int, sink, scale: float, max_q: int, window: int = 0, out=None):
    """Latent attention of sequences that all start at position 0, keys and values written out: q [T, H, D + R] rotated, kv
    [T, H, D + Dv], kr [T, R] the shared rotated keys (q, kr and ``out`` [T, H, Dv] may be column ranges of wider rows); ``gate``,
    ``sink`` as in latent_attention, ``gate_src`` columns as in head_matmul.  On the GPU only (bfloat16)."""
    if out is None:
        out = torch.empty(*q.shape[:2], kv.shape[2] - q.shape[2] + kr.shape[1], device=q.device, dtype=q.dtype)
    _k().hy_latent_expanded(q, kv, kr, q_start, gate, gate_src, g_off, sink, out, scale, max_q, window)
    return out


def moe_route(h, w_router, correction, top: int):
    if _gpu(h):
        return _k().hy_moe_route(h, w_router, correction, top)
    return ref.moe_route(h, w_router, correction, top)


def moe_ffn(h, idx, wt, w_up, w_down, act: int, act_dtype):
    if _gpu(h):
        return _k().hy_moe_ffn(h, idx, wt, w_up, w_down, act)
    return ref.moe_ffn(h, idx, wt, w_up, w_down, act, act_dtype)


# ---- post-norm residual stream, clamped GLU, windowed attention with sinks, linear-state recurrences ---------------


def rms_norm(x, w, eps: float, act_dtype, groups: int = 1, rows=None):
    """``groups`` > 1: every one of that many equal parts of a row is divided by its own root mean square.  ``rows`` (int64): of these
    rows of x only."""
    if _gpu(x):
        if groups > 1:
            return _k().hy_sandwich_join(None, None, x, None, w, None, None, groups, eps, _f32(act_dtype), False, True, rows)
        return _k().hy_rms_norm(x, w, eps, _f32(act_dtype), rows)
    return ref.rms_norm(x if rows is None else x.index_select(0, rows), w, eps, act_dtype, groups)


def scale_add_rms_norm(y, x, w, alpha: float, eps: float, act_dtype):
    """x (float32 residual, in place) <- rms_norm(alpha * x + y) * w; returns the updated rows in the activation
    dtype (x itself when that is float32)."""
    if _gpu(x):
        h = _k().hy_scale_add_rms_norm(y, x, w, alpha, eps, _f32(act_dtype))
        return x if _f32(act_dtype) else h
    return ref.scale_add_rms_norm(y, x, w, alpha, eps, act_dtype)


def glu(gu, limit: float, slope: float, shift: float, act_dtype):
    if _gpu(gu):
        return _k().hy_glu(gu, limit, slope, shift)
    return ref.glu(gu, limit, slope, shift, act_dtype)


def window_prep(qkv, H: int, G: int, D: int, Dv: int, v_first, lam, pos, tok_seq, block_table, q_norm, k_norm,
                eps: float, cos_sin, dims: int, kc, vc, emit_v: bool, v_off: int = -1, v_cos_sin=None, q_temp=None, ks=None):
    """``v_off`` >= 0: the column of qkv where the values start (default: after the keys); ``v_cos_sin``: a rotation
    table over all Dv columns that the values pass before they are cached; ``q_temp`` f32 [P]: a factor on the queries by
    position; ``ks`` (kc None): keys are values over their root mean square, only the factor is cached."""
    if _gpu(qkv):
        v = _k().hy_window_prep(qkv, H, G, D, Dv, v_first, lam, pos, tok_seq, block_table, q_norm, k_norm, eps, cos_sin,
                                dims, kc, vc, emit_v, v_off, v_cos_sin, q_temp, ks)
        return v if emit_v else None
    return ref.window_prep(qkv, H, G, D, Dv, v_first, lam, pos, tok_seq, block_table, q_norm, k_norm, eps, cos_sin,
                           dims, kc, vc, emit_v, v_off, v_cos_sin, q_temp, ks)


def pool_blocks(kc, vc, kp, vp, block_table, q_start, pos0, pool: int, max_q: int) -> None:
    """Means of the keys and values of the blocks of ``pool`` positions that this step's tokens complete, into the
    pooled caches.  ``max_q``: the most tokens any sequence brings in this step (sizes the launch grid)."""
    if _gpu(kc):
        _k().hy_pool_blocks(kc, vc, kp, vp, block_table, q_start, pos0, pool, max_q)
    else:
        ref.pool_blocks(kc, vc, kp, vp, block_table, q_start, pos0, pool)


def window_attention(qkv, kc, vc, block_table, q_start, pos, sink, gate, scale: float, window: int, keep_first: int,
                     H: int, act_dtype, max_q: int, chunk: int = 0, pool: int = 0, kp=None, vp=None, v_cos_sin=None,
                     g_off: int = -1, ks=None, out=None):
    """``max_q``: the most tokens any sequence brings in this step (sizes the launch grid).  ``chunk`` > 0: keys
    outside the query's own chunk of that many positions are hidden.  ``pool`` > 0: the pooled pairs of the blocks
    that lie wholly before a query's window join its softmax.  ``v_cos_sin`` [P, Dv]: every head's output is turned
    back by the query's position (the values were cached rotated); ``g_off`` >= 0: the output is multiplied element by
    element with sigmoid of qkv[:, g_off : g_off + H Dv].  The matrix-core kernel does both in its epilogue.
    ``ks`` f32 [NB, BS, G] (kc None): key j is value j times its factor, one cached row serves both.  ``out``: where the
    output goes, [T, H Dv] columns of wider rows (not with v_cos_sin or g_off)."""
    if _gpu(qkv):
        o = _k().hy_window_attention(qkv, kc, vc, block_table, q_start, pos, sink, gate, scale, window, keep_first,
                                     chunk, H, max_q, pool, kp if pool else None, vp if pool else None, v_cos_sin,
                                     g_off, ks, out)
        return o if out is None else out
    o = ref.window_attention(qkv, kc, vc, block_table, q_start, pos, sink, gate, scale, window, keep_first, H,
                             act_dtype, chunk, pool, kp, vp, ks)
    if v_cos_sin is not None or g_off >= 0:
        o = ref.unrotate_gate(o, pos, v_cos_sin, qkv if g_off >= 0 else None, g_off, H, vc.shape[3], act_dtype)
    if out is not None:
        out.copy_(o)
        return out
    return o


def short_conv(x, w, tok_seq, q_start, pos0, slots, hist, silu: bool = True, bias=None, x_off: int = 0, max_q: int = 0):
    """``max_q``: the most tokens any sequence brings in this step (with 1 the history is rewritten in the same pass; any value gives the
    same results; 0 = unknown)."""
    if _gpu(x):
        return _k().hy_short_conv(x, w, tok_seq, q_start, pos0, slots, hist, silu, bias, x_off, max_q)
    return ref.short_conv(x, w, q_start, pos0, slots, hist, silu, bias, x_off)


def delta_prep(y, ab, a_log, HK: int, H: int, D: int, q_mul: float):
    if _gpu(y):
        return _k().hy_delta_prep(y, ab, a_log, HK, H, D, q_mul)
    return ref.delta_prep(y, ab, a_log, HK, H, D, q_mul)


def decay_pow(z, inv_tau: float):
    if _gpu(z):
        _k().hy_decay_pow(z, inv_tau)
        return z
    return ref.decay_pow(z, inv_tau)


def low_rank_decay(a, w, b, inv_tau: float):
    """sigmoid(b + a @ w) ** inv_tau, float32: a [T, rank], w [rank, C], b [C]."""
    if _gpu(a) and w.shape[1] % 4 == 0:
        return _k().hy_low_rank_decay(a, w, b, inv_tau)
    return decay_pow(torch.addmm(b, a, w), inv_tau)


def linear_scan(proj, q_off: int, k_off: int, v_off: int, qscale, kscale, q_mul: float, decay, beta, q_start, pos0,
                slots, S, HK: int, H: int, D: int, Dv: int, vscale=None, max_q: int = 0, tiles_mb: int = 512):
    """``max_q``: the most tokens any sequence brings in this step (picks the kernel, any value gives the same
    results up to rounding; 0 = unknown).  ``tiles_mb``: scratch that the call may take for its chunks' tiles, for as long as it runs (28 to 32 KB per chunk and head;
    chunks whose tiles need more make them on their way)."""
    if _gpu(proj):
        return _k().hy_linear_scan(proj, q_off, k_off, v_off, qscale, kscale, q_mul, decay, beta, q_start, pos0, slots,
                                   S, HK, H, D, Dv, vscale, max_q, tiles_mb)
    return ref.linear_scan(proj, q_off, k_off, v_off, qscale, kscale, q_mul, decay, beta, q_start, pos0, slots, S, HK,
                           H, D, Dv, vscale)


def rows_step_pays(B: int, H: int, D: int, Dv: int, rank: int) -> bool:
    """rows_step or the launches that it stands for?  Every workgroup, one of a row and head, multiplies its head's decays out itself: few of them wait less for
    it than a launch takes, many pay for it from 100 MB of its weights between them on; and a lane of 256 x 256 states does not have the registers.  us, launches and one: 128 x 128, 32 heads, 1, 64
    and 128 rows: rank 16 10.0 and 6.6, 57 and 53, 97 and 94; 128 22 and 10, 72 and 68, 111 and 137; 256 36 and 13, 90 and 112, 132 and 216.  256 x 256, rank 16, 1 row of 4
    heads 10.1 and 13.5, 64 of 16 105 and 118; rank 128 22 and 17, 120 and 153.  Table: profiles/decode_forms.json, which tests/test_measured_rules.py
    replays."""
    if D == 256 and Dv > 128:
        return 64 <= rank <= 256 and B * H <= 400
    return rank <= 32 or rank <= 256 and B * H * rank * D <= (34_000_000 if B * H <= 2048 else 27_000_000)


def one_step_ok(proj, max_q: int, D: int, Dv: int, heads_per_key: int, *operands) -> bool:
    """May a recurrent mixer's part between its projections run as one launch (delta_step, rows_step, mlstm_step)?  For decode rows, max_q 1; ``operands``:
    what it reads 16 bytes at a time."""
    if max_q != 1 or not _gpu(proj) or proj.dtype != torch.bfloat16 or not proj.is_contiguous() or any(t.data_ptr() % 16 for t in (proj, *operands)):
        return False
    return _k().hy_state_mix_ok(D, Dv, heads_per_key, proj.shape[1])


def delta_step(proj, taps, ab, a_log, q_start, pos0, slots, hist, S, HK: int, H: int, D: int, Dv: int, q_mul: float, g_off: int, w, eps: float):
    """short_conv, delta_prep, linear_scan and head_norm_gate (SiLU gate) of q | k | v columns at 0 and a gate at g_off, 4 taps, where one_step_ok."""
    return _k().hy_delta_step(proj, taps, ab, a_log, q_start, pos0, slots, hist, S, HK, H, D, Dv, q_mul, g_off, w, eps)


def rows_step(proj, low, w2, b2, inv_tau: float, q_start, pos0, slots, S, H: int, D: int, Dv: int, q_mul: float, g_off: int, w, eps: float):
    """low_rank_decay, linear_scan and head_norm_gate (SiLU gate) of q | k | v columns at 0 and a gate at g_off, where one_step_ok."""
    return _k().hy_rows_step(proj, low, w2, b2, inv_tau, q_start, pos0, slots, S, H, D, Dv, q_mul, g_off, w, eps)


def mlstm_step(proj, gate_pre, q_start, pos0, slots, S, n, m, H: int, D: int, Dv: int, cap: float, g_off: int, w, eps: float):
    """mlstm_scan and mlstm_out, where one_step_ok."""
    return _k().hy_mlstm_step(proj, gate_pre, q_start, pos0, slots, S, n, m, H, D, Dv, cap, g_off, w, eps)


def head_norm_gate(o, src, g_off: int, w, eps: float, silu_gate: bool, act_dtype):
    if _gpu(o):
        return _k().hy_head_norm_gate(o, src, g_off, w, eps, silu_gate, _f32(act_dtype))
    return ref.head_norm_gate(o, src, g_off, w, eps, silu_gate, act_dtype)


def moe_route_topk(h, w_router, bias, top: int):
    if _gpu(h):
        return _k().hy_moe_route_topk(h, w_router, bias, top)
    return ref.moe_route_topk(h, w_router, bias, top)


def moe_glu_row_order(F: int) -> torch.Tensor:
    """Row order of a gated expert's [2F, d] gate-then-up matrix for the grouped MFMA path (F % 128 == 0): every
    128-row tile holds, for each of its two 64-row halves, 32 gate rows followed by the 32 up rows of the same
    outputs, so that a lane's accumulators hold a gate value and its up value."""
    n = torch.arange(2 * F)
    tile, local = n // 128, n % 128
    half, s, j = local // 64, (local % 64) // 16, local % 16
    out_col = tile * 64 + half * 32 + (s % 2) * 16 + j
    return out_col + (s >= 2) * F


def moe_glu_ffn(h, idx, wt, w_gu, w_down, limit: float, slope: float, shift: float, act_dtype, tiled: bool = False):
    """``tiled``: every expert's rows of w_gu are in :func:`moe_glu_row_order` (bfloat16 on the GPU, d and F on the
    128 grid): prompt-sized batches then run as grouped matrix-core GEMMs."""
    if _gpu(h):
        return _k().hy_moe_glu_ffn(h, idx, wt, w_gu, w_down, limit, slope, shift, tiled)
    if tiled:
        w_gu = w_gu[:, torch.argsort(moe_glu_row_order(w_gu.shape[1] // 2)).to(w_gu.device)]
    return ref.moe_glu_ffn(h, idx, wt, w_gu, w_down, limit, slope, shift, act_dtype)


# ---- pre-norm residual stream, per-layer token input, state-space and gated linear recurrences, grouped router ---


def add_rms_norm(y, x, w_out, eps: float, act_dtype, y2=None, gate2=None, w_y=None, emit: bool = True):
    """x (float32 residual, in place) <- x + v, v = y (+ sigmoid(gate2) y2), scaled to unit RMS and
    times w_y when that is given.  Returns in the activation dtype rms_norm(x) * w_out, or the updated rows
    themselves when w_out is None (x itself for float32), or None when ``emit`` is off."""
    if _gpu(x):
        h = _k().hy_add_rms_norm(y, x, w_out, eps, _f32(act_dtype), y2, gate2, w_y, emit)
        if not emit:
            return None
        return x if (w_out is None and _f32(act_dtype)) else h
    return ref.add_rms_norm(y, x, w_out, eps, act_dtype, y2, gate2, w_y, emit)


def token_gate(a, ids, table, col0: int, act_dtype):
    if _gpu(a):
        return _k().hy_token_gate(a, ids, table, col0)
    return ref.token_gate(a, ids, table, col0, act_dtype)


def ssm_prep(dt_pre, a_log):
    if _gpu(dt_pre):
        return _k().hy_ssm_prep(dt_pre, a_log)
    return ref.ssm_prep(dt_pre, a_log)


def gated_group_norm(o, skip_src, skip_off: int, skip_w, gate_src, g_off: int, w, groups: int, eps: float, act_dtype):
    if _gpu(o):
        return _k().hy_gated_group_norm(o, skip_src, skip_off, skip_w, gate_src, g_off, w, groups, eps, _f32(act_dtype))
    return ref.gated_group_norm(o, skip_src, skip_off, skip_w, gate_src, g_off, w, groups, eps, act_dtype)


def block_gates(u, w_gates, b_gates):
    """Gate pre-activations of a block-diagonal projection, float32: u [T, W] split into NB blocks of channels, block b
    times w_gates[b] ([W / NB, n]) plus b_gates[b] ([1, n], float32).  Returns [NB, T, n].  A library product with
    float32 accumulation and float32 output (its results are gates of a recurrence): bfloat16 operands go to the
    matrix cores as they are (their products are exact in float32), float32 operands to the float32 GEMM."""
    NB = w_gates.shape[0]
    T, W = u.shape
    ub = u.view(T, NB, W // NB).transpose(0, 1)
    if u.is_cuda and u.dtype == torch.bfloat16 and w_gates.dtype == torch.bfloat16:
        return torch.baddbmm(b_gates, ub, w_gates, out_dtype=torch.float32)
    return torch.baddbmm(b_gates, ub.float(), w_gates.float())


def rglru_scan(u, gates, sp, c: float, ysrc, y_off: int, q_start, pos0, slots, S, act_dtype, max_q: int = 0):
    """``max_q``: the most tokens any sequence brings in this step (sizes the launch grid; 0 = unknown)."""
    if _gpu(u):
        return _k().hy_rglru_scan(u, gates.contiguous(), sp, c, ysrc, y_off, q_start, pos0, slots, S, max_q)
    return ref.rglru_scan(u, gates, sp, c, ysrc, y_off, q_start, pos0, slots, S, act_dtype)


def moe_route_group(h, w_router, top: int, n_groups: int, keep: int, scale: float):
    if _gpu(h):
        return _k().hy_moe_route_group(h, w_router, top, n_groups, keep, scale)
    return ref.moe_route_group(h, w_router, top, n_groups, keep, scale)


# ---- sandwich residual stream, rotated values, retention -----------------------------------------------------------


def sandwich_join(y, x, w_y, w_out, groups: int, eps: float, act_dtype, y2=None, pair=None, emit: bool = True):
    """x (float32 residual, in place) <- x + group_rms_norm(v) * w_y with v = y (+ y2), or with ``pair`` = (w_a, w_b)
    v = (rms_norm(y) w_a + rms_norm(y2) w_b) / 2.  Returns group_rms_norm(x) * w_out in the activation dtype, or None
    when ``emit`` is off."""
    if _gpu(x):
        h = _k().hy_sandwich_join(y, y2, x, w_y, w_out if emit else None, pair[0] if pair else None,
                                  pair[1] if pair else None, groups, eps, _f32(act_dtype), True, emit)
        return h if emit else None
    return ref.sandwich_join(y, x, w_y, w_out, groups, eps, act_dtype, y2, pair, emit)


def unrotate_gate(o, pos, v_cos_sin, gate_src, g_off: int, H: int, Dv: int, act_dtype):
    if _gpu(o):
        return _k().hy_unrotate_gate(o, pos, v_cos_sin, gate_src, g_off, H, Dv)
    return ref.unrotate_gate(o, pos, v_cos_sin, gate_src, g_off, H, Dv, act_dtype)


def rotate_qk(proj, q_off: int, k_off: int, HQ: int, HK: int, D: int, dims: int, cos_sin, pos, q_mul: float,
              k_mul: float) -> None:
    if _gpu(proj):
        _k().hy_rotate_qk(proj, q_off, k_off, HQ, HK, D, dims if cos_sin is not None else 0, cos_sin, pos, q_mul, k_mul)
    else:
        ref.rotate_qk(proj, q_off, k_off, HQ, HK, D, dims, cos_sin, pos, q_mul, k_mul)


# ---- pre-norm stream with Dynamic Tanh norms, gated residuals and depth averages; PolyNorm ---------------------------


def dyn_tanh(x, wba, act_dtype):
    """tanh(alpha x) * w + b of the float32 stream; wba = w | b | alpha."""
    if _gpu(x):
        return _k().hy_dyn_tanh(x, wba, _f32(act_dtype))
    return ref.dyn_tanh(x, wba, act_dtype)


def gated_join(y, x, gate_src, g_off: int, gate_b, mult: float, wba, act_dtype, hist=None, run: int = -1, dwa=None,
               emit: bool = True):
    """x (float32 residual, in place) <- x + mult * sigmoid(gate) * y and, with ``dwa``, the weighted sum of that and
    the earlier layers' results in ``hist`` (where the layer's own result is kept).  Returns dyn_tanh(x, wba), or None
    when ``emit`` is off."""
    if _gpu(x):
        h = _k().hy_gated_join(y, x, gate_src, g_off, gate_b, mult, wba if emit else None, hist if dwa is not None else None,
                               run, dwa)
        return h if emit else None
    return ref.gated_join(y, x, gate_src, g_off, gate_b, mult, wba, act_dtype, hist, run, dwa, emit)


def poly_norm(z, F: int, abce, eps: float, act_dtype):
    """The PolyNorm activation of the first F columns of z [T, >= F]; returns [T, F]."""
    if _gpu(z):
        return _k().hy_poly_norm(z, F, abce, eps)
    return ref.poly_norm(z, F, abce, eps, act_dtype)


# ---- parallel stream: one layer norm per layer, both sublayers in one pair of products -------------------------------


def layer_norm_join(y, x, wb, eps: float, act_dtype, y2=None, emit: bool = True):
    """x (float32 residual, in place) <- x + y (+ y2), y None: x stays.  Returns layer_norm(x) * w + b (wb = w | b), or
    None when ``emit`` is off."""
    if _gpu(x):
        h = _k().hy_layer_norm_join(y, y2, x, wb if emit else None, eps, _f32(act_dtype))
        return h if emit else None
    return ref.layer_norm_join(y, x, wb, eps, act_dtype, y2, emit)


def glu_cols(src, off: int, F: int, limit: float, slope: float, shift: float, out) -> None:
    """The gated unit on columns off .. off + 2 F of src, into ``out`` [T, F] (a column range of wider rows)."""
    if _gpu(src):
        _k().hy_glu_cols(src, off, F, limit, slope, shift, out)
    else:
        ref.glu_cols(src, off, F, limit, slope, shift, out)


def norm_cols(src, off: int, n: int, w, eps: float):
    """RMS norm of n columns of src from ``off`` on, times w; [T, n] in src's dtype."""
    if _gpu(src):
        return _k().hy_norm_cols(src, off, n, w, eps)
    return ref.norm_cols(src, off, n, w, eps)


def conv_prep(proj, taps, tok_seq, q_start, pos0, slots, hist, pos, block_table, H: int, G: int, D: int, eps: float,
              q_temp, ks, vc, g_off: int, max_q: int):
    """Convolution, norms, temperature and cache write of an attention layer whose keys are values over their root mean
    square.  ``max_q``: the most tokens any sequence brings in this step (with 1 the history is rewritten in the same
    pass).  Returns (queries [T, H D], float32 gate columns [T, H] or None)."""
    if _gpu(proj):
        q, gate = _k().hy_conv_prep(proj, taps, tok_seq, q_start, pos0, slots, hist, pos, block_table, H, G, D, eps, q_temp,
                                    ks, vc, g_off, max_q)
        return q, (gate if g_off >= 0 else None)
    return ref.conv_prep(proj, taps, q_start, pos0, slots, hist, pos, tok_seq, block_table, H, G, D, eps, q_temp, ks, vc,
                         g_off)
