"""Projection GEMMs.

``linear(x, w)`` computes ``x @ w.T`` for weights stored [out, in] (HF layout); ``gate_up_silu`` is the fused K8+K9.
Routing is by measured shape:

* M <= 2 (single-stream decode): the hand-written GEMV (csrc/kernels/gemv.hip), 1 KiB row-contiguous weight
  streaming — beats hipBLASLt on every decode shape;
* M >= 3: the hand-written MFMA GEMM families with their fused epilogues — the decoder's residual add + RMSNorm
  partial sums on O / down (``gemv_resid`` -> ResidOut), the folded RMSNorm as a per-row scale on QKV / gate_up / LM
  head (a LazyNorm input), SwiGLU on gate_up: the skinny-M weight-streaming kernel (csrc/kernels/gemm_skinny.hip,
  M <= 128: jump-forward forwards, tail decode buckets) and the ping-pong tile GEMM (csrc/kernels/gemm_pp.hip) above,
  with the kernel, tile config and split-K of the measured plan (``gemm_plan.json``: per (N, K, epilogue) the best
  by M range, from ``scripts/tune_gemm_pp.py`` on one MI355X, random operands, cold weights; plan cfg >= 100 is
  skinny config cfg - 100);
* shapes that the plan does not list: up to 64 rows ``few_rows_plan``, from 128 on ``slab_rows_plan`` (``many_rows_plan``), between them ``mid_rows_plan``, where their measured ranges say that
  they win;
* hipBLASLt (torch.matmul) only where the plan records that the library wins by more than 3 % (the "plain library
  GEMM" rule), for unlisted shapes outside that range, or for shapes the kernel does not take (K % 64, N % 4).  CHRONOS_PP=lib|own|auto forces a side.
"""
from __future__ import annotations

import os
import sys
from dataclasses import dataclass
from typing import Callable, Optional

import torch

_pkg = sys.modules[__package__]


def _k():
    """The package's kernels.  (An import statement inside every function here cost a step of a hybrid decoder 30 us.)"""
    return _pkg._k()


# Largest M routed to the GEMV (gemv_ok).  Env CHRONOS_GEMV_MAX_M; scripts/single_stream.py A/Bs it (py_gemv_max_m).
# M = 2 goes to the skinny MFMA GEMM: the two-row GEMV streams at 1-3.5 TB/s against 4-5.5 at M = 1 and the skinny
# kernel's 3.4-4.9 at M = 3 (profiles/r3_gemm_table.md).
GEMV_MAX_M = int(os.environ.get("CHRONOS_GEMV_MAX_M", "1"))

# ---- the batched GEMM family (gemm_pp.hip) ----------------------------------------------------------------------
PP_MODE = os.environ.get("CHRONOS_PP", "auto")  # auto | own | lib
PP_PLAIN, PP_SWIGLU, PP_RESID = 0, 1, 2
# x rows (BM) / W rows (BN) per tile.  0-11: gemm_pp.hip (ping-pong); 12-35: gemm_lg.hip (software-pipelined: 12-19 and
# 29-31 the ring schedule, 20-28 the 64-deep slab schedule, 32-39 mid-M weight streaming with 64 W rows, 72-75 the
# same for M <= 32 with 32-row x tiles; 76-77 192 W rows x 128 x rows; 78-79 32-row x tiles with 7 / 12-stage rings;
# 80 = 20 on 32x32x16 MFMAs; 88 the 4-wave slab walk, 256 x 256 tiles, LDS-staged epilogue (gemm_slab.hip), 91 its loop on 32x32x16 MFMAs.
# Plans and programs from before may name 88 by any other id of 81-94: one kernel, but that 81-87 never took a split of K and do not now
_PP_BM = {0: 256, 1: 128, 2: 256, 3: 128, 4: 256, 5: 128, 6: 256, 7: 128, 8: 256, 9: 128, 10: 256, 11: 128,
          12: 256, 13: 128, 14: 256, 15: 128, 16: 256, 17: 128, 18: 256, 19: 128, 20: 256, 21: 256, 22: 128, 23: 128,
          24: 256, 25: 128, 26: 256, 27: 128, 28: 128, 29: 128, 30: 256, 31: 128, 32: 128, 33: 64, 34: 128, 35: 256,
          36: 64, 37: 128, 38: 64, 39: 64, 72: 32, 73: 32, 74: 32, 75: 32, 76: 128, 77: 128, 78: 32, 79: 32, 80: 256,
          **{c: 256 for c in range(81, 95)}}
_PP_BN = {0: 256, 1: 256, 2: 128, 3: 128, 4: 256, 5: 256, 6: 128, 7: 128, 8: 256, 9: 256, 10: 128, 11: 128,
          12: 256, 13: 256, 14: 128, 15: 128, 16: 256, 17: 256, 18: 128, 19: 128, 20: 256, 21: 256, 22: 256, 23: 128,
          24: 256, 25: 256, 26: 256, 27: 256, 28: 128, 29: 256, 30: 128, 31: 128, 32: 64, 33: 64, 34: 64, 35: 64, 36: 64, 37: 64, 38: 128, 39: 64, 72: 64, 73: 128, 74: 64, 75: 128, 76: 192, 77: 192, 78: 128, 79: 64, 80: 256,
          **{c: 256 for c in range(81, 95)}}
HB_FIRST, HB_LAST = 81, 94  # 88, its former ids, and 91
HB_SPLITK = (88, 89, 90, 91, 92, 93, 94)  # ... the ids that take a split-K
LG_FIRST = 12  # first gemm_lg.hip config: kResid partials every BN/2 columns (gemm_pp: BN/4)
# relative per-CU MAC rate of each tile config at full occupancy (gate_up M = 1024 / 16384 sweeps, profiles/r3_gemm_pp_*,
# profiles/r4_gemm_lg_*)
_PP_RATE = {0: 1.0, 1: 0.84, 2: 0.84, 3: 0.66, 4: 1.0, 5: 0.71, 6: 0.73, 7: 0.6, 8: 1.0, 9: 0.84, 10: 0.84, 11: 0.66,
            12: 0.95, 13: 0.7, 14: 0.7, 15: 0.75, 16: 0.98, 17: 0.7, 18: 0.7, 19: 0.75, 20: 1.05, 21: 0.7, 22: 0.7,
            23: 0.75, 24: 1.1, 25: 0.8, 26: 1.1, 27: 0.8, 28: 0.75, 29: 0.8, 30: 0.8, 31: 0.75, 32: 0.5,
            33: 0.4, 34: 0.5, 35: 0.55, 36: 0.4, 37: 0.5, 38: 0.5, 39: 0.4, 72: 0.3,
            73: 0.3, 74: 0.3, 75: 0.3, 76: 0.75, 77: 0.7, 78: 0.3, 79: 0.3, 80: 1.05,
            **{c: 1.15 for c in range(81, 95)}}
# skinny-M configs (gemm_skinny.hip SK_CONFIGS): plan id SK_BASE + c -> (RT: W tiles of 16 rows, MT: M <= 16 MT,
# NW: waves splitting K inside the workgroup)
SK_BASE = 100
_SK = {0: (1, 1, 16), 1: (2, 1, 8), 2: (4, 1, 4), 3: (2, 2, 8), 4: (4, 2, 4), 5: (2, 4, 4), 6: (4, 4, 4),
       7: (2, 8, 4), 8: (1, 2, 16), 9: (1, 4, 16), 10: (2, 4, 8), 11: (1, 1, 8)}
SKINNY_MAX_M = 128
# Configs that take any K % 64 (gemm_skinny.hip kSkinnyUneven): (W rows per workgroup, x rows, waves splitting K)
_UNEVEN = {112: (16, 32, 8), 113: (16, 64, 8), 114: (16, 16, 8), 115: (32, 16, 8)}
# Few rows, plain epilogue, shapes that the plan does not list: per largest M the configs that won somewhere on a grid of
# N = 512 .. 32768 by K = 512 .. 14336, and what a launch of each takes in us, fitted on that grid (cold weights; rms error 5 %):
# constant, split-K's second launch, per 64-deep step of a wave, per MB of weights, per 256 workgroups, per such step of each
# further round of 256 workgroups, per 100 MB of x that all workgroups read together.  The pick of the rule takes 3 % longer than the best config on average.
# profiles/few_rows_gemm.json: 86 shapes by 12 numbers of rows, every one measured with the library, the best config and the pick.
_FEW = ((16, {114: (2.4, 2.0, 0.77, 0.016, 0.23, 0.69, 3.4), 115: (2.2, 2.1, 1.4, 0.0082, 0.57, 1.3, 5.1),
              72: (2.2, 0.0, 0.16, 0.07, 1.2, 0.24, 8.3), 75: (1.7, 0.0, 0.28, 0.1, 1.4, 0.0, 10.0)}),
        (32, {112: (2.3, 2.1, 1.1, 0.0, 0.67, 0.9, 1.0), 72: (2.1, 0.0, 0.18, 0.052, 1.5, 0.22, 8.7),
              75: (1.8, 0.0, 0.29, 0.085, 1.7, 0.0, 12.0)}),
        (64, {113: (2.4, 2.3, 1.5, 0.0, 0.9, 1.0, 0.75), 72: (2.2, 0.0, 0.16, 0.0, 1.3, 0.19, 5.1),
              38: (3.0, 0.0, 0.31, 0.0, 0.54, 0.0, 35.0), 39: (2.4, 0.0, 0.21, 0.0, 1.2, 0.22, 14.0)}))
# Few rows, more weights than that: gemm_lg.hip's small tiles, K split over workgroups without tickets (gemm_split).  The same terms, and per M
# of partial sums, fitted on the "large" table of profiles/few_rows_gemm.json: 2 .. 32 rows at 65 shapes of 4 to 134 M elements (rms error 7 %;
# 33 .. 64 rows at 19 shapes of them, 10 % over all 65).
_FEW_LARGE = ((32, {72: (2.2, 2.32, 0.17, 0.0623, 1.53, 0.206, 1.66, 0.92), 74: (2.19, 2.32, 0.238, 0.049, 0.744, 0.186, 1.55, 1.02),
                    79: (2.6, 2.3, 0.172, 0.0595, 1.78, 0.225, 1.72, 0.917)}),
              (64, {39: (1.1, 2.7, 0.223, 0.0915, 0.94, 0.229, 0.0, 1.9), 38: (1.4, 2.7, 0.35, 0.105, 1.65, 0.259, 0.0, 1.7)}))
_plan_cache: dict = {}
_plan_table: Optional[dict] = None
_qplan_table: Optional[dict] = None


def _plan_file() -> dict:
    global _plan_table, _qplan_table
    if _plan_table is None:
        import json

        override = os.environ.get("CHRONOS_GEMM_PLAN")
        path = override or os.path.join(os.path.dirname(os.path.abspath(__file__)), "gemm_plan.json")
        try:
            with open(path) as fh:
                raw = json.load(fh)
        except FileNotFoundError:
            if override:  # an explicit A/B override that does not exist must not silently measure the library
                raise FileNotFoundError(f"CHRONOS_GEMM_PLAN={override!r}: no such plan file") from None
            raw = {}
        key = lambda k: tuple(int(v) for v in k.split(","))  # noqa: E731
        _plan_table = {key(k): rows for k, rows in raw.get("plans", {}).items()}
        _qplan_table = {key(k): rows for k, rows in raw.get("qplans", {}).items()}
    return _plan_table


QLG_BASE = 10  # qplan code >= QLG_BASE: gemm_lg.hip's fp8 config (code - QLG_BASE), row [M, code, split-K]
QLG_GEO = {0: (128, 256), 1: (256, 128), 2: (128, 128), 3: (128, 128),  # fp8 config -> (x rows, W rows) per tile
           4: (256, 256)}  # 4: the HB slab loop on the 32x32x64 fp8 MFMA (gemm_lg.hip F8HB)


def qplan_route(m: int, n: int, k: int, swiglu: bool) -> Optional[tuple[int, int]]:
    """W8A8 fp8 projection route from ops/gemm_plan.json "qplans" (``scripts/tune_gemm_pp.py --fp8``), rows
    [measured M, code(, split-K)] per (N, K, swiglu) read like the bf16 plan's: code 0 = the library's fp8 GEMM, 1 =
    fp8.hip (qgemv / block-scaled MFMA qgemm), QLG_BASE + c = gemm_lg.hip fp8 config c.  None = not measured."""
    _plan_file()
    rows = (_qplan_table or {}).get((n, k, int(swiglu)))
    if not rows:
        return None
    pick = next((r for r in rows if m <= r[0]), rows[-1])
    return int(pick[1]), int(pick[2]) if len(pick) > 2 else 1


def qplan_own(m: int, n: int, k: int, swiglu: bool) -> Optional[bool]:
    """True = a hand-written fp8 kernel (fp8.hip or gemm_lg.hip), False = the library, None = not measured."""
    r = qplan_route(m, n, k, swiglu)
    return None if r is None else r[0] != 0


def _sk_valid(c: int, m: int, n: int, k: int, mode: int, sk: int) -> bool:
    rt, mt, nw = _SK[c]
    if m > 16 * mt or k % (64 * nw * sk):
        return False
    return (rt % 2 == 0 and n % 2 == 0 and (n // 2) % (8 * rt) == 0) if mode == PP_SWIGLU else n % (16 * rt) == 0


def _sk_model(m: int, n: int, k: int, mode: int, cus: int = 256) -> Optional[tuple[int, int]]:
    """Cost-model pick of a skinny config: the narrowest x tile covering M, W tiles >= x tiles (x re-read bytes <=
    weight bytes), split-K until the grid covers the CUs twice."""
    best = None
    for c, (rt, mt, nw) in _SK.items():
        if m > 16 * mt or (mt > 1 and m <= 8 * mt):
            continue
        groups = (n // 2) // (8 * rt) if mode == PP_SWIGLU else n // (16 * rt)
        for sk in (1, 2, 4, 7, 8, 14, 16):
            if not _sk_valid(c, m, n, k, mode, sk):
                continue
            # a cross-workgroup split costs more than it hides (profiles/r3_gemm_table.md): only when the grid
            # would otherwise leave CUs idle; then the widest workgroups
            t = (sk > 1 and groups >= cus, rt < mt, -min(groups * sk, cus), sk, -nw, -rt)
            if best is None or t < best[0]:
                best = (t, (SK_BASE + c, sk))
    return best[1] if best else None


def _pp_valid(cfg: int, n: int, k: int, mode: int, sk: int, m: int = 0) -> bool:
    if cfg >= SK_BASE:
        return cfg - SK_BASE in _SK and _sk_valid(cfg - SK_BASE, m, n, k, mode, sk)
    bn = _PP_BN[cfg]
    if k % 64 or (k // 64) % sk or (HB_FIRST <= cfg <= HB_LAST and sk != 1 and cfg not in HB_SPLITK):
        return False
    return n % 4 == 0 if mode == PP_PLAIN else n % bn == 0


def _pp_model(m: int, n: int, k: int, mode: int, cus: int = 256) -> tuple[int, int]:
    """Cost-model pick for a shape the measured plan does not list: whole rounds of tiles over the CUs at each
    config's per-CU rate, plus the split-K slab traffic."""
    best, arg = None, (0, 1)
    for cfg in (0, 1, 2, 3):
        bm, bn = _PP_BM[cfg], _PP_BN[cfg]
        tiles = -(-m // bm) * -(-n // bn)
        for sk in (1, 2, 4):
            if not _pp_valid(cfg, n, k, mode, sk) or (sk > 1 and tiles * sk > 2 * cus):
                continue
            rounds = -(-tiles * sk // cus)
            t = rounds * bm * bn * (k // sk) / _PP_RATE[cfg] / 256.0 ** 2 + (sk > 1) * tiles * sk * bm * bn * 4 / 5e5
            if best is None or t < best:
                best, arg = t, (cfg, sk)
    return arg


def pp_plan(m: int, n: int, k: int, mode: int = PP_PLAIN) -> Optional[tuple[int, int]]:
    """(config, split-K) of the hand-written batched GEMM for this shape — config >= SK_BASE is the skinny kernel —
    or None for the library."""
    if m <= GEMV_MAX_M or PP_MODE == "lib":
        return None
    key = (m, n, k, mode)
    hit = _plan_cache.get(key, False)
    if hit is not False:
        return hit
    out = None
    if k % 64 == 0 and (n % 4 == 0 if mode == PP_PLAIN else n % 128 == 0):
        rows = _plan_file().get((n, k, mode))
        if PP_MODE == "own":
            out = (_sk_model(m, n, k, mode) if m <= SKINNY_MAX_M else None) or _pp_model(m, n, k, mode)
        elif rows:
            # rows [measured M, cfg, split-K] sorted by M: a measured M decides (previous M, M]; the last row also
            # everything above it.  cfg < 0 = the library measured faster.
            pick = next((r for r in rows if m <= r[0]), rows[-1])
            out = None if pick[1] < 0 else (pick[1], pick[2])
        # auto, shape never measured: the library (a hand-written config is routed only on a recorded A/B)
        if out is not None and not _pp_valid(out[0], n, k, mode, out[1], m):
            out = None
    _plan_cache[key] = out
    return out


def _library_streams(m: int, n: int, k: int) -> bool:
    """Shapes beyond _FEW's where the library reads the weights at 4 TB/s and these kernels do not.  us, library and the pick without this line:
    16 rows of 4096 x 8192 16.4 and 19.2, 8192 x 4096 16.1 and 18.5, 5120 x 5120 15.8 and 16.7, 8192 x 8192 29.5 and 31.2; 64 rows of 8192 x 4096 19.1
    and 20.6.  Not at other K, nor with more rows for fewer outputs: 16 rows of 4096 x 6400 23.6 and 14.5, 24 rows of 3584 x 7168 20.3 and 14.6, 64
    of 5632 x 5632 23.4 and 22.1.  Of 437 shapes 53 would be slower than the library by more than 3 % without this line, 7 are with it."""
    return n * k >= 25_000_000 and 2560 <= n <= 8192 and k <= 8192 and k % 1024 == 0 and (m <= 16 or n >= 4096 and m <= 32 or n > 7168)


def few_rows_plan(m: int, n: int, k: int) -> Optional[tuple[int, int]]:
    """(config, split-K) of the hand-written GEMM for few rows of a shape that no plan lists, or None (the GEMV or the
    library): of shapes that the kernels take (rows of w in 16s, at least one; K in 64s up to 2^20).  Where it wins, measured on the
    grid of _FEW, us, GEMV or library -> this:
    one row: K < 2048, where the GEMV's waves have one step each (5632 x 1024: 7.3 -> 5.7; 32768 x 512: 22 -> 9.7; at K = 2048 the
    two are level), and K % 512, which the GEMV does not take (1024 x 2816: 8.6 -> 5.7): no slower at any of 41 shapes;
    2 .. 64 rows: weights up to 12.5 M elements, from 33 rows on up to 7 M or K <= 2048 (2048 x 2048, 16 rows: 11.0 -> 6.4; 64 rows:
    11.6 -> 9.8), and where the library keeps half the chip idle, wide outputs of up to 48 rows, more weights too (22016 x 2048, 16 rows:
    41 -> 21): 1.54 times as fast on average over 622, one slower by more than 3 % (24 rows of 1536 x 5632, 10.3 -> 11.0);
    Beyond, 2 .. 64 rows: _FEW_LARGE, from 33 rows on for less than 12288 outputs, but for _library_streams: library -> this, 16 rows of 4096 x
    4096 15.7 -> 10.6, 4096 x 11008 37.6 -> 21.5, 12288 x 4096 27.7 -> 22.8; 64 rows of 4096 x 14336 39.9 -> 28.5, 2048 x 8192 22.3 -> 13.8;
    the wider ones are mid_rows_plan's.  (Both tables and the figures here are from before the ring tiles' weights were marked as read once, which takes 5 to
    12 % off 72, 74, 75, 79, 38 and 39.  Measured again with it, mid_rows_plan's among them: 1072 shapes 1.43 times as fast as the library, 8 slower by more than 3 %, the
    worst by 11 % (64 rows of 12288 x 5632, 34.2 -> 38.1); picks take 2 % longer than the best on average, 4 % from 33 rows on; of 84 shapes that are left to the library 61
    would be faster here by more than 3 %, up to 1.24 times, 8192 x 6144 by 2 to 40 rows.)  Tables: profiles/few_rows_gemm.json, which tests/test_measured_rules.py replays."""
    if 1 < m <= GEMV_MAX_M or PP_MODE != "auto":   # (programs set both while they run: nothing of them in the cache)
        return None
    key = (m, n, k, -1)
    hit = _plan_cache.get(key, False)
    if hit is not False:
        return hit
    nk, out = n * k, None
    if m == 1:
        ok = (k < 2048 or k % 512 != 0) and nk <= 100_000_000
    else:
        ok = m <= 64 and (nk <= 12_500_000 and (m <= 32 or k <= 2048 or nk <= 7_000_000) or
                                       m <= 48 and n >= 12288 and nk <= (40_000_000 if n < 16384 else 100_000_000))
    if ok and n > 0 and n % 16 == 0 and k % 64 == 0 and k <= 1 << 20 and (n, k, PP_PLAIN) not in _plan_file():
        best = None
        for cfg, c in next(models for most, models in _FEW if m <= most).items():
            bn, bm, nw = _UNEVEN.get(cfg) or (_PP_BN[cfg], _PP_BM[cfg], 1)
            for sk in (1, 2, 4, 8) if cfg in _UNEVEN else (1,):
                groups = -(-n // bn) * -(-m // bm) * sk
                if cfg in _UNEVEN and n % bn or k < 64 * sk or (sk > 1 and groups > 1024):
                    continue
                steps = k / (64 * sk * nw)
                t = (c[0] + c[1] * (sk > 1) + c[2] * steps + c[3] * nk * 2e-6 + c[4] * groups / 256
                     + c[5] * (-(-groups // 256) - 1) * steps + c[6] * m * k * groups * 2e-8)
                if best is None or t < best:
                    best, out = t, (cfg, sk)
    elif 1 < m <= 64 and n > 0 and n % 16 == 0 and 4_000_000 <= nk and (n + 128) * k < 1 << 30 and k % 64 == 0 and 0 < k <= 1 << 20 and (
            m <= 32 or n < 12288) and (n, k, PP_PLAIN) not in _plan_file() and not _library_streams(m, n, k):
        best = None
        for cfg, c in next(models for most, models in _FEW_LARGE if m <= most).items():
            for sk in (1, 2, 4, 8):
                groups, steps = -(-n // _PP_BN[cfg]) * sk, k / (64 * sk)
                if k // 64 % sk or (sk > 1 and groups > 2048):
                    continue
                t = (c[0] + c[1] * (sk > 1) + c[2] * steps + c[3] * nk * 2e-6 + c[4] * groups / 256
                     + c[5] * (-(-groups // 256) - 1) * steps + c[6] * m * k * groups * 2e-8 + c[7] * sk * m * n * 1e-6)
                if best is None or t < best:
                    best, out = t, (cfg, sk)
    _plan_cache[key] = out
    return out


# 65 .. 512 rows, and 33 .. 64 of 12288 outputs and more that few_rows_plan leaves: gemm_lg.hip's tiles of 64 W by 64 x rows (39, K split without
# tickets), 64 by 128 (32) and 128 by 128 (19).  The terms of _FEW_LARGE, fitted on profiles/mid_rows_gemm.json (rms error 7 %).
_MID = ((64, {39: (0.247, 3.535, 0.273, 0.037, 1.296, 0.257, 0.392, 2.906), 19: (3.26, 2.0, 0.378, 0.067, 0.0, 0.1, 1.6, 0.605)}),
        (128, {39: (2.318, 2.234, 0.227, 0.0, 1.264, 0.249, 0.892, 0.74), 32: (2.957, 2.0, 0.329, 0.0, 0.144, 0.377, 2.98, 1.176),
               19: (3.861, 2.0, 0.482, 0.0, 0.006, 0.1, 7.939, 0.496)}),
        (256, {39: (2.545, 2.395, 0.242, 0.0, 1.391, 0.232, 0.196, 0.936)}), (512, {39: (2.187, 2.426, 0.258, 0.0, 2.095, 0.234, 0.059, 0.607)}))


def mid_rows_plan(m: int, n: int, k: int) -> Optional[tuple[int, int]]:
    """(config, split-K) of the hand-written GEMM for rows and shapes that few_rows_plan, many_rows_plan and the measured plan leave, or None (the library):
    65 .. 128 rows, 33 .. 64 rows by 12288 outputs and more, 129 .. 256 rows by up to 4096 outputs, 257 .. 512 by up to 2048 with K <= 8192; outputs and K
    from 512 on, outputs to 153600, K to 32768 (28672 from 129 rows on) and 640 M weights, which is what was measured.  Rows beyond 64 count in 32s, so that a server's steps find their plan again.  us, library -> this: 80 rows of 1024 x 1024 10.9 ->
    6.6, 4096 x 4096 17.1 -> 13.9, 2048 x 5632 16.4 -> 12.2, 12288 x 4096 33.4 -> 28.0, 32768 x 1024 22.9 -> 17.0; 64 rows of 14336 x 4096 28.6 ->
    26.8, 32768 x 4096 62.2 -> 58.3 (39 would be 55.4: the model is off there); 192 rows of 1024 x 1024 10.7 -> 7.5, 2048 x 5632 21.2 -> 19.1; 512 rows of 1024 x 4096 15.8 -> 14.7.  On average 1.29
    (460 shapes of 65 .. 128 rows), 1.21 (105 of 33 .. 64), 1.21 (123 of 129 .. 256) and 1.10 times (86) as fast, of 774 shapes 35 slower by more than 3 %,
    the worst by 9 % (512 x 1408, 8.4 -> 9.2); 58 shapes beyond the fit's, up to 622 M weights and K = 32768: 1.29
    times, 5 slower, the worst by 7 %; and a library call costs the host 22 us, this 7.  Beyond these ranges the two are level or the
    library ahead.  Table: profiles/mid_rows_gemm.json, which tests/test_measured_rules.py replays."""
    if PP_MODE != "auto":
        return None
    m = m if m <= 64 else -(-m // 32) * 32
    key = (m, n, k, -5)
    hit = _plan_cache.get(key, False)
    if hit is not False:
        return hit
    out = best = None
    if ((m > 32 and n >= 12288 if m <= 64 else n >= 512 if m <= 128 else 512 <= n <= 4096 if m <= 256 else m <= 512 and 512 <= n <= 2048 and k <= 8192)
            and 512 <= k <= (32768 if m <= 128 else 28672) and n % 16 == 0 and k % 64 == 0 and n <= 153600 and n * k <= 640_000_000
            and (n, k, PP_PLAIN) not in _plan_file()):
        for cfg, c in next(models for most, models in _MID if m <= most).items():
            for sk in (1, 2, 4, 8) if cfg == 39 else (1,):
                groups, steps = -(-n // _PP_BN[cfg]) * -(-m // _PP_BM[cfg]) * sk, k / (64 * sk)
                if k // 64 % sk or (sk > 1 and (groups > 1024 or k // 64 // sk < 2)):
                    continue
                t = (c[0] + c[1] * (sk > 1) + c[2] * steps + c[3] * n * k * 2e-6 + c[4] * groups / 256
                     + c[5] * (-(-groups // 256) - 1) * steps + c[6] * m * k * groups * 2e-8 + c[7] * sk * m * n * 1e-6)
                if best is None or t < best:
                    best, out = t, (cfg, sk)
    _plan_cache[key] = out
    return out


# Configs of gemm_slices and of gemm_ring (csrc/kernels/bindings.cpp)
_SLICED = (19, 32, 33, 36, 38, 39, 72, 73, 74, 75, 78, 79, *_UNEVEN)
_RING = (19, 32, 38, 39, 72, 74, 75, 79)


def product_f32(x: torch.Tensor, w: torch.Tensor) -> Optional[torch.Tensor]:
    """x @ w.T as float32 [M, N], the product's sums before their rounding, where few_rows_plan or mid_rows_plan takes it, or None.  A vocabulary's logits: 8 rows of
    32768 x 1024 16 us as a rounded product and a conversion, 12 so."""
    (m, k), n = x.shape if x.dim() == 2 else (0, 0), w.shape[0]
    if not 0 < m <= 64 or n % 4 or not _plain_rows(x, w) or _registered(m, n, k) or (n + 128) * k >= 1 << 30:
        return None
    plan = few_rows_plan(m, n, k) or mid_rows_plan(m, n, k)
    if plan is None or plan[0] not in _SLICED:
        return None
    skinny = plan[0] >= SK_BASE
    return _k().gemm_f32(x, w, plan[0] - SK_BASE * skinny, plan[1], skinny)


def product_slices(x: torch.Tensor, w: torch.Tensor) -> Optional[torch.Tensor]:
    """The float32 slices [S, M, N] of x @ w.T where few_rows_plan splits K, or None: for kernels that take them in the product's place."""
    (m, k), n = x.shape if x.dim() == 2 else (0, 0), w.shape[0]
    if not 0 < m <= 64 or n % 8 or n > 8192 or not _plain_rows(x, w) or _registered(m, n, k):
        return None
    plan = few_rows_plan(m, n, k)
    if plan is None or plan[1] == 1 or (plan[0] >= SK_BASE and plan[0] not in _UNEVEN):
        return None
    skinny = plan[0] >= SK_BASE
    return _k().gemm_slices(x, w, plan[0] - SK_BASE * skinny, plan[1], skinny)


def product_parts(x: torch.Tensor, w: torch.Tensor) -> Optional[torch.Tensor]:
    """product_slices beyond 64 rows: the slices where linear()'s rules split K.  Product, its sum and the
    join behind it -> product and join, us: 113 rows of 1024 x 2816 12.1 -> 9.7, of 2048 x 5632 18.3 -> 15.0, 200 of 2048 x 2048 14.8 -> 11.5, 700 of 4096 x 11008 77 -> 71, 1351 of 4096 x
    14336 153 -> 149, 3000 of 2048 x 5632 88 -> 76; faster at all of 72 measured."""
    (m, k), n = x.shape if x.dim() == 2 else (0, 0), w.shape[0]
    if m <= 64 or n % 8 or n > 8192 or not _plain_rows(x, w) or _registered(m, n, k):
        return None
    plan = _linear_plan(m, n, k)
    if plan is None or plan[1] == 1 or plan[0] >= SK_BASE:
        return None
    return _k().gemm_slices(x, w, plan[0], plan[1], False)


# Many rows, shapes that the plan does not list: what a launch takes in us, fitted on a grid of M = 65 .. 8192, N = 512 .. 16384, K = 512 ..
# 8192 (rms error 8 %).  88 (gemm_slab.hip): constant, per half tile of the last round, per 64-deep step of a round of
# 256 x 256 tiles and of the halves, per M of results, per M of weights; 19 and 32 (128 x rows by 128 and 64 W rows): constant, per round of
# 256 tiles (there is one), per 256 tiles, per 64-deep step of these two, per M of weights.  Of all tile configs these three suffice, and the pick
# is the fastest of them.  Both grids, here and at _MANY_SPLIT: profiles/many_rows_gemm.json.
_MANY_88 = (2.6, 1.9, 1.17, 0.55, 0.52, 0.29)
_MANY_TILES = {19: (128, 2.9, 1.9, 1.2, 0.294, 0.15, 0.16), 32: (64, 2.7, 1.45, 0.46, 0.224, 0.083, 0.13)}
# ... and with an activation in 88's epilogue, the gated unit and the others; the same activation as a pass of its own: constant, per M of
# its inputs
_MANY_ACT = {True: ((2.1, 4.7, 1.22, 0.57, 0.41, 0.16), 4.45, (2.9, 0.44)), False: ((3.3, 2.2, 1.22, 0.55, 0.51, 0.17), 0.0, (2.8, 0.39))}
MANY_MIN = 128
# 88 with K split over workgroups (float32 slices and a launch that sums them), one round of tiles or of halves: constant, per slab of halves, of
# them as all CUs have one, of tiles, of them as all CUs have one, per M of all slices' results, per M of weights.  Fitted on 696 launches, M = 128 ..
# 3072, N = 1024 .. 6144, K = 1024 .. 14336 (rms error 8 %; the split picked takes 1 % longer than the best on average).
_MANY_SPLIT = (11.3, 0.51, 0.13, 0.80, 0.31, 1.09, 0.088)


def _many_tiles(m: int, n: int) -> tuple[int, int, bool]:
    """(whole rounds of 256 x 256 tiles, what is left for the last one, as halves?) of a launch on 256 CUs (chronos_slab.h slab_split, slab_tail)."""
    nt = -(-n // 256)
    t = -(-m // 256) * nt
    if 0 < m % 256 <= 128 and 2 * (m // 256 * nt % 256) + nt <= 256:
        return m // 256 * nt // 256, 2 * (m // 256 * nt % 256) + nt, True
    return (t // 256, 2 * (t % 256), True) if 0 < t % 256 <= 128 else (t // 256, t % 256, False)


def _third_idle(m: int, n: int, k: int) -> bool:
    """One long round of tiles, or of halves, that leaves a third of the CUs idle, where the library's other tile sizes need not: halves beyond
    K = 2048 (768 x 5632 x 8192 84 us, here 97; at K = 1024 and 2048 the two are level, and a library call costs the host more), whole tiles from 2048 on
    where there are more outputs than rows, in 256s (2446 x 4096 x 2048 39.5, here 45.1; ragged outputs cost the library as much, and tall products
    are hardly faster there: 8192 x 1280 x 2048 44.0 and 45.3)."""
    rounds, last, halves = _many_tiles(m, n)
    return rounds == 0 and last <= 170 and (halves and k > 2048 or not halves and n % 256 == 0 and n > m and k >= 2048)


def _many_slab(c, per_round: float, m: int, n: int, k: int) -> float:
    rounds, last, half = _many_tiles(m, n)
    rounds += last > 0 and not half
    return c[0] + per_round * rounds + (c[1] + c[3] * (k // 64)) * half + c[2] * rounds * (k // 64) + (c[4] * m + c[5] * k) * n * 1e-6


def _many_split(m: int, n: int, k: int) -> tuple[float, int]:
    nt, last, best = -(-n // 256), 0 < m % 256 <= 128, (float("inf"), 1)
    c = _MANY_SPLIT
    for s in range(2, 17):
        tiles, whole, slabs = -(-m // 256) * nt * s, m // 256 * nt * s, k // 64 // s
        if k // 64 % s or slabs < 2 or tiles > 256:
            continue
        half = 2 * whole + nt * s if last and 2 * whole + nt * s <= 256 else 2 * tiles if tiles <= 128 else 0
        t = slabs * (c[1] + c[2] * half / 256 if half else c[3] + c[4] * tiles / 256)
        best = min(best, (c[0] + t + (c[5] * s * m + c[6] * k) * n * 1e-6, s))
    return best


def _many_best(m: int, n: int, k: int) -> tuple[float, int]:
    best = (_many_slab(_MANY_88, 0.0, m, n, k), 88)
    for cfg, (bn, c0, c1, c2, c3, c4, c5) in _MANY_TILES.items():
        t = -(-m // 128) * -(-n // bn)
        if t > 256:   # (of no shape in either table are these tiles the faster ones beyond a round)
            continue
        steps = k // 64
        best = min(best, (c0 + c1 + c3 * steps + t / 256 * (c2 + c4 * steps) + c5 * n * k * 1e-6, cfg))
    return best


def _many_fits(m: int, n: int, k: int) -> bool:
    return k % 64 == 0 and 0 < k <= 1 << 20 and n > 0 and n % 4 == 0 and (max(m, n) + 384) * k < 1 << 30


def many_rows_plan(m: int, n: int, k: int) -> Optional[tuple[int, int]]:
    """(config, split-K) of the hand-written GEMM for at least 128 rows of a shape that no plan lists, or None (the library): from 64 tiles of 128 x rows
    by 64 W rows on, and K / 16 of them, but for _third_idle; (88, split-K) where at least 12 tiles of 256 x 256 are too few for the chip and the split's model is a
    tenth below the others' (51 shapes of _MANY_SPLIT's grid, 1.23 times as fast as the library, one 9 % slower; 768 x 4096 x 11008
    83 -> 71 us, 1024 x 4096 x 11008 102 -> 83; fewer tiles: the library's own splits are faster).  There, on the grid of _MANY_88: 1.14 times as
    fast as the library on average (302 shapes; 25 slower by more than 3 %, the worst by 14 %: whole or part rounds at K up to 2048, where the library's
    first loads and stores cost less, and rounds that are nearly full); at 260 shapes drawn off the grid 1.16 times (162; 16 slower, the worst 13 %);
    below the line 0.84 times.  A library call also costs the host 22 us, this 7.  Rows count in 128s, so that a server's
    steps of any size find their plan again.  (Measured with 256 x 256 tiles and halves only, on one card.  With 88's x tiles by rows, slab_rows_plan's
    and mid_rows_plan's picks among them, on another: 781 shapes 1.15 times as fast, 100 slower by more than 3 %, the worst by 23 %, most of them one round of 19 or 32,
    which were no faster there before: 256 x 4096 x 2048 13.4 and 16.4, 1536 x 2048 x 5632 44.4 and 54.0.)  Tables: profiles/many_rows_gemm.json, which tests/test_measured_rules.py replays."""
    if PP_MODE != "auto":
        return None
    m = -(-m // 128) * 128
    key = (m, n, k, -2)
    hit = _plan_cache.get(key, False)
    if hit is not False:
        return hit
    tiles = m // 128 * -(-n // 64)
    out = None
    if _many_fits(m, n, k) and tiles >= max(64, k // 16) and (n, k, PP_PLAIN) not in _plan_file():
        out = (_many_best(m, n, k)[1], 1)
        if out[0] == 88 and _third_idle(m, n, k):
            out = None
    if _many_fits(m, n, k) and -(-m // 256) * -(-n // 256) >= 12 and (n, k, PP_PLAIN) not in _plan_file():
        t, s = _many_split(m, n, k)
        if t < 0.9 * _many_best(m, n, k)[0]:
            out = (88, s)
    _plan_cache[key] = out
    return out


# 88 with the x tiles that gemm_slab.hip's slab_rows picks, K split or not: constant, the split's second launch, per 64-deep step of a round of 256 x 256
# tiles, per MB of weights, per round, per M of all slices' results, per M of results.  Fitted on profiles/slab_rows_gemm.json (rms error 8 %).
_SLAB_ROWS = (2.0, 2.11, 1.09, 0.118, 1.035, 1.238, 0.829)


def _slab_rounds(m: int, nt: int, s: int) -> float:
    """What slab_rows takes the launch for, in rounds of 256 x 256 tiles."""
    last = m % 256
    tail = nt * s if 0 < last <= 128 and nt * s <= 256 and 2 * (m // 256 * nt * s % 256) + nt * s <= 256 else 0
    tiles = (m // 256 if tail else -(-m // 256)) * nt * s
    rest = tiles % 256
    half = 2 * rest + tail if tail or rest <= 128 else 0
    full = tiles - rest if half else tiles
    best = -(-full // 256) + (0.57 if full else 0.63) * -(-half // 256)
    for rows, cost in ((128, 0.61), (160, 0.67), (192, 0.76), (224, 0.86)):
        t = cost * -(-(-(-m // rows) * nt * s) // 256)
        if t < best * (0.94 if best > 2.5 else 0.97):
            best = t
    return best


def slab_rows_plan(m: int, n: int, k: int) -> Optional[tuple[int, int]]:
    """many_rows_plan, or (88, split-K) in its place from 257 rows on, by 1024 to 8192 outputs, where the x tiles of 128 to 256 rows make that the faster one: in
    place of another split by 5 % by the model, of the library where it would have to reach 950 TFLOP/s, which at these sizes it does not.  us, before ->
    this: 1088 rows of 4096 x 14336 154 -> 119, of 11008 122 -> 98, 1500 153 -> 115, 1088 of 3648 x 8192 84 -> 70, 2100 of 4096 x 4096 82 -> 63.  Of 576 shapes 122 change, 1.18
    times as fast, one slower by more than 3 % (2446 x 2048 x 4096, 0.90).  Table: profiles/slab_rows_gemm.json, which tests/test_measured_rules.py replays."""
    out = many_rows_plan(m, n, k)
    if PP_MODE != "auto" or not 256 < m <= 4096 or out is not None and out[0] != 88:
        return out
    m = -(-m // 32) * 32
    key = (m, n, k, -6)
    hit = _plan_cache.get(key, False)
    if hit is not False:
        return hit
    if (1024 <= n <= 8192 and k >= 1024 and n * k <= 64_000_000 and _many_fits(m, n, k) and (n, k, PP_PLAIN) not in _plan_file()
            and (out is not None or mid_rows_plan(m, n, k) is None)):
        c, times = _SLAB_ROWS, {}
        for sk in (1, 2, 4, 8, out[1] if out else 1):
            if k // 64 % sk or k // 64 // sk < 2 or sk > 1 and -(-m // 256) * -(-n // 256) * sk > 768:
                continue
            r = _slab_rounds(m, -(-n // 256), sk)
            times[sk] = c[0] + c[2] * r * (k // 64 // sk) + c[3] * n * k * 2e-6 + c[4] * r + c[6] * m * n * 1e-6 + (sk > 1) * (c[1] + c[5] * sk * m * n * 1e-6)
        sk = min(times, key=times.get)
        if times[sk] < 0.95 * (times[out[1]] if out else 5 + 2 * m * n * k / 900e6):
            out = (88, sk)
    _plan_cache[key] = out
    return out


def _many_act_pays(m: int, n: int, k: int, glu: bool) -> bool:
    if not _many_fits(m, n, k) or glu and n % 256:
        return False
    c, per_round, apart = _MANY_ACT[glu]
    return _many_slab(c, per_round, m, n, k) < _many_best(m, n, k)[0] + apart[0] + apart[1] * m * n * 1e-6


def product_act(x: torch.Tensor, w: torch.Tensor, mode: int, limit: float = 0.0, slope: float = 0.0, shift: float = 0.0) -> Optional[torch.Tensor]:
    """x @ w.T with an activation in the epilogue (mode as in torch.ops.chronos.gemm_act: 3 a gated unit of w = [gate; up], 4 squared ReLU, 5
    GELU), or None where that does not pay: with up to 64 rows by _ring_more and _FEW_MORE, below 128 in the GEMV's or the ring tiles'
    epilogue where linear() takes those unsplit, from 128 on where the best product (many_rows_plan's or, below it, as if it were) and a pass of its
    own are faster by their models.  On the grid of _MANY_88, against the faster of the library and this product with
    its pass: gated units 1.12 times as fast (188 shapes; the worst 0.92), the others 1.15 (196; 0.90).  Both worst are long rounds that leave a
    third of the CUs idle (_third_idle); they stay, because the pass reads a rounded product: a step with it is further from float64 (0.0076 for 0.0067)."""
    m, (n, k) = x.numel() // max(1, x.shape[-1]), w.shape
    if PP_MODE != "auto" or x.dim() != 2 or not _plain_rows(x, w) or _registered(m, n, k):
        return None
    if m < MANY_MIN:
        cfg = _few_more(m, n, k, 2 if mode == 3 else 1)
        if m == 1 and not cfg and _linear_plan(1, n, k) is None and gemv_ok(1, n, k):
            return _k().gemv_act(x, w, mode, limit, slope, shift)
        plan = _linear_plan(m, n, k) if m > 64 or _ring_more(m, n, k) else None
        if plan is not None and plan[0] in _RING and plan[1] == 1 and (mode != 3 or n % _PP_BN[plan[0]] == 0):
            return _k().gemm_ring(x, w, plan[0], 1, mode, 0, 0, None, limit, slope, shift)[0]
        return _k().gemm_few(x, w, cfg, mode, 0, 0, None, limit, slope, shift)[0] if cfg else None
    glu = mode == 3
    rows = -(-m // 128) * 128
    key = (rows, n, k, -3 if glu else -4)
    pays = _plan_cache.get(key)
    if pays is None:
        pays = _plan_cache[key] = _many_act_pays(rows, n, k, glu)
    if not pays:
        return None
    return _k().gemm_act(x, w, mode, limit, slope, shift)


# Few rows with more to do behind the product (gemm_few): by the most rows (config up to 8 M elements of weights and for one row from 30 M on, beyond; the most of
# them where it wins with float32 outputs behind, with an activation, with a gated unit, whose config is always the second).  Measured at nine M = 1 .. 64
# on 25 shapes ("more behind" in profiles/few_rows_gemm.json), us, two launches -> one: 16 rows of 6144 x 2048 and 16 behind 16.2 -> 9.7, 12288 x 4096
# and 64 33.8 -> 30.1; 32 rows of that 34.6 -> 34.1; 16 rows of 8192 x 2048 with GELU 13.5 -> 10.6, 14336 x 4096 29.7 -> 30.7; gated units of 11264 x
# 2048 15.2 -> 16.7 (16 rows), 15.8 -> 20.0 (32), of 5632 x 1024 9.5 -> 6.9 (32).  On average 1.53, 1.40 and 1.20 times as fast
# where they are taken, the worst 0.91, those 16 rows: they stay, because the pass of its own reads a rounded product (a step's error against float64
# 0.0042, 0.0046 with it).
_FEW_MORE = ((16, 114, 115, 60e6, 24e6, 24e6), (32, 112, 116, 30e6, 24e6, 8e6), (64, 113, 117, 30e6, 24e6, 0))


def _few_more(m: int, n: int, k: int, kind: int) -> int:
    """Config of gemm_few, or 0: kind 0 float32 outputs behind, 1 an activation, 2 a gated unit."""
    if not 0 < m <= 64 or PP_MODE != "auto" or 1 < m <= GEMV_MAX_M or n % 32 or n <= 0 or k % 64 or not 0 < k <= 1 << 20:
        return 0
    for most, small, large, *limits in _FEW_MORE:
        if m <= most:
            if n * k > limits[kind]:
                return 0
            return (large if kind == 2 or 8e6 < n * k and (m > 1 or n * k < 30e6) else small) - SK_BASE
    return 0


def _ring_more(m: int, n: int, k: int) -> bool:
    """Whether up to 64 rows with more to do behind the product go to the ring tiles before gemm_few, whose workgroups of 32 weight rows are
    more than a round of 256 from 8192 rows on, and don't take K round from places of their own over large weights.  Two launches, gemm_few -> ring, us:
    gated units of 11264 x 2048, 4 rows 13.3, 15.0 -> 11.4, 16 rows 13.9, 16.8 -> 11.7, 64 rows 17.3, 24.0 -> 14.8; of 16384 x 1024, 16 rows
    10.6, 10.2 -> 8.4; GELU after 14336 x 1024, 32 rows 10.8, 12.4 -> 8.7; 12304 x 4096 with float32 rows, 4 rows 25.9, 26.3 -> 18.0, 16 rows
    25.2, 30.0 -> 18.8.  On this side: 8192 x 2048 with GELU 16 rows 10.6, ring 10.9, 64 rows 13.8, ring 14.5."""
    return m > 1 and n * k > 8_000_000 and (n > 8192 or n * k > 24_000_000)


def product_rows(x: torch.Tensor, w: torch.Tensor, n0: int, nf: int, bias: Optional[torch.Tensor]):
    """(x @ w[:n0].T, float32 x @ w[n0 : n0 + nf].T + bias) in one launch, or None where two are faster or one doesn't take these numbers of rows."""
    if x.dim() != 2 or not 0 < x.shape[0] <= 512 or n0 % 4 or nf < 1 or not _plain_rows(x, w) or _registered(x.shape[0], n0, w.shape[1]):
        return None
    m, (n, k) = x.shape[0], w.shape
    # the ring tiles also wherever gemm_few has no config.  Two launches -> one, us: 12304 x 4096, 64 rows 32.4 -> 25.3, 200 rows 49.1 -> 39.9;
    # 6160 x 2048, 100 rows 18.6 -> 12.7, 400 rows 26.5 -> 20.3; 3080 x 1024, 400 rows 13.0 -> 10.2.  512 rows are where this rule's
    # measurements ended and no line of speed (2064 x 2048, 512 rows 17.8 -> 13.2, 600 17.6 -> 13.2, 1500 23.6 -> 17.9).
    cfg = _few_more(m, n, k, 0)
    plan = _linear_plan(m, n0, k) if not cfg or _ring_more(m, n, k) else None
    if plan is not None and plan[0] in _RING and -(-(n0 + nf) // 4) * 4 <= n:   # (it stores in 4s)
        # the rows behind are one tile more, which must not be a round more
        bn, tiles = _PP_BN[plan[0]], -(-m // _PP_BM[plan[0]]) * plan[1]
        if -(-(-(-(n0 + nf) // bn) * tiles) // 256) <= -(-(-(-n0 // bn) * tiles) // 256):
            return _k().gemm_ring(x, w, plan[0], plan[1], 0, n0, nf, bias, 0.0, 0.0, 0.0)
    return _k().gemm_few(x, w, cfg, 0, n0, nf, bias, 0.0, 0.0, 0.0) if cfg else None


def join_rows_ok(m: int, k: int) -> bool:
    """Sizes at which a product's workgroups make a join's m rows of k columns themselves.  A decode step of four layers, us, joins as launches of
    their own -> in the products: one row of 1024 151 -> 144, of 2048 225 -> 214, of 4096 457 -> 446; 2 rows of 1024 155 -> 149; beyond, every workgroup's
    reading outweighs the launch: 3 rows of 1024 156 -> 158, 4 157 -> 160, 2 of 2048 231 -> 233."""
    return 0 < m and k % 256 == 0 and m * k <= (4096 if m == 1 else 2048)


def join_config(h: torch.Tensor, w: torch.Tensor, kind: int, n0: int = 0) -> int:
    """Config of gemm_join for the rows h that a post-norm join is to give, or 0 where the join and its product take two launches: kind 0 a product
    with float32 rows behind its first n0, 1 a plain one, 2 a gated unit, each where gemm_few's configs of one x tile have it alone."""
    m, (n, k) = h.shape[0], w.shape
    if not join_rows_ok(m, k) or n % 32 or n0 % 4 or not _plain_rows(h, w) or _registered(m, n0 or n, k):
        return 0
    if kind == 1:
        plan = _linear_plan(m, n, k)
        cfg = plan[0] - SK_BASE if plan is not None and plan[1] == 1 else 0
    else:
        cfg = 0 if _ring_more(m, n, k) else _few_more(m, n, k, kind)
    return cfg if cfg == 15 or (cfg == 14 and kind != 2) else 0


_Tensor, _WEIGHTS, _BF16 = torch.Tensor, (torch.Tensor, torch.nn.Parameter), torch.bfloat16
_autocast, _grad, _functorch, _forward_ad = torch.is_autocast_enabled, torch.is_grad_enabled, torch._C._are_functorch_transforms_active, torch.autograd.forward_ad


def _plain_rows(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Operands that the kernels take as they lie, and nothing that has to see the product (gradients, transforms,
    autocast, subclasses)."""
    return (type(x) is _Tensor and type(w) in _WEIGHTS and not _autocast("cuda") and x.dtype is _BF16 and w.dtype is _BF16 and w.dim() == 2
            and w.shape[1] == x.shape[-1] and w.is_cuda is x.is_cuda and w.get_device() == x.get_device()
            and not (_grad() and (x.requires_grad or w.requires_grad))
            and not _functorch() and _forward_ad._current_level < 0
            and x.is_contiguous() and w.is_contiguous() and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def pp_gemm(x: torch.Tensor, w: torch.Tensor, mode: int, plan: tuple[int, int], resid=None, part=None,
            eps: float = 1e-5, in_order: bool = False):
    """One launch of gemm_pp.hip (or gemm_skinny.hip for a skinny plan): returns (y, partials) — partials only for
    the residual epilogue.  ``in_order``: every workgroup sums K from its start (gemm_lg.hip's ring tiles may start elsewhere)."""
    if x.dim() != 2:
        x = x.reshape(-1, x.shape[-1])
    if plan[0] >= SK_BASE:
        return _k().gemm_skinny(x, w, mode, plan[0] - SK_BASE, plan[1], resid, part, eps)
    return _k().gemm_pp(x, w, mode, plan[0], plan[1], resid, part, eps, False, in_order)


# (M, N, K) -> bool predicate + kernel; extension point for further shape-specialised kernels
_custom: list[tuple[Callable[[int, int, int], bool], Callable[[torch.Tensor, torch.Tensor], torch.Tensor]]] = []


def register(pred: Callable[[int, int, int], bool], fn: Callable[[torch.Tensor, torch.Tensor], torch.Tensor]) -> None:
    _custom.append((pred, fn))


def _registered(m: int, n: int, k: int) -> bool:
    """Is a kernel registered for this product?  Then linear() calls it, and no launch that takes the product along with something else."""
    return bool(_custom) and any(pred(m, n, k) for pred, _ in _custom)


@dataclass
class ResidOut:
    """Output of a decode producer GEMV with the residual epilogue (``gemv_resid``): the new residual stream
    ``s = bf16(bf16(x @ w.T) + resid)`` and the per-workgroup partial sums of s^2 the next RMSNorm needs."""
    s: torch.Tensor
    part: torch.Tensor


@dataclass
class LazyNorm:
    """``rmsnorm(s) * w`` of a residual stream a ResidOut producer just wrote, not computed yet.

    Only built for models whose norm weights are folded into the consuming projections (``w`` is then ones).  A decode
    GEMV consumer (``linear`` / ``gate_up_silu`` / the fused QKV projection) applies it as one per-row scale of its
    outputs (csrc/kernels/gemv.hip NORMP: inv from the producer's partials), so the norm costs no launch; any other
    consumer calls ``materialize`` (the standalone RMSNorm kernel: equal up to rounding)."""
    s: torch.Tensor
    part: torch.Tensor
    w: torch.Tensor
    eps: float
    _y: Optional[torch.Tensor] = None

    @property
    def shape(self):
        return self.s.shape

    def rows(self) -> int:
        return self.s.numel() // self.s.shape[-1]

    def fusable(self) -> bool:
        return self.s.is_cuda and self._y is None

    def materialize(self) -> torch.Tensor:
        if self._y is None:
            from . import rmsnorm

            self._y = rmsnorm(self.s, self.w, self.eps)
        return self._y

    @staticmethod
    def force(x):
        """A tensor for anything that is not a GEMV consumer."""
        return x.materialize() if isinstance(x, LazyNorm) else x


def is_q(w) -> bool:
    """An fp8 projection weight (models/llama.py QTensor: e4m3 bytes ``q`` [N, K] + per-row scales ``s``)."""
    return not isinstance(w, torch.Tensor) and hasattr(w, "q") and hasattr(w, "s")


def gemv_q_ok(m: int, n: int, k: int) -> bool:
    """Shapes of the W8A16 decode GEMV (gemv.hip WQ: fp8 weights, bf16 activations): up to 4 rows (the fused
    norm / RoPE / residual epilogues: 2), whole 1 KiB weight chunks."""
    return m <= 4 and k % 1024 == 0 and n % 16 == 0


def _q_fallback(x, w, swiglu: bool = False) -> torch.Tensor:
    """fp8 weight off the W8A16 GEMV shapes: quantise the activations and run the W8A8 op."""
    from . import qlinear, quant_rows

    xq, xs = quant_rows(LazyNorm.force(x).reshape(-1, w.shape[1]))
    y = qlinear(xq, xs, w.q, w.s, swiglu)
    return y.view(*x.shape[:-1], y.shape[-1])


def gemv_resid(x: torch.Tensor, w: torch.Tensor, resid: torch.Tensor, in_order: bool = False) -> ResidOut:
    """Producer (O / down projection, TP=1): the new residual stream s = bf16(bf16(x @ w.T) + resid) and the RMSNorm
    partial sums of s^2, in one launch — the GEMV at M <= 2, the batched GEMM's kResid epilogue above.  ``w`` may be
    an fp8 QTensor at the W8A16 GEMV shapes (resid_ok(..., fp8=True)).  ``in_order``: as in :func:`linear`."""
    m, k = x.numel() // x.shape[-1], x.shape[-1]
    if is_q(w):
        s = torch.empty(resid.shape, dtype=resid.dtype, device=resid.device)
        part = _k().gemv_resid(x.reshape(-1, k), w.q, resid, s, w.s)
        return ResidOut(s, part)
    if m > GEMV_MAX_M:
        s, part = pp_gemm(x, w, PP_RESID, pp_plan(m, w.shape[0], k, PP_RESID), resid.reshape(m, -1), in_order=in_order)
        return ResidOut(s.view(resid.shape), part)
    s = torch.empty(resid.shape, dtype=resid.dtype, device=resid.device)
    part = _k().gemv_resid(x.reshape(-1, x.shape[-1]), w, resid, s)
    return ResidOut(s, part)


def resid_ok(m: int, n: int, k: int, fp8: bool = False) -> bool:
    """Shapes of the residual-epilogue producer: the M <= 2 GEMV shapes (gemv.hip kResid) and the batched GEMM's
    (gemm_pp.hip kResid) where the plan takes it; fp8 weights: the W8A16 GEMV shapes only."""
    if fp8:
        return m <= min(GEMV_MAX_M, 2) and gemv_q_ok(m, n, k)
    if m <= GEMV_MAX_M:
        return m <= 2 and gemv_ok(m, n, k)  # (the GEMV's residual epilogue: M <= 2)
    return pp_plan(m, n, k, PP_RESID) is not None


def gemv_ok(m: int, n: int, k: int, swiglu: bool = False) -> bool:
    """Shapes routed to the hand-written decode GEMV (csrc/kernels/gemv.hip): K % 512, N % 16, M <= GEMV_MAX_M (1 by
    default; M = 2 only below LM-head widths when raised)."""
    if k % 512 or n % 16:
        return False
    return m == 1 or (m <= GEMV_MAX_M and n <= 32768)


def mfma_swiglu_ok(m: int, n: int, k: int) -> bool:
    """Fused gate_up + SwiGLU on the MFMA GEMM: the measured winning range (3 <= M <= 128)."""
    return 3 <= m <= 128 and k % 64 == 0 and n % 128 == 0


def _gemv(x: torch.Tensor, w: torch.Tensor, swiglu: bool = False) -> torch.Tensor:
    k = x.shape[-1]
    y = _k().gemv(x.reshape(-1, k), w, swiglu)
    return y.view(*x.shape[:-1], y.shape[-1])


def mfma_gemm(x: torch.Tensor, w: torch.Tensor, swiglu: bool = False, stages: int = 3) -> torch.Tensor:
    k = x.shape[-1]
    y = _k().gemm(x.reshape(-1, k), w, swiglu, stages)
    return y.view(*x.shape[:-1], y.shape[-1])


def gate_up_silu(x: torch.Tensor, w_gu: torch.Tensor, in_order: bool = False) -> torch.Tensor:
    """silu(x @ gate.T) * (x @ up.T) with w_gu = [gate; up]: one fused launch (GEMV at M <= 2, the batched GEMM's
    SwiGLU epilogue above, with the folded input norm when x is a LazyNorm), else GEMM + silu_mul.  ``in_order``: as in :func:`linear`."""
    from . import silu_mul

    if is_q(w_gu):  # fp8 weights: the W8A16 GEMV (folded norm fused when x is a LazyNorm), else W8A8
        m, n, k = (x.rows() if isinstance(x, LazyNorm) else x.numel() // x.shape[-1]), w_gu.shape[0], x.shape[-1]
        if isinstance(x, LazyNorm) and x.fusable() and m <= 2 and gemv_q_ok(m, n, k):
            return _k().gemv_normp(x.s, x.part, x.eps, w_gu.q, True, w_gu.s)
        x = LazyNorm.force(x)
        if x.is_cuda and gemv_q_ok(m, n, k):
            y = _k().gemv(x.reshape(-1, k), w_gu.q, True, w_gu.s)
            return y.view(*x.shape[:-1], y.shape[-1])
        return _q_fallback(x, w_gu, True)
    if isinstance(x, LazyNorm):
        m, n, k = x.rows(), w_gu.shape[0], x.shape[-1]
        if x.fusable() and gemv_ok(m, n, k, swiglu=True):
            return _k().gemv_normp(x.s, x.part, x.eps, w_gu, True)
        plan = pp_plan(m, n, k, PP_SWIGLU) if x.fusable() else None
        if plan is not None:
            y, _ = pp_gemm(x.s, w_gu, PP_SWIGLU, plan, None, x.part, x.eps, in_order)
            return y.view(*x.shape[:-1], n // 2)
        x = x.materialize()
    if x.is_cuda:
        m, n, k = x.numel() // x.shape[-1], w_gu.shape[0], x.shape[-1]
        if gemv_ok(m, n, k, swiglu=True):
            return _gemv(x, w_gu, True)
        plan = pp_plan(m, n, k, PP_SWIGLU)
        if plan is not None:
            y, _ = pp_gemm(x, w_gu, PP_SWIGLU, plan, in_order=in_order)
            return y.view(*x.shape[:-1], n // 2)
        if mfma_swiglu_ok(m, n, k):
            return mfma_gemm(x, w_gu, True)
    return silu_mul(linear(x, w_gu, in_order=in_order))


def _linear_plan(m: int, n: int, k: int) -> Optional[tuple[int, int]]:
    """The rules' plan of a plain product whose operands _plain_rows takes, or None: one look-up for a shape that was here before."""
    key = (m, n, k, "linear", PP_MODE, GEMV_MAX_M)
    hit = _plan_cache.get(key, False)
    if hit is False:
        hit = (few_rows_plan(m, n, k) if m <= 64 else slab_rows_plan(m, n, k) if m >= MANY_MIN else None) or (mid_rows_plan(m, n, k) if 32 < m <= 512 else None)
        _plan_cache[key] = hit
    return hit


def linear(x, w: torch.Tensor, out: Optional[torch.Tensor] = None, in_order: bool = False) -> torch.Tensor:
    """x @ w.T.  ``in_order``: no workgroup of the hand-written tiles starts its sums over K elsewhere than at their start, as those over large weights
    otherwise do (gemm_lg.hip TURN), 4 to 10 % faster: for products in front of what is kept as bytes."""
    if is_q(w):  # fp8 weights: the W8A16 GEMV (folded norm fused when x is a LazyNorm), else W8A8
        m, n, k = (x.rows() if isinstance(x, LazyNorm) else x.numel() // x.shape[-1]), w.shape[0], x.shape[-1]
        if isinstance(x, LazyNorm) and x.fusable() and m <= 2 and gemv_q_ok(m, n, k):
            return _k().gemv_normp(x.s, x.part, x.eps, w.q, False, w.s)
        x = LazyNorm.force(x)
        if x.is_cuda and gemv_q_ok(m, n, k):
            y = _k().gemv(x.reshape(-1, k), w.q, False, w.s)
            return y.view(*x.shape[:-1], n)
        return _q_fallback(x, w)
    if isinstance(x, LazyNorm):
        m, n, k = x.rows(), w.shape[0], x.shape[-1]
        if x.fusable() and out is None and gemv_ok(m, n, k):
            return _k().gemv_normp(x.s, x.part, x.eps, w, False)
        plan = pp_plan(m, n, k, PP_PLAIN) if x.fusable() and out is None else None
        if plan is not None:
            y, _ = pp_gemm(x.s, w, PP_PLAIN, plan, None, x.part, x.eps, in_order)
            return y.view(*x.shape[:-1], n)
        x = x.materialize()
    if x.is_cuda:
        m, k = x.numel() // x.shape[-1], x.shape[-1]
        n = w.shape[0]
        few = None
        if out is None and m > 0 and _plain_rows(x, w):
            few = _linear_plan(m, n, k)
            if few is not None and not _custom and x.dim() == 2:   # (what follows, without the views)
                if few[1] > 1 and few[0] < SK_BASE and few[0] != 88:
                    return _k().gemm_split(x, w, few[0], few[1], in_order)
                return pp_gemm(x, w, PP_PLAIN, few, in_order=in_order)[0]
        if few is None and gemv_ok(m, n, k):
            return _gemv(x, w)
        for pred, fn in _custom:
            if pred(m, n, k):
                return fn(x, w)
        if few is not None and few[1] > 1 and few[0] < SK_BASE and few[0] != 88:   # a split without tickets
            return _k().gemm_split(x.reshape(-1, k), w, *few, in_order).view(*x.shape[:-1], n)
        plan = (few or pp_plan(m, n, k, PP_PLAIN)) if out is None else None
        if plan is not None:
            y, _ = pp_gemm(x, w, PP_PLAIN, plan, in_order=in_order)
            return y.view(*x.shape[:-1], n)
    if out is not None:
        return torch.matmul(x, w.t(), out=out)
    return torch.matmul(x, w.t())
