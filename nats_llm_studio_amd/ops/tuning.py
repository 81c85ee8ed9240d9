"""Launch-configuration selection for the quantised GEMV/GEMM kernels.

Measured per-shape winners (tools/tune_gemv.py on MI355X) live in `gemv_tuning.json`
next to this file: {"<type>:<rows>:<K>:<Mbucket>": [mode, waves, rt, ks]}. Shapes not in
the table use the heuristic below.
"""
from __future__ import annotations

import functools
import json
import math
import os

import numpy as np

_TABLE = None
_FORCED = set()        # keys of NLS_TUNING_EXTRA's entries: no rule below changes those launches
_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gemv_tuning.json")
MBUCKETS = (1, 2, 4, 8, 16, 32, 48, 64, 128, 256, 512, 1024, 2048)


def _mb(M: int) -> int:
    for b in MBUCKETS:
        if M <= b:
            return b
    return MBUCKETS[-1]


def key(segs, M: int) -> str:
    t = "+".join(str(s.w.type) for s in segs)
    rows = sum(s.w.rows for s in segs)
    return f"{t}:{rows}:{segs[0].w.K}:{_mb(M)}"


def table():
    global _TABLE
    if _TABLE is None:
        _TABLE = {}
        _FORCED.clear()
        if os.path.exists(_PATH):
            with open(_PATH) as f:
                _TABLE = {k: tuple(v) for k, v in json.load(f).items()}
        # A/B overrides without editing the table: NLS_TUNING_EXTRA='{"<key>": [..], ...}'
        # ... or from a file (NLS_TUNING_EXTRA_FILE, e.g. a fresh tune_gemv.py --out table), applied first
        path = os.environ.get("NLS_TUNING_EXTRA_FILE")
        if path:
            with open(path) as f:
                _TABLE.update({k: tuple(v) for k, v in json.load(f).items()})
        extra = os.environ.get("NLS_TUNING_EXTRA")
        if extra:
            _TABLE.update({k: tuple(v) for k, v in json.loads(extra).items()})
            _FORCED.update(json.loads(extra))
    return _TABLE


_MEMO, _MEMO_OF = {}, None


def memo() -> dict:
    """Configs worked out so far (ops.gemv_config), for the table as it is loaded."""
    global _MEMO, _MEMO_OF
    t = table()
    if _MEMO_OF is not t or len(_MEMO) > 8192:
        _MEMO, _MEMO_OF = {}, t
    return _MEMO


# Microseconds of a launch of quantised rows on shapes without a tuned entry, fitted to 39000 launches of 30 shapes (1536 to 128256 rows, K 1536 to 28672,
# Q4_K, Q5_K, Q6_K and Q8_0, the launch behind it included, weights streamed). (mode, waves, rt): workgroups that share a CU, and what a last round of at
# most one to a CU takes of a whole one; then of the launch: fixed, a round, a round's K (times bytes a weight up to 8 rows) / 4096, the same for each
# 16 rows, a second launch (RoPE, SwiGLU of split sums, norm), a million slab values, a MB of weights.
_FEW_US = (((0, 4, 1), 1, 1.0, (4.07, 0.97, 1.84, 0.0, 2.60, 0.0, 0.114)), ((0, 4, 2), 2, 0.6, (4.30, 3.00, 5.27, 0.0, 2.36, 0.0, 0.086)),
           ((1, 4, 1), 2, 0.6, (3.37, 2.95, 15.3, 0.0, 2.95, 8.58, 0.058)), ((1, 8, 1), 1, 1.0, (2.13, 3.30, 13.7, 0.0, 3.44, 10.2, 0.065)))
_SOME_US = (((0, 4, 1), 1, 1.0, (4.26, 0.90, 0.0, 3.37, 2.37, 0.0, 0.094)), ((0, 4, 2), 2, 0.6, (2.96, 4.73, 0.0, 6.48, 2.47, 0.0, 0.076)),
            ((1, 4, 1), 2, 0.7, (2.39, 4.79, 5.20, 4.62, 3.43, 2.29, 0.068)), ((1, 8, 1), 3, 0.5, (0.22, 10.4, 16.4, 5.76, 3.80, 2.97, 0.073)))
# ... above 64 rows, by (mode, rt): a round, its K / 4096, the same for the share of the block's rows in use, the second launch, a million slab values
_MID_US = {(2, 1): (2, 0.5, (9.03, 0.0, 54.3, 5.37, 1.39)), (2, 2): (1, 1.0, (5.49, 28.1, 7.31, 5.62, 1.81)), (2, 4): (1, 1.0, (7.70, 25.9, 25.6, 4.51, 1.62)),
           (3, 4): (2, 0.65, (5.94, 0.0, 40.2, 7.27, 0.74)), (3, 6): (2, 0.65, (8.91, 50.2, 0.0, 5.75, 1.20))}
_WEIGHT_BYTES = {8: 1.0625, 12: 0.5625, 13: 0.6875, 14: 0.8203}
_QUANT = frozenset(_WEIGHT_BYTES)


def _rounds(n: int, share: int, last: float) -> float:
    """Rounds of n workgroups, `share` of them to a CU; `last`: what a last round of at most one to a CU takes."""
    full, part = divmod(n, 256 * share)
    return full + (0.0 if not part else last if part <= 256 else 1.0)


@functools.lru_cache(maxsize=4096)
def _few_rule(rows, K: int, types, M: int, role: str):
    """The cheapest of paths A (up to 32 rows) and B for 2 to 64 rows of a shape without a tuned entry. us of all projections of a layer of a 2048-wide
    model at 2 / 4 / 16 / 32 / 48 rows, with the head, before and after (a rule that knew path B with 8 waves only from 9 rows on): Q4_K 164 -> 152,
    172 -> 155, 170 -> 170, 204 -> 203, 258 -> 241; Q5_K 181 -> 166, 186 -> 170, 226 -> 181, 247 -> 213, 265 -> 244; Q8_0 181 -> 175, 189 -> 180,
    237 -> 188, 262 -> 218, 271 -> 247."""
    nb, mt, total = K // 256, -(-M // 16), sum(rows)
    mb = sum(-(-n // 16) * 16 * K * _WEIGHT_BYTES[t] for n, t in zip(rows, types)) * 1e-6
    width = max(_WEIGHT_BYTES[t] for t in types) if M <= 8 else 1.0

    def us(fam, ks):
        (mode, waves, rt), share, last, c = fam
        tile = 16 * rt * (waves if mode else 1)
        k = _rounds(sum(-(-n // tile) for n in rows) * ks, share, last)
        kk = k * K / ks / 4096
        more = mode != 0 if role == "qkv" else ks > 1 if role in ("gateup", "lm_head") else True
        return (c[0] + c[1] * k + c[2] * kk * width + c[3] * kk * mt + c[4] * more + (c[5] * ks * M * total * 1e-6 if ks > 1 else 0.0) + c[6] * mb)
    (cfg, *_), ks = min(((f, ks) for f in (_FEW_US if M <= 8 else _SOME_US) for ks in (1, 2, 3, 4, 6, 8)
                         if (ks == 1 or f[0][0] == 1 and ks * 2 <= nb) and (f[0][0] == 1 or M <= 32)), key=lambda c: us(*c))
    return (*cfg, ks)


@functools.lru_cache(maxsize=4096)
def _mid_rule(rows, K: int, types, M: int, role: str):
    """65 to 255 rows: the cheapest of the LDS-dequant GEMM in blocks of 64 and 128 rows and (K-quants) the LDS-DMA GEMM in blocks of 64 and 96, 2.5 %
    behind the fastest of 90 configs on average. us of all projections of a layer of a 2048 / 4096-wide model with the head, 96 rows, before and
    after: Q4_K 377 -> 310, 555 -> 515; Q5_K 387 -> 325, 603 -> 530; Q8_0 (128-row tiles of path B, one launch on 16 of 256 CUs) 1042 -> 330, 1541 -> 550."""
    nb, total = K // 256, sum(rows)
    dma = 8 not in types                      # (raw Q8_0 tiles do not fit that kernel's LDS)

    def us(fam, ks):
        mode, rt = fam
        share, last, c = _MID_US[fam]
        bm = 64 * rt if mode == 2 else 16 * rt
        k = _rounds(sum(-(-n // 128) for n in rows) * -(-M // bm) * ks, share, last)
        kk = k * K / ks / 4096
        more = role != "gateup" or ks > 1
        return c[0] * k + c[1] * kk + c[2] * kk * min(M, bm) / bm + c[3] * more + (c[4] * ks * M * total * 1e-6 if ks > 1 else 0.0)
    (mode, rt), ks = min(((f, ks) for f in _MID_US for ks in (1, 2, 3, 4, 6, 8) if (ks == 1 or ks * 2 <= nb) and (dma or f[0] == 2)), key=lambda c: us(*c))
    return (mode, 8 if mode == 2 else 4, rt, ks)


def any_rows(segs, M: int):
    """More than 64 rows: the launch that takes rows of x and y at any place, through registers on both sides."""
    if not all(int(s.w.type) in _QUANT for s in segs):
        return (1, 8, 1, 1)      # MFMA GEMM: 128 weight rows x 128 activation rows per workgroup
    # LDS-dequant GEMM (mode 2): 128 weight rows x 256 (or 128) activation rows per workgroup;
    # split K until the grid covers the 256 CUs (the measured winners on the 8B shapes)
    tiles = sum((s.w.rows + 127) // 128 for s in segs) * ((M + 255) // 256)
    ks, nb = 1, segs[0].w.K // 256
    while tiles * ks < 256 and ks * 2 <= max(1, nb // 4):
        ks *= 2
    return (2, 8, 4 if M >= 192 else 2, ks)


def heuristic(segs, M: int):
    rows = sum(s.w.rows for s in segs)
    K = segs[0].w.K
    quant = all(int(s.w.type) in _QUANT for s in segs)
    # (up to 64 rows below 64 M weights: the others' bytes are most of their time, what the rule chooses there is 4 % faster, here 17 at 16 to 48 rows)
    if quant and 1 < M < 256 and (M > 64 or rows * K < 64 << 20):
        rule = _few_rule if M <= 64 else _mid_rule
        return rule(tuple(s.w.rows for s in segs), K, tuple(int(s.w.type) for s in segs), M, _role(segs))
    if M <= 8:
        # the batch-1 winners of every measured family (Llama-3-8B / -70B, Qwen2.5-7B, Mixtral; r03 sweeps,
        # profiles/b1_latency_r03.txt, profiles/b1_models_r03.txt): 4-wave workgroups; wide matrices (gate|up,
        # LM head) on path B's staged-x stream, fused Q|K|V on 32-row path-A tiles, the rest on 16-row ones.
        # The old (0, 8, 1, 1) default cost Llama-3-70B / Qwen2.5-7B ~30 % at batch 1.
        if rows >= 4 * K:
            return (1, 4, 2, 2) if rows >= 16 * K and K >= 1024 else (1, 4, 2, 1)
        return (0, 4, 2, 1) if len(segs) > 1 else (0, 4, 1, 1)
    if M > 64:
        if quant and (rows >= 4 * K or K >= 2 * rows):
            # wide (gate|up, LM head) and down-projection shapes: the quantised GEMM on the raw tile-blocks
            # (mode 9, 256 weight rows x 256 activation rows) won every measured one at M >= 256 -- Llama-3-8B
            # gate|up / LM head, Llama-3-70B gate|up / down / LM head by 10-20 % over mode 2
            # (profiles/tune_quant_70b_r05.txt); split K until the grid covers the 256 CUs.
            # Q8_0 too, path B / this (mode 2 where rows are not wide), us: 28672 x 4096 at 256 / 1000 / 3000 rows 120 / 113, 355 / 232, 1128 / 732,
            # 2048 x 8192 86 / 43, 85 / 59, 178 / 148, 6144 x 4096 51 / 36, 97 / 91, 250 / 223, but 16384 x 2048 at 256 37 / 49, 6144 x 4096 at 512 51 / 62
            tiles = sum((s.w.rows + 255) // 256 for s in segs) * ((M + 255) // 256)
            ks, nb = 1, K // 256
            while tiles * ks < 256 and ks * 2 <= min(8, max(1, nb // 4)):    # (ks <= 8: the tuned range)
                ks *= 2
            return (9, 8, 2, ks)
        return any_rows(segs, M)
    waves, rt = 8, 1
    tiles = sum((s.w.rows + waves * rt * 16 - 1) // (waves * rt * 16) for s in segs)
    ks = 1
    nb = K // 256
    while tiles * ks < 256 and ks * 2 <= max(1, nb // 2):
        ks *= 2
    return (1, waves, rt, ks)


def expert_heuristic(ws, T: int, per: float):
    """Path B config of a grouped launch over the experts `ws` (<= 8) for T tokens, `per` routed rows to an expert, or None: path A (up
    to 16 tokens) or the LDS-dequant GEMM. With few rows to an expert the launch is bound by the weights' bytes; path B streams
    them through registers, skips an expert's unused activation tiles, and wins as soon as its grid covers the 256 CUs.
    256 weight rows to a workgroup (us, path B / LDS-dequant GEMM / path A): Q5_K 8 x 8192 x 2048 at 8 / 24 / 64 / 96 tokens
    22 / - / 31, 25 / 40 / 62, 28 / 39 / -, 28 / 42 / -; at 128 37 / 43 even routing, 55 / 53 skewed, so not there; Q4_K 8 x 28672 x 4096 at
    24 tokens 107 / 197 / 237 (4 waves; with 8 waves 121: more than a workgroup to a CU). 64 weight rows: Q5_K 8 x 2048 x
    4096 at 16 / 24 / 64 tokens 16 / - / 15, 17 / 31 / 25, 20 / 32 / -; Q4_K 8 x 4096 x 4096 at 8 / 24 / 64 18 / - / 21, 22 / 30 / 39, 25 / 32 / -."""
    if T < 4 or not all(int(w.type) in (8, 12, 13, 14) for w in ws):
        return None
    big = sum((w.rows + 255) // 256 for w in ws)
    if big >= 256 and T <= 128 and per < 32:
        return (1, 4 if big > 256 and T <= 32 else 8, 2, 1)
    small = sum((w.rows + 63) // 64 for w in ws)
    if (small >= 512 and 4 < T <= 64) or (small >= 256 and 16 < T <= 64):
        return (1, 4, 1, 1)
    return None


def expert_gemm(ws, per: float, dma: bool = True):
    """Config (mode, waves, rt, ks) of a grouped launch over the experts `ws` (<= 8) at about `per` routed rows to an expert: the least time by rounds
    of workgroups over the 256 CUs, with microseconds of a round fitted to 14 shapes of eight experts and of eight out of 64 and 128, 768 to 28672 wide, at
    3 to 1500 rows (what it takes is 0.6 % behind the fastest on average). Mode 9 (256 x 256 tiles) takes long prompts, mode 3 (128 x 96, two
    workgroups to a CU) wide products of few rows and most counts of some hundred, mode 2 (128 x 256 and 128 x 128, multiplying only the 16-row tiles
    in use) few rows of narrow products. us at modes 2 rt 4 / 2 rt 2 / 3 rt 6 / 9: Q5_K 8192 x 2048 at 250 rows 150 / 159 / 127 / 146, at 540
    256 / 288 / 224 / 223, at 1000 418 / 488 / 411 / 360; Q6_K 2048 x 4096 at 50 rows 37 / 37 / 42 / 103, at 250 77 / 98 / 69 / 119; Q4_K
    28672 x 4096 at 64 rows 291 / 296 / 211 / 448, at 1000 2180 / 2661 / 2330 / 1813; Q6_K 4096 x 14336 at 64 rows 139 / 128 / 135 / 333, at 540
    660 / 741 / 623 / 782; Q4_K 1536 x 2048 of 128 at 24 rows 23 / 20 / 24 / 54. dma: mode 3 may be chosen."""
    return _expert_rule(len(ws), ws[0].rows, ws[0].K, frozenset(int(w.type) for w in ws), per, dma)


@functools.lru_cache(maxsize=4096)         # (a prompt's layers ask for the same)
def _expert_rule(E: int, N: int, K: int, types, per: float, dma: bool):
    far = per + per ** 0.5                 # rows of the larger experts

    def wgs(bn, bm):
        return E * -(-N // bn) * max(1, math.ceil(far / bm))

    def pair(n, us, one):                  # two workgroups to a CU; alone each is faster
        return us * one if n <= 256 else -(-n // 512) * us
    cand = {(2, 8, 4, 1): -(-wgs(128, 256) // 256) * (4.82 + 0.00558 * K + (4.24 + 0.00188 * K) * min(4, math.ceil(far / 64))),
            (2, 8, 2, 1): pair(wgs(128, 128), 9.93 + 0.00741 * K + (4.64 + 0.00191 * K) * min(4, math.ceil(far / 32)), 0.566)}
    if dma and types <= {12, 13, 14}:
        cand[3, 4, 6, 1] = pair(wgs(128, 96), 10.7 + 0.00812 * K + (8.09 + 0.00195 * K) * min(1, per / 96), 0.843)
    if types <= {8, 12, 13, 14}:
        cand[9, 8, 2, 1] = -(-wgs(256, 256) // 256) * (7.0 + 0.0233 * K + 20.0 * min(1, per / 256))
    return min(cand, key=cand.get)


def argmax_config(cfg, segs, M: int):
    """Config of a launch with an arg-max: path B unsplit ends in an atomic for every 16 weight rows and token, all on M neighbouring
    keys (32000 Q6_K rows, K = 4096, (1, 8, 1, 1): 62 us at 2 tokens, 108 at 8, 166 at 24, 248 at 64). Split in two, the reduce
    takes the maximum with few atomics: 26, 28, 34, 47; at K = 2048 2 / 8 / 24 / 64 tokens 58 / 105 / 150 / 217 -> 18 / 20 /
    25 / 34, one token 36 -> 19; on 16-row tiles, (1, 8, 1, 2), 24 / 26 / 30 / 36. Path A ends so as well (29 us at 2 tokens), where it was not measured
    with the arg-max."""
    if _FORCED and key(segs, M) in _FORCED:
        return cfg
    if (M <= 64 and sum(s.w.rows for s in segs) >= 8192 and segs[0].w.K >= 1024
            and (cfg[0] == 1 and 1 in cfg[2:] or cfg[0] == 0 and M > 1 and _tuned(segs, M) is None)):
        return (1, 4 if M == 1 else 8, 2, 2)
    return cfg


def dense_key(segs, M: int) -> str:
    return f"d:{sum(s.w.rows for s in segs)}:{segs[0].w.K}:{_mb(M)}"


# Microseconds of a round of workgroups, one to a CU: fixed (prologue, stores), and for 4096 of K, by (mode, rt, activation rows of a block). Fitted to
# 11700 launches of 33 shapes, 2048 to 152064 rows, K 2048 to 28672, at 70 to 4096 rows (each within 5 % on average).
_ROUND_US = {(10, 1, 256): (11.5, 101.5), (10, 1, 192): (8.5, 80.0), (10, 2, 256): (7.0, 60.0), (10, 2, 192): (6.0, 48.0), (10, 2, 320): (7.5, 71.5),
             (4, 2, 128): (4.5, 40.0)}


def _rows10(rt: int, tiles: int, M: int, ks: int) -> int:
    """Rows of mode 10's blocks: the launcher's choice (launch_dense10 of hgemm10.hip)."""
    def rounds(bm):
        return -(-tiles * -(-M // bm) * ks // 256) * bm
    low = 192 if rounds(192) * 100 < rounds(256) * (85 if rt == 1 else 100) else 256
    return 320 if rt == 2 and rounds(320) * 100 < rounds(low) * 97 else low


def dense_heuristic(segs, M: int, aligned: bool = True):
    """Dense f16 GEMM for shapes without a tuned "d:" entry, and above the tuned row counts: the cheapest of mode 10 with 256 or 128
    weight rows and mode 4 with 128 x 128 tiles, by the rounds of tiles over the 256 CUs; split-K slabs are written and read again.
    (A rule that took mode 4 below 1024 rows and mode 5 above ran a 32000-row head at 300 / 900 / 4096 rows in 161 / 742 / 2846 us;
    mode 10 takes 108 / 223 / 909.) aligned: the operands' row strides suit mode 10, whose stores are 4 columns wide."""
    aligned = aligned and all(s.w.rows % 4 == 0 and s.ycol % 4 == 0 for s in segs)
    return _dense_rule(tuple(s.w.rows for s in segs), segs[0].w.K, M, aligned)


@functools.lru_cache(maxsize=4096)         # (30 to 50 us to work out, and a prompt's launches ask once for each layer and projection)
def _dense_rule(rows, K: int, M: int, aligned: bool):
    nkt = K // 64

    def us(mode, rt, ks):
        bn = 256 if (mode, rt) == (10, 1) else 128
        tiles = sum((n + bn - 1) // bn for n in rows)
        bm = _rows10(rt, tiles, M, ks) if mode == 10 else 128
        fixed, per = _ROUND_US[mode, rt, bm]
        # one XCD's workgroups (it has every eighth weight tile) in rounds of its 32 CUs; a round that is not full takes 0.78 of its time at least
        full, part = divmod(-(-tiles // 8) * -(-M // bm) * ks, 32)
        n = full + (0.78 + 0.22 * part / 32 if part else 0)
        t = n * (fixed + per * K / ks / 4096)
        if bm == 320 and n > 4:
            t *= 1.05                     # (12288 x 4096 at 3200 rows 355 us, 313 on 256 x 256; 28672 x 4096 at 2880 7 % behind)
        slabs = ks * M * sum(rows)        # (f32 values; from 64 MB on they leave the caches)
        return t + ((7.0 if ks > 6 and M > 192 else 3.0) + 1.2e-6 * slabs + 4e-6 * max(0, slabs - (16 << 20)) if ks > 1 else 0.0)
    mode, rt, ks = min(((mode, rt, ks) for mode, rt in ([(10, 1), (10, 2)] if aligned else []) + [(4, 2)] for ks in range(1, 9)
                        if ks == 1 or nkt // ks >= 8), key=lambda c: us(*c))
    return (mode, 8 if mode == 10 or M < 128 else 16, rt, ks)


# What mode 11's forms are weighed against a launch of the other modes by, in microseconds: rounds of workgroups (of one XCD: it has every eighth weight
# tile, and 32 CUs; P is what a part of a round takes at least) times what a round takes, fixed and for 4096 of K; a MB of weights, which come from
# memory; a split's second launch (where there is none anyway), a million slab values, and those past 16 million, which leave the caches. By (mode, rt,
# activation rows of a block), fitted to 2000 launches of 27 shapes, 2048 to 57344 rows, K 2048 to 28672, at 128 to 4096 rows; 5 to 15 % each.
_DENSE_US = {(10, 1, 256): (0.5, 11.3, 94.7, 0.056, 14.9, 0.0, 1.27), (10, 1, 192): (0.7, 10.6, 76.5, 0.035, 7.3, 0.49, 0.57),
             (10, 2, 256): (0.6, 9.1, 59.9, 0.021, 7.7, 0.22, 0.87), (10, 2, 192): (0.78, 5.2, 47.8, 0.016, 6.9, 0.73, 0.52),
             (10, 2, 320): (0.5, 12.5, 70.3, 0.034, 7.3, 0.24, 0.63), (4, 2, 128): (0.85, 6.6, 30.8, 0.085, 6.0, 0.0, 0.59)}
# Mode 11's tiles are 32 nt weight rows x 32 mt activations, 3 <= nt <= 8, 3 <= mt <= 5 (the forms that are built); 9000 launches of the same shapes, 11 %
_NT11, _MT11 = (v.ravel() for v in np.meshgrid(np.arange(3, 9), np.arange(3, 6), indexing="ij"))


def _dense_us(rows, K: int, M: int, added: bool, mode: int, rt: int, ks: int) -> float:
    """Predicted time of a launch of mode 10 or 4 (those of mode 5 and other wave counts are taken for mode 4's)."""
    if mode != 10:
        mode, rt = 4, 2
    bn = 256 if (mode, rt) == (10, 1) else 128
    tiles = sum((n + bn - 1) // bn for n in rows)
    bm = _rows10(rt, tiles, M, ks) if mode == 10 else 128
    P, fixed, per, mb, second, slab, far = _DENSE_US[mode, rt, bm]
    full, part = divmod(-(-tiles // 8) * -(-M // bm) * ks, 32)
    n, slabs = full + (P + (1 - P) * part / 32 if part else 0.0), ks * M * sum(rows)
    return (n * (fixed + per * K / ks / 4096) + mb * sum(rows) * K * 2e-6
            + ((0.0 if added else second) + slab * slabs * 1e-6 + far * max(0, slabs - (16 << 20)) * 1e-6 if ks > 1 else 0.0))


def _best11(rows, K: int, M: int, added: bool):
    """(time, config) of mode 11's fastest form. All forms at once (0.1 ms a product; a prompt's length is new each time)."""
    ks = np.arange(1, 1 + max(1, min(8, K // 64 // 6)))[:, None]
    nt, mt = _NT11, _MT11
    tiles = sum(-(-n // (32 * nt)) for n in rows)
    full, part = np.divmod(-(-tiles // 8) * -(-M // (32 * mt)) * ks, 32)
    n = full + np.where(part > 0, 0.85 + 0.15 * part / 32, 0.0)
    slabs = np.where(ks > 1, ks * (M * sum(rows) * 1e-6), 0.0)
    t = (n * (2.16 + 0.201 * nt * mt + (0.39 + 0.252 * nt * mt + 3.41 * (nt + mt)) * K / ks / 4096) + 0.058 * sum(rows) * K * 2e-6
         + np.where(ks > 1, 0.0 if added else 5.6, 0.0) + 0.86 * slabs + 0.49 * np.maximum(0.0, slabs - 16.8))
    i = int(t.argmin())
    k, j = divmod(i, len(nt))
    return float(t.flat[i]), (11, 8, 512 + 16 * int(mt[j]) + int(nt[j]), k + 1)


def _launch_rows(segs):
    """Rows of a launch's segments, those whose f16 copies lie behind each other in one buffer (QWeight.expand_dense_group) as one. (Copies of
    their own may lie behind each other too, as the allocator deals them: the choice does not hang on that.)"""
    if len(segs) == 1:
        return (segs[0].w.rows,)
    rows, end = [], None
    for s in segs:
        d = getattr(s.w, "d16", None)
        at = (d.untyped_storage().data_ptr(), d.data_ptr()) if d is not None else None
        if at is not None and at == end:
            rows[-1] += s.w.rows
        else:
            rows.append(s.w.rows)
        end = None if at is None else (at[0], at[1] + 2 * s.w.rows * s.w.K)
    return tuple(rows)


MODE11_MAX_M = 2560          # (above, 256 x 256 tiles are as fast: 28672 x 4096 at 3000 rows 603 us, 633 on the best of mode 11, 2048 x 2048 45 and 45)


def _or_mode11(cfg, segs, M: int):
    """cfg, or mode 11's fastest form where that should be 5 % faster (times are known to 5 to 15 %: 1 % slower at worst on 138 measured products of 27 shapes,
    4.4 % faster on average). us before and after: 2048 x 2048 at 192 / 1500 rows 19 / 35 -> 14 / 29, 3072 x 2048 at 128 / 640 17 / 31 -> 15 / 19,
    16384 x 2048 at 128 / 512 30 / 45 -> 22 / 38, 6144 x 4096 at 320 / 640 39 / 53 -> 32 / 44, 5120 x 5120 at 128 / 1024 30 / 83 -> 25 / 71, 28672 x 4096 at 900
    210 -> 197. (Operands whose strides suit modes 10 and 11 only: stores are 4 columns wide. Unsplit blocks of 320 rows stay: faster in mode 11 where
    nothing but such launches runs, 85 -> 79 for 28672 x 4096 at 320 rows, but 80 either way in a step, between launches that draw less power.)"""
    if M > MODE11_MAX_M or any(s.w.rows % 4 or s.ycol % 4 for s in segs):
        return cfg
    return _mode11_or(tuple(cfg), _launch_rows(segs), segs[0].w.K, M, _role(segs) in ("o", "down"))


@functools.lru_cache(maxsize=4096)         # (a prompt's launches ask once for each layer and projection)
def _mode11_or(cfg, rows, K: int, M: int, added: bool):
    if len(rows) > 1:                      # (what was measured are whole products; a loaded model has Q, K and V copies behind each other)
        return cfg
    if cfg[0] == 10 and cfg[2:] == (2, 1) and _rows10(2, sum(-(-n // 128) for n in rows), M, 1) == 320:
        return cfg
    t, best = _best11(rows, K, M, added)
    return best if t < 0.95 * _dense_us(rows, K, M, added, cfg[0], cfg[2], cfg[3]) else cfg


def select_dense(segs, M: int):
    """Dense config, or None where the tuner measured the quantised GEMM faster (entry [-1])."""
    hit = table().get(dense_key(segs, M))
    if hit is not None and hit[0] < 0:
        return None
    # (the entries of 257 .. 320 and 513 .. 640 rows were measured at 512 and 1024, where other splits and blocks fill the rounds. us, entry / rule:
    # 28672 x 4096 at 320 rows, in blocks of 320, 89 / 81; 4096 x 4096 28.5 / 26.7 and 8192 x 8192 67 / 63, in four parts of K on blocks of 192;
    # 6144 x 4096 at 640 on mode 4 53 / 46, 10240 x 8192 149 / 120, 3584 x 3584 35 either way. 57344 x 8192 at 320 rows has an entry of its own: two
    # rounds of 320-row blocks there take 310 to 400, as the card holds its clock, 192 x 256 340 to 350)
    if dense_key(segs, M) not in _FORCED:
        if 256 < M <= 320 or 512 < M <= 640:
            hit = table().get(f"d:{sum(s.w.rows for s in segs)}:{segs[0].w.K}:{320 if M <= 320 else 640}")
        elif M > MBUCKETS[-1]:
            hit = None
    cfg = hit if hit is not None else dense_heuristic(segs, M)
    return cfg if dense_key(segs, M) in _FORCED else _or_mode11(cfg, segs, M)


# Llama-3-8B Q4_K_M shapes per projection role: the tuned entries an untuned shape of the same role borrows at
# the same batch bucket (M <= 64), e.g. Llama-3-70B / Qwen2.5-7B / Mixtral attention and dense FFN shapes
_ROLE_KEYS = {"qkv": "12+12+12:6144:4096", "o": "12:4096:4096", "gateup": "12:28672:4096", "down": "12:4096:14336",
              "lm_head": "14:128256:4096"}


def _role(segs) -> str:
    rows = sum(s.w.rows for s in segs)
    K = segs[0].w.K
    if len(segs) > 1:
        return "qkv"
    if rows >= 16 * K:
        return "lm_head"
    if rows >= 4 * K:
        return "gateup"
    if K >= 2 * rows:
        return "down"
    return "o"


def _role_entry(segs, M: int):
    """The Llama-3-8B entry of this shape's role and batch bucket, for a shape within 1.5x of that role's
    Llama-3-8B rows and K (Qwen2.5-7B, Mixtral attention: batch 16 / 64 2.70 / 4.30 vs 3.57 / 5.06 ms/step
    with the generic heuristic). Larger shapes keep the heuristic, whose split-K follows their own tile
    count (Llama-3-70B batch 64: 22.7 vs 24.4 ms/step borrowing); profiles/b1_models_r03.txt."""
    ref = _ROLE_KEYS[_role(segs)]
    _, rrows, rk = ref.split(":")
    rows, K = sum(s.w.rows for s in segs), segs[0].w.K
    near = lambda a, b: max(a, b) < 1.5 * min(a, b)
    if not (near(rows, int(rrows)) and near(K, int(rk))):
        return None
    return table().get(f"{ref}:{_mb(M)}")


def _tuned(segs, M: int):
    hit = table().get(key(segs, M))
    if hit is None and M <= 64 and os.environ.get("NLS_TUNING_ROLE", "1") == "1":
        hit = _role_entry(segs, M)
    return hit


def select(segs, M: int):
    hit = _tuned(segs, M)
    return hit if hit is not None else heuristic(segs, M)
