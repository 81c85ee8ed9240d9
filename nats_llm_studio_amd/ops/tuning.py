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


def heuristic(segs, M: int):
    rows = sum(s.w.rows for s in segs)
    K = segs[0].w.K
    if M <= 8:
        # the batch-1 winners of every measured family (Llama-3-8B / -70B, Qwen2.5-7B, Mixtral; r03 sweeps,
        # profiles/b1_latency_r03.txt, profiles/b1_models_r03.txt): 4-wave workgroups; wide matrices (gate|up,
        # LM head) on path B's staged-x stream, fused Q|K|V on 32-row path-A tiles, the rest on 16-row ones.
        # The old (0, 8, 1, 1) default cost Llama-3-70B / Qwen2.5-7B ~30 % at batch 1.
        if rows >= 4 * K:
            return (1, 4, 2, 2) if rows >= 16 * K and K >= 1024 else (1, 4, 2, 1)
        return (0, 4, 2, 1) if len(segs) > 1 else (0, 4, 1, 1)
    if M > 64:
        if all(int(s.w.type) in (12, 13, 14) for s in segs):
            if M >= 256 and (rows >= 4 * K or K >= 2 * rows):
                # wide (gate|up, LM head) and down-projection shapes: the quantised GEMM on the raw tile-blocks
                # (mode 9, 256 weight rows x 256 activation rows) won every measured one at M >= 256 -- Llama-3-8B
                # gate|up / LM head, Llama-3-70B gate|up / down / LM head by 10-20 % over mode 2
                # (profiles/tune_quant_70b_r05.txt); split K until the grid covers the 256 CUs
                tiles = sum((s.w.rows + 255) // 256 for s in segs) * ((M + 255) // 256)
                ks, nb = 1, K // 256
                while tiles * ks < 256 and ks * 2 <= min(8, max(1, nb // 4)):    # (ks <= 8: the tuned range)
                    ks *= 2
                return (9, 8, 2, ks)
            # LDS-dequant GEMM (mode 2): 128 weight rows x 256 (or 128) activation rows per workgroup;
            # split K until the grid covers the 256 CUs (the measured winners on the 8B shapes)
            tiles = sum((s.w.rows + 127) // 128 for s in segs) * ((M + 255) // 256)
            ks, nb = 1, K // 256
            while tiles * ks < 256 and ks * 2 <= max(1, nb // 4):
                ks *= 2
            return (2, 8, 4 if M >= 192 else 2, ks)
        return (1, 8, 1, 1)      # MFMA GEMM: 128 weight rows x 128 activation rows per workgroup
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
    25 / 34, one token 36 -> 19; on 16-row tiles, (1, 8, 1, 2), 24 / 26 / 30 / 36."""
    if _FORCED and key(segs, M) in _FORCED:
        return cfg
    if cfg[0] == 1 and 1 in cfg[2:] and M <= 64 and sum(s.w.rows for s in segs) >= 8192 and segs[0].w.K >= 1024:
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
    return hit if hit is not None else dense_heuristic(segs, M)


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


def select(segs, M: int):
    hit = table().get(key(segs, M))
    if hit is None and M <= 64 and os.environ.get("NLS_TUNING_ROLE", "1") == "1":
        hit = _role_entry(segs, M)
    return hit if hit is not None else heuristic(segs, M)
