"""Device ops of the config-driven decoder stacks: ctypes bindings of `_stack.so` (csrc/stack/*.hip, gfx950).

GPU tensors only: there is no eager form of these ops, a missing library raises. Operands are bf16 (f32 accumulation,
f32 norms / routing / softmax / recurrences) or, for 32-bit models, f32 throughout (f32 MFMA, or f32 in three bf16 parts)."""
from __future__ import annotations

import contextlib
import ctypes
import os
from functools import lru_cache
from typing import List, Optional

import torch

_PKG = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB_PATH = os.environ.get("NLS_STACK_SO") or os.path.join(_PKG, "_stack.so")

P, I, L, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_long, ctypes.c_float
SEGS = 6
EPI = {"none": 0, "silu": 1, "tanh": 2, "sigmoid": 3, "relu2": 4, "decay": 5, "gate": 6, "rope": 7,
       "geglu": 8, "sigpow": 9, "softcap": 10, "swiglu": 11, "siluglu": 12}
NO_BLOCK = 1 << 30       # LinSeg.cb: output columns are not blocked


class LinSeg(ctypes.Structure):
    """csrc/stack/lin.h LinSeg."""
    _fields_ = [("w", P), ("x", P), ("y", P), ("bias", P), ("gate", P), ("cs", P), ("pos", P), ("rows", P), ("xmap", P),
                ("wstride", L), ("ldx", L), ("ldy", L), ("xgs", L), ("ygs", L), ("yks", L),
                ("N", I), ("nsub", I), ("M", I), ("ng", I), ("epi", I), ("yact", I), ("cb", I), ("cstep", I),
                ("xdiv", I), ("ldg", I), ("half", I), ("alpha", F),
                ("ks", I), ("pad0", I)]


class LinArgs(ctypes.Structure):
    _fields_ = [("s", LinSeg * SEGS), ("tiles", P), ("ntiles", P), ("nseg", I), ("maxtiles", I),
                ("begin", I * (SEGS + 1)), ("nmt", I * SEGS)]


_SIGS = {
    "nls_lin_args_size": [],
    "nls_lin_small": [P, I, I, I, I, P],
    "nls_lin_gemm": [P, I, I, P],
    "nls_stack_embed": [P, P, P, P, I, I, F, P, P, L, I, P, P, L, I, P, I, I, I, P, P, P, P, I, P, P, P],
    "nls_norm_add": [P, L, P, I, L, P, P, L, P, L, P, P, P, P, L, P, I, I, I, F, I, I, I, I, L, P],
    "nls_row_norm": [P, L, P, P, P, P, P, L, P, L, I, I, F, I, I, I, P],
    "nls_poly_norm": [P, L, P, P, L, I, I, F, I, P],
    "nls_attn_rows": [P, P, P, L, P, P, P, P, P, P, L, P, P, L, I, I, I, I, I, I, I, I, I, F, I, P],
    "nls_talk_rows": [P, L, P, P, P, I, I, P, P, I, I, I, I, I, I, F, I, P, P, L, P, L, P, L, P, P, P, I, I, I, I, I, I, I, P],
    "nls_talk_decode": [P, L, P, P, P, I, I, P, P, I, I, I, I, I, I, F, I, P, P, L, P, L, P, L, P, P, P, I, I, I, P],
    "nls_talk_prefill": [P, L, P, P, P, I, I, P, I, I, I, I, I, I, F, I, P, P, L, P, L, P],
    "nls_gqa_attn": [P, L, P, P, P, I, I, P, P, I, I, I, I, I, F, P, L, P, L, P, P, P, I, I, I, I, I, P],
    "nls_gqa_prefill": [P, L, P, P, P, P, I, P, I, P, L, I, I, I, I, I, F, I, I, I, P],
    "nls_delta_conv": [P, L, P, P, L, P, L, P, L, P, P, I, I, I, I, I, I, I, I, P],
    "nls_delta_scan": [P, P, P, L, P, L, P, L, P, L, P, L, P, P, L, P, L, F, P, L, P, I, I, I, I, I, I, P, P, I, I, P],
    "nls_delta_step": [P, P, P, L, P, L, P, L, P, L, P, P, P, P, I, P, L, P, P, I, L, P, L, P, I, P, P, L, I, I, I, I, F, I, P],
    "nls_gla_scan": [P, P, P, L, P, L, F, P, L, P, P, L, P, L, F, P, L, P, I, I, I, I, I, P, P, I, I, P],
    "nls_gla_step": [P, P, P, L, P, L, P, P, P, I, F, F, P, L, P, I, P, P, L, P, L, P, L, I, I, I, F, I, P],
    "nls_attn_step": [P, L, P, P, P, I, I, P, P, I, I, I, I, F, P, L, P, L, I, I, P, P, P, P, P, P, L, P, L, P, P, P, I, F, F, P, L, P, P, P, L, P,
                      L, I, I, I, F, I, P],
    "nls_latent_rows": [P, L, I, P, P, L, P, L, I, I, I, P, P, P, P, P, L, I, F, I, P],
    "nls_stack_argmax": [P, L, I, P, I, P],
    "nls_moe_plan": [P, L, I, I, I, I, I, I, I, F, P, P, I, P, P, P, I, P, P],
    "nls_shift_mix": [P, L, P, P, L, P, L, L, P, P, I, I, I, P],
    "nls_wkv_scan": [P, P, P, L, P, L, P, P, L, P, L, P, L, P, L, I, P, I, I, I, I, P],
    "nls_scan_out": [P, L, P, P, L, P, L, I, I, I, F, I, P],
    "nls_wkv_step": [P, P, P, L, P, L, P, P, L, P, L, P, L, I, P, I, P, P, L, P, L, I, I, F, I, P],
    "nls_expand_plan": [P, I, I, P, I, I, P, P, P],
    "nls_latent_prefill": [P, L, I, P, L, I, P, P, P, L, P, P, I, P, I, P, L, I, I, I, I, I, I, I, F, P],
    "nls_latent_attn": [P, P, P, P, P, P, I, I, P, P, I, I, I, I, I, F, I, P],
}

_lib = None


def lib():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(f"HIP kernel library missing: {LIB_PATH} (run `python -m nats_llm_studio_amd.build`)")
        lb = ctypes.CDLL(LIB_PATH)
        for name, args in _SIGS.items():
            fn = getattr(lb, name)
            fn.argtypes = args
            fn.restype = I
        if lb.nls_lin_args_size() != ctypes.sizeof(LinArgs):
            raise RuntimeError("stale _stack.so: LinArgs layout mismatch (rebuild the kernels)")
        _lib = lb
    return _lib


def _check(rc: int, name: str):
    if rc != 0:
        raise RuntimeError(f"{name} failed with code {rc}")


def _p(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def stream(dev) -> int:
    return torch.cuda.current_stream(dev).cuda_stream


def pad_to(n: int, m: int) -> int:
    return (n + m - 1) // m * m


def act_ld(n: int) -> int:
    """Row stride of an activation that feeds a linear layer of n inputs: the packed weights' padded K."""
    return pad_to(n, 64)


# ---------------------------------------------------------------------------
# Linear layers
# ---------------------------------------------------------------------------

class PackedLinear:
    """[groups, N, K] weights in the packed layout of csrc/stack/lin.h (1 KiB sub-tiles in MFMA fragment order), bf16
    or f32. A plain matrix is one group; experts and per-head products are stacked groups."""

    def __init__(self, w: torch.Tensor, f32: bool, device):
        if w.dim() == 2:
            w = w[None]
        G, N, K = w.shape
        self.groups, self.N, self.K, self.f32 = G, N, K, f32
        dt, ks, el = (torch.float32, 16, 4) if f32 else (torch.bfloat16, 32, 8)
        Np, Kp = pad_to(N, 16), act_ld(K)
        self.nsub = Kp // ks
        self.data = torch.empty(G, Np * Kp, dtype=dt, device=device)
        step = max(1, (1 << 28) // (Np * Kp))               # groups per conversion pass
        for g0 in range(0, G, step):
            a = w[g0:g0 + step].to(device=device, dtype=dt)
            a = torch.nn.functional.pad(a, (0, Kp - K, 0, Np - N))
            a = a.view(-1, Np // 16, 16, Kp // ks, 4, el).permute(0, 1, 3, 4, 2, 5)
            self.data[g0:g0 + step] = a.reshape(-1, Np * Kp)
        self.wstride = Np * Kp * dt.itemsize

    @property
    def nbytes(self) -> int:
        return self.data.numel() * self.data.element_size()


class Seg:
    """One segment of a LinLaunch. y / x: 2-D buffers (row stride = their stride(0)); ycol / xcol: first column.
    xgs / ygs: column step per group. block = (cb, cstep): output column n -> (n / cb) * cstep + n % cb.
    routed = (entry list, xdiv): the rows are routed entries (x row = entry / xdiv, y row = entry).
    rope = (table, pos, pairs). alpha: constant of the epilogue (sigmoid, sigpow, softcap, swiglu); sigpow: `gate`,
    a vector, gives an exponent per column instead. geglu, swiglu, siluglu: the rows of w alternate gate and up, y has half as many
    columns. slabs: K splits that a launch may use; y holds that many slabs of slab_rows rows, or as many of a larger launch's rows as
    fit, added by the caller (LinLaunch.run returns how many were written)."""

    def __init__(self, w: PackedLinear, x: torch.Tensor, y: torch.Tensor, epi: str = "none", ycol: int = 0,
                 xcol: int = 0, xgs: int = 0, ygs: int = 0, block=None, bias=None, gate=None, routed=None, rope=None,
                 yrow: int = 0, xmap: Optional[torch.Tensor] = None, alpha: float = 1.0, slabs: int = 1, slab_rows: int = 0):
        if x.stride(1) != 1 or y.stride(1) != 1:
            raise ValueError("row-major operands")
        if xcol + (0 if routed else (w.groups - 1) * xgs) + act_ld(w.K) > x.stride(0):
            raise ValueError(f"x rows ({x.stride(0)}) do not cover the padded K of {w.K} inputs")
        if x.dtype != w.data.dtype:
            raise TypeError(f"activations must be {w.data.dtype}, got {x.dtype}")
        if (xcol * x.element_size()) % 16 or (x.stride(0) * x.element_size()) % 16 or (xgs * x.element_size()) % 16:
            raise ValueError("activation rows must be 16-byte aligned")
        self.w, self.y, self.x = w, y, x
        self.rows_cap = min(x.shape[0] * (routed[1] if routed else 1), y.shape[0] - yrow)
        if xmap is not None:               # x row of row m: xmap[m] (the caller keeps the entries inside x)
            self.rows_cap = min(xmap.numel(), y.shape[0] - yrow)
        s = self.s = LinSeg()
        s.w = w.data.data_ptr()
        s.x = x.data_ptr() + xcol * x.element_size()
        s.y = y.data_ptr() + (yrow * y.stride(0) + ycol) * y.element_size()
        s.bias, s.gate = _p(bias), _p(gate)
        s.ldg = gate.stride(0) if gate is not None else 0
        s.wstride, s.ldx, s.ldy, s.xgs, s.ygs = w.wstride, x.stride(0), y.stride(0), xgs, ygs
        s.N, s.nsub, s.ng, s.epi = w.N, w.nsub, w.groups, EPI[epi]
        s.yact = int(y.dtype != torch.float32)
        s.cb, s.cstep = block if block else (NO_BLOCK, 0)
        s.xdiv = 1
        if routed:
            s.rows, s.xdiv = routed[0].data_ptr(), routed[1]
        if rope:
            s.cs, s.pos, s.half = rope[0].data_ptr(), rope[1].data_ptr(), rope[2]
        s.xmap = _p(xmap)
        s.alpha = alpha
        if slabs * slab_rows > y.shape[0]:
            raise ValueError("y does not hold the slabs")
        s.ks, self.slabs, self.slab_rows = 1, slabs, slab_rows
        s.yks = slab_rows * y.stride(0)
        self.keep = (bias, gate, routed, rope, xmap)


def PAIR(nt: int, mt: int) -> int:
    """lin_gemm's config of lin_pair.hip's tile of 32 nt weight rows x 32 mt rows."""
    return 256 + 16 * nt + mt


# (weight rows, rows) of lin_gemm's configs
GEMM_TILES = {0: (64, 64), 1: (128, 64), 2: (128, 128), 3: (256, 128), 4: (256, 256), 5: (64, 64), 6: (192, 128), 7: (256, 256),
              8: (96, 64), 9: (160, 64), 10: (128, 64), 11: (96, 128), 12: (64, 32),
              **{PAIR(n, m): (32 * n, 32 * m) for n, m in ((4, 4), (4, 5), (5, 4), (6, 4), (6, 5), (8, 4), (8, 5))}}
THIN = 13                # config of products of up to 128 inputs straight from memory, 64 weight rows x 128 rows


# 32-bit operands: microseconds of 32 input columns on a CU that runs one workgroup of a tile, more for each further one, and how many run
# together; 0 to 2 in bf16 parts (lin_split.hip), 5 on the f32 MFMA (1.3 us more a launch). One workgroup to a CU splits and multiplies in turn, and
# the f32 MFMA is the faster one: 64 x 64, parts / f32, us: 65 x 4096 x 12288 356 / 226, 64 x 16384 x 4096 130 / 88, 256 x 2048 x 8704 249 / 162, in eight
# splits 64 x 2048 x 8704 41 / 28.6; with two it loses (128 x 10240 x 4096 138 / 147), with four it takes 1.4 times as long. Up to 128 inputs
# parts win (64 x 2048 x 128 6.9 / 7.6). 22 shapes x 16 row counts x 4 tiles x 1 to 8 splits lie 7 % around it, the tile it picks is 0.6 % behind the
# fastest on average, tile and splits 1.5 %. 64 x 64 / 128 x 64 / 128 x 128 in parts, us: 900 x 20096 x 2048 467 / 432 / 394 (f32 658), 1500 x 35888 x 4096
# 2621 / 2223 / 2020 (3440).
SPLIT_US = {0: (0.78, 0.30, 6), 1: (1.09, 0.49, 4), 2: (1.66, 0.87, 3), 5: (0.57, 0.57, 3)}

# bf16 launches of more than 64 rows, microseconds: fixed, then for a round of 256 workgroups of a tile, 1000 input columns of it, the same for the share of
# the CUs that a round uses, a MB of weights. Fitted to 13500 launches of 23 shapes (640 to 35888 outputs, 1024 to 17408 inputs, 65 to 3000 rows, 1 to 8
# splits of K) that lie 3 to 6 % around it. The tile it picks is 0.8 % behind the fastest of these on average; weighing rounds by a tile's multiply rate was
# 4 to 8 % behind (300 x 4096 x 9216 57 / 34 us, 200 x 14336 x 2048 31 / 25, 300 x 24576 x 4096 89 / 65, 800 x 10240 x 4096 83 / 68), the tiles without PAIR
# (lin_pair.hip) 5 % (300 x 10240 x 4096 47 / 38 us).
TILE_US = {5: (2.71, 2.74, 2.72, 0.71, 0.063), 8: (5.54, 0.23, 3.61, 0.69, 0.063), 10: (2.74, 3.17, 4.79, 0.88, 0.054), 11: (3.11, 3.76, 5.69, 1.14, 0.036),
           7: (2.85, 11.5, 14.1, 6.61, 0.0), 3: (1.65, 7.86, 9.78, 2.78, 0.057), 6: (2.86, 5.35, 7.53, 2.44, 0.056),
           PAIR(4, 4): (2.35, 5.38, 5.41, 1.75, 0.069), PAIR(4, 5): (2.60, 6.49, 6.51, 2.00, 0.048), PAIR(5, 4): (2.89, 6.35, 6.73, 1.61, 0.056),
           PAIR(6, 4): (2.70, 6.68, 6.49, 2.69, 0.074), PAIR(6, 5): (2.78, 8.07, 7.72, 2.91, 0.055), PAIR(8, 4): (1.20, 9.64, 8.21, 3.02, 0.079),
           PAIR(8, 5): (1.68, 11.3, 9.65, 3.38, 0.054)}


class LinLaunch:
    """A launch of up to SEGS independent linear layers, bound to its buffers once (only the row count and the launch
    config change from step to step)."""

    def __init__(self, segs: List[Seg], plan: "MoePlan" = None):
        self.segs, self.plan = segs, plan
        self.f32 = int(segs[0].w.f32)
        self.a = LinArgs()
        for i, s in enumerate(segs):
            self.a.s[i] = s.s
        self.a.nseg = len(segs)
        if plan is not None:
            self.a.tiles, self.a.ntiles = plan.tiles.data_ptr(), plan.ntiles.data_ptr()
        self._cfg = {}
        self._rows, self._ldy = segs[0].slab_rows, segs[0].y.stride(0)
        self.slab_rows = self._rows              # rows from slab to slab of the last run

    def _tiles(self, bn: int, bm: int, M: int) -> int:
        """Workgroups of a launch with bn x bm tiles."""
        n = 0
        for s in self.segs:
            nt = (s.w.N + bn - 1) // bn
            n += nt * (self.plan.expect_tiles(M, bm) if s.s.rows else s.w.groups * ((M + bm - 1) // bm))
        return n

    def config(self, M: int):
        """(False, mt, nw, rt): few-row kernel with mt activation tiles, nw waves and rt weight tiles per workgroup; or
        (True, c): GEMM config c."""
        if self.plan is not None:
            bm = self.plan.bm(M)
            if bm == 16:
                return False, 1, (4 if self._tiles(16, 16, M) >= 1536 else 8), 1
            if bm == 256:                 # (refused in 32 bits, whose tiles have up to 128 rows)
                return True, 7
            if self.f32:
                # (one list to an expert, each weight from memory once: two workgroups to a CU are not enough for parts either; eight experts of
                # 4096 x 3072, 8 to 38 rows each 125 us, on the f32 MFMA 114)
                if bm == 64 and M * self.plan.top <= 64 * self.plan.experts and self._tiles(64, 64, M) <= 512:
                    return True, 5
                return True, min((5, 0, 1) if bm == 64 else (2,), key=lambda c: self.split_us(c, M))
            if bm == 64:
                # short products are over before the deeper tiles' stages pay: 64 x 64 / chosen by rounds, us: 64 experts of 30 rows, 512 x 2048 28 / 41
                # and 2048 x 512 35 / 48; 8 of 30, 3072 x 2048 22.5 / 25.9; 32 of 30, 4096 x 1536 86 / 94; at 3072 inputs 24.2 / 23.6, from there
                # on 8 x 4096 x 6144 95 / 79, 8 x 6144 x 4096 79 / 77
                return True, 0 if self.segs[0].w.K < 3072 else self.balanced(M)
            return True, (3 if self._tiles(256, 128, M) >= 224 else 2)
        n16, n64 = self._tiles(16, 16, M), self._tiles(64, 64, M)
        ns = max(s.w.nsub for s in self.segs)
        if M <= 16:
            # 16 rows, streaming / GEMM, us: 10240 x 4096 23.7 / 18.2, 12288 x 2048 14.3 / 12.4, 17944 x 2048 18.7 / 16.4, 34816 x 4096 58.1 / 50.4, 8192 x
            # 2048 and narrower 9 / 11; 9 rows 19.2 / 18.7, 11.4 / 12.4, 17.4 / 16.9, 52.3 / 50.2
            if M > 12 and not self.f32 and ns >= 64 and n64 > 128:
                return True, 12 if n64 <= 256 else self.balanced(M)
            if M > 8 and n16 >= 1024:
                return False, 1, 4, 2
            return False, 1, (4 if ns <= 16 else 8 if n16 >= 320 or ns <= 32 else 16), 1
        if n16 <= 64:                     # a router's few outputs: split K over a workgroup's waves
            return False, 1, 16, 1
        if M <= 64 and not self.f32 and ns > 16:
            return self.few_rows(M, n64)
        if M <= 64:
            if n64 >= 250:
                return True, min((5, 0), key=lambda c: self.split_us(c, M)) if self.f32 else 0
            return False, 2, (4 if ns <= 16 else 8), (2 if M > 32 or n16 >= 640 else 1)
        if ns <= 4:                       # a step or two of K: all epilogue. 64 x 64 / 128 x 64 / straight from memory, us: 600 x 2048 x 64
            # 7.2 / 8.0 / 7.8, 2000 12.3 / 11.0 / 10.9, 4000 19.0 / 18.0 / 16.9; 4000 x 4096 x 64 25.4 / 23.5 / 19.2, 600 x 4096 x 128 7.8 / 7.9 / 8.7
            if not self.f32 and self._tiles(64, 128, M) >= 512:
                return True, THIN
            return True, (0 if M <= 2048 or not self.f32 else 1)
        if n64 < 96 and n16 <= 1024:
            return False, 1, 16, 1
        if self.f32:
            return True, min(SPLIT_US, key=lambda c: self.split_us(c, M))
        return True, min(self.tiles(M), key=lambda c: self.tile_us(c, M))

    def tiles(self, M: int):
        """The tiles that a bf16 launch of more than 64 rows chooses from."""
        cand = [5, 8, 10, 11] + ([7] if min(s.w.nsub for s in self.segs) >= 6 else [])       # (7: its DMA runs two steps ahead)
        if M <= 128 or any(getattr(s.s, "xmap", None) or getattr(s.s, "ldx", 0) >> 22 or s.w.nsub >> 16 for s in self.segs):
            return cand + [3, 6]                # (lin_pair.hip takes no row maps, and offsets of 32 bits)
        return cand + [c for c in TILE_US if c >= 256] + [3, 6]

    def tile_us(self, c: int, M: int, ks: int = 1) -> float:
        """About the microseconds of a bf16 launch on tile c in ks splits of K."""
        fixed, per_round, per_k, busy, mb = TILE_US[c]
        n = self._tiles(*GEMM_TILES[c], M) * ks
        # (long prompts: from the third round on the phased tile, whose workgroups stay, is faster in a running step, 2994 x 12288 x 4096 249 us, 269 on
        # PAIR(8, 5). Fewer rows fill its tiles badly: a pass of 600 on four products of 35888 x 4096 1.61 ms, 1.53 on PAIR(6, 5))
        if c >= 256 and n > 512 and M > 1024:
            return float("inf")
        k = max(s.w.nsub for s in self.segs) * 0.032 / ks
        return fixed + -(-n // 256) * (per_round + per_k * k) + n / 256 * busy * k + mb * 1.024e-3 * sum(s.w.groups * -(-s.w.N // 16) * s.w.nsub for s in self.segs)

    def balanced(self, M: int) -> int:
        """The GEMM config of launches with up to 64 rows to a tile, which read each weight once: the tile whose rounds of 256 workgroups
        sum up to the fewest weight rows; of equals the largest (four stages also keep such workgroups from sharing a CU while
        another has none), up to 40 rows the smallest. In a running step at 64 rows and K = 4096 (64 / 96 / 128 / 160 weight rows): N = 35888
        85 / 75 / 98 / 73 us, 34816 75 / 68 / 92 / 63, 24576 57 / 53 / 57 / 63; eight experts, N = 6144: 99 / 94 / 107 / 119, and N = 4096 at
        K = 6144: 115 / 99 / 82 / 85. Equals, 64 / 128 weight rows, one launch after another: 64 x 26880 50.4 / 44.5, 64 x 32000 54.0 / 52.3
        (in the step 65 / 68), 24 rows 41.7 / 43.7 and 47.8 / 51.0."""
        small = 1 if M <= 40 and self.plan is None else -1
        return min((10, 9, 8, 0), key=lambda c: (-(-self._tiles(*GEMM_TILES[c], M) // 256) * GEMM_TILES[c][0], small * GEMM_TILES[c][0]))

    def few_rows(self, M: int, n64: int):
        """17 to 64 rows, bound by the weights' bytes: the streaming kernel with the smallest tiles (weight rows x rows) that give each CU
        no more than one workgroup. 16 x 32 / 32 x 32 / 32 x 64, us: 24 x 4096 x 4096 13.4 / 19.0 / 15.1 (in the GEMM 19.4), 32 x 2048 x 9728
        28.7 / 40.6 / 33.1, 64 rows of it 31.5 / 42.6 / 52.7; 64 x 4096 x 17408 101.6 / 77.1 / 93.7, 40 rows of it 101.3 / 75.7 / 70.6;
        64 x 6144 x 2048 19.7 / 17.4 / 14.2."""
        if self._tiles(16, 32, M) <= 256:
            return False, 2, 8, 1
        if M > 48 and self._tiles(32, 32, M) <= 256:
            return False, 2, 8, 2
        if self._tiles(32, 64, M) <= 256:
            return False, 4, 8, 2
        if n64 <= 256:                    # 48 x 10240 x 4096: 27 us with 8 stages in flight, 35 streaming; 24 rows: 20 on 64 x 32, 24
            return (True, 5) if M > 32 else (True, 12) if self.segs[0].w.nsub >= 64 else (False, 2, 4, 2)
        return True, self.balanced(M)

    def split_us(self, c: int, M: int, ks: int = 1) -> float:
        """About the microseconds of an f32 launch on tile c in ks splits of K (without the 5 us that any takes)."""
        one, more, together = SPLIT_US[c]
        full, rest = divmod(-(-self._tiles(*GEMM_TILES[c], M) * ks // 256), together)
        step = full * (one + more * (together - 1)) + (one + more * (rest - 1) if rest else 0)
        return max(s.w.nsub for s in self.segs) / (2 * ks) * step + (1.3 if c == 5 else 0)

    def split_config(self, M: int):
        """(config, K splits) of a launch of up to slab_rows rows that may split K."""
        n16 = self._tiles(16, 16, M)
        # 64 x 32 tiles, up to one to a CU (a few more take a second round: 24 x 2560 x 4096 8.9 us in six splits, 12.9 in seven). 16 rows, streaming /
        # these, us: 4096 x 17408 27.5 / 25.6, 4096 x 8192 15.3 / 14.6, 4096 x 4096 9.1 / 9.6, 2048 x 8704 9.9 / 10.3; 24 rows 28.6 / 25.5, 19.3 / 15.5, 13.5 / 10.6,
        # 12.1 / 10.8; 5120 x 4096 15.6 / 11.8, 2560 x 4096 9.7 / 8.9, 640 x 6144 7.9 / 7.8. Short launches end before the ring's first stages are in:
        # 24 x 2048 x 2048 6.2 / 7.0, 1024 x 4096 6.8 / 7.2, 3072 x 2048 7.2 / 7.7. 14 x 7 layers x 17, 24 and 32 rows: 0.914 of streaming's time on average.
        Kd, n32 = self.segs[0].w.K, self._tiles(64, 32, M)
        if not self.f32 and (16 < M <= 32 and (Kd >= 6144 or n32 >= 64 or n32 * Kd >= 48 * 3072) or 12 < M <= 16 and n16 >= 256 and Kd >= 8192):
            return (True, 12), max(1, 256 // n32)
        if M <= 16:
            rt = 1 if M <= 8 else 2
            return (False, 1, 8, rt), -(-512 * rt // (2 * n16)) if M > 8 else -(-512 // n16)
        if M <= 32:
            return (False, 2, 4, 4 if n16 >= 256 else 2), 8
        if not self.f32 and M <= 64:      # one workgroup to a CU, 8 stages in flight: 64 x 4096 x 17408 34 us in 8 splits of 64 x 64 with
            small = self._tiles(64, 64, M)                                      # three, 31 in 4 (and half the slabs), 40 x 4096 x 9216 19, 18
            return ((True, 0), -(-512 // small)) if small > 256 else ((True, 5), 256 // small)
        c, ks = self.cheapest(M, self.segs[0].slabs)
        return (True, c), ks

    def cheapest(self, M: int, most: int):
        """(config, splits) of the least time for a launch with up to `most` slabs of K; each further slab is written and read again (about
        4 TB/s)."""
        s = self.segs[0]

        def us(c, ks):
            if self.f32:
                return self.split_us(c, M, ks) + (ks - 1) * M * s.w.N * 2e-6
            return self.tile_us(c, M, ks) + (ks - 1) * M * s.w.N * 2e-6
        return min(((c, ks) for c in (SPLIT_US if self.f32 else self.tiles(M)) for ks in range(1, max(1, min(most, s.w.nsub // 16)) + 1)), key=lambda v: us(*v))

    def tall_split(self, M: int):
        """(config, K splits) of more rows than slab_rows: as many slabs of M rows as y holds. A narrow product has fewer tiles than
        there are CUs, or lasts two rounds for a few more. 2000 x 4096 x 17408: 269 us in one round of 256 x 128 -> 209 in two splits of
        256 x 256 (292 -> 230 with the launch that adds the slabs); the passes of 600 tokens of a model 4096 wide 2446 -> 1895 us."""
        s = self.segs[0]
        c, ks = self.cheapest(M, min(s.slabs, s.y.shape[0] // self.slab_step(M)))
        return ((True, c), ks) if ks > 1 or c == 5 else (self.config(M), 1)

    def slab_step(self, M: int) -> int:
        """Rows from slab to slab: those the segment was bound for, or M of a larger launch, up to a multiple of 4 (the launch that adds
        the slabs takes no other distances where a row is not whole groups of 4 columns)."""
        return self._rows if M <= self._rows else (M + 3) & -4

    def choice(self, M: int):
        """(config, K splits) of a launch of M rows."""
        s = self.segs[0]
        splits = s.slabs > 1 and len(self.segs) == 1 and s.w.nsub >= 64
        if splits and M <= self._rows:
            cfg, ks = self.split_config(M)
            return cfg, max(1, min(ks, s.slabs, s.w.nsub // 16))
        if splits:
            return self.tall_split(M)
        return self.config(M), 1

    def run(self, M: int, st: int) -> int:
        """Returns the slabs of output rows that were written (1 unless a segment may split K), `slab_rows` rows apart."""
        if self.plan is not None:
            self.a.maxtiles = self.plan.max_tiles(M)
        for i, s in enumerate(self.segs):
            if (M * self.plan.top if s.s.rows else M) > s.rows_cap:
                raise ValueError(f"linear launch: {M} rows but the buffers hold {s.rows_cap}")
            self.a.s[i].M = M
        cfg = self._cfg.get(M)
        if cfg is None:
            if len(self._cfg) > 4096:
                self._cfg.clear()
            cfg = self._cfg[M] = self.choice(M)
        cfg, ks = cfg
        self.slab_rows = self.slab_step(M)
        self.a.s[0].ks, self.a.s[0].yks = ks, self.slab_rows * self._ldy
        if cfg[0]:
            _check(lib().nls_lin_gemm(ctypes.byref(self.a), self.f32, cfg[1], st), "nls_lin_gemm")
        else:
            _check(lib().nls_lin_small(ctypes.byref(self.a), self.f32, *cfg[1:], st), "nls_lin_small")
        return ks


class MoePlan:
    """Expert choice and routed-entry lists of one step (csrc/stack/stack_ops.hip moe_plan_kernel), shared by the layers
    of a step. Scores: sigmoid of the router logits, or their softmax; the `keep` groups with the largest score (the sum of
    their `group_best` best) of `groups` stay eligible; a chosen expert's weight is score * scale. tall: the products' tiles may have 256 rows (lin_gemm config 7)."""

    def __init__(self, cap: int, experts: int, top: int, groups: int, keep: int, scale: float, device, score: str = "sigmoid",
                 group_best: int = 2, tall: bool = False):
        self.tall = tall
        self.softmax, self.group_best = {"sigmoid": 0, "softmax": 1}[score], group_best
        self.experts, self.top, self.groups, self.keep, self.scale = experts, top, groups, keep, scale
        i32 = dict(dtype=torch.int32, device=device)
        self.topw = torch.zeros(cap * top, dtype=torch.float32, device=device)
        self.sel = torch.zeros(cap * top, **i32)
        self.rows = torch.zeros(cap * top, **i32)
        self.tiles = torch.zeros(self.max_tiles(cap, 16), 4, **i32)
        self.ntiles = torch.zeros(4, **i32)

    def bm(self, T: int) -> int:
        """Rows per tile of the expert products at T tokens."""
        avg = T * self.top / self.experts
        # 256 rows: eight experts of 875 rows took 251 -> 175 us at N = 6144, K = 2048 and 204 -> 149 us at N = 2048, K = 6144; from about
        # 160 rows on an expert's last tile wastes less than the phased kernel gains
        return 16 if avg <= 6 else 64 if avg <= 96 else 256 if self.tall and avg >= 160 else 128

    @staticmethod
    def takes_tall(f32: bool, *inputs: int) -> bool:
        """Whether products of these input widths run on 256-row tiles."""
        return not f32 and all(act_ld(k) >= 192 for k in inputs)

    def max_tiles(self, T: int, bm: Optional[int] = None) -> int:
        bm = bm or self.bm(T)
        n = T * self.top
        return max(1, min(n, self.experts + n // bm))

    def expect_tiles(self, T: int, bm: int) -> int:
        """About how many tiles T tokens make (launch rules)."""
        n = T * self.top
        return max(1, min(n, self.experts), n // bm)

    def run(self, z: torch.Tensor, T: int, st: int, ctx_len: Optional[torch.Tensor] = None):
        """ctx_len: rows without keys (a step's padding) are not routed."""
        _check(lib().nls_moe_plan(z.data_ptr(), z.stride(0), T, self.experts, self.top, self.groups, self.keep,
                                  self.softmax, self.group_best, self.scale, self.topw.data_ptr(), self.sel.data_ptr(), self.bm(T),
                                  self.rows.data_ptr(), self.tiles.data_ptr(), self.ntiles.data_ptr(),
                                  self.max_tiles(T), _p(ctx_len), st), "nls_moe_plan")


# ---------------------------------------------------------------------------
# Row kernels
# ---------------------------------------------------------------------------

def embed(ids, table: torch.Tensor, x: torch.Tensor, xb: Optional[torch.Tensor], T: int, st: int, prev=None,
          scale: float = 1.0, copies=(), pairs=None, positions=None, add: Optional[torch.Tensor] = None):
    """x = table[id] * scale (xb: its bf16 rounding). copies: up to two more of x in the activation type, of one row stride.
    pairs = (table, buckets, mul_prev, mul_cur, previous token of each slot, runs, tok_seq): plus the row of the token pair, and
    the slots' tokens move on. positions = (table, pos): plus the position's row. add: plus a vector."""
    nx, up = prev if prev is not None else (None, None)
    c0, c1 = (tuple(copies) + (None, None))[:2]
    pt, nb, mp, mc, pv, runs, seq = pairs if pairs is not None else (None, 0, 0, 0, None, None, None)
    tab, pos = positions if positions is not None else (None, None)
    _check(lib().nls_stack_embed(ids.data_ptr(), _p(nx), _p(up), table.data_ptr(), table.shape[0], table.shape[1], scale,
                                 x.data_ptr(), _p(xb), x.stride(0), T, _p(c0), _p(c1), c0.stride(0) if c0 is not None else 0,
                                 int(c0 is not None and c0.dtype == torch.float32), _p(pt), nb, mp, mc, _p(pv), _p(runs), _p(seq),
                                 _p(tab), tab.shape[0] if tab is not None else 0, _p(pos), _p(add), st), "nls_stack_embed")


def norm_add(y: torch.Tensor, w: Optional[torch.Tensor], x: torch.Tensor, xb: Optional[torch.Tensor], T: int, eps: float,
             st: int, plan: Optional[MoePlan] = None, shared_row0: int = -1, out_norm: Optional[torch.Tensor] = None,
             out: Optional[torch.Tensor] = None, rms: bool = False, slabs: int = 1, slab_rows: int = 0, out_norm2=None, out2=None,
             keep: bool = True, add: Optional[torch.Tensor] = None, groups: int = 1):
    """x[:T] += norm(y) * w, or += y without w (xb: a copy in the activation type); y may be the sum of `slabs` blocks of
    slab_rows rows. With `plan`, y holds the routed experts' rows (token-major) and from row `shared_row0` on the shared
    expert's, combined first. out = norm(x) * out_norm (what the next sublayers read, or the model's last norm), out2 the same
    with out_norm2. norm: layer norm, or RMS (of `groups` equal parts of a row each on its own). add: a vector that comes on top of
    x; keep False: the old x is left out."""
    D = y.shape[1] if w is None else w.numel()
    typed = out if out is not None else xb
    if out2 is not None and out2.stride(0) != out.stride(0):
        raise ValueError("norm_add: equal row strides of the outputs")
    _check(lib().nls_norm_add(y.data_ptr(), y.stride(0), _p(plan.topw) if plan else None, plan.top if plan else 0,
                              shared_row0, _p(w), x.data_ptr(), x.stride(0), _p(xb), xb.stride(0) if xb is not None else 0,
                              _p(out_norm), _p(out), _p(out_norm2), _p(out2), out.stride(0) if out is not None else 0, _p(add),
                              int(keep), D, T, eps, int(typed is not None and typed.dtype == torch.float32), int(rms), groups, slabs,
                              slab_rows * y.stride(0), st), "nls_norm_add")


def row_norm(x: torch.Tensor, rows: Optional[torch.Tensor], w: torch.Tensor, out: torch.Tensor, n: int, eps: float,
             st: int, rms: bool = False, w2=None, out2=None, gate: Optional[torch.Tensor] = None, groups: int = 1):
    """out[i] = norm(x[rows[i]]) * w (rows None: row i) (* gate[i]): layer norm, or RMS (of `groups` parts each on its own). out2: the
    same with w2."""
    if (out2 is not None and out2.stride(0) != out.stride(0)) or (gate is not None and gate.dtype != out.dtype):
        raise ValueError("row_norm: equal row strides of the outputs, a gate of their type")
    _check(lib().nls_row_norm(x.data_ptr(), x.stride(0), _p(rows), w.data_ptr(), out.data_ptr(), _p(w2), _p(out2), out.stride(0),
                              _p(gate), gate.stride(0) if gate is not None else 0, w.numel(), n, eps,
                              int(out.dtype == torch.float32), int(rms), groups, st), "nls_row_norm")


def poly_norm(z: torch.Tensor, act: torch.Tensor, out: torch.Tensor, N: int, T: int, eps: float, st: int):
    """out = a rms(z) + b rms(z^2) + c rms(z^3) + e over rows of N columns, powers by element; act: (a, b, c, e)."""
    if z.dtype != out.dtype or act.numel() != 4 or N > min(z.stride(0), out.stride(0)):
        raise ValueError("poly_norm: equal types, rows of N columns, four factors")
    _check(lib().nls_poly_norm(z.data_ptr(), z.stride(0), act.data_ptr(), out.data_ptr(), out.stride(0), N, T, eps,
                               int(out.dtype == torch.float32), st), "nls_poly_norm")


def argmax(logits: torch.Tensor, n: int, out: torch.Tensor, st: int):
    _check(lib().nls_stack_argmax(logits.data_ptr(), logits.stride(0), logits.shape[1], out.data_ptr(), n, st),
           "nls_stack_argmax")


def latent_rows(dq, wq, cq, dkv, wc, R: int, Rp: int, rot: int, cs, pos, slot, cache, T: int, eps: float, st: int):
    """cq = RMSNorm(dq) * wq; with `dkv`: the tokens' cache rows [RMSNorm(dkv[:R]) * wc | rotated dkv[R:]]."""
    _check(lib().nls_latent_rows(dq.data_ptr(), dq.stride(0), wq.numel(), wq.data_ptr(), cq.data_ptr(), cq.stride(0),
                                 _p(dkv), dkv.stride(0) if dkv is not None else 0, R, Rp, rot, _p(wc), cs.data_ptr(),
                                 pos.data_ptr(), slot.data_ptr(), _p(cache), cache.stride(0) if cache is not None else 0,
                                 T, eps, int(cq.dtype == torch.float32), st), "nls_latent_rows")


LATENT_TILES = (1, 2, 3, 4, 6, 8, 12, 16)     # padded latent widths / 64 the attention kernels are built for


def latent_pad(R: int) -> int:
    for n in LATENT_TILES:
        if R <= 64 * n:
            return 64 * n
    raise ValueError(f"latent width {R} > {64 * LATENT_TILES[-1]}")


def latent_head_groups(H: int, Rp: int) -> int:
    """Workgroups a (token, split) of latent_attention takes: 16 heads each, or 32 (csrc/stack/latent_attn.hip launch_r)."""
    return -(-H // (32 if H > 16 and Rp < 1024 else 16))


def rot_pad(rot: int) -> int:
    if rot > 128:
        raise ValueError(f"rotated width {rot} > 128")
    return 64 if rot <= 64 else 128


def latent_attention(q, cache, out, part, block_tables, block_size: int, tok_seq, ctx_len, T: int, H: int, ns: int,
                     Rp: int, rp: int, scale: float, st: int):
    po, pm = part if part is not None else (None, None)
    if ns > 1 and (po.numel() < T * H * ns * Rp or pm.numel() < T * H * ns * 2):
        raise ValueError("latent_attention: split workspace too small")
    _check(lib().nls_latent_attn(q.data_ptr(), cache.data_ptr(), out.data_ptr(), _p(po), _p(pm), block_tables.data_ptr(),
                                 block_tables.stride(0), block_size, tok_seq.data_ptr(), ctx_len.data_ptr(), T, H, ns,
                                 Rp, rp, scale, int(q.dtype == torch.float32), st), "nls_latent_attn")


BLOCK_INTS = 8           # int32 words per span / query block of the row plan (StackModel.row_blocks)
EXPAND_UNITS = {"key": (32, 64, 128), "rot": (32, 64), "value": (32, 64, 128)}      # per-head widths of latent_prefill


def expand_width(kind: str, n: int) -> Optional[int]:
    return next((w for w in EXPAND_UNITS[kind] if n <= w), None)


def expand_plan(spans, nspans: int, maxctx: int, block_tables, block_size: int, xmap, actx, st: int):
    """xmap: cache slots of the spans' contexts; actx (optional): key counts of the rows, cleared inside the spans."""
    _check(lib().nls_expand_plan(spans.data_ptr(), nspans, maxctx, block_tables.data_ptr(), block_tables.stride(0),
                                 block_size, xmap.data_ptr(), _p(actx), st), "nls_expand_plan")


def latent_prefill(qn, qns: int, q, Rp: int, qrs: int, kx, vx, cache, xmap, blocks, nblocks: int, waves: int, gate, out,
                   H: int, dku: int, dr: int, dv: int, vdim: int, scale: float, st: int, groups: int = 1):
    """Causal attention of query blocks over expanded keys / values; the rotated parts sit at column Rp of q and cache. groups: 2 splits a
    block's keys between two groups of waves (waves 4)."""
    _check(lib().nls_latent_prefill(qn.data_ptr(), qn.stride(0), qns, q.data_ptr() + Rp * q.element_size(), q.stride(0), qrs,
                                    kx.data_ptr(), vx.data_ptr(), cache.data_ptr() + Rp * cache.element_size(),
                                    cache.stride(0), xmap.data_ptr(), blocks.data_ptr(), nblocks, gate.data_ptr(),
                                    gate.stride(0), out.data_ptr(), out.stride(0), H, dku, dr, dv, vdim, waves, groups, scale, st),
           "nls_latent_prefill")


def shift_mix(x, mu, prev, out: torch.Tensor, runs, tok_seq, T: int, st: int):
    """out [mixes, rows, ld]: x + (previous token's x - x) * mu[s]; `prev` [slots, D] precedes each run's first row."""
    _check(lib().nls_shift_mix(x.data_ptr(), x.stride(0), mu.data_ptr(), prev.data_ptr(), prev.stride(0), out.data_ptr(),
                               out.stride(1), out.stride(0), runs.data_ptr(), tok_seq.data_ptr(), mu.shape[1], T,
                               int(out.dtype == torch.float32), st), "nls_shift_mix")


def wkv_scan(r, k, v, w, u, o, state, x, prev, runs, nruns: int, H: int, D: int, st: int):
    """The recurrence over each run's tokens; state [slots, H * D * D] and prev [slots, width] are carried on."""
    _check(lib().nls_wkv_scan(r.data_ptr(), k.data_ptr(), v.data_ptr(), r.stride(0), w.data_ptr(), w.stride(0),
                              u.data_ptr(), o.data_ptr(), o.stride(0), state.data_ptr(), state.stride(0), x.data_ptr(),
                              x.stride(0), prev.data_ptr(), prev.stride(0), prev.shape[1], runs.data_ptr(), nruns, H, D,
                              int(r.dtype == torch.float32), st), "nls_wkv_scan")


def wkv_step(r, k, v, w, u, state, x, prev, runs, nruns: int, norm, gate, out, H: int, D: int, eps: float, st: int):
    """wkv_scan and wkv_out of runs of one token each."""
    _check(lib().nls_wkv_step(r.data_ptr(), k.data_ptr(), v.data_ptr(), r.stride(0), w.data_ptr(), w.stride(0), u.data_ptr(),
                              state.data_ptr(), state.stride(0), x.data_ptr(), x.stride(0), prev.data_ptr(),
                              prev.stride(0), prev.shape[1], runs.data_ptr(), nruns, norm.data_ptr(), gate.data_ptr(),
                              gate.stride(0), out.data_ptr(), out.stride(0), H, D, eps, int(out.dtype == torch.float32),
                              st), "nls_wkv_step")


def scan_out(o, norm, gate, out, H: int, D: int, T: int, eps: float, st: int):
    """out = (o / rms(o) per head of D columns) * norm * gate."""
    _check(lib().nls_scan_out(o.data_ptr(), o.stride(0), norm.data_ptr(), gate.data_ptr(), gate.stride(0), out.data_ptr(),
                              out.stride(0), H, D, T, eps, int(out.dtype == torch.float32), st), "nls_scan_out")


# A chunked recurrence over 65 to 128 channels and more than 64 value columns, in microseconds: a workgroup has a CU to itself, so
# what counts is whole rounds of 256 of them, each as long as a segment. (launches, a token of the last pass, a token of the pass
# that finds what the segments end with, what segments add, the chain of their states: per segment in all, per segment of a run,
# workgroups of that pass per one of the last.) Fitted to 400 launches of 1 to 64 runs of 60 to 3500 tokens, 16 and 32 heads of
# 128 x 128, 1 to 16 segments: the count it picks is 0.6 % (gla) and 0.2 % (delta) behind the fastest on average.
SEGMENT_US = {"gla": (32.4, 0.3424, 0.1862, -10.0, 0.05, 0.0, 1), "delta": (52.5, 0.59, 0.35, -36.0, 0.2215, 9.0, 2),
              # the same on 64 value columns (narrow_shape), delta with the norm's launch behind it; 160 launches of 1 to 214 runs, 15 %
              "gla1": (9.17, 0.311, 0.0593, 3.97, 0.0404, 1.3, 1), "delta1": (12.9, 0.483, 0.182, 0.0, 0.0818, 12.4, 2)}


def segments_us(kind: str, tokens: int, wgs: float, nseg: int) -> float:
    """What a scan takes with nseg segments of its longest run (tokens); wgs: workgroups of that length, segments aside."""
    a, tok, tok_local, b, chain, link, lanes = SEGMENT_US[kind]
    size = -(-tokens // nseg) + 63 & ~63               # (segments are whole chunks of 64 tokens, the last one what is left)
    m = -(-tokens // size)
    size = min(size, tokens)
    us = a + -(-wgs * m // 256) * size * tok
    return us + (b + -(-wgs * lanes * (m - 1) // 256) * size * tok_local + chain * wgs * m + link * m if m > 1 else 0)


@lru_cache(maxsize=1024)
def segments(kind: str, T: int, tokens: int, wgs: int, most: int) -> int:
    """The fastest number of segments, up to `most`, of a scan over T rows whose runs have at most `tokens`; wgs: workgroups of
    one run. Short runs have one: the fit does not see what three launches cost them (100 tokens, us, one / two: gla 49.4 / 56.2, delta 79 / 112; 150
    tokens, one / three: gla 69 / 59, delta 113 / 126)."""
    if tokens < (129 if kind == "gla" else 192):
        return 1
    return min(range(1, max(1, min(-(-tokens // 64), most)) + 1), key=lambda s: segments_us(kind, tokens, wgs * T / tokens, s))


def gla_shape(T: int, nruns: int, H: int, V: int, D: int = 64, longest: Optional[int] = None):
    """(segments, groups of 64 value columns per workgroup) of a gla_scan launch; longest: tokens of the longest run, if known.
    Up to 64 channels two workgroups per CU, unless whole runs already give one: one segment up to 128 tokens (65 tokens, 32 heads of 64 x 128, us, one /
    two 26.6 / 34.8, 128 tokens 32.2 / 35.7, 150 in one / three 42.0 / 36.2), then as many as there are chunks of 64, since a segment has whole ones (333
    tokens cut for five 57, for six 42); 0.1 % behind the fastest count on average, no size slower than with T / 64 rounded down. There a CU holds
    several workgroups. With 65 to 128 channels that rule was 11 % behind, as it does not see a last round that is nearly empty (32 heads of 128 x 128, bf16: 6 runs of 650 tokens 382 us with 3
    segments, 265 with 1; 1 run of 333 tokens 93 us with 5, 63 with 6): the count is the one that segments_us finds fastest."""
    nt = 1 if V <= 64 else 2
    wgs = H * -(-V // (64 * nt))
    most = min(-(-512 // (wgs * nruns)), 16)             # (what bounds the scratch, too)
    if 64 < D <= 128 and nt == 2:
        return segments("gla", T, longest or -(-T // nruns), wgs, most), nt
    if longest is None:                                  # (no run can have more tokens than this)
        return 1 if wgs * nruns >= 256 else max(1, min(most, (T - nruns + 1) // 64)), nt
    return 1 if wgs * nruns >= 256 or longest <= 128 else min(most, -(-longest // 64)), nt


def narrow_shape(kind: str, shape, T: int, nruns: int, H: int, V: int, D: int, longest: Optional[int], f32: bool):
    """The shape of a launch over 65 to 128 channels and more than 64 value columns, or that of workgroups of 64 columns: half of the products to each,
    and (delta) LDS for four chunks, which the four waves prepare side by side; with 128 columns two of them do and two wait. They are the faster ones
    where whole rounds of CUs are not lost: twice as many, all at once (delta in 32 bits: always). The head's norm is then a launch of its own.
    us with 128 / 64 columns, 128 x 128, bf16: delta, 16 heads, 6 runs of 650 tokens 451 / 301, 7 of 86 79 / 63, 1 of 40 40 / 31, 1 of 700 228 / 198; 32
    heads, 1 of 330 189 / 152, 3 of 700 468 / 318, but 8 of 300 253 / 296; 32 bits 6 x 650 565 / 336, 214 of 16 519 / 474; plain, 16 heads, 1 of 330
    59 / 49, 6 of 650 209 / 196. What it picks is 1 % behind the fastest on average, 128 columns were 16 (32 bits: 30) and 6 (8) %."""
    nseg, nt = shape
    if nt != 2 or not 64 < D <= 128:
        return shape
    tokens = longest or -(-T // nruns)
    wide, narrow = H * -(-V // 128), H * -(-V // 64)
    most = min(-(-(256 if kind == "delta" else 512) // (wide * nruns)), 16, max(1, -(-tokens // 64)))     # (as much scratch as the shape's)
    fit = [s for s in range(1, most + 1) if narrow * nruns * s <= 256 or (s == 1 and f32 and kind == "delta")]
    us = lambda s: segments_us(kind + "1", tokens, narrow * T / tokens, s)
    best = min(fit, key=us, default=None)
    if best is None or not (f32 and kind == "delta") and us(best) >= segments_us(kind, tokens, wide * T / tokens, nseg):
        return shape
    return best, 1


def gla_scan(q, k, v, a, qscale: float, o, norm, gate, out, state, runs, nruns: int, H: int, D: int, V: int, eps: float, shape,
             seg, st: int):
    """Gated linear attention over each run's tokens: q, k [rows, H * D], v [rows, H * V] of one buffer (equal strides), decays
    a; state [slots, H * D * V] is carried on. With `out` (a head's columns fit a workgroup): its norm, `norm` and `gate`
    applied, else the plain outputs in `o` (scan_out follows). shape: gla_shape; seg: (states, decay products) scratch of its
    segments."""
    nseg, nt = shape
    if nseg > 1 and (seg[0].numel() < nruns * nseg * H * D * V or seg[1].numel() < nruns * nseg * H * D):
        raise ValueError("gla_scan: segment scratch too small")
    s0, s1 = seg if nseg > 1 else (None, None)
    f = out is not None
    _check(lib().nls_gla_scan(q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(0), a.data_ptr(), a.stride(0), qscale,
                              _p(o), o.stride(0) if o is not None else 0, norm.data_ptr() if f else None,
                              gate.data_ptr() if f else None, gate.stride(0) if f else 0, _p(out), out.stride(0) if f else 0,
                              eps, state.data_ptr(), state.stride(0), runs.data_ptr(), nruns, H, D, V, nseg, _p(s0), _p(s1), nt,
                              int(q.dtype == torch.float32), st), "nls_gla_scan")


def gla_step(q, k, v, a, gate_in, qscale: float, state, runs, nruns: int, norm, gate, out, H: int, D: int, V: int, eps: float,
             st: int, o=None):
    """gla_scan of runs of one token each (V a multiple of 4), with the norm and gate, or (norm None) the plain outputs in `o`.
    Decays `a`, or (None) from gate_in = (low-rank gate input, a2, bias, exponent): sigmoid(a2 low + bias) ^ exponent."""
    lo, a2, b, ia = gate_in if a is None else (None, None, None, 0.0)
    y = out if norm is not None else o
    _check(lib().nls_gla_step(q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(0), _p(a), a.stride(0) if a is not None else 0,
                              _p(lo), _p(a2), _p(b), a2.shape[1] if a2 is not None else 0, ia, qscale, state.data_ptr(),
                              state.stride(0), runs.data_ptr(), nruns, _p(norm), _p(gate),
                              gate.stride(0) if gate is not None else 0, _p(out), out.stride(0) if out is not None else 0, _p(o),
                              o.stride(0) if o is not None else 0, H, D, V, eps, int(q.dtype == torch.float32), st),
           "nls_gla_step")


def attn_step_fits(AH: int, AG: int, Dp: int, mfma: bool, window: int, H: int, D: int, V: int, f32: bool) -> int:
    """The most tokens whose attention and recurrence attn_step takes in one launch where that is the faster way (0: none): any
    number in bf16 (1 to 300 tokens behind 20 to 3000 keys 47 % less to 7 % more than one behind the other, 20 % less on average); in 32 bits (a
    workgroup per CU) up to 512 states (4 % more to 40 % less; 768 14 % less to 20 % more, 1024 up to 33 % more)."""
    if window or V % 4 or V > 1024 or -(-D // (256 // (V // 4))) > 16:
        return 0
    if f32:
        return 512 // max(H, attn_groups(AH, AG)) if Dp <= 256 else 0
    return 1 << 30 if mfma and Dp in (64, 128) else 0


def attn_step(aq, kc, vc, agate, aout, part, ns: int, block_tables, block_size: int, tok_seq, ctx_len, T: int, AH: int, AG: int, Dp: int,
              scale: float, sink: bool, q, k, v, a, gate_in, qscale: float, state, runs, norm, gate, out, H: int, D: int, V: int,
              eps: float, st: int):
    """gqa_attention of T single tokens without a window, and gla_step with a norm on the same tokens, in one launch."""
    po, pm, cnt = part
    if ns > 1 and (po.numel() < T * AH * ns * Dp or pm.numel() < T * AH * ns * 2 or cnt.numel() < T * attn_groups(AH, AG)):
        raise ValueError("attn_step: split workspace too small")
    lo, a2, b, ia = gate_in if a is None else (None, None, None, 0.0)
    _check(lib().nls_attn_step(aq.data_ptr(), aq.stride(0), kc.data_ptr(), vc.data_ptr(), block_tables.data_ptr(),
                               block_tables.stride(0), block_size, tok_seq.data_ptr(), ctx_len.data_ptr(), T, AH, AG, Dp, scale,
                               _p(agate), agate.stride(0) if agate is not None else 0, aout.data_ptr(), aout.stride(0), int(sink), ns,
                               po.data_ptr(), pm.data_ptr(), cnt.data_ptr(),
                               q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(0), _p(a), a.stride(0) if a is not None else 0,
                               _p(lo), _p(a2), _p(b), a2.shape[1] if a2 is not None else 0, ia, qscale, state.data_ptr(),
                               state.stride(0), runs.data_ptr(), norm.data_ptr(), gate.data_ptr(), gate.stride(0), out.data_ptr(),
                               out.stride(0), H, D, V, eps, int(q.dtype == torch.float32), st), "nls_attn_step")


# ---------------------------------------------------------------------------
# Delta rule
# ---------------------------------------------------------------------------

def delta_conv(z, w, y, fac, state, runs, tok_seq, T: int, nruns: int, H: int, G: int, D: int, V: int, st: int):
    """y = silu(causal convolution of z) per channel, [q: G * D | k: G * D | v: H * V]; w f32 [channels, taps]; the last taps - 1
    inputs are carried in state [slots, (taps - 1) * channels] (None for one tap). fac [rows, 2 G]: what makes the heads of q
    (times D^-1/2) and k unit vectors."""
    _check(lib().nls_delta_conv(z.data_ptr(), z.stride(0), w.data_ptr(), y.data_ptr(), y.stride(0), fac.data_ptr(), fac.stride(0),
                                _p(state), state.stride(0) if state is not None else 0, runs.data_ptr(), tok_seq.data_ptr(), T,
                                nruns, H, G, D, V, w.shape[1], int(z.dtype == torch.float32), st), "nls_delta_conv")


def delta_shape(T: int, nruns: int, H: int, D: int, V: int, longest: Optional[int] = None):
    """(segments, groups of 64 value columns per workgroup) of a delta_scan launch, as gla_shape. Segments cost a second pass over
    the tokens with D more columns: up to 64 channels they start where whole runs fill less than half the CUs, up to one workgroup per CU (16 heads of
    64 x 128, us: 128 tokens in one / two 69 / 70, 150 in one / three 93 / 72, 333 in one / two / six 183 / 157 / 109; 0.7 % behind the fastest count on
    average). With 65 to 128 channels that rule was 5.5 % behind (16 heads of 128 x 128: 6 runs of 650 tokens 517 us with 3
    segments, 444 with the 1 that segments_us finds)."""
    nt = 1 if V <= 64 else 2
    wgs = H * -(-V // (64 * nt))
    most = min(-(-256 // (wgs * nruns)), 16)             # (what bounds the scratch, too)
    if 64 < D <= 128 and nt == 2:
        return segments("delta", T, longest or -(-T // nruns), wgs, most), nt
    if longest is None:
        return 1 if wgs * nruns >= 128 else max(1, min(most, (T - nruns + 1) // 128)), nt
    return 1 if wgs * nruns >= 128 or longest <= 128 else min(most, -(-longest // 64)), nt


def delta_scan(q, k, v, fac, beta, a, o, norm, gate, out, state, runs, nruns: int, H: int, G: int, D: int, V: int, eps: float,
               shape, seg, st: int):
    """The delta rule over each run's tokens: q, k [rows, G * D], v [rows, H * V] of one buffer, the factors of delta_conv, beta
    [rows, H], decays a [rows, H * D]; otherwise as gla_scan. seg: (states, matrices) scratch of the segments."""
    nseg, nt = shape
    if nseg > 1 and (seg[0].numel() < nruns * nseg * H * D * V or seg[1].numel() < nruns * nseg * H * D * D):
        raise ValueError("delta_scan: segment scratch too small")
    s0, s1 = seg if nseg > 1 else (None, None)
    f = out is not None
    _check(lib().nls_delta_scan(q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(0), fac.data_ptr(), fac.stride(0),
                                beta.data_ptr(), beta.stride(0), a.data_ptr(), a.stride(0), _p(o), o.stride(0) if o is not None else 0,
                                norm.data_ptr() if f else None, gate.data_ptr() if f else None, gate.stride(0) if f else 0, _p(out),
                                out.stride(0) if f else 0, eps, state.data_ptr(), state.stride(0), runs.data_ptr(), nruns, H, G, D,
                                V, nseg, _p(s0), _p(s1), nt, int(q.dtype == torch.float32), st), "nls_delta_scan")


def delta_step(q, k, v, fac, beta, a, decay_in, gate, gate_in, ldz: int, state, runs, nruns: int, norm, out, H: int, G: int, D: int,
               V: int, eps: float, st: int):
    """delta_scan of runs of one token each (V a multiple of 4), with the norm and gate. Decays a, or (None) from decay_in =
    (low-rank input, a2, bias, exponent per channel): sigmoid(a2 low + bias) ^ exponent. The gate, or (None) from gate_in =
    (low-rank input, g2): sigmoid(g2 low). ldz: row stride of the low-rank inputs."""
    lo, a2, b, rate = decay_in if a is None else (None, None, None, None)
    lg, g2 = gate_in if gate is None else (None, None)
    _check(lib().nls_delta_step(q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(0), fac.data_ptr(), fac.stride(0),
                                beta.data_ptr(), beta.stride(0), _p(a), a.stride(0) if a is not None else 0, _p(lo), _p(a2), _p(b),
                                _p(rate), a2.shape[1] if a2 is not None else 0, _p(gate),
                                gate.stride(0) if gate is not None else 0, _p(lg), _p(g2), g2.shape[1] if g2 is not None else 0, ldz,
                                state.data_ptr(), state.stride(0), runs.data_ptr(), nruns, norm.data_ptr(), out.data_ptr(),
                                out.stride(0), H, G, D, V, eps, int(out.dtype == torch.float32), st), "nls_delta_step")


# ---------------------------------------------------------------------------
# Grouped-query attention
# ---------------------------------------------------------------------------

HEAD_WIDTHS = (32, 64, 128, 256)      # padded head widths of the MFMA attention kernels


def head_pad(D: int):
    """(padded head width, MFMA kernels): other widths run on the plain kernel, padded for its 16-byte loads."""
    for w in HEAD_WIDTHS:
        if D <= w:
            return w, True
    if D > 1024:
        raise ValueError(f"attention head width {D} > 1024")
    return pad_to(D, 32), False


def attn_groups(H: int, G: int) -> int:
    """Workgroups a (token, split) of gqa_attention takes."""
    return G * -(-(H // G) // 16)


def attn_rows(q, k, v, qn, kn, cs, pos, slot, qo, kc, vc, T: int, H: int, G: int, D: int, Dp: int, rot: int, eps: float, st: int,
              V: Optional[int] = None, head_norm: bool = False, key_tiles: bool = False):
    """Norm over the whole q and k projections (qn, kn: weights or None), rotation of the first `rot` columns of each head (cs
    None: none), then (head_norm) an RMS norm of each head of queries and keys on its own; queries to qo, keys and (as projected, V
    columns per head) values to the tokens' cache rows. q, k, v: f32 with one row stride. key_tiles: 16 slots of the key cache are a
    tile [G][Dp / 8][16][8] (slots in whole tiles)."""
    if key_tiles and kc.shape[0] % KEY_TILE:
        raise ValueError("attn_rows: a key cache of whole tiles")
    _check(lib().nls_attn_rows(q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(0), _p(qn), _p(kn), _p(cs),
                               pos.data_ptr(), slot.data_ptr(), qo.data_ptr(), qo.stride(0), kc.data_ptr(), vc.data_ptr(),
                               kc.stride(0), T, H, G, D, D if V is None else V, Dp, rot, int(head_norm),
                               int(key_tiles), eps,
                               int(qo.dtype == torch.float32), st),
           "nls_attn_rows")


def gqa_attention(q, kc, vc, gate, out, part, block_tables, block_size: int, tok_seq, ctx_len, T: int, H: int, G: int, Dp: int,
                  mfma: bool, ns: int, scale: float, st: int, window: int = 0, keep: int = 0, sink: bool = False):
    """Row-by-row attention (decoded tokens, short runs); a head gate (or None) is applied to the output. part: (partial
    outputs, (max, sum) pairs, ticket counters) of `ns` splits. window > 0: the newest `window` keys and the first `keep`;
    sink: the softmax's denominator holds one more, a score of 0 without a value."""
    po, pm, cnt = part
    if ns > 1 and (po.numel() < T * H * ns * Dp or pm.numel() < T * H * ns * 2 or cnt.numel() < T * attn_groups(H, G)):
        raise ValueError("gqa_attention: split workspace too small")
    _check(lib().nls_gqa_attn(q.data_ptr(), q.stride(0), kc.data_ptr(), vc.data_ptr(), block_tables.data_ptr(),
                              block_tables.stride(0), block_size, tok_seq.data_ptr(), ctx_len.data_ptr(), T, H, G, Dp, ns,
                              scale, _p(gate), gate.stride(0) if gate is not None else 0, out.data_ptr(), out.stride(0),
                              po.data_ptr(), pm.data_ptr(), cnt.data_ptr(), window, keep, int(sink), int(not mfma),
                              int(q.dtype == torch.float32), st), "nls_gqa_attn")


def gqa_prefill(q, kc, vc, xmap, blocks, nblocks: int, waves: int, gate, out, H: int, G: int, Dp: int, scale: float, st: int,
                window: int = 0, keep: int = 0, sink: bool = False, groups: int = 1):
    """Causal attention of query blocks over their sequences' paged keys and values (gate, window, keep, sink: as
    gqa_attention; groups: as latent_prefill)."""
    _check(lib().nls_gqa_prefill(q.data_ptr(), q.stride(0), kc.data_ptr(), vc.data_ptr(), xmap.data_ptr(), blocks.data_ptr(),
                                 nblocks, _p(gate), gate.stride(0) if gate is not None else 0, out.data_ptr(), out.stride(0), H, G,
                                 Dp, waves, groups, scale, window, keep, int(sink), st), "nls_gqa_prefill")


# ---------------------------------------------------------------------------
# Attention with mixed heads
# ---------------------------------------------------------------------------

KEY_TILE = 16                           # slots of a key tile
TALK_WIDTHS = (32, 64, 128)             # padded head widths of the prompt kernel, which takes up to 32 heads
TALK_SCRATCH = 256 << 20                # bytes of scores that a decode launch may hold


class TalkPlan:
    """Kernels and scratch sizes of an attention whose heads' softmax weights are mixed, heads padded to Dp columns. The MFMA kernels
    read keys in tiles of 16 slots (attn_rows: key_tiles), the plain one rows."""

    def __init__(self, H: int, G: int, Dp: int, window: int, ctx: int, f32: bool, device, scale: float = 1.0):
        self.H, self.G, self.Dp, self.window = H, G, Dp, window
        self.mfma = not f32 and Dp in HEAD_WIDTHS and H <= 128
        self.prefill = self.mfma and H <= 32 and Dp in TALK_WIDTHS and scale > 0
        self.groups, self.hs = attn_groups(H, G), pad_to(H, 8)
        self.ks = pad_to(min(window or ctx, ctx), 32) + 32              # keys of a row, from a multiple of 32 on
        self.device = device

    def matrix(self, talk: torch.Tensor) -> torch.Tensor:
        """The [H, H] matrix as the kernels read it."""
        if not self.mfma:
            return talk.to(device=self.device, dtype=torch.float32).contiguous()
        n = pad_to(self.H, 32) if self.H <= 64 else 128
        out = torch.zeros(n, n, dtype=torch.bfloat16, device=self.device)
        out[:self.H, :self.H] = talk.to(self.device)
        return out

    def rows(self, cap: int) -> int:
        """Rows of a decode launch."""
        return max(1, min(cap, TALK_SCRATCH // (4 * self.ks * self.hs)))

    def splits(self, T: int):
        """(splits of the scores, of the values, waves of a workgroup of the latter) at T rows."""
        n = T * self.groups
        ns1 = max(1, min(64, 2048 // n))
        if n >= 1024 or self.Dp > 128:
            return ns1, max(1, min(16, 1024 // n)), 1
        return ns1, max(1, min(16, 256 // n)), 4

    def plain_form(self, T: int):
        """(tokens of a workgroup of the scores, shares of the keys, tokens of a workgroup of the mix, shares, keys of a block, waves) of the
        plain kernels at T rows. Tokens share a workgroup, and so a tile of MFMA rows and their keys, once there are enough of them for the
        chip; fewer have their keys shared out instead. us of both launches with 1 / 2 / 4 tokens to a workgroup of the mix, at 400, 700 and 1203
        tokens of a prompt: 32 heads 125 / 94 / 127, 291 / 231 / 217, 726 / 545 / 491, 16 heads 61 / 66 / 81, 116 / 112 / 140, 267 / 199 / 231;
        one token and 1203 keys, 16 heads, in 1 / 4 / 16 shares 78 / 39 / 31."""
        most = max(1, 16 // (self.H // self.G))
        jobs = self.groups * -(-self.Dp // 64)
        tb1 = 1 if T <= 64 else min(most, -(-T * self.groups // 256))
        tb = 1
        while 2 * tb <= most and T * -(-jobs // 8) >= 340 * 2 * tb and 2 * tb * self.H * 36 <= 16384:
            tb *= 2
        kt = max(16, min(64, (16384 // (tb * self.H) - 4) // 16 * 16))
        nw = 4 if tb == 1 else 8
        ns1 = max(1, min(64, 1024 // (-(-T // tb1) * self.groups), -(-self.ks // 64)))
        ns = 1 if tb > 1 else max(1, min(16, 256 // (T * -(-jobs // nw)), -(-self.ks // kt)))
        return tb1, ns1, tb, ns, kt, nw

    def plain_buffers(self, T: int, ks: int, device):
        """What one call of the plain kernels over T rows needs, with ks keys to a row of scores: (scores, score statistics, partial outputs, counters)."""
        R = self.rows(T)
        forms = [(n, *self.plain_form(n)) for n in {R, T % R or R}]
        stats = max(n * ns1 for n, _, ns1, *_ in forms)
        part = max((n * ns for n, _, _, _, ns, _, _ in forms if ns > 1), default=0)
        cnt = max(n * -(-self.groups * -(-self.Dp // 64) // nw) for n, *_, nw in forms)
        f = [torch.empty(n, dtype=torch.float32, device=device) for n in (R * ks * self.H, stats * self.H * 2, part * self.H * self.Dp)]
        return (*f, torch.zeros(cnt, dtype=torch.int32, device=device))

    def scratch(self, cap: int):
        """Element counts of (scores, score statistics, partial outputs, counters)."""
        R = self.rows(cap)
        if not self.mfma:
            forms = [(T, *self.plain_form(T)) for T in range(1, R + 1)]
            part = max((T * ns for T, _, _, _, ns, _, _ in forms if ns > 1), default=0)
            return (R * self.ks * self.hs, max(T * ns1 for T, _, ns1, *_ in forms) * self.hs * 2, part * self.H * self.Dp,
                    min(R, 256) * -(-self.groups * -(-self.Dp // 64) // 4))
        part = max(T * self.splits(T)[1] for T in range(1, R + 1)) if R < 4096 else 16 * R
        return (R * self.ks * self.hs, max(T * self.splits(T)[0] for T in range(1, R + 1)) * self.hs * 2, part * self.H * self.Dp,
                R * self.groups)


def _allocating(device, st: int):
    """Allocations belong to stream st: memory of another stream could be handed out again while the kernels on st still use it."""
    if torch.cuda.current_stream(device).cuda_stream == st:
        return contextlib.nullcontext()
    return torch.cuda.stream(torch.cuda.ExternalStream(st, device) if st else torch.cuda.default_stream(device))


def talk_attention(plan: TalkPlan, q, kc, vc, talk, gate, out, scratch, block_tables, block_size: int, tok_seq, ctx_len, T: int,
                   V: int, scale: float, st: int):
    """Row-by-row attention with mixed heads (talk: TalkPlan.matrix); `gate`: a factor per output column, heads V columns apart."""
    p = plan
    ldg = gate.stride(0) if gate is not None else 0
    if gate is not None and gate.dtype != out.dtype:
        raise ValueError("talk_attention: a gate of the outputs' type")
    if not p.mfma:
        # (no plan of the contexts was needed before there were scores in memory: a table that holds more keys than the plan's rows gets longer rows)
        most = block_tables.shape[1] * block_size
        ks = max(p.ks, pad_to(min(p.window + 15, most) if p.window else most, 16))
        if not scratch or scratch[0].numel() < ks * p.H:
            with _allocating(q.device, st):
                scratch = p.plain_buffers(T, ks, q.device)
        sc, ss, po, cnt = scratch
        R = min(p.rows(T), sc.numel() // (ks * p.H))
        for t0 in range(0, T, R):
            n = min(R, T - t0)
            tb1, ns1, tb, ns, kt, nw = p.plain_form(n)
            if (ss.numel() < n * ns1 * p.H * 2 or (ns > 1 and (po.numel() < n * ns * p.H * p.Dp or cnt.numel() < n * -(-p.groups * -(-p.Dp // 64) // nw)))):
                raise ValueError("talk_attention: workspace too small")
            _check(lib().nls_talk_rows(q.data_ptr(), q.stride(0), kc.data_ptr(), vc.data_ptr(), block_tables.data_ptr(),
                                       block_tables.stride(0), block_size, tok_seq.data_ptr(), ctx_len.data_ptr(), t0, n, p.H, p.G, p.Dp, V,
                                       scale, p.window, talk.data_ptr(), _p(gate), ldg, out.data_ptr(), out.stride(0), sc.data_ptr(), ks,
                                       ss.data_ptr(), po.data_ptr(), cnt.data_ptr(), tb1, ns1, tb, ns, kt, nw,
                                       int(q.dtype == torch.float32), st), "nls_talk_rows")
        return
    sc, ss, po, cnt = scratch
    R = min(p.rows(T), sc.numel() // (p.ks * p.hs))
    for t0 in range(0, T, R):
        n = min(R, T - t0)
        ns1, ns, waves = p.splits(n)
        if (ss.numel() < n * ns1 * p.hs * 2 or cnt.numel() < n * p.groups or (ns > 1 and po.numel() < n * ns * p.H * p.Dp)):
            raise ValueError("talk_attention: workspace too small")
        _check(lib().nls_talk_decode(q.data_ptr(), q.stride(0), kc.data_ptr(), vc.data_ptr(), block_tables.data_ptr(),
                                     block_tables.stride(0), block_size, tok_seq.data_ptr(), ctx_len.data_ptr(), t0, n, p.H, p.G,
                                     p.Dp, V, scale, p.window, talk.data_ptr(), _p(gate), ldg, out.data_ptr(), out.stride(0),
                                     sc.data_ptr(), p.ks, ss.data_ptr(), po.data_ptr(), cnt.data_ptr(), ns1, ns, waves, st),
               "nls_talk_decode")


def talk_prefill(plan: TalkPlan, q, kc, vc, talk, gate, out, block_tables, block_size: int, blocks, nblocks: int, waves: int, V: int,
                 scale: float, st: int):
    """Attention with mixed heads of query blocks of up to 32 * waves tokens over their sequences' paged keys and values."""
    p = plan
    if not p.prefill or (gate is not None and gate.dtype != out.dtype):
        raise ValueError("talk_prefill: a shape of the row-by-row kernels, or a gate of another type")
    _check(lib().nls_talk_prefill(q.data_ptr(), q.stride(0), kc.data_ptr(), vc.data_ptr(), block_tables.data_ptr(),
                                  block_tables.stride(0), block_size, blocks.data_ptr(), nblocks, 2 * waves, p.H, p.G, p.Dp, V, scale, p.window, talk.data_ptr(), _p(gate),
                                  gate.stride(0) if gate is not None else 0, out.data_ptr(), out.stride(0), st), "nls_talk_prefill")
