// Tiled GEMM on packed f32 weights with the operands in three bf16 parts (prompt chunks, larger batches and routed experts of 32-bit models).
//
// v = h + m + l, each part the bf16 rounding of what the ones before left: 8 bits and a sign each, so the sum is v exactly (above 2^-110, below
// which the last part is no normal number). Of the nine products of parts the six above 2^-24 of x w are summed, the small ones of a step first,
// in the f32 accumulators of the bf16 MFMA: six of its products take 0.4 of the time of the f32 MFMA's one.
//
// A wave owns RT tiles of 16 weight rows, whose sub-tiles it loads straight into registers (they are in fragment order, nobody shares them) and
// splits there. The activation rows are shared: a stage of them (BM rows x 32 values) is loaded into registers two stages ahead, split once
// per workgroup and written to LDS as fragments. Both operands take a lane's eight k from the two f32 sub-tiles of a step (4 g .. + 3 of each).
// Sums that are not finite, and those below 2^-80, are computed again with the f32 MFMA, the wave's others stay: an infinite operand has no parts,
// and rows of operands below 2^-110 have fewer digits in theirs (beside operands up to 2^20 their sums are such).
//
// Against 64 bits 900 x 20096 x 2048 is off by 7.0e-7 of its norm (f32 MFMAs 8.1e-7), 1500 x 4096 x 17408 by 2.15e-6 (2.36e-6): six products
// of 32 inputs are 6 K / 32 roundings of a sum, where the f32 MFMA rounds at each input. 1500 x 35888 x 4096 runs at 217 TFLOP/s (f32 MFMAs 128),
// 1.3 PFLOP/s of bf16, what the bf16 GEMMs of this library reach. Four waves to a workgroup and three or four workgroups to a CU, so that one
// splits while another multiplies: one workgroup alone takes 2.6 times its MFMAs' time a step (1.65 us; three 3.5), eight waves of 128 x 128 or
// 256 x 128 with one or two to a CU 146 to 201 TFLOP/s, splits and loads placed between a wave's own MFMAs 0.95 of this.
#include "lin.h"

namespace nls_lin {

template <int NWV, int RT, int MT>
struct LS {
  static constexpr int BN = 16 * RT * NWV, BM = 16 * MT;
  static constexpr int XST = MT * 3 * 1024, LDS = 2 * XST;             // bytes of a stage's parts
  static constexpr int P = BM * 4 / (64 * NWV);                        // (row, lane group) pairs that a thread loads and splits
  static_assert(P * 64 * NWV == BM * 4 && LDS <= 160 * 1024, "stage");
};

struct Parts { u32x4 h, m, l; };

DEVI uint32_t pk_bf16(float a, float b) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, bf2{(__bf16)a, (__bf16)b});
}
DEVI float lo_f(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
DEVI float hi_f(uint32_t p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

DEVI Parts split8(const u32x4& u, const u32x4& v) {
  Parts p;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4 s = __builtin_bit_cast(f32x4, i < 2 ? u : v);
    float a = s[2 * i & 3], b = s[(2 * i & 3) + 1];
    p.h[i] = pk_bf16(a, b);
    a -= lo_f(p.h[i]);
    b -= hi_f(p.h[i]);
    p.m[i] = pk_bf16(a, b);
    a -= lo_f(p.m[i]);
    b -= hi_f(p.m[i]);
    p.l[i] = pk_bf16(a, b);
  }
  return p;
}

// Whether a sum is computed again with the f32 MFMA (a zero stays: rows of zeros are common). In integers, which leaves no branch: with one the
// first sum of a block was compiled to the value it had.
DEVI bool again(float v) {
  const uint32_t m = __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
  return (m >= 0x7f800000u) | (m - 1 < 0x17800000u - 1);       // inf and NaN, below 2^-80
}

template <int NWV, int RT, int MT, int WPE>
__global__ __launch_bounds__(64 * NWV, WPE) void lin_split_kernel(LinArgs a, int ntot) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lslds[];
  typedef LS<NWV, RT, MT> G;
  typedef LT<float> L;
  typedef LT<__bf16> B;
  constexpr int P = G::P;
  int listed, gap;
  lin_listed(a, G::BN, listed, gap);
  ntot -= gap;
  const int per = (ntot + 7) >> 3, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || id >= ntot) return;
  LinTile t;
  if (!lin_tile<G::BN, G::BM>(a, id < listed ? id : id + gap, t)) return;
  const LinSeg& S = a.s[t.seg];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int nsub = S.nsub, tot = nsub >> 1;
  const int jb = tot * t.ks / S.ks, nst = tot * (t.ks + 1) / S.ks - jb;     // this split's steps of 32 k
  const int nwt = (S.N + 15) >> 4;

  const uint8_t* wp[RT];
#pragma unroll
  for (int q = 0; q < RT; ++q)                       // (a tile past the matrix: its last one again, not stored)
    wp[q] = (const uint8_t*)S.w + (size_t)t.grp * S.wstride +
            ((size_t)min((t.n0 >> 4) + RT * wave + q, nwt - 1) * nsub + 2 * jb) * 1024 + lane * 16;
  // Pair i of this thread: fragment (row tile, step) f, row 4 q + rr of the tile, lane group gg. Sixteen lanes read four rows' 64 bytes; in the
  // fragment the quads of rows are permuted by group so that neither these writes nor the fragments' reads meet in a bank.
  const float* xp[P];
  uint32_t xd[P];
  const int rr = (lane >> 4) * 4 + ((lane >> 2) & 3), gg = lane & 3;
  auto slot = [](int grp, int row) __attribute__((always_inline)) {
    return 256 * grp + 16 * ((((row >> 2) ^ (0x2130 >> (4 * grp))) & 3) * 4 + (row & 3));
  };
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int mt = P * wave + i;
    int xr, yr;
    lin_row(S, t, 16 * mt + rr, xr, yr);
    xp[i] = (const float*)S.x + (size_t)xr * S.ldx + (size_t)t.grp * S.xgs + 32 * jb + 4 * gg;
    xd[i] = mt * 3072 + slot(gg, rr);
  }
  u32x4 wr[RT][2], xr[P][2];
  auto load_w = [&](int j) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < RT; ++q)
#pragma unroll
      for (int e = 0; e < 2; ++e) wr[q][e] = ld16(wp[q] + (size_t)min(j, nst - 1) * 2048 + 1024 * e);
  };
  auto load_x = [&](int j) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < P; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) xr[i][e] = ld16(xp[i] + (size_t)min(j, nst - 1) * 32 + 16 * e);
  };
  auto put_x = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const Parts p = split8(xr[i][0], xr[i][1]);
      uint8_t* d = lslds + stage * G::XST + xd[i];
      *reinterpret_cast<u32x4*>(d) = p.h;
      *reinterpret_cast<u32x4*>(d + 1024) = p.m;
      *reinterpret_cast<u32x4*>(d + 2048) = p.l;
    }
  };
  auto meet = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  f32x4 acc[RT][MT];
#pragma unroll
  for (int q = 0; q < RT; ++q)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[q][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int xo = slot(g, r);
  load_x(0);
  load_w(0);
  put_x(0);
  load_x(1);
  meet();
  for (int j = 0; j < nst; ++j) {
    const int s = j & 1;
    Parts w[RT];
#pragma unroll
    for (int q = 0; q < RT; ++q) w[q] = split8(wr[q][0], wr[q][1]);
    load_w(j + 1);
    put_x(s ^ 1);                                    // (that stage was read in the step before the last barrier)
    load_x(j + 2);
#pragma unroll
    for (int i = 0; i < MT; i += 2) {                // two row tiles side by side: chains of 2 RT accumulators
      Parts x[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const uint8_t* src = lslds + s * G::XST + (i + b) * 3072 + xo;
        x[b] = Parts{ld16(src), ld16(src + 1024), ld16(src + 2048)};
      }
      auto mul = [&](u32x4 Parts::*u, u32x4 Parts::*v) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < RT; ++q)
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[q][i + b] = B::mma(w[q].*u, x[b].*v, acc[q][i + b]);
      };
      mul(&Parts::l, &Parts::h);
      mul(&Parts::h, &Parts::l);
      mul(&Parts::m, &Parts::m);
      mul(&Parts::m, &Parts::h);
      mul(&Parts::h, &Parts::m);
      mul(&Parts::h, &Parts::h);
    }
    meet();
  }
  bool odd = false;
#pragma unroll
  for (int q = 0; q < RT; ++q)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) odd |= again(acc[q][i][e]);
  if (__any(odd))
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      int xr, yr;
      lin_row(S, t, 16 * i + r, xr, yr);
      const float* x = (const float*)S.x + (size_t)xr * S.ldx + (size_t)t.grp * S.xgs + 32 * jb + 4 * g;
#pragma unroll
      for (int q = 0; q < RT; ++q) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < 2 * nst; ++k) v = L::mma(ld16(wp[q] + (size_t)k * 1024), ld16(x + k * L::KS), v);
        asm volatile("" : "+v"(acc[q][i]));          // (looked at anew: kept from above, the answers would not fit beside the rest)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[q][i][e] = again(acc[q][i][e]) ? v[e] : acc[q][i][e];
      }
    }
  lin_epilogue<float>(S, t, acc, t.n0 + 16 * RT * wave + 4 * g, r);
}

template <int NWV, int RT, int MT, int WPE>
int split_t(LinArgs& a, hipStream_t st) {
  typedef LS<NWV, RT, MT> G;
  const int n = lin_count(a, G::BN, G::BM);
  if (n < 1) return -1;
  static bool attr = false;
  if (!attr) {
    if (hipFuncSetAttribute((const void*)lin_split_kernel<NWV, RT, MT, WPE>, hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS) != hipSuccess)
      return -1;
    attr = true;
  }
  hipLaunchKernelGGL((lin_split_kernel<NWV, RT, MT, WPE>), dim3((n + 7) / 8 * 8), dim3(64 * NWV), G::LDS, st, a, n);
  return (int)hipGetLastError();
}

int lin_split(LinArgs& a, int cfg, hipStream_t st) {
  if (cfg >= 256) cfg = 4;
  if (cfg == 4)                                      // (lists in tiles of more rows do not fit the 128 of the tile it runs on)
    for (int i = 0; i < a.nseg; ++i)
      if (a.s[i].rows) return -1;
  switch (cfg) {
    case 0: case 12: return split_t<4, 1, 4, 4>(a, st);
    case 1: case 8: case 9: case 10: return split_t<4, 2, 4, 4>(a, st);
    case 2: case 3: case 4: case 6: case 11: return split_t<4, 2, 8, 3>(a, st);
  }
  return -1;
}

}  // namespace nls_lin
