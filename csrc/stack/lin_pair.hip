// bf16 GEMM of some hundred rows on packed weights (gfx950): tiles in steps of 32 weight rows and 32 activations that fill one round of the chip, the
// two wave groups on alternate k-steps.
//
// 8 waves = 2 groups x 4; the four waves of a group are 2 x 2, each with 16 NT weight rows x 16 MT activation rows of the tile. Group g takes sub-tile g
// (32 of K) of every K-tile of 64, and the two halves of the sums meet in LDS at the end. A k-step is two sections a barrier apart: [read] NT + MT
// fragments, this group's half of the DMA of a later K-tile, lgkmcnt(0); [multiply] NT MT MFMAs from registers. Group 1 runs one section behind, so
// that on each SIMD one wave multiplies while the other reads.
// LDS is a ring of R = 3 or 4 K-tiles. A K-tile is read in sections 2 T (group 0) and 2 T + 1 (group 1); its slot is staged again, with K-tile T + R, in
// the two sections after. A group waits, counted, for its halves of K-tile T + 1 before the barrier that ends section 2 T + 1.
// Weight sub-tiles arrive verbatim (1 KiB, fragment order), activations as 8 rows x 128 bytes, the 16-byte chunks of a row permuted.
// What bounds a product of a few hundred rows is how fast a CU takes in operands: the tiles of lin_gemm.hip, whose waves all read and all multiply between
// two barriers, take 50 to 65 GB/s, this one 75 to 85. us of the best tile there and of this (rows x outputs x inputs, weights from memory):
// 300 x 10240 x 4096 46.8 -> 37.6, 640 57 -> 52, 800 83 -> 68, 200 x 14336 x 2048 30.8 -> 25.2, 400 x 20096 x 2048 50 -> 42, 300 x 24576 x 4096 89 -> 65,
// 640 x 6144 x 4096 52 -> 42; in four splits 300 x 4096 x 9216 40 -> 34, 640 x 4096 x 17408 92 -> 77. It needs its workgroups: a tile takes 0.4 us per 64
// inputs however few there are, so that 200 x 2048 x 2048 and 512 x 3072 x 2048 stay with smaller ones (9.5 against 12, 16 against 21), and where whole
// rounds fill, the phased 256 x 256 tile is the faster one (512 x 24576 x 4096 93 against 107).
#include "../kernels/lds_dma.h"
#include "lin.h"

namespace nls_lin {
using nls_dma::glds16;
using nls_dma::lds_addr;

template <int NT, int MT>
struct LP {
  static constexpr int BN = 32 * NT, BM = 32 * MT;
  static constexpr int TB = (BN + BM) * 128;              // a K-tile: weight row-tiles, then activations
  static constexpr int R = 4 * TB <= 160 * 1024 ? 4 : 3;  // K-tiles of the ring
  static constexpr int NW = BN / 16, RT = NW + BM / 16;   // row-tiles; a group stages one half (1 KiB) of each
  static constexpr int Q = RT / 4, X = RT % 4;            // ... a wave Q of them, the first X waves one more
  static constexpr bool ROWS = MT % 2 == 0;               // a group stores half of the rows, or half of the weight tiles
  static constexpr int NI = ROWS ? NT : NT / 2, NJ = ROWS ? MT / 2 : MT;
  static constexpr int LDS = R * TB > NT * MT * 4096 ? R * TB : NT * MT * 4096;
  static_assert(LDS <= 160 * 1024 && (ROWS || NT % 2 == 0), "tile");
};

template <int N>
DEVI void lp_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
DEVI void lp_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int NT, int MT>
__global__ __launch_bounds__(512, 1) void lin_pair_kernel(LinArgs a, int ntot) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lplds[];
  typedef LP<NT, MT> P;
  typedef LT<__bf16> L;
  constexpr int R = P::R, NJ = P::Q + (P::X ? 1 : 0), NW = P::NW;
  const int per = (ntot + 7) >> 3, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || id >= ntot) return;
  LinTile t;
  if (!lin_tile<P::BN, P::BM>(a, id, t)) return;
  const LinSeg& S = a.s[t.seg];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave >> 2, wc = wave & 3, wm = wc & 1, wn = wc >> 1;
  const int nsub = S.nsub, jb = (nsub >> 1) * t.ks / S.ks, nkt = (nsub >> 1) * (t.ks + 1) / S.ks - jb;     // this split's K-tiles
  const int nwt = ((S.N + 15) >> 4) - (t.n0 >> 4);

  // row-tile wc + 4 j (weights, then activations): sub-tile kg, or rows 8 kg .. + 7
  const char* Wb = (const char*)S.w + (size_t)t.grp * S.wstride + ((size_t)(t.n0 >> 4) * nsub + 2 * jb) * 1024;
  const char* Xb = (const char*)S.x + ((size_t)t.m0 * S.ldx + (size_t)t.grp * S.xgs + (size_t)jb * 64) * 2;
  uint32_t off[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int rt = wc + 4 * j, row = 16 * (rt - NW) + 8 * kg + (lane >> 3);
    off[j] = rt < NW ? (uint32_t)min(rt, nwt - 1) * (uint32_t)(nsub * 1024) + 1024u * kg + 16u * lane
                     : (uint32_t)min(row, t.cnt - 1) * (uint32_t)(S.ldx * 2) + 16u * ((lane & 7) ^ (lane >> 3));
  }
  const uint32_t base = __builtin_amdgcn_readfirstlane(lds_addr(lplds)) + 2048u * wc + 1024u * kg;
  auto dma = [&](int T, int slot) __attribute__((always_inline)) {
    const int tc = min(T, nkt - 1);                       // (past the end: the last K-tile again, which nothing reads)
    const char *wb = Wb + (size_t)tc * 2048, *xb = Xb + (size_t)tc * 128;
    const uint32_t dst = base + (uint32_t)slot * P::TB;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (4 * j + 3 < P::RT || wc + 4 * j < P::RT) glds16(wc + 4 * j < NW ? wb : xb, off[j], dst + 8192u * j);
  };
  auto wait_next = [&]() __attribute__((always_inline)) {
    if (P::X && wc < P::X) lp_wait<(R - 2) * (P::Q + 1)>();
    else lp_wait<(R - 2) * P::Q>();
  };

  const int wfo = wn * NT * 2048 + kg * 1024 + lane * 16, xfo = (NW + wm * MT) * 2048 + r * 128 + (((kg * 4 + g) ^ (r & 7)) << 4);
  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int T = 0; T < R - 1; ++T) dma(T, T);
  wait_next();
  lp_barrier();
  if (kg == 1) lp_barrier();
  int rd = 0, st = R - 1;                                 // slots of the K-tile that is read, and of the one that is staged
  for (int T = 0; T < nkt; ++T) {
    const uint8_t* p = lplds + rd * P::TB;
    u32x4 A[NT], B[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) B[j] = *reinterpret_cast<const u32x4*>(p + xfo + j * 2048);
#pragma unroll
    for (int i = 0; i < NT; ++i) A[i] = *reinterpret_cast<const u32x4*>(p + wfo + i * 2048);
    dma(T + R - 1, st);
    if (kg == 1) wait_next();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    lp_barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = L::mma(A[i], B[j], acc[i][j]);
    __builtin_amdgcn_s_setprio(0);
    if (kg == 0) wait_next();
    lp_barrier();
    rd = rd + 1 == R ? 0 : rd + 1;
    st = st + 1 == R ? 0 : st + 1;
  }
  if (kg == 0) lp_barrier();                              // barrier counts even again
  lp_wait<0>();                                           // the clamped DMAs past the end
  __syncthreads();
  // the groups' halves: group 1 gives the first half of the blocks, group 0 the others
  f32x4* ex = reinterpret_cast<f32x4*>(lplds) + (size_t)wc * NT * MT * 64 + lane;
  auto first = [](int i, int j) __attribute__((always_inline)) { return P::ROWS ? j < P::NJ : i < P::NI; };
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
      if (first(i, j) == (kg == 1)) ex[(i * MT + j) * 64] = acc[i][j];
  __syncthreads();
  f32x4 out[P::NI][P::NJ];
#pragma unroll
  for (int i = 0; i < P::NI; ++i)
#pragma unroll
    for (int j = 0; j < P::NJ; ++j) {
      const int i1 = P::ROWS ? i : i + P::NI, j1 = P::ROWS ? j + P::NJ : j;
      if (kg == 0) out[i][j] = acc[i][j] + ex[(i * MT + j) * 64];
      else out[i][j] = ex[(i1 * MT + j1) * 64] + acc[i1][j1];
    }
  lin_epilogue<__bf16>(S, t, out, t.n0 + 16 * NT * wn + (P::ROWS ? 0 : 16 * P::NI * kg) + 4 * g, 16 * MT * wm + (P::ROWS ? 16 * P::NJ * kg : 0) + r);
}

template <int NT, int MT>
int pair_t(LinArgs& a, hipStream_t st) {
  typedef LP<NT, MT> P;
  const int n = lin_count(a, P::BN, P::BM);
  if (n < 1) return -1;
  static bool attr = false;
  if (!attr) {
    if (hipFuncSetAttribute((const void*)lin_pair_kernel<NT, MT>, hipFuncAttributeMaxDynamicSharedMemorySize, P::LDS) != hipSuccess) return -1;
    attr = true;
  }
  hipLaunchKernelGGL((lin_pair_kernel<NT, MT>), dim3((n + 7) / 8 * 8), dim3(512), P::LDS, st, a, n);
  return (int)hipGetLastError();
}

// nt: weight rows of a tile / 32, mt: activation rows / 32
int lin_pair(LinArgs& a, int nt, int mt, hipStream_t st) {
  for (int i = 0; i < a.nseg && i < LIN_SEGS; ++i) {
    const LinSeg& S = a.s[i];                             // (row lists and maps; offsets inside a tile are 32 bits)
    if (S.rows || S.xmap || S.ldx >= (1 << 22) || S.nsub >= (1 << 16)) return -1;
  }
#define NLS_LP(NT, MT) \
  if (nt == NT && mt == MT) return pair_t<NT, MT>(a, st);
  NLS_LP(4, 4) NLS_LP(5, 4) NLS_LP(6, 4) NLS_LP(8, 4) NLS_LP(4, 5) NLS_LP(6, 5) NLS_LP(8, 5)
#undef NLS_LP
  return -1;
}

}  // namespace nls_lin
