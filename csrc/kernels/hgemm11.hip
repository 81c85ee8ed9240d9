// Dense f16 GEMM, "mode 11" of the qgemv dispatcher (gfx950): tiles in steps of 32 weight rows and 32 activations that fill one round of the chip, the
// two wave groups on alternate k-steps.
//
//   y[m, n] (epilogue) alpha * sum_k x[m, k] * W[n, k]      x f16 [M, K], W f16 [N, K] row-major
//
// 8 waves = 2 groups x 4; the four waves of a group are 2 x 2, each with 16 MT activation rows x 16 NT weight rows of the tile. Group g takes
// the k-steps (32 of K) of its parity, and the two halves meet in LDS at the end. A k-step is two sections a barrier apart: [read] NT + MT fragments,
// half of the DMA of a later K-tile, lgkmcnt(0); [multiply] NT MT MFMAs from registers. Group 1 runs one section behind, so that on each SIMD one
// wave multiplies while the other reads.
// What bounds a product of a few hundred rows is how fast a CU takes in operands: 57 GB/s with one K-tile of 64 in flight and copies of 16 rows x 64
// bytes, 80 with two and 8 rows x 128 bytes (tiles of 96 and 128 weight
// rows x 320 activations of a trial, 224 CUs; 16 x 64 bytes whose other half follows later: 48; with weights from memory 40 to
// 55). So LDS is a ring of R = 3 or 4
// K-tiles (mode 10: two), copies are whole lines, and tiles are nearer to squares: 160 x 224 makes 256 workgroups of 320 x 28672 and takes in 384 rows
// where 320 x 128 takes 448.
// A K-tile is read in sections 2 T (group 0) and 2 T + 1 (group 1); its slot is staged again, with K-tile T + R, in the two sections after. A group issues
// every other 8-row half of the row-tiles and waits, counted, for its halves of K-tile T + 1 before the barrier that ends section 2 T + 1.
// us of mode 10 (or 4) and of this, weights from memory: 6144 x 4096 with RoPE at 320 rows 39 -> 32 (and no launch behind it), 4096 x 4096 30 -> 28 in four
// parts, in a step of 320 rows 26 -> 21; 16384 x 2048 at 128 rows 30 -> 22, at 512 39 -> 38; 5120 x 5120 at 1024 83 -> 71; 28672 x 4096 at 256 70 and 71.
// Grid and split-K as mode 10.
#include "dense_epilogue.h"

namespace nls_hg11 {
using namespace nls_gemv;
using nls_dma::glds16;
using nls_dma::lds_addr;

template <int NT, int MT>
struct H11 {
  static constexpr int BN = 32 * NT, BM = 32 * MT;
  static constexpr int TB = (BN + BM) * 128;              // a K-tile of 64: weight rows, then activations
  static constexpr int R = 4 * TB <= 160 * 1024 ? 4 : 3;  // K-tiles of the ring
  static constexpr int RT = (BN + BM) / 16;               // row-tiles; a group stages one half (8 rows, 1 KiB) of each
  static constexpr int Q = RT / 4, X = RT % 4;            // ... a wave Q of them, the first X waves one more
  static constexpr int NA = (NT + 1) / 2;                 // weight tiles of a wave that group 0 stores
  static constexpr int LDS = R * TB > NT * MT * 4096 ? R * TB : NT * MT * 4096;
  static_assert(R * TB <= 160 * 1024 && LDS <= 160 * 1024, "LDS");
};

template <int N>
DEVI void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

template <int NT, int MT, bool ROPE>
DEVI void h11_tile(const Seg& S, int row0, int kslice, int ks, const GemvArgs& a, float* ws, uint8_t* lds) {
  typedef H11<NT, MT> C;
  constexpr int R = C::R, NJ = C::Q + (C::X ? 1 : 0), NA = C::NA, NW = C::BN / 16;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave >> 2, wc = wave & 3, wm = wc & 1, wn = wc >> 1;
  const int nkt_all = S.K / 64;
  const int t0 = (nkt_all * kslice) / ks, t1 = (nkt_all * (kslice + 1)) / ks;
  const int nkt = t1 - t0;
  const int M = a.M;

  // row-tile wc + 4 j (weights, then activations), rows 8 kg .. + 7 of it. Lane L -> row L >> 3, physical chunk L & 7 <- logical chunk
  // (L & 7) ^ (L >> 3), so that the rows of a fragment lie on different banks
  const char* Wb = (const char*)S.w + ((size_t)row0 * S.K + (size_t)t0 * 64) * 2;
  const char* Xb = (const char*)a.x + (size_t)t0 * 128;
  const uint32_t lc = ((lane & 7) ^ (lane >> 3)) * 16;
  uint32_t off[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int rt = wc + 4 * j, row = 16 * (rt < NW ? rt : rt - NW) + 8 * kg + (lane >> 3);
    off[j] = (rt < NW ? (uint32_t)min(row, S.rows - 1 - row0) * (uint32_t)(S.K * 2) : (uint32_t)min(row, M - 1) * (uint32_t)(a.ldx * 2)) + lc;
  }
  const uint32_t base = __builtin_amdgcn_readfirstlane(lds_addr(lds)) + 2048u * wc + 1024u * kg;
  auto dma = [&](int T, int slot) __attribute__((always_inline)) {
    const size_t kb = (size_t)min(T, nkt - 1) * 128;      // (past the end: the last K-tile again, which nothing reads)
    const char *wb = Wb + kb, *xb = Xb + kb;
    const uint32_t dst = base + (uint32_t)slot * C::TB;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (4 * j + 3 < C::RT || wc + 4 * j < C::RT) glds16(wc + 4 * j < NW ? wb : xb, off[j], dst + 8192u * j);
  };
  auto wait_next = [&]() __attribute__((always_inline)) {
    if (C::X && wc < C::X) wait_vm<(R - 2) * (C::Q + 1)>();
    else wait_vm<(R - 2) * C::Q>();
  };
  auto bar = []() __attribute__((always_inline)) {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  const int fro = (lane & 15) * 128 + (((kg * 4 + (lane >> 4)) ^ (lane & 7)) << 4);
  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  if (nkt > 0) {
#pragma unroll
    for (int T = 0; T < R - 1; ++T) dma(T, T);
    wait_next();
    bar();
    if (kg == 1) bar();
    int rd = 0, st = R - 1;                               // slots of the K-tile that is read, and of the one that is staged
    for (int T = 0; T < nkt; ++T) {
      const uint8_t* p = lds + rd * C::TB + fro;
      f16x8 FA[NT], FB[MT];
#pragma unroll
      for (int j = 0; j < MT; ++j) FB[j] = *reinterpret_cast<const f16x8*>(p + (NW + wm * MT + j) * 2048);
#pragma unroll
      for (int i = 0; i < NT; ++i) FA[i] = *reinterpret_cast<const f16x8*>(p + (wn * NT + i) * 2048);
      dma(T + R - 1, st);
      if (kg == 1) wait_next();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      bar();
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = mfma16(FA[i], FB[j], acc[i][j]);
      __builtin_amdgcn_s_setprio(0);
      if (kg == 0) wait_next();
      bar();
      rd = rd + 1 == R ? 0 : rd + 1;
      st = st + 1 == R ? 0 : st + 1;
    }
    if (kg == 0) bar();                                   // barrier counts even again
  }
  wait_vm<0>();                                           // the clamped DMAs past the end
  __syncthreads();
  // the groups' halves: group 1 gives tiles 0 .. NA - 1, group 0 the others
  f32x4* ex = reinterpret_cast<f32x4*>(lds) + (size_t)wc * NT * MT * 64 + lane;
#pragma unroll
  for (int i = 0; i < NT; ++i)
    if ((i < NA) == (kg == 1))
#pragma unroll
      for (int j = 0; j < MT; ++j) ex[(i * MT + j) * 64] = acc[i][j];
  __syncthreads();
  if (kg == 1) {
#pragma unroll
    for (int i = 0; i + NA < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = acc[NA + i][j];
  }
  f32x4 out[NA][MT];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int t = kg ? min(NA + i, NT - 1) : i;           // (an odd count: group 1's last tile is not stored)
#pragma unroll
    for (int j = 0; j < MT; ++j) out[i][j] = acc[i][j] + ex[(t * MT + j) * 64];
  }
  const int n0 = row0 + 16 * NT * wn;
  nls_dense::dense_epilogue<NA, MT, ROPE>(out, S, n0 + 16 * NA * kg, min(S.rows, n0 + (kg ? 16 * NT : 16 * NA)), wm * 16 * MT, kslice, ks, a, ws);
}

template <int NT, int MT, bool ROPE>
__global__ __launch_bounds__(512, 1) void hgemm11_kernel(SegList segs, GemvArgs a, int ks, float* ws, int ntiles, int nmb) {
  extern __shared__ __attribute__((aligned(16))) uint8_t h11lds[];
  constexpr int BM = H11<NT, MT>::BM;
  const int i = blockIdx.x, xcd = i & 7, j = i >> 3;
  const int kslice = j % ks;
  const int mb = (j / ks) % nmb;
  const int tile = (j / ks / nmb) * 8 + xcd;
  if (tile >= ntiles) return;
  const int m0 = mb * BM;
  Seg S = segs.s[0];
#pragma unroll
  for (int s = 1; s < 8; ++s)
    if (s < segs.nseg && tile >= segs.s[s].tile_begin) S = segs.s[s];
  a.m0 = m0;
  a.x += (size_t)m0 * a.ldx;
  const size_t esz = (a.epi == EPI_F32 || a.epi == EPI_ADD_F32 || a.epi == EPI_ARGMAX) ? 4 : 2;
  a.y = (char*)a.y + (size_t)m0 * a.ldy * esz;
  if (a.argmax) a.argmax += m0;
  a.M = min(BM, a.M - m0);
  h11_tile<NT, MT, ROPE>(S, (tile - S.tile_begin) * H11<NT, MT>::BN, kslice, ks, a, ws, h11lds);
}

template <int NT, int MT, bool ROPE>
int launch_e(const SegList& sl, int ntiles, int ks, float* ws, const GemvArgs& a, hipStream_t st) {
  typedef H11<NT, MT> C;
  const int nmb = (a.M + C::BM - 1) / C::BM;
  static bool attr = false;
  if (!attr) {   // > 64 KiB of dynamic LDS must be opted into
    if (hipFuncSetAttribute((const void*)hgemm11_kernel<NT, MT, ROPE>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS) != hipSuccess) return -1;
    attr = true;
  }
  hipLaunchKernelGGL((hgemm11_kernel<NT, MT, ROPE>), dim3((ntiles + 7) / 8 * 8 * nmb * ks), dim3(512), C::LDS, st, sl, a, ks, ws, ntiles, nmb);
  return (int)hipGetLastError();
}

// nt: weight rows of a tile / 32, mt: activation rows / 32
int launch_dense11(int nt, int mt, const SegList& sl, int ntiles, int ks, float* ws, const GemvArgs& a, hipStream_t st) {
#define NLS_H11(NT, MT) \
  if (nt == NT && mt == MT) return a.epi == EPI_ROPE ? launch_e<NT, MT, true>(sl, ntiles, ks, ws, a, st) : launch_e<NT, MT, false>(sl, ntiles, ks, ws, a, st);
#define NLS_H11N(MT) NLS_H11(3, MT) NLS_H11(4, MT) NLS_H11(5, MT) NLS_H11(6, MT) NLS_H11(7, MT) NLS_H11(8, MT)
  NLS_H11N(3) NLS_H11N(4) NLS_H11N(5)
#undef NLS_H11N
#undef NLS_H11
  return -1;
}

}  // namespace nls_hg11
