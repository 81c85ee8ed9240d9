// Dense f16 GEMM, "mode 10" of the qgemv dispatcher (gfx950): 256 x 256 tiles in 4 phases per 64-deep
// K-tile with the two wave groups staggered by one barrier (cdna_hip_programming.md "The 256^2 8-phase
// template": counted vmcnt, raw barriers, one LDS-DMA unit per phase, the per-phase interleave).
//
//   y[m, n] (epilogue) alpha * sum_k x[m, k] * W[n, k]      x f16 [M, K], W f16 [N, K] row-major
//
// Why (profiles/gemm_probes_r03.txt): mode 8's one-barrier-per-stage ring keeps all 8 waves in the same
// section at once -- every wave reads LDS and issues DMA together, then every wave runs MFMAs together,
// and with MFMAs off the kernel still takes 94 % of its time. Here:
//   * 8 waves = 2 groups (wr: 128 weight rows each) x 4 (wc: 64 activation rows each); a wave owns a
//     128 x 64 output block (8 x 4 accumulator tiles of v_mfma_f32_16x16x32_f16, weights as the A
//     operand so a lane ends with 4 consecutive output columns, as mode 8);
//   * a K-tile is 4 phases, each: [load section] ds_read the phase's fragments + issue one 16 KiB
//     LDS-DMA unit (2 global_load_lds_dwordx4 per lane) -> barrier -> lgkmcnt(0), 16 MFMAs at raised
//     priority -> vmcnt(6) -> barrier. Group 1 runs ONE barrier behind group 0, so on every SIMD (one wave
//     of each group) one wave's MFMAs overlap the other wave's LDS reads and DMA issue;
//   * fragment schedule per K-tile (quadrants of the wave's block): Q0 = weight rows 0-63 x act rows
//     0-31 (reads A(nq0) 8 + B(mh0) 4), Q1 = x act rows 32-63 (B(mh1) 4), Q2 = weight rows 64-127 (A(nq1)
//     8), Q3 = (nq1, mh0) from registers;
//   * the 64 KiB K-tile buffer is 4 units in the order they are needed -- U0 = A(nq0 of both groups),
//     U1 = B(mh0), U2 = B(mh1), U3 = A(nq1) -- and a unit is restaged as soon as its previous contents are
//     read (>= 2 phases, the WAR rule with a staggered group): U0(T) at phase Q2(T-2), U1(T) Q3(T-2),
//     U2(T) Q0(T-1), U3(T) Q1(T-1). Every unit is issued >= 5 phases before its first read and 3 units
//     stay in flight (vmcnt(6)), which the group stagger needs (a reader in group 0 is ordered only after
//     group 1's wait of the phase before);
//   * 2 K-tile buffers = 128 KiB of LDS, 1 workgroup per CU; 16-byte chunks XOR-swizzled per 4-row group
//     on the DMA source, as mode 8 (conflict-free ds_read_b128).
// Grid and split-K as mode 8: (tile, m-block, k-slice), every m-block and k-slice of a weight tile on one
// XCD. The epilogues are mode 8's (f32 / residual add / f16 / SwiGLU / split-K slabs / arg-max keys).
#include "dense_epilogue.h"

namespace nls_hg10 {
using namespace nls_gemv;
using nls_dma::glds16;
using nls_dma::lds_addr;

// BN = 256 (rt 1) or 128 (rt 2: narrow-N shapes get twice the workgroups -- Q|K|V, o at M = 512..2048): the
// weight half of a K-tile buffer and each wave's weight rows halve; the activation half, the phase schedule
// and the unit order stay, only the DMA instruction counts of the two weight units (and so the counted
// vmcnt of each phase) change.
// Row blocks of 64 MT rows: 256 (MT 4), or 192 (MT 3: the second half of a wave's rows is one tile), which 321 .. 384 rows and many
// larger counts fill better, or with 128 weight rows 320 (MT 5: the first half is three tiles; 18 KiB of LDS reads for 40 MFMAs of a wave, 14 for
// 24 at 192 rows), which 257 .. 320 and 513 .. 640 rows fill (launch_dense10).
constexpr int KT = 64;                       // K per tile
template <int BN, int MT>
struct H10 {
  static constexpr int BM = 64 * MT;
  static constexpr int AB = BN * KT * 2;     // weight half of a K-tile buffer (32 or 16 KiB)
  static constexpr int TB = AB + BM * KT * 2;
  static constexpr int LDS = 2 * TB;
  static constexpr int RTG = BN / 32;        // 16-row weight tiles per wave group (wr)
  static constexpr int NQH = RTG / 2;        // ... per quadrant half (nq)
  static constexpr int NA = BN / 128;        // DMA instructions per lane of a weight unit (U1: 2)
  static constexpr int NB1 = (MT + 1) / 2;   // ... of U1, and tiles of the first half of a wave's rows
  static constexpr int NB2 = MT - NB1;       // ... of U2
  // counted waits: the last three units issued stay in flight (units U0/U3 carry NA, U1 NB1, U2 NB2)
  static constexpr int VM_PRO = NA + NB1;          // after the prologue: U0(1) U1(1)
  static constexpr int VM_Q0 = NA + NB1 + NB2;     // U0(T+1) U1(T+1) U2(T+1)
  static constexpr int VM_Q1 = NA + NB1 + NB2;     // U1(T+1) U2(T+1) U3(T+1)
  static constexpr int VM_Q2 = 2 * NA + NB2;       // U2(T+1) U3(T+1) U0(T+2)
  static constexpr int VM_Q3 = 2 * NA + NB1; // U3(T+1) U0(T+2) U1(T+2)
};

DEVI int swz(int r) { return (0x1320 >> (4 * ((r >> 2) & 3))) & 3; }

template <int N>
DEVI void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

// unit u's (row-tile, k-step) subtiles; a subtile = 16 rows x 32 k = 1 KiB at (rt * 2 + ks) * 1 KiB of
// its operand region. A units (0, 3): weight row-tiles; B units (1, 2): activation row-tiles.
template <int BN, int MT>
DEVI int unit_rt(int u, int idx) {           // idx: row-tile slot of the unit
  // BN 256: U0: A {0-3, 8-11}; U3: A {4-7, 12-15}. BN 128: U0: A {0-1, 4-5}; U3: A {2-3, 6-7}.
  // U1: B {0,1,4,5,8,9,12,13}; U2: B {2,3,6,7,10,11,14,15}. MT 3: U1: B {0,1,3,4,6,7,9,10}; U2: B {2,5,8,11}
  // MT 5: U1: B {0-2, 5-7, 10-12, 15-17}; U2: B {3,4,8,9,13,14,18,19}
  constexpr int NQH = H10<BN, MT>::NQH, RTG = H10<BN, MT>::RTG, NB1 = H10<BN, MT>::NB1, NB2 = H10<BN, MT>::NB2;
  if (u == 0) return (idx % NQH) + RTG * (idx / NQH);
  if (u == 3) return NQH + (idx % NQH) + RTG * (idx / NQH);
  if (u == 1) return idx % NB1 + MT * (idx / NB1);
  return NB1 + idx % NB2 + MT * (idx / NB2);
}

template <int BN, int MT, bool ROPE>
DEVI void h10_tile(const Seg& S, int row0, int kslice, int ks, const GemvArgs& a, float* ws, uint8_t* lds) {
  typedef H10<BN, MT> C;
  constexpr int TB = C::TB, NQH = C::NQH, NA = C::NA, NB1 = C::NB1, NB2 = C::NB2;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 2, wc = wave & 3;
  const int nkt_all = S.K / KT;
  const int t0 = (nkt_all * kslice) / ks, t1 = (nkt_all * (kslice + 1)) / ks;
  const int nkt = t1 - t0;
  const int M = a.M;
  const act_t* Wd = reinterpret_cast<const act_t*>(S.w);

  // ---- DMA: unit u of K-tile T -> buffer T & 1. This wave issues subtiles idx = n * wave + j (j < n; n = NB1, NB2,
  // or NA for a weight unit) of every unit: row-tile unit_rt(u, idx >> 1), k-step idx & 1. Lane L -> row
  // 16 rt + (L >> 2), physical chunk L & 3 <- logical chunk (L & 3) ^ swz(L >> 2).
  const int lc = (lane & 3) ^ swz(lane >> 2);
  const uint32_t base = __builtin_amdgcn_readfirstlane(lds_addr(lds));
  auto dma = [&](int u, int T) __attribute__((always_inline)) {
    const int Tc = t0 + min(T, nkt - 1);       // clamped: past the end re-stages the last tile (same bytes)
    const bool bu = u == 1 || u == 2;
    const uint32_t buf = base + (uint32_t)(T & 1) * TB + (bu ? (uint32_t)C::AB : 0u);
    const int n = u == 1 ? NB1 : u == 2 ? NB2 : NA;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      if (j >= n) break;
      const int idx = n * wave + j;
      const int rt = unit_rt<BN, MT>(u, idx >> 1), kstep = idx & 1;
      const act_t* src;
      if (u == 1 || u == 2) {
        const int row = min(16 * rt + (lane >> 2), M - 1);
        src = a.x + (size_t)row * a.ldx;
      } else {
        const int row = min(row0 + 16 * rt + (lane >> 2), S.rows - 1);
        src = Wd + (size_t)row * S.K;
      }
      glds16(src + (size_t)Tc * KT + kstep * 32 + lc * 8, buf + (uint32_t)(rt * 2 + kstep) * 1024u);
    }
  };

  // ---- fragments: lane reads row (l & 15) of a 16-row subtile, logical chunk l >> 4
  const int fro = (lane & 15) * 64 + (((lane >> 4) ^ swz(lane & 15)) << 4);
  f16x8 FA[NQH][2], FB0[NB1][2], FB1[NB2][2];
  auto rdA = [&](int T, int nq) __attribute__((always_inline)) {
    const uint8_t* p = lds + (T & 1) * TB + fro;
#pragma unroll
    for (int i = 0; i < NQH; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s)
        FA[i][s] = *reinterpret_cast<const f16x8*>(p + ((wr * C::RTG + nq * NQH + i) * 2 + s) * 1024);
  };
  auto rdB = [&](auto& F, int T, int mh) __attribute__((always_inline)) {
    const uint8_t* p = lds + (T & 1) * TB + C::AB + fro;
#pragma unroll
    for (int i = 0; i < (mh ? NB2 : NB1); ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) F[i][s] = *reinterpret_cast<const f16x8*>(p + ((wc * MT + mh * NB1 + i) * 2 + s) * 1024);
  };
  f32x4 acc[2 * NQH][MT];
#pragma unroll
  for (int i = 0; i < 2 * NQH; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mma = [&](int nq, int mh, const auto& F) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < NQH; ++i)
#pragma unroll
        for (int j = 0; j < (mh ? NB2 : NB1); ++j)
          acc[nq * NQH + i][mh * NB1 + j] = mfma16(FA[i][s], F[j][s], acc[nq * NQH + i][mh * NB1 + j]);
  };
  auto bar = []() __attribute__((always_inline)) {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  if (nkt > 0) {
    // prologue: what the steady state would have issued before phase Q0(0): U0(0) U1(0) U2(0) U3(0) U0(1)
    // U1(1); K-tile 0 complete (2 units left in flight), then one barrier for all and group 1's stagger
    dma(0, 0);
    dma(1, 0);
    dma(2, 0);
    dma(3, 0);
    dma(0, 1);
    dma(1, 1);
    wait_vm<C::VM_PRO>();
    bar();
    if (wr == 1) bar();
    for (int T = 0; T < nkt; ++T) {
      // ---- Q0: (nq0, mh0); stage U2(T+1)
      rdA(T, 0);
      rdB(FB0, T, 0);
      dma(2, T + 1);
      bar();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_setprio(1);
      mma(0, 0, FB0);
      __builtin_amdgcn_s_setprio(0);
      wait_vm<C::VM_Q0>();
      bar();
      // ---- Q1: (nq0, mh1); stage U3(T+1)
      rdB(FB1, T, 1);
      dma(3, T + 1);
      bar();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_setprio(1);
      mma(0, 1, FB1);
      __builtin_amdgcn_s_setprio(0);
      wait_vm<C::VM_Q1>();
      bar();
      // ---- Q2: (nq1, mh1); stage U0(T+2)
      rdA(T, 1);
      dma(0, T + 2);
      bar();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_setprio(1);
      mma(1, 1, FB1);
      __builtin_amdgcn_s_setprio(0);
      wait_vm<C::VM_Q2>();
      bar();
      // ---- Q3: (nq1, mh0) from registers; stage U1(T+2)
      dma(1, T + 2);
      bar();
      __builtin_amdgcn_s_setprio(1);
      mma(1, 0, FB0);
      __builtin_amdgcn_s_setprio(0);
      wait_vm<C::VM_Q3>();
      bar();
    }
    if (wr == 0) bar();                         // barrier counts even again
  }
  wait_vm<0>();                                 // drain the clamped tail DMAs
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();

  nls_dense::dense_epilogue<2 * NQH, MT, ROPE>(acc, S, row0 + wr * (BN / 2), S.rows, wc * 16 * MT, kslice, ks, a, ws);
}

template <int BN, int MT, bool ROPE>
__global__ __launch_bounds__(512, 1) void hgemm10_kernel(SegList segs, GemvArgs a, int ks, float* ws, int ntiles,
                                                          int nmb) {
  extern __shared__ __attribute__((aligned(16))) uint8_t h10lds[];
  constexpr int BM = H10<BN, MT>::BM;
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
  const int row0 = (tile - S.tile_begin) * BN;       // (host tile counts use BN-row tiles)
  h10_tile<BN, MT, ROPE>(S, row0, kslice, ks, a, ws, h10lds);
}

template <int BN, int MT, bool ROPE>
int launch_e(const SegList& sl, int ntiles, int ks, float* ws, const GemvArgs& a, hipStream_t st) {
  constexpr int LDS = H10<BN, MT>::LDS, BM = H10<BN, MT>::BM;
  const int nmb = (a.M + BM - 1) / BM;
  const int grid = ((ntiles + 7) / 8) * 8 * nmb * ks;
  static bool attr = false;
  if (!attr) {   // > 64 KiB of dynamic LDS must be opted into
    if (hipFuncSetAttribute((const void*)hgemm10_kernel<BN, MT, ROPE>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) !=
        hipSuccess)
      return -1;
    attr = true;
  }
  hipLaunchKernelGGL((hgemm10_kernel<BN, MT, ROPE>), dim3(grid), dim3(512), LDS, st, sl, a, ks, ws, ntiles, nmb);
  return (int)hipGetLastError();
}

template <int BN, int MT>
int launch_t(const SegList& sl, int ntiles, int ks, float* ws, const GemvArgs& a, hipStream_t st) {
  return a.epi == EPI_ROPE ? launch_e<BN, MT, true>(sl, ntiles, ks, ws, a, st) : launch_e<BN, MT, false>(sl, ntiles, ks, ws, a, st);
}

// bn: weight rows per workgroup tile (256 or 128). Row blocks of 192 instead of 256 where their rounds over the 256 CUs, each three quarters as
// long, end earlier (Llama-3-8B at 384 rows: gate|up 99 -> 76 us, down 69 -> 57; 1500 rows: o 65 -> 56; 3000: down 308 -> 276). With 256 weight rows
// they must end a good deal earlier: 192 x 256 tiles multiply slower, and the last round is seldom full (28672 x 4096, rounds by length: 0.75 at
// 600 and 1100 rows 193 -> 169 and 292 -> 254 us, 0.875 at 3000 rows 638 -> 674, 0.9 at 2400 527 -> 537, 0.94 at 2048 417 -> 437).
// Blocks of 320 rows with 128 weight rows: a round of 224 workgroups reads 28672 x 4096 once, as do two of 192 x 256, for 320 rows instead of 384.
// In a running step of 320 rows 90.5 (384 rows, 192 x 256) -> 79.6 us, a head of 32000 92 -> 85; 640 rows 172 -> 162 and 186 -> 170.
int launch_dense10(int bn, const SegList& sl, int ntiles, int ks, float* ws, const GemvArgs& a, hipStream_t st) {
  auto rounds = [&](int bm) { return (long)((ntiles * ((a.M + bm - 1) / bm) * ks + 255) / 256) * bm; };
  const bool low = rounds(192) * 100 < rounds(256) * (bn == 256 ? 85 : 100);
  if (bn == 256) return low ? launch_t<256, 3>(sl, ntiles, ks, ws, a, st) : launch_t<256, 4>(sl, ntiles, ks, ws, a, st);
  if (bn == 128 && rounds(320) * 100 < (low ? rounds(192) : rounds(256)) * 97) return launch_t<128, 5>(sl, ntiles, ks, ws, a, st);
  if (bn == 128) return low ? launch_t<128, 3>(sl, ntiles, ks, ws, a, st) : launch_t<128, 4>(sl, ntiles, ks, ws, a, st);
  return -1;
}


}  // namespace nls_hg10
