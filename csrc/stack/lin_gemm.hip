// Tiled MFMA GEMM on packed bf16 weights (prompt chunks, large decode batches, routed experts with many rows), and on f32 weights where a CU has
// one workgroup (beyond that lin_split.hip is the faster one).
//
// BN weight rows x BM activation rows per workgroup; K advances two 1 KiB sub-tiles (64 bf16 / 32 f32 values) per
// step. Both operands arrive by LDS-DMA into NST-deep rings: weight sub-tiles verbatim (already in fragment order),
// activation sub-tiles with the 16-byte chunks of a row permuted on the DMA source (chunk ^ swz(row)), so every
// fragment is one conflict-free ds_read_b128. One raw barrier per step with a counted vmcnt leaves the later stages
// in flight. Routed rows (experts) are gathered by the DMA's per-lane source addresses.
// Tile ids are dealt to the 8 XCDs in contiguous ranges, a few m-tiles innermost (lin_tile): the workgroups that run
// together on an XCD form a block of weight and row tiles and read both through its L2.
// Weights of a tile that no other one shares (LinTile::once) come with the non-temporal hint: few rows make a launch a read of the weights, and
// without the hint they push the rows, caches and states of the step out of the caches (us in a running step, without / with: 64 x 35888 x 4096
// 75.7 / 59.7, 4.9 TB/s, 64 x 32000 68.7 / 55.5, eight experts of 50 rows 94.5 / 76.3 and 83.0 / 78.0). Weights of two row tiles need the L2 for the
// second one's read: with the hint eight experts of 75 rows took 142 -> 163 us.
// A CU takes in some 50 GB/s of a launch's operands whatever its waves and stages (96 workgroups read cold weights at 4.7 TB/s, 256 at 6.8), and
// the activation rows count as much as the weights: the 64 x 32 tile brings half as many of them as 64 x 64 (16 x 10240 x 4096 18.2 / 19.2 us, 24 rows
// 20.0 / 20.5; streamed with the rows from the caches, lin_small.hip, 23.7 and 24).
#include <type_traits>
#include "../kernels/lds_dma.h"
#include "lin.h"

namespace nls_lin {
using nls_dma::glds16;
using nls_dma::glds16_nt;
using nls_dma::lds_addr;
using nls_dma::wait_vm_lgkm0;

int lin_phased(LinArgs& a, hipStream_t st);      // lin_phased.hip
int lin_split(LinArgs& a, int cfg, hipStream_t st);      // lin_split.hip
int lin_thin(LinArgs& a, hipStream_t st);        // lin_thin.hip
int lin_pair(LinArgs& a, int nt, int mt, hipStream_t st);      // lin_pair.hip

template <int BN, int BM, int WN, int WM, int NST>
struct LG {
  static constexpr int NWV = WN * WM;
  static constexpr int NTW = BN / 16 / WN;          // weight tiles per wave
  static constexpr int MTW = BM / 16 / WM;          // row tiles per wave
  static constexpr int WST = BN * 128, XST = BM * 128, STG = WST + XST;   // bytes per stage
  static constexpr int NW = BN / 8 / NWV, NX = BM / 8 / NWV;              // DMA instructions per wave per stage
  static constexpr int LDS = NST * STG;
  static_assert(NW >= 1 && NX >= 2 && NX % 2 == 0 && NTW >= 1 && MTW >= 1, "tile too small for the wave count");
  static_assert(LDS <= 160 * 1024, "LDS");
};

// How a launch's weights are fetched: without the hint, with it, or as each tile asks (LinTile::once). Kernels of their own: one with both walks is
// twice the code, which a step's launches feel. Steps of four layers at 64 / 96 / 128 rows, us, both walks in a kernel / one: 148 MB of weights
// 180 / 181, 198 / 190, 207 / 194, 221 MB 210 / 205, 201 / 196, 209 / 202, 529 MB 236 / 234, 308 / 288, 321 / 298; without the hint 184, 189, 193;
// 198, 195, 202; 255, 306, 323.
enum Fetch : int { KEEP, STREAM, BY_TILE };

template <typename T, int BN, int BM, int WN, int WM, int NST, int FETCH>
__global__ __launch_bounds__(64 * WN * WM) void lin_gemm_kernel(LinArgs a, int ntot) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lglds[];
  typedef LG<BN, BM, WN, WM, NST> G;
  typedef LT<T> L;
  constexpr int NW = G::NW, NX = G::NX, NTW = G::NTW, MTW = G::MTW;
  int listed = ntot, gap = 0;
  if constexpr (FETCH == BY_TILE) lin_listed(a, BN, listed, gap);      // (a routed segment is fetched by tile)
  ntot -= gap;
  const int per = (ntot + 7) >> 3, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || id >= ntot) return;
  LinTile t;
  if (!lin_tile<BN, BM>(a, id < listed ? id : id + gap, t)) return;
  const LinSeg& S = a.s[t.seg];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wn = wave / WM, wm = wave % WM;
  const int nsub = S.nsub;
  const int jb = (nsub >> 1) * t.ks / S.ks, nst = (nsub >> 1) * (t.ks + 1) / S.ks - jb;     // this split's steps
  const int nwt = (S.N + 15) >> 4;

  const uint8_t* wbase = (const uint8_t*)S.w + (size_t)t.grp * S.wstride + lane * 16;
  const uint8_t* wsrc[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int q = NW * wave + i;                     // stage sub-tile: weight tile q >> 1, k half q & 1
    wsrc[i] = wbase + ((size_t)min((t.n0 >> 4) + (q >> 1), nwt - 1) * nsub + (q & 1)) * 1024;
  }
  const T* xsrc[NX / 2];
#pragma unroll
  for (int i = 0; i < NX / 2; ++i) {
    const int row = 16 * ((NX * wave) / 2 + i) + (lane >> 2);
    int xr, yr;
    lin_row(S, t, row, xr, yr);
    xsrc[i] = (const T*)S.x + (size_t)xr * S.ldx + (size_t)t.grp * S.xgs + ((lane & 3) ^ lin_swz(lane >> 2)) * L::EL;
  }
  const uint32_t base = __builtin_amdgcn_readfirstlane(lds_addr(lglds));
  const uint32_t wl = base + (uint32_t)(NW * wave) * 1024u;
  const uint32_t xl = base + G::WST + (uint32_t)(NX * wave) * 1024u;
  auto dma = [&](int j, int stage, auto once) __attribute__((always_inline)) {     // step j (clamped) -> stage
    const int jc = jb + min(j, nst - 1);
    const uint32_t so = (uint32_t)stage * G::STG;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      if constexpr (decltype(once)::value) glds16_nt(wsrc[i] + (size_t)jc * 2048, wl + so + i * 1024);
      else glds16(wsrc[i] + (size_t)jc * 2048, wl + so + i * 1024);
    }
#pragma unroll
    for (int i = 0; i < NX; ++i) glds16(xsrc[i >> 1] + (size_t)(2 * jc + (i & 1)) * L::KS, xl + so + i * 1024);
  };
  f32x4 acc[NTW][MTW];
#pragma unroll
  for (int i = 0; i < NTW; ++i)
#pragma unroll
    for (int j = 0; j < MTW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int xfo = r * 64 + ((g ^ lin_swz(r)) << 4);
  auto step = [&](int stage) __attribute__((always_inline)) {
    const uint8_t* wb = lglds + stage * G::STG + lane * 16;
    const uint8_t* xb = lglds + stage * G::STG + G::WST + xfo;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4 A[NTW], B[MTW];
#pragma unroll
      for (int i = 0; i < NTW; ++i) A[i] = *reinterpret_cast<const u32x4*>(wb + ((wn * NTW + i) * 2 + h) * 1024);
#pragma unroll
      for (int i = 0; i < MTW; ++i) B[i] = *reinterpret_cast<const u32x4*>(xb + ((wm * MTW + i) * 2 + h) * 1024);
#pragma unroll
      for (int i = 0; i < NTW; ++i)
#pragma unroll
        for (int jj = 0; jj < MTW; ++jj) acc[i][jj] = L::mma(A[i], B[jj], acc[i][jj]);
    }
  };
  constexpr int FL = (NST - 2) * (NW + NX);           // DMA instructions left in flight across the barrier
  // step j is in stage j % NST: NST steps to a pass of the loop, so that stages are constants and the accumulators stay where they are
  auto turn = [&](int j, int stage, auto once) __attribute__((always_inline)) {
    dma(j + NST - 1, (stage + NST - 1) % NST, once);  // that stage was last read in step j - 1: retired
    step(stage);
    wait_vm_lgkm0<FL>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto walk = [&](auto once) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NST - 1; ++j) dma(j, j, once);
    wait_vm_lgkm0<FL>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int j0 = 0;
    for (; j0 + NST <= nst; j0 += NST)
#pragma unroll
      for (int s = 0; s < NST; ++s) turn(j0 + s, s, once);
#pragma unroll
    for (int s = 0; s < NST - 1; ++s)
      if (j0 + s < nst) turn(j0 + s, s, once);        // (uniform)
  };
  if constexpr (FETCH == BY_TILE) {
    if (__builtin_amdgcn_readfirstlane(t.once)) walk(std::true_type{});
    else walk(std::false_type{});
  } else {
    walk(std::integral_constant<bool, FETCH == STREAM>{});
  }
  wait_vm_lgkm0<0>();                                 // the clamped tail DMAs land before the workgroup's LDS is freed
  lin_epilogue<T>(S, t, acc, t.n0 + 16 * wn * NTW + 4 * g, 16 * wm * MTW + r);
}

template <typename T, int BN, int BM, int WN, int WM, int NST, int FETCH>
int gemm_f(const LinArgs& a, int n, hipStream_t st) {
  typedef LG<BN, BM, WN, WM, NST> G;
  static bool attr = false;
  if (!attr) {
    if (hipFuncSetAttribute((const void*)lin_gemm_kernel<T, BN, BM, WN, WM, NST, FETCH>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS) != hipSuccess)
      return -1;
    attr = true;
  }
  hipLaunchKernelGGL((lin_gemm_kernel<T, BN, BM, WN, WM, NST, FETCH>), dim3((n + 7) / 8 * 8), dim3(64 * G::NWV), G::LDS, st,
                     a, n);
  return (int)hipGetLastError();
}

template <typename T, int BN, int BM, int WN, int WM, int NST>
int gemm_t(LinArgs& a, hipStream_t st) {
  const int n = lin_count(a, BN, BM);
  if (n < 1) return -1;
  int once = 0, several = 0;                          // segments of one row tile, and of more
  for (int i = 0; i < a.nseg; ++i) {
    once |= a.s[i].rows || a.s[i].M <= BM;
    several |= a.s[i].rows || a.s[i].M > BM;
  }
  if (!once) return gemm_f<T, BN, BM, WN, WM, NST, KEEP>(a, n, st);
  return several ? gemm_f<T, BN, BM, WN, WM, NST, BY_TILE>(a, n, st) : gemm_f<T, BN, BM, WN, WM, NST, STREAM>(a, n, st);
}

int lin_gemm(LinArgs& a, int cfg, hipStream_t st) {
  if (cfg >= 256) return lin_pair(a, cfg >> 4 & 15, cfg & 15, st);
  switch (cfg) {
    case 0: return gemm_t<__bf16, 64, 64, 2, 2, 3>(a, st);
    case 1: return gemm_t<__bf16, 128, 64, 4, 1, 3>(a, st);
    case 2: return gemm_t<__bf16, 128, 128, 2, 2, 2>(a, st);
    case 3: return gemm_t<__bf16, 256, 128, 4, 2, 3>(a, st);
    case 4: return gemm_t<__bf16, 256, 256, 4, 2, 2>(a, st);
    case 5: return gemm_t<__bf16, 64, 64, 2, 2, 8>(a, st);
    case 6: return gemm_t<__bf16, 192, 128, 4, 2, 3>(a, st);
    case 7: return lin_phased(a, st);
    case 8: return gemm_t<__bf16, 96, 64, 2, 2, 4>(a, st);
    case 9: return gemm_t<__bf16, 160, 64, 2, 2, 4>(a, st);
    case 10: return gemm_t<__bf16, 128, 64, 2, 2, 4>(a, st);
    case 11: return gemm_t<__bf16, 96, 128, 2, 2, 4>(a, st);
    case 12: return gemm_t<__bf16, 64, 32, 2, 1, 8>(a, st);
    case 13: return lin_thin(a, st);
  }
  return -1;
}

}  // namespace nls_lin

extern "C" {

// cfg: tile of the launch (BN x BM): 0 = 64 x 64, 1 = 128 x 64, 2 = 128 x 128, 3 = 256 x 128, 4 = 256 x 256 in two stages (a launch's
// own choice never is this one), 5 = 64 x 64 with 8 stages in flight (launches of at most one workgroup per CU),
// 6 = 192 x 128, 7 = 256 x 256 in phases, 8 = 96 x 64, 9 = 160 x 64, 10 = 128 x 64 with four stages, 11 = 96 x 128, 12 = 64 x 32 with 8 stages,
// 13 = 64 x 128 straight from memory (K up to 128, no routed rows), 256 + 16 nt + mt = 32 nt x 32 mt, two wave groups on alternate k-steps (no row
// lists and maps).
// f32: 5 = 64 x 64 on the f32 MFMA in three stages, 0, 1 and 2 in bf16 parts; the others run on one of these, but for 7 and 13 and for routed
// rows on 4 and from 256 on, which are refused.
int nls_lin_gemm(const void* args, int f32, int cfg, void* stream) {
  nls_lin::LinArgs a = *reinterpret_cast<const nls_lin::LinArgs*>(args);
  using namespace nls_lin;
  hipStream_t st = (hipStream_t)stream;
  return !f32 ? lin_gemm(a, cfg, st) : cfg == 5 ? gemm_t<float, 64, 64, 2, 2, 3>(a, st) : lin_split(a, cfg, st);
}

}  // extern "C"
