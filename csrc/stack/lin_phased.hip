// The large prompt GEMM on packed bf16 weights: 256 weight rows x 256 activation rows per workgroup, in four phases per 64-deep step.
//
// What bounds the 256 x 128 tile of lin_gemm.hip: a wave's 64 x 64 block reads 16 KB of fragments from LDS per step for 32 MFMAs, so
// the eight waves' reads (128 KB, 1024 cycles) last as long as their MFMAs (1024 cycles per SIMD), and its one barrier per step puts all
// waves into the same section at once. Here a wave owns 128 x 64 (24 KB for 64 MFMAs) and
//   * 8 waves = 2 groups (wr: 128 weight rows each) x 4 (wc: 64 rows each); group 1 runs one barrier behind group 0, so that on every
//     SIMD (a wave of each) one wave's MFMAs overlap the other's LDS reads and DMA;
//   * a step is 4 phases of 16 MFMAs: (weights 0, rows 0), (0, 1), (1, 1), (1, 0) of the halves of the wave's block; each phase reads
//     the fragments that it lacks and starts one 16 KB DMA unit: U0 = weight halves 0, U1 = row halves 0, U2 = row halves 1,
//     U3 = weight halves 1, each restaged as soon as both groups have read it (two phases later): U2 and U3 of the next step in phases
//     0 and 1, U0 and U1 of the one after it in phases 2 and 3. The last three units stay in flight (vmcnt(6));
//   * two 64 KB buffers, one workgroup per CU, which stays for several tiles: the DMA of the next tile's first steps takes the place of
//     the last steps' successors, so that it is under way during the epilogue.
// Weight sub-tiles are packed in fragment order and arrive verbatim; activation sub-tiles are swizzled as in lin_gemm.hip.
// 2000 x 35888 x 4096 (rows x weights x K): 743 us on 256 x 128 -> 490 us (1.20 PFLOP/s), 4096 x 35888 x 4096: 1311 -> 886 us (1.36), 4096 x 4096 x
// 17408, a single round of tiles: 521 -> 407 us (1.44); a workgroup for each tile instead: 644, 1165 and 422 us. What is left: 16 KB of
// LDS reads per 43 MFMAs, and rounds of tiles that the shape does not fill.
#include "../kernels/lds_dma.h"
#include "lin.h"

namespace nls_lin {
using nls_dma::glds16;
using nls_dma::lds_addr;

constexpr int PB = 256;                                  // weight and activation rows of a tile
constexpr int PHALF = PB * 128, PSTG = 2 * PHALF;        // bytes of an operand's half, of a step's buffer

template <int N>
DEVI void ph_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
DEVI void ph_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <typename P>
DEVI P* uniform(P* p) {                                  // (a value that the compiler does not see to be the wave's)
  const uint64_t v = (uint64_t)p;
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32)), lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  return (P*)((uint64_t)hi << 32 | lo);
}

// where a tile's operands start: weights by wave, rows by lane
struct PhTile {
  LinTile t;
  const uint8_t* w[2];
  const __bf16* x[2];
  int nst;                                               // steps
};

__global__ __launch_bounds__(512, 1) void lin_phased_kernel(LinArgs a, int ntot) {
  extern __shared__ __attribute__((aligned(16))) uint8_t phlds[];
  typedef LT<__bf16> L;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wr = wave >> 2, wc = wave & 3;
  // tile ids are dealt to the XCDs in contiguous ranges, which an XCD's workgroups walk together
  const int xcd = blockIdx.x & 7, nx = gridDim.x >> 3;
  int listed, gap;                                       // (of a routed first segment)
  lin_listed(a, PB, listed, gap);
  ntot -= gap;
  const int per = (ntot + 7) >> 3, last = min(ntot, (xcd + 1) * per);

  // DMA: in every unit a wave brings both sub-tiles (k halves) of one 16-row tile. Tiles 0 .. 3 and 8 .. 11 of the weights are U0, the
  // others U3; tiles with (tile & 2) == 0 of the rows are U1, the others U2.
  const int ta = (wave & 3) + 8 * (wave >> 2), tb = (wave & 1) + 4 * (wave >> 1);
  auto open = [&](int id, PhTile& p) __attribute__((always_inline)) -> int {      // tile id, if there is one; else -1
    if (id >= last || !lin_tile<PB, PB>(a, id < listed ? id : id + gap, p.t)) return -1;
    p.t.grp = __builtin_amdgcn_readfirstlane(p.t.grp);
    p.t.cnt = __builtin_amdgcn_readfirstlane(p.t.cnt);
    p.t.rows = uniform(p.t.rows);
    const LinSeg& S = a.s[p.t.seg];
    const int nsub = S.nsub, nwt = (S.N + 15) >> 4;
    const int jb = (nsub >> 1) * p.t.ks / S.ks;
    p.nst = (nsub >> 1) * (p.t.ks + 1) / S.ks - jb;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      p.w[h] = uniform((const uint8_t*)S.w + (size_t)p.t.grp * S.wstride +
                       ((size_t)min((p.t.n0 >> 4) + ta + 4 * h, nwt - 1) * nsub + 2 * jb) * 1024);
      int xr, yr;
      lin_row(S, p.t, 16 * (tb + 2 * h) + (lane >> 2), xr, yr);
      p.x[h] = (const __bf16*)S.x + (size_t)xr * S.ldx + (size_t)p.t.grp * S.xgs + ((lane & 3) ^ lin_swz(lane >> 2)) * L::EL +
               (size_t)jb * 2 * L::KS;
    }
    return id;
  };
  const uint32_t base = __builtin_amdgcn_readfirstlane(lds_addr(phlds));
  auto dma_w = [&](int h, const uint8_t* s, uint32_t buf) __attribute__((always_inline)) {      // U0 / U3
    const uint32_t d = base + buf + (uint32_t)(ta + 4 * h) * 2048u;
    glds16(s, lane * 16, d);
    glds16(s, lane * 16 + 1024, d + 1024u);
  };
  auto dma_x = [&](int h, const __bf16* s, uint32_t buf) __attribute__((always_inline)) {       // U1 / U2
    const uint32_t d = base + buf + PHALF + (uint32_t)(tb + 2 * h) * 2048u;
    glds16(s, d);
    glds16(s + L::KS, d + 1024u);
  };

  u32x4 A[4][2], B0[2][2], B1[2][2];
  const int xfo = r * 64 + ((g ^ lin_swz(r)) << 4);
  auto rd_w = [&](int h, uint32_t buf) __attribute__((always_inline)) {
    const uint8_t* p = phlds + buf + (8 * wr + 4 * h) * 2048 + lane * 16;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) A[i][s] = *reinterpret_cast<const u32x4*>(p + (2 * i + s) * 1024);
  };
  auto rd_x = [&](u32x4 (&B)[2][2], int h, uint32_t buf) __attribute__((always_inline)) {
    const uint8_t* p = phlds + buf + PHALF + (4 * wc + 2 * h) * 2048 + xfo;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) B[i][s] = *reinterpret_cast<const u32x4*>(p + (2 * i + s) * 1024);
  };
  f32x4 acc[8][4];
  auto mma = [&](int nh, int mh, const u32x4 (&B)[2][2]) __attribute__((always_inline)) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[4 * nh + i][2 * mh + j] = L::mma(A[i][s], B[j][s], acc[4 * nh + i][2 * mh + j]);
    __builtin_amdgcn_s_setprio(0);
  };
  auto reads_done = []() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };

  PhTile nxt;
  int id = open(xcd * per + (blockIdx.x >> 3), nxt);
  if (id < 0) return;
  // the four streams' next sources: halves 0 run two steps ahead of the multiplications, halves 1 one step
  const uint8_t *w0 = nxt.w[0], *w1 = nxt.w[1];
  const __bf16 *x0 = nxt.x[0], *x1 = nxt.x[1];
  uint32_t buf = 0;                                      // byte offset of the step's buffer
  dma_w(0, w0, 0);
  dma_x(0, x0, 0);
  dma_x(1, x1, 0);
  dma_w(1, w1, 0);
  dma_w(0, w0 += 2048, PSTG);
  dma_x(0, x0 += 2 * L::KS, PSTG);
  ph_wait<4>();                                          // step 0 has landed
  ph_barrier();
  for (;;) {
    const LinTile t = nxt.t;
    const int nst = nxt.nst, nid = open(id + nx, nxt);
    if (nid < 0) nxt.w[0] = w0, nxt.w[1] = w1, nxt.x[0] = x0, nxt.x[1] = x1;       // (staged, not used)
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // group 1 starts a barrier later and ends with the other one: left apart over the epilogue, it would wait with its last phase until group
    // 0's epilogue is done, and group 0 for its own
    if (wr == 1) ph_barrier();
    for (int j = 0; j < nst; ++j, buf ^= PSTG) {
      rd_w(0, buf);
      rd_x(B0, 0, buf);
      x1 = j + 1 == nst ? nxt.x[1] : x1 + 2 * L::KS;
      dma_x(1, x1, buf ^ PSTG);
      ph_barrier();
      reads_done();
      mma(0, 0, B0);
      ph_wait<6>();
      ph_barrier();

      rd_x(B1, 1, buf);
      w1 = j + 1 == nst ? nxt.w[1] : w1 + 2048;
      dma_w(1, w1, buf ^ PSTG);
      ph_barrier();
      reads_done();
      mma(0, 1, B1);
      ph_wait<6>();
      ph_barrier();

      rd_w(1, buf);
      w0 = j + 2 == nst ? nxt.w[0] : w0 + 2048;
      dma_w(0, w0, buf);
      ph_barrier();
      reads_done();
      mma(1, 1, B1);
      ph_wait<6>();
      ph_barrier();

      x0 = j + 2 == nst ? nxt.x[0] : x0 + 2 * L::KS;
      dma_x(0, x0, buf);
      ph_barrier();
      mma(1, 0, B0);
      ph_wait<6>();
      ph_barrier();
    }
    if (wr == 0) ph_barrier();
    lin_epilogue<__bf16>(a.s[t.seg], t, acc, t.n0 + 128 * wr + 4 * g, 64 * wc + r);
    if (nid < 0) break;
    id = nid;
  }
  ph_wait<0>();                                          // the staged tail lands before the workgroup's LDS is freed
}

int lin_phased(LinArgs& a, hipStream_t st) {
  const int n = lin_count(a, PB, PB);
  if (n < 1) return -1;
  for (int i = 0; i < a.nseg; ++i)
    if ((i && a.s[i].rows) || a.s[i].nsub / 2 / a.s[i].ks < 3) return -1;      // (the streams run two steps ahead, and a last tile's tail restages steps 1 and 2)
  static bool attr = false;
  if (!attr) {
    if (hipFuncSetAttribute((const void*)lin_phased_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * PSTG) != hipSuccess)
      return -1;
    attr = true;
  }
  hipLaunchKernelGGL(lin_phased_kernel, dim3(min((n + 7) / 8 * 8, 256)), dim3(512), 2 * PSTG, st, a, n);
  return (int)hipGetLastError();
}

}  // namespace nls_lin
