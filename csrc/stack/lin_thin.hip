// Products of few inputs (gfx950): up to four sub-tiles of K (128 bf16 values), as the second halves of low-rank projections are.
//
// Such a launch is its outputs: there is nothing to pipeline, and a workgroup of the tiled GEMM spends its time on the way to LDS and
// back. Here a wave takes 64 outputs of 32 rows straight from memory: packed weights are in fragment order already, a lane's 16 bytes
// of a row are its fragment. No LDS, no barrier, all loads of a wave in flight at once, and many waves to a CU cover the epilogue's loads.
// 64 x 64 through LDS / this, us: 4000 x 4096 x 64 25.4 / 19.2, 8000 43.7 / 32.2 (the outputs at 5 TB/s: 13), 4000 x 2048 x 64 with sigpow
// 19.0 / 16.9, five segments of 1024 columns with tanh 39.8 / 33.0; with less than two workgroups to a CU the smaller tiles spread further.
#include "lin.h"

namespace nls_lin {

template <int NS>
__global__ __launch_bounds__(256) void lin_thin_kernel(LinArgs a, int ntot) {
  typedef __bf16 T;
  typedef LT<T> L;
  const int per = (ntot + 7) >> 3, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || id >= ntot) return;
  LinTile t;
  if (!lin_tile<64, 128>(a, id, t)) return;
  const LinSeg& S = a.s[t.seg];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (32 * wave >= t.cnt) return;
  const int nsub = S.nsub, nwt = (S.N + 15) >> 4;
  const uint8_t* wb = (const uint8_t*)S.w + (size_t)t.grp * S.wstride + lane * 16;
  const u32x4 zero = {0, 0, 0, 0};
  u32x4 A[4][NS], B[2][NS];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    int xr, yr;
    lin_row(S, t, 32 * wave + 16 * j + r, xr, yr);
    const T* x = (const T*)S.x + (size_t)xr * S.ldx + (size_t)t.grp * S.xgs + g * L::EL;
#pragma unroll
    for (int h = 0; h < NS; ++h) B[j][h] = h < nsub ? *reinterpret_cast<const u32x4*>(x + h * L::KS) : zero;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int h = 0; h < NS; ++h)
      A[i][h] = h < nsub ? *reinterpret_cast<const u32x4*>(wb + ((size_t)min((t.n0 >> 4) + i, nwt - 1) * nsub + h) * 1024) : zero;
  f32x4 acc[4][2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < NS; ++h)
        if (h < nsub) acc[i][j] = L::mma(A[i][h], B[j][h], acc[i][j]);
    }
  lin_epilogue<T>(S, t, acc, t.n0 + 4 * g, 32 * wave + r);
}

int lin_thin(LinArgs& a, hipStream_t st) {
  const int n = lin_count(a, 64, 128);
  if (n < 1) return -1;
  int ns = 0;
  for (int i = 0; i < a.nseg; ++i) {
    if (a.s[i].rows || a.s[i].ks > 1) return -1;
    ns = max(ns, a.s[i].nsub);
  }
  const dim3 grid((n + 7) / 8 * 8), block(256);
  if (ns <= 2) hipLaunchKernelGGL(lin_thin_kernel<2>, grid, block, 0, st, a, n);
  else if (ns <= 4) hipLaunchKernelGGL(lin_thin_kernel<4>, grid, block, 0, st, a, n);
  else return -1;
  return (int)hipGetLastError();
}

}  // namespace nls_lin
