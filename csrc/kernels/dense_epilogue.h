// Epilogue of the dense f16 GEMMs (hgemm10.hip, hgemm11.hip): f32 / residual add / f16 / SwiGLU / split-K slabs / arg-max keys, or RoPE with
// the cache rows.
#pragma once
#include "qgemm_dma.h"

namespace nls_dense {
using namespace nls_gemv;

// A wave's NW x MT accumulator tiles: lane holds weight rows nb + 16i + 4(l >> 4) + e (those below nend are stored), activation
// row mb + 16j + (l & 15)
// ROPE: the RoPE epilogue, in kernels of its own: beside it the 256 x 256 tile spilled 21 registers
template <int NW, int MT, bool ROPE>
DEVI void dense_epilogue(f32x4 (&acc)[NW][MT], const Seg& S, int nb, int nend, int mb, int kslice, int ks, const GemvArgs& a, float* ws) {
  const int lane = threadIdx.x & 63;
  const int M = a.M;
  const int g4 = 4 * (lane >> 4), r16 = lane & 15;
  if (!ROPE && (ks > 1 || a.epi == EPI_SLABS)) {
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int n = nb + 16 * i + g4;
      if (n >= nend) continue;
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const int m = mb + 16 * j + r16;
        if (m >= M) continue;
        *reinterpret_cast<f32x4*>(ws + ((size_t)kslice * a.mtot + a.m0 + m) * a.pad + S.tile_begin_col + n) = acc[i][j];
      }
    }
    return;
  }
  const float al = a.alpha;
  if constexpr (ROPE) {
    // RoPE pairs (e, e + 1) of the lane's 4 consecutive weight rows: no cross-lane traffic
    if ((a.D & 3) || (a.ldq & 3)) {
      for (int i = 0; i < NW; ++i) {               // (moved up instead of unrolled: the general form is long)
        const int n = nb + 16 * i + g4;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          const int m = mb + 16 * j + r16;
          const f32x4 v = acc[0][j] * al;
          if (m < M && n < nend) {
            rope_store1(a, S.ycol + n, a.m0 + m, v[0], v[1]);
            rope_store1(a, S.ycol + n + 1, a.m0 + m, v[1], v[0]);
            rope_store1(a, S.ycol + n + 2, a.m0 + m, v[2], v[3]);
            rope_store1(a, S.ycol + n + 3, a.m0 + m, v[3], v[2]);
          }
#pragma unroll
          for (int k = 0; k + 1 < NW; ++k) acc[k][j] = acc[k + 1][j];
        }
      }
      return;
    }
    // 4 columns of one head: a row's slot and position once, 8-byte stores (one value at a time, with its own loads,
    // 3000 x 6144 x 4096 took 307 us, 181 this way)
    typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
    long sl[MT];
    const float* cs[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const int m = a.m0 + min(mb + 16 * j + r16, M - 1);
      sl[j] = a.slot[m];
      cs[j] = a.cs + (size_t)a.pos[m] * a.D;
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int n = nb + 16 * i + g4;
      if (n >= nend) continue;
      const int col = S.ycol + n, h = col / a.D, dd = col - h * a.D;
      f32x4 bias = {0.f, 0.f, 0.f, 0.f};
      if (a.bias) bias = f32x4{a.bias[col], a.bias[col + 1], a.bias[col + 2], a.bias[col + 3]};
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const int m = mb + 16 * j + r16;
        if (m >= M) continue;
        f32x4 v = acc[i][j] * al + bias;
        __bf16* d = nullptr;
        if (h < a.Hq + a.Hkv) {
          const float2 c0 = *reinterpret_cast<const float2*>(cs[j] + dd), c1 = *reinterpret_cast<const float2*>(cs[j] + dd + 2);
          v = f32x4{v[0] * c0.x - v[1] * c0.y, v[0] * c0.y + v[1] * c0.x, v[2] * c1.x - v[3] * c1.y, v[2] * c1.y + v[3] * c1.x};
          if (h < a.Hq) d = a.q_out + (size_t)(a.m0 + m) * a.ldq + col;
          else if (sl[j] >= 0) d = a.kc + ((size_t)sl[j] * a.Hkv + (h - a.Hq)) * a.D + dd;
        } else if (sl[j] >= 0) {
          d = a.vc + ((size_t)sl[j] * a.Hkv + (h - a.Hq - a.Hkv)) * a.D + dd;
        }
        if (d) *reinterpret_cast<bf4*>(d) = bf4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
      }
    }
    return;
  }
  if (a.epi == EPI_SWIGLU) {
#pragma unroll
    for (int i = 0; i < NW; ++i) {
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        f32x4 u;
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] = __shfl_xor(acc[i][j][e] * al, 32, 64);
        const int n16 = nb + 16 * i, m = mb + 16 * j + r16;
        if (lane < 32 && m < M && n16 < nend) {
          typedef _Float16 h4 __attribute__((ext_vector_type(4)));
          h4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (_Float16)(silu(acc[i][j][e] * al) * u[e]);
          *reinterpret_cast<h4*>(reinterpret_cast<act_t*>(a.y) + (size_t)m * a.ldy + S.ycol + (n16 >> 1) + g4) = o;
        }
      }
    }
    return;
  }
  if (a.epi != EPI_ARGMAX) {
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int n = nb + 16 * i + g4;
      if (n >= nend) continue;
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const int m = mb + 16 * j + r16;
        if (m >= M) continue;
        const f32x4 v = acc[i][j] * al;
        if (a.epi == EPI_ACT) {
          typedef _Float16 h4 __attribute__((ext_vector_type(4)));
          *reinterpret_cast<h4*>(reinterpret_cast<act_t*>(a.y) + (size_t)m * a.ldy + S.ycol + n) =
              h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
        } else {
          f32x4* p = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.y) + (size_t)m * a.ldy + S.ycol + n);
          *p = a.epi == EPI_ADD_F32 ? *p + v : v;
        }
      }
    }
  }
  if (a.argmax) {
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      unsigned long long k = 0ull;
#pragma unroll
      for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = nb + 16 * i + g4 + e;
          const unsigned long long kk = n < nend ? argmax_key(acc[i][j][e] * al, S.ycol + n) : 0ull;
          k = kk > k ? kk : k;
        }
      unsigned long long o = __shfl_xor(k, 16, 64);
      k = o > k ? o : k;
      o = __shfl_xor(k, 32, 64);
      k = o > k ? o : k;
      const int m = mb + 16 * j + r16;
      if (lane < 16 && m < M) atomicMax(a.argmax + m, k);
    }
  }
}

}  // namespace nls_dense
