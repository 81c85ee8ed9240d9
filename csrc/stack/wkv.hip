// "wkv" time mixing (gfx950): the token shift, the recurrence over runs of tokens, and the entry points of its single-token step
// (scan.h).
//
// The scan is sequential in the tokens of a run, so a position's result does not depend on how its sequence was cut
// into steps. Parallelism is (run, head, value columns) x lanes: a lane holds DP / PARTS key rows of CPL value columns in
// registers, PARTS neighbouring lanes cover the keys and close the sum with in-row lane exchanges (DPP). Few runs take
// many key parts (short per-token chains on all CUs). Tokens are staged in LDS in chunks of CH as f32, the next chunk's
// loads in flight while the current one runs.
#include <type_traits>
#include "scan.h"

namespace nls_wkv {
using namespace nls_scan;

// ---- token shift: m_s[t] = h[t] + (h[t - 1] - h[t]) * mu_s for NS mixes; h = the f32 residual row. The row before
// a run's first is the slot's previous token (zeros at position 0).
constexpr int NS = 5;
struct Mix {
  const float* x;
  const float* mu;      // [NS][D]
  const float* prev;    // [slots][prev stride]
  void* out;            // [NS][rows cap][ldo]
  const int* runs;      // [nruns][4]
  const int* tok_seq;   // row -> run
  long ldx, ldp, ldo, mstride;
  int D, f32;
};

template <typename T>
__global__ __launch_bounds__(256) void shift_mix_kernel(Mix p) {
  const int t = blockIdx.x;
  const int* run = p.runs + 4 * p.tok_seq[t];
  const int t0 = run[0], n = run[1], slot = run[2], pos0 = run[3];
  if (slot < 0 || t < t0 || t >= t0 + n) return;
  const float* h = p.x + (size_t)t * p.ldx;
  const float* q = t > t0 ? h - p.ldx : (pos0 > 0 ? p.prev + (size_t)slot * p.ldp : nullptr);
  T* o = reinterpret_cast<T*>(p.out) + (size_t)t * p.ldo;
  for (int i = blockIdx.y * 256 + threadIdx.x; i < p.D; i += gridDim.y * 256) {
    const float a = h[i], d = (q ? q[i] : 0.f) - a;
#pragma unroll
    for (int s = 0; s < NS; ++s) o[s * p.mstride + i] = (T)(a + d * p.mu[s * p.D + i]);
  }
}

// DP: key channels padded to a multiple of 32 (zeros past D). VEC: D = DP and 16-byte aligned rows (8 values of an operand's row to
// a thread: a quarter of the loads' addresses; 3500 tokens, 32 heads of 64: 433 -> 355 us)
template <typename T, int DP, int PARTS, int CPL, bool VEC>
__global__ __launch_bounds__(256) void wkv_scan_kernel(Scan p) {
  constexpr int WC = 256 / PARTS * CPL;          // value columns per workgroup
  constexpr int CH = DP <= 64 ? 32 : (DP <= 128 ? 16 : 8);   // tokens per staged chunk
  constexpr int R = DP / PARTS;                  // state rows per lane
  constexpr int LR = DP + 4;                     // LDS row stride
  constexpr int NV = (CH * DP + 255) / 256;      // staged values per thread and operand
  __shared__ __attribute__((aligned(16))) float rs[CH][LR], ks[CH][LR], ws[CH][LR];
  __shared__ __attribute__((aligned(16))) float vs[CH][WC], ruk[CH];
  const int* run = p.runs + 4 * blockIdx.y;
  const int t0 = run[0], n = run[1], slot = run[2], pos0 = run[3];
  if (slot < 0 || n < 1) return;
  const int D = p.D;
  const int ncb = (D + WC - 1) / WC;
  const int head = blockIdx.x / ncb, c0 = (blockIdx.x % ncb) * WC;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int part = lane & (PARTS - 1), col = (wave * (64 / PARTS) + lane / PARTS) * CPL;
  const int j = c0 + col;
  const size_t hb = (size_t)head * D;
  const T* rp = (const T*)p.r + hb;
  const T* kp = (const T*)p.k + hb;
  const T* vp = (const T*)p.v + hb;
  const float* wp = p.w + hb;
  float* st = p.state + (size_t)slot * p.sstride + hb * D;

  float S[CPL][R];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const int row = part * R + i;
      S[c][i] = (pos0 > 0 && row < D && j + c < D) ? st[(size_t)row * D + j + c] : 0.f;
    }
  float ur[DP / 16];                             // u of the bonus sums' columns
#pragma unroll
  for (int q = 0; q < DP / 16; ++q) {
    const int i = (threadIdx.x & 15) + 16 * q;
    ur[q] = i < D ? p.u[hb + i] : 0.f;
  }
  // these loads have arrived before the first chunk's go out: the loop over tokens would wait for all loads in flight otherwise
#pragma unroll
  for (int c = 0; c < CPL; ++c)
#pragma unroll
    for (int i = 0; i < R; ++i) asm volatile("" : "+v"(S[c][i]));
#pragma unroll
  for (int q = 0; q < DP / 16; ++q) asm volatile("" : "+v"(ur[q]));
  // the next chunk, as it lies in memory: no branch and no conversion, which would wait for the load, until it is staged (3500
  // tokens, 32 heads of 64: 748 us with a branch around each load, 10 round trips to memory a chunk; 433 without)
  constexpr int NU = (CH * WC + 255) / 256;
  typedef T tv8 __attribute__((ext_vector_type(8), aligned(16)));
  typedef float fv8 __attribute__((ext_vector_type(8), aligned(16)));
  static_assert(!VEC || (CH * DP == 2048 && CH * WC <= 2048), "8 values to a thread");
  T fr[VEC ? 1 : NV], fk[VEC ? 1 : NV], fv[VEC ? 1 : NU];
  float fw[VEC ? 1 : NV];
  tv8 r8, k8, v8;
  fv8 w8;
  const int et = threadIdx.x / (DP / 8), ei = threadIdx.x % (DP / 8) * 8;                               // VEC: a thread's token and keys
  const int vt = threadIdx.x % (CH * WC / 8) / (WC / 8), vi = threadIdx.x % (WC / 8) * 8;                 // and token and columns
  auto fetch = [&](int base) __attribute__((always_inline)) {
    if constexpr (VEC) {
      const size_t row = t0 + min(base + et, n - 1), vrow = t0 + min(base + vt, n - 1);
      r8 = *reinterpret_cast<const tv8*>(rp + row * p.ld + ei);
      k8 = *reinterpret_cast<const tv8*>(kp + row * p.ld + ei);
      w8 = *reinterpret_cast<const fv8*>(wp + row * p.ldw + ei);
      v8 = *reinterpret_cast<const tv8*>(vp + vrow * p.ld + c0 + vi);
      return;
    }
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const int e = threadIdx.x + q * 256, tt = e / DP, i = min(e % DP, D - 1);
      const size_t row = (size_t)(t0 + min(base + tt, n - 1));
      fr[VEC ? 0 : q] = rp[row * p.ld + i];
      fk[VEC ? 0 : q] = kp[row * p.ld + i];
      fw[VEC ? 0 : q] = wp[row * p.ldw + i];
    }
#pragma unroll
    for (int q = 0; q < NU; ++q) {
      const int e = threadIdx.x + q * 256, tt = e / WC, i = min(c0 + (e & (WC - 1)), D - 1);
      fv[VEC ? 0 : q] = vp[(size_t)(t0 + min(base + tt, n - 1)) * p.ld + i];
    }
  };
  fetch(0);
  for (int base = 0; base < n; base += CH) {
    __syncthreads();
    if constexpr (VEC) {
#pragma unroll
      for (int h = 0; h < 8; h += 4) {
        *reinterpret_cast<f32x4*>(&rs[et][ei + h]) = f32x4{(float)r8[h], (float)r8[h + 1], (float)r8[h + 2], (float)r8[h + 3]};
        *reinterpret_cast<f32x4*>(&ks[et][ei + h]) = f32x4{(float)k8[h], (float)k8[h + 1], (float)k8[h + 2], (float)k8[h + 3]};
        *reinterpret_cast<f32x4*>(&ws[et][ei + h]) = f32x4{w8[h], w8[h + 1], w8[h + 2], w8[h + 3]};
        *reinterpret_cast<f32x4*>(&vs[vt][vi + h]) = f32x4{(float)v8[h], (float)v8[h + 1], (float)v8[h + 2], (float)v8[h + 3]};
      }
    } else {
#pragma unroll
      for (int q = 0; q < NV; ++q) {
        const int e = threadIdx.x + q * 256, tt = e / DP, i = e % DP;
        if (tt < CH) {
          rs[tt][i] = i < D ? (float)fr[VEC ? 0 : q] : 0.f;
          ks[tt][i] = i < D ? (float)fk[VEC ? 0 : q] : 0.f;
          ws[tt][i] = i < D ? fw[VEC ? 0 : q] : 0.f;
        }
      }
#pragma unroll
      for (int q = 0; q < NU; ++q) {
        const int e = threadIdx.x + q * 256;
        if (e < CH * WC) vs[e / WC][e & (WC - 1)] = c0 + (e & (WC - 1)) < D ? (float)fv[VEC ? 0 : q] : 0.f;
      }
    }
    __syncthreads();
    if (base + CH < n) fetch(base + CH);
    // sum_i r u k of every staged token: 16 lanes each
#pragma unroll
    for (int t8 = 0; t8 < CH; t8 += 16) {
      const int tt = t8 + (threadIdx.x >> 4), l = threadIdx.x & 15;
      float a = 0.f;
      if (tt < CH)
#pragma unroll
        for (int q = 0; q < DP / 16; ++q) a += rs[tt][l + 16 * q] * ur[q] * ks[tt][l + 16 * q];
      // (row rotations: the exchanges of a butterfly over 16 lanes without the LDS round trips)
      a = dpp_add<0x121>(dpp_add<0x122>(dpp_add<0x124>(dpp_add<0x128>(a))));
      if (tt < CH && l == 0) ruk[tt] = a;
    }
    __syncthreads();
    // 8 tokens at a time, the next PF tokens' operands on their way while one is summed (a token's arithmetic takes less than
    // an LDS read); lane part q keeps token q's output. Three tokens ahead, unless f32 values wait one by one in the registers
    // (VEC false): those then leave room for two waves on a SIMD instead of three (100 runs of 50 tokens, 16 heads of 32: 32.7 us
    // against 26.7 with one token ahead; 8 runs of 300, 10 heads of 60: 52.0 against 49.2)
    constexpr int PF = R <= 4 && (VEC || sizeof(T) == 2) ? 3 : 1, RB = PF + 1;
    const int m = min(CH, n - base);
    f32x4 r4[RB][R / 4], k4[RB][R / 4], w4[RB][R / 4];
    float v1[RB][CPL];
    auto get = [&](int tt, int b) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < R / 4; ++q) {
        r4[b][q] = *reinterpret_cast<const f32x4*>(&rs[tt][part * R + 4 * q]);
        k4[b][q] = *reinterpret_cast<const f32x4*>(&ks[tt][part * R + 4 * q]);
        w4[b][q] = *reinterpret_cast<const f32x4*>(&ws[tt][part * R + 4 * q]);
      }
#pragma unroll
      for (int c = 0; c < CPL; ++c) v1[b][c] = vs[tt][col + c];
    };
    auto token = [&](int b, float (&o)[CPL]) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        float o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int i4 = 0; i4 < R / 4; ++i4)
#pragma unroll
          for (int e = 0; e < 4; e += 2) {
            const int i = 4 * i4 + e;
            o0 = fmaf(r4[b][i4][e], S[c][i], o0);
            o1 = fmaf(r4[b][i4][e + 1], S[c][i + 1], o1);
            S[c][i] = fmaf(w4[b][i4][e], S[c][i], k4[b][i4][e] * v1[b][c]);
            S[c][i + 1] = fmaf(w4[b][i4][e + 1], S[c][i + 1], k4[b][i4][e + 1] * v1[b][c]);
          }
        o[c] = sum_parts<PARTS>(o0 + o1);
      }
    };
#pragma unroll
    for (int i = 0; i < PF; ++i) get(i, i);
    for (int t8 = 0; t8 < m; t8 += 8) {
      float mine[CPL], o[CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) mine[c] = 0.f;
      const int last = m - 1 - t8, tt = t8 + (part & 7);
      const float rk = ruk[tt];
      if (last >= 7) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          get(min(t8 + q + PF, CH - 1), (q + PF) % RB);
          token(q % RB, o);
#pragma unroll
          for (int c = 0; c < CPL; ++c) mine[c] = part == q ? o[c] : mine[c];
        }
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          get(min(t8 + q + PF, CH - 1), (q + PF) % RB);
          if (q > last) continue;              // (uniform)
          token(q % RB, o);
#pragma unroll
          for (int c = 0; c < CPL; ++c) mine[c] = part == q ? o[c] : mine[c];
        }
      }
      if (part < 8 && part <= last)
#pragma unroll
        for (int c = 0; c < CPL; ++c)
          if (j + c < D) p.o[(size_t)(t0 + base + tt) * p.ldo + hb + j + c] = fmaf(rk, vs[tt][col + c], mine[c]);
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const int row = part * R + i;
      if (row < D && j + c < D) st[(size_t)row * D + j + c] = S[c][i];
    }
  // the run's last row is the next step's previous token (this layer's shift_mix, which reads it, came before)
  const int G = gridDim.x;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < p.width; i += G * 256)
    p.prev[(size_t)slot * p.ldp + i] = p.x[(size_t)(t0 + n - 1) * p.ldx + i];
}

// Sums of eight values over 32 lanes each: every exchange adds two of them, one for each half of the lanes (19 instructions; 8 x 5 one by one). Lane
// 16 a + 4 x + b ends with the sum of value a + 2 b.
DEVI float sum8_32(const float (&o)[8], int lane) {
  float h[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto s = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, o[2 * i]), __builtin_bit_cast(uint32_t, o[2 * i + 1]), false, false);
    h[i] = __builtin_bit_cast(float, (uint32_t)s[0]) + __builtin_bit_cast(float, (uint32_t)s[1]);
  }
  auto pair = [&](float a, float b, bool hi, auto dpp) __attribute__((always_inline)) {
    const int send = __builtin_bit_cast(int, hi ? a : b);
    return (hi ? b : a) + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, send, decltype(dpp)::value, 0xf, 0xf, true));
  };
  const float x = pair(h[0], h[1], lane & 1, std::integral_constant<int, 0xB1>{}), y = pair(h[2], h[3], lane & 1, std::integral_constant<int, 0xB1>{});
  return dpp_add<0x124>(dpp_add<0x128>(pair(x, y, lane & 2, std::integral_constant<int, 0x4E>{})));
}

// The scan of few runs, up to two workgroups for each CU. A wave takes a token's time to issue and to close its sums (240 cycles of the form above,
// however many waves share the CU), so here a column's keys lie over 32 lanes, two columns to a wave, the sums of eight tokens are closed together,
// and the next chunk is staged in a second buffer while one is summed, with a barrier for each. 3500 tokens, 32 heads of 64: 348 -> 244 us, 64 heads
// 351 -> 327, 16 and 32 heads of 128 533 -> 339 and 535 -> 450; 100 tokens 15.2 -> 12.4, 15.9 -> 17.1, 21.1 -> 15.1 and 22.9 -> 21.5. At two workgroups to a CU runs of up
// to 100 tokens of heads of 64 lose up to 1.2 us; the rule does not ask for their length, since the bits of a prompt must not depend on how it is cut. With
// four workgroups to a CU it would be slower (4 x 900, 32 heads of 64: 121 above, 173).
template <typename T, int DP, bool VEC>
__global__ __launch_bounds__(256) void wkv_few_kernel(Scan p) {
  constexpr int WC = 8, CH = 2048 / DP, R = DP / 32, LR = DP + 4, RQ = R < 4 ? 2 : 4, PF = 3, RB = PF + 1;
  struct Chunk {
    float r[CH][LR], k[CH][LR], w[CH][LR], v[CH][WC], ruk[CH];
  };
  __shared__ __attribute__((aligned(16))) Chunk ch[2];
  typedef T tv8 __attribute__((ext_vector_type(8), aligned(16)));
  typedef float fv8 __attribute__((ext_vector_type(8), aligned(16)));
  typedef float fq __attribute__((ext_vector_type(RQ)));
  const int* run = p.runs + 4 * blockIdx.y;
  const int t0 = run[0], n = run[1], slot = run[2], pos0 = run[3];
  if (slot < 0 || n < 1) return;
  const int head = blockIdx.x / (DP / WC), c0 = blockIdx.x % (DP / WC) * WC;
  const int lane = threadIdx.x & 63, part = lane & 31, col = 2 * (threadIdx.x >> 6) + (lane >> 5), j = c0 + col;
  const size_t hb = (size_t)head * DP;
  const T *rp = (const T*)p.r + hb, *kp = (const T*)p.k + hb, *vp = (const T*)p.v + hb;
  const float* wp = p.w + hb;
  float* st = p.state + (size_t)slot * p.sstride + hb * DP;
  const int et = threadIdx.x / (DP / 8), ei = threadIdx.x % (DP / 8) * 8, vt = threadIdx.x % CH;         // a thread's token and keys, its token's values
  float S[R], u[8];
#pragma unroll
  for (int i = 0; i < R; ++i) S[i] = pos0 > 0 ? st[(size_t)(part * R + i) * DP + j] : 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) u[i] = p.u[hb + ei + i];
  // (arrived before the first chunk's loads go out, which the loop over tokens would wait for otherwise)
#pragma unroll
  for (int i = 0; i < R; ++i) asm volatile("" : "+v"(S[i]));
#pragma unroll
  for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(u[i]));
  tv8 r8, k8, v8;
  fv8 w8;
  auto fetch = [&](int base) __attribute__((always_inline)) {        // (rows past the run: its last one)
    const size_t row = t0 + min(base + et, n - 1), vrow = t0 + min(base + vt, n - 1);
    if constexpr (!VEC) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        r8[e] = rp[row * p.ld + ei + e];
        k8[e] = kp[row * p.ld + ei + e];
        w8[e] = wp[row * p.ldw + ei + e];
        v8[e] = vp[vrow * p.ld + c0 + e];
      }
      return;
    }
    r8 = *reinterpret_cast<const tv8*>(rp + row * p.ld + ei);
    k8 = *reinterpret_cast<const tv8*>(kp + row * p.ld + ei);
    w8 = *reinterpret_cast<const fv8*>(wp + row * p.ldw + ei);
    v8 = *reinterpret_cast<const tv8*>(vp + vrow * p.ld + c0);
  };
  auto stage = [&](Chunk& c) __attribute__((always_inline)) {
    float a = 0.f;
#pragma unroll
    for (int h = 0; h < 8; h += 4) {
      *reinterpret_cast<f32x4*>(&c.r[et][ei + h]) = f32x4{(float)r8[h], (float)r8[h + 1], (float)r8[h + 2], (float)r8[h + 3]};
      *reinterpret_cast<f32x4*>(&c.k[et][ei + h]) = f32x4{(float)k8[h], (float)k8[h + 1], (float)k8[h + 2], (float)k8[h + 3]};
      *reinterpret_cast<f32x4*>(&c.w[et][ei + h]) = f32x4{w8[h], w8[h + 1], w8[h + 2], w8[h + 3]};
      *reinterpret_cast<f32x4*>(&c.v[vt][h]) = f32x4{(float)v8[h], (float)v8[h + 1], (float)v8[h + 2], (float)v8[h + 3]};
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) a += (float)r8[e] * u[e] * (float)k8[e];
    a = sum_parts<DP == 64 ? 8 : 16>(a);
    if (DP == 256) a += __shfl_xor(a, 16, 64);
    if (ei == 0) c.ruk[et] = a;
  };
  fetch(0);
  stage(ch[0]);
  fetch(CH);
  __syncthreads();
  int b = 0;
  for (int base = 0; base < n; base += CH, b ^= 1) {
    stage(ch[b ^ 1]);
    fetch(base + 2 * CH);
    const Chunk& c = ch[b];
    const int m = min(CH, n - base);
    fq r4[RB][R / RQ], k4[RB][R / RQ], w4[RB][R / RQ];
    float v1[RB];
    auto get = [&](int tt, int s) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < R / RQ; ++q) {
        r4[s][q] = *reinterpret_cast<const fq*>(&c.r[tt][part * R + RQ * q]);
        k4[s][q] = *reinterpret_cast<const fq*>(&c.k[tt][part * R + RQ * q]);
        w4[s][q] = *reinterpret_cast<const fq*>(&c.w[tt][part * R + RQ * q]);
      }
      v1[s] = c.v[tt][col];
    };
    auto token = [&](int s) __attribute__((always_inline)) {
      float o0 = 0.f, o1 = 0.f;
#pragma unroll
      for (int q = 0; q < R / RQ; ++q)
#pragma unroll
        for (int e = 0; e < RQ; e += 2) {
          const int i = RQ * q + e;
          o0 = fmaf(r4[s][q][e], S[i], o0);
          o1 = fmaf(r4[s][q][e + 1], S[i + 1], o1);
          S[i] = fmaf(w4[s][q][e], S[i], k4[s][q][e] * v1[s]);
          S[i + 1] = fmaf(w4[s][q][e + 1], S[i + 1], k4[s][q][e + 1] * v1[s]);
        }
      return o0 + o1;
    };
#pragma unroll
    for (int i = 0; i < PF; ++i) get(i, i);
    for (int t8 = 0; t8 < m; t8 += 8) {
      float o[8];
      const int last = m - 1 - t8;
      if (last >= 7) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          get(min(t8 + q + PF, CH - 1), (q + PF) % RB);
          o[q] = token(q % RB);
        }
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          get(min(t8 + q + PF, CH - 1), (q + PF) % RB);
          o[q] = 0.f;
          if (q <= last) o[q] = token(q % RB);           // (uniform)
        }
      }
      const float sum = sum8_32(o, lane);
      const int q = (lane >> 4 & 1) | (lane & 3) << 1, tt = t8 + q;
      if (!(lane & 12) && q <= last) p.o[(size_t)(t0 + base + tt) * p.ldo + hb + j] = fmaf(c.ruk[tt], c.v[tt][col], sum);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < R; ++i) st[(size_t)(part * R + i) * DP + j] = S[i];
  for (int i = blockIdx.x * 256 + threadIdx.x; i < p.width; i += gridDim.x * 256)
    p.prev[(size_t)slot * p.ldp + i] = p.x[(size_t)(t0 + n - 1) * p.ldx + i];
}

template <typename T, int DP, int PARTS>
int scan_v(const Scan& p, int nruns, hipStream_t st) {
  const dim3 grid(p.H * ((p.V + 256 / PARTS - 1) / (256 / PARTS)), nruns);
  if constexpr (DP >= 64) {
    auto whole = [](const void* q, long ld, size_t size) { return (uintptr_t)q % 16 == 0 && ld * size % 16 == 0; };
    const bool vec = p.D == DP && whole(p.r, p.ld, sizeof(T)) && whole(p.k, p.ld, sizeof(T)) && whole(p.v, p.ld, sizeof(T)) && whole(p.w, p.ldw, 4);
    if (PARTS == 16 && p.D == DP && p.H * nruns * (DP / 8) <= 512) {
      const dim3 few(p.H * (DP / 8), nruns);
      if (vec) hipLaunchKernelGGL((wkv_few_kernel<T, DP, true>), few, dim3(256), 0, st, p);
      else hipLaunchKernelGGL((wkv_few_kernel<T, DP, false>), few, dim3(256), 0, st, p);
      return (int)hipGetLastError();
    }
    if (vec) {
      hipLaunchKernelGGL((wkv_scan_kernel<T, DP, PARTS, 1, true>), grid, dim3(256), 0, st, p);
      return (int)hipGetLastError();
    }
  }
  hipLaunchKernelGGL((wkv_scan_kernel<T, DP, PARTS, 1, false>), grid, dim3(256), 0, st, p);
  return (int)hipGetLastError();
}

template <typename T, int DP>
int scan_d(const Scan& p, int nruns, hipStream_t st) {
  if (DP < 64 || p.H * nruns * ((p.V + 31) / 32) >= 256) return scan_v<T, DP, 8>(p, nruns, st);
  return scan_v<T, DP, DP < 64 ? 8 : 16>(p, nruns, st);
}

template <typename T>
int scan_t(const Scan& p, int nruns, hipStream_t st) {
  if (p.D <= 32) return scan_d<T, 32>(p, nruns, st);
  if (p.D <= 64) return scan_d<T, 64>(p, nruns, st);
  if (p.D <= 128) return scan_d<T, 128>(p, nruns, st);
  if (p.D <= 256) return scan_d<T, 256>(p, nruns, st);
  return -1;
}

Scan args(const void* r, const void* k, const void* v, long ld, const float* w, long ldw, const float* u, float* o, long ldo,
          float* state, long sstride, const float* x, long ldx, float* prev, long ldp, int width, const int* runs, int H, int D) {
  return Scan{r, k, v, w, u, o, state, x, prev, runs, ld, ldw, ldo, sstride, ldx, ldp, H, D, D, width, 1.f, nullptr, nullptr, nullptr, 0,
              0.f};
}

}  // namespace nls_wkv

extern "C" {
using namespace nls_wkv;

int nls_shift_mix(const float* x, long ldx, const float* mu, const float* prev, long ldp, void* out, long ldo,
                  long mstride, const int* runs, const int* tok_seq, int D, int T, int f32, void* stream) {
  if (T < 1 || D < 1) return -1;
  Mix p{x, mu, prev, out, runs, tok_seq, ldx, ldp, ldo, mstride, D, f32};
  const dim3 grid(T, T >= 256 ? 1 : min((D + 255) / 256, 16));
  if (f32) hipLaunchKernelGGL(shift_mix_kernel<float>, grid, dim3(256), 0, (hipStream_t)stream, p);
  else hipLaunchKernelGGL(shift_mix_kernel<__bf16>, grid, dim3(256), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

int nls_wkv_scan(const void* r, const void* k, const void* v, long ld, const float* w, long ldw, const float* u,
                 float* o, long ldo, float* state, long sstride, const float* x, long ldx, float* prev, long ldp,
                 int width, const int* runs, int nruns, int H, int D, int f32, void* stream) {
  if (nruns < 1 || H < 1 || D < 1) return -1;
  const Scan p = args(r, k, v, ld, w, ldw, u, o, ldo, state, sstride, x, ldx, prev, ldp, width, runs, H, D);
  return f32 ? scan_t<float>(p, nruns, (hipStream_t)stream) : scan_t<__bf16>(p, nruns, (hipStream_t)stream);
}

// every run has one token (or none); D a multiple of 4
int nls_wkv_step(const void* r, const void* k, const void* v, long ld, const float* w, long ldw, const float* u,
                 float* state, long sstride, const float* x, long ldx, float* prev, long ldp, int width, const int* runs,
                 int nruns, const float* norm, const void* gate, long ldg, void* out, long ldout, int H, int D, float eps,
                 int f32, void* stream) {
  const Scan p = args(r, k, v, ld, w, ldw, u, nullptr, 0, state, sstride, x, ldx, prev, ldp, width, runs, H, D);
  return f32 ? step_rows<float, WKV>(p, nruns, norm, gate, ldg, out, ldout, eps, (hipStream_t)stream)
             : step_rows<__bf16, WKV>(p, nruns, norm, gate, ldg, out, ldout, eps, (hipStream_t)stream);
}

// per-head norm of D columns, norm weight and gate of a recurrence's output rows
int nls_scan_out(const float* o, long ldo, const float* norm, const void* gate, long ldg, void* out, long ld, int H,
                 int D, int T, float eps, int f32, void* stream) {
  return f32 ? out_rows<float>(o, ldo, norm, gate, ldg, out, ld, H, D, T, eps, (hipStream_t)stream)
             : out_rows<__bf16>(o, ldo, norm, gate, ldg, out, ld, H, D, T, eps, (hipStream_t)stream);
}

}  // extern "C"
