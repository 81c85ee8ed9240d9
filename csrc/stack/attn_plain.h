// Causal attention over paged rows for any head widths in f32 arithmetic throughout (f32 MFMA): 32-bit models, and head widths that
// the bf16 MFMA kernels do not take.
//
// Workgroup = 16 rows of one key head, its waves split the keys 16 at a time and meet in LDS. The rows are the query heads of one
// token (up to 16 of them), or, where several tokens of a launch belong to one sequence, of 16 / heads tokens, so that a prompt's
// keys are read once for them; a group whose tokens belong to several sequences walks each one's keys.
// Per 16 keys and wave, with v_mfma_f32_16x16x4_f32:
//   S^T = K Q^T: lane 16 g + r loads 16 bytes of key r at column 16 s + 4 g, the operands of four MFMAs, and meets the same columns of
//   row r, which wait in LDS; it ends with the scores of keys 4 g .. 4 g + 3 and row r, so that maximum and rescale are two lane
//   exchanges and lane-local;
//   O^T += V^T P^T: those registers are the second operand as they stand; 16 bytes of value row 4 g + j at column 64 q + 4 r are
//   the first operand of the four tiles of columns 64 q + 4 m + e.
// Loads run one chunk of key columns and two of value columns ahead; nothing goes through LDS but the queries and the merge.
// A row also meets keys that it does not see (other sequences' and later tokens' of its group, those ahead of its window, the last one
// repeated), with a weight of 0, which an infinity or NaN among their values turns into NaN: rows whose result is not finite are summed
// once more over their own keys alone.
// What bounds it: the matrix pipe on prompts (32 cycles per MFMA, rows past a run's last token included), the walk over a row's keys on
// small grids. Three prompts of 300 tokens, 16 heads of 128 over 4: 823 us (one workgroup per row and head, a serial walk) -> 43 us;
// four decoded tokens behind 300 keys: 136 -> 16 us.
#pragma once
#include <type_traits>
#include "../kernels/common.h"

namespace nls_plain {

constexpr int MAXV = 1024, MAXK = 2048;     // value and key columns
constexpr int VB = 512;                     // value columns of a workgroup (its accumulators; wider values score twice)

struct PA {
  const void *q, *k, *v;
  void* out;
  const int* bt;              // block tables
  const int* tok_seq;
  const int* ctx_len;         // keys of each token (0: padded row)
  const float* gate;          // [T][ldg], a factor per token and head (null: none)
  long ldq, qhs;              // row and head strides of the queries
  long ldkv, khs;             // row and key-head strides of the cache
  long ldo, ohs;
  long ldg;
  int bts, bs, gs;            // gs: query heads per key head
  int Dk, Dv;                 // columns (Dk a multiple of 4)
  float scale;
  int window, keep, sink;     // window > 0: the newest `window` keys and the first `keep`; sink: one more in the denominator
  int T, tb, sub;             // tokens; tokens of a workgroup; workgroups that share a key head's query heads
};

template <typename T> DEVI f32x4 ld4(const T* p) {
  typedef T t4 __attribute__((ext_vector_type(4)));
  const t4 a = *reinterpret_cast<const t4*>(p);
  return f32x4{(float)a[0], (float)a[1], (float)a[2], (float)a[3]};
}

// Row `row` of a workgroup, its token t and query head h, over the keys that it sees. mls: the waves' maxima and sums, w: 64 NW floats.
template <typename T, int NW>
DEVI void redo_row(const PA& p, int t, int h, int row, int bz, const float* mls, float* w) {
  constexpr int NT = 64 * NW, C = VB / NT;
  const int ctx = p.ctx_len[t], low = p.window > 0 ? ctx - p.window : 0, v0 = bz * VB, dv = min(p.Dv - v0, VB);
  const int* bt = p.bt + (size_t)p.tok_seq[t] * p.bts;
  const T* q = reinterpret_cast<const T*>(p.q) + (size_t)t * p.ldq + (size_t)h * p.qhs;
  const T* kc = reinterpret_cast<const T*>(p.k) + (size_t)(h / p.gs) * p.khs;
  const T* vc = reinterpret_cast<const T*>(p.v) + (size_t)(h / p.gs) * p.khs + v0;
  auto slot = [&](int k) { return ((size_t)bt[k / p.bs] * p.bs + k % p.bs) * p.ldkv; };
  float m = -INFINITY, l = 0.f, acc[C];
  for (int i = 0; i < NW; ++i) m = fmaxf(m, mls[i * 32 + row]);
  for (int i = 0; i < NW; ++i)
    if (mls[i * 32 + row] != -INFINITY) l += mls[i * 32 + 16 + row] * expf(mls[i * 32 + row] - m);
  for (int i = 0; i < C; ++i) acc[i] = 0.f;
  for (int k0 = 0; k0 < ctx; k0 += NT) {
    const int n = min(NT, ctx - k0);
    const T* k = kc + slot(k0 + min((int)threadIdx.x, n - 1));
    float s = 0.f;
    for (int d = 0; d < p.Dk; d += 4) {
      const f32x4 x = ld4(k + d);
      for (int e = 0; e < 4; ++e) s = fmaf((float)q[d + e], x[e], s);
    }
    __syncthreads();                               // (the last keys' weights have been read)
    w[threadIdx.x] = expf(s * p.scale - m);
    __syncthreads();
    for (int i = 0; i < n; ++i) {
      if (k0 + i < low && k0 + i >= p.keep) continue;
      const T* v = vc + slot(k0 + i);
      for (int j = 0; j < C; ++j)
        if ((int)threadIdx.x + NT * j < dv) acc[j] = fmaf(w[i], (float)v[threadIdx.x + NT * j], acc[j]);
    }
  }
  const float f = (l > 0.f ? 1.f / l : 0.f) * (p.gate ? p.gate[(size_t)t * p.ldg + h] : 1.f);
  T* y = reinterpret_cast<T*>(p.out) + (size_t)t * p.ldo + (size_t)h * p.ohs + v0;
  for (int j = 0; j < C; ++j)
    if ((int)threadIdx.x + NT * j < dv) y[threadIdx.x + NT * j] = (T)(acc[j] * f);
}

// NQ: 64-column blocks of the values; NW: waves. Beside: other work of the launch, asked first, which answers whether the workgroup is its own or
// sets the place (bx, by, bz of gx) that it takes here. (A body called from two kernels compiled to other copies of the keys' registers in
// this one: 8 to 25 % slower at 128 columns in 32 bits.)
struct Alone {};
template <typename T, int NQ, int NW, class Beside>
__global__ __launch_bounds__(64 * NW) void attn_plain_kernel(PA p, Beside beside) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z, gx = gridDim.x;
  if constexpr (!std::is_same<Beside, Alone>::value)
    if (beside(sm, bx, by, bz, gx)) return;
  constexpr int KC = NQ > 2 ? 4 : 8;               // 16-column steps of a key chunk
  constexpr int ML = NW * 32 + 16;                 // floats of the waves' maxima and sums, rows that are not finite
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nks = (p.Dk + 15) >> 4, nc = (nks + KC - 1) / KC, ldl = nc * KC * 16 + 4;
  float *mls = sm, *ob = sm + ML, *qs = ob;        // (the merge takes the queries' place)
  int* bad = reinterpret_cast<int*>(sm + NW * 32);
  const int kh = (uint32_t)by / p.sub, h0 = ((uint32_t)by % p.sub) * 16;          // key head, first of its query heads
  const int gr = min(p.gs - h0, 16);                                          // query heads of this workgroup
  const int t0 = (gx - 1 - bx) * p.tb, tn = min(p.tb, p.T - t0);      // (later tokens see more keys)
  const int nrow = tn * gr;
  const int v0 = bz * VB, dv = min(p.Dv - v0, VB);                            // this workgroup's value columns
  const T* kc = reinterpret_cast<const T*>(p.k) + (size_t)kh * p.khs;
  const T* vc = reinterpret_cast<const T*>(p.v) + (size_t)kh * p.khs + v0;
  auto head = [&](int row) { return (size_t)kh * p.gs + h0 + row % gr; };
  for (int i = threadIdx.x; i < 4 * ldl; i += 64 * NW) {
    const int row = i / (ldl / 4), c = (i - row * (ldl / 4)) * 4;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (row < nrow && c < p.Dk) {
      const T* x = reinterpret_cast<const T*>(p.q) + (size_t)(t0 + row / gr) * p.ldq + head(row) * p.qhs + c;
      v = f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
    }
    *reinterpret_cast<f32x4*>(qs + row * ldl + c) = v;
  }
  __syncthreads();

  f32x4 o[NQ][4];
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[q][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = p.sink && wave == 0 ? 0.f : -INFINITY, l = p.sink && wave == 0 && g == 0 ? 1.f : 0.f;      // (l: four lanes' shares)
  for (int a = 0; a < tn;) {
    // tokens a .. b - 1 of the group belong to one sequence
    const int seq = p.tok_seq[t0 + a];
    int b = a, ctx = 0, low = 1 << 30;
    for (; b < tn && p.tok_seq[t0 + b] == seq; ++b) {
      const int c = p.ctx_len[t0 + b];
      ctx = max(ctx, c);
      if (c > 0) low = min(low, p.window > 0 ? max(c - p.window, 0) : 0);
    }
    const int tok = r / gr;
    const int rctx = r < nrow && tok >= a && tok < b ? p.ctx_len[t0 + tok] : 0, rlow = p.window > 0 ? rctx - p.window : 0;
    a = b;
    if (ctx <= 0) continue;
    const int* bt = p.bt + (size_t)seq * p.bts;
    // tiles that no row sees are left out: `skip` of them behind the kept keys' `nkt`
    const int lowt = low >> 4, nkt = min((p.keep + 15) >> 4, lowt), skip = lowt - nkt, ntile = ((ctx + 15) >> 4) - skip;
    auto key0 = [&](int t) { return (t < nkt ? t : t + skip) * 16; };
    auto slot = [&](int t) { return [&](int k) { return bt[k / p.bs] * p.bs + k % p.bs; }(min(key0(t) + r, ctx - 1)); };
    auto load_k = [&](f32x4 (&f)[KC], int s, int c) __attribute__((always_inline)) {
      const T* row = kc + (size_t)s * p.ldkv;
      const int c0 = c * (KC * 16) + 4 * g;
      if ((c + 1) * (KC * 16) <= p.Dk) {
#pragma unroll
        for (int i = 0; i < KC; ++i) f[i] = ld4(row + c0 + 16 * i);
      } else {
#pragma unroll
        for (int i = 0; i < KC; ++i) {             // (zeros past the last column: what is loaded there may not be finite)
          f[i] = ld4(row + min(c0 + 16 * i, p.Dk - 4));
          if (c0 + 16 * i >= p.Dk) f[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    };
    auto load_v = [&](f32x4 (&f)[4], const int (&s)[4], int q) __attribute__((always_inline)) {
      const int c0 = 64 * q + 4 * r;               // (columns past the last one are computed and not stored)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const T* row = vc + (size_t)s[j] * p.ldkv;
        if (!(dv & 3)) f[j] = ld4(row + min(c0, dv - 4));
        else
#pragma unroll
          for (int e = 0; e < 4; ++e) f[j][e] = (float)row[min(c0 + e, dv - 1)];
      }
    };
    if (wave >= ntile) continue;
    int sk = slot(wave);
    f32x4 kf[KC], kn[KC], vf[2][4];
    load_k(kf, sk, 0);
    for (int t = wave; t < ntile; t += NW) {
      const int sn = slot(min(t + NW, ntile - 1));
      int sv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) sv[j] = __shfl(sk, 4 * g + j, 64);
      load_v(vf[0], sv, 0);
      if (NQ > 1) load_v(vf[1], sv, 1);
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < nc; ++c) {
        if (c + 1 < nc) load_k(kn, sk, c + 1);
        else load_k(kn, sn, 0);
        const float* qr = qs + r * ldl + c * (KC * 16) + 4 * g;
#pragma unroll
        for (int i = 0; i < KC; ++i) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(qr + 16 * i);
#pragma unroll
          for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][j], x[j], s, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < KC; ++i) kf[i] = kn[i];
      }
      const int k0 = key0(t) + 4 * g;
      float mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = k0 + j;
        s[j] = k < rctx && (k >= rlow || k < p.keep) ? s[j] * p.scale : -INFINITY;
        mx = fmaxf(mx, s[j]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m, mx), base = mn == -INFINITY ? 0.f : mn;
      if (!__all(mn == m)) {
        const float alpha = m == -INFINITY ? 0.f : expf(m - base);
        l *= alpha;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[q][e] *= alpha;
        m = mn;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[j] = expf(s[j] - base);
        l += s[j];
      }
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[q][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[q & 1][j][e], s[j], o[q][e], 0, 0, 0);
        if (q + 2 < NQ) load_v(vf[q & 1], sv, q + 2);
      }
      sk = sn;
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (g == 0) {
    mls[wave * 32 + r] = m;
    mls[wave * 32 + 16 + r] = l;
  }
  __syncthreads();                                 // (the queries have been read, too)
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < NW; ++w) M = fmaxf(M, mls[w * 32 + r]);
  if (threadIdx.x < 16) bad[threadIdx.x] = 0;
  const float f = m == -INFINITY ? 0.f : expf(m - M);
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (64 * q >= dv) break;
    if (q) __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i)                    // columns 64 q + 16 g + 4 i .. of row r
      *reinterpret_cast<f32x4*>(ob + (wave * 16 + r) * 68 + 16 * g + 4 * i) =
          f32x4{o[q][0][i] * f, o[q][1][i] * f, o[q][2][i] * f, o[q][3][i] * f};
    __syncthreads();
    for (int i = threadIdx.x; i < nrow * 16; i += 64 * NW) {
      const int row = i >> 4, c = (i & 15) * 4;
      if (64 * q + c >= dv) continue;
      float mm = -INFINITY, ll = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) mm = fmaxf(mm, mls[w * 32 + row]);
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float mw = mls[w * 32 + row];
        if (mw != -INFINITY) ll += mls[w * 32 + 16 + row] * expf(mw - mm);
        v += *reinterpret_cast<const f32x4*>(ob + (w * 16 + row) * 68 + c);
      }
      const size_t tk = t0 + row / gr;
      v *= (ll > 0.f ? 1.f / ll : 0.f) * (p.gate ? p.gate[tk * p.ldg + head(row)] : 1.f);
      T* y = reinterpret_cast<T*>(p.out) + tk * p.ldo + head(row) * p.ohs + v0 + 64 * q + c;
      bool fin = true;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (64 * q + c + e < dv) {
          y[e] = (T)v[e];
          fin = fin && fabsf(v[e]) < INFINITY;
        }
      if (!fin) bad[row] = 1;
    }
  }
  __syncthreads();
  for (uint64_t again = __ballot(lane < nrow && bad[lane & 15]); again; again &= again - 1) {
    const int row = __builtin_ctzll(again);
    const PA* args = (const PA*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));                 // (read anew: kept from the start, they would not fit beside the loop's scalars)
    redo_row<T, NW>(*args, t0 + row / gr, kh * args->gs + h0 + row % gr, row, bz, mls, ob);
  }
}

inline size_t plain_lds(int Dk, int NQ, int NW) {
  const int KC = NQ > 2 ? 4 : 8, nc = ((Dk + 15) / 16 + KC - 1) / KC;
  return sizeof(float) * (NW * 32 + 16 + max(16 * (nc * KC * 16 + 4), NW * 16 * 68));
}

template <typename T, int NQ, int NW>
int launch_w(const PA& p, dim3 grid, hipStream_t st) {
  const size_t lds = plain_lds(p.Dk, NQ, NW);
  if (lds > 64 * 1024) {
    static bool attr = false;
    if (!attr && hipFuncSetAttribute((const void*)attn_plain_kernel<T, NQ, NW, Alone>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     160 * 1024) != hipSuccess)
      return -1;
    attr = true;
  }
  hipLaunchKernelGGL((attn_plain_kernel<T, NQ, NW, Alone>), grid, dim3(64 * NW), lds, st, p, Alone{});
  return (int)hipGetLastError();
}

// four waves once they fill the chip, eight (which halve the walk over a row's keys) on smaller grids
inline bool small(dim3 grid) { return (long)grid.x * grid.y <= 512; }

template <typename T, int NQ>
int launch_q(const PA& p, dim3 grid, hipStream_t st) {
  if (NQ <= 4 && small(grid)) return launch_w<T, NQ, NQ <= 4 ? 8 : 4>(p, grid, st);
  return launch_w<T, NQ, 4>(p, grid, st);
}

// the launch's tokens per workgroup and grid; false: refused
inline bool prepare(PA& p, int T_, int H, dim3& grid) {
  if (T_ < 1 || H < 1 || H > 65535 || p.gs < 1 || H % p.gs || p.Dk < 4 || p.Dk > MAXK || (p.Dk & 3) || p.Dv < 1 || (p.ldkv & 3) ||
      (p.khs & 3) || p.Dv > MAXV || p.bs < 1)
    return false;
  p.T = T_;
  p.sub = (p.gs + 15) / 16;
  // Up to 64 tokens each has a workgroup of its own. With more, a workgroup takes as many as leave one workgroup for each CU: a prompt's
  // tokens share their keys, those of several sequences are walked one after another. (Decoded tokens behind 300 keys, 16 heads of 128
  // over 4: 100 of them 47 us in groups of 4, 30 in groups of 2; 200, in groups of 4 either way, 52, and 74 in a workgroup each. 16
  // heads of 64 over 16: 65 tokens 167 us in groups of 16, 57 in groups of 5. One workgroup per row and head: 241, 403, 193 us.)
  const int heads = H / p.gs * p.sub;
  p.tb = T_ <= 64 ? 1 : min(max(1, 16 / p.gs), (int)(((long)T_ * heads + 255) / 256));
  grid = dim3((T_ + p.tb - 1) / p.tb, heads, (p.Dv + VB - 1) / VB);
  return true;
}

template <typename T>
int launch(PA p, int T_, int H, hipStream_t st) {
  dim3 grid;
  if (!prepare(p, T_, H, grid)) return -1;
  switch ((p.Dv + 63) / 64) {
    case 1: return launch_q<T, 1>(p, grid, st);
    case 2: return launch_q<T, 2>(p, grid, st);
    case 3: case 4: return launch_q<T, 4>(p, grid, st);
    default: return launch_q<T, 8>(p, grid, st);
  }
}

}  // namespace nls_plain
