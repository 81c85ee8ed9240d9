// Attention whose heads' softmax weights are mixed, over paged rows, for any head count and widths, f32 arithmetic throughout on f32 MFMA
// (32-bit models, shapes that the bf16 MFMA kernels do not take). See talk_attn.hip.
//
// Two launches, as the bf16 kernels' row-by-row form:
//   scores  a workgroup takes 16 rows (the query heads of a key head, of one token or of several beside each other) and a share of the
//           keys, its waves 16 keys at a time: S^T = K Q^T, so that a lane ends with four keys of one row. Scaled scores go to memory
//           [token][head][key], with each share's maximum and sum.
//   mix     a workgroup takes a few tokens, all heads of them, a share of the keys and some of the value columns. A block of 16 to 64 keys:
//           W^T = P^T talk^T for each token and 16 keys (P = exp(s - M) / L as it is loaded), through LDS, then O^T += V^T W^T, one
//           wave to 64 columns of a key head's rows. Normalised weights: shares of the keys add up, in the last workgroup to arrive.
// A tile's rows also meet keys that they do not see (later tokens' of the tile, those ahead of the window, the last one repeated) with a
// weight of 0, which an infinity or NaN among their values turns into NaN: tokens with a result that is not finite are summed once
// more over their own keys alone.
// What bounds it: decoded tokens the chain of a share (block table, keys, scores; then scores, mix, values), prompts the matrix pipe and the
// walk of a workgroup's keys (half of the time is the values' MFMAs). Before, one workgroup walked a token's keys on the vector units, twice: 16 heads
// of 128 over 4, 1203 keys in a window of 1024: one token 3290 us -> 31 for both launches, 1203 tokens of a prompt 6576 -> 199.
// Relative error against 64 bits, before and now, 16 heads of 128 over 4: one token and 53 keys 3.0e-7 -> 2.8e-7, 1203 keys 10.2e-7 -> 4.2e-7, 1203 tokens
// of a prompt 4.6e-7 -> 4.1e-7; 18 heads of 32 8.1e-7 -> 2.8e-7 at 1203 keys.
#pragma once
#include "../kernels/common.h"

namespace nls_talk {

struct TalkArgs {
  const void *q, *k, *v;      // q [T][ldq], heads Dp apart; k, v: paged [slots][G][Dp]
  void* out;                  // [T][ldo], heads Dp apart
  const void* gate;           // [T][ldg] of the activation type, a factor per column, heads V apart (null: none)
  const void* talk;           // plain: f32 [H][H]; MFMA kernels: bf16 [32 kk][32 kk], kk = ceil(H / 32), zero past H
  const int *bt, *tok_seq, *ctx_len;
  long ldq, ldo, ldg;
  int bts, bs, H, G, Dp, V;   // V: columns of a value head
  float scale;
  int window;                 // > 0: a token at position i sees j <= i if i - j < window
};

namespace plain {

constexpr int NW = 4, NT = 64 * NW;          // waves of the scores' workgroups
constexpr int KC = 8;         // 16-column steps of a key chunk
constexpr int KT = 64;        // keys of a block of the mix, at most

struct Rows {
  TalkArgs a;
  float *sc, *st, *part;      // scores [n][H][ks], share statistics [n][ns1][H][2], partial outputs [n][H][ns][Dp]
  int* cnt;                   // [n][workgroups of a token] zeros (left zero)
  long ks;                    // keys of a row, from 16 * (first visible / 16) on; a multiple of 16
  int t0, n;                  // tokens
  int sub;                    // workgroups that share a key head's query heads, 16 each
  int tb1, ns1;               // scores: tokens of a workgroup, shares of the keys
  int tb, ns, kt;             // mix: tokens of a workgroup, shares (one token), keys of a block
};

template <typename T> DEVI f32x4 ld4(const T* p) {
  typedef T t4 __attribute__((ext_vector_type(4)));
  const t4 a = *reinterpret_cast<const t4*>(p);
  return f32x4{(float)a[0], (float)a[1], (float)a[2], (float)a[3]};
}
DEVI f32x4 mma(float a, float b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// 16 states more behind the matrix pipe's last result, past the branch that ends its loop: a precaution, the compiler counts its wait across branches
DEVI void settle(f32x4& c) { asm volatile("s_nop 15" : "+v"(c)); }
DEVI int low_of(const TalkArgs& a, int ctx) { return a.window > 0 ? max(0, ctx - a.window) : 0; }

// tokens x .. y - 1 of a tile belong to one sequence: the keys that any of them sees
struct Run {
  int y, ctx, low;
  DEVI Run(const TalkArgs& a, int t0, int x, int tn) : y(x), ctx(0), low(1 << 30) {
    const int seq = a.tok_seq[t0 + x];
    for (; y < tn && a.tok_seq[t0 + y] == seq; ++y) {
      const int c = a.ctx_len[t0 + y];
      if (c <= 0) continue;
      ctx = max(ctx, c);
      low = min(low, low_of(a, c));
    }
  }
};

template <typename T>
__global__ __launch_bounds__(NT) void talk_rows_score_kernel(Rows p) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const TalkArgs& a = p.a;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, H = a.H, Dp = a.Dp, gs = H / a.G;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nks = (Dp + 15) >> 4, nc = (nks + KC - 1) / KC, ldl = nc * KC * 16 + 4;
  float *mls = sm, *qs = sm + NW * 32;
  const int kh = (int)blockIdx.y / p.sub, h0 = kh * gs + ((int)blockIdx.y % p.sub) * 16, gr = min(kh * gs + gs - h0, 16);
  const int tr0 = (int)(gridDim.x - 1 - blockIdx.x) * p.tb1, tn = min(p.tb1, p.n - tr0), t0 = p.t0 + tr0, nrow = tn * gr;
  const T* kc = (const T*)a.k + (size_t)kh * Dp;
  const size_t ldkv = (size_t)a.G * Dp;
  for (int i = threadIdx.x; i < 4 * ldl; i += NT) {
    const int row = i / (ldl / 4), c = (i - row * (ldl / 4)) * 4;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (row < nrow && c < Dp) {
      const T* x = (const T*)a.q + (size_t)(t0 + row / gr) * a.ldq + (size_t)(h0 + row % gr) * Dp + c;
      v = f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
    }
    *reinterpret_cast<f32x4*>(qs + row * ldl + c) = v;
  }
  __syncthreads();
  float m = -INFINITY, l = 0.f;
  const int tok = r / gr;
  for (int x = 0; x < tn;) {
    const Run run(a, t0, x, tn);
    const bool mine = r < nrow && tok >= x && tok < run.y;
    const int rctx = mine ? max(a.ctx_len[t0 + tok], 0) : 0, rlow = low_of(a, rctx), first = rlow & ~15;
    const int* bt = a.bt + (size_t)a.tok_seq[t0 + x] * a.bts;
    x = run.y;
    if (run.ctx <= 0) continue;
    const int tile0 = run.low >> 4, nt = ((run.ctx + 15) >> 4) - tile0, per = (nt + p.ns1 - 1) / p.ns1;
    const int ta = tile0 + min((int)blockIdx.z * per, nt), te = min(ta + per, tile0 + nt);
    float* dst = p.sc + ((size_t)(tr0 + tok) * H + h0 + r % gr) * p.ks;
    auto row_of = [&](int t) {
      const int k = min(16 * t + r, run.ctx - 1);
      return kc + ((size_t)bt[k / a.bs] * a.bs + k % a.bs) * ldkv;
    };
    auto load_k = [&](f32x4 (&f)[KC], const T* row, int c) __attribute__((always_inline)) {
      const int c0 = c * (KC * 16) + 4 * g;
#pragma unroll
      for (int i = 0; i < KC; ++i) {               // (zeros past the last column: what is loaded there may not be finite)
        f[i] = ld4(row + min(c0 + 16 * i, Dp - 4));
        if (c0 + 16 * i >= Dp) f[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    };
    if (ta + wave >= te) continue;
    f32x4 kf[KC], kn[KC];
    const T* row = row_of(ta + wave);
    load_k(kf, row, 0);
    for (int t = ta + wave; t < te; t += NW) {
      const T* next = row_of(min(t + NW, te - 1));
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < nc; ++c) {
        if (c + 1 < nc) load_k(kn, row, c + 1);
        else load_k(kn, next, 0);
        const float* qr = qs + r * ldl + c * (KC * 16) + 4 * g;
#pragma unroll
        for (int i = 0; i < KC; ++i) {
          const f32x4 q = *reinterpret_cast<const f32x4*>(qr + 16 * i);
#pragma unroll
          for (int j = 0; j < 4; ++j) s = mma(kf[i][j], q[j], s);
        }
#pragma unroll
        for (int i = 0; i < KC; ++i) kf[i] = kn[i];
      }
      settle(s);
      row = next;
      float mx = m;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 16 * t + 4 * g + j;
        s[j] = k >= rlow && k < rctx ? s[j] * a.scale : -INFINITY;
        mx = fmaxf(mx, s[j]);
      }
      if (16 * t >= first && 16 * t < rctx && 16 * t - first < p.ks) *reinterpret_cast<f32x4*>(dst + 16 * t - first + 4 * g) = s;
      const float base = mx == -INFINITY ? 0.f : mx;
      l *= m == -INFINITY ? 0.f : expf(m - base);
#pragma unroll
      for (int j = 0; j < 4; ++j) l += expf(s[j] - base);
      m = mx;
    }
  }
  // (the four lanes of a row have maxima of their own)
  float M = fmaxf(m, __shfl_xor(m, 16, 64));
  M = fmaxf(M, __shfl_xor(M, 32, 64));
  l *= m == -INFINITY ? 0.f : expf(m - M);
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (g == 0) {
    mls[wave * 32 + r] = M;
    mls[wave * 32 + 16 + r] = l;
  }
  __syncthreads();
  if ((int)threadIdx.x < nrow) {
    float mm = -INFINITY, ll = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) mm = fmaxf(mm, mls[w * 32 + threadIdx.x]);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = mls[w * 32 + threadIdx.x], lw = mls[w * 32 + 16 + threadIdx.x];
      ll += mw == -INFINITY ? lw : lw * expf(mw - mm);
    }
    const int tk = threadIdx.x / gr, h = h0 + threadIdx.x % gr;
    *reinterpret_cast<float2*>(p.st + (((size_t)(tr0 + tk) * p.ns1 + blockIdx.z) * H + h) * 2) = float2{mm, ll};
  }
}

// NW: waves, each with 64 value columns of a key head's rows; HB: head blocks of 16 that share a pass over a token's weights
template <typename T, int NW, int HB>
__global__ __launch_bounds__(64 * NW) void talk_rows_mix_kernel(Rows p) {
  constexpr int NT = 64 * NW;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const TalkArgs& a = p.a;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, H = a.H, Dp = a.Dp, gs = H / a.G;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nvb = (a.V + 63) >> 6, job = (int)blockIdx.y * NW + wave;
  const int tr0 = (int)(gridDim.x - 1 - blockIdx.x) * p.tb, tn = min(p.tb, p.n - tr0), t0 = p.t0 + tr0;
  const int kt = p.kt, ldw = kt + 4, hp = (H + 15) & ~15, nhb = hp >> 4;
  const bool own = H <= 64;                                              // the matrix in LDS
  float *ws = sm, *ml = ws + (size_t)p.tb * H * ldw, *tl = ml + 2 * (size_t)p.tb * H;
  int* slot = (int*)(tl + (own ? hp * hp : 0));                          // [2][KT]: this block's and the next one's
  int* bad = slot + 2 * KT;                                              // [tb], then the last share's flag
  const float* talk = (const float*)a.talk;
  const size_t ldkv = (size_t)a.G * Dp;
  // this wave's rows and value columns (a wave without any: those of the last, not stored)
  const bool on = job < a.G * p.sub * nvb;
  const int rb = min(job, a.G * p.sub * nvb - 1) / nvb, vb = min(job, a.G * p.sub * nvb - 1) - rb * nvb, kh = rb / p.sub;
  const int h0 = kh * gs + (rb - kh * p.sub) * 16, gr = min(kh * gs + gs - h0, 16), rtok = r / gr;
  const bool row = rtok < tn;
  const float* wrow = ws + ((size_t)(row ? rtok : 0) * H + h0 + r % gr) * ldw + 4 * g;
  const T* vc = (const T*)a.v + (size_t)kh * Dp + min(64 * vb + 4 * r, Dp - 4);
  for (int i = threadIdx.x >> 4; i < tn * H; i += NT / 16) {             // each head's maximum and 1 / sum over the shares, by 16 lanes
    const int tk = i / H, h = i - tk * H;
    const float* s = p.st + ((size_t)(tr0 + tk) * p.ns1 * H + h) * 2;
    float M = -INFINITY, L = 0.f;
    if (a.ctx_len[t0 + tk] > 0)
      for (int z = r; z < p.ns1; z += 16) {
        const float2 x = *reinterpret_cast<const float2*>(s + (size_t)z * H * 2);
        const float mn = fmaxf(M, x.x);
        L = (M == -INFINITY ? L : L * expf(M - mn)) + (x.x == -INFINITY ? x.y : x.y * expf(x.x - mn));
        M = mn;
      }
#pragma unroll
    for (int d = 1; d < 16; d *= 2) {
      const float mo = __shfl_xor(M, d, 64), lo = __shfl_xor(L, d, 64), mn = fmaxf(M, mo);
      L = (M == -INFINITY ? L : L * expf(M - mn)) + (mo == -INFINITY ? lo : lo * expf(mo - mn));
      M = mn;
    }
    if (r == 0) {
      ml[2 * i] = M;
      ml[2 * i + 1] = 1.f / L;
    }
  }
  if (own)
    for (int i = threadIdx.x; i < hp * hp; i += NT) {                    // transposed, zero past H
      const int s = i / hp, h = i - s * hp;
      tl[i] = s < H && h < H ? talk[(size_t)h * H + s] : 0.f;
    }
  if ((int)threadIdx.x < tn) bad[threadIdx.x] = 0;
  f32x4 o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
  int na = 1;                                                            // shares with keys
  bool any = false;
  for (int x = 0; x < tn;) {
    const Run run(a, t0, x, tn);
    const int xa = x;
    x = run.y;
    if (run.ctx <= 0) continue;
    const int* bt = a.bt + (size_t)a.tok_seq[t0 + xa] * a.bts;
    const int first = run.low & ~15, nb = (run.ctx - first + kt - 1) / kt, per = (nb + p.ns - 1) / p.ns;
    const int ba = min((int)blockIdx.z * per, nb), be = min(ba + per, nb);
    if (p.ns > 1) na = (nb + per - 1) / per;
    any = any || ba < be;
    auto put_slots = [&](int b) {
      if ((int)threadIdx.x < kt) {
        const int k = min(first + b * kt + (int)threadIdx.x, run.ctx - 1);
        slot[(b & 1) * KT + threadIdx.x] = bt[k / a.bs] * a.bs + k % a.bs;
      }
    };
    __syncthreads();                                                     // (the run before has been read)
    if (ba < be) put_slots(ba);
    for (int b = ba; b < be; ++b) {
      const int k0 = first + b * kt, nsub = min(kt, (run.ctx - k0 + 15) & ~15) >> 4;
      __syncthreads();                                                   // (the last block's weights have been read, the slots are written)
      f32x4 vf[KT / 16][4];
#pragma unroll
      for (int sb = 0; sb < KT / 16; ++sb)
#pragma unroll
        for (int i = 0; i < 4; ++i) vf[sb][i] = ld4(vc + (size_t)slot[(b & 1) * KT + 16 * min(sb, nsub - 1) + 4 * g + i] * ldkv);
      if (b + 1 < be) put_slots(b + 1);
      for (int j = wave; j < tn * nsub; j += NW) {                       // one token's 16 keys: lane (g, r) loads key r
        const int tk = j / nsub, sb = j - tk * nsub, k = k0 + 16 * sb + r;
        float* w = ws + (size_t)tk * H * ldw + 16 * sb + 4 * g;
        const bool in = tk >= xa && tk < run.y;
        const int ctx = in ? a.ctx_len[t0 + tk] : 0, low = low_of(a, ctx);
        const bool see = k >= low && k < ctx && k - (low & ~15) < p.ks;
        const float* s = p.sc + (size_t)(tr0 + tk) * H * p.ks + (see ? k - (low & ~15) : 0);
        const float* mt = ml + 2 * (size_t)tk * H;
        for (int c0 = 0; c0 < nhb; c0 += HB) {
          f32x4 acc[HB];
#pragma unroll
          for (int c = 0; c < HB; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (__any(see)) {
#pragma unroll 4
            for (int h = 0; h < hp; h += 4) {
              const int hh = h + g;
              const bool ok = see && hh < H;
              const int hs = min(hh, H - 1);
              const float v = ok ? s[(size_t)hs * p.ks] : 0.f;
              const float pr = ok ? expf(v - mt[2 * hs]) * mt[2 * hs + 1] : 0.f;
#pragma unroll
              for (int c = 0; c < HB; ++c) {
                const int col = 16 * (c0 + c) + r;
                const float tv = own ? tl[hh * hp + min(col, hp - 1)] : hh < H && col < H ? talk[(size_t)col * H + hh] : 0.f;
                acc[c] = mma(pr, tv, acc[c]);
              }
            }
          }
#pragma unroll
          for (int c = 0; c < HB; ++c) settle(acc[c]);
#pragma unroll
          for (int c = 0; c < HB; ++c)
            if (16 * (c0 + c) + r < H) *reinterpret_cast<f32x4*>(w + (size_t)(16 * (c0 + c) + r) * ldw) = acc[c];
        }
      }
      __syncthreads();
#pragma unroll
      for (int sb = 0; sb < KT / 16; ++sb) {
        f32x4 wf = *reinterpret_cast<const f32x4*>(wrow + 16 * min(sb, nsub - 1));
        if (!row || sb >= nsub) wf = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = mma(vf[sb][i][e], wf[i], o[e]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) settle(o[e]);
  // lane (g, r): columns 64 vb + 16 g + 4 i .. + 3 of row r
  auto put = [&](int tk, int h, int d, const f32x4& v) {
    const size_t t = t0 + tk;
    const T* ga = a.gate ? (const T*)a.gate + t * a.ldg + (size_t)h * a.V : nullptr;
    T* y = (T*)a.out + t * a.ldo + (size_t)h * Dp;
    bool fin = true;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (d + e < a.V) {
        y[d + e] = (T)(v[e] * (ga ? (float)ga[d + e] : 1.f));
        fin = fin && fabsf(v[e]) < INFINITY;
      }
    if (!fin) bad[tk] = 1;
  };
  auto each = [&](auto&& f) {
    if (on && row)
#pragma unroll
      for (int i = 0; i < 4; ++i) f(rtok, h0 + r % gr, 64 * vb + 16 * g + 4 * i, f32x4{o[0][i], o[1][i], o[2][i], o[3][i]});
  };
  __syncthreads();                                                       // (bad is written, the weights have been read)
  if (p.ns == 1) {
    each([&](int tk, int h, int d, const f32x4& v) {
      if (a.ctx_len[t0 + tk] > 0) put(tk, h, d, v);
    });
  } else {
    if (!any) return;
    if (na == 1) {
      each([&](int tk, int h, int d, const f32x4& v) { put(tk, h, d, v); });
    } else {
      each([&](int, int h, int d, const f32x4& v) {
        if (d < Dp) *reinterpret_cast<f32x4*>(p.part + (((size_t)tr0 * H + h) * p.ns + blockIdx.z) * Dp + d) = v;
      });
      // the last share to arrive adds them up
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0) {
        int* cp = p.cnt + (size_t)tr0 * gridDim.y + blockIdx.y;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const int old = __hip_atomic_fetch_add(cp, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int last = old == na - 1;
        if (last) {
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
          __hip_atomic_store(cp, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        bad[1] = last;
      }
      __syncthreads();
      if (!bad[1]) return;
      each([&](int tk, int h, int d, const f32x4&) {
        if (d >= Dp) return;
        const float* s = p.part + ((size_t)tr0 * H + h) * p.ns * Dp + d;
        f32x4 v = *reinterpret_cast<const f32x4*>(s);
        for (int z = 1; z < na; ++z) v += *reinterpret_cast<const f32x4*>(s + (size_t)z * Dp);
        put(tk, h, d, v);
      });
    }
  }
  __syncthreads();
  for (int tk = 0; tk < tn; ++tk) {
    if (!bad[tk]) continue;
    const size_t t = t0 + tk;
    const int low = low_of(a, a.ctx_len[t]), ctx = (int)min((long)a.ctx_len[t], (low & ~15) + p.ks);
    const int* bt = a.bt + (size_t)a.tok_seq[t] * a.bts;
    const float *mt = ml + 2 * (size_t)tk * H, *s = p.sc + (size_t)(tr0 + tk) * H * p.ks - (low & ~15);
    const int d = 64 * vb + lane;
    if (!on || d >= a.V) continue;
    for (int h = h0; h < h0 + gr; ++h) {
      float acc = 0.f;
      for (int k = low; k < ctx; ++k) {
        float w = 0.f;
        for (int i = 0; i < H; ++i) w = fmaf(talk[(size_t)h * H + i], expf(s[(size_t)i * p.ks + k] - mt[2 * i]) * mt[2 * i + 1], w);
        acc = fmaf(w, (float)((const T*)a.v)[((size_t)bt[k / a.bs] * a.bs + k % a.bs) * ldkv + (size_t)kh * Dp + d], acc);
      }
      ((T*)a.out)[t * a.ldo + (size_t)h * Dp + d] = (T)(acc * (a.gate ? (float)((const T*)a.gate)[t * a.ldg + (size_t)h * a.V + d] : 1.f));
    }
  }
}

template <class F>
bool lds_limit(F* f, size_t bytes) {
  return bytes <= 64 * 1024 || hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess;
}

template <typename T, int NW, int HB>
int launch_mix(const Rows& p, hipStream_t st) {
  const int H = p.a.H, hp = (H + 15) & ~15, njob = p.a.G * p.sub * ((p.a.V + 63) / 64);
  const size_t lds = sizeof(float) * ((size_t)p.tb * H * (p.kt + 4) + 2 * (size_t)p.tb * H + (H <= 64 ? hp * hp : 0) + 2 * KT + p.tb + 1);
  if (lds > 160 * 1024 || !lds_limit(talk_rows_mix_kernel<T, NW, HB>, lds)) return -1;
  hipLaunchKernelGGL((talk_rows_mix_kernel<T, NW, HB>), dim3((p.n + p.tb - 1) / p.tb, (njob + NW - 1) / NW, p.ns), dim3(64 * NW), lds, st, p);
  return (int)hipGetLastError();
}

// nw: 4 or 8 waves of the mix
template <typename T>
int launch(const Rows& p, int nw, hipStream_t st) {
  const int nks = (p.a.Dp + 15) / 16, ldl = (nks + KC - 1) / KC * KC * 16 + 4;
  const size_t lds = sizeof(float) * (NW * 32 + 16 * (size_t)ldl);
  if (lds > 160 * 1024 || !lds_limit(talk_rows_score_kernel<T>, lds)) return -1;
  hipLaunchKernelGGL(talk_rows_score_kernel<T>, dim3((p.n + p.tb1 - 1) / p.tb1, p.a.G * p.sub, p.ns1), dim3(NT), lds, st, p);
  const int rc = (int)hipGetLastError();
  if (rc) return rc;
  if (nw == 8) return p.a.H <= 16 ? launch_mix<T, 8, 1>(p, st) : launch_mix<T, 8, 2>(p, st);
  return p.a.H <= 16 ? launch_mix<T, 4, 1>(p, st) : launch_mix<T, 4, 2>(p, st);
}

}  // namespace plain
}  // namespace nls_talk
