// Decoded tokens of layers with attention and a gated linear recurrence side by side: both in one launch (gfx950).
//
// Neither reads what the other writes. The recurrence streams its states (64 tokens of 32 heads of 64 x 128: 134 MB read and written),
// the attention of few hundred keys is one chain of dependent loads, so each leaves idle what the other needs. Graph launches, bf16, 32
// heads of 128 over 8 beside 32 states of 64 x 128, us, one behind the other / together: 1 token behind 90 keys 12.1 / 7.1,
// behind 1500 16.4 / 11.0; with cold states and keys 16 tokens behind 90 and 1000 20 / 14 and 37 / 32, 64 tokens 43 / 37 and 101 / 86, 300 tokens 159 / 149 and
// 424 / 369. Of 375 sizes of 1 to 300 tokens behind 20 to 3000 keys 0.80 of the time on average; slower are 128 tokens and more behind 20 keys (61 /
// 65 to 138 / 141: three of four waves have no keys) and three sizes behind 3000 (1 to 6 %). The attention takes four waves and gives up the prefetch of
// the next keys: that leaves registers for three workgroups on a CU, of which two would not keep the states' loads in flight.
// In 32 bits the plain attention keeps all its registers, a CU holds one workgroup: that pays up to two rounds of states (3 tokens behind 330
// keys 24.9 / 20.1, 16 tokens 30.6 / 23.4; 32 tokens, 1024 states, 45.1 / 49.4).
#include "../kernels/attn_decode.h"
#include "attn_plain.h"
#include "scan.h"

namespace nls_both {
using namespace nls_attn;
using namespace nls_scan;

struct AT {
  const __bf16 *q, *k, *v;
  __bf16* out;
  const float* gate;
  float *part_o, *part_ml;
  int* cnt;
  const int *bt, *tok_seq, *ctx_len;
  long ldq, ldo, ldg;
  int bts, bs, T, G, gq, gy, ns;
  float scale;
  AttnMask mask;
};

// The states of the launch: workgroups from T * gy * ns on, one each; those before are the attention of a token's heads, a share of its keys.
template <int RPT>
struct TokenStates {
  static constexpr int lds = step_lds(256), waves = 3;
  int T, gy, ns;
  Scan p;
  StepOut y;
  DEVI bool operator()(uint8_t* sm, int& t, int& by, int& ngy, int& split) const {
    const int n = T * gy * ns, b = t;
    if (b < n) {
      const int u = b / T;
      split = u / gy;
      t = b - u * T;
      by = u - split * gy;
      ngy = gy;
      return false;
    }
    const int row = (b - n) / p.H;
    step_body<__bf16, GLA, 256, RPT>(reinterpret_cast<float*>(sm), p, y, b - n - row * p.H, p.H, row);
    return true;
  }
};

template <int D, int RPT>
int launch_rpt(const AT& a, const Scan& p, const StepOut& y, hipStream_t st) {
  hipLaunchKernelGGL((attn_decode_mfma_kernel<__bf16, 4, D, __bf16, false, false, TokenStates<RPT>>), dim3(a.T * (a.gy * a.ns + p.H)), dim3(256), 0,
                     st, a.q, a.ldq, a.k, a.v, a.bt, a.bts, a.tok_seq, a.ctx_len, a.G, a.gq, a.bs, a.scale, 0, a.ns, a.out, a.ldo, a.part_o, a.part_ml, a.cnt,
                     a.gate, a.ldg, a.mask, TokenStates<RPT>{a.T, a.gy, a.ns, p, y});
  return (int)hipGetLastError();
}

template <int D>
int launch(const AT& a, const Scan& p, const StepOut& y, hipStream_t st) {
  const int rpt = step_rpt(p.D, p.V, 256);
  return rpt <= 4 ? launch_rpt<D, 4>(a, p, y, st) : rpt <= 8 ? launch_rpt<D, 8>(a, p, y, st) : rpt <= 16 ? launch_rpt<D, 16>(a, p, y, st) : -1;
}

// 32-bit models: the same with the plain attention's grid of gx x gy
template <int NT, int RPT>
struct States {
  int gx, gy;
  Scan p;
  StepOut y;
  DEVI bool operator()(float* sm, int& bx, int& by, int& bz, int& ngx) const {
    const int n = gx * gy, b = bx;
    if (b < n) {
      by = b / gx;
      bx = b - by * gx;
      bz = 0;
      ngx = gx;
      return false;
    }
    const int row = (b - n) / p.H;
    step_body<float, GLA, NT, RPT>(sm, p, y, b - n - row * p.H, p.H, row);
    return true;
  }
};

template <int NQ, int RPT>
int plain_rpt(const nls_plain::PA& a, dim3 g, const Scan& p, const StepOut& y, hipStream_t st) {
  const size_t lds = max(nls_plain::plain_lds(a.Dk, NQ, 8), (size_t)step_lds(512));
  hipLaunchKernelGGL((nls_plain::attn_plain_kernel<float, NQ, 8, States<512, RPT>>), dim3(g.x * g.y + a.T * p.H), dim3(512), lds, st, a,
                     States<512, RPT>{(int)g.x, (int)g.y, p, y});
  return (int)hipGetLastError();
}

template <int NQ>
int plain_launch(const nls_plain::PA& a, dim3 g, const Scan& p, const StepOut& y, hipStream_t st) {
  const int rpt = step_rpt(p.D, p.V, 512);
  return rpt <= 4 ? plain_rpt<NQ, 4>(a, g, p, y, st) : rpt <= 8 ? plain_rpt<NQ, 8>(a, g, p, y, st) : -1;
}

int plain(nls_plain::PA a, int T, int H, const Scan& p, const StepOut& y, hipStream_t st) {
  dim3 g;
  if (a.Dk > 256 || a.Dv > 256 || !nls_plain::prepare(a, T, H, g) || !nls_plain::small(g)) return -1;       // (LDS: 36 KB)
  return a.Dv <= 64 ? plain_launch<1>(a, g, p, y, st) : a.Dv <= 128 ? plain_launch<2>(a, g, p, y, st) : plain_launch<4>(a, g, p, y, st);
}

}  // namespace nls_both

extern "C" {

// nls_gqa_attn (no window) and nls_gla_step (with a norm) of the same T rows, each a run of one token, in one launch.
// Dp 64 or 128 (32-bit: up to 256, ns and its scratch unused); at most 16 rows of a state per thread (step_rpt).
int nls_attn_step(const void* aq, long ldaq, const void* ak, const void* av, const int* bt, int bts, int bs, const int* tok_seq,
                  const int* ctx_len, int T, int AH, int AG, int Dp, float scale, const float* agate, long ldag, void* aout,
                  long ldaout, int sink, int ns, float* part_o, float* part_ml, int* cnt, const void* q, const void* k, const void* v, long ld, const float* a, long lda,
                  const void* low, const void* a2, const float* a2b, int rank, float ia, float qscale, float* state, long sstride,
                  const int* runs, const float* norm, const void* gate, long ldg, void* out, long ldout, int H,
                  int D, int V, float eps, int f32, void* stream) {
  using namespace nls_both;
  if (T < 1 || AG < 1 || AH < 1 || AH % AG || bs < 1 || Dp < 1 || !norm || !gate || !out) return -1;
  if (H < 1 || D < 1 || D > 256 || V < 4 || V > 1024 || (V & 3) || (sstride & 3)) return -1;
  if (!a && (!low || !a2 || !a2b || rank < 1 || ((uintptr_t)low & 15) || ((uintptr_t)a2 & 15) || (ld & 7))) return -1;
  const Scan p{q, k, v, a, nullptr, nullptr, state, nullptr, nullptr, runs, ld, lda, 0, sstride, 0, 0, H, D, V, 0, qscale,
               low, a2, a2b, rank, ia};
  const StepOut y{norm, gate, ldg, out, ldout, eps};
  if (f32)
    return plain({aq, ak, av, aout, bt, tok_seq, ctx_len, agate, ldaq, Dp, (long)AG * Dp, Dp, ldaout, Dp, ldag, bts, bs, AH / AG, Dp,
                  Dp, scale, 0, 0, sink}, T, AH, p, y, (hipStream_t)stream);
  if (bs < 16 || (ldaq & 7) || (ldaout & 3) || ns < 1 || ns > 64 || (ns > 1 && (!part_o || !part_ml || !cnt))) return -1;
  const int gq = AH / AG;
  const AT at{(const __bf16*)aq, (const __bf16*)ak, (const __bf16*)av, (__bf16*)aout, agate, part_o, part_ml, cnt, bt, tok_seq, ctx_len,
              ldaq, ldaout, ldag, bts, bs, T, AG, gq, AG * ((gq + 15) / 16), ns, scale, {0, 0, sink}};
  return Dp == 64 ? launch<64>(at, p, y, (hipStream_t)stream) : Dp == 128 ? launch<128>(at, p, y, (hipStream_t)stream) : -1;
}

}  // extern "C"
