// Dense attention for few query rows: decode steps (N_q = 1) and short chunks
// of queries against a long key range.
//
// The query heads that share a K / V head and their N_q queries are the
// R = group * N_q rows of one unit (b, K / V head), at most 32. K and V are
// then read once per unit, straight from their rows, and the key range is
// split over workgroups so that the chip is full whatever B * H_kv is:
//  1. row_attn_kernel: grid (split, unit). Each wave walks its own 32-key
//     steps of the split's range:
//       S^T = K Q^T       (A = K rows, B = Q in registers)
//       online softmax, fp32, log2 domain
//       O^T += V^T P^T    (A = V^T, B = P; see below)
//       row sums = 1 P^T  (the sums of exactly the rounded P used)
//     and the four waves' states are merged in LDS into one partial (O, m, l)
//     per row and split. With totals wanted, the scaled scores go to the
//     workspace too (4 bytes per row and key, beside 4 D bytes of K and V).
//  2. row_combine_kernel: merges a row's splits into out and lse, and adds
//     each key's softmax totals: exp2(score - lse), from the stored scores,
//     so K is not read again.
// V^T needs no transposition through memory: lane (c = lane % 16, g =
// lane / 16) loads the D / 16 values d = (D / 16) c .. of the eight keys its
// k-slots stand for (whole V rows per instruction), and byte permutes form
// the operand of output tile dt from element dt of each row. Row i of that
// tile is then d = (D / 16) i + dt, a fixed reordering of O's dims.
// fp32 inputs: every operand is split into bf16 hi and lo halves in registers
// and each product is three MFMA (a_hi b_hi + a_lo b_hi + a_hi b_lo), as in
// the other attention kernels.
//
// Bound: HBM (K and V read once). Measured with totals, bf16, 32 query heads on
// 8 K / V heads, D = 128, one query: 8 sequences of 32768 keys 222 us (5.1 TB/s
// of K, V, scores and totals; 1078 us as one workgroup per head over packed V
// and a second pass over K for the totals); one sequence of 4099 keys 20 us a
// call, host time included (78 us): 7.1 + 3.7 us of kernels in the profiler.
#include "attn_common.h"
#include "row_attn.h"

namespace cab {
namespace {

constexpr int STEP = 32;        // keys per wave step
// Rows per unit, and queries per head when totals are wanted, beyond which the
// general kernels are as fast or faster (bf16, causal, us, general -> here):
// 32 rows 28.3 -> 17.5 (32 heads on 8, 8 queries, 4099 keys), 39.0 -> 34.1 (12
// heads, 8000 keys); 64 rows 28.6 -> 29.4 (32 on 8, 16 queries, 4099 keys). With
// totals 24 queries 51.6 -> 44.2 (32 heads, 5000 keys), 32 queries 34.0 -> 37.3
// (32 heads, 2000 keys).
constexpr int MAX_ROWS = 32;
constexpr int MAX_TOTAL_QUERIES = 24;
constexpr int MAX_SPLITS = 256;
constexpr int KEYS_PER_WG = 1024;  // keys one row_combine workgroup totals
// Workgroups a plan aims at: two per CU run at a time (512, 1024 and 2048
// measured within 1 %; 1024 leaves the last round short where units are few).
constexpr int ROW_WGS = 1024;

// K and V are read once: non-temporal loads (8 sequences of 32768 keys, 8 K / V
// heads: 222 against 235 us).
template <typename T>
__device__ __forceinline__ T ld_stream(const char* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const T*>(p));
}

struct RowArgs {
  const char* q;
  const char* k;
  const char* v;
  int64_t qs[3], ks[3], vs[3];  // bytes: b, h, token
  int32_t Hkv, group, Nq, Nk, R, qoff, causal;
  int32_t steps, sps, splits;  // 32-key steps: all, per split; splits
  float c;                     // scale * log2(e)
  float* po;                   // [unit][R][splits][D]
  float* pm;                   // [unit][R][splits] running maxima (raw scores)
  float* pl;                   // [unit][R][splits] row sums
  float* s;                    // [unit][R][ld] scores * c, or null
  int64_t ld;
};

// One 32-key step's K and V values of a lane, as loaded.
template <cab_dtype_t DT, int HD>
struct StepRegs {
  static constexpr bool F32 = DT == CAB_F32;
  static constexpr int NDS = HD / 32;
  static constexpr int VB = HD / 16 * (F32 ? 4 : 2);  // V bytes per lane and key
  static constexpr int NV = VB / 8;                   // 8-byte pieces of them
  u32x4 k[2][NDS][F32 ? 2 : 1];
  u32x2 v[8][NV];
};

template <cab_dtype_t DT, int HD, bool TAIL>
__device__ __forceinline__ void load_step(StepRegs<DT, HD>& x, const char* kb, const char* vb,
                                          uint32_t koff, uint32_t voff, uint32_t krow, uint32_t vrow,
                                          int key0, int Nk, int l16, int g) {
  using SR = StepRegs<DT, HD>;
  const char* kp = kb + static_cast<int64_t>(key0) * krow;
  const char* vp = vb + static_cast<int64_t>(key0) * vrow;
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const bool in = !TAIL || key0 + 16 * tt + l16 < Nk;
#pragma unroll
    for (int ds = 0; ds < SR::NDS; ++ds)
#pragma unroll
      for (int p = 0; p < (SR::F32 ? 2 : 1); ++p) {
        x.k[tt][ds][p] = u32x4{0u, 0u, 0u, 0u};
        if (in)
          x.k[tt][ds][p] = ld_stream<u32x4>(kp + (koff + 16u * tt * krow) +
                                             (SR::F32 ? 128 : 64) * ds + 16 * p);
      }
  }
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int kr = 16 * (r >> 2) + (r & 3);  // + 4 g: this k-slot's key
    const bool in = !TAIL || key0 + kr + 4 * g < Nk;
#pragma unroll
    for (int n = 0; n < SR::NV; ++n) x.v[r][n] = u32x2{0u, 0u};
    if (in) {
      const char* p = vp + (voff + static_cast<uint32_t>(kr) * vrow);
      if constexpr (SR::NV == 1) {
        x.v[r][0] = ld_stream<u32x2>(p);
      } else {
#pragma unroll
        for (int n = 0; n < SR::NV; n += 2) {
          const u32x4 y = ld_stream<u32x4>(p + 8 * n);
          x.v[r][n] = u32x2{y[0], y[1]};
          x.v[r][n + 1] = u32x2{y[2], y[3]};
        }
      }
    }
  }
}

template <int QT, int HD>
struct RowAcc {
  f32x4 o[QT][HD / 16];  // O^T tile dt: row 4 g + r is d = (HD / 16) (4 g + r) + dt; query l16
  f32x4 l[QT];           // row sums (all four equal)
  float m[QT];           // running maxima of the raw scores
};

template <cab_dtype_t DT, int HD, int QT, bool SC>
__global__ __launch_bounds__(256, DT == CAB_F32 ? 1 : 2) void row_attn_kernel(RowArgs a) {
  constexpr bool F32 = DT == CAB_F32;
  constexpr bool BF16 = DT != CAB_F16;
  constexpr int NDS = HD / 32, NDT = HD / 16;
  using SR = StepRegs<DT, HD>;
  __shared__ f32x4 merge[4][NDT * 64];  // one query tile's O^T per wave
  __shared__ float sm[4][QT][16], sl[4][QT][16];

  const int split = blockIdx.x, unit = blockIdx.y;
  const int b = unit / a.Hkv, hk = unit - b * a.Hkv;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int lane = lane_id(), l16 = lane & 15, g = lane >> 4;
  const float c = a.c;
  const char* kb = a.k + b * a.ks[0] + hk * a.ks[1];
  const char* vb = a.v + b * a.vs[0] + hk * a.vs[1];
  const uint32_t krow = static_cast<uint32_t>(a.ks[2]), vrow = static_cast<uint32_t>(a.vs[2]);
  const uint32_t koff = l16 * krow + (F32 ? 32 : 16) * g;
  const uint32_t voff = 4 * g * vrow + SR::VB * l16;

  // Q^T operands of the rows r = 16 qt + l16 (zero past R), and how many
  // leading keys each row sees.
  u32x4 qh[QT][NDS], ql[QT][F32 ? NDS : 1];
  int lim[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int r = 16 * qt + l16;
    const int hg = r / a.Nq, t = r - hg * a.Nq;
    const bool in = r < a.R;
    lim[qt] = !in ? 0 : a.causal ? min(a.Nk, t + a.qoff + 1) : a.Nk;
    const char* qp = a.q + b * a.qs[0] + (static_cast<int64_t>(hk) * a.group + hg) * a.qs[1] + t * a.qs[2];
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) {
      if constexpr (F32) {
        f32x4 x0 = {0.f, 0.f, 0.f, 0.f}, x1 = x0;
        if (in) {
          x0 = *reinterpret_cast<const f32x4*>(qp + 128 * ds + 32 * g);
          x1 = *reinterpret_cast<const f32x4*>(qp + 128 * ds + 32 * g + 16);
        }
        split8(x0, x1, qh[qt][ds], ql[qt][ds]);
      } else {
        qh[qt][ds] = u32x4{0u, 0u, 0u, 0u};
        if (in) qh[qt][ds] = *reinterpret_cast<const u32x4*>(qp + 64 * ds + 16 * g);
      }
    }
  }
  RowAcc<QT, HD> st;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    st.l[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
    st.m[qt] = M_EMPTY;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) st.o[qt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const uint32_t one2 = BF16 ? 0x3f803f80u : 0x3c003c00u;
  const u32x4 ones = {one2, one2, one2, one2};
  // Keys below this are seen by every row (causal: by the first query).
  const int all_see = a.causal ? min(a.Nk, a.qoff + 1) : a.Nk;

  auto load = [&](int step, SR& x) {
    const int key0 = STEP * step;
    if (key0 + STEP <= a.Nk)
      load_step<DT, HD, false>(x, kb, vb, koff, voff, krow, vrow, key0, a.Nk, l16, g);
    else
      load_step<DT, HD, true>(x, kb, vb, koff, voff, krow, vrow, key0, a.Nk, l16, g);
  };
  auto compute = [&](int step, const SR& x) {
    const int key0 = STEP * step;
    // sc[qt][tt][r] = score(key key0 + 16 tt + 4 g + r, row 16 qt + l16)
    f32x4 sc[QT][2];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) sc[qt][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        if constexpr (F32) {
          u32x4 kh, kl;
          split8(__builtin_bit_cast(f32x4, x.k[tt][ds][0]), __builtin_bit_cast(f32x4, x.k[tt][ds][1]),
                 kh, kl);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) {
            sc[qt][tt] = mfma16<true>(kl, qh[qt][ds], sc[qt][tt]);
            sc[qt][tt] = mfma16<true>(kh, ql[qt][ds], sc[qt][tt]);
            sc[qt][tt] = mfma16<true>(kh, qh[qt][ds], sc[qt][tt]);
          }
        } else {
#pragma unroll
          for (int qt = 0; qt < QT; ++qt)
            sc[qt][tt] = mfma16<BF16>(x.k[tt][ds][0], qh[qt][ds], sc[qt][tt]);
        }
      }
    if (key0 + STEP > all_see) {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (key0 + 16 * tt + 4 * g + r >= lim[qt]) sc[qt][tt][r] = -INFINITY;
    }
    u32x4 pb[QT], pl[F32 ? QT : 1];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      if constexpr (SC) {
        const int row = 16 * qt + l16;
        if (row < a.R) {
          float* sp = a.s + (static_cast<int64_t>(unit) * a.R + row) * a.ld + key0 + 4 * g;
          *reinterpret_cast<f32x4*>(sp) = sc[qt][0] * c;
          *reinterpret_cast<f32x4*>(sp + 16) = sc[qt][1] * c;
        }
      }
      const float m0 = fmaxf(fmaxf(sc[qt][0][0], sc[qt][0][1]), fmaxf(sc[qt][0][2], sc[qt][0][3]));
      const float m1 = fmaxf(fmaxf(sc[qt][1][0], sc[qt][1][1]), fmaxf(sc[qt][1][2], sc[qt][1][3]));
      float mx = fmaxf(m0, m1), mdup = mx;
      colmax2(mx, mdup);
      if (__builtin_amdgcn_ballot_w64(mx > st.m[qt]) != 0) {
        const float mn = fmaxf(mx, st.m[qt]);
        const float alpha = __builtin_amdgcn_exp2f((st.m[qt] - mn) * c);
        st.l[qt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) st.o[qt][dt] *= alpha;
        st.m[qt] = mn;
      }
      const float nmc = -st.m[qt] * c;
      float p[2][4];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          p[tt][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[qt][tt][r], c, nmc));
      if constexpr (F32) {
        split8(f32x4{p[0][0], p[0][1], p[0][2], p[0][3]}, f32x4{p[1][0], p[1][1], p[1][2], p[1][3]},
               pb[qt], pl[qt]);
        st.l[qt] = mfma16<true>(ones, pl[qt], st.l[qt]);
        st.l[qt] = mfma16<true>(ones, pb[qt], st.l[qt]);
      } else {
        pb[qt] = u32x4{pack2<BF16>(p[0][0], p[0][1]), pack2<BF16>(p[0][2], p[0][3]),
                       pack2<BF16>(p[1][0], p[1][1]), pack2<BF16>(p[1][2], p[1][3])};
        st.l[qt] = mfma16<BF16>(ones, pb[qt], st.l[qt]);
      }
    }
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      if constexpr (F32) {
        u32x4 vh, vl;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t lo = x.v[2 * e][dt >> 1][dt & 1], hi = x.v[2 * e + 1][dt >> 1][dt & 1];
          const u32x2 y = split2(__uint_as_float(lo), __uint_as_float(hi));
          vh[e] = y[0];
          vl[e] = y[1];
        }
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
          st.o[qt][dt] = mfma16<true>(vl, pb[qt], st.o[qt][dt]);
          st.o[qt][dt] = mfma16<true>(vh, pl[qt], st.o[qt][dt]);
          st.o[qt][dt] = mfma16<true>(vh, pb[qt], st.o[qt][dt]);
        }
      } else {
        u32x4 vo;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t lo = x.v[2 * e][dt >> 2][(dt >> 1) & 1];
          const uint32_t hi = x.v[2 * e + 1][dt >> 2][(dt >> 1) & 1];
          vo[e] = __builtin_amdgcn_perm(hi, lo, dt & 1 ? 0x07060302u : 0x05040100u);
        }
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) st.o[qt][dt] = mfma16<BF16>(vo, pb[qt], st.o[qt][dt]);
      }
    }
  };

  const int end = min(a.steps, (split + 1) * a.sps);
  int step = split * a.sps + w;
  if constexpr (F32 || QT * HD > 128) {  // (two register sets would spill)
    SR x;
    for (; step < end; step += 4) {
      load(step, x);
      compute(step, x);
    }
  } else {
    // Two register sets: a step's loads are in flight while the one before
    // it is computed.
    SR x, y;
    if (step < end) load(step, x);
    for (; step < end; step += 8) {
      if (step + 4 < end) load(step + 4, y);
      compute(step, x);
      if (step + 4 < end) {
        if (step + 8 < end) load(step + 8, x);
        compute(step + 4, y);
      }
    }
  }

  // Merge of the four waves: common maximum, then the scaled O^T and row
  // sums added in wave order.
  if (g == 0) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) sm[w][qt][l16] = st.m[qt];
  }
  __syncthreads();
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const float m = fmaxf(fmaxf(sm[0][qt][l16], sm[1][qt][l16]), fmaxf(sm[2][qt][l16], sm[3][qt][l16]));
    const float f = __builtin_amdgcn_exp2f((st.m[qt] - m) * c);
    if (g == 0) sl[w][qt][l16] = st.l[qt][0] * f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) merge[w][dt * 64 + lane] = st.o[qt][dt] * f;
    __syncthreads();
    // Thread tid takes (dt, lane') pairs: row 16 qt + lane' % 16, values
    // d = NDT (4 (lane' / 16) + r) + dt.
    for (int e = threadIdx.x; e < NDT * 64; e += 256) {
      const int dt = e >> 6, ll = e & 63, row = 16 * qt + (ll & 15);
      const f32x4 o = (merge[0][e] + merge[1][e]) + (merge[2][e] + merge[3][e]);
      if (row < a.R) {
        float* po = a.po + ((static_cast<int64_t>(unit) * a.R + row) * a.splits + split) * HD;
#pragma unroll
        for (int r = 0; r < 4; ++r) po[NDT * (4 * (ll >> 4) + r) + dt] = o[r];
      }
    }
    const int row = 16 * qt + static_cast<int>(threadIdx.x);
    if (threadIdx.x < 16 && row < a.R) {
      const int64_t x = (static_cast<int64_t>(unit) * a.R + row) * a.splits + split;
      a.pm[x] = m;
      a.pl[x] = (sl[0][qt][l16] + sl[1][qt][l16]) + (sl[2][qt][l16] + sl[3][qt][l16]);
    }
    if (qt + 1 < QT) __syncthreads();
  }
}

struct CombineArgs {
  const float* po;
  const float* pm;
  const float* pl;
  const float* s;
  int64_t ld;
  int32_t H, Nq, Nk, splits;
  int32_t qoff, causal;
  float c;
  char* out;
  int64_t os[3];  // bytes
  float* lse;
  const float* old_scores;
  int64_t olds[2], n_old;
  float* scores;
  int64_t ss[2];
};

// Maximum and merged row sum of one row's splits, in every lane of a wave
// (pm, pl: the row's entries; splits <= MAX_SPLITS).
__device__ __forceinline__ void merge_row(const float* pm, const float* pl, int splits, float c,
                                          float& m, float& l) {
  constexpr int PER = MAX_SPLITS / 64;
  const int lane = lane_id();
  float pmv[PER], plv[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int x = 64 * i + lane;
    pmv[i] = x < splits ? pm[x] : M_EMPTY;
    plv[i] = x < splits ? pl[x] : 0.f;
  }
  m = fmaxf(fmaxf(pmv[0], pmv[1]), fmaxf(pmv[2], pmv[3]));
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, shfl_xor_f32(m, off));
  l = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) l += plv[i] * __builtin_amdgcn_exp2f((pmv[i] - m) * c);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) l += shfl_xor_f32(l, off);
}

// Workgroups (x, bh): x < Nq merges query x's splits into out and lse; the
// others add the totals of KEYS_PER_WG keys each.
template <cab_dtype_t DT, int HD>
__global__ __launch_bounds__(256) void row_combine_kernel(CombineArgs a) {
  const int bh = blockIdx.y;
  const int b = bh / a.H, h = bh - b * a.H;
  const int tid = threadIdx.x, w = tid >> 6;
  const float c = a.c;
  if (static_cast<int>(blockIdx.x) >= a.Nq) {
    constexpr int PER = KEYS_PER_WG / 256;
    __shared__ float lse2[MAX_ROWS];
    const int key0 = (blockIdx.x - a.Nq) * KEYS_PER_WG + tid;
    const float* srow = a.s + static_cast<int64_t>(bh) * a.Nq * a.ld;
    const float* orow = a.old_scores + (b * a.olds[0] + h * a.olds[1]);
    // The first query's scores and the old totals are loaded before the lse
    // is formed from the splits.
    float sv[PER], tot[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int key = key0 + 256 * i;
      sv[i] = key < a.Nk ? srow[key] : -INFINITY;
      tot[i] = key < a.n_old ? orow[key] : 0.f;
    }
    for (int t = w; t < a.Nq; t += 4) {
      const int64_t row = (static_cast<int64_t>(bh) * a.Nq + t) * a.splits;
      float m, l;
      merge_row(a.pm + row, a.pl + row, a.splits, c, m, l);
      // (a query without keys adds nothing; one whose sum is NaN makes the totals of
      // the keys it sees NaN, and of no others)
      if (lane_id() == 0) lse2[t] = l == 0.f ? INFINITY : m * c + __log2f(l);
    }
    __syncthreads();
    // Keys query t does not see hold scores of -inf; they add 0 whatever its lse.
    const int see = a.causal ? a.qoff + 1 : a.Nk;  // + t where causal
    float sum[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i)
      sum[i] = key0 + 256 * i < see ? __builtin_amdgcn_exp2f(sv[i] - lse2[0]) : 0.f;
#pragma unroll 4
    for (int t = 1; t < a.Nq; ++t) {
      const int lim = a.causal ? see + t : see;
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int key = key0 + 256 * i;  // (past the keys: a key of the row, not stored)
        const float p = __builtin_amdgcn_exp2f(srow[t * a.ld + (key < a.Nk ? key : 0)] - lse2[t]);
        sum[i] += key < lim ? p : 0.f;
      }
    }
    float* drow = a.scores + b * a.ss[0] + h * a.ss[1];
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (key0 + 256 * i < a.Nk) drow[key0 + 256 * i] = tot[i] + sum[i];
    return;
  }

  // Thread tid sums values d = 4 (tid % (HD / 4)) .. + 3 over every NG-th split.
  constexpr int TD = HD / 4, NG = 256 / TD;
  __shared__ f32x4 part[256];
  const int t = blockIdx.x;
  const int64_t row = (static_cast<int64_t>(bh) * a.Nq + t) * a.splits;
  const int grp = tid / TD;
  float m, l;
  merge_row(a.pm + row, a.pl + row, a.splits, c, m, l);
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int x = grp; x < a.splits; x += NG)
    o += reinterpret_cast<const f32x4*>(a.po + (row + x) * HD)[tid % TD] *
         __builtin_amdgcn_exp2f((a.pm[row + x] - m) * c);
  part[tid] = o;
  __syncthreads();
  if (grp != 0) return;
#pragma unroll
  for (int i = 1; i < NG; ++i) o += part[i * TD + tid];
  o *= l > 0.f ? 1.0f / l : 0.f;
  char* op = a.out + b * a.os[0] + h * a.os[1] + t * a.os[2];
  if constexpr (DT == CAB_F32)
    reinterpret_cast<f32x4*>(op)[tid] = o;
  else
    reinterpret_cast<u32x2*>(op)[tid] = u32x2{pack2<DT == CAB_BF16>(o[0], o[1]),
                                              pack2<DT == CAB_BF16>(o[2], o[3])};
  if (tid == 0 && a.lse)
    a.lse[static_cast<int64_t>(bh) * a.Nq + t] =
        l > 0.f ? (m * c + __log2f(l)) * 0.69314718055994531f : -INFINITY;
}

// The split of a problem and its workspace layout.
struct RowPlan {
  int64_t units, R, steps, sps, splits, ld;
  size_t off_pm, off_pl, off_s, bytes;
};

RowPlan row_plan(int64_t B, int64_t H, int64_t Hkv, int64_t Nq, int64_t Nk, int64_t D, bool scores) {
  RowPlan p;
  p.units = B * Hkv;
  p.R = H / Hkv * Nq;
  p.steps = ceil_div(Nk, STEP);
  const int64_t want = ceil_div(ROW_WGS, p.units);
  int64_t splits = want < MAX_SPLITS ? want : MAX_SPLITS;
  p.sps = round_up(ceil_div(p.steps, splits), 4);
  p.splits = ceil_div(p.steps, p.sps);
  p.ld = round_up(Nk, STEP);
  const int64_t rows = p.units * p.R;
  p.off_pm = static_cast<size_t>(rows * p.splits * D) * 4;
  p.off_pl = p.off_pm + static_cast<size_t>(round_up(rows * p.splits, 4)) * 4;
  p.off_s = p.off_pl + static_cast<size_t>(round_up(rows * p.splits, 4)) * 4;
  p.bytes = p.off_s + (scores ? static_cast<size_t>(rows * p.ld) * 4 : 0);
  return p;
}

template <cab_dtype_t DT, int HD, int QT>
void launch_rows(const RowArgs& a, dim3 grid, hipStream_t s) {
  if (a.s)
    row_attn_kernel<DT, HD, QT, true><<<grid, 256, 0, s>>>(a);
  else
    row_attn_kernel<DT, HD, QT, false><<<grid, 256, 0, s>>>(a);
}

template <cab_dtype_t DT, int HD>
void launch_dt(const RowArgs& a, dim3 grid, const CombineArgs& ca, dim3 cgrid, hipStream_t s) {
  if (a.R <= 16)
    launch_rows<DT, HD, 1>(a, grid, s);
  else
    launch_rows<DT, HD, 2>(a, grid, s);
  row_combine_kernel<DT, HD><<<cgrid, 256, 0, s>>>(ca);
}

}  // namespace

bool row_attn_applies(cab_dtype_t dtype, int64_t B, int64_t H, int64_t Hkv, int64_t Nq, int64_t Nk,
                      int64_t D, const int64_t* k_strides, const int64_t* v_strides, bool scores) {
  if (scores && Nq > MAX_TOTAL_QUERIES) return false;
  if (B < 1 || Hkv < 1 || H < Hkv || Nq < 1 || Nk < 1) return false;
  if (H / Hkv * Nq > MAX_ROWS || B * H > 65535) return false;  // grid.y
  // 32 rows of K and of V are addressed by 32-bit offsets.
  const int64_t lim = int64_t{1} << 24;
  return k_strides[2] <= lim && v_strides[2] <= lim;
}

size_t row_attn_workspace(int64_t B, int64_t H, int64_t Hkv, int64_t Nq, int64_t Nk, int64_t D,
                          bool scores) {
  return row_plan(B, H, Hkv, Nq, Nk, D, scores).bytes;
}

cab_status_t row_attn_launch(const char* fn, const RowAttnProblem& p, void* ws, hipStream_t s) {
  const RowPlan pl = row_plan(p.B, p.H, p.Hkv, p.Nq, p.Nk, p.D, p.scores != nullptr);
  const int64_t es = static_cast<int64_t>(dtype_size(p.dtype));
  char* wsb = static_cast<char*>(ws);
  RowArgs a;
  a.q = static_cast<const char*>(p.q);
  a.k = static_cast<const char*>(p.k);
  a.v = static_cast<const char*>(p.v);
  CombineArgs ca;
  for (int d = 0; d < 3; ++d) {
    a.qs[d] = p.qs[d] * es;
    a.ks[d] = p.ks[d] * es;
    a.vs[d] = p.vs[d] * es;
    ca.os[d] = p.os[d] * es;
  }
  a.Hkv = static_cast<int32_t>(p.Hkv);
  a.group = static_cast<int32_t>(p.H / p.Hkv);
  a.Nq = static_cast<int32_t>(p.Nq);
  a.Nk = static_cast<int32_t>(p.Nk);
  a.R = static_cast<int32_t>(pl.R);
  a.qoff = static_cast<int32_t>(p.Nk - p.Nq);
  a.causal = p.causal ? 1 : 0;
  a.steps = static_cast<int32_t>(pl.steps);
  a.sps = static_cast<int32_t>(pl.sps);
  a.splits = static_cast<int32_t>(pl.splits);
  a.c = static_cast<float>(static_cast<double>(p.scale) * 1.4426950408889634);
  a.po = reinterpret_cast<float*>(wsb);
  a.pm = reinterpret_cast<float*>(wsb + pl.off_pm);
  a.pl = reinterpret_cast<float*>(wsb + pl.off_pl);
  a.s = p.scores ? reinterpret_cast<float*>(wsb + pl.off_s) : nullptr;
  a.ld = pl.ld;
  ca.po = a.po;
  ca.pm = a.pm;
  ca.pl = a.pl;
  ca.s = a.s;
  ca.ld = a.ld;
  ca.H = static_cast<int32_t>(p.H);
  ca.Nq = a.Nq;
  ca.Nk = a.Nk;
  ca.splits = a.splits;
  ca.qoff = a.qoff;
  ca.causal = a.causal;
  ca.c = a.c;
  ca.out = static_cast<char*>(p.out);
  ca.lse = p.lse;
  ca.old_scores = p.old_scores;
  ca.n_old = p.old_scores ? p.n_old : 0;
  ca.scores = p.scores;
  for (int d = 0; d < 2; ++d) {
    ca.olds[d] = p.olds[d];
    ca.ss[d] = p.ss[d];
  }
  const dim3 grid(static_cast<unsigned>(pl.splits), static_cast<unsigned>(pl.units));
  const dim3 cgrid(static_cast<unsigned>(p.Nq + (p.scores ? ceil_div(p.Nk, KEYS_PER_WG) : 0)),
                   static_cast<unsigned>(p.B * p.H));
  auto go = [&](auto hd) {
    constexpr int HD = decltype(hd)::value;
    switch (p.dtype) {
      case CAB_BF16: launch_dt<CAB_BF16, HD>(a, grid, ca, cgrid, s); break;
      case CAB_F16: launch_dt<CAB_F16, HD>(a, grid, ca, cgrid, s); break;
      default: launch_dt<CAB_F32, HD>(a, grid, ca, cgrid, s); break;
    }
  };
  if (p.D == 64)
    go(std::integral_constant<int, 64>{});
  else
    go(std::integral_constant<int, 128>{});
  return launch_status(fn);
}

}  // namespace cab
