// Sequence mixers over packed row chunks: whole-row q/k RMSNorm + paged
// cache append, masked (causal / chunk-local / banded) paged softmax
// attention for arbitrary head sizes, and the token-serial decayed
// outer-product recurrence with per-sequence fp32 state slots.
//
// Storage dtype S is bf16 (raw u16) or fp32; scores, softmax, decays and the
// recurrent state are fp32.
#include "common.h"
#include "mix_attn.h"

#include <type_traits>

namespace {

template <typename S> __device__ __forceinline__ float ldf(const S* p);
template <> __device__ __forceinline__ float ldf<u16>(const u16* p) { return bf2f(*p); }
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <typename S> __device__ __forceinline__ void stf(S* p, float v);
template <> __device__ __forceinline__ void stf<u16>(u16* p, float v) { *p = f2bf(v); }
template <> __device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }

// ---------------------------------------------------------------- qk norm
// One workgroup per row.  q row [nq], k row [nk], v row [nv]; caches
// [P, G, page, dk|dv]; slot = page_index*page + offset.  V = 4: 4-element
// vector accesses (sizes and strides multiples of 4), V = 1: scalar.
template <typename S, int V>
__device__ __forceinline__ void ldvs(const S* p, float (&o)[4]) {
  if (V == 4) {
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = 0.f;
    if constexpr (sizeof(S) == 2) {
      const s16x4 v = *reinterpret_cast<const s16x4*>(p);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = bf2f((u16)v[j]);
    } else {
      const f32x4 v = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = v[j];
    }
  } else {
    o[0] = ldf<S>(p);
    o[1] = o[2] = o[3] = 0.f;
  }
}
template <typename S, int V>
__device__ __forceinline__ void stvs(S* p, const float (&o)[4]) {
  if (V == 4) {
    if constexpr (sizeof(S) == 2) {
      s16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = (short)f2bf(o[j]);
      *reinterpret_cast<s16x4*>(p) = v;
    } else {
      *reinterpret_cast<f32x4*>(p) = f32x4{o[0], o[1], o[2], o[3]};
    }
  } else {
    stf<S>(p, o[0]);
  }
}

// Rows of up to R * 256 * V stay in registers, keys and values in the first RK rounds, and all
// that the kernel reads is asked for before the sums, without a branch between (rows of 2048
// and 1024: six 4.5 -> 3.6 us, 7636 30.3 -> 23.2; with a branch around the further rounds of
// the keys 7636 x 4096 / 2048 48, 41 without).  PART: waves past a row load nothing (7636 rows
// of 64 9.9 us in the loop, 11.6 with all threads loading; from 768 on all have a share, and
// the branch costs 0.15 us of 3).  R = 0: any length.  NORM: weights for either.
template <typename S, int V, int R, int RK, bool NORM, bool PART>
__global__ void __launch_bounds__(256) qk_norm_cache_kernel(
    S* __restrict__ qout, const S* __restrict__ q, const S* __restrict__ k,
    const S* __restrict__ v, const S* __restrict__ qw, const S* __restrict__ kw,
    S* __restrict__ kc, S* __restrict__ vc, const i64* __restrict__ slots,
    float eps, int nq, int nk, int nv, int G, int dk, int dv, int page,
    i64 ldq, i64 ldk, i64 ldv) {
  __shared__ float red[8];
  const int t = blockIdx.x;
  const S* qr = q + (size_t)t * ldq;
  const S* kr = k + (size_t)t * ldk;
  const S* vr = v + (size_t)t * ldv;
  // (no branch between the loads: without weights of its own a side reads its row again)
  const S* qwr = qw ? qw : qr;
  const S* kwr = kw ? kw : kr;
  constexpr int N = R > 0 ? R : 1;
  float fq[N][4], fk[N][4], fv[N][4], wq[N][4], wk[N][4];
  const i64 sl = slots[t];
  float sq = 0.f, sk = 0.f;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63);
  if (R > 0 && (!PART || wave * V < max(nq, max(nk, nv)))) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = (threadIdx.x + r * 256) * V;
      ldvs<S, V>(qr + min(i, nq - V), fq[r]);
      if (r < RK) ldvs<S, V>(kr + min(i, nk - V), fk[r]);
      if (r < RK) ldvs<S, V>(vr + min(i, nv - V), fv[r]);
      if (NORM) ldvs<S, V>(qwr + min(i, nq - V), wq[r]);
      if (NORM && r < RK) ldvs<S, V>(kwr + min(i, nk - V), wk[r]);
    }
  }
  if (R > 0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = (threadIdx.x + r * 256) * V;
#pragma unroll
      for (int j = 0; j < V; ++j) {
        if (i < nq) sq += fq[r][j] * fq[r][j];
        if (r < RK && i < nk) sk += fk[r][j] * fk[r][j];
      }
    }
  } else {
    for (int i = threadIdx.x * V; i < nq; i += 256 * V) {
      ldvs<S, V>(qr + i, fq[0]);
#pragma unroll
      for (int j = 0; j < V; ++j) sq += fq[0][j] * fq[0][j];
    }
    for (int i = threadIdx.x * V; i < nk; i += 256 * V) {
      ldvs<S, V>(kr + i, fk[0]);
#pragma unroll
      for (int j = 0; j < V; ++j) sk += fk[0][j] * fk[0][j];
    }
  }
  sq = wave_sum_f32(sq);
  sk = wave_sum_f32(sk);
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = sq;
    red[4 + (threadIdx.x >> 6)] = sk;
  }
  __syncthreads();
  const float rq = qw ? 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)nq + eps) : 1.0f;
  const float rk = kw ? 1.0f / sqrtf((red[4] + red[5] + red[6] + red[7]) / (float)nk + eps) : 1.0f;
  const i64 pg = sl / page, off = sl % page;
  auto put_q = [&](int i, float (&f)[4], const float (&w4)[4]) {
    if (NORM && qw) {
#pragma unroll
      for (int j = 0; j < V; ++j) f[j] *= rq * w4[j];
    }
    stvs<S, V>(qout + (size_t)t * nq + i, f);
  };
  auto put_k = [&](int i, float (&f)[4], const float (&w4)[4]) {
    const int g = i / dk, d = i % dk;
    if (NORM && kw) {
#pragma unroll
      for (int j = 0; j < V; ++j) f[j] *= rk * w4[j];
    }
    stvs<S, V>(kc + (((size_t)pg * G + g) * page + off) * dk + d, f);
  };
  auto put_v = [&](int i, const float (&f)[4]) {
    const int g = i / dv, d = i % dv;
    stvs<S, V>(vc + (((size_t)pg * G + g) * page + off) * dv + d, f);
  };
  if (R > 0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = (threadIdx.x + r * 256) * V;
      if (i < nq) put_q(i, fq[r], wq[r]);
      if (r < RK && i < nk && sl >= 0) put_k(i, fk[r], wk[r]);
      if (r < RK && i < nv && sl >= 0) put_v(i, fv[r]);
    }
    return;
  }
  for (int i = threadIdx.x * V; i < nq; i += 256 * V) {
    ldvs<S, V>(qr + i, fq[0]);
    if (NORM) ldvs<S, V>(qwr + i, wq[0]);
    put_q(i, fq[0], wq[0]);
  }
  if (sl < 0) return;
  for (int i = threadIdx.x * V; i < nk; i += 256 * V) {
    ldvs<S, V>(kr + i, fk[0]);
    if (NORM) ldvs<S, V>(kwr + i, wk[0]);
    put_k(i, fk[0], wk[0]);
  }
  for (int i = threadIdx.x * V; i < nv; i += 256 * V) {
    ldvs<S, V>(vr + i, fv[0]);
    put_v(i, fv[0]);
  }
}

// -------------------------------------------------------- masked attention
// One wave per (row, query head), 4 waves per workgroup.  Keys are walked in
// tiles of 64 (one key per lane for the scores, one output channel per lane
// for P.V), online softmax across tiles.  MAXV = ceil(dv/64) accumulators.
template <typename S, int MAXV>
__global__ void __launch_bounds__(256) masked_attention_kernel(
    S* __restrict__ out, const S* __restrict__ q, const S* __restrict__ kc,
    const S* __restrict__ vc, const i32* __restrict__ bt,
    const i32* __restrict__ row_seq, const i32* __restrict__ positions,
    float scale, int n_rh, int H, int G, int dk, int dv, int page, int maxp,
    int chunk, int window, i64 ldq, float* __restrict__ part_o,
    float* __restrict__ part_ml, AttnExtra ex) {
  extern __shared__ float smem[];           // [4][dk + 64]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int rh = blockIdx.x * 4 + wave;
  if (rh >= n_rh) return;                    // whole wave exits together
  float* qs = smem + wave * (dk + 64);
  float* ps = qs + dk;
  const int t = rh / H, h = rh % H;
  const int g = h / (H / G);
  const int GV = G / ex.vshare, gv = g / ex.vshare;
  const int pos = positions[t];
  const i32* btr = bt + (size_t)row_seq[t] * maxp;
  int lo = 0;
  if (chunk > 0) lo = (pos / chunk) * chunk;
  if (window > 0 && pos - window + 1 > lo) lo = pos - window + 1;
  // always-visible leading keys outside the window sit in front of it in a
  // virtual key index: [lo - nf, lo) stands for the keys [0, nf)
  const int nf = ex.first > 0 ? min(ex.first, lo) : 0;
  const int vsh = lo - nf;
  const S* qr = q + (size_t)t * ldq + (size_t)h * dk;
  for (int d = lane; d < dk; d += 64) qs[d] = ldf<S>(qr + d) * scale;
  float m = AF_NEG_INF, l = 0.f;
  if (ex.sink) { m = ex.sink[h]; l = 1.f; }
  const float r1 = ex.r1 ? ex.r1[h] : 0.f, r2 = ex.r1 ? ex.r2[h] : 0.f;
  float acc[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) acc[i] = 0.f;
  for (int j0 = vsh; j0 <= pos; j0 += 64) {
    const int jv = j0 + lane;
    const int j = jv < lo ? jv - vsh : jv;
    float s = AF_NEG_INF;
    if (jv <= pos) {
      const int pg = btr[j / page];
      const S* kr = kc + (((size_t)pg * G + g) * page + (j % page)) * dk;
      float d0 = 0.f;
      for (int d = 0; d < dk; ++d) d0 += qs[d] * ldf<S>(kr + d);
      s = attn_softcap(d0, ex.cap);
      if (ex.r1) s -= attn_dist_bias(r1, r2, pos - j);
    }
    const float mn = fmaxf(m, wave_max_f32(s));
    const float corr = (m <= AF_NEG_INF) ? 0.f : expf(m - mn);
    const float p = (jv <= pos) ? expf(s - mn) : 0.f;
    l = l * corr + wave_sum_f32(p);
    m = mn;
    __builtin_amdgcn_wave_barrier();
    ps[lane] = p;                            // wave-private LDS: ordered without a block barrier
    __builtin_amdgcn_wave_barrier();
    const int cnt = min(64, pos - j0 + 1);
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int d = lane + 64 * i;
      float a = acc[i] * corr;
      if (d < dv) {
        for (int jj = 0; jj < cnt; ++jj) {
          const int jk = (j0 + jj) < lo ? j0 + jj - vsh : j0 + jj;
          const int pg = btr[jk / page];
          a += ps[jj] * ldf<S>(vc + (((size_t)pg * GV + gv) * page + (jk % page)) * ex.ldv + d);
        }
      }
      acc[i] = a;
    }
  }
  if (part_o) {                              // one unnormalised part per row
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int d = lane + 64 * i;
      if (d < dv) part_o[(size_t)rh * dv + d] = acc[i];
    }
    if (lane == 0) {
      part_ml[(size_t)rh * 2] = m;
      part_ml[(size_t)rh * 2 + 1] = l;
    }
    return;
  }
  const float inv = attn_head_gate<S>(ex, t, h) / l;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int d = lane + 64 * i;
    if (d < dv) stf<S>(out + (size_t)t * ex.ldo + (size_t)h * dv + d, acc[i] * inv);
  }
}

// ------------------------------------------------ row attention (decode)
// One workgroup per (row, K/V head): the GQ query heads of the group share
// every K and V load.  Keys are walked in super-tiles of `kt`:
//   A. scores: a key row is read by adjacent lanes, 16 bytes each, as the value
//      rows are: its lines are fetched whole and once, where one key per lane
//      walked 64 rows at a time and lost lines between its reads of them.  The
//      query slices stay in registers; partial dot products meet in lane swaps
//      and DPP, a lane ends with its share of them (scattered_sums).  One score
//      per (head, key) in LDS, beside the key's page;
//   B. per head: bias and cap, max, exp, sum over the tile (running max / sum /
//      rescale factor kept in LDS across super-tiles);
//   C. P.V: a value row is read by LPV adjacent lanes, each lane accumulates
//      its 16-byte slice for every head in registers.
// The partial outputs of the key groups are summed with lane swaps and DPP, across
// waves through LDS.  Serves decode steps and short prompt portions, bf16
// and fp32 storage; head sizes up to 64 lanes x 16 bytes.
// Few rows are bound by the chain position, block table, K, scores, V: its branches
// on the lane layout and the page size stand outside the unrolled loops, and no
// division is in it.  Eight key or value rows in flight per lane, or the next value rows
// asked for ahead, cost more in wavefronts than they hid; with eight heads in bf16 two key
// rows leave registers for a second wavefront.  Rows of 128 elements with the merge, one
// key per lane -> adjacent lanes, us (diff: both maps of 16 heads):
//     query / K/V heads    6 x 300 keys  6 x 1000     6 x 4000     128 x 1000
//     bf16  8 / 8          14.3 -> 10.9  20.3 -> 12.4 45.6 -> 25.1 142 -> 93
//          16 / 8          16.2 -> 11.9  22.3 -> 14.0 48.6 -> 26.8 145 -> 95
//          32 / 8          27.5 -> 14.4  32.9 -> 16.9 66.8 -> 32.0 202 -> 109
//          diff 16 / 8     32.2 -> 15.1  43.2 -> 21.2 87.7 -> 37.3 498 -> 147
//          diff 16 / 4     47.6 -> 20.5  54.4 -> 22.7 102 -> 44.5  275 -> 119
//     fp32 16 / 8          15.7 -> 13.1  26.5 -> 16.9 60.4 -> 38.6 228 -> 178
//          32 / 8          18.6 -> 15.8  28.9 -> 19.3 62.7 -> 42.5 238 -> 180
//          16 / 2          38.0 -> 21.3  41.5 -> 21.5 88.2 -> 51.2 123 -> 80
// 128 rows of 3000 keys, 16 / 8 heads, 398 -> 289 us (5.4 TB/s).  Of 4382 shapes the worst are
// fp32 heads of 33, 90 or 130 elements in groups of six, up to 1.1 of the time before.

// Sixteen bytes of a row in storage type, for loads that stay in flight across other work;
// zeros past the row's end.
template <typename S, bool VEC>
struct RawSlice {
  static constexpr int EPL = 16 / sizeof(S);
  union { f32x4 v; S e[EPL]; };
  __device__ __forceinline__ void load(const S* row, int e0, int n, bool wide = true) {
    if (VEC && wide) {
      v = *reinterpret_cast<const f32x4*>(row + min(e0, n - EPL));
    } else {
#pragma unroll
      for (int j = 0; j < EPL; ++j) e[j] = row[min(e0 + j, n - 1)];
    }
  }
  __device__ __forceinline__ void floats(int e0, int n, float (&o)[EPL]) const {
#pragma unroll
    for (int j = 0; j < EPL; ++j) o[j] = e0 + (VEC ? 0 : j) < n ? ldf<S>(e + j) : 0.f;
  }
};

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float add_half_f32(float v) {      // the other 32 lanes
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v),
                                                  false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
__device__ __forceinline__ float add_quarter_f32(float v) {   // the other 16 of 32 lanes
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v),
                                                  false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

// One level of sums over lanes that differ in bit B of their number (mirrored within 16 lanes):
// a lane without the bit gets a's sum, one with it b's.
template <int B>
__device__ __forceinline__ float meet(float a, float b, int lane) {
  if constexpr (B == 5 || B == 4) {
    const uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
    const auto r = B == 5 ? __builtin_amdgcn_permlane32_swap(x, y, false, false)
                          : __builtin_amdgcn_permlane16_swap(x, y, false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  } else {
    const bool has = lane >> B & 1;
    return (has ? b : a) + dpp_f32<B == 3 ? 0x140 : B == 2 ? 0x141 : B == 1 ? 0x4E : 0xB1>(
                               has ? a : b);
  }
}

// Sums of N values over groups of 1 << LOG2 adjacent lanes, each lane's share of them: value
// i of a lane is that of index i << min(LOG2, log2 N) | its number's low LOG2 bits reversed
// (the low ones of these where N is smaller).  Of every two values a lane hands its partner the
// one that the partner goes on with: N additions where every lane's adding up all N takes
// N * LOG2, half rate most of them (one row of 300 keys, 32 heads of 192 over 8 in fp32 23.8 ->
// 19.8 us).
template <int LOG2, int M, int N>
__device__ __forceinline__ void scattered_sums(float (&v)[N], int lane) {
  if constexpr (LOG2 > 0) {
    constexpr int HALF = M > 1 ? M / 2 : 1;
#pragma unroll
    for (int i = 0; i < HALF; ++i)
      v[i] = M > 1 ? meet<LOG2 - 1>(v[2 * i], v[2 * i + 1], lane)
                   : meet<LOG2 - 1>(v[i], v[i], lane);
    scattered_sums<LOG2 - 1, HALF>(v, lane);
  }
}

// Each value's sum over the lanes with the same low log2 bits of their number, in each of them
// (the branches, which all lanes take together, once for all N values).
template <int N>
__device__ __forceinline__ void strided_sums(float (&v)[N], int log2) {
#define EACH(...) do { _Pragma("unroll") for (int i = 0; i < N; ++i) __VA_ARGS__; } while (0)
  if (log2 < 6) EACH(v[i] = add_half_f32(v[i]));
  if (log2 < 5) EACH(v[i] = add_quarter_f32(v[i]));
  // rotations within 16 lanes, whose halves, quarters, ... are alike by then
  if (log2 < 4) EACH(v[i] += dpp_f32<0x128>(v[i]));
  if (log2 < 3) EACH(v[i] += dpp_f32<0x124>(v[i]));
  if (log2 < 2) EACH(v[i] += dpp_f32<0x122>(v[i]));
  if (log2 < 1) EACH(v[i] += dpp_f32<0x121>(v[i]));
#undef EACH
}

// NK = 2 (differential attention, ex.vshare == 2): the workgroup's heads are
// both maps of one value head, the first half on key head 2 gv, the second on
// 2 gv + 1, so that a value row is read once for both; grid.y and G count
// value heads, H all query heads.
template <typename S, int GQ, bool VEC, int NK = 1>
__global__ void __launch_bounds__(256, sizeof(S) == 2 && VEC && GQ == 4 ? 3 : 1) attn_rows_kernel(
    S* __restrict__ out, const S* __restrict__ q, const S* __restrict__ kc,
    const S* __restrict__ vc, const i32* __restrict__ bt,
    const i32* __restrict__ row_seq, const i32* __restrict__ positions,
    float scale, int H, int G, int hpg, int dk, int dv, int page, int page_log2,
    int q_wide, int maxp, int chunk, int window, i64 ldq, int lpk_log2, int lpv_log2,
    int kt, int nsplit,
    float* __restrict__ part_o, float* __restrict__ part_ml, AttnExtra ex) {
  // nsplit > 1: the visible keys are cut into nsplit ranges, one workgroup
  // each (grid.z = head blocks x nsplit).  With part_o, unnormalised outputs
  // and (max, sum) go to part_o [T, H, nsplit, dv] / part_ml [T, H, nsplit,
  // 2] for attn_split_combine_kernel (or diff_combine_kernel) to merge.
  constexpr int EPL = 16 / sizeof(S);
  // key and value rows in flight per lane
  constexpr int UK = sizeof(S) == 2 && GQ == 8 ? 2 : 4, UV = 4;
  extern __shared__ float smem[];
  const int dvp = EPL << lpv_log2;             // padded value width
  float* sc = smem;                            // [GQ][kt] scores, then probabilities
  float* red = sc + GQ * kt;                   // [4][GQ][dvp]
  float* m_run = red + 4 * GQ * dvp;           // [8]
  float* l_run = m_run + 8;                    // [8]
  float* corr = l_run + 8;                     // [8]
  float* r1s = corr + 8;                       // [8] distance-bias factors
  float* r2s = r1s + 8;                        // [8]
  i32* pgs = reinterpret_cast<i32*>(r2s + 8);  // [kt] pages of the tile's keys
  const int t = blockIdx.x, g = blockIdx.y;
  const bool own = NK == 2 || ex.vshare == 1;
  const int GV = own ? G : G / ex.vshare, gv = own ? g : g / ex.vshare;
  const int zh = (int)gridDim.z == nsplit ? 0 : blockIdx.z / nsplit;
  const int sp = blockIdx.z - zh * nsplit;
  const int h0 = g * hpg + zh * GQ;
  const int nh = min(GQ, hpg - zh * GQ);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lik = lane & ((1 << lpk_log2) - 1), kik = lane >> lpk_log2;
  const int kpk = 64 >> lpk_log2;
  const int liv = lane & ((1 << lpv_log2) - 1), kiv = lane >> lpv_log2;
  const int kpv = 64 >> lpv_log2;
  RawSlice<S, VEC> qr[GQ];                     // the lane's slice of each query
#pragma unroll
  for (int gg = 0; gg < GQ; ++gg)
    qr[gg].load(q + (size_t)t * ldq + (size_t)(h0 + min(gg, nh - 1)) * dk, lik * EPL, dk,
                q_wide);
  int pos = positions[t];
  const int qpos = pos;
  const i32* btr = bt + (size_t)row_seq[t] * maxp;
  int lo = 0;
  if (chunk > 0) lo = (pos / chunk) * chunk;
  if (window > 0 && pos - window + 1 > lo) lo = pos - window + 1;
  // always-visible leading keys outside the window sit in front of it in a
  // virtual key index: [wlo - nf, wlo) stands for the keys [0, nf)
  const int wlo = lo;
  const int vsh = lo - (ex.first > 0 ? min(ex.first, lo) : 0);
  lo = vsh;
  if (nsplit > 1) {   // this workgroup's share of [lo, pos]; may be empty
    const int per = (pos - lo + nsplit) / nsplit;
    lo += sp * per;
    pos = min(pos, lo + per - 1);
  }

  // where keys of the tile (virtual indexes, see above) lie: their page's place in the
  // block table and the place in it.  A page is a power of two of keys as a rule.
  auto places = [&](auto& jv, auto& at) {
    constexpr int N = sizeof(jv) / sizeof(int);
#pragma unroll
    for (int u = 0; u < N; ++u) jv[u] = jv[u] < wlo ? jv[u] - vsh : jv[u];
    if (page_log2 >= 0) {
#pragma unroll
      for (int u = 0; u < N; ++u) { at[u] = jv[u] & (page - 1); jv[u] >>= page_log2; }
    } else {
#pragma unroll
      for (int u = 0; u < N; ++u) { at[u] = jv[u] % page; jv[u] /= page; }
    }
  };
  float acc[GQ][EPL];
#pragma unroll
  for (int gg = 0; gg < GQ; ++gg)
#pragma unroll
    for (int j = 0; j < EPL; ++j) acc[gg][j] = 0.f;
  if (threadIdx.x < GQ) {
    // the sink joins the first key range only
    const bool sk = ex.sink && sp == 0 && (int)threadIdx.x < nh;
    m_run[threadIdx.x] = sk ? ex.sink[h0 + threadIdx.x] : AF_NEG_INF;
    l_run[threadIdx.x] = sk ? 1.f : 0.f;
    const bool rb = ex.r1 && (int)threadIdx.x < nh;
    r1s[threadIdx.x] = rb ? ex.r1[h0 + threadIdx.x] : 0.f;
    r2s[threadIdx.x] = rb ? ex.r2[h0 + threadIdx.x] : 0.f;
  }

  for (int tile0 = lo; tile0 <= pos; tile0 += kt) {
    const int nk = min(kt, pos + 1 - tile0);
    // ---- A: scores, a key's row over adjacent lanes ----
    int pgk[UK], atk[UK];
    auto look_up = [&](int kb) {
      int pi[UK];
#pragma unroll
      for (int u = 0; u < UK; ++u) pi[u] = tile0 + min(kb + u * 4 * kpk + kik, nk - 1);
      places(pi, atk);
#pragma unroll
      for (int u = 0; u < UK; ++u) pgk[u] = btr[pi[u]];
    };
    if (wave * kpk < nk) look_up(wave * kpk);
    for (int kb = wave * kpk; kb < nk; kb += 4 * UK * kpk) {
      RawSlice<S, VEC> kk[UK][NK];
#pragma unroll
      for (int u = 0; u < UK; ++u) {
        const S* kr = kc + (((size_t)pgk[u] * G + g) * NK * page + atk[u]) * dk;
#pragma unroll
        for (int m = 0; m < NK; ++m)           // the second map's rows lie behind the first's
          kk[u][m].load(kr + (size_t)m * page * dk, lik * EPL, dk);
        if (lik == 0) pgs[min(kb + u * 4 * kpk + kik, nk - 1)] = pgk[u];
      }
      if (kb + 4 * UK * kpk < nk) look_up(kb + 4 * UK * kpk);
      float qv[GQ][EPL];
#pragma unroll
      for (int gg = 0; gg < GQ; ++gg) qr[gg].floats(lik * EPL, dk, qv[gg]);
      float a[UK * GQ];
#pragma unroll
      for (int u = 0; u < UK; ++u) {
        float kf[NK][EPL];
#pragma unroll
        for (int m = 0; m < NK; ++m) kk[u][m].floats(lik * EPL, dk, kf[m]);
#pragma unroll
        for (int gg = 0; gg < GQ; ++gg) {
          const float (&kg)[EPL] = kf[gg / (GQ / NK)];
          a[u * GQ + gg] = 0.f;
#pragma unroll
          for (int e = 0; e < EPL; ++e) a[u * GQ + gg] += qv[gg][e] * kg[e];
        }
      }
      // a lane's share of the sums goes to LDS
      auto scatter = [&](auto log2) {
        constexpr int L = decltype(log2)::value, N = UK * GQ;
        constexpr int LN = N >= 32 ? 5 : N >= 16 ? 4 : N >= 8 ? 3 : 2, LS = L < LN ? L : LN;
        scattered_sums<L, N>(a, lane);
        int l = lik;
        asm volatile("" : "+v"(l));   // places in LDS of no layout are kept across rounds
        if (L > LN && (l & ((1 << (L - LS)) - 1))) return;
        const int mine = L > 0 ? (int)(__brev(l) >> (32 - L)) & ((1 << LS) - 1) : 0;
#pragma unroll
        for (int i = 0; i < N >> LS; ++i) {
          const int at = i << LS | mine, gg = at % GQ, kidx = kb + at / GQ * 4 * kpk + kik;
          if (kidx < nk) sc[gg * kt + kidx] = a[i] * scale;
        }
      };
      if (lpk_log2 == 4) scatter(std::integral_constant<int, 4>());
      else if (lpk_log2 == 3) scatter(std::integral_constant<int, 3>());
      else if (lpk_log2 == 5) scatter(std::integral_constant<int, 5>());
      else if (lpk_log2 == 6) scatter(std::integral_constant<int, 6>());
      else if (lpk_log2 == 2) scatter(std::integral_constant<int, 2>());
      else if (lpk_log2 == 1) scatter(std::integral_constant<int, 1>());
      else scatter(std::integral_constant<int, 0>());
    }
    __syncthreads();
    // ---- B: softmax statistics, wave w takes heads w, w+4, ... ----
    for (int gg = wave; gg < nh; gg += 4) {
      float* sr = sc + gg * kt;
      float mx = AF_NEG_INF;
      for (int i = lane; i < nk; i += 64) {
        float sv = sr[i];
        if (ex.cap > 0.f || ex.r1) {
          const int jv = tile0 + i;
          sv = attn_softcap(sv, ex.cap);
          if (ex.r1) sv -= attn_dist_bias(r1s[gg], r2s[gg], qpos - (jv < wlo ? jv - vsh : jv));
          sr[i] = sv;
        }
        mx = fmaxf(mx, sv);
      }
      mx = wave_max_f32(mx);
      const float m_old = m_run[gg];
      const float m_new = fmaxf(m_old, mx);
      float sum = 0.f;
      for (int i = lane; i < nk; i += 64) {
        const float p = expf(sr[i] - m_new);
        sr[i] = p;
        sum += p;
      }
      sum = wave_sum_f32(sum);
      if (lane == 0) {
        const float c = (m_old <= AF_NEG_INF) ? 0.f : expf(m_old - m_new);
        corr[gg] = c;
        l_run[gg] = l_run[gg] * c + sum;
        m_run[gg] = m_new;
      }
    }
    __syncthreads();
    // ---- C: accumulate P.V ----
    if (tile0 > lo) {
#pragma unroll
      for (int gg = 0; gg < GQ; ++gg) {
        const float c = gg < nh ? corr[gg] : 0.f;
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[gg][e] *= c;
      }
    }
    for (int kb = wave * kpv; kb < nk; kb += 4 * UV * kpv) {
      RawSlice<S, VEC> vv[UV];
      int pi[UV], at[UV];
#pragma unroll
      for (int u = 0; u < UV; ++u) pi[u] = tile0 + min(kb + u * 4 * kpv + kiv, nk - 1);
      places(pi, at);
#pragma unroll
      for (int u = 0; u < UV; ++u) {
        const int pg = pgs[min(kb + u * 4 * kpv + kiv, nk - 1)];
        vv[u].load(vc + (((size_t)pg * GV + gv) * page + at[u]) * ex.ldv, liv * EPL, dv);
      }
#pragma unroll
      for (int u = 0; u < UV; ++u) {
        const int kidx = kb + u * 4 * kpv + kiv;
        const bool valid = kidx < nk;
        float vf[EPL];
        vv[u].floats(liv * EPL, dv, vf);
#pragma unroll
        for (int gg = 0; gg < GQ; ++gg) {
          const float p = (valid && gg < nh) ? sc[gg * kt + kidx] : 0.f;
#pragma unroll
          for (int e = 0; e < EPL; ++e) acc[gg][e] += p * vf[e];
        }
      }
    }
    __syncthreads();   // scores of this tile are dead; next tile may overwrite
  }
  // ---- sum the key groups of a wave, then the 4 waves ----
#pragma unroll
  for (int gg = 0; gg < GQ; ++gg) strided_sums(acc[gg], lpv_log2);
  if (kiv == 0) {
#pragma unroll
    for (int gg = 0; gg < GQ; ++gg)
#pragma unroll
      for (int e = 0; e < EPL; ++e)
        red[(wave * GQ + gg) * dvp + liv * EPL + e] = acc[gg][e];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nh * dv; i += 256) {
    const int gg = i / dv, d = i % dv;
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) o += red[(w * GQ + gg) * dvp + d];
    if (!part_o)
      stf<S>(out + (size_t)t * ex.ldo + (size_t)(h0 + gg) * dv + d,
             o / l_run[gg] * attn_head_gate<S>(ex, t, h0 + gg));
    else
      part_o[(((size_t)t * H + h0 + gg) * nsplit + sp) * dv + d] = o;
  }
  if (part_o && threadIdx.x < nh) {
    float* ml = part_ml + (((size_t)t * H + h0 + threadIdx.x) * nsplit + sp) * 2;
    ml[0] = m_run[threadIdx.x];
    ml[1] = l_run[threadIdx.x];
  }
}

// One wave per (row, head): merge the nsplit (<= 64) partial softmaxes.
// Lane s weighs split s once; empty splits (max = -inf) weigh nothing and their partial
// outputs are not added.  Eight splits' are asked for together: one wait, not one each.
template <typename S>
__global__ void __launch_bounds__(256) attn_split_combine_kernel(
    S* __restrict__ out, const float* __restrict__ part_o,
    const float* __restrict__ part_ml, int n_rh, int H, int nsplit, int dv,
    AttnExtra ex) {
  const int rh = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (rh >= n_rh) return;
  const int t = rh / H, h = rh % H;
  const int lane = threadIdx.x & 63;
  const float* ml = part_ml + (size_t)rh * nsplit * 2;
  const float ms = lane < nsplit ? ml[2 * lane] : AF_NEG_INF;
  const float ls = lane < nsplit ? ml[2 * lane + 1] : 0.f;
  const float m = wave_max_f32(ms);
  const float w = ms > AF_NEG_INF ? expf(ms - m) : 0.f;
  const float inv = attn_head_gate<S>(ex, t, h) / wave_sum_f32(w * ls);
  S* orow = out + (size_t)t * ex.ldo + (size_t)h * dv;
  for (int d0 = 0; d0 < dv; d0 += 64) {
    const int d = d0 + lane;
    const float* po = part_o + (size_t)rh * nsplit * dv + min(d, dv - 1);
    float o = 0.f;
    for (int s0 = 0; s0 < nsplit; s0 += 8) {
      float p[8];   // an empty split's may hold anything, and is not added
#pragma unroll
      for (int u = 0; u < 8; ++u) p[u] = po[(size_t)min(s0 + u, nsplit - 1) * dv];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float ws = s0 + u < nsplit ? __shfl(w, s0 + u, 64) : 0.f;
        if (ws > 0.f) o += p[u] * ws;
      }
    }
    if (d < dv) stf<S>(orow + d, o * inv);
  }
}

// One wave per (row, head of a differential attention): merge the key splits
// of both maps, o = a1 - lam a2, o <- o / rms(o) * (1 - diff), times
// sigmoid(gate) per element (gate null: none).  The maps' query heads are
// laid out [K/V head][map][head of the group].
template <typename S, int NV>
__global__ void __launch_bounds__(256) diff_combine_kernel(
    S* __restrict__ out, const float* __restrict__ part_o,
    const float* __restrict__ part_ml, const S* __restrict__ gate, i64 ldg,
    float lam, float diff, float eps, int n_rh, int H, int hpg, int nsplit,
    int dv) {
  const int rh = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (rh >= n_rh) return;
  const int lane = threadIdx.x & 63;
  const int t = rh / H, h = rh % H;
  const int g = h / hpg, hg = h % hpg;
  float o[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) o[i] = 0.f;
#pragma unroll
  for (int mp = 0; mp < 2; ++mp) {
    const size_t ph = (size_t)t * 2 * H + (size_t)(g * 2 + mp) * hpg + hg;
    const float* ml = part_ml + ph * nsplit * 2;
    const float ms = lane < nsplit ? ml[2 * lane] : AF_NEG_INF;
    const float ls = lane < nsplit ? ml[2 * lane + 1] : 0.f;
    const float m = wave_max_f32(ms);
    const float w = ms > AF_NEG_INF ? expf(ms - m) : 0.f;
    const float ws = (mp ? -lam : 1.0f) * w / wave_sum_f32(w * ls);
    for (int s0 = 0; s0 < nsplit; s0 += 4) {
      float p[4][NV];                          // empty splits' are not added
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < NV; ++i)
          p[u][i] = part_o[(ph * nsplit + min(s0 + u, nsplit - 1)) * dv +
                           min(i * 64 + lane, dv - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (s0 + u >= nsplit || __shfl(w, s0 + u, 64) <= 0.f) continue;
        const float wv = __shfl(ws, s0 + u, 64);
#pragma unroll
        for (int i = 0; i < NV; ++i)
          if (i * 64 + lane < dv) o[i] += wv * p[u][i];
      }
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) ss += o[i] * o[i];
  const float f = (1.0f - diff) / sqrtf(wave_sum_f32(ss) / (float)dv + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int d = i * 64 + lane;
    if (d >= dv) continue;
    float v = o[i] * f;
    if (gate) v /= 1.0f + expf(-ldf<S>(gate + (size_t)t * ldg + (size_t)h * dv + d));
    stf<S>(out + (size_t)rh * dv + d, v);
  }
}

// ------------------------------------------------------------- linear scan
// Workgroup = (sequence, head, 32-column tile of dv); 256 threads = 16 row
// groups x 16 column pairs, or 512 = 16 x 32 columns.  A thread keeps RP consecutive
// rows of its columns of the state in registers (each q / k / decay value read from
// LDS feeds both of two columns).  Tokens are walked serially in blocks of TB: the
// block's q / k / decay rows are staged into LDS at once (rotary + scaling applied on
// the way in), the recurrence itself is strictly token by token in fp32, and both kernels use the
// same operations (scan_*) and sum the 16 row groups in the same order — so they
// give the same bits, and results do not depend on how a sequence is cut into
// chunks or on what else is in the step.
//
// linear_scan_kernel, few tokens per sequence: bound by moving the state; thread
// (r, c) = (tid >> 4, tid & 15) has columns c and c + 16, so that a state row
// moves in 64-byte pieces; partial outputs meet in LDS after the block of tokens.
// linear_scan_prompt_kernel: with few workgroups bound by vector instructions, 28 per
// token and wave on two waves per SIMD beside the staging (a quarter); the row groups are
// the 16 lanes of a DPP row, so the sum over rows needs no LDS and no second barrier.  A
// constant decay is not staged.  Its workgroups are four or eight waves, see launch_scan.
// Six sequences of 620..1900 tokens, 8 heads of 128 x 128, decays per channel:
// 787 -> 277 us; 16 heads, one decay per head, rotary: 770 -> 296 us (the row layout alone
// 711 and 698; four waves, two columns per thread, 350 and 333; element loads that were
// converted at once made every block wait for its successor).
// The 16 row groups of a token are summed as a tree: j with 15 - j, of the eight sums j with
// 7 - j, of the four 0 with 2 and 1 with 3, then the two.  In a 16-lane row these are mirrors
// and exchanges within quads; row16_sum_all leaves the sum in all lanes.
__device__ __forceinline__ float row16_sum_all(float v) {
  v += dpp_f32<0x140>(v);
  v += dpp_f32<0x141>(v);
  v += dpp_f32<0x4E>(v);
  v += dpp_f32<0xB1>(v);
  return v;
}

// The same sums of a block of tokens, each lane one token's: of every two tokens (then sums of
// two, four and eight lanes) a lane hands its partner the one that the partner goes on with,
// 15 additions for 16 tokens instead of 64.  DPP operands run at half rate, so the sums were a
// quarter of the prompt kernel's vector time: one sequence of 1900 tokens, 16 heads of 128
// 284 -> 240 us; 6 of 620..1900, 8 heads with decays per channel 337 -> 308.  (Each two tokens
// at once, with three values waiting instead of eight, 315.)
template <int TB>
struct Row16Sums {
  float p[8], sum;
  // tokens tt = 0 .. TB-1 in turn, tt known when compiled; sum is the lane's after the last
  __device__ __forceinline__ void add(int tt, float part, int lane) {
    const bool b3 = lane & 8, b2 = lane & 4, b1 = lane & 2, b0 = lane & 1;
    p[tt & 7] = part;
    if ((tt & 7) != 7) return;
    float s[4], u[2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      s[t] = (b3 ? p[2 * t + 1] : p[2 * t]) + dpp_f32<0x140>(b3 ? p[2 * t] : p[2 * t + 1]);
#pragma unroll
    for (int t = 0; t < 2; ++t)
      u[t] = (b2 ? s[2 * t + 1] : s[2 * t]) + dpp_f32<0x141>(b2 ? s[2 * t] : s[2 * t + 1]);
    const float v = (b1 ? u[1] : u[0]) + dpp_f32<0x4E>(b1 ? u[0] : u[1]);
    if (TB == 8) sum = v + dpp_f32<0xB1>(v);
    else if (!(tt & 8)) sum = v;
    else sum = (b0 ? v : sum) + dpp_f32<0xB1>(b0 ? sum : v);
  }
  // the token whose sum a lane has (TB == 8: from 8 on, nobody's)
  static __device__ __forceinline__ int token_of(int lane) {
    return (lane >> 3 & 1) | (lane >> 1 & 2) | (lane << 1 & 4) | (lane << 3 & 8);
  }
};

// The arithmetic of both kernels, every rounding spelled out: contraction is the
// compiler's choice per place otherwise, and a sequence's results must not depend
// on which kernel its neighbours in the step selected.
__device__ __forceinline__ void scan_rotate(float& x, float partner, float cs,
                                            float sn, bool low) {
#pragma clang fp contract(off)
  // pair (u, w) -> (u cos - w sin, w cos + u sin)
  x = fmaf(x, cs, partner * (low ? -sn : sn));
}

template <bool FAST>
__device__ __forceinline__ void scan_angle(float pos, float freq, float& sn,
                                           float& cs) {
#pragma clang fp contract(off)
  const float ang = pos * freq;
  if (FAST) { sn = __sinf(ang); cs = __cosf(ang); }
  else sincosf(ang, &sn, &cs);
}

// sigmoid(z)^inv_tau; log(sigmoid(z)) = min(z, 0) - log(1 + exp(-|z|)) does not
// overflow
template <bool FAST>
__device__ __forceinline__ float scan_decay(float z, float inv_tau) {
#pragma clang fp contract(off)
  if (FAST) {
    // All of it to the base 2, by the instructions: 9 of them where __logf alone is 11 (its
    // argument needs no care, it lies in 1 .. 2).  6 sequences of 620..1900 tokens, 8 heads
    // 305 -> 277 us.  A state adds up the bias of its decays, so the first exponent has the
    // rest of LOG2E, without which that was 1.02 of what it is with __expf and __logf.
    // Relative errors against 64 bits, z of deviation 1, with these / here: mean 3, inv_tau
    // 1/16, bias -4.32e-9 / -4.27e-9, rms 1.803e-8 / 1.801e-8; mean 0, inv_tau 1, 1.40e-8 /
    // 1.12e-8, 5.72e-8 / 4.76e-8.
    constexpr float LOG2E = 1.44269504088896341f;
    constexpr float REST = (float)(1.44269504088896341 - (double)LOG2E);
    const float y = -fabsf(z);
    const float l = __builtin_amdgcn_logf(
        1.0f + __builtin_amdgcn_exp2f(fmaf(y, LOG2E, y * REST)));
    return __builtin_amdgcn_exp2f(fmaf(fminf(z, 0.f), LOG2E, -l) * inv_tau);
  }
  const float l = log1pf(expf(-fabsf(z)));
  return expf((fminf(z, 0.f) - l) * inv_tau);
}

// one row of one column, one token: the state, then its share of the output
__device__ __forceinline__ void scan_row(float& st, float& o, float a, float k,
                                         float v, float q) {
#pragma clang fp contract(off)
  st = fmaf(a, st, k * v);
  o = fmaf(st, q, o);
}

// SCAN_TB: tokens of a block, 16 (8: keeps LDS under 64 KB), or one for decode steps, which
// staged the other 15 for nothing and held LDS for them (16 heads of 128 x 128, 6 rows 6.6 ->
// 5.2 us, 64 rows 39.8 -> 26.8, 5 TB/s).
template <typename S, int RP, int SCAN_TB>
__global__ void __launch_bounds__(256) linear_scan_kernel(
    float* __restrict__ out, float* __restrict__ state,
    const S* __restrict__ q, const S* __restrict__ k, const S* __restrict__ v,
    const S* __restrict__ zl, const float* __restrict__ zbias,
    const float* __restrict__ head_decay, const float* __restrict__ inv_freq,
    const i32* __restrict__ positions, const i32* __restrict__ cu,
    const i32* __restrict__ q_start, const i32* __restrict__ sslot,
    float q_scale, float k_scale, float inv_tau, int H, int dk, int dv,
    int rot, i64 ldq, i64 ldk, i64 ldv, i64 ldz) {
  constexpr int DKP = 16 * RP;         // padded rows: zeros beyond dk
  // bf16 operands carry 2^-9 relative rounding already: hardware
  // transcendentals there; fp32 storage keeps the precise library forms
  constexpr bool FAST = sizeof(S) == 2;
  extern __shared__ float smem[];      // [TB][3][DKP] + [TB][16][32] + [TB][32]
  const int b = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 32;
  const int t0 = cu[b], t1 = cu[b + 1];
  if (t1 <= t0) return;
  const int r = threadIdx.x >> 4, cc = threadIdx.x & 15;
  const int ca = c0 + cc, cb = c0 + cc + 16;
  const bool oka = ca < dv, okb = cb < dv;
  float* stage = smem;                         // [TB][3][DKP]: q, k, decay
  float* part = smem + SCAN_TB * 3 * DKP;      // [TB][16][32]
  float* vs = part + SCAN_TB * 512;            // [TB][32]
  float* sbase = state + (((size_t)sslot[b] * H + h) * dk) * dv;
  float sta[RP], stb[RP];
  const bool fresh = q_start[b] == 0;
#pragma unroll
  for (int ii = 0; ii < RP; ++ii) {
    const int i = r * RP + ii;
    sta[ii] = (!fresh && oka && i < dk) ? sbase[(size_t)i * dv + ca] : 0.f;
    stb[ii] = (!fresh && okb && i < dk) ? sbase[(size_t)i * dv + cb] : 0.f;
  }
  const float hd = head_decay ? head_decay[h] : 1.0f;
  const int half = rot >> 1;
  // raw operands of the next block, fetched while the current one computes
  constexpr int EPT = (SCAN_TB * DKP + 255) / 256;   // staged elements per thread
  float rq[EPT], rk[EPT], rqp[EPT], rkp[EPT], rz[EPT], rpos[EPT];
  float rv[(SCAN_TB * 32 + 255) / 256];
  // Every load is unconditional on a clamped address (invalid lanes are
  // zeroed afterwards), so all of a block's loads are in flight together
  // instead of one exposed memory latency per guarded element.
  auto fetch = [&](int tb) {
    const int nt = min(SCAN_TB, t1 - tb);
#pragma unroll
    for (int n = 0; n < EPT; ++n) {
      const int e = threadIdx.x + 256 * n;
      const int tt = e / DKP, i = e % DKP;
      const bool valid = tt < nt && i < dk;
      const int t = tb + min(tt, nt - 1), ic = min(i, dk - 1);
      const float a = ldf<S>(q + (size_t)t * ldq + (size_t)h * dk + ic);
      const float c = ldf<S>(k + (size_t)t * ldk + (size_t)h * dk + ic);
      rq[n] = valid ? a : 0.f;
      rk[n] = valid ? c : 0.f;
      rqp[n] = rkp[n] = rz[n] = rpos[n] = 0.f;
    }
    if (rot > 0) {
#pragma unroll
      for (int n = 0; n < EPT; ++n) {
        const int e = threadIdx.x + 256 * n;
        const int tt = e / DKP, i = e % DKP;
        const int t = tb + min(tt, nt - 1), ic = min(i, dk - 1);
        const int pi = ic < half ? ic + half : (ic < rot ? ic - half : ic);
        rqp[n] = ldf<S>(q + (size_t)t * ldq + (size_t)h * dk + pi);
        rkp[n] = ldf<S>(k + (size_t)t * ldk + (size_t)h * dk + pi);
        rpos[n] = (float)positions[t];
      }
    }
    if (zl) {
#pragma unroll
      for (int n = 0; n < EPT; ++n) {
        const int e = threadIdx.x + 256 * n;
        const int tt = e / DKP, i = e % DKP;
        const int t = tb + min(tt, nt - 1), ic = min(i, dk - 1);
        rz[n] = ldf<S>(zl + (size_t)t * ldz + (size_t)h * dk + ic);
      }
    }
#pragma unroll
    for (int n = 0; n < (SCAN_TB * 32 + 255) / 256; ++n) {
      const int e = threadIdx.x + 256 * n;
      const int tt = e >> 5, ci = c0 + (e & 31);
      const float x = ldf<S>(v + (size_t)(tb + min(tt, nt - 1)) * ldv +
                             (size_t)h * dv + min(ci, dv - 1));
      rv[n] = (tt < nt && ci < dv) ? x : 0.f;
    }
  };
  fetch(t0);
  for (int tb = t0; tb < t1; tb += SCAN_TB) {
    const int nt = min(SCAN_TB, t1 - tb);
    // ---- stage the block: rotate / scale q, k; evaluate the decays ----
#pragma unroll
    for (int n = 0; n < EPT; ++n) {
      const int e = threadIdx.x + 256 * n;
      const int tt = e / DKP, i = e % DKP;
      float* row = stage + (size_t)tt * 3 * DKP;
      float qv = rq[n], kv = rk[n], a = 0.f;
      if (tt < nt && i < dk) {
        if (i < rot) {
          const bool lowh = i < half;
          float sn, cs;
          scan_angle<FAST>(rpos[n], inv_freq[lowh ? i : i - half], sn, cs);
          scan_rotate(qv, rqp[n], cs, sn, lowh);
          scan_rotate(kv, rkp[n], cs, sn, lowh);
        }
        qv *= q_scale;
        kv *= k_scale;
        a = hd;
        if (zl) {
          a = scan_decay<FAST>(rz[n] + zbias[(size_t)h * dk + i], inv_tau);
        }
      }
      if (tt < SCAN_TB) {
        row[i] = qv;
        row[DKP + i] = kv;
        row[2 * DKP + i] = a;
      }
    }
#pragma unroll
    for (int n = 0; n < (SCAN_TB * 32 + 255) / 256; ++n) {
      const int e = threadIdx.x + 256 * n;
      if (e < SCAN_TB * 32) vs[e] = rv[n];
    }
    __syncthreads();
    if (tb + SCAN_TB < t1) fetch(tb + SCAN_TB);   // in flight during compute
    // ---- advance this thread's rows through the block, token by token ----
    auto step = [&](int tt) {
      const f32x2* sq = reinterpret_cast<const f32x2*>(
          stage + (size_t)tt * 3 * DKP + r * RP);
      const f32x2* sk = sq + DKP / 2;
      const f32x2* sa = sk + DKP / 2;
      const float va = vs[tt * 32 + cc], vb = vs[tt * 32 + cc + 16];
      float pa = 0.f, pb = 0.f;
#pragma unroll
      for (int i2 = 0; i2 < RP / 2; ++i2) {
        const f32x2 a2 = sa[i2], k2 = sk[i2], q2 = sq[i2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int ii = i2 * 2 + j;
          scan_row(sta[ii], pa, a2[j], k2[j], va, q2[j]);
          scan_row(stb[ii], pb, a2[j], k2[j], vb, q2[j]);
        }
      }
      part[tt * 512 + r * 32 + cc] = pa;
      part[tt * 512 + r * 32 + cc + 16] = pb;
    };
    if (nt == SCAN_TB) {
      // full block: fixed trip count, so the LDS reads of later tokens are
      // scheduled under the arithmetic of earlier ones
#pragma unroll
      for (int tt = 0; tt < SCAN_TB; ++tt) step(tt);
    } else {
      for (int tt = 0; tt < nt; ++tt) step(tt);
    }
    __syncthreads();
    // ---- o[t][c] = sum of the 16 row-group partials ----
    for (int e = threadIdx.x; e < nt * 32; e += 256) {
      const int tt = e >> 5, ci = e & 31;
      if (c0 + ci < dv) {
        const float* pr = part + tt * 512 + ci;
        float o[8];   // summed in the order of row16_sum_all
#pragma unroll
        for (int rr = 0; rr < 8; ++rr) o[rr] = pr[rr * 32] + pr[(15 - rr) * 32];
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) o[rr] += o[7 - rr];
        out[(size_t)(tb + tt) * H * dv + (size_t)h * dv + c0 + ci] =
            (o[0] + o[2]) + (o[1] + o[3]);
      }
    }
    // the next block's staging writes `stage`/`vs`, last read before the
    // barrier above; its partials are written after the next barrier
  }
#pragma unroll
  for (int ii = 0; ii < RP; ++ii) {
    const int i = r * RP + ii;
    if (i < dk && oka) sbase[(size_t)i * dv + ca] = sta[ii];
    if (i < dk && okb) sbase[(size_t)i * dv + cb] = stb[ii];
  }
}

// Rows of a token that a thread of the prompt kernel stages
constexpr int scan_rows(int rp, int threads) {
  return (rp >= 16 ? 8 : 16) * 16 * rp / threads;
}

// The sequence of a workgroup, and its rows.  The grid walks sequence by sequence, and the
// longest comes first where that decides what shares a CU and what is left to the end:
// beyond one workgroup per CU (256).  With a head of every sequence in turn two of the
// longest met on one CU, or one started last, and where their number shares a factor with 8
// an XCD has some of them only: 6 sequences of 620..1900 tokens in 384 workgroups 430 -> 328
// us, 32 of up to 1500 in 2048 1173 -> 660 and, with decays per channel, 1312 -> 650.  A lane
// per sequence finds the ranks; more than 64 sequences keep their order (70 of up to 700
// tokens 864 -> 815, 995 -> 900).
// Below 64 tokens per sequence the look at the lengths, a load that the workgroup waits for,
// costs 1 us of 13, and the ranks more with every sequence: the host says where they pay, with
// up to 16 sequences whose lengths it knows to differ by 16 and up to 32 that differ by 64,
// unless they fall already (in order / longest first: 8 and 12 of 3..114 in any order 1.05, 17
// to 24 1.03 to 1.11, 32 1.01, 32 of 3..45 0.93; 8 of falling lengths 0.98, 24 0.94).  Else
// they keep their order, and up to 256 workgroups a head of every sequence in turn.  1440
// calls of 3..128 sequences against a head of each in turn everywhere: 0.80 of it in the mean
// (16 of 10..76, 16 heads of 256 x 256 165 -> 119 us, 64 of 25..75, 16 of 128 x 128 in fp32
// 257 -> 203), lengths alike 1.00, at most 1.04.
// at most a token each, unlike, the longest 1.25 of the mean (and 256 tokens in the mean)
enum ScanLengths { LENS_UNKNOWN, LENS_ONE, LENS_DIFFER, LENS_UNEVEN };
enum ScanWalk { HEADS_IN_TURN, IN_ORDER, LONGEST_FIRST, LONGEST_FIRST_SHORT };
struct ScanRows { int b, t0, t1; };
__device__ __forceinline__ ScanRows scan_sequence(const i32* __restrict__ cu, int walk) {
  const int B = gridDim.z, turn = blockIdx.z;
  if (walk == IN_ORDER || B > 64 || B * gridDim.x * gridDim.y <= 256)
    return {turn, cu[turn], cu[turn + 1]};
  const int lane = min((int)threadIdx.x & 63, B - 1);
  const int from = cu[lane], len = cu[lane + 1] - from;
  // (lengths alike: nothing to win, and the ranks cost short ones 1 us of 48)
  if (walk == LONGEST_FIRST &&
      __builtin_amdgcn_readfirstlane(wave_max_f32((float)len) +
                                     wave_max_f32((float)-len) < 64.f))
    return {turn, __builtin_amdgcn_readlane(from, turn),
            __builtin_amdgcn_readlane(from, turn) + __builtin_amdgcn_readlane(len, turn)};
  int rank = 0;
  for (int j = 0; j < B; ++j) {
    const int other = __builtin_amdgcn_readlane(len, j);
    rank += other > len || (other == len && j < lane);
  }
  const int b = __ffsll((unsigned long long)__ballot(rank == turn)) - 1;
  const int t0 = __builtin_amdgcn_readlane(from, b);
  return {b, t0, t0 + __builtin_amdgcn_readlane(len, b)};
}

// The same recurrence for prompts.  A thread stages E consecutive rows of one token
// (one wide load each for q, k, the rotary partners and the decay logits, kept raw
// until the block before has been worked through) and computes RP rows of one column
// (NT = 512) or two (256); each lane of a 16-lane row keeps one token's sum.  Two LDS
// buffers, one barrier per block of tokens.
// APART (NT = 512, 16 columns): four waves stage and four compute, one of each per SIMD.
// With few workgroups the longest sequence's tokens follow one another, each the arithmetic
// of two waves and then their staging (28 vector instructions each and a quarter); so it is
// the arithmetic of one, beside the staging: 140 -> 100 ns a token with decays per channel,
// 124 -> 87 with one per head.  Every column is staged for twice as often, which costs where
// the chip is full.  (All four waves of 16 columns staging 267 -> 226 us.)  One loop holds both
// roles, and the registers of both: in bf16 with decays per channel 18 more than the 128 of RP
// = 8 (68 bytes of scratch a lane), elsewhere none.
template <typename S, int RP, bool ZL, int NT, int COLS>
__global__ void __launch_bounds__(NT, RP == 8 && sizeof(S) == 2 ? (NT == 512 ? 4 : 3) : 2)
linear_scan_prompt_kernel(
    float* __restrict__ out, float* __restrict__ state,
    const S* __restrict__ q, const S* __restrict__ k, const S* __restrict__ v,
    const S* __restrict__ zl, const float* __restrict__ zbias,
    const float* __restrict__ head_decay, const float* __restrict__ inv_freq,
    const i32* __restrict__ positions, const i32* __restrict__ cu,
    const i32* __restrict__ q_start, const i32* __restrict__ sslot,
    float q_scale, float k_scale, float inv_tau, int H, int dk, int dv,
    int rot, i64 ldq, i64 ldk, i64 ldv, i64 ldz, int walk) {
  constexpr int DKP = 16 * RP;
  constexpr bool FAST = sizeof(S) == 2;
  constexpr int TB = RP >= 16 ? 8 : 16;
  constexpr bool APART = COLS == 16 && NT == 512;   // half of the waves stage
  constexpr int WORK = APART ? NT / 2 : NT;
  constexpr int CPT = 16 * COLS / WORK;        // columns per thread
  constexpr int E = scan_rows(RP, WORK);
  const bool stages = !APART || threadIdx.x >= WORK, walks = !APART || threadIdx.x < WORK;
  const int tid = APART ? threadIdx.x % WORK : threadIdx.x;
  constexpr int BUF = TB * (3 * DKP + COLS);   // [TB][3][DKP], [TB][COLS]
  extern __shared__ float smem[];
  const bool by_sequence = walk != HEADS_IN_TURN;
  const ScanRows rows = by_sequence ? scan_sequence(cu, walk)
                                    : ScanRows{(int)blockIdx.x, cu[blockIdx.x], cu[blockIdx.x + 1]};
  const int b = __builtin_amdgcn_readfirstlane(rows.b);   // (known to be alike in all lanes)
  const int t0 = __builtin_amdgcn_readfirstlane(rows.t0);
  const int t1 = __builtin_amdgcn_readfirstlane(rows.t1);
  const int h = by_sequence ? blockIdx.x : blockIdx.y;
  const int c0 = (by_sequence ? blockIdx.y : blockIdx.z) * COLS;
  if (t1 <= t0) return;
  const int r = tid & 15, cc = tid >> 4;
  const int ca = c0 + CPT * cc;
  float* sbase = state + (((size_t)sslot[b] * H + h) * dk) * dv;
  float state_of[CPT][RP];
  const bool fresh = q_start[b] == 0;
#pragma unroll
  for (int ii = 0; ii < RP; ++ii) {
    const int i = r * RP + ii;
#pragma unroll
    for (int c = 0; c < CPT; ++c)
      state_of[c][ii] = (!fresh && ca + c < dv && i < dk)
                            ? sbase[i * dv + ca + c] : 0.f;
  }

  // what this thread stages: rows i0 .. i0+E-1 of token st of a block, and two
  // columns of v of token vt
  struct Raw { S x[E]; };
  const int st = tid * E / DKP, i0 = tid * E % DKP;
  const int vt = tid / (COLS / 2), vc = c0 + 2 * (tid % (COLS / 2));
  const bool have = i0 < dk, turn = i0 < rot;
  const int half = rot >> 1, ic = have ? i0 : 0;
  const bool lowh = i0 < half;
  const int pi = !turn ? ic : lowh ? i0 + half : i0 - half;
  float frq[E], bias[E];
#pragma unroll
  for (int j = 0; j < E; ++j) {
    frq[j] = turn ? inv_freq[(lowh ? i0 : i0 - half) + j] : 0.f;
    bias[j] = ZL ? zbias[(size_t)h * dk + ic + j] : 0.f;
  }
  const float hd = head_decay ? head_decay[h] : 1.0f;
  const S* qh = q + (size_t)h * dk;
  const S* kh = k + (size_t)h * dk;
  const S* zh = ZL ? zl + (size_t)h * dk : nullptr;
  const S* vh = v + (size_t)h * dv;
  Raw rq, rk, rqp, rkp, rz;
  S rv[2];
  int rpos = 0;
  auto wide = [](const S* p) { return *reinterpret_cast<const Raw*>(
      __builtin_assume_aligned(p, sizeof(Raw) < 16 ? sizeof(Raw) : 16)); };
  auto fetch = [&](int tb) {                   // addresses clamped into the chunk
    const size_t t = min(tb + st, t1 - 1);
    rq = wide(qh + t * ldq + ic);
    rk = wide(kh + t * ldk + ic);
    if (rot > 0) {
      rqp = wide(qh + t * ldq + pi);
      rkp = wide(kh + t * ldk + pi);
      rpos = positions[t];
    }
    if (ZL) rz = wide(zh + t * ldz + ic);
    if (vt < TB) {
      const S* vp = vh + (size_t)min(tb + vt, t1 - 1) * ldv;
      rv[0] = vp[min(vc, dv - 1)];
      rv[1] = vp[min(vc + 1, dv - 1)];
    }
  };
  // rotate / scale q and k, evaluate the decays; rows and tokens beyond the end
  // are zeros
  auto fill = [&](int nt, float* stage) {
    float qv[E], kv[E], av[E];
    const bool valid = have && st < nt;
#pragma unroll
    for (int j = 0; j < E; ++j) {
      qv[j] = ldf<S>(&rq.x[j]);
      kv[j] = ldf<S>(&rk.x[j]);
      av[j] = hd;
    }
    if (rot > 0) {
#pragma unroll
      for (int j = 0; j < E; ++j) {
        float sn, cs;                     // angle 0 where nothing is rotated
        scan_angle<FAST>((float)rpos, frq[j], sn, cs);
        float x = qv[j], y = kv[j];
        scan_rotate(x, ldf<S>(&rqp.x[j]), cs, sn, lowh);
        scan_rotate(y, ldf<S>(&rkp.x[j]), cs, sn, lowh);
        qv[j] = turn ? x : qv[j];
        kv[j] = turn ? y : kv[j];
      }
    }
    if (ZL) {
#pragma unroll
      for (int j = 0; j < E; ++j)
        av[j] = scan_decay<FAST>(ldf<S>(&rz.x[j]) + bias[j], inv_tau);
    }
#pragma unroll
    for (int j = 0; j < E; ++j) {
      qv[j] = valid ? qv[j] * q_scale : 0.f;
      kv[j] = valid ? kv[j] * k_scale : 0.f;
      av[j] = valid ? av[j] : 0.f;
    }
    // four-row pieces of the 16 row groups side by side: a lane row reads 256
    // contiguous bytes
    float* row = stage + (size_t)st * 3 * DKP;
    if constexpr (RP >= 4) {
      const int g = i0 / RP, w0 = i0 % RP;
#pragma unroll
      for (int w = 0; w < E; w += 4) {
        const int at = (((w0 + w) >> 2) * 16 + g) * 4;
        *reinterpret_cast<f32x4*>(row + at) = f32x4{qv[w], qv[w + 1], qv[w + 2], qv[w + 3]};
        *reinterpret_cast<f32x4*>(row + DKP + at) = f32x4{kv[w], kv[w + 1], kv[w + 2], kv[w + 3]};
        if (ZL)
          *reinterpret_cast<f32x4*>(row + 2 * DKP + at) = f32x4{av[w], av[w + 1], av[w + 2], av[w + 3]};
      }
    } else {
#pragma unroll
      for (int w = 0; w < E; ++w) {
        row[i0 + w] = qv[w];
        row[DKP + i0 + w] = kv[w];
        if (ZL) row[2 * DKP + i0 + w] = av[w];
      }
    }
    if (vt < TB) {
      float* vr = stage + TB * 3 * DKP + vt * COLS + (vc - c0);
      vr[0] = vt < nt && vc < dv ? ldf<S>(&rv[0]) : 0.f;
      vr[1] = vt < nt && vc + 1 < dv ? ldf<S>(&rv[1]) : 0.f;
    }
  };
  if (stages) {
    fetch(t0);
    fill(min(TB, t1 - t0), smem);
    fetch(min(t0 + TB, t1 - 1));
  }
  __syncthreads();
  int cur = 0;
  for (int tb = t0; tb < t1; tb += TB) {
    const int nt = min(TB, t1 - tb);
    if (stages && tb + TB < t1) {
      fill(min(TB, t1 - tb - TB), smem + (cur ^ BUF));
      fetch(min(tb + 2 * TB, t1 - 1));         // in flight during the arithmetic
    }
    if (walks) {
    const float* sb = smem + cur;
    const float* vb = sb + TB * 3 * DKP;
    float o[CPT];
#pragma unroll
    for (int c = 0; c < CPT; ++c) o[c] = 0.f;
    struct Token { float q[RP], k[RP], a[RP], v[CPT]; };
    auto read = [&](int tt) {
      const float* sq = sb + (size_t)tt * 3 * DKP;
      Token t;
      if constexpr (RP >= 4) {
#pragma unroll
        for (int w = 0; w < RP; w += 4) {
          const int at = ((w >> 2) * 16 + r) * 4;
          const f32x4 q4 = *reinterpret_cast<const f32x4*>(sq + at);
          const f32x4 k4 = *reinterpret_cast<const f32x4*>(sq + DKP + at);
          f32x4 a4 = {hd, hd, hd, hd};
          if (ZL) a4 = *reinterpret_cast<const f32x4*>(sq + 2 * DKP + at);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            t.q[w + j] = q4[j];
            t.k[w + j] = k4[j];
            t.a[w + j] = a4[j];
          }
        }
      } else {
#pragma unroll
        for (int w = 0; w < RP; ++w) {
          t.q[w] = sq[r * RP + w];
          t.k[w] = sq[DKP + r * RP + w];
          t.a[w] = ZL ? sq[2 * DKP + r * RP + w] : hd;
        }
      }
      if constexpr (CPT == 2) {
        const f32x2 v = *reinterpret_cast<const f32x2*>(vb + tt * COLS + 2 * cc);
        t.v[0] = v[0];
        t.v[1] = v[1];
      } else {
        t.v[0] = vb[tt * COLS + cc];
      }
      return t;
    };
    auto step = [&](const Token& t, float (&part)[CPT]) {
#pragma unroll
      for (int c = 0; c < CPT; ++c) part[c] = 0.f;
#pragma unroll
      for (int ii = 0; ii < RP; ++ii)
#pragma unroll
        for (int c = 0; c < CPT; ++c)
          scan_row(state_of[c][ii], part[c], t.a[ii], t.k[ii], t.v[c], t.q[ii]);
    };
    // a lane keeps the sums of token `mine`
    const int mine = Row16Sums<TB>::token_of(r);
    if (nt == TB) {
      // the next token's LDS reads run under this one's arithmetic: the fence keeps
      // them there, the one or two waves of a SIMD do not hide them otherwise
      Token t[2];
      Row16Sums<TB> sums[CPT];
      t[0] = read(0);
#pragma unroll
      for (int tt = 0; tt < TB; ++tt) {
        if (tt + 1 < TB) t[(tt + 1) & 1] = read(tt + 1);
        __builtin_amdgcn_sched_barrier(0);
        float part[CPT];
        step(t[tt & 1], part);
#pragma unroll
        for (int c = 0; c < CPT; ++c) sums[c].add(tt, part[c], r);
      }
#pragma unroll
      for (int c = 0; c < CPT; ++c) o[c] = sums[c].sum;
    } else {
      for (int tt = 0; tt < nt; ++tt) {
        float part[CPT];
        step(read(tt), part);
#pragma unroll
        for (int c = 0; c < CPT; ++c) {
          part[c] = row16_sum_all(part[c]);
          o[c] = mine == tt ? part[c] : o[c];
        }
      }
    }
    if (mine < nt) {
      float* op = out + (size_t)(tb + mine) * H * dv + (size_t)h * dv;
#pragma unroll
      for (int c = 0; c < CPT; ++c)
        if (ca + c < dv) op[ca + c] = o[c];
    }
    }
    __syncthreads();  // the next buffer is filled, this one read
    cur ^= BUF;
  }
  if (!walks) return;
#pragma unroll
  for (int ii = 0; ii < RP; ++ii) {
    const int i = r * RP + ii;
#pragma unroll
    for (int c = 0; c < CPT; ++c)
      if (i < dk && ca + c < dv) sbase[i * dv + ca + c] = state_of[c][ii];
  }
}

}  // namespace

AF_EXPORT int afm_qk_norm_cache(
    void* qout, const void* q, const void* k, const void* v, const void* qw,
    const void* kw, void* kc, void* vc, const void* slots, float eps, int T,
    int nq, int nk, int nv, int G, int dk, int dv, int page, i64 ldq, i64 ldk,
    i64 ldv, int dt, void* stream) {
  if (T == 0) return 0;
  if (nk != G * dk || nv != G * dv) return 9003;
  hipStream_t s = (hipStream_t)stream;
  auto al = [](const void* p) { return p == nullptr || (uintptr_t)p % 16 == 0; };
  const bool vec = dk % 4 == 0 && dv % 4 == 0 && nq % 4 == 0 && ldq % 4 == 0 &&
                   ldk % 4 == 0 && ldv % 4 == 0 && al(qout) && al(q) && al(k) &&
                   al(v) && al(qw) && al(kw) && al(kc) && al(vc);
  const int wide = max(nq, max(nk, nv));
  const bool any = nq > 0 && nk > 0 && nv > 0;
  const int narrow = max(nk, nv);
#define QKN(ST, V, R, RK, NORM, PART)                                         \
  qk_norm_cache_kernel<ST, V, R, RK, NORM, PART><<<T, 256, 0, s>>>((ST*)qout, (const ST*)q, \
      (const ST*)k, (const ST*)v, (const ST*)qw, (const ST*)kw, (ST*)kc,      \
      (ST*)vc, (const i64*)slots, eps, nq, nk, nv, G, dk, dv, page, ldq, ldk, \
      ldv)
#define QKR(ST, NORM)                                                         \
  do {                                                                        \
    if (!vec) QKN(ST, 1, 0, 0, NORM, false);                                  \
    else if (!any || wide > 4096) QKN(ST, 4, 0, 0, NORM, false);              \
    else if (wide <= 768) QKN(ST, 4, 1, 1, NORM, true);                       \
    else if (wide <= 1024) QKN(ST, 4, 1, 1, NORM, false);                     \
    else if (wide <= 2048 && narrow <= 1024) QKN(ST, 4, 2, 1, NORM, false);   \
    else if (wide <= 2048) QKN(ST, 4, 2, 2, NORM, false);                     \
    else if (narrow <= 1024) QKN(ST, 4, 4, 1, NORM, false);                   \
    else if (narrow <= 2048) QKN(ST, 4, 4, 2, NORM, false);                   \
    else QKN(ST, 4, 4, 4, NORM, false);                                       \
  } while (0)
  if (dt != 0 && dt != 1) return 9002;
  if (qw || kw) { if (dt == 0) QKR(u16, true); else QKR(float, true); }
  else { if (dt == 0) QKR(u16, false); else QKR(float, false); }
#undef QKR
#undef QKN
  return af_last_err();
}

template <typename S>
static int launch_attention(void* out, const void* q, const void* kc,
                            const void* vc, const void* bt, const void* row_seq,
                            const void* positions, float scale, int T, int H,
                            int G, int dk, int dv, int page, int maxp,
                            int chunk, int window, i64 ldq, int nsplit,
                            float* part_o, float* part_ml, AttnExtra ex,
                            hipStream_t s) {
  constexpr int EPL = 16 / (int)sizeof(S);
  if (dk <= 64 * EPL && dv <= 64 * EPL) {
    auto clog2 = [](int n) { int l = 0; while ((1 << l) < n) ++l; return l; };
    const int lpk = clog2((dk + EPL - 1) / EPL), lpv = clog2((dv + EPL - 1) / EPL);
    // both maps of a value head in one workgroup when its heads fit exactly
    const int pq = ex.vshare == 2 ? H / G * 2 : 0;
    const bool both = pq == 2 || pq == 4 || pq == 8;
    if (both) G /= 2;
    const int hpg = H / G;
    const int gq = hpg >= 8 ? 8 : hpg > 2 ? 4 : hpg;   // 1, 2, 4 or 8
    const int dvp = EPL << lpv;
    const int kt = dvp <= 128 ? 1024 : 512;
    const size_t sm = ((size_t)gq * kt + 4 * gq * dvp + 40 + kt) * sizeof(float);
    const bool vec = dk % EPL == 0 && dv % EPL == 0 && ex.ldv % EPL == 0 &&
                     (uintptr_t)kc % 16 == 0 && (uintptr_t)vc % 16 == 0;
    const int q_wide = ldq % EPL == 0 && (uintptr_t)q % 16 == 0;
    const int pl2 = page & (page - 1) ? -1 : clog2(page);
    dim3 grid(T, G, ((hpg + gq - 1) / gq) * nsplit);
#define ROWS(GQ, ...)                                                         \
  attn_rows_kernel<S, GQ, __VA_ARGS__><<<grid, 256, sm, s>>>(                 \
      (S*)out, (const S*)q, (const S*)kc, (const S*)vc, (const i32*)bt,       \
      (const i32*)row_seq, (const i32*)positions, scale, H, G, hpg, dk, dv,    \
      page, pl2, q_wide, maxp, chunk, window, ldq, lpk, lpv, kt, nsplit,      \
      part_o, part_ml, ex)
    if (both) {
      if (vec) {
        if (gq == 2) ROWS(2, true, 2); else if (gq == 4) ROWS(4, true, 2);
        else ROWS(8, true, 2);
      } else {
        if (gq == 2) ROWS(2, false, 2); else if (gq == 4) ROWS(4, false, 2);
        else ROWS(8, false, 2);
      }
    } else if (vec) {
      if (gq == 1) ROWS(1, true); else if (gq == 2) ROWS(2, true);
      else if (gq == 4) ROWS(4, true); else ROWS(8, true);
    } else {
      if (gq == 1) ROWS(1, false); else if (gq == 2) ROWS(2, false);
      else if (gq == 4) ROWS(4, false); else ROWS(8, false);
    }
#undef ROWS
    if (nsplit > 1 && out)
      attn_split_combine_kernel<S><<<(T * H + 3) / 4, 256, 0, s>>>(
          (S*)out, part_o, part_ml, T * H, H, nsplit, dv, ex);
    return af_last_err();
  }
  // very wide heads: one wave per (row, head), scalar key walk, no key splits
  if (!out && nsplit > 1) return 9003;
  const int n_rh = T * H;
  const int grid = (n_rh + 3) / 4;
  const size_t sm = (size_t)4 * (dk + 64) * sizeof(float);
#define ATT(MV)                                                              \
  masked_attention_kernel<S, MV><<<grid, 256, sm, s>>>(                      \
      (S*)out, (const S*)q, (const S*)kc, (const S*)vc, (const i32*)bt,      \
      (const i32*)row_seq, (const i32*)positions, scale, n_rh, H, G, dk, dv, \
      page, maxp, chunk, window, ldq, out ? nullptr : part_o,                \
      out ? nullptr : part_ml, ex)
  if (dv <= 64) ATT(1);
  else if (dv <= 128) ATT(2);
  else if (dv <= 256) ATT(4);
  else if (dv <= 512) ATT(8);
  else ATT(16);
#undef ATT
  return af_last_err();
}

// out null: the unmerged partial softmaxes stay in part_o / part_ml.
AF_EXPORT int afm_masked_attention(
    void* out, const void* q, const void* kc, const void* vc, const void* bt,
    const void* row_seq, const void* positions, float scale, int T, int H,
    int G, int dk, int dv, int page, int maxp, int chunk, int window, i64 ldq,
    int nsplit, void* part_o, void* part_ml, const void* sink, float cap,
    const void* r1, const void* r2, i64 ldv, int keep_first, int vshare,
    const void* gate, i64 ldg, i64 ldo, int dt, void* stream) {
  if (T == 0) return 0;
  if (out && (ldo < (i64)H * dv || (gate && ldg < H))) return 9003;
  if (G <= 0 || H % G || dv > 1024 || dk > 2048) return 9003;
  if (vshare < 1 || G % vshare) return 9003;
  if (nsplit < 1 || nsplit > 64 ||
      ((nsplit > 1 || !out) && (!part_o || !part_ml))) return 9003;
  if (ldv < dv || cap < 0.f || ((r1 == nullptr) != (r2 == nullptr))) return 9003;
  if (keep_first < 0) return 9003;
  const AttnExtra ex{(const float*)sink, (const float*)r1, (const float*)r2,
                     cap, ldv, keep_first, vshare, gate, ldg, ldo};
  hipStream_t s = (hipStream_t)stream;
  if (dt == 0)
    return launch_attention<u16>(out, q, kc, vc, bt, row_seq, positions, scale,
                                 T, H, G, dk, dv, page, maxp, chunk, window,
                                 ldq, nsplit, (float*)part_o, (float*)part_ml,
                                 ex, s);
  if (dt == 1)
    return launch_attention<float>(out, q, kc, vc, bt, row_seq, positions,
                                   scale, T, H, G, dk, dv, page, maxp, chunk,
                                   window, ldq, nsplit, (float*)part_o,
                                   (float*)part_ml, ex, s);
  return 9002;
}

// out [T, H*dv] from the partial softmaxes of 2H query heads laid out [key
// head pair][map][head of the group] (part_o [T, 2H, nsplit, dv], part_ml
// [T, 2H, nsplit, 2]); hpg query heads per K/V head.
AF_EXPORT int afm_diff_combine(void* out, const void* part_o,
                               const void* part_ml, const void* gate, i64 ldg,
                               float lam, float diff, float eps, int T, int H,
                               int hpg, int nsplit, int dv, int dt,
                               void* stream) {
  if (T == 0) return 0;
  if (nsplit < 1 || nsplit > 64 || hpg < 1 || H % hpg) return 9003;
  hipStream_t s = (hipStream_t)stream;
  const int n_rh = T * H;
#define DC(ST, NV)                                                            \
  diff_combine_kernel<ST, NV><<<(n_rh + 3) / 4, 256, 0, s>>>((ST*)out,        \
      (const float*)part_o, (const float*)part_ml, (const ST*)gate, ldg, lam, \
      diff, eps, n_rh, H, hpg, nsplit, dv)
#define DCV(ST)                                                               \
  do {                                                                        \
    if (dv <= 64) DC(ST, 1);                                                  \
    else if (dv <= 128) DC(ST, 2);                                            \
    else if (dv <= 256) DC(ST, 4);                                            \
    else if (dv <= 512) DC(ST, 8);                                            \
    else DC(ST, 16);                                                          \
  } while (0)
  if (dv > 1024) return 9003;
  if (dt == 0) DCV(u16);
  else if (dt == 1) DCV(float);
  else return 9002;
#undef DCV
#undef DC
  return af_last_err();
}

// out [T, H*dv] at row stride ldo from part_o [T, H, nsplit, dv] / part_ml [T,
// H, nsplit, 2]; gate [T, H] logits at row stride ldg, or null.
AF_EXPORT int afm_attn_split_combine(void* out, const void* part_o,
                                     const void* part_ml, int T, int H,
                                     int nsplit, int dv, const void* gate,
                                     i64 ldg, i64 ldo, int dt, void* stream) {
  if (T == 0) return 0;
  if (nsplit < 1 || nsplit > 64 || H < 1) return 9003;
  if (ldo < (i64)H * dv || (gate && ldg < H)) return 9003;
  const int n_rh = T * H;
  AttnExtra ex{};
  ex.gate = gate;
  ex.ldg = ldg;
  ex.ldo = ldo;
  hipStream_t s = (hipStream_t)stream;
  if (dt == 0)
    attn_split_combine_kernel<u16><<<(n_rh + 3) / 4, 256, 0, s>>>(
        (u16*)out, (const float*)part_o, (const float*)part_ml, n_rh, H, nsplit, dv, ex);
  else if (dt == 1)
    attn_split_combine_kernel<float><<<(n_rh + 3) / 4, 256, 0, s>>>(
        (float*)out, (const float*)part_o, (const float*)part_ml, n_rh, H, nsplit, dv, ex);
  else
    return 9002;
  return af_last_err();
}

template <typename S>
static int launch_scan(float* out, float* state, const void* q, const void* k,
                       const void* v, const void* zl, const float* zbias,
                       const float* head_decay, const float* inv_freq,
                       const i32* positions, const i32* cu, const i32* q_start,
                       const i32* sslot, float q_scale, float k_scale,
                       float inv_tau, int T, int B, int H, int dk, int dv,
                       int rot, i64 ldq, i64 ldk, i64 ldv, i64 ldz, int known,
                       hipStream_t s) {
  dim3 grid(B, H, (dv + 31) / 32);
  const int rp = (dk + 15) / 16;
  const int rpp = rp <= 2 ? 2 : rp <= 4 ? 4 : rp <= 8 ? 8 : 16;
  // From a block of tokens per sequence on the prompt kernel is the better one
  // (see there); its loads take E rows at once, so heads, halves of the rotated
  // part, strides and bases must be multiples of E elements (16 bytes at most).
  auto loads = [&](int threads) {
    const int E = scan_rows(rpp, threads);
    const size_t al = E * sizeof(S) < 16 ? E * sizeof(S) : 16;
    return T >= 16 * B && B <= 65535 && dk % E == 0 && (rot / 2) % E == 0 && ldq % E == 0 &&
           ldk % E == 0 && (!zl || ldz % E == 0) && (uintptr_t)q % al == 0 &&
           (uintptr_t)k % al == 0 && (uintptr_t)zl % al == 0;
  };
  // From 128 rows on with eight waves, which fill one another's waits, while that leaves
  // a workgroup or two to a CU; beyond, four waves do it with fewer instructions.  Four /
  // eight waves in us, sequences of 300 tokens, 128 rows: decays per channel, 192 groups
  // 67 / 61, 384 95 / 97 (of 50..1900 tokens 350 / 318), 768 133 / 149, 4096 585 / 679; one
  // decay per head 61 / 50, 85 / 80, 118 / 122, 530 / 579; 256 rows, 64 groups 113 / 107,
  // 384 179 / 221.  fp32: 128 rows, 192 groups 101 / 82, 384 140 / 153; one decay per head
  // 73 / 55, 96 / 88, 768 133 / 136, 4096 609 / 640.  What only eight waves can load (rows in
  // fours) is, on many groups, better off with them than with the token kernel at 128 rows in
  // bf16 (dk 100, 17 tokens 27 / 25) and with one decay per head (fp32, dk 100, 560 groups, 17
  // tokens 22 / 19, 50 tokens 47 / 31, 100 tokens 87 / 47; dk 124 breaks even at 24),
  // otherwise for longer prompts (fp32 17 tokens 32 / 44, 75 tokens 97 / 98, 225 tokens
  // 265 / 253).
  i64 groups = (i64)B * H * grid.z;
  const bool few = groups <= (rpp >= 16 || (sizeof(S) == 4 && zl) ? 256 : 512);
  const bool eight = rpp >= 8 && loads(512) &&
                     (few || (!loads(256) && ((rpp == 8 && (sizeof(S) == 2 || !zl)) ||
                                              T >= 128 * B)));
  const bool prompt = eight || loads(256);
  // Half of eight waves staging for the other half, 16 columns to a workgroup, where the
  // longest sequences decide: up to a workgroup per CU of these, or three (of which two are
  // there at once) where the caller knows them to be uneven.  All waves staging / apart in us: one sequence of 1900 tokens, 8
  // heads of 128 x 128 with decays per channel 267 / 190, 16 heads, one decay per head 235 /
  // 165; 4 of 300..700, 4 heads of 64 x 64 79 / 47, 8 of 256 x 256 222 / 158, in fp32 8 of 128
  // x 128 161 / 135; 3 of 58..82 19.2 / 18.2, but 4 of 49..58 16.2 / 16.7.  6 of 500..1900,
  // 384 groups 277 / 228, all of 1900 273 / 287; 768 groups 365 / 346, 391 / 373; 8 of
  // 200..1000, 512 groups 147 / 133, 1024 189 / 193; 512 groups of 256 x 256 182 / 187, in
  // fp32 161 / 190.
  const i64 narrow = (i64)B * H * ((dv + 15) / 16);
  const bool apart =
      loads(256) && (i64)T >= 64 * (i64)B &&
      narrow <= (known == LENS_UNEVEN && sizeof(S) == 2 && rpp <= 8 ? 768 : 256);
  if (apart) {
    grid.z = (dv + 15) / 16;
    groups = narrow;
  }
  const dim3 ordered(H, grid.z, B);
  const int walk = (i64)T >= 64 * (i64)B ? LONGEST_FIRST    // see scan_sequence
                   : groups <= 256        ? HEADS_IN_TURN
                   : known == LENS_DIFFER ? LONGEST_FIRST_SHORT : IN_ORDER;
  // Only where the caller says so: as many tokens as sequences may be one sequence's (50 of 51
  // sequences, 16 heads of 16 x 32 11 us in blocks of 16, 47 one by one).
  const bool single = !prompt && known == LENS_ONE;
  const size_t sm = (size_t)(single ? 1 : rpp >= 16 ? 8 : 16) * sizeof(float) *
                    (prompt ? 2 * (3 * 16 * rpp + 32) : 3 * 16 * rpp + 512 + 32);
#define SCAN_ARGS                                                            \
      out, state, (const S*)q, (const S*)k, (const S*)v, (const S*)zl, zbias, \
      head_decay, inv_freq, positions, cu, q_start, sslot, q_scale, k_scale, \
      inv_tau, H, dk, dv, rot, ldq, ldk, ldv, ldz
#define SCAN_PROMPT(RP, NT, COLS)                                                \
  do {                                                                       \
    if (zl)                                                                  \
      linear_scan_prompt_kernel<S, RP, true, NT, COLS>                       \
          <<<walk ? ordered : grid, NT, sm, s>>>(SCAN_ARGS, walk);           \
    else                                                                     \
      linear_scan_prompt_kernel<S, RP, false, NT, COLS>                      \
          <<<walk ? ordered : grid, NT, sm, s>>>(SCAN_ARGS, walk);           \
  } while (0)
#define SCAN(RP)                                                             \
  do {                                                                       \
    if (apart) SCAN_PROMPT(RP, 512, 16);                                     \
    else if (eight) SCAN_PROMPT((RP >= 8 ? RP : 8), 512, 32);                \
    else if (prompt) SCAN_PROMPT(RP, 256, 32);                               \
    else if (single)                                                         \
      linear_scan_kernel<S, RP, 1><<<grid, 256, sm, s>>>(SCAN_ARGS);         \
    else                                                                     \
      linear_scan_kernel<S, RP, (RP >= 16 ? 8 : 16)>                         \
          <<<grid, 256, sm, s>>>(SCAN_ARGS);                                 \
  } while (0)
  if (rp <= 2) SCAN(2);
  else if (rp <= 4) SCAN(4);
  else if (rp <= 8) SCAN(8);
  else SCAN(16);
#undef SCAN
#undef SCAN_PROMPT
#undef SCAN_ARGS
  return af_last_err();
}

// known: what the caller knows of the lengths (ScanLengths; any lengths are right).
AF_EXPORT int afm_linear_scan(
    void* out, void* state, const void* q, const void* k, const void* v,
    const void* zl, const void* zbias, const void* head_decay,
    const void* inv_freq, const void* positions, const void* cu,
    const void* q_start, const void* sslot, float q_scale, float k_scale,
    float inv_tau, int T, int B, int H, int dk, int dv, int rot, i64 ldq,
    i64 ldk, i64 ldv, i64 ldz, int dt, int known, void* stream) {
  if (B == 0) return 0;
  if (dk > 256 || dk < 1 || dv < 1) return 9003;
  if (rot < 0 || rot > dk || (rot & 1) || (rot && !inv_freq)) return 9003;
  if ((zl == nullptr) == (head_decay == nullptr)) return 9003;
  if (zl && !zbias) return 9003;
  hipStream_t s = (hipStream_t)stream;
  if (dt == 0)
    return launch_scan<u16>((float*)out, (float*)state, q, k, v, zl,
        (const float*)zbias, (const float*)head_decay, (const float*)inv_freq,
        (const i32*)positions, (const i32*)cu, (const i32*)q_start,
        (const i32*)sslot, q_scale, k_scale, inv_tau, T, B, H, dk, dv, rot,
        ldq, ldk, ldv, ldz, known, s);
  if (dt == 1)
    return launch_scan<float>((float*)out, (float*)state, q, k, v, zl,
        (const float*)zbias, (const float*)head_decay, (const float*)inv_freq,
        (const i32*)positions, (const i32*)cu, (const i32*)q_start,
        (const i32*)sslot, q_scale, k_scale, inv_tau, T, B, H, dk, dv, rot,
        ldq, ldk, ldv, ldz, known, s);
  return 9002;
}
