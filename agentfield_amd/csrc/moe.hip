// Routing, sorting and recombination of rows for the mixture feed-forward's
// exact dispatch (every expert runs its own rows).
//
// The projections are large; what the dispatch costs beside them is launches and
// waits: finding each expert's rows with a device-wide scan per expert made the
// host wait eight times per layer, and the rows were gathered and added back
// expert by expert in fp32 (1100 rows, 8 experts, 2 per row: 146 launches, 0.8 of
// 2.0 ms).  Here the rows are sorted by expert once, so that every expert's rows
// are one contiguous block: four launches and one wait for the block bounds.
#include "common.h"

#define MOE_MAX_K 8

// Router logits in fp32 (products of bf16 are exact), softmax over the k largest:
// equal logits go to the smaller expert.  A logit that is not a number counts as the
// largest, so that the row's weights show it.
// Few rows are bound by latency: with a wave per row the loop over the row waits for
// memory eight times (40 rows of 4096 over 8 experts 18.7 us, sorting included), with
// WAVES = 4 to a row most of its loads are out at once (10.8).  Many rows are bound by
// their instructions, and four waves sum every expert's logit four times over: there a
// wave takes a row.
template <int EM, int WAVES>
__global__ void __launch_bounds__(256) moe_route_kernel(
    i32* __restrict__ topi, float* __restrict__ topv, const u16* __restrict__ x,
    const u16* __restrict__ router, int T, int H, int E, int k) {
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = WAVES == 4 ? blockIdx.x : blockIdx.x * 4 + wid;
  if (t >= T) return;
  const u16* xr = x + (size_t)t * H;
  float acc[EM];
#pragma unroll
  for (int e = 0; e < EM; ++e) acc[e] = 0.f;
#pragma unroll WAVES == 4 ? 2 : 1
  for (int c = (WAVES == 4 ? threadIdx.x : lane) * 8; c < H; c += 512 * WAVES) {
    const s16x8 xv = *reinterpret_cast<const s16x8*>(xr + c);
    float xf[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) xf[j] = bf2f((u16)xv[j]);
#pragma unroll
    for (int e = 0; e < EM; ++e) {
      const s16x8 rv =
          *reinterpret_cast<const s16x8*>(router + (size_t)min(e, E - 1) * H + c);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[e] = fmaf(xf[j], bf2f((u16)rv[j]), acc[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < EM; ++e) acc[e] = wave_sum_f32(acc[e]);
  if constexpr (WAVES == 4) {
    __shared__ float part[4][EM];
#pragma unroll
    for (int e = 0; e < EM; ++e)
      if (lane == 0) part[wid][e] = acc[e];
    __syncthreads();
    if (wid) return;
#pragma unroll
    for (int e = 0; e < EM; ++e)
      acc[e] = (part[0][e] + part[1][e]) + (part[2][e] + part[3][e]);
  }
  unsigned long long used = 0;
  float best[MOE_MAX_K], sum = 0.f;
  int who[MOE_MAX_K];
#pragma unroll
  for (int j = 0; j < MOE_MAX_K; ++j) {
    if (j >= k) break;
    float b = 0.f;
    int w = -1;
#pragma unroll
    for (int e = 0; e < EM; ++e) {
      if (e >= E || (used >> e & 1)) continue;
      if (w < 0 || acc[e] > b || acc[e] != acc[e]) { b = acc[e]; w = e; }
    }
    used |= 1ull << w;
    best[j] = b;
    who[j] = w;
  }
  const float top = best[0];
#pragma unroll
  for (int j = 0; j < MOE_MAX_K; ++j)
    if (j < k) {
      best[j] = expf(best[j] - top);
      sum += best[j];
    }
#pragma unroll
  for (int j = 0; j < MOE_MAX_K; ++j)
    if (j < k && lane == j) {
      topi[(size_t)t * k + j] = who[j];
      topv[(size_t)t * k + j] = best[j] / sum;
    }
}

// Stable counting sort of the n = T*k (row, choice) entries by expert, in one
// block of 16 waves; a wave owns a contiguous stretch of entries.
//   offs [E+1]: first sorted position of every expert
//   row  [n]:   row of the entry at a sorted position
//   pos  [n]:   sorted position of an entry
#define MOE_MAX_E 64
__global__ void __launch_bounds__(1024) moe_sort_kernel(
    i32* __restrict__ offs, i32* __restrict__ row, i32* __restrict__ pos,
    const i32* __restrict__ topi, int n, int k, int E) {
  __shared__ i32 cnt[16][MOE_MAX_E];
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int per = ((n + 15) / 16 + 63) & ~63;
  const int i0 = wid * per, i1 = min(n, i0 + per);
  for (int i = threadIdx.x; i < 16 * MOE_MAX_E; i += 1024) (&cnt[0][0])[i] = 0;
  __syncthreads();
  int mine = 0;  // lane e counts expert e
  for (int i = i0; i < i1; i += 64) {
    const int e = (i + lane < i1) ? topi[i + lane] : -1;
    for (int w = 0; w < E; ++w) {
      const int c = __popcll(__ballot(e == w));
      if (lane == w) mine += c;
    }
  }
  if (lane < E) cnt[wid][lane] = mine;
  __syncthreads();
  if (wid == 0) {
    int tot = 0;
    for (int w = 0; w < 16; ++w) tot += cnt[w][lane];
    int incl = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    int at = incl - tot;
    if (lane < E) offs[lane] = at;
    if (lane == 0) offs[E] = n;
    for (int w = 0; w < 16; ++w) {
      const int c = cnt[w][lane];
      cnt[w][lane] = at;
      at += c;
    }
  }
  __syncthreads();
  int next = cnt[wid][lane];  // lane e: next position of expert e in this stretch
  for (int i = i0; i < i1; i += 64) {
    const int e = (i + lane < i1) ? topi[i + lane] : -1;
    for (int w = 0; w < E; ++w) {
      const unsigned long long m = __ballot(e == w);
      const int base = __shfl(next, w, 64);
      if (e == w) {
        const int p = base + __popcll(m & ((1ull << lane) - 1));
        pos[i + lane] = p;
        row[p] = (i + lane) / k;
      }
      if (lane == w) next += __popcll(m);
    }
  }
}

// out[t] = sum_j topv[t, j] * y[pos[t, j]] in fp32, rounded once: a block per row.
__global__ void __launch_bounds__(256) moe_combine_kernel(
    u16* __restrict__ out, const u16* __restrict__ y, const i32* __restrict__ pos,
    const float* __restrict__ topv, int H, int k) {
  const int t = blockIdx.x;
  for (int c = threadIdx.x * 8; c < H; c += 2048) {
    float o[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int j = 0; j < k; ++j) {
      const float g = topv[(size_t)t * k + j];
      const s16x8 v = *reinterpret_cast<const s16x8*>(
          y + (size_t)pos[(size_t)t * k + j] * H + c);
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = fmaf(g, bf2f((u16)v[i]), o[i]);
    }
    s16x8 r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = (short)f2bf(o[i]);
    *reinterpret_cast<s16x8*>(out + (size_t)t * H + c) = r;
  }
}

// Whether four waves share a row (see moe_route_kernel).  Routing, a wave / four waves per
// row in us: 8 experts, rows of 4096: 18.6 / 11.8 at 300 rows, 24.6 / 22.6 at 2000, 40.9 /
// 38.8 at 4096, 62 / 70 at 8192; rows of 1024: 12.5 / 12.0 at 1000, 16.8 / 18.4 at 2000; 2
// experts, rows of 4096: 16.3 / 15.9 at 2000, 17.2 / 20.2 at 3000; 32 experts, rows of
// 1024: 40.5 / 35.4 at 600, 45.8 / 48.0 at 800; 64 experts, rows of 2048: 95 / 60 at 200,
// 115 / 157 at 600, rows of 8192: 256 / 271 at 600.  A row of 256 is one load anyway (4
// experts, 1000 rows 9.7 / 10.5).
static bool route_shares_rows(int T, int H, int E) {
  if (H < 1024) return false;
  if (E > 32) return T <= min(H / 8, 512);
  if (E > 16) return T <= min(H / 2, 2048);
  return T <= min(H, E < 8 ? 2048 : 4096);
}

// topi [T, k] i32, topv [T, k] f32 (largest first, sum 1); offs / row / pos as
// moe_sort_kernel leaves them.
AF_EXPORT int af_moe_route(void* topi, void* topv, void* offs, void* row, void* pos,
                           const void* x, const void* router, int T, int H, int E,
                           int k, void* stream) {
  if (H % 8 || E < 1 || E > MOE_MAX_E || k < 1 || k > MOE_MAX_K || k > E) return 9001;
  if (T == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  const bool share = route_shares_rows(T, H, E);
#define AF_ROUTE_AS(EM, WAVES)                                                 \
  moe_route_kernel<EM, WAVES><<<WAVES == 4 ? T : (T + 3) / 4, 256, 0, st>>>(   \
      (i32*)topi, (float*)topv, (const u16*)x, (const u16*)router, T, H, E, k)
#define AF_ROUTE(EM) (share ? AF_ROUTE_AS(EM, 4) : AF_ROUTE_AS(EM, 1))
  if (E <= 8) AF_ROUTE(8);
  else if (E <= 16) AF_ROUTE(16);
  else if (E <= 32) AF_ROUTE(32);
  else AF_ROUTE(64);
#undef AF_ROUTE
#undef AF_ROUTE_AS
  moe_sort_kernel<<<1, 1024, 0, st>>>((i32*)offs, (i32*)row, (i32*)pos,
                                      (const i32*)topi, T * k, k, E);
  return af_last_err();
}

AF_EXPORT int af_moe_combine(void* out, const void* y, const void* pos,
                             const void* topv, int T, int H, int k,
                             void* stream) {
  if (H % 8) return 9001;
  if (T == 0) return 0;
  moe_combine_kernel<<<T, 256, 0, (hipStream_t)stream>>>(
      (u16*)out, (const u16*)y, (const i32*)pos, (const float*)topv, H, k);
  return af_last_err();
}
