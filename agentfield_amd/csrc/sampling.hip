// Token sampling over the LM-head logits.
//
// Greedy and temperature sampling share one argmax machine: temperature
// sampling uses the Gumbel-max trick (argmax(logits/T + g), g ~ Gumbel(0,1))
// so no sort or cumulative sum over the 128k vocab is needed and the whole
// step is hipGraph-capturable.  Randomness is a counter-based hash of
// (seed, step, b, v); the step counter lives in device memory and is bumped
// by a kernel inside the graph, so replays draw fresh samples.
//
// logits: [B, V] bf16;  temp: [B] f32 (0 => greedy);  out: [B] i32
// partial scratch: pv [B, SPLITS] f32, pi [B, SPLITS] i32
#include "common.h"

#define SMP_SPLITS 16
// rows from here on draw behind a bar (Draw): with fewer values a lane has not enough of
// them for it to pay (all rows unrestricted, a pass of 256 threads in 16 splits: 64 x 32003
// 18.3 us with the bar, 16.8 without; 64 x 128256 26.3 and 27.9, 128 x 128256 without top-k
// or top-p 19.5 and 23.5).  With top-k or top-p two vectors a lane are too few as well (16 x
// 65536, top-p 0.9, 14.6 and 14.0; 64 x 128256 0.9 of the time without), and a row whose
// top-k leaves fewer than one value in 64 draws without (all rows of 128256 with top-k 50, 64
// rows 18.8 and 18.0, 16 rows 14.6 and 14.1).
#define SMP_BAR 65536

__device__ __forceinline__ float u32_to_unit(uint32_t x) {
  return (x >> 8) * (1.f / 16777216.f) + (0.5f / 16777216.f);
}

// Gumbel(0,1) sample from u in (0,1).  The inner fast-math __logf(u) can
// round to EXACTLY 0 for u near 1, making -__logf(0) = +inf — which lets
// any token (including grammar-masked -1e30 rows) win the argmax.  Floor
// the inner result at 1e-30 (gumbel <= ~69, finite).
__device__ __forceinline__ float gumbel_of(float u) {
  const float nl = fmaxf(-__logf(u), 1e-30f);
  return -__logf(nl);
}

// A value and its noise, with the rounding spelled out (contraction is the compiler's
// choice per place otherwise, and equal values are told apart by the last bit): the draw
// without top-k and top-p in one step, the other, which compares x first, in two.
__device__ __forceinline__ float scaled_sum(float l, float invt, float g) {
  return fmaf(l, invt, g);
}
__device__ __forceinline__ float plain_sum(float x, float g) {
#pragma clang fp contract(off)
  return x + g;
}

__device__ __forceinline__ uint32_t hash3(uint32_t a, uint32_t b, uint32_t c) {
  // Wang/xxhash-style avalanche mix
  uint32_t h = a * 0x9E3779B1u + b * 0x85EBCA77u + c * 0xC2B2AE3Du + 0x27220A95u;
  h ^= h >> 15; h *= 0x2C1B3C6Du;
  h ^= h >> 12; h *= 0x297A2D39u;
  h ^= h >> 15;
  return h;
}

// Rows are read 16 bytes per lane.  V need not be a multiple of 8 (nor the row
// 16-byte aligned: an odd V shifts every row), so up to 7 values in front of
// the first 16-byte boundary and up to 7 behind the last go one by one, to
// split 0.  Four loads are in flight per thread: a split is ~1000 vectors at
// V = 128k, i.e. one round trip to memory instead of four.
template <class F>
__device__ __forceinline__ void each_logit(const u16* __restrict__ row, int V,
                                           int split, int nsplit, F f) {
  const int head =
      min(V, (int)(((16u - ((uint32_t)(uintptr_t)row & 15u)) & 15u) >> 1));
  const int nvec = (V - head) >> 3;
  const int per = (nvec + nsplit - 1) / nsplit;
  const int i0 = split * per, i1 = min(nvec, i0 + per);
  const u16* body = row + head;
  for (int i = i0 + (int)threadIdx.x; i < i1; i += 4 * 256) {
    s16x8 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[u] = *reinterpret_cast<const s16x8*>(
          body + (size_t)min(i + u * 256, i1 - 1) * 8);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i + u * 256 >= i1) break;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        f(bf2f((u16)v[u][j]), head + (i + u * 256) * 8 + j);
    }
  }
  if (split == 0) {
    const int t = threadIdx.x, tail = head + nvec * 8;
    if (t < head) f(bf2f(row[t]), t);
    if (tail + t < V) f(bf2f(row[tail + t]), tail + t);
  }
}

// The same with all lanes of a wave in f(value, index, there) together, those without a
// value of their own with there = false.  Eight values are passed over where the largest of
// none of the lanes' is `want`ed.
template <class Want, class F>
__device__ __forceinline__ void each_logit_in_step(const u16* __restrict__ row, int V,
                                                   int split, int nsplit, Want want, F f) {
  const int head =
      min(V, (int)(((16u - ((uint32_t)(uintptr_t)row & 15u)) & 15u) >> 1));
  const int nvec = (V - head) >> 3;
  const int per = (nvec + nsplit - 1) / nsplit;
  const int i0 = split * per, i1 = min(nvec, i0 + per);
  const u16* body = row + head;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63);
  for (int base = i0 + wave; base < i1; base += 4 * 256) {
    const int i = base + (int)(threadIdx.x & 63);
    s16x8 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[u] = *reinterpret_cast<const s16x8*>(
          body + (size_t)min(i + u * 256, i1 - 1) * 8);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (base + u * 256 >= i1) break;
      const bool there = i + u * 256 < i1;
      float m = AF_NEG_INF;                  // a median with infinity is the larger one
#pragma unroll
      for (int j = 0; j < 8; ++j)
        m = __builtin_amdgcn_fmed3f(m, bf2f((u16)v[u][j]), __builtin_inff());
      if (!__any(want(m))) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        f(bf2f((u16)v[u][j]), head + (i + u * 256) * 8 + j, there);
    }
  }
  if (split == 0 && wave == 0) {             // V >= 1
    const int t = threadIdx.x, tail = head + nvec * 8;
    if (head > 0) f(bf2f(row[min(t, V - 1)]), t, t < head);
    if (tail < V) f(bf2f(row[min(tail + t, V - 1)]), tail + t, tail + t < V);
  }
}

// Larger value wins, equal values go to the smaller index: the order in which
// threads and splits see a row does not matter.
__device__ __forceinline__ void take_best(float ov, int oi, float& best,
                                          int& bidx) {
  if (ov > best || (ov == best && oi < bidx)) { best = ov; bidx = oi; }
}

// The best of values with Gumbel noise, where a lane has many.  The noise is two
// logarithms, 22 instructions, that nearly no value needs: with w + 1/2 = 2^24 (1 - u), w a
// whole number, -log u >= 1 - u, so a value x can only pass the score `top` of another where
// w < 2^24 exp(x - top).  Eight steps of w (for the rounding of u and of the first
// logarithm, and the u that rounds to 1) and 2^0.002 make up for rounding of the noise;
// that of the scores themselves, which decides between equal values where 1/T is large, is
// up to 2^-24 of them for the sum and as much for a product that is rounded first: 2^-22
// of `top`.
struct Draw {
  float best = AF_NEG_INF, top = -__builtin_inff();   // this lane's, the wave's
  float lift = __builtin_inff();                      // 24 and what makes up for rounding
  int bidx = 0;
  uint32_t seed;
  int b;

  // all lanes of a wave; x counts where `there`, and `sum` adds noise to it
  template <class Sum>
  __device__ __forceinline__ void take(float x, int v, bool there, Sum sum) {
    const uint32_t h = hash3(seed, (uint32_t)b, (uint32_t)v);
    const float lim = __builtin_amdgcn_exp2f(fmaf(x - top, 1.44269504f, lift)) + 8.f;
    there = there && !((float)(~h >> 8) >= lim);
    if (!__any(there)) return;
    x = sum(gumbel_of(u32_to_unit(h)));
    if (there && (x > best || (x == best && v < bidx))) { best = x; bidx = v; }
    top = wave_max_f32(best);
    lift = fmaf(fabsf(top), 1.44269504f * 0x1p-22f, 24.002f);
  }
};

__device__ __forceinline__ void store_best(float best, int bidx,
                                           float* __restrict__ pv,
                                           i32* __restrict__ pi, int at) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(bidx, o, 64);
    take_best(ov, oi, best, bidx);
  }
  __shared__ float sv[4];
  __shared__ int si[4];
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sv[wid] = best; si[wid] = bidx; }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 4; ++w) take_best(sv[w], si[w], best, bidx);
    pv[at] = best;
    pi[at] = bidx;
  }
}

template <bool BAR>
__global__ void __launch_bounds__(256) sample_partial_kernel(
    float* __restrict__ pv, i32* __restrict__ pi, const u16* __restrict__ logits,
    const float* __restrict__ temp, const uint32_t* __restrict__ step,
    uint32_t seed, int V) {
  const int b = blockIdx.x, split = blockIdx.y;
  const float t = temp[b];
  const float invt = (t > 0.f) ? 1.f / t : 0.f;
  const uint32_t st = *step;
  if (BAR && t > 0.f) {
    Draw d;
    d.seed = seed ^ st;
    d.b = b;
    each_logit_in_step(logits + (size_t)b * V, V, split, SMP_SPLITS,
                       [](float) { return true; },
                       [&](float l, int v, bool there) {
      d.take(l * invt, v, there, [&](float g) { return scaled_sum(l, invt, g); });
    });
    store_best(d.best, d.bidx, pv, pi, b * SMP_SPLITS + split);
    return;
  }
  float best = AF_NEG_INF;
  int bidx = 0;
  each_logit(logits + (size_t)b * V, V, split, SMP_SPLITS, [&](float x, int v) {
    if (t > 0.f) {
      const float u = u32_to_unit(hash3(seed ^ st, (uint32_t)b, (uint32_t)v));
      x = scaled_sum(x, invt, gumbel_of(u));
    }
    if (x > best || (x == best && v < bidx)) { best = x; bidx = v; }
  });
  store_best(best, bidx, pv, pi, b * SMP_SPLITS + split);
}

// The last kernel of a draw: every reader of *step has finished, so it also
// moves the counter (one launch less, ~4.6 us each in a captured step).
__global__ void __launch_bounds__(64) sample_combine_kernel(
    i32* __restrict__ out, const float* __restrict__ pv,
    const i32* __restrict__ pi, uint32_t* __restrict__ step) {
  const int b = blockIdx.x;
  float best = AF_NEG_INF;
  int bidx = 0;
  if (threadIdx.x < SMP_SPLITS)
    take_best(pv[b * SMP_SPLITS + threadIdx.x],
              pi[b * SMP_SPLITS + threadIdx.x], best, bidx);
#pragma unroll
  for (int o = SMP_SPLITS / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(bidx, o, 64);
    take_best(ov, oi, best, bidx);
  }
  if (threadIdx.x == 0) {
    out[b] = bidx;
    if (b == 0) *step += 1u;
  }
}

// ---- top-k / top-p restriction --------------------------------------------
// Sort-free: a 256-bin histogram of logits over [rowmax-SPAN, rowmax]
// (bin 255 = max) gives, per row, the threshold above which the top-k count
// or top-p probability mass is reached; the Gumbel-max draw then ignores
// logits below the threshold.  Boundary-bin granularity is SPAN/256 ~ 0.08
// logits — the standard approximation for GPU nucleus sampling.
//
// Every pass runs SMP_SPLITS blocks per row: a row is 256 KB, and one block a
// row (64 of them on 256 CUs, one bin conflict after the other) took 173 us
// for the histogram and 52 us for the maximum at 64 x 128256.  The passes after
// the first fold the per-split results of the pass before in their prologue, so
// nothing but the three reads of the row and the draw's last step is launched: 346
// us -> 27 us; 24 with the bar of Draw, greedy rows without a histogram and the blocks of a
// CU from different rows.  (A draw to which top-k leaves few values takes 6.8 us, mostly its
// blocks' folding of all 16 histograms of their row, 32 KB each; one of all values, bound by
// their hashes, 13.9.)
#define TKP_BINS 256
#define TKP_SPAN 20.0f

// pass A: maximum of each split
__global__ void __launch_bounds__(256) row_max_kernel(
    float* __restrict__ rmax, const u16* __restrict__ logits, int V) {
  const int b = blockIdx.x, split = blockIdx.y;
  float best = AF_NEG_INF;
  each_logit(logits + (size_t)b * V, V, split, SMP_SPLITS,
             [&](float x, int) { best = fmaxf(best, x); });
  best = wave_max_f32(best);
  __shared__ float sv[4];
  if ((threadIdx.x & 63) == 0) sv[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0)
    rmax[b * SMP_SPLITS + split] =
        fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
}

__device__ __forceinline__ float row_max_of(const float* __restrict__ rmax,
                                            int b) {
  float m = rmax[b * SMP_SPLITS];
#pragma unroll
  for (int s = 1; s < SMP_SPLITS; ++s)
    m = fmaxf(m, rmax[b * SMP_SPLITS + s]);
  return m;
}

// pass B: histogram of counts and exp-mass per bin (temperature applied) of
// each split.  What bounds it is LDS atomics: at 64 x 128256 a float add per
// value takes 41 us and an integer one 2 us, whatever the conflicts.  So a value
// adds one 64-bit integer: 1 in the upper 20 bits, and below them its mass
// relative to its bin's upper edge (0.92..1) in units of 2^-24, which loses no
// more per value than a float does and nothing in the sum.  Every bin has 16
// copies, one per lane of a group of 16 (45 us -> 8 us).  A copy gets about 1/256 of
// a split row's values: the 20-bit count and the 44-bit mass hold rows of up to 2^27.
#define TKP_COPIES 16
#define TKP_MASS_BITS 44
__global__ void __launch_bounds__(256) tkp_hist_kernel(
    i32* __restrict__ hist_n, float* __restrict__ hist_m,
    const u16* __restrict__ logits, const float* __restrict__ rmax,
    const float* __restrict__ temp, int V) {
  const int split = blockIdx.y, b = blockIdx.x;
  const int copy = threadIdx.x & (TKP_COPIES - 1);
  const float t = temp[b];
  if (!(t > 0.f)) return;    // a greedy row takes its largest value: its histogram is not written
  __shared__ unsigned long long h[TKP_BINS * TKP_COPIES];
#pragma unroll
  for (int c = 0; c < TKP_COPIES; ++c) h[c * 256 + threadIdx.x] = 0;
  __syncthreads();
  const float invt = 1.f / t;
  const float mx = row_max_of(rmax, b) * invt;
  constexpr float STEP = TKP_SPAN / TKP_BINS;
  bool odd = false;  // a value that is not a number makes the mass one too
  each_logit(logits + (size_t)b * V, V, split, SMP_SPLITS, [&](float l, int) {
    const float x = l * invt;
    odd |= (x - mx) != (x - mx);
    int bin = (int)((x - (mx - TKP_SPAN)) * (TKP_BINS / TKP_SPAN));
    if (bin < 0) return;  // below span: negligible mass
    if (bin > TKP_BINS - 1) bin = TKP_BINS - 1;
    const float r = __expf(x - mx + (float)(TKP_BINS - 1 - bin) * STEP);
    atomicAdd(&h[bin * TKP_COPIES + copy],
              (1ull << TKP_MASS_BITS) +
                  (unsigned long long)(uint32_t)(r * 16777216.f + 0.5f));
  });
  odd = __syncthreads_or(odd);
  const int first = threadIdx.x * TKP_COPIES;
  int n = 0;
  unsigned long long m = 0;
#pragma unroll
  for (int c = 0; c < TKP_COPIES; ++c) {
    const unsigned long long q =
        h[first + ((c + threadIdx.x) & (TKP_COPIES - 1))];
    n += (int)(q >> TKP_MASS_BITS);
    m += q & ((1ull << TKP_MASS_BITS) - 1);
  }
  const size_t at = ((size_t)b * SMP_SPLITS + split) * TKP_BINS + threadIdx.x;
  hist_n[at] = n;
  hist_m[at] = odd ? __builtin_nanf("")
                   : __expf((float)((int)threadIdx.x - (TKP_BINS - 1)) * STEP) *
                         ((float)m * (1.f / 16777216.f));
}

// The threshold of a row (in temperature-scaled logit space): bins from the
// top until top-k count / top-p mass is covered.  Thread i holds bin 255 - i;
// an inclusive scan over the block gives count and mass down to that bin.
__device__ __forceinline__ float tkp_threshold(
    const i32* __restrict__ hist_n, const float* __restrict__ hist_m,
    float mx, int k, float p, int b) {
  const int i = threadIdx.x, lane = i & 63, wid = i >> 6;
  const size_t at = (size_t)b * SMP_SPLITS * TKP_BINS + (TKP_BINS - 1 - i);
  int cnt = 0;
  float mass = 0.f;
#pragma unroll
  for (int s = 0; s < SMP_SPLITS; ++s) {
    cnt += hist_n[at + s * TKP_BINS];
    mass += hist_m[at + s * TKP_BINS];
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int c = __shfl_up(cnt, o, 64);
    const float m = __shfl_up(mass, o, 64);
    if (lane >= o) { cnt += c; mass += m; }
  }
  __shared__ i32 wc[4];
  __shared__ float wm[4];
  __shared__ i32 hit[4];
  if (lane == 63) { wc[wid] = cnt; wm[wid] = mass; }
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wid) { cnt += wc[w]; mass += wm[w]; }
    total += wm[w];
  }
  const unsigned long long full = __ballot(cnt >= k || mass >= p * total);
  if (lane == 0) hit[wid] = full ? wid * 64 + (int)__ffsll(full) - 1 : TKP_BINS;
  __syncthreads();
  const int first = min(min(hit[0], hit[1]), min(hit[2], hit[3]));
  if (k == 1) return mx;  // exact: only the argmax survives
  return first < TKP_BINS
             ? mx - TKP_SPAN + (float)(TKP_BINS - 1 - first) *
                                   (TKP_SPAN / TKP_BINS)
             : mx - TKP_SPAN;
}

// pass C: Gumbel-argmax over {x/T >= threshold}
template <bool BAR>
__global__ void __launch_bounds__(256) tkp_sample_kernel(
    float* __restrict__ pv, i32* __restrict__ pi, const u16* __restrict__ logits,
    const float* __restrict__ temp, const float* __restrict__ rmax,
    const i32* __restrict__ hist_n, const float* __restrict__ hist_m,
    const i32* __restrict__ topk, const float* __restrict__ topp,
    const uint32_t* __restrict__ step, uint32_t seed, int V) {
  // a CU's blocks are of different rows, long and short (as blockIdx.x the four of a CU
  // were of one row: 64 x 128256 25.4 us, 24.2)
  const int split = blockIdx.y, b = (blockIdx.x + 8 * (split >> 2)) % gridDim.x;
  const u16* row = logits + (size_t)b * V;
  const float t = temp[b];
  if (!(t > 0.f)) {
    float best = AF_NEG_INF;
    int bidx = 0;
    each_logit(row, V, split, SMP_SPLITS, [&](float x, int v) {
      if (x > best || (x == best && v < bidx)) { best = x; bidx = v; }
    });
    store_best(best, bidx, pv, pi, b * SMP_SPLITS + split);
    return;
  }
  const float invt = 1.f / t;
  const int k = (topk[b] > 0) ? topk[b] : V;
  const float p = (topp[b] > 0.f && topp[b] < 1.f) ? topp[b] : 1.f;
  const float th =
      tkp_threshold(hist_n, hist_m, row_max_of(rmax, b) * invt, k, p, b);
  const uint32_t st = *step;
  if (BAR && k >= (V >> 6)) {                // of few values a bar spares nothing
    Draw d;
    d.seed = seed ^ st;
    d.b = b;
    each_logit_in_step(row, V, split, SMP_SPLITS,
                       [&](float l) { return !(l * invt < th); },
                       [&](float l, int v, bool there) {
      const float x = l * invt;
      there = there && !(x < th);
      if (__any(there)) d.take(x, v, there, [&](float g) { return plain_sum(x, g); });
    });
    store_best(d.best, d.bidx, pv, pi, b * SMP_SPLITS + split);
    return;
  }
  float best = AF_NEG_INF;
  int bidx = 0;
  each_logit(row, V, split, SMP_SPLITS, [&](float l, int v) {
    float x = l * invt;
    if (x < th) return;
    x = plain_sum(x, gumbel_of(u32_to_unit(hash3(seed ^ st, (uint32_t)b, (uint32_t)v))));
    if (x > best || (x == best && v < bidx)) { best = x; bidx = v; }
  });
  store_best(best, bidx, pv, pi, b * SMP_SPLITS + split);
}

// scratch of af_sample_topkp besides pv / pi: rmax [B, 16] f32,
// hist_n [B, 16, 256] i32, hist_m [B, 16, 256] f32.
AF_EXPORT int af_sample_topkp(void* out, void* pv, void* pi, void* rmax,
                              void* hist_n, void* hist_m, const void* logits,
                              const void* temp, const void* topk,
                              const void* topp, void* step, uint32_t seed,
                              int B, int V, void* stream) {
  if (B == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  dim3 g(B, SMP_SPLITS);
  row_max_kernel<<<g, 256, 0, st>>>((float*)rmax, (const u16*)logits, V);
  tkp_hist_kernel<<<g, 256, 0, st>>>((i32*)hist_n, (float*)hist_m,
                                     (const u16*)logits, (const float*)rmax,
                                     (const float*)temp, V);
  const auto draw = V > SMP_BAR ? tkp_sample_kernel<true> : tkp_sample_kernel<false>;
  draw<<<g, 256, 0, st>>>(
      (float*)pv, (i32*)pi, (const u16*)logits, (const float*)temp,
      (const float*)rmax, (const i32*)hist_n, (const float*)hist_m,
      (const i32*)topk, (const float*)topp, (const uint32_t*)step, seed, V);
  sample_combine_kernel<<<B, 64, 0, st>>>((i32*)out, (const float*)pv,
                                          (const i32*)pi, (uint32_t*)step);
  return af_last_err();
}

AF_EXPORT int af_sample(void* out, void* pv, void* pi, const void* logits,
                        const void* temp, void* step, uint32_t seed,
                        int B, int V, void* stream) {
  if (B == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  dim3 g1(B, SMP_SPLITS);
  const auto draw = V >= SMP_BAR ? sample_partial_kernel<true> : sample_partial_kernel<false>;
  draw<<<g1, 256, 0, st>>>(
      (float*)pv, (i32*)pi, (const u16*)logits, (const float*)temp,
      (const uint32_t*)step, seed, V);
  sample_combine_kernel<<<B, 64, 0, st>>>((i32*)out, (const float*)pv,
                                          (const i32*)pi, (uint32_t*)step);
  return af_last_err();
}

// Gather last-token logits rows: hidden [T,H] -> rows at idx [B] -> out [B,H]
__global__ void __launch_bounds__(256) gather_rows_kernel(
    u16* __restrict__ out, const u16* __restrict__ x, const i32* __restrict__ idx,
    int H) {
  const int b = blockIdx.x;
  const u16* src = x + (size_t)idx[b] * H;
  u16* dst = out + (size_t)b * H;
  for (int i = threadIdx.x * 8; i < H; i += 256 * 8)
    *reinterpret_cast<s16x8*>(dst + i) = *reinterpret_cast<const s16x8*>(src + i);
}

AF_EXPORT int af_gather_rows(void* out, const void* x, const void* idx, int B,
                             int H, void* stream) {
  if (H % 8) return 9001;
  if (B == 0) return 0;
  gather_rows_kernel<<<B, 256, 0, (hipStream_t)stream>>>(
      (u16*)out, (const u16*)x, (const i32*)idx, H);
  return af_last_err();
}
