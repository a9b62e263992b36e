// Paged decode attention (one query token per sequence) with GQA and
// split-K over the KV length ("flash-decoding" style).
//
// Shapes: q   [B, rows at stride qs] bf16, head h at offset h*D (post-RoPE)
//         kc  [npages, Hk, page_size, D] bf16
//         vc  [npages, Hk, page_size, D] bf16
//         bt  [B, max_pages] i32      block table
//         len [B] i32                 total tokens per seq (incl. current)
//         out [B, Hq*D] bf16 (contiguous)
// GQA group G = Hq/Hk in {1,2,4,8}.  D = 128.
//
// The K/V stream is the bound: 512 bytes per token and K/V head, used once.  A
// CU's share of the memory rate is ~9 bytes per clock, i.e. one token every ~54
// clocks, so a token may cost at most that in instructions and the loop must
// keep tens of KB per CU in flight.
//   grid (B x Hk, NSPLIT), K/V heads or sequences fastest, see heads_first (as three
//   dimensions 12 of 4500..8000 with G = 8 45.6 -> 46.6 us); block = 256 threads = 4
//   waves; a wave iteration takes
//   16 tokens (4 KB of K, 4 KB of V, 16 B per lane and load), the next tile's
//   eight loads are issued before the current tile's arithmetic.
//   Scores come from the matrix cores: K rows are the A operand straight from
//   the cache (lane = token, quarter of 32 dims), the group's query heads the
//   B operand (columns repeat when G < 16), accumulated over 4 x 32 dims.  The
//   result leaves lane (tg, h) = (lane>>4, lane&15) with head h's scores of the
//   four tokens tg*4..tg*4+3.
//   Running maximum, sum and output belong to a row of 16 lanes and its tokens
//   (every fourth group of four): nothing crosses lanes inside the loop but a
//   DPP broadcast of a head's weight along its row.  P V stays in fp32 vector
//   arithmetic (weights are never rounded): lane (tg, dl) owns dims
//   [dl*8, dl*8+8) and reads the same V rows whole, ~13 clocks per token at
//   G = 4.
//   Rows, then waves (through LDS), then splits (second kernel) merge once.
// A sequence's result has nothing of the others, unless the step's cut (decode_cut.h) is
// given: where that cuts unlike lengths in equal shares, the order of a sequence's fp32 sums
// depends on the lengths beside it, and so may the last bit of its bf16 results.
// Measured with 8 K/V heads, G = 4, against one lane group per token with a
// shuffle reduction per score: 24 sequences of 1800..8100 tokens (513 MB)
// 225 -> 108 us (4.7 TB/s), in equal shares 84 (6.1), 128 of 545 101 -> 49 us (5.8 TB/s),
// 1 of 8000 58 -> 16 us.  V is read with nontemporal loads, whole rows per instruction: 114
// -> 108 and 57.3 -> 52.5 us.  K is not: two instructions share each of its lines,
// and a line dropped between them is fetched twice (64 ragged sequences of up to
// 2000 tokens 60 -> 65 us with both, 59 with V only).  Not the loads' latency: eight
// waves per block (114 -> 125 us) and whole rows through LDS with two tiles per wave in
// flight (110.5 -> 112) do not help, nor do pages in order.
#include "decode_cut.h"

#include <type_traits>

#define AD_D 128
#define AD_MAXG 8

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8d;

__device__ __forceinline__ bf16x8d as_bf16x8d(s16x8 v) {
  union { s16x8 s; bf16x8d b; } u;
  u.s = v;
  return u.b;
}

// lane I of each 16-lane row, in all lanes of the row
template <int I>
__device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(
      0, __float_as_int(v), 0x150 + I, 0xf, 0xf, true));
}

template <int I, int N, class F>
__device__ __forceinline__ void each_head(F f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    each_head<I + 1, N>(f);
  }
}

// Partial layout: po [B, Hk, NSPLIT, G, D] f32; pml [B, Hk, NSPLIT, G, 2] f32
// (maximum in units of log2, sum; a split without tokens leaves po unwritten);
// CUT: [Hk, cap, G, ..], cap pieces, split s of sequence b at b * nsplit + s.
//
// TILED: page_size is a multiple of AD_TILE, so a tile lies in one page and its
// index is a scalar load; otherwise every lane looks its tokens' pages up.
//
// A block's part: rounds of sequence b from its skip'th on, sums to piece.  GO_ON: and `left`
// rounds of the sequences behind it.
template <int G, bool TILED, bool GO_ON>
__device__ __forceinline__ void attn_part(
    u16* __restrict__ out, float* __restrict__ po, float* __restrict__ pml,
    const u16* __restrict__ q, const u16* __restrict__ kc, const u16* __restrict__ vc,
    const i32* __restrict__ bt, const i32* __restrict__ len, float scale, int B, int Hk,
    int page_size, int page_shift, int max_pages, int nsplit, i64 qs, int win,
    float (*s_ml)[G][2], float (*s_o)[G][AD_D], int kvh, int b, int L, int skip, int rounds,
    size_t piece, int left) {
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tg = lane >> 4, dl = lane & 15;
  const int Hq = Hk * G;

  // (constant memory: the compiler looks nothing up by scalar loads behind a store, and a
  // vector load of a page waits for the tile that was asked for before it)
  typedef const __attribute__((address_space(4))) i32* pages;
  const pages tables = (pages)bt, lengths = (pages)len;
  pages btrow = tables + (size_t)b * max_pages;
  auto page_of = [&](int t) {
    return btrow[page_shift >= 0 ? t >> page_shift : t / page_size];
  };
  // a part: its visible tokens [t0, t1), tile grid; this wave's tile and the next one's page
  int c0, t0, t1, t, pg_next = 0;
  auto take = [&](int L, int skip, int rounds) {
    const Visible v = visible(L, win);
    c0 = v.tile0 + skip * ROUND;
    t1 = min(L, c0 + rounds * ROUND);
    t0 = max(v.first, c0);
    t = c0 + wid * AD_TILE;
  };
  take(L, skip, rounds);
  if (c0 >= t1) {                          // no tokens (uniform in the block)
    if (nsplit > 1) {
      if (threadIdx.x < G) {
        const size_t at = piece * G + threadIdx.x;
        pml[at * 2] = AF_NEG_INF;
        pml[at * 2 + 1] = 0.f;
      }
    } else {                               // an empty sequence
      for (int i = threadIdx.x; i < G * AD_D; i += 64 * AD_WAVES)
        out[(size_t)b * (Hq * AD_D) + kvh * G * AD_D + i] = 0;
    }
    return;
  }

  // query heads as B operand: lane holds head (lane & 15) % G, dims
  // 32 c + tg*8 .. +8
  s16x8 qf[4];
  auto load_q = [&]() {
    const u16* qp = q + (size_t)b * qs + (kvh * G + (dl & (G - 1))) * AD_D + tg * 8;
#pragma unroll
    for (int c = 0; c < 4; ++c) qf[c] = *reinterpret_cast<const s16x8*>(qp + c * 32);
  };
  const float sc = scale * 1.44269504088896f;  // softmax in powers of two

  auto page_off = [&](int t) {
    return page_shift >= 0 ? t & (page_size - 1) : t % page_size;
  };
  // K rows of tokens behind t1 may be read (their scores are dropped); V rows
  // are clamped to visible tokens, whose values are finite when weighed by 0
  auto load_tile = [&](int t, int page, s16x8* kf, s16x8* vf) {
    if (TILED) {
      const size_t base =
          (((size_t)page * Hk + kvh) * page_size + page_off(t)) * AD_D;
      const u16* kp = kc + base + dl * AD_D + tg * 8;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        kf[c] = *reinterpret_cast<const s16x8*>(kp + c * 32);
      const u16* vp = vc + base + dl * 8;
      const int lo = t0 - t, hi = t1 - 1 - t;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        vf[r] = __builtin_nontemporal_load(reinterpret_cast<const s16x8*>(
            vp + min(max(tg * 4 + r, lo), hi) * AD_D));
    } else {
      auto row = [&](int tok) {
        const int tc = min(max(tok, t0), t1 - 1);
        return (((size_t)page_of(tc) * Hk + kvh) * page_size + page_off(tc)) * AD_D;
      };
      const u16* kp = kc + row(t + dl) + tg * 8;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        kf[c] = *reinterpret_cast<const s16x8*>(kp + c * 32);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        vf[r] = __builtin_nontemporal_load(
            reinterpret_cast<const s16x8*>(vc + row(t + tg * 4 + r) + dl * 8));
    }
  };

  s16x8 kf[4], vf[4], kn[4], vn[4];
  auto begin = [&]() {                     // the wave's first tile
    load_q();
    if (t >= t1) return;
    load_tile(t, TILED ? page_of(t) : 0, kf, vf);
    if (TILED) pg_next = page_of(min(t + ROUND, t1 - 1));
  };
  begin();
  for (;;) {
    float m = AF_NEG_INF, l = 0.f, acc[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[g][j] = 0.f;
    for (; t < t1; t += ROUND) {
      if (t + ROUND < t1) {
        load_tile(t + ROUND, pg_next, kn, vn);
        if (TILED) pg_next = page_of(min(t + 2 * ROUND, t1 - 1));
      }
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c)
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8d(kf[c]),
                                                    as_bf16x8d(qf[c]), s, 0, 0, 0);
      float mn = m;
      bool ok[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tok = t + tg * 4 + r;
        ok[r] = tok >= t0 && tok < t1;
        s[r] = ok[r] ? s[r] * sc : AF_NEG_INF;
        mn = fmaxf(mn, s[r]);
      }
      float p[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        p[r] = ok[r] ? __builtin_amdgcn_exp2f(s[r] - mn) : 0.f;
      if (__any(mn > m)) {  // rare once the first tiles have been seen
        const float corr = __builtin_amdgcn_exp2f(m - mn);
        l *= corr;
        each_head<0, G>([&](auto g) {
          const float cg = row_bcast<g.value>(corr);
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[g.value][j] *= cg;
        });
        m = mn;
      }
      l += (p[0] + p[1]) + (p[2] + p[3]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = bf2f((u16)vf[r][j]);
        each_head<0, G>([&](auto g) {
          const float pg = row_bcast<g.value>(p[r]);
#pragma unroll
          for (int j = 0; j < 8; ++j)
            acc[g.value][j] = fmaf(pg, v[j], acc[g.value][j]);
        });
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) { kf[c] = kn[c]; vf[c] = vn[c]; }
    }

    // the slot's next sequence that has tokens: its loads travel while this part is merged
    const int of = b;
    const size_t to = piece;
    bool on = false;
    if (GO_ON && left > 0) {
      int L = 0;
      while (L <= 0 && b + 1 < B) {
        L = lengths[++b];
        ++piece;
      }
      on = L > 0;
      if (on) {
        const int rounds = min(left, visible(L, win).rounds);
        left -= rounds;
        btrow = tables + (size_t)b * max_pages;
        take(L, 0, rounds);
        begin();
      }
    }

    // fold the four rows (same dims, other tokens)
    float M = fmaxf(m, __shfl_xor(m, 16, 64));
    M = fmaxf(M, __shfl_xor(M, 32, 64));
    const float f = (m <= AF_NEG_INF) ? 0.f : __builtin_amdgcn_exp2f(m - M);
    l *= f;
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    each_head<0, G>([&](auto g) {
      const float fg = row_bcast<g.value>(f);
      float o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        o[j] = acc[g.value][j] * fg;
        o[j] += __shfl_xor(o[j], 16, 64);
        o[j] += __shfl_xor(o[j], 32, 64);
      }
      if (tg == 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) s_o[wid][g.value][dl * 8 + j] = o[j];
      }
    });
    if (lane < G) { s_ml[wid][lane][0] = M; s_ml[wid][lane][1] = l; }
    __syncthreads();

    // merge the waves: two elements per thread
    for (int i = threadIdx.x; i < G * AD_D / 2; i += 64 * AD_WAVES) {
      const int g = i / (AD_D / 2), d = (i % (AD_D / 2)) * 2;
      float Mx = s_ml[0][g][0];
#pragma unroll
      for (int w = 1; w < AD_WAVES; ++w) Mx = fmaxf(Mx, s_ml[w][g][0]);
      float L2 = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
      for (int w = 0; w < AD_WAVES; ++w) {
        const float c = (s_ml[w][g][0] <= AF_NEG_INF)
                            ? 0.f
                            : __builtin_amdgcn_exp2f(s_ml[w][g][0] - Mx);
        L2 += s_ml[w][g][1] * c;
        o0 += s_o[w][g][d] * c;
        o1 += s_o[w][g][d + 1] * c;
      }
      if (nsplit == 1) {
        const float inv = (L2 > 0.f) ? 1.f / L2 : 0.f;
        u16x2 ov = {f2bf(o0 * inv), f2bf(o1 * inv)};
        *reinterpret_cast<u16x2*>(out + (size_t)of * (Hq * AD_D) +
                                  (kvh * G + g) * AD_D + d) = ov;
      } else {
        const size_t at = to * G + g;
        *reinterpret_cast<f32x2*>(po + at * AD_D + d) = f32x2{o0, o1};
        if (d == 0) { pml[at * 2] = Mx; pml[at * 2 + 1] = L2; }
      }
    }
    if (!on) return;
    __syncthreads();                         // the sums are read
  }
}

// CUT: sequences are cut as the step's cut says (decode_cut.h).  The parts' code stands there
// twice: with one body for nsplit parts and for shares, what goes on behind a part cost those
// that do not 0.3 to 0.7 us.
template <int G, bool TILED, bool CUT>
__global__ void __launch_bounds__(64 * AD_WAVES, (G == 8 ? 3 : 4) - CUT) attn_decode_kernel(
    u16* __restrict__ out, float* __restrict__ po, float* __restrict__ pml,
    const u16* __restrict__ q, const u16* __restrict__ kc, const u16* __restrict__ vc,
    const i32* __restrict__ bt, const i32* __restrict__ len, const CutRow* __restrict__ cut,
    float scale, int B, int Hk, int page_size, int page_shift, int max_pages,
    int nsplit, int cap, i64 qs, int win, int faster) {
  __shared__ float s_ml[AD_WAVES][G][2];
  __shared__ float s_o[AD_WAVES][G][AD_D];
  // `faster`, the number of heads or of sequences, runs within x
  const int hi = blockIdx.x / faster, lo = blockIdx.x - hi * faster, split = blockIdx.y;
  const int kvh = faster == Hk ? lo : hi, b = faster == Hk ? hi : lo;
#define AD_PART(GO_ON, ...)                                                               \
  attn_part<G, TILED, GO_ON>(out, po, pml, q, kc, vc, bt, len, scale, B, Hk, page_size,   \
                             page_shift, max_pages, nsplit, qs, win, s_ml, s_o, kvh,      \
                             __VA_ARGS__)
  if constexpr (!CUT) {
    const int L = len[b], part = (visible(L, win).rounds + nsplit - 1) / nsplit;
    AD_PART(false, b, L, split * part, part, ((size_t)b * Hk + kvh) * nsplit + split, 0);
  } else {
    typedef const __attribute__((address_space(4))) CutRow* rows;
    const CutRow own = ((rows)cut)[b];
    const int share = own[0], part = own[2];
    if (share == 0) {
      AD_PART(false, b, own[1], split * part, part,
              (size_t)kvh * cap + b * nsplit + split, 0);
    } else {
      const int lane = threadIdx.x & 63, slot = split * B + b, at = slot * share;
      const CutRow seq = cut[min(lane, B - 1)];
      const unsigned long long behind = __ballot(lane < B && seq[3] > at);
      if (behind == 0) return;
      const int from = (int)__ffsll(behind) - 1;
      const int begin = from > 0 ? __builtin_amdgcn_readlane(seq[3], max(from - 1, 0)) : 0;
      const int now = min(share, __builtin_amdgcn_readlane(seq[3], from) - at);
      AD_PART(true, from, __builtin_amdgcn_readlane(seq[1], from), at - begin, now,
              (size_t)kvh * cap + slot + from, share - now);
    }
  }
#undef AD_PART
}

// Combine split partials: grid (B, Hq), one wave, 2 dims per lane.  A launch that is all
// latency: maxima, sums and partial outputs of up to NS splits (more go round again) are
// asked for together and wait once, not split by split (a decode step of 16 layers, one
// sequence of 387 tokens in 16 splits 1473 -> 1425 us, 12 of 4500..8000 in four 2074 ->
// 2050).  Splits behind the last repeat it; those without tokens, whose po was not
// written, are left out of the sum.
// CUT: the parts are asked for as if there were nsplit each, and again where there are
// shares, so that the cut is not waited for first.
template <int NS, bool CUT>
__global__ void __launch_bounds__(64) attn_decode_combine_kernel(
    u16* __restrict__ out, const float* __restrict__ po, const float* __restrict__ pml,
    const CutRow* __restrict__ cut, int Hq, int G, int nsplit, int cap) {
  const int b = blockIdx.x, h = blockIdx.y;
  const int kvh = h / G, g = h % G;
  const int Hk = Hq / G;
  const int lane = threadIdx.x;
  size_t first = CUT ? ((size_t)kvh * cap + b * nsplit) * G + g
                     : (((size_t)b * Hk + kvh) * nsplit) * G + g;
  int n = nsplit;

  f32x2 ml, v[NS];
  auto ask = [&](int s0) {
    ml = *reinterpret_cast<const f32x2*>(
        pml + (first + (size_t)min(s0 + lane, n - 1) * G) * 2);
#pragma unroll
    for (int i = 0; i < NS; ++i)
      v[i] = *reinterpret_cast<const f32x2*>(
          po + (first + (size_t)min(s0 + i, n - 1) * G) * AD_D + lane * 2);
  };
  if (CUT) {
    ask(0);
    const CutRow own = cut[b];
    const int share = own[0];
    if (share > 0) {
      const int start = b > 0 ? cut[b - 1][3] : 0, end = own[3], slot = start / share;
      n = end > start ? (end - 1) / share - slot + 1 : 0;
      first = ((size_t)kvh * cap + slot + b) * G + g;
      if (n > 0) ask(0);
    }
  }
  float L2 = 0.f, o0 = 0.f, o1 = 0.f, M = AF_NEG_INF;
  for (int s0 = 0; s0 < n; s0 += NS) {
    if (!CUT || s0 > 0) ask(s0);
    const bool mine = lane < NS && s0 + lane < n;
    const float pm = mine ? ml[0] : AF_NEG_INF, pl = mine ? ml[1] : 0.f;
    const float Mn = fmaxf(M, wave_max_f32(pm));
    const float back = (M <= AF_NEG_INF) ? 0.f : __builtin_amdgcn_exp2f(M - Mn);
    const float c = (pm <= AF_NEG_INF) ? 0.f : __builtin_amdgcn_exp2f(pm - Mn);
    L2 = L2 * back + wave_sum_f32(pl * c);
    o0 *= back;
    o1 *= back;
    M = Mn;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const float ci = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c), i));
      o0 = ci == 0.f ? o0 : fmaf(v[i][0], ci, o0);
      o1 = ci == 0.f ? o1 : fmaf(v[i][1], ci, o1);
    }
  }
  const float inv = (L2 > 0.f) ? 1.f / L2 : 0.f;
  u16x2 ov = {f2bf(o0 * inv), f2bf(o1 * inv)};
  *reinterpret_cast<u16x2*>(out + (size_t)b * (Hq * AD_D) + h * AD_D + lane * 2) = ov;
}

// Whether K/V heads run fastest in the grid.  With 8 of them every XCD then has one head of
// all sequences, long and short, where sequences first give it every eighth sequence
// (sequences / heads first in us: 32 of 300..1500 with 32 heads 83.5 / 71.3, 64 of
// 200..2000 with 8 heads, G = 8 68.9 / 58.9).  With fewer heads a sequence's heads and
// splits are spread over the XCDs and each looks up its pages anew: 8 of 300..3000 with 4
// heads 13.2 / 16.2, 16 of 1000 with 2 heads 11.8 / 14.3, 64 of 545 with 2 13.5 / 14.2;
// 4 heads unsplit: 128 of 100..1500 54.1 / 46.5, of 513..576 29.3 / 29.5.
static bool heads_first(int Hk, int nsplit) {
  return Hk >= 8 || (Hk >= 4 && nsplit == 1);
}

AF_EXPORT int af_attn_decode(void* out, void* po, void* pml, const void* q,
                             const void* kc, const void* vc, const void* bt,
                             const void* len, const void* cut, float scale, int B,
                             int Hq, int Hk, int D, int page_size, int max_pages,
                             int nsplit, int cap, i64 qs, int win, void* stream) {
  if (D != AD_D) return 9002;
  const int G = Hq / Hk;
  if (G < 1 || G > AD_MAXG || G * Hk != Hq) return 9003;
  if (B == 0) return 0;
  if (nsplit > 1 && cap < B * nsplit) return 9004;
  // B * nsplit shares are as many pieces and B - 1 at most
  const bool shares = cut && nsplit > 1 && nsplit <= 4 && B > 1 && B <= CUT_MAX &&
                      win <= 0 && cap >= B * (nsplit + 1) - 1;
  const int faster = heads_first(Hk, nsplit) ? Hk : B;
  const dim3 grid(B * Hk, nsplit), blk(64 * AD_WAVES);
  hipStream_t st = (hipStream_t)stream;
  const bool pow2 = (page_size & (page_size - 1)) == 0;
  const int shift = pow2 ? __builtin_ctz(page_size) : -1;
#define AF_LAUNCH2(GG, TT, CUT)                                                  \
  attn_decode_kernel<GG, TT, CUT><<<grid, blk, 0, st>>>(                         \
      (u16*)out, (float*)po, (float*)pml, (const u16*)q, (const u16*)kc,         \
      (const u16*)vc, (const i32*)bt, (const i32*)len, (const CutRow*)cut, scale, \
      B, Hk, page_size, shift, max_pages, nsplit, cap, qs, win, faster)
#define AF_LAUNCH1(GG, TT)                                                       \
  do {                                                                           \
    if (shares) AF_LAUNCH2(GG, TT, true);                                        \
    else AF_LAUNCH2(GG, TT, false);                                              \
  } while (0)
#define AF_LAUNCH(GG)                                                            \
  do {                                                                           \
    if (page_size % AD_TILE == 0) AF_LAUNCH1(GG, true);                          \
    else AF_LAUNCH1(GG, false);                                                  \
  } while (0)
  switch (G) {
    case 1: AF_LAUNCH(1); break;
    case 2: AF_LAUNCH(2); break;
    case 4: AF_LAUNCH(4); break;
    case 8: AF_LAUNCH(8); break;
    default: return 9003;
  }
#undef AF_LAUNCH
#undef AF_LAUNCH1
#undef AF_LAUNCH2
  if (nsplit > 1) {
    const dim3 g2(B, Hq);
#define AF_COMBINE(NS)                                                           \
  do {                                                                           \
    const auto merge = shares ? attn_decode_combine_kernel<NS, true>             \
                              : attn_decode_combine_kernel<NS, false>;           \
    merge<<<g2, 64, 0, st>>>((u16*)out, (const float*)po, (const float*)pml,     \
                             (const CutRow*)cut, Hq, G, nsplit, cap);             \
  } while (0)
    if (nsplit <= 4) AF_COMBINE(4);
    else if (nsplit <= 8) AF_COMBINE(8);
    else AF_COMBINE(16);
#undef AF_COMBINE
  }
  return af_last_err();
}

// The cut of a step whose embedding does not make it.
__global__ void __launch_bounds__(64) decode_cut_kernel(CutRow* __restrict__ cut,
                                                        const i32* __restrict__ len, int B,
                                                        int nsplit) {
  write_cut(cut, len, B, nsplit);
}

AF_EXPORT int af_decode_cut(void* cut, const void* len, int B, int nsplit, void* stream) {
  if (B < 1 || B > CUT_MAX || nsplit < 1) return 9002;
  decode_cut_kernel<<<1, 64, 0, (hipStream_t)stream>>>((CutRow*)cut, (const i32*)len, B, nsplit);
  return af_last_err();
}
