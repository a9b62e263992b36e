// Paged causal prefill attention (flash-style, GQA) on MFMA 32x32x16 bf16.
//
// q      : chunk rows at stride qs (view into the fused QKV buffer), head h
//          at offset h*D, D=128, packed by sequence (cu_seqlens of the CHUNK).
// kc/vc  : the paged KV cache [npages, Hk, page_size, D] — rope_cache has
//          already appended the chunk, so attention reads history + chunk
//          uniformly through the block table (chunked prefill falls out).
// qstart : per-seq absolute position of the chunk's first row (0 for a
//          full-prompt prefill; >0 when continuing a chunked prefill).
// out    : [chunk_T, Hq*D] bf16 contiguous.
//
// The rows of a sequence and the G query heads of one K/V head form G*len
// columns (column = row*G + head); a wave owns 32 of them.  Both products are
// computed transposed:
//   S^T [tokens x columns] = K Q^T: a lane gets 16 tokens of ONE column per 32
//     tokens, so maximum, sum and rescaling are per-lane values and a row
//     maximum crosses lanes once per tile (permlane32_swap).
//   O^T [dims x columns] = V^T P^T: the P fragment is the lane's own S^T
//     registers, rounded to bf16 in pairs; the contraction's token order inside
//     16 tokens is the one S^T came out in ({4h..4h+3, 8+4h..8+4h+3} for lane
//     half h), and V^T comes from row-major LDS by transposing reads
//     (ds_read_b64_tr_b16) in that order.  P never passes through LDS.
// K and V tiles go global -> LDS without registers (16 B per lane), chunks of 16 B
// permuted within the row by the row number, so that neither the b128 reads of K
// nor the transposing reads of V meet in a bank.
// Softmax works on powers of two; the running maximum moves only when a tile
// exceeds it by 2^6, which bounds P by 64 (relative rounding is unchanged) and
// saves rescaling the 64 output registers on most tiles.
//
//   attn_prefill_kernel  4 waves x 32 columns, K/V tiles of 64 tokens shared by
//     the block and double-buffered (64 KB, two blocks per CU: one wave's
//     exponentials run under the other's MFMA).  Bound by vector issue next to
//     the matrix cores (32 exponentials per lane and tile alone take half of the
//     tile's MFMA time, during which the cores are busy half of the time).  grid:
//     K/V head fastest, so with 8 of them an XCD's L2 keeps one head's K/V; late
//     (long) tiles start first.
//   attn_prefill_few_kernel  32 columns per block: sequences whose columns fit
//     one wave (verification of a few drafted tokens, single fed tokens), or all
//     of a batch too small to fill the chip with 128-column blocks.  The four
//     waves split the keys, each with private 32-token double buffers and no
//     barrier in the loop, and merge through LDS; with fewer than 256 blocks the
//     keys are also split over blocks and a second kernel merges.  Bound by the
//     latency of its transfers, which half a tile hides (129 KB of LDS, one block per
//     CU): ~4.2 TB/s of K/V where decode attention reaches 5.  P is kept to 16 bits
//     more: two bf16 terms, two products.
// Transfers: where pages hold whole tiles, the page of the tile after next is a scalar
// lookup behind the next tile's loads (as a vector load its wait drained them before
// this tile's arithmetic: 672 us and 43.9 against 628 and 37.0, one prompt of 8000 rows
// and 16 sequences of 5 rows behind up to 3000; with attend() as it is now 544 and
// 36.6).  The compiler still waits for them in front of the transposing reads, half a
// tile later; loads it does not know of changed little (628, 35.9).
// Fragment layouts (measured): A: lane holds A[m=lane&31][k=(lane>>5)*8+j]; B:
// B[k=(lane>>5)*8+j][n=lane&31]; C: reg r holds C[8*(r/4)+4*(lane>>5)+r%4][lane&31];
// transposing read: lane i of a group of 16 gets column i of 4 rows x 16 columns
// whose 8-byte pieces the group's lanes address row by row.
//
// Against 16x16x32 tiles of 64 columns with P through LDS and V transposed by
// scalar writes (one layer, 8 K/V heads, G = 4): one prompt of 8000 rows 2292 ->
// 544 us (229 -> 960 TFLOP/s), 20 of 300..700 384 -> 104 us, 8 x 2048 at G = 2
// 992 -> 232 us; 16 sequences of 5 rows behind 2400 tokens 387 -> 43 us.
#include "mfma_lines.h"

#define AP_D 128
#define AP_KV 64          // tokens per shared tile
#define AP_FEW 32         // tokens per wave-private tile
#define AP_ROWB 256       // bytes of a K or V row
#define AP_SPLITS 8       // shares of the keys at most

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) s16x8 lds_s16x8;

struct PrefillArgs {
  u16* out;
  const u16* q;
  const u16* kc;
  const u16* vc;
  const i32* bt;
  const i32* qstart;
  const i32* cu;
  float scale;      // positive
  float qmul;       // factor of q: the sign of the caller's scale, or a zero
  int nseq, Hq, Hk;
  i64 qs;
  int page_size, page_shift, max_pages, win;
  int few_cols;     // sequences of up to so many columns go to the few-kernel
};

__device__ __forceinline__ bf16x8 as_bf16x8(s16x8 v) {
  union { s16x8 s; bf16x8 b; } u;
  u.s = v;
  return u.b;
}

__device__ __forceinline__ float swap_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(v),
                                                  __float_as_int(v), false, false);
  return fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
}

// Sequence and place in it of work item `item`: items are pieces of 32 (FEW) or
// 128 columns, counted over the sequences that the kernel serves.
// By DPP and lane reads, with what the lanes have loaded: every workgroup waits for this, six
// shuffles one after the other and a second look at cu without (one prompt of 45 rows 9.2 ->
// 8.8 us, two of 200 18.6 -> 17.7, 20 of 300..680 96 -> 93).
struct Item { int seq, at, start, len; };
template <int G, bool FEW>
__device__ __forceinline__ Item find_item(const PrefillArgs& a, int item) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int s0 = 0; s0 < a.nseq; s0 += 64) {
    const int s = s0 + lane;
    int n = 0, start = 0, len = 0;
    if (s < a.nseq) {
      start = a.cu[s];
      len = a.cu[s + 1] - start;
      const int cols = len * G;
      if ((cols <= a.few_cols) == FEW) n = FEW ? (cols + 31) / 32 : (cols + 127) / 128;
    }
    int incl = n;   // the sum up to this lane: within 16 lanes, then over the rows before
#define AP_ADD(CTRL, ROWS) \
  incl += __builtin_amdgcn_update_dpp(0, incl, CTRL, ROWS, 0xf, false)
    AP_ADD(0x111, 0xf);
    AP_ADD(0x112, 0xf);
    AP_ADD(0x114, 0xf);
    AP_ADD(0x118, 0xf);
    AP_ADD(0x142, 0xa);
    AP_ADD(0x143, 0xc);
#undef AP_ADD
    const unsigned long long hit = __ballot(base + incl > item);
    if (hit) {
      const int l = __builtin_amdgcn_readfirstlane(__ffsll(hit) - 1);
      return {s0 + l,
              item - base - (__builtin_amdgcn_readlane(incl, l) - __builtin_amdgcn_readlane(n, l)),
              __builtin_amdgcn_readlane(start, l), __builtin_amdgcn_readlane(len, l)};
    }
    base += __builtin_amdgcn_readlane(incl, 63);
  }
  return {-1, 0, 0, 0};
}

// An entry of the block table whose index the wave shares, as a scalar load: after an LDS
// load the compiler makes it a vector load, and the wait for that drains the tile's loads.
__device__ __forceinline__ int table_entry(const i32* row, int i) {
  typedef const __attribute__((address_space(4))) i32 table_t;
  return ((table_t*)row)[__builtin_amdgcn_readfirstlane(i)];
}

// All but n of a wave's loads have landed, where the compiler can see it: it would wait
// for the next tile's loads as well in front of this tile's reads.
template <int N>
__device__ __forceinline__ void landed() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(vmcnt_only(N));
  asm volatile("" ::: "memory");
}

// Rows [row0, row0 + 4*N) of a K and a V tile whose first token is t0 into LDS:
// every instruction brings 4 rows (1 KB).  Tokens behind the last one repeat it
// (their weights are 0 and must meet finite values).
// page: the tile's page when it lies in one (TILED).
template <bool TILED, int N>
__device__ __forceinline__ void stage(const PrefillArgs& a, const i32* btrow,
                                      int kvh, int t0, int row0, int last,
                                      int page, lds_char* kl, lds_char* vl) {
  const int lane = threadIdx.x & 63;
  const int r4 = lane >> 4, slot = lane & 15;
  const int off0 =
      TILED ? (a.page_shift >= 0 ? t0 & (a.page_size - 1) : t0 % a.page_size) : 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int row = row0 + i * 4 + r4;
    size_t src;
    if (TILED) {
      src = ((size_t)page * a.Hk + kvh) * a.page_size + off0 +
            min(row, last - t0);
    } else {
      const int t = min(t0 + row, last);
      const int pi = a.page_shift >= 0 ? t >> a.page_shift : t / a.page_size;
      src = ((size_t)btrow[pi] * a.Hk + kvh) * a.page_size + (t - pi * a.page_size);
    }
    src *= AP_D;
    const int dst = (row0 + i * 4) * AP_ROWB;
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) uint32_t*)(
            a.kc + src + ((slot ^ (row & 15)) << 3)),
        (__attribute__((address_space(3))) uint32_t*)(kl + dst), 16, 0, 0);
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) uint32_t*)(
            a.vc + src + ((slot ^ ((row & 7) << 1)) << 3)),
        (__attribute__((address_space(3))) uint32_t*)(vl + dst), 16, 0, 0);
  }
}

// o += a b, in place: left to itself the compiler puts the result elsewhere and copies 64
// registers back per tile (together with the maximum in attend() 582 -> 569 us for one
// prompt of 8000 rows, 105 -> 93 for 20 of 300..700).  Two wait states for operands that
// were just written; who reads the sums other than as a sum again is behind settled().
__device__ __forceinline__ void add_product(f32x16& o, bf16x8 a, bf16x8 b) {
  asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0"
               : "+v"(o) : "v"(a), "v"(b));
}

// The matrix cores are done with the sums.
__device__ __forceinline__ void settled(f32x16 (&o)[4]) {
  asm volatile("s_nop 15\n\ts_nop 15" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]));
}

// A wave's columns and their running softmax.
struct Columns {
  s16x8 q[8];       // B operand, 8 x 16 dims
  f32x16 o[4];      // O^T, 4 x 32 dims
  float m, l;       // maximum of raw scores, sum over this lane half's tokens
  int qpos;         // absolute position of the column's row
};

// NB x 32 tokens from t0 of the tile at kl / vl.  masked: some column does not
// see some of them.  FINE: P as two bf16 terms.
template <int NB, bool FINE>
__device__ __forceinline__ void attend(Columns& c, const lds_char* kl,
                                       const lds_char* vl, int t0, float sc,
                                       int win, bool masked) {
  const int lane = threadIdx.x & 63;
  const int h = lane >> 5, n = lane & 31, i = lane & 15;
  f32x16 s[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[b][r] = 0.f;
  // operands are read one step ahead of their MFMA; the scheduling fences keep
  // the compiler from reading the whole tile ahead (it spilled 70 registers)
  const int kx = (h ^ (n & 15)) << 4;
  auto read_k = [&](int d, s16x8* f) {
    const lds_char* kp = kl + n * AP_ROWB + (kx ^ (d << 5));
#pragma unroll
    for (int b = 0; b < NB; ++b)
      f[b] = *reinterpret_cast<const lds_s16x8*>(kp + b * 32 * AP_ROWB);
  };
  s16x8 kf[2][NB];
  read_k(0, kf[0]);
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    if (d < 7) read_k(d + 1, kf[(d + 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < NB; ++b)
      s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          as_bf16x8(kf[d & 1][b]), as_bf16x8(c.q[d]), s[b], 0, 0, 0);
  }
  if (masked) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int t = t0 + b * 32 + 8 * (r / 4) + 4 * h + (r % 4);
        if (t > c.qpos || (win > 0 && t <= c.qpos - win))
          s[b][r] = -__builtin_inff();  // weight 0 under any positive scale
      }
  }
  // as a median with infinity: fmaxf first quiets NaNs that cannot signal, one more
  // instruction per score
  float mx[2] = {AF_NEG_INF, AF_NEG_INF};
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      mx[r & 1] = __builtin_amdgcn_fmed3f(mx[r & 1], s[b][r], __builtin_inff());
  const float top = swap_max(fmaxf(mx[0], mx[1]));
  if (__any((top - c.m) * sc > 6.f)) {
    settled(c.o);
    const float mn = fmaxf(c.m, top);
    const float corr = __builtin_amdgcn_exp2f((c.m - mn) * sc);
    c.m = mn;
    c.l *= corr;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) c.o[d][r] *= corr;
  }
  // a column that has seen nothing yet keeps weight 0 for masked tokens
  const float mz = (c.m <= AF_NEG_INF) ? 0.f : -c.m * sc;
  const int vx = ((4 * h + (i >> 2)) << 1);
  const lds_char* vp = vl + (4 * h + (i >> 2)) * AP_ROWB + (i & 1) * 8;
  const int ve = ((lane >> 4) & 1) * 2 + ((i & 3) >> 1);
  union VF { s16x4 half[2]; bf16x8 b; };
  auto read_v = [&](int k, VF* f) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const lds_char* at = vp + (((d * 4 + ve) ^ vx) << 4) + k * 16 * AP_ROWB;
      f[d].half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
      f[d].half[1] =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 8 * AP_ROWB));
    }
  };
  VF vf[2][4];
  read_v(0, vf[0]);
  float sum0 = 0.f, sum1 = 0.f;
  bf16x8 pf[2], pr[2];
  auto weigh = [&](int k, int u) {  // tokens 2u, 2u + 1 of the k-th 16
    const int r = (k & 1) * 8 + 2 * u;
    const float p0 = __builtin_amdgcn_exp2f(fmaf(s[k / 2][r], sc, mz));
    const float p1 = __builtin_amdgcn_exp2f(fmaf(s[k / 2][r + 1], sc, mz));
    sum0 += p0;
    sum1 += p1;
    bf16x8 &f = pf[k & 1], &e = pr[k & 1];
    f[2 * u] = (__bf16)p0;
    f[2 * u + 1] = (__bf16)p1;
    if (FINE) {
      e[2 * u] = (__bf16)(p0 - (float)f[2 * u]);
      e[2 * u + 1] = (__bf16)(p1 - (float)f[2 * u + 1]);
    }
  };
#pragma unroll
  for (int u = 0; u < 4; ++u) weigh(0, u);
  // a wave that has its weights goes first, so that the two of a SIMD do not multiply and
  // exponentiate in step (553 -> 535 us)
  __builtin_amdgcn_s_setprio(1);
#pragma unroll
  for (int k = 0; k < NB * 2; ++k) {  // 16 tokens; the next ones' weights in between, or
                                      // MFMA and vector unit take turns (569 -> 553 us)
    if (k + 1 < NB * 2) read_v(k + 1, vf[(k + 1) & 1]);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      __builtin_amdgcn_sched_barrier(0);
      add_product(c.o[d], vf[k & 1][d].b, pf[k & 1]);
      if (FINE) add_product(c.o[d], vf[k & 1][d].b, pr[k & 1]);
      if (k + 1 < NB * 2) weigh(k + 1, d);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_s_setprio(0);
  c.l += sum0 + sum1;
}

template <int G>
__device__ __forceinline__ void load_columns(const PrefillArgs& a, Columns& c,
                                             int row, int head, int seq_start,
                                             int len, int hist) {
  const int h = (threadIdx.x & 63) >> 5;
  const u16* qp = a.q + (size_t)(seq_start + min(row, len - 1)) * a.qs +
                  head * AP_D + h * 8;
#pragma unroll
  for (int d = 0; d < 8; ++d) c.q[d] = *reinterpret_cast<const s16x8*>(qp + d * 16);
  if (a.qmul != 1.f) {
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      union { s16x8 s; bf16x8 b; } u;
      u.s = c.q[d];
#pragma unroll
      for (int j = 0; j < 8; ++j) u.b[j] = (__bf16)((float)u.b[j] * a.qmul);
      c.q[d] = u.s;
    }
  }
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) c.o[d][r] = 0.f;
  c.m = AF_NEG_INF;
  c.l = 0.f;
  c.qpos = hist + min(row, len - 1);
}

template <int G, bool TILED>
__global__ void __launch_bounds__(256, 2) attn_prefill_kernel(PrefillArgs a,
                                                              int items) {
  constexpr int ROWS = 128 / G, WROWS = 32 / G;
  const int kvh = blockIdx.x % a.Hk;
  const Item it = find_item<G, false>(a, items - 1 - (int)(blockIdx.x / a.Hk));
  const int seq = it.seq, at = it.at;
  if (seq < 0) return;  // lengths on the device say less than the host's
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int seq_start = it.start, len = it.len;
  const int hist = a.qstart[seq];
  const i32* btrow = a.bt + (size_t)seq * a.max_pages;
  const int q0 = at * ROWS;

  __shared__ __attribute__((aligned(16))) char lds[2][2][AP_KV * AP_ROWB];
  auto kbuf = [&](int i) { return (lds_char*)&lds[i][0][0]; };
  auto vbuf = [&](int i) { return (lds_char*)&lds[i][1][0]; };

  const int col = lane & 31;
  const int row = q0 + wid * WROWS + col / G;
  const int qh = kvh * G + col % G;
  Columns c;
  load_columns<G>(a, c, row, qh, seq_start, len, hist);
  const float sc = a.scale * 1.44269504088896f;
  // positions of this wave's first and last row (none: no work but staging)
  const bool some = q0 + wid * WROWS < len;
  const int p0 = hist + q0 + wid * WROWS;
  const int p1 = hist + min(q0 + wid * WROWS + WROWS, len) - 1;

  // tokens visible to this block: history + chunk rows up to the causal bound,
  // and (sliding window) nothing below the first row's window
  const int last = hist + len - 1;
  const int ntiles = (min(last + 1, hist + q0 + ROWS) + AP_KV - 1) / AP_KV;
  int kt = a.win > 0 ? max(0, hist + q0 - a.win + 1) / AP_KV : 0;
  auto page_of = [&](int tile) {
    const int t = min(tile, ntiles - 1) * AP_KV;
    return table_entry(btrow, a.page_shift >= 0 ? t >> a.page_shift : t / a.page_size);
  };
  stage<TILED, 4>(a, btrow, kvh, kt * AP_KV, wid * 16, last,
                  TILED ? page_of(kt) : 0, kbuf(0), vbuf(0));
  int page = TILED ? page_of(kt + 1) : 0;
  int cur = 0;
  __syncthreads();
  for (; kt < ntiles; ++kt) {
    if (kt + 1 < ntiles) {
      stage<TILED, 4>(a, btrow, kvh, (kt + 1) * AP_KV, wid * 16, last, page,
                      kbuf(cur ^ 1), vbuf(cur ^ 1));
      if (TILED) page = page_of(kt + 2);
    }
    const int t0 = kt * AP_KV;
    if (some && t0 <= p1 && (a.win <= 0 || t0 + AP_KV - 1 > p0 - a.win)) {
      attend<2, false>(c, kbuf(cur), vbuf(cur), t0, sc, a.win,
                t0 + AP_KV - 1 > p0 || (a.win > 0 && t0 <= p1 - a.win));
    }
    __syncthreads();  // next tile has landed, this one is free
    cur ^= 1;
  }

  settled(c.o);
  const float l = c.l + __shfl_xor(c.l, 32, 64);
  if (row >= len) return;
  const float inv = (l > 0.f) ? 1.f / l : 0.f;
  u16* op = a.out + (size_t)(seq_start + row) * (a.Hq * AP_D) + qh * AP_D +
            4 * (lane >> 5);
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      s16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = (short)f2bf(c.o[d][r + j] * inv);
      *reinterpret_cast<s16x4*>(op + d * 32 + 2 * r) = v;
    }
}

// po [items, Hk, nsplit, 32, D] f32, pml [items, Hk, nsplit, 32, 2] f32: used
// with nsplit > 1 only.
template <int G, bool TILED>
__global__ void __launch_bounds__(256, 1) attn_prefill_few_kernel(
    PrefillArgs a, float* __restrict__ po, float* __restrict__ pml, int nsplit) {
  const int kvh = blockIdx.x % a.Hk;
  const Item it = find_item<G, true>(a, blockIdx.x / a.Hk);
  const int seq = it.seq, at = it.at;
  if (seq < 0) return;  // lengths on the device say less than the host's
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int seq_start = it.start, len = it.len;
  const int hist = a.qstart[seq];
  const i32* btrow = a.bt + (size_t)seq * a.max_pages;

  constexpr int TILE = AP_FEW * AP_ROWB, WROWS = 32 / G;
  // one array: with a second one the compiler waits for all loads before it reads
  __shared__ __attribute__((aligned(16))) char lds[4 * 4 * TILE + 1024];
  float (*s_m)[32] = reinterpret_cast<float (*)[32]>(lds + 16 * TILE), (*s_l)[32] = s_m + 4;
  auto kbuf = [&](int i) { return (lds_char*)&lds[(wid * 4 + i * 2) * TILE]; };
  auto vbuf = [&](int i) { return (lds_char*)&lds[(wid * 4 + i * 2 + 1) * TILE]; };

  const int col = lane & 31;
  const int row = at * WROWS + col / G, qh = kvh * G + col % G;
  const int nrows = min(WROWS, len - at * WROWS);
  Columns c;
  load_columns<G>(a, c, row, qh, seq_start, len, hist);
  const float sc = a.scale * 1.44269504088896f;
  const int last = hist + len - 1;
  const int p0 = hist + at * WROWS, p1 = p0 + nrows - 1;
  const int ntiles = (p1 + AP_FEW) / AP_FEW;
  const int first = a.win > 0 ? max(0, p0 - a.win + 1) / AP_FEW : 0;
  const int step = 4 * nsplit;
  auto page_of = [&](int tile) {
    const int t = min(tile, ntiles - 1) * AP_FEW;
    return table_entry(btrow, a.page_shift >= 0 ? t >> a.page_shift : t / a.page_size);
  };
  int kt = first + (int)blockIdx.y * 4 + wid, page = 0, cur = 0;
  if (kt < ntiles) {
    stage<TILED, 8>(a, btrow, kvh, kt * AP_FEW, 0, last, TILED ? page_of(kt) : 0,
                    kbuf(0), vbuf(0));
    if (TILED) page = page_of(kt + step);
  }
  for (; kt < ntiles; kt += step) {
    if (kt + step < ntiles) {
      stage<TILED, 8>(a, btrow, kvh, (kt + step) * AP_FEW, 0, last, page,
                      kbuf(cur ^ 1), vbuf(cur ^ 1));
      if (TILED) page = page_of(kt + 2 * step);
      landed<16>();      // all but the 16 loads just issued
    } else {
      landed<0>();
    }
    const int t0 = kt * AP_FEW;
    attend<1, true>(c, kbuf(cur), vbuf(cur), t0, sc, a.win,
                    t0 + AP_FEW - 1 > p0 || (a.win > 0 && t0 <= p1 - a.win));
    // this tile's reads are done before its buffer is filled again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    cur ^= 1;
  }

  // merge the waves: O^T as [wave][column][dim] in the tile buffers
  settled(c.o);
  const float l = c.l + __shfl_xor(c.l, 32, 64);
  __syncthreads();
  float* so = reinterpret_cast<float*>(lds);
  if (lane < 32) { s_m[wid][col] = c.m; s_l[wid][col] = l; }
  float* mine = so + (size_t)(wid * 32 + col) * AP_D + 4 * (lane >> 5);
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<f32x4*>(mine + d * 32 + 2 * r) =
          f32x4{c.o[d][r], c.o[d][r + 1], c.o[d][r + 2], c.o[d][r + 3]};
  __syncthreads();
  for (int i = threadIdx.x; i < nrows * G * (AP_D / 4); i += 256) {
    const int cc = i / (AP_D / 4), d = (i % (AP_D / 4)) * 4;
    float M = s_m[0][cc];
#pragma unroll
    for (int w = 1; w < 4; ++w) M = fmaxf(M, s_m[w][cc]);
    float L = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = (s_m[w][cc] <= AF_NEG_INF)
                          ? 0.f
                          : __builtin_amdgcn_exp2f((s_m[w][cc] - M) * sc);
      L += s_l[w][cc] * f;
      const f32x4 v = *reinterpret_cast<const f32x4*>(so + (size_t)(w * 32 + cc) * AP_D + d);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] += v[j] * f;
    }
    if (nsplit > 1) {
      const size_t to = ((size_t)blockIdx.x * nsplit + blockIdx.y) * 32 + cc;
      *reinterpret_cast<f32x4*>(po + to * AP_D + d) = o;
      if (d == 0) { pml[to * 2] = M; pml[to * 2 + 1] = L; }
      continue;
    }
    const float inv = (L > 0.f) ? 1.f / L : 0.f;
    s16x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (short)f2bf(o[j] * inv);
    *reinterpret_cast<s16x4*>(a.out +
                              (size_t)(seq_start + at * WROWS + cc / G) * (a.Hq * AP_D) +
                              (kvh * G + cc % G) * AP_D + d) = v;
  }
}

// Merge of the few-kernel's key splits; blocks as there.
template <int G>
__global__ void __launch_bounds__(256) attn_prefill_merge_kernel(
    PrefillArgs a, const float* __restrict__ po, const float* __restrict__ pml,
    int nsplit) {
  const int kvh = blockIdx.x % a.Hk;
  const Item it = find_item<G, true>(a, blockIdx.x / a.Hk);
  const int seq = it.seq, at = it.at;
  if (seq < 0) return;
  const int seq_start = it.start, len = it.len;
  const int row0 = at * (32 / G), nrows = min(32 / G, len - row0);
  const float sc = a.scale * 1.44269504088896f;
  const size_t from = (size_t)blockIdx.x * nsplit * 32;
  for (int i = threadIdx.x; i < nrows * G * (AP_D / 4); i += 256) {
    const int cc = i / (AP_D / 4), d = (i % (AP_D / 4)) * 4;
    // the splits' results are asked for together (those behind the last repeat it)
    f32x2 ml[AP_SPLITS];
    f32x4 part[AP_SPLITS];
#pragma unroll
    for (int s = 0; s < AP_SPLITS; ++s) {
      const size_t at = from + min(s, nsplit - 1) * 32 + cc;
      ml[s] = *reinterpret_cast<const f32x2*>(pml + at * 2);
      part[s] = *reinterpret_cast<const f32x4*>(po + at * AP_D + d);
    }
    float M = AF_NEG_INF;
#pragma unroll
    for (int s = 0; s < AP_SPLITS; ++s) M = fmaxf(M, ml[s][0]);
    float L = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < AP_SPLITS; ++s) {
      if (s >= nsplit) break;
      const float f = (ml[s][0] <= AF_NEG_INF) ? 0.f : __builtin_amdgcn_exp2f((ml[s][0] - M) * sc);
      L += ml[s][1] * f;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] += part[s][j] * f;
    }
    const float inv = (L > 0.f) ? 1.f / L : 0.f;
    s16x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (short)f2bf(o[j] * inv);
    *reinterpret_cast<s16x4*>(a.out +
                              (size_t)(seq_start + row0 + cc / G) * (a.Hq * AP_D) +
                              (kvh * G + cc % G) * AP_D + d) = v;
  }
}

// The kernels take the maximum of raw scores and mask before they scale, so scale
// must be positive there: a negative one changes the sign of q (exact), zero makes
// all scores zero.
// items: 128-column items of the sequences with more than few_cols columns; few:
// 32-column items of the others, their keys cut nsplit ways with the partial
// results in po / pml (all per K/V head).
AF_EXPORT int af_attn_prefill(void* out, void* po, void* pml, const void* q,
                              const void* kc, const void* vc, const void* bt,
                              const void* qstart, const void* cu_seqlens,
                              float scale, int nseq, int items, int few,
                              int few_cols, int nsplit, int Hq, int Hk, int D,
                              i64 qs, int page_size, int max_pages, int win,
                              void* stream) {
  if (D != AP_D) return 9002;
  const int G = Hq / Hk;
  if (G * Hk != Hq || (few > 0 && (nsplit < 1 || nsplit > AP_SPLITS))) return 9003;
  hipStream_t st = (hipStream_t)stream;
  const bool pow2 = (page_size & (page_size - 1)) == 0;
  const PrefillArgs a = {(u16*)out, (const u16*)q, (const u16*)kc, (const u16*)vc,
                         (const i32*)bt, (const i32*)qstart,
                         (const i32*)cu_seqlens,
                         scale > 0.f ? scale : scale < 0.f ? -scale : 1.f,
                         scale > 0.f ? 1.f : scale < 0.f ? -1.f : scale,
                         nseq, Hq, Hk, qs,
                         page_size, pow2 ? __builtin_ctz(page_size) : -1,
                         max_pages, win, few_cols};
  float* fo = (float*)po;
  float* fm = (float*)pml;
  const dim3 gf(few * Hk, nsplit);
#define AF_LAUNCH(GG)                                                           \
  do {                                                                          \
    if (items > 0) {                                                            \
      if (page_size % AP_KV == 0)                                               \
        attn_prefill_kernel<GG, true><<<items * Hk, 256, 0, st>>>(a, items);    \
      else                                                                      \
        attn_prefill_kernel<GG, false><<<items * Hk, 256, 0, st>>>(a, items);   \
    }                                                                           \
    if (few > 0) {                                                              \
      if (page_size % AP_FEW == 0)                                              \
        attn_prefill_few_kernel<GG, true><<<gf, 256, 0, st>>>(a, fo, fm, nsplit); \
      else                                                                      \
        attn_prefill_few_kernel<GG, false><<<gf, 256, 0, st>>>(a, fo, fm, nsplit); \
      if (nsplit > 1)                                                           \
        attn_prefill_merge_kernel<GG><<<few * Hk, 256, 0, st>>>(a, fo, fm, nsplit); \
    }                                                                           \
  } while (0)
  switch (G) {
    case 1: AF_LAUNCH(1); break;
    case 2: AF_LAUNCH(2); break;
    case 4: AF_LAUNCH(4); break;
    case 8: AF_LAUNCH(8); break;
    default: return 9003;
  }
#undef AF_LAUNCH
  return af_last_err();
}
