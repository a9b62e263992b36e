// Weight-streaming GEMMs for up to 128 rows:  Y[M,N] = X[M,K] @ W[N,K]^T with
// the step that follows it in a decoder layer.
//
// A decode step reads every weight once, so a layer's four projections are bound
// by the weight stream and by what a launch costs (~4.6 us in a captured step).
// Weights and X travel global -> LDS without registers, a whole 128-byte line per
// row and load: operand loads straight to registers (16 rows x 64 bytes per
// instruction) stop at ~7.6 TB/s of requests whatever is asked for, so X at 16
// rows doubled the time.  16-byte chunks are permuted within a line by the row
// number (the operand reads then do not meet in a bank).  Waits are counted, so that
// the loads of the next pieces stay in flight while one is multiplied.  All LDS of a
// kernel is one array: with a second one the compiler puts a full wait in front of
// the operand reads (SwiGLU over 28672 x 4096, one row: 38.7 us, 36.0 without it).
//
// gemm_rows_kernel, up to 16 rows: a block owns one tile of 16 weight rows (N =
//   4096 gives 256 tiles, one per CU; N = 28672 seven per CU) and K is split over
//   its 8 WAVES, which take 64-element pieces in turn, each through buffers of its
//   own: no barrier in the loop, no partial sums in memory and no second launch.
//   The waves' sums meet once, in LDS; results do not depend on M within this kernel.
//   The epilogue is the layer's next step: bf16 store, residual add in place,
//   SwiGLU (a tile is 8 gate and 8 up rows), or rotary embedding + page append (a
//   tile is 8 rotation pairs of a head, or 12 in 24 weight rows, see launch_rows).
//   RMSNorm (its weight is folded into W):
//   the loop multiplies every X fragment with itself (diagonal of X X^T, one
//   MFMA), so nobody has to leave row statistics behind.
// More rows: X would be read once per 16 weight rows, so here four or eight waves
//   share 64 or 128 weight rows and X, STAGES pieces in a ring with one barrier per
//   piece.
// gemm_parts_kernel, K split over blocks because N alone does not fill the chip: a
//   wave multiplies WT tiles of weights with a WT-th of X's rows (with WT = 1 every
//   wave reads all of X from LDS, 144 KB per piece at 128 rows; WT = 4 reads 96 KB).
//   The fp32 parts meet in the kernel that does the next step.  Bound by the parts
//   (16.8 MB at 128 rows, written at ~2.5 TB/s after the stream has ended: 7 of the 15
//   us of 4096 x 4096) and by starts, not by its loop: the loop below was no faster.
//   Unsplit, it also serves plain products of 97..128 rows without a norm, in blocks of
//   128 columns.
// gemm_tile_kernel, whole K (SwiGLU, plain): at 128 rows the loop of the kernel above
//   takes 0.47 us per piece without any load, nearly what the memory needs for the
//   128 weight rows of a piece (0.57), and the two did not overlap.  So half of the
//   waves take one half of a piece's K and half the other, each 64 weight rows by a
//   half of X's rows (64 KB of LDS reads per piece instead of 96), and the operands
//   of the next piece are read while one is multiplied: 0.2 us.  Rows of weights are
//   the first MFMA operand, so that a lane ends with four neighbouring columns of a
//   row; the norm scalars are made while the first pieces travel.  The epilogue takes
//   3 us instead of 8 of the 50.
//   SwiGLU over 28672 x 4096, alone / inside a step: 24 rows 40.1 -> 36.9, 64 rows
//   41.4 -> 38.9 / 44.2 -> 42.0, 80 rows (96 brought in instead of 128) 46.9 -> 41.8 /
//   51.7 -> 43.8, 128 rows 50.3 -> 48.0 / 57.2 -> 52.6; 16384 x 2048 at 128 rows 24.5 ->
//   19.6.  Deeper rings, in all or for the weights only, change nothing.
//
// Weight rows lie K * 2 bytes apart, usually a multiple of every channel
// interleave, so the rows of one piece come from the same memory channel and
// blocks that walk K in step ask the same channel for everything.  Blocks of an
// XCD therefore start at different pieces; where K is split the splits do that
// already and starting elsewhere costs a little (4096 x 4096 in four, 32 rows: 8.0 ->
// 8.8 us).  SwiGLU over 28672 x 4096: 42.9 -> 40.2 us at one row, 53.4 -> 45.2 at 64,
// 62.3 -> 57.3 at 128 (before the weights were streamed).  Two pieces per wave leave
// room for two blocks per CU, whose starts and ends overlap; three pieces with 8 rows
// of X each 36.4, four 43.7 (one block per CU).
// The order in which a column is summed depends on the kernel, the width of its
// blocks and the number of splits, and all three on M: the same row may differ by
// fp32 rounding between steps of different sizes.
// Measured in us, alone and repeated (inside a step 5-25% more), against the split-K
// kernel with two-stage buffers and its second launch (in brackets).  One row: 6144 x
// 4096 with rotary and append 10.7 (21.3 in three launches), 4096 x 4096 7.2 and 4096 x
// 14336 19.5 (together 44.4), SwiGLU over 28672 x 4096 36.0 = 6.5 TB/s (58.2).  16
// rows: 11.0, 8.0, 23.3, 41.2.  64 rows, without the closing launches: 13.1, 9.3,
// 23.3, 38.9 (16.7, o + down 44.8, 62.7).  128 rows: 16.9, 15.0, 27.5, 48.0 (library
// 25.6 and 57.5 + 5.2 for the first and the last, o + down 63.1).
#include "mfma_lines.h"

#include <climits>
#include <type_traits>

enum RowsEpi { EPI_PLAIN = 0, EPI_RESIDUAL = 1, EPI_SWIGLU = 2, EPI_ROPE = 3,
               EPI_PARTS = 4 };

struct RowsArgs {
  u16* out;            // [M, N] ([M, N/2] SwiGLU; [M, Hq*128] rope: q only)
  u16* residual;       // [M, N], updated in place (EPI_RESIDUAL)
  float* parts;        // [splits, M, N] (EPI_PARTS)
  const u16* X;
  const u16* W;
  int M, N, K;
  const float* ss;     // [M, 8] row sums of squares of X (norm 1)
  float eps;
  // EPI_ROPE
  const i32* pos;
  const float* table;  // [positions, 128]: cos | sin
  u16* kc;
  u16* vc;
  const i64* slot;
  int Hq, Hk, page_size;
};

// W row of row n of a 16-row tile
template <int EPI>
__device__ __forceinline__ int weight_row(const RowsArgs& a, int tile, int n) {
  if (EPI == EPI_SWIGLU) return (n < 8 ? 0 : (a.N >> 1) - 8) + tile * 8 + n;
  if (EPI == EPI_ROPE) {
    const int head = tile >> 3, j = tile & 7;
    return head * 128 + (head >= a.Hq + a.Hk ? j * 16 + n
                                             : j * 8 + n + (n < 8 ? 0 : 56));
  }
  return tile * 16 + n;
}

// The same of the 24-row tiles of EPI_ROPE, three groups of 8 rows: four rotation pairs of a
// head each, or eight rows of v.
__device__ __forceinline__ int rope_group_row(const RowsArgs& a, int group, int j) {
  const int head = group >> 4, at = group & 15;
  return head * 128 + (head >= a.Hq + a.Hk ? at * 8 + j : at * 4 + (j & 3) + (j & 4) * 16);
}

// Rotated q / k pair (dims d, d + 64) or plain v pair (dims d, d + 1) of row m to
// its place.  head counts q, k, v heads in turn.
__device__ __forceinline__ void put_rope(const RowsArgs& a, int m, int head, int d,
                                         float x1, float x2) {
  const bool is_q = head < a.Hq, is_v = head >= a.Hq + a.Hk;
  const i64 s = a.slot[m];
  const i64 page = (s >= 0) ? s / a.page_size : 0;
  const i64 off = (s >= 0) ? s % a.page_size : 0;
  if (is_v) {
    if (s < 0) return;
    u16* row = a.vc + (((size_t)page * a.Hk + head - a.Hq - a.Hk) * a.page_size +
                       off) * 128 + d;
    *reinterpret_cast<u16x2*>(row) = u16x2{f2bf(x1), f2bf(x2)};
    return;
  }
  const float* tab = a.table + (size_t)a.pos[m] * 128 + d;
  const float cs = tab[0], sn = tab[64];
  const u16 y1 = f2bf(x1 * cs - x2 * sn), y2 = f2bf(x2 * cs + x1 * sn);
  if (is_q) {
    u16* row = a.out + (size_t)m * (a.Hq * 128) + head * 128 + d;
    row[0] = y1;
    row[64] = y2;
  } else if (s >= 0) {
    u16* row = a.kc + (((size_t)page * a.Hk + head - a.Hq) * a.page_size + off) *
                          128 + d;
    row[0] = y1;
    row[64] = y2;
  }
}

// NORM: 0 none, 1 from ss, 2 computed from X.  PD pieces per wave in flight, with DRAIN
// until the next is needed.  Tiles of WL x 8 weight rows: 2, or 3 with EPI_ROPE.
template <int PD, int EPI, int NORM, int AUX, bool DRAIN, int WL>
__device__ __forceinline__ void rows_block(const RowsArgs& a, const int tile) {
  constexpr int NW = 8;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int n = lane & 15;

  static_assert(WL == 2 || (WL == 3 && EPI == EPI_ROPE), "tiles");
  constexpr int PIECE = WL * 1024;               // 8 WL rows x 64 elements
  constexpr int SLOT = PIECE + 2048;             // of W and of X
  constexpr int RS = 20;                         // column stride of the sums
  constexpr int RING = NW * PD * SLOT;
  constexpr int SUMS = NW * WL * 8 * RS * 4;
  // one array for everything: with a second one the compiler waits for all loads
  // in front of the loop's reads
  constexpr int TAIL = SUMS + (NW + 1) * 16 * 4;
  __shared__ __attribute__((aligned(16))) char lds[RING > TAIL ? RING : TAIL];
  lds_b* ring = (lds_b*)&lds[wid * PD * SLOT];

  // sources of this lane's chunks
  const int r8 = lane >> 3, ch = ((lane & 7) ^ r8) * 8 + wid * 64;
  const u16 *wp[WL], *xp[2];
#pragma unroll
  for (int g = 0; g < WL; ++g)
    wp[g] = a.W + (size_t)(WL == 3 ? rope_group_row(a, tile * 3 + g, r8)
                                   : weight_row<EPI>(a, tile, g * 8 + r8)) * a.K + ch;
#pragma unroll
  for (int g = 0; g < 2; ++g) xp[g] = a.X + (size_t)min(g * 8 + r8, a.M - 1) * a.K + ch;
  const int cnt = ((a.K >> 6) - wid + NW - 1) / NW;  // this wave's pieces
  const int rot = cnt > 0 ? (tile >> 3) % cnt : 0;
  auto load = [&](int i) {
    lds_b* to = ring + (i % PD) * SLOT;
    const int p = i + rot < cnt ? i + rot : i + rot - cnt;
    const size_t off = (size_t)p * (NW * 64);
#pragma unroll
    for (int g = 0; g < WL; ++g) load_line8<AUX>(wp[g] + off, to + g * 1024);
#pragma unroll
    for (int g = 0; g < 2; ++g)
      load_line8<KEEP>(xp[g] + off, to + PIECE + g * 1024);
  };
  f32x4 acc[WL - 1], sq = {0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < WL - 1; ++t) acc[t] = f32x4{0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < PD; ++s)
    if (s < cnt) load(s);
  for (int i = 0; i < cnt; ++i) {
    // piece i has landed when only the loads of the PD - 1 behind it are out
    if (!DRAIN && i + PD <= cnt)
      __builtin_amdgcn_s_waitcnt(vmcnt_only((WL + 2) * (PD - 1)));
    else
      __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    asm volatile("" ::: "memory");
    const lds_b* at = ring + (i % PD) * SLOT;
    // the second 16 rows of 24 end in the rows of X, whose products nobody stores
    bf16x8r w[2][WL - 1], x[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int t = 0; t < WL - 1; ++t) w[h][t] = frag(at + t * 2048, h);
      x[h] = frag(at + PIECE, h);
    }
    // the slot is read: fill it again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (i + PD < cnt) load(i + PD);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int t = 0; t < WL - 1; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[h], w[h][t], acc[t], 0, 0, 0);
      if (NORM == 2)
        sq = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[h], x[h], sq, 0, 0, 0);
    }
  }

  // meet in LDS: [wave][tile column][row]; + 4 spreads the columns over banks
  __syncthreads();
  float (*red)[WL * 8][RS] = reinterpret_cast<float (*)[WL * 8][RS]>(lds);
  float (*rsq)[16] = reinterpret_cast<float (*)[16]>(lds + SUMS);
  float* rstd = rsq[NW];
  *reinterpret_cast<f32x4*>(&red[wid][n][(lane >> 4) * 4]) = acc[0];
  if (WL == 3 && n < 8)
    *reinterpret_cast<f32x4*>(&red[wid][16 + n][(lane >> 4) * 4]) = acc[WL - 2];
  if (NORM == 2) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if ((lane >> 4) * 4 + r == n) rsq[wid][n] = sq[r];
  }
  __syncthreads();
  if (NORM != 0) {
    if ((int)threadIdx.x < a.M) {
      const int m = threadIdx.x;
      float s = 0.f;
      if (NORM == 2) {
#pragma unroll
        for (int w = 0; w < NW; ++w) s += rsq[w][m];
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) s += a.ss[m * 8 + j];
      }
      rstd[m] = rsqrtf(s * (1.f / (float)a.K) + a.eps);
    }
    __syncthreads();
  }
  auto total = [&](int c, int m) {
    float s = red[0][c][m];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += red[w][c][m];
    return NORM != 0 ? s * rstd[m] : s;
  };

  // two values per thread: neighbours, or a gate / rotation pair
  if constexpr (WL == 3) {
    const int m = threadIdx.x / 12, j = threadIdx.x % 12, c = (j >> 2) * 8, i = j & 3;
    if (m >= a.M) return;
    const int group = tile * 3 + (j >> 2), head = group >> 4, at = group & 15;
    if (head >= a.Hq + a.Hk)
      put_rope(a, m, head, at * 8 + 2 * i, total(c + 2 * i, m), total(c + 2 * i + 1, m));
    else
      put_rope(a, m, head, at * 4 + i, total(c + i, m), total(c + 4 + i, m));
    return;
  }
  const int m = threadIdx.x >> 3, j = threadIdx.x & 7;
  if (m >= a.M) return;
  if (EPI == EPI_SWIGLU) {
    const float g = total(j, m), u = total(8 + j, m);
    a.out[(size_t)m * (a.N >> 1) + tile * 8 + j] = f2bf(g / (1.f + __expf(-g)) * u);
  } else if (EPI == EPI_ROPE) {
    const int head = tile >> 3, jt = tile & 7;
    if (head >= a.Hq + a.Hk)
      put_rope(a, m, head, jt * 16 + 2 * j, total(2 * j, m), total(2 * j + 1, m));
    else
      put_rope(a, m, head, jt * 8 + j, total(j, m), total(8 + j, m));
  } else {
    const size_t at = (size_t)m * a.N + tile * 16 + 2 * j;
    float v0 = total(2 * j, m), v1 = total(2 * j + 1, m);
    if (EPI == EPI_RESIDUAL) {
      const u16x2 r = *reinterpret_cast<const u16x2*>(a.residual + at);
      v0 += bf2f(r[0]);
      v1 += bf2f(r[1]);
      *reinterpret_cast<u16x2*>(a.residual + at) = u16x2{f2bf(v0), f2bf(v1)};
      if (a.out == nullptr) return;
    }
    *reinterpret_cast<u16x2*>(a.out + at) = u16x2{f2bf(v0), f2bf(v1)};
  }
}

template <int PD, int EPI, int NORM, int AUX, bool DRAIN, int WL = 2>
__global__ void __launch_bounds__(512) gemm_rows_kernel(RowsArgs a) {
  rows_block<PD, EPI, NORM, AUX, DRAIN, WL>(a, blockIdx.x);
}

// Several plain products of as many rows in one launch, the longest inner dimension first:
// alone, those of small weights are launches and latency (rows against 2048 x 2048 4.1 us).
// Of a 1b hybrid layer, 6 rows: 8192 x 2048, 10240 x 2048 and 2048 x 2048 20.5 us in three
// launches, 15.2 in one (5.5 TB/s); 2048 x 8192, 2048 x 2048 and 2048 x 1024 17.0, 12.8; one
// row 19.6, 15.3 and 16.2, 10.5.  Two of larger weights gain the launch, 4096 x 4096 and
// 4096 x 14336 28.0, 26.4.
#define GROUP_MAX 4
struct RowsGroup {
  struct Part {
    u16* out;
    const u16 *X, *W;
    int N, K, tile0;
  } part[GROUP_MAX];
  int parts, M;
};

template <int AUX>
__global__ void __launch_bounds__(512) gemm_rows_group_kernel(RowsGroup g) {
  int i = 0;
  while (i + 1 < g.parts && (int)blockIdx.x >= g.part[i + 1].tile0) ++i;
  const RowsGroup::Part& p = g.part[i];
  RowsArgs a = {};
  a.out = p.out;
  a.X = p.X;
  a.W = p.W;
  a.M = g.M;
  a.N = p.N;
  a.K = p.K;
  rows_block<2, EPI_PLAIN, 0, AUX, false, 2>(a, blockIdx.x - p.tile0);
}

// All but N of a wave's loads have landed, its LDS reads are done, and so it is for
// every wave of the block.
template <int N>
__device__ __forceinline__ void wait_loads_and_meet() {
  static_assert(N == 0 || N == 3 || N == 4 || N == 6 || N == 8, "wait counts");
  if constexpr (N == 0)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  else if constexpr (N == 3)
    asm volatile("s_waitcnt vmcnt(3) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  else if constexpr (N == 4)
    asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  else if constexpr (N == 6)
    asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  else
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Split K: MT 16-row groups of X (even), ring of STAGES pieces of K = 64, the sums to
// the parts (EPI_PARTS); unsplit, EPI_PLAIN.  Grid (N / (16 NW), splits).
template <int MT, int NW, int WT, int STAGES, int EPI, int AUX>
__global__ void __launch_bounds__(64 * NW) gemm_parts_kernel(RowsArgs a) {
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int n = lane & 15;
  constexpr int PIECE = 2048;
  constexpr int STAGE = PIECE * (NW + MT);
  constexpr int XG = 2 * MT / NW;                // 8-row groups of X per wave
  constexpr int PER = 2 + XG;                    // loads per wave and stage
  static_assert(XG * NW == 2 * MT, "X rows divide among the waves");
  __shared__ __attribute__((aligned(16))) char lds[STAGES * STAGE];
  lds_b* ring = (lds_b*)&lds[0];

  const int tile = blockIdx.x * NW + wid;         // the 16 weight rows it fetches
  const int pieces = a.K >> 6;
  const int per = (pieces + (int)gridDim.y - 1) / (int)gridDim.y;
  const int p0 = (int)blockIdx.y * per;
  const int cnt = min(pieces, p0 + per) - p0;    // none empty (checked at launch)
  const int r8 = lane >> 3, ch = ((lane & 7) ^ r8) * 8 + p0 * 64;
  const u16* wp[2];
  const u16* xp[XG];
#pragma unroll
  for (int g = 0; g < 2; ++g)
    wp[g] = a.W + (size_t)weight_row<EPI_PARTS>(a, tile, g * 8 + r8) * a.K + ch;
#pragma unroll
  for (int g = 0; g < XG; ++g)
    xp[g] = a.X + (size_t)min((wid * XG + g) * 8 + r8, a.M - 1) * a.K + ch;
  const int rot = cnt == a.K >> 6 ? ((int)blockIdx.x >> 3) * 2 % cnt : 0;
  auto load = [&](int i) {
    lds_b* to = ring + (i % STAGES) * STAGE;
    const size_t off = (size_t)(i + rot < cnt ? i + rot : i + rot - cnt) * 64;
#pragma unroll
    for (int g = 0; g < 2; ++g)
      load_line8<AUX>(wp[g] + off, to + wid * PIECE + g * 1024);
#pragma unroll
    for (int g = 0; g < XG; ++g)
      load_line8<KEEP>(xp[g] + off, to + NW * PIECE + (wid * XG + g) * 1024);
  };
  constexpr int MW = MT / WT;
  static_assert(NW % WT == 0 && MT % WT == 0, "products divide among the waves");
  const int w0 = wid / WT * WT, m0 = wid % WT * MW;   // the products it computes
  f32x4 acc[WT][MW];
#pragma unroll
  for (int t = 0; t < WT; ++t)
#pragma unroll
    for (int m = 0; m < MW; ++m) acc[t][m] = f32x4{0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < cnt) load(s);
  for (int i = 0; i < cnt; ++i) {
    // stage i is complete for everybody, and stage i - 1 read by everybody
    if (i + STAGES - 2 < cnt) wait_loads_and_meet<PER * (STAGES - 2)>();
    else wait_loads_and_meet<0>();
    if (i + STAGES - 1 < cnt) load(i + STAGES - 1);
    const lds_b* at = ring + (i % STAGES) * STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8r w[WT];
#pragma unroll
      for (int t = 0; t < WT; ++t) w[t] = frag(at + (w0 + t) * PIECE, h);
#pragma unroll
      for (int m = 0; m < MW; ++m) {
        const bf16x8r x = frag(at + PIECE * (NW + m0 + m), h);
#pragma unroll
        for (int t = 0; t < WT; ++t)
          acc[t][m] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w[t], acc[t][m], 0, 0, 0);
      }
    }
  }

  // lane: column n of each tile, rows (m0 + m)*16 + (lane>>4)*4 + r
#pragma unroll
  for (int m = 0; m < MW; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = (m0 + m) * 16 + (lane >> 4) * 4 + r;
#pragma unroll
      for (int t = 0; t < WT; ++t) {
        const int c = (blockIdx.x * NW + w0 + t) * 16 + n;
        if (row >= a.M) continue;
        if (EPI == EPI_PARTS)
          a.parts[((size_t)blockIdx.y * a.M + row) * a.N + c] = acc[t][m][r];
        else
          a.out[(size_t)row * a.N + c] = f2bf(acc[t][m][r]);
      }
    }
}

// Four neighbours of a row of the caller's output, whose address is a multiple of 4 bytes
// only (the hardware needs no more for a store of 8).
typedef u16x4 __attribute__((aligned(4))) row_u16x4;

// Whole K: MT 16-row groups of X (even), NT 16-row tiles of weights (4 or 8), NW
// waves, a ring of STAGES pieces of K = 64.  Grid N / (16 NT).  EPI_PLAIN, EPI_SWIGLU.
template <int MT, int NT, int NW, int STAGES, int EPI, int NORM, int AUX>
__global__ void __launch_bounds__(64 * NW) gemm_tile_kernel(RowsArgs a) {
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int n = lane & 15;
  constexpr int PIECE = 2048;
  constexpr int STAGE = PIECE * (NT + MT);
  constexpr int WG = 2 * NT / NW;                // 8-row lines of W per wave
  constexpr int XH = 4 * MT / NW;                // 4-row half lines of X per wave
  constexpr int XG = (XH + 1) / 2;               // X loads, the last may be a half
  constexpr int PER = WG + XG;                   // loads per wave and stage
  constexpr int RP = NW / 2 / (NT / 4);          // parts of X's groups
  constexpr int MW = MT / RP;                    // X groups of a wave's products
  static_assert(WG * NW == 2 * NT && XH * NW == 4 * MT && MW * RP == MT, "shares");
  static_assert(NW * 2 * MW * 1024 <= STAGES * STAGE, "half of the sums fit");
  static_assert(STAGES >= 2 && STAGES <= 6 && PER * 4 < 64, "wait counts");
  // one array for everything: with a second one the compiler waits for all loads
  // in front of the loop's reads
  __shared__ __attribute__((aligned(16))) char lds[STAGES * STAGE + MT * 64];
  lds_b* const ring = (lds_b*)&lds[0];
  float* const rstd = reinterpret_cast<float*>(lds + STAGES * STAGE);

  const int cnt = a.K >> 6;
  const int r8 = lane >> 3;
  const u16* wp[WG];
  const u16* xp[XG];
#pragma unroll
  for (int g = 0; g < WG; ++g) {
    const int line = wid * WG + g;
    wp[g] = a.W + (size_t)weight_row<EPI>(a, blockIdx.x * NT + line / 2,
                                          (line & 1) * 8 + r8) * a.K +
            ((lane & 7) ^ r8) * 8;
  }
#pragma unroll
  for (int g = 0; g < XG; ++g) {
    const int row = wid * XH * 4 + g * 8 + r8;
    xp[g] = a.X + (size_t)min(row, a.M - 1) * a.K + ((lane & 7) ^ (row & 7)) * 8;
  }
  // the piece and slot to load next
  int pnext = ((int)blockIdx.x >> 3) * 2 % cnt, snext = 0;
  auto load = [&]() {
    lds_b* to = ring + snext * STAGE;
    const int off = pnext * 64;
#pragma unroll
    for (int g = 0; g < WG; ++g)
      load_line8<AUX>(wp[g] + off, to + (wid * WG + g) * 1024);
#pragma unroll
    for (int g = 0; g < XG; ++g)
      if (2 * g + 2 <= XH || lane < 32)
        load_line8<KEEP>(xp[g] + off, to + NT * PIECE + wid * XH * 512 + g * 1024);
    pnext = pnext + 1 == cnt ? 0 : pnext + 1;
    snext = snext + 1 == STAGES ? 0 : snext + 1;
  };
  // products: a half of every piece's K, 4 tiles of weights, a part of X's groups
  const int kh = wid / (NW / 2), role = wid % (NW / 2);
  const int w0 = role / RP * 4, m0 = role % RP * MW;
  f32x4 acc[4][MW];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int m = 0; m < MW; ++m) acc[t][m] = f32x4{0, 0, 0, 0};
  int slot = 0;                                  // of the piece to read next
  auto read = [&](bf16x8r (&w)[4], bf16x8r (&x)[MW]) {
    const lds_b* at = ring + slot * STAGE;
#pragma unroll
    for (int t = 0; t < 4; ++t) w[t] = frag(at + (w0 + t) * PIECE, kh);
#pragma unroll
    for (int m = 0; m < MW; ++m) x[m] = frag(at + (NT + m0 + m) * PIECE, kh);
    slot = slot + 1 == STAGES ? 0 : slot + 1;
  };
  // piece i + 1 is complete for everybody, and piece i read by everybody: its slot
  // is filled again, and while i is multiplied the operands of i + 1 are read
  auto step = [&](int i, const bf16x8r (&w)[4], const bf16x8r (&x)[MW],
                  bf16x8r (&wn)[4], bf16x8r (&xn)[MW]) {
    if (i + 1 < cnt) {
      meet<PER>(min(STAGES - 2, cnt - 2 - i));
      if (i + STAGES < cnt) load();
      read(wn, xn);
    } else {
      __builtin_amdgcn_s_waitcnt(vmcnt_only(0) & ~0x0f00);
    }
#pragma unroll
    for (int m = 0; m < MW; ++m)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        acc[t][m] =
            __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t], x[m], acc[t][m], 0, 0, 0);
  };
#pragma unroll 1
  for (int s = 0; s < min(STAGES, cnt); ++s) load();
  if (NORM == 1) {
    const int row = threadIdx.x;
    if (row < MT * 16) {
      const float* sp = a.ss + (size_t)min(row, a.M - 1) * 8;
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) s += sp[j];
      rstd[row] = rsqrtf(s * (1.f / (float)a.K) + a.eps);
    }
  }
  bf16x8r wa[4], xa[MW], wb[4], xb[MW];
  meet<PER>(min(STAGES, cnt) - 1);
  read(wa, xa);
#pragma unroll 1
  for (int i = 0; i < cnt; i += 2) {
    step(i, wa, xa, wb, xb);
    if (i + 1 < cnt) step(i + 1, wb, xb, wa, xa);
  }

  // the two waves of a product swap sums: each finishes two of its tiles
  __syncthreads();
  f32x4* give = reinterpret_cast<f32x4*>(lds) + (wid * 2 * MW) * 64 + lane;
  const f32x4* take = reinterpret_cast<const f32x4*>(lds) +
                      ((wid ^ (NW / 2)) * 2 * MW) * 64 + lane;
  f32x4 sum[2][MW];
  auto swap = [&](auto upper) {
    constexpr int U = decltype(upper)::value;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int m = 0; m < MW; ++m) {
        give[(t * MW + m) * 64] = acc[2 - 2 * U + t][m];
        sum[t][m] = acc[2 * U + t][m];
      }
  };
  if (kh == 0) swap(std::integral_constant<int, 0>{});
  else swap(std::integral_constant<int, 1>{});
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int m = 0; m < MW; ++m) sum[t][m] += take[(t * MW + m) * 64];

  // lane: row n of each group, columns (lane >> 4) * 4 .. + 4 of each tile
  const int tile = blockIdx.x * NT + w0 + kh * 2;
#pragma unroll
  for (int m = 0; m < MW; ++m) {
    const int row = (m0 + m) * 16 + n;
    if (NORM == 1) {
      const float f = rstd[row];
#pragma unroll
      for (int t = 0; t < 2; ++t) sum[t][m] *= f;
    }
    if (EPI == EPI_SWIGLU) {
      // gate rows lie in the lower lanes and up rows in the upper ones: the lower
      // lanes get both of the first tile, the upper ones both of the second
      u16x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const auto gu = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(sum[0][m][r]), __float_as_uint(sum[1][m][r]), false, false);
        const float v = __uint_as_float(gu[0]), u = __uint_as_float(gu[1]);
        o[r] = f2bf(v / (1.f + __expf(-v)) * u);
      }
      if (row < a.M)
        *reinterpret_cast<row_u16x4*>(a.out + (size_t)row * (a.N >> 1) +
                                  (tile + (lane >> 5)) * 8 + (lane >> 4 & 1) * 4) = o;
    } else if (row < a.M) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const size_t at = (size_t)row * a.N + (tile + t) * 16 + (lane >> 4) * 4;
        const f32x4 v = sum[t][m];
        *reinterpret_cast<row_u16x4*>(a.out + at) =
            u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
      }
    }
  }
}

// What adds the parts runs an eighth of the columns on each XCD (blockIdx.x): the tiles of
// the products that wrote them there, every eighth, all splits of which are on one XCD where
// the tiles are a multiple of 8.  The rotary launch walks heads, tiles of 128 columns; of
// tiles of 64 (QKV of 17 to 32 rows in several splits) a head is two XCDs', as its rotation
// pairs are.  With rows on the XCDs instead (row modulo 8, or any) the products that write the
// same parts next were slower, the launches themselves faster.  In us under the profiler, rows
// / columns, 20, 45, 80 and 128 rows: 6144 x 4096 11.0 12.7 15.2 17.2 / 11.0 11.4 13.5 14.8 and
// rotary 4.0 4.1 4.6 5.3 / 4.7 4.6 4.6 4.8; 4096 x 4096 8.3 9.4 13.1 15.1 / 8.2 9.0 10.5 12.2
// and its residual 2.8 4.0 4.1 4.8 / 4.0 4.7 4.8 4.8; 4096 x 14336 and its residual level.  A
// layer's four products with these, replayed: 17 rows 86.0 / 85.4, 32 89.3 / 88.7, 45 94.8 /
// 92.9, 64 99.2 / 97.2, 80 110.8 / 105.6, 128 125.8 / 121.9.

// The parts' sum + rotary positions + page append: grid (8, M, heads / 64), every eighth head
// a wave, a rotation (or value) pair per lane.
__global__ void __launch_bounds__(512) rows_rope_kernel(RowsArgs a, int splits) {
  const int m = blockIdx.y, lane = threadIdx.x & 63;
  const int head = blockIdx.x + 8 * (blockIdx.z * 8 + (threadIdx.x >> 6));
  if (head >= a.Hq + 2 * a.Hk) return;
  const bool is_v = head >= a.Hq + a.Hk;
  const int d = is_v ? 2 * lane : lane, step = is_v ? 1 : 64;
  float x1 = 0.f, x2 = 0.f;
  for (int s = 0; s < splits; ++s) {
    const float* p = a.parts + ((size_t)s * a.M + m) * a.N + head * 128 + d;
    x1 += p[0];
    x2 += p[step];
  }
  float q = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) q += a.ss[m * 8 + j];
  const float rstd = rsqrtf(q * (1.f / (float)a.K) + a.eps);
  put_rope(a, m, head, d, x1 * rstd, x2 * rstd);
}

// The parts' sum + residual (in place; a copy to `out` if given) + sums of squares
// of the new rows (if ss is given): grid (8, M), a block per eighth of a row, every eighth
// tile of `tile` columns (0: neighbours).
__global__ void __launch_bounds__(256) rows_residual_kernel(
    u16* __restrict__ residual, u16* __restrict__ out,
    const float* __restrict__ parts, float* __restrict__ ss, int M, int N,
    int splits, int tile) {
  const int m = blockIdx.y, nb = N / 8;
  __shared__ float red[4];
  float local = 0.f;
  for (int i = threadIdx.x * 2; i < nb; i += 512) {
    const int c = tile ? (i / tile * 8 + blockIdx.x) * tile + i % tile : blockIdx.x * nb + i;
    const u16x2 rv = *reinterpret_cast<const u16x2*>(residual + (size_t)m * N + c);
    float v0 = 0.f, v1 = 0.f;
#pragma unroll 4
    for (int s = 0; s < splits; ++s) {
      const f32x2 p =
          *reinterpret_cast<const f32x2*>(parts + ((size_t)s * M + m) * N + c);
      v0 += p[0];
      v1 += p[1];
    }
    const u16x2 o = {f2bf(v0 + bf2f(rv[0])), f2bf(v1 + bf2f(rv[1]))};
    *reinterpret_cast<u16x2*>(residual + (size_t)m * N + c) = o;
    if (out) *reinterpret_cast<u16x2*>(out + (size_t)m * N + c) = o;
    const float b0 = bf2f(o[0]), b1 = bf2f(o[1]);  // stats of the rounded value
    local += b0 * b0 + b1 * b1;
  }
  if (!ss) return;
  local = wave_sum_f32(local);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = local;
  __syncthreads();
  if (threadIdx.x == 0)
    ss[m * 8 + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// The parts' sum in bf16, rows optionally scaled by the RMSNorm scalar from ss.
__global__ void __launch_bounds__(256) rows_sum_kernel(
    u16* __restrict__ out, const float* __restrict__ parts,
    const float* __restrict__ ss, int M, int N, int splits, float inv_k,
    float eps) {
  const int m = blockIdx.x;
  const int c = (blockIdx.y * 256 + threadIdx.x) * 2;
  if (c >= N) return;
  float v0 = 0.f, v1 = 0.f;
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    const f32x2 p =
        *reinterpret_cast<const f32x2*>(parts + ((size_t)s * M + m) * N + c);
    v0 += p[0];
    v1 += p[1];
  }
  float rstd = 1.f;
  if (ss) {
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) q += ss[m * 8 + j];
    rstd = rsqrtf(q * inv_k + eps);
  }
  *reinterpret_cast<u16x2*>(out + (size_t)m * N + c) =
      u16x2{f2bf(v0 * rstd), f2bf(v1 * rstd)};
}

#define ROWS_MAX 16   // rows up to here: gemm_rows_kernel
#define ROWS_CUS 256

// Weights from here on are streamed past the caches, and X stays in them: SwiGLU
// over 28672 x 4096 40.5 -> 37.5 us at one row, 42.8 -> 40.1 at 64, 52.0 -> 50.0 at 128
// (before later changes); 4096 x 14336 21.4 -> 19.0, 23.3 -> 21.7, 27.6 -> 26.8.  Smaller
// ones are bound by latency, which is higher that way (2048 x 2048 5.1 us against
// 4.1 from memory, 3.9 against 2.9 from the L2).
static bool streamed(const RowsArgs& a) { return (i64)a.N * a.K >= (8 << 20); }

// With the norm computed, where some CUs have two blocks and others one, waves that wait
// for all they have asked for are faster at few rows.  Rotary, in flight / drained in us:
// 272 blocks, K 4096 11.5 / 10.9 at one row, 11.8 / 11.6 at 8, K 8192 20.0 / 17.7; 448
// blocks 12.8 / 12.6; but 512 13.6 / 13.6, K 8192 24.1 / 25.7; 256
// 8.5 / 9.8; 576 16.5 / 18.4; K 2048 from 272 blocks on 0 to 3% slower.
//
// Rotary, tiles that leave half of the CUs one more than the others: of 24 rows instead of 16
// all have as many, and X is read a third less often.  Blocks of 16 / 24 rows in us, one row
// and 16: 384 / 256, K 4096 11.1 / 10.7 and 13.3 / 11.0, K 8192 19.2 / 18.1 and 23.9 / 18.2;
// 264 / 176, K 4096 10.3 / 8.6 and 12.6 / 10.1; 768 / 512 18.0 / 17.8 and 20.2 / 18.4, K 2048
// 12.0 / 10.3 and 12.9 / 11.0; K 1024 level.  Not where 16 rows fill their rounds as well: 240
// / 160 7.7 / 8.3, 480 / 320 12.4 / 14.8, 960 / 640 21.7 / 22.1.  Nor where the second round
// of 24 is half empty and K long, one rule for all M, so that results do not depend on it: 1,
// 4, 8 and 16 rows, 528 / 352, K 5120 19.0 18.9 19.9 23.1 / 19.7 18.7 19.3 21.4; 576 / 384 19.7
// 19.8 21.0 23.6 / 20.0 20.5 21.6 21.9, K 6144 22.2 22.3 23.6 26.7 / 22.8 23.4 24.7 24.8; but
// K 3584 0.91 to 0.99 of the time at 352 to 384, K 4096 0.92 to 1.03, and from 416 tiles of 24
// on 0.90 to 0.99 at every K and M.  Longer rings (three and four pieces) and, to 8 rows, 8 rows
// of X instead of 16 change nothing.
static bool in_24s(const RowsArgs& a) {
  const int g = a.N / 16, g24 = a.N / 24, rounds = (g24 + ROWS_CUS - 1) / ROWS_CUS;
  return a.N % 24 == 0 && g > rounds * ROWS_CUS && rounds <= 2 &&
         (rounds == 1 || a.K < 4096 || g24 > 400);
}

template <int EPI, int NORM>
static void launch_rows(const RowsArgs& a, hipStream_t st) {
  const int g = a.N / 16;
  if constexpr (EPI == EPI_ROPE) {
    if (in_24s(a)) {
      if (streamed(a))
        gemm_rows_kernel<2, EPI, NORM, STREAM, false, 3><<<a.N / 24, 512, 0, st>>>(a);
      else
        gemm_rows_kernel<2, EPI, NORM, KEEP, false, 3><<<a.N / 24, 512, 0, st>>>(a);
      return;
    }
  }
  if (NORM == 2 && g > ROWS_CUS && g <= 448 && a.K >= 4096 && a.M <= 8)
    gemm_rows_kernel<2, EPI, NORM, STREAM, NORM == 2><<<g, 512, 0, st>>>(a);
  else if (streamed(a))
    gemm_rows_kernel<2, EPI, NORM, STREAM, false><<<g, 512, 0, st>>>(a);
  else
    gemm_rows_kernel<2, EPI, NORM, KEEP, false><<<g, 512, 0, st>>>(a);
}

// Blocks of 128 weight rows halve the reads of X; they pay where blocks of 64 are more
// than one to a CU (64 / 128 columns, SwiGLU, in us: 22016 x 4096, 344 or 172 blocks, 38.2
// / 31.5 at 32 rows, 58.2 / 44.8 at 128; 18432 x 4096 39.3 / 30.0, 57.2 / 43.7; 16384 x
// 4096, 256 or 128 blocks, 25.3 / 29.6, 34.1 / 43.2).  Up to 64 rows, more than one of them
// to a CU, the rings are short enough that two have room (57344 x 8192, 17 rows: 156 us in
// rings of 5, 149 of 3; 128256 x 8192 350, 323), otherwise longer (22016 x 4096 34.6 in 3,
// 31.5 in 5).  Plain products of 97..128 rows without a norm keep the loop of the split
// ones: 32000 x 2048 28.7 us, 27.2 there; 65536 x 2048 61.4, 58.5; 24576 x 4096 46.4, 45.2;
// but 128256 x 4096 with a norm 211, 215 there, 28672 x 4096 with SwiGLU 46.4, 48.2.  Small weights are here and gone: 4096 x 1024 at 32 rows
// 7.3 us in a ring of 5, 6.9 of 3.
template <int EPI, int NORM, int AUX>
static void launch_tile_as(const RowsArgs& a, hipStream_t st) {
  if (a.N % 128 == 0 && a.N > 64 * ROWS_CUS) {
    const int g = a.N / 128;
    if (a.M <= 32 && g <= ROWS_CUS)
      gemm_tile_kernel<2, 8, 8, 5, EPI, NORM, AUX><<<g, 512, 0, st>>>(a);
    else if (a.M <= 32)
      gemm_tile_kernel<2, 8, 8, 3, EPI, NORM, AUX><<<g, 512, 0, st>>>(a);
    else if (a.M <= 64 && g <= ROWS_CUS)
      gemm_tile_kernel<4, 8, 8, 4, EPI, NORM, AUX><<<g, 512, 0, st>>>(a);
    else if (a.M <= 64)
      gemm_tile_kernel<4, 8, 8, 3, EPI, NORM, AUX><<<g, 512, 0, st>>>(a);
    else if (a.M <= 96)
      gemm_tile_kernel<6, 8, 8, 4, EPI, NORM, AUX><<<g, 512, 0, st>>>(a);
    else if constexpr (EPI == EPI_PLAIN && NORM == 0)
      gemm_parts_kernel<8, 8, 4, 3, EPI, AUX><<<g, 512, 0, st>>>(a);
    else
      gemm_tile_kernel<8, 8, 8, 4, EPI, NORM, AUX><<<g, 512, 0, st>>>(a);
  } else {
    const int g = a.N / 64;
    const bool small = (i64)a.N * a.K <= (4 << 20);
    if (a.M <= 32 && small)
      gemm_tile_kernel<2, 4, 4, 3, EPI, NORM, KEEP><<<g, 256, 0, st>>>(a);
    else if (a.M <= 32)
      gemm_tile_kernel<2, 4, 4, 5, EPI, NORM, AUX><<<g, 256, 0, st>>>(a);
    else if (a.M <= 64)
      gemm_tile_kernel<4, 4, 8, 4, EPI, NORM, AUX><<<g, 512, 0, st>>>(a);
    else if (a.M <= 96)
      gemm_tile_kernel<6, 4, 4, 3, EPI, NORM, AUX><<<g, 256, 0, st>>>(a);
    else
      gemm_tile_kernel<8, 4, 8, 3, EPI, NORM, AUX><<<g, 512, 0, st>>>(a);
  }
}

template <int EPI, int NORM>
static void launch_tile(const RowsArgs& a, hipStream_t st) {
  if (streamed(a)) launch_tile_as<EPI, NORM, STREAM>(a, st);
  else launch_tile_as<EPI, NORM, KEEP>(a, st);
}

// Blocks of 128 weight rows pay from 33 rows on where they fill the chip with at least
// 12 pieces of K each (6144 x 4096 in 5 at 64 rows: 11.2 us against 12.8, 4096 x 14336
// in 8: 21.7 against 23.1; but 4096 x 4096 in 8, 8 pieces: 8.8 against 8.5 in 4), always
// above 64 rows.
static bool parts_in_128s(const RowsArgs& a, int splits) {
  if (a.N % 128 || a.M > 64) return a.N % 128 == 0;
  return a.N / 128 * splits >= 192 && a.K / 64 >= 12 * splits && (a.M > 32 || splits == 1);
}

template <int AUX>
static void launch_parts_as(const RowsArgs& a, int splits, hipStream_t st) {
  const bool wide = parts_in_128s(a, splits);
  const dim3 g(a.N / (wide ? 128 : 64), splits);
  if (a.M <= 64 && wide)
    gemm_parts_kernel<4, 8, 4, 3, EPI_PARTS, AUX><<<g, 512, 0, st>>>(a);
  else if (a.M <= 32)
    gemm_parts_kernel<2, 4, 1, 4, EPI_PARTS, AUX><<<g, 256, 0, st>>>(a);
  else if (a.M <= 64)
    gemm_parts_kernel<4, 4, 2, 4, EPI_PARTS, AUX><<<g, 256, 0, st>>>(a);
  else if (wide)
    gemm_parts_kernel<8, 8, 4, 3, EPI_PARTS, AUX><<<g, 512, 0, st>>>(a);
  else
    gemm_parts_kernel<8, 4, 2, 3, EPI_PARTS, AUX><<<g, 256, 0, st>>>(a);
}

static void launch_parts(const RowsArgs& a, int splits, hipStream_t st) {
  if (streamed(a)) launch_parts_as<STREAM>(a, splits, st);
  else launch_parts_as<KEEP>(a, splits, st);
}

static int check_rows(const RowsArgs& a, int splits) {
  if (a.M < 1 || a.M > 128) return 9005;
  if (a.N % 64 || a.K % 64 || a.K < 64) return 9006;
  const int pieces = a.K / 64;
  if (splits < 1 || splits > pieces) return 9003;
  const int per = (pieces + splits - 1) / splits;
  if ((splits - 1) * per >= pieces) return 9003;  // an empty split
  return 0;
}

// mode 0 plain, 1 residual add (in place, also to `out` if given), 2 SwiGLU,
// 4 residual add + row sums of squares of the result to ss_out [M, 8].
// norm 0 none, 1 RMSNorm scalar of X from ss [M, 8], 2 computed (<= 16 rows).
// parts [splits, M, N]: needed unless rows <= 16 (and mode 0..2), mode 2, or mode 0
// in one split.
AF_EXPORT int af_rows_linear(void* out, void* residual, void* parts, void* ss_out,
                             const void* X, const void* W, int M, int N, int K,
                             int splits, int mode, int norm, const void* ss,
                             float eps, void* stream) {
  RowsArgs a = {};
  a.out = (u16*)out;
  a.residual = (u16*)residual;
  a.parts = (float*)parts;
  a.X = (const u16*)X;
  a.W = (const u16*)W;
  a.M = M; a.N = N; a.K = K;
  a.ss = (const float*)ss;
  a.eps = eps;
  if (const int rc = check_rows(a, splits)) return rc;
  if (mode != 0 && mode != 2 && norm != 0) return 9008;
  if (mode == 0 || mode == 2 ? !out : !residual) return 9008;
  if ((mode == 4 && !ss_out) || (norm == 1 && !ss)) return 9008;
  hipStream_t st = (hipStream_t)stream;
  if (M <= ROWS_MAX && mode != 4) {
    if (mode == 0) {
      if (norm == 0) launch_rows<EPI_PLAIN, 0>(a, st);
      else if (norm == 1) launch_rows<EPI_PLAIN, 1>(a, st);
      else launch_rows<EPI_PLAIN, 2>(a, st);
    } else if (mode == 1) {
      launch_rows<EPI_RESIDUAL, 0>(a, st);
    } else if (mode == 2) {
      if (norm == 0) launch_rows<EPI_SWIGLU, 0>(a, st);
      else if (norm == 1) launch_rows<EPI_SWIGLU, 1>(a, st);
      else launch_rows<EPI_SWIGLU, 2>(a, st);
    } else {
      return 9008;
    }
    return af_last_err();
  }
  if (norm == 2) return 9008;
  if (mode == 2) {
    if (norm == 0) launch_tile<EPI_SWIGLU, 0>(a, st);
    else launch_tile<EPI_SWIGLU, 1>(a, st);
    return af_last_err();
  }
  if (mode == 0 && splits == 1) {
    if (norm == 0) launch_tile<EPI_PLAIN, 0>(a, st);
    else launch_tile<EPI_PLAIN, 1>(a, st);
    return af_last_err();
  }
  if (!parts) return 9008;
  launch_parts(a, splits, st);
  if (mode == 0) {
    const dim3 g(M, (N + 511) / 512);
    rows_sum_kernel<<<g, 256, 0, st>>>(a.out, a.parts, norm ? a.ss : nullptr, M, N,
                                       splits, 1.f / (float)K, eps);
  } else if (mode == 1 || mode == 4) {
    const int tile = parts_in_128s(a, splits) ? 128 : 64;
    rows_residual_kernel<<<dim3(8, M), 256, 0, st>>>(
        a.residual, a.out, a.parts, (float*)ss_out, M, N, splits, N % (8 * tile) ? 0 : tile);
  } else {
    return 9008;
  }
  return af_last_err();
}

// Up to GROUP_MAX plain products of M <= 16 rows each: out [M, N] = X [M, K] @ W [N, K]^T,
// described by n times (out, X, W, N, K).
AF_EXPORT int af_rows_group(const i64* desc, int n, int M, void* stream) {
  if (n < 1 || n > GROUP_MAX || M < 1 || M > ROWS_MAX) return 9008;
  RowsGroup g = {};
  g.parts = n;
  g.M = M;
  int order[GROUP_MAX] = {0, 1, 2, 3}, tiles = 0;
  for (int i = 1; i < n; ++i)
    for (int j = i; j > 0 && desc[order[j] * 5 + 4] > desc[order[j - 1] * 5 + 4]; --j) {
      const int t = order[j];
      order[j] = order[j - 1];
      order[j - 1] = t;
    }
  bool stream_past = false;
  for (int i = 0; i < n; ++i) {
    const i64* d = desc + order[i] * 5;
    RowsArgs a = {};
    a.out = (u16*)d[0];
    a.X = (const u16*)d[1];
    a.W = (const u16*)d[2];
    a.M = M;
    a.N = (int)d[3];
    a.K = (int)d[4];
    if (!a.out || d[3] < 64 || d[3] > INT_MAX || d[4] > INT_MAX) return 9008;
    if (const int rc = check_rows(a, 1)) return rc;
    g.part[i] = {a.out, a.X, a.W, a.N, a.K, tiles};
    tiles += a.N / 16;
    stream_past = stream_past || streamed(a);
  }
  hipStream_t st = (hipStream_t)stream;
  if (stream_past) gemm_rows_group_kernel<STREAM><<<tiles, 512, 0, st>>>(g);
  else gemm_rows_group_kernel<KEEP><<<tiles, 512, 0, st>>>(g);
  return af_last_err();
}

// Fused QKV projection of normed rows + rotary positions + page append: q
// [M, Hq*128] to `q`, k and v to their pages only.  Up to 16 rows compute the
// RMSNorm scalar themselves; more take it from ss.
AF_EXPORT int af_rows_qkv(void* q, void* parts, const void* X, const void* W,
                          const void* ss, int M, int Hq, int Hk, int D, int K,
                          int splits, float eps, const void* pos,
                          const void* table, void* kc, void* vc,
                          const void* slot, int page_size, void* stream) {
  if (D != 128) return 9002;
  if (Hq < 1 || Hk < 1 || page_size < 1) return 9003;
  RowsArgs a = {};
  a.out = (u16*)q;
  a.parts = (float*)parts;
  a.X = (const u16*)X;
  a.W = (const u16*)W;
  a.M = M; a.N = (Hq + 2 * Hk) * 128; a.K = K;
  a.ss = (const float*)ss;
  a.eps = eps;
  a.pos = (const i32*)pos;
  a.table = (const float*)table;
  a.kc = (u16*)kc;
  a.vc = (u16*)vc;
  a.slot = (const i64*)slot;
  a.Hq = Hq; a.Hk = Hk; a.page_size = page_size;
  if (const int rc = check_rows(a, splits)) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (M <= ROWS_MAX) {
    launch_rows<EPI_ROPE, 2>(a, st);
    return af_last_err();
  }
  if (!parts || !ss) return 9008;
  launch_parts(a, splits, st);
  const int heads = (Hq + 2 * Hk + 7) / 8;      // of an XCD
  rows_rope_kernel<<<dim3(8, M, (heads + 7) / 8), 64 * min(heads, 8), 0, st>>>(a, splits);
  return af_last_err();
}
