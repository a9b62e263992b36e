// Projections of the mixture feed-forward over rows sorted by expert: one launch for
// all experts,  Y[rows of e] = X[rows of e] @ W[e]^T, rows gathered through the sorted
// order where they are still the caller's, SwiGLU in the epilogue.
//
// Prompts of up to 200 rows per expert (down 250, above which the wide GEMM takes over)
// are bound by the experts' weights more than by the matrix cores (600 rows, 8 experts of
// 4096 x 14336, 2 per row: 2.8 GB or 435 us at 6.5 TB/s, 423 GFLOP or 280 us; 429 us of
// gate/up and 203 of down).  A block takes all rows of an expert, up to 288, against
// 128 weight rows, so the weights are read once; more rows are cut evenly, and the cuts
// of one block column run on one XCD at the same time.  Both operands go global -> LDS
// without registers, in stages of K = 64 (52 KB at 288 rows, three of them); half of the
// eight waves take one half of a piece's K and half the other, each 64 weight rows by
// half of the rows (144 registers of sums per lane, of the 256 that two waves leave).
// The loop is unrolled for the number of 16-row groups per wave, so few rows cost few
// products.
// Where experts' rows are uneven it still sees blocks of 288.  With 275 rows of every
// expert, more than it is sent now, the 52 KB per piece bounded it, which arrive at 12.3
// TB/s in all (loads alone 541 us of gate/up, products alone 387, both 600).  Weights
// through registers instead of LDS, 16 rows x 64 bytes per load, were slower there (640
// us, at half of the rows per wave 1420 with spills), and so were, at one row, rings
// short enough for two blocks to a CU (165 -> 182 us of the whole feed-forward).
// Feed-forward of 8 experts of 4096 x 14336 against one library product per expert and
// projection, gathered rows and a wait of the host for the block bounds: 20 rows 488 ->
// 429 us, 200 577 -> 474, 600 1119 -> 639.
#include "mfma_lines.h"

#include <type_traits>

enum MoeEpi { MOE_PLAIN = 0, MOE_SWIGLU = 2 };

#define MG_MT 18                       // 16-row groups of X per block
#define MG_ROWS (16 * MG_MT)
#define MG_NT 8                        // 16-row tiles of weights per block
#define MG_COLS (16 * MG_NT)
#define MG_NW 8                        // waves
#define MG_LDS (156 * 1024)
// Up to 192 rows the weights dominate: they are streamed past the caches, and blocks of
// an XCD start at different pieces of K, or they ask one memory channel for everything
// (40 rows: 307 us of gate/up without the first, 341 without the second, 276 with both).
// Above, pieces in step keep the rows of X in the L2 (512 rows of every expert: 2001 ->
// 1802 us of gate/up).
#define MG_FEW 6                       // 16-row groups per wave

struct MoeGemmArgs {
  u16* out;          // [n, N] ([n, N/2] SwiGLU), sorted rows
  const u16* X;      // rows [., K]
  const i32* row;    // [n] X row of a sorted position; null: the position
  const u16* W;      // [E, N, K]
  const i32* offs;   // [E + 1]
  int E, N, K;
};

// Rows pos0 .. pos0 + rows (up to 32 MW) of the sorted order against the weight rows of
// block column nb.
template <int MW, int EPI>
__device__ __forceinline__ void moe_tile(const MoeGemmArgs& a, char* lds, int e, int pos0,
                                         int rows, int nb, int rot) {
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4;
  constexpr int MT = 2 * MW, PIECE = 2048, STAGE = PIECE * (MG_NT + MT);
  constexpr int STAGES = MG_LDS / STAGE < 5 ? MG_LDS / STAGE : 5;
  constexpr int WG = 2;                          // 8-row lines of W per wave
  constexpr int XG = (MW + 1) / 2;               // lines of X, the last may be a half
  constexpr int PER = WG + XG;
  static_assert(STAGES >= 3 && PER * 3 < 64, "wait counts");
  lds_b* const ring = (lds_b*)lds;
  const int cnt = a.K >> 6, last = (a.N >> 4) - 1;

  const int r8 = lane >> 3;
  const u16 *wp[WG], *xp[XG];
#pragma unroll
  for (int g = 0; g < WG; ++g) {
    const int line = wid * WG + g, tile = min(nb * MG_NT + line / 2, last);
    const int r = EPI == MOE_SWIGLU
                      ? ((line & 1) ? (a.N >> 1) : 0) + tile * 8 + r8
                      : tile * 16 + (line & 1) * 8 + r8;
    wp[g] = a.W + ((size_t)e * a.N + r) * a.K + ((lane & 7) ^ r8) * 8;
  }
#pragma unroll
  for (int g = 0; g < XG; ++g) {
    const int i = wid * MW * 4 + g * 8 + r8;
    const int pos = pos0 + min(i, rows - 1);
    const int r = a.row ? a.row[pos] : pos;
    xp[g] = a.X + (size_t)r * a.K + ((lane & 7) ^ (i & 7)) * 8;
  }
  int pnext = MW <= MG_FEW ? rot : 0, snext = 0;
  auto load = [&]() {
    lds_b* to = ring + snext * STAGE;
    const int off = pnext * 64;
#pragma unroll
    for (int g = 0; g < WG; ++g)
      load_line8<MW <= MG_FEW ? STREAM : KEEP>(wp[g] + off,
                                                  to + (wid * WG + g) * 1024);
#pragma unroll
    for (int g = 0; g < XG; ++g)
      if (2 * g + 2 <= MW || lane < 32)
        load_line8<KEEP>(xp[g] + off, to + MG_NT * PIECE + wid * MW * 512 + g * 1024);
    pnext = pnext + 1 == cnt ? 0 : pnext + 1;
    snext = snext + 1 == STAGES ? 0 : snext + 1;
  };
  // products: a half of every piece's K, 4 tiles of weights, half of X's groups
  const int kh = wid / 4, w0 = (wid & 2) * 2, m0 = (wid & 1) * MW;
  f32x4 acc[4][MW];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int m = 0; m < MW; ++m) acc[t][m] = f32x4{0, 0, 0, 0};
#pragma unroll 1
  for (int s = 0; s < min(STAGES - 1, cnt); ++s) load();
  int slot = 0;
#pragma unroll 1
  for (int i = 0; i < cnt; ++i) {
    // piece i is complete for everybody, and piece i - 1 read by everybody
    meet<PER>(min(STAGES - 2, cnt - 1 - i));
    if (i + STAGES - 1 < cnt) load();
    const lds_b* at = ring + slot * STAGE;
    slot = slot + 1 == STAGES ? 0 : slot + 1;
    bf16x8r w[4], x[2][2];
#pragma unroll
    for (int t = 0; t < 4; ++t) w[t] = frag(at + (w0 + t) * PIECE, kh);
    // rows in pairs, the next pair behind the first two products of this one: the
    // compiler waits for all reads that are out before it uses one
    auto rows2 = [&](int p) {
#pragma unroll
      for (int m = 2 * p; m < min(2 * p + 2, MW); ++m)
        x[p & 1][m & 1] = frag(at + (MG_NT + m0 + m) * PIECE, kh);
    };
    rows2(0);
    __builtin_amdgcn_sched_group_barrier(0x100, MW > 1 ? 6 : 5, 0);
#pragma unroll
    for (int p = 0; 2 * p < MW; ++p) {
      if (2 * p + 2 < MW) rows2(p + 1);
#pragma unroll
      for (int m = 2 * p; m < min(2 * p + 2, MW); ++m)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t], x[p & 1][m & 1],
                                                              acc[t][m], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
    }
  }

  // the two waves of a product swap sums: each finishes two of its tiles
  __syncthreads();
  f32x4* give = reinterpret_cast<f32x4*>(lds) + wid * 2 * MW * 64 + lane;
  const f32x4* take = reinterpret_cast<const f32x4*>(lds) + (wid ^ 4) * 2 * MW * 64 + lane;
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

  // lane: row n of each group, columns 4 q .. + 4 of each tile
  const int tile = nb * MG_NT + w0 + kh * 2;
#pragma unroll
  for (int m = 0; m < MW; ++m) {
    const int r = (m0 + m) * 16 + n;
    u16* o = a.out + (size_t)(pos0 + r) * (EPI == MOE_SWIGLU ? a.N >> 1 : a.N);
    if (EPI == MOE_SWIGLU) {
      // gate rows lie in the lower lanes and up rows in the upper ones: the lower
      // lanes get both of the first tile, the upper ones both of the second
      u16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const auto gu = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(sum[0][m][j]), __float_as_uint(sum[1][m][j]), false, false);
        const float g = __uint_as_float(gu[0]), u = __uint_as_float(gu[1]);
        v[j] = f2bf(g / (1.f + __expf(-g)) * u);
      }
      const int mine = tile + (lane >> 5);
      if (r < rows && mine <= last)
        *reinterpret_cast<u16x4*>(o + mine * 8 + (q & 1) * 4) = v;
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const f32x4 v = sum[t][m];
        if (r < rows && tile + t <= last)
          *reinterpret_cast<u16x4*>(o + (tile + t) * 16 + q * 4) =
              u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
      }
    }
  }
}

// Grid: block columns x an upper bound of row tiles; blocks behind the last tile leave.
template <int EPI>
__global__ void __launch_bounds__(64 * MG_NW, 2) moe_gemm_kernel(MoeGemmArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[MG_LDS];
  const int lane = threadIdx.x & 63, id = blockIdx.x;
  const int cols = (a.N + MG_COLS - 1) / MG_COLS;
  // lane e: expert e's first position, rows, row tiles and first block
  const int o0 = a.offs[min(lane, a.E)];
  const int rows_e = lane < a.E ? a.offs[min(lane + 1, a.E)] - o0 : 0;
  const int nt_e = (rows_e + MG_ROWS - 1) / MG_ROWS;
  int end = nt_e * cols;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(end, o, 64);
    if (lane >= o) end += v;
  }
  const unsigned long long mine = __ballot(id < end);
  if (mine == 0) return;
  const int e = __builtin_ctzll(mine);             // the first that ends behind id
  const int nt = __builtin_amdgcn_readlane(nt_e, e);
  const int rows = __builtin_amdgcn_readlane(rows_e, e);
  const int p0 = __builtin_amdgcn_readlane(o0, e);
  const int local = id - (__builtin_amdgcn_readlane(end, e) - nt * cols);
  // row tiles of a block column eight blocks apart: on one XCD, at the same time
  const int whole = cols / 8 * 8;
  int t, nb;
  if (local < whole * nt) {
    const int g = local / (8 * nt), s = local - g * 8 * nt;
    t = s / 8;
    nb = g * 8 + s % 8;
  } else {
    const int s = local - whole * nt;
    t = s / (cols - whole);
    nb = whole + s % (cols - whole);
  }
  const int per = ((rows + nt - 1) / nt + 15) / 16 * 16;
  const int r0 = t * per, r = min(per, rows - r0);
  if (r <= 0) return;
  const int rot = (id >> 3) * 2 % (a.K >> 6);
#define MG_CASE(G) case G: moe_tile<G, EPI>(a, lds, e, p0 + r0, r, nb, rot); break
  switch ((r + 31) / 32) {                         // groups per wave
    MG_CASE(1); MG_CASE(2); MG_CASE(3); MG_CASE(4); MG_CASE(5); MG_CASE(6);
    MG_CASE(7); MG_CASE(8); MG_CASE(9);
  }
#undef MG_CASE
}

// epi 0 plain, 2 SwiGLU (W rows: gate, then up).  n sorted rows in all.
AF_EXPORT int af_moe_gemm(void* out, const void* X, const void* row, const void* W,
                          const void* offs, int n, int E, int N, int K, int epi,
                          void* stream) {
  if (E < 1 || E > 64 || N < 64 || N % 64 || K < 64 || K % 64) return 9006;
  if (n == 0) return 0;
  MoeGemmArgs a = {(u16*)out, (const u16*)X, (const i32*)row, (const u16*)W,
                   (const i32*)offs, E, N, K};
  const i64 tiles = (i64)n / MG_ROWS + min(E, n);
  const i64 grid = tiles * ((N + MG_COLS - 1) / MG_COLS);
  if (grid > 0x7fffffff) return 9007;
  hipStream_t st = (hipStream_t)stream;
  if (epi == MOE_PLAIN) moe_gemm_kernel<MOE_PLAIN><<<(int)grid, 64 * MG_NW, 0, st>>>(a);
  else if (epi == MOE_SWIGLU) moe_gemm_kernel<MOE_SWIGLU><<<(int)grid, 64 * MG_NW, 0, st>>>(a);
  else return 9008;
  return af_last_err();
}
