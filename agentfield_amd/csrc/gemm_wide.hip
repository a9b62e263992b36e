// Prompt GEMMs:  Y[M,N] = X[M,K] @ W[N,K]^T in bf16, plain or with SwiGLU behind it
// (W: gate rows, then up rows; Y[M,N/2]).
//
// Bound by the matrix cores.  One block per CU walks the tiles, 256 weight rows by 32 G
// rows of X (G = 4..8): G is the one whose rounds of 256 tiles cost least, so that rows
// just above a whole round do not pay for a second one.  Four waves, one per SIMD, each
// take 128 weight rows by 16 G rows; half of a 64-element piece of K is multiplied
// while the operands of the other half are read from LDS.  The sums are pinned to the
// accumulation registers by inline assembly: left to itself the compiler gives source and
// result different ones and copies between them (664 moves for 48 products).
//
// Both operands travel global -> LDS without registers, in whole 128-byte lines, three
// pieces deep for W and two for X (160 KB).  Loads are spread evenly over the products:
// asked for at once they come back at 64 bytes per clock and the wave stands (4096 x
// 14336, 4096 rows: 360 us, spread 320; those of X every 8 products instead of every 4
// another 0..3%).  One barrier per piece.  The stream of loads
// runs on into the block's next tile, so only the stores stand between tiles; a lane
// stores 16 bytes of a row (weight rows are permuted on their way into LDS so that it
// has eight neighbours), converted by the hardware (4.7 us less per tile).
// Eight waves of 128 x 64 read half as much again from LDS (4096 x 14336, 4096 rows: 331
// us against 316), products of 32 x 32 x 16 were slower still (361), and so were loads
// that warm the L2 ahead (376).
//
// Measured, library against this kernel in us: 14336 -> 4096 at 10077 rows 1104 / 829,
// 8192 rows 599 / 634; 4096 -> 4096 at 10077 rows 361 / 241, 8000 rows 179 / 189;
// 4096 -> 28672 with SwiGLU at 10077 rows 1746 + 164 / 1683, 8192 rows 1256 + 125 / 1330.
#include "mfma_lines.h"

typedef __attribute__((address_space(3))) void lds_v;

#define GW_BLOCKS 256
#define GW_COLS 256

enum WideEpi { WIDE_PLAIN = 0, WIDE_PARTS = 1, WIDE_SWIGLU = 2 };

struct WideArgs {
  u16* out;
  const u16* X;
  const u16* W;
  int M, N, K, tm, tn;     // tiles of rows and of columns
  // experts: rows sorted by expert, W [E, N, K]
  const i32* offs;         // [E + 1] first sorted row
  const i32* row;          // X row of a sorted row; null: itself
  int E;
  // WIDE_PARTS: partial sums [splits, M, N], split s over the s-th share of K
  float* parts;
  int splits;
};

// All tiles of a block.  EXPERTS: rows of X are gathered and tiles end with their
// expert's rows; lane e has expert e's first row, rows and the tiles up to its end.
template <int G, int EPI, bool EXPERTS>
__device__ __forceinline__ void wide_tiles(const WideArgs& a, char* lds, int first_e,
                                           int rows_e, int end_e) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int XR = 32 * G, WB = GW_COLS * 128, XB = XR * 128;
  constexpr bool GLU = EPI == WIDE_SWIGLU, PARTS = EPI == WIDE_PARTS;
  constexpr int OUT = GLU ? GW_COLS / 2 : GW_COLS;         // output columns per tile
  lds_b* const wring = (lds_b*)lds;
  lds_b* const xring = wring + 3 * WB;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4, r8 = lane >> 3;
  const int nt = EXPERTS ? __builtin_amdgcn_readlane(end_e, a.E - 1)
                         : a.tm * a.tn * (PARTS ? a.splits : 1);
  const int cnt = PARTS ? (a.K >> 6) / a.splits : a.K >> 6, cols = GLU ? a.N >> 1 : a.N;
  const unsigned ld = (unsigned)a.K * 2;

  // Rounds of 256 tiles; an XCD's 32 blocks take 8 x 4 neighbours, which share their
  // operands in its L2.  The last tile of a column is moved back inside the matrix (N >=
  // 256) and stores only what the one before it did not; so is, without experts, the last
  // tile of a row (M >= XR).
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  auto tile = [&](int round) { return (round * 8 + xcd) * (GW_BLOCKS / 8) + idx; };
  struct Place { int e, row, rows, fresh, tn, split; };           // rows from fresh on are new
  auto place = [&](int p) {
    Place at = {0, 0, a.M, 0, 0, 0};
    int tm = a.tm;
    if (EXPERTS) {
      at.e = __builtin_ctzll(__ballot(p < end_e));         // the first that ends behind p
      at.row = __builtin_amdgcn_readlane(first_e, at.e);
      at.rows = __builtin_amdgcn_readlane(rows_e, at.e);
      tm = (at.rows + XR - 1) / XR;
      p -= __builtin_amdgcn_readlane(end_e, at.e) - tm * a.tn;
    }
    if (PARTS) {
      at.split = p / (a.tm * a.tn);
      p -= at.split * a.tm * a.tn;
    }
    const int band = p / (8 * a.tn), high = min(8, tm - band * 8), in = p - band * 8 * a.tn;
    const int t = band * 8 + in % high, r = EXPERTS ? t * XR : min(t * XR, a.M - XR);
    at.row += r;
    at.rows -= r;
    at.fresh = EXPERTS ? 0 : t * XR - r;
    at.tn = in / high;
    return at;
  };
  const char *xb = (const char*)a.X, *wb;                  // of the tile being loaded
  unsigned xg[G], xgn[G];                                  // EXPERTS: lanes' rows, bytes
  auto seek_x = [&](int p) {                               // of the next tile
    const Place at = place(p);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int r = at.row + min((g * 4 + wid) * 8 + r8, at.rows - 1);
      xgn[g] = a.row ? a.row[r] : r;
    }
  };
  auto aim_x = [&](int p) {
    if (EXPERTS) {
#pragma unroll
      for (int g = 0; g < G; ++g) xg[g] = xgn[g] * ld + ((lane & 7) ^ r8) * 16;
    } else {
      const Place at = place(p);
      xb = (const char*)(a.X + (size_t)at.row * a.K + (PARTS ? at.split * cnt * 64 : 0));
    }
  };
  auto aim_w = [&](int p) {
    const Place at = place(p);
    wb = (const char*)(a.W + ((size_t)at.e * a.N + min(at.tn * OUT, cols - OUT)) * a.K +
                       (PARTS ? at.split * cnt * 64 : 0));
  };

  // A wave loads 8 lines (8 rows x 128 bytes) of W and G of X per piece.  Row 16 t + 4 q
  // + j of a 32-row group of W in LDS (t = 0, 1) is its row 8 q + 4 t + j, and with SwiGLU
  // a wave's 128 rows are 64 gate rows and the 64 up rows of the same columns.
  const unsigned swz = ((lane & 7) ^ r8) * 16;
  const unsigned xo = r8 * ld + swz, wo = ((r8 >> 2) * 8 + (r8 & 3)) * ld + swz;
  const unsigned w0 =
      GLU ? ((wid >> 1) * 64 + (wid & 1) * cols) * ld : wid * 64 * ld;
  auto load_w = [&](int g, lds_b* to, int k) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc((void*)wb, 0, 0xffffffffu, 0x00027000),
        (lds_v*)(to + (wid * 8 + g) * 1024), 16, wo,
        w0 + ((g >> 2) * 32 + (g & 1) * 16 + ((g >> 1) & 1) * 4) * ld + k, 0, 0);
  };
  auto load_x = [&](int g, lds_b* to, int k) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc((void*)xb, 0, 0xffffffffu, 0x00027000),
        (lds_v*)(to + (g * 4 + wid) * 1024), 16, EXPERTS ? xg[g] : xo,
        (EXPERTS ? 0 : (g * 4 + wid) * 8 * ld) + k, 0, 0);
  };
  // operands: lane (n, q) has k = 8 q .. + 8 of row n, at the first or second half
  const int wm = wid >> 1, wn = wid & 1;
  const int half0 = n * 128 + ((q ^ (n & 7)) * 16), half1 = half0 ^ 64;
  bf16x8r w[2][8], x[2][G];
  auto read_w = [&](int s, int t, const lds_b* at, int half) {
    w[s][t] = as_bf16x8r(
        *reinterpret_cast<const lds_v8*>(at + wn * 16384 + t * 2048 + half));
  };
  auto read_x = [&](int s, int m, const lds_b* at, int half) {
    x[s][m] = as_bf16x8r(
        *reinterpret_cast<const lds_v8*>(at + wm * G * 2048 + m * 2048 + half));
  };

  int round = 0, p = tile(0);
  if (p >= nt) return;
  if (EXPERTS) seek_x(p);
  aim_x(p);
  aim_w(p);
#pragma unroll
  for (int piece = 0; piece < 2; ++piece) {
#pragma unroll
    for (int g = 0; g < 8; ++g) load_w(g, wring + piece * WB, piece * 128);
#pragma unroll
    for (int g = 0; g < G; ++g) load_x(g, xring + piece * XB, piece * 128);
  }
  int kx = 2, kw = 2;                                      // next pieces to load
  __builtin_amdgcn_s_waitcnt(vmcnt_only(8 + G));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int t = 0; t < 8; ++t) read_w(0, t, wring, half0);
#pragma unroll
  for (int m = 0; m < G; ++m) read_x(0, m, xring, half0);
  int ws = 0, xs = 0;

  for (;;) {
    const int next = tile(round + 1);
    if (EXPERTS && next < nt) seek_x(next);
    f32x4 acc[8][G];
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int m = 0; m < G; ++m) {
        acc[t][m] = f32x4{0, 0, 0, 0};
        asm volatile("" : "+a"(acc[t][m]));
      }
    asm volatile("s_nop 7");                  // written before a product reads them
#define GW_MUL(s, c)                                                              \
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"                          \
               : "+a"(acc[(c) & 7][(c) >> 3])                                     \
               : "v"(w[s][(c) & 7]), "v"(x[s][(c) >> 3]))
#define GW_HERE __builtin_amdgcn_sched_barrier(0)
    // per half: an LDS read every 2 products, a load of X every 8, of W every G
    static_assert(4 * G >= 8 + G, "all operands are read within a half");
#pragma unroll 1
    for (int i = 0; i < cnt; ++i) {
      lds_b* const wat = wring + ws * WB;
      lds_b* const wold = wring + (ws == 0 ? 2 : ws - 1) * WB;   // of piece i - 1
      lds_b* const xat = xring + xs * XB;
      ws = ws == 2 ? 0 : ws + 1;
      xs ^= 1;
      const lds_b* wnx = wring + ws * WB;
      const lds_b* xnx = xring + xs * XB;
      // behind a tile's last piece the next tile's follow, behind the last tile the
      // last piece again
      if (kw == cnt) {
        if (next < nt) { aim_w(next); kw = 0; } else --kw;
      }
      const int ow = kw++ * 128;
      __builtin_amdgcn_s_waitcnt(0xc07f);                  // this half's operands
      asm volatile("" ::: "memory");
      GW_HERE;
#pragma unroll
      for (int c = 0; c < 8 * G; ++c) {
        GW_MUL(0, c);
        if (c % G == G / 2) {
          GW_HERE;
          load_w(c / G, wold, ow);
          GW_HERE;
        }
        if (c % 2 == 1 && c / 2 < 8 + G) {
          GW_HERE;
          if (c / 2 < 8) read_w(1, c / 2, wat, half1);
          else read_x(1, c / 2 - 8, xat, half1);
          GW_HERE;
        }
      }
      GW_HERE;
      if (kx == cnt) {
        if (next < nt) { aim_x(next); kx = 0; } else --kx;
      }
      const int ox = kx++ * 128;
      // the next piece has landed (8 loads of W behind it may be out), this one is read
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(vmcnt_only(8) & ~0x0f00);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      GW_HERE;
#pragma unroll
      for (int c = 0; c < 8 * G; ++c) {
        GW_MUL(1, c);
        if (c % 8 == 4) {
          GW_HERE;
          load_x(c / 8, xat, ox);
          GW_HERE;
        }
        if (c % 2 == 1 && c / 2 < 8 + G) {
          GW_HERE;
          if (c / 2 < 8) read_w(0, c / 2, wnx, half0);
          else read_x(0, c / 2 - 8, xnx, half0);
          GW_HERE;
        }
      }
      GW_HERE;
    }
#undef GW_MUL
#undef GW_HERE
    // the last products are through before their sums are read
    asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int m = 0; m < G; ++m) asm volatile("" : "+a"(acc[t][m]));

    // lane: row n of each group, columns 8 q .. + 8 of each pair of tiles
    const Place at = place(p);
    const int r0 = wm * G * 16 + n;
    const int c0 = min(at.tn * OUT, cols - OUT) + wn * (OUT / 2);
    u16* o = a.out + (size_t)(at.row + r0) * cols + c0 + q * 8;
    float* f4 = a.parts + ((size_t)at.split * a.M + at.row + r0) * cols + c0 + q * 8;
#pragma unroll
    for (int m = 0; m < G; ++m) {
      const bool mine = EXPERTS ? r0 + m * 16 < at.rows : r0 + m * 16 >= at.fresh;
      if (PARTS) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (mine && c0 + t * 32 >= at.tn * OUT) {
            *reinterpret_cast<f32x4*>(f4 + t * 32) = acc[t * 2][m];
            *reinterpret_cast<f32x4*>(f4 + t * 32 + 4) = acc[t * 2 + 1][m];
          }
        f4 += 16 * (size_t)cols;
        continue;
      }
      // a group of rows at a time, converted by all lanes: behind the branch the compiler
      // moved all sums to registers first, 256 of them instead of 140, and the experts'
      // kernels spilled 56 (8 experts of 14336 x 4096, two per row: 4096 rows 2430 -> 2378 us,
      // 1500 rows 1024 -> 1013, up to 1100 level; without experts nothing)
      __builtin_amdgcn_sched_barrier(0);
      bf16x8r v[GLU ? 2 : 4];
#pragma unroll
      for (int t = 0; t < (GLU ? 2 : 4); ++t) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float f = acc[t * 2 + (j >> 2)][m][j & 3];
          if (GLU)
            f = f * __builtin_amdgcn_rcpf(1.f + __expf(-f)) *
                acc[(GLU ? 4 : 0) + t * 2 + (j >> 2)][m][j & 3];
          v[t][j] = (__bf16)f;
        }
      }
#pragma unroll
      for (int t = 0; t < (GLU ? 2 : 4); ++t)
        if (mine && c0 + t * 32 >= at.tn * OUT) *reinterpret_cast<bf16x8r*>(o + t * 32) = v[t];
      o += 16 * (size_t)cols;
    }
    if (next >= nt) break;
    p = next;
    ++round;
  }
  __builtin_amdgcn_s_waitcnt(0);              // no load may land in a later block's LDS
#endif
}

template <int G, int EPI>
__global__ void __launch_bounds__(256, 1) gemm_wide_kernel(WideArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[(3 * GW_COLS + 2 * 32 * G) * 128];
  wide_tiles<G, EPI, false>(a, lds, 0, 0, 0);
}

// out = the sum of the parts, 8 values per thread, splits in their order.
__global__ void __launch_bounds__(256) wide_sum_kernel(u16* __restrict__ out,
                                                       const float* __restrict__ parts,
                                                       long long n8, int splits) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    const f32x4* at = reinterpret_cast<const f32x4*>(parts + (s * n8 + i) * 8);
    lo += at[0];
    hi += at[1];
  }
  bf16x8r v;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[j] = (__bf16)lo[j];
    v[j + 4] = (__bf16)hi[j];
  }
  *reinterpret_cast<bf16x8r*>(out + i * 8) = v;
}

// Microseconds per piece of K for G = 4..8, and per tile beside them, fitted to 2,175
// times (15 projections of four models, 256..9000 rows, every G).
#define GW_PIECE {0.766f, 0.911f, 1.054f, 1.195f, 1.333f}
#define GW_TILE 3.2f

// The same over rows sorted by expert.  Every block finds G by itself, from the number
// of tiles that the experts' rows make.
template <int EPI>
__global__ void __launch_bounds__(256, 1) gemm_wide_experts_kernel(WideArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[(3 * GW_COLS + 2 * 256) * 128];
  const int lane = threadIdx.x & 63;
  const int first = a.offs[min(lane, a.E)];
  const int rows = lane < a.E ? a.offs[min(lane + 1, a.E)] - first : 0;
  constexpr float piece[5] = GW_PIECE;
  int best = 0, end = 0;
  float least = 0.f;
#pragma unroll
  for (int g = 8; g >= 4; --g) {
    int sum = (rows + 32 * g - 1) / (32 * g) * a.tn;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(sum, o, 64);
      if (lane >= o) sum += v;
    }
    const int nt = __builtin_amdgcn_readlane(sum, 63);
    const float us =
        (float)((nt + GW_BLOCKS - 1) / GW_BLOCKS) * ((a.K >> 6) * piece[g - 4] + GW_TILE);
    if (best == 0 || us < least) { best = g; least = us; end = sum; }
  }
  switch (__builtin_amdgcn_readfirstlane(best)) {
    case 4: wide_tiles<4, EPI, true>(a, lds, first, rows, end); break;
    case 5: wide_tiles<5, EPI, true>(a, lds, first, rows, end); break;
    case 6: wide_tiles<6, EPI, true>(a, lds, first, rows, end); break;
    case 7: wide_tiles<7, EPI, true>(a, lds, first, rows, end); break;
    default: wide_tiles<8, EPI, true>(a, lds, first, rows, end);
  }
}

// G of least cost, which goes to *us
static int wide_groups(int M, int N, int K, int splits, float* us = nullptr) {
  static const float piece[5] = GW_PIECE;
  int best = 0;
  float least = 0.f;
  for (int g = M < 256 ? M / 32 : 8; g >= 4; --g) {
    const long long tiles =
        (long long)splits * ((M + 32 * g - 1) / (32 * g)) * ((N + GW_COLS - 1) / GW_COLS);
    const float cost =
        (float)((tiles + GW_BLOCKS - 1) / GW_BLOCKS) * (K / 64 / splits * piece[g - 4] + GW_TILE);
    if (best == 0 || cost < least) { best = g; least = cost; }
  }
  if (us) *us = least;
  return best;
}

static bool wide_ok(int M, int N, int K, int epi) {
  return (epi == WIDE_PLAIN || epi == WIDE_SWIGLU) && M >= 256 && N >= 256 && K >= 128 &&
         N % 64 == 0 && K % 64 == 0 &&
         // byte offsets within W are 32 bits wide, tiles are counted in 31
         ((long long)N / 2 + 256) * K * 2 < 0xffffffffll &&
         (long long)(M / 128 + 1) * (N / GW_COLS + 1) < 0x3fffffff;
}

// The time that the plain product should take, ns (1738 products of 256..14000 rows: 0.93
// of what was measured in the mean); 0 where it is not taken.
AF_EXPORT int af_gemm_wide_ns(int M, int N, int K) {
  float us = 0.f;
  if (wide_ok(M, N, K, WIDE_PLAIN)) wide_groups(M, N, K, 1, &us);
  return us < 2e6f ? (int)(us * 1000.f) : 2000000000;
}

// epi 0 plain, 2 SwiGLU.  groups: 4..8, 0 for the best.
AF_EXPORT int af_gemm_wide(void* out, const void* X, const void* W, int M, int N, int K,
                           int epi, int groups, void* stream) {
  if (!wide_ok(M, N, K, epi)) return 9021;
  if (groups == 0) groups = wide_groups(M, N, K, 1);
  hipStream_t st = (hipStream_t)stream;
  WideArgs a = {(u16*)out, (const u16*)X, (const u16*)W, M, N, K,
                (M + 32 * groups - 1) / (32 * groups), (N + GW_COLS - 1) / GW_COLS,
                nullptr, nullptr, 0, nullptr, 1};
#define GW_CASE(g)                                                                \
  case g:                                                                         \
    if (epi == WIDE_SWIGLU) gemm_wide_kernel<g, WIDE_SWIGLU><<<GW_BLOCKS, 256, 0, st>>>(a); \
    else gemm_wide_kernel<g, WIDE_PLAIN><<<GW_BLOCKS, 256, 0, st>>>(a);           \
    break
  switch (groups) {
    GW_CASE(4); GW_CASE(5); GW_CASE(6); GW_CASE(7); GW_CASE(8);
    default: return 9022;
  }
#undef GW_CASE
  return af_last_err();
}

// The number of shares of K, up to 16, that costs least: rounds of 256 blocks as above,
// but a piece never below 0.95 us while the weights come from HBM, and the parts written
// and read at 5.5 TB/s.  It names the fastest of 2..16 shares, or one within 6% of it.
AF_EXPORT int af_gemm_wide_splits(int M, int N, int K) {
  static const float piece[5] = GW_PIECE;
  if (M < 128 || N < 64 || K < 1024) return 1;
  const int pieces = K / 64;
  int best = 1;
  float least = 0.f;
  for (int s = 1; s <= 16 && pieces / s >= 8; ++s) {
    if (pieces % s) continue;
    for (int g = M < 256 ? M / 32 : 8; g >= 4; --g) {
      const long long tiles =
          (long long)s * ((M + 32 * g - 1) / (32 * g)) * ((N + GW_COLS - 1) / GW_COLS);
      const float p = piece[g - 4] < 0.95f ? 0.95f : piece[g - 4];
      const float us = (float)((tiles + GW_BLOCKS - 1) / GW_BLOCKS) * (pieces / s * p + GW_TILE) +
                       (float)s * M * N * 8e-6f / 5.5f;
      if (least == 0.f || us < least) { best = s; least = us; }
    }
  }
  return best;
}

// Plain, K in `splits` shares of whole pieces whose sums meet in parts [splits, M, N]:
// where the tiles of an output are fewer than the blocks.  14336 -> 4096, weights not in
// cache, library / this in us: 160 rows 84 / 42, 300 rows 74 / 55, 512 rows 92 / 71, 1000
// rows 138 / 106, of which the parts' way through memory takes a third.
AF_EXPORT int af_gemm_wide_split(void* out, void* parts, const void* X, const void* W, int M,
                                 int N, int K, int splits, int groups, void* stream) {
  if (M < 128 || splits < 1 || K / 64 % splits || K / 64 / splits < 2 ||
      !wide_ok(M < 256 ? 256 : M, N, K, WIDE_PLAIN) ||
      ((long long)M / 128 + 1) * (N / GW_COLS + 1) * splits > 0x3fffffff)
    return 9021;
  if (groups == 0) groups = wide_groups(M, N, K, splits);
  if (groups < 4 || groups > 8 || 32 * groups > M) return 9022;
  hipStream_t st = (hipStream_t)stream;
  WideArgs a = {(u16*)out, (const u16*)X, (const u16*)W, M, N, K,
                (M + 32 * groups - 1) / (32 * groups), (N + GW_COLS - 1) / GW_COLS,
                nullptr, nullptr, 0, (float*)parts, splits};
#define GW_CASE(g)                                                                \
  case g: gemm_wide_kernel<g, WIDE_PARTS><<<GW_BLOCKS, 256, 0, st>>>(a); break
  switch (groups) { GW_CASE(4); GW_CASE(5); GW_CASE(6); GW_CASE(7); GW_CASE(8); }
#undef GW_CASE
  const long long n8 = (long long)M * N / 8;
  wide_sum_kernel<<<(unsigned)((n8 + 255) / 256), 256, 0, st>>>((u16*)out, (const float*)parts,
                                                              n8, splits);
  return af_last_err();
}

// Rows sorted by expert, n in all: offs [E + 1], row [n] or null, W [E, N, K], x_rows rows
// of X.
AF_EXPORT int af_gemm_wide_experts(void* out, const void* X, const void* row, const void* W,
                                   const void* offs, int x_rows, int n, int E, int N, int K,
                                   int epi, void* stream) {
  if (!wide_ok(256, N, K, epi) || E < 1 || E > 64 || n < 0 || x_rows < 0 ||
      (long long)x_rows * K * 2 > 0xffffffffll ||
      ((long long)n / 128 + E) * (N / GW_COLS + 1) > 0x3fffffff)
    return 9021;
  if (n == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  WideArgs a = {(u16*)out, (const u16*)X, (const u16*)W, n, N, K, 0,
                (N + GW_COLS - 1) / GW_COLS, (const i32*)offs, (const i32*)row, E,
                nullptr, 1};
  if (epi == WIDE_SWIGLU)
    gemm_wide_experts_kernel<WIDE_SWIGLU><<<GW_BLOCKS, 256, 0, st>>>(a);
  else gemm_wide_experts_kernel<WIDE_PLAIN><<<GW_BLOCKS, 256, 0, st>>>(a);
  return af_last_err();
}
