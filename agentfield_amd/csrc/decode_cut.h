// How the sequences of a decode step are cut for its attention.  In nsplit parts each, the
// longest decide: 24 of 1800..8100 tokens in two are blocks of 900 to 4050 tokens, 97 us where
// as many tokens in sequences of one length take 86.  Where that leaves enough to win, all of
// them are cut as one row of rounds into as many equal shares instead: a block goes on into
// the next sequence, and its part of each is a piece, number slot + sequence.
//
// The cut follows from the lengths alone, which a step's layers have in common, so it is made
// once a step, beside the embedding, and read by scalar loads.  Found anew by every block of
// every layer and of every merge it cost 0.5 to 1.1 us a layer where lengths are alike: 16 of
// 513..576 tokens 14.4 us without a look at the lengths, 15.4 with, 14.3 so; 24 of 900..1000
// 24.2, 24.9, 24.0; 16 of 100..130 8.0, 8.8, 7.9.
#pragma once
#include "common.h"

#define AD_TILE 16   // tokens per wave iteration
#define AD_WAVES 4

// parts are whole rounds of the block's waves
constexpr int ROUND = AD_TILE * AD_WAVES;

// sequences that a cut is made for: a lane each
constexpr int CUT_MAX = 64;

// Visible tokens of a sequence are [first, L), its rounds begin at a whole tile.
struct Visible { int first, tile0, rounds; };
__device__ __forceinline__ Visible visible(int L, int win) {
  // sliding window (Mistral): only the last `win` tokens
  const int s0 = (win > 0 && L > win) ? L - win : 0;
  const int a0 = s0 & ~(AD_TILE - 1);
  return {s0, a0, (L - a0 + ROUND - 1) / ROUND};
}

// Sums over the lanes up to a lane's own
__device__ __forceinline__ int wave_scan(int v) {
#define AD_ADD(CTRL, ROWS) \
  v += __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false)
  AD_ADD(0x111, 0xf);   // a row's lanes 1, 2, 4 and 8 below
  AD_ADD(0x112, 0xf);
  AD_ADD(0x114, 0xf);
  AD_ADD(0x118, 0xf);
  AD_ADD(0x142, 0xa);   // the last lane of rows 0 and 2, then of the lower half
  AD_ADD(0x143, 0xc);
#undef AD_ADD
  return v;
}

// A row of the cut, of one sequence: rounds of a share (0: nsplit parts each), tokens, rounds
// of one of nsplit parts, rounds up to the sequence's end.  One scalar load instead of that of
// the length alone; the share as a load of its own was 0.5 us.
typedef __attribute__((ext_vector_type(4))) int CutRow;

// Writes B rows, one wave.  In us, nsplit parts / equal shares: 24 of 1800..8100 tokens in two
// 97 / 84, 9 of 1600..8000 in four 52 / 44, 24 of 800..4000 in two 50 / 48, 5 of 300..3000
// with 32 heads 38 / 30, 30 of up to 8000 with G = 8 118 / 92.  Four rounds are what going on
// takes (3 us: a merge more, loads from the start).
__device__ __forceinline__ void write_cut(CutRow* __restrict__ cut, const i32* __restrict__ len,
                                          int B, int nsplit) {
  const int lane = threadIdx.x & 63;
  const int L = lane < B ? len[lane] : 0;
  const int mine = max(visible(L, 0).rounds, 0);
  const int sum = wave_scan(mine), total = __builtin_amdgcn_readlane(sum, 63);
  const float most = wave_max_f32((float)mine);
  // the largest part against a share
  const bool even = most * (float)B <= (float)total + 4.f * (float)(B * nsplit);
  const int share = even ? 0 : (total + B * nsplit - 1) / (B * nsplit);
  if (lane < B) cut[lane] = CutRow{share, L, (mine + nsplit - 1) / nsplit, sum};
}
