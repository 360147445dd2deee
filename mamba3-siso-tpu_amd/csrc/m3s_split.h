// Sequences split over workgroups, for the forward and the backward scan.
//
// A scan workgroup takes one (b, h) sequence and holds its CU alone, so a launch costs
// ceil(B H / 256) sequence times however few sequences the last round holds: B=1, L=4096,
// H=32 ran its 32 chunks on 32 of 256 CUs. The sequences of that last, incomplete round
// are therefore cut into `segs` segments of chunks, one workgroup each. What a segment
// needs from the rest is the one P x N state that enters it, which two launches make first:
// every chunk's own share of the state, from zero and all chunks in parallel (the scan's
// state update alone: no scores, no readout), and the chain S <- 2^{A_last} S + share over
// the chunks, per state element. The scan forms its state by the same share and the same
// fma, so a split changes no bit of any result: a sequence's output does not depend on how
// many others are in its batch.
#pragma once

#include "m3s_common.h"
#include "m3s_internal.h"

namespace m3s {

struct Split {
  int whole;   // leading sequences that keep one workgroup
  int segs;    // segments of each later sequence (1: no split)
  // first chunk of segment s
  __host__ __device__ int seg_chunk(int s, int nc) const { return (int)((int64_t)nc * s / segs); }
  // chunks whose share the chain takes: all but the last (backward: the first) segment's
  __host__ __device__ int shares(int nc, bool reverse) const {
    return reverse ? nc - seg_chunk(1, nc) : seg_chunk(segs - 1, nc);
  }
};

// The rule: no split where the last round is full or more than half full (two segments
// would take a second round); else as many segments as fill that round, at most one per
// chunk and kMaxSegs, and only if a sequence's time falls by `min_saved` tokens, what the
// two launches cost. Forward, unsplit against split (H=32, traced): B=1 L=2048 113 -> 52 us,
// L=4096 207 -> 78, L=8192 403 -> 131 (of which the shares 14 / 20 / 40 and the chain 7 / 10
// / 17); three sequences' worth of rounds, B=16 L=2048 H=24: 247 -> 229; B=1 L=896 H=24, six
// chunks saved: 53 -> 37; B=4 L=512, two chunks saved, was slower split (37 -> 41).
// No split either where its states, `state_bytes` per chunk of each cut sequence (256 B a token
// and head at N = 128, P = 64; a layer's x, z and y rows are 384), come to more than kMaxBytes.
// Up to there it is always the faster: H=32 L=131072 (1 GiB) 6.25 -> 2.35 ms, H=4 L=1048576
// (1 GiB) 50 -> 17 ms, though each raw-mode share walks the angles of the chunks before it.
constexpr int kMaxSegs = 16;
constexpr int64_t kMaxBytes = int64_t(1) << 30;
inline Split plan_split(int64_t nseq, int nc, int chunk, int min_saved, int64_t state_bytes) {
  Split sp{(int)nseq, 1};
  const int rem = (int)(nseq % kFirstRound);
  if (rem == 0) return sp;
  int segs = kFirstRound / rem;
  segs = segs < nc ? segs : nc;
  segs = segs < kMaxSegs ? segs : kMaxSegs;
  if (segs < 2 || (nc - (nc + segs - 1) / segs) * chunk < min_saved) return sp;
  if (rem * (int64_t)nc * state_bytes > kMaxBytes) return sp;
  sp.whole = (int)(nseq - rem);
  sp.segs = segs;
  return sp;
}
// Workspace floats: per split sequence and share a P x N state and its decay (rounded up to
// 16 bytes).
inline int64_t split_floats(const Split& sp, int64_t nseq, int nc, int n, int pdim, bool reverse) {
  if (sp.segs < 2) return 0;
  const int64_t shares = (nseq - sp.whole) * sp.shares(nc, reverse);
  return shares * n * pdim + (shares + 3) / 4 * 4;
}

// Workgroup -> (sequence, segment): the unsplit sequences first, in xcd_remap order, then
// the split ones, a sequence's segments next to each other: its shares are written, chained
// and read on one XCD (2-3 us less per scan than segment by segment, which keeps the heads
// that share q and k rows together instead).
__device__ __forceinline__ void split_block(const Split& sp, int bid, int nwg, int& seq, int& seg) {
  if (bid < sp.whole) {
    seq = xcd_remap(bid, sp.whole);
    seg = 0;
    return;
  }
  const int i = xcd_remap(bid - sp.whole, nwg - sp.whole), r = i / sp.segs;
  seg = i - r * sp.segs;
  seq = sp.whole + r;
}

// A state in accumulator order: element 4 ((wave SPW + m) 64 + lane) + i is S[p][n] of wave
// `wave`'s tile m, p = 16 (wave % PB) + 4 (lane / 16) + i, n = 16 (wave / PB + NSTEP m) +
// lane % 16, as both scans' waves own it.
struct ChainParams {
  Split split;
  int nc, reverse;
  float* shares;        // (sequence, share) states in accumulator order
  const float* decay;   // (sequence, share) 2^{A_last}
  // what enters the first chunk (backward: the last): (B, H, P, N) or NULL, and in the
  // forward its trapezoid carry seed_coef v (x) k
  const float* s0;
  const float* seed_k;
  const float* seed_v;
  const float* seed_coef;
};

// The entering state of a sequence, one element: the seed plus its trapezoid carry (one fma,
// as the scans write it).
__device__ __forceinline__ float seeded(float s, float coef, float v, float k) {
  return fmaf(coef * v, k, s);
}

// The chain over the shares of the split sequences; the state entering a segment replaces
// the last share consumed before it. One thread per four state elements and sequence, the
// shares of kBatch chunks loaded ahead of their fmas. Bound by its one read of the shares.
template <int C, int N, int P>
__global__ void __launch_bounds__(256) state_chain_kernel(const ChainParams p) {
  constexpr int NW = C / 16, PB = P / 16, SPW = PB * (N / 16) / NW, NSTEP = NW / PB;
  constexpr int kBatch = 8;
  const int e = blockIdx.x * 256 + threadIdx.x;      // of N P / 4 (a multiple of 256)
  const int64_t r = blockIdx.y, bh = p.split.whole + r;
  const int nd = p.split.shares(p.nc, p.reverse), off = p.reverse ? p.split.seg_chunk(1, p.nc) : 0;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (p.s0) {
    const int lane = e & 63, wm = e >> 6, m = wm % SPW, wave = wm / SPW;
    const int n = (wave / PB + NSTEP * m) * 16 + (lane & 15);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (wave % PB) * 16 + 4 * (lane >> 4) + i;
      s[i] = p.s0[(bh * P + row) * N + n];
      if (p.seed_k) s[i] = seeded(s[i], p.seed_coef[bh], p.seed_v[bh * P + row], p.seed_k[bh * N + n]);
    }
  }
  f32x4* sh = reinterpret_cast<f32x4*>(p.shares) + r * nd * (N * P / 4) + e;
  const float* dec = p.decay + r * nd;
  int seg = p.reverse ? p.split.segs - 1 : 1;        // the next boundary: segment seg's start
  for (int i0 = 0; i0 < nd; i0 += kBatch) {
    f32x4 x[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int i = i0 + j < nd ? i0 + j : nd - 1;
      x[j] = sh[(int64_t)(p.reverse ? nd - 1 - i : i) * (N * P / 4)];
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (i0 + j < nd) {
        const int slot = p.reverse ? nd - 1 - (i0 + j) : i0 + j, c = slot + off;
        const float d = dec[slot];
#pragma unroll
        for (int k = 0; k < 4; ++k) s[k] = fmaf(s[k], d, x[j][k]);
        if (p.split.seg_chunk(seg, p.nc) == (p.reverse ? c : c + 1)) {
          sh[(int64_t)slot * (N * P / 4)] = s;
          seg += p.reverse ? -1 : 1;
        }
      }
    }
  }
}

}  // namespace m3s
