// Shared by the kernels of the attention with mixed heads (p3v_attn_mix.hip, p3v_mix_prompt.hip): how a prompt's key ranges are cut and dealt out.
#pragma once
#include "p3v_layered.h"

#define MIX_NEG (-1e30f)             // "no key yet": finite, so that differences of two of them stay 0
#define MIX_MAX_H 32
#define LOG2E 1.4426950408889634f

// A run = the key tiles [split * per, ..) of one query tile.  first query tile that sees 32-key tile T - 1, and how many do
__host__ __device__ static inline int mix_q_first(int past, int T) { const int d = 32 * (T - 1) - 15 - past; return d <= 0 ? 0 : (d + 15) >> 4; }
__host__ __device__ static inline int mix_q_count(int past, int L, int T) {
  return T > ((past + L - 1) >> 5) + 1 ? 0 : ((L + 15) >> 4) - mix_q_first(past, T);
}
// Run number `wid`.  With more runs than CUs in the order of their lengths: the full ones split by split, then the partial ones by
// decreasing length -- long runs that start late are what the last CUs wait for (2048 rows: 18 tiles' time instead of 23 - 27).  Else split by
// split, which takes 2 us less to find out.
struct MixRun { int qt, split, b; };
__device__ __forceinline__ MixRun mix_run(int wid, const AttnMixP& p) {
  const int per = p.tiles_per_split, n_qt = (p.L + 15) >> 4;
  for (int s = 0; s < p.n_split; ++s) {
    const int n = p.B * mix_q_count(p.past, p.L, p.by_length ? (s + 1) * per : s * per + 1);
    if (wid < n) return {n_qt - 1 - wid / p.B, s, wid % p.B};
    wid -= n;
  }
  const int lane = threadIdx.x & 63;
  for (int o0 = 0; o0 < (per - 1) * p.n_split; o0 += 64) {               // (length, split) pairs, a lane each
    const int o = o0 + lane, len = per - 1 - o / p.n_split, T = o % p.n_split * per + len;
    const int n = len > 0 ? p.B * (mix_q_count(p.past, p.L, T) - mix_q_count(p.past, p.L, T + 1)) : 0;
    int sum = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(sum, d);
      sum += lane >= d ? v : 0;
    }
    const unsigned long long hit = __ballot(wid < sum);
    if (hit) {
      const int l = __builtin_ctzll(hit), r = wid - __shfl(sum - n, l), q = __shfl(mix_q_first(p.past, T), l), sp = __shfl(o % p.n_split, l);
      return {__builtin_amdgcn_readfirstlane(q + r / p.B), __builtin_amdgcn_readfirstlane(sp), __builtin_amdgcn_readfirstlane(r % p.B)};
    }
    wid -= __shfl(sum, 63);
  }
  return {-1, 0, 0};
}

// When the last run of a prompt's, cut into runs of up to `per` key tiles, is done, in the time of a key tile.  The runs start by decreasing
// length; run i goes to shader engine i % MIX_ENGINES (XCD by XCD, then engine by engine in them) and waits for its first free CU.  The first
// engine has the longest of every MIX_ENGINES runs, and a run too many before the others: its end is the launch's.  MIX_RUN_FIXED: what a run
// costs besides its tiles.  (With one pool of CUs instead of engines the cut chosen by it was up to 1.2x behind the best, with these within 3 %.)
#define MIX_CUS 256
#define MIX_ENGINES 32
#define MIX_RUN_FIXED 2
#define MIX_PLAN_TILES 4096            // longest key range that is looked at in this detail
static int mix_runs_end(int B, int L, int past, int per, int cus, int fixed = MIX_RUN_FIXED) {
  int by_length[MIX_PLAN_TILES + 1], free_at[128] = {}, end = 0;
  for (int i = 0; i <= per; ++i) by_length[i] = 0;
  for (int q = 0; q < L; q += 16) {
    const int t = ((past + min(q + 15, L - 1)) >> 5) + 1;
    by_length[per] += t / per * B;
    if (t % per) by_length[t % per] += B;
  }
  const int n = min(max(cus / MIX_ENGINES, 1), 128);
  for (int len = per, i = 0, up_to = 0; len > 0; --len)
    for (up_to += by_length[len]; i < up_to; i += MIX_ENGINES) {
      int c = 0;
      for (int k = 1; k < n; ++k) c = free_at[k] < free_at[c] ? k : c;
      free_at[c] += len + fixed;
      end = max(end, free_at[c]);
    }
  return end;
}
