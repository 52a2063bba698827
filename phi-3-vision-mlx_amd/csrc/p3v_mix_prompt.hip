// Attention whose heads' scores are mixed before the softmax (p3v_attn_mix.hip), for prompts of 17 .. 32 heads, in two launches:
//
//   k_mix_scores   raw scores, their mixing, 2^(score - reference), rounded to bf16 -> P in memory
//   k_mix_values   P V, the sums, the sink, the gate -> output rows
//
// In one launch a workgroup holds the outputs of all heads of its 16 queries (192 KB of registers at 32 x 96) beside everything the scores
// need, so that nothing can be requested ahead and each phase waits for the one before it: 9.9 us for 16 queries x 32 keys, of which the
// matrix cores work 1.0 and the vector pipe 2.3.  Apart, no wave waits for another one: a wave owns 16 queries x 16 keys of all heads.
//
// k_mix_scores.  8 waves, the 16 queries' fragments of all heads in LDS (DC KB a head), key fragments straight from the cache.  The scores of
// a (query, key) pair are in ONE lane, a register per head; the mixing contracts over heads, which the matrix instruction wants spread over
// the four lane groups, eight heads each: four lane-group swaps per four registers turn that around, without LDS and without a barrier.
// The products are those of p3v_attn_mix.hip: talk is bf16 data and a score the sum of three bf16 terms, every product exact, the sums fp32.
// Runs of key tiles are cut and ordered as there, so that workgroups side by side walk the same keys (L2); a run costs its queries' way into LDS.
// The reference of a query's tile of 16 keys is its maximum's multiple of 64 (in powers of two): bf16 has fp32's exponent, so a reference
// within 32 of the maximum costs nothing, is the same for nearly all tiles, and two different ones differ by an exact power of two.  It needs
// no running state, so tiles are independent of each other.
//
// k_mix_values.  4 waves share 16 QW queries of one head, a 32-key step each in turn, and add up in LDS.
//
// 2048 rows of 32 heads x 96: keys 6 us, scores 73, values 39 (83 and 48 inside a model); the one launch and its merge 157 + 13.  The scores' CU takes 1.75 us for 16 x 16 pairs
// of all heads: key fragments 0.73 (64 bytes a cycle), matrix cores 0.37, LDS 0.37, vector instructions 0.6, two waves per SIMD to hide them
// behind each other.  Prompts whose scores would not fit the cache run the one launch, on the same fragments.
#include "p3v_attn_mix.h"

#define MIXP_XCDS 8

struct MixPromptP {
  AttnMixP a;
  bf16_t* P;                           // [B][query tiles][H][KT][2][16 queries][8 keys]
  float* M;                            // [B][query tiles][H][KT][16 queries]
  int KT;                              // 16-key tiles of a row of P
};

// ---------------------------------------------------------------- scores
// the four lane groups' registers turned around: x[a] of lane group g becomes x[g] of lane group a
__device__ __forceinline__ void groups_transpose(float& x0, float& x1, float& x2, float& x3) {
  uint32_t a = __float_as_uint(x0), b = __float_as_uint(x1), c = __float_as_uint(x2), d = __float_as_uint(x3);
  auto r = __builtin_amdgcn_permlane32_swap(a, c, false, false);
  a = r[0], c = r[1];
  auto s = __builtin_amdgcn_permlane32_swap(b, d, false, false);
  b = s[0], d = s[1];
  auto t = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  auto u = __builtin_amdgcn_permlane16_swap(c, d, false, false);
  a = t[0], b = t[1], c = u[0], d = u[1];
  asm("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));                          // (hipcc 7.2 folds the bitcast of result 1 into that of result 0)
  x0 = __uint_as_float(a), x1 = __uint_as_float(b), x2 = __uint_as_float(c), x3 = __uint_as_float(d);
}

template <int DC>
__global__ void __launch_bounds__(512) k_mix_scores(MixPromptP mp) {
  const AttnMixP& p = mp.a;
  extern __shared__ __attribute__((aligned(16))) u32x4_t QL[];           // [32 heads][DC][64 lanes]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lc = lane & 15, lg = lane >> 4;
  const uint32_t per_inv = (65535 + p.H / p.G) / (p.H / p.G), k_step = (uint32_t)p.kx_rows * p.dimp * 2;      // (h * per_inv >> 16: h / (H / G) for h < 32)
  const int past = p.past;
  const float sc = fabsf(p.scale) * LOG2E;                               // (a negative scale's sign goes into talk)
  const uint32_t flip = p.scale < 0.f ? 0x8000u : 0u;

  uint32_t neg_lo_w = 0x0000bf80u, neg_hi_w = 0xbf800000u;               // (from registers: as a constant the first becomes the inline -1.0,
  asm volatile("" : "+s"(neg_lo_w), "+s"(neg_hi_w));                     //  which this instruction reads as the second)
  const bf16x2_t neg_lo = __builtin_bit_cast(bf16x2_t, neg_lo_w), neg_hi = __builtin_bit_cast(bf16x2_t, neg_hi_w);
  bf16x8_t tf[2];                                                        // talk (A operand: row = mixed head, 8 raw heads), zero beyond H
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    u32x4_t w = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int h = m * 16 + lc, g = lg * 8 + j;
      const uint32_t v = h < p.H && g < p.H ? p.talk[h * p.H + g] ^ flip : 0;
      w[j >> 1] |= v << (16 * (j & 1));
    }
    tf[m] = __builtin_bit_cast(bf16x8_t, w);
  }

  const MixRun run = mix_run(blockIdx.x, p);
  if (run.qt < 0) return;
  const int b = run.b, q0 = run.qt * 16, first = p.pad_len ? p.pad_len[b] : 0, last = past + min(q0 + 15, p.L - 1);
  const int t1 = 2 * min((last >> 5) + 1, (run.split + 1) * p.tiles_per_split);        // 16-key tiles, whole pairs: what k_mix_values reads
  int kt = 2 * max(first >> 5, run.split * p.tiles_per_split) + wave;

  // ---- queries, whole rows, 16-byte piece by piece, to their fragments' places: 4 heads a wave
#pragma unroll
  for (int f = 0; f < DC; ++f) {
    const uint32_t e = f * 64 + lane, row = e / (4 * DC), c = e - row * (4 * DC);
    const uint32_t src = ((uint32_t)min(q0 + (int)row, p.L - 1) * p.dimp + c * 8) * 2, dst = c / 4 * 64 + c % 4 * 16 + row;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int h = wave * 4 + i;
      QL[h * DC * 64 + dst] = gload<u32x4_t>((gptr_t)p.q + ((size_t)b * p.H + min(h, p.H - 1)) * p.L * p.dimp * 2, src);
    }
  }
  const gptr_t kb = (gptr_t)p.kx + (size_t)b * p.G * k_step;
  const uint32_t k_lane = (uint32_t)lane * 16;
  constexpr int AHEAD = 4;
  bf16x8_t kf[AHEAD][DC];
  auto load_k = [&](int t, int h) {
    gptr_t k0 = kb + (size_t)((uint32_t)min(h, p.H - 1) * per_inv >> 16) * k_step + (size_t)t * 32 * p.dimp;
    asm volatile("" : "+s"(k0));                                         // (a scalar base and one 32-bit lane offset)
#pragma unroll
    for (int c = 0; c < DC; ++c) kf[h % AHEAD][c] = gload<bf16x8_t>(k0 + c * 1024, k_lane);
  };
  if (kt < t1) {
#pragma unroll
    for (int h = 0; h < AHEAD; ++h) load_k(kt, h);
  }
  __syncthreads();

  for (; kt < t1; kt += 8) {
    // ---- raw scores: lane (lg, lc) has keys 4 lg + r of query lc, a register per head
    f32x4_t sv[32];
    bf16x8_t qf[2][DC];
#pragma unroll
    for (int c = 0; c < DC; ++c) qf[0][c] = __builtin_bit_cast(bf16x8_t, QL[c * 64 + lane]);
#pragma unroll
    for (int h = 0; h < 32; ++h) {
      if (h < 31) {
#pragma unroll
        for (int c = 0; c < DC; ++c) qf[(h + 1) & 1][c] = __builtin_bit_cast(bf16x8_t, QL[((h + 1) * DC + c) * 64 + lane]);
      }
      sv[h] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < DC; ++c) sv[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[h % AHEAD][c], qf[h & 1][c], sv[h], 0, 0, 0);
      if (h + AHEAD < 32) load_k(kt, h + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- mixed: lane (lg, lc) has heads 16 m + 4 lg + j of query lc, a register per key
    f32x4_t mx[16][2];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float a = sv[j][r], b_ = sv[8 + j][r], c = sv[16 + j][r], d = sv[24 + j][r];
        groups_transpose(a, b_, c, d);
        sv[j][r] = a, sv[8 + j][r] = b_, sv[16 + j][r] = c, sv[24 + j][r] = d;
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {                                    // key 4 g + r
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = sv[8 * g + j][r];
        u32x4_t part[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t pk = pack_bf16x2(v[2 * j], v[2 * j + 1]);
            part[k][j] = pk;
            if (k < 2) {                                                 // what the pair leaves: exact (a dot product with (-1, 0), (0, -1))
              v[2 * j] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pk), neg_lo, v[2 * j], false);
              v[2 * j + 1] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pk), neg_hi, v[2 * j + 1], false);
            }
          }
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          f32x4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int k = 2; k >= 0; --k) a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tf[m], __builtin_bit_cast(bf16x8_t, part[k]), a, 0, 0, 0);
          mx[4 * g + r][m] = a;
        }
      }
    }
#pragma unroll
    for (int h = 0; h < AHEAD; ++h) load_k(min(kt + 8, t1 - 1), h);
    __builtin_amdgcn_sched_barrier(0);
    const int qpos = past + q0 + lc, key0 = kt * 16;
    if (key0 + 15 > past + q0 || key0 < first) {                       // some query of the tile does not see some key
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const bool live = key0 + k <= qpos && key0 + k >= first;
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int j = 0; j < 4; ++j) mx[k][m][j] = live ? mx[k][m][j] : -INFINITY;
      }
    }
    const size_t tile = ((size_t)b * ((p.L + 15) >> 4) + run.qt) * p.H * mp.KT + kt;
    char *pb = (char*)mp.P + tile * 512, *mb = (char*)mp.M + tile * 64;
    const uint32_t p_lane = (uint32_t)(lg * 4 * mp.KT) * 512 + lc * 16, m_lane = (uint32_t)(lg * 4 * mp.KT) * 64 + lc * 4;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float rm = fmaxf(mx[0][m][j], mx[1][m][j]);
#pragma unroll
        for (int k = 2; k < 16; k += 2) rm = fmaxf(fmaxf(rm, mx[k][m][j]), mx[k + 1][m][j]);
        const float ref = rm == -INFINITY ? MIX_NEG : ceilf(rm * sc * (1.f / 64.f) - 0.5f) * 64.f;
        u32x4_t w[2];
#pragma unroll
        for (int k = 0; k < 16; k += 2)
          w[k >> 3][(k >> 1) & 3] = pack_bf16x2(__builtin_amdgcn_exp2f(fmaf(mx[k][m][j], sc, -ref)), __builtin_amdgcn_exp2f(fmaf(mx[k + 1][m][j], sc, -ref)));
        if (m * 16 + lg * 4 + j < p.H) {
          char* dst = pb + (size_t)(m * 16 + j) * mp.KT * 512;
          *(u32x4_t*)(dst + p_lane) = w[0], *(u32x4_t*)(dst + p_lane + 256) = w[1];
          *(float*)(mb + (size_t)(m * 16 + j) * mp.KT * 64 + m_lane) = ref;
        }
      }
  }
}

// ---------------------------------------------------------------- values
template <int VC, int QW>
__global__ void __launch_bounds__(256, 2) k_mix_values(MixPromptP mp) {
  const AttnMixP& p = mp.a;
  constexpr int NV = 2 * VC;
  __shared__ f32x4_t red[4][2][NV][64];
  __shared__ float ml[4][QW][2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lc = lane & 15, lg = lane >> 4;
  // heads of an XCD side by side, long rows first
  const int nq = (p.L + 15) >> 4, nqb = (nq + QW - 1) / QW, hx = (p.H + MIXP_XCDS - 1) / MIXP_XCDS, xcd = blockIdx.x % MIXP_XCDS, nth = blockIdx.x / MIXP_XCDS;
  const int h = xcd * hx + nth % hx, rest = nth / hx, b = rest % p.B, qb = nqb - 1 - rest / p.B;
  if (h >= p.H || xcd * hx >= p.H) return;
  const int past = p.past, first = p.pad_len ? p.pad_len[b] : 0, g = h / (p.H / p.G);
  const int qt = qb * QW, n_t = min(QW, nq - qt);
  const int last = past + min((qt + n_t) * 16 - 1, p.L - 1);
  const int t0 = first >> 5, t1 = (last >> 5) + 1;

  const gptr_t pt = (gptr_t)mp.P + (((size_t)b * nq + qt) * p.H + h) * mp.KT * 512, mt = (gptr_t)mp.M + (((size_t)b * nq + qt) * p.H + h) * mp.KT * 64;
  const size_t tstep = (size_t)p.H * mp.KT;                              // tiles between two query tiles
  const gptr_t vb = (gptr_t)p.v + ((size_t)b * p.G + g) * (p.Tp >> 4) * p.vdimp * 32;
  const uint32_t p_lane = (uint32_t)lane * 16, m_lane = (uint32_t)((lg >> 1) * 16 + lc) * 4;
  const uint32_t v_lane = (uint32_t)(((lg >> 1) * p.vdimp + lc) * 16 + (lg & 1) * 8) * 2;
  int end[QW];                                                           // steps with keys that some query of the tile sees: k_mix_scores wrote those
#pragma unroll
  for (int i = 0; i < QW; ++i) end[i] = i < n_t ? ((past + min((qt + i) * 16 + 15, p.L - 1)) >> 5) + 1 : 0;

  f32x4_t o[QW][NV], ol[QW];
  float mr[QW];
  const u32x4_t ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  u32x4_t pf[2][QW];
  float mv[2][QW];
  bf16x8_t vf[2][NV];
  auto load = [&](int t, int s) {
#pragma unroll
    for (int i = 0; i < QW; ++i) {
      const int te = min(t, max(end[i] - 1, 0));                         // (past a tile's last step: that one again, not used)
      const size_t tile = min(i, n_t - 1) * tstep + 2 * te;
      gptr_t a = pt + tile * 512, m = mt + tile * 64;
      asm volatile("" : "+s"(a), "+s"(m));
      pf[s][i] = gload<u32x4_t>(a, p_lane);
      mv[s][i] = gload<float>(m, m_lane);
    }
    gptr_t v = vb + (size_t)t * 2 * p.vdimp * 32;
    asm volatile("" : "+s"(v));
#pragma unroll
    for (int d = 0; d < NV; ++d) vf[s][d] = gload<bf16x8_t>(v + d * 512, v_lane);
  };
  auto multiply = [&](int s, const u32x4_t (&w)[QW]) {
#pragma unroll
    for (int i = 0; i < QW; ++i) {
      const bf16x8_t pv = __builtin_bit_cast(bf16x8_t, w[i]);
      ol[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ones), pv, ol[i], 0, 0, 0);
#pragma unroll
      for (int d = 0; d < NV; ++d) o[i][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[s][d], pv, o[i][d], 0, 0, 0);
    }
  };
  // one step where every tile has the references the sums have (or no key); false: it has not, nothing done
  auto step = [&](int t, int s) {
    u32x4_t w[QW];
    bool other = false;
#pragma unroll
    for (int i = 0; i < QW; ++i) {
      const uint32_t seen = t < end[i] ? ~0u : 0u;                       // (a later query tile sees more steps)
      other |= seen && mv[s][i] != mr[i] && mv[s][i] != MIX_NEG;
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i][j] = pf[s][i][j] & seen;
    }
    if (__builtin_amdgcn_ballot_w64(other)) return false;
    multiply(s, w);
    return true;
  };
  // any step: references that differ are powers of two apart, so what is scaled here stays exact
  auto step_any = [&](int t, int s) {
    u32x4_t w[QW];
#pragma unroll
    for (int i = 0; i < QW; ++i) {
      const bool seen = t < end[i];
      const float m = seen ? mv[s][i] : MIX_NEG, mn = fmaxf(mr[i], rows_max(m)), al = __builtin_amdgcn_exp2f(mr[i] - mn);
      const float f = seen ? __builtin_amdgcn_exp2f(m - mn) : 0.f;
      mr[i] = mn;
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i][j] = seen ? pack_bf16x2(bf16lo(pf[s][i][j]) * f, bf16hi(pf[s][i][j]) * f) : 0u;
      ol[i] *= al;
#pragma unroll
      for (int d = 0; d < NV; ++d) o[i][d] *= al;
    }
    multiply(s, w);
  };
  int t = t0 + wave;
#pragma unroll
  for (int i = 0; i < QW; ++i) {
    ol[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f}, mr[i] = MIX_NEG;
#pragma unroll
    for (int d = 0; d < NV; ++d) o[i][d] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  }
  if (t < t1) {
    load(t, 0);
#pragma unroll
    for (int i = 0; i < QW; ++i) mr[i] = t < end[i] ? rows_max(mv[0][i]) : MIX_NEG;
  }
  for (; t < t1; t += 8) {                                               // nearly always all of them
    load(min(t + 4, t1 - 1), 1);
    if (!step(t, 0)) break;
    load(min(t + 8, t1 - 1), 0);
    if (t + 4 < t1 && !step(t + 4, 1)) {
      t += 4;
      break;
    }
  }
  for (; t < t1; t += 4) load(t, 0), step_any(t, 0);
  // ---- the four waves' sums, two query tiles at a time
#pragma unroll
  for (int i = 0; i < QW; ++i)
    if (lg == 0) ml[wave][i][0][lc] = mr[i], ml[wave][i][1][lc] = ol[i][0];
#pragma unroll
  for (int i0 = 0; i0 < QW; i0 += 2) {
    if (i0) __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int d = 0; d < NV; ++d) red[wave][i][d][lane] = o[i0 + i][d];
    __syncthreads();
#pragma unroll
    for (int u0 = 0; u0 < 2 * NV; u0 += 4) {
      const int u = u0 + wave, i = i0 + u / NV, d = u % NV, row_q = (qt + i) * 16 + lc, dd = d * 16 + lg * 4;
      if (i >= n_t || row_q >= p.L) continue;
      float m = MIX_NEG, l = 0.f;
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < 4; ++w) m = fmaxf(m, ml[w][i][0][lc]);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float f = __builtin_amdgcn_exp2f(ml[w][i][0][lc] - m);
        const f32x4_t v = red[w][i - i0][d][lane];
        l = fmaf(f, ml[w][i][1][lc], l);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = fmaf(f, v[r], acc[r]);
      }
      const size_t row = (size_t)b * p.L + row_q;
      const float sk = bf16_to_f32(p.sink[h]) * LOG2E, mm = fmaxf(m, sk), e = __builtin_amdgcn_exp2f(m - mm);
      const float gate = 1.f / (1.f + __expf(-bf16_to_f32(((const bf16_t*)p.gate)[row * p.ld + h])));
      const float f = e / (l * e + __builtin_amdgcn_exp2f(sk - mm)) * gate;
      bf16_t* dst = (bf16_t*)p.out + row * p.H * p.vdim + (size_t)h * p.vdim + dd;
      if (p.vdim % 4 == 0) {
        if (dd < p.vdim) *(u32x2_t*)dst = (u32x2_t){pack_bf16x2(acc[0] * f, acc[1] * f), pack_bf16x2(acc[2] * f, acc[3] * f)};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (dd + r < p.vdim) dst[r] = f32_to_bf16(acc[r] * f);
      }
    }
  }
}

// ---------------------------------------------------------------- keys
// The cache's rows of keys as MFMA fragments: 1 KB of 16 keys x 32 dimensions, lane by lane.  A fragment read out of rows takes 64 accesses of
// 16 bytes of the vector cache, which makes one a cycle; in this order it takes 16.
__global__ void __launch_bounds__(256) k_mix_keys(AttnMixP p, u32x4_t* dst) {
  const int n = p.dimp >> 3, t = blockIdx.x, row = blockIdx.y;           // 16-byte pieces of a key; tile of 16 keys; (sequence, key head)
  const u32x4_t* src = (const u32x4_t*)p.k + ((size_t)row * p.Tp + t * 16) * n;
  dst += ((size_t)row * p.kx_rows + t * 16) * n;
  for (int e = threadIdx.x; e < 16 * n; e += 256) dst[e] = src[(e & 15) * n + (e >> 4)];
}

// ---------------------------------------------------------------- host side
// The two launches take prompts whose scores in memory stay below this: written by one kernel and read by the next, they then mostly live in
// the 256 MB of last-level cache (half of them are never touched: causal).  us of the head split and the attention, 32 heads x 96, the one
// launch on rows of keys : on fragments : the two launches: 128 rows 49 : 45 : 34, 512 60 : 55 : 42, 2048 180 : 166 : 133, 2300 233 : 212 : 180,
// 3072 345 : 304 : 312, 4096 566 : 498 : 572; 256 rows behind 6000 148 : 138 : 120.
#define MIXP_BYTES (400l << 20)
static int64_t mixp_scores_bytes(int B, int L, int H, int n_keys) { return (int64_t)B * p3v_cdiv(L, 16) * H * 2 * p3v_cdiv(n_keys, 32) * (512 + 64); }
static bool mixp_two(int B, int L, int H, int n_keys) { return mixp_scores_bytes(B, L, H, n_keys) <= MIXP_BYTES; }
static int64_t mixp_keys_bytes(int B, int G, int dim, int n_keys) { return (int64_t)B * G * p3v_cdiv(n_keys, 32) * 32 * p3v_cdiv(dim, 32) * 64; }

extern "C" int64_t p3v_attn_mix_prompt_ws_bytes(int B, int L, int H, int G, int dim, int vdim, int n_keys, int f32) {
  // not: fewer than 16 rows (8: 24.9 : 26.3 us) and key heads shared by 4, 8 .. heads, which one wave takes together (32 heads, 8 of keys: 256 rows
  // 41 : 33 us, but 1024 58 : 64, 2 x 900 73 : 73)
  if (B <= 0 || L < 16 || H <= 16 || G <= 0 || H % G || H / G % 4 == 0 || n_keys < L) return 0;
  const int plan = p3v_attn_mix_plan(B, L, H, G, dim, vdim, n_keys, f32);
  if (!plan) return 0;                                                   // the any-size kernel
  return mixp_keys_bytes(B, G, dim, n_keys) +
         (mixp_two(B, L, H, n_keys) ? mixp_scores_bytes(B, L, H, n_keys) : plan > 1 ? p3v_attn_mix_ws_bytes(B, L, H, vdim, plan) : 0);
}

// Key tiles of a run: whole rounds of the waves' tiles (4 tiles of 32 keys), the cut whose last CU is done first
static int mixp_run_tiles(int B, int L, int past) {
  const int tiles = ((past + L - 1) >> 5) + 1;
  if (tiles > MIX_PLAN_TILES) return 64;
  static thread_local int last[4] = {};                                  // (asked for again by every layer of a prompt)
  if (last[0] == B && last[1] == L && last[2] == past) return last[3];
  int best = tiles, best_end = 1 << 30;
  for (int per = 4; per < tiles + 4; per += per < 32 ? 4 : per / 16 * 4) {
    const int end = mix_runs_end(B, L, past, min(per, tiles), MIX_CUS, 1);
    if (end <= best_end) best_end = end, best = per;
  }
  last[0] = B, last[1] = L, last[2] = past, last[3] = best;
  return best;
}

template <int DC>
static int launch_scores(const MixPromptP& mp, hipStream_t s) {
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_mix_scores<DC>, hipFuncAttributeMaxDynamicSharedMemorySize, 32 * DC * 1024) != hipSuccess) return P3V_ERR_HIP;
    attr_set = true;
  }
  hipLaunchKernelGGL((k_mix_scores<DC>), dim3(mp.a.runs), dim3(512), 32 * DC * 1024, s, mp);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}
template <int VC, int QW>
static int launch_values_qw(const MixPromptP& mp, int blocks, hipStream_t s) {
  hipLaunchKernelGGL((k_mix_values<VC, QW>), dim3(blocks), dim3(256), 0, s, mp);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}
// 64 queries a workgroup, which read their values once, where that still makes two workgroups a CU (2048 rows inside a prompt 53 -> 48 us), else 32
// (512 rows 43 -> 41)
template <int VC>
static int launch_values(const MixPromptP& mp, hipStream_t s) {
  const int rows = MIXP_XCDS * p3v_cdiv(mp.a.H, MIXP_XCDS) * mp.a.B, qt = p3v_cdiv(mp.a.L, 16);
  if (rows * p3v_cdiv(qt, 4) >= 2 * MIX_CUS) return launch_values_qw<VC, 4>(mp, rows * p3v_cdiv(qt, 4), s);
  return launch_values_qw<VC, 2>(mp, rows * p3v_cdiv(qt, 2), s);
}

extern "C" int p3v_attn_mix_prompt(const p3v_mix_args_t* a, void* ws, int64_t ws_bytes, void* stream) {
  const int rc = p3v_mix_check(a);
  if (rc != P3V_OK) return rc;
  if (!a->q || !a->talk || !a->sink || !a->gate || !a->out || !ws) return P3V_ERR_ARG;
  const int n_keys = a->past + a->L, dimp = p3v_cdiv(a->dim, 32) * 32, vdimp = p3v_cdiv(a->vdim, 32) * 32;
  const int64_t need = a->d_past || a->dimp != dimp || a->vdimp != vdimp ? 0 : p3v_attn_mix_prompt_ws_bytes(a->B, a->L, a->H, a->G, a->dim, a->vdim, n_keys, a->f32);
  if (!need) return P3V_ERR_UNSUPPORTED;
  if (ws_bytes < need || ((uintptr_t)ws & 15)) return P3V_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  MixPromptP mp = {attn_mix_params(a), nullptr, nullptr, 2 * p3v_cdiv(n_keys, 32)};
  AttnMixP& p = mp.a;
  p.kx = (const bf16_t*)ws, p.kx_rows = 16 * mp.KT;
  hipLaunchKernelGGL(k_mix_keys, dim3(mp.KT, p.B * p.G), dim3(256), 0, s, p, (u32x4_t*)ws);
  P3V_CHECK_LAUNCH();
  char* rest = (char*)ws + mixp_keys_bytes(p.B, p.G, p.dim, n_keys);
  if (!mixp_two(p.B, p.L, p.H, n_keys)) {
    p.n_split = p3v_attn_mix_plan(p.B, p.L, p.H, p.G, p.dim, p.vdim, n_keys, 0), p.ws = (float*)rest;
    return mix_prefill(p, n_keys, s);
  }
  mp.P = (bf16_t*)rest, mp.M = (float*)(rest + (size_t)p.B * p3v_cdiv(p.L, 16) * p.H * mp.KT * 512);
  p.tiles_per_split = mixp_run_tiles(p.B, p.L, p.past);
  p.n_split = p3v_cdiv(p3v_cdiv(n_keys, 32), p.tiles_per_split);
  for (int sp = 0; sp < p.n_split; ++sp) p.runs += p.B * mix_q_count(p.past, p.L, sp * p.tiles_per_split + 1);
  p.by_length = p.runs > MIX_CUS;
  const int e = p.dimp == 32 ? launch_scores<1>(mp, s) : p.dimp == 64 ? launch_scores<2>(mp, s) : p.dimp == 96 ? launch_scores<3>(mp, s) : launch_scores<4>(mp, s);
  if (e != P3V_OK) return e;
  return p.vdimp == 32 ? launch_values<1>(mp, s) : p.vdimp == 64 ? launch_values<2>(mp, s) : p.vdimp == 96 ? launch_values<3>(mp, s) : launch_values<4>(mp, s);
}
