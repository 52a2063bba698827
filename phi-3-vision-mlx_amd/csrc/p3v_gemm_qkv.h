// The qkv projection with the head split, the rotation and the KV append in its epilogue: p3v_gemm_qkv =
// p3v_gemm(qkv_proj) + p3v_rope_kv_append in the launch of the GEMM alone.  Shared by the kernels of every tile.
//
// What makes it fit the accumulator layout (a lane holds 4 consecutive output columns of one row, p3v_gemm256_epi.h):
//   * Q and K tiles: _rotate_half pairs dimension d with d + hd/2 (phi.py:419-423).  The tile's W rows are fetched in PAIR order --
//     a wave's 64 tile columns are 32 consecutive pairs: blocks 0, 1 their first halves, blocks 2, 3 their second halves (the DMA takes
//     any W row for any tile row: the same trick as the SiLU epilogue's gate / up rows) -- so both halves of a pair sit in ONE lane
//     (acc[i][j][r] and acc[i][j + 2][r]) and the rotation is lane-local.  16 pairs never straddle a head (hd/2 = 48 or 32).
//   * V tiles: the cache keeps V TRANSPOSED ([.., hd, t]).  These tiles are computed with the operand roles swapped -- W rows fill the
//     tile's A side, the tokens its B side (a tile of R x 256 then holds R dimensions of 256 tokens; the K loop does not care) -- so a lane holds 4 consecutive TOKENS of
//     one V dimension, and 8 after the v_permlane16_swap: one 16-byte store into a V^T row (rows whose length is not a multiple of 8
//     -- CLIP's 577-token crops -- shift the run inside the row: still one dwordx4 store at even offsets, three stores at odd ones).
// Arithmetic: exactly p3v_gemm's + p3v_rope_kv_append's (the Linear output rounded to bf16, rotation in fp32 on those values,
// q_scale before the one rounding): bit-identical to the two launches (tests/test_kernels_gpu.py::test_gemm_qkv_fused).
#pragma once
#include "p3v_common.h"

struct QkvP {
  const float* cos_t; const float* sin_t;        // [B / tab_div, tab_t, hd / 2] or both null: plain head split (CLIP)
  bf16_t* q_out; bf16_t* k_dst; bf16_t* v_dst;   // [B, nh, L, hd], [B, nkv, dst_t, hd], [B, nkv, hd, dst_t]
  int L, nh, nkv, hd, past, dpos0, dst_t, tab_t, tab_div;
  float q_scale;
};

// The V^T epilogue stores runs of eight tokens, which may cross the end of ONE batch row: several rows of fewer than 7 tokens do not fit
// (the run's last token would need two or more steps), and the launchers decline them.
static inline bool qkv_rows_ok(int B, int L) { return B == 1 || L >= 7; }

// W row fetched for tile column `rr` (0 .. tile width - 1) of a Q / K tile whose first pair is p0; row0 = first W row of the region
__device__ __forceinline__ int qkv_pair_row(const QkvP& q, int row0, int p0, int rr) {
  const int half = q.hd >> 1;
  const int wcol = rr >> 6, ni = (rr & 63) >> 4, c = rr & 15;
  const int P = p0 + wcol * 32 + (ni & 1) * 16 + c;
  return row0 + (P / half) * q.hd + P % half + (ni >> 1) * half;
}

// Q / K tile: acc[g][i][j] = block row i (16 tokens from m_first) of column group g, blocks 0, 1 = first halves of pairs pw + 32 g .. + 31,
// blocks 2, 3 = second.  The rotation tables cost 4 sixteen-byte loads per block row and group: requested G block rows at a time, a turn.
// W4 (p3v_gemm256.hip, one wave per SIMD: nothing else covers a trip to memory): three turns' tables are on their way while a fourth's row is
// rotated (256 rows x 9216 x 3072 in one round 77 -> 67 us), the sums stay in accumulation registers until their row's turn (p3v_gemm256_epi.h), and
// rows beyond M, which that kernel's requests clamp to row M - 1, are stored as that row, bit for bit, instead of being branched around.
template <int NI, int G, bool W4, int NG>
__device__ __forceinline__ void qkv_epilogue_rot_groups(const QkvP& q, f32x4_t (&acc)[NG][NI][4], const bf16_t* bias, bool is_k, int row0, int pw,
                                                        int m_first, int M, int lane) {
  const int fc = lane & 15, fq = lane >> 4, half = q.hd >> 1;
  const bool rot = q.cos_t != nullptr;
  const float qs = is_k ? 1.f : q.q_scale;
  constexpr int TURNS = (NI + G - 1) / G, RING = W4 ? 4 : 1;
  int d0[NG][2];
  u32x2_t b1[NG][2], b2[NG][2];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int P = pw + g * 32 + j * 16 + fq * 4, head = P / half;
      d0[g][j] = P - head * half;
      b1[g][j] = b2[g][j] = (u32x2_t){0u, 0u};
      if (bias) {
        b1[g][j] = *(const u32x2_t*)(bias + row0 + head * q.hd + d0[g][j]);
        b2[g][j] = *(const u32x2_t*)(bias + row0 + head * q.hd + d0[g][j] + half);
      }
    }
  // (b, l) of the lane's row in block 0; later blocks are 16 tokens further on (one division per tile, not per block)
  const int m00 = m_first + fc;
  int b0 = 0, l0 = m00 < M ? m00 : M - 1;
  if (l0 >= q.L) { b0 = l0 / q.L; l0 -= b0 * q.L; }
  struct Turn { float4 cs[G][2], sn[G][2]; int bb[G], ll[G]; } ring[RING];
  auto ask = [&](int turn) {
    Turn& t = ring[turn % RING];
    const int g = turn / TURNS;
#pragma unroll
    for (int ii = 0; ii < G; ++ii) {
      const int i = turn % TURNS * G + ii;
      if (i >= NI) continue;
      int l = l0 + i * 16, b = b0;
      if (m00 + i * 16 >= M) l = l0 + (M - 1 - (m00 < M ? m00 : M - 1));   // clamped rows
      while (l >= q.L) { l -= q.L; ++b; }
      t.bb[ii] = b, t.ll[ii] = l;
      if (rot) {
        const size_t trow = ((size_t)(b / q.tab_div) * q.tab_t + q.past + l) * half;
#pragma unroll
        for (int j = 0; j < 2; ++j) { t.cs[ii][j] = *(const float4*)(q.cos_t + trow + d0[g][j]); t.sn[ii][j] = *(const float4*)(q.sin_t + trow + d0[g][j]); }
      }
    }
  };
#pragma unroll
  for (int turn = 0; turn < RING; ++turn) ask(turn);
#pragma unroll
  for (int turn = 0; turn < NG * TURNS; ++turn) {
    if (!W4 && turn) ask(turn);
    Turn& t = ring[turn % RING];
    const int g = turn / TURNS;
    // the block this lane stores after the swap: jj = fq & 1, its columns 8 * (fq >> 1) .. + 8
    const int Ps = pw + g * 32 + (fq & 1) * 16, head_s = Ps / half, d_s = Ps - head_s * half + (fq >> 1) * 8;
#pragma unroll
    for (int ii = 0; ii < G; ++ii) {
      const int i = turn % TURNS * G + ii;
      if (i >= NI) continue;
      if constexpr (W4) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) asm volatile("" : "+a"(acc[g][i][j]));
      }
      const int b = t.bb[ii], l = t.ll[ii];
      uint32_t pk1[2][2], pk2[2][2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float cs[4] = {t.cs[ii][j].x, t.cs[ii][j].y, t.cs[ii][j].z, t.cs[ii][j].w}, sn[4] = {t.sn[ii][j].x, t.sn[ii][j].y, t.sn[ii][j].z, t.sn[ii][j].w};
        float o1[4], o2[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v1 = r & 1 ? bf16hi(b1[g][j][r >> 1]) : bf16lo(b1[g][j][r >> 1]), v2 = r & 1 ? bf16hi(b2[g][j][r >> 1]) : bf16lo(b2[g][j][r >> 1]);
          const float a0 = bf16_round(acc[g][i][j][r] + v1), a1 = bf16_round(acc[g][i][j + 2][r] + v2);   // the Linear's bf16 output
          if (rot) {
            p3v_rope_pair(a0, a1, cs[r], sn[r], qs, o1[r], o2[r]);
          } else {
            o1[r] = qs != 1.f ? a0 * qs : a0;
            o2[r] = qs != 1.f ? a1 * qs : a1;
          }
        }
        pk1[j][0] = pack_bf16x2(o1[0], o1[1]), pk1[j][1] = pack_bf16x2(o1[2], o1[3]);
        pk2[j][0] = pack_bf16x2(o2[0], o2[1]), pk2[j][1] = pack_bf16x2(o2[2], o2[3]);
      }
      u32x4_t w1, w2;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        auto s1 = __builtin_amdgcn_permlane16_swap(pk1[0][k], pk1[1][k], false, false);
        w1[k] = s1[0], w1[2 + k] = s1[1];
        auto s2 = __builtin_amdgcn_permlane16_swap(pk2[0][k], pk2[1][k], false, false);
        w2[k] = s2[0], w2[2 + k] = s2[1];
      }
      if (W4 || m00 + i * 16 < M) {
        bf16_t* dst = is_k ? q.k_dst + (((size_t)b * q.nkv + head_s) * q.dst_t + q.dpos0 + l) * q.hd
                           : q.q_out + (((size_t)b * q.nh + head_s) * q.L + l) * q.hd;
        *(u32x4_t*)(dst + d_s) = w1;
        *(u32x4_t*)(dst + d_s + half) = w2;
      }
    }
    if (W4 && turn + RING < NG * TURNS) ask(turn + RING);
  }
}
template <int NI, int G = (NI < 4 ? NI : 4)>
__device__ __forceinline__ void qkv_epilogue_rot(const QkvP& q, f32x4_t (&acc)[NI][4], const bf16_t* bias, bool is_k, int row0, int pw,
                                                 int m_first, int M, int lane) {
  qkv_epilogue_rot_groups<NI, G, false, 1>(q, *reinterpret_cast<f32x4_t (*)[1][NI][4]>(&acc), bias, is_k, row0, pw, m_first, M, lane);
}

// V tile (operand roles swapped): acc[g][i][j] = block row i of 16 V dimensions from fv_first (index into [nkv * hd]), block column j of
// 16 tokens from t_first + 64 g.  bias_v = bias + first W row of the V region, or null.  fv_end: dimensions from there on are not stored.
// W4: as above; runs that all lie at even offsets inside one batch row each are stored in one straight line.
template <int NI, bool W4, int NG>
__device__ __forceinline__ void qkv_epilogue_vt_groups(const QkvP& q, f32x4_t (&acc)[NG][NI][4], const bf16_t* bias_v, int fv_first, int t_first,
                                                       int M, int lane, int fv_end) {
  const int fc = lane & 15, fq = lane >> 4;
  // (an even token offset: the run is dword-aligned -- 16-byte aligned for one batch row, or rows of L % 8 == 0 tokens; any row length, e.g.
  // CLIP's 577-token crops, start one token later in every crop -- one dwordx4 store either way)
  typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
  float bv[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int fv = fv_first + i * 16 + fc;
    bv[i] = bias_v && fv < fv_end ? bf16_to_f32(bias_v[fv]) : 0.f;
  }
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    int tt[2], ll[2];
    bf16_t* run[2];                                            // where the lane's run of 8 tokens of dimension fv_first + fc goes
    bool plain = true;
#pragma unroll
    for (int jp = 0; jp < 2; ++jp) {
      const int t = t_first + g * 64 + (2 * jp + (fq & 1)) * 16 + (fq >> 1) * 8;      // 8 consecutive tokens t .. t + 7
      const int b = t < q.L ? 0 : t / q.L, l = t - b * q.L;
      tt[jp] = t, ll[jp] = l;
      run[jp] = q.v_dst + ((size_t)b * q.nkv * q.hd + fv_first + fc) * (size_t)q.dst_t + q.dpos0 + l;
      plain &= t + 8 <= M && l + 8 <= q.L && !(l & 1);
    }
    plain = W4 && fv_first + NI * 16 <= fv_end && __builtin_amdgcn_ballot_w64(plain) == ~0ull;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if constexpr (W4) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) asm volatile("" : "+a"(acc[g][i][j]));
      }
      const int fv = fv_first + i * 16 + fc;
#pragma unroll
      for (int jp = 0; jp < 2; ++jp) {
        uint32_t pk[2][2];
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
          const f32x4_t& c = acc[g][i][2 * jp + jj];
          pk[jj][0] = pack_bf16x2(c[0] + bv[i], c[1] + bv[i]), pk[jj][1] = pack_bf16x2(c[2] + bv[i], c[3] + bv[i]);
        }
        u32x4_t w;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          auto sw = __builtin_amdgcn_permlane16_swap(pk[0][k], pk[1][k], false, false);
          w[k] = sw[0], w[2 + k] = sw[1];
        }
        const int t = tt[jp], l = ll[jp];
        bf16_t* dst = run[jp] + (size_t)(i * 16) * q.dst_t;
        if (plain) {
          *(u32x4_a4*)dst = w;
        } else if (t < M && fv < fv_end) {
          if (t + 8 <= M && l + 8 <= q.L) {                      // the run lies in one batch row
            if (!(l & 1)) {
              *(u32x4_a4*)dst = w;
            } else {                                             // odd offset: first token, three dwords of token pairs, last token
              typedef uint32_t u32x3_a4 __attribute__((ext_vector_type(3), aligned(4)));
              dst[0] = (bf16_t)w[0];
              const u32x3_a4 mid = {__builtin_amdgcn_alignbyte(w[1], w[0], 2), __builtin_amdgcn_alignbyte(w[2], w[1], 2),
                                    __builtin_amdgcn_alignbyte(w[3], w[2], 2)};
              *(u32x3_a4*)(dst + 1) = mid;
              dst[7] = (bf16_t)(w[3] >> 16);
            }
          } else {                                               // the ragged end of the prompt, or a run across two batch rows
            for (int e = 0; e < 8 && t + e < M; ++e) {
              bf16_t* d = l + e < q.L ? dst + e : dst + e - q.L + (size_t)q.nkv * q.hd * q.dst_t;
              *d = (bf16_t)(w[e >> 1] >> (16 * (e & 1)));
            }
          }
        }
      }
    }
  }
}
template <int NI>
__device__ __forceinline__ void qkv_epilogue_vt(const QkvP& q, f32x4_t (&acc)[NI][4], const bf16_t* bias_v, int fv_first, int t_first,
                                                int M, int lane, int fv_end = 0x7fffffff) {
  qkv_epilogue_vt_groups<NI, false, 1>(q, *reinterpret_cast<f32x4_t (*)[1][NI][4]>(&acc), bias_v, fv_first, t_first, M, lane, fv_end);
}
