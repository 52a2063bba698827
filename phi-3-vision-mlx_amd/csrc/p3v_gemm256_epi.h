// Shared by the large GEMM kernels (p3v_gemm256.hip, p3v_gemm_pc.hip): launch parameters and the epilogue.
#pragma once
#include "p3v_gemm_qkv.h"

#define P3V_EPI_QKV 100                // internal: the qkv projection with split + RoPE + KV append in the epilogue (p3v_gemm_qkv.h)

#define P3V_EPI_PART 101               // internal: the fp32 partial sums of one slice of K, out [slices, M, N] (p3v_gemm_slices, p3v_gemm.hip)

#define TK 64

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

struct Gemm256P {
  const bf16_t* A; const bf16_t* W; void* out; const bf16_t* bias; const void* resid;
  int M, N, K, lda, ldw, ldo;
  QkvP q;                                // P3V_EPI_QKV only
  int slices;                            // P3V_EPI_PART only: slice z takes the K-tiles z nk / slices .. (z + 1) nk / slices
};

// ---- epilogue: 16 MB x 16 NB outputs per wave, STRAIGHT FROM THE ACCUMULATORS.  The MFMAs take the W fragment as their
// first operand, so a 16 x 16 block comes out transposed: lane (c = lane & 15, q = lane >> 4) holds, for output row
// m = block row c, the FOUR CONSECUTIVE columns 4q .. 4q+3 (the plain operand order gives four rows of one column, which is
// what would make a tile go through a wave-private LDS image: 64 ds_write_b32 + 32 ds_read_b128 per lane and tile,
// ~4 us per tile).  fp32 outputs: those four values are one 16-byte store.  bf16 outputs: the lane pairs (q, q ^ 1) trade the
// packed halves of two neighbouring column blocks with v_permlane16_swap, after which every lane owns 8 consecutive columns
// = one 16-byte store (even q: block 2jp, odd q: block 2jp + 1; columns 8 * (q >> 1) .. + 8 of it).  No LDS, no barrier:
// a wave starts its stores as soon as ITS last MFMA is done.
// acc[i][j]: block row i (16 output rows), block column j (16 W rows) of the wave's outputs, which start at (m0, n0); the launchers see to
// it that the columns are whole tiles.  Reads and writes go through buffer descriptors at the wave's first output, whose bounds check drops
// the rows beyond M: no branch around a store, so a wave's conversions and stores run in one straight line.
template <int EPI, int MB, int NB, bool AGPR = false>
__device__ __forceinline__ void gemm256_epilogue(const Gemm256P& p, f32x4_t (&acc)[MB][NB], int m0, int n0, int lane) {
  constexpr bool SILU = P3V_GATED(EPI), F32 = EPI == P3V_EPI_BIAS_RESID_F32 || EPI == P3V_EPI_F32 || EPI == P3V_EPI_SCALE_RESID_F32;
  constexpr bool RESID = EPI == P3V_EPI_RESID_BF16 || EPI == P3V_EPI_BIAS_RESID_F32 || EPI == P3V_EPI_SCALE_RESID_F32;
  constexpr bool BIAS = EPI == P3V_EPI_BIAS || EPI == P3V_EPI_BIAS_QGELU || EPI == P3V_EPI_BIAS_GELU || EPI == P3V_EPI_BIAS_RESID_F32 || EPI == P3V_EPI_SCALE_RESID_F32;
  constexpr int ES = F32 ? 4 : 2;                                        // bytes of an output
  const int fc = lane & 15, fq = lane >> 4;
  const size_t first = ((size_t)m0 * p.ldo + n0) * ES;
  const __amdgpu_buffer_rsrc_t rs_o = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)p.out + first, 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_r = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)p.resid + (RESID ? first : 0), 0, 0x7fffffff, 0x00020000);
  // (bytes from the wave's first output; beyond the descriptor for rows beyond M)
  auto row = [&](int i) { return m0 + fc + i * 16 < p.M ? (fc + i * 16) * p.ldo * ES : (int)0x80000000; };
  // A row's turn: nothing moves across it (the scheduler would bring all residual loads forward, and spill).  AGPR: the sums lie in accumulation
  // registers and are to stay there until then (the allocator would read them all at once).
  auto take = [&](int i) {
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (AGPR)
#pragma unroll
      for (int j = 0; j < NB; ++j) asm volatile("" : "+a"(acc[i][j]));
  };
  if constexpr (SILU) {
    // wave columns: blocks 0, 1 = gate, blocks 2, 3 = up of the SAME 32 output columns n0 + [0, 32)
    const int col = ((fq & 1) * 16 + (fq >> 1) * 8) * ES;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      take(i);
      uint32_t pk[2][2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        // reference rounds gate/up to bf16 (Linear output) and every elementwise op after it (phi.py:469-471)
#pragma unroll
        for (int h = 0; h < 2; ++h) pk[j][h] = p3v_gated2(EPI, acc[i][j][2 * h], acc[i][j][2 * h + 1], acc[i][2 + j][2 * h], acc[i][2 + j][2 * h + 1]);
      }
      u32x4_t w;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        auto sw = __builtin_amdgcn_permlane16_swap(pk[0][k], pk[1][k], false, false);
        w[k] = sw[0], w[2 + k] = sw[1];
      }
      __builtin_amdgcn_raw_buffer_store_b128(w, rs_o, row(i) + col, 0, 0);
    }
  } else {
    float bias[BIAS ? NB : 1][4];
    if constexpr (BIAS) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        u32x2_t bw = {0u, 0u};
        if (p.bias) bw = *(const u32x2_t*)(p.bias + n0 + j * 16 + fq * 4);
        bias[j][0] = bf16lo(bw[0]), bias[j][1] = bf16hi(bw[0]), bias[j][2] = bf16lo(bw[1]), bias[j][3] = bf16hi(bw[1]);
      }
    }
    // (residual rows are requested RN turns ahead, as far as registers go: one wave per SIMD, which nothing else covers, has most)
    constexpr int RN = AGPR ? (F32 ? 4 : MB) : F32 && MB > 4 ? 1 : 2;
    if constexpr (F32) {
      u32x4_t rws[RN][NB];
      auto ask = [&](int i) {
        if constexpr (RESID)
#pragma unroll
          for (int j = 0; j < NB; ++j) rws[i % RN][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_r, row(i) + fq * 16 + j * 64, 0, 0);
      };
#pragma unroll
      for (int i = 0; i < RN && i < MB; ++i) ask(i);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        take(i);
        const int at = row(i) + fq * 16;
        auto& rw = rws[i % RN];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          f32x4_t v = acc[i][j];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (EPI == P3V_EPI_BIAS_RESID_F32) v[r] += bias[j][r];
            if (EPI == P3V_EPI_SCALE_RESID_F32) v[r] *= bias[j][r];  // (`bias` carries the per-column scale)
          }
          if constexpr (RESID) v += __builtin_bit_cast(f32x4_t, rw[j]);
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), rs_o, at + j * 64, 0, 0);
        }
        if (i + RN < MB) ask(i + RN);
      }
    } else {
      u32x4_t rws[RN][NB / 2];
      u32x2_t rws1[RN];
      // (the block without a partner, NB odd: four columns, 8 bytes)
      auto pair_at = [&](int i) { return row(i) + ((fq & 1) * 16 + (fq >> 1) * 8) * 2; };
      auto one_at = [&](int i) { return row(i) + ((NB - 1) * 16 + fq * 4) * 2; };
      auto ask = [&](int i) {
        if constexpr (RESID) {
#pragma unroll
          for (int jp = 0; jp < NB / 2; ++jp) rws[i % RN][jp] = __builtin_amdgcn_raw_buffer_load_b128(rs_r, pair_at(i) + jp * 64, 0, 0);
          if constexpr (NB & 1) rws1[i % RN] = __builtin_amdgcn_raw_buffer_load_b64(rs_r, one_at(i), 0, 0);
        }
      };
#pragma unroll
      for (int i = 0; i < RN && i < MB; ++i) ask(i);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        take(i);
        const int at = pair_at(i), at1 = one_at(i);
        auto& rw = rws[i % RN];
        auto& rw1 = rws1[i % RN];
        uint32_t pk[NB][2];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[r] = acc[i][j][r];
            if constexpr (BIAS) v[r] += bias[j][r];
            if (EPI == P3V_EPI_BIAS_QGELU) v[r] = v[r] * p3v_sigmoid(1.702f * v[r]);
            else if (EPI == P3V_EPI_BIAS_GELU) v[r] = p3v_gelu_erf(v[r]);
          }
          pk[j][0] = pack_bf16x2(v[0], v[1]), pk[j][1] = pack_bf16x2(v[2], v[3]);
        }
        auto add = [](uint32_t r, uint32_t w) { return pack_bf16x2(bf16lo(r) + bf16lo(w), bf16hi(r) + bf16hi(w)); };   // resid + bf16(acc)
#pragma unroll
        for (int jp = 0; jp < NB / 2; ++jp) {
          u32x4_t w;
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            auto sw = __builtin_amdgcn_permlane16_swap(pk[2 * jp][k], pk[2 * jp + 1][k], false, false);
            w[k] = sw[0], w[2 + k] = sw[1];
          }
          if constexpr (RESID)
#pragma unroll
            for (int k = 0; k < 4; ++k) w[k] = add(rw[jp][k], w[k]);
          __builtin_amdgcn_raw_buffer_store_b128(w, rs_o, at + jp * 64, 0, 0);
        }
        if constexpr (NB & 1) {
          u32x2_t w = {pk[NB - 1][0], pk[NB - 1][1]};
          if constexpr (RESID) w[0] = add(rw1[0], w[0]), w[1] = add(rw1[1], w[1]);
          __builtin_amdgcn_raw_buffer_store_b64(w, rs_o, at1, 0, 0);
        }
        if (i + RN < MB) ask(i + RN);
      }
    }
  }
}
