// Dense projection  C[M,N] = A[M,K] * W[N,K]^T  on the gfx950 matrix cores.
//
// Both operands are K-contiguous, which is exactly the MFMA A/B fragment order
// (each lane owns 8 consecutive k), so no transposes anywhere.
//
//   tile      128(M) x 128(N) x 64(K), 256 threads = 4 waves as 2(M) x 2(N),
//             each wave 64x64 = 4x4 v_mfma_f32_16x16x32_bf16 accumulators
//   staging   global_load_lds_dwordx4 (LDS-DMA, 1 KiB = 8 rows x 128 B per
//             wave-instruction), two LDS buffers (64 KiB), one barrier per K tile
//   LDS       rows of 128 B; 16-B chunk c of row r is stored at chunk c^(r&7)
//             (XOR swizzle applied on the per-lane SOURCE address because the
//             DMA destination is lane-linear; the same XOR on the ds_read_b128
//             side) -> conflict-free fragment reads
//   epilogue  compile-time variant (bias / quick-GELU / erf-GELU / residual /
//             SiLU*up / patch-embed row remap), straight from the accumulators: the
//             MFMAs take the W fragment FIRST, so a lane holds 4 consecutive columns
//             of one output row; bf16 outputs pair two column blocks with
//             v_permlane16_swap -> 16-byte stores of 8 consecutive columns, no LDS
//             staging.
//
// Roofline: MFMA-bound for M >= ~512 (2*M*N*K flops vs (M+N)*K*2 bytes).
#include <stdlib.h>
#include <string.h>


#include "p3v_gemm_qkv.h"

#define P3V_EPI_QKV 100                // internal: qkv projection with split + RoPE + KV append in the epilogue (p3v_gemm_qkv.h)

#define BM 128
#define BN 128
#define BK 64
#define TILE_BYTES (BM * BK * 2)   // 16 KiB per operand tile
#define GEMM_LDS (4 * TILE_BYTES)   // two stages of an A and a W tile: 64 KiB -> two workgroups per CU

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

struct GemmP {
  const bf16_t* A; const bf16_t* W; void* out; const bf16_t* bias; const void* resid; const bf16_t* pos;
  int M, N, K, lda, ldw, ldo, ppi;
  int kslice;   // split-K (EPI_F32 only): workgroup z covers k in [z*kslice, (z+1)*kslice) and writes fp32 partial z ([M, ldo] each)
  QkvP q;       // P3V_EPI_QKV only
};


__device__ __forceinline__ void load8_bf16(const bf16_t* p, float* v) {
  const u32x4_t w = *(const u32x4_t*)p;
#pragma unroll
  for (int j = 0; j < 4; ++j) { v[2 * j] = bf16lo(w[j]); v[2 * j + 1] = bf16hi(w[j]); }
}
__device__ __forceinline__ void store8_bf16(bf16_t* p, const float* v) {
  u32x4_t w;
#pragma unroll
  for (int j = 0; j < 4; ++j) w[j] = pack_bf16x2(v[2 * j], v[2 * j + 1]);
  *(u32x4_t*)p = w;
}

template <int EPI, int ORD = 0>
__global__ void __launch_bounds__(256, 2) k_gemm(GemmP p) {
  constexpr bool SILU = P3V_GATED(EPI), QKV = EPI == P3V_EPI_QKV;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: LDS-DMA bases stay in SGPRs
  const int wr = wave >> 1, wc = wave & 1;
  const int n_out_tile = SILU ? BN / 2 : BN;
  // XCD-aware tile order: the dispatcher places workgroup i on XCD i % 8 (speed only, never correctness), so
  // give each XCD a contiguous run of tiles; inside a run tiles walk N fastest within a band of 8 M-tiles,
  // i.e. the tiles resident on one XCD share A row panels and W panels through that XCD's 4 MiB L2.
  int m_t, n_t;
  {
    const int gx = gridDim.x, gy = gridDim.y, nwg = gx * gy, wid = blockIdx.y * gx + blockIdx.x;
    const int q = nwg >> 3, r = nwg & 7, xcd = wid & 7, loc = wid >> 3;
    const int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + loc;       // bijective for any nwg
    constexpr int BAND = 8;
    const int band = id / (BAND * gx), in_band = id % (BAND * gx);
    const int rows = min(BAND, gy - band * BAND);
    m_t = band * BAND + in_band % rows;
    n_t = in_band / rows;
  }
  const int m0 = m_t * BM;
  int n0 = n_t * n_out_tile;
  // P3V_EPI_QKV (p3v_gemm_qkv.h): column tiles 0 .. nq-1 are Q, then K (both fetched in rotation-pair order), then V, whose tiles
  // are computed with the operand roles swapped (W rows on the tile's A side, tokens on its B side)
  bool swapped = false, is_k = false;
  int row0 = 0;
  if (QKV) {
    const int nq_t = p.q.nh * p.q.hd / BN, nk_t = p.q.nkv * p.q.hd / BN;
    swapped = n_t >= nq_t + nk_t;
    is_k = !swapped && n_t >= nq_t;
    row0 = swapped ? (p.q.nh + p.q.nkv) * p.q.hd : is_k ? p.q.nh * p.q.hd : 0;
    n0 = (n_t - (swapped ? nq_t + nk_t : is_k ? nq_t : 0)) * BN;       // first column INSIDE the region
  }

  // ---- staging addresses: wave w issues 4 DMA pieces per operand, piece q covers tile rows (w*4+q)*8 .. +8
  const int srow = lane >> 3, schunk = lane & 7;
  // byte offsets from p.A / p.W: the DMA is issued in its MUBUF form (`buffer_load ... lds`).  A pending `global_load_lds`
  // is, for the compiler's wait-count model, a FLAT access of both memories, and every later s_waitcnt becomes
  // vmcnt(0) / lgkmcnt(0): the counted lgkmcnt on the fragment reads below was silently a full wait.
  unsigned a_src[4], b_src[4];
  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, 0xffffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_ww = __builtin_amdgcn_make_buffer_rsrc((void*)p.W, 0, 0xffffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_a = QKV && swapped ? rs_ww : rs_x, rs_w = QKV && swapped ? rs_x : rs_ww;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = (wave * 4 + q) * 8 + srow;                 // tile row 0..127
    const int sw = (schunk ^ (r & 7)) * 8;                   // swizzled source chunk (elements)
    int ar = m0 + r;
    ar = ar < p.M ? ar : p.M - 1;
    int br;
    if (SILU) {
      const int wcol = r >> 6, ni = (r & 63) >> 4, c = r & 15;
      br = n0 + wcol * 32 + (ni & 1) * 16 + c;
      br = (br < p.N ? br : p.N - 1) + (ni >> 1) * p.N;      // up rows live N rows below the gate rows
    } else if (QKV) {
      br = qkv_pair_row(p.q, row0, n0 >> 1, r);
    } else {
      br = n0 + r;
      br = br < p.N ? br : p.N - 1;
    }
    if (QKV && swapped) {                                    // A side: W rows row0 + n0 + r; B side: token rows (clamped)
      a_src[q] = (unsigned)(((size_t)(row0 + n0 + r) * p.ldw + sw) * 2);
      b_src[q] = (unsigned)(((size_t)ar * p.lda + sw) * 2);
    } else {
      a_src[q] = (unsigned)(((size_t)ar * p.lda + sw) * 2);
      b_src[q] = (unsigned)(((size_t)br * p.ldw + sw) * 2);
    }
  }
  const int kz = p.kslice ? (int)blockIdx.z : 0;              // split-K slice (0 when not split)
  const int nk = (p.kslice ? p.kslice : p.K) / BK, kt0 = kz * nk;

  auto stage = [&](int kt, int buf) {
    unsigned char* base = smem + buf * (2 * TILE_BYTES);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int piece = (wave * 4 + q) * 1024;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, (lptr_t)(base + piece), 16, a_src[q], (kt0 + kt) * (BK * 2), 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_w, (lptr_t)(base + TILE_BYTES + piece), 16, b_src[q], (kt0 + kt) * (BK * 2), 0, 0);
    }
  };

  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

  // fragment read offsets (bytes) inside a tile: row = base + (lane&15), logical chunk = kk*4 + (lane>>4)
  const int frow = lane & 15, fchunk = lane >> 4;

  stage(0, 0);
  for (int kt = 0; kt < nk; ++kt) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (ORD == 0 && kt + 1 < nk) stage(kt + 1, (kt + 1) & 1);
    const unsigned char* ta = smem + (kt & 1) * (2 * TILE_BYTES);
    const unsigned char* tb = ta + TILE_BYTES;
    // All 16 fragment reads of the K-tile are requested up front (64 VGPRs) and the MFMAs of the first k-step start as
    // soon as ITS eight have landed (LDS returns in order -> counted lgkmcnt): one exposed LDS latency per K-tile instead
    // of four (hipcc otherwise recycles two A registers and waits lgkmcnt(0) before every run of eight MFMAs).
    bf16x8_t af[2][4], bfr[2][4];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = wr * 64 + i * 16 + frow;
        af[kk][i] = *(const bf16x8_t*)(ta + r * 128 + (((kk * 4 + fchunk) ^ (r & 7)) << 4));
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = wc * 64 + j * 16 + frow;
        bfr[kk][j] = *(const bf16x8_t*)(tb + r * 128 + (((kk * 4 + fchunk) ^ (r & 7)) << 4));
      }
    }
    if (ORD == 1 && kt + 1 < nk) stage(kt + 1, (kt + 1) & 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[kk][j], af[kk][i], acc[i][j], 0, 0, 0);   // W first: transposed block
      if (ORD == 2 && kk == 0) {
        __builtin_amdgcn_sched_barrier(0);
        if (kt + 1 < nk) stage(kt + 1, (kt + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // ---- epilogue straight from the accumulators (not staged through LDS between two barriers).  The
  // MFMAs take the W fragment first, so a 16 x 16 block comes out transposed: lane (c = lane & 15, q = lane >> 4) holds the four
  // consecutive columns 4q .. 4q+3 of output row c.  fp32 outputs store them as they are (16 bytes); bf16 outputs first trade
  // packed halves of two neighbouring column blocks between lanes q and q ^ 1 (v_permlane16_swap): 8 consecutive columns per lane.
  if constexpr (QKV) {
    if (!swapped) qkv_epilogue_rot<4>(p.q, acc, p.bias, is_k, row0, (n0 >> 1) + wc * 32, m0 + wr * 64, p.M, lane);
    else qkv_epilogue_vt<4>(p.q, acc, p.bias ? p.bias + row0 : nullptr, n0 + wr * 64, m0 + wc * 64, p.M, lane);
    return;
  }
  const int fc = lane & 15, fq = lane >> 4;
  const int mrow0 = m0 + wr * 64 + fc;                         // + i * 16
  if (SILU) {
    // wave tile columns: [0,32) gate, [32,64) up for output columns n0 + wc*32 + [0,32)
    const int n = n0 + wc * 32 + (fq & 1) * 16 + (fq >> 1) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t pk[2][2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int h = 0; h < 2; ++h) pk[j][h] = p3v_gated2(EPI, acc[i][j][2 * h], acc[i][j][2 * h + 1], acc[i][2 + j][2 * h], acc[i][2 + j][2 * h + 1]);
      }
      u32x4_t w;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        auto sw = __builtin_amdgcn_permlane16_swap(pk[0][k], pk[1][k], false, false);
        w[k] = sw[0], w[2 + k] = sw[1];
      }
      const int m = mrow0 + i * 16;
      if (m < p.M && n < p.N) *(u32x4_t*)((bf16_t*)p.out + (size_t)m * p.ldo + n) = w;
    }
    return;
  }

  float bias[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + wc * 64 + j * 16 + fq * 4;
    u32x2_t bw = {0u, 0u};
    if (p.bias && n < p.N) bw = *(const u32x2_t*)(p.bias + n);
    bias[j][0] = bf16lo(bw[0]), bias[j][1] = bf16hi(bw[0]), bias[j][2] = bf16lo(bw[1]), bias[j][3] = bf16hi(bw[1]);
  }
  if (EPI == P3V_EPI_BIAS_RESID_F32 || EPI == P3V_EPI_F32 || EPI == P3V_EPI_PATCH || EPI == P3V_EPI_SCALE_RESID_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = mrow0 + i * 16;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + wc * 64 + j * 16 + fq * 4;
        if (m < p.M && n < p.N) {
          const size_t o = (size_t)m * p.ldo + n;
          size_t oo = o;
          float4 v = make_float4(acc[i][j][0] + bias[j][0], acc[i][j][1] + bias[j][1], acc[i][j][2] + bias[j][2], acc[i][j][3] + bias[j][3]);
          if (EPI == P3V_EPI_SCALE_RESID_F32)                  // (`bias` carries the per-column scale)
            v = make_float4(acc[i][j][0] * bias[j][0], acc[i][j][1] * bias[j][1], acc[i][j][2] * bias[j][2], acc[i][j][3] * bias[j][3]);
          if (EPI == P3V_EPI_BIAS_RESID_F32 || EPI == P3V_EPI_SCALE_RESID_F32) {
            const float4 r4 = *(const float4*)((const float*)p.resid + o);
            v.x += r4.x, v.y += r4.y, v.z += r4.z, v.w += r4.w;
          } else if (EPI == P3V_EPI_PATCH) {
            const int img = m / p.ppi, pi = m % p.ppi;
            const u32x2_t pw = *(const u32x2_t*)(p.pos + (size_t)(1 + pi) * p.N + n);
            v.x += bf16lo(pw[0]), v.y += bf16hi(pw[0]), v.z += bf16lo(pw[1]), v.w += bf16hi(pw[1]);
            oo = ((size_t)img * (p.ppi + 1) + 1 + pi) * p.ldo + n;
          }
          if (EPI == P3V_EPI_F32) oo += (size_t)kz * p.M * p.ldo;
          *(float4*)((float*)p.out + oo) = v;
        }
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = mrow0 + i * 16;
#pragma unroll
    for (int jp = 0; jp < 2; ++jp) {
      uint32_t pk[2][2];
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int j = 2 * jp + jj;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] = acc[i][j][r] + bias[j][r];
          if (EPI == P3V_EPI_BIAS_QGELU) v[r] = v[r] * p3v_sigmoid(1.702f * v[r]);
          else if (EPI == P3V_EPI_BIAS_GELU) v[r] = p3v_gelu_erf(v[r]);
        }
        pk[jj][0] = pack_bf16x2(v[0], v[1]), pk[jj][1] = pack_bf16x2(v[2], v[3]);
      }
      u32x4_t w;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        auto sw = __builtin_amdgcn_permlane16_swap(pk[0][k], pk[1][k], false, false);
        w[k] = sw[0], w[2 + k] = sw[1];
      }
      const int n = n0 + wc * 64 + (2 * jp + (fq & 1)) * 16 + (fq >> 1) * 8;
      if (m < p.M && n < p.N) {
        const size_t o = (size_t)m * p.ldo + n;
        if (EPI == P3V_EPI_RESID_BF16) {                       // out = resid + bf16(acc): the packed words ARE bf16(acc)
          const u32x4_t rw = *(const u32x4_t*)((const bf16_t*)p.resid + o);
#pragma unroll
          for (int k = 0; k < 4; ++k) w[k] = pack_bf16x2(bf16lo(rw[k]) + bf16lo(w[k]), bf16hi(rw[k]) + bf16hi(w[k]));
        }
        *(u32x4_t*)((bf16_t*)p.out + o) = w;
      }
    }
  }
}

template <int EPI, int ORD>
static int launch_gemm_v(const GemmP& p, hipStream_t s) {
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm<EPI, ORD>, hipFuncAttributeMaxDynamicSharedMemorySize, GEMM_LDS) != hipSuccess)
      return P3V_ERR_HIP;
    attr_set = true;
  }
  const int n_tile = P3V_GATED(EPI) ? BN / 2 : BN;
  dim3 grid(p3v_cdiv(p.N, n_tile), p3v_cdiv(p.M, BM), p.kslice ? p.K / p.kslice : 1);
  hipLaunchKernelGGL((k_gemm<EPI, ORD>), grid, dim3(256), GEMM_LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}

template <int EPI>
static int launch_gemm(const GemmP& p, hipStream_t s) { return launch_gemm_v<EPI, 0>(p, s); }

int p3v_gemm256_try(const p3v_gemm_args_t* a, int mb, int nb, hipStream_t s);   // p3v_gemm256.hip: tiles of 32 mb x 64 nb, P3V_ERR_UNSUPPORTED if the shape does not fit
static int gemm128(const p3v_gemm_args_t* a, hipStream_t s);

// How many leading rows go to the 256 x 256 kernel (a multiple of 256, or M for all of them); the rest runs on the 128 x 128 kernel in a second
// launch on the same stream.  The machine holds 256 big workgroups or 512 small ones per round; a round of big tiles costs 1, a round of small ones
// 0.675, a last round that leaves every CU at most one small workgroup 0.42 -- the cheapest whole-round packing, e.g. 2531 x 16384 (gate_up): 8 x 64 =
// 512 big tiles = 2 rounds + 4 x 128 small = 1 round.  It runs where gemm_tile_choice names no tile: short K (< 1024), columns that no tile divides, and
// sizes where no tile promises 2 %.  The prices were measured on the eight-wave form of the big tile (1.31 PFLOP/s; 1.40 - 1.55 on four waves), a shorter
// K's on its 128-KiB prologue and staged epilogue; they have not been taken again.
static int gemm_big_rows(const p3v_gemm_args_t* a) {
  const int n_big = P3V_GATED(a->epilogue) ? 128 : 256, n_small = n_big / 2;
  if (a->M < 1024 || a->N % n_big || a->epilogue == P3V_EPI_PATCH) return 0;
  if (const int force = p3v_tuning().gemm_big_rows; force >= 0) return min(force / 256 * 256, a->M);   // tests: pin the split
  const int mt = p3v_cdiv(a->M, 256), nt_big = a->N / n_big, nt_small = p3v_cdiv(a->N, n_small);
  // a short K loop leaves the big tile's prologue and epilogue exposed (one workgroup per CU)
  const float big_round = a->K >= 2048 ? 1.0f : 1.0f + 0.25f * (2048 - a->K) / 1024.f;
  float best = 1e30f;
  int best_rows = 0;
  for (int ms = 0; ms <= mt; ++ms) {
    const int rows_big = min(ms * 256, a->M), rows_small = a->M - rows_big;
    const long big = (long)ms * nt_big, small = (long)p3v_cdiv(rows_small, 128) * nt_small;
    float c = (float)((big + 255) / 256) * big_round;
    if (small) {
      const long full = small / 512, rest = small % 512;
      c += 0.675f * full + (rest == 0 ? 0.f : rest <= 256 ? 0.42f : 0.675f);
    }
    if (big && small) c += 0.04f;                       // the second launch
    if (c < best - 1e-4f) { best = c; best_rows = rows_big; }
  }
  return best_rows;
}

// The plan by whole rounds (*mb, *nb: a tile of 32 mb x 64 nb), or false: the packing above (or 128 x 128 tiles).  A launch lasts whole rounds of the
// chip's workgroups, so what counts is how a tile height divides the rows: 2531 x 3072 is 120 tiles of 256 x 256 (half the chip idle) but 240 of
// 128 x 256.  Times of one round in us, K-tiles of 64 = t, fitted to M = 1100 .. 9809 x the decoder's and the vision tower's projections: the flat tiles of
// p3v_gemm_pc.hip 6.6 + 0.69 t (128 x 256), 7.9 + 0.79 t (160 x 256), 5.5 + 0.61 t (128 x 192); the tall ones 9.5 + 1.28 t (256 x 256), 8.2 + 1.27 t (224 x
// 256), 8.1 + 1.11 t (256 x 192), a twentieth more per K-tile from the second round on (power); 512 tiles of 128 x 128 6.0 + 0.785 t, up to 256 of them 4.4 +
// 0.635 t.  A tile has to promise 5 %; short K loops (< 1024) stay.  The tall tiles' times are those of their eight-wave form (the four-wave one: 8.3 + 1.2 t
// at a full chip, gemm_tile_choice), so this is not what p3v_gemm runs: it is the choice's starting point, and the qkv projection's rule below 1024 rows.
static bool gemm_tile_plan(const p3v_gemm_args_t* a, int rows_big, int* mb, int* nb) {
  const bool gated = P3V_GATED(a->epilogue);
  if (a->M <= 256 || a->K < 1024 || a->epilogue == P3V_EPI_PATCH || p3v_tuning().gemm_128 || p3v_tuning().gemm_big_rows >= 0) return false;
  struct Tile { int mb, nb; float f, c, more; };
  static const Tile tiles[] = {{8, 4, 9.5f, 1.285f, 0.07f}, {7, 4, 8.2f, 1.27f, 0.03f}, {8, 3, 8.1f, 1.106f, 0.f},
                               {5, 4, 7.9f, 0.79f, 0.05f},  {4, 4, 6.6f, 0.69f, 0.05f}, {4, 3, 5.5f, 0.61f, 0.f}};
  const float kt = (float)(a->K / BK);
  auto time = [&](const Tile& t, int M) {
    const int rounds = p3v_cdiv((long)p3v_cdiv(M, 32 * t.mb) * (a->N / (gated ? 32 * t.nb : 64 * t.nb)), 256);
    return rounds * (t.f + t.c * kt) + (rounds > 1 ? (rounds - 1) * t.more * kt : 0.f);
  };
  float best = rows_big ? time(tiles[0], rows_big) : 0.f;
  if (rows_big < a->M) {
    const long small = (long)p3v_cdiv(a->M - rows_big, BM) * p3v_cdiv(a->N, gated ? BN / 2 : BN), rest = small % 512;
    best += (small / 512 + (rest > 256)) * (6.0f + 0.785f * kt) + (rest > 0 && rest <= 256 ? 4.4f + 0.635f * kt : 0.f) + (rows_big ? 3.8f : 0.f);
  }
  best *= 0.95f;
  bool found = false;
  for (const Tile& t : tiles) {
    if (a->N % (gated ? 32 * t.nb : 64 * t.nb) || (gated && t.nb != 4)) continue;
    const float c = time(t, a->M);
    if (c < best) { best = c; *mb = t.mb; *nb = t.nb; found = true; }
  }
  return found;
}

// The tile that p3v_gemm runs, 10 mb + nb, or 0: the packing.  The plan above knows rounds; how long one lasts also depends on how full it is
// (power: 24 workgroups of 256 x 256 over 128 K-tiles 137 us, 240 of them 155), and the tiles of 192 rows are priced here alone.  t K-tiles, r
// rounds of which u are filled: once + r (f + c t) + u fill t, and per round what a gated, a 32-bit residual or a GELU epilogue takes more; fitted to
// 20 heights, 257 .. 9809 rows, of eight projections of the decoder and the vision tower with their weights from memory (3 - 5 % of a time at
// most sizes).  Another tile than the plan's has to promise 2 %.  Where it names a tile, that is within 0.3 % of the fastest measured one on average, 8.7 %
// at most below 1000 rows and 6.4 % beyond (profiles/gemm_bf16_tile_sweep.txt, 130 sizes).  Measured (us, the plan on these kernels -> this): 2300 x 16384 x 3072
// (gate | up) 192 -> 169, 2531 193 -> 187, 768 67 -> 60; 2531 x 9216 x 3072 115 -> 107, 4096 175 -> 163; 3072 x 8192: 6000 rows 238 -> 219, 8192 313 -> 286;
// 2048 x 10496 x 3072 117 -> 107.
static int gemm_tile_choice(const p3v_gemm_args_t* a, int rows_big) {
  int mb = 0, nb = 0;
  const int plan = gemm_tile_plan(a, rows_big, &mb, &nb) ? 10 * mb + nb : 0;
  if (a->M <= 256 || a->K < 1024 || a->epilogue == P3V_EPI_PATCH || p3v_tuning().gemm_128 || p3v_tuning().gemm_big_rows >= 0) return plan;
  struct Tile { int mb, nb; float once, f, c, fill, gated, f32, act; };
  static const Tile tiles[] = {{8, 4, 2.9f, 8.3f, 0.94f, 0.258f, 1.4f, 7.1f, 0.f}, {7, 4, 3.1f, 7.f, 0.857f, 0.214f, 1.4f, 6.3f, 0.f},
                               {6, 4, 3.9f, 5.5f, 0.765f, 0.193f, 1.8f, 5.2f, 0.f}, {8, 3, 3.f, 6.3f, 0.754f, 0.207f, 0.f, 5.3f, 0.f},
                               {6, 3, 5.9f, 3.9f, 0.6f, 0.166f, 0.f, 3.9f, 0.f}, {5, 4, 5.2f, 2.5f, 0.698f, 0.199f, 1.8f, 4.1f, 1.8f},
                               {4, 4, 5.4f, 1.6f, 0.64f, 0.167f, 1.4f, 3.4f, 1.5f}, {4, 3, 6.5f, 3.6f, 0.467f, 0.144f, 0.f, 2.5f, 1.1f}};
  const bool gated = P3V_GATED(a->epilogue), f32 = a->epilogue == P3V_EPI_BIAS_RESID_F32 || a->epilogue == P3V_EPI_SCALE_RESID_F32 || a->epilogue == P3V_EPI_F32;
  const bool act = a->epilogue == P3V_EPI_BIAS_QGELU || a->epilogue == P3V_EPI_BIAS_GELU;
  const float kt = (float)(a->K / BK);
  auto time = [&](const Tile& t, int M) {
    const long n = (long)p3v_cdiv(M, 32 * t.mb) * (a->N / (gated ? 32 * t.nb : 64 * t.nb));
    const float used = n / 256.f, rounds = (float)((n + 255) / 256);
    return t.once + rounds * (t.f + (gated ? t.gated : f32 ? t.f32 : act ? t.act : 0.f) + t.c * kt) + used * t.fill * kt;
  };
  float best = 0.f;
  if (plan) {
    for (const Tile& t : tiles)
      if (plan == 10 * t.mb + t.nb) best = time(t, a->M);
  } else {
    if (rows_big) best = time(tiles[0], rows_big);
    if (rows_big < a->M) {
      const long small = (long)p3v_cdiv(a->M - rows_big, BM) * p3v_cdiv(a->N, gated ? BN / 2 : BN), rest = small % 512;
      best += (small / 512 + (rest > 256)) * (6.0f + 0.95f * kt) + (rest > 0 && rest <= 256 ? 4.4f + 0.85f * kt : 0.f) + (rows_big ? 3.8f : 0.f);
    }
  }
  best *= 0.98f;
  int choice = plan;
  for (const Tile& t : tiles) {
    if (a->N % (gated ? 32 * t.nb : 64 * t.nb) || (gated && t.nb != 4)) continue;
    const float c = time(t, a->M);
    if (c < best) best = c, choice = 10 * t.mb + t.nb;
  }
  return choice;
}

extern "C" int p3v_gemm_plan(int M, int N, int K, int epilogue) {
  if (M <= 0 || N <= 0 || K <= 0 || epilogue < 0 || epilogue > P3V_EPI_GELU_MUL) return 0;
  p3v_gemm_args_t a = {};
  a.M = M, a.N = N, a.K = K, a.epilogue = epilogue;
  int mb, nb;
  return gemm_tile_plan(&a, p3v_tuning().gemm_128 ? 0 : gemm_big_rows(&a), &mb, &nb) ? 10 * mb + nb : 0;
}

int p3v_gemm_skinny_slices(int M, int N, int K, int epilogue);   // p3v_gemm_skinny.hip: 0 = not one of its shapes
static int splitk_slices(int M, int N, int K, int epilogue);
extern "C" int p3v_gemm_tile(int M, int N, int K, int epilogue) {
  if (M <= 0 || N <= 0 || K <= 0 || epilogue < 0 || epilogue > P3V_EPI_GELU_MUL) return 0;
  p3v_gemm_args_t a = {};
  a.M = M, a.N = N, a.K = K, a.epilogue = epilogue;
  if (K % BK || p3v_gemm_skinny_slices(M, N, K, epilogue) || splitk_slices(M, N, K, epilogue) > 1) return 0;      // (p3v_gemm tries these first)
  return gemm_tile_choice(&a, p3v_tuning().gemm_128 ? 0 : gemm_big_rows(&a));
}

// ---- split-K for prompt-sized-but-small M (17 .. 256 rows: short chat prompts, the text group of a mixed batch).  One
// 128-row tile leaves N / 128 = 24 .. 128 workgroups, each walking the WHOLE K loop with one tile in flight: an iteration is
// one DMA round trip (~0.6 us), so down_proj (K = 8192) took 78 us for a 50 MB weight matrix and a 17..256-token prefill
// 8.3-9.5 ms, flat in the length.  Here S slices of K run as gridDim.z (fp32 partials [S, M, N] in the CALLER's workspace:
// p3v_gemm_ws_bytes() sizes it, the library never allocates) and a second launch adds them in slice order (deterministic)
// and applies the epilogue.  Without a workspace of that size the shape runs on the one-pass kernels.
template <int EPI>
__global__ void __launch_bounds__(256) k_splitk_reduce(const float* __restrict__ part, void* __restrict__ out, const void* __restrict__ resid,
                                                       const bf16_t* __restrict__ col_scale, int M, int N, int ldp, int ldo, int S) {
  constexpr bool SILU = P3V_GATED(EPI);             // part holds [gate | up] columns (2N), out N columns
  const int per_row = N / 8;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)M * per_row) return;
  const int m = (int)(i / per_row), n = (int)(i - (long)m * per_row) * 8;
  float v[8] = {0, 0, 0, 0, 0, 0, 0, 0}, u[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
  for (int z = 0; z < S; ++z) {
    const float* pr = part + ((size_t)z * M + m) * ldp + n;
    const float4 a0 = *(const float4*)pr, a1 = *(const float4*)(pr + 4);
    v[0] += a0.x; v[1] += a0.y; v[2] += a0.z; v[3] += a0.w; v[4] += a1.x; v[5] += a1.y; v[6] += a1.z; v[7] += a1.w;
    if (SILU) {
      const float4 b0 = *(const float4*)(pr + N), b1 = *(const float4*)(pr + N + 4);
      u[0] += b0.x; u[1] += b0.y; u[2] += b0.z; u[3] += b0.w; u[4] += b1.x; u[5] += b1.y; u[6] += b1.z; u[7] += b1.w;
    }
  }
  const size_t o = (size_t)m * ldo + n;
  if (SILU) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = p3v_gated(EPI, v[e], u[e]);
  } else if (EPI == P3V_EPI_RESID_BF16) {
    float r[8];
    load8_bf16((const bf16_t*)resid + o, r);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = r[e] + bf16_round(v[e]);
  }
  if (EPI == P3V_EPI_SCALE_RESID_F32 || EPI == P3V_EPI_BIAS_RESID_F32) {
    float c[8] = {0, 0, 0, 0, 0, 0, 0, 0};          // (col_scale carries the bias of the latter; may be null)
    if (EPI == P3V_EPI_SCALE_RESID_F32 || col_scale) load8_bf16(col_scale + n, c);
    const float* r = (const float*)resid + o;
    const float4 r0 = *(const float4*)r, r1 = *(const float4*)(r + 4);
    if (EPI == P3V_EPI_BIAS_RESID_F32) {
      *(float4*)((float*)out + o) = make_float4(r0.x + (v[0] + c[0]), r0.y + (v[1] + c[1]), r0.z + (v[2] + c[2]), r0.w + (v[3] + c[3]));
      *(float4*)((float*)out + o + 4) = make_float4(r1.x + (v[4] + c[4]), r1.y + (v[5] + c[5]), r1.z + (v[6] + c[6]), r1.w + (v[7] + c[7]));
      return;
    }
    *(float4*)((float*)out + o) = make_float4(r0.x + c[0] * v[0], r0.y + c[1] * v[1], r0.z + c[2] * v[2], r0.w + c[3] * v[3]);
    *(float4*)((float*)out + o + 4) = make_float4(r1.x + c[4] * v[4], r1.y + c[5] * v[5], r1.z + c[6] * v[6], r1.w + c[7] * v[7]);
    return;
  }
  store8_bf16((bf16_t*)out + o, v);
}

// The reduction of a split whose consumer is an RMSNorm (o_proj / down_proj of a short prompt): adds the S partials in slice order,
// out = resid + bf16(sum) exactly as k_splitk_reduce<P3V_EPI_RESID_BF16>, and writes RMSNorm(out) beside it -- the residual stream
// and the next projection's input from ONE launch instead of two.  A workgroup per row, a thread per 8 columns (every load of the
// launch in flight at once: with k_rmsnorm_r's one wave per row, 128 rows keep 128 waves busy and the launch takes longer than the
// two it replaces).  The sum of squares is k_rmsnorm_r's, bit for bit: that kernel's lane l adds p = lo*lo + fl(hi*hi) of its chunks
// l, l + 64, ... one pair at a time; here every thread computes the four p of ITS chunk, and wave 0 adds them in that order.
// What bounds it is the launch and its trips to memory: residual and gain are requested ahead of the partials' sums (behind them they were a second
// trip: a 128-token prompt with 62 of these launches 3147 -> 3128 us, four steps of 15 rows with 124 9387 -> 9359).
__global__ void __launch_bounds__(384) k_splitk_reduce_norm(const float* __restrict__ part, bf16_t* __restrict__ out, const bf16_t* __restrict__ resid,
                                                            const u32x4_t* __restrict__ norm_w, u32x4_t* __restrict__ normed, int M, int N,
                                                            int ldo, int S, float inv_h, float eps) {
  __shared__ float ps[6 * 4][64];
  __shared__ float r_sh;
  const int row = blockIdx.x, c = threadIdx.x, lane = c & 63, wv = c >> 6, chunks = N / 8;
  u32x4_t v = {0u, 0u, 0u, 0u}, g = {0u, 0u, 0u, 0u};
  if (c < chunks) {
    const size_t o = (size_t)row * ldo + c * 8;
    const u32x4_t rr = *(const u32x4_t*)(resid + o);             // (residual and gain are requested with the partials, not behind them)
    g = norm_w[c];
    __builtin_amdgcn_sched_barrier(0);
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
    for (int z = 0; z < S; ++z) {
      const float* pr = part + ((size_t)z * M + row) * N + c * 8;
      const float4 a0 = *(const float4*)pr, a1 = *(const float4*)(pr + 4);
      acc[0] += a0.x; acc[1] += a0.y; acc[2] += a0.z; acc[3] += a0.w; acc[4] += a1.x; acc[5] += a1.y; acc[6] += a1.z; acc[7] += a1.w;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = (e & 1 ? bf16hi(rr[e >> 1]) : bf16lo(rr[e >> 1])) + bf16_round(acc[e]);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = pack_bf16x2(acc[2 * j], acc[2 * j + 1]);
    *(u32x4_t*)(out + o) = v;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float lo = bf16lo(v[j]), hi = bf16hi(v[j]);
    float hh = hi * hi;
    asm volatile("" : "+v"(hh));                                // (one rounding of hi*hi, then ONE fma: k_rmsnorm_r's compiled form)
    ps[wv * 4 + j][lane] = __builtin_fmaf(lo, lo, hh);
  }
  __syncthreads();
  if (wv == 0) {
    float ss = ps[0][lane];
#pragma unroll
    for (int k = 1; k < 24; ++k) {
      ss += ps[k][lane];
      asm volatile("" : "+v"(ss));
    }
    const float r = rsqrtf(wave_sum(ss) * inv_h + eps);
    if (lane == 0) r_sh = r;
  }
  __syncthreads();
  if (c < chunks) {
    const float r = r_sh;
    u32x4_t o4;
#pragma unroll
    for (int j = 0; j < 4; ++j) o4[j] = rms_pair(v[j], r, g[j]);
    normed[(size_t)row * chunks + c] = o4;
  }
}

// number of K slices for a shape (1 = not a split-K shape)
static int splitk_slices(int M, int N, int K, int epilogue) {
  const P3vTuning& t = p3v_tuning();
  const bool silu = P3V_GATED(epilogue);
  if (t.gemm_no_splitk || M <= 16 || M > t.gemm_splitk_max_m /* beyond, every projection has >= 256 tiles anyway */ ||
      N % 128 || K % 512)
    return 1;
  if (epilogue != P3V_EPI_NONE && epilogue != P3V_EPI_RESID_BF16 && epilogue != P3V_EPI_SCALE_RESID_F32 && !silu) return 1;
  const int w_rows = silu ? 2 * N : N;                        // SiLU: [gate; up] taken as 2N plain output columns
  const int tiles = p3v_cdiv(M, BM) * (w_rows / BN);
  int S = 1;
  while (S < t.gemm_splitk_max_s && tiles * S < t.gemm_splitk_wgs && (K / (2 * S)) % BK == 0 && K / (2 * S) >= 2 * BK) S *= 2;
  return S;
}

int p3v_splitk_slices(int M, int N, int K, int epilogue) { return splitk_slices(M, N, K, epilogue); }

int p3v_gemm_skinny_try(const p3v_gemm_args_t* a, hipStream_t s);
int p3v_gemm_skinny_tall(const p3v_gemm_args_t* a, hipStream_t s);

extern "C" int64_t p3v_gemm_ws_bytes(int M, int N, int K, int epilogue) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int sk = p3v_gemm_skinny_slices(M, N, K, epilogue);
  const int S = sk ? sk : splitk_slices(M, N, K, epilogue);
  if (S == 1) return 0;
  return (int64_t)S * M * (P3V_GATED(epilogue) ? 2 * N : N) * 4;
}
int p3v_gemm_skinny_most_slices(int M, int N, int K, int epilogue);   // p3v_gemm_skinny.hip: with a workspace for its 96-column tiles
extern "C" int64_t p3v_gemm_ws_most_bytes(int M, int N, int K, int epilogue) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int sk = p3v_gemm_skinny_most_slices(M, N, K, epilogue);
  return sk > 1 ? (int64_t)sk * M * (P3V_GATED(epilogue) ? 2 * N : N) * 4 : p3v_gemm_ws_bytes(M, N, K, epilogue);
}

// ---- out = resid + bf16(A W^T) and normed = RMSNorm(out) (include/p3v.h): only where the projection runs as K slices anyway
int p3v_gemm_skinny_partials(const p3v_gemm_args_t* a, int* S_out, hipStream_t s);   // p3v_gemm_skinny.hip
extern "C" int p3v_gemm_resid_norm(const p3v_gemm_args_t* a, const uint16_t* norm_w, float eps, uint16_t* normed, void* stream) {
  if (!a || !a->A || !a->W || !a->out || !a->resid || !norm_w || !normed) return P3V_ERR_ARG;
  if (a->epilogue != P3V_EPI_RESID_BF16 || a->M <= 0 || a->N <= 0 || a->K <= 0 || a->K % BK || a->N % 8 || a->ldo % 8 || a->ldo < a->N) return P3V_ERR_ARG;
  if (a->lda < a->K || a->ldw < a->K || a->lda % 8 || a->ldw % 8) return P3V_ERR_ARG;
  if (((uintptr_t)a->A | (uintptr_t)a->W | (uintptr_t)a->out | (uintptr_t)a->resid | (uintptr_t)norm_w | (uintptr_t)normed | (uintptr_t)a->ws) & 15)
    return P3V_ERR_ARG;
  if (a->N > 6 * 64 * 8 || a->bias || (size_t)a->N * a->ldw * 2 >= (1ull << 32)) return P3V_ERR_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  int S = 0;
  const int rc = p3v_gemm_skinny_partials(a, &S, s);           // P3V_ERR_UNSUPPORTED (nothing launched) unless the shape splits
  if (rc != P3V_OK) return rc;
  hipLaunchKernelGGL(k_splitk_reduce_norm, dim3(a->M), dim3(384), 0, s, (const float*)a->ws, (bf16_t*)a->out, (const bf16_t*)a->resid,
                     (const u32x4_t*)norm_w, (u32x4_t*)normed, a->M, a->N, a->ldo, S, 1.0f / (float)a->N, eps);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}

// the second launch of a split: adds the S fp32 partials [S, M, W rows] in slice order and applies the epilogue
int p3v_splitk_reduce(const float* part, const p3v_gemm_args_t* a, int S, hipStream_t s) {
  const bool silu = P3V_GATED(a->epilogue);
  const int w_rows = silu ? 2 * a->N : a->N;
  const long items = (long)a->M * (a->N / 8);
  const dim3 grid((unsigned)p3v_cdiv(items, 256));
  if (a->epilogue == P3V_EPI_GELU_MUL)
    hipLaunchKernelGGL(k_splitk_reduce<P3V_EPI_GELU_MUL>, grid, dim3(256), 0, s, part, a->out, a->resid, a->col_scale, a->M, a->N, w_rows, a->ldo, S);
  else if (silu) hipLaunchKernelGGL(k_splitk_reduce<P3V_EPI_SILU_MUL>, grid, dim3(256), 0, s, part, a->out, a->resid, a->col_scale, a->M, a->N, w_rows, a->ldo, S);
  else if (a->epilogue == P3V_EPI_SCALE_RESID_F32)
    hipLaunchKernelGGL(k_splitk_reduce<P3V_EPI_SCALE_RESID_F32>, grid, dim3(256), 0, s, part, a->out, a->resid, a->col_scale, a->M, a->N, w_rows, a->ldo, S);
  else if (a->epilogue == P3V_EPI_BIAS_RESID_F32)
    hipLaunchKernelGGL(k_splitk_reduce<P3V_EPI_BIAS_RESID_F32>, grid, dim3(256), 0, s, part, a->out, a->resid, a->bias, a->M, a->N, w_rows, a->ldo, S);
  else if (a->epilogue == P3V_EPI_RESID_BF16)
    hipLaunchKernelGGL(k_splitk_reduce<P3V_EPI_RESID_BF16>, grid, dim3(256), 0, s, part, a->out, a->resid, a->col_scale, a->M, a->N, w_rows, a->ldo, S);
  else hipLaunchKernelGGL(k_splitk_reduce<P3V_EPI_NONE>, grid, dim3(256), 0, s, part, a->out, a->resid, a->col_scale, a->M, a->N, w_rows, a->ldo, S);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}

// returns P3V_ERR_UNSUPPORTED when the shape is not one for split-K (or the caller gave no workspace for it)
static int gemm_splitk(const p3v_gemm_args_t* a, hipStream_t s) {
  const bool silu = P3V_GATED(a->epilogue);
  const int S = splitk_slices(a->M, a->N, a->K, a->epilogue);
  if (S == 1) return P3V_ERR_UNSUPPORTED;
  const int w_rows = silu ? 2 * a->N : a->N;
  if (!a->ws || a->ws_bytes < (int64_t)S * a->M * w_rows * 4) return P3V_ERR_UNSUPPORTED;
  if ((uintptr_t)a->ws & 15) return P3V_ERR_ARG;
  float* part = (float*)a->ws;
  GemmP p = {a->A, a->W, part, nullptr, nullptr, nullptr, a->M, w_rows, a->K, a->lda, a->ldw, w_rows, 0, a->K / S, {}};
  const int rc = launch_gemm<P3V_EPI_F32>(p, s);
  if (rc != P3V_OK) return rc;
  return p3v_splitk_reduce(part, a, S, s);
}

// ---- K slices on the flat tiles (p3v_gemm_pc.hip): residual projections of some hundred rows, whose tiles leave most of the chip idle.
// 300 x 3072 has 48 tiles of 128 x 192 and 1154 x 1024 (two image crops) 40 of 128 x 256: as many slices of K as one round of the chip takes,
// whole K-tiles each, fp32 partials in the caller's workspace, and a second launch that adds them in slice order.  Measured in us, with the
// RMSNorm behind it where there is one, against the paths of p3v_gemm (+ p3v_rmsnorm): 300 x 3072 x 8192 44.6 -> 31.7, 512 56.2 -> 39.3,
// 1000 90.5 -> 59.5, 1536 91.8 -> 78.6; 512 x 3072 x 3072 31.8 -> 25.8, 1100 51.5 -> 37.5; 577 x 1024 x 4096 (bias, fp32 residual) 60.6 -> 22.8,
// 2308 58.8 -> 33.8, 4039 60.9 -> 45.5.
// The rule: one round's time by tile, fitted to those and 40 more (within 2 us): a constant for both launches, the K-tiles of the longest slice,
// and 0.2 us per MB of partials written and read.  It has to promise 5 % over one pass on one of the flat tiles (gemm_tile_plan's times) and
// the 6 us of the norm's own launch (up to 256 rows over the kernel for few rows, from where that needs two passes over a long K: 256 x 3072 x
// 8192 35.2 -> 30.8, 160 29.2 -> 27.8, 128 24.7 -> 25.4); the sizes it turns down measured slower (1300 x 3072 x 3072: 42.1 against 40.5; 1154 x 1024 x 1024: 21.1, 15.7).
struct SlicePlan { int S, mb, nb; };
static SlicePlan gemm_slices_plan(int M, int N, int K, int epilogue) {
  const P3vTuning& t = p3v_tuning();
  const SlicePlan none = {0, 0, 0};
  if (!t.gemm_slices || (t.gemm_slices < 0 && M <= (K < 8192 ? 256 : 192)) || K % BK) return none;
  if (epilogue != P3V_EPI_RESID_BF16 && epilogue != P3V_EPI_BIAS_RESID_F32 && epilogue != P3V_EPI_SCALE_RESID_F32) return none;
  if (t.gemm_slices > 0) {
    const SlicePlan p = {t.gemm_slices / 100, t.gemm_slices / 10 % 10, t.gemm_slices % 10};
    return p.S < 1 || p.S > K / BK || !p.nb || N % (64 * p.nb) ? none : p;
  }
  struct Tile { int mb, nb; float f, c, one_f, one_c; };
  static const Tile tiles[] = {{4, 3, 13.3f, 0.64f, 5.5f, 0.61f}, {4, 4, 14.f, 0.72f, 6.6f, 0.69f}, {5, 4, 15.f, 0.87f, 7.9f, 0.79f}};
  const int nk = K / BK;
  float one = 1e30f, best = 1e30f;
  SlicePlan plan = none;
  for (const Tile& t : tiles) {
    if (N % (64 * t.nb)) continue;
    const long n = (long)p3v_cdiv(M, 32 * t.mb) * (N / (64 * t.nb));
    one = fminf(one, (float)p3v_cdiv(n, 256) * (t.one_f + t.one_c * nk));
    for (int S = 2; S <= 16 && n * S <= 256 && nk >= 3 * S; ++S) {
      const float c = t.f + t.c * p3v_cdiv(nk, S) + 0.2f * S * M * N * 4e-6f;
      if (c < best) best = c, plan = {S, t.mb, t.nb};
    }
  }
  return best < 0.95f * (one + (epilogue == P3V_EPI_RESID_BF16 ? 6.f : 0.f)) ? plan : none;
}

extern "C" int64_t p3v_gemm_slices_ws_bytes(int M, int N, int K, int epilogue) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return (int64_t)gemm_slices_plan(M, N, K, epilogue).S * M * N * 4;
}

int p3v_gemm256_slices(const p3v_gemm_args_t* a, float* part, int S, int mb, int nb, hipStream_t s);   // p3v_gemm256.hip

extern "C" int p3v_gemm_slices(const p3v_gemm_args_t* a, const uint16_t* norm_w, float eps, uint16_t* normed, void* stream) {
  if (!a || !a->A || !a->W || !a->out || !a->resid || !norm_w != !normed) return P3V_ERR_ARG;
  if (a->M <= 0 || a->N <= 0 || a->K <= 0 || a->K % BK || a->N % 8 || a->ldo % 8 || a->ldo < a->N) return P3V_ERR_ARG;
  if (a->lda < a->K || a->ldw < a->K || a->lda % 8 || a->ldw % 8) return P3V_ERR_ARG;
  if (((uintptr_t)a->A | (uintptr_t)a->W | (uintptr_t)a->out | (uintptr_t)a->resid | (uintptr_t)a->bias | (uintptr_t)a->col_scale | (uintptr_t)norm_w | (uintptr_t)normed | (uintptr_t)a->ws) & 15)
    return P3V_ERR_ARG;
  const bool scale = a->epilogue == P3V_EPI_SCALE_RESID_F32;
  if (scale != (a->col_scale != nullptr)) return P3V_ERR_ARG;
  if (a->bias && a->epilogue != P3V_EPI_BIAS_RESID_F32) return P3V_ERR_ARG;
  if (norm_w && (a->epilogue != P3V_EPI_RESID_BF16 || a->N > 6 * 64 * 8)) return P3V_ERR_UNSUPPORTED;
  const SlicePlan p = gemm_slices_plan(a->M, a->N, a->K, a->epilogue);
  if (!p.S || !a->ws || a->ws_bytes < (int64_t)p.S * a->M * a->N * 4) return P3V_ERR_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  float* part = (float*)a->ws;
  if (const int rc = p3v_gemm256_slices(a, part, p.S, p.mb, p.nb, s); rc != P3V_OK) return rc;
  if (!norm_w) return p3v_splitk_reduce(part, a, p.S, s);
  hipLaunchKernelGGL(k_splitk_reduce_norm, dim3(a->M), dim3(384), 0, s, part, (bf16_t*)a->out, (const bf16_t*)a->resid,
                     (const u32x4_t*)norm_w, (u32x4_t*)normed, a->M, a->N, a->ldo, p.S, 1.0f / (float)a->N, eps);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}

extern "C" int p3v_gemm(const p3v_gemm_args_t* a, void* stream) {
  if (!a || !a->A || !a->W || !a->out) return P3V_ERR_ARG;
  if (a->M < 0 || a->N <= 0 || a->K <= 0 || a->K % BK || a->N % 8 || a->ldo % 8) return P3V_ERR_ARG;
  if (a->lda < a->K || a->ldw < a->K || a->lda % 8 || a->ldw % 8) return P3V_ERR_ARG;
  if (((uintptr_t)a->A | (uintptr_t)a->W | (uintptr_t)a->out | (uintptr_t)a->resid | (uintptr_t)a->bias | (uintptr_t)a->pos) & 15)
    return P3V_ERR_ARG;
  if ((a->epilogue == P3V_EPI_BIAS_RESID_F32 || a->epilogue == P3V_EPI_RESID_BF16) && !a->resid) return P3V_ERR_ARG;
  if (a->epilogue == P3V_EPI_PATCH && (!a->pos || a->patches_per_img <= 0)) return P3V_ERR_ARG;
  if (a->epilogue < 0 || a->epilogue > P3V_EPI_GELU_MUL) return P3V_ERR_ARG;
  if (a->epilogue == P3V_EPI_SCALE_RESID_F32 && (!a->resid || !a->col_scale || ((uintptr_t)a->col_scale & 15) || a->bias)) return P3V_ERR_ARG;
  if (a->M == 0) return P3V_OK;
  {                                                            // operands are addressed with 32-bit byte offsets (buffer loads)
    const size_t w_rows = (size_t)a->N * (P3V_GATED(a->epilogue) ? 2 : 1);
    if ((size_t)a->M * a->lda * 2 >= (1ull << 32) || w_rows * a->ldw * 2 >= (1ull << 32)) return P3V_ERR_UNSUPPORTED;
  }
  hipStream_t s = (hipStream_t)stream;
  if (const int t = p3v_tuning().gemm_tile; t > 0) return p3v_gemm256_try(a, t / 10, t % 10, s);
  if (!a->bias) {                                              // 17 .. 256 rows: the weight-streaming kernel (p3v_gemm_skinny.hip)
    const int rc = p3v_gemm_skinny_try(a, s);
    if (rc != P3V_ERR_UNSUPPORTED) return rc;
  }
  {
    int rc = gemm_splitk(a, s);
    if (rc == P3V_ERR_UNSUPPORTED) rc = p3v_gemm_skinny_tall(a, s);
    if (rc != P3V_ERR_UNSUPPORTED) return rc;
  }
  const bool big_tiles = !p3v_tuning().gemm_128;
  const int rows_big = big_tiles ? gemm_big_rows(a) : 0;
  if (const int t = gemm_tile_choice(a, rows_big)) {
    const int rc = p3v_gemm256_try(a, t / 10, t % 10, s);
    if (rc != P3V_ERR_UNSUPPORTED) return rc;
  }
  if (rows_big > 0) {
    p3v_gemm_args_t top = *a;
    top.M = rows_big;
    const int rc = p3v_gemm256_try(&top, 8, 4, s);
    if (rc == P3V_OK && rows_big < a->M) {
      const bool f32_out = a->epilogue == P3V_EPI_BIAS_RESID_F32 || a->epilogue == P3V_EPI_F32 || a->epilogue == P3V_EPI_SCALE_RESID_F32;
      const size_t out_row = (size_t)a->ldo * (f32_out ? 4 : 2);
      p3v_gemm_args_t rest = *a;
      rest.M = a->M - rows_big;
      rest.A = a->A + (size_t)rows_big * a->lda;
      rest.out = (char*)a->out + rows_big * out_row;
      if (a->resid) rest.resid = (const char*)a->resid + rows_big * out_row;
      return gemm128(&rest, s);
    }
    if (rc != P3V_ERR_UNSUPPORTED) return rc;
  }
  return gemm128(a, s);
}

static int gemm128(const p3v_gemm_args_t* a, hipStream_t s) {
  const GemmP p = {a->A, a->W, a->out, a->epilogue == P3V_EPI_SCALE_RESID_F32 ? a->col_scale : a->bias, a->resid, a->pos,
                   a->M, a->N, a->K, a->lda, a->ldw, a->ldo, a->patches_per_img, 0, {}};
  switch (a->epilogue) {
    case P3V_EPI_NONE: return launch_gemm<P3V_EPI_NONE>(p, s);
    case P3V_EPI_BIAS: return launch_gemm<P3V_EPI_BIAS>(p, s);
    case P3V_EPI_BIAS_QGELU: return launch_gemm<P3V_EPI_BIAS_QGELU>(p, s);
    case P3V_EPI_BIAS_GELU: return launch_gemm<P3V_EPI_BIAS_GELU>(p, s);
    case P3V_EPI_BIAS_RESID_F32: return launch_gemm<P3V_EPI_BIAS_RESID_F32>(p, s);
    case P3V_EPI_RESID_BF16: return launch_gemm<P3V_EPI_RESID_BF16>(p, s);
    case P3V_EPI_SILU_MUL: return launch_gemm<P3V_EPI_SILU_MUL>(p, s);
    case P3V_EPI_GELU_MUL: return launch_gemm<P3V_EPI_GELU_MUL>(p, s);
    case P3V_EPI_PATCH: return launch_gemm<P3V_EPI_PATCH>(p, s);
    case P3V_EPI_F32: return launch_gemm<P3V_EPI_F32>(p, s);
    case P3V_EPI_SCALE_RESID_F32: return launch_gemm<P3V_EPI_SCALE_RESID_F32>(p, s);
    default: return P3V_ERR_ARG;
  }
}

// ---- the qkv projection with the head split, the rotation and the KV append in its epilogue (p3v_gemm_qkv.h)
int p3v_gemm_skinny_qkv(const p3v_gemm_args_t* a, const QkvP& q, bool tall, hipStream_t s);   // p3v_gemm_skinny.hip

int p3v_gemm_skinny_qkv_merge(const p3v_gemm_args_t* a, const QkvP& q, void* ws, int64_t ws_bytes, hipStream_t s);   // p3v_gemm_skinny.hip
int p3v_qkv_flat_tiles(const QkvP& q, int M, int mb);                                        // p3v_gemm_pc.hip
int p3v_gemm256_flat_qkv(const p3v_gemm_args_t* a, const QkvP& q, int mb, hipStream_t s);      // p3v_gemm256.hip

// The qkv projection in one launch on tiles of 32 mb rows x 256 columns (p3v_gemm_pc.hip up to 160 rows, p3v_gemm256.hip from 192) or, mb = 1, of 128 x 128
// (k_gemm): mb, or 0.
// Below 1024 rows the alternative is p3v_gemm and the split as a launch of its own: the same tile saves that launch for 4 us of epilogue (900 x
// 9216 x 3072 59.0 -> 55.2 us, 768 55.9 -> 52.7), as long as one round of the chip takes the tiles, of which there are more (a V tile's rows are
// dimensions, its columns 256 tokens).  From 1024 rows on every tile is priced as in gemm_tile_choice, 128 x 128 ones (two a CU: whole rounds of 512, and
// the last one by whether it holds more than 256) for K <= 1024 alone, where their short prologue counts; fitted to 219 sizes: 21 heights, 1024 .. 16384 rows,
// of nine projections with K = 256 .. 3072, and 2 .. 17 image crops (profiles/gemm_qkv_tile_sweep.txt).  The tile it names is 0.7 % slower than the fastest on
// average, 15 % at most (K = 256); each projection left out of the fit: 1.0 %, 15 %.  At the decoder's own widths, 9216 x 3072, it is the fastest at each
// of the 42 sizes of one and four prompts.  Measured, us, a fit without short K -> this: 1536 x 4608 x 512 16.7 -> 14.8, 8192 60 -> 56; 2048 x 9216 x 3072 104 ->
// 103, 4096 205 -> 198; 11 crops 58.9 -> 56.6.
static int qkv_tile_plan(const p3v_gemm_args_t* a, const QkvP& q) {
  const int pin = p3v_tuning().gemm_qkv_flat;
  if (!pin || a->M <= 256 || (q.nh * q.hd) % 256 || (q.nkv * q.hd) % 256) return 0;
  if (pin > 0) return pin;
  if (p3v_tuning().gemm_128) return 0;
  if (a->M < 1024) {
    p3v_gemm_args_t plain = *a;
    int mb = 0, nb = 0;
    if (splitk_slices(a->M, a->N, a->K, a->epilogue) > 1 || !gemm_tile_plan(&plain, 0, &mb, &nb) || nb != 4 || (mb != 4 && mb != 5)) return 0;
    return p3v_qkv_flat_tiles(q, a->M, mb) <= 256 ? mb : 0;
  }
  static const struct { int mb; float once, f, c, fill, out; } tiles[] = {{2, 4.32f, 3.74f, 0.182f, 0.389f, 0.f},    {3, 4.68f, 4.67f, 0.318f, 0.398f, 0.f},
                                                                          {4, 5.11f, 4.64f, 0.507f, 0.312f, 1.77f},  {5, 5.38f, 6.17f, 0.584f, 0.358f, 1.52f},
                                                                          {6, 4.1f, 9.78f, 0.685f, 0.372f, 1.88f},   {7, 4.67f, 10.44f, 0.802f, 0.38f, 2.24f},
                                                                          {8, 4.96f, 11.85f, 0.879f, 0.446f, 2.45f}};
  const float kt = (float)(a->K / BK);
  float best = 1e30f;
  int mb = 0;
  if (a->K <= 1024) {
    const long n = (long)(a->N / BN) * p3v_cdiv(a->M, BM), rest = n % 512;
    best = 4.63f + n / 512 * (2.09f + 0.516f * kt) + (rest > 0) * (1.58f + 0.423f * kt) + (rest > 256) * (1.03f + 0.036f * kt) + n / 512.f * (3.72f + 0.272f * kt);
    mb = 1;
  }
  for (const auto& t : tiles) {
    const int n = p3v_qkv_flat_tiles(q, a->M, t.mb);
    const float c = t.once + p3v_cdiv(n, 256) * (t.f + t.c * kt) + n / 256.f * (t.fill * kt + t.out);
    if (c < best) best = c, mb = t.mb;
  }
  return mb;
}

extern "C" int p3v_gemm_qkv_tile(int M, int n_q, int n_kv, int K) {
  if (M <= 0 || n_q <= 0 || n_kv <= 0 || K <= 0 || n_q % 32 || n_kv % 32 || K % BK) return 0;
  p3v_gemm_args_t a = {};
  QkvP q = {};
  a.M = M, a.N = n_q + 2 * n_kv, a.K = K, a.epilogue = P3V_EPI_NONE;
  q.nh = n_q / 32, q.nkv = n_kv / 32, q.hd = 32;
  return qkv_tile_plan(&a, q);
}

static int gemm_qkv(const p3v_gemm_args_t* a, const p3v_qkv_split_t* sp, void* merge_ws, int64_t merge_bytes, bool tall, void* stream) {
  if (!a || !sp || !a->A || !a->W || !sp->q_out || !sp->k_dst || !sp->v_dst || (!sp->cos_t) != (!sp->sin_t)) return P3V_ERR_ARG;
  if (a->epilogue != P3V_EPI_NONE && a->epilogue != P3V_EPI_BIAS) return P3V_ERR_ARG;
  if (a->epilogue == P3V_EPI_BIAS && !a->bias) return P3V_ERR_ARG;
  const int nh = sp->n_heads, nkv = sp->n_kv, hd = sp->hd, half = hd / 2;
  if (sp->B <= 0 || sp->L <= 0 || nh <= 0 || nkv <= 0 || hd <= 0 || sp->tab_div <= 0 || !(sp->q_scale > 0.f)) return P3V_ERR_ARG;
  if (a->M != sp->B * sp->L || a->N != (nh + 2 * nkv) * hd || a->K % BK || a->lda < a->K || a->ldw < a->K || a->lda % 8 || a->ldw % 8) return P3V_ERR_ARG;
  if (((uintptr_t)a->A | (uintptr_t)a->W | (uintptr_t)a->bias | (uintptr_t)sp->q_out | (uintptr_t)sp->k_dst | (uintptr_t)sp->v_dst |
       (uintptr_t)sp->cos_t | (uintptr_t)sp->sin_t) & 15)
    return P3V_ERR_ARG;
  // what the fused epilogue needs (anything else: P3V_ERR_UNSUPPORTED, the caller runs p3v_gemm + p3v_rope_kv_append):
  // prompt-sized M; rotation pairs in blocks of 16 inside a head; whole 128-column tiles per region; an 8-aligned append offset
  const int dpos0 = sp->dst_off_is_past ? sp->past : 0;
  // (batch rows of any length -- the V^T runs are then stored at whatever offset they fall on, qkv_epilogue_vt)
  if (hd % 32 || half % 16 || dpos0 % 8 || sp->dst_t % 8 || !qkv_rows_ok(sp->B, sp->L) || p3v_tuning().gemm_no_qkv_fuse) return P3V_ERR_UNSUPPORTED;
  if ((size_t)a->M * a->lda * 2 >= (1ull << 32) || (size_t)a->N * a->ldw * 2 >= (1ull << 32)) return P3V_ERR_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  QkvP q = {sp->cos_t, sp->sin_t, sp->q_out, sp->k_dst, sp->v_dst, sp->L, nh, nkv, hd, sp->past, dpos0, sp->dst_t, sp->tab_t, sp->tab_div,
            sp->q_scale};
  if (merge_ws) return p3v_gemm_skinny_qkv_merge(a, q, merge_ws, merge_bytes, s);
  if (tall) return p3v_gemm_skinny_qkv(a, q, true, s);
  const int mb = qkv_tile_plan(a, q);
  if (mb > 1) return p3v_gemm256_flat_qkv(a, q, mb, s);
  if (!mb && a->M < 1024) return p3v_gemm_skinny_qkv(a, q, false, s);  // 17 .. 256 rows: the weight-streaming kernel (or "unsupported")
  if ((nh * hd) % BN || (nkv * hd) % BN || p3v_tuning().gemm_128) return P3V_ERR_UNSUPPORTED;
  const GemmP p = {a->A, a->W, nullptr, a->bias, nullptr, nullptr, a->M, a->N, a->K, a->lda, a->ldw, 0, 0, 0, q};
  return launch_gemm<P3V_EPI_QKV>(p, s);
}
extern "C" int p3v_gemm_qkv(const p3v_gemm_args_t* a, const p3v_qkv_split_t* sp, void* stream) { return gemm_qkv(a, sp, nullptr, 0, false, stream); }
extern "C" int p3v_gemm_qkv_one_pass(const p3v_gemm_args_t* a, const p3v_qkv_split_t* sp, void* stream) { return gemm_qkv(a, sp, nullptr, 0, true, stream); }
extern "C" int p3v_gemm_qkv_merge(const p3v_gemm_args_t* a, const p3v_qkv_split_t* sp, void* ws, int64_t ws_bytes, void* stream) {
  return ws ? gemm_qkv(a, sp, ws, ws_bytes, false, stream) : P3V_ERR_ARG;
}
