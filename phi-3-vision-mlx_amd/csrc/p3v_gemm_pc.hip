// Flat-tile variant of the dense projection for prefill-sized problems (p3v_gemm's tile plan decides): 128 x 256, 160 x 256 or 128 x 192
// outputs x 64 of K, for the shapes whose 256 x 256 tiles leave a round of the chip half empty.
//   waves    12: eight CONSUMERS as 2(M) x 4(N), each 64 .. 80 x 48 .. 64 outputs, and four PRODUCERS (one per SIMD) that only issue the
//            LDS-DMA and wait for it.  A K-tile of a flat tile has half the MFMAs of a 256 x 256 one but three quarters of its bytes: with
//            the MFMA waves issuing the DMA themselves (p3v_gemm256.hip's form) a 128 x 256 K-tile takes 1.14 us with two LDS buffers and
//            0.85 with three, most of it DMA issue in front of the MFMAs; here 0.81 (0.65 with 192 workgroups).
//   staging  S = 3 (128 x 192: 4) LDS buffers; one barrier per K-tile, in the middle of it: the fragments of one 32-wide half are
//            multiplied while those of the other are read, so a K-tile's buffer is free, and refilled, half a K-tile before its last MFMA.
//   bound    the LDS-DMA: 88 - 98 KB/us and CU in pieces of 8 rows x 128 B (profiles/lds_dma_probe.txt), i.e. 0.5 us for the 48 KB of a 128 x 256 K-tile against 0.45 of
//            MFMAs; larger tiles do not fit the 168 registers that twelve waves leave each other.
// 2531 x 3072 x 8192 (+ residual) 117 -> 105 us (1.21 PFLOP/s), 9809 x 1024 x 4096 (+ fp32 residual) 95 -> 73, 2048 x 9472 x 3072 114 -> 97.
// Same K order and epilogue as the other tiles: bit-identical results.
// P3V_EPI_QKV: split, rotation and KV append in the epilogue, tiles of 64 and 96 rows too (qkv_tile_plan, p3v_gemm.hip, has the rule and the
// times; a K-tile of 64 x 256 takes as long as one of 128 x 256, waiting for its weights, but a short K gets through the chip sooner).
// P3V_EPI_PART: the tiles of one slice of K after the other, fp32 partials (p3v_gemm_slices, p3v_gemm.hip, which has the rule and the times).
// (Tried and left out: touching the lines of later K-tiles ahead of the DMA, one dword per line -- 64 lines cost the address path as
//  much as four pieces: 105 -> 137 us; 4 consumers of twice the size without producers: 121 us.)
#include "p3v_gemm256_epi.h"

struct TilePc {                        // where the requests of an output tile's K-tiles come from
  int a_off[8], b_off[8]; __amdgpu_buffer_rsrc_t rs_a, rs_b;
};
struct PlacePc { int m0, n0, z, swapped, is_k, row0; };           // z: slice of K; the others P3V_EPI_QKV: V tile (operand roles swapped) / K region / first W row of the region

#define GPC_BUF(mb, nb) ((32 * (mb) + 64 * (nb)) * TK * 2)
#define GPC_STAGES(mb, nb) (160 * 1024 / GPC_BUF(mb, nb) < 4 ? 160 * 1024 / GPC_BUF(mb, nb) : 4)

// MB, NB: 16-row / 16-column blocks of a consumer wave (2 x 4 waves: a tile of 32 MB rows x 64 NB columns)
template <int EPI, int MB, int NB>
__global__ void __launch_bounds__(768, 1) k_gemm_pc(Gemm256P p) {
  constexpr bool SILU = P3V_GATED(EPI);
  static_assert(NB == 4 || (NB == 3 && !SILU), "");
  constexpr int TM = 32 * MB, TN = 64 * NB, A_BYTES = TM * TK * 2, BUF_BYTES = A_BYTES + TN * TK * 2;
  constexpr int S = GPC_STAGES(MB, NB), PER = MB + 2 * NB;        // LDS buffers; requests of a producer wave per K-tile
  static_assert(S >= 3 && (S - 1) * PER < 64, "");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: LDS-DMA bases stay in SGPRs
  constexpr int n_out_tile = SILU ? TN / 2 : TN;
  constexpr bool PART = EPI == P3V_EPI_PART, QKV = EPI == P3V_EPI_QKV;
  static_assert(!QKV || NB == 4, "both halves of 32 rotation pairs in a wave");
  // (QKV: column tiles 0 .. nq - 1 are Q, the others K; behind them the V tiles, TM rows of W_v by TN tokens -- p3v_gemm_qkv.h)
  const int nq = QKV ? p.q.nh * p.q.hd / TN : 0, v_rows = QKV ? p.q.nkv * p.q.hd : 0, vx = QKV ? (p.M + TN - 1) / TN : 0;
  const int gx = QKV ? nq + v_rows / TN : (p.N + n_out_tile - 1) / n_out_tile, gy = (p.M + TM - 1) / TM;
  const int nwg = QKV ? gx * gy + vx * ((v_rows + TM - 1) / TM) : PART ? gx * gy * p.slices : gx * gy;
  const int nk = p.K / TK;

  // ---- PERSISTENT over output tiles: workgroup b takes tiles b, b + G, b + 2G, ... (G = gridDim.x, a multiple of 8, so a
  // workgroup's tiles keep its XCD in the XCD-aware order below), one stream of K-tiles across all of them.
  // PART: the slices one after the other, so an XCD keeps to one slice of K or two: A and W pass each L2 once, whatever the tile order.
  auto place = [&](int wid) {
    const int q = nwg >> 3, r = nwg & 7, xcd = wid & 7, loc = wid >> 3;
    int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + loc;
    PlacePc t = {0, 0, 0, 0, 0, 0};
    if (PART) t.z = id / (gx * gy), id -= t.z * (gx * gy);
    if (QKV && id >= gx * gy) {
      id -= gx * gy;
      t.swapped = 1, t.row0 = (p.q.nh + p.q.nkv) * p.q.hd, t.m0 = id % vx * TN, t.n0 = id / vx * TM;
      return t;
    }
    constexpr int BAND = 4;
    const int band = id / (BAND * gx), in_band = id % (BAND * gx);
    const int rows = min(BAND, gy - band * BAND);
    int x = in_band / rows;
    t.m0 = (band * BAND + in_band % rows) * TM;
    if (QKV && x >= nq) t.is_k = 1, t.row0 = p.q.nh * p.q.hd, x -= nq;
    t.n0 = x * n_out_tile;                                        // (QKV: first column INSIDE the region)
    return t;
  };
  auto k_begin = [&](int z) { return PART ? z * nk / p.slices : 0; };
  auto k_end = [&](int z) { return PART ? (z + 1) * nk / p.slices : nk; };
  if ((int)blockIdx.x >= nwg) return;
  int total = 0;                                                  // K-tiles of this workgroup
  if (PART) {
    for (int wid = blockIdx.x; wid < nwg; wid += gridDim.x) {
      const int z = place(wid).z;
      total += k_end(z) - k_begin(z);
    }
  } else {
    total = ((nwg - 1 - (int)blockIdx.x) / (int)gridDim.x + 1) * nk;
  }

  if (wave >= 8) {
    // ---- PRODUCERS.  A request = 8 tile rows x 128 B (1 KiB) by LDS-DMA; the 16-byte chunks of a row are swizzled on the source side.
    // Buffer addressing (SGPR descriptor + 32-bit per-lane byte offset + SGPR K offset): no vector ALU work at all.
    const int pw = wave - 8, srow = pw * 8 + (lane >> 3), sw = ((lane & 7) ^ (lane >> 3)) * 8;
    int dk = 0, dk_end = nk;                                      // the K-tiles still to be requested for the tile in hand
    TilePc dt;   // (declared outside the template: a builtin called with a member of a DEPENDENT type is only checked at
                 //  instantiation, fails there in the HOST pass -- no such builtin -- and hipcc silently drops the host stub)
    auto aim = [&](int wid) {
      const PlacePc t = place(wid);
      const int m0 = t.m0, n0 = t.n0;
      dk = k_begin(t.z), dk_end = k_end(t.z);
      const bool v = QKV && t.swapped;                            // V tile: W rows fill the A side, tokens the B side
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int rr = q * 32 + srow;
        int br = n0 + rr;
        if (SILU)                                     // a group of 64 tile columns = 32 gate rows + the 32 up rows of the same outputs
          br = min(n0 + (rr >> 6) * 32 + ((rr >> 4) & 1) * 16 + (rr & 15), p.N - 1) + ((rr & 63) >> 5) * p.N;
        else if (QKV)                                 // pair order (both halves of a rotation pair in one lane)
          br = v ? min(m0 + rr, p.M - 1) : qkv_pair_row(p.q, t.row0, n0 >> 1, rr);
        else
          br = min(br, p.N - 1);
        const int ar = v ? min(n0 + rr, v_rows - 1) - n0 : min(m0 + rr, p.M - 1) - m0;
        dt.a_off[q] = (ar * (v ? p.ldw : p.lda) + sw) * 2;
        dt.b_off[q] = (int)(((unsigned)br * (unsigned)(v ? p.lda : p.ldw) + (unsigned)sw) * 2u);   // < 2^32: checked by the launcher
      }
      const bf16_t* pa = v ? p.W + (size_t)(t.row0 + n0) * p.ldw : p.A + (size_t)m0 * p.lda;
      const bf16_t* pb = v ? p.A : p.W;
      dt.rs_a = __builtin_amdgcn_make_buffer_rsrc((void*)pa, 0, 0xffffffff, 0x00020000);
      dt.rs_b = __builtin_amdgcn_make_buffer_rsrc((void*)pb, 0, 0xffffffff, 0x00020000);
    };
    int dwid = blockIdx.x, slot = 0;                              // the tile in hand, and the next K-tile's buffer
    aim(dwid);
    auto request = [&]() {
      unsigned char* base = smem + slot * (int)BUF_BYTES + pw * 1024;
      const int na = MB, nb = 2 * NB, a_bytes = A_BYTES;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (q < na) {
          lptr_t dst = (lptr_t)(base + q * 4096);
          const int vo = dt.a_off[q];
          __builtin_amdgcn_raw_ptr_buffer_load_lds(dt.rs_a, dst, 16, vo, dk * (TK * 2), 0, 0);
        }
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (q < nb) {
          lptr_t dst = (lptr_t)(base + a_bytes + q * 4096);
          const int vo = dt.b_off[q];
          __builtin_amdgcn_raw_ptr_buffer_load_lds(dt.rs_b, dst, 16, vo, dk * (TK * 2), 0, 0);
        }
      }
      slot = slot == S - 1 ? 0 : slot + 1;
      if (++dk == dk_end) {
        dwid += gridDim.x;
        if (dwid < nwg) aim(dwid);
      }
    };
    for (int g = 0; g < min(S, total); ++g) request();
    for (int g = 0; g < total; ++g) {
      // K-tile g has landed when only the younger ones' requests are out: S - 1 of them at first, then S - 2, fewer at the end
      const int young = min(g == 0 ? S - 1 : S - 2, total - 1 - g);
      if (young >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S > 3 ? 3 : 0) * PER) : "memory");
      else if (young == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PER) : "memory");
      else if (young == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();                               // K-tile g is there; K-tile g - 1 is in the consumers' registers
      if (g > 0 && g - 1 + S < total) request();
    }
    return;
  }

  // ---- CONSUMERS: the fragments of one 32-wide half of a K-tile are multiplied while those of the next are fetched
  const int wr = wave >> 2, wc = wave & 3;
  const int frow = lane & 15, fchunk = lane >> 4;
  const int fo0 = frow * 128 + ((fchunk ^ (frow & 7)) << 4), fo1 = frow * 128 + (((4 + fchunk) ^ (frow & 7)) << 4);
  f32x4_t acc[MB][NB];
  bf16x8_t fa[2][MB], fb[2][NB];                                  // the fragments of the two halves
  auto fetch = [&](int n, int kk, int buf) {                      // fragment n: the columns' first, then the rows' (the MFMAs walk row by row)
    const unsigned char* t = smem + buf * BUF_BYTES + (kk ? fo1 : fo0);
    if (n < NB) fb[kk][n] = *(const bf16x8_t*)(t + A_BYTES + (wc * NB + n) * 2048);
    else fa[kk][n - NB] = *(const bf16x8_t*)(t + (wr * MB + n - NB) * 2048);
  };
  auto half = [&](int kk, bool fetches, int fbuf) {               // all MFMAs of one half, between them (early) the fetches of the other
    constexpr int C = (MB * NB + 3) / 4;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (2 * c < C && (kk == 0 || fetches)) {
#pragma unroll
        for (int n = 0; n < MB + NB; ++n)
          if (n >= 2 * (MB + NB) * c / C && n < 2 * (MB + NB) * (c + 1) / C) fetch(n, kk ^ 1, fbuf);
      }
#pragma unroll
      for (int m = 4 * c; m < 4 * c + 4 && m < MB * NB; ++m)
        acc[m / NB][m % NB] =                                    // (W fragment first: the block comes out TRANSPOSED, see the epilogue)
            __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[kk][m % NB], fa[kk][m / NB], acc[m / NB][m % NB], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int slot = 0;                                                   // LDS buffer of the K-tile in hand
  __builtin_amdgcn_s_barrier();
  for (int wid = blockIdx.x; wid < nwg; wid += gridDim.x) {
    const PlacePc t = place(wid);
    const int m0 = t.m0, n0 = t.n0, nkt = k_end(t.z) - k_begin(t.z);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < MB + NB; ++n) fetch(n, 0, slot);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (int kt = 0; kt < nkt; ++kt) {
      const int nslot = slot == S - 1 ? 0 : slot + 1;
      const bool last = kt + 1 == nkt;                             // (nothing is fetched behind a tile's last K-tile: the epilogue needs the registers)
      half(0, true, slot);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // the K-tile in hand is in registers: its buffer is given back
      if (!last || wid + (int)gridDim.x < nwg) __builtin_amdgcn_s_barrier();
      half(1, !last, nslot);
      slot = nslot;
    }
    int lane_e = lane;                                            // (opaque: what the epilogue derives from it is not to be held through the K loop)
    asm volatile("" : "+v"(lane_e));
    if constexpr (PART) {
      Gemm256P part = p;
      part.out = (float*)p.out + (size_t)t.z * p.M * p.ldo;
      gemm256_epilogue<P3V_EPI_F32, MB, NB>(part, acc, m0 + wr * MB * 16, n0 + wc * (n_out_tile / 4), lane_e);
    } else if constexpr (QKV) {
      if (!t.swapped) qkv_epilogue_rot<MB, 2>(p.q, acc, p.bias, t.is_k, t.row0, (n0 >> 1) + wc * 32, m0 + wr * MB * 16, p.M, lane_e);
      else qkv_epilogue_vt<MB>(p.q, acc, p.bias ? p.bias + t.row0 : nullptr, n0 + wr * MB * 16, m0 + wc * 64, p.M, lane_e, v_rows);
    } else {
      gemm256_epilogue<EPI, MB, NB>(p, acc, m0 + wr * MB * 16, n0 + wc * (n_out_tile / 4), lane_e);  // straight from the accumulators: p3v_gemm256_epi.h
    }
  }
}

int p3v_gemm256_cus();                                             // p3v_gemm256.hip

int p3v_qkv_flat_tiles(const QkvP& q, int M, int mb);

template <int EPI, int MB, int NB>
static int launch_pc_v(const Gemm256P& p, hipStream_t s) {
  constexpr int LDS = GPC_STAGES(MB, NB) * GPC_BUF(MB, NB);
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm_pc<EPI, MB, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return P3V_ERR_HIP;
    attr_set = true;
  }
  const int n_cu = p3v_gemm256_cus();
  if (!n_cu) return P3V_ERR_HIP;
  int tiles = p3v_cdiv(p.N, P3V_GATED(EPI) ? 32 * NB : 64 * NB) * p3v_cdiv(p.M, 32 * MB) * (EPI == P3V_EPI_PART ? p.slices : 1);
  if (EPI == P3V_EPI_QKV) tiles = p3v_qkv_flat_tiles(p.q, p.M, MB);
  hipLaunchKernelGGL((k_gemm_pc<EPI, MB, NB>), dim3(min(tiles, n_cu)), dim3(768), LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}

// output tiles of the qkv projection on tiles of 32 mb rows x 256 columns
int p3v_qkv_flat_tiles(const QkvP& q, int M, int mb) {
  return (q.nh + q.nkv) * q.hd / 256 * p3v_cdiv(M, 32 * mb) + p3v_cdiv(q.nkv * q.hd, 32 * mb) * p3v_cdiv(M, 256);
}

template <int EPI>
static int launch_pc(const Gemm256P& p, int mb, int nb, hipStream_t s) {
  if constexpr (!P3V_GATED(EPI) && EPI != P3V_EPI_QKV)
    if (nb == 3) return launch_pc_v<EPI, 4, 3>(p, s);
  if constexpr (EPI == P3V_EPI_QKV) {
    if (mb == 2) return launch_pc_v<EPI, 2, 4>(p, s);
    if (mb == 3) return launch_pc_v<EPI, 3, 4>(p, s);
  }
  return mb == 4 ? launch_pc_v<EPI, 4, 4>(p, s) : launch_pc_v<EPI, 5, 4>(p, s);
}

int p3v_gemm_pc(const Gemm256P& p, int epi, int mb, int nb, hipStream_t s) {
  switch (epi) {
    case P3V_EPI_NONE: return launch_pc<P3V_EPI_NONE>(p, mb, nb, s);
    case P3V_EPI_BIAS: return launch_pc<P3V_EPI_BIAS>(p, mb, nb, s);
    case P3V_EPI_BIAS_QGELU: return launch_pc<P3V_EPI_BIAS_QGELU>(p, mb, nb, s);
    case P3V_EPI_BIAS_GELU: return launch_pc<P3V_EPI_BIAS_GELU>(p, mb, nb, s);
    case P3V_EPI_BIAS_RESID_F32: return launch_pc<P3V_EPI_BIAS_RESID_F32>(p, mb, nb, s);
    case P3V_EPI_RESID_BF16: return launch_pc<P3V_EPI_RESID_BF16>(p, mb, nb, s);
    case P3V_EPI_SILU_MUL: return launch_pc<P3V_EPI_SILU_MUL>(p, mb, nb, s);
    case P3V_EPI_GELU_MUL: return launch_pc<P3V_EPI_GELU_MUL>(p, mb, nb, s);
    case P3V_EPI_F32: return launch_pc<P3V_EPI_F32>(p, mb, nb, s);
    case P3V_EPI_SCALE_RESID_F32: return launch_pc<P3V_EPI_SCALE_RESID_F32>(p, mb, nb, s);
    case P3V_EPI_QKV: return launch_pc<P3V_EPI_QKV>(p, mb, nb, s);
    case P3V_EPI_PART: return launch_pc<P3V_EPI_PART>(p, mb, nb, s);
    default: return P3V_ERR_UNSUPPORTED;
  }
}
