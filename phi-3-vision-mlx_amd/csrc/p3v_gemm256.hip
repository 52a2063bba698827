// Large-tile variant of the dense projection for prefill-sized problems (K % 64 == 0, columns in whole tiles; p3v_gemm decides which rows of a
// problem it gets and in which of its tiles):
//   256(M) x 256(N) x 64(K) tile (template: 224 or 192 rows, or 192 columns, for problems whose rounds they fill better), 256 threads = 4 waves as
//   2(M) x 2(N), one per SIMD, each 128 x 128 = 8 x 8 v_mfma_f32_16x16x32_bf16 blocks: 256 accumulation registers, 4 MFMAs per LDS fragment read.
//   Why     what bounds it is power and the LDS: with 8 waves of 128 x 64 (2.67 MFMAs a fragment) a K-tile's fragment reads and its LDS-DMA
//           together take all 2048 cycles of its MFMAs at 128 B a cycle; with 128 x 128 a wave reads a third less.  Matrix pipe busy of the CUs' cycles,
//           8 waves -> 4: 4096 x 4096 x 8192 0.73 -> 0.84, gate | up of 2531 rows 0.64 -> 0.76, at a lower clock for the same power (1.98 -> 1.84 GHz,
//           2.21 -> 2.06; profiles/gemm256_four_waves_pmc.txt).
//   Loop    half a K-tile (64 MFMAs) is multiplied while the other half's 16 fragments are read, one every two MFMAs; ONE barrier per K-tile, in
//           the first half, where this K-tile is in registers and the next one in LDS: the buffers change hands there, and the requests of K-tiles
//           to come go out one every six MFMAs from then on (LDS-DMA, 1 KiB each; W three K-tiles ahead, A two, or three where 160 KiB hold
//           them).  A wave has nobody to cover for it, so nothing in the loop waits for memory unless the request is late.  The order of reads,
//           the places of requests and a second barrier were tried both ways: no difference.  Without requests the loop is 20 % faster, without
//           fragment reads 6 %, from an L2-hot K-tile 9 % (power again).  W three and A two K-tiles ahead against the other way round: 5 - 10 %
//           with weights from memory (768 x 9216 x 3072 65 -> 60 us), nothing from the last-level cache.
//   Same XOR-swizzled LDS image and the same epilogues as p3v_gemm.hip; stored straight from the accumulators.
// Measured, us, 8 waves -> this: 4096^3 110 -> 98 (1.40 PFLOP/s), 8192^3 777 -> 710 (1.55), 16384 x 3072 x 8192 604 -> 554; without a pause and with weights from
// memory 2048 x 16384 x 3072 (gate | up) 179 -> 149, 9809 808 -> 710, 2531 x 10496 x 3072 157 -> 127 (with the tiles' choice); inside a prompt of 2531
// tokens gate_up 217 -> 198, qkv 147 -> 133.
#include <stdlib.h>

#include <type_traits>

#include "p3v_gemm256_epi.h"

struct Aim256 { int a_off[8], b_off[8]; __amdgpu_buffer_rsrc_t rs_a, rs_b; };   // where the requests of an output tile's K-tiles come from
// (declared outside the template: a builtin called with a member of a DEPENDENT type is only checked at instantiation, fails there in the
//  HOST pass -- no such builtin -- and hipcc silently drops the host stub)
struct Place256 { int m0, n0, swapped, is_k, row0; };             // P3V_EPI_QKV: V tile (operand roles swapped) / K region / first W row of the region

#define G256_BUF(mb, nb) (32 * ((mb) + (nb)) * TK * 2)            // bytes of a K-tile
#define G256_SA(mb, nb) (3 * G256_BUF(mb, nb) <= 160 * 1024 ? 3 : 2)   // LDS buffers of A's half (of W's: 3)

// MB, NB: 16-row / 16-column blocks of a wave (2 x 2 waves: a tile of 32 MB rows x 32 NB columns)
template <int EPI, int MB, int NB>
__global__ void __launch_bounds__(256, 1) k_gemm256(Gemm256P p) {
  constexpr bool SILU = P3V_GATED(EPI), QKV = EPI == P3V_EPI_QKV;
  static_assert(MB >= 6 && MB <= 8 && (NB == 8 || (NB == 6 && !SILU && !QKV)), "");
  constexpr int TM = 32 * MB, TN = 32 * NB, A_BYTES = TM * TK * 2, B_BYTES = TN * TK * 2;
  constexpr int SA = G256_SA(MB, NB), B0 = SA * A_BYTES;          // the LDS buffers: SA of A, three of W behind them
  constexpr int GB = NB == 8 ? 4 : 6, NG = NB / GB;               // a wave's column blocks in groups: 64 columns are the epilogues' unit
  constexpr int NM = MB * NB, NF = MB + NB;                       // MFMAs and fragments of half a K-tile; a wave's requests per K-tile
  constexpr int TURN = 2 * NF + 4 < NM - 1 ? 2 * NF + 4 : NM - 2, STEP = 3 * NM / (2 * NF);      // the first half's MFMA where buffers change hands; MFMAs per request
  static_assert(TURN >= 2 * NF - 1 && TURN < NM, "");
  constexpr int YOUNG = SA == 3 ? NF : NB;                        // requests younger than those of the next K-tile, at a turn
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: LDS-DMA bases stay in SGPRs
  const int wr = wave >> 1, wc = wave & 1;
  constexpr int n_out_tile = SILU ? TN / 2 : TN;
  // (QKV: column tiles 0 .. nq - 1 are Q, the others K; behind them the V tiles, TM rows of W_v by TN tokens -- p3v_gemm_qkv.h)
  const int nq = QKV ? p.q.nh * p.q.hd / TN : 0, v_rows = QKV ? p.q.nkv * p.q.hd : 0, vx = QKV ? (p.M + TN - 1) / TN : 0;
  const int gx = QKV ? nq + v_rows / TN : (p.N + n_out_tile - 1) / n_out_tile, gy = (p.M + TM - 1) / TM;
  const int nwg = QKV ? gx * gy + vx * ((v_rows + TM - 1) / TM) : gx * gy;
  const int nk = p.K / TK;

  // ---- PERSISTENT over output tiles: workgroup b takes tiles b, b + G, b + 2G, ... (G = gridDim.x, a multiple of 8, so a workgroup's tiles
  // keep its XCD in the XCD-aware order below), one stream of K-tiles across all of them.
  auto place = [&](int wid) {
    const int q = nwg >> 3, r = nwg & 7, xcd = wid & 7, loc = wid >> 3;
    int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + loc;
    Place256 t = {0, 0, 0, 0, 0};
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

  // What only a tile's end needs of the launch's parameters is read again there (a scalar load): held in registers through the K loop, it
  // would push the loop's own scalars out.
  auto again = [&]() {
    typedef const __attribute__((address_space(4))) unsigned char* cptr_t;
    cptr_t a = (cptr_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return (const void*)(a + __builtin_offsetof(Gemm256P, q));
  };

  // ---- REQUESTS.  One = 8 tile rows x 128 B (1 KiB) of LDS-DMA by a wave, 32 rows by all four; the 16-byte chunks of a row are swizzled on
  // the source side.  Buffer addressing (SGPR descriptor + 32-bit per-lane byte offset + SGPR K offset): no vector ALU work at all.
  // W, which comes from memory, runs three K-tiles ahead of the products, A, which the launch before wrote, SA; behind the last K-tile both repeat it
  // (into buffers that nobody reads any more), so that every K-tile has the same requests and the counted waits hold to the end.
  const int sw = ((tid & 7) ^ ((tid >> 3) & 7)) * 8;
  Aim256 aim;
  int wa = blockIdx.x, ka = 0, wb = blockIdx.x, kb = 0;           // the K-tiles to be requested next: output tile, K
  auto aim_a = [&]() {
    const Place256 t = place(wa);
    const bool v = QKV && t.swapped;                              // V tile: W rows fill the A side, tokens the B side
    int srow = tid >> 3;                                          // (opaque: what follows from it is not to be held through the K loop)
    asm volatile("" : "+v"(srow));
#pragma unroll
    for (int q = 0; q < MB; ++q) {
      const int rr = q * 32 + srow, ar = v ? min(t.n0 + rr, v_rows - 1) - t.n0 : min(t.m0 + rr, p.M - 1) - t.m0;
      aim.a_off[q] = (ar * (v ? p.ldw : p.lda) + sw) * 2;
    }
    const bf16_t* pa = v ? p.W + (size_t)(t.row0 + t.n0) * p.ldw : p.A + (size_t)t.m0 * p.lda;
    aim.rs_a = __builtin_amdgcn_make_buffer_rsrc((void*)pa, 0, 0xffffffff, 0x00020000);
  };
  auto aim_b = [&]() {
    const Place256 t = place(wb);
    const bool v = QKV && t.swapped;
    int srow = tid >> 3;
    asm volatile("" : "+v"(srow));
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int rr = q * 32 + srow;
      int br;
      if (SILU)                                       // a group of 64 tile columns = 32 gate rows + the 32 up rows of the same outputs
        br = min(t.n0 + (rr >> 6) * 32 + ((rr >> 4) & 1) * 16 + (rr & 15), p.N - 1) + ((rr & 63) >> 5) * p.N;
      else if (QKV)                                   // pair order (both halves of a rotation pair in one lane)
        br = v ? min(t.m0 + rr, p.M - 1) : qkv_pair_row(p.q, t.row0, t.n0 >> 1, rr);
      else
        br = min(t.n0 + rr, p.N - 1);
      aim.b_off[q] = (int)(((unsigned)br * (unsigned)(v ? p.lda : p.ldw) + (unsigned)sw) * 2u);   // < 2^32: checked by the launcher
    }
    const bf16_t* pb = v ? p.A : p.W;
    aim.rs_b = __builtin_amdgcn_make_buffer_rsrc((void*)pb, 0, 0xffffffff, 0x00020000);
  };
  auto next_a = [&]() {
    if (++ka < nk) return;
    if (wa + (int)gridDim.x < nwg) wa += gridDim.x, ka = 0, aim_a();
    else ka = nk - 1;
  };
  auto next_b = [&]() {
    if (++kb < nk) return;
    if (wb + (int)gridDim.x < nwg) wb += gridDim.x, kb = 0, aim_b();
    else kb = nk - 1;
  };
  auto request = [&](int n, int as, int bs) {                     // A's first: it is needed first
    if (n < MB) {
      lptr_t dst = (lptr_t)(smem + as + n * 4096 + wave * 1024);
      const int vo = aim.a_off[n & 7];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(aim.rs_a, dst, 16, vo, ka * (TK * 2), 0, 0);
    } else {
      lptr_t dst = (lptr_t)(smem + (int)B0 + bs + (n - (int)MB) * 4096 + wave * 1024);
      const int vo = aim.b_off[(n - (int)MB) & 7];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(aim.rs_b, dst, 16, vo, kb * (TK * 2), 0, 0);
    }
  };
  int wid = blockIdx.x;
  if (wid >= nwg) return;
  aim_a(), aim_b();
#pragma unroll
  for (int t = 0; t < 3; ++t) {
#pragma unroll
    for (int n = t < SA ? 0 : MB; n < NF; ++n) request(n, t * A_BYTES, t * B_BYTES);
    if (t < SA) next_a();
    next_b();
  }

  // ---- PRODUCTS: the fragments of one 32-wide half of a K-tile are multiplied while those of the next half are read
  const int frow = lane & 15, fo = frow * 128 + (((lane >> 4) ^ (frow & 7)) << 4);
  int as = 0, bs = 0;                                             // the buffers of the K-tile in hand
  f32x4_t acc[NG][MB][GB];
  bf16x8_t fa[2][MB], fb[2][NB];
  auto fetch = [&](int n, int kk, int as, int bs) {               // the first row block, the columns', then the other rows' (the MFMAs walk row by row)
    const int f = fo ^ (kk * 64);
    if (n == 0) fa[kk][0] = *(const bf16x8_t*)(smem + as + wr * (MB * 2048) + f);
    else if (n <= NB) fb[kk][n - 1] = *(const bf16x8_t*)(smem + B0 + bs + wc * (NB * 2048) + f + (n - 1) * 2048);
    else fa[kk][n - NB] = *(const bf16x8_t*)(smem + as + wr * (MB * 2048) + f + (n - NB) * 2048);
  };
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(SA == 3 ? 2 * NF : NF + NB) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int n = 0; n < NF; ++n) fetch(n, 0, 0, 0);
  bool landed = false;                                            // this wave's requests of the next K-tile have been waited for
  for (;;) {
    const Place256 t = place(wid);
    auto k_tile = [&](auto first) {                               // (first: the sums of an output tile start here)
      constexpr bool FIRST = decltype(first)::value;
      const int an = as == (SA - 1) * A_BYTES ? 0 : as + A_BYTES, bn = bs == 2 * B_BYTES ? 0 : bs + B_BYTES;
      auto mfma = [&](int kk, int m) {                            // (W fragment first: the block comes out TRANSPOSED, see the epilogue)
        const int i = m / NB, j = m % NB;
        f32x4_t& c = acc[j / GB][i][j % GB];
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[kk][j], fa[kk][i], FIRST && kk == 0 ? (f32x4_t){0.f, 0.f, 0.f, 0.f} : c, 0, 0, 0);
      };
      auto ask = [&](int m) {                                     // the requests that have their place in front of MFMA m (of both halves)
        m -= TURN + 2;
        if (m >= 0 && m % STEP == 0 && m / STEP < NF) request(m / STEP, as, bs);
        if (m == 2 * NM - 1 - (TURN + 2))
#pragma unroll
          for (int n = m / STEP + 1; n < NF; ++n) request(n, as, bs);
      };
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        if (m % 2 == 0 && m / 2 < NF) fetch(m / 2, 1, as, bs);
        if (m == TURN) {                                          // the next K-tile is in LDS, this one in registers: its buffers are given back
          if (!landed) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNG) : "memory");
          landed = false;
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
        }
        ask(m);
        mfma(0, m);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        if (m % 2 == 0 && m / 2 < NF) fetch(m / 2, 0, an, bn);
        ask(NM + m);
        mfma(1, m);
        __builtin_amdgcn_sched_barrier(0);
      }
      next_a(), next_b();
      as = an, bs = bn;
    };
    k_tile(std::true_type{});
#pragma unroll 1
    for (int kt = 1; kt < nk; ++kt) k_tile(std::false_type{});

    // What the next K-tile's turn waits for, waited for NOW, ahead of the epilogue's stores: the vector-memory counter cannot tell loads from
    // stores, so behind them the same wait would last until they have drained (all 256 CUs store at once: 5 - 10 us per tile).
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNG) : "memory");
    landed = true;
    int lane_e = lane;                                            // (opaque, as in aim_a)
    asm volatile("" : "+v"(lane_e));
    if constexpr (QKV) {
      QkvP q;
      __builtin_memcpy(&q, again(), sizeof(q));
      if (!t.swapped) qkv_epilogue_rot_groups<MB, 1, true>(q, acc, p.bias, t.is_k, t.row0, (t.n0 >> 1) + wc * 64, t.m0 + wr * MB * 16, p.M, lane_e);
      else qkv_epilogue_vt_groups<MB, true>(q, acc, p.bias ? p.bias + t.row0 : nullptr, t.n0 + wr * MB * 16, t.m0 + wc * 128, p.M, lane_e, v_rows);
    } else {
#pragma unroll
      for (int g = 0; g < NG; ++g)
        gemm256_epilogue<EPI, MB, GB, true>(p, acc[g], t.m0 + wr * MB * 16, t.n0 + wc * (n_out_tile / 2) + g * (SILU ? 32 : GB * 16), lane_e);
    }
    if (wid + (int)gridDim.x >= nwg) break;
    wid += gridDim.x;
    if constexpr (QKV) {                                          // (read once more: that epilogue needs the registers)
#pragma unroll
      for (int n = 0; n < NF; ++n) fetch(n, 0, as, bs);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                // (the requests that repeat the last K-tile: LDS is given back behind them)
}

int p3v_gemm256_cus();
int p3v_qkv_flat_tiles(const QkvP& q, int M, int mb);

template <int EPI, int MB, int NB>
static int launch_gemm256_v(const Gemm256P& p, hipStream_t s) {
  constexpr int TM = 32 * MB, TN = 32 * NB, LDS = (G256_SA(MB, NB) * TM + 3 * TN) * TK * 2;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm256<EPI, MB, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return P3V_ERR_HIP;
    attr_set = true;
  }
  const int n_cu = p3v_gemm256_cus();
  if (!n_cu) return P3V_ERR_HIP;
  int tiles = p3v_cdiv(p.N, P3V_GATED(EPI) ? TN / 2 : TN) * p3v_cdiv(p.M, TM);
  if (EPI == P3V_EPI_QKV) tiles = p3v_qkv_flat_tiles(p.q, p.M, MB);
  const int persist = p3v_tuning().gemm_persistent;                // 0: one workgroup per tile, else the persistent loop
  dim3 grid(persist ? min(tiles, n_cu) : tiles);
  hipLaunchKernelGGL((k_gemm256<EPI, MB, NB>), grid, dim3(256), LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}

// persistent grid: one workgroup per CU, a multiple of 8 (XCDs); 0: no device
int p3v_gemm256_cus() {
  static int n_cu = 0;
  if (!n_cu) {
    int dev = 0;
    hipDeviceProp_t pr;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&pr, dev) != hipSuccess) return 0;
    n_cu = pr.multiProcessorCount / 8 * 8;
  }
  return n_cu;
}

template <int EPI>
static int launch_gemm256(const Gemm256P& p, int mb, int nb, hipStream_t s) {
  if constexpr (!P3V_GATED(EPI) && EPI != P3V_EPI_QKV)
    if (nb == 3) return mb == 6 ? launch_gemm256_v<EPI, 6, 6>(p, s) : launch_gemm256_v<EPI, 8, 6>(p, s);
  if (mb == 6) return launch_gemm256_v<EPI, 6, 8>(p, s);
  if (mb == 7) return launch_gemm256_v<EPI, 7, 8>(p, s);
  return launch_gemm256_v<EPI, 8, 8>(p, s);
}
int p3v_gemm_pc(const Gemm256P& p, int epi, int mb, int nb, hipStream_t s);       // p3v_gemm_pc.hip: the flat tiles

// called by p3v_gemm (which decides how many rows get the big tile); returns P3V_ERR_UNSUPPORTED to fall back
int p3v_gemm256_try(const p3v_gemm_args_t* a, int mb, int nb, hipStream_t s) {
  // the tiles there are (the knob "gemm_tile" may ask for any); a gated epilogue needs whole gate / up pairs of a group of four column blocks
  const int tile = 10 * mb + nb;
  if (tile != 84 && tile != 74 && tile != 64 && tile != 54 && tile != 44 && (P3V_GATED(a->epilogue) || (tile != 83 && tile != 63 && tile != 43))) return P3V_ERR_UNSUPPORTED;
  const int n_tile = P3V_GATED(a->epilogue) ? 32 * nb : 64 * nb;
  if (a->N % n_tile || a->K % TK || a->epilogue == P3V_EPI_PATCH) return P3V_ERR_UNSUPPORTED;
  const size_t w_rows = (size_t)a->N * (P3V_GATED(a->epilogue) ? 2 : 1);
  if (w_rows * a->ldw * 2 >= ((size_t)1 << 32) || (size_t)256 * a->lda * 2 >= ((size_t)1 << 31) || (size_t)256 * a->ldo * 4 >= ((size_t)1 << 31)) return P3V_ERR_UNSUPPORTED;  // 32-bit buffer offsets
  const Gemm256P p = {a->A, a->W, a->out, a->epilogue == P3V_EPI_SCALE_RESID_F32 ? a->col_scale : a->bias, a->resid, a->M, a->N, a->K, a->lda, a->ldw, a->ldo, {}};
  if (mb < 6) return p3v_gemm_pc(p, a->epilogue, mb, nb, s);
  switch (a->epilogue) {
    case P3V_EPI_NONE: return launch_gemm256<P3V_EPI_NONE>(p, mb, nb, s);
    case P3V_EPI_BIAS: return launch_gemm256<P3V_EPI_BIAS>(p, mb, nb, s);
    case P3V_EPI_BIAS_QGELU: return launch_gemm256<P3V_EPI_BIAS_QGELU>(p, mb, nb, s);
    case P3V_EPI_BIAS_GELU: return launch_gemm256<P3V_EPI_BIAS_GELU>(p, mb, nb, s);
    case P3V_EPI_BIAS_RESID_F32: return launch_gemm256<P3V_EPI_BIAS_RESID_F32>(p, mb, nb, s);
    case P3V_EPI_RESID_BF16: return launch_gemm256<P3V_EPI_RESID_BF16>(p, mb, nb, s);
    case P3V_EPI_SILU_MUL: return launch_gemm256<P3V_EPI_SILU_MUL>(p, mb, nb, s);
    case P3V_EPI_GELU_MUL: return launch_gemm256<P3V_EPI_GELU_MUL>(p, mb, nb, s);
    case P3V_EPI_F32: return launch_gemm256<P3V_EPI_F32>(p, mb, nb, s);
    case P3V_EPI_SCALE_RESID_F32: return launch_gemm256<P3V_EPI_SCALE_RESID_F32>(p, mb, nb, s);
    default: return P3V_ERR_UNSUPPORTED;
  }
}

// the K slices of p3v_gemm_slices (p3v_gemm.hip): fp32 partials [S, M, N] of a whole problem on a flat tile
int p3v_gemm256_slices(const p3v_gemm_args_t* a, float* part, int S, int mb, int nb, hipStream_t s) {
  const int tile = 10 * mb + nb;
  if ((tile != 54 && tile != 44 && tile != 43) || a->N % (64 * nb) || a->K % TK || S < 1 || S > a->K / TK) return P3V_ERR_UNSUPPORTED;
  if ((size_t)80 * a->N * 4 >= ((size_t)1 << 31)) return P3V_ERR_UNSUPPORTED;   // the partials' 32-bit store offsets, 80 rows of a wave at most
  if ((size_t)a->N * a->ldw * 2 >= ((size_t)1 << 32) || (size_t)a->M * a->lda * 2 >= ((size_t)1 << 32)) return P3V_ERR_UNSUPPORTED;  // 32-bit buffer offsets
  const Gemm256P p = {a->A, a->W, part, nullptr, nullptr, a->M, a->N, a->K, a->lda, a->ldw, a->N, {}, S};
  return p3v_gemm_pc(p, P3V_EPI_PART, mb, nb, s);
}

// the qkv projection on tiles of 32 mb rows (qkv_tile_plan, p3v_gemm.hip)
int p3v_gemm256_flat_qkv(const p3v_gemm_args_t* a, const QkvP& q, int mb, hipStream_t s) {
  if (mb < 2 || mb > 8 || a->K % TK || (q.nh * q.hd) % 256 || (q.nkv * q.hd) % 256) return P3V_ERR_UNSUPPORTED;
  if ((size_t)a->N * a->ldw * 2 >= ((size_t)1 << 32) || (size_t)a->M * a->lda * 2 >= ((size_t)1 << 32) || (size_t)256 * a->ldw * 2 >= ((size_t)1 << 31)) return P3V_ERR_UNSUPPORTED;
  const Gemm256P p = {a->A, a->W, nullptr, a->bias, nullptr, a->M, a->N, a->K, a->lda, a->ldw, 0, q, 0};
  if (mb > 5) return launch_gemm256<P3V_EPI_QKV>(p, mb, 4, s);
  return p3v_gemm_pc(p, P3V_EPI_QKV, mb, 4, s);
}
