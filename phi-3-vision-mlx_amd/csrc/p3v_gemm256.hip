// Large-tile variant of the dense projection for prefill-sized problems (K % 64 == 0, columns in whole tiles; p3v_gemm decides which rows of a
// problem it gets and in which of its tiles):
//   256(M) x 256(N) x 64(K) tile (template: 224 rows, or 192 columns, for problems whose rounds they fill better), 512 threads = 8 waves
//   as 2(M) x 4(N), each wave 128 x 64 = 8 x 4 v_mfma_f32_16x16x32_bf16 accumulators (128 registers), 2.67 MFMAs per LDS fragment read
//   (the 128x128 kernel: 2.0) and 25 % less global->LDS traffic per flop.
//   K-tile t lives in LDS buffer t&1 (2 x 64 KiB); a tile is four quadrants (64 x 32 accumulators = 16 MFMAs each).  K-tile t+1 is
//   requested by LDS-DMA during the first two quadrants of K-tile t, A behind the first's fragment reads, B behind the second's: measured
//   against a quarter per quadrant (the last one then has only 16 MFMAs to land before the vmcnt(0)) +12 % at 4096^3 (1170 -> 1310 TF/s),
//   against all of it up front +7 % (eight DMA issues ahead of the first fragment reads delay the first MFMA).  The fragment reads are
//   software-pipelined: the fragments of the next quadrant are requested before the MFMAs of this one (second A-fragment buffer: all 256
//   registers, and one or two spilled in the gated and erf-GELU forms, reloaded once per output tile: no difference measured), +1.5-2 % at
//   4096^3 / 8192^3 (1.28 -> 1.30, 1.32 -> 1.34 PFLOP/s).  One vmcnt(0) + barrier per K-tile.  No barrier inside a tile: the waves
//   de-phase, one wave's fragment reads overlap another's MFMAs.
//   Same XOR-swizzled LDS image and the same epilogues as p3v_gemm.hip; stored straight from the accumulators.
#include <stdlib.h>

#include "p3v_gemm256_epi.h"

struct Tile256 {
  int m0, n0; int a_off[4], b_off[4]; __amdgpu_buffer_rsrc_t rs_a;
  int swapped, is_k, row0;              // P3V_EPI_QKV: V tile (operand roles swapped) / K region / first W row of the region
};

#ifdef P3V_G256_DEBUG                                            // tools/gemm256_timeline.py: per-wave stamps inside the K loop of ONE workgroup
__device__ unsigned long long p3v_g256dbg[8 * 64 * 8];
#define G_S(k) do { __builtin_amdgcn_sched_barrier(0); asm volatile("s_memtime %0" : "=s"(g_s[k])); __builtin_amdgcn_sched_barrier(0); } while (0)
#define G_FLUSH(it) do { if (blockIdx.x == P3V_G256_DEBUG && (threadIdx.x & 63) == 0 && (it) < 64) { for (int k_ = 0; k_ < 8; ++k_) p3v_g256dbg[((threadIdx.x >> 6) * 64 + (it)) * 8 + k_] = g_s[k_]; } } while (0)
extern "C" int p3v_g256dbg_read(unsigned long long* out) {
  return hipMemcpyFromSymbol(out, HIP_SYMBOL(p3v_g256dbg), sizeof(unsigned long long) * 8 * 64 * 8) == hipSuccess ? 0 : -1;
}
#else
#define G_S(k) do { } while (0)
#define G_FLUSH(it) do { } while (0)
#endif
// MB, NB: 16-row / 16-column blocks of a wave (2 x 4 waves: a tile of 32 MB rows x 64 NB columns)
template <int EPI, int MB, int NB>
__global__ void __launch_bounds__(512, 1) k_gemm256(Gemm256P p) {
  constexpr bool SILU = P3V_GATED(EPI), QKV = EPI == P3V_EPI_QKV;
  static_assert((MB == 7 || MB == 8) && (NB == 4 || (NB == 3 && !SILU)) && (!QKV || (MB == 8 && NB == 4)), "");
  constexpr int TM = 32 * MB, TN = 64 * NB, A_BYTES = TM * TK * 2, BUF_BYTES = A_BYTES + TN * TK * 2;
  constexpr int M0 = (MB + 1) / 2, M1 = MB - M0, N1 = NB - 2;                  // blocks of the two halves of a wave's rows / columns
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: LDS-DMA bases stay in SGPRs
  const int wr = wave >> 2, wc = wave & 3;
  constexpr int n_out_tile = SILU ? TN / 2 : TN;
  const int gx = (p.N + n_out_tile - 1) / n_out_tile, gy = (p.M + TM - 1) / TM, nwg = gx * gy;
  // (P3V_EPI_QKV: N = (nh + 2 nkv) * hd; column tiles 0 .. nq-1 are Q, then K, then V -- p3v_gemm_qkv.h)
  const int nq_t = QKV ? p.q.nh * p.q.hd / TN : 0, nk_t = QKV ? p.q.nkv * p.q.hd / TN : 0;

  // ---- PERSISTENT over output tiles: workgroup b takes tiles b, b + G, b + 2G, ... (G = gridDim.x, a multiple of 8,
  // so a workgroup's tiles keep its XCD in the XCD-aware order below).  The K-tile stream runs ACROSS tile seams: during the
  // last K-tile of a tile the first K-tile of the workgroup's NEXT tile is requested into the other LDS buffer, and the
  // epilogue (staged through the buffer that was just consumed) runs under that DMA -- the 64-KiB cold fetch that opened every
  // tile (HBM latency + 4 x 16 KiB, ~2 us) was 15-20 % of a K = 1024 tile (the ViT projections) and 5 % at K = 3072.
  using Tile = Tile256;   // (declared outside the template: a builtin called with a member of a DEPENDENT type is only checked at
                          //  instantiation, fails there in the HOST pass -- no such builtin -- and hipcc silently drops the host stub)
  const int srow = tid >> 3, schunk = tid & 7;
  auto make_tile = [&](int wid, Tile& t) {
    const int q = nwg >> 3, r = nwg & 7, xcd = wid & 7, loc = wid >> 3;
    const int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + loc;
    constexpr int BAND = 4;
    const int band = id / (BAND * gx), in_band = id % (BAND * gx);
    const int rows = min(BAND, gy - band * BAND);
    const int m_t = band * BAND + in_band % rows, n_t = in_band / rows;
    t.m0 = m_t * TM, t.n0 = n_t * n_out_tile;
    t.swapped = t.is_k = t.row0 = 0;
    if (QKV) {
      t.swapped = n_t >= nq_t + nk_t;
      t.is_k = !t.swapped && n_t >= nq_t;
      t.row0 = t.swapped ? (p.q.nh + p.q.nkv) * p.q.hd : t.is_k ? p.q.nh * p.q.hd : 0;
      t.n0 = (n_t - (t.swapped ? nq_t + nk_t : t.is_k ? nq_t : 0)) * TN;        // first column INSIDE the region
    }
    // DMA sources: instruction qq covers 64 tile rows, this thread: row tid/8, chunk tid%8.
    // Buffer addressing (SGPR descriptor + 32-bit per-lane byte offset + SGPR K offset): a request is `s_mov m0` +
    // `buffer_load_dwordx4 ... offen lds` with no vector ALU work at all.
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
      const int rr = qq * 64 + srow;
      const int sw = (schunk ^ (rr & 7)) * 8;
      const int ar = min(t.m0 + rr, p.M - 1) - t.m0;
      int br;
      if (SILU) {                                   // wave column group wcol (64 tile rows) = 32 gate + 32 up rows
        const int wcol = rr >> 6, ni = (rr & 63) >> 4, c = rr & 15;
        br = min(t.n0 + wcol * 32 + (ni & 1) * 16 + c, p.N - 1) + (ni >> 1) * p.N;
      } else if (QKV) {                             // Q / K: pair order (both halves of a rotation pair in one lane)
        br = qkv_pair_row(p.q, t.row0, t.n0 >> 1, rr);
      } else {
        br = min(t.n0 + rr, p.N - 1);
      }
      if (QKV && t.swapped) {
        // V tile: the tile's rows are the 256 W rows row0 + n0 .. (A side), its columns the tokens m0 .. (B side)
        t.a_off[qq] = (rr * p.ldw + sw) * 2;                                                  // from W + (row0 + n0) * ldw
        t.b_off[qq] = (int)(((unsigned)(t.m0 + ar) * (unsigned)p.lda + (unsigned)sw) * 2u);    // from A, clamped token row
      } else {
        t.a_off[qq] = (ar * p.lda + sw) * 2;
        t.b_off[qq] = (int)(((unsigned)br * (unsigned)p.ldw + (unsigned)sw) * 2u);   // < 2^32: checked by the launcher
      }
    }
    t.rs_a = QKV && t.swapped ? __builtin_amdgcn_make_buffer_rsrc((void*)(p.W + (size_t)(t.row0 + t.n0) * p.ldw), 0, 0xffffffff, 0x00020000)
                              : __builtin_amdgcn_make_buffer_rsrc((void*)(p.A + (size_t)t.m0 * p.lda), 0, 0xffffffff, 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)p.W, 0, 0xffffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, 0xffffffff, 0x00020000);   // (V tiles: tokens on the B side)
  auto dma_a = [&](const Tile& t, int kt, int buf) {             // (4 MB pieces of 8 rows over eight waves: an odd MB leaves half of them out of the last round)
    unsigned char* base = smem + buf * (int)BUF_BYTES + wave * 1024;
    const int n = MB;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q < n / 2 || (q == n / 2 && (n & 1) && wave < 4)) {
        lptr_t dst = (lptr_t)(base + q * 8192);
        const int vo = t.a_off[q];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(t.rs_a, dst, 16, vo, kt * (TK * 2), 0, 0);
      }
    }
  };
  auto dma_b = [&](const Tile& t, int kt, int buf) {
    unsigned char* base = smem + buf * (int)BUF_BYTES + (int)A_BYTES + wave * 1024;
    const __amdgpu_buffer_rsrc_t rs = (QKV && t.swapped) ? rs_x : rs_w;
    const int n = NB;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q < n) {
        lptr_t dst = (lptr_t)(base + q * 8192);
        const int vo = t.b_off[q];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 16, vo, kt * (TK * 2), 0, 0);
      }
    }
  };

  const int frow = lane & 15, fchunk = lane >> 4;
  const int nk = p.K / TK;
  int wid = blockIdx.x;
  if (wid >= nwg) return;
  Tile cur_t;
  make_tile(wid, cur_t);
  dma_a(cur_t, 0, 0);
  dma_b(cur_t, 0, 0);
  int gk = 0;                                                     // K-tiles consumed so far: LDS buffer = gk & 1
  bool landed = false;                                            // this wave's pieces of the K-tile about to be consumed are already in LDS
  for (;;) {
  const int m0 = cur_t.m0, n0 = cur_t.n0;
  const bool has_next = wid + (int)gridDim.x < nwg;
  f32x4_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

#ifdef P3V_G256_DEBUG
  unsigned long long g_s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#endif
  for (int kt = 0; kt < nk; ++kt, ++gk) {
    G_S(0);
    // (first K-tile of a later tile: waited for BEFORE the previous tile's stores were issued, below -- a vmcnt(0) here would
    //  wait for those stores to drain; so the barrier is the raw one, __syncthreads() would add that wait back)
    if (!(kt == 0 && landed)) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    G_S(1);
    __builtin_amdgcn_s_barrier();
    G_S(2);
    const bool last = kt + 1 == nk;
    const bool more = !last || has_next;                          // something to prefetch: this tile's next K-tile, or the next tile's first
    const int nb = (gk + 1) & 1;
    const unsigned char* ta = smem + (gk & 1) * BUF_BYTES + wr * MB * 2048;                       // this wave's rows
    const unsigned char* tb = smem + (gk & 1) * BUF_BYTES + A_BYTES + wc * NB * 2048;             // its columns
    bf16x8_t af[M0][2], af1[M1][2], bf0[2][2], bf1[N1][2];
    auto read = [&](const unsigned char* t, int first, auto& dst) {
#pragma unroll
      for (int i = 0; i < (int)(sizeof(dst) / sizeof(dst[0])); ++i)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const int r = (first + i) * 16 + frow;
          dst[i][kk] = *(const bf16x8_t*)(t + r * 128 + (((kk * 4 + fchunk) ^ (frow & 7)) << 4));
        }
    };
    auto quad = [&](int i0, int j0, auto& a, auto& bf) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < (int)(sizeof(a) / sizeof(a[0])); ++i)
#pragma unroll
          for (int j = 0; j < (int)(sizeof(bf) / sizeof(bf[0])); ++j)
            acc[i0 + i][j0 + j] =                    // (W fragment first: the block comes out TRANSPOSED, see the epilogue)
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[j][kk], a[i][kk], acc[i0 + i][j0 + j], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    };
    // the next K-tile's two halves: A requested in phase 0, B in phase 1, each behind the phase's fragment reads
    auto dma_next = [&](bool b_side) {
      if (!more) return;
      if (!last) {
        if (b_side) dma_b(cur_t, kt + 1, nb);
        else dma_a(cur_t, kt + 1, nb);
      } else {                                                    // the next tile's offsets are computed here, once per tile, and
        Tile nt;                                                  // die at once: kept live through the K loop they are spilled
        make_tile(wid + gridDim.x, nt);                           // (the kernel sits at the 256-register limit)
        if (b_side) dma_b(nt, 0, nb);
        else dma_a(nt, 0, nb);
      }
    };
    // (Measured and removed: the eight LDS-DMA pieces of a wave SPREAD over the first two quads, one piece every four
    //  MFMAs, instead of two bursts of four in front of them -- 18-30 % SLOWER on every shape.  tools/gemm256_timeline.py: a
    //  piece costs its wave ~80-150 cycles of instruction issue wherever it stands (580-750 cycles for 12 fragment reads + 4
    //  pieces, ~300 for 8 + 4, against 1024 for the K-tile's 64 MFMAs); inside a quad those cycles come out of the wave's own
    //  MFMA stream, in front of it the partner wave's MFMAs cover most of them.)
    // (Likewise measured and removed: the SIMD partners' DMA bursts at different places -- waves 0-3 in front of quads 0 / 1,
    //  waves 4-7 behind them -- so that the two waves of a SIMD are not both in their "reads + 4 pieces" stretch right after
    //  the barrier: 4-13 % slower on the big-tile shapes.)
    // software-pipelined fragment reads: the fragments of phase p+1 are requested BEFORE the MFMAs of phase p (second A
    // fragment buffer, 224 of 256 registers), so only the first reads after the barrier expose their LDS latency
    read(tb, 0, bf0);
    read(ta, 0, af);
    dma_next(false);
    read(tb, 2, bf1);
    __builtin_amdgcn_sched_barrier(0);
    G_S(3);
    quad(0, 0, af, bf0);
    __builtin_amdgcn_sched_barrier(0);
    G_S(4);
    read(ta, M0, af1);
    dma_next(true);
    __builtin_amdgcn_sched_barrier(0);
    G_S(5);
    quad(0, 2, af, bf1);
    __builtin_amdgcn_sched_barrier(0);
    G_S(6);
    quad(M0, 2, af1, bf1);
    quad(M0, 0, af1, bf0);
    G_S(7);
    G_FLUSH(kt);
  }

  // The next tile's first K-tile was requested during the last K-tile above: wait for it NOW, ahead of the epilogue's stores.  The
  // vector-memory counter cannot tell loads from stores, so behind the stores the same wait would last until they have drained
  // (all 256 CUs store at once: the HBM write rate, 5-10 us per tile); this way the next tile's first 64 MFMAs run under the drain.
  if (has_next) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    landed = true;
  }
  if constexpr (QKV) {
    if (!cur_t.swapped) qkv_epilogue_rot<MB>(p.q, acc, p.bias, cur_t.is_k, cur_t.row0, (n0 >> 1) + wc * 32, m0 + wr * MB * 16, p.M, lane);
    else qkv_epilogue_vt<MB>(p.q, acc, p.bias ? p.bias + cur_t.row0 : nullptr, n0 + wr * 128, m0 + wc * 64, p.M, lane);
  } else {
    gemm256_epilogue<EPI, MB, NB>(p, acc, m0 + wr * MB * 16, n0 + wc * (SILU ? 32 : NB * 16), lane);    // straight from the accumulators: p3v_gemm256_epi.h
  }
  if (!has_next) break;
  wid += gridDim.x;
  make_tile(wid, cur_t);
  }                                                             // next tile of this workgroup
}

int p3v_gemm256_cus();

template <int EPI, int MB, int NB>
static int launch_gemm256_v(const Gemm256P& p, hipStream_t s) {
  constexpr int TM = 32 * MB, TN = 64 * NB, LDS = 2 * (TM + TN) * TK * 2;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm256<EPI, MB, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return P3V_ERR_HIP;
    attr_set = true;
  }
  const int n_cu = p3v_gemm256_cus();
  if (!n_cu) return P3V_ERR_HIP;
  const int tiles = p3v_cdiv(p.N, P3V_GATED(EPI) ? TN / 2 : TN) * p3v_cdiv(p.M, TM);
  const int persist = p3v_tuning().gemm_persistent;                // 0: one workgroup per tile, else the persistent loop
  dim3 grid(persist ? min(tiles, n_cu) : tiles);
  hipLaunchKernelGGL((k_gemm256<EPI, MB, NB>), grid, dim3(512), LDS, s, p);
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
    if (nb == 3) return launch_gemm256_v<EPI, 8, 3>(p, s);
  if constexpr (EPI != P3V_EPI_QKV)
    if (mb == 7) return launch_gemm256_v<EPI, 7, 4>(p, s);
  return launch_gemm256_v<EPI, 8, 4>(p, s);
}
int p3v_gemm_pc(const Gemm256P& p, int epi, int mb, int nb, hipStream_t s);       // p3v_gemm_pc.hip: the flat tiles

// the qkv projection with split + RoPE + KV append in the epilogue (p3v_gemm_qkv, p3v_gemm.hip): rows of `a` on big tiles
int p3v_gemm256_qkv(const p3v_gemm_args_t* a, const QkvP& q, hipStream_t s) {
  if (a->N % 256 || a->K % TK || (q.nh * q.hd) % 256 || (q.nkv * q.hd) % 256) return P3V_ERR_UNSUPPORTED;
  if ((size_t)a->N * a->ldw * 2 >= ((size_t)1 << 32) || (size_t)a->M * a->lda * 2 >= ((size_t)1 << 32)) return P3V_ERR_UNSUPPORTED;
  const Gemm256P p = {a->A, a->W, nullptr, a->bias, nullptr, a->M, a->N, a->K, a->lda, a->ldw, 0, q};
  return launch_gemm256<P3V_EPI_QKV>(p, 8, 4, s);
}

// called by p3v_gemm (which decides how many rows get the big tile); returns P3V_ERR_UNSUPPORTED to fall back
int p3v_gemm256_try(const p3v_gemm_args_t* a, int mb, int nb, hipStream_t s) {
  // the tiles there are (the knob "gemm_tile" may ask for any); a gated epilogue needs whole gate / up pairs of a wave's four column blocks
  const int tile = 10 * mb + nb;
  if (tile != 84 && tile != 74 && tile != 54 && tile != 44 && (P3V_GATED(a->epilogue) || (tile != 83 && tile != 43))) return P3V_ERR_UNSUPPORTED;
  const int n_tile = P3V_GATED(a->epilogue) ? 32 * nb : 64 * nb;
  if (a->N % n_tile || a->K % TK || a->epilogue == P3V_EPI_PATCH) return P3V_ERR_UNSUPPORTED;
  const size_t w_rows = (size_t)a->N * (P3V_GATED(a->epilogue) ? 2 : 1);
  if (w_rows * a->ldw * 2 >= ((size_t)1 << 32) || (size_t)256 * a->lda * 2 >= ((size_t)1 << 31)) return P3V_ERR_UNSUPPORTED;  // 32-bit buffer offsets
  const Gemm256P p = {a->A, a->W, a->out, a->epilogue == P3V_EPI_SCALE_RESID_F32 ? a->col_scale : a->bias, a->resid, a->M, a->N, a->K, a->lda, a->ldw, a->ldo, {}};
  if (mb < 7) return p3v_gemm_pc(p, a->epilogue, mb, nb, s);
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
  if ((size_t)a->N * a->ldw * 2 >= ((size_t)1 << 32) || (size_t)a->M * a->lda * 2 >= ((size_t)1 << 32)) return P3V_ERR_UNSUPPORTED;  // 32-bit buffer offsets
  const Gemm256P p = {a->A, a->W, part, nullptr, nullptr, a->M, a->N, a->K, a->lda, a->ldw, a->N, {}, S};
  return p3v_gemm_pc(p, P3V_EPI_PART, mb, nb, s);
}

// the qkv projection on flat tiles of 32 mb rows (qkv_flat_plan, p3v_gemm.hip)
int p3v_gemm256_flat_qkv(const p3v_gemm_args_t* a, const QkvP& q, int mb, hipStream_t s) {
  if (mb < 2 || mb > 5 || a->K % TK || (q.nh * q.hd) % 256 || (q.nkv * q.hd) % 256) return P3V_ERR_UNSUPPORTED;
  if ((size_t)a->N * a->ldw * 2 >= ((size_t)1 << 32) || (size_t)a->M * a->lda * 2 >= ((size_t)1 << 32) || (size_t)256 * a->ldw * 2 >= ((size_t)1 << 31)) return P3V_ERR_UNSUPPORTED;
  const Gemm256P p = {a->A, a->W, nullptr, a->bias, nullptr, a->M, a->N, a->K, a->lda, a->ldw, 0, q, 0};
  return p3v_gemm_pc(p, P3V_EPI_QKV, mb, 4, s);
}
