// Prompt-sized-but-short projections  C[M, N] = A[M, K] * W[N, K]^T  for 9 .. 256 rows: a 128-token chat prompt, the text
// group of a mixed batch, a 9..128-row decode batch.  At these M the GEMM is a WEIGHT STREAM (2 * 128 * N * K flops against N * K * 2
// bytes: ~13 GFLOP for the 100 MB of gate_up, both worth ~10-17 us), and what decides its speed is how many K-tiles a workgroup
// has on the wire: the 128 x 128-tile kernel (p3v_gemm.hip) holds ONE ahead and pays a DMA round trip (~1.3 us at this load) per
// K-tile -- gate_up 34 us + 5 us for the reduction of the split it needs to reach 256 workgroups, 2.9 TB/s.  Here:
//   tile      128(M) x 64(N) x 64(K): twice the workgroups per weight matrix, so gate_up (256 tiles) and qkv (144) run in one pass
//             and the others with a smaller split over K (o_proj 4, down 4 slices: one workgroup per CU, partials <= a quarter of
//             the weight bytes).  The kernel's bound: every workgroup re-reads the A panel from L2 beside its weight stream from
//             HBM, and in one CU the two add up -- the same requests without any compute take as long as gate_up, 30 us at 128
//             rows (rows 6144 bytes apart; weights alone 18.5, both packed 25.9: profiles/lds_dma_probe.txt).  Rows of A and W 128 bytes further apart: gate_up 30.2 ->
//             27.7, qkv 26 -> 24.3, but down 22.6 -> 25.4; the weights lie unpadded, as the other kernels and the loader have them.
//             128 x 128 tiles (W x 2 staged, half the workgroups) in one pass are not faster up to 128 rows; where the K slices that fill the
//             chip again are summed inside the launch they are (p3v_gemm_merge, at the end).  Beyond 128 rows they are wherever 64 columns take two
//             rounds of the chip and 128 one: gate_up of 129 / 192 / 256 rows 45.5 -> 30.4, 44.5 -> 32.6, 45.3 -> 36.2 us, qkv 34.7 -> 27.2, 35.9 -> 30.9,
//             40.4 -> 36.2 (6144 columns, one round either way: 18.2 against 23.3).  257 .. 384 rows whose tiles are more than half a round and no more than
//             one (sk_tall): 9216 x 3072 37.6 -> 25.6 at 266, 41.2 -> 33.0 at 384, qkv 42.3 -> 28.1, 46.6 -> 35.8 (slices of K before); gated ones would
//             take two rounds (44.7 against 54.6).
//             Plain partials of a long K: 128 x 96 tiles in up to 8 slices where that is a workgroup for more CUs than 64 columns reach (3072 columns:
//             256 against 192), each of which then asks for less (448 against 768 KB of 8192 at 128 rows; the requests alone 16.5 -> 11.5 us).  With the
//             reduction, 3072 x 8192: 128 rows 24.2 -> 21.8 us, 64 rows 19.9 -> 17.3, 40 rows 18.4 -> 16.3, 160 rows 28.5 -> 23.3, 200 30.3 -> 24.9, 256 34.7 ->
//             28.0 (four slices); x 6144 at 100 rows (12 K-tiles a slice) 19.8 -> 18.0, at 200 25.3 -> 21.8; x 4096 at 200 (16) 19.0 -> 17.3; x 3072 would have 6
//             K-tiles a slice up to 128 rows (15.5 -> 16.6) and 12 beyond (15.4 -> 15.8): slices of fewer than 12 and 16 stay on 64 columns.
//   staging   LDS-DMA into a ring of 6 stages (A 16 KiB + W 8 KiB each), 5 in flight behind a counted vmcnt; one workgroup per CU
//             (<= 64 rows: 64-row tiles, A 8 KiB per stage -- a third less staged per K-tile, the same sums bit for bit: 60 -> 53 us
//             per decoder layer at 17 rows)
//   waves     8: four CONSUMERS (stacked along M, 32 rows x 64 columns each: acc[2][4]; W fragment first
//             in the MFMA, so the epilogue is the register-direct one of the other GEMM kernels, p3v_gemm256_epi.h) and four
//             PRODUCERS that only issue the DMA and wait for it; one barrier per K-tile hands a landed stage over and a drained
//             one back.  (With the MFMA waves issuing their own DMA a K-tile cost the SUM of its DMA issue, ~800 cycles for 24 KB,
//             and its fragment reads + MFMAs, ~400.)
//   K slices  gridDim.z; fp32 partials [S, M, ldp] in the caller's workspace, added in slice order by k_splitk_reduce (p3v_gemm.hip)
// (tools/scratch/gemm_skinny_regw_r5.hip: the variant that keeps each wave's W fragments out of LDS -- global loads straight into a
// register ring 8 K-tiles deep, A alone through LDS -- measured slower on every shape: profiles/r05_skinny_gemm.txt.)
#include "p3v_gemm_qkv.h"

#define SK_BM 128
#define SK_BK 64
#define SK_TN 64                    // tile width, but 96 for partial sums of a long K (sk_plan), 128 for MERGE and one pass of many rows (sk_one_pass_tn, sk_tall)
#ifndef SK_ABL
#define SK_ABL 0                    // timing experiments: 1 = A always K-tile 0 (one L2/L1-hot tile), 2 = W likewise, 3 = no MFMAs after K-tile 0
#endif
#define SK_A_BYTES (SK_BM * SK_BK * 2)

typedef __attribute__((address_space(3))) void* lptr_t;

template <int TN, int TM = SK_BM> struct SkCfg {
  static_assert(TM == 128 || (TM == 64 && TN <= 96), "64-row tiles: prompts / batches of <= 64 rows, 64- and 96-column tiles");
  static constexpr int NS = TN == 64 ? 6 : TN == 96 ? 5 : 4;   // ring stages (NS - 1 ahead)
  static constexpr int A_BYTES = TM * SK_BK * 2, W_BYTES = TN * SK_BK * 2, STAGE = A_BYTES + W_BYTES, LDS = NS * STAGE;
  static constexpr int AQ = TM / 32, WQ = TN / 32;             // A / W pieces (8 rows x 128 B) per producer wave and stage
  static constexpr int PER = AQ + WQ;                          // DMA instructions per producer wave and stage
  static constexpr int NI = TN == 128 ? 4 : TM / 64;           // 16-row blocks per consumer wave ...
  static constexpr int NJ = TN == 96 ? 6 : 4;                  // ... and 16-column blocks
};

// s_waitcnt vmcnt(PER * n) for a uniform run-time n = stages that may stay in flight (PER: DMA instructions per stage)
template <int PER>
__device__ __forceinline__ void sk_wait_stages(int n) {
  switch (n) {
    case 1: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER) : "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PER) : "memory"); break;
    case 3: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * PER) : "memory"); break;
    case 4: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * PER < 63 ? 4 * PER : 63) : "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
}

struct SkinnyP {
  const bf16_t* A; const bf16_t* W; void* out; const void* resid;
  int M, N, K, lda, ldw, ldo;      // N = output columns (SiLU: W holds 2N rows, gate rows then up rows)
  const bf16_t* col_scale;         // P3V_EPI_SCALE_RESID_F32
  int kslice;                      // 0: one pass with the epilogue; else K columns per slice, fp32 partials
  QkvP q;                          // P3V_EPI_QKV only (p3v_gemm_qkv.h): head split + rotation + KV append in the epilogue
  float* xpart; unsigned* xflag;   // MERGE: partial tiles [tile][slice][consumer wave][block][lane] x 4, counters [tile][consumer wave] (multiples of 4 between launches)
  int nk_part;                     // MERGE: K-tiles of a slice other than the last
  unsigned polls;                  // MERGE: how often the last slice looks at a counter before it gives up
};

#define P3V_EPI_QKV 100            // internal, as in the other GEMM kernels

// MERGE: gridDim.z slices of K, summed inside the launch (see p3v_gemm_merge below)
template <int EPI, bool PART, int TN, int TM = SK_BM, bool MERGE = false>
__global__ void __launch_bounds__(512, 1) k_gemm_skinny(SkinnyP p) {
  typedef SkCfg<TN, TM> C;
  static_assert(TM == SK_BM || EPI != P3V_EPI_QKV, "the qkv epilogue's V tiles are 128 dimensions tall");
  static_assert(!MERGE || (!PART && TN == 128), "merged slices: 128-column tiles");
  constexpr bool SILU = P3V_GATED(EPI);
  constexpr int NS = C::NS, NI = C::NI, NJ = C::NJ;
  static_assert(TN != 96 || (PART && !P3V_GATED(EPI)), "96-column tiles: plain partial sums");
  static_assert(NS - 2 <= 4 && (NS - 2) * C::PER < 64, "sk_wait_stages covers 4 stages in flight");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr bool QKV = EPI == P3V_EPI_QKV;
  static_assert(!QKV || !PART, "the qkv epilogue needs whole sums");
  constexpr int n_out_tile = SILU ? TN / 2 : TN;
  int n0 = blockIdx.x * n_out_tile, m0 = blockIdx.y * TM;
  const int kz = blockIdx.z;
  const bool last = !MERGE || kz == (int)gridDim.z - 1;          // the slice that adds the others' sums to its own
  const int nk = MERGE ? (last ? p.K / SK_BK - kz * p.nk_part : p.nk_part) : (PART ? p.kslice : p.K) / SK_BK, kt0 = kz * (MERGE ? p.nk_part : nk);
  // P3V_EPI_QKV (p3v_gemm_qkv.h), a one-dimensional grid: first the Q and K tiles (128 tokens x 32 rotation pairs, W rows fetched in
  // pair order), M-tile-major; then the V tiles with the operand roles swapped (128 V dimensions on the tile's A side, 64 tokens on
  // its B side), so that a lane ends up with consecutive TOKENS of one dimension for the transposed cache.
  bool swapped = false, is_k = false;
  int row0 = 0;
  if (QKV) {
    const int nq_t = p.q.nh * p.q.hd / TN, nk_t = p.q.nkv * p.q.hd / TN, nqk = nq_t + nk_t, mt = (p.M + SK_BM - 1) / SK_BM;
    int t = blockIdx.x;
    if (t < nqk * mt) {
      const int n_t = t % nqk;
      m0 = (t / nqk) * SK_BM;
      is_k = n_t >= nq_t;
      row0 = is_k ? p.q.nh * p.q.hd : 0;
      n0 = (n_t - (is_k ? nq_t : 0)) * TN;                     // first column INSIDE the region
    } else {
      t -= nqk * mt;
      const int nv_t = p.q.nkv * p.q.hd / SK_BM;
      swapped = true;
      row0 = (p.q.nh + p.q.nkv) * p.q.hd;
      n0 = (t % nv_t) * SK_BM;                                 // first V dimension of the tile (its A side)
      m0 = (t / nv_t) * TN;                                    // first token (its B side)
    }
  }

  if (wave >= 4) {
    // ---- PRODUCERS: wave pw stages 4 A pieces and WQ W pieces per K-tile, a piece = 8 tile rows x 128 B (1 KiB), the 16-byte
    // chunks of a row XOR-swizzled on the SOURCE side (the DMA destination is lane-linear).
    // SiLU: a 64-column group of the tile = gate rows (blocks 0, 1) and the up rows (blocks 2, 3) of the same 32 output columns.
    const int srow = lane >> 3, schunk = lane & 7, pw = wave - 4;
    unsigned a_src[4], w_src[4];                                 // (fixed sizes: see the note in stage())
    __amdgpu_buffer_rsrc_t rs_a = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, 0xffffffff, 0x00020000);
    __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)p.W, 0, 0xffffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rs_x = rs_a;
    if (QKV && swapped) { rs_a = rs_w; rs_w = rs_x; }           // the tile's A side reads W rows, its B side token rows
#pragma unroll
    for (int q = 0; q < C::AQ; ++q) {
      const int r = (pw * C::AQ + q) * 8 + srow;
      if (QKV && swapped) {
        a_src[q] = (unsigned)(((size_t)(row0 + n0 + r) * p.ldw + ((schunk ^ (r & 7)) * 8)) * 2);
      } else {
        const int ar = min(m0 + r, p.M - 1);
        a_src[q] = (unsigned)(((size_t)ar * p.lda + ((schunk ^ (r & 7)) * 8)) * 2);
      }
    }
#pragma unroll
    for (int q = 0; q < C::WQ; ++q) {
      const int r = (pw * C::WQ + q) * 8 + srow;
      if (QKV && swapped) {
        const int ar = min(m0 + r, p.M - 1);
        w_src[q] = (unsigned)(((size_t)ar * p.lda + ((schunk ^ (r & 7)) * 8)) * 2);
        continue;
      }
      int br;
      if (SILU) br = min(n0 + (r >> 6) * 32 + ((r >> 4) & 1) * 16 + (r & 15), p.N - 1) + ((r >> 5) & 1) * p.N;
      else if (QKV) br = qkv_pair_row(p.q, row0, n0 >> 1, r);
      else br = min(n0 + r, p.N - 1);
      w_src[q] = (unsigned)(((size_t)br * p.ldw + ((schunk ^ (r & 7)) * 8)) * 2);
    }
    auto stage = [&](int kt, int slot) {
      // (every argument of the builtin is a local of NON-DEPENDENT type: a type-dependent one defers the check to instantiation,
      // where the HOST pass does not know the builtin and hipcc silently drops the kernel's host stub)
      unsigned char* base = smem + slot * (int)C::STAGE;
      const int koff = (kt0 + kt) * (SK_BK * 2), koff_a = SK_ABL == 1 ? 0 : koff, koff_w = SK_ABL == 2 ? 0 : koff;
      const int wq = C::WQ, aq = C::AQ, a_bytes = C::A_BYTES;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q < aq) {
          lptr_t dst = (lptr_t)(base + (pw * aq + q) * 1024);
          const unsigned vo = a_src[q];
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, dst, 16, vo, koff_a, 0, 0);
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q < wq) {
          lptr_t dst = (lptr_t)(base + a_bytes + (pw * wq + q) * 1024);
          const unsigned vo = SK_ABL == 2 ? a_src[q] : w_src[q];
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_w, dst, 16, vo, koff_w, 0, 0);
        }
      }
    };
    for (int st = 0; st < min(NS - 1, nk); ++st) stage(st, st);
    int slot = 0;
    for (int kt = 0; kt < nk; ++kt) {
      sk_wait_stages<C::PER>(min(NS - 2, nk - 1 - kt));        // stage kt has landed when only the younger stages are still out
      __builtin_amdgcn_s_barrier();                             // tells the consumers; and they are done reading kt - 1
      if (kt + NS - 1 < nk) stage(kt + NS - 1, slot == 0 ? NS - 1 : slot - 1);   // ... whose slot takes K-tile kt + NS - 1
      slot = slot == NS - 1 ? 0 : slot + 1;
    }
    return;
  }

  // ---- CONSUMERS: wave (wr, wc) owns NI x 16 rows from wr * NI * 16 and the 64 columns of group wc
  const int wr = TN == 128 ? wave >> 1 : wave, wc = TN == 128 ? wave & 1 : 0;
  f32x4_t acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int frow = lane & 15, fchunk = lane >> 4;
  {
    int slot = 0;
    for (int kt = 0; kt < nk; ++kt) {
      __builtin_amdgcn_s_barrier();                             // K-tile kt is in LDS (every producer waited for its pieces)
      const unsigned char* ta = smem + slot * C::STAGE;
      const unsigned char* tb = ta + C::A_BYTES;
      bf16x8_t af[2][NI], bfr[2][NJ];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int r = (wr * NI + i) * 16 + frow;
          af[kk][i] = *(const bf16x8_t*)(ta + r * 128 + (((kk * 4 + fchunk) ^ (r & 7)) << 4));
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const int r = wc * 64 + j * 16 + frow;
          bfr[kk][j] = *(const bf16x8_t*)(tb + r * 128 + (((kk * 4 + fchunk) ^ (r & 7)) << 4));
        }
      }
      __builtin_amdgcn_sched_barrier(0);                        // all fragment reads out before the first MFMA (counted lgkmcnt)
#pragma unroll
      for (int kk = 0; kk < (SK_ABL == 3 ? (kt == 0 ? 2 : 0) : 2); ++kk)
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[kk][j], af[kk][i], acc[i][j], 0, 0, 0);   // W first: transposed block
      slot = slot == NS - 1 ? 0 : slot + 1;
    }
  }

  if constexpr (MERGE) {
    // A wave of another slice writes its blocks past the caches, waits until they are there and counts itself in; the last slice's wave of
    // the same place waits for all of them and adds them in slice order.  Its workgroups come last in dispatch order, so whatever they
    // wait for runs or has run; it has more K-tiles than the others, whose sums are on their way meanwhile.
    // A counter is a multiple of 4 between launches and counts modulo 4 (at most three others: merge_plan).  The waiting wave puts it back
    // to 0; one that gave up cannot, the late ones are still to count themselves in: it adds what they leave to the next multiple, so that
    // the next launch on this workspace, which starts behind them, waits for its own partials again.
    const int tile = (int)blockIdx.x, others = (int)gridDim.z - 1;
    // (rows and, in a V tile, tokens beyond M: nothing is stored for them)
    const bool live = (QKV && swapped ? m0 + wc * 64 : m0 + wr * NI * 16) < p.M;
    unsigned* flag = p.xflag + tile * 4 + wave;
    constexpr int WAVE_BYTES = NI * 4 * 1024;
    const __amdgpu_buffer_rsrc_t rs_p = __builtin_amdgcn_make_buffer_rsrc((void*)(p.xpart + (size_t)(tile * others) * (WAVE_BYTES)), 0, others * 4 * WAVE_BYTES, 0x00020000);
    const int my = lane * 16;
    if (!last) {
      if (!live) return;
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i][j]), rs_p, my + (i * 4 + j) * 1024, (kz * 4 + wave) * WAVE_BYTES, 16);   // (16: sc1)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (lane == 0) __hip_atomic_fetch_add(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    if (live) {
      bool late = true;
      for (unsigned n = 0; n < p.polls; ++n) {
        if ((__builtin_amdgcn_readfirstlane(__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) & 3u) == (unsigned)others) { late = false; break; }
        __builtin_amdgcn_s_sleep(1);
      }
      asm volatile("" ::: "memory");
      auto load = [&](u32x4_t (&v)[NI][4], int z) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) v[i][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_p, my + (i * 4 + j) * 1024, (z * 4 + wave) * WAVE_BYTES, 16);
      };
      auto add = [&](const u32x4_t (&v)[NI][4]) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] += __builtin_bit_cast(f32x4_t, v[i][j]);
      };
      u32x4_t v[NI][4];
      for (int z = 0; z < others; ++z) { load(v, z); add(v); }   // (two slices' loads at once: no faster)
      if (late) {                                                // loud, not wrong
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4_t){__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
      }
      if (lane == 0) {
        if (late) __hip_atomic_fetch_add(flag, 4u - (unsigned)others, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else __hip_atomic_store(flag, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }

  // ---- epilogue, straight from the accumulators: lane (fc = lane & 15, fq = lane >> 4) holds columns 4 fq .. 4 fq + 3 of block
  //      row fc (see p3v_gemm256_epi.h)
  if constexpr (QKV) {
    if (!swapped) qkv_epilogue_rot<NI>(p.q, acc, nullptr, is_k, row0, (n0 >> 1) + wc * 32, m0 + wr * NI * 16, p.M, lane);
    else qkv_epilogue_vt<NI>(p.q, acc, nullptr, n0 + wr * NI * 16, m0 + wc * 64, p.M, lane);
    return;
  }
  const int fc = lane & 15, fq = lane >> 4;
  const int mrow0 = m0 + wr * NI * 16 + fc;
  if constexpr (PART) {
    // fp32 partial of slice kz, [M, ldp] with ldp = W rows: SiLU keeps [gate | up] as 2N plain columns (k_splitk_reduce's layout)
    const int ldp = SILU ? 2 * p.N : p.N;
    float* part = (float*)p.out + (size_t)kz * p.M * ldp;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int m = mrow0 + i * 16;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int nn = SILU ? n0 + wc * 32 + (j & 1) * 16 + fq * 4 : n0 + wc * 64 + j * 16 + fq * 4;
        if (m < p.M && nn < p.N)
          *(float4*)(part + (size_t)m * ldp + nn + (SILU ? (j >> 1) * p.N : 0)) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
      }
    }
    return;
  }
  if constexpr (SILU) {
    const int n = n0 + wc * 32 + (fq & 1) * 16 + (fq >> 1) * 8;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
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
  if constexpr (EPI == P3V_EPI_SCALE_RESID_F32) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int m = mrow0 + i * 16;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + wc * 64 + j * 16 + fq * 4;
        if (m < p.M && n < p.N) {
          const size_t o = (size_t)m * p.ldo + n;
          const u32x2_t c = *(const u32x2_t*)(p.col_scale + n);
          const float4 r4 = *(const float4*)((const float*)p.resid + o);
          *(float4*)((float*)p.out + o) = make_float4(r4.x + acc[i][j][0] * bf16lo(c[0]), r4.y + acc[i][j][1] * bf16hi(c[0]),
                                                      r4.z + acc[i][j][2] * bf16lo(c[1]), r4.w + acc[i][j][3] * bf16hi(c[1]));
        }
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int m = mrow0 + i * 16;
#pragma unroll
    for (int jp = 0; jp < 2; ++jp) {
      uint32_t pk[2][2];
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int j = 2 * jp + jj;
        pk[jj][0] = pack_bf16x2(acc[i][j][0], acc[i][j][1]), pk[jj][1] = pack_bf16x2(acc[i][j][2], acc[i][j][3]);
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

// K slices for a shape on this kernel: 0 = not one of its shapes; 1 = one pass; S > 1 = S slices + the reduction launch.
// One workgroup per CU: the largest S <= 8 whose tiles * S still fit one round of the chip (slices of >= 6 K-tiles).
extern "C" int p3v_gemm_rows_slices(int M, int N, int K, int epilogue);            // p3v_gemm_rows.hip: 9 .. 32 rows, weights straight to registers
int p3v_gemm_rows_launch(const p3v_gemm_args_t* a, float* part, hipStream_t s);
struct SkPlan { int S, tn; };                                     // slices, tile columns
static SkPlan sk_plan(int M, int N, int K, int epilogue, bool wide);
static int sk_slices(int M, int N, int K, int epilogue) { return sk_plan(M, N, K, epilogue, false).S; }
int p3v_gemm_skinny_slices(int M, int N, int K, int epilogue) {
  const int rs = p3v_gemm_rows_slices(M, N, K, epilogue);
  return rs ? rs : sk_slices(M, N, K, epilogue);
}
// Columns of a one-pass tile: rounds of the chip times what a K-tile asks for, 32 KB on 128 columns and 24 on 64 (the header's figures)
static int sk_one_pass_tn(int M, int rows) {
  const int pin = p3v_tuning().gemm_skinny_tn, mt = p3v_cdiv(M, SK_BM);
  if (M <= 64 || rows % 128) return SK_TN;
  if (pin > 0) return pin == 128 ? 128 : SK_TN;
  return p3v_cdiv(mt * (rows / 128), 256) * 4 < p3v_cdiv(mt * (rows / 64), 256) * 3 ? 128 : SK_TN;
}
// Rows beyond the knob's: one round of 128 x 128 tiles in one pass, where p3v_gemm would run slices of K through a workspace
int p3v_splitk_slices(int M, int N, int K, int epilogue);            // p3v_gemm.hip
static bool sk_tall(int M, int N, int K, int epilogue) {
  const P3vTuning& t = p3v_tuning();
  if (t.gemm_no_skinny || t.gemm_skinny_tn == SK_TN || M <= t.gemm_skinny_max_m || M > 3 * SK_BM || epilogue != P3V_EPI_NONE || N % 128 || K % SK_BK) return false;
  const int tiles = p3v_cdiv(M, SK_BM) * (N / 128);
  return tiles > 128 && tiles <= 256 && p3v_splitk_slices(M, N, K, epilogue) > 1;
}
extern "C" int p3v_gemm_one_pass_pays(int M, int N, int K, int epilogue) { return M > 0 && N > 0 && K > 0 && sk_tall(M, N, K, epilogue); }
// wide: whether the caller's workspace holds the partials of 96-column tiles too (p3v_gemm_ws_most_bytes)
static SkPlan sk_plan(int M, int N, int K, int epilogue, bool wide) {
  const P3vTuning& t = p3v_tuning();
  const bool silu = P3V_GATED(epilogue);
  if (t.gemm_no_skinny || M <= 8 || M > t.gemm_skinny_max_m || K % SK_BK || N % (silu ? 32 : 64)) return {0, SK_TN};
  if (epilogue != P3V_EPI_NONE && epilogue != P3V_EPI_RESID_BF16 && epilogue != P3V_EPI_SCALE_RESID_F32 && !silu) return {0, SK_TN};
  const int mt = p3v_cdiv(M, SK_BM), tiles = mt * ((silu ? 2 * N : N) / SK_TN);
  if (t.gemm_skinny_s > 0) return {K % (t.gemm_skinny_s * SK_BK) ? 1 : t.gemm_skinny_s, SK_TN};
  auto slices = [&](int n) {
    int best = 1;
    for (int S = 2; S <= 8; ++S)
      if (K % (S * SK_BK) == 0 && K / S >= 6 * SK_BK && n * S <= t.gemm_splitk_wgs) best = S;
    return best;
  };
  const int S = slices(tiles);
  if (S == 1) return {1, sk_one_pass_tn(M, silu ? 2 * N : N)};
  if (!wide || silu || N % 96 || t.gemm_skinny_tn == SK_TN) return {S, SK_TN};
  const int tiles96 = mt * (N / 96), S96 = slices(tiles96);
  return S96 > 1 && tiles96 * S96 > tiles * S && K / S96 >= (mt > 1 ? 16 : 12) * SK_BK ? SkPlan{S96, 96} : SkPlan{S, SK_TN};
}
int p3v_gemm_skinny_most_slices(int M, int N, int K, int epilogue) {
  const int rs = p3v_gemm_rows_slices(M, N, K, epilogue);
  return rs ? rs : sk_plan(M, N, K, epilogue, true).S;
}

// 96-column tiles: plain partial sums
template <int TM>
static int launch_skinny96(const SkinnyP& p, int S, hipStream_t s) {
  typedef SkCfg<96, TM> C;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm_skinny<P3V_EPI_NONE, true, 96, TM>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS) != hipSuccess) return P3V_ERR_HIP;
    attr_set = true;
  }
  hipLaunchKernelGGL((k_gemm_skinny<P3V_EPI_NONE, true, 96, TM>), dim3(p.N / 96, p3v_cdiv(p.M, TM), S), dim3(512), C::LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}
// 128-column tiles in one pass
template <int EPI>
static int launch_skinny128(const SkinnyP& p, int grid_x, int grid_y, hipStream_t s) {
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm_skinny<EPI, false, 128>, hipFuncAttributeMaxDynamicSharedMemorySize, SkCfg<128>::LDS) != hipSuccess) return P3V_ERR_HIP;
    attr_set = true;
  }
  hipLaunchKernelGGL((k_gemm_skinny<EPI, false, 128>), dim3(grid_x, grid_y), dim3(512), SkCfg<128>::LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}
template <int EPI, int TM>
static int launch_skinny_tm(const SkinnyP& p, int S, hipStream_t s) {
  typedef SkCfg<SK_TN, TM> C;
  static bool attr_set[2] = {false, false};
  const bool part = S > 1;
  if (!attr_set[part]) {
    const void* fn = part ? (const void*)k_gemm_skinny<EPI, true, SK_TN, TM> : (const void*)k_gemm_skinny<EPI, false, SK_TN, TM>;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS) != hipSuccess) return P3V_ERR_HIP;
    attr_set[part] = true;
  }
  const int n_tile = P3V_GATED(EPI) ? SK_TN / 2 : SK_TN;
  const dim3 grid(p.N / n_tile, p3v_cdiv(p.M, TM), S);
  if (part) hipLaunchKernelGGL((k_gemm_skinny<EPI, true, SK_TN, TM>), grid, dim3(512), C::LDS, s, p);
  else hipLaunchKernelGGL((k_gemm_skinny<EPI, false, SK_TN, TM>), grid, dim3(512), C::LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}
// <= 64 rows: 64-row tiles (the A panel is two thirds of what a 128-row tile stages per K-tile; half of it would be clamped copies)
template <int EPI>
static int launch_skinny(const SkinnyP& p, int S, hipStream_t s) {
  if (const int rows = P3V_GATED(EPI) ? 2 * p.N : p.N; S == 1 && sk_one_pass_tn(p.M, rows) == 128) return launch_skinny128<EPI>(p, rows / 128, p3v_cdiv(p.M, SK_BM), s);
  return p.M <= 64 && !p3v_tuning().gemm_skinny_tm128 ? launch_skinny_tm<EPI, 64>(p, S, s) : launch_skinny_tm<EPI, SK_BM>(p, S, s);
}

int p3v_splitk_reduce(const float* part, const p3v_gemm_args_t* a, int S, hipStream_t s);   // p3v_gemm.hip

// the K-slice launch alone (fp32 partials into a->ws; *S_out slices): P3V_ERR_UNSUPPORTED, nothing launched, unless the shape is
// one this kernel splits and the workspace holds the partials
int p3v_gemm_skinny_partials(const p3v_gemm_args_t* a, int* S_out, hipStream_t s) {
  const bool silu = P3V_GATED(a->epilogue);
  const int w_rows = silu ? 2 * a->N : a->N;
  const int RS = a->bias ? 0 : p3v_gemm_rows_slices(a->M, a->N, a->K, a->epilogue);
  if (RS > 1 && a->ws && a->ws_bytes >= (int64_t)RS * a->M * w_rows * 4) {        // 9 .. 32 rows: the register-streaming kernel's K slices
    if ((uintptr_t)a->ws & 15) return P3V_ERR_ARG;
    *S_out = RS;
    return p3v_gemm_rows_launch(a, (float*)a->ws, s);
  }
  if (RS == 1) return P3V_ERR_UNSUPPORTED;                       // (runs in one pass: no partials)
  SkPlan pl = sk_plan(a->M, a->N, a->K, a->epilogue, true);
  if (pl.tn == 96 && a->ws_bytes < (int64_t)pl.S * a->M * w_rows * 4) pl = sk_plan(a->M, a->N, a->K, a->epilogue, false);
  const int S = pl.S;
  if (S <= 1 || !a->ws || a->ws_bytes < (int64_t)S * a->M * w_rows * 4) return P3V_ERR_UNSUPPORTED;
  if ((uintptr_t)a->ws & 15) return P3V_ERR_ARG;
  *S_out = S;
  const SkinnyP p = {a->A, a->W, a->ws, a->resid, a->M, a->N, a->K, a->lda, a->ldw, a->ldo, a->col_scale, a->K / S, {}, nullptr, nullptr, 0, 0};
  if (pl.tn == 96) return a->M <= 64 && !p3v_tuning().gemm_skinny_tm128 ? launch_skinny96<64>(p, S, s) : launch_skinny96<SK_BM>(p, S, s);
  if (silu) return launch_skinny<P3V_EPI_SILU_MUL>(p, S, s);                       // (partials: the activation is the reduction's)
  if (a->epilogue == P3V_EPI_RESID_BF16) return launch_skinny<P3V_EPI_RESID_BF16>(p, S, s);
  return launch_skinny<P3V_EPI_NONE>(p, S, s);
}

// P3V_ERR_UNSUPPORTED: not a shape for this kernel (the caller goes on to the other GEMM paths).  A split that finds no workspace of
// p3v_gemm_ws_bytes() runs as one pass.
int p3v_gemm_skinny_try(const p3v_gemm_args_t* a, hipStream_t s) {
  if (p3v_gemm_skinny_slices(a->M, a->N, a->K, a->epilogue) == 0) return P3V_ERR_UNSUPPORTED;
  if (p3v_gemm_rows_slices(a->M, a->N, a->K, a->epilogue) == 1) {                  // 9 .. 32 rows, one pass
    const int rr = p3v_gemm_rows_launch(a, nullptr, s);
    if (rr != P3V_ERR_UNSUPPORTED) return rr;
  }
  int S = 1;
  const int rc = p3v_gemm_skinny_partials(a, &S, s);
  if (rc == P3V_OK) return p3v_splitk_reduce((const float*)a->ws, a, S, s);
  if (rc != P3V_ERR_UNSUPPORTED) return rc;
  if (sk_slices(a->M, a->N, a->K, a->epilogue) == 0) return P3V_ERR_UNSUPPORTED;   // (a rows shape whose slices found no workspace and that the tile kernel does not take)
  const SkinnyP p = {a->A, a->W, a->out, a->resid, a->M, a->N, a->K, a->lda, a->ldw, a->ldo, a->col_scale, 0, {}, nullptr, nullptr, 0, 0};
  if (a->epilogue == P3V_EPI_SCALE_RESID_F32) return launch_skinny<P3V_EPI_SCALE_RESID_F32>(p, 1, s);
  if (a->epilogue == P3V_EPI_SILU_MUL) return launch_skinny<P3V_EPI_SILU_MUL>(p, 1, s);
  if (a->epilogue == P3V_EPI_GELU_MUL) return launch_skinny<P3V_EPI_GELU_MUL>(p, 1, s);
  if (a->epilogue == P3V_EPI_RESID_BF16) return launch_skinny<P3V_EPI_RESID_BF16>(p, 1, s);
  return launch_skinny<P3V_EPI_NONE>(p, 1, s);
}

// p3v_gemm without the workspace of its slices
int p3v_gemm_skinny_tall(const p3v_gemm_args_t* a, hipStream_t s) {
  if (a->bias || !sk_tall(a->M, a->N, a->K, a->epilogue)) return P3V_ERR_UNSUPPORTED;
  const SkinnyP p = {a->A, a->W, a->out, a->resid, a->M, a->N, a->K, a->lda, a->ldw, a->ldo, a->col_scale, 0, {}, nullptr, nullptr, 0, 0};
  return launch_skinny128<P3V_EPI_NONE>(p, a->N / 128, p3v_cdiv(a->M, SK_BM), s);
}

// ---- the qkv projection of a short prompt with the head split, the rotation and the KV append in the epilogue (p3v_gemm_qkv's
// 17 .. 256-row case): one pass (the epilogue needs whole sums), Q / K tiles + V tiles in a one-dimensional grid.
// P3V_ERR_UNSUPPORTED (nothing launched) where the shape is not this kernel's.
int p3v_gemm_skinny_qkv(const p3v_gemm_args_t* a, const QkvP& q, bool tall, hipStream_t s) {
  const P3vTuning& t = p3v_tuning();
  if (tall && (!sk_tall(a->M, a->N, a->K, P3V_EPI_NONE) || (q.nh * q.hd) % 128 || (q.nkv * q.hd) % 128)) return P3V_ERR_UNSUPPORTED;
  if (t.gemm_no_skinny || a->M <= 8 || (a->M > t.gemm_skinny_max_m && !tall) || a->K % SK_BK || a->bias) return P3V_ERR_UNSUPPORTED;
  if ((q.nh * q.hd) % 64 || (q.nkv * q.hd) % SK_BM) return P3V_ERR_UNSUPPORTED;   // whole Q / K tiles of 32 pairs, whole V tiles of 128 dims
  const SkinnyP p = {a->A, a->W, nullptr, nullptr, a->M, a->N, a->K, a->lda, a->ldw, 0, nullptr, 0, q, nullptr, nullptr, 0, 0};
  if ((q.nh * q.hd) % 128 == 0 && (q.nkv * q.hd) % 128 == 0 && (tall || sk_one_pass_tn(a->M, a->N) == 128))
    return launch_skinny128<P3V_EPI_QKV>(p, a->N / 128 * p3v_cdiv(a->M, SK_BM), 1, s);
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm_skinny<P3V_EPI_QKV, false, SK_TN>, hipFuncAttributeMaxDynamicSharedMemorySize, SkCfg<SK_TN>::LDS) != hipSuccess)
      return P3V_ERR_HIP;
    attr_set = true;
  }
  const int mt = p3v_cdiv(a->M, SK_BM), tiles = ((q.nh + q.nkv) * q.hd / 64) * mt + (q.nkv * q.hd / SK_BM) * p3v_cdiv(a->M, 64);
  hipLaunchKernelGGL((k_gemm_skinny<P3V_EPI_QKV, false, SK_TN>), dim3(tiles), dim3(512), SkCfg<SK_TN>::LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}

// ---- K slices that meet inside the launch: qkv of 17 .. 128 rows, gated projections of 105 .. 128.
// What these launches wait for is the bytes a CU requests, the A panel from L2 among them (the header), and qkv keeps only 144 CUs busy
// besides: on 128-column tiles a CU asks for half the A bytes per weight byte, and slices of K bring the workgroups back to one for
// (nearly) every CU.  Their fp32 sums through a launch of their own would cost what that gains; here the last slice's workgroup of a tile
// takes them over (k_gemm_skinny, MERGE).  It has a few K-tiles more than the others, while whose sums are under way (qkv 18 : 15 : 15 of
// 48; 16 each: 24.8 us, 20 : 14 : 14 23.5).  qkv 27.7 -> 22.4 us at 128 rows, 27.6 -> 19.0 at 64, 22.7 -> 18 at 17; gate_up 29.5 -> 26.9 at
// 128, 27.2 -> 26.3 at 112, 26.1 -> 26.1 at 104 (64 rows, on 64-row tiles of the one-pass form: 22.0 : 23.1).  Every slice finishing a
// share of the blocks instead: 26.8 and 30.9, the hand-over through memory then being behind everybody's products.
#define SK_MERGE_FLAGS 4096        // bytes of counters in front of the partials (zero before the first launch; every launch leaves them multiples of 4)
struct MergePlan { int S, nk_part, tiles; };
static MergePlan merge_plan(int M, int N, int K, int epilogue, bool qkv) {
  const MergePlan none = {0, 0, 0};
  const P3vTuning& t = p3v_tuning();
  const int rows = P3V_GATED(epilogue) ? 2 * N : N, nk = K / SK_BK, tiles = rows / 128;
  if (t.gemm_no_skinny || t.gemm_no_merge || M <= (qkv ? 16 : 104) || M > SK_BM || K % SK_BK || rows % 128 || N % 32) return none;
  if (!qkv && !P3V_GATED(epilogue)) return none;
  const int S = tiles ? 256 / tiles : 0;                         // one workgroup per CU
  if (S < 2 || S > 4 || nk < 8 * S || tiles * 4 * 4 > SK_MERGE_FLAGS) return none;
  return {S, (nk - (nk + 15) / 16) / S, tiles};
}
extern "C" int64_t p3v_gemm_merge_ws_bytes(int M, int N, int K, int epilogue, int qkv) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const MergePlan pl = merge_plan(M, N, K, epilogue, qkv != 0);
  return pl.S ? SK_MERGE_FLAGS + (int64_t)pl.tiles * (pl.S - 1) * (SK_BM * 128 * 4) : 0;
}
template <int EPI>
static int launch_merge(SkinnyP p, const MergePlan& pl, void* ws, hipStream_t s) {
  typedef SkCfg<128> C;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm_skinny<EPI, false, 128, SK_BM, true>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS) != hipSuccess) return P3V_ERR_HIP;
    attr_set = true;
  }
  p.xflag = (unsigned*)ws, p.xpart = (float*)((unsigned char*)ws + SK_MERGE_FLAGS), p.nk_part = pl.nk_part, p.polls = p3v_tuning().gemm_merge_polls < 0 ? 1u << 22 : (unsigned)p3v_tuning().gemm_merge_polls;
  hipLaunchKernelGGL((k_gemm_skinny<EPI, false, 128, SK_BM, true>), dim3(pl.tiles, 1, pl.S), dim3(512), C::LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}
static int merge_args(const p3v_gemm_args_t* a, const void* ws, int64_t ws_bytes, const MergePlan& pl) {
  if (!pl.S || !ws || ws_bytes < SK_MERGE_FLAGS + (int64_t)pl.tiles * (pl.S - 1) * (SK_BM * 128 * 4)) return P3V_ERR_UNSUPPORTED;
  if ((uintptr_t)ws & 15) return P3V_ERR_ARG;
  const size_t rows = (size_t)a->N * (P3V_GATED(a->epilogue) ? 2 : 1);
  return (size_t)a->M * a->lda * 2 >= (1ull << 32) || rows * a->ldw * 2 >= (1ull << 32) ? P3V_ERR_UNSUPPORTED : P3V_OK;
}
extern "C" int p3v_gemm_merge(const p3v_gemm_args_t* a, void* ws, int64_t ws_bytes, void* stream) {
  if (!a || !a->A || !a->W || !a->out || a->M <= 0 || a->N <= 0 || a->K <= 0 || a->K % SK_BK) return P3V_ERR_ARG;
  if (a->lda < a->K || a->ldw < a->K || a->lda % 8 || a->ldw % 8 || a->ldo % 8 || a->ldo < a->N) return P3V_ERR_ARG;
  if (((uintptr_t)a->A | (uintptr_t)a->W | (uintptr_t)a->out) & 15) return P3V_ERR_ARG;
  if (a->bias) return P3V_ERR_UNSUPPORTED;
  const MergePlan pl = merge_plan(a->M, a->N, a->K, a->epilogue, false);
  const int rc = merge_args(a, ws, ws_bytes, pl);
  if (rc != P3V_OK) return rc;
  const SkinnyP p = {a->A, a->W, a->out, nullptr, a->M, a->N, a->K, a->lda, a->ldw, a->ldo, nullptr, 0, {}, nullptr, nullptr, 0, 0};
  hipStream_t s = (hipStream_t)stream;
  return a->epilogue == P3V_EPI_GELU_MUL ? launch_merge<P3V_EPI_GELU_MUL>(p, pl, ws, s) : launch_merge<P3V_EPI_SILU_MUL>(p, pl, ws, s);
}
// p3v_gemm_qkv's case (p3v_gemm.hip has checked the call)
int p3v_gemm_skinny_qkv_merge(const p3v_gemm_args_t* a, const QkvP& q, void* ws, int64_t ws_bytes, hipStream_t s) {
  if (a->bias || (q.nh * q.hd) % 128 || (q.nkv * q.hd) % 128) return P3V_ERR_UNSUPPORTED;
  const MergePlan pl = merge_plan(a->M, a->N, a->K, P3V_EPI_NONE, true);
  const int rc = merge_args(a, ws, ws_bytes, pl);
  if (rc != P3V_OK) return rc;
  const SkinnyP p = {a->A, a->W, nullptr, nullptr, a->M, a->N, a->K, a->lda, a->ldw, 0, nullptr, 0, q, nullptr, nullptr, 0, 0};
  return launch_merge<P3V_EPI_QKV>(p, pl, ws, s);
}
