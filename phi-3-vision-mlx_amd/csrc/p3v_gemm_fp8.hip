// Prompts of the fp8 weight format: W8A8 projection on the gfx950 fp8 matrix cores.
//
//   C[M,N] = (sa[m] * sw[n]) * sum_k A8[m,k] * W8[n,k]        A8, W8 = OCP e4m3 bytes, K contiguous
//
// replaces the reference's QuantizedLinear call sites (phi_3_vision_mlx.py:264, 291-305) for prompt-sized inputs:
// weights are the per-output-row-scaled e4m3 bytes of `quantize_model=True` (the same bytes the decode GEMV streams),
// activations are quantised on the fly, one fp32 scale per token row (p3v_quant_fp8_rows, fused with the RMSNorm that
// precedes qkv_proj / gate_up_proj).
//
//   MFMA      v_mfma_scale_f32_16x16x128_f8f6f4 with both block scales = 1.0 (E8M0 0x7f): the only fp8 form that runs at
//             twice the bf16 rate on this chip (the unscaled 16x16x32 fp8 MFMA runs at the bf16 rate).  A lane holds 32
//             k bytes of its row (lane & 15) for k-block lane >> 4 -- the SAME bytes for A and B, so which k they are
//             does not matter (the kernel takes 16-byte chunks fchunk and fchunk + 4: bank-conflict-free reads).
//   tile      chosen by time (f8_tile_plan).  Flat ones, 128 or 160(M) x 256 / 192 / 128(N) x 128(K), and small ones: 768
//             threads: 8 CONSUMER waves as 2(M) x 4(N), ONE MFMA per 16 x 16 block and K-tile, and 4 PRODUCER waves that only
//             request K-tiles by LDS-DMA (as p3v_gemm_pc.hip): rows of 128 BYTES, 16-byte chunk c of row r stored at chunk
//             c ^ (r & 7), swizzled on the source address; three buffers of a K-tile (four from 128 x 192 down, up to eight of small ones: what
//             160 KiB hold), so a request has two or three K-tiles' time to land.  Tall ones, 192, 224 or 256 x 256, on FOUR waves that request and
//             multiply (k_gemm_f8_w4).
//             What bounds it: the requests, 60 ns per four 1-KiB pieces of a CU with the weights from memory, 40 with all of it in the L2s
//             (a K-tile of 192 x 256, 0.64 us of MFMAs, takes 0.81 - 0.85 and 0.73 where 12 - 60 CUs are at it), and, with all CUs at it, the
//             chip's power (0.97 - 1.03): the same launches on all-zero operands are 20-25 % faster.  The tall tiles against the flat ones, us, weights
//             from memory, launch behind launch: gate | up (16384 x 3072) 2300 rows
//             122 -> 93, 2531 124 -> 106, 4096 198 -> 164, 8192 367 -> 327 (2.5 PFLOP/s); 9216 x 3072 2531 rows 71 -> 61, 4096 106 -> 97; 3072 x 8192
//             3500 92 -> 69, 4096 99 -> 79; 3072 x 3072 4096 50 -> 37.  One round of flat tiles that fills the chip stays ahead of one of tall ones
//             that does not: 3072 x 8192 at 2531 rows 59 (128 rows), 62 (192).
//             Some hundred rows leave most CUs without a 128 x 128 tile, and no slices of K can bring them in (another order of the sums would reach the next
//             row quantiser).  Tiles of 32 x 64, 64 x 64, 64 x 128 and 96 x 128 do: a K-tile of 12 - 28 KB is 0.23 - 0.45 us of a CU's requests instead of
//             0.5, with up to eight buffers of it in flight.  us, 128 x 128 -> the small one: 3072 x 8192 137 rows 31.0 -> 18.0 (32 x 64), 276 31.2 -> 21.5
//             (64 x 64), 512 39.3 -> 30.1 (64 x 128), 803 33.2 -> 32.9 (96 x 128); 3072 x 3072 137 rows 15.1 -> 9.1, 276 15.5 -> 11.2; 9216 x 3072 137 rows 15.9
//             -> 14.2; gate | up 128 rows 23.0 -> 20.1.  Tiles of 96 x 64 and 128 x 64 are hardly ever the fastest, by 3 % then.
//   epilogue  scales, then none / residual add / SiLU(gate) * up, bf16 out, straight from the accumulators (p3v_gemm256_epi.h).
#include <stdlib.h>

#include <type_traits>

#include "p3v_gemm_qkv.h"

#define P3V_EPI_QKV 100                // internal: the qkv projection with split + RoPE + KV append in the epilogue (p3v_gemm_qkv.h)
#define TKB 128                        // K bytes (= fp8 elements) per K-tile

typedef __attribute__((address_space(3))) void* lptr_t;
typedef __attribute__((ext_vector_type(8))) int i32x8_t;

struct GemmF8P {
  const uint8_t* A; const float* sa; const uint8_t* W; const float* sw; bf16_t* out; const bf16_t* resid;
  int M, N, K, lda, ldw, ldo;
  QkvP q;                              // P3V_EPI_QKV only
};
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));   // (scales: any float address)

struct PlaceF8 { int m0, n0, swapped, is_k, row0; };             // P3V_EPI_QKV: V tile (operand roles swapped) / K region / first W row of the region
struct TileF8 { int a_off[8], b_off[8]; __amdgpu_buffer_rsrc_t rs_a, rs_b; };   // where the requests of an output tile's K-tiles come from

#define F8_BUF(mb, nb) ((32 * (mb) + 64 * (nb)) * TKB)
#define F8_STAGES(mb, nb) f8_stages(160 * 1024 / F8_BUF(mb, nb), F8_BUF(mb, nb))
constexpr int f8_stages(int fit, int buf) { return buf >= 32 * 1024 ? (fit < 4 ? fit : 4) : fit < 8 ? fit : 8; }

// s_waitcnt vmcnt(PER n): all but the n youngest K-tiles of PER requests each have landed
template <int PER>
__device__ __forceinline__ void f8_wait(int n) {
#define F8_WAIT(k) case k: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(k * PER < 63 ? k * PER : 63) : "memory"); break;
  switch (n) {
    F8_WAIT(1) F8_WAIT(2) F8_WAIT(3) F8_WAIT(4) F8_WAIT(5) F8_WAIT(6) F8_WAIT(7)
    default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
#undef F8_WAIT
}

// A wave's 16 MB x 16 NB sums at rows mrow0 - fc .., outputs from column nw on, straight from the accumulators: lane (fc = lane & 15, fq = lane >> 4)
// holds columns 4 fq .. 4 fq + 3 of block row fc; lanes q and q ^ 1 trade packed halves of two neighbouring column blocks: 16-byte stores.
template <int EPI, int MB, int NB>
__device__ __forceinline__ void f8_epilogue(const GemmF8P& p, const f32x4_t (&acc)[MB][NB], int mrow0, int nw, int fq) {
  constexpr bool SILU = EPI == P3V_EPI_SILU_MUL;
  constexpr int HB = SILU ? NB / 2 : NB;                           // column blocks of outputs of a wave
  float sc[NB][4];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = SILU ? nw + j % HB * 16 + fq * 4 + j / HB * p.N : nw + j * 16 + fq * 4;
    const f32x4_a4 c = *(const f32x4_a4*)(p.sw + n);
    sc[j][0] = c[0], sc[j][1] = c[1], sc[j][2] = c[2], sc[j][3] = c[3];
  }
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int m = mrow0 + i * 16;
    const float s = p.sa[min(m, p.M - 1)];
    uint32_t pk[HB][2];
#pragma unroll
    for (int j = 0; j < HB; ++j) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = acc[i][j][r] * (s * sc[j][r]);
        if (SILU) {
          // gate / up are bf16 Linear outputs, every elementwise op after them rounds to bf16 (phi.py:469-471)
          const float g = bf16_round(v[r]), u = bf16_round(acc[i][(HB + j) % NB][r] * (s * sc[(HB + j) % NB][r]));
          v[r] = bf16_round(g * bf16_round(1.f / (1.f + __expf(-g)))) * u;
        }
      }
      pk[j][0] = pack_bf16x2(v[0], v[1]), pk[j][1] = pack_bf16x2(v[2], v[3]);
    }
#pragma unroll
    for (int jp = 0; jp < HB / 2; ++jp) {
      u32x4_t w;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        auto sw = __builtin_amdgcn_permlane16_swap(pk[2 * jp][k], pk[2 * jp + 1][k], false, false);
        w[k] = sw[0], w[2 + k] = sw[1];
      }
      const int n = nw + (2 * jp + (fq & 1)) * 16 + (fq >> 1) * 8;
      if (m < p.M) {
        const size_t o = (size_t)m * p.ldo + n;
        if (EPI == P3V_EPI_RESID_BF16) {
          const u32x4_t rw = *(const u32x4_t*)(p.resid + o);
#pragma unroll
          for (int k = 0; k < 4; ++k) w[k] = pack_bf16x2(bf16lo(rw[k]) + bf16lo(w[k]), bf16hi(rw[k]) + bf16hi(w[k]));
        }
        *(u32x4_t*)(p.out + o) = w;
      }
    }
    if (HB & 1) {                                     // the block without a partner: four columns, 8 bytes
      const int n = nw + (HB - 1) * 16 + fq * 4;
      if (m < p.M) {
        const size_t o = (size_t)m * p.ldo + n;
        u32x2_t w = {pk[HB - 1][0], pk[HB - 1][1]};
        if (EPI == P3V_EPI_RESID_BF16) {
          const u32x2_t rw = *(const u32x2_t*)(p.resid + o);
#pragma unroll
          for (int k = 0; k < 2; ++k) w[k] = pack_bf16x2(bf16lo(rw[k]) + bf16lo(w[k]), bf16hi(rw[k]) + bf16hi(w[k]));
        }
        *(u32x2_t*)(p.out + o) = w;
      }
    }
  }
}

// MB, NB: 16-row / 16-column blocks of a consumer wave (2 x 4 waves: a tile of 32 MB rows x 64 NB columns)
template <int EPI, int MB, int NB>
__global__ void __launch_bounds__(768, 1) k_gemm_f8(GemmF8P p) {
  constexpr bool SILU = EPI == P3V_EPI_SILU_MUL, QKV = EPI == P3V_EPI_QKV;
  static_assert(!QKV || NB == 4, "both halves of 32 rotation pairs in a wave");
  static_assert(NB % 2 == 0 || !SILU, "a wave's column blocks: gate, then up of the same outputs");
  constexpr int HB = SILU ? NB / 2 : NB;                           // column blocks of outputs of a wave
  constexpr int TM = 32 * MB, TN = 64 * NB, A_BYTES = TM * TKB, BUF_BYTES = F8_BUF(MB, NB);
  constexpr int S = F8_STAGES(MB, NB), PER = MB + 2 * NB;          // LDS buffers; requests of a producer wave per K-tile
  static_assert(S >= 3 && S <= 8 && (S - 1) * PER < 64, "f8_wait");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int n_out_tile = SILU ? TN / 2 : TN;
  // (QKV: column tiles 0 .. nq - 1 are Q, the others K; behind them the V tiles, TM rows of W_v by TN tokens)
  const int nq = QKV ? p.q.nh * p.q.hd / TN : 0;
  const int gx = QKV ? nq + p.q.nkv * p.q.hd / TN : p.N / n_out_tile, gy = (p.M + TM - 1) / TM;
  const int vx = QKV ? (p.M + TN - 1) / TN : 0, vy = QKV ? p.q.nkv * p.q.hd / TM : 0, nwg = gx * gy + vx * vy;
  const int nk = p.K / TKB;

  // persistent over output tiles, XCD-aware order (as p3v_gemm_pc.hip): each XCD gets a contiguous run of tiles, bands of 4 M tiles
  auto place = [&](int wid) {
    const int q = nwg >> 3, r = nwg & 7, xcd = wid & 7, loc = wid >> 3;
    int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + loc;
    const bool v = QKV && id >= gx * gy;
    if (v) id -= gx * gy;
    const int cx = v ? vx : gx, cy = v ? vy : gy;
    constexpr int BAND = 4;
    const int band = id / (BAND * cx), in_band = id % (BAND * cx);
    const int rows = min(BAND, cy - band * BAND);
    const int y = band * BAND + in_band % rows, x = in_band / rows;
    PlaceF8 t = {y * TM, x * n_out_tile, 0, 0, 0};
    if (v) t = {x * TN, y * TM, 1, 0, (p.q.nh + p.q.nkv) * p.q.hd};          // first token, first row of the V region
    else if (QKV && x >= nq) t.is_k = 1, t.n0 -= nq * TN, t.row0 = p.q.nh * p.q.hd;
    return t;
  };
  if ((int)blockIdx.x >= nwg) return;
  const int n_mine = (nwg - 1 - (int)blockIdx.x) / (int)gridDim.x + 1, total = n_mine * nk;      // output tiles, K-tiles of this workgroup

  if (wave >= 8) {
    // ---- PRODUCERS (p3v_gemm_pc.hip)
    const int pw = wave - 8, srow = pw * 8 + (lane >> 3), sw = ((lane & 7) ^ (lane >> 3)) * 16;
    TileF8 dt;    // (declared outside the template: a builtin called with a member of a DEPENDENT type is only checked at
                  //  instantiation, fails there in the HOST pass -- no such builtin -- and hipcc silently drops the host stub)
    auto aim = [&](int wid) {
      const PlaceF8 t = place(wid);
      const int m0 = t.m0, n0 = t.n0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int rr = q * 32 + srow;
        int br = QKV ? qkv_pair_row(p.q, t.row0, n0 >> 1, rr) : min(n0 + rr, p.N - 1);
        if (SILU) {                                               // a wave's 16 HB gate rows + the 16 HB up rows of the same outputs
          const int in = rr % (NB * 16);
          br = n0 + rr / (NB * 16) * (HB * 16) + in % (HB * 16) + in / (HB * 16) * p.N;
        }
        dt.a_off[q] = (min(m0 + rr, p.M - 1) - m0) * p.lda + sw;
        dt.b_off[q] = (int)((unsigned)br * (unsigned)p.ldw + (unsigned)sw);
        if (QKV && t.swapped) {                                   // W rows fill the A side, tokens the B side
          dt.a_off[q] = rr * p.ldw + sw;
          dt.b_off[q] = (int)((unsigned)min(m0 + rr, p.M - 1) * (unsigned)p.lda + (unsigned)sw);
        }
      }
      const uint8_t* pa = QKV && t.swapped ? p.W + (size_t)(t.row0 + n0) * p.ldw : p.A + (size_t)m0 * p.lda;
      const uint8_t* pb = QKV && t.swapped ? p.A : p.W;
      dt.rs_a = __builtin_amdgcn_make_buffer_rsrc((void*)pa, 0, 0xffffffff, 0x00020000);
      dt.rs_b = __builtin_amdgcn_make_buffer_rsrc((void*)pb, 0, 0xffffffff, 0x00020000);
    };
    int dwid = blockIdx.x, dk = 0, slot = 0;                      // the next K-tile to request, and its buffer
    aim(dwid);
    auto request = [&]() {
      unsigned char* base = smem + slot * (int)BUF_BYTES + pw * 1024;
      const int na = MB, nb = 2 * NB, a_bytes = A_BYTES;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (q < na) {
          lptr_t dst = (lptr_t)(base + q * 4096);
          const int vo = dt.a_off[q];
          __builtin_amdgcn_raw_ptr_buffer_load_lds(dt.rs_a, dst, 16, vo, dk * TKB, 0, 0);
        }
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (q < nb) {
          lptr_t dst = (lptr_t)(base + a_bytes + q * 4096);
          const int vo = dt.b_off[q];
          __builtin_amdgcn_raw_ptr_buffer_load_lds(dt.rs_b, dst, 16, vo, dk * TKB, 0, 0);
        }
      }
      slot = slot == S - 1 ? 0 : slot + 1;
      if (++dk == nk) {
        dk = 0;
        dwid += gridDim.x;
        if (dwid < nwg) aim(dwid);
      }
    };
    for (int g = 0; g < min(S, total); ++g) request();
    for (int g = 0; g < total; ++g) {
      // K-tile g has landed when only the younger ones' requests are out: S - 1 of them at first, then S - 2, fewer at the end
      f8_wait<PER>(min(g == 0 ? S - 1 : S - 2, total - 1 - g));
      __builtin_amdgcn_s_barrier();                               // K-tile g is there; K-tile g - 1 is in the consumers' registers
      if (g > 0 && g - 1 + S < total) request();
    }
    return;
  }

  // ---- CONSUMERS.  One MFMA takes a whole K-tile of a 16 x 16 block, so a K-tile is cut by rows: while the first M0 row blocks are
  // multiplied the other M1 are fetched (then all of it is in registers and its buffer is given back), while those are multiplied
  // column by column the next K-tile's first row blocks and, behind each column, its new fragment are.
  constexpr int M0 = (MB + 1) / 2, M1 = MB - M0;
  const int wr = wave >> 2, wc = wave & 3;
  const int frow = lane & 15, fchunk = lane >> 4;
  // lane (row frow, k-block fchunk) owns the 16-byte chunks fchunk and fchunk + 4 of its 128-byte row (A and B alike, so the k
  // permutation cancels; contiguous chunks would put the 16 lanes of a ds_read_b128 group on 8 bank slots)
  const int fo0 = frow * 128 + ((fchunk ^ (frow & 7)) << 4), fo1 = frow * 128 + (((4 + fchunk) ^ (frow & 7)) << 4);
  f32x4_t acc[MB][NB];
  i32x8_t fa[MB], fb[NB];
  auto fetch = [&](i32x8_t& f, const unsigned char* t) {
    const u32x4_t lo = *(const u32x4_t*)(t + fo0), hi = *(const u32x4_t*)(t + fo1);
    f = (i32x8_t){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
  };
  auto fetch_a = [&](int i, int buf) { fetch(fa[i], smem + buf * BUF_BYTES + (wr * MB + i) * 2048); };
  auto fetch_b = [&](int j, int buf) { fetch(fb[j], smem + buf * BUF_BYTES + A_BYTES + (wc * NB + j) * 2048); };
  auto mma = [&](int i, int j) {                                  // (W fragment first: the block comes out TRANSPOSED, see the epilogue)
    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j], fa[i], acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
  };
  int slot = 0;                                                   // LDS buffer of the K-tile in hand
  __builtin_amdgcn_s_barrier();
  for (int wid = blockIdx.x; wid < nwg; wid += gridDim.x) {
    const PlaceF8 at = place(wid);
    const int m0 = at.m0, n0 = at.n0;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < M0; ++i) fetch_a(i, slot);
#pragma unroll
    for (int j = 0; j < NB; ++j) fetch_b(j, slot);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt) {
      const int nslot = slot == S - 1 ? 0 : slot + 1;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
#pragma unroll
        for (int i = 0; i < M0; ++i) mma(i, j);
        if (j == 0) {
#pragma unroll
          for (int i = 0; i < M1; ++i) fetch_a(M0 + i, slot);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // the K-tile in hand is in registers: its buffer is given back
      if (kt + 1 < nk || wid + (int)gridDim.x < nwg) __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        if (j == 0) {
#pragma unroll
          for (int i = 0; i < M0; ++i) fetch_a(i, nslot);
        }
#pragma unroll
        for (int i = 0; i < M1; ++i) mma(M0 + i, j);
        __builtin_amdgcn_sched_barrier(0);
        fetch_b(j, nslot);
        __builtin_amdgcn_sched_barrier(0);
      }
      slot = nslot;
    }

    const int fc = lane & 15, fq = lane >> 4;
    if constexpr (QKV) {                                           // the same products of sum and scales, then p3v_gemm_qkv's epilogues
      if (at.swapped) {
        float st[4][4], sr[MB];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) st[j][r] = p.sa[min(m0 + wc * 64 + j * 16 + fq * 4 + r, p.M - 1)];
#pragma unroll
        for (int i = 0; i < MB; ++i) sr[i] = p.sw[at.row0 + n0 + (wr * MB + i) * 16 + fc];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] *= st[j][r] * sr[i];
        qkv_epilogue_vt<MB>(p.q, acc, nullptr, n0 + wr * MB * 16, m0 + wc * 64, p.M, lane);
      } else {
        f32x4_a4 sc[4];
        float st[MB];
#pragma unroll
        for (int j = 0; j < 4; ++j) sc[j] = *(const f32x4_a4*)(p.sw + qkv_pair_row(p.q, at.row0, n0 >> 1, wc * 64 + j * 16 + fq * 4));
#pragma unroll
        for (int i = 0; i < MB; ++i) st[i] = p.sa[min(m0 + (wr * MB + i) * 16 + fc, p.M - 1)];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] *= st[i] * sc[j][r];
        static_assert(!QKV || MB % 2 == 0, "");
#pragma unroll
        for (int i = 0; i < MB; i += 2) {                          // (two block rows' table values at a time: the registers of twelve waves)
          f32x4_t part[2][4];
#pragma unroll
          for (int j = 0; j < 4; ++j) part[0][j] = acc[i][j], part[1][j] = acc[i + 1][j];
          qkv_epilogue_rot<2>(p.q, part, nullptr, at.is_k, at.row0, (n0 >> 1) + wc * 32, m0 + (wr * MB + i) * 16, p.M, lane);
        }
      }
      continue;
    }
    f8_epilogue<EPI, MB, NB>(p, acc, m0 + wr * MB * 16 + fc, n0 + wc * (n_out_tile / 4), fq);
  }
}

// A wave's sums of 64 columns of W (column group g of NG; SiLU: 32 gate, then the 32 up rows of the same outputs) at rows m0 .., outputs from n0 on:
// as f8_epilogue, in one straight line (p3v_gemm256_epi.h: buffer stores whose bounds check drops the rows beyond M; the sums stay in
// accumulation registers until their row's turn; scales and residual rows are requested ahead, one wave per SIMD has nobody to cover for it).
template <int EPI, int MB, int NG>
__device__ __forceinline__ void f8_epilogue_w4(const GemmF8P& p, f32x4_t (&acc)[NG][MB][4], int m0, int n0, int lane) {
  constexpr bool SILU = EPI == P3V_EPI_SILU_MUL, RESID = EPI == P3V_EPI_RESID_BF16;
  constexpr int NOUT = SILU ? 32 : 64;                             // outputs of a group
  const int fc = lane & 15, fq = lane >> 4;
  float s[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) s[i] = p.sa[min(m0 + fc + i * 16, p.M - 1)];
  f32x4_t sc[NG][4];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int j = 0; j < 4; ++j) sc[g][j] = *(const f32x4_a4*)(p.sw + n0 + g * NOUT + (SILU ? j % 2 * 16 + j / 2 * p.N : j * 16) + fq * 4);
  const size_t first = ((size_t)m0 * p.ldo + n0) * 2;
  const __amdgpu_buffer_rsrc_t rs_o = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)p.out + first, 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_r = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)p.resid + (RESID ? first : 0), 0, 0x7fffffff, 0x00020000);
  auto at = [&](int i) { return m0 + fc + i * 16 < p.M ? (fc + i * 16) * p.ldo * 2 + ((fq & 1) * 16 + (fq >> 1) * 8) * 2 : (int)0x80000000; };
  constexpr int TURNS = NG * MB, RN = 6;
  u32x4_t rw[RESID ? RN : 1][2];
  auto ask = [&](int t) {
    if constexpr (RESID)
#pragma unroll
      for (int jp = 0; jp < 2; ++jp) rw[t % RN][jp] = __builtin_amdgcn_raw_buffer_load_b128(rs_r, at(t % MB) + t / MB * NOUT * 2 + jp * 64, 0, 0);
  };
#pragma unroll
  for (int t = 0; t < RN; ++t) ask(t);
#pragma unroll
  for (int t = 0; t < TURNS; ++t) {
    const int g = t / MB, i = t % MB;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+a"(acc[g][i][j]));
    float v[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[j][r] = acc[g][i][j][r] * (s[i] * sc[g][j][r]);
    uint32_t pk[4][2];
    constexpr int NJ = SILU ? 2 : 4;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        pk[j][h] = SILU ? p3v_gated2(EPI, v[j][2 * h], v[j][2 * h + 1], v[(2 + j) % 4][2 * h], v[(2 + j) % 4][2 * h + 1]) : pack_bf16x2(v[j][2 * h], v[j][2 * h + 1]);
#pragma unroll
    for (int jp = 0; jp < NJ / 2; ++jp) {
      u32x4_t w;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        auto sw = __builtin_amdgcn_permlane16_swap(pk[2 * jp][k], pk[2 * jp + 1][k], false, false);
        w[k] = sw[0], w[2 + k] = sw[1];
      }
      if constexpr (RESID)
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = pack_bf16x2(bf16lo(rw[t % RN][jp][k]) + bf16lo(w[k]), bf16hi(rw[t % RN][jp][k]) + bf16hi(w[k]));
      __builtin_amdgcn_raw_buffer_store_b128(w, rs_o, at(i) + g * NOUT * 2 + jp * 64, 0, 0);
    }
    if (t + RN < TURNS) ask(t + RN);
  }
}

// Tall tiles: 256, 224 or 192 rows x 256 columns on FOUR waves of 16 MB x 128 outputs, one per SIMD, that request and multiply (p3v_gemm256.hip's form).
// The eight consumers of the flat tiles keep the LDS busy for more cycles than their MFMAs take (160 x 256: 1531 against 1288 a K-tile, reads and
// DMA); these read 4 MFMAs' worth a fragment: 1536 of 2061.  One MFMA takes a whole K-tile of a block, and both operands' fragments of one K-tile
// fill 128 registers, so a K-tile is multiplied column block by column block: its W fragments arrive as they are needed (the first two a K-tile
// early), A's, all of the next K-tile, in the second register set meanwhile.  The sets change places with every K-tile: the loop takes two; an odd
// last one moves the second set into the first, 64 moves an output tile (1300 x 9216 x 3200 48 us on the flat tiles, 34 here; gate | up of 2048
// rows, K = 2944: 102, 80).  One barrier per K-tile, behind its last W fragment; from there on until the next one a request every few MFMAs, A two K-tiles
// ahead, W three.
struct AimF8 { int a_off[8], b_off[8]; __amdgpu_buffer_rsrc_t rs_a, rs_b; };     // (declared outside the template: see TileF8's use)
template <int EPI, int MB>
__global__ void __launch_bounds__(256, 1) k_gemm_f8_w4(GemmF8P p) {
  constexpr bool SILU = EPI == P3V_EPI_SILU_MUL;
  constexpr int NB = 8, NG = 2, TM = 32 * MB, TN = 256, A_BYTES = TM * TKB, B_BYTES = TN * TKB, B0 = 2 * A_BYTES;    // LDS: two buffers of A, three of W
  constexpr int NM = MB * NB, NF = MB + NB;                        // MFMAs and requests of a K-tile
  constexpr int TURN = 2 * (NB - 2) + 4, STEP = (NM - TURN - 2) / NF;                              // where buffers change hands; MFMAs per request behind it
  constexpr bool ZERO = MB == 8;                                   // (the allocator spills the sums if they start in the first MFMAs)
  static_assert(STEP >= 2 && 2 * MB <= TURN && NM - TURN - 1 >= 4 + 2 * MB, "");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 1, wc = wave & 1;
  constexpr int n_out_tile = SILU ? TN / 2 : TN;
  const int gx = p.N / n_out_tile, gy = (p.M + TM - 1) / TM, nwg = gx * gy, nk = p.K / TKB;
  auto place = [&](int wid) {                                      // persistent, XCD-aware order, as above
    const int q = nwg >> 3, r = nwg & 7, xcd = wid & 7, loc = wid >> 3;
    const int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + loc;
    constexpr int BAND = 4;
    const int band = id / (BAND * gx), in_band = id % (BAND * gx), rows = min(BAND, gy - band * BAND);
    const PlaceF8 t = {(band * BAND + in_band % rows) * TM, in_band / rows * n_out_tile, 0, 0, 0};
    return t;
  };
  const int sw = ((tid & 7) ^ ((tid >> 3) & 7)) * 16;
  AimF8 aim;
  int wa = blockIdx.x, ka = 0, wb = blockIdx.x, kb = 0;            // the K-tiles to be requested next: output tile, K
  auto aim_a = [&]() {
    const PlaceF8 t = place(wa);
    int srow = tid >> 3;                                           // (opaque: what follows from it is not to be held through the K loop)
    asm volatile("" : "+v"(srow));
#pragma unroll
    for (int q = 0; q < MB; ++q) aim.a_off[q] = (min(t.m0 + q * 32 + srow, p.M - 1) - t.m0) * p.lda + sw;
    aim.rs_a = __builtin_amdgcn_make_buffer_rsrc((void*)(p.A + (size_t)t.m0 * p.lda), 0, 0xffffffff, 0x00020000);
  };
  auto aim_b = [&]() {
    const PlaceF8 t = place(wb);
    int srow = tid >> 3;
    asm volatile("" : "+v"(srow));
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int rr = q * 32 + srow, in = rr & 63;
      const int br = SILU ? t.n0 + (rr >> 6) * 32 + (in & 31) + (in >> 5) * p.N : t.n0 + rr;   // (SiLU: 32 gate rows + the 32 up rows of the same outputs)
      aim.b_off[q] = (int)((unsigned)br * (unsigned)p.ldw + (unsigned)sw);
    }
    aim.rs_b = __builtin_amdgcn_make_buffer_rsrc((void*)p.W, 0, 0xffffffff, 0x00020000);
  };
  // (behind the last K-tile the requests repeat it: every K-tile has the same number of them, and the counted waits hold to the end)
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
  auto request = [&](int n, int as, int bs) {
    if (n < MB) {
      lptr_t dst = (lptr_t)(smem + as + n * 4096 + wave * 1024);
      const int vo = aim.a_off[n & 7];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(aim.rs_a, dst, 16, vo, ka * TKB, 0, 0);
    } else {
      lptr_t dst = (lptr_t)(smem + (int)B0 + bs + (n - (int)MB) * 4096 + wave * 1024);
      const int vo = aim.b_off[(n - (int)MB) & 7];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(aim.rs_b, dst, 16, vo, kb * TKB, 0, 0);
    }
  };
  int wid = blockIdx.x;
  if (wid >= nwg) return;
  aim_a(), aim_b();
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int n = 0; n < NF; ++n) request(n, t * A_BYTES, t * B_BYTES);
    next_a(), next_b();
  }
#pragma unroll
  for (int n = MB; n < NF; ++n) request(n, 0, 2 * B_BYTES);
  next_b();

  const int frow = lane & 15, fchunk = lane >> 4;
  const int fo0 = frow * 128 + ((fchunk ^ (frow & 7)) << 4);       // (chunks fchunk and fchunk + 4 of the row, as above)
  int as = 0, bs = 0;                                              // the buffers of the K-tile in hand
  f32x4_t acc[NG][MB][4];
  i32x8_t fa[2][MB], fb[NB];
  auto half = [&](i32x8_t& f, int h, const unsigned char* t) {     // a half of a fragment
    const u32x4_t v = *(const u32x4_t*)(t + (fo0 ^ (h * 64)));
#pragma unroll
    for (int k = 0; k < 4; ++k) f[4 * h + k] = (int)v[k];
  };
  auto read_b = [&](int n, int bs) { half(fb[n >> 1], n & 1, smem + B0 + bs + wc * (NB * 2048) + (n >> 1) * 2048); };
  auto read_a = [&](i32x8_t (&f)[MB], int n, int as) { half(f[n >> 1], n & 1, smem + as + wr * (MB * 2048) + (n >> 1) * 2048); };
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NF + NB) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int n = 0; n < 4; ++n) read_b(n, 0);
#pragma unroll
  for (int n = 0; n < 2 * MB; ++n) read_a(fa[0], n, 0);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NB) : "memory");
  for (;;) {
    const PlaceF8 t = place(wid);
    bool first_pair = true;
    auto k_tile = [&](auto first, auto odd) {                      // (first of an output tile: the sums start here, and the next K-tile has been waited for)
      constexpr bool FIRST = decltype(first)::value;
      constexpr int P = decltype(odd)::value;
      const int an = as ^ A_BYTES, bn = bs == 2 * B_BYTES ? 0 : bs + B_BYTES;
      auto mma = [&](int m) {                                      // (W fragment first: the block comes out TRANSPOSED)
        const int j = m / MB, i = m % MB;
        f32x4_t& c = acc[j / 4][i][j % 4];
        c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j], fa[P][i], FIRST ? (f32x4_t){0.f, 0.f, 0.f, 0.f} : c, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
        __builtin_amdgcn_sched_barrier(0);
      };
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < TURN; ++m) {
        if (m < 2 * (NB - 2)) read_b(4 + m, bs);
        mma(m);
      }
      // the next K-tile is in LDS, this one in registers: its buffers are given back
      if (!(ZERO && P == 0 ? first_pair : FIRST)) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NB) : "memory");
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int m = TURN; m < NM; ++m) {
        if (m > TURN) {                                            // the next K-tile's first two fragments of W, and all of A's
          const int n = m - TURN - 1;
          if (n < 4) read_b(n, bn);
          else if (n < 4 + 2 * MB) read_a(fa[1 - P], n - 4, an);
        }
        if (m >= TURN + 2 && (m - TURN - 2) % STEP == 0 && (m - TURN - 2) / STEP < NF) request((m - TURN - 2) / STEP, as, bs);
        mma(m);
      }
      // (an MFMA has no side effects: without this the first K-tile's are moved down, behind the branches, to where the second one's need them)
#pragma unroll
      for (int m = 0; m < NM; ++m) asm volatile("" : "+a"(acc[m / MB / 4][m % MB][m / MB % 4]));
      next_a(), next_b();
      as = an, bs = bn;
    };
    if constexpr (ZERO)
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        acc[m / MB / 4][m % MB][m / MB % 4] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[m / MB / 4][m % MB][m / MB % 4]));
      }
    if constexpr (!ZERO) {
      k_tile(std::true_type{}, std::integral_constant<int, 0>{});
      k_tile(std::false_type{}, std::integral_constant<int, 1>{});
    }
#pragma unroll 1
    for (int kt = ZERO ? 0 : 2; kt + 1 < nk; kt += 2) {
      k_tile(std::false_type{}, std::integral_constant<int, 0>{});
      k_tile(std::false_type{}, std::integral_constant<int, 1>{});
      first_pair = false;
    }
    if (nk & 1) {                                                  // the next output tile starts in the first register set again
      k_tile(std::false_type{}, std::integral_constant<int, 0>{});
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[0][i] = fa[1][i];
    }
    // (what the next K-tile's turn waits for, waited for ahead of the epilogue's stores, which the same counter counts)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NB) : "memory");
    int lane_e = lane;                                             // (opaque, as in aim_a)
    asm volatile("" : "+v"(lane_e));
    f8_epilogue_w4<EPI, MB, NG>(p, acc, t.m0 + wr * MB * 16, t.n0 + wc * (n_out_tile / 2), lane_e);
    if (wid + (int)gridDim.x >= nwg) break;
    wid += gridDim.x;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                 // (the requests that repeat the last K-tile: LDS is given back behind them)
}
int p3v_gemm256_cus();                                             // p3v_gemm256.hip

template <int EPI, int MB>
static int launch_f8_w4(const GemmF8P& p, hipStream_t s) {
  constexpr int LDS = (2 * 32 * MB + 3 * 256) * TKB;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm_f8_w4<EPI, MB>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return P3V_ERR_HIP;
    attr_set = true;
  }
  const int n_cu = p3v_gemm256_cus();
  if (!n_cu) return P3V_ERR_HIP;
  const int tiles = p.N / (EPI == P3V_EPI_SILU_MUL ? 128 : 256) * p3v_cdiv(p.M, 32 * MB);
  hipLaunchKernelGGL((k_gemm_f8_w4<EPI, MB>), dim3(min(tiles, n_cu)), dim3(256), LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}

template <int EPI, int MB, int NB>
static int launch_f8_v(const GemmF8P& p, hipStream_t s) {
  constexpr int LDS = F8_STAGES(MB, NB) * F8_BUF(MB, NB);
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k_gemm_f8<EPI, MB, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return P3V_ERR_HIP;
    attr_set = true;
  }
  const int n_cu = p3v_gemm256_cus();
  if (!n_cu) return P3V_ERR_HIP;
  int tiles = p.N / (EPI == P3V_EPI_SILU_MUL ? 32 * NB : 64 * NB) * p3v_cdiv(p.M, 32 * MB);
  if (EPI == P3V_EPI_QKV) tiles = (p.q.nh + p.q.nkv) * p.q.hd / (64 * NB) * p3v_cdiv(p.M, 32 * MB) + p.q.nkv * p.q.hd / (32 * MB) * p3v_cdiv(p.M, 64 * NB);
  hipLaunchKernelGGL((k_gemm_f8<EPI, MB, NB>), dim3(min(tiles, n_cu)), dim3(768), LDS, s, p);
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}

// The tile that takes least time, which is returned (us).  t K-tiles, r rounds of which u are filled (a fuller chip runs slower: power, and the outputs'
// way to memory): once + r (f + c t) + u (fill t + out), a gated or residual epilogue's more per round; fitted to 24 heights, 128 .. 9809 rows, of 15
// projections of K = 256 .. 8192 (even and odd numbers of K-tiles) with their weights from memory (4 - 8 % of a time; profiles/gemm_fp8_tile_sweep.txt).  What it
// names is 0.2 % slower than the fastest of the seven on average over those 360 sizes, 6.8 % at most (with each projection's own times left out of the
// fit: the same).  The fit to K = 3072 and 8192 alone that this one replaces: 1.4 %, 20 % at most, at short K (4096 x 384, 1300 rows 9.8 -> 8.9 us; 9216 x 3072,
// 1024 rows 31.3 -> 29.9); rounds alone: 7.7 % at K = 3072 and 8192.
// The four small tiles are fitted to 14 heights, 64 .. 1300 rows, of the same projections (the second table there): what the plan names is 0.8 % slower than
// the fastest of eleven on average, 25 % at most (803 x 9216 x 640 as before them), and 17.5 % faster than the fastest of seven (3 % slower at most).
static int f8_cus() { const int n = p3v_gemm256_cus(); return n ? n : 256; }     // (no device: host queries)
struct F8Tile { int mb, nb; float once, f, gated, resid, c, fill, out; };
static float f8_tile_plan(int M, int N, int K, int ldo, int epilogue, int& mb, int& nb) {
  static const F8Tile tiles[] = {{4, 4, 4.82f, 0.1f, 1.75f, 1.45f, 0.779f, 0.023f, 2.48f},  {5, 4, 5.01f, 0.71f, 2.18f, 1.85f, 0.804f, 0.103f, 2.57f},
                                 {4, 3, 5.72f, 0.42f, 0.f, 1.64f, 0.569f, 0.054f, 1.86f},   {4, 2, 3.87f, 0.21f, 0.76f, 0.72f, 0.492f, 0.017f, 1.44f},
                                 {8, 4, 5.02f, 3.29f, 1.82f, 2.34f, 0.98f, 0.269f, 2.46f},  {7, 4, 5.18f, 2.09f, 1.69f, 1.88f, 0.897f, 0.2f, 2.45f},
                                 {6, 4, 4.97f, 1.57f, 1.4f, 1.25f, 0.847f, 0.141f, 2.36f},
                                 {3, 2, 3.395f, 0.f, 0.869f, 0.236f, 0.42f, 0.108f, 1.499f}, {2, 2, 3.051f, 0.f, 0.679f, 0.014f, 0.431f, 0.021f, 0.975f},
                                 {2, 1, 2.443f, 0.888f, 0.f, 0.103f, 0.293f, 0.f, 0.475f},   {1, 1, 2.35f, 0.602f, 0.f, 0.227f, 0.234f, 0.f, 0.138f}};
  const int n_cu = f8_cus(), pin = p3v_tuning().gemm_f8_narrow;
  const bool silu = epilogue == P3V_EPI_SILU_MUL, resid = epilogue == P3V_EPI_RESID_BF16;
  const float kt = (float)(K / TKB);
  float best = -1.f;
  for (const auto& t : tiles) {
    const int n_tile = silu ? 32 * t.nb : 64 * t.nb;
    if (N % n_tile || (silu && t.nb % 2)) continue;
    if (t.mb > 5 && ((t.mb < 8 && K < 2 * TKB) || ldo >= 1 << 22)) continue;      // (four waves: two K-tiles come first below 256 rows; 32-bit store offsets)
    const long n = (long)(N / n_tile) * p3v_cdiv(M, 32 * t.mb);
    const float rounds = (float)p3v_cdiv(n, (long)n_cu), used = (float)n / (float)n_cu;
    float c = t.once + rounds * (t.f + (silu ? t.gated : resid ? t.resid : 0.f) + t.c * kt) + used * (t.fill * kt + t.out);
    if (pin == 10 * t.mb + t.nb || (pin == 0 && t.mb == 4 && t.nb == 4) || (pin == 1 && t.mb == 4 && t.nb == 2)) c = 0.f;
    if (best < 0.f || c < best) best = c, mb = t.mb, nb = t.nb;
  }
  return best;
}

template <int EPI>
static int launch_f8(const GemmF8P& p, hipStream_t s) {
  int mb = 0, nb = 0;
  f8_tile_plan(p.M, p.N, p.K, p.ldo, EPI, mb, nb);
  if constexpr (EPI != P3V_EPI_SILU_MUL)
    if (nb == 3) return launch_f8_v<EPI, 4, 3>(p, s);
  if constexpr (EPI != P3V_EPI_SILU_MUL)
    if (nb == 1) return mb == 1 ? launch_f8_v<EPI, 1, 1>(p, s) : launch_f8_v<EPI, 2, 1>(p, s);
  if (nb == 2) return mb == 2 ? launch_f8_v<EPI, 2, 2>(p, s) : mb == 3 ? launch_f8_v<EPI, 3, 2>(p, s) : launch_f8_v<EPI, 4, 2>(p, s);
  if (mb == 8) return launch_f8_w4<EPI, 8>(p, s);
  if (mb == 7) return launch_f8_w4<EPI, 7>(p, s);
  if (mb == 6) return launch_f8_w4<EPI, 6>(p, s);
  return mb == 5 ? launch_f8_v<EPI, 5, 4>(p, s) : launch_f8_v<EPI, 4, 4>(p, s);
}

extern "C" int p3v_gemm_fp8_tile(int M, int N, int K, int epilogue) {
  if (M <= 0 || N <= 0 || K <= 0 || K % TKB || N % 128 || (epilogue != P3V_EPI_NONE && epilogue != P3V_EPI_RESID_BF16 && epilogue != P3V_EPI_SILU_MUL)) return 0;
  int mb = 0, nb = 0;
  f8_tile_plan(M, N, K, N, epilogue, mb, nb);
  return 10 * mb + nb;
}

extern "C" int p3v_gemm_fp8(const p3v_gemm_fp8_args_t* a, void* stream) {
  if (!a || !a->A || !a->a_scale || !a->W || !a->w_scale || !a->out) return P3V_ERR_ARG;
  const int n_tile = 128;                              // SILU: 128 outputs per wide tile; plain: the narrow tile
  if (a->M < 0 || a->N <= 0 || a->K <= 0 || a->K % TKB || a->N % n_tile || a->ldo % 8) return P3V_ERR_ARG;
  if (a->lda < a->K || a->ldw < a->K || a->lda % 16 || a->ldw % 16) return P3V_ERR_ARG;
  if (((uintptr_t)a->A | (uintptr_t)a->W | (uintptr_t)a->out | (uintptr_t)a->resid) & 15) return P3V_ERR_ARG;
  if (a->epilogue == P3V_EPI_RESID_BF16 && !a->resid) return P3V_ERR_ARG;
  const size_t w_rows = (size_t)a->N * (a->epilogue == P3V_EPI_SILU_MUL ? 2 : 1);
  if (w_rows * a->ldw >= ((size_t)1 << 32) || (size_t)256 * a->lda >= ((size_t)1 << 31)) return P3V_ERR_UNSUPPORTED;   // 32-bit buffer offsets
  if (a->M == 0) return P3V_OK;
  const GemmF8P p = {a->A, a->a_scale, a->W, a->w_scale, a->out, a->resid, a->M, a->N, a->K, a->lda, a->ldw, a->ldo, {}};
  hipStream_t s = (hipStream_t)stream;
  switch (a->epilogue) {
    case P3V_EPI_NONE: return launch_f8<P3V_EPI_NONE>(p, s);
    case P3V_EPI_RESID_BF16: return launch_f8<P3V_EPI_RESID_BF16>(p, s);
    case P3V_EPI_SILU_MUL: return launch_f8<P3V_EPI_SILU_MUL>(p, s);
    default: return P3V_ERR_ARG;
  }
}

// Whether one launch beats the two.  It writes and reads 47 MB less (2531 rows), but runs on 128 x 256 tiles alone.  Both sides as in f8_tile_plan; the split +
// rotation, 3.5 us + 8.8 ns a row of 9216 and two fifths more beyond 40 MB of outputs, are what makes the rule agree best with 30 whole prompts of 256 .. 7000
// tokens at the decoder's widths run either way (it names the slower one for five, by 2.4 us a layer at most) and with 24 sizes of other widths launch
// behind launch.  (Launch behind launch, with the projection's outputs in the caches, they would be 3.7 us + 7.9 ns, and 2531 tokens would go the slower
// way by 13 us.)  us a layer, two - one, in a prompt: 768 tokens 5, 2531 13, 4096 37, 6000 16, but 256 -5, 1024 -7, 1800 -10, 2700 -11, where tiles of
// other heights fill their rounds; 8192 -15, where the rule says one (launch behind launch: +30).
// (Tiles of 192 and 224 rows on four waves under this epilogue, with one wave per SIMD to run it: no faster than the faster of the two at any size.)
static float qkv_fp8_gain(int M, int n_q, int n_kv, int K) {       // us that one launch saves
  int mb, nb;
  const int N = n_q + 2 * n_kv, n_cu = f8_cus();
  const float kt = (float)(K / TKB), out = (float)M * (float)N;
  const long tiles = (long)(n_q + n_kv) / 256 * p3v_cdiv(M, 128) + (long)n_kv / 128 * p3v_cdiv(M, 256);
  const float one = 6.66f + p3v_cdiv(tiles, (long)n_cu) * (1.73f + 0.62f * kt) + (float)tiles / (float)n_cu * (0.2f * kt + 4.23f);
  return f8_tile_plan(M, N, K, N, P3V_EPI_NONE, mb, nb) + 3.5f + 9.5e-7f * out + 4e-7f * fmaxf(out - 2e7f, 0.f) - one;
}
static bool qkv_fp8_sizes(int M, int n_q, int n_kv, int K) { return M > 0 && K > 0 && n_q > 0 && n_kv > 0 && n_q % 256 == 0 && n_kv % 256 == 0; }
extern "C" int p3v_gemm_qkv_fp8_pays(int M, int n_q, int n_kv, int K) { return qkv_fp8_sizes(M, n_q, n_kv, K) && qkv_fp8_gain(M, n_q, n_kv, K) > 0.f; }
// With an int8 cache behind it the split + rotation store the codes too (p3v_rope_kv_quantize), and a quantiser's launch goes with them: one launch has to
// gain 5 us more, and more than that the longer both take: the chip is then at its power limit, where 128 x 256 tiles on twelve waves cost more than their time
// (8192 tokens: the two pairs of launches are equal, but gate_up and attention beside the pair are 2 and 5 % faster).  The threshold is fitted to whole prompts of 137 .. 14000
// tokens at the decoder's widths, 95 lengths run either way, 35 of them on two to five machines: it names the slower side by 9 us a layer at most (4150 .. 4300 tokens on
// one machine, 8130 on another; 1.3 % of the prompt), elsewhere by no more than the runs of one side differ.  us a layer, two - one: 400 tokens -4.6, 577 -3.7, 768 0.4, 803 -19, 1800
// -16, 2300 -10, 2531 -5 .. 3, 2670 2, 3300 -7 and -18, 3500 0 and -7, 3900 -8.4, 4000 2 and 6, 4050 28, 4096 13 .. 30, 4150 -9 and -5, 4300 -5 and 3, 4500 -15, 5150 1, 5170 4, 5200 6, 6000 -2 and 4, 6100 -1 and 8, 6500 -15 and -5,
// 6750 41, 7000 0, 7300 -25 .. -37, 7800 -32, 8000 1 .. 20, 8192 -52, -40, -22 and 9, 10000 -14 and -8, 12288 0.
extern "C" int p3v_gemm_qkv_fp8_stored_pays(int M, int n_q, int n_kv, int K) {
  if (!qkv_fp8_sizes(M, n_q, n_kv, K)) return 0;
  const float out = (float)M * (float)(n_q + 2 * n_kv);
  return out <= 7.5e7f && qkv_fp8_gain(M, n_q, n_kv, K) > 5.f + 3.2e-7f * fmaxf(out - 2.4e7f, 0.f);
}

// p3v_gemm_fp8 (epilogue NONE) + p3v_rope_kv_append in one launch, bit for bit, on 128 x 256 tiles: the projection's 47 MB (2531 rows) are
// neither written nor read again.
extern "C" int p3v_gemm_qkv_fp8(const p3v_gemm_fp8_args_t* a, const p3v_qkv_split_t* sp, void* stream) {
  if (!a || !sp || !a->A || !a->a_scale || !a->W || !a->w_scale || !sp->q_out || !sp->k_dst || !sp->v_dst || (!sp->cos_t) != (!sp->sin_t)) return P3V_ERR_ARG;
  const int nh = sp->n_heads, nkv = sp->n_kv, hd = sp->hd;
  if (sp->B <= 0 || sp->L <= 0 || nh <= 0 || nkv <= 0 || hd <= 0 || sp->tab_div <= 0 || !(sp->q_scale > 0.f) || a->epilogue != P3V_EPI_NONE) return P3V_ERR_ARG;
  if (a->M != sp->B * sp->L || a->N != (nh + 2 * nkv) * hd || a->K <= 0 || a->K % TKB || a->lda < a->K || a->ldw < a->K || a->lda % 16 || a->ldw % 16) return P3V_ERR_ARG;
  if (((uintptr_t)a->A | (uintptr_t)a->W | (uintptr_t)sp->q_out | (uintptr_t)sp->k_dst | (uintptr_t)sp->v_dst | (uintptr_t)sp->cos_t | (uintptr_t)sp->sin_t) & 15) return P3V_ERR_ARG;
  const int dpos0 = sp->dst_off_is_past ? sp->past : 0;
  if (hd % 32 || (hd / 2) % 16 || (nh * hd) % 256 || (nkv * hd) % 256 || dpos0 % 8 || sp->dst_t % 8 || !qkv_rows_ok(sp->B, sp->L) ||
      p3v_tuning().gemm_no_qkv_fuse) return P3V_ERR_UNSUPPORTED;
  if ((size_t)a->N * a->ldw >= ((size_t)1 << 32) || (size_t)a->M * a->lda >= ((size_t)1 << 32) || (size_t)256 * a->lda >= ((size_t)1 << 31) ||
      (size_t)256 * a->ldw >= ((size_t)1 << 31)) return P3V_ERR_UNSUPPORTED;                                  // 32-bit buffer offsets
  const GemmF8P p = {a->A, a->a_scale, a->W, a->w_scale, nullptr, nullptr, a->M, a->N, a->K, a->lda, a->ldw, 0,
                     {sp->cos_t, sp->sin_t, sp->q_out, sp->k_dst, sp->v_dst, sp->L, nh, nkv, hd, sp->past, dpos0, sp->dst_t, sp->tab_t, sp->tab_div, sp->q_scale}};
  return launch_f8_v<P3V_EPI_QKV, 4, 4>(p, (hipStream_t)stream);
}

// ---------------------------------------------------------------- activation quantiser (one wave per token row)
// q[m, k] = e4m3(h[m, k] * (1 / s[m])),  s[m] = max_k |h[m, k]| / 448 (1 for an all-zero row; 1 / s rounded to fp32 once per
// row -- 8 million IEEE divisions per call kept the first version VALU-bound),  h = x, or -- with a norm weight --
// h = bf16(x * rsqrt(mean x^2 + eps) * g): exactly the row p3v_rmsnorm would have written (phi.py:478-479, 482, 484).
// The row is read ONCE and stays in registers (CH 16-byte chunks per lane: 6 for K = 3072, 16 for K = 8192) through the
// sum of squares, the maximum and the conversion: 3 bytes of traffic per element.
// The gain is requested with the row (a second trip behind the sum of squares otherwise), and where the row fills the lanes' chunks (FULL: K = 3072,
// 8192) nothing is masked: the branches around every chunk kept its arithmetic behind the last load.  us: 128 x 3072 with the norm 4.4 -> 3.8, 640
// 5.0 -> 4.2, 2531 9.6 -> 8.5, 8192 21.5 -> 17.6; 2531 x 8192 without 14.8 -> 14.0 (62 MB: 4.4 TB/s).  Not for 3072 without the norm: 128 rows
// 3.0 -> 3.2, 2531 6.9 either way.
template <bool NORM, int CH, bool FULL>
__global__ void __launch_bounds__(256) k_quant_fp8_rows(const u32x4_t* __restrict__ x, const u32x4_t* __restrict__ g,
                                                        u32x2_t* __restrict__ q, float* __restrict__ scale, int rows,
                                                        int chunks, float inv_h, float eps) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const u32x4_t* xr = x + (size_t)row * chunks;
  constexpr bool G_AHEAD = NORM && CH <= 6;                        // (16 chunks: too many registers)
  u32x4_t v[CH], gv[G_AHEAD ? CH : 1];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = i * 64 + lane;
    v[i] = FULL || c < chunks ? xr[c] : (u32x4_t){0u, 0u, 0u, 0u};
    if constexpr (G_AHEAD) gv[i] = FULL || c < chunks ? g[c] : (u32x4_t){0u, 0u, 0u, 0u};
  }
  float r = 1.f;
  if (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = bf16lo(v[i][j]), b = bf16hi(v[i][j]);
        ss += a * a + b * b;
      }
    r = rsqrtf(wave_sum(ss) * inv_h + eps);
  }
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = i * 64 + lane;
    if (NORM && (FULL || c < chunks)) {
      const u32x4_t w = G_AHEAD ? gv[i % (G_AHEAD ? CH : 1)] : g[c];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i][j] = rms_pair(v[i][j], r, w[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) amax = fmaxf(amax, fmaxf(fabsf(bf16lo(v[i][j])), fabsf(bf16hi(v[i][j]))));
  }
  amax = wave_max(amax);
  const float s = amax > 0.f ? amax / 448.f : 1.f;
  const float inv = 1.f / s;
  if (lane == 0) scale[row] = s;
  u32x2_t* qr = q + (size_t)row * chunks;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = i * 64 + lane;
    if (FULL || c < chunks) {
      u32x2_t o;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        int w = 0;
        w = __builtin_amdgcn_cvt_pk_fp8_f32(bf16lo(v[i][2 * j]) * inv, bf16hi(v[i][2 * j]) * inv, w, false);
        w = __builtin_amdgcn_cvt_pk_fp8_f32(bf16lo(v[i][2 * j + 1]) * inv, bf16hi(v[i][2 * j + 1]) * inv, w, true);
        o[j] = (uint32_t)w;
      }
      qr[c] = o;
    }
  }
}

template <bool NORM, int CH>
static void launch_quant(const uint16_t* x, const uint16_t* norm_w, float eps, uint8_t* q, float* scale, int rows, int K, hipStream_t s) {
  const auto fn = (NORM || CH > 6) && K == CH * 512 ? k_quant_fp8_rows<NORM, CH, NORM || (CH > 6)> : k_quant_fp8_rows<NORM, CH, false>;
  hipLaunchKernelGGL(fn, dim3(p3v_cdiv(rows, 4)), dim3(256), 0, s, (const u32x4_t*)x, (const u32x4_t*)norm_w, (u32x2_t*)q, scale, rows, K / 8, 1.0f / K, eps);
}

extern "C" int p3v_quant_fp8_rows(const uint16_t* x, const uint16_t* norm_w, float eps, uint8_t* q, float* scale, int rows,
                                  int K, void* stream) {
  if (!x || !q || !scale || rows < 0 || K <= 0 || K % 8 || K > 16 * 64 * 8) return P3V_ERR_ARG;
  if (((uintptr_t)x | (uintptr_t)norm_w) & 15 || (uintptr_t)q & 7) return P3V_ERR_ARG;
  if (rows == 0) return P3V_OK;
  hipStream_t s = (hipStream_t)stream;
  const int ch = p3v_cdiv(K / 8, 64);
  if (norm_w) {
    if (ch <= 6) launch_quant<true, 6>(x, norm_w, eps, q, scale, rows, K, s);
    else launch_quant<true, 16>(x, norm_w, eps, q, scale, rows, K, s);
  } else {
    if (ch <= 6) launch_quant<false, 6>(x, norm_w, eps, q, scale, rows, K, s);
    else launch_quant<false, 16>(x, norm_w, eps, q, scale, rows, K, s);
  }
  P3V_CHECK_LAUNCH();
  return P3V_OK;
}
