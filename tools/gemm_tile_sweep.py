"""Every tile of the large GEMMs over the sizes that their tile choices are fitted to (gemm_tile_choice, qkv_tile_plan: csrc/p3v_gemm.hip; f8_tile_plan:
csrc/p3v_gemm_fp8.hip): us per launch, weights from memory, graphs of one tile's launches replayed in turn without a pause, so that all share one power state.

    python3 tools/gemm_tile_sweep.py bf16|fp8|qkv [rows,rows,...]        # prints the table; `choice`: the tile that the library takes by itself
"""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import torch

from phi_3_vision_mlx_amd import _lib, ops

ROWS = [128, 192, 257, 320, 400, 512, 577, 640, 768, 900, 1024, 1154, 1300, 1536, 1800, 2048, 2300, 2531, 2885, 3500, 4096, 5193, 6000, 8192, 9809]
BF16 = [(8192, 3072, "silu"), (9216, 3072, "none"), (3072, 3072, "resid"), (3072, 8192, "resid"), (4096, 1024, "qgelu"), (1024, 4096, "resid_f32"), (1024, 1024, "resid_f32"),
        (10496, 3072, "none"), (3072, 8192, "scale"), (3072, 4096, "gelu"), (3072, 3072, "gelu"), (4096, 1024, "gelu")]
FP8 = [(8192, 3072, "silu"), (9216, 3072, "none"), (3072, 3072, "resid"), (3072, 8192, "resid"), (4096, 1024, "resid"), (9216, 1024, "none"), (8192, 1024, "silu"), (4096, 384, "none"),
       (9216, 640, "none"), (5120, 1664, "silu"), (4096, 2048, "resid"), (6144, 512, "silu"), (2048, 256, "none"), (8192, 2944, "silu"), (9216, 3200, "none")]
QKV = [(1, 0, 32, 32, 96, 3072), (1, 0, 16, 16, 96, 512), (1, 0, 32, 32, 96, 768), (1, 0, 32, 8, 96, 3072), (1, 0, 8, 8, 96, 1024), (4, 0, 32, 32, 96, 3072)] + [(b, 577, 16, 16, 64, 1024) for b in (2, 3, 5, 9, 13, 17)]
EACH, REPS = 1.2e-3, 4                                           # seconds of one tile's turn; turns


def in_turn(knob, pins, run, flops, rate):
    """us of run() with `knob` at each of `pins` (None: the library refuses)."""
    graphs = []
    for v in pins:
        saved = ops.set_tuning(knob, v)
        torch.cuda.synchronize()
        s = torch.cuda.Stream()
        try:
            with torch.cuda.stream(s):
                ok = run()
                torch.cuda.synchronize()
                g = torch.cuda.CUDAGraph()
                if ok:
                    with torch.cuda.graph(g, stream=s):
                        run()
            graphs.append(g if ok else None)
        except RuntimeError:
            graphs.append(None)
        finally:
            ops.set_tuning(knob, saved)
    n, ev = max(1, int(EACH * rate / flops)), []
    for rep in range(REPS + 1):
        for i, g in enumerate(graphs):
            if g is not None:
                e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
                e[0].record()
                for _ in range(n):
                    g.replay()
                e[1].record()
                if rep:
                    ev.append((i, e))
    torch.cuda.synchronize()
    t = [sorted(e[0].elapsed_time(e[1]) * 1e3 / n for j, e in ev if j == i) for i in range(len(pins))]
    return [x[len(x) // 2] if x else None for x in t]


def row(label, M, choice, times, per):                           # choice: the tile of the library's own choice
    print(f"{label:<28}{M:>6}{choice:>8}" + "".join(f"{t / per:>8.1f}" if t else f"{'-':>8}" for t in times), flush=True)


def weights(n, k, bytes_each, make):
    return [make(n, k) for _ in range(max(3, min(60, int(4.5e8 / (n * k * bytes_each)) + 1)))]


def sweep_bf16(rows):
    tiles = [84, 74, 64, 83, 63, 54, 44, 43]
    print("N x K (epilogue)                 M  choice     own" + "".join(f"{t:>8}" for t in tiles) + "    (own: the choice itself, no pin)")
    for N, K, epi in BF16:
        wn = 2 * N if epi == "silu" else N
        w = weights(wn, K, 2, lambda n, k: (torch.randn((n, k), device="cuda") * k ** -0.5).bfloat16())
        v = torch.randn((N,), device="cuda").bfloat16()
        for M in rows:
            a = [torch.randn((M, K), device="cuda").bfloat16() for _ in range(2)]
            r = torch.randn((M, N), device="cuda", dtype=torch.float32 if epi in ("resid_f32", "scale") else torch.bfloat16)
            out = torch.empty_like(r)
            kw = {"silu": dict(epilogue=ops.EPI_SILU_MUL), "none": dict(epilogue=ops.EPI_NONE), "resid": dict(epilogue=ops.EPI_RESID_BF16, resid=r), "qgelu": dict(epilogue=ops.EPI_BIAS_QGELU, bias=v),
                  "gelu": dict(epilogue=ops.EPI_BIAS_GELU, bias=v), "resid_f32": dict(epilogue=ops.EPI_BIAS_RESID_F32, resid=r, bias=v),
                  "scale": dict(epilogue=ops.EPI_SCALE_RESID_F32, resid=r, col_scale=v)}[epi]

            def run():
                for i, x in enumerate(w):
                    ops.gemm(a[i % 2], x, out=out, **kw)
                return True
            times = in_turn("gemm_tile", [-1] + tiles, run, len(w) * 2.0 * M * wn * K, 1.1e15)
            row(f"{N}{'(x2)' if epi == 'silu' else ''} x {K} {epi}", M, _lib.lib().p3v_gemm_tile(M, N, K, kw["epilogue"]), times, len(w))


def sweep_fp8(rows):
    tiles = [44, 54, 43, 42, 64, 74, 84, 32, 22, 21, 11]
    print("N x K (epilogue)                 M  choice" + "".join(f"{t:>8}" for t in tiles))

    def codes(n, k):
        return (torch.randn((n, k), device="cuda") * 100).clamp(-440, 440).to(torch.float8_e4m3fn).view(torch.uint8)
    for N, K, epi in FP8:
        wn = 2 * N if epi == "silu" else N
        e = {"silu": ops.EPI_SILU_MUL, "none": ops.EPI_NONE, "resid": ops.EPI_RESID_BF16}[epi]
        w, ws = weights(wn, K, 1, codes), (torch.rand((wn,), device="cuda") + 0.5) * 1e-4
        for M in rows:
            a, sa, r = [codes(M, K) for _ in range(2)], torch.rand((M,), device="cuda") + 0.5, torch.randn((M, N), device="cuda").bfloat16()
            out = torch.empty_like(r)

            def run():
                for i, x in enumerate(w):
                    ops.gemm_fp8(a[i % 2], sa, x, ws, e, resid=r if epi == "resid" else None, out=out)
                return _lib.lib().p3v_gemm_fp8_tile(M, N, K, e) in tiles
            usable = [t for t in tiles if N % (32 * (t % 10) if epi == "silu" else 64 * (t % 10)) == 0 and not (epi == "silu" and t % 2)]
            times = dict(zip(usable, in_turn("gemm_f8_narrow", usable, run, len(w) * 2.0 * M * wn * K, 2e15)))
            row(f"{N}{'(x2)' if epi == 'silu' else ''} x {K} {epi}", M, _lib.lib().p3v_gemm_fp8_tile(M, N, K, e), [times.get(t) for t in tiles], len(w))


def sweep_qkv(rows):
    tiles = [1, 2, 3, 4, 5, 6, 7, 8]
    print("B x L, heads / kv x dim, K       M  choice     own" + "".join(f"{t:>8}" for t in tiles) + "    (32 t rows a tile; 1: 128 x 128)")
    for B, L0, nh, nkv, hd, K in QKV:
        for L in [L0] if L0 else [r // B for r in rows]:
            M, N, Tp = B * L, (nh + 2 * nkv) * hd, (L + 127) // 128 * 128
            w = [(torch.randn((N, K), device="cuda") * K ** -0.5).bfloat16() for _ in range(12)]
            # (image crops, L0: a bias and no rotation)
            a, cos = torch.randn((M, K), device="cuda").bfloat16(), None if L0 else torch.rand((B, Tp, hd // 2), device="cuda")
            bias = torch.randn((N,), device="cuda").bfloat16() if L0 else None
            q, k, v = (torch.zeros(s, device="cuda", dtype=torch.bfloat16) for s in ((B, nh, L, hd), (B, nkv, Tp, hd), (B, nkv, hd, Tp)))

            def run():
                return all([ops.gemm_qkv(a, x, cos, cos, q, k, v, B, L, nh, nkv, hd, 0, Tp, True, Tp, 1, q_scale=0.5, bias=bias) for x in w])
            times = in_turn("gemm_qkv_flat", [-1] + tiles, run, len(w) * 2.0 * M * N * K, 1.1e15)
            row(f"{B} x {L}, {nh} / {nkv} x {hd}, {K}", M, _lib.lib().p3v_gemm_qkv_tile(M, nh * hd, nkv * hd, K), times, len(w))


if __name__ == "__main__":
    rows = [int(x) for x in sys.argv[2].split(",")] if len(sys.argv) > 2 else ROWS
    ops.set_tuning("gemm_big_rows", -1)
    {"bf16": sweep_bf16, "fp8": sweep_fp8, "qkv": sweep_qkv}[sys.argv[1]](rows)
