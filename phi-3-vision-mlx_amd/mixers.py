"""The mixers of the layered decoders: what a layer does between its norm and its output projection.

A mixer holds the device weights of one layer that has them (another layer may use the same object) and takes the rows of ONE packed
projection of the layer's input:

    w_in                     the packed projection; its rows are padded with zeros to whole GEMM tiles
    n_out, o                 columns of the mixer's output, the output projection
    buffers(B, L, n_keys)    {name: (elements, dtype)} of scratch; layers share a buffer of the largest size
    plan(B, L, n_keys)       what a call's launches are planned for (a one-token call: the cache capacity, so that eager and captured
                             steps run alike)
    run(y, out, rows, bufs, call, plan)
                             call.tail: only the outputs of each sequence's last token are read; a mixer that saves work by it returns these
                             rows, else None
"""
from dataclasses import dataclass
from typing import Any

import torch

from . import ops
from .cache import latent_width, round_up
from .config import GlaMixer, LatentMixer, Mixer
from .ops import BF16, F32


@dataclass
class Call:
    """One call of the stack: B rows of L new tokens behind `past` columns (d_past: the same from device memory), of which `keep` stay."""
    B: int
    L: int
    past: int
    keep: int
    d_past: Any = None
    pad_len: Any = None
    v_first: Any = None
    tail: bool = False


def packed(mats):
    """Matrices that read the same input as one, in whole GEMM tiles (the 256-column ones where it is wide): the padding rows are zero
    and nobody reads their outputs."""
    w = torch.cat(mats)
    n = round_up(w.shape[0], 256 if w.shape[0] >= 2048 else 64)
    return torch.cat([w, w.new_zeros((n - w.shape[0], w.shape[1]))]).contiguous()


class MixedHeads:
    """Attention whose heads' scores are mixed before the softmax (config.Mixer)."""

    def __init__(self, m, w, p, dev, cfg):
        def t(name):
            return w[p + name].to(dev, BF16).contiguous()
        self.m, self.eps, self.T = m, cfg.norm_eps, F32 if cfg.dtype == "float32" else BF16
        self.w_in, self.o, self.n_out = packed([t("q"), t("k"), t("v"), t("g")]), t("o"), m.heads * m.vdim
        self.norms = (t("q.norm"), t("k.norm"))
        self.talk, self.sink, self.vmix = t("talk"), t("sink"), float(w[p + "vmix"]) if p + "vmix" in w else 0.0
        self.v_col = (m.heads + m.kv_heads) * m.dim              # first value column of the packed projection

    def plan(self, B, L, n_keys):
        m = self.m
        # Two launches on fragments of the keys, or one on their rows.  Wide heads fill the one launch's registers: two.  Else
        # - a single tile of 32 keys does not pay for the fragments' launch and the scores' way through memory.  us of head split and attention, one launch : two, 16, 32 and,
        #   two tiles, 33 tokens: 32 heads x 96 24.5 : 25.5, 25.0 : 26.0, 28.1 : 26.9; 24 x 64 19.7 : 20.4, 19.9 : 21.2, 24.3 : 21.4; 18 x 96 / 48 16.9 : 20.1, 17.3 : 21.1, 22.0 : 21.9; 32 x
        #   128 36.3 : 27.7.  Whole prompts of 17 .. 32 tokens 2.5 % faster, captured, and 4 .. 6 where the host is what they wait for; a few tokens behind earlier ones
        #   are two tiles: 16 behind 32 30.9 : 26.2.
        # - few new tokens of many rows behind long caches do not pay for the copy of all keys, once they fill the chip in one launch: 12 rows of 96 behind 2000 234 : 293, 8 of 40 behind
        #   3000 179 : 205, 6 of 40 behind 3000 144 : 159, but 4 of 128 behind 4000 1.23x faster in two, 2 of 24 behind 16000 1.51x.  The line is fitted to 1506 sizes of 1 .. 16 rows of 24 ..
        #   600 tokens behind 0 .. 16000 at 32 x 96 and 24 x 64: 0.4 % behind the faster form on average (two launches always: 0.9 %, 41 % at most), 17 % at most.
        narrow, copied = round_up(m.dim, 32) + round_up(m.vdim, 32) <= 192, 2e-6 * B * m.kv_heads * n_keys * round_up(m.dim, 32)      # MB of keys
        one = narrow and (n_keys <= 32 or (n_keys > L and B * -(-L // 16) >= 10 and copied >= 80 + 0.5 * L))
        if not one and ops.mix_prompt_ws_bytes(B, L, m.heads, m.kv_heads, m.dim, m.vdim, n_keys, self.T):
            return -1
        return ops.mix_plan(B, L, m.heads, m.kv_heads, m.dim, m.vdim, n_keys, self.T)

    def buffers(self, B, L, n_keys):
        m, plan = self.m, self.plan(B, L, n_keys)
        if plan < 0:                                             # (of the whole prompt, and of its last tile: Call.tail)
            ws = max(ops.mix_prompt_ws_bytes(B, n, m.heads, m.kv_heads, m.dim, m.vdim, n_keys, self.T) for n in (L, ops.MIX_TAIL))
        else:
            ws = ops.mix_ws_bytes(B, L, m.heads, m.vdim, plan)
        return {"q": (B * L * m.heads * round_up(m.dim, 32), self.T), "attn_ws": (ws // 4, F32)}

    def run(self, y, out, rows, bufs, call, plan):
        m = self.m
        tail = call.tail and plan < 0
        got = ops.attention_mixed(y, bufs["q"], rows.k, rows.v, out, self.norms, self.talk, self.sink, call.B, call.L, m.heads, m.kv_heads, m.dim,
                                  m.vdim, self.eps, m.scale, call.past, v_first=call.v_first if m.v_mix else None, vmix=self.vmix,
                                  pad_len=call.pad_len, d_past=call.d_past, ws=bufs["attn_ws"], n_split=plan, tail=tail)
        return got if tail else None

    def values(self, y):
        return y[:, self.v_col:self.v_col + self.m.kv_heads * self.m.vdim]


class LatentHeads:
    """Latent attention (config.LatentMixer).  A few new tokens attend in the latent space: the up-projections of keys and values are
    applied to the query and to the attended latent.  A prompt expands keys and values of all its columns once and attends over those."""

    def __init__(self, m, w, p, dev, cfg):
        def t(name):
            return w[p + name].to(dev, BF16)
        self.m, self.eps, self.T = m, cfg.norm_eps, F32 if cfg.dtype == "float32" else BF16
        self.w_in, self.o, self.n_out = packed([t("q"), t("dkv"), t("g")]), t("o").contiguous(), m.heads * m.vdim
        self.c_norm, self.sink = t("dkv.norm").contiguous(), t("sink").contiguous()
        rankp, dimp = round_up(m.rank, 64), round_up(m.dim, 32)

        def wide(a):                                             # the latent's padding meets zeros
            return torch.nn.functional.pad(a, (0, rankp - m.rank)).contiguous()
        self.uk, self.uv = wide(t("uk")), wide(t("uv"))
        ukt = self.uk.view(m.heads, m.dim, rankp).transpose(1, 2)
        self.ukt = torch.nn.functional.pad(ukt, (0, dimp - m.dim)).contiguous()

    def plan(self, B, L, n_keys):
        return ops.latent_plan(self.m, B, L, n_keys, self.T)

    def buffers(self, B, L, n_keys):
        m, plan = self.m, self.plan(B, L, n_keys)
        if plan > 0:                                             # in the latent space, keys split `plan` ways
            hp = round_up(m.heads, 16)
            return {"q": (B * L * hp * latent_width(m), self.T), "attn_ws": (ops.latent_ws_bytes(m, B, L, plan) // 4, F32)}
        if plan < 0:                                             # expanded
            n = round_up(n_keys, 64)
            return {"kx": (B * n * m.heads * m.dim, self.T), "vx": (B * n * m.heads * m.vdim, self.T)}
        return {}

    def run(self, y, out, rows, bufs, call, plan):
        ops.attention_latent(self, y, out, rows.c, rows.cos, rows.sin, bufs, call, plan)


class LinearState:
    """Gated linear attention (config.GlaMixer)."""

    def __init__(self, m, w, p, dev, cfg):
        def t(name):
            return w[p + name].to(dev, BF16).contiguous()
        self.m, self.eps, self.T = m, cfg.norm_eps, F32 if cfg.dtype == "float32" else BF16
        self.w_in, self.o, self.n_out = packed([t("q"), t("k"), t("v"), t("g"), t("a1")]), t("o"), m.heads * m.vdim
        self.a2, self.a2_b, self.norm = t("a2"), t("a2.b"), t("norm")
        self.rank = self.a2.shape[1]
        if w[p + "a1"].shape[0] != self.rank:
            raise ValueError(f"{p}a1 has {w[p + 'a1'].shape[0]} rows, {p}a2 {self.rank} columns")

    def plan(self, B, L, n_keys):
        return ops.gla_plan(self.m, B, L, self.T)

    def buffers(self, B, L, n_keys):
        return {"gla_ws": (ops.gla_ws_bytes(self.m, B, L, self.plan(B, L, n_keys)) // 4, F32)}

    def run(self, y, out, rows, bufs, call, plan):
        ops.gated_linear_attention(self, y, out, rows.s, bufs.get("gla_ws"), call, plan)


MIXERS = {Mixer: MixedHeads, LatentMixer: LatentHeads, GlaMixer: LinearState}
