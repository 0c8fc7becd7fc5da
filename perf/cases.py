"""The measured workloads of the quantized-decode framework: decode, prompt and expert layers, whole
decode steps and compiled graphs, at the sizes of this repository's configurations and over the ranges
around them.

Every case names a `kind` (one way a program uses the framework) and its sizes:

  linear        the same projection of every layer of a decode step, captured in one graph (1..16 rows)
  decode_attn   decode attention of every layer over a resident KV cache, captured in one graph
  decode        whole decode steps of an int8 model through DecodeEngine's step graphs -> logits
  prompt        a whole prompt through DecodeEngine.prefill and the next token's logits
  attn_block    one attention layer over prompt rows (AttentionDecode.prefill) -> hidden rows, KV cache
  mlp_block     one SwiGLU MLP over prompt rows (SwiGLUDecode.prefill) -> hidden rows
  moe           one mixture-of-experts MLP (MoEDecode.run), decode batches and prompt chunks
  graph_mlp     an af.compile program called with host arrays
  graph_sdpa    an af.compile program of causal attention over device ports

Weights are drawn as N(0, 0.02) in each format's own code layout, hidden rows as N(0, 1)."""
import ctypes
import math

import numpy as np
import torch

LINEAR_FMTS = ("int8", "q4_0", "fp16", "blockwise", "lut4", "q4_k", "q6_k")
BLOCK_FMTS = ("int8", "int8", "q4_0", "fp16", "blockwise", "lut4", "q4_k")
MOE_FMTS = ("q4_0", "q4_0", "q4_k", "q6_k", "blockwise")
EPS = 1e-5
STD = 0.02


# ----------------------------------------------------------------------------- the cases
def listed():
    return [
        # the o-projection of 16 layers in a one-sequence int8 decode step: the smallest call, all
        # weight stream and launch latency
        {"name": "linear_int8_1row", "kind": "linear", "fmt": "int8", "N": 4096, "K": 4096, "M": 1, "calls": 16},
        # the gate projection of a Q4_0 checkpoint for 4 sequences (or 4 speculated tokens)
        {"name": "linear_q4_0_4rows", "kind": "linear", "fmt": "q4_0", "N": 11008, "K": 4096, "M": 4, "calls": 8},
        # attention of a 16-sequence batch over long contexts, the KV-cache stream
        {"name": "decode_attn_16x8192", "kind": "decode_attn", "B": 16, "H": 32, "KV": 8, "D": 128, "ctx": 8192,
         "calls": 2},
        # the headline workload: tokens of the 32-layer int8 decode at position 2048
        {"name": "decode_int8_32_layers", "kind": "decode", "layers": 32, "D": 4096, "KV": 8, "F": 11008,
         "V": 32000, "pos": 2048, "steps": 8, "sampled": False},
        # a chat turn: a 65-token prompt through the model, to the first token's logits
        {"name": "prompt_65_tokens", "kind": "prompt", "fmt": "int8", "layers": 8, "D": 4096, "KV": 8, "F": 11008,
         "V": 32000, "n": 65},
        # one attention layer of the 2048-token prompt
        {"name": "attn_block_2048", "kind": "attn_block", "fmt": "int8", "D": 4096, "KV": 8, "m": 2048, "pos0": 0},
        # one MLP of the 2048-token prompt: the largest matrix products
        {"name": "mlp_block_2048", "kind": "mlp_block", "fmt": "int8", "D": 4096, "F": 11008, "m": 2048},
        # the MLP of a short, ragged prompt over a 4-bit checkpoint
        {"name": "mlp_block_q4_0_100", "kind": "mlp_block", "fmt": "q4_0", "D": 4096, "F": 11008, "m": 100},
        # a decode batch of 16 tokens through an 8-expert layer
        {"name": "moe_16_tokens", "kind": "moe", "fmt": "q4_0", "E": 8, "k": 2, "D": 4096, "F": 14336, "T": 16},
        # a prompt of 300 tokens through the same layer
        {"name": "moe_300_tokens", "kind": "moe", "fmt": "q4_0", "E": 8, "k": 2, "D": 4096, "F": 14336, "T": 300},
        # an int8 program called with host arrays, one row in and out
        {"name": "graph_mlp_1row", "kind": "graph_mlp", "compress": "int8", "D": 2048, "F": 5632, "M": 1},
        # af.sdpa of a 512-token causal sequence, 32 query heads on 8 key/value heads
        {"name": "graph_sdpa_512", "kind": "graph_sdpa", "H": 32, "KV": 8, "D": 128, "S": 512, "causal": True},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "decode_attn", "decode", "prompt", "attn_block", "attn_block", "mlp_block",
                       "mlp_block", "moe", "moe", "graph_mlp", "graph_sdpa"])
    if kind == "linear":
        N, K = 16 * _log(rng, 64, 1376), 256 * _log(rng, 4, 43)
        return {"kind": kind, "fmt": rng.choice(LINEAR_FMTS), "N": N, "K": K, "M": _log(rng, 1, 16),
                "calls": max(2, min(16, (1 << 28) // (N * K)))}
    if kind == "decode_attn":
        D, KV = rng.choice([64, 128, 128]), rng.choice([2, 4, 8, 8])
        B, ctx = _log(rng, 1, 16), _log(rng, 128, 8192)
        return {"kind": kind, "B": B, "H": KV * rng.choice([1, 4, 4, 8]), "KV": KV, "D": D, "ctx": ctx,
                "calls": max(2, min(16, (1 << 28) // (B * KV * ctx * D)))}
    if kind == "decode":
        return {"kind": kind, "layers": _log(rng, 1, 16), "D": 4096, "KV": rng.choice([8, 8, 32]), "F": 11008,
                "V": rng.choice([32000, 32000, 50257]), "pos": _log(rng, 64, 4096), "steps": rng.randint(1, 8),
                "sampled": rng.random() < 0.5}
    D = 128 * rng.choice([8, 16, 16, 24, 32, 32])
    if kind == "prompt":
        return {"kind": kind, "fmt": rng.choice(BLOCK_FMTS), "layers": _log(rng, 1, 8), "D": D,
                "KV": D // 128 // rng.choice([1, 4]), "F": 256 * (D * 43 // 16 // 256), "V": 32000, "n": _log(rng, 3, 1200)}
    if kind == "attn_block":
        m = _log(rng, 2, 2048)
        return {"kind": kind, "fmt": rng.choice(BLOCK_FMTS), "D": D, "KV": D // 128 // rng.choice([1, 4, 8]), "m": m,
                "pos0": rng.choice([0, 0, _log(rng, 16, 2048)])}
    if kind == "mlp_block":
        return {"kind": kind, "fmt": rng.choice(BLOCK_FMTS), "D": D, "F": 256 * _log(rng, D // 128, D * 43 // 16 // 256),
                "m": _log(rng, 2, 2048)}
    if kind == "moe":
        D = 256 * _log(rng, 4, 16)
        E = rng.choice([8, 8, 16, 60])
        return {"kind": kind, "fmt": rng.choice(MOE_FMTS), "E": E, "k": rng.choice([2, 2, 4]), "D": D,
                "F": 256 * _log(rng, 3, 14336 * 4096 * 8 // (D * E * 256) if E * D > 32 * 1024 else 56), "T": _log(rng, 1, 512)}
    if kind == "graph_mlp":
        return {"kind": kind, "compress": rng.choice(["int8", "int8", "blockwise", None]), "D": 128 * rng.randint(4, 16),
                "F": 128 * rng.randint(8, 44), "M": _log(rng, 1, 64)}
    KV = rng.choice([2, 4, 8])
    return {"kind": kind, "H": KV * rng.choice([1, 4]), "KV": KV, "D": rng.choice([64, 128, 128]), "S": _log(rng, 16, 1024),
            "causal": rng.random() < 0.7}


# ----------------------------------------------------------------------------- weights
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)


def _bytes(g, *shape):
    """Two 4-bit codes a byte, each N(7.5, 2.3) rounded: what a block quantizer leaves."""
    lo, hi = ((_randn(g, *shape) * 2.3 + 7.5).round_().clamp_(0, 15).to(torch.uint8) for _ in range(2))
    return lo | (hi << 4)


def _weight(g, fmt, N, K):
    """Codes and scales of one [N, K] matrix in the layout of format `fmt`."""
    if fmt == "fp16":
        return _randn(g, N, K) * STD, None
    if fmt in ("int8", "blockwise"):
        q = (_randn(g, N, K) * 36).round_().clamp_(-127, 127).to(torch.int8)
        n = (N,) if fmt == "int8" else (N, K // 32)
        return q, ((torch.rand(n, generator=g, device="cuda") * 0.4 + 0.8) * (STD / 36)).half()
    codes = _bytes(g, N, K // 2)
    if fmt == "q4_0":
        return codes, ((torch.rand((N, K // 32), generator=g, device="cuda") * 0.4 + 0.8) * (STD / 2.3)).half()
    if fmt == "lut4":
        return codes, (torch.linspace(-3.2, 3.2, 16, device="cuda") * STD + 1e-3 * torch.randn((N, 16), generator=g, device="cuda")).half()
    if fmt == "q4_k":       # per 256 weights: {d, dmin}, then per pair of 32-weight sub-blocks {sc, sc, m, m}
        sc = torch.randint(20, 64, (N, K // 256, 4, 2), generator=g, device="cuda", dtype=torch.int32)
        h = torch.empty((N, K // 256, 5), dtype=torch.int32, device="cuda")
        h[..., 0] = _bits(STD / 2.3 / 42) | (_bits(7.5 * STD / 2.3 / 42) << 16)
        h[..., 1:] = sc[..., 0] | (sc[..., 1] << 8) | (sc[..., 0] << 16) | (sc[..., 1] << 24)
        return codes, h.reshape(N, -1)
    side = torch.empty((N, K // 32, 3), dtype=torch.int32, device="cuda")       # q6_k
    side[..., :2] = torch.randint(-2**31, 2**31 - 1, (N, K // 32, 2), generator=g, device="cuda", dtype=torch.int32)
    sc = torch.randint(20, 100, (N, K // 32, 2), generator=g, device="cuda", dtype=torch.int32)
    side[..., 2] = sc[..., 0] | (sc[..., 1] << 8) | (_bits(STD / 18 / 60) << 16)
    return codes, side.reshape(N, -1)


def _bits(v):
    return int(np.float16(v).view(np.uint16))


def _fp16(v):
    return float(np.float16(v))


def _dense(fmt, w, s):
    """The weights of a format in 64 bits, from its definition."""
    N = w.shape[0]
    if fmt == "fp16":
        return w.double()
    if fmt == "int8":
        return w.double() * s.double()[:, None]
    if fmt == "blockwise":
        return (w.view(N, -1, 32).float() * s.float()[..., None]).half().double().view(N, -1)
    lo, hi = w & 15, w >> 4
    if fmt == "lut4":
        return torch.gather(s, 1, torch.stack([lo, hi], -1).view(N, -1).long()).double()
    if fmt == "q4_0":       # bytes of word [superblock][g][block]: {e0 e2} {e4 e6} {e1 e3} {e5 e7}
        v = torch.stack([lo, hi], -1).view(N, -1, 4, 4, 2, 4)                   # [sb, g, block, odd, i]
        v = v.permute(0, 1, 3, 2, 5, 4).reshape(N, -1, 32)                      # [block][g][i][odd]
        return ((v.float() - 8) * s.float()[..., None]).half().double().view(N, -1)
    if fmt == "q4_k":
        h = s.view(N, -1, 5)
        d, dm = _fp16(STD / 2.3 / 42), _fp16(7.5 * STD / 2.3 / 42)
        sm = torch.stack([(h[..., 1:] >> (8 * i)) & 255 for i in range(4)], -1).float()   # [N, nb, pair, 4]
        q = torch.stack([lo.view(N, -1, 4, 32), hi.view(N, -1, 4, 32)], 3).float()
        return (d * sm[..., :2, None] * q - dm * sm[..., 2:, None]).half().double().reshape(N, -1)
    side = s.view(N, -1, 3)                                                     # q6_k
    lo4 = torch.stack([lo.view(N, -1, 4, 4), hi.view(N, -1, 4, 4)], 3).reshape(N, -1, 32)
    H = torch.stack([(side[..., :2] >> (8 * j)) & 255 for j in range(4)], -1)   # [N, chunk, half word, j]
    h2 = torch.stack([(H >> (2 * q)) & 3 for q in range(4)], 3).reshape(N, -1, 32)
    sc = torch.stack([side[..., 2] & 255, (side[..., 2] >> 8) & 255], -1).float()
    ds = _fp16(STD / 18 / 60) * sc
    q = (lo4.int() | (h2 << 4)).float() - 32
    return (q.view(N, -1, 2, 16) * ds[..., None]).half().double().reshape(N, -1)


def _wbytes(fmt, N, K):
    return {"fp16": 2 * N * K, "int8": N * K + 2 * N, "blockwise": N * K + N * K // 16, "q4_0": N * K // 2 + N * K // 16,
            "lut4": N * K // 2 + 32 * N, "q4_k": N * K // 2 + N * K // 256 * 20, "q6_k": N * K // 2 + N * K // 32 * 12}[fmt]


def _matmul(x, fmt, w, s, rows=8192):
    """x @ W^T in 64 bits, a few weight rows at a time."""
    return torch.cat([x @ _dense(fmt, w[r:r + rows], None if s is None else s[r:r + rows]).T for r in range(0, w.shape[0], rows)], -1)


# ----------------------------------------------------------------------------- 64-bit pieces
def _rms(x, g):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * g.double()


def _unpair(y, heads):
    """Projection rows in rope-pair order (d, d + dh/2 side by side) to natural head order."""
    return y.view(*y.shape[:-1], heads, -1, 2).transpose(-1, -2).reshape(*y.shape[:-1], heads, -1)


def _rope64(x, cos, sin):
    a, b = x.chunk(2, -1)
    return x * cos[:, None] + torch.cat([-b, a], -1) * sin[:, None]


def _rope_tables(n, dh):
    a = torch.arange(n, dtype=torch.float64)[:, None] / 10000.0 ** (torch.arange(0, dh, 2, dtype=torch.float64) / dh)
    a = torch.cat([a, a], 1)
    return a.cos().half().numpy(), a.sin().half().numpy()


def _attend(q, k, v, off):
    """q [m, H, D] over k, v [KV, n, D]; query i sees rows 0 .. off + i."""
    m, H, D = q.shape
    KV, n = k.shape[:2]
    out = torch.empty_like(q)
    seen = torch.arange(n, device=q.device)[None] <= off + torch.arange(m, device=q.device)[:, None]
    for h in range(H):
        s = (q[:, h] @ k[h * KV // H].T) / math.sqrt(D)
        out[:, h] = s.masked_fill(~seen, -math.inf).softmax(-1) @ v[h * KV // H]
    return out


def _attn64(x, L, kc, vc, pos0, H, KV, cos, sin):
    """The attention layer on rows x at positions pos0..; kc, vc [KV, M, dh] are written."""
    m = x.shape[0]
    y = _matmul(_rms(x, L["an"]), *L["qkv"])
    dh = y.shape[1] // (H + 2 * KV)
    q, k, v = y.split([H * dh, KV * dh, KV * dh], 1)
    c, s = cos[pos0:pos0 + m], sin[pos0:pos0 + m]
    q, k = _rope64(_unpair(q, H), c, s), _rope64(_unpair(k, KV), c, s)
    kc[:, pos0:pos0 + m], vc[:, pos0:pos0 + m] = k.transpose(0, 1), v.view(m, KV, dh).transpose(0, 1)
    a = _attend(q, kc[:, :pos0 + m], vc[:, :pos0 + m], pos0)
    return x + _matmul(a.reshape(m, -1), *L["wo"])


def _mlp64(x, L):
    y = _matmul(_rms(x, L["mn"]), *L["gu"])
    return x + _matmul(torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2], *L["down"])


# ----------------------------------------------------------------------------- a model
def _raw_layer(g, fmt, D, KV, F):
    nkv = KV * 128
    L = {"an": 1 + 0.1 * _randn(g, D), "mn": 1 + 0.1 * _randn(g, D)}
    if KV:
        L["qkv"], L["wo"] = (fmt, *_weight(g, fmt, D + 2 * nkv, D)), (fmt, *_weight(g, fmt, D, D))
    if F:
        L["gu"], L["down"] = (fmt, *_weight(g, fmt, 2 * F, D)), (fmt, *_weight(g, fmt, D, F))
    return L


def _raw_model(c, seed):
    g = _gen(seed)
    layers = [_raw_layer(g, c.get("fmt", "int8"), c["D"], c["KV"], c["F"]) for _ in range(c["layers"])]
    m = {"layers": layers, "fn": 1 + 0.1 * _randn(g, c["D"]), "embed": _randn(g, c["V"], c["D"]) * STD,
         "head": _randn(g, c["V"], c["D"]) * STD, "g": g}
    rng = np.random.default_rng(seed)
    m["tokens"] = rng.integers(0, c["V"], c.get("n", c.get("steps", 1))).tolist()
    return m


def _linear(t):
    from aneforge_amd import _engine as E
    fmt, w, s = t
    return E.Linear(fmt, w, s, w.shape[0], w.shape[1] * (2 if w.dtype == torch.uint8 else 1))


def _engine(raw, D, KV, F, V, M):
    from aneforge_amd import _engine as E
    from aneforge_amd.llm import LlamaConfig
    cfg = LlamaConfig(dim=D, n_layers=len(raw["layers"]), n_heads=D // 128, n_kv_heads=KV, ffn_dim=F, vocab=V, norm_eps=EPS)
    layers = [(E.AttentionDecode.from_linears(cfg, _linear(L["qkv"]), _linear(L["wo"]), L["an"]),
               E.SwiGLUDecode.from_linears(cfg, _linear(L["gu"]), _linear(L["down"]), L["mn"])) for L in raw["layers"]]
    return E.DecodeEngine(cfg, layers, raw["embed"], E.Linear("fp16", raw["head"], None, V, D), raw["fn"], M,
                          rope_tables=_rope_tables(M, 128))


def _cache_rows(g, KV, n):
    return _randn(g, KV, n, 128), _randn(g, KV, n, 128)


class _Captured:
    """Launches captured into a graph on a stream of their own."""

    def __init__(self, fn):
        from aneforge_amd import _hip
        self.hip, self.exec, self.stream = _hip, ctypes.c_void_p(), torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(self.stream):
            fn()                                           # first launches load the kernels
            _hip.call("afx_graph_begin", self.stream.cuda_stream)
            try:
                fn()
            finally:
                _hip.call("afx_graph_end", self.stream.cuda_stream, ctypes.byref(self.exec))
        torch.cuda.synchronize()

    def launch(self):
        self.hip.call("afx_graph_launch", self.exec, self.stream.cuda_stream)

    def __del__(self):
        if self.exec:
            self.hip.call("afx_graph_destroy", self.exec)


# ----------------------------------------------------------------------------- inputs of each kind
def _in_linear(c, seed):
    g = _gen(seed)
    ws = [_weight(g, c["fmt"], c["N"], c["K"]) for _ in range(c["calls"])]
    return ws, [_randn(g, c["M"], c["K"]) for _ in ws]


def _in_decode_attn(c, seed):
    g = _gen(seed)
    return [(_randn(g, c["B"], c["H"], c["D"]), _randn(g, c["B"], c["KV"], c["ctx"], c["D"]),
             _randn(g, c["B"], c["KV"], c["ctx"], c["D"])) for _ in range(c["calls"])]


def _in_block(c, seed):
    g = _gen(seed)
    F = c.get("F", 0)
    L = _raw_layer(g, c["fmt"], c["D"], c.get("KV", 0), F)
    return L, _randn(g, c["m"], c["D"]), _cache_rows(g, c.get("KV", 1), c.get("pos0", 0))


def _in_moe(c, seed):
    g = _gen(seed)
    E, D, F, fmt = c["E"], c["D"], c["F"], c["fmt"]
    experts = [[_weight(g, fmt, n, k) for n, k in ((F, D), (F, D), (D, F))] for _ in range(E)]
    return experts, _randn(g, E, D) * STD, 1 + 0.1 * _randn(g, D), _randn(g, c["T"], D)


def _in_graph_mlp(c, seed):
    r = np.random.default_rng(seed)
    w = [(r.standard_normal(s, np.float32) * np.float32(STD)) for s in ((c["F"], c["D"]), (c["F"], c["D"]), (c["D"], c["F"]))]
    return w, 1 + 0.1 * r.standard_normal(c["D"], np.float32), r.standard_normal((c["M"], c["D"]), np.float32)


def _in_graph_sdpa(c, seed):
    g = _gen(seed)
    return [_randn(g, 1, h, c["S"], c["D"]) for h in (c["H"], c["KV"], c["KV"])]


# ----------------------------------------------------------------------------- prepare
def prepare(case, seed):
    c, kind = case, case["kind"]
    from aneforge_amd import _kernels as K
    st = {"c": c}
    if kind == "linear":
        ws, xs = _in_linear(c, seed)
        split = torch.empty(8 * c["M"] * c["N"], dtype=torch.float32, device="cuda")
        ys = [torch.empty((c["M"], c["N"]), dtype=torch.float16, device="cuda") for _ in ws]
        st.update(out=ys, keep=(ws, xs, split), graph=_Captured(
            lambda: [K.linear(c["fmt"], w, s, x, y=y, ws=split) for (w, s), x, y in zip(ws, xs, ys)]))
    elif kind == "decode_attn":
        ins = _in_decode_attn(c, seed)
        outs = [torch.empty_like(q) for q, _, _ in ins]
        ws = torch.zeros(K.attn_ws_bytes(c["B"], c["H"], c["KV"], c["D"], c["ctx"]) // 4 + 1, dtype=torch.float32, device="cuda")
        st.update(out=outs, keep=(ins, ws), graph=_Captured(
            lambda: [K.decode_attn(q, k, v, o=o, ctx_len=c["ctx"], ws=ws) for (q, k, v), o in zip(ins, outs)]))
    elif kind == "decode":
        raw = _raw_model(c, seed)
        eng = _engine(raw, c["D"], c["KV"], c["F"], c["V"], c["pos"] + c["steps"] + 8)
        for mixer, _ in eng.layers:
            mixer.kc[0, :, :c["pos"]], mixer.vc[0, :, :c["pos"]] = _cache_rows(raw["g"], c["KV"], c["pos"])
        if c["sampled"]:
            eng.set_sampling(0.8, 0.9, 40, [0.5], c["steps"] - 1)
        else:
            eng._graphs()
        st.update(eng=eng, tokens=raw["tokens"])
    elif kind == "prompt":
        raw = _raw_model(c, seed)
        st.update(eng=_engine(raw, c["D"], c["KV"], c["F"], c["V"], c["n"] + 8), tokens=raw["tokens"])
    elif kind in ("attn_block", "mlp_block"):
        L, x0, (k0, v0) = _in_block(c, seed)
        from aneforge_amd import _engine as E
        from aneforge_amd.llm import LlamaConfig
        D, pos0, m = c["D"], c.get("pos0", 0), c["m"]
        cfg = LlamaConfig(dim=D, n_layers=1, n_heads=D // 128, n_kv_heads=c.get("KV", 1), ffn_dim=c.get("F", 256), vocab=64, norm_eps=EPS)
        embed = torch.zeros((64, D), dtype=torch.float16, device="cuda")
        head = E.Linear("fp16", embed, None, 64, D)
        # the half of the layer that the case leaves out gets a small stand-in
        qkv, wo = (_linear(L["qkv"]), _linear(L["wo"])) if kind == "attn_block" else (head, head)
        gu, down = (_linear(L["gu"]), _linear(L["down"])) if kind == "mlp_block" else (head, head)
        mixer, mlp = E.AttentionDecode.from_linears(cfg, qkv, wo, L["an"]), E.SwiGLUDecode.from_linears(cfg, gu, down, L["mn"])
        eng = E.DecodeEngine(cfg, [(mixer, mlp)], embed, head, L["an"], pos0 + m + 8,
                             rope_tables=_rope_tables(pos0 + m + 8, 128))
        if kind == "attn_block" and pos0:
            mixer.kc[0, :, :pos0], mixer.vc[0, :, :pos0] = k0, v0
        st.update(eng=eng, layer=mixer if kind == "attn_block" else mlp, x0=x0, x=torch.empty_like(x0), bufs=eng._prefill_buffers(m))
    elif kind == "moe":
        experts, router, norm, h0 = _in_moe(c, seed)
        from aneforge_amd import moe
        from aneforge_amd._engine import QuantizedWeight
        from aneforge_amd.llm import LayerSpec, LlamaConfig
        D, F = c["D"], c["F"]
        cpu = lambda t: t.cpu().numpy()
        qw = lambda t, n, k: QuantizedWeight(c["fmt"], cpu(t[0]), cpu(t[1]), (n, k))
        lw = {"mlp_norm": cpu(norm), "router": cpu(router), "wgate_exps": [qw(e[0], F, D) for e in experts],
              "wup_exps": [qw(e[1], F, D) for e in experts], "wdown_exps": [qw(e[2], D, F) for e in experts]}
        del experts
        cfg = LlamaConfig(dim=D, n_layers=1, n_heads=D // 128, n_kv_heads=D // 128, ffn_dim=F, vocab=64, norm_eps=EPS,
                          extra={"n_experts": c["E"], "n_experts_per_tok": c["k"], "norm_topk_prob": True})
        layer = moe.MoEDecode(lw, cfg, LayerSpec(mlp="moe"), None)
        st.update(layer=layer, bufs=layer._make_bufs(c["T"]), h0=h0, h=torch.empty_like(h0))
    elif kind == "graph_mlp":
        import aneforge_amd as af
        (wg, wu, wd), gamma, x = _in_graph_mlp(c, seed)
        t = af.input((c["M"], c["D"]))
        n = t.rms_norm(gamma, EPS)
        st.update(model=af.compile(t + (n.linear(wg).silu() * n.linear(wu)).linear(wd), compress=c["compress"]), x=x)
    else:
        import aneforge_amd as af
        ins = _in_graph_sdpa(c, seed)
        ports = [af.input(tuple(t.shape)) for t in ins]
        m = af.compile(af.sdpa(*ports, is_causal=c["causal"]))
        for (name, _), t in zip(m._inputs, ins):
            m.input_view(name).copy_(t)
        torch.cuda.synchronize()
        st["model"] = m
    return st


# ----------------------------------------------------------------------------- run
def run(st):
    c, kind = st["c"], st["c"]["kind"]
    if kind in ("linear", "decode_attn"):
        st["graph"].launch()
        return st["out"]
    if kind == "decode":
        eng = st["eng"]
        eng.reset(st["tokens"], pos0=c["pos"], zero_state=False)
        if c["sampled"]:
            eng.run(c["steps"] - 1, 0)
            eng.run_sampled(1)
        else:
            eng.run(c["steps"] - 1, 1)
        return eng.logits
    if kind == "prompt":
        eng = st["eng"]
        eng.prefill(st["tokens"])
        with torch.cuda.stream(eng.stream):
            eng.enqueue_layers()
            eng.enqueue_head()
        return eng.logits
    if kind in ("attn_block", "mlp_block"):
        st["x"].copy_(st["x0"])
        st["layer"].prefill(st["eng"], st["x"], c.get("pos0", 0), st["bufs"])
        return [st["x"], st["layer"].kc, st["layer"].vc] if kind == "attn_block" else st["x"]
    if kind == "moe":
        st["h"].copy_(st["h0"])
        st["layer"].run(st["h"], st["bufs"])
        return st["h"]
    if kind == "graph_mlp":
        return st["model"](st["x"])
    st["model"].execute()
    return st["model"].output_view()


# ----------------------------------------------------------------------------- 64-bit results
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        ws, xs = _in_linear(c, seed)
        return [_matmul(x.double(), c["fmt"], w, s) for (w, s), x in zip(ws, xs)]
    if kind == "decode_attn":
        return [torch.stack([_attend(q[b:b + 1].double(), k[b].double(), v[b].double(), c["ctx"] - 1)[0] for b in range(c["B"])])
                for q, k, v in _in_decode_attn(c, seed)]
    if kind in ("decode", "prompt"):
        raw = _raw_model(c, seed)
        pos0 = c.get("pos", 0)
        n = len(raw["tokens"])
        H, KV = c["D"] // 128, c["KV"]
        x = raw["embed"][raw["tokens"]].double()
        cos, sin = (torch.from_numpy(t).cuda().double() for t in _rope_tables(pos0 + n, 128))
        for L in raw["layers"]:
            kc, vc = (torch.zeros((KV, pos0 + n, 128), dtype=torch.float64, device="cuda") for _ in range(2))
            if pos0:
                k0, v0 = _cache_rows(raw["g"], KV, pos0)
                kc[:, :pos0], vc[:, :pos0] = k0.double(), v0.double()
            x = _mlp64(_attn64(x, L, kc, vc, pos0, H, KV, cos, sin), L)
        return _rms(x[-1:], raw["fn"]) @ raw["head"].double().T
    if kind in ("attn_block", "mlp_block"):
        L, x0, (k0, v0) = _in_block(c, seed)
        if kind == "mlp_block":
            return _mlp64(x0.double(), L)
        KV, pos0, M = c["KV"], c["pos0"], c["pos0"] + c["m"] + 8
        kc, vc = (torch.zeros((KV, M, 128), dtype=torch.float64, device="cuda") for _ in range(2))
        kc[:, :pos0], vc[:, :pos0] = k0.double(), v0.double()
        cos, sin = (torch.from_numpy(t).cuda().double() for t in _rope_tables(M, 128))
        return [_attn64(x0.double(), L, kc, vc, pos0, c["D"] // 128, KV, cos, sin), kc[None], vc[None]]
    if kind == "moe":
        experts, router, norm, h0 = _in_moe(c, seed)
        hn = _rms(h0.double(), norm).half().double()
        # routing as it is defined: fp16 probabilities, the lowest index among exact ties
        p = (hn @ router.double().T).softmax(-1).half().double()
        order = torch.sort(-p, dim=-1, stable=True).indices[:, :c["k"]]
        gate = torch.gather(p, 1, order)
        gate = gate / gate.sum(-1, keepdim=True)
        out = h0.double()
        for e, (wg, wu, wd) in enumerate(experts):
            t, slot = (order == e).nonzero(as_tuple=True)
            if t.numel():
                a = torch.nn.functional.silu(_matmul(hn[t], c["fmt"], *wg)) * _matmul(hn[t], c["fmt"], *wu)
                out[t] += gate[t, slot, None] * _matmul(a, c["fmt"], *wd)
        return out
    if kind == "graph_mlp":
        (wg, wu, wd), gamma, x = _in_graph_mlp(c, seed)
        q = lambda w: _compressed(w, c["compress"])
        x = x.astype(np.float16).astype(np.float64)
        n = x / np.sqrt((x * x).mean(-1, keepdims=True) + EPS) * gamma.astype(np.float16)
        g, u = n @ q(wg).T, n @ q(wu).T
        return x + (g / (1 + np.exp(-g)) * u) @ q(wd).T
    q, k, v = (t[0].double() for t in _in_graph_sdpa(c, seed))
    return _attend(q.transpose(0, 1), k, v, 0 if c["causal"] else c["S"]).transpose(0, 1)[None]


def _compressed(w, compress):
    """A host weight as its encoding holds it: int8 codes and an fp16 scale per row, or per 32 weights."""
    if compress is None:
        return w.astype(np.float16).astype(np.float64)
    r = w.reshape(-1, w.shape[1] if compress == "int8" else 32)
    s = np.maximum(np.abs(r).max(1, keepdims=True) / np.float32(127), np.float32(1e-8))
    q = np.clip(np.rint(r / s), -127, 127)
    v = q.astype(np.float64) * s.astype(np.float16).astype(np.float64)
    return (v if compress == "int8" else v.astype(np.float16).astype(np.float64)).reshape(w.shape)


# ----------------------------------------------------------------------------- work and tolerance
def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        n = c["calls"]
        return {"bytes": n * (_wbytes(c["fmt"], c["N"], c["K"]) + 2 * c["M"] * (c["N"] + c["K"])), "flops": 2 * n * c["M"] * c["N"] * c["K"]}
    if kind == "decode_attn":
        n = c["calls"] * c["B"] * c["D"]
        return {"bytes": 4 * n * (c["KV"] * c["ctx"] + c["H"]), "flops": 4 * n * c["H"] * c["ctx"]}
    if kind in ("decode", "prompt"):
        D, F, nkv = c["D"], c["F"], c["KV"] * 128
        fmt, n = c.get("fmt", "int8"), c.get("n", c.get("steps"))
        pos = c.get("pos", 0)
        elems = c["layers"] * (2 * D * D + 2 * nkv * D + 3 * F * D)
        wb = sum(_wbytes(fmt, *s) for s in ((D + 2 * nkv, D), (D, D), (2 * F, D), (D, F))) * c["layers"]
        rows = sum(pos + i + 1 for i in range(n))
        kv = 4 * c["layers"] * nkv
        # decode steps read the weights and the cache once each; a prompt reads the weights twice
        # (all but its last token together, then the last)
        reads, kvb = (n, kv * rows) if kind == "decode" else (2, 2 * kv * n)
        return {"bytes": reads * wb + kvb + 2 * c["V"] * D + 2 * n * D, "flops": 2 * n * elems + 4 * c["layers"] * D * rows + 2 * c["V"] * D}
    if kind == "attn_block":
        D, m, p, nkv = c["D"], c["m"], c["pos0"], c["KV"] * 128
        return {"bytes": _wbytes(c["fmt"], D + 2 * nkv, D) + _wbytes(c["fmt"], D, D) + 4 * m * D + 4 * nkv * (p + m),
                "flops": 2 * m * D * (2 * D + 2 * nkv) + 4 * D * sum(p + i + 1 for i in range(m))}
    if kind == "mlp_block":
        D, F, m = c["D"], c["F"], c["m"]
        return {"bytes": _wbytes(c["fmt"], 2 * F, D) + _wbytes(c["fmt"], D, F) + 4 * m * D, "flops": 6 * m * D * F}
    if kind == "moe":
        D, F, n = c["D"], c["F"], c["T"] * c["k"]
        active = c["E"] * (1 - (1 - c["k"] / c["E"]) ** c["T"])              # experts that some token routes to
        return {"bytes": active * (_wbytes(c["fmt"], 2 * F, D) + _wbytes(c["fmt"], D, F)) + 4 * c["T"] * D, "flops": 6 * n * D * F}
    if kind == "graph_mlp":
        D, F, M = c["D"], c["F"], c["M"]
        fmt = c["compress"] or "fp16"
        return {"bytes": 2 * _wbytes(fmt, F, D) + _wbytes(fmt, D, F) + 8 * M * D, "flops": 6 * M * D * F}
    S = c["S"]
    return {"bytes": 4 * c["D"] * S * (c["H"] + c["KV"]), "flops": 4 * c["H"] * c["D"] * (S * (S + 1) // 2 if c["causal"] else S * S)}


def tolerance(case):
    kind = case["kind"]
    # about four times the distance from the 64-bit results: fp16 outputs of one fp32-accumulated
    # product or softmax are 2e-4 from them, blocks, which round a few more times in fp16 between their
    # products, 3e-4 to 5e-4, and whole models, which pass those roundings through every layer, up to 6e-3
    rel = {"linear": 1e-3, "decode_attn": 1e-3, "graph_sdpa": 2e-3, "attn_block": 2e-3, "mlp_block": 2e-3, "moe": 2e-3, "graph_mlp": 2e-3,
           "decode": 2e-2, "prompt": 2e-2}[kind]
    return {"rel": rel}
