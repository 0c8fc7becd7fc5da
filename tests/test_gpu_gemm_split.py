"""The split GEMM (every packed format, row tiles, K slices and K groups) and the grouped experts on it,
against fp64 products with the oracle's dequantised weights.

Bar: an output differs from the fp64 product by its own rounding (half an fp16 ulp, 2^-11 relative) and
by the fp32 accumulation, at most K * 2^-24 of the sum of the terms' magnitudes; the SwiGLU epilogue
rounds gate and up to fp16 first and takes the repository's fp16 bar."""
import os

import numpy as np
import pytest

from _util import check_f16, check_hidden, dev, host, say
from oracle import ref

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

FMTS = ["int8", "q4_0", "fp16", "blockwise", "lut4", "q4_k", "q6_k"]


@pytest.fixture(scope="module")
def K():
    from aneforge_amd import _kernels
    return _kernels


def _weights(K, fmt, N, Kd, rng):
    """(codes, scale, fp64 weights) of a random [N, Kd] matrix on the device."""
    if fmt == "int8":
        q = rng.integers(-127, 128, (N, Kd), dtype=np.int8)
        s = (np.abs(rng.normal(0, 0.02, N)) / 127 + 1e-5).astype(np.float16)
        return dev(q), dev(s), ref.dequant_w8(q, s).astype(np.float64)
    if fmt == "fp16":
        w = (rng.standard_normal((N, Kd)) * 0.02).astype(np.float16)
        return dev(w), None, w.astype(np.float64)
    if fmt == "blockwise":
        q = rng.integers(-127, 128, (N, Kd), dtype=np.int8)
        s = (np.abs(rng.normal(0, 0.02, (N, Kd // 32))) / 127 + 1e-5).astype(np.float16)
        return dev(q), dev(s), ref.dequant_blockwise(q, s).astype(np.float64)
    if fmt == "lut4":
        packed = rng.integers(0, 256, (N, Kd // 2), dtype=np.uint8)
        cb = np.sort(rng.normal(0, 0.02, (N, 16)), axis=1).astype(np.float16)
        idx = np.empty((N, Kd), np.int64)
        idx[:, 0::2], idx[:, 1::2] = packed & 15, packed >> 4
        return dev(packed), dev(cb), np.take_along_axis(cb.astype(np.float64), idx, axis=1)
    if fmt == "q4_0":
        b = ref.quantize_q4_0((rng.standard_normal((N, Kd)) * 0.05).astype(np.float32))
        return (*K.q4_repack(dev(b), N, Kd), ref.dequant_q4_0_f16(b, N, Kd).astype(np.float64))
    nb = N * Kd // 256
    if fmt == "q4_k":
        b = rng.integers(0, 256, (nb, 144), dtype=np.uint8)
        b[:, :4] = (np.abs(rng.standard_normal((nb, 2))) * 0.0005 + 1e-5).astype(np.float16).view(np.uint8).reshape(nb, 4)
        b = b.reshape(N, -1)
        return (*K.q4_k_repack(dev(b), N, Kd), ref.dequant_q4_k_f16(b, N, Kd).astype(np.float16).astype(np.float64))
    b = rng.integers(0, 256, (nb, 210), dtype=np.uint8)
    b[:, 208:210] = (np.abs(rng.standard_normal(nb)) * 0.0005 + 1e-5).astype(np.float16).view(np.uint8).reshape(nb, 2)
    b = b.reshape(N, -1)
    return (*K.q6_k_repack(dev(b), N, Kd), ref.dequant_q6_k_f16(b, N, Kd).astype(np.float16).astype(np.float64))


def _bound(x, W, want):
    mag = np.abs(x.astype(np.float64)) @ np.abs(W).T
    return np.abs(want) * 2.0 ** -11 + mag * W.shape[1] * 2.0 ** -24 + 2.0 ** -24


# (slices, features / 32, row tiles / 16): every kernel built, the slice counts around the K = 1280 row's ten
# chunks (one short slice, one chunk each), and more than one row tile
CONFIGS = [(1, 2, 1), (3, 4, 1), (10, 2, 2), (2, 4, 2), (4, 2, 3), (1, 4, 3), (16, 2, 4), (1, 4, 4), (3, 2, 6), (2, 4, 6),
           (1, 2, 8), (7, 4, 8)]


@pytest.mark.parametrize("fmt", FMTS)
def test_every_tile_and_slice_count(K, fmt, monkeypatch):
    rng = np.random.default_rng(len(fmt))
    N, Kd = 16 * 17, 1280                                   # a ragged feature tile, K not a power of two
    w, s, W = _weights(K, fmt, N, Kd, rng)
    ws = torch.empty(16 * 256 * 512, dtype=torch.float32, device="cuda")
    cfgs = CONFIGS + ([(1, 8, 4), (2, 8, 6)] if fmt in ("int8", "q4_0") else []) + ([(1, 8, 8), (5, 8, 8)] if fmt == "int8" else [])
    for S, nw, mt in cfgs:
        M = 16 * mt + 5 if S % 2 else 16 * mt - 3           # past one row tile, and short of it
        x = rng.standard_normal((M, Kd)).astype(np.float16)
        want = x.astype(np.float64) @ W.T
        say(f"gemm_split {fmt} M={M} N={N} K={Kd} slices={S} nw={nw} mt={mt}")
        monkeypatch.setenv("AFX_GEMM_SPLIT", f"{S}.{nw}.{mt}")
        y = torch.full((M, N), 7.0, dtype=torch.float16, device="cuda")
        K.gemm_split(fmt, w, s, dev(x), y, ws=ws)
        got = host(y)
        assert (np.abs(got - want) <= _bound(x, W, want)).all(), (S, nw, mt)
        again = torch.empty_like(y)
        K.gemm_split(fmt, w, s, dev(x), again, ws=ws)       # the slices' sum has a fixed order
        assert np.array_equal(host(again).view(np.uint16), got.view(np.uint16))


@pytest.mark.parametrize("fmt", ["int8", "q4_k"])
@pytest.mark.parametrize("cfg", ["1.2.2", "5.4.2"])
@pytest.mark.parametrize("ldy_pad", [0, 5])                 # 5: rows that take no 8- or 16-byte stores
def test_epilogues(K, fmt, cfg, ldy_pad, monkeypatch):
    monkeypatch.setenv("AFX_GEMM_SPLIT", cfg)
    rng = np.random.default_rng(7 + ldy_pad)
    M, N, Kd = 37, 96, 768
    w, s, W = _weights(K, fmt, N, Kd, rng)
    x = rng.standard_normal((M, Kd)).astype(np.float16)
    xp = torch.zeros((M, Kd + 16), dtype=torch.float16, device="cuda")
    xp[:, :Kd] = dev(x)
    bias = (rng.standard_normal(N) * 0.1).astype(np.float16)
    r = rng.standard_normal((M, N)).astype(np.float16)
    ws = torch.empty(8 * 128 * 64, dtype=torch.float32, device="cuda")
    lin = x.astype(np.float64) @ W.T
    say(f"gemm_split epilogues {fmt} cfg={cfg} ldy+{ldy_pad}")

    def out(cols, dtype=torch.float16):
        return torch.zeros((M, cols + ldy_pad), dtype=dtype, device="cuda")[:, :cols]
    y = K.gemm_split(fmt, w, s, xp[:, :Kd], out(N), bias=dev(bias), ws=ws)
    want = lin + bias.astype(np.float64)
    assert (np.abs(host(y) - want) <= _bound(x, W, want) + np.abs(lin) * 2.0 ** -23).all()
    y = K.gemm_split(fmt, w, s, xp[:, :Kd], out(N, torch.float32), epi="f32", ws=ws)
    assert (np.abs(host(y) - lin) <= _bound(x, W, lin)).all()
    y = out(N)
    y.copy_(dev(r))
    K.gemm_split(fmt, w, s, xp[:, :Kd], y, residual=y, epi="resid", ws=ws)
    check_hidden(host(y), ref.r16(r.astype(np.float64) + ref.r16(lin)), what="resid")
    y = K.gemm_split(fmt, w, s, xp[:, :Kd], out(N // 2), epi="swiglu", ws=ws)
    check_f16(host(y), ref.r16(ref.silu(ref.r16(lin[:, 0::2])) * ref.r16(lin[:, 1::2])), what="swiglu")


def test_workspace_limits_the_slices_and_bad_shapes_raise(K, monkeypatch):
    rng = np.random.default_rng(3)
    w, s, W = _weights(K, "int8", 64, 512, rng)
    x = rng.standard_normal((20, 512)).astype(np.float16)
    want = x.astype(np.float64) @ W.T
    monkeypatch.setenv("AFX_GEMM_SPLIT", "4.2.2")
    per = 2 * 2 * 2048                                      # bytes of one slice: mt * nw * 2 KB tiles
    for nbytes in (0, 2 * per, 3 * per + 8, 4 * per):
        ws = torch.empty(nbytes // 4, dtype=torch.float32, device="cuda") if nbytes else None
        guard = torch.full((20, 64), 7.0, dtype=torch.float16, device="cuda")
        y = K.gemm_split("int8", w, s, dev(x), guard, ws=ws)
        assert (np.abs(host(y) - want) <= _bound(x, W, want)).all(), nbytes
    with pytest.raises(RuntimeError, match="K %"):
        K.gemm_split("int8", w[:, :64].contiguous(), s, dev(x[:, :64].copy()), torch.empty((20, 64), dtype=torch.float16, device="cuda"))
    monkeypatch.delenv("AFX_GEMM_SPLIT")
    assert K.gemm_split_plan("int8", 20, 64, 64) == (False, 0)      # K = 64: afx_gemm's
    assert K.gemm_split_plan("q4_0", 64, 4096, 4096)[0]


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("E,T,k", [(3, 70, 2), (130, 33, 2), (5, 4, 3), (20, 4, 3)])
def test_grouped_experts(K, fmt, E, T, k):
    """Skewed routing: one expert takes every token (several row tiles), others one row, some none; 130
    experts need more than one pass over the counts; 4 tokens where the format has no skinny MFMA kernel (the
    K-quants with the 20 experts only)."""
    rng = np.random.default_rng(E + T)
    D, F = 512, 256
    say(f"grouped experts {fmt} E={E} T={T} k={k}")
    used = [E - 1] + [int(e) for e in rng.choice(E - 1, min(E - 1, 4), replace=False)]
    pick = [[E - 1] + [int(e) for e in rng.choice(used[1:], k - 1, replace=False)] for _ in range(T)]
    cnt, lst = np.zeros(E, np.int32), np.zeros((E, T), np.int32)
    for t in range(T):
        for sl, e in enumerate(pick[t]):
            lst[e, cnt[e]] = t * k + sl
            cnt[e] += 1
    gu, gus, G = [], [], {}
    dn, dns, Dn = [], [], {}
    zero_g, zero_d = _weights(K, fmt, 2 * F, D, rng), _weights(K, fmt, D, F, rng)
    for e in range(E):
        a, b = (_weights(K, fmt, 2 * F, D, rng), _weights(K, fmt, D, F, rng)) if e in used else (zero_g, zero_d)
        gu.append(a[0]); gus.append(a[1]); G[e] = a[2]
        dn.append(b[0]); dns.append(b[1]); Dn[e] = b[2]
    cat = lambda ts: None if ts[0] is None else torch.cat(ts)
    x = (rng.standard_normal((T, D)) * 0.5).astype(np.float16)
    act = K.moe_gateup(fmt, cat(gu), cat(gus), dev(x), k, E, F, dev(cnt), dev(lst))
    a = host(act)
    y = host(K.moe_down(fmt, cat(dn), cat(dns), act, T, k, E, F, D, dev(cnt), dev(lst)))
    for t in range(T):
        for sl, e in enumerate(pick[t]):
            lin = ref.r16(x[t].astype(np.float64) @ G[e].T)
            i = t * k + sl
            check_f16(a[i], ref.r16(ref.silu(lin[0::2]) * lin[1::2]), what=f"gate/up token {t} expert {e}")
            want = a[i].astype(np.float64) @ Dn[e].T
            assert (np.abs(y[i] - want) <= _bound(a[i][None], Dn[e], want[None])[0]).all(), (t, e)


@pytest.mark.parametrize("T,E,k", [(33, 8, 2), (300, 8, 2), (65, 130, 4), (64, 3, 3)])
def test_topk_lists_of_many_tokens(K, T, E, k):
    """More than 32 tokens: the gates, choices and lists are those of the one-workgroup form on 32 tokens
    at a time, joined in token order."""
    say(f"moe_topk T={T} E={E} k={k}")
    rng = np.random.default_rng(T)
    lg = np.round(rng.standard_normal((T, E)).astype(np.float32), 1)     # ties
    gate, sel, cnt, lst = (host(t) for t in K.moe_topk(dev(lg), k, True))
    gates, sels, joined = [], [], [[] for _ in range(E)]
    for t0 in range(0, T, 32):
        g, s, c, l = (host(t) for t in K.moe_topk(dev(lg[t0:t0 + 32]), k, True))
        gates.append(g); sels.append(s)
        for e in range(E):
            joined[e] += [int(i) + t0 * k for i in l[e, :c[e]]]
    assert np.array_equal(gate.view(np.uint32), np.concatenate(gates).view(np.uint32))
    assert np.array_equal(sel, np.concatenate(sels))
    for e in range(E):
        assert cnt[e] == len(joined[e]) and lst[e, :cnt[e]].tolist() == joined[e]


@pytest.mark.parametrize("M", [17, 300])
def test_router_rows_past_16(K, M):
    """A linear with few outputs and many rows: the row groups run in workgroups of their own."""
    say(f"fp16 router rows M={M}")
    rng = np.random.default_rng(M)
    w, _, W = _weights(K, "fp16", 8, 4096, rng)
    x = rng.standard_normal((M, 4096)).astype(np.float16)
    want = x.astype(np.float64) @ W.T
    got = host(K.linear("fp16", w, None, dev(x), out_f32=True))
    assert (np.abs(got - want) <= _bound(x, W, want)).all()


@pytest.mark.parametrize("M,N,Kd,epi", [(4000, 4096, 64, "f16"), (257, 272, 128, "resid"), (300, 2320, 192, "swiglu"),
                                        (2000, 5504, 128, "f32")])
def test_gemm_256_tiles(K, M, N, Kd, epi):
    """fp16 weights over 256 x 256 tiles (AFX_GEMM_WL=7; the default where they fill the chip, as in the
    first shape) against the 128 x 128 form: the same sums in the same order, so the same bytes, with
    ragged rows and columns and an odd and an even number of K steps."""
    rng = np.random.default_rng(M + N)
    w = dev((rng.standard_normal((N, Kd)) * 0.05).astype(np.float16))
    x = dev(rng.standard_normal((M, Kd)).astype(np.float16))
    r = rng.standard_normal((M, N)).astype(np.float16)
    outs, old = [], os.environ.get("AFX_GEMM_WL")
    try:
        for wl in (None, "6", "7"):
            os.environ.pop("AFX_GEMM_WL", None)
            if wl:
                os.environ["AFX_GEMM_WL"] = wl
            say(f"gemm 256 tiles M={M} N={N} K={Kd} {epi} WL={wl}")
            y = dev(r) if epi == "resid" else None
            outs.append(host(K.gemm("fp16", w, None, x, y=y, residual=y, epi=epi)))
    finally:
        os.environ.pop("AFX_GEMM_WL", None)
        if old is not None:
            os.environ["AFX_GEMM_WL"] = old
    np.testing.assert_array_equal(outs[0], outs[1])
    np.testing.assert_array_equal(outs[2], outs[1])


@pytest.mark.parametrize("compress", [None, "int8", "int4", "blockwise"])
@pytest.mark.parametrize("rows", [17, 64])
def test_compiled_matmul_rows(compress, rows):
    """A compiled graph's matmuls of 17 and 64 rows, two of them sharing the program's workspace, against
    the same matmuls row by row in batches of 16 (the linear kernels): both within their own rounding of
    the fp64 product, so within two fp16 ulps and the two accumulations' bound of each other."""
    import aneforge_amd as af
    rng = np.random.default_rng(rows)
    D, F = 512, 2048
    w1 = (rng.standard_normal((F, D)) / np.sqrt(D)).astype(np.float32)
    w2 = (rng.standard_normal((D, F)) / np.sqrt(F)).astype(np.float32)

    def net(n):
        x = af.input((n, D))
        h = x.linear(w1)
        return af.compile(h.relu().linear(w2), compress=compress, compress_atol=1.0)
    x = rng.standard_normal((rows, D)).astype(np.float16)
    say(f"compiled matmul rows={rows} {compress}")
    full = net(rows)
    got = [np.asarray(full(x)) for _ in range(3)]
    part = net(16)
    pad = np.concatenate([x, np.zeros((-rows % 16, D), np.float16)])
    want = np.concatenate([np.asarray(part(pad[i:i + 16])) for i in range(0, len(pad), 16)])[:rows]
    np.testing.assert_array_equal(got[1], got[0])
    np.testing.assert_array_equal(got[2], got[0])
    # an intermediate that rounds the other way moves by an ulp (2^-10 relative at most) and its share of
    # an output is a sum of such moves over F terms: sqrt(F / 2) * 2^-10 * |h| |w| at 6 deviations
    tol = 6 * np.sqrt(F / 2) * 2.0 ** -10 * np.abs(want).std() / np.sqrt(F) * 2 + 2.0 ** -10 * np.abs(want)
    assert (np.abs(got[0] - want) <= tol).all()


def test_three_rows_with_scales_off_the_mfma_alignment(K):
    """3 rows of a large int8 matrix take the skinny MFMA kernel only where its 8-byte scale loads do."""
    rng = np.random.default_rng(5)
    N, Kd = 2048, 4096
    w, s, W = _weights(K, "int8", N, Kd, rng)
    off = torch.empty(N + 1, dtype=torch.float16, device="cuda")[1:]
    off.copy_(s)
    x = rng.standard_normal((3, Kd)).astype(np.float16)
    want = x.astype(np.float64) @ W.T
    for sc in (s, off):
        say(f"int8 3 rows scale at {sc.data_ptr() % 16}")
        assert (np.abs(host(K.linear("int8", w, sc, dev(x))) - want) <= _bound(x, W, want)).all()


def test_codebook_rows_past_the_split_range(K):
    """Activation rows that span 2 GiB (a stride of 2^27) stay on the vector kernels, in two launches."""
    rng = np.random.default_rng(6)
    w, s, W = _weights(K, "lut4", 16, 256, rng)
    x = rng.standard_normal((9, 256)).astype(np.float16)
    wide = torch.empty((9, 1 << 27), dtype=torch.float16, device="cuda")[:, :256]
    wide.copy_(dev(x))
    want = x.astype(np.float64) @ W.T
    say("lut4 9 rows, row stride 2^27")
    assert (np.abs(host(K.linear("lut4", w, s, wide)) - want) <= _bound(x, W, want)).all()


@pytest.mark.parametrize("fmt", ["int8", "q4_0", "blockwise"])
def test_three_rows_that_span_2_gib(K, fmt):
    """3 rows of a large matrix on a stride of 400 M elements stay on the vector kernel, as 2 rows do."""
    rng = np.random.default_rng(7)
    w, s, W = _weights(K, fmt, 2048, 4096, rng)
    x = rng.standard_normal((3, 4096)).astype(np.float16)
    wide = torch.empty((3, 400_000_000), dtype=torch.float16, device="cuda")[:, :4096]
    wide.copy_(dev(x))
    want = x.astype(np.float64) @ W.T
    say(f"{fmt} 3 rows, row stride 400M")
    got = host(K.linear(fmt, w, s, wide))
    assert (np.abs(got - want) <= _bound(x, W, want)).all()
    np.testing.assert_array_equal(got[:2], host(K.linear(fmt, w, s, wide[:2])))


@pytest.mark.parametrize("slices", [1, 3])
def test_unused_infinite_codebook_entry(K, slices, monkeypatch):
    """Entry 0 is infinite and no weight names it: the slices' odd last chunks must not bring it in."""
    monkeypatch.setenv("AFX_GEMM_SPLIT", f"{slices}.2.1")
    rng = np.random.default_rng(8)
    N, Kd = 64, 128 * 9
    idx = rng.integers(1, 16, (N, Kd))
    packed = (idx[:, 0::2] | (idx[:, 1::2] << 4)).astype(np.uint8)
    cb = rng.normal(0, 0.02, (N, 16)).astype(np.float16)
    cb[:, 0] = np.inf
    W = np.take_along_axis(cb.astype(np.float64), idx, axis=1)
    x = rng.standard_normal((7, Kd)).astype(np.float16)
    want = x.astype(np.float64) @ W.T
    say(f"lut4 infinite entry, {slices} slices")
    y = torch.empty((7, N), dtype=torch.float16, device="cuda")
    K.gemm_split("lut4", dev(packed), dev(cb), dev(x), y, ws=torch.empty(1 << 16, dtype=torch.float32, device="cuda"))
    assert (np.abs(host(y) - want) <= _bound(x, W, want)).all()


def test_misaligned_weights_keep_their_kernels():
    """A plan is taken only for weights and scales on 16 bytes; the workspace keeps what it outgrew."""
    from aneforge_amd import _engine as E
    w = torch.zeros((4096, 4096), dtype=torch.int8, device="cuda")
    s = torch.zeros(4097, dtype=torch.float16, device="cuda")
    assert E.split_plan(E.Linear("int8", w, s[:4096], 4096, 4096), 64)[0]
    assert E.split_plan(E.Linear("int8", w, s[1:], 4096, 4096), 64) == (False, 0)
    eng = E.DecodeEngine.__new__(E.DecodeEngine)
    a = eng.gemm_scratch(1000)
    assert eng.gemm_scratch(500) is a
    b = eng.gemm_scratch(1004)
    assert b.numel() >= 2 * a.numel() and eng._gws[0] is a


@pytest.mark.parametrize("fmt,M,N,Kd", [("fp16", 128, 2048, 512), ("q4_k", 100, 4096, 2816), ("blockwise", 200, 2816, 512),
                                        ("q6_k", 512, 5632, 256), ("int8", 300, 5504, 512)])
def test_planned_tiles(K, fmt, M, N, Kd):
    """The plan's own tile and slices, with the workspace it asks for, on both sides of one and two workgroups per CU."""
    rng = np.random.default_rng(M)
    w, s, W = _weights(K, fmt, N, Kd, rng)
    x = rng.standard_normal((M, Kd)).astype(np.float16)
    n = K.gemm_split_plan(fmt, M, N, Kd)[1]
    want = x.astype(np.float64) @ W.T
    say(f"planned {fmt} M={M} N={N} K={Kd} workspace {n}")
    y = torch.empty((M, N), dtype=torch.float16, device="cuda")
    K.gemm_split(fmt, w, s, dev(x), y, ws=torch.empty(n // 4, dtype=torch.float32, device="cuda") if n else None)
    assert (np.abs(host(y) - want) <= _bound(x, W, want)).all()


@pytest.mark.parametrize("fmt,M,N,Kd", [("fp16", 8, 4096, 11008), ("fp16", 16, 512, 5120), ("fp16", 3, 2048, 5632),
                                        ("q4_k", 8, 1024, 4096), ("lut4", 5, 512, 5120), ("q6_k", 11, 256, 2048)])
def test_few_rows_without_a_workspace_keep_the_faster_kernel(K, fmt, M, N, Kd):
    """Without a workspace K is not cut, and these rows are faster on the kernels that take any N: the same
    bytes as the first N - 4 features by themselves, which only those kernels take."""
    rng = np.random.default_rng(N + M)
    w, s, W = _weights(K, fmt, N, Kd, rng)
    x = rng.standard_normal((M, Kd)).astype(np.float16)
    say(f"few rows without a workspace {fmt} M={M} N={N} K={Kd}")
    y = host(K.linear(fmt, w, s, dev(x), out_f32=True))
    part = host(K.linear(fmt, w[:N - 4], None if s is None else s[:N - 4], dev(x), out_f32=True))
    want = x.astype(np.float64) @ W.T
    assert (np.abs(y - want) <= _bound(x, W, want)).all()
    np.testing.assert_array_equal(y[:, :N - 4], part)


@pytest.mark.parametrize("fmt,M,N,Kd,cfg", [("q4_k", 8, 8192, 2048, "1.2.1"), ("lut4", 16, 8192, 2048, "1.2.1"), ("q6_k", 20, 8192, 2048, "1.2.1")])
def test_few_rows_without_a_workspace_take_an_uncut_tile(K, fmt, M, N, Kd, cfg, monkeypatch):
    """Where the split GEMM is the faster without a workspace too, it takes the tile that is best uncut (64
    features), not the one its slices would want: the bytes of that tile."""
    rng = np.random.default_rng(N + M)
    w, s, W = _weights(K, fmt, N, Kd, rng)
    x = rng.standard_normal((M, Kd)).astype(np.float16)
    say(f"uncut tile {fmt} M={M} N={N} K={Kd}")
    want = x.astype(np.float64) @ W.T
    y = host(K.linear(fmt, w, s, dev(x), out_f32=True))
    assert (np.abs(y - want) <= _bound(x, W, want)).all()
    monkeypatch.setenv("AFX_GEMM_SPLIT", cfg)
    fixed = torch.empty((M, N), dtype=torch.float32, device="cuda")
    np.testing.assert_array_equal(y, host(K.gemm_split(fmt, w, s, dev(x), fixed, epi="f32")))


@pytest.mark.parametrize("fmt,M,cfg", [("lut4", 20, "2.8"), ("int8", 20, "1.8"), ("q4_0", 130, "1.8.8"), ("fp16", 20, "1.2.5")])
def test_override_that_no_kernel_has(K, fmt, M, cfg, monkeypatch):
    """A fixed choice for which no kernel is built: the plan's own, by its bytes."""
    rng = np.random.default_rng(M)
    N, Kd = 272, 512
    w, s, W = _weights(K, fmt, N, Kd, rng)
    x = rng.standard_normal((M, Kd)).astype(np.float16)
    ws = torch.empty(1 << 18, dtype=torch.float32, device="cuda")
    run = lambda: host(K.gemm_split(fmt, w, s, dev(x), torch.full((M, N), 7.0, dtype=torch.float32, device="cuda"), epi="f32", ws=ws))
    want = run()
    exact = x.astype(np.float64) @ W.T
    assert (np.abs(want - exact) <= _bound(x, W, exact)).all()
    say(f"override {cfg} {fmt} M={M}")
    monkeypatch.setenv("AFX_GEMM_SPLIT", cfg)
    np.testing.assert_array_equal(run(), want)


def _with_sentinel(K, fmt, w, s, x, W, nbytes, what):
    """gemm_split with the first nbytes of a larger buffer as its workspace: the result, and nothing written past them."""
    buf = torch.full((nbytes // 4 + (1 << 21),), 7.0, dtype=torch.float32, device="cuda")
    n = nbytes // 4
    say(f"{what} workspace {nbytes}")
    y = K.gemm_split(fmt, w, s, dev(x), torch.empty((x.shape[0], W.shape[0]), dtype=torch.float16, device="cuda"), ws=buf[:n] if n else None)
    want = x.astype(np.float64) @ W.T
    assert (np.abs(host(y) - want) <= _bound(x, W, want)).all(), what
    assert bool((buf[n:] == 7.0).all()), what
    return buf[:n]


@pytest.mark.parametrize("M", [20, 5])
def test_slices_stay_inside_the_workspace(K, M, monkeypatch):
    """Fixed to four slices of 2 x 2 tiles: none, two, three or all of them as the workspace holds them."""
    rng = np.random.default_rng(M)
    w, s, W = _weights(K, "int8", 64, 512, rng)
    x = rng.standard_normal((M, 512)).astype(np.float16)
    monkeypatch.setenv("AFX_GEMM_SPLIT", "4.2.2")
    per = 2 * 2 * 128 * min(M, 16)                          # bytes of one slice
    for nbytes, slices in ((0, 1), (2 * per, 2), (3 * per + 8, 3), (4 * per, 4)):
        ws = _with_sentinel(K, "int8", w, s, x, W, nbytes, f"M={M} slices={slices}")
        if slices > 1:                                      # the last slice that fits is written
            assert bool((ws[(slices - 1) * per // 4:slices * per // 4] != 7.0).any())


@pytest.mark.parametrize("fmt,M,N,Kd", [("fp16", 100, 1024, 2816), ("q4_k", 100, 4096, 2816), ("blockwise", 40, 3072, 3072),
                                        ("q6_k", 5, 4096, 4096), ("int8", 13, 2048, 4096), ("lut4", 16, 4096, 2048), ("q4_0", 64, 4096, 4096)])
def test_planned_slices_stay_inside_the_planned_workspace(K, fmt, M, N, Kd):
    """The plan's own slices, with exactly the bytes that it asks for, and with half of them."""
    rng = np.random.default_rng(M + 1)
    w, s, W = _weights(K, fmt, N, Kd, rng)
    x = rng.standard_normal((M, Kd)).astype(np.float16)
    nbytes = K.gemm_split_plan(fmt, M, N, Kd)[1]
    assert nbytes > 0                                       # a shape whose K is cut
    _with_sentinel(K, fmt, w, s, x, W, nbytes, f"planned {fmt} M={M}")
    _with_sentinel(K, fmt, w, s, x, W, nbytes // 32 * 16, f"half {fmt} M={M}")


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("cfg", ["1.2.1", "3.4.2"])
def test_rows_keep_to_themselves(K, fmt, cfg, monkeypatch):
    """Rows of NaN and infinities, the last one (which rows past the end repeat) among them, leave the bytes of
    the others as they are."""
    monkeypatch.setenv("AFX_GEMM_SPLIT", cfg)
    rng = np.random.default_rng(11)
    M, N, Kd = 37, 272, 1280
    w, s, _ = _weights(K, fmt, N, Kd, rng)
    x = rng.standard_normal((M, Kd)).astype(np.float16)
    ws = torch.empty(1 << 18, dtype=torch.float32, device="cuda")
    say(f"rows keep to themselves {fmt} {cfg}")
    run = lambda a: host(K.gemm_split(fmt, w, s, dev(a), torch.empty((M, N), dtype=torch.float32, device="cuda"), epi="f32", ws=ws))
    clean = run(x)
    odd = [3, 16, M - 1]
    x[3], x[16, 1279], x[M - 1, 5] = np.nan, np.inf, -np.inf
    got = run(x)
    rest = np.delete(np.arange(M), odd)
    np.testing.assert_array_equal(got[rest], clean[rest])
    assert not np.isfinite(got[odd].astype(np.float64)).all()
    assert np.isnan(got[3]).all()
