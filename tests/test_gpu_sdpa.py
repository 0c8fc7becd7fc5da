"""afx_sdpa (many queries, plain and causal) against fp64 attention, and against the decode kernel it stands in
for.  Bar: the fp16 output's own rounding (2^-11 relative) plus 2^-12 of the largest |v| seen: both
kernels' scores and sums are fp32, whose exponents move a weight by at most about |score| * 2^-23 * 4."""
import numpy as np
import pytest

from _util import dev, host, say

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _want(q, k, v, scale, causal):
    H, Sq, D = q.shape
    Hkv, Skv = k.shape[:2]
    out = np.empty((H, Sq, D))
    for h in range(H):
        s = q[h].astype(np.float64) @ k[h * Hkv // H].astype(np.float64).T * scale
        if causal:
            s[np.arange(Skv)[None] > np.arange(Sq)[:, None] + Skv - Sq] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        vv = v[h * Hkv // H].astype(np.float64)
        out[h] = np.einsum("qk,kd->qd", p, np.where(np.isfinite(vv), vv, 0))
    return out


def _run(q, k, v, scale, causal):
    from aneforge_amd import _kernels as K
    o = torch.full(q.shape, 7.0, dtype=torch.float16, device="cuda")
    return host(K.sdpa(dev(q), dev(k), dev(v), o, scale, causal))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,Hkv,Sq,Skv,causal", [(1, 1, 1, 1, True), (2, 1, 16, 16, True), (4, 2, 63, 63, True), (3, 3, 64, 64, False),
                                                 (2, 2, 65, 65, True), (4, 1, 130, 130, True), (2, 2, 200, 321, False), (2, 1, 40, 300, True),
                                                 (1, 1, 17, 129, False), (8, 8, 257, 257, True)])
def test_matches_fp64(D, H, Hkv, Sq, Skv, causal):
    say(f"sdpa H={H} Hkv={Hkv} Sq={Sq} Skv={Skv} D={D} causal={causal}")
    rng = np.random.default_rng(D + Sq + Skv)
    q = rng.standard_normal((H, Sq, D)).astype(np.float16)
    k, v = (rng.standard_normal((Hkv, Skv, D)).astype(np.float16) for _ in range(2))
    for scale in (1.0 / D ** 0.5, -0.3, 1.0):               # plain, negative, peaked
        want = _want(q, k, v, scale, causal)
        got = _run(q, k, v, scale, causal)
        assert (np.abs(got - want) <= np.abs(want) * 2.0 ** -11 + np.abs(v).max() * 2.0 ** -12).all(), scale


@pytest.mark.parametrize("causal", [False, True])
def test_no_less_precise_than_the_decode_kernel(causal):
    from aneforge_amd import _kernels as K
    H, Hkv, S, D = 8, 2, 300, 128
    say(f"sdpa precision S={S} causal={causal}")
    rng = np.random.default_rng(5)
    q = rng.standard_normal((H, S, D)).astype(np.float16)
    k, v = (rng.standard_normal((Hkv, S, D)).astype(np.float16) for _ in range(2))
    want = _want(q, k, v, D ** -0.5, causal)
    qd, kd, vd = dev(q), dev(k)[None], dev(v)[None]
    o = torch.empty_like(qd)
    K.decode_attn(qd, kd, vd, o=o, ctx_len=S, causal_off=0 if causal else -1, q_strides=(D, S * D), kv_strides=(0, S * D), B=S, Hq=H)
    err = [np.linalg.norm(x.astype(np.float64) - want) for x in (_run(q, k, v, D ** -0.5, causal), host(o))]
    assert err[0] <= 1.01 * err[1]                          # both at the fp16 output's rounding


@pytest.mark.parametrize("D,Skv", [(64, 64), (128, 64), (128, 49)])
def test_weights_keep_their_fp32_bits(D, Skv):
    """Differences of nearly equal weights: a dimension adds one key's weight times 2^15 and takes off the
    next one's.  Scores are single fp16 products and the largest is 0, and the products and differences are
    exact, so what is off is the fp32 weights' own last places (a hundred of them make a difference): as far
    as the decode kernel's, up to how those happen to round.  Weights of 22 bits are off by ten times that."""
    from aneforge_amd import _kernels as K
    Sq = 70
    say(f"sdpa weight bits D={D} Skv={Skv}")
    rng = np.random.default_rng(D + Skv)
    q, k, v = np.zeros((1, Sq, D), np.float16), np.zeros((1, Skv, D), np.float16), np.zeros((1, Skv, D), np.float16)
    q[0, :, 0] = rng.uniform(0.5, 2.0, Sq)
    for j in range((Skv - 1) // 2):
        a = np.float16(-rng.uniform(2.0 ** -8, 2.0 ** -5))
        k[0, 2 * j, 0], k[0, 2 * j + 1, 0] = a, np.nextafter(a, np.float16(0))
        v[0, 2 * j, j], v[0, 2 * j + 1, j] = 2.0 ** 15, -2.0 ** 15
    got = _run(q, k, v, 0.37, False).astype(np.float64)
    qd, kd, vd = dev(q), dev(k)[None], dev(v)[None]
    o = torch.empty_like(qd)
    K.decode_attn(qd, kd, vd, o=o, ctx_len=Skv, scale=0.37, q_strides=(D, Sq * D), kv_strides=(0, Skv * D), B=Sq, Hq=1)
    want = _want(q, k, v, 0.37, False)
    err = [np.linalg.norm(x.astype(np.float64) - want) / np.linalg.norm(want) for x in (got, host(o))]
    assert err[0] <= 1.5 * err[1], err


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_values_hidden_by_the_causal_mask_do_not_leak(bad):
    H, S, D = 2, 150, 64
    say(f"sdpa causal with v = {bad} in row 70")
    rng = np.random.default_rng(9)
    q, k, v = (rng.standard_normal((H, S, D)).astype(np.float16) for _ in range(3))
    v[:, 70, 3] = bad
    got = _run(q, k, v, D ** -0.5, True)
    want = _want(q, k, v, D ** -0.5, True)
    assert np.isfinite(got[:, :70]).all()
    assert (np.abs(got[:, :70] - want[:, :70]) <= np.abs(want[:, :70]) * 2.0 ** -11 + 4 * 2.0 ** -12).all()
    assert not np.isfinite(got[:, 70:, 3].astype(np.float64)).any()
    rest = np.delete(np.arange(D), 3)
    assert (np.abs(got[:, 70:][..., rest] - want[:, 70:][..., rest]) <= np.abs(want[:, 70:][..., rest]) * 2.0 ** -11 + 4 * 2.0 ** -12).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal,Sq,Skv", [(False, 70, 200), (True, 150, 150), (True, 40, 300), (False, 16, 33)])
def test_infinite_values_reach_the_queries_that_see_them(causal, Sq, Skv, D):
    """An infinity in v gives its sign in every query that sees it (two of opposite signs, or a NaN: NaN),
    in blocks that the mask cuts and in whole ones; as in the decode kernel."""
    from aneforge_amd import _kernels as K
    H, Hkv = 4, 2
    say(f"sdpa infinite values causal={causal} Sq={Sq} Skv={Skv} D={D}")
    rng = np.random.default_rng(Skv + D)
    q = rng.standard_normal((H, Sq, D)).astype(np.float16)
    k, v = (rng.standard_normal((Hkv, Skv, D)).astype(np.float16) for _ in range(2))
    v[0, 3, 1], v[0, 20, 5], v[0, 30, 5], v[1, 5, 9], v[1, Skv - 1, 2] = np.inf, np.inf, -np.inf, np.nan, -np.inf
    if Skv > 130:
        v[1, 100, 40], v[0, 129, 63] = np.inf, -np.inf
    seen = np.arange(Skv)[None] <= np.arange(Sq)[:, None] + (Skv - Sq if causal else Skv)
    want = _want(q, k, v, D ** -0.5, causal)                # finite values only: now the others
    for h in range(H):
        vv = v[h * Hkv // H].astype(np.float64)
        for key, d in zip(*np.nonzero(~np.isfinite(vv))):
            with np.errstate(invalid="ignore"):             # inf - inf: NaN
                want[h, seen[:, key], d] += vv[key, d]
    got = _run(q, k, v, D ** -0.5, causal)
    qd, kd, vd = dev(q), dev(k)[None], dev(v)[None]
    o = torch.empty_like(qd)
    K.decode_attn(qd, kd, vd, o=o, ctx_len=Skv, causal_off=Skv - Sq if causal else -1, q_strides=(D, Sq * D),
                  kv_strides=(0, Skv * D), B=Sq, Hq=H)
    fine = np.isfinite(want)
    for out, name in ((got, "sdpa"), (host(o), "decode")):
        np.testing.assert_array_equal(out[~fine].astype(np.float64), want[~fine], err_msg=name)
        assert (np.abs(out[fine] - want[fine]) <= np.abs(want[fine]) * 2.0 ** -11 + 5 * 2.0 ** -12).all(), name


def test_bad_arguments_raise():
    from aneforge_amd import _kernels as K
    t = torch.zeros((2, 16, 32), dtype=torch.float16, device="cuda")
    with pytest.raises(RuntimeError, match="head dim 32"):
        K.sdpa(t, t, t, torch.empty_like(t), 1.0)
    q = torch.zeros((2, 20, 64), dtype=torch.float16, device="cuda")
    kv = torch.zeros((2, 16, 64), dtype=torch.float16, device="cuda")
    with pytest.raises(RuntimeError, match="bad lengths"):
        K.sdpa(q, kv, kv, torch.empty_like(q), 1.0, causal=True)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal,Sq,Skv,key", [(False, 70, 200, 3), (False, 70, 64, 63), (True, 150, 150, 149), (True, 150, 150, 70), (True, 40, 300, 5)])
def test_nan_scores_reach_the_queries_that_see_them(causal, Sq, Skv, key, D):
    """A NaN key row (also one that is all a query sees of its half) makes the queries that see it NaN, as in the
    decode kernel, and no others."""
    from aneforge_amd import _kernels as K
    H = 2
    say(f"sdpa NaN key {key} causal={causal} Sq={Sq} Skv={Skv} D={D}")
    rng = np.random.default_rng(key)
    q = rng.standard_normal((H, Sq, D)).astype(np.float16)
    k, v = (rng.standard_normal((H, Skv, D)).astype(np.float16) for _ in range(2))
    k[1, key, 7] = np.nan
    got = _run(q, k, v, D ** -0.5, causal)
    qd, kd, vd = dev(q), dev(k)[None], dev(v)[None]
    o = torch.empty_like(qd)
    K.decode_attn(qd, kd, vd, o=o, ctx_len=Skv, causal_off=Skv - Sq if causal else -1, q_strides=(D, Sq * D),
                  kv_strides=(0, Skv * D), B=Sq, Hq=H)
    nan = np.zeros(got.shape, bool)
    nan[1, max(0, key - (Skv - Sq)) if causal else 0:] = True
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(np.isnan(host(o)), nan)
