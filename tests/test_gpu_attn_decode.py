"""Attention of a few query rows: the streaming kernel against float64 and the
tiled kernels."""
import numpy as np
import pytest

from browsergrad_amd import _native as N
from oracle import ops as O

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def bridge():
    from browsergrad_amd.bridge import HipRealizerBridge
    with HipRealizerBridge(device=0) as br:
        yield br


def _put(br, x, dtype):
    """(handle, the values it holds in float64)"""
    if dtype == "bfloat16":
        bits = O.f32_to_bf16_bits(x)
        return br.upload(bits, x.shape, dtype), O.bf16_bits_to_f32(bits).astype(np.float64)
    y = x.astype(dtype)
    return br.upload(y, x.shape, dtype), y.astype(np.float64)


def _run(br, hs, dtype, **kw):
    br.set_launch_log(True)
    br.take_launch_log()
    h = br.attention_ex(*hs, in_dtype=dtype, out_dtype="float32", **kw)
    log = br.take_launch_log()
    br.set_launch_log(False)
    y = br.to_numpy(h)
    br.release(h)
    return y, log


# One key block and less, a run that no wavefront step divides, key slices
# (few heads, long runs), every number of rows, head dims below 64.
@pytest.mark.parametrize("b,h,sq,sk,d", [(1, 1, 1, 64, 64), (2, 3, 1, 65, 64), (8, 12, 1, 1024, 64), (3, 1, 2, 515, 32),
                                         (1, 2, 3, 1000, 8), (2, 2, 4, 129, 48), (1, 12, 1, 4099, 64),
                                         (1, 1, 4, 20000, 64), (64, 16, 1, 100, 64)])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("causal", [False, True])
def test_decode_attention(bridge, b, h, sq, sk, d, dtype, causal):
    rng = np.random.default_rng(sk + d)
    (hq, q), (hk, k), (hv, v) = (_put(bridge, rng.standard_normal((b, h, n, d)).astype(F32), dtype)
                                 for n in (sq, sk, sk))
    kw = dict(batch=b, heads=h, sq=sq, sk=sk, d=d, scale=d ** -0.5, causal=causal)
    y, log = _run(bridge, (hq, hk, hv), dtype, **kw)
    streams = dtype == "float32" or sq <= 2  # more 16-bit rows run on the matrix cores
    assert all(("attention_decode" in r["kernel"]) == streams for r in log), log
    if not streams:  # checked against its own bound with the tiled kernels' tests
        return
    if dtype == "float32":
        from browsergrad_amd.semantic import launch_plan
        a = N.AttentionDesc()
        a.batch, a.heads, a.sq, a.sk, a.d, a.causal = b, h, sq, sk, d, int(causal)
        a.in_dtype = a.out_dtype = N.BG_F32
        assert [(r["grid"], r["block"]) for r in log] == [(e["grid"], e["block"])
                                                         for e in launch_plan("attention", a)["launches"]]
    s = q @ k.transpose(0, 1, 3, 2) * d ** -0.5
    if causal:
        s = np.where(np.triu(np.ones((sq, sk), bool), 1), -np.inf, s)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    truth, mass = p @ v, p @ np.abs(v)
    # P is rounded to the operands' type; sums are float32 (scores within 1e-5)
    u = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8, "float32": 0.0}[dtype]
    assert np.all(np.abs(y - truth) <= (u + 3e-5) * mass)
    tiled, log = _run(bridge, (hq, hk, hv), dtype, tiled=True, **kw)
    assert not any("attention_decode" in r["kernel"] for r in log)
    err = [np.linalg.norm(t - truth) / np.linalg.norm(truth) for t in (y, tiled)]
    assert err[0] <= 1.05 * err[1] + 2.0 ** -23, err
    for x in (hq, hk, hv):
        bridge.release(x)


# Heads on both sides of one a CU, runs of keys on both sides of a step of four
# and eight wavefronts (32 16-bit or 16 float32 rows each) and of the 512 rule.
@pytest.mark.parametrize("h,sk,waves", [(256, 64, 8), (5, 255, 8), (5, 257, 8), (256, 512, 8), (256, 513, 16),
                                        (257, 64, 4), (300, 127, 4), (300, 129, 4), (257, 513, 4), (5, 129, 8)])
@pytest.mark.parametrize("dtype,sq", [("float16", 1), ("bfloat16", 2), ("float32", 1), ("float32", 3)])
def test_decode_wavefronts(bridge, h, sk, waves, dtype, sq):
    if dtype == "float32":
        waves = 8 if h > 256 and sq > 2 or sk <= 128 else 16
    d = 24
    rng = np.random.default_rng(sk)
    (hq, q), (hk, k), (hv, v) = (_put(bridge, rng.standard_normal((1, h, n, d)).astype(F32), dtype)
                                 for n in (sq, sk, sk))
    y, log = _run(bridge, (hq, hk, hv), dtype, batch=1, heads=h, sq=sq, sk=sk, d=d, scale=d ** -0.5)
    assert len(log) == 1 and "attention_decode_kernel" in log[0]["kernel"] and log[0]["block"][0] == 64 * waves
    if dtype == "float32":
        from browsergrad_amd.semantic import launch_plan
        a = N.AttentionDesc()
        a.batch, a.heads, a.sq, a.sk, a.d = 1, h, sq, sk, d
        a.in_dtype = a.out_dtype = N.BG_F32
        assert [(r["grid"], r["block"]) for r in log] == [(e["grid"], e["block"])
                                                         for e in launch_plan("attention", a)["launches"]]
    s = q @ k.transpose(0, 1, 3, 2) * d ** -0.5
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    u = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8, "float32": 0.0}[dtype]
    assert np.all(np.abs(y - p @ v) <= (u + 3e-5) * (p @ np.abs(v)))
    for x in (hq, hk, hv):
        bridge.release(x)


def test_decode_attention_views_and_rounded_scores(bridge):
    """K and V inside one [B, S, 2, H, D] cache, output [B, Sq, H, D]; and two
    scores that round to one 16-bit value share their weight."""
    b, sk, h, d = 2, 200, 3, 64
    rng = np.random.default_rng(4)
    cache, q = rng.standard_normal((b, sk, 2, h, d)).astype(np.float16), rng.standard_normal((b, 2, h, d)).astype(np.float16)
    hc, hq = bridge.upload(cache, cache.shape, "float16"), bridge.upload(q, q.shape, "float16")
    st = (sk * 2 * h * d, d, 2 * h * d)
    y, log = _run(bridge, (hq, hc, hc), "float16", batch=b, heads=h, sq=2, sk=sk, d=d, scale=0.125,
                  q_view=(0, 2 * h * d, d, h * d), k_view=(0, *st), v_view=(h * d, *st), o_strides=(2 * h * d, d, h * d))
    assert "attention_decode_kernel" in log[0]["kernel"]
    q64, k64, v64 = (t.astype(np.float64).transpose(0, 2, 1, 3) for t in (q, cache[:, :, 0], cache[:, :, 1]))
    s = q64 @ k64.transpose(0, 1, 3, 2) * 0.125
    p = np.exp(s - s.max(-1, keepdims=True))
    truth = (p / p.sum(-1, keepdims=True) @ v64).transpose(0, 2, 1, 3)
    assert np.all(np.abs(y.reshape(truth.shape) - truth) <= 2.0 ** -10 * 4)
    one = np.zeros((1, 1, 1, 64), np.float16)
    one[..., :2] = 1
    k, v = np.full((1, 1, 64, 64), 0, np.float16), np.zeros((1, 1, 64, 64), np.float16)
    k[0, 0, :, 0] = -1024
    k[0, 0, 0, :2], k[0, 0, 1, :2], v[0, 0, 0], v[0, 0, 1] = (1024, 1024), (1025, 1024), 1, -1
    hs = [bridge.upload(t, t.shape, "float16") for t in (one, k, v)]
    kw = dict(batch=1, heads=1, sq=1, sk=64, d=64, scale=1 / 64)
    assert np.all(_run(bridge, hs, "float16", round_scores=True, **kw)[0] == 0)
    assert np.all(_run(bridge, hs, "float16", **kw)[0] < 0)


def test_decode_attention_special_values(bridge):
    """NaN scores reach the output; float32 scores below -1e20 leave the
    reference's zeros; an infinite key wins nothing when its score is -inf."""
    q, k, v = np.ones((1, 3, 1, 4), F32), np.ones((1, 3, 70, 4), F32), np.ones((1, 3, 70, 4), F32)
    k[0, 0, 5, 0], k[0, 1], k[0, 2, 7, 0] = np.nan, -1e25, -np.inf
    hs = [bridge.upload(t, t.shape, "float32") for t in (q, k, v)]
    kw = dict(batch=1, heads=3, sq=1, sk=70, d=4, scale=1.0)
    y, log = _run(bridge, hs, "float32", **kw)
    t, _ = _run(bridge, hs, "float32", tiled=True, **kw)
    assert "attention_decode_kernel" in log[0]["kernel"]
    assert np.array_equal(np.isnan(y), np.isnan(t)) and np.isnan(y[0, 0]).all()
    assert np.all(y[0, 1] == 0) and np.all(t[0, 1] == 0)
    assert np.allclose(y[0, 2], t[0, 2], atol=1e-6) and np.allclose(y[0, 2], 1)
