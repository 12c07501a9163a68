"""float32 attention on the bf16 matrix core (three bf16 parts of each value):
against float64 and the float32 kernel, the launch plan, and the values the
parts cannot hold."""
import numpy as np
import pytest

from browsergrad_amd import _native as N

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def bridge():
    from browsergrad_amd.bridge import HipRealizerBridge
    with HipRealizerBridge(device=0) as br:
        yield br


def _run(br, hs, **kw):
    br.set_launch_log(True)
    br.take_launch_log()
    h = br.attention_ex(*hs, in_dtype="float32", out_dtype="float32", **kw)
    log = br.take_launch_log()
    br.set_launch_log(False)
    y = br.to_numpy(h)
    br.release(h)
    return y, log


def _truth(q, k, v, scale, causal):
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    with np.errstate(all="ignore"):
        s = q @ k.transpose(0, 1, 3, 2) * scale
        if causal:
            s = np.where(np.triu(np.ones(s.shape[-2:], bool), 1), -np.inf, s)
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        return p @ v, p @ np.abs(v)


# Two tiles and more, ragged key and query counts, more queries than keys, every
# padded head dim, odd head dims (4-byte loads), one workgroup and many.
@pytest.mark.parametrize("b,h,sq,sk,d", [(1, 1, 5, 65, 64), (2, 3, 128, 128, 16), (1, 2, 130, 200, 64), (1, 2, 300, 97, 32),
                                         (2, 2, 64, 200, 7), (1, 1, 257, 257, 33), (4, 12, 1000, 1000, 64),
                                         (1, 3, 31, 1025, 48), (3, 1, 96, 128, 24)])
@pytest.mark.parametrize("causal", [False, True])
def test_split_attention(bridge, b, h, sq, sk, d, causal):
    rng = np.random.default_rng(sq + sk + d)
    q, k, v = (rng.standard_normal((b, h, n, d)).astype(F32) for n in (sq, sk, sk))
    hs = [bridge.upload(t, t.shape, "float32") for t in (q, k, v)]
    kw = dict(batch=b, heads=h, sq=sq, sk=sk, d=d, scale=d ** -0.5, causal=causal)
    y, log = _run(bridge, hs, **kw)
    from browsergrad_amd.semantic import launch_plan
    a = N.AttentionDesc()
    a.batch, a.heads, a.sq, a.sk, a.d, a.causal = b, h, sq, sk, d, int(causal)
    a.in_dtype = a.out_dtype = N.BG_F32
    plan = launch_plan("attention", a)["launches"]
    assert "split_fa32_fwd_kernel" in log[0]["kernel"] and plan[0]["family"] == "split_fa32_fwd_kernel"
    assert [(r["grid"], r["block"]) for r in log] == [(e["grid"], e["block"]) for e in plan]
    truth, mass = _truth(q, k, v, d ** -0.5, causal)
    # scores carry sqrt(D) roundings of |q||k|/sqrt(D) (about 1e-6), sums sqrt(Sk)
    assert np.all(np.abs(y - truth) <= (4e-6 + 2.0 * np.sqrt(sk) * 2.0 ** -24) * mass)
    old, log = _run(bridge, hs, tiled=True, **kw)
    assert "split" not in log[0]["kernel"]
    err = [np.linalg.norm(t - truth) / np.linalg.norm(truth) for t in (y, old)]
    assert err[0] <= 1.05 * err[1] + 2.0 ** -25, err
    for x in hs:
        bridge.release(x)


# One round of 256 workgroups, one workgroup more with few and with more than
# three key tiles a query block, and causal averages of 3 and 11 / 3 tiles.
@pytest.mark.parametrize("h,sq,sk,causal,family", [
    (256, 128, 128, False, "split_fa32_fwd_kernel"), (257, 128, 128, False, "fa32_fwd_kernel"),
    (260, 8, 192, False, "fa32_fwd_kernel"), (260, 8, 193, False, "split_fa32_fwd_kernel"),
    (130, 256, 256, True, "fa32_fwd_kernel"), (130, 320, 320, True, "split_fa32_fwd_kernel")])
def test_kernel_choice(bridge, h, sq, sk, causal, family):
    d = 8
    rng = np.random.default_rng(h + sk)
    q, k, v = (rng.standard_normal((1, h, n, d)).astype(F32) for n in (sq, sk, sk))
    hs = [bridge.upload(t, t.shape, "float32") for t in (q, k, v)]
    y, log = _run(bridge, hs, batch=1, heads=h, sq=sq, sk=sk, d=d, scale=d ** -0.5, causal=causal)
    from browsergrad_amd.semantic import launch_plan
    a = N.AttentionDesc()
    a.batch, a.heads, a.sq, a.sk, a.d, a.causal = 1, h, sq, sk, d, int(causal)
    a.in_dtype = a.out_dtype = N.BG_F32
    plan = launch_plan("attention", a)["launches"]
    assert plan[0]["family"] == family and f"{len(family)}{family}" in log[0]["kernel"]
    assert [(r["grid"], r["block"]) for r in log] == [(e["grid"], e["block"]) for e in plan]
    truth, mass = _truth(q, k, v, d ** -0.5, causal)
    assert np.all(np.abs(y - truth) <= (4e-6 + 2.0 * np.sqrt(sk) * 2.0 ** -24) * mass)


def test_split_attention_mask_and_views(bridge):
    """An additive mask (with a row of -inf, which gives zeros) and Q, K, V as
    views of one projection with an odd head dim."""
    b, h, s, d = 2, 3, 150, 64
    rng = np.random.default_rng(2)
    q, k, v = (rng.standard_normal((b, h, s, d)).astype(F32) for _ in range(3))
    mask = rng.uniform(-0.5, 0.5, (b, 1, s, s)).astype(F32)
    mask[rng.random(mask.shape) < 0.05] = -np.inf
    mask[:, :, 5] = -np.inf
    hs = [bridge.upload(t, t.shape, "float32") for t in (q, k, v, mask)]
    y = bridge.to_numpy(bridge.flash_attention(*hs, b, h, s, s, d, 0.125, "float32"))
    sc = q.astype(np.float64) @ k.astype(np.float64).transpose(0, 1, 3, 2) * 0.125 + mask
    m = sc.max(-1, keepdims=True)
    p = np.exp(sc - np.where(np.isfinite(m), m, 0))
    truth = p @ v.astype(np.float64) / np.where(m == -np.inf, 1, p.sum(-1, keepdims=True))
    assert np.all(y[:, :, 5] == 0) and np.max(np.abs(y - truth)) <= 2e-5
    B, S, H, D = 2, 150, 3, 21
    x = rng.standard_normal((B, S, 3, H, D)).astype(F32)
    hx = bridge.upload(x, x.shape, "float32")
    st = (S * 3 * H * D, D, 3 * H * D)
    y, log = _run(bridge, (hx, hx, hx), batch=B, heads=H, sq=S, sk=S, d=D, scale=0.3, causal=True, q_view=(0, *st),
                  k_view=(H * D, *st), v_view=(2 * H * D, *st), o_strides=(S * H * D, D, H * D))
    assert "split_fa32_fwd_kernel" in log[0]["kernel"]
    truth, mass = _truth(*(np.ascontiguousarray(x[:, :, i].transpose(0, 2, 1, 3)) for i in range(3)), 0.3, True)
    assert np.all(np.abs(y.reshape(B, S, H, D).transpose(0, 2, 1, 3) - truth) <= 1e-5 * mass)


@pytest.mark.parametrize("d", [7, 16, 32, 33, 64])
@pytest.mark.parametrize("causal", [False, True])
def test_redo_is_the_float32_kernel(bridge, d, causal):
    """A workgroup that met a NaN gives the float32 kernel's bits, every padded
    head dim and both kinds of load; the other head does not notice."""
    rng = np.random.default_rng(d)
    b, h, s = 1, 2, 300
    q, k, v = (rng.standard_normal((b, h, s, d)).astype(F32) for _ in range(3))
    kw = dict(batch=b, heads=h, sq=s, sk=s, d=d, scale=d ** -0.5, causal=causal)
    hs = [bridge.upload(t, t.shape, "float32") for t in (q, k, v)]
    clean, _ = _run(bridge, hs, **kw)
    v[0, 0, 0, d - 1] = np.nan  # every query of the head sees it
    hs[2] = bridge.upload(v, v.shape, "float32")
    y, log = _run(bridge, hs, **kw)
    t, _ = _run(bridge, hs, tiled=True, **kw)
    assert "split_fa32_fwd_kernel" in log[0]["kernel"] and np.isnan(t[0, 0, :, d - 1]).all()
    assert np.array_equal(y[0, 0], t[0, 0], equal_nan=True) and np.array_equal(y[0, 1], clean[0, 1])


@pytest.mark.parametrize("e", [-100, -115, -120])
def test_split_attention_small_values(bridge, e):
    """V, or K with Q scaled up, at 2^-100 to 2^-120: the bits of the unscaled
    call, since such values take no other path."""
    rng = np.random.default_rng(4)
    b, h, s, d = 1, 2, 200, 64
    q, k, v = (rng.uniform(1, 2, (b, h, s, d)).astype(F32) * rng.choice([-1, 1], (b, h, s, d)).astype(F32)
               for _ in range(3))
    kw = dict(batch=b, heads=h, sq=s, sk=s, d=d, scale=2.0 ** -4)

    def run(*x):
        hs = [bridge.upload(t, t.shape, "float32") for t in x]
        y, log = _run(bridge, hs, **kw)
        assert "split_fa32_fwd_kernel" in log[0]["kernel"]
        for t in hs:
            bridge.release(t)
        return y.astype(np.float64)

    base = run(q, k, v)
    f = F32(2.0 ** e)
    assert np.array_equal(run(q * F32(2.0 ** 60), k * f, v), run(q * F32(2.0 ** (60 + e)), k, v))
    y = run(q, k, v * f)
    normal = np.abs(y) >= 2.0 ** -126  # (below, the result itself rounds)
    assert np.array_equal(y[normal], (base * 2.0 ** e)[normal]) and np.mean(normal) > 0.9


def test_split_attention_small_weights(bridge):
    """Weights of 2^-122 of the largest, whose key has V = 0, keep their bits: the
    scores' roundings (122 * 2^-24, times ln 2) and a few units bound the error."""
    s, d = 130, 64
    rng = np.random.default_rng(6)
    q, k = np.zeros((1, 1, 8, d), F32), np.zeros((1, 1, s, d), F32)
    q[..., 0] = 1
    k[0, 0, 1:, 0] = -122 * np.log(2) + rng.uniform(-1, 1, s - 1)
    v = rng.uniform(1, 2, (1, 1, s, d)).astype(F32)
    v[0, 0, 0] = 0
    hs = [bridge.upload(t, t.shape, "float32") for t in (q, k, v)]
    y, log = _run(bridge, hs, batch=1, heads=1, sq=8, sk=s, d=d, scale=1.0)
    assert "split_fa32_fwd_kernel" in log[0]["kernel"]
    truth, _ = _truth(q, k, v, 1.0, False)
    assert np.all(np.abs(y - truth) <= (123 * 3 + 8) * 2.0 ** -24 * truth)


@pytest.mark.parametrize("what", ["nan_k", "inf_v", "neg_inf_k", "tiny_v", "tiny_k", "huge_q"])
def test_split_attention_special_values(bridge, what):
    """What the parts cannot hold, and tiny values, give what the float32 kernel gives."""
    rng = np.random.default_rng(8)
    b, h, s, d = 1, 2, 140, 64
    q, k, v = (rng.standard_normal((b, h, s, d)).astype(F32) for _ in range(3))
    if what == "nan_k":
        k[0, 0, 70, 3] = np.nan
    elif what == "inf_v":
        v[0, 1, 3, 7] = np.inf
    elif what == "neg_inf_k":
        q[..., 0], k[0, 0, 9, 0] = 1, -np.inf
    elif what == "tiny_v":
        v[0, 0] *= F32(2.0 ** -130)
    elif what == "tiny_k":
        k[0, 0] *= F32(2.0 ** -120)
    else:
        q[0, 0, 4] *= F32(3e37)
    hs = [bridge.upload(t, t.shape, "float32") for t in (q, k, v)]
    kw = dict(batch=b, heads=h, sq=s, sk=s, d=d, scale=0.125)
    y, log = _run(bridge, hs, **kw)
    t, _ = _run(bridge, hs, tiled=True, **kw)
    assert "split_fa32_fwd_kernel" in log[0]["kernel"]
    assert np.array_equal(np.isnan(y), np.isnan(t)) and np.array_equal(np.isposinf(y), np.isposinf(t))
    fin = np.isfinite(t)
    _, mass = _truth(q, k, np.where(np.isfinite(v), v, 0), 0.125, False)
    if what != "huge_q":  # (scores of 1e37 round to 1e30: any order of their sum picks the same key only by luck)
        ok = fin & np.isfinite(mass)
        assert np.all(np.abs(y[ok].astype(np.float64) - t[ok]) <= 2e-5 * mass[ok] + 2.0 ** -148)
