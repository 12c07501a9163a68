"""float32 GEMM on the bf16 matrix core (three bf16 parts of each value): every
tile shape and K split against float64, the launch plan, and the values the
parts cannot hold."""
import ctypes as C

import numpy as np
import pytest
import torch

from browsergrad_amd import _native as N

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def bridge():
    from browsergrad_amd.bridge import HipRealizerBridge
    with HipRealizerBridge(device=0) as br:
        yield br


def _gemm(br, a, b, trans_b, **kw):
    m, k = a.shape[-2:]
    n = b.shape[-2] if trans_b else b.shape[-1]
    hs = {x: br.upload(kw[x], kw[x].shape, "float32") for x in ("bias", "residual") if kw.get(x) is not None}
    ha, hb = br.upload(a, a.shape, "float32"), br.upload(b, b.shape, "float32")
    br.set_launch_log(True)
    br.take_launch_log()
    h = br.matmul_ex(ha, hb, m=m, n=n, k=k, trans_b=trans_b, **{**kw, **hs})
    log = br.take_launch_log()
    br.set_launch_log(False)
    y = br.to_numpy(h)
    for x in (ha, hb, h, *hs.values()):
        br.release(x)
    return y, log


def _plan(m, n, k, trans_b):
    d = N.MatmulDesc()
    d.batch, d.m, d.n, d.k = 1, m, n, k
    d.lda, d.ldb, d.ldc = k, k if trans_b else n, n
    d.trans_b, d.in_dtype, d.out_dtype = int(trans_b), N.BG_F32, N.BG_F32
    from browsergrad_amd.semantic import launch_plan
    return launch_plan("gemm", d)


# One of each tile shape (256 x 256, 256 x 128, 128 x 128, 64 x 128) with whole
# and ragged tiles, K slices, K of one step and less, rows that allow no
# 16-byte load, and a stage that K does not fill.
SHAPES = [(4096, 4096, 64), (4001, 4003, 37), (2047, 3072, 100), (1500, 1500, 1500), (512, 1024, 768), (200, 2100, 515),
          (65, 2200, 2049), (40, 3000, 700), (1, 9000, 500), (129, 65, 17), (300, 200, 5), (64, 128, 16)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("trans_b", [False, True])
def test_split_gemm_against_float64(bridge, m, n, k, trans_b):
    """Within the rounding bound of a K-term float32 sum, and in the 2-norm no
    further from float64 than the float32 matrix instruction (5% and half a
    rounding for the chance of the draw); the launches are the planned ones."""
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)).astype(F32)
    b = rng.standard_normal((n, k) if trans_b else (k, n)).astype(F32)
    bias, res = rng.standard_normal(n).astype(F32), rng.standard_normal((m, n)).astype(F32)
    y, log = _gemm(bridge, a, b, trans_b, bias=bias, act=N.ACT_RELU, residual=res)
    plan = _plan(m, n, k, trans_b)
    assert "gemm32_split_kernel" in log[0]["kernel"]
    assert [(r["grid"], r["block"]) for r in log] == [(e["grid"], e["block"]) for e in plan["launches"]]
    assert log[0]["staticLds"] == plan["ldsBytes"] or abs(log[0]["staticLds"] - plan["ldsBytes"]) <= 512
    a64, b64 = a.astype(np.float64), (b.T if trans_b else b).astype(np.float64)
    truth = np.maximum(a64 @ b64 + bias, 0) + res
    mass = np.abs(a64) @ np.abs(b64) + np.abs(bias) + np.abs(res)
    assert np.all(np.abs(y - truth) <= 2.0 * np.sqrt(k + 2) * 2.0 ** -24 * mass)
    plain, _ = _gemm(bridge, a, b, trans_b)
    unsplit, _ = _gemm(bridge, a, b, trans_b, f32_unsplit=True)
    truth = a64 @ b64
    err = [np.linalg.norm(v - truth) / np.linalg.norm(truth) for v in (plain, unsplit)]
    assert err[0] <= 1.05 * err[1] + 2.0 ** -25, err


@pytest.mark.parametrize("m,n", [(300, 200), (4096, 4096)])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("near", [0.0, 1 + 2.0 ** -8])
def test_few_terms_lose_no_precision(bridge, m, n, k, near):
    """Random values, and mantissas near 1 + 2^-8, whose dropped part products are
    largest (2^-24 of the product): K = 1 is the rounded product, up to K = 4 the
    float32 kernel runs, and from K = 5 on no error (2-norm, largest over the mass)
    is above the float32 kernel's."""
    rng = np.random.default_rng(k)

    def draw(*shape):
        if near == 0.0:
            return rng.standard_normal(shape).astype(F32)
        x = F32(near) + F32(2.0 ** -23) * rng.integers(-64, 0, shape).astype(F32)
        return x * rng.choice([-1, 1], shape).astype(F32)

    a, b = draw(m, k), draw(k, n)
    y, log = _gemm(bridge, a, b, False)
    if k == 1:
        assert np.array_equal(y, a * b)
    if k <= 4:
        assert "gemm32_kernel" in log[0]["kernel"]
        return
    assert "gemm32_split_kernel" in log[0]["kernel"]
    unsplit, _ = _gemm(bridge, a, b, False, f32_unsplit=True)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    truth, mass = a64 @ b64, np.abs(a64) @ np.abs(b64)
    err = [(np.linalg.norm(v - truth), np.max(np.abs(v - truth) / mass)) for v in (y, unsplit)]
    assert err[0][0] <= err[1][0] and err[0][1] <= err[1][1], err


def test_split_gemm_batched(bridge):
    """Batches of their own A and C, with B shared (stride 0) or their own."""
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((3, 130, 70)).astype(F32), rng.standard_normal((3, 70, 140)).astype(F32)
    for shared in (False, True):
        y, log = _gemm(bridge, a, b[0] if shared else b, False, batch=3, stride_b=0 if shared else 70 * 140)
        assert "gemm32_split_kernel" in log[0]["kernel"]
        truth = a.astype(np.float64) @ (b[:1] if shared else b).astype(np.float64)
        mass = np.abs(a).astype(np.float64) @ np.abs(b[:1] if shared else b).astype(np.float64)
        assert np.all(np.abs(y.reshape(truth.shape) - truth) <= 2.0 * np.sqrt(70) * 2.0 ** -24 * mass)


@pytest.mark.parametrize("m,n,k", [(70, 2100, 515), (300, 300, 40), (4096, 4096, 48)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_split_gemm_special_values(bridge, m, n, k, trans_b):
    """Infinities, NaNs, the largest values and values whose third part would
    fall below bf16's smallest step give what float32 products give."""
    rng = np.random.default_rng(9)
    a = rng.standard_normal((m, k)).astype(F32)
    b = rng.standard_normal((k, n)).astype(F32)
    a[3, 5], a[7, 1], a[11, 2], b[2, 9], b[k - 1, n - 1] = np.inf, np.nan, 3.4e38, -np.inf, -3.4e38
    a[20], b[:, 30] = 0, 0
    a[40] *= F32(2.0 ** -115)
    a[41] *= F32(2.0 ** -140)
    b[:, 50] *= F32(2.0 ** -120)
    bm = np.ascontiguousarray(b.T) if trans_b else b
    y, log = _gemm(bridge, a, bm, trans_b)
    assert "gemm32_split_kernel" in log[0]["kernel"]
    with np.errstate(all="ignore"):
        truth = a.astype(np.float64) @ b.astype(np.float64)
        mass = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
        f32 = truth.astype(F32)
    assert np.array_equal(np.isnan(y), np.isnan(f32))
    # (a sum within its own rounding of the largest float may go either way)
    clear = ~np.isnan(f32) & ((mass < 3e38) | ~np.isfinite(mass))
    assert np.array_equal(np.isposinf(y)[clear], np.isposinf(f32)[clear])
    assert np.array_equal(np.isneginf(y)[clear], np.isneginf(f32)[clear])
    fin = clear & np.isfinite(mass)
    bound = 2.0 * np.sqrt(k) * 2.0 ** -24 * mass[fin] + k * 2.0 ** -149
    assert np.all(np.abs(y[fin].astype(np.float64) - truth[fin]) <= bound)


@pytest.mark.parametrize("m,n,k", [(300, 300, 40), (1001, 1003, 37), (2048, 1027, 64), (4096, 4096, 48)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_redo_is_the_float32_kernel(bridge, m, n, k, trans_b):
    """A tile that met a NaN gives the float32 kernel's bits (the same order of
    sums); tiles that did not keep theirs."""
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, k)).astype(F32)
    b = rng.standard_normal((n, k) if trans_b else (k, n)).astype(F32)
    clean, _ = _gemm(bridge, a, b, trans_b)
    a[m - 1, k - 1] = np.nan
    y, log = _gemm(bridge, a, b, trans_b)
    unsplit, other = _gemm(bridge, a, b, trans_b, f32_unsplit=True)
    assert "gemm32_split_kernel" in log[0]["kernel"] and "gemm32_kernel" in other[0]["kernel"]
    tile = _plan(m, n, k, trans_b)["tile"][0]
    first = (m - 1) // tile * tile
    assert np.array_equal(y[first:], unsplit[first:], equal_nan=True) and np.isnan(y[m - 1]).all()
    assert np.array_equal(y[:first], clean[:first])


@pytest.mark.parametrize("e", [-100, -109, -115, -126, -135, -145])
@pytest.mark.parametrize("m,n,k", [(70, 2100, 515), (300, 300, 40), (4096, 4096, 48)])
def test_split_gemm_small_values(bridge, m, n, k, e):
    """Full 24-bit mantissas down to float32's subnormals, against a B scaled up:
    within the bound of float32 sums, element by element, and (where scaling loses
    no bits) the unscaled product's very bits: such values take no other path."""
    rng = np.random.default_rng(-e)
    base = rng.uniform(1, 2, (m, k)).astype(F32) * rng.choice([-1, 1], (m, k)).astype(F32)
    b = rng.standard_normal((k, n)).astype(F32)
    a = (base.astype(np.float64) * 2.0 ** e).astype(F32)
    up = b * F32(2.0 ** 60)
    y, log = _gemm(bridge, a, up, False)
    assert "gemm32_split_kernel" in log[0]["kernel"]
    a64, b64 = a.astype(np.float64), up.astype(np.float64)
    assert np.all(np.abs(y - a64 @ b64) <= 2.0 * np.sqrt(k) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)))
    if e >= -126:
        plain, _ = _gemm(bridge, base, b, False)
        assert np.array_equal(y.astype(np.float64), plain.astype(np.float64) * 2.0 ** (60 + e))
    mixed = base.copy()
    mixed[5, 3] = a[5, 3]  # one of them among ordinary values
    y, _ = _gemm(bridge, mixed, b, False)
    m64, b64 = mixed.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(y - m64 @ b64) <= 2.0 * np.sqrt(k) * 2.0 ** -24 * (np.abs(m64) @ np.abs(b64)))


def test_split_gemm_no_allocation(bridge):
    """Without workspace for the K slices the call takes fewer of them and
    still runs."""
    m, n, k = 1000, 4096, 4096
    a, b = torch.randn(m, k, device="cuda"), torch.randn(n, k, device="cuda")
    c = torch.zeros(m, n, device="cuda")
    d = N.MatmulDesc()
    d.batch, d.m, d.n, d.k = 1, m, n, k
    d.lda, d.ldb, d.ldc, d.trans_b = k, k, n, 1
    d.in_dtype = d.out_dtype = N.BG_F32
    torch.cuda.synchronize()
    assert _plan(m, n, k, True)["kSlices"] * m * n * 4 > 16 << 20
    assert bridge._lib.bg_matmul_noalloc(bridge._ctx, C.byref(d), a.data_ptr(), b.data_ptr(), None, c.data_ptr()) == 0
    bridge.synchronize()
    truth = a.double() @ b.double().T
    assert float((c.double() - truth).norm() / truth.norm()) < 1e-6
