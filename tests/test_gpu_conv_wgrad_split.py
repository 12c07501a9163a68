"""Convolution weight gradients on the bf16 matrix core (three bf16 parts of each
value) against float64: tiles, rows and images that end inside a chunk of
eight positions, groups, strides, dilation, 1-D / 3-D / transposed layers, the
sizes on both sides of the rule, and the values the parts cannot hold."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def bridge():
    from browsergrad_amd.bridge import HipRealizerBridge
    with HipRealizerBridge(device=0) as br:
        yield br


def _exact(x, dy, kernel, stride, pad, dil, groups, transposed):
    """dw and the same sum over absolute values, in float64."""
    r = len(kernel)
    fn = getattr(torch.nn.functional, f"conv{'_transpose' if transposed else ''}{r}d")
    c, o = x.shape[1], dy.shape[1]
    shape = (c, o // groups, *kernel) if transposed else (o, c // groups, *kernel)
    res = []
    for f in (lambda t: t, np.abs):
        w = torch.zeros(shape, dtype=torch.float64, requires_grad=True)
        y = fn(torch.from_numpy(f(x).astype(np.float64)), w, None, stride=stride, padding=pad, dilation=dil,
               groups=groups)
        y.backward(torch.from_numpy(f(dy).astype(np.float64)))
        res.append(w.grad.numpy())
    return res


def _run(br, x, dy, kernel, stride, pad, dil, groups, transposed):
    hx, hd = br.upload(x, x.shape, "float32"), br.upload(dy, dy.shape, "float32")
    h = br.conv_ex("backward_weight", hd, hx, n=x.shape[0], c_in=x.shape[1], c_out=dy.shape[1], in_size=x.shape[2:],
                   out_size=dy.shape[2:], k=kernel, stride=stride, pad=pad, dilation=dil, groups=groups,
                   transposed=transposed)
    y = br.to_numpy(h)
    for t in (hx, hd, h):
        br.release(t)
    return y


def _data(n, c, o, size, kernel, stride, pad, dil, transposed, seed):
    rng = np.random.default_rng(seed)
    if transposed:
        out = [(i - 1) * s - 2 * p + d * (k - 1) + 1 for i, k, s, p, d in zip(size, kernel, stride, pad, dil)]
    else:
        out = [(i + 2 * p - d * (k - 1) - 1) // s + 1 for i, k, s, p, d in zip(size, kernel, stride, pad, dil)]
    return rng.standard_normal((n, c, *size)).astype(F32), rng.standard_normal((n, o, *out)).astype(F32)


# n, c, o, size, kernel, stride, pad, dilation, groups, transposed
CASES = [
    (2, 16, 130, (8, 8), (3, 3), (1, 1), (1, 1), (1, 1), 1, False),     # chunks end with rows; two row tiles
    (3, 15, 70, (9, 9), (3, 3), (1, 1), (1, 1), (1, 1), 1, False),      # odd image: dy element by element
    (5, 32, 70, (14, 14), (2, 2), (1, 1), (0, 1), (1, 1), 1, False),    # 13 x 15: dy element by element
    (6, 140, 70, (14, 14), (1, 1), (1, 1), (0, 0), (1, 1), 1, False),   # 196: a chunk's halves in two images
    (3, 140, 20, (6, 10), (1, 1), (1, 1), (0, 0), (1, 1), 1, False),    # 60 positions, two row groups
    (2, 16, 3, (13, 11), (3, 3), (1, 1), (1, 1), (1, 1), 1, False),     # few rows
    (4, 64, 128, (28, 28), (3, 3), (2, 2), (1, 1), (1, 1), 1, False),   # stride
    (2, 40, 64, (16, 12), (2, 3), (1, 1), (0, 2), (2, 2), 1, False),    # dilation, uneven padding
    (2, 64, 256, (14, 14), (3, 3), (1, 1), (1, 1), (1, 1), 2, False),   # groups
    (5, 200, 20, (16,), (1,), (1,), (0,), (1,), 1, False),              # 1-D, one tap
    (2, 8, 32, (3, 5, 10), (2, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), 1, False),  # 3-D
    (2, 128, 32, (9, 10), (3, 3), (2, 2), (1, 1), (1, 1), 1, True),     # transposed: the operands change places
    (2, 16, 16, (8, 7), (3, 3), (1, 1), (1, 1), (1, 1), 1, False),      # rows of 7: the other kernel
    (1, 16, 16, (8, 15), (3, 3), (1, 1), (1, 1), (1, 1), 1, False),     # 120 positions: the other kernel
    (1, 16, 16, (8, 16), (3, 3), (1, 1), (1, 1), (1, 1), 1, False),     # 128: the first on this one
]


@pytest.mark.parametrize("n,c,o,size,kernel,stride,pad,dil,groups,transposed", CASES)
def test_weight_gradient_against_float64(bridge, n, c, o, size, kernel, stride, pad, dil, groups, transposed):
    """|dw - truth| <= 8 sqrt(K) 2^-24 mass + 1e-6 (the bound of a K-term float32
    sum, as for the other weight gradients)."""
    x, dy = _data(n, c, o, size, kernel, stride, pad, dil, transposed, n + c + o)
    want, mass = _exact(x, dy, kernel, stride, pad, dil, groups, transposed)
    got = _run(bridge, x, dy, kernel, stride, pad, dil, groups, transposed).reshape(want.shape)
    terms = n * int(np.prod((x if transposed else dy).shape[2:]))
    assert (np.abs(got - want) <= 8 * np.sqrt(terms) * 2.0**-24 * mass + 1e-6).all()


@pytest.mark.parametrize("e", [-100, -115, -126])
@pytest.mark.parametrize("o", [40, 130])
def test_small_values_take_no_other_path(bridge, e, o):
    """dy at 2^-100 to 2^-126 against an x scaled up, and the other way round:
    the unscaled gradient's bits."""
    geo = ((3, 3), (1, 1), (1, 1), (1, 1))
    x, dy = _data(2, 16, o, (10, 10), *geo, False, 5)
    x, dy = (np.sign(t) * (F32(1) + np.abs(t) % F32(1)) for t in (x, dy))
    base = _run(bridge, x, dy, *geo, 1, False).astype(np.float64)
    lo, up = F32(2.0**e), F32(2.0**60)
    for a, b in ((x * up, dy * lo), (x * lo, dy * up)):
        assert np.array_equal(_run(bridge, a, b, *geo, 1, False).astype(np.float64), base * 2.0**(60 + e))


@pytest.mark.parametrize("value", [2.0**-120, 1e-40, np.inf, np.nan, 3.4e38])
def test_values_the_parts_cannot_hold(bridge, value):
    """A dy value infinite, NaN or one whose leading part rounds to infinity (the
    workgroup's float32 sums), or a tiny one, gives what float32 gives."""
    geo = ((3, 3), (1, 1), (1, 1), (1, 1))
    x, dy = _data(2, 16, 40, (10, 10), *geo, False, 5)
    x = np.abs(x) + F32(1)
    dy[:, 7] = 0
    dy[1, 7, 4, 5] = value
    with np.errstate(all="ignore"):
        want, mass = _exact(x, dy, *geo, 1, False)
        got = _run(bridge, x, dy, *geo, 1, False)
        one = (x[1, :, 3:6, 4:7] * F32(value)).astype(F32)  # row 7 has this one term
    assert np.array_equal(got[7], one, equal_nan=True)
    rest = [i for i in range(40) if i != 7]
    assert (np.abs(got[rest] - want[rest]) <= 8 * np.sqrt(200) * 2.0**-24 * mass[rest] + 1e-6).all()
