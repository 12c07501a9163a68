"""Calls on a captured stream: split GEMMs and decode attention run in one slice,
and scratch that a graph names outlives the growth of its slot."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def bridge():
    from browsergrad_amd.bridge import HipRealizerBridge
    with HipRealizerBridge(device=0) as br:
        br.set_profiling(False)
        yield br


def _gemm(br, rng):
    m, k, n = 300, 3072, 200
    a, b = rng.standard_normal((m, k)).astype(F32), rng.standard_normal((k, n)).astype(F32)
    ha, hb = br.upload(a, a.shape, "float32"), br.upload(b, b.shape, "float32")
    return (lambda: br.matmul_ex(ha, hb, m=m, n=n, k=k)), a.astype(np.float64) @ b, k


def _decode(br, rng):
    s, d = 9000, 64
    q, k, v = (rng.standard_normal((1, 1, t, d)).astype(F32) for t in (1, s, s))
    hs = [br.upload(x, x.shape, "float32") for x in (q, k, v)]
    x = q[0, 0].astype(np.float64) @ k[0, 0].T / 8
    p = np.exp(x - x.max())
    return (lambda: br.attention_ex(*hs, batch=1, heads=1, sq=1, sk=s, d=d, scale=1 / 8, causal=False,
                                    in_dtype="float32", out_dtype="float32")), (p / p.sum()) @ v[0, 0], s


@pytest.mark.parametrize("make", [_gemm, _decode])
def test_captured_call_takes_no_scratch(bridge, make):
    """Replayed with eager calls between; |y - truth| <= 8 sqrt(K) 2^-24 max|mass|."""
    br = bridge
    fn, want, terms = make(br, np.random.default_rng(3))
    br.set_launch_log(True)
    br.take_launch_log()
    warm = fn()
    eager = br.take_launch_log()
    assert len(eager) == 2, eager  # slices and their merge
    br.synchronize()
    br.release(warm)  # its block serves the captured call's output
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.ExternalStream(br.stream_ptr())):
        h = fn()
    assert len(br.take_launch_log()) == 1
    br.set_launch_log(False)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        y = br.to_numpy(h).reshape(want.shape)
        assert np.abs(y - want).max() <= 8 * np.sqrt(terms) * 2.0**-24 * max(1.0, 8 * np.abs(want).max())
        br.release(fn())
        br.synchronize()
    br.release(h)


def _skinny(br, rng, m, n, k, dtype):
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    if dtype == "float16":
        a, b = a.astype(np.float16), np.ascontiguousarray(b.T.astype(np.float16))
    else:
        a, b = a.astype(F32), b.astype(F32)
    ha, hb = br.upload(a, a.shape, dtype), br.upload(b, b.shape, dtype)
    return lambda: br.matmul_ex(ha, hb, m=m, n=n, k=k, trans_b=dtype == "float16", in_dtype=dtype,
                                out_dtype="float32")


def _transposed_b(br, rng, n):
    a, b = rng.standard_normal((96, 512)).astype(np.float16), rng.standard_normal((512, n)).astype(np.float16)
    ha, hb = br.upload(a, a.shape, "float16"), br.upload(b, b.shape, "float16")
    return lambda: br.matmul_ex(ha, hb, m=96, n=n, k=512, in_dtype="float16", out_dtype="float32")


def _conv(br, rng, c):
    x, dy = rng.standard_normal((2, c, 28, 28)).astype(F32), rng.standard_normal((2, 64, 28, 28)).astype(F32)
    hx, hd = br.upload(x, x.shape, "float32"), br.upload(dy, dy.shape, "float32")
    return lambda: br.conv_ex("backward_weight", hd, hx, n=2, c_in=c, c_out=64, in_size=(28, 28), out_size=(28, 28),
                              k=(3, 3), stride=(1, 1), pad=(1, 1), dilation=(1, 1))


# A call that keeps something in scratch, and a larger one in the same slot.
@pytest.mark.parametrize("small,large", [
    (lambda br, g: _skinny(br, g, 1, 4096, 4096, "float32"), lambda br, g: _skinny(br, g, 64, 8192, 2048, "float16")),
    (lambda br, g: _skinny(br, g, 32, 2048, 4096, "float16"), lambda br, g: _skinny(br, g, 64, 8192, 4096, "float16")),
    (lambda br, g: _transposed_b(br, g, 300), lambda br, g: _transposed_b(br, g, 9000)),
    (lambda br, g: _conv(br, g, 16), lambda br, g: _conv(br, g, 512))], ids=["f32", "f16", "b", "conv"])
def test_captured_scratch_outlives_growth(small, large):
    """Replays after the slot has grown give the eager call's bits, and do not
    write what took the memory since."""
    from browsergrad_amd.bridge import HipRealizerBridge
    rng = np.random.default_rng(11)
    with HipRealizerBridge(device=0) as br:
        br.set_profiling(False)
        fn, grow = small(br, rng), large(br, rng)
        warm = fn()
        want = br.to_numpy(warm).copy()
        br.release(warm)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=torch.cuda.ExternalStream(br.stream_ptr())):
            h = fn()
        eager = br.to_numpy(g := grow()).copy()
        br.release(g)
        fill = [br.upload(np.full(1 << 19, 7, F32), (1 << 19,), "float32") for _ in range(16)]
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(br.to_numpy(h), want)
            assert all((br.to_numpy(f) == 7).all() for f in fill)
            again = grow()
            assert np.array_equal(br.to_numpy(again), eager)
            br.release(again)
        del graph
