"""Calls on a captured stream: what takes partial sums from the context's scratch
outside a capture runs in one slice inside it, so that a replay does not
depend on scratch that a later call may grow."""
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
