"""Optimizer updates larger than the last-level cache."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bridge():
    from browsergrad_amd.bridge import HipRealizerBridge
    with HipRealizerBridge(device=0) as br:
        yield br


@pytest.mark.parametrize("op", ["SGD_UPDATE", "ADAMW_UPDATE_M", "ADAMW_UPDATE_V", "ADAMW_UPDATE_PARAM", "ADAM_UPDATE_M",
                                "ADAM_UPDATE_V", "ADAM_UPDATE_PARAM"])
def test_optimizer_large_call_matches_small_calls(bridge, op):
    """A call that streams more than the last-level cache (nontemporal loads
    and stores) gives the same bits as the same elements in calls that do not."""
    import torch
    arity = 4 if op == "ADAMW_UPDATE_PARAM" else 3 if op.startswith("ADAM_") else 2
    n = {2: 23_000_003, 3: 17_000_001, 4: 15_000_003}[arity]
    g = torch.Generator().manual_seed(3)
    host = [torch.randn(n, generator=g).abs_().numpy() for _ in range(arity)]
    kw = dict(lr=6e-4, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.1, step=7)

    def update(lo, hi):
        hs = [bridge.upload(x[lo:hi], (hi - lo,), "float32") for x in host]
        h = bridge.optimizer_update(op, hs, hi - lo, **kw)
        y = bridge.to_numpy(h)
        for x in (*hs, h):
            bridge.release(x)
        return y

    big, step = update(0, n), 4_000_000
    assert n * 4 * (arity + 1) > 256 << 20
    assert np.array_equal(big, np.concatenate([update(i, min(n, i + step)) for i in range(0, n, step)]))
