"""LogUp-GKR batches with more instances than a workgroup has threads (a round's descriptors are then
searched in several steps) and with instances that join in different layers, against the oracle; and launches that fail."""
import gkr_mi355x as G
import numpy as np
import oracle as O
import pytest
from test_gpu_lookup import _check, _make

pytestmark = pytest.mark.gpu
KINDS = (O.LOOKUP_GRAND_PRODUCT, O.LOOKUP_LOGUP_GENERIC, O.LOOKUP_LOGUP_MULTIPLICITIES, O.LOOKUP_LOGUP_SINGLES)


@pytest.mark.parametrize("count,nvs", [(1, (3,)), (255, (2, 3)), (256, (3,)), (257, (4, 2, 3)), (600, (2, 3, 5))])
def test_many_instances(gpu_ctx, count, nvs):
    spec = [(KINDS[i % 4], nvs[i % len(nvs)]) for i in range(count)]
    _check(gpu_ctx, _make(np.random.default_rng(count), spec), count)


def test_large_beside_small(gpu_ctx):
    """Several workgroups per instance beside one-workgroup instances."""
    _check(gpu_ctx, _make(np.random.default_rng(7), [(2, 13), (0, 2), (1, 11), (3, 12), (2, 2)]), 7)


def test_refused_launches(monkeypatch):
    """Whichever launch the runtime refuses, the call fails and the next one on the context gives the proof:
    what a launch that did not run would have counted is not waited for."""
    monkeypatch.setenv("GKR_ASYNC_LAUNCH", "0")
    ctx = G.Context(0)
    batch = _make(np.random.default_rng(3), [(2, 9), (0, 5), (1, 11)])
    _check(ctx, batch, 3)
    for launch in range(1, 40, 3):
        ctx.debug(G.DEBUG_REFUSE_LAUNCH, launch)
        with pytest.raises(G.GkrError):
            _check(ctx, batch, 3)
        _check(ctx, batch, 3)
    ctx.close()
