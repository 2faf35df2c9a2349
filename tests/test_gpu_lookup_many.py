"""LogUp-GKR batches with more instances than a workgroup has threads (a round's descriptors are then
searched in several steps) and with instances that join in different layers, against the oracle."""
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
