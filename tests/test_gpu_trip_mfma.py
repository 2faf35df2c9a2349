"""Product sumchecks whose trips run on the matrix cores (csrc/trip_mfma.h): vectors on both sides of the
trip rule, with values at the ends of the digit ranges (0, P - 1, P / 2 and its neighbours, bytes of 0x7f
and 0x80), where the balanced digits and the int32 sums are largest.  Against the oracle."""
import numpy as np
import pytest

import gkr_mi355x as G
import oracle as O

pytestmark = pytest.mark.gpu
P = G.P
EDGE = np.array([0, 1, P - 1, P // 2, P // 2 + 1, P // 2 - 1, 0x7F7F7F7F, 0x3F7F7F7F, 0x40808080, 0x00808080,
                 0x007F7F7F, 0x3F808080, 0x40000000, 0x7F808080], dtype=np.uint32) % P


def vec(n, what, seed):
    rng = np.random.default_rng(seed)
    if what == "edges":
        return EDGE[rng.integers(0, len(EDGE), size=(n, 4))]
    if what == "same":  # every digit product of one sign: the largest sums
        return np.full((n, 4), 0x3F808080, dtype=np.uint32)
    return rng.integers(0, P, size=(n, 4), dtype=np.uint32)


@pytest.mark.parametrize("logn", [16, 17, 18, 19, 20])
@pytest.mark.parametrize("what", ["edges", "same", "uniform"])
def test_product_sumcheck(gpu_ctx, logn, what):
    n = 1 << logn
    a, b = vec(n, what, logn), vec(n, what, logn + 100)
    gch, och = G.PoseidonChannel(), O.Channel()
    got = gpu_ctx.sumcheck_product(gpu_ctx.qvec_upload(a), gpu_ctx.qvec_upload(b), gch)
    assert got == O.sumcheck_product(a, b, och)
    assert gch.digest() == och.digest()


@pytest.mark.parametrize("logn", [17, 20])
def test_without_launches_ahead(monkeypatch, logn):
    """The same trips launched once their challenges are known (no launcher thread)."""
    monkeypatch.setenv("GKR_ASYNC_LAUNCH", "0")
    ctx = G.Context(0)
    n = 1 << logn
    a, b = vec(n, "edges", 5), vec(n, "uniform", 6)
    assert ctx.sumcheck_product(ctx.qvec_upload(a), ctx.qvec_upload(b), G.PoseidonChannel()) == \
        O.sumcheck_product(a, b, O.Channel())
    va, vb = ctx.qvec_upload(a), ctx.qvec_upload(b)
    assert ctx.sumcheck_product_noalloc(va.device_ptr, vb.device_ptr, n, G.PoseidonChannel()) == \
        O.sumcheck_product(a, b, O.Channel())
    ctx.close()


@pytest.mark.parametrize("logn", [16, 17, 18, 19])
@pytest.mark.parametrize("what", ["edges", "same", "uniform"])
def test_eq_weighted_trips(gpu_ctx, logn, what):
    """The Mul layer's eq-sumcheck over full QM31 operands."""
    n = 1 << logn
    a, b = vec(n, what, logn), vec(n, what, logn + 50)
    gch, och = G.PoseidonChannel(), O.Channel()
    pt = gch.draw_qm31s(logn)
    assert pt == och.draw_qm31s(logn)
    v = (1, 2, 3, 4)
    assert gpu_ctx.reduce_mul_layer(pt, v, a, b, gch) == O.reduce_mul_layer(pt, v, a, b, och)
    assert gch.digest() == och.digest()
