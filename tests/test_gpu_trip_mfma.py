"""Product sumchecks whose trips run on the matrix cores (csrc/trip_mfma.h): vectors on both sides of the
trip rule, with values at the ends of the digit ranges (0, P - 1, P / 2 and its neighbours, bytes of 0x7f
and 0x80), where the balanced digits and the int32 sums are largest; and layers whose first trip is of one or
two rounds, so that a matrix-core trip folds one or two challenges.  Against the oracle."""
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


@pytest.mark.parametrize("k", [(1 << 18) + 3, (1 << 20) + 5])
@pytest.mark.parametrize("kind", [0, 1])
def test_matmul_after_a_short_first_trip(gpu_ctx, k, kind):
    """Inner sizes over 2^18 and 2^20: the first trip, which adds the weight side's partials, takes two rounds
    and one, and the next one folds as many challenges."""
    A, B = O.synthetic(1, k, kind, 7), O.synthetic(k, 2, kind, 8)
    A[0, :len(EDGE)], B[-len(EDGE):, 0] = EDGE, EDGE
    a, b = gpu_ctx.upload(A), gpu_ctx.upload(B)
    gch, och = G.PoseidonChannel(), O.Channel()
    r = gch.draw_qm31s(1)
    assert r == och.draw_qm31s(1)
    v = gpu_ctx.matmul_output_claim(a, b, r)
    assert v == O.matmul_output_claim(A, B, r)
    assert gpu_ctx.prove_matmul_layer(r, v, a, b, gch) == O.prove_matmul_layer(r, v, A, B, och)
    assert gch.digest() == och.digest()


def test_activation_after_a_short_first_trip(gpu_ctx):
    """2^21 padded entries: the fused first trip takes one round and the next one folds its challenge."""
    X = O.synthetic(61, 16385, 0, 9)
    X[0, :len(EDGE)], X[-1, -len(EDGE):] = EDGE, EDGE
    gch, och = G.PoseidonChannel(), O.Channel()
    pt = gch.draw_qm31s(21)
    assert pt == och.draw_qm31s(21)
    got = gpu_ctx.prove_activation_layer(pt, (1, 2, 3, 4), gpu_ctx.upload(X), 5, gch, 10)
    ref = O.prove_activation_layer(pt, (1, 2, 3, 4), X, 5, och, 10)
    for key in ("eq_round_polys", "claimed_sum", "mult_round_polys", "mult_final_eval", "input_eval"):
        assert got[key] == ref[key], key
    assert (got["multiplicities"] == ref["multiplicities"]).all()
    assert gch.digest() == och.digest()
