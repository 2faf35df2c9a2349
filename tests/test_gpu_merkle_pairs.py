"""Weight commitments whose leaf pairs come from the table of int8-range pairs (csrc/merkle.h): the
matrices are large enough for the table to be used, and mix pairs inside and outside its range, odd row
counts (a padding leaf beside a real one), padded columns and single-row grids.  Against the oracle.
And the time: a matrix that is partly in the range must not take longer than one that is all outside."""
import time

import numpy as np
import pytest

import gkr_mi355x as G
import oracle as O

pytestmark = pytest.mark.gpu
P = G.P


@pytest.fixture(scope="module")
def ctx():
    c = G.Context(0)
    # a batch large enough to build the table (2^18 leaf pairs); later, smaller ones use it too
    big = c.synthetic(1024, 512, 1, 5)
    c.weight_commitment(big)
    yield c
    c.close()


def edges(rows, cols, seed):
    """int8 range with its ends, the values next to them and a few general ones."""
    rng = np.random.default_rng(seed)
    m = rng.integers(-127, 128, size=(rows, cols)).astype(np.int64)
    m = np.where(m < 0, m + P, m)
    pick = np.array([0, 127, 128, P - 1, P - 127, P - 128, P - 129, 1 << 30, 255, 65025])
    hit = rng.random((rows, cols)) < 0.2
    return np.where(hit, pick[rng.integers(0, len(pick), size=(rows, cols))], m).astype(np.uint32)


@pytest.mark.parametrize("rows,cols", [(2, 1), (3, 5), (1, 7), (2, 2), (17, 3), (64, 33), (127, 9), (33, 64)])
def test_roots_match_oracle(ctx, rows, cols):
    for kind, m in (("edges", edges(rows, cols, rows * 100 + cols)), ("int8", O.synthetic(rows, cols, 1, rows + cols)),
                    ("m31", O.synthetic(rows, cols, 0, rows + cols))):
        assert ctx.weight_commitment(ctx.upload(m)) == O.weight_commitment(m), kind


def test_opening_matches_oracle(ctx):
    m = edges(24, 12, 3)
    ch, och = G.PoseidonChannel(), O.Channel()
    pt = ch.draw_qm31s(5 + 4)
    assert pt == och.draw_qm31s(9)
    proof = G.Proof()
    cm = ctx.prove_weight_opening(ctx.upload(m), pt, ch, proof)
    cm_o, felts = O.mle_opening(O.col_major_mle(m), pt, och)
    assert cm == cm_o and proof.serialize()[-1 - len(felts):-1] == felts
    assert ch.digest() == och.digest()


def test_with_and_without_the_table(ctx):
    """The same roots from a context that has built no table."""
    m = edges(300, 70, 9)
    plain = G.Context(0)
    assert ctx.weight_commitment(ctx.upload(m)) == plain.weight_commitment(plain.upload(m))
    plain.close()


@pytest.mark.parametrize("launch", [1, 2, 3])
def test_refused_launch(launch):
    """A launch of the commitment that the runtime refuses (the table's, a level's, the next) fails the call,
    and nothing of it is kept: the same call then gives the root."""
    c, m = G.Context(0), O.synthetic(1024, 512, 1, 5)
    w = c.upload(m)
    c.debug(G.DEBUG_REFUSE_LAUNCH, launch)
    with pytest.raises(G.GkrError):
        c.weight_commitment(w)
    root = c.weight_commitment(w)
    small = edges(64, 33, 2)  # below the size that builds the table: the kept one, if any
    assert c.weight_commitment(c.upload(small)) == O.weight_commitment(small)
    plain = G.Context(0)
    assert root == plain.weight_commitment(plain.upload(m))
    plain.close()
    c.close()


def test_partly_in_range_takes_no_longer(ctx):
    """Lanes with a pair in the table and lanes without stay in step: the hashes of a wave are then at most
    those of a matrix outside the range.  Out of step the mixed one took 1.4 to 2.7 times as long."""
    rng = np.random.default_rng(4)
    other = rng.integers(1 << 20, 1 << 30, size=(2048, 2048)).astype(np.uint32)
    small = rng.integers(0, 128, size=other.shape).astype(np.uint32)

    def best(m):
        w, ts = ctx.upload(m), []
        for _ in range(5):
            w.invalidate()
            t = time.perf_counter()
            ctx.weight_commitment(w)
            ts.append(time.perf_counter() - t)
        return min(ts)

    outside = best(other)
    for share in (0.05, 0.5, 0.9):
        mixed = best(np.where(rng.random(other.shape) < share, other, small))
        assert mixed < 1.2 * outside, (share, mixed, outside)


def test_words_past_the_field_are_hashed_as_they_are(ctx, write_words):
    """P and the words above it are no entries of the table: they keep the leaf of their own word."""
    w = ctx.upload(np.zeros((64, 64), dtype=np.uint32))
    zero = ctx.weight_commitment(w)
    write_words(w, 3 * 64 + 5, [P])
    w.invalidate()
    plain = G.Context(0)
    got = ctx.weight_commitment(w)
    assert got == plain.weight_commitment(plain.wrap_device(w.device_ptr, 64, 64)) and got != zero
    plain.close()
