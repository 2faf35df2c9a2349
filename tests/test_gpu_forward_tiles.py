"""The forward product over int8-range weights around its tile shapes (csrc/gemm.h): row counts on both
sides of each rule (1, 2, 4 and 8 row tiles of 32; few and many tile steps), ragged columns and inner
sizes with and without K splits, and activations of one digit plane and of four.  Against exact integers.
And the time of products with little work or few columns, by products that do more."""
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
    yield c
    c.close()


def exact(a, b):
    """A * B mod P over 16-bit halves of A, centered int8 B: every partial sum below 2^53."""
    bc = np.where(b > P // 2, b.astype(np.int64) - P, b.astype(np.int64)).astype(np.float64)
    lo = ((a & 0xFFFF).astype(np.float64) @ bc).astype(np.int64)
    hi = ((a >> 16).astype(np.float64) @ bc).astype(np.int64)
    return ((lo + (hi % P) * 65536) % P).astype(np.uint32)


@pytest.mark.parametrize("m", [1, 32, 33, 64, 97, 128, 224, 225, 300, 513])
@pytest.mark.parametrize("k,n", [(40, 70), (1100, 257), (3000, 31), (96, 4099)])
def test_tile_rules(ctx, m, k, n):
    b = O.synthetic(k, n, 1, 7)
    b[0, 0], b[-1, -1] = 127, P - 127
    dev = ctx.upload(b)
    for kind in (1, 0):  # one digit plane, then four, then one again (the mask words take turns)
        a = O.synthetic(m, k, kind, 11 + m)
        assert np.array_equal(ctx.matmul_forward(ctx.upload(a), dev).download(), exact(a, b))
    a = O.synthetic(m, k, 1, 12 + m)
    assert np.array_equal(ctx.matmul_forward(ctx.upload(a), dev).download(), exact(a, b))


# many tile steps, so that wider tiles than one per wave are taken: 4 x 2, 2 x 2 and 2 x 1, each with
# its last tiles past the matrix's edges
@pytest.mark.parametrize("m,k,n", [(513, 3900, 4099), (200, 9400, 4099), (33, 8200, 4099)])
def test_wide_tiles(ctx, m, k, n):
    b = O.synthetic(k, n, 1, 7)
    b[0, 0], b[-1, -1] = 127, P - 127
    dev = ctx.upload(b)
    for kind in (1, 0):
        a = O.synthetic(m, k, kind, 11 + m)
        assert np.array_equal(ctx.matmul_forward(ctx.upload(a), dev).download(), exact(a, b))


def test_one_high_value_takes_the_general_path(ctx):
    """A single entry of A outside the int8 range, in the last row: one tile per wave and wider ones."""
    for m, k, n in ((300, 200, 300), (257, 4000, 7500)):
        a, b = O.synthetic(m, k, 1, 5), O.synthetic(k, n, 1, 6)
        a[-1, -1] = 1 << 20
        assert np.array_equal(ctx.matmul_forward(ctx.upload(a), ctx.upload(b)).download(), exact(a, b))


def test_four_planes_two_column_tiles_per_wave(ctx):
    """33 x 129 tiles of many steps: enough for two column tiles per wave, the last wave's second one past
    the edge."""
    a, b = O.synthetic(1030, 3100, 0, 8), O.synthetic(3100, 4099, 1, 9)
    assert np.array_equal(ctx.matmul_forward(ctx.upload(a), ctx.upload(b)).download(), exact(a, b))


def best(ctx, *products):
    """Seconds of the fastest of 60 calls of each product (m, k, n, kind of A, kind of B; kind 0: values over
    the whole field), called in turn: a host thread that moves meanwhile slows all of them."""
    ops = [(ctx.synthetic(m, k, a, 3), ctx.synthetic(k, n, b, 4), ctx.synthetic(m, n, 1, 5)) for m, k, n, a, b in products]
    times = [[] for _ in ops]
    for _ in range(60):
        for (a, b, c), ts in zip(ops, times):
            ctx.synchronize()
            t = time.perf_counter()
            ctx.matmul_forward_into(a, b, c)
            ctx.synchronize()
            ts.append(time.perf_counter() - t)
    return [min(ts) for ts in times]


def test_small_products_are_not_slowed_by_wide_tiles(ctx):
    """512 rows of few tile steps take about as long as 32 rows (latency and launches; 1.4 times with tiles
    of 4 x 2), and 64 columns less than 700 (on one XCD of eight they took longer)."""
    rows512, rows32 = best(ctx, (512, 576, 1536, 1, 1), (32, 576, 1536, 1, 1))
    assert rows512 < 1.3 * rows32
    narrow, wide = best(ctx, (4096, 5120, 64, 1, 1), (4096, 5120, 700, 1, 1))
    assert narrow < 0.9 * wide


def test_general_activations_have_splits_enough(ctx):
    """A wave's chain of K steps is what a product with few waves waits for: one general row takes 1.4 times
    an int8 row's time (1.8 with splits for one plane), and 96 int8 rows by 13824 x 13824 1.1 times 64 rows'
    (1.5 with a single split)."""
    general, int8 = best(ctx, (1, 5120, 13824, 0, 1), (1, 5120, 13824, 1, 1))
    assert general < 1.6 * int8
    rows96, rows64 = best(ctx, (96, 13824, 13824, 1, 1), (64, 13824, 13824, 1, 1))
    assert rows96 < 1.3 * rows64


def test_loads_of_general_weights_are_in_flight_together(ctx):
    """One row by weights of four digit planes reads the weights whatever the row's range, and one plane of it
    has a quarter of the multiplications: 0.86 of a general row's time (0.98 with two loads in flight)."""
    int8, general = best(ctx, (1, 5120, 13824, 1, 0), (1, 5120, 13824, 0, 0))
    assert int8 < 0.93 * general


def test_rows_for_a_grid_of_two_layers():
    """2^23 + 1 row tiles of one column: the four-plane kernel's workgroups fill two layers of the grid."""
    m = (1 << 28) + 3
    c = G.Context(0)
    a, b = c.synthetic(m, 1, 0, 3), c.upload(np.array([[P - 5]], dtype=np.uint32))
    got = c.matmul_forward(a, b).download().reshape(-1)
    x = a.download().reshape(-1)
    for i in range(0, m, 1 << 25):
        v = x[i:i + (1 << 25)].astype(np.int64) * -5 % P
        assert np.array_equal(got[i:i + (1 << 25)], v.astype(np.uint32)), i
    c.close()
