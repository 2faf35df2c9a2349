"""The norm layers' device pass (csrc/norm.hip: statistics, vectors and evaluations without a host round
trip) at shapes around its workgroups, and walk steps whose scale is a resident matrix: a fresh claim
proved from the same pass, a scale longer and shorter than the width, and one that is not canonical, on
the host (refused before any launch) and resident (found by the device pass)."""
import numpy as np
import pytest

import gkr_mi355x as G
import oracle as O

pytestmark = pytest.mark.gpu
P = G.P


@pytest.mark.parametrize("rows,cols,dim", [(1, 2, 2), (3, 1023, 1023), (2, 1025, 700), (5, 4097, 5000), (65, 33, 33),
                                           (1, 9000, 9000)])
@pytest.mark.parametrize("kind", [G.STEP_LAYERNORM, G.STEP_RMSNORM])
def test_layers_match_oracle(gpu_ctx, rows, cols, dim, kind):
    x = O.synthetic(rows, cols, 0, rows * 7 + cols)
    x[0, 0] = P - 1
    gch, och = G.PoseidonChannel(), O.Channel()
    nv = (rows - 1).bit_length() + (cols - 1).bit_length()
    pt = gch.draw_qm31s(nv)
    assert pt == och.draw_qm31s(nv)
    m = gpu_ctx.upload(x)
    if kind == G.STEP_LAYERNORM:
        got = gpu_ctx.prove_norm_layer(kind, pt, (1, 2, 3, 4), m, dim, gch)
        ref = O.prove_layernorm_layer(pt, (1, 2, 3, 4), x, dim, och)
    else:
        g = np.random.default_rng(3).integers(0, P, size=cols, dtype=np.uint32)
        got = gpu_ctx.prove_norm_layer(kind, pt, (1, 2, 3, 4), m, dim, gch, gamma=g)
        ref = O.prove_rmsnorm_layer(pt, (1, 2, 3, 4), x, dim, och, g)
    assert gch.digest() == och.digest()
    for key in ("input_eval", "output_eval", "rsqrt_eval", "p0_round_polys", "lin_round_polys", "logup_round_polys",
                "mult_round_polys", "row_stats0", "row_stats1", "claimed_sum", "gamma_eval"):
        assert got[key] == ref[key], key
    assert (got["multiplicities"] == ref["multiplicities"]).all()


@pytest.mark.parametrize("ng", [0, 1, 40, 64, 200])
def test_fresh_walk_step(gpu_ctx, ng):
    """A fresh RMSNorm step against the output claim and the layer called one after the other."""
    x = gpu_ctx.upload(O.synthetic(6, 64, 1, 9))
    g = np.random.default_rng(ng).integers(0, P, size=ng, dtype=np.uint32) if ng else None
    gm = gpu_ctx.upload(g.reshape(1, -1)) if ng else None
    a, b = G.PoseidonChannel(), G.PoseidonChannel()
    proof = G.Proof()
    point, value = G.prove_walk(gpu_ctx, a, [(G.STEP_RMSNORM, G.CLAIM_FRESH, x, gm, 0, 0, 64)], proof)
    pt = b.draw_qm31s(9)
    v = gpu_ctx.norm_output_claim(G.STEP_RMSNORM, x, 64, pt, gamma=g)
    b.mix_secure_field(v)
    d = gpu_ctx.prove_norm_layer(G.STEP_RMSNORM, pt, v, x, 64, b, gamma=g)
    assert a.digest() == b.digest() and point == pt and value == d["input_eval"]
    assert proof.layer_claim_value(0) == v


def test_scale_not_canonical(gpu_ctx):
    x = gpu_ctx.synthetic(4, 16, 1, 3)
    g = np.ones(16, dtype=np.uint32)
    g[11] = P
    with pytest.raises(G.GkrError, match="gamma value 11 not canonical"):
        gpu_ctx.prove_norm_layer(G.STEP_RMSNORM, [(0, 0, 0, 0)] * 6, (0, 0, 0, 0), x, 16, G.PoseidonChannel(), gamma=g)


@pytest.mark.parametrize("claim", [G.CLAIM_FRESH, G.CLAIM_CHAINED])
@pytest.mark.parametrize("ng,at,bad", [(16, 0, P), (16, 11, P), (40, 39, 0xFFFFFFFF), (200, 199, P), (200, 64, P + 1)])
def test_resident_scale_not_canonical(gpu_ctx, write_words, claim, ng, at, bad):
    """A walk's scale is checked where it is: inside the width (16 columns), past it, and past the padded
    matrix (64 entries); the first bad value is named, and a good scale in its place is then accepted."""
    x = gpu_ctx.synthetic(4, 16, 1, 3)
    good = np.full((1, ng), 7, dtype=np.uint32)
    g = gpu_ctx.upload(good)
    write_words(g, at, [bad] * (ng - at))
    step = [(G.STEP_RMSNORM, claim, x, g, 0, 0, 16)]
    start = dict(init_point=[(1, 2, 3, 4)] * 6, init_value=(1, 0, 0, 0)) if claim == G.CLAIM_CHAINED else {}
    with pytest.raises(G.GkrError, match="gamma value %d not canonical" % at):
        G.prove_walk(gpu_ctx, G.PoseidonChannel(), step, G.Proof(), **start)
    write_words(g, at, good[0, at:])
    ch, ref = G.PoseidonChannel(), G.PoseidonChannel()
    up = gpu_ctx.upload(good)
    got = G.prove_walk(gpu_ctx, ch, step, G.Proof(), **start)
    assert got == G.prove_walk(gpu_ctx, ref, [step[0][:3] + (up,) + step[0][4:]], G.Proof(), **start)
    assert ch.digest() == ref.digest()


def test_more_rows_than_a_launch_takes(gpu_ctx):
    """2^25 + 1 rows pad to 2^26, whose waves a launch does not take: refused before anything is launched."""
    x = gpu_ctx.synthetic((1 << 25) + 1, 1, 1, 3)
    with pytest.raises(G.GkrError, match="norm layer of 33554433 rows"):
        gpu_ctx.norm_output_claim(G.STEP_RMSNORM, x, 1, [(1, 0, 0, 0)] * 26)
