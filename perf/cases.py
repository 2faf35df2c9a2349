"""The workloads this framework is timed on.

A case is a dict of plain values: its "kind" and the sizes of one call.  The
listed cases are the layers and phases of a proof at the sizes of this
repository's own configurations (SmolLM2-135M with one token, Qwen2.5-14B with
64 tokens, the 256^3 matmul, the 2^28 product sumcheck); draw() gives more of
the same kinds over the ranges those sizes stand for.  The calls are the ones a
prover program makes through the C ABI (and the binding's walk), with result
buffers that it keeps.  Every result is a field element, a hash or a count, so
two correct implementations agree on every word.
"""
import ctypes as C
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stwo-ml_amd"))

import gkr_mi355x as G  # noqa: E402

P = (1 << 31) - 1
_context = []


def context():
    """The program's device context, kept for its whole life."""
    if not _context:
        _context.append(G.Context(0))
    return _context[0]


def lg(v):
    return max(0, (v - 1).bit_length())


def pow2(v):
    return 1 << lg(v)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one decoded token through a SmolLM2-135M layer (9 query heads, 3 kv heads of 64): the smallest
        # steps, where launches, waits and the transcript are all there is
        {"name": "decode_walk", "kind": "walk", "tokens": 1, "hidden": 576, "inter": 1536, "q": 576, "kv": 192,
         "heads": 9},
        # a 64-token prompt through a Qwen2.5-14B layer: seven matmuls, SiLU and softmax lookups
        {"name": "prefill_walk", "kind": "walk", "tokens": 64, "hidden": 5120, "inter": 13824, "q": 5120, "kv": 1024,
         "heads": 40},
        # a single matmul layer over full-range values (weights that are not int8)
        {"name": "matmul_256", "kind": "matmul", "m": 256, "k": 256, "n": 256, "values": "m31"},
        # the MLP gate weight shared by the activation blocks of a batch of eight
        {"name": "simd_gate", "kind": "simd", "blocks": 8, "m": 64, "k": 5120, "n": 13824},
        # attention scores through softmax-exp with the default 2^20 table
        {"name": "softmax_scores", "kind": "activation", "rows": 2560, "cols": 64, "act": 4, "table": 20},
        # SwiGLU's element-wise product
        {"name": "swiglu_mul", "kind": "mul", "rows": 64, "cols": 13824},
        # the two RMSNorms of a block, with learned scales
        {"name": "rmsnorm", "kind": "norm", "norm": "rms", "rows": 64, "cols": 5120, "layers": 2},
        # the witness of the gate product for a longer prompt
        {"name": "forward_prefill", "kind": "forward", "m": 512, "k": 5120, "n": 13824, "values": "int8"},
        # the product sumcheck alone at its largest configured size
        {"name": "sumcheck_2p28", "kind": "sumcheck", "log_n": 28},
        # the weight commitments of a Qwen2.5-14B layer, after its weights changed
        {"name": "commit_layer", "kind": "commit", "hidden": 5120, "inter": 13824, "q": 5120, "kv": 1024},
        # one weight opened at a claim point
        {"name": "opening_q", "kind": "opening", "k": 5120, "n": 5120},
        # the LogUp-GKR batch over the activation tables of 48 layers
        {"name": "lookup_tables", "kind": "lookup", "instances": 96, "log_n": 16},
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi], odd as often as not."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    return max(lo, min(hi, v | 1 if rng.random() < 0.5 else v))


def draw(rng):
    kind = rng.choice(["walk", "matmul", "simd", "activation", "mul", "norm", "forward", "sumcheck", "commit",
                       "opening", "lookup"])
    c = {"kind": kind}
    if kind == "walk":
        heads = rng.choice([4, 9, 16, 40])
        c.update(tokens=_size(rng, 1, 64), hidden=_size(rng, 256, 5120), inter=_size(rng, 512, 13824),
                 q=64 * heads, kv=64 * max(1, heads // rng.choice([1, 3, 4])), heads=heads)
    elif kind == "matmul":
        c.update(m=_size(rng, 1, 256), k=_size(rng, 64, 13824), n=_size(rng, 64, 13824),
                 values=rng.choice(["int8", "m31"]))
    elif kind == "simd":
        c.update(blocks=_size(rng, 1, 16), m=_size(rng, 1, 64), k=_size(rng, 64, 5120), n=_size(rng, 64, 13824))
    elif kind == "activation":
        act = rng.choice([2, 3, 4, 5])
        c.update(rows=_size(rng, 1, 512), cols=_size(rng, 64, 2048), act=act, table=20 if act == 4 else 16)
    elif kind == "mul":
        c.update(rows=_size(rng, 1, 64), cols=_size(rng, 64, 13824))
    elif kind == "norm":
        c.update(norm=rng.choice(["rms", "layer"]), rows=_size(rng, 1, 64), cols=_size(rng, 64, 5120), layers=1)
    elif kind == "forward":
        c.update(m=_size(rng, 1, 512), k=_size(rng, 64, 5120), n=_size(rng, 64, 13824),
                 values=rng.choice(["int8", "int8", "m31"]))
    elif kind == "sumcheck":
        c.update(log_n=rng.randint(8, 28))
    elif kind == "commit":
        h = _size(rng, 192, 5120)
        c.update(hidden=h, inter=_size(rng, h, 13824), q=h, kv=_size(rng, 64, 1024))
    elif kind == "opening":
        c.update(k=_size(rng, 64, 5120), n=_size(rng, 64, 5120))
    else:
        c.update(instances=_size(rng, 1, 96), log_n=rng.randint(6, 16))
    return c


# ------------------------------------------------------------------ inputs
class Inputs:
    """Seeded matrices in device memory, as a program that owns its tensors hands them over."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.keep = []

    def values(self, shape, values):
        """Quantized weights and activations ("int8": [-127, 127], negatives as P + v) or uniform M31."""
        if values == "int8":
            v = torch.randint(-127, 128, shape, generator=self.gen, device="cuda", dtype=torch.int32)
            return torch.where(v < 0, v + P, v)
        return torch.randint(0, P, shape, generator=self.gen, device="cuda", dtype=torch.int32)

    def matrix(self, rows, cols, values):
        t = self.values((rows, cols), values)
        self.keep.append(t)
        return context().wrap_device(t.data_ptr(), rows, cols)

    def point(self, n):
        return torch.randint(0, P, (n, 4), generator=self.gen, device="cuda", dtype=torch.int32).cpu().numpy()


class Buffer:
    """n QM31 (or another count of u32 words) of a result, and its address for the C ABI."""

    def __init__(self, n, words=4):
        self.a = np.zeros((max(1, n), words), dtype=np.int32)

    def q(self, i=0):
        return C.cast(self.a.ctypes.data + 16 * i, C.POINTER(G.GkrQM31))

    def u32(self):
        return C.cast(self.a.ctypes.data, C.POINTER(C.c_uint32))


def _q(words):
    x = G.GkrQM31()
    x.v[:] = [int(w) for w in words]
    return x


def _channel(seed):
    """The caller's transcript before the call."""
    ch = G.PoseidonChannel()
    ch.mix_u64(seed)
    return ch


def _walk_state(st, steps, max_felts):
    st["steps"], st["n_steps"] = G.make_steps(steps), len(steps)
    st["words"] = np.zeros((max_felts, 8), dtype=np.uint32)


def prepare(case, seed):
    ctx, inp, kind = context(), Inputs(seed), case["kind"]
    st = {"case": case, "seed": seed, "inputs": inp}
    F = G.CLAIM_FRESH
    if kind == "walk":
        m, h, i, q, kv = (case[k] for k in ("tokens", "hidden", "inter", "q", "kv"))
        x, xo, xg, xd = (inp.matrix(m, c, "int8") for c in (h, q, h, i))
        steps = [(G.STEP_MATMUL, F, x, inp.matrix(h, q, "int8"), 0, 0),
                 (G.STEP_MATMUL, F, x, inp.matrix(h, kv, "int8"), 0, 0),
                 (G.STEP_MATMUL, F, x, inp.matrix(h, kv, "int8"), 0, 0),
                 (G.STEP_MATMUL, F, xo, inp.matrix(q, h, "int8"), 0, 0),
                 (G.STEP_MATMUL, F, xg, inp.matrix(h, i, "int8"), 0, 0),
                 (G.STEP_MATMUL, F, xg, inp.matrix(h, i, "int8"), 0, 0),
                 (G.STEP_ACTIVATION, F, inp.matrix(m, i, "m31"), None, 5, 16),
                 (G.STEP_MATMUL, F, xd, inp.matrix(i, h, "int8"), 0, 0)]
        if m > 1:
            steps.append((G.STEP_ACTIVATION, F, inp.matrix(case["heads"] * m, m, "m31"), None, 4, 16))
        st["mats"] = [s[2] for s in steps] + [s[3] for s in steps]
        _walk_state(st, steps, 2 * (1 << 16) + 4096 * len(steps))
    elif kind == "norm":
        steps, st["mats"] = [], []
        for _ in range(case["layers"]):
            x, g = inp.matrix(case["rows"], case["cols"], "int8"), None
            if case["norm"] == "rms":  # a 12-bit learned scale per column
                t = torch.randint(1, 1 << 12, (1, case["cols"]), generator=inp.gen, device="cuda", dtype=torch.int32)
                inp.keep.append(t)
                g = ctx.wrap_device(t.data_ptr(), 1, case["cols"])
            steps.append((G.STEP_RMSNORM if case["norm"] == "rms" else G.STEP_LAYERNORM, F, x, g, 0, 0, case["cols"]))
            st["mats"] += [x, g]
        _walk_state(st, steps, ((1 << 17) + 8192) * len(steps))
    elif kind == "matmul":
        st["a"] = inp.matrix(case["m"], case["k"], case["values"])
        st["b"] = inp.matrix(case["k"], case["n"], case["values"])
    elif kind == "simd":
        st["blocks"] = [inp.matrix(case["m"], case["k"], "int8") for _ in range(case["blocks"])]
        st["b"] = inp.matrix(case["k"], case["n"], "int8")
        st["handles"] = (C.c_void_p * case["blocks"])(*[x.handle for x in st["blocks"]])
        st["weights"] = Buffer(case["blocks"])
        st["weights"].a[:] = inp.point(case["blocks"])
        st["value"] = _q(inp.point(1)[0])
    elif kind == "activation":
        st["x"] = inp.matrix(case["rows"], case["cols"], "m31")
        t, nv = case["table"], lg(case["rows"]) + lg(case["cols"])
        st["eq"], st["mults"], st["mult_polys"] = Buffer(4 * nv), Buffer(1 << t, 1), Buffer(2 * t)
        o = st["out"] = G.GkrLogupOut()
        o.eq_round_polys, o.mult_round_polys = st["eq"].q(), st["mult_polys"].q()
        o.multiplicities = st["mults"].u32()
    elif kind == "mul":
        st["x"] = inp.matrix(case["rows"], case["cols"], "int8")
        st["y"] = inp.matrix(case["rows"], case["cols"], "int8")
        st["eq"] = Buffer(4 * (lg(case["rows"]) + lg(case["cols"])))
        st["out"] = G.GkrMulOut()
        st["out"].eq_round_polys = st["eq"].q()
    elif kind == "forward":
        st["a"] = inp.matrix(case["m"], case["k"], "int8" if case["values"] == "int8" else "m31")
        st["b"] = inp.matrix(case["k"], case["n"], case["values"])
        st["c_values"] = torch.zeros((case["m"], case["n"]), dtype=torch.int32, device="cuda")
        st["c"] = ctx.wrap_device(st["c_values"].data_ptr(), case["m"], case["n"])
    elif kind == "sumcheck":
        n = 1 << case["log_n"]
        st["fa"], st["fb"] = ctx.qvec_synthetic(n, 2 * seed + 1), ctx.qvec_synthetic(n, 2 * seed + 2)
    elif kind == "commit":
        h, i, q, kv = (case[k] for k in ("hidden", "inter", "q", "kv"))
        st["weights"] = [inp.matrix(r, c, "int8")
                         for r, c in ((h, q), (h, kv), (h, kv), (q, h), (h, i), (h, i), (i, h))]
        st["handles"] = (C.c_void_p * 7)(*[w.handle for w in st["weights"]])
        st["roots"] = Buffer(7, 8)
    elif kind == "opening":
        st["b"] = inp.matrix(case["k"], case["n"], "int8")
        st["nv"] = lg(case["k"]) + lg(case["n"])
        st["words"] = np.zeros((1 << 15, 8), dtype=np.uint32)
    elif kind == "lookup":
        n, ni, nl = 1 << case["log_n"], case["instances"], case["log_n"]
        alpha = inp.point(1)[0]
        tables = torch.randint(0, P, (ni, n), generator=inp.gen, device="cuda", dtype=torch.int32)
        den = torch.empty((ni, n, 4), dtype=torch.int32, device="cuda")
        den[..., 0] = (int(alpha[0]) + P - tables.to(torch.int64)).remainder(P).to(torch.int32)
        for j in range(1, 4):
            den[..., j] = int(alpha[j])
        num = torch.randint(0, 8, (ni, n), generator=inp.gen, device="cuda", dtype=torch.int32)
        inp.keep += [den, num]
        st["instances"] = (G.GkrLookupInstance * ni)()
        for i in range(ni):
            s = st["instances"][i]
            s.kind, s.n_vars = G.LOOKUP_LOGUP_MULTIPLICITIES, nl
            s.numerators, s.denominators = num[i].data_ptr(), den[i].data_ptr()
        rounds = nl * (nl - 1) // 2
        st["buffers"] = {"claims": Buffer(2 * ni), "polys": Buffer(4 * rounds), "lens": Buffer(rounds, 1),
                         "masks": Buffer(4 * nl * ni), "point": Buffer(nl), "verify": Buffer(2 * ni)}
        b, o = st["buffers"], G.GkrLookupBatch()
        o.output_claims, o.round_polys, o.round_poly_lens = b["claims"].q(), b["polys"].q(), b["lens"].u32()
        o.masks, o.ood_point, o.claims_to_verify = b["masks"].q(), b["point"].q(), b["verify"].q()
        st["out"] = o
    if kind in ("matmul", "simd"):
        T, nv = lg(case["k"]), lg(case["m"]) + lg(case["n"])
        st["point"], st["polys"] = Buffer(nv), Buffer(3 * T)
        st["finals"], st["next"] = Buffer(3), Buffer(lg(case["m"]) + T)
    if kind in ("activation", "mul"):
        st["nv"] = lg(case["rows"]) + lg(case["cols"])
        st["point"] = Buffer(st["nv"])
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------ one pass
def _struct_q(o, names):
    return np.array([list(getattr(o, k).v) for k in names], dtype=np.int64)


def _digest(ch):
    return np.array(ch.export_state(), dtype=np.int64)


def run(st):
    L, ctx, case, kind = G.lib(), context(), st["case"], st["case"]["kind"]
    if kind in ("walk", "norm"):  # the walk on one channel, its proof serialized as it is made
        ch, proof = _channel(st["seed"]), G.Proof()
        proof.stream_to(st["words"])
        point, value = G.prove_walk(ctx, ch, st["steps"], proof, n_steps=st["n_steps"])
        n = proof.serialize_into(st["words"])
        return {"proof": st["words"][:n].view(np.int32), "point": np.array(point + [value], dtype=np.int64)}
    if kind == "forward":  # the product, finished: the program reads it on its own stream
        G._check(L.gkr_matmul_forward_into(ctx.handle, st["a"].handle, st["b"].handle, st["c"].handle))
        ctx.synchronize()
        return st["c_values"]
    if kind == "commit":  # the weights were updated: the roots kept on them no longer hold
        for w in st["weights"]:
            w.invalidate()
        G._check(L.gkr_weight_commitments(ctx.handle, st["handles"], 7,
                                          C.cast(st["roots"].a.ctypes.data, C.POINTER(G.GkrFelt))))
        return st["roots"].a
    ch = _channel(st["seed"])
    if kind == "matmul":  # a fresh output claim, then the layer
        G._check(L.gkr_channel_draw_qm31s(ch.handle, lg(case["m"]) + lg(case["n"]), st["point"].q()))
        v, nv = G.GkrQM31(), lg(case["m"]) + lg(case["n"])
        a, b, f = st["a"].handle, st["b"].handle, st["finals"]
        G._check(L.gkr_matmul_output_claim(ctx.handle, a, b, st["point"].q(), nv, C.byref(v)))
        G._check(L.gkr_channel_mix_secure_field(ch.handle, C.byref(v)))
        G._check(L.gkr_prove_matmul_layer(ctx.handle, st["point"].q(), nv, C.byref(v), a, b, ch.handle, None,
                                          st["polys"].q(), f.q(0), f.q(1), st["next"].q(), f.q(2)))
        return {"claim": np.array(list(v.v)), "polys": st["polys"].a, "finals": f.a, "next": st["next"].a,
                "channel": _digest(ch)}
    if kind == "simd":
        nv, f = lg(case["m"]) + lg(case["n"]), st["finals"]
        G._check(L.gkr_channel_draw_qm31s(ch.handle, nv, st["point"].q()))
        G._check(L.gkr_prove_matmul_layer_simd(ctx.handle, st["point"].q(), nv, C.byref(st["value"]), st["handles"],
                                               st["weights"].q(), case["blocks"], st["b"].handle, ch.handle, None,
                                               st["polys"].q(), f.q(0), f.q(1), st["next"].q(), f.q(2)))
        return {"polys": st["polys"].a, "finals": f.a, "next": st["next"].a, "channel": _digest(ch)}
    if kind == "activation":  # a drawn claim, as a walk's fresh activation step
        v, o = G.GkrQM31(), st["out"]
        G._check(L.gkr_channel_draw_qm31s(ch.handle, st["nv"], st["point"].q()))
        G._check(L.gkr_channel_draw_qm31(ch.handle, C.byref(v)))
        G._check(L.gkr_prove_activation_layer(ctx.handle, st["point"].q(), st["nv"], C.byref(v), st["x"].handle,
                                              case["act"], case["table"], ch.handle, None, C.byref(o)))
        evals = ("claimed_sum", "w_eval", "in_eval", "out_eval", "mult_final_eval", "mult_claimed_sum", "input_eval",
                 "output_eval", "gamma", "beta")
        return {"eq": st["eq"].a, "mults": st["mults"].a, "mult_polys": st["mult_polys"].a,
                "evals": _struct_q(o, evals), "channel": _digest(ch)}
    if kind == "mul":
        v, o = G.GkrQM31(), st["out"]
        G._check(L.gkr_channel_draw_qm31s(ch.handle, st["nv"], st["point"].q()))
        G._check(L.gkr_mul_output_claim(ctx.handle, st["x"].handle, st["y"].handle, st["point"].q(), st["nv"],
                                        C.byref(v)))
        G._check(L.gkr_channel_mix_secure_field(ch.handle, C.byref(v)))
        G._check(L.gkr_prove_mul_layer(ctx.handle, st["point"].q(), st["nv"], C.byref(v), st["x"].handle,
                                       st["y"].handle, ch.handle, None, C.byref(o)))
        return {"claim": np.array(list(v.v)), "eq": st["eq"].a,
                "evals": _struct_q(o, ("lhs_eval", "rhs_eval", "alpha", "next_value")), "channel": _digest(ch)}
    if kind == "sumcheck":
        r = ctx.sumcheck_product(st["fa"], st["fb"], ch)
        return {"polys": np.array(r["round_polys"], dtype=np.int64), "challenges": np.array(r["challenges"]),
                "finals": np.array([r["final_a_eval"], r["final_b_eval"]], dtype=np.int64)}
    if kind == "opening":
        proof = G.Proof()
        ctx.prove_weight_opening(st["b"], ch.draw_qm31s(st["nv"]), ch, proof)
        n = proof.serialize_into(st["words"])
        return {"proof": st["words"][:n].view(np.int32), "channel": _digest(ch)}
    G._check(L.gkr_prove_lookup_batch(ctx.handle, ch.handle, st["instances"], case["instances"], C.byref(st["out"])))
    return dict({k: b.a for k, b in st["buffers"].items()}, channel=_digest(ch))


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """bytes: every input read once (an int8-range weight as one byte), every result written once.
    flops: a matrix product's multiply-adds, and a Poseidon hash's 32-bit multiply-adds (107 cubes of a
    252-bit element, each a square and a product of nine limbs), two operations each."""
    kind = case["kind"]
    hash_ops = 2 * 107 * (45 + 81)
    if kind == "walk":
        m, h, i, q, kv = (case[k] for k in ("tokens", "hidden", "inter", "q", "kv"))
        weights = h * q + 2 * h * kv + q * h + 3 * h * i
        acts = m * (h + q + h + 2 * i + (case["heads"] * m if m > 1 else 0))
        return {"bytes": weights + 4 * acts + 32 * (1 << 16) * (2 if m > 1 else 1), "flops": 0}
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": (1 if case["values"] == "int8" else 4) * k * n + 4 * m * k, "flops": 0}
    if kind == "simd":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": k * n + 4 * case["blocks"] * m * k, "flops": 0}
    if kind == "activation":
        return {"bytes": 4 * case["rows"] * case["cols"] + 4 * 2 * (1 << case["table"]), "flops": 0}
    if kind == "mul":
        return {"bytes": 8 * case["rows"] * case["cols"], "flops": 0}
    if kind == "norm":
        return {"bytes": case["layers"] * (4 * case["rows"] * case["cols"] + 32 * (1 << 16)), "flops": 0}
    if kind == "forward":
        m, k, n = case["m"], case["k"], case["n"]
        w = 1 if case["values"] == "int8" else 4
        return {"bytes": w * k * n + 4 * m * k + 4 * m * n, "flops": 2 * m * k * n}
    if kind == "sumcheck":
        return {"bytes": 2 * 16 << case["log_n"], "flops": 0}
    if kind == "commit":
        h, i, q, kv = (case[k] for k in ("hidden", "inter", "q", "kv"))
        n = h * q + 2 * h * kv + q * h + 3 * h * i
        return {"bytes": 4 * n, "flops": n * hash_ops}
    if kind == "opening":
        n = case["k"] * case["n"]
        return {"bytes": 4 * n, "flops": 2 * n * hash_ops}
    n = case["instances"] << case["log_n"]
    return {"bytes": 20 * n, "flops": 0}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The forward product in float64 over 16-bit halves (every partial sum below 2^53).  The other
    results are transcripts of a proof and have no counterpart outside a prover."""
    if case["kind"] != "forward" or case["m"] * case["k"] * case["n"] > 1 << 36:
        return None
    inp = Inputs(seed)
    a = inp.values((case["m"], case["k"]), case["values"]).cpu().to(torch.int64)
    b = inp.values((case["k"], case["n"]), case["values"]).cpu().to(torch.int64)
    total = torch.zeros((case["m"], case["n"]), dtype=torch.int64)
    for i in range(2):
        for j in range(2):
            x, y = ((a >> (16 * i)) & 0xFFFF).double(), ((b >> (16 * j)) & 0xFFFF).double()
            part = (x @ y).to(torch.int64).remainder(P)
            total = (total + part * ((1 << (16 * (i + j))) % P)).remainder(P)
    return total.to(torch.int32)
