"""What the framework's speed is measured on: its online gates and their
dealer's key generation, each through the Python entry points that a program
calls, both parties on one GPU.

Every output is an integer: key bytes, DCF share bits, or additive shares
mod 2^64.  Two implementations of a gate agree bit for bit on the same dealer
material, so the tolerance is "exact" everywhere.  A share is also
pseudo-random (an AES keystream or a PRG walk decides it), so it has no value
that plain 64-bit arithmetic could give: exact() returns None.

Kinds of cases (field "kind"):
  dcf         per-element comparison keys at public masked points, both
              parties (the batch evaluation of SUF's PFSS backend)
  dcf_gen     the dealer's comparison keys
  trunc       one truncation gate over a batch, both parties
  spline      a piecewise-cubic activation, online phase as a HIP graph
  softmax_ln  causal softmax rows and a LayerNorm, online phase as a HIP graph
  matmul      Beaver product with its truncation, online phase as a HIP graph
  composite   a gate with boolean outputs (predicates, selector network)
  layer       a GPT-2-shaped transformer layer, online phase as a HIP graph
A program captures the fixed chains of launches once (suf_amd.tasks.capture)
and replays them; the single gates are called directly.
"""
import math

import numpy as np
import torch

from suf_amd import composite, layer, layernorm, matmul_gate, native, pfss, softmax, spline, tasks

F = 12  # fractional bits of the fixed-point values
M64 = (1 << 64) - 1
T62, T63 = 1 << 62, 1 << 63
GROUPS = {"xor": native.GROUP_XOR, "add": native.GROUP_ADD}
MODES = {"bit": native.DCF_OUT_BIT, "bytes": native.DCF_OUT_BYTES,
         "packed": native.DCF_OUT_PACKED}
TRUNCS = {"tr": native.TRUNC_TR, "ars": native.TRUNC_ARS, "gapars": native.TRUNC_GAPARS}

# The two shapes of composite gate: the sign output of a ReLU, and one over
# every predicate kind and connective (four pieces, two boolean outputs).
COMPOSITES = {
    "drelu": {"alpha": [0, T63], "preds": [],
              "pieces": [{"arith": [1], "bools": [("const", 1)]},
                         {"arith": [0], "bools": [("const", 0)]}]},
    "mixed": {"alpha": [0, T62, T63, T63 + T62],
              "preds": [("lt", 1000), ("ltlow", 12, 2048), ("msb",), ("msb_add", 5000)],
              "pieces": [
                  {"arith": [7], "bools": [("and", ("var", 0), ("not", ("var", 1))),
                                           ("or", ("var", 2), ("var", 3))]},
                  {"arith": [11], "bools": [("xor", ("var", 1), ("var", 3)), ("const", 1)]},
                  {"arith": [13], "bools": [("not", ("var", 0)),
                                            ("and", ("or", ("var", 1), ("var", 2)), ("var", 3))]},
                  {"arith": [17], "bools": [("const", 0), ("var", 2)]}]},
}


def listed():
    return [
        # A handful of comparisons on their own: the selection of a few
        # hundred values, one key per value.  Latency decides.
        {"name": "dcf_few", "kind": "dcf", "n": 300, "in_bits": 64, "payload": 1, "group": "xor",
         "mode": "bit"},
        # The batch the framework's headline is quoted on.
        {"name": "dcf_batch", "kind": "dcf", "n": 1 << 20, "in_bits": 64, "payload": 1,
         "group": "xor", "mode": "bit"},
        # Whole additive u64 shares on a narrower ring, a ragged batch.
        {"name": "dcf_shares_u64", "kind": "dcf", "n": 50021, "in_bits": 32, "payload": 8,
         "group": "add", "mode": "bytes"},
        # The dealer's half of a quarter of the headline batch.
        {"name": "dcf_keys", "kind": "dcf_gen", "n": 1 << 18, "in_bits": 64, "payload": 1,
         "group": "xor"},
        # A faithful arithmetic shift of a 128 x 768 activation: carry, wrap
        # and sign comparisons under one broadcast key.
        {"name": "trunc_ars_128x768", "kind": "trunc", "trunc": "ars", "f": 12, "n": 128 * 768},
        # SiLU / GeLU-shaped activation at the size of the benchmark.
        {"name": "spline_2p20", "kind": "spline", "n": 1 << 20, "per_party": True},
        # Attention's softmax and a LayerNorm at GPT-2-small's sizes, 128 tokens.
        {"name": "softmax_ln_128", "kind": "softmax_ln", "heads": 12, "seq": 128, "rows": 128,
         "cols": 768, "per_party": True},
        # A longer odd context, fewer heads, an odd width.
        {"name": "softmax_ln_300", "kind": "softmax_ln", "heads": 4, "seq": 300, "rows": 300,
         "cols": 1001, "per_party": True},
        # A shared-times-shared product at an MLP's shape.
        {"name": "matmul_128x768x3072", "kind": "matmul", "M": 128, "K": 768, "N": 3072},
        # The same kind of product where no dimension fits a tile.
        {"name": "matmul_77x300x1000", "kind": "matmul", "M": 77, "K": 300, "N": 1000},
        # A gate of four predicates and two boolean outputs over a few
        # thousand values: many broadcast keys, small batch.
        {"name": "composite_mixed_4096", "kind": "composite", "gate": "mixed", "n": 4096},
        # The whole layer.
        {"name": "layer_gpt2_small_128", "kind": "layer", "seq": 128, "d": 768, "heads": 12,
         "ffn": 3072, "per_party": True},
    ]


def _spread(rng, lo, hi):
    """An integer of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["dcf", "dcf", "dcf_gen", "trunc", "spline", "softmax_ln", "matmul",
                       "matmul", "composite", "layer"])
    if kind == "dcf":
        mode = rng.choice(["bit", "bit", "packed", "bytes"])
        payload = rng.choice([8, 16, 20]) if mode == "bytes" else 1
        return {"kind": kind, "n": _spread(rng, 60, (1 << 20) if payload == 1 else 1 << 18),
                "in_bits": rng.choice([64, 64, 32, rng.randint(8, 63)]), "payload": payload,
                "group": rng.choice(["xor", "add"]), "mode": mode}
    if kind == "dcf_gen":
        return {"kind": kind, "n": _spread(rng, 60, 1 << 18),
                "in_bits": rng.choice([64, 64, 32, rng.randint(8, 63)]),
                "payload": rng.choice([1, 1, 8, 16]), "group": rng.choice(["xor", "add"])}
    if kind == "trunc":
        return {"kind": kind, "trunc": rng.choice(["tr", "ars", "gapars"]),
                "f": rng.choice([F, F, 2 * F, rng.randint(8, 16)]),
                "n": _spread(rng, 256, 1 << 18)}
    if kind == "spline":
        return {"kind": kind, "n": _spread(rng, 500, 1 << 20), "per_party": rng.random() < 0.5}
    if kind == "softmax_ln":
        seq = _spread(rng, 8, 400)
        return {"kind": kind, "heads": rng.randint(1, max(1, min(16, 110000 // (seq * seq)))),
                "seq": seq, "rows": _spread(rng, 1, 400), "cols": _spread(rng, 64, 2048),
                "per_party": rng.random() < 0.5}
    if kind == "matmul":
        tile = rng.choice([1, 1, 32])
        at = lambda lo, hi: max(tile, _spread(rng, lo, hi) // tile * tile)  # noqa: E731
        return {"kind": kind, "M": at(1, 256), "K": at(16, 1024), "N": at(16, 2048)}
    if kind == "composite":
        return {"kind": kind, "gate": rng.choice(sorted(COMPOSITES)),
                "n": _spread(rng, 100, 1 << 16)}
    heads = rng.choice([2, 4, 8, 12])
    return {"kind": kind, "seq": 32 * rng.randint(1, 4), "d": 64 * heads, "heads": heads,
            "ffn": 64 * heads * rng.choice([2, 4]), "per_party": rng.random() < 0.5}


class _Rand:
    """Seeded words and fixed-point values on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))
        self.host = np.random.default_rng(int(seed))

    def words(self, *shape):
        return torch.randint(-T63, T63 - 1, shape, dtype=torch.int64, device="cuda",
                             generator=self.g)

    def fixed(self, n, sigma=1.0, clip=None):
        v = torch.randn(n, device="cuda", generator=self.g) * sigma
        v = v if clip is None else v.clamp(-clip, clip)
        return (v * (1 << F)).round().to(torch.int64)

    def shares(self, v):
        s = self.words(v.numel())
        return s, v - s

    def prg_state(self):
        return self.host.integers(0, 256, pfss.PRG_STATE_BYTES, dtype=np.uint8).tobytes()

    def seed(self):
        return int(self.host.integers(1, 1 << 40))


def _pair(n):
    return [torch.empty(n, dtype=torch.int64, device="cuda") for _ in range(2)]


def _dcf_material(case, r):
    n, bits = case["n"], case["in_bits"]
    low = M64 if bits == 64 else (1 << bits) - 1
    low = low - (1 << 64) if low >> 63 else low
    alpha = r.words(n) & low
    payload = torch.zeros(case["payload"], dtype=torch.uint8, device="cuda")
    payload[0] = 1
    seeds = r.words(n, 4 * ((case["payload"] + 15) // 16)).view(torch.uint8)
    return alpha, payload, seeds, low


def _graph(case, fn):
    """fn() captured under the case's keystream policy."""
    with pfss.keystream_per_party(case.get("per_party", False)):
        return tasks.capture(fn)


def prepare(case, seed):
    r = _Rand(seed)
    prg = r.prg_state()
    kind = case["kind"]
    st = {"case": dict(case), "prg": prg}
    if kind == "dcf":
        alpha, payload, seeds, low = _dcf_material(case, r)
        st["keys"] = pfss.dcf_gen(GROUPS[case["group"]], case["in_bits"], prg, alpha, payload,
                                  seeds)
        st["xs"] = (r.fixed(case["n"]) + alpha) & low
    elif kind == "dcf_gen":
        st["alpha"], st["payload"], st["seeds"], _ = _dcf_material(case, r)
    elif kind == "trunc":
        rnd = r.host.integers(0, M64, native.TRUNC_RAND_WORDS, dtype=np.uint64, endpoint=True)
        st["keys"] = pfss.trunc_gen(TRUNCS[case["trunc"]], case["f"], prg, rnd)
        x = (r.fixed(case["n"], 1.0) * r.fixed(case["n"], 4.0))
        x = x.abs() if case["trunc"] == "tr" else x
        mask = int(rnd[0])
        st["xhat"] = x + (mask - (1 << 64) if mask >> 63 else mask)
    elif kind == "spline":
        n = case["n"]
        alpha, coeffs = spline.spline_spec(F, seed=r.seed())
        gate = spline.SplineGate(n, alpha, coeffs, prg, F, seed=r.seed())
        x, out = r.shares(r.fixed(n, 3.0, 8.0)), _pair(n)
        # The truncations' key-only halves first, on the same stream.
        st["graph"] = _graph(case, lambda: gate.eval2(
            x, out, prep=(tasks.Prepared(None, [gate.truncs()]), 0)))
        st["out"], st["keep"] = out, (gate, x)
    elif kind == "softmax_ln":
        rows, cols = case["rows"], case["cols"]
        offs = softmax.causal_offsets(case["heads"], case["seq"])
        sm = softmax.SoftmaxBlock(offs, prg, F, seed=r.seed())
        ln = layernorm.LayerNormBlock(rows, cols, prg, F, seed=r.seed())
        xs, so = r.shares(r.fixed(int(offs[-1]), 2.0)), _pair(int(offs[-1]))
        xl, lo = r.shares(r.fixed(rows * cols)), _pair(rows * cols)

        def both():
            prep = tasks.Prepared(None, [sm.truncs() + ln.truncs()])
            sm.eval2(xs, so, prep=(prep, 0))
            ln.eval2(xl, lo, prep=(prep, 0))

        st["graph"] = _graph(case, both)
        st["out"], st["keep"] = so + lo, (sm, ln, xs, xl)
    elif kind == "matmul":
        M, K, N = case["M"], case["K"], case["N"]
        gate = matmul_gate.BeaverMatmulTrunc(M, K, N, prg, F, seed=r.seed())
        X, W = r.shares(r.fixed(M * K)), r.shares(r.fixed(K * N, 0.02))
        out = _pair(M * N)
        st["graph"] = _graph(case, lambda: gate.eval2(X, W, out))
        st["out"], st["keep"] = out, (gate, X, W)
    elif kind == "composite":
        n, spec = case["n"], COMPOSITES[case["gate"]]
        gate = composite.CompositeGate(spec, n, prg, seed=r.seed())
        mask = gate.r_in - (1 << 64) if gate.r_in >> 63 else gate.r_in
        st["gate"], st["xhat"] = gate, r.fixed(n) + mask
        st["bools"] = _pair(n * gate.ell)
        st["words"] = _pair(n * gate.r)
    else:
        seq, d, heads, ffn = case["seq"], case["d"], case["heads"], case["ffn"]
        weight = lambda k, m: r.fixed(k * m, 0.02).cpu().numpy().reshape(k, m)  # noqa: E731
        weights = {"Wqkv": weight(d, 3 * d), "Wout": weight(d, d), "W1": weight(d, ffn),
                   "W2": weight(ffn, d)}
        net = layer.TransformerLayer(prg, weights, seq=seq, d=d, heads=heads, ffn=ffn,
                                     frac_bits=F, seed=r.seed())
        x, out = r.shares(r.fixed(seq * d)), _pair(seq * d)
        st["graph"] = _graph(case, lambda: net.eval2(x, out))
        st["out"], st["keep"] = out, (net, x)
    return st


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    case, prg = state["case"], state["prg"]
    if case["kind"] == "dcf":
        return [pfss.dcf_eval(GROUPS[case["group"]], case["in_bits"], case["payload"], prg, keys,
                              state["xs"], MODES[case["mode"]], case["payload"])
                for keys in state["keys"]]
    if case["kind"] == "dcf_gen":
        return list(pfss.dcf_gen(GROUPS[case["group"]], case["in_bits"], prg, state["alpha"],
                                 state["payload"], state["seeds"]))
    if case["kind"] == "trunc":
        return [pfss.trunc_eval(TRUNCS[case["trunc"]], case["f"], prg, key, state["xhat"])
                for key in state["keys"]]
    state["gate"].eval2(state["xhat"], state["bools"], state["words"])
    return state["bools"] + state["words"]


def work(case):
    """Bytes of each input and output once; a u64 multiply-add counts as two
    operations.  The PRG's and keystreams' AES rounds are in neither."""
    kind = case["kind"]
    if kind in ("dcf", "dcf_gen"):
        n, plen = case["n"], case["payload"]
        key = pfss.dcf_key_bytes(case["in_bits"], plen)
        if kind == "dcf_gen":
            return {"bytes": n * (2 * key + 8 + 32 * ((plen + 15) // 16)), "flops": 0}
        out = {"bit": 1.0, "packed": 0.125, "bytes": plen}[case["mode"]]
        return {"bytes": n * 2 * (key + 8 + out), "flops": 0}
    if kind == "trunc":
        return {"bytes": case["n"] * 2 * 16, "flops": 0}
    if kind == "spline":
        # Per element and party: x, three triples of three words, the output.
        return {"bytes": case["n"] * 2 * 8 * 11, "flops": case["n"] * 24}
    if kind == "softmax_ln":
        heads, seq, n = case["heads"], case["seq"], case["rows"] * case["cols"]
        scores = heads * seq * (seq + 1) // 2
        # Scores: x, nExp's nine triple words, the product's a and c, out.
        # LayerNorm: x, the square's three triple words, the product's two, out.
        return {"bytes": scores * 2 * 8 * 13 + n * 2 * 8 * 7 + heads * seq * 2 * 8 * 10 +
                case["rows"] * 2 * 8 * 13, "flops": scores * 32 + n * 16}
    if kind == "matmul":
        M, K, N = case["M"], case["K"], case["N"]
        # Shares and triple shares of both operands, C and the output.
        return {"bytes": 8 * 4 * (M * K + K * N + M * N), "flops": 8 * M * K * N}
    if kind == "composite":
        return {"bytes": case["n"] * (8 + 2 * 8 * 3 + 2 * 8 * 9), "flops": 0}
    seq, d, heads, ffn = case["seq"], case["d"], case["heads"], case["ffn"]
    weights = 4 * d * d + 2 * d * ffn
    scores = heads * seq * (seq + 1) // 2
    nbytes = 2 * weights + 2 * 8 * (2 * seq * d + 6 * 2 * seq * d + scores * 12 + 9 * seq * ffn +
                                    heads * (5 * seq * d // heads + 2 * seq * seq))
    return {"bytes": nbytes, "flops": 4 * seq * weights + 8 * 2 * seq * seq * d}


def tolerance(case):
    return "exact"


def exact(case, seed):
    return None
