"""The boolean network's split over a gate's segments (one wave per segment of
64 elements, up to 8 waves; two and one where the triples exceed 128 and 256
MB): both parties' shares equal the oracle's two-party composition for one
segment, more segments than waves and up to 8 outputs, at whole and partial
groups of 64 elements, and the large batches' equal those of their own parts."""
import numpy as np
import pytest
import torch

import test_gpu_composite as base
from gpu_util import say
from suf_amd import composite, native

pytestmark = pytest.mark.gpu


def _spec(pieces, ell):
    rng = np.random.default_rng(pieces + ell)
    cuts = sorted({int(v) for v in rng.integers(1, 1 << 63, pieces - 1)}) if pieces > 1 else []
    preds = [("lt", 1 << 62), ("ltlow", 9, 100), ("msb",)]
    exprs = [("and", ("var", 0), ("var", 1)), ("or", ("var", 2), ("not", ("var", 1))),
             ("xor", ("var", 0), ("var", 2)), ("not", ("var", 2))]
    # A gate takes 32 wrap bits, one per variable: 14 expressions, then constants.
    pool = [exprs[k % 4] for k in range(14)] + [("const", k & 1) for k in range(pieces * ell)]
    order = rng.permutation((len(cuts) + 1) * ell)
    bools = {int(o): pool[k] for k, o in enumerate(order)}
    return {"alpha": [0] + cuts, "preds": preds,
            "pieces": [{"arith": [k + 3], "bools": [bools[k * ell + j] for j in range(ell)]}
                       for k in range(len(cuts) + 1)]}


@pytest.mark.parametrize("pieces,ell,n", [(1, 1, 33), (1, 8, 65), (3, 5, 64), (9, 8, 200),
                                          (20, 2, 1000), (7, 3, 129), (30, 1, 63)])
def test_segments(pieces, ell, n):
    native.call("sufhip_init", 0)
    base._run(_spec(pieces, ell), n, 11 + n, share_check=True)


@pytest.mark.parametrize("n", [104000 + 37, 208000 + 5])
def test_batches_past_the_cache_equal_their_parts(n):
    """A batch on two waves and on one, against the same triples and bits cut
    into parts that take a wave per segment."""
    say("composite network n=%d" % n)
    native.call("sufhip_init", 0)
    gate = composite.CompositeGate(_spec(5, 2), n, base.STATE, seed=3)
    assert 128 << 20 < n * gate.T * 48 and (n * gate.T * 48 > 256 << 20) == (n > 200000)
    g = torch.Generator(device="cuda").manual_seed(n)
    for t in gate.pred + gate.cutb:
        t.copy_(torch.randint(0, 2, t.shape, dtype=torch.uint8, device="cuda", generator=g))
    call = lambda a: native.call("sufhip_composite_bool2", native.ctypes.byref(a), None)  # noqa: E731
    whole = [torch.empty(n * 2, dtype=torch.int64, device="cuda") for _ in range(2)]
    call(gate.args(whole))
    step = 60000
    for lo in range(0, n, step):
        m = min(step, n - lo)
        cut = lambda t: t.reshape(-1, n)[:, lo:lo + m].contiguous()  # noqa: E731
        out = [torch.empty(m * 2, dtype=torch.int64, device="cuda") for _ in range(2)]
        a = gate.args(out)
        a.n = m
        held = []
        for p in (0, 1):
            parts = [cut(t) for t in (gate.pred[p], gate.cutb[p], gate.bit_tri[p], gate.tri[p])]
            held.append(parts)
            a.pred[p], a.cut[p], a.bit_tri[p], a.tri[p] = (t.data_ptr() for t in parts)
        call(a)
        for p in (0, 1):
            assert torch.equal(out[p], whole[p][2 * lo:2 * (lo + m)]), (lo, p)
