"""The boolean network's split over a gate's segments (one wave per segment of
64 elements, up to 8 waves): both parties' shares equal the oracle's two-party
composition for one segment, more segments than waves and up to 8 outputs, at
whole and partial groups of 64 elements."""
import numpy as np
import pytest

import test_gpu_composite as base
from suf_amd import native

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
