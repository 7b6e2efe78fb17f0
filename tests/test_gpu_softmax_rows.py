"""How the softmax block deals rows to workgroups on the GPU: shares equal the
launch-by-launch path's for one row, rows of one element, lengths at the
limits of one, two and four scores per lane and of six and eight rows per
workgroup, more rows than one pass of the chip takes, and either keystream
policy."""
import numpy as np
import pytest
import torch

import test_gpu_softmax_ln as base
from gpu_util import say, u64
from suf_amd import native, pfss, softmax

pytestmark = pytest.mark.gpu


def _lens(shape, seed):
    rng = np.random.default_rng(seed)
    rows, longest = shape
    lens = rng.integers(1, longest + 1, rows)
    lens[rng.integers(0, rows)] = longest
    return lens


@pytest.mark.parametrize("per_party", [False, True])
@pytest.mark.parametrize("shape", [(1, 1), (1, 512), (40, 1), (9, 96), (9, 97), (70, 192),
                                   (70, 193), (300, 384), (300, 385), (2100, 20), (1600, 130)])
def test_rows_match_step_path(shape, per_party):
    say("softmax rows=%d longest=%d per_party=%d" % (shape + (per_party,)))
    native.call("sufhip_init", 0)
    lens = _lens(shape, 5 + shape[0])
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    n = int(offs[-1])
    x = base._pair_dev(*base._share(base._scores(offs, 31), 32))
    sm = softmax.SoftmaxBlock(offs, base.STATE, base.F, seed=9)
    got, ref = ([torch.full((n + 2,), -3, dtype=torch.int64, device="cuda") for _ in range(2)]
                for _ in range(2))
    with pfss.keystream_per_party(per_party):
        sm.eval2(x, [t[:n] for t in got])
    sm.eval2(x, [t[:n] for t in ref], fused=False)
    for p in (0, 1):
        assert np.array_equal(u64(got[p]), u64(ref[p])), p
