"""LayerNorm of more rows than the GPU has CUs (256 lanes per row, two rows to
a CU): shares equal the launch-per-step path's at row counts on both sides of
the rule and widths at its limits."""
import numpy as np
import pytest
import torch

import test_gpu_softmax_ln as base
from gpu_util import say, u64
from suf_amd import layernorm, native, pfss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(256, 40), (257, 1), (257, 256), (300, 1001), (700, 513),
                                       (260, 1024), (259, 1025), (1100, 70)])
def test_many_rows_match_step_path(rows, cols):
    say("layernorm rows=%d cols=%d" % (rows, cols))
    native.call("sufhip_init", 0)
    x = pfss.host_normal_fixed(61, 1.0, 0.0, base.F, rows * cols)
    xs = base._pair_dev(*base._share(x, 62))
    ln = layernorm.LayerNormBlock(rows, cols, base.STATE, base.F, seed=15)
    outs = []
    for fused in (True, False):
        out = [torch.full((rows * cols + 2,), -3, dtype=torch.int64, device="cuda")
               for _ in range(2)]
        ln.eval2(xs, [t[:rows * cols] for t in out], fused=fused)
        outs.append([u64(t) for t in out])
    for p in (0, 1):
        assert np.array_equal(outs[0][p][:-2], outs[1][p][:-2]), p
        assert np.array_equal(outs[0][p][-2:], outs[1][p][-2:])
