"""Truncation gates whose keys are walked per element, on the GPU, over what a
tile's points may share: one value, a short interval around the mask, an
interval across 0, anything.  Shares equal the oracle's and reconstruct the
shift, for one party at a time and for both in one launch, at tiles of
8-lane walks and of one-lane walks and with carry keys above and below the
full-domain table's width."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
from gpu_util import CUS, dev, say, u64
from suf_amd import native, pfss

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1
STATE = ol.mt64_bytes(3, ol.PRG_STATE_BYTES).tobytes()
PRG = ol.Prg(STATE)


def _signed(v):
    return v - (1 << 64) if v >> 63 else v


@pytest.mark.parametrize("shape", ["equal", "near", "wrap", "random"])
@pytest.mark.parametrize("kind,f,n", [
    (ol.TRUNC_TR, 12, 1), (ol.TRUNC_ARS, 12, 9), (ol.TRUNC_ARS, 24, 300),
    (ol.TRUNC_TR, 16, CUS * 128 + 1), (ol.TRUNC_ARS, 12, CUS * 64 + 3),
    (ol.TRUNC_ARS, 12, CUS * 128 + 129), (ol.TRUNC_ARS, 24, 98304 + 5),
    (ol.TRUNC_GAPARS, 20, CUS * 256 + 7), (ol.TRUNC_GAPARS, 31, 50)])
def test_tiles(kind, f, n, shape):
    say("trunc tiles kind=%d f=%d n=%d shape=%s" % (kind, f, n, shape))
    native.call("sufhip_init", 0)
    rng = np.random.default_rng(n + f)
    rnd = rng.integers(0, 1 << 64, ol.TRUNC_RAND_WORDS, dtype=np.uint64)
    if shape == "wrap":
        rnd[0] = np.uint64(3)
    r = int(rnd[0])
    lim = (1 << 62) - 1 if kind == ol.TRUNC_GAPARS else (1 << 63) - 1
    if shape == "equal":
        x = [12345 << 7] * n
    elif shape == "random":
        x = [int(v) for v in rng.integers(-lim, lim, n)]
    else:
        x = [int(v) for v in rng.integers(-(1 << 29), 1 << 29, n)]
    if kind == ol.TRUNC_TR:
        x = [abs(v) for v in x]
    xhat = np.array([(v + r) & M64 for v in x], dtype=np.uint64)
    xd = dev(xhat)
    keys = pfss.trunc_gen(kind, f, STATE, rnd)
    ok = ol.trunc_gen(PRG, kind, f, rnd)
    one = [pfss.trunc_eval(kind, f, STATE, k, xd) for k in keys]
    wb = native.load().sufhip_trunc_work_bytes(f, n)
    work = [torch.empty(wb // 8, dtype=torch.int64, device="cuda") for _ in range(2)]
    both = [torch.empty(n, dtype=torch.int64, device="cuda") for _ in range(2)]
    st = pfss._state_buf(STATE)
    for k, w in zip(keys, work):
        native.call("sufhip_trunc_prepare", kind, f, st, k.data_ptr(), k.numel(), n, w.data_ptr(),
                    wb, pfss._stream())
    native.call("sufhip_trunc_finish2", kind, f, st, keys[0].data_ptr(), keys[1].data_ptr(),
                keys[0].numel(), xd.data_ptr(), n, both[0].data_ptr(), both[1].data_ptr(),
                work[0].data_ptr(), work[1].data_ptr(), wb, pfss._stream())
    y = [u64(t) for t in one]
    for p in (0, 1):
        assert np.array_equal(u64(both[p]), y[p])
    rec = y[0] + y[1]
    want = np.array([(v >> f) & M64 for v in x], dtype=np.uint64)
    assert np.array_equal(rec, want)
    idx = np.unique(np.concatenate([[0, n - 1], rng.integers(0, n, min(n, 40))]))
    for p in (0, 1):
        assert np.array_equal(y[p][idx], ol.trunc_eval(PRG, kind, f, ok[p], xhat[idx]))
