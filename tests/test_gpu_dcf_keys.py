"""sufhip_dcf_eval_keys on the GPU: the bits of many broadcast keys at the same
points equal the one-key evaluation's and the oracle's, whatever the points
share: all equal, a short interval (a long common prefix), an interval across
0 (no common prefix), anything; for tiles of 8-lane walks and of one-lane
walks with an expanded subtree, few-bit keys, more keys than one launch takes
and, from 1024 points per CU on, launches of one key width."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
from gpu_util import CUS, dev, host, say
from suf_amd import native, pfss

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


def _points(shape, n, centre, rng):
    if shape == "equal":
        return np.full(n, centre, dtype=np.uint64)
    if shape == "random":
        return rng.integers(0, 1 << 64, n, dtype=np.uint64)
    base = 0 if shape == "wrap" else centre
    return np.array([(base + int(d)) & M64 for d in rng.integers(-(1 << 20), 1 << 20, n)],
                    dtype=np.uint64)


@pytest.mark.parametrize("shape", ["equal", "near", "wrap", "random"])
@pytest.mark.parametrize("n,bits", [
    (1, [64]), (9, [1, 64, 12]), (300, [64] * 3 + [5]), (8 * CUS + 1, [64, 64]),
    (257 * CUS + 3, [64, 9]), (4096, [64] * 20 + [12] * 2), (70000, [64] * 21), (65, [17] * 65),
    (1024 * CUS - 1, [12, 64, 5]), (1024 * CUS + 77, [12, 64, 64, 9, 64, 12] + [64] * 4 + [3] * 45)])
def test_bits_match_single_key_evaluation(n, bits, shape):
    say("dcf_eval_keys n=%d keys=%d shape=%s" % (n, len(bits), shape))
    native.call("sufhip_init", 0)
    rng = np.random.default_rng(n + len(bits))
    state = ol.mt64_bytes(23, ol.PRG_STATE_BYTES).tobytes()
    prg = ol.Prg(state)
    centre = int(rng.integers(1 << 62, 1 << 63))
    xs = _points(shape, n, centre, rng)
    xd = dev(xs)
    jobs = (native.DcfKeyJob * (2 * len(bits)))()
    out = torch.full((2 * len(bits), n + 8), 7, dtype=torch.uint8, device="cuda")
    keys = []
    for q, b in enumerate(bits):
        m = (1 << b) - 1
        # Thresholds at a point, beside one and anywhere.
        theta = [int(xs[q % n]), int(xs[-1]) + 1, int(rng.integers(0, 1 << 63))][q % 3] & m
        seed = rng.integers(0, 256, size=(1, 32), dtype=np.uint8)
        k = pfss.dcf_gen(0, b, state, dev(np.array([theta], dtype=np.uint64)),
                         dev(np.array([1], dtype=np.uint8)), dev(seed))
        for p in (0, 1):
            j = 2 * q + p
            jobs[j] = (k[p].data_ptr(), k[p].shape[-1], out[j].data_ptr(), b)
        keys.append((b, theta, k))
    native.call("sufhip_dcf_eval_keys", pfss._state_buf(state), jobs, len(jobs), xd.data_ptr(), n,
                pfss._stream())
    got = host(out)
    assert (got[:, n:] == 7).all()
    for q, (b, theta, k) in enumerate(keys):
        m = np.uint64((1 << b) - 1)
        assert np.array_equal(got[2 * q, :n] ^ got[2 * q + 1, :n],
                              ((xs & m) < np.uint64(theta)).astype(np.uint8)), q
        for p in (0, 1):
            one = host(pfss.dcf_eval(0, b, 1, state, k[p], xd, broadcast=True))
            assert np.array_equal(got[2 * q + p, :n], one), (q, p)
        kh = host(k[0])[0]
        for i in sorted({0, n // 2, n - 1}):
            ref = ol.myl7_eval(prg, 0, b, kh, int(xs[i] & m), 1)[0] & 1
            assert got[2 * q, i] == ref, (q, i)


def test_bad_jobs_are_refused():
    say("dcf_eval_keys refused")
    xs = torch.zeros(4, dtype=torch.int64, device="cuda")
    key = torch.zeros(2152, dtype=torch.uint8, device="cuda")
    out = torch.zeros(4, dtype=torch.uint8, device="cuda")
    state = pfss._state_buf(bytes(128))
    job = (native.DcfKeyJob * 1)()
    for bad in ((None, 2152, out.data_ptr(), 64), (key.data_ptr(), 2151, out.data_ptr(), 64),
                (key.data_ptr(), 2152, None, 64), (key.data_ptr(), 2152, out.data_ptr(), 65)):
        job[0] = bad
        with pytest.raises(native.SufHipError):
            native.call("sufhip_dcf_eval_keys", state, job, 1, xs.data_ptr(), 4, pfss._stream())
    job[0] = (key.data_ptr(), 2152, out.data_ptr(), 64)
    native.call("sufhip_dcf_eval_keys", state, job, 1, xs.data_ptr(), 0, pfss._stream())
    native.call("sufhip_dcf_eval_keys", state, job, 0, xs.data_ptr(), 4, pfss._stream())
