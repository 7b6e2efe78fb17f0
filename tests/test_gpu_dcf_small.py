"""Small DCF batches on the GPU (8 lanes per walk up to 160 walks per CU, two
up to 320, one above): shares equal the oracle's at the edges of a wave's
walks, of one pass of the chip and of the rule that picks the kernel."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
from gpu_util import dev, host, say, u64
from suf_amd import native, pfss

pytestmark = pytest.mark.gpu

CUS = 256
QUAD, PAIR = 160 * CUS, 320 * CUS  # the largest batches of 8-lane and 2-lane walks


@pytest.fixture(scope="module", autouse=True)
def _init():
    native.call("sufhip_init", 0)


@pytest.mark.parametrize("n,in_bits,plen,group", [
    (1, 64, 1, 0), (7, 1, 1, 1), (8, 13, 16, 1), (9, 64, 20, 0), (65, 32, 8, 1), (511, 37, 40, 1),
(128 * CUS + 1, 9, 8, 1), (QUAD // 2 - 3, 8, 20, 0), (QUAD, 8, 1, 0), (QUAD + 1, 8, 8, 1),
    (QUAD + 31, 11, 5, 0), (256 * CUS - 1, 7, 1, 1), (256 * CUS + 33, 10, 16, 0),
    (QUAD // 2 + 1, 6, 33, 1), (PAIR, 9, 1, 0), (PAIR + 1, 8, 8, 1),
    (PAIR + 64 * 7 + 5, 11, 1, 0)])
@pytest.mark.parametrize("broadcast", [False, True])
def test_small_batches_match_oracle(n, in_bits, plen, group, broadcast):
    say("dcf small n=%d in_bits=%d plen=%d group=%d bcast=%d" % (n, in_bits, plen, group, broadcast))
    rng = np.random.default_rng(n + in_bits)
    state = ol.mt64_bytes(31, ol.PRG_STATE_BYTES).tobytes()
    prg = ol.Prg(state)
    nk = 1 if broadcast else n
    mask = np.uint64((1 << in_bits) - 1)
    alpha = rng.integers(0, 2**63, size=nk).astype(np.uint64) & mask
    payload = rng.integers(1, 256, size=plen, dtype=np.uint8)
    payload[0] |= 1
    seeds = rng.integers(0, 256, size=(nk, 32 * ((plen + 15) // 16)), dtype=np.uint8)
    xs = alpha + rng.integers(0, 7, size=n).astype(np.uint64) - np.uint64(3)
    xs[::3] = rng.integers(0, 2**63, size=len(xs[::3])).astype(np.uint64) * np.uint64(2)
    keys = pfss.dcf_gen(group, in_bits, state, dev(alpha), dev(payload), dev(seeds))
    xd = dev(xs)
    picked = sorted(set(range(0, n, max(1, n // 97))) | {n - 1, max(0, n - 9)})
    bits = []
    for k in keys:
        kh = host(k[torch.tensor(picked if not broadcast else [0], device="cuda")])
        full = host(pfss.dcf_eval(group, in_bits, plen, state, k, xd, native.DCF_OUT_BYTES, plen,
                                  broadcast=broadcast))
        bit = host(pfss.dcf_eval(group, in_bits, plen, state, k, xd, broadcast=broadcast))
        words = u64(pfss.dcf_eval(group, in_bits, plen, state, k, xd, native.DCF_OUT_PACKED,
                                  broadcast=broadcast))
        for j, i in enumerate(picked):
            x = int(xs[i] & mask)
            ref = ol.myl7_eval(prg, group, in_bits, kh[0 if broadcast else j], x, plen)
            assert full[i].tobytes() == ref.tobytes(), i
        assert np.array_equal(bit, full[:, 0] & 1)
        packed = np.unpackbits(words.view(np.uint8), bitorder="little")
        assert np.array_equal(packed[:n], bit) and not packed[n:].any()
        bits.append(bit)
    assert np.array_equal(bits[0] ^ bits[1],
                          np.where((xs & mask) < alpha, payload[0] & 1, 0).astype(np.uint8))
