"""DCF batches on the GPU by the lanes their walks take (8 up to 160 walks per
CU, and for bits from 256 to 320; two up to 384; one above): shares equal the
oracle's at the edges of a wave's walks, of one pass of the chip and of the
rule that picks the kernel, for short and 64-level keys."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
from gpu_util import CUS, best_us, dev, host, say, u64
from suf_amd import native, pfss

pytestmark = pytest.mark.gpu

# The largest batches of 8-lane walks, of 8-lane walks of bits past a full
# pass of 2-lane ones, and of 2-lane walks.
QUAD, AGAIN, PAIR = 160 * CUS, 320 * CUS, 384 * CUS


@pytest.fixture(scope="module", autouse=True)
def _init():
    native.call("sufhip_init", 0)


@pytest.mark.parametrize("n,in_bits,plen,group", [
    (1, 64, 1, 0), (7, 1, 1, 1), (8, 13, 16, 1), (9, 64, 20, 0), (65, 32, 8, 1), (511, 37, 40, 1),
(128 * CUS + 1, 9, 8, 1), (QUAD // 2 - 3, 8, 20, 0), (QUAD, 8, 1, 0), (QUAD + 1, 8, 8, 1),
    (QUAD + 31, 11, 5, 0), (256 * CUS - 1, 7, 1, 1), (256 * CUS + 33, 10, 16, 0),
    (QUAD // 2 + 1, 6, 33, 1), (PAIR, 9, 1, 0), (PAIR + 1, 8, 8, 1),
    (PAIR + 64 * 7 + 5, 11, 1, 0),
    (50021, 32, 8, 1), (QUAD + 77, 64, 16, 1), (QUAD // 2 + 33, 64, 20, 0), (QUAD + 5, 64, 1, 0),
    (256 * CUS, 64, 1, 1), (AGAIN, 64, 1, 0), (AGAIN - 64 * 3 - 11, 21, 16, 0),
    (AGAIN + 1, 64, 1, 0), (PAIR - 3, 40, 8, 1), (PAIR // 2 - 5, 37, 20, 1),
    (PAIR // 3 + 5, 64, 40, 0), (PAIR // 64 + 7, 6, 1024, 1), (PAIR // 2 + 21, 33, 17, 1)])
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


def test_many_chunks_past_the_two_lane_limit():
    """64-chunk payloads on either side of the limit where a lane takes a walk:
    a third more walks cost about as much more, not one lane running an
    element's 64 walks in turn (50 times)."""
    state = ol.mt64_bytes(31, ol.PRG_STATE_BYTES).tobytes()
    in_bits, plen = 16, 1024
    us = {}
    for n in (18 * CUS // 4, 25 * CUS // 4):
        xs = torch.arange(n, dtype=torch.int64, device="cuda")
        seeds = torch.randint(0, 256, (n, 32 * 64), dtype=torch.uint8, device="cuda")
        payload = torch.ones(plen, dtype=torch.uint8, device="cuda")
        k0, _ = pfss.dcf_gen(1, in_bits, state, xs, payload, seeds)
        out = torch.empty((n, plen), dtype=torch.uint8, device="cuda")
        us[n] = best_us(lambda: pfss.dcf_eval(1, in_bits, plen, state, k0, xs, native.DCF_OUT_BYTES,
                                              plen, out=out), reps=4, tries=5)
    say("dcf 64 chunks: %s us" % us)
    few, many = us.values()
    assert many < 4 * few
