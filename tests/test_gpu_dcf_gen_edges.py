"""DCF key generation at the edges of its lane groups on the GPU (8 lanes per
chunk of a key pair, 8 chunks to a wave, one pass 128 chunks per CU): both
parties' key bytes equal the oracle's, for one key, whole and partial waves,
several chunks and more than one pass, and nothing is written past a key."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
from gpu_util import dev, host, say
from suf_amd import native, pfss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,in_bits,plen,group", [
    (1, 64, 1, 0), (1, 1, 1, 1), (3, 13, 33, 1), (7, 64, 16, 0), (8, 32, 8, 1), (9, 5, 20, 0),
    (128 * 256 + 3, 6, 1, 1), (128 * 128 + 1, 4, 17, 0)])
def test_keys_match_oracle(n, in_bits, plen, group):
    say("dcf_gen n=%d in_bits=%d plen=%d group=%d" % (n, in_bits, plen, group))
    native.call("sufhip_init", 0)
    rng = np.random.default_rng(100 * n + in_bits)
    state = ol.mt64_bytes(17, ol.PRG_STATE_BYTES).tobytes()
    prg = ol.Prg(state)
    # Bits of alpha above in_bits are ignored.
    alpha = rng.integers(0, 2**63, size=n).astype(np.uint64)
    payload = rng.integers(0, 256, size=(n, plen), dtype=np.uint8)
    chunks = (plen + 15) // 16
    seeds = rng.integers(0, 256, size=(n, 32 * chunks), dtype=np.uint8)
    kb = pfss.dcf_key_bytes(in_bits, plen)
    out = torch.full((2, n * kb + 16), 0xA5, dtype=torch.uint8, device="cuda")
    a, p, s = dev(alpha), dev(payload), dev(seeds)
    native.call("sufhip_dcf_gen", group, in_bits, pfss._state_buf(state), a.data_ptr(),
                p.data_ptr(), plen, 0, s.data_ptr(), n, out[0].data_ptr(), out[1].data_ptr(),
                pfss._stream())
    got = host(out)
    assert (got[:, n * kb:] == 0xA5).all()
    mask = (1 << in_bits) - 1
    for i in sorted(set(range(0, n, max(1, n // 61))) | {n - 1}):
        ref = ol.myl7_gen(prg, group, in_bits, int(alpha[i]) & mask, payload[i].tobytes(), seeds[i])
        for party in (0, 1):
            assert got[party, i * kb:(i + 1) * kb].tobytes() == ref[party].tobytes(), (i, party)
