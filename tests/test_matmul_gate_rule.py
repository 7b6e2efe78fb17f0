"""Which products the matmul gate runs in its padded matrix-core form (CPU)."""
import pytest

pytest.importorskip("torch")
from suf_amd.matmul_gate import padded_form  # noqa: E402


@pytest.mark.parametrize("M,K,N,padded", [
    (0, 32, 32, False), (32, 0, 32, False), (1, 1, 1, True), (32, 4096, 32, True),
    (32, 4097, 32, False), (1 << 21, 32, 64, True),            # whole extents: as large as ever
    (84544, 1, 1, True), (84576, 1, 1, False),                 # padding outputs, k < 12
    (1, 11, 84544, True), (1, 11, 84576, False),
    (1, 12, 219000, True), (1, 23, 220000, False), (1, 24, 220000, True),
    (1 << 20, 16, 16, True), (1 << 20, 15, 16, False),
    (1500, 1, 2500, True), (31, 1, 524288, True),              # little padding
    (1 << 20, 24, 1, True), (65535 * 32, 31, 1, True), (65535 * 32 + 1, 31, 1, False),
    (3, 300, 1 << 21, False), (3, 300, 1 << 20, True)])        # planes of 4 GiB
def test_padded_form(M, K, N, padded):
    assert padded_form(M, K, N) is padded
