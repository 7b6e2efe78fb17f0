"""The matmul gate where a dimension is no multiple of 32 (planes padded with
zero digits, matrix cores): both parties' shares equal the launch-per-step
form's on the VALU kernel for the same dealer material, on reused buffers and
at every split of the opens (1, 4 and 16 k per lane, tiles)."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
from gpu_util import dev, host, say, u64
from suf_amd import layer, matmul_gate, native

pytestmark = pytest.mark.gpu

STATE = ol.mt64_bytes(3, ol.PRG_STATE_BYTES).tobytes()


@pytest.mark.parametrize("M,K,N,f", [
    (1, 1, 1, 12), (1, 16, 33, 8), (31, 33, 65, 13), (32, 100, 64, 12), (33, 64, 32, 12),
    (77, 300, 1000, 12), (3, 129, 2000, 12), (40, 1023, 2050, 12), (5, 1023, 2100, 12),
    (250, 160, 31, 12), (64, 64, 64, 12), (32, 96, 480, 12), (31, 32, 33, 12)])
def test_ragged_gate_equals_step_form(M, K, N, f):
    say("matmul gate ragged %dx%dx%d f=%d" % (M, K, N, f))
    native.call("sufhip_init", 0)
    rng = np.random.default_rng(M + K + N)
    gate = matmul_gate.BeaverMatmulTrunc(M, K, N, STATE, f, seed=7)
    step = matmul_gate.BeaverMatmulTrunc(M, K, N, STATE, f, seed=7, use_mfma=False)
    assert gate.fused and not step.fused
    for turn in range(2):
        x = (rng.normal(0, 1, M * K) * (1 << f)).astype(np.int64)
        w = (rng.normal(0, 0.05, K * N) * (1 << f)).astype(np.int64)
        x0 = rng.integers(0, 1 << 64, M * K, dtype=np.uint64)
        w0 = rng.integers(0, 1 << 64, K * N, dtype=np.uint64)
        X = (dev(x0), dev(x.view(np.uint64) - x0))
        W = (dev(w0), dev(w.view(np.uint64) - w0))
        got = [torch.full((M * N + 3,), -7, dtype=torch.int64, device="cuda") for _ in range(2)]
        ref = [torch.empty(M * N, dtype=torch.int64, device="cuda") for _ in range(2)]
        gate.eval2(X, W, got)
        step.eval2(X, W, ref)
        for p in (0, 1):
            assert np.array_equal(u64(got[p])[:M * N], u64(ref[p])), (turn, p)
            assert (host(got[p])[M * N:] == -7).all()
        if M * K * N <= 1 << 22:
            z = x.reshape(M, K).astype(object) @ w.reshape(K, N).astype(object)
            want = np.array([int(v) >> f for v in z.ravel()], dtype=np.int64)
            assert np.array_equal(host(ref[0] + ref[1]), want)


@pytest.mark.parametrize("batches,rows,cols,k_is_col", [
    (1, 1, 1, 1), (2, 33, 47, 1), (3, 31, 70, 0), (1, 96, 100, 0)])
def test_padded_planes(batches, rows, cols, k_is_col):
    """A padded split writes every byte of its planes: those of the source
    padded with zeros, with and without + a0."""
    say("kb_split padded %d %dx%d kc=%d" % (batches, rows, cols, k_is_col))
    native.call("sufhip_init", 0)
    rng = np.random.default_rng(rows + cols)
    rp, cp = (-(-v // 32) * 32 for v in (rows, cols))
    src, a0 = (rng.integers(0, 1 << 64, (batches, rows, cols), dtype=np.uint64) for _ in range(2))

    def padded(a):
        big = np.zeros((batches, rp, cp), dtype=np.uint64)
        big[:, :rows, :cols] = a
        return dev(big)

    want, want_x, got, got_x = (layer.kb_planes(batches, rp, cp).fill_(-1) for _ in range(4))
    layer.kb_split([(padded(src), want, batches, rp, cp, k_is_col),
                    (padded(src + a0), want_x, batches, rp, cp, k_is_col)])
    layer.kb_split([(dev(src), got, batches, rows, cols, k_is_col, got_x, dev(a0))], pad=True)
    assert torch.equal(got, want) and torch.equal(got_x, want_x)


def test_bad_extents_are_refused():
    say("kb_split bad extents")
    planes = layer.kb_planes(1, 64, 64)
    src = torch.zeros(64 * 64, dtype=torch.int64, device="cuda")
    job = (native.KbOpenJob * 1)()
    job[0].a[0] = job[0].a[1] = src.data_ptr()
    job[0].planes, job[0].batches, job[0].rows, job[0].cols = planes.data_ptr(), 1, 64, 64
    for vr, vc, stride in ((65, 64, 0), (64, 0, 0), (0, 5, 0), (-1, 3, 0), (33, 33, 1)):
        job[0].valid_rows, job[0].valid_cols, job[0].a_stride[2] = vr, vc, stride
        with pytest.raises(native.SufHipError):
            native.call("sufhip_kb_open_split_batch", job, 1, None)


@pytest.mark.parametrize("M,K,N", [(1 << 18, 1, 1), (2, 11, 90000), (300000, 16, 3)])
def test_thin_gate_keeps_the_step_form(M, K, N):
    """Products that padding would blow up: the shares of the launch-per-step
    form, and no more memory than it takes."""
    say("matmul gate thin %dx%dx%d" % (M, K, N))
    native.call("sufhip_init", 0)
    rng = np.random.default_rng(M)
    x, w = (rng.integers(-(1 << 14), 1 << 14, s) for s in (M * K, K * N))
    x0, w0 = (rng.integers(0, 1 << 64, s, dtype=np.uint64) for s in (M * K, K * N))
    X = (dev(x0), dev(x.view(np.uint64) - x0))
    W = (dev(w0), dev(w.view(np.uint64) - w0))
    held, outs = [], []
    for use_mfma in (True, False):
        before = torch.cuda.memory_allocated()
        gate = matmul_gate.BeaverMatmulTrunc(M, K, N, STATE, 12, seed=7, use_mfma=use_mfma)
        held.append(torch.cuda.memory_allocated() - before)
        out = [torch.empty(M * N, dtype=torch.int64, device="cuda") for _ in range(2)]
        gate.eval2(X, W, out)
        outs.append([u64(o) for o in out])
        del gate
    assert held[0] <= held[1]
    for p in (0, 1):
        assert np.array_equal(outs[0][p], outs[1][p])
    z = x.reshape(M, K) @ w.reshape(K, N)
    assert np.array_equal((outs[0][0] + outs[0][1]).view(np.int64), z.ravel() >> 12)
