"""The library's per-stream scratch (workspace) across HIP graph capture:
a call that needs scratch, run once eagerly, can then be captured; the
captured buffer outlives aq_release_workspace and a larger eager call, so
the graph keeps replaying the same bits; and a call that would need more
scratch than the stream holds is refused while the stream is capturing
(nothing is allocated under capture), with a message that says what to do."""
from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from alpacca_amd import _lib, synth
from alpacca_amd.qmatrix import DenseMatrix, QuantMatrix

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_captured_scratch_survives_release_and_growth():
    d = torch.device("cuda", 0)
    rows, cols, M = 2048, 2048, 16  # the exact-fp16 kernel: X pieces and split partials
    qm = QuantMatrix(synth.random_matrix_bytes("Q4_K", rows, cols, seed=1), "Q4_K", rows, cols)
    X = torch.from_numpy(synth.random_x(cols, seed=2, batch=M)).to(d)
    Y = torch.empty((M, rows), device=d)
    s = torch.cuda.Stream(d)
    h = s.cuda_stream
    lib = _lib.ensure_device()
    lib.aq_release_workspace(ctypes.c_void_p(h))  # start from no scratch on this stream
    with torch.cuda.stream(s):
        qm.matmul_t_device(X.data_ptr(), M, Y.data_ptr(), h)  # eager: sizes the scratch
    s.synchronize()
    want = Y.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        qm.matmul_t_device(X.data_ptr(), M, Y.data_ptr(), h)
    for _ in range(3):
        Y.zero_()
        with torch.cuda.stream(s):
            g.replay()
        s.synchronize()
        assert torch.equal(Y, want)
    # release, then a larger eager call on the same stream (new, larger scratch)
    _lib.check(lib.aq_release_workspace(ctypes.c_void_p(h)))
    X2 = torch.from_numpy(synth.random_x(cols, seed=3, batch=8 * M)).to(d)
    Y2 = torch.empty((8 * M, rows), device=d)
    with torch.cuda.stream(s):
        qm.matmul_t_device(X2.data_ptr(), 8 * M, Y2.data_ptr(), h)
    s.synchronize()
    for _ in range(3):
        Y.zero_()
        with torch.cuda.stream(s):
            g.replay()
        s.synchronize()
        assert torch.equal(Y, want)
    # the stream works eagerly as before
    with torch.cuda.stream(s):
        qm.matmul_t_device(X.data_ptr(), M, Y.data_ptr(), h)
    s.synchronize()
    assert torch.equal(Y, want)


def test_capture_refuses_scratch_growth():
    """Under capture the call fails on the host (no kernel is launched) and
    names the remedy; the stream is usable afterwards."""
    d = torch.device("cuda", 0)
    rows, cols = 2048, 2048
    qm = QuantMatrix(synth.random_matrix_bytes("Q4_K", rows, cols, seed=4), "Q4_K", rows, cols)
    s = torch.cuda.Stream(d)
    h = s.cuda_stream
    lib = _lib.ensure_device()
    lib.aq_release_workspace(ctypes.c_void_p(h))
    X = torch.from_numpy(synth.random_x(cols, seed=5, batch=64)).to(d)
    Y = torch.empty((64, rows), device=d)
    g = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError, match="eagerly before capture"):
        with torch.cuda.graph(g, stream=s):
            qm.matmul_t_device(X.data_ptr(), 64, Y.data_ptr(), h)
    with torch.cuda.stream(s):
        qm.matmul_t_device(X.data_ptr(), 64, Y.data_ptr(), h)
    s.synchronize()
    ref = qm.matmul_t(X.cpu().numpy())
    assert np.array_equal(Y.cpu().numpy(), ref)


@pytest.mark.parametrize("dtype", ["F16", "BF16", "F32"])
def test_dense_capture_without_scratch(dtype):
    """A dense matmul_t captured on a stream that holds no scratch runs without
    any for this many weight rows; the error of a call that does need some is
    not left behind.  Bar 1e-5 of max|Y| between the fp32 sums over 256 columns
    in two orders."""
    d = torch.device("cuda", 0)
    rows, cols, M = 4224, 256, 5
    W = DenseMatrix(synth.dense_values_bytes(dtype, rows, cols, seed=4), dtype, rows, cols)
    X = torch.from_numpy(synth.random_x(cols, seed=5, batch=M)).to(d)
    want = W.matmul_t(X.cpu().numpy())
    Y = torch.empty((M, rows), device=d)
    s = torch.cuda.Stream(d)
    h = s.cuda_stream
    _lib.check(_lib.ensure_device().aq_release_workspace(ctypes.c_void_p(h)))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        W.matmul_t_device(X.data_ptr(), M, Y.data_ptr(), h)
    for _ in range(3):
        Y.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            g.replay()
        s.synchronize()
        assert np.abs(Y.cpu().numpy() - want).max() < 1e-5 * np.abs(want).max()
    with pytest.raises(ValueError):  # its own message, not the refused scratch
        W.matmul_t_device(X.data_ptr(), -1, Y.data_ptr(), h)


@pytest.mark.parametrize("M", [5, 70])
@pytest.mark.parametrize("dtype", ["F16", "BF16", "F32"])
def test_dense_fp32_same_bits_without_scratch(dtype, M):
    """A dense matmul_t at fp32 gives the same bits whether the stream holds
    scratch for it or not, and for any M: captured without any, and in an
    eager call; rows that are corrected or formed again among them (the
    largest and smallest floats, an infinity, a NaN, a wide range)."""
    d = torch.device("cuda", 0)
    rows, cols = 4200, 352
    W = DenseMatrix(synth.dense_values_bytes(dtype, rows, cols, seed=7), dtype, rows, cols)
    Xh = synth.random_x(cols, seed=8, batch=M)
    Xh[0, 9] = 1e9
    Xh[1, 3], Xh[1, 300:303] = 1e5, 1e-6
    Xh[2, 5] = np.inf
    Xh[3, 6], Xh[3, 7] = 3.4e38, 1e-36
    if M > 20:
        Xh[20, 8] = np.nan
        Xh[33] = 0.0
        Xh[64] *= np.float32(1e-36)
    X = torch.from_numpy(Xh).to(d)
    Y = torch.empty((M, rows), device=d)
    s = torch.cuda.Stream(d)
    h = s.cuda_stream
    _lib.check(_lib.ensure_device().aq_release_workspace(ctypes.c_void_p(h)))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        W.matmul_t_device(X.data_ptr(), M, Y.data_ptr(), h, "fp32")
    got = []
    for _ in range(3):
        Y.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            g.replay()
        s.synchronize()
        got.append(Y.cpu().numpy().view(np.uint32))
    want = W.matmul_t(Xh, precision="fp32").view(np.uint32)
    assert all(np.array_equal(y, want) for y in got)
    cut = np.concatenate([W.matmul_t(Xh[a:b], precision="fp32") for a, b in ((0, 3), (3, M))])
    assert np.array_equal(cut.view(np.uint32), want)


def test_dense_scratch_is_bounded():
    """A dense matmul_t of many rows of X runs in slices: the stream's scratch for
    their pieces stays at 256 MiB (the pieces of all 24,000 rows: 590 MB), and a
    slice's end changes no bits at fp32."""
    d = torch.device("cuda", 0)
    rows, cols, M = 96, 4096, 24000
    W = DenseMatrix(synth.dense_values_bytes("F32", rows, cols, seed=9), "F32", rows, cols)
    X = torch.randn((M, cols), device=d)
    Y = torch.empty((M, rows), device=d)
    s = torch.cuda.Stream(d)
    h = s.cuda_stream
    W.matmul_t_device(X.data_ptr(), 2, Y.data_ptr(), None, "fp32")
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info(d)[0]
    W.matmul_t_device(X.data_ptr(), M, Y.data_ptr(), h, "fp32")
    s.synchronize()
    assert free - torch.cuda.mem_get_info(d)[0] <= (256 + 64) << 20
    got = Y.cpu().numpy()
    per = (1 << 28) // (6 * (cols + 32) + 80) // 256 * 256
    for r in (0, per - 3, 2 * per - 3, M - 6):
        want = W.matmul_t(X[r:r + 6].cpu().numpy(), precision="fp32")
        assert np.array_equal(got[r:r + 6].view(np.uint32), want.view(np.uint32)), r
    _lib.check(_lib.ensure_device().aq_release_workspace(ctypes.c_void_p(h)))


@pytest.mark.parametrize("dtype", ["F16", "F32", "Q4_K"])
def test_threads_share_a_stream(dtype):
    """Host threads that call on one stream (calls on host arrays all run on
    the null stream) share its scratch: each call's pieces of X and partials
    stay its own until its launches are queued, also while another thread's
    larger call outgrows the buffer.  Every result has the bits of the same
    call made alone."""
    rows, cols = 640, 2048
    cls = QuantMatrix if dtype == "Q4_K" else DenseMatrix
    data = (synth.random_matrix_bytes(dtype, rows, cols, seed=6) if dtype == "Q4_K" else
            synth.dense_values_bytes(dtype, rows, cols, seed=6))
    W = cls(data, dtype, rows, cols)
    # growing batches, of different sizes from thread to thread
    Xs = [[synth.random_x(cols, seed=100 * t + i, batch=17 + 40 * i + 11 * t) for i in range(6)]
          for t in range(4)]
    want = [[W.matmul_t(X) for X in row] for row in Xs]
    _lib.check(_lib.ensure_device().aq_release_workspace(None))
    start = threading.Barrier(len(Xs))
    bad = []

    def work(t):
        try:
            start.wait(30)
            for _ in range(5):
                for X, w in zip(Xs[t], want[t]):
                    if not np.array_equal(W.matmul_t(X).view(np.uint32), w.view(np.uint32)):
                        bad.append((t, X.shape[0]))
        except Exception as e:  # noqa: BLE001 (a thread's error is the test's)
            bad.append((t, repr(e)))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(len(Xs))]
    for th in threads:
        th.start()
    for th in threads:
        th.join(60)
    assert not bad, bad[:8]
    assert not any(th.is_alive() for th in threads)
