"""Dense F32 / F16 / BF16 matrices (DenseMatrix): the reference keeps such
weights as float32 arrays and multiplies with NumPy (model.py:269-281,
quants.py:517-523, tensor.py:82-113).

The oracle's decode is pinned by known bit patterns (IEEE half and bfloat16
encodings of exact values, subnormals, signed zero, infinity); the device
path by the f64 product over the same decoded values (2e-5 / 1e-2
normalized), exact row gathers, and greedy tokens of a
model with dense matrices equal to the oracle's.
"""
from __future__ import annotations

import numpy as np
import pytest

from alpacca_amd import gguf, synth
from alpacca_amd.qmatrix import DENSE_DTYPES, DenseMatrix, QuantMatrix
from oracle.qmatrix_ref import DenseRef, normalized_error
from oracle.quants_ref import dense_decode
from tests.f64 import f64_of_bits

DENSE = ("F32", "F16", "BF16")


def test_dense_decode_known_answers():
    f16 = np.array([0x3C00, 0xC000, 0x0001, 0x7BFF, 0x8000, 0x7C00, 0x3555], "<u2")
    got = dense_decode(f16.view(np.uint8).tobytes(), f16.size, "F16")
    want = [1.0, -2.0, 2.0 ** -24, 65504.0, -0.0, np.inf, 1365 / 4096]
    assert np.array_equal(got, np.array(want, np.float32))
    assert np.signbit(got[4])
    bf = np.array([0x3F80, 0xC040, 0x0001, 0x7F7F, 0x3EAB], "<u2")
    got = dense_decode(bf.view(np.uint8).tobytes(), bf.size, "BF16")
    want = np.array([0x3F800000, 0xC0400000, 0x00010000, 0x7F7F0000, 0x3EAB0000],
                    np.uint32).view(np.float32)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert got[0] == 1.0 and got[1] == -3.0
    f32 = np.array([1.5, -0.0, 3.4e38, 1e-45], np.float32)
    assert np.array_equal(dense_decode(f32.tobytes(), 4, "F32").view(np.uint32), f32.view(np.uint32))
    with pytest.raises(ValueError):
        dense_decode(b"\0" * 6, 4, "F16")


def test_synth_bf16_rounds_to_nearest_even():
    v = synth.dense_values_bytes("BF16", 4, 64, seed=3).view("<u2")
    ref = np.random.default_rng(3).standard_normal(256).astype(np.float32) * np.float32(0.02)
    back = (v.astype(np.uint32) << 16).view(np.float32)
    # |error| at most half a bf16 ulp (2^-8 relative)
    assert np.all(np.abs(back - ref) <= np.abs(ref) * 2.0 ** -8)


@pytest.mark.parametrize("dtype", DENSE)
def test_dense_matrix_rejects_bad_arguments(dtype):
    w = DENSE_DTYPES[dtype]
    with pytest.raises(ValueError, match="multiple of 32"):
        DenseMatrix(b"\0" * (4 * 48 * w), dtype, 4, 48)
    with pytest.raises(ValueError, match="bytes, expected"):
        DenseMatrix(b"\0" * (4 * 64 * w - 2), dtype, 4, 64)
    with pytest.raises(ValueError, match="not Q4_K"):
        DenseMatrix(b"\0" * 64, "Q4_K", 1, 32)
    with pytest.raises(ValueError):  # QuantMatrix keeps the reference's rejection
        QuantMatrix(b"\0" * (4 * 64 * w), dtype, 4, 64)


def test_gguf_keeps_dense_matrices(tmp_path):
    from alpacca_amd.model import Tensor, synthetic_llama_1b
    hp, tensors = synthetic_llama_1b(seed=1, n_layer=1, n_embd=256, n_head=2, n_kv=1,
                                     n_ff=512, n_vocab=96, n_ctx_train=256)
    tensors["blk.0.attn_q.weight"] = Tensor("F16", (256, 256), synth.dense_values_bytes("F16", 256, 256, 1))
    tensors["blk.0.ffn_up.weight"] = Tensor("BF16", (512, 256), synth.dense_values_bytes("BF16", 512, 256, 2))
    f32 = np.random.default_rng(4).standard_normal((96, 256)).astype(np.float32)
    tensors["output.weight"] = Tensor("F32", (96, 256), f32)
    p = tmp_path / "d.gguf"
    gguf.write_model(p, hp, tensors)
    with gguf.GGUFReader(p) as g:
        assert g.tensors["blk.0.attn_q.weight"].dtype == "F16"
        back = gguf.read_tensors(g)
        assert back["blk.0.attn_q.weight"].dtype == "F16"
        assert bytes(back["blk.0.attn_q.weight"].data) == tensors["blk.0.attn_q.weight"].data.tobytes()
        assert bytes(back["blk.0.ffn_up.weight"].data) == tensors["blk.0.ffn_up.weight"].data.tobytes()
        assert back["output.weight"].dtype == "F32" and back["output.weight"].shape == (96, 256)
        assert bytes(back["output.weight"].data) == f32.tobytes()
        assert back["blk.0.attn_norm.weight"].data.dtype == np.float32
        del back


# ---------------------------------------------------------------- GPU parity --

SHAPES = [(64, 32), (300, 512), (2048, 2048), (4096, 4096), (96, 14336)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DENSE)
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_dense_matvec_vs_f64(dtype, rows, cols):
    data = synth.dense_values_bytes(dtype, rows, cols, seed=rows + cols, std=1.0)
    W = DenseMatrix(data, dtype, rows, cols)
    ref = DenseRef(data, dtype, rows, cols)
    x = synth.random_x(cols, seed=cols)
    y = W.matvec(x)
    assert normalized_error(y, ref.matvec_f64(x), ref.row_norms(), x) < 2e-5
    assert np.array_equal(W.rows_at([0, rows - 1, rows // 2]), ref.rows_at([0, rows - 1, rows // 2]))
    with pytest.raises(IndexError):
        W.row(rows)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DENSE)
@pytest.mark.parametrize("M", [5, 70, 512])
def test_dense_matmul_t_vs_f64(dtype, M):
    rows, cols = 1000, 2048
    data = synth.dense_values_bytes(dtype, rows, cols, seed=M, std=1.0)
    W = DenseMatrix(data, dtype, rows, cols)
    ref = DenseRef(data, dtype, rows, cols)
    X = synth.random_x(cols, seed=M, batch=M)
    want = ref.matmul_t_f64(X)
    norms = ref.row_norms()
    for prec, tol in (("fp32", 2e-5), ("bf16", 1e-2)):
        Y = W.matmul_t(X, precision=prec)
        err = max(normalized_error(Y[i], want[i], norms, X[i]) for i in range(M))
        assert err < tol, (prec, err)


@pytest.mark.gpu
def test_dense_rejected_by_multi_launches():
    import torch
    from alpacca_amd.qmatrix import matvec_multi_device
    W = DenseMatrix(synth.dense_values_bytes("F16", 64, 64), "F16", 64, 64)
    x = torch.zeros(64, device="cuda")
    y = torch.zeros(64, device="cuda")
    with pytest.raises(ValueError, match="aq_matvec"):
        matvec_multi_device([W], x.data_ptr(), [y.data_ptr()])


@pytest.mark.gpu
@pytest.mark.parametrize("dense", ["F16", "BF16", "F32"])
def test_model_with_dense_matrices_greedy(tmp_path, dense):
    """Some matrices dense (the reference's F16 / F32 GGUFs), the rest
    quantized: greedy tokens equal the oracle's, also through a GGUF file."""
    from alpacca_amd.model import Model, Tensor, synthetic_llama_1b
    from oracle.model_ref import RefModel
    hp, tensors = synthetic_llama_1b(seed=7, n_layer=2, n_embd=256, n_head=4, n_kv=2,
                                     n_ff=512, n_vocab=700, n_ctx_train=512)
    for i, name in enumerate(["blk.0.attn_q.weight", "blk.0.ffn_down.weight",
                              "blk.1.attn_v.weight", "blk.1.ffn_gate.weight",
                              "token_embd.weight"]):
        rows, cols = tensors[name].shape
        tensors[name] = Tensor(dense, (rows, cols),
                               synth.dense_values_bytes(dense, rows, cols, seed=50 + i))
    prompt = list(np.random.default_rng(11).integers(0, hp.n_vocab, 40))
    m = Model(hp, tensors)
    assert not m.fused
    toks = m.generate_greedy(prompt, 12)
    ref_toks, margins = RefModel(hp, tensors).greedy(prompt, 12)
    assert toks == ref_toks, (toks, ref_toks, min(margins))
    p = tmp_path / "m.gguf"
    gguf.write_model(p, hp, tensors)
    assert gguf.load_model(p).generate_greedy(prompt, 12) == toks


# Tile kernel (aq_matmul_dn.hip): sizes that end inside a tile of each shape and
# inside a 64-column stage.  Bar: 2^-22 of ||W_r|| ||x_m|| from the pieces and
# as much again for the fp32 sums.
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DENSE)
@pytest.mark.parametrize("M,rows,cols", [(2, 1, 32), (33, 130, 96), (130, 300, 1056)])
def test_dense_tile_shapes_vs_f64(dtype, M, rows, cols, monkeypatch):
    data = synth.dense_values_bytes(dtype, rows, cols, seed=rows, std=1.0)
    W = DenseMatrix(data, dtype, rows, cols)
    ref = DenseRef(data, dtype, rows, cols)
    X = synth.random_x(cols, seed=M, batch=M)
    X[0] *= 1e30
    X[1] *= 1e-30
    want, norms = ref.matmul_t_f64(X), ref.row_norms()
    first = None
    for shape in range(4):
        monkeypatch.setenv("AQ_MATMUL_TILE", str(shape))
        for prec in ("fp32", "auto"):
            Y = W.matmul_t(X, precision=prec)
            err = max(normalized_error(Y[i], want[i], norms, X[i]) for i in range(M))
            assert err < 2.0 ** -21, (shape, prec, err)
            if prec == "fp32":
                first = Y if first is None else first
                assert np.array_equal(Y.view(np.uint32), first.view(np.uint32)), shape
    assert np.array_equal(W.matmul_t(X[:1], precision="fp32").view(np.uint32),
                          first[:1].view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DENSE)
def test_dense_matmul_t_nonfinite(dtype):
    """Infinities and NaNs in X and in the weights give what float32 products
    give, and leave the other rows and columns alone.  Bar: the rounding of a sum
    of cols float32 products, cols 2^-24 of the sum of |x| |w|, for each output
    (weights of zero against the largest x leave the rest of its row's sum)."""
    M, rows, cols = 40, 64, 128
    w = np.random.default_rng(1).standard_normal((rows, cols)).astype(np.float32)
    w[20:40, 8] = 0.0
    if dtype == "BF16":
        w = (w.view(np.uint32) & 0xFFFF0000).view(np.float32)
    X = synth.random_x(cols, seed=2, batch=M)
    X[3, 5], X[4, 6], X[5, 7] = np.inf, -np.inf, np.nan
    X[6, 8] = 3.4e38
    for bad_w in (False, True):
        if bad_w:
            w[7, 9], w[8, 10] = np.inf, np.nan
        data = (w.astype(np.float16).view(np.uint8) if dtype == "F16" else
                (w.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8) if dtype == "BF16"
                else w.view(np.uint8)).reshape(-1)
        wv = w.astype(np.float16).astype(np.float64) if dtype == "F16" else w.astype(np.float64)
        with np.errstate(invalid="ignore", over="ignore"):
            want = (X.astype(np.float64) @ wv.T).astype(np.float32)
        Y = DenseMatrix(data, dtype, rows, cols).matmul_t(X)
        fin = np.isfinite(want)
        assert np.array_equal(np.isnan(want), np.isnan(Y))
        assert np.array_equal(want[~fin & ~np.isnan(want)], Y[~fin & ~np.isnan(want)])
        with np.errstate(invalid="ignore"):
            bar = (np.abs(X).astype(np.float64) @ np.abs(wv).T) * cols * 2.0 ** -24
        assert (np.abs(Y[fin].astype(np.float64) - want[fin]) <= bar[fin]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("bad_w", [False, True])
@pytest.mark.parametrize("dtype", DENSE)
def test_dense_matmul_t_nonfinite_split(dtype, bad_w):
    """Infinities and NaNs with K split over workgroups (few weight rows, 4096
    columns): of the tile kernel, where every split forms its own columns of a
    row again, and, with an infinite weight, of the fp32 kernel.  Bar as above."""
    M, rows, cols = 6, 40, 4096
    rng = np.random.default_rng(5)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    w = (w.view(np.uint32) & 0xFFFF0000).view(np.float32)
    if bad_w:
        w[7, 3000] = np.inf
    data = (w.astype(np.float16).view(np.uint8) if dtype == "F16" else
            (w.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8) if dtype == "BF16"
            else w.view(np.uint8)).reshape(-1)
    wv = w.astype(np.float16).astype(np.float64) if dtype == "F16" else w.astype(np.float64)
    X = synth.random_x(cols, seed=6, batch=M)
    X[1, 70], X[2, 4000] = np.inf, np.nan
    X[3, 100], X[3, 3900] = np.inf, -np.inf
    X[4, 5], X[4, 2500] = np.inf, 1e-36
    with np.errstate(invalid="ignore"):
        want = X.astype(np.float64) @ wv.T
        bar = (np.abs(X).astype(np.float64) @ np.abs(wv).T) * cols * 2.0 ** -24
    W = DenseMatrix(data, dtype, rows, cols)
    for prec in ("auto", "fp32"):
        Y = W.matmul_t(X, precision=prec).astype(np.float64)
        fin = np.isfinite(want)
        assert np.array_equal(want[~fin], Y[~fin], equal_nan=True), prec
        assert (np.abs(Y[fin] - want[fin]) <= bar[fin]).all(), prec


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DENSE)
@pytest.mark.parametrize("cols", [64, 2080])
def test_dense_matmul_t_wide_range_rows(dtype, cols, monkeypatch):
    """Rows of X whose elements lie far apart: what is left of a sum when the
    weight of the largest element is zero has the accuracy of float32 products.
    Bar: cols 2^-24 of the sum of |x| |w|, for each output.  F16 keeps 22 bits of
    elements down to 2^-28 of the row's largest in its two pieces (row 0), adds
    what they lack of up to eight smaller ones (rows 1 - 3: one, eight, and nine
    of them, the last is formed again in float32 as rows 17, 18, 35 are); with
    a split of K (auto, 2080 columns) and without, the same bits in every tile
    shape at fp32."""
    M, rows = 37, 150
    rng = np.random.default_rng(cols)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    w = (w.view(np.uint32) & 0xFFFF0000).view(np.float32)
    w[:, 7] = 0.0
    X = synth.random_x(cols, seed=cols, batch=M)
    X[0] = rng.uniform(0.5, 1.0, cols) * rng.choice([-1.0, 1.0], cols)
    X[0, 7] = 2.0 ** 27
    for i, n in ((1, 1), (2, 8), (3, 9)):
        # small values against weights of 2^13, so that the sum shows them
        X[i] = rng.uniform(0.5, 1.0, cols) * rng.choice([-1.0, 1.0], cols)
        X[i, 7], X[i, 8:] = 2.0 ** 27, 0.0
        X[i, cols - 3 * n::3] = rng.uniform(1.0, 2.0, n) * 2.0 ** -21
    w[::2, cols - 40:] *= np.float32(2.0 ** 13)
    X[17, 7] = 1e8
    X[18] = 1.0
    X[18, 7] = 1e20
    X[35] = np.ldexp(X[35], rng.integers(-90, 90, cols))
    X[36] = 0.0
    X[36, 7], X[36, 9] = 3e38, 1e-30
    data = (w.astype(np.float16).view(np.uint8) if dtype == "F16" else
            (w.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8) if dtype == "BF16"
            else w.view(np.uint8)).reshape(-1)
    wv = w.astype(np.float16).astype(np.float64) if dtype == "F16" else w.astype(np.float64)
    want = X.astype(np.float64) @ wv.T
    bar = (np.abs(X).astype(np.float64) @ np.abs(wv).T) * cols * 2.0 ** -24
    W = DenseMatrix(data, dtype, rows, cols)
    first = None
    for shape in (None, 0, 1, 2, 3):
        if shape is not None:
            monkeypatch.setenv("AQ_MATMUL_TILE", str(shape))
        for prec in ("auto", "fp32"):
            Y = W.matmul_t(X, precision=prec)
            bad = np.argwhere(np.abs(Y.astype(np.float64) - want) > bar)
            assert not len(bad), (shape, prec, bad[:5])
            if prec == "fp32":
                first = Y if first is None else first
                assert np.array_equal(Y.view(np.uint32), first.view(np.uint32)), shape


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DENSE)
@pytest.mark.parametrize("w_exp", [0, -118])
def test_dense_matmul_t_tiny_values(dtype, w_exp):
    """Values of X down to float32's subnormals, and F32 / BF16 weights below
    2^-110 (where three bf16 pieces stop holding 24 bits), give what float32
    products give.  Bar: cols 2^-24 of the sum of |x| |w| and cols of float32's
    smallest subnormals, for each output."""
    M, rows, cols = 20, 140, 96
    rng = np.random.default_rng(3)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    if w_exp and dtype != "F16":
        w[::3] = np.ldexp(w[::3], w_exp)
        w[1, 5] = np.ldexp(np.float32(1.2345678), w_exp)
    w = (w.view(np.uint32) & 0xFFFF0000).view(np.float32) if dtype == "BF16" else w
    data = (w.astype(np.float16).view(np.uint8) if dtype == "F16" else
            (w.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8) if dtype == "BF16"
            else w.view(np.uint8)).reshape(-1)
    wv = w.astype(np.float16).astype(np.float64) if dtype == "F16" else w.astype(np.float64)
    X = synth.random_x(cols, seed=4, batch=M)
    for i, e in enumerate((-105, -112, -116, -120, -124, -128, -140, 100, 118)):
        X[i] = np.ldexp(X[i], e)
    X[10, 3] = np.ldexp(np.float32(1.2345678), -115)
    X[11] = np.ldexp(X[11], rng.integers(-125, 100, cols))
    x64 = f64_of_bits(X)
    wv = wv if dtype == "F16" else f64_of_bits(w)
    want = x64 @ wv.T
    bar = (np.abs(x64) @ np.abs(wv).T) * cols * 2.0 ** -24 + cols * 2.0 ** -149
    W = DenseMatrix(data, dtype, rows, cols)
    for prec in ("auto", "fp32"):
        Y = f64_of_bits(W.matmul_t(X, precision=prec))
        bad = np.argwhere(np.abs(Y - want) > bar)
        assert not len(bad), (prec, bad[:5], len(bad))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DENSE)
def test_dense_matmul_t_one_wide_row(dtype):
    """One row of X wider than the matvec kernel stages in LDS (K = 53,248 is a
    405B-class ffn_down) runs as well."""
    rows, cols = 3, 53248
    data = synth.dense_values_bytes(dtype, rows, cols, seed=1, std=1.0)
    W, ref = DenseMatrix(data, dtype, rows, cols), DenseRef(data, dtype, rows, cols)
    X = synth.random_x(cols, seed=2, batch=1)
    err = normalized_error(W.matmul_t(X)[0], ref.matmul_t_f64(X)[0], ref.row_norms(), X[0])
    assert err < 2.0 ** -21, err
