"""Decode attention against a float64 softmax at long contexts and wide score
ranges.  The attention weights are e^(s - max) computed as
2^((s - max) log2 e) on the hardware exp2, whose rounded product adds a
relative error of about |s - max| 2^-24 ln 2 to each weight; this pins the
resulting error of the outputs where the scores span tens of units (the
reference computes float32 np.exp, model.py:447-455; the bar is taken
against float64, the exact softmax)."""
from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest

from alpacca_amd import _lib
from tests.f64 import f64_of_bits

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _attention_f64(q, K, V, group):
    """q (n_head, hd), K/V (n_pos, n_kv, hd): the exact softmax attention."""
    n_head, hd = q.shape
    out = np.empty((n_head, hd))
    for h in range(n_head):
        kv = h // group
        s = K[:, kv, :].astype(np.float64) @ q[h].astype(np.float64) / np.sqrt(hd)
        w = np.exp(s - s.max())
        out[h] = (w @ V[:, kv, :].astype(np.float64)) / w.sum()
    return out


@pytest.mark.parametrize("n_ctx,pos,q_scale", [(2304, 2303, 1.0), (2304, 2175, 12.0),
                                               (4096, 4095, 25.0), (8192, 6000, 6.0)])
@pytest.mark.parametrize("hd", [64, 128])
def test_attention_vs_f64_wide_scores(n_ctx, pos, q_scale, hd):
    """Scores with standard deviations of about 1, 12, 25 and 6 units (q
    scaled; keys ~ N(0, 1)): outputs within 1e-5 of max|V| of the float64
    softmax, and the measured maximum printed for the record."""
    n_head, n_kv = 32, 8
    rng = np.random.default_rng(n_ctx + hd + int(q_scale))
    q = (rng.standard_normal((n_head, hd)) * q_scale).astype(np.float32)
    K = rng.standard_normal((n_ctx, n_kv, hd)).astype(np.float32)
    V = rng.standard_normal((n_ctx, n_kv, hd)).astype(np.float32)
    d = torch.device("cuda", 0)
    kc = torch.from_numpy(np.ascontiguousarray(K.transpose(1, 0, 2))).to(d)
    vc = torch.from_numpy(np.ascontiguousarray(V.transpose(1, 0, 2))).to(d)
    qd = torch.from_numpy(q.reshape(-1)).to(d)
    out = torch.empty(n_head * hd, device=d)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    lib = _lib.ensure_device()
    _lib.check(lib.aq_attention(P(qd), P(kc), P(vc), n_head, n_kv, hd, n_ctx, None, pos,
                                P(out), None))
    got = out.cpu().numpy().reshape(n_head, hd).astype(np.float64)
    want = _attention_f64(q, K[:pos + 1], V[:pos + 1], n_head // n_kv)
    err = np.abs(got - want).max() / np.abs(V).max()
    s_span = float(np.abs(q).max() * np.sqrt(hd))
    print(f"attention n_ctx={n_ctx} pos={pos} hd={hd} q_scale={q_scale}: "
          f"max|out - f64| / max|V| = {err:.2e}", flush=True)
    assert err < 1e-5, (err, s_span)


@pytest.mark.parametrize("hd,T,vscale,qscale", [(64, 130, 1e25, 1.0), (128, 1100, 1e-25, 6.0),
                                                (64, 65, 1.0, 1e-20)])
def test_attention_batch_three_pieces_vs_f64(hd, T, vscale, qscale):
    """The batched attention cuts q, K, V and the weights into three bf16
    pieces (24 bits, fp32's exponent range, no scaling): against float64 at
    magnitudes far from one, and the same bits when the tokens come in several
    calls (which at head_dim 128 run four-wave workgroups, the 1100 tokens
    eight-wave ones).  Bar 1e-5 max|V|, as for the decode form above."""
    n_head, n_kv, pos0 = 32, 8, 70
    n_ctx = pos0 + T
    rng = np.random.default_rng(hd + T)
    q = (rng.standard_normal((T, n_head * hd)) * qscale).astype(np.float32)
    K = rng.standard_normal((n_kv, n_ctx, hd)).astype(np.float32)
    V = (rng.standard_normal((n_kv, n_ctx, hd)) * vscale).astype(np.float32)
    kc, vc, qd = (torch.from_numpy(a).to("cuda") for a in (K, V, q))
    lib = _lib.ensure_device()
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731

    def run(cuts):
        out = torch.empty((T, n_head * hd), device="cuda")
        for a, b in zip(cuts, cuts[1:]):
            _lib.check(lib.aq_attention_batch(p(qd[a:b]), p(kc), p(vc), b - a, n_head, n_kv, hd,
                                              n_ctx, None, pos0 + a, p(out[a:b]), None))
        return out.cpu().numpy()

    whole = run([0, T])
    cut = sorted({0, 3, T // 3, T // 2 + 1, T})
    assert np.array_equal(whole.view(np.uint32), run(cut).view(np.uint32))
    for h in (0, 5, 31):
        kv = h // (n_head // n_kv)
        s = q[:, h * hd:(h + 1) * hd].astype(np.float64) @ K[kv].astype(np.float64).T / math.sqrt(hd)
        s[np.arange(n_ctx)[None, :] > pos0 + np.arange(T)[:, None]] = -np.inf
        w = np.exp(s - s.max(axis=1, keepdims=True))
        want = (w / w.sum(axis=1, keepdims=True)) @ V[kv].astype(np.float64)
        err = np.abs(whole[:, h * hd:(h + 1) * hd] - want).max() / np.abs(V).max()
        assert err < 1e-5, (h, err)


@pytest.mark.parametrize("hd,T", [(64, 100), (128, 70), (64, 2)])
def test_attention_batch_nonfinite(hd, T):
    """Infinities and NaNs in q, K and V, and finite values that round to a
    bf16 infinity, give what the float32 softmax over the positions a row sees
    gives (a score of -inf is a weight of zero), and leave the rows that do not
    see them alone.  Bar 1e-5 max|V| of each dimension, as above."""
    n_head, n_kv, pos0 = 8, 2, 9
    n_ctx = pos0 + T
    rng = np.random.default_rng(hd * T)
    q = rng.standard_normal((T, n_head, hd)).astype(np.float32)
    K = rng.standard_normal((n_kv, n_ctx, hd)).astype(np.float32)
    V = rng.standard_normal((n_kv, n_ctx, hd)).astype(np.float32)
    q[..., 0], q[..., 1] = 1.0, np.float32(2.0 ** -126)
    K[0, 2, 0] = -np.inf                      # no weight
    K[0, 4, 1] = np.finfo(np.float32).max     # adds 4 to the score
    V[0, 5, 3] = np.inf                       # that dimension infinite
    V[1, 6, 7] = np.finfo(np.float32).max     # finite products
    if T > 60:
        V[1, pos0 + 40, 2] = np.nan           # seen from token 40 on
        q[50, 3, 5] = np.nan
        q[20, 1, 2] = np.inf
    qd, kc, vc = (torch.from_numpy(a).to("cuda") for a in (q, K, V))
    out = torch.empty((T, n_head, hd), device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    _lib.check(_lib.ensure_device().aq_attention_batch(p(qd), p(kc), p(vc), T, n_head, n_kv, hd,
                                                       n_ctx, None, pos0, p(out), None))
    got = out.cpu().numpy()
    with np.errstate(all="ignore"):
        for t in range(T):
            n = pos0 + t + 1
            for h in range(n_head):
                kv = h // (n_head // n_kv)
                s = (K[kv, :n].astype(np.float64) @ q[t, h].astype(np.float64)) / math.sqrt(hd)
                w = np.exp(s - s.max())
                want = (w / w.sum()) @ V[kv, :n].astype(np.float64)
                fin = np.isfinite(want)
                g = got[t, h]
                assert np.array_equal(np.isnan(want), np.isnan(g)), (t, h)
                assert np.array_equal(want[~fin], g[~fin], equal_nan=True), (t, h)
                bar = np.abs(V[kv, :n].astype(np.float64)).max(axis=0)
                assert (np.abs(g - want)[fin] <= 1e-5 * bar[fin]).all(), (t, h)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("what", ["v", "v_late", "k", "q", "q_some"])
def test_attention_batch_tiny_values(hd, what):
    """Values whose 24 bits three bf16 pieces do not hold (below 2^-110): V of
    that size (v_late: in one dimension, from position 70 on), and K or q of that
    size against q or K so large that their scores matter (q_some: in every fifth
    row, one dimension).  Bar 1e-5 max|V| of each dimension against float64, as
    above, and the same bits when the tokens come in several calls."""
    n_head, n_kv, T = 8, 2, 100
    rng = np.random.default_rng(hd)
    q = rng.standard_normal((T, n_head, hd)).astype(np.float32)
    K = rng.standard_normal((n_kv, T, hd)).astype(np.float32)
    V = rng.standard_normal((n_kv, T, hd)).astype(np.float32)
    if what == "v":
        V = np.ldexp(V, -118)
    elif what == "v_late":
        V[:, :70, 3] = 0.0
        V[:, 70:, 3] = np.ldexp(V[:, 70:, 3], -118)
    elif what == "q_some":
        q[::5, :, 1] = np.ldexp(q[::5, :, 1], -118)
        q[1::5, :, 1] = q[2::5, :, 1] = q[3::5, :, 1] = q[4::5, :, 1] = 0.0
        K[:, ::2, 1] = np.ldexp(np.abs(K[:, ::2, 1]), 119)
    else:
        q = np.ldexp(q, -116 if what == "q" else 115)
        K = np.ldexp(K, 118 if what == "q" else -117)
    qd, kc, vc = (torch.from_numpy(a).to("cuda") for a in (q, K, V))
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    lib = _lib.ensure_device()

    def run(cuts):
        out = torch.empty((T, n_head, hd), device="cuda")
        for a, b in zip(cuts, cuts[1:]):
            _lib.check(lib.aq_attention_batch(p(qd[a:b]), p(kc), p(vc), b - a, n_head, n_kv, hd,
                                              T, None, a, p(out[a:b]), None))
        return out.cpu().numpy()

    got = run([0, T])
    assert np.array_equal(got.view(np.uint32), run([0, 3, 37, 72, T]).view(np.uint32))
    got, q, K, V = (f64_of_bits(a) for a in (got, q, K, V))
    for t in range(T):
        for h in range(n_head):
            kv = h // (n_head // n_kv)
            s = (K[kv, :t + 1] @ q[t, h]) / math.sqrt(hd)
            w = np.exp(s - s.max())
            v = V[kv, :t + 1]
            want = (w / w.sum()) @ v
            bar = 1e-5 * np.abs(v).max(axis=0)
            err = np.abs(got[t, h] - want)
            assert (err <= bar).all(), (t, h, (err - bar).max())
