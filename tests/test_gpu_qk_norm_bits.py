"""RMSNorm of Q and K rows to the last bit: 1 / sqrt as a correctly rounded
square root and division, not the hardware's reciprocal square root (1 ulp).
Inputs are small whole numbers, so a row's sum of squares is exact in any order
and numpy's f32 arithmetic gives the kernel's value."""
import ctypes
import math

import numpy as np
import pytest

import iris_testlib as tl

pytestmark = pytest.mark.gpu
EPS = np.float32(1e-6)


@pytest.fixture(scope="module")
def lib():
    return tl.hip()


def norm_bits(x, w, cos, sin):
    """bf16 bits of x / sqrt(mean(x^2) + eps) * w in f32, its pairs rotated with
    one fused product each (float64 holds a product of two f32 exactly);
    x [rows][heads][128] whole numbers, w [rows][128], cos and sin [rows][64]"""
    x = x.astype(np.float32)
    ss = (x * x).sum(-1, dtype=np.float32, keepdims=True)
    inv = np.float32(1) / np.sqrt(ss / np.float32(128) + EPS)
    n = x * inv * w[:, None]
    x0, x1, c, s = n[..., 0::2], n[..., 1::2], cos[:, None], sin[:, None]
    r0 = x0.astype(np.float64) * c - (x1 * s).astype(np.float64)
    r1 = x0.astype(np.float64) * s + (x1 * c).astype(np.float64)
    return tl.to_bf16(np.stack([r0, r1], -1).astype(np.float32).reshape(x.shape))


def tables(rng, S, rope):
    ang = rng.uniform(-3, 3, (S, 64))
    return (np.cos(ang), np.sin(ang)) if rope else (np.ones((S, 64)), np.zeros((S, 64)))


@pytest.mark.parametrize("S,H,split,rope", [(1024, 8, 1024, False), (257, 3, 100, False), (1024, 8, 300, True),
                                            (130, 5, 60, True), (70, 30, 0, True), (3, 1, 2, False)])
def test_prepared_rows(lib, S, H, split, rope):
    """Whole and part-empty rounds of 8 heads. 2 x 1 M values: a last-bit error of 1 / sqrt in a fifth of the rows moves several over a bf16 rounding line"""
    rng = np.random.default_rng(S)
    h, S_pad = H * 128, (S + 63) // 64 * 64
    qkv = rng.integers(-9, 10, (S, 3, H, 128))
    ws = (1 + 0.3 * rng.standard_normal((4, 128))).astype(np.float32)
    cos, sin = (t.astype(np.float32) for t in tables(rng, S, rope))
    dqkv, q, k, vt = tl.Dev.of(tl.to_bf16(qkv)), tl.Dev(S * h * 2), tl.Dev(S * h * 2), tl.Dev(h * S_pad * 2)
    dw, dt = [tl.Dev.of(w) for w in ws], [tl.Dev.of(np.repeat(t, 2, 1)) for t in (cos, sin)]
    a = tl.QkPrepArgs(dqkv.ptr, 3 * h, h, 2 * h, q.ptr, k.ptr, vt.ptr, S_pad, S, H, dw[0].ptr, dw[1].ptr, dw[2].ptr,
                      dw[3].ptr, split, *((t.ptr if rope else None) for t in dt), 0, EPS, 0, None, None)
    assert lib.iris_hip_qk_prepare(ctypes.byref(a)) == 0, lib.iris_hip_last_error()
    assert lib.iris_hip_sync() == 0
    first = np.arange(S)[:, None] < split
    for i, dev in ((0, q), (1, k)):
        ref = norm_bits(qkv[:, i], np.where(first, ws[i], ws[2 + i]), cos, sin)
        assert np.array_equal(dev.get(np.uint16, (S, H, 128)), ref), i


@pytest.mark.parametrize("S,H,split,rope", [(512, 8, 200, False), (4000, 4, 1000, False), (4000, 9, 33, False),
                                            (512, 8, 512, True), (4000, 9, 0, True)])
def test_query_prologue(lib, S, H, split, rope):
    """The attention's own normalisation of its query rows against the same
    launch on rows normalised here: with keys 64 e_j and values e_j an output
    is the softmax of 5.66 q itself, where a query's last bf16 bit shows. Both
    block shapes (4 and 8 waves)."""
    rng = np.random.default_rng(S + H)
    raw = rng.integers(-9, 10, (S, H, 128))
    wa, wb = (1 + 0.3 * rng.standard_normal((2, 128))).astype(np.float32)
    cos, sin = (t.astype(np.float32) for t in tables(rng, S, rope))
    qn = norm_bits(raw, np.where(np.arange(S)[:, None] < split, wa, wb), cos, sin)
    k = np.broadcast_to(64 * np.eye(128, dtype=np.float32)[:, None], (128, H, 128))
    vt = np.broadcast_to(np.eye(128, dtype=np.float32), (H, 128, 128))
    draw, dqn, dk, dvt = (tl.Dev.of(v) for v in (tl.to_bf16(raw), qn, tl.to_bf16(k), tl.to_bf16(vt)))
    dwa, dwb, dc, ds, o = tl.Dev.of(wa), tl.Dev.of(wb), tl.Dev.of(cos), tl.Dev.of(sin), tl.Dev(S * H * 256)
    got = []
    for q, tail in ((draw, (dwa.ptr, dwb.ptr, split, EPS, *((t.ptr if rope else None) for t in (dc, ds)))), (dqn, ())):
        a = tl.AttnArgs(q.ptr, dk.ptr, dvt.ptr, o.ptr, H * 128, H * 128, 128, H * 128, S, 128, H, 1, 0, 0, 0, 0,
                        1 / math.sqrt(128), 0, 128, 0, 0, 0, 0, 0, 0.0, *tail)
        assert lib.iris_hip_attention(ctypes.byref(a)) == 0, lib.iris_hip_last_error()
        got.append(o.get(np.uint16, (S, H, 128)))
    assert np.array_equal(got[0], got[1])
