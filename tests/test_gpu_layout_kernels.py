"""The layout and conversion kernels at the edges of their blocks: remainders,
unaligned buffers, few pixels."""
import ctypes

import numpy as np
import pytest

import iris_testlib as tl

pytestmark = pytest.mark.gpu
VP, I = ctypes.c_void_p, ctypes.c_int


@pytest.fixture(scope="module")
def lib():
    lib = tl.hip()
    lib.iris_hip_f32_to_bf16.argtypes = [VP, VP, ctypes.c_size_t]
    lib.iris_hip_vae_front.argtypes = [VP, VP, I, I, I, VP, VP, I, VP, VP]
    lib.iris_hip_vae_enc_out.argtypes = [VP, VP, I, I, I, VP, VP, VP, VP]
    lib.iris_hip_vae_img_in.argtypes = [VP, VP, I, I]
    lib.iris_hip_gn_apply.argtypes = [VP, I, VP, I, I, I, VP, VP]
    return lib


@pytest.mark.parametrize("n,skip", [(1, 0), (8, 0), (2056, 0), (2051, 0), (2056, 1), (100000, 2)])
def test_f32_to_bf16(lib, n, skip):
    """Whole 16-byte chunks, a remainder, and buffers off their alignment by
    `skip` elements: round to nearest even, infinities and NaN kept."""
    x = np.random.default_rng(n).standard_normal(n + skip).astype(np.float32)
    x[skip:skip + 4] = np.array([np.inf, -np.inf, np.nan, 1.00390625], np.float32)[:min(4, n)]
    d, o = tl.Dev.of(x), tl.Dev((n + skip) * 2)
    assert lib.iris_hip_f32_to_bf16(o.ptr + 2 * skip, d.ptr + 4 * skip, n) == 0
    got = o.get(np.uint16, (n + skip,))[skip:]
    want = tl.to_bf16(x[skip:])
    nan = np.isnan(x[skip:])
    assert np.array_equal(got[~nan], want[~nan]) and np.all(np.isnan(tl.bf16_to_f32(got[nan])))


@pytest.mark.parametrize("C,hw", [(128, 1), (128, 31), (128, 33), (128, 256), (96, 65), (40, 32)])
def test_nchw_to_tokens(lib, C, hw):
    x = np.random.default_rng(hw).standard_normal((C, hw)).astype(np.float32)
    d, o = tl.Dev.of(x), tl.Dev(C * hw * 2)
    assert lib.iris_hip_nchw_to_tokens(o.ptr, d.ptr, C, hw) == 0
    assert np.array_equal(o.get(np.uint16, (hw, C)), tl.to_bf16(np.ascontiguousarray(x.T)))


@pytest.mark.parametrize("N,K,act", [(8192, 3072, 1), (8195, 520, 0), (17 * 512, 512, 1), (8192, 4096, 0)])
def test_gemv_rows(lib, N, K, act):
    """Products of enough rows for four to a wave, a ragged last wave: the
    same bits as the same rows a few at a time."""
    rng = np.random.default_rng(N + K)
    w = tl.to_bf16((rng.standard_normal((N, K)) * 0.03).astype(np.float32))
    x, b = rng.standard_normal(K).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    dw, dx, db, dy, dz = tl.Dev.of(w), tl.Dev.of(x), tl.Dev.of(b), tl.Dev(N * 4), tl.Dev(N * 4)
    assert lib.iris_hip_gemv(dy.ptr, dw.ptr, dx.ptr, db.ptr, N, K, act) == 0
    for n0 in range(0, N, 4096):
        n = min(4096, N - n0)
        assert lib.iris_hip_gemv(dz.ptr + 4 * n0, dw.ptr + 2 * n0 * K, dx.ptr, db.ptr + 4 * n0, n, K, act) == 0
    y, z = dy.get(np.float32, (N,)), dz.get(np.float32, (N,))
    assert np.array_equal(y, z)
    xs = x.astype(np.float64) / (1 + np.exp(-x.astype(np.float64))) if act else x
    assert tl.rel_l2(y, tl.bf16_to_f32(w).astype(np.float64) @ xs + b) < 1e-5


@pytest.mark.parametrize("z,h,w,conv", [(32, 1, 1, True), (16, 5, 7, True), (32, 4, 8, False), (3, 2, 3, True)])
def test_vae_front(lib, z, h, w, conv):
    """Few pixels, z below the 8-channel chunk, with and without the 1x1."""
    rng = np.random.default_rng(z + h)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    lat, sc, sh, pw, pb = f(4 * z, h, w), f(4 * z), f(4 * z), f(z, z), f(z)
    o = tl.Dev(4 * h * w * 64 * 2)
    d = [tl.Dev.of(a) for a in (lat, sc, sh, pw, pb)]
    assert lib.iris_hip_vae_front(o.ptr, d[0].ptr, z, h, w, d[1].ptr, d[2].ptr, 0, d[3].ptr if conv else None,
                                  d[4].ptr if conv else None) == 0
    y = lat.astype(np.float64) * sc[:, None, None] + sh[:, None, None]
    y = y.reshape(z, 2, 2, h, w).transpose(3, 1, 4, 2, 0).reshape(2 * h, 2 * w, z)
    if conv:
        y = y @ pw.astype(np.float64).T + pb
    got = tl.bf16_to_f32(o.get(np.uint16, (2 * h, 2 * w, 64)))
    assert tl.rel_l2(got[..., :z], y) < 4e-3 and not got[..., z:].any()


@pytest.mark.parametrize("z,h,w,conv", [(32, 2, 2, True), (16, 6, 10, True), (16, 5, 7, False), (90, 2, 6, True)])
def test_vae_enc_out(lib, z, h, w, conv):
    """Few pixels, odd sides (the last row and column have no latent), and
    more channels than LDS holds."""
    rng = np.random.default_rng(z + h)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    lh, lw = h // 2, w // 2
    m, qw, qb, sc, sh = f(h, w, 2 * z), f(2 * z, 2 * z), f(2 * z), f(4 * z), f(4 * z)
    o = tl.Dev.of(np.zeros((4 * z, lh, lw), np.float32))
    d = [tl.Dev.of(a) for a in (m, qw, qb, sc, sh)]
    assert lib.iris_hip_vae_enc_out(o.ptr, d[0].ptr, z, h, w, d[1].ptr if conv else None,
                                    d[2].ptr if conv else None, d[3].ptr, d[4].ptr) == 0
    y = m.astype(np.float64)
    if conv:
        y = y @ qw.astype(np.float64).T + qb
    y = y[:2 * lh, :2 * lw, :z].reshape(lh, 2, lw, 2, z).transpose(4, 1, 3, 0, 2).reshape(4 * z, lh, lw)
    assert tl.rel_l2(o.get(np.float32, (4 * z, lh, lw)), (y - sh[:, None, None]) * sc[:, None, None]) < 1e-5


@pytest.mark.parametrize("H,W", [(1, 1), (3, 11), (16, 32)])
def test_vae_img_in(lib, H, W):
    x = np.random.default_rng(H).standard_normal((3, H, W)).astype(np.float32)
    o = tl.Dev(H * W * 64 * 2)
    d = tl.Dev.of(x)
    assert lib.iris_hip_vae_img_in(o.ptr, d.ptr, H, W) == 0
    got = o.get(np.uint16, (H, W, 64))
    assert np.array_equal(got[..., :3], tl.to_bf16(np.ascontiguousarray(x.transpose(1, 2, 0)))) and not got[..., 3:].any()


@pytest.mark.parametrize("pix,C", [(1, 64), (33, 512), (17, 96), (7, 24)])
@pytest.mark.parametrize("swish", [0, 1])
def test_gn_apply(lib, pix, C, swish):
    """Channel counts that are and are not powers of two, f32 input with the
    raw copy, against float64 within the bf16 rounding of the result."""
    rng = np.random.default_rng(pix + C)
    x, ab = rng.standard_normal((pix, C)).astype(np.float32), rng.standard_normal((2, C)).astype(np.float32)
    dx, da, dy, dr = tl.Dev.of(x), tl.Dev.of(ab), tl.Dev(pix * C * 2), tl.Dev(pix * C * 2)
    assert lib.iris_hip_gn_apply(dx.ptr, 0, da.ptr, pix, C, swish, dy.ptr, dr.ptr) == 0
    t = x.astype(np.float64) * ab[0] + ab[1]
    t = t / (1 + np.exp(-t)) if swish else t
    assert tl.rel_l2(tl.bf16_to_f32(dy.get(np.uint16, (pix, C))), t) < 4e-3
    assert np.array_equal(dr.get(np.uint16, (pix, C)), tl.to_bf16(x))
