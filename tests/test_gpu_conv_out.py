"""The output convolution (3x3, cin -> 3) with the image conversion, from bf16
and from the f32 stream with its GroupNorm scale, shift and swish on the way
in, against float64: edges of the 30 x 16 tiles, channel counts round a
128-channel step, blocks that take several tiles."""
import ctypes

import numpy as np
import pytest

import iris_testlib as tl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    lib = tl.hip()
    vp, i = ctypes.c_void_p, ctypes.c_int
    lib.iris_hip_vae_conv_out.argtypes = [vp, vp, vp, i, i, i, vp, vp]
    lib.iris_hip_vae_conv_out_norm.argtypes = [vp, vp, vp, vp, i, i, i, vp, vp]
    return lib


@pytest.mark.parametrize("H,W,cin", [(1, 1, 128), (16, 30, 128), (17, 31, 128), (15, 61, 256), (33, 29, 8),
                                     (34, 64, 136), (640, 481, 16)])
@pytest.mark.parametrize("norm", [False, True])
def test_conv_out_f64(lib, H, W, cin, norm):
    rng = np.random.default_rng(H * W + cin)
    x = rng.standard_normal((H, W, cin)).astype(np.float32)
    ab = (rng.standard_normal((2, cin)) + 0.5).astype(np.float32)
    w = (0.5 * rng.standard_normal((9, cin, 3)) / np.sqrt(9 * cin)).astype(np.float32)
    b = (0.1 * rng.standard_normal(3)).astype(np.float32)
    wt = np.zeros((9, cin, 4), np.float32)
    wt[:, :, :3] = w
    if norm:
        t = x.astype(np.float64) * ab[0] + ab[1]
        g = t / (1.0 + np.exp(-t))
        # the activation: a rounded scale and shift, exp of a rounded argument, a reciprocal and a product
        gerr = 2.0 ** -23 * ((np.abs(x * ab[0]) + np.abs(t)) * 1.2 + (4 + np.abs(t)) * np.abs(g))
    else:
        x = tl.bf16_to_f32(tl.to_bf16(x))
        g, gerr = x.astype(np.float64), np.zeros(x.shape)
    pad = lambda a: np.pad(a, ((1, 1), (1, 1), (0, 0)))  # noqa: E731
    gp, ep = pad(g), pad(gerr)
    ref, err = np.zeros((H, W, 3)) + b, np.zeros((H, W, 3)) + np.abs(b) * 2.0 ** -24
    n = 9 * cin + 10
    for tap in range(9):
        dy, dx = divmod(tap, 3)
        gs, es = gp[dy:dy + H, dx:dx + W], ep[dy:dy + H, dx:dx + W]
        ref += gs @ w[tap].astype(np.float64)
        err += (np.abs(gs) * n * 2.0 ** -24 + es) @ np.abs(w[tap]).astype(np.float64)
    dx_ = tl.Dev.of(x if norm else tl.to_bf16(x))
    dab, dw, db = tl.Dev.of(ab), tl.Dev.of(wt), tl.Dev.of(np.r_[b, 0].astype(np.float32))
    rgb, f = tl.Dev(H * W * 3), tl.Dev(3 * H * W * 4)
    if norm:
        rc = lib.iris_hip_vae_conv_out_norm(rgb.ptr, f.ptr, dx_.ptr, dab.ptr, H, W, cin, dw.ptr, db.ptr)
    else:
        rc = lib.iris_hip_vae_conv_out(rgb.ptr, f.ptr, dx_.ptr, H, W, cin, dw.ptr, db.ptr)
    assert rc == 0, lib.iris_hip_last_error()
    assert lib.iris_hip_sync() == 0
    got = f.get(np.float32, (3, H, W)).transpose(1, 2, 0)
    assert (np.abs(got - ref) <= err).all()
    v = np.clip((got + np.float32(1.0)) * np.float32(0.5) * np.float32(255.0), 0, 255)
    assert np.array_equal(rgb.get(np.uint8, (H, W, 3)), (v + np.float32(0.5)).astype(np.uint8))
