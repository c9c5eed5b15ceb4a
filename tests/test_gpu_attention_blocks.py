"""The attention's two block shapes: launches whose 128-query blocks fit one
round take 4 waves, larger ones 8. A head's result does not depend on which:
the first heads of a launch past the line, bit for bit, and float64."""
import ctypes
import math

import numpy as np
import pytest

import iris_testlib as tl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    return tl.hip()


def bf(x):
    return tl.bf16_to_f32(tl.to_bf16(x))


@pytest.mark.parametrize("S,mask,causal,group,bias,fused", [
    (1, None, 0, 0, 0, False), (63, None, 0, 0, 0, True), (64, None, 1, 2, 0, True), (65, None, 1, 2, 0, True),
    (127, (0, 100, 0, 0), 0, 0, 0, True), (128, None, 0, 0, 0.7, True), (129, None, 1, 4, 0, False),
    (193, (0, 64, 96, 190), 0, 0, 0, True), (256, (70, 200, 0, 0), 0, 0, 0, False), (300, None, 0, 0, -1.0, True)])
def test_block_shapes_bitwise(lib, S, mask, causal, group, bias, fused):
    """Rows around the 64-key tiles and the 128-query blocks, key ranges that
    leave tiles masked, causal with grouped queries, a key bias, with and
    without the Q prologue whose weight line falls inside a wave."""
    cus = int(lib.iris_hip_device_name().decode().rsplit(",", 1)[1].split()[0])
    g = max(group, 1)
    few = 8
    many = (cus // -(-S // 128) // g + 1) * g + g      # past one round of 128-query blocks
    rng = np.random.default_rng(S)
    S_pad, split = (S + 63) // 64 * 64, S // 2 + 3
    q = rng.standard_normal((S, many, 128)).astype(np.float32)
    k = rng.standard_normal((S, many // g, 128)).astype(np.float32)
    v = rng.standard_normal((S, many // g, 128)).astype(np.float32)
    wa, wb = (1 + 0.3 * rng.standard_normal((2, 128))).astype(np.float32)
    ang = rng.uniform(-3, 3, (S, 64)).astype(np.float32)
    cs, sn = np.cos(ang), np.sin(ang)
    vt = np.zeros((many // g, 128, S_pad), np.float32)
    vt[:, :, :S] = v.transpose(1, 2, 0)
    dq, dk, dvt = tl.Dev.of(tl.to_bf16(q)), tl.Dev.of(tl.to_bf16(k)), tl.Dev.of(tl.to_bf16(vt))
    dw = [tl.Dev.of(a) for a in (wa, wb, cs, sn)]
    lo0, hi0, lo1, hi1 = mask or (0, S, 0, 0)
    outs, names = [], []
    for H in (few, many):
        o = tl.Dev(S * H * 128 * 2)
        a = tl.AttnArgs(dq.ptr, dk.ptr, dvt.ptr, o.ptr, many * 128, many // g * 128, S_pad, H * 128, S, S, H, 1, 0, 0,
                        0, 0, 1 / math.sqrt(128), lo0, hi0, lo1, hi1, causal, group, S // 3, bias,
                        *((dw[0].ptr, dw[1].ptr, split, 1e-6, dw[2].ptr, dw[3].ptr) if fused else ()))
        assert lib.iris_hip_profile_enable(1) == 0
        assert lib.iris_hip_attention(ctypes.byref(a)) == 0, lib.iris_hip_last_error()
        recs = (tl.KernelTime * 4)()
        assert lib.iris_hip_profile_read(recs, 4) == 1 and lib.iris_hip_profile_enable(0) == 0
        names.append(recs[0].kernel.decode())
        outs.append(o.get(np.uint16, (S, H, 128))[:, :few])
        o.close()
    assert names[0].endswith(", 4>") and not names[1].endswith(", 4>"), names
    assert np.array_equal(outs[0], outs[1])
    at = np.arange(S)
    ok = ((at >= lo0) & (at < hi0) | (at >= lo1) & (at < hi1))[None] & (~np.bool_(causal) | (at[None] <= at[:, None]))
    for h in range(few):
        x = bf(q[:, h]).astype(np.float64)
        if fused:
            x = x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-6) * np.where(at[:, None] < split, wa, wb)
            x0, x1 = x[:, 0::2], x[:, 1::2]
            x = np.stack([x0 * cs - x1 * sn, x1 * cs + x0 * sn], -1).reshape(S, 128)
        sc = x @ bf(k[:, h // g]).astype(np.float64).T / math.sqrt(128) + bias * (at[None] >= S // 3)
        sc = np.where(ok, sc, -np.inf)
        p = np.exp(sc - sc.max(1, keepdims=True))
        ref = p / p.sum(1, keepdims=True) @ bf(v[:, h // g]).astype(np.float64)
        assert tl.rel_l2(tl.bf16_to_f32(outs[0][:, h]), ref) < 1e-2, h
