"""iris_hip_conv3x3_tiled: 3x3 convolutions on 16 x 16 pixel tiles, against
float64, and the GroupNorm sums of each tile."""
import ctypes

import numpy as np
import pytest

import iris_testlib as tl

pytestmark = pytest.mark.gpu
EPI_F32, EPI_BF16, EPI_ADD = 0, 1, 5


@pytest.fixture(scope="module")
def lib():
    lib = tl.hip()
    lib.iris_hip_conv3x3_tiled.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    return lib


def bf(x):
    return tl.bf16_to_f32(tl.to_bf16(x))


def conv64(x, w, b, up):
    if up:
        x = x.repeat(2, 0).repeat(2, 1)
    H, W = x.shape[:2]
    xp = np.pad(x.astype(np.float64), ((1, 1), (1, 1), (0, 0)))
    out = np.zeros((H, W, w.shape[0])) + b
    for tap in range(9):
        dy, dx = tap // 3, tap % 3
        out += xp[dy:dy + H, dx:dx + W] @ w[:, tap].astype(np.float64).T
    return out


@pytest.mark.parametrize("H,W,cin,cout,up,tiled", [
    (176, 192, 64, 128, 0, True),      # one channel chunk, whole tiles
    (173, 190, 128, 128, 0, True),     # two chunks (both patch buffers), ragged on both sides
    (96, 97, 256, 512, 0, True),       # four chunks, four channel tiles
    (160, 208, 64, 256, 1, True),      # through the upsample
    (150, 190, 128, 256, 1, True),     # upsample, ragged
    (1, 1, 64, 128, 0, True),          # one pixel
    (16, 17, 64, 128, 0, True),    # two tiles
    (170, 193, 64, 192, 0, False),     # a part-empty channel tile: the other kernel
])
def test_conv3x3_tiled(lib, H, W, cin, cout, up, tiled):
    """Every epilogue against float64 (f32 sums: 1e-5; bf16 output: 4e-3),
    repeatable bit for bit, which kernel ran, and with the sums requested the
    sum and sum of squares per tile and group of what was written."""
    G = 32
    rng = np.random.default_rng(H + W + cin)
    x = bf(rng.standard_normal((H >> up, W >> up, cin)).astype(np.float32))
    w = bf((rng.standard_normal((cout, 9, cin)) / np.sqrt(9 * cin)).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    ref = conv64(x, w, b, up)
    dx, dw, db = tl.Dev.of(tl.to_bf16(x)), tl.Dev.of(tl.to_bf16(w)), tl.Dev.of(b)
    x0 = rng.standard_normal((H, W, cout)).astype(np.float32)
    ty, tx = -(-H // 16), -(-W // 16)
    gn = cout % (4 * G) == 0
    for epi in (EPI_F32, EPI_BF16, EPI_ADD):
        got = []
        for _ in range(2):
            o = tl.Dev(H * W * cout * 2) if epi == EPI_BF16 else tl.Dev.of(x0)
            part = tl.Dev.of(np.zeros((max(ty * tx, -(-H * W // 256)), G, 2)))
            c = tl.Conv3x3(dx.ptr, dw.ptr, o.ptr, db.ptr, H, W, cin, cout, up, cout, epi, 1, None, 0,
                           part.ptr if gn else None, G if gn else 0)
            n = ctypes.c_int(-1)
            assert lib.iris_hip_profile_enable(1) == 0
            assert lib.iris_hip_conv3x3_tiled(ctypes.byref(c), ctypes.byref(n)) == 0, lib.iris_hip_last_error()
            recs = (tl.KernelTime * 4)()
            assert lib.iris_hip_profile_read(recs, 4) == 1 and lib.iris_hip_profile_enable(0) == 0
            assert (b"patch" in recs[0].kernel) == tiled, recs[0].kernel
            assert n.value == (0 if not gn else ty * tx if tiled else -(-H * W // 256))
            got.append((o.get(np.uint16 if epi == EPI_BF16 else np.float32, (H, W, cout)),
                        part.get(np.float64, (max(ty * tx, -(-H * W // 256)), G, 2))))
            o.close()
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
        y = tl.bf16_to_f32(got[0][0]) if epi == EPI_BF16 else got[0][0]
        want = ref + x0 if epi == EPI_ADD else ref
        assert tl.rel_l2(y, want) < (4e-3 if epi == EPI_BF16 else 1e-5)
        if gn and tiled:
            pad = np.zeros((ty * 16, tx * 16, cout))
            pad[:H, :W] = want
            t = pad.reshape(ty, 16, tx, 16, G, cout // G)
            sums = np.stack([t.sum((1, 3, 5)), (t * t).sum((1, 3, 5))], -1).reshape(ty * tx, G, 2)
            # f32 sums of 256 x 4 .. 16 values: their rounding against the sum of magnitudes
            np.testing.assert_allclose(got[0][1], sums, rtol=1e-4, atol=2e-2)


@pytest.mark.parametrize("H,W,cin,cout,up", [(32, 32, 512, 512, 0), (20, 22, 256, 128, 1), (16, 16, 512, 256, 0),
                                             (33, 18, 512, 128, 0)])
def test_conv3x3_tiled_split(lib, H, W, cin, cout, up):
    """Few tiles and a workspace: split over the input channels, partials
    reduced in order: every epilogue against float64, repeatable; no sums."""
    rng = np.random.default_rng(H + cin)
    x = bf(rng.standard_normal((H >> up, W >> up, cin)).astype(np.float32))
    w = bf((rng.standard_normal((cout, 9, cin)) / np.sqrt(9 * cin)).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    ref = conv64(x, w, b, up)
    dx, dw, db = tl.Dev.of(tl.to_bf16(x)), tl.Dev.of(tl.to_bf16(w)), tl.Dev.of(b)
    x0 = rng.standard_normal((H, W, cout)).astype(np.float32)
    nb = 8 * H * W * cout * 4
    ws, part = tl.Dev(nb), tl.Dev(4096 * 64 * 8)
    for epi in (EPI_F32, EPI_BF16, EPI_ADD):
        got, split = [], False
        for _ in range(2):
            o = tl.Dev(H * W * cout * 2) if epi == EPI_BF16 else tl.Dev.of(x0)
            c = tl.Conv3x3(dx.ptr, dw.ptr, o.ptr, db.ptr, H, W, cin, cout, up, cout, epi, 0, ws.ptr, nb, part.ptr, 32)
            n = ctypes.c_int(-1)
            assert lib.iris_hip_profile_enable(1) == 0
            assert lib.iris_hip_conv3x3_tiled(ctypes.byref(c), ctypes.byref(n)) == 0, lib.iris_hip_last_error()
            recs = (tl.KernelTime * 4)()
            k = lib.iris_hip_profile_read(recs, 4)
            assert lib.iris_hip_profile_enable(0) == 0
            names = [r.kernel for r in recs[:k]]
            split = any(b"reduce" in m for m in names)
            assert any(b"patch" in m for m in names) and (n.value == 0) == split, (names, n.value)
            got.append(o.get(np.uint16 if epi == EPI_BF16 else np.float32, (H, W, cout)))
            o.close()
        assert split and np.array_equal(got[0], got[1])
        y = tl.bf16_to_f32(got[0]) if epi == EPI_BF16 else got[0]
        assert tl.rel_l2(y, ref + x0 if epi == EPI_ADD else ref) < (4e-3 if epi == EPI_BF16 else 1e-5)


@pytest.mark.parametrize("H,W,cin,cout,up", [(64, 48, 256, 512, 0), (61, 50, 128, 256, 0), (33, 31, 512, 128, 0),
                                             (64, 64, 128, 256, 1), (50, 34, 64, 128, 1)])
def test_conv3x3_tiled_few_tiles(lib, H, W, cin, cout, up):
    """Tiles of 64 channels (twice the tiles of 128 still have a CU each):
    whole, ragged and upsampled, over one and several chunks."""
    test_conv3x3_tiled(lib, H, W, cin, cout, up, True)


@pytest.mark.parametrize("G", [8, 16, 32])
def test_conv3x3_tiled_wide_groups(lib, G):
    """Groups of 128, 64 and 32 channels: wider than, as wide as and within a
    64-channel tile."""
    H = W = 16
    cin, cout = 64, 1024
    rng = np.random.default_rng(G)
    x = bf(rng.standard_normal((H, W, cin)).astype(np.float32))
    w = bf((rng.standard_normal((cout, 9, cin)) / np.sqrt(9 * cin)).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    dx, dw, db = tl.Dev.of(tl.to_bf16(x)), tl.Dev.of(tl.to_bf16(w)), tl.Dev.of(b)
    o, part = tl.Dev(H * W * cout * 4), tl.Dev(G * 16)
    c = tl.Conv3x3(dx.ptr, dw.ptr, o.ptr, db.ptr, H, W, cin, cout, 0, cout, EPI_F32, 1, None, 0, part.ptr, G)
    n = ctypes.c_int(-1)
    assert lib.iris_hip_conv3x3_tiled(ctypes.byref(c), ctypes.byref(n)) == 0, lib.iris_hip_last_error()
    assert n.value == 1
    ref = conv64(x, w, b, 0)
    assert tl.rel_l2(o.get(np.float32, (H, W, cout)), ref) < 1e-5
    t = ref.reshape(H * W, G, cout // G)
    # f32 sums of 64 to 128 values per thread, their rounding against the sum of magnitudes
    np.testing.assert_allclose(part.get(np.float64, (G, 2)), np.stack([t.sum((0, 2)), (t * t).sum((0, 2))], -1),
                               rtol=1e-4, atol=5e-2)


@pytest.mark.parametrize("cout,G,ok", [(1024, 4, True), (512, 2, True), (512, 1, False), (512, 3, False), (384, 2, False)])
def test_conv3x3_tiled_groups_of_the_other_kernel(lib, cout, G, ok):
    """Groups wider than a tile's 128 channels run on, or are refused by, the
    other kernel, with its bits and sums and the number of its row tiles."""
    H, W, cin = 20, 15, 64
    rng = np.random.default_rng(G)
    x = rng.standard_normal((H, W, cin)).astype(np.float32)
    w = (rng.standard_normal((cout, 9, cin)) / np.sqrt(9 * cin)).astype(np.float32)
    dx, dw = tl.Dev.of(tl.to_bf16(x)), tl.Dev.of(tl.to_bf16(w))
    got = []
    for tiled in (0, 1):
        o, part = tl.Dev.of(np.zeros((H, W, cout), np.float32)), tl.Dev.of(np.zeros((2, G, 2)))
        c = tl.Conv3x3(dx.ptr, dw.ptr, o.ptr, None, H, W, cin, cout, 0, cout, EPI_F32, 1, None, 0, part.ptr, G)
        n = ctypes.c_int(-1)
        rc = lib.iris_hip_conv3x3_tiled(ctypes.byref(c), ctypes.byref(n)) if tiled else lib.iris_hip_conv3x3(ctypes.byref(c))
        assert (rc == 0) == ok, (tiled, lib.iris_hip_last_error())
        if tiled and ok:
            assert n.value == 2
        got.append((o.get(np.uint32, (H, W, cout)), part.get(np.uint64, (2, G, 2))))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("H,W,cin,cout,up,tiled", [
    (128, 128, 512, 512, 0, True),     # one round of tiles
    (144, 144, 512, 512, 0, True),     # 1.27 rounds of tiles, 162 row tiles: 94 us, 93 there and 4 in the pass after
    (132, 132, 512, 512, 1, True),     # upsampled 90, 92 there
    (176, 176, 512, 512, 0, True),     # 1.89 rounds: 105, 112 there
    (180, 180, 512, 512, 0, False),    # 2.25 rounds, 254 row tiles: 145, 114 there
    (180, 180, 512, 512, 1, False),    # 138, 115 there
    (192, 192, 512, 512, 0, True),     # 2.25 rounds, 288 row tiles: 148, 187 there
    (360, 360, 512, 256, 0, False),    # 248, 225 there
    (360, 360, 256, 128, 0, False),    # 87, 82 there
    (90, 166, 512, 512, 0, False),     # tiles overshoot: 93, 67 there
    (17, 640, 512, 512, 0, False),     # by 1.9: 94, 62 there
])
def test_conv3x3_tiled_rounds(lib, H, W, cin, cout, up, tiled):
    """Past one tile per CU the kernel measured faster runs, and gives what the
    other gives up to the order of the sums and a rounding to bf16."""
    rng = np.random.default_rng(H)
    x = rng.standard_normal(((H >> up) * (W >> up) * cin), np.float32)
    w = rng.standard_normal(cout * 9 * cin, np.float32) / np.float32(np.sqrt(9 * cin))
    dx, dw = tl.Dev.of(tl.to_bf16(x)), tl.Dev.of(tl.to_bf16(w))
    outs = []
    for other in (0, 1):
        o = tl.Dev(H * W * cout * 2)
        c = tl.Conv3x3(dx.ptr, dw.ptr, o.ptr, None, H, W, cin, cout, up, cout, EPI_BF16, 1, None, 0, None, 0)
        assert lib.iris_hip_profile_enable(1) == 0
        rc = lib.iris_hip_conv3x3(ctypes.byref(c)) if other else lib.iris_hip_conv3x3_tiled(ctypes.byref(c), None)
        assert rc == 0, lib.iris_hip_last_error()
        recs = (tl.KernelTime * 4)()
        assert lib.iris_hip_profile_read(recs, 4) == 1 and lib.iris_hip_profile_enable(0) == 0
        assert (b"patch" in recs[0].kernel) == (tiled and not other), recs[0].kernel
        outs.append(tl.bf16_to_f32(o.get(np.uint16, (H, W, cout))))
    assert tl.rel_l2(outs[0], outs[1]) < 4e-3


@pytest.mark.parametrize("H,W,cin,cout,up,split", [
    (173, 190, 128, 128, 0, False),   # 128-channel tiles, ragged
    (61, 50, 128, 256, 0, False),     # 64-channel tiles
    (64, 64, 128, 256, 1, False),     # through the upsample
    (32, 32, 512, 512, 0, True),      # partial sums, then the conversion
    (20, 23, 64, 192, 0, False),      # the other kernel, then the conversion
])
def test_conv3x3_add_bf16(lib, H, W, cin, cout, up, split):
    """The residual epilogue leaving in bf16: the bits of IRIS_EPI_ADD followed
    by the conversion."""
    lib.iris_hip_conv3x3_add_bf16.argtypes = [ctypes.c_void_p] * 2
    lib.iris_hip_f32_to_bf16.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    rng = np.random.default_rng(H + cin)
    dx = tl.Dev.of(tl.to_bf16(rng.standard_normal((H >> up, W >> up, cin)).astype(np.float32)))
    dw = tl.Dev.of(tl.to_bf16((rng.standard_normal((cout, 9, cin)) / np.sqrt(9 * cin)).astype(np.float32)))
    db = tl.Dev.of(rng.standard_normal(cout).astype(np.float32))
    x0 = rng.standard_normal((H, W, cout)).astype(np.float32)
    nb = 8 * H * W * cout * 4
    ws = tl.Dev(nb) if split else None
    got = []
    for direct in (True, False):
        o, y = tl.Dev.of(x0), tl.Dev.of(np.zeros((H, W, cout), np.uint16))
        c = tl.Conv3x3(dx.ptr, dw.ptr, o.ptr, db.ptr, H, W, cin, cout, up, cout, EPI_ADD, 0, ws.ptr if split else None,
                       nb if split else 0, None, 0)
        if direct:
            assert lib.iris_hip_conv3x3_add_bf16(ctypes.byref(c), y.ptr) == 0, lib.iris_hip_last_error()
        else:
            assert lib.iris_hip_conv3x3_tiled(ctypes.byref(c), None) == 0, lib.iris_hip_last_error()
            assert lib.iris_hip_f32_to_bf16(y.ptr, o.ptr, H * W * cout) == 0
        assert lib.iris_hip_sync() == 0
        got.append(y.get(np.uint16, (H, W, cout)))
    assert np.array_equal(got[0], got[1]) and tl.bf16_to_f32(got[0]).std() > 0.5
    c.epi = EPI_F32
    assert lib.iris_hip_conv3x3_add_bf16(ctypes.byref(c), y.ptr) != 0


@pytest.mark.parametrize("H,W,cin,cout,up,G", [(17, 33, 64, 256, 2, 32), (16, 16, 128, 384, 2, 0), (20, 21, 64, 320, 0, 0),
                                               (16, 32, 64, 256, 1, 2), (16, 16, 64, 512, 2, 2)])
def test_conv3x3_narrow_tiles(lib, H, W, cin, cout, up, G):
    """The implicit GEMM with few tiles: 128 channels each (a part-empty last
    one too), 256 where a GroupNorm's group is wider; float64 outputs and sums."""
    lib.iris_hip_conv3x3.argtypes = [ctypes.c_void_p]
    rng = np.random.default_rng(H + cout)
    shape = (2 * H, 2 * W, cin) if up == 2 else (H >> up, W >> up, cin)
    x = bf(rng.standard_normal(shape).astype(np.float32))
    w = bf((rng.standard_normal((cout, 9, cin)) / np.sqrt(9 * cin)).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    if up == 2:   # one row and column of zeros after the image, stride 2
        ref = conv64(np.pad(x, ((0, 1), (0, 1), (0, 0))), w, b, 0)[1:-1:2, 1:-1:2]
    else:
        ref = conv64(x, w, b, up)
    blocks = -(-H * W // 256)
    dx, dw, db = tl.Dev.of(tl.to_bf16(x)), tl.Dev.of(tl.to_bf16(w)), tl.Dev.of(b)
    o, part = tl.Dev(H * W * cout * 4), tl.Dev(blocks * max(G, 1) * 16)
    c = tl.Conv3x3(dx.ptr, dw.ptr, o.ptr, db.ptr, H, W, cin, cout, up, cout, EPI_F32, 1, None, 0,
                   part.ptr if G else None, G)
    assert lib.iris_hip_conv3x3(ctypes.byref(c)) == 0, lib.iris_hip_last_error()
    assert lib.iris_hip_sync() == 0
    assert tl.rel_l2(o.get(np.float32, (H, W, cout)), ref) < 1e-5
    if G:
        pad = np.zeros((blocks * 256, cout))
        pad[:H * W] = ref.reshape(-1, cout)
        t = pad.reshape(blocks, 256, G, cout // G)
        # f32 sums of 16 values, their rounding against the sum of magnitudes
        np.testing.assert_allclose(part.get(np.float64, (blocks, G, 2)),
                                   np.stack([t.sum((1, 3)), (t * t).sum((1, 3))], -1), rtol=1e-4, atol=5e-2)
