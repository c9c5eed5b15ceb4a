"""iris_hip_gemm_ring (small tiles, loads in waves of their own) against the
two-stage kernel, bit for bit, and against float64; and the products of few
rows for which iris_hip_gemm_fill takes it."""
import ctypes

import numpy as np
import pytest

import iris_testlib as tl

pytestmark = pytest.mark.gpu
EPI_F32, EPI_BF16, EPI_GATED_ADD, EPI_SWIGLU, EPI_F32_T, EPI_ADD = range(6)
WS = 32 << 20


@pytest.fixture(scope="module")
def lib():
    lib = tl.hip()
    vp, sz, i = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int
    lib.iris_hip_gemm_ring.argtypes = [vp, i, i, i, vp, sz]
    lib.iris_hip_gemm_splitk.argtypes = [vp, i, vp, sz]
    lib.iris_hip_gemm_fill.argtypes = [vp, vp, sz]
    return lib


def bf(x):
    return tl.bf16_to_f32(tl.to_bf16(x))


class Product:
    """One problem on the device; run(call) gives its output on fresh memory."""

    def __init__(self, M, N, K, epi, pad=0):
        rng = np.random.default_rng(M * 7 + N + K + epi)
        self.a, self.w = bf(rng.standard_normal((M, K), np.float32)), bf(rng.standard_normal((N, K), np.float32) * 0.03)
        self.vec = rng.standard_normal(N).astype(np.float32)
        nout = N // 2 if epi == EPI_SWIGLU else N
        self.shape = (N, M + pad) if epi == EPI_F32_T else (M, nout + pad)
        self.x0 = rng.standard_normal(self.shape).astype(np.float32)
        self.bf16 = epi in (EPI_BF16, EPI_SWIGLU)
        self.dims, self.epi, self.ldo, self.nout = (M, N, K), epi, self.shape[1], nout
        self.dev = [tl.Dev.of(tl.to_bf16(self.a)), tl.Dev.of(tl.to_bf16(self.w)), tl.Dev.of(self.vec)]

    def run(self, lib, call):
        M, N, K = self.dims
        o = tl.Dev.of(tl.to_bf16(self.x0) if self.bf16 else self.x0)
        vec = None if self.epi == EPI_SWIGLU else self.dev[2].ptr
        pr = tl.GemmProblem(self.dev[0].ptr, self.dev[1].ptr, o.ptr, vec, M, N, K, K, K, self.ldo, self.epi)
        assert call(ctypes.byref(pr)) == 0, lib.iris_hip_last_error()
        assert lib.iris_hip_sync() == 0
        r = o.get(np.uint16 if self.bf16 else np.float32, self.shape)
        o.close()
        return r

    def exact(self):
        M, N, K = self.dims
        y = self.a.astype(np.float64) @ self.w.astype(np.float64).T
        if self.epi == EPI_SWIGLU:
            g = np.concatenate([y[:, c * 64:c * 64 + 32] for c in range(N // 64)], 1)
            u = np.concatenate([y[:, c * 64 + 32:c * 64 + 64] for c in range(N // 64)], 1)
            return g / (1 + np.exp(-g)) * u
        if self.epi == EPI_F32_T:
            return (y + self.vec).T
        x0 = self.x0[:, :self.nout]
        return {EPI_GATED_ADD: x0 + self.vec * y, EPI_ADD: x0 + y + self.vec}.get(self.epi, y + self.vec)


@pytest.mark.parametrize("rows,M,N,K,splits", [(64, 1, 128, 64, 1), (64, 37, 192, 448, 1), (64, 65, 320, 1024, 3),
                                               (128, 128, 128, 192, 1), (128, 129, 448, 640, 2),
                                               (128, 300, 1344, 2560, 5)])
@pytest.mark.parametrize("epi", range(6))
def test_gemm_ring_bitwise(lib, rows, M, N, K, splits, epi):
    """Edges of tiles and of the ring (K of fewer steps than stages, of one
    more, long), every epilogue, an output row stride that takes the
    element-wise stores: the bits of the two-stage kernel at the same number of
    chunks, the columns past the output untouched, the float64 product within
    f32 summation (1e-5) or the bf16 rounding of the result (4e-3)."""
    ws = tl.Dev(WS)
    for pad in (0, 3):
        p = Product(M, N, K, epi, pad)
        got = p.run(lib, lambda pr: lib.iris_hip_gemm_ring(pr, 1, rows, splits, ws.ptr, WS))
        want = p.run(lib, lambda pr: lib.iris_hip_gemm_splitk(pr, splits, ws.ptr, WS))
        assert np.array_equal(got, want)
        y = p.exact()
        g = (tl.bf16_to_f32(got) if p.bf16 else got)[:, :y.shape[1]]
        assert tl.rel_l2(g, y) < (4e-3 if p.bf16 else 1e-5)
    ws.close()


@pytest.mark.parametrize("rows", [64, 128])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("shapes", [
    [(37, 192, 448, EPI_BF16), (128, 320, 448, EPI_F32)],
    [(1, 128, 64, EPI_F32), (130, 192, 1024, EPI_GATED_ADD), (64, 448, 320, EPI_ADD)],
    [(65, 64, 640, EPI_SWIGLU), (3, 321, 192, EPI_F32_T), (129, 130, 448, EPI_BF16), (64, 128, 2560, EPI_GATED_ADD)]])
def test_gemm_ring_several_problems(lib, shapes, splits, rows):
    """2 to 4 problems of different rows, columns, K and epilogues in one
    launch, whole and split over K (K of one step is not): each the bits of the
    two-stage kernel on that problem alone."""
    ps = [Product(*s) for s in shapes]
    ws, outs = tl.Dev(WS), []
    arr = (tl.GemmProblem * len(ps))()
    for i, p in enumerate(ps):
        M, N, K = p.dims
        outs.append(tl.Dev.of(tl.to_bf16(p.x0) if p.bf16 else p.x0))
        arr[i] = tl.GemmProblem(p.dev[0].ptr, p.dev[1].ptr, outs[i].ptr, None if p.epi == EPI_SWIGLU else p.dev[2].ptr,
                                M, N, K, K, K, p.ldo, p.epi)
    assert lib.iris_hip_gemm_ring(arr, len(ps), rows, splits, ws.ptr, WS) == 0, lib.iris_hip_last_error()
    assert lib.iris_hip_sync() == 0
    for p, o in zip(ps, outs):
        want = p.run(lib, lambda pr: lib.iris_hip_gemm_splitk(pr, splits, ws.ptr, WS))
        assert np.array_equal(o.get(np.uint16 if p.bf16 else np.float32, p.shape), want), p.dims
    ws.close()


@pytest.mark.parametrize("M,N,K,epi,ring", [(1, 6144, 2560, EPI_BF16, True), (37, 2560, 9728, EPI_GATED_ADD, True),
                                            (64, 19456, 2560, EPI_SWIGLU, True), (65, 3840, 3840, EPI_F32, True),
                                            (128, 2560, 4096, EPI_GATED_ADD, True),
                                            (129, 2560, 4096, EPI_GATED_ADD, False),
                                            (512, 6144, 2560, EPI_BF16, True), (256, 128, 3072, EPI_F32_T, False)])
def test_gemm_fill_few_rows(lib, M, N, K, epi, ring):
    """The text encoder's and the captions' products around the 128-row line
    of the rule, through iris_hip_gemm_fill: which kernel runs, repeatable,
    against float64."""
    ws = tl.Dev(WS)
    p = Product(M, N, K, epi)
    got = []
    for _ in range(2):
        assert lib.iris_hip_profile_enable(1) == 0
        got.append(p.run(lib, lambda pr: lib.iris_hip_gemm_fill(pr, ws.ptr, WS)))
        recs = (tl.KernelTime * 4)()
        n = lib.iris_hip_profile_read(recs, 4)
        assert lib.iris_hip_profile_enable(0) == 0
        assert any(b"ring" in r.kernel for r in recs[:n]) == ring, [r.kernel for r in recs[:n]]
    assert np.array_equal(got[0], got[1])
    y = p.exact()
    assert tl.rel_l2(tl.bf16_to_f32(got[0]) if p.bf16 else got[0], y) < (4e-3 if p.bf16 else 1e-5)
    ws.close()


def test_gemm_ring_repeat_bitwise(lib):
    """A long K over every stage of the ring, many blocks: 20 launches give the
    same bits (a load that is read before it is there would not)."""
    ws = tl.Dev(WS)
    p = Product(128, 19456, 2560, EPI_SWIGLU)
    for rows in (64, 128):
        first = p.run(lib, lambda pr: lib.iris_hip_gemm_ring(pr, 1, rows, 1, ws.ptr, WS))
        for _ in range(20):
            assert np.array_equal(first, p.run(lib, lambda pr: lib.iris_hip_gemm_ring(pr, 1, rows, 1, ws.ptr, WS)))
    ws.close()


def test_gemm_ring_rejects(lib):
    """Tile heights it does not have, a workspace too small for the chunks."""
    p = Product(64, 128, 512, EPI_F32)
    o = tl.Dev(64 * 128 * 4)
    pr = tl.GemmProblem(p.dev[0].ptr, p.dev[1].ptr, o.ptr, None, 64, 128, 512, 512, 512, 128, EPI_F32)
    assert lib.iris_hip_gemm_ring(ctypes.byref(pr), 1, 96, 1, None, 0) != 0
    assert lib.iris_hip_gemm_ring(ctypes.byref(pr), 1, 64, 2, o.ptr, 16) != 0
