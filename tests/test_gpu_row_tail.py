"""iris_hip_gemm_fill_tail: products split over K whose row passes run in the
reduce launch give the bits of the separate calls; where the products are not
split, or the rows are not the normalisation's, those calls run."""
import ctypes

import numpy as np
import pytest

import iris_testlib as tl

pytestmark = pytest.mark.gpu
EPI_F32, EPI_GATED_ADD = 0, 2
LN_MOD, RMS = 0, 2
WS = 64 << 20


class Tail(ctypes.Structure):
    _fields_ = [("x", ctypes.c_void_p), ("w", ctypes.c_void_p), ("gate", ctypes.c_void_p), ("eps", ctypes.c_float),
                ("norm", ctypes.c_void_p)]


@pytest.fixture(scope="module")
def lib():
    lib = tl.hip()
    vp, sz, i = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int
    lib.iris_hip_gemm_fill_tail.argtypes = [vp, i, vp, sz, vp]
    lib.iris_hip_gemm_fill_n.argtypes = [vp, i, vp, sz]
    lib.iris_hip_rms_gated_add.argtypes = [vp, vp, vp, vp, i, i, ctypes.c_float, i]
    return lib


def kernels(lib, call):
    assert lib.iris_hip_profile_enable(1) == 0
    assert call() == 0, lib.iris_hip_last_error()
    recs = (tl.KernelTime * 16)()
    n = lib.iris_hip_profile_read(recs, 16)
    assert lib.iris_hip_profile_enable(0) == 0
    return [r.kernel.decode() for r in recs[:n]]


@pytest.mark.parametrize("rows,N,K,kind,fused", [
    ((128,), 2560, 4096, "rms", True), ((512,), 2560, 9728, "rms", True), ((130,), 64, 2048, "rms", True),
    ((37,), 2560, 4096, "rms", False),       # few rows
    ((512, 256), 3072, 3072, "ln", True), ((100, 1, 30), 1028, 2048, "ln", True),
    ((1120,), 3840, 3840, "sand", True), ((96,), 3840, 10240, "sand", False), ((133,), 4096, 2048, "sand_last", True),
    ((200,), 4100, 2048, "rms", False),      # wider than a block's row
    ((4608,), 3072, 512, "rms", False),      # not split
])
def test_row_tail_bitwise(lib, rows, N, K, kind, fused):
    rng = np.random.default_rng(sum(rows) + N)
    M, sand = sum(rows), kind.startswith("sand")
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    x0, gate, w, scale, shift = f(M, N), f(N), f(N), f(N), f(N)
    A, ws, y = tl.Dev.of(tl.to_bf16(f(M, K))), tl.Dev(WS), tl.Dev(M * N * 4)
    W = [tl.Dev.of(tl.to_bf16(f(N, K) * 0.03)) for _ in rows]
    d = [tl.Dev.of(v) for v in (gate, w, scale, shift)]
    outs, names = [], []
    for tail_call in (True, True, False):
        x, a = tl.Dev.of(x0), tl.Dev.of(np.zeros((M, N), np.uint16))
        norm = tl.NormArgs(x.ptr, N, a.ptr, N, 1, M, N, LN_MOD if kind == "ln" else RMS, 1e-6, rows[0], 0,
                           d[3].ptr, d[2].ptr, d[1].ptr, d[2].ptr, d[3].ptr, d[0].ptr)
        probs, r0 = [], 0
        for m, wt in zip(rows, W):
            probs.append(tl.GemmProblem(A.ptr + r0 * K * 2, wt.ptr, (y if sand else x).ptr + r0 * N * 4,
                                        None if sand else d[0].ptr, m, N, K, K, K, N,
                                        EPI_F32 if sand else EPI_GATED_ADD))
            r0 += m
        arr = (tl.GemmProblem * len(probs))(*probs)
        has_norm = kind != "sand_last"
        if tail_call:
            t = Tail(x.ptr if sand else None, d[1].ptr if sand else None, d[0].ptr if sand else None, 1e-5,
                     ctypes.cast(ctypes.pointer(norm), ctypes.c_void_p) if has_norm else None)
            names.append(kernels(lib, lambda: lib.iris_hip_gemm_fill_tail(arr, len(probs), ws.ptr, WS, ctypes.byref(t))))
        else:
            assert lib.iris_hip_gemm_fill_n(arr, len(probs), ws.ptr, WS) == 0
            if sand:
                assert lib.iris_hip_rms_gated_add(x.ptr, y.ptr, d[1].ptr, d[0].ptr, M, N, 1e-5, 0) == 0
            if has_norm:
                assert lib.iris_hip_rownorm(ctypes.byref(norm)) == 0
            assert lib.iris_hip_sync() == 0
        outs.append((x.get(np.float32, (M, N)), a.get(np.uint16, (M, N))))
    assert any("reduce_rows" in n for n in names[0]) == fused, names[0]
    for got in outs[:2]:
        assert np.array_equal(got[0], outs[2][0]) and np.array_equal(got[1], outs[2][1])
    assert not np.array_equal(outs[0][0], x0)


def test_row_tail_other_rows(lib):
    """A normalisation of other rows than the products update: the separate calls."""
    M, N, K = 192, 512, 4096
    rng = np.random.default_rng(3)
    A, W = (tl.Dev.of(tl.to_bf16(rng.standard_normal((r, K)).astype(np.float32))) for r in (M, N))
    x, a, w, ws = tl.Dev.of(np.ones((M, N), np.float32)), tl.Dev(M * N * 2), tl.Dev.of(np.ones(N, np.float32)), tl.Dev(WS)
    norm = tl.NormArgs(x.ptr + N * 4, N, a.ptr, N, 1, M - 1, N, RMS, 1e-6, M, 0, None, None, w.ptr)
    pr = tl.GemmProblem(A.ptr, W.ptr, x.ptr, None, M, N, K, K, K, N, EPI_GATED_ADD)
    t = Tail(None, None, None, 0.0, ctypes.cast(ctypes.pointer(norm), ctypes.c_void_p))
    names = kernels(lib, lambda: lib.iris_hip_gemm_fill_tail(ctypes.byref(pr), 1, ws.ptr, WS, ctypes.byref(t)))
    assert not any("reduce_rows" in n for n in names) and any("rownorm" in n for n in names), names
