"""Host side of the text encoder's downloads, on the CPU: iris_qwen3.c compiled
against stand-ins for the device calls. A download is a copy that happens only
when it is waited for, so one left behind by an exit is seen, and layers can be
made to fail."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import iris_testlib as tl

STUBS = r"""
#include "iris_hip.h"
#include "iris_synth.h"
#include <stdlib.h>
#include <string.h>
int fail_gemm_at = -1, gemms, fail_rows_at = -1, rows_calls, clobbered, no_pinned;
struct { void *dst; const void *src; size_t n; int on; } down[8];
void reset(void) { memset(down, 0, sizeof(down)); clobbered = no_pinned = 0; fail_gemm_at = fail_rows_at = -1; }
int pending(void) { int n = 0; for (int i = 0; i < 8; i++) n += down[i].on; return n; }
int iris_hip_init(int d) { (void)d; return 0; }
const char *iris_hip_last_error(void) { return "stub"; }
void *iris_hip_malloc(size_t n) { return calloc(1, n); }
void iris_hip_free(void *p) { free(p); }
void *iris_hip_host_malloc(size_t n) { return no_pinned ? NULL : calloc(1, n); }
void iris_hip_host_free(void *p) { free(p); }
int iris_hip_sync(void) { return 0; }
int iris_hip_memcpy_h2d(void *d, const void *s, size_t n) { memcpy(d, s, n); return 0; }
int iris_hip_memcpy_d2h(void *d, const void *s, size_t n) { memcpy(d, s, n); return 0; }
int iris_hip_download(void *d, const void *s, size_t n, int slot) {
    clobbered += down[slot].on;   /* over a copy that nobody waited for */
    down[slot].dst = d; down[slot].src = s; down[slot].n = n; down[slot].on = 1;
    return 0;
}
int iris_hip_download_wait(int slot) {
    if (!down[slot].on) return -1;
    memcpy(down[slot].dst, down[slot].src, down[slot].n);
    down[slot].on = 0;
    return 0;
}
static float *stream;   /* the residual stream: every gated product adds 1 to it */
static int width;
int iris_hip_embed_rows(float *x, const uint16_t *t, const int *ids, int S, int h, int vocab) {
    (void)t; (void)vocab;
    stream = x; width = h;
    for (int i = 0; i < S * h; i++) x[i] = ids[i / h] + (i % h) * 1e-3f;
    return 0;
}
int iris_hip_copy_rows(float *d, int ldd, const float *s, int lds, int rows, int cols) {
    if (rows_calls++ == fail_rows_at) return -1;
    for (int r = 0; r < rows; r++) memcpy(d + (size_t)r * ldd, s + (size_t)r * lds, cols * sizeof(float));
    return 0;
}
static int gemm(const iris_gemm_problem_t *p) {
    if (gemms++ == fail_gemm_at) return -1;
    if (p->out == stream)
        for (int i = 0; i < p->M * width; i++) stream[i] += 1.0f;
    return 0;
}
int iris_hip_gemm_fill(const iris_gemm_problem_t *p, float *ws, size_t n) { (void)ws; (void)n; return gemm(p); }
int iris_hip_gemm_fill_tail(const iris_gemm_problem_t *p, int k, float *ws, size_t n, const iris_row_tail_t *t) {
    (void)k; (void)ws; (void)n; (void)t;
    return gemm(p);
}
int iris_hip_rownorm(const iris_norm_args_t *a) { (void)a; return 0; }
int iris_hip_kv_prepare(const iris_qkprep_args_t *a) { (void)a; return 0; }
int iris_hip_attention(const iris_attn_args_t *a) { (void)a; return 0; }
"""
H, LAYERS, PER_LAYER = 256, 28, 4     # products of a layer: qkv, o, gate/up, down


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("qwen3_host")
    host, inc = os.path.join(tl.ROOT, "iris.c_amd", "host"), os.path.join(tl.ROOT, "include")
    (d / "stubs.c").write_text(STUBS)
    so = str(d / "libqwen3_host.so")
    subprocess.run(["gcc", "-O1", "-fPIC", "-shared", "-fopenmp", "-I", inc, "-o", so, str(d / "stubs.c")] +
                   [os.path.join(host, f) for f in ("iris_qwen3.c", "iris_synth.c", "iris_st.c")] + ["-lm"], check=True)
    lib = ctypes.CDLL(so)
    lib.qwen3_model_create_synthetic.restype = ctypes.c_void_p
    lib.qwen3_model_create_synthetic.argtypes = [ctypes.c_int] * 6 + [ctypes.c_uint64]
    lib.qwen3_forward.restype = ctypes.c_void_p
    lib.qwen3_forward.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_int]
    lib.qwen3_model_set_extraction_mode.argtypes = [ctypes.c_void_p, ctypes.c_int]
    lib.qwen3_model_free.argtypes = [ctypes.c_void_p]
    return lib


def set_int(lib, **kw):
    for k, v in kw.items():
        ctypes.c_int.in_dll(lib, k).value = v


def forward(lib, m, S):
    """One encode; the rows, or None where it failed."""
    set_int(lib, gemms=0, rows_calls=0)
    ids = np.arange(S, dtype=np.int32)
    p = lib.qwen3_forward(m, ids.ctypes.data, None, S)
    if not p:
        return None
    n = S * lib.qwen3_model_text_dim(ctypes.c_void_p(m))
    out = np.ctypeslib.as_array(ctypes.cast(p, tl.FP), shape=(n,)).reshape(S, -1).copy()
    ctypes.CDLL(None).free(ctypes.c_void_p(p))
    return out


def expect(S, layers):
    rows = np.arange(S, dtype=np.float32)[:, None] + np.arange(H, dtype=np.float32) * np.float32(1e-3)
    outs, x, at = {}, rows, 0
    for i in range(max(layers) + 1):
        x = x + np.float32(1) + np.float32(1)      # o and down
        outs[i] = x
    return np.concatenate([outs[i] for i in layers], 1)


@pytest.mark.parametrize("mode,layers", [(0, (8, 17, 26)), (1, (LAYERS - 2,))])
@pytest.mark.parametrize("S", [37, 512])
@pytest.mark.parametrize("no_pinned", [0, 1])
def test_rows(lib, S, mode, layers, no_pinned):
    """Both sides of the 1 MiB line, both modes: the extracted layers side by
    side, also where no pinned memory is to be had."""
    lib.reset()
    set_int(lib, no_pinned=no_pinned)
    m = lib.qwen3_model_create_synthetic(H, 64, 2, 1, LAYERS, 1024, 1)
    assert m
    lib.qwen3_model_set_extraction_mode(m, mode)
    got = forward(lib, m, S)
    assert lib.pending() == 0
    lib.qwen3_model_free(m)
    np.testing.assert_allclose(got, expect(S, layers), rtol=1e-6)


@pytest.mark.parametrize("gemm_at,rows_at", [(0, -1), (9 * PER_LAYER, -1), (20 * PER_LAYER + 3, -1),
                                             (27 * PER_LAYER - 1, -1), (-1, 0), (-1, 1), (-1, 2)])
def test_failed_layer_leaves_no_download(lib, gemm_at, rows_at):
    """A layer that fails before, between and after the extracted ones, and a
    failing copy of each: nothing is in flight when the call returns, and the
    next call's rows are right."""
    lib.reset()
    set_int(lib, fail_gemm_at=gemm_at, fail_rows_at=rows_at)
    m = lib.qwen3_model_create_synthetic(H, 64, 2, 1, LAYERS, 1024, 1)
    assert m
    assert forward(lib, m, 512) is None
    assert lib.pending() == 0
    set_int(lib, fail_gemm_at=-1, fail_rows_at=-1)
    got = forward(lib, m, 512)
    lib.qwen3_model_free(m)
    assert ctypes.c_int.in_dll(lib, "clobbered").value == 0
    np.testing.assert_allclose(got, expect(512, (8, 17, 26)), rtol=1e-6)
