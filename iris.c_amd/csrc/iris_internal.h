/* iris_internal.h - declarations shared by the HIP layer's translation units. */
#pragma once
#include "iris_dev.h"
#include "../../include/iris_hip.h"

hipStream_t iris_stream(void);
int iris_cu_count(void);   /* compute units of the bound device (0 before init) */
int iris_set_error(const char *fmt, ...);
int iris_check(hipError_t e, const char *what);
int iris_launch_check(const char *what);

/* Row pass after products split over K (iris_hip_gemm_fill_tail): the
 * partials of up to 4 problems (rows start[i] .. of problem i, chunks[i] of
 * them stride[i] apart) update the rows of x, then norm is taken of them. vec:
 * the gate per column (NULL: 1); w: Z-Image's RMSNorm of the product's row
 * with this weight and eps before the gate (NULL: none). */
typedef struct {
    const float *ws[4], *vec[4];
    long long stride[4];
    int chunks[4], start[4], n, cols, ldx, has_norm;
    float *x;
    const float *w;
    float eps;
    iris_norm_args_t norm;
} iris_reduce_rows_t;
int iris_reduce_rows(const iris_reduce_rows_t *r, int rows);

/* Per-launch timing for the library's profile (iris_hip_profile_enable):
 * while enabled and the stream is not being captured, each launch is
 * bracketed by two events on the library stream. begin returns the record
 * index, or -1 when nothing is recorded. */
int iris_prof_begin(const char *kernel, long long grid);
void iris_prof_end(int idx);

#define IRIS_LAUNCH(kernel, grid, block, smem, stream, ...)                                                   \
    do {                                                                                                      \
        const dim3 iris_grid_ = (grid);                                                                       \
        const int iris_prof_ = iris_prof_begin(#kernel, (long long)iris_grid_.x * iris_grid_.y * iris_grid_.z); \
        hipLaunchKernelGGL(kernel, iris_grid_, block, smem, stream, __VA_ARGS__);                            \
        iris_prof_end(iris_prof_);                                                                            \
    } while (0)
