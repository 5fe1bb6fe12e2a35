// mmq_launch.h -- host functions that the MMQ sources share: the few-column GEMM
// (mmq_few.hip), the f16 prefill GEMM (mmq_f16.hip) and the parts of mmq.hip that
// api.hip's routes use.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "qmm_device.h"

// quantize_q8_1.hip: hip_qmm_quantize_q8_1_planar with the header bits of `keep` only
// (q8_1_header_mask of the weights' type for an op's own copy)
int qmm_quantize_planar(const float *x, int64_t K, int64_t ncols, int64_t x_col_stride, int8_t *qs, void *ds,
                        uint32_t keep, hipStream_t s);

// mmq.hip: whether the few-column kernel takes this shape (given aligned operands),
// the kernel of hip_qmm_mmq on aligned operands (a HIP_QMM_KERNEL_ value, K % 256 ==
// 0), the weight checks of its dispatch, and the sum of K-split partials
bool few_cols_type(int type, int64_t K, int64_t nrows, int64_t ncols);
int mmq_kernel_of(int type, int64_t K, int64_t nrows, int64_t ncols);
int mmq_check_weights(int type, const void *w, int64_t K, int64_t row_stride);
int mmq_add_partials(const float *partial, int split, int64_t nrows, int64_t ncols, float *dst, int64_t dst_col_stride,
                     hipStream_t s);

// mmq_few.hip: the GEMM for at most 32 columns: whether it takes these weight rows,
// its K split, and whether its 16-row workgroups that hold all of K run
bool mmq_few_takes(int type, int64_t K, const void *w, int64_t row_stride);
int mmq_few_split_k(int64_t K, int64_t nrows);
bool mmq_few_whole_k(int type, int64_t K, int64_t nrows, int64_t ncols);
int mmq_few_launch(int type, const void *w, int64_t K, int64_t nrows, int64_t row_stride, const int8_t *yqs,
                   const void *yds, int64_t ncols, float *dst, int64_t dst_col_stride, int split, float *partial,
                   const qmm::MmqGlu &glu, hipStream_t s);

// mmq_f16.hip: the large-grid Q4_K / Q5_K / Q6_K GEMM on f16 matrix cores
struct MmqF16Plan {
    bool use, wide;
    int split;
};
MmqF16Plan mmq_f16_plan(int type, int64_t K, int64_t nrows, int64_t ncols, bool glu);
size_t mmq_f16_panel_bytes(int64_t K, int64_t ncols);
int mmq_f16_quantize(const float *x, int64_t K, int64_t ncols, int64_t x_col_stride, void *panels, hipStream_t s);
int mmq_f16_launch(int type, bool wide, const void *w, int64_t K, int64_t nrows, int64_t row_stride,
                   const void *panels, int64_t ncols, float *dst, int64_t dst_col_stride, float *partial, int split,
                   const qmm::MmqGlu &glu, hipStream_t s);
