// api.hip -- op-level entry points of libggml_hip_qmm.so: workspace sizing and
// the MUL_MAT dispatch (GEMV for <= 8 columns, MMQ above, and the few-column
// Q4_K GEMM for 5-8 columns of large matrices), mirroring
// ggml_cuda_mul_mat's choice between MMVQ and MMQ
// (src/ggml/cuda/mulmat.zig:576-639; mmvq.zig:128-173; mmq.zig:865-917).
#include "../../include/ggml_hip_qmm.h"
#include "mmq_launch.h"
#include "qmm_device.h"

#include <atomic>
#include <mutex>

using namespace qmm;

extern "C" int hip_qmm_mmq(int type, const void *w, int64_t K, int64_t nrows, int64_t row_stride,
                           const int8_t *y_qs, const void *y_ds, int64_t ncols, float *dst,
                           int64_t dst_col_stride, void *workspace, size_t workspace_size, void *stream);
extern "C" size_t hip_qmm_mmq_workspace_size(int type, int64_t K, int64_t nrows, int64_t ncols);

// gemv.hip: 2-4 f32 columns (or twice the kernel's columns as two grid rows)
// through the quantize-in-GEMV kernel, or hipErrorNotSupported for shapes it
// does not take.
int qmm_mul_mat_fx_cols(int type, const void *w, int64_t K, int64_t nrows, int64_t row_stride, const float *x,
                        int64_t ncols, int64_t x_col_stride, float *dst, int64_t dst_col_stride, void *stream);
// gemv.hip: 2-8 f32 columns of a small matrix through the one-column kernel
// (grid y = column), or hipErrorNotSupported where it does not win.
int qmm_mul_mat_fx_percol(int type, const void *w, int64_t K, int64_t nrows, int64_t row_stride, const float *x,
                          int64_t ncols, int64_t x_col_stride, float *dst, int64_t dst_col_stride, void *stream);

namespace {
size_t q8_1_bytes(int64_t K, int64_t ncols) {
    const int64_t Kp = pad_k(K);
    return (size_t)(ncols * Kp) + (size_t)(ncols * (Kp / QK8)) * 4u;  // qs plane, then ds plane
}
size_t align256(size_t v) { return (v + 255) / 256 * 256; }

// Whether 2-8 columns go to the MMQ dispatch (the few-column kernel,
// mmq_few.hip) rather than the GEMV.  The GEMV's time grows with the columns
// (each wave re-reads every column's activation slice), the few-column
// kernel's hardly does; the few-column kernel is at its best on long rows (K
// >= 8192, where the GEMV's per-wave activation slices are longest) and on
// >= 12288 rows (an unsplit grid, two K halves per workgroup), while on
// 6144-8192 rows of K = 4096 its split grid loses to the GEMV.  Crossovers
// measured on the op (hip_qmm_mul_mat, us, GEMV path against few-column):
//   - Q4_K: from 5 columns at K >= 8192 on >= 4096 rows (4096x14336: 19.6
//     against 16.4) and on >= 12288 rows (14336x4096 at 5: 14.8 against 14.0;
//     12288x4096 13.9 against 13.4), from 6 at K >= 8192 on >= 2048 rows, from
//     7 on >= 6144 rows; the GEMV stays ahead on smaller matrices (4096x4096 at
//     8 columns: 9.7 against 11.1);
//   - Q5_K: from 4 columns on >= 24M weights of long rows or >= 12288 rows
//     (14336x4096 at 4: 18.0 against 16.0), from 6 on other >= 24M weights
//     (6144x4096 at 4 / 5 / 6: 10.5 / 12.9 / 13.9 against 13.5 / 13.5 / 13.6),
//     8 columns from 12M (4096x4096 11.8 against 11.5);
//   - Q8_0: from 4 columns on >= 24M weights of long rows or >= 12288 rows
//     (4096x14336 at 4: 24.0 against 21.1), 8 columns from 12M on long rows;
//     6144x4096 keeps the GEMV (12.4-14.4 against 14.8-15.1 at 4-8 columns);
//   - Q4_0: on >= 24M weights, from 4 columns on >= 12288 rows (14336x4096:
//     17.9 against 16.5) and on long rows of <= 2048 (2048x14336: 15.2 against
//     14.9), from 5 on other long rows (4096x14336 at 4 / 5: 17.3 / 19.9
//     against 17.9 / 17.9); 6144x4096 keeps the GEMV (9.7-13.2 against
//     13.4-13.7); 8 columns from 12M on long rows;
//   - IQ4_XS: from 5 columns on >= 24M weights of long rows or >= 12288 rows
//     (14336x4096: 18.5 against 18.0; 2048x14336: 16.6 against 15.3), 8
//     columns from 12M on long rows;
//   - Q6_K (two 16-deep sub-blocks per MFMA up to 8 columns): on >= 24M
//     weights from 4 columns on long rows or >= 12288 rows (4096x14336 at 4 /
//     8: 24.7 / 27.9 against 22.4 / 22.3; 14336x4096 at 4: 24.3 against 21.1;
//     2048x14336 at 4: 20.5 against 17.6), from 5 on >= 8192 rows (8192x4096
//     at 4 / 5: 15.4 / 17.4 against 16.7 / 16.7), from 6 on the rest
//     (6144x4096 at 5 / 6: 14.7 / 16.6 against 16.1 / 16.2); 7 columns from
//     12M (4096x4096 13.0 against 12.7), 8 columns on rows of K >= 8192 at <=
//     2048 rows; the GEMV stays ahead on 4096x4096 at 5, 6 and 8 columns (10.7
//     / 12.3 / 11.3 against 12.7 / 12.8 / 12.9) and on 1024x4096.
//   At 3 columns the one-launch GEMV with the quantization fused in stays
//   (Q5_K 14336x4096 16.5 against 15.9; Q8_0 4096x14336 22.4 against 20.9).
bool few_cols_wins(int type, int64_t K, int64_t nrows, int64_t ncols) {
    if (K % 256 != 0 || ncols > 8 || !few_cols_type(type, K, nrows, ncols)) return false;
    const int64_t elems = nrows * K;
    const bool large = elems >= ((int64_t)24 << 20), mid = elems >= ((int64_t)12 << 20), long_rows = K >= 8192;
    const bool strong = large && (long_rows || nrows >= 12288);  // the few-column kernel's best grids
    switch (type) {
    case TYPE_Q4_K:
        if (long_rows && nrows >= 4096) return ncols >= 5;
        if (nrows >= 12288) return ncols >= 5;
        if (long_rows && nrows >= 2048) return ncols >= 6;
        if (nrows >= 6144) return ncols >= 7;
        return false;
    case TYPE_Q5_K: return (strong && ncols >= 4) || (large && ncols >= 6) || (mid && ncols == 8);
    case TYPE_Q8_0: return (strong && ncols >= 4) || (mid && long_rows && ncols == 8);
    case TYPE_Q4_0:
        return (strong && ncols >= (long_rows && nrows > 2048 && nrows < 12288 ? 5 : 4)) ||
               (mid && long_rows && ncols == 8);
    case TYPE_IQ4_XS: return (strong && ncols >= 5) || (mid && long_rows && ncols == 8);
    case TYPE_Q6_K:
        return (strong && ncols >= 4) || (large && nrows >= 8192 && ncols >= 5) || (large && ncols >= 6) ||
               (mid && ncols == 7) || (mid && long_rows && nrows <= 2048 && ncols == 8);
    default: return false;
    }
}

// Whether 3-8 columns go to the few-column kernel beyond few_cols_wins because its
// 16-row workgroups hold all of K there (mmq_few_whole_k): one launch after the
// quantizer and no partials, so the workspace needs nothing beyond the Q8_1 planes
// and hip_qmm_mul_mat_uses_mmq (which sizes for partials) does not report it.  The
// least columns at which quantizer + GEMM is ahead of the GEMV, by rows and K, from
// graph-timed calls (GEMV -> few, us): Q4_K 4096x4096 at 5 / 6 / 8 7.6 -> 7.4, 8.9 ->
// 7.4, 9.5 -> 7.4 (at 4 6.9 / 7.3), 6144x2048 at 3 7.3 -> 6.8, 2048x4096 at 7 8.0 ->
// 7.1; rows below 2048 keep the GEMV (1024x4096 at 8 5.3 / 6.9; Q4_0
// 2048x8192 at 6 10.3 / 10.9), and so do the shapes
// of hip_qmm_mul_mat_per_column and, on at most 4096 rows and K, the columns that one
// launch of the quantize-in-GEMV kernel takes: their results are the one-column
// kernel's.
bool few_whole_wins(int type, int64_t K, int64_t nrows, int64_t ncols) {
    if (K % 256 != 0 || ncols < 3 || ncols > 8 || nrows < 2048 || !few_cols_type(type, K, nrows, ncols) ||
        !mmq_few_whole_k(type, K, nrows, ncols) || hip_qmm_mul_mat_per_column(type, K, nrows, ncols))
        return false;
    if (nrows <= 4096 && K <= 4096 && ncols <= (type == TYPE_Q8_0 ? 8 : type == TYPE_IQ4_XS ? 6 : 4)) return false;
    //                          K < 4096, K < 8192, more
    static constexpr int8_t least[6][3][3] = {
        // rows from 2048   4096         6144
        {{9, 7, 6}, {5, 6, 4}, {3, 5, 4}},  // Q4_K
        {{9, 5, 5}, {4, 5, 4}, {4, 5, 4}},  // Q5_K
        {{9, 5, 5}, {5, 5, 4}, {4, 4, 4}},  // Q6_K
        {{9, 9, 5}, {5, 5, 4}, {5, 5, 4}},  // Q8_0
        {{9, 7, 7}, {8, 7, 5}, {8, 8, 5}},  // Q4_0
        {{9, 6, 6}, {6, 6, 5}, {6, 7, 5}},  // IQ4_XS
    };
    const int t = type == TYPE_Q4_K ? 0 : type == TYPE_Q5_K ? 1 : type == TYPE_Q6_K ? 2 : type == TYPE_Q8_0 ? 3
                : type == TYPE_Q4_0 ? 4 : 5;
    return ncols >= least[t][nrows >= 6144 ? 2 : nrows >= 4096 ? 1 : 0][K >= 8192 ? 2 : K >= 4096 ? 1 : 0];
}

// Shape-only (the workspace sizing): the MMQ dispatch takes these columns.
bool use_mmq(int type, int64_t K, int64_t nrows, int64_t ncols) {
    return K % 256 == 0 && (ncols > 8 || few_cols_wins(type, K, nrows, ncols));
}

// At the call: up to 8 columns go to the few-column kernel only where it takes
// the rows (16-byte-aligned rows for the 2- and 8-byte-aligned types); the
// MMQ tile would be slower than the GEMV there.
bool use_mmq_rows(int type, int64_t K, int64_t nrows, int64_t ncols, const void *w, int64_t row_stride) {
    return (use_mmq(type, K, nrows, ncols) || few_whole_wins(type, K, nrows, ncols)) &&
           (ncols > 8 || mmq_few_takes(type, K, w, row_stride));
}

// Whether gate/up/GLU over ncols columns runs the fused MMQ: where each
// product alone would run the MMQ tile kernel (not the GEMV and not the
// few-column kernel; the reference's shouldFuseMulMatQ likewise leaves the
// matmuls its few-row MMQ and MMVQ take, src/ggml/cuda/mulmat.zig:560-567).
bool glu_fuses_mmq(int type, int64_t K, int64_t nrows, int64_t ncols) {
    return ncols >= 2 && use_mmq(type, K, nrows, ncols) && !few_cols_type(type, K, nrows, ncols);
}

// Whether gate/up/GLU over ncols columns runs the few-column kernel on both
// weights with the GLU in its epilogue (one quantizer and one launch) rather
// than two products and the GLU kernel (two quantizers, two GEMVs or few-column
// GEMMs with their K-split reductions, one GLU).  Both weights' rows give the
// grid twice the workgroups, so it needs no K split from 4096 rows on.  Measured
// (whole call, us, graph-timed, unfused -> fused): Q4_K 14336x4096 at 2 / 4 / 9 /
// 16 / 32 columns 25.1 -> 21.3, 27.9 -> 20.8, 31.3 -> 22.1, 32.6 -> 22.6, 43.2 ->
// 30.1; 8192x4096 at 4 / 16 25.7 -> 13.9, 28.7 -> 14.5; 4096x4096 at 4 / 8 16.1 ->
// 12.7, 21.2 -> 12.7; Q5_K 14336x4096 at 13 34.6 -> 25.6; Q6_K at 4 44.1 -> 33.3;
// Q8_0 at 4 39.1 -> 30.1; Q4_0 at 8 34.8 -> 25.2; IQ4_XS at 8 38.4 -> 27.6.  The
// unfused route stays where it measured level or faster: few columns of small or
// long-row matrices, whose one-launch GEMVs have no quantizer (Q4_K 4096x4096 at
// 2 11.7 against 13.0; Q6_K 5120x8192 at 2 32.5 / 34.0; Q4_0 4096x8192 at 4 22.0 /
// 24.6; IQ4_XS 14336x14336 at 2 70.2 / 78.5, 5120x8192 at 3 26.3 / 26.6), and
// below 4096 rows or 12M weights, where the unsplit grid is too small (Q4_K
// 1024x8192 at 4 16.4 against 19.6).
bool glu_few(int type, int64_t K, int64_t nrows, int64_t ncols) {
    if (K % 256 != 0 || nrows < 4096 || nrows * K < ((int64_t)12 << 20) || !few_cols_type(type, K, nrows, ncols))
        return false;
    if (nrows < 5120) return ncols >= (type == TYPE_Q4_0 || type == TYPE_IQ4_XS ? 8 : 4);
    switch (type) {
    case TYPE_Q6_K:
    case TYPE_Q4_0: return ncols >= 3;
    case TYPE_IQ4_XS: return ncols >= 4;
    default: return ncols >= 2;
    }
}

// The unfused gate/up/GLU's workspace: the gate and up products, then
// hip_qmm_mul_mat's own workspace.
size_t glu_unfused_bytes(int type, int64_t K, int64_t nrows, int64_t ncols) {
    return align256((size_t)2 * (size_t)nrows * (size_t)ncols * sizeof(float)) +
           hip_qmm_mul_mat_workspace_size(type, K, nrows, ncols);
}
// Workspace of the f16 route: the panels, then the K-split partials.
size_t f16_bytes(const MmqF16Plan &pl, int64_t K, int64_t nrows, int64_t ncols) {
    const size_t partials = pl.split > 1 ? (size_t)pl.split * (size_t)nrows * (size_t)ncols * sizeof(float) : 0;
    return align256(mmq_f16_panel_bytes(K, ncols)) + partials;
}

// The f16 route of a product (w_gate null) or of gate/up/GLU, or
// hipErrorNotSupported where it does not apply: a shape that the plan leaves to
// the int8 kernels, operands they would check further, or a workspace that does
// not hold the panels (they are twice the Q8_1 planes, so a caller's workspace of
// the required size keeps the int8 kernels).
int f16_route(int type, const void *w, const void *w_gate, int64_t K, int64_t nrows, int64_t row_stride,
              const float *x, int64_t ncols, int64_t x_col_stride, int glu_op, float glu_alpha, float glu_limit,
              float *dst, int64_t dst_col_stride, void *workspace, size_t workspace_size, void *stream) {
    const MmqF16Plan pl = mmq_f16_plan(type, K, nrows, ncols, w_gate != nullptr);
    if (!pl.use || !w || (uintptr_t)x % 16 || x_col_stride % 4 || dst_col_stride < nrows ||
        mmq_check_weights(type, w, K, row_stride) || (w_gate && mmq_check_weights(type, w_gate, K, row_stride)) ||
        workspace_size < f16_bytes(pl, K, nrows, ncols))
        return (int)hipErrorNotSupported;
    hipStream_t s = (hipStream_t)stream;
    float *partial = pl.split > 1 ? (float *)((uint8_t *)workspace + align256(mmq_f16_panel_bytes(K, ncols))) : nullptr;
    const MmqGlu glu{(const uint8_t *)w_gate, glu_op, glu_alpha, glu_limit};
    if (int e = mmq_f16_quantize(x, K, ncols, x_col_stride, workspace, s)) return e;
    if (int e = mmq_f16_launch(type, pl.wide, w, K, nrows, row_stride, workspace, ncols, dst, dst_col_stride, partial,
                               pl.split, glu, s))
        return e;
    return partial ? mmq_add_partials(partial, pl.split, nrows, ncols, dst, dst_col_stride, s) : 0;
}
}  // namespace

extern "C" int hip_qmm_version(void) { return (0 << 16) | 1; }

extern "C" int64_t hip_qmm_row_padding(void) { return ROW_PAD; }

extern "C" size_t hip_qmm_mul_mat_workspace_size(int type, int64_t K, int64_t nrows, int64_t ncols) {
    if (K <= 0 || ncols <= 0) return 0;
    size_t n = q8_1_bytes(K, ncols);
    if (nrows > 0 && use_mmq(type, K, nrows, ncols)) n = align256(n) + hip_qmm_mmq_workspace_size(type, K, nrows, ncols);
    return n;
}

extern "C" size_t hip_qmm_mul_mat_workspace_preferred(int type, int64_t K, int64_t nrows, int64_t ncols) {
    const size_t need = hip_qmm_mul_mat_workspace_size(type, K, nrows, ncols);
    const MmqF16Plan pl = mmq_f16_plan(type, K, nrows, ncols, false);
    const size_t f16 = pl.use ? f16_bytes(pl, K, nrows, ncols) : 0;
    return f16 > need ? f16 : need;
}

extern "C" int hip_qmm_mul_mat_uses_mmq(int type, int64_t K, int64_t nrows, int64_t ncols) {
    return K > 0 && nrows > 0 && ncols > 1 && use_mmq(type, K, nrows, ncols) ? 1 : 0;
}

extern "C" int hip_qmm_kernel(int op, int type, int64_t K, int64_t nrows, int64_t ncols) {
    const bool legacy = type == TYPE_Q8_0 || type == TYPE_Q4_0;
    const bool known = legacy || type == TYPE_Q4_K || type == TYPE_Q5_K || type == TYPE_Q6_K || type == TYPE_IQ4_XS;
    if (!known || K <= 0 || nrows <= 0 || ncols <= 0 || K % (legacy ? QK8 : QK_K)) return -1;
    if (op == HIP_QMM_OP_MMQ) return K % QK_K ? -1 : mmq_kernel_of(type, K, nrows, ncols);
    if (op == HIP_QMM_OP_MUL_MAT) {
        if (ncols == 1 || K % QK_K || !(use_mmq(type, K, nrows, ncols) || few_whole_wins(type, K, nrows, ncols)))
            return HIP_QMM_KERNEL_GEMV;
        return ncols > 8 && mmq_f16_plan(type, K, nrows, ncols, false).use ? HIP_QMM_KERNEL_F16
                                                                           : mmq_kernel_of(type, K, nrows, ncols);
    }
    if (op == HIP_QMM_OP_MUL_MAT_GLU) {
        if (ncols == 1 && K <= 32768) return HIP_QMM_KERNEL_GEMV;
        if (glu_fuses_mmq(type, K, nrows, ncols))
            return mmq_f16_plan(type, K, nrows, ncols, true).use ? HIP_QMM_KERNEL_F16 : HIP_QMM_KERNEL_TILE;
        return glu_few(type, K, nrows, ncols) ? HIP_QMM_KERNEL_FEW : HIP_QMM_KERNEL_UNFUSED;
    }
    return -1;
}

extern "C" int hip_qmm_mul_mat(int type, const void *w, int64_t K, int64_t nrows, int64_t row_stride,
                               const float *x, int64_t ncols, int64_t x_col_stride, float *dst,
                               int64_t dst_col_stride, void *workspace, size_t workspace_size, void *stream) {
    if (ncols <= 0 || !workspace || !x || !dst) return (int)hipErrorInvalidValue;
    // columns must not overlap, whichever kernel the shape picks
    if (ncols > 1 && (dst_col_stride < nrows || x_col_stride < K)) return (int)hipErrorInvalidValue;
    if (workspace_size < hip_qmm_mul_mat_workspace_size(type, K, nrows, ncols)) return (int)hipErrorInvalidValue;
    if ((uintptr_t)workspace % 16) return (int)hipErrorInvalidValue;
    // One column: the quantization runs inside the GEMV (one launch), which
    // measured faster than quantizer + GEMV on every decode shape (e.g. Q4_K
    // 1024x4096 3.3 vs 5.1 us, 14336x4096 8.5 vs 9.6 us, Q6_K 4096x14336 with
    // K shares 14.9 vs 15.6 us).
    if (ncols == 1 && K <= 32768 && K % QK8 == 0 && (uintptr_t)x % 16 == 0)
        return hip_qmm_mul_mat_vec_f32(type, w, K, nrows, row_stride, x, dst, stream);
    if (ncols >= 2 && ncols <= 8 && !use_mmq_rows(type, K, nrows, ncols, w, row_stride)) {
        const int e = qmm_mul_mat_fx_percol(type, w, K, nrows, row_stride, x, ncols, x_col_stride, dst,
                                            dst_col_stride, stream);
        if (e != (int)hipErrorNotSupported) return e;
    }
    if (ncols >= 2 && ncols <= 8 && !use_mmq_rows(type, K, nrows, ncols, w, row_stride)) {
        const int e = qmm_mul_mat_fx_cols(type, w, K, nrows, row_stride, x, ncols, x_col_stride, dst, dst_col_stride,
                                          stream);
        if (e != (int)hipErrorNotSupported) return e;
    }
    if (ncols > 8) {
        const int e = f16_route(type, w, nullptr, K, nrows, row_stride, x, ncols, x_col_stride, 0, 0.0f, 0.0f, dst,
                                dst_col_stride, workspace, workspace_size, stream);
        if (e != (int)hipErrorNotSupported) return e;
    }
    const int64_t Kp = pad_k(K);
    int8_t *qs = (int8_t *)workspace;
    void *ds = (uint8_t *)workspace + ncols * Kp;
    if (int e = qmm_quantize_planar(x, K, ncols, x_col_stride, qs, ds, q8_1_header_mask(type), (hipStream_t)stream))
        return e;
    if (ncols <= 8 && !use_mmq_rows(type, K, nrows, ncols, w, row_stride))
        return hip_qmm_mul_mat_vec(type, w, K, nrows, row_stride, qs, ds, ncols, dst, dst_col_stride, stream);
    if (K % 256 == 0) {
        // few-column calls without partials may end before the aligned offset
        const size_t off = align256(q8_1_bytes(K, ncols));
        const bool rest = workspace_size > off;
        return hip_qmm_mmq(type, w, K, nrows, row_stride, qs, ds, ncols, dst, dst_col_stride,
                           rest ? (uint8_t *)workspace + off : nullptr, rest ? workspace_size - off : 0, stream);
    }
    // Q8_0 / Q4_0 rows whose length is not a multiple of 256 (the MMQ K-step):
    // GEMV over column groups of 8.
    for (int64_t c0 = 0; c0 < ncols; c0 += 8) {
        const int64_t nc = ncols - c0 < 8 ? ncols - c0 : 8;
        const uint8_t *dsb = (const uint8_t *)ds + c0 * (Kp / QK8) * 4;
        if (int e = hip_qmm_mul_mat_vec(type, w, K, nrows, row_stride, qs + c0 * Kp, dsb, nc,
                                        dst + c0 * dst_col_stride, dst_col_stride, stream))
            return e;
    }
    return 0;
}

extern "C" int hip_qmm_mul_mat_glu_fused(int type, int64_t K, int64_t nrows, int64_t ncols) {
    return K > 0 && nrows > 0 && (glu_fuses_mmq(type, K, nrows, ncols) || (ncols > 8 && glu_few(type, K, nrows, ncols)))
               ? 1
               : 0;
}

extern "C" size_t hip_qmm_mul_mat_glu_workspace_size(int type, int64_t K, int64_t nrows, int64_t ncols) {
    if (K <= 0 || nrows <= 0 || ncols <= 0) return 0;
    if (glu_fuses_mmq(type, K, nrows, ncols)) return q8_1_bytes(K, ncols);
    return glu_unfused_bytes(type, K, nrows, ncols);  // one column: only used when the fused GEMV cannot run
}

extern "C" size_t hip_qmm_mul_mat_glu_workspace_preferred(int type, int64_t K, int64_t nrows, int64_t ncols) {
    const size_t need = hip_qmm_mul_mat_glu_workspace_size(type, K, nrows, ncols);
    if (K <= 0 || nrows <= 0 || ncols <= 0 || !glu_fuses_mmq(type, K, nrows, ncols)) return need;
    const MmqF16Plan pl = mmq_f16_plan(type, K, nrows, ncols, true);
    const size_t f16 = pl.use ? f16_bytes(pl, K, nrows, ncols) : 0;
    return f16 > need ? f16 : need;
}

extern "C" int hip_qmm_mul_mat_glu(int type, const void *w, const void *w_gate, int64_t K, int64_t nrows,
                                   int64_t row_stride, const float *x, int64_t ncols, int64_t x_col_stride,
                                   int glu_op, float glu_alpha, float glu_limit, float *dst, int64_t dst_col_stride,
                                   void *workspace, size_t workspace_size, void *stream) {
    if (ncols <= 0 || nrows <= 0 || K <= 0 || !w || !w_gate || !x || !dst || !glu_op_valid(glu_op))
        return (int)hipErrorInvalidValue;
    if (ncols > 1 && (dst_col_stride < nrows || x_col_stride < K)) return (int)hipErrorInvalidValue;
    if (ncols == 1 && K <= 32768 && K % QK8 == 0 && (uintptr_t)x % 16 == 0)
        return hip_qmm_mul_mat_vec_fused(type, w, w_gate, K, nrows, row_stride, x, nullptr, nullptr, glu_op,
                                         glu_alpha, glu_limit, dst, stream);
    if (!workspace || (uintptr_t)workspace % 256 ||
        workspace_size < hip_qmm_mul_mat_glu_workspace_size(type, K, nrows, ncols))
        return (int)hipErrorInvalidValue;
    if (glu_fuses_mmq(type, K, nrows, ncols)) {
        const int f16 = f16_route(type, w, w_gate, K, nrows, row_stride, x, ncols, x_col_stride, glu_op, glu_alpha,
                                  glu_limit, dst, dst_col_stride, workspace, workspace_size, stream);
        if (f16 != (int)hipErrorNotSupported) return f16;
        const int64_t Kp = pad_k(K);
        int8_t *qs = (int8_t *)workspace;
        void *ds = (uint8_t *)workspace + ncols * Kp;
        if (int e = qmm_quantize_planar(x, K, ncols, x_col_stride, qs, ds, q8_1_header_mask(type), (hipStream_t)stream))
            return e;
        return hip_qmm_mmq_glu(type, w, w_gate, K, nrows, row_stride, qs, ds, ncols, glu_op, glu_alpha, glu_limit,
                               dst, dst_col_stride, stream);
    }
    if (glu_few(type, K, nrows, ncols) && mmq_few_takes(type, K, w, row_stride) &&
        mmq_few_takes(type, K, w_gate, row_stride) && !mmq_check_weights(type, w, K, row_stride) &&
        !mmq_check_weights(type, w_gate, K, row_stride) && dst_col_stride >= nrows) {
        const int64_t Kp = pad_k(K);
        int8_t *qs = (int8_t *)workspace;
        void *ds = (uint8_t *)workspace + ncols * Kp;
        if (int e = qmm_quantize_planar(x, K, ncols, x_col_stride, qs, ds, q8_1_header_mask(type), (hipStream_t)stream))
            return e;
        const MmqGlu glu{(const uint8_t *)w_gate, glu_op, glu_alpha, glu_limit};
        return mmq_few_launch(type, w, K, nrows, row_stride, qs, ds, ncols, dst, dst_col_stride, 1, nullptr, glu,
                              (hipStream_t)stream);
    }
    float *g = (float *)workspace, *u = g + nrows * ncols;
    const size_t off = align256((size_t)2 * (size_t)nrows * (size_t)ncols * sizeof(float));
    void *rest = (uint8_t *)workspace + off;
    if (int e = hip_qmm_mul_mat(type, w_gate, K, nrows, row_stride, x, ncols, x_col_stride, g, nrows, rest,
                                workspace_size - off, stream))
        return e;
    if (int e = hip_qmm_mul_mat(type, w, K, nrows, row_stride, x, ncols, x_col_stride, u, nrows, rest,
                                workspace_size - off, stream))
        return e;
    return hip_qmm_glu_f32(glu_op, glu_alpha, glu_limit, nrows, ncols, g, nrows, u, nrows, dst, dst_col_stride,
                           stream);
}

// ---------------------------------------------------------------- allocation-free MUL_MAT
//
// For callers that cannot allocate (code under HIP graph capture, serving
// loops, harnesses that forbid hipMalloc): hip_qmm_mul_mat with its workspace
// taken from a fixed device array instead of an argument.  Each device holds
// its own copy of the array for the life of the process.  Its device address
// is looked up once per device, with that device current, and kept; host
// code never passes the array's name (a host-side stand-in) to a kernel.
// Every call on one device shares its array: calls that overlap on one GPU
// race, and a call leaves its scratch contents behind (nothing in the op
// reads scratch before writing it, so no clearing is needed).
//
// The array holds hip_qmm_mul_mat_workspace_preferred of every shape that is
// accepted, so the kernel, and with it the result, is that of a call with that
// workspace.  A required size of 32 MiB bounds ncols * K * 9/8, so the f16 route's
// panels, 288 K bytes for each 128 columns begun, take at most 64 MiB + 288 K, 82
// MiB with its K <= 65536, and its K split's partials, of at most 256 tiles of 256 x
// 128 f32, at most 32 MiB.

static __device__ __align__(256) uint8_t scratch[HIP_QMM_NOALLOC_ARRAY_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::atomic<void *> scratch_addr[MAX_DEVICES];
std::mutex scratch_mu;

int current_device_scratch(void **out) {
    int dev = -1;
    if (hipError_t e = hipGetDevice(&dev)) return (int)e;
    if (dev < 0 || dev >= MAX_DEVICES) return (int)hipErrorInvalidDevice;
    void *p = scratch_addr[dev].load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> lock(scratch_mu);
        p = scratch_addr[dev].load(std::memory_order_relaxed);
        if (!p) {
            if (hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch))) return (int)e;
            if (!p) return (int)hipErrorInvalidSymbol;
            scratch_addr[dev].store(p, std::memory_order_release);
        }
    }
    *out = p;
    return 0;
}
}  // namespace

extern "C" int hip_qmm_mul_mat_noalloc(int type, const void *w, int64_t K, int64_t nrows, int64_t row_stride,
                                       const float *x, int64_t ncols, int64_t x_col_stride, float *dst,
                                       int64_t dst_col_stride, void *stream) {
    if (ncols <= 0 || K <= 0) return (int)hipErrorInvalidValue;
    if (hip_qmm_mul_mat_workspace_size(type, K, nrows, ncols) > (size_t)HIP_QMM_NOALLOC_SCRATCH_BYTES)
        return (int)hipErrorInvalidValue;
    void *ws = nullptr;
    if (int e = current_device_scratch(&ws)) return e;
    return hip_qmm_mul_mat(type, w, K, nrows, row_stride, x, ncols, x_col_stride, dst, dst_col_stride, ws,
                           (size_t)HIP_QMM_NOALLOC_ARRAY_BYTES, stream);
}
