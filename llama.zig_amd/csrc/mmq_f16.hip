// mmq_f16.hip -- prefill GEMM of the Q4_K, Q5_K and Q6_K weights on the f16
// matrix cores, exact in its integer block products.
//
// The int8 MMQ (mmq_q4k_dma.hip, mmq_q5k_dma.hip) is bound by vector work: per
// output and 32-deep block it converts an int32 dot (v_cvt_f32_i32 takes 4.2
// cycles a wave64 here, an FMA from two waves 2.6) and needs a second MFMA for
// the scale outer product.  This kernel removes both.  A weight code q (4 or 5
// bits) times its 6-bit sub-block scale is at most 31 * 63 = 1953, exact in
// f16; the masked code is taken as the f16 subnormal q * 2^-24, which
// v_pk_mul_f16 and the f16 MFMA take exactly.  The activation codes are f16
// integers.  Two v_mfma_f32_32x32x16_f16 then give sc_j * dot_j * 2^-24 of a
// 32-deep block exactly in f32 (|sc * dot| < 2^24), and an output costs one FMA
// with the column's d8 (kept as d8 * 2^24).  d and the min term are applied
// once per super-block as in the int8 kernels, in the same order, so the
// outputs of Q4_K and Q5_K equal the unsplit int8 MMQ's bit for bit (Q6_K's
// scales take two operands each, see Raw<TYPE_Q6_K>).
//
// Per 32x32 tile and 32-deep block (one wave, two waves per SIMD) the matrix
// cores take 67 cycles, the FMAs 43, the super-block terms 21, decoding 18 (at
// four column tiles a wave), LDS reads 14 and transfers 11, each measured as
// what its removal saves: 174 cycles in sum where the whole takes 162, so they
// hardly overlap (the int8 kernel takes about 220).  What is left is the sum of
// matrix and vector work and the clock, which falls to 1.95-2.1 GHz under it.
//
// Layout.  A workgroup of NW waves takes 32 * NW weight rows by 32 * NCT
// columns; every wave holds 32 rows: its super-block is decoded once into 16
// MFMA operands in registers (its raw bytes are loaded a super-block ahead) and
// meets every column tile.  The columns come as panels, written by
// quantize_panels in the order the MFMA lanes read them: a panel is 32 columns
// of one super-block, 16 operands of 64 lanes x 16 bytes, then d8 * 2^24 (f32)
// and s8 (f16).  Panels move to LDS with global_load_lds_dwordx4, double
// buffered, one barrier per super-block, and each LDS read is one conflict-free
// ds_read_b128.  The transfers and the weight loads are spread over the step's
// pairs (issued together at its start they stalled the waves: 200 against 162
// cycles a pair).
#include <type_traits>

#include "../../include/ggml_hip_qmm.h"
#include "mmq_dma.h"
#include "mmq_launch.h"
#include "qmm_device.h"

using namespace qmm;
using namespace qmm_dma;

namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int PANEL_BYTES = 18432;   // 16 KiB of codes, 1 KiB of d8, 512 B of s8, 512 B unused
constexpr int PANEL_D = 16384;       // d8 * 2^24: [sub-block / 4][column][sub-block % 4] f32
constexpr int PANEL_S = 17408;       // s8: [column][sub-block] f16
constexpr int PANEL_UNIT = 4;        // panels per super-block are a multiple of this (the widest tile)

constexpr int F16_MAX_K = 65536;  // keeps the panels of a call without a workspace argument within its array (api.hip)

constexpr int F16_CUS = 256;   // 256 x 128 tiles resident at once, one per CU
constexpr int F16_REST = 128;  // a last round of at most this many tiles runs as quarter tiles

__host__ __device__ constexpr int64_t panel_count(int64_t ncols) {
    return (ncols + 32 * PANEL_UNIT - 1) / (32 * PANEL_UNIT) * PANEL_UNIT;
}

// f32 columns -> panels [super-block][panel].  One workgroup per panel and
// super-block: a thread quantizes 8 consecutive values of a column as
// quantize_q8_1_planar8 does (same codes and headers), which are one lane's 16
// bytes of one operand: sub-block j, values 16h + 8m + {0, 2, 1, 3, 4, 6, 5, 7}
// go to operand 2j + m, lane half h (the value order is the one in which the
// weight nibbles come out of their masks).  Columns past ncols are zeros.
// The chunks pass through LDS, rotated by their index so that the writes
// spread over the banks, and leave in one contiguous run.
__global__ __launch_bounds__(256) void quantize_panels(const float *__restrict__ x, int64_t ncols,
                                                       int64_t x_col_stride, uint8_t *__restrict__ out,
                                                       int64_t npanels) {
    __shared__ alignas(16) uint8_t st[PANEL_BYTES];
    const int sb = blockIdx.x, panel = blockIdx.y;
    const int k8 = threadIdx.x & 31;  // 8 values k8 * 8 .. of the super-block: 4j + 2h + m
    const int chunk = ((k8 >> 2) * 2 + (k8 & 1)) * 2 + ((k8 >> 1) & 1);  // operand 2j + m, lane half h
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = (threadIdx.x >> 5) + 8 * i;
        const int64_t col = (int64_t)panel * 32 + c;
        float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        if (col < ncols) {
            const float *p = x + col * x_col_stride + (int64_t)sb * QK_K + k8 * 8;
            const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
            v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        }
        const Q8Quad r = q8_1_quantize_quad(v);
        auto pair = [](uint32_t w, int lo, int hi) {
            return f16_bits((float)(int8_t)(w >> (8 * lo))) | f16_bits((float)(int8_t)(w >> (8 * hi))) << 16;
        };
        *reinterpret_cast<uint4 *>(st + (chunk * 32 + ((c + chunk) & 31)) * 16) =
            make_uint4(pair(r.lo, 0, 2), pair(r.lo, 1, 3), pair(r.hi, 0, 2), pair(r.hi, 1, 3));
        if ((threadIdx.x & 3) == 0) {
            const int j = k8 >> 2;
            *reinterpret_cast<float *>(st + PANEL_D + (j >> 2) * 512 + c * 16 + (j & 3) * 4) =
                h2f(r.ds) * 16777216.0f;
            *reinterpret_cast<uint16_t *>(st + PANEL_S + c * 16 + j * 2) = (uint16_t)(r.ds >> 16);
        }
    }
    __syncthreads();
    uint4 *o = reinterpret_cast<uint4 *>(out + ((int64_t)sb * npanels + panel) * PANEL_BYTES);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int u = threadIdx.x + 256 * i, ch = u >> 5;
        o[u] = *reinterpret_cast<const uint4 *>(st + (ch * 32 + (((u & 31) + ch) & 31)) * 16);
    }
    if (threadIdx.x < 96)
        o[PANEL_D / 16 + threadIdx.x] = *reinterpret_cast<const uint4 *>(st + PANEL_D + threadIdx.x * 16);
}

// A lane's raw bytes of its row and their decoding into MFMA operands, in SEGS
// segments of a super-block.  Segment g's loads are NL(g) 16-byte loads, issued
// one segment ahead; decode(g) gives, for each of its JS sub-blocks, M operands
// per K half (M = 2 for Q6_K: two f16 parts of a product), and leaves the row
// header (d | dmin << 16) and, for the types with mins, the min term's operand.
__device__ __forceinline__ v2h pk(uint32_t u) { return __builtin_bit_cast(v2h, u); }
__device__ __forceinline__ uint32_t bits(v2h h) { return __builtin_bit_cast(uint32_t, h); }
// two bytes of `bytes` picked by sel (0x07BB07AA) as exact f16: 0x64nn is 1024 + nn
__device__ __forceinline__ v2h bytes_f16(uint32_t bytes, uint32_t sel) {
    const v2h k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
    return pk(__builtin_amdgcn_perm(0x64646464u, bytes, sel)) - k1024;
}

template <int TYPE>
struct Raw {  // Q4_K, Q5_K
    static constexpr bool Q5 = TYPE == TYPE_Q5_K;
    static constexpr int BYTES = Q5 ? Q5K_BYTES : Q4K_BYTES, SEGS = 1, JS = 8, M = 1;
    static constexpr bool MINS = true;
    static constexpr int NL(int) { return Q5 ? 6 : 5; }
    uint4 hdr, qs[4], qh;
    v4h am;

    __device__ __forceinline__ void load(int, int k, const uint8_t *blk, int lh) {
        if (k == 0) hdr = ld_u128(blk);
        else if (k < 5) qs[k - 1] = ld_u128(blk + (Q5 ? 48 : 16) + 32 * (k - 1) + 16 * lh);
        else qh = ld_u128(blk + 16 + 16 * lh);
    }
    __device__ __forceinline__ uint32_t row_header() const { return hdr.x; }
    // A operands 2j, 2j + 1: sc_j * q as subnormals.  A low nibble is masked to
    // q; a high one in place to 16 q, so its factor is sc / 16.
    template <int SEG>
    __device__ __forceinline__ void decode(int lh, v8h (&A)[16]) {
        const uint32_t s0 = hdr.y, s1 = hdr.z, s2 = hdr.w;
        const uint32_t sc03 = s0 & 0x3F3F3F3Fu, sc47 = (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u);
        const uint32_t mn03 = s1 & 0x3F3F3F3Fu, mn47 = ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
        // the min term's A operand: this half's four mins (K slots 4h..4h+3)
        const uint32_t mnb = lh ? mn47 : mn03;
        am = __builtin_bit_cast(v4h, make_uint2(bits(bytes_f16(mnb, 0x07010700u)), bits(bytes_f16(mnb, 0x07030702u))));
        const v2h k16th = {(_Float16)0.0625f, (_Float16)0.0625f};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t scw = c < 2 ? sc03 : sc47;
            const v2h sl = bytes_f16(scw, (c & 1) ? 0x07020702u : 0x07000700u);
            const v2h sh = bytes_f16(scw, (c & 1) ? 0x07030703u : 0x07010701u) * k16th;
            const uint32_t q[4] = {qs[c].x, qs[c].y, qs[c].z, qs[c].w};
            const uint32_t hb[4] = {qh.x, qh.y, qh.z, qh.w};
            uint32_t lo[8], hi[8];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
#pragma unroll
                for (int o = 0; o < 2; ++o) {  // bytes 0 and 2, then 1 and 3
                    const uint32_t b = o ? q[d] >> 8 : q[d];
                    uint32_t l = b & 0x000F000Fu, h = b & 0x00F000F0u;
                    if constexpr (Q5) {
                        // bits 2c and 2c + 1 of the element's byte: to bits 4 and 8 of its half
                        const uint32_t g = o ? hb[d] >> 8 : hb[d];
                        l |= (2 * c < 4 ? g << (4 - 2 * c) : g >> (2 * c - 4)) & 0x00100010u;
                        h |= (g << (7 - 2 * c)) & 0x01000100u;
                    }
                    lo[2 * d + o] = bits(pk(l) * sl);
                    hi[2 * d + o] = bits(pk(h) * sh);
                }
            }
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                A[4 * c + m] = __builtin_bit_cast(v8h, make_uint4(lo[4 * m], lo[4 * m + 1], lo[4 * m + 2], lo[4 * m + 3]));
                A[4 * c + 2 + m] =
                    __builtin_bit_cast(v8h, make_uint4(hi[4 * m], hi[4 * m + 1], hi[4 * m + 2], hi[4 * m + 3]));
            }
        }
    }
};

// Q6_K: q - 32 (6 bits) times an int8 scale needs 13 bits.  The scale is split
// into its even part and its low bit: (q - 32) * even has at most 11 significant
// bits, (q - 32) * bit is q - 32 or 0, so both are exact in f16, and the four
// MFMAs of a 32-deep block add up exactly (|sum| <= 32 * 128 * 128 * 32 = 2^24).
// Lane half h holds elements 16h..16h+15 of every sub-block, which share one
// scale.  Segment n is the half super-block n.
template <>
struct Raw<TYPE_Q6_K> {
    static constexpr int BYTES = Q6K_BYTES, SEGS = 2, JS = 4, M = 2;
    static constexpr bool MINS = false;
    static constexpr int NL(int seg) { return seg == 0 ? 5 : 3; }
    uint4 ql[2], qh, sc;
    uint32_t d;
    v4h am;  // unused

    __device__ __forceinline__ void load(int seg, int k, const uint8_t *blk, int lh) {
        if (k < 2) ql[k] = ld16_u(blk + 64 * seg + 32 * k + 16 * lh);
        else if (k == 2) qh = ld16_u(blk + 128 + 32 * seg + 16 * lh);
        else if (k == 3) sc = ld16_u(blk + 192);
        else d = ld_u16(blk + 208);
    }
    __device__ __forceinline__ uint32_t row_header() const { return d; }
    // A operands 4g + 2m' + part of sub-block g: m' the K half, part 0 the even scale, 1 its low bit
    template <int SEG>
    __device__ __forceinline__ void decode(int lh, v8h (&A)[16]) {
        const uint32_t s0 = SEG ? sc.z : sc.x, s1 = SEG ? sc.w : sc.y;  // scales 8 SEG + 2g + h
        const uint32_t hb[4] = {qh.x, qh.y, qh.z, qh.w};
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int scale = (int8_t)((g < 2 ? s0 : s1) >> (16 * (g & 1) + 8 * lh));
            const _Float16 ev = (_Float16)(float)(scale & ~1);
            const v2h even = {ev, ev};
            const uint32_t odd = 0u - (uint32_t)(scale & 1);
            const uint4 &qv = ql[g & 1];
            const uint32_t q[4] = {qv.x, qv.y, qv.z, qv.w};
            uint32_t hi[8], lo[8];
#pragma unroll
            for (int dw = 0; dw < 4; ++dw)
#pragma unroll
                for (int o = 0; o < 2; ++o) {  // bytes 0 and 2, then 1 and 3
                    const uint32_t b = q[dw] >> (8 * o + (g < 2 ? 0 : 4));
                    const int sh = 2 * g + 8 * o - 4;  // bits 2g, 2g + 1 of the byte to bits 4, 5
                    const uint32_t t = sh < 0 ? hb[dw] << -sh : hb[dw] >> sh;
                    // u = q as the subnormal u * 2^-24; minus 32 * 2^-24
                    const v2h v = pk((b & 0x000F000Fu) | (t & 0x00300030u)) - pk(0x00200020u);
                    hi[2 * dw + o] = bits(v * even);
                    lo[2 * dw + o] = bits(v) & odd;
                }
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                A[4 * g + 2 * m] = __builtin_bit_cast(v8h, make_uint4(hi[4 * m], hi[4 * m + 1], hi[4 * m + 2], hi[4 * m + 3]));
                A[4 * g + 2 * m + 1] =
                    __builtin_bit_cast(v8h, make_uint4(lo[4 * m], lo[4 * m + 1], lo[4 * m + 2], lo[4 * m + 3]));
            }
        }
    }
};

// The tiles of one launch: tiles [base, base + n) of the banded order over a gx
// x gy grid (mmq_tile_order's), dealt so that each XCD gets one contiguous run;
// with quads, four workgroups per tile take its quarters (row half l % 2,
// column half l / 2 % 2).
struct TileGrid {
    int gx, gy, base, n;
    bool quads;
};

__device__ __forceinline__ void f16_tile(const TileGrid &g, int l, int &bx, int &by) {
    const int t = g.quads ? l >> 2 : l;
    const int q = g.n >> 3, r = g.n & 7, xcd = t & 7;
    const int v = g.base + (g.quads ? t : (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (t >> 3));
    const int band = v / (MMQ_BAND * g.gy), idx = v - band * (MMQ_BAND * g.gy);
    const int rows = g.gx - band * MMQ_BAND < MMQ_BAND ? g.gx - band * MMQ_BAND : MMQ_BAND;
    bx = band * MMQ_BAND + idx % rows;
    by = idx / rows;
    if (g.quads) {
        bx = 2 * bx + (l & 1);
        by = 2 * by + (l >> 1 & 1);
    }
}

template <int TYPE, int NCT, int NW>
__global__ __launch_bounds__(64 * NW, 2) void mmq_f16_kernel(const uint8_t *__restrict__ w, int nsb, int64_t nrows,
                                                             int64_t row_stride, const uint8_t *__restrict__ panels,
                                                             int64_t ncols, float *__restrict__ dst,
                                                             int64_t dst_col_stride, float *__restrict__ partial,
                                                             TileGrid tg, int gz, MmqGlu glu) {
    using R = Raw<TYPE>;
    constexpr int STAGE = NCT * PANEL_BYTES;
    constexpr int PER = NCT * 18 / NW;  // 1 KiB transfers per wave and step
    static_assert(NCT * 18 % NW == 0 && NCT <= PANEL_UNIT, "whole transfers per wave");
    __shared__ alignas(16) uint8_t sB0[STAGE], sB1[STAGE];
    __shared__ alignas(16) uint32_t rowh[NW][32];  // (d | dmin << 16) of the wave's rows
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const uint32_t lane16 = lane * 16;

    int bx, by;
    f16_tile(tg, (int)blockIdx.x, bx, by);
    if (bx * (glu.gate ? 16 * NW : 32 * NW) >= nrows || by * 32 * NCT >= ncols) return;  // uniform
    const int z = (int)blockIdx.y;
    const int kb0 = (int)((int64_t)nsb * z / gz), kb1 = (int)((int64_t)nsb * (z + 1) / gz);

    // this lane's weight row; rows past the end repeat the last one (never stored)
    const bool fused = glu.gate != nullptr;  // uniform
    const int trow = wave * 32 + li;
    const int64_t orow = fused ? (int64_t)bx * (16 * NW) + mmq_glu_tile_row(trow) : (int64_t)bx * (32 * NW) + trow;
    const uint8_t *ap = (fused && (trow & 2) == 0 ? glu.gate : w) + (orow < nrows ? orow : nrows - 1) * row_stride;

    const int64_t bstep = panel_count(ncols) * PANEL_BYTES;
    const uint8_t *bbase = panels + (int64_t)by * STAGE + wave * 1024;
    R raw;
    auto dma = [&](int k, int sb, uint8_t *s) {
        dma16(bbase + sb * bstep + NW * k * 1024 + lane16, s + (wave + NW * k) * 1024);
    };
    auto load = [&](int seg, int k, int sb) { raw.load(seg, k, ap + (int64_t)sb * R::BYTES, lh); };

    v16f acc[NCT];
#pragma unroll
    for (int t = 0; t < NCT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;

    // Contract segment SEG of super-block `cur` in s.  Meanwhile, spread over the
    // segment's pairs: the panel transfers of super-block `nxt` into snext (in the
    // first segment) and the raw bytes of the next segment.
    auto segment = [&](auto seg, const uint8_t *s, int cur, int nxt, uint8_t *snext) __attribute__((always_inline)) {
        constexpr int SEG = decltype(seg)::value, NSEG = (SEG + 1) % R::SEGS;
        v8h A[16];
        if (SEG == 0) rowh[wave][li] = raw.row_header();  // both lane halves store the same word
        raw.template decode<SEG>(lh, A);
        const v4h am = raw.am;

        // pairs p = (column tile t, sub-block j): pair p + 1's MFMAs and pair
        // p + 2's LDS reads are issued before pair p's FMAs
        constexpr int NP = R::JS * NCT, NDMA = SEG == 0 ? PER : 0, NOPS = NDMA + R::NL(NSEG);
        constexpr int SPREAD = NP * 2 / 3;  // the memory operations' pairs: the first two thirds
        v8h bop[2][2];
        v16f out[2], accb;
        float4 dq[2];
        const v16f zero = {0};
        auto ldb = [&](int p, int m) {
            const int t = p / R::JS, j = SEG * R::JS + p % R::JS;
            return *reinterpret_cast<const v8h *>(s + t * PANEL_BYTES + j * 2048 + m * 1024 + lane16);
        };
        auto mfmas = [&](int p, v16f &r) {
            const int a = p % R::JS * 2 * R::M;
            r = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[a], bop[p & 1][0], zero, 0, 0, 0);
            if constexpr (R::M == 2) r = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[a + 1], bop[p & 1][0], r, 0, 0, 0);
            r = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[a + R::M], bop[p & 1][1], r, 0, 0, 0);
            if constexpr (R::M == 2) r = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[a + 3], bop[p & 1][1], r, 0, 0, 0);
        };
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            bop[p][0] = ldb(p, 0);
            bop[p][1] = ldb(p, 1);
        }
        mfmas(0, out[0]);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int t = p / R::JS, j = p % R::JS;
            const uint8_t *bt = s + t * PANEL_BYTES;
            __builtin_amdgcn_sched_barrier(0);
            if (j == 0) {
#pragma unroll
                for (int h = 0; h < R::JS / 4; ++h)
                    dq[h] = *reinterpret_cast<const float4 *>(bt + PANEL_D + (SEG * R::JS / 4 + h) * 512 + li * 16);
            }
            const float4 d4 = dq[j >> 2];
            const float d8 = (j & 3) == 0 ? d4.x : (j & 3) == 1 ? d4.y : (j & 3) == 2 ? d4.z : d4.w;
            if (p + 1 < NP) mfmas(p + 1, out[(p + 1) & 1]);
#pragma unroll
            for (int k = 0; k < NOPS; ++k)
                if (k * SPREAD / NOPS == p) {
                    // the next segment's bytes first where it is in this super-block
                    constexpr int L0 = NSEG == 0 ? NDMA : 0;
                    if (k >= L0 && k < L0 + R::NL(NSEG)) load(NSEG, k - L0, NSEG == 0 ? nxt : cur);
                    else dma(NSEG == 0 ? k : k - R::NL(NSEG), nxt, snext);
                }
            if (p + 2 < NP) {
                bop[p & 1][0] = ldb(p + 2, 0);
                bop[p & 1][1] = ldb(p + 2, 1);
            }
            const v16f &S = out[p & 1];
#pragma unroll
            for (int v = 0; v < 16; ++v) accb[v] = j == 0 ? S[v] * d8 : fmaf(S[v], d8, accb[v]);
            if (j == R::JS - 1) {  // acc += d * accb - dmin * sum_j m_j * s8_j
                v16f P = zero;
                if constexpr (R::MINS) {
                    const v4h bm = *reinterpret_cast<const v4h *>(bt + PANEL_S + li * 16 + 8 * lh);
                    P = __builtin_amdgcn_mfma_f32_32x32x8f16(am, bm, zero, 0, 0, 0);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint4 hw = *reinterpret_cast<const uint4 *>(&rowh[wave][8 * q + 4 * lh]);
                    const uint32_t hh[4] = {hw.x, hw.y, hw.z, hw.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const v2h dm = pk(hh[i]);
                        const int v = 4 * q + i;
                        if constexpr (R::MINS) acc[t][v] = fmaf(-(float)dm[1], P[v], acc[t][v]);
                        acc[t][v] = fmaf((float)dm[0], accb[v], acc[t][v]);
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](const uint8_t *s, int cur, int nxt, uint8_t *snext) __attribute__((always_inline)) {
        segment(std::integral_constant<int, 0>{}, s, cur, nxt, snext);
        if constexpr (R::SEGS == 2) segment(std::integral_constant<int, 1>{}, s, cur, nxt, snext);
    };

#pragma unroll
    for (int k = 0; k < PER; ++k) dma(k, kb0, sB0);
#pragma unroll
    for (int k = 0; k < R::NL(0); ++k) load(0, k, kb0);
    wait_vmem();
    __syncthreads();
    // the last step reloads its own super-block into the idle buffer: no branch
    // in the step, and never a read past the row
    for (int sb = kb0; sb < kb1; sb += 2) {
        step(sB0, sb, sb + 1 < kb1 ? sb + 1 : kb1 - 1, sB1);
        wait_vmem();
        __syncthreads();
        if (sb + 1 < kb1) {
            step(sB1, sb + 1, sb + 2 < kb1 ? sb + 2 : kb1 - 1, sB0);
            wait_vmem();
            __syncthreads();
        }
    }
#pragma unroll
    for (int t = 0; t < NCT; ++t) {
        const int64_t c = (int64_t)(by * NCT + t) * 32 + li;
        if (c >= ncols) continue;
        float *o = partial ? partial + ((int64_t)z * ncols + c) * nrows : dst + c * dst_col_stride;
        if (fused) store_glu_column(o, (int64_t)bx * (16 * NW) + wave * 16 + 2 * lh, nrows, acc[t], glu);
        else store_tile_column(o, (int64_t)bx * (32 * NW) + wave * 32 + 4 * lh, nrows, acc[t]);
    }
}

// One launch of 256 x 128 tiles (NCT 4, NW 8) or 128 x 64 ones (2, 4).
template <int TYPE, int NCT, int NW>
int launch_tiles(const TileGrid &tg, const void *w, int64_t K, int64_t nrows, int64_t row_stride,
                 const uint8_t *panels, int64_t ncols, float *dst, int64_t dst_col_stride, float *partial, int split,
                 const MmqGlu &glu, hipStream_t s) {
    const dim3 grid((unsigned)(tg.quads ? 4 * tg.n : tg.n), (unsigned)split);
    hipLaunchKernelGGL((mmq_f16_kernel<TYPE, NCT, NW>), grid, dim3(64 * NW), 0, s, (const uint8_t *)w,
                       (int)(K / QK_K), nrows, row_stride, panels, ncols, dst, dst_col_stride, partial, tg, split, glu);
    return (int)hipGetLastError();
}

template <int TYPE>
int launch_type(bool wide, const void *w, int64_t K, int64_t nrows, int64_t row_stride, const uint8_t *panels,
                int64_t ncols, float *dst, int64_t dst_col_stride, float *partial, int split, const MmqGlu &glu,
                hipStream_t s) {
    const int64_t rows = (wide ? 256 : 128) / (glu.gate ? 2 : 1), cols = wide ? 128 : 64;
    const int64_t gx = (nrows + rows - 1) / rows, gy = (ncols + cols - 1) / cols;
    if (gx * gy > 0x1FFFFFFF || split < 1 || split > 64) return (int)hipErrorInvalidValue;
    TileGrid tg{(int)gx, (int)gy, 0, (int)(gx * gy), false};
    if (!wide)
        return launch_tiles<TYPE, 2, 4>(tg, w, K, nrows, row_stride, panels, ncols, dst, dst_col_stride, partial,
                                        split, glu, s);
    const int rest = tg.n % F16_CUS;
    if (split == 1 && tg.n > F16_CUS && rest > 0 && rest <= F16_REST) {
        tg.n -= rest;
        if (int e = launch_tiles<TYPE, 4, 8>(tg, w, K, nrows, row_stride, panels, ncols, dst, dst_col_stride, partial,
                                             split, glu, s))
            return e;
        const TileGrid quads{tg.gx, tg.gy, tg.n, rest, true};
        return launch_tiles<TYPE, 2, 4>(quads, w, K, nrows, row_stride, panels, ncols, dst, dst_col_stride, partial,
                                        split, glu, s);
    }
    return launch_tiles<TYPE, 4, 8>(tg, w, K, nrows, row_stride, panels, ncols, dst, dst_col_stride, partial, split,
                                    glu, s);
}

}  // namespace

// Which products take this kernel, and how: modelled times in us of the choices
// against the int8 MMQ's, fitted to a sweep of every choice on 180 shapes
// (512-28672 rows, K 512-14336, 33-2048 columns, plain and gate/up-fused; whole
// calls, graph-timed).  A choice is taken 5 % below the int8 model: on the sweep
// the chosen times are 1.25x (Q6_K), 1.02x (Q5_K) and 1.005x (Q4_K) better in the
// geometric mean, of 1.27x, 1.03x and 1.017x with perfect choices, and the worst
// one is 10 % slower (Q4_K 9184x2304 at 1286).  Per 16 super-blocks of K:
//   - a round of 256 wide tiles takes 77 us (Q5_K 1.14, Q6_K 1.7 times that), a
//     last round 38 / 57 as quarter tiles of up to 64 / 128 tiles, else 68-78 (it
//     leaves CUs idle, and the others run at a higher clock); narrow tiles (128
//     x 64, two per CU) take 32 up to 256 workgroups and 51 up to 512;
//   - the int8 kernels take 55 / 62 / 109 (Q4_K, Q5_K, Q6_K) per round of 512 of
//     their 128 x 64 tiles.
// To these come a fixed part, the outputs' write and a K split's partials.
// Measured (us, int8 -> here): Q4_K 14336x4096 at 512 / 1000 / 2048 columns
// 111 -> 94, 195 -> 183, 374 -> 346, gate/up-fused at 2048 700 -> 650;
// 4096x4096 at 2048 120 -> 106; 14336x14336 at 200 185 -> 167; Q5_K 4096x14336
// at 512 124 -> 110.  Q6_K 4096x14336 at 128 / 512 / 2048 68.5 -> 61, 206 -> 145,
// 734 -> 491; 14336x4096 at 300 / 512 188 -> 123, 226 -> 146; 4096x4096 at 512
// 76 -> 56.  The int8 kernels stay ahead on the smaller grids of Q4_K and Q5_K
// (4096x4096 at 200 / 512: 28 / 41 against 37 / 45; 14336x4096 at 128 / 256: 37 /
// 57 against 41 / 61), whose nibbles they unpack for a fraction of what the
// decoding here costs on few column tiles.
MmqF16Plan mmq_f16_plan(int type, int64_t K, int64_t nrows, int64_t ncols, bool glu) {
    MmqF16Plan best{false, false, 1};
    if ((type != TYPE_Q4_K && type != TYPE_Q5_K && type != TYPE_Q6_K) || K <= 0 || K % QK_K != 0 || K > F16_MAX_K ||
        nrows <= 0 || nrows > 0x7FFFFFFF || ncols <= 32 || ncols > 65535)
        return best;
    const bool q6 = type == TYPE_Q6_K, q5 = type == TYPE_Q5_K;
    const int64_t nsb = K / QK_K, rows = glu ? 2 * nrows : nrows;  // both weights' rows
    auto tiles = [&](int64_t r, int64_t c) { return ((rows + r - 1) / r) * ((ncols + c - 1) / c); };
    const double per16 = (double)nsb / 16, scale = q6 ? 1.71 : q5 ? 1.14 : 1.0;
    const double outs = (double)nrows * (double)ncols * 4.0 / 4.0e6;
    auto reduce = [&](int split) { return split > 1 ? 2.9 + (double)split * 2.2 * outs : 0.0; };
    const int64_t wide = tiles(256, 128), narrow = tiles(128, 64);
    // the int8 kernels: rounds of 512 tiles, and the latency of one tile's own steps
    const int split8 = glu ? 1 : hip_qmm_mmq_split_k(type, K, nrows, ncols);
    const double rounds8 = (double)narrow / 512 + (narrow > 512 ? 0.14 : 0.0);
    const double body8 = per16 * (q6 ? 109.0 : q5 ? 62.0 : 55.0) * rounds8;
    const double chain8 = (double)nsb / split8 * (q6 ? 6.1 : q5 ? 2.3 : 1.9);
    double least = 0.95 * ((body8 > chain8 ? body8 : chain8) + (q6 ? 7.3 : 5.6) + outs + reduce(split8));
    auto consider = [&](bool w, int split, double t) {
        if (t < least) {
            least = t;
            best = MmqF16Plan{true, w, split};
        }
    };
    for (int split = 1; split <= 16; ++split) {
        if (nsb % split || (split > 1 && (glu || nsb / split < 4))) continue;
        const double part = per16 / split * scale;
        if (split == 1 || wide * split <= F16_CUS) {
            const int64_t n = wide * split, full = n / F16_CUS, rest = n % F16_CUS;
            const bool quads = full > 0 && rest > 0 && rest <= F16_REST;
            const double last = rest == 0 ? 0.0 : quads ? (rest <= 64 ? 38.4 : 57.0)
                                : 67.5 + 0.08 * (double)(rest > 128 ? rest - 128 : 0);
            consider(true, split, part * (76.8 * (double)full + last) + 9.4 + (quads ? 4.0 : 0.0) + outs + reduce(split));
        }
        if (q6 && (split == 1 || narrow * split <= 2 * F16_CUS)) {
            const int64_t n = narrow * split, full = n / (2 * F16_CUS), rest = n % (2 * F16_CUS);
            const double last = rest == 0 ? 0.0 : rest <= F16_CUS ? 31.6 : 51.3;
            consider(false, split, part * (51.3 * (double)full + last) + 7.0 + outs + reduce(split));
        }
    }
    return best;
}

// Bytes of the panels of ncols columns of K values (K a multiple of 256).
size_t mmq_f16_panel_bytes(int64_t K, int64_t ncols) {
    return (size_t)(K / QK_K) * (size_t)panel_count(ncols) * PANEL_BYTES;
}

int mmq_f16_quantize(const float *x, int64_t K, int64_t ncols, int64_t x_col_stride, void *panels, hipStream_t s) {
    const int64_t np = (ncols + 31) / 32;
    if (np > 65535) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(quantize_panels, dim3((unsigned)(K / QK_K), (unsigned)np), dim3(256), 0, s, x, ncols,
                       x_col_stride, (uint8_t *)panels, panel_count(ncols));
    return (int)hipGetLastError();
}

// The GEMM over panels: 256 x 128 tiles (wide) or 128 x 64; `split` K parts
// into `partial` (then added by the caller) when above 1; gate/up-fused with
// glu.gate (unsplit).  Weight rows 16-byte aligned, checked by the caller.
int mmq_f16_launch(int type, bool wide, const void *w, int64_t K, int64_t nrows, int64_t row_stride,
                   const void *panels, int64_t ncols, float *dst, int64_t dst_col_stride, float *partial, int split,
                   const MmqGlu &glu, hipStream_t s) {
    const uint8_t *p = (const uint8_t *)panels;
    switch (type) {
    case TYPE_Q4_K:
        return launch_type<TYPE_Q4_K>(wide, w, K, nrows, row_stride, p, ncols, dst, dst_col_stride, partial, split, glu, s);
    case TYPE_Q5_K:
        return launch_type<TYPE_Q5_K>(wide, w, K, nrows, row_stride, p, ncols, dst, dst_col_stride, partial, split, glu, s);
    case TYPE_Q6_K:
        return launch_type<TYPE_Q6_K>(wide, w, K, nrows, row_stride, p, ncols, dst, dst_col_stride, partial, split, glu, s);
    default: return (int)hipErrorInvalidValue;
    }
}
