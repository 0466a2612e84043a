// Host side of the small-M / prefill LUT GEMM: shape policy, workspace layout,
// pre-passes (activation permutation, residual coefficients) and the launch.
#include <limits.h>
#include <stdlib.h>

#include "gemm_launch.h"
#include "gemm_wide_kernel.h"
#include "host_common.h"

#include <algorithm>
#include <atomic>

namespace flute {

flute_status gemm_launch_segs(int bf16, int mb, int mw, const GemmParams &p, dim3 grid, int lds, hipStream_t stream);
flute_status gemm_wide_f16(int mb, int b1, int b2, int slices, const WideParams &p, hipStream_t stream);
flute_status gemm_wide_bf16(int mb, int b1, int b2, int slices, const WideParams &p, hipStream_t stream);

namespace {

struct GemmShape {
    int mb, kw, mw;       // 16-row blocks per wavefront, k ways, m ways
    int wg_per_cu;        // workgroups the policy expects to be resident per CU
};

// Rows of A per workgroup.  One or two 16-row blocks per wavefront with eight k ways (the
// launch is then a weight stream, like the GEMV) as long as one workgroup per 16 (32) rows
// and tile fits the device in one round and the indices are not re-read too often: every
// chunk of rows streams its tile again, and beyond about 64 MB (100 MB) of index traffic
// the next shape wins.  Measured: M = 32, 4096 -> 12288: 18.0 us with 16 rows, 24.6 us
// with 64; M = 64: 21.5 us with 32 rows, 26.0 us with 64; M = 256, 4096 -> 4096: 23.8 us
// with 32 rows, 29.0 us with 64; M = 96, 12288 -> 4096: 31.6 us with 32 rows, 37.8 us
// with 16, 34.7 us with 64.  Otherwise four blocks per wavefront: 64 rows per workgroup
// with eight k ways while that fits the device in one round, else 128 rows (two m groups,
// four k ways); further rows go to gridDim.y.  The tables plus staging take most of a
// CU's LDS, so one workgroup per CU is resident.  FLUTE_GEMM_ROWS = 16, 32, 64 or 128
// forces the shape (a tuning and test knob, like FLUTE_GEMV_RW), 256 or 512 the many-row kernel.
// Two streams are one launch in 16-row workgroups and two in all others, so for two chunks of rows
// (M = 17 ... 32) the next shape wins from 80 MB on only: (3, 3) bits, 12288 -> 4096 30.8 us with 16 rows,
// 41.2 with 32; (2, 4) 32.7 and 35.6; (3, 3), 4096 -> 12288 32.5 and 34.4.  A 4-bit stream, though, has
// its one-instruction lookups in a launch of its own only (`fast_stream`), which is worth the second
// launch where a 16-row workgroup would have a K range of 4096 or more: (4, 1) bits, M = 32 with 16
// rows and 32, 4096 -> 12288 34.2 and 30.2 us (rank 16: 42.2, 39.5), 8192 -> 6144 in two slices 35.9 and
// 32.1, 12288 -> 4096 in four 31.7 and 35.2, 2048 -> 12288 22.4 and 25.4; M = 96, 4096 -> 4096 33.1 and 30.2.
GemmShape choose_gemm_shape(int M, int tiles, int64_t index_bytes, int G, bool two_streams, bool fast_stream) {
    {
        const int v = tuning().gemm_rows;
        if (v == 16) return {1, 8, 1, 1};
        if (v == 32) return {2, 8, 1, 1};
        if (v == 64) return {4, 8, 1, 1};
        if (v == 128) return {4, 4, 2, 1};
    }
    if (M <= 16) return {1, 8, 1, 1};
    const int chunks16 = (M + 15) / 16, chunks32 = (M + 31) / 32;
    const int64_t units16 = (int64_t)tiles * chunks16, limit16 = (int64_t)(two_streams && chunks16 == 2 ? 80 : 64) << 20;
    int slices = 1;                                     // of K, as gemm_rows would cut it
    while (units16 * slices * 2 <= kNumCU && G / (slices * 2) >= 16) slices *= 2;
    const bool fast_wins = two_streams && fast_stream && G / slices >= 64;
    if (units16 <= kNumCU && chunks16 * index_bytes <= limit16 && !fast_wins)
        return {1, 8, 1, 1};
    if ((int64_t)tiles * chunks32 <= kNumCU && chunks32 * index_bytes <= (int64_t)100 << 20)
        return {2, 8, 1, 1};
    const int chunks64 = (M + 63) / 64;
    if ((int64_t)tiles * chunks64 <= kNumCU) return {4, 8, 1, 1};
    return {4, 4, 2, 1};
}

bool fast_stream(const flute_linear &w) { return (w.b1 == 4 || w.b2 == 4) && w.group_size >= 64; }

// The residual coefficients of a call's weights, xb[i][m, r] = sum_k A[m, k] * resB[i][r, k] in fp32:
// 16-row by 16-rank blocks in as many slices of K as the chip has CUs for, 512 columns (one step of a
// workgroup) or more each.
struct CoeffPlan {
    int rows, ranks, slices;                            // blocks
    size_t floats() const { return slices > 1 ? (size_t)slices * rows * ranks * 256 : 0; }
    size_t tickets() const { return (size_t)rows * ranks; }
};
CoeffPlan plan_coeff(const flute_linear *ws, int count, int M) {
    CoeffPlan c = {(M + 15) / 16, 0, 1};
    for (int i = 0; i < count; ++i) c.ranks += (ws[i].R + 15) / 16;
    while (c.slices < 16 && (int64_t)c.rows * c.ranks * c.slices * 2 <= kNumCU && ws[0].K / (c.slices * 2) >= 512)
        c.slices *= 2;
    if (c.slices < 4) c.slices = 1;                     // (partial sums are read in fours)
    return c;
}

flute_status launch_coeff(const CoeffPlan &plan, const flute_linear *ws, int count, const void *A, int64_t lda,
                          float *const *xb, int M, int is_bf16, float *part, int *tickets, hipStream_t stream) {
    CoeffParams p = {};
    p.A = (const uint16_t *)A;
    p.lda = lda;
    p.M = M;
    p.K = ws[0].K;
    p.aligned = ((uintptr_t)A & 15) == 0 && lda % 8 == 0;
    p.kper = (p.K / 32 + plan.slices - 1) / plan.slices * 32;
    p.part = part;
    p.tickets = tickets;
    int n = 0, ranks = 0;
    for (int i = 0; i < count; ++i) {
        if (ws[i].R == 0) continue;
        p.resB[n] = (const uint16_t *)ws[i].resB;
        p.xb[n] = xb[i];
        p.R[n] = ws[i].R;
        p.rank0[n++] = ranks;
        p.aligned &= ((uintptr_t)ws[i].resB & 15) == 0;
        ranks += (ws[i].R + 15) / 16;
    }
    for (; n < kGemmMaxSegs; ++n) p.rank0[n] = INT_MAX;
    const dim3 grid(plan.rows, plan.ranks, plan.slices);
    if (is_bf16) hipLaunchKernelGGL(gemm_coeff_kernel<true>, grid, dim3(1024), 0, stream, p);
    else hipLaunchKernelGGL(gemm_coeff_kernel<false>, grid, dim3(1024), 0, stream, p);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

// LDS plan of one launch: pair tables (+ staging on the fast path), sized against the
// reduction tree and the totals tile that reuse the same memory afterwards.
// A single 4-bit stream with at most two LUT groups per 128-row tile gets 64-lane
// replication (256 bytes per entry, 64 KB per group, first table at LDS offset 0: the
// layout the one-instruction address needs).  Everything else: as much replication as
// the budget allows, 32 lanes at most.
int plan_lds(GemmParams &p, const GemmShape &shape) {
    const int ngrp = p.seg[0].gs >= 128 ? 1 : 128 / p.seg[0].gs;
    const bool perm = p.nstreams == 1 && p.bits[0] == 4 && ngrp <= 2 &&
                      !tuning().gemm_no_perm;
    const int table_budget = (shape.mb == 1 ? 64 : 96) * 1024 / p.nstreams;
    int lds_tables = 0;
    for (int s = 0; s < p.nstreams; ++s) {
        const int entries = ngrp << (2 * p.bits[s]);
        int rl = 5;
        while (rl > 0 && (entries << rl) * 4 > table_budget) --rl;
        if (perm) rl = 6;
        p.rep_log2[s] = rl;
        p.tab_off[s] = lds_tables;
        lds_tables += (entries << rl) * 4;
    }
    p.lean = 0;
    if (perm) {                                  // per-wavefront tile staging behind the tables
        // four blocks per wavefront and one LUT group per tile: the lean loop, whose tiles go
        // straight into two staging buffers per wavefront
        p.lean = shape.mb == 4 && ngrp == 1 && !tuning().gemm_no_lean;
        p.stage_off = lds_tables;
        lds_tables += shape.kw * shape.mw * (p.lean ? 8192 : 4096);
        if (p.lean) {                            // one progress word per wavefront
            p.prog_off = lds_tables;
            lds_tables += 64;
            p.balance = !tuning().gemm_no_balance;
        }
    }
    const int slot_bytes = shape.mb * 8 * 64 * 16;
    const int lds_reduce = (shape.kw / 2) * shape.mw * slot_bytes;
    const int lds_tile = shape.mw * shape.mb * 16 * 132 * 4 + 16;   // totals tile + ticket flag
    int lds = lds_tables > lds_reduce ? lds_tables : lds_reduce;
    if (lds_tile > lds) lds = lds_tile;
    // the hand-overs between the k ways: eight 16 KB areas, then eight of 8 KB behind the totals tile
    if (p.scatter && lds < 17 * 4096 + 8 * 8192) lds = 17 * 4096 + 8 * 8192;
    return lds;
}

}  // namespace

}  // namespace flute

namespace flute {
namespace {

// How the many-row kernel would serve a call; rows = 0: the other kernels do.
struct WidePlan {
    int rows;      // rows of A per workgroup: 512 or 256
    int ksplit;
};

// The many-row kernel or the others, and its shape.  Each form's time is a line in what it has to
// do, in microseconds, fitted to measurements (4-bit stream, bfloat16; `steps` = 64-k tiles of all
// streams that a workgroup takes, `rounds` = workgroups / 256 CUs, rounded up):
//   128-row workgroups of gemm_kernel.h   8 + 0.43 a tile (64-row ones 0.26) per round; two
//                                         streams are two launches, other widths 15 % more
//   512-row workgroups                    14 a round + 0.95 ... 1.35 a step (the clock falls as the chip
//                                         fills); slices of K cost 5 each (256 KB written, read)
//   256-row workgroups                    14 a round + 0.65 ... 0.90 a step; slices 2.5 each
// e.g. M = 1024, 4096 -> 12288: 120 / 92 / 118 us (estimated 105 / 94 / 122); M = 512: 74 / 61
// (two slices) / 61; M = 512, 12288 -> 4096: 59 / 77 (four) / 65 (four), the others stay; two
// streams (4, 1) at M = 1024, 4096 -> 12288: 263 / 165 / 190, at M = 192: 76 / - / 60 (two).
// Calls that the 16- and 32-row workgroups serve in one round stay with them (M = 128,
// 4096 -> 12288: 27 us there, 41 us here).
// (several weights in one launch: `tiles` counts theirs; `other_us` is other_forms' estimate)
double other_forms(int M, int tiles, int G, int streams, bool four_bit, const GemmShape &other) {
    const int rows_other = other.mb * other.mw * 16;
    const int64_t units_other = (int64_t)tiles * ((M + rows_other - 1) / rows_other);
    int ks_other = 1;
    while (units_other * ks_other * 2 <= kNumCU && ks_other < 4 && G / (ks_other * 2) >= other.kw * 2) ks_other *= 2;
    const double per_tile = (other.mw == 1 ? 0.26 : 0.43) * (four_bit && streams == 1 ? 1.0 : 1.15);
    return streams * (double)((units_other * ks_other + kNumCU - 1) / kNumCU) * (8.0 + per_tile * G / ks_other) +
           (ks_other > 1 ? 5.0 : 0.0);
}

WidePlan choose_wide(int M, int tiles, int G, int streams, double other_us, const GemmShape &other) {
    {
        const int v = tuning().gemm_rows;
        if (v == 512 || v == 256) {
            const int k = tuning().gemm_ksplit;
            return {v, k > 1 ? (k < G ? k : G) : 1};
        }
        if (v) return {0, 1};
    }
    if (other.mb < 4) return {0, 1};
    double best = other_us;
    WidePlan plan = {0, 1};
    for (int rows = 512; rows >= 256; rows /= 2) {
        const int64_t units = (int64_t)tiles * ((M + rows - 1) / rows);
        for (int ks = 1; ks <= 8 && G / ks >= 8; ks *= 2) {
            const int64_t groups = units * ks, rounds = (groups + kNumCU - 1) / kNumCU;
            const double fill = groups < kNumCU ? (double)groups / kNumCU : 1.0;
            const double step = rows == 512 ? 0.95 + 0.40 * fill : 0.65 + 0.25 * fill;
            const double us = rounds * (14.0 + step * streams * ((G + ks - 1) / ks)) +
                              (ks > 1 ? (rows == 512 ? 5.0 : 2.5) * ks : 0.0);
            if (us < best) {
                best = us;
                plan = {rows, ks};
            }
        }
    }
    return plan;
}

// Up to four weights over the same rows of A: C[i] = A @ W[i]^T (+ residual, bias).  They share
// their LUT's type and K; weights of one width pair go in one launch.
flute_status gemm_wide(const flute_linear *ws, int count, const void *A, void *const *C, const int64_t *ldc, int M,
                       int64_t lda, int act_dtype, WidePlan plan, hipStream_t stream) {
    const int K = ws[0].K, G = K / 64, lut_dtype = ws[0].lut_dtype;
    const int out_bf16 = act_dtype == FLUTE_BF16;
    const bool scale_rows = act_dtype == FLUTE_BF16 && lut_dtype == FLUTE_F16;
    const int mb = plan.rows / 128;
    const int mtiles = (M + plan.rows - 1) / plan.rows, mblk = mtiles * plan.rows / 16;
    const int gper = (G + plan.ksplit - 1) / plan.ksplit, slices = (G + gper - 1) / gper;
    FLUTE_REQUIRE(slices <= 65535, FLUTE_ERR_UNSUPPORTED, "flute_gemm: %d slices of K exceed the grid", slices);

    // what a weight needs of the activations: one image per distinct rotation
    int image_of[kWideMaxSegs], owner[kWideMaxSegs], images = 0;
    for (int i = 0; i < count; ++i) {
        int k = 0;
        while (k < images && !(ws[owner[k]].signs == ws[i].signs && ws[owner[k]].awq == ws[i].awq &&
                               ws[owner[k]].rot_block == ws[i].rot_block))
            ++k;
        if (k == images) owner[images++] = i;
        image_of[i] = k;
    }
    auto up4 = [](size_t n) { return (n + 3) & ~(size_t)3; };
    const size_t image_floats = (size_t)K * mblk * 8, rot_floats = up4((size_t)M * K / 2);
    const size_t shift_floats = scale_rows ? up4(M) : 0;
    size_t xb_floats = 0, part_xb = 0, want_tickets = 0;
    int tiles = 0;
    for (int i = 0; i < count; ++i) {
        xb_floats += up4((size_t)M * ws[i].R);
        const CoeffPlan c = plan_coeff(ws + i, 1, M);
        part_xb = std::max(part_xb, c.floats());
        want_tickets = std::max(want_tickets, c.tickets());
        tiles += ws[i].N / 128;
    }
    const size_t part_floats = slices > 1 ? (size_t)slices * mtiles * tiles * plan.rows * 128 : 0;
    size_t total = part_floats + xb_floats + part_xb + 64;
    for (int k = 0; k < images; ++k) total += image_floats + shift_floats + (ws[owner[k]].signs ? rot_floats : 0);
    float *base = nullptr;
    int *tickets = nullptr;
    want_tickets = std::max(want_tickets, (size_t)mtiles * tiles) + 1;
    flute_status st = get_workspace(total, want_tickets, stream, &base, &tickets);
    if (st != FLUTE_OK) return st;
    float *const xb_part = base + part_floats;
    float *next = xb_part + part_xb;

    const u4_t *image[kWideMaxSegs];
    const int *shift[kWideMaxSegs];
    const void *rows[kWideMaxSegs];
    int64_t ldr[kWideMaxSegs];
    for (int k = 0; k < images; ++k) {
        const flute_linear &w = ws[owner[k]];
        rows[k] = A;
        ldr[k] = lda;
        if (w.signs) {
            // (the rotation knows its rows' largest exponents)
            int *const row_shift = scale_rows ? (int *)(next + rot_floats) : nullptr;
            st = fht_launch(A, lda, w.signs, w.awq, next, K, M, K, act_dtype, 0, w.rot_block, stream, nullptr, row_shift);
            if (st != FLUTE_OK) return st;
            rows[k] = next;
            ldr[k] = K;
            next += rot_floats;
        }
        shift[k] = nullptr;
        if (scale_rows && w.signs) {
            shift[k] = (const int *)next;
            next += shift_floats;
        } else if (scale_rows) {
            hipLaunchKernelGGL(gemm_rowshift_kernel, dim3(M), dim3(256), 0, stream, (const uint16_t *)rows[k], ldr[k], K,
                               (int *)next);
            FLUTE_HIP_CHECK(hipGetLastError());
            shift[k] = (const int *)next;
            next += shift_floats;
        }
        const int64_t blocks = (int64_t)(2 * G) * ((M + 15) / 16);
        const int grid = (int)((blocks + 3) / 4 < 8192 ? (blocks + 3) / 4 : 8192);
        hipLaunchKernelGGL(gemm_image_kernel, dim3(grid), dim3(256), 0, stream, (const uint16_t *)rows[k], (u4_t *)next, M,
                           ldr[k], 2 * G, mblk, out_bf16, (int)(lut_dtype == FLUTE_BF16),
                           (int)(((uintptr_t)rows[k] & 15) == 0 && ldr[k] % 8 == 0), shift[k]);
        FLUTE_HIP_CHECK(hipGetLastError());
        image[k] = (const u4_t *)next;
        next += image_floats;
    }
    float *xb[kWideMaxSegs] = {};
    for (int i = 0; i < count; ++i) {
        if (ws[i].R == 0) continue;
        xb[i] = next;
        next += up4((size_t)M * ws[i].R);
        // (weights of different rotations have different rows: one launch each)
        st = launch_coeff(plan_coeff(ws + i, 1, M), ws + i, 1, rows[image_of[i]], ldr[image_of[i]], xb + i, M, out_bf16,
                          xb_part, tickets, stream);
        if (st != FLUTE_OK) return st;
    }
    bool done[kWideMaxSegs] = {};
    for (int i = 0; i < count; ++i) {
        if (done[i]) continue;
        WideParams p = {};
        p.M = M;
        p.G = G;
        p.mblk = mblk;
        p.mtiles = mtiles;
        p.gper = gper;
        p.out_bf16 = out_bf16;
        p.P = base;
        p.tickets = tickets;
        // the sum does not depend on the order of the streams beyond fp32 rounding: the wider first
        const int b1 = ws[i].b1 > ws[i].b2 ? ws[i].b1 : ws[i].b2, b2 = ws[i].b1 + ws[i].b2 - b1;
        for (int k = i; k < count; ++k) {
            const flute_linear &w = ws[k];
            const bool swap = w.b2 > w.b1;
            if (done[k] || (swap ? w.b2 : w.b1) != b1 || (swap ? w.b1 : w.b2) != b2) continue;
            done[k] = true;
            WideSeg &g = p.seg[p.nsegs++];
            g.q[0] = (const uint8_t *)(swap ? w.q2 : w.q1);
            g.q[1] = (const uint8_t *)(swap ? w.q1 : w.q2);
            g.lut[0] = (const uint16_t *)(swap ? w.lut2 : w.lut1);
            g.lut[1] = (const uint16_t *)(swap ? w.lut1 : w.lut2);
            g.Ap = image[image_of[k]];
            g.rowshift = shift[image_of[k]];
            g.xb = xb[k];
            g.resA = (const uint16_t *)w.resA;
            g.bias = (const uint16_t *)w.bias;
            g.C = C[k];
            g.ldc = ldc[k];
            g.tile0 = p.ntiles;
            g.gs = w.group_size;
            g.lut_rows = w.lut_rows;
            g.R = w.R;
            g.vec_store = (ldc[k] % 8 == 0) && (((uintptr_t)C[k] & 15) == 0);
            p.ntiles += w.N / 128;
        }
        st = lut_dtype == FLUTE_BF16 ? gemm_wide_bf16(mb, b1, b2, slices, p, stream)
                                     : gemm_wide_f16(mb, b1, b2, slices, p, stream);
        if (st != FLUTE_OK) return st;
    }
    workspace_done(stream);
    return FLUTE_OK;
}

// Up to four weights of one width pair, group size and rotation over the same rows of A through the
// small-M kernel, in the given shape: one launch of each pre-pass and one (per stream) of the kernel.
flute_status gemm_rows(const flute_linear *ws, int count, const void *A, void *const *C, const int64_t *ldc, int M,
                       int64_t lda, int act_dtype, const GemmShape &shape, hipStream_t stream) {
    const flute_linear *w = ws;                         // what they share
    flute_status st;
    GemmParams p = {};
    p.nstreams = w->b2 > 0 ? 2 : 1;
    p.bits[0] = w->b1;
    p.bits[1] = w->b2;
    p.M = M;
    p.G = w->K / 64;
    p.out_bf16 = act_dtype == FLUTE_BF16;
    int tiles = 0;
    bool any_res = false;
    for (int i = 0; i < kGemmMaxSegs; ++i) {
        p.tile0[i] = i < count ? tiles : INT_MAX;
        if (i >= count) continue;
        GemmSeg &g = p.seg[i];
        g.q[0] = (const uint8_t *)ws[i].q1;
        g.q[1] = (const uint8_t *)ws[i].q2;
        g.lut[0] = (const uint16_t *)ws[i].lut1;
        g.lut[1] = (const uint16_t *)ws[i].lut2;
        g.gs = ws[i].group_size;
        g.lut_rows = ws[i].lut_rows;
        g.R = ws[i].R;
        g.resA = (const uint16_t *)ws[i].resA;
        g.bias = (const uint16_t *)ws[i].bias;
        g.C = C[i];
        g.ldc = ldc[i];
        g.vec_store = (ldc[i] % 8 == 0) && (((uintptr_t)C[i] & 15) == 0);
        any_res |= ws[i].R > 0;
        tiles += ws[i].N / 128;
    }
    p.mblk_total = (M + 15) / 16;

    // ---- grid and K split --------------------------------------------------------
    const int mchunks = (p.mblk_total + shape.mb * shape.mw - 1) / (shape.mb * shape.mw);
    const int64_t units = (int64_t)tiles * mchunks;
    p.mblk_pad = mchunks * shape.mb * shape.mw;
    const int64_t cap = (int64_t)kNumCU * shape.wg_per_cu;
    // K is split until the grid reaches one workgroup per CU, while every wavefront keeps
    // two tiles or more; with four blocks of rows per wavefront at most four ways, because
    // the workgroup that arrives last reads every 32 KB partial tile of its unit back
    // (measured at M = 64: 12288 -> 4096 29.7 us four ways, 36.4 us eight ways; 4096 -> 4096
    // 21.8 us four ways, 23.0 us two ways, 24.6 us eight ways).
    const int max_split = shape.mb == 1 ? 64 : 4;
    int ksplit = 1;
    while (units * ksplit * 2 <= cap && ksplit * 2 <= max_split &&
           p.G / (ksplit * 2) >= shape.kw * 2)
        ksplit *= 2;
    {
        const int v = tuning().gemm_ksplit;
        if (v >= 1 && v <= p.G) ksplit = v;
    }
    p.gper = (p.G + ksplit - 1) / ksplit;
    ksplit = (p.G + p.gper - 1) / p.gper;
    p.ksplit = ksplit;
    // Four blocks per wavefront and K ranges that start on a multiple of the k ways: the image is
    // written in the order the k ways want their blocks and they hand blocks to each other
    // instead of reducing through a tree (gemm_kernel.h; FLUTE_GEMM_NO_HANDOVER keeps the tree).
    p.scatter = 0;
    if (shape.mb == 4 && shape.kw * shape.mw == 8 && p.gper % shape.kw == 0 && !tuning().gemm_no_handover)
        p.scatter = shape.kw == 4 ? 1 : 2;
    const int block_xor = p.scatter;
    FLUTE_REQUIRE(mchunks <= 65535 && ksplit <= 65535, FLUTE_ERR_UNSUPPORTED,
                  "flute_gemm: M=%d exceeds the grid", M);

    // ---- workspace: [partial images][xb][Ap] -----------------------------------------
    const size_t image = (size_t)shape.mw * shape.mb * 8 * 64 * 4;
    const int zparts = ksplit * ((p.nstreams == 2 && shape.mb > 1) ? 2 : 1);
    const size_t p_floats = zparts > 1 ? (size_t)zparts * units * image : 0;
    const CoeffPlan coeff = plan_coeff(ws, count, M);
    size_t xb_floats = any_res ? coeff.floats() : 0;
    for (int i = 0; i < count; ++i) xb_floats += ((size_t)M * ws[i].R + 3) & ~(size_t)3;
    const size_t ap_floats = (size_t)p.G * 2 * p.mblk_pad * 64 * 4;
    const size_t rot_floats = w->signs ? ((size_t)M * w->K / 2 + 4) & ~(size_t)3 : 0;
    // bfloat16 activations presented as float16 operands: one power-of-two scale per row
    const bool scale_rows = act_dtype == FLUTE_BF16 && w->lut_dtype == FLUTE_F16;
    const size_t shift_floats = scale_rows ? ((size_t)M + 3) & ~(size_t)3 : 0;
    float *base = nullptr;
    int *tickets = nullptr;
    const size_t want_tickets = std::max((size_t)units, any_res ? coeff.tickets() : 0) + 1;
    st = get_workspace(p_floats + xb_floats + ap_floats + rot_floats + shift_floats + 64, want_tickets, stream, &base,
                       &tickets);
    if (st != FLUTE_OK) return st;
    p.P = base;
    p.tickets = tickets;
    float *xb = base + p_floats;
    u4_t *Ap = (u4_t *)(xb + xb_floats);
    p.Ap = Ap;
    int *rowshift = scale_rows
        ? (int *)(base + p_floats + xb_floats + ap_floats + rot_floats) : nullptr;
    auto launch_rowshift = [&](const void *rows, int64_t ld) -> flute_status {
        hipLaunchKernelGGL(gemm_rowshift_kernel, dim3(M), dim3(256), 0, stream,
                           (const uint16_t *)rows, ld, w->K, rowshift);
        FLUTE_HIP_CHECK(hipGetLastError());
        p.rowshift = rowshift;
        return FLUTE_OK;
    };
    // One block of rows per wavefront on the single-stream 4-bit fast path: the kernel reads
    // A itself (16-byte pieces of a row, put into operand order in registers), so the
    // pre-pass launch is dropped.  Needs 16-byte aligned rows; rotated rows are read the same way
    // (the rotation can write the image itself, but only without a residual and row scales).
    const bool direct = [&] {
        const int ngrp = w->group_size >= 128 ? 1 : 128 / w->group_size;
        return shape.mb == 1 && p.nstreams == 1 && w->b1 == 4 && ngrp <= 2 && !tuning().gemm_no_perm &&
               !tuning().gemm_no_direct;
    }();
    if (w->signs && !any_res && !scale_rows) {
        // the rotation writes the operand image itself: one launch instead of two
        FhtOperandOut image_out = {(uint32_t *)Ap, p.mblk_pad, (int)(w->lut_dtype == FLUTE_BF16), block_xor};
        st = fht_launch(A, lda, w->signs, w->awq, nullptr, 0, M, w->K, act_dtype, 0, w->rot_block,
                        stream, &image_out);
        if (st != FLUTE_OK) return st;
    } else {
        if (w->signs) {
            // the residual coefficients and the row scales need the rotated rows as rows:
            // rotated copy first, then the ordinary pre-pass on it
            void *Arot = (void *)(Ap + (size_t)p.G * 2 * p.mblk_pad * 64);
            st = fht_launch(A, lda, w->signs, w->awq, Arot, w->K, M, w->K, act_dtype, 0,
                            w->rot_block, stream, nullptr, rowshift);
            if (st != FLUTE_OK) return st;
            A = Arot;
            lda = w->K;
            p.rowshift = rowshift;                      // (the rotation knows its rows' largest exponents)
        } else if (scale_rows) {
            st = launch_rowshift(A, lda);
            if (st != FLUTE_OK) return st;
        }
        const int64_t total = (int64_t)p.G * 2 * p.mblk_pad * 64;
        const int blocks = (int)((total + 255) / 256 < 4096 ? (total + 255) / 256 : 4096);
        const bool rows16 = ((uintptr_t)A & 15) == 0 && lda % 8 == 0;
        if (direct && rows16) {
            p.A8 = (const u4_t *)A;
            p.lda8 = lda / 8;
            p.a_bf16 = act_dtype == FLUTE_BF16;
        } else if (rows16) {
            // 16-byte aligned rows: one coalesced 16-byte load per thread and a transpose
            // inside each quad (M = 256, K = 4096: 2.2 us against 5.2 us for the gathers)
            hipLaunchKernelGGL(gemm_prep_quad_kernel, dim3(blocks), dim3(256), 0, stream,
                               (const uint16_t *)A, Ap, M, lda, p.G, p.mblk_pad,
                               (int)(act_dtype == FLUTE_BF16), (int)(w->lut_dtype == FLUTE_BF16),
                               rowshift, (const uint32_t *)w->lut1,
                               (int)(((size_t)w->lut_rows << w->b1) * 2 / 64), block_xor);
        } else {
            hipLaunchKernelGGL(gemm_prep_kernel, dim3(blocks), dim3(256), 0, stream,
                               (const uint16_t *)A, Ap, M, lda, p.G, p.mblk_pad,
                               (int)(act_dtype == FLUTE_BF16), (int)(w->lut_dtype == FLUTE_BF16),
                               (int)((((uintptr_t)A & 3) == 0) && (lda % 2 == 0)), rowshift, block_xor);
        }
        FLUTE_HIP_CHECK(hipGetLastError());
    }
    if (any_res) {
        float *next = xb + coeff.floats(), *to[kGemmMaxSegs] = {};
        for (int i = 0; i < count; ++i) {
            if (ws[i].R == 0) continue;
            to[i] = next;
            p.seg[i].xb = next;
            p.seg[i].vec_res = ws[i].R % 8 == 0 && ((uintptr_t)ws[i].resA & 15) == 0 && ((uintptr_t)next & 15) == 0;
            next += ((size_t)M * ws[i].R + 3) & ~(size_t)3;
        }
        st = launch_coeff(coeff, ws, count, A, lda, to, M, p.out_bf16, xb, tickets, stream);
        if (st != FLUTE_OK) return st;
    }

    // Two streams with four blocks per wavefront: one launch per stream through the
    // single-stream kernels (the two-stream kernel does not fit the register file at
    // that size); both write partial tiles and the last workgroup of the second launch
    // folds everything, exactly as a K split does.
    const bool per_stream = p.nstreams == 2 && shape.mb > 1;
    const int passes = per_stream ? 2 : 1;
    const dim3 grid(tiles, mchunks, ksplit);
    for (int pass = 0; pass < passes; ++pass) {
        GemmParams q = p;
        if (per_stream) {
            q.nstreams = 1;
            for (int i = 0; i < count; ++i) {
                q.seg[i].q[0] = p.seg[i].q[pass];
                q.seg[i].lut[0] = p.seg[i].lut[pass];
            }
            q.bits[0] = p.bits[pass];
        }
        q.z_base = pass * ksplit;
        q.ztotal = passes * ksplit;
        const int lds = plan_lds(q, shape);
        FLUTE_REQUIRE(lds <= kLdsPerCU, FLUTE_ERR_UNSUPPORTED,
                      "flute_gemm: %d bytes of LDS exceed the %d of one CU", lds, kLdsPerCU);
        const int bf16 = w->lut_dtype == FLUTE_BF16;
        st = count > 1 ? gemm_launch_segs(bf16, shape.mb, shape.mw, q, grid, lds, stream)
             : bf16    ? launch_gemm_shape<true, false>(shape.mb, shape.mw, q, grid, lds, stream)
                       : launch_gemm_shape<false, false>(shape.mb, shape.mw, q, grid, lds, stream);
        if (st != FLUTE_OK) return st;
    }
    workspace_done(stream);
    return FLUTE_OK;
}

}  // namespace
}  // namespace flute

using namespace flute;

extern "C" flute_status flute_gemm(const flute_linear *w, const void *A, void *C, int M,
                                   int64_t lda, int64_t ldc, int act_dtype, void *stream_) {
    flute_status st = validate_linear(w, 1, "flute_gemm");
    if (st != FLUTE_OK) return st;
    FLUTE_REQUIRE(act_dtype == FLUTE_F16 || act_dtype == FLUTE_BF16, FLUTE_ERR_INVALID,
                  "flute_gemm: activations must be float16 or bfloat16");
    FLUTE_REQUIRE(M >= 0, FLUTE_ERR_INVALID, "flute_gemm: M must be >= 0 (got %d)", M);
    if (M == 0) return FLUTE_OK;
    FLUTE_REQUIRE(A != nullptr && C != nullptr, FLUTE_ERR_INVALID,
                  "flute_gemm: A and C must not be NULL");
    FLUTE_REQUIRE(lda >= w->K && ldc >= w->N, FLUTE_ERR_INVALID,
                  "flute_gemm: row strides must cover a row (lda=%lld < K=%d or ldc=%lld < N=%d)",
                  (long long)lda, w->K, (long long)ldc, w->N);
    FLUTE_REQUIRE(((uintptr_t)A & 1) == 0 && ((uintptr_t)C & 1) == 0, FLUTE_ERR_INVALID,
                  "flute_gemm: A and C must be 2-byte aligned");
    hipStream_t stream = (hipStream_t)stream_;

    const GemmShape shape = choose_gemm_shape(M, w->N / 128, w->q1_bytes + (w->b2 > 0 ? w->q2_bytes : 0), w->K / 64,
                                              w->b2 > 0, fast_stream(*w));
    const int streams = w->b2 > 0 ? 2 : 1;
    const WidePlan wide = choose_wide(M, w->N / 128, w->K / 64, streams,
                                      other_forms(M, w->N / 128, w->K / 64, streams, w->b1 == 4, shape), shape);
    if (wide.rows) return gemm_wide(w, 1, A, &C, &ldc, M, lda, act_dtype, wide, stream);
    return gemm_rows(w, 1, A, &C, &ldc, M, lda, act_dtype, shape, stream);
}

extern "C" flute_status flute_gemm_multi(const flute_linear *ws, int count, const void *A, void *const *C,
                                         const int64_t *ldc, int M, int64_t lda, int act_dtype, void *stream) {
    FLUTE_REQUIRE(ws && C && ldc && count >= 1 && count <= kWideMaxSegs, FLUTE_ERR_INVALID,
                  "flute_gemm_multi: 1..%d weights", kWideMaxSegs);
    for (int i = 0; i < count; ++i) {
        flute_status st = validate_linear(&ws[i], 1, "flute_gemm_multi");
        if (st != FLUTE_OK) return st;
        FLUTE_REQUIRE(ws[i].K == ws[0].K && ws[i].lut_dtype == ws[0].lut_dtype, FLUTE_ERR_INVALID,
                      "flute_gemm_multi: the weights must share K and the LUT's type");
        FLUTE_REQUIRE(M <= 0 || (C[i] && ((uintptr_t)C[i] & 1) == 0 && ldc[i] >= ws[i].N), FLUTE_ERR_INVALID,
                      "flute_gemm_multi: output %d must be 2-byte aligned rows of N or more", i);
    }
    FLUTE_REQUIRE(act_dtype == FLUTE_F16 || act_dtype == FLUTE_BF16, FLUTE_ERR_INVALID,
                  "flute_gemm_multi: activations must be float16 or bfloat16");
    FLUTE_REQUIRE(M >= 0 && (M == 0 || (A && ((uintptr_t)A & 1) == 0 && lda >= ws[0].K)), FLUTE_ERR_INVALID,
                  "flute_gemm_multi: A must be 2-byte aligned rows of K or more");
    if (M == 0) return FLUTE_OK;
    // One launch of the many-row kernel where the weights together are better off there than each
    // in its own best form: they share the activations' image, and a chip that one weight's tiles
    // leave partly idle (or cut into slices of K) is filled.  Gate and up, 2 x 4096 -> 12288, M = 509:
    // 2 x 65.8 us in two slices each, 98.7 together.
    // Small calls share everything in front of the kernel, and its launch.
    const int streams = ws[0].b2 > 0 ? 2 : 1, G = ws[0].K / 64;
    bool widths = true, all = true;
    int tiles = 0;
    int64_t bytes = 0;
    for (int i = 0; i < count; ++i) {
        const flute_linear &w = ws[i];
        widths &= w.b1 == ws[0].b1 && w.b2 == ws[0].b2;
        all &= w.group_size == ws[0].group_size && w.signs == ws[0].signs && w.awq == ws[0].awq &&
               w.rot_block == ws[0].rot_block;
        tiles += w.N / 128;
        bytes += w.q1_bytes + (w.b2 > 0 ? w.q2_bytes : 0);
    }
    if (widths) {
        const GemmShape shape = choose_gemm_shape(M, tiles, bytes, G, streams == 2, fast_stream(ws[0]));
        const WidePlan plan = choose_wide(M, tiles, G, streams, other_forms(M, tiles, G, streams, ws[0].b1 == 4, shape),
                                          shape);
        if (plan.rows) return gemm_wide(ws, count, A, C, ldc, M, lda, act_dtype, plan, (hipStream_t)stream);
        if (all) return gemm_rows(ws, count, A, C, ldc, M, lda, act_dtype, shape, (hipStream_t)stream);
    }
    for (int i = 0; i < count; ++i) {
        flute_status st = flute_gemm(&ws[i], A, C[i], M, lda, ldc[i], act_dtype, stream);
        if (st != FLUTE_OK) return st;
    }
    return FLUTE_OK;
}

namespace flute {
namespace {

// h = silu(g) * u, eight values a thread, fp32 inside, one rounding.  Bound by its three streams.
__global__ void __launch_bounds__(256) silu_mul_kernel(const uint16_t *g, const uint16_t *u, uint16_t *h, int64_t pieces,
                                                       int bf16) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < pieces; i += (int64_t)gridDim.x * 256) {
        const u4_t a = *(const u4_t *)(g + i * 8), b = *(const u4_t *)(u + i * 8);
        u4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t r = 0;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const uint16_t x = (uint16_t)(a[e] >> (16 * s)), y = (uint16_t)(b[e] >> (16 * s));
                const float f = bf16 ? bf2f(x) : h2f(x);
                const float t = f / (1.0f + expf(-f)) * (bf16 ? bf2f(y) : h2f(y));
                r |= (uint32_t)round_act(t, bf16) << (16 * s);
            }
            o[e] = r;
        }
        *(u4_t *)(h + i * 8) = o;
    }
}

}  // namespace
}  // namespace flute

extern "C" flute_status flute_silu_mul(const void *g, const void *u, void *h, int64_t count, int act_dtype, void *stream) {
    FLUTE_REQUIRE(act_dtype == FLUTE_F16 || act_dtype == FLUTE_BF16, FLUTE_ERR_INVALID,
                  "flute_silu_mul: float16 or bfloat16");
    FLUTE_REQUIRE(count >= 0 && count % 8 == 0, FLUTE_ERR_INVALID, "flute_silu_mul: count must be a multiple of 8");
    if (count == 0) return FLUTE_OK;
    FLUTE_REQUIRE(g && u && h && (((uintptr_t)g | (uintptr_t)u | (uintptr_t)h) & 15) == 0, FLUTE_ERR_INVALID,
                  "flute_silu_mul: g, u and h must be 16-byte aligned");
    const int64_t blocks = (count / 8 + 255) / 256;
    hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t *)g, (const uint16_t *)u, (uint16_t *)h, count / 8, (int)(act_dtype == FLUTE_BF16));
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

#ifdef FLUTE_STAMPS
// Instrumented builds only: where the kernels write their phase times (NULL switches them off).
extern "C" int flute_debug_stamps(void *buf) {
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(flute::g_gemm_stamps), &buf, sizeof(buf));
}
#endif
