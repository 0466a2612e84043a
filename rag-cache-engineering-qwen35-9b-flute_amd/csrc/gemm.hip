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
flute_status gemm_few_f16(int mb, const GemmParams &p, dim3 grid, hipStream_t stream);
flute_status gemm_few_bf16(int mb, const GemmParams &p, dim3 grid, hipStream_t stream);
flute_status gemm_few_f16_segs(int mb, const GemmParams &p, dim3 grid, hipStream_t stream);
flute_status gemm_few_bf16_segs(int mb, const GemmParams &p, dim3 grid, hipStream_t stream);
flute_status gemm_wide_f16(int mb, int b1, int b2, int slices, const WideParams &p, hipStream_t stream);
flute_status gemm_wide_bf16(int mb, int b1, int b2, int slices, const WideParams &p, hipStream_t stream);

namespace {

struct GemmShape {
    int mb, kw, mw;       // 16-row blocks per wavefront, k ways, m ways
    int wg_per_cu;        // workgroups the policy expects to be resident per CU
};

// Slices of K of 64-row and 128-row workgroups: split until the grid reaches one workgroup per CU, while every
// wavefront keeps two tiles or more, at most four, because the workgroup that arrives
// last reads every partial tile of its unit back (64 rows, M = 64: 12288 -> 4096 29.7 us four ways,
// 36.4 eight ways; 4096 -> 4096 21.8 four ways, 23.0 two ways, 24.6 eight ways).
int slices_of_k(int64_t units, int G, const GemmShape &shape) {
    int ks = 1;
    while (units * ks * 2 <= (int64_t)kNumCU * shape.wg_per_cu && ks < 4 && G / (ks * 2) >= shape.kw * 2) ks *= 2;
    return ks;
}

// Width pairs (the wider first) that the few-row kernel takes in one launch: all but (4, 4), whose tables
// and staged codes take 192 KB of LDS (a launch per stream, M = 8, 4096 -> 4096 16.3 us; the kernel before it,
// which took both with half of the tables' replicas, 20.9).
bool few_takes(int b1, int b2) { return !(b1 == 4 && b2 == 4); }

// Microseconds of a call (one round = a workgroup per CU; `turns` = K tiles of a wavefront), fitted to
// measurements on tiles of 16 and 32 rows: a fixed part, what some calls of 32 rows have in front (few_reads)
// and, per round, prologue, sums and epilogue, then what a wavefront's tile costs.
// 16 and 32 rows, us: M = 32, 4096 -> 12288 13.2 / 14.4; M = 64 25.6 / 17.1; M = 200, 4096 -> 4096 24.0 / 16.6; over
// random shapes and against the other kernels: profiles/gemm_shape_choice.txt.  (A launch in front of 16-row
// workgroups is not in it.)
// The slices of K are those of the least estimate: a slice more saves turns and costs the last arrival its share
// of the partial tiles, which it reads four at a time, slower the more workgroups do.  Any number of them, so that
// turns come out whole, down to one a wavefront.  us with 1, 2, 4, 8, 12, 16 slices: M = 8, 12288 -> 1024 29.0, 18.2,
// 11.9, 9.6, 9.3, 10.0; 2048 -> 1024 7.7, 7.2, 6.3, 6.8, 7.6, 8.5 (other shapes: same file).
struct FewPlan {
    double us;
    int slices;
};
FewPlan plan_few(int mb, int M, int tiles, int G, int b1, int b2) {
    static const double tile_us[5] = {0.0, 0.6, 0.75, 1.2, 1.15};
    const int64_t units = (int64_t)tiles * ((M + 16 * mb - 1) / (16 * mb));
    const double tile = (tile_us[b1] + tile_us[b2]) * (mb == 1 ? 1.0 : 1.09);
    const double launches = b2 && !few_takes(std::max(b1, b2), std::min(b1, b2)) ? 2.0 : 1.0;
    FewPlan best = {1e30, 1};
    for (int ks = 1; ks <= 32 && (ks == 1 || (units * ks <= kNumCU && ks < G)); ++ks) {
        const int turns = ((G + ks - 1) / ks + 7) / 8;
        const int64_t rounds = (units * ks + kNumCU - 1) / kNumCU;
        const double share = 0.6 + 0.9 * (double)(units * ks) / kNumCU;
        const double fold = ks == 1 ? 0.0 : mb == 1 ? 0.6 + 0.65 * ((ks + 3) / 4) * share : 0.4 + 1.0 * ((ks + 3) / 4) * share;
        const double us = (mb == 1 ? 1.5 : 3.5) + rounds * ((mb == 1 ? 4.0 : 5.0) * launches + tile * turns) + fold * launches;
        if (us < best.us) best = {us, ks};
    }
    return best;
}

// The same for 64-row (in one round) and 128-row workgroups of gemm_kernel.h: 8 us + 0.26 (0.43) a tile
// per round, two streams are two launches, other widths 15 % more.
GemmShape other_shape(int M, int tiles) {
    return (int64_t)tiles * ((M + 63) / 64) <= kNumCU ? GemmShape{4, 8, 1, 1} : GemmShape{4, 4, 2, 1};
}
double other_us(int M, int tiles, int G, int streams, bool four_bit) {
    const GemmShape other = other_shape(M, tiles);
    const int rows = other.mb * other.mw * 16;
    const int64_t units = (int64_t)tiles * ((M + rows - 1) / rows);
    const int ks = slices_of_k(units, G, other);
    const double per_tile = (other.mw == 1 ? 0.26 : 0.43) * (four_bit && streams == 1 ? 1.0 : 1.15);
    return streams * (double)((units * ks + kNumCU - 1) / kNumCU) * (8.0 + per_tile * G / ks) + (ks > 1 ? 2.5 * ks : 0.0);
}

// Rows of A per workgroup and what the call then takes.  One or two 16-row blocks per wavefront with
// eight k ways (gemm_few_kernel.h) while there are few rows, else four blocks: 64 rows per workgroup
// with eight k ways while that fits the device in one round, else 128 rows (two m groups, four k ways);
// further rows go to gridDim.y.  The tables plus staging take most of a CU's LDS, so one workgroup per
// CU is resident.  FLUTE_GEMM_ROWS = 16, 32, 64 or 128 forces the shape (a tuning and test knob, like
// FLUTE_GEMV_RW), 256 or 512 the many-row kernel.
GemmShape choose_gemm_shape(int M, int tiles, int G, int b1, int b2, double &us) {
    const int v = tuning().gemm_rows;
    const double other = other_us(M, tiles, G, b2 ? 2 : 1, b1 == 4);
    us = other;
    if (v == 16) return {1, 8, 1, 1};
    if (v == 32) return {2, 8, 1, 1};
    if (v == 64) return {4, 8, 1, 1};
    if (v == 128) return {4, 4, 2, 1};
    const double few1 = plan_few(1, M, tiles, G, b1, b2).us, few2 = plan_few(2, M, tiles, G, b1, b2).us;
    // (row blocks that gridDim.y holds)
    const bool fits1 = M <= 65535 * 16, fits2 = M <= 65535 * 32;
    if (M <= 16 || (fits1 && few1 <= few2 && few1 < other)) {
        us = few1;
        return {1, 8, 1, 1};
    }
    // The estimate of 64 rows is up to 2.5 us short where the two are close and a workgroup has few
    // tiles (less with more: M = 256 and 512, 12288 -> 4096 stay).  64 and 32 rows: M = 225,
    // 5248 -> 2816 29.2 / 23.3 us; M = 300, 6912 -> 1792 32.2 / 27.6; M = 39, 1664 -> 12288 18.2 / 14.5;
    // M = 672, 10432 -> 896 43.2 / 40.1; (3, 3) bits, M = 218, 1408 -> 6912 42.5 / 29.1.
    const GemmShape shape = other_shape(M, tiles);
    const double short_by = shape.mw == 1
        ? std::min(2.5, std::max(-1.5, 6.5 - G / slices_of_k((int64_t)tiles * ((M + 63) / 64), G, shape) / 16.0)) : -1.5;
    if (fits2 && few2 < other + short_by) {
        // 1.5 more against the many-row kernel, whose estimate has a launch in front as many of these calls have.
        // Over 40 random shapes beside that boundary the choice loses 1.6 % on the mean against the better of the two,
        // with 0 ... 4 us in its place 1.5, 1.3 (1 us), 1.6 (2), 1.2 (3), 1.4 (4): the line lies anywhere there.  The
        // estimates miss most where many turns come in several rounds: M = 338, 4992 -> 8064, (1, 4) bits 102.8 us, 256
        // rows 86.6 (profiles/gemm_shape_choice.txt).
        us = few2 + 1.5;
        return {2, 8, 1, 1};
    }
    return other_shape(M, tiles);
}

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

// The pre-pass of rows of A: coefficients of `count` weights (those with a residual; plan NULL: none)
// and what `image` asks for (blocks 0: nothing), in one launch.  image.up: the rows are silu(A) * up.
flute_status launch_pre(const CoeffPlan *plan, const flute_linear *ws, int count, const void *A, int64_t lda,
                        float *const *xb, int M, int is_bf16, float *part, int *tickets, ImageParams image,
                        hipStream_t stream) {
    CoeffParams p = {};
    int n = 0, ranks = 0;
    if (plan) {
        p.A = (const uint16_t *)A;
        p.up = image.up;
        p.lda = lda;
        p.M = M;
        p.K = ws[0].K;
        p.aligned = ((uintptr_t)A & 15) == 0 && lda % 8 == 0;
        p.kper = (p.K / 32 + plan->slices - 1) / plan->slices * 32;
        p.rows = plan->rows;
        p.ranks = plan->ranks;
        p.slices = plan->slices;
        p.part = part;
        p.tickets = tickets;
        for (int i = 0; i < count; ++i) {
            if (ws[i].R == 0) continue;
            p.resB[n] = (const uint16_t *)ws[i].resB;
            p.xb[n] = xb[i];
            p.R[n] = ws[i].R;
            p.rank0[n++] = ranks;
            p.aligned &= ((uintptr_t)ws[i].resB & 15) == 0;
            ranks += (ws[i].R + 15) / 16;
        }
    }
    for (; n < kGemmMaxSegs; ++n) p.rank0[n] = INT_MAX;
    // Coefficients and the search for scales are work for sixteen wavefronts; a small image alone is
    // spread over the chip in workgroups of four.  A share of the image is four rows, or a 1 KB block a
    // wavefront; workgroups beyond those resident at once would only queue (4096 x 12288: 512 workgroups
    // of sixteen wavefronts 33 us, 2048 39, 6144 44; 2048 of four 36).
    const int64_t ncoeff = (int64_t)p.rows * p.ranks * p.slices;
    const int waves = ncoeff || image.find || (int64_t)image.blocks * image.segs > 32 * kNumCU ? 16 : 4;
    // (whole rows: two a workgroup where four leave CUs without one.  The block 2048/8192 on 300 rows 80.5 us with
    // four, 74.9 with two; 509 rows, 12288 -> 4096 64.2 and 63.1)
    if (image.find) image.find = (int64_t)image.blocks * 4 < kNumCU ? 2 : 4;
    const int64_t shares = image.find ? (int64_t)image.blocks * (16 / image.find)
                                      : ((int64_t)image.blocks * image.segs + waves - 1) / waves;
    const int64_t grid = ncoeff + std::min<int64_t>(shares, 32 / waves * kNumCU);
    FLUTE_REQUIRE(grid <= 0x7fffffff, FLUTE_ERR_UNSUPPORTED, "flute_gemm: %lld workgroups exceed the grid", (long long)grid);
    if (grid == 0) return FLUTE_OK;
    const dim3 threads(64 * waves), blocks((unsigned)grid);
    if (image.up) {
        if (is_bf16) hipLaunchKernelGGL((gemm_pre_kernel<true, true>), blocks, threads, 0, stream, p, image);
        else hipLaunchKernelGGL((gemm_pre_kernel<false, true>), blocks, threads, 0, stream, p, image);
    } else if (is_bf16) {
        hipLaunchKernelGGL((gemm_pre_kernel<true, false>), blocks, threads, 0, stream, p, image);
    } else {
        hipLaunchKernelGGL((gemm_pre_kernel<false, false>), blocks, threads, 0, stream, p, image);
    }
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

// Scales of bfloat16 rows by a launch of their own (rows that gemm_pre_kernel does not look through).
flute_status launch_rowshift(const void *rows, int64_t ld, int M, int K, int *shift, hipStream_t stream) {
    hipLaunchKernelGGL(gemm_rowshift_kernel, dim3(M), dim3(256), 0, stream, (const uint16_t *)rows, ld, K, shift);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

// LDS plan of one launch of gemm_kernel, one stream: the pair table (+ staging on the fast path), sized
// against the reduction tree and the totals tile that reuse the same memory afterwards.
// 4 bits with at most two LUT groups per 128-row tile get 64-lane replication (256 bytes per entry,
// 64 KB per group, table at LDS offset 0: the layout the one-instruction address needs).  Everything
// else: as much replication as the budget allows, 32 lanes at most.
int plan_lds(GemmParams &p, const GemmShape &shape) {
    const int ngrp = p.seg[0].gs >= 128 ? 1 : 128 / p.seg[0].gs;
    const bool perm = p.bits[0] == 4 && ngrp <= 2 && !tuning().gemm_no_perm;
    const int table_budget = 96 * 1024, entries = ngrp << (2 * p.bits[0]);
    int rl = 5;
    while (rl > 0 && (entries << rl) * 4 > table_budget) --rl;
    if (perm) rl = 6;
    p.rep_log2[0] = rl;
    p.tab_off[0] = 0;
    int lds_tables = (entries << rl) * 4;
    p.lean = 0;
    if (perm) {                                  // per-wavefront tile staging behind the table
        // one LUT group per tile: the lean loop, whose tiles go straight into two staging buffers
        // per wavefront
        p.lean = ngrp == 1 && !tuning().gemm_no_lean;
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
    const int rows = shape.mw * shape.mb * 16;
    bool residual = false;
    for (const GemmSeg &g : p.seg) residual |= g.R > 0;
    const int lds_tile = gemm_residual_offset(rows) + (residual ? rows * 132 * 4 : 0);
    int lds = lds_tables > lds_reduce ? lds_tables : lds_reduce;
    if (lds_tile > lds) lds = lds_tile;
    // the hand-overs between the k ways: eight 16 KB areas, then eight of 8 KB behind the totals tile, in part those
    // of the residual's tile
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

// The many-row kernel or the others (`us`), and its shape.  Each form's time is a line in what it has to
// do, in microseconds, fitted to measurements (4-bit stream, bfloat16; `steps` = 64-k tiles of all
// streams that a workgroup takes, `rounds` = workgroups / 256 CUs, rounded up; several weights in one
// launch: `tiles` counts theirs):
//   512-row workgroups                    14 a round + 0.95 ... 1.35 a step (the clock falls as the chip
//                                         fills); slices of K cost 5 each (256 KB written, read)
//   256-row workgroups                    11 a round + 0.60 ... 0.80 a step; slices 2.5 each
// e.g. 128-row, 512-row and 256-row workgroups at M = 1024, 4096 -> 12288: 120 / 92 / 118 us (estimated
// 107 / 94 / 124); M = 512: 74 / 61 (two slices) / 61; M = 512, 12288 -> 4096: 59 / 77 (four) / 65
// (four), the others stay; two streams (4, 1) at M = 1024, 4096 -> 12288: 263 / 165 / 190; (3, 3) at
// M = 600, 4096 -> 4096: 32-row workgroups 80, 256-row ones in two slices 61 (estimated 64).
WidePlan choose_wide(int M, int tiles, int G, int streams, double us_others) {
    {
        const int v = tuning().gemm_rows;
        if (v == 512 || v == 256) {
            const int k = tuning().gemm_ksplit;
            return {v, k > 1 ? (k < G ? k : G) : 1};
        }
        if (v) return {0, 1};
    }
    if (M <= 16) return {0, 1};
    double best = us_others;
    WidePlan plan = {0, 1};
    for (int rows = 512; rows >= 256; rows /= 2) {
        const int64_t units = (int64_t)tiles * ((M + rows - 1) / rows);
        for (int ks = 1; ks <= 8 && G / ks >= 8; ks *= 2) {
            const int64_t groups = units * ks, rounds = (groups + kNumCU - 1) / kNumCU;
            const double fill = groups < kNumCU ? (double)groups / kNumCU : 1.0;
            const double step = rows == 512 ? 0.95 + 0.40 * fill : 0.60 + 0.20 * fill;
            const double us = rounds * ((rows == 512 ? 14.0 : 11.0) + step * streams * ((G + ks - 1) / ks)) +
                              (ks > 1 ? (rows == 512 ? 5.0 : 2.5) * ks : 0.0);
            if (us < best) {
                best = us;
                plan = {rows, ks};
            }
        }
    }
    return plan;
}

// Up to four weights over the same rows of A in one launch: C[i] = A @ W[i]^T (+ residual, bias).  They
// share their widths, LUT's type and K.
// up: the rows are silu(A) * up (rows that takes_silu allows, of one stride).
flute_status gemm_wide(const flute_linear *ws, int count, const void *A, void *const *C, const int64_t *ldc, int M,
                       int64_t lda, int act_dtype, WidePlan plan, hipStream_t stream, const void *up = nullptr) {
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
    // the weights of each image side by side, and their coefficients
    flute_linear of[kWideMaxSegs][kWideMaxSegs];
    int members[kWideMaxSegs][kWideMaxSegs], ofs[kWideMaxSegs] = {};
    CoeffPlan coeff[kWideMaxSegs];
    for (int i = 0; i < count; ++i) {
        const int k = image_of[i];
        members[k][ofs[k]] = i;
        of[k][ofs[k]++] = ws[i];
        xb_floats += up4((size_t)M * ws[i].R);
        tiles += ws[i].N / 128;
    }
    for (int k = 0; k < images; ++k) {
        coeff[k] = plan_coeff(of[k], ofs[k], M);
        part_xb = std::max(part_xb, coeff[k].floats());
        want_tickets = std::max(want_tickets, coeff[k].tickets());
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
    float *xb[kWideMaxSegs] = {};
    for (int i = 0; i < count; ++i) {
        if (ws[i].R == 0) continue;
        xb[i] = next;
        next += up4((size_t)M * ws[i].R);
    }
    for (int k = 0; k < images; ++k) {
        const flute_linear &w = ws[owner[k]];
        const void *rows = A;
        int64_t ldr = lda;
        int *row_shift = nullptr;
        if (w.signs) {
            // (the rotation knows its rows' largest exponents)
            row_shift = scale_rows ? (int *)(next + rot_floats) : nullptr;
            st = fht_launch(A, lda, w.signs, w.awq, next, K, M, K, act_dtype, 0, w.rot_block, stream, nullptr, row_shift);
            if (st != FLUTE_OK) return st;
            rows = next;
            ldr = K;
            next += rot_floats;
        } else if (scale_rows) {
            row_shift = (int *)next;
        }
        if (scale_rows) next += shift_floats;
        shift[k] = row_shift;
        image[k] = (const u4_t *)next;
        ImageParams im = {};
        im.A = (const uint16_t *)rows;
        im.up = (const uint16_t *)up;
        im.Ap = (u4_t *)next;
        im.lda = ldr;
        im.rowshift = row_shift;
        im.M = M;
        im.segs = 2 * G;
        im.blocks = (M + 15) / 16;
        im.mblk = mblk;
        im.in_bf16 = out_bf16;
        im.out_bf16 = lut_dtype == FLUTE_BF16;
        im.wide = 1;
        next += image_floats;
        const bool find = scale_rows && !w.signs, rows16 = ((uintptr_t)rows & 15) == 0 && ldr % 8 == 0;
        im.find = find && rows16 && K <= find_reach();
        if (find && !im.find) {
            st = launch_rowshift(rows, ldr, M, K, row_shift, stream);
            if (st != FLUTE_OK) return st;
        }
        if (!rows16) {
            const int64_t blocks = (int64_t)im.segs * im.blocks;
            const int grid = (int)((blocks + 3) / 4 < 8192 ? (blocks + 3) / 4 : 8192);
            hipLaunchKernelGGL(gemm_image_kernel, dim3(grid), dim3(256), 0, stream, im.A, im.Ap, M, ldr, im.segs, mblk,
                               im.in_bf16, im.out_bf16, (const int *)row_shift);
            FLUTE_HIP_CHECK(hipGetLastError());
            im.blocks = 0;
        }
        // (weights of different rotations have different rows: a launch each)
        float *to[kWideMaxSegs];
        for (int j = 0; j < ofs[k]; ++j) to[j] = xb[members[k][j]];
        st = launch_pre(coeff[k].ranks ? &coeff[k] : nullptr, of[k], ofs[k], rows, ldr, to, M, out_bf16, xb_part, tickets,
                        im, stream);
        if (st != FLUTE_OK) return st;
    }
    WideParams p = {};
    p.nsegs = count;
    p.M = M;
    p.G = G;
    p.mblk = mblk;
    p.mtiles = mtiles;
    p.gper = gper;
    p.out_bf16 = out_bf16;
    p.P = base;
    p.tickets = tickets;
    // the sum does not depend on the order of the streams beyond fp32 rounding: the wider first
    const bool swap = ws[0].b2 > ws[0].b1;
    for (int i = 0; i < count; ++i) {
        const flute_linear &w = ws[i];
        WideSeg &g = p.seg[i];
        g.q[0] = (const uint8_t *)(swap ? w.q2 : w.q1);
        g.q[1] = (const uint8_t *)(swap ? w.q1 : w.q2);
        g.lut[0] = (const uint16_t *)(swap ? w.lut2 : w.lut1);
        g.lut[1] = (const uint16_t *)(swap ? w.lut1 : w.lut2);
        g.Ap = image[image_of[i]];
        g.rowshift = shift[image_of[i]];
        g.xb = xb[i];
        g.resA = (const uint16_t *)w.resA;
        g.bias = (const uint16_t *)w.bias;
        g.C = C[i];
        g.ldc = ldc[i];
        g.tile0 = p.ntiles;
        g.gs = w.group_size;
        g.lut_rows = w.lut_rows;
        g.R = w.R;
        g.vec_store = (ldc[i] % 8 == 0) && (((uintptr_t)C[i] & 15) == 0);
        p.ntiles += w.N / 128;
    }
    const int b1 = swap ? ws[0].b2 : ws[0].b1, b2 = swap ? ws[0].b1 : ws[0].b2;
    st = lut_dtype == FLUTE_BF16 ? gemm_wide_bf16(mb, b1, b2, slices, p, stream)
                                 : gemm_wide_f16(mb, b1, b2, slices, p, stream);
    if (st != FLUTE_OK) return st;
    workspace_done(stream);
    return FLUTE_OK;
}

// Whether 16-row workgroups that read A themselves look for their rows' scales too, instead of a launch in front
// (3 us of the device and as much of the host): every workgroup reads whole rows for it, sixteen of 12288 columns
// in about those 3 us.  The launch in front and this, us a call: M = 8, 4096 -> 12288 14.6 / 12.5; M = 16 14.9 / 13.5;
// M = 2, 12288 -> 1024 13.8 / 11.3; M = 16, 12288 -> 4096 16.0 / 16.0; M = 6, 1152 -> 512, (2, 3) bits 12.0 / 10.2.
bool few_finds(int M, int K, int64_t workgroups) {
    const int64_t rounds = (workgroups + kNumCU - 1) / kNumCU;
    return rounds * std::min(M, 16) * K <= 16 * 12288;
}

// Whether workgroups of few rows read A themselves.  Sixteen rows always do.  Thirty-two do where that leaves no
// launch in front, and where a launch that only looks for scales in few, long rows is the shorter for it; beside
// coefficients of more ranks (few_coeff) the image costs nothing, and bfloat16 rows in front of a float16 LUT cost
// each turn of the loop their conversions (0.3 us; six turns bear them).  The image and A itself, us a call: M = 200,
// 4096 -> 4096 19.5 / 16.6; bfloat16 rows, float16 LUT: M = 48, 12288 -> 4096, (4, 1) bits, six turns 29.0 / 27.0;
// M = 64, 4096 -> 12288, eight turns 20.0 / 21.3 (both sides of other shapes: profiles/gemm_shape_choice.txt).
bool few_reads(const GemmShape &shape, bool scale_rows, bool rotated, int K, int gper) {
    if (shape.mb == 1) return true;
    return !scale_rows || ((rotated || K > 8192) && (gper + 7) / 8 <= 6);
}

// Residuals whose coefficients the few-row kernel can form: one operand of ranks.
bool few_coeff(const flute_linear &w) { return w.R > 0 && w.R <= 16 && ((uintptr_t)w.resB & 15) == 0; }

// Up to four weights of one width pair, group size and rotation over the same rows of A through the
// small-M kernel, in the given shape: one launch of each pre-pass and one (per stream) of the kernel.
// up: as gemm_wide's.
flute_status gemm_rows(const flute_linear *ws, int count, const void *A, void *const *C, const int64_t *ldc, int M,
                       int64_t lda, int act_dtype, const GemmShape &shape, hipStream_t stream, const void *up = nullptr) {
    const flute_linear *w = ws;                         // what they share
    flute_status st;
    GemmParams p = {};
    p.nstreams = w->b2 > 0 ? 2 : 1;
    // (the sum does not depend on the order of the streams beyond fp32 rounding: the wider first)
    const bool few = shape.mb <= 2, swap = few && w->b2 > w->b1;
    p.bits[0] = swap ? w->b2 : w->b1;
    p.bits[1] = swap ? w->b1 : w->b2;
    p.M = M;
    p.G = w->K / 64;
    p.out_bf16 = act_dtype == FLUTE_BF16;
    int tiles = 0;
    bool any_res = false;
    for (int i = 0; i < kGemmMaxSegs; ++i) {
        p.tile0[i] = i < count ? tiles : INT_MAX;
        if (i >= count) continue;
        GemmSeg &g = p.seg[i];
        g.q[swap] = (const uint8_t *)ws[i].q1;
        g.q[!swap] = (const uint8_t *)ws[i].q2;
        g.lut[swap] = (const uint16_t *)ws[i].lut1;
        g.lut[!swap] = (const uint16_t *)ws[i].lut2;
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
    int ksplit = few ? plan_few(shape.mb, M, tiles, p.G, p.bits[0], p.nstreams == 2 ? p.bits[1] : 0).slices
                     : slices_of_k(units, p.G, shape);
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
    // Two streams where no kernel takes both (four blocks of rows per wavefront: they do not fit the
    // register file; twice 4 bits): one launch per stream, both write partial
    // tiles and the last workgroup of the second launch folds everything, exactly as a K split does.
    const bool per_stream = p.nstreams == 2 && !(few && few_takes(p.bits[0], p.bits[1]));
    const int zparts = ksplit * (per_stream ? 2 : 1);
    const size_t p_floats = zparts > 1 ? (size_t)zparts * units * image : 0;
    // bfloat16 activations presented as float16 operands: one power-of-two scale per row
    const bool scale_rows = act_dtype == FLUTE_BF16 && w->lut_dtype == FLUTE_F16;
    const bool rows16 = w->signs || (((uintptr_t)A & 15) == 0 && lda % 8 == 0);
    // (float16 rows in front of a bfloat16 LUT are converted by the image: the kernel converts the other pair only)
    const bool narrows = act_dtype == FLUTE_F16 && w->lut_dtype == FLUTE_BF16;
    const bool reads = few && rows16 && !narrows && (w->signs ? w->K : lda) <= few_lda() && !up && !tuning().gemm_no_direct;
    p.find = reads && shape.mb == 1 && scale_rows && !w->signs && few_finds(M, w->K, units * ksplit);
    // Residuals of up to 16 ranks whose rows the kernel reads, and needs nothing else of a launch in front for: it
    // forms their coefficients beside its products (gemm_few_kernel.h).
    bool coeff_in = reads && !per_stream && few_reads(shape, scale_rows, w->signs != nullptr, w->K, p.gper) &&
                    (!scale_rows || w->signs || p.find);
    for (int i = 0; i < count; ++i) coeff_in &= few_coeff(ws[i]);
    const bool coeff_pre = any_res && !coeff_in;
    p.find &= !coeff_pre;
    for (int i = 0; i < count; ++i) p.seg[i].resB = coeff_in ? (const uint16_t *)ws[i].resB : nullptr;
    const CoeffPlan coeff = plan_coeff(ws, count, M);
    size_t xb_floats = coeff_pre ? coeff.floats() : 0;
    for (int i = 0; i < count && coeff_pre; ++i) xb_floats += ((size_t)M * ws[i].R + 3) & ~(size_t)3;
    const size_t rot_floats = w->signs ? ((size_t)M * w->K / 2 + 4) & ~(size_t)3 : 0;
    const size_t shift_floats = scale_rows ? ((size_t)M + 3) & ~(size_t)3 : 0;
    // Few rows: the kernel reads A itself where that pays (16-byte pieces of a row, put into
    // operand order in registers), so the pre-pass launch is dropped, and the image with it.  Needs
    // 16-byte aligned rows; rotated rows are read the same way (the rotation can write the image itself,
    // but only without a residual and row scales).
    const bool image_of_rotation = w->signs && !any_res && !scale_rows;
    const bool direct = reads && !image_of_rotation &&
                        (coeff_pre ? shape.mb == 1 : few_reads(shape, scale_rows, w->signs != nullptr, w->K, p.gper));
    const size_t ap_floats = direct ? 0 : (size_t)p.G * 2 * p.mblk_pad * 64 * 4;
    float *base = nullptr;
    int *tickets = nullptr;
    const size_t want_tickets = std::max((size_t)units, coeff_pre ? coeff.tickets() : 0) + 1;
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
    if (image_of_rotation) {
        // the rotation writes the operand image itself: one launch instead of two
        FhtOperandOut image_out = {(uint32_t *)Ap, p.mblk_pad, (int)(w->lut_dtype == FLUTE_BF16), block_xor};
        st = fht_launch(A, lda, w->signs, w->awq, nullptr, 0, M, w->K, act_dtype, 0, w->rot_block,
                        stream, &image_out);
        if (st != FLUTE_OK) return st;
    } else {
        if (w->signs) {
            // the residual coefficients and the row scales need the rotated rows as rows:
            // rotated copy first, then the ordinary pre-pass on it
            void *Arot = (void *)((float *)Ap + ap_floats);
            st = fht_launch(A, lda, w->signs, w->awq, Arot, w->K, M, w->K, act_dtype, 0,
                            w->rot_block, stream, nullptr, rowshift);
            if (st != FLUTE_OK) return st;
            A = Arot;
            lda = w->K;
        }
        p.rowshift = rowshift;                          // (the rotation knows its rows' largest exponents)
        if (p.find) p.rowshift = nullptr;
        const bool find = scale_rows && !w->signs && !p.find;
        ImageParams im = {};
        im.A = (const uint16_t *)A;
        im.up = (const uint16_t *)up;
        im.lda = lda;
        im.rowshift = p.find ? nullptr : rowshift;
        im.M = M;
        im.segs = 2 * p.G;
        im.mblk = p.mblk_pad;
        im.in_bf16 = act_dtype == FLUTE_BF16;
        im.out_bf16 = w->lut_dtype == FLUTE_BF16;
        im.block_xor = block_xor;
        im.find = find && rows16 && w->K <= find_reach();
        if (find && !im.find) {
            st = launch_rowshift(A, lda, M, w->K, rowshift, stream);
            if (st != FLUTE_OK) return st;
        }
        if (direct) {
            p.A8 = (const u4_t *)A;
            p.lda8 = lda / 8;
            p.a_bf16 = act_dtype == FLUTE_BF16;
            im.blocks = im.find ? (M + 15) / 16 : 0;    // (the scales alone)
        } else if (rows16) {
            im.Ap = Ap;
            im.blocks = p.mblk_pad;
            im.warm = (const uint32_t *)w->lut1;
            im.warm_lines = (int)(((size_t)w->lut_rows << w->b1) * 2 / 64);
        } else {
            const int64_t total = (int64_t)p.G * 2 * p.mblk_pad * 64;
            const int blocks = (int)((total + 255) / 256 < 4096 ? (total + 255) / 256 : 4096);
            hipLaunchKernelGGL(gemm_prep_kernel, dim3(blocks), dim3(256), 0, stream,
                               (const uint16_t *)A, Ap, M, lda, p.G, p.mblk_pad,
                               (int)(act_dtype == FLUTE_BF16), (int)(w->lut_dtype == FLUTE_BF16),
                               (int)((((uintptr_t)A & 3) == 0) && (lda % 2 == 0)), rowshift, block_xor);
            FLUTE_HIP_CHECK(hipGetLastError());
        }
        float *next = xb + coeff.floats(), *to[kGemmMaxSegs] = {};
        for (int i = 0; i < count; ++i) {
            if (ws[i].R == 0 || coeff_in) continue;
            to[i] = next;
            p.seg[i].xb = next;
            p.seg[i].vec_res = ws[i].R % 4 == 0 && ((uintptr_t)ws[i].resA & 7) == 0 && ((uintptr_t)next & 15) == 0;
            next += ((size_t)M * ws[i].R + 3) & ~(size_t)3;
        }
        st = launch_pre(coeff_pre ? &coeff : nullptr, ws, count, A, lda, to, M, p.out_bf16, xb, tickets, im, stream);
        if (st != FLUTE_OK) return st;
    }

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
        const int bf16 = w->lut_dtype == FLUTE_BF16;
        if (few) {
            st = count > 1 ? (bf16 ? gemm_few_bf16_segs : gemm_few_f16_segs)(shape.mb, q, grid, stream)
                           : (bf16 ? gemm_few_bf16 : gemm_few_f16)(shape.mb, q, grid, stream);
        } else {
            const int lds = plan_lds(q, shape);
            FLUTE_REQUIRE(lds <= kLdsPerCU, FLUTE_ERR_UNSUPPORTED,
                          "flute_gemm: %d bytes of LDS exceed the %d of one CU", lds, kLdsPerCU);
            st = count > 1 ? gemm_launch_segs(bf16, shape.mb, shape.mw, q, grid, lds, stream)
                 : bf16    ? launch_gemm_shape<true, false>(shape.mb, shape.mw, q, grid, lds, stream)
                           : launch_gemm_shape<false, false>(shape.mb, shape.mw, q, grid, lds, stream);
        }
        if (st != FLUTE_OK) return st;
    }
    workspace_done(stream);
    return FLUTE_OK;
}

// How a call is served.
struct GemmPlan {
    bool together;     // all weights in one launch of the kernel (one weight always is)
    GemmShape shape;   // of the small-M kernel
    WidePlan wide;     // rows > 0: the many-row kernel instead
};

// One launch of the many-row kernel where the weights together are better off there than each in its
// own best form: they share the activations' image, and a chip that one weight's tiles leave partly
// idle (or cut into slices of K) is filled.  Gate and up, 2 x 4096 -> 12288, M = 509: 2 x 65.8 us in
// two slices each, 98.7 together.  Small calls share everything in front of the kernel, and its
// launch.
GemmPlan plan_gemm(const flute_linear *ws, int count, int M) {
    const int streams = ws[0].b2 > 0 ? 2 : 1, G = ws[0].K / 64;
    bool widths = true, all = true;
    int tiles = 0;
    for (int i = 0; i < count; ++i) {
        const flute_linear &w = ws[i];
        widths &= w.b1 == ws[0].b1 && w.b2 == ws[0].b2;
        all &= w.group_size == ws[0].group_size && w.signs == ws[0].signs && w.awq == ws[0].awq &&
               w.rot_block == ws[0].rot_block;
        tiles += w.N / 128;
    }
    GemmPlan plan = {};
    if (!widths) return plan;
    double us = 0.0;
    plan.shape = choose_gemm_shape(M, tiles, G, ws[0].b1, ws[0].b2, us);
    plan.wide = choose_wide(M, tiles, G, streams, us);
    plan.together = plan.wide.rows || all;
    return plan;
}

// Whether a call forms silu(gate) * up on its way to the operand image: calls that have one, of rows that are not
// rotated (the rotation wants the rows themselves, as do coefficients of factors that are not aligned, and
// the few-row kernel where it forms the coefficients: their sums have an order of their own).
bool takes_silu(const flute_linear &w, const GemmPlan &plan, int act_dtype) {
    if (!plan.wide.rows && plan.shape.mb == 2 && few_coeff(w) && !tuning().gemm_no_direct &&
        (act_dtype == FLUTE_BF16) == (w.lut_dtype == FLUTE_BF16) && few_takes(std::max(w.b1, w.b2), std::min(w.b1, w.b2)))
        return false;
    return !w.signs && ((uintptr_t)w.resB & 15) == 0 && (plan.wide.rows || plan.shape.mb > 1) &&
           (w.K <= find_reach() || (act_dtype == FLUTE_BF16) == (w.lut_dtype == FLUTE_BF16));
}

}  // namespace
}  // namespace flute

using namespace flute;

extern "C" int flute_gemm_rows(const flute_linear *ws, int count, int M) {
    if (!ws || count < 1 || count > kWideMaxSegs || M < 1) return -1;
    for (int i = 0; i < count; ++i)
        if (validate_linear(&ws[i], 1, "flute_gemm_rows") != FLUTE_OK) return -1;
    const GemmPlan plan = plan_gemm(ws, count, M);
    return !plan.together ? 0 : plan.wide.rows ? plan.wide.rows : 16 * plan.shape.mb * plan.shape.mw;
}

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

    const GemmPlan plan = plan_gemm(w, 1, M);
    if (plan.wide.rows) return gemm_wide(w, 1, A, &C, &ldc, M, lda, act_dtype, plan.wide, stream);
    return gemm_rows(w, 1, A, &C, &ldc, M, lda, act_dtype, plan.shape, stream);
}

extern "C" int flute_gemm_takes_silu(const flute_linear *w, int M, int act_dtype) {
    if (!w || M < 1 || validate_linear(w, 1, "flute_gemm_takes_silu") != FLUTE_OK) return 0;
    return takes_silu(*w, plan_gemm(w, 1, M), act_dtype);
}

extern "C" flute_status flute_gemm_silu(const flute_linear *w, const void *gate, const void *up, void *C, int M,
                                        int64_t lda, int64_t ldc, int act_dtype, void *stream) {
    flute_status st = validate_linear(w, 1, "flute_gemm_silu");
    if (st != FLUTE_OK) return st;
    FLUTE_REQUIRE(act_dtype == FLUTE_F16 || act_dtype == FLUTE_BF16, FLUTE_ERR_INVALID,
                  "flute_gemm_silu: activations must be float16 or bfloat16");
    FLUTE_REQUIRE(M >= 0, FLUTE_ERR_INVALID, "flute_gemm_silu: M must be >= 0 (got %d)", M);
    if (M == 0) return FLUTE_OK;
    FLUTE_REQUIRE(gate && up && C && lda >= w->K && ldc >= w->N && lda % 8 == 0 && (((uintptr_t)gate | (uintptr_t)up) & 15) == 0 &&
                      ((uintptr_t)C & 1) == 0,
                  FLUTE_ERR_INVALID, "flute_gemm_silu: gate and up must be 16-byte aligned rows, C rows of N or more");
    const GemmPlan plan = plan_gemm(w, 1, M);
    FLUTE_REQUIRE(takes_silu(*w, plan, act_dtype), FLUTE_ERR_UNSUPPORTED,
                  "flute_gemm_silu: this call has no operand image (flute_gemm_takes_silu); use flute_silu_mul and flute_gemm");
    if (plan.wide.rows) return gemm_wide(w, 1, gate, &C, &ldc, M, lda, act_dtype, plan.wide, (hipStream_t)stream, up);
    return gemm_rows(w, 1, gate, &C, &ldc, M, lda, act_dtype, plan.shape, (hipStream_t)stream, up);
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
    const GemmPlan plan = plan_gemm(ws, count, M);
    if (plan.wide.rows) return gemm_wide(ws, count, A, C, ldc, M, lda, act_dtype, plan.wide, (hipStream_t)stream);
    if (plan.together) return gemm_rows(ws, count, A, C, ldc, M, lda, act_dtype, plan.shape, (hipStream_t)stream);
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
        *(u4_t *)(h + i * 8) = bf16 ? silu_mul8<true>(a, b) : silu_mul8<false>(a, b);
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
