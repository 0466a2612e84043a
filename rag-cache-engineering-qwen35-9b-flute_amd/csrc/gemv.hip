// Launchers of the M = 1 LUT GEMV family: single weight, merged gate/up with
// SiLU*mul, several weights sharing one input, and the two-launch MLP block.
#include "gemv_kernel.h"
#include "gemv4_kernel.h"
#include "host_common.h"

#include <atomic>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>

namespace flute {

namespace {

// What has to be known before a GEMV launch can finish a row: the rotated input of every weight
// that carries a residual, and the residual coefficients xb[r] = sum_k x[k] * resB[r][k] (fp32, x
// rotated and rounded to the activation type where the weight is rotated).  One launch for all
// weights of a call, and every workgroup transforms the input itself (a few microseconds of one CU)
// instead of waiting for another launch to do it.  The butterflies are fht_dev.h's in the same order,
// so the rotated row has the bits of flute_fht; a lane's sum runs over its columns in ascending order,
// then a fixed tree, then over the wavefronts of the residual row in order.
// What bounds it: latency.  The row, its multipliers and a wavefront's first columns of its residual
// row are requested together; what follows is LDS passes between barriers, then a step of eight
// columns a lane for every 512 * (8 / rows) columns, rows = residual rows per workgroup, as few as
// leave a workgroup per CU.  (One wavefront a residual row, eight rows a workgroup: rotated q/k/v of
// rank 16, K = 4096, 7.2 us, now 6.0; rank 16, K = 11520, not rotated, 10.8, now 4.0; rank 8, K = 12288,
// rotated, the call 26.7, now 21.2.)
constexpr int kPreThreads = 512, kPreWaves = kPreThreads / 64;

struct PreSeg {
    const uint16_t *resB;
    const float *signs, *awq;
    float *xb;
    uint16_t *xrot;         // where the first workgroup of this weight leaves the rotated row, or NULL
    int R;
    int block0;             // first workgroup of this weight
    int vec_b, vec_m;       // resB / signs and awq allow 16-byte loads
};

struct PreParams {
    PreSeg seg[kGemvMaxSegs];
    const uint16_t *x;
    int nsegs, K, act_bf16, rot_block;
    int rows;               // residual rows per workgroup: 1, 2, 4 or 8
};

__device__ __forceinline__ void pre_unpack8(const uint4 raw, int bf16, float (&f)[8]) {
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const uint16_t h = (uint16_t)(w[q >> 1] >> (16 * (q & 1)));
        f[q] = bf16 ? bf2f(h) : h2f(h);
    }
}

__device__ __forceinline__ uint4 pre_load8(const uint16_t *p, int vec) {
    if (vec) return *(const uint4 *)p;
    uint32_t w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = (uint32_t)p[2 * q] | ((uint32_t)p[2 * q + 1] << 16);
    return make_uint4(w[0], w[1], w[2], w[3]);
}

__device__ __forceinline__ void pre_mul8(const float *p, int vec, float (&f)[8]) {
    if (vec) {
        const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 4);
        f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
        f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) f[q] = p[q];
    }
}

// WHOLE: rows that transform_row reaches (buf holds K floats); else, segment by segment, the longest
// segment or chunk of blocks.
template <bool WHOLE>
__global__ void __launch_bounds__(kPreThreads) gemv_pre_kernel(const PreParams p) {
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ float sums[kPreWaves];
    float *const buf = (float *)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int si = 0;
    while (si + 1 < p.nsegs && (int)blockIdx.x >= p.seg[si + 1].block0) ++si;
    const PreSeg &w = p.seg[si];
    const int part = blockIdx.x - w.block0;
    const int share = kPreWaves / p.rows;               // wavefronts of a residual row
    const int r = part * p.rows + wave / share, c = wave % share;
    const bool mine = r < w.R;
    const uint16_t *const row = w.resB + (size_t)(mine ? r : 0) * p.K;
    // columns of this lane: (h * share + c) * 512 + lane * 8, h = 0, 1, ...
    const int col0 = c * 512 + lane * 8, step = share * 512;
    constexpr int AHEAD = 4;                            // steps requested up front
    uint4 first[AHEAD];
    if (mine) {
#pragma unroll
        for (int h = 0; h < AHEAD; ++h)
            if (h * step < p.K) first[h] = pre_load8(row + min(col0 + h * step, p.K - 8), w.vec_b);
    }
    float acc = 0.0f;
    // products of this lane's columns in [off, off + count), x from `get`
    auto dot = [&](int off, int count, auto get) {
        if (!mine) return;
        auto take = [&](int k, const uint4 raw) {
            float b[8], x[8];
            pre_unpack8(raw, p.act_bf16, b);
            get(k, x);
#pragma unroll
            for (int q = 0; q < 8; ++q) acc = fmaf(x[q], b[q], acc);
        };
#pragma unroll
        for (int h = 0; h < AHEAD; ++h) {
            const int k = col0 + h * step;
            if (k >= off && k < off + count) take(k, first[h]);
        }
        int k = col0 + AHEAD * step;
        if (k < off) k += (off - k + step - 1) / step * step;
        for (; k < off + count; k += step) take(k, pre_load8(row + k, w.vec_b));
    };
    // eight finished columns of the rotated row: rounded to the activation type, kept in fp32 at `to`
    auto rotated = [&](int k, float (&t)[8], const float (&sg)[8], float inv, float (&back)[8]) {
#pragma unroll
        for (int q = 0; q < 8; ++q) t[q] = t[q] * sg[q] * inv;
        if (w.awq) {
            float sc[8];
            pre_mul8(w.awq + k, w.vec_m, sc);
#pragma unroll
            for (int q = 0; q < 8; ++q) t[q] = t[q] / sc[q];
        }
        uint16_t o[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            o[q] = round_act(t[q], p.act_bf16);
            back[q] = p.act_bf16 ? bf2f(o[q]) : h2f(o[q]);
        }
        if (w.xrot && part == 0)
            *(uint4 *)(w.xrot + k) =
                make_uint4((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16),
                           (uint32_t)o[4] | ((uint32_t)o[5] << 16), (uint32_t)o[6] | ((uint32_t)o[7] << 16));
    };
    if (w.signs == nullptr) {
        dot(0, p.K, [&](int k, float (&x)[8]) { pre_unpack8(*(const uint4 *)(p.x + k), p.act_bf16, x); });
    } else if constexpr (WHOLE) {
        float sg[4][8];
        transform_row<4>(
            buf, p.K, p.rot_block, tid, kPreThreads,
            [&](int h, int j, float (&f)[8]) {
                pre_unpack8(*(const uint4 *)(p.x + j), p.act_bf16, f);
                pre_mul8(w.signs + j, w.vec_m, sg[h]);
                if (w.awq) {
                    float s[8];
                    pre_mul8(w.awq + j, w.vec_m, s);
#pragma unroll
                    for (int q = 0; q < 8; ++q) f[q] *= s[q];
                }
            },
            [&](int h, int j, float (&f)[8], int nst) {
                float b[8];
                rotated(j, f, sg[h], inv_sqrt_pow2(nst), b);
                *(float4 *)(buf + (row_slot(j) ^ 0)) = make_float4(b[0], b[1], b[2], b[3]);
                *(float4 *)(buf + (row_slot(j) ^ 4)) = make_float4(b[4], b[5], b[6], b[7]);
            });
        __syncthreads();
        dot(0, p.K, [&](int k, float (&x)[8]) {
            const float4 a = *(const float4 *)(buf + row_slot(k)), b = *(const float4 *)(buf + (row_slot(k) ^ 4));
            x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
            x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
        });
    } else {
        for (int off = 0; off < p.K;) {
            int count, nst;
            if (p.rot_block > 0) {
                nst = 31 - __builtin_clz((unsigned)p.rot_block);
                count = min((16384 / p.rot_block) * p.rot_block, p.K - off);
            } else {
                nst = 31 - __builtin_clz((unsigned)(p.K - off));
                count = 1 << nst;
            }
            const float inv = inv_sqrt_pow2(nst);
            for (int j = tid * 8; j < count; j += kPreThreads * 8) {
                float f[8];
                pre_unpack8(*(const uint4 *)(p.x + off + j), p.act_bf16, f);
                if (w.awq) {
                    float s[8];
                    pre_mul8(w.awq + off + j, w.vec_m, s);
#pragma unroll
                    for (int q = 0; q < 8; ++q) f[q] *= s[q];
                }
                fht_head(f, lane, nst);
                const int s0 = fht_slot(j);             // a multiple of 8: slot(j + q) = s0 ^ q
#pragma unroll
                for (int q = 0; q < 8; ++q) buf[s0 ^ q] = f[q];
            }
            __syncthreads();
            fht_tail(buf, count, nst, 9, tid, kPreThreads);
            for (int j = tid * 8; j < count; j += kPreThreads * 8) {
                float sg[8], t[8], b[8];
                pre_mul8(w.signs + off + j, w.vec_m, sg);
                const int s0 = fht_slot(j);
#pragma unroll
                for (int q = 0; q < 8; ++q) t[q] = buf[s0 ^ q];
                rotated(off + j, t, sg, inv, b);
#pragma unroll
                for (int q = 0; q < 8; ++q) buf[s0 ^ q] = b[q];
            }
            __syncthreads();
            dot(off, count, [&](int k, float (&x)[8]) {
                const int s0 = fht_slot(k - off);
#pragma unroll
                for (int q = 0; q < 8; ++q) x[q] = buf[s0 ^ q];
            });
            off += count;
            if (off < p.K) __syncthreads();             // the next segment reuses the buffer
        }
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) acc += __shfl_xor(acc, m);
    if (lane == 0) sums[wave] = acc;
    __syncthreads();
    if (lane == 0 && c == 0 && mine) {
        float total = sums[wave];
        for (int i = 1; i < share; ++i) total += sums[wave + i];
        w.xb[r] = total;
    }
}

int entries_log2(int bits) { return bits == 3 ? 6 : 8; }
int entry_bytes_log2(int bits) { return bits >= 3 ? 2 : (bits == 2 ? 3 : 4); }

struct Plan {
    GemvParams p;
    int pair;               // 10 * b1 + b2 when the widths are a pair the lean kernel serves with two tables, else 0
    bool k_group;           // the LUT is grouped along K (single weight, lean kernel only)
    bool lean;              // the lean kernel serves the launch (make_plan lays the tables out for it)
    size_t lds_bytes;
    int grid_x;
    int threads;
    int total_tickets;
    size_t p_floats;        // partial sums
    size_t xb_floats;       // residual coefficients
    size_t xrot_halves;     // pre-rotated inputs of weights that carry a residual
    bool lut_bf16;
    // pre-kernels: residual coefficients (and the rotation they need)
    struct Pre {
        const uint16_t *resB;
        const float *signs, *awq;
        int R, seg;
        int share;              // index of an earlier entry with the same rotation, or -1
        size_t xb_off, xrot_off;
    } pre[kGemvMaxSegs];
    int npre;
    int rot_block;
};

// Wavefronts of a workgroup of `rw` rows: eight when each still has two loads or more and the grid is
// at most one workgroup per CU, or two per CU of eight-row workgroups with a long K range (the general
// kernel; the lean one takes wider slices there, see make_plan).  Otherwise four, fewer for very short K.
int choose_waves(int rows, int G, int split, int rw) {
    const int forced = tuning().gemv_waves;
    if (forced == 1 || forced == 2 || forced == 4 || forced == 8) return forced;
    const int units = (G / split) / (32 / rw);
    const long wgs = (long)(rows / rw) * split;
    const bool eight = units >= 16 && (wgs <= kNumCU || (wgs <= 2 * kNumCU && units >= 32 && rw == 8));
    return eight ? 8 : (units >= 4 ? 4 : (units >= 2 ? 2 : 1));
}

// Shape of the launch for `rows` output rows over G tiles of K.  A workgroup
// owns `rw` rows.  The library's own policy splits K only where a workgroup's K range
// would be very long over few rows: the exchange between workgroups (partial sums
// written through, a ticket, the last arrival reading them back) is three memory round
// trips, and up to K = 24576 the unsplit launch measured faster for every narrow shape
// (N = 128...3072; e.g. N = 1024, K = 4096: 4.5 us against 5.9 / 10.4 / 11.4 us split
// 2 / 4 / 8 ways; N = 512, K = 24576: 7.7 against 8.2 / 11.5).  From K = 32768 on, four
// ways win up to 512 rows and two ways up to 1024 (K = 32768: N = 128 6.8 against
// 8.7 us, N = 512 7.5 against 9.0, N = 1024 8.3 against 9.2; K = 65536: N = 512 8.8
// against 19.0, N = 1024 12.8 against 20.9); 2048 rows and more stay unsplit (11.0
// against 14.3 us).  A caller's explicit split is honoured.
void choose_shape(int rows, int G, int split_req, int *rw, int *split, int *waves,
                  bool may_split = true) {
    int best_rw = tuning().gemv_rw;
    if (best_rw != 8 && best_rw != 16 && best_rw != 32) {
        // The narrowest slices whose grid is still resident at once (three four-wavefront
        // workgroups per CU): a second round of workgroups costs far more than wider
        // slices do (8192 rows at K = 4096: 512 sixteen-row workgroups 7.3 us, 1024
        // eight-row ones 13.2 us; 16384 rows: 11.3 us with 32 rows against 15.3 with 16).
        best_rw = 32;
        for (int cand : {8, 16}) {
            if (rows / cand <= 3 * kNumCU) { best_rw = cand; break; }
        }
        // A grid of exactly one or two 16-row workgroups per CU, unsplit, measured best
        // where K is long enough to give each of them eight wavefronts (4096 rows at
        // K = 12288: 256 workgroups, 8.5 us against 9.2 us for 512 eight-row ones and
        // 9.5 us for 768 with a three-way K split).
        if (rows % (16 * kNumCU) == 0 && rows / (16 * kNumCU) <= 2 && G / 2 >= 64) {
            best_rw = 16;
        }
    }
    int sp = split_req;
    if (sp > 0) {
        // a wavefront load spans 32/rw tiles of K: widen the slices until the K
        // range of one split is a whole number of loads
        while (G % sp == 0 && (G / sp) % (32 / best_rw) != 0 && best_rw < 32) best_rw *= 2;
    } else {
        sp = 1;
        // (not with a rotation fused into the prologue: its blocks would have to fit the slices)
        if (may_split && G >= 512 && rows <= 512 && G % 4 == 0) sp = 4;
        else if (may_split && G >= 512 && rows <= 1024 && G % 2 == 0) sp = 2;
        while ((G / sp) % (32 / best_rw) != 0 && best_rw < 32) best_rw *= 2;
    }
    *rw = best_rw;
    *split = sp;
    *waves = choose_waves(rows, G, sp, best_rw);
}

// 10 * b1 + b2 of a launch that the lean kernel takes with two tables, 0: one 4-bit width, -1: neither.
int lean_pair(const flute_linear *segs, int count) {
    const int b1 = segs[0].b1;
    int b2 = 0;
    bool four = true, same = true;
    for (int i = 0; i < count; ++i) {
        four &= segs[i].b1 == 4 && (segs[i].b2 == 0 || segs[i].b2 == 4);
        same &= segs[i].b1 == b1;
        if (segs[i].b2 > 0) {
            if (b2 == 0) b2 = segs[i].b2;
            same &= segs[i].b2 == b2;
        }
    }
    if (four) return 0;
    if (!same) return -1;
    // a single narrow stream ((3, 0) is one of upstream's pairs): the two-table instantiation
    // of its width with the second table unused
    if (b2 == 0) b2 = b1 == 3 ? 3 : (b1 == 2 ? 3 : 4);
    const int code = 10 * b1 + b2;
    return code == 41 || code == 14 || code == 33 || code == 24 || code == 23 ? code : -1;
}

// LDS bytes of its tables: 4^b entries of 128 bytes a stream, of which a launch of one width has one;
// a 1-bit stream's nibble table has 16 entries of 256 bytes.
size_t lean_table_bytes(int pair) {
    const auto tab = [](int b) { return b == 1 ? (size_t)16 * 256 : ((size_t)1 << (2 * b)) * 128; };
    return pair == 0 ? tab(4) : tab(pair / 10) + tab(pair % 10);
}

// Whether the lean kernel takes a launch: widths as above, one LUT group per half tile (its row
// slices lie in one half), LUT rows that can be read through the scalar cache, gate and up with one
// input and rotation (the activations are staged once), a load or more per wavefront, and LDS for the
// tables (32 KB, two-table pairs 36 KB at most) beside the activations.
bool lean_serves(const flute_linear *segs, int count, int gs_tiles, int rw, int waves, int silu_mul) {
    if (lean_pair(segs, count) < 0 || tuning().gemv_no_fast || !(waves == 4 || waves == 8)) return false;
    if (tuning().gemv_table_log2 >= 12 && tuning().gemv_table_log2 < 15) return false;   // (smaller tables are asked for)
    for (int i = 0; i < count; ++i) {
        if (segs[i].group_size < 64 || ((uintptr_t)segs[i].lut1 & 3) || (segs[i].b2 && ((uintptr_t)segs[i].lut2 & 3)))
            return false;
    }
    if (silu_mul) {
        const flute_linear &g = segs[0], &u = segs[1];
        if (g.signs != u.signs || g.awq != u.awq || (g.signs && (g.R > 0) != (u.R > 0))) return false;
    }
    const int gpi = 32 / rw;
    return gs_tiles % gpi == 0 && gs_tiles / gpi >= waves &&
           36 * 1024 + gs_tiles * 128 + kGemvRedBytes + 1024 <= kLdsPerCU;
}

// Fill a launch plan for `count` weights that share x.  silu_mul couples
// weights 0 and 1 into one output.
flute_status make_plan(const flute_linear *segs, int count, const void *x, void *const *outs,
                       int act_dtype, int split, int silu_mul, const char *who, Plan *plan) {
    FLUTE_REQUIRE(count >= 1 && count <= kGemvMaxSegs, FLUTE_ERR_INVALID,
                  "%s: 1..%d weights per launch (got %d)", who, kGemvMaxSegs, count);
    FLUTE_REQUIRE(x != nullptr, FLUTE_ERR_INVALID, "%s: x is NULL", who);
    FLUTE_REQUIRE(((uintptr_t)x & 15) == 0, FLUTE_ERR_INVALID,
                  "%s: x must be 16-byte aligned (the kernels read it 16 bytes at a time)", who);
    FLUTE_REQUIRE(act_dtype == FLUTE_F16 || act_dtype == FLUTE_BF16, FLUTE_ERR_INVALID,
                  "%s: activations must be float16 or bfloat16", who);
    for (int i = 0; i < count; ++i) {
        flute_status st = validate_linear(&segs[i], count == 1 && !silu_mul ? kModeKGroupOk : 0, who);
        if (st != FLUTE_OK) return st;
        FLUTE_REQUIRE(outs[i] != nullptr, FLUTE_ERR_INVALID, "%s: output %d is NULL", who, i);
        FLUTE_REQUIRE(((uintptr_t)outs[i] & 1) == 0, FLUTE_ERR_INVALID,
                      "%s: output %d must be 2-byte aligned", who, i);
        FLUTE_REQUIRE(segs[i].K == segs[0].K, FLUTE_ERR_INVALID,
                      "%s: all weights of one launch must share K (%d vs %d)", who, segs[i].K,
                      segs[0].K);
        FLUTE_REQUIRE(segs[i].lut_dtype == segs[0].lut_dtype, FLUTE_ERR_UNSUPPORTED,
                      "%s: all weights of one launch must share the LUT dtype", who);
        FLUTE_REQUIRE(segs[i].rot_block == segs[0].rot_block, FLUTE_ERR_UNSUPPORTED,
                      "%s: all weights of one launch must share the rotation block", who);
    }
    const bool lut_bf16 = segs[0].lut_dtype == FLUTE_BF16;
    FLUTE_REQUIRE(!(lut_bf16 && act_dtype == FLUTE_F16), FLUTE_ERR_UNSUPPORTED,
                  "%s: a bfloat16 LUT with float16 activations is not served (the pair product "
                  "runs in the LUT's type and float16 does not convert to bfloat16 exactly)",
                  who);
    if (silu_mul) {
        FLUTE_REQUIRE(count == 2 && segs[0].N == segs[1].N, FLUTE_ERR_INVALID,
                      "%s: gate and up must agree in N (%d vs %d)", who, segs[0].N,
                      count == 2 ? segs[1].N : -1);
    }
    const int K = segs[0].K;
    const int G = K / 64;
    FLUTE_REQUIRE(split <= 0 || G % split == 0, FLUTE_ERR_INVALID,
                  "%s: split %d must divide K/64 = %d", who, split, G);

    const int split_in = split;
    GemvParams &p = plan->p;
    std::memset(&p, 0, sizeof(p));
    int rows = 0;
    for (int i = 0; i < (silu_mul ? 1 : count); ++i) rows += segs[i].N;
    int rw, waves;
    bool rotated = false;
    for (int i = 0; i < count; ++i) rotated |= segs[i].signs != nullptr;
    // (the library's own K split was measured on single weights only: merged gate/up launches
    // split when the caller asks for it)
    choose_shape(rows, G, split, &rw, &split, &waves, !rotated && !silu_mul);
    const bool k_group = segs[0].k_group != 0;
    if (k_group) {
        // Only the lean kernel serves this form: four or eight wavefronts, each with an even
        // number (two at least) of loads of 32 / rw tiles.  The workgroup stages its LUT rows in
        // LDS, 64 bytes per (row, K group), at most kKGroupPieces 16-byte pieces per thread, whole
        // K groups per split.  The shape chosen above is kept where it fits; else wider slices or
        // another wavefront count; else, where the library chooses the split, a larger one.
        auto ok = [&](int sp, int rw_, int wv) {
            if (G % sp || (G / sp) % 2 || (G / sp) % (32 / rw_)) return false;
            const int units = (G / sp) / (32 / rw_);
            if (!(wv == 4 || (wv == 8 && rw_ <= 16)) || units % wv) return false;
            const int u = units / wv;
            return u >= 2 && u % 2 == 0 &&
                   (long)rw_ * (G / sp / 2) * 2 <= (long)kKGroupPieces * wv * 64;
        };
        auto settle = [&](int sp) {
            if (ok(sp, rw, waves)) return true;
            for (int r = rw; r <= 32; r *= 2)
                for (int wv : {4, 8})
                    if (ok(sp, r, wv)) {
                        rw = r;
                        waves = wv;
                        return true;
                    }
            return false;
        };
        bool done = settle(split);
        for (int sp = split * 2; !done && split_in <= 0 && sp <= G / 2 && G % sp == 0; sp *= 2) {
            choose_shape(rows, G, sp, &rw, &split, &waves, false);
            done = settle(split);
        }
        FLUTE_REQUIRE(done, FLUTE_ERR_UNSUPPORTED,
                      "%s: K=%d at split %d does not divide into the loads of the kernel that serves "
                      "a LUT grouped along K (K/split must be a multiple of 512 whose LUT rows fit a "
                      "workgroup's staging); try another split", who, K, split);
    }
    // A lean launch of which fewer workgroups stay on a CU than its narrow slices need: wider slices
    // instead of a second round.  Four wavefronts (tables and activations of a long K range over many rows
    // leave no room for three workgroups): 32 rows.  One token, 16-row slices and these: 11264 -> 12288, (4, 1)
    // bits 41.7 -> 25.9 us, 12288 -> 12288 20.9 -> 18.0, (2, 4) bits 33.4 -> 31.2; where all are resident either
    // width measures the same.  Eight wavefronts (the registers leave room for one workgroup; 257 to 512 eight-row
    // ones): 16 rows, which are one per CU and fill half of the chip or more; 32 rows leave up to three quarters
    // of it idle.  The launch alone with 8, 16 and 32 rows: 8192 -> 3072, 4 bits 7.9 / 5.9 / 7.5 us, (3, 3) 11.5 /
    // 8.7 / 13.0; 12288 -> 2176, (4, 1) 9.5 / 9.5 / 14.8; 12288 -> 3968, rotated, (2, 4) 19.9 / 16.4 / 21.9.
    if (tuning().gemv_rw == 0 && rw < 32 && !k_group && lean_serves(segs, count, G / split, rw, waves, silu_mul)) {
        const size_t lds = lean_table_bytes(lean_pair(segs, count)) + (size_t)(G / split) * 128 + kGemvRedBytes + 512;
        const long holds = std::min<long>(waves == 4 ? 3 : 1, (long)(kLdsPerCU / lds));
        if ((long)(rows / rw) * split > holds * kNumCU) {
            rw = waves == 8 ? 2 * rw : 32;
            waves = choose_waves(rows, G, split, rw);
        }
    }
    FLUTE_REQUIRE((G / split) % (32 / rw) == 0, FLUTE_ERR_UNSUPPORTED,
                  "%s: K/64/split = %d is not a whole number of wavefront loads", who, G / split);
    const int gs_tiles = G / split;
    const int kc = gs_tiles * 64;
    const int spt = 128 / rw;
    plan->lean = !k_group && lean_serves(segs, count, gs_tiles, rw, waves, silu_mul);

    bool any_fused_rot = false;
    const int fht_block = segs[0].rot_block;
    plan->npre = 0;
    plan->rot_block = fht_block;
    size_t xb_off = 0, xrot_off = 0;
    int n0 = 0, col = 0, ticket = 0;
    size_t tab_bytes = 0;
    // LDS: tables/scratch | x slice | row sums.  The table stride is the largest
    // that still lets the whole grid be resident at once (one round of
    // workgroups), since a second round repeats the start-up latency.
    int budget = tuning().gemv_table_log2;
    if (budget < 12 || budget > 17) {
        long wgs = 0;
        for (int i = 0; i < (silu_mul ? 1 : count); ++i) wgs += (long)(segs[i].N / rw) * split;
        long per_cu = (wgs + kNumCU - 1) / kNumCU;
        // The lean kernel needs the full 32 KB table and is built for three workgroups per CU; grids
        // of many rounds gain more from it than from a fourth resident workgroup with a half-size
        // table in the general kernel (4096 -> 248320: 104 us against 127 us).
        if (per_cu > (plan->lean ? 3 : 4)) per_cu = plan->lean ? 3 : 4;
        if (per_cu < 1) per_cu = 1;
        const long fixed = kc * 2 + 4096;
        budget = 14;
        for (int cand = 15; cand >= 14; --cand)
            if (((1L << cand) + fixed) * per_cu <= kLdsPerCU) { budget = cand; break; }
    }
    for (int i = 0; i < count; ++i) {
        const flute_linear &w = segs[i];
        GemvSeg &sg = p.seg[i];
        sg.resA = (const uint16_t *)w.resA;
        sg.bias = (const uint16_t *)w.bias;
        sg.out = (uint16_t *)outs[i];
        sg.N = w.N;
        sg.R = w.R;
        sg.gs = k_group ? 128 : w.group_size;       // (a LUT grouped along K: group_size is not read)
        sg.lut_rows = w.lut_rows;
        sg.nstreams = w.b2 > 0 ? 2 : 1;
        sg.n0 = n0;
        sg.col0 = (silu_mul && i == 1) ? 0 : col;
        sg.ticket0 = (silu_mul && i == 1) ? 0 : ticket;
        n0 += w.N;
        if (!(silu_mul && i == 1)) {
            col += (w.N / 128) * spt;
            ticket += (w.N / 128) * spt;
        }
        // Rotating inside the GEMV makes every workgroup transform the whole row itself
        // (about 5 us of VALU work per CU at K = 4096); a separate rotation launch in
        // front measured slower still (a dependent launch costs more than that), so it
        // stays an opt-in.
        const bool prerotate = w.signs != nullptr && w.R == 0 &&
                               tuning().gemv_prerotate != 0;
        if (w.R > 0 || prerotate) {
            // the residual needs x . resB[r] before any row can finish: computed by a
            // small kernel in front, on the rotated input when the weight is rotated
            Plan::Pre &pre = plan->pre[plan->npre++];
            pre.resB = (const uint16_t *)w.resB;
            pre.signs = w.signs;
            pre.awq = w.awq;
            pre.R = w.R;
            pre.seg = i;
            pre.xb_off = xb_off;
            pre.share = -1;
            for (int j = 0; j + 1 < plan->npre && w.signs; ++j)
                if (plan->pre[j].signs == w.signs && plan->pre[j].awq == w.awq) pre.share = j;
            pre.xrot_off = pre.share >= 0 ? plan->pre[pre.share].xrot_off : xrot_off;
            xb_off += (size_t)((w.R + 3) & ~3);
            if (w.signs && pre.share < 0) xrot_off += (size_t)K;
            sg.signs = nullptr;                     // the kernel reads the pre-rotated row
            sg.awq = nullptr;
        } else {
            sg.signs = w.signs;
            sg.awq = w.awq;
            any_fused_rot |= w.signs != nullptr;
        }
        const int ngrp_log2 = k_group || plan->lean || w.group_size >= 128 ? 0 : ilog2(128 / w.group_size);
        for (int st = 0; st < sg.nstreams; ++st) {
            GemvStream &gs = sg.st[st];
            gs.q = (const uint8_t *)(st ? w.q2 : w.q1);
            gs.lut = (const uint16_t *)(st ? w.lut2 : w.lut1);
            gs.bits = st ? w.b2 : w.b1;
            int es = budget - entries_log2(gs.bits) - ngrp_log2;
            if (es > 7) es = 7;             // 32 replicas cover the 32 LDS banks
            if (es < entry_bytes_log2(gs.bits)) es = entry_bytes_log2(gs.bits);
            if (k_group || plan->lean) es = 7;   // (k_group: no table but the lean kernel's LUT rows, sized below)
            gs.es = es;
            const size_t tb = k_group ? (size_t)(kc / 128) * (rw * 64 + (rw / 8) * 64)
                                      : ((size_t)1 << (entries_log2(gs.bits) + es)) << ngrp_log2;
            if (tb > tab_bytes) tab_bytes = tb;
        }
    }
    size_t scratch = 0;
    if (fht_block > 0) {
        bool any_rot = false;
        for (int i = 0; i < count; ++i) any_rot |= segs[i].signs != nullptr;
        FLUTE_REQUIRE(any_rot, FLUTE_ERR_INVALID, "%s: a rotation block needs rotation signs", who);
        FLUTE_REQUIRE(is_pow2(fht_block) && fht_block >= 32 && fht_block <= 16384 &&
                          K % fht_block == 0,
                      FLUTE_ERR_INVALID,
                      "%s: rotation block must be a power of two in [32, 16384] dividing K", who);
        FLUTE_REQUIRE(kc % fht_block == 0, FLUTE_ERR_UNSUPPORTED,
                      "%s: K slice %d of split %d is not a whole number of %d-column rotation "
                      "blocks",
                      who, kc, split, fht_block);
        if (any_fused_rot) scratch = (size_t)kc * 4;
    } else if (any_fused_rot) {
        scratch = (size_t)make_segments(K, 0).len[0] * 4;
    }
    p.fht_block = fht_block;
    p.nsegs = count;
    p.K = K;
    p.split = split;
    p.gs_tiles = gs_tiles;
    p.lpg_log2 = ilog2(2 * rw);
    p.p_stride = (n0 + 31) & ~31;
    p.silu_mul = silu_mul;
    p.act_bf16 = act_dtype == FLUTE_BF16;
    p.x = (const uint16_t *)x;

    // Mixed widths (and 3 + 3 bits) in the lean kernel: both tables of a weight stand side by
    // side (4^b entries of 128 bytes each).  Decided here because it sets the table region;
    // the launcher may still send the launch to the general kernel, which needs less.
    plan->pair = 0;
    plan->k_group = k_group;
    if (plan->lean) {
        const int code = lean_pair(segs, count);
        if (code) {
            plan->pair = code;
            if (lean_table_bytes(code) > tab_bytes) tab_bytes = lean_table_bytes(code);
            // (4, 1) where every weight has both streams: the kernel walks the 1-bit stream first
            // (the sum of the two streams does not depend on their order beyond fp32 rounding, and
            // the order is fixed, so results stay deterministic).  With the narrow stream in front
            // all of its loads go out in the prologue: 4096 -> 12288 measured 9.7 us against 11.1 us.
            bool all_two = true;
            for (int i = 0; i < count; ++i) all_two &= segs[i].b2 > 0;
            if (code == 41 && all_two) {
                for (int i = 0; i < count; ++i) std::swap(p.seg[i].st[0], p.seg[i].st[1]);
                plan->pair = 14;
            }
        }
    }
    // A fused rotation transforms its slice at once where a thread's pieces reach it (an unsplit row, or
    // blocks beyond those that stay in a wavefront) and the fp32 slice in LDS costs no workgroup a CU
    // would otherwise hold.
    p.rot_whole = 0;
    if (plan->lean && any_fused_rot && (fht_block > 256 || (fht_block == 0 && split == 1)) &&
        kc <= transform_reach(kRotPieces, waves * 64)) {
        const auto total = [&](size_t head) {
            return ((head + 255) & ~(size_t)255) + ((kc * 2 + 15) & ~15) + kGemvRedBytes + 16 + 8 * 4;
        };
        const size_t whole = std::max(tab_bytes, (size_t)kc * 4), now = std::max(tab_bytes, scratch);
        const long per_cu = std::min<long>(((long)col * split + kNumCU - 1) / kNumCU, 16 / waves);
        const long holds = std::min<long>(per_cu, kLdsPerCU / total(now));
        if (kLdsPerCU / total(whole) >= (size_t)std::max(holds, 1L)) {
            p.rot_whole = 1;
            scratch = std::max(scratch, (size_t)kc * 4);
        }
    }
    size_t region0 = tab_bytes > scratch ? tab_bytes : scratch;
    region0 = (region0 + 255) & ~(size_t)255;
    p.lds_x = (int)region0;
    p.lds_red = p.lds_x + ((kc * 2 + 15) & ~15);
    // row sums [2][8][32], the ticket flag (16 bytes), then one word per wavefront for the
    // row maximum of a bfloat16 slice (not the row-sum area: a merged launch restages for its
    // second output while the first output's sums are still waiting to be folded)
    plan->lds_bytes = (size_t)p.lds_red + kGemvRedBytes + 16 + 8 * 4;
    FLUTE_REQUIRE(plan->lds_bytes <= (size_t)kLdsPerCU, FLUTE_ERR_UNSUPPORTED,
                  "%s: K=%d at split %d needs %zu B of LDS (limit %d)", who, K, split,
                  plan->lds_bytes, kLdsPerCU);
    plan->grid_x = col;
    plan->threads = waves * 64;
    plan->total_tickets = ticket;
    plan->p_floats = split > 1 ? (size_t)split * p.p_stride : 0;
    plan->xb_floats = xb_off;
    plan->xrot_halves = xrot_off;
    plan->lut_bf16 = lut_bf16;
    return FLUTE_OK;
}

template <bool BF16, int BFIX>
flute_status launch_typed(Plan &plan, hipStream_t stream) {
    static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
    if (!attr_done) {
        FLUTE_HIP_CHECK(hipFuncSetAttribute((const void *)gemv_kernel<BF16, BFIX>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize,
                                            (int)kLdsPerCU));
        attr_done = true;
    }
    dim3 grid(plan.grid_x, plan.p.split);
    hipLaunchKernelGGL((gemv_kernel<BF16, BFIX>), grid, dim3(plan.threads), plan.lds_bytes, stream,
                       plan.p);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

template <int LPGL, int NW, int PF, bool BF16, bool WALK>
flute_status launch_fast4_grid(const Plan &plan, int gx, hipStream_t stream) {
    static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
    if (!attr_done) {
        FLUTE_HIP_CHECK(hipFuncSetAttribute((const void *)gemv4_kernel<LPGL, NW, PF, BF16, WALK>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize,
                                            (int)kLdsPerCU));
        attr_done = true;
    }
    dim3 grid(gx, plan.p.split);
    hipLaunchKernelGGL((gemv4_kernel<LPGL, NW, PF, BF16, WALK>), grid, dim3(NW * 64), plan.lds_bytes,
                       stream, plan.p);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

// A grid of several rounds of (four-wavefront) workgroups: as many workgroups as are resident at
// once walk over the row slices instead, which stages the activations once per workgroup and lets a
// slice's first loads travel under the previous slice's last products.  Their number, or 0.
int walking_grid(Plan &plan) {
    // three workgroups per CU is what the kernel's registers allow (3 wavefronts per SIMD)
    const int per_cu = tuning().gemv4_walk >= 0 ? (tuning().gemv4_walk < 3 ? tuning().gemv4_walk : 3) : 3;
    const int resident = per_cu * kNumCU;
    if (per_cu == 0 || plan.p.split != 1 || !(plan.p.nsegs == 1 || plan.p.silu_mul) ||
        plan.lds_bytes * per_cu > (size_t)kLdsPerCU || plan.grid_x <= resident)
        return 0;
    plan.p.slices = plan.grid_x;
    plan.p.xcd_runs = tuning().gemv_xcd && resident % 8 == 0;
    return resident;
}

template <int LPGL, int NW, int PF, bool BF16>
flute_status launch_fast4(Plan &plan, hipStream_t stream) {
    plan.p.slices = 0;
    if constexpr (NW == 4) {                     // (eight-wavefront workgroups serve short grids only)
        if (const int resident = walking_grid(plan))
            return launch_fast4_grid<LPGL, NW, PF, BF16, true>(plan, resident, stream);
    }
    return launch_fast4_grid<LPGL, NW, PF, BF16, false>(plan, plan.grid_x, stream);
}

// Loads a lane keeps in flight in the lean kernel: 4 when that divides the loads of a
// wavefront, else 2; 0 when the launch does not fit the kernel (the wavefronts would get
// different or odd numbers of loads: two loads feed one matrix product).
int pick_prefetch(const Plan &plan, int nw) {
    const int gpi = 64 >> plan.p.lpg_log2;
    if (plan.p.gs_tiles % gpi) return 0;
    const int units = plan.p.gs_tiles / gpi;
    if (units % nw) return 0;
    const int u = units / nw;
    if (u < 2 || (u & 1)) return 0;
    const int pf = tuning().gemv4_pf;
    if ((pf == 2 || pf == 4) && u % pf == 0) return pf;
    return u % 4 == 0 ? 4 : 2;
}

template <int LPGL, int NW, bool BF16>
flute_status launch_fast4_pf(Plan &plan, hipStream_t stream) {
    switch (pick_prefetch(plan, NW)) {
        case 2: return launch_fast4<LPGL, NW, 2, BF16>(plan, stream);
        default: return launch_fast4<LPGL, NW, 4, BF16>(plan, stream);
    }
}

template <int LPGL, bool BF16>
flute_status launch_fast4_shape(Plan &plan, int nw, hipStream_t stream) {
    return nw == 4 ? launch_fast4_pf<LPGL, 4, BF16>(plan, stream)
                   : launch_fast4_pf<LPGL, 8, BF16>(plan, stream);
}

template <bool BF16>
flute_status launch_width(Plan &plan, hipStream_t stream) {
    // one width for the whole launch -> the instantiation specialised for it
    int bits = plan.p.seg[0].st[0].bits;
    for (int i = 0; i < plan.p.nsegs; ++i) {
        for (int st = 0; st < plan.p.seg[i].nstreams; ++st) {
            if (plan.p.seg[i].st[st].bits != bits) bits = 0;
        }
    }
    const int nw = plan.threads / 64;
    // (a contiguous run of row slices per XCD: every weight's slices must come in eights)
    plan.p.xcd_runs = tuning().gemv_xcd != 0;
    for (int i = 0; i < plan.p.nsegs; ++i)
        if (((plan.p.seg[i].N >> 7) * (256 >> plan.p.lpg_log2)) % 8 != 0) plan.p.xcd_runs = 0;
    if (plan.k_group) {
        // only the lean kernel knows this form: no general-kernel route
        const int pf = pick_prefetch(plan, nw);
        FLUTE_REQUIRE(pf != 0 && (nw == 4 || (nw == 8 && plan.p.lpg_log2 <= 5)), FLUTE_ERR_UNSUPPORTED,
                      "flute_gemv: K=%d at split %d with %d-row workgroups of %d wavefronts does not "
                      "divide into the loads of the kernel that serves a LUT grouped along K; try "
                      "another split", plan.p.K, plan.p.split, 1 << (plan.p.lpg_log2 - 1), nw);
        plan.p.slices = 0;
        return launch_gemv_kgroup(plan.p, plan.grid_x, nw, pf, plan.lds_bytes, BF16, stream);
    }
    if (plan.lean) {
        int pf = pick_prefetch(plan, nw);
        if (plan.pair == 0 && pf != 0) {
            switch (plan.p.lpg_log2) {
                case 4: return launch_fast4_shape<4, BF16>(plan, nw, stream);
                case 5: return launch_fast4_shape<5, BF16>(plan, nw, stream);
                default: return launch_fast4_shape<6, BF16>(plan, nw, stream);
            }
        }
        plan.p.slices = 0;
        if (pf != 0 && (nw == 4 || plan.p.lpg_log2 <= 5)) {
            // a 1-bit stream with loads that come in eights: the deep ring (launch_pair's pf 8)
            const int u = (plan.p.gs_tiles / (64 >> plan.p.lpg_log2)) / nw;
            if (pf == 4 && plan.pair == 14 && u % 8 == 0 && tuning().gemv4_pf == 0) pf = 8;
            // Grids beyond the resident workgroups walk here too (one weight: gate and up are never that
            // wide; 32-row slices: choose_shape has no more workgroups of narrower ones than are resident),
            // both tables kept while the slices share their LUT rows.  The call, one workgroup per
            // slice and walking:
            //   4096 -> 151936, (4, 1) bits  90.2 -> 79.5 us       4096 -> 248320, 3 bits        93.8 -> 86.3
            //   4096 -> 128000, (2, 4)       87.6 -> 82.5          4096 -> 51200, (1, 4), rotated 42.4 -> 33.1
            //   4096 -> 167552, (3, 3)      111.8 -> 110.2         1024 -> 51200, (3, 3)         17.5 -> 14.3
            int gx = plan.grid_x;
            if (nw == 4 && pf >= 4 && plan.p.nsegs == 1 && plan.p.lpg_log2 == 6)
                if (const int resident = walking_grid(plan)) gx = resident;
            return (plan.pair == 41 || plan.pair == 14)
                       ? launch_gemv_pair_1bit(plan.p, plan.pair, gx, nw, pf, plan.lds_bytes, BF16, stream)
                       : launch_gemv_pair_wide(plan.p, plan.pair, gx, nw, pf, plan.lds_bytes, BF16, stream);
        }
        // K ranges that do not divide into equal, even numbers of loads: the lean kernel's ragged form, which
        // is the faster one wherever it fits.  One token, the general kernel and this one, the launch alone:
        //   3968 -> 2 x 11520, (1, 4) bits   30.0 -> 22.8 us      11520 -> 3968             25.7 -> 11.1
        //   2944 -> 2 x 11904, rotated       23.5 -> 19.0         11904 -> 2944, rotated    20.6 -> 17.4
        //   1152 -> 2 x 4480, (2, 4) bits    19.2 -> 14.8         4480 -> 1152              12.8 -> 9.1
        //   2432 -> 2 x 2304, (3, 3), rotated 20.8 -> 16.1        4032 -> 2048, 512, 512    9.5 -> 6.4
        //   2112 -> 144000: the call 57.9 -> 33.1 (a walking grid), (3, 3) bits 81.3 -> 64.2
        // and of the pairs' walking grid, the call: 3008 -> 100352, (2, 3) bits 58.6 -> 52.8, 3 bits 35.2 -> 30.2;
        // 1600 -> 90112, (4, 1) 28.9 -> 26.6
        int gx = plan.grid_x;
        if (nw == 4 && (plan.pair == 0 || plan.p.nsegs == 1) && plan.p.lpg_log2 == 6)
            if (const int resident = walking_grid(plan)) gx = resident;
        return (plan.pair == 0 || plan.pair == 14 || plan.pair == 41)
                   ? launch_gemv_ragged_a(plan.p, plan.pair, gx, nw, plan.lds_bytes, BF16, stream)
                   : launch_gemv_ragged_b(plan.p, plan.pair, gx, nw, plan.lds_bytes, BF16, stream);
    }
    switch (bits) {
        case 4: return launch_typed<BF16, 4>(plan, stream);
        case 3: return launch_typed<BF16, 3>(plan, stream);
        case 2: return launch_typed<BF16, 2>(plan, stream);
        case 1: return launch_typed<BF16, 1>(plan, stream);
        default: break;
    }
    // mixed widths: the pairs deployed artifacts hold ((1,4) x45, (4,1) x24, (2,3) x3, (2,4) x6
    // in upstream's census, flute_extended/__init__.py:226-233) have instantiations of their own
    int b1 = plan.p.seg[0].st[0].bits, b2 = 0;
    bool pair = true;
    for (int i = 0; i < plan.p.nsegs; ++i) {
        pair &= plan.p.seg[i].st[0].bits == b1;
        if (plan.p.seg[i].nstreams == 2) {
            if (b2 == 0) b2 = plan.p.seg[i].st[1].bits;
            pair &= plan.p.seg[i].st[1].bits == b2;
        }
    }
    if (pair) {
        switch (10 * b1 + b2) {
            case 14: return launch_typed<BF16, 14>(plan, stream);
            case 41: return launch_typed<BF16, 41>(plan, stream);
            case 23: return launch_typed<BF16, 23>(plan, stream);
            case 24: return launch_typed<BF16, 24>(plan, stream);
            default: break;
        }
    }
    return launch_typed<BF16, 0>(plan, stream);
}

// Scratch memory a launch needs beyond its operands: partial sums of a K split, tickets,
// residual coefficients, pre-rotated inputs.
struct ScratchNeed {
    size_t floats, ints;
};
ScratchNeed scratch_need(const Plan &plan) {
    if (!(plan.p_floats || plan.npre)) return {0, 0};
    const size_t xb_pad = (plan.xb_floats + 3) & ~(size_t)3;
    return {plan.p_floats + xb_pad + (plan.xrot_halves + 1) / 2 + 64, (size_t)plan.total_tickets + 1};
}

// fixed_base/fixed_tickets: caller-provided scratch (the allocation-free entry point);
// null = the library's per-device workspace, grown on demand.
flute_status launch(Plan &plan, int act_dtype, hipStream_t stream, float *fixed_base = nullptr,
                    int *fixed_tickets = nullptr) {
    if (plan.p_floats || plan.npre) {
        const size_t xb_pad = (plan.xb_floats + 3) & ~(size_t)3;
        const ScratchNeed need = scratch_need(plan);
        float *base = fixed_base;
        int *tickets = fixed_tickets;
        flute_status st = FLUTE_OK;
        if (!base) st = get_workspace(need.floats, need.ints, stream, &base, &tickets);
        if (st != FLUTE_OK) return st;
        plan.p.P = base;
        plan.p.tickets = tickets;
        float *xb_base = base + plan.p_floats;
        uint16_t *xrot_base = (uint16_t *)(xb_base + xb_pad);
        PreParams pp = {};
        pp.x = plan.p.x;
        pp.K = plan.p.K;
        pp.act_bf16 = plan.p.act_bf16;
        pp.rot_block = plan.rot_block;
        // as few residual rows per workgroup as leave one per CU
        int ranks = 0;
        for (int i = 0; i < plan.npre; ++i) ranks += plan.pre[i].R;
        pp.rows = 1;
        while (pp.rows < kPreWaves && ranks > kNumCU * pp.rows) pp.rows *= 2;
        const bool whole = plan.p.K <= transform_reach(4, kPreThreads);
        int blocks = 0;
        size_t lds = 0;
        for (int i = 0; i < plan.npre; ++i) {
            const Plan::Pre &pre = plan.pre[i];
            uint16_t *const xr = xrot_base + pre.xrot_off;
            float *const xb = xb_base + pre.xb_off;
            if (pre.signs) {
                const size_t cols = whole ? (size_t)plan.p.K
                                    : plan.rot_block > 0 ? (size_t)(16384 / plan.rot_block) * plan.rot_block
                                                         : (size_t)make_segments(plan.p.K, 0).len[0];
                FLUTE_REQUIRE(cols <= 16384 && plan.p.K <= 65504, FLUTE_ERR_UNSUPPORTED,
                              "flute_gemv: the rotation of K=%d columns is not served", plan.p.K);
                lds = cols * 4;
                plan.p.seg[pre.seg].xsrc = xr;
            }
            if (pre.R > 0) plan.p.seg[pre.seg].xb = xb;
            const int rowblocks = (pre.R + pp.rows - 1) / pp.rows;
            if (rowblocks == 0 && pre.share >= 0) continue;      // another weight's rotation is all it needs
            PreSeg &g = pp.seg[pp.nsegs++];
            g.resB = pre.resB;
            g.signs = pre.signs;
            g.awq = pre.awq;
            g.xb = xb;
            g.xrot = pre.signs && pre.share < 0 ? xr : nullptr;
            g.R = pre.R;
            g.block0 = blocks;
            g.vec_b = ((uintptr_t)pre.resB & 15) == 0;
            g.vec_m = ((uintptr_t)pre.signs & 15) == 0 && ((uintptr_t)pre.awq & 15) == 0;
            blocks += rowblocks ? rowblocks : 1;
        }
        if (blocks) {
            static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
            if (!attr_done) {
                for (const void *k : {(const void *)gemv_pre_kernel<true>, (const void *)gemv_pre_kernel<false>})
                    FLUTE_HIP_CHECK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 16384 * 4));
                attr_done = true;
            }
            if (whole) hipLaunchKernelGGL(gemv_pre_kernel<true>, dim3(blocks), dim3(kPreThreads), lds, stream, pp);
            else hipLaunchKernelGGL(gemv_pre_kernel<false>, dim3(blocks), dim3(kPreThreads), lds, stream, pp);
            FLUTE_HIP_CHECK(hipGetLastError());
        }
    }
    const flute_status st = plan.lut_bf16 ? launch_width<true>(plan, stream) : launch_width<false>(plan, stream);
    if ((plan.p_floats || plan.npre) && !fixed_base) workspace_done(stream);
    return st;
}

// ---- the allocation-free variant's scratch ------------------------------------------
// One fixed array per device, part of the code object: held from the time the library is
// loaded on a device until the process ends.  Layout: [tickets: kNoAllocTickets ints]
// [partial sums, residual coefficients, pre-rotated input: the rest as floats].
constexpr size_t kNoAllocBytes = (size_t)2 << 20;
constexpr size_t kNoAllocTickets = 4096;
constexpr size_t kNoAllocFloats = (kNoAllocBytes - kNoAllocTickets * sizeof(int)) / sizeof(float);
constexpr int kMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

__global__ void zero_ints_kernel(int *dst, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = 0;
}

static std::mutex g_scratch_mu;
static unsigned char *g_scratch_ptr[kMaxDevices] = {};

// Device address of this device's copy of the array (the array's name is a host-side
// stand-in, not a device address): resolved once per device, with that device current.
flute_status noalloc_scratch(unsigned char **out, hipStream_t stream) {
    int dev = 0;
    FLUTE_HIP_CHECK(hipGetDevice(&dev));
    FLUTE_REQUIRE(dev >= 0 && dev < kMaxDevices, FLUTE_ERR_UNSUPPORTED,
                  "flute_gemv_noalloc: device ordinal %d beyond %d", dev, kMaxDevices);
    std::lock_guard<std::mutex> guard(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        // resolving the symbol may load the code object: not something to do inside a capture
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        FLUTE_HIP_CHECK(hipStreamIsCapturing(stream, &cap));
        FLUTE_REQUIRE(cap == hipStreamCaptureStatusNone, FLUTE_ERR_INVALID,
                      "flute_gemv_noalloc: the first call on device %d that needs the scratch array "
                      "resolves its address and must not be under stream capture; make one such "
                      "call outside the capture first", dev);
        unsigned char *ptr = nullptr;
        FLUTE_HIP_CHECK(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
        FLUTE_REQUIRE(ptr != nullptr, FLUTE_ERR_HIP,
                      "flute_gemv_noalloc: the scratch array has no address on device %d", dev);
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return FLUTE_OK;
}

}  // namespace

}  // namespace flute

using namespace flute;

extern "C" {

flute_status flute_gemv(const flute_linear *w, const void *x, void *y, int act_dtype, int split,
                        void *stream) {
    Plan plan;
    void *outs[1] = {y};
    flute_status st = make_plan(w, 1, x, outs, act_dtype, split, 0, "flute_gemv", &plan);
    if (st != FLUTE_OK) return st;
    return launch(plan, act_dtype, (hipStream_t)stream);
}

flute_status flute_gemv_noalloc(const flute_linear *w, const void *x, void *y, int act_dtype,
                                int split, void *stream) {
    Plan plan;
    void *outs[1] = {y};
    flute_status st = make_plan(w, 1, x, outs, act_dtype, split, 0, "flute_gemv_noalloc", &plan);
    if (st != FLUTE_OK) return st;
    const ScratchNeed need = scratch_need(plan);
    FLUTE_REQUIRE(need.floats <= kNoAllocFloats && need.ints <= kNoAllocTickets,
                  FLUTE_ERR_UNSUPPORTED,
                  "flute_gemv_noalloc: this launch needs %zu B of scratch and %zu tickets; the fixed "
                  "array holds %zu B and %zu tickets (N=%d, K=%d, R=%d, split=%d). Use flute_gemv, "
                  "or a smaller split",
                  need.floats * sizeof(float), need.ints, kNoAllocFloats * sizeof(float),
                  kNoAllocTickets, w->N, w->K, w->R, plan.p.split);
    if (need.floats == 0) return launch(plan, act_dtype, (hipStream_t)stream);
    unsigned char *ptr = nullptr;
    st = noalloc_scratch(&ptr, (hipStream_t)stream);
    if (st != FLUTE_OK) return st;
    int *tickets = (int *)ptr;
    float *base = (float *)(ptr + kNoAllocTickets * sizeof(int));
    if (plan.p.split > 1) {
        // the array keeps the last call's contents: tickets must start at zero (a fill
        // kernel, not a memset node, so that the call can be captured into a graph)
        const int n = (int)need.ints;
        hipLaunchKernelGGL(zero_ints_kernel, dim3((n + 255) / 256), dim3(256), 0,
                           (hipStream_t)stream, tickets, n);
        FLUTE_HIP_CHECK(hipGetLastError());
    }
    return launch(plan, act_dtype, (hipStream_t)stream, base, tickets);
}

flute_status flute_gemv_mlp(const flute_linear *gate, const flute_linear *up, const void *x,
                            void *h, int act_dtype, int split, void *stream) {
    FLUTE_REQUIRE(gate && up, FLUTE_ERR_INVALID, "flute_gemv_mlp: gate/up descriptor is NULL");
    flute_linear segs[2] = {*gate, *up};
    void *outs[2] = {h, h};
    Plan plan;
    flute_status st = make_plan(segs, 2, x, outs, act_dtype, split, 1, "flute_gemv_mlp", &plan);
    if (st != FLUTE_OK) return st;
    return launch(plan, act_dtype, (hipStream_t)stream);
}

flute_status flute_gemv_multi(const flute_linear *segs, int count, const void *x,
                              void *const *outs, int act_dtype, int split, void *stream) {
    FLUTE_REQUIRE(segs && outs, FLUTE_ERR_INVALID, "flute_gemv_multi: NULL argument");
    Plan plan;
    flute_status st =
        make_plan(segs, count, x, outs, act_dtype, split, 0, "flute_gemv_multi", &plan);
    if (st != FLUTE_OK) return st;
    return launch(plan, act_dtype, (hipStream_t)stream);
}

flute_status flute_mlp_block(const flute_linear *gate, const flute_linear *up,
                             const flute_linear *down, const void *x, void *h, void *y,
                             int act_dtype, void *stream) {
    FLUTE_REQUIRE(gate && up && down, FLUTE_ERR_INVALID, "flute_mlp_block: NULL descriptor");
    FLUTE_REQUIRE(down->K == gate->N, FLUTE_ERR_INVALID,
                  "flute_mlp_block: down K (%d) must equal gate/up N (%d)", down->K, gate->N);
    flute_status st = flute_gemv_mlp(gate, up, x, h, act_dtype, 0, stream);
    if (st != FLUTE_OK) return st;
    return flute_gemv(down, h, y, act_dtype, 0, stream);
}

int flute_pick_split(int N, int K) {
    if (N <= 0 || K <= 0 || N % 128 || K % 64) return 1;
    int rw, split, waves;
    choose_shape(N, K / 64, 0, &rw, &split, &waves);
    return split;
}

int flute_gemv_rows(const flute_linear *ws, int count, int *waves) {
    if (!ws || count < 1 || count > kGemvMaxSegs) return -1;
    Plan plan;
    alignas(16) char dummy[16] = {};                        // never dereferenced
    void *outs[kGemvMaxSegs];
    for (void *&o : outs) o = dummy;
    if (make_plan(ws, count, dummy, outs, ws[0].lut_dtype == FLUTE_BF16 ? FLUTE_BF16 : FLUTE_F16, 0, 0, "flute_gemv_rows",
                  &plan) != FLUTE_OK)
        return -1;
    if (waves) *waves = plan.threads / 64;
    return 1 << (plan.p.lpg_log2 - 1);
}

int64_t flute_gemv_lds_bytes(const flute_linear *w, int split) {
    Plan plan;
    alignas(16) char dummy_x[16] = {}, dummy_y[16] = {};    // never dereferenced
    void *outs[1] = {dummy_y};
    if (make_plan(w, 1, dummy_x, outs, (w && w->lut_dtype == FLUTE_BF16) ? FLUTE_BF16 : FLUTE_F16,
                  split, 0, "flute_gemv_lds_bytes", &plan) != FLUTE_OK)
        return 0;
    return (int64_t)plan.lds_bytes;
}

}  // extern "C"

#ifdef FLUTE_STAMPS
// Instrumented builds only: where the lean kernel writes its phase times (NULL switches them off).
extern "C" int flute_debug_gemv_stamps(void *buf) {
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(g_gemv_stamps), &buf, sizeof(buf));
}
#endif
