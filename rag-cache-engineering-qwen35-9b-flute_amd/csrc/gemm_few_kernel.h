// LUT GEMM for few rows (workgroups of 16 or 32 rows of A):  C[M, N] = A[M, K] @ (W1 (+ W2))^T, fp32
// accumulate, one rounding.  The operands' layout is that of gemm_kernel.h: a lane's chunk of codes
// is what it needs of the matrix instruction's row side, the weights never exist as a dense tile.
//
// Workgroup = eight wavefronts on one 128-row tile of the weight; wavefront w takes the K tiles w,
// w + 8, ... of the workgroup's slice of K, for MB blocks of 16 rows of A, both streams of a tile one
// after the other on the same activations.  What bounds it: such a launch is a few trips to memory and
// through LDS around a loop of a few microseconds (M = 48, 12288 -> 4096, four slices of K, six tiles a
// wavefront: 4 bits 8 us of loop in a launch of 16, (4, 1) bits 13 of 22), so a second stream costs its
// loop here and not a launch of its own, and the eight wavefronts' sums cross LDS once, every thread
// adding the eight terms of the outputs it then stores, instead of a tree of three steps with two
// barriers each and a totals tile behind it.
#pragma once

#include "gemm_kernel.h"

namespace flute {

// Lookup tables of a stream in LDS.  An entry holds `slots` copies, split evenly over the LUT groups
// of the 128-row tile, so that the lanes of an instruction lie on different banks.  4 and 3 bits: an
// entry is a pair of weights (a dword).  2 and 1 bits: the four weights of a byte (a nibble) of
// codes, half an operand, which halves the lookups and their addresses.  4 bits: 256 bytes an entry,
// table at LDS offset 0, so that one v_perm_b32 drops a code byte into the address.
template <int B>
struct FewTable {
    static constexpr int entries = B == 4 ? 256 : B == 3 ? 64 : B == 2 ? 256 : B == 1 ? 16 : 0;
    static constexpr int stride_log2 = B == 4 ? 8 : 7;
    static constexpr int unit = B >= 3 ? 4 : 8;
    static constexpr int slots = (1 << stride_log2) / unit;
    static constexpr int bytes = entries << stride_log2;
    static constexpr int stage = B * 1024;                       // one tile of codes
};

template <int B1, int B2, int MB>
constexpr int few_lds_bytes() {
    constexpr int loop = FewTable<B1>::bytes + FewTable<B2>::bytes + 8 * (FewTable<B1>::stage + FewTable<B2>::stage);
    constexpr int sums = 8 * MB * 8 * 64 * 16 + 16;              // every wavefront's accumulators, a flag
    return loop > sums ? loop : sums;
}

// Bytes of a launch: behind the above, the scales of sixteen rows that a workgroup looks for itself, and every
// wavefront's residual coefficients.
template <int B1, int B2, int FORM>
constexpr int few_lds_total() {
    constexpr int MB = FORM == 1 || FORM == 4 ? 1 : 2;
    return few_lds_bytes<B1, B2, MB>() + (MB == 1 ? 64 : 0) + (FORM >= 4 ? 8 * MB * 64 * 16 : 0);
}

// What a thread contributes to a table: the LUT values its entries are made of, requested with the
// kernel's first loads; `build` waits for them only.
template <int B>
struct FewLut {
    uint32_t v[B == 4 ? 6 : B == 3 ? 2 : B == 2 ? 4 : 2];

    // lanes per entry, and the LUT group of this lane's 16 bytes of an entry
    static constexpr int lanes = B == 4 ? 16 : 8;
    __device__ __forceinline__ void load(const GemmSeg &w, int s, int t, int lane, int wave) {
        const int lg = __builtin_ctz((unsigned)w.gs);            // a power of two, 16 or more
        const int ngrp = lg >= 7 ? 1 : 128 >> lg;
        const int gl = ((lane & (lanes - 1)) * ngrp) / lanes;
        const int row = min(lg >= 7 ? (t * 128) >> lg : t * ngrp + gl, w.lut_rows - 1);
        const uint16_t *lr = w.lut[s] + ((size_t)row << B);
        if constexpr (B == 4) {                                  // codes 32 * wave + 4 * it + lane / 16
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = lr[4 * i + (lane >> 4)];
            v[4] = lr[2 * wave];
            v[5] = lr[2 * wave + 1];
        } else if constexpr (B == 3) {                           // code 8 * wave + lane / 8
            v[0] = lr[lane >> 3];
            v[1] = lr[wave];
        } else {
#pragma unroll
            for (int i = 0; i < (1 << B); ++i) v[i] = lr[i];
        }
    }
    // B == 2: value i of the four.  A shift: selects over v became an array in scratch memory, in front of the
    // table's barrier (4096 -> 4096, M = 8: 2 bits 8.5 -> 7.8 us, (2, 4) 11.1 -> 10.5, (2, 3) 11.2 -> 10.5).
    __device__ __forceinline__ uint32_t of4(int i) const {
        const uint64_t four = (uint64_t)(v[0] | (v[1] << 16)) | ((uint64_t)(v[2] | (v[3] << 16)) << 32);
        return (uint32_t)(four >> (16 * i)) & 0xffffu;
    }
    __device__ __forceinline__ void build(unsigned char *table, int lane, int wave) const {
        u4_t *const to = (u4_t *)table + lane;                   // an instruction writes 64 / lanes entries
        if constexpr (B == 4) {
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const uint32_t d = v[it & 3] | (v[4 + (it >> 2)] << 16);
                to[(wave * 8 + it) * 64] = u4_t{d, d, d, d};
            }
        } else if constexpr (B == 3) {
            const uint32_t d = v[0] | (v[1] << 16);
            to[wave * 64] = u4_t{d, d, d, d};
        } else if constexpr (B == 2) {
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                const int code = wave * 32 + it * 8 + (lane >> 3);
                const uint32_t lo = of4(code & 3) | (of4((code >> 2) & 3) << 16);
                const uint32_t hi = of4((code >> 4) & 3) | (of4(code >> 6) << 16);
                to[(wave * 4 + it) * 64] = u4_t{lo, hi, lo, hi};
            }
        } else if (wave < 2) {
            const int code = wave * 8 + (lane >> 3);
            const uint32_t lo = ((code & 1) ? v[1] : v[0]) | (((code & 2) ? v[1] : v[0]) << 16);
            const uint32_t hi = ((code & 4) ? v[1] : v[0]) | (((code & 8) ? v[1] : v[0]) << 16);
            to[wave * 64] = u4_t{lo, hi, lo, hi};
        }
    }
};

// One stream of a workgroup's tile: its codes on their way from memory to the matrix operands.
template <int B>
struct FewStream {
    u4_t raw[B];               // a tile on its way from memory, contiguous 1 KB rows
    uint32_t Q[4 * B];         // this lane's chunk of the tile in work
    uint32_t lb[4];            // table column of this lane for the rows (wx, v)
    uint32_t wr[B], rd[B];     // staging: where a lane puts its piece of a row, where its chunk's pieces are
    const uint8_t *p;

    // A tile passes through LDS on its way (contiguous loads cost the address path a quarter of what
    // loads of whole chunks do).  Piece i of chunk c = 4 * a + kg is q = B * c + i = 4 * B * a + m; it
    // lies at m * 16 + (a ^ (m & 7)): lanes that write neighbouring pieces and lanes that read the
    // chunks of neighbouring rows both meet different banks.
    __device__ __forceinline__ void init(const GemmSeg &w, int s, int64_t tile, uint32_t table, uint32_t stage, int lane) {
        typedef FewTable<B> T;
        p = w.q[s] + tile * (1024 * B) + lane * 16;
        const int rho = lane & 15, kg = lane >> 4, wx = rho >> 3;
#pragma unroll
        for (int i = 0; i < B; ++i) {
            const uint32_t q = i * 64 + lane, m = q % (4 * B), a = q / (4 * B);
            wr[i] = stage + (m * 16 + (a ^ (m & 7))) * 16;
            const uint32_t mr = B * kg + i;
            rd[i] = stage + (mr * 16 + ((uint32_t)rho ^ (mr & 7))) * 16;
        }
        const int lg = __builtin_ctz((unsigned)w.gs);
        const int ngrp = lg >= 7 ? 1 : 128 >> lg;
        const int reps = lg >= 7 ? T::slots : T::slots >> (7 - lg);
        const int r = ngrp == 1 ? lane & (T::slots - 1) : ((kg * 8 + (rho & 7)) ^ (wx * 16)) & (reps - 1);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int gl = ngrp == 1 ? 0 : (wx * 64 + v * 16) >> lg;
            lb[v] = table + (gl * reps + r) * T::unit;
        }
    }
    __device__ __forceinline__ void load() {
#pragma unroll
        for (int i = 0; i < B; ++i) raw[i] = __builtin_nontemporal_load((const u4_t *)(p + i * 1024));
    }
    typedef __attribute__((address_space(3))) u4_t *LdsQuad;
    __device__ __forceinline__ void put() const {
#pragma unroll
        for (int i = 0; i < B; ++i) *(LdsQuad)(uintptr_t)wr[i] = raw[i];
    }
    __device__ __forceinline__ void get() {
#pragma unroll
        for (int i = 0; i < B; ++i) {
            const u4_t v = *(LdsQuad)(uintptr_t)rd[i];
#pragma unroll
            for (int e = 0; e < 4; ++e) Q[4 * i + e] = v[e];
        }
    }
    // operand (rows v, d; half j of the tile)
    __device__ __forceinline__ u4_t operand(int j, int v, int d) const {
        if constexpr (B >= 3) {
            return fetch_operand<B, B == 4>(Q, j, v, d, lb[v], FewTable<B>::stride_log2);
        } else {
            typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
            typedef const __attribute__((address_space(3))) u2_t *LdsPair;
            u4_t w;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const int bit = 2 * B * ((2 * j + kt) * 16 + v * 4 + d * 2);       // four codes: 4 * B bits
                const uint32_t code = __builtin_amdgcn_ubfe(Q[bit >> 5], bit & 31, 4 * B);
                const u2_t two = *(LdsPair)(uintptr_t)((code << FewTable<B>::stride_log2) + lb[v]);
                w[2 * kt] = two[0];
                w[2 * kt + 1] = two[1];
            }
            return w;
        }
    }
};
template <>
struct FewStream<0> {};

// Rows held scaled by 2^-shift that carry a residual: their sums are scaled back to 2^-few_lift of their
// magnitude ahead of the residual, and by the rest in the epilogue.  Partial sums of such a row stay
// below 2^(shift + 34) (operands below 2, two float16 LUT values, K up to 2^16), so up to shift 92 they
// fit fp32 as they are; beyond, they may leave its range where the row's sum does not, and are kept
// 2^36 smaller, as is the residual (which loses bits below 2^-90 there, next to a row of 2^93 or more).
__device__ __forceinline__ int few_lift(int shift) { return shift > 92 ? 36 : 0; }

// B2 == 0: one stream (launches of one stream each may share a fold, p.z_base and p.ztotal).
// SEGS: several weights in the launch.
// FORM: 1: 16 rows, of A or of the image; 2: 32 rows of the image; 3: 32 rows of A; 4, 5: as 1 and 3, of A, with the
// residual's coefficients.  (Forms of their own: what 32 rows need to read A themselves costs the image's launches
// 0.6 us where they step over it, and a loop for each in one kernel costs more, in registers and in code that every
// launch fetches.)
template <int FORM, bool BF16, int B1, int B2, bool SEGS>
__global__ void __launch_bounds__(512) gemm_few_kernel(const GemmParams p) {
    static_assert(FORM >= 1 && FORM <= 5, "16 or 32 rows");
    constexpr int MB = FORM == 1 || FORM == 4 ? 1 : 2;
    constexpr bool COEFF = FORM >= 4;
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int KW = 8, NT = 512;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int si = 0;
    if constexpr (SEGS)
        si = ((int)blockIdx.x >= p.tile0[1]) + ((int)blockIdx.x >= p.tile0[2]) + ((int)blockIdx.x >= p.tile0[3]);
    const GemmSeg &w = p.seg[SEGS ? si : 0];
    const int t = SEGS ? blockIdx.x - p.tile0[si] : blockIdx.x;
    const int mb0 = blockIdx.y * MB;                   // first 16-row block
    const int z = blockIdx.z;
    const int rho = lane & 15, kg = lane >> 4;

    const int gbeg = z * p.gper, gend = min(p.G, gbeg + p.gper);
    const int g0 = gbeg + wave;
    int left = g0 < gend ? (gend - g0 + KW - 1) / KW : 0;   // tiles of this wavefront
    // A wavefront without tiles addresses the first one of the slice instead: the loads below are then
    // unconditional like everyone's, and the compiler can count them.
    const int g_first = left > 0 ? g0 : gbeg;

    // ---- activations: A itself where its rows are whole 16-byte pieces, put into operand order in registers,
    // or the image (its blocks are padded to whole workgroups) ------------------------------------------
    const bool direct = FORM >= 3 || (FORM == 1 && p.A8 != nullptr);
    const bool find = MB == 1 && p.find;
    // Four lanes to the 64 bytes of a row, as the address path likes it (lane per row and piece: 64 accesses an
    // instruction, not 16), in the order of rows that to_operand leaves as 0 ... 15.  Rows beyond M repeat the
    // last: nobody stores their outputs.
    const int load_row = ((lane >> 2) & 3) * 4 + (lane >> 4);
    int a_shift[MB];                                    // of row rho
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) a_shift[mb] = 0;
    // (uniform base, 32-bit offsets of a lane: few_lda bounds the stride)
    const int64_t jstep = direct ? 4 : (int64_t)p.mblk_pad * 64, gstep = direct ? 8 : 2 * jstep;
    const u4_t *ap = (direct ? p.A8 + (int64_t)mb0 * 16 * p.lda8 : p.Ap + (int64_t)mb0 * 64) + (int64_t)g_first * gstep;
    uint32_t a_ofs[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
        a_ofs[mb] = direct ? ((uint32_t)(min((mb0 + mb) * 16 + load_row, p.M - 1) - mb0 * 16) * (uint32_t)p.lda8 + (lane & 3)) * 16
                           : mb * 1024 + lane * 16;
    auto load_a = [&](u4_t (&Aj)[MB], int64_t ofs) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) Aj[mb] = *(const u4_t *)((const char *)(ap + ofs) + a_ofs[mb]);
    };
    // COEFF: the residual's coefficients, A @ resB^T over this slice of K, as one more operand of sixteen weights: rank
    // r in the place of row r.  They cost the loop an eighth of its products and a load of half its codes' size
    // instead of a launch in front: M = 8, 4096 -> 4096, rank 16 14.0 -> 10.0 us; M = 48, 12288 -> 4096, (4, 1) bits
    // 30.3 -> 26.5; M = 22, 6912 -> 4224, (2, 3) bits 27.4 -> 18.2 (of which 5 by 32-row workgroups); M = 200, 4096 ->
    // 4096 23.7 -> 20.2.  fp32 sums of products of the activations' own type.
    const u4_t *bp = COEFF ? (const u4_t *)w.resB + (int64_t)g_first * 8 : nullptr;
    const uint32_t b_ofs = COEFF ? ((uint32_t)min(load_row, w.R - 1) * (uint32_t)(p.G * 8) + (lane & 3)) * 16 : 0;
    u4_t RB0 = {0u, 0u, 0u, 0u}, RB1 = {0u, 0u, 0u, 0u};
    f4_t xacc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) xacc[mb] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto load_b = [&](u4_t &to, int ofs) {
        if constexpr (COEFF) to = *(const u4_t *)((const char *)(bp + ofs) + b_ofs);
    };
    // A lane has loaded piece lane & 3 of its row, eight consecutive k; the matrix cores want lane kg * 16 + rho to
    // hold the pairs (2*kg, 2*kg + 1) of all four pieces of row rho, in the LUT's 16-bit type: dwords change
    // places with the lane's upper two bits, then with the lower two.
    auto transposed = [&](u4_t v) {
        uint32_t q[4] = {v[0], v[1], v[2], v[3]};
        transpose_lanes16(q);
        transpose_quad(q, lane);
        return u4_t{q[0], q[1], q[2], q[3]};
    };
    auto to_operand = [&](u4_t (&T)[MB], u4_t rb) {
        if (!direct) return;
        if constexpr (COEFF) rb = transposed(rb);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) T[mb] = transposed(T[mb]);
        if constexpr (!BF16) {
            if (p.a_bf16) {
                typedef float f2_t __attribute__((ext_vector_type(2)));
                typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    if constexpr (COEFF) xacc[mb] = mfma16<true>(rb, T[mb], xacc[mb]);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        T[mb][e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(
                            (f2_t{ldexpf(__builtin_bit_cast(float, T[mb][e] << 16), -a_shift[mb]),
                                  ldexpf(__builtin_bit_cast(float, T[mb][e] & 0xffff0000u), -a_shift[mb])}), h2_t));
                }
                return;
            }
        }
        if constexpr (COEFF)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) xacc[mb] = mfma16<BF16>(rb, T[mb], xacc[mb]);
    };

    // ---- first loads, in the order they are waited for: LUT values, codes, activations ------------
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    constexpr int tab2 = FewTable<B1>::bytes, stage0 = tab2 + FewTable<B2>::bytes;
    constexpr int stage_wave = FewTable<B1>::stage + FewTable<B2>::stage;
    const uint32_t stage = lds0 + stage0 + (uint32_t)wave * stage_wave;
    // (the residual's first sixteen ranks in front of all: what comes behind them can still be counted)
    const bool residual = COEFF || (w.R > 0 && p.z_base + z == 0);
    uint16_t res_a[4] = {0, 0, 0, 0};
    float res_x[MB][4];
    const uint16_t *const res_row = w.resA + (int64_t)(t * 128 + (rho >> 3) * 64 + wave * 8 + (rho & 7)) * w.R;
    auto residual_load = [&](int r0) {
        const int k0 = r0 + kg * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            res_a[e] = k0 + e < w.R ? res_row[k0 + e] : (uint16_t)0;
            if constexpr (!COEFF)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    res_x[mb][e] = k0 + e < w.R ? w.xb[(int64_t)min((mb0 + mb) * 16 + rho, p.M - 1) * w.R + k0 + e] : 0.0f;
        }
    };
    if (residual) residual_load(0);
    int unscale[MB];                                    // (with a residual: sums leave the loop's scale at once)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
        unscale[mb] = w.R > 0 && p.rowshift ? p.rowshift[min((mb0 + mb) * 16 + rho, p.M - 1)] : 0;
    FewLut<B1> lut1;
    FewLut<B2 ? B2 : 1> lut2;
    FewStream<B1> s1;
    FewStream<B2> s2;
    u4_t A0[MB], A1[MB];
    lut1.load(w, 0, t, lane, wave);
    if constexpr (B2 > 0) lut2.load(w, 1, t, lane, wave);
    const int64_t tile = (int64_t)t * p.G + g_first;
    s1.init(w, 0, tile, lds0, stage, lane);
    if constexpr (B2 > 0) s2.init(w, 1, tile, lds0 + tab2, stage + FewTable<B1>::stage, lane);
    __builtin_amdgcn_sched_barrier(0);
    s1.load();
    if constexpr (B2 > 0) s2.load();
    load_a(A0, 0);
    load_b(RB0, 0);
    load_a(A1, jstep);
    load_b(RB1, 4);
    __builtin_amdgcn_sched_barrier(0);
    if (direct && p.rowshift)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) a_shift[mb] = p.rowshift[min((mb0 + mb) * 16 + rho, p.M - 1)];
    lut1.build(smem, lane, wave);
    if constexpr (B2 > 0) lut2.build(smem + tab2, lane, wave);
    // bfloat16 rows in front of a float16 LUT: each wavefront looks two of the workgroup's rows through for
    // their scales (few_finds).
    int *const found = (int *)(smem + few_lds_bytes<B1, B2, MB>());
    if (find) {
        const int pieces = p.G * 8;                     // of a row
        for (int r = wave; r < 16 && mb0 * 16 + r < p.M; r += 8) {
            const u4_t *const row = p.A8 + (int64_t)(mb0 * 16 + r) * p.lda8;
            uint32_t e = 0;
            for (int i = 0; i < pieces; i += 512) {     // (past the end: the last piece again)
                u4_t v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = row[min(i + u * 64 + lane, pieces - 1)];
#pragma unroll
                for (int u = 0; u < 8; ++u) e = max(e, bf16_max_exp8(make_uint4(v[u][0], v[u][1], v[u][2], v[u][3])));
            }
            e = wavefront_max(e);
            if (lane == 0) found[r] = bf16_row_shift(e);
        }
    }
    __syncthreads();
    if (find) {
        a_shift[0] = found[min(rho, p.M - 1 - mb0 * 16)];
        if constexpr (COEFF) unscale[0] = a_shift[0];
    }

    f4_t acc[MB][8];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[mb][i] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // ---- the K loop: codes a tile and a half ahead (through LDS), activations half a tile or more -------
    auto next_codes = [&](bool more) {
        s1.put();
        if constexpr (B2 > 0) s2.put();
        if (more) {                                     // else: a harmless reload
            s1.p += KW * 1024 * B1;
            if constexpr (B2 > 0) s2.p += KW * 1024 * B2;
        }
        s1.load();
        if constexpr (B2 > 0) s2.load();
    };
    // A turn is one run of operand pairs (half a tile: four of the first stream, four of the second), MB products
    // an operand.  The lookups run two pairs ahead of the products that consume them, from one half and
    // stream into the next, and the next tile's codes leave the staging behind the last of them, so that LDS
    // latency hides behind matrix work.
    constexpr int STREAMS = B2 > 0 ? 2 : 1, HALF = 4 * STREAMS, PAIRS = 2 * HALF, AHEAD = 2;
    u4_t W[AHEAD + 1][2];
    auto lookup = [&](int u) {
        const int j = u / HALF, v = u & 3;
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            if constexpr (B2 > 0) W[u % (AHEAD + 1)][d] = (u & 4) ? s2.operand(j, v, d) : s1.operand(j, v, d);
            else W[u % (AHEAD + 1)][d] = s1.operand(j, v, d);
        }
    };
    auto get_codes = [&]() {
        s1.get();
        if constexpr (B2 > 0) s2.get();
    };
    if (left > 0) {
        next_codes(left > 1);
        get_codes();
    }
    while (left > 0) {
        // the two wavefronts of a SIMD (w and w + 4) take turns at the higher priority
        if ((left + (wave >> 2)) & 1) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) lookup(u);
        to_operand(A0, RB0);
#pragma unroll
        for (int u = 0; u < PAIRS; ++u) {
            if (u + AHEAD < PAIRS) lookup(u + AHEAD);
            if (u + AHEAD == PAIRS) get_codes();
            if (u == HALF) {
                if (left > 1) {
                    ap += KW * gstep;
                    if constexpr (COEFF) bp += KW * 8;
                }
                load_a(A0, 0);
                load_b(RB0, 0);
                // issue order activations -> codes: the wait for these activations at the top of the next
                // round then does not include the codes'
                __builtin_amdgcn_sched_barrier(0);
                next_codes(left > 2);
                __builtin_amdgcn_sched_barrier(0);
                to_operand(A1, RB1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    acc[mb][(u & 3) * 2 + d] = mfma16<BF16>(W[u % (AHEAD + 1)][d], u < HALF ? A0[mb] : A1[mb],
                                                            acc[mb][(u & 3) * 2 + d]);
            __builtin_amdgcn_sched_barrier(0);
        }
        load_a(A1, jstep);
        load_b(RB1, 4);
        __builtin_amdgcn_sched_barrier(0);
        --left;
    }
    __builtin_amdgcn_s_setprio(0);

    // ---- residual: + xb @ resA^T, in fp32 products onto the sums of the first slice (COEFF: of each) ---
    // Wavefront i takes the outputs of accumulator i, sixteen ranks a step, of which lane group kg holds
    // four (the order of ranks is free as long as both operands agree): a few loads a lane, requested
    // with the first loads of one slice, where the threads of the last arrival read eight rows of resA
    // each behind the exchange.  Sums of rows that are held scaled are
    // scaled back ahead of it, in every slice: a residual may be of another magnitude than its row, and
    // is added at its own (few_lift).
    if (w.R > 0 && (p.rowshift || find)) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[mb][i][q] = ldexpf(acc[mb][i][q], unscale[mb] - few_lift(unscale[mb]));
    }
    if constexpr (COEFF) {                              // of all wavefronts, in their order
        f4_t *const part = (f4_t *)(smem + few_lds_bytes<B1, B2, MB>() + (MB == 1 ? 64 : 0));
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) part[(wave * MB + mb) * 64 + lane] = xacc[mb];
        __syncthreads();                                // tables and staging are dead
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            f4_t sum = part[mb * 64 + lane];
#pragma unroll
            for (int u = 1; u < 8; ++u) sum += part[(u * MB + mb) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) res_x[mb][e] = kg * 4 + e < w.R ? sum[e] : 0.0f;
        }
    }
    if (residual) {
        f4_t sum[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) sum[mb] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
        for (int r0 = 0; r0 < w.R; r0 += 16) {
            if (r0 > 0) residual_load(r0);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    sum[mb] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.out_bf16 ? bf2f(res_a[e]) : h2f(res_a[e]),
                                                                  res_x[mb][e], sum[mb], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (i != wave) continue;                    // uniform
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[mb][i][q] += ldexpf(sum[mb][q], -few_lift(unscale[mb]));
        }
    }

    // ---- sums of the eight wavefronts ---------------------------------------------------------
    // Four outputs of one row = one f4: accumulator i of lane (kg, rho) holds row rho, outputs
    // (kg >> 1) * 64 + i * 8 + (kg & 1) * 4 ... + 3.  A wavefront's area is in that order, the lane's
    // low bits XORed with the outputs' so that the sixteen (eight) threads that serve a row of C side
    // by side read different banks.
    if constexpr (!COEFF) __syncthreads();              // tables and staging are dead
    f4_t *const red = (f4_t *)smem;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            red[(wave * MB + mb) * 512 + i * 64 + (lane ^ i ^ ((kg & 1) << 2))] = acc[mb][i];
    __syncthreads();
    constexpr int PW = 4 * MB;                          // outputs per thread: 16 * MB rows, 128 columns in all
    const int ml = tid / (128 / PW), n_in = (tid % (128 / PW)) * PW;
    float y[PW];
#pragma unroll
    for (int e = 0; e < MB; ++e) {
        const int n = n_in + 4 * e, i = (n >> 3) & 7, lo = (n >> 2) & 1;
        const f4_t *from = red + (ml >> 4) * 512 + i * 64 + ((((n >> 6) * 2 + lo) * 16 + (ml & 15)) ^ i ^ (lo << 2));
        f4_t sum = from[0];
#pragma unroll
        for (int u = 1; u < 8; ++u) sum += from[u * MB * 512];
#pragma unroll
        for (int q = 0; q < 4; ++q) y[4 * e + q] = sum[q];
    }

    // ---- across workgroups: partial sums and a ticket, the last arrival adds them in z order ---------
    if (p.ztotal > 1) {
        const int unit = blockIdx.y * gridDim.x + blockIdx.x, zmine = p.z_base + z;
        constexpr int image = NT * PW;
        const int64_t zstride = (int64_t)gridDim.x * gridDim.y * image;
        float *const mine = p.P + (int64_t)unit * image + tid * 4;
#pragma unroll
        for (int e = 0; e < MB; ++e)
            ws_store16(mine + zmine * zstride + e * (NT * 4), f4_t{y[4 * e], y[4 * e + 1], y[4 * e + 2], y[4 * e + 3]});
        ws_stores_done();
        __syncthreads();
        int *const flag = (int *)(smem + 8 * MB * 8 * 64 * 16);
        if (tid == 0) {
            const int old = __hip_atomic_fetch_add(p.tickets + unit, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *flag = old == p.ztotal - 1;
            if (old == p.ztotal - 1)
                __hip_atomic_store(p.tickets + unit, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!*flag) return;
        f4_t sum[MB];
#pragma unroll
        for (int e = 0; e < MB; ++e) sum[e] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
        for (int z0 = 0; z0 < p.ztotal; z0 += 4) {      // past the last slice: that one again, not added
#pragma unroll
            for (int e = 0; e < MB; ++e) {
                const float *s[4];
                f4_t v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) s[i] = mine + min(z0 + i, p.ztotal - 1) * zstride + e * (NT * 4);
                ws_load16x4(s[0], s[1], s[2], s[3], v[0], v[1], v[2], v[3]);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (z0 + i < p.ztotal) sum[e] += v[i];
            }
        }
#pragma unroll
        for (int e = 0; e < MB; ++e)
#pragma unroll
            for (int q = 0; q < 4; ++q) y[4 * e + q] = sum[e][q];
    }

    // ---- epilogue: scale back, bias, one rounding, store ------------------------------------------
    const int m = blockIdx.y * (16 * MB) + ml;
    if (m >= p.M) return;
    const int n0 = t * 128 + n_in;
    if (p.rowshift || find) {                           // exact
        const int row_shift = find ? found[ml] : p.rowshift[m], sh = w.R == 0 ? row_shift : few_lift(row_shift);
#pragma unroll
        for (int e = 0; e < PW; ++e) y[e] = ldexpf(y[e], sh);
    }
    if (w.bias) {
#pragma unroll
        for (int e = 0; e < PW; ++e) y[e] += load_act(w.bias, n0 + e, p.out_bf16);
    }
    uint32_t o[PW / 2];
#pragma unroll
    for (int e = 0; e < PW / 2; ++e)
        o[e] = (uint32_t)round_act(y[2 * e], p.out_bf16) | ((uint32_t)round_act(y[2 * e + 1], p.out_bf16) << 16);
    uint16_t *const dst = (uint16_t *)w.C + (size_t)m * w.ldc + n0;
    if (w.vec_store) {
        if constexpr (MB == 2) *(u4_t *)dst = u4_t{o[0], o[1], o[2], o[3]};
        else *(uint2 *)dst = make_uint2(o[0], o[1]);
    } else {
#pragma unroll
        for (int e = 0; e < PW / 2; ++e) {
            dst[2 * e] = (uint16_t)o[e];
            dst[2 * e + 1] = (uint16_t)(o[e] >> 16);
        }
    }
}

}  // namespace flute
