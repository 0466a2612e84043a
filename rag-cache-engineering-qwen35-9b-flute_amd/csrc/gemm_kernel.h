// LUT GEMM for M > 1 on the gfx950 matrix cores:  C[M, N] = A[M, K] @ W^T,
// W[n, k] = LUT[n / gs][idx[n, k]], fp32 accumulate, one rounding.
//
// The weights never exist as a dense tile anywhere.  A lane loads one 16*b-byte
// chunk of the idxN blob, which holds 8 rows x 16 k of one 128 x 64 tile, turns
// the codes into 16-bit LUT values through a pair table in LDS (one lookup = two
// weights) and feeds the result straight into v_mfma_f32_16x16x32 as the
// row-side operand.  The blob's chunk order is the operand order of that
// instruction up to a lane permutation:
//
//   MFMA lane l:  rho = l & 15 (operand row), kg = l >> 4 (k group of 8 values)
//   chunk         th  = (rho >> 3) * 32 + (rho & 7) * 4 + kg     (wx, lane>>2, lane&3)
//   operand (v, d, j), j = half of the 64-k tile:
//       row  n = t*128 + wx*64 + v*16 + d*8 + (rho & 7)
//       slot s = ktl*4 + s2*2 + e  ->  k = g*64 + (2j + ktl)*16 + 2*kg + 8*s2 + e
//
// so one chunk yields the 16 operands (v, d, j) of its 16 rows, and the
// activations only have to present the same k order: a pre-pass writes them as
// Ap[g][j][m / 16][lane = kg*16 + m % 16][8 values], one 16-byte load per operand.
// The product is formed as C^T (rows of W on the MFMA row side), so a lane ends
// up with four consecutive n of one m.
//
// Workgroup = KW x MW wavefronts on one 128-row tile: wavefront (kw, mw) walks the
// k-tiles kw, kw + KW, ... for MB blocks of 16 rows of A.  Partial sums meet in a
// tree through LDS, then (gridDim.z > 1) across workgroups through fp32 partials
// and a ticket; the last arrival folds them in a fixed order.
#pragma once


#include "gemm_common.h"

namespace flute {

#ifdef FLUTE_STAMPS
// Instrumented builds only: per-wavefront phase times (s_memrealtime, 10 ns units) and the shader
// clock count across the K loop, written to the buffer flute_debug_stamps() was given.
static __device__ long long *g_gemm_stamps = nullptr;
#define FLUTE_STAMP(slot)                                                                       \
    do {                                                                                        \
        if (g_gemm_stamps && (threadIdx.x & 63) == 0)                                           \
            g_gemm_stamps[(((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * \
                              (blockDim.x / 64) * 8 + (threadIdx.x >> 6) * 8 + (slot)] =        \
                (slot) == 7 ? (long long)__builtin_readcyclecounter()                           \
                            : (long long)__builtin_amdgcn_s_memrealtime();                      \
    } while (0)
#else
#define FLUTE_STAMP(slot) do { } while (0)
#endif
constexpr int kGemmMaxSegs = 4;

// LDS of gemm_kernel behind its loop: the totals of `rows` rows as fp32 rows of 132, a ticket flag, and (a
// residual) as many rows again, which overlap the areas of the k ways' hand-overs.
constexpr int gemm_residual_offset(int rows) { return rows * 132 * 4 + 16; }

// One weight of a launch.
struct GemmSeg {
    const uint8_t *q[2];
    const uint16_t *lut[2];
    void *C;
    const float *xb;       // [M, R] fp32 residual coefficients (A @ resB^T) or NULL
    const uint16_t *resA;  // [N, R] activation dtype
    const uint16_t *resB;  // few rows that form xb themselves (R <= 16): [R, K] activation dtype; else NULL
    const uint16_t *bias;  // [N] activation dtype
    int64_t ldc;
    int gs, lut_rows, R;
    int vec_res;           // R % 4 == 0 and rows of resA and xb allow loads of four ranks
    int vec_store;         // C rows allow 16-byte stores
};

// Up to four weights of one width pair and group size over the same rows: gridDim.x counts the
// 128-row tiles of all of them.
struct GemmParams {
    int tile0[kGemmMaxSegs];   // first tile of each weight; past the last one INT_MAX
    GemmSeg seg[kGemmMaxSegs];
    const u4_t *Ap;        // permuted activations, LUT dtype, rows padded to 16
    float *P;              // split-K partial images
    int *tickets;
    int bits[2];
    int tab_off[2];        // byte offset of each stream's pair tables in LDS
    int rep_log2[2];       // log2 of the table replication (lanes per entry)
    int stage_off;         // byte offset of the per-wavefront tile staging buffers (4 KB, lean loop: 8 KB)
    int lean;              // 1: the launch uses the lean loop's instantiation
    int prog_off;          // lean loop: byte offset of one progress word per wavefront
    int balance;           // lean loop: 1 = the wavefront of a SIMD that is behind gets the higher priority
    int scatter;           // four blocks per wavefront: the mode of image_block_xor the image was written with;
                           // not 0: the k ways hand blocks to each other instead of reducing through the tree
    int nstreams;
    int M, G;
    int mblk_total;        // ceil(M / 16)
    int mblk_pad;          // blocks Ap holds per half tile: gridDim.y * MW * MB
    int ksplit, gper;      // gridDim.z and k-tiles per z slice
    int z_base, ztotal;    // partial tiles: this launch writes [z_base, z_base + gridDim.z) of
                           // ztotal (several launches, one per stream, may share a fold)
    int out_bf16;          // dtype of C, resA, bias
    const u4_t *A8;        // few rows: A itself, rows of lda8 16-byte pieces, no pre-pass (or NULL)
    int64_t lda8;
    int a_bf16;            // dtype of A there
    int find;              // A8 of one type and a LUT of the other: workgroups look for their rows' scales themselves
    const int *rowshift;   // [M] or NULL: row m of the operands holds A[m] * 2^-rowshift[m]
};

// Strides of A (elements) at which the offsets of a few-row workgroup's lanes within its rows fit 32 bits.
constexpr int64_t few_lda() { return (int64_t)1 << 25; }

// Activation pre-pass of rows that are not 16-byte aligned (others: gemm_pre_kernel):
// Ap[g][j][mb][lane][slot] in the LUT's 16-bit type.
// block_xor: the mode of image_block_xor (common.h).
static __global__ void __launch_bounds__(256) gemm_prep_kernel(const uint16_t *A, u4_t *Ap, int M,
                                                        int64_t lda, int G, int mblk,
                                                        int in_bf16, int out_bf16, int pairs,
                                                        const int *rowshift, int block_xor) {
    const int64_t total = (int64_t)G * 2 * mblk * 64;
    for (int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; o < total;
         o += (int64_t)gridDim.x * blockDim.x) {
        const int lane = (int)(o & 63);
        const int64_t rest = o >> 6;
        const int gj = (int)(rest / mblk);
        const int g = gj >> 1, j = gj & 1;
        const int mb = (int)(rest % mblk) ^ image_block_xor(g, block_xor);
        const int m = mb * 16 + (lane & 15), kg = lane >> 4;
        uint32_t out[4] = {0u, 0u, 0u, 0u};
        if (m < M) {
            const int shift = rowshift ? rowshift[m] : 0;
#pragma unroll
            for (int s = 0; s < 4; ++s) {              // s = ktl*2 + s2
                const int k = g * 64 + (2 * j + (s >> 1)) * 16 + 2 * kg + 8 * (s & 1);
                // k is even: one 32-bit load per pair where the rows are 4-byte aligned
                uint16_t a0, a1;
                if (pairs) {
                    const uint32_t pair = *(const uint32_t *)(A + m * lda + k);
                    a0 = (uint16_t)(pair & 0xffffu);
                    a1 = (uint16_t)(pair >> 16);
                } else {
                    a0 = A[m * lda + k];
                    a1 = A[m * lda + k + 1];
                }
                if (in_bf16 != out_bf16) {
                    a0 = round_act(ldexpf(in_bf16 ? bf2f(a0) : h2f(a0), -shift), out_bf16);
                    a1 = round_act(ldexpf(in_bf16 ? bf2f(a1) : h2f(a1), -shift), out_bf16);
                }
                out[s] = (uint32_t)a0 | ((uint32_t)a1 << 16);
            }
        }
        u4_t v = {out[0], out[1], out[2], out[3]};
        Ap[o] = v;
    }
}

// Lane J of this lane's quad.
template <int J>
__device__ __forceinline__ uint32_t quad_bcast(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, J * 0x55, 0xf, 0xf, true);
}
// The activation image of the many-row kernel (wide_piece) from rows that are not 16-byte aligned (others:
// gemm_pre_kernel): a wavefront moves one 1 KB block, sixteen rows by 64 bytes.
static __global__ void __launch_bounds__(256) gemm_image_kernel(const uint16_t *A, u4_t *Ap, int M, int64_t lda, int segs,
                                                         int mblk, int in_bf16, int out_bf16,
                                                         const int *rowshift) {
    const int lane = threadIdx.x & 63;
    const int64_t blocks = (int64_t)segs * ((M + 15) >> 4);          // (16-row block, 32-k segment)
    for (int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); b < blocks; b += (int64_t)gridDim.x * 4) {
        int mb, seg;
        if (blocks <= 0x7fffffff) {                      // uniform; a 64-bit division costs some hundred instructions
            mb = (int)((uint32_t)b / (uint32_t)segs);
            seg = (int)((uint32_t)b - (uint32_t)mb * (uint32_t)segs);
        } else {
            mb = (int)(b / segs);
            seg = (int)(b - (int64_t)mb * segs);
        }
        const int m = min(mb * 16 + (lane >> 2), M - 1); // rows past the end repeat the last: nobody stores their products
        const uint16_t *src = A + (int64_t)m * lda + seg * 32 + (lane & 3) * 8;
        u4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (uint32_t)src[2 * e] | ((uint32_t)src[2 * e + 1] << 16);
        if (in_bf16 != out_bf16) {
            const int shift = rowshift ? rowshift[m] : 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint16_t lo = (uint16_t)(v[e] & 0xffffu), hi = (uint16_t)(v[e] >> 16);
                const float flo = ldexpf(in_bf16 ? bf2f(lo) : h2f(lo), -shift);
                const float fhi = ldexpf(in_bf16 ? bf2f(hi) : h2f(hi), -shift);
                v[e] = (uint32_t)round_act(flo, out_bf16) | ((uint32_t)round_act(fhi, out_bf16) << 16);
            }
        }
        Ap[((int64_t)seg * mblk + mb) * 64 + (lane & 3) * 16 + (lane >> 2)] = v;
    }
}

// bfloat16 rows in front of float16 operands: shift[m] = the power of two that brings the
// largest magnitude of row m to [1, 2) (bf16_row_shift), one workgroup per row.
static __global__ void __launch_bounds__(256) gemm_rowshift_kernel(const uint16_t *A, int64_t lda, int K,
                                                            int *shift) {
    __shared__ uint32_t slots[4];
    const uint16_t *row = A + (int64_t)blockIdx.x * lda;
    uint32_t e = 0;
    if ((((uintptr_t)row) & 15) == 0) {                // uniform per row
        for (int k = threadIdx.x * 8; k < K; k += 256 * 8) {
            if (k + 8 <= K) e = max(e, bf16_max_exp8(*(const uint4 *)(row + k)));
            else for (int q = k; q < K; ++q) e = max(e, (uint32_t)(row[q] >> 7) & 0xffu);
        }
    } else {
        for (int k = threadIdx.x; k < K; k += 256) e = max(e, (uint32_t)(row[k] >> 7) & 0xffu);
    }
    e = workgroup_max(e, slots, threadIdx.x, 256);
    if (threadIdx.x == 0) shift[blockIdx.x] = bf16_row_shift(e);
}

// xb[m, r] = sum_k A[m, k] * resB[r, k] in fp32: sixteen rows by sixteen ranks per workgroup on the
// matrix cores, sixteen wavefronts taking the 32-k pieces of K in turn, their sums added in wavefront
// order.  K is what there is to spread: a call of few rows has few such blocks, and a wavefront's
// loads (sixteen rows each) are a chain of trips to memory; `slices` slices of K leave their sums in
// `part`, and the last arrival of a block adds them in slice order.  M = 48, K = 12288, R = 16: 22.8
// us in one slice, 6.3 in sixteen.
struct CoeffParams {
    const uint16_t *A;
    const uint16_t *up;        // (SILU) as ImageParams
    const uint16_t *resB[kGemmMaxSegs];
    float *xb[kGemmMaxSegs];
    int R[kGemmMaxSegs];
    int rank0[kGemmMaxSegs];   // first block of ranks of each weight; past the last one INT_MAX
    int64_t lda;
    int M, K, aligned, kper;
    int rows, ranks, slices;   // blocks
    float *part;
    int *tickets;
};
template <bool BF16, bool SILU>
__device__ __forceinline__ void coeff_block(const CoeffParams &p, int index, f4_t (&red)[16][64]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int bz = index / (p.rows * p.ranks), in_slice = index - bz * (p.rows * p.ranks);
    const int by = in_slice / p.rows, bx = in_slice - by * p.rows;
    const int si = (by >= p.rank0[1]) + (by >= p.rank0[2]) + (by >= p.rank0[3]);
    const int M = p.M, K = p.K, R = p.R[si], rb = by - p.rank0[si], aligned = p.aligned;
    float *const xb = p.xb[si];
    f4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const int k0 = bz * p.kper + wave * 32, k1 = min(bz * p.kper + p.kper, K);
    // Rows that allow it are loaded as four lanes to the 64 bytes of a row: a lane per row and piece, the order
    // of the matrix operands, is 64 accesses of the address path an instruction and not 16, and that path
    // bounds these workgroups; the lanes are put in order behind the load (ds_bpermute).  The pre-pass of
    // M = 98, K = 1536, three weights of rank 16 4.5 us, before 7.2; M = 86, K = 1792 4.7, before 6.0; M = 48, K = 12288 6.4, before 6.8.
    if (aligned) {                                      // uniform
        const int m = min(bx * 16 + (lane >> 2), M - 1), rr = min(rb * 16 + (lane >> 2), R - 1);
        const uint16_t *a = p.A + (int64_t)m * p.lda + (lane & 3) * 8, *b = p.resB[si] + (int64_t)rr * K + (lane & 3) * 8;
        const uint16_t *up = SILU ? p.up + (int64_t)m * p.lda + (lane & 3) * 8 : nullptr;
        const int from = ((lane & 15) * 4 + (lane >> 4)) << 2;
        auto ordered = [&](u4_t v) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)v[e]);
            return v;
        };
        constexpr int U = 4;                            // steps whose loads go out together
        for (int k = k0; k < k1; k += 512 * U) {
            u4_t va[U], vb[U], vu[SILU ? U : 1];
#pragma unroll
            for (int i = 0; i < U; ++i) {
                if (k + 512 * i >= k1) break;           // uniform
                va[i] = *(const u4_t *)(a + k + 512 * i);
                vb[i] = *(const u4_t *)(b + k + 512 * i);
                if constexpr (SILU) vu[i] = *(const u4_t *)(up + k + 512 * i);
            }
#pragma unroll
            for (int i = 0; i < U; ++i) {
                if (k + 512 * i >= k1) break;
                if constexpr (SILU) va[i] = silu_mul8<BF16>(va[i], vu[i]);
                acc = mfma16<BF16>(ordered(vb[i]), ordered(va[i]), acc);
            }
        }
    } else {
        const int m = min(bx * 16 + (lane & 15), M - 1), rr = min(rb * 16 + (lane & 15), R - 1);
        const uint16_t *a = p.A + (int64_t)m * p.lda + (lane >> 4) * 8, *b = p.resB[si] + (int64_t)rr * K + (lane >> 4) * 8;
        auto load8 = [&](const uint16_t *p) {
            u4_t v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (uint32_t)p[2 * e] | ((uint32_t)p[2 * e + 1] << 16);
            return v;
        };
        for (int k = k0; k < k1; k += 512) acc = mfma16<BF16>(load8(b + k), load8(a + k), acc);
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave == 0) {
        for (int w = 1; w < 16; ++w) acc += red[w][lane];
        if (p.slices > 1) {
            const int block = in_slice, Z = p.slices;
            const int64_t step = (int64_t)p.rows * p.ranks * 256;            // floats of one slice
            float *const mine = p.part + (int64_t)block * 256 + lane * 4;
            ws_store16(mine + bz * step, acc);
            ws_stores_done();
            int old = 0;
            if (lane == 0) old = __hip_atomic_fetch_add(p.tickets + block, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__builtin_amdgcn_readfirstlane(old) != Z - 1) return;
            if (lane == 0) __hip_atomic_store(p.tickets + block, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            acc = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
            for (int z = 0; z < Z; z += 4) {                                 // (slices come in fours)
                f4_t v[4];
                const float *s = mine + z * step;
                ws_load16x4(s, s + step, s + 2 * step, s + 3 * step, v[0], v[1], v[2], v[3]);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc += v[i];
            }
        }
        const int mo = bx * 16 + (lane & 15), r0 = rb * 16 + (lane >> 4) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (mo < M && r0 + e < R) xb[(int64_t)mo * R + r0 + e] = acc[e];
    }
}

// What a launch over rows of A (16-byte aligned) has to have in front of it, in one launch: the operand
// image, the power-of-two scale of every row (bfloat16 rows in front of float16 operands), the residual
// coefficients.  The first workgroups take the coefficients, the longest chain of the three; the others
// a share of the image each.  As launches of their own: M = 48, K = 12288, rank 16 image 4.2 and
// coefficients 6.9 us one after the other; M = 509, K = 12288, bfloat16 rows, scales 3.1 and image 6.8.
struct ImageParams {
    const uint16_t *A;
    const uint16_t *up;        // (SILU) an element of the rows is silu(A's) * this one, rounded; rows as A's
    u4_t *Ap;                  // or NULL: only the scales are wanted
    int64_t lda;
    int *rowshift;             // [M] or NULL; find: written here, else read
    const uint32_t *warm;      // LUT rows the launch behind reads first: one touch per 64-byte line
    int M, segs;               // rows, 32-k segments of a row
    int blocks;                // 16-row blocks to write
    int mblk;                  // 16-row blocks the image holds per segment
    int in_bf16, out_bf16;
    int wide;                  // 1: pieces as they are (wide_piece), rows past the end repeat the last; 0: operands of
                               // gemm_kernel.h, rows past the end zero
    int block_xor;             // wide == 0: mode of image_block_xor
    int find;                  // look for the scales first: the rows (2 or 4) that a workgroup then takes whole, or 0
    int warm_lines;
};

constexpr int kPieceMax = 8;   // 16-byte pieces of a row quarter that a thread holds where it looks for scales
constexpr int find_reach() { return kPieceMax * 64 * 32; }       // columns, four rows a workgroup

__device__ __forceinline__ u4_t image_convert(u4_t raw, int in_bf16, int out_bf16, int shift) {
    if (in_bf16 != out_bf16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint16_t lo = (uint16_t)(raw[e] & 0xffffu), hi = (uint16_t)(raw[e] >> 16);
            const float flo = ldexpf(in_bf16 ? bf2f(lo) : h2f(lo), -shift);
            const float fhi = ldexpf(in_bf16 ? bf2f(hi) : h2f(hi), -shift);
            raw[e] = (uint32_t)round_act(flo, out_bf16) | ((uint32_t)round_act(fhi, out_bf16) << 16);
        }
    }
    return raw;
}

// Piece q (lane & 3) of 32-k segment `seg` of row m into the image; the four lanes of a quad hold the
// pieces of one row's segment.
__device__ __forceinline__ void image_store(const ImageParams &p, int m, int seg, u4_t raw) {
    const int q = threadIdx.x & 3;
    u4_t out = raw;
    int mb = m >> 4;
    if (!p.wide) {                                      // uniform
        // piece j of a segment holds its dwords 4j .. 4j + 3; operand kg is the dwords
        // {kg, kg + 4, kg + 8, kg + 12} = element kg of the pieces 0 .. 3
#define FLUTE_TAKE(J)                                                                          \
        {                                                                                      \
            const uint32_t b0 = quad_bcast<J>(raw[0]), b1 = quad_bcast<J>(raw[1]);             \
            const uint32_t b2 = quad_bcast<J>(raw[2]), b3 = quad_bcast<J>(raw[3]);             \
            out[J] = (q & 2) ? ((q & 1) ? b3 : b2) : ((q & 1) ? b1 : b0);                      \
        }
        FLUTE_TAKE(0) FLUTE_TAKE(1) FLUTE_TAKE(2) FLUTE_TAKE(3)
#undef FLUTE_TAKE
        mb ^= image_block_xor(seg >> 1, p.block_xor);
    }
    p.Ap[((int64_t)seg * p.mblk + mb) * 64 + q * 16 + (m & 15)] = out;
}

// ROWS rows by all segments: a quad per segment and row, 256 / ROWS quads of a row side by side.
template <bool BF16, bool SILU, int ROWS>
__device__ __forceinline__ void find_rows(const ImageParams &p, int b, int nb, uint32_t *slots) {
    constexpr int STEP = 256 / ROWS, PIECES = kPieceMax * ROWS / 4;
    const int tid = threadIdx.x, lane = tid & 63, r = (tid >> 2) & (ROWS - 1), s0 = tid / (4 * ROWS);
    for (int m0 = b * ROWS; m0 < p.blocks * 16; m0 += nb * ROWS) {
        const int m = m0 + r;
        const int64_t at = (int64_t)min(m, p.M - 1) * p.lda + (lane & 3) * 8;
        u4_t raw[PIECES];
        uint32_t e = 0;
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
            if (s0 + i * STEP < p.segs) raw[i] = *(const u4_t *)(p.A + at + (s0 + i * STEP) * 32);
        if constexpr (SILU) {
            u4_t up[PIECES];
#pragma unroll
            for (int i = 0; i < PIECES; ++i)
                if (s0 + i * STEP < p.segs) up[i] = *(const u4_t *)(p.up + at + (s0 + i * STEP) * 32);
#pragma unroll
            for (int i = 0; i < PIECES; ++i)
                if (s0 + i * STEP < p.segs) raw[i] = silu_mul8<BF16>(raw[i], up[i]);
        }
        if (m >= p.M && !p.wide) {
#pragma unroll
            for (int i = 0; i < PIECES; ++i) raw[i] = u4_t{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
            if (s0 + i * STEP < p.segs) e = max(e, bf16_max_exp8(make_uint4(raw[i][0], raw[i][1], raw[i][2], raw[i][3])));
        e = dpp_max<0xB1>(e);                           // the quad
        e = dpp_max<0x4E>(e);
        if constexpr (ROWS == 2) e = max(e, (uint32_t)__shfl_xor((int)e, 8));
        e = max(e, (uint32_t)__shfl_xor((int)e, 16));
        e = max(e, (uint32_t)__shfl_xor((int)e, 32));
        __syncthreads();                                // (the rows before are done with the slots)
        if ((lane & 3) == 0 && lane < 4 * ROWS) slots[(tid >> 6) * 4 + r] = e;      // [wave][row]
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 16; ++w) e = max(e, slots[w * 4 + r]);
        const int shift = bf16_row_shift(e);
        if (tid < 4 * ROWS && (tid & 3) == 0 && m < p.M) p.rowshift[m] = shift;
        if (p.Ap) {
#pragma unroll
            for (int i = 0; i < PIECES; ++i)
                if (s0 + i * STEP < p.segs) image_store(p, m, s0 + i * STEP, image_convert(raw[i], p.in_bf16, p.out_bf16, shift));
        }
    }
}

template <bool BF16, bool SILU>
__global__ void __launch_bounds__(1024) gemm_pre_kernel(const CoeffParams c, const ImageParams p) {
    __shared__ f4_t red[16][64];
    const int ncoeff = c.rows * c.ranks * c.slices;
    if ((int)blockIdx.x < ncoeff) {
        coeff_block<BF16, SILU>(c, blockIdx.x, red);
        return;
    }
    const int b = blockIdx.x - ncoeff, nb = gridDim.x - ncoeff, tid = threadIdx.x, lane = tid & 63;
    {
        const int line = b * (int)blockDim.x + tid;
        if (line < p.warm_lines) {
            const uint32_t seen = __builtin_nontemporal_load(p.warm + (size_t)line * 16);
            asm volatile("" ::"v"(seen));
        }
    }
    // a row past the end: the last one again (wide) or zeros
    auto offset = [&](int m, int seg) { return (int64_t)min(m, p.M - 1) * p.lda + seg * 32 + (lane & 3) * 8; };
    if (p.find) {
        if (p.find == 2) find_rows<BF16, SILU, 2>(p, b, nb, (uint32_t *)red);
        else find_rows<BF16, SILU, 4>(p, b, nb, (uint32_t *)red);
        return;
    }
    // a wavefront moves one 1 KB block of the image, sixteen rows by 64 bytes, at a time
    const int waves = blockDim.x >> 6;
    const int64_t total = (int64_t)p.blocks * p.segs;
    for (int64_t w = (int64_t)b * waves + (tid >> 6); w < total; w += (int64_t)nb * waves) {
        int mb, seg;
        if (total <= 0x7fffffff) {                      // uniform; a 64-bit division costs some hundred instructions
            mb = (int)((uint32_t)w / (uint32_t)p.segs);
            seg = (int)((uint32_t)w - (uint32_t)mb * (uint32_t)p.segs);
        } else {
            mb = (int)(w / p.segs);
            seg = (int)(w - (int64_t)mb * p.segs);
        }
        const int m = mb * 16 + (lane >> 2);
        u4_t raw = {0u, 0u, 0u, 0u};
        if (m < p.M || p.wide) {
            raw = *(const u4_t *)(p.A + offset(m, seg));
            if constexpr (SILU) raw = silu_mul8<BF16>(raw, *(const u4_t *)(p.up + offset(m, seg)));
        }
        const int shift = p.rowshift ? p.rowshift[min(m, p.M - 1)] : 0;
        image_store(p, m, seg, image_convert(raw, p.in_bf16, p.out_bf16, shift));
    }
}

// The 2B-bit code of pair p of a chunk held as 4*B dwords (all indices constant
// after unrolling).
template <int B>
__device__ __forceinline__ uint32_t pair_code(const uint32_t (&Q)[4 * B], int p) {
    const int bit = 2 * B * p, dw = bit >> 5, sh = bit & 31;
    if (sh + 2 * B <= 32) return __builtin_amdgcn_ubfe(Q[dw], sh, 2 * B);
    return __builtin_amdgcn_alignbit(Q[dw + 1 < 4 * B ? dw + 1 : dw], Q[dw], sh) &
           ((1u << (2 * B)) - 1u);
}

template <int B>
__device__ __forceinline__ void load_chunk(uint32_t (&Q)[4 * B], const uint8_t *chunk) {
    const u4_t *src = (const u4_t *)chunk;
#pragma unroll
    for (int i = 0; i < B; ++i) {
        const u4_t v = __builtin_nontemporal_load(src + i);
        Q[4 * i + 0] = v[0];
        Q[4 * i + 1] = v[1];
        Q[4 * i + 2] = v[2];
        Q[4 * i + 3] = v[3];
    }
}

// The four lookups of operand (j, v, d).  PERM (4-bit codes, 64-lane replication,
// table on a 64 KB boundary of LDS): the code is a whole byte of the chunk and the
// entry stride is 256 bytes, so one v_perm_b32 drops it into byte 1 of the lane's
// column address.
template <int B, bool PERM>
__device__ __forceinline__ u4_t fetch_operand(const uint32_t (&Q)[4 * B], int j, int v, int d,
                                              uint32_t lbase, int code_shift) {
    typedef const __attribute__((address_space(3))) uint32_t *LdsWord;
    u4_t w;
#pragma unroll
    for (int s = 0; s < 4; ++s) {                      // s = ktl*2 + s2
        const int p = (2 * j + (s >> 1)) * 16 + v * 4 + d * 2 + (s & 1);
        uint32_t addr;
        if constexpr (PERM) {
            static_assert(B == 4, "byte codes");
            addr = __builtin_amdgcn_perm(Q[p >> 2], lbase, 0x03020000u | ((4u + (p & 3)) << 8));
        } else {
            addr = (pair_code<B>(Q, p) << code_shift) + lbase;
        }
        w[s] = *(LdsWord)addr;
    }
    return w;
}

// Half (32 k) of a 64-k tile of one stream: 8 operands x MB MFMAs.  The lookups
// run one pair of operands ahead of the MFMAs that consume them, in two
// alternating register sets, so the LDS latency hides behind matrix work.
//   lbase[v] : LDS byte address of this lane's column of the table that serves
//              rows (wx, v) (the LUT group may depend on wx and v when gs < 128)
template <int B, int MB, bool BF16, bool PERM = false>
__device__ __forceinline__ void half_mma(const uint32_t (&Q)[4 * B], int j, const u4_t (&Aj)[MB],
                                         f4_t (&acc)[MB][8], const uint32_t (&lbase)[4],
                                         int code_shift) {
    constexpr int AHEAD = 2;                             // pairs of operands in flight
    u4_t W[AHEAD + 1][2];
#pragma unroll
    for (int v = 0; v < AHEAD; ++v) {
        W[v][0] = fetch_operand<B, PERM>(Q, j, v, 0, lbase[v], code_shift);
        W[v][1] = fetch_operand<B, PERM>(Q, j, v, 1, lbase[v], code_shift);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        if (v + AHEAD < 4) {
            W[(v + AHEAD) % (AHEAD + 1)][0] =
                fetch_operand<B, PERM>(Q, j, v + AHEAD, 0, lbase[v + AHEAD], code_shift);
            W[(v + AHEAD) % (AHEAD + 1)][1] =
                fetch_operand<B, PERM>(Q, j, v + AHEAD, 1, lbase[v + AHEAD], code_shift);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                acc[mb][v * 2 + d] =
                    mfma16<BF16>(W[v % (AHEAD + 1)][d], Aj[mb], acc[mb][v * 2 + d]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Block mb of an activation half: 16 bytes per lane at src + mb KB, as a statement the compiler
// does not take for a load (no wait of its own follows).
__device__ __forceinline__ void lean_load16(u4_t &dst, const u4_t *src, int mb) {
    switch (mb) {                                       // the offset is an immediate
        case 0: asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(dst) : "v"(src) : "memory"); break;
        case 1: asm volatile("global_load_dwordx4 %0, %1, off offset:1024" : "=&v"(dst) : "v"(src) : "memory"); break;
        case 2: asm volatile("global_load_dwordx4 %0, %1, off offset:2048" : "=&v"(dst) : "v"(src) : "memory"); break;
        default: asm volatile("global_load_dwordx4 %0, %1, off offset:3072" : "=&v"(dst) : "v"(src) : "memory"); break;
    }
}

// One stream of B1-bit codes, four blocks of rows per wavefront (fewer rows: gemm_few_kernel.h).
// LEAN (one 4-bit stream, one LUT group per tile): every vector memory
// instruction of the kernel is written out and so is every wait for one.  The tile goes straight
// into LDS (global_load_lds_dwordx4), which frees the sixteen registers a tile in flight would
// hold; the compiler cannot count such loads next to its own (it answers one in flight with
// vmcnt(0) in front of the next use of any loaded register), hence all or nothing.
template <int MB, int KW, int MW, bool BF16, int B1, bool PERM = false, bool LEAN = false, bool SEGS = false>
__global__ void __launch_bounds__(64 * KW * MW) gemm_kernel(const GemmParams p) {
    static_assert(MB == 4 && KW * MW == 8, "64 or 128 rows");
    static_assert(!LEAN || (PERM && B1 == 4), "lean loop: fast path, operand image");
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int NT = 64 * KW * MW;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kw = wave % KW, mw = wave / KW;
    // (instantiations of their own for several weights: the tile numbers have to be read before the
    // weight's arguments can be, and M = 256, 4096 -> 12288 went from 36.6 to 37.6 us with it)
    int si = 0;
    if constexpr (SEGS)
        si = ((int)blockIdx.x >= p.tile0[1]) + ((int)blockIdx.x >= p.tile0[2]) + ((int)blockIdx.x >= p.tile0[3]);
    const GemmSeg &w = p.seg[SEGS ? si : 0];
    const int t = SEGS ? blockIdx.x - p.tile0[si] : blockIdx.x;
    FLUTE_STAMP(0);
    const int mb0 = (blockIdx.y * MW + mw) * MB;       // first 16-row block of this wavefront
    const int z = blockIdx.z;
    const int rho = lane & 15, kg = lane >> 4;
    const int wx = rho >> 3;
    const int th = wx * 32 + (rho & 7) * 4 + kg;

    const int gbeg = z * p.gper, gend = min(p.G, gbeg + p.gper);
    const bool active = mb0 < p.mblk_total;            // whole wavefront
    const int g0 = gbeg + kw;
    int left = (active && g0 < gend) ? (gend - g0 + KW - 1) / KW : 0;   // tiles of this wavefront
    const int64_t jstep = (int64_t)p.mblk_pad * 64;    // u4 units between the halves of a tile
    // Ap is padded to whole workgroups of blocks (zeros), so every block index below
    // gridDim.y * MW * MB is loadable.
    // A wavefront without tiles addresses the first tile of the K range instead: its
    // loads below are then unconditional like everyone's, and the compiler can count them.
    const int g_first = left > 0 ? g0 : gbeg;
    const u4_t *ap = p.Ap + ((int64_t)g_first * 2 * p.mblk_pad + mb0) * 64 + lane;
    auto load_a = [&](u4_t (&Aj)[MB], const u4_t *src) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) Aj[mb] = src[mb * 64];
    };
    // fast path: first tile and first activation operands are requested before the
    // tables are built, so their latency hides behind the build
    u4_t R[4], A0[MB], A1[MB];
    const uint8_t *tp = w.q[0] + ((int64_t)t * p.G + g_first) * 4096 + lane * 16;
    auto load_tile = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) R[i] = __builtin_nontemporal_load((const u4_t *)(tp + i * 1024));
    };
    const int ngrp = w.gs >= 128 ? 1 : 128 / w.gs;
    uint32_t lutv[2] = {0u, 0u};                       // fast path: LUT row(s), one value per lane
    if constexpr (PERM) {
#pragma unroll
        for (int gl = 0; gl < 2; ++gl) {
            if (LEAN || gl >= ngrp) break;
            int row = w.gs >= 128 ? (t * 128) / w.gs : t * ngrp + gl;
            row = min(row, w.lut_rows - 1);
            lutv[gl] = w.lut[0][((size_t)row << 4) + (lane & 15)];
        }
        // Unconditional, after the LUT row: the table build below then waits for the LUT
        // values only, not for the first tile (a conditional load here made that wait a
        // wait for everything).
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!LEAN) {
            load_tile();
            load_a(A0, ap);
            load_a(A1, ap + jstep);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // ---- lean loop: hand-written loads ------------------------------------------------
    // LDS staging: two 4 KB buffers per wavefront; tile n lives in buffer n & 1.  Lane L of row i
    // asks for the 16-byte piece that belongs at position L of that row (the same layout the
    // register path writes: slot order and rotation of the quarters).
    const uint32_t lds_base0 =
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    const uint32_t lean_stage =
        __builtin_amdgcn_readfirstlane(lds_base0 + p.stage_off + (uint32_t)wave * 8192u);
    const int lean_kt = ((lane & 3) - (lane >> 4)) & 3;
    const uint32_t lean_even = (uint32_t)((lane >> 2) * 64 + lean_kt * 16);
    const uint32_t lean_odd = (uint32_t)(((lane >> 2) ^ 1) * 64 + lean_kt * 16);
    const uint8_t *lean_tq = w.q[0] + ((int64_t)t * p.G + g_first) * 4096;   // wavefront-uniform
    auto lean_tile = [&](int buf) {                    // four loads, straight into LDS
        const uint32_t m0v = lean_stage + (uint32_t)buf * 4096u;
        // (the pointer is the same in every lane; the compiler cannot see that through the
        // wavefront-dependent tile count)
        const uint64_t a64 = (uint64_t)(uintptr_t)lean_tq;
        const uint8_t *tq_s = (const uint8_t *)(uintptr_t)join_address_halves(
            __builtin_amdgcn_readfirstlane((int)(uint32_t)a64),
            __builtin_amdgcn_readfirstlane((int)(uint32_t)(a64 >> 32)));
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %1, %3 offset:0 nt\n\t"
                     "global_load_lds_dwordx4 %2, %3 offset:1024 nt\n\t"
                     "global_load_lds_dwordx4 %1, %3 offset:2048 nt\n\t"
                     "global_load_lds_dwordx4 %2, %3 offset:3072 nt"
                     :: "s"(m0v), "v"(lean_even), "v"(lean_odd), "s"(tq_s) : "memory", "m0");
    };
    if constexpr (LEAN) {
        int row = (t * 128) / w.gs;
        row = min(row, w.lut_rows - 1);
        const uint16_t *lp = w.lut[0] + ((size_t)row << 4) + (lane & 15);
        uint32_t lv;
        asm volatile("global_load_ushort %0, %1, off" : "=&v"(lv) : "v"(lp) : "memory");
        lean_tile(0);                                  // tile 0
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) lean_load16(A0[mb], ap, mb);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) lean_load16(A1[mb], ap + jstep, mb);
        // the LUT value is the oldest load: 4 + 2 MB younger ones may stay in flight
        asm volatile("s_waitcnt vmcnt(%1)" : "+v"(lv) : "n"(4 + 2 * MB) : "memory");
        lutv[0] = lv;
    }

    // ---- pair tables ------------------------------------------------------------
    if constexpr (PERM) {
        // 64 replicas per entry: a wavefront writes one entry per instruction, every
        // lane the same dword, built from two lane reads of the LUT row it holds.
        const int wave_u = __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
        for (int gl = 0; gl < 2; ++gl) {
            if (gl >= ngrp) break;
            const uint32_t lv = lutv[gl];
            uint32_t *tab = (uint32_t *)(smem + p.tab_off[0]) + (gl << 14);
            for (int code = wave_u; code < 256; code += NT / 64) {
                const uint32_t lo = __builtin_amdgcn_readlane(lv, code & 15);
                const uint32_t hi = __builtin_amdgcn_readlane(lv, code >> 4);
                tab[code * 64 + lane] = lo | (hi << 16);
            }
        }
    } else {
        const int rl = p.rep_log2[0];
        const int total = ngrp << (2 * B1 + rl);
        uint32_t *tab = (uint32_t *)(smem + p.tab_off[0]);
        for (int i = tid; i < total; i += NT) {
            const int code = (i >> rl) & ((1 << (2 * B1)) - 1);
            const int gl = i >> (rl + 2 * B1);
            int row = w.gs >= 128 ? (t * 128) / w.gs : t * ngrp + gl;
            row = min(row, w.lut_rows - 1);
            const uint16_t *lr = w.lut[0] + ((size_t)row << B1);
            tab[i] = (uint32_t)lr[code & ((1 << B1) - 1)] | ((uint32_t)lr[code >> B1] << 16);
        }
    }
    if constexpr (LEAN) {
        if (lane == 0)
            *(uint32_t *)(smem + p.prog_off + wave * 4) = (uint32_t)__builtin_amdgcn_readfirstlane(left);
    }
    __syncthreads();
    FLUTE_STAMP(1);
    FLUTE_STAMP(7);

    f4_t acc[MB][8];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[mb][i] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const uint32_t lds_base =
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    auto table_bases = [&](uint32_t (&lb)[4], int s, int b) {
        const int rl = p.rep_log2[s];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = wx * 64 + v * 16;
            const int gl = w.gs >= 128 ? 0 : row / w.gs;
            lb[v] = lds_base + p.tab_off[s] +
                    (((gl << (2 * b + rl)) + (lane & ((1 << rl) - 1))) << 2);
        }
    };

    if (active) {
        if constexpr (PERM) {
            // 4-bit fast path.  A 64-byte chunk per lane is the worst pattern for the
            // vector memory pipe (one 64-byte sector per lane and instruction), so the
            // 4 KB tile is fetched as four fully contiguous 1 KB rows instead, dropped
            // into a per-wavefront LDS buffer and read back chunk by chunk.  Slot
            // order and a rotation of the four quarters keep both sides free of bank
            // conflicts: piece (chunk c, quarter kt) lives at
            //     (c ^ ((c >> 4) & 1)) * 64 + ((kt + (c >> 2)) & 3) * 16.
            typedef __attribute__((address_space(3))) u4_t *LdsQuad;
            uint32_t lb[4];
            table_bases(lb, 0, 4);
            const uint32_t stage = lds_base + p.stage_off + wave * 4096;
            const int rotw = ((lane & 3) + ((lane >> 4) & 3)) & 3;
            const uint32_t wb_even = stage + (lane >> 2) * 64 + rotw * 16;
            const uint32_t wb_odd = stage + ((lane >> 2) ^ 1) * 64 + rotw * 16;
            const int slot = th ^ ((th >> 4) & 1);
            uint32_t rb[4];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) rb[kt] = stage + slot * 64 + ((kt + (rho & 3)) & 3) * 16;

            uint32_t Q[16];
            constexpr int64_t qstep = (int64_t)KW * 4096;
            const int64_t astep = (int64_t)KW * 2 * p.mblk_pad * 64;
            auto stage_write = [&]() {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    *(LdsQuad)(uintptr_t)(((i & 1) ? wb_odd : wb_even) + i * 1024) = R[i];
            };
            auto stage_read = [&]() {
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    const u4_t v = *(LdsQuad)(uintptr_t)rb[kt];
                    Q[4 * kt + 0] = v[0];
                    Q[4 * kt + 1] = v[1];
                    Q[4 * kt + 2] = v[2];
                    Q[4 * kt + 3] = v[3];
                }
            };
            if constexpr (LEAN) {
                // One round = one tile of this wavefront.  Vector memory instructions of a round,
                // in issue order: the tile after next (4, into the LDS buffer just read out), the
                // next tile's first-half operands (MB), its second-half operands (MB).  Inside a
                // half the weight operands are outermost: an operand serves all blocks of rows
                // and is replaced by the next half's right away, so lookups and products
                // alternate four by four (measured against blocks of rows outermost with the
                // lookups bunched behind the last two blocks: 1 % faster; the explicit waits of
                // either order cost no time, a wavefront's loads are there when it asks).
                // The products of an accumulator come in the same order as in the other loop.
                u4_t W[8];
                uint32_t Q8[8];
                const uint32_t lb0 = lb[0];
                const uint32_t rbase = lean_stage + slot * 64;
                const int rot = rho & 3;
                uint32_t cur = 0;                         // LDS buffer of this round's tile: 0 or 4096
                auto read_codes = [&](int j, uint32_t boff) {
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) {
                        const u4_t v = *(LdsQuad)(uintptr_t)(rbase + boff + (((2 * j + kk + rot) & 3) << 4));
                        Q8[4 * kk + 0] = v[0];
                        Q8[4 * kk + 1] = v[1];
                        Q8[4 * kk + 2] = v[2];
                        Q8[4 * kk + 3] = v[3];
                    }
                };
                auto operand = [&](int o) -> u4_t {
                    typedef const __attribute__((address_space(3))) uint32_t *LdsWord;
                    const int v = o >> 1, d = o & 1;
                    u4_t w;
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4)       // q4 = ktl * 2 + s2
                        w[q4] = *(LdsWord)__builtin_amdgcn_perm(
                            Q8[(q4 >> 1) * 4 + v], lb0, 0x03020000u | ((4u + d * 2 + (q4 & 1)) << 8));
                    return w;
                };
                // `between` runs after the first operand's products: work that has to follow LDS
                // reads issued in front of the half finds them complete there
                auto half = [&](u4_t (&Aj)[MB], const u4_t *next, auto &&between) {
#pragma unroll
                    for (int o = 0; o < 8; ++o) {
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb) acc[mb][o] = mfma16<BF16>(W[o], Aj[mb], acc[mb][o]);
                        if (o == 0) {
                            __builtin_amdgcn_sched_barrier(0);
                            between();
                        }
                        W[o] = operand(o);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) lean_load16(Aj[mb], next, mb);
                    __builtin_amdgcn_sched_barrier(0);
                };
                auto wait_half = [&](u4_t (&Aj)[MB], auto younger) {
                    asm volatile("s_waitcnt vmcnt(%4)" : "+v"(Aj[0]), "+v"(Aj[1]), "+v"(Aj[2]), "+v"(Aj[3])
                                 : "n"(decltype(younger)::value) : "memory");
                };
                // (the same in every lane: a scalar count gives a scalar loop)
                left = __builtin_amdgcn_readfirstlane(left);
                if (left > 0) {
                    // tile 0 is the oldest load in flight: both activation halves may stay
                    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * MB) : "memory");
                    read_codes(0, 0);
#pragma unroll
                    for (int o = 0; o < 8; ++o) W[o] = operand(o);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    if (left > 1) lean_tq += qstep;
                    lean_tile(1);                         // tile 1 (or a harmless reload)
                }
                const int wave_hi = __builtin_amdgcn_readfirstlane(wave >> 2);
                // Progress of the two wavefronts of a SIMD (w and w + 4): every round a wavefront
                // posts the tiles it has left and reads the other's figure of a round ago; the one
                // that is behind (or level) runs at the higher priority.  Against taking turns tile
                // by tile (FLUTE_GEMM_NO_BALANCE) the second wavefront of a SIMD leaves the loop
                // 0.8 us after the first instead of 1.9 us; worth 1 % at M = 256, nothing elsewhere.
                typedef __attribute__((address_space(3))) uint32_t *LdsProg;
                const uint32_t prog_mine = lds_base0 + p.prog_off + (uint32_t)wave * 4u;
                const uint32_t prog_other = lds_base0 + p.prog_off + (uint32_t)(wave ^ 4) * 4u;
                int other_left = left;
                while (left > 0) {
                    uint32_t seen = 0;
                    if (p.balance) {
                        if (left >= other_left) __builtin_amdgcn_s_setprio(1);
                        else __builtin_amdgcn_s_setprio(0);
                        *(LdsProg)(uintptr_t)prog_mine = (uint32_t)left;
                        seen = *(LdsProg)(uintptr_t)prog_other;
                    } else {
                        if ((left + wave_hi) & 1) __builtin_amdgcn_s_setprio(1);
                        else __builtin_amdgcn_s_setprio(0);
                    }
                    const u4_t *apn = left > 1 ? ap + astep : ap;
                    // this tile's first-half operands (and, older, the tile itself) have arrived;
                    // the second-half operands may still be in flight
                    wait_half(A0, std::integral_constant<int, MB>());
                    read_codes(1, cur);                   // this tile, second half
                    __builtin_amdgcn_sched_barrier(0);
                    half(A0, apn, [&] {
                        // the tile after next goes into the buffer just read out: not before
                        // those reads have returned (four products later they have)
                            asm volatile("s_waitcnt lgkmcnt(0)"
                                     : "+v"(Q8[0]), "+v"(Q8[1]), "+v"(Q8[2]), "+v"(Q8[3]), "+v"(Q8[4]),
                                       "+v"(Q8[5]), "+v"(Q8[6]), "+v"(Q8[7]) :: "memory");
                        if (left > 2) lean_tq += qstep;
                        lean_tile(cur != 0);
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    // second-half operands and (older) the next tile have arrived; the tile after
                    // next and the next first-half operands may be in flight
                    wait_half(A1, std::integral_constant<int, 4 + MB>());
                    read_codes(0, cur ^ 4096u);           // next tile, first half
                    __builtin_amdgcn_sched_barrier(0);
                    half(A1, apn + jstep, [] {});
                    ap = apn;
                    cur ^= 4096u;
                    --left;
                    if (p.balance) other_left = __builtin_amdgcn_readfirstlane((int)seen);
                }
                // nothing may land in LDS or in a register once the tree reuses them
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            } else {
            if (left > 0) {
                stage_write();                            // first tile, requested before the tables
                if (left > 1) tp += qstep;
                load_tile();                              // second tile (or a harmless reload)
            }
            while (left > 0) {
                // The two wavefronts of a SIMD (wavefront w and w + 4) take turns at the higher
                // priority, tile by tile, so that neither falls a tile behind the other
                // (measured with the builds interleaved: about 1 % at M = 256 and M = 1024).
                if ((left + (wave >> 2)) & 1) __builtin_amdgcn_s_setprio(1);
                else __builtin_amdgcn_s_setprio(0);
                stage_read();                             // this tile's chunk
                __builtin_amdgcn_sched_barrier(0);
                half_mma<4, MB, BF16, true>(Q, 0, A0, acc, lb, 8);
                if (left > 1) ap += astep;
                load_a(A0, ap);                           // half a tile ahead of its use
                // issue order activations -> tile: the wait for these activations at the
                // top of the next iteration then does not include the tile load
                __builtin_amdgcn_sched_barrier(0);
                stage_write();                            // next tile, requested a whole tile ago
                if (left > 2) tp += qstep;
                load_tile();                              // the tile after it
                __builtin_amdgcn_sched_barrier(0);
                half_mma<4, MB, BF16, true>(Q, 1, A1, acc, lb, 8);
                load_a(A1, ap + jstep);
                __builtin_amdgcn_sched_barrier(0);
                --left;
            }
            }
            __builtin_amdgcn_s_setprio(0);
        } else {
            uint32_t lb[4];
            table_bases(lb, 0, B1);
            const int cs = p.rep_log2[0] + 2;
            uint32_t Qa[4 * B1], Qb[4 * B1];
            const uint8_t *qp = w.q[0] + (((int64_t)t * p.G + g0) * 64 + th) * (16 * B1);
            constexpr int64_t qstep = (int64_t)KW * 64 * 16 * B1;
            const int64_t astep = (int64_t)KW * 2 * p.mblk_pad * 64;
            if (left > 0) {
                load_chunk<B1>(Qa, qp);
                load_a(A0, ap);
                load_a(A1, ap + jstep);
            }
            // One tile: the next chunk is requested first (a whole tile ahead), the
            // activation halves of the next tile as soon as their registers are free.
            auto step = [&](const uint32_t (&Qc)[4 * B1], uint32_t (&Qn)[4 * B1], bool more) {
                if (more) {                              // else: harmless reload of this tile
                    qp += qstep;
                    ap += astep;
                }
                load_chunk<B1>(Qn, qp);
                __builtin_amdgcn_sched_barrier(0);
                half_mma<B1, MB, BF16, PERM>(Qc, 0, A0, acc, lb, cs);
                load_a(A0, ap);
                __builtin_amdgcn_sched_barrier(0);
                half_mma<B1, MB, BF16, PERM>(Qc, 1, A1, acc, lb, cs);
                load_a(A1, ap + jstep);
                __builtin_amdgcn_sched_barrier(0);
            };
            while (left > 0) {
                step(Qa, Qb, left > 1);
                if (--left == 0) break;
                step(Qb, Qa, left > 1);
                --left;
            }
        }
    }

    // a lean loop's loads land in LDS and registers without the compiler's knowledge: none may
    // be in flight when the tree reuses either (wavefronts without work have issued some too)
    if constexpr (LEAN) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // ---- tree over the KW wavefronts of one m group, through LDS ------------------
    f4_t *red = (f4_t *)smem;                           // slot = [MB*8][64] f4
#ifdef FLUTE_STAMPS
    if (g_gemm_stamps && lane == 0) {
        long long *sl = g_gemm_stamps + (((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * (NT / 64) * 8 + wave * 8;
        sl[7] = (long long)__builtin_readcyclecounter() - sl[7];
    }
#endif
    FLUTE_STAMP(2);
    __syncthreads();                                    // tables are dead from here
    FLUTE_STAMP(3);
    // Four blocks of rows per wavefront and the image in the order of image_block_xor: accumulator j
    // of k way kw holds block j ^ x(kw).  Instead of the tree every wavefront hands the blocks it
    // does not keep to the k way that keeps them: accumulators 2 and 3 to the k way whose 0 and 1
    // they are, then accumulator 1 to the one whose 0 it is; with eight k ways two of them then
    // hold the same block and the odd one gives its sums to the even one.  The same bytes cross
    // LDS as in the tree and the sums are the same (every addition commutes), but all eight
    // wavefronts move them, barriers go, and four or eight wavefronts write the totals tile.
    const bool scattered = p.scatter != 0;
    if (scattered) {
        constexpr int P1 = KW == 4 ? 2 : 4, P2 = KW == 4 ? 1 : 2;   // partners of the two hand-overs
        f4_t *mine1 = red + (size_t)wave * 1024;
        const f4_t *theirs1 = red + (size_t)(wave ^ P1) * 1024;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            mine1[i * 64 + lane] = acc[2][i];
            mine1[(8 + i) * 64 + lane] = acc[3][i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            acc[0][i] += theirs1[i * 64 + lane];
            acc[1][i] += theirs1[(8 + i) * 64 + lane];
        }
        __syncthreads();
        // second hand-over: behind the region the totals tile takes (17 * 4 KB from the start), which the
        // residual's tile takes too (residual_tile waits)
        f4_t *mine2 = red + 4352 + (size_t)wave * 512;
        const f4_t *theirs2 = red + 4352 + (size_t)(wave ^ P2) * 512;
#pragma unroll
        for (int i = 0; i < 8; ++i) mine2[i * 64 + lane] = acc[1][i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[0][i] += theirs2[i * 64 + lane];
        if constexpr (KW == 8) {
            // k ways kw and kw ^ 1 hold the same block: between the (smaller) totals tile
            // and the second hand-over's areas
            f4_t *pair3 = red + 2176 + (size_t)(wave >> 1) * 512;
            if (kw & 1) {
#pragma unroll
                for (int i = 0; i < 8; ++i) pair3[i * 64 + lane] = acc[0][i];
            }
            __syncthreads();
            if (!(kw & 1)) {
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[0][i] += pair3[i * 64 + lane];
            }
        }
    }
#pragma unroll
    for (int step = KW / 2; step >= 1; step >>= 1) {
        if (scattered) break;
        if (kw >= step && kw < 2 * step) {
            f4_t *slot = red + (size_t)((kw - step) * MW + mw) * (MB * 8 * 64);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int i = 0; i < 8; ++i) slot[(mb * 8 + i) * 64 + lane] = acc[mb][i];
        }
        __syncthreads();
        if (kw < step) {
            const f4_t *slot = red + (size_t)(kw * MW + mw) * (MB * 8 * 64);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[mb][i] += slot[(mb * 8 + i) * 64 + lane];
        }
        __syncthreads();
    }

    FLUTE_STAMP(4);
    // ---- totals of the workgroup as a row-major fp32 tile in LDS --------------------
    constexpr int ROWS = MW * MB * 16;                  // rows of C this workgroup owns
    constexpr int LDT = 128 + 4;                        // padded row: conflict-free both ways
    float *tile = (float *)smem;
    // Residual, xb @ resA^T, as a tile of its own behind the totals' (gemm_residual_offset): fp32 products on
    // the matrix cores, sixteen ranks a step, of which lane group kg holds four (the order of ranks is free
    // as long as both operands agree); wavefront i takes the outputs 16 * i ... + 15 of every row.  resA and
    // xb are read once each; every thread reading the eight rows of resA behind its outputs and adding rank by
    // rank: M = 1271, 1344 -> 3200, 3 bits, rank 16, the launch 40.6 us, now 27; M = 256,
    // 4096 -> 12288, 4 bits, rank 16, the call 54.5 and 42.4; M = 300, 4096 -> 4096 39.8 and 32.8.
    float *const rtile = (float *)(smem + gemm_residual_offset(ROWS));
    auto residual_tile = [&] {
        constexpr int BLOCKS = ROWS / 16;
        f4_t sum[BLOCKS];
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) sum[b] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
        const uint16_t *const ra = w.resA + (int64_t)(t * 128 + wave * 16 + rho) * w.R;
#pragma unroll 1
        for (int r0 = 0; r0 < w.R; r0 += 16) {
            const int k0 = r0 + kg * 4;
            uint32_t h[2] = {0u, 0u};
            f4_t x[BLOCKS];
#pragma unroll
            for (int b = 0; b < BLOCKS; ++b) x[b] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
            if (w.vec_res) {                            // uniform
                if (k0 < w.R) {
                    const uint2 raw = *(const uint2 *)(ra + k0);
                    h[0] = raw.x;
                    h[1] = raw.y;
#pragma unroll
                    for (int b = 0; b < BLOCKS; ++b)
                        x[b] = *(const f4_t *)(w.xb + (int64_t)min((int)blockIdx.y * ROWS + b * 16 + rho, p.M - 1) * w.R + k0);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (k0 + e >= w.R) continue;
                    h[e >> 1] |= (uint32_t)ra[k0 + e] << (16 * (e & 1));
#pragma unroll
                    for (int b = 0; b < BLOCKS; ++b)
                        x[b][e] = w.xb[(int64_t)min((int)blockIdx.y * ROWS + b * 16 + rho, p.M - 1) * w.R + k0 + e];
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint16_t one = (uint16_t)(h[e >> 1] >> (16 * (e & 1)));
                const float a = p.out_bf16 ? bf2f(one) : h2f(one);
#pragma unroll
                for (int b = 0; b < BLOCKS; ++b)
                    sum[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, x[b][e], sum[b], 0, 0, 0);
            }
        }
        // Its tile lies where the k ways have handed blocks to each other (theirs2, pair3): a wavefront may be past
        // its reads while another is not.  (Of several slices barriers lie between, as they do behind the tree.)
        if (scattered && p.ztotal == 1) __syncthreads();
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) *(f4_t *)(rtile + (b * 16 + rho) * LDT + wave * 16 + kg * 4) = sum[b];
    };
    if (scattered) {                                    // the totals of block x(kw) are in accumulator 0
        if (KW == 4 || !(kw & 1)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = (mw * MB + image_block_xor(kw, p.scatter)) * 16 + rho;
            const int n0 = (kg >> 1) * 64 + (i >> 1) * 16 + (i & 1) * 8 + (kg & 1) * 4;
            *(f4_t *)(tile + row * LDT + n0) = acc[0][i];
        }
        }
    } else if (kw == 0) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int row = (mw * MB + mb) * 16 + rho;
                const int n0 = (kg >> 1) * 64 + (i >> 1) * 16 + (i & 1) * 8 + (kg & 1) * 4;
                *(f4_t *)(tile + row * LDT + n0) = acc[mb][i];
            }
    }
    if (w.R > 0 && p.ztotal == 1) residual_tile();      // (of several slices the last arrival forms it)
    __syncthreads();

    FLUTE_STAMP(5);
    // Every thread now serves pieces of 8 consecutive outputs of one row: 16 threads
    // write one 256-byte row segment of C.
    constexpr int PIECES = ROWS * 16;
    const int unit = blockIdx.y * gridDim.x + blockIdx.x;           // (m chunk, n tile)
    const size_t image = (size_t)ROWS * 128;                        // floats per unit per z
    const size_t zstride = (size_t)gridDim.x * gridDim.y * image;
    if (p.ztotal > 1) {
        // across workgroups: partial tiles + ticket; the last arrival folds them in z order
        float *mine = p.P + (size_t)(p.z_base + z) * zstride + (size_t)unit * image;
        for (int idx = tid; idx < PIECES; idx += NT) {
            const int ml = idx >> 4, n8 = idx & 15;
            ws_store16(mine + ml * 128 + n8 * 8, *(const f4_t *)(tile + ml * LDT + n8 * 8));
            ws_store16(mine + ml * 128 + n8 * 8 + 4, *(const f4_t *)(tile + ml * LDT + n8 * 8 + 4));
        }
        ws_stores_done();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        int *flag = (int *)(tile + ROWS * LDT);
        if (tid == 0) {
            const int old = __hip_atomic_fetch_add(p.tickets + unit, 1, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
            *flag = (old == p.ztotal - 1);
        }
        __syncthreads();
        if (!*flag) return;
        if (tid == 0)
            __hip_atomic_store(p.tickets + unit, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (w.R > 0) {
            residual_tile();
            __syncthreads();
        }
    }

    // ---- epilogue: residual, bias, one rounding, store -------------------------------
    for (int idx = tid; idx < PIECES; idx += NT) {
        const int ml = idx >> 4, n8 = idx & 15;
        const int m = blockIdx.y * ROWS + ml;
        if (m >= p.M) continue;
        const int n0 = t * 128 + n8 * 8;
        float y[8];
        if (p.ztotal > 1) {
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = 0.0f;
            const float *src = p.P + (size_t)unit * image + ml * 128 + n8 * 8;
            for (int z0 = 0; z0 < p.ztotal; z0 += 2) {
                const float *s0 = src + z0 * zstride;
                const float *s1 = z0 + 1 < p.ztotal ? s0 + zstride : s0;
                f4_t a, b, c, d;
                ws_load16x4(s0, s0 + 4, s1, s1 + 4, a, b, c, d);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    y[e] += a[e];
                    y[4 + e] += b[e];
                }
                if (z0 + 1 < p.ztotal) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        y[e] += c[e];
                        y[4 + e] += d[e];
                    }
                }
            }
        } else {
            const f4_t lo = *(const f4_t *)(tile + ml * LDT + n8 * 8);
            const f4_t hi = *(const f4_t *)(tile + ml * LDT + n8 * 8 + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[e] = lo[e];
                y[4 + e] = hi[e];
            }
        }
        if (p.rowshift) {                               // undo the row's activation scaling (exact)
            const int sh = p.rowshift[m];
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = ldexpf(y[e], sh);
        }
        if (w.R > 0) {
            const f4_t lo = *(const f4_t *)(rtile + ml * LDT + n8 * 8);
            const f4_t hi = *(const f4_t *)(rtile + ml * LDT + n8 * 8 + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[e] += lo[e];
                y[4 + e] += hi[e];
            }
        }
        if (w.bias) {
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] += load_act(w.bias, n0 + e, p.out_bf16);
        }
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = (uint32_t)round_act(y[2 * e], p.out_bf16) |
                   ((uint32_t)round_act(y[2 * e + 1], p.out_bf16) << 16);
        uint16_t *dst = (uint16_t *)w.C + (size_t)m * w.ldc + n0;
        if (w.vec_store) {
            *(u4_t *)dst = u4_t{o[0], o[1], o[2], o[3]};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                dst[2 * e] = (uint16_t)o[e];
                dst[2 * e + 1] = (uint16_t)(o[e] >> 16);
            }
        }
    }
    FLUTE_STAMP(6);
}

}  // namespace flute
