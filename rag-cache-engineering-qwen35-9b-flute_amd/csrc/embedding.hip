// Embedding rows out of a palettized table: a gather through the idxN layout, the
// second stream, the low-rank residual and the un-rotation of tied (rotated) tables,
// in the dtype ladder of the upstream module (scripts/palettized_modules.py:1998-2015,
// 2298-2335):
//     w   = lut1[n / gs][idx1[n, :]]  (+ lut2[...] in the LUT's 16-bit type, stream 1 first)
//     row = float(w) + resA[n, :] @ resB                (fp32)
//     row = row @ T^T  when the table is rotated          (adjoint transform, fp32)
//     out = row rounded once to the LUT's type
#include "fht_dev.h"
#include "host_common.h"
#include "verdicts.h"

#include <atomic>
#include <chrono>

namespace flute {

namespace {

constexpr int kEmbThreads = 256;

struct EmbParams {
    const uint8_t *q[2];
    const uint16_t *lut[2];
    const uint16_t *resA, *resB;
    const float *signs;
    const int64_t *ids;
    uint16_t *out;
    int bits[2];
    int nstreams;
    int N, K, gs, lut_rows, R;
    int bf16;        // LUT / output / residual dtype
    int block;       // rotation block (0: descending power-of-two segments)
    int vec_out;     // rows of out allow 16-byte stores
};

// A thread's share of a row is quarter kt of tile g: sixteen consecutive columns, whose codes lie
// in the four chunks c4 = 0 ... 3 of the row's chunk group (columns c4*2 + 8*s2 (+1) of the quarter
// are the pairs s2 = 0, 1 of chunk c4), 4*B consecutive bits each: byte B*v + (4*B*d)/8 of the
// quarter's 4*B bytes.  Sixteen neighbouring threads' bytes are the 256*B ones of four chunk groups.
__device__ __forceinline__ uint32_t chunk_codes(const uint8_t *p, int b, int d) {
    if (b == 4) return *(const uint16_t *)(p + 2 * d);
    if (b == 3) return (((uint32_t)p[d] | ((uint32_t)p[d + 1] << 8)) >> (4 * d)) & 0xfffu;
    if (b == 2) return p[d];
    return (uint32_t)*p >> (4 * d);
}

__device__ __forceinline__ float to_f(uint32_t h, int bf16) {
    return bf16 ? bf2f((uint16_t)h) : h2f((uint16_t)h);
}

// The grid's first workgroup looks all ids over and leaves its verdict in host memory, 1 = every id lies in the
// table, 2 = some do not.
__device__ __forceinline__ void check_ids(const EmbParams &p, int64_t count, int *check) {
    __shared__ int bad;
    const int tid = threadIdx.x;
    if (tid == 0) bad = 0;
    __syncthreads();
    int mine = 0;
    for (int64_t i = tid; i < count; i += 8 * kEmbThreads) {
        int64_t id[8];                                  // (past the end: the last one again)
#pragma unroll
        for (int u = 0; u < 8; ++u) id[u] = p.ids[i + u * kEmbThreads < count ? i + u * kEmbThreads : count - 1];
#pragma unroll
        for (int u = 0; u < 8; ++u) mine |= id[u] < 0 || id[u] >= p.N;
    }
    if (mine) bad = 1;
    __syncthreads();
    if (tid == 0) __hip_atomic_store(check, bad ? 2 : 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Rows of up to 4096 columns: one workgroup per requested row, sixteen consecutive columns a thread, all segments
// of a rotated row side by side.  What bounds it: for few rows the chain id -> codes -> values -> butterfly -> store,
// for many vector and LDS instructions, so widths and types are decided outside the loops over the values, the LUT
// row lies in LDS as fp32 (16-bit LDS reads take four times a dword's), the codes of a stream are requested together,
// stages between lanes exchange halves in registers, the ones above cross LDS once, and stores are
// contiguous.  In a graph, the kernel below and this one, us: 1000 rows of 4096 columns, 4 bits, rotated 13.8 / 9.9, plain
// 11.0 / 8.5; 4000 rotated 45.1 / 25; 2000 of 3136, (1, 4) bits, rotated 32.5 / 17.5; 64 rotated 6.5 / 4.4.
constexpr int kEmbRow = kEmbThreads * 16;
// Dynamic LDS of a wavefront: its 1024 columns in fp32 (rotated), or as it stores them.
__host__ __device__ constexpr int emb_wave_bytes(bool rotated) { return rotated ? 4096 : 2048; }

// Codes of the columns k ... k + 15 of a row as chunks c4 = 0 ... 3 (from = the row's place in its tile row).
template <int B>
__device__ __forceinline__ void row_codes(const uint8_t *from, int k, int d, uint32_t (&c)[4]) {
    const uint8_t *const at = from + (size_t)(k >> 6) * (1024 * B) + ((k >> 4) & 3) * (4 * B);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint8_t *const q = at + i * 16 * B;
        if constexpr (B == 4) c[i] = *(const uint16_t *)(q + 2 * d);
        else if constexpr (B == 3) c[i] = ((uint32_t)q[d] | ((uint32_t)q[d + 1] << 8)) >> (4 * d);
        else if constexpr (B == 2) c[i] = q[d];
        else c[i] = (uint32_t)*q >> (4 * d);
    }
}
// Their values out of the LUT row, fp32 in LDS.
template <int B>
__device__ __forceinline__ void row_values(const float *lut, const uint32_t (&c)[4], float (&f)[16]) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int i = (j >> 1) & 3, shift = 2 * (j >> 3) + (j & 1);         // in codes
        f[j] = lut[__builtin_amdgcn_ubfe(c[i], B * shift, B)];
    }
}

template <bool BF16, bool ROT>
__global__ void __launch_bounds__(kEmbThreads) embedding_row_kernel(const EmbParams p, int64_t count, int *check) {
    extern __shared__ __align__(16) uint8_t lds[];
    float *const buf = (float *)lds;                    // (ROT, segments beyond 1024 columns)
    __shared__ float luts[2][16];
    const int tid = threadIdx.x, lane = tid & 63;
    if (check && blockIdx.x == 0) {
        check_ids(p, count, check);
        return;
    }
    const int64_t row = (int64_t)blockIdx.x - (check ? 1 : 0);
    const int64_t n64 = p.ids[row];
    uint16_t *const out = p.out + (size_t)row * p.K;
    if (n64 < 0 || n64 >= p.N) {                        // refused on the host; never read out of range
        for (int k = tid; k < p.K; k += kEmbThreads) out[k] = 0;
        return;
    }
    const int n = (int)n64, G = p.K >> 6;
    const int wx = (n >> 6) & 1, v = (n >> 4) & 3, d = (n >> 3) & 1, r8 = n & 7;
    const bool mine = tid * 16 < p.K;
    const int k = min(tid * 16, p.K - 16);
    uint32_t c[2][4];
    auto codes = [&](int s) {
        const int b = p.bits[s];
        const uint8_t *const from = p.q[s] + (size_t)(n >> 7) * G * (1024 * b) + (wx * 32 + r8 * 4) * (16 * b) + b * v;
        switch (b) {                                    // uniform, around all of a stream's loads
            case 4: row_codes<4>(from, k, d, c[s]); break;
            case 3: row_codes<3>(from, k, d, c[s]); break;
            case 2: row_codes<2>(from, k, d, c[s]); break;
            default: row_codes<1>(from, k, d, c[s]); break;
        }
    };
    auto act = [](uint16_t h) { return BF16 ? bf2f(h) : h2f(h); };
    float sg[ROT ? 16 : 1];
    if constexpr (ROT) {
#pragma unroll
        for (int e = 0; e < 16; ++e) sg[e] = p.signs[k + e];
    }
    codes(0);
    if (p.nstreams == 2) codes(1);
    {
        const int grp = min(n / p.gs, p.lut_rows - 1), s = tid >> 4, e = tid & 15;
        if (tid < 32 && s < p.nstreams && e < (1 << p.bits[s])) luts[s][e] = act(p.lut[s][((size_t)grp << p.bits[s]) + e]);
    }
    __syncthreads();                                    // the LUT rows are in
    float f[16];
    auto values = [&](int s, float (&t)[16]) {
        switch (p.bits[s]) {
            case 4: row_values<4>(luts[s], c[s], t); break;
            case 3: row_values<3>(luts[s], c[s], t); break;
            case 2: row_values<2>(luts[s], c[s], t); break;
            default: row_values<1>(luts[s], c[s], t); break;
        }
    };
    values(0, f);
    if (p.nstreams == 2) {
        float t[16];
        values(1, t);
        // the 16-bit add of the module: exact sum, one rounding to the LUT's type
#pragma unroll
        for (int j = 0; j < 16; ++j) f[j] = act(round_act(f[j] + t[j], BF16));
    }
    if (p.R > 0) {
        float sum[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) sum[j] = 0.0f;
        for (int r = 0; r < p.R; ++r) {
            const float a = act(p.resA[(size_t)n * p.R + r]);
            const uint16_t *const b = p.resB + (size_t)r * p.K + k;
#pragma unroll
            for (int j = 0; j < 16; ++j) sum[j] = fmaf(a, act(b[j]), sum[j]);
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) f[j] += sum[j];
    }
    auto pair = [](float a, float b) { return (uint32_t)round_act(a, BF16) | ((uint32_t)round_act(b, BF16) << 16); };
    // A wavefront's 1024 columns out, sixteen bytes a lane side by side: its lanes' 32 bytes change places through
    // LDS on the way (as two stores 32 bytes apart: 1000 plain rows of 4096 columns 11.5 us, 8.5).
    // (the wavefront's own part of the dynamic memory, which the stages across wavefronts use otherwise)
    auto store16 = [&] {
        if ((tid >> 6) * 1024 >= p.K) return;           // a whole wavefront past the end
        uint4 *const at = (uint4 *)(lds + (tid >> 6) * emb_wave_bytes(ROT));
#pragma unroll
        for (int h = 0; h < 2; ++h)
            at[2 * lane + (h ^ ((lane >> 2) & 1))] = make_uint4(pair(f[8 * h], f[8 * h + 1]), pair(f[8 * h + 2], f[8 * h + 3]),
                                                                pair(f[8 * h + 4], f[8 * h + 5]), pair(f[8 * h + 6], f[8 * h + 7]));
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int i = h * 64 + lane, col = (tid >> 6) * 1024 + i * 8;
            if (col >= p.K) continue;
            const uint4 o = at[i ^ ((i >> 3) & 1)];
            if (p.vec_out) {
                *(uint4 *)(out + col) = o;
            } else {
                const uint32_t w[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) *(uint32_t *)(out + col + 2 * e) = w[e];
            }
        }
    };
    if constexpr (!ROT) {
        store16();
    } else {
        // the adjoint transform: ten stages within a wavefront (1024 columns), the one or two above across
        // wavefronts through LDS
        const int nst = column_stages(k, p.K, p.block);
#pragma unroll
        for (int e = 0; e < 16; ++e) f[e] *= sg[e];
        stages_in_thread(f);
        if (__all(nst >= 10)) {
            stage_all_lanes<1>(f, lane);
            stage_all_lanes<2>(f, lane);
            stage_all_lanes<4>(f, lane);
            stage_all_lanes<8>(f, lane);
            stage_all_lanes<16>(f, lane);
            stage_all_lanes<32>(f, lane);
        } else {
            stage_some_lanes<1>(f, lane, nst > 4);
            stage_some_lanes<2>(f, lane, nst > 5);
            stage_some_lanes<4>(f, lane, nst > 6);
            stage_some_lanes<8>(f, lane, nst > 7);
            stage_some_lanes<16>(f, lane, nst > 8);
            stage_some_lanes<32>(f, lane, nst > 9);
        }
        const float inv = inv_sqrt_pow2(nst);
        const int top = column_stages(0, p.K, p.block); // the longest segment is the first
        // (a segment beyond 1024 columns takes whole wavefronts)
        if (__any(mine && nst <= 10)) {
#pragma unroll
            for (int e = 0; e < 16; ++e) f[e] *= inv;
            store16();
        } else if (mine) {
            // piece q of thread t (16 bytes) lies at t * 4 + (q ^ (t >> 1 & 3)): writers side by side, and readers
            // of consecutive pieces, meet different banks
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *(float4 *)(buf + tid * 16 + ((q ^ ((tid >> 1) & 3)) << 2)) = make_float4(f[4 * q], f[4 * q + 1], f[4 * q + 2], f[4 * q + 3]);
        }
        if (top <= 10) return;                          // uniform
        __syncthreads();
        // Four columns of each of the 2^T chunks of 1024 a thread: the stages between chunks, and a store of
        // eight bytes a lane side by side.
        auto across = [&](auto stages, int chunk0) {
            constexpr int T = decltype(stages)::value, E = 1 << T;
            float w[4][E];
#pragma unroll
            for (int h = 0; h < E; ++h) {
                const int t = (chunk0 + h) * 64 + (tid >> 2);
                const float4 x = *(const float4 *)(buf + t * 16 + (((tid & 3) ^ ((t >> 1) & 3)) << 2));
                w[0][h] = x.x; w[1][h] = x.y; w[2][h] = x.z; w[3][h] = x.w;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) stages_in_thread(w[q]);
            const float scale = inv_sqrt_pow2(10 + T);
#pragma unroll
            for (int h = 0; h < E; ++h) {
                uint16_t *const to = out + (chunk0 + h) * 1024 + tid * 4;
                const uint32_t lo = pair(w[0][h] * scale, w[1][h] * scale), hi = pair(w[2][h] * scale, w[3][h] * scale);
                if (p.vec_out) {
                    *(uint2 *)to = make_uint2(lo, hi);
                } else {
                    *(uint32_t *)to = lo;
                    *(uint32_t *)(to + 2) = hi;
                }
            }
        };
        if (top == 12) {
            across(std::integral_constant<int, 2>(), 0);
        } else {
            across(std::integral_constant<int, 1>(), 0);
            if (p.block == 2048 && p.K == 4096) across(std::integral_constant<int, 1>(), 2);
        }
    }
}

// Rows of more than 4096 columns.  One workgroup per requested row, sixteen consecutive columns a thread, 4096 a
// step, segments of a rotated row one after the other.  What bounds it: the chain id -> codes -> values ->
// butterfly -> store, so everything a phase needs is requested together (the LUT row goes to LDS beside the codes
// and signs, a value costs one LDS read) and the first ten stages of the butterfly stay in registers.  In a graph,
// 4 bits, rotated and plain, us: 1000 rows of 4160 columns 17.3 / 12.9, of 8192 26.9 / 18.3, of 12288 35.3 / 27.2;
// 64 of 8192 11.2 / 7.2; 4000 of 8192 78.5 / 54.3, which cannot do without 131 MB of lines read (a row's codes are an
// eighth of those they lie in) and 66 MB written, 39 us at a copy's rate.
// check != NULL: the first workgroup of the grid looks all ids over instead (check_ids).
__global__ void __launch_bounds__(kEmbThreads) embedding_kernel(const EmbParams p, int64_t count, int *check) {
    extern __shared__ __align__(16) uint8_t lds[];
    float *buf = (float *)lds;
    __shared__ uint16_t luts[2][16];
    const int tid = threadIdx.x;
    if (check && blockIdx.x == 0) {
        check_ids(p, count, check);
        return;
    }
    const int64_t at = (int64_t)blockIdx.x - (check ? 1 : 0);
    const int64_t n64 = p.ids[at];
    uint16_t *out = p.out + (size_t)at * p.K;
    if (n64 < 0 || n64 >= p.N) {                  // refused on the host; never read out of range
        for (int k = tid; k < p.K; k += kEmbThreads) out[k] = 0;
        return;
    }
    const int n = (int)n64;
    const int G = p.K >> 6;
    const int grp = min(n / p.gs, p.lut_rows - 1);
    const int wx = (n >> 6) & 1, v = (n >> 4) & 3, d = (n >> 3) & 1, r8 = n & 7;
    const uint8_t *q[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) q[s] = p.q[s] + (size_t)(n >> 7) * G * (1024 * p.bits[s]);
    if (tid < 32) {
        const int s = tid >> 4, e = tid & 15;
        if (s < p.nstreams && e < (1 << p.bits[s])) luts[s][e] = p.lut[s][((size_t)grp << p.bits[s]) + e];
    }
    const uint8_t *src[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) src[s] = q[s] + (wx * 32 + r8 * 4) * (16 * p.bits[s]) + p.bits[s] * v;
    // codes of the columns k ... k + 15 (k a multiple of 16), as chunk c4 of stream s
    auto codes = [&](int s, int k, uint32_t (&c)[4]) {
        const int b = p.bits[s];
        const uint8_t *at_k = src[s] + (size_t)(k >> 6) * (1024 * b) + ((k >> 4) & 3) * (4 * b);
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = chunk_codes(at_k + i * 16 * b, b, d);
    };
    auto values = [&](int k, const uint32_t (&c)[2][4], float (&f)[16]) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int i = (j >> 1) & 3, shift = 2 * (j >> 3) + (j & 1);    // in codes
            const int b = p.bits[0];
            f[j] = to_f(luts[0][(c[0][i] >> (b * shift)) & ((1 << b) - 1)], p.bf16);
        }
        if (p.nstreams == 2) {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int i = (j >> 1) & 3, shift = 2 * (j >> 3) + (j & 1);
                const int b = p.bits[1];
                // the 16-bit add of the module: exact sum, one rounding to the LUT's type
                f[j] = to_f(round_act(f[j] + to_f(luts[1][(c[1][i] >> (b * shift)) & ((1 << b) - 1)], p.bf16), p.bf16), p.bf16);
            }
        }
        if (p.R > 0) {
            float sum[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) sum[j] = 0.0f;
            for (int r = 0; r < p.R; ++r) {
                const float a = to_f(p.resA[(size_t)n * p.R + r], p.bf16);
                const uint16_t *row = p.resB + (size_t)r * p.K + k;
#pragma unroll
                for (int j = 0; j < 16; ++j) sum[j] = fmaf(a, to_f(row[j], p.bf16), sum[j]);
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) f[j] += sum[j];
        }
    };
    auto store = [&](int k, const float (&f)[16]) {
        uint32_t o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            o[e] = (uint32_t)round_act(f[2 * e], p.bf16) | ((uint32_t)round_act(f[2 * e + 1], p.bf16) << 16);
        if (p.vec_out) {
            *(uint4 *)(out + k) = make_uint4(o[0], o[1], o[2], o[3]);
            *(uint4 *)(out + k + 8) = make_uint4(o[4], o[5], o[6], o[7]);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) *(uint32_t *)(out + k + 2 * e) = o[e];
        }
    };
    constexpr int STEP = kEmbThreads * 16;
    const int lane = tid & 63;
    uint32_t c[2][4];
    {
        // codes of this thread's first columns, beside the LUT row
        const int k = min(tid * 16, p.K - 16);
        codes(0, k, c[0]);
        if (p.nstreams == 2) codes(1, k, c[1]);
    }
    __syncthreads();                                      // the LUT rows are in

    if (p.signs == nullptr) {
        for (int k = tid * 16; k < p.K; k += STEP) {
            if (k >= STEP) {
                codes(0, k, c[0]);
                if (p.nstreams == 2) codes(1, k, c[1]);
            }
            float f[16];
            values(k, c, f);
            store(k, f);
        }
        return;
    }
    // rotated table: the adjoint transform of the row, segment by segment
    for (int off = 0; off < p.K;) {
        int cols, nst;
        if (p.block > 0) {
            nst = 31 - __builtin_clz((unsigned)p.block);
            cols = min((16384 / p.block) * p.block, p.K - off);
        } else {
            nst = 31 - __builtin_clz((unsigned)(p.K - off));
            cols = 1 << nst;
        }
        const float inv = inv_sqrt_pow2(nst);
        for (int j = tid * 16; j < cols; j += STEP) {
            const int k = off + j;
            float sg[16], f[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) sg[e] = p.signs[k + e];
            if (k >= STEP || off > 0) {
                codes(0, k, c[0]);
                if (p.nstreams == 2) codes(1, k, c[1]);
            }
            values(k, c, f);
#pragma unroll
            for (int e = 0; e < 16; ++e) f[e] *= sg[e];
            fht_head(f, lane, nst);
            if (nst <= 10) {
#pragma unroll
                for (int e = 0; e < 16; ++e) f[e] *= inv;
                store(k, f);
            } else {
                const int s0 = fht_slot(j);               // a multiple of 16: slot(j + q) = s0 ^ q
#pragma unroll
                for (int e = 0; e < 16; ++e) buf[s0 ^ e] = f[e];
            }
        }
        if (nst > 10) {
            __syncthreads();
            fht_tail(buf, cols, nst, 10, tid, kEmbThreads);
            for (int j = tid * 16; j < cols; j += STEP) {
                const int s0 = fht_slot(j);
                float f[16];
#pragma unroll
                for (int e = 0; e < 16; ++e) f[e] = buf[s0 ^ e] * inv;
                store(off + j, f);
            }
            __syncthreads();                              // the next segment reuses the buffer
        }
        off += cols;
    }
}

// Pinned words the kernel leaves its verdict on a call's ids in.
Verdicts g_verdicts;

flute_status verdict_memory(void **mem) {
    FLUTE_HIP_CHECK(hipHostMalloc(mem, Verdicts::kBytes, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent));
    return FLUTE_OK;
}

}  // namespace

}  // namespace flute

using namespace flute;

namespace {

flute_status embedding(const flute_linear *w, const int64_t *ids, int64_t count, void *out, hipStream_t stream,
                       int *check) {
    flute_status st = validate_linear(w, 1, "flute_embedding");
    if (st != FLUTE_OK) return st;
    FLUTE_REQUIRE(count >= 0 && count <= 0x7fffffffLL, FLUTE_ERR_INVALID,
                  "flute_embedding: count must be in [0, 2^31)");
    if (count == 0) return FLUTE_OK;
    FLUTE_REQUIRE(ids != nullptr && out != nullptr, FLUTE_ERR_INVALID,
                  "flute_embedding: ids and out must not be NULL");
    FLUTE_REQUIRE(w->bias == nullptr, FLUTE_ERR_INVALID, "flute_embedding: an embedding has no bias");
    FLUTE_REQUIRE(w->awq == nullptr, FLUTE_ERR_INVALID,
                  "flute_embedding: an embedding table carries no activation scale");
    FLUTE_REQUIRE(((uintptr_t)ids & 7) == 0, FLUTE_ERR_INVALID,
                  "flute_embedding: ids are int64 and must be 8-byte aligned");
    FLUTE_REQUIRE(((uintptr_t)out & 3) == 0, FLUTE_ERR_INVALID,
                  "flute_embedding: out must be 4-byte aligned");
    EmbParams p = {};
    p.q[0] = (const uint8_t *)w->q1;
    p.q[1] = (const uint8_t *)w->q2;
    p.lut[0] = (const uint16_t *)w->lut1;
    p.lut[1] = (const uint16_t *)w->lut2;
    p.bits[0] = w->b1;
    p.bits[1] = w->b2;
    p.nstreams = w->b2 > 0 ? 2 : 1;
    p.resA = (const uint16_t *)w->resA;
    p.resB = (const uint16_t *)w->resB;
    p.R = w->R;
    p.signs = w->signs;
    p.ids = ids;
    p.out = (uint16_t *)out;
    p.N = w->N;
    p.K = w->K;
    p.gs = w->group_size;
    p.lut_rows = w->lut_rows;
    p.bf16 = w->lut_dtype == FLUTE_BF16;
    p.block = w->rot_block;
    p.vec_out = ((uintptr_t)out & 15) == 0;             // (rows are K * 2 bytes, K a multiple of 64)
    FLUTE_REQUIRE(!w->signs || w->rot_block <= 0 ||
                      (is_pow2(w->rot_block) && w->rot_block >= 32 && w->rot_block <= 16384 && w->K % w->rot_block == 0),
                  FLUTE_ERR_INVALID,
                  "flute_embedding: rotation block must be a power of two in [32, 16384] dividing K");
    const dim3 grid((unsigned)(count + (check ? 1 : 0))), threads(kEmbThreads);
    if (w->K <= kEmbRow) {
        const int form = 2 * p.bf16 + (w->signs != nullptr);
        const size_t lds = (size_t)((w->K + 1023) / 1024) * emb_wave_bytes(w->signs != nullptr);
        if (form == 3) hipLaunchKernelGGL((embedding_row_kernel<true, true>), grid, threads, lds, stream, p, count, check);
        else if (form == 2) hipLaunchKernelGGL((embedding_row_kernel<true, false>), grid, threads, lds, stream, p, count, check);
        else if (form == 1) hipLaunchKernelGGL((embedding_row_kernel<false, true>), grid, threads, lds, stream, p, count, check);
        else hipLaunchKernelGGL((embedding_row_kernel<false, false>), grid, threads, lds, stream, p, count, check);
        FLUTE_HIP_CHECK(hipGetLastError());
        return FLUTE_OK;
    }
    size_t lds = 0;
    if (w->signs) {
        int columns = w->K;                             // that lie in LDS together
        if (w->rot_block <= 0) columns = make_segments(w->K, 0).len[0];
        else if (w->K > 16384) columns = (16384 / w->rot_block) * w->rot_block;
        lds = (size_t)columns * 4;
        static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
        if (!attr_done) {
            FLUTE_HIP_CHECK(hipFuncSetAttribute((const void *)embedding_kernel,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, 98304));
            attr_done = true;
        }
    }
    hipLaunchKernelGGL(embedding_kernel, grid, threads, lds, stream, p, count, check);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

}  // namespace

extern "C" flute_status flute_embedding(const flute_linear *w, const int64_t *ids, int64_t count,
                                        void *out, void *stream) {
    return embedding(w, ids, count, out, (hipStream_t)stream, nullptr);
}

extern "C" flute_status flute_embedding_checked(const flute_linear *w, const int64_t *ids, int64_t count,
                                                void *out, void *stream_, int *in_range) {
    FLUTE_REQUIRE(in_range != nullptr, FLUTE_ERR_INVALID, "flute_embedding_checked: in_range must not be NULL");
    hipStream_t stream = (hipStream_t)stream_;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    FLUTE_HIP_CHECK(hipStreamIsCapturing(stream, &cap));
    FLUTE_REQUIRE(cap == hipStreamCaptureStatusNone, FLUTE_ERR_INVALID,
                  "flute_embedding_checked: no value can reach the host while the stream is capturing; "
                  "flute_embedding writes zeros for an id outside the table");
    *in_range = 1;
    if (count == 0) return flute_embedding(w, ids, count, out, stream_);
    Verdicts::Word word;
    flute_status st = (flute_status)g_verdicts.take(word, verdict_memory);
    if (st != FLUTE_OK) return st;
    st = embedding(w, ids, count, out, stream, word.get());
    if (st != FLUTE_OK) {
        // (an error left by an earlier call may be reported behind a launch that went out: the word is
        // not another call's before the stream has done with it)
        if (st == FLUTE_ERR_HIP) (void)hipStreamSynchronize(stream);
        return st;
    }
    // The verdict comes from the grid's first workgroup, usually while the rows are still being
    // gathered; a stream that has much to do before it is waited for without spinning.
    int verdict = 0;
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    while (!(verdict = __atomic_load_n(word.get(), __ATOMIC_ACQUIRE)) && std::chrono::steady_clock::now() < until)
        __builtin_ia32_pause();
    if (!verdict) {
        FLUTE_HIP_CHECK(hipStreamSynchronize(stream));
        verdict = __atomic_load_n(word.get(), __ATOMIC_ACQUIRE);
        FLUTE_REQUIRE(verdict != 0, FLUTE_ERR_HIP, "flute_embedding_checked: the launch left no verdict");
    }
    *in_range = verdict == 1;
    return FLUTE_OK;
}
