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

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>

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

// One workgroup per requested row, sixteen consecutive columns a thread.  What bounds it: the chain
// id -> codes -> values -> butterfly -> store, so everything a phase needs is requested together
// (the LUT row goes to LDS beside the codes and signs, a value costs one LDS read) and the first ten
// stages of the butterfly stay in registers.  (One pair at a time, byte loads of the codes and trips
// to memory for the LUT, all stages in LDS: 15.2 us for 1000 rotated rows of 4096 columns, 4 bits,
// against 13.6; the check of the ids as five launches and a copy before it: 71 us a call against 27.)
// check != NULL: the first workgroup of the grid looks all ids over instead and leaves its verdict
// in host memory, 1 = every id lies in the table, 2 = some do not.
__global__ void __launch_bounds__(kEmbThreads) embedding_kernel(const EmbParams p, int64_t count, int *check) {
    extern __shared__ __align__(16) uint8_t lds[];
    float *buf = (float *)lds;
    __shared__ uint16_t luts[2][16];
    const int tid = threadIdx.x;
    if (check && blockIdx.x == 0) {
        __shared__ int bad;
        if (tid == 0) bad = 0;
        __syncthreads();
        int mine = 0;
        for (int64_t i = tid; i < count; i += kEmbThreads) mine |= p.ids[i] < 0 || p.ids[i] >= p.N;
        if (mine) bad = 1;
        __syncthreads();
        if (tid == 0) __hip_atomic_store(check, bad ? 2 : 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
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

// ---- verdicts ----------------------------------------------------------------------------
// Pinned words the kernel leaves its verdict on a call's ids in, one per call that waits for it:
// taken and given back under a lock, at most kVerdicts at a time (a further call waits for one).
constexpr int kVerdicts = 64, kVerdictStride = 16;        // one per 64-byte line
std::mutex g_verdict_mu;
std::condition_variable g_verdict_cv;
int *g_verdict_mem = nullptr;
uint64_t g_verdict_free = ~(uint64_t)0;

flute_status take_verdict(int *slot, int **word) {
    std::unique_lock<std::mutex> lock(g_verdict_mu);
    if (!g_verdict_mem) {
        void *mem = nullptr;
        FLUTE_HIP_CHECK(hipHostMalloc(&mem, kVerdicts * kVerdictStride * sizeof(int),
                                      hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent));
        g_verdict_mem = (int *)mem;
    }
    g_verdict_cv.wait(lock, [] { return g_verdict_free != 0; });
    *slot = __builtin_ctzll(g_verdict_free);
    g_verdict_free &= ~((uint64_t)1 << *slot);
    *word = g_verdict_mem + *slot * kVerdictStride;
    __atomic_store_n(*word, 0, __ATOMIC_RELAXED);
    return FLUTE_OK;
}
void give_verdict(int slot) {
    {
        std::lock_guard<std::mutex> lock(g_verdict_mu);
        g_verdict_free |= (uint64_t)1 << slot;
    }
    g_verdict_cv.notify_one();
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
    size_t lds = 0;
    if (w->signs) {
        if (w->rot_block > 0) {
            FLUTE_REQUIRE(is_pow2(w->rot_block) && w->rot_block >= 32 && w->rot_block <= 16384 &&
                              w->K % w->rot_block == 0,
                          FLUTE_ERR_INVALID,
                          "flute_embedding: rotation block must be a power of two in [32, 16384] "
                          "dividing K");
            lds = (size_t)(w->K <= 16384 ? w->K : (16384 / w->rot_block) * w->rot_block) * 4;
        } else {
            lds = (size_t)make_segments(w->K, 0).len[0] * 4;
        }
        static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
        if (!attr_done) {
            FLUTE_HIP_CHECK(hipFuncSetAttribute((const void *)embedding_kernel,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, 98304));
            attr_done = true;
        }
    }
    hipLaunchKernelGGL(embedding_kernel, dim3((unsigned)(count + (check ? 1 : 0))), dim3(kEmbThreads), lds, stream, p,
                       count, check);
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
    int slot = 0, *word = nullptr;
    flute_status st = take_verdict(&slot, &word);
    if (st != FLUTE_OK) return st;
    st = embedding(w, ids, count, out, stream, word);
    if (st != FLUTE_OK) {
        give_verdict(slot);                             // nothing was launched
        return st;
    }
    // The verdict comes from the grid's first workgroup, usually while the rows are still being
    // gathered; a stream that has much to do before it is waited for without spinning.
    int verdict = 0;
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    while (!(verdict = __atomic_load_n(word, __ATOMIC_ACQUIRE)) && std::chrono::steady_clock::now() < until)
        __builtin_ia32_pause();
    if (!verdict) {
        FLUTE_HIP_CHECK(hipStreamSynchronize(stream));
        verdict = __atomic_load_n(word, __ATOMIC_ACQUIRE);
        FLUTE_REQUIRE(verdict != 0, FLUTE_ERR_HIP, "flute_embedding_checked: the launch left no verdict");
    }
    give_verdict(slot);
    *in_range = verdict == 1;
    return FLUTE_OK;
}
