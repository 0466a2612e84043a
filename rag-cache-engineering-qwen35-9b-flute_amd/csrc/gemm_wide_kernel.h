// LUT GEMM for many rows:  C[M, N] = A[M, K] @ (W1 (+ W2))^T (+ xb @ resA^T) (+ bias),
// for up to four weights that share their number of rows and columns of A in one launch.
//
// A workgroup of eight wavefronts owns ROWS = 128 * MB rows of A and one 128-row tile of a weight,
// and every weight of a K tile is looked up ONCE per workgroup: the wavefronts turn an eighth of
// the tile's codes each into 16-bit values and write them to LDS in the order the matrix cores
// read them; then each takes all its operands from there against its own 16 * MB rows of A.  (The kernel of
// gemm_kernel.h looks a weight up once per 64 rows and wavefront; at many rows its lookups and
// their addresses, 2.3 instructions beside each matrix product, fill the issue port.  Here it is
// 1.1.)  The order of k inside a tile is free as long as both operands agree, and with the weights
// rearranged on their way through LDS it is the natural one.
//
// What bounds it (M = N = 4096, K = 12288): power.  Matrix instructions alone, in this structure,
// take 242 us of a sustained launch; the activations out of L2 (64 KB a tile) add 34 us, lookups
// and their stores 25 us, the weight operands out of LDS 9 us, each by lowering the clock: the
// matrix pipe is busy 93 % of the loop's cycles.  32x32x16 products reach 10 % less at the same
// power, and re-reading A straight from its rows costs the address path 64 cycles an instruction
// (sixteen rows) against 17 for an image in operand order, hence the image (wide_piece).
#pragma once

#include "gemm_common.h"

namespace flute {

constexpr int kWideMaxSegs = 4;

struct WideSeg {
    const uint8_t *q[2];
    const uint16_t *lut[2];
    const u4_t *Ap;        // activations in the LUT's 16-bit type as operands (wide_piece)
    const int *rowshift;   // [M] or NULL: row m of Ap holds the activations * 2^-rowshift[m]
    const float *xb;       // [M, R] residual coefficients (A @ resB^T) where R > 0
    const uint16_t *resA;  // [N, R] activation dtype
    const uint16_t *bias;  // [N] activation dtype or NULL
    void *C;
    int64_t ldc;
    int tile0;             // first tile of the launch that belongs to this weight
    int gs, lut_rows, R;
    int vec_store;         // C rows allow 16-byte stores
};

struct WideParams {
    WideSeg seg[kWideMaxSegs];
    int nsegs;
    int M, G;
    int mblk;              // 16-row blocks an image holds per half tile
    int mtiles, ntiles;    // units: ROWS rows by 128 outputs, over all weights
    int gper;              // K tiles per slice; gridDim.y slices
    int out_bf16;          // dtype of C, resA, bias
    float *P;              // [slice][unit] partial tiles where gridDim.y > 1
    int *tickets;
};

typedef const __attribute__((address_space(1))) uint8_t *GlobalBytes;
typedef const __attribute__((address_space(1))) u4_t *GlobalQuad;
typedef const __attribute__((address_space(1))) uint32_t *GlobalWord;

// One quarter (16 k) of a chunk: 4*B bytes.
template <int B>
__device__ __forceinline__ void wide_load_codes(uint32_t (&raw)[B], GlobalBytes p) {
    if constexpr (B == 4) {
        const u4_t v = __builtin_nontemporal_load((GlobalQuad)p);
        raw[0] = v[0]; raw[1] = v[1]; raw[2] = v[2]; raw[3] = v[3];
    } else {
#pragma unroll
        for (int i = 0; i < B; ++i) raw[i] = __builtin_nontemporal_load((GlobalWord)p + i);
    }
}

// The 8*B code bits of the four pairs (d, s2) of row quarter v, for v = 0 ... 3, then exchanged
// among the lanes: afterwards this lane holds the codes of its own row quarter v = lane >> 4 for
// the four chunks c = 0 ... 3 of a row, i.e. of eight consecutive k.
template <int B>
__device__ __forceinline__ void wide_spread_codes(uint32_t (&q)[4], const uint32_t (&raw)[B]) {
    if constexpr (B == 4) {
        q[0] = raw[0]; q[1] = raw[1]; q[2] = raw[2]; q[3] = raw[3];
    } else if constexpr (B == 3) {
        q[0] = raw[0];
        q[1] = __builtin_amdgcn_alignbit(raw[1], raw[0], 24);
        q[2] = __builtin_amdgcn_alignbit(raw[2], raw[1], 16);
        q[3] = raw[2] >> 8;
    } else if constexpr (B == 2) {
        q[0] = raw[0]; q[1] = raw[0] >> 16; q[2] = raw[1]; q[3] = raw[1] >> 16;
    } else {
        q[0] = raw[0]; q[1] = raw[0] >> 8; q[2] = raw[0] >> 16; q[3] = raw[0] >> 24;
    }
    transpose_lanes16(q);
}

// LDS: three buffers of one dequantised tile (16 KB each), then the pair tables of the streams: one
// entry of 32 dwords per pair code, split evenly over the LUT groups of the tile.
constexpr int kWideBuf = 16384, kWideEntryLog2 = 7;
template <int B1, int B2>
constexpr int wide_lds_bytes() {
    return 3 * kWideBuf + (((1 << (2 * B1)) + (B2 ? (1 << (2 * B2)) : 0)) << kWideEntryLog2);
}

template <bool BF16, int B1, int B2, int MB>
__global__ void __launch_bounds__(512, 2) gemm_wide_kernel(const WideParams p) {
    static_assert(MB == 4 || MB == 2, "64 or 32 rows per wavefront");
    extern __shared__ __align__(16) unsigned char smem[];
    typedef const __attribute__((address_space(3))) uint32_t *LdsWord;
    typedef __attribute__((address_space(3))) u4_t *LdsQuad;
    constexpr int NS = B2 > 0 ? 2 : 1;
    constexpr int SH = kWideEntryLog2;
    constexpr int ROWS = 128 * MB, NT = 512;
    constexpr bool WHOLE = MB == 2;                     // a product phase is a whole tile, not half a one
    using I1 = std::integral_constant<int, B1>;
    using I2 = std::integral_constant<int, B2 ? B2 : 1>;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // Unit of this workgroup: consecutive workgroups go to consecutive XCDs, so an XCD takes a
    // contiguous run of units, ordered in columns of four m tiles: what runs on it at a time
    // shares rows of A and tiles of W in its L2.
    int mt, nt;
    {
        const int units = p.mtiles * p.ntiles;
        const int xcd = blockIdx.x & 7, base = units >> 3, rem = units & 7;
        const int u = xcd * base + min(xcd, rem) + (blockIdx.x >> 3);
        const int col = 4 * p.ntiles;
        const int grp = u / col, in = u - grp * col;
        const int gm = min(4, p.mtiles - grp * 4);
        nt = in / gm;
        mt = grp * 4 + (in - nt * gm);
    }
    const int unit = mt * p.ntiles + nt;
    int si = 0;
    while (si + 1 < p.nsegs && nt >= p.seg[si + 1].tile0) ++si;
    const WideSeg &w = p.seg[si];
    const int t128 = nt - w.tile0;                      // tile of this weight
    const int g0 = blockIdx.y * p.gper, G = min(p.gper, p.G - g0);

    // ---- this lane's part of a tile's codes --------------------------------------------
    // (wavefronts w and w + 4 take the d = 0 and d = 1 rows of the same chunks)
    const int slice = wave & 3;
    const int c = lane >> 4, r = (lane >> 2) & 3, kt = lane & 3;
    const int th = slice * 16 + r * 4 + c;
    const int rowq = lane >> 4;                         // row quarter v after the exchange
    const uint64_t q1 = (uint64_t)(uintptr_t)w.q[0] + ((uint64_t)t128 * p.G + g0) * (1024 * B1);
    const uint64_t q2 = NS == 2 ? (uint64_t)(uintptr_t)w.q[1] + ((uint64_t)t128 * p.G + g0) * (1024 * B2) : 0;
    const uint32_t qofs1 = th * (16 * B1) + kt * (4 * B1), qofs2 = th * (16 * B2) + kt * (4 * B2);
    // tile g of stream s (past the end: the last tile again, so that every load is unconditional)
    auto load_codes = [&](auto bits, int s, auto &raw, int g) {
        constexpr int B = decltype(bits)::value;
        uint64_t t = (s ? q2 : q1) + (uint64_t)min(g, G - 1) * (1024 * B);
        asm volatile("" : "+s"(t));                     // keep it a scalar base plus a lane offset
        wide_load_codes<B>(raw, (GlobalBytes)t + (s ? qofs2 : qofs1));
    };
    const int odd = G & 1;                              // the loop of a single stream takes two tiles a turn
    uint32_t raw0[2][B1], raw1[2][B1], rawb[B2 ? B2 : 1], raw2[B2 ? B2 : 1];
    load_codes(I1(), 0, raw0[0], 0);
    if constexpr (NS == 1) load_codes(I1(), 0, raw0[1], 1);
    else load_codes(I2(), 1, rawb, 0);
    load_codes(I1(), 0, raw1[0], NS == 1 ? 3 : 1);

    // ---- pair tables -------------------------------------------------------------------
    const int gs = w.gs;
    const int ngrp = gs >= 128 ? 1 : 128 / gs;
    const int rep_log2 = SH - 2 - (31 - __builtin_clz(ngrp));     // dwords per entry and group
    // The LUT rows of the tile go to LDS first (the third buffer, written from the loop on only):
    // the entries then cost LDS reads, not a chain of trips to memory.
    uint16_t *const rows = (uint16_t *)(smem + 2 * kWideBuf);
    auto fetch_rows = [&](const uint16_t *lut, int b, uint16_t *to) {
        if (tid < ngrp << b) {
            int row = gs >= 128 ? (t128 * 128) / gs : t128 * ngrp + (tid >> b);
            row = min(row, w.lut_rows - 1);
            to[tid] = lut[((size_t)row << b) + (tid & ((1 << b) - 1))];
        }
    };
    fetch_rows(w.lut[0], B1, rows);
    if constexpr (NS == 2) fetch_rows(w.lut[1], B2, rows + 128);
    __syncthreads();
    auto build = [&](const uint16_t *lr, auto bits, uint32_t *tab) {
        constexpr int b = decltype(bits)::value;
        constexpr int quads = 1 << (2 * b + SH - 4);
#pragma unroll 4
        for (int i = tid; i < quads; i += NT) {
            const int code = i >> (SH - 4);
            const int word = (i & ((1 << (SH - 4)) - 1)) * 4;
            const uint16_t *row = lr + ((word >> rep_log2) << b);    // a group has four replicas or more
            const uint32_t v = (uint32_t)row[code & ((1 << b) - 1)] | ((uint32_t)row[code >> b] << 16);
            *(u4_t *)(tab + i * 4) = u4_t{v, v, v, v};
        }
    };
    uint32_t *const tab1 = (uint32_t *)(smem + 3 * kWideBuf);
    build(rows, I1(), tab1);
    if constexpr (NS == 2) build(rows + 128, I2(), tab1 + (1 << (2 * B1 + SH - 2)));

    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    // column of this lane in the tables: the LUT group of its rows (wx = slice >> 1, row quarter),
    // then the lane's replica
    const int my_group = ngrp == 1 ? 0 : (((slice >> 1) * 64 + rowq * 16) * ngrp) >> 7;
    uint32_t col[2];
    col[0] = lds0 + 3 * kWideBuf + (((my_group << rep_log2) + (lane & ((1 << rep_log2) - 1))) << 2);
    col[1] = col[0] + (1u << (2 * B1 + SH));

    // ---- where the weights go in a buffer ------------------------------------------------
    // Block (o, j) = 1 KB holds matrix operand (16 rows o, half j of the tile's k) in lane order;
    // row i of block o = pr*2 + blk is n = pr*32 + (i >> 2)*8 + blk*4 + (i & 3), so that the two
    // blocks of a pair give a lane eight consecutive outputs of C.  A slot's low three bits are
    // XORed with kt << 1 (kt = the 16-k quarter it belongs to): eight lanes that write together
    // then lie on different banks, and readers stay a permutation of 128 bytes.
    const uint32_t wofs = (uint32_t)(((slice >> 1) * 4 + (lane >> 5) * 2 + (slice & 1)) * 2 + (kt >> 1)) * 1024u;
    const int my_d = wave >> 2;
    const int wslot = (kt & 1) * 32 + ((lane >> 4) & 1) * 8 + my_d * 4 + r;
    const uint32_t waddr = lds0 + wofs + (uint32_t)((wslot ^ (kt << 1)) * 16);
    const int rslot = lane ^ ((lane >> 5) << 1);
    uint32_t raddr[2];
    raddr[0] = lds0 + (uint32_t)(rslot * 16);
    raddr[1] = lds0 + (uint32_t)((rslot ^ 4) * 16) + 1024u;

    // ---- activations ----------------------------------------------------------------------
    const int m0 = mt * ROWS + wave * (16 * MB);
    const uint64_t abase = (uint64_t)(uintptr_t)w.Ap + ((uint64_t)(2 * g0) * p.mblk + (m0 >> 4)) * 1024;
    u4_t A[2][2][MB];                                   // [set][half][block]; half-tile phases: one set
    auto load_a = [&](u4_t (&dst)[MB], int j, int g) {
        uint64_t ab = abase + (uint64_t)(2 * min(g, G - 1) + j) * p.mblk * 1024;
        asm volatile("" : "+s"(ab));
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) dst[mb] = *(GlobalQuad)((GlobalBytes)ab + (uint32_t)(lane * 16) + mb * 1024);
    };

    f4_t acc[MB][8];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[mb][i] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // ---- this wavefront's share of a tile: the pairs s2 = 0, 1 of one d ----------------------------
    uint32_t Q[4], addr[2][4];
    u4_t val[2];
    auto spread = [&](auto bits, const auto &raw) {
        constexpr int B = decltype(bits)::value;
        wide_spread_codes<B>(Q, raw);
#pragma unroll
        for (int i = 0; i < 4; ++i) Q[i] >>= my_d * 4 * B;
    };
    auto address = [&](auto bits, int s, int s2, int i) {
        constexpr int B = decltype(bits)::value;
        addr[s2][i] = (__builtin_amdgcn_ubfe(Q[i], 2 * B * s2, 2 * B) << SH) + col[s];
    };
    auto lookups = [&](int s2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) val[s2][i] = *(LdsWord)(uintptr_t)addr[s2][i];
    };
    auto put = [&](int s2, uint32_t buf) { *(LdsQuad)(uintptr_t)(waddr + buf + s2 * 256) = val[s2]; };

    __syncthreads();                                     // tables are in place

    // ---- first tiles -----------------------------------------------------------------------
    auto whole = [&](auto bits, int s, const auto &raw, uint32_t buf) {
        spread(bits, raw);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
#pragma unroll
            for (int i = 0; i < 4; ++i) address(bits, s, s2, i);
            lookups(s2);
            put(s2, buf);
        }
    };
    load_a(A[0][0], 0, 0);
    if constexpr (WHOLE) load_a(A[0][1], 1, 0);
    whole(I1(), 0, raw0[0], 0);
    if constexpr (NS == 1) {
        whole(I1(), 0, raw0[1], kWideBuf);
        uint32_t rawc[B1];
        load_codes(I1(), 0, rawc, 2);
        load_codes(I1(), 0, raw1[1], 3);
        spread(I1(), rawc);
    } else {
        whole(I2(), 1, rawb, kWideBuf);
        spread(I1(), raw1[0]);
        load_codes(I2(), 1, raw2, 1);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        address(I1(), 0, 0, i);
        if constexpr (WHOLE) address(I1(), 0, 1, i);
    }
    __syncthreads();

    // ---- the K loop ----------------------------------------------------------------------------
    // A step = one tile of one stream.  It is taken in load phases and product phases that
    // alternate: a load phase stores what the last one's lookups returned, fetches weight operands
    // from LDS, issues the lookups of a tile two steps ahead and loads activations; a product
    // phase is 32 matrix instructions that form the next lookups' addresses besides.  Wavefronts
    // w + 4 run one phase behind wavefronts w with a barrier after every phase, so the two
    // wavefronts of a SIMD take turns: one keeps the matrix pipe busy while the other loads.
    // With 64 rows per wavefront 32 products are half a tile (32 k), with 32 rows a tile.
    // Tile t lies in buffer t % 3.  Tile t + 2 is looked up during step t and stored one load phase
    // later each time, so its buffer's last reader (tile t - 1) is a step away, and so is its first.
    uint32_t rd = 0, wr = 2 * kWideBuf, wr_before = kWideBuf;
    u4_t W[WHOLE ? 16 : 8];
    auto phase_end = [&] {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto operands = [&](int j, u4_t *dst) {
        uint32_t from = raddr[j] + rd;
        asm volatile("" : "+v"(from));                  // opaque: the constant parts stay instruction offsets
#pragma unroll
        for (int o = 0; o < 8; ++o) dst[o] = *(LdsQuad)(uintptr_t)(from + o * 2048u);
    };
    // MB products: block o against the blocks of rows, back and forth: of two neighbouring
    // instructions one operand stays the same (2 % more products at the same power in a loop of
    // nothing else)
    auto products = [&](int o, const u4_t &wo, const u4_t (&Aj)[MB]) {
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const int mb = (o & 1) ? MB - 1 - i : i;
            acc[mb][o] = mfma16<BF16>(wo, Aj[mb], acc[mb][o]);
        }
    };
    auto turn = [&] {
        wr_before = wr;
        rd = rd == 2 * kWideBuf ? 0u : rd + kWideBuf;
        wr = wr == 2 * kWideBuf ? 0u : wr + kWideBuf;
    };
    // MB = 4, half j of a step: what to load beside the operands, and what the product phase
    // prepares for the next half's lookups: `first` once, then `then(i)` for i = 0 ... 3
    auto half = [&](int j, auto load_more, auto first, auto then) {
        put(1 - j, j ? wr : wr_before);                 // (the very first one stores tile 1's last piece again)
        operands(j, W);
        __builtin_amdgcn_sched_barrier(0);
        lookups(j);
        load_more();
        __builtin_amdgcn_sched_barrier(0);
        // the operands are here (LDS answers in order: everything older too), the lookups may be out
        asm volatile("s_waitcnt lgkmcnt(4)" ::: "memory");
        phase_end();
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int o = 0; o < 8; ++o) {
            products(o, W[o], A[0][j]);
            if (o == 3) first();
            if (o >= 4) then(o - 4);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        phase_end();
    };
    // MB = 2, a whole step with the activations of `now`
    auto full = [&](u4_t (&now)[2][MB], auto load_more, auto first, auto then) {
        put(0, wr_before);                              // (the very first one stores tile 1 again)
        put(1, wr_before);
        operands(0, W);
        operands(1, W + 8);
        __builtin_amdgcn_sched_barrier(0);
        lookups(0);
        lookups(1);
        load_more();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(8)" ::: "memory");
        phase_end();
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int o = 0; o < 16; ++o) {
            products(o & 7, W[o], now[o >> 3]);
            if (o == 3) first();
            if (o >= 4 && !(o & 1) && o < 12) then((o - 4) >> 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        phase_end();
        turn();
    };
    if (wave >= 4) phase_end();                          // one phase behind
    if constexpr (!WHOLE && NS == 1) {
        auto step = [&](auto &raw, auto &other, int t) {
            half(0, [&] {
                load_a(A[0][1], 1, t);
                load_codes(I1(), 0, raw, t + 4);
            }, [] {}, [&](int i) { address(I1(), 0, 1, i); });
            half(1, [&] { load_a(A[0][0], 0, t + 1); }, [&] { spread(I1(), other); },
                 [&](int i) { address(I1(), 0, 0, i); });
            turn();
        };
        int t = 0;
        if (odd) {
            step(raw1[1], raw1[0], 0);
            t = 1;
        }
        for (; t < G; t += 2) {
            step(raw1[0], raw1[1], t);
            step(raw1[1], raw1[0], t + 1);
        }
    } else if constexpr (!WHOLE) {
        for (int g = 0; g < G; ++g) {
            half(0, [&] {
                load_a(A[0][1], 1, g);
                load_codes(I1(), 0, raw1[0], g + 2);
            }, [] {}, [&](int i) { address(I1(), 0, 1, i); });
            half(1, [&] {}, [&] { spread(I2(), raw2); }, [&](int i) { address(I2(), 1, 0, i); });
            turn();
            half(0, [&] { load_codes(I2(), 1, raw2, g + 2); }, [] {}, [&](int i) { address(I2(), 1, 1, i); });
            half(1, [&] { load_a(A[0][0], 0, g + 1); }, [&] { spread(I1(), raw1[0]); },
                 [&](int i) { address(I1(), 0, 0, i); });
            turn();
        }
    } else if constexpr (NS == 1) {
        auto step = [&](auto &now, auto &next, auto &raw, auto &other, int t) {
            full(now, [&] {
                load_a(next[0], 0, t + 1);
                load_a(next[1], 1, t + 1);
                load_codes(I1(), 0, raw, t + 4);
            }, [&] { spread(I1(), other); }, [&](int i) {
                address(I1(), 0, 0, i);
                address(I1(), 0, 1, i);
            });
        };
        int t = 0;
        if (odd) {
            step(A[0], A[1], raw1[1], raw1[0], 0);
            t = 1;
            for (; t < G; t += 2) {
                step(A[1], A[0], raw1[0], raw1[1], t);
                step(A[0], A[1], raw1[1], raw1[0], t + 1);
            }
        } else {
            for (; t < G; t += 2) {
                step(A[0], A[1], raw1[0], raw1[1], t);
                step(A[1], A[0], raw1[1], raw1[0], t + 1);
            }
        }
    } else {
        auto both = [&](auto &now, auto &next, int g) {
            full(now, [&] {
                load_a(next[0], 0, g + 1);
                load_codes(I1(), 0, raw1[0], g + 2);
            }, [&] { spread(I2(), raw2); }, [&](int i) {
                address(I2(), 1, 0, i);
                address(I2(), 1, 1, i);
            });
            full(now, [&] {
                load_a(next[1], 1, g + 1);
                load_codes(I2(), 1, raw2, g + 2);
            }, [&] { spread(I1(), raw1[0]); }, [&](int i) {
                address(I1(), 0, 0, i);
                address(I1(), 0, 1, i);
            });
        };
        int g = 0;
        for (; g + 1 < G; g += 2) {
            both(A[0], A[1], g);
            both(A[1], A[0], g + 1);
        }
        if (g < G) both(A[0], A[1], g);
    }
    if (wave < 4) phase_end();                           // as many barriers as the others

    // ---- K slices: partial tiles in register order; the last arrival adds them in slice order --------
    const int rho = lane & 15, kg = lane >> 4;
    if (gridDim.y > 1) {
        const int z = blockIdx.y, Z = gridDim.y;
        const size_t image = (size_t)ROWS * 128, zstride = (size_t)p.mtiles * p.ntiles * image;
        float *const mine = p.P + (size_t)unit * image + tid * 4;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int i = 0; i < 8; ++i) ws_store16(mine + z * zstride + (mb * 8 + i) * (NT * 4), acc[mb][i]);
        ws_stores_done();
        __syncthreads();
        int *flag = (int *)smem;                         // the tile buffers are dead
        if (tid == 0) {
            const int old = __hip_atomic_fetch_add(p.tickets + unit, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *flag = old == Z - 1;
            if (old == Z - 1)
                __hip_atomic_store(p.tickets + unit, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!*flag) return;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            f4_t sum[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) sum[i] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
            for (int zz = 0; zz < Z; ++zz) {
                if (zz == z) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) sum[i] += acc[mb][i];
                } else {
                    // read around the caches of this XCD, all eight blocks in flight
                    f4_t got[8];
                    ws_load16x8(mine + zz * zstride + mb * 8 * (NT * 4), NT * 4, got);
#pragma unroll
                    for (int i = 0; i < 8; ++i) sum[i] += got[i];
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[mb][i] = sum[i];
        }
    }

    // ---- epilogue: scale back, residual, bias, one rounding, store ----------------------------
    if (w.rowshift) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int sh = w.rowshift[min(m0 + mb * 16 + rho, p.M - 1)];
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[mb][i][e] = ldexpf(acc[mb][i][e], sh);
        }
    }
    if (w.R > 0) {
        // + xb @ resA^T, the fp32 coefficients as they are: fp32 matrix products onto the sums, sixteen
        // ranks a step, of which lane group kg holds four (the order of ranks is free as long as both
        // operands agree).  resA is read once for all the rows of a wavefront.  (As three 16-bit terms of
        // rows scaled to [1, 2), which in float16 lost the low bits of all but a row's largest
        // coefficients: M = 1000, 4096 -> 12288, (1, 4) bits, rank 16, 191 us a forward against 171.)
        const bool vec = w.R % 4 == 0 && ((uintptr_t)w.resA & 7) == 0 && ((uintptr_t)w.xb & 15) == 0;
#pragma unroll 1
        for (int r0 = 0; r0 < w.R; r0 += 16) {
            const int k0 = r0 + kg * 4;
            float a[8][4];
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const int n = t128 * 128 + (o >> 1) * 32 + (rho >> 2) * 8 + (o & 1) * 4 + (rho & 3);
                const uint16_t *const row = w.resA + (size_t)n * w.R;
                uint32_t h[2] = {0u, 0u};
                if (vec) {
                    if (k0 < w.R) {
                        const uint2 raw = *(const uint2 *)(row + k0);
                        h[0] = raw.x;
                        h[1] = raw.y;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (k0 + e < w.R) h[e >> 1] |= (uint32_t)row[k0 + e] << (16 * (e & 1));
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint16_t one = (uint16_t)(h[e >> 1] >> (16 * (e & 1)));
                    a[o][e] = p.out_bf16 ? bf2f(one) : h2f(one);
                }
            }
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const float *const row = w.xb + (size_t)min(m0 + mb * 16 + rho, p.M - 1) * w.R;
                f4_t x = {0.0f, 0.0f, 0.0f, 0.0f};
                if (vec) {
                    if (k0 < w.R) x = *(const f4_t *)(row + k0);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (k0 + e < w.R) x[e] = row[k0 + e];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int o = 0; o < 8; ++o)
                        acc[mb][o] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[o][e], x[e], acc[mb][o], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int pr = 0; pr < 4; ++pr) {
        const int n0 = t128 * 128 + pr * 32 + kg * 8;
        float bias[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) bias[e] = 0.0f;
        if (w.bias) {
#pragma unroll
            for (int e = 0; e < 8; ++e) bias[e] = load_act(w.bias, n0 + e, p.out_bf16);
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int m = m0 + mb * 16 + rho;
            if (m >= p.M) continue;
            float y[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[e] = acc[mb][2 * pr][e] + bias[e];
                y[4 + e] = acc[mb][2 * pr + 1][e] + bias[4 + e];
            }
            uint32_t o[4];
            if (p.out_bf16) {
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (uint32_t)f2bf(y[2 * e]) | ((uint32_t)f2bf(y[2 * e + 1]) << 16);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (uint32_t)f2h(y[2 * e]) | ((uint32_t)f2h(y[2 * e + 1]) << 16);
            }
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
    }
}

}  // namespace flute
