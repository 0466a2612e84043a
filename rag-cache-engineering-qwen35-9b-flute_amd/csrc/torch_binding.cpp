// flute_extended._C_native: the decode and prefill entry points of the operator surface as a
// compiled PyTorch-ROCm extension over the C ABI (include/flute_hip.h).  Upstream builds its
// kernels into a pybind11 module `flute_extended._C` (src/bindings.cpp:230-546); this file is
// that module's counterpart for the entries an eager decode loop calls per token:
//
//   qgemm_gemv_stream, qgemm_gemv_fht_stream, qgemm_gemv_splitk_stream,
//   qgemm_gemv_splitk_fht_stream            (src/bindings.cpp:277-354)
//   qgemm_gemv_multi, qgemm_gemv_mlp        (src/bindings.cpp:368-384)
//   qgemm_cutlass_streaming, qgemm_dual_stream   (src/bindings.cpp:245-270)
//   qgemm_linear, qgemm_linear_multi, qgemm_linear_mlp, embedding_rows, operand_addresses
//                                           (what a module's forward calls; no upstream counterpart)
//   Forwards                                (the forwards of the module layer themselves, for the calls that
//                                           need nothing but the library)
//
// Same positional signatures, same conventions (empty tensor = absent operand, N from the
// blob's byte count, RuntimeError on every contract violation, fresh outputs, launches on the
// current stream of the input's device) and the same checks, in the same order and with the
// same messages, as the ctypes mirror in flute_extended/_C.py, which stays the binding for
// everything else and the fallback when this module is not built.  Host code only: nothing
// here runs on the device, the kernels are in libflute_hip.so.
#include <torch/extension.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <cstring>
#include <functional>
#include <map>
#include <sstream>
#include <string>
#include <vector>

#include "flute_hip.h"

namespace {

using torch::Tensor;

int act_code(const Tensor &t) { return t.scalar_type() == at::kBFloat16 ? FLUTE_BF16 : FLUTE_F16; }
bool is_act(const Tensor &t) {
    return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16;
}
// the name Python prints for a dtype
const char *dtype_name(const Tensor &t) {
    switch (t.scalar_type()) {
        case at::kBFloat16: return "torch.bfloat16";
        case at::kHalf: return "torch.float16";
        case at::kFloat: return "torch.float32";
        case at::kDouble: return "torch.float64";
        case at::kByte: return "torch.uint8";
        case at::kChar: return "torch.int8";
        case at::kShort: return "torch.int16";
        case at::kInt: return "torch.int32";
        case at::kLong: return "torch.int64";
        case at::kBool: return "torch.bool";
        default: return c10::toString(t.scalar_type());
    }
}

void *stream_of(const Tensor &t) {
    return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}
Tensor aligned16(const Tensor &t) {
    // fresh allocations are 256-byte aligned; views and slices may not be
    return ((uintptr_t)t.data_ptr() % 16 == 0) ? t : t.clone();
}
void check_status(flute_status st) {
    TORCH_CHECK(st == FLUTE_OK, flute_last_error());
}

struct Shape2 {
    int64_t M, K;
};

// What the library's argument checks need to know about a tensor (flute_tensor): no tensor
// type crosses the C ABI.  `name` keeps the printed dtype alive for the duration of the call.
struct Record {
    flute_tensor t = {};
    std::string name;
};
void record(Record &r, const Tensor *t) {
    if (t == nullptr || !t->defined()) {
        r.t.present = 0;
        return;
    }
    r.t.present = 1;
    r.t.numel = t->numel();
    r.t.ndim = (int32_t)t->dim();
    for (int64_t i = 0; i < t->dim() && i < 4; ++i) r.t.size[i] = t->size(i);
    switch (t->scalar_type()) {
        case at::kHalf: r.t.dtype = FLUTE_F16; break;
        case at::kBFloat16: r.t.dtype = FLUTE_BF16; break;
        case at::kFloat: r.t.dtype = FLUTE_F32; break;
        case at::kByte: r.t.dtype = FLUTE_U8; break;
        default:
            r.t.dtype = -1;
            r.name = dtype_name(*t);
            r.t.dtype_name = r.name.c_str();
    }
    r.t.contiguous = t->is_contiguous() ? 1 : 0;
    r.t.device = t->is_cuda() ? (int32_t)t->device().index() : -1;
    r.t.data = t->numel() ? t->data_ptr() : nullptr;
}

// The checks of the input matrix: flute_check_input (one copy for this binding and the ctypes
// mirror).
Shape2 check_2d_input(const char *who, const Tensor &A, bool need_m1) {
    Record r;
    record(r, &A);
    check_status(flute_check_input(who, &r.t, need_m1 ? 1 : 0));
    return {A.size(0), A.size(1)};
}

struct Described {
    flute_linear w;
    int64_t N;
    Tensor keep1, keep2;    // re-aligned blobs, alive until the launch is queued
};

uint32_t gs_mask(const std::vector<int> &allowed) {
    uint32_t m = 0;
    for (int g : allowed) m |= 1u << (31 - __builtin_clz((unsigned)g));
    return m;
}

const std::vector<int> kGsAll = {16, 32, 64, 128, 256, 512, 1024, 2048};
const std::vector<int> kGsPlain = {64, 128, 256, 512, 1024, 2048};

// The checks of one weight's tensors: flute_describe_linear; this function records what it was
// handed and re-aligns blobs that torch may hand over as views.
Described describe(const char *who, const Tensor &A, int64_t K, const Tensor &indices,
                   const Tensor &lut, int64_t b1, const Tensor &indices2, const Tensor &lut2,
                   int64_t b2, const Tensor &resB, const Tensor &resA, const Tensor &bias,
                   int64_t gs, const c10::optional<Tensor> &signs, c10::optional<Tensor> awq,
                   int64_t rot_block, const std::vector<int> &gs_allowed, int64_t max_rank) {
    Described d;
    d.keep1 = (indices.defined() && indices.is_cuda()) ? aligned16(indices) : indices;
    d.keep2 = (b2 > 0 && indices2.defined() && indices2.is_cuda()) ? aligned16(indices2) : indices2;
    Record rA, rI, rL, rI2, rL2, rRB, rRA, rBias, rS, rAwq;
    record(rA, &A);
    record(rI, &d.keep1);
    record(rL, &lut);
    record(rI2, &d.keep2);
    record(rL2, &lut2);
    record(rRB, &resB);
    record(rRA, &resA);
    record(rBias, &bias);
    record(rS, signs.has_value() ? &*signs : nullptr);
    record(rAwq, awq.has_value() ? &*awq : nullptr);
    flute_operands ops = {};
    ops.A = rA.t;
    ops.indices = rI.t;
    ops.lut = rL.t;
    ops.indices2 = rI2.t;
    ops.lut2 = rL2.t;
    ops.resB = rRB.t;
    ops.resA = rRA.t;
    ops.bias = rBias.t;
    ops.signs = rS.t;
    ops.awq = rAwq.t;
    ops.K = K;
    ops.b1 = (int32_t)b1;
    ops.b2 = (int32_t)b2;
    ops.group_size = (gs >= INT32_MIN && gs <= INT32_MAX) ? (int32_t)gs : -1;
    ops.rot_block = (int32_t)rot_block;
    ops.max_rank = (int32_t)max_rank;
    ops.gs_allowed = gs_mask(gs_allowed);
    check_status(flute_describe_linear(who, &ops, &d.w, &d.N));
    return d;
}

Tensor gemv(const char *who, const Tensor &A_in, const Tensor &indices, const Tensor &lut,
            int64_t b1, const Tensor &indices2, const Tensor &lut2, int64_t b2, const Tensor &resB,
            const Tensor &resA, const Tensor &bias, int64_t gs,
            const c10::optional<Tensor> &signs, const c10::optional<Tensor> &awq, int64_t split,
            int64_t rot_block, const std::vector<int> &gs_allowed, int64_t max_rank) {
    const Shape2 s = check_2d_input(who, A_in, true);
    if (s.K == 0 || indices.numel() == 0) {
        // degenerate shapes never reach the device (src/kernel_gemv.cu:456-461 upstream)
        const int64_t N = (s.K == 0 && lut.dim() == 2) ? lut.size(0) * gs : 0;
        return torch::zeros({1, N}, A_in.options());
    }
    Described d = describe(who, A_in, s.K, indices, lut, b1, indices2, lut2, b2, resB, resA, bias,
                           gs, signs, awq, rot_block, gs_allowed, max_rank);
    const Tensor A = aligned16(A_in);
    c10::DeviceGuard guard(A.device());
    Tensor C = torch::empty({1, d.N}, A.options());
    check_status(flute_gemv(&d.w, A.data_ptr(), C.data_ptr(), act_code(A), (int)split, stream_of(A)));
    return C;
}

Tensor gemm(const char *who, const Tensor &A_in, const Tensor &indices, const Tensor &lut,
            int64_t b1, const Tensor &indices2, const Tensor &lut2, int64_t b2, const Tensor &resB,
            const Tensor &resA, const Tensor &bias, int64_t gs,
            const c10::optional<Tensor> &signs = c10::nullopt,
            const c10::optional<Tensor> &awq = c10::nullopt) {
    const Shape2 s = check_2d_input(who, A_in, false);
    if (s.K == 0 || s.M == 0 || indices.numel() == 0) {
        const int64_t rb = (s.K * b1) / 8;
        const int64_t N = s.K == 0 ? 0 : indices.numel() / (rb > 1 ? rb : 1);
        return torch::zeros({s.M, N}, A_in.options());
    }
    Described d = describe(who, A_in, s.K, indices, lut, b1, indices2, lut2, b2, resB, resA, bias,
                           gs, signs, awq, 0, kGsAll, 256);
    const Tensor A = aligned16(A_in);
    c10::DeviceGuard guard(A.device());
    Tensor C = torch::empty({s.M, d.N}, A.options());
    check_status(flute_gemm(&d.w, A.data_ptr(), C.data_ptr(), (int)s.M, s.K, d.N, act_code(A),
                            stream_of(A)));
    return C;
}

// ---- M = 1 GEMV family --------------------------------------------------------------

Tensor qgemm_gemv_stream(const Tensor &A, const Tensor &indices, const Tensor &lut, int64_t b1,
                         const Tensor &indices2, const Tensor &lut2, int64_t b2,
                         const Tensor &resB, const Tensor &resA, const Tensor &bias, int64_t gs) {
    return gemv("qgemm_gemv_stream", A, indices, lut, b1, indices2, lut2, b2, resB, resA, bias, gs,
                c10::nullopt, c10::nullopt, 0, 0, kGsPlain, 16);
}

Tensor qgemm_gemv_fht_stream(const Tensor &A, const Tensor &indices, const Tensor &lut, int64_t b1,
                             const Tensor &indices2, const Tensor &lut2, int64_t b2,
                             const Tensor &resB, const Tensor &resA, const Tensor &bias, int64_t gs,
                             const c10::optional<Tensor> &signs, const c10::optional<Tensor> &s) {
    return gemv("qgemm_gemv_fht_stream", A, indices, lut, b1, indices2, lut2, b2, resB, resA, bias,
                gs, signs, s, 0, 0, kGsPlain, 16);
}

Tensor qgemm_gemv_splitk_stream(const Tensor &A, const Tensor &indices, const Tensor &lut,
                                int64_t b1, const Tensor &indices2, const Tensor &lut2, int64_t b2,
                                const Tensor &resB, const Tensor &resA, const Tensor &bias,
                                int64_t gs, int64_t split) {
    return gemv("qgemm_gemv_splitk_stream", A, indices, lut, b1, indices2, lut2, b2, resB, resA,
                bias, gs, c10::nullopt, c10::nullopt, split, 0, kGsAll, 256);
}

Tensor qgemm_gemv_splitk_fht_stream(const Tensor &A, const Tensor &indices, const Tensor &lut,
                                    int64_t b1, const Tensor &indices2, const Tensor &lut2,
                                    int64_t b2, const Tensor &resB, const Tensor &resA,
                                    const Tensor &bias, int64_t gs,
                                    const c10::optional<Tensor> &signs,
                                    const c10::optional<Tensor> &s, int64_t split,
                                    int64_t rot_block) {
    return gemv("qgemm_gemv_splitk_fht_stream", A, indices, lut, b1, indices2, lut2, b2, resB, resA,
                bias, gs, signs, s, split, rot_block, kGsAll, 256);
}

// ---- segment-table entries -----------------------------------------------------------

constexpr int kSegCols = 15;   // q1 lut1 q2 lut2 resB resA bias C N R b1 b2 gs signs s

int64_t check_seg_inputs(const char *who, const Tensor &A, const Tensor &seg_table, int64_t rows) {
    TORCH_CHECK(A.dim() == 2 && A.size(0) == 1 && is_act(A) && A.is_contiguous(), who,
                ": A must be a contiguous [1, K] float16/bfloat16 tensor");
    TORCH_CHECK(seg_table.device().is_cpu() && seg_table.scalar_type() == at::kLong &&
                    seg_table.dim() == 2 && seg_table.size(1) == kSegCols,
                who, ": seg_table must be a CPU int64 [count, 15] tensor");
    const int64_t count = seg_table.size(0);
    TORCH_CHECK(rows < 0 || count == rows, who, ": seg_table must have ", rows, " rows (got ",
                count, ")");
    TORCH_CHECK(rows >= 0 || (count >= 1 && count <= 4), who,
                ": 1..4 segments per launch (got ", count, ")");
    return count;
}

void seg_descs(const char *who, const Tensor &A, const Tensor &seg_table, int lut_dtype,
               std::vector<flute_linear> &descs, std::vector<void *> &outs) {
    const int64_t K = A.size(1);
    const Tensor table = seg_table.contiguous();
    const int64_t *v = table.data_ptr<int64_t>();
    const int64_t count = table.size(0);
    descs.assign(count, flute_linear{});
    outs.assign(count, nullptr);
    static const char *names[] = {"q1", "q2", "resB", "resA", "signs", "s"};
    static const int cols[] = {0, 2, 4, 5, 13, 14};
    for (int64_t i = 0; i < count; ++i) {
        const int64_t *r = v + i * kSegCols;
        for (int c = 0; c < 6; ++c)
            TORCH_CHECK(r[cols[c]] % 16 == 0, who, ": segment ", i, " pointer ", names[c],
                        " must be 16-byte aligned");
        TORCH_CHECK(r[0] != 0 && r[1] != 0, who, ": segment ", i, " has no stream-1 indices/lut");
        TORCH_CHECK(r[12] > 0, who, ": segment ", i, " group_size must be positive");
        flute_linear &w = descs[i];
        const int64_t N = r[8], R = r[9], b1 = r[10], b2 = r[11], gs = r[12];
        w.q1 = (const void *)r[0];
        w.lut1 = (const void *)r[1];
        w.q2 = (const void *)r[2];
        w.lut2 = (const void *)r[3];
        w.resB = (const void *)r[4];
        w.resA = (const void *)r[5];
        w.bias = (const void *)r[6];
        w.signs = (const float *)r[13];
        w.awq = (const float *)r[14];
        w.N = (int)N;
        w.K = (int)K;
        w.R = (int)R;
        w.b1 = (int)b1;
        w.b2 = (int)b2;
        w.group_size = (int)gs;
        w.q1_bytes = N * K * b1 / 8;
        w.q2_bytes = N * K * b2 / 8;
        w.lut_rows = (int)((N + gs - 1) / gs);
        w.lut_dtype = lut_dtype;
        outs[i] = (void *)r[7];
    }
}

// lut_dtype: None (float16) or a torch.dtype
int lut_code(const pybind11::object &lut_dtype) {
    if (lut_dtype.is_none()) return FLUTE_F16;
    return lut_dtype.is(pybind11::module_::import("torch").attr("bfloat16")) ? FLUTE_BF16 : FLUTE_F16;
}

void gemv_multi_table(const Tensor &A_in, const Tensor &seg_table, int lut, int64_t split) {
    const char *who = "qgemm_gemv_multi";
    check_seg_inputs(who, A_in, seg_table, -1);
    TORCH_CHECK(A_in.is_cuda(), who, ": A must be a CUDA (HIP) tensor");
    std::vector<flute_linear> descs;
    std::vector<void *> outs;
    seg_descs(who, A_in, seg_table, lut, descs, outs);
    for (size_t i = 0; i < outs.size(); ++i)
        TORCH_CHECK(outs[i] != nullptr, who, ": segment ", i, " has no output pointer");
    const Tensor A = aligned16(A_in);
    c10::DeviceGuard guard(A.device());
    check_status(flute_gemv_multi(descs.data(), (int)descs.size(), A.data_ptr(), outs.data(),
                                  act_code(A), (int)split, stream_of(A)));
}

void qgemm_gemv_multi(const Tensor &A, const Tensor &seg_table, const pybind11::object &lut_dtype, int64_t split) {
    gemv_multi_table(A, seg_table, lut_code(lut_dtype), split);
}

Tensor gemv_mlp_table(const Tensor &A_in, const Tensor &seg_table, const Tensor &C, int lut, int64_t split) {
    const char *who = "qgemm_gemv_mlp";
    check_seg_inputs(who, A_in, seg_table, 2);
    TORCH_CHECK(C.scalar_type() == A_in.scalar_type() && C.is_contiguous(), who,
                ": C must be a contiguous ", dtype_name(A_in), " output buffer");
    const Tensor table = seg_table.contiguous();   // alive while v is read
    const int64_t *v = table.data_ptr<int64_t>();
    const int64_t N = v[8];
    TORCH_CHECK(v[kSegCols + 8] == N && C.numel() == N, who, ": gate/up/C must agree in N");
    TORCH_CHECK(A_in.is_cuda() && C.is_cuda(), who, ": A and C must be CUDA (HIP) tensors");
    TORCH_CHECK(C.device() == A_in.device(), who, ": C must live on A's device ",
                A_in.device().str());
    std::vector<flute_linear> descs;
    std::vector<void *> outs;
    seg_descs(who, A_in, seg_table, lut, descs, outs);
    const Tensor A = aligned16(A_in);
    c10::DeviceGuard guard(A.device());
    check_status(flute_gemv_mlp(&descs[0], &descs[1], A.data_ptr(), C.data_ptr(), act_code(A),
                                (int)split, stream_of(A)));
    return C;
}

Tensor qgemm_gemv_mlp(const Tensor &A, const Tensor &seg_table, const Tensor &C, const pybind11::object &lut_dtype,
                      int64_t split) {
    return gemv_mlp_table(A, seg_table, C, lut_code(lut_dtype), split);
}

// ---- GEMM family ------------------------------------------------------------------------

Tensor qgemm_cutlass_streaming(const Tensor &A, const Tensor &indices, const Tensor &lut,
                               int64_t b1, int64_t gs, int64_t q_layout) {
    TORCH_CHECK(q_layout == 1, "qgemm_cutlass_streaming: only q_layout=1 (the idxN blob) is served");
    const Tensor e8 = torch::empty({0}, A.options().dtype(at::kByte));
    const Tensor e16 = torch::empty({0}, A.options());
    return gemm("qgemm_cutlass_streaming", A, indices, lut, b1, e8, e16, 0, e16, e16, e16, gs);
}

Tensor qgemm_dual_stream(const Tensor &A, const Tensor &indices, const Tensor &lut, int64_t b1,
                         const Tensor &indices2, const Tensor &lut2, int64_t b2,
                         const Tensor &resB, const Tensor &resA, const Tensor &bias, int64_t gs) {
    return gemm("qgemm_dual_stream", A, indices, lut, b1, indices2, lut2, b2, resB, resA, bias, gs);
}

// ---- one call per module forward ----------------------------------------------------------

Tensor qgemm_linear(const Tensor &A, const Tensor &indices, const Tensor &lut, int64_t b1,
                    const c10::optional<Tensor> &indices2, const c10::optional<Tensor> &lut2, int64_t b2,
                    const c10::optional<Tensor> &resB, const c10::optional<Tensor> &resA,
                    const c10::optional<Tensor> &bias, int64_t gs, const c10::optional<Tensor> &signs,
                    const c10::optional<Tensor> &awq) {
    const auto held = [](const c10::optional<Tensor> &t) { return t.has_value() ? *t : Tensor(); };
    if (A.dim() == 2 && A.size(0) == 1)
        return gemv("qgemm_linear", A, indices, lut, b1, held(indices2), held(lut2), b2, held(resB), held(resA),
                    held(bias), gs, signs, awq, 0, 0, kGsAll, 256);
    return gemm("qgemm_linear", A, indices, lut, b1, held(indices2), held(lut2), b2, held(resB), held(resA),
                held(bias), gs, signs, awq);
}

// The layers of a call on several rows, each (indices, lut, b1, indices2, lut2, b2, resB, resA, bias, gs,
// signs, s) with None for what it has not.
Described described(const char *who, const Tensor &A, int64_t K, const pybind11::tuple &l) {
    const auto opt = [](const pybind11::handle &h) {
        return h.is_none() ? c10::optional<Tensor>() : c10::optional<Tensor>(h.cast<Tensor>());
    };
    const auto held = [](const pybind11::handle &h) { return h.is_none() ? Tensor() : h.cast<Tensor>(); };
    TORCH_CHECK(l.size() == 12, who, ": a layer has 12 operands");
    return describe(who, A, K, l[0].cast<Tensor>(), l[1].cast<Tensor>(), l[2].cast<int64_t>(), held(l[3]), held(l[4]),
                    l[5].cast<int64_t>(), held(l[6]), held(l[7]), held(l[8]), l[9].cast<int64_t>(), opt(l[10]), opt(l[11]),
                    0, kGsAll, 256);
}

std::vector<Described> described_all(const char *who, const Tensor &A, int64_t K, const std::vector<pybind11::tuple> &layers,
                                     size_t count) {
    std::vector<Described> d;
    for (size_t i = 0; i < count; ++i) d.push_back(described(who, A, K, layers[i]));
    return d;
}

// Layers on the rows of A: outputs of one row side by side, or one below the other (`stacked`, layers of
// equal N).
Tensor gemm_layers(const char *who, const Tensor &A, const Shape2 &s, const std::vector<Described> &d, bool stacked) {
    std::vector<flute_linear> ws;
    int64_t total = 0;
    for (const Described &one : d) {
        ws.push_back(one.w);
        total += one.N;
    }
    TORCH_CHECK(!stacked || d[0].N == d[1].N, who, ": gate and up must agree in N");
    const Tensor out = stacked ? torch::empty({2, s.M, d[0].N}, A.options()) : torch::empty({s.M, total}, A.options());
    std::vector<void *> C;
    std::vector<int64_t> ldc;
    char *at = (char *)out.data_ptr();
    for (const Described &one : d) {
        C.push_back(at);
        at += 2 * one.N * (stacked ? s.M : 1);
        ldc.push_back(stacked ? one.N : total);
    }
    check_status(flute_gemm_multi(ws.data(), (int)ws.size(), A.data_ptr(), C.data(), ldc.data(), (int)s.M, s.K, act_code(A),
                                  stream_of(A)));
    return out;
}

// silu(first) * second of two stacked outputs.
Tensor gated(const Tensor &out, const Tensor &A) {
    const Tensor g = out.select(0, 0), u = out.select(0, 1), h = torch::empty_like(g);
    check_status(flute_silu_mul(g.data_ptr(), u.data_ptr(), h.data_ptr(), g.numel(), act_code(A), stream_of(A)));
    return h;
}

// Several layers on the same rows: their outputs side by side, or silu(first) * second.
// Layers of one rotation (the same signs and s at the same address) share the rotated rows.
Tensor qgemm_linear_multi(const Tensor &A_in, const std::vector<pybind11::tuple> &layers, bool silu_mul) {
    const char *who = "qgemm_linear_multi";
    const Shape2 s = check_2d_input(who, A_in, false);
    TORCH_CHECK(!layers.empty() && layers.size() <= 4 && (!silu_mul || layers.size() == 2), who,
                ": 1..4 layers, two for silu_mul");
    const Tensor A = aligned16(A_in);
    c10::DeviceGuard guard(A.device());
    const Tensor out = gemm_layers(who, A, s, described_all(who, A, s.K, layers, layers.size()), silu_mul);
    return silu_mul ? gated(out, A) : out;
}

// down of the gated product of stacked gate and up outputs.
Tensor gated_down(const Tensor &out, const Described &d) {
    const Tensor g = out.select(0, 0), u = out.select(0, 1);
    const int64_t M = g.size(0), K = g.size(1);
    const Tensor C = torch::empty({M, d.N}, g.options());
    const int act = act_code(g);
    void *const stream = stream_of(g);
    if (flute_gemm_takes_silu(&d.w, (int)M, act)) {
        check_status(flute_gemm_silu(&d.w, g.data_ptr(), u.data_ptr(), C.data_ptr(), (int)M, K, d.N, act, stream));
    } else {
        check_status(flute_silu_mul(g.data_ptr(), u.data_ptr(), g.data_ptr(), g.numel(), act, stream));
        check_status(flute_gemm(&d.w, g.data_ptr(), C.data_ptr(), (int)M, K, d.N, act, stream));
    }
    return C;
}

// A gated block on several rows: down(silu(gate(A)) * up(A)) of the layers gate, up and down.
Tensor qgemm_linear_mlp(const Tensor &A_in, const std::vector<pybind11::tuple> &layers) {
    const char *who = "qgemm_linear_mlp";
    const Shape2 s = check_2d_input(who, A_in, false);
    TORCH_CHECK(layers.size() == 3, who, ": three layers: gate, up, down");
    const Tensor A = aligned16(A_in);
    c10::DeviceGuard guard(A.device());
    const Tensor out = gemm_layers(who, A, s, described_all(who, A, s.K, layers, 2), true), g = out.select(0, 0);
    return gated_down(out, described(who, g, g.size(1), layers[2]));
}

// Rows `ids` (int64, contiguous, flat) of a table, and whether every id lay in it (true where
// nobody asked).
std::pair<Tensor, bool> embedding_rows(const Tensor &ids, const Tensor &indices, const Tensor &lut, int64_t N,
                                       int64_t K, int64_t b1, int64_t gs, const c10::optional<Tensor> &indices2,
                                       const c10::optional<Tensor> &lut2, int64_t b2,
                                       const c10::optional<Tensor> &resB, const c10::optional<Tensor> &resA,
                                       const c10::optional<Tensor> &signs, int64_t rot_block, bool check_ids) {
    const char *who = "embedding_gather";
    const auto held = [](const c10::optional<Tensor> &t) { return t.has_value() ? *t : Tensor(); };
    c10::DeviceGuard guard(lut.device());
    const Tensor out = torch::empty({ids.numel(), K}, lut.options());
    // (the row whose type and device the checks compare the operands with)
    const Tensor like = ids.numel() ? out.narrow(0, 0, 1) : torch::empty({1, K}, lut.options());
    Described d = describe(who, like, K, indices, lut, b1, held(indices2), held(lut2), b2, held(resB), held(resA),
                           Tensor(), gs, signs, c10::nullopt, rot_block, kGsAll, 256);
    TORCH_CHECK(d.N == N, who, ": blob holds N=", d.N, ", not ", N);
    TORCH_CHECK(ids.scalar_type() == at::kLong && ids.is_contiguous() && ids.device() == lut.device(), who,
                ": ids must be contiguous int64 on the table's device");
    int in_range = 1;
    flute_status st;
    {
        pybind11::gil_scoped_release unlocked;            // the checked form waits for the launch's verdict
        st = check_ids ? flute_embedding_checked(&d.w, ids.data_ptr<int64_t>(), ids.numel(), out.data_ptr(),
                                                 stream_of(lut), &in_range)
                       : flute_embedding(&d.w, ids.data_ptr<int64_t>(), ids.numel(), out.data_ptr(), stream_of(lut));
    }
    check_status(st);
    return {out, in_range != 0};
}

// Addresses of what the members' launches read, seven to a member in a fixed order, 0 for what is absent:
// palettized_modules._operand_ptrs as it stands there (the dictionaries that a module's attribute lookup
// ends in, in its order, then the lookup itself).
pybind11::tuple operand_addresses(const pybind11::sequence &members) {
    namespace py = pybind11;
    static PyObject *const names[] = {PyUnicode_InternFromString("indices"), PyUnicode_InternFromString("lut"),
                                      PyUnicode_InternFromString("indices2"), PyUnicode_InternFromString("lut2"),
                                      PyUnicode_InternFromString("resA"), PyUnicode_InternFromString("resB"),
                                      PyUnicode_InternFromString("bias")};
    static PyObject *const buffers = PyUnicode_InternFromString("_buffers"), *const parameters = PyUnicode_InternFromString("_parameters");
    const size_t count = members.size();
    py::tuple out(7 * count);
    for (size_t i = 0; i < count; ++i) {
        const py::object m = members[i];
        py::object places[3];
        PyObject **const own = _PyObject_GetDictPtr(m.ptr());
        if (own && *own) {
            PyObject *const b = PyDict_GetItemWithError(*own, buffers), *const p = PyDict_GetItemWithError(*own, parameters);
            if (b && p && PyDict_Check(b) && PyDict_Check(p)) {          // a module
                PyObject *const three[3] = {*own, b, p};
                for (int n = 0; n < 3; ++n) places[n] = py::reinterpret_borrow<py::object>(three[n]);
            }
        }
        for (int n = 0; n < 7; ++n) {
            py::object t;
            for (const py::object &place : places) {
                if (!place) continue;
                if (PyObject *const found = PyDict_GetItemWithError(place.ptr(), names[n])) {
                    t = py::reinterpret_borrow<py::object>(found);
                    break;
                }
            }
            if (!t) {                                                    // (only what is not there counts as absent)
                t = py::reinterpret_steal<py::object>(PyObject_GetAttr(m.ptr(), names[n]));
                if (!t) {
                    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) throw py::error_already_set();
                    PyErr_Clear();
                    t = py::none();
                }
            }
            out[7 * i + n] = THPVariable_Check(t.ptr()) ? py::int_((size_t)THPVariable_Unpack(t.ptr()).data_ptr()) : py::int_(0);
        }
    }
    return out;
}

// ---- the module layer's forwards ------------------------------------------------------------
// palettized_modules' forwards of the calls that need nothing but the library: every operand in the type and
// on the device that the launch reads, nobody watching, no switch set.  Each method answers None for any other
// call, and the Python forward then runs from its beginning.  Everything is read out of the modules on each
// call (the dictionaries that attribute lookup ends in); nothing is kept from one call for the next but
// which entry serves a shape, by its numbers.  What is used behind a call into Python (hooks, attributes of
// modules, the choice of an entry: other threads run there, and may replace what a module holds) is held by a
// reference.  One token, 4096 -> 1024: 10.1 us of host time a call in
// Python, 7 here; q/k/v of several rows 22 and 9, of rotated ones 39 and 16; a gated block of 22 rows 43 and
// 19; a thousand embedding rows 16 and 13, half of them the wait for the verdict on the ids.
namespace names {
#define FLUTE_NAME(n) PyObject *const n = PyUnicode_InternFromString(#n)
FLUTE_NAME(_buffers); FLUTE_NAME(_parameters); FLUTE_NAME(_modules); FLUTE_NAME(_dev_cache); FLUTE_NAME(_logical);
FLUTE_NAME(_merge_state); FLUTE_NAME(_forward_hooks); FLUTE_NAME(_forward_pre_hooks); FLUTE_NAME(_backward_hooks);
FLUTE_NAME(_backward_pre_hooks); FLUTE_NAME(_current_level); FLUTE_NAME(environ); FLUTE_NAME(forward); FLUTE_NAME(indices);
FLUTE_NAME(lut); FLUTE_NAME(indices2); FLUTE_NAME(lut2); FLUTE_NAME(resA); FLUTE_NAME(resB); FLUTE_NAME(bias);
FLUTE_NAME(bitwidth); FLUTE_NAME(bitwidth2); FLUTE_NAME(group_size); FLUTE_NAME(N); FLUTE_NAME(K); FLUTE_NAME(reference);
FLUTE_NAME(rot_signs); FLUTE_NAME(awq_scale); FLUTE_NAME(fold_order); FLUTE_NAME(signs); FLUTE_NAME(awq); FLUTE_NAME(has_stream2);
FLUTE_NAME(q_proj); FLUTE_NAME(k_proj); FLUTE_NAME(v_proj); FLUTE_NAME(gate_proj); FLUTE_NAME(up_proj); FLUTE_NAME(down_proj);
FLUTE_NAME(act_fn); FLUTE_NAME(ok); FLUTE_NAME(device); FLUTE_NAME(dtype); FLUTE_NAME(ptrs); FLUTE_NAME(sources);
FLUTE_NAME(seg_table); FLUTE_NAME(out);
#undef FLUTE_NAME
}  // namespace names

// A dictionary's value (borrowed), or nullptr.
PyObject *item(PyObject *dict, PyObject *name) {
    PyObject *const v = PyDict_GetItemWithError(dict, name);
    if (!v && PyErr_Occurred()) throw pybind11::error_already_set();
    return v;
}

// The dictionaries of a module that its attributes are looked up in.
struct Places {
    PyObject *own = nullptr, *buffers = nullptr, *parameters = nullptr;
    explicit Places(PyObject *m) {
        PyObject **const d = _PyObject_GetDictPtr(m);
        if (!d || !*d) return;
        buffers = item(*d, names::_buffers);
        parameters = item(*d, names::_parameters);
        if (buffers && parameters && PyDict_CheckExact(buffers) && PyDict_CheckExact(parameters)) own = *d;
    }
    PyObject *find(PyObject *name) const {
        PyObject *v = item(own, name);
        if (!v) v = item(buffers, name);
        if (!v || v == Py_None) {
            PyObject *const w = item(own, name) ? nullptr : item(parameters, name);
            if (w) v = w;
        }
        return v;
    }
    bool integer(PyObject *name, int64_t &v) const {
        PyObject *const o = item(own, name);
        if (!o || !PyLong_CheckExact(o)) return false;
        v = PyLong_AsLongLong(o);
        if (v == -1 && PyErr_Occurred()) throw pybind11::error_already_set();
        return true;
    }
};

// The operands of one layer as its module holds them.
struct Layer {
    Tensor indices, lut, indices2, lut2, resB, resA, bias, signs, awq;
    Tensor rotation;                                    // the module's own signs
    int64_t b1 = 0, b2 = 0, gs = 0, N = 0, K = 0;
    bool scaled = false;
    int64_t rank() const { return resB.defined() ? resB.size(0) : 0; }
    Described described(const char *who, const Tensor &A) const {
        const auto opt = [](const Tensor &t) { return t.defined() ? c10::optional<Tensor>(t) : c10::optional<Tensor>(); };
        return describe(who, A, K, indices, lut, b1, indices2, lut2, b2, resB, resA, bias, gs, opt(signs), opt(awq), 0, kGsAll, 256);
    }
};

class Forwards {
  public:
    Forwards(pybind11::object linear_type, pybind11::object linear_forward, pybind11::object embedding_type,
             pybind11::dict census, pybind11::object gemv_choice, pybind11::object is_silu)
        : linear_type_(std::move(linear_type)), linear_forward_(std::move(linear_forward)),
          embedding_type_(std::move(embedding_type)), census_(std::move(census)), gemv_choice_(std::move(gemv_choice)),
          is_silu_(std::move(is_silu)) {
        namespace py = pybind11;
        os_ = py::module_::import("os");
        environ_ = os_.attr("environ");
        if (py::hasattr(environ_, "_data")) environ_data_ = environ_.attr("_data");
        parameter_type_ = py::module_::import("torch.nn").attr("Parameter");
        forward_ad_ = py::module_::import("torch.autograd.forward_ad");
        transforms_ = py::module_::import("torch._C._functorch").attr("peek_interpreter_stack");
        global_hooks_ = py::module_::import("torch.nn.modules.module").attr("_has_any_global_hook");
        for (const char *n : {"FLUTE_NO_FHT_FUSE", "FLUTE_ROTATION", "FLUTE_NO_SPLITK", "FLUTE_NO_WIDE_PREF", "FLUTE_NO_MERGE"})
            switches_.push_back(py::bytes(n));
        for (const char *n : {"gemv_splitk", "gemv_splitk_fht", "gemv", "gemv_fht", "dual_stream", "per_group_lut", "gemm_multi",
                              "gemv_multi", "gemv_mlp", "embedding_gather"})
            routes_.push_back(py::str(n));
    }

    pybind11::object linear(pybind11::handle m, pybind11::handle x_) {
        Tensor x;
        if (!plain_input(x_.ptr(), x) || !no_switch()) return pybind11::none();
        const Tensor x2 = rows_of(x);
        Layer l;
        if (!x2.is_contiguous() || !read(m.ptr(), x2, l)) return pybind11::none();
        const int64_t M = x2.size(0);
        Tensor y;
        if (M == 1) {
            if (!one_row(x2, l, y)) return pybind11::none();
        } else {
            if (M < 1 || !several_rows(x2, l)) return pybind11::none();
            count_rows(M, l);
            const Described d = l.described("qgemm_linear", x2);
            y = gemm_described(x2, d);
        }
        return wrap(shaped(y, x));
    }

    pybind11::object qkv(pybind11::handle m, pybind11::handle x_) {
        Tensor x;
        Members members;
        if (!plain_input(x_.ptr(), x) || !no_switch() ||
            !children(m.ptr(), {names::q_proj, names::k_proj, names::v_proj}, members))
            return pybind11::none();
        if (x.numel() == x.size(-1)) {
            const Tensor out = grouped(m.ptr(), members, 3, x, false);
            if (!out.defined()) return pybind11::none();
            count(kGemvMulti);
            return wrap(x.dim() == 3 ? out.view({1, 1, out.size(1)}) : out);
        }
        const Tensor x2 = rows_of(x);
        std::vector<Layer> layers(3);
        if (!together(members, 3, x2, layers)) return pybind11::none();
        const Shape2 s = {x2.size(0), x2.size(1)};
        const Tensor A = aligned16(x2);
        c10::DeviceGuard guard(A.device());
        std::vector<Described> d;
        for (const Layer &l : layers) d.push_back(l.described("qgemm_linear_multi", A));
        const Tensor y = gemm_layers("qgemm_linear_multi", A, s, d, false);
        count(kGemmMulti);
        return wrap(shaped(y, x));
    }

    pybind11::object mlp(pybind11::handle m, pybind11::handle x_) {
        Tensor x;
        Members members;
        if (!plain_input(x_.ptr(), x) || !no_switch() ||
            !children(m.ptr(), {names::gate_proj, names::up_proj, names::down_proj}, members))
            return pybind11::none();
        const bool one = x.numel() == x.size(-1);
        if (one) {
            if (!own_call(members, 2, 3)) return pybind11::none();
            Layer down;
            const Tensor h = grouped(m.ptr(), members, 2, x, true, [&](const Tensor &h) { return read(members[2].ptr(), h, down); });
            if (!h.defined()) return pybind11::none();
            count(kGemvMlp);
            Tensor y;
            if (!one_row(h, down, y)) {                 // (the product is there: the module's own call)
                const pybind11::object out = pybind11::reinterpret_steal<pybind11::object>(
                    PyObject_CallOneArg(members[2].ptr(), wrap(h).ptr()));
                if (!out) throw pybind11::error_already_set();
                y = THPVariable_Unpack(out.ptr());
            }
            return wrap(x.dim() == 3 ? y.view({x.size(0), x.size(1), y.size(1)}) : y);
        }
        if (!is_silu(m.ptr())) return pybind11::none();
        const Tensor x2 = rows_of(x);
        std::vector<Layer> layers(2);
        Layer down;
        if (!own_call(members, 2, 3) || !together(members, 2, x2, layers) || layers[0].N != layers[1].N ||
            !read(members[2].ptr(), x2, down, layers[0].N) || !several_rows(x2, down))
            return pybind11::none();
        const char *who = "qgemm_linear_mlp";
        const Shape2 s = {x2.size(0), x2.size(1)};
        const Tensor A = aligned16(x2);
        c10::DeviceGuard guard(A.device());
        std::vector<Described> d;
        for (const Layer &l : layers) d.push_back(l.described(who, A));
        const Tensor out = gemm_layers(who, A, s, d, true);
        const Tensor y = gated_down(out, down.described(who, out.select(0, 0)));
        count(kGemmMulti);
        count_rows(s.M, down);
        return wrap(shaped(y, x));
    }

    pybind11::object embedding(pybind11::handle m, pybind11::handle ids_) {
        namespace py = pybind11;
        if ((PyObject *)Py_TYPE(m.ptr()) != embedding_type_.ptr() || !THPVariable_CheckExact(ids_.ptr())) return py::none();
        const Tensor ids = THPVariable_Unpack(ids_.ptr());
        if (!ids.is_cuda() || ids.scalar_type() != at::kLong || !ids.is_contiguous() || at::isTensorSubclassLike(ids)) return py::none();
        const Places at(m.ptr());
        Layer l;
        if (!at.own || item(at.own, names::reference) != Py_False || !numbers(at, l)) return py::none();
        PyObject *const two = item(at.own, names::has_stream2);
        if (two != Py_True && two != Py_False) return py::none();
        if (!tensor(at, names::indices, l.indices) || !tensor(at, names::lut, l.lut) || !tensor(at, names::indices2, l.indices2) ||
            !tensor(at, names::lut2, l.lut2) || !tensor(at, names::resA, l.resA) || !tensor(at, names::resB, l.resB) ||
            !l.indices.defined() || !l.lut.defined() || l.lut.device() != ids.device())
            return py::none();
        if (two == Py_False) l.b2 = 0;
        PyObject *const signs = item(at.own, names::rot_signs);
        if (!signs || !table_signs(at, signs, ids.device(), l.signs)) return py::none();
        const auto opt = [](const Tensor &t) { return t.defined() ? c10::optional<Tensor>(t) : c10::optional<Tensor>(); };
        c10::DeviceGuard guard(ids.device());
        const bool capturing = c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
        const auto got = embedding_rows(ids.reshape({-1}), l.indices, l.lut, l.N, l.K, l.b1, l.gs, opt(l.indices2), opt(l.lut2), l.b2,
                                        opt(l.resB), opt(l.resA), opt(l.signs), 0, !capturing);
        if (!got.second) return py::none();             // (the Python forward says what is wrong)
        count(kEmbeddingGather);
        if (ids.dim() == 1) return wrap(got.first);
        std::vector<int64_t> shape(ids.sizes().begin(), ids.sizes().end());
        shape.push_back(l.K);
        return wrap(got.first.view(shape));
    }

  private:
    enum Route { kGemvSplitk, kGemvSplitkFht, kGemv, kGemvFht, kDualStream, kPerGroupLut, kGemmMulti, kGemvMulti, kGemvMlp,
                 kEmbeddingGather, kNone };

    typedef std::array<pybind11::object, 3> Members;    // projections of a block

    static pybind11::object wrap(const Tensor &t) { return pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(t)); }
    static Tensor rows_of(const Tensor &x) { return x.dim() == 2 ? x : x.reshape({-1, x.size(-1)}); }
    static Tensor shaped(const Tensor &y, const Tensor &x) {
        if (x.dim() == 2) return y;
        std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
        shape.back() = y.size(1);
        return y.reshape(shape);
    }

    // An ordinary 16-bit tensor on a device, which nobody differentiates or maps over.
    bool plain_input(PyObject *o, Tensor &x) const {
        if (!THPVariable_CheckExact(o)) return false;
        const Tensor &t = THPVariable_Unpack(o);
        if (!t.is_cuda() || !is_act(t) || t.dim() < 2 || t.requires_grad() || at::isTensorSubclassLike(t) || t.numel() == 0) return false;
        x = t;
        return true;
    }

    // None of the environment's switches is set (os.environ's own dictionary: lookups in os.environ decode).
    bool no_switch() const {
        if (!environ_data_ || !PyDict_CheckExact(environ_data_.ptr())) return false;
        PyObject *const now = PyObject_GetAttr(os_.ptr(), names::environ);
        if (!now) throw pybind11::error_already_set();
        const bool same = now == environ_.ptr();
        Py_DECREF(now);
        if (!same) return false;
        for (const pybind11::bytes &s : switches_)
            if (item(environ_data_.ptr(), s.ptr())) return false;
        return true;
    }

    // The tensor a module holds under a name (undefined: it has none); false: the Python forward has to look.
    bool tensor(const Places &at, PyObject *name, Tensor &t) const {
        PyObject *const o = at.find(name);
        if (o == Py_None) return true;
        if (!o || !(THPVariable_CheckExact(o) || (PyObject *)Py_TYPE(o) == parameter_type_.ptr())) return false;
        t = THPVariable_Unpack(o);
        return true;
    }

    static bool numbers(const Places &at, Layer &l) {
        return at.integer(names::bitwidth, l.b1) && at.integer(names::bitwidth2, l.b2) && at.integer(names::group_size, l.gs) &&
               at.integer(names::N, l.N) && at.integer(names::K, l.K);
    }

    // A vector of the rotation as the kernels read it: itself, or the copy the module keeps of it (`_on`).
    static bool vector_on(const Places &at, PyObject *key, PyObject *source, const c10::Device &device, Tensor &v) {
        if (!THPVariable_CheckExact(source)) return false;
        const Tensor &t = THPVariable_Unpack(source);
        if (t.device() == device && t.scalar_type() == at::kFloat && t.is_contiguous()) {
            v = t;
            return true;
        }
        PyObject *const entry = cached(item(at.own, names::_dev_cache), key, device);
        if (!entry || !PyTuple_CheckExact(entry) || PyTuple_GET_SIZE(entry) != 4 || PyTuple_GET_ITEM(entry, 0) != source) return false;
        if (PyLong_AsVoidPtr(PyTuple_GET_ITEM(entry, 1)) != t.data_ptr()) return false;
        PyObject *const version = PyTuple_GET_ITEM(entry, 2);
        if (version != Py_None && (t.is_inference() || PyLong_AsLongLong(version) != (long long)t._version())) return false;
        PyObject *const value = PyTuple_GET_ITEM(entry, 3);
        if (!THPVariable_Check(value)) return false;
        v = THPVariable_Unpack(value);
        return true;
    }

    // dict[(key, device)], borrowed.
    static PyObject *cached(PyObject *dict, PyObject *key, const c10::Device &device) {
        if (!dict || !PyDict_CheckExact(dict)) return nullptr;
        const pybind11::object d = pybind11::reinterpret_steal<pybind11::object>(THPDevice_New(device));
        const pybind11::object k = pybind11::reinterpret_steal<pybind11::object>(PyTuple_Pack(2, key, d.ptr()));
        return item(dict, k.ptr());
    }

    // PalettizedEmbedding._signs_on where it finds its copy.
    static bool table_signs(const Places &at, PyObject *signs, const c10::Device &device, Tensor &v) {
        if (signs == Py_None) return true;
        if (!THPVariable_CheckExact(signs)) return false;
        const Tensor &t = THPVariable_Unpack(signs);
        if (t.device() == device) {
            v = t;
            return true;
        }
        PyObject *const entry = cached(item(at.own, names::_logical), names::signs, device);
        if (!entry || !PyTuple_CheckExact(entry) || PyTuple_GET_SIZE(entry) != 2) return false;
        PyObject *const k = PyTuple_GET_ITEM(entry, 0), *const c = PyTuple_GET_ITEM(entry, 1);
        if (!THPVariable_Check(k) || !THPVariable_Check(c)) return false;
        const Tensor &kept = THPVariable_Unpack(k);
        if (kept.scalar_type() != t.scalar_type() || kept.sizes() != t.sizes() || !same_bytes(kept, t)) return false;
        v = THPVariable_Unpack(c);
        return true;
    }
    // Two tensors whose values are the bytes at their addresses in host memory, and the same ones.
    static bool same_bytes(const Tensor &a, const Tensor &b) {
        return a.is_cpu() && b.is_cpu() && a.is_contiguous() && b.is_contiguous() && !a.is_neg() && !b.is_neg() &&
               a.scalar_type() == b.scalar_type() && a.numel() == b.numel() && std::memcmp(a.data_ptr(), b.data_ptr(), a.nbytes()) == 0;
    }

    // The operands of module m as launches on rows like x's read them; K: columns of its rows.  False: something
    // has to be converted, copied, refused or done otherwise.
    bool read(PyObject *m, const Tensor &x, Layer &l, int64_t K = -1) const {
        if ((PyObject *)Py_TYPE(m) != linear_type_.ptr()) return false;
        const Places at(m);
        if (!at.own || item(at.own, names::reference) != Py_False || !numbers(at, l) || l.K != (K < 0 ? x.size(1) : K)) return false;
        if (!tensor(at, names::indices, l.indices) || !tensor(at, names::lut, l.lut) || !tensor(at, names::indices2, l.indices2) ||
            !tensor(at, names::lut2, l.lut2) || !tensor(at, names::resB, l.resB) || !tensor(at, names::resA, l.resA) ||
            !tensor(at, names::bias, l.bias) || !l.indices.defined() || !l.lut.defined())
            return false;
        if (l.indices2.defined() != l.lut2.defined() || l.resA.defined() != l.resB.defined()) return false;
        if (!l.indices2.defined()) l.b2 = 0;
        if (!is_act(l.lut) || l.lut.requires_grad() || l.lut.device() != x.device() ||
            (l.lut.scalar_type() == at::kBFloat16 && x.scalar_type() != at::kBFloat16))
            return false;
        for (const Tensor *t : {&l.resB, &l.resA, &l.bias})
            if (t->defined() && (t->device() != x.device() || t->scalar_type() != x.scalar_type() || !t->is_contiguous() ||
                                 at::isTensorSubclassLike(*t)))
                return false;
        if (l.resB.defined() && l.resB.dim() != 2) return false;
        PyObject *const rotation = item(at.own, names::rot_signs);
        if (!rotation) return false;
        if (rotation == Py_None) return true;
        if (!vector_on(at, names::signs, rotation, x.device(), l.signs)) return false;
        l.rotation = THPVariable_Unpack(rotation);
        PyObject *const scale = item(at.own, names::awq_scale), *const order = item(at.own, names::fold_order);
        if (!scale || !order) return false;
        if (scale == Py_None) return true;
        if (!PyUnicode_CheckExact(order)) return false;
        if (PyUnicode_CompareWithASCIIString(order, "rotate_then_awq") != 0) return true;
        l.scaled = true;
        return vector_on(at, names::awq, scale, x.device(), l.awq);
    }

    // What several_rows has beyond read: PalettizedLinear._gemm_operands.
    bool several_rows(const Tensor &x, const Layer &l) const {
        if (c10::GradMode::is_enabled())
            for (const Tensor *t : {&l.bias, &l.resA, &l.resB})
                if (t->defined() && t->requires_grad()) return false;
        if (watched()) return false;
        const int64_t M = x.size(0), rank = l.rank();
        if (rank > 256 || !(rank <= 16 || M * rank * (l.N + l.K) <= (int64_t)1 << 27)) return false;
        if (l.bias.defined() && (l.bias.dim() != 1 || l.bias.numel() != l.N)) return false;
        if (l.rotation.defined() && !(l.K % 32 == 0 && l.K >= 32 && l.K <= 65504 && l.K < 32768)) return false;
        if (l.b2 && l.lut2.scalar_type() != l.lut.scalar_type()) return false;
        return l.gs >= 16 && l.gs <= 2048 && (l.gs & (l.gs - 1)) == 0 && l.N % 128 == 0 && l.K % 64 == 0;
    }

    // Forward-mode derivatives or function transforms in force.
    bool watched() const {
        const pybind11::object level = forward_ad_.attr(pybind11::handle(names::_current_level));
        if (PyLong_AsLong(level.ptr()) >= 0) return true;
        const pybind11::object stack = pybind11::reinterpret_steal<pybind11::object>(PyObject_CallNoArgs(transforms_.ptr()));
        if (!stack) throw pybind11::error_already_set();
        return !stack.is_none();
    }

    // One row through the one-token launch; false: the shape is not its.
    bool one_row(const Tensor &x, const Layer &l, Tensor &y) {
        const Route route = gemv_route(l);
        if (route == kNone) return false;
        count(route);
        const auto opt = [](const Tensor &t) { return t.defined() ? c10::optional<Tensor>(t) : c10::optional<Tensor>(); };
        y = gemv("qgemm_linear", x, l.indices, l.lut, l.b1, l.indices2, l.lut2, l.b2, l.resB, l.resA, l.bias, l.gs, opt(l.signs),
                 opt(l.awq), 0, 0, kGsAll, 256);
        return true;
    }

    Tensor gemm_described(const Tensor &x, const Described &d) const {
        const Tensor A = aligned16(x);
        c10::DeviceGuard guard(A.device());
        const Tensor C = torch::empty({A.size(0), d.N}, A.options());
        check_status(flute_gemm(&d.w, A.data_ptr(), C.data_ptr(), (int)A.size(0), A.size(1), d.N, act_code(A), stream_of(A)));
        return C;
    }

    // Which entry of the package takes one row of a shape, by its numbers (palettized_modules._gemv_choice).
    Route gemv_route(const Layer &l) {
        const std::array<int64_t, 7> key = {l.b1, l.b2, l.gs, l.N, l.K, l.rank(), l.rotation.defined()};
        const auto known = gemv_routes_.find(key);
        if (known != gemv_routes_.end()) return known->second;
        const pybind11::object name = gemv_choice_(l.b1, l.b2, l.gs, l.N, l.K, l.rank(), l.rotation.defined());
        Route route = kNone;
        for (int r = kGemvSplitk; r <= kGemvFht && !name.is_none(); ++r)
            if (name.equal(routes_[r])) route = (Route)r;
        if (gemv_routes_.size() >= 4096) gemv_routes_.clear();
        return gemv_routes_[key] = route;
    }

    void count(Route r) const {
        PyObject *const name = routes_[r].ptr(), *const before = item(census_.ptr(), name);
        const pybind11::int_ now(before ? PyLong_AsLongLong(before) + 1 : 1);
        if (PyDict_SetItem(census_.ptr(), name, now.ptr())) throw pybind11::error_already_set();
    }
    void count_rows(int64_t M, const Layer &l) const { count(M <= 16 && l.rank() <= 16 ? kDualStream : kPerGroupLut); }

    // Children of a block out of its dictionary of modules.
    static bool children(PyObject *m, std::initializer_list<PyObject *> which, Members &out) {
        PyObject **const d = _PyObject_GetDictPtr(m);
        if (!d || !*d) return false;
        PyObject *const modules = item(*d, names::_modules);
        if (!modules || !PyDict_CheckExact(modules)) return false;
        size_t i = 0;
        for (PyObject *name : which) {
            PyObject *const child = item(modules, name);
            if (!child || child == Py_None || item(*d, name)) return false;
            out[i++] = pybind11::reinterpret_borrow<pybind11::object>(child);
        }
        return true;
    }
    bool is_silu(PyObject *m) const {
        const pybind11::object act = pybind11::reinterpret_steal<pybind11::object>(PyObject_GetAttr(m, names::act_fn));
        if (!act) throw pybind11::error_already_set();
        return PyObject_IsTrue(is_silu_(act).ptr()) == 1;
    }

    // palettized_modules._own_call and no global hooks: calling these modules is calling the class's forward.
    bool own_call(const Members &members, int first, int last) const {
        const pybind11::object f = pybind11::reinterpret_steal<pybind11::object>(PyObject_GetAttr(linear_type_.ptr(), names::forward));
        if (!f) throw pybind11::error_already_set();
        if (f.ptr() != linear_forward_.ptr()) return false;
        for (int i = first; i < last; ++i) {
            if ((PyObject *)Py_TYPE(members[i].ptr()) != linear_type_.ptr()) return false;
            PyObject *const own = *_PyObject_GetDictPtr(members[i].ptr());
            if (!own || item(own, names::forward)) return false;
            for (PyObject *hooks : {names::_forward_hooks, names::_forward_pre_hooks, names::_backward_hooks, names::_backward_pre_hooks}) {
                PyObject *const h = item(own, hooks);
                if (!h || PyObject_IsTrue(h) != 0) return false;
            }
        }
        const pybind11::object any = pybind11::reinterpret_steal<pybind11::object>(PyObject_CallNoArgs(global_hooks_.ptr()));
        if (!any) throw pybind11::error_already_set();
        return PyObject_IsTrue(any.ptr()) == 0;          // (the registries themselves, empty)
    }

    // palettized_modules._layers_on.
    bool together(const Members &members, int n, const Tensor &x, std::vector<Layer> &layers) const {
        if (x.size(0) < 2 || !x.is_contiguous() || !own_call(members, 0, n)) return false;
        for (int i = 0; i < n; ++i) {
            Layer &l = layers[i];
            if (!read(members[i].ptr(), x, l) || !several_rows(x, l) || l.lut.scalar_type() != layers[0].lut.scalar_type()) return false;
            if (i && l.rotation.defined() && layers[0].rotation.defined() && !l.scaled && !layers[0].scaled) {
                // one rotation, one address: its members share the rotated rows
                if (l.rotation.is_same(layers[0].rotation) || same_bytes(l.rotation, layers[0].rotation)) l.signs = layers[0].signs;
            }
        }
        return true;
    }

    // The decode launch of a block whose table still holds (state of FusedPalettizedMLP and SplitQKV): its output,
    // or an undefined tensor.  `also`: what else has to hold before the launch.
    Tensor grouped(PyObject *block, const Members &members, int n, const Tensor &x, bool mlp,
                   const std::function<bool(const Tensor &)> &also = nullptr) const {
        namespace py = pybind11;
        if (x.dim() > 3 || !x.is_contiguous()) return Tensor();
        const auto held_item = [](const py::object &dict, PyObject *name) {
            return py::reinterpret_borrow<py::object>(item(dict.ptr(), name));     // (empty: it has none)
        };
        const py::object state = py::reinterpret_borrow<py::object>(item(*_PyObject_GetDictPtr(block), names::_merge_state));
        if (!state || !PyDict_CheckExact(state.ptr()) || item(state.ptr(), names::ok) != Py_True) return Tensor();
        PyObject *const device = item(state.ptr(), names::device), *const dtype = item(state.ptr(), names::dtype);
        if (!device || !THPDevice_Check(device) || ((THPDevice *)device)->device != x.device() || !dtype || !THPDtype_Check(dtype) ||
            ((THPDtype *)dtype)->scalar_type != x.scalar_type())
            return Tensor();
        const py::object ptrs = held_item(state, names::ptrs), sources = held_item(state, names::sources),
                         table = held_item(state, names::seg_table), out_ = held_item(state, names::out);
        if (!ptrs || !PyTuple_CheckExact(ptrs.ptr()) || !sources || !PyList_CheckExact(sources.ptr()) || !table || !out_ ||
            !THPVariable_Check(table.ptr()) || !THPVariable_Check(out_.ptr()))
            return Tensor();
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(sources.ptr()); ++i) {
            const py::object s = py::reinterpret_borrow<py::object>(PyList_GET_ITEM(sources.ptr(), i));  // (member, name, tensor, version)
            if (!PyTuple_CheckExact(s.ptr()) || PyTuple_GET_SIZE(s.ptr()) != 4) return Tensor();
            const py::object t = py::reinterpret_steal<py::object>(
                PyObject_GetAttr(PyTuple_GET_ITEM(s.ptr(), 0), PyTuple_GET_ITEM(s.ptr(), 1)));
            if (!t) throw py::error_already_set();
            PyObject *const version = PyTuple_GET_ITEM(s.ptr(), 3);
            if (t.ptr() != PyTuple_GET_ITEM(s.ptr(), 2) || !THPVariable_Check(t.ptr()) ||
                (version != Py_None && PyLong_AsLongLong(version) != (long long)THPVariable_Unpack(t.ptr())._version()))
                return Tensor();
        }
        // (the addresses last: from here to the launch nothing calls into Python, so nobody frees what they name)
        py::list held;
        for (int i = 0; i < n; ++i) held.append(members[i]);
        const py::tuple now = operand_addresses(held);
        const int same = PyObject_RichCompareBool(now.ptr(), ptrs.ptr(), Py_EQ);
        if (same < 0) throw py::error_already_set();
        if (!same) return Tensor();
        const Places first(members[0].ptr());
        Tensor lut;
        int64_t K;
        if (!first.own || !first.integer(names::K, K) || K != x.size(-1) || !tensor(first, names::lut, lut) || !lut.defined())
            return Tensor();
        const Tensor out = THPVariable_Unpack(out_.ptr()), x2 = rows_of(x);
        if (also && !also(out)) return Tensor();
        const int code = lut.scalar_type() == at::kBFloat16 ? FLUTE_BF16 : FLUTE_F16;
        if (mlp) return gemv_mlp_table(x2, THPVariable_Unpack(table.ptr()), out, code, 0);
        gemv_multi_table(x2, THPVariable_Unpack(table.ptr()), code, 0);
        return out;
    }

    pybind11::object linear_type_, linear_forward_, embedding_type_, os_, environ_, environ_data_, parameter_type_, forward_ad_,
        transforms_, global_hooks_;
    pybind11::dict census_;
    pybind11::object gemv_choice_, is_silu_;
    std::vector<pybind11::bytes> switches_;
    std::vector<pybind11::str> routes_;
    std::map<std::array<int64_t, 7>, Route> gemv_routes_;
};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    namespace py = pybind11;
    m.doc() = "compiled PyTorch-ROCm binding of the idxN LUT linear layer (libflute_hip.so)";
    m.def("abi_version", []() { return flute_abi_version(); });
    m.def("qgemm_gemv_stream", &qgemm_gemv_stream);
    m.def("qgemm_gemv_fht_stream", &qgemm_gemv_fht_stream);
    m.def("qgemm_gemv_splitk_stream", &qgemm_gemv_splitk_stream, py::arg("A"), py::arg("indices"),
          py::arg("lut"), py::arg("bitwidth"), py::arg("indices2"), py::arg("lut2"),
          py::arg("bitwidth2"), py::arg("resB"), py::arg("resA"), py::arg("bias"),
          py::arg("group_size"), py::arg("split") = 0);
    m.def("qgemm_gemv_splitk_fht_stream", &qgemm_gemv_splitk_fht_stream, py::arg("A"),
          py::arg("indices"), py::arg("lut"), py::arg("bitwidth"), py::arg("indices2"),
          py::arg("lut2"), py::arg("bitwidth2"), py::arg("resB"), py::arg("resA"), py::arg("bias"),
          py::arg("group_size"), py::arg("signs"), py::arg("s"), py::arg("split") = 0,
          py::arg("rot_block") = 0);
    m.def("qgemm_linear", &qgemm_linear);
    py::class_<Forwards>(m, "Forwards")
        .def(py::init<py::object, py::object, py::object, py::dict, py::object, py::object>())
        .def("linear", &Forwards::linear)
        .def("qkv", &Forwards::qkv)
        .def("mlp", &Forwards::mlp)
        .def("embedding", &Forwards::embedding);
    m.def("embedding_rows", &embedding_rows);
    m.def("operand_addresses", &operand_addresses);
    m.def("qgemm_linear_multi", &qgemm_linear_multi);
    m.def("qgemm_linear_mlp", &qgemm_linear_mlp);
    m.def("qgemm_gemv_multi", &qgemm_gemv_multi, py::arg("A"), py::arg("seg_table"),
          py::arg("lut_dtype") = py::none(), py::arg("split") = 0);
    m.def("qgemm_gemv_mlp", &qgemm_gemv_mlp, py::arg("A"), py::arg("seg_table"), py::arg("C"),
          py::arg("lut_dtype") = py::none(), py::arg("split") = 0);
    m.def("qgemm_cutlass_streaming", &qgemm_cutlass_streaming, py::arg("A"), py::arg("indices"),
          py::arg("lut"), py::arg("bitwidth"), py::arg("group_size"), py::arg("q_layout") = 1);
    m.def("qgemm_dual_stream", &qgemm_dual_stream, py::arg("A"), py::arg("indices"), py::arg("lut"),
          py::arg("bitwidth"), py::arg("indices2"), py::arg("lut2"), py::arg("bitwidth2"),
          py::arg("resB"), py::arg("resA"), py::arg("bias"), py::arg("group_size") = 512);
}
