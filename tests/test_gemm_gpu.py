"""GPU parity of the M > 1 LUT GEMM (MFMA) against the oracle, through the
flute_extended op surface (which calls the C ABI).

Tolerance: relative L2 <= 1e-3 for fp16 outputs (the benchmark contract's figure
for fp32 accumulate + one 16-bit rounding), <= 4e-3 for bf16 outputs, whose final
rounding alone is 2^-9.  The oracle is the fp64 closed form.  Index decoding is
checked bit-exactly: with A = identity rows (one-hot in k) the GEMM must return
the dequantised columns exactly, because a single product with 1.0 and a sum of
zeros involves no rounding.
"""
import pytest
import torch

import flute_extended as fx
import flute_oracle as O
from _util import gemm_rows, make_weight, make_x, rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = 1e-3
TOL_BF16 = 4e-3


def _exact(w, x):
    return O.linear_exact(x, w["blob"].numpy(), w["lut"], w["N"], w["K"], w["gs"], w["bits"],
                          w["blob2"].numpy() if w["bits2"] else None, w["lut2"], w["bits2"],
                          w["resA"], w["resB"], w["bias"])


def _dual(w, x):
    return fx.qgemm_dual_stream(x.to(DEV), w["blob_d"], w["lut_d"], w["bits"], w["gs"],
                                indices2=w.get("blob2_d"), lut2=w.get("lut2_d"),
                                bitwidth2=w["bits2"], resB=w.get("resB_d"), resA=w.get("resA_d"),
                                bias=w.get("bias_d"))


SINGLE = [
    # M, N, K, bits, gs
    (2, 128, 64, 4, 128),
    (16, 256, 512, 4, 128),
    (17, 256, 512, 4, 128),
    (33, 384, 1024, 4, 256),           # N not a multiple of the group size
    (64, 512, 1024, 4, 128),
    (100, 512, 1024, 4, 64),
    (128, 256, 2048, 4, 32),
    (130, 256, 1024, 4, 16),
    (256, 1024, 4096, 4, 128),
    (300, 256, 704, 4, 128),           # K/64 = 11: ragged over the k ways
    (8, 512, 1024, 3, 128),
    (48, 512, 1024, 3, 32),
    (8, 512, 1024, 2, 128),
    (200, 256, 1024, 2, 16),
    (8, 512, 1024, 1, 64),
    (96, 256, 1024, 1, 128),
]


@pytest.mark.parametrize("M,N,K,bits,gs", SINGLE)
def test_gemm_single_stream_fp16(M, N, K, bits, gs):
    w = make_weight(N, K, bits, gs, seed=M + N + K + bits, device=DEV)
    x = make_x(M, K, seed=11)
    y = fx.qgemm_per_group_lut(x.to(DEV), w["blob_d"], w["lut_d"], bitwidth=bits, group_size=gs,
                               indices_layout=f"idx{bits}").cpu()
    assert y.shape == (M, N) and y.dtype == torch.float16
    assert rel_l2(y, _exact(w, x).half()) <= TOL
    y2 = fx.qgemm_per_group_lut(x.to(DEV), w["blob_d"], w["lut_d"], bitwidth=bits, group_size=gs,
                                indices_layout=f"idx{bits}").cpu()
    assert torch.equal(y, y2)                           # deterministic


@pytest.mark.parametrize("rows", ["16", "32", "64", "128"])
@pytest.mark.parametrize("M,N,K,bits,gs", [c for c in SINGLE if c[0] > 16])
def test_gemm_every_workgroup_shape(tuning_env, rows, M, N, K, bits, gs):
    """The library picks the rows of A per workgroup (16, 32, 64 or 128) from M, N and K; at
    the small N of these cases it would always pick 16, so each shape is forced in turn
    (FLUTE_GEMM_ROWS) and must give the oracle's result."""
    tuning_env("FLUTE_GEMM_ROWS", rows)
    w = make_weight(N, K, bits, gs, seed=M + N + K + bits, device=DEV)
    x = make_x(M, K, seed=11)
    y = fx.qgemm_per_group_lut(x.to(DEV), w["blob_d"], w["lut_d"], bitwidth=bits, group_size=gs,
                               indices_layout=f"idx{bits}").cpu()
    assert rel_l2(y, _exact(w, x).half()) <= TOL


@pytest.mark.parametrize("rows", ["16", "32", "64", "128"])
def test_gemm_two_streams_residual_bias_every_workgroup_shape(tuning_env, rows):
    tuning_env("FLUTE_GEMM_ROWS", rows)
    M, N, K = 40, 256, 1024
    for lut_dtype, act_dtype in ((torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16)):
        w = make_weight(N, K, 4, 128, seed=7, bits2=2, rank=8, bias=True, lut_dtype=lut_dtype,
                        act_dtype=act_dtype, device=DEV)
        x = make_x(M, K, seed=13, dtype=act_dtype)
        y = _dual(w, x).cpu()
        ref = _exact(w, x).to(act_dtype)
        assert rel_l2(y, ref) <= (TOL if act_dtype == torch.float16 else TOL_BF16)


@pytest.mark.parametrize("M,N,K,gs", [(5, 256, 512, 128), (16, 512, 1024, 64), (33, 384, 1024, 256),
                                      (130, 256, 2048, 128)])
@pytest.mark.parametrize("act,lut", [(torch.float16, torch.float16), (torch.bfloat16, torch.float16),
                                     (torch.bfloat16, torch.bfloat16)])
def test_gemm_direct_activations_match_the_pre_pass(tuning_env, M, N, K, gs, act, lut):
    """With one 16-row block per wavefront the kernel reads A itself and transposes the
    pieces in registers; FLUTE_GEMM_NO_DIRECT=1 sends the same call through the activation
    pre-pass.  Both present identical operands, so the outputs are bit-identical; rows that
    are not 16-byte aligned take the pre-pass by themselves."""
    w = make_weight(N, K, 4, gs, seed=M + N, lut_dtype=lut, act_dtype=act, bias=True, device=DEV)
    x = make_x(M, K, seed=17, dtype=act)
    xd = x.to(DEV)
    y = _dual(w, xd)
    assert rel_l2(y.cpu(), _exact(w, x).to(act)) <= (TOL if act == torch.float16 else TOL_BF16)
    tuning_env("FLUTE_GEMM_NO_DIRECT", "1")
    assert torch.equal(_dual(w, xd), y)
    tuning_env("FLUTE_GEMM_NO_DIRECT", None)
    shifted = torch.zeros(M * K + 1, dtype=act, device=DEV)
    shifted[1:] = xd.reshape(-1)
    assert torch.equal(_dual(w, shifted[1:].reshape(M, K)), y)


@pytest.mark.parametrize("M,K,bits,bits2,act,lut,rot", [
    (17, 64, 4, 0, torch.float16, torch.float16, False),           # one row in the second block, one tile of K
    (32, 576, 3, 3, torch.bfloat16, torch.bfloat16, False),        # more wavefronts with a second tile than without
    (33, 1088, 4, 3, torch.float16, torch.float16, False),         # a workgroup with a single row
    (63, 1024, 2, 0, torch.bfloat16, torch.bfloat16, True),
    (40, 8256, 4, 1, torch.bfloat16, torch.float16, False),        # scales from a launch in front
    (48, 1024, 1, 4, torch.bfloat16, torch.float16, True),         # scales from the rotation
])
def test_gemm_32_row_workgroups_read_the_rows_themselves(tuning_env, M, K, bits, bits2, act, lut, rot):
    """32-row workgroups on the rows of A and on the operand image: equal bits, at any stride of the rows."""
    tuning_env("FLUTE_GEMM_ROWS", "32")
    w = make_weight(256, K, bits, 128, seed=M + K, bits2=bits2, lut_dtype=lut, act_dtype=act, bias=True, device=DEV)
    signs = O.rotation_signs(K, 3).to(DEV) if rot else None
    wide = torch.full((M, K + 24), float("nan"), dtype=act, device=DEV)
    x = make_x(M, K, seed=M, dtype=act).to(DEV)
    x[0] *= 1e3
    x[M - 1] = 0
    wide[:, 8:K + 8] = x
    import ctypes
    from flute_extended import _lib
    kind = lambda t: _lib.BF16 if t == torch.bfloat16 else _lib.F16
    d = _lib.FluteLinear()
    d.q1, d.lut1, d.q1_bytes, d.b1 = w["blob_d"].data_ptr(), w["lut_d"].data_ptr(), w["blob_d"].numel(), bits
    if bits2:
        d.q2, d.lut2, d.q2_bytes, d.b2 = w["blob2_d"].data_ptr(), w["lut2_d"].data_ptr(), w["blob2_d"].numel(), bits2
    d.N, d.K, d.group_size, d.lut_rows, d.lut_dtype, d.bias = 256, K, 128, 2, kind(lut), w["bias_d"].data_ptr()
    if rot:
        d.signs = signs.data_ptr()

    def run(a):
        C = torch.zeros(M, 256, dtype=act, device=DEV)
        assert _lib.lib.flute_gemm(ctypes.byref(d), a.data_ptr(), C.data_ptr(), M, a.stride(0), 256, kind(act),
                                   torch.cuda.current_stream().cuda_stream) == 0, _lib.last_error()
        return C

    rows = run(x)
    assert torch.equal(run(wide[:, 8:K + 8]), rows)
    tuning_env("FLUTE_GEMM_NO_DIRECT", "1")
    assert torch.equal(run(x), rows)
    if not rot:
        assert rel_l2(rows.cpu(), _exact(w, x.cpu()).to(act)) <= (TOL if act == torch.float16 else TOL_BF16)


@pytest.mark.parametrize("M,K,bits,bits2,rank,act,lut", [
    (2, 64, 4, 0, 1, torch.float16, torch.float16), (17, 576, 3, 3, 16, torch.bfloat16, torch.bfloat16),
    (33, 1088, 4, 2, 5, torch.float16, torch.float16), (15, 4160, 1, 0, 15, torch.bfloat16, torch.float16),
    (40, 8256, 4, 1, 16, torch.bfloat16, torch.float16), (16, 1024, 4, 4, 8, torch.float16, torch.float16),
    (20, 1024, 2, 1, 17, torch.float16, torch.float16)])
@pytest.mark.parametrize("rows,slices", [(16, "1"), (16, "2"), (32, "1"), (32, "3")])
def test_gemm_few_rows_residual_of_one_operand_of_ranks(tuning_env, M, K, bits, bits2, rank, act, lut, rows, slices):
    """Residuals of up to 16 ranks, whose coefficients the few-row kernel forms beside its products, slice of K
    by slice, and those that a launch in front forms (more ranks, twice 4 bits, 32 rows that need scales)."""
    tuning_env("FLUTE_GEMM_ROWS", str(rows))
    tuning_env("FLUTE_GEMM_KSPLIT", slices)
    w = make_weight(256, K, bits, 128, seed=M + K, bits2=bits2, rank=rank, lut_dtype=lut, act_dtype=act, bias=True, device=DEV)
    x = make_x(M, K, seed=M, dtype=act)
    x[M // 2] *= 1e2
    y = _dual(w, x).cpu()
    ref = _exact(w, x).to(act)
    for m in range(M):
        assert rel_l2(y[m], ref[m]) <= (TOL if act == torch.float16 else TOL_BF16), m
    tuning_env("FLUTE_GEMM_NO_DIRECT", "1")                # the launch in front: one rounding of the type apart
    assert rel_l2(y, _dual(w, x).cpu()) <= (2 ** -11 if act == torch.float16 else 2 ** -8)


@pytest.mark.parametrize("M,N,K,bits,bits2,rank", [(2, 128, 1024, 4, 0, 0), (8, 256, 1408, 4, 1, 0), (15, 512, 7616, 1, 4, 8),
                                                  (3, 256, 2752, 3, 3, 8), (20, 1152, 3136, 4, 1, 0), (48, 512, 12288, 4, 0, 16),
                                                  (5, 128, 65472, 2, 0, 0)])
def test_gemm_few_rows_in_as_many_slices_as_pay(M, N, K, bits, bits2, rank):
    """The slices of K that the rule chooses, in numbers that are no power of two and down to a tile a wavefront:
    against the oracle, and repeats bit for bit (the last arrival adds in slice order)."""
    w = make_weight(N, K, bits, 128, seed=M + K, bits2=bits2, rank=rank, bias=True, device=DEV)
    x = make_x(M, K, seed=M)
    y = _dual(w, x)
    assert gemm_rows(M, (N, K, bits, bits2, 128)) <= 32
    assert rel_l2(y.cpu(), _exact(w, x).half()) <= TOL
    for _ in range(3):
        assert torch.equal(_dual(w, x), y)


DUAL = [
    # M, N, K, bits, gs, bits2, rank, bias
    (8, 512, 1024, 4, 128, 1, 0, False),
    (16, 512, 1024, 1, 128, 4, 0, True),
    (16, 512, 1024, 3, 128, 3, 16, True),
    (4, 512, 1024, 2, 64, 3, 0, False),
    (12, 512, 1024, 4, 128, 4, 4, False),
    (16, 256, 2048, 4, 512, 0, 64, True),
    (5, 256, 1024, 4, 16, 2, 256, False),
    (40, 256, 1024, 4, 128, 2, 8, True),               # beyond upstream's M <= 16
]


@pytest.mark.parametrize("M,K", [(2, 64), (15, 448), (16, 512), (17, 576), (33, 4160), (16, 12288), (16, 12352), (5, 16448)])
def test_gemm_scales_found_by_the_workgroups_match_the_pre_pass(tuning_env, M, K):
    """bfloat16 rows in front of a float16 LUT in 16-row workgroups, below and above the size up to which
    the workgroups look for the scales themselves: the same bits as with the scales of the pre-pass."""
    tuning_env("FLUTE_GEMM_ROWS", "16")
    w = make_weight(256, K, 4, 128, seed=K, device=DEV)
    x = make_x(M, K, seed=M, dtype=torch.bfloat16)
    x[0] *= 1e30
    x[M // 2] *= 1e-30
    if M > 2:
        x[M - 1] = 0
    if M > 4:
        x[3, K - 1] = float("inf")

    def run():
        return fx.qgemm_per_group_lut(x.to(DEV), w["blob_d"], w["lut_d"], bitwidth=4, group_size=128,
                                      indices_layout="idx4")
    direct = run()
    tuning_env("FLUTE_GEMM_NO_DIRECT", "1")
    assert torch.equal(direct.nan_to_num(7.0), run().nan_to_num(7.0))
    # row by row: a scale that both ways get wrong would be lost beside rows of 1e30.  A row's norm bears sixteen
    # of its 256 values rounding the other way (2^-8 of a value each, 2^-12 of the norm); a wrong scale is a factor of 2
    want = _exact(w, x).bfloat16()
    for m in torch.isfinite(x).all(dim=1).nonzero().flatten().tolist():
        assert rel_l2(direct[m].cpu(), want[m]) <= TOL, m


@pytest.mark.parametrize("M,N,K,bits,gs,bits2,rank,bias", DUAL)
def test_gemm_dual_stream_fp16(M, N, K, bits, gs, bits2, rank, bias):
    w = make_weight(N, K, bits, gs, seed=M + N + bits2, bits2=bits2, rank=rank, bias=bias,
                    device=DEV)
    x = make_x(M, K, seed=13)
    y = _dual(w, x).cpu()
    assert y.shape == (M, N)
    assert rel_l2(y, _exact(w, x).half()) <= TOL
    assert torch.equal(y, _dual(w, x).cpu())


@pytest.mark.parametrize("bits,bits2", [(4, 0), (3, 0), (2, 0), (1, 0), (4, 1), (1, 4), (3, 3), (2, 4), (3, 2), (4, 4), (1, 2),
                                        (1, 1), (2, 2), (1, 3), (4, 3)])
@pytest.mark.parametrize("M,N,K,gs,rows,slices", [
    (1, 128, 64, 128, "16", None),      # one tile of K: seven wavefronts without one
    (16, 256, 576, 16, "16", "2"),      # nine tiles in slices of five and four
    (17, 128, 1088, 64, "16", "3"),     # the second block holds one row
    (31, 256, 704, 32, "32", None),     # eleven tiles over eight wavefronts
    (33, 384, 1024, 256, "32", "4"),    # two tiles share a LUT row, the last has its own
])
def test_gemm_few_row_workgroups(tuning_env, M, N, K, gs, rows, slices, bits, bits2):
    """16- and 32-row workgroups, every width alone and the pairs of one launch and of two, at the
    edges of their tiles.  The sums are fp32 over exact 16-bit weights, so what is left is the one
    rounding of the output (2^-11 of a value at most): TOL."""
    tuning_env("FLUTE_GEMM_ROWS", rows)
    if slices:
        tuning_env("FLUTE_GEMM_KSPLIT", slices)
    w = make_weight(N, K, bits, gs, seed=M + bits, bits2=bits2, rank=8, bias=True, device=DEV)
    x = make_x(M, K, seed=5)
    y = _dual(w, x).cpu()
    assert rel_l2(y, _exact(w, x).half()) <= TOL
    assert torch.equal(y, _dual(w, x).cpu())


@pytest.mark.parametrize("lut_dtype,act_dtype", [(torch.bfloat16, torch.bfloat16),
                                                 (torch.float16, torch.bfloat16)])
def test_gemm_dtype_mixes(lut_dtype, act_dtype):
    M, N, K = 48, 512, 2048
    w = make_weight(N, K, 4, 128, seed=5, lut_dtype=lut_dtype, act_dtype=act_dtype, bias=True,
                    device=DEV)
    x = make_x(M, K, seed=3, dtype=act_dtype)
    y = _dual(w, x).cpu()
    assert y.dtype == act_dtype
    ref = _exact(w, x).to(act_dtype)                   # the reference forward uses x.float()
    tol = TOL if act_dtype == torch.float16 else TOL_BF16
    assert rel_l2(y, ref) <= tol


@pytest.mark.parametrize("rows", [None, "16", "32", "64", "256"])
@pytest.mark.parametrize("M,K,bits2,rank", [(1, 64, 0, 0), (16, 1088, 3, 0), (17, 576, 0, 16), (40, 1024, 1, 5), (33, 2048, 4, 24)])
def test_gemm_float16_rows_in_front_of_a_bfloat16_lut(tuning_env, rows, M, K, bits2, rank):
    """The C entry points round such rows to the LUT's type on their way to the matrix cores, in every workgroup
    shape; the residual takes the rows as they are.  (The bindings and the module layer keep the pair away.)"""
    import ctypes
    from flute_extended import _lib
    if rows:
        tuning_env("FLUTE_GEMM_ROWS", rows)
    w = make_weight(256, K, 4, 128, seed=M, bits2=bits2, rank=rank, lut_dtype=torch.bfloat16, device=DEV)
    x = make_x(M, K, seed=K)
    d = _lib.FluteLinear()
    d.q1, d.lut1, d.q1_bytes, d.b1 = w["blob_d"].data_ptr(), w["lut_d"].data_ptr(), w["blob_d"].numel(), 4
    if bits2:
        d.q2, d.lut2, d.q2_bytes, d.b2 = w["blob2_d"].data_ptr(), w["lut2_d"].data_ptr(), w["blob2_d"].numel(), bits2
    if rank:
        d.resB, d.resA, d.R = w["resB_d"].data_ptr(), w["resA_d"].data_ptr(), rank
    d.N, d.K, d.group_size, d.lut_rows, d.lut_dtype = 256, K, 128, 2, _lib.BF16
    xd = x.to(DEV)
    ds, outs = (_lib.FluteLinear * 2)(d, d), [torch.zeros(M, 256, dtype=torch.float16, device=DEV) for _ in range(3)]
    stream = torch.cuda.current_stream().cuda_stream
    assert _lib.lib.flute_gemm(ctypes.byref(d), xd.data_ptr(), outs[0].data_ptr(), M, K, 256, _lib.F16, stream) == 0
    assert _lib.lib.flute_gemm_multi(ds, 2, xd.data_ptr(), (ctypes.c_void_p * 2)(*[o.data_ptr() for o in outs[1:]]),
                                     (ctypes.c_int64 * 2)(256, 256), M, K, _lib.F16, stream) == 0
    want = _exact(dict(w, resA=None, resB=None), x.bfloat16()).double()
    if rank:
        want = want + (x.double() @ w["resB"].double().t()) @ w["resA"].double().t()
    for y in outs:
        assert rel_l2(y.cpu(), want.half()) <= TOL


@pytest.mark.parametrize("bits,gs", [(4, 128), (3, 64), (2, 16), (1, 128), (4, 32)])
def test_gemm_one_hot_rows_return_dequantised_columns(bits, gs):
    N, K = 256, 128
    w = make_weight(N, K, bits, gs, seed=bits * 7 + gs, device=DEV)
    eye = torch.eye(K, dtype=torch.float16)             # M = K = 128 one-hot rows
    y = fx.qgemm_per_group_lut(eye.to(DEV), w["blob_d"], w["lut_d"], bitwidth=bits,
                               group_size=gs, indices_layout=f"idx{bits}").cpu()
    W = O.dequant(w["blob"].numpy(), w["lut"], N, K, gs, bits)       # [N, K] fp32 of fp16 values
    assert torch.equal(y, W.t().half())


def test_gemm_matches_gemv_rows():
    """Row m of the GEMM equals the M = 1 kernel on that row up to summation order."""
    N, K = 512, 4096
    w = make_weight(N, K, 4, 128, seed=21, device=DEV)
    x = make_x(8, K, seed=2)
    y = _dual(w, x).cpu()
    for m in (0, 7):
        ym = fx.qgemm_gemv_splitk_stream(x[m:m + 1].to(DEV), w["blob_d"], w["lut_d"], 4, 128).cpu()
        assert rel_l2(y[m:m + 1], ym) <= TOL


def test_gemm_strided_views_and_empty():
    N, K = 256, 512
    w = make_weight(N, K, 4, 128, seed=9, device=DEV)
    x = make_x(24, K, seed=4)
    y = _dual(w, x).cpu()
    assert torch.equal(_dual(w, x[:0]).cpu(), torch.zeros(0, N, dtype=torch.float16))
    assert torch.equal(_dual(w, x[3:19]).cpu(), _dual(w, x[3:19].clone()).cpu())
    assert rel_l2(_dual(w, x[3:19]).cpu(), y[3:19]) <= TOL   # same rows through another shape


def test_gemm_full_size_linearity():
    """At the benchmark's full shape the oracle is too slow; use linearity instead:
    gemm(a*x1 + x2) == a*gemm(x1) + gemm(x2) within rounding, and row consistency
    between M = 256 and M = 16 launches (different shapes of the same kernel)."""
    N, K = 12288, 4096
    gen = torch.Generator(device=DEV).manual_seed(0)
    blob = torch.randint(0, 256, (N * K // 2,), dtype=torch.uint8, device=DEV, generator=gen)
    lut = (torch.randn(N // 128, 16, device=DEV, generator=gen) * 0.02).sort(dim=1).values.half()
    x = torch.randn(256, K, device=DEV, generator=gen).half()
    run = lambda a: fx.qgemm_per_group_lut(a, blob, lut, bitwidth=4, group_size=128,
                                           indices_layout="idx4")
    y = run(x)
    y16 = run(x[32:48])
    assert rel_l2(y[32:48], y16) <= TOL
    y1 = fx.qgemm_gemv_splitk_stream(x[5:6], blob, lut, 4, 128)
    assert rel_l2(y[5:6], y1) <= TOL
    z = run((2.0 * x[:64].float() + x[64:128].float()).half())
    assert rel_l2(z, 2.0 * y[:64].float() + y[64:128].float()) <= 3e-3


@pytest.mark.parametrize("N,K,M,lut_dtype", [(12288, 4096, 256, torch.bfloat16), (4096, 12288, 256, torch.bfloat16),
                                             (12288, 4096, 1024, torch.float16), (1024, 4096, 200, torch.bfloat16)])
def test_lean_loop_is_bit_identical_to_the_scheduled_loop(tuning_env, N, K, M, lut_dtype):
    """Four-block workgroups run the loop with hand-written loads and waits by default and the
    compiler-scheduled loop under FLUTE_GEMM_NO_LEAN=1: same sums in the same order, so the
    outputs must be equal bit for bit.  Full benchmark shapes: the blobs are large enough for tile
    addresses with bit 31 set to occur."""
    gen = torch.Generator(device=DEV).manual_seed(N + K + M)
    blob = torch.randint(0, 256, (N * K // 2,), dtype=torch.uint8, device=DEV, generator=gen)
    lut = (torch.randn(N // 128, 16, device=DEV, generator=gen) * 0.02).sort(dim=1).values.to(lut_dtype)
    x = torch.randn(M, K, device=DEV, generator=gen).bfloat16()
    run = lambda: fx.qgemm_per_group_lut(x, blob, lut, bitwidth=4, group_size=128, indices_layout="idx4")
    if M >= 1000:                                       # (the rule gives it to the many-row kernel)
        tuning_env("FLUTE_GEMM_ROWS", "128")
    elif N == 1024:                                     # (and this one to 16-row workgroups)
        tuning_env("FLUTE_GEMM_ROWS", "64")
    assert gemm_rows(M, (N, K, 4, 0, 128)) in (64, 128)
    lean = run()
    tuning_env("FLUTE_GEMM_NO_LEAN", "1")
    scheduled = run()
    tuning_env("FLUTE_GEMM_NO_LEAN", None)
    assert torch.equal(lean, scheduled)
    y1 = fx.qgemm_gemv_splitk_stream(x[7:8], blob, lut, 4, 128)        # and against the M = 1 kernel
    assert rel_l2(lean[7:8], y1) <= 4e-3                               # (bf16 outputs: one rounding each)


@pytest.mark.parametrize("N,K,M,rot", [(12288, 4096, 256, False), (4096, 12288, 256, False), (4096, 12288, 200, True),
                                       (12288, 4096, 1000, True), (1024, 4096, 300, True)])
def test_hand_overs_between_the_k_ways_equal_the_tree(tuning_env, N, K, M, rot):
    """Workgroups of four-block wavefronts end with hand-overs between their k ways (the activation
    image is written with the blocks in the order those expect) and, under FLUTE_GEMM_NO_HANDOVER=1,
    with the reduction tree over the image in plain order: the same additions, so equal bit for
    bit, whether the image comes from the pre-pass or from the rotation that writes it itself,
    with ragged M, four k ways (K = 4096) and eight (K = 12288)."""
    import ctypes
    from flute_extended import _lib
    import fht
    gen = torch.Generator(device=DEV).manual_seed(N + K + M)
    blob = torch.randint(0, 256, (N * K // 2,), dtype=torch.uint8, device=DEV, generator=gen)
    lut = (torch.randn(N // 128, 16, device=DEV, generator=gen) * 0.02).sort(dim=1).values.bfloat16().contiguous()
    x = torch.randn(M, K, device=DEV, generator=gen).bfloat16()
    signs = O.rotation_signs(K, 3).to(DEV) if rot else None
    if N == 1024 or M >= 1000:                          # (the rule gives the latter to the many-row kernel)
        tuning_env("FLUTE_GEMM_ROWS", "128")
    assert gemm_rows(M, (N, K, 4, 0, 128)) in (64, 128)
    d = _lib.FluteLinear()
    d.q1, d.lut1, d.q1_bytes = blob.data_ptr(), lut.data_ptr(), blob.numel()
    d.N, d.K, d.b1, d.group_size, d.lut_rows, d.lut_dtype = N, K, 4, 128, N // 128, _lib.BF16
    if rot:
        d.signs = signs.data_ptr()

    def run():
        C = torch.zeros(M, N, dtype=torch.bfloat16, device=DEV)
        st = _lib.lib.flute_gemm(ctypes.byref(d), x.data_ptr(), C.data_ptr(), M, K, N, _lib.BF16,
                                 torch.cuda.current_stream().cuda_stream)
        assert st == 0, _lib.last_error()
        return C

    handed = run()
    tuning_env("FLUTE_GEMM_NO_HANDOVER", "1")
    tree = run()
    tuning_env("FLUTE_GEMM_NO_HANDOVER", None)
    assert torch.equal(handed, tree)
    xr = fht.fht_apply(x, signs, backend="kernel") if rot else x
    y1 = fx.qgemm_gemv_splitk_stream(xr[M - 1:M], blob, lut, 4, 128)   # and against the M = 1 kernel
    assert rel_l2(handed[M - 1:M], y1) <= 4e-3


@pytest.mark.parametrize("rank", [5, 16, 24])
@pytest.mark.parametrize("rows,M", [("64", 64), ("64", 130), ("128", 128), ("128", 200)])
@pytest.mark.parametrize("N,K", [(256, 1024), (1024, 4096)])
def test_hand_overs_beside_a_residual_equal_the_tree(tuning_env, N, K, rows, M, rank):
    """One stream in one slice of K: the residual's tile takes memory that the k ways have just handed blocks
    over in, with four k ways (128 rows) and eight (64).  The bits of the reduction tree, which does not use that
    memory, and the oracle's values, row by row (a block overwritten early would be lost in a launch-wide norm)."""
    tuning_env("FLUTE_GEMM_ROWS", rows)
    tuning_env("FLUTE_GEMM_KSPLIT", "1")
    w = make_weight(N, K, 4, 128, seed=M + rank, rank=rank, bias=True, device=DEV)
    x = make_x(M, K, seed=rank)
    handed = _dual(w, x)
    tuning_env("FLUTE_GEMM_NO_HANDOVER", "1")
    assert torch.equal(handed, _dual(w, x))
    want = _exact(w, x).half()
    assert max(rel_l2(y, v) for y, v in zip(handed.cpu(), want)) <= TOL


@pytest.mark.parametrize("kind", ["outliers", "tiny", "huge", "mixed"])
@pytest.mark.parametrize("M,rows", [(8, None), (40, None), (130, "64"), (300, "128")])
def test_gemm_bf16_activations_beyond_the_float16_range(tuning_env, kind, M, rows):
    """bfloat16 rows that float16 cannot hold (|x| > 65504 or < 6e-8) in front of a float16
    LUT: every row is scaled by its own power of two before it meets the matrix cores and
    scaled back afterwards, so the result is the reference forward's (x.float() @ W.t()),
    never inf or 0.  Rows of very different magnitude share a launch."""
    if rows:
        tuning_env("FLUTE_GEMM_ROWS", rows)
    N, K = 256, 1024
    w = make_weight(N, K, 4, 128, seed=29, act_dtype=torch.bfloat16, device=DEV)
    x = make_x(M, K, seed=31, dtype=torch.float32)
    if kind == "outliers":
        x[::3, 5] = 1.0e5
        x[1, K - 1] = -3.0e5
    elif kind == "tiny":
        x *= 1.0e-7
    elif kind == "huge":
        x[: M // 2] *= 1.0e30
    else:
        x[::2] *= 1.0e-6
        x[1::2, ::64] *= 1.0e5
    x = x.to(torch.bfloat16)
    y = _dual(w, x).cpu()
    assert torch.isfinite(y).all()
    ref = O.linear_reference(x, w["blob"].numpy(), w["lut"], N, K, 128, 4)   # same rounding point
    assert torch.isfinite(ref).all()
    # row by row: a launch-wide norm would let the large rows hide the small ones
    for m in range(M):
        assert rel_l2(y[m], ref[m]) <= TOL, f"row {m}"


@pytest.mark.parametrize("bits,gs", [(1, 128), (2, 64), (3, 128), (4, 128), (4, 16), (3, 32)])
def test_scalar_twin_differential_chain(bits, gs):
    """Upstream's differential chain (test_flute.py:172-223): the fast kernel on the idxN
    blob, the scalar twin on the LOGICAL packed rows and the twin on the blob.  The twin
    shares no code with the fast path (one thread per output, bit-position decode, LUT in
    global memory), so agreement means both read the format the same way: the two twin
    layouts must agree bit for bit (same sums in the same order), twin and fast kernel
    within fp32 reassociation, and all three exactly on one-hot rows."""
    M, K, N = 64, 512, 256
    w = make_weight(N, K, bits, gs, seed=43 + bits, device=DEV)
    logical = torch.from_numpy(O.logical_packed_rows(w["idx"].numpy(), bits)).to(DEV)
    assert logical.shape == (N, K * bits // 8)
    x = make_x(M, K, seed=44).to(DEV)
    fast = fx.qgemm_per_group_lut(x, w["blob_d"], w["lut_d"], bitwidth=bits, group_size=gs,
                                  indices_layout=f"idx{bits}")
    twin = fx.qgemm_per_group_lut(x, logical, w["lut_d"], bitwidth=bits, group_size=gs,
                                  backend="debug_simple", indices_layout=f"idx{bits}")
    twin_blob = fx.qgemm_debug_simple(x, w["blob_d"], w["lut_d"], bits, gs, q_layout=1)
    assert torch.equal(twin, twin_blob)
    assert rel_l2(fast.cpu(), twin.cpu()) <= 5e-4
    assert rel_l2(twin.cpu(), _exact(w, x.cpu()).half()) <= TOL
    eye = torch.eye(K, dtype=torch.float16, device=DEV)
    W = O.dequant(w["blob"].numpy(), w["lut"], N, K, gs, bits).t().half()
    assert torch.equal(fx.qgemm_debug_simple(eye, logical, w["lut_d"], bits, gs).cpu(), W)
    assert torch.equal(fx.qgemm_debug_simple(eye, w["blob_d"], w["lut_d"], bits, gs, q_layout=1).cpu(), W)
    assert torch.equal(fx.qgemm_per_group_lut(eye, w["blob_d"], w["lut_d"], bitwidth=bits,
                                              group_size=gs, indices_layout=f"idx{bits}").cpu(), W)


def test_scalar_twin_refusals_and_bf16():
    w = make_weight(256, 128, 4, 128, seed=47, lut_dtype=torch.bfloat16, device=DEV)
    x = make_x(3, 128, seed=48, dtype=torch.bfloat16).to(DEV)
    y = fx.qgemm_debug_simple(x, w["blob_d"], w["lut_d"], 4, 128, q_layout=1)
    assert y.dtype == torch.bfloat16
    assert rel_l2(y.cpu(), _exact(w, x.cpu()).bfloat16()) <= TOL
    with pytest.raises(RuntimeError):
        fx.qgemm_debug_simple(x, w["blob_d"][:-1], w["lut_d"], 4, 128)        # truncated
    with pytest.raises(RuntimeError):
        fx.qgemm_debug_simple(x, w["blob_d"], w["lut_d"][:, :8], 4, 128)      # wrong LUT width
    with pytest.raises(RuntimeError):
        fx.qgemm_debug_simple(x, w["blob_d"], w["lut_d"], 5, 128)


# ---- many rows: every weight looked up once per workgroup (gemm_wide_kernel.h) ------------------
WIDE = [
    # M, N, K, bits, gs, bits2, rank, bias, lut, act
    (1, 128, 64, 4, 128, 0, 0, False, torch.float16, torch.float16),       # one tile, one row
    (33, 384, 192, 4, 64, 0, 0, True, torch.bfloat16, torch.bfloat16),     # odd number of tiles
    (257, 256, 320, 4, 16, 0, 0, False, torch.float16, torch.float16),     # eight LUT groups a tile
    (513, 256, 512, 3, 128, 0, 5, False, torch.float16, torch.float16),    # one row past a workgroup
    (511, 256, 448, 2, 32, 0, 0, False, torch.bfloat16, torch.bfloat16),
    (130, 128, 1088, 1, 256, 0, 0, True, torch.float16, torch.float16),
    (300, 256, 512, 4, 128, 1, 16, True, torch.float16, torch.float16),
    (300, 256, 512, 1, 128, 4, 0, False, torch.bfloat16, torch.bfloat16),  # the wider stream second
    (100, 256, 576, 3, 64, 3, 40, False, torch.bfloat16, torch.bfloat16),  # ranks beyond one 32-wide step
    (300, 256, 512, 2, 16, 4, 0, False, torch.float16, torch.float16),
    (300, 256, 448, 2, 256, 3, 0, False, torch.float16, torch.bfloat16),   # rows scaled into float16
    (70, 512, 512, 4, 64, 4, 8, True, torch.float16, torch.bfloat16),      # two 32 KB tables
    (130, 256, 512, 1, 64, 1, 0, False, torch.float16, torch.float16),
    (130, 256, 512, 3, 128, 1, 0, False, torch.float16, torch.bfloat16),
]


@pytest.mark.parametrize("rows,slices", [("512", None), ("256", None), ("512", "3"), ("256", "5")])
@pytest.mark.parametrize("M,N,K,bits,gs,bits2,rank,bias,lut,act", WIDE)
def test_gemm_many_row_workgroups(tuning_env, rows, slices, M, N, K, bits, gs, bits2, rank, bias, lut, act):
    """The many-row kernel at the edges of its tiles, forced with FLUTE_GEMM_ROWS = 512 / 256, with
    and without slices of K (FLUTE_GEMM_KSPLIT), against the closed form; repeats bit identical.
    One rounding of an fp32 sum to the output type: 2^-12 of a value at most in float16, 2^-9 in
    bfloat16, the tolerances of this file."""
    tuning_env("FLUTE_GEMM_ROWS", rows)
    if slices:
        tuning_env("FLUTE_GEMM_KSPLIT", slices)
    w = make_weight(N, K, bits, gs, seed=M + N + K + bits, bits2=bits2, rank=rank, bias=bias, lut_dtype=lut,
                    act_dtype=act, device=DEV)
    x = make_x(M, K, seed=43, dtype=act)
    y = _dual(w, x)
    assert rel_l2(y.cpu(), _exact(w, x).to(act)) <= (TOL if act == torch.float16 else TOL_BF16)
    assert torch.equal(y, _dual(w, x))


@pytest.mark.parametrize("rot", [False, True])
@pytest.mark.parametrize("M,N,K,bits2,rows", [(1100, 12288, 1024, 0, 256), (600, 4096, 4096, 1, 256), (600, 12288, 512, 1, 512)])
def test_gemm_many_rows_by_the_rule_agree_with_the_other_kernels(tuning_env, M, N, K, bits2, rows, rot):
    """Sizes the launcher gives to the many-row kernel by itself, plain and rotated, against the 128-row
    workgroups: the same fp32 sums in another order, one rounding."""
    w = make_weight(N, K, 4, 128, seed=3, bits2=bits2, rank=16, bias=True, device=DEV)
    x = make_x(M, K, seed=5).to(DEV)
    signs = O.rotation_signs(K, 3).to(DEV) if rot else None
    shape = (N, K, 4, bits2, 128)

    def run():
        return fx.qgemm_linear(x, w["blob_d"], w["lut_d"], 4, w.get("blob2_d"), w.get("lut2_d"), bits2, w["resB_d"],
                               w["resA_d"], w["bias_d"], 128, signs, None).cpu()
    assert gemm_rows(M, shape) == rows
    y = run()
    tuning_env("FLUTE_GEMM_ROWS", "128")
    assert gemm_rows(M, shape) == 128
    assert rel_l2(y, run()) <= TOL


@pytest.mark.parametrize("rank", [5, 8, 24])
@pytest.mark.parametrize("M,K", [(2, 64), (17, 2048), (40, 8192), (33, 12288), (300, 4096)])
@pytest.mark.parametrize("form", ["f16", "bf16 over f16", "bf16 over f16, rotated"])
@pytest.mark.parametrize("rows", [None, "256", "512"])
def test_gemm_residual_slices_and_row_scales(tuning_env, rows, M, K, rank, form):
    """Residual coefficients in one, four and sixteen slices of K, and those that the few-row kernel forms; ranks
    that are loaded four at a time (multiples of four) and one by one; row scales found by the rotation, by the
    workgroups and by the launch in front, rows over a wide range of magnitudes; the small-M kernels and both
    workgroups of the many-row kernel."""
    if rows:
        tuning_env("FLUTE_GEMM_ROWS", rows)
    N, act = 256, torch.float16 if form == "f16" else torch.bfloat16
    w = make_weight(N, K, 4, 128, seed=M + K + rank, bits2=1, rank=rank, act_dtype=act, device=DEV)
    x = make_x(M, K, seed=M, dtype=act)
    if act is torch.bfloat16:
        x = x * torch.logspace(-6, 6, M).unsqueeze(1).to(act)
    signs = O.rotation_signs(K, 3) if "rotated" in form else None
    y = fx.qgemm_linear(x.to(DEV), w["blob_d"], w["lut_d"], 4, w["blob2_d"], w["lut2_d"], 1, w["resB_d"],
                        w["resA_d"], None, 128, None if signs is None else signs.to(DEV), None).cpu()
    ref = _exact(w, x if signs is None else O.fht_reference(x, signs))
    scale = ref.abs().amax(dim=1, keepdim=True)
    assert rel_l2(y.double() / scale, ref / scale) <= (TOL if act is torch.float16 else TOL_BF16)


@pytest.mark.parametrize("rank", [7, 20, 21])
@pytest.mark.parametrize("rows", ["512", "256", "128"])
@pytest.mark.parametrize("act", [torch.float16, torch.bfloat16])
def test_gemm_residual_coefficients_of_very_different_magnitude(tuning_env, rows, rank, act):
    """Ranks whose coefficients fall by 2^20 and whose resA grows by as much, so that each adds the same
    to the output: the coefficients are fp32 and stay so in every kernel.  With a zero LUT the output
    is the residual alone, fp32 sums rounded once.  The 128-row workgroups sum the fp32 products sixteen ranks a
    step in a tile of their own, the many-row kernel in its accumulators, so the two may differ by a rounding."""
    M, N, K = 130, 256, 512
    tuning_env("FLUTE_GEMM_ROWS", rows)
    w = make_weight(N, K, 4, 128, seed=7, act_dtype=act, device=DEV)
    g = torch.Generator().manual_seed(rank)
    step = torch.logspace(0, -20, rank, base=2.0)
    resB = (torch.randn(rank, K, generator=g) * 64 * step.unsqueeze(1)).to(act)
    resA = (torch.randn(N, rank, generator=g) * 0.004 / step).to(act)
    x = make_x(M, K, seed=rank, dtype=act)

    def run():
        return fx.qgemm_linear(x.to(DEV), w["blob_d"], w["lut_d"] * 0, 4, None, None, 0, resB.to(DEV),
                               resA.to(DEV), None, 128, None, None).cpu()
    want = (x.double() @ resB.double().t()) @ resA.double().t()
    y = run()
    assert rel_l2(y, want) <= (TOL if act is torch.float16 else TOL_BF16)
    # against the rounded 64-bit result: 2 % of the values may round the other way (fp32 sums are off
    # by 2^-20 of a value or less, a rounding step is 2^-10 or 2^-7 of it)
    assert (y != want.to(act)).float().mean() <= 0.02


@pytest.mark.parametrize("rows", ["512", "256"])
def test_gemm_residual_of_infinite_operands(tuning_env, rows):
    """An overflowing coefficient and an infinite entry of resA give the infinities and NaN that fp32
    products give, in their rows and columns and nowhere else."""
    M, N, K, rank, act = 40, 256, 256, 6, torch.bfloat16
    w = make_weight(N, K, 4, 128, seed=9, act_dtype=act, rank=rank, device=DEV)
    x = make_x(M, K, seed=3, dtype=act)
    x[5] = 1.0e30
    resB, resA = w["resB"].clone(), w["resA"].clone()
    resB[2] = 1.0e30
    x[:5, 0] += 1
    resA[17, 4] = float("inf")
    run = lambda: fx.qgemm_linear(x.to(DEV), w["blob_d"], w["lut_d"], 4, None, None, 0, resB.to(DEV), resA.to(DEV),
                                  None, 128, None, None).cpu().float()
    tuning_env("FLUTE_GEMM_ROWS", "128")
    want = run()
    tuning_env("FLUTE_GEMM_ROWS", rows)
    y = run()
    assert torch.isinf(want[5]).any() and torch.isinf(want[:, 17]).any()
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isinf(y), torch.isinf(want))
    assert torch.equal(torch.sign(y[torch.isinf(y)]), torch.sign(want[torch.isinf(want)]))


@pytest.mark.parametrize("M,K,rows", [(2, 64, None), (17, 2048, "32"), (33, 12288, "32"), (70, 4160, "64"), (300, 1088, "256"),
                                      (513, 16384, "512"), (40, 16448, "32"), (9, 20480, None)])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("rank", [0, 20])
def test_gemm_pre_pass_of_scaled_rows(tuning_env, M, K, rows, offset, rank):
    """Row scales, image and coefficients of bfloat16 rows over a float16 LUT in one launch: rows of
    every magnitude, the last group of four partly past the end, K at and beyond what a workgroup holds
    of four rows, rows that are not 16-byte aligned (the kernels of their own).  Products are exact in
    fp32 and scales powers of two, so a row is off by its one rounding to bfloat16: 2^-9 of a value."""
    if rows:
        tuning_env("FLUTE_GEMM_ROWS", rows)
    N = 256
    w = make_weight(N, K, 4, 128, seed=M + K, rank=rank, act_dtype=torch.bfloat16, device=DEV)
    x = make_x(M, K, seed=5, dtype=torch.bfloat16) * (2.0 ** torch.randint(-60, 60, (M, 1))).to(torch.bfloat16)
    flat = torch.zeros(M * K + 8, dtype=torch.bfloat16, device=DEV)
    xd = flat[offset:offset + M * K].reshape(M, K)
    xd.copy_(x)
    y = _dual(w, xd).cpu().double()
    want = _exact(w, x).double()
    assert bool(((y - want).norm(dim=1) <= 2.0 ** -8 * want.norm(dim=1)).all())


@pytest.mark.parametrize("M", [3, 16, 17, 40])
@pytest.mark.parametrize("rank", [1, 15, 17, 256])
@pytest.mark.parametrize("exponent", [-100, 0, 100])
def test_gemm_few_rows_residual_far_from_its_row(M, rank, exponent):
    """Rows held scaled by 2^exponent, a residual 2^-exponent of them and a zero LUT: the residual is
    added at its own magnitude (scaled with its row it would leave the range of fp32).  fp32 sums over K and
    the ranks are off by (K + rank) * 2^-24 of the sum of magnitudes, the rounding by 2^-9 of a value."""
    N, K, act = 256, 1088, torch.bfloat16
    w = make_weight(N, K, 4, 128, seed=M + rank, act_dtype=act, device=DEV)
    g = torch.Generator().manual_seed(M * rank)
    x = torch.ldexp(torch.randn(M, K, generator=g), torch.tensor(exponent)).to(act)
    resB = torch.ldexp(torch.randn(rank, K, generator=g), torch.tensor(-exponent)).to(act)
    resA = torch.ldexp(torch.randn(N, rank, generator=g), torch.tensor(-exponent // 2)).to(act)
    y = fx.qgemm_linear(x.to(DEV), w["blob_d"], w["lut_d"] * 0, 4, None, None, 0, resB.to(DEV), resA.to(DEV),
                        None, 128, None, None).cpu().double()
    xb, a = x.double() @ resB.double().t(), resA.double().t()
    magnitude = (x.double().abs() @ resB.double().abs().t()) @ a.abs()
    assert bool(((y - xb @ a).abs() <= 2.0 ** -8 * (xb @ a).abs() + (K + rank) * 2.0 ** -24 * magnitude).all())


@pytest.mark.parametrize("M,rows,slices", [(3, "16", "1"), (17, "16", "2"), (40, "32", "1"), (40, "32", "2")])
def test_gemm_few_rows_residual_of_rows_at_the_end_of_the_range(tuning_env, M, rows, slices):
    """Rows of 2^127 whose partial sums leave the range of fp32 and whose sums do not: the odd tiles of K
    take back what the even ones add, up to one element of half the size.  fp32 sums over K and the ranks
    are off by (K + rank) * 2^-24 of the sum of magnitudes, the rounding by 2^-9 of a value."""
    tuning_env("FLUTE_GEMM_ROWS", rows)
    tuning_env("FLUTE_GEMM_KSPLIT", slices)
    N, K, rank, act = 256, 1024, 8, torch.bfloat16
    w = make_weight(N, K, 4, 128, seed=M, act_dtype=act, device=DEV)
    sign = 1.0 - 2.0 * (torch.arange(K) // 64 % 2)
    x = (sign * 2.0 ** 127).repeat(M, 1).to(act)
    x[:, 0] = 2.0 ** 126
    g = torch.Generator().manual_seed(M)
    resB = torch.ldexp(torch.randn(rank, K, generator=g), torch.tensor(-127)).to(act)
    resA = torch.ldexp(torch.randn(N, rank, generator=g), torch.tensor(117)).to(act)
    y = fx.qgemm_linear(x.to(DEV), w["blob_d"], torch.ones_like(w["lut_d"]), 4, None, None, 0, resB.to(DEV),
                        resA.to(DEV), None, 128, None, None).cpu().double()
    xb, a = x.double() @ resB.double().t(), resA.double().t()
    want = x.double().sum(dim=1, keepdim=True) + xb @ a
    magnitude = (x.double().abs() @ resB.double().abs().t()) @ a.abs()
    assert bool(((y - want).abs() <= 2.0 ** -8 * want.abs() + (K + rank) * 2.0 ** -24 * magnitude).all())
