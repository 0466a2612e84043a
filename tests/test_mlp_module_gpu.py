"""GPU parity of the merged gate/up launch, the grouped launch, the MLP block
and the module layer's kernel mode against the oracle / the reference mode."""
import ctypes

import pytest
import torch

import flute_extended as fx
import flute_oracle as O
import palettized_modules as pm
from flute_extended import _lib
from _util import gemm_rows, make_weight, make_x, rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = 1e-3


def _row(w, out=None, signs=None, awq=None):
    p = lambda t: 0 if t is None else t.data_ptr()
    return [p(w["blob_d"]), p(w["lut_d"]), p(w.get("blob2_d")), p(w.get("lut2_d")),
            p(w.get("resB_d")), p(w.get("resA_d")), p(w.get("bias_d")), p(out), w["N"],
            0 if w["resB"] is None else w["resB"].shape[0], w["bits"], w["bits2"], w["gs"],
            p(signs), p(awq)]


def _exact(w, x):
    return O.linear_exact(x, w["blob"].numpy(), w["lut"], w["N"], w["K"], w["gs"], w["bits"],
                          w["blob2"].numpy() if w["bits2"] else None, w["lut2"], w["bits2"],
                          w["resA"], w["resB"], w["bias"])


@pytest.mark.parametrize("gspec,uspec", [
    (dict(bits=4), dict(bits=4)),
    (dict(bits=4, bits2=1, gs=64), dict(bits=1, bits2=4, rank=8, bias=True)),
    (dict(bits=3, gs=32), dict(bits=2, rank=4)),
])
def test_merged_gate_up_silu(gspec, uspec):
    N, K = 1024, 2048
    g = make_weight(N, K, seed=1, device=DEV, **gspec)
    u = make_weight(N, K, seed=2, device=DEV, **uspec)
    x = make_x(1, K, seed=3)
    out = torch.zeros(1, N, dtype=torch.float16, device=DEV)
    table = torch.tensor([_row(g), _row(u)], dtype=torch.int64)
    y = fx.qgemm_gemv_mlp(x.to(DEV), table, out)
    assert y.data_ptr() == out.data_ptr()
    ref = O.silu_mul_exact(_exact(g, x), _exact(u, x)).half()
    assert rel_l2(y.cpu(), ref) <= TOL
    y1 = y.clone()
    fx.qgemm_gemv_mlp(x.to(DEV), table, out)
    assert torch.equal(out, y1)


def test_merged_gate_up_with_different_rotations():
    N, K = 512, 4096
    g = make_weight(N, K, seed=1, device=DEV)
    u = make_weight(N, K, seed=2, device=DEV)
    x = make_x(1, K, seed=3)
    sg, su = O.rotation_signs(K, 1).to(DEV), O.rotation_signs(K, 2).to(DEV)
    out = torch.zeros(1, N, dtype=torch.float16, device=DEV)
    table = torch.tensor([_row(g, signs=sg), _row(u, signs=su)], dtype=torch.int64)
    y = fx.qgemm_gemv_mlp(x.to(DEV), table, out).cpu()
    ref = O.silu_mul_exact(_exact(g, O.fht_reference(x, sg.cpu())),
                           _exact(u, O.fht_reference(x, su.cpu()))).half()
    assert rel_l2(y, ref) <= TOL


@pytest.mark.parametrize("rank", [0, 8])
def test_merged_gate_up_different_rotations_bfloat16_rows_float16_lut(rank):
    """bfloat16 activations in front of float16 LUTs are scaled per staged row, and a member with
    its own signs makes the launch stage the row a second time while the first output's partial
    row sums still wait in LDS: the scaling's scratch words must not be those sums.  Every gate
    row is checked (the first rows of each slice were the ones at risk), with magnitudes beyond
    float16's range so the scaling is exercised."""
    N, K = 512, 4096
    bf = torch.bfloat16
    g = make_weight(N, K, seed=11, rank=rank, act_dtype=bf, device=DEV)
    u = make_weight(N, K, seed=12, rank=rank, act_dtype=bf, device=DEV)
    x = (make_x(1, K, seed=13).float() * 3.0e5).to(bf)
    sg, su = O.rotation_signs(K, 1).to(DEV), O.rotation_signs(K, 2).to(DEV)
    out = torch.zeros(1, N, dtype=bf, device=DEV)
    table = torch.tensor([_row(g, signs=sg), _row(u, signs=su)], dtype=torch.int64)
    y = fx.qgemm_gemv_mlp(x.to(DEV), table, out).cpu()
    yg = _exact(g, O.fht_reference(x, sg.cpu()))
    yu = _exact(u, O.fht_reference(x, su.cpu()))
    ref = O.silu_mul_exact(yg, yu)
    assert torch.isfinite(y).all()
    assert rel_l2(y, ref.to(bf)) <= TOL           # same rounding point as the reference forward
    # row by row: one bfloat16 rounding (2^-9) of a value whose factors are exact to ~1e-6
    # (values far below bfloat16's normal range, where SiLU of a large negative sum underflows,
    # are left to the norm above)
    big = ref.double().abs() > 1e-30
    err = (y.double() - ref.double()).abs()[big] / ref.double().abs()[big]
    assert int(big.sum()) > N // 4 and float(err.max()) <= 2.0 ** -8
    # each member alone through the single-weight entry gives the same sums
    yg1 = fx.qgemm_gemv_stream(x.to(DEV), g["blob_d"], g["lut_d"], 4, 128, rot_signs=sg,
                               **({"resA": g["resA_d"], "resB": g["resB_d"]} if rank else {})).cpu()
    assert rel_l2(yg1, yg.to(bf)) <= TOL


def test_grouped_launch():
    K = 2048
    ws = [make_weight(512, K, seed=1, device=DEV),
          make_weight(256, K, bits=3, gs=64, bits2=3, rank=8, seed=2, device=DEV),
          make_weight(128, K, bits=2, gs=32, bias=True, seed=3, device=DEV)]
    outs = [torch.zeros(1, w["N"], dtype=torch.float16, device=DEV) for w in ws]
    x = make_x(1, K, seed=4)
    table = torch.tensor([_row(w, o) for w, o in zip(ws, outs)], dtype=torch.int64)
    assert fx.qgemm_gemv_multi(x.to(DEV), table) is None
    for w, o in zip(ws, outs):
        assert rel_l2(o.cpu(), _exact(w, x).half()) <= TOL


def _desc(w):
    d = _lib.FluteLinear()
    d.q1, d.lut1 = w["blob_d"].data_ptr(), w["lut_d"].data_ptr()
    d.q1_bytes = w["blob_d"].numel()
    d.N, d.K, d.b1, d.group_size = w["N"], w["K"], w["bits"], w["gs"]
    d.lut_rows = w["lut"].shape[0]
    d.lut_dtype = _lib.F16 if w["lut"].dtype == torch.float16 else _lib.BF16
    return d


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_mlp_block_through_the_c_abi(dtype):
    """Benchmark configuration 2 at full size: gate/up 4096 -> 12288, SiLU*mul,
    down 12288 -> 4096, called straight through flute_mlp_block."""
    H, I = 4096, 12288
    g = make_weight(I, H, seed=1, device=DEV)
    u = make_weight(I, H, seed=2, device=DEV)
    d = make_weight(H, I, seed=3, device=DEV)
    x = make_x(1, H, seed=4, dtype=dtype)
    xd = x.to(DEV)
    h = torch.zeros(1, I, dtype=dtype, device=DEV)
    y = torch.zeros(1, H, dtype=dtype, device=DEV)
    dg, du, dd = _desc(g), _desc(u), _desc(d)
    act = _lib.F16 if dtype == torch.float16 else _lib.BF16
    st = _lib.lib.flute_mlp_block(ctypes.byref(dg), ctypes.byref(du), ctypes.byref(dd),
                                  xd.data_ptr(), h.data_ptr(), y.data_ptr(), act,
                                  torch.cuda.current_stream().cuda_stream)
    assert st == 0, _lib.last_error()
    torch.cuda.synchronize()
    h_ref = O.silu_mul_exact(_exact(g, x), _exact(u, x)).to(dtype)
    tol = TOL if dtype == torch.float16 else 4e-3      # bf16: the output rounding alone is 2^-9
    assert rel_l2(h.cpu(), h_ref) <= tol
    assert rel_l2(y.cpu(), _exact(d, h.cpu()).to(dtype)) <= tol


def _modules(w, **kw):
    args = dict(bias=w["bias"], resA=w["resA"], resB=w["resB"], indices2=w["blob2"],
                lut2=w["lut2"], bitwidth2=w["bits2"] or None)
    args.update(kw)
    ref = pm.PalettizedLinear(w["blob"], w["lut"], w["bits"], w["gs"], w["N"], w["K"],
                              reference=True, **args)
    ker = pm.PalettizedLinear(w["blob"], w["lut"], w["bits"], w["gs"], w["N"], w["K"],
                              reference=False, **args).to(DEV)
    return ref, ker


@pytest.mark.parametrize("spec", [dict(), dict(bits2=2, rank=8, bias=True), dict(bits=3, gs=32)])
@pytest.mark.parametrize("rot", [False, True])
def test_module_kernel_mode_matches_reference_mode_m1(spec, rot):
    N, K = 512, 1024
    w = make_weight(N, K, seed=5, **spec)
    kw = dict(rotation_seed=9, rotation_k=K) if rot else {}
    ref, ker = _modules(w, **kw)
    x = make_x(1, K, seed=6)
    pm.ROUTE_CENSUS.clear()
    y = ker(x.to(DEV).reshape(1, 1, K))
    assert y.shape == (1, 1, N)
    assert rel_l2(y.cpu().reshape(1, N), ref(x)) <= TOL
    assert list(pm.ROUTE_CENSUS) == ["gemv_splitk_fht" if rot else "gemv_splitk"]


def test_fused_mlp_module():
    H, I = 1024, 2048
    wg, wu, wd = (make_weight(I, H, seed=1), make_weight(I, H, seed=2, bits2=1),
                  make_weight(H, I, seed=3))
    refs, kers = zip(*[_modules(w) for w in (wg, wu, wd)])
    act = torch.nn.functional.silu
    mref = pm.FusedPalettizedMLP(*refs, act)
    mker = pm.FusedPalettizedMLP(*kers, act)
    x = make_x(1, H, seed=7)
    pm.ROUTE_CENSUS.clear()
    y = mker(x.to(DEV))
    assert pm.ROUTE_CENSUS.get("gemv_mlp") == 1 and mker._merge_state["ok"]
    assert rel_l2(y.cpu(), mref(x)) <= 2e-3       # two 16-bit roundings (h, then y) on each side


def test_merged_tables_follow_moved_and_converted_members():
    """The cached segment table holds raw addresses.  A member moved to the CPU and back has
    new buffers: the table is rebuilt (stale addresses would be a memory fault).  Residual
    factors kept in float16 are converted once for bfloat16 activations, so the merged
    launch still serves them."""
    H, I = 512, 1024
    wg, wu, wd = (make_weight(I, H, seed=1, rank=8), make_weight(I, H, seed=2, rank=8),
                  make_weight(H, I, seed=3))
    refs, kers = zip(*[_modules(w) for w in (wg, wu, wd)])
    act = torch.nn.functional.silu
    mref, mker = pm.FusedPalettizedMLP(*refs, act), pm.FusedPalettizedMLP(*kers, act)
    x = make_x(1, H, seed=7)
    y0 = mker(x.to(DEV))
    first = mker._merge_state
    assert first["ok"]
    mker.gate_proj.to("cpu")
    mker.gate_proj.to(DEV)
    y1 = mker(x.to(DEV))
    assert mker._merge_state is not first and mker._merge_state["ok"]
    assert torch.equal(y0, y1)
    # bfloat16 activations against float16 residual factors: merged launch, not the fallback
    xb = make_x(1, H, seed=8, dtype=torch.bfloat16)
    pm.ROUTE_CENSUS.clear()
    yb = mker(xb.to(DEV))
    assert pm.ROUTE_CENSUS.get("gemv_mlp") == 1
    assert rel_l2(yb.cpu(), mref(xb)) <= 8e-3     # bf16 h and y, residual factors rounded to bf16


def test_fused_mlp_module_replays_from_a_graph():
    """The module layer is host-bound in eager mode (tens of microseconds of Python per
    call against ~20 us of kernels), so decode loops capture it in a HIP graph.  Every
    replay, with eager work and synchronisations in between, must reproduce the eager
    result bit for bit, also after the input buffer's contents change."""
    H, I = 1024, 2048
    wg, wu, wd = make_weight(I, H, seed=1), make_weight(I, H, seed=2), make_weight(H, I, seed=3)
    kers = [_modules(w)[1] for w in (wg, wu, wd)]
    mker = pm.FusedPalettizedMLP(*kers, torch.nn.functional.silu)
    x = make_x(1, H, seed=7).to(DEV)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):                        # warm-up: workspaces, merge state
        for _ in range(3):
            mker(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = mker(x)
    for seed in (7, 8, 9):
        x.copy_(make_x(1, H, seed=seed).to(DEV))
        graph.replay()
        torch.cuda.synchronize()
        got = y.clone()
        want = mker(x)                                   # eager work between the replays
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("M,spec,route", [
    (8, dict(), "dual_stream"),
    (16, dict(bits2=2, rank=8, bias=True), "dual_stream"),
    (40, dict(bits2=2, rank=8, bias=True), "per_group_lut"),
    (130, dict(bits=3, gs=32), "per_group_lut"),
])
@pytest.mark.parametrize("rot", [False, True])
def test_module_kernel_mode_matches_reference_mode_prefill(M, spec, route, rot):
    """M > 1 goes to the MFMA GEMM: one call for the whole layer where nothing has to see its terms (the
    bias is a parameter, and gradients are on: the cases without one), else the fused small-M entry up
    to 16 rows and the plain entry, the module adding the terms, above.  The census names the entry
    that serves such rows term by term in either case."""
    N, K = 512, 1024
    w = make_weight(N, K, seed=5, **spec)
    kw = dict(rotation_seed=9, rotation_k=K) if rot else {}
    ref, ker = _modules(w, **kw)
    x = make_x(M, K, seed=6)
    pm.ROUTE_CENSUS.clear()
    y = ker(x.to(DEV))
    assert y.shape == (M, N)
    assert rel_l2(y.cpu(), ref(x)) <= (TOL if M <= 16 else 2e-3)   # module-side adds round twice
    assert list(pm.ROUTE_CENSUS) == [route]


@pytest.mark.parametrize("M,lda_pad,act,lut,rank", [
    (8, 0, torch.bfloat16, torch.float16, 0),       # the rotated-input configuration
    (8, 0, torch.float16, torch.float16, 0),
    (40, 0, torch.bfloat16, torch.bfloat16, 0),     # several 16-row blocks, padded rows
    (24, 64, torch.bfloat16, torch.float16, 0),     # rows of A further apart than K
    (100, 0, torch.float16, torch.float16, 0),      # 64-row workgroups
    (8, 0, torch.float16, torch.float16, 4),        # residual: rotated rows are kept as rows
    (24, 64, torch.float16, torch.float16, 4),
])
def test_gemm_with_rotation_through_the_c_abi(M, lda_pad, act, lut, rank):
    """flute_gemm rotates its input itself when the descriptor carries signs (block-128
    form and the full-K form).  Without a residual the rotation writes the activations
    straight in the order the matrix cores read them; with one, as rows first."""
    N, K = 512, 4096
    w = make_weight(N, K, seed=11, lut_dtype=lut, act_dtype=act, rank=rank, device=DEV)
    x = make_x(M, K, seed=12, dtype=act)
    lda = K + lda_pad
    xd = torch.zeros(M, lda, dtype=act, device=DEV)
    xd[:, :K] = x.to(DEV)
    for block in (128, 0):
        signs = O.rotation_signs(K, 3)
        sd = signs.to(DEV)
        d = _desc(w)
        d.signs, d.rot_block = sd.data_ptr(), block
        if rank:
            d.resA, d.resB, d.R = w["resA_d"].data_ptr(), w["resB_d"].data_ptr(), rank
        C = torch.zeros(M, N, dtype=act, device=DEV)
        st = _lib.lib.flute_gemm(ctypes.byref(d), xd.data_ptr(), C.data_ptr(), M, lda, N,
                                 _lib.F16 if act == torch.float16 else _lib.BF16,
                                 torch.cuda.current_stream().cuda_stream)
        assert st == 0, _lib.last_error()
        xr = O.block_fht_reference(x, 128, signs) if block else O.fht_reference(x, signs)
        # the rotated activations are rounded to the activation type before the GEMM
        xr = xr.to(act)
        ref = O.linear_exact(xr, w["blob"].numpy(), w["lut"], N, K, w["gs"], w["bits"],
                             None, None, 0, None, None, None).double()
        if rank:
            ref = ref + (xr.double() @ w["resB"].double().t()) @ w["resA"].double().t()
        tol = 1.5e-3 if act == torch.float16 else 4e-3
        assert rel_l2(C.cpu(), ref.to(act)) <= tol


@pytest.mark.parametrize("rot", [False, True])
def test_split_qkv_module(rot):
    """One token: one grouped launch writes Q|K|V side by side; several tokens: the
    per-module chain and a concatenation.  Both against the reference-mode modules."""
    K = 1024
    ws = [make_weight(512, K, seed=1), make_weight(256, K, bits=3, gs=64, bits2=3, rank=8, seed=2),
          make_weight(256, K, bits=4, gs=128, bias=True, seed=3)]
    kw = dict(rotation_seed=4, rotation_k=K) if rot else {}
    pairs = [_modules(w, **kw) for w in ws]
    ref = pm.SplitQKV(*[p[0] for p in pairs])
    ker = pm.SplitQKV(*[p[1] for p in pairs])
    x = make_x(1, K, seed=5)
    pm.ROUTE_CENSUS.clear()
    y = ker(x.to(DEV).reshape(1, 1, K))
    assert y.shape == (1, 1, 1024)
    assert pm.ROUTE_CENSUS.get("gemv_multi") == 1 and ker._merge_state["ok"], ker._merge_state
    assert rel_l2(y.cpu().reshape(1, -1), ref(x)) <= TOL
    y2 = ker(x.to(DEV))                                  # persistent output, same values
    assert torch.equal(y2.cpu(), y.cpu().reshape(1, -1))
    xs = make_x(5, K, seed=6)
    assert rel_l2(ker(xs.to(DEV)).cpu(), ref(xs)) <= 2e-3


@pytest.mark.parametrize("rot", [False, True])
def test_many_rows_in_one_call_and_autograd_beside_it(rot):
    """More than sixteen rows of a two-stream layer with residual and bias are one library call whose
    only rounding is the last (2^-11 relative at most, so TOL); where autograd wants the bias, or the
    bias has another type, the terms are added one by one as before."""
    N, K, M = 256, 512, 40
    w = make_weight(N, K, seed=5, bits2=1, rank=8, bias=True)
    kw = dict(rotation_seed=9, rotation_k=K) if rot else {}
    ref, ker = _modules(w, **kw)
    x = make_x(M, K, seed=6)
    with torch.no_grad():
        want = ref(x)
        y = ker(x.to(DEV))
    assert not y.requires_grad and rel_l2(y.cpu(), want) <= TOL
    z = ker(x.to(DEV))                                  # gradients on: the bias is a parameter
    assert z.requires_grad and rel_l2(z.detach().cpu(), want) <= 2e-3
    z.float().sum().backward()
    assert torch.equal(ker.bias.grad.cpu().float(), torch.full((N,), float(M)))
    with torch.no_grad():
        ker.bias = torch.nn.Parameter(ker.bias.detach().float())
        assert ker(x.to(DEV)).dtype == torch.float32    # as torch adds a float32 bias


@pytest.mark.parametrize("M", [2, 17, 200, 600, 3000])
@pytest.mark.parametrize("spec,act,rot", [
    (dict(), torch.float16, False), (dict(bits2=1, rank=8), torch.bfloat16, True),
    (dict(bits=3, gs=64, rank=5, bias=True), torch.float16, True), (dict(lut_dtype=torch.bfloat16), torch.bfloat16, False)])
def test_layers_on_the_same_rows_in_one_call(monkeypatch, M, spec, act, rot):
    """q/k/v side by side and silu(gate) * up for more than one token: launches of one weight and of
    several, whole and ragged row blocks, the small-M kernel and (M = 3000) the many-row kernel, shared
    rotated rows, against the members one by one, which round once per output (and the product three
    times): two roundings of the type apart."""
    widths = (spec.get("bits", 4), spec.get("bits2", 0), spec.get("gs", 128))
    assert (gemm_rows(M, *[(n, 1024) + widths for n in (1024, 256, 256)]) >= 256) == (M == 3000)
    assert (gemm_rows(M, *[(n, 1024) + widths for n in (1024, 1024)]) >= 256) == (M == 3000)
    K, rounding = 1024, 2 ** -11 if act is torch.float16 else 2 ** -8
    kw = dict(rotation_seed=9, rotation_k=K) if rot else {}
    layers = [_modules(make_weight(n, K, seed=i, act_dtype=act, **spec), **kw)[1] for i, n in
              enumerate((1024, 256, 256, 1024))]
    x = make_x(M, K, seed=6, dtype=act).to(DEV)
    qkv = pm.SplitQKV(*layers[:3])
    mlp = pm.FusedPalettizedMLP(layers[0], layers[3], torch.nn.Identity(), torch.nn.SiLU())
    with torch.no_grad():
        for block, n in ((qkv, 1536), (mlp, 1024)):
            pm.ROUTE_CENSUS.clear()
            y = block(x.view(1, M, K))
            assert y.shape == (1, M, n) and y.dtype == act and list(pm.ROUTE_CENSUS) == ["gemm_multi"]
            monkeypatch.setenv("FLUTE_NO_MERGE", "1")
            want = block(x)
            monkeypatch.delenv("FLUTE_NO_MERGE")
            assert rel_l2(y.cpu().view(M, n), want.cpu()) <= 2 * rounding
        # somebody who watches a member's call sees it
        seen = []
        handle = layers[0].register_forward_hook(lambda *a: seen.append(1))
        pm.ROUTE_CENSUS.clear()
        qkv(x), mlp(x)
        handle.remove()
        assert len(seen) == 2 and "gemm_multi" not in pm.ROUTE_CENSUS
    if spec.get("bias") and M > 16:                     # (the small-M entry never tracked the bias)
        assert qkv(x).requires_grad and mlp(x).requires_grad


@pytest.mark.parametrize("rows", [16, 32, 64, 128, 256, 512])
@pytest.mark.parametrize("M", [2, 33, 530])
@pytest.mark.parametrize("K,N,spec,act", [
    (256, 1152, dict(rank=16), torch.bfloat16), (128, 2176, dict(rank=5, bias=True), torch.float16),
    (512, 640, dict(lut_dtype=torch.bfloat16, bits2=1), torch.bfloat16)])
def test_block_in_one_call_equals_its_parts(tuning_env, rows, M, K, N, spec, act):
    """silu(gate) * up formed on the way to the operand image, in every shape of the down projection's
    launch, whole and ragged row blocks, scaled rows (two and four a workgroup) and coefficients: the bits of the
    product as a tensor and the down projection of it."""
    gate, up = (_modules(make_weight(N, K, seed=i))[1] for i in range(2))
    if "lut_dtype" in spec:
        gate, up = (_modules(make_weight(N, K, seed=i, lut_dtype=spec["lut_dtype"]))[1] for i in range(2))
    down = _modules(make_weight(K, N, seed=3, act_dtype=act, **spec))[1]
    x = make_x(M, K, seed=6, dtype=act)
    x[M // 2] *= 100.0
    x = x.to(DEV)
    with torch.no_grad():
        tuning_env("FLUTE_GEMM_ROWS", str(rows))
        h = pm._rows_together((gate, up), x, True)
        want, got = down(h), pm.FusedPalettizedMLP(gate, up, down, torch.nn.SiLU())(x)
    assert torch.equal(got, want)


def test_layers_wrapped_on_the_object_are_called_one_by_one():
    """A forward set on one object (placement libraries wrap modules so) is called, as torch would."""
    K = 1024
    layers = [_modules(make_weight(n, K, seed=i))[1] for i, n in enumerate((256, 128, 128))]
    seen, inner = [], layers[1].forward
    layers[1].forward = lambda x: (seen.append(1), inner(x))[1]
    qkv, x = pm.SplitQKV(*layers), make_x(5, K, seed=6).to(DEV)
    with torch.no_grad():
        y = qkv(x)
        assert seen == [1] and torch.equal(y[:, 256:384], inner(x))


@pytest.mark.parametrize("rows", [16, 32, 64, 128])
@pytest.mark.parametrize("M", [2, 33, 130])
@pytest.mark.parametrize("spec,act,rot", [
    (dict(), torch.bfloat16, False), (dict(gs=64), torch.float16, True), (dict(gs=32), torch.float16, False),
    (dict(bits=3, rank=5, bias=True), torch.bfloat16, True), (dict(bits=2, bits2=4, rank=16), torch.float16, False),
    (dict(lut_dtype=torch.bfloat16, rank=8), torch.bfloat16, False)])
def test_several_weights_in_every_workgroup_shape(tuning_env, rows, M, spec, act, rot):
    """The launch of several weights in every shape of the small-M kernel: its loops, ragged row
    blocks, slices of K, weights that begin inside the grid.  fp32 sums (K terms: far below the type's
    rounding), so it and the members one by one, which sum in slices of their own, differ by one
    rounding each; the reference mode rounds the rotated rows, each stream, residual and bias (four)."""
    K, rounding = 1024, 2 ** -11 if act is torch.float16 else 2 ** -8
    kw = dict(rotation_seed=9, rotation_k=K) if rot else {}
    tuning_env("FLUTE_GEMM_ROWS", str(rows))
    pairs = [_modules(make_weight(n, K, seed=i, act_dtype=act, **spec), **kw) for i, n in enumerate((384, 128, 256))]
    x = make_x(M, K, seed=6, dtype=act)
    pm.ROUTE_CENSUS.clear()
    with torch.no_grad():
        y = pm.SplitQKV(*[p[1] for p in pairs])(x.to(DEV))
        want = torch.cat([p[1](x.to(DEV)) for p in pairs], dim=-1)
    assert pm.ROUTE_CENSUS["gemm_multi"] == 1
    assert rel_l2(y.cpu(), want.cpu()) <= rounding
    assert rel_l2(y.cpu(), torch.cat([p[0](x) for p in pairs], dim=-1)) <= 2 * rounding    # half a unit each


@pytest.mark.parametrize("rows,slices", [(512, None), (256, None), (512, 3), (256, 3)])
@pytest.mark.parametrize("M", [130, 600])
@pytest.mark.parametrize("spec,gss,act,seeds", [
    (dict(), (128, 128, 128), torch.bfloat16, None),                          # one image, rows scaled
    (dict(rank=16), (128, 64, 256), torch.bfloat16, (9, 9, 9)),               # groups differ, one rotation
    (dict(bits2=1, rank=16), (64, 64, 64), torch.bfloat16, (9, 4, 9)),        # two rotations, two images
    (dict(bits=1, bits2=4, rank=16), (128, 128, 128), torch.float16, (9, 9, 4)),
    (dict(bits=3, rank=5, bias=True), (128, 32, 128), torch.float16, None),
    (dict(lut_dtype=torch.bfloat16, rank=8), (128, 128, 128), torch.bfloat16, (1, 2, 3))])
def test_several_weights_in_many_row_workgroups(tuning_env, rows, slices, M, spec, gss, act, seeds):
    """The many-row kernel with several weights in the launch: where a weight begins, its own strides,
    bias, group size and coefficients, partial tiles numbered over all of them, one image of the
    activations per rotation, rotated rows with scales.  Against the members one by one in the same
    kernel (one rounding apart) and the reference mode (four roundings)."""
    K, rounding = 1024, 2 ** -11 if act is torch.float16 else 2 ** -8
    tuning_env("FLUTE_GEMM_ROWS", str(rows))
    if slices:
        tuning_env("FLUTE_GEMM_KSPLIT", str(slices))
    pairs = []
    for i, (n, gs) in enumerate(zip((384, 128, 256), gss)):
        kw = dict(rotation_seed=seeds[i], rotation_k=K) if seeds else {}
        pairs.append(_modules(make_weight(n, K, gs=gs, seed=i, act_dtype=act, **spec), **kw))
    x = make_x(M, K, seed=6, dtype=act)
    pm.ROUTE_CENSUS.clear()
    with torch.no_grad():
        y = pm.SplitQKV(*[p[1] for p in pairs])(x.to(DEV))
        again = pm.SplitQKV(*[p[1] for p in pairs])(x.to(DEV))
        want = torch.cat([p[1](x.to(DEV)) for p in pairs], dim=-1)
    assert pm.ROUTE_CENSUS["gemm_multi"] == 2 and torch.equal(y, again)
    assert rel_l2(y.cpu(), want.cpu()) <= rounding
    assert rel_l2(y.cpu(), torch.cat([p[0](x) for p in pairs], dim=-1)) <= 2 * rounding    # half a unit each


def _both_ways(monkeypatch, compiled, block, x):
    """(output, census) of a call through the compiled forward, which has to take it, and through Python's."""
    with torch.no_grad():
        block(x)                                        # (copies and tables that the module keeps)
        pm.ROUTE_CENSUS.clear()
        one = compiled(block, x)
        assert one is not None
        taken = dict(pm.ROUTE_CENSUS)
        pm.ROUTE_CENSUS.clear()
        with monkeypatch.context() as patch:
            patch.setattr(pm, "_forwards", None)
            two = block(x)
        assert taken == pm.ROUTE_CENSUS and one.shape == two.shape and torch.equal(one, two)


@pytest.mark.skipif(fx._C.native is None, reason="the compiled binding is not built or switched off")
@pytest.mark.parametrize("shape", [(1,), (1, 1), (2,), (1, 17), (3, 2, 5)])
@pytest.mark.parametrize("spec,act,rot", [
    (dict(), torch.float16, None), (dict(bits2=1, rank=8, bias=True), torch.bfloat16, None),
    (dict(bits=3, gs=64, rank=16), torch.float16, "same"), (dict(bits=2, bits2=4, gs=16), torch.float16, "awq"),
    (dict(lut_dtype=torch.bfloat16, rank=64), torch.bfloat16, "different")])
def test_compiled_forwards_equal_the_python_ones(monkeypatch, shape, spec, act, rot):
    K, F = 256, 384

    def member(n, k, seed):
        kw = {}
        if rot:
            kw = dict(rotation_seed=seed if rot == "different" else 5, rotation_k=k)
        if rot == "awq":
            kw["awq_scale"] = torch.rand(k, generator=torch.Generator().manual_seed(1)) + 0.5
        return _modules(make_weight(n, k, seed=seed, act_dtype=act, **spec), **kw)[1]
    x = make_x(int(torch.tensor(shape).prod()), K, seed=3, dtype=act).view(*shape, K).to(DEV)
    gate, up, down = member(F, K, 1), member(F, K, 2), member(K, F, 3)
    pm._flute()
    fw = pm._forwards
    _both_ways(monkeypatch, fw.linear, gate, x)
    if len(shape) < 3 or shape[0] > 1:
        _both_ways(monkeypatch, fw.qkv, pm.SplitQKV(gate, up, member(128, K, 4)), x)
        _both_ways(monkeypatch, fw.mlp, pm.FusedPalettizedMLP(gate, up, down, torch.nn.SiLU()), x)
    w = make_weight(256, K, seed=7, lut_dtype=spec.get("lut_dtype", torch.float16), bits2=spec.get("bits2", 0))
    table = pm.PalettizedEmbedding(w["blob"], w["lut"], 4, 128, 256, K, indices2=w["blob2"], lut2=w["lut2"], reference=False,
                                   bitwidth2=w["bits2"] or None, **(dict(rotation_seed=1, rotation_k=K) if rot else {})).to(DEV)
    _both_ways(monkeypatch, fw.embedding, table, torch.randint(0, 256, shape, device=DEV))


@pytest.mark.skipif(fx._C.native is None, reason="the compiled binding is not built or switched off")
@pytest.mark.parametrize("M", [1, 20])
def test_compiled_forwards_leave_other_calls_to_python(monkeypatch, M):
    """Conversions, switches, subclasses, watchers and derivatives: the compiled forwards answer None."""
    from torch.autograd import forward_ad
    K = 256
    pm._flute()
    fw = pm._forwards

    def layer(n=256, **spec):
        return _modules(make_weight(n, K, seed=n, rank=8, bias=True, **spec))[1]
    a, b, c = layer(), layer(), layer()
    qkv, mlp = pm.SplitQKV(a, b, c), pm.FusedPalettizedMLP(a, b, c, torch.nn.SiLU())
    x = make_x(M, K, seed=3).to(DEV)

    def refused(which=("linear", "qkv", "mlp"), x=x):
        blocks = dict(linear=a, qkv=qkv, mlp=mlp)
        return [fw.__getattribute__(n)(blocks[n], x) is None for n in which] == [True] * len(which)
    with torch.no_grad():
        for block in (a, qkv, mlp):
            block(x)
        assert not refused(("linear",)) and not refused(("qkv",)) and not refused(("mlp",))
        for name in ("FLUTE_NO_FHT_FUSE", "FLUTE_NO_MERGE", "FLUTE_ROTATION", "FLUTE_NO_SPLITK", "FLUTE_NO_WIDE_PREF"):
            monkeypatch.setenv(name, "0")
            assert refused()
            monkeypatch.delenv(name)
        assert refused(x=x.float()) and refused(x=x.cpu()) and refused(x=x[:0]) and refused(x=x[:, :64].contiguous())
        assert refused(x=x.clone().requires_grad_(True))
        for watch in (lambda m: m.register_forward_hook(lambda *a: None), lambda m: m.register_forward_pre_hook(lambda *a: None)):
            handle = watch(c)
            assert refused(("mlp",)) and (M == 1 or refused(("qkv",)))
            handle.remove()
        if M > 1:
            with forward_ad.dual_level():
                assert refused()
            mlp.act_fn = torch.nn.GELU()
            assert refused(("mlp",))
            mlp.act_fn = torch.nn.SiLU()
        kept = a.resA
        a.resA = a.resA.float()
        assert refused()
        a.resA = kept
        c.__class__ = type("Other", (pm.PalettizedLinear,), {})
        assert refused(("mlp",)) and (M == 1 or refused(("qkv",)))
        c.__class__ = pm.PalettizedLinear
        a.lut = a.lut.clone()                           # the decode tables hold the old one's address
        assert M > 1 or refused(("qkv", "mlp"))
        block(x), qkv(x), mlp(x)
        assert not refused(("linear",)) and not refused(("qkv",)) and not refused(("mlp",))
        w = make_weight(256, K, seed=7)
        table = pm.PalettizedEmbedding(w["blob"], w["lut"], 4, 128, 256, K, reference=False).to(DEV)
        ids = torch.arange(5, device=DEV)
        assert fw.embedding(table, ids) is not None and fw.embedding(table, ids.int()) is None
        assert fw.embedding(table, ids + 256) is None and fw.embedding(table, ids.cpu()) is None
    if M > 1:
        assert a.bias.requires_grad and refused()       # with gradients on


def _block_of(kind, M, K=256):
    """A block of residual layers.  One row: q/k/v or gate and up hold a factor of another type, so that the decode
    table has it by a copy, whose source is looked at on each call."""
    members = [_modules(make_weight(256, K, seed=i, rank=8, bias=True))[1] for i in range(3)]
    for m in members[:0 if M > 1 else 3 if kind == "qkv" else 2]:
        m.resA = m.resA.float()
    return pm.SplitQKV(*members) if kind == "qkv" else pm.FusedPalettizedMLP(*members, torch.nn.SiLU())


@pytest.mark.skipif(fx._C.native is None, reason="the compiled binding is not built or switched off")
@pytest.mark.parametrize("kind,M,when", [("qkv", 1, "sources"), ("mlp", 1, "sources"), ("mlp", 1, "hooks"), ("qkv", 5, "hooks"),
                                         ("mlp", 5, "hooks")])
def test_compiled_forwards_hold_what_a_call_into_python_replaces(monkeypatch, kind, M, when):
    """Projections and the decode table that go away while the compiled forward asks Python something (another
    thread may run there): the call ends on what it began with."""
    import gc
    pm._flute()
    compiled, it, x, calls = getattr(pm._forwards, kind), _block_of(kind, M), make_x(M, 256, seed=3).to(DEV), []

    def vanish():
        if calls:
            return
        calls.append(1)
        for n in ("q_proj", "k_proj", "v_proj") if kind == "qkv" else ("gate_proj", "up_proj", "down_proj"):
            setattr(it, n, _modules(make_weight(256, 256, seed=9))[1])
        if when == "sources":                           # (at the hooks it has not been read yet)
            it._merge_state = None
        gc.collect()

    class Empty(dict):
        def __bool__(self):
            vanish()
            return False
    inner = torch.nn.Module.__getattr__

    def looked_up(self, name):
        found = inner(self, name)
        vanish()
        return found
    with torch.no_grad():
        want = it(x).clone()
        with monkeypatch.context() as patch:
            if when == "hooks":
                patch.setattr(torch.nn.modules.module, "_global_forward_hooks", Empty())
            else:
                patch.setattr(torch.nn.Module, "__getattr__", looked_up)
            y = compiled(it, x)
        assert calls and y is not None and torch.equal(y, want)


@pytest.mark.skipif(fx._C.native is None, reason="the compiled binding is not built or switched off")
@pytest.mark.parametrize("kind", ["qkv", "mlp"])
def test_compiled_decode_tables_are_looked_at_behind_every_call_into_python(monkeypatch, kind):
    """An operand that is replaced while the sources of a decode table's copies are looked up: its address in the
    table is no longer its own, and the call is left to Python."""
    pm._flute()
    it, x, calls = _block_of(kind, 1), make_x(1, 256, seed=3).to(DEV), []
    inner, first = torch.nn.Module.__getattr__, it.q_proj if kind == "qkv" else it.gate_proj

    def looked_up(self, name):
        found = inner(self, name)
        if not calls:
            calls.append(1)
            first._buffers["lut"] = first._buffers["lut"].clone()
        return found
    with torch.no_grad():
        want = it(x).clone()
        with monkeypatch.context() as patch:
            patch.setattr(torch.nn.Module, "__getattr__", looked_up)
            assert getattr(pm._forwards, kind)(it, x) is None and calls
        assert torch.equal(it(x), want)
