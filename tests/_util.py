"""Seeded synthetic weights shaped like the benchmark configurations: uniform
b-bit indices, per-group LUT ~ N(0, 0.02) sorted ascending, activations ~ N(0, 1)."""
import numpy as np
import torch

from flute_extended import idxN


def make_weight(N, K, bits=4, gs=128, seed=0, lut_dtype=torch.float16, bits2=0, rank=0,
                bias=False, act_dtype=torch.float16, device="cpu"):
    g = torch.Generator().manual_seed(seed)
    w = {"N": N, "K": K, "bits": bits, "gs": gs, "bits2": bits2}
    rows = (N + gs - 1) // gs

    def stream(b):
        idx = torch.randint(0, 1 << b, (N, K), generator=g, dtype=torch.uint8)
        lut = (torch.randn(rows, 1 << b, generator=g) * 0.02).sort(dim=1).values.to(lut_dtype)
        blob = torch.from_numpy(idxN.pack_idxn(idx.numpy(), b))
        return idx, lut, blob

    w["idx"], w["lut"], w["blob"] = stream(bits)
    if bits2:
        w["idx2"], w["lut2"], w["blob2"] = stream(bits2)
    else:
        w["idx2"] = w["lut2"] = w["blob2"] = None
    if rank:
        w["resB"] = (torch.randn(rank, K, generator=g) * 0.05).to(act_dtype)
        w["resA"] = (torch.randn(N, rank, generator=g) * 0.05).to(act_dtype)
    else:
        w["resB"] = w["resA"] = None
    w["bias"] = (torch.randn(N, generator=g) * 0.1).to(act_dtype) if bias else None
    if device != "cpu":
        for k, v in list(w.items()):
            if torch.is_tensor(v) and k not in ("idx", "idx2"):
                w[k + "_d"] = v.to(device)
    return w


def gemm_rows(M, *shapes):
    """Rows of A per workgroup that the library takes for weights (N, K, bits, bits2, gs) together:
    16 ... 128 the small-M kernel, 256 or 512 the many-row kernel."""
    from flute_extended import _lib
    return _lib.lib.flute_gemm_rows(_weights(shapes), len(shapes), M)


def gemv_rows(*shapes):
    """(output rows, wavefronts) of a workgroup in the one-token launch of weights (N, K, bits, bits2, gs)."""
    import ctypes
    from flute_extended import _lib
    waves = ctypes.c_int(0)
    return _lib.lib.flute_gemv_rows(_weights(shapes), len(shapes), ctypes.byref(waves)), waves.value


def _weights(shapes):
    from flute_extended import _lib
    ws = (_lib.FluteLinear * len(shapes))()
    for w, (N, K, bits, bits2, gs) in zip(ws, shapes):
        w.N, w.K, w.b1, w.b2, w.group_size, w.lut_rows = N, K, bits, bits2, gs, -(-N // gs)
        w.lut_dtype = _lib.F16
        w.q1 = w.lut1 = 16                    # (looked at for alignment only)
        w.q1_bytes = N * K * bits // 8
        if bits2:
            w.q2 = w.lut2 = 16
            w.q2_bytes = N * K * bits2 // 8
    return ws


def make_x(M, K, seed=1, dtype=torch.float16):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(M, K, generator=g).to(dtype)


def rel_l2(a, b):
    a, b = a.detach().double().flatten(), b.detach().double().flatten()
    return float((a - b).norm() / b.norm().clamp_min(1e-30))
