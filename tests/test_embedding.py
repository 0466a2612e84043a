"""PalettizedEmbedding: the row gather through the idxN layout.

CPU: the module's torch path against the oracle composition (dequant rows, 16-bit
stream add, fp32 residual, adjoint rotation).  GPU: the HIP gather through the C ABI.
Without a residual or a rotation the result is a pure gather plus one exactly rounded
add, so it must be bit-identical; with them the summation order differs and the
tolerance is relative L2 <= 1e-3.
"""
import ctypes

import pytest
import torch

import flute_oracle as O
import palettized_modules as pm
from _util import make_weight, rel_l2

DEV = "cuda:0"
CASES = [
    # bits, gs, bits2, rank, rot
    (4, 128, 0, 0, False),
    (3, 64, 0, 0, False),
    (2, 16, 0, 0, False),
    (1, 128, 0, 0, False),
    (4, 128, 2, 0, False),
    (3, 32, 3, 0, False),
    (4, 128, 0, 8, False),
    (4, 64, 1, 4, True),
    (4, 128, 0, 0, True),
]


def _module(w, rot, reference):
    kw = dict(rotation_seed=7, rotation_k=w["K"]) if rot else {}
    lut_res = lambda t: None if t is None else t.to(w["lut"].dtype)
    return pm.PalettizedEmbedding(w["blob"], w["lut"], w["bits"], w["gs"], w["N"], w["K"],
                                  indices2=w["blob2"], lut2=w["lut2"],
                                  bitwidth2=w["bits2"] or None, resA=lut_res(w["resA"]),
                                  resB=lut_res(w["resB"]), reference=reference, **kw)


def _oracle(w, ids, rot):
    return O.embedding_reference(ids, w["blob"].numpy(), w["lut"], w["N"], w["K"], w["gs"],
                                 w["bits"], w["blob2"].numpy() if w["bits2"] else None, w["lut2"],
                                 w["bits2"], w["resA"], w["resB"],
                                 O.rotation_signs(w["K"], 7) if rot else None)


@pytest.mark.parametrize("bits,gs,bits2,rank,rot", CASES)
def test_reference_path_matches_oracle(bits, gs, bits2, rank, rot):
    N, K = 384, 192
    w = make_weight(N, K, bits, gs, seed=bits + gs, bits2=bits2, rank=rank)
    ids = torch.tensor([[0, 1, 127, 128], [383, 200, 5, 5]])
    y = _module(w, rot, True)(ids)
    assert y.shape == (2, 4, K) and y.dtype == torch.float16
    ref = _oracle(w, ids, rot)
    if rank == 0 and not rot:
        assert torch.equal(y, ref)
    else:
        assert rel_l2(y, ref) <= 1e-3


def test_contract_errors():
    w = make_weight(256, 128, seed=1)
    m = _module(w, False, True)
    with pytest.raises(ValueError, match="integer"):
        m(torch.zeros(3))
    with pytest.raises(ValueError, match=r"\[0, 256\)"):
        m(torch.tensor([256]))
    with pytest.raises(ValueError, match=r"\[0, 256\)"):
        m(torch.tensor([-1]))
    with pytest.raises(ValueError, match="num_embeddings"):
        pm.PalettizedEmbedding(w["blob"], w["lut"], 4, 128, 256, 128, num_embeddings=100)
    with pytest.raises(ValueError, match="BOTH"):
        pm.PalettizedEmbedding(w["blob"], w["lut"], 4, 128, 256, 128, indices2=w["blob"])
    assert (m.num_embeddings, m.embedding_dim) == (256, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("bits,gs,bits2,rank,rot", CASES)
def test_hip_gather_matches_oracle(bits, gs, bits2, rank, rot):
    N, K = 512, 4096 if rot else 1024
    w = make_weight(N, K, bits, gs, seed=bits * 3 + gs, bits2=bits2, rank=rank)
    g = torch.Generator().manual_seed(3)
    ids = torch.randint(0, N, (3, 17), generator=g)
    ids[0, 0], ids[0, 1] = 0, N - 1
    m = _module(w, rot, False).to(DEV)
    pm.ROUTE_CENSUS.clear()
    y = m(ids.to(DEV))
    assert y.shape == (3, 17, K) and y.dtype == torch.float16
    assert pm.ROUTE_CENSUS.get("embedding_gather") == 1
    ref = _oracle(w, ids, rot)
    if rank == 0 and not rot:
        assert torch.equal(y.cpu(), ref)
    else:
        assert rel_l2(y.cpu(), ref) <= 1e-3
    assert torch.equal(m(ids.to(DEV)), y)                       # deterministic


@pytest.mark.gpu
def test_hip_gather_bf16_table_and_refusals():
    import flute_extended as fx
    N, K = 256, 512
    w = make_weight(N, K, 4, 128, seed=9, lut_dtype=torch.bfloat16, bits2=2)
    ids = torch.arange(0, N, 7)
    y = fx.embedding_gather(ids.to(DEV), w["blob"].to(DEV), w["lut"].to(DEV), N, K, 4, 128,
                            indices2=w["blob2"].to(DEV), lut2=w["lut2"].to(DEV), bitwidth2=2)
    ref = O.embedding_reference(ids, w["blob"].numpy(), w["lut"], N, K, 128, 4,
                                w["blob2"].numpy(), w["lut2"], 2)
    assert y.dtype == torch.bfloat16 and torch.equal(y.cpu(), ref)
    with pytest.raises(RuntimeError, match=r"\[0, 256\)"):
        fx.embedding_gather(torch.tensor([300], device=DEV), w["blob"].to(DEV), w["lut"].to(DEV),
                            N, K, 4, 128)
    with pytest.raises(RuntimeError, match="integer"):
        fx.embedding_gather(torch.zeros(2, device=DEV), w["blob"].to(DEV), w["lut"].to(DEV), N, K,
                            4, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 192, 1088, 2048, 4160, 12288])
@pytest.mark.parametrize("bits,bits2", [(1, 0), (3, 2), (4, 1), (2, 3)])
@pytest.mark.parametrize("block", [None, 0, 32])
def test_hip_gather_column_edges(K, bits, bits2, block):
    """Rows shorter and longer than a workgroup's sixteen columns a thread, every width's place in
    a chunk (all eight rows of a chunk group, both halves of a tile), segments within and beyond the
    stages held in registers.  Unrotated rows are a gather: bit exact."""
    import flute_extended as fx
    if block and K % block:
        pytest.skip("blocks divide K")
    N = 256
    w = make_weight(N, K, bits, 64, seed=K + bits, bits2=bits2)
    ids = torch.arange(0, N, 5)
    signs = None if block is None else O.rotation_signs(K, 3)
    kw = {} if not bits2 else dict(indices2=w["blob2"].to(DEV), lut2=w["lut2"].to(DEV), bitwidth2=bits2)
    y = fx.embedding_gather(ids.to(DEV), w["blob"].to(DEV), w["lut"].to(DEV), N, K, bits, 64,
                            signs=None if signs is None else signs.to(DEV), rot_block=block or 0, **kw)
    row = O.embedding_reference(ids, w["blob"].numpy(), w["lut"], N, K, 64, bits,
                                w["blob2"].numpy() if bits2 else None, w["lut2"], bits2)
    if signs is None:
        assert torch.equal(y.cpu(), row)
        return
    # the adjoint in blocks is the block transform of the signed row without signs behind it
    one = torch.ones(K)
    want = O.fht_adjoint_reference(row.float(), signs) if not block else \
        O.block_fht_reference(row.float() * signs, block, one)
    assert rel_l2(y.cpu(), want) <= 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("K,block", [(1024, 0), (1088, 0), (3072, 0), (3136, 0), (4032, 0), (4096, 0), (4096, 1024), (4096, 2048),
                                     (2048, 2048), (4096, 4096), (4160, 0)])
@pytest.mark.parametrize("dtype,bits2", [(torch.float16, 0), (torch.bfloat16, 3)])
def test_rotated_rows_of_every_mix_of_segments(K, block, dtype, bits2):
    """Segments in one wavefront, across two and four, several beside each other, and the rows the longer kernel
    takes: the rotation of the gathered rows, also into rows of four-byte alignment."""
    import ctypes
    import flute_extended as fx
    from flute_extended import _C, _lib
    N = 256
    w = make_weight(N, K, 4, 128, seed=K, bits2=bits2, lut_dtype=dtype, device=DEV)
    ids = torch.arange(0, N, 7, device=DEV)
    signs = O.rotation_signs(K, 3).to(DEV)
    kw = dict(indices2=w["blob2_d"], lut2=w["lut2_d"], bitwidth2=bits2) if bits2 else {}
    args = (ids, w["blob_d"], w["lut_d"], N, K, 4, 128)
    y = fx.embedding_gather(*args, signs=signs, rot_block=block, **kw)
    row = fx.embedding_gather(*args, **kw)
    want = _C.fht_backward(row.float(), signs, block).to(dtype)
    # (odd numbers of stages scale by a multiple of sqrt(2), a product the kernel may round once with the type:
    # a unit in the last place where the fp32 product lies at a tie)
    off = (y.float() - want.float()).abs()
    assert bool((off <= want.float().abs() * torch.finfo(dtype).eps).all()) and int((off > 0).sum()) <= 1e-3 * off.numel()
    like = torch.empty(1, K, dtype=dtype, device=DEV)
    none = torch.empty(0, dtype=dtype, device=DEV)
    d, _, keep = _C._describe("test", like, K, w["blob_d"], w["lut_d"], 4, w.get("blob2_d"), w.get("lut2_d"), bits2, none, none,
                              none, 128, signs, None, block)
    out = torch.zeros(ids.numel() * K + 2, dtype=dtype, device=DEV)
    _lib.check(_lib.lib.flute_embedding(ctypes.byref(d), ids.data_ptr(), ids.numel(), out.data_ptr() + 4, _C._stream_of(out)))
    assert torch.equal(out[2:].view(-1, K), y)


@pytest.mark.gpu
def test_ids_are_checked_by_the_launch():
    """One id outside the table anywhere, the first and the last one included, is refused, from
    several threads at a time; the next good call is served."""
    from concurrent.futures import ThreadPoolExecutor
    N, K = 256, 128
    m = _module(make_weight(N, K, seed=2), True, False).to(DEV)
    good = torch.arange(N, device=DEV).repeat(5)
    want = m(good)
    for at in (0, 700, len(good) - 1):
        for value in (-1, N, 1 << 40):
            ids = good.clone()
            ids[at] = value
            with pytest.raises(ValueError, match=r"\[0, 256\)"):
                m(ids)

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
            y = m(good)
            torch.cuda.current_stream().synchronize()
            return torch.equal(y.cpu(), want_cpu)
    want_cpu = want.cpu()
    with ThreadPoolExecutor(4) as pool:
        assert all(pool.map(work, range(16)))


def test_verdict_words_come_back_whichever_way_a_call_ends(tmp_path):
    """The words that checked gathers wait on: a call that ends early, by an error as well, gives its
    word back; an allocation that fails takes none; with all of them out a call waits for one."""
    import os
    import subprocess
    from conftest import PKG
    (tmp_path / "t.cpp").write_text(r"""
#include "verdicts.h"
#include <assert.h>
#include <stdlib.h>
#include <atomic>
#include <memory>
#include <thread>
#include <vector>
using flute::Verdicts;
static int none(void **) { return 7; }
static int some(void **p) { return (*p = aligned_alloc(64, Verdicts::kBytes)) ? 0 : 1; }
static int fails(Verdicts &v) {                       // what a call does whose wait ends in an error
    Verdicts::Word w;
    if (int e = v.take(w, some)) return e;
    assert(*w.get() == 0);
    *w.get() = 5;
    return 3;
}
int main() {
    Verdicts v;
    { Verdicts::Word w; assert(v.take(w, none) == 7); }
    for (int i = 0; i < 3 * Verdicts::kWords; ++i) assert(fails(v) == 3);
    std::vector<std::unique_ptr<Verdicts::Word>> all;
    for (int i = 0; i < Verdicts::kWords; ++i) {
        all.emplace_back(new Verdicts::Word);
        assert(v.take(*all.back(), some) == 0);
        for (int k = 0; k < i; ++k) assert(all[k]->get() != all[i]->get());
    }
    std::atomic<bool> served{false};
    std::thread one([&] { Verdicts::Word w; v.take(w, some); served = true; });
    assert(!served);
    all.pop_back();
    one.join();
    assert(served);
    return 0;
}
""")
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-std=c++17", "-pthread", "-I", os.path.join(PKG, "csrc"), str(tmp_path / "t.cpp"), "-o", exe],
                   check=True)
    subprocess.run([exe], check=True, timeout=60)
