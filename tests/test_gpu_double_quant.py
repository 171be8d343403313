"""Nested ("double") quantisation on the GPU at the sizes where its kernels can go wrong, bit-exact against the CPU
oracle: every nested block size (one to sixteen waves of a nested block), lengths that end inside a lane's four values,
inside a nested block and inside a workgroup, maps that the bisection must hand to the full scan or settle ties on."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _compress(ta, absmax, D, off, nested):
    lib = ta._lib.load()
    nb = absmax.numel()
    q = torch.full((nb + 16,), 0xA5, dtype=torch.uint8, device=DEV)
    a2 = torch.full(((nb + nested - 1) // nested + 4,), -7.0, device=DEV)
    a_dev, D_dev = absmax.to(DEV), D.to(DEV)
    ta._lib.check(lib.nf4hip_dq_compress(a_dev.data_ptr(), nb, nested, D_dev.data_ptr(), off, q.data_ptr(), a2.data_ptr(),
                                         torch.cuda.current_stream().cuda_stream))
    assert bool((q[nb:] == 0xA5).all()) and bool((a2[-4:] == -7.0).all()), "wrote past its output"
    return q[:nb].cpu(), a2[:-4].cpu()


@pytest.mark.parametrize("nested", [64, 128, 256, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("nb", [1, 3, 63, 257, 1021, 1024, 4099, 50001])
def test_compress_sizes(ta, oracle, nested, nb):
    print(f"compress nested={nested} nb={nb}", flush=True)
    absmax = torch.rand(nb, generator=torch.Generator().manual_seed(nb + nested)) * 0.1
    D = oracle.create_dynamic_map()
    q, a2 = _compress(ta, absmax, D, 0.04, nested)
    q_o, a2_o = oracle.C().dq_compress(absmax, D, 0.04, nested)
    assert torch.equal(q, q_o) and torch.equal(a2, a2_o)


def _maps(oracle):
    D = oracle.create_dynamic_map()
    g = torch.Generator().manual_seed(5)
    coarse = (D * 16).round() / 16  # runs of equal entries: the first of a run is the answer
    yield "dynamic", D
    yield "runs of equal entries", coarse
    yield "descending", D.flip(0).contiguous()
    yield "shuffled", D[torch.randperm(256, generator=g)].contiguous()
    yield "without zero", torch.where(D == 0, torch.tensor(1e-3), D).sort().values
    yield "infinite end", torch.cat([D[:-1], torch.tensor([float("inf")])])
    yield "nan", torch.where(torch.arange(256) == 100, torch.tensor(float("nan")), D)


def test_compress_maps_and_ties(ta, oracle):
    """Values on map entries, exactly half way between neighbours, an ulp to either side, beyond both ends, all-zero
    nested blocks, infinities and NaN."""
    for name, D in _maps(oracle):
        print(f"compress map: {name}", flush=True)
        finite = oracle.create_dynamic_map()
        mid = (finite[:-1] + finite[1:]) / 2
        v = torch.cat([finite, mid, torch.nextafter(mid, torch.tensor(2.0)), torch.nextafter(mid, torch.tensor(-2.0))])
        blocks = [torch.cat([c, torch.zeros(63 - len(c)), torch.tensor([1.0])]) for c in v.split(63)]  # r / max|r| = r
        blocks += [torch.zeros(64), torch.full((64,), 1e-39), torch.linspace(-3, 3, 64), torch.linspace(-3, 3, 63)]
        absmax = torch.cat(blocks)
        absmax[-70], absmax[-200] = float("inf"), float("nan")
        q, a2 = _compress(ta, absmax, D, 0.0, 64)
        q_o, a2_o = oracle.C().dq_compress(absmax, D, 0.0, 64)
        assert torch.equal(a2, a2_o), name
        assert torch.equal(q, q_o), (name, (q != q_o).nonzero().flatten()[:8].tolist())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,blocksize,nested", [(1, 64, 256), (65, 64, 64), (8192 * 3 + 5, 64, 256), (300_001, 128, 4096), (8192 * 64, 4096, 256),
                                                (40_000, 1024, 2048), (16_777_216 + 64, 64, 256)])
def test_quantize_dq(ta, oracle, dtype, n, blocksize, nested):
    """One call: codes, nested codes and second level bit for bit, the offset as the float64 mean rounded once."""
    print(f"quantize_dq {dtype} n={n} {blocksize}/{nested}", flush=True)
    w = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 0.02).to(dtype)
    qw, q, a2, m256, off, code = ta.functional.quantize_nf4_dq(w.to(DEV), blocksize, nested)
    qw_o, absmax_o = oracle.C().quantize(w, blocksize)
    off_o = float(absmax_o.double().mean().to(torch.float32))
    assert off.shape == (1,) and off.item() == off_o and ta.functional._offset_value(off) == off_o
    D = oracle.create_dynamic_map()
    assert torch.equal(m256.cpu(), D) and torch.equal(code.cpu(), oracle.nf4_lut())
    q_o, a2_o = oracle.C().dq_compress(absmax_o, D, off_o, nested)
    assert torch.equal(qw.cpu(), qw_o) and torch.equal(q.cpu(), q_o) and torch.equal(a2.cpu(), a2_o)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("blocksize", [64, 512, 1024, 4096])
def test_quantize_workgroup_edges(ta, oracle, dtype, blocksize):
    """The last workgroup whole, one element short, one element over; thresholds and their neighbours, infinities, NaN and
    denormals in a whole workgroup and in the ragged one."""
    thr = torch.tensor([(0xBF591CD9 - (1 << 32)), 0x3D22FAFF, 0x3F5C89D9], dtype=torch.int32).view(torch.float32)
    one = torch.tensor([1.0, -1.0, float("inf"), float("nan"), float("-inf"), 1e-39, 0.0, -0.0])
    special = torch.cat([thr, torch.nextafter(thr, one[:1]), torch.nextafter(thr, one[1:2]), one])
    span = 8192 if blocksize < 4096 else 16384
    for n in (span - 1, span, span + 1, 2 * span, 3 * span + 9):
        print(f"quantize edges {dtype} {blocksize} n={n}", flush=True)
        w = torch.rand(n, generator=torch.Generator().manual_seed(n)) * 2 - 1
        for at in (0, blocksize - 20, n - len(special)):
            w[at:at + len(special)] = special
        w[2 * blocksize:3 * blocksize] = 0.0
        w = w.to(dtype)
        qw, absmax, _ = ta.quantize_nf4(w.to(DEV), blocksize)
        qw_o, absmax_o = oracle.C().quantize(w, blocksize)
        assert torch.equal(absmax.cpu(), absmax_o) and torch.equal(qw.cpu().flatten(), qw_o.flatten()), n


def test_statistics_in_one_call_or_two(ta):
    """nf4hip_quantize_dq is nf4hip_quantize and nf4hip_dq_statistics, which functional.quantize_nf4_dq launches apart; what the
    second refuses."""
    L = ta._lib
    lib = L.load()
    n, stream = 64 * 5003, torch.cuda.current_stream().cuda_stream
    w = torch.randn(n, device=DEV, dtype=torch.bfloat16)
    want = ta.functional.quantize_nf4_dq(w)
    D = ta.functional.dynamic_map(w.device)
    got = [torch.empty_like(t) for t in want]
    need = lib.nf4hip_quantize_dq_workspace_bytes(n, 64)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    qw, q, a2, m256, off, code = (t.data_ptr() for t in got)
    L.check(lib.nf4hip_quantize_dq(w.data_ptr(), L.BF16, n, 64, 256, D.data_ptr(), qw, q, a2, off, m256, code, ws.data_ptr(), need, stream))
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    absmax = torch.rand(5003, device=DEV)

    def statistics(absmax=absmax.data_ptr(), n=5003, nested=256, offset=off, ws_bytes=L.DQ_STATISTICS_WORKSPACE_BYTES):
        return lib.nf4hip_dq_statistics(absmax, n, nested, D.data_ptr(), q, a2, offset, None, None, ws.data_ptr(), ws_bytes, stream)

    assert statistics() == 0 and statistics(n=0) == L.E_SHAPE and statistics(nested=96) == L.E_BLOCKSIZE
    assert statistics(offset=None) == L.E_NULL and statistics(absmax=absmax.data_ptr() + 4) == L.E_ALIGN
    assert statistics(ws_bytes=L.DQ_STATISTICS_WORKSPACE_BYTES - 1) == L.E_WORKSPACE
    torch.cuda.synchronize()
    assert got[4].item() == float(absmax.cpu().double().mean().to(torch.float32))


def test_offset_of_more_values_than_one_round_of_loads(ta):
    """4.8 M blocks: every workgroup of the sum takes more full rounds than it loads at a time, and a remainder."""
    n = 64 * (512 * 9300 + 5)
    w = torch.randn(n, device=DEV, dtype=torch.bfloat16)
    off = ta.functional.quantize_nf4_dq(w)[4]
    qw, absmax, code = ta.quantize_nf4(w)
    assert off.item() == float(absmax.cpu().double().mean().to(torch.float32))
    # beyond the last-level cache weight and output are streamed past it: what a part alone, which is not, gives
    m = 64 * 100_003
    part = ta.quantize_nf4(w[-m:].clone())
    assert torch.equal(part[0].flatten(), qw.flatten()[-m // 2:]) and torch.equal(part[1], absmax[-100_003:])
    dense = ta.dequantize_nf4(qw, absmax, code, 64, torch.bfloat16, (n,))
    assert torch.equal(dense[-m:], ta.dequantize_nf4(*part, 64, torch.bfloat16, (m,)))


@pytest.mark.parametrize("n,blocksize,nested", [(7, 64, 256), (8192 + 8, 64, 64), (8192 * 5 + 3, 256, 256), (100_000, 64, 4096)])
def test_dequantize_nested_sizes(ta, oracle, n, blocksize, nested):
    print(f"dequantize nested n={n} {blocksize}/{nested}", flush=True)
    g = torch.Generator().manual_seed(n)
    nb = (n + blocksize - 1) // blocksize
    packed = torch.randint(0, 256, ((n + 1) // 2,), dtype=torch.uint8, generator=g)
    D = oracle.create_dynamic_map()
    absmax = torch.rand(nb, generator=g) * 0.1
    q, a2 = oracle.C().dq_compress(absmax, D, 0.03, nested)
    nq = ta.NestedAbsmax(q.to(DEV), a2.to(DEV), D.to(DEV), 0.03, nested)
    plain = oracle.C().dq_reconstruct(q, a2, D, 0.03, nested)
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        out = ta.dequantize_nf4(packed.to(DEV), nq, ta.nf4_code(DEV), blocksize, dtype, (n,))
        want = oracle.C().dequantize(packed, plain, oracle.nf4_lut(), blocksize, dtype, (n,))
        assert torch.equal(out.cpu().view(torch.uint8), want.view(torch.uint8)), dtype
