"""``nf4hip_stream``: the fused matmul for up to 128 rows of bf16 or fp16 x, at the edges of its tiles -- rows of x around
16 / 32 / 64 / 128, ragged weight rows, one k step, a partial unit of four steps, K split over workgroups -- on fp32 and nested
absmax and larger blocksizes, against a float64 product over the HIP-dequantised weight."""

import ctypes

import pytest
import torch

DEV = "cuda"
U = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}  # half an ulp over the value: 8 and 11 significant bits
A = 1 << 20  # fake, aligned device address: validation dereferences nothing


def _weight(ta, N, K, blocksize, nested, dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = torch.empty(N, K, device=DEV).normal_(0, 0.02, generator=g).to(dtype)
    qw, absmax, code = ta.quantize_nf4(w, blocksize)
    return qw, (ta.compress_absmax(absmax) if nested else absmax), code


def _plan(ta, M, N, K):
    plan = (ctypes.c_int * 4)()
    ta._lib.check(ta._lib.load().nf4hip_stream_plan(M, N, K, ctypes.byref(plan)))
    return tuple(plan)


def _check(y, x, deq, bias):
    """Each product is exact in fp32; a sum takes at most K / 16 MFMA accumulations and a handful of merges, each within
    2**-23 of the sum of magnitudes (two roundings); the result is rounded once."""
    ref, size = x.double() @ deq.double().t(), x.double().abs() @ deq.double().abs().t()
    if bias is not None:
        ref, size = ref + bias.double(), size + bias.double().abs()
    bound = U[y.dtype] * ref.abs() + (x.shape[1] / 16 + 16) * 2.0**-23 * size + 2.0**-24
    worst = ((y.double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, f"{worst:.3f} of the bound"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,blocksize,nested,bias", [
    (1, 1, 64, 64, False, True), (5, 63, 64, 64, True, False), (16, 64, 192, 64, False, False), (17, 65, 256, 64, True, True),
    (32, 300, 320, 64, False, True), (33, 129, 1344, 64, True, False), (64, 1000, 2880, 64, False, True), (65, 257, 1024, 128, False, False),
    (100, 515, 1536, 256, True, True), (128, 4098, 4096, 64, False, True), (128, 96, 28672, 64, True, False), (48, 4096, 4096, 64, True, False),
    (20, 40000, 512, 64, False, False), (16, 8192, 28672, 64, True, False), (129, 300, 320, 64, True, True), (1000, 1000, 2880, 64, False, True), (2, 8192, 2048, 2048, False, True),
])
def test_stream_matches_float64(ta, dtype, M, N, K, blocksize, nested, bias):
    print(f"stream M={M} [{N},{K}] bs={blocksize} nested={nested} bias={bias} {dtype}", flush=True)
    qw, stats, code = _weight(ta, N, K, blocksize, nested, dtype, M + N)
    g = torch.Generator(device=DEV).manual_seed(K)
    x = torch.empty(M, K, device=DEV).normal_(0, 1, generator=g).to(dtype)
    b = torch.empty(N, device=DEV).normal_(0, 1, generator=g).to(dtype) if bias else None
    deq = ta.dequantize_nf4(qw, stats, code, blocksize, dtype, (N, K))
    run = lambda: ta.functional._matmul_nf4_on(x, qw, b, stats, code, blocksize, dtype, (N, K), "stream")
    y = run()
    _check(y, x, deq, b)
    assert torch.equal(run(), y)  # the workspace is left as it was found, sums have one order


# (M, N, K, rows of x per tile, weight rows per tile, K splits): every tile the kernel is built for, with K a multiple of 256 (four
# absmax per load where blocksize is 64) and not (a partial unit), with one workgroup per tile and with K split; ragged M and N, and
# units of K that the k groups share unevenly where more than one group shares them.
TILES = [
    (11, 16, 2176, 16, 64, 1), (3, 16, 16960, 16, 64, 6), (4, 16, 2304, 16, 64, 1), (13, 16, 16640, 16, 64, 6),
    (9, 16765, 1088, 16, 128, 1), (2, 5448, 6208, 16, 128, 5), (1, 16412, 1280, 16, 128, 1), (15, 5656, 6400, 16, 128, 5),
    (7, 33001, 1088, 16, 256, 1), (5, 17122, 4224, 16, 256, 3), (10, 33001, 1024, 16, 256, 1), (6, 16686, 4352, 16, 256, 3),
    (19, 16, 2176, 32, 64, 1), (17, 16, 17472, 32, 64, 6), (29, 16, 2304, 32, 64, 1), (19, 16, 16896, 32, 64, 6),
    (33, 8764, 1088, 32, 128, 1), (1373, 67, 6976, 32, 128, 5), (34, 8332, 1280, 32, 128, 1), (1358, 65, 6912, 32, 128, 5),
    (31, 33001, 1088, 32, 256, 1), (79, 5517, 4160, 32, 256, 3), (21, 33001, 1024, 32, 256, 1), (71, 6274, 4352, 32, 256, 3),
    (36, 16940, 1152, 64, 128, 1), (1402, 129, 6976, 64, 128, 5), (35, 17382, 1280, 64, 128, 1), (1382, 134, 6656, 64, 128, 5),
    (47, 33001, 1088, 64, 256, 1), (1249, 774, 4160, 64, 256, 3), (61, 33001, 1024, 64, 256, 1), (34, 17161, 4352, 64, 256, 3),
    (101, 33001, 1088, 128, 256, 1), (99, 16972, 2752, 128, 256, 3), (125, 33001, 1024, 128, 256, 1), (851, 2345, 2816, 128, 256, 3),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("nested", [False, True])
@pytest.mark.parametrize("M,N,K,rows,width,splits", TILES)
def test_every_tile(ta, dtype, nested, M, N, K, rows, width, splits):
    print(f"tile {rows}x{width} / {splits}: M={M} [{N},{K}] nested={nested} {dtype}", flush=True)
    L, lib = ta._lib, ta._lib.load()
    need = lib.nf4hip_stream_workspace_bytes(M, N, K)
    assert _plan(ta, M, N, K)[:3] == (rows, width, splits) and (need > 0) == (splits > 1)
    qw, stats, code = _weight(ta, N, K, 64, nested, dtype, M + N)
    x = torch.empty(M, K, device=DEV).normal_(0, 1, generator=torch.Generator(device=DEV).manual_seed(K)).to(dtype)
    b = torch.empty(N, device=DEV).normal_(0, 1, generator=torch.Generator(device=DEV).manual_seed(N)).to(dtype)
    deq = ta.dequantize_nf4(qw, stats, code, 64, dtype, (N, K))
    ws = torch.zeros(need + 4096, dtype=torch.uint8, device=DEV)
    head = (x.data_ptr(), L.F16 if dtype == torch.float16 else L.BF16, M, qw.data_ptr())
    first = None
    for _ in range(2):
        out = torch.full((M + 1, N), float("nan"), dtype=dtype, device=DEV)
        tail = (code.data_ptr(), b.data_ptr(), N, K, 64, out.data_ptr(), ws.data_ptr() if need else None, need, ta.functional._stream())
        if nested:
            L.check(lib.nf4hip_stream_dq(*head, stats.q.data_ptr(), stats.absmax2.data_ptr(), stats.map256.data_ptr(), stats.offset, stats.blocksize, *tail))
        else:
            L.check(lib.nf4hip_stream(*head, stats.data_ptr(), *tail))
        _check(out[:M], x, deq, b)
        assert out[M].isnan().all() and not ws[:65536 * 4].any() and not ws[need:].any()
        first = out if first is None else first
        assert torch.equal(out[:M], first[:M])


def test_every_tile_is_listed(ta):
    """The list above names the tiles the library plans (checked without a GPU), each with and without a split of K, whole and
    partial units."""
    seen = set()
    for M, N, K, rows, width, splits in TILES:
        assert _plan(ta, M, N, K)[:3] == (rows, width, splits), (M, N, K, _plan(ta, M, N, K))
        seen.add((rows, width, K % 256 == 0, splits > 1))
    tiles = [(16, 64), (16, 128), (16, 256), (32, 64), (32, 128), (32, 256), (64, 128), (64, 256), (128, 256)]
    assert seen == {(*tile, whole, split) for tile in tiles for whole in (False, True) for split in (False, True)}
    g = torch.Generator().manual_seed(0)
    for _ in range(2000):  # ... and no other
        M, N, K = (int(2.0 ** (lo + (hi - lo) * torch.rand(1, generator=g).item())) for lo, hi in ((0, 12), (0, 17), (0, 9)))
        if ta._lib.load().nf4hip_stream_served(M, N, 64 * K):
            assert _plan(ta, M, N, 64 * K)[:2] in tiles


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [16, 32, 64, 128])
def test_stream_recovers_dequantised_weights(ta, dtype, M):
    """One-hot rows of x: every output is one product 1.0 * w and must be nf4hip_dequantize's value bit for bit."""
    print(f"stream one-hot M={M} {dtype}", flush=True)
    N, K = 272, 1088
    qw, absmax, code = _weight(ta, N, K, 64, False, dtype, 3)
    cols = torch.randint(0, K, (M,), generator=torch.Generator().manual_seed(M))
    x = torch.zeros(M, K, dtype=dtype)
    x[torch.arange(M), cols] = 1.0
    y = ta.functional._matmul_nf4_on(x.to(DEV), qw, None, absmax, code, 64, dtype, (N, K), "stream")
    deq = ta.dequantize_nf4(qw, absmax, code, 64, dtype, (N, K))
    assert torch.equal(y, deq[:, cols.to(DEV)].t())


@pytest.mark.gpu
def test_stream_infinities_stay_in_their_row(ta):
    print("stream infinities", flush=True)
    N, K, M = 300, 2880, 33
    qw, absmax, code = _weight(ta, N, K, 64, False, torch.float16, 4)
    x = torch.ones(M, K, dtype=torch.float16, device=DEV)
    x[5, 7], x[32, K - 1] = float("inf"), float("nan")
    y = ta.matmul_nf4(x, qw, None, absmax, code, 64, torch.float16, (N, K))
    others = [m for m in range(M) if m not in (5, 32)]
    assert y[others].isfinite().all() and y[32].isnan().all() and not y[5].isfinite().any()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,refused", [(24, 512, 4096, True), (128, 4096, 14336, True), (8, 300, 2880, True), (256, 1024, 8192, True),
                                           (24, 512, 64 * 47, False)])
def test_capture_on_a_stream_without_a_workspace(ta, monkeypatch, M, N, K, refused):
    """bf16 calls that would record a slower plan than the eager call's are refused, with the way out in the message; those that
    were always taken without a workspace, and fp16, which has no other kernel, go on and say so.  (The stream is only said
    to be capturing.)"""
    print(f"capture without workspace M={M} [{N},{K}]", flush=True)
    F = ta.functional
    for dtype in (torch.bfloat16, torch.float16):
        qw, absmax, code = _weight(ta, N, K, 64, False, dtype, 5)
        x = torch.randn(M, K, device=DEV).to(dtype)
        deq = ta.dequantize_nf4(qw, absmax, code, 64, dtype, (N, K))
        call = lambda: F.matmul_nf4(x, qw, None, absmax, code, 64, dtype, (N, K))
        with monkeypatch.context() as m:
            m.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
            m.setattr(F._workspace_pool, "_live", {})
            if refused and dtype == torch.bfloat16:
                with pytest.raises(RuntimeError, match="reserve_workspace"):
                    call()
            else:
                with pytest.warns(UserWarning, match="without a workspace"):
                    y = call()
                _check(y, x, deq, None)
        _check(call(), x, deq, None)


@pytest.mark.gpu
def test_stream_capture_without_scratch_and_autograd(ta):
    print("stream capture / autograd", flush=True)
    F = ta.functional
    N, K, M = 512, 4096, 24
    assert ta._lib.load().nf4hip_stream_workspace_bytes(M, N, K) > 0
    qw, absmax, code = _weight(ta, N, K, 64, False, torch.float16, 5)
    x = torch.randn(M, K, device=DEV).half()
    args = (qw, None, absmax, code, 64, torch.float16, (N, K))
    deq = ta.dequantize_nf4(qw, absmax, code, 64, torch.float16, (N, K))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    saved = F._workspace_pool._live
    try:
        F._workspace_pool._live = {}
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = F.matmul_nf4(x, *args)
    finally:
        F._workspace_pool._live = saved
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        _check(y, x, deq, None)
    # what has to be differentiated goes to the torch operation, as it always has
    xg = x.clone().requires_grad_(True)
    F.matmul_nf4(xg, *args).sum().backward()
    torch.testing.assert_close(xg.grad[0].float(), deq.float().sum(0), rtol=1e-2, atol=1e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,blocksize,nested,bias", [
    (129, 300, 320, 64, False, True), (200, 65, 2880, 64, True, False), (256, 512, 64, 64, False, False), (1025, 1024, 4096, 64, True, True),
    (513, 1000, 1536, 128, False, False), (2048, 4096, 2048, 64, False, False), (130, 32768, 2048, 64, True, False), (300, 264, 28672, 64, False, True),
])
@pytest.mark.parametrize("scratch", [True, False])
def test_gemm_streamed_beyond_128_rows(ta, M, N, K, blocksize, nested, bias, scratch):
    """``nf4hip_gemm`` on the streaming kernel for more than 128 rows of x (several tiles of x rows, K split or not)."""
    print(f"streamed gemm M={M} [{N},{K}] bs={blocksize} nested={nested} bias={bias} scratch={scratch}", flush=True)
    F, lib = ta.functional, ta._lib.load()
    assert lib.nf4hip_gemm_streamed(M, N, K)
    qw, stats, code = _weight(ta, N, K, blocksize, nested, torch.bfloat16, M + N)
    g = torch.Generator(device=DEV).manual_seed(K)
    x = torch.empty(M, K, device=DEV).normal_(0, 1, generator=g).to(torch.bfloat16)
    b = torch.empty(N, device=DEV).normal_(0, 1, generator=g).to(torch.bfloat16) if bias else None
    deq = ta.dequantize_nf4(qw, stats, code, blocksize, torch.bfloat16, (N, K))
    if scratch:
        run = lambda: F._matmul_nf4_on(x, qw, b, stats, code, blocksize, torch.bfloat16, (N, K), "gemm")
    else:  # the streaming kernel takes any plan without
        if nested:
            stats = ta.reconstruct_absmax(stats)

        def run():
            out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
            ta._lib.check(lib.nf4hip_stream(x.data_ptr(), 0, M, qw.data_ptr(), stats.data_ptr(), code.data_ptr(), None if b is None else b.data_ptr(), N, K,
                                            blocksize, out.data_ptr(), None, 0, F._stream()))
            return out

    y = run()
    _check(y, x, deq, b)
    assert torch.equal(run(), y)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,split", [(24, 512, 64 * 47, True), (100, 300, 64 * 61, True), (300, 1000, 1024, False)])
def test_gemm_without_the_workspace(ta, M, N, K, split):
    """Calls that nf4hip_gemm takes without the workspace it asks for (K in no equal ranges) or that need none: NULL, too small a
    one, one that is not aligned and one that was not asked for, which stay as they are."""
    print(f"gemm without workspace M={M} [{N},{K}]", flush=True)
    F, lib, L = ta.functional, ta._lib.load(), ta._lib
    need = lib.nf4hip_gemm_workspace_bytes(M, N, K)
    assert (need > 0) == split and lib.nf4hip_gemm_streamed(M, N, K)
    qw, absmax, code = _weight(ta, N, K, 64, False, torch.bfloat16, M + N)
    x = torch.randn(M, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(K)).to(torch.bfloat16)
    deq = ta.dequantize_nf4(qw, absmax, code, 64, torch.bfloat16, (N, K))
    ws = torch.full((4 << 20,), 0x5A, dtype=torch.uint8, device=DEV)
    assert need < ws.numel() - 16
    cases = [(None, 0), (ws.data_ptr(), 4096), (ws.data_ptr() + 2, ws.numel() - 16)] + ([] if split else [(ws.data_ptr(), ws.numel())])
    first = None
    for ptr, nbytes in cases:
        out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        L.check(lib.nf4hip_gemm(x.data_ptr(), L.BF16, M, qw.data_ptr(), absmax.data_ptr(), code.data_ptr(), None, N, K, 64, out.data_ptr(), ptr, nbytes,
                                F._stream()))
        first = out if first is None else first
        assert torch.equal(out, first) and bool((ws == 0x5A).all())
    _check(first, x, deq, None)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,blocksize,written", [(700, 3000, 5056, 64, True), (700, 3000, 5120, 64, False), (700, 3000, 5120, 128, True),
                                                     (700, 3000, 5120, 256, False), (200, 300, 2880, 64, False), (128, 3000, 5056, 64, False),
                                                     (512, 8192, 28672, 64, True)])
def test_nested_absmax_written_out(ta, monkeypatch, M, N, K, blocksize, written):
    """More than 128 rows of x on nested absmax: the fp32 absmax is written out first where the kernel that serves the call reads
    the nested form value by value; the bits are those of the kernel on the nested form."""
    print(f"nested absmax M={M} [{N},{K}] bs={blocksize}", flush=True)
    F, L, lib = ta.functional, ta._lib, ta._lib.load()
    qw, nq, code = _weight(ta, N, K, blocksize, True, torch.bfloat16, 9)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    calls, real = [], F.reconstruct_absmax
    monkeypatch.setattr(F, "reconstruct_absmax", lambda nq: calls.append(1) or real(nq))
    y = F._matmul_nf4_on(x, qw, None, nq, code, blocksize, torch.bfloat16, (N, K), "gemm")
    assert bool(calls) == written
    need = lib.nf4hip_gemm_workspace_bytes(M, N, K)
    ws = torch.zeros(max(need, 16), dtype=torch.uint8, device=DEV)
    out = torch.empty_like(y)
    L.check(lib.nf4hip_gemm_dq(x.data_ptr(), L.BF16, M, qw.data_ptr(), nq.q.data_ptr(), nq.absmax2.data_ptr(), nq.map256.data_ptr(), nq.offset, nq.blocksize,
                               code.data_ptr(), None, N, K, blocksize, out.data_ptr(), ws.data_ptr(), need, F._stream()))
    assert torch.equal(out, y)


def test_gemm_streamed_rule(ta):
    """Tiles of 128 x 256 fill the chip once at most (half of it with few k steps); beyond 32-bit offsets never.  Of these
    nf4hip_gemm leaves long rows to the other kernel's 256-row tiles in pieces where their models say so."""
    lib = ta._lib.load()
    served = lib.nf4hip_stream_served
    for M, N, K, streamed in ((986, 4384, 27520, 0), (1343, 4864, 26560, 0), (2005, 3236, 20224, 0), (512, 8192, 28672, 0), (315, 8768, 27648, 1),
                              (2048, 4096, 14336, 1), (512, 4096, 14336, 1), (302, 19800, 12672, 1), (129, 8192, 28672, 1)):
        assert served(M, N, K) and lib.nf4hip_gemm_streamed(M, N, K) == streamed, (M, N, K)
    assert served(128, 1 << 20, 4096) and served(2048, 4096, 4096) and not served(2049, 4096, 4096) and served(256, 32768, 2048)
    assert not served(257, 32768, 2048) and not served(256, 32768, 1024) and served(256, 16384, 1024) and not served(1 << 18, 64, 8192)
    assert not served(128, 1 << 26, 4096) and not served(0, 64, 64) and not served(8, 64, 96)


def test_stream_arguments_and_workspace(ta):
    """Checked before any HIP call; the workspace holds what the plan can need and is optional."""
    L = ta._lib
    lib = L.load()

    def call(x=A, dt=L.F16, M=8, packed=A, absmax=A, lut=A, bias=None, N=64, K=4096, bs=64, out=A, w=None, wb=0):
        return lib.nf4hip_stream(x, dt, M, packed, absmax, lut, bias, N, K, bs, out, w, wb, None)

    assert call(x=None) == L.E_NULL and call(absmax=None) == L.E_NULL and call(dt=L.F32) == L.E_DTYPE and call(bs=96) == L.E_BLOCKSIZE
    assert call(M=0) == L.E_SHAPE and call(M=257, N=32768) == L.E_SHAPE and call(K=96) == L.E_SHAPE and call(K=192, bs=128) == L.E_SHAPE
    assert call(K=1 << 24) == L.E_SHAPE and call(N=1 << 30) == L.E_SHAPE
    assert call(out=A + 2) == L.E_ALIGN and call(w=A + 8, wb=1 << 20) == L.E_ALIGN
    for M in (1, 16, 17, 33, 65, 128):
        for N, K in ((1, 64), (1024, 4096), (4096, 14336), (128256, 4096), (8192, 28672)):
            need = lib.nf4hip_stream_workspace_bytes(M, N, K)
            assert need == 0 or 65536 * 4 < need <= 65536 * 4 + 256 * 256 * 128 * 4
    assert lib.nf4hip_stream_workspace_bytes(129, 64, 64) == 0 and lib.nf4hip_stream_workspace_bytes(8, 64, 96) == 0


def test_fp16_route(ta):
    F = ta.functional
    hf = torch.float16

    def route(M, N, K, x=None, bias=None):
        return F.fused_route(torch.empty(M, K, dtype=hf) if x is None else x, bias, 64, hf, (N, K))

    assert route(2048, 64, 4096) == "stream" and route(2049, 64, 4096) == "dequant+linear" and route(512, 32768, 256) == "dequant+linear"
    # what differentiates or transforms stays with the torch operation
    xg = torch.empty(2, 4096, dtype=hf, requires_grad=True)
    assert route(2, 64, 4096, xg) == "dequant+linear"
    with torch.no_grad():
        assert route(2, 64, 4096, xg) == "stream"
    with torch.autograd.forward_ad.dual_level():
        assert route(2, 64, 4096) == "dequant+linear"
    seen = []
    torch.func.vmap(lambda row: (seen.append(route(1, 64, 4096, row)), row)[1])(torch.zeros(2, 1, 4096, dtype=hf))
    assert seen == ["dequant+linear"]
    # ... and so do weights that are too small or lie elsewhere
    n = 64 * 4096
    x, book = torch.empty(2, 4096, dtype=hf), torch.empty(16)
    whole = dict(qweight=torch.empty(n // 2, 1, dtype=torch.uint8), bias=None, absmax=torch.empty(n // 64), quant_map=book, n=n, blocksize=64)
    ok = lambda **kw: F._weight_complete(x, **{**whole, **kw})
    assert ok() and not ok(absmax=torch.empty(n // 64 - 1)) and not ok(qweight=torch.empty(n // 2 - 1, 1, dtype=torch.uint8))
    assert not ok(quant_map=torch.empty(15)) and not ok(bias=torch.empty(64, dtype=hf, device="meta")) and not ok(absmax=whole["absmax"].to("meta"))
    nested = lambda device: F.NestedAbsmax(torch.empty(n // 64, dtype=torch.uint8, device=device), None, None, 0.0)
    assert ok(absmax=nested("cpu")) and not ok(absmax=nested("meta"))
