"""GPU parity tests: the HIP kernels, called through the C ABI, against the CPU oracle.

quantize / dequantize: bit-exact.  matmul: rtol = atol = 2e-2 against the float64-accumulated
dequantize-then-matmul (the tolerance the north star states for bf16).
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _weights(shape, seed, dtype=torch.bfloat16, std=0.02):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g, dtype=torch.float32) * std).to(dtype)


def _acts(shape, seed, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g, dtype=torch.float32).to(dtype)


def _sync_print(msg):
    print(msg, flush=True)


# ------------------------------------------------------------------------------------------------
# quantize
# ------------------------------------------------------------------------------------------------


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize(
    "shape",
    [(2, 2), (1, 1), (3, 21), (64, 64), (64, 1376), (7, 999), (512, 4096), (1, 64 * 5 + 2)],
)
def test_quantize_bit_exact(ta, oracle, dtype, shape):
    _sync_print(f"quantize {dtype} {shape}")
    w = _weights(shape, seed=sum(shape), dtype=dtype)
    qw, absmax, code = ta.quantize_nf4(w.to(DEV))
    qw_o, absmax_o = oracle.C().quantize(w, 64)
    assert qw.shape == qw_o.shape and qw.dtype == torch.uint8
    assert torch.equal(qw.cpu(), qw_o)
    assert torch.equal(absmax.cpu(), absmax_o)
    assert torch.equal(code.cpu(), oracle.nf4_lut())


@pytest.mark.parametrize("blocksize", [64, 128, 256, 512, 1024, 2048, 4096])
def test_quantize_blocksizes(ta, oracle, blocksize):
    _sync_print(f"quantize blocksize {blocksize}")
    w = _weights((37, 1000), seed=blocksize)  # partial last block for every blocksize
    qw, absmax, _ = ta.quantize_nf4(w.to(DEV), blocksize=blocksize)
    qw_o, absmax_o = oracle.C().quantize(w, blocksize)
    assert torch.equal(qw.cpu(), qw_o)
    assert torch.equal(absmax.cpu(), absmax_o)


def test_quantize_corner_cases(ta, oracle):
    _sync_print("quantize corner cases")
    w = torch.zeros(4, 64, dtype=torch.bfloat16)
    w[1, 5] = 0.5  # a block with a single non-zero
    w[2] = torch.linspace(-1, 1, 64).to(torch.bfloat16)  # contains +-absmax exactly
    w[3, ::2] = -3.0
    qw, absmax, _ = ta.quantize_nf4(w.to(DEV))
    qw_o, absmax_o = oracle.C().quantize(w, 64)
    assert torch.equal(qw.cpu(), qw_o)
    assert torch.equal(absmax.cpu(), absmax_o)
    codes = oracle.unpack_codes(qw.cpu(), w.numel()).view(4, 64)
    assert (codes[0] == 0).all() and absmax[0].item() == 0.0  # zero block: 0*inf = NaN -> code 0
    assert codes[1, 5] == 15 and (codes[1, :5] == 7).all()
    assert codes[2, 0] == 0 and codes[2, 63] == 15
    # zero block dequantizes to -0.0 (code 0 is -1.0, times absmax 0)
    deq = ta.dequantize_nf4(qw, absmax, ta.nf4_code(DEV), 64, torch.bfloat16, w.shape)
    assert (deq[0].cpu().view(torch.int16) == -32768).all()


def test_quantize_exhaustive_bf16(ta, oracle):
    """Every finite bf16 bit pattern, in blocks whose absmax is pinned to a chosen value."""
    _sync_print("quantize exhaustive bf16")
    bits = torch.arange(0, 1 << 16, dtype=torch.int32).to(torch.int16)
    vals = bits.view(torch.bfloat16)
    vals = vals[torch.isfinite(vals.float())]
    for amax in [2.0**-7, 0.025146484375, 0.0517578125, 0.10595703125, 1.0, 3.5, 65280.0]:
        v = vals[vals.float().abs() <= amax]
        pad = (-v.numel()) % 63
        v = torch.cat([v, torch.zeros(pad, dtype=torch.bfloat16)]).view(-1, 63)
        w = torch.cat([torch.full((v.shape[0], 1), amax, dtype=torch.bfloat16), v], dim=1).contiguous()
        qw, absmax, _ = ta.quantize_nf4(w.to(DEV))
        qw_o, absmax_o = oracle.C().quantize(w, 64)
        assert torch.equal(qw.cpu(), qw_o), f"absmax {amax}"
        assert torch.equal(absmax.cpu(), absmax_o)


# ------------------------------------------------------------------------------------------------
# dequantize
# ------------------------------------------------------------------------------------------------


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lut_mode", ["f32", "rounded"])
def test_dequantize_exhaustive(ta, oracle, dtype, lut_mode):
    """16 codes x every non-negative finite bf16 absmax."""
    _sync_print(f"dequantize exhaustive {dtype} {lut_mode}")
    bits = torch.arange(0, 0x7F80, dtype=torch.int32).to(torch.int16)
    amax = bits.view(torch.bfloat16).float()  # 32640 values
    nb = amax.numel()
    codes = (torch.arange(64) % 16).to(torch.uint8).repeat(nb, 1)  # each block holds all 16 codes, 4 times
    packed = ((codes[:, 0::2] << 4) | codes[:, 1::2]).reshape(-1, 1).contiguous()
    lut = oracle.nf4_lut()
    if lut_mode == "rounded":
        lut = lut.to(dtype).float()
    out = ta.dequantize_nf4(packed.to(DEV), amax.to(DEV), lut.to(DEV), 64, dtype, (nb, 64))
    ref = oracle.C().dequantize(packed, amax, lut, 64, dtype, (nb, 64))
    assert torch.equal(out.cpu().view(torch.int16 if dtype != torch.float32 else torch.int32),
                       ref.view(torch.int16 if dtype != torch.float32 else torch.int32))


@pytest.mark.parametrize("shape", [(2, 2), (3, 21), (64, 1376), (7, 999), (256, 4096)])
@pytest.mark.parametrize("blocksize", [64, 256, 4096])
def test_dequantize_shapes(ta, oracle, shape, blocksize):
    _sync_print(f"dequantize {shape} {blocksize}")
    w = _weights(shape, seed=3)
    qw, absmax = oracle.C().quantize(w, blocksize)
    out = ta.dequantize_nf4(qw.to(DEV), absmax.to(DEV), ta.nf4_code(DEV), blocksize, torch.bfloat16, shape)
    ref = oracle.C().dequantize(qw, absmax, oracle.nf4_lut(), blocksize, torch.bfloat16, shape)
    assert torch.equal(out.cpu().view(torch.int16), ref.view(torch.int16))
    # round trip bound: |deq - w| <= absmax * (largest code gap)/2 (+ bf16 rounding)
    err = (out.cpu().float() - w.float()).abs().view(-1)
    bound = absmax.repeat_interleave(blocksize)[: err.numel()] * (0.3038072 / 2 + 2**-8)
    assert (err <= bound).all()


# 16-bit outputs of 64 and 192 MiB and one element more (rule of how codes are read and the output is written), the last span of a workgroup
# cut off; fp32 outputs reach the same sizes with half the elements
@pytest.mark.parametrize("n", [2**24, 2**24 + 1, 2**25, 2**25 + 1, 3 * 2**24 + 7, 3 * 2**25, 3 * 2**25 + 1])
def test_dequantize_large_outputs(ta, n):
    _sync_print(f"dequantize large {n}")
    g = torch.Generator(device=DEV).manual_seed(n)
    packed = torch.randint(0, 256, ((n + 1) // 2, 1), dtype=torch.uint8, device=DEV, generator=g)
    absmax = torch.rand((n + 63) // 64, device=DEV, generator=g) * 0.1 + 1e-3
    lut = ta.nf4_code(DEV)
    codes = torch.stack([packed.view(-1) >> 4, packed.view(-1) & 15], dim=1).view(-1)[:n]
    nq = ta.compress_absmax(absmax)
    for stats, values in ((absmax, absmax), (nq, ta.functional.reconstruct_absmax(nq))):
        want = lut[codes.int()] * values.repeat_interleave(64)[:n]  # one product, rounded once to fp32 and once to the output's type
        for dtype in (torch.bfloat16, torch.float16, torch.float32) if n <= 3 * 2**24 + 7 else (torch.bfloat16,):
            assert torch.equal(ta.dequantize_nf4(packed, stats, lut, 64, dtype, (n,)), want.to(dtype)), (dtype, stats is nq)


def test_nested_absmax(ta, oracle):
    _sync_print("nested absmax")
    w = _weights((1024, 1024), seed=11)
    qw, absmax = oracle.C().quantize(w, 64)
    nq = ta.compress_absmax(absmax.to(DEV))
    D = oracle.create_dynamic_map()
    assert torch.equal(nq.map256.cpu(), D)
    off = oracle.C().dq_offset(absmax)
    assert nq.offset == off
    q_o, a2_o = oracle.C().dq_compress(absmax, D, off)
    assert torch.equal(nq.q.cpu(), q_o)
    assert torch.equal(nq.absmax2.cpu(), a2_o)
    rec = ta.reconstruct_absmax(nq)
    rec_o = oracle.C().dq_reconstruct(q_o, a2_o, D, off)
    assert torch.equal(rec.cpu(), rec_o)
    deq = ta.dequantize_nf4(qw.to(DEV), nq, ta.nf4_code(DEV), 64, torch.bfloat16, w.shape)
    deq_o = oracle.C().dequantize(qw, rec_o, oracle.nf4_lut(), 64, torch.bfloat16, w.shape)
    assert torch.equal(deq.cpu().view(torch.int16), deq_o.view(torch.int16))


@pytest.mark.parametrize("map_has_zero", [True, False])
def test_nested_absmax_all_equal_block(ta, oracle, map_has_zero):
    """A nested block whose absmax values all equal the offset has residual 0 everywhere: it stores
    the code of 0.0, or code 0 when the map holds no 0.0 -- as the oracle does."""
    _sync_print(f"nested absmax, zero block, map_has_zero={map_has_zero}")
    absmax = torch.full((512,), 0.25)
    absmax[256:] = torch.linspace(0.1, 0.4, 256)  # second nested block: ordinary
    D = oracle.create_dynamic_map()
    if not map_has_zero:
        D = torch.where(D == 0, torch.full_like(D, 1e-6), D)
    off = 0.25
    q_o, a2_o = oracle.C().dq_compress(absmax, D, off)
    lib = ta._lib.load()
    q = torch.empty(512, dtype=torch.uint8, device=DEV)
    a2 = torch.empty(2, dtype=torch.float32, device=DEV)
    a_dev, D_dev = absmax.to(DEV), D.to(DEV)
    ta._lib.check(lib.nf4hip_dq_compress(a_dev.data_ptr(), 512, 256, D_dev.data_ptr(), off, q.data_ptr(), a2.data_ptr(),
                                         torch.cuda.current_stream().cuda_stream))
    assert torch.equal(q.cpu(), q_o) and torch.equal(a2.cpu(), a2_o)
    assert a2_o[0] == 0 and len(set(q_o[:256].tolist())) == 1


# ------------------------------------------------------------------------------------------------
# matmul
# ------------------------------------------------------------------------------------------------


def _matmul_case(ta, oracle, M, N, K, blocksize=64, bias=False, nested=False, seed=0, x_shape=None):
    w = _weights((N, K), seed=1000 + seed)
    x = _acts(x_shape or (M, K), seed=2000 + seed)
    b = _acts((N,), seed=3000 + seed) if bias else None
    qw, absmax = oracle.C().quantize(w, blocksize)
    lut = oracle.nf4_lut()
    absmax_dev = absmax.to(DEV)
    absmax_ref = absmax
    if nested:
        absmax_dev = ta.compress_absmax(absmax.to(DEV))
        absmax_ref = ta.reconstruct_absmax(absmax_dev).cpu()
    y = ta.matmul_nf4(x.to(DEV), qw.to(DEV), None if b is None else b.to(DEV), absmax_dev, lut.to(DEV), blocksize,
                      torch.bfloat16, (N, K))
    ref = oracle.matmul_4bit_f64(x, qw, b, absmax_ref, lut, blocksize, torch.bfloat16, (N, K))
    assert y.shape == ref.shape and y.dtype == torch.bfloat16
    torch.testing.assert_close(y.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)
    return y, ref


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 15, 16])
def test_gemv_rows(ta, oracle, M):
    _sync_print(f"gemv M={M}")
    assert ta.functional.fused_route(torch.empty(M, 1024, dtype=torch.bfloat16), None, 64, torch.bfloat16, (256, 1024)) == "gemv"
    _matmul_case(ta, oracle, M, 256, 1024, seed=M)


@pytest.mark.parametrize(
    "N,K",
    [(16, 512), (48, 512), (100, 1024), (130, 2048), (1024, 4096), (4096, 4096), (1000, 14336), (2048 + 16, 8192),
     (300, 28672), (77, 32768 + 512), (8, 1 << 20)],  # the last: K split over 64 to 256 workgroups
)
@pytest.mark.parametrize("M", [1, 2, 4, 5, 16])
def test_gemv_shapes(ta, oracle, N, K, M):
    _sync_print(f"gemv N={N} K={K} M={M}")
    _matmul_case(ta, oracle, M, N, K, seed=N + K + M)


@pytest.mark.parametrize("K", [2048, 10240])
@pytest.mark.parametrize("M", [1, 2, 4, 8, 11, 16])
def test_gemv_x_outside_fp16_range(ta, oracle, M, K):
    """For 8192 < K <= 16384 the decode kernels multiply in fp16 after scaling x into range -- per lane in the row and
    quad kernels, per row of x in the tile kernel (M = 11, 16) -- (K = 10240; K = 2048 takes the bf16 arithmetic): rows
    of x far above fp16's largest value, far below its smallest, of mixed magnitudes, and with the largest finite
    bf16."""
    _sync_print(f"gemv x outside the fp16 range M={M} K={K}")
    N = 192
    w = _weights((N, K), seed=77)
    qw, absmax = oracle.C().quantize(w, 64)
    lut = oracle.nf4_lut()
    base = _acts((M, K), seed=78 + M).float()
    scales = [1e6, 2.0**100, 2.0**-60, 70000.0]
    for case in range(5):
        x = base.clone()
        if case < 4:
            x *= scales[case]
        else:  # one huge value per row among ordinary ones, and the largest finite bf16 in row 0
            x[:, 5::211] *= 1e8
            x[0, 1000] = 3.3895313892515355e38
        x = x.to(torch.bfloat16)
        y = ta.matmul_nf4(x.to(DEV), qw.to(DEV), None, absmax.to(DEV), lut.to(DEV), 64, torch.bfloat16, (N, K))
        ref = oracle.matmul_4bit_f64(x, qw, None, absmax, lut, 64, torch.float32, (N, K)).double()
        got = y.cpu().double()
        assert bool(torch.isfinite(got).all()), f"case {case}: non-finite output"
        # the tolerance of the matmul, scaled with the magnitude of each row of x
        mag = x.double().abs().amax(dim=1, keepdim=True).clamp_min(1e-300)
        typical = x.double().pow(2).mean(dim=1, keepdim=True).sqrt()
        tol = 2e-2 * typical + 2e-2 * ref.abs() + 1e-6 * mag
        assert bool(((got - ref).abs() <= tol).all()), f"case {case}: max excess {((got - ref).abs() - tol).max().item():.3g}"
    # infinities and NaNs in x reach the outputs of their row
    x = base.clone().to(torch.bfloat16)
    x[0, 3] = float("inf")
    y = ta.matmul_nf4(x.to(DEV), qw.to(DEV), None, absmax.to(DEV), lut.to(DEV), 64, torch.bfloat16, (N, K)).cpu()
    assert not bool(torch.isfinite(y[0].float()).any())
    if M > 1:
        assert bool(torch.isfinite(y[1:].float()).all())


@pytest.mark.parametrize("blocksize", [128, 512, 4096])
@pytest.mark.parametrize("M", [3, 7])
def test_gemv_blocksizes(ta, oracle, blocksize, M):
    _sync_print(f"gemv blocksize={blocksize} M={M}")
    _matmul_case(ta, oracle, M, 272, 4096, blocksize=blocksize, seed=blocksize)


@pytest.mark.parametrize("N,K", [(64, 1376), (2, 32), (33, 96), (5, 2048 + 32)])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_gemv_rows_odd_k(ta, oracle, N, K, M):
    """The row-streaming kernel needs only K % 32 == 0: quantisation blocks may straddle rows
    (K = 1376 is the intermediate size of the reference's own llama2-like test model)."""
    _sync_print(f"gemv rows odd K N={N} K={K} M={M}")
    assert ta.functional.fused_route(torch.empty(M, K, dtype=torch.bfloat16), None, 64, torch.bfloat16, (N, K)) == "gemv"
    _matmul_case(ta, oracle, M, N, K, seed=N + K)


def test_gemv_bias_and_batch_dims(ta, oracle):
    _sync_print("gemv bias / leading dims")
    y, _ = _matmul_case(ta, oracle, 6, 320, 1024, bias=True, seed=5, x_shape=(2, 3, 1024))
    assert y.shape == (2, 3, 320)


@pytest.mark.parametrize("M", [1, 4, 16])
def test_gemv_nested(ta, oracle, M):
    _sync_print(f"gemv nested M={M}")
    _matmul_case(ta, oracle, M, 1024, 8192, nested=True, seed=70 + M)


@pytest.mark.parametrize("M", [1, 4])
def test_gemv_large_k_bit_matches_dequantize_then_matmul(ta, oracle, M):
    """For K > 16384 the decode kernel rounds every weight as bf16(lut * absmax): with x = one-hot
    rows the output must equal the dequantised weight column bit for bit."""
    _sync_print(f"gemv exact M={M}")
    N, K = 192, 16384 + 2048
    w = _weights((N, K), seed=77)
    qw, absmax = oracle.C().quantize(w, 64)
    deq = oracle.C().dequantize(qw, absmax, oracle.nf4_lut(), 64, torch.bfloat16, (N, K))
    x = torch.zeros(M, K, dtype=torch.bfloat16)
    cols = [5, 4097, 16383 + 64, K - 1][:M]
    for m, c in enumerate(cols):
        x[m, c] = 1.0
    y = ta.matmul_nf4(x.to(DEV), qw.to(DEV), None, absmax.to(DEV), ta.nf4_code(DEV), 64, torch.bfloat16, (N, K))
    for m, c in enumerate(cols):
        assert torch.equal(y[m].cpu().view(torch.int16), deq[:, c].contiguous().view(torch.int16))


def test_gemv_repeatable_and_workspace_reuse(ta, oracle):
    """Split-K partial sums are added in a fixed order: repeated calls are bit-identical, and calls
    of different shapes can share the workspace back to back."""
    _sync_print("gemv repeatability")
    outs = []
    for it in range(3):
        y, _ = _matmul_case(ta, oracle, 4, 1024, 4096, seed=42)
        outs.append(y.cpu())
        _matmul_case(ta, oracle, 16, 512, 2048, seed=43)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_split_k_hand_off_holds_over_many_launches(ta):
    """2000 launches on ONE workspace, alternating between four calls whose partial sums cross workgroups (decode
    tile kernel with K split eight ways, row kernel with a long K, streaming kernel with one tile of x rows and with
    several): every result must equal the first of its kind bit for bit and every arrival counter must be back at
    zero.  The comparison runs on the device; the host looks at the verdict every 100 launches and stops at the
    first mismatch."""
    _sync_print("split-K hand-off, 2000 launches on one workspace")
    L, lib = ta._lib, ta._lib.load()
    code = ta.nf4_code(DEV)
    g = torch.Generator(device=DEV).manual_seed(7)
    calls = []
    for kind, M, N, K in [("gemv", 16, 6144, 4096), ("gemv", 1, 512, 32768), ("gemm", 64, 1024, 4096), ("gemm", 256, 1024, 8192)]:
        n = N * K
        packed = torch.randint(0, 256, (n // 2,), dtype=torch.uint8, device=DEV, generator=g)
        absmax = torch.rand(n // 64, device=DEV, generator=g) * 0.05 + 0.01
        x = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
        need = (lib.nf4hip_gemv_workspace_bytes if kind == "gemv" else lib.nf4hip_gemm_workspace_bytes)(M, N, K)
        assert need > 65536 * 4, f"{kind} M={M} [{N},{K}] is expected to split K over workgroups"
        calls.append((kind, M, N, K, packed, absmax, x, need, torch.empty(M, N, dtype=torch.bfloat16, device=DEV)))
    ws = torch.zeros(max(c[7] for c in calls), dtype=torch.uint8, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream

    def launch(c):
        kind, M, N, K, packed, absmax, x, _, out = c
        fn = lib.nf4hip_gemv if kind == "gemv" else lib.nf4hip_gemm
        L.check(fn(x.data_ptr(), L.BF16, M, packed.data_ptr(), absmax.data_ptr(), code.data_ptr(), None, N, K, 64,
                   out.data_ptr(), ws.data_ptr(), ws.numel(), stream))

    first = []
    for c in calls:
        launch(c)
        first.append(c[8].clone())
    bad = torch.zeros((), dtype=torch.bool, device=DEV)
    for it in range(2000):
        c = calls[it % len(calls)]
        c[8].zero_()
        launch(c)
        bad |= (c[8].view(torch.int16) != first[it % len(calls)].view(torch.int16)).any()
        if it % 100 == 99:
            assert not bool(bad), f"a result changed between launches {it - 99} and {it}"
    assert not bool(ws[: 65536 * 4].any()), "arrival counters not back at zero"


@pytest.fixture
def fused_gemm(ta, monkeypatch):
    """Route every call of more than 128 rows to ``nf4hip_gemm`` (the default router prefers HIP dequantize + a dense GEMM for
    some shapes); up to 128 rows ``nf4hip_stream`` serves them anyway."""
    monkeypatch.setattr(ta.functional, "DENSE_ROUTE_MIN_M", 1 << 30)


def _fused_route_of(M):
    return "stream" if M <= 128 else "gemm"


@pytest.mark.parametrize("M,N,K", [(9000, 260, 512), (4100, 1024, 1024)])
def test_dense_route(ta, oracle, M, N, K):
    """Default route for many rows of x: nf4hip_dequantize + dense GEMM."""
    _sync_print(f"dequant+gemm M={M} N={N} K={K}")
    assert ta.functional.fused_route(torch.empty(M, K, dtype=torch.bfloat16), None, 64, torch.bfloat16, (N, K)) == "dequant+gemm"
    _matmul_case(ta, oracle, M, N, K, seed=M + N + K + 1)


@pytest.mark.parametrize("M,N,K", [(200, 128, 4096), (129, 1024, 4096), (3000, 1024, 4096)])
def test_dense_route_forced(ta, oracle, M, N, K, monkeypatch):
    """The same route on shapes whose own route is the fused kernel."""
    _sync_print(f"dequant+gemm (forced) M={M} N={N} K={K}")
    monkeypatch.setattr(ta.functional, "fused_route", lambda *a, **k: "dequant+gemm")
    _matmul_case(ta, oracle, M, N, K, seed=M + N + K + 1)


@pytest.mark.parametrize(
    "M,N,K",
    [(17, 128, 64), (32, 130, 128), (128, 128, 512), (100, 100, 1344), (300, 384, 1024), (512, 1024, 4096), (257, 4096, 1024)],
)
def test_gemm_shapes(ta, oracle, M, N, K, fused_gemm):
    _sync_print(f"gemm M={M} N={N} K={K}")
    assert ta.functional.fused_route(torch.empty(M, K, dtype=torch.bfloat16), None, 64, torch.bfloat16, (N, K)) == _fused_route_of(M)
    _matmul_case(ta, oracle, M, N, K, seed=M + N + K)


@pytest.mark.parametrize("M,N,K,kw", [
    (20, 28672, 512, {}), (49, 28672, 512, {}), (64, 28700, 576, {"nested": True}), (128, 28700, 576, {"bias": True}), (129, 28672, 640, {"nested": True}),
    (300, 28930, 512, {"blocksize": 256}), (512, 28672, 1024, {}), (700, 4 * 28672, 128, {"bias": True}),
])
def test_gemm_route_tall_weights(ta, oracle, M, N, K, kw, fused_gemm):
    """Tall weights through the streaming kernel and the fused GEMM kernel (ragged M and N, odd and even numbers
    of k steps, fewer k steps than pipeline stages)."""
    _sync_print(f"gemm (tall) M={M} N={N} K={K} {kw}")
    assert ta.functional.fused_route(torch.empty(M, K, dtype=torch.bfloat16), None, kw.get("blocksize", 64), torch.bfloat16, (N, K)) == _fused_route_of(M)
    _matmul_case(ta, oracle, M, N, K, seed=M + K, **kw)


@pytest.mark.parametrize("N,streamed", [(256, 1), (9000, 0)])
def test_gemm_recovers_dequantized_weight_bit_exact(ta, oracle, fused_gemm, N, streamed):
    """x = identity makes every output a single product 1.0 * w: the expansion in either fused kernel
    (nf4_gemm_stream.h, nf4_gemm_wide.hip) must equal nf4hip_dequantize bit for bit."""
    _sync_print(f"gemm identity N={N}")
    K = 512
    assert ta._lib.load().nf4hip_gemm_streamed(K, N, K) == streamed
    w = _weights((N, K), seed=9)
    qw, absmax = oracle.C().quantize(w, 64)
    x = torch.eye(K, dtype=torch.bfloat16)
    y = ta.matmul_nf4(x.to(DEV), qw.to(DEV), None, absmax.to(DEV), ta.nf4_code(DEV), 64, torch.bfloat16, (N, K))
    deq = oracle.C().dequantize(qw, absmax, oracle.nf4_lut(), 64, torch.bfloat16, (N, K))
    assert torch.equal(y.cpu().t().contiguous().view(torch.int16), deq.view(torch.int16))


def test_gemm_bias_nested_blocksize(ta, oracle, fused_gemm, monkeypatch):
    _sync_print("gemm bias/nested/blocksize")
    _matmul_case(ta, oracle, 64, 256, 1024, bias=True, seed=1)
    _matmul_case(ta, oracle, 64, 256, 1024, nested=True, seed=2)
    _matmul_case(ta, oracle, 64, 256, 1024, blocksize=256, seed=3)
    for K in (64, 128, 192, 256, 320):  # 1..5 k steps: the nested absmax look-ups are staged across steps
        _matmul_case(ta, oracle, 40, 300, K, nested=True, bias=True, seed=4 + K)
        _matmul_case(ta, oracle, 200, 300, K, nested=True, seed=5 + K)
        assert not ta._lib.load().nf4hip_gemm_streamed(200, 16900, K)  # the same steps in the other kernel, on either form of absmax
        _matmul_case(ta, oracle, 200, 16900, K, seed=6 + K)
        with monkeypatch.context() as m:
            m.setattr(ta.functional, "NESTED_RECONSTRUCT_MIN_M", 1 << 30)
            _matmul_case(ta, oracle, 200, 16900, K, nested=True, seed=7 + K)


@pytest.mark.parametrize("case", ["fp32", "fp16", "fp16_K_not_64", "K_not_64", "n_lt_block"])
def test_fallback_route(ta, oracle, case):
    """Shapes/dtypes outside the fused kernels take HIP dequantize + dense matmul, as
    bitsandbytes.matmul_4bit does; fp16 only where the streaming kernel does not take the shape."""
    _sync_print(f"fallback {case}")
    dtype = {"fp32": torch.float32, "fp16": torch.float16, "fp16_K_not_64": torch.float16}.get(case, torch.bfloat16)
    N, K = {"K_not_64": (64, 1376), "fp16_K_not_64": (64, 1376), "n_lt_block": (2, 2)}.get(case, (96, 256))
    w = _weights((N, K), seed=5, dtype=dtype)
    x = _acts((7, K), seed=6, dtype=dtype)
    b = _acts((N,), seed=7, dtype=dtype)
    qw, absmax = oracle.C().quantize(w, 64)
    assert ta.functional.fused_route(x, b, 64, dtype, (N, K)) == ("stream" if case == "fp16" else "dequant+linear")
    y = ta.matmul_nf4(x.to(DEV), qw.to(DEV), b.to(DEV), absmax.to(DEV), ta.nf4_code(DEV), 64, dtype, (N, K))
    ref = oracle.matmul_4bit_f64(x, qw, b, absmax, oracle.nf4_lut(), 64, dtype, (N, K))
    torch.testing.assert_close(y.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)


def test_matmul_randomized_sweep_large(ta):
    """Seeded sweep over matmul_nf4 at sizes the CPU oracle would take too long for
    (N up to 40000, K up to 28672, M up to 48: row / quad / tile kernels with their exact and
    long-list variants, the streaming kernel), each against a float64-accumulated
    matmul over sampled rows of the HIP-dequantized weight (pinned bit-exact against the oracle by the
    tests above)."""
    rng = torch.Generator().manual_seed(4321)

    def pick(options):
        return options[int(torch.randint(0, len(options), (1,), generator=rng))]

    code = ta.nf4_code(DEV)
    seen = set()
    for case in range(120):
        M = pick([1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 13, 16, 17, 24, 33, 48])
        K = pick([512, 1024, 2048, 3072, 4096, 6144, 8192, 14336, 16384 + 512, 28672])
        N = pick([1, 5, 16, 31, 64, 100, 128, 257, 1000, 2049, 4096, 6000, 14336, 20000, 40000])
        if N * K > 600_000_000:
            N = 4096
        blocksize = pick([64, 64, 64, 128, 256, 512])
        bias = pick([False, True])
        nested = pick([False, False, True])
        _sync_print(f"large sweep {case}: M={M} N={N} K={K} bs={blocksize} bias={bias} nested={nested}")
        g = torch.Generator(device=DEV).manual_seed(case)
        w = (torch.randn(N, K, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
        x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
        b = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16) if bias else None
        qw, absmax, _ = ta.quantize_nf4(w, blocksize)
        state = ta.compress_absmax(absmax) if nested else absmax
        deq = ta.dequantize_nf4(qw, state, code, blocksize, torch.bfloat16, (N, K))
        seen.add(ta.functional.fused_route(x, b, blocksize, torch.bfloat16, (N, K)))
        y = ta.matmul_nf4(x, qw, b, state, code, blocksize, torch.bfloat16, (N, K))
        rows = torch.randint(0, N, (min(N, 256),), generator=g, device=DEV)
        ref = x.double() @ deq[rows].double().t()
        if bias:
            ref = ref + b[rows].double()
        torch.testing.assert_close(y[:, rows].double(), ref, rtol=2e-2, atol=2e-2)
        del w, x, qw, absmax, deq, y
    assert seen == {"gemv", "stream"}


def test_gemm_randomized_sweep(ta, fused_gemm):
    """Seeded sweep over the streaming kernel (up to 128 rows of x, and through ``nf4hip_gemm`` on most of the shapes beyond)
    and the fused GEMM kernel (more than 128 tiles with a short K): ragged
    M and N, 1..33 k steps every blocksize, bias, nested absmax; against a float64-accumulated
    matmul over the HIP-dequantized weight."""
    rng = torch.Generator().manual_seed(8765)

    def pick(options):
        return options[int(torch.randint(0, len(options), (1,), generator=rng))]

    code = ta.nf4_code(DEV)
    for case in range(90):
        M = pick([17, 31, 33, 64, 65, 100, 128, 129, 200, 255, 256, 257, 400, 511, 513, 600])
        K = pick([64, 128, 192, 256, 320, 512, 1024, 2048 + 64, 4096, 14336])  # K splits of 1, 2, 4, 8
        N = pick([2, 31, 64, 255, 256, 257, 1000, 4096 + 18, 9000])
        blocksize = pick([b for b in (64, 64, 128, 256, 512, 1024, 2048) if K % b == 0])
        bias = pick([False, True])
        nested = pick([False, False, True])
        _sync_print(f"gemm sweep {case}: M={M} N={N} K={K} bs={blocksize} bias={bias} nested={nested}")
        g = torch.Generator(device=DEV).manual_seed(1000 + case)
        w = (torch.randn(N, K, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
        x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
        b = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16) if bias else None
        qw, absmax, _ = ta.quantize_nf4(w, blocksize)
        state = ta.compress_absmax(absmax) if nested else absmax
        deq = ta.dequantize_nf4(qw, state, code, blocksize, torch.bfloat16, (N, K))
        assert ta.functional.fused_route(x, b, blocksize, torch.bfloat16, (N, K)) == _fused_route_of(M)
        y = ta.matmul_nf4(x, qw, b, state, code, blocksize, torch.bfloat16, (N, K))
        ref = x.double() @ deq.double().t()
        if bias:
            ref = ref + b.double()
        torch.testing.assert_close(y.double(), ref, rtol=2e-2, atol=2e-2)


def test_full_size_properties(ta):
    """Llama-3-8B FFN shape at full size through size-independent properties: quantize is
    idempotent on its own dequantisation, and gemv is linear in x."""
    _sync_print("full size properties")
    N, K = 14336, 4096
    g = torch.Generator(device=DEV).manual_seed(1)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    qw, absmax, code = ta.quantize_nf4(w)
    deq = ta.dequantize_nf4(qw, absmax, code, 64, torch.bfloat16, (N, K))
    qw2, absmax2, _ = ta.quantize_nf4(deq)
    deq2 = ta.dequantize_nf4(qw2, absmax2, code, 64, torch.bfloat16, (N, K))
    assert torch.equal(deq.view(torch.int16), deq2.view(torch.int16))
    x1 = torch.randn(1, K, generator=g, device=DEV).to(torch.bfloat16)
    x2 = torch.randn(1, K, generator=g, device=DEV).to(torch.bfloat16)
    y1 = ta.matmul_nf4(x1, qw, None, absmax, code, 64, torch.bfloat16, (N, K)).float()
    y2 = ta.matmul_nf4(x2, qw, None, absmax, code, 64, torch.bfloat16, (N, K)).float()
    y12 = ta.matmul_nf4(torch.cat([x1, x2]), qw, None, absmax, code, 64, torch.bfloat16, (N, K)).float()
    torch.testing.assert_close(y12[0], y1[0], rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(y12[1], y2[0], rtol=2e-2, atol=2e-2)
    ref = (x1.float() @ deq.float().t())
    torch.testing.assert_close(y1, ref, rtol=2e-2, atol=2e-2)
    big = ta.matmul_nf4(torch.cat([x1, x2]).repeat(128, 1), qw, None, absmax, code, 64, torch.bfloat16, (N, K)).float()
    torch.testing.assert_close(big[0], ref[0], rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(big[254], ref[0], rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("N,K", [(8192, 8192), (1024, 8192), (28672, 8192), (8192, 28672)])
def test_llama70b_shapes_double_quant(ta, N, K):
    """Llama-3-70B projection shapes with 8-bit double-quantized absmax (nested blocksize 256 plus
    offset), M in {1, 4, 8, 16, 2048}, at full size: every route against a float64-accumulated matmul over
    the HIP-dequantized weight (itself pinned bit-exact against the oracle at small sizes), and the
    fused kernels' nested path against their fp32-absmax path on the reconstructed absmax."""
    _sync_print(f"70B double-quant N={N} K={K}")
    g = torch.Generator(device=DEV).manual_seed(5000 + N + K)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    qw, absmax, code = ta.quantize_nf4(w)
    nested = ta.compress_absmax(absmax)
    absmax_rec = ta.reconstruct_absmax(nested)
    deq = ta.dequantize_nf4(qw, nested, code, 64, torch.bfloat16, (N, K))
    assert torch.equal(deq, ta.dequantize_nf4(qw, absmax_rec, code, 64, torch.bfloat16, (N, K)))
    rows = torch.randint(0, N, (64,), generator=g, device=DEV)
    for M in (1, 4, 8, 16, 2048):
        x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
        y = ta.matmul_nf4(x, qw, None, nested, code, 64, torch.bfloat16, (N, K))
        ref = x.double() @ deq[rows].double().t()
        torch.testing.assert_close(y[:, rows].double(), ref, rtol=2e-2, atol=2e-2)
        if M <= 16:
            # bit for bit the same kernel's result on the reconstructed fp32 absmax: with the LDS-staged kernel wherever it
            # applies and with it held off (the library's own rule may send the two forms of absmax to different kernels)
            lib = ta._lib.load()
            for mode in (1, 0):
                assert lib.nf4hip_gemv_prefer_staged(mode) == 0
                try:
                    y3 = ta.matmul_nf4(x, qw, None, nested, code, 64, torch.bfloat16, (N, K))
                    y4 = ta.matmul_nf4(x, qw, None, absmax_rec, code, 64, torch.bfloat16, (N, K))
                finally:
                    assert lib.nf4hip_gemv_prefer_staged(-1) == 0
                assert torch.equal(y3, y4), f"nested and reconstructed absmax differ, M = {M}, staged mode {mode}"
                torch.testing.assert_close(y3[:, rows].double(), ref, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("N,K", [(28672, 4096), (128256, 4096), (16384 + 16, 4096)])
def test_gemv_every_m_on_large_weights(ta, N, K):
    """Every decode kernel at full size (fused gate/up projection, lm_head, and a shape just past
    2^26 weights with a ragged last tile -- M = 5..8 is served by the quad kernel up to that size and
    by the MFMA tile kernel beyond): against a float64-accumulated matmul over sampled rows of the
    HIP-dequantized weight, which is itself pinned bit-exact against the oracle at small sizes."""
    _sync_print(f"gemv every M, large N={N} K={K}")
    g = torch.Generator(device=DEV).manual_seed(N + K)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    qw, absmax, code = ta.quantize_nf4(w)
    deq = ta.dequantize_nf4(qw, absmax, code, 64, torch.bfloat16, (N, K))
    rows = torch.cat([torch.randint(0, N, (61,), generator=g, device=DEV), torch.tensor([0, N - 2, N - 1], device=DEV)])
    bias = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    for M in (1, 2, 3, 4, 5, 6, 7, 8, 12, 16):
        x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
        assert ta.functional.fused_route(x, bias, 64, torch.bfloat16, (N, K)) == "gemv"
        y = ta.matmul_nf4(x, qw, bias, absmax, code, 64, torch.bfloat16, (N, K))
        ref = x.double() @ deq[rows].double().t() + bias[rows].double()
        torch.testing.assert_close(y[:, rows].double(), ref, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("nested", [False, True])
def test_stream_route_short_wide_weight(ta, nested):
    """17..32 rows of x on a short, very wide weight, with bias, against a float64-accumulated matmul over sampled rows of the
    HIP-dequantized weight; sixteen of the rows alone (the same kernel, beyond K = 16384) give the same bits."""
    N, K = 2048, 20480
    _sync_print(f"stream, short wide weight nested={nested}")
    g = torch.Generator(device=DEV).manual_seed(99)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    qw, absmax, code = ta.quantize_nf4(w)
    state = ta.compress_absmax(absmax) if nested else absmax
    deq = ta.dequantize_nf4(qw, state, code, 64, torch.bfloat16, (N, K))
    rows = torch.cat([torch.randint(0, N, (61,), generator=g, device=DEV), torch.tensor([0, N - 2, N - 1], device=DEV)])
    bias = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    for M in (17, 20, 31, 32):
        x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
        assert ta.functional.fused_route(x, bias, 64, torch.bfloat16, (N, K)) == "stream"
        assert ta.functional.fused_route(x[:16], bias, 64, torch.bfloat16, (N, K)) == "stream"
        y = ta.matmul_nf4(x.reshape(1, M, K), qw, bias, state, code, 64, torch.bfloat16, (N, K))
        assert y.shape == (1, M, N)
        ref = x.double() @ deq[rows].double().t() + bias[rows].double()
        torch.testing.assert_close(y[0][:, rows].double(), ref, rtol=2e-2, atol=2e-2)
        y16 = ta.matmul_nf4(x[16:32] if M >= 32 else x[:16], qw, bias, state, code, 64, torch.bfloat16, (N, K))
        assert torch.equal(y16, y[0][16:32] if M >= 32 else y[0][:16])


@pytest.mark.parametrize("M", [1, 3, 8, 16])
def test_gemv_exact_variants_recover_dequantized_weights(ta, oracle, M):
    """K > 16384 selects the decode kernels' exact-weights variants: with one-hot rows of x every
    output is a single product 1.0 * w, so it must equal nf4hip_dequantize's value bit for bit."""
    _sync_print(f"gemv exact one-hot M={M}")
    N, K = 272, 32768
    w = _weights((N, K), seed=77)
    qw, absmax = oracle.C().quantize(w, 64)
    lut = oracle.nf4_lut()
    cols = torch.randint(0, K, (M,), generator=torch.Generator().manual_seed(M))
    x = torch.zeros(M, K, dtype=torch.bfloat16)
    x[torch.arange(M), cols] = 1.0
    assert ta.functional.fused_route(x, None, 64, torch.bfloat16, (N, K)) == "gemv"
    y = ta.matmul_nf4(x.to(DEV), qw.to(DEV), None, absmax.to(DEV), lut.to(DEV), 64, torch.bfloat16, (N, K))
    deq = oracle.C().dequantize(qw, absmax, lut, 64, torch.bfloat16, (N, K))
    assert torch.equal(y.cpu().view(torch.int16), deq[:, cols].t().contiguous().view(torch.int16))


def test_gemv_randomized_sweep(ta, oracle):
    """Seeded sweep over the decode kernels' planning space: ragged N (tile, band and batch tails),
    K from one phase to several slices, every M, bias, nested absmax and larger blocksizes, each
    against the float64 oracle."""
    rng = torch.Generator().manual_seed(1234)

    def pick(options):
        return options[int(torch.randint(0, len(options), (1,), generator=rng))]

    for case in range(48):
        M = pick([1, 2, 3, 4, 5, 7, 8, 9, 12, 16])
        K = pick([512, 1024, 1536, 2048, 3072, 4096, 5120, 6144, 8192, 11264])
        N = pick([1, 3, 15, 16, 17, 100, 127, 128, 129, 257, 400, 515, 1000, 2049])
        blocksize = pick([64, 64, 64, 128, 256, 512])
        bias = pick([False, False, True])
        nested = pick([False, False, True]) and (N * K // blocksize) >= 1
        _sync_print(f"sweep {case}: M={M} N={N} K={K} bs={blocksize} bias={bias} nested={nested}")
        assert ta.functional.fused_route(torch.empty(M, K, dtype=torch.bfloat16), None, blocksize, torch.bfloat16, (N, K)) == "gemv"
        _matmul_case(ta, oracle, M, N, K, blocksize=blocksize, bias=bias, nested=nested, seed=10 * case)
