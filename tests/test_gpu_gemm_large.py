"""``nf4hip_gemm`` on large calls: the kernel of nf4_gemm_wide.hip with its tiles cut along K, pieces that meet in the workspace
(256-row tiles on long rows, 128-row tiles from K = 2^24 on), and the general kernel of nf4_gemm.hip (x of 4 GB and more), against
a float64 product over the HIP-dequantised weight."""

import pytest
import torch

DEV = "cuda"
COUNTERS = 65536 * 4


def _weight(ta, N, K, nested, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    packed = torch.randint(0, 256, (N * K // 2, 1), dtype=torch.uint8, device=DEV, generator=g)
    absmax = torch.rand(N * K // 64, device=DEV, generator=g) * 0.05 + 0.01
    return packed, (ta.compress_absmax(absmax) if nested else absmax), ta.nf4_code(DEV)


def _gemm(ta, x, packed, stats, code, bias, N, K, out, ws, nbytes):
    L, lib = ta._lib, ta._lib.load()
    b = None if bias is None else bias.data_ptr()
    w = None if ws is None else ws.data_ptr()
    if isinstance(stats, ta.NestedAbsmax):
        return lib.nf4hip_gemm_dq(x.data_ptr(), L.BF16, x.shape[0], packed.data_ptr(), stats.q.data_ptr(), stats.absmax2.data_ptr(),
                                  stats.map256.data_ptr(), stats.offset, stats.blocksize, code.data_ptr(), b, N, K, 64, out.data_ptr(), w, nbytes,
                                  ta.functional._stream())
    return lib.nf4hip_gemm(x.data_ptr(), L.BF16, x.shape[0], packed.data_ptr(), stats.data_ptr(), code.data_ptr(), b, N, K, 64, out.data_ptr(), w,
                           nbytes, ta.functional._stream())


def _check(y, x, deq, bias, terms):
    """`terms` additions that are not of an exact zero, each within 2**-23 of the sum of magnitudes (two roundings), merges
    of eight pieces, one rounding of the result."""
    xd = x.double()
    ref, size = xd @ deq.double().t(), xd.abs() @ deq.double().abs().t()
    if bias is not None:
        ref, size = ref + bias.double(), size + bias.double().abs()
    bound = 2.0**-8 * ref.abs() + (terms + 16) * 2.0**-23 * size + 2.0**-24
    assert ((y.double() - ref).abs() <= bound).all()


def test_plan_beyond_the_streaming_offsets(ta):
    """17..128 rows keep tiles of 128 rows and their pieces along K; x of 4 GB and more is taken in whole 256-row tiles."""
    lib, plan = ta._lib.load(), ta.functional._gemm_plan
    for M, N, K in ((64, 300, 1 << 24), (17, 264, (1 << 24) + 64), (32, 4096, 1 << 24)):
        assert not lib.nf4hip_gemm_streamed(M, N, K)
        tiles = (N + 255) // 256
        assert plan(M, N, K) == (128, tiles, 8, 8 * tiles)
        assert lib.nf4hip_gemm_workspace_bytes(M, N, K) == COUNTERS + 8 * tiles * 128 * 256 * 4
    assert plan(65600, 300, 32832) == (256, 257 * 2, 1, 514) and lib.nf4hip_gemm_workspace_bytes(65600, 300, 32832) == 0
    assert plan(128, 300, 1 << 24) == (256, 2, 1, 2)  # x of exactly 4 GB


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,nested,bias", [(64, 300, 1 << 24, False, True), (17, 264, (1 << 24) + 64, True, False), (100, 40, 1 << 24, False, False)])
def test_cut_tiles_at_k_of_2_to_24(ta, M, N, K, nested, bias):
    """Eight pieces per tile: 4096 elements per row of x are not zero (so the bound stays tight), spread over all pieces and dense
    at every piece's ends; five calls on one workspace give the same bits and leave its counters at zero."""
    print(f"cut tiles M={M} [{N},{K}] nested={nested} bias={bias}", flush=True)
    lib = ta._lib.load()
    need = lib.nf4hip_gemm_workspace_bytes(M, N, K)
    assert need > COUNTERS and not lib.nf4hip_gemm_streamed(M, N, K)
    packed, stats, code = _weight(ta, N, K, nested, M)
    g = torch.Generator(device=DEV).manual_seed(N)
    ends = (torch.arange(9, device=DEV) * (K // 64) // 8 * 64).unsqueeze(1) + torch.arange(-128, 128, device=DEV)
    ends = ends.flatten().clamp(0, K - 1).unique()
    cols = torch.cat([ends.expand(M, -1), torch.randint(0, K, (M, 4096 - ends.numel()), device=DEV, generator=g)], 1)
    x = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV)
    x.scatter_(1, cols, torch.empty(cols.shape, device=DEV).normal_(0, 1, generator=g).to(torch.bfloat16))
    b = torch.empty(N, device=DEV).normal_(0, 1, generator=g).to(torch.bfloat16) if bias else None
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    assert _gemm(ta, x, packed, stats, code, b, N, K, out, None, 0) == ta._lib.E_WORKSPACE
    ws = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device=DEV)
    ws[:COUNTERS] = 0  # (partial sums are in any state)
    first = None
    for _ in range(5):
        out.fill_(float("nan"))
        ta._lib.check(_gemm(ta, x, packed, stats, code, b, N, K, out, ws, need))
        first = out.clone() if first is None else first
        assert torch.equal(out, first)
    assert not ws[:COUNTERS].any() and bool((ws[need:] == 0x5A).all())
    rows = sorted({0, 31, N // 2, N - 2, N - 1})
    deq = torch.cat([ta.dequantize_nf4(packed[r * K // 2:(r + 1) * K // 2],
                                       (ta.reconstruct_absmax(stats) if nested else stats)[r * (K // 64):(r + 1) * (K // 64)], code, 64, torch.bfloat16,
                                       (1, K)) for r in rows])
    _check(first[:, rows], x, deq, None if b is None else b[rows], 4096)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,nested,pieces", [(512, 8192, 28672, False, 4), (1249, 4096, 24064, True, 3), (2005, 3236, 20224, False, 2),
                                                 (986, 4384, 27520 + 64, False, 3)])
def test_cut_256_row_tiles(ta, M, N, K, nested, pieces):
    """Ragged M and N, an odd number of k steps (pieces of unequal length); five calls on one workspace give the same bits."""
    print(f"cut 256-row tiles M={M} [{N},{K}] nested={nested}", flush=True)
    lib = ta._lib.load()
    tiles = ((M + 255) // 256) * ((N + 255) // 256)
    assert not lib.nf4hip_gemm_streamed(M, N, K) and ta.functional._gemm_plan(M, N, K) == (256, tiles, pieces, tiles * pieces)
    need = lib.nf4hip_gemm_workspace_bytes(M, N, K)
    assert need == COUNTERS + tiles * pieces * 256 * 256 * 4
    packed, stats, code = _weight(ta, N, K, nested, M)
    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.empty(M, K, device=DEV).normal_(0, 1, generator=g).to(torch.bfloat16)
    b = torch.empty(N, device=DEV).normal_(0, 1, generator=g).to(torch.bfloat16)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    assert _gemm(ta, x, packed, stats, code, b, N, K, out, None, 0) == ta._lib.E_WORKSPACE
    ws = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device=DEV)
    ws[:COUNTERS] = 0
    first = None
    for _ in range(5):
        out.fill_(float("nan"))
        ta._lib.check(_gemm(ta, x, packed, stats, code, b, N, K, out, ws, need))
        first = out.clone() if first is None else first
        assert torch.equal(out, first)
    assert not ws[:COUNTERS].any() and bool((ws[need:] == 0x5A).all())
    _check(first, x, ta.dequantize_nf4(packed, stats, code, 64, torch.bfloat16, (N, K)), b, K // 16)


@pytest.mark.gpu
@pytest.mark.parametrize("nested", [False, True])
def test_x_of_more_than_4_gb(ta, nested):
    M, N, K = 65600, 300, 32832  # ragged in every direction, an odd number of k steps
    print(f"general kernel M={M} [{N},{K}] nested={nested}", flush=True)
    assert M * K * 2 > 1 << 32
    packed, stats, code = _weight(ta, N, K, nested, 5)
    g = torch.Generator(device=DEV).manual_seed(6)
    x = torch.empty(M, K, dtype=torch.bfloat16, device=DEV).normal_(0, 1, generator=g)
    b = torch.empty(N, device=DEV).normal_(0, 1, generator=g).to(torch.bfloat16)
    out = torch.full((M + 1, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    ta._lib.check(_gemm(ta, x, packed, stats, code, b, N, K, out, None, 0))
    deq = ta.dequantize_nf4(packed, stats, code, 64, torch.bfloat16, (N, K))
    rows = torch.cat([torch.arange(40), torch.randint(0, M, (80,), generator=torch.Generator().manual_seed(1)), torch.arange(M - 70, M)]).to(DEV)
    _check(out[rows], x[rows], deq, b, K // 16)
    assert out[:M].isfinite().all() and out[M].isnan().all()
