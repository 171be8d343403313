"""Operands smaller than a call needs are answered by torch or refused on the host: no kernel reads past their end."""

import pytest
import torch

DEV = "cuda"
bf = torch.bfloat16

# gemv, streaming kernel, gemm
SHAPES = [(1, 64, 1024), (4, 64, 1376), (16, 64, 1024), (45, 64, 1024), (300, 64, 1024)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_bias_of_another_size_has_no_kernel(ta, M, N, K):
    F = ta.functional
    x, w = torch.empty(M, K, dtype=bf), torch.empty(N, K, dtype=bf)
    assert F.fused_route(x, torch.empty(N, dtype=bf), 64, bf, (N, K)) != "dequant+linear"
    for shape in ((), (1,), (N - 1,), (N + 1,), (M + 1, N)):
        bias = torch.empty(shape, dtype=bf)
        assert F.fused_route(x, bias, 64, bf, (N, K)) == "dequant+linear", shape
        assert not F.linear_possible(x, w, bias), shape


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_bias_of_another_size_is_torchs(ta, M, N, K):
    print(f"short bias {M} [{N}, {K}]", flush=True)
    F = ta.functional
    qw, absmax, code = ta.quantize_nf4((torch.randn(N, K, device=DEV) * 0.02).to(bf))
    x = torch.randn(M, K, device=DEV).to(bf)
    args = (absmax, code, 64, bf, (N, K))
    w = ta.dequantize_nf4(qw, *args)
    one = torch.ones(1, dtype=bf, device=DEV)
    assert torch.equal(ta.matmul_nf4(x, qw, one, *args), torch.nn.functional.linear(x, w, one))
    with pytest.raises(RuntimeError):
        ta.matmul_nf4(x, qw, torch.ones(N - 1, dtype=bf, device=DEV), *args)
    assert F.matmul_nf4_epilogue(x, qw, one, *args) is None
    whole = torch.randn(N, dtype=bf, device=DEV)  # (one row of N values is N values)
    assert torch.equal(ta.matmul_nf4(x, qw, whole, *args), ta.matmul_nf4(x, qw, whole.reshape(1, N), *args))


def test_statistics_and_tables_too_small_are_refused(ta):
    F = ta.functional
    cpu = torch.device("cpu")
    assert F._code_book(torch.zeros(16, dtype=bf)).dtype is torch.float32
    with pytest.raises(ValueError):
        F._code_book(torch.zeros(15))
    assert F._plain_absmax(torch.zeros(5), 5, cpu).numel() == 5
    with pytest.raises(ValueError):
        F._plain_absmax(torch.zeros(4), 5, cpu)
    with pytest.raises(RuntimeError):
        F._plain_absmax(torch.zeros(5, device="meta"), 5, cpu)
    nested = lambda q=513, a2=3, m=256: F.NestedAbsmax(torch.zeros(q, dtype=torch.uint8), torch.zeros(a2), torch.zeros(m), 0.0, 256)
    F._nested_args(nested(), 513, cpu)
    for short in (nested(q=512), nested(a2=2), nested(m=255)):
        with pytest.raises(ValueError):
            F._nested_args(short, 513, cpu)
    with pytest.raises(RuntimeError):
        F._nested_args(nested(), 513, torch.device("meta"))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [*SHAPES, (1, 33, 32), (3, 33, 96)])  # (blocks that straddle rows, the last one cut off)
def test_short_operands_raise(ta, M, N, K):
    print(f"short operands {M} [{N}, {K}]", flush=True)
    F = ta.functional
    qw, absmax, code = ta.quantize_nf4((torch.randn(N, K, device=DEV) * 0.02).to(bf))
    assert absmax.numel() == -(-N * K // 64)
    x = torch.randn(M, K, device=DEV).to(bf)
    rest = (64, bf, (N, K))
    want = torch.nn.functional.linear(x.double(), ta.dequantize_nf4(qw, absmax, code, *rest).double())
    # (bf16 rounding of the result, 2^-9, and of a weight where the route rounds it)
    assert float((ta.matmul_nf4(x, qw, None, absmax, code, *rest).double() - want).norm() / want.norm()) < 1e-2
    nq = F.compress_absmax(absmax)
    short = F.NestedAbsmax(nq.q, nq.absmax2[:-1], nq.map256, nq.offset, nq.blocksize)
    for q, a, c in ((qw[:-1], absmax, code), (qw, absmax[:-1], code), (qw, absmax, code[:15]), (qw, short, code),
                    (qw, F.NestedAbsmax(nq.q, nq.absmax2, nq.map256[:255], nq.offset, nq.blocksize), code)):
        with pytest.raises(ValueError):
            ta.matmul_nf4(x, q, None, a, c, *rest)
        with pytest.raises(ValueError):
            ta.dequantize_nf4(q, a, c, *rest)
    with pytest.raises(RuntimeError):
        ta.matmul_nf4(x, qw, None, absmax.cpu(), code, *rest)
    with pytest.raises(ValueError):
        F.compress_absmax(absmax, map256=nq.map256[:255])
