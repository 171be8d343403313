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
