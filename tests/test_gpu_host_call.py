"""The native host side of a fused matmul: the same bits as the call through the interpreter for everything it takes, and what it
does not take -- views, odd alignment, other types, transforms, streams without scratch -- answered or refused as there."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _weight(ta, N, K, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(N + K)
    return ta.quantize_nf4((torch.randn(N, K, generator=g, device=DEV) * 0.02).to(dtype))


@pytest.fixture
def both(ta, monkeypatch):
    """call(f): f's answer with the native step and how often that was taken, and f's answer without it."""
    lib = ta._lib.load()

    def call(f):
        taken = []

        def counting(*args, inner=lib.host_matmul):
            out = inner(*args)
            taken.append(out is not None)
            return out

        with monkeypatch.context() as m:
            m.setattr(lib, "host_matmul", counting)
            a = f()
        with monkeypatch.context() as m:
            m.setattr(lib, "host_matmul", lambda *args: None)
            b = f()
        return a, sum(taken), b

    return call


@pytest.mark.parametrize("dtype,lead,N,K,biased", [
    (torch.bfloat16, (1,), 512, 1024, False),       # row kernel
    (torch.bfloat16, (3,), 515, 2880, True),        # quad kernel, odd N
    (torch.bfloat16, (2, 8), 4096, 4096, True),     # three dimensions
    (torch.bfloat16, (), 512, 1024, False),         # a vector
    (torch.bfloat16, (45,), 5003, 2880, True),      # streaming kernel
    (torch.bfloat16, (192,), 512, 1024, False),     # prompt, kept on the fused route
    (torch.float16, (4,), 1024, 1024, True),
])  # fmt: skip
def test_same_bits(ta, both, monkeypatch, dtype, lead, N, K, biased):
    print(f"host call {dtype} {lead} [{N}, {K}]", flush=True)
    qw, absmax, code = _weight(ta, N, K, dtype)
    x = torch.randn(*lead, K, device=DEV).to(dtype)
    bias = torch.randn(N, device=DEV).to(dtype) if biased else None
    args = (qw, bias, absmax, code, 64, dtype, (N, K))
    if lead == (192,):  # (whatever the dense route's time is on this card)
        monkeypatch.setitem(ta.functional._route_measured, ta.functional._route_key(x.device, 192, N, K, 64, False, False), "gemm")
    ta.matmul_nf4(x, *args)  # (the stream's scratch)
    a, taken, b = both(lambda: ta.matmul_nf4(x, *args))
    assert torch.equal(a, b) and a.shape == (*lead, N) and a.dtype is dtype and a.is_contiguous()
    assert taken == 1


def test_nested_statistics_are_not_asked_about(ta, monkeypatch):
    asked = []
    monkeypatch.setattr(ta._lib.load(), "host_matmul", lambda *args: asked.append(1))
    qw, *nested, code = ta.functional.quantize_nf4_dq((torch.randn(512, 1024, device=DEV) * 0.02).bfloat16())
    for M in (1, 45):
        x = torch.randn(M, 1024, device=DEV).bfloat16()
        ta.functional.matmul_nf4_dq(x, qw, None, *nested, code, 64, 256, torch.bfloat16, (512, 1024))
    assert not asked


def test_not_taken(ta, both):
    N, K = 512, 1024
    qw, absmax, code = _weight(ta, N, K)
    base = torch.randn(9, 2 * K + 8, device=DEV).bfloat16()
    rest = (64, torch.bfloat16, (N, K))
    flat = torch.randn(4 * K + 8, device=DEV).bfloat16()
    cases = {
        "strided x": (base[:2, :K], qw, absmax, code),
        "unaligned x": (flat[3:3 + K].view(1, K), qw, absmax, code),
        "fp64 absmax": (base[:1, :K].contiguous(), qw, absmax.double(), code),
        "bf16 map": (base[:1, :K].contiguous(), qw, absmax, code.bfloat16()),
        "strided absmax": (base[:1, :K].contiguous(), qw, torch.stack([absmax, absmax], 1)[:, 0], code),
        "subclass": (base[:1, :K].contiguous().as_subclass(type("Sub", (torch.Tensor,), {})), qw, absmax, code),
    }
    for name, (x, q, a, c) in cases.items():
        print("host call, not taken:", name, flush=True)
        got, taken, want = both(lambda x=x, q=q, a=a, c=c: ta.matmul_nf4(x, q, None, a, c, *rest))
        assert taken == 0 and torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor)), name
    x = base[:1, :K].contiguous()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):  # whether or not the pool's stream has scratch already
        got, _, want = both(lambda: ta.matmul_nf4(x, qw, None, absmax, code, *rest))
    stream.synchronize()
    assert torch.equal(got, want)
    with pytest.raises(ValueError):
        ta.matmul_nf4(x, qw[:-1], None, absmax, code, *rest)
    with pytest.raises(ValueError):
        ta.matmul_nf4(x, qw, None, absmax[:-1], code, *rest)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda row: ta.matmul_nf4(row, qw, None, absmax, code, *rest))(base[:2, :K].contiguous())
