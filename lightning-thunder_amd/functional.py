"""Tensor-level NF4 ops on PyTorch-ROCm tensors, backed by ``libnf4hip.so``.

These are the functions the executor registers as operators.  They mirror what the reference
gets from bitsandbytes at thunder/transforms/quantization.py:35-39,63:

* :func:`quantize_nf4`      -- ``bitsandbytes.functional.quantize_4bit(w, quant_type="nf4")``
* :func:`dequantize_nf4`    -- ``bitsandbytes.functional.dequantize_4bit``
* :func:`matmul_nf4`        -- ``bitsandbytes.matmul_4bit(x, qweight.t(), bias, quant_state)``

All tensors must live on the GPU (``device.type == "cuda"`` on ROCm builds of torch); kernels are
queued on ``torch.cuda.current_stream()`` and nothing synchronises.
"""

from __future__ import annotations

import ctypes
import math
import os
import warnings
from dataclasses import dataclass

import torch

from . import _lib
from ._workspace import WorkspacePool

SUPPORTED_BLOCKSIZES = (64, 128, 256, 512, 1024, 2048, 4096)

# K beyond which a call that no model above claims goes to dequantize + dense GEMM even for a few rows of x
LONG_K = 16384
# From this many rows of x on, HIP dequantize followed by the dense library GEMM is a candidate
# (the fused GEMM kernels re-expand the weight tile once per 256 rows of x and reach 1.0-1.15
# PFLOP/s, the library GEMM 1.1-1.5 PFLOP/s and the dequantize kernel runs at HBM speed); see
# _fused_gemm_wins for which of the two serves a shape.  Raise it to force the fused, allocation-free
# kernels everywhere.
DENSE_ROUTE_MIN_M = 17

_DTYPE_CODE = {torch.bfloat16: _lib.BF16, torch.float16: _lib.F16, torch.float32: _lib.F32}

# fp32 NF4 code values (QLoRA), index = 4-bit code; the table bitsandbytes stores as QuantState.code
NF4_CODE = (
    -1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
    -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
    0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
    0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0,
)  # fmt: skip


_code_masters: dict[tuple[str, torch.dtype], torch.Tensor] = {}


def nf4_code(device=None, dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """The 16-entry code book as a new tensor (``quant_map`` / ``QuantState.code``).  One master copy
    per device is kept and cloned, so that only the first call on a device pays a host-to-device
    copy (which synchronises the stream)."""
    dev = torch.device(device) if device is not None else torch.device("cpu")
    if dev.type == "cuda" and dev.index is None:
        dev = torch.device("cuda", torch.cuda.current_device())
    key = (str(dev), dtype)
    master = _code_masters.get(key)
    if master is None:
        master = torch.tensor(NF4_CODE, dtype=torch.float32, device=dev).to(dtype)
        _code_masters[key] = master
    return master.clone()


_map_masters: dict[str, torch.Tensor] = {}


def _dynamic_map_values() -> torch.Tensor:
    """Built on the CPU in fp32 whatever the process's default device and dtype are: the result is kept, and quantised
    weights depend on its last bits."""
    data: list[float] = []
    for i in range(7):
        boundaries = torch.linspace(0.1, 1, 2**i + 1, dtype=torch.float32, device="cpu")
        means = (boundaries[:-1] + boundaries[1:]) / 2.0
        scale = 10 ** (-6 + i)
        data += (scale * means).tolist()
        data += (-scale * means).tolist()
    data += [0.0, 1.0]
    assert len(data) == 256
    data.sort()
    return torch.tensor(data, dtype=torch.float32, device="cpu")


def _dynamic_map_master(device=None) -> torch.Tensor:
    """The map as this package's own tensor, one per device (default: torch's default device): read it, never hand it
    out (``dynamic_map`` gives copies)."""
    dev = torch.device(device) if device is not None else torch.get_default_device()
    if dev.type == "cuda" and dev.index is None:
        dev = torch.device("cuda", torch.cuda.current_device())
    master = _map_masters.get(str(dev))
    if master is None:
        master = _map_masters[str(dev)] = _dynamic_map_values().to(dev)
    return master


def dynamic_map(device=None) -> torch.Tensor:
    """The 256-entry signed "dynamic" 8-bit code bitsandbytes uses for nested absmax quantisation
    (``create_dynamic_map(signed=True, max_exponent_bits=7, total_bits=8)``), as a new tensor.  One master copy per
    device is kept and cloned: building it on the host and copying it over took 0.1 ms of every nested quantisation."""
    return _dynamic_map_master(device).clone()


@dataclass
class NestedAbsmax:
    """absmax in nested ("double quantised") form: ``map256[q] * absmax2[i // blocksize] + offset``."""

    q: torch.Tensor  # uint8 [nblocks]
    absmax2: torch.Tensor  # fp32 [ceil(nblocks / blocksize)]
    map256: torch.Tensor  # fp32 [256]
    offset: float
    blocksize: int = 256


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream() -> int:
    """hipStream_t of the current stream of the current device (the raw query where this torch has
    it: it skips building a Stream object, a third of the host time of a small call)."""
    if _raw_stream is not None:
        return _raw_stream(torch.cuda.current_device())
    return torch.cuda.current_stream().cuda_stream


class _on_device:
    """``torch.cuda.device(dev)`` that does nothing when ``dev`` is already current."""

    def __init__(self, device: torch.device):
        idx = device.index
        self._ctx = None if idx is None or idx == torch.cuda.current_device() else torch.cuda.device(idx)

    def __enter__(self):
        if self._ctx is not None:
            self._ctx.__enter__()

    def __exit__(self, *exc):
        if self._ctx is not None:
            return self._ctx.__exit__(*exc)


def _require_gpu(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError(f"NF4 HIP ops need GPU tensors, got a tensor on {t.device}")


def _require_device(device: torch.device, *tensors: torch.Tensor) -> None:
    for t in tensors:
        if t is not None and t.device != device:
            raise RuntimeError(f"NF4 HIP ops need all operands on one device, got a tensor on {t.device} beside one on {device}")


def _aligned(t: torch.Tensor) -> torch.Tensor:
    """Contiguous and 16-byte aligned view or copy of ``t``."""
    t = t.contiguous()
    if t.data_ptr() % 16:
        t = t.clone(memory_format=torch.contiguous_format)
    return t


def _code_book(quant_map: torch.Tensor) -> torch.Tensor:
    """``quant_map`` as the kernels read it: sixteen fp32 values."""
    if quant_map.numel() < 16:
        raise ValueError(f"quant_map holds {quant_map.numel()} values, need 16")
    return _aligned(quant_map if quant_map.dtype is torch.float32 else quant_map.to(torch.float32))


def _plain_absmax(absmax: torch.Tensor, nblocks: int, device: torch.device) -> torch.Tensor:
    """fp32 statistics of ``nblocks`` blocks as the kernels read them."""
    _require_device(device, absmax)
    if absmax.numel() < nblocks:
        raise ValueError(f"absmax holds {absmax.numel()} entries, need {nblocks}")
    return _aligned(absmax if absmax.dtype is torch.float32 else absmax.to(torch.float32))


def _check_blocksize(blocksize: int) -> None:
    if blocksize not in SUPPORTED_BLOCKSIZES:
        raise ValueError(f"blocksize must be one of {SUPPORTED_BLOCKSIZES}, got {blocksize}")


# ------------------------------------------------------------------------------------------------
# quantize / dequantize
# ------------------------------------------------------------------------------------------------


def quantize_nf4(w: torch.Tensor, blocksize: int = 64):
    """Blockwise NF4 quantisation of ``w`` (bf16/f16/f32, any shape, flattened row-major).

    Returns ``(qweight uint8 [(n+1)//2, 1], absmax fp32 [ceil(n/blocksize)], code fp32 [16])``,
    the tensors the reference stores as ``<w>``, ``<w>.absmax`` and ``<w>.code``
    (thunder/transforms/quantization.py:87-89).
    """
    _check_blocksize(blocksize)
    _require_gpu(w)
    if w.dtype not in _DTYPE_CODE:
        raise TypeError(f"cannot quantize dtype {w.dtype}")
    lib = _lib.load()
    w = _aligned(w.detach())
    n = w.numel()
    with _on_device(w.device):
        packed = torch.empty(((n + 1) // 2, 1), dtype=torch.uint8, device=w.device)
        absmax = torch.empty(((n + blocksize - 1) // blocksize,), dtype=torch.float32, device=w.device)
        _lib.check(lib.nf4hip_quantize(w.data_ptr(), _DTYPE_CODE[w.dtype], n, blocksize, packed.data_ptr(), absmax.data_ptr(), _stream()))
    return packed, absmax, nf4_code(w.device)


def dequantize_nf4(qweight, absmax, quant_map, blocksize, dtype, shape) -> torch.Tensor:
    """``cast(quant_map[code] * absmax[block])`` reshaped to ``shape``; ``absmax`` is an fp32
    tensor or a :class:`NestedAbsmax`."""
    _check_blocksize(blocksize)
    if dtype not in _DTYPE_CODE:
        raise TypeError(f"cannot dequantize to dtype {dtype}")
    shape = tuple(int(s) for s in shape)
    n = math.prod(shape)
    lib = _lib.load()
    _require_gpu(qweight, quant_map)
    qweight = _aligned(qweight)
    if qweight.numel() < (n + 1) // 2:
        raise ValueError(f"qweight holds {qweight.numel()} bytes, shape {shape} needs {(n + 1) // 2}")
    _require_device(qweight.device, quant_map)
    quant_map = _code_book(quant_map)
    nblocks = (n + blocksize - 1) // blocksize
    with _on_device(qweight.device):
        out = torch.empty(shape, dtype=dtype, device=qweight.device)
        if isinstance(absmax, NestedAbsmax):
            nq = _nested_args(absmax, nblocks, qweight.device)
            _lib.check(
                lib.nf4hip_dequantize_dq(qweight.data_ptr(), nq[0].data_ptr(), nq[1].data_ptr(), nq[2].data_ptr(), nq[3], nq[4],
                                         quant_map.data_ptr(), n, blocksize, out.data_ptr(), _DTYPE_CODE[dtype], _stream())
            )  # fmt: skip
        else:
            absmax = _plain_absmax(absmax, nblocks, qweight.device)
            _lib.check(
                lib.nf4hip_dequantize(qweight.data_ptr(), absmax.data_ptr(), quant_map.data_ptr(), n, blocksize,
                                      out.data_ptr(), _DTYPE_CODE[dtype], _stream())
            )  # fmt: skip
    return out


# ------------------------------------------------------------------------------------------------
# nested (double) quantisation of absmax
# ------------------------------------------------------------------------------------------------


def _nested_args(nq: NestedAbsmax, nblocks: int, device: torch.device):
    """Nested statistics of ``nblocks`` blocks as the kernels read them."""
    _require_device(device, nq.q, nq.absmax2, nq.map256)
    if nq.q.numel() < nblocks:
        raise ValueError(f"nested absmax holds {nq.q.numel()} codes, need {nblocks}")
    if nq.absmax2.numel() * nq.blocksize < nblocks or nq.map256.numel() < 256:
        raise ValueError(f"nested absmax holds {nq.absmax2.numel()} values for blocks of {nq.blocksize} and a map of {nq.map256.numel()}, need "
                         f"values for {nblocks} codes and a map of 256")
    return (_aligned(nq.q), _aligned(nq.absmax2.to(torch.float32)), _aligned(nq.map256.to(torch.float32)), float(nq.offset), int(nq.blocksize))


def compress_absmax(absmax: torch.Tensor, nested_blocksize: int = 256, map256: torch.Tensor | None = None) -> NestedAbsmax:
    """bitsandbytes' ``compress_statistics=True``: subtract the mean, then 8-bit blockwise quantise.
    The mean is taken in float64 and rounded to fp32 once, so it does not depend on reduction order."""
    _check_blocksize(nested_blocksize)
    _require_gpu(absmax)
    if map256 is not None:
        _require_device(absmax.device, map256)
        if map256.numel() < 256:
            raise ValueError(f"map256 holds {map256.numel()} values, need 256")
    lib = _lib.load()
    absmax = _aligned(absmax.to(torch.float32))
    nb = absmax.numel()
    offset = float(absmax.double().mean().to(torch.float32)) if nb else 0.0
    with _on_device(absmax.device):
        if map256 is None:
            map256 = dynamic_map(absmax.device)
        map256 = _aligned(map256.to(torch.float32))
        q = torch.empty(nb, dtype=torch.uint8, device=absmax.device)
        absmax2 = torch.empty(((nb + nested_blocksize - 1) // nested_blocksize,), dtype=torch.float32, device=absmax.device)
        _lib.check(lib.nf4hip_dq_compress(absmax.data_ptr(), nb, nested_blocksize, map256.data_ptr(), offset, q.data_ptr(), absmax2.data_ptr(), _stream()))
    return NestedAbsmax(q, absmax2, map256, offset, nested_blocksize)


def reconstruct_absmax(nq: NestedAbsmax) -> torch.Tensor:
    lib = _lib.load()
    nb = nq.q.numel()
    _require_gpu(nq.q)
    q, a2, m, off, bs = _nested_args(nq, nb, nq.q.device)
    with _on_device(q.device):
        out = torch.empty(nb, dtype=torch.float32, device=q.device)
        _lib.check(lib.nf4hip_dq_reconstruct(q.data_ptr(), a2.data_ptr(), m.data_ptr(), off, nb, bs, out.data_ptr(), _stream()))
    return out


# Nested state as plain tensors (what a state dict can hold): absmax_q uint8 [nblocks], nested_absmax fp32
# [ceil(nblocks / nested_blocksize)], nested_quant_map fp32 [256], nested_offset fp32 [1].  The C ABI takes the
# offset by value; reading it back from the device costs a synchronisation, so it is read once per tensor and
# again only after the tensor was written to (torch bumps ``_version`` on every in-place write) or rebound to other
# storage.  The value is kept ON the tensor object: it dies with it, so a new tensor that happens to get a dead one's
# id and address (CPython reuses ids, the caching allocator reuses addresses) can never see a stale value.
_OFFSET_ATTR = "_nf4hip_offset_value"


def _remember_offset(nested_offset: torch.Tensor, value: float) -> None:
    setattr(nested_offset, _OFFSET_ATTR, (nested_offset.data_ptr(), nested_offset._version, value))


def _offset_value(nested_offset) -> float:
    if not isinstance(nested_offset, torch.Tensor):
        return float(nested_offset)
    hit = getattr(nested_offset, _OFFSET_ATTR, None)
    if hit is not None and hit[0] == nested_offset.data_ptr() and hit[1] == nested_offset._version:
        return hit[2]
    value = float(nested_offset.reshape(-1)[0].item())
    _remember_offset(nested_offset, value)
    return value


def nested_state(absmax_q, nested_absmax, nested_quant_map, nested_offset, nested_blocksize: int = 256) -> NestedAbsmax:
    return NestedAbsmax(absmax_q, nested_absmax, nested_quant_map, _offset_value(nested_offset), int(nested_blocksize))


def quantize_nf4_dq(w: torch.Tensor, blocksize: int = 64, nested_blocksize: int = 256):
    """NF4 quantisation with double-quantised statistics (bitsandbytes' ``compress_statistics=True``).  Returns
    ``(qweight, absmax_q, nested_absmax, nested_quant_map, nested_offset, code)``; ``nested_offset`` is a one-element
    fp32 tensor so that it can live in a state dict."""
    if not w.is_cuda or w.numel() == 0 or w.dtype not in _DTYPE_CODE:
        qw, absmax, code = quantize_nf4(w, blocksize)
        nq = compress_absmax(absmax, nested_blocksize)
        offset = torch.tensor([nq.offset], dtype=torch.float32, device=qw.device)
        _remember_offset(offset, float(nq.offset))
        return qw, nq.q, nq.absmax2, nq.map256, offset, code
    _check_blocksize(blocksize)
    _check_blocksize(nested_blocksize)
    lib = _lib.load()
    w = _aligned(w.detach())
    dev, n = w.device, w.numel()
    nblocks = (n + blocksize - 1) // blocksize
    with _on_device(dev):
        # the long kernel first: what the others need is prepared while it runs ([28672, 8192]: 138 -> 129.5 us)
        stream, sums = _stream(), _lib.DQ_STATISTICS_WORKSPACE_BYTES
        qw = torch.empty(((n + 1) // 2, 1), dtype=torch.uint8, device=dev)
        scratch = torch.empty(sums + 4 * nblocks, dtype=torch.uint8, device=dev)  # partial sums, absmax in fp32: nobody keeps them
        absmax = scratch.data_ptr() + sums
        _lib.check(lib.nf4hip_quantize(w.data_ptr(), _DTYPE_CODE[w.dtype], n, blocksize, qw.data_ptr(), absmax, stream))
        q = torch.empty(nblocks, dtype=torch.uint8, device=dev)
        absmax2 = torch.empty(((nblocks + nested_blocksize - 1) // nested_blocksize,), dtype=torch.float32, device=dev)
        map256, code, offset = (torch.empty(k, dtype=torch.float32, device=dev) for k in (256, 16, 1))
        _lib.check(lib.nf4hip_dq_statistics(absmax, nblocks, nested_blocksize, _dynamic_map_master(dev).data_ptr(), q.data_ptr(),
                                            absmax2.data_ptr(), offset.data_ptr(), map256.data_ptr(), code.data_ptr(), scratch.data_ptr(),
                                            sums, stream))
        _offset_value(offset)  # one read back, behind all three kernels: the matmuls' C ABI takes the offset by value
    return qw, q, absmax2, map256, offset, code


def dequantize_nf4_dq(qweight, absmax_q, nested_absmax, nested_quant_map, nested_offset, quant_map, blocksize, nested_blocksize,
                      dtype, shape) -> torch.Tensor:
    nq = nested_state(absmax_q, nested_absmax, nested_quant_map, nested_offset, nested_blocksize)
    return dequantize_nf4(qweight, nq, quant_map, blocksize, dtype, shape)


def matmul_nf4_dq(x, qweight, bias, absmax_q, nested_absmax, nested_quant_map, nested_offset, quant_map, blocksize,
                  nested_blocksize, dtype, shape) -> torch.Tensor:
    """:func:`matmul_nf4` on double-quantised statistics given as tensors: ``absmax`` is replaced by ``(absmax_q,
    nested_absmax, nested_quant_map, nested_offset)`` and ``nested_blocksize`` follows ``blocksize``."""
    nq = nested_state(absmax_q, nested_absmax, nested_quant_map, nested_offset, nested_blocksize)
    return matmul_nf4(x, qweight, bias, nq, quant_map, blocksize, dtype, shape)


# ------------------------------------------------------------------------------------------------
# matmul
# ------------------------------------------------------------------------------------------------

# 65 MiB -- 256 partial tiles of 256 x 256 floats (nf4hip_linear's two pieces of 128 tiles) and the counter region -- is the
# most any kernel asks for, so a stream's buffer is allocated once.
_workspace_pool = WorkspacePool(65 << 20, "NF4 matmul")


def _gemv_workspace(device: torch.device, nbytes: int, stream: int | None = None) -> torch.Tensor:
    """Zero-initialised scratch of the split-K kernels for (device, stream); the kernels leave their
    counters zeroed, so it is reused without clearing.  Raises instead of allocating under capture."""
    return _workspace_pool.get(device, nbytes, stream)


def reserve_workspace(device=None, nbytes: int | None = None) -> int:
    """Give the current stream of ``device`` its matmul workspace now (for example before capturing a
    graph on a stream that has not run an NF4 matmul yet).  Returns the buffer's size in bytes."""
    dev = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    with _on_device(dev):
        return _workspace_pool.reserve(dev, nbytes)


def _gemm_plan(M: int, N: int, K: int) -> tuple[int, int, int, int]:
    """``(rows of x per tile, tiles, pieces per tile along K, workgroups)`` of the fused GEMM for this shape: the
    library's own answer (``nf4hip_gemm_plan``), so that the time models below never restate a launcher's rules."""
    plan = (ctypes.c_int * 4)()
    _lib.check(_lib.load().nf4hip_gemm_plan(M, N, K, ctypes.byref(plan)))
    return plan[0], plan[1], plan[2], plan[3]


def _dense_gemm_us(M: int, N: int, K: int) -> float:
    """Model of the dense route for more than 128 rows of x, kernel time: the dequantize pass (10 us with the gap to the
    GEMM + 0.45 us per million weights) plus the library GEMM, 3 us + flops / rate with 1 / rate = 1 / cap(M) + 85 / t in s per PFLOP: cap
    is the rate the library reaches for M rows of x on a full, power-limited chip (1.0 PFLOP/s at 256 rows, 1.3
    at 512, 1.4 at 1024, 1.5 at 2048, 1.6 at 4096, 1.68 beyond, times K / (K + 512) for the start and end of the
    k loop) and t the number of 128 x 128 output tiles (few
    tiles leave CUs idle).  Measured (kernel trace) / modelled, us: [4096, 4096] M = 512 / 2048 / 8192: 42 / 74 / 217 vs
    45 / 74 / 214; [1024, 4096] M = 512 / 8192: 25 / 72 vs 30 / 68; [14336, 4096] M = 512 / 2048 / 8192: 89 / 236 / 676 vs 99 /
    227 / 684; [4096, 14336] M = 512 / 2048: 110 / 250 vs 136 / 232; lm_head M = 512 / 2048 / 8192: 788 / 1850 / 6191 vs 735 /
    1868 / 6005."""
    cap = 1.0 if M <= 256 else 1.3 if M <= 512 else 1.4 if M <= 1024 else 1.5 if M <= 2048 else 1.6 if M <= 4096 else 1.68
    cap *= K / (K + 512.0)
    t = ((M + 127) // 128) * ((N + 127) // 128)
    per_pflop = 1.0 / cap + 85.0 / t
    return 10.0 + 0.45 * N * K / 1e6 + 3.0 + 2.0 * M * N * K * per_pflop / 1e9


def _fused_gemm_wins(M: int, N: int, K: int, nested: bool = False) -> bool:
    """Is ``nf4hip_gemm`` faster than dequantize + dense GEMM (calls that ``_stream_takes`` leaves)?  Both sides are
    modelled from measurements on MI355X, the fused one by its launcher (``nf4hip_gemm_us``).  While the streaming kernel
    serves the call, that stands against what ``nf4hip_linear`` takes behind the dequantize pass, 3-18 % longer than the
    library GEMM the dense model describes (fused measured / modelled vs dense route, us: M = 1457 [3616, 14528] 203 / 213 vs 183,
    M = 2957 [2235, 10944] 163 / 169 vs 171, M = 2392 [1332, 17344] 141 / 146 vs 186, M = 2691 [664, 9088] 57 / 60 vs 94).  Beyond, the
    fused kernel runs at 1.0-1.15 PFLOP/s, the library GEMM at up to 1.5, but the dense route first writes the bf16 weight: the two
    cross near 1024 rows of x (fused vs dense, us, M = 1024 / 2048: [14336, 4096] 117 / 232 vs 118 / 198; [28672, 4096] 239 / 473 vs 238 /
    405; [28672, 8192] 442 / 881 vs 466 / 789; lm_head [128256, 4096] 978 / 1938 vs 1099 / 1831).  A tie goes to the fused kernel,
    which needs no transient bf16 weight."""
    # nested absmax: the fp32 absmax is written out ahead of the fused kernel (_matmul_nf4_on), 2-7 % on top; the
    # dequantize pass of the dense route resolves the codes itself at no measurable cost
    lib = _lib.load()
    margin = 1.15 if lib.nf4hip_gemm_streamed(M, N, K) else 1.03
    return lib.nf4hip_gemm_us(M, N, K) * (1.05 if nested else 1.0) <= margin * _dense_gemm_us(M, N, K)


# Many rows of x: the fused GEMM and dequantize + dense GEMM are within a few per cent of each other over a wide range
# of shapes, and which one leads moves with the board (clocks under a power limit, the library's GEMM heuristics).  The
# time models above are the answer where nothing can be measured (on the CPU, under stream capture); otherwise the
# first call of a shape on a device times both routes once -- a few launches each -- and every later call takes the
# faster one.  fp16 in the range of the streaming kernel: that kernel against dequantize + the library's GEMM, which no model
# predicts (it is 2.3 times to 0.86 times as fast from 1000 rows on: M = 1375 [512, 24320] 60 vs 138 us, M = 1388 [4284, 15168] 229 vs 197, M = 1003
# [4224, 3904] 60 vs 52; below 1000 rows the kernel was ahead on every shape tried, and is the answer where nothing is measured).
# NF4HIP_CALIBRATE=0 switches the measurement off.
CALIBRATE_MIN_M = 129
_route_measured: dict[tuple, str] = {}


def _route_key(device: torch.device, M: int, N: int, K: int, blocksize: int, nested: bool, has_bias: bool, f16: bool = False) -> tuple:
    index = device.index if device.index is not None else (torch.cuda.current_device() if device.type == "cuda" else -1)
    return (device.type, index, M, N, K, blocksize, nested, has_bias, f16)


def _calibration_enabled() -> bool:
    return os.environ.get("NF4HIP_CALIBRATE", "1") != "0"


def _library_gemm_allowed() -> bool:
    """Is dequantize + the vendor library's GEMM ("dequant+libgemm") one of the routes that are timed against each
    other?  Yes unless NF4HIP_LIBRARY_GEMM=0, which keeps every fused-eligible call on this package's own kernels.  It
    is only ever chosen by measurement, and only when it beats both hand-written routes by more than 3 %."""
    return os.environ.get("NF4HIP_LIBRARY_GEMM", "1") != "0"


def _measure_route(key: tuple, candidates: dict, launches: int = 3) -> str:
    """Time every candidate (a callable per route name) on the current stream: one untimed call, then ``launches``
    calls between two events; remember and return the fastest.  The vendor library's GEMM ("dequant+libgemm") has to
    beat the best hand-written route by more than 3 %; a candidate within 2 % of the best that needs no transient
    dense weight ("gemm", "stream") is preferred."""
    times = {}
    for name, fn in candidates.items():
        fn()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(launches):
            fn()
        e1.record()
        e1.synchronize()
        times[name] = e0.elapsed_time(e1)
    best = min(times, key=times.get)
    own = {name: t for name, t in times.items() if name != "dequant+libgemm"}
    if best == "dequant+libgemm" and own and min(own.values()) <= 1.03 * times[best]:
        best = min(own, key=own.get)
    for fused in ("gemm", "stream"):
        if fused in times and times[fused] <= 1.02 * times[best]:
            best = fused
    _route_measured[key] = best
    return best


STREAM_MAX_M = 128
STREAM_F16_MAX_M = 2048
STREAM_LONG_WEIGHT = 1 << 25


def _is_plain(*tensors) -> bool:
    """Can these be handed to a kernel by address?  No: anything that differentiates, transforms, traces or casts -- the
    fp16 route without a kernel of its own is a torch operation, which does all of that."""
    if torch.is_autocast_enabled("cuda") or torch._C._len_torch_dispatch_stack() or torch._C._functorch.peek_interpreter_stack() is not None:
        return False
    if torch.autograd.forward_ad._current_level >= 0 or torch.overrides._len_torch_function_stack():
        return False
    grad = torch.is_grad_enabled()
    return all(t is None or (type(t) in (torch.Tensor, torch.nn.Parameter) and not (grad and t.requires_grad)) for t in tensors)


def _stream_takes(M: int, N: int, K: int, f16: bool) -> bool:
    """Does ``nf4hip_stream`` serve M rows of bf16 or fp16 x (K a multiple of 64 and of the blocksize)?

    bf16, 17..128 rows: always (graph replay, cold weights, us, against the former kernels: [4096, 4096] M = 32 / 64 / 128 18.0 / 18.7 /
    28.3 vs 9.7 / 14.2 / 26.9; [14336, 4096] 24.7 / 27.3 / 35.8 vs 14.5 / 20.0 / 32.9; lm_head [128256, 4096] 112.7 / 124.8 / 171.0 vs
    77.8 / 98.7 / 139.2).  5..16 rows: where K is no multiple of 512, which the decode kernels need ([5003, 2880] M = 8 18.8 vs
    9.5), and from 2^25 elements on beyond K = 16384, where those reproduce every weight's rounding and are slow ([8192, 28672]
    M = 8 / 16 38.7 / 45.0 vs 36.3 / 35.4, nested absmax 45.5 / 51.1 vs 35.4 / 36.3).  Smaller weights stay in the kernel that
    their epilogue forms run in.
    fp16, up to 128 rows: always; the alternative writes the dense weight first ([14336, 4096] M = 4: 47 vs 13).  Up to 2048
    rows, while the kernel's tiles fill the chip once: a candidate, measured against that route per shape (M = 256 / 512 / 1024 / 2048
    [1024, 4096] 21.0 / 23.6 / 26.8 / 33.2 vs 10.8 / 13.3 / 20.8 / 28.5; [4096, 4096] 34.7 / 40.0 / 52.7 / 75.9 vs 20.1 / 27.3 / 50.7 / 72.2;
    [4096, 14336] 90.6 / 113.9 / 146.8 / 226.1 vs 48.7 / 74.8 / 130.2 / 228.4; beyond 2048, nothing was).
    Never beyond the kernel's 32-bit offsets into a weight."""
    if K >= 1 << 24 or N * (K // 64) >= 1 << 31:
        return False
    if f16:
        return M <= STREAM_MAX_M or (M <= STREAM_F16_MAX_M and bool(_lib.load().nf4hip_stream_served(M, N, K)))
    return 16 < M <= STREAM_MAX_M or 4 < M <= 16 and (K % 512 != 0 or (K > 16384 and N * K >= STREAM_LONG_WEIGHT))


def _weight_complete(x, qweight, bias, absmax, quant_map, n: int, blocksize: int) -> bool:
    """Are the operands of an fp16 call as large as its n weights need and on one device?  Where not, the route through
    ``torch.nn.functional.linear`` answers, or raises, as it always has."""
    nested = isinstance(absmax, NestedAbsmax)
    return ((nested or absmax.numel() >= n // blocksize) and qweight.numel() >= n // 2 and quant_map.numel() >= 16
            and all(t is None or t.device == x.device for t in (qweight, bias, absmax.q if nested else absmax)))


def _decode_takes(M: int, K: int, blocksize: int) -> bool:
    """Does ``nf4hip_gemv`` serve M rows of bf16 x?  Up to four rows: the row and quad kernels, whose blocks may straddle
    weight rows; up to sixteen: the others."""
    return K % 32 == 0 if M <= 4 else M <= 16 and K % 512 == 0 and K % blocksize == 0


def fused_route(x: torch.Tensor, bias, blocksize: int, dtype: torch.dtype, shape, nested: bool = False) -> str:
    """Which kernel serves this call: ``"gemv"`` (a decode kernel), ``"stream"`` (``nf4hip_stream``: the fused kernel between a
    decode step and a prompt, and for fp16), ``"gemm"`` (``nf4hip_gemm``, fused), ``"dequant+gemm"`` (HIP dequantize, then the
    hand-written dense MFMA kernel ``nf4hip_linear``, because that is the faster of the two for many rows of x),
    ``"dequant+libgemm"`` (HIP dequantize, then the vendor library's GEMM; only when measured faster) or ``"dequant+linear"``
    (dequantize + ``torch.nn.functional.linear``, for dtypes and shapes no kernel here takes).

    Mirrors bitsandbytes.matmul_4bit: the fused single-row kernel when the shape allows, else
    dequantize followed by a dense matmul.
    """
    N, K = shape
    M = x.numel() // K if K else 0
    # (a bias of another size than N is torch's to broadcast or to refuse: the kernels read one value per weight row)
    if x.dtype is not dtype or M <= 0 or N <= 0 or blocksize not in SUPPORTED_BLOCKSIZES or (bias is not None and (bias.dtype is not dtype or bias.numel() != N)):
        return "dequant+linear"
    if dtype is torch.float16:
        serves = (K % 64 == 0 and K % blocksize == 0 and _stream_takes(M, N, K, True) and _is_plain(x, bias)
                  and (bias is None or bias.shape == (N,)))
        if not serves:
            return "dequant+linear"
        return "stream" if M <= STREAM_MAX_M else _route_measured.get(_route_key(x.device, M, N, K, blocksize, nested, bias is not None, True), "stream")
    if dtype is not torch.bfloat16 or (N * K) % 2:
        return "dequant+linear"
    if M <= 4 and _decode_takes(M, K, blocksize):
        return "gemv"
    if K % 64 or K % blocksize:
        return "dequant+linear"
    if _stream_takes(M, N, K, False):
        return "stream"
    if _decode_takes(M, K, blocksize):
        return "gemv"
    measured = _route_measured.get(_route_key(x.device, M, N, K, blocksize, nested, bias is not None))
    if measured is not None:
        return measured  # both routes were timed on this device for this shape (_measure_route)
    if _fused_gemm_wins(M, N, K, nested):
        return "gemm"  # expanding the weight tiles in registers beats writing the bf16 weight out
    # (a few rows of x beyond the streaming kernel's offsets: the k loop of a tile is long)
    return "dequant+gemm" if M >= DENSE_ROUTE_MIN_M or K > LONG_K else "gemm"


def matmul_nf4(x, qweight, bias, absmax, quant_map, blocksize, dtype, shape) -> torch.Tensor:
    """``x @ dequantize(qweight).T + bias`` with the signature of the reference operator
    ``bnb_matmul_nf4`` (thunder/transforms/quantization.py:34).  ``absmax`` may be a
    :class:`NestedAbsmax`."""
    if type(shape) is not tuple or len(shape) != 2 or type(shape[0]) is not int or type(shape[1]) is not int:
        shape = tuple(int(s) for s in shape)
        assert len(shape) == 2
    N, K = shape
    assert x.shape[-1] == K, f"{x.shape=}, rhs {shape=}"
    _require_gpu(x, qweight, quant_map, bias)
    nested = isinstance(absmax, NestedAbsmax)
    route = fused_route(x, bias, blocksize, dtype, shape, nested)
    if route == "stream" and dtype is torch.float16 and not _weight_complete(x, qweight, bias, absmax, quant_map, N * K, blocksize):
        route = "dequant+linear"
    if (route in ("gemm", "dequant+gemm", "stream") and x.numel() >= CALIBRATE_MIN_M * K and _calibration_enabled()
            and not torch.cuda.is_current_stream_capturing()):
        M, f16 = x.numel() // K, route == "stream"  # (bf16 is streamed up to 128 rows only)
        key = _route_key(x.device, M, N, K, blocksize, nested, bias is not None, f16)
        if key not in _route_measured:
            with _on_device(x.device):
                names = ["stream", "dequant+linear"] if f16 else ["gemm", "dequant+gemm"] + (["dequant+libgemm"] if _library_gemm_allowed() else [])
                route = _measure_route(key, {
                    name: (lambda name=name: _matmul_nf4_on(x, qweight, bias, absmax, quant_map, blocksize, dtype, shape, name))
                    for name in names
                })
    return _matmul_nf4_on(x, qweight, bias, absmax, quant_map, blocksize, dtype, shape, route)


# Nested absmax beyond this many rows of x: the fp32 absmax may be written out first (nf4hip_dq_reconstruct, 4 bytes per block into
# a transient buffer, 2-15 us; same two roundings, same bits).  Always ahead of the kernel of nf4_gemm_wide.hip, which resolves an 8-bit
# code through two more loads per block and k step (us, nested kernel / reconstruct + fp32 kernel / fp32 kernel alone: [28672, 8192]
# M = 512 242 / 226 / 213, M = 2048 930 / 854 / 837; [8192, 28672] M = 1024 481 / 439 / 425).  The streaming kernel loads the
# statistics of four k steps at a time where blocksize is 64 and K a multiple of 256, and hardly at all from blocksize 256 on (M = 320
# [7040, 11264] 77.5 / 80.5 / 74.2, M = 1403 [4164, 10240] 147.1 / 147.8 / 141.9); in between, per step and lane, which a call has to be
# long for to pay another launch (K % 256 != 0: M = 2047 [2816, 12352] 205 / 182 / 179, M = 602 [3016, 5056] 41.0 / 38.7 / 32.8, M = 200
# [1024, 2880] 12.4 / 13.2, M = 140 [600, 1088] 7.6 / 9.6; blocksize 128: M = 1403 [4164, 10240] 163 / 150, M = 200 [4096, 4096] 23.3 / 23.9).
NESTED_RECONSTRUCT_MIN_M = 128
NESTED_RECONSTRUCT_MIN_US = 30


def _matmul_nf4_on(x, qweight, bias, absmax, quant_map, blocksize, dtype, shape, route: str) -> torch.Tensor:
    """:func:`matmul_nf4` on a given route (one of ``fused_route``'s answers).

    A decode call on a small weight is as long as this function, so what needs no conversion is handed to the library in one native
    step (csrc/host_call.cpp; [4096, 4096], one row, 4.6 us of kernel: ``matmul_nf4`` 9.5 -> 5.3 us, of which the launch is 2.9).  What that
    step does not take -- views, other types, a stream without a workspace, tensors inside a transform -- comes back and is
    served below, as are nested statistics, which it is not asked for."""
    N, K = shape
    if route in ("dequant+linear", "dequant+gemm", "dequant+libgemm"):
        w = dequantize_nf4(qweight, absmax, quant_map, blocksize, dtype, shape).to(x.dtype)
        if route == "dequant+gemm":
            return linear_bf16(x, w, bias)  # the hand-written dense kernel
        return torch.nn.functional.linear(x, w, bias)

    device = x.device
    if device.index != torch._C._cuda_getDevice():
        with torch.cuda.device(device):
            return _matmul_nf4_on(x, qweight, bias, absmax, quant_map, blocksize, dtype, shape, route)
    lib = _lib.load()
    stream = _stream() if _raw_stream is None else _raw_stream(device.index)
    nested = isinstance(absmax, NestedAbsmax)
    if not nested:
        entry = "nf4hip_gemv" if route == "gemv" else "nf4hip_stream" if x.dtype is torch.float16 else "nf4hip_gemm"
        out = lib.host_matmul(*lib.host_calls[entry], x, qweight, absmax, quant_map, bias, N, K, blocksize,
                              _workspace_pool.peek(device.index, stream), stream)  # fmt: skip
        if out is not None:
            if type(out) is int:
                _lib.check(out)
            return out
    flat = x.dim() == 2
    x2 = _aligned(x if flat else x.reshape(-1, K))
    M = x2.shape[0]
    qweight = _aligned(qweight)
    if qweight.numel() < N * K // 2:
        raise ValueError(f"qweight holds {qweight.numel()} bytes, shape {shape} needs {N * K // 2}")
    _require_device(device, qweight, quant_map, bias)
    quant_map = _code_book(quant_map)
    b = None if bias is None else bias.contiguous()
    nblocks = -(-N * K // blocksize)  # (up to four rows of x a block may straddle weight rows, and the last may be cut off)
    out = x2.new_empty((M, N)) if type(x2) is torch.Tensor else torch.empty((M, N), dtype=x.dtype, device=device)
    if route == "gemv":
        need = lib.nf4hip_gemv_workspace_bytes(M, N, K)
        ws = _gemv_workspace(device, need, stream)
        fn, fn_dq = lib.nf4hip_gemv, lib.nf4hip_gemv_dq
    else:  # K split over workgroups: partial tiles and counters.  Under capture, on a stream that has none yet, what can do without does
        if x.dtype is torch.float16:
            need, fn, fn_dq = lib.nf4hip_stream_workspace_bytes(M, N, K), lib.nf4hip_stream, lib.nf4hip_stream_dq
        else:
            need, fn, fn_dq = lib.nf4hip_gemm_workspace_bytes(M, N, K), lib.nf4hip_gemm, lib.nf4hip_gemm_dq
        ws = _workspace_pool.get_or_none(device, need, stream) if need else None
    ws_ptr, ws_bytes = (None, 0) if ws is None else (ws.data_ptr(), ws.numel())
    bptr = None if b is None else b.data_ptr()
    code, x_ptr, out_ptr = _DTYPE_CODE[x.dtype], x2.data_ptr(), out.data_ptr()
    if (nested and route != "gemv" and M > NESTED_RECONSTRUCT_MIN_M
            and (not (route == "stream" or lib.nf4hip_gemm_streamed(M, N, K))
                 or ((blocksize == 128 or K % 256) and lib.nf4hip_gemm_us(M, N, K) > NESTED_RECONSTRUCT_MIN_US))):
        absmax, nested = reconstruct_absmax(absmax), False
    if nested:
        q, a2, m256, off, nbs = _nested_args(absmax, nblocks, device)
        rc = fn_dq(x_ptr, code, M, qweight.data_ptr(), q.data_ptr(), a2.data_ptr(), m256.data_ptr(), off, nbs,
                   quant_map.data_ptr(), bptr, N, K, blocksize, out_ptr, ws_ptr, ws_bytes, stream)  # fmt: skip
    else:
        absmax = _plain_absmax(absmax, nblocks, device)
        rc = fn(x_ptr, code, M, qweight.data_ptr(), absmax.data_ptr(), quant_map.data_ptr(), bptr,
                N, K, blocksize, out_ptr, ws_ptr, ws_bytes, stream)  # fmt: skip
    if ws is None and need:
        if rc == _lib.E_WORKSPACE:
            _gemv_workspace(device, need, stream)  # raises: a capture on a stream that has none
        if rc == 0:
            warnings.warn(f"NF4 matmul: [{N}, {K}] captured on a stream without a workspace, so K is not split over workgroups: a slower "
                          "kernel than the eager call's. Run the call once on this stream before the capture, or call reserve_workspace().",
                          stacklevel=3)
    _lib.check(rc)
    return out if flat else out.reshape(*x.shape[:-1], N)


def linear_possible(x: torch.Tensor, w: torch.Tensor, bias=None) -> bool:
    """Does ``linear_bf16`` take these operands (bf16, K a multiple of 64 and at least 128, a bias of N values or none)?"""
    K = w.shape[-1]
    return (x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and (bias is None or bias.dtype == torch.bfloat16)
            and w.dim() == 2 and (bias is None or bias.numel() == w.shape[0])
            and x.shape[-1] == K and K % 64 == 0 and K >= 128 and x.numel() > 0 and w.numel() > 0)


def linear_bf16(x: torch.Tensor, w: torch.Tensor, bias=None) -> torch.Tensor:
    """``torch.nn.functional.linear(x, w, bias)`` for bf16 operands on the hand-written dense MFMA kernel
    (``nf4hip_linear``): the GEMM that follows ``dequantize_nf4`` on the dequantize + linear route of
    bitsandbytes.matmul_4bit (MatMul4Bit.forward, reached from thunder/transforms/quantization.py:39).  ``w`` is [N, K]."""
    if not linear_possible(x, w, bias):
        raise ValueError(f"linear_bf16: bf16 operands with K a multiple of 64 (>= 128) and a bias of N values or none only, got x {tuple(x.shape)} "
                         f"{x.dtype}, w {tuple(w.shape)} {w.dtype}, bias {None if bias is None else tuple(bias.shape)}")
    _require_gpu(x, w, bias)
    lib = _lib.load()
    N, K = w.shape
    x2 = _aligned(x.reshape(-1, K))
    w = _aligned(w)
    M = x2.shape[0]
    b = None if bias is None else bias.contiguous()
    with _on_device(x.device):
        out = torch.empty((M, N), dtype=torch.bfloat16, device=x.device)
        stream = _stream()
        need = lib.nf4hip_linear_workspace_bytes(M, N, K)
        ws = _gemv_workspace(x.device, need, stream) if need else None
        ws_ptr, ws_bytes = (None, 0) if ws is None else (ws.data_ptr(), ws.numel())
        _lib.check(lib.nf4hip_linear(x2.data_ptr(), _lib.BF16, M, w.data_ptr(), None if b is None else b.data_ptr(), N, K,
                                     out.data_ptr(), ws_ptr, ws_bytes, stream))
    return out.reshape(*x.shape[:-1], N)


# ---- the decode kernels with an epilogue ---------------------------------------------------------------------


def epilogue_served(rows: int, shape, blocksize: int = 64, dtype: torch.dtype = torch.bfloat16, nested: bool = False, *,
                    rowscale_parts: int = 0, silu_pairs: bool = False, resid_norm: bool = False) -> bool:
    """Will ``matmul_nf4_epilogue`` serve ``rows`` rows of bf16 x on an [N, K] weight with this epilogue
    (``rowscale_parts``: the number of partial sums a row scale would be given, 0 for none)?  The library's own answer
    for the current device; for callers that must know before they launch the first kernel of a chain."""
    N, K = (int(s) for s in shape)
    if nested or dtype != torch.bfloat16 or blocksize not in SUPPORTED_BLOCKSIZES:
        return False
    flags = (_lib.EPI_ROWSCALE if rowscale_parts else 0) | (_lib.EPI_SILU_PAIRS if silu_pairs else 0) | (_lib.EPI_RESID_NORM if resid_norm else 0)
    return bool(_lib.load().nf4hip_gemv_epilogue_served(rows, N, K, blocksize, flags, rowscale_parts))


def matmul_nf4_epilogue(x, qweight, bias, absmax, quant_map, blocksize, dtype, shape, *, rowscale=None, silu_pairs=False,
                        resid_norm=None):
    """``matmul_nf4`` at decode shapes with the step that follows (or precedes) the linear in a decoder layer done by
    the thread that finishes each output (``nf4hip_gemv_epilogue``), one launch instead of two:

    * ``resid_norm=(resid, norm_weight)``: ``r = resid + linear(x)``; returns ``(r, xnext, sumsq)`` with
      ``xnext = r * norm_weight`` (not yet divided by the rms) and ``sumsq`` [rows, parts] partial sums of ``r**2``.
    * ``rowscale=(sumsq, eps)``: ``x`` is such an ``xnext``; the sums are multiplied by ``rsqrt(sumsq.sum(-1) / K + eps)``,
      which makes the result ``linear(rms_norm(r) * norm_weight)``.
    * ``silu_pairs``: weight rows 2j / 2j+1 are gate row j / up row j; returns ``silu(gate) * up`` [rows, N/2].

    Each output is what ``matmul_nf4`` and the step would store, bit for bit (``rowscale`` aside), except at 5..16
    rows on a weight of 2^25 elements and more with K > 16384: there the plain product runs in another kernel
    (``_stream_takes``), with the same weights and another order of its sums.

    Returns None where the library does not serve the case (more than sixteen rows of x, nested absmax, other dtypes,
    one row of x with K > 16384, ...; ``epilogue_served`` answers beforehand): the caller then runs
    ``matmul_nf4`` and the step by itself."""
    N, K = (int(s) for s in shape)
    x2 = x.reshape(-1, K)
    M = x2.shape[0]
    if isinstance(absmax, NestedAbsmax) or M > 16 or not x2.is_cuda:
        return None
    if (x.dtype is not torch.bfloat16 or dtype is not torch.bfloat16 or (bias is not None and (bias.dtype is not dtype or bias.numel() != N))
            or M == 0 or N <= 0 or blocksize not in SUPPORTED_BLOCKSIZES or (N * K) % 2 or not _decode_takes(M, K, blocksize)):
        return None
    lib = _lib.load()
    _require_device(x2.device, qweight, quant_map, bias)
    x2, qweight = _aligned(x2), _aligned(qweight)
    if qweight.numel() < N * K // 2:
        raise ValueError(f"qweight holds {qweight.numel()} bytes, too few for {shape}")
    quant_map, absmax = _code_book(quant_map), _plain_absmax(absmax, -(-N * K // blocksize), x2.device)
    b = None if bias is None else bias.contiguous()
    epi = _lib.Epilogue()
    keep = []  # tensors whose addresses the struct holds
    with _on_device(x2.device):
        out = None
        if rowscale is not None:
            sumsq, eps = rowscale
            if sumsq.dtype != torch.float32 or sumsq.dim() != 2 or sumsq.shape[0] != M or not sumsq.is_contiguous():
                raise ValueError(f"rowscale: sumsq must be a contiguous fp32 [rows, parts] tensor, got {sumsq.dtype} {tuple(sumsq.shape)}")
            epi.flags |= _lib.EPI_ROWSCALE
            epi.eps, epi.in_sumsq, epi.in_parts = float(eps), sumsq.data_ptr(), sumsq.shape[1]
            keep.append(sumsq)
        if silu_pairs:
            if N % 2:
                return None
            epi.flags |= _lib.EPI_SILU_PAIRS
        if resid_norm is not None:
            resid, norm_weight = resid_norm
            if resid.shape != (M, N) or resid.dtype != torch.bfloat16 or norm_weight.shape != (N,) or norm_weight.dtype != torch.bfloat16:
                raise ValueError(f"resid_norm: need bf16 resid [{M}, {N}] and norm_weight [{N}], got {tuple(resid.shape)} {resid.dtype}, "
                                 f"{tuple(norm_weight.shape)} {norm_weight.dtype}")
            parts = lib.nf4hip_gemv_norm_parts(M, N, K)
            if parts <= 0:
                return None
            resid, norm_weight = resid.contiguous(), norm_weight.contiguous()
            r_out, xnext = torch.empty_like(resid), torch.empty_like(resid)
            out_sumsq = torch.empty((M, parts), dtype=torch.float32, device=x2.device)
            epi.flags |= _lib.EPI_RESID_NORM
            epi.resid_in, epi.norm_weight = resid.data_ptr(), norm_weight.data_ptr()
            epi.resid_out, epi.xnext_out, epi.out_sumsq = r_out.data_ptr(), xnext.data_ptr(), out_sumsq.data_ptr()
            keep += [resid, norm_weight]
        else:
            out = torch.empty((M, N // 2 if silu_pairs else N), dtype=torch.bfloat16, device=x2.device)
        stream = _stream()
        ws = _gemv_workspace(x2.device, lib.nf4hip_gemv_workspace_bytes(M, N, K), stream)
        rc = lib.nf4hip_gemv_epilogue(x2.data_ptr(), _lib.BF16, M, qweight.data_ptr(), absmax.data_ptr(), quant_map.data_ptr(),
                                      None if b is None else b.data_ptr(), N, K, blocksize, None if out is None else out.data_ptr(),
                                      ws.data_ptr(), ws.numel(), ctypes.byref(epi), stream)
    if rc == _lib.E_SHAPE:
        return None
    _lib.check(rc)
    if resid_norm is not None:
        return r_out, xnext, out_sumsq
    return out.reshape(*x.shape[:-1], out.shape[-1])
