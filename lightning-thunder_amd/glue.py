"""Decode-step glue: ctypes binding of ``libnf4hip_decode.so`` (C ABI in ``include/nf4hip_decode.h`` and
``include/nf4hip_decode_chain.h``).

Three kernels for the work between the 4-bit linears of a Llama decode step -- residual add +
RMSNorm, rotary embedding + KV-cache update + grouped-query attention, SiLU(gate) * up -- and a row
argmax for greedy sampling, used by ``decode.Llama`` / ``decode.greedy_decode`` when ``LlamaConfig.hip_glue`` is set; and
``decode_chain``, the whole step as one kernel.  The reference leaves this work to its other
executors (thunder/executors/sdpaex.py, nvFuser / torch.compile fusions); it is not part of the
bitsandbytes path.  There is no CPU fallback: without the built library these functions raise.
"""

from __future__ import annotations

import ctypes
import os
import threading

import torch

from ._workspace import WorkspacePool

LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libnf4hip_decode.so")

_vp, _i32, _i64, _f32 = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
# every symbol include/nf4hip_decode.h declares: name -> (restype, argtypes)
SYMBOLS = {
    "nf4hip_decode_last_error": (ctypes.c_char_p, []),
    "nf4hip_decode_add_rmsnorm": (_i32, [_vp, _vp, _vp, _f32, _i64, _i64, _vp, _vp]),
    "nf4hip_decode_attention_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i32]),
    "nf4hip_decode_attention": (_i32, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i64, _vp, _vp, ctypes.c_size_t, _vp]),
    "nf4hip_decode_silu_mul": (_i32, [_vp, _i64, _i64, _vp, _vp]),
    "nf4hip_decode_silu_mul_pairs": (_i32, [_vp, _i64, _i64, _vp, _vp]),
    "nf4hip_decode_argmax": (_i32, [_vp, _i64, _i64, _vp, _vp, _vp]),
}
# include/nf4hip_decode_chain.h
CHAIN_SYMBOLS = {
    "nf4hip_decode_chain_workspace_bytes": (ctypes.c_size_t, [_i64, _i64, _i64, _i32, _i32, _i64, _i64, _i64]),
    "nf4hip_decode_chain": (_i32, [_vp, _vp, _vp, _vp, _f32, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i32, _i32, _i64, _i64, _i64, _i32, _vp, _vp,
                                   ctypes.c_size_t, _vp]),
    "nf4hip_decode_chain_joined": (_i32, [_vp, _vp, _vp, _vp, _f32, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i32, _i32, _i64, _i64, _i64, _i32, _i32, _i32,
                                          _vp, _vp, ctypes.c_size_t, _vp]),
}

_lib = None
_lock = threading.Lock()
_workspace_pool = WorkspacePool(1 << 20, "decode attention")  # split-key partials and counters


def _workspace(device: torch.device, nbytes: int) -> torch.Tensor:
    """Zero-initialised scratch of the attention kernel for (device, current stream); the kernel leaves
    its counters zeroed, so the buffer is reused without clearing.  Raises instead of allocating under
    capture."""
    return _workspace_pool.get(device, nbytes)


def load(path: str | None = None) -> ctypes.CDLL:
    """Load (once) and return the shared library; raises if it has not been built."""
    global _lib
    if _lib is not None and path is None:
        return _lib
    with _lock:
        if _lib is not None and path is None:
            return _lib
        p = path or LIB_PATH
        if not os.path.exists(p):
            raise RuntimeError(
                f"{p} not found: the HIP extension has not been built "
                "(run `python -c 'import __graft_entry__ as g; g.build()'` or `make -C lightning-thunder_amd/csrc`). "
                "There is no CPU fallback."
            )
        lib = ctypes.CDLL(p)
        for name, (restype, argtypes) in {**SYMBOLS, **CHAIN_SYMBOLS}.items():
            fn = getattr(lib, name)
            fn.restype, fn.argtypes = restype, argtypes
        if path is None:
            _lib = lib
        return lib


def _check(lib, rc: int) -> None:
    if rc != 0:
        raise RuntimeError(lib.nf4hip_decode_last_error().decode())


def _bf16_cuda(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if not (t.is_cuda and t.dtype == torch.bfloat16 and t.is_contiguous()):
            raise ValueError(f"expected a contiguous bf16 tensor on the GPU, got {t.dtype} {t.device} contiguous={t.is_contiguous()}")


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(t: torch.Tensor) -> int:
    idx = t.device.index if t.device.index is not None else torch.cuda.current_device()
    if _raw_stream is not None:
        return _raw_stream(idx)
    return torch.cuda.current_stream(t.device).cuda_stream


def add_rmsnorm(x: torch.Tensor, delta: torch.Tensor | None, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """``x += delta`` in place (skipped when ``delta`` is None), then returns ``rms_norm(x) * weight``.
    ``x``, ``delta`` [rows, d], ``weight`` [d]."""
    lib = load()
    _bf16_cuda(x, weight, *(() if delta is None else (delta,)))
    rows, d = x.shape
    if delta is not None and delta.shape != x.shape:
        raise ValueError(f"{delta.shape=} != {x.shape=}")
    y = torch.empty_like(x)
    with torch.cuda.device(x.device):
        _check(lib, lib.nf4hip_decode_add_rmsnorm(x.data_ptr(), None if delta is None else delta.data_ptr(), weight.data_ptr(),
                                                  float(eps), rows, d, y.data_ptr(), _stream(x)))
    return y


def attention_decode(qkv: torch.Tensor, pos: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, kcache: torch.Tensor,
                     vcache: torch.Tensor, n_head: int, n_kv_head: int) -> torch.Tensor:
    """One new token per sequence: rotary embedding of the q and k heads in ``qkv`` [B, (H + 2 Hkv) hd],
    the new k / v rows written into ``kcache`` / ``vcache`` [B, Hkv, max_seq, hd] at position ``pos``
    (a one-element int64 tensor on the GPU), attention over rows 0..pos.  Returns [B, H hd]."""
    lib = load()
    _bf16_cuda(qkv, kcache, vcache)
    B, Hkv, max_seq, hd = kcache.shape
    if Hkv != n_kv_head or qkv.shape != (B, (n_head + 2 * n_kv_head) * hd) or vcache.shape != kcache.shape:
        raise ValueError(f"{qkv.shape=} {kcache.shape=} {vcache.shape=} do not fit {n_head=} {n_kv_head=}")
    if not (pos.is_cuda and pos.dtype == torch.int64 and pos.numel() == 1):
        raise ValueError("pos must be a one-element int64 tensor on the GPU")
    for t in (cos, sin):
        if not (t.is_cuda and t.dtype == torch.float32 and t.is_contiguous() and t.shape == (max_seq, hd)):
            raise ValueError(f"rotary tables must be contiguous fp32 [{max_seq}, {hd}] on the GPU")
    out = torch.empty((B, n_head * hd), dtype=torch.bfloat16, device=qkv.device)
    with torch.cuda.device(qkv.device):
        need = lib.nf4hip_decode_attention_workspace_bytes(B, n_head, hd)
        ws = _workspace(qkv.device, need) if need else None
        _check(lib, lib.nf4hip_decode_attention(qkv.data_ptr(), pos.data_ptr(), cos.data_ptr(), sin.data_ptr(), kcache.data_ptr(),
                                                vcache.data_ptr(), B, n_head, n_kv_head, hd, max_seq, out.data_ptr(),
                                                None if ws is None else ws.data_ptr(), 0 if ws is None else ws.numel(), _stream(qkv)))
    return out


def silu_mul(gate_up: torch.Tensor, pairs: bool = False) -> torch.Tensor:
    """``silu(gate) * up`` for ``gate_up`` [rows, 2 dff] = (gate | up), or with ``pairs`` gate and up interleaved
    (column 2j = gate j, column 2j + 1 = up j).  Returns [rows, dff]."""
    lib = load()
    _bf16_cuda(gate_up)
    rows, two = gate_up.shape
    dff = two // 2
    out = torch.empty((rows, dff), dtype=torch.bfloat16, device=gate_up.device)
    fn = lib.nf4hip_decode_silu_mul_pairs if pairs else lib.nf4hip_decode_silu_mul
    with torch.cuda.device(gate_up.device):
        _check(lib, fn(gate_up.data_ptr(), rows, dff, out.data_ptr(), _stream(gate_up)))
    return out


def decode_chain_served(device: torch.device, batch: int, n_layer: int, d_model: int, n_head: int, n_kv_head: int, d_ff: int, vocab: int,
                        max_seq: int) -> bool:
    """Has ``decode_chain`` a plan for these shapes on ``device``?"""
    with torch.cuda.device(device):
        return load().nf4hip_decode_chain_workspace_bytes(batch, n_layer, d_model, n_head, n_kv_head, d_ff, vocab, max_seq) > 0


def decode_chain_pays(batch: int, n_layer: int, d_model: int, n_head: int, max_seq: int, vocab: int) -> bool:
    """Is a step as one kernel faster than one launch per linear, over the positions of a cache of this length?

    Modelled from graph replays of both on one MI355X (us, launches / one kernel; four query heads per kv head).  A layer gains by its
    width, as six exchanges between workgroups take about as long as five launches of small kernels: eight layers, 512 positions, 1 / 3 / 8 / 16
    sequences, d 1024 (d_ff 4096) 213 / 245, 236 / 286, 274 / 320, 308 / 359; d 1536 (4096) 229 / 235, 261 / 274, 314 / 307, 366 / 351; d 2048
    (8192) 254 / 231, 302 / 284, 365 / 308, 432 / 376; d 3072 (8192) 316 / 269, 363 / 320, 430 / 373, 524 / 443; d 4096 (14336) 448 / 355,
    476 / 395, 531 / 453, 619 / 543.  Two sequences gain more than one or three (d 2048, six layers, 100 positions 229 / 210), and with up to four a
    large output head gains too (d 2048, two layers, two sequences, 500 positions, vocabulary 43000 / 99000: 91 / 91, 110 / 106).  A layer loses 4 to 7 ns
    per key of a range of keys, of which a workgroup has one (four layers, d 4096: one sequence at 4000 / 12000 / 20000 positions 235 / 207, 278 / 271,
    356 / 379; eight at 4000 / 8000 / 10900 352 / 338, 442 / 455, 504 / 544; sixteen at 2048 / 4000 / 5600 388 / 374, 473 / 490, 543 / 588; d 2048, one at
    8000 / 20000 181 / 198, 245 / 296): the position is not known where a step is recorded, so the middle of the cache stands for it.  The launch
    that fills the scratch and the wait for all workgroups cost 7..14 us a step (one layer of d 2048, 1 / 3 / 8 sequences 50 / 55, 56 / 66, 67 / 70; two
    79 / 80, 90 / 96, 108 / 104; four 139 / 130, 159 / 158, 197 / 172; one layer of d 4096 75 / 70, 81 / 82, 90 / 90).  Over 407 drawn models (d 512..4096,
    1..24 layers, 1..16 sequences, up to 20000 positions) the side that this picks is 0.1 % slower than the faster one on average, 6 % at most."""
    width = d_model / 1024
    keys = max_seq / 2 / max(1, min(8, 1024 // (batch * n_head))) / 1000
    head = width * vocab / 1e5
    if batch <= 2:
        layer, gain = (3.6 * width - 3.9 - 6.7 * keys, 2.8 * head - 10) if batch == 1 else (3.0 * width - 1.2 - 4.5 * keys, 2.8 * head - 11.5)
    elif batch <= 4:
        layer, gain = 4.0 * width - 5.0 - 4.5 * keys, 1.6 * head - 14
    else:
        layer, gain = 4.0 * width - 4.7 - 5.5 * keys, -11.5
        if d_model >= 2048 or (batch > 8 and d_model >= 1536):
            layer = max(4.0 * width - 4.7, 8.0) - 5.5 * keys
    return n_layer * layer + gain >= 0


def _chain_misfit(x, linears, norms, pos, cos, sin, kcache, vcache, n_head: int, n_kv_head: int, d_ff: int, vocab: int) -> str | None:
    """What, if anything, keeps these operands from being read as a decode step of these sizes."""
    n_layer, B, Hkv, max_seq, hd = kcache.shape
    d = x.shape[1]
    if x.shape != (B, n_head * hd) or vcache.shape != kcache.shape or Hkv != n_kv_head or len(linears) != 4 * n_layer + 1 or len(norms) != 2 * n_layer + 1:
        return f"{x.shape=} {kcache.shape=} {vcache.shape=}, {len(linears)} linears and {len(norms)} norms do not fit {n_head=} {n_kv_head=}"
    if not (pos.device == x.device and pos.dtype == torch.int64 and pos.numel() == 1):
        return "pos must be a one-element int64 tensor on the GPU"
    for t in (cos, sin):
        if not (t.device == x.device and t.dtype == torch.float32 and t.is_contiguous() and t.shape == (max_seq, hd)):
            return f"rotary tables must be contiguous fp32 [{max_seq}, {hd}] on the GPU"
    shapes = [((n_head + 2 * n_kv_head) * hd, d), (d, d), (2 * d_ff, d), (d, d_ff)] * n_layer + [(vocab, d)]
    for (qweight, absmax, quant_map), (n, k) in zip(linears, shapes):
        if not (qweight.is_contiguous() and qweight.numel() * qweight.element_size() >= n * k // 2
                and absmax.dtype == torch.float32 and absmax.is_contiguous() and absmax.numel() >= n * k // 64
                and quant_map.dtype == torch.float32 and quant_map.is_contiguous() and quant_map.numel() >= 16):
            return f"a 4-bit weight does not hold [{n}, {k}] in blocks of 64"
        if qweight.device != x.device or absmax.device != x.device or quant_map.device != x.device:
            return "a 4-bit weight lies on another device"
    for w in norms:
        if w.numel() != d:
            return f"norm weight of {w.numel()} elements, expected {d}"
    for t in (kcache, vcache, *norms):
        if t.device != x.device:
            return "a cache or a norm weight lies on another device"
    return None


def decode_chain_takes(x, linears, norms, pos, cos, sin, kcache, vcache, n_head: int, d_ff: int, vocab: int) -> bool:
    """Would ``decode_chain`` take these operands on their device?  (Everything lies on it, 16-byte aligned, in the types, sizes and
    layouts that the kernel reads, and the library has a plan for the shapes.)"""
    n_layer, B, Hkv, max_seq, _ = kcache.shape
    if not x.is_cuda or not decode_chain_served(x.device, B, n_layer, x.shape[1], n_head, Hkv, d_ff, vocab, max_seq):
        return False
    bf16 = [x, kcache, vcache, *norms]
    if not all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.data_ptr() % 16 == 0 for t in [*bf16, cos, sin, *(t for lin in linears for t in lin)]):
        return False
    return (all(t.dtype == torch.bfloat16 and t.is_contiguous() for t in bf16)
            and _chain_misfit(x, linears, norms, pos, cos, sin, kcache, vcache, n_head, Hkv, d_ff, vocab) is None)


def decode_chain(x: torch.Tensor, linears, norms, eps: float, pos: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, kcache: torch.Tensor,
                 vcache: torch.Tensor, n_head: int, n_kv_head: int, d_ff: int, vocab: int, max_workgroups: int = 0, checked: bool = False, first_members: int = 0,
                 more_members: int = 0) -> torch.Tensor:
    """A whole decode step from the embedded tokens ``x`` [B, d] to the logits [B, vocab] (``nf4hip_decode_chain``).

    ``linears``: (qweight, absmax, quant_map) of every layer's QKV, output, gate-up and down projection in that order, then of the
    output head; ``norms``: the two norm weights of every layer in order, then the final one.  ``kcache`` / ``vcache``
    [n_layer, B, n_kv_head, max_seq, 128].  Two launches on the current stream; the scratch is this call's own (under
    capture it belongs to the graph).  ``checked``: ``decode_chain_takes`` has just said yes to these operands.
    ``max_workgroups``, ``first_members``, ``more_members``: fewer workgroups, or some of them late; the answer is the same."""
    lib = load()
    if not checked:
        _bf16_cuda(x, kcache, vcache, *norms)
        misfit = _chain_misfit(x, linears, norms, pos, cos, sin, kcache, vcache, n_head, n_kv_head, d_ff, vocab)
        if misfit is not None:
            raise ValueError(misfit)
    n_layer, B, _, max_seq, _ = kcache.shape
    d = x.shape[1]
    layers = []
    for i in range(n_layer):
        layers += [t.data_ptr() for lin in linears[4 * i: 4 * i + 4] for t in lin] + [norms[2 * i + 1].data_ptr(), norms[2 * i + 2].data_ptr()]
    layer_ptrs = (ctypes.c_void_p * len(layers))(*layers)
    head_ptrs = (ctypes.c_void_p * 3)(*(t.data_ptr() for t in linears[-1]))
    out = torch.empty((B, vocab), dtype=torch.bfloat16, device=x.device)
    with torch.cuda.device(x.device):
        need = lib.nf4hip_decode_chain_workspace_bytes(B, n_layer, d, n_head, n_kv_head, d_ff, vocab, max_seq)
        ws = torch.empty(max(need, 1), dtype=torch.uint8, device=x.device)
        _check(lib, lib.nf4hip_decode_chain_joined(x.data_ptr(), layer_ptrs, head_ptrs, norms[0].data_ptr(), float(eps), pos.data_ptr(), cos.data_ptr(),
                                                   sin.data_ptr(), kcache.data_ptr(), vcache.data_ptr(), B, n_layer, d, n_head, n_kv_head, d_ff, vocab,
                                                   max_seq, max_workgroups, first_members, more_members, out.data_ptr(), ws.data_ptr(), ws.numel(), _stream(x)))
    return out


def argmax_into(logits: torch.Tensor, out: torch.Tensor, pos: torch.Tensor | None = None) -> None:
    """``out[r] = logits[r].argmax()`` for ``logits`` [rows, vocab] bf16 and ``out`` int64 with ``rows`` elements;
    ``pos`` (a one-element int64 tensor on the GPU), when given, is advanced by one in the same launch."""
    lib = load()
    _bf16_cuda(logits)
    rows, vocab = logits.shape
    if not (out.is_cuda and out.dtype == torch.int64 and out.is_contiguous() and out.numel() == rows):
        raise ValueError(f"out must be a contiguous int64 GPU tensor of {rows} elements, got {out.dtype} {tuple(out.shape)}")
    if pos is not None and not (pos.is_cuda and pos.dtype == torch.int64 and pos.numel() == 1):
        raise ValueError("pos must be a one-element int64 tensor on the GPU")
    with torch.cuda.device(logits.device):
        _check(lib, lib.nf4hip_decode_argmax(logits.data_ptr(), rows, vocab, out.data_ptr(), None if pos is None else pos.data_ptr(),
                                             _stream(logits)))
