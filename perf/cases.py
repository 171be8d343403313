"""What a user of this package has it do, as cases that can be timed and compared.

Four kinds of work, each through the package's public entry points:

* ``linear``     -- one 4-bit linear: ``matmul_nf4`` / ``matmul_nf4_dq`` (the operators behind every quantised
                    ``nn.Linear``) or, for ``entry == "module"``, a ``jit``-ed ``nn.Linear`` itself.  From one row of x
                    (a decode step) over a few dozen (a batch being served) to thousands (prefill).
* ``quantize``   -- a dense weight to NF4, with fp32 or double-quantised statistics: what loading a model runs per weight.
* ``dequantize`` -- NF4 back to a dense weight: the reverse transform, and the first half of the reference's own route.
* ``step``       -- one token of a Llama-architecture decoder with every linear in NF4, replayed from a HIP graph as
                    ``decode.greedy_decode`` replays it.  Its answer is the logits and the caches: the logits of random
                    weights have close runners-up, so a token sampled from them would compare nothing.

Weights ~ N(0, 0.02), activations ~ N(0, 1), as in the repository's configurations and benchmark.
"""

import importlib
import math

import torch

ta = importlib.import_module("lightning-thunder_amd")
decode = importlib.import_module("lightning-thunder_amd.decode")

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
NESTED_BLOCKSIZE = 256


def _linear(m, n, k, **kw):
    return {"kind": "linear", "entry": "op", "m": m, "n": n, "k": k, "dtype": "bf16", "blocksize": 64, "nested": False, "bias": False, **kw}


def _codec(kind, n, k, **kw):
    return {"kind": kind, "n": n, "k": k, "dtype": "bf16", "blocksize": 64, "nested": False, **kw}


def _step(batch, pos, **kw):
    return {"kind": "step", "batch": batch, "pos": pos, "max_seq": 640, "layers": 32, "d_model": 4096, "d_ff": 14336, "vocab": 128256, **kw}


def listed():
    return [
        # a single small linear, called as a module at one token: latency and host work
        {**_linear(1, 4096, 4096), "entry": "module", "name": "module_m1"},
        # a half-precision model at a small batch
        {**_linear(4, 14336, 4096, dtype="fp16"), "name": "linear_fp16_m4"},
        # the output head at a batch of sixteen: the longest stream of weights a decode step has
        {**_linear(16, 128256, 4096), "name": "linear_head_m16"},
        # the down projection of a 70B-class layer with double quantisation, batch of sixteen
        {**_linear(16, 8192, 28672, nested=True), "name": "linear_down70_dq_m16"},
        # a serving batch between decode and prefill
        {**_linear(64, 14336, 4096), "name": "linear_m64"},
        # odd sizes and a bias: 45 rows of x, an odd number of weight rows, a row that is no multiple of the larger tiles
        {**_linear(45, 5003, 2880, bias=True), "name": "linear_ragged_m45"},
        # a chunk of a prompt through a long reduction
        {**_linear(512, 4096, 14336), "name": "linear_m512"},
        # a whole prompt through a 70B-class gate projection with double quantisation: the largest
        {**_linear(2048, 28672, 8192, nested=True), "name": "linear_gate70_dq_m2048"},
        # loading a model with double quantisation, one weight
        {**_codec("quantize", 28672, 8192, nested=True), "name": "quantize_dq"},
        # restoring a dense weight
        {**_codec("dequantize", 14336, 4096), "name": "dequantize"},
        # one token of the 8B-class decoder, one sequence and eight
        {**_step(1, 512), "name": "step_b1"},
        {**_step(8, 576), "name": "step_b8"},
    ]


MAX_WEIGHT = 128256 * 4096
MAX_FLOP = 2 * 2048 * 28672 * 8192


def _log_int(rng, low, high, multiple=1):
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high, max(low, round(v / multiple) * multiple))


def draw(rng):
    kind = rng.choices(["linear", "quantize", "dequantize", "step"], [12, 2, 2, 2])[0]
    if kind == "step":
        # the same decoder with fewer layers, other widths, batches and contexts
        d_model = rng.choice([2048, 4096])
        max_seq = _log_int(rng, 128, 4096, 64)
        return _step(_log_int(rng, 1, 16), rng.randrange(max_seq // 2, max_seq), max_seq=max_seq, layers=rng.randrange(2, 9), d_model=d_model,
                     d_ff=_log_int(rng, 2 * d_model, 4 * d_model, 512), vocab=_log_int(rng, 32000, 128256, 8))
    while True:
        n, k = _log_int(rng, 512, 131072, rng.choice([1, 8, 64, 256])), _log_int(rng, 1024, 28672, rng.choice([64, 256, 512]))
        if n * k > MAX_WEIGHT:
            continue
        blocksize = 128 if k % 128 == 0 and rng.random() < 0.2 else 64
        nested = rng.random() < 0.25
        if kind == "quantize":
            return _codec(kind, n, k, dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]), blocksize=blocksize, nested=nested)
        if kind == "dequantize":
            return _codec(kind, n, k, dtype=rng.choice(["bf16", "bf16", "fp16"]), blocksize=blocksize, nested=nested)
        # decode, serving batches, prompts
        low, high = rng.choices([(1, 16), (17, 128), (129, 2048)], [3, 1, 2])[0]
        m = _log_int(rng, low, high)
        if 2 * m * n * k <= MAX_FLOP:
            return _linear(m, n, k, dtype=rng.choice(["bf16"] * 4 + ["fp16"]), blocksize=blocksize, nested=nested, bias=rng.random() < 0.25)


def _normal(shape, std, dtype, g):
    return torch.empty(shape, device="cuda", dtype=torch.float32).normal_(0.0, std, generator=g).to(dtype)


def _cfg(case):
    d = case["d_model"]
    return decode.LlamaConfig(n_layer=case["layers"], d_model=d, n_head=d // 128, n_kv_head=d // 512, d_ff=case["d_ff"], vocab=case["vocab"],
                              max_seq=case["max_seq"], fused_projections=True, hip_glue=True, gate_up_interleaved=True)


def _prepare_step(case, seed, g):
    cfg = _cfg(case)
    model = ta.jit(decode.build_llama(cfg, device="cuda", seed=seed), transforms=[ta.BitsAndBytesLinearQuant4bit()])
    B = case["batch"]
    kcache, vcache = decode.new_caches(cfg, B)
    for cache in (kcache, vcache):  # what a prompt of `pos` tokens leaves behind
        for layer in cache:
            layer[:, :, : case["pos"]] = _normal((B, cfg.n_kv_head, case["pos"], cfg.head_dim), 1.0, torch.bfloat16, g)
    tok = torch.randint(0, cfg.vocab, (B, 1), generator=g, device="cuda")
    pos = torch.full((1,), case["pos"], device="cuda", dtype=torch.long)
    out = {"kcache": kcache, "vcache": vcache}

    def step():
        out["logits"] = model(tok, pos, kcache, vcache)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(side):
        step()
        step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            step()
    torch.cuda.current_stream().wait_stream(side)
    return {"kind": "step", "graph": graph, "out": out, "keep": (model, tok, pos)}


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "step":
        return _prepare_step(case, seed, g)
    n, k, dtype, blocksize, nested = case["n"], case["k"], DTYPES[case["dtype"]], case["blocksize"], case["nested"]
    w = _normal((n, k), 0.02, dtype, g)
    state = {"kind": kind, "nested": nested, "blocksize": blocksize}
    if kind == "quantize":
        return {**state, "w": w}
    if kind == "linear":
        state["x"] = _normal((case["m"], k), 1.0, dtype, g)
        state["bias"] = _normal((n,), 1.0, dtype, g) if case["bias"] else None
        if case["entry"] == "module":
            linear = torch.nn.Linear(k, n, bias=case["bias"], device="cuda", dtype=dtype).requires_grad_(False)
            linear.weight.copy_(w)
            return {**state, "kind": "module", "module": ta.jit(linear, transforms=[ta.BitsAndBytesLinearQuant4bit()])}
    if nested:
        quantized = ta.functional.quantize_nf4_dq(w, blocksize, NESTED_BLOCKSIZE)
        state["qweight"], state["stats"] = quantized[0], (*quantized[1:], blocksize, NESTED_BLOCKSIZE, dtype, (n, k))
    else:
        qweight, absmax, code = ta.quantize_nf4(w, blocksize)
        state["qweight"], state["stats"] = qweight, (absmax, code, blocksize, dtype, (n, k))
    return state


def run(state):
    kind = state["kind"]
    if kind == "step":
        state["graph"].replay()
        return state["out"]
    if kind == "module":
        return state["module"](state["x"])
    if kind == "quantize":
        if state["nested"]:
            return ta.functional.quantize_nf4_dq(state["w"], state["blocksize"], NESTED_BLOCKSIZE)
        return ta.quantize_nf4(state["w"], state["blocksize"])
    if kind == "dequantize":
        f = ta.functional.dequantize_nf4_dq if state["nested"] else ta.dequantize_nf4
        return f(state["qweight"], *state["stats"])
    f = ta.functional.matmul_nf4_dq if state["nested"] else ta.matmul_nf4
    return f(state["x"], state["qweight"], state["bias"], *state["stats"])


def _stored_bytes(n, k, blocksize, nested):
    """Codes and statistics of an NF4 weight."""
    blocks = -(-n * k // blocksize)
    return (n * k + 1) // 2 + (blocks + 4 * -(-blocks // NESTED_BLOCKSIZE) + 1024 if nested else 4 * blocks) + 64


def work(case):
    kind = case["kind"]
    if kind == "step":
        cfg, B = _cfg(case), case["batch"]
        d, hd, keys = cfg.d_model, cfg.head_dim, case["pos"] + 1
        weights = [((cfg.n_head + 2 * cfg.n_kv_head) * hd, d), (cfg.n_head * hd, d), (2 * cfg.d_ff, d), (d, cfg.d_ff)]
        cache = 2 * 2 * B * cfg.n_kv_head * keys * hd
        nbytes = cfg.n_layer * (sum(_stored_bytes(n, k, 64, False) for n, k in weights) + cache + 4 * d)
        flops = 2 * B * cfg.n_layer * (sum(n * k for n, k in weights) + 2 * cfg.n_head * hd * keys)
        return {"bytes": nbytes + _stored_bytes(cfg.vocab, d, 64, False) + 2 * B * (cfg.vocab + d), "flops": flops + 2 * B * cfg.vocab * d}
    n, k, size = case["n"], case["k"], SIZE[case["dtype"]]
    nbytes = _stored_bytes(n, k, case["blocksize"], case["nested"])
    if kind == "linear":
        m = case["m"]
        return {"bytes": nbytes + size * (m * k + m * n + (n if case["bias"] else 0)), "flops": 2 * m * n * k}
    return {"bytes": nbytes + size * n * k, "flops": 2 * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quantize", "dequantize"):
        return "exact"
    if kind == "linear":
        # Measured against the float64 product, over the listed and 24 drawn shapes: bf16 2.0e-3..2.7e-3 and at most 1.1e-2
        # (the rounding of the weights, or of the code book, and of the result); fp16 2.1e-4..2.9e-4 and at most 1.3e-3.
        return {"rel": 1e-2, "max": 4.4e-2} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 5.2e-3}
    # bf16 activations rounded in another order, layer after layer.  Measured between the three forms of the step (norms and
    # activation in the linears' epilogues, as kernels between them, as PyTorch operations): logits 0.0075..0.0115 times the
    # square root of the number of layers and at most 0.04..0.055 times it in one value.
    depth = math.sqrt(case["layers"])
    return {"rel": 0.03 * depth, "max": 0.16 * depth}
