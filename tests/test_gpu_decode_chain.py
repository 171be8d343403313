"""The decode step as one kernel (nf4hip_decode_chain): ABI checks without a GPU; on the GPU against the PyTorch step of the same
quantized model, and bit for bit against itself with fewer workgroups, in a replayed graph and beside other steps."""

import ctypes
import importlib
import math
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda:0"


@pytest.fixture(scope="module")
def glue():
    return importlib.import_module("lightning-thunder_amd.glue")


@pytest.fixture(scope="module")
def D():
    return importlib.import_module("lightning-thunder_amd.decode")


def test_symbols_and_argument_errors(glue):
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", "nf4hip_decode_chain.h")).read(), flags=re.S)
    declared = sorted(set(re.findall(r"\b(nf4hip_decode_\w+)\s*\(", text)))
    assert declared == sorted(glue.CHAIN_SYMBOLS)
    lib = glue.load()
    need = lib.nf4hip_decode_chain_workspace_bytes
    assert need(1, 32, 4096, 32, 8, 14336, 128256, 640) > 0 and need(16, 1, 2048, 16, 4, 4096, 32000, 4096) > 0
    # 17 sequences, head size 64, eight query heads per kv head, K > 4096, d_ff no multiple of 256 or beyond 16384, vocab no multiple of 8
    for shape in [(17, 2, 4096, 32, 8, 14336, 32000, 640), (1, 2, 2048, 32, 8, 8192, 32000, 640), (1, 2, 4096, 32, 4, 14336, 32000, 640),
                  (1, 2, 8192, 64, 16, 28672, 32000, 640), (1, 2, 4096, 32, 8, 14400, 32000, 640), (1, 2, 4096, 32, 8, 16640, 32000, 640),
                  (1, 2, 4096, 32, 8, 14336, 32001, 640), (1, 0, 4096, 32, 8, 14336, 32000, 640)]:
        assert need(*shape) == 0, shape
    # the longest caches whose scores fit LDS: 2880 keys in each of eight, four and two ranges
    for batch, longest in ((1, 23033), (4, 23033), (8, 11517), (16, 5759)):
        assert need(batch, 1, 4096, 32, 8, 14336, 8000, longest) > 0 and need(batch, 1, 4096, 32, 8, 14336, 8000, longest + 1) == 0, batch
    A = 4096  # non-null, 16-byte aligned fake device address: validation never dereferences
    err = lambda: lib.nf4hip_decode_last_error().decode()

    def call(layers=(A,) * 14, head=(A,) * 3, x=A, batch=1, ws_bytes=1 << 40):
        return lib.nf4hip_decode_chain(x, (ctypes.c_void_p * 14)(*layers), (ctypes.c_void_p * 3)(*head), A, 1e-5, A, A, A, A, A, batch, 1, 4096, 32, 8,
                                       14336, 32000, 640, 0, A, A, ws_bytes, None)

    for first, more in ((-1, 0), (1, -1), (1, 1 << 17)):
        assert lib.nf4hip_decode_chain_joined(A, (ctypes.c_void_p * 14)(*(A,) * 14), (ctypes.c_void_p * 3)(A, A, A), A, 1e-5, A, A, A, A, A, 1, 1, 4096, 32, 8,
                                              14336, 32000, 640, 0, first, more, A, A, 1 << 40, None) == -1 and "number of workgroups" in err()
    assert call(x=None) == -1 and "null" in err()
    assert call(batch=17) == -1 and "not served" in err()
    assert call(ws_bytes=4096) == -1 and "workspace" in err()
    assert call(x=A + 2) == -1 and "aligned" in err()
    assert call(layers=(A,) * 13 + (None,)) == -1 and "null" in err()
    assert call(head=(A, A + 8, A)) == -1 and "aligned" in err()


def _model(D, ta, batch, layers, d, d_ff, vocab, max_seq, seed=1):
    cfg = D.LlamaConfig(n_layer=layers, d_model=d, n_head=d // 128, n_kv_head=d // 512, d_ff=d_ff, vocab=vocab, max_seq=max_seq,
                        fused_projections=True, hip_glue=True, gate_up_interleaved=True)
    model = ta.jit(D.build_llama(cfg, device=DEV, seed=seed), transforms=[ta.BitsAndBytesLinearQuant4bit()])
    g = torch.Generator(device=DEV).manual_seed(seed)
    kc, vc = D.new_caches(cfg, batch, DEV)
    kc.normal_(generator=g)
    vc.normal_(generator=g)
    tok = torch.randint(0, vocab, (batch, 1), generator=g, device=DEV)
    return cfg, model, kc, vc, tok


@pytest.fixture
def chain_calls(glue, monkeypatch):
    """Counts the calls of glue.decode_chain, caps their workgroups and makes some late; every step that the kernel serves is one, also where launches
    are faster."""
    calls = {"n": 0, "workgroups": 0, "late": {}}
    real = glue.decode_chain

    def counted(*args, **kw):
        calls["n"] += 1
        return real(*args, max_workgroups=calls["workgroups"], **calls["late"], **kw)

    monkeypatch.setattr(glue, "decode_chain", counted)
    monkeypatch.setattr(glue, "decode_chain_pays", lambda *a: True)
    return calls


# batch, layers, d_model, d_ff, vocab, max_seq, position: 1, 2 and more rows of x (two ways to operands), one to four K ranges of the down
# projection (the last of them shorter), parts of K that are not whole, rows that are no whole tile, no cached key, one key, ragged
# ranges of keys
SHAPES = [(1, 2, 4096, 14336, 8000, 128, 0), (1, 2, 1024, 2304, 1000, 640, 333), (7, 2, 1024, 4096, 1000, 640, 17), (2, 2, 1024, 2304, 1000, 640, 1), (3, 2, 2048, 5632, 8008, 640, 17), (5, 1, 4096, 16384, 1000, 640, 333),
          (9, 2, 2048, 4096, 1000, 2048, 2047), (16, 2, 4096, 8448, 8000, 640, 639), (16, 1, 4096, 12288, 1000, 300, 16)]


@pytest.mark.gpu
@pytest.mark.parametrize("batch,layers,d,d_ff,vocab,max_seq,p", SHAPES)
def test_chain_against_the_pytorch_step(D, ta, chain_calls, batch, layers, d, d_ff, vocab, max_seq, p):
    print(f"chain {batch=} {layers=} {d=} {d_ff=} {vocab=} {max_seq=} {p=}", flush=True)
    cfg, model, kc, vc, tok = _model(D, ta, batch, layers, d, d_ff, vocab, max_seq)
    pos = torch.full((1,), p, device=DEV, dtype=torch.long)
    kr, vr = kc.clone(), vc.clone()
    with torch.no_grad():
        out = model(tok, pos, kc, vc)
        assert chain_calls["n"] == 1
        cfg.hip_glue = False
        ref = model(tok, pos, kr, vr)
    rel = lambda a, b: ((a.float() - b.float()).norm() / b.float().norm()).item()
    # bf16 activations rounded in another order, layer after layer: 0.012 * sqrt(layers) measured between the forms of the step
    bound = 0.03 * math.sqrt(layers)
    assert rel(out, ref) < bound
    for c, r in ((kc, kr), (vc, vr)):
        assert rel(c[:, :, :, p], r[:, :, :, p]) < bound
        c[:, :, :, p] = 0
        r[:, :, :, p] = 0
        assert torch.equal(c, r)  # no other row is written


@pytest.mark.gpu
@pytest.mark.parametrize("batch,p", [(1, 0), (1, 512), (5, 3), (8, 576), (9, 100), (16, 639)])
def test_same_bits_as_launch_by_launch_at_8b_shapes(D, ta, chain_calls, monkeypatch, batch, p):
    """Every sum is taken in the order of the kernels that the step of one launch per linear runs there."""
    print(f"chain bits {batch=} {p=}", flush=True)
    cfg, model, kc, vc, tok = _model(D, ta, batch, 2, 4096, 14336, 32000, 640)
    pos = torch.full((1,), p, device=DEV, dtype=torch.long)
    kr, vr = kc.clone(), vc.clone()
    with torch.no_grad():
        out = model(tok, pos, kc, vc)
        assert chain_calls["n"] == 1
        monkeypatch.setattr(D.Llama, "_decode_step_chain", lambda *a: None)
        ref = model(tok, pos, kr, vr)
    assert chain_calls["n"] == 1
    assert torch.equal(out, ref) and torch.equal(kc, kr) and torch.equal(vc, vr)


# ranges of keys that reach into the second part of the scores' LDS (from 2048 keys on): just so, in the middle, the longest that there are;
# whole rounds of 192 keys and 160 values and one more  (vocabulary: one where the launches' head takes its sums in the same order)
LONG = [(1, 23033, 16384), (1, 23033, 16392), (1, 23033, 20011), (1, 23033, 23032), (5, 13817, 13816), (8, 11517, 11516), (16, 5759, 384), (16, 5759, 386),
        (16, 5759, 4097), (16, 5759, 5758)]


@pytest.mark.gpu
@pytest.mark.parametrize("batch,max_seq,p", LONG)
def test_long_contexts_same_bits_as_launch_by_launch(D, ta, chain_calls, monkeypatch, batch, max_seq, p):
    print(f"chain long {batch=} {max_seq=} {p=}", flush=True)
    cfg, model, kc, vc, tok = _model(D, ta, batch, 1, 4096, 14336, 32000, max_seq)
    pos = torch.full((1,), p, device=DEV, dtype=torch.long)
    kr, vr = kc.clone(), vc.clone()
    step = D.Llama._decode_step_chain
    seen = []
    for q in (p // 2, p - 1):  # (a key that counts, early and late)
        for k, v in ((kc, vc), (kr, vr)):
            k[:, -1:, :, q], v[:, -1:, :, q] = 3.0, 50.0
        with torch.no_grad():
            monkeypatch.setattr(D.Llama, "_decode_step_chain", step)
            out = model(tok, pos, kc, vc)
            monkeypatch.setattr(D.Llama, "_decode_step_chain", lambda *a: None)
            ref = model(tok, pos, kr, vr)
        assert torch.equal(out, ref) and torch.equal(kc, kr) and torch.equal(vc, vr)
        seen.append(out)
    assert chain_calls["n"] == 2 and not torch.equal(seen[0][-1], seen[1][-1])


@pytest.mark.gpu
@pytest.mark.parametrize("batch,layers,d,d_ff,p", [(1, 2, 4096, 14336, 300), (1, 2, 2048, 5632, 40), (5, 2, 2048, 5632, 300), (3, 2, 4096, 14336, 300), (16, 1, 4096, 8192, 37), (2, 35, 1024, 2048, 77)])
def test_fewer_workgroups_same_bits(D, ta, chain_calls, batch, layers, d, d_ff, p):
    """Tasks are dealt by the shape alone; (35 layers are two launches)."""
    print(f"chain workgroups {batch=} {layers=} {d=} {d_ff=}", flush=True)
    cfg, model, kc, vc, tok = _model(D, ta, batch, layers, d, d_ff, 1000, 640)
    pos = torch.full((1,), p, device=DEV, dtype=torch.long)
    ref = None
    for workgroups in (0, 255, 37, 3, 1):
        chain_calls["workgroups"] = workgroups
        k, v = kc.clone(), vc.clone()
        with torch.no_grad():
            got = (model(tok, pos, k, v), k, v)
        if ref is None:
            ref = got
            assert not ref[0].isnan().any()
        assert all(torch.equal(a, b) for a, b in zip(got, ref)), workgroups
    assert chain_calls["n"] == 5


CTL_BYTES, CTL_MEMBERS = 1024, 32  # decode_chain.h: per launch, the arrivals and then how many shared each phase


@pytest.mark.gpu
@pytest.mark.parametrize("batch,layers,d,d_ff", [(1, 3, 4096, 14336), (1, 2, 1024, 2304), (6, 2, 2048, 5632), (2, 2, 4096, 14336), (16, 2, 4096, 8448), (3, 35, 1024, 2048)])
def test_late_workgroups_join_same_bits(D, ta, glue, chain_calls, monkeypatch, batch, layers, d, d_ff):
    """Workgroups that are late take part from the next phase or layer on; those that never get a turn leave.  (35 layers are two launches.)"""
    print(f"chain late {batch=} {layers=} {d=} {d_ff=}", flush=True)
    cfg, model, kc, vc, tok = _model(D, ta, batch, layers, d, d_ff, 1000, 640)
    pos = torch.full((1,), 300, device=DEV, dtype=torch.long)
    step = lambda k, v: model(tok, pos, k, v)
    with torch.no_grad():
        ref = [kc.clone(), vc.clone()]
        ref.insert(0, step(*ref))
        real, scratch = torch.empty, []

        def empty(*args, **kw):
            t = real(*args, **kw)
            if kw.get("dtype") is torch.uint8:
                scratch.append(t)
            return t

        # first, more: one, then one more per phase; few, never more; all but one late; one late; odd steps, past all of them; most, never more
        for first, more in ((1, 1), (3, 0), (1, 1 << 16), (255, 1), (37, 50), (100, 0)):
            chain_calls["late"] = {"first_members": first, "more_members": more}
            got = [kc.clone(), vc.clone()]
            scratch.clear()
            with monkeypatch.context() as m:
                m.setattr(torch, "empty", empty)
                got.insert(0, step(*got))
            assert all(torch.equal(a, b) for a, b in zip(got, ref)), (first, more)
            ws = max(scratch, key=lambda t: t.numel())
            cus = torch.cuda.get_device_properties(0).multi_processor_count
            for launch in range(-(-layers // 32)):
                ctl = ws[launch * CTL_BYTES:(launch + 1) * CTL_BYTES].view(torch.int32).tolist()
                phases = 4 * min(32, layers - 32 * launch) + (1 if 32 * (launch + 1) >= layers else 0)
                members = ctl[CTL_MEMBERS:CTL_MEMBERS + phases]
                # what was settled: phase by phase for less than a quarter, then layer by layer, until all are there (the device is idle:
                # all have arrived when the second phase is settled)
                want, i = [0] * phases, 0
                while i < phases:
                    m = min(cus, first + i * more)
                    stop = i if m == cus or 4 * m < cus else min(i | 3, phases - 1)
                    want[i:stop + 1] = [m] * (stop + 1 - i)
                    i = phases if m == cus else stop + 1
                assert ctl[0] == cus and members == want, (first, more, ctl[0], members)


@pytest.mark.gpu
def test_chain_graph_replays_and_streams(D, ta, chain_calls):
    """Replays with new tokens and positions equal the eager step, with eager steps between them; steps of three models at a time on
    as many streams give what they give alone."""
    cfg, model, kc, vc, tok = _model(D, ta, 8, 2, 2048, 5632, 1000, 640)
    pos = torch.full((1,), 100, device=DEV, dtype=torch.long)
    ke, ve = kc.clone(), vc.clone()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.no_grad(), torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):  # (no call on this stream before: the step brings its own scratch)
            out = model(tok, pos, kc, vc)
    torch.cuda.synchronize()
    for i in range(12):
        t = torch.randint(0, 1000, (8, 1), device=DEV)
        tok.copy_(t)
        pos.fill_(100 + 7 * i)
        graph.replay()
        with torch.no_grad():
            eager = model(t, torch.full((1,), 100 + 7 * i, device=DEV, dtype=torch.long), ke, ve)
        assert torch.equal(eager, out) and torch.equal(ke, kc) and torch.equal(ve, vc), i

    models = [_model(D, ta, b, 2, 2048, 5632, 1000, 640, seed=b) for b in (1, 4, 9)]
    streams = [torch.cuda.Stream() for _ in models]
    pos.fill_(200)
    with torch.no_grad():
        alone = [m(t, pos, k.clone(), v.clone()) for _, m, k, v, t in models]
        torch.cuda.synchronize()
        for _ in range(5):
            got = []
            for s, (_, m, k, v, t) in zip(streams, models):
                with torch.cuda.stream(s):
                    got.append(m(t, pos, k.clone(), v.clone()))
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, alone))


@pytest.mark.gpu
def test_chain_position_outside_the_cache_and_other_routes(D, ta, chain_calls):
    cfg, model, kc, vc, tok = _model(D, ta, 2, 1, 1024, 2048, 1000, 64)
    k, v = kc.clone(), vc.clone()
    with torch.no_grad():
        for p in (64, -1):
            model(tok, torch.full((1,), p, device=DEV, dtype=torch.long), k, v)
    torch.cuda.synchronize()
    assert torch.equal(k, kc) and torch.equal(v, vc) and chain_calls["n"] == 2
    # caches in another layout, seventeen sequences: the step of several launches, as before
    pos = torch.full((1,), 5, device=DEV, dtype=torch.long)
    apart = torch.zeros((1, 2, 2, 64, 256), device=DEV, dtype=torch.bfloat16)
    with torch.no_grad(), pytest.raises(ValueError):
        model(tok, pos, apart[..., :128], apart[..., 128:])
    kb, vb = D.new_caches(cfg, 17, DEV)
    with torch.no_grad():
        assert model(tok[:1].expand(17, 1).contiguous(), pos, kb, vb).shape == (17, 1000)
    assert chain_calls["n"] == 2


@pytest.mark.gpu
def test_chain_infinities_and_nan(D, ta, chain_calls):
    """A value of +inf in one sequence's cache stays in that sequence, and a NaN there makes its logits NaN, without a wait that lasts."""
    cfg, model, kc, vc, tok = _model(D, ta, 4, 2, 1024, 2048, 1000, 64)
    pos = torch.full((1,), 40, device=DEV, dtype=torch.long)
    with torch.no_grad():
        ref = model(tok, pos, kc.clone(), vc.clone())
        for bad in (float("inf"), float("nan")):
            v = vc.clone()
            v[0, 1, 0, 3, 5] = bad
            out = model(tok, pos, kc.clone(), v)
            assert out[1].isnan().all()  # (an infinite residual has an infinite rms)
            assert torch.equal(out[[0, 2, 3]], ref[[0, 2, 3]])


def test_caches_of_one_tensor_per_layer_are_left_to_the_launches(D):
    cfg = D.LlamaConfig(n_layer=2, d_model=1024, n_head=8, n_kv_head=2, d_ff=256, vocab=64, max_seq=16, fused_projections=True, hip_glue=True,
                        gate_up_interleaved=True)
    model = D.build_llama(cfg, device="cpu")
    kc, vc = D.new_caches(cfg, 1, "cpu")
    for k, v in ((list(kc), list(vc)), (tuple(kc), vc), (kc, list(vc))):
        assert model._decode_step_chain(torch.zeros(1, 1024, dtype=torch.bfloat16), torch.zeros(1, dtype=torch.long), k, v) is None


@pytest.mark.gpu
def test_caches_of_one_tensor_per_layer(D, ta, chain_calls, monkeypatch):
    cfg, model, kc, vc, tok = _model(D, ta, 5, 2, 1024, 2048, 1000, 64)
    pos = torch.full((1,), 30, device=DEV, dtype=torch.long)
    kl, vl = [c.clone() for c in kc], [c.clone() for c in vc]
    with torch.no_grad():
        got = model(tok, pos, kl, vl)
        assert chain_calls["n"] == 0
        monkeypatch.setattr(D.Llama, "_decode_step_chain", lambda *a: None)
        ref = model(tok, pos, kc, vc)
    assert torch.equal(got, ref) and torch.equal(torch.stack(kl), kc) and torch.equal(torch.stack(vl), vc)


def test_a_model_that_is_refused_is_asked_about_once(D, glue, monkeypatch):
    """Shapes first: a model that the kernel does not serve pays one query per eager step, not a look at every weight."""
    cfg = D.LlamaConfig(n_layer=2, d_model=1024, n_head=8, n_kv_head=8, d_ff=256, vocab=64, max_seq=16, fused_projections=True, hip_glue=True,
                        gate_up_interleaved=True)
    model = D.build_llama(cfg, device="cpu")
    kc, vc = D.new_caches(cfg, 1, "cpu")
    asked = []
    monkeypatch.setattr(glue, "decode_chain_served", lambda *a: asked.append(a[1:]))
    monkeypatch.setattr(D, "_planned_nf4", lambda lin: pytest.fail("a weight was looked at"))
    assert model._decode_step_chain(torch.zeros(1, 1024, dtype=torch.bfloat16), torch.zeros(1, dtype=torch.long), kc, vc) is None
    assert asked == [(1, 2, 1024, 8, 8, 256, 64, 16)]


def test_rule_of_use(D, glue, monkeypatch):
    """Where both steps were timed, the rule names the faster one (cases within 2 % left out)."""
    # batch, layers, d_model, max_seq, vocabulary (32000)
    faster = [(b, l, 4096, 640) for b in (1, 3, 8, 16) for l in (2, 8, 32)] + [(b, 8, d, 640) for b in (1, 3, 8, 16) for d in (2048, 3072)]
    faster += [(8, 2, 2048, 640), (16, 3, 2048, 640), (1, 32, 4096, 20480), (4, 32, 4096, 11000), (8, 32, 4096, 5696), (16, 32, 4096, 4096)]
    slower = [(b, l, 1024, 640) for b in (1, 3, 8) for l in (8, 32)] + [(b, 1, 512, 64) for b in (1, 8)] + [(3, 8, 1536, 640)]
    slower += [(1, 1, 2048, 640), (3, 2, 2048, 640), (3, 3, 2048, 640), (8, 1, 2048, 640), (16, 1, 4096, 640), (1, 4, 2048, 20480), (4, 4, 2048, 20480)]
    faster += [(2, 6, 2048, 192), (2, 7, 1536, 192, 59152), (2, 6, 2048, 3968, 37328), (2, 3, 2048, 3136, 62520), (2, 4, 2048, 1856, 115400), (9, 5, 1536, 2624), (11, 7, 1536, 1664)]
    faster += [(1, 2, 2048, 768, 96376), (2, 2, 2048, 448, 99304)]
    slower += [(4, 2, 2048, 2816), (3, 2, 2048, 256), (3, 3, 2048, 1472, 45712), (13, 3, 1024, 5568), (1, 2, 2048, 640, 44248)]
    pays = lambda b, l, d, s, vocab=32000: glue.decode_chain_pays(b, l, d, d // 128, s, vocab)
    assert all(pays(*c) for c in faster) and not any(pays(*c) for c in slower)

    cfg = D.LlamaConfig(n_layer=1, d_model=512, n_head=4, n_kv_head=1, d_ff=256, vocab=64, max_seq=16, fused_projections=True, hip_glue=True,
                        gate_up_interleaved=True)
    model = D.build_llama(cfg, device="cpu")
    monkeypatch.setattr(glue, "decode_chain_served", lambda *a: True)
    monkeypatch.setattr(D, "_planned_nf4", lambda lin: pytest.fail("a weight was looked at"))
    assert model._decode_step_chain(torch.zeros(1, 512, dtype=torch.bfloat16), torch.zeros(1, dtype=torch.long), *D.new_caches(cfg, 1, "cpu")) is None
