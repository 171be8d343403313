"""Decode attention with four query heads of a kv group per workgroup (head size 128, 128 such workgroups and more): numbers of
cached keys around what a request of the workgroup (64 keys, 16 rows) and a round of them (256) cover, one and several splits, two
workgroups per kv head, empty splits; against a float64 softmax."""

import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
glue = importlib.import_module("lightning-thunder_amd.glue")


@pytest.mark.parametrize("B,H,Hkv,max_seq,p", [
    (2, 32, 8, 64, 0), (4, 32, 8, 64, 1), (2, 32, 8, 300, 257), (8, 32, 8, 140, 127), (8, 32, 8, 140, 129), (32, 32, 8, 40, 31), (32, 32, 8, 40, 33),
    (32, 32, 8, 520, 256), (33, 32, 8, 520, 257), (64, 16, 2, 300, 299), (8, 16, 4, 4096, 4095), (16, 32, 4, 2100, 2050),
])
def test_grouped_attention(B, H, Hkv, max_seq, p):
    print(f"grouped attention B={B} H={H}/{Hkv} max_seq={max_seq} p={p}", flush=True)
    hd = 128
    g = torch.Generator(device=DEV).manual_seed(B + p)
    rnd = lambda *shape: torch.empty(*shape, device=DEV).normal_(0, 1, generator=g).to(torch.bfloat16)
    kc, vc, qkv = rnd(B, Hkv, max_seq, hd), rnd(B, Hkv, max_seq, hd), rnd(B, (H + 2 * Hkv) * hd)
    # no rotation (it is tested where its rounding is compared): q and the new key are then known exactly
    cos, sin = torch.ones(max_seq, hd, device=DEV), torch.zeros(max_seq, hd, device=DEV)
    pos = torch.tensor([p], device=DEV)
    heads = qkv.view(B, H + 2 * Hkv, hd)
    kref, vref = kc.clone(), vc.clone()
    kref[:, :, p], vref[:, :, p] = heads[:, H:H + Hkv], heads[:, H + Hkv:]
    out = glue.attention_decode(qkv, pos, cos, sin, kc, vc, H, Hkv)
    assert torch.equal(kc, kref) and torch.equal(vc, vref)  # row p written, nothing else
    assert torch.equal(glue.attention_decode(qkv, pos, cos, sin, kc, vc, H, Hkv), out)  # counters back at zero, one order of sums
    K, V = (t[:, :, : p + 1].double().repeat_interleave(H // Hkv, 1) for t in (kref, vref))
    w = torch.softmax((K @ heads[:, :H].double().unsqueeze(-1)).squeeze(-1) / hd**0.5, -1)
    ref = (w.unsqueeze(-2) @ V).squeeze(-2).reshape(B, H * hd)
    # result in bf16 (2^-8); a weight is exp of a score of magnitude up to ~10 that 130 fp32 roundings of terms adding up to ~8
    # and the scaling by log2(e) leave within 2^-16: relative error of a weight, twice that with their sum, of sums over |v| <= 6
    bound = 2.0**-8 * ref.abs() + 2 * 2.0**-16 * 6
    assert ((out.double().reshape(B, -1) - ref).abs() <= bound).all()


@pytest.mark.parametrize("p", [0, 70, 300, 513])
def test_grouped_attention_gives_the_bits_of_a_workgroup_per_head(p):
    """Four sequences (128 workgroups: grouped) against each of them alone (a workgroup per head); both split the keys in 8."""
    print(f"grouped attention, same bits, p={p}", flush=True)
    B, H, Hkv, hd, max_seq = 4, 32, 8, 128, 640
    g = torch.Generator(device=DEV).manual_seed(p)
    rnd = lambda *shape: torch.empty(*shape, device=DEV).normal_(0, 1, generator=g)
    kc, vc, qkv = (rnd(*shape).to(torch.bfloat16) for shape in ((B, Hkv, max_seq, hd), (B, Hkv, max_seq, hd), (B, (H + 2 * Hkv) * hd)))
    angle = rnd(max_seq, hd // 2).repeat(1, 2)
    cos, sin, pos = angle.cos(), angle.sin(), torch.tensor([p], device=DEV)
    alone = [glue.attention_decode(qkv[b:b + 1].clone(), pos, cos, sin, kc[b:b + 1].clone(), vc[b:b + 1].clone(), H, Hkv) for b in range(B)]
    assert torch.equal(glue.attention_decode(qkv, pos, cos, sin, kc, vc, H, Hkv), torch.cat(alone))
