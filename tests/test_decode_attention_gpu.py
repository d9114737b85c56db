"""Decode attention with a window, a sink, learned extras, a cap or an entry gate: steps of more items than CUs."""
import pytest
import torch

from distributed_llm_inference_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("form", ["window", "extras", "bias", "cap", "entry gate"])
@pytest.mark.parametrize("Hq,Hkv,D", [(16, 8, 64), (32, 8, 128)])
def test_many_items_have_the_bits_of_few(form, Hq, Hkv, D):
    """33 and 32 sequences of 8 key heads: above and at the 256 items up to which a CU holds one workgroup. A sequence's result is its own: the bits
    of steps of three sequences, whose numbers other tests hold against 64 bits. Lengths around blocks and beyond the table of biases."""
    K = ops.load()
    g = torch.Generator(device=DEV).manual_seed(D)
    B = 33
    ctx = [(0, 1, 31, 32, 33, 63, 127, 200, 511)[i % 9] + 3 * (i // 9) for i in range(B)]
    nb = [c // 32 + 1 for c in ctx]
    table = torch.full((B, max(nb)), -1, dtype=torch.int32)
    at = 0
    for b in range(B):
        table[b, :nb[b]] = torch.arange(at, at + nb[b])
        at += nb[b]
    kv = torch.randn(at, Hkv, 2, 32 * D, device=DEV, generator=g).bfloat16()
    qkv = torch.randn(B, (Hq + 2 * Hkv) * D, device=DEV, generator=g).bfloat16()
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    temp, bias, sink, gate, egate = r(Hq).exp(), r(97, Hq), r(Hq), r(B, Hq), r(B, Hq * D).bfloat16()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    table, cl = table.to(DEV), i32(ctx)

    def run(a, b):
        out = torch.full((b - a, Hq * D), float("nan"), device=DEV, dtype=torch.bfloat16)
        args = (out, qkv[a:b], kv, i32(list(range(b - a + 1))), cl[a:b], table, i32(list(range(a, b))))
        if form == "window":
            K.paged_attention_window(*args, None, 1, Hq, Hkv, D, D ** -0.5, 1, 100, True)
        elif form in ("extras", "bias"):
            K.paged_attention_biased(*args, 1, Hq, Hkv, D, D ** -0.5, temp, bias if form == "bias" else None, sink, gate[a:b])
        else:
            K.paged_attention_capped(*args, 1, Hq, Hkv, D, D ** -0.5, 100, 5.0 if form == "cap" else 0.0, egate[a:b] if form != "cap" else None)
        return out
    whole, parts = run(0, B), torch.cat([run(a, a + 3) for a in range(0, B, 3)])
    assert bool(torch.isfinite(whole.float()).all()) and torch.equal(whole, parts) and torch.equal(run(0, 32), parts[:32])
