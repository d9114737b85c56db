"""Heads on shared key rows (fp32, matrix cores): rounds that begin inside a block, tiles whose heads begin inside a value head."""
import pytest
import torch

from distributed_llm_inference_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Gk,per,G,d,dv,window,keep,chunk", [
    (1, 16, 4, 512, 128, 0, 0, 0),         # four value heads a tile: eight units, a wave each
    (1, 16, 4, 512, 128, 37, 3, 0),        # a window that begins at any key, and kept first keys
    (1, 16, 2, 576, 256, 0, 0, 100),       # chunks that begin inside a block
    (2, 20, 5, 64, 64, 0, 0, 0),           # tiles of 16 and 4 heads, value heads of 8 across tiles
    (1, 12, 3, 64, 196, 50, 0, 0),         # value rows beyond a tile of 64
    (2, 32, 2, 80, 128, 0, 0, 0),          # two tiles of one value head
    (1, 24, 4, 48, 320, 0, 0, 0),          # tiles that do not end with a value head: more than eight units
])
def test_heads_on_shared_key_rows(Gk, per, G, d, dv, window, keep, chunk):
    K, dev = ops.load(), "cuda"
    g = torch.Generator(device=dev).manual_seed(5)
    H, lens = Gk * per, [1, 31, 130, 263]
    blocks = [(n + 31) // 32 for n in lens]
    table = torch.full((len(lens), max(blocks)), -1, dtype=torch.int32)
    order = torch.randperm(sum(blocks), generator=torch.Generator().manual_seed(6)).int()
    for b, n in enumerate(blocks):
        table[b, :n] = order[sum(blocks[:b]):][:n]
    # ...of each sequence its last tokens
    pos = torch.cat([torch.arange(max(0, n - 6), n) for n in lens]).int()
    seq = torch.cat([torch.full((min(6, n),), b) for b, n in enumerate(lens)]).int()
    T = pos.numel()
    kc = torch.randn(sum(blocks), Gk, 32, d, device=dev, generator=g)
    vc = torch.randn(sum(blocks), G, 32, dv, device=dev, generator=g)
    q = torch.randn(T, H * d, device=dev, generator=g) * (2 / d ** 0.5)
    sink = torch.randn(H, device=dev, generator=g)
    out = torch.full((T, H * dv), 7.0, device=dev)
    K.multi_attention(out, q, d, kc, vc, 0, pos.to(dev), seq.to(dev), table.to(dev), H, d, dv, 1, 1.0, window, keep, 0.0, 0.0, 1.0, 1e-5,
                      None, chunk, sink)
    for t in range(T):
        p = int(pos[t])
        lo = max(0, p - window + 1) if window else 0
        lo = max(lo, p // chunk * chunk) if chunk else lo
        js = torch.cat([torch.arange(min(keep, lo)), torch.arange(lo, p + 1)])
        blk, row = table[int(seq[t])][js // 32].long().to(dev), (js % 32).to(dev)
        for h in range(H):
            s = kc[blk, h // per, row].double() @ q[t, h * d:(h + 1) * d].double()
            w = torch.softmax(torch.cat([s, sink[h:h + 1].double()]), 0)[:-1]
            want = w @ vc[blk, h // (H // G), row].double()
            got = out[t, h * dv:(h + 1) * dv].double()
            # a score's error is at most d / 4 + 2 roundings of its products' sum |q k| <= 2 |k| (about 2 sqrt(d)), a weight's about that;
            # the sums over keys add their own 2^-24 a term: 600 roundings bound the rows here, none is near it
            assert (got - want).abs().max() <= 600 * 2.0 ** -24 * (w @ vc[blk, h // (H // G), row].double().abs()).max(), (t, h)
