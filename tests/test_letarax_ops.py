"""Each mechanism of the Letarax design alone: the package's torch operations (CPU) and HIP kernels (`gpu` marker)
against the one-function-per-mechanism plain model in `letarax_oracle`, on sizes that are not powers of two."""
import math

import numpy as np
import pytest
import torch

import letarax_oracle as O
from distributed_llm_inference_amd.ops import reference as R

gpu = pytest.mark.gpu


def close(a, b, tol):
    a, b = a.double().cpu(), b.double().cpu()
    err = float((a - b).abs().max() / (b.abs().max() + 1e-12))
    assert err < tol, f"relative error {err:.3g} over {tol}"


def rnd(*shape, seed=0, std=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std


# ---- torch operations (what the CPU executor is made of) -------------------------------------------------------------

def test_torch_offset_norm():
    x, w = rnd(5, 36), rnd(36, seed=1, std=0.3)
    close(R.rmsnorm(x, w, 1e-5, unit_offset=True), O.offset_rmsnorm(x, w, 1e-5), 1e-6)
    close(R.rmsnorm(x, w, 1e-5), O.plain_rmsnorm(x, w, 1e-5), 1e-6)


@pytest.mark.parametrize("window,ctx", [(1, 0), (5, 0), (5, 9), (40, 3), (100, 0)])
def test_torch_window_sink_attention(window, ctx):
    T, H, G, d, dv = 23, 4, 2, 12, 20
    q, k, v = rnd(T, H, d, seed=1), rnd(T, G, d, seed=2), rnd(T, G, dv, seed=3)
    ref = O.sink_window_attention(q, k, v, 0.3, window)
    got = R.attention(q[ctx:], k, v, ctx, 0.3, window=window, sink=True)
    close(got, ref[ctx:], 1e-5)


def test_torch_sink_takes_weight():
    """Scores far below zero: the sink holds the weight and the output vanishes (a plain softmax would return v)."""
    q, k, v = torch.full((1, 1, 4), 10.0), torch.full((1, 1, 4), -10.0), torch.ones(1, 1, 3)
    assert float(R.attention(q, k, v, 0, 1.0, window=4, sink=True).abs().max()) < 1e-6
    assert float(R.attention(q, k, v, 0, 1.0, window=4, sink=False).min()) > 0.99


@pytest.mark.parametrize("K", [1, 2, 4, 7])
def test_torch_short_conv_carried(K):
    x, taps = rnd(19, 10, seed=1), rnd(10, K, seed=2)
    ref = O.causal_short_conv(x, taps)
    prev = torch.zeros(K - 1, 10)
    outs = []
    for lo, hi in [(0, 1), (1, 3), (3, 4), (4, 12), (12, 19)]:
        y, prev = R.short_conv(x[lo:hi], prev, taps)
        outs.append(y)
    close(torch.cat(outs), ref, 1e-6)


def test_torch_delta_rule_carried():
    T, G, H, d, dv = 17, 2, 4, 7, 9
    q, k = O.unit_vectors(rnd(T, G, d, seed=1).double()).float(), O.unit_vectors(rnd(T, G, d, seed=2).double()).float()
    v, beta, decay = rnd(T, H, dv, seed=3), torch.sigmoid(rnd(T, H, seed=4)), torch.sigmoid(rnd(T, H, seed=5) + 2)
    S = torch.zeros(H, d, dv)
    outs = []
    for lo, hi in [(0, 5), (5, 6), (6, 17)]:
        o, S = R.gated_delta_rule(q[lo:hi], k[lo:hi], v[lo:hi], beta[lo:hi], decay[lo:hi], S)
        outs.append(o)
    got = torch.cat(outs)
    for h in range(H):
        ref = O.gated_delta_rule(q[:, h // 2].double(), k[:, h // 2].double(), v[:, h].double(), beta[:, h].double(), decay[:, h].double())
        close(got[:, h], ref, 1e-5)


# ---- HIP kernels -------------------------------------------------------------------------------------------------------

@pytest.fixture(scope="module")
def K():
    from distributed_llm_inference_amd import ops
    return ops.load()


def dev(t, dt=torch.float32):
    return t.to(device="cuda", dtype=dt).contiguous()


@gpu
@pytest.mark.parametrize("dt,tol", [(torch.float32, 2e-6), (torch.bfloat16, 1e-5)])
@pytest.mark.parametrize("M,N,Kd", [(1, 4, 36), (23, 48, 32), (70, 100, 52), (5, 322, 200), (129, 65, 7), (64, 64, 64), (300, 36, 136)])
def test_gemm_any(K, dt, tol, M, N, Kd):
    x, w, b = dev(rnd(M, Kd, seed=1), dt), dev(rnd(N, Kd, seed=2), dt), dev(rnd(N, seed=3))
    out = torch.zeros(M, N, device="cuda")
    K.gemm_any(out, x, w, b, 0)
    close(out, O.linear(x.cpu(), w.cpu(), b.cpu()), tol)
    if dt == torch.bfloat16:           # output in the operand type
        out16 = torch.zeros(M, N, device="cuda", dtype=dt)
        K.gemm_any(out16, x, w, None, 0)
        close(out16, O.linear(x.cpu(), w.cpu()), 1e-2)


TILED = [(1, 16, 512), (16, 34, 520), (15, 2050, 2056),               # the weight stream: its least K, K beyond whole chunks, a ragged last tile
         (17, 36, 512), (33, 4100, 64), (300, 2048, 1024),            # tiles of 32 and 48 rows, one and several K groups, one stage
         (64, 2048, 1088), (65, 64, 192), (301, 8192, 256), (200, 2056, 1024), (1000, 1030, 320),
         (512, 2048, 1024), (500, 2040, 1088), (2000, 4100, 128), (1030, 4096, 320), (2336, 224, 1024)]      # tiles of 64 rows; two groups on 32 x 32
GATED = [(9, 48, 1024), (40, 48, 1024), (70, 528, 320), (250, 2048, 1024), (250, 1040, 1088), (700, 4112, 192)]


def test_gemm_any_shapes_reach_every_kernel():
    from distributed_llm_inference_amd import ops
    form = ops.load(build_if_missing=True).gemm_any_form
    for f32 in (False, True):
        assert {form(M, N, K, 1, f32, 0) for M, N, K in TILED} == {1, 64642, 64641, 48642, 48641, 32642, 32641, 32324, 32322, 32321}
        assert {form(M, 2 * F, K, 1, f32, 1) for M, F, K in GATED} == {1, 64642, 64641, 32642, 32641}
        assert form(40, 64, 100, 1, f32, 0) == 0


@gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,Kd", TILED)
def test_gemm_any_tiles_and_weight_stream(K, dt, M, N, Kd):
    """A sum of K products in fp32, in any order: every entry within K roundings of the sum of the magnitudes (and, where the
    output is 16 bits wide, within one more of bf16)."""
    x, w, b = dev(rnd(M, Kd, seed=1), dt), dev(rnd(N, Kd, seed=2), dt), dev(rnd(N, seed=3))
    ref = (x.double() @ w.double().t() + b.double()).cpu()
    mag = (x.double().abs() @ w.double().abs().t() + b.double().abs()).cpu()
    wide = torch.full((M, N + 8), 7.0, device="cuda")
    K.gemm_any(wide[:, :N], x, w, b, 0)
    assert bool(((wide[:, :N].double().cpu() - ref).abs() <= (Kd + 1) * 2.0 ** -24 * mag).all())
    assert bool((wide[:, N:] == 7.0).all())
    if dt == torch.bfloat16:
        for pad in (0, 4):                                       # rows in whole 16-byte pieces, and not
            out = torch.full((M, N + pad), 7.0, device="cuda", dtype=dt)
            K.gemm_any(out[:, :N], x, w, b, 0)
            assert bool(((out[:, :N].double().cpu() - ref).abs() <= (Kd + 1) * 2.0 ** -24 * mag + 2.0 ** -8 * ref.abs()).all())
            assert bool((out[:, N:] == 7.0).all())


@gpu
@pytest.mark.parametrize("dt,tol", [(torch.float32, 5e-6), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("M,F,Kd", GATED)
def test_gemm_any_gated_tiles(K, dt, tol, M, F, Kd):
    test_gemm_any_gated(K, dt, tol, M, F, Kd)


@gpu
@pytest.mark.parametrize("dt,tol", [(torch.float32, 5e-6), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("M,F,Kd", [(9, 16, 36), (70, 48, 72), (3, 176, 200)])
def test_gemm_any_gated(K, dt, tol, M, F, Kd):
    from distributed_llm_inference_amd.ops.packing import interleave_gate_up
    x, wg, wu = dev(rnd(M, Kd, seed=1), dt), dev(rnd(F, Kd, seed=2, std=Kd ** -0.5), dt), dev(rnd(F, Kd, seed=3, std=Kd ** -0.5), dt)
    bg, bu = dev(rnd(F, seed=4)), dev(rnd(F, seed=5))
    w = interleave_gate_up(wg, wu).contiguous()
    b = interleave_gate_up(bg.unsqueeze(1), bu.unsqueeze(1)).reshape(-1).contiguous()
    out = torch.zeros(M, F, device="cuda", dtype=dt)
    K.gemm_any(out, x, w, b, 1)
    ref = O.gelu_tanh(O.linear(x.cpu(), wg.cpu(), bg.cpu())) * O.linear(x.cpu(), wu.cpu(), bu.cpu())
    close(out, ref, tol)


@gpu
@pytest.mark.parametrize("H", [37, 4, 4100, 16388])
def test_norm32_row_widths(K, H):
    """Rows of no whole 16-byte pieces, of one, of one unit more than the most threads, and beyond what registers hold."""
    test_norm32_forms(K, H)


@gpu
@pytest.mark.parametrize("H", [36, 200, 1000])
def test_norm32_forms(K, H):
    T, eps = 7, 1e-5
    x, y = rnd(T, H, seed=1, std=3.0), rnd(T, H, seed=2, std=0.7)
    wb, wn = rnd(H, seed=3, std=0.3), rnd(H, seed=4, std=0.3)
    xd, out = dev(x), torch.zeros(T, H, device="cuda")
    K.norm32(out, xd, None, None, dev(wn), None, eps, 1.0)
    close(out, O.offset_rmsnorm(x, wn, eps), 2e-6)
    K.norm32(out, xd, dev(y), dev(wb), dev(wn), None, eps, 1.0)            # post-norm, add, next pre-norm
    x2 = x.double() + O.offset_rmsnorm(y, wb, eps)
    close(xd, x2, 2e-6)
    close(out, O.offset_rmsnorm(x2, wn, eps), 2e-6)
    xd2 = dev(x)
    K.norm32(None, xd2, dev(y), dev(wb), None, None, eps, 1.0)
    close(xd2, x2, 2e-6)
    rows = torch.tensor([5, 0, 5], dtype=torch.int32, device="cuda")
    out16 = torch.zeros(3, H, device="cuda", dtype=torch.bfloat16)
    K.norm32(out16, dev(x), None, None, dev(wn), rows, eps, 0.0)               # gathered rows, plain weight, bf16 out
    close(out16, O.plain_rmsnorm(x[[5, 0, 5]], wn, eps), 1e-2)


def paged(K, q, k, v, scale, window, sink, dt, chunks, blocks_perm=None):
    """Runs kv_store + window_attention over one sequence given in `chunks`, blocks handed out in a scrambled order."""
    T, H, d = q.shape
    G, dv = k.shape[1], v.shape[2]
    nb = (T + 31) // 32
    order = list(range(nb + 3))[::-1] if blocks_perm is None else blocks_perm
    table = torch.full((3, nb), -1, dtype=torch.int32)
    table[1, :nb] = torch.tensor(order[:nb], dtype=torch.int32)
    table = table.cuda()
    kc = torch.zeros(nb + 3, G, 32, d, device="cuda", dtype=dt)
    vc = torch.zeros(nb + 3, G, 32, dv, device="cuda", dtype=dt)
    outs, lo = [], 0
    for n in chunks:
        qkv = dev(torch.cat([q[lo:lo + n].reshape(n, -1), k[lo:lo + n].reshape(n, -1), v[lo:lo + n].reshape(n, -1)], dim=1))
        pos = torch.arange(lo, lo + n, dtype=torch.int32, device="cuda")
        seq = torch.ones(n, dtype=torch.int32, device="cuda")
        K.kv_store(qkv, None, None, 0, kc, vc, pos, seq, table, G, d, dv, H * d)
        out = torch.zeros(n, H * dv, device="cuda", dtype=dt)
        K.window_attention(out, qkv, kc, vc, pos, seq, table, H, G, d, dv, scale, window, sink)
        outs.append(out.float().cpu().reshape(n, H, dv))
        lo += n
    return torch.cat(outs)


@gpu
@pytest.mark.parametrize("dt,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("H,G,d,dv,window", [(4, 2, 12, 20, 5), (3, 3, 64, 64, 96), (2, 1, 7, 130, 1), (8, 2, 128, 32, 70), (1, 1, 36, 36, 1000)])
def test_window_attention_kernel(K, dt, tol, H, G, d, dv, window):
    T = 150
    q, k, v = rnd(T, H, d, seed=1), rnd(T, G, d, seed=2), rnd(T, G, dv, seed=3)
    if dt == torch.bfloat16:
        k, v = k.bfloat16().float(), v.bfloat16().float()
    ref = O.sink_window_attention(q, k, v, d ** -0.5, window)
    close(paged(K, q, k, v, d ** -0.5, window, True, dt, [150]), ref, tol)
    close(paged(K, q, k, v, d ** -0.5, window, True, dt, [31, 2, 1, 1, 64, 33, 18]), ref, tol)


@gpu
def test_window_attention_edge_and_sink(K):
    """One key with a large score right at the window's far edge (seen) and one step beyond (not seen), 200 tokens
    back across block edges; and scores so low that only the sink has weight."""
    T, d, window = 260, 8, 200
    for back, seen in [(window - 1, True), (window, False)]:
        q, k, v = torch.zeros(T, 1, d), torch.zeros(T, 1, d), rnd(T, 1, 4, seed=1)
        ask, beacon = 255, 255 - back
        q[ask, 0, 0], k[beacon, 0, 0] = 6.0, 6.0
        out = paged(K, q, k, v, 1.0, window, True, torch.float32, [250, 3, 1, 1, 1, 4])
        close(out, O.sink_window_attention(q, k, v, 1.0, window), 1e-5)
        near_beacon = float((out[ask, 0] - v[beacon, 0]).abs().max()) < 1e-3
        assert near_beacon == seen
    q, k, v = torch.full((40, 1, d), 3.0), torch.full((40, 1, d), -3.0), torch.ones(40, 1, 4)
    assert float(paged(K, q, k, v, 1.0, 16, True, torch.float32, [40]).abs().max()) < 1e-6
    assert float(paged(K, q, k, v, 1.0, 16, False, torch.float32, [40]).min()) > 0.999


@gpu
def test_value_mixing_in_store(K):
    T, G, d, dv, H = 5, 2, 8, 12, 2
    qkv1, qkv2 = dev(rnd(T, H * d + G * d + G * dv, seed=1)), dev(rnd(T, H * d + G * d + G * dv, seed=2))
    table = torch.tensor([[0]], dtype=torch.int32, device="cuda")
    pos, seq = torch.arange(T, dtype=torch.int32, device="cuda"), torch.zeros(T, dtype=torch.int32, device="cuda")
    kc, vc = torch.zeros(1, G, 32, d, device="cuda"), torch.zeros(1, G, 32, dv, device="cuda")
    vf, lam = torch.zeros(T * G * dv, device="cuda"), torch.tensor([0.3], device="cuda")
    K.kv_store(qkv1, vf, None, 1, kc, vc, pos, seq, table, G, d, dv, H * d)
    v1 = qkv1[:, H * d + G * d:].cpu()
    close(vc[0, :, :T].permute(1, 0, 2).reshape(T, -1), v1, 1e-7)
    K.kv_store(qkv2, vf, lam, 2, kc, vc, pos, seq, table, G, d, dv, H * d)
    close(vc[0, :, :T].permute(1, 0, 2).reshape(T, -1), O.mix_values(qkv2[:, H * d + G * d:].cpu(), v1, float(lam)), 1e-6)
    close(kc[0, :, :T].permute(1, 0, 2).reshape(T, -1), qkv2[:, H * d:H * d + G * d].cpu(), 1e-7)


def ragged(lens, ctxs, slots):
    qs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    t = lambda a: torch.tensor(np.asarray(a, dtype=np.int32), device="cuda")
    return t(qs), t(ctxs), t(slots)


@gpu
@pytest.mark.parametrize("Kt", [1, 2, 4, 9])
def test_short_conv_kernel(K, Kt):
    C, T = 70, 45
    x, taps = rnd(T, C + 6, seed=1), rnd(C, Kt, seed=2)
    ref = O.silu(O.causal_short_conv(x[:, :C], taps))
    carry = torch.full((3, max(Kt - 1, 1), C), 7.0, device="cuda")          # stale contents: a first step must not read them
    outs, lo = [], 0
    for n in [1, 1, 2, 20, 3, 18]:
        z = dev(x[lo:lo + n])
        y = torch.zeros(n, C, device="cuda")
        qs, ctx, sl = ragged([n], [lo], [2])
        K.short_conv(y, z, carry, dev(taps), qs, ctx, sl, n)
        outs.append(y.cpu())
        lo += n
    close(torch.cat(outs), ref, 1e-5)


@gpu
@pytest.mark.parametrize("C", [4, 72, 1028, 2052])
def test_short_conv_of_four_taps_in_pieces(K, C):
    """Channels in whole pieces, portions on either side of the 8 tokens that a thread takes, beside a sequence that goes on behind them."""
    T = 52
    x, x2, taps = rnd(T, C + 4, seed=1), rnd(40, C + 4, seed=3), rnd(C, 4, seed=2)
    ref, ref2 = (O.silu(O.causal_short_conv(v[:, :C], taps)) for v in (x, x2))
    carry = torch.full((3, 3, C), 7.0, device="cuda")
    outs, outs2, lo, lo2 = [], [], 0, 0
    for n, n2 in [(1, 2), (2, 1), (7, 17), (8, 1), (9, 8), (17, 9), (8, 2)]:
        z = dev(torch.cat([x[lo:lo + n], x2[lo2:lo2 + n2]]))
        y = torch.full((n + n2, C), 9.0, device="cuda")
        qs, ctx, sl = ragged([n, n2], [lo, lo2], [2, 0])
        K.short_conv(y, z, carry, dev(taps), qs, ctx, sl, max(n, n2))
        outs.append(y[:n].cpu())
        outs2.append(y[n:].cpu())
        lo, lo2 = lo + n, lo2 + n2
    close(torch.cat(outs), ref, 1e-5)
    close(torch.cat(outs2), ref2, 1e-5)


@gpu
@pytest.mark.parametrize("G,H,d,dv", [(1, 1, 7, 9), (2, 4, 32, 32), (2, 6, 16, 48), (1, 2, 160, 72), (1, 1, 128, 128), (3, 3, 64, 20)])
def test_delta_rule_kernel(K, G, H, d, dv):
    T, C = 40, 2 * G * d + H * dv
    y = torch.cat([O.unit_vectors(rnd(T, G, d, seed=1).double()).float().reshape(T, -1) * d ** -0.5,
                   O.unit_vectors(rnd(T, G, d, seed=2).double()).float().reshape(T, -1), rnd(T, H * dv, seed=3)], dim=1)
    z = rnd(T, 5 + 2 * H, seed=4)                                            # [pad | beta logits | decay logits]
    A_log, dtb = rnd(H, seed=5, std=0.5), rnd(H, seed=6, std=0.5)
    state = torch.full((4, H, d, dv), 3.0, device="cuda")                    # stale
    outs, lo = [], 0
    for n in [1, 2, 17, 1, 19]:
        o = torch.zeros(n, H * dv, device="cuda")
        qs, ctx, sl = ragged([n], [lo], [3])
        K.delta_rule(o, dev(y[lo:lo + n]), dev(z[lo:lo + n]), state, dev(A_log), dev(dtb), qs, ctx, sl, G, H, d, dv, 5, 5 + H, n)
        outs.append(o.cpu())
        lo += n
    got = torch.cat(outs).reshape(T, H, dv)
    beta = torch.sigmoid(z[:, 5:5 + H].double())
    a = z[:, 5 + H:].double() + dtb.double()
    decay = torch.exp(-torch.exp(A_log.double()) * torch.log1p(torch.exp(a)))
    yq, yk, yv = y[:, :G * d].reshape(T, G, d), y[:, G * d:2 * G * d].reshape(T, G, d), y[:, 2 * G * d:].reshape(T, H, dv)
    for h in range(H):
        g = h // (H // G)
        ref = O.gated_delta_rule(yq[:, g].double(), yk[:, g].double(), yv[:, h].double(), beta[:, h], decay[:, h])
        close(got[:, h], ref, 2e-5)


@gpu
@pytest.mark.parametrize("G,H,d,dv", [(1, 2, 64, 16), (2, 4, 128, 48), (1, 1, 128, 128), (3, 3, 64, 64)])
def test_delta_rule_in_chunks(K, G, H, d, dv):
    """Prompt portions that run in chunks of 32 on the matrix cores, beside sequences with a token or two: whole chunks, remainders,
    states carried from step to step and from and to the token-by-token kernel, stale slots, a decay that forgets within a chunk."""
    C = 2 * G * d + H * dv
    steps = [[33, 1, 0, 64], [2, 96, 40, 31], [1, 1, 1, 1], [70, 32, 5, 3]]
    A_log, dtb = rnd(H, seed=5, std=0.5), rnd(H, seed=6, std=0.5)
    A_log[0] = 2.5                                                           # (log decays down to some -20 a token)
    lens = [sum(s[b] for s in steps) for b in range(4)]
    ys, zs = [], []
    for b, T in enumerate(lens):
        unit = lambda s: O.unit_vectors(rnd(T, G, d, seed=s + b).double()).float().reshape(T, -1)
        ys.append(torch.cat([unit(10) * d ** -0.5, unit(20), rnd(T, H * dv, seed=30 + b)], dim=1))
        zs.append(rnd(T, 5 + 2 * H, seed=40 + b))
    state = torch.full((7, H, d, dv), 3.0, device="cuda")                    # stale
    slots, at, got = [3, 0, 6, 2], [0] * 4, [[] for _ in range(4)]
    for ns in steps:
        o = torch.full((sum(ns), H * dv), 9.0, device="cuda")
        take = lambda src: dev(torch.cat([src[b][at[b]:at[b] + ns[b]] for b in range(4)]))
        qs, ctx, sl = ragged(ns, at, slots)
        K.delta_rule(o, take(ys), take(zs), state, dev(A_log), dev(dtb), qs, ctx, sl, G, H, d, dv, 5, 5 + H, max(ns))
        for b, part in enumerate(o.cpu().split(ns)):
            got[b].append(part)
            at[b] += ns[b]
    for b in range(4):
        y, z, T = ys[b], zs[b], lens[b]
        beta = torch.sigmoid(z[:, 5:5 + H].double())
        decay = torch.exp(-torch.exp(A_log.double()) * torch.log1p(torch.exp(z[:, 5 + H:].double() + dtb.double())))
        yq, yk, yv = y[:, :G * d].reshape(T, G, d), y[:, G * d:2 * G * d].reshape(T, G, d), y[:, 2 * G * d:].reshape(T, H, dv)
        for h in range(H):
            g = h // (H // G)
            ref = O.gated_delta_rule(yq[:, g].double(), yk[:, g].double(), yv[:, h].double(), beta[:, h], decay[:, h])
            close(torch.cat(got[b]).reshape(T, H, dv)[:, h], ref, 2e-5)
    assert bool((state[[1, 4, 5]] == 3.0).all())


def _delta_run(K, lens, G, H, d, dv, max_q, seed, ctx=0, edit=None, tail=()):
    """The kernel's read-outs and states for sequences of these lengths and the plain recurrence in 64 bits for the same inputs
    (`edit` changes them first), all on the GPU. States start from random ones where ctx > 0."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *shape: torch.randn(*shape, device="cuda", generator=g)
    B, T = len(lens), sum(lens)
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1).reshape(T, -1)
    y = torch.cat([unit(r(T, G, d)) * d ** -0.5, unit(r(T, G, d)), r(T, H * dv)], dim=1)
    z, A_log, dtb, S0 = r(T, 2 * H), r(H) * 0.5, r(H) * 0.5, r(B, H, d, dv) * 0.3
    if edit:
        edit(y, z, A_log, dtb)
    qs, cx, sl = ragged(lens, [ctx] * B, list(range(B)))
    state, o = S0.clone(), torch.full((T, H * dv), 9.0, device="cuda")
    K.delta_rule(o, y, z, state, A_log, dtb, qs, cx, sl, G, H, d, dv, 0, H, max_q, *tail)
    beta, decay = torch.sigmoid(z[:, :H].double()), torch.exp(-torch.exp(A_log.double()) * torch.nn.functional.softplus(z[:, H:].double() + dtb.double()))
    heads = lambda x: x.reshape(T, G, d).double().repeat_interleave(H // G, 1)
    q, k, v = heads(y[:, :G * d]), heads(y[:, G * d:2 * G * d]), y[:, 2 * G * d:].reshape(T, H, dv).double()
    ref, S_ref, t = torch.zeros(T, H, dv, device="cuda", dtype=torch.float64), [], 0
    for b, n in enumerate(lens):
        S = S0[b].double() if ctx else torch.zeros(H, d, dv, device="cuda", dtype=torch.float64)
        for t in range(t, t + n):
            S = S * decay[t][:, None, None]
            S = S + k[t][:, :, None] * (beta[t][:, None] * (v[t] - (k[t][:, :, None] * S).sum(1)))[:, None]
            ref[t] = (q[t][:, :, None] * S).sum(1)
        t += n > 0
        S_ref.append(S)
    return o.reshape(T, H, dv), state, ref, torch.stack(S_ref)


def rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@gpu
@pytest.mark.parametrize("n,G,H,d,dv", [(64, 8, 32, 128, 128), (300, 2, 8, 128, 64), (700, 4, 8, 64, 64)])
def test_delta_rule_in_chunks_is_no_less_exact(K, n, G, H, d, dv):
    """Against 64 bits, portions in chunks have no more error than the same portions token by token (which `max_q` 2 asks for), in the
    read-outs and in the states they leave. Measured: 0.73 to 0.77 and 0.96 to 0.98 of it (with one 32-bit chain throughout: 1.04 to
    1.12 and 1.09 to 1.13)."""
    def error(max_q):
        assert (K.scan_route(2, 1, H, d, dv, n, max_q) == 2) == (max_q == n)
        runs = [_delta_run(K, [n], G, H, d, dv, max_q, seed) for seed in range(8)]
        return [rel(torch.cat([r[i] for r in runs]), torch.cat([r[i + 2] for r in runs])) for i in (0, 1)]
    chunks, tokens = error(n), error(2)
    assert chunks[0] <= 0.9 * tokens[0] and chunks[1] <= tokens[1], (chunks, tokens)


@gpu
@pytest.mark.parametrize("log_a", [5.0, 60.0, 100.0])
def test_delta_rule_in_chunks_forgets_all(K, log_a):
    """Decays of exactly zero between tokens that keep e^-1 of the state (for the largest `log_a`: all of them, exp(A_log) being infinite)."""
    def edit(y, z, A_log, dtb):
        A_log[0], dtb[0] = log_a, 0.0
        z[:, 2] = -min(log_a, 60.0)
        z[5::7, 2] = 30.0
    assert K.scan_route(2, 2, 2, 64, 32, 164, 100) == 2
    o, state, ref, S = _delta_run(K, [100, 64], 1, 2, 64, 32, 100, 8, ctx=4, edit=edit)
    close(o, ref, 2e-5)
    close(state, S, 2e-5)


@gpu
@pytest.mark.parametrize("what", ["q", "k", "v", "beta", "decay"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_delta_rule_in_chunks_keeps_a_bad_value_to_later_tokens(K, what, value):
    """A value that is no number or infinite in token 41 of the first sequence (head 1, or the key head of heads 0 and 1; value column 5)
    leaves the read-outs and states finite where they are token by token: earlier tokens, other heads, sequences and columns."""
    G, H, d, dv = 2, 4, 64, 32
    assert K.scan_route(2, 2, H, d, dv, 170, 100) == 2
    def edit(y, z, A_log, dtb):
        if what in "qkv":
            y[41, {"q": 3, "k": G * d + 3, "v": 2 * G * d + dv + 5}[what]] = value
        else:
            z[41, {"beta": 1, "decay": H + 1}[what]] = value
    chunks, tokens = (_delta_run(K, [100, 70], G, H, d, dv, q, 9, ctx=4, edit=edit) for q in (100, 2))
    for a, b in zip(chunks[:2], tokens[:2]):
        assert torch.equal(a.isfinite(), b.isfinite()) and bool(a.isfinite().any())
        close(a[a.isfinite()], b[a.isfinite()], 2e-5)
    assert bool(chunks[0][:41].isfinite().all()) and bool(chunks[0][100:].isfinite().all())


@gpu
def test_delta_rule_in_chunks_longer_than_announced(K):
    """A portion longer than `max_q` says runs all of its tokens, in chunks as token by token."""
    for lens, max_q in [([200, 3, 64], 64), ([1, 110, 300], 100)]:
        assert K.scan_route(2, 3, 2, 64, 32, sum(lens), max_q) == 2
        o, state, ref, S = _delta_run(K, lens, 1, 2, 64, 32, max_q, 7, ctx=4)
        close(o, ref, 2e-5)
        close(state, S, 2e-5)


# (us token by token, in chunks, apart, of 32 or 16 heads of 128 x 128 unless said otherwise)
@pytest.mark.parametrize("rule,lens,lead,H,d,dv,route", [
    (2, [64], 0, 32, 128, 128, 2), (2, [48], 0, 32, 128, 128, 0), (2, [47], 0, 32, 128, 128, 0),          # 27.5 / 24.8, 22.6 / 24.7
    (2, [64] * 4, 0, 32, 128, 128, 0), (2, [512] * 4, 0, 32, 128, 128, 2), (2, [96] * 5, 0, 32, 128, 128, 2),   # 41 / 55, ..., 106 / 81
    (2, [48] * 64, 0, 32, 128, 128, 0), (2, [128] * 16, 0, 32, 64, 64, 0), (2, [2048], 0, 32, 128, 128, 2),     # 516 / 665, 73 / 88, 780 / 242
    (2, [1] * 64 + [64], 64, 32, 128, 128, 3), (2, [1] * 64 + [64], 0, 32, 128, 128, 0), (2, [1] * 64 + [1024], 64, 32, 128, 128, 3),
    (2, [1] * 128 + [256] * 4, 128, 32, 128, 128, 3), (2, [1] * 64 + [20], 64, 32, 128, 128, 0), (2, [1] * 16 + [300], 16, 4, 64, 64, 2),
    (1, [48], 0, 16, 128, 128, 2), (1, [128] * 16, 0, 16, 128, 128, 0), (1, [48] * 4, 0, 16, 128, 128, 0),      # 20 / 15, 120 / 127, 26 / 33
    (1, [1] * 128 + [256], 128, 16, 128, 128, 3), (1, [1] * 64 + [1024], 64, 8, 64, 64, 2), (1, [300], 0, 16, 128, 528, 0),
    (0, [300], 0, 16, 128, 128, 0), (2, [300], 0, 16, 96, 96, 0), (2, [300], 0, 16, 128, 40, 0), (2, [48] * 65536, 0, 1, 128, 128, 0)])
def test_a_step_takes_the_route_that_measured_faster(K, rule, lens, lead, H, d, dv, route):
    assert K.scan_route(rule, len(lens), H, d, dv, sum(lens), max(lens), lead) == route


@gpu
@pytest.mark.parametrize("lens,lead,G,H,d,dv", [([1] * 40 + [200, 3, 33], 40, 4, 16, 128, 128), ([1] * 20 + [1000], 20, 2, 4, 64, 64),
                                                ([1] * 70 + [128], 70, 8, 32, 128, 128), ([1] * 64 + [130], 64, 8, 16, 64, 128)])
def test_delta_rule_mixed_step(K, lens, lead, G, H, d, dv):
    """Single tokens in front of prompt portions (announced or not), against 64 bits: 3e-7 of the 2-norm, where 1.1e-7 is the most that
    any route was measured at."""
    for n in (lead, 0):
        o, state, ref, S = _delta_run(K, lens, G, H, d, dv, max(lens), 3, ctx=5, tail=(n,))
        assert rel(o, ref) < 3e-7 and rel(state, S) < 3e-7
    assert K.scan_route(2, len(lens), H, d, dv, sum(lens), max(lens), lead) >= 2


@gpu
def test_unit_heads_and_gated_headnorm(K):
    T, heads, d = 6, 5, 13
    x = rnd(T, heads * d + 3, seed=1)
    xd = dev(x)
    K.unit_heads(xd[:, :heads * d], heads, d, 2, 0.25, 1e-6)
    ref = O.unit_vectors(x[:, :heads * d].reshape(T, heads, d).double())
    ref[:, :2] *= 0.25
    close(xd[:, :heads * d], ref.reshape(T, -1), 1e-6)
    close(xd[:, heads * d:], x[:, heads * d:], 1e-7)
    dv = 9
    o, gate, w = rnd(T, heads * dv, seed=2), rnd(T, heads * dv + 4, seed=3), rnd(dv, seed=4)
    out = torch.zeros(T, heads * dv, device="cuda")
    K.gated_headnorm(out, dev(o), dev(gate)[:, 2:2 + heads * dv], dev(w), heads, dv, 1e-5)
    ref = O.plain_rmsnorm(o.reshape(T, heads, dv), w, 1e-5) * O.silu(gate[:, 2:2 + heads * dv].double()).reshape(T, heads, dv)
    close(out, ref.reshape(T, -1), 1e-5)


def fragment_paged(K, q, k, v, scale, window, sink, chunks):
    """The MFMA attention path: bf16 fused q|k|v rows, fragment-ordered cache written without rotation, windowed kernel."""
    T, H, D = q.shape
    G = k.shape[1]
    nb = (T + 31) // 32
    table = torch.full((2, nb), -1, dtype=torch.int32)
    table[1] = torch.arange(nb - 1, -1, -1, dtype=torch.int32) + 2
    table = table.cuda()
    kv = torch.zeros(nb + 2, G, 2, 32 * D, device="cuda", dtype=torch.bfloat16)
    zero = torch.zeros(1, D // 2, device="cuda")
    outs, lo = [], 0
    for n in chunks:
        qkv = dev(torch.cat([q[lo:lo + n].reshape(n, -1), k[lo:lo + n].reshape(n, -1), v[lo:lo + n].reshape(n, -1)], dim=1), torch.bfloat16)
        pos = torch.arange(lo, lo + n, dtype=torch.int32, device="cuda")
        seq = torch.ones(n, dtype=torch.int32, device="cuda")
        K.rope_kvwrite(qkv, None, 1, None, kv, zero, zero, pos, seq, table, H, G, D, False)
        out = torch.zeros(n, H * D, device="cuda", dtype=torch.bfloat16)
        qs, ctx, sl = ragged([n], [lo], [1])
        K.paged_attention_window(out, qkv, kv, qs, ctx, table, sl, None, n, H, G, D, scale, 1, window, sink)
        outs.append(out.float().cpu().reshape(n, H, D))
        lo += n
    return torch.cat(outs)


@gpu
@pytest.mark.parametrize("H,G,D,window", [(4, 2, 64, 5), (4, 4, 64, 96), (8, 1, 128, 70), (3, 1, 128, 1), (2, 1, 64, 1000), (4, 2, 128, 33)])
def test_windowed_mfma_attention(K, H, G, D, window):
    T = 330
    bf = lambda t: t.bfloat16().float()
    q, k, v = bf(rnd(T, H, D, seed=1)), bf(rnd(T, G, D, seed=2)), bf(rnd(T, G, D, seed=3))
    ref = O.sink_window_attention(q, k, v, D ** -0.5, window)
    close(fragment_paged(K, q, k, v, D ** -0.5, window, True, [330]), ref, 2e-2)                       # prefill-shaped kernel
    close(fragment_paged(K, q, k, v, D ** -0.5, window, True, [200, 2, 1, 1, 1, 64, 33, 28]), ref, 2e-2)   # portions and single tokens


@gpu
def test_windowed_mfma_attention_edge_and_sink(K):
    T, D, window = 300, 64, 200
    for back, seen in [(window - 1, True), (window, False)]:
        for chunks in ([300], [290, 3, 1, 1, 1, 4]):
            q, k, v = torch.zeros(T, 1, D), torch.zeros(T, 1, D), rnd(T, 1, D, seed=1).bfloat16().float()
            ask, beacon = 294, 294 - back
            q[ask, 0, 0], k[beacon, 0, 0] = 6.0, 6.0
            out = fragment_paged(K, q, k, v, 1.0, window, True, chunks)
            close(out, O.sink_window_attention(q, k, v, 1.0, window), 2e-2)
            assert (float((out[ask, 0] - v[beacon, 0]).abs().max()) < 5e-2) == seen
    q, k, v = torch.full((40, 1, D), 1.0), torch.full((40, 1, D), -1.0), torch.ones(40, 1, D)
    assert float(fragment_paged(K, q, k, v, 1.0, 16, True, [40]).abs().max()) < 1e-6
    assert float(fragment_paged(K, q, k, v, 1.0, 16, False, [40]).min()) > 0.99


@gpu
def test_value_mix_kernel(K):
    T, cols, off = 5, 24, 40
    a, b = rnd(T, off + cols, seed=1).bfloat16(), rnd(T, off + cols, seed=2).bfloat16()
    vf, lam = torch.zeros(T * cols, device="cuda"), torch.tensor([0.3], device="cuda")
    ad, bd = a.cuda(), b.cuda()
    K.value_mix(ad, vf, None, 1, off, cols)
    close(vf.view(T, cols), a[:, off:].float(), 1e-7)
    K.value_mix(bd, vf, lam, 2, off, cols)
    close(bd[:, off:], O.mix_values(b[:, off:].float(), a[:, off:].float(), float(lam)), 1e-2)
    close(bd[:, :off], b[:, :off].float(), 1e-7)
