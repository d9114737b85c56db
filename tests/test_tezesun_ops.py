"""Every mechanism of the Tezesun design alone: the package's torch operations (CPU) and its HIP kernels (`gpu` marker)
against the plain float64 functions of `tezesun_oracle`, on small inputs made here."""
import math

import pytest
import torch

import tezesun_oracle as O

F64 = torch.float64


def rnd(*shape, seed=0, std=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed), dtype=F64) * std


def close(got, ref, tol=2e-5):
    ref = ref.to(F64)
    err = (got.detach().cpu().to(F64) - ref).abs().max().item() / max(1.0, ref.abs().max().item())
    assert err < tol, err


# ---- torch operations (the CPU executor's) ---------------------------------------------------------------------------
def test_xielu_and_token_shift():
    from distributed_llm_inference_amd.ops import reference as R
    z = rnd(7, 33, seed=1, std=3.0)
    for p, q in [(0.3, -0.7), (-2.0, 1.5), (0.0, 0.0)]:
        close(R.xielu(z.float(), torch.tensor(p), torch.tensor(q)), O.xielu(z, torch.tensor(p, dtype=F64), torch.tensor(q, dtype=F64)))
    h, mu = rnd(9, 20, seed=2), torch.rand(20, dtype=F64)
    ref = O.token_shift(h, mu)
    a, last = R.token_shift(h[:4].float(), torch.zeros(20), mu.float())           # in two portions: the last row is carried
    b, _ = R.token_shift(h[4:].float(), last, mu.float())
    close(torch.cat([a, b]), ref)


@pytest.mark.parametrize("interleaved", [True, False])
@pytest.mark.parametrize("dims,D", [(8, 8), (4, 10), (2, 2)])
def test_partial_rotation_and_scaled_frequencies(interleaved, dims, D):
    from distributed_llm_inference_amd.models.rope import rope_table
    from distributed_llm_inference_amd.models.spec import RopeScaling
    from distributed_llm_inference_amd.ops import reference as R
    # (the last one: a band that lies beyond the rotated entries, which the clamps turn inside out: no frequency is rescaled)
    for sc in (None, {"factor": 4.0, "original": 64, "fast": 16.0, "slow": 2.0}, {"factor": 6.0, "original": 1000, "fast": 24.0, "slow": 1.5},
               {"factor": 3.0, "original": 10 ** 7, "fast": 16.0, "slow": 2.0}):
        rot = {"dims": dims, "base": 100.0, **({"scaling": sc} if sc else {})}
        rs = RopeScaling(factor=sc["factor"], rope_type="yarn", beta_fast=sc["fast"], beta_slow=sc["slow"],
                         original_max_position_embeddings=sc["original"], ramp_floor=True) if sc else None
        cos, sin = rope_table(dims, 100.0, rs, 50)
        rc, rsn = O.rope_angles(rot, 50)
        close(cos, rc, 1e-6)
        close(sin, rsn, 1e-6)
        x = rnd(50, 3, D, seed=3)
        got = R.rope_partial(x.float(), cos, sin, torch.arange(50), interleaved)
        close(got, O.rotate(x, rc, rsn, interleaved))
        # positions are the tokens' own, not their place in the step
        got = R.rope_partial(x[:5].float(), cos, sin, torch.tensor([40, 41, 42, 43, 44]), interleaved)
        close(got, O.rotate(x[:5], rc[40:45], rsn[40:45], interleaved))


def _rglru_weights(W, nb, taps, H, seed):
    bw = W // nb
    return {"y": rnd(W, H, seed=seed, std=H ** -0.5), "y.b": rnd(W, seed=seed + 1, std=0.3), "x": rnd(W, H, seed=seed + 2, std=H ** -0.5),
            "x.b": rnd(W, seed=seed + 3, std=0.3), "conv": rnd(W, taps, seed=seed + 4, std=0.6), "conv.b": rnd(W, seed=seed + 5, std=0.2),
            "ra": rnd(nb, bw, bw, seed=seed + 6, std=bw ** -0.5), "ra.b": rnd(nb, bw, seed=seed + 7, std=0.5),
            "ri": rnd(nb, bw, bw, seed=seed + 8, std=bw ** -0.5), "ri.b": rnd(nb, bw, seed=seed + 9, std=0.5),
            "lam": rnd(W, seed=seed + 10, std=1.5) - 2.0, "o": torch.eye(W, dtype=F64)}


@pytest.mark.parametrize("W,nb,taps", [(24, 3, 3), (16, 1, 1), (10, 10, 5)])
def test_recurrent_unit_in_portions(W, nb, taps):
    """conv -> block gates -> recurrence over several calls with the carried inputs and state, against the whole sequence."""
    from distributed_llm_inference_amd.ops import reference as R
    H, T = 12, 40
    w, h = _rglru_weights(W, nb, taps, H, 20), rnd(T, H, seed=5)
    ref = O.rglru(h, w)
    carry, S, outs, t0 = torch.zeros(taps - 1, W), torch.zeros(W), [], 0
    for n in (1, 2, 17, 1, 19):
        hp = h[t0:t0 + n].float()
        y = R.gelu_tanh(hp @ w["y"].float().T + w["y.b"].float())
        u, carry = R.short_conv(hp @ w["x"].float().T + w["x.b"].float(), carry, w["conv"].float())
        u = u + w["conv.b"].float()
        gr, gi = torch.sigmoid(R.block_linear(u, w["ra"], w["ra.b"])), torch.sigmoid(R.block_linear(u, w["ri"], w["ri.b"]))
        st, S = R.rglru_scan(u, gr, gi, w["lam"], S)
        outs.append(st * y)
        t0 += n
    close(torch.cat(outs), ref, 5e-5)


def test_attention_mask_with_kept_tokens_and_cap():
    from distributed_llm_inference_amd.ops import reference as R
    T, d, dv = 30, 6, 5
    q, k, v = rnd(T, 2, d, seed=6), rnd(T, 1, d, seed=7), rnd(T, 1, dv, seed=8)
    for window, keep, cap in [(4, 3, 2.0), (1, 0, 0.0), (7, 9, 0.5), (0, 0, 1.0)]:
        ok = O.visible(T, window, keep)
        ref = []
        for hh in range(2):
            s = (q[:, hh] @ k[:, 0].T) * 0.7
            if cap > 0:
                s = cap * torch.tanh(s / cap)
            ref.append(torch.softmax(s.masked_fill(~ok, float("-inf")), -1) @ v[:, 0])
        got = R.attention(q[10:].float(), k.float(), v.float(), 10, 0.7, window=window, keep_first=keep, softcap=cap)
        close(got, torch.stack(ref, 1)[10:])


# ---- HIP kernels ------------------------------------------------------------------------------------------------------
def _K():
    from distributed_llm_inference_amd import ops
    return ops.load()


def _meta(seqs, dev):
    """seqs: [(slot, q_len, ctx)] -> tok_pos, tok_seq, q_start, ctx, slots (int32 on the device)."""
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    pos = [c + i for _, n, c in seqs for i in range(n)]
    seq = [s for s, n, _ in seqs for _ in range(n)]
    qs = [0]
    for _, n, _ in seqs:
        qs.append(qs[-1] + n)
    return i32(pos), i32(seq), i32(qs), i32([c for _, _, c in seqs]), i32([s for s, _, _ in seqs])


@pytest.mark.gpu
def test_norm_residual_shift_and_carried_rows_hip():
    """par_norm + token_shift over two steps of two sequences that sit in slots used before: positions 0 start from zeros,
    portions go on from the slot's carried row."""
    K, dev, H = _K(), "cuda", 40
    x = rnd(12, H, seed=1)                      # sequence a: rows 0..6 (7 tokens), sequence b: rows 7..11 (5 tokens)
    w, mu, ls1, ls2 = 1.0 + rnd(H, seed=2, std=0.1), torch.rand(H, dtype=F64), rnd(H, seed=3), rnd(H, seed=4)
    ya, yb = rnd(12, H, seed=5), rnd(12, H, seed=6)
    w2 = 1.0 + rnd(H, seed=7, std=0.1)
    f = lambda t: t.float().to(dev).contiguous()
    carry = torch.full((5, H), 7.0, device=dev)      # stale rows
    got_s, got_n2 = {}, {}
    for step, (ra, rb) in enumerate([((0, 3), (7, 9)), ((3, 7), (9, 12))]):
        rows = list(range(*ra)) + list(range(*rb))
        tok_pos, tok_seq, *_ = _meta([(3, ra[1] - ra[0], ra[0]), (1, rb[1] - rb[0], rb[0] - 7)], dev)
        h = f(x[rows])
        n32, xn, xs = torch.zeros(len(rows), H, device=dev), torch.zeros(len(rows), H, device=dev), torch.zeros(len(rows), H, device=dev)
        K.par_norm(xn, n32, h, None, None, None, None, f(w), None, tok_seq, 1e-5)
        K.token_shift(xs, n32, carry, f(mu), tok_pos, tok_seq)
        K.par_norm(xn, n32, h, f(ya[rows]), f(yb[rows]), f(ls1), f(ls2), f(w2), carry, tok_seq, 1e-5)
        for i, r in enumerate(rows):
            got_s[r], got_n2[r] = xs[i].cpu(), xn[i].cpu()
    for lo, hi in ((0, 7), (7, 12)):
        n = O.rms(x[lo:hi], 1e-5) * w
        ref_s = O.token_shift(n, mu)
        ref_n2 = O.rms(x[lo:hi] + ls1 * ya[lo:hi] + ls2 * yb[lo:hi], 1e-5) * w2
        close(torch.stack([got_s[r] for r in range(lo, hi)]), ref_s)
        close(torch.stack([got_n2[r] for r in range(lo, hi)]), ref_n2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,d,dv,maps,window,keep,cap,dims,inter", [
    (4, 2, 16, 24, 2, 40, 5, 10.0, 8, True), (2, 1, 8, 8, 1, 0, 0, 0.0, 8, False), (3, 3, 12, 70, 2, 3, 50, 0.0, 4, True),
    (2, 2, 72, 130, 1, 33, 0, 3.0, 0, False), (6, 1, 10, 16, 2, 64, 1, 25.0, 10, True)])
def test_rotation_cache_write_and_attention_hip(dtype, H, G, d, dv, maps, window, keep, cap, dims, inter):
    """rope_cache_write + multi_attention over a paged cache whose blocks are in no order: a prompt portion, then another
    that crosses block edges, then single tokens, against whole-sequence attention; two maps combined, normed and gated."""
    K, dev = _K(), "cuda"
    T, eps, lam, post, scale = 150, 1e-5, 0.37, 0.6, 0.3
    q, k = rnd(T, H * maps, d, seed=1), rnd(T, G * maps, d, seed=2)
    v, gate = rnd(T, G, dv, seed=3), rnd(T, H * dv, seed=4)
    if dtype == torch.bfloat16:             # inputs that the cache holds exactly
        k, v = k.bfloat16().to(F64), v.bfloat16().to(F64)
    rot = {"dims": dims, "base": 50.0}
    cos, sin = O.rope_angles(rot, T) if dims else (None, None)
    qr, kr = (O.rotate(q, cos, sin, inter), O.rotate(k, cos, sin, inter)) if dims else (q, k)
    ok = O.visible(T, window, keep)
    heads = []
    for hh in range(H):
        g, per = hh // (H // G), []
        for mp in range(maps):
            s = (qr[:, maps * hh + mp] @ kr[:, maps * g + mp].T) * scale
            if cap > 0:
                s = cap * torch.tanh(s / cap)
            per.append(torch.softmax(s.masked_fill(~ok, float("-inf")), -1) @ v[:, g])
        heads.append(O.rms(per[0] - lam * per[1], eps) * post if maps == 2 else per[0])
    ref = torch.cat(heads, -1) * (torch.sigmoid(gate) if maps == 2 else 1.0)
    nblk = 9
    kc = torch.zeros(nblk, G, 32, maps * d, device=dev, dtype=dtype)
    vc = torch.zeros(nblk, G, 32, dv, device=dev, dtype=dtype)
    table = torch.full((3, 6), -1, dtype=torch.int32, device=dev)
    table[1, :5] = torch.tensor([7, 2, 5, 0, 3], dtype=torch.int32)
    f = lambda t: t.float().to(dev).contiguous() if t is not None else None
    z_all = torch.cat([q.reshape(T, -1), k.reshape(T, -1), v.reshape(T, -1)], 1)
    qn, kn, vn = H * maps * d, G * maps * d, G * dv
    got, t0 = [], 0
    for n in (50, 47, 1, 1, 1, 50):
        tok_pos, tok_seq, *_ = _meta([(1, n, t0)], dev)
        z = f(z_all[t0:t0 + n])
        out = torch.zeros(n, H * dv, device=dev, dtype=dtype)
        K.rope_cache_write(z, H * maps, d, 0, None, 0, z[:, qn:], kn, G * maps, d, 0, kn, vn, False, kc, vc, dims, inter, f(cos), f(sin), tok_pos, tok_seq, table)
        K.multi_attention(out, z, maps * d, kc, vc, 0, tok_pos, tok_seq, table, H, d, dv, maps, scale, window, keep, cap, lam, post, eps,
                          f(gate[t0:t0 + n]) if maps == 2 else None)
        got.append(out.float().cpu())
        t0 += n
    close(torch.cat(got), ref, 2e-5 if dtype == torch.float32 else 2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("over_workgroups", [False, True])
@pytest.mark.parametrize("W,nb,taps", [(24, 3, 3), (16, 1, 1), (100, 100, 4), (320, 4, 2)])
def test_recurrent_unit_hip(W, nb, taps, over_workgroups):
    """short_conv_act + gemm_blocks + rglru_scan: two sequences in one step (a long portion that is scanned in segments
    beside a single token), several steps, slots that held other values, against the whole sequences."""
    K, dev, H = _K(), "cuda", 12
    bw = W // nb
    w = _rglru_weights(W, nb, taps, H, 30)
    ha, hb = rnd(700, H, seed=8), rnd(40, H, seed=9)
    ref_a, ref_b = O.rglru(ha, w), O.rglru(hb, w)
    f = lambda t: t.float().to(dev).contiguous()
    pre = lambda h: torch.cat([h @ w["y"].T + w["y.b"], h @ w["x"].T + w["x.b"]], 1)
    za, zb = pre(ha), pre(hb)
    wg, bg = f(torch.cat([w["ra"], w["ri"]], 1)), f(torch.cat([w["ra.b"], w["ri.b"]], 1).reshape(-1))
    clam = f(8.0 * O.softplus(w["lam"]))
    carry, state = torch.full((4, max(taps - 1, 1), W), 3.0, device=dev), torch.full((4, W), -2.0, device=dev)
    got_a, got_b, a0, b0 = [], [], 0, 0
    for na, nb_ in [(300, 1), (1, 1), (20, 2), (379, 36)]:
        seqs = [(2, nb_, b0), (0, na, a0)]
        _, _, q_start, ctx, slots = _meta(seqs, dev)
        z = f(torch.cat([zb[b0:b0 + nb_], za[a0:a0 + na]]))
        n = na + nb_
        u, gates, out = torch.zeros(n, W, device=dev), torch.zeros(n, 2 * W, device=dev), torch.zeros(n, W, device=dev)
        K.short_conv_act(u, z[:, W:], carry, f(w["conv"]), f(w["conv.b"]), q_start, ctx, slots, max(na, nb_), False)
        K.gemm_blocks(gates, u, wg, bg, bw, 2 * bw)
        ws = torch.zeros(int(K.rglru_scan_ws_floats(n, 2, W)), device=dev) if over_workgroups else None
        K.rglru_scan(out, u, gates, z[:, :W], clam, state, q_start, ctx, slots, bw, max(na, nb_), ws)
        got_b.append(out[:nb_].cpu())
        got_a.append(out[nb_:].cpu())
        a0, b0 = a0 + na, b0 + nb_
    close(torch.cat(got_a), ref_a, 5e-5)
    close(torch.cat(got_b), ref_b, 5e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("portions,over_workgroups", [((1,) * 40, False), ((40,), False), ((7, 300), False), ((300, 9), True)])
def test_recurrent_unit_of_closed_gates_hip(portions, over_workgroups):
    """Decay gates so far negative that 1 - a^2 falls below the normal range, and to 0, with decay rates from 0.002 up: finite, and within 2^-20 of the terms
    summed. A gate r below the normal range may be 0: its root is then off by up to sqrt(2 c 2^-126), c being the rate."""
    K, dev, T = _K(), "cuda", sum(portions)
    lam = torch.tensor([-8.0, -6.5, -5.0, -3.5, 0.0, 3.0], dtype=F64).repeat_interleave(11)
    W = len(lam)
    gr = torch.stack([torch.linspace(-104.0, -60.0, W, dtype=F64)[torch.randperm(W, generator=torch.Generator().manual_seed(t))] for t in range(T)]).float()
    u, gi, clam = rnd(T, W, seed=1).float(), rnd(T, W, seed=2).float(), (8.0 * O.softplus(lam)).float()
    la = -clam.to(F64) * torch.sigmoid(gr.to(F64))
    b = torch.sqrt(-torch.expm1(2 * la)) * torch.sigmoid(gi.to(F64)) * u.to(F64)
    S, want = torch.zeros(W, dtype=F64), []
    for t in range(T):
        S = torch.exp(la[t]) * S + b[t]
        want.append(S)
    bound = 2.0 ** -20 * b.abs().cumsum(0) + (torch.sqrt(2 * clam.to(F64) * 2.0 ** -126) * u.to(F64).abs()).cumsum(0)
    state, got, at = torch.full((2, W), 5.0, device=dev), [], 0
    for n in portions:
        i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
        sl = slice(at, at + n)
        out = torch.zeros(n, W, device=dev)
        ws = torch.zeros(int(K.rglru_scan_ws_floats(n, 1, W)), device=dev) if over_workgroups else None
        K.rglru_scan(out, u[sl].to(dev), torch.cat([gr, gi], 1)[sl].to(dev), torch.full((n, W), 3.0, device=dev), clam.to(dev), state, i32([0, n]), i32([at]), i32([1]),
                     W, n, ws)
        got.append(out.cpu().to(F64))
        at += n
        assert bool(((state[1].cpu().to(F64) - want[at - 1]).abs() <= bound[at - 1]).all())
    g = float(torch.nn.functional.gelu(torch.tensor(3.0, dtype=F64), approximate="tanh"))
    assert bool(((torch.cat(got) - g * torch.stack(want)).abs() <= g * bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rate", [0.05, 3.0])
def test_recurrent_unit_of_one_token_to_the_last_places_hip(rate):
    """A token's input alone, sqrt(1 - a^2): half of what the gate (two units in the last place) and the series (one) leave, and the root's half unit."""
    K, dev, W = _K(), "cuda", 1 << 18
    gr = torch.linspace(-5.0, 5.0, W).to(dev)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    state = torch.zeros(1, W, device=dev)
    one = torch.ones(1, W, device=dev)
    K.rglru_scan(torch.zeros(1, W, device=dev), one, torch.cat([gr, 100.0 * one[0]])[None], one, torch.full((W,), rate, device=dev), state, i32([0, 1]), i32([0]), i32([0]),
                 W, 1, None)
    want = torch.sqrt(-torch.expm1(-2.0 * torch.full((), rate, device=dev).to(F64) * torch.sigmoid(gr.to(F64))))
    unit = 2.0 ** (torch.frexp(want).exponent.to(F64) - 24)
    assert float(((state[0].to(F64) - want).abs() / unit).max()) <= 2.0


BLOCKS = [(16, 48, 512, 3), (9, 40, 520, 4), (40, 36, 128, 3), (300, 72, 1088, 5), (200, 448, 128, 32), (1900, 448, 128, 32), (500, 1020, 1024, 2)]


def test_block_products_reach_streams_and_tiles():
    from distributed_llm_inference_amd import ops
    form = ops.load(build_if_missing=True).gemm_any_form
    for f32 in (False, True):
        assert {form(M, N, k, nb, f32, 0) for M, N, k, nb in BLOCKS} >= {1, 64642, 64641, 48641, 32324, 32321}


def test_block_products_of_one_stage_by_their_output():
    from distributed_llm_inference_amd import ops
    form = ops.load(build_if_missing=True).gemm_any_form
    for M, N, nb in ((1900, 640, 32), (312, 640, 32), (1900, 4096, 1), (700, 640, 8)):          # us in tiles / general, fp32 out: 65.6 / 51.7, 15.9 / 13.3, 15.4 / 14.1, 9.9 / 9.0
        assert form(M, N, 64, nb, False, 0, True) == 0 and form(M, N, 64, nb, False, 0, False) != 0 and form(M, N, 32, nb, True, 0, True) == 0
    assert form(312, 448, 64, 8, False, 0, True) == form(312, 448, 64, 8, False, 0, False) != 0                                             # (the chip not full)


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("dt,ot", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("M,N,k,nb", BLOCKS)
def test_block_products_streams_and_tiles_hip(M, N, k, nb, dt, ot, bias):
    """Every block against 64 bits, read from and written into rows with gaps between the blocks. A sum of k products in fp32, in any order:
    within k roundings of the sum of the magnitudes (one more for the bias, and one of bf16 where the output is)."""
    K, dev, xs, os_ = _K(), "cuda", k + 16, N + 8
    g = torch.Generator(device=dev).manual_seed(M + N)
    x, w = torch.randn(M, nb * xs, device=dev, generator=g).to(dt), torch.randn(nb, N, k, device=dev, generator=g).to(dt)
    b = torch.randn(nb * N, device=dev, generator=g) if bias else None
    out = torch.full((M, nb * os_), 7.0, device=dev, dtype=ot)
    K.gemm_blocks(out, x, w, b, xs, os_)
    for i in range(nb):
        xi, wi = x[:, i * xs:i * xs + k].double(), w[i].double()
        bi = b[i * N:(i + 1) * N].double() if bias else torch.zeros(N, device=dev, dtype=F64)
        ref, mag = xi @ wi.t() + bi, xi.abs() @ wi.abs().t() + bi.abs()
        bound = (k + 1) * 2.0 ** -24 * mag + (2.0 ** -8 * ref.abs() if ot == torch.bfloat16 else 0.0)
        assert bool(((out[:, i * os_:i * os_ + N].double() - ref).abs() <= bound).all()), i
        assert bool((out[:, i * os_ + N:(i + 1) * os_] == 7.0).all()), i


@pytest.mark.gpu
@pytest.mark.parametrize("ot", [torch.float32, torch.bfloat16])
def test_block_products_of_one_stage_hip(ot):
    test_block_products_streams_and_tiles_hip(313, 636, 64, 32, torch.bfloat16, ot, True)


@pytest.mark.gpu
def test_block_products_activation_and_scale_hip():
    K, dev = _K(), "cuda"
    x, w, b = rnd(37, 5 * 12, seed=1), rnd(5, 7, 12, seed=2), rnd(5, 7, seed=3)
    ref = torch.einsum("tbi,boi->tbo", x.reshape(37, 5, 12), w) + b
    out = torch.zeros(37, 5 * 7, device=dev)
    K.gemm_blocks(out, x.float().to(dev), w.float().to(dev).contiguous(), b.float().to(dev).reshape(-1).contiguous(), 12, 7)
    close(out, ref.reshape(37, -1))
    # blocks that read overlapping-free slices of wider rows and write into wider rows (bf16 operands, fp32 sums)
    xb, wb = rnd(20, 3 * 24, seed=4).bfloat16(), rnd(3, 10, 16, seed=5).bfloat16()
    out = torch.zeros(20, 3 * 12, device=dev)
    K.gemm_blocks(out, xb.to(dev), wb.to(dev).contiguous(), None, 24, 12)
    ref = torch.einsum("tbi,boi->tbo", xb.to(F64).reshape(20, 3, 24)[:, :, :16], wb.to(F64))
    close(out.reshape(20, 3, 12)[:, :, :10], ref, 1e-5)
    z = rnd(9, 50, seed=6, std=3.0)
    p, q = torch.tensor(0.4, dtype=F64), torch.tensor(-1.1, dtype=F64)
    act = torch.zeros(9, 50, device=dev)
    K.xielu(act, z.float().to(dev), torch.stack([O.softplus(p), 0.5 + O.softplus(q)]).float().to(dev))
    close(act, O.xielu(z, p, q))
    lg = rnd(4, 30, seed=7).float().to(dev)
    ref = lg.cpu().to(F64).clone()
    ref[:, :25] *= 1.7
    K.scale_rows(lg, 25, 1.7)
    close(lg, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("M,F,ld", [(3, 1024, 1024), (5, 1022, 1024), (4, 260, 261), (1, 4, 4)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_xielu_rows_in_pieces_and_one_by_one(M, F, ld, dt):
    """Whole pieces of four and rows that are not, both sides of where the negative branch changes, zeros and large magnitudes. Negative side: |q|
    times two roundings of what the exponential and v leave, and of the sum's terms."""
    K, dev = _K(), "cuda"
    z = rnd(M, ld, seed=1, std=2.0)
    z[0, :4] = torch.tensor([0.0, -0.5, -3e38, 100.0])            # (q 3e38 = 3.15e38 is below the largest float, 3.4e38: with 1.3 the sum is infinite in any fp32 form)
    z = z.float()[:, :F]
    act, pq = torch.full((M, F), 7.0, device=dev, dtype=dt), torch.tensor([0.8, 1.05])
    K.xielu(act, z.to(dev), pq.to(dev))
    v, (p, q) = z.to(F64), pq.to(F64)
    ref = torch.where(v > 0, p * v * v, q * (torch.expm1(v.clamp(max=0)) - v)) + 0.5 * v
    bound = 2.0 ** -22 * (torch.where(v > 0, p * v * v, q * (1 + v.abs())) + 0.5 * v.abs()) + (2.0 ** -8 * ref.abs() if dt == torch.bfloat16 else 0)
    assert bool(((act.cpu().to(F64) - ref).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,F,ld", [(512, 1024, 1024), (511, 1024, 1024), (514, 1022, 1024), (520, 1024, 1025), (1, 1 << 19, 1 << 19)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_xielu_on_both_sides_of_the_line(M, F, ld, dt):
    """2^19 entries, from which on a thread takes four where the rows allow: the same entries one by one, to the bit."""
    K, dev = _K(), "cuda"
    z, pq = rnd(M, ld, seed=1, std=2.0).float().to(dev)[:, :F], torch.tensor([0.8, 1.05], device=dev)
    act, few = torch.full((M, F), 7.0, device=dev, dtype=dt), torch.full((M, F), 7.0, device=dev, dtype=dt)
    K.xielu(act, z, pq)
    for m in range(0, M, 64):
        for c in range(0, F, 4096):
            K.xielu(few[m:m + 64, c:c + 4096], z[m:m + 64, c:c + 4096], pq)
    assert torch.equal(act, few) and not bool((few == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("F", [65537, 65540])
def test_xielu_of_more_entries_than_a_dimension_has_threads(F):
    """A little over 2^32 entries one by one, and over 2^30 pieces of four, for which a launch has a second dimension: every row as one row by itself."""
    K, dev, M = _K(), "cuda", F
    z, pq = rnd(1, F, seed=1, std=2.0).float().to(dev), torch.tensor([0.8, 1.05], device=dev)
    one, act = torch.zeros(1, F, device=dev, dtype=torch.bfloat16), torch.full((M, F), 7.0, device=dev, dtype=torch.bfloat16)
    K.xielu(one, z, pq)
    K.xielu(act, z.expand(M, F), pq)
    assert all(torch.equal(a, one.expand(len(a), F)) for a in act.split(4096))


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,d,dv,maps,window,keep,cap,dims,inter", [
    (4, 2, 16, 24, 2, 40, 5, 10.0, 8, True), (2, 1, 8, 8, 1, 0, 0, 0.0, 8, False), (3, 3, 24, 70, 2, 3, 50, 0.0, 4, True),
    (2, 2, 72, 130, 1, 33, 0, 3.0, 0, False), (6, 1, 40, 16, 2, 64, 1, 25.0, 10, True), (1, 1, 104, 300, 1, 0, 0, 0.0, 16, False),
    (2, 1, 56, 80, 2, 31, 33, 12.0, 14, True)])
def test_tile_attention_hip(H, G, d, dv, maps, window, keep, cap, dims, inter):
    """The matrix-core attention kernel (bf16, values key-contiguous in the cache) on two sequences that share steps with
    different portions (down to single tokens), blocks in no order, against whole-sequence attention."""
    K, dev, dtype = _K(), "cuda", torch.bfloat16
    T, eps, lam, post, scale = 150, 1e-5, 0.37, 0.6, 0.3
    q, k = rnd(T, H * maps, d, seed=1), rnd(T, G * maps, d, seed=2)
    v, gate = rnd(T, G, dv, seed=3).bfloat16().to(F64), rnd(T, H * dv, seed=4)
    cos, sin = O.rope_angles({"dims": dims, "base": 50.0}, T) if dims else (None, None)
    qr, kr = (O.rotate(q, cos, sin, inter), O.rotate(k, cos, sin, inter)) if dims else (q, k)
    qr, kr = qr.bfloat16().to(F64), kr.bfloat16().to(F64)          # (what the kernel reads: rotated in fp32, then rounded)
    ok = O.visible(T, window, keep)
    heads = []
    for hh in range(H):
        g, per = hh // (H // G), []
        for mp in range(maps):
            s = (qr[:, maps * hh + mp] @ kr[:, maps * g + mp].T) * scale
            if cap > 0:
                s = cap * torch.tanh(s / cap)
            per.append(torch.softmax(s.masked_fill(~ok, float("-inf")), -1) @ v[:, g])
        heads.append(O.rms(per[0] - lam * per[1], eps) * post if maps == 2 else per[0])
    ref = torch.cat(heads, -1) * (torch.sigmoid(gate) if maps == 2 else 1.0)
    nblk = 12
    kc = torch.zeros(nblk, G, 32, maps * d, device=dev, dtype=dtype)
    vt = torch.zeros(nblk, G, dv, 32, device=dev, dtype=dtype)
    table = torch.full((3, 6), -1, dtype=torch.int32, device=dev)
    table[1, :5] = torch.tensor([7, 2, 5, 0, 3], dtype=torch.int32)
    table[2, :5] = torch.tensor([11, 1, 9, 4, 6], dtype=torch.int32)
    f = lambda t: t.float().to(dev).contiguous() if t is not None else None
    z_all = torch.cat([q.reshape(T, -1), k.reshape(T, -1), v.reshape(T, -1)], 1)
    qn, kn, vn = H * maps * d, G * maps * d, G * dv
    got_a, got_b, a0, b0 = [], [], 0, 0
    for na, nb in zip((50, 47, 1, 1, 1, 50), (1, 20, 30, 1, 34, 64)):      # (the fourth step brings single tokens only)
        tok_pos, tok_seq, q_start, ctx, slots = _meta([(2, nb, b0), (1, na, a0)], dev)
        z = f(torch.cat([z_all[b0:b0 + nb], z_all[a0:a0 + na]]))
        gt = f(torch.cat([gate[b0:b0 + nb], gate[a0:a0 + na]]))
        n = na + nb
        out, q16 = torch.zeros(n, H * dv, device=dev, dtype=dtype), torch.zeros(n, qn, device=dev, dtype=dtype)
        K.rope_cache_write(z, H * maps, d, 0, q16, qn, z[:, qn:], kn, G * maps, d, 0, kn, vn, True, kc, vt, dims, inter, f(cos), f(sin),
                           tok_pos, tok_seq, table)
        part = torch.zeros(int(K.tile_attention_part_floats(2, H, G, dv, maps)), device=dev)
        K.tile_attention(out, q16, maps * d, kc, vt, q_start, ctx, slots, table, max(na, nb), H, d, dv, maps, scale, window, keep, cap, lam,
                         post, eps, gt if maps == 2 else None, part)
        got_b.append(out[:nb].float().cpu())
        got_a.append(out[nb:].float().cpu())
        a0, b0 = a0 + na, b0 + nb
    close(torch.cat(got_a), ref, 2e-2)
    close(torch.cat(got_b), ref, 2e-2)


@pytest.mark.gpu
def test_tile_attention_caps_and_weights_to_the_last_places_hip():
    """What the key splits of single-token steps leave for the merge, in fp32: the capped score of one key (the cap a power of two: the tanh's error alone) and
    values of a first block rescaled by the weight that a second block's maximum leaves them. One unit in the last place and a rounding each."""
    K, dev, bf, B, H, d, dv = _K(), "cuda", torch.bfloat16, 1024, 16, 8, 8
    i32 = lambda v: v.to(torch.int32).to(dev)
    units = lambda got, want: float(((got.to(F64) - want).abs() / 2.0 ** (torch.frexp(want).exponent.to(F64) - 24)).max())

    def parts(x, blocks, cap):
        q = torch.zeros(B, H, d, device=dev, dtype=bf)
        q[:, :, 0] = x
        kc, vt = torch.zeros(2, 1, 32, d, device=dev, dtype=bf), torch.zeros(2, 1, dv, 32, device=dev, dtype=bf)
        kc[-1, :, :, 0], vt[0] = 1.0, 1.0                     # block 0: scores of 0, values of 1; block 1: scores of x, values of 0
        part = torch.zeros(int(K.tile_attention_part_floats(B, H, 1, dv, 1)), device=dev)
        assert part.numel() == B * H * (dv + 2)               # (one split)
        n = torch.full((B,), 31 if blocks == [1] else 63)
        K.tile_attention(torch.zeros(B, H * dv, device=dev, dtype=bf), q.view(B, -1), d, kc, vt, i32(torch.arange(B + 1)), i32(n), i32(torch.arange(B)),
                         i32(torch.tensor(blocks)).repeat(B, 1), 1, H, d, dv, 1, 1.0, 0, 0, cap, 0.0, 1.0, 1e-5, None, part)
        return part.view(B, H, dv + 2)

    for lo, hi in ((0.5, 8.0), (-40.0, -2.0)):
        x = torch.linspace(lo, hi, B * H, device=dev).view(B, H).to(bf)
        assert units(parts(x, [1], 8.0)[:, :, dv], 8.0 * torch.tanh(x.to(F64) / 8.0)) <= 1.5
    x = torch.linspace(0.25, 80.0, B * H, device=dev).view(B, H).to(bf)
    assert units(parts(x, [0, 1], 0.0)[:, :, :dv], (32.0 * torch.exp(-x.to(F64)))[:, :, None].expand(-1, -1, dv)) <= 1.5


@pytest.mark.gpu
@pytest.mark.parametrize("window,keep,chunk", [(100, 0, 0), (100, 70, 0), (64, 33, 0), (31, 300, 0), (1, 1, 0), (0, 0, 96), (70, 0, 96), (0, 0, 1)])
@pytest.mark.parametrize("H,G,d,dv,cap", [(4, 2, 64, 64, 0.0), (8, 1, 72, 128, 20.0), (3, 3, 128, 24, 0.0)])
@pytest.mark.parametrize("lens", [[(0, 200), (300, 131), (0, 0), (64, 1), (95, 33)], [(401, 17)], [(33, 1), (0, 1), (200, 1)]])
def test_tile_attention_blocks_seen_in_full_hip(lens, H, G, d, dv, cap, window, keep, chunk):
    """Blocks without masks on the edges of windows, kept first tokens and chunks; the tiles of sequences of different lengths, last ones first, an empty one
    among them. Weights are rounded to bf16 (the sum is of the unrounded ones), the result once more; fp32 scores move a weight by less than 2^-11 of itself."""
    K, dev, bf = _K(), "cuda", torch.bfloat16
    lens = [(c, n) for c, n in lens if n or max(m for _, m in lens) > 1]
    nb, B = [(c + n + 31) // 32 for c, n in lens], len(lens)
    table = torch.full((B, max(nb) + 1), -1, dtype=torch.int32)
    perm = torch.randperm(sum(nb), generator=torch.Generator().manual_seed(5)).int().split(nb)
    for b in range(B):
        table[b, :nb[b]] = perm[b]
    kc, vt = rnd(sum(nb), G, 32, d, seed=1).to(bf), rnd(sum(nb), G, dv, 32, seed=2).to(bf)
    starts = torch.tensor([0] + [n for _, n in lens]).cumsum(0)
    q, mq = rnd(int(starts[-1]), H * d, seed=3).to(bf), max(n for _, n in lens)
    out = torch.full((len(q), H * dv), 9.0, device=dev, dtype=bf)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    part = torch.zeros(int(K.tile_attention_part_floats(B, H, G, dv, 1)), device=dev)
    K.tile_attention(out, q.to(dev), d, kc.to(dev), vt.to(dev), starts.int().to(dev), i32([c for c, _ in lens]), i32(list(range(B))), table.to(dev), mq, H, d, dv, 1,
                     d ** -0.5, window, keep, cap, 0.0, 1.0, 1e-5, None, part, chunk)
    for b, (c, n) in enumerate(lens):
        blk = table[b, :nb[b]].long()
        k, v = kc[blk].to(F64).permute(1, 0, 2, 3).reshape(G, -1, d)[:, :c + n], vt[blk].to(F64).permute(1, 0, 3, 2).reshape(G, -1, dv)[:, :c + n]
        i, j = torch.arange(c, c + n)[:, None], torch.arange(c + n)[None]
        see = (j <= i) & (((i - j < window) | (j < keep)) if window else True) & ((j >= i // chunk * chunk) if chunk else True)
        rows = slice(int(starts[b]), int(starts[b + 1]))
        for h in range(H):
            s = q[rows, h * d:(h + 1) * d].to(F64) @ k[h // (H // G)].T * d ** -0.5
            s = cap * torch.tanh(s / cap) if cap else s
            w = torch.softmax(s.masked_fill(~see, float("-inf")), -1)
            want, room = w @ v[h // (H // G)], w @ v[h // (H // G)].abs()
            got = out[rows, h * dv:(h + 1) * dv].cpu().to(F64)
            assert bool(((got - want).abs() <= (2.0 ** -8 + 2.0 ** -11) * room + 2.0 ** -8 * want.abs() + 1e-6).all()), (b, h)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,Gk,d,dv,window,keep,cap,chunk,sink", [
    (16, 4, 1, 64, 64, 0, 0, 0.0, 0, True), (8, 8, 1, 16, 4, 0, 0, 0.0, 0, False), (24, 3, 1, 48, 68, 90, 5, 0.0, 0, True), (40, 2, 2, 32, 128, 0, 0, 20.0, 0, False),
    (16, 1, 1, 576, 512, 0, 0, 0.0, 130, True), (16, 1, 1, 592, 64, 0, 0, 0.0, 0, False), (16, 16, 1, 64, 128, 70, 0, 0.0, 0, False)])
def test_fp32_heads_of_one_key_row(H, G, Gk, d, dv, window, keep, cap, chunk, sink):
    """Heads that share a key row in fp32: positions around the rounds of 128 keys, tiles of heads that are not whole, several value heads a
    tile, window with kept first keys, chunks, blocks that are missing, padding rows; sizes on both sides of what the matrix cores
    take.  Scores of magnitude s carry d roundings of 2^-24 s, weights and sums as many again: 2^-24 (4 d + 4 keys) in all."""
    from distributed_llm_inference_amd import ops
    K = ops.load()
    torch.manual_seed(11)
    pos = [0, 15, 16, 127, 128, 129, 300, 31, 5, 9]
    seq = [0, 0, 0, 0, 0, 0, 0, 1, -1, 2]
    mb, T = 12, len(pos)
    nb = 3 * mb
    table = torch.randperm(nb).view(3, mb).int()
    table[0, 1] = -1                                                   # a block that is not there
    table[2] = nb + 5
    kc, vc = torch.randn(nb, Gk, 32, d), torch.randn(nb, G, 32, dv + 4)
    q, gate, sk = torch.randn(T, H * d) * d ** -0.5, torch.randn(T, H * dv), torch.randn(H)
    out = torch.full((T, H * dv), 9.0, device="cuda")
    dev = lambda x: x.cuda()
    K.multi_attention(out, dev(q), d, dev(kc), dev(vc), 4, dev(torch.tensor(pos, dtype=torch.int32)), dev(torch.tensor(seq, dtype=torch.int32)), dev(table), H, d, dv, 1,
                      1.5, window, keep, cap, 0.0, 1.0, 1e-5, dev(gate), chunk, dev(sk) if sink else None)
    out = out.cpu().double()
    for t in range(T):
        s = seq[t]
        if s < 0:
            assert bool((out[t] == 0).all())
            continue
        ok = (table[s] >= 0) & (table[s] < nb)
        bl = table[s].clamp(0, nb - 1).long()
        key, val = kc[bl].permute(0, 2, 1, 3).reshape(mb * 32, Gk, d).double(), vc[bl].permute(0, 2, 1, 3).reshape(mb * 32, G, dv + 4)[:, :, 4:].double()
        j = torch.arange(mb * 32)
        vis = (j <= pos[t]) & ok.repeat_interleave(32)
        if window:
            vis &= (j > pos[t] - window) | (j < keep)
        if chunk:
            vis &= j >= pos[t] // chunk * chunk
        for h in range(H):
            sc = 1.5 * key[vis][:, h // (H // Gk)] @ q[t, h * d:(h + 1) * d].double()
            sc = cap * torch.tanh(sc / cap) if cap else sc
            m = sc.max() if len(sc) else torch.tensor(0.0).double()
            e = (sc - m).exp()
            den = e.sum() + ((sk[h].double() - m).exp() if sink else 0.0)
            ref = (e @ val[vis][:, h // (H // G)] / den if len(sc) else torch.zeros(dv).double()) * torch.sigmoid(gate[t, h * dv:(h + 1) * dv].double())
            err = float((out[t, h * dv:(h + 1) * dv] - ref).abs().max())
            assert err <= 2.0 ** -24 * 4 * (d + pos[t] + 1) * max(1.0, float(ref.abs().max())), (t, h, err)
