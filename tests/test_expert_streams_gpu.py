"""Experts of steps with 16 rows an expert and more: the weight stream takes an expert's 32-row tiles two at a time."""
import pytest
import torch

from distributed_llm_inference_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[1, 33, 64, 65, 97, 0, 16, 17], [128, 0, 0, 0, 0, 0, 0, 0], [48, 49, 31, 32, 129, 2, 80, 96]])
@pytest.mark.parametrize("kind,N", [(0, 4090), (1, 4090), (2, 4100)])
@pytest.mark.parametrize("k", [1152, 2048])
def test_tiles_two_at_a_time(counts, kind, N, k):
    """Experts of one to five tiles, three and four halves of a pair, ragged last columns; sums of k products in fp32, what the activation makes of
    them, one rounding of 16-bit results. Rows of no token and what lies behind the tiles stay as they were or are never read."""
    K = ops.load()
    E, T, tr, bf = len(counts), sum(counts), 32, torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(k + N)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    nt = (T + tr - 1) // tr + E
    assert 2 * (nt - E) >= E and not K.moe_short(nt, E, N, k, False, kind) and not K.moe_wide(nt, E, N, kind == 0)
    sel = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=torch.Generator().manual_seed(k))].int().cuda()
    wts, row_w = torch.rand(T, device="cuda", generator=g) + 0.5, torch.full((tr * nt,), float("nan"), device="cuda")
    tiles, row_tok, pair_row = (torch.full((n,), 77777, dtype=torch.int32, device="cuda") for n in (1 + nt, tr * nt, T))
    K.moe_plan(tiles, row_tok, pair_row, sel, T, 1, E, tr, wts, row_w)
    x, w, w2 = r(tr * nt if kind == 0 else T, k).to(bf), (r(E, N, k) * k ** -0.5).to(bf), (r(E, N, k) * k ** -0.5).to(bf)
    out = torch.full((tr * nt, N), 3.0, device="cuda", dtype=torch.float32 if kind == 0 else bf)
    if kind == 0:
        K.moe_down(out, x, w, tiles, row_tok, nt, tr)
    else:
        K.moe_up(out, x, w if kind == 1 else None, w2, tiles, row_tok, nt, 0.0, tr, row_w if kind == 2 else None)
    assert bool((out[int(tiles[0]) * tr:] == 3.0).all())
    eps = (k + 1) * 2.0 ** -24
    for e in range(E):
        at = torch.nonzero(sel == e).squeeze(1)
        rows = pair_row[at].long()
        a = (x[rows] if kind == 0 else x[at]).double()
        if kind == 2:
            a = a * wts[at].double()[:, None]
        p, m = a @ w[e].double().t(), eps * (a.abs() @ w[e].double().abs().t())
        q, n = a @ w2[e].double().t(), (eps + 2.0 ** -23) * (a.abs() @ w2[e].double().abs().t())
        if kind == 0:
            ref, bound = p, m
        elif kind == 1:
            s = p * torch.sigmoid(p)
            ref, bound = s * q, 1.1 * m * (q.abs() + n) + s.abs() * n
        else:
            u = torch.relu(q)
            ref, bound = u * u, 2 * u * n + n * n
        if kind:
            bound = bound + (2.0 ** -8 + 2.0 ** -20) * ref.abs()
        assert bool(((out[rows].double() - ref).abs() <= bound).all()), e
