"""The sampler's order of its candidates: by value, equal values by index, at the sizes where the sort changes its way of exchanging."""
import pytest
import torch

from distributed_llm_inference_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [4, 60, 64, 68, 128, 132, 256, 260, 512, 516, 1020, 1024])
@pytest.mark.parametrize("values", [3, 100, 0])          # (how many different ones; 0: hardly two alike)
def test_candidates_in_order(V, values):
    K, R = ops.load(), 5
    g = torch.Generator(device="cuda").manual_seed(V + values)
    lg = torch.randn(R, V, device="cuda", generator=g)
    if values:
        lg = torch.randint(-values // 2, values // 2, (R, V), device="cuda", generator=g).float() / values
    lg[0, V // 2] = -float("inf")
    f = lambda v: torch.full((R,), v, device="cuda")
    out, steps = (torch.zeros(R, dtype=torch.int32, device="cuda") for _ in range(2))
    probs, ids = torch.zeros(R, V, device="cuda"), torch.zeros(R, V, dtype=torch.int32, device="cuda")
    K.sample(out, lg, f(0.7), torch.full((R,), V, dtype=torch.int32, device="cuda"), f(1.0), torch.arange(R, device="cuda"), steps, V, probs, ids)
    order = torch.sort(lg.cpu(), dim=1, descending=True, stable=True).indices
    for r in range(R):
        assert torch.equal(ids[r].cpu().long(), order[r]), r
        want = torch.softmax(lg[r].cpu().double()[order[r]] / 0.7, 0)
        assert (probs[r].cpu().double() - want).abs().max() <= 1e-5      # (__expf and a sum of 1024 fp32 terms: both below 2^-17)
        assert 0 <= int(out[r]) < V
