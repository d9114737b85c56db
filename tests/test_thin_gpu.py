"""Weight stream of at most 16 rows with all of K in a workgroup (`gemm_thin`, `gemm_thin_qkv`) and the steps that run on it."""
import pytest
import torch

from distributed_llm_inference_amd import ops
from distributed_llm_inference_amd.ops import packing

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


@pytest.fixture(scope="module")
def K():
    return ops.load()


def rand(*shape, seed, std=1.0):
    return (torch.randn(*shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed)) * std).bfloat16()


def normed(x, w, eps):
    """The rows as the GEMM reads them: normalised in 64 bits, then bf16, and how far a value can be from that (32-bit sums, the next bf16)."""
    y = x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + eps) * w.double()
    return y.bfloat16().double(), 2.0 ** -8 * y.abs()


# K of one k-step a wave and less, of ragged chunks, of one, two and seven chunks; two waves a row above 2048; N below, at and beyond 256 tiles
@pytest.mark.parametrize("M,N,Kd", [(1, 128, 128), (2, 48, 384), (15, 100, 2048), (16, 256, 640), (1, 4224, 2048), (3, 160, 2176), (7, 96, 4096), (8, 4160, 1152)])
@pytest.mark.parametrize("epi", [2, 4, 6])
def test_gemm_thin(K, M, N, Kd, epi):
    N = (N + 31) // 32 * 32 if epi == 4 else N
    x, w, g = rand(M, Kd + 8, seed=1)[:, :Kd], rand(N, Kd, seed=2, std=Kd ** -0.5), rand(Kd, seed=3) + 1
    b, r = rand(N, seed=4), rand(M, N + 8, seed=5)[:, :N]
    n_out = N // 2 if epi == 4 else N
    out = torch.full((M, n_out + 8), 7.0, device=DEV, dtype=torch.float32 if epi == 6 else torch.bfloat16)
    xv, slack = (x.double(), torch.zeros_like(x, dtype=F64)) if epi == 2 else normed(x, g, 1e-5)
    ref, mag = xv @ w.double().t(), (Kd + 1) * 2.0 ** -24 * (xv.abs() @ w.double().abs().t()) + slack @ w.double().abs().t()
    if epi == 4:
        wi = packing.interleave_gate_up(w[:N // 2], w[N // 2:])
        K.gemm_thin(out[:, :n_out], x, packing.pack_weight(wi), g, 1e-5, None, None, N, 4)
        a, u = ref[:, :N // 2], ref[:, N // 2:]
        want = a * torch.sigmoid(a) * u                # (silu's slope is at most 1.1; __expf and v_rcp_f32: a few units of 2^-22)
        bound = 1.1 * mag[:, :N // 2] * u.abs() + (a * torch.sigmoid(a)).abs() * mag[:, N // 2:] + (2.0 ** -8 + 2.0 ** -20) * want.abs() + 1.1 * mag[:, :N // 2] * mag[:, N // 2:]
    elif epi == 2:
        K.gemm_thin(out[:, :n_out], x, packing.pack_weight(w), None, 0.0, b, r, N, 2)
        want = ref + b.double() + r.double()
        bound = mag + 2.0 ** -8 * want.abs() + 2.0 ** -22 * (b.double().abs() + r.double().abs())
    else:
        K.gemm_thin(out[:, :n_out], x, packing.pack_weight(w), g, 1e-5, None, None, N, 6)
        want, bound = ref, mag
    assert bool(((out[:, :n_out].double() - want).abs() <= bound + 1e-30).all())
    assert bool((out[:, n_out:] == 7.0).all())


@pytest.mark.parametrize("M,Hq,Hkv,D,Kd", [(1, 4, 2, 64, 256), (15, 32, 4, 64, 2048), (2, 8, 8, 128, 1024), (7, 32, 8, 128, 4096), (3, 6, 2, 128, 2176)])
@pytest.mark.parametrize("bias", [False, True])
def test_gemm_thin_qkv_is_the_gemm_and_the_rotation(K, M, Hq, Hkv, D, Kd, bias):
    """The same sums through `gemm_thin` and `rope_kvwrite`: the same bits, in q's rows and in the cache; a row without a block leaves the cache alone."""
    N = (Hq + 2 * Hkv) * D
    x, w, g = rand(M, Kd, seed=1), packing.pack_weight(rand(N, Kd, seed=2, std=Kd ** -0.5)), rand(Kd, seed=3) + 1
    pb = rand(N, seed=4) if bias else None
    cos, sin = torch.rand(50, D // 2, device=DEV), torch.rand(50, D // 2, device=DEV)
    pos = torch.arange(M, device=DEV, dtype=torch.int32) * 3 + 1
    seq = torch.arange(M, device=DEV, dtype=torch.int32)
    table = torch.randperm(2 * M, device=DEV).to(torch.int32).view(M, 2)
    table[M - 1, 1] = -1
    pos[M - 1] = 40 if M > 1 else 1
    sums = torch.empty(M, N, device=DEV)
    K.gemm_thin(sums, x, w, g, 1e-5, None, None, N, 6)
    want, got = (torch.zeros(M, N, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    kv0, kv1 = (torch.zeros(2 * M, Hkv, 2, 32 * D, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    K.rope_kvwrite(want, sums, 1, pb, kv0, cos, sin, pos, seq, table, Hq, Hkv, D, True)
    K.gemm_thin_qkv(got, x, w, g, 1e-5, pb, kv1, cos, sin, pos, seq, table, Hq, Hkv, D)
    # (another number of waves adds K in another order: both within K roundings of the sum, then one of bf16)
    for a, b in ((got[:, :Hq * D], want[:, :Hq * D]), (kv1, kv0)):
        assert float((a.double() - b.double()).norm()) <= 2.0 ** -9 * float(b.double().norm())
        assert bool(((a == 0) == (b == 0)).all())
    assert M == 1 or bool((kv1[table[M - 1, 0].long()] == 0).all())


def test_gemm_thin_refuses_what_it_cannot_hold(K):
    w, g = packing.pack_weight(rand(128, 4096, seed=1)), rand(4096, seed=2)
    out = torch.empty(16, 128, device=DEV)
    for x in (rand(17, 128, seed=3), rand(9, 4096, seed=3)):
        with pytest.raises(RuntimeError, match="gemm_thin|packed weight size"):
            K.gemm_thin(out, x, w, g, 1e-5, None, None, 128, 6)


@pytest.mark.parametrize("model,rows", [("tiny-llama-gpu-test", 3), ("tiny-qwen2-gpu-test", 16)])
@pytest.mark.parametrize("part", [(0, 0, 4, True, True), (1, 1, 3, False, False)])
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
def test_steps_of_few_rows(model, rows, part, kv):
    """Prompt and captured decode steps of a stage, whole or in the middle, on `gemm_thin` and on the kernels of larger steps."""
    from distributed_llm_inference_amd.models import weights as W
    from distributed_llm_inference_amd.models.partition import StagePlan
    from distributed_llm_inference_amd.models.spec import BUILTIN_SPECS
    from distributed_llm_inference_amd.models.stage_gpu import GpuStage
    from distributed_llm_inference_amd.runtime.batch import StepBatch
    spec, plan = BUILTIN_SPECS[model], StagePlan(part[0], 3 if part[0] else 1, *part[1:])
    outs = []
    for thin in (0, 16):
        ex = GpuStage(spec, plan, W.random_stage_weights(spec, plan, seed=1, device=DEV, dtype=torch.bfloat16), device=DEV, max_slots=rows, max_seq_len=96,
                      num_blocks=3 * rows, max_batch=rows, max_tokens=64, kv_dtype=kv)
        ex._thin_rows = thin
        new = lambda q, c, ids, **kw: StepBatch(slots=list(range(rows)), q_lens=[q] * rows, ctx_lens=[c] * rows, sample=[1] * rows, temperature=[0.7] * rows,
                                                top_k=[5] * rows, top_p=[0.9] * rows, seeds=list(range(rows)), sample_steps=[0] * rows, token_ids=ids, **kw)
        tables = dict(table_slots=list(range(rows)), table_blocks=[[3 * i, 3 * i + 1, 3 * i + 2] for i in range(rows)])
        n = 4 if rows < 4 else 1                        # (12 or 16 tokens: few rows of a prompt too)
        ids = torch.arange(rows * n, dtype=torch.int32) * 7 % spec.vocab_size
        x = None if plan.has_embed else rand(rows * n, spec.hidden_size, seed=9, std=3.0)
        got = [ex.forward(new(n, 0, None, **tables), ids if plan.has_embed else x).float().clone()]
        for s in range(3):
            step = new(1, n + s, [(5 * i + s) % spec.vocab_size for i in range(rows)])
            out = ex.decode_step(step, None if plan.has_embed else rand(rows, spec.hidden_size, seed=10 + s, std=3.0))
            got.append((ex._mb_state(0, rows).wk.logits[:rows, :spec.vocab_size] if plan.has_head else out).float().clone())
        assert ex.graph_replays == 3 and ex._mb_state(0, rows).ctx.tolist() == [n + 3] * rows
        outs.append(got)
    for a, b in zip(*outs):                             # (bf16 roundings of other sums, through two or four layers)
        assert float((a - b).norm()) <= 0.03 * float(b.norm())
