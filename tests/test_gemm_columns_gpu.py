"""Streaming GEMMs of up to 128 rows with 64 columns a workgroup, whole in K or split: the shapes at which the choice changes."""
import pytest
import torch

from distributed_llm_inference_amd import ops
from distributed_llm_inference_amd.ops import packing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,Kd,choice", [
    (768, 1024, (1, 1)), (776, 1152, (1, 2)),         # a K that is walked whole, the first that is split
    (4104, 2048, (1, 4)), (8192, 4096, (1, 2)),       # a last block of 8 columns, the widest that is split
    (8200, 4096, (1, 1)), (8200, 4224, (2, 2)),       # whole from there on, unless K is long
    (16384, 1152, (1, 1)), (16392, 1152, (2, 1)),     # the widest with 64 columns
])
@pytest.mark.parametrize("M", [1, 17, 64, 65, 128])
def test_columns_and_splits(N, Kd, choice, M):
    K, dev = ops.load(), "cuda"
    assert tuple(K.gemm_config(M, N, Kd, 0, True)) == choice
    g = torch.Generator(device=dev).manual_seed(N + Kd + M)
    x = torch.randn(M, Kd, device=dev, generator=g).bfloat16()
    w = torch.randn(N, Kd, device=dev, generator=g).bfloat16()
    res = torch.randn(M, N, device=dev, generator=g).bfloat16()
    ws = torch.empty(4 * M * N, device=dev)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    out = torch.full((M, N), 7.0, device=dev)
    K.gemm(out, x, packing.pack_weight(w), None, None, ws, N, 0, 0, 0)
    bound = Kd * 2.0 ** -24 * size                    # a rounding of the sum for every product
    assert ((out - want).abs() <= bound).all()
    out16 = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
    K.gemm(out16, x, packing.pack_weight(w), None, res, ws, N, 2, 0, 0)
    full = want + res.double()
    assert ((out16.double() - full).abs() <= bound + 2.0 ** -8 * full.abs()).all()      # (and the result's own)
    if M in (17, 128):                                # e4m3 weights, and e4m3 rows as well: exact products of what is stored
        wq, sc = packing.pack_weight_fp8(w)
        back = packing.unpack_weight_fp8(wq, sc, N, Kd).double()
        K.gemm_w8(out, x, wq, sc, None, None, ws, N, 0, 0, 0)
        assert ((out - x.double() @ back.t()).abs() <= (Kd + 2) * 2.0 ** -24 * (x.double().abs() @ back.abs().t())).all()
        wq, sc = packing.pack_weight_a8w8(w)
        xq, xs = torch.empty(M, Kd, device=dev, dtype=torch.uint8), torch.empty(M, device=dev)
        K.quant_rows(xq, xs, x)
        K.gemm_a8w8(out, xq, xs, wq, sc, None, None, ws, N, 0, 0, 0)
        two = torch.empty_like(out)
        K.gemm_a8w8(two, xq, xs, wq, sc, None, None, ws, N, 0, 1, 2)      # (128 columns, whole)
        assert ((out - two).abs() <= 2 * (Kd + 2) * 2.0 ** -24 * 1.2 * size).all()
