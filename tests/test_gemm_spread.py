"""How far a GEMM of more than 256 rows is spread when it has the chip for itself (`gemm_spread`)."""
import pytest


@pytest.fixture(scope="module")
def K():
    from distributed_llm_inference_amd import ops
    return ops.load(build_if_missing=True)


def splits(M, N, kt, target):
    s = min(8, (target if target > 1 else 128) // ((M + 255) // 256 * ((N + 255) // 256)))
    while s > 1 and kt // s < 8:
        s -= 1
    return max(s, 1)


def test_never_more_splits_than_fit_and_room_for_them(K):
    for M in (257, 300, 512, 513, 1000, 1531, 2048, 4100):
        for N in (16, 128, 1000, 2048, 4096, 6144, 14336, 28672):
            for kt in (1, 7, 16, 17, 32, 64, 88, 224):
                t = int(K.gemm_spread(M, N, kt))
                tiles = (M + 255) // 256 * ((N + 255) // 256)
                assert 1 < t <= 256 and splits(M, N, kt, t) <= splits(M, N, kt, 256)
                assert tiles * (splits(M, N, kt, t) - 1) * 65536 <= int(K.gemm_ws_floats(M, N, kt * 64))


def test_splits_that_measured_fastest(K):
    # us: all that fit -> these
    for M, N, kt, s in ((300, 4096, 64, 4), (512, 4096, 64, 4), (300, 4096, 224, 5), (300, 4096, 112, 5), (1024, 2048, 88, 4),        # 46 -> 38, 75 -> 69, 57 -> 48, 54 -> 44
                        (768, 4096, 224, 4), (2048, 4096, 224, 2)):                                                                # 87 -> 86, 173
        t = int(K.gemm_spread(M, N, kt))
        assert splits(M, N, kt, t) in (s, s + 1 if kt == 224 and M == 300 else s), (M, N, kt, t)
    assert int(K.gemm_spread(1531, 14336, 64)) == 256 and int(K.gemm_spread(2048, 28672, 64)) == 256                              # halves of the last round
