"""i32 layers whose values leave int8: the digit-plane products on the int8
matrix cores (gemm_i8.hip), bit-exact against the wrapping integer sum.

Values at the edges of one to four signed base-256 digits, digit counts that
differ from tile to tile (planes a tile does not have are read as zeros), K
of fewer 64-wide chunks than the four waves that split it, more than 64 chunks
a wave (the counts register is reloaded), and ragged M, N and K; on the 64x64
tiles that small layers take and, forced, inside each 128x128 variant."""
from __future__ import annotations

import numpy as np
import pytest

from mlir_edsl_hip import _native

pytestmark = pytest.mark.gpu

# The last value of a digit count and the first of the next, both signs.
EDGES = np.array([0, 127, 128, -128, -129, 32639, 32640, -32896, -32897, 8355711, 8355712, -8421504, -8421505,
                  2**31 - 1, -2**31], dtype=np.int64)


def _operands(kind, rng, M, K, N):
    if kind == "edges":
        return rng.choice(EDGES, (M, K)), rng.choice(EDGES, (K, N))
    if kind == "wide_x":
        return rng.integers(-30000, 30000, (M, K)), rng.integers(-128, 128, (K, N))
    if kind == "full":
        return rng.integers(-2**31, 2**31, (M, K)), rng.integers(-2**31, 2**31, (K, N))
    X, W = rng.integers(-100, 100, (M, K)), rng.integers(-100, 100, (K, N))  # "mixed"
    X[:, K // 2:] *= 300
    W[:K // 3] *= 70000
    X[M // 2, 0] = 2**31 - 1
    W[0, N // 2] = -2**31
    return X, W


@pytest.mark.parametrize("kind", ["edges", "wide_x", "full", "mixed"])
@pytest.mark.parametrize("M, K, N", [(1, 1, 1), (65, 33, 17), (64, 64, 64), (200, 300, 257), (130, 1000, 129)])
def test_digit_planes_are_exact(M, K, N, kind):
    import torch
    from mlir_edsl_hip.device import dense_launch, set_i8_variant
    rng = np.random.default_rng(M + 3 * K + 7 * N)
    X, W = (a.astype(np.int32) for a in _operands(kind, rng, M, K, N))
    b = rng.integers(-2**31, 2**31, N).astype(np.int32)
    # int64 products wrap modulo 2^64, which keeps the low 32 bits exact.
    exp = (X.astype(np.int64) @ W.astype(np.int64) + b).astype(np.uint64).astype(np.uint32).astype(np.int32)
    tX, tW, tb = (torch.from_numpy(a).cuda() for a in (X, W, b))
    try:
        for variant in (-1, 0, 3):
            set_i8_variant(variant)
            for epi, want in ((_native.EPI_BIAS, exp), (_native.EPI_BIAS_RELU, np.maximum(exp, 0))):
                Y = torch.full((M, N), 7, dtype=torch.int32, device="cuda")
                dense_launch(tX, tW, tb, Y, epi)
                torch.cuda.synchronize()
                plan = _native.last_plan()
                assert ("tile=64x64" if variant < 0 else f"variant={variant}") in plan, plan
                assert np.array_equal(Y.cpu().numpy(), want), (kind, plan)
    finally:
        set_i8_variant(-1)


def test_more_chunks_than_a_counts_register():
    """K of 4 * 64 chunks and some: a wave of the 64x64 tile reads its counts
    in two registers full; the second half holds the wide values."""
    import torch
    from mlir_edsl_hip.device import dense_launch
    M, K, N = 70, 64 * 4 * 64 + 200, 40
    rng = np.random.default_rng(5)
    X, W = rng.integers(-100, 100, (M, K)), rng.integers(-100, 100, (K, N))
    X[:, K - 150:] *= 1000
    W[K - 300:K - 200] *= 20000
    X, W = X.astype(np.int32), W.astype(np.int32)
    exp = (X.astype(np.int64) @ W.astype(np.int64)).astype(np.uint64).astype(np.uint32).astype(np.int32)
    Y = torch.full((M, N), 7, dtype=torch.int32, device="cuda")
    dense_launch(torch.from_numpy(X).cuda(), torch.from_numpy(W).cuda(), None, Y, _native.EPI_NONE)
    torch.cuda.synchronize()
    assert "tile=64x64" in _native.last_plan()
    assert np.array_equal(Y.cpu().numpy(), exp)
