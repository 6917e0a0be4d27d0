"""The 16x16 tiles for small outputs (gemm_f32_small.hip): one group of K to
more than the eight a wave loads at once, waves without a group, K tails of
every residue class, M and N below, at and past a tile, operands off 16-byte
alignment with NaN in every padding element, and every epilogue."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import assert_f32_parity
from mlir_edsl_hip import _native

pytestmark = pytest.mark.gpu

_EPIS = [(_native.EPI_NONE, False, "none"), (_native.EPI_RELU, False, "relu"), (_native.EPI_BIAS, True, "none"),
         (_native.EPI_BIAS_RELU, True, "relu"), (_native.EPI_BIAS_LEAKY, True, "leaky"),
         (_native.EPI_BIAS_IF_RELU, True, "if_relu")]


def _view(torch, a, pad, off, fill):
    rows, cols = a.shape
    buf = torch.full(((rows + 1) * (cols + pad) + off,), fill, device="cuda")
    v = buf[off:off + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]
    v.copy_(torch.from_numpy(a))
    return v, buf


@pytest.mark.parametrize("pad, off", [(0, 0), (3, 1)])
@pytest.mark.parametrize("M, K, N", [(1, 1, 1), (16, 16, 16), (17, 15, 33), (2, 31, 5), (65, 63, 17), (70, 64, 70),
                                     (3, 448, 31), (3, 449, 31), (33, 1023, 40), (100, 1024, 300), (1, 1024, 8192)])
def test_small_tiles(M, K, N, pad, off):
    import torch
    from mlir_edsl_hip.device import dense_launch
    rng = np.random.default_rng(M + 3 * K + 7 * N + pad)
    X = rng.standard_normal((M, K), dtype=np.float32)
    W = (rng.standard_normal((K, N), dtype=np.float32) / np.float32(np.sqrt(K))).astype(np.float32)
    b = rng.uniform(-0.1, 0.1, N).astype(np.float32)
    tX, _ = _view(torch, X, pad, off, float("nan"))
    tW, _ = _view(torch, W, pad, off, float("nan"))
    tb = torch.from_numpy(b).cuda()
    for epi, has_bias, act in _EPIS:
        tY, ybuf = _view(torch, np.full((M, N), 5.0, np.float32), pad, off, 7.0)
        dense_launch(tX, tW, tb if has_bias else None, tY, epi, 0.125)
        torch.cuda.synchronize()
        plan = _native.last_plan()
        assert plan.startswith("gemm_f32_small tile=16x16 "), plan
        assert_f32_parity(tY.cpu().numpy(), oracle.dense_f32_chains(X, W, b if has_bias else None, act, 0.125), K)
        tY.fill_(7.0)
        assert (ybuf == 7.0).all()  # nothing else was written
