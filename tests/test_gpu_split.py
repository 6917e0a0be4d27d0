"""fp32 layers on the bf16 matrix cores (gemm_f32_split.hip): the three tiles
at sizes that divide and do not divide them (M, N and K remainders, rows off
16-byte alignment, NaN in every padding element), every epilogue, and the
values that do not split exactly -- denormal, near the largest float, infinite,
NaN -- which the tile that holds them recomputes on fp32 MFMA."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import assert_f32_parity
from mlir_edsl_hip import _native

pytestmark = pytest.mark.gpu

# (M, K, N): the split tile the planner takes
SHAPES = [((2048, 512, 4096), "256x128x16"), ((2500, 1030, 2496), "256x128x16"), ((4001, 1007, 4001), "256x128x16"),
          ((2048, 1024, 2048), "128x128x32_w8"), ((2001, 543, 2003), "128x128x32_w8"),
          ((4096, 256, 4096), "128x128x16"), ((4000, 271, 4001), "128x128x16")]

_EPIS = [(_native.EPI_NONE, False, "none"), (_native.EPI_BIAS, True, "none"), (_native.EPI_RELU, False, "relu"),
         (_native.EPI_BIAS_RELU, True, "relu"), (_native.EPI_LEAKY, False, "leaky"),
         (_native.EPI_BIAS_LEAKY, True, "leaky"), (_native.EPI_IF_RELU, False, "if_relu"),
         (_native.EPI_BIAS_IF_RELU, True, "if_relu")]


def _inputs(M, K, N, seed):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((M, K), dtype=np.float32)
    W = (rng.standard_normal((K, N), dtype=np.float32) / np.float32(np.sqrt(K))).astype(np.float32)
    return X, W, rng.uniform(-0.1, 0.1, N).astype(np.float32)


def _view(torch, a, pad, off, fill):
    rows, cols = a.shape
    buf = torch.full(((rows + 1) * (cols + pad) + off,), fill, device="cuda")
    v = buf[off:off + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]
    v.copy_(torch.from_numpy(a))
    return v, buf


@pytest.mark.parametrize("shape, tile", SHAPES, ids=["x".join(map(str, s)) for s, _ in SHAPES])
def test_split_tiles(shape, tile):
    import torch
    from mlir_edsl_hip.device import dense_launch
    M, K, N = shape
    X, W, b = _inputs(M, K, N, M + K + N)
    tb = torch.from_numpy(b).cuda()
    ref = oracle.dense_f32_chains(X, W, b, "relu")
    for pad, off in ((0, 0), (3, 1)):
        tX, tW = (_view(torch, a, pad, off, float("nan"))[0] for a in (X, W))
        tY, ybuf = _view(torch, np.full((M, N), 5.0, np.float32), pad, off, 7.0)
        dense_launch(tX, tW, tb, tY, _native.EPI_BIAS_RELU)
        torch.cuda.synchronize()
        if pad == 0:
            assert f"split=bf16x6 tile={tile} " in _native.last_plan(), _native.last_plan()
        got = tY.cpu().numpy()
        assert_f32_parity(got, ref, K)
        tY.fill_(7.0)
        assert (ybuf == 7.0).all()  # nothing else was written
    # No larger error than the fp32 MFMA tile it replaces.
    exact = torch.relu(tX.double() @ tW.double() + tb.double()).cpu().numpy()
    norm = np.linalg.norm(exact)
    err = np.linalg.norm(got - exact) / norm
    assert err <= 1.25e-7 * np.sqrt(K / 256), err  # one fp32 chain: 2.9e-7 at K = 256, growing with sqrt(K)


@pytest.mark.parametrize("epi, has_bias, act", _EPIS)
def test_split_epilogues(epi, has_bias, act):
    import torch
    from mlir_edsl_hip.device import dense_launch
    M, K, N = 2001, 512, 2003
    X, W, b = _inputs(M, K, N, epi)
    X[5] = 0.0  # sums of +0: -0 in the bias column gives +0
    b[7], b[8] = -0.0, np.nan
    tX, tW, tb = (torch.from_numpy(a).cuda() for a in (X, W, b))
    Y = torch.full((M, N), 7.0, device="cuda")
    dense_launch(tX, tW, tb if has_bias else None, Y, epi, 0.125)
    torch.cuda.synchronize()
    assert "split=bf16x6" in _native.last_plan()
    got = Y.cpu().numpy()
    assert_f32_parity(got, oracle.dense_f32_chains(X, W, b if has_bias else None, act, 0.125), K)
    assert not np.signbit(got[5][got[5] == 0]).any()


# Operands with few terms a sum, where fp32 rounds once a term: one nonzero value
# a row or a column, n of them in different steps, rows of two and full columns
# that meet at one k, and half of all zero on one or both sides.
@pytest.mark.parametrize("what", ["one_a_row", "one_a_column", "two_a_row", "eight_a_row", "thirty_a_row",
                                  "one_in_common", "relu", "relu_both"])
@pytest.mark.parametrize("M, K, N", [(2500, 1030, 2496), (2001, 543, 2003), (4000, 271, 4001)],
                         ids=["256x128", "128x128_w8", "128x128"])
def test_sparse_operands_lose_no_precision(M, K, N, what):
    import torch
    from mlir_edsl_hip.device import dense_launch, set_f32_config
    g = torch.Generator(device="cuda").manual_seed(K)
    X = torch.randn(M, K, device="cuda", generator=g)
    W = torch.randn(K, N, device="cuda", generator=g)
    r, c = torch.arange(M, device="cuda"), torch.arange(N, device="cuda")
    if what == "one_a_column":
        d = torch.zeros_like(W)
        d[c % K, c] = W[0]
        W = d
    elif what.startswith("relu"):
        X.relu_()
        if what == "relu_both":
            W.relu_()
    elif what == "one_in_common":
        X[:, 2:] = 0.0
        W[1] = 0.0
    else:
        d = torch.zeros_like(X)
        n = {"one_a_row": 1, "two_a_row": 2, "eight_a_row": 8, "thirty_a_row": 30}[what]
        step = K // 30
        for j in range(n):  # rows start all over K
            d[r, (r + j * step) % K] = X[:, j]
        X = d
    exact = X.double() @ W.double()
    terms = exact != 0
    anyshape = _native.f32_config_names().index("f32_128x128x32_mfma16_anyshape")

    def errors(cfg):
        y = torch.full((M, N), 7.0, device="cuda")
        set_f32_config(cfg)
        try:
            dense_launch(X, W, None, y, _native.EPI_NONE)
            torch.cuda.synchronize()
        finally:
            set_f32_config(-1)
        assert ("split=bf16x6" in _native.last_plan()) == (cfg < 0)
        d = y.double() - exact
        assert (d[~terms] == 0).all()
        return (d.norm() / exact.norm()).item(), (d[terms] / exact[terms]).abs().max().item()

    (rel, largest), (rel32, _) = errors(-1), errors(anyshape)
    # Eight products are within 2^-33 of the exact one and the seven small ones, at
    # most 2^-7 of it, round at 2^-24 of themselves: 0.4 % on top of one rounding.
    assert rel <= rel32 * 1.004, (rel, rel32)
    if what.startswith("one"):
        assert largest <= 2.0**-24 * (1 + 7 * 2.0**-7), largest


@pytest.mark.parametrize("M, K, N", [(2048, 512, 4096), (2001, 543, 2003), (4096, 256, 4096)],
                         ids=["256x128", "128x128_w8", "128x128"])
def test_values_that_do_not_split(M, K, N):
    """Denormal, huge, infinite and NaN operands give what the fp32 tiles
    give; the tiles that hold none of them keep their bits."""
    import torch
    from mlir_edsl_hip.device import dense_launch, set_f32_config
    X, W, b = _inputs(M, K, N, 3 * M + K)
    tX, tW, tb = (torch.from_numpy(a).cuda() for a in (X, W, b))

    def run(x, w, cfg=-1):
        y = torch.full((M, N), 7.0, device="cuda")
        set_f32_config(cfg)
        try:
            dense_launch(x, w, tb, y, _native.EPI_BIAS)
            torch.cuda.synchronize()
        finally:
            set_f32_config(-1)
        assert ("split=bf16x6" in _native.last_plan()) == (cfg < 0)
        return y

    anyshape = _native.f32_config_names().index("f32_128x128x32_mfma16_anyshape")
    clean = run(tX, tW)
    for value in (1e-40, -3.0e-38 / 2**12, 3.4e38, float("inf"), float("nan")):
        x, w = tX.clone(), tW.clone()
        x[M - 1, K - 1] = value
        w[1, 3] = value
        got, want = run(x, w), run(x, w, anyshape)
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
        ok = torch.isfinite(want)
        # both sum the same fp32 products; 1e-4 sqrt(K) is the parity bar at unit scale
        scale = want.abs().clamp_min(1.0)
        assert (((got - want).abs() / scale)[ok] <= 1e-4 * K**0.5).all()
        # Tiles of other rows and columns are untouched: 256 rows and columns from the edges.
        assert torch.equal(got[:M - 512, 512:], clean[:M - 512, 512:])


# What the split cannot hold, where it shows in the result: values below 2^-109,
# whose last remainder bf16 cuts (the first three: without the recomputation
# the first and the third are off by 1e-5 and more), and products whose parts
# underflow.
@pytest.mark.parametrize("xs, ws", [(-124, 100), (-110, 60), (-118, 0), (-62, -62), (-50, -50), (-75, -60)])
@pytest.mark.parametrize("M, K, N", [(2048, 512, 4096), (2001, 543, 2003), (4000, 271, 4001)],
                         ids=["256x128", "128x128_w8", "128x128"])
def test_tiny_operands_keep_fp32_precision(M, K, N, xs, ws):
    import torch
    from mlir_edsl_hip.device import dense_launch, set_f32_config
    X, W, _ = _inputs(M, K, N, K)
    X, W = np.ldexp(X, xs), np.ldexp(W * np.float32(np.sqrt(K)), ws)
    tX, tW = torch.from_numpy(X).cuda(), torch.from_numpy(W).cuda()
    exact = tX.double() @ tW.double()
    rel = []
    for cfg in (-1, _native.f32_config_names().index("f32_128x128x32_mfma16_anyshape")):
        y = torch.full((M, N), 7.0, device="cuda")
        set_f32_config(cfg)
        try:
            dense_launch(tX, tW, None, y, _native.EPI_NONE)
            torch.cuda.synchronize()
        finally:
            set_f32_config(-1)
        rel.append(((y.double() - exact).norm() / exact.norm()).item())
    # Both sum the same fp32 products where the tile is recomputed, in another
    # order of K steps; 2^-26 a sum is what the test of the sums lets pass.
    assert rel[0] <= 1.05 * rel[1] + 2.0**-26, rel


@pytest.mark.parametrize("M, K, N", [(2048, 512, 4096), (2001, 543, 2003), (4000, 271, 4001)],
                         ids=["256x128", "128x128_w8", "128x128"])
def test_denormals_alone_and_among_other_values(M, K, N):
    """A row whose only value is a denormal gives correctly rounded products, a
    row of zeros zeros, and ordinary rows keep their precision."""
    import torch
    from mlir_edsl_hip.device import dense_launch
    X, W, _ = _inputs(M, K, N, K + 1)
    X[:, K // 2] = 1e-40
    X[7], X[M - 1], X[11] = 0.0, 0.0, 0.0
    X[7, K - 1], X[M - 1, 3] = 1.2345e-39, -3e-41
    W[K - 1] *= np.float32(2.0**80)
    W[K - 2, 5] = -1e-42
    W[:, 9] = 0.0
    Y = torch.full((M, N), 7.0, device="cuda")
    dense_launch(torch.from_numpy(X).cuda(), torch.from_numpy(W).cuda(), None, Y, _native.EPI_NONE)
    torch.cuda.synchronize()
    assert "split=bf16x6" in _native.last_plan()
    got = Y.cpu().numpy()
    assert np.array_equal(got[7], X[7, K - 1] * W[K - 1])
    assert np.array_equal(got[M - 1], X[M - 1, 3] * W[3])
    assert (got[11] == 0).all() and (got[:, 9] == 0).all()
    rows = np.delete(np.arange(M), [7, M - 1, 11])
    exact = X[rows].astype(np.float64) @ W.astype(np.float64)
    err = np.linalg.norm(got[rows] - exact) / np.linalg.norm(exact)
    assert err <= 1.25e-7 * np.sqrt(K / 256), err
