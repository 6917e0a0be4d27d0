"""The small-M kernel on W rows of any alignment, with K splits that are not
powers of two (as many workgroups as fill the CUs once or twice)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import assert_f32_parity
from mlir_edsl_hip import _native

pytestmark = pytest.mark.gpu


# W's rows start on 128-byte lines (streamed loads), on 16-byte ones, or on
# neither (both cached, column blocks mapped by XCD: total workgroups that 8
# does and does not divide); N that ends inside a lane's four columns, at its
# end, or one column into a block.
@pytest.mark.parametrize("M, K, N, pad, off", [
    (16, 1040, 4096, 0, 0),    # 128-byte rows
    (16, 1040, 4096, 4, 4),    # 16-byte rows
    (16, 1040, 4097, 0, 0), (3, 1040, 4098, 0, 1), (20, 1040, 4099, 1, 3), (48, 1040, 4097, 0, 2),
    (64, 1040, 8191, 0, 0), (33, 1029, 1000, 1, 0), (1, 1029, 5, 0, 0), (17, 1029, 3, 0, 0),
])
def test_rows_of_any_alignment(M, K, N, pad, off):
    import torch
    from mlir_edsl_hip.device import dense_launch
    rng = np.random.default_rng(M + 3 * K + 7 * N + pad + off)
    X = rng.standard_normal((M, K), dtype=np.float32)
    W = (rng.standard_normal((K, N), dtype=np.float32) / np.float32(np.sqrt(K))).astype(np.float32)
    b = rng.uniform(-0.1, 0.1, N).astype(np.float32)
    buf = torch.full((K * (N + pad) + off,), float("nan"), device="cuda")
    tW = buf[off:].view(K, N + pad)[:, :N]
    tW.copy_(torch.from_numpy(W))
    ybuf = torch.full((M * (N + pad) + off + 8,), 7.0, device="cuda")  # nothing past the rows is written
    tY = ybuf[off:off + M * (N + pad)].view(M, N + pad)[:, :N]
    dense_launch(torch.from_numpy(X).cuda(), tW, torch.from_numpy(b).cuda(), tY, _native.EPI_BIAS_RELU)
    torch.cuda.synchronize()
    assert _native.last_plan().startswith("gemv_f32"), _native.last_plan()
    assert_f32_parity(tY.cpu().numpy(), oracle.dense_f32_chains(X, W, b, "relu"), K)
    assert (ybuf[:off] == 7.0).all() and (ybuf[off + M * (N + pad):] == 7.0).all()
    if pad:
        gap = ybuf[off:off + M * (N + pad)].view(M, N + pad)[:, N:]
        assert (gap == 7.0).all()


# Wide N, where a split that fills the rounds of the CUs would need more than
# the 16 MiB of partials that the allocation-free launch has: the automatic
# plan, the same for both entries, stays within them.
@pytest.mark.parametrize("M, K, N", [(48, 2048, 33024), (64, 1030, 40001), (16, 1024, 50257), (64, 2048, 8320)])
def test_automatic_splits_fit_the_fixed_scratch(M, K, N):
    import torch
    g = torch.Generator(device="cuda").manual_seed(N)
    X = torch.randn(M, K, device="cuda", generator=g)
    W = torch.randn(K, N, device="cuda", generator=g)
    b = torch.randn(N, device="cuda", generator=g)
    Y, Z = torch.zeros(M, N, device="cuda"), torch.zeros(M, N, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    L = _native.lib()
    for fn, out in ((L.edsl_hip_dense_f32_launch, Y), (L.edsl_hip_dense_f32_launch_noalloc, Z)):
        rc = fn(X.data_ptr(), K, W.data_ptr(), N, b.data_ptr(), out.data_ptr(), N, M, N, K, _native.EPI_BIAS, 0.0,
                stream)
        assert rc == 0, _native.last_error()
    torch.cuda.synchronize()
    assert torch.equal(Y, Z)
    assert torch.allclose(Y, torch.addmm(b, X, W), rtol=0, atol=1e-4 * K ** 0.5)


# Three and four row blocks on plans with fewer slices of K than the workgroups of
# powers of two had: one set of accumulators was 1.85e-7, 2.04e-7 and 1.54e-7 from
# float64 there, slices as many as before 1.59e-7, 1.77e-7 and 1.47e-7.
@pytest.mark.parametrize("M, K, N, bound", [(37, 4232, 1760, 1.65e-7), (39, 4735, 1596, 1.85e-7), (42, 2529, 1295, 1.5e-7)])
def test_fewer_slices_keep_their_precision(M, K, N, bound):
    import torch
    from mlir_edsl_hip.device import dense_launch
    g = torch.Generator(device="cuda").manual_seed(K)
    X = torch.randn(M, K, device="cuda", generator=g)
    W = torch.randn(K, N, device="cuda", generator=g)
    Y = torch.empty(M, N, device="cuda")
    dense_launch(X, W, None, Y, _native.EPI_NONE)
    exact = X.double() @ W.double()
    assert _native.last_plan().startswith("gemv_f32 mb=3 "), _native.last_plan()
    assert ((Y.double() - exact).norm() / exact.norm()).item() <= bound


# A K tail needs two splits, whose partials do not fit from N = 32769 at M = 64
# on: the allocation-free launch refuses such a layer where the small-M kernel
# has it, and takes it where a tile does.
@pytest.mark.parametrize("M, K, N, fits", [(64, 2049, 40001, False), (64, 4104, 40000, False), (64, 2049, 32765, True),
                                           (64, 2047, 40001, True), (64, 4088, 40000, True)])
def test_k_tails_and_the_fixed_scratch(M, K, N, fits):
    import torch
    g = torch.Generator(device="cuda").manual_seed(N)
    X = torch.randn(M, K, device="cuda", generator=g)
    W = torch.randn(K, N, device="cuda", generator=g)
    Y = torch.zeros(M, N, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    args = (X.data_ptr(), K, W.data_ptr(), N, None, Y.data_ptr(), N, M, N, K, _native.EPI_NONE, 0.0, stream)
    rc = _native.lib().edsl_hip_dense_f32_launch_noalloc(*args)
    torch.cuda.synchronize()
    if fits:
        assert rc == 0, _native.last_error()
    else:
        assert rc == -5 and f"needs {512 * (N + 3 & ~3)} bytes" in str(_native.last_error()), _native.last_error()
        assert not Y.any()
        assert _native.lib().edsl_hip_dense_f32_launch(*args) == 0, _native.last_error()
        torch.cuda.synchronize()
    assert torch.allclose(Y, X @ W, rtol=0, atol=1e-4 * K ** 0.5)
