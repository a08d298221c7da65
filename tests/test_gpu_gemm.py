"""GPU parity of the gemm layout's tiles (MFMA, many activation rows): one and
two 64-row activation tiles per workgroup at the edges of both, special values
in the weights and in the activations (which send a tile through its second,
hi-term pass), and outputs whose exact zero sends one wave through the
reference chain."""
import numpy as np
import pytest

import oracle
from demonic_amd import workloads as W
from parity import check, check_bound, check_or_bound
from test_gpu_parity import case, run_rd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fuse", [0, 2])
@pytest.mark.parametrize("pair", [1, 2])
@pytest.mark.parametrize("m,k,n", [(65, 64, 256), (128, 4096, 257), (129, 1088, 512), (300, 192, 1030)])
def test_one_and_two_activation_tiles(hip, m, k, n, pair, fuse, monkeypatch):
    monkeypatch.setenv("DMC_HIP_RD_MFMA_KIND", "8")
    monkeypatch.setenv("DMC_HIP_GEMM_PAIR", str(pair))
    monkeypatch.setenv("DMC_HIP_GEMM_FUSE", str(fuse))
    x, w = case(m, k, n, seed=m + k + n, edge=True)
    x[0, 3], x[1, 5], x[64, k - 1] = np.inf, np.nan, -np.inf  # whole rows that are not finite
    x[2, 7], w[9, 7] = np.float32(1e-45), 0x7F80              # inf against the least subnormal
    w[11, :], x[3, :] = 0, 0
    x[4, :] = np.float32(-1e-38)
    w[12, :] = 0x0001                                         # every product of row 4 underflows
    w[13, : k // 2], w[13, k // 2:] = 0x3F80, 0xBF80          # cancels exactly against a constant row
    x[5, :] = 1
    y_ref = oracle.matmul_bf16_t(x, w)
    assert y_ref[5, 13] == 0 and np.isposinf(y_ref[2, 9])
    check_or_bound(run_rd(hip, x, w), y_ref, x, W.bf16_to_f32(w), f"gemm pair={pair} fuse={fuse} {m}x{k}x{n}")


@pytest.mark.parametrize("slices", [1, 4])
def test_a_lone_cancelling_output_takes_the_chain(hip, slices, monkeypatch):
    """One output in 80 x 300 whose sum is exactly zero, K long enough for
    several rounds of the wave's chain: the reference's bits."""
    m, k, n = 80, 3008, 300
    monkeypatch.setenv("DMC_HIP_RD_MFMA_KIND", "8")
    monkeypatch.setenv("DMC_HIP_GEMM_MAX_SLICES", str(slices))
    x, w = case(m, k, n, seed=5, scale=0.02)
    x[70] = 1
    w[200, : k // 2], w[200, k // 2:] = 0x3F80, 0xBF80
    y_ref = oracle.matmul_bf16_t(x, w)
    assert y_ref[70, 200] == 0
    y = run_rd(hip, x, w)
    assert y[70, 200].view(np.uint32) == y_ref[70, 200].view(np.uint32)
    check(y, y_ref, what="lone zero")
    for r in (0, 70, 79):
        check_bound(y[r], y_ref[r], x[r], W.bf16_to_f32(w), what=f"lone zero row {r}")
