"""GPU parity of the gemm layout's tiles (MFMA, many activation rows): one and
two 64-row activation tiles per workgroup at the edges of both, with special
values in the weights and in the activations, which send a tile through its
second, hi-term pass."""
import numpy as np
import pytest

import oracle
from demonic_amd import workloads as W
from parity import check_or_bound
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
