"""GPU parity of the f32 group kernels at 5 and more activation rows: W read
once per 8 rows (4 where a lane holds 3 or 4 windows), the rows split over
the groups of one launch."""
import numpy as np
import pytest

import oracle
from parity import check, check_bound
from test_gpu_f32 import edge

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [5, 8, 9, 17, 40])
@pytest.mark.parametrize("n,k", [(33, 4), (300, 2048), (17, 2052), (40, 4096), (16, 4100), (35, 7168), (18, 7172),
                                 (50, 14336)])
def test_group_rows_f32(hip, n, k, m, monkeypatch):
    monkeypatch.setenv("DMC_HIP_F32_GROUP_M", "2")
    rng = np.random.default_rng(n + k + m)
    x = edge(rng.standard_normal((m, k)).astype(np.float32), rng)
    w = edge(rng.standard_normal((n, k)).astype(np.float32), rng)
    w[5] = 0
    x[m - 1], w[6, : k // 2], w[6, k // 2:] = np.float32(1e-30), np.float32(1e-30), np.float32(-1e-30)
    y_ref = oracle.matmul_f32(x, np.ascontiguousarray(w.T))
    with hip.DeviceBuffer.from_numpy(x) as dx, hip.DeviceBuffer.from_numpy(w) as dw, hip.DeviceBuffer(4 * m * n) as dy:
        p = hip.plan_f32(m, k, n, x_addr=dx.addr, w_addr=dw.addr)
        most = 4 if k > 7168 else 8
        assert (p.rows_per_group, p.grid_y, p.mt) == (16, -(-m // most), -(-m // -(-m // most))), p
        hip.gemv_f32_rd(dx, dw, dy, m, k, n)
        hip.synchronize()
        y = dy.download(np.float32, (m, n))
    check(y, y_ref, what=f"f32 rows m={m} n={n} k={k}")
    check_bound(y[m - 1], y_ref[m - 1], x[m - 1], w, what="the tiny row")
    if m <= 16:  # the drop-in's W @ x writes the same kernels' outputs transposed
        check(hip.matmul_f32_gpu(w, np.ascontiguousarray(x.T)), np.ascontiguousarray(y_ref.T), what="W @ x")
