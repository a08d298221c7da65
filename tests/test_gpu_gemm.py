"""GPU parity of the gemm layout's tiles (MFMA, many activation rows): one and
two 64-row activation tiles per workgroup at the edges of both, special values
in the weights and in the activations (which send a tile through its second,
hi-term pass), and outputs whose exact zero sends one wave through the
reference chain."""
import pathlib
import subprocess
import sys

import numpy as np
import pytest

import oracle
from demonic_amd import workloads as W
from parity import check, check_bound, check_classes, check_or_bound
from test_gpu_parity import case, run_cs_dev, run_rd

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


ROUTES = [  # (environment, K, W stored [k,n])
    pytest.param({"DMC_HIP_RD_MFMA_KIND": "8", "DMC_HIP_GEMM_MAX_SLICES": "1"}, 3008, False, id="gemm"),
    pytest.param({"DMC_HIP_RD_MFMA_KIND": "8", "DMC_HIP_GEMM_MAX_SLICES": "4"}, 3008, False, id="gemm-slices"),
    pytest.param({"DMC_HIP_RD_MFMA_KIND": "7"}, 3008, False, id="rows16"),
    pytest.param({"DMC_HIP_RD_MFMA_KIND": "6"}, 3008, False, id="wide"),
    pytest.param({"DMC_HIP_RD_GEMM_ROWS": "2", "DMC_HIP_GEMM_MAX_SLICES": "1"}, 3001, False, id="rows"),
    pytest.param({"DMC_HIP_RD_GEMM_ROWS": "2"}, 3001, False, id="rows-slices"),
    pytest.param({"DMC_HIP_CS_GEMM": "2", "DMC_HIP_GEMM_MAX_SLICES": "1"}, 3001, True, id="columns"),
    pytest.param({"DMC_HIP_CS_GEMM": "2"}, 3001, True, id="columns-slices"),
]


def on_route(hip, x, w, columns):
    return run_cs_dev(hip, x, w) if columns else run_rd(hip, x, w)


@pytest.mark.parametrize("env,k,columns", ROUTES)
def test_zero_sums_take_the_reference_chain(hip, env, k, columns, monkeypatch):
    """Sums that come out exactly zero, alone in 80 x 300 and many in one wave,
    K long enough for several rounds of the wave's chain:
    - full cancellation of ordinary products (the reference: +0);
    - products that all underflow, positive and then, past k = 2000, negative,
      in a row that is not all tiny since its largest element meets a weight
      of 0 (the reference chain: -0);
    - products that cancel after the chain has overflowed (the reference: inf)."""
    m, n = 80, 300
    for name, value in env.items():
        monkeypatch.setenv(name, value)
    x, w = case(m, k, n, seed=5, scale=0.02)
    x[:, :4] = 0.25
    x[70] = 1
    half = k // 2
    w[200] = 0
    w[200, :half], w[200, half:2 * half] = 0x3F80, 0xBF80
    x[30] = np.float32(1e-38)
    x[30, 0], x[30, 2000:] = 1, np.float32(-1e-38)
    w[100], w[100, 0] = 0x0001, 0
    w[240:260], w[240:260, 0] = 0x0001, 0
    w[50] = 0
    w[50, 0:2], w[50, 2:4] = 0x7F62, 0xFF62  # 3e38 twice, -3e38 twice
    with np.errstate(over="ignore"):
        y_ref = oracle.matmul_bf16_t(x, w)
    assert y_ref[70, 200] == 0 and np.isposinf(y_ref[70, 50])
    assert all(y_ref[30, c] == 0 and np.signbit(y_ref[30, c]) for c in [100, *range(240, 260)])
    y = on_route(hip, x, w, columns)
    for r, c in ((70, 200), (70, 50), (30, 100), (30, 240), (30, 259)):
        assert y[r, c].view(np.uint32) == y_ref[r, c].view(np.uint32), (r, c, y[r, c], y_ref[r, c])
    check_or_bound(y, y_ref, x, W.bf16_to_f32(w), what="zero sums")


@pytest.mark.parametrize("env,k,columns", ROUTES[4:])
def test_small_elements_beside_large_ones_keep_their_bits(hip, env, k, columns, monkeypatch):
    """Activation elements down to the least subnormal in rows whose largest
    element meets a weight of 0, and small elements against large weights: f32
    keeps all 24 bits of them (three bf16 terms alone lose those under 2^-133)."""
    m, n = 40, 300
    for name, value in env.items():
        monkeypatch.setenv(name, value)
    rng = np.random.default_rng(11)
    x, w = case(m, k, n, seed=6, scale=0.02)
    for r, top in ((3, -112), (17, -125), (33, -136)):
        x[r] = np.ldexp(rng.standard_normal(k), top).astype(np.float32)
        x[r, 5] = 1
    x[34], x[34, 0], x[34, 1] = 0, 1, np.ldexp(np.float32(1), -140)
    x[35, 9], x[36, 2] = np.inf, np.nan  # whole rows that are not finite, in the same tiles
    w[::3, 5] = 0
    w[::3, 6:] = W.bf16_rne(np.ldexp(rng.standard_normal((n + 2) // 3 * (k - 6)), 60).astype(np.float32)).reshape(-1, k - 6)
    w[7], w[7, 0], w[7, 1] = 0, 0x2180, 0x7F00  # 2^-60 and 2^127: 2^-13 with row 34
    w[8, 3] = 0x7F80
    y_ref = oracle.matmul_bf16_t(x, w)
    assert abs(y_ref[34, 7] - 2.0 ** -13) < 1e-9
    y = on_route(hip, x, w, columns)
    wf = W.bf16_to_f32(w)
    check_classes(y, y_ref, "mixed rows")
    fin = np.all(np.isfinite(wf), axis=1)
    for r in np.flatnonzero(np.all(np.isfinite(x), axis=1)):
        check_bound(y[r, fin], y_ref[r, fin], x[r], wf[fin], what=f"mixed row {r}")
    for r in (3, 17, 33):  # every product carries the same 24 bits: a few roundings away
        cols = np.flatnonzero(w[:, 5] == 0)
        want = wf[cols].astype(np.float64) @ x[r].astype(np.float64)
        size = np.abs(wf[cols].astype(np.float64)) @ np.abs(x[r].astype(np.float64))
        # 3 roundings per k-block, at most 12 per sum of blocks, 1 for the small parts
        assert np.all(np.abs(y[r, cols] - want) <= 16 * 2.0 ** -24 * size + 2.0 ** -148), r


def planted(m, k, n, seed):
    """Edge data, with special values, zero rows and underflow where they fit; (x, w [n,k], reference)."""
    x, w = case(m, k, n, seed=seed, edge=True)
    if k > 2 and n > 4 and m > 3:
        x[0, k - 1], w[1, k - 1], w[n - 1, k - 1] = np.inf, 0x7F80, 0x3F80  # in the last chunk and the last element
        x[1, 0], w[1, 0] = np.float32(1e-45), 0xFF80
        w[2, :], x[2, :] = 0, 0
        x[3, :], w[3, :] = np.float32(-1e-38), 0x0001
    return x, w, oracle.matmul_bf16_t(x, w)


@pytest.mark.parametrize("offset", [0, 2])
@pytest.mark.parametrize("m,k,n", [(5, 65, 257), (16, 4097, 300), (17, 1003, 256), (33, 4104, 255), (64, 63, 513),
                                   (65, 130, 1030), (200, 2050, 259), (7, 1, 6), (6, 8191, 130)])
def test_rows_of_any_length_and_alignment(hip, m, k, n, offset, monkeypatch):
    """The gemm layout on rows whose length is no multiple of 64, W at the end
    of its region and 0 or 2 bytes into it: nothing past K takes part (the next
    row starts with what it likes, the last row ends the region)."""
    monkeypatch.setenv("DMC_HIP_RD_GEMM_ROWS", "2")
    x, w, y_ref = planted(m, k, n, seed=m + k + n)
    buf = np.zeros(w.size + offset // 2, np.uint16)
    buf[offset // 2:] = w.reshape(-1)
    with hip.DeviceBuffer.from_numpy(buf) as dw, hip.DeviceBuffer.from_numpy(x) as dx, \
            hip.DeviceBuffer(4 * m * n) as dy:
        p = hip.plan("rd", m, k, n, x_addr=dx.addr, w_addr=dw.addr + offset)
        assert (p.slices, p.mt, p.rows_per_group) == (-8, 16 if m <= 16 else 32 if m <= 32 else 64, 256), p
        hip.gemv_rd(dx, dw.addr + offset, dy, m, k, n)
        hip.synchronize()
        y = dy.download(np.float32, (m, n))
    check_or_bound(y, y_ref, x, W.bf16_to_f32(w), f"gemm rows {m}x{k}x{n}+{offset}")


@pytest.mark.parametrize("offset", [0, 2])
@pytest.mark.parametrize("m,k,n,batch", [(17, 65, 257, 1), (33, 4097, 300, 1), (64, 63, 255, 1), (65, 1000, 513, 1),
                                         (20, 128, 64, 3), (40, 70, 131, 2), (18, 1, 9, 1), (130, 2048, 1024, 1),
                                         (16, 129, 259, 1), (5, 4097, 300, 1), (7, 64, 130, 3), (1, 66, 1, 1)])
def test_columns_on_the_gemm_layout(hip, m, k, n, batch, offset, monkeypatch):
    """W [k,n] per batch slice on the gemm layout: partial column blocks, odd N
    (the last element shares a dword with what follows the matrix), K tails,
    several slices of k and of the batch, W 0 or 2 bytes into its region."""
    monkeypatch.setenv("DMC_HIP_CS_GEMM", "2")
    zs = [planted(m, k, n, seed=m + k + n + z) for z in range(batch)]
    x = np.stack([z[0] for z in zs])
    wt = np.stack([np.ascontiguousarray(z[1].T) for z in zs])
    buf = np.zeros(wt.size + offset // 2, np.uint16)
    buf[offset // 2:] = wt.reshape(-1)
    with hip.DeviceBuffer.from_numpy(buf) as dw, hip.DeviceBuffer.from_numpy(x) as dx, \
            hip.DeviceBuffer(4 * batch * m * n) as dy:
        p = hip.plan("cs", m, k, n, batch=batch, rs=k * n, x_addr=dx.addr, w_addr=dw.addr + offset)
        assert p.rows_or_rw == -256 and p.mt == (16 if m <= 16 else 32 if m <= 32 else 64), p
        hip.gemv_cs(dx, dw.addr + offset, dy, m, k, n, batch, m * k, k * n)
        hip.synchronize()
        y = dy.download(np.float32, (batch, m, n))
    for z, (xz, wz, y_ref) in enumerate(zs):
        check_or_bound(y[z], y_ref, xz, W.bf16_to_f32(wz), f"gemm cols {m}x{k}x{n} slice {z}")


@pytest.mark.parametrize("m,k,n,batch,shared", [(20, 300, 70, 3, True), (130, 200, 300, 2, True),
                                                (130, 1000, 259, 3, False)])
def test_columns_of_padded_batches_and_a_shared_x(hip, m, k, n, batch, shared, monkeypatch):
    """Weight slices further apart than k * n, one activation matrix for all
    slices (ls = 0) or one each, and several activation tiles per slice (their
    own order of tiles over the XCDs)."""
    monkeypatch.setenv("DMC_HIP_CS_GEMM", "2")
    rng = np.random.default_rng(m + k + n)
    rs = k * n + 37
    buf = W.bf16_rne(rng.standard_normal(batch * rs).astype(np.float32))
    x = rng.standard_normal((1 if shared else batch, m, k)).astype(np.float32)
    with hip.DeviceBuffer.from_numpy(buf) as dw, hip.DeviceBuffer.from_numpy(x) as dx, \
            hip.DeviceBuffer(4 * batch * m * n) as dy:
        assert hip.plan("cs", m, k, n, batch=batch, rs=rs, x_addr=dx.addr, w_addr=dw.addr).rows_or_rw == -256
        hip.gemv_cs(dx, dw, dy, m, k, n, batch, 0 if shared else m * k, rs)
        hip.synchronize()
        y = dy.download(np.float32, (batch, m, n))
    for z in range(batch):
        wz = np.ascontiguousarray(buf[z * rs:z * rs + k * n].reshape(k, n).T)
        check(y[z], oracle.matmul_bf16_t(x[0 if shared else z], wz), what=f"slice {z}")


@pytest.mark.parametrize("m,k,n", [(33, 257, 300), (40, 4097, 600), (17, 1000, 259)])
def test_columns_that_hold_zeros(hip, m, k, n, monkeypatch):
    """Whole weight columns of zeros, unequal blocks of zeros that an activation
    row's few nonzero elements never meet, and small integers, whose sums
    cancel often: +0 as in the reference, one slice of k and several."""
    monkeypatch.setenv("DMC_HIP_CS_GEMM", "2")
    rng = np.random.default_rng(m + n)
    x, w = case(m, k, n, seed=m + k, scale=0.02)
    w[n // 3:] = 0
    w[0], w[n - 1, 0] = 0, 0x8000
    w[1, k // 2:] = 0
    x[2], x[2, k - 1] = 0, 3  # one-hot
    x[3], x[4] = 0, -0.0
    x[5:12] = rng.integers(-1, 2, (7, k))
    w[2:60] = W.bf16_rne(rng.integers(-1, 2, (58, k)).astype(np.float32))
    y_ref = oracle.matmul_bf16_t(x, w)
    assert y_ref[2, 1] == 0 and (y_ref[5:12, 2:60] == 0).any()
    for slices in ("1", "64"):
        monkeypatch.setenv("DMC_HIP_GEMM_MAX_SLICES", slices)
        check(run_cs_dev(hip, x, w), y_ref, what=f"zeros, at most {slices} slices")


FIRST_CALL_CAPTURED = """
import sys
import numpy as np
sys.path[:0] = [{root!r}, {root!r} + "/tests"]
import demonic_amd as hip, oracle
from demonic_amd import workloads as W
from parity import check
from test_gpu_parity import case
assert hip.available()
for m, k, n, columns in {shapes!r}:
    x, w = case(m, k, n, seed=m, scale=0.02)
    y_ref = oracle.matmul_bf16_t(x, w)
    with hip.DeviceBuffer.from_numpy(np.ascontiguousarray(w.T) if columns else w) as dw, \\
            hip.DeviceBuffer.from_numpy(x) as dx, hip.DeviceBuffer(4 * m * n) as dy:
        call = lambda: (hip.gemv_cs if columns else hip.gemv_rd)(dx, dw, dy, m, k, n)
        with hip.Graph() as g:
            call()
        got = []
        for rep in range(3):
            dy.upload(np.full(m * n, np.nan, np.float32))
            g.launch()
            hip.synchronize()
            got.append(dy.download(np.float32, (m, n)))
        call()
        hip.synchronize()
        eager = dy.download(np.float32, (m, n))
    check(eager, y_ref, what="eager")
    assert all(np.array_equal(y.view(np.uint32), eager.view(np.uint32)) for y in got)
    print("ok", m, k, n, flush=True)
"""


@pytest.mark.parametrize("shapes", [[(5, 4097, 3000, False), (40, 4097, 2000, False), (64, 1024, 8192, True)],
                                    [(17, 4096, 14336, True)], [(128, 4096, 2048, False)]])
def test_a_first_call_inside_a_capture(hip, shapes):
    """A process whose first GEMV is made while capturing: accepted, and bit for
    bit the eager call's result, whose split of k does not depend on what ran
    before."""
    root = str(pathlib.Path(__file__).resolve().parent.parent)
    r = subprocess.run([sys.executable, "-c", FIRST_CALL_CAPTURED.format(root=root, shapes=shapes)],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.count("ok") == len(shapes), r.stdout + r.stderr


GROWN_AFTER_CAPTURE = """
import sys
import numpy as np
sys.path[:0] = [{root!r}, {root!r} + "/tests"]
import demonic_amd as hip, oracle
from parity import check
from test_gpu_parity import case
assert hip.available()
m, k, n, m2, k2, n2 = 40, 4097, 2000, 4096, 4096, 4100
x, w = case(m, k, n, seed=1, scale=0.02)
x2, w2 = case(m2, k2, n2, seed=2, scale=0.02)
p, p2 = (hip.plan("rd", *s, x_addr=256, w_addr=256) for s in ((m, k, n), (m2, k2, n2)))
assert 0 < p.workspace_bytes <= 64 << 20 < p2.workspace_bytes, (p, p2)
y_ref = oracle.matmul_bf16_t(x, w)
bufs = dw, dx, dw2, dx2 = [hip.DeviceBuffer.from_numpy(a) for a in (w, x, w2, x2)]
with hip.DeviceBuffer(4 * m * n) as dy, hip.DeviceBuffer(4 * m2 * n2) as dy2:
    with hip.Graph() as g:
        hip.gemv_rd(dx, dw, dy, m, k, n)
    hip.gemv_rd(dx2, dw2, dy2, m2, k2, n2)
    hip.synchronize()
    rows = [0, 1, m2 - 1]
    check(dy2.download(np.float32, (m2, n2))[rows], oracle.matmul_bf16_t(x2[rows], w2), what="larger call")
    for rep in range(2):
        dy.upload(np.full(m * n, np.nan, np.float32))
        g.launch()
        hip.synchronize()
        check(dy.download(np.float32, (m, n)), y_ref, what="replay")
    g.destroy()
    hip.gemv_rd(dx, dw, dy, m, k, n)
    hip.synchronize()
    check(dy.download(np.float32, (m, n)), y_ref, what="after the graph")
print("ok", flush=True)
"""


def test_a_graph_outlives_the_workspace_it_was_captured_on(hip):
    """A later call that needs more than the 64 MiB a capture reserves: the
    outgrown workspace stays while the graph lives."""
    root = str(pathlib.Path(__file__).resolve().parent.parent)
    r = subprocess.run([sys.executable, "-c", GROWN_AFTER_CAPTURE.format(root=root)], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr
