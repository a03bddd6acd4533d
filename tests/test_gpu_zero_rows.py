"""What a clearing run (tsp_plan_run with zero_c) clears: the split row-blocks
and, once the caller has C, the rows no tile covers; everything else is
stored whole."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_spmm import assert_close, random_b, reference

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(tsp):
    if not tsp.device_available():
        pytest.fail("no gfx950 device: GPU tests need an MI355X")
    return tsp


def matrix(tsp, rng, rows, cols, prec, hub):
    """Runs of empty rows longer than a row-block, and `hub` long rows."""
    lens = rng.integers(0, 12, rows)
    lens[rng.random(rows) < 0.3] = 0
    for r0 in range(64, rows, 192):
        lens[r0:r0 + 96] = 0
    if hub:
        lens[rng.choice(rows, hub, replace=False)] = cols // 2
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(cols, int(l), replace=False)) for l in lens]).astype(np.int32)
    v = rng.uniform(-1, 1, rp[-1]).astype(np.float32)
    return tsp.Csr(rows, cols, rp, ci, v.astype(np.float16).view(np.uint16) if prec == 0 else v, prec)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("rows,hub", [(1, 0), (8, 1), (517, 0), (517, 3), (1000, 5)])
def test_clearing_run_over_garbage(gpu, orc, prec, rows, hub):
    tsp = gpu
    hip, host = tsp.load()
    rng = np.random.default_rng(rows * 10 + hub + prec)
    A = matrix(tsp, rng, rows, 700, prec, hub)
    if prec == 1:
        A.val = orc.round_tf32_array(A.val)
    B, cbp = random_b(tsp, rng, A.cols, 96, prec)
    if prec == 1:
        B = orc.round_tf32_array(B)
    Cref, Cabs = reference(orc, A, B, 96)
    for gamma, delta in ((2.0, 1.5), (5.0, 3.0)):
        plan = tsp.Plan.from_csr(tsp.matrix_split(A, gamma, delta), A.rows, A.cols, cbp, prec, B)
        try:
            for th in (4, 1 << 20, 4):              # split row-blocks, none, split again
                plan.set_th(th, th, th)
                for rep in range(3):                # the plan's own C
                    plan.run()
                    assert_close(plan.download_c()[:, :96], Cref, Cabs, prec, f"th={th} rep={rep}")
            dc = C.c_void_p()
            assert host.tsp_plan_device_c(plan.p, C.byref(dc)) == 0
            for th in (4, 1 << 20):
                plan.set_th(th, th, th)
                for fill in (0xFF, 0x7F):           # NaN, a large value
                    # (the null stream is not ordered with the plan's)
                    assert hip.tsp_memset(dc, fill, A.rows * cbp * 4) == 0 and hip.tsp_device_sync() == 0
                    plan.run()
                    Cg = plan.download_c()
                    assert_close(Cg[:, :96], Cref, Cabs, prec, f"shared th={th} fill={fill}")
                    assert (Cg[:, 96:] == 0).all()
        finally:
            plan.close()


def test_row_blocks_off_the_grid(gpu, orc):
    """Sub-CSRs whose row-blocks do not start at multiples of 8."""
    tsp = gpu
    hip, host = tsp.load()
    rng = np.random.default_rng(5)
    A = matrix(tsp, rng, 40, 300, 0, 1)
    B, cbp = random_b(tsp, rng, A.cols, 32, 0)
    Cref, Cabs = reference(orc, A, B, 32)
    subs = tsp.matrix_split(A, 5.0, 3.0)
    shift = 4
    for s in subs:
        s.orig_row = s.orig_row + shift
    plan = tsp.Plan.from_csr(subs, A.rows + shift, A.cols, cbp, 0, B)
    try:
        plan.set_th(4, 4, 4)
        dc = C.c_void_p()
        assert host.tsp_plan_device_c(plan.p, C.byref(dc)) == 0
        for _ in range(2):
            assert hip.tsp_memset(dc, 0xFF, (A.rows + shift) * cbp * 4) == 0 and hip.tsp_device_sync() == 0
            plan.run()
            Cg = plan.download_c()
            assert (Cg[:shift] == 0).all()
            assert_close(Cg[shift:], Cref, Cabs, 0, "shifted rows")
    finally:
        plan.close()
