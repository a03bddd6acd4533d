"""Launches that leave the tasks per wave to the library add up the sums of a
split row-block inside a workgroup: every class, format and precision, chunk
counts that group four tasks, two tasks or none, task counts that do not fill
the last workgroup, row-blocks whose pieces straddle workgroups, empty split
tasks between pieces, and pieces in any order."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_spmm import assert_close, random_b, random_matrix, reference

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(tsp):
    if not tsp.device_available():
        pytest.fail("no gfx950 device: GPU tests need an MI355X")
    return tsp


def pack(arr, bm, bn, prec):
    """Packed values and offsets of dense canonical tiles."""
    n = bm * bn
    bits = np.unpackbits(arr["bitmap"].view(np.uint8), bitorder="little").reshape(-1, arr["bitmap"].size * 64
                                                                                   // max(len(arr["dense"]) // n, 1))
    bits = bits[:, :n].astype(bool)
    dense = arr["dense"].reshape(-1, n)
    vptr = np.concatenate([[0], np.cumsum(bits.sum(1))]).astype(np.int32)
    return np.concatenate([dense[bits], np.zeros(4, dense.dtype)]), vptr


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("bm,packed", [(8, False), (8, True), (16, False), (16, True), (64, False)])
@pytest.mark.parametrize("colB", [32, 64, 128, 192, 256, 512])
def test_sums_in_group(gpu, orc, prec, bm, packed, colB):
    tsp = gpu
    hip, _ = tsp.load()
    rng = np.random.default_rng(1000 * bm + colB + prec)
    # (64-row tiles add up in the workgroup from 4096 waves on)
    rows_n = 1100 if bm == 64 else 203
    A = random_matrix(tsp, rng, rows_n, 1500, 90 if bm == 64 else 30, prec, heavy_rows=6)
    if prec == 1:
        A.val = orc.round_tf32_array(A.val)
    B, cbp = random_b(tsp, rng, A.cols, colB, prec)
    if prec == 1:
        B = orc.round_tf32_array(B)
    Cref, Cabs = reference(orc, A, B, colB)
    sub = tsp.Csr(A.rows, A.cols, A.rowptr, A.colidx, A.val, prec)
    sub.orig_row = np.arange(A.rows, dtype=np.int32)
    t = tsp.tile_create(sub, A.cols, bm, prec)
    arr = t.arrays()
    bn = t.bn
    rows, cs = tsp.pretreatment(t, 1 if bm == 64 else 2)
    assert (rows >> 31).sum() > 20
    schedules = [(rows, cs, np.arange(t.tilenum))]
    # an empty piece after every third task
    r2, c2 = [], [0]
    for k in range(len(rows)):
        r2.append(rows[k]); c2.append(cs[k + 1])
        if k % 3 == 0:
            r2.append(rows[k]); c2.append(cs[k + 1])
    schedules.append((np.array(r2, np.uint32), np.array(c2, np.int32), np.arange(t.tilenum)))
    # the tasks in any order, their tiles with them
    order = rng.permutation(len(rows))
    perm = np.concatenate([np.arange(cs[k], cs[k + 1]) for k in order])
    c3 = np.concatenate([[0], np.cumsum(np.diff(cs)[order])]).astype(np.int32)
    schedules.append((rows[order], c3, perm))
    pval, vptr = pack(arr, bm, bn, prec) if packed else (None, None)
    for si, (rw, c, perm) in enumerate(schedules):
        bufs = {}

        def up(name, a):
            a = np.ascontiguousarray(a)
            p = C.c_void_p()
            assert hip.tsp_malloc(C.byref(p), max(a.nbytes, 16)) == 0
            assert hip.tsp_memcpy_h2d(p, a.ctypes.data_as(C.c_void_p), a.nbytes) == 0
            bufs[name] = p

        try:
            up("col", arr["tile_colidx"].reshape(-1, bn)[perm]); up("rows", rw); up("cs", c); up("B", B)
            up("C", np.zeros((A.rows, cbp), np.float32))
            if packed:
                a2 = {"bitmap": arr["bitmap"].reshape(t.tilenum, -1)[perm].reshape(-1),
                      "dense": arr["dense"].reshape(t.tilenum, -1)[perm].reshape(-1)}
                pval, vptr = pack(a2, bm, bn, prec)
                up("val", pval); up("vptr", vptr); up("bmp", a2["bitmap"])
                st = hip.tsp_spmm_launch_packed(bm, prec, len(rw), cbp, bufs["val"], bufs["bmp"], bufs["vptr"],
                                                bufs["rows"], bufs["cs"], bufs["B"], bufs["C"], bufs["col"], A.rows,
                                                None, 0, 0, 0, 0)
            else:
                up("val", arr["dense"].reshape(t.tilenum, -1)[perm])
                st = hip.tsp_spmm_launch(bm, prec, len(rw), cbp, bufs["val"], bufs["rows"], bufs["cs"], bufs["B"],
                                         bufs["C"], bufs["col"], A.rows, None)
            assert st == 0 and hip.tsp_device_sync() == 0
            out = np.zeros((A.rows, cbp), np.float32)
            assert hip.tsp_memcpy_d2h(out.ctypes.data_as(C.c_void_p), bufs["C"], out.nbytes) == 0
        finally:
            for p in bufs.values():
                hip.tsp_free(p)
        assert_close(out[:, :colB], Cref, Cabs, prec, f"bm={bm} packed={packed} colB={colB} schedule {si}")
