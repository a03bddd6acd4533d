"""The work that users of this library have it do, as cases that can be timed.

Every case is one pass through the public entry points: a step of a plan
(``Plan.run``), a launch of one row-block class on the caller's own device
buffers (``tsp_switch_v*``, ``tsp_spmm_launch_packed``), the conversion of a
CSR matrix to tiles on the device (``tsp_tile_create_device``, with
``tsp_tiles_pack_device`` for the packed format), and the whole way from a
host CSR matrix to its first product.  The matrices are the shapes of the
benchmark's five configurations and of the test fixture dc2.mtx, and generic
banded, uniform and block-sparse ones around them.
"""
import ctypes
import math
import zlib

import numpy as np
import torch

import tilespmm_amd as tsp

# Settings that a program pins after it has tuned once, as the benchmark's
# replay flags do (the tuned settings of the RMAT workloads).
PINNED_TF32 = dict(th=16, fmt=2, w=64, stages=2, tpw=4, order=1, place=1, lane=1, b3=1, hot=16 << 20)
PINNED_FP16 = dict(th=32, fmt=2, w=64, stages=2, tpw=4, order=2, place=1, lane=1, b3=0, hot=16 << 20)

MAX_ROW = 10000          # longest power-law row, as in the benchmark's generator


def _case(name, op, kind, rows, cols, mean, prec, colB, **more):
    return dict(dict(op=op, kind=kind, rows=rows, cols=cols, mean=mean, prec=prec, colB=colB), **more,
                **({"name": name} if name else {}))


def listed():
    return [
        # the smallest repeated product (an iterative solver's inner step, a
        # small graph): bound by launches
        _case("step_uniform_small", "step", "uniform", 4096, 4096, 8, "fp16", 32),
        # a stencil operator applied to a block of vectors
        _case("step_laplacian", "step", "laplacian", 262144, 262144, 5, "fp16", 128),
        # an ordinary skewed matrix in fp32 storage, no tuning run
        _case("step_powerlaw_tf32", "step", "powerlaw", 1 << 20, 1 << 20, 16, "tf32", 128),
        # the largest: graph propagation over an RMAT graph of 4 million
        # vertices with settings pinned from an earlier tuning
        _case("step_rmat_tf32", "step", "rmat", 1 << 22, 1 << 22, 16, "tf32", 64, pinned=True),
        # the reference's dispatcher name on the caller's buffers: block-pruned
        # weights, the densest tiles and the widest product
        _case("launch_blocks_fp16", "launch", "blocks", 65536, 65536, 1311, "fp16", 256, bm=16, fmt="dense"),
        # graph propagation from packed tiles, library defaults
        _case("launch_rmat_packed", "launch", "rmat", 1 << 20, 1 << 20, 16, "fp16", 128, bm=8, fmt="packed"),
        # a banded matrix with ragged sizes through the tallest class, raw fp32 operands
        _case("launch_banded_tf32", "launch", "banded", 100003, 99991, 24, "tf32", 96, bm=64, fmt="dense"),
        # a circuit matrix with one dense row (dc2's shape): split row-blocks,
        # a cleared C, atomics
        _case("launch_circuit_fp16", "launch", "circuit", 116835, 116835, 6, "fp16", 32, bm=8, fmt="dense"),
        # a new matrix every time: small and irregular
        _case("tile_circuit_fp16", "tile", "circuit", 116835, 116835, 6, "fp16", 0, bm=8, pack=False),
        # the largest conversion
        _case("tile_rmat_tf32", "tile", "rmat", 1 << 22, 1 << 22, 16, "tf32", 0, bm=8, pack=False),
        # tiles and then their packed form, 16-row class
        _case("tile_pack_powerlaw_tf32", "tile", "powerlaw", 1 << 20, 1 << 20, 16, "tf32", 0, bm=16, pack=True),
        # from a host CSR matrix to the first product: policy, row split,
        # plan, thresholds from the cost model, one step
        _case("build_banded_fp16", "build", "banded", 200003, 200003, 24, "fp16", 64),
    ]


def draw(rng):
    op = rng.choice(["step", "step", "launch", "launch", "launch", "tile", "tile", "build"])
    kind = rng.choice(["uniform", "laplacian", "powerlaw", "rmat", "blocks", "banded", "circuit"])
    prec = rng.choice(["fp16", "tf32"])
    bm = rng.choice([8, 8, 16, 16, 64])
    colB = rng.choice([8, 32, 64, 96, 128, 200, 256, 512])
    nnz = 2.0 ** rng.uniform(15, 22 if op == "build" else 24.5)
    mean = {"laplacian": 5, "circuit": 6}.get(kind) or int(round(2.0 ** rng.uniform(2, 6)))
    if kind == "blocks":
        mean *= 8                                 # a few dense blocks per row of blocks
    rows = max(512, int(nnz / mean))
    rows = min(rows, (1 << 28) // colB)           # C of at most 1 GB
    cols = rows
    if kind == "laplacian":
        side = max(16, int(math.sqrt(rows)))
        rows = cols = side * side
    elif kind == "rmat":
        scale = max(10, int(math.log2(rows)))
        rows = cols = 1 << scale
        mean = max(2, mean // 2)
    elif kind in ("uniform", "powerlaw", "banded", "blocks"):
        rows += rng.randrange(0, 63)              # ragged last row-blocks
        cols = max(512, int(rows * rng.uniform(0.5, 1.5)))
        if kind == "blocks":
            cols = max(cols, 4 * mean)
    case = _case(None, op, kind, rows, cols, mean, prec, 0 if op == "tile" else colB)
    if op == "launch":
        case.update(bm=bm, fmt="dense" if bm == 64 else rng.choice(["dense", "packed"]))
    elif op == "tile":
        case.update(bm=bm, pack=rng.random() < 0.4)
    elif op == "step" and kind == "rmat" and colB % 64 == 0:
        case.update(pinned=rng.random() < 0.5)
    return case


# ---- matrices ---------------------------------------------------------------

def _powerlaw_lengths(u, mean):
    """Row lengths clip(round(x * u^(-1/1.1)), 1, MAX_ROW) with x chosen for the mean."""
    base = u.pow(-1.0 / 1.1)
    lo, hi = 0.0, float(mean)
    for _ in range(30):
        x = 0.5 * (lo + hi)
        if float((base * x).round().clamp(1, MAX_ROW).mean()) < mean:
            lo = x
        else:
            hi = x
    return (base * hi).round().clamp(1, MAX_ROW).long()


def _keys(case, g):
    """Sorted distinct row * cols + column of the matrix's entries, on the GPU."""
    kind, m, n, mean = case["kind"], case["rows"], case["cols"], case["mean"]
    dev = "cuda"

    def ints(hi, size):
        return torch.randint(0, hi, (size,), generator=g, device=dev, dtype=torch.int64)

    if kind == "uniform":
        r = torch.arange(m, device=dev).repeat_interleave(mean)
        return torch.unique(r * n + ints(n, m * mean))
    if kind == "powerlaw":
        u = 1.0 - torch.rand(m, generator=g, device=dev, dtype=torch.float64)
        length = torch.minimum(_powerlaw_lengths(u, mean), torch.tensor(n, device=dev))
        r = torch.repeat_interleave(torch.arange(m, device=dev), length)
        return torch.unique(r * n + ints(n, r.numel()))
    if kind == "laplacian":
        side = int(math.isqrt(m))
        i = torch.arange(m, device=dev)
        y, x = i // side, i % side
        parts = [i * n + i]
        for ok, d in ((y > 0, -side), (x > 0, -1), (x < side - 1, 1), (y < side - 1, side)):
            parts.append((i * n + i + d)[ok])
        return torch.sort(torch.cat(parts))[0]
    if kind == "banded":
        half = 2 * mean
        r = torch.arange(m, device=dev).repeat_interleave(mean)
        c = (r * n) // m + ints(2 * half + 1, m * mean) - half
        return torch.unique(r * n + c.clamp(0, n - 1))
    if kind == "blocks":
        nb = (m + 15) // 16
        cb = (n + 15) // 16
        per = max(1, mean // 16)
        b = torch.unique(torch.arange(nb, device=dev).repeat_interleave(per) * cb + ints(cb, nb * per))
        br, bc = (b // cb) * 16, (b % cb) * 16
        o = torch.arange(16, device=dev)
        r = (br[:, None, None] + o[None, :, None]).expand(-1, 16, 16).reshape(-1)
        c = (bc[:, None, None] + o[None, None, :]).expand(-1, 16, 16).reshape(-1)
        singles = m * 6                            # scattered single entries between the blocks
        r = torch.cat([r, ints(m, singles)])
        c = torch.cat([c, ints(n, singles)])
        ok = (r < m) & (c < n)
        return torch.unique(r[ok] * n + c[ok])
    if kind == "rmat":
        scale = int(math.log2(m))
        edges = m * mean
        r = torch.zeros(edges, device=dev, dtype=torch.int64)
        c = torch.zeros(edges, device=dev, dtype=torch.int64)
        for _ in range(scale):                     # quadrants (.57, .19, .19, .05)
            u = torch.rand(edges, generator=g, device=dev)
            r = r * 2 + (u >= 0.76)
            c = c * 2 + (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
        return torch.unique(torch.cat([r * n + c, c * n + r]))
    # circuit: a few neighbours per row, a dense row and a dense column
    r = torch.arange(m, device=dev).repeat_interleave(mean - 2)
    near = (r + ints(2049, r.numel()) - 1024).clamp(0, n - 1)
    far = ints(n, r.numel())
    c = torch.where(ints(4, r.numel()) > 0, near, far)
    i = torch.arange(n, device=dev)
    hub = int(ints(n, 1))
    return torch.unique(torch.cat([r * n + c, i * n + i, hub * n + i, i * n + hub]))


def _matrix(case, seed):
    """CSR on the GPU: (ptr int32, idx int32, val in the storage type), and the generator."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    m, n = case["rows"], case["cols"]
    if case["op"] == "tile":
        # as many tiles with every seed, so that outputs can be compared: the
        # matrix of this size with its whole 64-row blocks and its columns
        # turned by amounts of the seed's own
        g0 = torch.Generator(device="cuda")
        g0.manual_seed(zlib.crc32(repr((case["kind"], m, n, case["mean"])).encode()))
        keys = _keys(case, g0)
        full = m // 64 * 64
        by_rows = 64 * int(torch.randint(0, full // 64, (1,), generator=g, device="cuda"))
        by_cols = int(torch.randint(0, n, (1,), generator=g, device="cuda"))
        r = keys // n
        c = (keys - r * n + by_cols) % n
        keys = torch.sort(torch.where(r < full, (r + by_rows) % full, r) * n + c)[0]
    else:
        keys = _keys(case, g)
    nnz = keys.numel()
    r = keys // n
    idx = (keys - r * n).int()
    count = torch.bincount(r, minlength=m)
    ptr = torch.zeros(m + 1, device="cuda", dtype=torch.int32)
    ptr[1:] = torch.cumsum(count, 0).int()
    if case["kind"] == "rmat":                     # 1 / degree
        val = (1.0 / count[r].double()).float()
    elif case["kind"] == "laplacian":
        val = torch.where(idx.long() == r, 4.0, -1.0)
    elif case["kind"] == "blocks":
        val = torch.randn(nnz, generator=g, device="cuda")
    else:
        val = torch.rand(nnz, generator=g, device="cuda") * 2 - 1
    return ptr, idx, val.to(_dtype(case)), g


def _dtype(case):
    return torch.float16 if case["prec"] == "fp16" else torch.float32


def _prec(case):
    return tsp.PREC_FP16 if case["prec"] == "fp16" else tsp.PREC_TF32


def _width(case):
    return 32 if case["colB"] <= 32 else -(-case["colB"] // 64) * 64


def _dense(case, g):
    """B, row-major, the padded columns zero."""
    n, w, cb = case["cols"], _width(case), case["colB"]
    B = torch.zeros(n, w, device="cuda", dtype=_dtype(case))
    if case["kind"] == "blocks":
        B[:, :cb] = torch.randn(n, cb, generator=g, device="cuda")
    else:
        B[:, :cb] = torch.rand(n, cb, generator=g, device="cuda") * 2 - 1
    return B


# ---- device buffers of the library as tensors ---------------------------------

class _View:
    """Memory of the library for torch.as_tensor, which keeps this object, and
    so the memory's owner, for as long as the tensor lives."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": typestr,
                                         "version": 3, "strides": None}


def _tensor(ptr, shape, typestr, owner):
    dt = {"<f4": torch.float32, "<f2": torch.float16, "<i4": torch.int32, "<i8": torch.int64}[typestr]
    if 0 in shape:
        return torch.zeros(shape, dtype=dt, device="cuda")
    return torch.as_tensor(_View(ptr, shape, typestr, owner), device="cuda")


def _ok(status):
    if status != 0:
        raise RuntimeError("status %d" % status)


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


class _Tiles:
    """Tiles made on the device from a device CSR matrix; freed with the object."""

    def __init__(self, case, ptr, idx, val, pack):
        hip, _ = tsp.load()
        self.hip, self.t = hip, tsp.DevTiles()
        self.pval, self.vptr, self.nvals = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_longlong()
        bm, prec = case["bm"], _prec(case)
        bn = tsp.tile_bn(bm, prec)
        _ok(hip.tsp_tile_create_device(ctypes.byref(self.t), case["rows"], case["cols"], idx.numel(), _p(ptr), _p(idx),
                                       _p(val), bm, bn, prec, None))
        if pack:
            _ok(hip.tsp_tiles_pack_device(self.t.tilenum, bm, bn, prec, self.t.d_val, self.t.d_bitmap,
                                          ctypes.byref(self.nvals), ctypes.byref(self.pval), ctypes.byref(self.vptr),
                                          None))

    def tensors(self):
        t = self.t
        v = "<f2" if t.prec == tsp.PREC_FP16 else "<f4"
        out = {"tile_ptr": _tensor(t.d_tile_ptr, (t.tilem + 1,), "<i4", self),
               "tile_nnz": _tensor(t.d_tile_nnz, (t.tilenum + 1,), "<i4", self),
               "colidx": _tensor(t.d_tile_colidx, (t.tilenum, t.bn), "<i4", self),
               "val": _tensor(t.d_val, (t.tilenum, t.bm, t.bn), v, self),
               "bitmap": _tensor(t.d_bitmap, (t.tilenum, t.bitmap_words), "<i8", self)}
        if self.pval:
            out["pval"] = _tensor(self.pval.value, (self.nvals.value,), v, self)
            out["vptr"] = _tensor(self.vptr.value, (t.tilenum + 1,), "<i4", self)
        return out

    def free(self):
        if self.t.d_tile_ptr:
            self.hip.tsp_dev_tiles_free(ctypes.byref(self.t))
        for p in (self.pval, self.vptr):
            if p:
                self.hip.tsp_free(p)
        self.pval, self.vptr = ctypes.c_void_p(), ctypes.c_void_p()

    def __del__(self):
        self.free()


def _schedule(case, tiles):
    """Task schedule of one class on the device, its threshold from the cost model."""
    _, host = tsp.load()
    bm, prec, w = case["bm"], _prec(case), _width(case)
    prm = tsp.ThParams()
    _ok(host.tsp_th_params_probe(0, bm, prec, w, ctypes.byref(prm)))
    tile_ptr = tiles.tensors()["tile_ptr"].cpu().numpy()
    _, top = tsp.optimal_th(bm, w, tile_ptr, prm)
    first = np.arange(tiles.t.tilem, dtype=np.int32) * bm
    m = tsp.Tile_matrix()
    m.tilem, m.tilenum, m.bm, m.bn, m.prec = tiles.t.tilem, tiles.t.tilenum, bm, tiles.t.bn, prec
    m.tile_ptr = tile_ptr.ctypes.data_as(ctypes.POINTER(ctypes.c_int))
    m.orig_tile_row_idx = first.ctypes.data_as(ctypes.POINTER(ctypes.c_int))
    n, rows, cs = ctypes.c_int(), ctypes.POINTER(ctypes.c_uint)(), ctypes.POINTER(ctypes.c_int)()
    _ok(host.tsp_tile_pretreatment(ctypes.byref(m), int(top[0]), ctypes.byref(n), ctypes.byref(rows),
                                   ctypes.byref(cs)))
    r = np.ctypeslib.as_array(rows, (n.value,)).copy()
    c = np.ctypeslib.as_array(cs, (n.value + 1,)).copy()
    host.tsp_free_host(ctypes.cast(rows, ctypes.c_void_p))
    host.tsp_free_host(ctypes.cast(cs, ctypes.c_void_p))
    return n.value, torch.from_numpy(r.view(np.int32)).cuda(), torch.from_numpy(c).cuda(), bool((r >> 31).any())


# ---- plans ------------------------------------------------------------------

def _host_csr(case, ptr, idx, val):
    v = val.cpu().numpy()
    return tsp.Csr(case["rows"], case["cols"], ptr.cpu().numpy(), idx.cpu().numpy(),
                   v.view(np.uint16) if case["prec"] == "fp16" else v, _prec(case))


def _plan(case, A, B):
    """Policy, row split and plan, with the cost model's thresholds."""
    prec, w = _prec(case), _width(case)
    gamma, delta = tsp.predict(tsp.features(A, 9.5, case["colB"]), prec)
    plan = tsp.Plan.from_csr(tsp.matrix_split(A, gamma, delta), case["rows"], case["cols"], w, prec, B)
    if not case.get("pinned"):
        plan.tune(False)
        return plan
    pin = PINNED_TF32 if case["prec"] == "tf32" else PINNED_FP16
    plan.set_th(pin["th"], pin["th"], pin["th"])
    for bm in (16, 8):
        if plan.tilenum(bm):
            plan.set_format(bm, pin["fmt"])
            plan.set_variant(bm, pin["w"], pin["stages"], pin["tpw"], pin["order"])
            plan.set_placement(bm, pin["place"])
            plan.set_lane_indices(bm, bool(pin["lane"]))
            plan.set_b_3byte(bm, bool(pin["b3"]))
    plan.set_hot_rows(pin["hot"])
    return plan


def _plan_c(case, plan):
    c = ctypes.c_void_p()
    _ok(tsp.load()[1].tsp_plan_device_c(plan.p, ctypes.byref(c)))
    return _tensor(c.value, (case["rows"], _width(case)), "<f4", plan)


# ---- the interface ------------------------------------------------------------

def prepare(case, seed):
    ptr, idx, val, g = _matrix(case, seed)
    op = case["op"]
    if op == "tile":
        return {"case": case, "ptr": ptr, "idx": idx, "val": val, "tiles": None}
    B = _dense(case, g)
    if op == "launch":
        packed = case["fmt"] == "packed"
        tiles = _Tiles(case, ptr, idx, val, packed)
        n, rows, cs, split = _schedule(case, tiles)
        C = torch.zeros(case["rows"], _width(case), device="cuda")
        hip, _ = tsp.load()
        t, w, prec = tiles.t, _width(case), _prec(case)
        if packed:
            args = (case["bm"], prec, n, w, tiles.pval, t.d_bitmap, tiles.vptr, _p(rows), _p(cs), _p(B), _p(C),
                    t.d_tile_colidx, case["rows"], None, 0, 0, 0, 0)
            fn = hip.tsp_spmm_launch_packed
        else:
            args = (prec, n, w, t.d_val, _p(rows), _p(cs), _p(B), _p(C), t.d_tile_colidx, case["rows"], None)
            fn = {64: hip.tsp_switch_v64, 16: hip.tsp_switch_v16, 8: hip.tsp_switch_v8}[case["bm"]]
        return {"case": case, "tiles": tiles, "keep": (rows, cs, B), "C": C, "split": split, "fn": fn, "args": args}
    A = _host_csr(case, ptr, idx, val)
    B = B.cpu().numpy()
    if op == "build":
        return {"case": case, "A": A, "B": B, "plan": None}
    plan = _plan(case, A, B)
    return {"case": case, "plan": plan, "C": _plan_c(case, plan)}


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "step":
        state["plan"].run()
        return state["C"]
    if op == "launch":
        if state["split"]:                         # split row-blocks are added to C
            state["C"].zero_()
        _ok(state["fn"](*state["args"]))
        return state["C"]
    if op == "tile":
        if state["tiles"] is not None:             # the matrix before this one
            state["tiles"].free()
        state["tiles"] = _Tiles(case, state["ptr"], state["idx"], state["val"], case["pack"])
        return state["tiles"].tensors()
    if state["plan"] is not None:
        state["plan"].close()
    plan = state["plan"] = _plan(case, state["A"], state["B"])
    C = _plan_c(case, plan)
    plan.run()
    return C


def _entries(case):
    """Expected entries of the matrix."""
    m, n, mean, kind = case["rows"], case["cols"], case["mean"], case["kind"]
    if kind == "blocks":
        return m * (max(1, mean // 16) * 16 + 6)
    if kind == "rmat":
        return m * mean * 1.9
    if kind == "banded":
        return m * mean * 0.89                     # columns drawn twice in the band
    if kind == "circuit":
        return m * (mean + 1)
    return m * mean


def work(case):
    m, n, s, nnz = case["rows"], case["cols"], 2 if case["prec"] == "fp16" else 4, _entries(case)
    if case["op"] == "tile":
        bm = case["bm"]
        bn = (32 if bm == 64 else 16) if s == 2 else (16 if bm == 64 else 8)
        distinct = nnz / (min(bm, 16) if case["kind"] == "blocks" else max(1, bm / 4) if case["kind"] == "banded" else 1)
        tiles = distinct / bn + 0.5 * m / bm
        out = 4 * m / bm + tiles * (4 + 4 * bn + s * bm * bn + bm * bn / 8)
        if case["pack"]:
            out += nnz * s + 4 * tiles
        return {"bytes": 4 * (m + 1) + nnz * (4 + s) + out, "flops": 0}
    return {"bytes": 4 * (m + 1) + nnz * (4 + s) + n * case["colB"] * s + 4 * m * case["colB"],
            "flops": 2 * nnz * case["colB"]}


def tolerance(case):
    # tiles are moved, not computed; products are summed in 32 bits, parts of
    # a split row-block in no fixed order (the same inputs twice: up to 2.5e-7,
    # a single value 5e-5, in rows of 100000 entries)
    return "exact" if case["op"] == "tile" else {"rel": 1e-6, "max": 2e-4}


def _round_tf32(x):
    """fp32 to the nearest value with 10 mantissa bits, ties to even (finite values)."""
    b = x.view(torch.int32)
    return ((b + 0xFFF + ((b >> 13) & 1)) & ~0x1FFF).view(torch.float32)


def exact(case, seed):
    if case["op"] == "tile":
        return None
    ptr, idx, val, g = _matrix(case, seed)
    B = _dense(case, g)
    if case["prec"] == "tf32":                     # the operands of the operator are tf32 values
        val, B = _round_tf32(val), _round_tf32(B)
    out = torch.empty(case["rows"], _width(case), device="cuda", dtype=torch.float64)
    A = torch.sparse_csr_tensor(ptr, idx, val.double(), size=(case["rows"], case["cols"]))
    for c in range(0, _width(case), 64):
        out[:, c:c + 64] = A @ B[:, c:c + 64].double().contiguous()
    return out
