"""The tiled symmetric operator of the PCG (``ysp_bsr3_tiles_*``, ``YSP_VALUES_TILED``) through
the C ABI on random symmetric block graphs of sizes around a tile (1, 255, 256, 257 rows),
a slice (64 rows) and the launch (several tiles, the last one nearly empty), with empty
rows, rows of very different lengths, any order of the points, an initial guess and FP32
values: the solution against numpy.linalg.solve and the iteration count against the
mirrored operator's.

Tolerance: the systems are diagonally dominant (condition number below 10), so a relative
residual of t leaves a relative error of at most 10 t; FP32 values change the solution by at
most 10 eps32 per unit of the operator, 2e-6 with a factor of two to spare."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(nv, degree, seed, hub=0, isolated=0):
    """Upper 3x3 blocks (positions, values) of a symmetric, diagonally dominant operator."""
    rng = np.random.default_rng(seed)
    a = rng.integers(0, nv, degree * nv)
    b = (a + np.rint(rng.normal(0, 12, a.size)).astype(np.int64)) % nv
    if hub:
        a = np.r_[a, np.zeros(hub, dtype=np.int64)]
        b = np.r_[b, rng.permutation(nv)[:hub]]
    keep = (a != b) & (a >= isolated) & (b >= isolated)
    pairs = np.unique(np.sort(np.stack([a[keep], b[keep]], 1), axis=1), axis=0)
    off = rng.uniform(-1, 1, (len(pairs), 3, 3))
    weight = np.zeros(nv)
    np.add.at(weight, pairs.ravel(), 3.0)
    diag = np.zeros((nv, 3, 3))
    diag[:, [0, 1, 2], [0, 1, 2]] = 1.5 * weight[:, None] + 1.0
    pos = np.concatenate([np.stack([np.arange(nv)] * 2, 1), pairs])
    vals = np.concatenate([diag, off])
    order = np.lexsort((pos[:, 1], pos[:, 0]))
    pos, vals = pos[order], vals[order]
    A = np.zeros((3 * nv, 3 * nv))
    for (r, c), B in zip(pos, vals):
        A[3 * r:3 * r + 3, 3 * c:3 * c + 3] = B
        if r != c:
            A[3 * c:3 * c + 3, 3 * r:3 * r + 3] = B.T
    return 3 * pos, vals, np.linalg.inv(diag), A


class _Operator:
    def __init__(self, pos, vals, minv, n, points):
        from yasps_amd import _lib, device as dev
        self.lib, self.dev, self.L, self.n = _lib.load(), dev, _lib, n
        lib, s = self.lib, dev.stream()
        nb, nv = len(pos), n // 3
        self.values = dev.to_device(vals.reshape(-1), "float64")
        positions = dev.to_device(pos.reshape(-1), "uint32")
        self.row_ptr = dev.empty(nv + 1, "uint32")
        self.col, self.src = dev.empty(2 * nb, "uint32"), dev.empty(2 * nb, "uint32")
        count = C.c_uint32(0)
        _lib.check(lib.ysp_bsr3_build(dev.ptr(positions), nb, None, 0, n, dev.ptr(self.row_ptr),
                                      dev.ptr(self.col), dev.ptr(self.src), 2 * nb, C.byref(count), s),
                   "build")
        self.nnz = count.value
        self.v64 = dev.empty(9 * ((self.nnz + 63) // 64 * 64), "float64")
        _lib.check(lib.ysp_bsr3_gather_values(dev.ptr(self.values), None, dev.ptr(self.src), self.nnz,
                                              dev.ptr(self.v64), None, s), "gather")
        self.minv = dev.to_device(minv.reshape(-1), "float64")
        self.minv32 = dev.to_device(minv.reshape(-1).astype(np.float32), "float32")
        slices = (nv + 255) // 256 * 4
        self.rows, self.lens = dev.empty(nv, "uint32"), dev.empty(nv, "uint32")
        self.slice_start, work = dev.empty(slices + 1, "uint32"), dev.empty(2 * nv, "uint32")
        p = None if points is None else dev.to_device(points.reshape(-1), "float64")
        _lib.check(lib.ysp_bsr3_tiles_layout(
            dev.ptr(self.row_ptr), dev.ptr(self.col), self.nnz, n, dev.ptr(p), dev.ptr(self.rows),
            dev.ptr(self.lens), dev.ptr(self.slice_start), dev.ptr(work), C.byref(count), s), "layout")
        self.entries = count.value
        if not self.entries:
            return
        self.entry, source = dev.empty(self.entries, "uint32"), dev.empty(self.entries, "uint32")
        _lib.check(lib.ysp_bsr3_tiles_entries(
            dev.ptr(self.row_ptr), dev.ptr(self.col), dev.ptr(self.src), n, dev.ptr(self.rows),
            dev.ptr(self.slice_start), dev.ptr(work), dev.ptr(self.entry), dev.ptr(source), s), "entries")
        self.t64 = dev.empty(9 * self.entries, "float64")
        self.t32 = dev.empty(9 * self.entries, "float32")
        _lib.check(lib.ysp_bsr3_tiles_values(dev.ptr(self.values), dev.ptr(source), self.entries,
                                             dev.ptr(self.t64), dev.ptr(self.t32), s), "values")

    def solve(self, rhs, tol, tiled, f32=False, guess=None, max_iterations=2000):
        dev, L = self.dev, self.L
        if tiled:
            d = L.TiledValues(dev.ptr(self.rows), dev.ptr(self.lens), dev.ptr(self.slice_start),
                              dev.ptr(self.entry), self.entries,
                              dev.ptr(self.t32 if f32 else self.t64), int(f32))
            values, fmt = C.addressof(d), L.VALUES_TILED
        else:
            values, fmt = dev.ptr(self.v64), L.VALUES_F64
        b = dev.to_device(rhs, "float64")
        x = dev.zeros(self.n, "float64")
        x.fill_(np.nan)
        g = None if guess is None else dev.to_device(guess, "float64")
        work, st = dev.zeros(5 * self.n, "float64"), dev.zeros(12288, "float64")
        stats = L.PcgStats()
        rc = self.lib.ysp_pcg3_solve(
            max_iterations, tol, 1, dev.ptr(self.row_ptr), dev.ptr(self.col), values, fmt, self.nnz,
            dev.ptr(self.minv32 if f32 else self.minv), int(f32), dev.ptr(b), self.n, dev.ptr(x),
            dev.ptr(g), int(g is None), dev.ptr(work), dev.ptr(st), C.byref(stats), dev.stream())
        return rc, dev.to_host(x), stats


@pytest.mark.parametrize("nv,degree", [(1, 1), (2, 1), (63, 3), (64, 3), (255, 4), (256, 4), (257, 4),
                                       (513, 7), (700, 20)])
@pytest.mark.parametrize("points", ["line", "random", "same", "none"])
def test_tiled_pcg_equals_dense_solve(nv, degree, points):
    print(f"tiles nv={nv} degree={degree} points={points}", flush=True)
    rng = np.random.default_rng(nv)
    pos, vals, minv, A = _system(nv, degree, seed=nv, isolated=nv // 5)
    n = 3 * nv
    p = {"line": np.stack([np.arange(nv)] * 3, 1) * 1.0, "random": rng.standard_normal((nv, 3)),
         "same": np.ones((nv, 3)), "none": None}[points]
    op = _Operator(pos, vals, minv, n, p)
    assert op.entries >= len(pos) and sorted(op.dev.to_host(op.rows, "uint32")) == list(range(nv))
    b = rng.standard_normal(n)
    xs = np.linalg.solve(A, b)
    rc0, _, st0 = op.solve(b, 1e-12, False)
    rc, x, st = op.solve(b, 1e-12, True)
    assert rc >= 0 and abs(st.iterations - st0.iterations) <= 1
    assert np.linalg.norm(x - xs) <= 1e-11 * np.linalg.norm(xs)
    # an initial guess (a plain product with the operator first)
    rc, x, st = op.solve(b, 1e-12, True, guess=xs + 1e-3 * rng.standard_normal(n))
    assert rc >= 0 and np.linalg.norm(x - xs) <= 1e-11 * np.linalg.norm(xs)
    rc, x, _ = op.solve(b, 1e-10, True, f32=True)
    assert rc >= 0 and np.linalg.norm(x - xs) <= 2e-6 * np.linalg.norm(xs)
    # the limit of iterations, as the mirrored operator reports it
    if st0.iterations > 2:
        assert op.solve(b, 1e-12, True, max_iterations=2)[0] == op.solve(
            b, 1e-12, False, max_iterations=2)[0] == -4


def test_rows_too_long_for_tiles_are_refused():
    print("tiles: hub row", flush=True)
    pos, vals, minv, _ = _system(300, 3, seed=9, hub=200)
    assert _Operator(pos, vals, minv, 900, None).entries == 0


def test_scene_uses_tiles_and_matches_mirrored():
    """A cube above the size from which the solver reads tiles, against the mirrored copy."""
    from yasps_amd import _lib, device as dev
    from yasps_amd.scenes import cube_scene, build_yasps_scene
    print("tiles: n=32 cube", flush=True)
    x = {}
    for source in ("auto", "mirrored"):
        s0, _ = build_yasps_scene(cube_scene(32, seed=1), threshold_mode="relative_residual")
        h = s0.minimizer.computeNumericValue()
        h.value_source = source
        assert (h.full.tiles is not None) and h.full.tiles.entries < 0.9 * h.full.nnz
        x[source] = dev.to_host(s0.minimizeEnergy(tolerance=1e-10)[0]).copy()
        # what the solve read
        tiled = source == "auto"
        assert h.pcg_values()[1] == (_lib.VALUES_TILED if tiled else _lib.VALUES_F64)
        assert h.full.tiles.valid64 == tiled and not h.full.tiles.valid32
    assert np.linalg.norm(x["auto"] - x["mirrored"]) <= 1e-8 * np.linalg.norm(x["mirrored"])


def test_mixed_solve_through_tiles():
    """FP32 tiles in the Krylov loop, FP64 refinement: the true residual, and the FP64
    solution to the tolerance times the condition of the cube (below 1e3)."""
    from yasps_amd import _lib, device as dev
    from yasps_amd.hessian import vector
    from yasps_amd.scenes import cube_scene, build_yasps_scene
    print("tiles: n=32 cube, mixed", flush=True)
    x = {}
    for precision in ("fp64", "mixed"):
        s0, _ = build_yasps_scene(cube_scene(32, seed=1), threshold_mode="relative_residual",
                                  precision=precision)
        x[precision] = s0.minimizeEnergy(tolerance=1e-10)[0].reshape(-1).clone()
        h = s0.minimizer.activeHessian
        mixed = precision == "mixed"
        assert h.pcg_values(f32=mixed)[1] == _lib.VALUES_TILED
        assert h.full.tiles.valid32 == mixed and h.full.tiles.valid64 == (not mixed)
        g = h.gradient.value
        r = h.spmv(vector(h.rows, x[precision].clone())).value - g
        assert float(r.norm() / g.norm()) <= 1.01e-10
    assert float((x["mixed"] - x["fp64"]).norm() / x["fp64"].norm()) <= 1e-7


def test_product_pass_over_tiles():
    """One pass of the loop's product on prepared state: p = z + p0, q = A z + q0 in tile order."""
    from yasps_amd import _lib, device as dev
    from yasps_amd.hessian import vector
    from yasps_amd.scenes import cube_scene, build_yasps_scene
    print("tiles: product pass", flush=True)
    s0, _ = build_yasps_scene(cube_scene(32, seed=1))
    h = s0.minimizer.computeNumericValue()
    n, f = h.rows, h.full
    values, fmt = h.pcg_values()
    assert fmt == _lib.VALUES_TILED
    work, scalars = dev.zeros(5 * n, "float64"), dev.zeros(12288, "float64")
    _lib.check(_lib.load().ysp_pcg3_product_pass(
        dev.ptr(f.row_ptr), dev.ptr(f.col), values, fmt, f.nnz, n, dev.ptr(work), dev.ptr(scalars), 1,
        dev.stream()), "ysp_pcg3_product_pass")
    z, p, q = (dev.to_host(work)[k * n:(k + 1) * n] for k in (1, 2, 4))
    assert np.array_equal(z, 1.0 + 0.01 * (np.arange(n) % 7)) and np.array_equal(p, z + 0.5)
    rows = dev.to_host(f.tiles.rows, "uint32").astype(np.int64)
    order = (3 * rows[:, None] + np.arange(3)).ravel()
    zn = np.empty(n)
    zn[order] = z
    want = h.spmv(vector().updateValue(zn)).get()[order] + 0.25
    # sums of at most 96 entries in another order: 96 x 3 eps of the largest product
    scale = np.abs(dev.to_host(h.blocks_flattened)).max() * np.abs(z).max()
    assert np.abs(q - want).max() <= 288 * np.finfo(np.float64).eps * scale * 3
