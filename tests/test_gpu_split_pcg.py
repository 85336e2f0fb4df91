"""The two-kernel PCG loop over the split operator: iterates at every iteration limit around
the host's status reads (after 4, 12 and 28 iterations), from zero and from a guess, with all,
some and no rows taken by workgroups of their own, against the textbook recurrence on the
assembled system; convergence at the first iteration and negative curvature."""
import ctypes as C

import numpy as np
import pytest

from yasps_amd.scenes import contact_scene, build_contact_scene

pytestmark = pytest.mark.gpu
SCENE = dict(bodies_x=2, bodies_z=1, cells=4, radius=0.12, cloth_m=9, max_pairs=10 ** 9, seed=0)


@pytest.fixture(scope="module")
def system():
    from yasps_amd import device as dev
    s0, _ = build_contact_scene(contact_scene(**SCENE), threshold_mode="relative_residual")
    s0.minimizeEnergy(tolerance=1e-10)
    hs = s0.minimizer.activeHessian
    n = hs.rows
    H = np.asarray(hs.dense())
    inv = dev.to_host(hs.diagonal_blocks_inverse)
    M = np.zeros((n, n))
    for w, d0, g0 in zip(hs.wrt, hs.diagonal_blocks_start_cpu, hs.gradient_segments_start_cpu):
        k = w.size
        for i in range(w.numInstances):
            a, b = int(g0) + i * k, int(d0) + i * k * k
            M[a:a + k, a:a + k] = inv[b:b + k * k].reshape(k, k)
    return s0, hs, H, M, dev.to_host(hs.gradient.value)


def _solve(hs, max_it, tol, guess=None, long_row=0, sign=1.0, source="f64"):
    from yasps_amd import _lib, device as dev
    f, n = hs.split, hs.rows
    x, work, scalars = dev.zeros(n, "float64"), dev.zeros(5 * n, "float64"), dev.zeros(12288, "float64")
    held = f.v64 * sign if source == "f64" else hs.full_values_f32()
    values, fmt = dev.ptr(held), int(source == "f32")
    if source == "upper":
        hs.value_source = "upper"
        values, fmt = hs.solve_values()
        hs.value_source = "auto"
    st = _lib.PcgStats()
    g = None if guess is None else dev.to_device(guess, "float64")
    rc = _lib.load().ysp_pcg_solve_full(
        max_it, tol, 1, dev.ptr(f.row_ptr), dev.ptr(f.col), values, fmt, f.nnz, long_row,
        dev.ptr(hs.diagonal_blocks_inverse), _lib.u32_array(hs.diagonal_blocks_start_cpu[:-1]),
        _lib.u32_array([w.numInstances for w in hs.wrt]), _lib.u32_array([w.size for w in hs.wrt]),
        _lib.u32_array(hs.gradient_segments_start_cpu[:-1]), len(hs.wrt),
        dev.ptr(hs.gradient.value), n, dev.ptr(x), dev.ptr(g), int(g is None), dev.ptr(work),
        dev.ptr(scalars), C.byref(st), dev.stream())
    return rc, st, dev.to_host(x)


def _rounded(hs):
    """The operator with every entry of the split block-CSR rounded to FP32 (a block of the
    static and one of the dynamic part at the same place are entries of their own)."""
    from yasps_amd import device as dev
    f, A = hs.split, np.zeros((hs.rows // 3, 3, hs.rows // 3, 3))
    v = dev.to_host(f.v64).reshape(9, -1)[:, :f.nnz].T.reshape(-1, 3, 3)
    row = np.repeat(np.arange(f.nbr), np.diff(dev.to_host(f.row_ptr, "uint32").astype(np.int64)))
    np.add.at(A, (row, slice(None), dev.to_host(f.col, "uint32")[:f.nnz].astype(np.int64)),
              v.astype(np.float32).astype(np.float64))
    return A.reshape(hs.rows, hs.rows)


def _pcg(H, M, b, x, iterations):
    r = b - H @ x
    z = M @ r
    p, rz = z, r @ z
    for _ in range(iterations):
        q = H @ p
        alpha = rz / (p @ q)
        x, r = x + alpha * p, r - alpha * q
        z = M @ r
        rz, old = r @ z, rz
        p = z + rz / old * p
    return x, rz, r @ r


@pytest.mark.parametrize("long_row", [0, 1, 4, 1 << 30])
@pytest.mark.parametrize("max_it", [1, 3, 4, 5, 12, 13])
def test_iterates(system, max_it, long_row):
    _, hs, H, M, b = system
    for guess in (None, np.random.default_rng(1).normal(size=b.size) * 1e-3):
        print(f"{max_it} iterations, long rows from {long_row}, guess {guess is not None}", flush=True)
        rc, st, x = _solve(hs, max_it, 1e-30, guess, long_row)
        want, rz, rr = _pcg(H, M, b, np.zeros_like(b) if guess is None else guess, max_it)
        assert rc == -4 and st.iterations == max_it
        # rounding of a dot or product (1e-14 here), amplified by the recurrence: 1e-11 after 5
        # iterations is the bound of the long-row test, a factor 10 for the 13 here
        assert np.linalg.norm(x - want) <= 1e-10 * np.linalg.norm(want)
        assert abs(st.delta - rz) <= 1e-8 * rz and abs(st.rr - rr) <= 1e-8 * rr


@pytest.mark.parametrize("source", ["f32", "upper"])
@pytest.mark.parametrize("long_row", [0, 4])
def test_iterates_from_other_values(system, long_row, source):
    _, hs, H, M, b = system
    A = _rounded(hs) if source == "f32" else H
    for max_it in (1, 5, 13):
        print(f"{max_it} iterations, long rows from {long_row}, {source}", flush=True)
        rc, st, x = _solve(hs, max_it, 1e-30, None, long_row, source=source)
        want, rz, rr = _pcg(A, M, b, np.zeros_like(b), max_it)
        assert rc == -4 and st.iterations == max_it
        assert np.linalg.norm(x - want) <= 1e-10 * np.linalg.norm(want)      # as above
        assert abs(st.delta - rz) <= 1e-8 * rz and abs(st.rr - rr) <= 1e-8 * rr


def test_first_iteration_and_negative_curvature(system):
    _, hs, H, M, b = system
    # a residual tolerance that one iteration meets, and none before it
    _, _, rr = _pcg(H, M, b, np.zeros_like(b), 1)
    tol = 1.01 * np.sqrt(rr) / np.linalg.norm(b)
    rc, st, _ = _solve(hs, 50, tol)
    assert rc == (1 if tol < 1 else 0) and st.iterations == rc
    rc, st, _ = _solve(hs, 50, 1e-10, sign=-1.0)
    assert rc == -5 and st.iterations == 1
