"""The PCG loop over a split operator too large for the two-kernel iteration (above 600,000
entries: p formed in a kernel of its own, one vector gathered per entry): iterates at the
iteration limits around the host's status reads, from zero and from a guess, with all, some
and no rows taken by workgroups of their own and every value source, against the textbook
recurrence on the host; convergence at the first iteration and negative curvature."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

from yasps_amd.scenes import contact_scene, build_contact_scene

pytestmark = pytest.mark.gpu
SCENE = dict(bodies_x=4, bodies_z=3, cells=12, cloth_m=160, max_pairs=150_000, seed=0)


@pytest.fixture(scope="module")
def system():
    from yasps_amd import device as dev
    s0, _ = build_contact_scene(contact_scene(**SCENE), threshold_mode="relative_residual")
    s0.minimizeEnergy(tolerance=0.5)
    hs = s0.minimizer.activeHessian
    f, n = hs.split, hs.rows
    assert f.nnz > 600_000
    stride = (f.nnz + 63) // 64 * 64
    rp = dev.to_host(f.row_ptr, "uint32").astype(np.int64)
    assert np.diff(rp).max() > 128                       # rows with workgroups of their own
    v = dev.to_host(f.v64).reshape(9, stride)[:, :f.nnz].T.reshape(-1, 3, 3)
    H = sp.bsr_matrix((v, dev.to_host(f.col, "uint32")[:f.nnz].astype(np.int64), rp), shape=(n, n)).tocsr()
    inv, blocks = dev.to_host(hs.diagonal_blocks_inverse), []
    for w, d0 in zip(hs.wrt, hs.diagonal_blocks_start_cpu):
        k, c = w.size, w.numInstances
        blocks.append(sp.bsr_matrix((inv[int(d0):int(d0) + c * k * k].reshape(c, k, k),
                                     np.arange(c), np.arange(c + 1)), shape=(c * k, c * k)))
    return s0, hs, H, sp.block_diag(blocks, format="csr"), dev.to_host(hs.gradient.value)


def _solve(hs, max_it, tol, guess=None, long_row=0, source="f64", sign=1.0):
    from yasps_amd import _lib, device as dev
    f, n = hs.split, hs.rows
    x, work, scalars = dev.zeros(n, "float64"), dev.zeros(5 * n, "float64"), dev.zeros(12288, "float64")
    work.fill_(np.nan)
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


@pytest.mark.parametrize("source", ["f64", "f32", "upper"])
@pytest.mark.parametrize("long_row", [0, 1, 1 << 30])
@pytest.mark.parametrize("max_it", [1, 4, 5, 13])
def test_iterates(system, max_it, long_row, source):
    _, hs, H, M, b = system
    # FP32 values: the operator rounded entry by entry, the arithmetic stays FP64
    A = sp.csr_matrix((H.data.astype(np.float32).astype(np.float64), H.indices, H.indptr), H.shape) \
        if source == "f32" else H
    for guess in (None, np.random.default_rng(1).normal(size=b.size) * 1e-3):
        print(f"{max_it} iterations, long rows from {long_row}, {source}, guess {guess is not None}", flush=True)
        rc, st, x = _solve(hs, max_it, 1e-30, guess, long_row, source)
        want, rz, rr = _pcg(A, M, b, np.zeros_like(b) if guess is None else guess, max_it)
        assert rc == -4 and st.iterations == max_it
        # rounding of a dot or product (1e-14 here), amplified by the recurrence, as for small
        # operators
        assert np.linalg.norm(x - want) <= 1e-10 * np.linalg.norm(want)
        assert abs(st.delta - rz) <= 1e-8 * rz and abs(st.rr - rr) <= 1e-8 * rr


def test_first_iteration_and_negative_curvature(system):
    _, hs, H, M, b = system
    _, _, rr = _pcg(H, M, b, np.zeros_like(b), 1)
    tol = 1.01 * np.sqrt(rr) / np.linalg.norm(b)
    rc, st, _ = _solve(hs, 50, tol)
    assert rc == (1 if tol < 1 else 0) and st.iterations == rc
    rc, st, _ = _solve(hs, 50, 1e-10, sign=-1.0)
    assert rc == -5 and st.iterations == 1
