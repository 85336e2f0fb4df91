"""PSD projection of element Hessians on the GPU at the spectra where an eigensolver can go
wrong, against the oracle (``oracle/projection.py``, numpy eigh): a 6 x 6 inner Hessian of a
quadratic form with a chosen spectrum, and SNH tets in deformations whose 9 x 9 Hessians
have repeated, zero and large negative eigenvalues.

Tolerance: a backward-stable symmetric eigen-decomposition puts an error of a small
multiple of N eps |A| on V f(d) V^T; both sides have one, and the element sums add a few
roundings: 64 N eps of the largest entry."""
import numpy as np
import pytest

from oracle import newton, projection
from yasps_amd.scenes import cube_scene, build_yasps_scene

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
rng0 = np.random.default_rng(5)
BASIS = np.linalg.qr(rng0.standard_normal((6, 6)))[0]


def _with(spectrum, scale=1.0):
    return scale * (BASIS * np.asarray(spectrum)) @ BASIS.T


QS = {
    "diagonal": np.diag([3.0, -2.0, 0.0, 5.0, -1e-3, 1.0]),
    "exchange": np.fliplr(np.eye(6)),
    "tridiagonal": np.diag(np.ones(5), 1) + np.diag(np.ones(5), -1),
    "split": np.kron(np.eye(3), [[0.0, 1.0], [1.0, 0.0]]),
    "ones": -np.ones((6, 6)),
    "repeated": _with([-1, -1, -1, 2, 2, 2]),
    "negative definite": _with([-1, -2, -3, -4, -5, -6]),
    "rank one": _with([-7, 0, 0, 0, 0, 0]),
    "graded": _with([1.0, -1e-3, 1e-6, -1e-6, 1e-9, 0.0]),
    "large": _with([1, -2, 3, -4, 5, -6], 1e150),
    "nearly diagonal": np.diag([1.0, -1.0, 2.0, -2.0, 3.0, -3.0]) + 1e-13 * (np.ones((6, 6)) - np.eye(6)),
}


def _quadratic_scene(Q, method):
    from yasps_amd import scene
    from yasps_amd.energies import quadratic_form
    s0 = scene("projection")
    m = s0.addMesh("mesh")
    v = m.addPrimitive("vertices", numInstances=4)
    pos = v.addAttribute("position", rows=3, cols=1)
    pos.updateValue(np.arange(12.0))
    el = m.addPrimitive("elements", numInstances=1)
    to_v = el.addConnectivity("to_vertices", v, np.arange(4)[None], 4)
    lp = el.addAttribute("local_position", through=to_v, source=pos)
    e = el.addAttribute("energy", computed_attribute=quadratic_form(lp, np.eye(6, 12), Q))
    s0.addEnergy(e, [pos], projection_method=method)
    s0.addMinimizeTarget([pos])
    return s0


@pytest.mark.parametrize("method", [1, 2])
@pytest.mark.parametrize("name", list(QS))
def test_inner_hessian_spectra(name, method):
    print(f"projection {name} method {method}", flush=True)
    Q = 0.5 * (QS[name] + QS[name].T)
    want = np.zeros((12, 12))
    want[:6, :6] = projection.project(Q, method)
    got = _quadratic_scene(Q, method).minimizer.computeNumericValue().dense()
    assert np.abs(got - want).max() <= 64 * 6 * EPS * np.abs(Q).max()


DEFORMATIONS = {
    "uniform compression": 0.3 * np.eye(3),
    "collapsed": np.zeros((3, 3)),
    "flat": np.diag([1.0, 1.0, 0.0]),
    "inverted": np.diag([1.0, 1.0, -1.0]),
    "stretched": np.diag([40.0, 1.0, 0.1]),
    "sheared": np.array([[1.0, 2.0, 0.0], [0.0, 1.0, -3.0], [0.0, 0.0, 0.5]]),
}


@pytest.mark.parametrize("method", [1, 2])
@pytest.mark.parametrize("name", list(DEFORMATIONS) + ["noise"])
def test_tet_hessians(name, method):
    from yasps_amd import device as dev
    print(f"tet projection {name} method {method}", flush=True)
    cs = cube_scene(3, noise=0.5 if name == "noise" else 0.0, seed=2)
    if name != "noise":
        # the fixed face too: every tet in the same state
        cs.position = cs.rest @ DEFORMATIONS[name].T
    st = newton.fast_structure(cs)
    asm = newton.evaluate(cs, st, method)
    s0, _ = build_yasps_scene(cs, projection_method=method)
    hs = s0.minimizer.computeNumericValue()
    got = dev.to_host(hs.blocks_flattened)
    assert np.abs(got - asm.values).max() <= 64 * 9 * EPS * np.abs(asm.values).max()
