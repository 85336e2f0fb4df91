"""The closed form of the hinge energy's derivatives against central differences of the
energy with 60 digits: flat, bent, nearly folded both ways, a sliver, a small hinge far from
the origin."""
import mpmath as mp
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps
K, THETA0, LEN = 3.7, 0.2, 1.3


def _hinge(angle, height=1.0, scale=1.0, shift=0.0):
    """Edge along a skew direction, faces at the dihedral angle pi - |angle|."""
    q = np.array([[0, 0, 0], [1, 0, 0], [0.3, height, 0],
                  [0.8, -0.9 * np.cos(angle), 0.9 * np.sin(angle)]])
    R = np.linalg.qr(np.random.default_rng(1).normal(size=(3, 3)))[0]
    return scale * (q @ R.T) + shift


HINGES = {"flat": (_hinge(0.0), 1.0), "bent": (_hinge(1.1), 1.0), "bent back": (_hinge(-2.0), 1.0),
          "folded": (_hinge(np.pi - 1e-3), 1e-3), "folded back": (_hinge(1e-3 - np.pi), 1e-3),
          "sliver": (_hinge(0.7, height=1e-3), 1.0), "far": (_hinge(0.4, scale=1e-2, shift=2.0), 1.0)}


def _energy(x):
    q = [mp.matrix(x[3 * i:3 * i + 3]) for i in range(4)]

    def cross(a, b):
        return mp.matrix([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2],
                          a[0] * b[1] - a[1] * b[0]])

    def dot(a, b):
        return sum(a[i] * b[i] for i in range(3))
    n0, n1 = cross(q[0] - q[2], q[1] - q[2]), cross(q[1] - q[3], q[0] - q[3])
    e = q[1] - q[0]
    theta = 2 * mp.atan2(dot(cross(n0, n1), e) / mp.sqrt(dot(e, e)),
                         dot(n0, n1) + mp.sqrt(dot(n0, n0) * dot(n1, n1)))
    return K * (theta - mp.mpf(THETA0)) ** 2 * mp.mpf(LEN)


def _derivatives(x):
    """Central differences at 60 digits: truncation and cancellation below 1e-20."""
    with mp.workdps(60):
        x = [mp.mpf(float(v)) for v in x]
        h = mp.mpf(10) ** -16 * max(abs(a - b) for a in x[:3] for b in x[3:6])

        def at(*moves):
            y = list(x)
            for i, d in moves:
                y[i] += d
            return _energy(y)
        g = [float((at((i, h)) - at((i, -h))) / (2 * h)) for i in range(12)]
        H = np.zeros((12, 12))
        for i in range(12):
            for j in range(i, 12):
                H[i, j] = H[j, i] = float((at((i, h), (j, h)) - at((i, h), (j, -h)) -
                                           at((i, -h), (j, h)) + at((i, -h), (j, -h))) / (4 * h * h))
        return float(_energy(x)), np.array(g), H


def test_hinge_derivatives():
    from yasps_amd import scene, device as dev, energies as en
    x = np.array([h[0] for h in HINGES.values()])
    n = len(x)
    s0 = scene("s")
    m = s0.addMesh("m")
    v = m.addPrimitive("v", numInstances=4 * n)
    pos = v.addAttribute("position", rows=3, cols=1)
    pos.updateValue(x.reshape(-1, 3))
    v.addConstant("rest", rows=3, cols=1).updateValue(x.reshape(-1, 3))
    el = m.addPrimitive("el", numInstances=n)
    e2v = el.addConnectivity("e2v", v, np.arange(4 * n).reshape(n, 4), 4)
    att = el.addAttribute("e", computed_attribute=en.bending(
        el.addAttribute("p", through=e2v, source=pos),
        el.addAttribute("r", through=e2v, source=v["rest"]), K))
    params = dev.to_device(np.tile([THETA0, LEN], n), "float64")
    att.expression.element_params = lambda: params
    s0.addEnergy(att, projection_method=0)
    s0.addMinimizeTarget([pos])
    hs = s0.minimizer.computeNumericValue()
    D, grad = hs.dense(), dev.to_host(hs.gradient.value)
    values = dev.to_host(att.compute().value).reshape(n)
    for i, (name, (q, fold)) in enumerate(HINGES.items()):
        E, g, H = _derivatives(q.reshape(-1))
        # a normal loses |a| |b| / |n| of its digits, the angle 1 / (distance from the fold),
        # theta - theta0 what cancels there
        kappa = 1.0
        for o in (2, 3):
            a, b = q[0] - q[o], q[1] - q[o]
            kappa = max(kappa, np.linalg.norm(a) * np.linalg.norm(b) / np.linalg.norm(np.cross(a, b)))
        theta = THETA0 + np.sqrt(E / (K * LEN))
        tol = 50 * EPS * kappa * max(1 / fold, theta / abs(theta - THETA0))
        err = [abs(values[i] - E) / E, np.abs(grad[12 * i:12 * i + 12] - g).max() / np.abs(g).max(),
               np.abs(D[12 * i:12 * i + 12, 12 * i:12 * i + 12] - H).max() / np.abs(H).max()]
        print(name, err, tol, flush=True)
        assert max(err) <= tol, name
