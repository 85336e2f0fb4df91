"""Element evaluations queued on two streams without a host wait between them: the Hessians that
one call holds between its launches are not the other's. Staged assembly sums in a fixed
order, so every result has the bits that the same scene gives alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _membranes(n, seed):
    """n StVK membranes with vertices of their own, most of them compressed (indefinite)."""
    from yasps_amd import scene, energies as en
    rng = np.random.default_rng(seed)
    rest = np.tile([[0.0, 0, 0], [1, 0, 0], [0, 1, 0]], (n, 1))
    x = rest * 0.7 + 0.1 * rng.normal(size=rest.shape)
    s0 = scene("s")
    m = s0.addMesh("m")
    v = m.addPrimitive("v", numInstances=3 * n)
    pos = v.addAttribute("position", rows=3, cols=1)
    pos.updateValue(x)
    v.addConstant("rest", rows=3, cols=1).updateValue(rest)
    el = m.addPrimitive("el", numInstances=n)
    e2v = el.addConnectivity("e2v", v, np.arange(3 * n).reshape(n, 3), 3)
    p = el.addAttribute("p", through=e2v, source=pos)
    r = el.addAttribute("r", through=e2v, source=v["rest"])
    att = el.addAttribute("e", computed_attribute=en.stvk_membrane(r, p, 1e3, 8e2, 0.01, 0.05))
    s0.addEnergy(att, projection_method=2)
    s0.addMinimizeTarget([pos])
    return s0.minimizer.computeNumericValue()


def _tets(n, seed):
    """SNH tets and inertia of a cube (6 n^3 tets), many of the tets in the projection's queue."""
    from yasps_amd.scenes import cube_scene, build_yasps_scene
    s0, _ = build_yasps_scene(cube_scene(n, seed=seed))
    return s0.minimizer.computeNumericValue()


@pytest.mark.parametrize("scene,sizes", [(_membranes, (200_000, 300)), (_membranes, (300, 200_000)),
                                         (_membranes, (20_000, 20_000)), (_tets, (32, 4)),
                                         (_tets, (4, 32)), (_tets, (16, 16))])
@pytest.mark.parametrize("default", [False, True])
def test_two_streams_keep_their_hessians(scene, sizes, default):
    from yasps_amd import device as dev
    t = dev.torch()
    print(f"element streams {scene.__name__} {sizes} default {default}", flush=True)
    hs = [scene(n, k) for k, n in enumerate(sizes)]
    want = [(h.gradient.value.clone(), h.blocks_flattened.clone()) for h in hs]
    streams = [t.cuda.Stream(), t.cuda.default_stream() if default else t.cuda.Stream()]
    t.cuda.synchronize()
    for _ in range(4):
        for h in hs:
            h.gradient.value.fill_(np.nan)
            h.blocks_flattened.fill_(np.nan)
        t.cuda.synchronize()
        for h, s in zip(hs, streams):
            with t.cuda.stream(s):
                h.compute(check=False)
        t.cuda.synchronize()
        for h, (g, b) in zip(hs, want):
            assert t.equal(h.gradient.value, g) and t.equal(h.blocks_flattened, b)
    for s in streams:                                    # the flags queued on each stream
        with t.cuda.stream(s):
            from yasps_amd.hessian import check_deferred
            check_deferred()
