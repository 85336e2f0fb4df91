"""Staged assembly of an energy whose vertices are not 3 wide (staged blocks are 3 x 3): refused
by the deferred check, with nothing written, also where one wavefront holds elements with one
slot per vertex beside elements with other slots."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ERR_UNSUPPORTED = -6
GUARD = 4096                          # words before and after everything the call may write


@pytest.mark.parametrize("method", [0, 2])
@pytest.mark.parametrize("n", [1, 64, 131])
@pytest.mark.parametrize("mixed", ["one slot", "three slots", "both"])
def test_staged_nine_wide_energy_is_refused(mixed, n, method):
    from yasps_amd import _lib, device as dev
    from yasps_amd.energies import KIND_IDS
    print(f"staged 9-wide energy: {mixed}, {n} elements, method {method}", flush=True)
    lib, K = _lib.load(), 3
    three = {"one slot": np.zeros(n, bool), "three slots": np.ones(n, bool),
             "both": np.arange(n) % 2 == 1}[mixed]
    first = 2 + 9 * np.arange(n)
    idx = np.where(three[:, None], first[:, None] + [0, 3, 6], np.stack([first, 0 * first, 0 * first], 1))
    size = np.where(three[:, None], 3, [9, 0, 0])
    perm = np.where(three[:, None], [1, 2, 3], [1, 0, 0])
    pairs = np.where(three, 6, 1)
    up = dev.to_device
    outer = up(np.concatenate([[0], np.cumsum(pairs)]).astype(np.uint32), "uint32")
    lookups = up(np.zeros(int(pairs.sum())), "uint32")
    starts = up(np.array([0, 9 * n], np.uint32), "uint32")
    diag = up(np.array([0, 81 * n], np.uint32), "uint32")
    bodies = up(np.tile(np.eye(3).ravel(), n) + 0.1, "float64")
    count = up(np.array([n], np.uint32), "uint32")
    e2v = up(np.arange(n, dtype=np.uint32), "uint32")
    arrays = [dev.zeros(2 * GUARD + m, "float64") for m in (9 * n, 81 * n, 81 * n, 81 * n * 6, 9 * n)]
    for a in arrays:                  # gradient, blocks, diagonal blocks, staged blocks and gradient
        a.fill_(7.25)
    at = [dev.ptr(a) + 8 * GUARD for a in arrays]
    keep = [up(idx.astype(np.uint32).ravel(), "uint32"), up(size.astype(np.uint16).ravel(), "uint16"),
            up(perm.astype(np.int16).ravel(), "int16")]
    sa = _lib.ScatterArgs(dev.ptr(keep[0]), dev.ptr(keep[1]), dev.ptr(keep[2]), dev.ptr(lookups),
                          dev.ptr(outer), K, 1, dev.ptr(diag), dev.ptr(starts), at[0], at[1], at[2],
                          at[3], at[4], 9)
    u = _lib.UnionF64(1, 9, dev.ptr(count))
    u.data[0] = dev.ptr(bodies)
    scene = up(np.array([1.0]), "float64")
    rc = lib.ysp_eval_element_energy(KIND_IDS["affine_orthogonality"], C.byref(u), None, dev.ptr(e2v), n,
                                     dev.ptr(scene), dev.ptr(scene), method, C.byref(sa), dev.stream())
    assert rc == 0
    assert lib.ysp_check_deferred(dev.stream()) == ERR_UNSUPPORTED
    for a in arrays:
        assert bool((a == 7.25).all())
    assert lib.ysp_check_deferred(dev.stream()) == 0
