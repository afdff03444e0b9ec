"""lbm_moments and lbm_init_equilibrium pass their arrays in chunks of 2^17
cells through several host threads: every cell arrives, at sizes around one
chunk and one thread, with either output left out, and from several calling
threads at once. lbm_moments_noalloc (one kernel, one plain copy) is the
reference, bit for bit."""
import ctypes
import threading

import numpy as np
import pytest

from lbm_amd import capi, scenario

pytestmark = pytest.mark.gpu


def domain(shape, storage="f32", solid=False):
    d = capi.Domain(*shape, 0.6, q=19, storage=storage)
    if solid:
        mask = np.ones(shape[::-1], dtype=np.uint8)
        mask[1:3, 1:4, 2:5] = 0
        d.set_solid_mask(mask)
    scenario.cavity(*shape, lid=(0.05, 0.0, 0.0)).apply(d)
    d.finalize()
    return d


def fields(shape, seed):
    rng = np.random.default_rng(seed)
    return 1 + 1e-2 * rng.standard_normal(shape[::-1]), 0.02 * rng.standard_normal(shape[::-1] + (3,))


# 2^17 = 64 * 64 * 32 cells a chunk; 2^15 cells a MiB
@pytest.mark.parametrize("solid", [False, True])
@pytest.mark.parametrize("shape", [(5, 6, 7), (32, 32, 31), (64, 64, 32), (131, 67, 15), (64, 64, 33), (101, 97, 107)])
def test_every_cell_arrives(shape, solid):
    rho, u = fields(shape, 1)
    d = domain(shape, "f64s", solid)
    d.init_equilibrium(rho, u)
    r, v = d.moments()
    fluid = np.ones(shape[::-1], dtype=bool)
    if solid:
        fluid[1:3, 1:4, 2:5] = False
    # sums of 19 fp64 values near 1/36 .. 1/3 that make up rho and rho u
    assert np.abs(r - rho)[fluid].max() < 1e-13 and np.abs(v - u)[fluid].max() < 1e-13
    d.step(3)
    r, v = d.moments()
    r0, v0 = d.moments_noalloc()
    assert np.array_equal(r.view(np.uint64), r0.view(np.uint64))
    assert np.array_equal(v.view(np.uint64), v0.view(np.uint64))
    lib, ptr = capi.load(), lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    r1, v1 = np.empty_like(r), np.empty_like(v)
    assert lib.lbm_moments(d._h, ptr(r1), None) == 0 and lib.lbm_moments(d._h, None, ptr(v1)) == 0
    assert np.array_equal(r1, r) and np.array_equal(v1, v)
    d.close()


def test_domains_on_several_threads():
    shapes = [(40, 41, 42), (70, 60, 50), (20, 21, 22), (90, 50, 40)]
    doms = [domain(s) for s in shapes]
    bad = []

    def work(i):
        rho, u = fields(shapes[i], i)
        for _ in range(5):
            doms[i].init_equilibrium(rho, u)
            doms[i].step(2)
            out.setdefault(i, []).append(doms[i].moments())

    out = {}
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(doms))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, d in enumerate(doms):
        ref = d.moments_noalloc()
        for got in out[i]:
            bad += [i] * (not all(np.array_equal(a, b) for a, b in zip(got, ref)))
        d.close()
    assert not bad
