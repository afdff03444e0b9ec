"""lbm_init_equilibrium restarts a domain: whatever the domain did before (steps
in either form, fields read, a field written), the run that follows is that of
a new domain with the same initial fields, bit for bit, in both layouts. The
first step takes stored values from the non-fluid cells, so these are part of
it: in the walls' faces, in solid cells inside the box, and where an earlier
two-step pass or an earlier read wrote rule values."""
import numpy as np
import pytest

from lbm_amd import capi, scenario

pytestmark = pytest.mark.gpu

SHAPE = (70, 12, 10)


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def domain(storage, layout, spp, solid):
    d = capi.Domain(*SHAPE, 0.6, q=19, storage=storage, layout=layout)
    if solid:
        mask = np.ones(SHAPE[::-1], dtype=np.uint8)
        mask[3:5, 4:7, 20:24] = 0
        d.set_solid_mask(mask)
    scenario.cavity(*SHAPE, lid=(0.05, 0.02, 0.0)).apply(d)
    d.finalize()
    d.set_time_blocking(spp)
    return d


def fields(seed):
    rng = np.random.default_rng(seed)
    return 1 + 0.02 * rng.random(SHAPE[::-1]), 0.02 * rng.standard_normal(SHAPE[::-1] + (3,))


def run(d, seed, steps=5):
    d.init_equilibrium(*fields(seed))
    d.step(steps)
    return d.moments() + (d.get_pdf(),)


BEFORE = {
    "steps": lambda d: d.step(7),
    "moments": lambda d: (d.step(6), d.moments()),
    "whole field": lambda d: (d.step(6), d.get_pdf()),
    "written field": lambda d: d.set_pdf(d.get_pdf() * 1.01),
}


@pytest.mark.parametrize("before", sorted(BEFORE))
@pytest.mark.parametrize("solid", [False, True])
@pytest.mark.parametrize("storage,layout,spp", [("f64", "ab", 0), ("f32", "ab", 1), ("f32", "ab", 2), ("f16", "ab", 2),
                                                ("f32", "aa", 0)])
def test_restart_equals_a_new_domain(storage, layout, spp, solid, before):
    fresh = domain(storage, layout, spp, solid)
    ref = run(fresh, 2)
    fresh.close()
    used = domain(storage, layout, spp, solid)
    used.init_equilibrium(*fields(1))
    BEFORE[before](used)
    got = run(used, 2)
    used.close()
    # (ghost cells that serve no fluid cell are never read: edges keep what was written)
    inner = (slice(1, -1),) * 3
    for a, b in zip(got[:2] + (got[2][inner],), ref[:2] + (ref[2][inner],)):
        assert np.array_equal(bits(a), bits(b))


@pytest.mark.parametrize("layout", ["ab", "aa"])
def test_restart_after_reads_equals_the_oracle(layout):
    """fp64 in the reference's operation order, against the CPU oracle started
    anew with the field the restart writes."""
    from oracle import ora
    d = domain("f64", layout, 0, False)
    d.init_equilibrium(*fields(1))
    d.step(4)
    d.moments()
    d.init_equilibrium(*fields(2))
    f0 = d.get_pdf()
    o = ora.OracleDomain(*SHAPE, 0.6, q=19)
    scenario.cavity(*SHAPE, lid=(0.05, 0.02, 0.0)).apply(o)
    o.finalize()
    start = o.get_pdf()
    start[1:-1, 1:-1, 1:-1] = f0[1:-1, 1:-1, 1:-1]
    o.set_pdf(start)
    d.step(5)
    o.step(5)
    inner = (slice(1, -1),) * 3
    assert np.array_equal(bits(d.get_pdf()[inner]), bits(o.get_pdf()[inner]))
    d.close()
    o.close()
