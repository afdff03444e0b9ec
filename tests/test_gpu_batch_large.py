"""Batches whose buffers take more than 2 GiB at fp32, most of it in packed rows
between walls, step with the pulls sent ahead of the cell kinds: every domain's
field is that of the domain stepped alone, bit for bit. One domain brings the
size, the others the conditions: edges between lids, walls, inflow, outflow and
pressure, more conditions than a rule word names, solid cells and a periodic
axis."""
import numpy as np
import pytest

from lbm_amd import capi, scenario

pytestmark = pytest.mark.gpu

X, Y, Z = 70, 10, 9
REST = (0.0, 0.0, 0.0, 1.0)
FACES = {"x0": (0, 0, 0, Y + 1, 0, Z + 1), "xmax": (X + 1, X + 1, 0, Y + 1, 0, Z + 1),
         "y0": (0, X + 1, 0, 0, 0, Z + 1), "ymax": (0, X + 1, Y + 1, Y + 1, 0, Z + 1),
         "z0": (0, X + 1, 0, Y + 1, 0, 0), "zmax": (0, X + 1, 0, Y + 1, Z + 1, Z + 1)}
LID, LID2 = (capi.MOVINGWALL, (0.05, 0.01, 0.0, 1.0)), (capi.MOVINGWALL, (0.03, 0.0, 0.02, 1.0))
FLOW = {"x0": (capi.INFLOW, (0.04, 0.0, 0.0, 1.0)), "xmax": (capi.OUTFLOW, REST)}
GEOMETRIES = {
    "walls": {},
    "two lids": {"zmax": LID, "ymax": LID2},
    "channel with a lid": {**FLOW, "ymax": LID},
    "pressure": {"x0": FLOW["x0"], "xmax": (capi.PRESSURE, (0.0, 0.0, 0.0, 1.01)), "zmax": LID},
    "many lids": {},
    "periodic z": {"y0": LID},
}


def small(geometry):
    d = capi.Domain(X, Y, Z, 0.8, q=19, storage="f32", periodic=(0, 0, geometry == "periodic z"))
    if geometry == "walls":
        mask = np.ones((Z, Y, X), dtype=np.uint8)
        mask[2:5, 3:7, 20:33] = 0
        d.set_solid_mask(mask)
    for face, box in FACES.items():
        if geometry != "periodic z" or face[0] != "z":
            d.set_boundary_box(capi.NOSLIP, REST, *box)
    for face, cond in GEOMETRIES[geometry].items():
        d.set_boundary_box(*cond, *FACES[face])
    if geometry == "many lids":
        for x in range(1, 46):
            d.set_boundary_box(capi.MOVINGWALL, (0.001 * x, 0.0, 0.0, 1.0), x, x, 0, Y + 1, Z + 1, Z + 1)
    return d


def domains():
    big = (61, 700, 360)  # packed: fewer than 64 values a row with the ghosts
    doms = [small(g) for g in GEOMETRIES] + [capi.Domain(*big, 0.7, q=19, storage="f32")]
    scenario.cavity(*big, lid=(0.05, 0.02, 0.0)).apply(doms[-1])
    rng = np.random.default_rng(11)
    for d in doms:
        d.finalize()
        d.set_time_blocking(1)
        shape = (d.zl, d.yl, d.xl)
        d.init_equilibrium(1 + 0.02 * rng.random(shape), 0.02 * rng.standard_normal(shape + (3,)))
    return doms


def test_large_batch_equals_domains_alone():
    batched, alone = domains(), domains()
    assert 2 * sum(d.info()["field_bytes"] for d in batched) > 2 << 30
    b = capi.Batch(batched)
    for n in (7, 4):
        print("large batch:", n, "steps", flush=True)
        b.step(n)
        b.sync()
        for d in alone:
            d.step(n)
        for got, ref, name in zip(batched, alone, [*GEOMETRIES, "large cavity"]):
            for x, y in zip(got.moments(), ref.moments()):
                assert np.array_equal(x.view(np.uint64), y.view(np.uint64)), name
            if name in GEOMETRIES:
                x, y = (d.get_pdf()[1:-1, 1:-1, 1:-1] for d in (got, ref))
                assert np.array_equal(np.ascontiguousarray(x).view(np.uint64), np.ascontiguousarray(y).view(np.uint64)), name
    assert not b.status().any()
    b.close()
    for d in batched + alone:
        d.close()
