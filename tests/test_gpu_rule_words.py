"""Cells whose links that are not NoSlip share one condition take its values
together (the rule words of lbm_finalize), in the cell tiles and before a
walled pass. The near-boundary list kernel, which evaluates link after link,
is the reference, bit for bit on every fluid cell: edges between lids, walls,
inflow and outflow, edges of two different lids, conditions beyond the 31 that
a rule word can name, and FreeSlip beside a lid."""
import numpy as np
import pytest

from lbm_amd import capi

pytestmark = pytest.mark.gpu

X, Y, Z = 131, 10, 9  # padded rows in every storage, of more than one tile
REST = (0.0, 0.0, 0.0, 1.0)
FACES = {"x0": (0, 0, 0, Y + 1, 0, Z + 1), "xmax": (X + 1, X + 1, 0, Y + 1, 0, Z + 1),
         "y0": (0, X + 1, 0, 0, 0, Z + 1), "ymax": (0, X + 1, Y + 1, Y + 1, 0, Z + 1),
         "z0": (0, X + 1, 0, Y + 1, 0, 0), "zmax": (0, X + 1, 0, Y + 1, Z + 1, Z + 1)}
LID, LID2 = ("movingwall", (0.05, 0.01, 0.0, 1.0)), ("movingwall", (0.03, 0.0, 0.02, 1.0))
FLOW = {"x0": ("inflow", (0.04, 0.0, 0.0, 1.0)), "xmax": ("outflow", REST)}
GEOMETRIES = {
    "lid": {"zmax": LID},
    "two lids": {"zmax": LID, "ymax": LID2},
    "channel": FLOW,
    "channel with a lid": {**FLOW, "ymax": LID},
    "pressure": {"x0": FLOW["x0"], "xmax": ("pressure", (0.0, 0.0, 0.0, 1.01)), "zmax": LID},
    "many lids": {"zmax": None},
    "freeslip": {"zmax": LID, "y0": ("freeslip", REST)},
}
KIND = {"noslip": capi.NOSLIP, "movingwall": capi.MOVINGWALL, "inflow": capi.INFLOW, "outflow": capi.OUTFLOW,
        "pressure": capi.PRESSURE, "freeslip": capi.FREESLIP}


def run(geometry, storage, q, vec=0, spp=1):
    d = capi.Domain(X, Y, Z, 0.8, q=q, storage=storage)
    for face, box in FACES.items():
        d.set_boundary_box(KIND["noslip"], REST, *box)
    for face, cond in GEOMETRIES[geometry].items():
        if cond:
            d.set_boundary_box(KIND[cond[0]], cond[1], *FACES[face])
    if geometry == "many lids":
        for x in range(1, 46):
            d.set_boundary_box(KIND["movingwall"], (0.001 * x, 0.0, 0.0, 1.0), x, x, 0, Y + 1, Z + 1, Z + 1)
    d.finalize()
    d.set_tuning(vec)
    d.set_time_blocking(spp)
    rng = np.random.default_rng(5)
    d.init_equilibrium(1 + 0.02 * rng.random((Z, Y, X)), 0.02 * rng.standard_normal((Z, Y, X, 3)))
    d.step(7)
    out = d.get_pdf()[1:-1, 1:-1, 1:-1]
    d.close()
    return np.ascontiguousarray(out).view(np.uint64)


@pytest.mark.parametrize("storage", ["f32", "f16", "bf16", "f64", "f64s"])
@pytest.mark.parametrize("geometry", list(GEOMETRIES))
def test_rule_words_equal_links_one_by_one(geometry, storage):
    for q in (15, 19, 27):
        print("rule words:", geometry, storage, q, flush=True)
        ref = run(geometry, storage, q, vec=4 if storage in ("f16", "bf16") else 1)
        np.testing.assert_array_equal(run(geometry, storage, q), ref)
        if storage in ("f32", "f16", "bf16") and geometry != "freeslip":
            np.testing.assert_array_equal(run(geometry, storage, q, spp=2), ref)
