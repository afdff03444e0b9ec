"""Which form the cell tiles take by the share of x lines with links
(StepPlan::ahead), and in place by how full row tiles are (StepPlan::aa_rows):
on either side of each line, the bits of the build with 64-bit element indices,
which has plane tiles and reads the link words first."""
import numpy as np
import pytest

from lbm_amd import capi, scenario

pytestmark = pytest.mark.gpu

REST = (0.0, 0.0, 0.0, 1.0)
LID = (0.05, 0.01, 0.0, 1.0)
# name: periodic axes, faces (kind, parameters)
GEOMETRIES = {
    "box": ((1, 1, 1), {}),
    "plates": ((1, 1, 0), {"z0": (capi.NOSLIP, REST), "zmax": (capi.MOVINGWALL, LID)}),
    "duct": ((1, 0, 0), {"y0": (capi.NOSLIP, REST), "ymax": (capi.NOSLIP, REST), "z0": (capi.NOSLIP, REST),
                         "zmax": (capi.MOVINGWALL, LID)}),
    "x plates": ((0, 1, 1), {"x0": (capi.NOSLIP, REST), "xmax": (capi.MOVINGWALL, (0.0, 0.05, 0.02, 1.0))}),
    "open ends": ((0, 1, 0), {"z0": (capi.NOSLIP, REST), "zmax": (capi.NOSLIP, REST),
                              "x0": (capi.INFLOW, (0.04, 0.0, 0.0, 1.0)), "xmax": (capi.OUTFLOW, REST)}),
    "block": ((1, 1, 1), {}),
}
STORAGES = ["f32", "f64", "f64s", "f16", "bf16"]


def run(geometry, shape, q, storage, layout="ab", width=32, steps=7):
    per, faces = GEOMETRIES[geometry]
    d = capi.Domain(*shape, 0.8, q=q, storage=storage, periodic=per, layout=layout)
    if geometry == "block":
        mask = np.ones(shape[::-1], dtype=np.uint8)
        mask[2:4, 3:5, 5:12] = 0
        d.set_solid_mask(mask)
    sc = scenario.Scenario(geometry, *shape)
    for face, (kind, p) in faces.items():
        sc.boundaries.append(scenario.Boundary(kind, p, scenario.face_box(face, *shape), "", face))
    sc.apply(d)
    d.finalize()
    d.set_time_blocking(1)
    d.set_index_width(width)
    rng = np.random.default_rng(3)
    d.init_equilibrium(1 + 0.02 * rng.random(shape[::-1]), 0.02 * rng.standard_normal(shape[::-1] + (3,)))
    d.step(steps)
    out = d.get_pdf()[1:-1, 1:-1, 1:-1]
    d.close()
    return np.ascontiguousarray(out).view(np.uint64)


# packed rows and row tiles; the share of lines with links is below a third for
# plates, the block and the 12 x 13 x 11 duct, above for the 131 x 12 x 9 duct
@pytest.mark.parametrize("storage", STORAGES)
@pytest.mark.parametrize("geometry", list(GEOMETRIES))
def test_cell_tiles_equal_64_bit_build(geometry, storage):
    for q in (15, 19, 27):
        for shape in ((12, 13, 11), (131, 12, 9)):
            print("cell forms:", geometry, storage, q, shape, flush=True)
            np.testing.assert_array_equal(run(geometry, shape, q, storage), run(geometry, shape, q, storage, width=64))


# rows in place: full tiles (128), a nearly empty last one (131), three quarters (144)
@pytest.mark.parametrize("storage", STORAGES)
@pytest.mark.parametrize("geometry", list(GEOMETRIES))
def test_in_place_tiles_equal_64_bit_build(geometry, storage):
    for x in (128, 131, 144):
        for steps in (6, 7):
            print("in place:", geometry, storage, x, steps, flush=True)
            a, b = (run(geometry, (x, 10, 9), 19, storage, layout="aa", width=w, steps=steps) for w in (32, 64))
            np.testing.assert_array_equal(a, b)
