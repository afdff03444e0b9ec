"""Row tiles (64 consecutive cells of one row per wavefront) against the plane
tiling (64 consecutive cells of a plane, taken where lbm_set_index_width asks
for 64-bit elements). Both give every cell the same arithmetic, so the fields
must agree bit for bit: at row lengths one short of, equal to and one past a
multiple of 64 cells, at the shortest rows that take row tiles, with walls,
solids and every periodic axis, in both layouts."""
import numpy as np
import pytest

from lbm_amd import capi, scenario, workloads

pytestmark = pytest.mark.gpu

# fp32, fp64 and 16-bit rows are padded (not packed) from 62, 30 and 126 cells
CASES = [(x, "f32") for x in (62, 63, 64, 65, 96, 127, 128, 129)]
CASES += [(x, "f64") for x in (32, 33, 64, 65)] + [(x, "f64s") for x in (40, 64)]
CASES += [(x, "f16") for x in (126, 128, 130)] + [(x, "bf16") for x in (127, 192)]


def run(dims, storage, q, layout, geometry, width):
    periodic = (True,) * 3 if geometry == "box" else (False,) * 3
    d = capi.Domain(*dims, 0.7, q=q, storage=storage, layout=layout, periodic=periodic)
    if geometry == "cavity":
        scenario.cavity(*dims, lid=(0.05, 0.02, 0.0)).apply(d)
    elif geometry == "channel":
        workloads.sphere_channel(*dims, seed=3).apply(d)
    d.set_index_width(width)
    d.finalize()
    if layout == "ab":
        d.set_time_blocking(1)
    rng = np.random.default_rng(9)
    shape = dims[::-1]
    d.init_equilibrium(1 + 0.02 * rng.random(shape), 0.02 * rng.standard_normal(shape + (3,)))
    d.step(5)
    out = d.get_pdf()
    d.close()
    return out.view(np.uint64)


@pytest.mark.parametrize("layout", ["ab", "aa"])
@pytest.mark.parametrize("x,storage", CASES)
def test_row_tiles_equal_plane_tiles(x, storage, layout):
    for geometry, q in (("box", 19), ("cavity", 19), ("channel", 27)):
        dims = (x, 9, 7) if geometry != "channel" else (x, 12, 11)
        print("row tiles:", dims, storage, layout, geometry, q, flush=True)
        rows, planes = (run(dims, storage, q, layout, geometry, w) for w in (32, 64))
        np.testing.assert_array_equal(rows, planes)


# fields beyond 32 MiB, whose cell tiles sweep every other step backwards:
# padded rows (row tiles) and packed ones (plane tiles), plane counts that
# leave a remainder of tiles
@pytest.mark.parametrize("dims,storage", [((97, 83, 61), "f32"), ((60, 91, 87), "f32"), ((130, 101, 71), "f16"),
                                          ((61, 59, 37), "f64s")])
@pytest.mark.parametrize("geometry", ["box", "cavity"])
def test_turning_sweeps(dims, storage, geometry):
    fields = []
    for layout, spp in (("ab", 1), ("aa", 0), ("ab", 2)):
        if spp == 2 and storage == "f64s":
            continue
        print("sweeps:", dims, storage, geometry, layout, spp, flush=True)
        d = capi.Domain(*dims, 0.7, storage=storage, layout=layout, periodic=(geometry == "box",) * 3)
        if geometry == "cavity":
            scenario.cavity(*dims, lid=(0.05, 0.02, 0.0)).apply(d)
        d.finalize()
        if layout == "ab":
            d.set_time_blocking(spp)
        rng = np.random.default_rng(5)
        d.init_equilibrium(1 + 0.02 * rng.random(dims[::-1]), 0.02 * rng.standard_normal(dims[::-1] + (3,)))
        d.step(3)
        d.step(4)
        fields.append([m.view(np.uint64) for m in d.moments()])
        d.close()
    for f in fields[1:]:
        for got, want in zip(f, fields[0]):
            np.testing.assert_array_equal(got, want)


def test_turning_sweeps_of_a_batch():
    sizes = [(33 + 4 * i, 40, 31 + 3 * i) for i in range(12)]  # 12 cavities, 114 MB a buffer

    def domains():
        out = []
        for s in sizes:
            d = capi.Domain(*s, 0.7, storage="f32")
            scenario.cavity(*s, lid=(0.05, 0.02, 0.0)).apply(d)
            d.finalize()
            out.append(d)
        return out

    alone, together = domains(), domains()
    for d in alone:
        d.set_time_blocking(1)
        d.step(7)
    with_batch = capi.Batch(together)
    with_batch.step(3)
    with_batch.step(4)
    for a, b in zip(alone, together):
        for x, y in zip(a.moments(), b.moments()):
            np.testing.assert_array_equal(x.view(np.uint64), y.view(np.uint64))
    with_batch.close()
    for d in alone + together:
        d.close()
