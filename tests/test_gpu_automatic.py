"""The automatic setting on either side of each line between single steps and
two-step passes: lbm_get_steps_per_launch names the form that lbm_step takes,
and both forms give the bits of single steps."""
import ctypes

import numpy as np
import pytest

from lbm_amd import capi, scenario

MIB = 1 << 20


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def test_steps_per_launch_refuses_null():
    n = ctypes.c_int()
    assert capi.load().lbm_get_steps_per_launch(None, ctypes.byref(n)) == -1


# periodic: 3 * 2^16 cells; walls, every cell fluid: both buffers over 256 MiB
# (112^3 and 120^3 cavities; 96^3 and 100 x 100 x 60 are within it); walls and
# solid cells in the box: 3 000 000 cells
LINES = [
    ((64, 64, 47), "periodic", 1), ((64, 64, 48), "periodic", 2),
    ((12, 12, 12), "walls", 1), ((96, 96, 96), "walls", 1), ((100, 100, 60), "walls", 1),
    ((112, 112, 112), "walls", 1), ((120, 120, 120), "walls", 2),
    ((208, 120, 120), "solids", 1), ((209, 120, 120), "solids", 2),
]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,kind,steps", LINES)
def test_form_taken_and_its_bits(shape, kind, steps):
    per = (int(kind == "periodic"),) * 3
    fluid = np.ones(shape[::-1], dtype=np.uint8)
    if kind == "solids":
        fluid[3:9, 4:30, 20:41] = 0
    out = []
    for spp in (0, 1):
        d = capi.Domain(*shape, 0.6, q=19, storage="f32", periodic=per)
        if kind == "solids":
            d.set_solid_mask(fluid)
        if kind != "periodic":
            scenario.cavity(*shape, lid=(0.05, 0.02, 0.0)).apply(d)
        with pytest.raises(KeyError):
            d.info()["steps_per_launch"]
        d.finalize()
        d.set_time_blocking(spp)
        info = d.info()
        assert info["steps_per_launch"] == (1 if spp else steps)
        if spp == 0 and kind == "walls" and shape[0] > 100:
            assert (2 * info["field_bytes"] > 256 * MIB) == (steps == 2)
        if spp == 0:
            d.set_time_blocking(2)
            assert d.info()["steps_per_launch"] == 2
            d.set_time_blocking(0)
        rng = np.random.default_rng(3)
        d.init_equilibrium(1 + 1e-3 * rng.standard_normal(shape[::-1]), 0.02 * rng.standard_normal(shape[::-1] + (3,)))
        d.step(7)
        out.append(d.moments())
        d.close()
    m = fluid.astype(bool)
    for a, b in zip(*out):
        assert np.array_equal(bits(a[m]), bits(b[m]))
