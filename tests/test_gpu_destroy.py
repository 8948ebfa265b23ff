"""EmDeeGPU_destroy gives back all device memory of a system, its rigid bodies' included."""
import ctypes

import numpy as np
import pytest

from emdee_amd.water_box import water_box, MASS, CHARGE, EPS_OO, SIG_OO, KCOUL

pytestmark = pytest.mark.gpu

NMOL = 8000


@pytest.mark.parametrize("rigid", [True, False])
def test_memory_returns(gpu, rigid):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    R, types, mol, L = water_box(NMOL, 2)

    def cycle():
        md = gpu.system(1, 1, 7.0, 1.0, 3 * NMOL, types, MASS, mol if rigid else None)
        gpu.EmDee_set_pair_model(md, 1, 1, gpu.EmDee_pair_lj_cut(EPS_OO, SIG_OO), KCOUL)
        gpu.EmDee_set_pair_model(md, 2, 2, gpu.EmDee_pair_none(), KCOUL)
        gpu.EmDee_set_coul_model(md, gpu.EmDee_coul_damped(0.3))
        gpu.upload(md, "charges", CHARGE[types - 1])
        gpu.upload(md, "coordinates", R)
        gpu.upload(md, "box", np.array([L]))
        gpu.EmDeeGPU_destroy(ctypes.byref(md))
        assert gpu.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    base = min(cycle() for _ in range(4))
    last = max([cycle() for _ in range(64)][-4:])
    # a system's body arrays are 7 doubles per atom and 36 per body, 3.6 MB: 64 systems that kept theirs would be short
    # of 230 MB; the card's free memory itself moves by some 40 MB either way
    assert base - last < 100 << 20
