"""Fields read back in the order of the upload, whatever the list builds have
made of the order on the device."""
import numpy as np
import pytest

from fjsph_amd import abi
from tests.test_gpu_parity import _engine, _small_cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [abi.STATE_NP1, abi.STATE_N], ids=["np1", "n"])
@pytest.mark.parametrize("name", ["drop3d", "dam2d"])
def test_host_order(name, which):
    case = dict(_small_cases())[name]
    print(f"[fields] {name} n={case.n}", flush=True)
    eng = _engine(case)
    x0, dim = eng.field("X"), case.settings.dim
    eng.integrate_no_update()
    for _ in range(3):
        eng.integrate_step()
    assert np.abs(eng.field("X", which) - x0).max() < case.settings.particle_step
    k = np.arange(eng.n, dtype=np.float64)
    for f, v in (("P", k), ("V", np.stack([k + a for a in range(dim)], 1)), ("CELLID", k),
                 ("L", k[:, None] + np.arange(dim * dim) / 16)):
        eng.set_field(f, v, which)
        assert np.array_equal(eng.field(f, which), v), f
    eng.close()
