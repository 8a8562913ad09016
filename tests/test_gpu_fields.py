"""Fields read back in the order of the upload, whatever the list builds have
made of the order on the device."""
import numpy as np
import pytest

from fjsph_amd import abi, cases
from tests.test_gpu_parity import _engine, _small_cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [abi.STATE_NP1, abi.STATE_N], ids=["np1", "n"])
@pytest.mark.parametrize("name", ["drop3d", "dam2d", "large"])
def test_host_order(name, which):
    """"large" has more particles than are reordered by one launch a state."""
    case = dict(_small_cases()).get(name) or cases.fluid_block(2, 560, dx=1e-3, precision=abi.PREC_MIXED, H_fac=2.0)
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


@pytest.mark.parametrize("n", [64, 1023, 2048, 2049, 4097])
def test_state_copy(n):
    """The step's end copies one state over the other in one launch: sizes
    around the launch's blocks of 16 KB (2048 scalars, 4096 integers), odd
    ones with a remainder of 4 and 8 B."""
    case = cases.fluid_block(3, 17, dx=1e-3, precision=abi.PREC_FP64, H_fac=2.0, sig=0.07)
    for f in ("x", "v", "rho", "p", "m", "b"):
        setattr(case, f, np.ascontiguousarray(getattr(case, f)[:n]))
    case.blocks = [dict(first=0, last=n, is_fluid=1)]
    print(f"[fields] state copy n={n}", flush=True)
    eng = _engine(case)
    eng.integrate_no_update()
    eng.integrate_step()
    for f in abi.F:
        assert np.array_equal(eng.field(f, abi.STATE_N), eng.field(f, abi.STATE_NP1)), f
    eng.close()


def test_a_growing_set_gives_its_spare_state_back():
    """Small sets keep buffers for a whole state's reordering; a set that
    grows past the size up to which they are used frees them.  They are more
    than the growth of everything else here, so the context shrinks."""
    import ctypes as C
    case = cases.pipe_inlet_3d(diameter=9.1e-3, dx=5e-5, mode=0, precision=abi.PREC_MIXED, exit_to_delete=100.0)
    print(f"[fields] growing set n={case.n}", flush=True)
    assert case.n < 300_000
    eng = _engine(case)
    eng.set_reorder_interval(1)
    eng.integrate_no_update()
    eng.integrate_step()

    def free():
        b, total = C.c_size_t(), C.c_size_t()
        assert eng.lib.hipMemGetInfo(C.byref(b), C.byref(total)) == 0
        return b.value

    before = free()
    for _ in range(30):
        eng.integrate_step()
        if eng.n > case.n:
            break
    assert eng.n > 300_000
    eng.integrate_step()
    assert free() > before
    eng.close()
