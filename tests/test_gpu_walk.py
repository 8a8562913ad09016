"""List walks at the edges of their rows: isolated clusters of k particles, so
that every target has k - 1 neighbours (no row at all, rows of one to four
entries, a second row with one) and the waves mix lanes with and without
entries.  Pair sums against the oracle; FP64 to summation order, mixed to the
FP32 pair terms (as test_gpu_parity.py).  And blocks short enough that two or
four waves share a target's list."""
import numpy as np
import pytest

from fjsph_amd import abi, cases
from tests.parity import assert_close, same_neighbour_sets
from tests.test_gpu_parity import FP64_PASS, FP64_STEP, MIXED_STEP, _engine, _oracle, _small_cases

pytestmark = pytest.mark.gpu

SIZES = (1, 2, 3, 4, 5, 6, 8, 9, 13)


def _clusters(dim, sizes, precision, ale):
    dx = 1e-3
    c = cases.fluid_block(dim, 2, dx=dx, precision=precision, H_fac=2.0, sig=0.07)
    s = c.settings
    s.ale = ale
    rng = np.random.default_rng(17)
    pts, k = [], 0
    for rep in range(6):
        for size in sizes:
            at = np.array([k % 8, (k // 8) % 8, 0.0])[:dim] * 12 * dx
            # well separated points of a cluster: a jittered corner of the lattice
            g = np.array([[i, j, m][:dim] for m in range(3) for j in range(3) for i in range(2)], dtype=float)
            g = np.unique(g, axis=0)
            g = g[rng.permutation(len(g))[:min(size, len(g))]]
            pts.append(at + dx * (g + rng.uniform(-0.1, 0.1, g.shape)))
            k += 1
    x = np.concatenate(pts)
    n = len(x)
    c.x = np.ascontiguousarray(x)
    c.v = rng.uniform(-0.1, 0.1, x.shape)
    c.rho = s.rho_rest * (1.0 + rng.uniform(-5e-3, 5e-3, n))
    b = s.rho_rest * s.speed_sound ** 2 / s.gam
    c.p = b * ((c.rho / s.rho_rest) ** s.gam - 1.0)
    c.m = np.full(n, s.rho_rest * dx ** dim)
    c.b = np.full(n, abi.FREE, dtype=np.int32)
    c.n_bound = 0
    c.blocks = [dict(first=0, last=n, is_fluid=1)]
    return c


@pytest.mark.parametrize("precision", [abi.PREC_FP64, abi.PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("dim,ale,sizes", [(2, 0, SIZES), (3, 0, SIZES), (3, 1, SIZES), (3, 0, (1,))],
                         ids=["2d", "3d", "3d-ale", "3d-lone"])
def test_row_remainders(dim, ale, sizes, precision):
    case = _clusters(dim, sizes, precision, ale)
    print(f"[walk] {dim}D ale={ale} sizes={sizes} n={case.n} precision={precision}", flush=True)
    eng, orc = _engine(case), _oracle(case)
    eng.build_neighbours()
    orc.build_neighbours()
    off_e, idx_e = eng.neighbours()
    off_o, idx_o, _ = orc.neighbours()
    assert same_neighbour_sets(off_e, idx_e, off_o, idx_o)
    tol = FP64_PASS if precision == abi.PREC_FP64 else MIXED_STEP
    npd_e, npd_o = eng.dsph_prestep(), orc.dsph_prestep()
    assert abs(npd_e - npd_o) <= tol * abs(npd_o)
    # sums that do not pass through the correction matrix, whose inverse is
    # ill-conditioned for a handful of neighbours
    for f in ("KERNSUM", "COLOUR"):
        assert_close(f, eng.field(f), orc.field(f), tol)
    eng.detect_surface()
    orc.detect_surface()
    assert np.array_equal(eng.field("SURF"), orc.field("SURF"))
    eng.dissipation_terms()
    orc.dissipation_terms()
    assert_close("AVISC", eng.field("AVISC"), orc.field("AVISC"), tol)
    if sizes == (1,):
        npd_o = 1.0 / case.settings.particle_step ** dim  # no pair gives it
    eng.acc_rrho(npd_o)
    orc.acc_rrho(npd_o)
    assert_close("ACC", eng.field("ACC"), orc.field("ACC"), tol)
    eng.close()


@pytest.mark.parametrize("precision", [abi.PREC_FP64, abi.PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("targets", [16, 64, 128, 192])
@pytest.mark.parametrize("name", ["dam2d", "jet3d_ale", "drop3d"])
def test_shared_lists(name, targets, precision):
    """Start-up pass and two steps with blocks of few targets: in mixed
    precision four waves to a list (16, 64), two (128), one (192), and a run's
    mixture of them."""
    case = dict(_small_cases())[name]
    case.settings.precision = precision
    print(f"[walk] {name}: n={case.n} {targets} targets a block, precision={precision}", flush=True)
    eng, orc = _engine(case), _oracle(case)
    eng.set_block_targets(targets)
    eng.integrate_no_update()
    orc.integrate_no_update()
    for _ in range(2):
        ie, io = eng.integrate_step(), orc.integrate_step()
        if precision == abi.PREC_FP64:
            assert ie["iterations"] == io["iterations"]
    tol = FP64_STEP if precision == abi.PREC_FP64 else MIXED_STEP
    assert np.array_equal(eng.field("SURF"), orc.field("SURF"))
    for f in ("X", "V", "RHO", "ACC", "RRHO", "LAM", "AVISC"):
        assert_close(f, eng.field(f), orc.field(f), tol)
    eng.close()


@pytest.mark.parametrize("precision", [abi.PREC_FP64, abi.PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("targets", [0, 8, 70, 512])
@pytest.mark.parametrize("cells", [(9, 1), (1, 9), (12, 9), (300, 2), (7, 1, 1), (1, 1, 7), (2, 9, 1), (5, 4, 6)],
                         ids=lambda c: "x".join(map(str, c)))
def test_block_shapes(cells, targets, precision):
    """Neighbour sets for clouds of every aspect (cut-off cells along the
    axes), blocks of one cell to the whole cloud.  Half the particles lie on
    a lattice whose step divides the cut-off, so that some pairs are a
    rounding from it on either side."""
    dim, dx = len(cells), 1e-3
    c = cases.fluid_block(dim, 2, dx=dx, precision=precision, H_fac=2.0, sig=0.07)
    rng = np.random.default_rng(5)
    step = dx * (dim - 1)
    g = np.stack(np.meshgrid(*[np.arange(max(1, round((4 * k - 1) * dx / step))) for k in cells], indexing="ij"), -1)
    g = g.reshape(-1, dim) * step
    loose = rng.random(len(g)) < 0.5
    g[loose] += rng.uniform(-0.4, 0.4, (loose.sum(), dim)) * step
    c.x = np.ascontiguousarray(g[rng.permutation(len(g))])
    n = len(c.x)
    c.v, c.rho, c.p = np.zeros((n, dim)), np.full(n, c.settings.rho_rest), np.zeros(n)
    c.m, c.b = np.full(n, c.settings.rho_rest * dx ** dim), np.full(n, abi.FREE, dtype=np.int32)
    c.n_bound, c.blocks = 0, [dict(first=0, last=n, is_fluid=1)]
    print(f"[walk] cells {cells} n={n} {targets} targets a block, precision={precision}", flush=True)
    eng, orc = _engine(c), _oracle(c)
    eng.set_block_targets(targets)
    eng.build_neighbours()
    orc.build_neighbours()
    off_e, idx_e = eng.neighbours()
    off_o, idx_o, _ = orc.neighbours()
    assert same_neighbour_sets(off_e, idx_e, off_o, idx_o)
    assert np.array_equal(eng.neighbour_counts(), np.diff(off_e))
    eng.close()


@pytest.mark.parametrize("cells", [2, 2047, 2048, 2049, 4096, 4097, 600_000])
def test_cell_scan(cells):
    """Lists of two clusters at the ends of a row of cells: the cell counts'
    scan at its tiles' edges (2048 cells), one tile to several hundred."""
    c = _clusters(2, (13,), abi.PREC_FP64, 0)
    k = len(c.x) // 2
    cs = 4 * c.settings.particle_step * (1.0 + 1e-7)
    c.x -= c.x.min(axis=0)
    c.x[:, 1] *= 1e-3
    c.x[:, 0] = np.where(np.arange(len(c.x)) < k, c.x[:, 0] % (0.5 * cs), c.x[:, 0] % (0.5 * cs) + (cells - 0.75) * cs)
    c.x[0, 0], c.x[k, 0] = 0.0, (cells - 0.9) * cs
    print(f"[walk] scan of {cells} cells n={c.n}", flush=True)
    eng, orc = _engine(c), _oracle(c)
    eng.build_neighbours()
    orc.build_neighbours()
    off_e, idx_e = eng.neighbours()
    off_o, idx_o, _ = orc.neighbours()
    assert same_neighbour_sets(off_e, idx_e, off_o, idx_o)
    eng.close()


@pytest.mark.parametrize("cells", [2048 * 1024, 2048 * 1024 + 1, 2048 * 1300 + 77])
def test_cell_scan_of_many_tiles(cells):
    """The same over a row of more cells than tiles' sums are added up
    directly for (1024 tiles): the last such size, one tile more, and a
    number of tiles and of cells in the last that are no multiples of
    anything.  One particle to four cells, the sparsest grid there may be."""
    c = _clusters(2, (13,), abi.PREC_FP64, 0)
    dx, n = c.settings.particle_step, cells // 4
    cs = 4 * dx * (1.0 + 1e-7)
    rng = np.random.default_rng(31)
    c.x = np.stack([rng.uniform(0.0, (cells - 1) * cs, n), rng.uniform(0.0, 0.5 * cs, n)], 1)
    c.x[7], c.x[n // 2] = 0.0, ((cells - 0.9) * cs, 0.0)
    c.v, c.rho, c.p = np.zeros((n, 2)), np.full(n, c.settings.rho_rest), np.zeros(n)
    c.m, c.b = np.full(n, c.settings.rho_rest * dx ** 2), np.full(n, abi.FREE, dtype=np.int32)
    c.blocks = [dict(first=0, last=n, is_fluid=1)]
    print(f"[walk] scan of {cells} cells n={n}", flush=True)
    eng, orc = _engine(c), _oracle(c)
    eng.build_neighbours()
    orc.build_neighbours()
    off_e, idx_e = eng.neighbours()
    off_o, idx_o, _ = orc.neighbours()
    assert same_neighbour_sets(off_e, idx_e, off_o, idx_o)
    eng.close()
