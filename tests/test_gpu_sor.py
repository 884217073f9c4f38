"""The tiled red-black and lexicographic SOR (solvers 5 and 1) on the GPU
against the oracle, bit for bit, where the tiles can go wrong: grids around the one-tile limit (64 interior points a
side), sides that leave a remainder of every kind after the owned points of
the larger tiles, sweep counts around a launch's, solves that stop inside one,
the three forms of the division by the diagonal (array coefficients, one
value, one power of two) and quotients that are zero, tiny or huge."""
import numpy as np
import pytest

from wolfd2_amd import api, case

pytestmark = pytest.mark.gpu


def _grid(kind, nx, ny):
    x, y = case.uniform_nodes(nx, ny, 1.0, (ny - 1) / (nx - 1))
    if kind == "stretched":
        x, y = x ** 1.25, y ** 0.8
    return case.compute_grid(x, y)


def _fields(g, seed, scale, blank):
    rng = np.random.default_rng(seed)
    f = [scale * rng.standard_normal((g.ncol, g.ld)) for _ in range(3)]
    if blank:   # a quiescent part: right-hand side and pressure zero
        for a in f:
            a[:, : 1 + g.nx // 2] = 0.0
    return f


def _check(oracle, g, nx, ny, msorit, sortol, seed, scale=1.0, blank=False, solver=5):
    reg = case.cavity_regions(nx, ny)
    prm = case.Params.from_physical(1e-3, 1.0, 1e-3, nPpeSolver=solver, msorit=msorit, sortol=sortol)
    u, v, p = _fields(g, seed, scale, blank)
    a, b = p.copy(), p.copy()
    na = api.ppe(reg, g, prm, u, v, a)
    nb = oracle.ppe(reg, g, prm, u, v, b)
    assert na == nb
    assert np.array_equal(a[: ny + 2, : nx + 2], b[: ny + 2, : nx + 2], equal_nan=True)
    return na


@pytest.mark.parametrize("solver", [5, 1])
@pytest.mark.parametrize("kind", ["uniform", "stretched"])
@pytest.mark.parametrize("nx,ny", [(5, 5), (65, 65), (65, 7), (64, 66), (66, 65), (73, 74), (75, 130), (257, 40),
                                   (385, 90), (401, 450)])
def test_tiled_sor_sizes(oracle, kind, nx, ny, solver):
    print(f"tiled sor {solver} {kind} {nx} x {ny}", flush=True)
    _check(oracle, _grid(kind, nx, ny), nx, ny, 31, 1e-30, nx, solver=solver)


@pytest.mark.parametrize("nx", [49, 65, 129])   # one value; one power of two; one power of two over tiles
@pytest.mark.parametrize("solver,msorit", [(5, m) for m in (1, 2, 13, 14, 15, 28, 29)] +
                         [(1, m) for m in (1, 16, 17, 33, 64, 65, 200)])
def test_tiled_sor_sweep_counts(oracle, nx, solver, msorit):
    print(f"tiled sor {solver} sweeps {nx} {msorit}", flush=True)
    g = _grid("uniform", nx, nx)
    assert _check(oracle, g, nx, nx, msorit, 1e-30, 1, solver=solver) == msorit
    _check(oracle, g, nx, nx, msorit, 1e30, 2, solver=solver)   # stops at the first sweep that may


@pytest.mark.parametrize("kind", ["uniform", "stretched"])
@pytest.mark.parametrize("nx", [50, 65, 97])
@pytest.mark.parametrize("solver", [5, 1])
def test_tiled_sor_stops_inside_a_launch(oracle, kind, nx, solver):
    g = _grid(kind, nx, nx)
    stops = {_check(oracle, g, nx, nx, 6000, tol, 3, scale=1e-3, solver=solver) for tol in 10.0 ** -np.arange(1.0, 9.0)}
    print(f"tiled sor {solver} stops {kind} {nx} {sorted(stops)}", flush=True)
    assert len(stops) > 2


@pytest.mark.parametrize("kind", ["uniform", "stretched"])
@pytest.mark.parametrize("nx", [50, 65, 97])
@pytest.mark.parametrize("scale,blank", [(1.0, True), (0.0, False), (1e-250, False), (1e250, False), (1e308, False)])
@pytest.mark.parametrize("solver", [5, 1])
def test_tiled_sor_extreme_quotients(oracle, kind, nx, scale, blank, solver):
    print(f"tiled sor {solver} quotients {kind} {nx} {scale} {blank}", flush=True)
    _check(oracle, _grid(kind, nx, nx), nx, nx, 17, 1e-300, 4, scale, blank, solver)
