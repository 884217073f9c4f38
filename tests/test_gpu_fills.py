"""The boundary fills on the GPU against the oracle, bit for bit, where their
work split can go wrong: sides around the workgroup's lanes and the staged
rows of the outlet recurrences (1024), and regions one and two cells wide
(whose opposite sides touch the same columns)."""
import numpy as np
import pytest

from wolfd2_amd import api, case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", ["west", "east", "south", "north"])
@pytest.mark.parametrize("kind", ["fully_dev", "mass_cons"])
@pytest.mark.parametrize("n", [6, 1025, 1026, 2050])
def test_outlet_fills_at_the_edges_of_the_staged_rows(oracle, side, kind, n):
    print(f"outlet fills {side} {kind} {n}", flush=True)
    nx, ny = (9, n) if side in ("west", "east") else (n, 9)
    reg = case.make_regions(nx, ny, walls=[(1, 1, s, "no_slip", 0.5, 0.1) for s in ("west", "east", "south", "north")
                                           if s != side], outlets=[(1, 1, side, kind, 0.2, 0.3, 0.4)])
    _check(oracle, reg, nx, ny, n)


@pytest.mark.parametrize("ib", [(3, 4), (3, 5), (2, 8)])
def test_fills_of_narrow_regions(oracle, ib):
    print(f"narrow regions {ib}", flush=True)
    nx, ny = 13, 12
    reg = case.make_regions(nx, ny, nreg=(3, 3), i_borders=ib, j_borders=ib,
                            walls=[(2, 2, s, "no_slip", 0.3, 0.2) for s in ("west", "east", "south", "north")],
                            outlets=[(3, 1, "east", "mass_cons", 0.0, 0.0, 0.0)])
    _check(oracle, reg, nx, ny, 7)


def _check(oracle, reg, nx, ny, seed):
    rng = np.random.default_rng(seed)
    f = [rng.standard_normal((ny + 2, nx + 2)) for _ in range(3)]
    for name in ("vel_bound_cond", "vel_outflow_bcs"):
        a, b = [x.copy() for x in f[:2]], [x.copy() for x in f[:2]]
        getattr(api, name)(reg, *a)
        getattr(oracle, name)(reg, nx + 2, *b)
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), name
    a, b = f[2].copy(), f[2].copy()
    api.pres_bound_cond(reg, a)
    oracle.pres_bound_cond(reg, nx + 2, b)
    assert np.array_equal(a, b)
