"""Kernels that split their work into tiles, strips or windows, at the sizes
where the split can go wrong: momentum tiles of 64 x 4 rows with and without
constant metrics, the q-l iteration's windows of chain rows and their repeat
where rows couple too far, multigrid tiles of 52 and 56 owned points and
levels below them, the adjoint's tiles and windows."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_mg import _random_state
from test_oracle import _poisson_exact
from wolfd2_amd import api, case, workloads
from wolfd2_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _grid(kind, nx, ny):
    x, y = case.uniform_nodes(nx, ny, 1.0, (ny - 1) / (nx - 1))
    if kind == "stretched":
        x, y = x ** 1.2, y ** 0.9
    return case.compute_grid(x, y)


def _state(g, seed, amp=0.1):
    rng = np.random.default_rng(seed)
    f = [np.zeros((g.ncol, g.ld)) for _ in range(3)]
    for a in f:
        a[: g.ny + 2, : g.nx + 2] = amp * rng.standard_normal((g.ny + 2, g.nx + 2))
    return f


def _step_bitwise(oracle, g, prm, seed):
    reg = case.cavity_regions(g.nx, g.ny)
    f = _state(g, seed)
    sol = api.Solver(g, reg, prm)
    sol.set_fields(*f)
    tg = sol.step(1)
    out = sol.get_fields()
    stats = sol.ql_stats()
    sol.close()
    ref = [a.copy() for a in f]
    to = oracle.run(reg, g, prm, *ref, 1)
    assert np.array_equal(np.asarray(tg)[:, :2], np.asarray(to)[:, :2])
    S = np.s_[: g.ny + 2, : g.nx + 2]
    for name, a, b in zip("uvp", out, ref):
        assert np.array_equal(a[S], b[S], equal_nan=True), name
    return stats


@pytest.mark.parametrize("kind", ["uniform", "stretched"])
@pytest.mark.parametrize("nx,ny", [(5, 5), (64, 6), (65, 5), (66, 9), (130, 67), (513, 453)])
def test_momentum_tiles_bitwise_vs_oracle(oracle, kind, nx, ny):
    print(f"momentum tiles {kind} {nx} x {ny}", flush=True)
    prm = case.Params.from_physical(1e-4, 1.0, 1e-2, nPpeSolver=5, msorit=3, mqiter=4)
    _step_bitwise(oracle, _grid(kind, nx, ny), prm, nx)


@pytest.mark.parametrize("dt,repeats", [(1e-4, 0), (1e-3, 1), (1e-2, 1), (50.0, 1)])
def test_chain_windows_of_weakly_dominant_rows(oracle, dt, repeats):
    """From strong dominance to rows whose coupling outlasts the windows'
    halos, where the iteration is repeated on the whole chains."""
    print(f"chain windows dt {dt}", flush=True)
    prm = case.Params.from_physical(dt, 1.0, 1.0, nPpeSolver=5, msorit=3, mqiter=3)
    stats = _step_bitwise(oracle, _grid("uniform", 90, 70), prm, 11)
    assert stats == {"loops": 1, "repeats": repeats}


@pytest.mark.parametrize("dt,repeats", [(1e-4, 0), (1e-3, 1), (50.0, 1)])
def test_mixed_chain_windows_against_the_whole_chains(dt, repeats):
    """FP32 windows (and their repeat) against the bit-exact FP32 chains: the
    two differ by FP32 rounding of the iterates, 2^-24 times what three
    unconverged iterations amplify it by (10^2)."""
    g = _grid("uniform", 90, 70)
    reg = case.cavity_regions(g.nx, g.ny)
    prm = case.Params.from_physical(dt, 1.0, 1.0, nPpeSolver=5, msorit=3, mqiter=3)
    out = []
    for win in (1, 0):
        old = lib().wd2_set_window_chains(win)
        try:
            sol = api.Solver(g, reg, prm)
            sol.set_precision("mixed")
            sol.set_fields(*_state(g, 12))
            sol.step(1)
            out.append(sol.get_fields())
            assert sol.ql_stats() == {"loops": win, "repeats": win * repeats}
            sol.close()
        finally:
            lib().wd2_set_window_chains(old)
    S = np.s_[: g.ny + 2, : g.nx + 2]
    for name, a, b in zip("uv", *out):
        e = np.linalg.norm(a[S] - b[S]) / np.linalg.norm(b[S])
        print(f"mixed windows dt {dt} {name} {e:.1e}", flush=True)
        assert e < 1e-5, name


@pytest.mark.parametrize("graph", [False, True])
def test_mixed_steps_do_not_depend_on_earlier_runs(graph):
    """A mixed run gives the same bits on a context that has met chains the
    windows cannot take as on a new one, and as graph replays."""
    g = _grid("uniform", 90, 70)
    reg = case.cavity_regions(g.nx, g.ny)
    prm = [case.Params.from_physical(dt, 1.0, 1.0 / re, nPpeSolver=7, msorit=100, sortol=1e-8, mqiter=20)
           for dt, re in ((50.0, 1.0), (2e-4, 1000.0))]
    out = []
    for weak_first in (True, False):
        sol = api.Solver(g, reg, prm[0])
        sol.set_precision("mixed")
        sol.set_graph(graph and weak_first)
        if weak_first:
            sol.set_fields(*_state(g, 12))
            sol.step(2)
        sol.set_params(prm[1])
        sol.set_fields(*_state(g, 13))
        tab = sol.step(4)
        out.append((np.asarray(tab), *sol.get_fields()))
        if weak_first:
            assert sol.ql_stats()["repeats"] >= 2   # the first run's steps
            assert (sol.graph_stats()["replayed"] > 0) == graph
        sol.close()
    S = np.s_[: g.ny + 2, : g.nx + 2]
    assert np.array_equal(out[0][0], out[1][0])
    for name, a, b in zip("uvp", out[0][1:], out[1][1:]):
        assert np.array_equal(a[S], b[S]), name


@pytest.mark.parametrize("ncx,ncy", [(8, 8), (56, 56), (64, 64), (72, 64), (104, 112), (112, 104), (120, 16),
                                     (16, 136), (208, 224)])
def test_mg_tile_edges_against_the_sparse_solution(oracle, ncx, ncy):
    x, y = case.uniform_nodes(ncx + 1, ncy + 1, 1.0, ncy / ncx)
    g = case.compute_grid(x, y)
    reg = case.cavity_regions(g.nx, g.ny)
    u, v, p = _random_state(g, reg, oracle, ncx)
    prm = case.Params(dk=1e-2, re=1.0, nPpeSolver=7, msorit=200, sortol=1e-15)
    exact = _poisson_exact(reg, g, prm, u, v, p)
    n = api.ppe(reg, g, prm, u, v, p)
    S = np.s_[2:g.ny + 1, 2:g.nx + 1]
    err = np.abs(p[S] - exact[S]).max() / np.abs(exact[S]).max()
    print(f"mg {ncx} x {ncy}: {n} V-cycles, {err:.1e}", flush=True)
    assert 0 < n < 200
    assert err < 1e-10


@pytest.mark.parametrize("n", [80, 96, 128])
def test_mg_bottom_widths_agree(n):
    """The bottom kernel from 32 or from 64 cells a side (a first coarse level
    of 40 to 64 is a tile launch or the bottom's own): both V-cycles reach the same
    solution to the solve's own tolerance."""
    g, reg, prm = workloads.cavity(n, 1000.0, 2e-4, nPpeSolver=7, msorit=100, sortol=1e-10)
    out = []
    for bside in (32, 64):
        sol = api.Solver(g, reg, prm)
        sol.set_precision("mixed")
        check(lib().wd2_ctx_mg_set_tune(sol.ctx, 512, 1, bside))
        assert sol.mg_tune()["bside"] == bside
        z = np.zeros((g.ncol, g.ld))
        sol.set_fields(z, z, z)
        sol.cold_start()
        t = np.asarray(sol.step(2))
        last = C.c_double(0)
        lib().wd2_ctx_ppe_divergence(sol.ctx, C.byref(last), None, 1)
        assert last.value < prm.sortol
        out.append((t[:, 1], *sol.get_fields()))
        sol.close()
    S = np.s_[: g.ny + 2, : g.nx + 2]
    assert np.all(np.abs(out[0][0] - out[1][0]) <= 1)
    for name, a, b in zip("uvp", out[0][1:], out[1][1:]):
        assert np.abs(a[S] - b[S]).max() <= 1e-6 * np.abs(b[S]).max(), name


def test_mg_tune_reports_the_width_that_runs():
    """The FP64 path's bottom kernel holds 32 cells a side, and tuning FP64
    leaves the mixed path's width as it was set."""
    g, reg, prm = workloads.cavity(128, 1000.0, 2e-4, nPpeSolver=7, msorit=100, sortol=1e-10)
    sol = api.Solver(g, reg, prm)
    z = np.zeros((g.ncol, g.ld))
    sol.set_fields(z, z, z)
    for bside in (32, 64):
        sol.set_mg_tune(256, 0, bside)
        assert sol.mg_tune()["bside"] == 32
        assert sol.mg_autotune()["bside"] == 32
        sol.set_precision("mixed")
        assert sol.mg_tune()["bside"] == bside
        assert sol.mg_autotune()["bside"] in (32, 64)
        sol.set_precision("fp64")
    sol.close()


@pytest.mark.parametrize("first,other", [("fp64", "mixed"), ("mixed", "fp64")])
def test_mg_shape_set_between_precisions(first, other):
    """A bottom width set while the context's precision is not that of the
    levels' coefficients: the next solve in their precision runs them in its
    own shape, with the bits of a run that set nothing."""
    g, reg, prm = workloads.cavity(128, 1000.0, 2e-4, nPpeSolver=7, msorit=100, sortol=1e-10)
    out = []
    for change in (True, False):
        sol = api.Solver(g, reg, prm)
        sol.set_precision(first)
        sol.set_mg_tune(256, 0, 64)
        z = np.zeros((g.ncol, g.ld))
        sol.set_fields(z, z, z)
        sol.cold_start()
        sol.step(2)
        f = sol.get_fields()
        if change:
            sol.set_precision(other)
            sol.set_mg_tune(256, 0, 64)
            assert lib().wd2_ctx_mg_kernel_time(sol.ctx, 4, 2, C.byref(C.c_double(0))) == 0
            sol.set_precision(first)
        sol.set_fields(*f)
        out.append((np.asarray(sol.step(2)), *sol.get_fields()))
        sol.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nx,ny,dt,lid", [(65, 33, 2e-3, 1.0), (73, 41, 2e-3, 1.0), (65, 33, 0.022, 0.05)])
def test_adjoint_tiles_dot_product(nx, ny, dt, lid):
    """<w, J d> = <J^T w, d> between the tangent-linear pass and the adjoint,
    at tile edges, and with rows too weakly dominant for the windows (the last
    case, on the whole chains); 1e-9 as the solvers' tolerances allow."""
    print(f"adjoint tiles {nx} x {ny} dt {dt}", flush=True)
    x, y = case.uniform_nodes(nx, ny, 1.0, 1.0)
    g = case.compute_grid(x, y)
    reg = case.cavity_regions(nx, ny)
    prm = case.Params.from_physical(dt, 1.0, 1e-2, nPpeSolver=7, msorit=100, sortol=1e-15, qtol=1e-15, mqiter=80)
    sol = api.Solver(g, reg, prm)
    sol.set_bc_profile(1, 1, case.NORTH, case.VAR_U, lid * workloads.lid_modes(x, y, reg, seed=5))
    z = np.zeros((g.ncol, g.ld))
    sol.set_fields(z, z, z)
    sol.step(3)
    rng = np.random.default_rng(nx)
    masks = [np.zeros((g.ncol, g.ld)) for _ in range(3)]
    masks[0][workloads.interior_u(g)] = 1
    masks[1][workloads.interior_v(g)] = 1
    masks[2][2:ny + 1, 2:nx + 1] = 1
    w = [m * rng.standard_normal((g.ncol, g.ld)) for m in masks]
    d = [m * rng.standard_normal((g.ncol, g.ld)) for m in masks]
    adj = api.Adjoint(sol, 2)
    tab = adj.forward(2)
    assert np.all(tab[:, 0] > 0)
    r = adj.backward(*w)
    whole = 2 if lid < 1 else 0   # of its two steps
    assert adj.window_stats() == {"windows": 2 - whole, "chains": whole}
    t = adj.tangent(*d, np.zeros((4, 2, max(nx, ny) + 2)))
    assert r["stats"]["adj_unconverged"] == 0 and t["stats"]["adj_unconverged"] == 0
    tl = sum(float(np.sum(a * t[k])) for a, k in zip(w, ("duN", "dvN", "dpN")))
    ad = sum(float(np.sum(a * r[k])) for a, k in zip(d, ("u0_bar", "v0_bar", "p0_bar")))
    print(f"  {tl:.12e} {ad:.12e}", flush=True)
    assert abs(tl - ad) <= 1e-9 * abs(ad)
