"""Ensembles: every member of a batched, uneven-size ensemble advances exactly
as a single-grid run of the same scenario (and, in FP64, as the oracle)."""
import numpy as np
import pytest

from tsuner_amd import scenarios as S
from tsuner_amd.ensemble import Ensemble
from tsuner_amd.solver import Solver

pytestmark = pytest.mark.gpu


def members():
    out = [S.gaussian_source(n=n, dx=40.0, seed=seed) for n, seed in ((48, 1), (70, 2), (61, 3), (130, 4))]
    sc = S.sediment_shelf(n=90, ny=45, dx=40.0, inflow=False, seed=5)
    out.append(sc)
    return out


def test_fp64_members_equal_oracle_and_single(oracle):
    scs = members()
    ens = Ensemble(scs, precision="fp64", tile_rows=[8, 16, 5, 32, 3])
    ens.step(12)
    for i, sc in enumerate(scs):
        print("member %d %s" % (i, sc.name), flush=True)
        o = oracle.from_scenario(sc)
        o.step(12)
        W = ens.state(i)
        assert np.array_equal(W, o.state()), "member %d differs from the oracle" % i
        t, dt, n = ens.time(i)
        assert (t, dt, n) == (o.t, o.dt, 12)


def test_fp64_mixed_bedload_laws_equal_oracle(oracle):
    """A member with Grass bedload makes the whole ensemble take the general
    bedload kernel; the Ashida-Michiue members must still equal the oracle
    bit for bit (their single-grid runs take the branch-free variant)."""
    scs = [S.gaussian_source(n=48, dx=40.0, seed=1),
           S.gaussian_source(n=70, dx=40.0, seed=2, bedload_law=S.BEDLOAD_GRASS, grass_ag=1e-3),
           S.gaussian_source(n=61, dx=40.0, seed=3)]
    ens = Ensemble(scs, precision="fp64", tile_rows=[8, 16, 5])
    ens.step(12)
    for i, sc in enumerate(scs):
        print("member %d %s law %d" % (i, sc.name, sc.scheme["bedload_law"]), flush=True)
        o = oracle.from_scenario(sc)
        o.step(12)
        assert np.array_equal(ens.state(i), o.state()), "member %d differs from the oracle" % i
        g = Solver.from_scenario(sc, precision="fp64", tile_rows=16)
        g.step(12)
        assert np.array_equal(ens.state(i), g.state()), "member %d differs from its single-grid run" % i


def test_fp32_members_equal_single_solver():
    scs = members()
    ens = Ensemble(scs, precision="fp32")
    ens.step(15)
    for i, sc in enumerate(scs):
        g = Solver.from_scenario(sc, precision="fp32", tile_rows=16)
        g.step(15)
        assert np.array_equal(ens.state(i), g.state()), "member %d" % i
        assert ens.time(i) == g.time()


def test_graph_replay_and_stop_step():
    scs = members()
    a = Ensemble(scs, precision="fp32")
    b = Ensemble(scs, precision="fp32", graph_chunk=4)
    b.set_stop_step(10)
    a.step(10)
    b.step(12)          # three replays of four steps; the last two steps are no-ops
    for i in range(len(scs)):
        assert b.time(i)[2] == 10
        assert np.array_equal(a.state(i), b.state(i))
        b.mass(i)


def test_autotune_keeps_results(tmp_path, monkeypatch):
    from tsuner_amd import autotune
    monkeypatch.setenv("XDG_CACHE_HOME", str(tmp_path))
    scs = members()
    ref = Ensemble(scs, precision="fp32")
    ref.step(6)
    ens = Ensemble(scs, precision="fp32")
    choice = autotune.tune_ensemble(ens, "fp32", candidates=(4, 16), steps=2, log=print)
    assert set(choice) == {max(s.npx, s.npy) for s in scs}
    ens.step(6)
    for i in range(len(scs)):
        assert np.array_equal(ref.state(i), ens.state(i))
    assert (tmp_path / "tsuner_amd" / "tile_rows.json").exists()


def inflow_members():
    """Members with boundary series of their own: two N-wave shelves of
    different sizes driven through the left side (different series lengths
    and spacings), the reference's westport example driven through all four
    sides, and a walled member beside them."""
    from ingest_files import westport_scenario
    a = S.sediment_shelf(n=64, ny=40, dx=40.0, seed=6, t_series=60.0)   # its series ends within the test
    b = S.sediment_shelf(n=97, ny=33, dx=40.0, seed=7, t_series=2000.0)
    b.tCC = b.tCC[::2].copy()
    b.CC = np.ascontiguousarray(b.CC[::2])
    c = westport_scenario()
    d = S.gaussian_source(n=50, dx=40.0, seed=8)
    return [a, b, c, d]


def test_fp64_inflow_members_equal_oracle(oracle):
    """Per-member inflow series (VolumeSolver.cu:172-215 read at each
    member's own time) in one batched launch: every member equals the
    oracle bit for bit, through and past the end of its series."""
    scs = inflow_members()
    ens = Ensemble(scs, precision="fp64", tile_rows=[8, 5, 16, 4])
    orc = [oracle.from_scenario(sc) for sc in scs]
    for chunk in range(3):
        ens.step(60)
        for i, (sc, o) in enumerate(zip(scs, orc)):
            o.step(60)
            print("chunk %d member %d %s t=%.1f" % (chunk, i, sc.name, o.t), flush=True)
            assert np.array_equal(ens.state(i), o.state()), "member %d differs from the oracle" % i
            assert ens.time(i) == (o.t, o.dt, 60 * (chunk + 1))


def test_fp32_inflow_members_equal_single_solver():
    scs = inflow_members()
    ens = Ensemble(scs, precision="fp32", graph_chunk=10)
    ens.step(40)
    for i, sc in enumerate(scs):
        g = Solver.from_scenario(sc, precision="fp32", tile_rows=16)
        g.step(40)
        assert np.array_equal(ens.state(i), g.state()), "member %d" % i
        assert ens.time(i) == g.time()


def test_inflow_member_without_series_is_refused():
    from tsuner_amd import _lib
    sc = S.sediment_shelf(n=40, ny=20, dx=40.0)
    sc.CC = None
    sc.tCC = None
    with pytest.raises(_lib.TsuError) as e:
        Ensemble([sc], precision="fp32")
    assert "tsu_ensemble_set_inflow" in str(e.value)


@pytest.mark.parametrize("n", [1, 2, 3])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("chunk", [0, 4])
def test_halves_on_two_streams_equal_single_solver(n, order, chunk):
    """One member (one half), two, and three of unequal sizes; calls that
    enqueue whole chunks, a remainder and a single step, with work on the
    ensemble's stream (a mass sum) between them."""
    scs = [S.gaussian_source(n=k, dx=40.0, seed=k, order=order) for k in (48, 130, 61)][:n]
    ens = Ensemble(scs, precision="fp32", graph_chunk=chunk)
    masses = []
    for k in (9, 1, 4, 0):
        ens.step(k, sync=False)
        masses.append([ens.mass(i) for i in range(n)])
    for i, sc in enumerate(scs):
        g = Solver.from_scenario(sc, precision="fp32")
        for k, m in zip((9, 1, 4, 0), masses):
            g.step(k)
            assert g.mass() == m[i]
        assert np.array_equal(ens.state(i), g.state()), "member %d" % i
        assert ens.time(i) == g.time()


@pytest.mark.parametrize("nx,ny", [(1, 1), (63, 5), (1100, 801)])
def test_fp32_states_keep_hi_and_lo_parts(nx, ny):
    """FP64 planes -> float pairs (q: floats) -> FP64 planes; the last grid's
    five planes take more than one transfer of 4 Mi values."""
    rng = np.random.default_rng(nx)
    V = rng.normal(size=(5, ny, nx)) * 10.0 ** rng.integers(-42, 6, size=(5, ny, nx))
    V.reshape(5, -1)[:, 0] = [0.0, -0.0, 1e-45, 3e38, 1e-300]
    want = V.astype(np.float32).astype(np.float64)
    for f in (0, 3, 4):
        want[f] += (V[f] - want[f]).astype(np.float32).astype(np.float64)
    sc = S.Scenario("random", S.base_params(nx, ny, 10.0, 10.0), S.default_scheme(), V, np.ones((ny, nx), np.int32))
    s = Solver.from_scenario(sc, precision="fp32", init_dt=False)
    assert np.array_equal(s.state(), want)
    ens = Ensemble([sc, sc], precision="fp32")
    for i in range(2):
        assert np.array_equal(ens.state(i), want)
        for f in range(5):
            assert np.array_equal(ens.plane(i, f), want[f])


@pytest.mark.parametrize("nx,ny", [(128, 128), (127, 130)])
def test_fp32_states_converted_on_the_host_and_on_the_device(nx, ny):
    """The largest states whose FP64 values the host splits and joins, and
    larger ones, whose the device does: the same floats, q without low parts."""
    rng = np.random.default_rng(nx)
    V = rng.normal(size=(5, ny, nx)) * 10.0 ** rng.integers(-42, 6, size=(5, ny, nx))
    V.reshape(5, -1)[:, 0] = [0.0, -0.0, 1e-45, 3e38, 1e-300]
    want = V.astype(np.float32).astype(np.float64)
    for f in (0, 3, 4):
        want[f] += (V[f] - want[f]).astype(np.float32).astype(np.float64)
    sc = S.Scenario("random", S.base_params(nx, ny, 10.0, 10.0), S.default_scheme(), V, np.ones((ny, nx), np.int32))
    other = S.gaussian_source(n=64, dx=20.0, seed=1)
    assert np.array_equal(Solver.from_scenario(sc, precision="fp32", init_dt=False).state(), want)
    ens = Ensemble([other, sc], precision="fp32")
    assert np.array_equal(ens.state(1), want)
    for f in range(5):
        assert np.array_equal(ens.plane(1, f), want[f])
        assert np.array_equal(ens.plane(0, f), ens.state(0)[f])


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("chunk", [0, 2])
def test_short_and_long_calls_alternate(order, chunk):
    """Calls of one launch for both halves and calls that fork them (here from
    21 single-stage and 11 two-stage steps on), eager and in graphs of either,
    against the single solver."""
    scs = [S.gaussian_source(n=k, dx=40.0, seed=k, order=order) for k in (300, 181, 240)]
    ens = Ensemble(scs, precision="fp32", graph_chunk=chunk)
    calls = (1, 2, 24, 3, 25, 2, 10)
    for k in calls:
        ens.step(k, sync=False)
    for i, sc in enumerate(scs):
        g = Solver.from_scenario(sc, precision="fp32")
        g.step(sum(calls))
        assert np.array_equal(ens.state(i), g.state()), "member %d" % i
        assert ens.time(i) == g.time()
