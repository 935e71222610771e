"""The many-days kernel (the graph-free path of step_days) against the eager path,
one launch per day and part, which the parity tests pin to the oracle: every state
field, the day's outputs and the daily station series, bit for bit.

The sizes are where it can go wrong: grids below, at and above one wavefront, call
lengths that take different wavefront tables (levels per wavefront) and that make the
ring of transported volumes wrap, members, and cells with lakes, reservoirs, inland
sinks and no land."""
import concurrent.futures
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(wg, w, f, members, calls, profiled, start=None):
    m = wg.WaterBalanceModel(w, n_members=members)
    if start is not None:
        m.set_state(start(m.get_state()))
    rng = np.random.default_rng(3)
    if members > 1:
        m.set_member_params(gamma=rng.uniform(0.2, 4.0, (members, w.n)), cfa=rng.uniform(0.7, 1.3, (members, w.n)))
        m.set_forcing_perturbation(np.arange(5, 5 + members, dtype=np.uint64))
    m.set_stations(np.unique(np.concatenate([w.basin_outlet, [0, w.n // 2]])).astype(np.int32))
    m.load_forcing(f)
    day, daily = 0, []
    for k in calls:
        m.step_days(day, day % 365 + 1, k, profiled=profiled)
        daily.append(m.station_discharge(max_days=k)[1])
        day += k
    states = [m.get_state(q) for q in range(members)]
    outs = [m.day_outputs(q) for q in range(members)]
    total = m.station_discharge()[0]
    m.close()
    return states, outs, total, np.concatenate(daily, axis=1)


@pytest.mark.parametrize("rows, cols, members, calls", [
    (1, 1, 1, [3, 9]), (7, 9, 1, [9, 1]), (8, 8, 2, [4]), (5, 13, 1, [10]),
    (40, 50, 1, [3] * 14), (40, 50, 3, [40, 33, 2, 70]), (30, 41, 1, [120]), (40, 50, 70, [5, 33])])
def test_many_days_equals_eager(wg, rows, cols, members, calls):
    print("case: many days", rows, cols, members, calls[:3], flush=True)
    w = wg.World(wg.regional_spec(seed=rows * 100 + cols, nrows=rows, ncols=cols, edge_cases=rows * cols > 60,
                                  glolake_every=9, res_every=14))
    if w.n > 100:
        w.contfreq[::37] = 0.0  # cells without land keep a zero volume
    f = w.forcing(seed=2, day0=0, n_days=sum(calls))
    a = run(wg, w, f, members, calls, False)
    b = run(wg, w, f, members, calls, True)
    for q in range(members):
        for k in b[0][q]:
            assert np.array_equal(np.asarray(a[0][q][k]), np.asarray(b[0][q][k]), equal_nan=True), (q, k)
        for k in b[1][q]:
            assert np.array_equal(a[1][q][k], b[1][q][k], equal_nan=True), (q, k)
    assert np.array_equal(a[2], b[2], equal_nan=True)
    assert np.array_equal(a[3], b[3], equal_nan=True)


def same(a, b):
    return np.array_equal(np.asarray(a), np.asarray(b), equal_nan=True)


@pytest.mark.parametrize("members", [1, 3])
def test_start_states_that_are_not_numbers(wg, members):
    """Storages and land fractions that are no numbers, or become none within a day (the
    power of a slightly negative soil), spread downstream as in one launch per day."""
    print("case: many days, start states that are not numbers", members, flush=True)
    w = wg.World(wg.regional_spec(seed=9, nrows=20, ncols=31, glolake_every=9, res_every=14))
    f = w.forcing(seed=2, day0=0, n_days=12)

    def start(st):
        st["started"] = 1
        st["soil"][3::41] = -1.8e-19
        st["laf"][10::67] = st["laf_prev"][10::67] = np.nan
        st["laf"][11::67] = 0.0
        st["laf_prev"][12::67] = np.nan
        st["river"][13::97] = np.nan
        st["snow_elev"][20::53, 1:] = 12.0
        st["snow_elev"][21::53, 5] = np.nan
        st["snow_elev"][22::53, 6] = np.inf
        st["laf"][20::53] = np.nan
        return st

    a = run(wg, w, f, members, [4, 8], False, start)
    b = run(wg, w, f, members, [4, 8], True, start)
    assert np.isnan(b[0][0]["laf"]).any() and not np.isnan(b[0][0]["laf"]).all()
    for q in range(members):
        assert all(same(a[0][q][k], b[0][q][k]) for k in b[0][q]), [k for k in b[0][q] if not same(a[0][q][k], b[0][q][k])]
        assert all(same(a[1][q][k], b[1][q][k]) for k in b[1][q]), [k for k in b[1][q] if not same(a[1][q][k], b[1][q][k])]
    assert same(a[2], b[2]) and same(a[3], b[3])


@pytest.mark.parametrize("members, days", [(12, 9), (17, 9), (71, 4)])
def test_members_one_by_one_and_in_twos(wg, members, days):
    """Workgroups of one member while every wavefront has a SIMD of its own (12 members
    of 80 wavefronts, 17 of 52 with two levels each), of two beyond, the last one half
    empty (71)."""
    print("case: many days, members", members, days, flush=True)
    w = wg.World(wg.regional_spec(seed=6, nrows=40, ncols=50))
    f = w.forcing(seed=3, day0=0, n_days=days)
    a = run(wg, w, f, members, [days], False)
    b = run(wg, w, f, members, [days], True)
    for q in range(members):
        assert all(np.array_equal(np.asarray(a[0][q][k]), np.asarray(b[0][q][k]), equal_nan=True) for k in b[0][q]), q
    assert np.array_equal(a[2], b[2], equal_nan=True) and np.array_equal(a[3], b[3], equal_nan=True)


@pytest.mark.parametrize("members, use, pot", [(71, True, False), (71, False, True), (5, True, False), (3, True, True)])
def test_members_with_water_use_and_potential_runoff(wg, members, use, pot):
    """The options whose fields each day reads and writes beside the state, with members
    in workgroups of two (71 members of 32 wavefronts and more) and of one."""
    print("case: many days, options", members, use, pot, flush=True)
    w = wg.World(wg.regional_spec(seed=8, nrows=40, ncols=50, glolake_every=9, res_every=14))
    f = w.forcing(seed=3, day0=0, n_days=17)
    rng = np.random.default_rng(4)
    scale = np.asarray(w.cell_area)[None, :, None] * 6e4  # 2 mm a month, in m3
    tabs = [rng.uniform(a, b, (1, w.n, 12)) * scale for a, b in ((-0.3, 20.0), (0.0, 0.5), (1.0, 2.0), (0.2, 0.9))]
    frgi = rng.uniform(0.0, 1.0, w.n)
    smax = (np.tile(w.smax, (members, 1)) * rng.uniform(0.8, 1.2, (members, w.n))).astype(np.float32)
    out = []
    for profiled in (False, True):
        m = wg.WaterBalanceModel(w, n_members=members, options={"subtract_use": 2} if use else None)
        m.set_member_params(smax=smax)
        m.set_forcing_perturbation(np.arange(5, 5 + members, dtype=np.uint64))
        m.set_stations(w.basin_outlet)
        if use:
            m.set_water_use(*tabs, frgi, delayed=1)
        if pot:
            m.pot_cell_runoff_output(True)
        m.load_forcing(f)
        for a, b in ((0, 4), (4, 17)):
            m.step_days(a, 60 + a, b - a, profiled=profiled)
        got = {"sum": m.station_discharge()[0]}
        for q in (0, 1, members // 2, members - 1):
            got.update({f"{k} {q}": v for k, v in {**m.get_state(q), **m.day_outputs(q)}.items()})
            if use:
                got[f"use {q}"] = m.water_use_state(q)
            if pot:
                got[f"pot {q}"] = m.pot_cell_runoff(q)
        out.append(got)
        m.close()
    assert all(same(out[0][k], out[1][k]) for k in out[1]), [k for k in out[1] if not same(out[0][k], out[1][k])]
    assert not use or np.abs(out[0]["use 0"]).max() > 0
    assert not pot or np.abs(out[0]["pot 0"]).max() > 0


def test_two_handles_that_each_fill_the_chip(wg):
    """Launches of two handles, from two threads, that each have more wavefronts than the
    chip holds (2,000 cells, 130 members): workgroups of both hold its slots in any mixture,
    and each handle's days are those it steps alone."""
    print("case: many days, two handles at once", flush=True)
    w = wg.World(wg.regional_spec(seed=6, nrows=40, ncols=50))
    f = w.forcing(seed=3, day0=0, n_days=24)
    barrier = threading.Barrier(2)

    def steps(first_seed, together):
        m = wg.WaterBalanceModel(w, n_members=130)
        m.set_forcing_perturbation(np.arange(first_seed, first_seed + 130, dtype=np.uint64))
        m.set_stations(w.basin_outlet)
        m.load_forcing(f)
        for rep in range(4):
            if together:
                barrier.wait(60)
            m.step_days(0, 1, 24)
        out = m.station_discharge(max_days=24)
        states = [m.get_state(q) for q in (0, 64, 129)]
        m.close()
        return out, states

    alone = [steps(1, False), steps(500, False)]
    with concurrent.futures.ThreadPoolExecutor(2) as pool:
        both = list(pool.map(lambda seed: steps(seed, True), (1, 500)))
    for a, b in zip(alone, both):
        assert same(a[0][0], b[0][0]) and same(a[0][1], b[0][1])
        for x, y in zip(a[1], b[1]):
            assert all(same(x[k], y[k]) for k in x)


def test_launch_count_of_a_call_longer_than_the_ring(wg):
    """6,000 members of 180 cells: the ring's 2 GiB hold 248 days, so 250 days are two
    launches, and wg_last_timing says so."""
    print("case: many days, launches of 6,000 members", flush=True)
    w = wg.World(wg.regional_spec(seed=0, nrows=12, ncols=15))
    m = wg.WaterBalanceModel(w, n_members=6000)
    m.load_forcing(w.forcing(seed=3, day0=0, n_days=250))
    m.step_days(0, 1, 40)
    assert m.timing()[1][2] == 1
    m.step_days(0, 1, 250)
    assert (2 << 30) // (6000 * w.n * 8) == 248 and m.timing()[1][2] == 2
    m.close()


def test_autotune_on_the_many_days_path(wg):
    """The tuner's saved state leaves the tables and the ring alone that its own first
    call of the many-days kernel makes."""
    print("case: many days, autotune of 12 days", flush=True)
    w = wg.World(wg.regional_spec(seed=4, nrows=20, ncols=21))
    f = w.forcing(seed=3, day0=0, n_days=30)
    out = []
    for tune in (True, False):
        m = wg.WaterBalanceModel(w)
        m.load_forcing(f)
        if tune:
            m.autotune(n_days=12)
        m.step_days(0, 1, 30)
        out.append(m.get_state())
        m.close()
    for k in out[0]:
        assert np.array_equal(np.asarray(out[0][k]), np.asarray(out[1][k])), k


@pytest.mark.parametrize("rows, cols, members", [(2, 2, 1), (2, 2, 300), (20, 21, 12), (40, 50, 1)])
@pytest.mark.parametrize("days", [1, 3])
def test_autotune_on_few_days_leaves_long_calls_on_the_many_days_path(wg, rows, cols, members, days):
    """Whatever the tuner finds fastest for one day or three, thirty are one launch; an
    explicit configuration with another chain mode still takes two launches a day."""
    print("case: many days, autotune on few days", rows, cols, members, days, flush=True)
    w = wg.World(wg.regional_spec(seed=4, nrows=rows, ncols=cols))
    m = wg.WaterBalanceModel(w, n_members=members)
    m.load_forcing(w.forcing(seed=3, day0=0, n_days=30))
    cfg, _ = m.autotune(n_days=days)
    m.step_days(0, 1, 30)
    assert m.timing()[1][2] == 1, cfg
    m.set_launch_config(256, 256, 5, 0)
    m.step_days(0, 1, 30)
    assert m.timing()[1][2] == 61
    m.close()


@pytest.mark.parametrize("members, chain", [(1, 512), (5, 256)])
def test_autotune_keeps_the_defaults_of_short_calls(wg, members, chain):
    """Tuned on many days, mode 3 keeps the tile, workgroup and chunk that calls of one
    or two days run with."""
    print("case: many days, autotune defaults", members, flush=True)
    w = wg.World(wg.regional_spec(seed=4, nrows=20, ncols=21))
    m = wg.WaterBalanceModel(w, n_members=members)
    m.load_forcing(w.forcing(seed=3, day0=0, n_days=12))
    cfg, _ = m.autotune(n_days=12)
    m.close()
    if cfg[3] != 3:
        pytest.skip("one launch per day and part was faster on 12 days")
    assert tuple(cfg) == (256, chain, 5, 3)
