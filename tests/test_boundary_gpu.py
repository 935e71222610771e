"""The boundary calls that reorder on the device: states and member parameters in
reference order go in and come out bit for bit, also the values that arithmetic would
change (-0.0, infinities, NaN, subnormals), on grids below and above the pieces in
which sub-cells and parameter rows pass the staging buffer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows, cols, members", [(1, 1, 1), (7, 9, 2), (40, 50, 13)])
def test_boundary_calls_keep_bits_and_order(wg, rows, cols, members):
    print("case: boundary calls", rows, cols, members, flush=True)
    w = wg.World(wg.regional_spec(seed=rows * 100 + cols, nrows=rows, ncols=cols))
    rng = np.random.default_rng(rows)
    m = wg.WaterBalanceModel(w, n_members=members)
    blank = m.get_state(0)
    odd = np.array([-0.0, np.inf, -np.inf, np.nan, 5e-324])

    def draw():
        st = {}
        for k, v in blank.items():
            if k == "started":
                continue
            a = rng.integers(-2**31, 2**31, v.shape) if v.dtype.kind == "i" else rng.normal(size=v.shape) * 1e3
            st[k] = a.astype(v.dtype)
            if v.dtype.kind == "f":
                st[k].flat[rng.integers(0, st[k].size, 5)] = odd
        return st

    def same(q, st):
        got = m.get_state(q)
        return [k for k in st if got[k].tobytes() != st[k].tobytes()]

    common, own = draw(), draw()
    m.set_state(common)
    m.set_state(own, member=members - 1)
    for q in range(members - 1):
        assert same(q, common) == []
    assert same(members - 1, own) == []
    m.close()

    # member parameters and the daily series: every member as a model of its own
    gamma, cfa = rng.uniform(0.2, 4.0, (members, w.n)), rng.uniform(0.7, 1.3, (members, w.n))
    smax = (np.tile(w.smax, (members, 1)) * rng.uniform(0.8, 1.2, (members, w.n))).astype(np.float32)
    forcing = w.forcing(seed=2, day0=0, n_days=4)

    def series(q0, q1, max_days):
        e = wg.WaterBalanceModel(w, n_members=q1 - q0)
        e.set_member_params(gamma=gamma[q0:q1], cfa=cfa[q0:q1], smax=smax[q0:q1])
        e.set_stations(w.basin_outlet)
        e.load_forcing(forcing)
        e.step_days(0, 1, 4)
        daily = e.station_discharge(max_days=max_days)[1]
        out = e.day_outputs(q1 - q0 - 1)
        e.close()
        return daily, out

    together, last = series(0, members, 6)
    assert not together[:, 4:].any()  # days that were not stepped stay as they were
    for q in range(0, members, 6):
        alone, out = series(q, q + 1, 3)
        assert np.array_equal(together[q, :3], alone[0])
        if q == members - 1:
            assert all(np.array_equal(last[k], out[k]) for k in out)
