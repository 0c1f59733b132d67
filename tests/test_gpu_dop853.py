"""GPU DOP853 (gamd_dop853) against the oracle's restatement of gala's
dop853 driven with nbatch=1 (one adaptive system per orbit), which the
oracle matches bit for bit against gala's own compiled dop853.cpp
(tests/test_oracle_ref.py).

Bars: identical accepted-step counts for all but a tiny fraction of orbits
(an ulp-level difference can flip one accept/reject decision), final states
within 1e-8 relative where the step sequences agree, and dense output within
1e-8 relative (the stated DOP853 tolerance)."""
import numpy as np
import pytest

from gala_amd import workloads
from oracle import oracle as O
from tests.helpers import mw_oracle, mw_product, state_rel_err, vcirc_oracle

pytestmark = pytest.mark.gpu


def _energy(orc, w):
    return O.value(orc, np.ascontiguousarray(w[:3])) + 0.5 * np.sum(w[3:] ** 2, axis=0)


def test_per_orbit_uneven_parity():
    """16,384 orbits of the 1,048,576-orbit uneven workload over their FULL
    integration times (up to 10 Gyr): the 1,024 longest by the pilot pass
    (the orbits that set the launch's length, up to ~23,700 step attempts)
    and 15,360 drawn at random from the rest.

    Over these times a third of the orbits (those through the 0.07 kpc
    nucleus) are chaotic: in the oracle itself a one-ulp change of the
    initial state, or building it with gala's own -Ofast instead of IEEE
    flags, moves their final states by up to O(1).  Orbits insensitive to
    both (response <= 1e-10) must match within 1e-8 (the stated DOP853 bar);
    the chaotic ones cannot match any ulp-different implementation and are
    held to the oracle's energy-error distribution instead.  Status codes
    must be identical for all, and the share of orbits whose accepted-step
    count differs may not exceed what a one-ulp change causes in the oracle."""
    from gala_amd import _device as dev
    from gala_amd.integrate import dop853, pilot_order
    orc = mw_oracle()
    w_all, T_all = workloads.composite_dop853(vcirc_oracle(orc), n=1048576, seed=1)
    pot = mw_product()
    order = dev.to_host(pilot_order(pot, w_all, 0.0, T_all, 1.0, rtol=1e-8, atol=1e-10))
    rest = np.random.default_rng(2).choice(order[1024:], 15360, replace=False)
    sel = np.sort(np.concatenate([order[:1024], rest]))
    w0, T = np.ascontiguousarray(w_all[:, sel]), np.ascontiguousarray(T_all[sel])
    longest = np.isin(sel, order[:1024])
    ref, st_ref, stats_ref = O.dop853_orbits(orc, w0, 0.0, T, 1.0, atol=1e-10, rtol=1e-8)
    sens = np.zeros(w0.shape[1])
    for k, direction in ((0, np.inf), (1, -np.inf), (5, np.inf)):
        pert = w0.copy()
        pert[k] = np.nextafter(pert[k], direction)
        alt, _, stats_k = O.dop853_orbits(orc, pert, 0.0, T, 1.0, atol=1e-10, rtol=1e-8)
        sens = np.maximum(sens, state_rel_err(alt, ref))
        if k == 0:
            stats_alt = stats_k
    build = state_rel_err(O.dop853_orbits(orc, w0, 0.0, T, 1.0, atol=1e-10, rtol=1e-8,
                                          fast=True)[0], ref)
    calm = (sens <= 1e-10) & (build <= 1e-10)
    res = dop853(pot, w0, 0.0, T, 1.0, rtol=1e-8, atol=1e-10)
    w = dev.to_host(res["w_final"])
    st = dev.to_host(res["status"])
    stats = dev.to_host(res["stats"])
    assert np.array_equal(st, st_ref)
    same = stats[:, 1] == stats_ref[:, 1]
    own = (stats_alt[:, 1] == stats_ref[:, 1]).mean()
    flip = np.any(stats[:, :3] != stats_ref[:, :3], axis=1)
    err = state_rel_err(w, ref)
    e0 = _energy(orc, w0)
    de_gpu = np.abs(_energy(orc, w) - e0) / np.abs(e0)
    de_ref = np.abs(_energy(orc, ref) - e0) / np.abs(e0)
    ch = ~calm
    print(f"{len(sel)} orbits, max attempts {stats_ref[:, 0].max()}; identical accepted-step "
          f"counts GPU {same.mean():.4f}, oracle under a one-ulp change {own:.4f}.  "
          f"{calm.sum()} insensitive orbits ({calm.mean():.1%}; of the longest 1,024: "
          f"{calm[longest].sum()}): error median {np.median(err[calm]):.2e}, max "
          f"{err[calm].max():.2e}, {flip[calm].sum()} with other step counts.  {ch.sum()} "
          f"chaotic: |dE/E| median GPU {np.median(de_gpu[ch]):.2e} oracle "
          f"{np.median(de_ref[ch]):.2e}, 99% {np.percentile(de_gpu[ch], 99):.2e} / "
          f"{np.percentile(de_ref[ch], 99):.2e}, max {de_gpu[ch].max():.2e} / {de_ref[ch].max():.2e}")
    bad = np.nonzero(calm & (err > 1e-8))[0]
    for i in bad[:10]:
        print(f"orbit {sel[i]}: err {err[i]:.3e} sens {sens[i]:.1e} build {build[i]:.1e} "
              f"naccpt gpu {stats[i, 1]} oracle {stats_ref[i, 1]} T {T[i]:.1f}")
    assert 1.0 - same.mean() <= 3.0 * (1.0 - own) + 0.005
    assert calm.mean() >= 0.55
    assert len(bad) == 0
    assert np.median(err[calm]) < 1e-12
    assert flip[calm].mean() <= 0.01
    assert np.median(de_gpu[ch]) <= 2.0 * np.median(de_ref[ch])
    assert np.percentile(de_gpu[ch], 99) <= 2.0 * np.percentile(de_ref[ch], 99)
    assert de_gpu[ch].max() <= 3.0 * de_ref[ch].max()


def test_dense_output_parity():
    from gala_amd.potential import Hamiltonian
    orc = mw_oracle()
    rng = np.random.default_rng(5)
    n = 64
    w0 = np.vstack([rng.uniform(3, 20, (3, n)), rng.normal(0, 0.12, (3, n))])
    t = np.linspace(0.0, 600.0, 301)
    ref, st, _ = O.dop853(orc, w0, t, atol=1e-10, rtol=1e-10, nbatch=1, save_all=True)
    orbit = Hamiltonian(mw_product()).integrate_orbit(
        w0, t=t, Integrator="dopri853", Integrator_kwargs=dict(atol=1e-10, rtol=1e-10, nbatch=1))
    w = orbit.w()
    assert w.shape == (6, 301, n)
    assert np.max(state_rel_err(w, ref)) < 1e-8
    # interpolant at the interval ends reproduces the first output exactly
    assert np.array_equal(w[:, 0], w0)


def test_status_codes_and_errors():
    from gala_amd.integrate import dop853
    from gala_amd import _device as dev
    from gala_amd.potential import Hamiltonian
    pot = mw_product()
    w0 = np.array([[8.0], [0.0], [0.0], [0.0], [0.2], [0.0]])
    # nmax exceeded -> -2 (dop853.cpp:340-347)
    res = dop853(pot, w0, 0.0, 5000.0, 1.0, rtol=1e-12, atol=1e-12, nmax=5)
    assert dev.to_host(res["status"])[0] == -2
    st_o = O.dop853_orbits(mw_oracle(), w0, 0.0, 5000.0, 1.0, atol=1e-12, rtol=1e-12, nmax=5)[1]
    assert st_o[0] == -2
    with pytest.raises(RuntimeError):
        Hamiltonian(pot).integrate_orbit(w0[:, 0], dt=1.0, n_steps=5000, Integrator="dop853",
                                         Integrator_kwargs=dict(nmax=5, nbatch=1))
    # h0 = 0 -> Hairer's initial step guess (dop853.cpp:18-86), still correct
    res = dop853(pot, w0, 0.0, 500.0, 0.0, rtol=1e-10, atol=1e-10)
    ref = O.dop853_orbits(mw_oracle(), w0, 0.0, 500.0, 1.0, atol=1e-10, rtol=1e-10)[0]
    assert state_rel_err(dev.to_host(res["w_final"]), ref)[0] < 1e-8


def test_queue_order_invariance():
    """The work-queue order changes which lane runs an orbit, never its result."""
    from gala_amd.integrate import dop853
    from gala_amd import _device as dev
    orc = mw_oracle()
    w0, T = workloads.composite_dop853(vcirc_oracle(orc), n=5000, seed=9)
    T = T * 0.05
    pot = mw_product()
    a = dop853(pot, w0, 0.0, T, 1.0, rtol=1e-8, atol=1e-10)
    order = np.random.default_rng(0).permutation(w0.shape[1]).astype(np.int32)
    b = dop853(pot, w0, 0.0, T, 1.0, rtol=1e-8, atol=1e-10, order=order, block=128)
    assert np.array_equal(dev.to_host(a["w_final"]), dev.to_host(b["w_final"]))
    assert np.array_equal(dev.to_host(a["stats"]), dev.to_host(b["stats"]))


@pytest.mark.parametrize("layout", ["milky_way", "generic"])
def test_wide_tail_matches_one_lane_per_orbit(layout, monkeypatch):
    """The last orbits of each wave finish spread over 4-lane quads (at most
    16 left) and then 16-lane rows (at most 4 left); that changes the lane
    layout only, never a bit of the result (final states, status codes and
    step statistics), including the stiffness test, which nstiff=3 runs every
    few steps.  GAMD_DOP853_WIDE: 0 one lane to the end, 1 rows only, 2 (the
    default) quads then rows."""
    from gala_amd.integrate import dop853
    from gala_amd import _device as dev
    from gala_amd.potential import HernquistPotential, PlummerPotential
    orc = mw_oracle()
    w0, T = workloads.composite_dop853(vcirc_oracle(orc), n=3000, seed=21)
    T = T * 0.05
    if layout == "milky_way":
        pot = mw_product()
    else:
        pot = HernquistPotential(m=1e11, c=2.0) + PlummerPotential(m=1e10, b=1.0,
                                                                   origin=[1.0, 0.5, -0.2])
    out = {}
    for wide in ("0", "1", "2"):
        monkeypatch.setenv("GAMD_DOP853_WIDE", wide)
        for nstiff in (0, 3):
            r = dop853(pot, w0, 0.0, T, 1.0, rtol=1e-8, atol=1e-10, nstiff=nstiff)
            out[wide, nstiff] = [dev.to_host(r[k]) for k in ("w_final", "status", "stats")]
    for wide in ("1", "2"):
        for nstiff in (0, 3):
            for a, b in zip(out["0", nstiff], out[wide, nstiff]):
                assert np.array_equal(a, b)
    assert np.all(out["2", 0][1] == 1)


@pytest.mark.parametrize("n", [1, 4, 5, 17, 65])
def test_rows_equal_one_lane_on_extreme_orbits(n, monkeypatch):
    """A row's lanes hold one component each, take the tableau from each
    other's registers and share the Milky-Way evaluator's roots and logarithm;
    whatever the state, the results are one lane's, bit for bit: planar orbits
    (zeros of either sign), orbits through the centre, radii where the shared
    reciprocal over- or underflows, a start at the centre (NaN), with and
    without dense output, for a few steps at least."""
    from gala_amd.integrate import dop853
    from gala_amd import _device as dev
    rng = np.random.default_rng(31)
    w0 = np.vstack([rng.uniform(-20, 20, (3, n)), rng.normal(0, 0.12, (3, n))])
    edge = np.zeros((6, 9))
    edge[:, 0] = [8.0, 0.0, 0.0, 0.0, 0.2, 0.0]
    edge[:, 1] = [8.0, -0.0, -0.0, 0.0, -0.2, -0.0]
    edge[:, 2] = [0.0, 0.0, 5.0, 0.0, 0.0, 0.1]
    edge[:, 3] = [1e-3, 0.0, 0.0, 0.0, 1e-3, 0.0]
    edge[:, 4] = [1e100, 1e99, -1e100, 0.1, 0.2, 0.3]
    edge[:, 5] = [1e-100, 1e-101, 1e-100, 0.0, 0.0, 1e-5]
    edge[:, 6] = [0.0, 0.0, 0.0, 0.1, 0.0, 0.0]
    edge[:, 7] = [3.0, 1e-310, 2.0, -0.1, 0.0, 1e-310]
    edge[:, 8] = [1e160, 0.0, 0.0, 0.0, 0.0, 0.0]
    m = min(n, 9)
    w0[:, n - m:] = edge[:, 9 - m:]
    pot = mw_product()
    t_out = np.linspace(0.0, 40.0, 9)
    out = {}
    for wide in ("0", "1", "2"):
        monkeypatch.setenv("GAMD_DOP853_WIDE", wide)
        for dense in (None, t_out):
            r = dop853(pot, w0, 0.0, 40.0, 1.0, rtol=1e-8, atol=1e-10, nmax=300, t_out=dense,
                       n_tail=n)
            out[wide, dense is None] = [dev.to_host(r[k]) for k in ("w_final", "status", "stats")]
            if dense is not None:
                done = out[wide, False][1] == 1
                out[wide, False].append(dev.to_host(r["w_out"])[:, :, done])
    for wide in ("1", "2"):
        for final_only in (True, False):
            for a, b in zip(out["0", final_only], out[wide, final_only]):
                same = a == b
                if a.dtype == np.float64:  # NaN equals NaN; zeros keep their sign
                    same = np.where(np.isnan(a), np.isnan(b),
                                    same & (np.signbit(a) == np.signbit(b)))
                assert np.all(same), (wide, final_only)


def test_dedicated_tail_waves_match():
    """n_tail > 0 runs the queue order's first orbits on dedicated 16-lane
    rows from the start; the results are those of the one-lane kernel, bit
    for bit, for the longest-first order and for a shuffled one."""
    from gala_amd.integrate import dop853
    from gala_amd import _device as dev
    orc = mw_oracle()
    w0, T = workloads.composite_dop853(vcirc_oracle(orc), n=6000, seed=23)
    T = T * 0.05
    pot = mw_product()
    base = dop853(pot, w0, 0.0, T, 1.0, rtol=1e-8, atol=1e-10)
    ref = [dev.to_host(base[k]) for k in ("w_final", "status", "stats")]
    lpt = workloads.cost_order(w0, T, pot.gradient, spread=1)
    shuffled = np.random.default_rng(1).permutation(w0.shape[1]).astype(np.int32)
    for order in (lpt, shuffled):
        for n_tail in (4, 37, 512, 100000):
            r = dop853(pot, w0, 0.0, T, 1.0, rtol=1e-8, atol=1e-10, order=order, n_tail=n_tail)
            for k, a in zip(("w_final", "status", "stats"), ref):
                assert np.array_equal(dev.to_host(r[k]), a), (k, n_tail)


@pytest.mark.parametrize("layout", ["milky_way", "generic"])
def test_dense_output_same_in_every_lane_layout(layout, monkeypatch):
    """With dense output too, the orbits that set a launch's length move to
    4-lane quads and 16-lane rows (at the queue's end, and from the start
    for the n_tail longest); every sample, final state, status and step count
    equals one lane per orbit to the end, bit for bit."""
    from gala_amd.integrate import dop853, pilot_order
    from gala_amd import _device as dev
    from gala_amd.potential import HernquistPotential, PlummerPotential
    orc = mw_oracle()
    w0, T = workloads.composite_dop853(vcirc_oracle(orc), n=3000, seed=27)
    T = T * 0.05
    t_out = np.linspace(0.0, 500.0, 33)
    if layout == "milky_way":
        pot = mw_product()
    else:
        pot = HernquistPotential(m=1e11, c=2.0) + PlummerPotential(m=1e10, b=1.0,
                                                                   origin=[1.0, 0.5, -0.2])
    keys = ("w_out", "w_final", "status", "stats")
    monkeypatch.setenv("GAMD_DOP853_WIDE", "0")
    ref = [dev.to_host(v) for v in
           (dop853(pot, w0, 0.0, T, 1.0, rtol=1e-8, atol=1e-10, t_out=t_out)[k] for k in keys)]
    st = ref[2]
    reached = (t_out[:, None] <= T[None, :]) & (st == 1)[None, :]
    print(f"{reached.sum()} samples reached of {reached.size}")
    order = pilot_order(pot, w0, 0.0, T, 1.0, rtol=1e-8, atol=1e-10)
    for wide, n_tail, o in (("1", 0, None), ("2", 0, None), ("2", 256, order),
                            ("2", 100000, order)):
        monkeypatch.setenv("GAMD_DOP853_WIDE", wide)
        r = dop853(pot, w0, 0.0, T, 1.0, rtol=1e-8, atol=1e-10, t_out=t_out, order=o,
                   n_tail=n_tail)
        got = [dev.to_host(r[k]) for k in keys]
        m = np.broadcast_to(reached[None], ref[0].shape)
        assert np.array_equal(got[0][m], ref[0][m]), (wide, n_tail)
        for k, a, b in zip(keys[1:], ref[1:], got[1:]):
            assert np.array_equal(a, b), (wide, n_tail, k)


def test_order_entries_naming_no_orbit_are_skipped():
    """gamd_dop853 skips order entries outside 0..N-1 and keeps
    GAMD_STATUS_NOT_RUN (0) for the orbits the order does not name.  Here
    the first 200,000 of 262,144 slots name no orbit (more slots than the
    persistent grid has lanes): waves whose draws bring nothing must draw
    again, so every named orbit still runs, with the results of a run over
    the named orbits alone."""
    import torch
    from gala_amd import _device as dev
    from gala_amd import _lib
    from gala_amd.integrate import dop853
    lib = _lib.load()
    pot = mw_product()
    n = 262144
    w0, T = workloads.composite_dop853(vcirc_oracle(mw_oracle()), n=n, seed=41)
    T = T * 0.01
    named = np.sort(np.random.default_rng(2).choice(n, n - 200000, replace=False))
    order = np.concatenate([np.full(200000, -1), named]).astype(np.int32)
    w0d, t1 = dev.to_dev(w0), dev.to_dev(T)
    t0 = torch.zeros(n, dtype=torch.float64, device="cuda")
    h0 = torch.ones(n, dtype=torch.float64, device="cuda")
    wfin = torch.full((6, n), np.nan, dtype=torch.float64, device="cuda")
    status = torch.full((n,), 99, dtype=torch.int32, device="cuda")
    stats = torch.zeros((n, 4), dtype=torch.int64, device="cuda")
    ordd = dev.to_dev(order, dtype=torch.int32)
    print(f"{n} slots, {named.size} naming orbits", flush=True)
    rc = lib.gamd_dop853(pot.c_handle, w0d.data_ptr(), n, t0.data_ptr(), t1.data_ptr(),
                         h0.data_ptr(), 1e-8, 1e-10, 0, 0, 0.0, None, 0, None, wfin.data_ptr(),
                         status.data_ptr(), stats.data_ptr(), ordd.data_ptr(), 0, 0,
                         dev.stream_ptr())
    assert rc == 0
    st = dev.to_host(status)
    assert np.all(st[np.setdiff1d(np.arange(n), named)] == 0)
    ref = dop853(pot, np.ascontiguousarray(w0[:, named]), 0.0, np.ascontiguousarray(T[named]),
                 1.0, rtol=1e-8, atol=1e-10)
    assert np.array_equal(st[named], dev.to_host(ref["status"]))
    assert np.array_equal(dev.to_host(wfin)[:, named], dev.to_host(ref["w_final"]))
    assert np.array_equal(dev.to_host(stats)[named], dev.to_host(ref["stats"]))


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("nmax", [0, 40])
def test_rows_without_an_orbit_repeat_another(n, nmax, monkeypatch):
    """A few orbits of very different lengths, some stopped by nmax, on rows
    from the start, from the queue's end or dedicated: a row whose orbit has
    ended repeats another row's, and every orbit's final state, status, step
    counts and dense samples are those of one lane per orbit, bit for bit."""
    from gala_amd.integrate import dop853
    from gala_amd import _device as dev
    w0, _ = workloads.composite_dop853(vcirc_oracle(mw_oracle()), n=n, seed=5)
    T = 40.0 * 3.0 ** (np.arange(n) % 4)
    t_out = np.linspace(0.0, 40.0, 9)
    out = {}
    for wide, n_tail in (("0", 0), ("1", 0), ("2", 0), ("2", n)):
        monkeypatch.setenv("GAMD_DOP853_WIDE", wide)
        r = dop853(mw_product(), w0, 0.0, T, 1.0, rtol=1e-9, atol=1e-10, nmax=nmax, n_tail=n_tail)
        d = dop853(mw_product(), w0, 0.0, T, 1.0, rtol=1e-9, atol=1e-10, nmax=nmax, n_tail=n_tail,
                   t_out=t_out)
        out[wide, n_tail] = [dev.to_host(r[k]) for k in ("w_final", "status", "stats")] + [
            dev.to_host(d[k]) for k in ("w_final", "status", "stats")]
        if not nmax:  # samples past an orbit's last step are left as they were
            out[wide, n_tail].append(dev.to_host(d["w_out"]))
    for got in out.values():
        for a, b in zip(out["0", 0], got):
            np.testing.assert_array_equal(a, b)
