"""GPU SCF expansion (the SCF component of the potential table) against the
Fortran golden vectors (rtol 1e-6, as gala's test_accp_fortran.py) and the
oracle (1e-12), plus SCF orbits against the oracle."""
import numpy as np
import pytest

from gala_amd import workloads
from oracle import oracle as O
from tests.helpers import rel_err, state_rel_err
from tests.test_oracle_scf import NAMES, fortran_case

pytestmark = pytest.mark.gpu


def product_scf(m, r_s, S, T, G=None):
    from gala_amd.potential import SCFPotential
    from gala_amd.units import UnitSystem
    units = UnitSystem(G=G) if G is not None else None
    return SCFPotential(m=m, r_s=r_s, Snlm=S, Tnlm=T, units=units)


@pytest.mark.parametrize("name", NAMES)
def test_fortran_golden(name):
    xyz, S, T, accp = fortran_case(name)
    pot = product_scf(1.0, 1.0, S, T, G=1.0)
    np.testing.assert_allclose(pot.energy(xyz), -accp[:, -1], rtol=1e-6)
    g = pot.gradient(xyz)
    np.testing.assert_allclose(g.T, accp[:, :3], rtol=1e-6, atol=1e-7 * np.abs(accp[:, :3]).max())


def test_oracle_parity_benchmark_coefficients():
    S, T = workloads.scf_coefficients()
    pot = product_scf(1e12, 20.0, S, T)
    orc = [O.scf(1e12, 20.0, S, T)]
    rng = np.random.default_rng(0)
    r = np.exp(rng.uniform(np.log(1.0), np.log(200.0), 2000))
    q = r * rng.normal(size=(3, 2000)) / np.linalg.norm(rng.normal(size=(3, 2000)), axis=0)
    q = r / np.linalg.norm(q, axis=0) * q
    assert np.max(rel_err(pot.energy(q), O.value(orc, q))) < 1e-12
    g, go = pot.gradient(q), O.gradient(orc, q)
    assert np.max(np.abs(g - go) / np.linalg.norm(go, axis=0)) < 1e-11
    rho, rho_o = pot.density(q), O.density(orc, q)
    assert np.max(np.abs(rho - rho_o) / np.max(np.abs(rho_o))) < 1e-11


def test_generic_layout_matches():
    """A shifted SCF component takes the generic evaluator path; it must agree
    with the oracle as well."""
    from gala_amd.potential import SCFPotential
    S, T = workloads.scf_coefficients(nmax=4, lmax=3, seed=2)
    q0 = np.array([0.5, -0.2, 0.1])
    pot = SCFPotential(m=1e11, r_s=5.0, Snlm=S, Tnlm=T, origin=q0)
    orc = [O.scf(1e11, 5.0, S, T, q0=q0)]
    q = np.random.default_rng(1).uniform(-30, 30, (3, 500))
    g, go = pot.gradient(q), O.gradient(orc, q)
    assert np.max(np.abs(g - go) / np.linalg.norm(go, axis=0)) < 1e-11


@pytest.mark.parametrize("nmax,lmax", [(0, 0), (1, 0), (2, 1), (10, 6), (10, 5), (0, 10), (3, 8),
                                       (20, 10)])
def test_every_size_matches_oracle(nmax, lmax):
    """Smallest and largest tables, rows of one batch and of several, the
    written-out size beside its neighbours; inner, outer and ordinary radii.
    T_nl0 is not zero here and must not matter.  The bounds are those of
    test_oracle_parity_benchmark_coefficients at ordinary radii."""
    S, T = workloads.scf_coefficients(nmax, lmax, seed=nmax + lmax)
    T[:, :, 0] = 0.25
    pot = product_scf(1e12, 20.0, S, T)
    orc = [O.scf(1e12, 20.0, S, T)]
    rng = np.random.default_rng(nmax * 16 + lmax)
    n = 333
    q = rng.normal(size=(3, n))
    q *= np.exp(rng.uniform(np.log(1.0), np.log(200.0), n)) / np.linalg.norm(q, axis=0)
    v, vo = pot.energy(q), O.value(orc, q)
    assert np.max(np.abs(v - vo) / np.max(np.abs(vo))) < 1e-12
    g, go = pot.gradient(q), O.gradient(orc, q)
    assert np.max(np.abs(g - go) / np.max(np.linalg.norm(go, axis=0))) < 1e-11
    rho, rho_o = pot.density(q), O.density(orc, q)
    assert np.max(np.abs(rho - rho_o) / np.max(np.abs(rho_o))) < 1e-11
    # on the axis the value is finite and the gradient's angular part is 0 / 0
    ax = np.array([[0.0, 0.0], [0.0, 0.0], [3.0, -40.0]])
    np.testing.assert_allclose(pot.energy(ax), O.value(orc, ax), rtol=1e-11)
    assert np.isnan(pot.gradient(ax)).all()


def test_scf_leapfrog_and_dop853_parity():
    from gala_amd import _device as dev
    from gala_amd.integrate import dop853, leapfrog
    S, T = workloads.scf_coefficients()
    pot = product_scf(1e12, 20.0, S, T)
    orc = [O.scf(1e12, 20.0, S, T)]

    def vc(q):
        g = O.gradient(orc, q)
        r = np.linalg.norm(q, axis=0)
        return np.sqrt(r * np.abs(np.sum(g * q / r, axis=0)))
    w0, dt, _ = workloads.scf_leapfrog(vc, n=256, seed=3)
    t = np.arange(401) * dt
    ref = O.leapfrog(orc, w0, t, save_all=False)
    _, wf = leapfrog(pot, w0, dt, 400, save=False)
    assert np.max(state_rel_err(dev.to_host(wf), ref)) < 1e-10
    # the whole workload length: 10,000 steps (5 Gyr).  The expansion's random
    # S_nlm, T_nlm make the potential triaxial and a fifth of these orbits
    # chaotic: in the oracle itself a one-ulp change of the initial state, or
    # gala's -Ofast build flags instead of IEEE ones, moves their final
    # states by up to O(1).  Orbits insensitive to both (response below
    # 1e-12) must match within 1e-10; the chaotic ones are held to the
    # oracle's energy-error distribution.
    t = np.arange(10001) * dt
    ref = O.leapfrog(orc, w0, t, save_all=False)
    pert = w0.copy()
    pert[0] = np.nextafter(pert[0], np.inf)
    sens = state_rel_err(O.leapfrog(orc, pert, t, save_all=False), ref)
    build = state_rel_err(O.leapfrog(orc, w0, t, save_all=False, fast=True), ref)
    _, wf = leapfrog(pot, w0, dt, 10000, save=False)
    w = dev.to_host(wf)
    err = state_rel_err(w, ref)
    calm = (sens < 1e-12) & (build < 1e-12)
    ch = ~calm
    e0 = O.value(orc, w0[:3]) + 0.5 * np.sum(w0[3:] ** 2, axis=0)
    de_gpu = np.abs(O.value(orc, w[:3]) + 0.5 * np.sum(w[3:] ** 2, axis=0) - e0) / np.abs(e0)
    de_ref = np.abs(O.value(orc, ref[:3]) + 0.5 * np.sum(ref[3:] ** 2, axis=0) - e0) / np.abs(e0)
    print(f"10,000 steps: {calm.sum()} of {len(calm)} orbits insensitive, max error "
          f"{err[calm].max():.2e}; the other {ch.sum()}: |dE/E| median GPU "
          f"{np.median(de_gpu[ch]):.2e} oracle {np.median(de_ref[ch]):.2e}, max GPU "
          f"{de_gpu[ch].max():.2e} oracle {de_ref[ch].max():.2e}")
    assert calm.mean() >= 0.7
    assert err[calm].max() < 1e-10
    assert np.median(de_gpu[ch]) <= 2.0 * np.median(de_ref[ch])
    assert de_gpu[ch].max() <= 3.0 * de_ref[ch].max()
    res = dop853(pot, w0[:, :64], 0.0, 300.0, 1.0, rtol=1e-8, atol=1e-10)
    ref2, st, _ = O.dop853_orbits(orc, w0[:, :64], 0.0, 300.0, 1.0, atol=1e-10, rtol=1e-8)
    assert np.array_equal(dev.to_host(res["status"]), st)
    assert np.median(state_rel_err(dev.to_host(res["w_final"]), ref2)) < 1e-9
