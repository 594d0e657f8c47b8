"""GPU parity of the convergence power spectrum and <Map^2> against the CPU FP64 oracle.

Point values (P(k, z), the Limber integrand, Pell) agree to rounding (1e-12 relative); the adaptive
integrals (P_kappa, <Map^2>) take the oracle's decision sequence, so their point counts are equal
and their values agree to rounding too (1e-10).
"""
import math

import numpy as np
import pytest

import threepoint_amd as tp
from threepoint_amd import workloads as W

pytestmark = pytest.mark.gpu
A = 2.9088820866e-4


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return np.abs(a - b) / np.maximum(np.abs(b), 1e-300)


@pytest.mark.parametrize("flags", [0, tp.PK_LINEAR])
def test_pk_at_z_matches_oracle(fid_tables, fid_oracle, flags):
    rng = np.random.default_rng(7)
    n = 400
    kz = np.stack([np.exp(rng.uniform(np.log(1e-4), np.log(1e2), n)), rng.uniform(0, 3.0, n)], 1)
    kz[:4, 1] = [0.0, 1e-6, 3.0, 2.9999999]
    g = fid_tables.pk_at_z(kz, flags=flags)
    name = "linear_pk_at_z" if flags & tp.PK_LINEAR else "pk_nonlinear"
    o = np.array([fid_oracle.scalar(name, k, z) for k, z in kz])
    r = rel(g, o)
    print("P(k, z) flags %d max rel %.3e" % (flags, r.max()))
    assert r.max() < 1e-12


@pytest.mark.parametrize("flags", [0, tp.PK_LINEAR, tp.PK_T17])
def test_limber_integrand_matches_oracle(fid_tables, fid_oracle, flags):
    rng = np.random.default_rng(11)
    n = 400
    lz = np.stack([np.exp(rng.uniform(0, np.log(1e5), n)), rng.uniform(0, 3.0, n)], 1)
    lz[:3, 1] = [0.0, 0.99e-5, 3.0]
    g = fid_tables.limber_pkappa(lz, flags=flags)
    o = np.array([fid_oracle.scalar("limber_pkappa", l, z, flags) for l, z in lz])
    assert g[0] == 0 and g[1] == 0
    r = rel(g[2:], o[2:])
    print("limber flags %d max rel %.3e" % (flags, r.max()))
    assert r.max() < 1e-12


@pytest.mark.parametrize("flags", [0, tp.PK_LINEAR, tp.PK_T17])
def test_far_wavenumbers_match_oracle(fid_tables, fid_oracle, flags):
    """k and ell of 1e-60 to 1e60, far outside the range of the short FP64 forms: the values the library's functions
    give there, to the rounding of (3 + n_s) ln k (550 ulp; the oracle takes powers).  A k that is no number is refused."""
    rng = np.random.default_rng(13)
    k = 10 ** rng.uniform(-60, 60, 300)
    z = rng.uniform(0.05, 3.0, 300)
    kz = np.stack([k, z], 1)
    if not flags & tp.PK_T17:
        name = "linear_pk_at_z" if flags & tp.PK_LINEAR else "pk_nonlinear"
        o = np.array([fid_oracle.scalar(name, *p) for p in kz])
        assert rel(fid_tables.pk_at_z(kz, flags=flags), o).max() < 1e-11
    o = np.array([fid_oracle.scalar("limber_pkappa", *p, flags) for p in kz])
    assert rel(fid_tables.limber_pkappa(kz, flags=flags), o).max() < 1e-11
    o = np.array([fid_oracle.scalar("pell", l, 0.0, 1.0, flags) for l in k])
    assert rel(fid_tables.pell(k, flags=flags), o).max() < 1e-11
    for call in (fid_tables.pk_at_z, fid_tables.limber_pkappa):
        with pytest.raises(tp.TpError, match="non-finite"):
            call(np.array([[-1.0, 1.0]]), flags=flags)


@pytest.mark.parametrize("flags,sigma", [(0, 0.0), (tp.PK_T17, 0.0), (0, 0.3)])
def test_pell_matches_oracle(fid_tables, fid_oracle, flags, sigma):
    """sigma = 0.3 with the reference's default density n (bispectrum.hpp:120-121, integer division
    included): the shape noise then dominates; sigma = 0 tests the Limber sum itself."""
    ell = np.concatenate([[0.0], np.geomspace(1, 5e4, 120)])
    n = 4096 * 4096 // 10 // 10 * math.pi * math.pi / 180 / 180
    g = fid_tables.pell(ell, flags=flags, sigma=sigma, n_gal=n)
    o = np.array([fid_oracle.scalar("pell", l, sigma, n, flags) for l in ell])
    assert g[0] == 0.5 * sigma * sigma / n
    r = rel(g[1:], o[1:])
    print("Pell flags %d sigma %g max rel %.3e" % (flags, sigma, r.max()))
    assert r.max() < 1e-12


def test_pkappa_batch_matches_oracle(gpu_ctx, fid_nz):
    """Two cosmologies, multipoles interleaved: the batched cubature reproduces each integral's
    one-at-a-time decision sequence (equal point counts)."""
    c2 = tp.Cosmology(h=0.65, sigma8=0.9, omb=0.045, ns=0.95, w=-0.9, om=0.35)
    tabs = tp.CosmologyTables([W.fiducial(), c2], fid_nz, 100, 3.0, gpu_ctx)
    from _oracle import Oracle
    orcs = [Oracle(W.fiducial(), fid_nz), Oracle(c2, fid_nz)]
    ell = np.geomspace(1, 1e5, 24)
    ic = np.arange(24) % 2
    v, e, n = tabs.pkappa_batch(ell, ic, reltol=1e-6)
    for i in range(24):
        ov, oe, on = orcs[ic[i]].convergence_power_spectrum(ell[i], 1e-6)
        assert n[i] == on, (i, n[i], on)
        assert abs(v[i] / ov - 1) < 1e-10 and abs(e[i] / oe - 1) < 1e-6


@pytest.mark.parametrize("flags,sigma", [(0, 0.0), (tp.PK_T17, 0.0), (0, 0.3)])
def test_map2_batch_matches_oracle(fid_tables, fid_oracle, flags, sigma):
    th = np.array([0.5, 1.0, 2.0, 4.0, 8.0, 16.0, 32.0]) * A
    v, e, n = fid_tables.map2_batch(th, reltol=1e-5, flags=flags, sigma=sigma, ngal=30.0)
    for i, t in enumerate(th):
        ov, oe, on = fid_oracle.map2(t, 1e-5, flags, sigma, 30.0)
        assert n[i] == on, (i, n[i], on)
        assert abs(v[i] / ov - 1) < 1e-10


def test_map2_shape_noise_closed_form(fid_tables):
    """Size-independent property: <Map^2> with noise minus without = sigma^2 / (2 n) / (8 pi theta^2)."""
    th = np.geomspace(0.5, 64, 25) * A
    m0 = fid_tables.map2_batch(th, reltol=1e-7)[0]
    m1 = fid_tables.map2_batch(th, reltol=1e-7, sigma=0.3, ngal=30.0)[0]
    cf = 0.09 / (2 * 30.0 / A ** 2) / (8 * np.pi * th ** 2)
    assert np.max(np.abs((m1 - m0) / cf - 1)) < 1e-5


def test_power_with_tabulated_pk(gpu_ctx, fid_nz):
    """The tabulated linear P(k) input feeds the power spectrum as it feeds the bispectrum."""
    from _oracle import Oracle
    c = W.fiducial()
    eh = Oracle(c, fid_nz)
    kh = np.geomspace(1e-5, 1e3, 300)
    pk = np.array([eh.scalar("linear_pk", k) for k in kh]) * 1.05
    tabs = tp.CosmologyTables([c], fid_nz, 100, 3.0, gpu_ctx, pk=(kh, pk))
    orc = Oracle(c, fid_nz, pk=(kh, pk))
    ell = np.geomspace(10, 1e4, 9)
    g = tabs.pell(ell)
    o = np.array([orc.scalar("pell", l, 0.0, 1.0, 0) for l in ell])
    assert rel(g, o).max() < 1e-12
    v, e, n = tabs.map2_batch(np.array([2.0, 8.0]) * A)
    for i, t in enumerate([2.0, 8.0]):
        ov, oe, on = orc.map2(t * A, 1e-5)
        assert n[i] == on and abs(v[i] / ov - 1) < 1e-10


@pytest.mark.parametrize("n", [16, 40, 1100])
@pytest.mark.parametrize("flags,sigma,reltol", [(0, 0.0, 1e-5), (tp.PK_T17, 0.3, 5e-6), (tp.PK_LINEAR, 0.0, 1e-3)])
def test_map2_batch_sizes_agree(fid_tables, n, flags, sigma, reltol):
    """Integrals finished on the device, in either workgroup size, and in rounds take the same steps in the same
    order: equal bits."""
    th = np.geomspace(0.3, 100, n) * A
    v, e, m = fid_tables.map2_batch(th, reltol=reltol, flags=flags, sigma=sigma, ngal=30.0)
    pick = np.unique(np.linspace(0, n - 1, 45).astype(int))
    for c in np.array_split(pick, 4):  # fewer than 16 to a call
        rv, re, rm = fid_tables.map2_batch(th[c], reltol=reltol, flags=flags, sigma=sigma, ngal=30.0)
        assert np.array_equal(v[c], rv) and np.array_equal(e[c], re) and np.array_equal(m[c], rm)


@pytest.mark.parametrize("reltol", [5e-6, 5e-5])
def test_map2_integrals_that_outgrow_the_device(gpu_ctx, fid_nz, reltol):
    """A coarsely tabulated P(k) has kinks: integrals that would hold more regions than the device keeps of one (all of
    them at the tighter tolerance) are evaluated in rounds, with the bits of smaller calls; a round limit ends the
    call."""
    kh = np.geomspace(1e-4, 50, 12)
    tabs = tp.CosmologyTables([W.fiducial()], fid_nz, 100, 3.0, gpu_ctx, pk=(kh, 2e4 * (kh / 0.02) / (1 + (kh / 0.02) ** 2.5)))
    th = np.geomspace(0.5, 64, 28) * A
    v, e, m = tabs.map2_batch(th, reltol=reltol, flags=tp.PK_LINEAR)
    held = (m // 17 + 1) // 2
    print("regions held: %d to %d" % (held.min(), held.max()))
    assert held.max() > 1024 or reltol > 5e-6
    for c in (slice(0, 14), slice(14, 28)):
        rv, re, rm = tabs.map2_batch(th[c], reltol=reltol, flags=tp.PK_LINEAR)
        assert np.array_equal(v[c], rv) and np.array_equal(e[c], re) and np.array_equal(m[c], rm)
    gpu_ctx.set_batch_limits(max_rounds=3)
    try:
        with pytest.raises(tp.TpError, match=r"code 4\).*round limit"):
            tabs.map2_batch(th, reltol=1e-5)
    finally:
        gpu_ctx.set_batch_limits()


def test_map2_of_tabulated_pk_takes_the_device_where_it_fits(gpu_ctx, fid_nz):
    """A table fine enough for the tolerance takes the device (one launch), a coarse one rounds, unless the tolerance is
    loose.  A fine table that is rough from entry to entry is taken for smooth: integrals that then hold more regions than
    the device keeps of one are finished in rounds.  The bits of calls in rounds (fewer than 16 integrals) each time."""
    th = np.geomspace(0.5, 64, 28) * A
    seen = set()
    for nk, rough, reltol, device in [(500, 0.0, 1e-4, True), (150, 0.0, 1e-4, False), (12, 0.0, 1e-3, True),
                                      (1000, 0.0, 3e-5, False), (1000, 0.02, 1e-4, True)]:
        kh = np.geomspace(1e-4, 50, nk)
        pk = 2e4 * (kh / 0.02) / (1 + (kh / 0.02) ** 2.5) * (1 + rough * (-1.0) ** np.arange(nk))
        tabs = tp.CosmologyTables([W.fiducial()], fid_nz, 100, 3.0, gpu_ctx, pk=(kh, pk))
        v, e, m = tabs.map2_batch(th, reltol=reltol)
        launches, outgrown = gpu_ctx.stats()["launches"], int(((m // 17 + 1) // 2 > 1024).sum())
        print("%d entries, %g: %d launches, %d of 28 outgrown" % (nk, reltol, launches, outgrown))
        assert (launches == 1) == (device and not outgrown)
        seen.add((device, outgrown > 0))
        for c in (slice(0, 14), slice(14, 28)):
            rv, re, rm = tabs.map2_batch(th[c], reltol=reltol)
            assert np.array_equal(v[c], rv) and np.array_equal(e[c], re) and np.array_equal(m[c], rm)
    assert {(True, False), (True, True)} <= seen


def test_power_rejects_bad_arguments(fid_tables):
    with pytest.raises(tp.TpError):
        fid_tables.map2_batch(np.array([0.0]))
    with pytest.raises(tp.TpError):
        fid_tables.pell(np.array([10.0]), flags=8)
    with pytest.raises(tp.TpError):
        fid_tables.pkappa_batch(np.array([10.0]), icosmo=np.array([3]))


def test_map2_and_t1_kept_pools_bit_identical(gpu_ctx, fid_tables):
    """<Map^2> and T1 batches give the same bits with their integrators reused or freshly allocated."""
    th = np.array([0.5, 2.0, 8.0, 32.0]) * A
    pairs = np.array([[4, 8, 8, 6, 6, 12], [8, 8, 8, 8, 8, 8]], dtype=float) * A
    area, ngal = (5 * 60 * A) ** 2, 30 / A ** 2
    try:
        m_ref = fid_tables.map2_batch(th, reltol=1e-5)
        t_ref = fid_tables.map3_cov_t1(pairs, area, 0.0, 0.3, ngal, tp.PK_T17, reltol=1e-3)
        m_again = fid_tables.map2_batch(th, reltol=1e-5)
        t_again = fid_tables.map3_cov_t1(pairs, area, 0.0, 0.3, ngal, tp.PK_T17, reltol=1e-3)
        gpu_ctx.set_keep_pool_bytes(0)
        m_fresh = fid_tables.map2_batch(th, reltol=1e-5)
        t_fresh = fid_tables.map3_cov_t1(pairs, area, 0.0, 0.3, ngal, tp.PK_T17, reltol=1e-3)
    finally:
        gpu_ctx.set_keep_pool_bytes(1 << 34)
    for r in (m_again, m_fresh):
        for a, b in zip(m_ref, r):
            assert np.array_equal(a, b)
    for r in (t_again, t_fresh):
        for a, b in zip(t_ref, r):
            assert np.array_equal(a, b)
