"""The short FP64 forms of the bispectrum and power-spectrum arithmetic against the C library's, both from the kernels'
own functions (threepoint_amd/csrc/tp_device.h, tp_power_dev.h) built for the host: over every size of ell and every
n_eff, far outside a survey's too, the short forms give a number where the library's give one, to rounding, and none
where those give none (a call with a non-finite value is refused)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
SRC = r"""
#include "tp_power_dev.h"
// the z-only factors of BiHalofit (Takahashi et al. 2020, app. B)
static TpNode64 node(double D1, double sigma8, double rs, double ne, double fK, double h, double ns, double norm)
{
    const double ln10 = 2.302585092994045684, L = log10(D1 * sigma8), hr = h / rs;
    TpNode64 N;
    N.wz = 1e-9; N.ks = rs / fK; N.lnks = log(N.ks); N.inv_rs = 1. / rs;
    N.lnA0 = ln10 * (-2.167 - 2.944 * L - 1.106 * L * L - 2.865 * L * L * L);
    N.c1 = pow(10., 0.182 + 0.57 * ne); N.m031ln10 = -0.310 * ln10;
    N.bn = pow(10., -3.428 - 2.681 * L + 1.624 * L * L - 0.095 * L * L * L); N.cn = pow(10., 0.159 - 1.107 * ne);
    N.a0ln = ln10 * (-4.348 - 3.006 * ne - 0.5745 * ne * ne); N.a1ln = ln10 * pow(10., -0.9 + 0.2 * ne);
    N.acap = 1. - (2. / 3.) * ns;
    N.b0ln = ln10 * (-1.731 - 2.845 * ne - 1.4995 * ne * ne - 0.2811 * ne * ne * ne); N.b1ln = ln10 * 0.007;
    N.fn = pow(10., -10.533 - 16.838 * ne - 9.3048 * ne * ne - 1.8263 * ne * ne * ne);
    N.gn = pow(10., 2.787 + 2.405 * ne + 0.4577 * ne * ne); N.hn = pow(10., -1.118 - 0.394 * ne);
    N.mn = pow(10., -2.605 - 2.434 * L + 5.71 * L * L); N.nn = pow(10., -4.468 - 3.08 * L + 1.035 * L * L);
    N.mun = pow(10., 15.312 + 22.977 * ne + 10.9579 * ne * ne + 1.6586 * ne * ne * ne);
    N.nun = pow(10., 1.347 + 1.246 * ne + 0.4525 * ne * ne);
    N.pn = pow(10., 0.071 - 0.433 * ne); N.en = pow(10., -0.632 + 0.646 * ne);
    N.D1sq = D1 * D1; N.dn = pow(10., -0.483 + 0.892 * L - 0.043); N.lnkoff = log(2997.9 / rs);
    N.pk_pref = h * h * h * 2 * tpd::kPi * tpd::kPi * norm * norm / (hr * hr * hr);
    return N;
}
// rows of D1, sigma8, r_sigma, n_eff, f_K, h, n_s, norm, l1, l2, l3; nk > 0: the tabulated P(k)
extern "C" void run(int n, const double *a, int nk, const double *k, const double *p, const int *idx, double *lib,
                    double *fast)
{
    for (int i = 0; i < n; ++i, a += 11) {
        const TpNode64 N = node(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7]);
        TpEH64 E{a[5], 0.9, 0.1, 0.43 * 110, 0.3 * a[5] * a[5], 1.02, 2.0, 3. + a[6], 2.718281828, {}};
        E.tab.k = k; E.tab.p = p; E.tab.idx = idx; E.tab.nk = nk; E.tab.ng = 1;
        TpPointPre P;
        tp_point_pre<double>(a[8], a[9], a[10], &P);
        double q[3], lq[3];
        for (int j = 0; j < 3; ++j) { q[j] = P.l[j] * N.ks; lq[j] = P.ll[j] + N.lnks; }
        lib[i] = N.wz * tp_bispec_node<double, TpMathAny<double>>(N, E, q, lq, P.f2t, P.lr1, P.r2);
        fast[i] = N.wz * tp_bispec_node<double>(N, E, q, lq, P.f2t, P.lr1, P.r2);
    }
}

// a double whose functions are the library's: the power-spectrum templates take the short forms for double only
struct Lib {
    double v;
    Lib(double x = 0) : v(x) {}
};
static Lib operator+(Lib a, Lib b) { return a.v + b.v; }
static Lib operator-(Lib a, Lib b) { return a.v - b.v; }
static Lib operator*(Lib a, Lib b) { return a.v * b.v; }
static Lib operator/(Lib a, Lib b) { return a.v / b.v; }
static Lib operator-(Lib a) { return -a.v; }
static Lib pow(Lib a, Lib b) { return std::pow(a.v, b.v); }
static Lib exp(Lib a) { return std::exp(a.v); }
static Lib log(Lib a) { return std::log(a.v); }
static Lib sqrt(Lib a) { return std::sqrt(a.v); }
static Lib log1p(Lib a) { return std::log1p(a.v); }
static Lib fabs(Lib a) { return std::fabs(a.v); }
static double tp_dbl(Lib a) { return a.v; }

// rows of h, n_s, norm, Omega_m, w, ell (or k), z; form 0: the Limber integrand, 1: P(k, z), 2: the precomputed z-node,
// 3: the same without its branch for a far k
extern "C" void power(int n, const double *a, const double *tab, int n_z, int flags, int form, double *lib, double *fast)
{
    for (int i = 0; i < n; ++i, a += 7) {
        TpCosmoConst C{};
        C.h = a[0]; C.ns = a[1]; C.norm = a[2]; C.om = a[3]; C.ow = 1 - a[3]; C.w = a[4]; C.zmax = 3; C.n_z = n_z;
        C.eh_sqrt_alnu = 0.9; C.eh_sh = 110; C.eh_omh2 = a[3] * a[0] * a[0]; C.eh_theta2 = 1.02; C.eh_cL = 2;
        C.limber_pref = 1e-9;
        if (form == 1) {
            TpZAtT<Lib> Z;
            TpZAtT<double> Y;
            tp_z_at<Lib>(tab, n_z, 3, a[6], &Z);
            tp_z_at<double>(tab, n_z, 3, a[6], &Y);
            lib[i] = tp_pk_at<Lib>(C, Z, a[5], a[6], flags).v;
            fast[i] = tp_pk_at<double>(C, Y, a[5], a[6], flags);
            continue;
        }
        lib[i] = tp_limber_pk<Lib>(C, tab, n_z, a[5], a[6], flags).v;
        if (form == 0) {
            fast[i] = tp_limber_pk<double>(C, tab, n_z, a[5], a[6], flags);
            continue;
        }
        TpPNode N;
        tp_pnode_make(C, tab, n_z, a[6], &N);
        fast[i] = form == 2 ? tp_limber_pk_node<true>(C, N, a[5], log(a[5]), flags)
                            : tp_limber_pk_node<false>(C, N, a[5], log(a[5]), flags);
    }
}
"""


@pytest.fixture(scope="module")
def forms(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("node")
    (d / "t.hip").write_text(SRC)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", "-shared", "-fPIC", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-I" + os.path.join(ROOT, "threepoint_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"), str(d / "t.hip"), "-o", str(d / "t.so")],
                   check=True, stderr=subprocess.DEVNULL)
    return ctypes.CDLL(str(d / "t.so"))


# n_eff of a LCDM universe is -2.95 to -1.5; a given P(k) can have any.  The tolerance: the two forms share every
# argument but alpha_n and beta_n (an ulp each), arguments reach 700, and an ulp of one changes the exponential by
# 700 2^-53 = 8e-14; some thirty of them meet in a value, whose terms do not cancel in these triangles.
@pytest.mark.parametrize("tabulated", [False, True])
@pytest.mark.parametrize("ne", [(-2.95, -0.8), (-1.0, 4.0)])
@pytest.mark.parametrize("ell", [(0, 5), (-5, 8), (-60, 60)])
def test_short_forms_are_finite_where_the_library_forms_are(forms, ne, ell, tabulated):
    n, rng = 100000, np.random.default_rng(1)
    a = np.empty((n, 11))
    for j, (lo, hi) in enumerate([(-1.5, 0), (-1, 0.7), (-5, 1.3)]):
        a[:, j] = 10 ** rng.uniform(lo, hi, n)
    a[:, 3] = rng.uniform(*ne, n)
    a[:, 4] = 10 ** rng.uniform(-1, 3.7, n)
    a[:, 5], a[:, 6], a[:, 7] = rng.uniform(0.5, 0.9, n), rng.uniform(0.8, 1.2, n), 10 ** rng.uniform(-5, -3, n)
    l, r, phi = 10 ** rng.uniform(*ell, n), rng.uniform(0.5, 1, n), rng.uniform(0, 2.5, n)
    a[:, 8], a[:, 9], a[:, 10] = l, l * r, l * np.sqrt(1 + r * r + 2 * r * np.cos(phi))
    k = np.geomspace(1e-4, 50, 12)
    p = 2e4 * (k / 0.02) / (1 + (k / 0.02) ** 2.5)
    idx = np.zeros(1, np.int32)
    lib, fast = np.empty(n), np.empty(n)
    ptr = [v.ctypes.data_as(ctypes.c_void_p) for v in (a, k, p, idx, lib, fast)]
    forms.run(n, ptr[0], 12 if tabulated else 0, ptr[1], ptr[2], ptr[3], ptr[4], ptr[5])
    fin = np.isfinite(lib)
    assert fin.sum() > 1000
    assert np.array_equal(np.isfinite(fast), fin)
    seen = fin & (np.abs(lib) > 1e-280)
    d = np.abs(fast[seen] / lib[seen] - 1)
    print("finite %.3f, largest difference %.1e" % (fin.mean(), d.max()))
    assert d.max() < 1e-11


@pytest.fixture(scope="module")
def z_tables():
    from _oracle import Oracle
    from threepoint_amd import workloads as W
    t = Oracle(W.fiducial(), W.fiducial_nz()).tables()
    return np.concatenate([t[k] for k in ("f_K", "g", "D1", "r_sigma", "n_eff", "ncur")]), len(t["f_K"])


# The tolerance: as above, with one power (1 + Delta^2)^beta, beta < 5, over another.  Form 3 is for the multipoles of T1,
# up to 1e15 and down to where a bisected domain could reach.
@pytest.mark.parametrize("form, ell", [(0, (-1, 6)), (0, (-300, 300)), (1, (-6, 3)), (1, (-300, 300)), (2, (-1, 6)),
                                       (2, (-300, 300)), (3, (-65, 15))])
@pytest.mark.parametrize("flags", [0, 1, 2, 3])
def test_power_spectrum_of_any_wavenumber(forms, z_tables, form, ell, flags):
    n, rng = 100000, np.random.default_rng(2)
    a = np.column_stack([rng.uniform(0.5, 0.9, n), rng.uniform(0.8, 1.2, n), 10 ** rng.uniform(-5, -3, n),
                         rng.uniform(0.1, 0.9, n), rng.uniform(-1.5, -0.5, n), 10 ** rng.uniform(*ell, n),
                         rng.uniform(0.02, 3, n)])
    tab, n_z = z_tables
    lib, fast = np.empty(n), np.empty(n)
    a_, t_, l_, f_ = (v.ctypes.data_as(ctypes.c_void_p) for v in (a, tab, lib, fast))
    forms.power(n, a_, t_, n_z, flags, form, l_, f_)
    fin = np.isfinite(lib)
    assert fin.sum() > 1000
    assert np.array_equal(np.isfinite(fast), fin)
    seen = fin & (np.abs(lib) > 1e-280)
    d = np.abs(fast[seen] / lib[seen] - 1)
    print("finite %.3f, largest difference %.1e" % (fin.mean(), d.max()))
    assert d.max() < 5e-12
