"""The FP32 mode of the library against its FP64 path.

The FP32 mode keeps the flow fields, the stencils and the Gauss-Seidel
solve in FP32, and keeps FP64 for the volume-fraction fluxes and mass sums,
the contact-line slip velocity and the pressure correction.  The pressure
solve's FFT+TDMA modes are FP64 by default; registered in the flow class
they are FP32, warm-started from the last correction, and iterative
refinement on the FP64 residual of the FFT+TDMA operator brings the
correction back to FP64-level accuracy.
Bars (stated here, measured against the FP64 GPU path on identical initial
states):

* velocity and pressure, relative L2 error after 20 steps <= 1e-5;
* volume drift over the run <= 1e-12 (the mass correction is FP64);
* phi stays in [0, 1];
* the pressure correction solves its Poisson problem to the refinement
  tolerance (default 1e-7, the relative rounding of the FP32 velocities it
  corrects; an FP32 solve alone reaches ~1e-6), or to 1e-10 when set so.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import felharness as H
from felharness import D, I
from felmpf import config as C
from felmpf.driver import GpuRun

pytestmark = pytest.mark.gpu


def _interior(cfg, a):
    return a[3:cfg.nk + 3, 3:cfg.nj + 3, 3:cfg.ni + 3]


@pytest.mark.parametrize("fp32_modes", [True, False], ids=["fp32_refine", "fp64_modes"])
@pytest.mark.parametrize("make", [C.droplet_impact, C.sessile_droplet],
                         ids=["droplet_impact", "sessile_droplet"])
def test_fp32_mode_tracks_fp64(make, fp32_modes):
    """Both FP32 configurations: FP32 pressure-solve modes with FP64
    refinement (the benchmark's FP32+refine) and FP64 modes."""
    base = make()
    cfg = base.scaled(64, 16, 32) if base.name == "droplet_impact" else base.scaled(32, 32, 32)
    out = {}
    for prec in (64, 32):
        g = GpuRun(cfg, precision=prec, fp32_modes=fp32_modes and prec == 32)
        assert H.gpu().felgpu_precision_() == prec
        v0 = _interior(cfg, g.field("phi1")).sum()
        g.steps(20)
        out[prec] = {f: _interior(cfg, g.field(f)) for f in ("u", "v", "w", "p", "phi1")}
        out[prec]["drift"] = abs(out[prec]["phi1"].sum() - v0) / v0
        g.close()
    assert H.gpu().felgpu_precision_() == 64  # closing the FP32 run restores FP64
    for f in ("u", "v", "w", "p"):
        a, b = out[64][f], out[32][f]
        err = np.linalg.norm(a - b) / np.linalg.norm(a)
        assert err <= 1e-5, (f, err)
    assert out[32]["drift"] <= 1e-12, out[32]["drift"]
    phi = out[32]["phi1"]
    assert phi.min() >= 0.0 and phi.max() <= 1.0


def _poisson_stats(reset):
    v = [ctypes.c_longlong(0) for _ in range(3)] + [ctypes.c_double(0) for _ in range(2)]
    H.gpu().felgpu_poisson_stats_(ctypes.byref(ctypes.c_int(reset)), *map(ctypes.byref, v))
    return {k: x.value for k, x in zip(("solves", "warm", "refine", "first", "final"), v)}


def _set_refinement(steps, tol):
    H.gpu().felgpu_set_refinement_(ctypes.byref(ctypes.c_int(steps)),
                                   ctypes.byref(ctypes.c_double(tol)))


@pytest.mark.parametrize("fp32_modes,tol,bar", [(True, 1e-7, 2e-7), (True, 1e-10, 1e-9),
                                                (False, None, 1e-12)],
                         ids=["fp32_modes_default", "fp32_modes_1e-10", "fp64_modes"])
def test_fp32_pressure_correction(fp32_modes, tol, bar):
    """The pressure correction solves its Poisson problem to the bar.  In
    the FP32+refine mode the solves from the second on are warm-started
    from the last correction, and each ends at the refinement tolerance of
    the FFT+TDMA operator's relative residual (default 1e-7; 1e-10 set
    through felgpu_set_refinement_); the bar is on the monitor's operator
    (uniform coefficients), which differs from the FFT+TDMA operator's
    residual in the rounding of the wall rows."""
    cfg = C.droplet_impact().scaled(64, 16, 32)
    if tol is not None:
        _set_refinement(3, tol)
    g = GpuRun(cfg, precision=32, fp32_modes=fp32_modes)
    try:
        _poisson_stats(1)
        g.steps(3)
        st = _poisson_stats(1)
        if fp32_modes:
            # the second and third solves start from the last correction (the
            # first from whatever the array holds: zeros in a fresh run, or
            # an earlier run's array at the same address; the residual
            # check makes any starting guess safe)
            assert st["solves"] == 3 and st["warm"] >= 2, st
            assert st["final"] <= tol, st
        else:
            assert st["solves"] == 0, st
        lib = H.gpu()
        fn = lib.felgpu_poisson_residual_
        fn.restype = ctypes.c_double
        div, dp = g.view("div"), g.view("dp")  # registered: resolved to the device copies
        r = fn(ctypes.byref(ctypes.c_int(cfg.ni)), ctypes.byref(ctypes.c_int(cfg.nj)),
               ctypes.byref(ctypes.c_int(cfg.nk)), ctypes.byref(ctypes.c_double(cfg.rhog)),
               ctypes.byref(ctypes.c_double(1 / cfg.dx)), ctypes.byref(ctypes.c_double(1 / cfg.dy)),
               ctypes.byref(ctypes.c_double(1 / cfg.dz)), div.ctypes.data_as(ctypes.c_void_p),
               dp.ctypes.data_as(ctypes.c_void_p))
        assert r <= bar, r
    finally:
        g.close()
        _set_refinement(3, 1e-7)


def test_warm_start_after_the_correction_array_is_gone():
    """The address of the last FP32 solve's correction may since hold a
    flow-class array of the same size: the next solve starts cold instead of
    reading it as FP64."""
    g = H.Grid(16, 8, 16)
    lib = H.gpu()
    lib.felgpu_set_precision_(ctypes.byref(ctypes.c_int(32)))
    reg = []

    def register(a, fp64, upload=1):
        fn = lib.felgpu_register_fp64_ if fp64 else lib.felgpu_register_
        fn(ctypes.c_void_p(a.ctypes.data), ctypes.byref(ctypes.c_int64(a.nbytes)),
           ctypes.byref(ctypes.c_int(upload)))
        reg.append(a)

    def drop(a):
        lib.felgpu_unregister_(ctypes.c_void_p(a.ctypes.data))
        reg[:] = [x for x in reg if x is not a]

    try:
        r = np.random.default_rng(55)
        div, div2, old, new = (g.zeros() for _ in range(4))
        g.interior(div)[...] = r.standard_normal((g.nk, g.nj, g.ni))
        g.interior(div)[...] -= g.interior(div).mean()
        div2[...] = div
        modes = [np.zeros(g.ni * g.nj * g.nk) for _ in range(2)]
        head = [I(g.ni), I(g.nj), I(g.nk)]
        pc = [np.zeros(g.nj + 6) for _ in range(7)]
        fft = [np.zeros(g.nj + 6) for _ in range(3)]
        H.call_gpu("cal_coef_prs", I(g.nj), D(1.0), D(1.0), D(1.0), D(1.0), *pc)
        H.call_gpu("cal_coef_solp_fft", I(g.nj), pc[2], pc[3], *fft)
        sv = np.array([g.ni, g.nj, g.nk], dtype=np.int32)
        wk = [np.zeros(64) for _ in range(3)]

        def solve(rhs, dp):
            H.call_gpu("solp_fft_tdma1", *head, wk[0], rhs, *modes)
            H.call_gpu("solp_fft_tdma2", I(0), I(1), sv, D(1.0), D(1.0), D(1.0), *fft, *wk, *modes)
            H.call_gpu("solp_fft_tdma3", *head, wk[0], *modes, dp)
            lib.felgpu_download_(ctypes.c_void_p(dp.ctypes.data))
            return g.interior(dp).copy()

        for a in (div, old):
            register(a, True)
        for a in modes:
            register(a, False, 0)
        first = solve(div, old)
        drop(old)
        old[...] = r.standard_normal(g.shape)
        register(old, False)  # the same address, now a flow-class array
        register(div2, True)
        register(new, True)
        second = solve(div2, new)
        assert np.linalg.norm(first - second) <= 1e-5 * np.linalg.norm(first)
    finally:
        for a in list(reg):
            drop(a)
        lib.felgpu_set_precision_(ctypes.byref(ctypes.c_int(64)))


class Poisson32:
    """FP32 pressure solves on registered arrays of one small grid."""

    def __init__(self):
        self.g, self.lib, self.reg = H.Grid(16, 8, 16), H.gpu(), []
        g = self.g
        self.modes = [np.zeros(g.ni * g.nj * g.nk) for _ in range(2)]
        self.div, self.dp = g.zeros(), g.zeros()
        r = np.random.default_rng(57)
        g.interior(self.div)[...] = r.standard_normal((g.nk, g.nj, g.ni))
        g.interior(self.div)[...] -= g.interior(self.div).mean()
        pc = [np.zeros(g.nj + 6) for _ in range(7)]
        self.fft = [np.zeros(g.nj + 6) for _ in range(3)]
        H.call_gpu("cal_coef_prs", I(g.nj), D(1.0), D(1.0), D(1.0), D(1.0), *pc)
        H.call_gpu("cal_coef_solp_fft", I(g.nj), pc[2], pc[3], *self.fft)

    def __enter__(self):
        self.lib.felgpu_set_precision_(ctypes.byref(ctypes.c_int(32)))
        for a in (self.div, self.dp):
            self.register(a, self.lib.felgpu_register_fp64_)
        for a in self.modes:
            self.register(a, self.lib.felgpu_register_)
        return self

    def register(self, a, fn):
        fn(ctypes.c_void_p(a.ctypes.data), ctypes.byref(ctypes.c_int64(a.nbytes)),
           ctypes.byref(ctypes.c_int(1)))
        self.reg.append(a)

    def drop(self, a):
        self.lib.felgpu_unregister_(ctypes.c_void_p(a.ctypes.data))
        self.reg = [x for x in self.reg if x is not a]

    def solve(self):
        g = self.g
        head, wk = [I(g.ni), I(g.nj), I(g.nk)], [np.zeros(64) for _ in range(3)]
        sv = np.array([g.ni, g.nj, g.nk], dtype=np.int32)
        H.call_gpu("solp_fft_tdma1", *head, wk[0], self.div, *self.modes)
        H.call_gpu("solp_fft_tdma2", I(0), I(1), sv, D(1.0), D(1.0), D(1.0), *self.fft, *wk,
                   *self.modes)
        H.call_gpu("solp_fft_tdma3", *head, wk[0], *self.modes, self.dp)
        self.lib.felgpu_download_(ctypes.c_void_p(self.dp.ctypes.data))
        return g.interior(self.dp).copy()

    def __exit__(self, *exc):
        for a in list(self.reg):
            self.drop(a)
        self.lib.felgpu_set_precision_(ctypes.byref(ctypes.c_int(64)))


@pytest.mark.parametrize("given_back", [True, False], ids=["given back", "registered again"])
def test_no_warm_start_from_another_registration(given_back):
    """The last correction's address may since hold another FP64 array, or have
    been registered again: the next solve does not start from what it holds
    (NaN here)."""
    with Poisson32() as p:
        first = p.solve()
        if given_back:
            p.drop(p.dp)
        p.dp[...] = np.nan
        p.register(p.dp, p.lib.felgpu_register_fp64_)
        second = p.solve()
    assert np.linalg.norm(first - second) <= 1e-5 * np.linalg.norm(first)


@pytest.mark.parametrize("value", [np.nan, -np.inf, 1e30])
def test_no_warm_start_from_a_useless_guess(value):
    """A correction array that was overwritten since the last solve, with values
    that no refinement brings back, does not spoil the next solve; a right-hand
    side with a NaN still gives NaN."""
    with Poisson32() as p:
        first = p.solve()
        p.dp[5, 6, 7] = value
        p.lib.felgpu_upload_(ctypes.c_void_p(p.dp.ctypes.data))
        second = p.solve()
        p.div[5, 6, 7] = np.nan
        p.lib.felgpu_upload_(ctypes.c_void_p(p.div.ctypes.data))
        third = p.solve()
    assert np.linalg.norm(first - second) <= 1e-5 * np.linalg.norm(first)
    assert np.isnan(third).all()


def test_fp32_precision_is_per_array_class():
    """Flow arrays registered with felgpu_register_ are FP32, arrays
    registered with felgpu_register_fp64_ stay FP64; a kernel asked to read
    the wrong class is refused before anything runs (checked on the host)."""
    g = H.Grid(16, 8, 16)
    lib = H.gpu()
    lib.felgpu_set_precision_(ctypes.byref(ctypes.c_int(32)))
    arrays = []
    try:
        rng = np.random.default_rng(50)
        phi = rng.random(g.shape)
        rho = g.zeros()
        for a, fp64 in ((phi, True), (rho, False)):
            n = ctypes.c_int64(a.nbytes)
            up = ctypes.c_int(1)
            reg = lib.felgpu_register_fp64_ if fp64 else lib.felgpu_register_
            reg(ctypes.c_void_p(a.ctypes.data), ctypes.byref(n), ctypes.byref(up))
            arrays.append(a)
        H.call_gpu("cal_arith_mean", I(g.ni), I(g.nj), I(g.nk), phi, D(0.81), D(1e-3), rho)
        lib.felgpu_download_(ctypes.c_void_p(rho.ctypes.data))
        want = (0.81 * (1.0 - phi) + 1e-3 * phi).astype(np.float32).astype(np.float64)
        assert np.array_equal(rho, want)
    finally:
        for a in arrays:
            lib.felgpu_unregister_(ctypes.c_void_p(a.ctypes.data))
        lib.felgpu_set_precision_(ctypes.byref(ctypes.c_int(64)))


def test_fp32_weno_with_subnormal_differences():
    """FP32 WENO5 on a u field whose differences are subnormal floats (the
    largest below 2.9e-39, where 1/x overflows), advected by v = w = 1:
    every output is finite and adv_u is not all zero."""
    g = H.Grid(16, 8, 16, 1.0, 1.0, 1.0)
    lib = H.gpu()
    lib.felgpu_set_precision_(ctypes.byref(ctypes.c_int(32)))
    arrays = []
    try:
        rng = np.random.default_rng(53)
        u = (np.float32(1e-39) * rng.uniform(-1, 1, g.shape).astype(np.float32)).astype(np.float64)
        assert 0 < np.abs(np.diff(u, axis=2)).max() < 2.9e-39
        vel = [u, np.ones(g.shape), np.ones(g.shape)]
        adv = [g.zeros() for _ in range(3)]
        for a in vel + adv:
            n = ctypes.c_int64(a.nbytes)
            lib.felgpu_register_(ctypes.c_void_p(a.ctypes.data), ctypes.byref(n),
                                 ctypes.byref(ctypes.c_int(1)))
            arrays.append(a)
        H.call_gpu("cal_advu_weno5", I(g.ni), I(g.nj), I(g.nk), D(1.0), D(1.0), D(1.0), *vel, *adv)
        for a in adv:
            lib.felgpu_download_(ctypes.c_void_p(a.ctypes.data))
            assert np.isfinite(a).all()
        assert np.abs(g.interior(adv[0])).max() > 0
    finally:
        for a in arrays:
            lib.felgpu_unregister_(ctypes.c_void_p(a.ctypes.data))
        lib.felgpu_set_precision_(ctypes.byref(ctypes.c_int(64)))


def test_poisson_residual_equals_the_oracle():
    """felgpu_poisson_residual_ (the FP64 residual operator of the
    refinement, srcs/solp_fft_tdma4.f:55-72) against orc_poisson_residual on
    the same seeded div and dp: relative residual and its absolute form."""
    g = H.Grid(32, 16, 32, 1 / 32, 1 / 16, 1 / 32)
    r = np.random.default_rng(54)
    div, dp = r.standard_normal(g.shape), r.standard_normal(g.shape)
    lib, orc = H.gpu(), H.oracle()
    fn = lib.felgpu_poisson_residual_
    fn.restype = ctypes.c_double
    got = fn(ctypes.byref(ctypes.c_int(g.ni)), ctypes.byref(ctypes.c_int(g.nj)),
             ctypes.byref(ctypes.c_int(g.nk)), ctypes.byref(ctypes.c_double(0.81)),
             ctypes.byref(ctypes.c_double(1 / g.dx)), ctypes.byref(ctypes.c_double(1 / g.dy)),
             ctypes.byref(ctypes.c_double(1 / g.dz)), div.ctypes.data_as(ctypes.c_void_p),
             dp.ctypes.data_as(ctypes.c_void_p))
    orc.orc_poisson_residual.restype = ctypes.c_double
    orc.orc_poisson_residual.argtypes = [ctypes.c_int] * 3 + [ctypes.c_double] * 4 + \
        [ctypes.c_void_p] * 3
    eabs = ctypes.c_double(0.0)
    want = orc.orc_poisson_residual(g.ni, g.nj, g.nk, 0.81, 1 / g.dx, 1 / g.dy, 1 / g.dz,
                                    div.ctypes.data, dp.ctypes.data, ctypes.addressof(eabs))
    assert abs(got / want - 1.0) <= 1e-13, (got, want)
