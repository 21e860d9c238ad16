"""The launch shapes that depend on the grid: chunk lengths of the marching
kernels, tile edges and remainders, each against the oracle on the sizes where
a shape changes."""
import numpy as np
import pytest

import adjoint_cases as A
import felharness as H
from felharness import D, I, Grid
from test_gpu_kernels import check, grad, run_both

pytestmark = pytest.mark.gpu


# (64 x 4 blocks; one plane per thread up to 8: 4^3 and the odd grids march one
# plane, 130 x 40 x 40 two, 200 x 100 x 70 eight)
@pytest.mark.parametrize("ni,nj,nk", [(4, 4, 4), (63, 5, 9), (66, 7, 18), (130, 40, 40),
                                      (200, 100, 70)])
@pytest.mark.parametrize("flat", [False, True], ids=["interface", "flat"])
def test_mthinc_flux_and_truncation_shapes(ni, nj, nk, flat):
    """solphi_mthinc1 with and without interface cells, and the truncation
    pass of solphi_mthinc3.  Bars: the fluxes' Gauss sums differ from the
    oracle's by the rounding of an 8-term sum and of the device's exp (1e-13
    of the largest flux); phin by the mass offset's sum order."""
    g = Grid(ni, nj, nk, 1 / 16, 1 / 16, 1 / 16)
    r = np.random.default_rng(ni + nj + nk)
    phi = np.full(g.shape, 0.75) if flat else H.smooth_phi(g, r)
    gx, gy, gz = grad(g, phi)
    u, v, w = (H.random_vel(g, r, 0.5) for _ in range(3))
    u[3, 3, 3] = v[4, 4, 4] = w[5, 5, 5] = 0.0
    head = [I(g.ni), I(g.nj), I(g.nk), D(1 / g.dx), D(1 / g.dy), D(1 / g.dz)]
    old = [r.standard_normal(g.shape) for _ in range(3)]

    def flux():
        return head + [D(0.01), D(1.0), phi.copy(), gx.copy(), gy.copy(), gz.copy(), u.copy(),
                       v.copy(), w.copy()] + [x.copy() for x in old]
    check(*run_both("solphi_mthinc1", flux), rtol=1e-13)
    phin = np.clip(phi + 0.01 * r.standard_normal(g.shape), -0.05, 1.05)

    def trunc():
        return [I(0)] + head + [D(1.0), gx.copy(), gy.copy(), gz.copy(), phi.copy(), phin.copy()]
    a, b = run_both("solphi_mthinc3", trunc)
    # the offset's two sums of n terms are taken in another order: each is off
    # by at most n eps times itself; phin moves by offset p^2 (1-p) <= 4/27 offset
    p = np.clip(g.interior(phin), 0.0, 1.0)
    bar = 4 / 27 * 2 * p.size * 1.2e-16 * p.sum() / (p * p * (1 - p)).sum() + 1e-15
    assert np.max(np.abs(a[-1] - b[-1])) <= bar


class Resident:
    """Arrays registered with the library for one test."""

    def __init__(self, *arrays):
        self.lib, self.arrays = H.gpu(), arrays

    def __enter__(self):
        for a in self.arrays:
            self.lib.felgpu_register_(H.ctypes.c_void_p(a.ctypes.data),
                                      H.ctypes.byref(H.ctypes.c_int64(a.nbytes)),
                                      H.ctypes.byref(H.ctypes.c_int(1)))
        return self

    def fetch(self):
        for a in self.arrays:
            self.lib.felgpu_download_(H.ctypes.c_void_p(a.ctypes.data))

    def __exit__(self, *exc):
        for a in self.arrays:
            self.lib.felgpu_unregister_(H.ctypes.c_void_p(a.ctypes.data))


# sizes at which the marching kernels take 1, 2, 4 and (the normals) 16 planes
MARCH = [(4, 4, 4), (61, 7, 13), (130, 40, 40), (70, 50, 160), (260, 124, 130)]


@pytest.mark.parametrize("ni,nj,nk", MARCH)
def test_marching_stencils_shapes(ni, nj, nk):
    """Normals on four staggerings with their curvature, WENO5, and stress with
    its divergence on resident arrays: bit for bit the oracle's."""
    g = Grid(ni, nj, nk, 1 / 16, 1 / 12, 1 / 20)
    r = np.random.default_rng(ni * nj + nk)
    head = [I(ni), I(nj), I(nk), D(1 / g.dx), D(1 / g.dy), D(1 / g.dz)]
    grads = [r.standard_normal(g.shape) for _ in range(3)]
    rn, kap = [g.zeros(3) for _ in range(4)], g.zeros(3)
    vel, mu = [r.standard_normal(g.shape) for _ in range(3)], r.uniform(0.1, 1.0, g.shape)
    adv, vis = [g.zeros() for _ in range(3)], [g.zeros() for _ in range(3)]
    s, tau = g.zeros(6), g.zeros(6)
    outs = rn + [kap] + adv + [s, tau] + vis

    def calls(call):
        for st, o in zip(((1, 1, 1), (0, 0, 1), (0, 1, 0), (1, 0, 0)), rn):
            call("calrn", *head, *[I(v) for v in st], *grads, o)
        call("calrkap", *head, *rn, kap)
        call("cal_advu_weno5", *head, *vel, *adv)
        call("calsij", *head, *vel, s)
        call("cal_arith_tau", *head[:3], s, mu, tau)
        call("cal_div_tensor", *head, tau, *vis)

    calls(H.call_oracle)
    want = [o.copy() for o in outs]
    for o in outs:
        o[...] = 0.0
    with Resident(*grads, *vel, mu, *outs) as res:
        calls(H.call_gpu)
        res.fetch()
    for a, b in zip(want, outs):
        assert np.array_equal(a, b)


# even x and z (ghost images in the launches: the smallest grid, one and several
# blocks a row) and an odd size of each (refresh launches); partial sums of the
# stop test for one launch and for two
@pytest.mark.parametrize("ni,nj,nk", [(4, 4, 4), (66, 7, 18), (130, 9, 6), (33, 8, 10), (8, 5, 9),
                                      (8, 8, 340), (8, 8, 1400)])
@pytest.mark.parametrize("resident", [False, True], ids=["coefficients", "viscosity"])
def test_viscous_solve_with_any_ghosts(ni, nj, nk, resident):
    """solu_sor4 from ghosts that are no periodic images: the values that its
    pairs read through bndu's shifted sources are the ones the refreshes of the
    oracle leave, bit for bit, whether the coefficients are arrays or formed
    from the viscosity."""
    g = Grid(ni, nj, nk, 1 / 16, 1 / 12, 1 / 20)
    r = np.random.default_rng(ni * nj + nk)
    head = [I(ni), I(nj), I(nk)]
    rmu, rho, rhon, phi, l1, l2 = (r.uniform(0.05, 1.0, g.shape) for _ in range(6))
    src = [r.standard_normal(g.shape) for _ in range(3)]
    start = [r.standard_normal(g.shape) for _ in range(3)]

    def solve(call, coef, uvw):
        call("cal_arith_coef_vis", *head, D(1 / g.dx), D(1 / g.dy), D(1 / g.dz), rmu, *coef)
        call("solu_sor4", I(0), I(0), np.full(6, -1, np.int32), I(1), *head,
             np.zeros(8, np.int32), np.zeros(8), np.zeros(8), I(1), I(0), D(0.01), rho, rhon,
             *coef, *src, *uvw, D(0.25), D(g.dy), l1, l2, phi)

    want, got = [x.copy() for x in start], [x.copy() for x in start]
    solve(H.call_oracle, [g.zeros() for _ in range(45)], want)
    coef = [g.zeros() for _ in range(45)]
    if resident:
        with Resident(rmu, rho, rhon, phi, l1, l2, *src, *coef, *got) as res:
            solve(H.call_gpu, coef, got)
            for a in got:
                res.lib.felgpu_download_(H.ctypes.c_void_p(a.ctypes.data))
    else:
        solve(H.call_gpu, coef, got)
    for a, b in zip(want, got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("ni,nj,nk", [(5, 4, 4), (66, 5, 18)])
def test_weno_zero_and_non_finite_values(ni, nj, nk):
    """WENO5 where the transport velocity is zero (both sides count), where a
    weight sum leaves the range of the short reciprocal, and at infinities and
    NaN: bit for bit the oracle's."""
    g = Grid(ni, nj, nk, 1 / 16, 1 / 12, 1 / 20)
    r = np.random.default_rng(ni)
    head = [I(ni), I(nj), I(nk), D(1 / g.dx), D(1 / g.dy), D(1 / g.dz)]
    plain = [r.standard_normal(g.shape) for _ in range(3)]
    still = [np.where(r.random(g.shape) < 0.9, 0.0, x) for x in plain]
    large = [5.0e36 * x for x in plain]

    def both(vel):
        a, b = run_both("cal_advu_weno5",
                        lambda: head + [x.copy() for x in vel] + [g.zeros() for _ in range(3)])
        return a[-3:], b[-3:]
    for vel in (plain, [0.0 * x for x in plain], still, large):
        for x, y in zip(*both(vel)):
            # the library does not form the side that a zero multiplies, whose
            # overflow is the oracle's NaN
            assert np.all((x == y) | np.isnan(x))
    assert not np.isnan(both(still)[0][0]).any()
    u = np.where(r.random(g.shape) < 0.03, r.choice([np.inf, -np.inf, np.nan], g.shape), 0.0)
    want, got = both([u, g.zeros(), g.zeros()])
    quiet = np.isfinite(u) & np.isfinite(np.roll(u, 1, 0)) & np.isfinite(np.roll(u, -1, 0))
    assert np.isnan(want[0][quiet]).any()
    assert np.array_equal(want[0][quiet], got[0][quiet], equal_nan=True)


@pytest.mark.parametrize("flip", [False, True])
def test_weno_zero_velocity_beside_an_overflowing_side(flip):
    """WENO5 across a still direction where one side's weights overflow and the
    other's, whose smoothness indicators vanish, do not: both sides count, and the
    oracle's NaN is the library's."""
    g = Grid(5, 16, 4, 1.0, 1.0, 1.0)
    ramp = -2.0 ** 330 * np.maximum(0.0, 10.0 - np.arange(g.nj + 6))  # slope, then flat
    u = np.empty(g.shape)
    u[...] = (ramp[::-1] if flip else ramp)[None, :, None]

    def args():
        return [I(g.ni), I(g.nj), I(g.nk), D(1.0), D(1.0), D(1.0), u.copy(), g.zeros(),
                np.ones(g.shape), g.zeros(), g.zeros(), g.zeros()]
    want, got = run_both("cal_advu_weno5", args)
    assert np.isnan(want[-3]).any() and (g.interior(want[-3]) == 0.0).any()
    for a, b in zip(want[-3:], got[-3:]):
        assert np.array_equal(a, b, equal_nan=True)


# rows of odd and even length, the image's end inside a 16-byte run (0 to 3
# elements over), less than one block
@pytest.mark.parametrize("ni,nj,nk", [(4, 4, 4), (5, 5, 5), (7, 5, 4), (33, 8, 10), (130, 9, 6)])
def test_viscous_coefficients_on_the_image(ni, nj, nk):
    """The 45 coefficient arrays over the whole padded image, in FP64 bit for
    bit the oracle's, in FP32 within the rounding of their 4-point means and
    products (fewer than 16 operations of 2^-24 each)."""
    g = Grid(ni, nj, nk, 1 / 16, 1 / 12, 1 / 20)
    mu = np.random.default_rng(ni * nj * nk).uniform(0.1, 1.0, g.shape)
    args = [I(ni), I(nj), I(nk), D(16.0), D(12.0), D(20.0)]
    want, got = ([np.full(g.shape, 7.0) for _ in range(45)] for _ in range(2))
    H.call_oracle("cal_arith_coef_vis", *args, mu, *want)
    H.call_gpu("cal_arith_coef_vis", *args, mu, *got)
    for a, b in zip(want, got):
        assert np.array_equal(a, b)
    low = [np.full(g.shape, 7.0) for _ in range(45)]
    H.gpu().felgpu_set_precision_(H.ctypes.byref(H.ctypes.c_int(32)))
    try:
        H.call_gpu("cal_arith_coef_vis", *args, mu, *low)
    finally:
        H.gpu().felgpu_set_precision_(H.ctypes.byref(H.ctypes.c_int(64)))
    for a, b in zip(want, low):
        assert np.max(np.abs(a - b)) <= 16 * 2.0 ** -24 * np.max(np.abs(a))


# lines of 4 and 5 cells (ends that share elements) and of 6 and 7 (the first
# whose two ends are folded in registers) in x and z, the shortest columns in y
@pytest.mark.parametrize("ni,nj,nk", [(4, 4, 4), (5, 4, 6), (6, 5, 5), (7, 6, 4), (6, 4, 7)])
@pytest.mark.parametrize("case", ["bndu", "bndu_bp", "bnd_periodic"])
def test_ghost_adjoints_on_short_lines(ni, nj, nk, case):
    """The transposed ghost fills and wall rows equal the oracle's, to the
    rounding of the slip coefficients' adjoints."""
    g = Grid(ni, nj, nk, 1 / 16, 1 / 12, 1 / 20)
    c = {"bndu": A.Bndu, "bndu_bp": A.BnduP, "bnd_periodic": A.Periodic}[case](g, ni + 7 * nk)
    x, y = c.inputs(), c.out_adjoints()
    want = c.adjoint(H.call_oracle, {k: v.copy() for k, v in y.items()})
    got = c.adjoint(H.call_gpu, {k: v.copy() for k, v in y.items()})
    for k in x:
        assert np.max(np.abs(want[k] - got[k])) <= 1e-13 * max(1.0, np.max(np.abs(want[k])))


# rows of even and odd length, the image's last run whole or cut
@pytest.mark.parametrize("ni,nj,nk", [(4, 4, 4), (5, 5, 5), (7, 4, 6), (33, 8, 10), (130, 9, 6)])
def test_streamed_differences_shapes(ni, nj, nk):
    """Face gradients (one 1/dy and one per row) and the surface force by 16-byte
    runs: bit for bit the oracle's, with the elements they leave untouched."""
    g = Grid(ni, nj, nk, 1 / 16, 1 / 12, 1 / 20)
    r = np.random.default_rng(ni + nj + nk)
    f = [r.standard_normal(g.shape) for _ in range(10)]
    rk = r.standard_normal((3,) + g.shape)
    scales = [D(16.0), D(12.0), D(20.0)]
    for dy in (np.full(nj + 6, 12.0), r.uniform(8.0, 16.0, nj + 6)):
        check(*run_both("cal_grad_p2uvw", lambda: [
            I(0), I(nj), I(ni), I(nj), I(nk), scales[0], dy, scales[2]] + [x.copy() for x in f[:4]]))
    check(*run_both("cal_grad_prs", lambda: [I(ni), I(nj), I(nk)] + scales +
                    [x.copy() for x in f[:4]]))
    check(*run_both("calfst", lambda: [I(ni), I(nj), I(nk), D(0.81), D(8.1e-4), D(5.5)] +
                    [x.copy() for x in f[4:7]] + [rk.copy()] + [x.copy() for x in f[7:10]]))
