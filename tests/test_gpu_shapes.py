"""The launch shapes that depend on the grid: chunk lengths of the marching
kernels, tile edges and remainders, each against the oracle on the sizes where
a shape changes."""
import contextlib

import numpy as np
import pytest

import adjoint_cases as A
import felharness as H
from felharness import D, I, Grid
from test_gpu_kernels import check, grad, run_both

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def mode(which):
    """The library in another of its modes: "fp32" or "tangent"."""
    lib, c = H.gpu(), H.ctypes
    fn, on, off = {"fp32": (lib.felgpu_set_precision_, 32, 64),
                   "tangent": (lib.felgpu_set_tangent_, 1, 0)}[which]
    fn(c.byref(c.c_int(on)))
    try:
        yield
    finally:
        fn(c.byref(c.c_int(off)))


def float32(a):
    """Values that the FP32 mode holds as they are."""
    return a.astype(np.float32).astype(np.float64)


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


# f(-3..2) of a stencil whose weight sum has a significand of all ones, the one
# that a residual correction of an approximate reciprocal may leave a unit in the
# last place low, depending on where it starts (in each the derivative's last
# place depends on it)
ALL_ONES = [
    "0x1.5ac933da37283p-2 0x1.9c3cd63e28b70p-1 0x1.4b960e74a5b97p-2 -0x1.46ec1717aa384p+0 "
    "0x1.c64089d23ece5p-1 0x1.bfed443a534cep-2",
    "-0x1.e0d0c00daaa40p-1 0x1.a5e2ededb21eep-8 -0x1.1c496df700f17p+0 -0x1.1473ce69d79eep+0 "
    "0x1.708b7879a8d94p+0 -0x1.ae807168d09b5p-5",
    "-0x1.38543e84c0de1p-1 0x1.cafdb732b9abbp+0 -0x1.db1dde593df6ep-1 -0x1.6de1ffbe532ecp-2 "
    "0x1.af8e923357f13p-1 -0x1.eb88eec79bd85p-3",
    "-0x1.24246dde22f0bp+0 0x1.db3439dc6af07p+0 -0x1.7a3ac98873e55p-1 -0x1.63d200ecd1183p-2 "
    "0x1.f1578407ff970p-1 0x1.ff18f61497003p-1",
]


@pytest.mark.parametrize("stencil", ALL_ONES, ids=range(4))
@pytest.mark.parametrize("down", [False, True])
def test_weno_weight_sums_of_all_ones(stencil, down):
    """WENO5 at such a weight sum: bit for bit the oracle's."""
    g = Grid(16, 4, 4, 1.0, 1.0, 1.0)
    f = np.zeros(g.ni)
    f[4:10] = [float.fromhex(x) for x in stencil.split()]
    if down:  # the mirrored stencil, carried the other way
        f = -f[::-1]
    u, v = np.full(g.shape, -1.0 if down else 1.0), g.zeros()
    v[:, :, 3:g.ni + 3] = f  # constant in y, where it carries itself

    def args():
        return [I(g.ni), I(g.nj), I(g.nk), D(1.0), D(1.0), D(1.0), u.copy(), v.copy(), g.zeros(),
                g.zeros(), g.zeros(), g.zeros()]
    want, got = run_both("cal_advu_weno5", args)
    assert np.any(want[-2])
    for a, b in zip(want[-3:], got[-3:]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("down", [False, True])
def test_weno_fp32_jump_beside_the_stencil(down):
    """WENO5 in FP32 on cells whose upwind stencil ends before a jump of 2^20:
    the weights are those of the values the stencil holds.  Small whole numbers
    up to the jump, so the differences and indicators are exact; the bar is 16
    roundings of the largest term |u|/6 (2 + 7 + 11) |d| of a derivative, |d| <= 6
    the differences in a stencil."""
    g = Grid(32, 4, 4, 1.0, 1.0, 1.0)
    r = np.random.default_rng(20)
    u = g.zeros()
    u[...] = 8.0 + r.integers(-3, 4, g.ni + 6)
    u[:, :, 20] = 2.0 ** 20
    sign = -1.0 if down else 1.0
    u = sign * (u[:, :, ::-1].copy() if down else u)

    def args():
        return [I(g.ni), I(g.nj), I(g.nk), D(1.0), D(1.0), D(1.0), u.copy(), g.zeros(), g.zeros(),
                g.zeros(), g.zeros(), g.zeros()]
    with mode("fp32"):
        want, got = run_both("cal_advu_weno5", args)
    clear = slice(3, 18)  # up to the cell that only misses the jump with f(2)
    if down:
        clear = slice(g.ni + 6 - 18, g.ni + 6 - 3)
    a, b = (g.interior(x[-3])[..., clear.start - 3:clear.stop - 3] for x in (want, got))
    assert np.min(np.max(np.abs(a), axis=(0, 1))) > 0.0
    assert np.max(np.abs(a - b)) <= 16 * 2.0 ** -24 * 11.0 / 6.0 * 20.0 * 6.0


def test_weno_fp32_non_finite_values():
    """WENO5 in FP32 at infinities and NaN in a still flow: the cells that the
    oracle leaves finite are the library's."""
    g = Grid(66, 5, 18, 1 / 16, 1 / 12, 1 / 20)
    r = np.random.default_rng(66)
    u = np.where(r.random(g.shape) < 0.03, r.choice([np.inf, -np.inf, np.nan], g.shape), 0.0)
    with mode("fp32"):
        want, got = run_both("cal_advu_weno5", lambda: [
            I(g.ni), I(g.nj), I(g.nk), D(16.0), D(12.0), D(20.0), u.copy()] + [
                g.zeros() for _ in range(5)])
    quiet = np.isfinite(u) & np.isfinite(np.roll(u, 1, 2)) & np.isfinite(np.roll(u, -1, 2))
    assert np.isnan(want[-3][quiet]).any()
    assert np.array_equal(want[-3][quiet], got[-3][quiet], equal_nan=True)


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


@pytest.mark.parametrize("ni,nj,nk", [(4, 4, 4), (5, 5, 5), (33, 8, 10), (130, 9, 6)])
@pytest.mark.parametrize("which", ["fp32", "tangent"])
def test_streamed_differences_in_the_other_modes(ni, nj, nk, which):
    """The same kernels with four elements a run and with one: bit for bit the
    oracle's in the tangent mode, in FP32 within the rounding of a scale, two
    operations and the store, relative to each element."""
    g = Grid(ni, nj, nk, 1 / 16, 1 / 12, 1 / 20)
    r = np.random.default_rng(ni * nj + nk)
    f = [float32(r.standard_normal(g.shape)) for _ in range(10)]
    rk = float32(r.standard_normal((3,) + g.shape))
    dy = r.uniform(8.0, 16.0, nj + 6)
    scales = [D(16.0), D(12.0), D(20.0)]
    with mode(which):
        both = [run_both("cal_grad_p2uvw", lambda: [I(0), I(nj), I(ni), I(nj), I(nk), scales[0],
                                                    dy.copy(), scales[2]] +
                         [x.copy() for x in f[:4]]),
                run_both("cal_grad_prs", lambda: [I(ni), I(nj), I(nk)] + scales +
                         [x.copy() for x in f[:4]]),
                run_both("calfst", lambda: [I(ni), I(nj), I(nk), D(0.81), D(8.1e-4), D(5.5)] +
                         [x.copy() for x in f[4:7]] + [rk.copy()] + [x.copy() for x in f[7:10]])]
    eps = 4 * 2.0 ** -24 if which == "fp32" else 0.0
    for want, got in both:
        for a, b in zip(want, got):
            if isinstance(a, np.ndarray):
                assert np.all(np.abs(a - b) <= eps * np.abs(a))


@pytest.mark.parametrize("ni,nj,nk", [(4, 4, 4), (66, 7, 18), (130, 9, 6), (33, 8, 10), (8, 5, 9)])
@pytest.mark.parametrize("which", ["fp32", "tangent"])
@pytest.mark.parametrize("resident", [False, True], ids=["coefficients", "viscosity"])
def test_viscous_solve_with_any_ghosts_in_the_other_modes(ni, nj, nk, which, resident):
    """As test_viscous_solve_with_any_ghosts, interior values: bit for bit the
    oracle's in the tangent mode; in FP32 within 16 roundings a sweep of the
    largest velocity, 21 sweeps at most (a source read from the wrong ghost is off
    by the size of the velocities)."""
    g = Grid(ni, nj, nk, 1 / 16, 1 / 12, 1 / 20)
    r = np.random.default_rng(ni * nj + nk)
    head = [I(ni), I(nj), I(nk)]
    rmu, rho, rhon = (float32(r.uniform(0.5, 1.0, g.shape)) for _ in range(3))
    phi, l1, l2 = (r.uniform(0.05, 1.0, g.shape) for _ in range(3))
    src, start = ([float32(r.standard_normal(g.shape)) for _ in range(3)] for _ in range(2))

    def solve(call, coef, uvw):
        call("cal_arith_coef_vis", *head, D(1 / g.dx), D(1 / g.dy), D(1 / g.dz), rmu, *coef)
        call("solu_sor4", I(0), I(0), np.full(6, -1, np.int32), I(1), *head,
             np.zeros(8, np.int32), np.zeros(8), np.zeros(8), I(1), I(0), D(0.001), rho, rhon,
             *coef, *src, *uvw, D(0.25), D(g.dy), l1, l2, phi)

    want, got = [x.copy() for x in start], [x.copy() for x in start]
    solve(H.call_oracle, [g.zeros() for _ in range(45)], want)
    coef = [g.zeros() for _ in range(45)]
    with mode(which):
        if resident:
            lib = H.gpu()
            flow, phase = [rmu, rho, rhon, *src, *coef, *got], [phi, l1, l2]
            try:
                for a in flow + phase:
                    fn = lib.felgpu_register_ if any(a is x for x in flow) else lib.felgpu_register_fp64_
                    fn(H.ctypes.c_void_p(a.ctypes.data), H.ctypes.byref(H.ctypes.c_int64(a.nbytes)),
                       H.ctypes.byref(H.ctypes.c_int(1)))
                solve(H.call_gpu, coef, got)
                for a in got:
                    lib.felgpu_download_(H.ctypes.c_void_p(a.ctypes.data))
            finally:
                for a in flow + phase:
                    lib.felgpu_unregister_(H.ctypes.c_void_p(a.ctypes.data))
        else:
            solve(H.call_gpu, coef, got)
    for a, b in zip(want, got):
        if which == "tangent":
            assert np.array_equal(a, b)
        else:
            a, b = g.interior(a), g.interior(b)
            assert np.max(np.abs(a - b)) <= 21 * 16 * 2.0 ** -24 * np.max(np.abs(a))
