"""The deposition's evaluation forms -- rows of merged Gauss-Legendre nodes,
wide kernels on every fourth column with interpolation between, launches whose
points are split into slices -- against the FP64 oracle, at the sizes where
their dispatch changes."""
from types import SimpleNamespace

import numpy as np
import pytest

from helpers import max_norm_err, oracle_range
from test_host_prep_and_emulation import _emu

# FP32 evaluation: coordinates up to 8 standard deviations carry a rounding of
# 2^-24 each, so a kernel value at the 1e-3 level of its peak (|a| ~ 3.7) is off
# by 2 a |a| 2^-24 ~ 1.6e-6 of itself at most, its peak region by far less; the
# merged and interpolated forms add 5e-8 of the peak.  (Kernels much narrower
# than a bin are left out: what reaches the next bins is a difference of erf
# values close to 1.)
TOL = 2e-6


def _points(n, ex, ey, seed, hi=4.0):
    """Kernel points all over (and around) the grid, widths log-uniform over
    every form: erf differences to kernels wider than the grid."""
    rng = np.random.default_rng(seed)
    x = rng.uniform(ex.first - 0.2, ex.last + 0.2, n)
    y = rng.uniform(ey.first - 0.2, ey.last + 0.2, n)
    sx = np.exp(rng.uniform(np.log(0.3 * ex.step), np.log(hi), n))
    sy = sx * np.exp(rng.uniform(-0.7, 0.7, n))
    return x, y, sx, sy, rng.uniform(0.1, 1.0, n)


@pytest.mark.parametrize("cov_mult", [1, -1, 0])
@pytest.mark.parametrize("nx,ny", [(200, 300), (75, 100), (28, 40)])
def test_single_kernels_of_every_width(sfh, emu, O, nx, ny, cov_mult):
    """One kernel at a time, widths in small steps across every change of form."""
    ex, ey = sfh.edges_range(-0.5, 2.5, nx + 1), sfh.edges_range(18.0, 30.0, ny + 1)
    ox, oy = oracle_range(O, ex), oracle_range(O, ey)
    worst = 0.0
    for k, s in enumerate(np.geomspace(0.3 * ex.step, 3.0, 60)):
        p = [np.array([v]) for v in (1.0 + 0.013 * k, 24.1 + 0.017 * k, s, s * (0.6 + 0.02 * (k % 40)), 1.0)]
        ref, pr = O.bin_cmd_smooth(*p[:4], cov_mult, p[4], ox, oy)
        mat, pe = _emu(emu, O, *p, cov_mult, ox, oy)
        assert pe == pr
        worst = max(worst, max_norm_err(mat, ref))
    assert worst <= TOL, worst


@pytest.mark.parametrize("kind,bound", [("asym", 2.2e-6), ("cov", 3.3e-6), ("corr", 3.3e-6)])
def test_tails_of_templates(sfh, emu, O, kind, bound):
    """Every bin above 1e-6 of a template's maximum.  A kernel's value there is 2^-20
    of its peak: two roundings of an exponent of 20 (20 ln 2 2^-24 = 8e-7), and of
    its coordinates |a| < 3.7 (2 |a| da, da = 2^-25 |a| for each of two in the
    asymmetric kernel, 1.6e-6, and of three with the shear, 2.4e-6).  What the forms
    leave out is below that."""
    from sfh_amd import synth
    edges = synth.edges_200x300()
    ex, ey = oracle_range(O, edges[0]), oracle_range(O, edges[1])
    for la, mh, seed in ((6.74, -2.5, 100), (8.16, -1.14, 105), (8.72, -0.23, 107), (9.86, 0.0, 111)):
        sp, cm = synth.template_points(synth.TemplateSpec(la, mh, seed), 1200, edges, 120.0,
                                       correlation=0.6 if kind == "corr" else None)
        p = (sp.colors, sp.mags, sp.color_err, sp.mag_err, sp.weights)
        cov_mult, cm = 0 if kind == "asym" else 1, cm if kind == "corr" else None
        ref, _ = O.bin_cmd_smooth(*p[:4], cov_mult, p[4], ex, ey, cmult=cm, nthreads=8)
        mat, _ = _emu(emu, O, *p, cov_mult, ex, ey, cmult=cm)
        big = ref > 1e-6 * ref.max()
        worst = np.max(np.abs(mat[big] - ref[big]) / ref[big])
        assert worst <= bound, (worst, la, mh, seed)


# few high rows, fine columns, and kernels of about two columns much higher than wide
STEEP = [(200, 300, 2.0, 34.0, 1, None), (200, 300, 2.0, 40.0, 1, None), (200, 300, 1.78, 30.0, -1, None),
         (1000, 300, 1.8, 30.0, 1, None), (300, 5, 1.96, 3.357, -1, None), (300, 5, 2.45, 5.29, 1, None)]


def _sheared():
    """(nx, ny, sigma_x in columns, sigma_y / sigma_x, cov_mult, cmult): sigma_x
    across every change of form, sigma_y / sigma_x from 1/100 to 100, grids of few
    high rows and of fine columns, and the shears of correlations close to 1."""
    rng = np.random.default_rng(5)
    for nx, ny in ((200, 300), (300, 5), (1000, 4), (75, 100), (28, 40)):
        for sxc in np.geomspace(1.5, 0.6 * nx, 24):
            for ratio in np.geomspace(0.01, 100.0, 9) * rng.uniform(0.8, 1.25):
                yield nx, ny, sxc, ratio, 1, None
                yield nx, ny, sxc, ratio, -1, None
                r = 1.0 - 10.0 ** rng.uniform(-5.0, 0.0)
                yield nx, ny, sxc, ratio, 1, rng.choice([-1, 1]) * r / np.sqrt(1.0 - r * r) / ratio
                yield nx, ny, sxc, ratio, 1, rng.normal() * 10.0 ** rng.uniform(-1.0, 1.0)
    yield from STEEP


def _check_sheared(sfh, O, case, evaluate):
    """A kernel next to a row's middle node (between the nodes a kernel much
    narrower than a row has no part on the grid): finite, and within the
    coordinates' rounding.  With T the largest row coordinate |t| of the
    footprint, a row's t is off by dt = 3 2^-24 T and a column's a = u + g t by
    |g| dt and its own 3 2^-24 |u|, |u| < 8.  A value exp(-t^2 / 2 - a^2) is off
    by t dt + 2 a da of itself; relative to the peak's (at t_p, a_p) the factor
    2 a exp(a_p^2 - a^2) is below 2 (a_p + 0.43)."""
    nx, ny, sxc, ratio, cov_mult, cm = case
    ex, ey = sfh.edges_range(-0.5, 2.5, nx + 1), sfh.edges_range(18.0, 30.0, ny + 1)
    x, y, sx = 1.0 + 0.3 * ex.step, 18.0 + (ny // 2 + 0.51) * ey.step, sxc * ex.step
    sy = ratio * sx
    p = [np.array([v]) for v in (x, y, sx, sy, 1.0)]
    cmult = None if cm is None else np.array([cm])
    ref, _ = O.bin_cmd_smooth(*p[:4], cov_mult, p[4], oracle_range(O, ex), oracle_range(O, ey), cmult=cmult)
    mat = evaluate(p, cov_mult, ex, ey, cmult)
    assert np.isfinite(mat).all(), case
    peak = ref.max()
    if peak < 1e-9:            # a ridge that misses the bins: the oracle's own erf differences are noise
        return
    eps = 2.0 ** -24
    t = (18.0 + (np.arange(ny)[:, None] + 0.5 + 0.387 * np.array([-1, 0, 1])) * ey.step - y) / sy
    T = np.abs(t[np.abs(np.arange(ny) - ny // 2) <= max(1, round(5.0 * sy / ey.step)) + 1]).max()
    g = (cov_mult if cm is None else cm) * ratio / np.sqrt(2.0)
    col, row = np.unravel_index(ref.argmax(), ref.shape)
    a = np.abs((-0.5 + (col + 0.5) * ex.step - x) / (np.sqrt(2.0) * sx) + g * t[row])
    k = np.argmin(0.5 * t[row] ** 2 + a ** 2)
    dt = 3.0 * eps * T
    tol = TOL + abs(t[row, k]) * dt + 2.0 * (a[k] + 0.43) * (abs(g) * dt + 3.0 * eps * 8.0)
    worst = np.max(np.abs(mat - ref)) / peak
    assert worst <= tol, (worst, tol, case)


def test_sheared_kernels(sfh, emu, O):
    """The shift g t of a row's columns moves its ridge far out of the strips,
    whose products have to stay finite."""
    for case in _sheared():
        _check_sheared(sfh, O, case, lambda p, cov_mult, ex, ey, cmult: _emu(
            emu, O, *p, cov_mult, oracle_range(O, ex), oracle_range(O, ey), cmult=cmult)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("case", STEEP)
def test_sheared_kernels_on_the_device(sfh, gpu_ctx, O, case):
    _check_sheared(sfh, O, case, lambda p, cov_mult, ex, ey, cmult: sfh.bin_cmd_smooth(
        *p[:4], cov_mult, weights=p[4], edges=(ex, ey)).weights)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,n", [(200, 300, 1), (200, 300, 1500), (201, 77, 65), (33, 40, 63), (29, 41, 64),
                                     (28, 17, 129), (17, 5, 40), (16, 9, 300), (3, 2, 10), (1, 2, 5)])
@pytest.mark.parametrize("cov_mult", [1, -1, 0])
def test_one_template(sfh, gpu_ctx, O, nx, ny, n, cov_mult):
    """Grids around the strips' and nodes' edges, point counts around a chunk's,
    split over slices (one template leaves the chip idle)."""
    ex, ey = sfh.edges_range(-0.5, 2.5, nx + 1), sfh.edges_range(18.0, 21.0, ny + 1)
    p = _points(n, ex, ey, n + nx)
    ref, _ = O.bin_cmd_smooth(*p[:4], cov_mult, p[4], oracle_range(O, ex), oracle_range(O, ey))
    h = sfh.bin_cmd_smooth(*p[:4], cov_mult, weights=p[4], edges=(ex, ey))
    assert np.max(np.abs(h.weights - ref)) <= TOL * np.max(np.abs(ref))


@pytest.mark.gpu
@pytest.mark.parametrize("xo", [33, 35, 37])
def test_wide_footprint_of_erf_differences(sfh, gpu_ctx, emu, O, xo):
    """Edges so far from 0 that adding steps to them rounds to multiples of 64
    steps: the columns come out wider than the step that the footprint is counted
    in, so an erf-difference kernel's footprint spans 2 xo + 1 > 63 columns, which
    the shear's ridge crosses from end to end.  Against the host build, which
    takes a footprint column by column (the oracle rounds every column's
    coordinate, which here moves columns by half a width)."""
    first = 2.0 ** 58
    ex, ey = sfh.Range(first, 1.0, 401), sfh.edges_range(18.0, 21.0, 41)
    q = SimpleNamespace(cov_mult=1)
    sx = (2.0 * xo - 0.5) / 15.0                        # round(15 sx / 2) = xo
    for x in (128, 192, 256):
        xa, xb = x + 1 - xo, x + 1 + xo
        step = ((first + (xb - 0.5)) - (first + (xa - 0.5))) / (xb - xa)
        assert xb - xa + 1 > 63 and step / (2.0 * np.sqrt(2.0) * sx) > 0.12
        q.colors, q.mags, q.color_err, q.mag_err, q.weights = p = [np.array([v]) for v in (first + x, 19.5, sx, 0.2, 1.0)]
        for c in (100.0, -100.0):
            ref, _ = _emu(emu, O, *p, 1, oracle_range(O, ex), oracle_range(O, ey), cmult=np.array([c]))
            assert ref[xa - 1:xb].max(axis=1).min() > 1e-4 * ref.max()
            h = sfh.deposit_batch(sfh.PointBatch([q], (ex, ey), cmult_list=[np.array([c])])).cpu().numpy()
            assert np.max(np.abs(h[0] - ref.ravel(order="F"))) <= TOL * ref.max(), (x, c)


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [2, 130])
def test_batch_equals_single_templates(sfh, gpu_ctx, nt):
    """Templates of uneven point counts (none, one, a chunk and more) in one
    launch, sliced (2) and not (130), against the one-template call: FP32
    rounding of the output and the order of the FP64 sums apart, the same."""
    ex, ey = sfh.edges_range(-0.5, 2.5, 121), sfh.edges_range(18.0, 24.0, 141)

    class P:
        pass

    pts = []
    for t in range(nt):
        q = P()
        n = [0, 1, 64, 65, 200][t % 5] if nt > 2 else [65, 700][t]
        q.colors, q.mags, q.color_err, q.mag_err, q.weights = _points(n, ex, ey, t)
        q.cov_mult = 1
        pts.append(q)
    out = sfh.deposit_batch(sfh.PointBatch(pts, (ex, ey))).cpu().numpy()
    for t in range(nt):
        q = pts[t]
        h = sfh.bin_cmd_smooth(q.colors, q.mags, q.color_err, q.mag_err, 1, weights=q.weights, edges=(ex, ey))
        ref = h.weights.ravel(order="F")
        if not q.weights.size:
            assert not out[t].any() and not ref.any()
            continue
        assert np.max(np.abs(out[t] - ref)) <= 1e-7 * np.max(np.abs(ref))
