"""The deposition's evaluation forms -- rows of merged Gauss-Legendre nodes,
wide kernels on every fourth column with interpolation between, launches whose
points are split into slices -- against the FP64 oracle, at the sizes where
their dispatch changes."""
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
