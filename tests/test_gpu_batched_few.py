"""The batched fg! with few walkers: the narrow FP64 tiles (32 and 64 walkers),
the narrow split-K gradient and the log-likelihood-only call, at the edges
where their dispatch changes, against one walker at a time on the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,T,B", [(60, 3, 1), (257, 17, 2), (5000, 50, 31), (5000, 257, 32), (4999, 33, 33),
                                   (10001, 129, 64), (4097, 300, 65), (2000, 16, 128), (2000, 700, 129)])
@pytest.mark.parametrize("precision,tol_ll", [("f64", 1e-12), ("bf16x2", 1e-5), ("fp32", 1e-5)])
def test_few_walkers_against_oracle(sfh, O, gpu_ctx, N, T, B, precision, tol_ll):
    from sfh_amd import synth
    models = synth.synthetic_templates(N, T, seed=T)
    rng = np.random.default_rng(B)
    x = rng.uniform(100, 1000, T)
    data = synth.poisson_data(models.astype(np.float64) @ x, seed=3)
    X = synth.walkers(x, B, 0.2, seed=4)
    tpl = sfh.HIPTemplates(models)
    nll, G = sfh.fg_batched(X, tpl, data, precision=precision)
    ll_only, none = sfh.fg_batched(X, tpl, data, precision=precision, want_G=False)
    assert none is None and np.array_equal(ll_only, nll)
    for b in sorted({0, B // 2, B - 1}):
        ref_nl, ref_G, _ = O.fg(models, data, X[:, b])
        assert abs(nll[b] - ref_nl) <= tol_ll * abs(ref_nl)
        # G = sum_i C_i (1 - n_i / m_i), m from the composite: BF16 hi+lo operands
        # are off by 2^-17 of themselves each (FP32 ones and their sums by less),
        # so each of the two products by 2^-16
        q = data / (models.astype(np.float64) @ X[:, b])
        assert np.all(np.abs(G[:, b] - ref_G) <= 2.0 ** -16 * (models.T.astype(np.float64) @ (np.abs(1 - q) + q)))


@pytest.mark.parametrize("N,T,B", [(100, 50, 500), (700, 300, 257), (1500, 40, 300), (3000, 600, 130), (4200, 257, 385),
                                   (9000, 20, 140)])
@pytest.mark.parametrize("precision", ["f64", "bf16x2", "fp32"])
def test_every_split_and_tile_is_summed_once(sfh, gpu_ctx, N, T, B, precision):
    """The gradient's bins in 1, 1, 2, 5, 8 and more splits over the XCDs: every
    walker and template against FP64 products, within the bound above."""
    from sfh_amd import synth
    models = synth.synthetic_templates(N, T, seed=T)
    x = np.random.default_rng(B).uniform(100, 1000, T)
    data = synth.poisson_data(models.astype(np.float64) @ x, seed=3)
    X = synth.walkers(x, B, 0.2, seed=4)
    _, G = sfh.fg_batched(X, sfh.HIPTemplates(models), data, precision=precision)
    C = models.astype(np.float64)
    q = data[:, None] / (C @ X)
    assert np.all(np.abs(G - C.T @ (1 - q)) <= 2.0 ** -16 * (C.T @ (np.abs(1 - q) + q)))
