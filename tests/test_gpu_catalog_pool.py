"""Catalogues in recycled memory: sizes that grow and shrink from call to call,
several alive at once, two contexts and two host threads -- the same results
as in fresh memory."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _population(sfh, ctx, mass, seed):
    from sfh_amd import mock, synth
    m, mags = synth.isochrone(9.0, -1.0, 500, 7, mmax_imf=120.0)
    cat = sfh.generate_stars_mass(m, np.stack(mags, axis=1), ["B", "V"], mass, mock.Kroupa2001(0.08, 120.0),
                                  dist_mod=24.0, seed=seed, catalog=True, ctx=ctx)
    obs = sfh.model_cmd(cat, [synth.photerr] * 2, [synth.completeness] * 2, seed=seed + 1)
    r = cat.arrays() + obs.arrays()[1:]
    cat.close()
    return r, obs


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def test_recycled_catalogues(sfh, gpu_ctx):
    sizes = [2e3, 5e4, 3e4, 2e3, 5e4, 1e3]
    fresh = []
    for k, mass in enumerate(sizes):
        ctx = sfh.Context(0)
        r, obs = _population(sfh, ctx, mass, k)
        obs.close()
        ctx.close()
        fresh.append(r)
    ctx, alive = sfh.Context(0), []
    for rep in range(3):
        for k, mass in enumerate(sizes):
            r, obs = _population(sfh, ctx, mass, k)
            assert _same(r, fresh[k])
            alive.append((k, obs))
            if len(alive) > 3:
                alive.pop(0)[1].close()
            for j, o in alive:                         # the others' memory was not touched
                assert np.array_equal(o.arrays()[1], fresh[j][3])
    for _, o in alive:
        o.close()
    ctx.close()


def test_two_threads(sfh, gpu_ctx):
    want = [_population(sfh, gpu_ctx, 2e4, k)[0] for k in range(2)]
    bad = []

    def work(k):
        ctx = sfh.Context(0)
        for _ in range(4):
            r, obs = _population(sfh, ctx, 2e4, k)
            obs.close()
            if not _same(r, want[k]):
                bad.append(k)
        ctx.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


def test_failed_allocations_give_the_pools_back(sfh, gpu_ctx):
    """An allocation that does not fit, of any kind and in any context, first
    empties the pools of all contexts.  The sizes are refused by the runtime at
    once (petabytes), so nothing is filled up."""
    import ctypes

    import torch

    def buffer(ctx):
        p = ctypes.c_void_p()
        ctx.check(ctx.lib.sfh_buffer_alloc(ctx.handle, 1 << 50, ctypes.byref(p)))

    def templates(ctx):
        sfh.HIPTemplates(ctx=ctx, device_ptr=x.data_ptr(), shape=(1 << 30, 1 << 18))

    def data(ctx):
        sfh.HIPData(ctx=ctx, device_ptr=x.data_ptr(), nbins=1 << 47)

    x = torch.zeros(16, dtype=torch.float64, device="cuda")
    a, b = sfh.Context(0), sfh.Context(0)
    r, obs = _population(sfh, a, 4e5, 3)                # sizes the scratch buffers
    obs.close()
    for alloc in (buffer, templates, data):
        for ctx in (a, b):
            again, obs = _population(sfh, a, 4e5, 3)
            assert _same(again, r)
            obs.close()
            free = torch.cuda.mem_get_info()[0]
            with pytest.raises(sfh.DeviceError):
                alloc(ctx)
            assert torch.cuda.mem_get_info()[0] >= free + (10 << 20)
    again, obs = _population(sfh, a, 4e5, 3)            # and the contexts go on working
    assert _same(again, r)
    obs.close()
    a.close()
    b.close()
