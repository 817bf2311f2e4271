"""The fused loss and gradient over facet-ordered tasks (mx_adjoint_step) at
the edges of its work list (needs an MI355X): facets without photons, with one
photon, with just under, at and just over one task's photons, runs longer than
one workgroup, more facets than the accumulators of the unordered kernels held
in LDS, and parameters in other layouts.  It equals the unordered kernels
(frames, replay with MX_AJ_SUMS, chain rule) on the same photons to 1e-11 of
each column's largest value in both precisions: every photon's derivatives are
the same bits, and sums of n <= 3e5 terms of both signs differ by a few times
log2(n) units of 1.1e-16 of their largest partial sums, some 1e3 units here."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(gpu, n_facets, counts, seed):
    """Photons sent through the middle of the lens towards points on facets of
    a CAT array (counts[f] of them for facet f), order -5 or -6, onto the CCD
    nearest in y; in random order, a few of them without weight."""
    import torch
    from marxs_amd import configs
    from marxs_amd.adjoint import AdjointProblem
    inst, parts = configs.cat_rowland_instrument(n_facets)
    rng = np.random.default_rng(seed)
    facet = np.repeat(np.arange(n_facets), counts)
    facet = rng.permutation(facet)
    n = len(facet)
    pos4d = np.array([e.pos4d for e in parts['gratings'].elements])
    centre, ey, ez = pos4d[facet, :3, 3], pos4d[facet, :3, 1], pos4d[facet, :3, 2]
    target = centre + ey * rng.uniform(-.9, .9, (n, 1)) + ez * rng.uniform(-.9, .9, (n, 1))
    d = -target / np.linalg.norm(target, axis=1)[:, None]
    pos = target - 500. * d
    t = lambda x, dt: torch.as_tensor(np.ascontiguousarray(x), dtype=dt, device=gpu)  # noqa: E731
    weight = rng.uniform(0.1, 1., n)
    weight[rng.random(n) < 0.02] = 0.
    return AdjointProblem(parts['gratings'], parts['ccds'], t(pos.T, torch.float64), t(d.T, torch.float64),
                          t(rng.uniform(0.5, 0.9, n), torch.float64), t(weight, torch.float64),
                          t(facet, torch.int32), t(rng.choice([-5, -6], n), torch.int32),
                          t(rng.integers(0, 16, n), torch.int32))


def _unordered(prob, theta, period, precision):
    import torch
    from marxs_amd import _lib
    from marxs_amd.adjoint import _launch
    pb = prob.buffers
    stream = torch.cuda.current_stream(prob.device).cuda_stream
    pb['theta'].copy_(theta)
    pb['period'].copy_(period)
    pb['accum'].zero_()
    _lib.check(_lib.lib.mx_facet_pose(ctypes.byref(prob._pose_args(0)), ctypes.c_void_p(stream)))
    one = prob._args(pb['geom'], precision, grad=pb['accum'], moments=pb['moments'])
    one.flags, one.lds_accumulate, one.y_shift = _lib.MX_AJ_SUMS, int(prob.F <= 315), prob.y_shift
    _launch(one, stream)
    _lib.check(_lib.lib.mx_facet_pose(ctypes.byref(prob._pose_args(2)), ctypes.c_void_p(stream)))
    return pb['loss'][0].clone(), pb['grad7'].clone(), pb['geom'].clone()


@pytest.mark.parametrize('counts', ['edges', 'even', 'long', 'one facet'])
@pytest.mark.parametrize('precision', [64, 32])
def test_step_equals_unordered_kernels(gpu, counts, precision):
    import torch
    if counts == 'edges':
        c = np.resize([0, 1, 127, 128, 129, 0, 256, 300], 320)
    elif counts == 'even':
        c = np.full(401, 37)
    elif counts == 'long':
        c = np.zeros(60, dtype=int)
        c[[3, 59]] = 5000, 300000
    else:
        c = np.zeros(50, dtype=int)
        c[17] = 4097
    prob = _problem(gpu, len(c), c, len(c))
    g = torch.Generator(device=gpu).manual_seed(1)
    theta = prob.theta0 + 1e-4 * torch.randn(prob.theta0.shape, dtype=torch.float64, device=gpu, generator=g)
    loss, gt, gp = prob.loss_and_grad(theta, prob.period0, precision)
    geom = prob.buffers['geom'].clone()
    assert torch.equal(prob.buffers['theta'], theta) and torch.equal(prob.buffers['grad7'][:, :6], gt)
    again = prob.loss_and_grad(theta, prob.period0, precision)
    assert torch.equal(loss, again[0]) and torch.equal(gt, again[1]) and torch.equal(gp, again[2])
    loss_u, g7, geom_u = _unordered(prob, theta, prob.period0, precision)
    assert torch.equal(geom, geom_u)
    assert abs(loss.item() - loss_u.item()) <= 1e-12 * abs(loss_u.item())
    got = torch.cat([gt, gp[:, None]], 1)
    scale = torch.abs(g7).max(0).values
    assert bool((torch.abs(got - g7) <= 1e-11 * scale).all())
    assert bool((got[torch.as_tensor(c == 0, device=gpu)] == 0).all())


def test_parameter_layouts(gpu):
    """A strided view, single precision and a broadcast period mean the same
    parameters."""
    import torch
    prob = _problem(gpu, 50, np.full(50, 20), 2)
    wide = torch.zeros((50, 12), dtype=torch.float64, device=gpu)
    wide[:, ::2] = prob.theta0.to(torch.float32)
    want = prob.loss_and_grad(wide[:, ::2].contiguous(), prob.period0.clone(), 64)
    for theta in (wide[:, ::2], wide[:, ::2].to(torch.float32)):
        got = prob.loss_and_grad(theta, prob.period0[:1].clone(), 64)
        for a, b in zip(got, want):
            assert torch.equal(a, b)
            assert a.is_contiguous() and a.dtype == torch.float64
