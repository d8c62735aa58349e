"""The FP64 kernels' Moffat tables against the Bessel functions sample by sample (the same kernels
with no room for a table): every kind, orders from the smallest to beyond the table's, sheared and
shifted profiles, single drawings, batches and gradients."""
import numpy as np
import pytest

import galsim_amd as g
from galsim_amd import _lib, diff, render
from galsim_amd.batch import BatchPlan

pytestmark = pytest.mark.gpu

# both evaluate the transform to a few 1e-15 of its value at k = 0, and an image pixel sums
# N^2 samples of at most that over N^2
TOL = 2e-14
BETAS = [1.6, 1.8, 2.0, 2.3, 3.0, 3.4, 4.0, 5.9, 6.0, 7.5]


def _profiles(beta):
    m = g.Moffat(beta=beta, fwhm=0.7)
    e = g.Exponential(half_light_radius=0.6, flux=100.).shear(g1=0.3, g2=-0.2)
    return [g.Convolve([e, m]), g.Convolve([e, m.shear(g1=-0.4, g2=0.5)]),
            g.Convolve([g.Gaussian(sigma=0.3), m, g.Moffat(beta=2.7, half_light_radius=0.5)]),
            g.Convolve([e, m.shift(0.3, -0.2)]) + m, m]


def _no_tables(monkeypatch):
    monkeypatch.setattr(render, 'moffat_tables',
                        lambda recs, leaves, margin=0: (leaves, np.zeros(len(recs), np.int64)))


@pytest.mark.parametrize("beta", BETAS)
def test_images_match_sample_by_sample(beta, monkeypatch):
    profs = _profiles(beta)
    n = len(profs)
    nx, ny = np.array([64, 33, 190, 64, 128]), np.array([48, 65, 64, 300, 128])
    offs = np.random.default_rng(3).uniform(-0.5, 0.5, (n, 2))
    plan = BatchPlan(profs, nx, ny, 0.2, offs, precision='f64')
    sel = plan.host_leaves['type'] == _lib.LEAF_MOFFAT
    assert (plan.host_leaves['ntab'][sel] > 0).any() == (beta <= 6. or n > 2)
    plan.run()
    one = profs[0].drawImage(nx=64, ny=48, scale=0.2, offset=tuple(offs[0]),
                             dtype=np.float64).array
    _no_tables(monkeypatch)
    ref = BatchPlan(profs, nx, ny, 0.2, offs, precision='f64')
    assert not ref.host_leaves['ntab'][sel].any()
    ref.run()
    for i in range(n):
        peak = float(ref.stamp(i).abs().max())
        assert float((plan.stamp(i) - ref.stamp(i)).abs().max()) < TOL * peak, i
    assert np.abs(one - plan.stamp(0).cpu().numpy()).max() < TOL * np.abs(one).max()


@pytest.mark.parametrize("fit_beta", [False, True])
def test_gradients_match_as_parameters_move(fit_beta, monkeypatch):
    """Parameters far from those the plan was made for: the tables follow each step's records, and
    samples and orders beyond their room take the Bessel functions."""
    import torch
    rng = np.random.default_rng(5)
    n = 12
    cols = [rng.uniform(50., 200., n), rng.uniform(0.4, 1.2, n), rng.uniform(-0.3, 0.3, n),
            rng.uniform(-0.3, 0.3, n), rng.uniform(-0.3, 0.3, n), rng.uniform(-0.3, 0.3, n),
            rng.uniform(0.6, 0.9, n)]
    if fit_beta:
        cols.append(rng.uniform(2., 5.5, n))
    theta0 = np.stack(cols, axis=1)
    theta = theta0.copy()
    theta[:, 6] *= np.geomspace(0.02, 40., n)
    if fit_beta:
        theta[:, 7] = np.linspace(1.3, 8., n)
    t0 = torch.from_numpy(theta).cuda()

    def both():
        model = diff.ExpMoffat(theta0, 40, 40, scale=0.2, beta=3., precision='f64',
                               fit_beta=fit_beta)
        t = t0.clone().requires_grad_(True)
        img = model.render(t)
        cot = torch.cos(torch.arange(img.numel(), dtype=torch.float64, device='cuda'))
        torch.autograd.backward(img, grad_tensors=cot)
        return img.detach(), t.grad

    img, grad = both()
    _no_tables(monkeypatch)
    rimg, rgrad = both()
    assert float((img - rimg).abs().max()) < TOL * float(rimg.abs().max())
    scale = rgrad.abs().max(dim=1, keepdim=True).values
    # d/dbeta is a central difference of step 1e-4, good to about 1e-11 in either
    assert float(((grad - rgrad).abs() / scale).max()) < (1e-10 if fit_beta else 1e-12)
