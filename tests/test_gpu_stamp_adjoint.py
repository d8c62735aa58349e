"""The one-kernel adjoint of N = 128 and 192 stamps (gsmi_adjoint_stamps_f32) against the FP64
adjoint kernels: every program shape and Moffat form, windows of one pixel, odd sides and the whole
grid, with and without aliased samples, sheared PSFs, and the order derivative."""
import numpy as np
import pytest

import galsim_amd as g
from galsim_amd import _lib, diff

pytestmark = pytest.mark.gpu


def _profile(shape, p, i):
    hlr, g1, g2, fwhm = p[i]
    psf = {'moffat': lambda: g.Moffat(beta=3., fwhm=fwhm),
           'moffat2.5': lambda: g.Moffat(beta=2.5, fwhm=fwhm),
           'moffat3.3': lambda: g.Moffat(beta=3.3, fwhm=fwhm)}.get(
               shape[1], lambda: g.Kolmogorov(fwhm=fwhm))()
    if i % 3 == 1:
        psf = psf.shear(g1=0.2, g2=-0.1)
    gal = {'exp': lambda: g.Exponential(half_light_radius=hlr, flux=200.),
           'sersic': lambda: g.Sersic(2.5, half_light_radius=hlr, flux=200.),
           'bulge_disk': lambda: g.Exponential(half_light_radius=hlr, flux=200.) +
           g.Sersic(2.5, half_light_radius=0.5 * hlr, flux=100.)}[shape[0]]()
    return g.Convolve([gal.shear(g1=g1, g2=g2), psf])


@pytest.mark.parametrize("shape", [('exp', 'moffat'), ('exp', 'moffat2.5'), ('exp', 'moffat3.3'),
                                   ('exp', 'kolmogorov'), ('sersic', 'kolmogorov'),
                                   ('bulge_disk', 'kolmogorov')])
@pytest.mark.parametrize("scale", [0.13, 0.28])
def test_adjoint_matches_fp64(shape, scale):
    import torch
    sides = np.array([(1, 1), (64, 63), (33, 128), (128, 128), (127, 5), (191, 192), (192, 190),
                      (150, 40)])
    n = len(sides)
    rng = np.random.default_rng(n + int(100 * scale))
    p = np.stack([rng.uniform(0.2, 0.4, n), rng.uniform(-0.3, 0.3, n), rng.uniform(-0.3, 0.3, n),
                  rng.uniform(0.62, 0.9, n)], axis=1)
    offs = rng.uniform(-0.5, 0.5, (n, 2))
    profs = [_profile(shape, p, i) for i in range(n)]
    beta = shape[1].startswith('moffat')
    out = {}
    for prec in ('f32', 'f64'):
        d = diff.DiffPlan(profs, sides[:, 0], sides[:, 1], scale, offs, prec,
                          moffat_generic=beta and shape[1] != 'moffat', shape_gradients=beta)
        if prec == 'f32':
            assert {b[0] for b in d._stamp_bins} <= {128, 192} and d._stamp_bins
            cot = torch.randn(d.plan.out.numel(), dtype=torch.float64,
                              generator=torch.Generator().manual_seed(1)).cuda()
        d.forward()
        out[prec] = d.adjoint(cot).cpu().numpy()
        f0 = d.fields0.cpu().numpy()
    ref, got = out['f64'], out['f32']
    assert np.isfinite(got).all()
    # a field's gradient is a sum over the k-image of random-sign terms good to a few 1e-7 each (the
    # order derivative 1e-6); they are compared in units of the stamp's largest sensitivity.  A
    # Sersic's q-derivative is a difference of neighbouring spline values in FP32, 5e-5 off in the
    # general FP32 kernels too
    s = np.abs(ref) * np.maximum(np.abs(f0), 1e-3)
    err = np.abs(got - ref) * np.maximum(np.abs(f0), 1e-3) / s.max(axis=1, keepdims=True)
    assert err.max() < (1e-5 if shape[0] == 'exp' else 1e-4), np.unravel_index(err.argmax(), err.shape)


def test_rejected_stamps_get_nan():
    import torch
    e, m = g.Exponential(half_light_radius=0.6, flux=1e3), g.Moffat(beta=3, fwhm=0.7)
    d = diff.DiffPlan([g.Convolve([e, m])] * 3, 48, 48, 0.2, precision='f32')
    cot = torch.ones(d.plan.out.numel(), dtype=torch.float32, device='cuda')
    ref = d.adjoint(cot).clone()
    o = d.plan._o_stamp + _lib.STAMP_DTYPE.itemsize + _lib.STAMP_DTYPE.fields['Nk'][1]
    d.plan.dev[o:o + 4].view(torch.int32).fill_(256)
    got = d.adjoint(cot)
    assert torch.isnan(got[1]).all()
    assert torch.equal(got[0], ref[0]) and torch.equal(got[2], ref[2])
