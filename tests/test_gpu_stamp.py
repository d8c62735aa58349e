"""The one-kernel drawing of N = 128 and 192 stamps (gsmi_draw_stamps_f32) against the FP64
kernels and the fold + row kernels, where its tiles and alias passes can go wrong: odd and even
sides from one pixel to the whole grid, no aliased samples, a few, and nearly one per cell, every
program shape and Moffat form, an inner shift (another shape), and non-finite stamps."""
import numpy as np
import pytest

import galsim_amd as g
from galsim_amd import _lib, batch
from galsim_amd.batch import BatchPlan

pytestmark = pytest.mark.gpu

# FP32 sums of an N x N inverse transform: about log2(N^2) roundings of 6e-8 on terms whose
# absolute sum is the peak pixel, leaf values good to a few ulp (Sersic's spline ten)
TOL = 3e-6


def _gal(kind, hlr, g1, g2):
    d = g.Exponential(half_light_radius=hlr, flux=300.)
    if kind == 'bulge_disk':
        d = d + g.Sersic(2.5, half_light_radius=0.5 * hlr, flux=100.)
    if kind == 'sersic':
        d = g.Sersic(4.0, half_light_radius=hlr, flux=100.)
    return d.shear(g1=g1, g2=g2)


def _psf(kind, fwhm):
    if kind.startswith('moffat'):
        return g.Moffat(beta=float(kind[6:]), fwhm=fwhm)
    return g.Kolmogorov(fwhm=fwhm)


def _general(plan):
    """The plan drawn by the fold and row kernels of any shape and size."""
    plan.stamp_groups, plan.wide_groups, plan.list_groups = [], [], list(plan.groups)
    plan.run()
    return plan


def _peak_rel(a, b):
    return float((a.double() - b.double()).abs().max() / b.double().abs().max())


SHAPES = [('bulge_disk', 'kolmogorov'), ('exp', 'moffat3'), ('exp', 'moffat2.5'),
          ('exp', 'moffat3.3'), ('sersic', 'kolmogorov'), ('exp', 'kolmogorov')]


@pytest.mark.parametrize("gal,psf", SHAPES)
@pytest.mark.parametrize("scale", [0.13, 0.2, 0.28])
@pytest.mark.parametrize("whole", [True, False])
def test_stamps_match_fp64_and_list_kernels(gal, psf, scale, whole, monkeypatch):
    monkeypatch.setattr(batch, 'STAMP_MIN', 0 if whole else 1000)
    sides = [(1, 1), (2, 3), (64, 64), (63, 65), (127, 128), (128, 127), (128, 128), (129, 40),
             (190, 191), (192, 192), (33, 192)]
    rng = np.random.default_rng(int(100 * scale) + len(gal) + len(psf))
    profs, offs = [], rng.uniform(-0.5, 0.5, (len(sides), 2))
    for i, (nx, ny) in enumerate(sides):
        gm, ph = rng.uniform(0., 0.6), rng.uniform(0., np.pi)
        hlr = min(0.01 * scale * max(nx, ny, 64), 0.4)
        p = _psf(psf, rng.uniform(0.62, 0.9))
        if i % 4 == 1:
            p = p.shear(g1=0.1, g2=-0.15)          # the PSF's form has a kx ky term
        profs.append(g.Convolve([_gal(gal, hlr, gm * np.cos(2 * ph), gm * np.sin(2 * ph)), p]))
    nx, ny = np.array(sides).T
    plan = BatchPlan(profs, nx, ny, scale, offs, precision='f32')
    assert {x[0] for x in plan.stamp_fit} <= {128, 192} and plan.stamp_fit
    assert bool(plan.stamp_groups) == whole
    plan.out.fill_(float('nan'))
    plan.run()
    lists = _general(BatchPlan(profs, nx, ny, scale, offs, precision='f32'))
    ref = _general(BatchPlan(profs, nx, ny, scale, offs, precision='f64'))
    for i in range(len(sides)):
        assert _peak_rel(plan.stamp(i), ref.stamp(i)) < TOL, (sides[i], plan.recs['Nk'])
        assert _peak_rel(plan.stamp(i), lists.stamp(i)) < TOL, sides[i]
    assert not plan.status().any()


def test_stamp_path_is_left_for_other_sizes_and_shapes(monkeypatch):
    """Beyond one alias per axis, another program shape, or FP64: the fold and row kernels."""
    monkeypatch.setattr(batch, 'STAMP_MIN', 0)
    def plan(prof, scale=0.2, precision='f32'):
        return BatchPlan([prof] * 2, 64, 64, scale, precision=precision)
    e, m = g.Exponential(half_light_radius=0.4), g.Moffat(beta=3, fwhm=0.7)
    assert plan(g.Convolve([e, m])).stamp_groups
    assert not plan(g.Convolve([e, m]), precision='f64').stamp_groups
    assert plan(g.Convolve([e, m]), precision='f64').wide_groups
    assert not plan(g.Convolve([e, m, g.Gaussian(sigma=0.1)]), precision='f64').wide_groups
    assert not plan(g.Convolve([e, m, g.Gaussian(sigma=0.1)])).stamp_groups
    assert not plan(g.Convolve([e.shift(0.1, 0.2), m])).stamp_groups
    coarse = plan(g.Convolve([e, m]), scale=0.9)
    assert int(coarse.recs['Nk'].max()) >= 2 * int(coarse.recs['N'].max())
    assert not coarse.stamp_groups
    coarse.run()
    ref = plan(g.Convolve([e, m]), scale=0.9, precision='f64')
    ref.run()
    assert _peak_rel(coarse.stamp(0), ref.stamp(0)) < TOL


def test_stamp_status_and_rejected_stamps(monkeypatch):
    """A stamp whose flux overflows FP32 is flagged and the next run clears the flag; a record
    that is not of the launch's size is left undrawn and flagged."""
    import torch
    monkeypatch.setattr(batch, 'STAMP_MIN', 0)
    e, m = g.Exponential(half_light_radius=0.6, flux=1e3), g.Moffat(beta=3, fwhm=0.7)
    profs = [g.Convolve([e, m]), g.Convolve([e.withFlux(1e38), m.withFlux(1e5)]),
             g.Convolve([e, m])]
    plan = BatchPlan(profs, 48, 48, 0.2, precision='f32')
    plan.run()
    assert plan.status().tolist() == [0, _lib.STAMP_NONFINITE, 0]
    ref = plan.out.clone()
    size = _lib.STAMP_DTYPE.itemsize
    o = plan._o_stamp + 2 * size + _lib.STAMP_DTYPE.fields['Nk'][1]
    word = plan.dev[o:o + 4].view(torch.int32)
    good = int(word)
    word.fill_(2 * 128)                                   # Nk = 2 N: two aliases per axis
    plan.out.fill_(7.)
    plan.run()
    assert plan.status().tolist() == [0, _lib.STAMP_NONFINITE, _lib.STAMP_NONFINITE]
    assert bool((plan.stamp(2) == 7.).all())
    word.fill_(good)
    plan.run()
    assert plan.status().tolist() == [0, _lib.STAMP_NONFINITE, 0]
    assert torch.equal(plan.stamp(2), ref[plan.stamp_offset[2]:][:48 * 48].view(48, 48))


@pytest.mark.parametrize("gal,psf", [SHAPES[0], SHAPES[3], SHAPES[4], SHAPES[5]])
@pytest.mark.parametrize("N", [256, 384, 512, 768, 1024, 1536, 2048, 3072, 4096])
def test_wide_sizes_match_fp64_kernels(gal, psf, N):
    """The column and row kernels of every larger size, with and without aliased samples: windows
    of the whole grid, one row, an odd few, and one more than a row chunk."""
    rng = np.random.default_rng(N + len(gal))
    for scale in (0.15, 0.28):
        sides = [(N, N - 1), (N - 2, 1), (N - 1, 33), (17, N - 3)]
        profs = []
        for nx, ny in sides:
            gm, ph = rng.uniform(0., 0.5), rng.uniform(0., np.pi)
            profs.append(g.Convolve([_gal(gal, 0.4, gm * np.cos(2 * ph), gm * np.sin(2 * ph)),
                                     _psf(psf, rng.uniform(0.62, 0.9))]))
        offs = rng.uniform(-0.5, 0.5, (len(sides), 2))
        nx, ny = np.array(sides).T
        plan = BatchPlan(profs, nx, ny, scale, offs, precision='f32')
        assert [x[0] for x in plan.wide_groups] == [N], plan.fft_sizes()
        plan.out.fill_(float('nan'))
        plan.run()
        ref = _general(BatchPlan(profs, nx, ny, scale, offs, precision='f64'))
        for i in range(len(sides)):
            peak = float(ref.stamp(0).abs().max())
            err = float((plan.stamp(i).double() - ref.stamp(i)).abs().max()) / peak
            assert err < TOL, (sides[i], scale)
        assert not plan.status().any()


@pytest.mark.parametrize("gal,psf", SHAPES)
@pytest.mark.parametrize("N", [128, 192, 256, 384, 512, 768, 1024, 1536, 2048])
def test_wide_fp64_matches_general_kernels(gal, psf, N):
    """The FP64 column and row kernels, samples beside the Exponential's clip rows included, in a
    batch and (a window of one shape) through drawImage."""
    rng = np.random.default_rng(N + len(psf))
    for scale in (0.15, 0.23):
        sides = [(N, N - 1), (N - 2, 1), (N - 1, 33), (17, N - 3)]
        profs = []
        for i, (nx, ny) in enumerate(sides):
            gm, ph = rng.uniform(0., 0.5), rng.uniform(0., np.pi)
            p = _psf(psf, rng.uniform(0.62, 0.9))
            if i == 1:
                p = p.shear(g1=0.1, g2=-0.15)
            hlr = 0.12 if N <= 192 else 0.4
            profs.append(g.Convolve([_gal(gal, hlr, gm * np.cos(2 * ph), gm * np.sin(2 * ph)),
                                     p]))
        offs = rng.uniform(-0.5, 0.5, (len(sides), 2))
        nx, ny = np.array(sides).T
        plan = BatchPlan(profs, nx, ny, scale, offs, precision='f64')
        assert [x[0] for x in plan.wide_groups] == [N], plan.fft_sizes()
        plan.out.fill_(float('nan'))
        plan.run()
        ref = _general(BatchPlan(profs, nx, ny, scale, offs, precision='f64'))
        for i in range(len(sides)):
            assert _peak_rel(plan.stamp(i), ref.stamp(i)) < 2e-14, (sides[i], scale)
        one = profs[3].drawImage(nx=17, ny=N - 3, scale=scale, offset=tuple(offs[3]),
                                 dtype=np.float64).array
        b = ref.stamp(3).cpu().numpy()
        assert np.abs(one - b).max() < 2e-14 * np.abs(b).max()
        assert not plan.status().any()


@pytest.mark.parametrize("precision", ['f32', 'f64'])
def test_sizes_drawn_together_and_apart(precision):
    """Every wide size in one launch (few stamps) against each by itself, and beside a size the list
    kernels draw (N = 64): their prepass leaves the other stamps' status alone."""
    sizes = [64, 128, 192, 256, 384, 512, 768, 1024, 1536, 2048] + \
        ([3072, 4096] if precision == 'f32' else [])
    gsp = g.GSParams(minimum_fft_size=64)
    profs, nx, ny = [], [], []
    for i, N in enumerate(sizes):
        e = g.Exponential(half_light_radius=0.1, flux=200., gsparams=gsp).shear(g1=0.2, g2=0.1)
        profs.append(g.Convolve([e, g.Kolmogorov(fwhm=0.3, gsparams=gsp)]))
        nx.append(N - i % 2)
        ny.append(N if i % 3 else 19)
    bad = {'f32': 1e38, 'f64': 1e306}[precision]
    e = g.Exponential(half_light_radius=0.1, flux=bad, gsparams=gsp).shear(g1=0.2, g2=0.1)
    profs += [g.Convolve([e, g.Kolmogorov(fwhm=0.3, flux=1e5, gsparams=gsp)])] * 2
    nx, ny = np.array(nx + [128, 384]), np.array(ny + [100, 300])
    plan = BatchPlan(profs, nx, ny, 0.1, precision=precision)
    assert [x[0] for x in plan.list_groups] == [64]
    for use in (False, True):
        if use:
            plan.use_schedule()
        plan.out.fill_(7.)
        plan.run()
        st = plan.status()
        assert (st[:-2] == 0).all() and (st[-2:] == _lib.STAMP_NONFINITE).all(), (use, st)
        together = plan.out.clone()
        for i in range(len(sizes)):
            one = BatchPlan([profs[i]], nx[i], ny[i], 0.1, precision=precision)
            one.run()
            # the same bodies with another number of threads
            assert _peak_rel(plan.stamp(i), one.stamp(0)) < (2e-7 if precision == 'f32' else 1e-15)
    ref = _general(BatchPlan(profs[:-2], nx[:-2], ny[:-2], 0.1, precision='f64')) \
        if precision == 'f64' else None
    if ref is not None:
        for i in range(len(sizes)):
            a = together[int(plan.stamp_offset[i]):][:int(nx[i] * ny[i])]
            assert _peak_rel(a, ref.stamp(i).reshape(-1)) < 2e-14
