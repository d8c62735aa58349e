"""The work a user of galsim_amd has it do, as cases that can be timed and checked.

Each case is a dict of plain values; ``prepare`` builds what a program holds before the call
(profiles, a lowered batch, a differentiable model, device arrays), ``run`` makes one pass through
the public entry points, ``exact`` restates the result in 64-bit numpy / torch alone.

Kinds
  draw        GSObject.drawImage(method='fft') of one Exponential x Moffat galaxy, FP64, host image
              out: the per-object loop of a script
  real        drawImage(method='no_pixel') of a sheared Exponential + Gaussian + Moffat sum
  bulge_disk  BatchPlan of (Exponential + Sersic) x Kolmogorov galaxies planned from a config,
              uneven stamps, FP32: a survey simulation
  kolm        BatchPlan of Exponential x Kolmogorov galaxies on uneven (odd and even) stamps
  moffat      BatchPlan of Exponential x Moffat galaxies on one stamp size
  sersic      BatchPlan of large high-n Sersic x Kolmogorov galaxies at drawImage's own sizes
  grad        forward and backward of ExpMoffat: the step of a fit, one cotangent per pixel
  rfft        rfft2 then irfft2 of a device image (Image.calculate_fft / calculate_inverse_fft)
  cfft        fft2 and ifft2 of a complex device image with shifts
"""
import math

import numpy as np
import torch

SCALE = 0.2                       # arcsec per pixel


# -- the cases -----------------------------------------------------------------------------------
def listed():
    return [
        # one postage stamp at a time from a script: planning, launches and the copy back count
        {'name': 'draw_64', 'kind': 'draw', 'nx': 64, 'ny': 64},
        # one big, odd-sided, rectangular galaxy image in FP64
        {'name': 'draw_1001x769', 'kind': 'draw', 'nx': 1001, 'ny': 769},
        # a surface-brightness image evaluated at the pixel centres, copied to the host
        {'name': 'real_1000x1024', 'kind': 'real', 'nx': 1000, 'ny': 1024},
        # the benchmark's survey batch: every FFT size in one work list, replayed as a HIP graph
        {'name': 'bulge_disk_4096', 'kind': 'bulge_disk', 'n': 4096, 'graph': True},
        # a small batch of a per-exposure loop, drawn once by the default per-size launches
        {'name': 'bulge_disk_100', 'kind': 'bulge_disk', 'n': 100, 'graph': False},
        # uneven stamps, odd sides among them, drawn once by the default per-size launches
        {'name': 'kolm_500', 'kind': 'kolm', 'n': 500, 'lo': 32, 'hi': 255, 'precision': 'f32'},
        # FP64 stamps of one size, as a validation batch draws them
        {'name': 'moffat_f64_256', 'kind': 'moffat', 'n': 256, 'side': 64, 'precision': 'f64'},
        # bright, extended galaxies: FFT grids of 384 to 3072
        {'name': 'sersic_64', 'kind': 'sersic', 'n': 64},
        # the step of a 7-parameter fit of equal stamps
        {'name': 'grad_1024', 'kind': 'grad', 'n': 1024, 'lo': 64, 'hi': 64,
         'precision': 'f32', 'fit_beta': False},
        # the step of an 8-parameter fit (the Moffat beta free) of uneven stamps
        {'name': 'grad_beta_1024', 'kind': 'grad', 'n': 1024, 'lo': 32, 'hi': 128,
         'precision': 'f32', 'fit_beta': True},
        # an image and its half-plane transform, there and back
        {'name': 'rfft_2048', 'kind': 'rfft', 'm': 2048, 'n': 2048},
        # complex arrays of ragged sizes (1174 = 2 x 587, 1500 = 4 x 3 x 125), shifted
        {'name': 'cfft_1174x1500', 'kind': 'cfft', 'm': 1174, 'n': 1500},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _even(v):
    return v + v % 2


def draw(rng):
    kind = rng.choice(['draw', 'real', 'bulge_disk', 'kolm', 'moffat', 'sersic', 'grad', 'rfft',
                       'cfft'])
    if kind == 'draw':
        return {'kind': kind, 'nx': _log_int(rng, 32, 1000), 'ny': _log_int(rng, 32, 1000)}
    if kind == 'real':
        return {'kind': kind, 'nx': _log_int(rng, 64, 1024), 'ny': _log_int(rng, 64, 1000)}
    if kind == 'bulge_disk':
        return {'kind': kind, 'n': _log_int(rng, 16, 4096), 'graph': rng.random() < 0.5}
    if kind == 'kolm':
        hi = rng.randint(64, 255)
        return {'kind': kind, 'n': _log_int(rng, 8, 500), 'lo': rng.randint(24, 48), 'hi': hi,
                'precision': rng.choice(['f32', 'f64'])}
    if kind == 'moffat':
        return {'kind': kind, 'n': _log_int(rng, 8, 512), 'side': rng.randint(24, 192),
                'precision': rng.choice(['f32', 'f64'])}
    if kind == 'sersic':
        return {'kind': kind, 'n': rng.randint(4, 64)}
    if kind == 'grad':
        lo = rng.randint(24, 64)
        precision = rng.choice(['f32', 'f32', 'f64'])
        return {'kind': kind, 'n': _log_int(rng, 16, 1024 if precision == 'f32' else 96),
                'lo': lo, 'hi': rng.randint(lo, 128), 'precision': precision,
                'fit_beta': rng.random() < 0.5}
    return {'kind': kind, 'm': _even(_log_int(rng, 64, 2048)),
            'n': _even(_log_int(rng, 64, 2048))}


# -- inputs --------------------------------------------------------------------------------------
def _rng(seed, tag):
    return np.random.default_rng([int(seed) & 0x7fffffff, tag])


def _draw_params(case, seed):
    """One galaxy whose size suits the stamp (about a tenth of its side)."""
    r = _rng(seed, 1)
    side = max(case['nx'], case['ny']) * SCALE
    g, phi = r.uniform(0., 0.5), r.uniform(0., math.pi)
    return {'hlr': side * r.uniform(0.04, 0.1), 'flux': 10. ** r.uniform(2., 5.),
            'g1': g * math.cos(2 * phi), 'g2': g * math.sin(2 * phi),
            'fwhm': r.uniform(0.6, 1.0), 'beta': r.uniform(2.5, 4.5),
            'offset': (r.uniform(-0.5, 0.5), r.uniform(-0.5, 0.5))}


def _real_params(case, seed):
    r = _rng(seed, 2)
    side = max(case['nx'], case['ny']) * SCALE
    g, phi = r.uniform(0., 0.5), r.uniform(0., math.pi)
    return {'disk': side * r.uniform(0.05, 0.1), 'sigma': side * r.uniform(0.01, 0.05),
            'rd': side * r.uniform(0.01, 0.03), 'beta': r.uniform(2.2, 4.2),
            'flux': r.uniform(10., 1000., 3), 'g1': g * math.cos(2 * phi),
            'g2': g * math.sin(2 * phi), 'offset': r.uniform(-0.5, 0.5, 2)}


def _sides(case):
    """Stamp sides of the uneven kinds: the case's own, whatever the inputs."""
    r = _rng(case['n'], 1000 + case['lo'] * 256 + case['hi'])
    nx = r.integers(case['lo'], case['hi'] + 1, case['n'])
    ny = r.integers(case['lo'], case['hi'] + 1, case['n'])
    return nx, ny


def _gal_params(n, seed, tag):
    """Exponential galaxies: hlr ~ U(0.4, 1.6)", |g| ~ U(0, 0.5), sub-pixel offsets, seeing
    fwhm ~ U(0.6, 1.0)", Moffat beta ~ U(2.5, 4.5)."""
    r = _rng(seed, tag)
    g, phi = r.uniform(0., 0.5, n), r.uniform(0., math.pi, n)
    return {'flux': 10. ** r.uniform(2., 5., n), 'hlr': r.uniform(0.4, 1.6, n),
            'g1': g * np.cos(2 * phi), 'g2': g * np.sin(2 * phi),
            'dx': r.uniform(-0.5, 0.5, n), 'dy': r.uniform(-0.5, 0.5, n),
            'fwhm': r.uniform(0.6, 1.0, n), 'beta': r.uniform(2.5, 4.5, n)}


def _grad_inputs(case, seed):
    """(theta0, theta, sides, cotangent parts): the initial guess the grids come from, the
    parameters of the step a little off it, and per-pixel noise for the cotangent."""
    n = case['n']
    p = _gal_params(n, seed, 5)
    r = _rng(seed, 6)
    beta = p['beta'] if case['fit_beta'] else np.full(n, 3.)
    theta0 = np.stack([p['flux'], p['hlr'], p['g1'], p['g2'], p['dx'], p['dy'], p['fwhm']],
                      axis=1)
    theta = theta0 * (1. + 0.02 * r.standard_normal(theta0.shape))
    if case['fit_beta']:
        theta0 = np.concatenate([theta0, beta[:, None]], axis=1)
        theta = np.concatenate([theta, (beta * (1. + 0.02 * r.uniform(-1., 1., n)))[:, None]],
                               axis=1)
    sides = _sides(case)[0]
    return theta0, theta, beta, sides


def _cotangent(case, seed, order, sides):
    """dL/dI of a fit, flat in the drawn order: unit noise plus a smooth misfit under the
    galaxy, rounded to FP32 so that both precisions take the same numbers."""
    out = []
    for i in order:
        s = int(sides[i])
        r = _rng(seed, 7 + 16 * int(i))
        y = (np.arange(s) - 0.5 * (s - 1))[:, None]
        x = (np.arange(s) - 0.5 * (s - 1))[None, :]
        bump = np.exp(-0.5 * (x * x + y * y) / (0.08 * s) ** 2)
        a, b, c = r.uniform(1., 3., 3)
        out.append((r.standard_normal((s, s)) + bump * (a + 0.3 * b * x - 0.3 * c * y)).ravel())
    return np.concatenate(out).astype(np.float32)


def _bulge_disk(case, seed):
    """The catalogue (sizes, Sersic indices, shears, hence the stamp sides) is the case's own;
    fluxes, bulge fractions, position angles and seeing are the inputs'."""
    import galsim_amd as g
    from galsim_amd import config, workloads
    n = case['n']
    p = workloads.bulge_disk_params(n, n)
    sizes = np.array([workloads.stamp_size(workloads.bulge_disk_profile(g, p, i), SCALE)
                      for i in range(n)])
    r = _rng(seed, 4)
    gm, phi = np.hypot(p['g1'], p['g2']), r.uniform(0., math.pi, n)
    p.update(g1=gm * np.cos(2 * phi), g2=gm * np.sin(2 * phi), bfrac=r.uniform(0., 0.6, n),
             flux=10. ** r.uniform(2., 5., n), psf_fwhm=r.uniform(0.6, 1.0, n))
    return config.plan_config(workloads.bulge_disk_config(p, sizes), n, 'f32', seed=1)


def _fft_input(case, seed):
    """A noisy image (real) or a noisy transform (complex) of unit variance."""
    gen = torch.Generator(device='cpu').manual_seed(int(seed) & 0x7fffffff)
    shape = (case['m'], case['n'])
    if case['kind'] == 'rfft':
        return torch.randn(shape, generator=gen, dtype=torch.float64)
    return torch.complex(torch.randn(shape, generator=gen, dtype=torch.float64),
                         torch.randn(shape, generator=gen, dtype=torch.float64))


def prepare(case, seed):
    import galsim_amd as g
    from galsim_amd.batch import BatchPlan
    kind = case['kind']
    if kind == 'draw':
        p = _draw_params(case, seed)
        gal = g.Exponential(half_light_radius=p['hlr'], flux=p['flux'])
        gal = gal.shear(g1=p['g1'], g2=p['g2'])
        prof = g.Convolve([gal, g.Moffat(beta=p['beta'], fwhm=p['fwhm'])])
        return {'kind': kind, 'prof': prof, 'nx': case['nx'], 'ny': case['ny'],
                'offset': p['offset']}
    if kind == 'real':
        p = _real_params(case, seed)
        gal = (g.Exponential(half_light_radius=p['disk'], flux=p['flux'][0]) +
               g.Gaussian(sigma=p['sigma'], flux=p['flux'][1])).shear(g1=p['g1'], g2=p['g2'])
        prof = gal + g.Moffat(beta=p['beta'], scale_radius=p['rd'], flux=p['flux'][2])
        return {'kind': kind, 'prof': prof, 'nx': case['nx'], 'ny': case['ny'],
                'offset': tuple(p['offset'])}
    if kind == 'bulge_disk':
        plan = BatchPlan(None, None, None, None, lowered=_bulge_disk(case, seed))
        if case['graph']:
            plan.use_schedule()
            plan.capture()
        return {'kind': kind, 'plan': plan, 'graph': case['graph']}
    if kind in ('kolm', 'moffat'):
        n = case['n']
        p = _gal_params(n, seed, 3)
        nx, ny = _sides(case) if kind == 'kolm' else (case['side'], case['side'])
        profs = []
        for i in range(n):
            gal = g.Exponential(half_light_radius=p['hlr'][i], flux=p['flux'][i])
            gal = gal.shear(g1=p['g1'][i], g2=p['g2'][i])
            psf = (g.Kolmogorov(fwhm=p['fwhm'][i]) if kind == 'kolm' else
                   g.Moffat(beta=3., fwhm=p['fwhm'][i]))
            profs.append(g.Convolve([gal, psf]))
        plan = BatchPlan(profs, nx, ny, SCALE, offsets=np.stack([p['dx'], p['dy']], axis=1),
                         precision=case['precision'])
        return {'kind': kind, 'plan': plan, 'graph': False}
    if kind == 'sersic':
        from galsim_amd import workloads
        # the galaxies' sizes and indices, hence the sides, are the case's; the rest the inputs'
        n = case['n']
        p = workloads.large_sersic_params(n, n)
        sides = [workloads.large_sersic_profile(g, p, i).getGoodImageSize(SCALE)
                 for i in range(n)]
        r = _rng(seed, 8)
        p.update(flux=10. ** r.uniform(3., 5., n), psf_fwhm=r.uniform(0.7, 0.9, n))
        profs = [workloads.large_sersic_profile(g, p, i) for i in range(n)]
        plan = BatchPlan(profs, sides, sides, SCALE, offsets=r.uniform(-0.5, 0.5, (n, 2)),
                         precision='f32')
        plan.use_schedule()
        return {'kind': kind, 'plan': plan, 'graph': False}
    if kind == 'grad':
        from galsim_amd import diff
        theta0, theta, beta, sides = _grad_inputs(case, seed)
        model = diff.ExpMoffat(theta0, sides, sides, scale=SCALE, beta=beta,
                               precision=case['precision'], fit_beta=case['fit_beta'])
        order = np.argsort(model.dplan.plan.stamp_offset)
        cot = torch.from_numpy(_cotangent(case, seed, order, sides)).cuda()
        if case['precision'] == 'f64':
            cot = cot.double()
        return {'kind': kind, 'model': model, 'theta': torch.from_numpy(theta).cuda(),
                'cot': cot}
    return {'kind': kind, 'a': _fft_input(case, seed).cuda()}


# -- one pass ------------------------------------------------------------------------------------
def run(state):
    kind = state['kind']
    if kind == 'draw':
        return state['prof'].drawImage(nx=state['nx'], ny=state['ny'], scale=SCALE,
                                       offset=state['offset'], dtype=np.float64).array
    if kind == 'real':
        return state['prof'].drawImage(nx=state['nx'], ny=state['ny'], scale=SCALE,
                                       offset=state['offset'], method='no_pixel',
                                       dtype=np.float64).array
    if kind == 'grad':
        t = state['theta'].detach().requires_grad_(True)
        img = state['model'].render(t)
        torch.autograd.backward(img, grad_tensors=state['cot'])
        return {'image': img.detach(), 'grad': [t.grad[:, k] for k in range(t.shape[1])]}
    if kind in ('rfft', 'cfft'):
        from galsim_amd import fft
        if kind == 'rfft':
            k = fft.rfft2(state['a'], shift_out=True)
            return {'k': k, 'x': fft.irfft2(k, shift_in=True)}
        return {'fwd': fft.fft2(state['a'], shift_in=True, shift_out=True),
                'inv': fft.ifft2(state['a'], shift_out=True)}
    if state['graph']:
        return state['plan'].replay()
    return state['plan'].run()


# -- what a pass cannot do without ---------------------------------------------------------------
def _good_fft(n):
    """Smallest 2^k or 3 2^k that is at least n (and at least 2)."""
    k = math.ceil(math.log2(max(n, 2)) - 1e-12)
    return 3 * 2 ** (k - 2) if n <= 3 * 2 ** (k - 2) and k >= 2 else 2 ** k


def _fft_flops(m, n, real):
    """Radix-2 count of a 2-d transform of m x n (half of it for real data)."""
    return 5. * m * n * math.log2(m * n) * (0.5 if real else 1.)


def _stamp_flops(ny, nx, leaves):
    """A drawn stamp: each half-plane sample of the k-image takes about 10 operations per leaf
    and 10 for the axis factors, then the real inverse transform."""
    N = max(128, _good_fft(max(nx, ny)))
    return 0.5 * N * N * 10. * (leaves + 1) + _fft_flops(N, N, True)


def work(case):
    kind = case['kind']
    elem = 4 if case.get('precision', 'f32') == 'f32' else 8
    if kind == 'draw':
        return {'bytes': 8 * case['nx'] * case['ny'] + 512,
                'flops': _stamp_flops(case['ny'], case['nx'], 2)}
    if kind == 'real':
        return {'bytes': 8 * case['nx'] * case['ny'] + 512,
                'flops': 60. * case['nx'] * case['ny']}
    if kind == 'bulge_disk':
        # 24,900 pixels on average over the parameter distribution; 700 bytes of records a stamp
        return {'bytes': case['n'] * (4 * 24900 + 700),
                'flops': case['n'] * _stamp_flops(158, 158, 3)}
    if kind in ('kolm', 'moffat'):
        nx, ny = _sides(case) if kind == 'kolm' else ([case['side']] * case['n'],) * 2
        return {'bytes': float(sum(elem * int(x) * int(y) + 500 for x, y in zip(nx, ny))),
                'flops': float(sum(_stamp_flops(int(y), int(x), 2) for x, y in zip(nx, ny)))}
    if kind == 'sersic':
        # drawImage's own sides: 1.8 million pixels on average
        return {'bytes': case['n'] * (4 * 1800000 + 600),
                'flops': case['n'] * _stamp_flops(1340, 1340, 2)}
    if kind == 'grad':
        s = [int(v) for v in _sides(case)[0]]
        # image out, cotangent in, parameters in and gradients out; two transforms and the leaf
        # values with their derivatives
        return {'bytes': float(sum(2 * elem * v * v + 128 + 700 for v in s)),
                'flops': float(sum(3. * _stamp_flops(v, v, 2) for v in s))}
    m, n = case['m'], case['n']
    if kind == 'rfft':
        w = n // 2 + 1
        # image in, half-plane out, half-plane in, image out
        return {'bytes': 2. * (8 * m * n + 16 * m * w), 'flops': 2. * _fft_flops(m, n, True)}
    # one array in, two out
    return {'bytes': 3. * 16 * m * n, 'flops': 2. * _fft_flops(m, n, False)}


def tolerance(case):
    """About four times the error against ``exact`` that was measured (relative, 2-norm): FP64
    7e-16 (transforms) to 1.8e-15 (images, which another library of elementary functions moves by
    an ulp or two per factor), FP32 images and gradients 0.7e-7 to 3.3e-7 (a Sersic's spline in
    32 bits is several times coarser than the closed forms), the gradient of a free Moffat beta
    7e-6 (a difference of nearly equal integrals)."""
    kind = case['kind']
    if kind in ('rfft', 'cfft'):
        return {'rel': 3e-15}
    if kind == 'draw':
        return {'rel': 1e-14}
    if kind == 'real':
        # 4e-15 with coordinates from the pixel's indices; coordinates summed along a row, as
        # GalSim has them, are 1e-13 off
        return {'rel': 2e-14}
    if case.get('precision', 'f32') == 'f64':
        # a central difference in FP64 gives the beta gradient
        return {'rel': (1e-7 if case['fit_beta'] else 1e-12) if kind == 'grad' else 1e-14}
    if kind == 'grad':
        return {'rel': 3e-5 if case['fit_beta'] else 2e-6}
    return {'rel': 2e-6}


# -- the same results in 64 bits -----------------------------------------------------------------
HLR_TO_R0 = 1. / 1.6783469900166605          # Exponential scale radius per half-light radius
KOLM_K0 = 2.992939911888651                  # k0 lambda / r0 of the Kolmogorov transform
KOLM_FWHM = 0.9758634299                     # fwhm per lambda / r0
KOLM_HLR = 0.5548101137                      # half-light radius per lambda / r0
FOLD, MAXK_T, KACC, XACC, MIN_HLR = 5e-3, 1e-3, 1e-5, 1e-5, 5.


def _moffat_u(nu, x):
    """x^nu K_nu(x) for x >= 0 (nu a float or a tensor that broadcasts), from K_nu(x) =
    int_0^inf exp(-x cosh t) cosh(nu t) dt (A&S 9.6.24) by the trapezoid rule with step 1/5: the
    integrand is analytic in |Im t| < pi/2, so the rule is good to about exp(-5 pi^2)."""
    nu = torch.as_tensor(nu, dtype=torch.float64, device=x.device)
    pos = x > 0
    xs = torch.where(pos, x, torch.ones_like(x))
    acc = 0.5 * torch.exp(-xs)
    top = float(torch.acosh(1. + 60. / xs.min()).item())
    h = 0.2
    for m in range(1, int(top / h) + 2):
        acc = acc + torch.exp(-xs * math.cosh(m * h)) * torch.cosh(nu * (m * h))
    at0 = torch.exp((nu - 1.) * math.log(2.) + torch.lgamma(nu))
    return torch.where(pos, h * acc * xs ** nu, at0 + torch.zeros_like(x))


def _moffat_k(beta, k):
    """Unit-flux Moffat transform at k = |k| rD: 4 / (Gamma(beta-1) 2^beta) k^nu K_nu(k)."""
    b = torch.as_tensor(beta, dtype=torch.float64, device=k.device)
    return 4. * torch.exp(-torch.lgamma(b - 1.) - b * math.log(2.)) * _moffat_u(b - 1., k)


def _moffat_rd(fwhm, beta):
    return fwhm / (2. * (2. ** (1. / beta) - 1.) ** 0.5)


def _moffat_sizes(fwhm, beta):
    """(maxk, stepk): the transform falls to the maxk threshold; all but the folding threshold
    of the flux, and five half-light radii, inside pi / stepk."""
    rd = _moffat_rd(fwhm, beta)
    lo, hi = 0., 60.
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        v = float(_moffat_k(beta, torch.tensor([mid], dtype=torch.float64))[0])
        lo, hi = (mid, hi) if v > MAXK_T else (lo, mid)
    R = FOLD ** (0.5 / (1. - beta))
    R = min(R, math.sqrt(XACC ** (1. / (1. - beta)) - 1.))
    R = max(R, MIN_HLR * math.sqrt(0.5 ** (1. / (1. - beta)) - 1.))
    return lo / rd, math.pi / (R * rd)


def _kolm_sizes(fwhm):
    """(maxk, stepk) of the Kolmogorov transform exp(-(k / k0)^(5/3)); its folding radius is
    that of its r^(-11/3) wing, sb -> C r^(-11/3) with C = 2^(5/3) Gamma(11/6) (5/6) /
    (pi Gamma(1/6)) in units of k0, which holds the folding threshold outside R."""
    k0 = KOLM_K0 * KOLM_FWHM / fwhm
    C = 2. ** (5. / 3.) * (5. / 6.) * math.gamma(11. / 6.) / (math.pi * math.gamma(1. / 6.))
    R = (2. * math.pi * C / (5. / 3. * FOLD)) ** 0.6
    R = max(R, MIN_HLR * KOLM_K0 * KOLM_HLR)
    return (-math.log(KACC)) ** 0.6 * k0, math.pi / R * k0


def _exp_sizes(hlr):
    r0 = hlr * HLR_TO_R0
    logx = math.log(FOLD)
    R = -logx
    for _ in range(3):
        R = math.log(1. + R) - logx
    return MAXK_T ** (-1. / 3.) / r0, math.pi / (max(R, MIN_HLR / HLR_TO_R0) * r0)


def _grid(hlr, g, psf_sizes, nx, ny, dx, dy):
    """(N, Nk, ux, uy) of a sheared Exponential x PSF drawn on nx x ny pixels: the shear
    stretches by sqrt((1+g)/(1-g)); convolution takes the smallest maxk and adds the folding
    radii in quadrature, the pixel among them; an offset adds its length."""
    maxk_e, stepk_e = _exp_sizes(hlr)
    s = math.sqrt((1. + g) / (1. - g))
    maxk = min(maxk_e * s, psf_sizes[0]) * SCALE
    stepk = SCALE / math.sqrt((stepk_e / s) ** -2 + psf_sizes[1] ** -2)
    ux = dx - (0.5 if nx % 2 == 0 else 0.)
    uy = dy - (0.5 if ny % 2 == 0 else 0.)
    if ux != 0. or uy != 0.:
        stepk = math.pi / (math.pi / stepk + math.hypot(ux, uy))
    stepk = 1. / math.sqrt(stepk ** -2 + math.pi ** -2)
    maxk = min(maxk, 2. / MAXK_T)
    N = 2 * ((math.ceil(2. * math.pi / stepk * (1. - 1e-12)) + 1) // 2)
    N = max(N, 2 * (max(nx, ny) // 2), max(nx, ny))
    N = max(_good_fft(N), 128)
    dk = 2. * math.pi / N
    Nk = N if math.pi > maxk else 2 * math.ceil(maxk / dk)
    return N, Nk, ux, uy


def _image(hlr, flux, g1, g2, psf, N, Nk, nx, ny, ux, uy, device):
    """Pixels of the sheared Exponential times psf(kx, ky), pixel-convolved: the inverse DFT of
    every k sample |kx|, |ky| <= Nk/2 on the N grid, as two products with the DFT matrices."""
    hk = Nk // 2
    j = torch.arange(-hk, hk + 1, dtype=torch.float64, device=device)
    k = j * (2. * math.pi / N)
    kx, ky = k[None, :], k[:, None]
    den = (1. - (g1 * g1 + g2 * g2)) ** 0.5
    ax = ((1. + g1) * kx + g2 * ky) / den / SCALE
    ay = (g2 * kx + (1. - g1) * ky) / den / SCALE
    q = (ax * ax + ay * ay) * (hlr * HLR_TO_R0) ** 2
    gal = torch.where(q > KACC ** (-1. / 1.5) - 1., torch.zeros_like(q), flux * (1. + q) ** -1.5)
    sinc = torch.sinc(k / (2. * math.pi))
    F = gal * psf(torch.sqrt(kx * kx + ky * ky) / SCALE) * (sinc[None, :] * sinc[:, None])

    def dft(n, u):
        p = torch.arange(n, dtype=torch.float64, device=device) - n // 2
        # the whole turns of p j / N go exactly, in integers
        whole = torch.remainder(p[:, None] * j[None, :], float(N)) * (2. * math.pi / N)
        ph = whole - u * k[None, :]
        return torch.complex(torch.cos(ph), torch.sin(ph))

    Ex, Ey = dft(nx, ux), dft(ny, uy)
    return (Ey @ (F.to(torch.complex128) @ Ex.T)).real / (N * N)


def _exact_real(case, seed):
    p = _real_params(case, seed)
    nx, ny = case['nx'], case['ny']
    u = [p['offset'][0] - (0.5 if nx % 2 == 0 else 0.), p['offset'][1] - (0.5 if ny % 2 == 0
                                                                       else 0.)]
    x = ((np.arange(nx) - nx // 2 - u[0]) * SCALE)[None, :]
    y = ((np.arange(ny) - ny // 2 - u[1]) * SCALE)[:, None]
    den = math.sqrt(1. - p['g1'] ** 2 - p['g2'] ** 2)
    sx = ((1. - p['g1']) * x - p['g2'] * y) / den
    sy = (-p['g2'] * x + (1. + p['g1']) * y) / den
    r2 = sx * sx + sy * sy
    r0 = p['disk'] * HLR_TO_R0
    out = p['flux'][0] / (2. * math.pi * r0 ** 2) * np.exp(-np.sqrt(r2) / r0)
    out = out + p['flux'][1] / (2. * math.pi * p['sigma'] ** 2) * np.exp(-0.5 * r2 /
                                                                        p['sigma'] ** 2)
    b, rd = p['beta'], p['rd']
    m = (x * x + y * y) / rd ** 2
    # GalSim's Moffat ends where its surface brightness has fallen by xvalue_accuracy^(b/(b-1))
    out = out + np.where(m > XACC ** (1. / (1. - b)) - 1., 0.,
                         p['flux'][2] * (b - 1.) / (math.pi * rd ** 2) * (1. + m) ** -b)
    return out * SCALE ** 2


def _exact_grad(case, seed):
    theta0, theta, beta, sides = _grad_inputs(case, seed)
    dev = 'cuda' if torch.cuda.is_available() else 'cpu'
    grids = []
    for i, t in enumerate(theta0):
        s = int(sides[i])
        N, Nk, _, _ = _grid(t[1], math.hypot(t[2], t[3]), _moffat_sizes(t[6], beta[i]), s, s,
                            t[4], t[5])
        grids.append((N, Nk, s))
    order = np.argsort([gr[0] for gr in grids], kind='stable')
    cot = torch.from_numpy(_cotangent(case, seed, order, sides)).to(dev).double()
    th = torch.from_numpy(theta).to(dev).requires_grad_(True)
    images, at = [], 0
    for i in order:
        N, Nk, s = grids[i]
        t = th[i]
        b = t[7] if case['fit_beta'] else torch.tensor(3., dtype=torch.float64, device=dev)
        shift = 0.5 if s % 2 == 0 else 0.
        rd = _moffat_rd(t[6], b)
        img = _image(t[1], t[0], t[2], t[3], lambda k: _moffat_k(b, k * rd),
                     N, Nk, s, s, t[4] - shift, t[5] - shift, dev).reshape(-1)
        img.backward(cot[at:at + s * s])
        at += s * s
        images.append(img.detach())
    return {'image': torch.cat(images), 'grad': [th.grad[:, k] for k in range(th.shape[1])]}


def exact(case, seed):
    kind = case['kind']
    dev = 'cuda' if torch.cuda.is_available() else 'cpu'
    if kind in ('bulge_disk', 'sersic'):
        # a Sersic's transform is the framework's own table by definition (as in GalSim):
        # there is no value of it to 64 bits apart from the table
        return None
    if kind == 'draw':
        p = _draw_params(case, seed)
        nx, ny = case['nx'], case['ny']
        N, Nk, ux, uy = _grid(p['hlr'], math.hypot(p['g1'], p['g2']),
                              _moffat_sizes(p['fwhm'], p['beta']), nx, ny, *p['offset'])
        rd = _moffat_rd(p['fwhm'], p['beta'])
        return _image(p['hlr'], p['flux'], p['g1'], p['g2'],
                      lambda k: _moffat_k(p['beta'], k * rd), N, Nk, nx, ny, ux, uy,
                      dev).cpu().numpy()
    if kind == 'real':
        return _exact_real(case, seed)
    if kind in ('kolm', 'moffat'):
        n = case['n']
        p = _gal_params(n, seed, 3)
        nx, ny = _sides(case) if kind == 'kolm' else ([case['side']] * n,) * 2
        grids = []
        for i in range(n):
            sizes = (_kolm_sizes(p['fwhm'][i]) if kind == 'kolm' else
                     _moffat_sizes(p['fwhm'][i], 3.))
            grids.append(_grid(p['hlr'][i], math.hypot(p['g1'][i], p['g2'][i]), sizes,
                               int(nx[i]), int(ny[i]), p['dx'][i], p['dy'][i]))
        out = []
        for i in np.argsort([gr[0] for gr in grids], kind='stable'):
            N, Nk, ux, uy = grids[i]
            if kind == 'kolm':
                k0 = KOLM_K0 * KOLM_FWHM / p['fwhm'][i]

                def psf(k):
                    return torch.exp(-(k / k0) ** (5. / 3.))
            else:
                rd = _moffat_rd(p['fwhm'][i], 3.)

                def psf(k):
                    return _moffat_k(3., k * rd)
            out.append(_image(p['hlr'][i], p['flux'][i], p['g1'][i], p['g2'][i], psf, N, Nk,
                              int(nx[i]), int(ny[i]), ux, uy, dev).reshape(-1))
        return torch.cat(out)
    if kind == 'grad':
        return _exact_grad(case, seed)
    a = _fft_input(case, seed).numpy()
    if kind == 'rfft':
        k = np.fft.fftshift(np.fft.rfft2(a), axes=(0,))
        return {'k': torch.from_numpy(k), 'x': torch.from_numpy(a)}
    return {'fwd': torch.from_numpy(np.fft.fftshift(np.fft.fft2(np.fft.fftshift(a)))),
            'inv': torch.from_numpy(np.fft.fftshift(np.fft.ifft2(a)))}
