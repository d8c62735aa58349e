"""Benchmark: batched FP32 drawImage(method='fft') of 4096 bulge+disk galaxies (Exponential disk +
Sersic bulge, sheared, convolved with Kolmogorov, pixel-integrated, 0.2"/px, stamps 48..256 px)
on one MI355X, against the plain per-stamp FP64 GPU path and the CPU oracle.

python bench.py [--gpus 1] [--steps K] [--warmup W] [--n 4096] [--cpu-seconds 15]
Prints one JSON line on stdout; progress goes to stderr.
"""
import argparse
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = ("stamps/s fwd & fwd+bwd, batched FP32 vs plain FP64 GPU at <=1e-5 peak-rel err")
HBM_PEAK_GBS = 8000.
FP32_PEAK_TFLOPS = 157.3          # MI355X vector FP32, counting packed (two-per-lane) FMAs
FP32_NONPACKED_TFLOPS = 78.6      # the same without packed FP32, which this build leaves out


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def kernel_flops(rec):
    """Algorithmic FLOPs per stamp for the two kernels: k-space products (8 per factor per
    half-plane sample of the Nk grid) + column inverse DFTs (5 N log2 N per column) for the fold
    kernel; half-length complex DFT per output row (5 (N/2) log2(N/2)) plus the real-split
    (~10 per element) for the row kernel."""
    N, Nk, ny, nfac = rec
    fold = 8. * nfac * Nk * (Nk / 2 + 1) + 5. * N * math.log2(N) * (N / 2 + 1)
    rows = ny * (5. * (N / 2) * math.log2(N / 2) + 10. * (N / 2))
    return fold, rows


def kernel_bytes(rec, nx, fsize):
    """Algorithmic HBM bytes per stamp: the fold kernel writes ny (N/2+1) complex rows of the
    column transform; the row kernel reads them and writes nx ny pixels."""
    N, Nk, ny, nfac = rec
    col = ny * (N / 2 + 1) * 2 * fsize
    return col + 64, col + nx * ny * fsize


def fwd_bwd_bench(args, torch):
    """Forward+backward of the chi^2 fit workload: 1024 Exponential x Moffat(beta=3) stamps of
    64x64, FP32, noisy targets (sigma = 1% of each stamp's peak), gradient with respect to
    (flux, hlr, g1, g2, dx, dy, psf_fwhm) through the adjoint kernels.  Also the same step on
    the plain per-stamp FP64 GPU path (one stamp per launch sequence), and the FP32 gradients
    against the FP64 ones."""
    from galsim_amd import diff, workloads
    n = args.fit_n
    p = workloads.exp_moffat_params(n, seed=args.seed + 1)
    theta = np.stack([p['flux'], p['hlr'], p['g1'], p['g2'], p['offset'][:, 0],
                      p['offset'][:, 1], p['psf_fwhm']], axis=1)
    t_true = torch.tensor(theta, dtype=torch.float64, device='cuda')
    rng = np.random.default_rng(args.seed + 2)
    t_fit = t_true * torch.tensor(1. + 0.02 * rng.standard_normal(theta.shape),
                                  dtype=torch.float64, device='cuda')

    def setup(prec, rows):
        model = diff.ExpMoffat(theta[rows], 64, 64, scale=0.2, beta=3.0, precision=prec)
        with torch.no_grad():
            img = model.render(t_true[rows]).double()
        sig = torch.empty_like(img)
        gen = torch.Generator(device='cpu').manual_seed(args.seed + 3)
        noise = torch.randn(img.shape, generator=gen, dtype=torch.float64).cuda()
        for s_img, s_sig in zip(model.dplan.stamps(img), model.dplan.stamps(sig)):
            s_sig.fill_(0.01 * float(s_img.abs().max()))
        target = (img + sig * noise).to(img.dtype)
        return model, target, 1. / sig

    def step(model, t, target, isig):
        t = t.detach().requires_grad_(True)
        r = (model.render(t).double() - target) * isig
        (r * r).sum().backward()
        return t.grad

    rows = np.arange(n)
    m32, tg32, is32 = setup('f32', rows)
    for _ in range(args.warmup):
        step(m32, t_fit, tg32, is32)
    torch.cuda.synchronize()
    k = max(args.steps, 1)
    t0 = time.perf_counter()
    for _ in range(k):
        g32 = step(m32, t_fit, tg32, is32)
    torch.cuda.synchronize()
    ms = 1e3 * (time.perf_counter() - t0) / k
    with torch.no_grad():
        for _ in range(2):
            m32.render(t_fit)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(k):
            m32.render(t_fit)
        torch.cuda.synchronize()
        ms_fwd = 1e3 * (time.perf_counter() - t0) / k
    log("fwd+bwd FP32 eager (%d stamps): %.3f ms/step (forward alone %.3f ms)"
        % (n, ms, ms_fwd))
    # the same step captured in one HIP graph (the chi^2 gradient fed straight to backward, so no
    # reduction enters the graph) and replayed
    tg = t_fit.detach().clone().requires_grad_(True)
    w2 = 2. * is32 * is32

    def body():
        if tg.grad is not None:
            tg.grad.zero_()
        img = m32.render(tg)
        torch.autograd.backward(img, grad_tensors=((img.double() - tg32) * w2).to(img.dtype))

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            body()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        body()
    settle(graph.replay, torch)
    t0 = time.perf_counter()
    for _ in range(k):
        graph.replay()
    torch.cuda.synchronize()
    ms_graph = 1e3 * (time.perf_counter() - t0) / k
    graph_err = float(((tg.grad - g32).abs() / g32.abs().clamp(min=1e-30)).max())
    rate = n / (ms_graph * 1e-3)
    log("fwd+bwd FP32 graph: %.3f ms/step, %.0f stamps/s (graph vs eager gradient rel diff "
        "%.1e)" % (ms_graph, rate, graph_err))
    # FP64 batched gradients for the accuracy figure
    m64, tg64, is64 = setup('f64', rows)
    g64 = step(m64, t_fit, tg64, is64)
    scale = (g64.abs() * t_fit.abs().clamp(min=1.)).max(dim=1, keepdim=True).values
    err = ((g32 - g64).abs() * t_fit.abs().clamp(min=1.) / scale).max().item()
    log("FP32 vs FP64 gradient: max error / largest sensitivity = %.2e" % err)
    # the adjoint alone: J^T v for one cotangent v in both precisions (the FP64 chi^2 cotangent at
    # t_fit).  The chi^2 gradient above also carries each precision's own forward image through
    # residuals 100x smaller than the peak, which magnifies the FP32 image error 100-fold.
    with torch.no_grad():
        img64 = m64.render(t_fit).double()
        cot = 2. * (img64 - tg64) * is64 * is64

    def vjp(model):
        t = t_fit.detach().requires_grad_(True)
        img = model.render(t)
        (g,) = torch.autograd.grad(img, t, grad_outputs=cot.to(img.dtype))
        return g

    j32, j64 = vjp(m32), vjp(m64)
    scale_j = (j64.abs() * t_fit.abs().clamp(min=1.)).max(dim=1, keepdim=True).values
    err_adj = ((j32 - j64).abs() * t_fit.abs().clamp(min=1.) / scale_j).max().item()
    log("FP32 vs FP64 adjoint (same cotangent): max error / largest sensitivity = %.2e" % err_adj)
    # plain per-stamp FP64 path
    mp = min(args.plain_sample, n, 64)
    singles = [setup('f64', np.array([i])) for i in range(mp)]
    for i in range(min(4, mp)):
        step(singles[i][0], t_fit[i:i + 1], singles[i][1], singles[i][2])
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i, (mm, tg, isg) in enumerate(singles):
        step(mm, t_fit[i:i + 1], tg, isg)
    torch.cuda.synchronize()
    plain = mp / (time.perf_counter() - t0)
    log("plain FP64 per-stamp fwd+bwd: %.0f stamps/s (%d stamps)" % (plain, mp))
    return {"value": round(rate, 1), "unit": "stamps/s", "ms_per_step": round(ms_graph, 4),
            "eager_ms_per_step": round(ms, 4), "forward_ms_per_step": round(ms_fwd, 4),
            "graph_vs_eager_grad_rel_diff": graph_err,
            "workload": "%d Exponential x Moffat(beta=3) 64x64 stamps, FP32, chi^2 against "
                        "noisy targets (sigma = 1%% of peak), gradient w.r.t. flux, hlr, g1, g2, "
                        "dx, dy, psf_fwhm via the adjoint kernels" % n,
            "plain_fp64_gpu_fwd_bwd_stamps_per_s": round(plain, 1),
            "speedup_vs_plain_fp64_gpu": round(rate / plain, 2),
            "grad_err_fp32_vs_fp64": err,
            "adjoint_err_fp32_vs_fp64_same_cotangent": err_adj,
            "grad_err_note": "errors are max |g32 - g64| |theta| over the stamp's largest "
                             "|g64| |theta|; grad_err compares the chi^2 gradients (each "
                             "precision with its own targets and forward image), "
                             "adjoint_err feeds one FP64 chi^2 cotangent to both adjoints"}


def fit_bench(args, torch):
    """The batched fit workload: 8192 Exponential x Moffat stamps with sides in {32, 48, 64, 96,
    128}, beta ~ U(2.5, 4.5), noisy targets at S/N ~ U(20, 200); 50 Adam steps on (flux, hlr,
    g1, g2, dx, dy, psf_fwhm, beta), each step one HIP graph launch.
    Reports fit throughput, peak device memory, and the parameters against the same fit run
    with the FP64 kernels on a subset."""
    from galsim_amd import fit
    n = args.fit_batch
    steps = 50
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base_mem = torch.cuda.memory_allocated()
    t0 = time.perf_counter()
    model, theta, init, target, isig, scale, betas, sides = fit.exp_moffat_fit_problem(
        n, seed=args.seed + 7, precision='f32')
    f = fit.BatchFit(model, init, target, isig, scale)
    f.capture()
    t_setup = time.perf_counter() - t0
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    f.replay(steps)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    peak = torch.cuda.max_memory_allocated() - base_mem
    rate = n / wall
    est32 = f.theta.cpu().numpy()
    chi = (f.chi2().cpu().numpy() / sides.astype(float) ** 2)
    log("fit: %d stamps x %d Adam steps in %.3f s (%.1f ms/step) -> %.0f stamps/s; peak "
        "device memory %.2f GB; median chi2/pixel %.3f" % (n, steps, wall, 1e3 * wall / steps,
                                                           rate, peak / 1e9, np.median(chi)))
    # the same fit with the FP64 kernels on a subset (graph replays as well)
    m = min(n, args.fit_compare)
    sub = fit.exp_moffat_fit_problem(m, seed=args.seed + 7, precision='f64')
    f64 = fit.BatchFit(sub[0], sub[2], sub[3], sub[4], sub[5])
    f64.capture()
    f64.replay(steps)
    torch.cuda.synchronize()
    est64 = f64.theta.cpu().numpy()
    sub32 = fit.exp_moffat_fit_problem(m, seed=args.seed + 7, precision='f32')
    f32 = fit.BatchFit(sub32[0], sub32[2], sub32[3], sub32[4], sub32[5])
    f32.capture()
    f32.replay(steps)
    torch.cuda.synchronize()
    d = np.abs(f32.theta.cpu().numpy() - est64) / scale
    err_truth = np.abs(est32 - theta) / scale
    log("fit FP32 vs FP64 (%d stamps): max |diff| / scale per parameter %s" % (
        m, np.round(d.max(axis=0), 6)))
    return {"value": round(rate, 1), "unit": "stamps/s (50 Adam steps each)",
            "n_stamps": n, "adam_steps": steps, "ms_per_step": round(1e3 * wall / steps, 3),
            "setup_s": round(t_setup, 2), "peak_device_memory_GB": round(peak / 1e9, 3),
            "median_chi2_per_pixel": round(float(np.median(chi)), 4),
            "param_diff_fp32_vs_fp64_fit_max_over_scale": {
                k: float(v) for k, v in zip(('flux', 'hlr', 'g1', 'g2', 'dx', 'dy', 'psf_fwhm',
                                             'beta'), d.max(axis=0))},
            "param_scale": scale.tolist(),
            "median_abs_error_vs_truth_over_scale": float(np.median(err_truth)),
            "workload": "%d Exponential x Moffat(beta ~ U(2.5, 4.5)) stamps, sides in {32, 48, "
                        "64, 96, 128}, FP32, S/N ~ U(20, 200); 8 parameters fitted (flux, hlr, "
                        "g1, g2, dx, dy, psf_fwhm, beta)" % n}


def large_bench(args, torch):
    """Large stamps: 64 Sersic galaxies (n ~ U(3, 6) in steps of 0.05, hlr ~ U(2, 6)") under
    Kolmogorov(0.8") at drawImage's own stamp sizes, FP32 batched (FFT grids of 512 to 4096),
    with the error of every stamp whose grid the FP64 kernels take (N <= 2048) against them."""
    from galsim_amd import workloads
    from galsim_amd.batch import BatchPlan
    n = args.large_n
    t0 = time.perf_counter()
    profs, nx, ny, offs, p = workloads.build('large_sersic', n, seed=args.seed + 11)
    plan = BatchPlan(profs, nx, ny, 0.2, offs, precision='f32')
    plan.autotune(reps=2)
    plan.capture()
    t_setup = time.perf_counter() - t0
    settle(plan.replay, torch)
    k = 5
    t0 = time.perf_counter()
    for _ in range(k):
        plan.replay()
    torch.cuda.synchronize()
    ms = 1e3 * (time.perf_counter() - t0) / k
    Ns = np.empty(n, dtype=int)
    Ns[plan.order] = plan.recs['N']
    # every stamp against the FP64 kernels (the FP64 work lists take these grids in one
    # workgroup's LDS; otherwise each stamp draws through the FP64 per-stamp path)
    try:
        plan64 = BatchPlan(profs, nx, ny, 0.2, offs, precision='f64')
        plan64.run()
        torch.cuda.synchronize()
        ref64 = [plan64.stamp(i) for i in range(n)]
    except Exception:                                          # noqa: BLE001
        ref64 = []
        for i in range(n):
            im = profs[i].drawImage(nx=int(nx[i]), ny=int(ny[i]), scale=0.2, dtype=np.float64,
                                    precision='f64')
            ref64.append(torch.from_numpy(im.array).cuda())
    errs = []
    for i in range(n):
        a = plan.stamp(i).double()
        b = ref64[i]
        errs.append(float((a - b).abs().max() / b.abs().max()))
    # a sample against the FP64 oracle (numpy), for the FP32 batch and the FP64 kernels both
    from oracle import draw as od
    sample = [int(i) for i in np.argsort(Ns)[::max(1, n // max(args.large_oracle, 1))]]
    sample = sample[:args.large_oracle]
    orc = []
    for i in sample:
        ref = workloads.large_sersic_profile(od, p, i).drawImage(int(nx[i]), int(ny[i]),
                                                                 scale=0.2)
        a = plan.stamp(i).double().cpu().numpy()
        b = ref64[i].cpu().numpy()
        orc.append({"stamp": i, "N": int(Ns[i]),
                    "fp32_vs_oracle": float(np.max(np.abs(a - ref)) / np.max(np.abs(ref))),
                    "fp64_vs_oracle": float(np.max(np.abs(b - ref)) / np.max(np.abs(ref)))})
    # the same galaxies on stamps of 1024^2 (grids drawImage sizes at 1024 or less) or 2048^2
    # (the rest), so the FFT grids are the 1024 and 2048 the configuration names wherever the
    # profile allows (drawImage keeps a larger grid where the profile needs one)
    sides = np.where(Ns <= 1024, 1024, 2048)
    plan_p = BatchPlan(profs, sides, sides, 0.2, offs, precision='f32')
    plan_p.autotune(reps=1)
    plan_p.capture()
    settle(plan_p.replay, torch)
    t0 = time.perf_counter()
    for _ in range(3):
        plan_p.replay()
    torch.cuda.synchronize()
    ms_p = 1e3 * (time.perf_counter() - t0) / 3
    Np = np.empty(n, dtype=int)
    Np[plan_p.order] = plan_p.recs['N']
    errs_p = []
    for i in range(n):
        b = torch.from_numpy(profs[i].drawImage(nx=int(sides[i]), ny=int(sides[i]), scale=0.2,
                                                offset=tuple(offs[i]), dtype=np.float64,
                                                precision='f64').array).cuda()
        a = plan_p.stamp(i).double()
        errs_p.append(float((a - b).abs().max() / b.abs().max()))
    pinned = {"value": round(n / (ms_p * 1e-3), 1), "unit": "stamps/s",
              "ms_per_step": round(ms_p, 3),
              "fft_sizes": {str(a): b for a, b in plan_p.fft_sizes().items()},
              "stamp_sides": {"1024": int((sides == 1024).sum()),
                              "2048": int((sides == 2048).sum())},
              "peak_rel_err_fp32_vs_fp64_drawimage": {"max": max(errs_p),
                                                      "median": float(np.median(errs_p)),
                                                      "stamps_compared": n}}
    log("large Sersic on 1024^2 / 2048^2 stamps: %.2f ms (%.0f stamps/s), FFT sizes %s; FP32 vs "
        "FP64 drawImage over all %d stamps: max %.2e" % (ms_p, n / (ms_p * 1e-3),
                                                        plan_p.fft_sizes(), n, max(errs_p)))
    del plan_p
    log("large Sersic: %d stamps FP32 in %.2f ms (%.0f stamps/s), FFT sizes %s; FP32 vs FP64 "
        "peak-rel error over all %d stamps: max %.2e; vs the oracle on %d stamps: FP32 max "
        "%.2e, FP64 max %.2e" % (n, ms, n / (ms * 1e-3), plan.fft_sizes(), n, max(errs),
                                 len(orc), max([o['fp32_vs_oracle'] for o in orc] or [0.]),
                                 max([o['fp64_vs_oracle'] for o in orc] or [0.])))
    return {"value": round(n / (ms * 1e-3), 1), "unit": "stamps/s", "ms_per_step": round(ms, 3),
            "n_stamps": n, "fft_sizes": {str(a): b for a, b in plan.fft_sizes().items()},
            "setup_s": round(t_setup, 2),
            "peak_rel_err_fp32_vs_fp64": {"max": max(errs), "median": float(np.median(errs)),
                                          "stamps_compared": n,
                                          "per_stamp": [round(e, 10) for e in errs],
                                          "N_per_stamp": [int(v) for v in Ns]},
            "vs_fp64_oracle_sample": orc,
            "pinned_grids": pinned,
            "workload": "Sersic n ~ U(3, 6) step 0.05, hlr ~ U(2, 6) arcsec, x Kolmogorov "
                        "0.8 arcsec x Pixel, FP32; FFT grids are drawImage's own sizes for these "
                        "profiles (listed in fft_sizes); pinned_grids draws the same galaxies on "
                        "1024^2 / 2048^2 stamps so the grids are the 1024 and 2048 the "
                        "configuration names (3072 where a profile needs more)"}


def _config0_cpu_worker(job):
    """One CPU process of the multi-core baseline: oracle drawImage of stamps i0, i0 + step, ...
    of the 256-stamp Exponential x Moffat workload until the time budget is spent."""
    i0, step, n, seed, seconds = job
    os.environ['OMP_NUM_THREADS'] = '1'
    from galsim_amd import workloads
    from oracle import draw as od
    p = workloads.exp_moffat_params(n, seed)
    workloads.exp_moffat_profile(od, p, i0).drawImage(64, 64, scale=0.2)    # warm caches
    done = 0
    t0 = time.perf_counter()
    i = i0
    while time.perf_counter() - t0 < seconds:
        workloads.exp_moffat_profile(od, p, i % n).drawImage(
            64, 64, scale=0.2, offset=tuple(p['offset'][i % n]))
        done += 1
        i += step
    return done, time.perf_counter() - t0


def config0_bench(args, torch):
    """The reference's CPU-runnable case: 256 seeded Exponential x Moffat(beta=3, fwhm=0.7")
    stamps of 64x64 at 0.2"/px, FP64.  The plain per-stamp GPU path (one stamp per launch
    sequence, pre-planned), the batched FP64 path (work lists replayed from a HIP graph), the
    error of both against the oracle, and the oracle on 1 core and on the host's cores (one
    process per core, up to 16)."""
    from galsim_amd import workloads
    from galsim_amd.batch import BatchPlan
    from oracle import draw as od
    n = 256
    profs, nx, ny, offs, p = workloads.build('exp_moffat', n, seed=args.seed + 5)
    singles = [BatchPlan([profs[i]], nx[i:i + 1], ny[i:i + 1], 0.2, offs[i:i + 1],
                         precision='f64') for i in range(n)]
    for s_ in singles[:8]:
        s_.run()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for s_ in singles:
        s_.run()
    torch.cuda.synchronize()
    plain = n / (time.perf_counter() - t0)
    plan = BatchPlan(profs, nx, ny, 0.2, offs, precision='f64')
    plan.autotune(reps=2)
    plan.capture()
    settle(plan.replay, torch)
    k = 20
    t0 = time.perf_counter()
    for _ in range(k):
        plan.replay()
    torch.cuda.synchronize()
    ms = 1e3 * (time.perf_counter() - t0) / k
    worst = 0.
    for i in range(0, n, 16):
        ref = workloads.exp_moffat_profile(od, p, i).drawImage(64, 64, scale=0.2,
                                                               offset=tuple(offs[i]))
        a = plan.stamp(i).cpu().numpy()
        b = singles[i].stamp(0).cpu().numpy()
        worst = max(worst, float(np.max(np.abs(a - ref)) / np.max(np.abs(ref))),
                    float(np.max(np.abs(b - ref)) / np.max(np.abs(ref))))
    log("config0 (256 Exp x Moffat 64x64 FP64): plain per-stamp %.0f stamps/s, batched %.3f ms "
        "(%.0f stamps/s); max peak-rel error vs oracle %.2e" % (plain, ms, n / (ms * 1e-3),
                                                               worst))
    out = {"workload": "256 Exponential x Moffat(beta=3, fwhm=0.7) 64x64 stamps, 0.2 arcsec/px, "
                       "FP64, seeded hlr/shear/offset",
           "plain_fp64_gpu_stamps_per_s": round(plain, 1),
           "batched_fp64_gpu_stamps_per_s": round(n / (ms * 1e-3), 1),
           "batched_fp64_ms_per_step": round(ms, 4),
           "max_peak_rel_err_vs_oracle": worst}
    if not args.no_cpu:
        import multiprocessing as mp
        secs = max(args.cpu_seconds / 2., 2.)
        d1, t1 = _config0_cpu_worker((0, 1, n, args.seed + 5, secs))
        cores = max(1, min(16, os.cpu_count() or 1))
        ctx = mp.get_context('spawn')
        with ctx.Pool(cores) as pool:
            res = pool.map(_config0_cpu_worker,
                           [(c, cores, n, args.seed + 5, secs) for c in range(cores)])
        multi = sum(d for d, _ in res) / max(t for _, t in res)
        log("config0 CPU oracle: %.1f stamps/s on 1 core, %.1f on %d processes"
            % (d1 / t1, multi, cores))
        out["cpu_oracle_1_core_stamps_per_s"] = round(d1 / t1, 2)
        out["cpu_oracle_multicore_stamps_per_s"] = round(multi, 2)
        out["cpu_oracle_processes"] = cores
    return out


def settle(fn, torch, ms=30.):
    """Run fn (at least twice) until about ``ms`` ms of wall time have passed: after host-side
    set-up the GPU's clocks take ~25 ms of work to settle, and a short timed region right after
    an idle gap reads several % slow."""
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    n = 0
    while n < 2 or (time.perf_counter() - t0) * 1e3 < ms:
        fn()
        torch.cuda.synchronize()
        n += 1


def fft_module_bench(args, torch):
    """galsim_amd.fft on device-resident float64 images: rfft2 then irfft2 (shift_in and
    shift_out, as Image.calculate_fft / calculate_inverse_fft use them) for square sizes, timed
    with HIP events on the current stream.  Algorithmic bytes per pair: rfft2 reads 8 M N and
    writes 16 M (N/2 + 1); irfft2 reads 16 M (N/2 + 1) and writes 8 M N."""
    from galsim_amd import fft as gfft
    res = {}
    for N in (1174, 1536, 2048, 3072, 4096):
        x = torch.randn((N, N), dtype=torch.float64, device='cuda')
        for _ in range(args.fft_warmup):
            gfft.irfft2(gfft.rfft2(x, True, True), True, True)
        settle(lambda: gfft.irfft2(gfft.rfft2(x, True, True), True, True), torch)
        k = args.fft_pairs
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(k):
            y = gfft.irfft2(gfft.rfft2(x, True, True), True, True)
        e1.record()
        torch.cuda.synchronize()
        ms = e0.elapsed_time(e1) / k
        err = float((y - x).abs().max() / x.abs().max())
        W = N // 2 + 1
        nbytes = 2 * (8 * N * N + 16 * N * W)
        res[str(N)] = {"ms_per_pair": round(ms, 4), "algorithmic_GB_per_s":
                       round(nbytes / (ms * 1e-3) / 1e9, 1), "round_trip_err": err}
        log("fft module %dx%d: rfft2+irfft2 %.3f ms (%.0f GB/s algorithmic), round trip %.1e"
            % (N, N, ms, nbytes / (ms * 1e-3) / 1e9, err))
    return res


def real_space_bench(args, torch):
    """Real-space drawing (drawImage method='no_pixel' of analytic profiles): the pixel fill
    kernel on a device-resident 4096 x 4096 FP64 image of a sheared bulge + disk (Sersic n = 4
    + Exponential), timed with HIP events on the current stream; algorithmic bytes 8 per pixel
    (written once, nothing read).  Also the per-call time of drawImage for a 64 x 64 stamp and
    the oracle's fill of a 256 x 256 image on one core."""
    import galsim_amd as g
    from galsim_amd import real, _lib
    from galsim_amd.position import BoundsI
    from galsim_amd.transform import _Transform
    from oracle import draw as od, xdraw as ox

    def bulge_disk(m):
        return m.Add(m.Sersic(4., half_light_radius=0.6, flux=0.4).shear(g1=0.05, g2=0.1),
                     m.Exponential(half_light_radius=1.2, flux=0.6).shear(g1=0.3, g2=-0.1))
    scale = 0.2
    N = 4096
    prof = _Transform(bulge_disk(g), np.array([[1. / scale, 0.], [0., 1. / scale]]),
                      (0.3, -0.2), scale ** 2)
    b = BoundsI(-N // 2, N // 2 - 1, -N // 2, N // 2 - 1)
    recs = np.ascontiguousarray(real.components(prof, b, 1.))
    out = torch.empty((N, N), dtype=torch.float64, device='cuda')
    stream = torch.cuda.current_stream().cuda_stream
    L = _lib.lib()

    def fill():
        _lib.check(L.gsmi_draw_real_f64(recs.ctypes.data, len(recs), None, N, N, 0,
                                        out.data_ptr(), stream), "gsmi_draw_real_f64")
    settle(fill, torch)
    k = 20
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(k):
        fill()
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / k
    gbps = 8. * N * N / (ms * 1e-3) / 1e9
    flux = float(out.sum()) * 1.
    # drawImage per call, 64 x 64 stamps
    obj = bulge_disk(g)
    for _ in range(5):
        obj.drawImage(nx=64, ny=64, scale=scale, method='no_pixel')
    t0 = time.perf_counter()
    calls = 200
    for _ in range(calls):
        obj.drawImage(nx=64, ny=64, scale=scale, method='no_pixel')
    per_call_us = (time.perf_counter() - t0) / calls * 1e6
    # the oracle on one core
    oobj = bulge_disk(od)
    t0 = time.perf_counter()
    reps = 0
    while reps < 3 or time.perf_counter() - t0 < 2.:
        ox.draw_image_sb(oobj, -128, 127, -128, 127, scale, method='no_pixel',
                         offset=(0.3, -0.2))
        reps += 1
    cpu_px = reps * 256 * 256 / (time.perf_counter() - t0)
    log("real-space fill 4096^2 bulge+disk FP64: %.3f ms (%.2e pixels/s, %.0f GB/s written, "
        "flux %.6f); drawImage no_pixel 64^2 %.0f us/call; oracle %.2e pixels/s on 1 core"
        % (ms, N * N / (ms * 1e-3), gbps, flux, per_call_us, cpu_px))
    return {"workload": "sheared Sersic(n=4) + Exponential, 4096 x 4096 FP64 image, 0.2 "
                        "arcsec/px, method='no_pixel'",
            "fill_ms": round(ms, 4), "pixels_per_s": round(N * N / (ms * 1e-3), 1),
            "roofline": {"bound": "hbm", "achieved": round(gbps, 1), "peak": 8000.,
                         "unit": "GB/s", "frac": round(gbps / 8000., 4),
                         "algorithmic_bytes_per_launch": 8 * N * N},
            "image_flux": flux,
            "drawimage_64x64_us_per_call": round(per_call_us, 1),
            "cpu_oracle_pixels_per_s_1_core": round(cpu_px, 1)}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument('--gpus', type=int, default=1)
    ap.add_argument('--steps', type=int, default=50)
    # after the host-side set-up (planning, tuning, graph capture) the GPU's clocks take about
    # 25 ms of work to settle: the first steps after an idle gap run ~8% slower
    ap.add_argument('--warmup', type=int, default=40)
    ap.add_argument('--n', type=int, default=4096)
    ap.add_argument('--seed', type=int, default=0)
    ap.add_argument('--plain-sample', type=int, default=256)
    ap.add_argument('--cpu-seconds', type=float, default=15.)
    ap.add_argument('--no-cpu', action='store_true')
    ap.add_argument('--fit-n', type=int, default=1024)
    ap.add_argument('--no-fit', action='store_true')
    ap.add_argument('--fit-batch', type=int, default=8192)
    ap.add_argument('--fit-compare', type=int, default=256)
    ap.add_argument('--no-batch-fit', action='store_true')
    ap.add_argument('--large-n', type=int, default=64)
    ap.add_argument('--no-large', action='store_true')
    ap.add_argument('--large-oracle', type=int, default=4,
                    help='stamps of the large-stamp workload checked against the numpy oracle')
    ap.add_argument('--no-fft-module', action='store_true')
    ap.add_argument('--fft-module-only', action='store_true',
                    help='only run the FFT-module leg (rfft2 + irfft2 of 1174^2, 1536^2, '
                         '2048^2, 3072^2 and 4096^2 float64 images) and exit')
    ap.add_argument('--fft-pairs', type=int, default=10)
    ap.add_argument('--fft-warmup', type=int, default=2)
    ap.add_argument('--no-real-space', action='store_true')
    ap.add_argument('--no-config0', action='store_true')
    ap.add_argument('--copy-calibration', type=int, default=0, metavar='MIB',
                    help='only run a plain device copy of MIB MiB (3 times) and exit; used to '
                         'scale the FETCH_SIZE/WRITE_SIZE counters')
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get('WORLD_SIZE', '1')) != 1:
        print("bench.py measures one GPU only: this build renders every stamp on a single "
              "MI355X (--gpus 1); stamps are independent, so more GPUs would shard the stamp "
              "list with no communication.", file=sys.stderr)
        sys.exit(2)

    import torch
    torch.cuda.set_device(0)
    if args.copy_calibration:
        n = args.copy_calibration * (1 << 20) // 4
        x = torch.ones(n, dtype=torch.float32, device='cuda')
        y = torch.empty_like(x)
        for _ in range(3):
            y.copy_(x)
        torch.cuda.synchronize()
        log("copied %d MiB three times" % args.copy_calibration)
        return
    if args.fft_module_only:
        fft_module_bench(args, torch)
        return
    import galsim_amd as g
    from galsim_amd import workloads
    from galsim_amd.batch import BatchPlan

    t0 = time.perf_counter()
    profs, nx, ny, offs, params = workloads.build('bulge_disk', args.n, seed=args.seed)
    t_build = time.perf_counter() - t0
    t0 = time.perf_counter()
    plan = BatchPlan(profs, nx, ny, 0.2, offs, precision='f32')
    t_plan = time.perf_counter() - t0
    log("workload: %d stamps, build %.2fs, plan %.2fs, FFT sizes %s" % (
        args.n, t_build, t_plan, plan.fft_sizes()))

    # --- the per-FFT-size launches (one fold + one row launch per size), event-timed --------
    evs = []

    def mk(kind, N):
        e = torch.cuda.Event(enable_timing=True)
        evs[-1].append((kind, N, e))
        return e

    def kernel_times(p, steps):
        del evs[:]
        for _ in range(2):
            p.run()
        torch.cuda.synchronize()
        for _ in range(steps):
            evs.append([])
            p.run(events=mk)
        torch.cuda.synchronize()
        fold, rows = {}, {}
        for step in evs:
            for k in range(len(step) - 1):
                kind, N, e = step[k]
                d = e.elapsed_time(step[k + 1][2])
                (fold if kind == 'fold' else rows).setdefault(N, []).append(d)
        return ({N: float(np.mean(v)) for N, v in fold.items()},
                {N: float(np.mean(v)) for N, v in rows.items()})

    bins_fold, bins_rows = kernel_times(plan, min(args.steps, 10))
    t_bins = sum(bins_fold.values()) + sum(bins_rows.values())
    log("per-size launches: fold %.3f ms + rows %.3f ms per step; fold per-N ms %s" % (
        sum(bins_fold.values()), sum(bins_rows.values()),
        {N: round(v, 4) for N, v in bins_fold.items()}))

    # --- work lists: every FFT size in one fold and one row launch, tiles and grid tuned on
    # this batch, the whole step captured in a HIP graph ---------------------------------------
    t0 = time.perf_counter()
    tuning = plan.autotune()
    t_tune = time.perf_counter() - t0
    log("autotune (%.1fs): cols %s chunks %s rows %s grid %s -> %.3f ms" % (
        t_tune, tuning['cols'], tuning['chunks'], tuning['rows'], tuning['grid'], tuning['ms']))
    fold_ms, rows_ms = kernel_times(plan, min(args.steps, 10))
    plan.capture()

    # --- timed region: K graph launches of the batched FP32 forward ---------------------------
    for _ in range(args.warmup):
        plan.replay()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        plan.replay()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    ms_per_step = 1e3 * wall / args.steps
    value = args.n / (wall / args.steps)
    log("batched FP32 (graph): %.3f ms/step, %.0f stamps/s" % (ms_per_step, value))
    recs = plan.recs
    nfac = {}
    flops = {'fold': 0., 'rows': 0.}
    for r in recs:
        rec = (int(r['N']), int(r['Nk']), int(r['ny']), r['op_count'])
        # factors: LEAF + PHASE + SCALE ops (each a complex multiply-accumulate per sample)
        f, rw = kernel_flops((rec[0], rec[1], rec[2], 5))
        flops['fold'] += f
        flops['rows'] += rw
    # the whole step: the kernels compiled per FFT size (one workgroup per stamp at N = 128 and
    # 192, which touches memory for its pixels only; columns and rows above), and the fold and
    # row work lists of any size they do not take
    t_fold = sum(fold_ms.values())
    t_rows = sum(rows_ms.values())
    t_dom = t_fold + t_rows
    in_lds = {g[0] for g in plan.stamp_groups}
    step_bytes = sum(4. * int(r['nx']) * int(r['ny']) if int(r['N']) in in_lds else
                     sum(kernel_bytes((int(r['N']), int(r['Nk']), int(r['ny']), 5), int(r['nx']),
                                      4)) for r in recs)
    n_launch = len(plan.stamp_groups) + (3 if plan.wide_groups else 0) + \
        (3 if plan.list_groups else 0)
    achieved = (flops['fold'] + flops['rows']) / (t_dom * 1e-3) / 1e12
    log("step: %.3f ms of kernels over %d launches" % (t_dom, n_launch))
    roofline = {
        "kernel": "draw_stamp_f32 + fold_cols + row_pixels (the whole step)",
        # vector ALU issue bounds the kernels (no matrix-core work on this path)
        "bound": "valu",
        "achieved": round(achieved, 4),
        "peak": FP32_PEAK_TFLOPS,
        "unit": "TFLOP/s",
        "frac": round(achieved / FP32_PEAK_TFLOPS, 6),
        "traffic": None,
        "algorithmic_bytes_per_step": step_bytes,
        "hbm_GBps_algorithmic": round(step_bytes / (t_dom * 1e-3) / 1e9, 2),
        "hbm_frac_algorithmic": round(step_bytes / (t_dom * 1e-3) / 1e9 / HBM_PEAK_GBS, 6),
        "avg_launch_ms": round(t_dom / max(n_launch, 1), 5),
        "launches_per_step": n_launch,
        "frac_of_nonpacked_fp32_peak": round(achieved / FP32_NONPACKED_TFLOPS, 6),
    }

    # --- config-driven planning (vectorised, galsim_amd.config) and end to end ---------------
    from galsim_amd import config as gcfg
    cfg = workloads.bulge_disk_config(params, nx)
    gcfg.plan_config(cfg, args.n, 'f32')                 # tables built once, outside timing
    t0 = time.perf_counter()
    hp = gcfg.plan_config(cfg, args.n, 'f32')
    t_plan_cfg = time.perf_counter() - t0
    same = bool(np.array_equal(hp.recs['N'], np.asarray(
        [plan.recs['N'][plan.rec_of[i]] for i in range(args.n)])))
    e2e = []
    for _ in range(3):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        hp = gcfg.plan_config(cfg, args.n, 'f32')
        cplan = BatchPlan(None, None, None, None, lowered=hp)
        cplan.use_schedule(tuning['cols'], tuning['rows'], tuning['grid'], tuning['grid'],
                           tuning['chunks'])
        cplan.run()
        torch.cuda.synchronize()
        e2e.append(time.perf_counter() - t0)
        del cplan
    e2e_rate = args.n / min(e2e)
    log("config-driven planning: %.1f ms for %d stamps (per-object planning %.0f ms); end to "
        "end (plan + upload + launch, output on the device) %.0f stamps/s; same FFT sizes: %s"
        % (1e3 * t_plan_cfg, args.n, 1e3 * t_plan, e2e_rate, same))

    # --- accuracy: FP32 batch against the FP64 kernels on every stamp -------------------------
    plan64 = BatchPlan(profs, nx, ny, 0.2, offs, precision='f64')
    plan64.run()
    torch.cuda.synchronize()
    worst = 0.
    for i in range(args.n):
        a = plan.stamp(i).double()
        b = plan64.stamp(i)
        worst = max(worst, float((a - b).abs().max() / b.abs().max()))
    log("max peak-relative error FP32 vs FP64 over %d stamps: %.3e" % (args.n, worst))

    # --- plain per-stamp FP64 GPU path (one stamp per launch, pre-planned) -------------------
    m = min(args.plain_sample, args.n)
    singles = [BatchPlan([profs[i]], nx[i:i + 1], ny[i:i + 1], 0.2, offs[i:i + 1],
                         precision='f64') for i in range(m)]
    for s in singles[:8]:
        s.run()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for s in singles:
        s.run()
    torch.cuda.synchronize()
    plain_rate = m / (time.perf_counter() - t0)
    log("plain FP64 per-stamp GPU path: %.0f stamps/s (%d stamps)" % (plain_rate, m))
    # end-to-end drawImage (host planning + one transfer + launches + copy back) per stamp
    m2 = min(64, args.n)
    t0 = time.perf_counter()
    for i in range(m2):
        profs[i].drawImage(nx=int(nx[i]), ny=int(ny[i]), scale=0.2, dtype=np.float64)
    drawimage_rate = m2 / (time.perf_counter() - t0)
    log("drawImage FP64 end to end: %.0f stamps/s" % drawimage_rate)

    fwd_bwd = None if args.no_fit else fwd_bwd_bench(args, torch)
    batch_fit = None if (args.no_fit or args.no_batch_fit) else fit_bench(args, torch)
    large = None if args.no_large else large_bench(args, torch)
    fft_mod = None if args.no_fft_module else fft_module_bench(args, torch)
    config0 = None if args.no_config0 else config0_bench(args, torch)
    real_space = None if args.no_real_space else real_space_bench(args, torch)

    # --- CPU baseline: the oracle's C++ restatement (oracle/cpu_draw.cpp), all cores and 1 ----
    cpu = None
    if not args.no_cpu:
        from oracle import cpu_port, draw as od
        cpu_port.build()
        oprofs = [workloads.bulge_disk_profile(od, params, i) for i in range(args.n)]
        t0 = time.perf_counter()
        cb = cpu_port.Batch(oprofs, nx, ny, 0.2, offs)       # sizes, leaf constants, tables
        t_cplan = time.perf_counter() - t0
        # the cores this process may run on (the GPU box gives one GPU's job 16)
        cores = max(1, min(16, len(os.sched_getaffinity(0))))
        cb.draw(cores)                                          # warm-up
        reps = []
        for _ in range(5):
            t0 = time.perf_counter()
            cb.draw(cores)
            reps.append(time.perf_counter() - t0)
        t_all = float(np.median(reps))
        # one core: a prefix of the same workload sized to about cpu_seconds / 3 per repeat
        t0 = time.perf_counter()
        cb.draw(1, 0, min(128, args.n))
        per = (time.perf_counter() - t0) / min(128, args.n)
        n1 = int(max(64, min(args.n, args.cpu_seconds / 3. / max(per, 1e-6))))
        reps1 = []
        for _ in range(3):
            t0 = time.perf_counter()
            cb.draw(1, 0, n1)
            reps1.append(time.perf_counter() - t0)
        t_one = float(np.median(reps1))
        # the port against the FP64 GPU kernels, every stamp
        port_err = 0.
        for i in range(args.n):
            ref = plan64.stamp(i).cpu().numpy()
            port_err = max(port_err, float(np.max(np.abs(cb.outs[i] - ref)) /
                                           np.max(np.abs(ref))))
        cpu = {"value": round(args.n / t_all, 1), "unit": "stamps/s", "cores": cores,
               "kind": "port",
               "sample": "all %d stamps of the same workload (same sizes and offsets), drawn by "
                         "the oracle's C++ restatement (oracle/cpu_draw.cpp: k fills, products, "
                         "phases, wrap, mixed-radix FFT, crop), one stamp per thread, median of "
                         "5 after a warm-up; host planning (%.1f s, sizes and Sersic tables from "
                         "the numpy oracle) excluded" % (args.n, t_cplan),
               "value_1_core": round(n1 / t_one, 1),
               "sample_1_core": "first %d stamps, median of 3" % n1,
               "port_vs_gpu_fp64_peak_rel_max": port_err}
        log("CPU baseline (C++ restatement): %.0f stamps/s on %d cores, %.0f on 1 core; max "
            "peak-rel vs the FP64 GPU kernels %.1e" % (args.n / t_all, cores, n1 / t_one,
                                                       port_err))

    out = {
        "metric": METRIC,
        "value": round(value, 1),
        "unit": "stamps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": "bulge+disk (Exponential + Sersic n in 1.5..4, sheared) x "
                               "Kolmogorov x Pixel, FP32, 0.2 arcsec/px",
                   "n_stamps": args.n, "stamp_sides": "48..256",
                   "fft_sizes": {str(k): v for k, v in plan.fft_sizes().items()},
                   "seed": args.seed},
        "roofline": roofline,
        "cpu_baseline": cpu,
        "fwd_bwd": fwd_bwd,
        "batch_fit": batch_fit,
        "large_stamps": large,
        "fft_module_f64": fft_mod,
        "real_space_f64": real_space,
        "config0_exp_moffat_fp64": config0,
        "plain_fp64_gpu_stamps_per_s": round(plain_rate, 1),
        "speedup_vs_plain_fp64_gpu": round(value / plain_rate, 2),
        "drawimage_fp64_end_to_end_stamps_per_s": round(drawimage_rate, 1),
        "max_peak_rel_err_fp32_vs_fp64": worst,
        "host_plan_s": round(t_plan, 3),
        "host_plan_config_s": round(t_plan_cfg, 4),
        "end_to_end_config_stamps_per_s": round(e2e_rate, 1),
        "end_to_end_note": "config-driven planning (vectorised) + one host-to-device copy of "
                           "the records + the tuned launches, output left on the device",
        "schedule": {"launches": "one launch per FFT size that a workgroup holds, an axis "
                                 "prepass, a column and a row launch for the others, replayed "
                                 "from one HIP graph",
                     "cols_per_group": {str(k): v for k, v in tuning['cols'].items()},
                     "rows_per_group": {str(k): v for k, v in tuning['rows'].items()},
                     "fold_chunks_per_item": {str(k): v for k, v in tuning['chunks'].items()},
                     "grid": tuning['grid'], "autotune_s": round(t_tune, 2),
                     "per_size_launches_ms_per_step": round(t_bins, 4),
                     "work_list_ms_per_step": round(t_fold + t_rows, 4)},
    }
    print(json.dumps(out), flush=True)


if __name__ == '__main__':
    main()
