// One-kernel drawing of small stamps in FP32: a workgroup draws a whole stamp, its wrapped
// N-grid held in LDS from the first k-space sample to the last pixel.
//
// The two-kernel path (gsmi_kernels.hip) carries every stamp's column transform through a scratch
// buffer in memory: 8 bytes written and read per wrapped cell against 4 bytes of output per
// pixel, and a second launch.  For N = 128 and 192 the N/2 packed columns of N values (64 and
// 147 KB) fit the 160 KB of LDS one workgroup may hold, so nothing but the pixels leaves the CU.
//
// Steps of a workgroup (barriers between them):
//   1. tables: leaf constants, the Sersic spline coefficients, the N twiddles, the axis factors
//      X(kx), kx = 0..Nk/2, and Y(ky), ky = 0..Nk/2 (Y(-ky) is its conjugate: the hoisted factors
//      are sincs, shifts and constants);
//   2. cells: samples are evaluated in pairs (kx, ky), (kx, -ky), which share the circular PSF's
//      value, the products X Y and most of the quadratic forms.  A thread keeps one ky for all
//      its columns.  Aliased samples (|kx| or |ky| beyond N/2) follow as their own compact
//      passes that add to the cells;
//   3. columns: the inverse DFT along ky, in place, as two passes of radix C1 and C2 with
//      C1 C2 = N; a value's final place is its digit-reversed index (row_slot);
//   4. rows: the real inverse DFT along x of the rows inside the output window, also in place in
//      two passes, the first forming E + i O from the packed columns and the second writing the
//      pixels.
//
// Bound: VALU issue (154 lane instructions per cell for a bulge + disk, samples and both
// transforms; 49 M wave instructions = 80 us of the 128 us of the N = 128 launch below), then the
// waits at the barriers; LDS is busy a third of the time.  Measured on 4096 bulge + disk stamps,
// whose N = 128 and 192 sizes took 483 us in the fold and row kernels: 128 us and 156 us.
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "../../include/gsmi.h"
#include "device_program.h"
#include "launch.h"
#include "stamp_cells.h"

namespace gsmi {
namespace {

// Radices, LDS geometry and workgroup size of each FFT size.  A column is L values apart from the
// next and holds element r at r + r / PADR: with these, the lanes of a half-wave fall on different
// banks (64-bit accesses, 32 slots) up to two or three of them, in every pass.  128: two
// workgroups of 8 waves per CU (LDS), 4 waves per SIMD; 192: one of 12 waves, 3 per SIMD.
template <int N>
struct Shape;
template <>
struct Shape<128> {
    static constexpr int C1 = 16, C2 = 8, R1 = 8, R2 = 8, L = 143, PADR = 8, T = 512, WAVES = 4;
};
template <>
struct Shape<192> {
    static constexpr int C1 = 16, C2 = 12, R1 = 8, R2 = 12, L = 197, PADR = 48, T = 768, WAVES = 3;
};

template <int N>
__device__ __forceinline__ constexpr int pad(int r)
{
    return r + r / Shape<N>::PADR;
}

// Place within its column of output row y of the column transform (before padding).
template <int N>
__device__ __forceinline__ constexpr int row_slot(int y)
{
    return (y % Shape<N>::C1) * Shape<N>::C2 + y / Shape<N>::C1;
}

// In-place inverse DFT of the H columns: radix C1 over elements C2 apart, the twiddle, then radix
// C2 over each run of C2 elements.
template <int N>
__device__ __forceinline__ void column_dft(cplx<float>* buf, const cplx<float>* tw)
{
    using S = Shape<N>;
    constexpr int H = N / 2, L = S::L, T = S::T, C1 = S::C1, C2 = S::C2;
    for (int t = threadIdx.x; t < H * C2; t += T) {
        const unsigned c = unsigned(t) / C2;
        const int b = t - int(c) * C2;
        cplx<float>* p = buf + c * L + b;
        cplx<float> v[C1];
        // element b + s C2 is s C2 + s C2 / PADR past b (C2 divides PADR, or PADR divides C2)
#pragma unroll
        for (int s = 0; s < C1; ++s) v[s] = p[s * C2 + s * C2 / S::PADR];
        bfly<C1>(v);
#pragma unroll
        for (int k = 1; k < C1; ++k) v[k] = cmul(v[k], tw[b * k]);
#pragma unroll
        for (int s = 0; s < C1; ++s) p[s * C2 + s * C2 / S::PADR] = v[s];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < H * C1; t += T) {
        const unsigned c = unsigned(t) / C1;
        const int k1 = t - int(c) * C1;
        cplx<float>* p = buf + c * L + pad<N>(k1 * C2);
        cplx<float> v[C2];
#pragma unroll
        for (int b = 0; b < C2; ++b) v[b] = p[b];
        bfly<C2>(v);
#pragma unroll
        for (int b = 0; b < C2; ++b) p[b] = v[b];
    }
    __syncthreads();
}

// Real inverse DFT along x of ny rows (window rows y0.. of the N-grid) and the pixels.
template <int N>
__device__ __forceinline__ void row_dft(cplx<float>* buf, const cplx<float>* tw, int x0, int y0,
                                        int nx, int ny, float* __restrict__ out, bool& bad)
{
    using S = Shape<N>;
    constexpr int M = N / 2, L = S::L, T = S::T, R1 = S::R1, R2 = S::R2;
    constexpr int U = R2 / 2;
    const float inv_ny = 1.f / float(ny);
    for (int t = threadIdx.x; t < ny * U; t += T) {
        const int u = fdiv(t, inv_ny);
        const int idx = t - u * ny;
        const int yy = y0 + idx < 0 ? y0 + idx + N : y0 + idx;
        cplx<float>* p = buf + pad<N>(row_slot<N>(yy));
        const int b0 = u, b1 = u ? R2 - u : R2 / 2;      // columns b + R2 s; unit 0: 0 and R2/2
        cplx<float> va[R1], vb[R1];
#pragma unroll
        for (int s = 0; s < R1; ++s) {
            va[s] = p[(b0 + R2 * s) * L];
            vb[s] = p[(b1 + R2 * s) * L];
        }
        c2r_inputs<R1, R2>(b0, [&](int c) { return tw[c]; }, va, vb);
        bfly<R1>(va);
        bfly<R1>(vb);
#pragma unroll
        for (int k = 1; k < R1; ++k) {
            va[k] = cmul(va[k], tw[2 * b0 * k]);
            vb[k] = cmul(vb[k], tw[2 * b1 * k]);
        }
#pragma unroll
        for (int s = 0; s < R1; ++s) {
            p[(b0 + R2 * s) * L] = va[s];
            p[(b1 + R2 * s) * L] = vb[s];
        }
    }
    __syncthreads();
    const float norm = 1.f / (float(N) * float(N));
    for (int t = threadIdx.x; t < ny * R1; t += T) {
        const int k1 = t % R1;
        const int idx = t / R1;
        const int yy = y0 + idx < 0 ? y0 + idx + N : y0 + idx;
        const cplx<float>* p = buf + pad<N>(row_slot<N>(yy)) + k1 * R2 * L;
        cplx<float> v[R2];
#pragma unroll
        for (int b = 0; b < R2; ++b) v[b] = p[b * L];
        bfly<R2>(v);
        // every output of a row's transform sums every input with a unit-modulus weight, so one
        // output per thread shows a non-finite value anywhere in the row's spectrum
        bad |= !isfinite(v[0].x + v[0].y);
        float* o = out + size_t(idx) * nx;
#pragma unroll
        for (int k2 = 0; k2 < R2; ++k2) {
            const int q = 2 * (k1 + R1 * k2);            // pixels q, q + 1 of the N-periodic row
            int col = q - x0;
            col = col >= N ? col - N : (col < 0 ? col + N : col);
            int col1 = col + 1;
            col1 = col1 >= N ? col1 - N : col1;
            if (col < nx) o[col] = v[k2].x * norm;
            if (col1 < nx) o[col1] = v[k2].y * norm;
        }
    }
}

// LDS of a stamp: its columns, the decoded leaves, the coefficients of its Sersic table (ncoef
// quadruples), the twiddles and the axis factors.
template <int N>
__host__ __device__ constexpr size_t stamp_lds(int ncoef, int hk)
{
    return sizeof(cplx<float>) * (size_t(N / 2) * Shape<N>::L + N + 2 * (hk + 1)) +
           sizeof(LeafC<float>) * kProgLeaves + 16 * size_t(ncoef);
}

// Grid: one workgroup per stamp (all of FFT size N and program shape SIG).  A stamp the launch
// cannot draw (another size or shape, a window off the grid, tables beyond its LDS) is left
// undrawn with its status flagged.
template <int N, int SIG>
__global__ void __launch_bounds__(Shape<N>::T, Shape<N>::WAVES)
draw_stamp_f32(gsmi_stamp* __restrict__ stamps, const gsmi_op* __restrict__ ops,
               const gsmi_leaf* __restrict__ leaves, Tables<float> tb, TwiddleSet<float> tws,
               int lds_bytes, float* __restrict__ out)
{
    using S = Shape<N>;
    constexpr int H = N / 2, T = S::T;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    gsmi_stamp* st = stamps + blockIdx.x;
    const int hk = st->Nk / 2;
    const gsmi_op* sops = ops + st->op_begin;
    const int nops = st->op_count;
    const gsmi_leaf* sleaves = leaves + st->leaf_begin;
    bool ok = matches_static<SIG>(sops, nops, sleaves);
    constexpr int ss = sersic_slot<SIG>();
    int ncoef = 0;
    if constexpr (ss >= 0)
        if (ok) {
            ncoef = sleaves[ss].ntab - 1;
            ok = sleaves[ss].cliprows >= 0 && ncoef >= 1;
        }
    const int x0 = st->x0, y0 = st->y0, nx = st->nx, ny = st->ny;
    if (!ok || st->N != N || hk < H || hk >= N || x0 < -H || x0 + nx > H || y0 < -H ||
        y0 + ny > H || stamp_lds<N>(ncoef, hk) > size_t(lds_bytes)) {
        if (threadIdx.x == 0) st->status = GSMI_STAMP_NONFINITE;
        return;
    }
    cplx<float>* buf = reinterpret_cast<cplx<float>*>(smem_raw);
    // 16-byte aligned: H L is even
    static_assert((H * S::L) % 2 == 0, "float4 alignment of the coefficients");
    float4* cfl = reinterpret_cast<float4*>(buf + H * S::L);
    LeafC<float>* lc = reinterpret_cast<LeafC<float>*>(cfl + ncoef);
    cplx<float>* tw = reinterpret_cast<cplx<float>*>(lc + kProgLeaves);
    cplx<float>* X = tw + N;
    cplx<float>* Y = X + hk + 1;
    const float dk = float(st->dk);
    {
        int stride;
        const cplx<float>* g = tws.pick(N, &stride);
        for (int e = threadIdx.x; e < N; e += T) tw[e] = g[e * stride];
        const gsmi_op* aops = sops + nops;
        for (int e = threadIdx.x; e < 2 * (hk + 1); e += T) {
            const bool xaxis = e <= hk;
            const int m = xaxis ? e : e - (hk + 1);
            X[e] = axis_factor<float>(aops, st->axis_count, sleaves, float(m) * dk, xaxis);
        }
    }
    StaticPair<SIG> pair;
    pair.dk = dk;
    pair.tb = tb;
    if (int(threadIdx.x) < kStaticPrograms[SIG].nl)
        lc[threadIdx.x] = leaf_consts_t<float>(sleaves[threadIdx.x], tb);
#pragma unroll
    for (int l = 0; l < kStaticPrograms[SIG].nl; ++l) pair.li[l] = leaf_ints(sleaves[l]);
    if constexpr (ss >= 0) {
        const float4* src = tb.coef + sleaves[ss].cliprows / 4;
        for (int e = threadIdx.x; e < ncoef; e += T) cfl[e] = src[e];
        pair.tb.coef = cfl;
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < kStaticPrograms[SIG].nl; ++l) pair.lr[l] = uniform_leaf(lc[l]);
    pair.even = pair.lr[kStaticPrograms[SIG].nl - 1].q1 == 0.f;
    fill_cells<N, S::L, T>(pair, [](int r) { return pad<N>(r); }, hk, X, Y, 0, H, buf);
    column_dft<N>(buf, tw);
    bool bad = false;
    row_dft<N>(buf, tw, x0, y0, nx, ny, out + st->out_offset, bad);
    const int any = __syncthreads_or(bad);
    if (threadIdx.x == 0) st->status = any ? GSMI_STAMP_NONFINITE : 0;
}

template <int N, int SIG>
int launch(const gsmi_stamp* stamps, int nstamps, const gsmi_op* ops, const gsmi_leaf* leaves,
           Tables<float> tb, TwiddleSet<float> tws, size_t lds, float* out, void* stream)
{
    auto fn = draw_stamp_f32<N, SIG>;
    int rc = allow_lds(reinterpret_cast<const void*>(fn), lds);
    if (rc) return rc;
    hipLaunchKernelGGL(fn, dim3(nstamps), dim3(Shape<N>::T), lds,
                       reinterpret_cast<hipStream_t>(stream), const_cast<gsmi_stamp*>(stamps), ops,
                       leaves, tb, tws, int(lds), out);
    return hip_check(hipGetLastError(), "draw_stamp launch");
}

template <int N>
int dispatch(int program, const gsmi_stamp* stamps, int nstamps, const gsmi_op* ops,
             const gsmi_leaf* leaves, Tables<float> tb, TwiddleSet<float> tws, size_t lds,
             float* out, void* stream)
{
    switch (program) {
      case 1: return launch<N, 1>(stamps, nstamps, ops, leaves, tb, tws, lds, out, stream);
      case 2: return launch<N, 2>(stamps, nstamps, ops, leaves, tb, tws, lds, out, stream);
      case 3: return launch<N, 3>(stamps, nstamps, ops, leaves, tb, tws, lds, out, stream);
      case 4: return launch<N, 4>(stamps, nstamps, ops, leaves, tb, tws, lds, out, stream);
    }
    set_error("gsmi_draw_stamps_f32: unknown program shape");
    return GSMI_E_ARG;
}

}  // namespace
}  // namespace gsmi

using namespace gsmi;

extern "C" {

int64_t gsmi_draw_stamps_lds(int N, int max_Nk, int max_ncoef)
{
    if (max_Nk < N || max_Nk >= 2 * N || max_ncoef < 0) return -1;
    if (N == 128) return int64_t(stamp_lds<128>(max_ncoef, max_Nk / 2));
    if (N == 192) return int64_t(stamp_lds<192>(max_ncoef, max_Nk / 2));
    return -1;
}

int gsmi_draw_stamps_f32(const gsmi_stamp* stamps, int nstamps, int N, int max_Nk, int max_ncoef,
                         int program, const gsmi_op* ops, const gsmi_leaf* leaves,
                         const double* tables, const float* tables32, float* out, void* stream)
{
    if (!stamps || !ops || !leaves || !out || nstamps < 0) {
        set_error("gsmi_draw_stamps_f32: null buffer or negative count");
        return GSMI_E_ARG;
    }
    const int64_t lds = gsmi_draw_stamps_lds(N, max_Nk, max_ncoef);
    if (lds < 0 || size_t(lds) > lds_limit()) {
        set_error("gsmi_draw_stamps_f32: unsupported size N = " + std::to_string(N) + ", Nk = " +
                  std::to_string(max_Nk));
        return GSMI_E_SIZE;
    }
    if (nstamps == 0) return GSMI_OK;
    const TwiddleSet<float> tws = twiddle_set<float>();
    if (!tws.p2 || !tws.p3) {
        set_error("twiddle table allocation failed");
        return GSMI_E_HIP;
    }
    const Tables<float> tb{tables, tables32, reinterpret_cast<const float4*>(tables32)};
    if (N == 128)
        return dispatch<128>(program, stamps, nstamps, ops, leaves, tb, tws, size_t(lds), out,
                             stream);
    return dispatch<192>(program, stamps, nstamps, ops, leaves, tb, tws, size_t(lds), out, stream);
}

}
