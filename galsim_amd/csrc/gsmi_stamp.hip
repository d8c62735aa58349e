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
#include "moffat_shape.h"
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
               int lds_bytes, const cplx<float>* __restrict__ scratch, float* __restrict__ out)
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
    tb.radial = scratch + st->axis_offset;
    StaticPair<float, SIG> pair;
    pair.leaves = sleaves;
    pair.Nk = st->Nk;
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

// ---------------------------------------------------------------------------------------------
// Adjoint of draw_stamp_f32: the gradients of one stamp's fields by one workgroup, in the reverse
// order of the drawing and again without leaving the CU.  Rows: the real DFT (sign +) of each
// residual row into the packed columns.  Columns: column_dft gives Rhat.  Samples: every k-image
// sample is visited once as (kx, +-ky), kx, ky = 0..Nk/2, with its seed A = w Rhat(kx, ky) / N^2
// -- w = 1 at kx = 0, else 2; beyond the grid Rhat is read at the congruent cell -- and adds
// Re[dF/dfield A] to the sums (gsmi_adjoint.hip derives this).  A leaf's scale and Jacobian
// gradients are combinations of three moments, sum g kx^2, g kx ky, g ky^2 with g = flux dphi/dq
// times the rest of the program times the seed, formed at the end in FP64.
// The general kernels write the rows to scratch and read them back column by column, walk one
// sample at a time and reduce the partials of every eight columns in a launch of its own.
// Measured on 1024 Exponential x Moffat(3) stamps of 64 x 64 (N = 128 and 192): 233 us in those
// launches, 90 us here; with the beta derivatives on uneven stamps 535 us, 118 us and 24 us for
// the radial tables (272 us with the order derivative's quadrature per sample).  Bound by VALU
// issue.
// ---------------------------------------------------------------------------------------------

// Unit-flux value and q-derivative of leaf l of shape SIG (eval_leafc_d's forms on q).
template <int SIG>
__device__ __forceinline__ void radial_d(int l, const LeafC<float>& C, const LeafI& I,
                                         const Tables<float>& tb, float q, float* phi, float* dphi)
{
    const int type = kStaticPrograms[SIG].type[l];
    if (type == GSMI_LEAF_EXPONENTIAL) {
        const float r = __builtin_amdgcn_rsqf(1.f + q);
        const float p = q > C.p[0] ? 0.f : r * r * r;
        *phi = p;
        *dphi = -1.5f * p * (r * r);
    } else if (type == GSMI_LEAF_KOLMOGOROV) {
        const float t = __builtin_amdgcn_exp2f((5.f / 6.f) * __builtin_amdgcn_logf(q));
        const float p = __builtin_amdgcn_exp2f(-1.44269504088896341f * t);
        *phi = p;
        *dphi = q > 0.f ? (-5.f / 6.f) * t * __builtin_amdgcn_rcpf(q) * p : 0.f;
    } else if (type == GSMI_LEAF_SERSIC) {
        if (q >= C.p[1]) {
            const float r = __builtin_amdgcn_rsqf(q), iq = r * r;
            *phi = (C.p[2] + C.p[3] * r) * iq;
            *dphi = -(C.p[2] + 1.5f * C.p[3] * r) * iq * iq;
        } else if (q < C.p[0]) {
            *phi = 1.f + q * (C.p[4] + q * C.p[5]);
            *dphi = C.p[4] + 2.f * q * C.p[5];
        } else {
            const float lk = 0.34657359027997264f * __builtin_amdgcn_logf(q);   // ln(q) / 2
            float dS;
            const float S = spline_eq32_d(sersic_table<float>(tb, I.aux), I.ntab, lk, C.t0, C.t1,
                                          C.t2, &dS);
            const float iq = __builtin_amdgcn_rcpf(q);
            *phi = S * iq;
            *dphi = (0.5f * dS - S) * iq * iq;
        }
    } else {
        const float k = __builtin_amdgcn_sqrtf(fmaxf(q, 0.f));
        const float e = __expf(-k);
        switch (I.kind) {
          case 1:
            *phi = moffat_trunc_spline<float>(sersic_table<float>(tb, I.aux), I.ntab, q, k,
                                              C.p[1], dphi);
            break;
          case 15: *phi = e; *dphi = k > 0.f ? ddiv(-0.5f * e, k) : 0.f; break;
          case 25: *phi = e * (1.f + k); *dphi = -0.5f * e; break;
          case 35: *phi = e * (3.f + (3.f + k) * k); *dphi = -0.5f * e * (1.f + k); break;
          case 0:
            if constexpr (SIG == kMoffatTableProgram) {
                float x;
                const float4* e = I.ntab > 0 ? moffat_entry(tb.radial + I.aux, q, &x) : nullptr;
                if (e) {
                    *phi = moffat_eval(e[0], x);
                    *dphi = moffat_eval(e[1], x);
                } else {
                    const float2 gd = moffat_off_table(C, k);
                    *phi = gd.x;
                    *dphi = gd.y;
                }
            } else {
                moffat_generic_f32(C, k, phi, dphi);
            }
            break;
          default: moffat_int_kind_f32(I.kind, k, phi, dphi); break;
        }
    }
}

// d/dnu of the Moffat transform at q.
__device__ __noinline__ float moffat_shape_off_table(float nu, float k)
{
    return moffat_dg_dnu_f32(nu, k);
}
template <int SIG>
__device__ __forceinline__ float moffat_shape(const LeafC<float>& C, const LeafI& I,
                                              const Tables<float>& tb, float q)
{
    if constexpr (SIG == kMoffatTableProgram) {
        float x;
        const float4* e = I.ntab > 0 ? moffat_entry(tb.radial + I.aux, q, &x) : nullptr;
        if (e) return moffat_eval(e[2], x);
    }
    return moffat_shape_off_table(C.p[0] - 1.f, __builtin_amdgcn_sqrtf(fmaxf(q, 0.f)));
}

// Row DFTs of the residual: H(c) = sum_q R(q) e^{2 pi i c q / N} of each window row into the
// packed columns, column c at buf + col_slot(c) L, row y at pad(y); column 0 holds H(0) + i H(N/2)
// (both real).  z(m) = R(2m) + i R(2m+1), m = b + R2 s, takes radix R1 over s, the twiddle, and
// radix R2 over b: c = k1 + R1 k2 ends at column k1 R2 + k2.  Runs k1 and R1 - k1 hold the pairs
// Z(c), Z(N/2 - c) that give H(c) = E + w^c O, E = (Z(c) + conj Z(N/2-c)) / 2, O = (Z(c) -
// conj Z(N/2-c)) / 2i, and H(N/2 - c) = conj E - conj(w^c O).
template <int N>
__device__ __forceinline__ constexpr int col_slot(int c)
{
    return (c % Shape<N>::R1) * Shape<N>::R2 + c / Shape<N>::R1;
}

template <int N>
__device__ __forceinline__ void residual_rows(cplx<float>* buf, const cplx<float>* tw,
                                              const float* __restrict__ in, int x0, int y0, int nx,
                                              int ny)
{
    using S = Shape<N>;
    constexpr int L = S::L, T = S::T, R1 = S::R1, R2 = S::R2, U = R1 / 2;
    for (int t = threadIdx.x; t < ny * R2; t += T) {
        const int idx = unsigned(t) / unsigned(R2);
        const int b = t - idx * R2;
        const int yy = y0 + idx < 0 ? y0 + idx + N : y0 + idx;
        const float* r = in + size_t(idx) * nx;
        cplx<float> v[R1];
#pragma unroll
        for (int s = 0; s < R1; ++s) {
            const int q = 2 * (b + R2 * s);
            int col = q - x0;
            col = col >= N ? col - N : (col < 0 ? col + N : col);
            int col1 = col + 1;
            col1 = col1 >= N ? col1 - N : col1;
            v[s] = {col < nx ? r[col] : 0.f, col1 < nx ? r[col1] : 0.f};
        }
        bfly<R1>(v);
        cplx<float>* p = buf + b * L + pad<N>(yy);
        p[0] = v[0];
#pragma unroll
        for (int k = 1; k < R1; ++k) p[R2 * k * L] = cmul(v[k], tw[2 * b * k]);
    }
    __syncthreads();
    const float inv_ny = 1.f / float(ny);
    // H(c), H(M - c) from Z(c) = zc, Z(M - c) = zm
    auto split = [&](cplx<float>& zc, cplx<float>& zm, int c) {
        const cplx<float> E = {0.5f * (zc.x + zm.x), 0.5f * (zc.y - zm.y)};
        const cplx<float> O = {0.5f * (zc.y + zm.y), 0.5f * (zm.x - zc.x)};
        const cplx<float> wo = cmul(O, tw[c]);
        zc = cadd(E, wo);
        zm = {E.x - wo.x, wo.y - E.y};
    };
    for (int t = threadIdx.x; t < ny * U; t += T) {
        const int u = fdiv(t, inv_ny);
        const int idx = t - u * ny;
        const int yy = y0 + idx < 0 ? y0 + idx + N : y0 + idx;
        const int k0 = u, k1 = u ? R1 - u : R1 / 2;          // unit 0: runs 0 and R1/2
        cplx<float>* p0 = buf + k0 * R2 * L + pad<N>(yy);
        cplx<float>* p1 = buf + k1 * R2 * L + pad<N>(yy);
        cplx<float> va[R2], vb[R2];
#pragma unroll
        for (int b = 0; b < R2; ++b) {
            va[b] = p0[b * L];
            vb[b] = p1[b * L];
        }
        bfly<R2>(va);
        bfly<R2>(vb);
        if (u == 0) {
            // c = R1 k pairs with R1 (R2 - k); c = R1/2 + R1 k with R1/2 + R1 (R2 - 1 - k)
            va[0] = {va[0].x + va[0].y, va[0].x - va[0].y};
#pragma unroll
            for (int k = 1; k < R2 / 2; ++k) split(va[k], va[R2 - k], R1 * k);
            // c = N/4 is its own partner: H = E + i O = Z
#pragma unroll
            for (int k = 0; k < R2 / 2; ++k) split(vb[k], vb[R2 - 1 - k], R1 / 2 + R1 * k);
        } else {
#pragma unroll
            for (int k = 0; k < R2; ++k) split(va[k], vb[R2 - 1 - k], k0 + R1 * k);
        }
#pragma unroll
        for (int b = 0; b < R2; ++b) {
            p0[b * L] = va[b];
            p1[b * L] = vb[b];
        }
    }
    __syncthreads();
}

// Grid: one workgroup per stamp.  grad: GSMI_GRAD_FIELDS doubles per stamp; NaN for a stamp the
// launch does not take.
template <int N, int SIG, bool SHAPE>
__global__ void __launch_bounds__(Shape<N>::T, Shape<N>::WAVES)
grad_stamp_f32(const gsmi_stamp* __restrict__ stamps, const gsmi_op* __restrict__ ops,
               const gsmi_leaf* __restrict__ leaves, Tables<float> tb, TwiddleSet<float> tws,
               int lds_bytes, const cplx<float>* __restrict__ scratch,
               const float* __restrict__ resid, double* __restrict__ grad)
{
    using S = Shape<N>;
    constexpr int H = N / 2, T = S::T, L = S::L;
    constexpr int nl = kStaticPrograms[SIG].nl;
    constexpr int PER = 5;                     // flux, the three moments, shape
    constexpr int NA = PER * nl + 3;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double red[(T / 64) * NA];
    const gsmi_stamp* st = stamps + blockIdx.x;
    double* g = grad + size_t(blockIdx.x) * GSMI_GRAD_FIELDS;
    const int hk = st->Nk / 2;
    const gsmi_op* sops = ops + st->op_begin;
    const int nops = st->op_count;
    const gsmi_leaf* sleaves = leaves + st->leaf_begin;
    const int x0 = st->x0, y0 = st->y0, nx = st->nx, ny = st->ny;
    if (!matches_static<SIG>(sops, nops, sleaves) || st->N != N || hk < H || hk >= N || x0 < -H ||
        x0 + nx > H || y0 < -H || y0 + ny > H || stamp_lds<N>(0, hk) > size_t(lds_bytes)) {
        if (threadIdx.x < GSMI_GRAD_FIELDS) g[threadIdx.x] = NAN;
        return;
    }
    cplx<float>* buf = reinterpret_cast<cplx<float>*>(smem_raw);
    LeafC<float>* lc = reinterpret_cast<LeafC<float>*>(buf + H * L);
    cplx<float>* tw = reinterpret_cast<cplx<float>*>(lc + kProgLeaves);
    cplx<float>* X = tw + N;
    cplx<float>* Y = X + hk + 1;
    const float dk = float(st->dk);
    {
        int stride;
        const cplx<float>* gt = tws.pick(N, &stride);
        for (int e = threadIdx.x; e < N; e += T) tw[e] = gt[e * stride];
        const gsmi_op* aops = sops + nops;
        for (int e = threadIdx.x; e < 2 * (hk + 1); e += T) {
            const bool xaxis = e <= hk;
            const int m = xaxis ? e : e - (hk + 1);
            X[e] = axis_factor<float>(aops, st->axis_count, sleaves, float(m) * dk, xaxis);
        }
        // rows outside the window are zero
        if (ny < N)
            for (int e = threadIdx.x; e < H * L; e += T) buf[e] = {0.f, 0.f};
    }
    tb.radial = scratch + st->axis_offset;
    LeafI li[kProgLeaves];
    if (int(threadIdx.x) < nl)
        lc[threadIdx.x] = leaf_consts_t<float>(sleaves[threadIdx.x], tb);
#pragma unroll
    for (int l = 0; l < nl; ++l) li[l] = leaf_ints(sleaves[l]);
    __syncthreads();
    LeafC<float> lr[kProgLeaves];
#pragma unroll
    for (int l = 0; l < nl; ++l) lr[l] = uniform_leaf(lc[l]);
    const bool even = lr[nl - 1].q1 == 0.f;
    residual_rows<N>(buf, tw, resid + st->out_offset, x0, y0, nx, ny);
    column_dft<N>(buf, tw);

    // FP32 sums of at most four samples, added up in FP64: the terms have random signs, and a
    // longer FP32 sum costs digits of the small fields
    float acc[NA];
    double sum[NA];
#pragma unroll
    for (int f = 0; f < NA; ++f) {
        acc[f] = 0.f;
        sum[f] = 0.;
    }
    int pending = 0;
    const float inv_n2 = 1.f / (float(N) * float(N));
    const int nk = hk + 1;
    const float inv_nk = 1.f / float(nk);
    for (int t = threadIdx.x; t < nk * nk; t += T) {
        const int i = fdiv(t, inv_nk);
        const int m = t - i * nk;
        // seeds of (i, m) and (i, -m): Rhat at rows m and -m mod N of column i, or the conjugates
        // at rows -m and m of column N - i
        const bool far = i > H;
        const int c = far ? N - i : i;
        const int rp = row_slot<N>(m < N ? m : m - N), rn = row_slot<N>(m == 0 ? 0 : N - m);
        const cplx<float>* col = buf + col_slot<N>(c == H ? 0 : c) * L;
        const cplx<float> zp = col[rp + rp / S::PADR], zn = col[rn + rn / S::PADR];
        cplx<float> ap = zp, an = zn;
        if (far) {
            ap = cconj(zn);
            an = cconj(zp);
        } else if (i == 0) {
            ap = {0.5f * (zp.x + zn.x), 0.5f * (zp.y - zn.y)};       // (Z(m) + conj Z(-m)) / 2
            an = cconj(ap);
        } else if (i == H) {
            ap = {0.5f * (zp.y + zn.y), 0.5f * (zn.x - zp.x)};       // (Z(m) - conj Z(-m)) / 2i
            an = cconj(ap);
        }
        // the conjugate sample (0, -m) stands in the sum by itself, (i, .) also for -i
        const float wgt = i == 0 ? inv_n2 : 2.f * inv_n2;
        const cplx<float> x = X[i], y = Y[m];
        const cplx<float> xp = cmul(x, y), xn = cmul(x, cconj(y));
        cplx<float> Zp = cmul(ap, xp), Zn = cmul(an, xn);
        const float wn = m == 0 ? 0.f : wgt;                          // (i, -0) is (i, 0)
        Zp.x *= wgt; Zp.y *= wgt;
        Zn.x *= wn; Zn.y *= wn;
        const float kx = float(i) * dk, ky = float(m) * dk;
        const float xx = kx * kx, xy = kx * ky, yy = ky * ky;
        float vp[kProgLeaves] = {}, vn[kProgLeaves] = {}, php[nl], phn[nl], dp[nl], dn[nl];
#pragma unroll
        for (int l = 0; l < nl; ++l) {
            const LeafC<float>& C = lr[l];
            const float a = C.q0 * xx + C.q2 * yy, b = C.q1 * xy;
            radial_d<SIG>(l, C, li[l], tb, a + b, &php[l], &dp[l]);
            if (l == nl - 1 && even) {
                phn[l] = php[l];
                dn[l] = dp[l];
            } else {
                radial_d<SIG>(l, C, li[l], tb, a - b, &phn[l], &dn[l]);
            }
            vp[l] = C.flux * php[l];
            vn[l] = C.flux * phn[l];
        }
        const float Pp = static_ops<float, SIG>(vp, -1, 0.f);
        const float Pn = static_ops<float, SIG>(vn, -1, 0.f);
        acc[PER * nl] += kx * (Pp * Zp.y + Pn * Zn.y);
        acc[PER * nl + 1] += ky * (Pp * Zp.y - Pn * Zn.y);
        acc[PER * nl + 2] += Pp * Zp.x + Pn * Zn.x;
#pragma unroll
        for (int l = 0; l < nl; ++l) {
            // Re[(dP/dv_l) Z]
            const float tp = static_grad<float, SIG>(vp, l) * Zp.x;
            const float tn = static_grad<float, SIG>(vn, l) * Zn.x;
            acc[PER * l] += tp * php[l] + tn * phn[l];
            const float gp = tp * dp[l], gn = tn * dn[l];
            acc[PER * l + 1] += xx * (gp + gn);
            acc[PER * l + 2] += xy * (gp - gn);
            acc[PER * l + 3] += yy * (gp + gn);
            if constexpr (SHAPE) {
                if (kStaticPrograms[SIG].type[l] == GSMI_LEAF_MOFFAT) {
                    const LeafC<float>& C = lr[l];
                    const float a = C.q0 * xx + C.q2 * yy, b = C.q1 * xy;
                    const float hp = moffat_shape<SIG>(C, li[l], tb, a + b);
                    float hn = hp;
                    if (l != nl - 1 || !even) hn = moffat_shape<SIG>(C, li[l], tb, a - b);
                    acc[PER * l + 4] += tp * hp + tn * hn;
                }
            }
        }
        if (++pending == 2) {
            pending = 0;
#pragma unroll
            for (int f = 0; f < NA; ++f) {
                sum[f] += double(acc[f]);
                acc[f] = 0.f;
            }
        }
    }
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
#pragma unroll
    for (int f = 0; f < NA; ++f) {
        double x = sum[f] + double(acc[f]);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
        if (lane == 0) red[wave * NA + f] = x;
    }
    __syncthreads();
    if (int(threadIdx.x) < NA) {
        double x = 0.;
        for (int w = 0; w < T / 64; ++w) x += red[w * NA + threadIdx.x];
        red[threadIdx.x] = x;                  // column threadIdx.x of wave 0: read only here
    }
    __syncthreads();
    if (threadIdx.x < GSMI_GRAD_FIELDS) {
        const int f = threadIdx.x;
        const int l = f / GSMI_GRAD_PER_LEAF, k = f - l * GSMI_GRAD_PER_LEAF;
        double v = 0.;
        if (f >= GSMI_GRAD_PER_LEAF * GSMI_GRAD_MAXLEAF) {
            v = red[PER * nl + (f - GSMI_GRAD_PER_LEAF * GSMI_GRAD_MAXLEAF)];
        } else if (l < nl) {
            const double* M = red + PER * l;
            const gsmi_leaf& R = sleaves[l];
            const double *j = R.jac, s = R.scale, fs2 = 2. * R.flux * s * s;
            switch (k) {
              case 0: v = M[0]; break;
              case 1:
                v = 2. * R.flux * s * ((j[0] * j[0] + j[1] * j[1]) * M[1] +
                                       2. * (j[0] * j[2] + j[1] * j[3]) * M[2] +
                                       (j[2] * j[2] + j[3] * j[3]) * M[3]);
                break;
              case 2: v = fs2 * (j[0] * M[1] + j[2] * M[2]); break;
              case 3: v = fs2 * (j[1] * M[1] + j[3] * M[2]); break;
              case 4: v = fs2 * (j[0] * M[2] + j[2] * M[3]); break;
              case 5: v = fs2 * (j[1] * M[2] + j[3] * M[3]); break;
              default: v = R.flux * M[4];
            }
        }
        g[f] = v;
    }
}

// The FP32 Moffat tables of every stamp that has room for one (grid: nstamps x the workgroups
// sharing a stamp).
__global__ void __launch_bounds__(kThreads)
moffat_tables_f32(const gsmi_stamp* __restrict__ stamps, const gsmi_op* __restrict__ ops,
                  const gsmi_leaf* __restrict__ leaves, cplx<float>* __restrict__ scratch)
{
    const gsmi_stamp* st = stamps + blockIdx.x;
    for (int o = 0; o < st->op_count; ++o) {
        const gsmi_op op = ops[st->op_begin + o];
        if (op.code != GSMI_OP_LEAF) continue;
        const gsmi_leaf& L = leaves[st->leaf_begin + op.arg];
        if (L.type == GSMI_LEAF_MOFFAT && L.kind != 1 && L.ntab > 0)
            moffat_table_build_f32(L, st->dk, st->Nk / 2, blockIdx.y, gridDim.y,
                                   scratch + st->axis_offset + L.table);
    }
}

template <int N, int SIG>
int launch(const gsmi_stamp* stamps, int nstamps, const gsmi_op* ops, const gsmi_leaf* leaves,
           Tables<float> tb, TwiddleSet<float> tws, size_t lds, const cplx<float>* scratch,
           float* out, void* stream)
{
    auto fn = draw_stamp_f32<N, SIG>;
    int rc = allow_lds(reinterpret_cast<const void*>(fn), lds);
    if (rc) return rc;
    hipLaunchKernelGGL(fn, dim3(nstamps), dim3(Shape<N>::T), lds,
                       reinterpret_cast<hipStream_t>(stream), const_cast<gsmi_stamp*>(stamps), ops,
                       leaves, tb, tws, int(lds), scratch, out);
    return hip_check(hipGetLastError(), "draw_stamp launch");
}

template <int N, int SIG, bool SHAPE>
int launch_grad(const gsmi_stamp* stamps, int nstamps, const gsmi_op* ops,
                const gsmi_leaf* leaves, Tables<float> tb, TwiddleSet<float> tws, size_t lds,
                const cplx<float>* scratch, const float* resid, double* grad, void* stream)
{
    auto fn = grad_stamp_f32<N, SIG, SHAPE>;
    int rc = allow_lds(reinterpret_cast<const void*>(fn), lds);
    if (rc) return rc;
    hipLaunchKernelGGL(fn, dim3(nstamps), dim3(Shape<N>::T), lds,
                       reinterpret_cast<hipStream_t>(stream), stamps, ops, leaves, tb, tws,
                       int(lds), scratch, resid, grad);
    return hip_check(hipGetLastError(), "grad_stamp launch");
}

template <int N>
int dispatch_grad(int program, bool shape, const gsmi_stamp* stamps, int nstamps,
                  const gsmi_op* ops, const gsmi_leaf* leaves, Tables<float> tb,
                  TwiddleSet<float> tws, size_t lds, const cplx<float>* scratch,
                  const float* resid, double* grad, void* stream)
{
#define GSMI_GRAD(SIG, SHAPE)                                                                   \
    return launch_grad<N, SIG, SHAPE>(stamps, nstamps, ops, leaves, tb, tws, lds, scratch,      \
                                      resid, grad, stream)
    switch (program) {
      case 1: GSMI_GRAD(1, false);
      case 2: if (shape) GSMI_GRAD(2, true); else GSMI_GRAD(2, false);
      case 3: GSMI_GRAD(3, false);
      case 4: GSMI_GRAD(4, false);
      case 5: if (shape) GSMI_GRAD(5, true); else GSMI_GRAD(5, false);
    }
#undef GSMI_GRAD
    set_error("gsmi_adjoint_stamps_f32: unknown program shape");
    return GSMI_E_ARG;
}

template <int N>
int dispatch(int program, const gsmi_stamp* stamps, int nstamps, const gsmi_op* ops,
             const gsmi_leaf* leaves, Tables<float> tb, TwiddleSet<float> tws, size_t lds,
             const cplx<float>* scratch, float* out, void* stream)
{
    switch (program) {
      case 1:
        return launch<N, 1>(stamps, nstamps, ops, leaves, tb, tws, lds, scratch, out, stream);
      case 2:
        return launch<N, 2>(stamps, nstamps, ops, leaves, tb, tws, lds, scratch, out, stream);
      case 3:
        return launch<N, 3>(stamps, nstamps, ops, leaves, tb, tws, lds, scratch, out, stream);
      case 4:
        return launch<N, 4>(stamps, nstamps, ops, leaves, tb, tws, lds, scratch, out, stream);
      case 5:
        return launch<N, 5>(stamps, nstamps, ops, leaves, tb, tws, lds, scratch, out, stream);
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
                         const double* tables, const float* tables32, const void* scratch,
                         float* out, void* stream)
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
    const cplx<float>* scr = reinterpret_cast<const cplx<float>*>(scratch);
    if (N == 128)
        return dispatch<128>(program, stamps, nstamps, ops, leaves, tb, tws, size_t(lds), scr, out,
                             stream);
    return dispatch<192>(program, stamps, nstamps, ops, leaves, tb, tws, size_t(lds), scr, out,
                         stream);
}

int gsmi_adjoint_stamps_f32(const gsmi_stamp* stamps, int nstamps, int N, int max_Nk, int program,
                            int shape, const gsmi_op* ops, const gsmi_leaf* leaves,
                            const double* tables, const float* tables32, const void* scratch,
                            const float* resid, double* grad, void* stream)
{
    if (!stamps || !ops || !leaves || !resid || !grad || nstamps < 0) {
        set_error("gsmi_adjoint_stamps_f32: null buffer or negative count");
        return GSMI_E_ARG;
    }
    const int64_t lds = gsmi_draw_stamps_lds(N, max_Nk, 0);
    if (lds < 0 || size_t(lds) > lds_limit()) {
        set_error("gsmi_adjoint_stamps_f32: unsupported size N = " + std::to_string(N) +
                  ", Nk = " + std::to_string(max_Nk));
        return GSMI_E_SIZE;
    }
    if (nstamps == 0) return GSMI_OK;
    const TwiddleSet<float> tws = twiddle_set<float>();
    if (!tws.p2 || !tws.p3) {
        set_error("twiddle table allocation failed");
        return GSMI_E_HIP;
    }
    const Tables<float> tb{tables, tables32, reinterpret_cast<const float4*>(tables32)};
    const cplx<float>* scr = reinterpret_cast<const cplx<float>*>(scratch);
    if (N == 128)
        return dispatch_grad<128>(program, shape != 0, stamps, nstamps, ops, leaves, tb, tws,
                                  size_t(lds), scr, resid, grad, stream);
    return dispatch_grad<192>(program, shape != 0, stamps, nstamps, ops, leaves, tb, tws,
                              size_t(lds), scr, resid, grad, stream);
}

int gsmi_moffat_tables_f32(const gsmi_stamp* stamps, int nstamps, const gsmi_op* ops,
                           const gsmi_leaf* leaves, void* scratch, void* stream)
{
    if (!stamps || !ops || !leaves || !scratch || nstamps < 0) {
        set_error("gsmi_moffat_tables_f32: null buffer or negative count");
        return GSMI_E_ARG;
    }
    if (nstamps == 0) return GSMI_OK;
    const int parts = nstamps >= 1024 ? 1 : nstamps > 128 ? 1024 / nstamps : 8;
    hipLaunchKernelGGL(moffat_tables_f32, dim3(nstamps, parts), dim3(kThreads), 0,
                       reinterpret_cast<hipStream_t>(stream), stamps, ops, leaves,
                       reinterpret_cast<cplx<float>*>(scratch));
    return hip_check(hipGetLastError(), "moffat_tables launch");
}

}
