// Pieces shared by the kernels that draw stamps of a specialised program shape: pair
// evaluation of the program, the fold of its samples onto packed columns in LDS, and the
// butterflies of the in-place transforms.
#pragma once

#include <hip/hip_runtime.h>

#include "device_program.h"

namespace gsmi {

// Radix 16 (e^{+2 pi i}) as radix 4 over n1 and radix 4 over n2 with n = 4 n1 + n2, k = k1 + 4 k2.
template <typename F>
__device__ __forceinline__ void bfly16(cplx<F>* v)
{
    const F c1 = F(0.92387953251128675613), s1 = F(0.38268343236508977173);   // cos, sin pi/8
    const F h = F(0.70710678118654752440);
    cplx<F> a[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
        cplx<F> u[4] = {v[n2], v[n2 + 4], v[n2 + 8], v[n2 + 12]};
        bfly4(u);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) a[n2][k1] = u[k1];
    }
    // w16^(n2 k1): w = (c1, s1), w^2 = (h, h), w^3 = (s1, c1), w^4 = i, w^6 = (-h, h),
    // w^9 = (-c1, -s1)
    a[1][1] = cmul(a[1][1], cplx<F>{c1, s1});
    a[1][2] = {h * (a[1][2].x - a[1][2].y), h * (a[1][2].x + a[1][2].y)};
    a[1][3] = cmul(a[1][3], cplx<F>{s1, c1});
    a[2][1] = {h * (a[2][1].x - a[2][1].y), h * (a[2][1].x + a[2][1].y)};
    a[2][2] = {-a[2][2].y, a[2][2].x};
    a[2][3] = {-h * (a[2][3].x + a[2][3].y), h * (a[2][3].x - a[2][3].y)};
    a[3][1] = cmul(a[3][1], cplx<F>{s1, c1});
    a[3][2] = {-h * (a[3][2].x + a[3][2].y), h * (a[3][2].x - a[3][2].y)};
    a[3][3] = cmul(a[3][3], cplx<F>{-c1, -s1});
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        cplx<F> u[4] = {a[0][k1], a[1][k1], a[2][k1], a[3][k1]};
        bfly4(u);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = u[k2];
    }
}

template <int R, typename F>
__device__ __forceinline__ void bfly(cplx<F>* v)
{
    static_assert(R == 4 || R == 8 || R == 12 || R == 16, "radix");
    if constexpr (R == 4) bfly4(v);
    if constexpr (R == 8) bfly8(v);
    if constexpr (R == 12) bfly12(v);
    if constexpr (R == 16) bfly16(v);
}

// Moffat of non-special beta off the table: out of line, as few samples or none take it.
static __device__ __noinline__ float2 moffat_off_table(const LeafC<float>& C, float k)
{
    float g, dg;
    moffat_generic_f32(C, k, &g, &dg);
    return {g, dg};
}

// Value of leaf l of shape SIG from its quadratic form q = |k'|^2 s^2.
template <int SIG>
__device__ __forceinline__ float radial_static(int l, const LeafC<float>& C, const LeafI& I,
                                               const Tables<float>& tb, float q)
{
    const int type = kStaticPrograms[SIG].type[l];
    if (type == GSMI_LEAF_SERSIC) return C.flux * sersic_f32(C, tb.coef, I.ntab, q);
    if (type == GSMI_LEAF_MOFFAT) {
        // eval_leafc's Moffat forms on k = sqrt(q)
        const float k = sqrtf(fmaxf(q, 0.f));
        float g, dg;
        switch (I.kind) {
          case 1:
            return C.flux * moffat_trunc_spline<float>(sersic_table<float>(tb, I.aux), I.ntab, q,
                                                       k, C.p[1], nullptr);
          case 15: return C.flux * __expf(-k);
          case 25: return C.flux * __expf(-k) * (1.f + k);
          case 35: return C.flux * __expf(-k) * (3.f + (3.f + k) * k);
          case 0:
            // (the out-of-line call costs every kind of a kernel registers: 46 -> 51 us on 1024
            // stamps of beta = 3, so kernels without tables do without it)
            if constexpr (SIG == kMoffatTableProgram) {
                float x;
                const float4* e = I.ntab > 0 ? moffat_entry(tb.radial + I.aux, q, &x) : nullptr;
                return C.flux * (e ? moffat_eval(e[0], x) : moffat_off_table(C, k).x);
            }
            moffat_generic_f32(C, k, &g, &dg);
            return C.flux * g;
          default: moffat_int_kind_f32(I.kind, k, &g, &dg); return C.flux * g;
        }
    }
    LeafI J = I;
    J.type = type;
    return radial_f32(C, J, tb, q);
}

// The program at (i dk, m dk) and (i dk, -m dk) of a stamp of shape SIG (real values: radial
// leaves only).  The last leaf, the PSF, is evaluated once when its form has no kx ky term.
template <typename F, int SIG>
struct StaticPair;
template <int SIG>
struct StaticPair<float, SIG> {
    LeafC<float> lr[kProgLeaves];
    LeafI li[kProgLeaves];
    Tables<float> tb;
    float dk;
    bool even;               // q1 of the last leaf is zero
    const gsmi_leaf* leaves;
    int Nk;

    __device__ __forceinline__ void operator()(int i, int m, float* p, float* n) const
    {
        constexpr int nl = kStaticPrograms[SIG].nl;
        const float kx = float(i) * dk, ky = float(m) * dk;
        const float xx = kx * kx, xy = kx * ky, yy = ky * ky;
        float vp[kProgLeaves] = {}, vn[kProgLeaves] = {};
#pragma unroll
        for (int l = 0; l < nl; ++l) {
            const LeafC<float>& C = lr[l];
            const float a = C.q0 * xx + C.q2 * yy;
            if (l == nl - 1) {
                vp[l] = radial_static<SIG>(l, C, li[l], tb, a + C.q1 * xy);
                vn[l] = vp[l];
                if (!even) vn[l] = radial_static<SIG>(l, C, li[l], tb, a - C.q1 * xy);
            } else {
                vp[l] = radial_static<SIG>(l, C, li[l], tb, a + C.q1 * xy);
                vn[l] = radial_static<SIG>(l, C, li[l], tb, a - C.q1 * xy);
            }
        }
        *p = static_ops<float, SIG>(vp, -1, 0.f);
        *n = static_ops<float, SIG>(vn, -1, 0.f);
    }
};

// The same in FP64: each leaf by the forms of the general kernels (the clip rows of the reference,
// k' through the Jacobian), the PSF shared as above.
template <int SIG>
struct StaticPair<double, SIG> {
    LeafC<double> lr[kProgLeaves];
    LeafI li[kProgLeaves];
    Tables<double> tb;
    double dk;
    bool even;
    const gsmi_leaf* leaves;
    int Nk;

    __device__ __forceinline__ void operator()(int i, int m, double* p, double* n) const
    {
        constexpr int nl = kStaticPrograms[SIG].nl;
        const double kx = double(i) * dk, ky = double(m) * dk;
        double vp[kProgLeaves] = {}, vn[kProgLeaves] = {};
#pragma unroll
        for (int l = 0; l < nl; ++l) {
            LeafI I = li[l];
            I.type = kStaticPrograms[SIG].type[l];
            vp[l] = eval_leafc<double>(lr[l], I, leaves + l, tb, kx, ky, i, m, Nk);
            if (l == nl - 1 && even)
                vn[l] = vp[l];
            else
                vn[l] = eval_leafc<double>(lr[l], I, leaves + l, tb, kx, -ky, i, -m, Nk);
        }
        *p = static_ops<double, SIG>(vp, -1, 0.);
        *n = static_ops<double, SIG>(vn, -1, 0.);
    }
};

// Fill packed columns [c0, c0 + ncol) of a stamp's wrapped N-grid: cell (c, r) at
// buf[(c - c0) * L + pad(r)], column 0 holding cell(0, r) + i cell(N/2, r) (both Hermitian along
// ky, so their transforms are real).  hk = Nk/2 < N: a cell has at most one aliased sample per
// axis.  X(kx), kx <= hk and Y(ky), 0 <= ky <= hk: the axis factors (Y(-ky) is conj Y(ky): the
// hoisted factors are sincs, shifts and constants).  T threads; ends with a barrier.
//
// Samples come in pairs (kx, ky), (kx, -ky), which share the circular PSF's value, the products
// X Y and most of the quadratic forms; where T and N/2 allow, a thread keeps one ky for all its
// columns.  Aliased samples follow as compact passes that add to the cells: evaluated in the
// primary pass they would idle most lanes of every wave.
template <int N, int L, int T, typename F, typename Pad, typename P>
__device__ __forceinline__ void fill_cells(const P& pair, const Pad& pad, int hk,
                                           const cplx<F>* X, const cplx<F>* Y, int c0,
                                           int ncol, cplx<F>* buf)
{
    constexpr int H = N / 2;
    const int tid = threadIdx.x;
    const int a = N - hk;                    // aliased rows: |ky| from a to N/2
    const int na = H - a + 1;                // a <= N/2 as Nk >= N
    // F(i, m) and F(i, -m), m >= 0
    auto sample = [&](int i, int m, cplx<F> x, cplx<F> y, cplx<F>* fp,
                      cplx<F>* fn) {
        F p, n;
        pair(i, m, &p, &n);
        const F ac = x.x * y.x, bd = x.y * y.y, ad = x.x * y.y, bc = x.y * y.x;
        *fp = {p * (ac - bd), p * (ad + bc)};
        *fn = {n * (ac + bd), n * (bc - ad)};
    };
    // primary samples: rows j and N - j, j < N/2 (row N/2 belongs to the next pass)
    auto primary = [&](int cl, int j, cplx<F> y) {
        cplx<F> fp, fn;
        sample(c0 + cl, j, X[c0 + cl], y, &fp, &fn);
        buf[cl * L + pad(j)] = fp;
        if (j) buf[cl * L + pad(N - j)] = fn;
    };
    if constexpr (T % H == 0) {
        const int j = tid % H;
        const cplx<F> y = Y[j];
        for (int cl = tid / H; cl < ncol; cl += T / H) primary(cl, j, y);
    } else if constexpr (H % T == 0) {
        for (int j = tid; j < H; j += T) {
            const cplx<F> y = Y[j];
            for (int cl = 0; cl < ncol; ++cl) primary(cl, j, y);
        }
    } else {
        for (int t = tid; t < ncol * H; t += T) {
            const int cl = unsigned(t) / unsigned(H);
            const int j = t - cl * H;
            primary(cl, j, Y[j]);
        }
    }
    __syncthreads();
    const float inv_na = 1.f / float(na);
    // aliased rows of these columns: ky = N - j adds to row N - j's congruent, -j, and ky = j - N
    // to row j; row N/2 takes both of ky = +-N/2
    for (int t = tid; t < ncol * na; t += T) {
        const int cl = fdiv(t, inv_na);
        const int j = a + (t - cl * na);
        cplx<F> fp, fn;
        sample(c0 + cl, N - j, X[c0 + cl], Y[N - j], &fp, &fn);
        cplx<F>* col = buf + cl * L;
        if (j == H) {
            col[pad(H)] = cadd(fp, fn);
        } else {
            cplx<F>& lo = col[pad(j)];
            cplx<F>& hi = col[pad(N - j)];
            lo = cadd(lo, fn);
            hi = cadd(hi, fp);
        }
    }
    __syncthreads();
    // samples of columns kx = N/2..hk.  kx > N/2 is congruent to kx - N < 0, whose cells are the
    // conjugates at -ky of column kx: they add to column N - kx.  Column N/2 itself takes both
    // signs and goes to the imaginary part of column 0.  wj, wn: that column's folded values at
    // rows j and N - j.
    const int cf = max(c0, a);               // first column here with an aliased kx
    const int nyq = c0 == 0 ? 1 : 0;
    const int nv = max(0, c0 + ncol - cf) + nyq;
    auto alias_kx = [&](int k) { return k < nyq ? H : N - (cf + k - nyq); };
    auto add_alias = [&](int kx, int j, cplx<F> wj, cplx<F> wn) {
        cplx<F>* col = buf + (kx == H ? 0 : N - kx - c0) * L;
        cplx<F> dj = cconj(wn), dn = cconj(wj);
        if (kx == H) {
            const cplx<F> cj = cadd(wj, dj), cn = cadd(wn, dn);
            dj = {-cj.y, cj.x};
            dn = {-cn.y, cn.x};
        }
        cplx<F>& lo = col[pad(j)];
        lo = cadd(lo, dj);
        if (j != 0 && j != H) {
            cplx<F>& hi = col[pad(N - j)];
            hi = cadd(hi, dn);
        }
    };
    for (int t = tid; t < nv * H; t += T) {
        const int k = unsigned(t) / unsigned(H);
        const int j = t - k * H;
        const int kx = alias_kx(k);
        cplx<F> fp, fn;
        sample(kx, j, X[kx], Y[j], &fp, &fn);
        add_alias(kx, j, fp, fn);
    }
    __syncthreads();
    for (int t = tid; t < nv * na; t += T) {
        const int k = fdiv(t, inv_na);
        const int j = a + (t - k * na);
        const int kx = alias_kx(k);
        cplx<F> fp, fn;
        sample(kx, N - j, X[kx], Y[N - j], &fp, &fn);
        if (j == H) fp = fn = cadd(fp, fn);
        add_alias(kx, j, fn, fp);
    }
    __syncthreads();
}

// v(c) = E + i O of the real inverse transform along x, E = Z(c) + conj Z(N/2 - c), O = (Z(c) -
// conj Z(N/2 - c)) w^c with w = e^{2 pi i / N}, and v(N/2 - c) = conj E + i conj O, which has the
// same two inputs.
template <typename F>
__device__ __forceinline__ void c2r_pair(cplx<F> zc, cplx<F> zm, cplx<F> wc,
                                         cplx<F>* v, cplx<F>* vm)
{
    const cplx<F> E = {zc.x + zm.x, zc.y - zm.y};
    const cplx<F> O = cmul(cplx<F>{zc.x - zm.x, zc.y + zm.y}, wc);
    *v = {E.x - O.y, E.y + O.x};
    *vm = {E.x + O.y, O.x - E.y};
}

// The inputs of units b0 and b1 = Q - b0 (unit 0: b0 = 0 and b1 = Q/2) of the first, radix-R pass
// of that transform over columns b + Q s, Q = (N/2) / R, formed in place from the columns'
// values; column 0 is the packed pair (Z(0), Z(N/2)), both real.  w(c) = e^{2 pi i c / N}.
template <int R, int Q, typename F, typename W>
__device__ __forceinline__ void c2r_inputs(int b0, const W& w, cplx<F>* va, cplx<F>* vb)
{
    if (b0 == 0) {
        // column Q s pairs with Q (R - s); column Q/2 + Q s with Q/2 + Q (R - 1 - s)
        va[0] = {va[0].x + va[0].y, va[0].x - va[0].y};
#pragma unroll
        for (int s = 1; s < R / 2; ++s) c2r_pair(va[s], va[R - s], w(Q * s), &va[s], &va[R - s]);
        cplx<F> same;
        c2r_pair(va[R / 2], va[R / 2], w(Q * R / 2), &va[R / 2], &same);
#pragma unroll
        for (int s = 0; s < R / 2; ++s)
            c2r_pair(vb[s], vb[R - 1 - s], w(Q / 2 + Q * s), &vb[s], &vb[R - 1 - s]);
    } else {
#pragma unroll
        for (int s = 0; s < R; ++s)
            c2r_pair(va[s], vb[R - 1 - s], w(b0 + Q * s), &va[s], &vb[R - 1 - s]);
    }
}

}  // namespace gsmi
