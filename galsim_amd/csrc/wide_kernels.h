// Drawing of stamps of a specialised program shape in two kernels compiled per FFT size (FP32 at
// N = 128 to 4096, FP64 at 128 to 2048): columns of the wrapped grid to the scratch buffer, then
// its rows to pixels.
//
// fold_cols: a workgroup takes CC packed columns at a time: fill_cells puts their cells in LDS, an
// in-place DFT of two or three radix passes runs along ky, and the rows of the output window go
// to the scratch columns (contiguous, 128-byte aligned).
// row_pixels: a workgroup takes R output rows.  Its first pass reads them straight from the
// scratch columns into registers -- R consecutive values of a column at a time, so R of 16 or 32
// (8 at the largest sizes, where LDS ends) decides how much of each 128-byte line is used --
// forms E + i O and does the first radix pass; the others run in place in LDS, the last one
// writing the pixels.
//
// Against the kernels for any shape and size: half the LDS (no ping-pong buffers), samples in
// +-ky pairs, every index of the transforms a constant, and full lines of scratch per row chunk
// (those read 1024 / (N/2) rows, 8 bytes of each line at N = 2048).
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "../../include/gsmi.h"
#include "device_program.h"
#include "launch.h"
#include "stamp_cells.h"

namespace gsmi {
namespace {

// In-place transform of length N = C1 C2 C3 (C3 = 1: two passes) on a padded LDS line.  Pass 1
// runs over elements N/C1 apart, pass 2 over C3 apart within each block of N/C1, pass 3 over runs
// of C3; output y ends at slot(y).  A line carries one slot of padding per last-radix run and, with
// three passes, one per N/C1 block: the strides of every pass and of the output order are then odd
// or contiguous across lanes, so LDS accesses spread over the banks, and all of them are
// compile-time offsets from a unit's first element.
template <int N_, int C1_, int C2_, int C3_>
struct Line {
    static constexpr int N = N_, C1 = C1_, C2 = C2_, C3 = C3_;
    static constexpr bool three = C3 > 1;
    static constexpr int last = three ? C3 : C2;
    static constexpr int NB = N / C1;
    static constexpr int STEP = NB + NB / last + (three ? 1 : 0);   // pad(r + NB) - pad(r)
    static_assert(C1 * C2 * C3 == N, "radices");
    __host__ __device__ static constexpr int pad(int r)
    {
        return r + r / last + (three ? r / NB : 0);
    }
    static constexpr int L = (C1 * STEP) | 1;
    __device__ static __forceinline__ int slot(int y)
    {
        if constexpr (three)
            return (y % C1) * STEP + (y / C1 % C2) * (C3 + 1) + y / (C1 * C2);
        else
            return (y % C1) * STEP + y / C1;
    }
};

// Passes 2 (of three) over nline lines: tw(m) = e^{2 pi i m / NB}.
template <typename S, int T, typename F, typename W>
__device__ __forceinline__ void middle_pass(cplx<F>* buf, int nline, const W& w)
{
    constexpr int U = S::C1 * S::C3;
    for (int t = threadIdx.x; t < nline * U; t += T) {
        const int line = unsigned(t) / unsigned(U);
        const int q = t - line * U;
        const int k1 = unsigned(q) / unsigned(S::C3);
        const int b = q - k1 * S::C3;
        cplx<F>* p = buf + line * S::L + k1 * S::STEP + b;
        cplx<F> v[S::C2];
#pragma unroll
        for (int s = 0; s < S::C2; ++s) v[s] = p[s * (S::C3 + 1)];
        bfly<S::C2>(v);
#pragma unroll
        for (int k = 1; k < S::C2; ++k) v[k] = cmul(v[k], w(b * k));
#pragma unroll
        for (int s = 0; s < S::C2; ++s) p[s * (S::C3 + 1)] = v[s];
    }
    __syncthreads();
}

// Columns: CC per chunk, T threads, the waves per SIMD the LDS leaves room for; twiddles in LDS up
// to N = 2048.
template <typename F, int N>
struct Cols;
#define GSMI_COLS(F, N, C1, C2, C3, CC_, T_, WAVES_)                                            \
    template <>                                                                                 \
    struct Cols<F, N> : Line<N, C1, C2, C3> {                                                   \
        static constexpr int CC = CC_, T = T_, WAVES = WAVES_;                                  \
        static constexpr bool lds_tw = N <= 2048;                                               \
        static_assert(CC % 2 == 0 && (N / 2) % CC == 0, "even chunks that divide the columns");  \
    };
GSMI_COLS(float, 128, 8, 16, 1, 16, 256, 4)
GSMI_COLS(float, 192, 12, 16, 1, 12, 256, 4)
GSMI_COLS(float, 256, 16, 16, 1, 16, 256, 4)
GSMI_COLS(float, 384, 12, 4, 8, 8, 256, 4)
GSMI_COLS(float, 512, 8, 8, 8, 8, 256, 3)
GSMI_COLS(float, 768, 12, 8, 8, 4, 256, 4)
GSMI_COLS(float, 1024, 16, 8, 8, 4, 256, 3)
GSMI_COLS(float, 1536, 12, 16, 8, 4, 512, 4)
GSMI_COLS(float, 2048, 16, 16, 8, 2, 512, 4)
GSMI_COLS(float, 3072, 12, 16, 16, 2, 512, 4)
GSMI_COLS(float, 4096, 16, 16, 16, 2, 512, 4)
GSMI_COLS(double, 128, 8, 16, 1, 8, 256, 2)
GSMI_COLS(double, 192, 12, 16, 1, 8, 256, 2)
GSMI_COLS(double, 256, 16, 16, 1, 8, 256, 2)
GSMI_COLS(double, 384, 12, 4, 8, 4, 256, 2)
GSMI_COLS(double, 512, 8, 8, 8, 4, 256, 2)
GSMI_COLS(double, 768, 12, 8, 8, 2, 256, 2)
GSMI_COLS(double, 1024, 16, 8, 8, 2, 256, 2)
GSMI_COLS(double, 1536, 12, 16, 8, 2, 512, 2)
GSMI_COLS(double, 2048, 16, 16, 8, 2, 512, 2)
#undef GSMI_COLS

// Rows: R per workgroup, T threads.
template <typename F, int N>
struct Rows;
#define GSMI_ROWS(F, N, D1, D2, D3, R_, T_, WAVES_)                                             \
    template <>                                                                                 \
    struct Rows<F, N> : Line<N / 2, D1, D2, D3> {                                               \
        static constexpr int R = R_, T = T_, WAVES = WAVES_;                                    \
    };
GSMI_ROWS(float, 128, 8, 8, 1, 32, 128, 4)
GSMI_ROWS(float, 192, 8, 12, 1, 32, 256, 4)
GSMI_ROWS(float, 256, 8, 16, 1, 32, 256, 4)
GSMI_ROWS(float, 384, 12, 16, 1, 32, 256, 3)
GSMI_ROWS(float, 512, 8, 8, 4, 16, 256, 4)
GSMI_ROWS(float, 768, 12, 8, 4, 16, 256, 2)
GSMI_ROWS(float, 1024, 8, 8, 8, 16, 512, 4)
GSMI_ROWS(float, 1536, 12, 8, 8, 8, 256, 2)
GSMI_ROWS(float, 2048, 16, 8, 8, 8, 256, 2)
GSMI_ROWS(float, 3072, 12, 16, 8, 8, 512, 2)
GSMI_ROWS(float, 4096, 16, 16, 8, 8, 512, 2)
GSMI_ROWS(double, 128, 8, 8, 1, 16, 128, 2)
GSMI_ROWS(double, 192, 8, 12, 1, 16, 128, 2)
GSMI_ROWS(double, 256, 8, 16, 1, 16, 128, 2)
GSMI_ROWS(double, 384, 12, 16, 1, 16, 128, 2)
GSMI_ROWS(double, 512, 8, 8, 4, 8, 128, 2)
GSMI_ROWS(double, 768, 12, 8, 4, 8, 128, 2)
GSMI_ROWS(double, 1024, 8, 8, 8, 8, 256, 2)
GSMI_ROWS(double, 1536, 12, 8, 8, 4, 128, 2)
GSMI_ROWS(double, 2048, 16, 8, 8, 4, 128, 2)
#undef GSMI_ROWS

template <typename F, int N>
__host__ __device__ constexpr size_t cols_lds(int ncoef)
{
    return sizeof(cplx<F>) * (size_t(Cols<F, N>::CC) * Cols<F, N>::L + (Cols<F, N>::lds_tw ? N : 0)) +
           sizeof(LeafC<F>) * kProgLeaves + 16 * size_t(ncoef);
}

template <typename F, int N>
constexpr size_t rows_lds = sizeof(cplx<F>) * size_t(Rows<F, N>::R) * Rows<F, N>::L;

// Grid: (ceil(N/2 / (CC per_wg)), stamps): per_wg chunks of CC columns each.  A stamp the launch
// cannot draw is flagged and its scratch left as it was.
template <typename F, int N, int SIG, int T>
__device__ __forceinline__ void fold_cols_body(gsmi_stamp* __restrict__ st, int block,
                                               const gsmi_op* __restrict__ ops,
                                               const gsmi_leaf* __restrict__ leaves, Tables<F> tb,
                                               TwiddleSet<F> tws, int lds_bytes, int per_wg,
                                               cplx<F>* __restrict__ scratch)
{
    using S = Cols<F, N>;
    constexpr int H = N / 2, CC = S::CC;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int hk = st->Nk / 2;
    const gsmi_op* sops = ops + st->op_begin;
    const gsmi_leaf* sleaves = leaves + st->leaf_begin;
    bool ok = matches_static<SIG>(sops, st->op_count, sleaves);
    constexpr int ss = sersic_slot<SIG>();
    int ncoef = 0;
    if constexpr (sizeof(F) == 4 && ss >= 0)                // FP32 stages its Sersic cubics
        if (ok) {
            ncoef = sleaves[ss].ntab - 1;
            ok = sleaves[ss].cliprows >= 0 && ncoef >= 1;
        }
    const int y0 = st->y0, ny = st->ny;
    if (!ok || st->N != N || hk < H || hk >= N || y0 < -H || y0 + ny > H ||
        cols_lds<F, N>(ncoef) > size_t(lds_bytes)) {
        if (threadIdx.x == 0) atomicOr(&st->status, GSMI_STAMP_NONFINITE);
        return;
    }
    cplx<F>* buf = reinterpret_cast<cplx<F>*>(smem_raw);
    float4* cfl = reinterpret_cast<float4*>(buf + CC * S::L);
    LeafC<F>* lc = reinterpret_cast<LeafC<F>*>(cfl + ncoef);
    cplx<F>* twl = reinterpret_cast<cplx<F>*>(lc + kProgLeaves);
    int stride;
    const cplx<F>* twg = tws.pick(N, &stride);
    if constexpr (S::lds_tw)
        for (int e = threadIdx.x; e < N; e += T) twl[e] = twg[e * stride];
    auto tw = [&](int m) { return S::lds_tw ? twl[m] : twg[m * stride]; };
    if constexpr (sizeof(F) == 4) tb.radial = scratch + st->axis_offset;
    else tb.radial = reinterpret_cast<const double*>(scratch + st->axis_offset);
    StaticPair<F, SIG> pair;
    pair.leaves = sleaves;
    pair.Nk = st->Nk;
    pair.dk = F(st->dk);
    pair.tb = tb;
    if (int(threadIdx.x) < kStaticPrograms[SIG].nl)
        lc[threadIdx.x] = leaf_consts_t<F>(sleaves[threadIdx.x], tb);
#pragma unroll
    for (int l = 0; l < kStaticPrograms[SIG].nl; ++l) pair.li[l] = leaf_ints(sleaves[l]);
    if constexpr (sizeof(F) == 4 && ss >= 0) {
        const float4* src = tb.coef + sleaves[ss].cliprows / 4;
        for (int e = threadIdx.x; e < ncoef; e += T) cfl[e] = src[e];
        pair.tb.coef = cfl;
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < kStaticPrograms[SIG].nl; ++l) pair.lr[l] = uniform_leaf(lc[l]);
    pair.even = pair.lr[kStaticPrograms[SIG].nl - 1].q1 == F(0);
    const cplx<F>* X = scratch + st->axis_offset;      // X(0..hk), then Y(-hk..hk)
    const cplx<F>* Y = X + hk + 1 + hk;
    const size_t cs = col_stride(st);
    cplx<F>* out = scratch + st->scratch_offset;
    const float inv_ny = 1.f / float(ny);
    const int cend = min(H, (block + 1) * per_wg * CC);
    for (int c0 = block * per_wg * CC; c0 < cend; c0 += CC) {
        fill_cells<N, S::L, T>(pair, [](int r) { return S::pad(r); }, hk, X, Y, c0, CC, buf);
        for (int t = threadIdx.x; t < CC * S::NB; t += T) {
            const int cl = unsigned(t) / unsigned(S::NB);
            const int b = t - cl * S::NB;
            cplx<F>* p = buf + cl * S::L + S::pad(b);
            cplx<F> v[S::C1];
#pragma unroll
            for (int s = 0; s < S::C1; ++s) v[s] = p[s * S::STEP];
            bfly<S::C1>(v);
#pragma unroll
            for (int k = 1; k < S::C1; ++k) v[k] = cmul(v[k], tw(b * k));
#pragma unroll
            for (int s = 0; s < S::C1; ++s) p[s * S::STEP] = v[s];
        }
        __syncthreads();
        if constexpr (S::three)
            middle_pass<S, T>(buf, CC, [&](int m) { return tw(S::C1 * m); });
        constexpr int NR = N / S::last;                    // runs of a column
        for (int t = threadIdx.x; t < CC * NR; t += T) {
            const int cl = unsigned(t) / unsigned(NR);
            const int run = t - cl * NR;
            cplx<F>* p = buf + cl * S::L + S::pad(run * S::last);
            cplx<F> v[S::last];
#pragma unroll
            for (int b = 0; b < S::last; ++b) v[b] = p[b];
            bfly<S::last>(v);
#pragma unroll
            for (int b = 0; b < S::last; ++b) p[b] = v[b];
        }
        __syncthreads();
        for (int e = threadIdx.x; e < CC * ny; e += T) {
            const int cl = fdiv(e, inv_ny);
            const int row = e - cl * ny;
            const int p = y0 + row;
            const cplx<F> v = buf[cl * S::L + S::slot(p < 0 ? p + N : p)];
            const int c = c0 + cl;
            if (c == 0) {
                // the packed column: column 0 in the real part, column N/2 in the imaginary part
                out[row] = {v.x, F(0)};
                out[size_t(H) * cs + row] = {v.y, F(0)};
            } else {
                out[size_t(c) * cs + row] = v;
            }
        }
        __syncthreads();
    }
}

template <typename F, int N, int SIG>
__global__ void __launch_bounds__((Cols<F, N>::T), (Cols<F, N>::WAVES))
fold_cols(gsmi_stamp* __restrict__ stamps, const gsmi_op* __restrict__ ops,
          const gsmi_leaf* __restrict__ leaves, Tables<F> tb, TwiddleSet<F> tws,
          int lds_bytes, int per_wg, cplx<F>* __restrict__ scratch)
{
    fold_cols_body<F, N, SIG, Cols<F, N>::T>(stamps + blockIdx.y, blockIdx.x, ops, leaves, tb, tws,
                                             lds_bytes, per_wg, scratch);
}

template <typename F, int N, int T>
__device__ __forceinline__ void row_pixels_body(gsmi_stamp* __restrict__ st, int block,
                                                const cplx<F>* __restrict__ scratch,
                                                TwiddleSet<F> tws, F* __restrict__ out)
{
    using S = Rows<F, N>;
    constexpr int M = N / 2, R = S::R, Q = S::NB, U = Q / 2, D1 = S::C1;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cplx<F>* buf = reinterpret_cast<cplx<F>*>(smem_raw);
    const int r0 = block * R;
    const int nx = st->nx, x0 = st->x0;
    const int nrow = min(R, st->ny - r0);
    if (st->N != N || nrow <= 0 || x0 < -M || x0 + nx > M) return;
    int stride;
    const cplx<F>* twg = tws.pick(N, &stride);
    auto tw = [&](int m) { return twg[m * stride]; };
    const unsigned cs = col_stride(st);                    // N/2 columns of it stay below 2^24
    const cplx<F>* in = scratch + st->scratch_offset + r0;
    for (int t = threadIdx.x; t < R * U; t += T) {
        const int row = t % R;
        const int u = t / R;
        if (row >= nrow) continue;
        const int b0 = u, b1 = u ? Q - u : Q / 2;
        const cplx<F>* z = in + row;
        cplx<F> va[D1], vb[D1];
#pragma unroll
        for (int s = 0; s < D1; ++s) {
            va[s] = z[unsigned(b0 + Q * s) * cs];
            vb[s] = z[unsigned(b1 + Q * s) * cs];
        }
        if (u == 0) va[0].y = z[unsigned(M) * cs].x;         // the packed pair (Z(0), Z(N/2))
        c2r_inputs<D1, Q>(b0, tw, va, vb);
        bfly<D1>(va);
        bfly<D1>(vb);
#pragma unroll
        for (int k = 1; k < D1; ++k) {
            va[k] = cmul(va[k], tw(2 * b0 * k));
            vb[k] = cmul(vb[k], tw(2 * b1 * k));
        }
        cplx<F>* pa = buf + row * S::L + S::pad(b0);
        cplx<F>* pb = buf + row * S::L + S::pad(b1);
#pragma unroll
        for (int s = 0; s < D1; ++s) {
            pa[s * S::STEP] = va[s];
            pb[s * S::STEP] = vb[s];
        }
    }
    __syncthreads();
    if constexpr (S::three)
        middle_pass<S, T>(buf, nrow, [&](int m) { return tw(2 * D1 * m); });
    constexpr int KK = M / S::last;                        // runs of a row, in output order
    const F norm = F(1) / (F(N) * F(N));
    bool bad = false;
    F* o = out + st->out_offset + size_t(r0) * nx;
    for (int t = threadIdx.x; t < nrow * KK; t += T) {
        const int row = unsigned(t) / unsigned(KK);
        const int kk = t - row * KK;                       // outputs kk + KK k, k < last
        const cplx<F>* p = buf + row * S::L + S::slot(kk);
        cplx<F> v[S::last];
#pragma unroll
        for (int b = 0; b < S::last; ++b) v[b] = p[b];
        bfly<S::last>(v);
        // every output of a row's transform sums every input with a unit-modulus weight, so one
        // output per thread shows a non-finite value anywhere in the row's spectrum
        bad |= !isfinite(v[0].x + v[0].y);
        F* orow = o + size_t(row) * nx;
#pragma unroll
        for (int k = 0; k < S::last; ++k) {
            const int q = 2 * (kk + KK * k);               // pixels q, q + 1 of the N-periodic row
            int col = q - x0;
            col = col >= N ? col - N : (col < 0 ? col + N : col);
            int col1 = col + 1;
            col1 = col1 >= N ? col1 - N : col1;
            if (col < nx) orow[col] = v[k].x * norm;
            if (col1 < nx) orow[col1] = v[k].y * norm;
        }
    }
    if (__syncthreads_or(bad) && threadIdx.x == 0) atomicOr(&st->status, GSMI_STAMP_NONFINITE);
}

// Grid: (ceil(max ny / R), stamps).
template <typename F, int N>
__global__ void __launch_bounds__((Rows<F, N>::T), (Rows<F, N>::WAVES))
row_pixels(gsmi_stamp* __restrict__ stamps, const cplx<F>* __restrict__ scratch,
           TwiddleSet<F> tws, F* __restrict__ out)
{
    row_pixels_body<F, N, Rows<F, N>::T>(stamps + blockIdx.y, blockIdx.x, scratch, tws, out);
}

// ---------------------------------------------------------------------------------------------
// Several FFT sizes in one launch of each kernel: a launch of a handful of workgroups takes 6 to
// 12 us whatever its size, one per FFT size and kernel, and each launch has a tail.  The bodies run
// with kAnyT threads and the LDS of the largest size present, so beyond kMergeBlocks column
// workgroups (64 per CU) the launches per size win by their occupancy.  Measured, apart |
// together, us: bulge + disk batches of 400 stamps (1080 workgroups) 180 | 127, 2400 (4696) 423 |
// 387, 4096 (8968) 636 | 625; Sersic batches of 16 (5248) 385 | 312, 48 (13752) 823 | 787, 64
// (24064) 1283 | 1330.  FP64, whose bodies hold 512-thread workgroups to two waves per SIMD, ends
// at 4 per CU: 256 stamps of two sizes (2300) 80 | 130.
// ---------------------------------------------------------------------------------------------
template <typename F>
constexpr int kMergeBlocks = sizeof(F) == 4 ? 16384 : 1024;
constexpr int kAnyT = 512;
constexpr int kMaxSizes = 16;
struct SizeList {
    int n;
    int N[kMaxSizes];
    int first[kMaxSizes];          // first stamp
    int per[kMaxSizes];            // workgroups per stamp
    int start[kMaxSizes + 1];      // first workgroup

    __device__ __forceinline__ int find(int b, int* stamp, int* block) const
    {
        int k = 0;
        while (k + 1 < n && b >= start[k + 1]) ++k;
        const int r = b - start[k];
        *stamp = first[k] + r / per[k];
        *block = r % per[k];
        return N[k];
    }
};

#define GSMI_F32_SIZES(X) X(128) X(192) X(256) X(384) X(512) X(768) X(1024) X(1536) X(2048) \
    X(3072) X(4096)
#define GSMI_F64_SIZES(X) X(128) X(192) X(256) X(384) X(512) X(768) X(1024) X(1536) X(2048)

template <typename F, int SIG>
__global__ void __launch_bounds__(kAnyT, (sizeof(F) == 4 ? 4 : 2))
fold_cols_any(gsmi_stamp* __restrict__ stamps, SizeList sizes, const gsmi_op* __restrict__ ops,
              const gsmi_leaf* __restrict__ leaves, Tables<F> tb, TwiddleSet<F> tws, int lds_bytes,
              cplx<F>* __restrict__ scratch)
{
    int stamp, block;
    const int N = sizes.find(blockIdx.x, &stamp, &block);
    switch (N) {
#define GSMI_SIZE(NN)                                                                           \
      case NN:                                                                                  \
        fold_cols_body<F, NN, SIG, kAnyT>(stamps + stamp, block, ops, leaves, tb, tws,          \
                                          lds_bytes, 1, scratch);                               \
        break;
#ifdef GSMI_WIDE_F64
      GSMI_F64_SIZES(GSMI_SIZE)
#else
      GSMI_F32_SIZES(GSMI_SIZE)
#endif
#undef GSMI_SIZE
    }
}

template <typename F>
__global__ void __launch_bounds__(kAnyT, (sizeof(F) == 4 ? 4 : 2))
row_pixels_any(gsmi_stamp* __restrict__ stamps, SizeList sizes,
               const cplx<F>* __restrict__ scratch, TwiddleSet<F> tws, F* __restrict__ out)
{
    int stamp, block;
    const int N = sizes.find(blockIdx.x, &stamp, &block);
    switch (N) {
#define GSMI_SIZE(NN)                                                                           \
      case NN: row_pixels_body<F, NN, kAnyT>(stamps + stamp, block, scratch, tws, out); break;
#ifdef GSMI_WIDE_F64
      GSMI_F64_SIZES(GSMI_SIZE)
#else
      GSMI_F32_SIZES(GSMI_SIZE)
#endif
#undef GSMI_SIZE
    }
}

template <typename F, int N, int SIG>
int launch_cols(const gsmi_stamp* stamps, int nstamps, int ncoef, const gsmi_op* ops,
                const gsmi_leaf* leaves, Tables<F> tb, TwiddleSet<F> tws,
                cplx<F>* scratch, void* stream)
{
    auto fn = fold_cols<F, N, SIG>;
    const size_t lds = cols_lds<F, N>(ncoef);
    int rc = allow_lds(reinterpret_cast<const void*>(fn), lds);
    if (rc) return rc;
    const int chunks = N / 2 / Cols<F, N>::CC;
    // several chunks per workgroup share its set-up while the launch keeps 4096 of them
    int per = 1;
    while (per < chunks && size_t(nstamps) * size_t(chunks / (2 * per)) >= 4096) per *= 2;
    const dim3 grid((chunks + per - 1) / per, nstamps);
    const int threads = Cols<F, N>::T;
    hipLaunchKernelGGL(fn, grid, dim3(threads), lds,
                       reinterpret_cast<hipStream_t>(stream), const_cast<gsmi_stamp*>(stamps), ops,
                       leaves, tb, tws, int(lds), per, scratch);
    return hip_check(hipGetLastError(), "fold_cols launch");
}

template <typename F, int N>
int launch_wide(const gsmi_stamp* stamps, int nstamps, int max_ny, int ncoef, int program,
                const gsmi_op* ops, const gsmi_leaf* leaves, Tables<F> tb,
                TwiddleSet<F> tws, cplx<F>* scratch, F* out, void* stream)
{
    int rc = GSMI_E_ARG;
    switch (program) {
#define GSMI_WIDE(SIG)                                                                          \
      case SIG:                                                                                 \
        rc = launch_cols<F, N, SIG>(stamps, nstamps, ncoef, ops, leaves, tb, tws, scratch, stream); \
        break;
      GSMI_WIDE(1)
      GSMI_WIDE(2)
      GSMI_WIDE(3)
      GSMI_WIDE(4)
#undef GSMI_WIDE
      case kMoffatTableProgram:
        if constexpr (sizeof(F) == 4) {
            rc = launch_cols<F, N, kMoffatTableProgram>(stamps, nstamps, ncoef, ops, leaves, tb,
                                                        tws, scratch, stream);
            break;
        }
        [[fallthrough]];
      default: set_error("unknown program shape");
    }
    if (rc) return rc;
    auto fn = row_pixels<F, N>;
    using S = Rows<F, N>;
    const dim3 grid((max_ny + S::R - 1) / S::R, nstamps);
    const size_t lds = rows_lds<F, N>;
    if ((rc = allow_lds(reinterpret_cast<const void*>(fn), lds))) return rc;
    hipLaunchKernelGGL(fn, grid, dim3(S::T), lds, reinterpret_cast<hipStream_t>(stream),
                       const_cast<gsmi_stamp*>(stamps), scratch, tws, out);
    return hip_check(hipGetLastError(), "row_pixels launch");
}


// The kernels of every stamp, at most 32768 at a time: they are the grids' second dimension.
template <typename F, int N>
int launch_wide_all(const gsmi_stamp* stamps, int nstamps, int max_ny, int ncoef, int program,
                    const gsmi_op* ops, const gsmi_leaf* leaves, Tables<F> tb, TwiddleSet<F> tws,
                    cplx<F>* scratch, F* out, void* stream)
{
    int rc = GSMI_OK;
    for (int s0 = 0; s0 < nstamps && !rc; s0 += 32768)
        rc = launch_wide<F, N>(stamps + s0, nstamps - s0 < 32768 ? nstamps - s0 : 32768, max_ny,
                               ncoef, program, ops, leaves, tb, tws, scratch, out, stream);
    return rc;
}

template <typename F>
int launch_any(const gsmi_stamp* stamps, const SizeList& cols, const SizeList& rows, size_t lds_c,
               size_t lds_r, int program, const gsmi_op* ops, const gsmi_leaf* leaves,
               Tables<F> tb, TwiddleSet<F> tws, cplx<F>* scratch, F* out, void* stream)
{
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    gsmi_stamp* st = const_cast<gsmi_stamp*>(stamps);
    int rc = GSMI_E_ARG;
    auto cols_of = [&](auto fn) {
        rc = allow_lds(reinterpret_cast<const void*>(fn), lds_c);
        if (rc) return;
        hipLaunchKernelGGL(fn, dim3(cols.start[cols.n]), dim3(kAnyT), lds_c, s, st, cols, ops,
                           leaves, tb, tws, int(lds_c), scratch);
        rc = hip_check(hipGetLastError(), "fold_cols launch");
    };
    switch (program) {
      case 1: cols_of(fold_cols_any<F, 1>); break;
      case 2: cols_of(fold_cols_any<F, 2>); break;
      case 3: cols_of(fold_cols_any<F, 3>); break;
      case 4: cols_of(fold_cols_any<F, 4>); break;
#ifndef GSMI_WIDE_F64
      case kMoffatTableProgram: cols_of(fold_cols_any<F, kMoffatTableProgram>); break;
#endif
      default: set_error("unknown program shape");
    }
    if (rc) return rc;
    auto fn = row_pixels_any<F>;
    if ((rc = allow_lds(reinterpret_cast<const void*>(fn), lds_r))) return rc;
    hipLaunchKernelGGL(fn, dim3(rows.start[rows.n]), dim3(kAnyT), lds_r, s, st, rows, scratch, tws,
                       out);
    return hip_check(hipGetLastError(), "row_pixels launch");
}

// Every group: one axis-factor launch over their stamps, then both kernels for all of them when
// there are several sizes and at most kMergeBlocks column workgroups, else size by size.
template <typename F>
int draw_groups(const gsmi_stamp* stamps, const gsmi_size_group* groups, int ngroups, int ncoef,
                int program, const gsmi_op* ops, const gsmi_leaf* leaves, Tables<F> tb,
                TwiddleSet<F> tws, cplx<F>* scratch, F* out, void* stream)
{
    SizeList cols{}, rows{};
    size_t lds_c = 0, lds_r = 0;
    int lo = 0x7fffffff, hi = 0;
    int64_t blocks = 0;
    for (int g = 0; g < ngroups; ++g) {
        const gsmi_size_group& G = groups[g];
        lo = G.first < lo ? G.first : lo;
        hi = G.first + G.count > hi ? G.first + G.count : hi;
        int chunks = 0, R = 1;
        size_t c = 0, r = 0;
        switch (G.N) {
#define GSMI_SIZE(NN)                                                                           \
          case NN:                                                                              \
            chunks = NN / 2 / Cols<F, NN>::CC;                                                  \
            R = Rows<F, NN>::R;                                                                 \
            c = cols_lds<F, NN>(ncoef);                                                         \
            r = rows_lds<F, NN>;                                                                \
            break;
#ifdef GSMI_WIDE_F64
          GSMI_F64_SIZES(GSMI_SIZE)
#else
          GSMI_F32_SIZES(GSMI_SIZE)
#endif
#undef GSMI_SIZE
        }
        blocks += int64_t(G.count) * chunks;
        if (blocks > kMergeBlocks<F> || g >= kMaxSizes) continue;
        lds_c = c > lds_c ? c : lds_c;
        lds_r = r > lds_r ? r : lds_r;
        cols.N[g] = rows.N[g] = G.N;
        cols.first[g] = rows.first[g] = G.first;
        cols.per[g] = chunks;
        rows.per[g] = (G.max_ny + R - 1) / R;
        cols.start[g + 1] = cols.start[g] + G.count * chunks;
        rows.start[g + 1] = rows.start[g] + G.count * rows.per[g];
        cols.n = rows.n = g + 1;
    }
    int rc = launch_axis_factors<F>(stamps + lo, hi - lo, ops, leaves, scratch, stream);
    if (rc) return rc;
    if (ngroups > 1 && ngroups <= kMaxSizes && blocks <= kMergeBlocks<F>)
        return launch_any<F>(stamps, cols, rows, lds_c, lds_r, program, ops, leaves, tb, tws,
                             scratch, out, stream);
    for (int g = 0; g < ngroups && !rc; ++g) {
        const gsmi_size_group& G = groups[g];
        switch (G.N) {
#define GSMI_SIZE(NN)                                                                           \
          case NN:                                                                              \
            rc = launch_wide_all<F, NN>(stamps + G.first, G.count, G.max_ny, ncoef, program,    \
                                        ops, leaves, tb, tws, scratch, out, stream);            \
            break;
#ifdef GSMI_WIDE_F64
          GSMI_F64_SIZES(GSMI_SIZE)
#else
          GSMI_F32_SIZES(GSMI_SIZE)
#endif
#undef GSMI_SIZE
        }
    }
    return rc;
}

}  // namespace
}  // namespace gsmi
