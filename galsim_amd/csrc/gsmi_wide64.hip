// FP64 entry points of the per-size column and row kernels (wide_kernels.h).
#include "wide_kernels.h"

#define GSMI_WIDE_SIZES(X) X(128) X(192) X(256) X(384) X(512) X(768) X(1024) X(1536) X(2048)

using namespace gsmi;

extern "C" {

int64_t gsmi_draw_wide_lds_f64(int N, int max_Nk)
{
    if (max_Nk < N || max_Nk >= 2 * N) return -1;
    switch (N) {
#define GSMI_SIZE(NN)                                                                           \
      case NN: {                                                                                \
        const size_t a = cols_lds<double, NN>(0), b = rows_lds<double, NN>;                        \
        return int64_t(a > b ? a : b);                                                          \
      }
      GSMI_WIDE_SIZES(GSMI_SIZE)
#undef GSMI_SIZE
      default: return -1;
    }
}

int gsmi_draw_wide_f64(const gsmi_stamp* stamps, int nstamps, int N, int max_Nk, int max_ny,
                       int program, const gsmi_op* ops, const gsmi_leaf* leaves,
                       const double* tables, const int32_t* cliprows, void* scratch,
                       double* out, void* stream)
{
    if (!stamps || !ops || !leaves || !scratch || !out || nstamps < 0 || max_ny <= 0) {
        set_error("gsmi_draw_wide_f64: null buffer, negative count or empty stamps");
        return GSMI_E_ARG;
    }
    const int64_t lds = gsmi_draw_wide_lds_f64(N, max_Nk);
    if (lds < 0 || size_t(lds) > lds_limit()) {
        set_error("gsmi_draw_wide_f64: unsupported size N = " + std::to_string(N) + ", Nk = " +
                  std::to_string(max_Nk));
        return GSMI_E_SIZE;
    }
    if (program < 1 || program > 4) {
        set_error("gsmi_draw_wide_f64: unknown program shape");
        return GSMI_E_ARG;
    }
    if (nstamps == 0) return GSMI_OK;
    const TwiddleSet<double> tws = twiddle_set<double>();
    if (!tws.p2 || !tws.p3) {
        set_error("twiddle table allocation failed");
        return GSMI_E_HIP;
    }
    int rc = launch_axis_factors<double>(stamps, nstamps, ops, leaves, scratch, stream);
    if (rc) return rc;
    const Tables<double> tb{tables, cliprows};
    cplx<double>* scr = reinterpret_cast<cplx<double>*>(scratch);
    switch (N) {
#define GSMI_SIZE(NN)                                                                           \
      case NN:                                                                                  \
        return launch_wide_all<double, NN>(stamps, nstamps, max_ny, 0, program, ops, leaves, tb,         \
                                       tws, scr, out, stream);
      GSMI_WIDE_SIZES(GSMI_SIZE)
#undef GSMI_SIZE
      default: return GSMI_E_SIZE;
    }
}

}
