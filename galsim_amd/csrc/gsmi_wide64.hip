// FP64 entry points of the per-size column and row kernels (wide_kernels.h).
#define GSMI_WIDE_F64
#include "wide_kernels.h"

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
      GSMI_F64_SIZES(GSMI_SIZE)
#undef GSMI_SIZE
      default: return -1;
    }
}

int gsmi_draw_wide_f64(const gsmi_stamp* stamps, const gsmi_size_group* groups, int ngroups,
                       int program, const gsmi_op* ops, const gsmi_leaf* leaves,
                       const double* tables, const int32_t* cliprows, void* scratch, double* out,
                       void* stream)
{
    if (!stamps || !groups || ngroups < 1 || !ops || !leaves || !scratch || !out) {
        set_error("gsmi_draw_wide_f64: null buffer or no group");
        return GSMI_E_ARG;
    }
    if (program < 1 || program > 4) {
        set_error("gsmi_draw_wide_f64: unknown program shape");
        return GSMI_E_ARG;
    }
    for (int g = 0; g < ngroups; ++g) {
        const gsmi_size_group& G = groups[g];
        if (G.first < 0 || G.count < 1 || G.max_ny < 1) {
            set_error("gsmi_draw_wide_f64: bad group");
            return GSMI_E_ARG;
        }
        const int64_t lds = gsmi_draw_wide_lds_f64(G.N, G.max_Nk);
        if (lds < 0 || size_t(lds) > lds_limit()) {
            set_error("gsmi_draw_wide_f64: unsupported size N = " + std::to_string(G.N) +
                      ", Nk = " + std::to_string(G.max_Nk));
            return GSMI_E_SIZE;
        }
    }
    const TwiddleSet<double> tws = twiddle_set<double>();
    if (!tws.p2 || !tws.p3) {
        set_error("twiddle table allocation failed");
        return GSMI_E_HIP;
    }
    return draw_groups<double>(stamps, groups, ngroups, 0, program, ops, leaves,
                              Tables<double>{tables, cliprows}, tws,
                              reinterpret_cast<cplx<double>*>(scratch), out, stream);
}

}
