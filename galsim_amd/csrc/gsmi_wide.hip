// FP32 entry points of the per-size column and row kernels (wide_kernels.h).
#include "wide_kernels.h"

using namespace gsmi;

extern "C" {

int64_t gsmi_draw_wide_lds(int N, int max_Nk, int max_ncoef)
{
    if (max_Nk < N || max_Nk >= 2 * N || max_ncoef < 0) return -1;
    switch (N) {
#define GSMI_SIZE(NN)                                                                           \
      case NN: {                                                                                \
        const size_t a = cols_lds<float, NN>(max_ncoef), b = rows_lds<float, NN>;                  \
        return int64_t(a > b ? a : b);                                                          \
      }
      GSMI_F32_SIZES(GSMI_SIZE)
#undef GSMI_SIZE
      default: return -1;
    }
}

int gsmi_draw_wide_f32(const gsmi_stamp* stamps, const gsmi_size_group* groups, int ngroups,
                       int max_ncoef, int program, const gsmi_op* ops, const gsmi_leaf* leaves,
                       const double* tables, const float* tables32, void* scratch, float* out,
                       void* stream)
{
    if (!stamps || !groups || ngroups < 1 || !ops || !leaves || !scratch || !out) {
        set_error("gsmi_draw_wide_f32: null buffer or no group");
        return GSMI_E_ARG;
    }
    if (program < 1 || program > kMoffatTableProgram) {
        set_error("gsmi_draw_wide_f32: unknown program shape");
        return GSMI_E_ARG;
    }
    for (int g = 0; g < ngroups; ++g) {
        const gsmi_size_group& G = groups[g];
        if (G.first < 0 || G.count < 1 || G.max_ny < 1) {
            set_error("gsmi_draw_wide_f32: bad group");
            return GSMI_E_ARG;
        }
        const int64_t lds = gsmi_draw_wide_lds(G.N, G.max_Nk, max_ncoef);
        if (lds < 0 || size_t(lds) > lds_limit()) {
            set_error("gsmi_draw_wide_f32: unsupported size N = " + std::to_string(G.N) +
                      ", Nk = " + std::to_string(G.max_Nk));
            return GSMI_E_SIZE;
        }
    }
    const TwiddleSet<float> tws = twiddle_set<float>();
    if (!tws.p2 || !tws.p3) {
        set_error("twiddle table allocation failed");
        return GSMI_E_HIP;
    }
    return draw_groups<float>(stamps, groups, ngroups, max_ncoef, program, ops, leaves,
                              Tables<float>{tables, tables32, reinterpret_cast<const float4*>(tables32)}, tws,
                              reinterpret_cast<cplx<float>*>(scratch), out, stream);
}

}
