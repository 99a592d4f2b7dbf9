// Size dispatch: each launcher is defined once per size family (f_g0 .. f_g3,
// see kw_kernels.hpp); the entry points below hand a call to the family that
// holds the line length, and every other grid to the generic-length family
// (kw_generic.hip): contiguous-axis work whose length is not compiled or whose
// row count is odd, column passes whose length is not compiled.
#include "kw_launch.hpp"

namespace kw {

// The small-grid forms of the contiguous-axis updates run where the lanes of all row
// pairs and axes fit about half the chip at these kernels' registers.  Measured, us per
// step with the large-grid forms -> with the small ones: 256^2 35.6 -> 30.1, 64 maps of
// 128^2 (66 k lanes a group) 64.1 -> 59.9, 1024^2 power law 109.8 -> 103.1; beyond, the sixteen
// scan lines of 256^2 to 640^2 lose (197.7 -> 201.6 at 150 k lanes, 218.5 at 300 k) and
// 160^3 (512 k lanes an axis) 289 -> 324.  Plans of a batch share the chip with the others'
// kernels and take half as many (small 3): the scan lines 176 -> 163 us a step; eleven other
// mixes (2 to 90 instances, 2 to 4 plans, 96^2 to 1024 x 768) differ less between the two limits
// than between two runs.
bool z_small(const Geom& g, int nb, int tpl, int groups) {
  if (g.small == 0) return false;
  return g.small == 2 || (int64_t)(g.rows / 2) * tpl * nb * groups <= (g.small == 3 ? 75000 : 150000);
}

#define KW_DECL4(RET, NAME, ...) \
  RET NAME##_g0(__VA_ARGS__, bool*); RET NAME##_g1(__VA_ARGS__, bool*); RET NAME##_g2(__VA_ARGS__, bool*); RET NAME##_g3(__VA_ARGS__, bool*);
#define KW_TRY4(NAME, ...)                                    \
  do {                                                        \
    bool h = false;                                           \
    hipError_t e = NAME##_g0(__VA_ARGS__, &h); if (h) return e; \
    e = NAME##_g1(__VA_ARGS__, &h); if (h) return e;            \
    e = NAME##_g2(__VA_ARGS__, &h); if (h) return e;            \
    e = NAME##_g3(__VA_ARGS__, &h); if (h) return e;            \
    return hipErrorInvalidValue;                              \
  } while (0)

KW_DECL4(hipError_t, launch_zfwd, const Geom&, int, const float*, int64_t, float2*, int64_t, const float2*, hipStream_t)
KW_DECL4(hipError_t, launch_zinv, const Geom&, int, const float2*, int64_t, float*, int64_t, const float2*, float, hipStream_t)
KW_DECL4(hipError_t, launch_init_u, const Geom&, int, const Fields&, const Inst*, const float2*, hipStream_t)
KW_DECL4(hipError_t, launch_src_build, const Geom&, int, const Fields&, const Inst*, const float2*, int, hipStream_t)
KW_DECL4(hipError_t, launch_momentum, const Geom&, int, const Fields&, const Inst*, const float2*, hipStream_t)
KW_DECL4(hipError_t, launch_mass, const Geom&, int, const Fields&, const Inst*, const float2*, int, hipStream_t, bool)
KW_DECL4(hipError_t, launch_eos, const Geom&, int, const Fields&, const Inst*, const float2*, int, hipStream_t)
KW_DECL4(hipError_t, launch_col, const Geom&, int, const Fields&, const Ops&, const Inst*, const ColArgs&, int, hipStream_t)
KW_DECL4(hipError_t, launch_adj_eos, const Geom&, int, const Fields&, const AdjFields&, const Inst*, const float2*, int, hipStream_t)
KW_DECL4(hipError_t, launch_adj_mom, const Geom&, int, const Fields&, const AdjFields&, const Inst*, const float2*, int, hipStream_t)
KW_DECL4(hipError_t, launch_adj_abs1, const Geom&, int, const Fields&, const AdjFields&, const Inst*, const float2*, hipStream_t)
KW_DECL4(hipError_t, launch_adj_sum, const Geom&, int, const Fields&, const AdjFields&, const Inst*, const float2*, hipStream_t)

hipError_t launch_zfwd(const Geom& g, int nb, const float* f, int64_t fs, float2* spec, int64_t ss, const float2* tw, hipStream_t st) {
  if (generic_z(g)) return launch_zfwd_gen(g, nb, f, fs, spec, ss, tw, st);
  KW_TRY4(launch_zfwd, g, nb, f, fs, spec, ss, tw, st);
}
hipError_t launch_zinv(const Geom& g, int nb, const float2* spec, int64_t ss, float* f, int64_t fs, const float2* tw, float scale, hipStream_t st) {
  if (generic_z(g)) return launch_zinv_gen(g, nb, spec, ss, f, fs, tw, scale, st);
  KW_TRY4(launch_zinv, g, nb, spec, ss, f, fs, tw, scale, st);
}
hipError_t launch_init_u(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, hipStream_t st) {
  if (generic_z(g)) return launch_init_u_gen(g, nb, fl, inst, tw, st);
  KW_TRY4(launch_init_u, g, nb, fl, inst, tw, st);
}
hipError_t launch_src_build(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, int which, hipStream_t st) {
  if (generic_z(g)) return launch_src_build_gen(g, nb, fl, inst, tw, which, st);
  KW_TRY4(launch_src_build, g, nb, fl, inst, tw, which, st);
}
hipError_t launch_momentum(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, hipStream_t st) {
  if (generic_z(g)) return launch_momentum_gen(g, nb, fl, inst, tw, st);
  KW_TRY4(launch_momentum, g, nb, fl, inst, tw, st);
}
hipError_t launch_mass(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, int flags, hipStream_t st, bool sreg) {
  if (generic_z(g)) return launch_mass_gen(g, nb, fl, inst, tw, flags, st);
  KW_TRY4(launch_mass, g, nb, fl, inst, tw, flags, st, sreg);
}
hipError_t launch_eos(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, int flags, hipStream_t st) {
  if (generic_z(g)) return launch_eos_gen(g, nb, fl, inst, tw, flags, st);
  KW_TRY4(launch_eos, g, nb, fl, inst, tw, flags, st);
}
hipError_t launch_col(const Geom& g, int nb, const Fields& fl, const Ops& ops, const Inst* inst, const ColArgs& a, int nline, hipStream_t st) {
  if (!compiled_size(nline)) return launch_col_gen(g, nb, fl, ops, inst, a, nline, st);
  KW_TRY4(launch_col, g, nb, fl, ops, inst, a, nline, st);
}

hipError_t launch_adj_eos(const Geom& g, int nb, const Fields& fl, const AdjFields& af, const Inst* inst, const float2* tw, int t, hipStream_t st) {
  if (generic_z(g)) return launch_adj_eos_gen(g, nb, fl, af, inst, tw, t, st);
  KW_TRY4(launch_adj_eos, g, nb, fl, af, inst, tw, t, st);
}
hipError_t launch_adj_mom(const Geom& g, int nb, const Fields& fl, const AdjFields& af, const Inst* inst, const float2* tw, int t, hipStream_t st) {
  if (generic_z(g)) return launch_adj_mom_gen(g, nb, fl, af, inst, tw, t, st);
  KW_TRY4(launch_adj_mom, g, nb, fl, af, inst, tw, t, st);
}
hipError_t launch_adj_abs1(const Geom& g, int nb, const Fields& fl, const AdjFields& af, const Inst* inst, const float2* tw, hipStream_t st) {
  if (generic_z(g)) return launch_adj_abs1_gen(g, nb, fl, af, inst, tw, st);
  KW_TRY4(launch_adj_abs1, g, nb, fl, af, inst, tw, st);
}
hipError_t launch_adj_sum(const Geom& g, int nb, const Fields& fl, const AdjFields& af, const Inst* inst, const float2* tw, hipStream_t st) {
  if (generic_z(g)) return launch_adj_sum_gen(g, nb, fl, af, inst, tw, st);
  KW_TRY4(launch_adj_sum, g, nb, fl, af, inst, tw, st);
}

}  // namespace kw
