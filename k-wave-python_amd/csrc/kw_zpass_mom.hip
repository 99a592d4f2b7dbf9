// Momentum launcher of one size family (compiled once per family, -DKW_GROUP=0..3).
#include "kw_kernels.hpp"

namespace kw {

hipError_t KW_GNAME(launch_momentum)(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, hipStream_t st, bool* handled) {
#define KW_C(S)                                                                                                          \
  case S:                                                                                                                \
    if (z_small(g, nb, ZCfg<S>::TPL, g.nd))                                                                              \
      hipLaunchKernelGGL(k_momentum_small<S>, zgrid(g, ZCfg<S, true>::L, nb, g.nd), dim3(ZCfg<S, true>::NT), 0, st, g, fl, inst, tw); \
    else                                                                                                                 \
      hipLaunchKernelGGL(k_momentum<S>, zgrid(g, ZCfg<S>::L, nb, g.nd), dim3(ZCfg<S>::NT), 0, st, g, fl, inst, tw);      \
    break;
  KW_ZDISPATCH(KW_C)
#undef KW_C
  return hipGetLastError();
}

}  // namespace kw
