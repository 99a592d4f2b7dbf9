// Momentum launcher of one size family (compiled once per family, -DKW_GROUP=0..3).
#include "kw_kernels.hpp"

namespace kw {

// Real elements of a launch above which k_momentum stages its tables before it loads its
// operands.  While an axis's u, dt/rho0 and spectrum stay in the caches its time is latency,
// and all loads at once win; from memory the rate decides, and loads that start behind the
// tables win.  us, all at once -> staged: 192^3 80 -> 87, 256 x 256 x 192 136 -> 142 (12.6 M
// elements); 256^3 (16.8 M) 194 -> 191, 384^3 805 -> 785, 640 x 512 x 256 1195 -> 1144, 512^3
// 1840 -> 1755.
constexpr int64_t kMomStaged = 14000000;

hipError_t KW_GNAME(launch_momentum)(const Geom& g, int nb, const Fields& fl, const Inst* inst, const float2* tw, hipStream_t st, bool* handled) {
#define KW_C(S)                                                                                                          \
  case S:                                                                                                                \
    if (z_small(g, nb, ZCfg<S>::TPL, g.nd))                                                                              \
      hipLaunchKernelGGL(k_momentum_small<S>, zgrid(g, ZCfg<S, true>::L, nb, g.nd), dim3(ZCfg<S, true>::NT), 0, st, g, fl, inst, tw); \
    else if (nb * g.ntot > kMomStaged)                                                                                   \
      hipLaunchKernelGGL((k_momentum<S, true>), zgrid(g, ZCfg<S>::L, nb, g.nd), dim3(ZCfg<S>::NT), 0, st, g, fl, inst, tw); \
    else                                                                                                                 \
      hipLaunchKernelGGL((k_momentum<S, false>), zgrid(g, ZCfg<S>::L, nb, g.nd), dim3(ZCfg<S>::NT), 0, st, g, fl, inst, tw); \
    break;
  KW_ZDISPATCH(KW_C)
#undef KW_C
  return hipGetLastError();
}

}  // namespace kw
