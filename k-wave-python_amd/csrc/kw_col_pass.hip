// Strided-axis (column) pass launcher of one size family (compiled once per
// family, -DKW_GROUP=0..3; see kw_kernels.hpp).
#include <algorithm>
#include <mutex>

#include "kw_host.hpp"
#include "kw_kernels.hpp"

namespace kw {

constexpr int kColDevices = 64;

// Workgroups of k_col<S, L, OPS> resident on the current device at once, at most
// `most` per compute unit (0 if the runtime cannot say).  Queried once per kernel and device.
template <int S, int L, bool OPS, int PV>
static int col_resident(int most) {
  static std::mutex mu;
  static struct { int per_cu, cus; } per_dev[kColDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kColDevices) return 0;
  std::lock_guard<std::mutex> lock(mu);
  auto& d = per_dev[dev];
  if (d.per_cu == 0 && (hipOccupancyMaxActiveBlocksPerMultiprocessor(&d.per_cu, reinterpret_cast<const void*>(&k_col<S, L, OPS, 1, PV>),
                                                                     ColCfg<S, L, 1, PV>::NT, 0) != hipSuccess ||
                        hipDeviceGetAttribute(&d.cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || d.per_cu <= 0))
    d.per_cu = -1;
  return d.per_cu > 0 ? std::min(d.per_cu, most) * d.cus : 0;
}

// Workgroups per instance of a column pass: every tile its own workgroup, or -
// when the tiles of all instances exceed what is resident at once - a resident
// grid (a multiple of the 8 XCDs) whose workgroups loop over tiles and load the
// next tile's input during the current one.  a.persist selects the passes that
// loop (bit 0 those with spectral jobs, bit 1 the FFT-only ones); a.grid > 0
// sets the looping grid (tests).  Results do not depend on either: every column
// is transformed the same way.
//
// FFT-only passes over lengths with a factor 3 (E = 12) loop on three waves a SIMD, not the four
// their registers allow, once a buffer exceeds 27 MB (the L2s hold 32).  us a y-pass, four ->
// three: 384^3 280 -> 258, 192^3 39.0 -> 36.7, 256 x 384 x 128 68 -> 64, 512 x 48 x 512 55 -> 48,
// 256 x 192 x 160 42.5 -> 36.8, 512 x 96 x 256 56.5 -> 58.4; below, 64 x 192 x 512 (25 MB)
// 27.9 -> 33.3, 96 x 96 x 512 21.0 -> 23.5.  With a factor 5 three lose (320^3 149 -> 173).
template <int S, int L, bool OPS, int PV>
static int col_grid(const ColArgs& a, int tiles, int nb) {
  using C = ColCfg<S, L, 1, PV>;
  if (!(a.persist & (OPS ? 1 : 2))) return tiles;
  if (a.grid > 0) return std::min(tiles, a.grid);
  const bool three = !OPS && C::E == 12 && (int64_t)sizeof(float2) * a.nouter * a.ncols * S * nb > 27000000;
  const int res = col_resident<S, L, OPS, PV>(three ? std::max(1, 12 * 64 / C::NT) : 1 << 20);
  if (res <= 0 || (int64_t)tiles * nb <= res) return tiles;
  const int per = std::max(8, (res / nb) & ~7);
  return std::min(tiles, per);
}

// One launch at tile width LW: wide tiles when they still give at least 1024
// workgroups (or a.wide is set), the narrow col_lsmall width otherwise (small grids).
template <int S, int LW, bool OPS, int PV>
static hipError_t col_launch_v(const Geom& g, int nb, const Fields& fl, const Ops& ops, const Inst* inst, const ColArgs& a,
                               hipStream_t st) {
  constexpr int LS = col_lsmall<S>();
  const int ntw = (a.ncols + LW - 1) / LW;
  if ((int64_t)a.nouter * nb * ntw >= 1024 || LW == LS || a.wide) {
    const int gx = col_grid<S, LW, OPS, PV>(a, a.nouter * ntw, nb);
    const ColArgs al = col_blocks(a, gx);
    hipLaunchKernelGGL((k_col<S, LW, OPS, 1, PV>), dim3(col_gridx(al, ColCfg<S, LW, 1, PV>::NT), nb), dim3(ColCfg<S, LW, 1, PV>::NT), 0, st, g, fl, ops, inst, al);
  } else {
    const int nt = (a.ncols + LS - 1) / LS;
    const int gx = col_grid<S, LS, OPS, PV>(a, a.nouter * nt, nb);
    const ColArgs al = col_blocks(a, gx);
    hipLaunchKernelGGL((k_col<S, LS, OPS, 1, PV>), dim3(col_gridx(al, ColCfg<S, LS, 1, PV>::NT), nb), dim3(ColCfg<S, LS, 1, PV>::NT), 0, st, g, fl, ops, inst, al);
  }
  return hipGetLastError();
}

// The small-grid form (k_col_small) where it applies: plan variant 0, the default
// tile choice, few enough jobs, all groups' exchange buffers within 64 KiB.
template <int S, bool OPS>
static bool col_small_fits(const ColArgs& a) {
  using C = ColCfg<S, col_lsmall2<S>()>;
  const int groups = OPS ? a.njob : 1;
  return groups <= (OPS ? kColSmallJobs : 1) && groups * C::NT <= 1024 && sizeof(float2) * C::LDS * groups <= 65536;
}
template <int S, bool OPS>
static hipError_t col_launch_small(const Geom& g, int nb, const Fields& fl, const Ops& ops, const Inst* inst, const ColArgs& a,
                                   hipStream_t st) {
  constexpr int L = col_lsmall2<S>();
  using C = ColCfg<S, L>;
  const int groups = OPS ? a.njob : 1;
  const ColArgs al = col_blocks(a, a.nouter * ((a.ncols + L - 1) / L));
  const dim3 grid(col_gridx(al, C::NT * groups), nb, OPS ? 1 : a.nbuf);
  hipLaunchKernelGGL((k_col_small<S, L, OPS>), grid, dim3(C::NT * groups), sizeof(float2) * C::LDS * groups, st, g, fl, ops, inst, al);
  return hipGetLastError();
}

// the plan variant a.pv where the length has one, variant 0 otherwise
template <int S, int LW, bool OPS>
static hipError_t col_launch(const Geom& g, int nb, const Fields& fl, const Ops& ops, const Inst* inst, const ColArgs& a,
                             hipStream_t st) {
  if constexpr (has_plan_variant(S)) {
    if (a.pv && a.small < 2) return col_launch_v<S, LW, OPS, 1>(g, nb, fl, ops, inst, a, st);
  }
  if (a.small && col_small_fits<S, OPS>(a)) {
    if (a.small == 2 || col_small_lanes(a, S, nb) <= kColSmallLanes) return col_launch_small<S, OPS>(g, nb, fl, ops, inst, a, st);
  }
  return col_launch_v<S, LW, OPS, 0>(g, nb, fl, ops, inst, a, st);
}

template <int W>
constexpr int half_width() { return W / 2 < 1 ? 1 : W / 2; }

// Tile widths: FFT-only passes col_lbig or half of it, passes with spectral jobs
// col_lops or half of it (a.tile selects; the plan picks by timing both).
hipError_t KW_GNAME(launch_col)(const Geom& g, int nb, const Fields& fl, const Ops& ops, const Inst* inst, const ColArgs& a, int nline, hipStream_t st, bool* handled) {
#define KW_C(S)                                                                                                          \
  case S:                                                                                                                \
    if (a.mode == 2)                                                                                                     \
      return a.tile ? col_launch<S, half_width<col_lops<S>()>(), true>(g, nb, fl, ops, inst, a, st)                      \
                    : col_launch<S, col_lops<S>(), true>(g, nb, fl, ops, inst, a, st);                                   \
    return a.tile ? col_launch<S, half_width<col_lbig<S>()>(), false>(g, nb, fl, ops, inst, a, st)                       \
                  : col_launch<S, col_lbig<S>(), false>(g, nb, fl, ops, inst, a, st);
  *handled = true;
  switch (nline) {
    KW_GROUP_SIZES(KW_C)
    default: *handled = false; return hipSuccess;
  }
#undef KW_C
  return hipGetLastError();
}

}  // namespace kw
