// Time-loop kernels of the k-space pseudospectral solver (gfx950).
//
// Every kernel works on a *batch* of same-shape instances (blockIdx.y is the
// instance) and reads the instance's step counter from device memory, so that
// one captured sequence serves every step and finished instances drop out.
//
// z-pass kernels own the contiguous axis: a workgroup takes L pairs of grid
// rows, runs the real<->half-complex transform of both rows of a pair as one
// complex FFT (row a in the real part, row b in the imaginary part), and fuses
// the pointwise physics of the step between the inverse and forward transforms.
// Column kernels own the strided axes; the outermost-axis pass applies the
// spectral multipliers (regenerated in registers from 1-D tables) between its
// forward and inverse transforms.
#pragma once
#include "kw_fft.hpp"
#include "kw_launch.hpp"
#include "kw_types.hpp"

namespace kw {

// ---------------------------------------------------------------------------
// z-pass configuration
// ---------------------------------------------------------------------------
constexpr int pow2floor(int v) {
  int p = 1;
  while (p * 2 <= v) p *= 2;
  return p;
}
constexpr int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

#ifndef KW_ZPV
#define KW_ZPV 0
#endif
// NAR: the narrow form of small grids, one wavefront per workgroup (or per group of
// lanes of a workgroup) where the line length leaves a wavefront room for it.
template <int N_, bool NAR = false>
struct ZCfg {
  static constexpr int N = N_;
  // radix plan of the row passes: KW_ZPV=2 selects the radix-4 plan (4 elements per
  // thread) for power-of-two lengths
  static constexpr int PV = (KW_ZPV == 2 && (N & (N - 1)) == 0) ? 2 : 0;
  using F = FftShape<N, 1, PV>;
  static constexpr int E = F::E;
  static constexpr int TPL = F::TPL;
  static constexpr int L0 = clampi(pow2floor(2048 / N), 1, 64);
  static constexpr int L = NAR ? clampi(64 / TPL, 1, 64) : (L0 * TPL < 64) ? clampi(64 / TPL, L0, 64) : L0;  // row pairs per workgroup
  static constexpr int NT = TPL * L;
  static constexpr bool WS = NAR && NT == 64;  // lines_sync without workgroup barriers
  static constexpr int NH = N / 2 + 1;
  static constexpr int IT = (L * NH + NT - 1) / NT;  // spectrum values of a row per thread
  using Idx = RowIdx<N>;
  static constexpr int LDS = Idx::size(L);
};

// Global-memory views of pointers.  Pointers read from parameter blocks are
// generic to the compiler, and generic (flat) loads also count against the LDS
// wait counter, so every LDS wait inside a transform would drain them too; the
// global view keeps them on the vector-memory counter alone.
#define KW_AS1 __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ const KW_AS1 T* gp(const T* p) { return (const KW_AS1 T*)p; }
template <class T>
__device__ __forceinline__ KW_AS1 T* gw(T* p) { return (KW_AS1 T*)p; }
// float2 through a global view, by components (the vector type's members take
// generic references)
__device__ __forceinline__ float2 ld2(const KW_AS1 float2* p, int64_t i) {
  const KW_AS1 float2& v = p[i];
  return make_float2(v.x, v.y);
}
__device__ __forceinline__ void st2(KW_AS1 float2* p, int64_t i, float2 v) {
  KW_AS1 float2& d = p[i];
  d.x = v.x;
  d.y = v.y;
}

__device__ __forceinline__ float ld(const float* p, int64_t i, int s) { return gp(p)[i * s]; }

// step an instance is at
__device__ __forceinline__ int step_of(const Fields& fl, int b) { return gp(fl.tdev)[b] + fl.toff; }

// Record sensor s of instance b at step t: interpolated pressure and velocities, running
// maximum, minimum and sum of squares.
__device__ __forceinline__ void gather_point(const Geom& g, const Fields& fl, const Inst& I, int b, int t, int s) {
  if (I.sens_kind == 0 || t >= I.nt || t < I.rec_start || s >= I.nsens) return;
  const int64_t off = b * g.ntot;
  const int64_t row = (int64_t)(t - I.rec_start) * I.nsens + s;
  auto sample = [&](const float* f) {
    float acc = 0.f;
    for (int c = 0; c < I.ncorner; ++c) {
      const int64_t ii = I.sidx[(int64_t)s * I.ncorner + c];
      const float w = I.sens_kind == 2 ? I.sw[(int64_t)s * I.ncorner + c] : 1.f;
      acc += w * f[off + ii];
    }
    return acc;
  };
  if (I.rec_p || I.agg_p) {
    const float v = sample(fl.p);
    if (I.rec_p) I.rec_p[row] = v;
    if (I.agg_p) {
      float* a = I.agg_p;
      if (t == I.rec_start) { a[s] = v; a[I.nsens + s] = v; a[2 * I.nsens + s] = v * v; }
      else { a[s] = fmaxf(a[s], v); a[I.nsens + s] = fminf(a[I.nsens + s], v); a[2 * I.nsens + s] += v * v; }
    }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (i >= g.nd) continue;
    if (I.rec_u[i]) I.rec_u[i][row] = sample(fl.u[i]);
    if (I.rec_uc[i]) I.rec_uc[i][row] = sample(fl.uc[i]);
  }
}
// The workgroups a column pass has beyond its own (ColArgs::gath): the sensors of the step
// before, whose fields nothing changes before the next update.  A kernel of its own would
// add its launch and one chain of latencies, 4 to 5 us, to every step (with the counter
// advanced once a block as well, us per step: 128^2 30.0 -> 25.7, 512^2 power law 51.3 ->
// 48.4, 64 maps of 128^2 58.5 -> 54.7).  Up to kGatherInPass sensors (kw_abi.hip).
__device__ __forceinline__ void gather_blocks(const Geom& g, const Fields& fl, const Inst* inst, const ColArgs& a) {
  if (blockIdx.z) return;
  const int b = blockIdx.y;
  gather_point(g, fl, inst[b], b, step_of(fl, b) - 1, ((int)blockIdx.x - a.gx) * (int)blockDim.x + (int)threadIdx.x);
}

// absorption / dispersion coefficient at idx given c0^2 there
__device__ __forceinline__ float tau_at(const Inst& I, int64_t idx, float c2) {
  return I.tau ? ld(I.tau, idx, I.tau_s) : I.tau_c * exp2f(I.ym1h * log2f(c2));
}
__device__ __forceinline__ float eta_at(const Inst& I, int64_t idx, float c2) {
  return I.eta ? ld(I.eta, idx, I.eta_s) : I.eta_c * exp2f(I.yh * log2f(c2));
}

// pml value of axis `ax` at grid row r, contiguous position n
__device__ __forceinline__ float pml_at(const float* const* tab, const Geom& g, int ax, int r, int n) {
  if (ax == g.nd - 1) return gp(tab[ax])[n];
  if (ax == 0) return gp(tab[0])[g.nd == 2 ? r : r / g.n[1]];
  return gp(tab[1])[r % g.n[1]];
}

// Load the half spectra of the L row pairs of this workgroup into LDS as the
// full spectrum of z = a + i b (Hermitian extension of each half spectrum).  All of
// a thread's loads (pair_load) are issued before its first LDS write (pair_put), so
// their latencies overlap instead of adding up.
template <class C>
__device__ __forceinline__ void pair_put(float2* lds, const float2 (&As)[C::IT], const float2 (&Bs)[C::IT], int tid) {
  constexpr int N = C::N;
  const typename C::Idx idx{};
#pragma unroll
  for (int it = 0; it < C::IT; ++it) {
    const int e = tid + it * C::NT;
    if ((it + 1) * C::NT > C::L * C::NH && e >= C::L * C::NH) break;
    const int p = e / C::NH, k = e % C::NH;
    const float2 A = As[it], B = Bs[it];
    // the self-conjugate columns 0 and N/2 keep their real parts (both writes go to one slot)
    const bool self = k == 0 || (N % 2 == 0 && k == N / 2);
    const float2 lo = self ? make_float2(A.x, B.x) : make_float2(A.x - B.y, A.y + B.x);
    const float2 hi = self ? lo : make_float2(A.x + B.y, B.x - A.y);
    lds[idx(k, p)] = lo;
    lds[idx(k == 0 ? 0 : N - k, p)] = hi;
  }
}

// Rows (even in number) and columns are clamped into the grid rather than tested: a test
// puts every load into a block of its own, which the compiler then waits for one by one.
// What the clamped lanes read belongs to lines that are never stored.
template <class C>
__device__ __forceinline__ void pair_load(float2 (&As)[C::IT], float2 (&Bs)[C::IT], const float2* __restrict__ spec_, int row0, int rows,
                                          int pitch, int tid) {
  const auto spec = gp(spec_);
#pragma unroll
  for (int it = 0; it < C::IT; ++it) {
    const int e = min(tid + it * C::NT, C::L * C::NH - 1);
    const int p = e / C::NH, k = e % C::NH;
    const int ra = min(row0 + 2 * p, rows - 2);
    As[it] = ld2(spec, (int64_t)ra * pitch + k);
    Bs[it] = ld2(spec, (int64_t)(ra + 1) * pitch + k);
  }
}

// After a forward FFT of z = a + i b (in LDS), split into the two half spectra.
template <class C>
__device__ __forceinline__ void store_pair_spec(const float2* lds, float2* __restrict__ spec_, int row0, int rows, int pitch, int tid) {
  constexpr int N = C::N;
  const auto spec = gw(spec_);
  const typename C::Idx idx{};
  float2 Z[C::IT], Zc[C::IT];
#pragma unroll
  for (int it = 0; it < C::IT; ++it) {
    const int e = min(tid + it * C::NT, C::L * C::NH - 1);
    const int p = e / C::NH, k = e % C::NH;
    Z[it] = lds[idx(k, p)];
    Zc[it] = lds[idx(k == 0 ? 0 : N - k, p)];
  }
#pragma unroll
  for (int it = 0; it < C::IT; ++it) {
    const int e = tid + it * C::NT;
    const int p = e / C::NH, k = e % C::NH;
    const int ra = row0 + 2 * p;  // both rows of a pair are inside the grid, or neither
    if (((it + 1) * C::NT <= C::L * C::NH || e < C::L * C::NH) && ra < rows) {
      st2(spec, (int64_t)ra * pitch + k, make_float2(0.5f * (Z[it].x + Zc[it].x), 0.5f * (Z[it].y - Zc[it].y)));
      st2(spec, (int64_t)(ra + 1) * pitch + k, make_float2(0.5f * (Z[it].y + Zc[it].y), -0.5f * (Z[it].x - Zc[it].x)));
    }
  }
}

// full spectra of row pairs in LDS -> real values of both rows at the owned positions
template <class C>
__device__ __forceinline__ void inv_from_lds(float2* lds, const float2* __restrict__ tw, int tid, float2 (&out)[C::E]) {
  const typename C::Idx idx{};
  const int j0 = tid % C::TPL, c = tid / C::TPL;
  line_sync<C::WS>();
#pragma unroll
  for (int m = 0; m < C::E; ++m) out[m] = lds[idx(j0 + m * C::TPL, c)];
  line_sync<C::WS>();
  fft_reg<C::N, +1, typename C::Idx, 1, C::PV, C::WS>(out, lds, tw, c, j0, idx);
}

// half spectra of a row pair -> real values of both rows at the owned positions
template <class C>
__device__ __forceinline__ void inv_to_regs(float2* lds, const float2* __restrict__ spec, const float2* __restrict__ tw,
                                            int row0, int rows, int pitch, int tid, float2 (&out)[C::E]) {
  float2 As[C::IT], Bs[C::IT];
  pair_load<C>(As, Bs, spec, row0, rows, pitch, tid);
  line_sync<C::WS>();
  pair_put<C>(lds, As, Bs, tid);
  inv_from_lds<C>(lds, tw, tid, out);
}

// real values of a row pair at the owned positions -> half spectra of both rows
// (stored where `store` holds)
template <class C>
__device__ __forceinline__ void fwd_from_regs(float2* lds, float2 (&v)[C::E], float2* __restrict__ spec,
                                              const float2* __restrict__ tw, int row0, int rows, int pitch, int tid, bool store = true) {
  const typename C::Idx idx{};
  const int j0 = tid % C::TPL, c = tid / C::TPL;
  fft_reg<C::N, -1, typename C::Idx, 1, C::PV, C::WS>(v, lds, tw, c, j0, idx);
  line_sync<C::WS>();
#pragma unroll
  for (int m = 0; m < C::E; ++m) lds[idx(j0 + m * C::TPL, c)] = v[m];
  line_sync<C::WS>();
  if (store) store_pair_spec<C>(lds, spec, row0, rows, pitch, tid);
  // leave the buffer free: a following transform writes it in its first stage
  // while slower waves could still be reading the pair spectra here
  line_sync<C::WS>();
}

// Source value added/imposed at (row r, position n) for a CSR source term.
// Returns true when (r, n) is a source point; v receives scale * signal(t).
__device__ __forceinline__ bool csr_lookup(const Src& s, int r, int n, int t, float& v) {
  int lo = gp(s.row_ptr)[r], hi = gp(s.row_ptr)[r + 1];
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    const int c = gp(s.col)[mid];
    if (c == n) {
      v = gp(s.scale)[mid] * gp(s.sig)[(int64_t)gp(s.sigrow)[mid] * s.len + t];
      return true;
    }
    if (c < n) lo = mid + 1; else hi = mid;
  }
  return false;
}

// Filtered sources: the dense pattern (PATTERN, value sig(t) * pattern) and the
// inverse transform of the multi-row source's spectrum (CHAIN).  mode is SRC_NONE once
// the signal has ended.  The point-source modes (DIRICHLET, NOCORR) are applied
// afterwards by a rolled pass over the owned source points, which keeps their lookup
// out of the unrolled code.
__device__ __forceinline__ int src_mode_at(const Src& s, int t) { return t < s.len ? s.mode : SRC_NONE; }
__device__ __forceinline__ float src_inline(const Src& s, int mode, float f, int64_t idx, float fac, float sig_t, float chv) {
  if (mode == SRC_PATTERN) return fmaf(fac, sig_t * gp(s.pattern)[idx], f);
  if (mode == SRC_CHAIN) return fmaf(fac, chv, f);
  return f;
}
// the source values at a thread's elements (iA: its first element)
template <class C>
__device__ __forceinline__ void filtered_source(const Src& s, int mode, int t, int64_t iA, float2* lds, const Fields& fl, const Geom& g, int b,
                                                const float2* tw, int row0, int rows, int tid, float2 (&ch)[C::E]) {
  if (mode == SRC_CHAIN) {
    inv_to_regs<C>(lds, fl.spec[s.chain_buf] + b * g.nspec, tw, row0, rows, g.nhp, tid, ch);
  } else {
    const float sig_t = gp(s.sig)[t];
    const auto pat = gp(s.pattern);
#pragma unroll
    for (int m = 0; m < C::E; ++m) ch[m] = make_float2(sig_t * pat[iA + m * C::TPL], sig_t * pat[iA + C::N + m * C::TPL]);
  }
}
template <class C>
__device__ __forceinline__ void add_filtered_source(const Src& s, int mode, int t, float fac, int64_t iA, float2* lds, const Fields& fl,
                                                    const Geom& g, int b, const float2* tw, int row0, int rows, int tid, float2 (&v)[C::E]) {
  if (mode != SRC_CHAIN && mode != SRC_PATTERN) return;
  float2 ch[C::E];
  filtered_source<C>(s, mode, t, iA, lds, fl, g, b, tw, row0, rows, tid, ch);
#pragma unroll
  for (int m = 0; m < C::E; ++m) v[m] = make_float2(fmaf(fac, ch[m].x, v[m].x), fmaf(fac, ch[m].y, v[m].y));
}
__device__ __forceinline__ bool src_is_point(int mode) { return mode == SRC_DIRICHLET || mode == SRC_NOCORR; }
__device__ __forceinline__ float src_point(int mode, float f, float fac, float v) { return mode == SRC_DIRICHLET ? fac * v : fmaf(fac, v, f); }

// PML-weighted update of a velocity or split-density component, s (s f - a b); the fused
// multiply-add is spelled out so that every form of a step rounds alike (kw_fft.hpp, cmul).
__device__ __forceinline__ float pml_update(float s, float f, float a, float b) { return s * fmaf(s, f, -(a * b)); }
// A value other terms are added to is rounded here, not contracted into the addition.
__device__ __forceinline__ void rounded(float& v) { asm("" : "+v"(v)); }

// Register-array element (m, h) with a run-time m (selects, no indexed registers).
template <int E>
__device__ __forceinline__ float get_lane(const float2 (&a)[E], int m, int h) {
  float v = 0.f;
#pragma unroll
  for (int k = 0; k < E; ++k)
    if (k == m) v = h ? a[k].y : a[k].x;
  return v;
}
template <int E>
__device__ __forceinline__ void set_lane(float2 (&a)[E], int m, int h, float v) {
#pragma unroll
  for (int k = 0; k < E; ++k)
    if (k == m) { if (h) a[k].y = v; else a[k].x = v; }
}

// Minimum waves per SIMD the register allocator must leave room for (kernels
// with short register arrays only; 1 = unconstrained).  Measured at 512^3: every
// floor that forces spills loses (the mass kernel forced from 2 waves to 3 spilled 23
// registers, 2155 -> 2948 us; the momentum kernel forced from 3 to 4, 1904 -> 2808 us).
//
// What bounds the updates on large grids is memory (512^3: mass 1686 us = 4.5 TB/s of
// its algorithmic bytes, eos 811 us = 4.6, momentum 1750 us = 4.6; a plain copy reaches
// 5.0), once their loads are issued in batches: element loops with a test inside (the
// nonlinear flag, a source mode, a clamped row) had compiled into one block per element,
// each load waited for alone.  Straight-line loops with the tests around them took the
// mass kernel from 1970 to 1686 us at 512^3 and from 264 to 187 us at 256^3, eos from 902
// to 811 and from 126 to 102 us, momentum from 198 to 186 us at 256^3, and 256^3 steps from
// 1287 to 1159 us.  Momentum has a second order of its loads for larger grids (kMomStaged).
#ifndef KW_WPE_MOM
#define KW_WPE_MOM 1
#endif
#ifndef KW_WPE_MASS
#define KW_WPE_MASS 1
#endif
#ifndef KW_WPE_EOS
#define KW_WPE_EOS 1
#endif
#ifndef KW_WPE_COL
#define KW_WPE_COL 1
#endif
#ifndef KW_WPE_COLOPS
#define KW_WPE_COLOPS 4  // the prefetch of the next job input would take it to 130 VGPRs, 3 waves
#endif
#ifndef KW_COL_SMALL_MIN
#define KW_COL_SMALL_MIN 2
#endif
#define KW_WPE(N, W) __attribute__((amdgpu_waves_per_eu((FftShape<N>::E <= 8 ? (W) : 1))))

// Stage-ordered twiddles (kw_fft.hpp stage_tw_*) of an N-point plan from the
// natural table src[m] = exp(-2 pi i m / N), one stage at a time so that every
// index is a compile-time expression of the entry; loads (into registers) and LDS
// writes are separate, so that every load is in flight before the first write.
template <int N, int PV, int NT, int S = 1, int K = 0, int M>
__device__ __forceinline__ void load_stage_tw(float2 (&r)[M], const float2* src, int tid) {
  if constexpr (S < plan_nstages(N, PV)) {
    constexpr int R = plan_stage_radix(N, S, PV), NS = plan_ns_before(N, S, PV);
    constexpr int TWS = N / (NS * R), CNT = NS * (R - 1), IT = (CNT + NT - 1) / NT;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int e = min(tid + i * NT, CNT - 1);
      r[K + i] = ld2(gp(src), (e % (R - 1) + 1) * (e / (R - 1)) * TWS);
    }
    load_stage_tw<N, PV, NT, S + 1, K + IT>(r, src, tid);
  }
}
template <int N, int PV, int NT, int S = 1, int K = 0, int M>
__device__ __forceinline__ void put_stage_tw(const float2 (&r)[M], float2* dst, int tid) {
  if constexpr (S < plan_nstages(N, PV)) {
    constexpr int R = plan_stage_radix(N, S, PV), NS = plan_ns_before(N, S, PV);
    constexpr int B = stage_tw_base<N, PV>(S), CNT = NS * (R - 1), IT = (CNT + NT - 1) / NT;
#pragma unroll
    for (int i = 0; i < IT; ++i)
      if (tid + i * NT < CNT) dst[B + tid + i * NT] = r[K + i];
    put_stage_tw<N, PV, NT, S + 1, K + IT>(r, dst, tid);
  }
}
template <int N, int PV>
constexpr int stage_tw_loads(int nt) {
  int k = 0;
  for (int s = 1; s < plan_nstages(N, PV); ++s)
    k += (plan_ns_before(N, s, PV) * (plan_stage_radix(N, s, PV) - 1) + nt - 1) / nt;
  return k < 1 ? 1 : k;
}

#define KW_ZPASS_PROLOGUE KW_ZPASS_PROLOGUE_AS(ZCfg<N>)
#define KW_ZPASS_PROLOGUE_AS(...)                                      \
  using C = __VA_ARGS__;                                               \
  __shared__ float2 lds[C::LDS];                                       \
  __shared__ float2 twl[stage_tw_size<N, C::PV>()];                    \
  const int tid = threadIdx.x;                                         \
  {                                                                    \
    float2 twr_[stage_tw_loads<N, C::PV>(C::NT)];                      \
    load_stage_tw<N, C::PV, C::NT>(twr_, tw_g, tid);                   \
    put_stage_tw<N, C::PV, C::NT>(twr_, twl, tid);                     \
  }                                                                    \
  __syncthreads();                                                     \
  const float2* tw = twl;                                              \
  const int b = blockIdx.y;                                            \
  const int row0 = blockIdx.x * 2 * C::L;                              \
  const int rows = g.rows;                                             \
  const int j0 = tid % C::TPL, pc = tid / C::TPL;                      \
  const int ra = row0 + 2 * pc;                                        \
  (void)j0; (void)ra;

// The updates' prologue: the twiddles and the contiguous-axis PML (PTAB, or null) are
// loaded into registers here and put into LDS by KW_ZPASS_PUT, once the kernel has
// issued the loads of its operands and first spectrum (the transform's first barrier
// publishes them).
#define KW_ZPASS_EARLY(PTAB)                                           \
  using C = ZCfg<N>;                                                   \
  __shared__ float2 lds[C::LDS];                                       \
  __shared__ float2 twl[stage_tw_size<N, C::PV>()];                    \
  __shared__ float pmlz[N];                                            \
  const int tid = threadIdx.x;                                         \
  const int b = blockIdx.y;                                            \
  const Inst& I = inst[b];                                             \
  float2 twr[stage_tw_loads<N, C::PV>(C::NT)];                         \
  load_stage_tw<N, C::PV, C::NT>(twr, tw_g, tid);                      \
  constexpr int PZ = (N + C::NT - 1) / C::NT;                          \
  float pzr[PZ];                                                       \
  const float* const ptab = PTAB;                                      \
  if (ptab) {                                                          \
    _Pragma("unroll") for (int i_ = 0; i_ < PZ; ++i_) pzr[i_] = gp(ptab)[min(tid + i_ * C::NT, N - 1)]; \
  }                                                                    \
  const float2* tw = twl;                                              \
  const int row0 = blockIdx.x * 2 * C::L;                              \
  const int rows = g.rows;                                             \
  const int j0 = tid % C::TPL, pc = tid / C::TPL;                      \
  const int ra = row0 + 2 * pc;                                        \
  (void)j0; (void)ra;
#define KW_ZPASS_PUT                                                   \
  put_stage_tw<N, C::PV, C::NT>(twr, twl, tid);                        \
  if (ptab) {                                                          \
    _Pragma("unroll") for (int i_ = 0; i_ < PZ; ++i_)                  \
      if (tid + i_ * C::NT < N) pmlz[tid + i_ * C::NT] = pzr[i_];      \
  }

// ---------------------------------------------------------------------------
// generic real <-> half-spectrum transforms along the contiguous axis
// ---------------------------------------------------------------------------
template <int N, bool NAR>
__global__ __launch_bounds__((ZCfg<N, NAR>::NT)) void k_zfwd(Geom g, const float* __restrict__ f, int64_t fstride, float2* __restrict__ spec,
                                                      int64_t sstride, const float2* __restrict__ tw_g) {
  KW_ZPASS_PROLOGUE_AS(ZCfg<N, NAR>)
  const auto fb = gp(f + b * fstride);
  float2 v[C::E];
  const int64_t iA = (int64_t)min(ra, rows - 2) * N + j0;  // row counts are even here
#pragma unroll
  for (int m = 0; m < C::E; ++m) v[m] = make_float2(fb[iA + m * C::TPL], fb[iA + N + m * C::TPL]);
  fwd_from_regs<C>(lds, v, spec + b * sstride, tw, row0, rows, g.nhp, tid);
}

template <int N, bool NAR>
__global__ __launch_bounds__((ZCfg<N, NAR>::NT)) void k_zinv(Geom g, const float2* __restrict__ spec, int64_t sstride, float* __restrict__ f,
                                                      int64_t fstride, const float2* __restrict__ tw_g, float scale) {
  KW_ZPASS_PROLOGUE_AS(ZCfg<N, NAR>)
  const auto fb = gw(f + b * fstride);
  float2 v[C::E];
  inv_to_regs<C>(lds, spec + b * sstride, tw, row0, rows, g.nhp, tid, v);
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int n = j0 + m * C::TPL;
    if (ra < rows) fb[(int64_t)ra * N + n] = scale * v[m].x;
    if (ra + 1 < rows) fb[(int64_t)(ra + 1) * N + n] = scale * v[m].y;
  }
}

// Element addressing shared by the step kernels.  A thread owns positions
// n = j0 + m * TPL of the two rows ra, ra + 1 of its pair.  Row counts are even,
// so both rows of a pair are inside the grid or both outside (tail workgroups of
// small grids); loads use rows clamped into the grid so that the unrolled
// element loops carry no branches and their loads issue together, and only the
// stores are guarded.  Values computed for rows outside the grid are never stored.
#define KW_ROWS_CLAMPED                                                          \
  const bool inside = ra < rows;                                                 \
  const int rA = min(ra, rows - 2);                                              \
  const int64_t iA = (int64_t)rA * N + j0; /* element (m, h): iA + h N + m TPL */

// pml multipliers of the rows of a thread along axis ax (1 for the contiguous axis)
__device__ __forceinline__ void pml_rows(const float* const* tab, const Geom& g, int ax, int rA, float (&ph)[2]) {
  if (ax == g.nd - 1) { ph[0] = ph[1] = 1.f; return; }
  ph[0] = pml_at(tab, g, ax, rA, 0);
  ph[1] = pml_at(tab, g, ax, rA + 1, 0);
}

// ---------------------------------------------------------------------------
// momentum: u_i = pml_sg (pml_sg u_i - dt/rho0_sg * grad_i p) (+ source), then
// forward transform of u_i along z (for the divergence).  blockIdx.z = axis.
// ---------------------------------------------------------------------------
// STAGED (rule kMomStaged): the tables are in LDS before the operands are loaded.
template <int N, bool STAGED>
__global__ __launch_bounds__(ZCfg<N>::NT) KW_WPE(N, KW_WPE_MOM) void k_momentum(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ tw_g) {
  const int ax = blockIdx.z;
  const bool zax = ax == g.nd - 1;
  KW_ZPASS_EARLY(!STAGED && zax ? inst[blockIdx.y].pmlsg[ax] : nullptr)
  const int t = step_of(fl, b);
  if constexpr (STAGED) {
    if (t >= I.nt) return;
    put_stage_tw<N, C::PV, C::NT>(twr, twl, tid);
    __syncthreads();
    if (zax)
      for (int i = tid; i < N; i += C::NT) pmlz[i] = gp(I.pmlsg[ax])[i];
  }
  KW_ROWS_CLAMPED
  float2* sp = fl.spec[ax] + b * g.nspec;
  const auto u = gw(fl.u[ax] + b * g.ntot);
  const Src& src = I.srcu[ax];
  float ph[2];
  pml_rows(I.pmlsg, g, ax, rA, ph);
  // operands of the update, fetched before the transform so their latency overlaps it
  float2 uo[C::E], dr[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    uo[m] = make_float2(u[i0], u[i0 + N]);
    dr[m] = make_float2(ld(I.dtr0[ax], i0, I.dtr0_s), ld(I.dtr0[ax], i0 + N, I.dtr0_s));
  }
  float2 gv[C::E], As[C::IT], Bs[C::IT];
  pair_load<C>(As, Bs, sp, row0, rows, g.nhp, tid);
  if constexpr (STAGED) {
    __syncthreads();
  } else {
    if (t >= I.nt) return;
    KW_ZPASS_PUT
  }
  pair_put<C>(lds, As, Bs, tid);
  inv_from_lds<C>(lds, tw, tid, gv);
  const int smode = src_mode_at(src, t);
  // straight-line element loops: a test inside would split them into blocks whose loads
  // and stores the compiler cannot move past each other
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const float sz = zax ? pmlz[j0 + m * C::TPL] : 1.f;
    gv[m].x = pml_update(sz * ph[0], uo[m].x, dr[m].x, gv[m].x);
    gv[m].y = pml_update(sz * ph[1], uo[m].y, dr[m].y, gv[m].y);
  }
  add_filtered_source<C>(src, smode, t, src.fac[ax], iA, lds, fl, g, b, tw, row0, rows, tid, gv);
  if (inside) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      u[iA + m * C::TPL] = gv[m].x;
      u[iA + N + m * C::TPL] = gv[m].y;
    }
  }
  if (src_is_point(smode) && inside) {
    for (int h = 0; h < 2; ++h) {
      const int r = ra + h;
      if (gp(src.row_ptr)[r] == gp(src.row_ptr)[r + 1]) continue;
      for (int m = 0; m < C::E; ++m) {
        const int n = j0 + m * C::TPL;
        float v;
        if (!csr_lookup(src, r, n, t, v)) continue;
        const float uv = src_point(smode, get_lane(gv, m, h), src.fac[ax], v);
        u[(int64_t)r * N + n] = uv;
        set_lane(gv, m, h, uv);
      }
    }
  }
  fwd_from_regs<C>(lds, gv, sp, tw, row0, rows, g.nhp, tid);
}

// ---------------------------------------------------------------------------
// mass conservation (+ equation of state when no fractional Laplacian is needed)
// SREG: the pressure source term is staged in registers once per element
// (CHAIN: the inverse transform of its filtered spectrum; PATTERN: sig(t) times
// the dense filtered pattern) and added to every split density from there.
// The other instantiation serves plans without such a source and the steps
// after the signal has ended.
// CAP: the adjoint replay of a nonlinear plan also keeps each axis's Dop_i u_i
// (Fields::adjD).  A template switch rather than a runtime test, so the
// stepping kernels' code, and with it their FP32 contractions, stays unchanged.
// ---------------------------------------------------------------------------
template <int N, int ND, bool SREG, bool CAP>
__global__ __launch_bounds__(ZCfg<N>::NT) KW_WPE(N, KW_WPE_MASS) void k_mass(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ tw_g, int flags) {
  KW_ZPASS_EARLY(inst[blockIdx.y].pml[ND - 1])
  const int t = step_of(fl, b);
  KW_ROWS_CLAMPED
  const int64_t off = b * g.ntot;
  const Src& src = I.srcp;
  const int smode = src_mode_at(src, t);
  const bool filtered = SREG && (smode == SRC_CHAIN || smode == SRC_PATTERN);
  const bool powerlaw = flags & (FLAG_POWERLAW_ABS | FLAG_POWERLAW_DISP);
  float ph[ND][2];
#pragma unroll
  for (int i = 0; i < ND; ++i) pml_rows(I.pml, g, i, rA, ph[i]);
  // per owned element and row: the coefficient dt (2 rho_old + rho0) of the
  // density update (dt rho0 when linear; rho_old = sum of the split densities
  // of the previous step, kept in rhot), and the running sums of div u and of
  // the new densities
  // rho0 stays in registers for the outputs at the end where that costs no occupancy (3-D,
  // power-of-two lengths: two waves per SIMD either way).  A re-read there misses L2 at
  // large grids, about 4 bytes per voxel of extra HBM traffic; the 2-D kernels would drop
  // from three waves per SIMD to two, the mixed-radix ones from two to one.
  constexpr bool R0R = ND == 3 && C::E <= 16 && (N & (N - 1)) == 0;
  // (Every loop below is straight-line over its elements, with tests around whole loops:
  // a test inside puts each load into a block of its own that is waited for alone.)
  float2 qv[C::E], divu[C::E], rt[C::E], r0v[R0R ? C::E : 1];
  float2 ch[SREG ? C::E : 1];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    qv[m] = make_float2(ld(I.rho0, i0, I.rho0_s), ld(I.rho0, i0 + N, I.rho0_s));
    if constexpr (R0R) r0v[m] = qv[m];
    divu[m] = make_float2(0.f, 0.f);
    rt[m] = make_float2(0.f, 0.f);
  }
  if (flags & FLAG_NONLINEAR) {
    const auto rhot = gp(fl.rhoi + off);
    float2 ro[C::E];
#pragma unroll
    for (int m = 0; m < C::E; ++m) ro[m] = make_float2(rhot[iA + m * C::TPL], rhot[iA + N + m * C::TPL]);
#pragma unroll
    for (int m = 0; m < C::E; ++m) qv[m] = make_float2(fmaf(2.f, ro[m].x, qv[m].x), fmaf(2.f, ro[m].y, qv[m].y));
  }
#pragma unroll
  for (int m = 0; m < C::E; ++m) qv[m] = cscale(qv[m], I.dt);
  float2 As[C::IT], Bs[C::IT];
  pair_load<C>(As, Bs, fl.spec[0] + b * g.nspec, row0, rows, g.nhp, tid);
  if (t >= I.nt) return;
  KW_ZPASS_PUT
  __syncthreads();
  if constexpr (SREG) {
    if (filtered) filtered_source<C>(src, smode, t, iA, lds, fl, g, b, tw, row0, rows, tid, ch);
  }
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const auto rho = gw(fl.rho[i] + off);
    // old split density, fetched before the transform so its latency overlaps it
    // (for short register arrays; the long mixed-radix ones load it in place)
    constexpr bool PF = C::E <= 16;
    float2 ro[C::E];
    if constexpr (PF) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) ro[m] = make_float2(rho[iA + m * C::TPL], rho[iA + N + m * C::TPL]);
    }
    float2 d[C::E];
    if (i > 0) pair_load<C>(As, Bs, fl.spec[i] + b * g.nspec, row0, rows, g.nhp, tid);
    __syncthreads();
    pair_put<C>(lds, As, Bs, tid);
    inv_from_lds<C>(lds, tw, tid, d);
    if constexpr (!PF) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) ro[m] = make_float2(rho[iA + m * C::TPL], rho[iA + N + m * C::TPL]);
    }
    if constexpr (CAP) {
      if (inside) {
        const auto dd = gw(fl.adjD + (int64_t)i * gridDim.y * g.ntot + off);
#pragma unroll
        for (int m = 0; m < C::E; ++m) {
          dd[iA + m * C::TPL] = d[m].x;
          dd[iA + N + m * C::TPL] = d[m].y;
        }
      }
    }
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const float sz = (i == ND - 1) ? pmlz[j0 + m * C::TPL] : 1.f;
      ro[m] = make_float2(pml_update(sz * ph[i][0], ro[m].x, qv[m].x, d[m].x), pml_update(sz * ph[i][1], ro[m].y, qv[m].y, d[m].y));
    }
    if constexpr (SREG) {
      if (filtered) {
        const float fac = src.fac[i];
#pragma unroll
        for (int m = 0; m < C::E; ++m) ro[m] = make_float2(fmaf(fac, ch[m].x, ro[m].x), fmaf(fac, ch[m].y, ro[m].y));
      }
    }
    if (inside) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        rho[iA + m * C::TPL] = ro[m].x;
        rho[iA + N + m * C::TPL] = ro[m].y;
      }
    }
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      rounded(ro[m].x);
      rounded(ro[m].y);
      divu[m] = cadd(divu[m], d[m]);
      rt[m] = cadd(rt[m], ro[m]);
    }
  }
  if (src_is_point(smode) && inside) {
    // point sources: update the owned source points of every split density and
    // rebuild their density sums (same order of additions as the loop above)
    for (int h = 0; h < 2; ++h) {
      const int r = ra + h;
      if (gp(src.row_ptr)[r] == gp(src.row_ptr)[r + 1]) continue;
      for (int m = 0; m < C::E; ++m) {
        const int n = j0 + m * C::TPL;
        float v;
        if (!csr_lookup(src, r, n, t, v)) continue;
        const int64_t idx = off + (int64_t)r * N + n;
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < ND; ++i) {
          const auto rho = gw(fl.rho[i]);
          const float x = src_point(smode, rho[idx], src.fac[i], v);
          rho[idx] = x;
          sum += x;
        }
        set_lane(rt, m, h, sum);
      }
    }
  }
  if (fl.rhot && inside) {
    const auto rhot = gw(fl.rhot + off);
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      rhot[iA + m * C::TPL] = rt[m].x;
      rhot[iA + N + m * C::TPL] = rt[m].y;
    }
  }
  float2 r0e[C::E];  // rho0 again: the lines this block read at its start, from L2 if still there
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    if constexpr (R0R) r0e[m] = r0v[m];
    else r0e[m] = make_float2(ld(I.rho0, iA + m * C::TPL, I.rho0_s), ld(I.rho0, iA + N + m * C::TPL, I.rho0_s));
  }
  if (powerlaw) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) divu[m] = make_float2(r0e[m].x * divu[m].x, r0e[m].y * divu[m].y);
  } else {
    float2 c2v[C::E], q[C::E];
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const int64_t i0 = iA + m * C::TPL;
      c2v[m] = make_float2(ld(I.c0sq, i0, I.c0sq_s), ld(I.c0sq, i0 + N, I.c0sq_s));
      q[m] = rt[m];
    }
    if (flags & FLAG_STOKES) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        const int64_t i0 = iA + m * C::TPL;
        q[m].x = fmaf(tau_at(I, i0, c2v[m].x) * r0e[m].x, divu[m].x, q[m].x);
        q[m].y = fmaf(tau_at(I, i0 + N, c2v[m].y) * r0e[m].y, divu[m].y, q[m].y);
      }
      if (fl.adjA && inside) {  // adjoint replay: the Stokes operand
#pragma unroll
        for (int m = 0; m < C::E; ++m) {
          gw(fl.adjA)[off + iA + m * C::TPL] = r0e[m].x * divu[m].x;
          gw(fl.adjA)[off + iA + N + m * C::TPL] = r0e[m].y * divu[m].y;
        }
      }
    }
    if (flags & FLAG_NONLINEAR) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        const int64_t i0 = iA + m * C::TPL;
        q[m].x += ld(I.bona, i0, I.bona_s) * rt[m].x * rt[m].x / (2.f * r0e[m].x);
        q[m].y += ld(I.bona, i0 + N, I.bona_s) * rt[m].y * rt[m].y / (2.f * r0e[m].y);
      }
    }
#pragma unroll
    for (int m = 0; m < C::E; ++m) divu[m] = make_float2(c2v[m].x * q[m].x, c2v[m].y * q[m].y);
    if (inside) {
      const auto p = gw(fl.p + off);
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        p[iA + m * C::TPL] = divu[m].x;
        p[iA + N + m * C::TPL] = divu[m].y;
      }
    }
  }
  if (!powerlaw) {
    fwd_from_regs<C>(lds, divu, fl.spec[0] + b * g.nspec, tw, row0, rows, g.nhp, tid);
  } else {
    if (flags & FLAG_POWERLAW_ABS) fwd_from_regs<C>(lds, divu, fl.spec[0] + b * g.nspec, tw, row0, rows, g.nhp, tid);
    if (flags & FLAG_POWERLAW_DISP) fwd_from_regs<C>(lds, rt, fl.spec[1] + b * g.nspec, tw, row0, rows, g.nhp, tid);
  }
}

// ---------------------------------------------------------------------------
// equation of state with power-law absorption / dispersion
// p = c0^2 (rho + tau F^-1[|k|^{y-2} F[rho0 div u]] - eta F^-1[|k|^{y-1} F[rho]] + B/A rho^2 / (2 rho0))
// ---------------------------------------------------------------------------
template <int N>
__global__ __launch_bounds__(ZCfg<N>::NT) KW_WPE(N, KW_WPE_EOS) void k_eos(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ tw_g, int flags) {
  KW_ZPASS_EARLY((const float*)nullptr)
  const int t = step_of(fl, b);
  KW_ROWS_CLAMPED
  const int64_t off = b * g.ntot;
  const auto rhot = gw(fl.rhot + off);
  float2 rtv[C::E], c2v[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    rtv[m] = make_float2(rhot[i0], rhot[i0 + N]);
    c2v[m] = make_float2(ld(I.c0sq, i0, I.c0sq_s), ld(I.c0sq, i0 + N, I.c0sq_s));
  }
  if (t >= I.nt) return;
  KW_ZPASS_PUT
  __syncthreads();
  float2 av[C::E], bv[C::E];
  if (flags & FLAG_POWERLAW_ABS) inv_to_regs<C>(lds, fl.spec[0] + b * g.nspec, tw, row0, rows, g.nhp, tid, av);
  if (flags & FLAG_POWERLAW_DISP) inv_to_regs<C>(lds, fl.spec[1] + b * g.nspec, tw, row0, rows, g.nhp, tid, bv);
  if (inside && fl.adjA && (flags & FLAG_POWERLAW_ABS)) {  // adjoint replay: keep the operands
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      gw(fl.adjA)[off + iA + m * C::TPL] = av[m].x;
      gw(fl.adjA)[off + iA + N + m * C::TPL] = av[m].y;
    }
  }
  if (inside && fl.adjB && (flags & FLAG_POWERLAW_DISP)) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      gw(fl.adjB)[off + iA + m * C::TPL] = bv[m].x;
      gw(fl.adjB)[off + iA + N + m * C::TPL] = bv[m].y;
    }
  }
  float2 q[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) q[m] = rtv[m];
  if (flags & FLAG_POWERLAW_ABS) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const int64_t i0 = iA + m * C::TPL;
      q[m] = make_float2(fmaf(tau_at(I, i0, c2v[m].x), av[m].x, q[m].x), fmaf(tau_at(I, i0 + N, c2v[m].y), av[m].y, q[m].y));
    }
  }
  if (flags & FLAG_POWERLAW_DISP) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const int64_t i0 = iA + m * C::TPL;
      q[m] = make_float2(fmaf(-eta_at(I, i0, c2v[m].x), bv[m].x, q[m].x), fmaf(-eta_at(I, i0 + N, c2v[m].y), bv[m].y, q[m].y));
    }
  }
  if (flags & FLAG_NONLINEAR) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const int64_t i0 = iA + m * C::TPL;
      q[m].x += ld(I.bona, i0, I.bona_s) * rtv[m].x * rtv[m].x / (2.f * ld(I.rho0, i0, I.rho0_s));
      q[m].y += ld(I.bona, i0 + N, I.bona_s) * rtv[m].y * rtv[m].y / (2.f * ld(I.rho0, i0 + N, I.rho0_s));
    }
  }
#pragma unroll
  for (int m = 0; m < C::E; ++m) av[m] = make_float2(c2v[m].x * q[m].x, c2v[m].y * q[m].y);
  if (inside) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      gw(fl.p)[off + iA + m * C::TPL] = av[m].x;
      gw(fl.p)[off + iA + N + m * C::TPL] = av[m].y;
    }
  }
  fwd_from_regs<C>(lds, av, fl.spec[0] + b * g.nspec, tw, row0, rows, g.nhp, tid);
}

// ---------------------------------------------------------------------------
// t = 0 initial-value override: u_i = dt/(2 rho0_sg_i) grad_i p0, rho_j = p0 / (c0^2 D)
// ---------------------------------------------------------------------------
template <int N>
__global__ __launch_bounds__(ZCfg<N>::NT) void k_init_u(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ tw_g) {
  KW_ZPASS_PROLOGUE
  const int ax = blockIdx.z;
  const Inst& I = inst[b];
  const int64_t off = b * g.ntot;
  float2 gv[C::E];
  inv_to_regs<C>(lds, fl.spec[ax] + b * g.nspec, tw, row0, rows, g.nhp, tid, gv);
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int n = j0 + m * C::TPL;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = ra + h;
      if (r >= rows) continue;
      const int64_t idx = (int64_t)r * N + n;
      gw(fl.u[ax])[off + idx] = 0.5f * ld(I.dtr0[ax], idx, I.dtr0_s) * (h ? gv[m].y : gv[m].x);
      if (ax == 0) {
        const float pv = gw(fl.p)[off + idx], c2 = ld(I.c0sq, idx, I.c0sq_s);
        float rs = 0.f;
        for (int j = 0; j < g.nd; ++j) {
          const float rv = pv / (c2 * I.p0div[j]);
          gw(fl.rho[j])[off + idx] = rv;
          rs += rv;
        }
        if (fl.rhot) gw(fl.rhot)[off + idx] = rs;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// build the z-spectrum of a multi-row additive source at step t (mode CHAIN)
// which = -1: pressure source, 0..2: velocity component
// ---------------------------------------------------------------------------
template <int N, bool NAR>
__global__ __launch_bounds__((ZCfg<N, NAR>::NT)) void k_src_build(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ tw_g, int which) {
  KW_ZPASS_PROLOGUE_AS(ZCfg<N, NAR>)
  const Inst& I = inst[b];
  const int t = step_of(fl, b);
  const Src& s = which < 0 ? I.srcp : I.srcu[which];
  if (t >= I.nt || s.mode != SRC_CHAIN || t >= s.len) return;
  const auto sp = gw(fl.spec[s.chain_buf] + b * g.nspec);
  const int rend = min(row0 + 2 * C::L, rows);
  const int e0 = gp(s.row_ptr)[row0], e1 = gp(s.row_ptr)[rend];
  if (e0 == e1) {
    for (int e = tid; e < C::L * C::NH; e += C::NT) {
      const int p = e / C::NH, k = e % C::NH;
      const int r0 = row0 + 2 * p;
      if (r0 < rows) st2(sp, (int64_t)r0 * g.nhp + k, make_float2(0.f, 0.f));
      if (r0 + 1 < rows) st2(sp, (int64_t)(r0 + 1) * g.nhp + k, make_float2(0.f, 0.f));
    }
    return;
  }
  const typename C::Idx idx{};
  for (int e = tid; e < N * C::L; e += C::NT) lds[idx(e % N, e / N)] = make_float2(0.f, 0.f);
  __syncthreads();
  float* fb = reinterpret_cast<float*>(lds);
  for (int e = e0 + tid; e < e1; e += C::NT) {
    int r = row0;
    while (gp(s.row_ptr)[r + 1] <= e) ++r;
    const int p = (r - row0) >> 1, h = (r - row0) & 1;
    fb[2 * idx(gp(s.col)[e], p) + h] = gp(s.scale)[e] * gp(s.sig)[(int64_t)gp(s.sigrow)[e] * s.len + t];
  }
  __syncthreads();
  float2 v[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) v[m] = lds[idx(j0 + m * C::TPL, pc)];
  __syncthreads();
  fwd_from_regs<C>(lds, v, fl.spec[s.chain_buf] + b * g.nspec, tw, row0, rows, g.nhp, tid);
}

// ---------------------------------------------------------------------------
// strided column passes
// ---------------------------------------------------------------------------
// sin(x)/x and cos(x) by their Taylor series through x^14 (truncation error
// below 2e-10 for |x| <= 2, which covers c_ref dt |k| / 2 at any stable CFL);
// larger arguments fall back to the library functions.
// The k-space operators of the outermost-axis pass take |k|^2 = kx^2 + ky^2 + kz^2
// (no square root on the common path).  kappa = sinc(x) and cos(x) for
// x = c_ref dt |k| / 2 from x^2: Taylor polynomials in x^2 up to x^2 = 4 (FP32
// rounding), sin(x)/x and cos(x) beyond.
// BIG = false: the caller has tested x^2 <= 4, for a whole line at once.
template <bool BIG = true>
__device__ __forceinline__ float sinc_k2(float x2) {
  if (BIG && x2 > 4.f) {
    const float x = sqrtf(x2);
    return sinf(x) / x;
  }
  float p = -1.f / 1307674368000.f;                 // -1/15!
  p = fmaf(p, x2, 1.f / 6227020800.f);              //  1/13!
  p = fmaf(p, x2, -1.f / 39916800.f);               // -1/11!
  p = fmaf(p, x2, 1.f / 362880.f);                  //  1/9!
  p = fmaf(p, x2, -1.f / 5040.f);                   // -1/7!
  p = fmaf(p, x2, 1.f / 120.f);                     //  1/5!
  p = fmaf(p, x2, -1.f / 6.f);                      // -1/3!
  return fmaf(p, x2, 1.f);
}
template <bool BIG = true>
__device__ __forceinline__ float cos_k2(float x2) {
  if (BIG && x2 > 4.f) return cosf(sqrtf(x2));
  float p = -1.f / 87178291200.f;                   // -1/14!
  p = fmaf(p, x2, 1.f / 479001600.f);               //  1/12!
  p = fmaf(p, x2, -1.f / 3628800.f);                // -1/10!
  p = fmaf(p, x2, 1.f / 40320.f);                   //  1/8!
  p = fmaf(p, x2, -1.f / 720.f);                    // -1/6!
  p = fmaf(p, x2, 1.f / 24.f);                      //  1/4!
  p = fmaf(p, x2, -0.5f);                           // -1/2!
  return fmaf(p, x2, 1.f);
}
// |k|^a from |k|^2 for |k| > 0 (the fractional Laplacian is 0 at |k| = 0)
__device__ __forceinline__ float kpow2(float km2, float a) { return km2 == 0.f ? 0.f : exp2f(0.5f * a * log2f(km2)); }

// Spectral factor of a job at the lane's E elements: kappa(|k|) = sinc (GRAD, DIV; also
// the common factor of an input whose jobs are all of these), cos (SRCKAPPA), the
// fractional powers, 1 otherwise.  The kind and the range of the arguments are tested
// around the loops, not per element: on any stable time step every argument is within
// the polynomials' range (kx2max: the largest kx^2 of the axis), and the loops are
// straight-line code.
template <int E>
__device__ __forceinline__ void job_factor(int kind, float kap, const float (&km2)[E], float kmax2, const Ops& ops, float (&f)[E]) {
  if (kind == XK_FRAC1 || kind == XK_FRAC2) {
    const float a = kind == XK_FRAC1 ? ops.frac1 : ops.frac2;
#pragma unroll
    for (int m = 0; m < E; ++m) f[m] = kpow2(km2[m], a);
  } else if (kap > 0.f && (kind == XK_GRAD || kind == XK_DIV || kind == XK_SRCKAPPA)) {
    const float k2 = kap * kap;
    if (__any(k2 * kmax2 > 4.f)) {
#pragma unroll
      for (int m = 0; m < E; ++m) f[m] = kind == XK_SRCKAPPA ? cos_k2(k2 * km2[m]) : sinc_k2(k2 * km2[m]);
    } else if (kind == XK_SRCKAPPA) {
#pragma unroll
      for (int m = 0; m < E; ++m) f[m] = cos_k2<false>(k2 * km2[m]);
    } else {
#pragma unroll
      for (int m = 0; m < E; ++m) f[m] = sinc_k2<false>(k2 * km2[m]);
    }
  } else {
#pragma unroll
    for (int m = 0; m < E; ++m) f[m] = 1.f;
  }
}

// v = st times a job's operator and 1/ntot: the tabled vector (in v) times its factor, or
// the factor alone.
template <int E>
__device__ __forceinline__ void apply_job(bool tabled, const float2 (&st)[E], const float (&f)[E], float inv, float2 (&v)[E]) {
  if (tabled) {
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = cscale(cmul(st[m], cscale(v[m], f[m])), inv);
  } else {
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = cscale(cscale(st[m], f[m]), inv);
  }
}

// Consecutive workgroup ids go to different XCDs (round robin over 8); give each
// XCD a contiguous range of tiles so neighbouring tiles share its L2.
__device__ __forceinline__ int xcd_remap(int bid, int nblk) {
  const int nfull = nblk & ~7;
  if (bid >= nfull) return bid;
  return (bid & 7) * (nfull >> 3) + (bid >> 3);
}

template <int N, int L, int EM = 1, int PV = 0>
struct ColCfg {
  using F = FftShape<N, EM, PV>;
  static constexpr int E = F::E;
  static constexpr int TPL = F::TPL;
  static constexpr int NT = TPL * L;
  using Idx = ColIdx<L>;
  static constexpr int LDS = Idx::size(N);
};

template <int N>
constexpr int col_lbig() { return clampi(pow2floor(8192 / N), 1, 64); }
template <int N>
constexpr int col_lsmall() { return col_lbig<N>() / 4 < 1 ? 1 : col_lbig<N>() / 4; }
// Tiles of the outermost-axis pass with spectral jobs: half as wide, since that
// kernel holds more registers (at 512: 942 vs 1015 us for the gradient pass,
// 1197 vs 1335 us for the divergence pass).
template <int N>
constexpr int col_lops() { return col_lbig<N>() / 2 < 1 ? 1 : col_lbig<N>() / 2; }

template <int N, int L, bool OPS, int EM = 1, int PV = 0>
__global__ __launch_bounds__((ColCfg<N, L, EM, PV>::NT)) KW_WPE(N, (OPS ? KW_WPE_COLOPS : KW_WPE_COL)) void k_col(Geom g, Fields fl, Ops ops, const Inst* __restrict__ inst, ColArgs a) {
  if (a.gath && (int)blockIdx.x >= a.gx) return gather_blocks(g, fl, inst, a);
  using C = ColCfg<N, L, EM, PV>;
  __shared__ float2 lds[C::LDS];
  __shared__ float2 twl[stage_tw_size<N, PV>()];
  const typename C::Idx idx{};
  const int tid = threadIdx.x;
  const int b = blockIdx.y;
  if (fl.tdev && step_of(fl, b) >= inst[b].nt) return;
  {
    float2 twr[stage_tw_loads<N, PV>(C::NT)];
    load_stage_tw<N, PV, C::NT>(twr, ops.tw[a.axis], tid);
    put_stage_tw<N, PV, C::NT>(twr, twl, tid);
  }
  __syncthreads();
  const int ntile = (a.ncols + L - 1) / L;
  const int lid = xcd_remap(blockIdx.x, a.gx);
  const int c = tid % L, j0 = tid / L;
  const float2* tw = twl;
  const int ntiles = a.nouter * ntile;
  // Tile lt: its lane's column, clamped into the spectrum (a lane beyond it transforms a
  // copy of the last column and does not store it: tests around single loads would have
  // the compiler wait for each alone).
  auto tile_base = [&](int lt, bool& in) -> int64_t {
    const int o = lt / ntile, col = (lt - o * ntile) * L + c;
    in = col < a.ncols;
    return (int64_t)b * g.nspec + (int64_t)o * a.ostride + min(col, a.ncols - 1) + (int64_t)j0 * a.estride;
  };
  const int64_t step = (int64_t)C::TPL * a.estride;

  float2 v[C::E];
  if constexpr (!OPS) {
    // software pipeline over the buffers and tiles: the loads of the next buffer
    // (after a tile's last buffer, the first buffer of this workgroup's next tile)
    // are in flight while the current one is transformed and stored
    float2 nx[C::E];
    bool vt = false;
    int64_t bt = tile_base(min(lid, ntiles - 1), vt);
    {
      const auto bp = gp(fl.spec[a.bufs[0]]);
#pragma unroll
      for (int m = 0; m < C::E; ++m) nx[m] = ld2(bp, bt + m * step);
    }
    for (int lt = lid; lt < ntiles; lt += a.gx) {
      const int ltn = lt + a.gx;
      bool vn = false;
      const int64_t bn = tile_base(min(ltn, ntiles - 1), vn);
      for (int q = 0; q < a.nbuf; ++q) {
        const auto bp = gw(fl.spec[a.bufs[q]]);
#pragma unroll
        for (int m = 0; m < C::E; ++m) v[m] = nx[m];
        if (q + 1 < a.nbuf || ltn < ntiles) {
          const bool last = q + 1 == a.nbuf;
          const auto bq = gp(fl.spec[a.bufs[last ? 0 : q + 1]]);
          const int64_t bx = last ? bn : bt;
#pragma unroll
          for (int m = 0; m < C::E; ++m) nx[m] = ld2(bq, bx + m * step);
        }
        if (a.mode == 0) fft_reg<N, -1, typename C::Idx, EM, PV>(v, lds, tw, c, j0, idx);
        else fft_reg<N, +1, typename C::Idx, EM, PV>(v, lds, tw, c, j0, idx);
        if (vt) {
#pragma unroll
          for (int m = 0; m < C::E; ++m) st2(bp, bt + m * step, v[m]);
        }
      }
      bt = bn;
      vt = vn;
    }
  } else {
  // forward, multiply, inverse (outermost axis = axis 0), over the tiles lid,
  // lid + G, ... of this instance (G = workgroups per instance: one tile each when
  // the grid covers every tile, else a resident grid that loops; with the
  // XCD-aware lid, the tiles an XCD runs at one time are neighbours).
  const float kap = inst[b].kap;
  // Operator values read between the transforms come from LDS, so no global
  // latency sits between a forward and an inverse transform: the x wavenumbers,
  // the x-axis operator vectors of up to two tabled jobs (loaded once), and per
  // column of the tile the value of every y/z-axis job.  (The twiddle barrier
  // above has passed; the first transform's barriers publish these before they
  // are read, and the previous tile's last reads of cop sit before its last
  // transform's barriers.)
  __shared__ float kxs[N];
  __shared__ float2 xop[2][N];
  __shared__ float2 cop[kMaxJobs][L];
  for (int i_ = tid; i_ < N; i_ += C::NT) kxs[i_] = gp(ops.k[0])[i_];
  for (int j = 0, slot = 0; j < a.njob; ++j) {
    const XJob jb = a.job[j];
    const float2* t = jb.kind == XK_GRAD ? ops.grad[jb.axis] : jb.kind == XK_DIV ? ops.div[jb.axis]
                    : jb.kind == XK_UNSTAGGER ? ops.unst[jb.axis] : nullptr;
    if (!t || jb.axis != 0) continue;
    if (slot < 2)
      for (int i_ = tid; i_ < N; i_ += C::NT) xop[slot][i_] = ld2(gp(t), i_);
    ++slot;
  }
  const float kxe = gp(ops.k[0])[N / 2];  // the axis's largest wavenumber
  // The next distinct input is loaded while the current one is transformed and
  // its jobs stored: issued after those stores, its loads would also wait for
  // them (the vector-memory counter drains in order).  Within a tile, not when
  // one of the jobs before it writes that buffer; after a tile's last input, the
  // next tile's first input (other columns, so never written by this tile).
  // Only for short register arrays (the mixed-radix ones would lose occupancy).
  constexpr bool PRE = C::E <= 8;
  float2 nx[PRE ? C::E : 1];
  bool next_loaded = false;  // nx holds this tile's first input
  for (int lt = lid; lt < ntiles; lt += a.gx) {
    const int o = lt / ntile, tile = lt % ntile;
    const int col = tile * L + c;
    bool valid = false;
    const int64_t base = tile_base(lt, valid);
    int iy, iz;
    if (g.nd == 2) { iy = valid ? col : 0; iz = 0; }
    else { iy = o; iz = valid ? col : 0; }
    for (int j = 0; j < a.njob; ++j) {
      const XJob jb = a.job[j];
      const float2* t = jb.kind == XK_GRAD ? ops.grad[jb.axis] : jb.kind == XK_DIV ? ops.div[jb.axis]
                      : jb.kind == XK_UNSTAGGER ? ops.unst[jb.axis] : nullptr;
      if (!t || jb.axis == 0) continue;
      for (int cc = tid; cc < L; cc += C::NT) {
        const int colc = min(tile * L + cc, a.ncols - 1);
        const int ia = (jb.axis == 1 && g.nd == 3) ? o : colc;
        cop[j][cc] = ld2(gp(t), ia);
      }
    }
    float kyz2 = 0.f;
    {
      const float ky = gp(ops.k[1])[iy];
      kyz2 = ky * ky;
      if (g.nd == 3) { const float kz = gp(ops.k[2])[iz]; kyz2 = fmaf(kz, kz, kyz2); }
    }
    const float kmax2 = fmaf(kxe, kxe, kyz2);
    float2 st[C::E];
    int cur_in = -1, pre_in = next_loaded ? a.job[0].in : -1;
    bool kgroup = false;  // the current input's spectrum carries kappa / ntot
    next_loaded = false;
    int slot = 0;  // x-table slot of the next x-axis job
    for (int j = 0; j < a.njob; ++j) {
      const XJob jb = a.job[j];
      if (jb.in != cur_in) {
        cur_in = jb.in;
        if (PRE && pre_in == cur_in) {
#pragma unroll
          for (int m = 0; m < C::E; ++m) st[m] = nx[PRE ? m : 0];
        } else {
          const auto src = gp(fl.spec[jb.in]);
#pragma unroll
          for (int m = 0; m < C::E; ++m) st[m] = ld2(src, base + m * step);
          // wait here, not at the transform: there the compiler could not tell these loads
          // from the ones issued ahead below and would wait for both
#pragma unroll
          for (int m = 0; m < C::E; ++m) asm volatile("" : "+v"(st[m].x), "+v"(st[m].y));
        }
        pre_in = -1;
        int k = j + 1;
        while (k < a.njob && a.job[k].in == cur_in) ++k;
        if constexpr (PRE) {
          int from = -1;  // what to load ahead
          int64_t nbase = base;
          if (k < a.njob) {
            bool clobbered = false;
            for (int i = j; i < k; ++i) clobbered |= a.job[i].out == a.job[k].in;
            if (!clobbered) from = pre_in = a.job[k].in;
          } else if (lt + a.gx < ntiles) {
            bool vn;
            nbase = tile_base(lt + a.gx, vn);
            from = a.job[0].in;
            next_loaded = true;
          }
          if (from >= 0) {
            const auto nsrc = gp(fl.spec[from]);
#pragma unroll
            for (int m = 0; m < C::E; ++m) nx[m] = ld2(nsrc, nbase + m * step);
          }
        }
        fft_reg<N, -1, typename C::Idx, EM, PV>(st, lds, tw, c, j0, idx);
        // When every job on this input is a gradient or divergence, the common
        // factor kappa(|k|) / ntot is applied to the spectrum once (the x
        // wavenumbers in LDS are published by the transform's barriers).
        kgroup = true;
        for (int i = j; i < k; ++i) kgroup &= a.job[i].kind == XK_GRAD || a.job[i].kind == XK_DIV;
        if (kgroup) {
          float km2[C::E], f[C::E];
#pragma unroll
          for (int m = 0; m < C::E; ++m) { const float kx = kxs[j0 + m * C::TPL]; km2[m] = fmaf(kx, kx, kyz2); }
          job_factor(XK_GRAD, kap, km2, kmax2, ops, f);
#pragma unroll
          for (int m = 0; m < C::E; ++m) st[m] = cscale(st[m], f[m] * ops.inv_ntot);
        }
      }
      // where this job's operator values live: the per-column values, an x-table
      // slot, or (a third x-axis table) global memory
      const bool tabled = jb.kind == XK_GRAD || jb.kind == XK_DIV || jb.kind == XK_UNSTAGGER;
      if (tabled && jb.axis != 0) {
        const float2 colv = cop[j][c];
#pragma unroll
        for (int m = 0; m < C::E; ++m) v[m] = colv;
      } else if (tabled) {
        if (slot < 2) {
#pragma unroll
          for (int m = 0; m < C::E; ++m) v[m] = xop[slot][j0 + m * C::TPL];
        } else {
          const auto gtab = gp(jb.kind == XK_GRAD ? ops.grad[0] : jb.kind == XK_DIV ? ops.div[0] : ops.unst[0]);
#pragma unroll
          for (int m = 0; m < C::E; ++m) v[m] = ld2(gtab, j0 + m * C::TPL);
        }
        ++slot;
      }
      if (kgroup) {
#pragma unroll
        for (int m = 0; m < C::E; ++m) v[m] = cmul(st[m], v[m]);
      } else {
        float km2[C::E], f[C::E];
#pragma unroll
        for (int m = 0; m < C::E; ++m) { const float kx = kxs[j0 + m * C::TPL]; km2[m] = fmaf(kx, kx, kyz2); }
        job_factor(jb.kind, kap, km2, kmax2, ops, f);
        apply_job<C::E>(tabled, st, f, ops.inv_ntot, v);
      }
      fft_reg<N, +1, typename C::Idx, EM, PV>(v, lds, tw, c, j0, idx);
      if (valid) {
        const auto dst = gw(fl.spec[jb.out]);
#pragma unroll
        for (int m = 0; m < C::E; ++m) st2(dst, base + m * step, v[m]);
      }
    }
  }
  }
}

// ---------------------------------------------------------------------------
// column passes of small grids
// ---------------------------------------------------------------------------
// Where the tiles of k_col leave most of the chip idle, a pass is one chain of
// latencies: load, transforms one job after the other, store.  This form shortens the
// chain and gives the same bits: tiles of at most one or two wavefronts (col_lsmall2),
// one group of lanes per job (each loads and transforms its job's input itself, so a
// pass costs one forward and one inverse transform whatever its jobs; stores wait
// until every group has read, since jobs may write each other's input) or per buffer
// (blockIdx.z), and every load of the pass, operator values included, issued at once.
constexpr int kColSmallJobs = 4;  // jobs of a small-grid pass (one group of lanes each)
template <int N>
constexpr int col_lsmall2() { return clampi(64 / FftShape<N>::TPL, KW_COL_SMALL_MIN, 32); }

template <int N, int L, bool OPS>
__global__ __launch_bounds__((ColCfg<N, L>::NT * (OPS ? kColSmallJobs : 1))) void k_col_small(Geom g, Fields fl, Ops ops, const Inst* __restrict__ inst, ColArgs a) {
  if (a.gath && (int)blockIdx.x >= a.gx) return gather_blocks(g, fl, inst, a);
  using C = ColCfg<N, L>;
  constexpr bool WS = C::NT == 64;
  extern __shared__ float2 lds_all[];
  __shared__ float2 twl[stage_tw_size<N>()];
  const typename C::Idx idx{};
  const int grp = OPS ? (int)threadIdx.x / C::NT : 0;
  const int tid = threadIdx.x - grp * C::NT;
  const int b = blockIdx.y;
  float2* const lds = lds_all + grp * C::LDS;
  const int ntile = (a.ncols + L - 1) / L;
  const int lid = xcd_remap(blockIdx.x, a.gx);
  const int o = lid / ntile, tile = lid % ntile;
  const int c = tid % L, j0 = tid / L;
  const int col = tile * L + c;
  const bool valid = col < a.ncols;
  const int64_t base = (int64_t)b * g.nspec + (int64_t)o * a.ostride + min(col, a.ncols - 1);
  const XJob jb = OPS ? a.job[grp] : XJob{};
  const int ibuf = OPS ? jb.in : a.bufs[blockIdx.z];
  float2 v[C::E];
  {
    const auto src = gp(fl.spec[ibuf]);
#pragma unroll
    for (int m = 0; m < C::E; ++m) v[m] = ld2(src, base + (int64_t)(j0 + m * C::TPL) * a.estride);
  }
  constexpr int TW = stage_tw_loads<N, 0>(C::NT);
  float2 twr[TW];
  load_stage_tw<N, 0, C::NT>(twr, ops.tw[a.axis], tid);
  // operator values of this lane's lines: the x wavenumbers, |k|^2 of the other axes, the job's
  // x-axis vector or its per-column value
  float kx[OPS ? C::E : 1], kyz2 = 0.f, kap = 0.f, kxe = 0.f;
  float2 opx[OPS ? C::E : 1], colv = make_float2(1.f, 0.f);
  const float2* tab = nullptr;
  if constexpr (OPS) {
    const int colc = min(col, a.ncols - 1);
    tab = jb.kind == XK_GRAD ? ops.grad[jb.axis] : jb.kind == XK_DIV ? ops.div[jb.axis] : jb.kind == XK_UNSTAGGER ? ops.unst[jb.axis] : nullptr;
    kap = inst[b].kap;
    kxe = gp(ops.k[0])[N / 2];
#pragma unroll
    for (int m = 0; m < C::E; ++m) kx[m] = gp(ops.k[0])[j0 + m * C::TPL];
    if (tab && jb.axis == 0) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) opx[m] = ld2(gp(tab), j0 + m * C::TPL);
    } else if (tab) {
      colv = ld2(gp(tab), (jb.axis == 1 && g.nd == 3) ? o : colc);
    }
    const float ky = gp(ops.k[1])[g.nd == 2 ? (valid ? col : 0) : o];
    kyz2 = ky * ky;
    if (g.nd == 3) { const float kz = gp(ops.k[2])[valid ? col : 0]; kyz2 = fmaf(kz, kz, kyz2); }
  }
  if (fl.tdev && step_of(fl, b) >= inst[b].nt) return;
  if (grp == 0) put_stage_tw<N, 0, C::NT>(twr, twl, tid);
  __syncthreads();
  if constexpr (!OPS) {
    if (a.mode == 0) fft_reg<N, -1, typename C::Idx, 1, 0, WS>(v, lds, twl, c, j0, idx);
    else fft_reg<N, +1, typename C::Idx, 1, 0, WS>(v, lds, twl, c, j0, idx);
  } else {
    fft_reg<N, -1, typename C::Idx, 1, 0, WS>(v, lds, twl, c, j0, idx);
    // the jobs next to this one on the same input (k_col: one common factor when all of
    // them are gradients or divergences)
    bool kgroup = true;
    for (int i = grp; i >= 0 && a.job[i].in == jb.in; --i) kgroup &= a.job[i].kind == XK_GRAD || a.job[i].kind == XK_DIV;
    for (int i = grp; i < a.njob && a.job[i].in == jb.in; ++i) kgroup &= a.job[i].kind == XK_GRAD || a.job[i].kind == XK_DIV;
    float km2[C::E], f[C::E];
#pragma unroll
    for (int m = 0; m < C::E; ++m) km2[m] = fmaf(kx[m], kx[m], kyz2);
    job_factor(jb.kind, kap, km2, fmaf(kxe, kxe, kyz2), ops, f);
    if (!(tab && jb.axis == 0)) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) opx[m] = colv;
    }
    if (kgroup) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) v[m] = cmul(cscale(v[m], f[m] * ops.inv_ntot), opx[m]);
    } else {
      float2 st[C::E];
#pragma unroll
      for (int m = 0; m < C::E; ++m) { st[m] = v[m]; v[m] = opx[m]; }
      apply_job<C::E>(tab != nullptr, st, f, ops.inv_ntot, v);
    }
    __syncthreads();  // every group has read its input
    fft_reg<N, +1, typename C::Idx, 1, 0, WS>(v, lds, twl, c, j0, idx);
  }
  if (valid) {
    const auto dst = gw(fl.spec[OPS ? jb.out : ibuf]);
#pragma unroll
    for (int m = 0; m < C::E; ++m) st2(dst, base + (int64_t)(j0 + m * C::TPL) * a.estride, v[m]);
  }
}

// ---------------------------------------------------------------------------
// contiguous-axis updates of small grids
// ---------------------------------------------------------------------------
// The updates above walk their axes one after the other on workgroups sized for
// bandwidth; on a small grid that is a long chain of latencies on few compute units.
// These forms give the same bits from one wavefront per row group and axis: the
// transforms of the axes run side by side, their results meet once in LDS, every load
// of the kernel is issued at its start, and a wavefront's exchanges need no workgroup
// barrier (lines of 1024 take two wavefronts and keep the barriers).
#define KW_ZSMALL_PROLOGUE(GROUPS)                                                                    \
  using C = ZCfg<N, true>;                                                                            \
  constexpr int G = GROUPS;                                                                           \
  static_assert(C::NT % 64 == 0, "a group is whole wavefronts");                                      \
  __shared__ float2 lds_all[G][C::LDS];                                                               \
  __shared__ float2 twl[stage_tw_size<N, C::PV>()];                                                   \
  const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x / C::NT);                           \
  const int tid = (int)threadIdx.x - grp * C::NT;                                                     \
  float2* const lds = lds_all[grp];                                                                   \
  const float2* tw = twl;                                                                             \
  const int b = blockIdx.y;                                                                           \
  const int row0 = blockIdx.x * 2 * C::L;                                                             \
  const int rows = g.rows;                                                                            \
  const int j0 = tid % C::TPL, pc = tid / C::TPL;                                                     \
  const int ra = row0 + 2 * pc;                                                                       \
  const Inst& I = inst[b];                                                                            \
  constexpr int TWN = stage_tw_loads<N, C::PV>(G * C::NT);                                            \
  float2 twr[TWN];

// momentum (k_momentum): one group, blockIdx.z = axis
template <int N>
__global__ __launch_bounds__((ZCfg<N, true>::NT)) void k_momentum_small(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ tw_g) {
  KW_ZSMALL_PROLOGUE(1)
  const int ax = blockIdx.z;
  float2* const sp = fl.spec[ax] + b * g.nspec;
  float2 As[C::IT], Bs[C::IT];
  pair_load<C>(As, Bs, sp, row0, rows, g.nhp, tid);
  load_stage_tw<N, C::PV, G * C::NT>(twr, tw_g, threadIdx.x);
  const int t = step_of(fl, b);
  KW_ROWS_CLAMPED
  const auto u = gw(fl.u[ax] + b * g.ntot);
  const Src& src = I.srcu[ax];
  const bool zax = ax == g.nd - 1;
  float2 uo[C::E], dr[C::E];
  float pz[C::E], ph[2];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    uo[m] = make_float2(u[i0], u[i0 + N]);
    dr[m] = make_float2(ld(I.dtr0[ax], i0, I.dtr0_s), ld(I.dtr0[ax], i0 + N, I.dtr0_s));
    pz[m] = 1.f;
  }
  if (zax) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) pz[m] = gp(I.pmlsg[ax])[j0 + m * C::TPL];
  }
  pml_rows(I.pmlsg, g, ax, rA, ph);
  if (t >= I.nt) return;
  put_stage_tw<N, C::PV, G * C::NT>(twr, twl, threadIdx.x);
  pair_put<C>(lds, As, Bs, tid);
  float2 gv[C::E];
  inv_from_lds<C>(lds, tw, tid, gv);
  const int smode = src_mode_at(src, t);
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    gv[m].x = pml_update(pz[m] * ph[0], uo[m].x, dr[m].x, gv[m].x);
    gv[m].y = pml_update(pz[m] * ph[1], uo[m].y, dr[m].y, gv[m].y);
  }
  add_filtered_source<C>(src, smode, t, src.fac[ax], iA, lds, fl, g, b, tw, row0, rows, tid, gv);
  if (inside) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      u[iA + m * C::TPL] = gv[m].x;
      u[iA + N + m * C::TPL] = gv[m].y;
    }
  }
  if (src_is_point(smode) && inside) {
    for (int h = 0; h < 2; ++h) {
      const int r = ra + h;
      if (gp(src.row_ptr)[r] == gp(src.row_ptr)[r + 1]) continue;
      for (int m = 0; m < C::E; ++m) {
        const int n = j0 + m * C::TPL;
        float v;
        if (!csr_lookup(src, r, n, t, v)) continue;
        const float uv = src_point(smode, get_lane(gv, m, h), src.fac[ax], v);
        u[(int64_t)r * N + n] = uv;
        set_lane(gv, m, h, uv);
      }
    }
  }
  fwd_from_regs<C>(lds, gv, sp, tw, row0, rows, g.nhp, tid);
}

// mass conservation (k_mass): group i holds axis i; the divergence terms and the new split
// densities of the axes meet in LDS and are added in axis order.  One form serves plans
// with and without a filtered source and the adjoint replay (Fields::adjD).
template <int N, int ND>
__global__ __launch_bounds__((ZCfg<N, true>::NT * ND)) void k_mass_small(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ tw_g, int flags) {
  KW_ZSMALL_PROLOGUE(ND)
  __shared__ float2 exd[ND][C::E * C::NT], exr[ND][C::E * C::NT];
  float2 As[C::IT], Bs[C::IT];
  pair_load<C>(As, Bs, fl.spec[grp] + b * g.nspec, row0, rows, g.nhp, tid);
  load_stage_tw<N, C::PV, G * C::NT>(twr, tw_g, threadIdx.x);
  const int t = step_of(fl, b);
  KW_ROWS_CLAMPED
  const int64_t off = b * g.ntot;
  const Src& src = I.srcp;
  const bool powerlaw = flags & (FLAG_POWERLAW_ABS | FLAG_POWERLAW_DISP);
  const auto rho = gw(fl.rho[grp] + off);
  float2 ro[C::E], r0v[C::E], qv[C::E], c2v[C::E];
  float pz[C::E], ph[2];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    ro[m] = make_float2(rho[i0], rho[i0 + N]);
    r0v[m] = make_float2(ld(I.rho0, i0, I.rho0_s), ld(I.rho0, i0 + N, I.rho0_s));
    c2v[m] = make_float2(ld(I.c0sq, i0, I.c0sq_s), ld(I.c0sq, i0 + N, I.c0sq_s));
    pz[m] = 1.f;
  }
  if (flags & FLAG_NONLINEAR) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) qv[m] = make_float2(gp(fl.rhoi)[off + iA + m * C::TPL], gp(fl.rhoi)[off + iA + N + m * C::TPL]);
  }
  if (grp == ND - 1) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) pz[m] = gp(I.pml[ND - 1])[j0 + m * C::TPL];
  }
  pml_rows(I.pml, g, grp, rA, ph);
  if (t >= I.nt) return;
  const int smode = src_mode_at(src, t);
  const bool filtered = smode == SRC_CHAIN || smode == SRC_PATTERN;
  put_stage_tw<N, C::PV, G * C::NT>(twr, twl, threadIdx.x);
  pair_put<C>(lds, As, Bs, tid);
  __syncthreads();  // twiddles
  float2 d[C::E], ch[C::E], res[C::E];
  inv_from_lds<C>(lds, tw, tid, d);
  if (filtered) filtered_source<C>(src, smode, t, iA, lds, fl, g, b, tw, row0, rows, tid, ch);
  const float fac = src.fac[grp];
  if (flags & FLAG_NONLINEAR) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) qv[m] = make_float2(fmaf(2.f, qv[m].x, r0v[m].x), fmaf(2.f, qv[m].y, r0v[m].y));
  } else {
#pragma unroll
    for (int m = 0; m < C::E; ++m) qv[m] = r0v[m];
  }
#pragma unroll
  for (int m = 0; m < C::E; ++m)
    res[m] = make_float2(pml_update(pz[m] * ph[0], ro[m].x, I.dt * qv[m].x, d[m].x), pml_update(pz[m] * ph[1], ro[m].y, I.dt * qv[m].y, d[m].y));
  if (filtered) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) res[m] = make_float2(fmaf(fac, ch[m].x, res[m].x), fmaf(fac, ch[m].y, res[m].y));
  }
  if (inside) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      rho[iA + m * C::TPL] = res[m].x;
      rho[iA + N + m * C::TPL] = res[m].y;
    }
  }
  if (fl.adjD && inside) {  // adjoint replay: Dop_i u_i
    const auto dd = gw(fl.adjD + (int64_t)grp * gridDim.y * g.ntot + off);
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      dd[iA + m * C::TPL] = d[m].x;
      dd[iA + N + m * C::TPL] = d[m].y;
    }
  }
  if (src_is_point(smode) && inside) {
    for (int h = 0; h < 2; ++h) {
      const int r = ra + h;
      if (gp(src.row_ptr)[r] == gp(src.row_ptr)[r + 1]) continue;
      for (int m = 0; m < C::E; ++m) {
        const int n = j0 + m * C::TPL;
        float v;
        if (!csr_lookup(src, r, n, t, v)) continue;
        const float x = src_point(smode, get_lane(res, m, h), fac, v);
        rho[(int64_t)r * N + n] = x;
        set_lane(res, m, h, x);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    exd[grp][m * C::NT + tid] = d[m];
    exr[grp][m * C::NT + tid] = res[m];
  }
  __syncthreads();
  float2 divu[C::E], rt[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    float2 ds = make_float2(0.f, 0.f), rs = ds;
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      ds = cadd(ds, exd[i][m * C::NT + tid]);
      rs = cadd(rs, exr[i][m * C::NT + tid]);
    }
    divu[m] = ds;
    rt[m] = rs;
  }
  // group 0: p (or rho0 div u) and its transform; group 1: the density sum and, with
  // dispersion, its transform
  if (grp == 1 && fl.rhot && inside) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      gw(fl.rhot)[off + iA + m * C::TPL] = rt[m].x;
      gw(fl.rhot)[off + iA + N + m * C::TPL] = rt[m].y;
    }
  }
  if (grp == 0) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      float out[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t idx = iA + h * N + m * C::TPL;
        const float r0 = h ? r0v[m].y : r0v[m].x;
        const float du = h ? divu[m].y : divu[m].x;
        const float rtv = h ? rt[m].y : rt[m].x;
        if (powerlaw) {
          out[h] = r0 * du;
        } else {
          float q = rtv;
          const float c2 = h ? c2v[m].y : c2v[m].x;
          if (flags & FLAG_STOKES) {
            q = fmaf(tau_at(I, idx, c2) * r0, du, q);
            if (fl.adjA && inside) gw(fl.adjA)[off + idx] = r0 * du;
          }
          if (flags & FLAG_NONLINEAR) q += ld(I.bona, idx, I.bona_s) * rtv * rtv / (2.f * r0);
          out[h] = c2 * q;
        }
      }
      if (inside && !powerlaw) {
        gw(fl.p)[off + iA + m * C::TPL] = out[0];
        gw(fl.p)[off + iA + N + m * C::TPL] = out[1];
      }
      rt[m] = make_float2(out[0], out[1]);
    }
  }
  const bool fwd = grp == 0 ? (!powerlaw || (flags & FLAG_POWERLAW_ABS)) : grp == 1 && (flags & FLAG_POWERLAW_DISP);
  if (!C::WS || fwd) fwd_from_regs<C>(lds, rt, fl.spec[grp] + b * g.nspec, tw, row0, rows, g.nhp, tid, fwd);
}

// equation of state with power-law terms (k_eos): group 0 transforms the absorption
// operand, group 1 the dispersion operand
template <int N>
__global__ __launch_bounds__((ZCfg<N, true>::NT * 2)) void k_eos_small(Geom g, Fields fl, const Inst* __restrict__ inst, const float2* __restrict__ tw_g, int flags) {
  KW_ZSMALL_PROLOGUE(2)
  __shared__ float2 ex[C::E * C::NT], exc[C::E * C::NT];
  const bool abs = flags & FLAG_POWERLAW_ABS, disp = flags & FLAG_POWERLAW_DISP;
  float2 As[C::IT], Bs[C::IT];
  pair_load<C>(As, Bs, fl.spec[grp] + b * g.nspec, row0, rows, g.nhp, tid);
  load_stage_tw<N, C::PV, G * C::NT>(twr, tw_g, threadIdx.x);
  const int t = step_of(fl, b);
  KW_ROWS_CLAMPED
  const int64_t off = b * g.ntot;
  float2 rtv[C::E], c2v[C::E], r0v[C::E], bav[C::E], co[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    c2v[m] = make_float2(ld(I.c0sq, i0, I.c0sq_s), ld(I.c0sq, i0 + N, I.c0sq_s));
    rtv[m] = make_float2(gp(fl.rhot)[off + i0], gp(fl.rhot)[off + i0 + N]);
  }
  if (flags & FLAG_NONLINEAR) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const int64_t i0 = iA + m * C::TPL;
      r0v[m] = make_float2(ld(I.rho0, i0, I.rho0_s), ld(I.rho0, i0 + N, I.rho0_s));
      bav[m] = make_float2(ld(I.bona, i0, I.bona_s), ld(I.bona, i0 + N, I.bona_s));
    }
  }
  if (t >= I.nt) return;
  put_stage_tw<N, C::PV, G * C::NT>(twr, twl, threadIdx.x);
  pair_put<C>(lds, As, Bs, tid);
  // this group's coefficient, tau or eta
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    if (grp == 0 && abs) co[m] = make_float2(tau_at(I, i0, c2v[m].x), tau_at(I, i0 + N, c2v[m].y));
    if (grp == 1 && disp) co[m] = make_float2(eta_at(I, i0, c2v[m].x), eta_at(I, i0 + N, c2v[m].y));
  }
  __syncthreads();  // twiddles
  float2 v[C::E];
  inv_from_lds<C>(lds, tw, tid, v);
  float* const keep = grp == 0 ? (abs ? fl.adjA : nullptr) : (disp ? fl.adjB : nullptr);
  if (inside && keep) {  // adjoint replay: keep the operands
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      gw(keep)[off + iA + m * C::TPL] = v[m].x;
      gw(keep)[off + iA + N + m * C::TPL] = v[m].y;
    }
  }
  if (grp == 1 && disp) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      ex[m * C::NT + tid] = v[m];
      exc[m * C::NT + tid] = co[m];
    }
  }
  __syncthreads();
  if (grp == 0) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const float2 bv = disp ? ex[m * C::NT + tid] : make_float2(0.f, 0.f), eta = disp ? exc[m * C::NT + tid] : make_float2(0.f, 0.f);
      float out[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float rt = h ? rtv[m].y : rtv[m].x;
        float q = rt;
        if (abs) q = fmaf(h ? co[m].y : co[m].x, h ? v[m].y : v[m].x, q);
        if (disp) q = fmaf(-(h ? eta.y : eta.x), h ? bv.y : bv.x, q);
        if (flags & FLAG_NONLINEAR) q += (h ? bav[m].y : bav[m].x) * rt * rt / (2.f * (h ? r0v[m].y : r0v[m].x));
        out[h] = (h ? c2v[m].y : c2v[m].x) * q;
      }
      if (inside) {
        gw(fl.p)[off + iA + m * C::TPL] = out[0];
        gw(fl.p)[off + iA + N + m * C::TPL] = out[1];
      }
      v[m] = make_float2(out[0], out[1]);
    }
  }
  if (!C::WS || grp == 0) fwd_from_regs<C>(lds, v, fl.spec[0] + b * g.nspec, tw, row0, rows, g.nhp, tid, grp == 0);
}

// Supported line lengths, in four radix families.  Launcher files are compiled
// once per family (-DKW_GROUP=0..3) so the many template instantiations build
// in parallel; KW_GROUP_SIZES lists the family of the current translation unit
// and KW_GNAME(f) names its launcher f_g<family>.
#define KW_SIZES_G0(X) X(16) X(32) X(64) X(128) X(256) X(512) X(1024)
#define KW_SIZES_G1(X) X(24) X(48) X(96) X(192) X(384) X(768)
#define KW_SIZES_G2(X) X(40) X(80) X(160) X(320) X(640)
#define KW_SIZES_G3(X) X(56) X(112) X(224) X(448)
#define KW_FOR_SIZES(X) KW_SIZES_G0(X) KW_SIZES_G1(X) KW_SIZES_G2(X) KW_SIZES_G3(X)
#define KW_CAT_(a, b) a##b
#define KW_CAT(a, b) KW_CAT_(a, b)
#ifdef KW_GROUP
#define KW_GROUP_SIZES KW_CAT(KW_SIZES_G, KW_GROUP)
#define KW_GNAME(f) KW_CAT(f##_g, KW_GROUP)
#endif

inline bool size_supported_impl(int n) {
  switch (n) {
#define KW_CASE(S) case S: return true;
    KW_FOR_SIZES(KW_CASE)
#undef KW_CASE
    default: return false;
  }
}

// Whether a contiguous-axis kernel takes its small-grid form: tpl lanes per row pair in
// each of `groups` groups or grid layers (kw_dispatch.hip).
bool z_small(const Geom& g, int nb, int tpl, int groups);

inline dim3 zgrid(const Geom& g, int lpairs, int nb, int nz) {
  const int npairs = (g.rows + 1) / 2;
  return dim3((npairs + lpairs - 1) / lpairs, nb, nz);
}

// switch over the current family's sizes; a size outside it leaves *handled false
#define KW_ZDISPATCH(NAME)                                                 \
  *handled = true;                                                         \
  switch (g.nz) {                                                          \
    KW_GROUP_SIZES(NAME)                                                   \
    default: *handled = false; return hipSuccess;                          \
  }

}  // namespace kw
