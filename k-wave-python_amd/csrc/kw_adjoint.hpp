// Reverse-time (discrete adjoint) kernels of the step, for the
// gradient of a sensor-trace functional with respect to the sound speed.
//
// Forward step t (kw_kernels.hpp; reference kspace_solver.py:691-747):
//   u_i = a_i^2 u_i - a_i beta_i Gop_i p,   rho_i = b_i^2 rho_i - b_i dt rho0 Dop_i u_i + s_i,
//   p = c^2 sum_i rho_i,                    y = S p
// with a = pml_sg, b = pml, beta_i = dt / rho0_sg_i.  The operator tables are
// Hermitian, so Gop_i^T = -Dop_i and Dop_i^T = -Gop_i: the reverse step is the
// forward one with gradient and divergence swapped.  One reverse step:
//   k_adj_scatter   pbar += S^T r_t
//   k_adj_eos       rbar_i += c^2 pbar; cbar += 2 p pbar / c; R = sum_i fac_i rbar_i;
//                   w_i = b_i dt rho0 rbar_i -> F_z;  rbar_i = b_i^2 rbar_i
//   (x/y passes)    Gop_i on w_i
//   k_adj_mom       ubar_i += Gop_i w_i; v_i = a_i beta_i ubar_i -> F_z; ubar_i = a_i^2 ubar_i
//   (x/y passes)    Dop_i on v_i
//   k_adj_sum       pbar = sum_i Dop_i v_i
//   k_adj_srcgrad   cbar += -(scale / c) sig(t) [K R] at the source points
//
// Absorbing media (linear): the equation of state gains c^2 (tau A - eta B),
// A = L1[rho0 d] (Stokes: rho0 d), d = sum_i Dop_i u_i, B = L2[sum rho]; the forward
// replay keeps A and B of every step (Fields::adjA/adjB).  With w = c^2 pbar:
//   cbar += w ((y-1) tau A - y eta B) / c,  rbar_i += w - L2[eta w],
//   and the gradient jobs act on b dt rho0 rbar_i - rho0 L1[tau w] (Stokes: tau w).
// For the power law k_adj_abs1 forms tau w and eta w (forward z-FFT into spectra 0
// and 1) and the speed term; the fractional column passes apply L1, L2; k_adj_eos
// then reads both back.
//
// Dirichlet pressure source: at its points the step overwrote every rho_i with
// fac_i sig / (D c^2), so cbar gains -2 fac_i v rbar_i / c there and rbar_i is
// cleared before it is carried back through the mass update.
//
// B/A (nonlinear): rbar_i also gains w B/A S^t / rho0, the gradient-job input is
// scaled by (2 S^{t-1} + rho0) / rho0, and -2 dt sum_i b_i d_i^t rbar_i goes to every
// rbar_j of step t-1 (S and d_i = Dop_i u_i kept by the replay).
//
// What bounds the sweep: on large grids memory, so every thread's loads are issued in
// straight-line batches (sources and PML rows without per-element branches); on small ones
// the chain of latencies of a workgroup, so the small forms run one wavefront per row
// group and axis (kw_kernels.hpp, the same rule z_small and the same bits).  Measured, us a
// launch before -> now: 64^3 power law with B/A k_adj_eos 41 -> 11.4, k_adj_abs1 20 -> 10.9,
// k_adj_mom 9 -> 7.6, k_adj_sum 7 -> 5.0; 1024^2 lossless eos 28.7 -> 14.1, mom 16.2 -> 13.5,
// sum 8.7 -> 7.4; 128^3 (large forms) eos 79.5 -> 51.1 (lossless 34.8 -> 24.9), abs1 33.8 ->
// 20.8, mom 27.6 -> 26.9.
#pragma once
#include "kw_kernels.hpp"

namespace kw {

// One element of the mass update's adjoint along an axis: the input w of the gradient job
// and the density adjoint rn carried back.  The roundings are spelled out, since the large-
// and small-grid forms must agree (kw_fft.hpp, cmul).
struct AdjElem { float w, rn; };
__device__ __forceinline__ AdjElem adj_elem(float rbt, float s, float dt, float r0, float nl, float dbar) {
  return {fmaf(-r0, dbar, s * dt * r0 * nl * rbt), s * s * rbt};
}

// Operands of a thread's elements shared by the axes: w = c^2 pbar, rho0, the B/A term of
// the equation of state, the nonlinear factor of the mass update, the Stokes term tau w.
// adj_load also adds the speed gradient's own term (lossless, Stokes).
template <class C, int ABS>
struct AdjOps {
  float2 wc[C::E], r0[C::E], ba[C::E], nl[C::E], tw[C::E];
};
template <class C, int ABS>
__device__ __forceinline__ void adj_load(AdjOps<C, ABS>& o, const AdjFields& af, const Inst& I, int64_t off, int64_t iA, bool speed,
                                         bool inside) {
  constexpr int N = C::N;
  const auto pb = gp(af.pb + off);
  float2 c2[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    c2[m] = make_float2(ld(I.c0sq, i0, I.c0sq_s), ld(I.c0sq, i0 + N, I.c0sq_s));
    o.r0[m] = make_float2(ld(I.rho0, i0, I.rho0_s), ld(I.rho0, i0 + N, I.rho0_s));
    o.wc[m] = make_float2(pb[i0], pb[i0 + N]);
  }
  if (ABS != 2 && speed) {  // the power law's speed terms are k_adj_abs1's
    // p = c^2 sum rho  ->  dJ/dc += 2 c sum(rho) pbar = 2 p pbar / c
    const auto cb = gw(af.cb + off);
    const auto pt = gp(af.pt + off);
    float2 ga[C::E], cv[C::E];
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const int64_t i0 = iA + m * C::TPL;
      ga[m] = make_float2(2.f * pt[i0] * o.wc[m].x / sqrtf(c2[m].x), 2.f * pt[i0 + N] * o.wc[m].y / sqrtf(c2[m].y));
      cv[m] = make_float2(cb[i0], cb[i0 + N]);
    }
    if constexpr (ABS == 1) {  // Stokes: tau = -2 a c, d tau/dc = tau / c, operand A = rho0 d
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        const int64_t i0 = iA + m * C::TPL;
        ga[m].x = fmaf(c2[m].x * o.wc[m].x * tau_at(I, i0, c2[m].x) / sqrtf(c2[m].x), gp(af.At)[off + i0], ga[m].x);
        ga[m].y = fmaf(c2[m].y * o.wc[m].y * tau_at(I, i0 + N, c2[m].y) / sqrtf(c2[m].y), gp(af.At)[off + i0 + N], ga[m].y);
      }
    }
    if (inside) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        cb[iA + m * C::TPL] = cv[m].x + ga[m].x;
        cb[iA + N + m * C::TPL] = cv[m].y + ga[m].y;
      }
    }
  }
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    o.wc[m] = make_float2(c2[m].x * o.wc[m].x, c2[m].y * o.wc[m].y);
    rounded(o.wc[m].x);
    rounded(o.wc[m].y);
    o.nl[m] = make_float2(1.f, 1.f);
    o.ba[m] = make_float2(0.f, 0.f);
    if constexpr (ABS == 1) {
      const int64_t i0 = iA + m * C::TPL;
      o.tw[m] = make_float2(tau_at(I, i0, c2[m].x) * o.wc[m].x, tau_at(I, i0 + N, c2[m].y) * o.wc[m].y);
    } else {
      o.tw[m] = make_float2(0.f, 0.f);
    }
  }
  if (af.nonlin) {  // EOS: c^2 B/A S^2 / (2 rho0);  mass: d_i (2 S^{t-1} + rho0) / rho0
    float2 S[C::E], Sp[C::E];
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const int64_t i0 = iA + m * C::TPL;
      S[m] = make_float2(gp(af.St)[off + i0], gp(af.St)[off + i0 + N]);
      Sp[m] = make_float2(gp(af.Sp)[off + i0], gp(af.Sp)[off + i0 + N]);
      o.ba[m] = make_float2(ld(I.bona, i0, I.bona_s), ld(I.bona, i0 + N, I.bona_s));
    }
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      o.ba[m] = make_float2(o.wc[m].x * o.ba[m].x * S[m].x / o.r0[m].x, o.wc[m].y * o.ba[m].y * S[m].y / o.r0[m].y);
      o.nl[m] = make_float2(1.f + 2.f * Sp[m].x / o.r0[m].x, 1.f + 2.f * Sp[m].y / o.r0[m].y);
    }
  }
}
// Dirichlet point at a thread's elements: rho_i = fac_i v after the mass update, v = sig /
// (D c^2).  Its speed term goes to gd, and rbt carries no adjoint further back.
template <class C>
__device__ __forceinline__ void adj_dirichlet(const Src& src, float fac, const Inst& I, int t, int rA, int j0, int64_t iA, float2 (&rbt)[C::E],
                                              float2 (&gd)[C::E]) {
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    float v;
    gd[m] = make_float2(0.f, 0.f);
    if (csr_lookup(src, rA, j0 + m * C::TPL, t, v)) {
      gd[m].x = -2.f * fac * v * rbt[m].x / sqrtf(ld(I.c0sq, iA + m * C::TPL, I.c0sq_s));
      rbt[m].x = 0.f;
    }
    if (csr_lookup(src, rA + 1, j0 + m * C::TPL, t, v)) {
      gd[m].y = -2.f * fac * v * rbt[m].y / sqrtf(ld(I.c0sq, iA + C::N + m * C::TPL, I.c0sq_s));
      rbt[m].y = 0.f;
    }
  }
}

// ABS: 0 lossless, 1 Stokes, 2 power law (spectra 0 and 1 hold L1[tau w], L2[eta w])
template <int N, int ND, int ABS>
__global__ __launch_bounds__(ZCfg<N>::NT) void k_adj_eos(Geom g, Fields fl, AdjFields af, const Inst* __restrict__ inst,
                                                         const float2* __restrict__ tw_g, int t) {
  KW_ZPASS_PROLOGUE
  const Inst& I = inst[b];
  float2 l1[ABS == 2 ? C::E : 1], l2[ABS == 2 ? C::E : 1];
  if constexpr (ABS == 2) {
    inv_to_regs<C>(lds, fl.spec[0] + b * g.nspec, tw, row0, rows, g.nhp, tid, l1);
    if (af.disp) {
      inv_to_regs<C>(lds, fl.spec[1] + b * g.nspec, tw, row0, rows, g.nhp, tid, l2);
    } else {
#pragma unroll
      for (int m = 0; m < C::E; ++m) l2[m] = make_float2(0.f, 0.f);
    }
  }
  __shared__ float pmlz[N];
  for (int i_ = tid; i_ < N; i_ += C::NT) pmlz[i_] = gp(I.pml[ND - 1])[i_];
  __syncthreads();
  KW_ROWS_CLAMPED
  const int64_t off = b * g.ntot;
  const Src& src = I.srcp;
  const bool srcon = src.mode != SRC_NONE && t < src.len;
  const bool dir = srcon && src.mode == SRC_DIRICHLET;
  float ph[ND][2];
#pragma unroll
  for (int i = 0; i < ND; ++i) pml_rows(I.pml, g, i, rA, ph[i]);
  AdjOps<C, ABS> o;
  adj_load<C, ABS>(o, af, I, off, iA, true, inside);
  // B/A: the adjoint of S^{t-1} through the mass update's factor, -2 dt sum_i b_i d_i rbar_i,
  // goes to every rbar_j of the step before (added after the axis loop)
  float2 sb[C::E], rs[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) rs[m] = sb[m] = make_float2(0.f, 0.f);
  const int64_t nf = (int64_t)gridDim.y * g.ntot;
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const auto rb = gw(af.rb[i] + off);
    float2 rbt[C::E], w[C::E];
#pragma unroll
    for (int m = 0; m < C::E; ++m) rbt[m] = make_float2(rb[iA + m * C::TPL], rb[iA + N + m * C::TPL]);
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      rbt[m] = cadd(cadd(rbt[m], o.wc[m]), o.ba[m]);
      if constexpr (ABS == 2) rbt[m] = csub(rbt[m], l2[m]);
    }
    if (dir) {
      float2 gd[C::E];
      adj_dirichlet<C>(src, src.fac[i], I, t, rA, j0, iA, rbt, gd);
      if (inside) {
        const auto cb = gw(af.cb + off);
#pragma unroll
        for (int m = 0; m < C::E; ++m) {
          cb[iA + m * C::TPL] += gd[m].x;
          cb[iA + N + m * C::TPL] += gd[m].y;
        }
      }
    }
    const float fac = src.fac[i];
    float2 rn[C::E], sc[C::E];
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const float sz = (i == ND - 1) ? pmlz[j0 + m * C::TPL] : 1.f;
      sc[m] = make_float2(sz * ph[i][0], sz * ph[i][1]);
      const float2 db = ABS == 2 ? l1[ABS == 2 ? m : 0] : o.tw[m];
      const AdjElem a = adj_elem(rbt[m].x, sc[m].x, I.dt, o.r0[m].x, o.nl[m].x, db.x);
      const AdjElem c = adj_elem(rbt[m].y, sc[m].y, I.dt, o.r0[m].y, o.nl[m].y, db.y);
      w[m] = make_float2(a.w, c.w);
      rn[m] = make_float2(a.rn, c.rn);
      rs[m] = make_float2(fmaf(fac, rbt[m].x, rs[m].x), fmaf(fac, rbt[m].y, rs[m].y));
    }
    if (af.nonlin) {
      const auto Dt = gp(af.Dt + (int64_t)i * nf + off);
      float2 dv[C::E];
#pragma unroll
      for (int m = 0; m < C::E; ++m) dv[m] = make_float2(Dt[iA + m * C::TPL], Dt[iA + N + m * C::TPL]);
#pragma unroll
      for (int m = 0; m < C::E; ++m)
        sb[m] = make_float2(fmaf(-2.f * I.dt * sc[m].x * dv[m].x, rbt[m].x, sb[m].x), fmaf(-2.f * I.dt * sc[m].y * dv[m].y, rbt[m].y, sb[m].y));
    }
    if (inside) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        rb[iA + m * C::TPL] = rn[m].x;
        rb[iA + N + m * C::TPL] = rn[m].y;
      }
    }
    fwd_from_regs<C>(lds, w, fl.spec[i] + b * g.nspec, tw, row0, rows, g.nhp, tid);
  }
  if (af.nonlin && inside) {
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const auto rb = gw(af.rb[i] + off);
      float2 r[C::E];
#pragma unroll
      for (int m = 0; m < C::E; ++m) r[m] = make_float2(rb[iA + m * C::TPL], rb[iA + N + m * C::TPL]);
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        rb[iA + m * C::TPL] = r[m].x + sb[m].x;
        rb[iA + N + m * C::TPL] = r[m].y + sb[m].y;
      }
    }
  }
  if (srcon && inside) {
    const auto R = gw(af.R + off);
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      R[iA + m * C::TPL] = rs[m].x;
      R[iA + N + m * C::TPL] = rs[m].y;
    }
  }
}

// Small grids: group i holds axis i (see the small-grid updates in kw_kernels.hpp).
template <int N, int ND, int ABS>
__global__ __launch_bounds__((ZCfg<N, true>::NT * ND)) void k_adj_eos_small(Geom g, Fields fl, AdjFields af, const Inst* __restrict__ inst,
                                                                            const float2* __restrict__ tw_g, int t) {
  KW_ZSMALL_PROLOGUE(ND)
  __shared__ float2 ex1[ND][C::E * C::NT], ex2[ND][C::E * C::NT];
  float2 As[ABS == 2 ? C::IT : 1], Bs[ABS == 2 ? C::IT : 1];
  if constexpr (ABS == 2) pair_load<C>(As, Bs, fl.spec[grp == 0 ? 0 : 1] + b * g.nspec, row0, rows, g.nhp, tid);
  load_stage_tw<N, C::PV, G * C::NT>(twr, tw_g, threadIdx.x);
  KW_ROWS_CLAMPED
  const int64_t off = b * g.ntot;
  const Src& src = I.srcp;
  const auto rb = gw(af.rb[grp] + off);
  float2 rbt[C::E], dv[C::E];
  float pz[C::E], ph[2];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    rbt[m] = make_float2(rb[iA + m * C::TPL], rb[iA + N + m * C::TPL]);
    pz[m] = 1.f;
  }
  if (grp == ND - 1) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) pz[m] = gp(I.pml[ND - 1])[j0 + m * C::TPL];
  }
  pml_rows(I.pml, g, grp, rA, ph);
  if (af.nonlin) {
    const auto Dt = gp(af.Dt + ((int64_t)grp * gridDim.y + b) * g.ntot);
#pragma unroll
    for (int m = 0; m < C::E; ++m) dv[m] = make_float2(Dt[iA + m * C::TPL], Dt[iA + N + m * C::TPL]);
  }
  put_stage_tw<N, C::PV, G * C::NT>(twr, twl, threadIdx.x);
  if constexpr (ABS == 2) pair_put<C>(lds, As, Bs, tid);
  AdjOps<C, ABS> o;
  adj_load<C, ABS>(o, af, I, off, iA, grp == 0, inside);
  __syncthreads();  // twiddles
  float2 l1[ABS == 2 ? C::E : 1];
  if constexpr (ABS == 2) {
    float2 lv[C::E];
    inv_from_lds<C>(lds, tw, tid, lv);
    if (grp < 2) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) ex1[grp][m * C::NT + tid] = lv[m];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < C::E; ++m) l1[m] = ex1[0][m * C::NT + tid];
    if (af.disp) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) lv[m] = ex1[1][m * C::NT + tid];
    } else {
#pragma unroll
      for (int m = 0; m < C::E; ++m) lv[m] = make_float2(0.f, 0.f);
    }
    __syncthreads();  // ex1 is used again
#pragma unroll
    for (int m = 0; m < C::E; ++m) rbt[m] = csub(cadd(cadd(rbt[m], o.wc[m]), o.ba[m]), lv[m]);
  } else {
#pragma unroll
    for (int m = 0; m < C::E; ++m) rbt[m] = cadd(cadd(rbt[m], o.wc[m]), o.ba[m]);
  }
  const bool srcon = src.mode != SRC_NONE && t < src.len;
  if (srcon && src.mode == SRC_DIRICHLET) {
    float2 gd[C::E];
    adj_dirichlet<C>(src, src.fac[grp], I, t, rA, j0, iA, rbt, gd);
#pragma unroll
    for (int m = 0; m < C::E; ++m) ex2[grp][m * C::NT + tid] = gd[m];
    __syncthreads();
    if (grp == 0 && inside) {
      const auto cb = gw(af.cb + off);
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        float2 c = make_float2(cb[iA + m * C::TPL], cb[iA + N + m * C::TPL]);
#pragma unroll
        for (int i = 0; i < ND; ++i) c = cadd(c, ex2[i][m * C::NT + tid]);
        cb[iA + m * C::TPL] = c.x;
        cb[iA + N + m * C::TPL] = c.y;
      }
    }
    __syncthreads();  // ex2 is used again
  }
  float2 w[C::E], rn[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const float2 sc = make_float2(pz[m] * ph[0], pz[m] * ph[1]);
    const float2 db = ABS == 2 ? l1[ABS == 2 ? m : 0] : o.tw[m];
    const AdjElem a = adj_elem(rbt[m].x, sc.x, I.dt, o.r0[m].x, o.nl[m].x, db.x);
    const AdjElem c = adj_elem(rbt[m].y, sc.y, I.dt, o.r0[m].y, o.nl[m].y, db.y);
    w[m] = make_float2(a.w, c.w);
    rn[m] = make_float2(a.rn, c.rn);
    ex1[grp][m * C::NT + tid] = rbt[m];
    if (af.nonlin) ex2[grp][m * C::NT + tid] = make_float2(-2.f * I.dt * sc.x * dv[m].x, -2.f * I.dt * sc.y * dv[m].y);
  }
  __syncthreads();
  if (af.nonlin) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      float2 sb = make_float2(0.f, 0.f);
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        const float2 p = ex2[i][m * C::NT + tid], r = ex1[i][m * C::NT + tid];
        sb = make_float2(fmaf(p.x, r.x, sb.x), fmaf(p.y, r.y, sb.y));
      }
      rounded(rn[m].x);
      rounded(rn[m].y);
      rn[m] = cadd(rn[m], sb);
    }
  }
  if (inside) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      rb[iA + m * C::TPL] = rn[m].x;
      rb[iA + N + m * C::TPL] = rn[m].y;
    }
  }
  if (grp == 0 && srcon && inside) {
    const auto R = gw(af.R + off);
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      float2 rs = make_float2(0.f, 0.f);
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        const float2 r = ex1[i][m * C::NT + tid];
        rs = make_float2(fmaf(src.fac[i], r.x, rs.x), fmaf(src.fac[i], r.y, rs.y));
      }
      R[iA + m * C::TPL] = rs.x;
      R[iA + N + m * C::TPL] = rs.y;
    }
  }
  fwd_from_regs<C>(lds, w, fl.spec[grp] + b * g.nspec, tw, row0, rows, g.nhp, tid);
}

// Power-law pre-pass of a reverse step: w = c^2 pbar,
//   cbar += 2 p pbar / c + w ((y-1) tau A - y eta B) / c,
// and the forward z-FFTs of tau w (spectrum 0) and eta w (spectrum 1, with dispersion).
// first, second: the parts a workgroup's group of lanes forms; the speed term is the first's.
template <class C>
__device__ __forceinline__ void adj_abs1_elems(const AdjFields& af, const Inst& I, int64_t off, int64_t iA, bool inside, bool first, bool second,
                                               float2 (&tv)[C::E], float2 (&ev)[C::E]) {
  constexpr int N = C::N;
  const auto pb = gp(af.pb + off);
  const auto pt = gp(af.pt + off);
  const auto cb = gw(af.cb + off);
  float2 c2[C::E], w[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    c2[m] = make_float2(ld(I.c0sq, i0, I.c0sq_s), ld(I.c0sq, i0 + N, I.c0sq_s));
    w[m] = make_float2(pb[i0], pb[i0 + N]);
  }
  float2 tau[C::E], eta[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    tau[m] = eta[m] = make_float2(0.f, 0.f);
    if (first) tau[m] = make_float2(tau_at(I, i0, c2[m].x), tau_at(I, i0 + N, c2[m].y));
    if (af.disp) eta[m] = make_float2(eta_at(I, i0, c2[m].x), eta_at(I, i0 + N, c2[m].y));
  }
  if (first) {
    float2 P[C::E], A[C::E], B[C::E], cv[C::E];
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      const int64_t i0 = iA + m * C::TPL;
      P[m] = make_float2(pt[i0], pt[i0 + N]);
      A[m] = make_float2(gp(af.At)[off + i0], gp(af.At)[off + i0 + N]);
      B[m] = make_float2(0.f, 0.f);
      cv[m] = make_float2(cb[i0], cb[i0 + N]);
    }
    if (af.disp) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) B[m] = make_float2(gp(af.Bt)[off + iA + m * C::TPL], gp(af.Bt)[off + iA + N + m * C::TPL]);
    }
    auto speed = [&](float c2v, float pbar, float pv, float ta, float et, float a, float bb) {
      const float c = sqrtf(c2v), ww = c2v * pbar;
      float gc = fmaf(ww * af.ym1 * ta / c, a, 2.f * pv * pbar / c);
      if (af.disp) gc = fmaf(-(ww * af.y * et / c), bb, gc);
      return gc;
    };
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      cv[m].x += speed(c2[m].x, w[m].x, P[m].x, tau[m].x, eta[m].x, A[m].x, B[m].x);
      cv[m].y += speed(c2[m].y, w[m].y, P[m].y, tau[m].y, eta[m].y, A[m].y, B[m].y);
    }
    if (inside) {
#pragma unroll
      for (int m = 0; m < C::E; ++m) {
        cb[iA + m * C::TPL] = cv[m].x;
        cb[iA + N + m * C::TPL] = cv[m].y;
      }
    }
  }
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const float2 ww = make_float2(c2[m].x * w[m].x, c2[m].y * w[m].y);
    tv[m] = make_float2(tau[m].x * ww.x, tau[m].y * ww.y);
    ev[m] = make_float2(eta[m].x * ww.x, eta[m].y * ww.y);
  }
}

template <int N>
__global__ __launch_bounds__(ZCfg<N>::NT) void k_adj_abs1(Geom g, Fields fl, AdjFields af, const Inst* __restrict__ inst,
                                                          const float2* __restrict__ tw_g) {
  KW_ZPASS_PROLOGUE
  const Inst& I = inst[b];
  KW_ROWS_CLAMPED
  float2 tv[C::E], ev[C::E];
  adj_abs1_elems<C>(af, I, b * g.ntot, iA, inside, true, true, tv, ev);
  fwd_from_regs<C>(lds, tv, fl.spec[0] + b * g.nspec, tw, row0, rows, g.nhp, tid);
  if (af.disp) fwd_from_regs<C>(lds, ev, fl.spec[1] + b * g.nspec, tw, row0, rows, g.nhp, tid);
}

template <int N>
__global__ __launch_bounds__((ZCfg<N, true>::NT * 2)) void k_adj_abs1_small(Geom g, Fields fl, AdjFields af, const Inst* __restrict__ inst,
                                                                            const float2* __restrict__ tw_g) {
  KW_ZSMALL_PROLOGUE(2)
  load_stage_tw<N, C::PV, G * C::NT>(twr, tw_g, threadIdx.x);
  KW_ROWS_CLAMPED
  float2 tv[C::E], ev[C::E];
  adj_abs1_elems<C>(af, I, b * g.ntot, iA, inside, grp == 0, grp == 1, tv, ev);
  put_stage_tw<N, C::PV, G * C::NT>(twr, twl, threadIdx.x);
  if (grp == 1) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) tv[m] = ev[m];
  }
  __syncthreads();  // twiddles
  const bool fwd = grp == 0 || af.disp;
  if (!C::WS || fwd) fwd_from_regs<C>(lds, tv, fl.spec[grp] + b * g.nspec, tw, row0, rows, g.nhp, tid, fwd);
}

template <int N, bool NAR>
__global__ __launch_bounds__((ZCfg<N, NAR>::NT)) void k_adj_mom(Geom g, Fields fl, AdjFields af, const Inst* __restrict__ inst,
                                                                const float2* __restrict__ tw_g, int t) {
  using C = ZCfg<N, NAR>;
  __shared__ float2 lds[C::LDS];
  __shared__ float2 twl[stage_tw_size<N, C::PV>()];
  const int tid = threadIdx.x, b = blockIdx.y, ax = blockIdx.z;
  const int row0 = blockIdx.x * 2 * C::L, rows = g.rows;
  const int j0 = tid % C::TPL, pc = tid / C::TPL, ra = row0 + 2 * pc;
  const float2* tw = twl;
  float2* sp = fl.spec[ax] + b * g.nspec;
  float2 As[C::IT], Bs[C::IT], twr[stage_tw_loads<N, C::PV>(C::NT)];
  pair_load<C>(As, Bs, sp, row0, rows, g.nhp, tid);
  load_stage_tw<N, C::PV, C::NT>(twr, tw_g, tid);
  const Inst& I = inst[b];
  KW_ROWS_CLAMPED
  const auto ub = gw(af.ub[ax] + b * g.ntot);
  // velocity source of this axis at step t: dirichlet points drop their adjoint; for an
  // additive one dJ/du_i^t goes to U (its speed term needs K applied, k_adj_srcgrad)
  const Src& us = I.srcu[ax];
  const bool uon = us.mode != SRC_NONE && t < us.len;
  const bool udir = uon && us.mode == SRC_DIRICHLET;
  float* const Ub = uon && !udir && af.U[ax] ? af.U[ax] + b * g.ntot : nullptr;
  const bool zax = ax == g.nd - 1;
  float2 uo[C::E], dr[C::E];
  float pz[C::E], ph[2];
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const int64_t i0 = iA + m * C::TPL;
    uo[m] = make_float2(ub[i0], ub[i0 + N]);
    dr[m] = make_float2(ld(I.dtr0[ax], i0, I.dtr0_s), ld(I.dtr0[ax], i0 + N, I.dtr0_s));
    pz[m] = 1.f;
  }
  if (zax) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) pz[m] = gp(I.pmlsg[ax])[j0 + m * C::TPL];
  }
  pml_rows(I.pmlsg, g, ax, rA, ph);
  put_stage_tw<N, C::PV, C::NT>(twr, twl, tid);
  pair_put<C>(lds, As, Bs, tid);
  float2 gv[C::E];
  inv_from_lds<C>(lds, tw, tid, gv);
#pragma unroll
  for (int m = 0; m < C::E; ++m) uo[m] = cadd(uo[m], gv[m]);
  if (udir) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      float v;
      if (csr_lookup(us, rA, j0 + m * C::TPL, t, v)) uo[m].x = 0.f;
      if (csr_lookup(us, rA + 1, j0 + m * C::TPL, t, v)) uo[m].y = 0.f;
    }
  }
  if (Ub && inside) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      gw(Ub)[iA + m * C::TPL] = uo[m].x;
      gw(Ub)[iA + N + m * C::TPL] = uo[m].y;
    }
  }
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    const float2 s = make_float2(pz[m] * ph[0], pz[m] * ph[1]);
    gv[m] = make_float2(s.x * dr[m].x * uo[m].x, s.y * dr[m].y * uo[m].y);
    uo[m] = make_float2(s.x * s.x * uo[m].x, s.y * s.y * uo[m].y);
  }
  if (inside) {
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      ub[iA + m * C::TPL] = uo[m].x;
      ub[iA + N + m * C::TPL] = uo[m].y;
    }
  }
  fwd_from_regs<C>(lds, gv, sp, tw, row0, rows, g.nhp, tid);
}

template <int N, int ND>
__global__ __launch_bounds__(ZCfg<N>::NT) void k_adj_sum(Geom g, Fields fl, AdjFields af, const Inst* __restrict__ inst,
                                                         const float2* __restrict__ tw_g) {
  KW_ZPASS_PROLOGUE
  (void)inst;
  KW_ROWS_CLAMPED
  float2 acc[C::E];
#pragma unroll
  for (int m = 0; m < C::E; ++m) acc[m] = make_float2(0.f, 0.f);
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    float2 d[C::E];
    inv_to_regs<C>(lds, fl.spec[i] + b * g.nspec, tw, row0, rows, g.nhp, tid, d);
#pragma unroll
    for (int m = 0; m < C::E; ++m) acc[m] = cadd(acc[m], d[m]);
  }
  if (inside) {
    const auto pb = gw(af.pb + b * g.ntot);
#pragma unroll
    for (int m = 0; m < C::E; ++m) {
      pb[iA + m * C::TPL] = acc[m].x;
      pb[iA + N + m * C::TPL] = acc[m].y;
    }
  }
}

template <int N, int ND>
__global__ __launch_bounds__((ZCfg<N, true>::NT * ND)) void k_adj_sum_small(Geom g, Fields fl, AdjFields af, const Inst* __restrict__ inst,
                                                                            const float2* __restrict__ tw_g) {
  KW_ZSMALL_PROLOGUE(ND)
  __shared__ float2 ex[ND][C::E * C::NT];
  float2 As[C::IT], Bs[C::IT], d[C::E];
  pair_load<C>(As, Bs, fl.spec[grp] + b * g.nspec, row0, rows, g.nhp, tid);
  load_stage_tw<N, C::PV, G * C::NT>(twr, tw_g, threadIdx.x);
  KW_ROWS_CLAMPED
  (void)I;
  put_stage_tw<N, C::PV, G * C::NT>(twr, twl, threadIdx.x);
  pair_put<C>(lds, As, Bs, tid);
  __syncthreads();  // twiddles
  inv_from_lds<C>(lds, tw, tid, d);
#pragma unroll
  for (int m = 0; m < C::E; ++m) ex[grp][m * C::NT + tid] = d[m];
  __syncthreads();
  if (grp || !inside) return;
  const auto pb = gw(af.pb + b * g.ntot);
#pragma unroll
  for (int m = 0; m < C::E; ++m) {
    float2 acc = make_float2(0.f, 0.f);
#pragma unroll
    for (int i = 0; i < ND; ++i) acc = cadd(acc, ex[i][m * C::NT + tid]);
    pb[iA + m * C::TPL] = acc.x;
    pb[iA + N + m * C::TPL] = acc.y;
  }
}

}  // namespace kw
