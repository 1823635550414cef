// sph_ghost.h -- the per-particle arithmetic of the ghosts and of the end of
// the force loop, shared by their kernels and by the tiles that do it
// themselves (sph_tile.h).  Contraction is off, so that both round alike.
#pragma once

#include "sph_loops.h"

namespace sphl {

// The smoothing-length iteration of one particle: the current h, its
// bracket, and (after ghost_step) the finished density.
struct GhostState {
  float h, left, right;
};
// Density sums of a particle: raw before ghost_step, final after a step that
// converged.
struct DensSums {
  float rho, rho_dh, wc, wc_dh, divv, rx, ry, rz;
};

// One step of runner_do_ghost (runner_ghost.c:1217-1461) on the raw sums at
// g.h: hydro_end_density (hydro.h:613-662, a = 1, H = 0), one Newton-Raphson
// / bisection step, and the tolerance test.  Returns true when the particle
// goes again at the new g.h (its sums are then of no further use); false
// when it has converged: g.h is the final h and `a` the finished density.
__device__ __forceinline__ bool ghost_step(const GhostArgs &ga, float m,
                                           GhostState &g, DensSums &a) {
#pragma clang fp contract(off)
  const float h_old = g.h;
  const float h_old_dim = h_old * h_old * h_old;
  const float h_old_dim_m1 = h_old * h_old;
  float left = g.left, right = g.right;
  float h_new;
  bool no_ngb = false;
  bool done = false;
  if ((double)a.wc < 1.e-5 * (double)kRoot) {
    no_ngb = true;
    h_new = 2.f * h_old;
  } else {
    const float h_inv = 1.0f / h_old;
    const float hid = h_inv * h_inv * h_inv;
    const float hid1 = hid * h_inv;
    a.rho = (a.rho + m * kRoot) * hid;
    a.rho_dh = (a.rho_dh - kDim * m * kRoot) * hid1;
    a.wc = (a.wc + kRoot) * hid;
    a.wc_dh = (a.wc_dh - kDim * kRoot) * hid1;
    const float rho_inv = 1.f / a.rho;
    a.rx *= hid1 * rho_inv;
    a.ry *= hid1 * rho_inv;
    a.rz *= hid1 * rho_inv;
    a.divv *= hid1 * rho_inv;
    const float n_sum = a.wc * h_old_dim;
    const float f = n_sum - ga.eta_dim;
    const float f_prime = a.wc_dh * h_old_dim + kDim * a.wc * h_old_dim_m1;
    if (n_sum < ga.eta_dim)
      left = fmaxf(left, h_old);
    else if (n_sum > ga.eta_dim)
      right = fminf(right, h_old);
    if (((h_old >= ga.h_max) && (f < 0.f)) ||
        ((h_old <= ga.h_min) && (f > 0.f))) {
      done = true;
      h_new = h_old;
    } else {
      h_new = h_old - f / (f_prime + 1.17549435e-38f);
      h_new = fminf(h_new, 2.f * h_old);
      h_new = fmaxf(h_new, 0.5f * h_old);
      h_new = fmaxf(h_new, left);
      h_new = fminf(h_new, right);
    }
  }
  if (!done && fabsf(h_new - h_old) > ga.eps * h_old) {
    float hn;
    if ((h_new == left && h_old == right) || (h_old == left && h_new == right))
      hn = cbrtf(0.5f * (left * left * left + right * right * right));
    else
      hn = h_new;
    if (hn < ga.h_max && hn > ga.h_min) {
      g.h = hn;
      g.left = left;
      g.right = right;
      return true;
    }
    if (hn <= ga.h_min) {
      g.h = ga.h_min;
    } else {
      g.h = ga.h_max;
      if (no_ngb) {
        // hydro_part_has_no_neighbours (hydro.h:791-825)
        const float hinv = 1.0f / g.h;
        const float hid = hinv * hinv * hinv;
        a.rho = m * kRoot * hid;
        a.wc = kRoot * hid;
        a.rho_dh = 0.f;
        a.wc_dh = 0.f;
        a.rx = a.ry = a.rz = 0.f;
        a.divv = 0.f;
      }
    }
  }
  return false;
}

// A particle whose iteration has converged: its h and finished density, and
// hydro_prepare_gradient + hydro_reset_gradient (hydro.h:671-750).
__device__ __forceinline__ void ghost_finish(const DevParts &d,
                                             const GhostArgs &ga, int i,
                                             float h, const DensSums &a) {
#pragma clang fp contract(off)
  d.h[i] = h;
  d.redo[i] = 0;
  d.rho[i] = a.rho;
  d.rho_dh[i] = a.rho_dh;
  d.wc[i] = a.wc;
  d.wc_dh[i] = a.wc_dh;
  d.divv[i] = a.divv;
  d.rotx[i] = a.rx;
  d.roty[i] = a.ry;
  d.rotz[i] = a.rz;
  const float curl_v = sqrtf(a.rx * a.rx + a.ry * a.ry + a.rz * a.rz);
  const float abs_div_v = fabsf(a.divv);
  const float u = d.u[i];
  const float P = kGasGm1 * u * a.rho;
  const float c = sqrtf(kGasGamma * P / a.rho);
  const float bal = abs_div_v / (abs_div_v + curl_v + 0.0001f * c / h);
  const float common = h * kDimInv / a.wc;
  float fgh;
  if (h > 0.9999f * ga.h_max) {
    fgh = 0.f;
  } else {
    const float gW = common * a.wc_dh;
    fgh = (gW < -0.9999f) ? 0.f : common * a.rho_dh / (1.f + gW);
  }
  d.P[i] = P;
  d.c[i] = c;
  d.f[i] = fgh;
  d.bal[i] = bal;
  const float alpha = d.alpha[i];
  // the gradient record, built here from the values at hand
  if (ga.grad_rec)
    d.rg[rec_slot(d, i)] = grad_rec_of(d, i, a.rho, u, c, alpha);
  if (ga.fresh_grad) return;  // the gradient loop starts from these itself
  d.vsig[i] = 2.f * c;
  d.avmax[i] = alpha;
  d.lapu[i] = 0.f;
  d.ng[i] = 0;
}

// runner_do_extra_ghost (runner_ghost.c:1016-1111) on one active particle
// whose gradient sums the caller holds: hydro_end_gradient,
// hydro_prepare_force (hydro.h:840-954, a = 1), hydro_reset_acceleration and
// timestep_limiter_prepare_force.
__device__ __forceinline__ void extra_ghost_one(const DevParts &d,
                                                const GhostArgs &ga, int i,
                                                int8_t tb, float vsig,
                                                float lapu_sum, float avmax) {
#pragma clang fp contract(off)
  const float h = d.h[i];
  const float h_inv = 1.0f / h;
  const float hid1 = h_inv * h_inv * h_inv * h_inv;
  const float lapu = lapu_sum * (2.f * hid1);
  d.lapu[i] = lapu;
  const float dt_alpha =
      tb <= 0 ? 0.f : (float)((double)(1LL << (tb + 1)) * ga.time_base);
  const float ksp = h * kGamma;
  const float ksp_inv = 1.f / ksp;
  const float rho = d.rho[i];
  const float u = d.u[i];
  const float P = kGasGm1 * u * rho;
  const float c = sqrtf(kGasGamma * P / rho);
  const float sct_inv = c * ksp_inv;
  const float divv = d.divv[i];
  const float div_v_dt =
      dt_alpha == 0.f ? 0.f : (divv - d.divv_prev[i]) / dt_alpha;
  const float S = divv < 0.f ? ksp * ksp * fmaxf(0.f, -div_v_dt) : 0.f;
  const float alpha_loc = ga.alpha_max * S / (c * c + S);
  float alpha = d.alpha[i];
  if (alpha_loc > alpha) {
    alpha = alpha_loc;
  } else {
    const float tr = dt_alpha * sct_inv * ga.visc_length;
    alpha += alpha_loc * tr;
    alpha /= (1.f + tr);
  }
  alpha = fmaxf(alpha, ga.alpha_min);
  d.alpha[i] = alpha;
  d.divv_prev[i] = divv;
  d.divv_dt[i] = div_v_dt;
  const float dtpi = vsig * ksp_inv;
  const float sqrt_u_inv = 1.f / sqrtf(u);
  float adt = ga.diff_beta * ksp * lapu * sqrt_u_inv;
  const float ad0 = d.adiff[i];
  adt -= (ad0 - ga.diff_alpha_min) * dtpi;
  float na = ad0 + adt * dt_alpha;
  na = fmaxf(na, ga.diff_alpha_min);
  const float lim = ga.diff_alpha_max * (1.f - avmax / ga.alpha_max);
  const float adiff = fminf(na, lim);
  d.adiff[i] = adiff;
  // the force record, built here from the values at hand
  if (ga.force_rec)
    d.rf[rec_slot(d, i)] =
        force_rec_of(d, i, tb, h, rho, P, c, alpha, adiff, u);
  if (ga.fresh_force) return;
  d.ax[i] = 0.f;
  d.ay[i] = 0.f;
  d.az[i] = 0.f;
  d.udt[i] = 0.f;
  d.hdt[i] = 0.f;
  d.nf[i] = 0;
  d.mintb[i] = (int8_t)(kNumTimeBins + 1);
}

// runner_do_end_hydro_force (runner_others.c:815-870) -> hydro_end_force on
// the h_dt sum of one particle.
__device__ __forceinline__ float end_force_hdt(float hdt, float h) {
#pragma clang fp contract(off)
  return hdt * (h * kDimInv);
}

}  // namespace sphl
