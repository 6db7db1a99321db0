// Step kernels, one per reference kernel: diagnostics, resets, mass fluxes,
// divergence, RK update, buoyancy, pressure tendency, end-of-step updates.
// Every kernel has the signature (M, KArg) so a recorded or encoded program can
// launch it by name; the thread mapping follows the reference dispatch grid.
#include "te_device.hpp"
#include "te_kernels.hpp"
#include "pointwise.hpp"

namespace te {

__global__ __launch_bounds__(256) void k_update_diagnostics_moist(uint32_t* M, KArg a) { update_diagnostics_moist_body(M, a, te_block(a)); }

__global__ __launch_bounds__(256) void k_update_diagnostics(uint32_t* M, KArg a) { update_diagnostics_body(M, a, te_block(a)); }

__global__ __launch_bounds__(256) void k_stage_tendency_reset(uint32_t* M, KArg a) { stage_tendency_reset_body(M, a, te_block(a)); }

__global__ __launch_bounds__(256) void k_stage_state_reset(uint32_t* M, KArg a) { stage_state_reset_body(M, a, te_block(a)); }

// massflux_from_state.wgsl:111-137
__global__ __launch_bounds__(256) void k_massflux_from_state(uint32_t* M, KArg a) {
  {
    const Dims g = dims(a.q[0], 0);
    if (te_flat_levels(a, te_block(a), (uint32_t)(g.sJ * g.sK), [&](uint32_t w, int width, int k) {
          if (k < g.nz) {
            const float r = fq(a.q[4])[k];
            F4 u = ld4(a.q[1], w, width), v = ld4(a.q[2], w, width);
            for (int e = 0; e < width; ++e) {
              u.v[e] = r * u.v[e];
              v.v[e] = r * v.v[e];
            }
            st4(a.q[6], w, width, u);
            st4(a.q[7], w, width, v);
          }
          F4 m = ld4(a.q[3], w, width);
          const bool edge = k == 0 || k == g.nz;
          const float rf = edge ? 0.0f : fq(a.q[5])[k];
          for (int e = 0; e < width; ++e) m.v[e] = edge ? 0.0f : rf * m.v[e];
          st4(a.q[8], w, width, m);
        }))
      return;
  }
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  const float *u = fq(a.q[1]), *v = fq(a.q[2]), *w = fq(a.q[3]), *rho0 = fq(a.q[4]), *rf0 = fq(a.q[5]);
  float *rru = fq(a.q[6]), *rrv = fq(a.q[7]), *rrw = fq(a.q[8]);
  int64_t c = g.idx(i, j, k);
  if (k < g.nz) {
    rru[c] = rho0[k] * u[c];
    rrv[c] = rho0[k] * v[c];
  }
  rrw[c] = (k == 0 || k == g.nz) ? 0.0f : rf0[k] * w[c];
}

__global__ __launch_bounds__(256) void k_massflux_div(uint32_t* M, KArg a) { massflux_div_body(M, a, te_block(a)); }

// After the stage's substeps: divergence3d of the mean velocities,
// velocity_to_massflux, div_massflux of the fluxes and build_sadv
// (timestep.js:2056-2075) in one launch.  The mean velocities are read from
// fields of their own (the last substep writes them there), so that no thread
// of the launch reads what another one writes.  10 words per cell instead of
// 16, one launch instead of four: 17.3 us became 6 at 64 x 64 x 40, 42 became
// 30 at 192 x 192 x 80.
// p: 1-3 mean u, v, w, 4 rho0, 5 rf0, 6-8 rru, rrv, rrw, 9 mh, 10 divx,
// 11 div3d (if bound), 12 th0, 13 th, 14 sadv, 30 metric.  Grid: whole.
__global__ __launch_bounds__(256) void k_mean_massflux(uint32_t* M, KArg a) {
  TE_TID3
  const Dims g = dims(a.q[0], 0);
  const int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  const float *u = fq(a.q[1]), *v = fq(a.q[2]), *w = fq(a.q[3]), *rho0 = fq(a.q[4]), *rf0 = fq(a.q[5]),
              *mh = fq(a.q[9]), *hm = fq(a.q[30]);
  const int64_t sj = g.sJ, sk = g.sk(), c = g.idx(i, j, k);
  const bool below = k < g.nz, div = i <= g.nx + 2 && j <= g.ny + 2 && below;
  const bool inner = a.p[11] != 0 && below && i >= 0 && i < g.nx && j >= 0 && j < g.ny;
  const float uc = u[c], vc = v[c], wc = w[c], th = below ? fq(a.q[13])[c] : 0.0f;
  const float up = div ? u[c + 1] : 0.0f, vp = div ? v[c + sj] : 0.0f, wp = div ? w[c + sk] : 0.0f;
  const float r = below ? rho0[k] : 1.0f, t0 = below ? fq(a.q[12])[k] - 3e+02f : 0.0f;
  auto fw = [&](int kk, float x) { return (kk == 0 || kk == g.nz) ? 0.0f : x * rf0[kk]; };
  const float mu = uc * r, mv = vc * r, mw = fw(k, wc), mwp = div ? fw(k + 1, wp) : 0.0f;
  const float uh = div ? hm_uh(hm, g, i) : 0.0f, vh = div ? hm_vh(hm, g, j) : 0.0f, mhk = div ? mh[k] : 0.0f;
  auto divergence = [&](float u0, float u1, float v0, float v1, float w0, float w1) {
    return fma_((w1 - w0) * g.rdz, mhk, fma_((u1 - u0) * g.rdx, uh, ((v1 - v0) * g.rdy) * vh));
  };
  const float dx = divergence(mu, up * r, mv, vp * r, mw, mwp), d3 = divergence(uc, up, vc, vp, wc, wp);
  fq(a.q[6])[c] = below ? mu : uc;  // level nz keeps the mean velocity
  fq(a.q[7])[c] = below ? mv : vc;
  fq(a.q[8])[c] = mw;
  if (div) fq(a.q[10])[c] = dx;
  if (inner) fq(a.q[11])[c] = (ab(d3) < 1e-30f) ? 0.0f : d3;
  if (below) fq(a.q[14])[c] = t0 + th;
}

// velocity_to_massflux.wgsl:111-134
__global__ __launch_bounds__(256) void k_velocity_to_massflux(uint32_t* M, KArg a) {
  {
    const Dims g = dims(a.q[0], 0);
    if (te_flat_levels(a, te_block(a), (uint32_t)(g.sJ * g.sK), [&](uint32_t w, int width, int k) {
          if (k < g.nz) {
            const float r = fq(a.q[1])[k];
            F4 u = ld4(a.q[3], w, width), v = ld4(a.q[4], w, width);
            for (int e = 0; e < width; ++e) {
              u.v[e] = u.v[e] * r;
              v.v[e] = v.v[e] * r;
            }
            st4(a.q[3], w, width, u);
            st4(a.q[4], w, width, v);
          }
          const bool edge = k == 0 || k == g.nz;
          F4 m = ld4(a.q[5], w, width);
          const float rf = edge ? 0.0f : fq(a.q[2])[k];
          for (int e = 0; e < width; ++e) m.v[e] = edge ? 0.0f : m.v[e] * rf;
          st4(a.q[5], w, width, m);
        }))
      return;
  }
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  const float *rho0 = fq(a.q[1]), *rf0 = fq(a.q[2]);
  float *rru = fq(a.q[3]), *rrv = fq(a.q[4]), *rrw = fq(a.q[5]);
  int64_t c = g.idx(i, j, k);
  if (k < g.nz) {
    rru[c] = rru[c] * rho0[k];
    rrv[c] = rrv[c] * rho0[k];
  }
  rrw[c] = (k == 0 || k == g.nz) ? 0.0f : rrw[c] * rf0[k];
}

// div_massflux.wgsl:125-147
__global__ __launch_bounds__(256) void k_div_massflux(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 2 || j > g.ny + 2 || k >= g.nz) return;
  const float *rru = fq(a.q[1]), *rrv = fq(a.q[2]), *rrw = fq(a.q[3]), *mh = fq(a.q[4]),
              *hm = fq(a.q[30]);
  float* divx = fq(a.q[5]);
  const int64_t sj = g.sJ, sk = g.sk(), c = g.idx(i, j, k);
  divx[c] = fma_((rrw[c + sk] - rrw[c]) * g.rdz, mh[k],
                 fma_((rru[c + 1] - rru[c]) * g.rdx, hm_uh(hm, g, i), ((rrv[c + sj] - rrv[c]) * g.rdy) * hm_vh(hm, g, j)));
}

// divergence3d.wgsl:125-147
__global__ __launch_bounds__(256) void k_divergence3d(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz;
  if (i >= g.nx || j >= g.ny || k >= g.nz) return;
  const float *u = fq(a.q[1]), *v = fq(a.q[2]), *w = fq(a.q[3]), *mh = fq(a.q[4]), *hm = fq(a.q[30]);
  float* dv = fq(a.q[5]);
  const int64_t sj = g.sJ, sk = g.sk(), c = g.idx(i, j, k);
  float d = fma_((w[c + sk] - w[c]) * g.rdz, mh[k],
                 fma_((u[c + 1] - u[c]) * g.rdx, hm_uh(hm, g, i), ((v[c + sj] - v[c]) * g.rdy) * hm_vh(hm, g, j)));
  dv[c] = (ab(d) < 1e-30f) ? 0.0f : d;
}

// buoyancy_apply.wgsl:111-129
__global__ __launch_bounds__(256) void k_buoyancy_apply(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz + 1;
  if (i >= g.nx || j >= g.ny || k > g.nz - 1) return;
  const float *buoy = fq(a.q[1]), *c1 = fq(a.q[2]), *c2 = fq(a.q[3]);
  float* wten = fq(a.q[4]);
  const int64_t sk = g.sk(), c = g.idx(i, j, k);
  wten[c] = wten[c] + fma_(c1[k], buoy[c - sk], c2[k] * buoy[c]);
}

// rk_update.wgsl:111-132
__global__ __launch_bounds__(256) void k_rk_update(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int stag = ldi(a.q[1], 0);
  int i = gx, j = gy, k = gz;
  int iMax = stag == 2 ? g.nx : g.nx - 1, jMax = stag == 3 ? g.ny : g.ny - 1, kLo = stag == 4 ? 1 : 0;
  if (i > iMax || j > jMax || k < kLo || k >= g.nz) return;
  const float *phiA = fq(a.q[2]), *tend = fq(a.q[3]);
  float* phi = fq(a.q[4]);
  float dttmp = ldf(a.q[5], 0);
  int64_t c = g.idx(i, j, k);
  phi[c] = fma_(dttmp, tend[c], phiA[c]);
}

__global__ __launch_bounds__(256) void k_build_sadv(uint32_t* M, KArg a) { build_sadv_body(M, a, te_block(a)); }

// apply_thterm.wgsl:111-127
__global__ __launch_bounds__(256) void k_apply_thterm(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  if (gx >= g.nx || gy >= g.ny || gz >= g.nz) return;
  const float *dv = fq(a.q[1]), *thterm = fq(a.q[2]);
  float* tend = fq(a.q[3]);
  int64_t c = g.idx(gx, gy, gz);
  tend[c] = fma_(-dv[c], thterm[c], tend[c]);
}

// turb_add_tendency.wgsl:111-127
__global__ __launch_bounds__(256) void k_turb_add_tendency(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  const float* src = fq(a.q[1]);
  float* dst = fq(a.q[2]);
  float scale = ldf(a.q[3], 0);
  int64_t c = g.idx(i, j, k);
  dst[c] = fma_(scale, src[c], dst[c]);
}

// turb_zero.wgsl:103-116
__global__ __launch_bounds__(256) void k_turb_zero(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  if (gx >= g.sJ || gy >= g.sK || gz > g.nz + 1) return;
  fq(a.q[1])[gx + (int64_t)g.sJ * (gy + (int64_t)g.sK * gz)] = 0.0f;
}

// tke_advance.wgsl:111-129
__global__ __launch_bounds__(256) void k_tke_advance(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz + 1;
  if (i >= g.nx || j >= g.ny || k > g.nz - 1) return;
  const float *tkea = fq(a.q[1]), *tketen = fq(a.q[2]);
  float dttmp = ldf(a.q[3], 0);
  int64_t c = g.idx(i, j, k);
  float v = fma_(dttmp, tketen[c], tkea[c]);
  fq(a.q[4])[c] = (v < 1e-10f) ? 0.0f : v;
}

// ppx_finish.wgsl:111-126
__global__ __launch_bounds__(256) void k_ppx_finish(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  if (gx >= g.nx || gy >= g.ny || gz >= g.nz) return;
  int64_t c = g.idx(gx, gy, gz);
  float* ppx = fq(a.q[2]);
  ppx[c] = fq(a.q[1])[c] + ppx[c];
}
__global__ __launch_bounds__(256) void k_ppx_finish_xy(uint32_t* M, KArg a) { ppx_finish_xy_body(M, a, te_block(a)); }

// diabatic_unapply.wgsl:111-140
__global__ __launch_bounds__(256) void k_diabatic_unapply(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  if (gx >= g.nx || gy >= g.ny || gz >= g.nz) return;
  float dt = ldf(a.q[1], 0);
  int64_t c = g.idx(gx, gy, gz);
  for (int q = 0; q < 4; ++q) {
    float* s = fq(a.q[2 + q]);
    float* r = fq(a.q[6 + q]);
    s[c] = fma_(-dt, r[c], s[c]);
    r[c] = s[c];
  }
}

__global__ __launch_bounds__(256) void k_diabatic_rates(uint32_t* M, KArg a) { diabatic_rates_body(M, a, te_block(a)); }

__global__ __launch_bounds__(256) void k_pressure_tendency(uint32_t* M, KArg a) { pressure_tendency_body(M, a, te_block(a)); }

__global__ __launch_bounds__(256) void k_update_rho_prs(uint32_t* M, KArg a) { update_rho_prs_body(M, a, te_block(a)); }

__global__ __launch_bounds__(256) void k_diabatic_finish(uint32_t* M, KArg a) { diabatic_finish_body(M, a, te_block(a)); }

// stability_max.wgsl:120-178 (adapt_dt = 1): max over the grid of the
// squared advective Courant number c2 = x^2 + y^2 + z^2 (x = (u_i + u_i+1)
// dt / (2 dx) uh, and alike) and of the squared diffusion number of kmh,
// khh, kmv at levels k >= 1, into two words: the bits of non-negative floats
// order like the floats, so an unsigned max of the bits is the float max
// and the result does not depend on the order of the workgroups.  Each
// workgroup reduces in LDS and adds one global atomic per word.
__global__ __launch_bounds__(256) void k_stability_max(uint32_t* M, KArg a) {
  __shared__ uint32_t red[2];
  const uint32_t t = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
  if (t == 0) {
    red[0] = 0u;
    red[1] = 0u;
  }
  __syncthreads();
  int gx, gy, gz;
  te_tid3(a, te_block(a), gx, gy, gz);
  const Dims g = dims(a.q[0], 0);
  float c2 = 0.0f, m = 0.0f;
  if (gx < (int)a.n[0] && gy < (int)a.n[1] && gz < (int)a.n[2] && gx < g.nx && gy < g.ny && gz < g.nz) {
    const uint32_t* P = a.q[1];
    const float dtdx = ldf(P, 0), dtdy = ldf(P, 1), dtdz = ldf(P, 2), ksdx = ldf(P, 3), ksdy = ldf(P, 4);
    const int twoD = ldi(P, 5), withKs = ldi(P, 6);
    const float *u = fq(a.q[2]), *v = fq(a.q[3]), *w = fq(a.q[4]), *mh = fq(a.q[5]), *hm = fq(a.q[30]);
    const int64_t c = g.idx(gx, gy, gz);
    const float uh = hm_uh(hm, g, gx), vh = hm_vh(hm, g, gy);
    const float x = ((u[c] + u[c + 1]) * dtdx) * uh;
    const float z = ((w[c] + w[c + g.sk()]) * dtdz) * mh[gz];
    if (twoD != 0) {
      c2 = fma_(x, x, z * z);
    } else {
      const float y = ((v[c] + v[c + g.sJ]) * dtdy) * vh;
      c2 = fma_(z, z, fma_(x, x, y * y));
    }
    if (withKs != 0 && gz >= 1) {
      const float K[3] = {fq(a.q[6])[c], fq(a.q[8])[c], fq(a.q[7])[c]};  // kmh, khh, kmv
      for (int n = 0; n < 3; ++n) {
        const float aa = ((K[n] * ksdx) * uh) * uh;
        float tt = aa;
        if (twoD == 0) {
          const float bb = ((K[n] * ksdy) * vh) * vh;
          tt = fma_(aa, aa, bb * bb);
        }
        m = mx(m, tt);
      }
    }
  }
  atomicMax(&red[0], __float_as_uint(c2));
  atomicMax(&red[1], __float_as_uint(m));
  __syncthreads();
  if (t == 0) {
    atomicMax(a.q[9], red[0]);
    atomicMax(a.q[9] + 1, red[1]);
  }
}

}  // namespace te
