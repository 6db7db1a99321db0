// Pointwise and short-stencil dispatches whose workgroups may also run inside
// a batch (te_batch_part): the body takes its arguments and its workgroup, and
// the kernel of each dispatch passes its launch's own.  One thread per point
// (TE_TID3_OF), or runs of words where the launch is flat (te_flat).
#pragma once
#include "te_device.hpp"

namespace te {

// rayleigh_damping.wgsl:111-164
TE_DEV void rayleigh_damping_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz;
  if (i > g.nx || j > g.ny || k > g.nz) return;
  const float *u = fq(a.q[1]), *v = fq(a.q[2]), *w = fq(a.q[3]), *th = fq(a.q[4]), *u0 = fq(a.q[5]),
              *v0 = fq(a.q[6]), *tauh = fq(a.q[7]), *tauf = fq(a.q[8]), *hdx = fq(a.q[14]),
              *hdy = fq(a.q[15]), *avg = fq(a.q[18]), *th0 = fq(a.q[19]);
  float *uten = fq(a.q[10]), *vten = fq(a.q[11]), *wten = fq(a.q[12]), *thten = fq(a.q[13]);
  float rdalpha = ldf(a.q[9], 0);
  int lateral = ldi(a.q[16], 0), toAverage = ldi(a.q[17], 0);
  const int64_t c = g.idx(i, j, k);
  // the four fields loaded before the first store (the loads go out together)
  const float uc = u[c], vc = v[c], thc = th[c], wc = w[c];
  if (k < g.nz) {
    float t = tauh[k];
    float ur = toAverage != 0 ? avg[k] : u0[k];
    float vr = toAverage != 0 ? avg[g.nz + k] : v0[k];
    if (j < g.ny) uten[c] = ((-rdalpha) * t) * (uc - ur);
    if (i < g.nx) vten[c] = ((-rdalpha) * t) * (vc - vr);
    if (i < g.nx && j < g.ny) {
      float d = toAverage != 0 ? (th0[k] - avg[2 * g.nz + k]) + thc : thc;
      thten[c] = ((-rdalpha) * t) * d;
    }
  }
  if (i < g.nx && j < g.ny) {
    float tf = tauf[k];
    if (lateral != 0 && k < g.nz) tf = mx(mx(tf, hdx[i]), hdy[j]);
    wten[c] = ((-rdalpha) * tf) * wc;
  }
}

// turb_rho_faces.wgsl:111-151
TE_DEV void turb_rho_faces_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx - 2, j = gy - 2, k = gz;
  if (i > g.nx + 1 || j > g.ny + 1 || k > g.nz) return;
  const float *rho = fq(a.q[1]), *c1 = fq(a.q[2]), *c2 = fq(a.q[3]);
  float *rr = fq(a.q[4]), *rf = fq(a.q[5]);
  const uint32_t *os = a.q[6], *ot = a.q[7];
  const int64_t sk = g.sk(), c = g.idx(i, j, k);
  // rf formed before either store (the loads go out together)
  float r;
  if (k == 0) {
    r = fma_(ldf(os, 0), rho[c], ldf(os, 1) * rho[c + sk]);
    if (g.nz >= 3) r = fma_(ldf(os, 2), rho[c + 2 * sk], r);
  } else if (k == g.nz) {
    r = fma_(ldf(ot, 0), rho[c - sk], ldf(ot, 1) * rho[c - 2 * sk]);
    if (g.nz >= 3) r = fma_(ldf(ot, 2), rho[c - 3 * sk], r);
  } else {
    r = fma_(c1[k], rho[c - sk], c2[k] * rho[c]);
  }
  if (k < g.nz) rr[c] = 1.0f / rho[c];
  rf[c] = r;
}

// turb_def_centers.wgsl:139-168
TE_DEV void turb_def_centers_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx - 1, j = gy - 1, k = gz;
  if (i > g.nx + 1 || j > g.ny + 1 || k >= g.nz) return;
  const float *u = fq(a.q[1]), *v = fq(a.q[2]), *w = fq(a.q[3]), *rho = fq(a.q[4]), *mh = fq(a.q[5]),
              *hm = fq(a.q[30]);
  const int64_t sj = g.sJ, sk = g.sk(), c = g.idx(i, j, k);
  // every value formed before the first store (the loads go out together)
  const float r0 = rho[c];
  const float s11 = ((r0 * (u[c + 1] - u[c])) * g.rdx) * hm_uh(hm, g, i);
  const float s22 = ((r0 * (v[c + sj] - v[c])) * g.rdy) * hm_vh(hm, g, j);
  const float s33 = ((r0 * (w[c + sk] - w[c])) * g.rdz) * mh[k];
  const float rcorner = 0.25f * ((rho[c - 1 - sj] + r0) + (rho[c - 1] + rho[c - sj]));
  const float s12 =
      (0.5f * fma_((u[c] - u[c - sj]) * g.rdy, hm_vf(hm, g, j), ((v[c] - v[c - 1]) * g.rdx) * hm_uf(hm, g, i))) * rcorner;
  fq(a.q[6])[c] = s11;
  fq(a.q[7])[c] = s22;
  fq(a.q[8])[c] = s33;
  fq(a.q[9])[c] = s12;
}

// turb_def_faces.wgsl:125-151
TE_DEV void turb_def_faces_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz + 1;
  if (i > g.nx + 1 || j > g.ny + 1 || k > g.nz - 1) return;
  const float *u = fq(a.q[1]), *v = fq(a.q[2]), *w = fq(a.q[3]), *rf = fq(a.q[4]), *mf = fq(a.q[5]),
              *hm = fq(a.q[30]);
  const int64_t sj = g.sJ, sk = g.sk(), c = g.idx(i, j, k);
  float mfu = 0.5f * (mf[k] + mf[k]);
  float mfv = 0.5f * (mf[k] + mf[k]);
  // both values formed before the first store
  const float s13 =
      ((0.5f * fma_((w[c] - w[c - 1]) * g.rdx, hm_uf(hm, g, i), ((u[c] - u[c - sk]) * g.rdz) * mfu)) * 0.5f) * (rf[c - 1] + rf[c]);
  const float s23 =
      ((0.5f * fma_((w[c] - w[c - sj]) * g.rdy, hm_vf(hm, g, j), ((v[c] - v[c - sk]) * g.rdz) * mfv)) * 0.5f) * (rf[c - sj] + rf[c]);
  fq(a.q[6])[c] = s13;
  fq(a.q[7])[c] = s23;
}

// turb_def_assemble.wgsl:111-149
TE_DEV void turb_def_assemble_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz + 1;
  if (i >= g.nx || j >= g.ny || k > g.nz - 1) return;
  const float *s11 = fq(a.q[1]), *s22 = fq(a.q[2]), *s33 = fq(a.q[3]), *s12 = fq(a.q[4]),
              *s13 = fq(a.q[5]), *s23 = fq(a.q[6]), *c1 = fq(a.q[7]), *c2 = fq(a.q[8]), *rf = fq(a.q[9]);
  const int64_t sj = g.sJ, sk = g.sk(), c = g.idx(i, j, k);
  float A = c1[k], B = c2[k];
  float t11 = fma_(A * s11[c - sk], s11[c - sk], (B * s11[c]) * s11[c]);
  float t22 = fma_(A * s22[c - sk], s22[c - sk], (B * s22[c]) * s22[c]);
  float t33 = fma_(A * s33[c - sk], s33[c - sk], (B * s33[c]) * s33[c]);
  auto sq2 = [&](int64_t p, int64_t q) { return fma_(s12[p], s12[p], s12[q] * s12[q]); };
  float lo = sq2(c - sk, c + 1 + sj - sk) + sq2(c + sj - sk, c + 1 - sk);
  float hi = sq2(c, c + 1 + sj) + sq2(c + sj, c + 1);
  float t12 = 0.25f * fma_(A, lo, B * hi);
  float t13 = 0.5f * fma_(s13[c], s13[c], s13[c + 1] * s13[c + 1]);
  float t23 = 0.5f * fma_(s23[c], s23[c], s23[c + sj] * s23[c + sj]);
  float rrf = 1.0f / (rf[c] * rf[c]);
  fq(a.q[10])[c] = (4.0f * (t13 + t23)) * rrf;
  fq(a.q[11])[c] = fma_(2.0f, (t11 + t22) + t33, 4.0f * t12) * rrf;
}

// saturation mixing ratios over liquid / ice (turb_nm.wgsl:204-230)
TE_DEV float mp_rslf(float p, float t) {
  float esl = 611.2f * fast_exp((17.67f * (t - 273.15f)) / (t - 29.65f));
  esl = mn(esl, p * 0.5f);
  return ((RD / RV) * esl) / (p - esl);
}
TE_DEV float mp_rsif(float p, float t) {
  float esi = 611.2f * fast_exp((21.874557f * (t - 273.15f)) / (t - 7.66f));
  esi = mn(esi, p * 0.5f);
  return ((RD / RV) * esi) / (p - esi);
}

// turb_nm.wgsl:236-355 (moist squared buoyancy frequency)
TE_DEV void turb_nm_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz + 1;
  if (i >= g.nx || j >= g.ny || k > g.nz - 1) return;
  const float *thP = fq(a.q[1]), *ppP = fq(a.q[2]), *th0 = fq(a.q[3]), *pi0 = fq(a.q[4]),
              *prs = fq(a.q[5]), *qv = fq(a.q[6]), *qc = fq(a.q[7]), *qr = fq(a.q[8]), *qi = fq(a.q[9]),
              *qs = fq(a.q[10]), *qg = fq(a.q[11]), *c1 = fq(a.q[12]), *c2 = fq(a.q[13]), *mf = fq(a.q[14]);
  float *nm = fq(a.q[15]), *sat = fq(a.q[17]);
  int moist = ldi(a.q[16], 0), wantSat = ldi(a.q[18], 0);
  const int64_t sk = g.sk(), c = g.idx(i, j, k);
  const float nmsat = 1e-10f, eps = RD / RV, reps = RV / RD, gAcc = 9.81f;
  const float LV1 = 3134708.0f, LV2 = 2.32e+03f, LS1 = 2898463.5f, LS2 = 236.0f;
  float thA = th0[k - 1] + thP[c - sk];
  float thB = th0[k] + thP[c];
  if (moist == 0) {
    if (wantSat != 0) sat[c] = 0.0f;
    nm[c] = ((fast_log(thB / thA) * gAcc) * g.rdz) * mf[k];
    return;
  }
  float piA = pi0[k - 1] + ppP[c - sk], piB = pi0[k] + ppP[c];
  float tA = thA * piA, tB = thB * piB;
  float qtA = ((((qv[c - sk] + qc[c - sk]) + qr[c - sk]) + qi[c - sk]) + qs[c - sk]) + qg[c - sk];
  float qtB = ((((qv[c] + qc[c]) + qr[c]) + qi[c]) + qs[c]) + qg[c];
  float qciA = (qv[c - sk] + qc[c - sk]) + qi[c - sk];
  float qciB = (qv[c] + qc[c]) + qi[c];
  float thvA = (thA * fma_(reps, qv[c - sk], 1.0f)) / (1.0f + qtA);
  float thvB = (thB * fma_(reps, qv[c], 1.0f)) / (1.0f + qtB);
  float rmf = g.rdz * mf[k];
  float A = c1[k], B = c2[k];
  float pavg = fma_(A, prs[c - sk], B * prs[c]);
  float tavg = fma_(A, tA, B * tB);
  float qtavg = fma_(A, qtA, B * qtB);
  float qciavg = fma_(A, qciA, B * qciB);
  // The three temperature ranges only choose lam's operands (liquid, ice, or
  // both blended by ff); lam and the logarithms it needs are evaluated once,
  // below, for the saturated points alone.
  bool satd = false, blend = false;
  float qvs1 = 0.0f, lh1 = 0.0f, drdt1 = 0.0f, qvs2 = 0.0f, lh2 = 0.0f, drdt2 = 0.0f, cpml = 0.0f, ff = 0.0f;
  if (tavg >= 273.15f) {
    float qvs = mp_rslf(pavg, tavg);
    float ql = mx(qciavg - qvs, 0.0f);
    if (ql > nmsat) {
      satd = true;
      float qvl = mx(qciavg - ql, 0.0f);
      cpml = fma_(CPL, ql, fma_(CPV, qvl, CP));
      qvs1 = qvs;
      lh1 = fma_(-LV2, tavg, LV1);
      drdt1 = ((17.67f * (273.15f - 29.65f)) * qvs) / ((tavg - 29.65f) * (tavg - 29.65f));
    }
  } else if (tavg <= 233.15f) {
    float qvs = mp_rsif(pavg, tavg);
    float qice = mx(qciavg - qvs, 0.0f);
    if (qice > nmsat) {
      satd = true;
      float qvl = mx(qciavg - qice, 0.0f);
      cpml = fma_(CPI, qice, fma_(CPV, qvl, CP));
      qvs1 = qvs;
      lh1 = fma_(-LS2, tavg, LS1);
      drdt1 = ((21.874557f * (273.15f - 7.66f)) * qvs) / ((tavg - 7.66f) * (tavg - 7.66f));
    }
  } else {
    ff = (tavg - 233.15f) / (273.15f - 233.15f);
    float qvsl = mp_rslf(pavg, tavg), qvsi = mp_rsif(pavg, tavg);
    float qvs = fma_(ff, qvsl, (1.0f - ff) * qvsi);
    float qice = mx(0.0f, (1.0f - ff) * (qciavg - qvs));
    float ql = mx(0.0f, ff * (qciavg - qvs));
    if (ql + qice > nmsat) {
      satd = blend = true;
      float qvl = mx(0.0f, (qciavg - ql) - qice);
      cpml = fma_(CPI, qice, fma_(CPL, ql, fma_(CPV, qvl, CP)));
      qvs1 = qvsl;
      lh1 = fma_(-LV2, tavg, LV1);
      drdt1 = ((17.67f * (273.15f - 29.65f)) * qvsl) / ((tavg - 29.65f) * (tavg - 29.65f));
      qvs2 = qvsi;
      lh2 = fma_(-LS2, tavg, LS1);
      drdt2 = ((21.874557f * (273.15f - 7.66f)) * qvsi) / ((tavg - 7.66f) * (tavg - 7.66f));
    }
  }
  if (wantSat != 0) sat[c] = satd ? 1.0f : 0.0f;
  float out;
  if (satd) {
    const float dlnT = fast_log(tB / tA) * rmf;
    const float dlnQt = fast_log((1.0f + qtB) / (1.0f + qtA)) * rmf;
    auto lam = [&](float qvs, float lh, float drdt) {
      float gamma = ((gAcc * (1.0f + qtavg)) * (1.0f + (lh * qvs) / (RD * tavg))) / fma_(lh, drdt, cpml);
      return gAcc * fma_(dlnT + gamma / tavg, 1.0f + (tavg * drdt) / (eps + qvs), -dlnQt);
    };
    const float n1 = lam(qvs1, lh1, drdt1);
    out = blend ? fma_(ff, n1, (1.0f - ff) * lam(qvs2, lh2, drdt2)) : n1;
  } else {
    out = (gAcc * fast_log(thvB / thvA)) * rmf;
  }
  nm[c] = out;
}

// turb_km_kh.wgsl:125-187; IMG: then the halo fill of kmh, kmv, khh, khv on
// a periodic domain (nx, ny >= 4; timestep.js:1593 haloFill): each cell
// writes its periodic images, the cells of levels 1 and nz-1 also the images
// of levels 0 and nz (not written here; no thread of the launch reads K).
template <bool IMG>
__device__ __forceinline__ void turb_km_kh_at(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  const Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz + 1;
  if (i >= g.nx || j >= g.ny || k > g.nz - 1) return;
  const float *tkea = fq(a.q[1]), *nm = fq(a.q[2]), *mf = fq(a.q[3]), *hm = fq(a.q[30]);
  float *kmh = fq(a.q[4]), *kmv = fq(a.q[5]), *khh = fq(a.q[6]), *khv = fq(a.q[7]), *lenscl = fq(a.q[8]),
        *dissten = fq(a.q[9]);
  float kmScale = ldf(a.q[10], 0), kmFixed = ldf(a.q[11], 0), turbfac = ldf(a.q[12], 0);
  const int64_t c = g.idx(i, j, k);
  const float c_m = 0.1f, c_l = 0.8165f, ri_c = 0.25f, tke_min = 1e-10f, nm_min = 1e-06f, small_len_frac = 0.001f;
  float cmz = mx(0.001f, turbfac * c_m);
  float ce1z = ((cmz * c_l) * c_l) * (1.0f / ri_c - 1.0f);
  float ce2z = mx(0.0f, fma_(cmz * 3.1415927f, 3.1415927f, -ce1z));
  float dzk = (1.0f / g.rdz) / mf[k];
  float grdscl = fast_pow((((1.0f / g.rdx) / hm_uh(hm, g, i)) * ((1.0f / g.rdy) / hm_vh(hm, g, j))) * dzk, 0.33333334f);
  float rgrdscl = 1.0f / grdscl;
  // the cell's operands, loaded once before the stores below
  const float tkc = tkea[c], nmc = nm[c], dissc = dissten[c];
  float tk, len;
  if (tkc <= tke_min) {
    tk = tke_min;
    len = small_len_frac * grdscl;
  } else {
    tk = tkc;
    len = grdscl;
    if (nmc > nm_min) {
      len = c_l * sqrtf(tk / nmc);
      len = mn(len, grdscl);
      len = mx(len, small_len_frac * grdscl);
    }
  }
  lenscl[c] = len;
  dissten[c] = dissc + ((fma_(ce2z * len, rgrdscl, ce1z) * tk) * sqrtf(tk)) / len;
  float km = kmFixed > 0.0f ? kmFixed : ((cmz * sqrtf(tk)) * len) * kmScale;
  kmh[c] = km;
  kmv[c] = km;
  float prinv = 3.0f;
  if (nmc > nm_min) prinv = mn(fma_(2.0f * len, rgrdscl, 1.0f), 3.0f);
  khh[c] = km * prinv;
  khv[c] = km * prinv;
  if (IMG) {
    float* F[4] = {kmh, kmv, khh, khv};
    const float v[4] = {km, km, km * prinv, km * prinv};
    const int64_t sk = g.sk(), e = k == 1 ? -sk : (k == g.nz - 1 ? sk : 0);
    const int64_t e2 = k == 1 && k == g.nz - 1 ? sk : 0;  // nz = 2: level 1 is next to both
    float ev[4], ev2[4];
    for (int q = 0; q < 4; ++q) {
      ev[q] = e != 0 ? F[q][c + e] : 0.0f;
      ev2[q] = e2 != 0 ? F[q][c + e2] : 0.0f;
    }
    for (int q = 0; q < 4; ++q) {
      halo_from<false>(g, {false, false}, F[q], i, j, c, v[q], {});
      if (e != 0) halo_from<false>(g, {false, false}, F[q], i, j, c + e, ev[q], {});
      if (e2 != 0) halo_from<false>(g, {false, false}, F[q], i, j, c + e2, ev2[q], {});
    }
  }
}

// turb_dissipative_heating.wgsl:139-194
TE_DEV void turb_dissipative_heating_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz;
  if (i >= g.nx || j >= g.ny || k >= g.nz) return;
  const float *dissten = fq(a.q[1]), *pi0 = fq(a.q[2]), *ppi = fq(a.q[3]), *qv = fq(a.q[4]),
              *qc = fq(a.q[5]), *qr = fq(a.q[6]), *qi = fq(a.q[7]), *qs = fq(a.q[8]), *qg = fq(a.q[9]),
              *sfc = fq(a.q[12]);
  float* thten = fq(a.q[10]);
  const uint32_t* op = a.q[11];
  int moist = ldi(op, 0), bbc3 = ldi(op, 1), zntField = ldi(op, 4);
  float znt = ldf(op, 2), dz1 = ldf(op, 3);
  const int64_t sk = g.sk(), c = g.idx(i, j, k);
  const float cv = CP - RD, cvv = CPV - RV, cpdcv = CP / (CP - RD);
  float epsd;
  if (k == 0 && bbc3 != 0) {
    float ust = sfc[3 * sk + g.idx(i, j, 0)];
    float z0 = zntField != 0 ? sfc[4 * sk + g.idx(i, j, 0)] : znt;
    epsd = (((ust * ust) * ust) * fast_log((dz1 + z0) / z0)) / (0.4f * dz1);
  } else {
    epsd = 0.5f * (dissten[c] + dissten[c + sk]);
  }
  float pi = pi0[k] + ppi[c];
  float dheat;
  if (moist != 0) {
    float cvm = fma_(2106.0f, (qi[c] + qs[c]) + qg[c], fma_(4.19e+03f, qc[c] + qr[c], fma_(cvv, qv[c], cv)));
    dheat = epsd / ((cpdcv * cvm) * pi);
  } else {
    dheat = epsd / (CP * pi);
  }
  thten[c] = thten[c] + dheat;
}

// turb_gettau.wgsl:111-143
TE_DEV void turb_gettau_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx - 1, j = gy - 1, k = gz;
  if (i > g.nx || j > g.ny || k >= g.nz) return;
  const float *kmh = fq(a.q[1]), *kmv = fq(a.q[2]);
  float *t11 = fq(a.q[3]), *t22 = fq(a.q[4]), *t33 = fq(a.q[5]), *t12 = fq(a.q[6]), *t13 = fq(a.q[7]),
        *t23 = fq(a.q[8]);
  const int64_t sj = g.sJ, sk = g.sk(), c = g.idx(i, j, k);
  // every operand loaded before the first store (the loads go out together;
  // t13 / t23 and kmv at the column's first level are read but not used)
  const float tem = kmh[c] + kmh[c + sk];
  const float q = ((kmh[c - 1 - sj] + kmh[c]) + (kmh[c - 1] + kmh[c - sj])) +
                  ((kmh[c - 1 - sj + sk] + kmh[c + sk]) + (kmh[c - 1 + sk] + kmh[c - sj + sk]));
  const float a11 = t11[c], a22 = t22[c], a33 = t33[c], a12 = t12[c], a13 = t13[c], a23 = t23[c];
  const float kv = kmv[c], kvx = kmv[c - 1], kvy = kmv[c - sj];
  t11[c] = a11 * tem;
  t22[c] = a22 * tem;
  t33[c] = a33 * tem;
  t12[c] = a12 * (0.25f * q);
  if (k >= 1 && k <= g.nz - 1 && i >= 0 && j >= 0) {
    t13[c] = a13 * (kvx + kv);
    t23[c] = a23 * (kvy + kv);
  }
}

// tke_sources.wgsl:111-129
TE_DEV void tke_sources_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz + 1;
  if (i >= g.nx || j >= g.ny || k > g.nz - 1) return;
  const int64_t c = g.idx(i, j, k);
  const float *khv = fq(a.q[1]), *nm = fq(a.q[2]), *dissten = fq(a.q[3]), *epst = fq(a.q[4]);
  fq(a.q[5])[c] = fma_(-khv[c], nm[c], -dissten[c]) + epst[c];
}

// turb_scalar_flux_h.wgsl:125-148
TE_DEV void turb_scalar_flux_h_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz;
  if (i > g.nx || j > g.ny || k >= g.nz) return;
  const float *s = fq(a.q[1]), *rho = fq(a.q[2]), *khh = fq(a.q[3]), *hm = fq(a.q[30]);
  float leNum = ldf(a.q[4], 0);
  const int64_t sj = g.sJ, sk = g.sk(), c = g.idx(i, j, k);
  // both fluxes formed before the first store (the loads go out together)
  const float fx = (((((-0.125f * (rho[c] + rho[c - 1])) * leNum) * ((khh[c] + khh[c - 1]) + (khh[c + sk] + khh[c - 1 + sk]))) *
                     (s[c] - s[c - 1])) * g.rdx) * hm_uf(hm, g, i);
  const float fy = (((((-0.125f * (rho[c] + rho[c - sj])) * leNum) * ((khh[c] + khh[c - sj]) + (khh[c + sk] + khh[c - sj + sk]))) *
                     (s[c] - s[c - sj])) * g.rdy) * hm_vf(hm, g, j);
  fq(a.q[5])[c] = fx;
  fq(a.q[6])[c] = fy;
}

// tke_flux_h.wgsl:125-146
TE_DEV void tke_flux_h_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx, j = gy, k = gz + 1;
  if (i > g.nx || j > g.ny || k > g.nz - 1) return;
  const float *t = fq(a.q[1]), *rf = fq(a.q[2]), *kmh = fq(a.q[3]), *hm = fq(a.q[30]);
  const int64_t sj = g.sJ, c = g.idx(i, j, k);
  // both fluxes formed before the first store
  const float fx =
      (((((-0.25f * (rf[c] + rf[c - 1])) * 2.0f) * (kmh[c] + kmh[c - 1])) * (t[c] - t[c - 1])) * g.rdx) * hm_uf(hm, g, i);
  const float fy =
      (((((-0.25f * (rf[c] + rf[c - sj])) * 2.0f) * (kmh[c] + kmh[c - sj])) * (t[c] - t[c - sj])) * g.rdy) * hm_vf(hm, g, j);
  fq(a.q[4])[c] = fx;
  fq(a.q[5])[c] = fy;
}

// update_diagnostics_moist.wgsl:128-184
TE_DEV void update_diagnostics_moist_body(uint32_t* M, const KArg& a, const Blk& blk) {
  {
    const Dims g = dims(a.q[0], 0);
    if (te_flat_levels(a, blk, (uint32_t)(g.sJ * g.sK), [&](uint32_t w, int width, int k) {
          if (k >= g.nz) return;
          const float reps = RV / RD, repsm1 = reps - 1.0f;
          const float t0 = fq(a.q[3])[k], p0 = fq(a.q[4])[k], qv0k = fq(a.q[5])[k], qc0k = fq(a.q[6])[k],
                      qi0k = fq(a.q[7])[k], rt0 = fq(a.q[8])[k];
          const F4 thP = ld4(a.q[1], w, width), ppP = ld4(a.q[2], w, width), qv = ld4(a.q[9], w, width),
                   qc = ld4(a.q[10], w, width), qr = ld4(a.q[11], w, width), qi = ld4(a.q[12], w, width),
                   qs = ld4(a.q[13], w, width), qg = ld4(a.q[14], w, width);
          F4 thv, ppterm, piadv, thterm, buoy;
          for (int e = 0; e < width; ++e) {
            const float qvv = mx(qv.v[e], 0.0f);
            const float liq = qc.v[e] + qr.v[e];
            const float ice = (qi.v[e] + qs.v[e]) + qg.v[e];
            const float qli = mx(0.0f, liq + ice);
            const float cpli = fma_(CPL, mx(0.0f, liq), CPI * mx(0.0f, ice));
            const float th = t0 + thP.v[e];
            const float pi = p0 + ppP.v[e];
            const float cpm = fma_(CPV, qvv, CP) + cpli;
            const float cvm = 1.0f / (fma_(CVV, qvv, CV) + cpli);
            thv.v[e] = (th * fma_(reps, qvv, 1.0f)) / ((1.0f + qvv) + qli);
            piadv.v[e] = pi;
            ppterm.v[e] = ((pi * ROVCP) * cpm) * cvm;
            thterm.v[e] = (th * fma_(-ROVCP, cpm, fma_(RV, qvv, RD))) * cvm;
            buoy.v[e] = GRAV * (fma_(thP.v[e], rt0, repsm1 * (qvv - qv0k)) - ((qli - qc0k) - qi0k));
          }
          st4(a.q[15], w, width, thv);
          st4(a.q[16], w, width, ppterm);
          st4(a.q[17], w, width, piadv);
          st4(a.q[18], w, width, thterm);
          st4(a.q[19], w, width, buoy);
        }))
      return;
  }
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k >= g.nz) return;
  const float *thP = fq(a.q[1]), *ppP = fq(a.q[2]), *th0 = fq(a.q[3]), *pi0 = fq(a.q[4]),
              *qv0 = fq(a.q[5]), *qc0 = fq(a.q[6]), *qi0 = fq(a.q[7]), *rth0 = fq(a.q[8]),
              *qv = fq(a.q[9]), *qc = fq(a.q[10]), *qr = fq(a.q[11]), *qi = fq(a.q[12]),
              *qs = fq(a.q[13]), *qg = fq(a.q[14]);
  float *thv = fq(a.q[15]), *ppterm = fq(a.q[16]), *piadv = fq(a.q[17]), *thterm = fq(a.q[18]),
        *buoy = fq(a.q[19]);
  int64_t c = g.idx(i, j, k);
  const float reps = RV / RD, repsm1 = reps - 1.0f;
  float qvv = mx(qv[c], 0.0f);
  float liq = qc[c] + qr[c];
  float ice = (qi[c] + qs[c]) + qg[c];
  float qli = mx(0.0f, liq + ice);
  float cpli = fma_(CPL, mx(0.0f, liq), CPI * mx(0.0f, ice));
  float th = th0[k] + thP[c];
  float pi = pi0[k] + ppP[c];
  float cpm = fma_(CPV, qvv, CP) + cpli;
  float cvm = 1.0f / (fma_(CVV, qvv, CV) + cpli);
  thv[c] = (th * fma_(reps, qvv, 1.0f)) / ((1.0f + qvv) + qli);
  piadv[c] = pi;
  ppterm[c] = ((pi * ROVCP) * cpm) * cvm;
  thterm[c] = (th * fma_(-ROVCP, cpm, fma_(RV, qvv, RD))) * cvm;
  buoy[c] = GRAV * (fma_(thP[c], rth0[k], repsm1 * (qvv - qv0[k])) - ((qli - qc0[k]) - qi0[k]));
}

// update_diagnostics.wgsl:114-144 (dry)
TE_DEV void update_diagnostics_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k >= g.nz) return;
  const float *thP = fq(a.q[1]), *ppP = fq(a.q[2]), *th0 = fq(a.q[3]), *pi0 = fq(a.q[4]),
              *rth0 = fq(a.q[8]);
  float *thv = fq(a.q[5]), *ppterm = fq(a.q[6]), *piadv = fq(a.q[7]), *buoy = fq(a.q[9]);
  const float rddcv = RD / (CP - RD);
  int64_t c = g.idx(i, j, k);
  float pi = pi0[k] + ppP[c];
  thv[c] = th0[k] + thP[c];
  piadv[c] = pi;
  ppterm[c] = pi * rddcv;
  buoy[c] = (GRAV * thP[c]) * rth0[k];
}

// stage_tendency_reset.wgsl:110-129
TE_DEV void stage_tendency_reset_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  int64_t c = g.idx(i, j, k);
  fq(a.q[1])[c] = 0.0f;
  fq(a.q[2])[c] = 0.0f;
  fq(a.q[3])[c] = 0.0f;
}

// stage_state_reset.wgsl:110-138
TE_DEV void stage_state_reset_body(uint32_t* M, const KArg& a, const Blk& blk) {
  if (te_flat(a, blk, [&](uint32_t w, int width) {
        const int src[5] = {1, 2, 3, 4, 10};
        for (int q = 0; q < 5; ++q) st4(a.q[5 + q], w, width, ld4(a.q[src[q]], w, width));
      }))
    return;
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  int64_t c = g.idx(i, j, k);
  // u <- u_a, v <- v_a, w <- w_a, pp3d <- ppi, ppd <- ppx
  const int src[5] = {1, 2, 3, 4, 10};
  for (int q = 0; q < 5; ++q) fq(a.q[5 + q])[c] = fq(a.q[src[q]])[c];
}

// massflux_from_state then div_massflux (div_massflux.wgsl:125-147) in one
// launch: each cell stores its mass fluxes and forms the divergence from its
// own and its i+1, j+1, k+1 neighbours' fluxes, each the product
// massflux_from_state stores there (so the same bits), instead of reading them
// back.  p: 1-8 as massflux_from_state's, 9 mh, 10 divx.  Grid: whole.
TE_DEV void massflux_div_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  const Dims g = dims(a.q[0], 0);
  const int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  const float *u = fq(a.q[1]), *v = fq(a.q[2]), *w = fq(a.q[3]), *rho0 = fq(a.q[4]), *rf0 = fq(a.q[5]),
              *mh = fq(a.q[9]), *hm = fq(a.q[30]);
  const int64_t sj = g.sJ, sk = g.sk(), c = g.idx(i, j, k);
  auto fw = [&](int kk, int64_t cc) { return (kk == 0 || kk == g.nz) ? 0.0f : rf0[kk] * w[cc]; };
  const bool div = i <= g.nx + 2 && j <= g.ny + 2 && k < g.nz;
  const float r = k < g.nz ? rho0[k] : 0.0f;
  const float uc = k < g.nz ? u[c] : 0.0f, vc = k < g.nz ? v[c] : 0.0f;
  const float up = div ? u[c + 1] : 0.0f, vp = div ? v[c + sj] : 0.0f;
  const float mw = fw(k, c), mwp = div ? fw(k + 1, c + sk) : 0.0f;
  const float mu = r * uc, mv = r * vc;
  // the divergence formed before the first store (its profile and metric
  // loads go out with the others)
  const float d = div ? fma_((mwp - mw) * g.rdz, mh[k],
                             fma_((r * up - mu) * g.rdx, hm_uh(hm, g, i), ((r * vp - mv) * g.rdy) * hm_vh(hm, g, j)))
                      : 0.0f;
  if (k < g.nz) {
    fq(a.q[6])[c] = mu;
    fq(a.q[7])[c] = mv;
  }
  fq(a.q[8])[c] = mw;
  if (div) fq(a.q[10])[c] = d;
}

// build_sadv.wgsl:111-127
TE_DEV void build_sadv_body(uint32_t* M, const KArg& a, const Blk& blk) {
  {
    const Dims g = dims(a.q[0], 0);
    if (te_flat_levels(a, blk, (uint32_t)(g.sJ * g.sK), [&](uint32_t w, int width, int k) {
          if (k >= g.nz) return;
          const float t0 = fq(a.q[1])[k] - 3e+02f;
          F4 s = ld4(a.q[2], w, width);
          for (int e = 0; e < width; ++e) s.v[e] = t0 + s.v[e];
          st4(a.q[3], w, width, s);
        }))
      return;
  }
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k >= g.nz) return;
  const float *th0 = fq(a.q[1]), *thP = fq(a.q[2]);
  int64_t c = g.idx(i, j, k);
  fq(a.q[3])[c] = (th0[k] - 3e+02f) + thP[c];
}

// ppx_finish, then the halo fill of ppx on a periodic domain (nx, ny >= 4;
// timestep.js:1593 haloFill): each cell writes its periodic images.
TE_DEV void ppx_finish_xy_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  const Dims g = dims(a.q[0], 0);
  if (gx >= g.nx || gy >= g.ny || gz >= g.nz) return;
  const float* pp = fq(a.q[1]);
  float* ppx = fq(a.q[2]);
  update_with_halo(g, open_sides(a, 3), ppx, gx, gy, gz, 0, [&](int64_t c) { return pp[c] + ppx[c]; });
}

// diabatic_rates.wgsl:111-137
TE_DEV void diabatic_rates_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  if (gx >= g.nx || gy >= g.ny || gz >= g.nz) return;
  float dt = ldf(a.q[1], 0);
  float rdt = 1.0f / dt;
  int64_t c = g.idx(gx, gy, gz);
  for (int q = 0; q < 4; ++q) {
    const float* s = fq(a.q[2 + q]);
    float* r = fq(a.q[6 + q]);
    r[c] = (s[c] - r[c]) * rdt;
  }
}

// pressure_tendency.wgsl:234-291
TE_DEV void pressure_tendency_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  if (gx >= g.nx || gy >= g.ny || gz >= g.nz) return;
  const float *th = fq(a.q[1]), *qv = fq(a.q[2]), *rho = fq(a.q[3]), *ppi = fq(a.q[4]),
              *thten = fq(a.q[5]), *qpten = fq(a.q[6]), *th0 = fq(a.q[7]), *pi0 = fq(a.q[8]),
              *qvt = fq(a.q[13]);
  float* ppten = fq(a.q[11]);
  float dt = ldf(a.q[9], 0);
  int hasDiabatic = ldi(a.q[10], 0), hasStepTend = ldi(a.q[12], 0), moist = ldi(a.q[14], 0);
  const int k = gz;
  int64_t c = g.idx(gx, gy, gz);
  const float rp00 = 1.0f / P00, rddcv = RD / (CP - RD);
  float tem = 0.0001f * 0.0001f;
  float tht = hasStepTend != 0 ? thten[c] : 0.0f;
  if (moist == 0) {
    float p = 0.0f;
    if (ab(dt * tht) > tem) {
      float thnew = fma_(dt, tht, th[c]);
      float pinew = fast_pow(((rho[c] * (th0[k] + thnew)) * RD) * rp00, rddcv) - pi0[k];
      p = (pinew - ppi[c]) / dt;
    }
    ppten[c] = p;
    return;
  }
  float qvten = qvt[c];
  // every operand loaded with the tendencies (one wait for memory), whether
  // or not the cell takes the update
  const float thc = th[c], qvc = qv[c], rhoc = rho[c], ppic = ppi[c], qp = hasDiabatic != 0 ? qpten[c] : 0.0f;
  float p = 0.0f;
  if (ab(dt * tht) > tem || ab(dt * qvten) > 1e-14f) {
    float thnew = fma_(dt, tht, thc);
    float qvnew = fma_(dt, qvten, qvc);
    float pinew = fast_pow(((rhoc * (th0[k] + thnew)) * fma_(RV, qvnew, RD)) * rp00, rddcv) - pi0[k];
    p = (pinew - ppic) / dt;
  }
  if (hasDiabatic != 0) p = p + qp;
  ppten[c] = p;
}

// update_rho_prs.wgsl:234-267
TE_DEV void update_rho_prs_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  if (gx >= g.nx || gy >= g.ny || gz >= g.nz) return;
  int moist = ldi(a.q[1], 0);
  const float *thP = fq(a.q[2]), *ppP = fq(a.q[3]), *th0 = fq(a.q[4]), *pi0 = fq(a.q[5]),
              *qv = fq(a.q[6]);
  float *prs = fq(a.q[7]), *rho = fq(a.q[8]);
  const int k = gz;
  int64_t c = g.idx(gx, gy, gz);
  const float cpdrd = CP / RD;
  float pi = pi0[k] + ppP[c];
  float th = th0[k] + thP[c];
  float p = P00 * fast_pow(pi, cpdrd);
  prs[c] = p;
  float rmix = moist != 0 ? fma_(mx(0.0f, qv[c]), RV, RD) : RD;
  rho[c] = p / ((th * pi) * rmix);
}

// The end of a moist step in one pass over its cells: diabatic_unapply
// (diabatic_unapply.wgsl:111-140), update_rho_prs, diabatic_rates
// (diabatic_rates.wgsl:111-137) and ppx_finish with ppx's halo fill, for a step
// that changes no state between them (no mass correction, no microphysics).
// All are pointwise: 20 words per cell instead of 36, and two launches fewer;
// a step of 192 x 192 x 80 went from 3020 to 2980 us, one of 64 x 64 x 40
// stayed at 372.
// p: 1 -> dt, 2-5 pp3d, th, qv, qc, 6-9 their tendencies, 10 th0, 11 pi0,
// 12 prs, 13 rho, 14 ppx, 15 -> open x, open y.
TE_DEV void diabatic_finish_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  const Dims g = dims(a.q[0], 0);
  const int i = gx, j = gy, k = gz;
  if (i >= g.nx || j >= g.ny || k >= g.nz) return;
  const float dt = ldf(a.q[1], 0), rdt = 1.0f / dt;
  const int64_t c = g.idx(i, j, k);
  const Sides open = open_sides(a, 15);
  float* ppx = fq(a.q[14]);
  HaloCell h;
  if (open.x || open.y) h = halo_cell<true>(g, open, ppx, i, j, k, 0, c);
  else h = halo_cell<false>(g, open, ppx, i, j, k, 0, c);
  const float x = ppx[c], th0 = fq(a.q[10])[k], pi0 = fq(a.q[11])[k];
  float s[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) s[q] = fma_(-dt, fq(a.q[6 + q])[c], fq(a.q[2 + q])[c]);
  const float pi = pi0 + s[0], th = th0 + s[1];
  const float p = P00 * fast_pow(pi, CP / RD);
  const float rmix = fma_(mx(0.0f, s[2]), RV, RD);
  const float rho = p / ((th * pi) * rmix);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    fq(a.q[2 + q])[c] = s[q];
    fq(a.q[6 + q])[c] = (s[q] - s[q]) * rdt;  // (not 0 where s is not finite)
  }
  fq(a.q[12])[c] = p;
  fq(a.q[13])[c] = rho;
  if (open.x || open.y) halo_put<true>(g, open, ppx, i, j, c, s[0] + x, h);
  else halo_put<false>(g, open, ppx, i, j, c, s[0] + x, h);
}

// tke_advance (levels 1 .. nz-1) then the halo fill of tke
// (tke_advance.wgsl:111-129, timestep.js:1593 haloFill); arguments as
// tke_advance's, 5 -> open x, open y.
TE_DEV void tke_advance_xy_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  const Dims g = dims(a.q[0], 0);
  const int i = gx, j = gy, k = gz + 1;
  if (i >= g.nx || j >= g.ny || k > g.nz - 1) return;
  const float *tkea = fq(a.q[1]), *tketen = fq(a.q[2]);
  const float dttmp = ldf(a.q[3], 0);
  update_with_halo(g, open_sides(a, 5), fq(a.q[4]), i, j, k, 1, [&](int64_t c) {
    const float v = fma_(dttmp, tketen[c], tkea[c]);
    return (v < 1e-10f) ? 0.0f : v;
  });
}

// turb_zero (turb_zero.wgsl, timestep.js:1070-1072) of up to 8 fields in one
// launch over the whole grid [strideJ, strideK, nz+1].  p[1..8] fields,
// p[9] -> field count.
TE_DEV void zero_fields_body(uint32_t* M, const KArg& a, const Blk& blk) {
  if (te_flat(a, blk, [&](uint32_t w, int width) {
        const int n = ldi(a.q[9], 0);
        F4 z;
        z.v[0] = z.v[1] = z.v[2] = z.v[3] = 0.0f;
        for (int q = 0; q < 8; ++q) {
          if (q >= n) break;
          st4(a.q[1 + q], w, width, z);
        }
      }))
    return;
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  if (gx >= g.sJ || gy >= g.sK || gz > g.nz) return;
  const int64_t c = gx + (int64_t)g.sJ * (gy + (int64_t)g.sK * gz);
  const int n = ldi(a.q[9], 0);
  for (int q = 0; q < 8; ++q) {
    if (q >= n) break;
    fq(a.q[1 + q])[c] = 0.0f;
  }
}

// stage_tendency_reset (stage_tendency_reset.wgsl:111-129) followed by
// turb_add_tendency of the three SGS / damping momentum tendencies:
// dst = fma(scale, src, 0), the bits of adding src*scale to the cleared field.
// p: 1-3 uten vten wten, 4-6 their sources, 7 -> scale.  Grid: whole.
TE_DEV void tendency_reset_add_body(uint32_t* M, const KArg& a, const Blk& blk) {
  if (te_flat(a, blk, [&](uint32_t w, int width) {
        const float sc = ldf(a.q[7], 0);
        for (int q = 0; q < 3; ++q) {
          F4 d = ld4(a.q[4 + q], w, width);
          for (int e = 0; e < width; ++e) d.v[e] = fma_(sc, d.v[e], 0.0f);
          st4(a.q[1 + q], w, width, d);
        }
      }))
    return;
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  const int64_t c = g.idx(i, j, k);
  const float scale = ldf(a.q[7], 0);
  for (int q = 0; q < 3; ++q) fq(a.q[1 + q])[c] = fma_(scale, fq(a.q[4 + q])[c], 0.0f);
}

// Up to 4 buffer copies of a.n[0] words each (the state swap of
// timestep.js:766-774): p[1..4] sources, p[5..8] destinations, p[9] -> count.
TE_DEV void copy_fields_body(uint32_t* M, const KArg& a, const Blk& blk) {
  if (te_flat(a, blk, [&](uint32_t w, int width) {
        const int n = ldi(a.q[9], 0);
        for (int f = 0; f < 4; ++f) {
          if (f >= n) break;
          st4(a.q[5 + f], w, width, ld4(a.q[1 + f], w, width));
        }
      }))
    return;
  const uint32_t q = (uint32_t)(blk.x * TE_BX) + (uint32_t)blk.tx;
  if (q >= a.n[0]) return;
  const int n = ldi(a.q[9], 0);
  for (int f = 0; f < 4; ++f) {
    if (f >= n) break;
    a.q[5 + f][q] = a.q[1 + f][q];
  }
}

// rk_update of a scalar (stagger 1) then its halo fill (rk_update.wgsl:111-132,
// timestep.js:1593 haloFill); arguments as rk_update's, 6 -> open x, open y.
TE_DEV void rk_update_xy_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  const Dims g = dims(a.q[0], 0);
  const int i = gx, j = gy, k = gz;
  if (i >= g.nx || j >= g.ny || k >= g.nz) return;
  const float *phiA = fq(a.q[2]), *tend = fq(a.q[3]);
  const float dttmp = ldf(a.q[5], 0);
  update_with_halo(g, open_sides(a, 6), fq(a.q[4]), i, j, k, 0, [&](int64_t c) { return fma_(dttmp, tend[c], phiA[c]); });
}

// turb_openbc_flux.wgsl:111-140
TE_DEV void turb_openbc_flux_body(uint32_t* M, const KArg& a, const Blk& blk) {
  TE_TID3_OF(blk)
  Dims g = dims(a.q[0], 0);
  const int n = gx, k = gy;
  if (k > g.nz) return;
  float *fx = fq(a.q[1]), *fy = fq(a.q[2]);
  int openx = ldi(a.q[3], 0), openy = ldi(a.q[3], 1);
  if (openx != 0 && n <= g.ny) {
    fx[g.idx(0, n, k)] = fx[g.idx(1, n, k)];
    fx[g.idx(g.nx, n, k)] = fx[g.idx(g.nx - 1, n, k)];
  }
  if (openy != 0 && n <= g.nx) {
    fy[g.idx(n, 0, k)] = fy[g.idx(n, 1, k)];
    fy[g.idx(n, g.ny, k)] = fy[g.idx(n, g.ny - 1, k)];
  }
}

}  // namespace te
