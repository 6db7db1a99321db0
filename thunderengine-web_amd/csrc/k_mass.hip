// apmasscon dry-mass conservation at the end of the step: row, level and
// total sums in double-float (float pairs) in a fixed sequential order, so
// every launch reproduces the reference's bits; then the uniform pi'
// correction with prs and rho from the corrected state.
#include "te_device.hpp"
#include "te_kernels.hpp"

namespace te {

struct DFs {
  float x, y;
};
// f_df_add (mass_row_sums.wgsl:120-127)
TE_DEV void df_add(DFs& acc, float x) {
  float s = acc.x + x;
  float bb = s - acc.x;
  float err = (acc.x - (s - bb)) + (x - bb);
  acc.x = s;
  acc.y = acc.y + err;
}
// f_df_add_pair (mass_level_sums.wgsl:98-102)
TE_DEV void df_add_pair(DFs& acc, float vx, float vy) {
  df_add(acc, vx);
  acc.y = acc.y + vy;
}

// mass_row_sums.wgsl:134-170: per row (j, k) the sums over i, in order.  A
// workgroup takes MASS_ROWS rows: its threads form the rows' terms tile by tile
// with coalesced loads (the divisions too), and one lane per row and sum adds a
// tile from LDS in the reference's order.  One thread per row read every row at
// the row stride: 57 us at 120 x 120 x 40, now 10.
#define MASS_ROWS 16
#define MASS_TILE 64
__global__ __launch_bounds__(256) void k_mass_row_sums(uint32_t* M, KArg a) {
  __shared__ float term[2][MASS_ROWS][MASS_TILE + 1];
  const Dims g = dims(a.q[0], 0);
  const float *rho = fq(a.q[1]), *pi0 = fq(a.q[2]), *pp3d = fq(a.q[3]), *mh = fq(a.q[4]),
              *hm = fq(a.q[30]);
  const int id = (int)threadIdx.x, wave = id / 64, lane = id % 64;
  // rows numbered over the launch grid [ny, nz]
  const int nj = (int)a.n[0], rows = nj * (int)a.n[1];
  const int row0 = (int)blockIdx.x * MASS_ROWS;
  // summing lane: row `id % MASS_ROWS` of sum `id / MASS_ROWS`
  const int mine = row0 + id % MASS_ROWS, which = id / MASS_ROWS;
  DFs s{0.0f, 0.0f};
  for (int i0 = 0; i0 < g.nx; i0 += MASS_TILE) {
    const int i = i0 + lane;
#pragma unroll
    for (int q = 0; q < MASS_ROWS / 4; ++q) {
      const int r = q * 4 + wave, row = row0 + r;
      const int k = row / nj, j = row - k * nj;
      if (row >= rows || i >= g.nx || j >= g.ny || k >= g.nz) continue;
      const int64_t c = g.idx(i, j, k);
      const float rvh = 1.0f / hm_vh(hm, g, j), rmh = 1.0f / mh[k];
      term[0][r][lane] = ((rho[c] * (1.0f / hm_uh(hm, g, i))) * rvh) * rmh;
      term[1][r][lane] = pi0[k] + pp3d[c];
    }
    __syncthreads();
    if (which < 2 && mine < rows) {
      const int n = min(MASS_TILE, g.nx - i0);
      for (int t = 0; t < n; ++t) df_add(s, term[which][id % MASS_ROWS][t]);
    }
    __syncthreads();
  }
  const int k = mine / nj, j = mine - k * nj;
  if (which < 2 && mine < rows && j < g.ny && k < g.nz) {
    float* out = fq(a.q[5 + which]);
    const int64_t r = ((int64_t)k * g.sK + j) * 2;
    out[r] = s.x;
    out[r + 1] = s.y;
  }
}

// mass_level_sums.wgsl:118-146: per level the sums over its rows, in order.
// One wave per level: its lanes fetch 64 rows at a time, two of them add (34 us
// with one thread per level at 120 x 120 x 40, now 5).
__global__ __launch_bounds__(256) void k_mass_level_sums(uint32_t* M, KArg a) {
  __shared__ float part[2][64][2];
  const Dims g = dims(a.q[0], 0);
  const int k = (int)blockIdx.x, lane = (int)threadIdx.x;
  if (k >= g.nz) return;
  DFs s{0.0f, 0.0f};
  for (int j0 = 0; j0 < g.ny; j0 += 64) {
    const int j = j0 + lane;
    if (j < g.ny) {
      const int64_t r = ((int64_t)k * g.sK + j) * 2;
      for (int q = 0; q < 2; ++q) {
        const float* rows = fq(a.q[1 + q]);
        part[q][lane][0] = rows[r];
        part[q][lane][1] = rows[r + 1];
      }
    }
    __syncthreads();
    if (lane < 2) {
      const int n = min(64, g.ny - j0);
      for (int t = 0; t < n; ++t) df_add_pair(s, part[lane][t][0], part[lane][t][1]);
    }
    __syncthreads();
  }
  if (lane < 2) {
    float* lev = fq(a.q[3 + lane]);
    lev[k * 2] = s.x;
    lev[k * 2 + 1] = s.y;
  }
}

// mass_reference_init.wgsl:118-142: the reference dry mass, once (ref[2]).
__global__ __launch_bounds__(256) void k_mass_reference_init(uint32_t* M, KArg a) {
  TE_TID3
  if (gx != 0) return;
  Dims g = dims(a.q[0], 0);
  const float* lev1 = fq(a.q[1]);
  float* ref = fq(a.q[2]);
  if (ref[2] != 0.0f) return;
  DFs s{0.0f, 0.0f};
  for (int k = 0; k < g.nz; ++k) df_add_pair(s, lev1[k * 2], lev1[k * 2 + 1]);
  ref[0] = s.x;
  ref[1] = s.y;
  ref[2] = 1.0f;
}

// f_powm1 (mass_correction_apply.wgsl:121-128).  The |r| > 0.05 branch calls
// the WGSL pow builtin; the correctly rounded pow stands in for it.
TE_DEV float powm1(float r, float a) {
  if (ab(r) > 0.05f) return fast_pow(1.0f + r, a) - 1.0f;
  return r * fma_(r, fma_(a * (a - 1.0f), 0.5f, (((r * a) * (a - 1.0f)) * (a - 2.0f)) / 6.0f), a);
}

// mass_correction_apply.wgsl:258-321.  Grid [nx, ny, nz].  The totals over the
// levels are formed by two lanes of each workgroup (by every thread for itself: 20
// us at 120 x 120 x 40, now 15).
__global__ __launch_bounds__(256) void k_mass_correction_apply(uint32_t* M, KArg a) {
  __shared__ DFs total[2];
  __shared__ float part[2][64][2];
  const Dims g = dims(a.q[0], 0);
  const int id = (int)(threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z));
  const int threads = (int)(blockDim.x * blockDim.y * blockDim.z);
  DFs s{0.0f, 0.0f};
  for (int k0 = 0; k0 < g.nz; k0 += 64) {
    for (int q = id; q < 256; q += threads) {  // (sum, level, part)
      const int kk = k0 + q / 2 % 64;
      if (kk < g.nz) part[q / 128][q / 2 % 64][q % 2] = fq(a.q[2 + q / 128])[kk * 2 + q % 2];
    }
    __syncthreads();
    if (id < 2) {
      const int n = min(64, g.nz - k0);
      for (int t = 0; t < n; ++t) df_add_pair(s, part[id][t][0], part[id][t][1]);
      total[id] = s;
    }
    __syncthreads();
  }
  TE_TID3
  const int i = gx, j = gy, k = gz;
  if (i >= g.nx || j >= g.ny || k >= g.nz) return;
  const int moist = ldi(a.q[1], 0);
  const float *ref = fq(a.q[4]), *thP = fq(a.q[5]), *th0 = fq(a.q[7]), *pi0 = fq(a.q[8]), *qv = fq(a.q[9]);
  float *pp3d = fq(a.q[6]), *prs = fq(a.q[10]), *rho = fq(a.q[11]), *out = fq(a.q[12]);
  const DFs m2 = total[0], pp2 = total[1];
  const float rddcv = RD / (CP - RD);
  const float r = ((ref[0] - m2.x) + (ref[1] - m2.y)) / m2.x;
  const float p2 = pp2.x + pp2.y;
  const float tem = (powm1(r, rddcv) * p2) / (float)((g.nx * g.ny) * g.nz);
  if (i == 0 && j == 0 && k == 0) {
    out[0] = tem; out[1] = m2.x; out[2] = p2; out[3] = r; out[4] = m2.y;
  }
  const int64_t c = g.idx(i, j, k);
  const float pp = pp3d[c] + tem;
  pp3d[c] = pp;
  const float cpdrd = CP / RD;
  const float pi = pi0[k] + pp;
  const float th = th0[k] + thP[c];
  const float p = P00 * fast_pow(pi, cpdrd);
  prs[c] = p;
  const float rmix = moist != 0 ? fma_(mx(0.0f, qv[c]), RV, RD) : RD;
  rho[c] = p / ((th * pi) * rmix);
}

}  // namespace te
