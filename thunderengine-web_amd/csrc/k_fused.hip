// Launches that replace a run of reference dispatches (encoder option
// `fuse`).  Each produces the same bits as the run it replaces on every
// field the step carries.
#include "te_device.hpp"
#include <type_traits>

#include "te_kernels.hpp"
#include "pointwise.hpp"

namespace te {

// Periodic halos of up to 8 fields in one launch.  Replaces, per field, the
// pair bc_periodic_x + bc_periodic_y (bc_periodic_x.wgsl:111-133,
// bc_periodic_y.wgsl:111-133; timestep.js haloFill): the x pass copies
// interior columns into the i-halo of every row, the y pass then copies whole
// rows (including the fresh i-halo) into the j-halo, so every halo cell ends
// as the image f[i mod nx, j mod ny, k] of an interior cell; this kernel
// writes exactly those images.
// Grid: x = halo cells of one level (7 rows of strideJ, then ny rows of 7),
// y = k in [0, nz].  p[1..8] fields, p[9] -> field count.
__global__ __launch_bounds__(256) void k_bc_periodic_xy(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  const int k = gy;
  if (k > g.nz) return;
  const int rowCells = 7 * g.sJ;
  int i, j;
  if (gx < rowCells) {
    const int r = gx / g.sJ;           // 0..6 -> j = -3..-1, ny..ny+3
    i = gx - r * g.sJ - 3;
    j = r < 3 ? r - 3 : g.ny + (r - 3);
  } else {
    const int t = gx - rowCells;       // ny rows x 7 halo columns, row by row
    j = t / 7;
    const int cidx = t - j * 7;
    if (j >= g.ny) return;
    i = cidx < 3 ? cidx - 3 : g.nx + (cidx - 3);
  }
  const int si = ((i % g.nx) + g.nx) % g.nx, sj = ((j % g.ny) + g.ny) % g.ny;
  const int64_t dst = g.idx(i, j, k), src = g.idx(si, sj, k);
  const int n = ldi(a.q[9], 0);
  for (int q = 0; q < 8; ++q) {
    if (q >= n) break;
    float* f = fq(a.q[1 + q]);
    f[dst] = f[src];
  }
}

// Halos of up to 8 fields on a domain with an open side, in one launch.
// Replaces, per field, bc_periodic_x or bc_open_x and bc_periodic_y or
// bc_open_y in haloFill's order (timestep.js haloFill: the periodic passes,
// then the open ones).  Each pass copies whole lines of the other direction,
// halo included, so a halo cell ends as the value at (sx(i), sy(j)): on a
// periodic axis the image modulo n; on an open one the nearest cell of
// [0, last], last = n - 1 (n for a field on that axis' faces), for the three
// cells past either end, and the cell itself beyond them (bc_open_x.wgsl:111-131
// fills three).  No source is itself filled, so every cell can be written at
// once.  The fill moves a few percent of the field and is bound by the launch:
// 120 x 120 x 40 with 7 species has 188 of these passes per step at 3.0-3.4 us
// each; one launch for the 4 fields of a substep takes about what one pass did.
// Grid as k_bc_periodic_xy.  p[1..8] fields, p[9] -> count, open x, open y and
// per field 1 (on x faces), 2 (on y faces) or 0.
TE_DEV bool halo_cell_at(const Dims& g, int n, int& i, int& j) {
  const int rowCells = 7 * g.sJ;
  if (n < rowCells) {
    const int r = n / g.sJ;            // 0..6 -> j = -3..-1, ny..ny+3
    i = n - r * g.sJ - 3;
    j = r < 3 ? r - 3 : g.ny + (r - 3);
    return true;
  }
  const int t = n - rowCells;          // ny rows x 7 halo columns, row by row
  j = t / 7;
  const int cidx = t - j * 7;
  i = cidx < 3 ? cidx - 3 : g.nx + (cidx - 3);
  return j < g.ny;
}
TE_DEV int halo_source(int q, int cells, bool open, int last) {
  if (!open) return ((q % cells) + cells) % cells;
  return q < 0 ? 0 : (q > last && q <= last + 3 ? last : q);
}
__global__ __launch_bounds__(256) void k_bc_open_xy(uint32_t* M, KArg a) {
  TE_TID3
  const Dims g = dims(a.q[0], 0);
  const int k = gy;
  if (k > g.nz) return;
  int i, j;
  if (!halo_cell_at(g, gx, i, j)) return;
  const uint32_t* P = a.q[9];
  const int n = ldi(P, 0);
  const bool openx = ldi(P, 1) != 0, openy = ldi(P, 2) != 0;
  const int64_t dst = g.idx(i, j, k);
  float v[8];
  bool fill[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    fill[q] = false;
    if (q < n) {
      const int on = ldi(P, 3 + q);
      const int64_t src =
          g.idx(halo_source(i, g.nx, openx, g.nx - 1 + (on == 1)), halo_source(j, g.ny, openy, g.ny - 1 + (on == 2)), k);
      fill[q] = src != dst;
      if (fill[q]) v[q] = fq(a.q[1 + q])[src];
    }
  }
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (fill[q]) fq(a.q[1 + q])[dst] = v[q];
}

__global__ __launch_bounds__(256) void k_rk_update_xy(uint32_t* M, KArg a) { rk_update_xy_body(M, a, te_block(a)); }

__global__ __launch_bounds__(256) void k_tke_advance_xy(uint32_t* M, KArg a) { tke_advance_xy_body(M, a, te_block(a)); }

__global__ __launch_bounds__(256) void k_zero_fields(uint32_t* M, KArg a) { zero_fields_body(M, a, te_block(a)); }

// turb_add_tendency (dst = fma(scale, src, dst) over the whole grid) for up
// to 4 independent triples: p[1..4] sources, p[5..8] destinations,
// p[9..12] -> scales, p[13] -> count.
__global__ __launch_bounds__(256) void k_add_fields(uint32_t* M, KArg a) {
  if (te_flat(a, te_block(a), [&](uint32_t w, int width) {
        const int n = ldi(a.q[13], 0);
        for (int q = 0; q < 4; ++q) {
          if (q >= n) break;
          const float sc = ldf(a.q[9 + q], 0);
          const F4 s = ld4(a.q[1 + q], w, width);
          F4 d = ld4(a.q[5 + q], w, width);
          for (int e = 0; e < width; ++e) d.v[e] = fma_(sc, s.v[e], d.v[e]);
          st4(a.q[5 + q], w, width, d);
        }
      }))
    return;
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  const int64_t c = g.idx(i, j, k);
  const int n = ldi(a.q[13], 0);
  for (int q = 0; q < 4; ++q) {
    if (q >= n) break;
    float* dst = fq(a.q[5 + q]);
    dst[c] = fma_(ldf(a.q[9 + q], 0), fq(a.q[1 + q])[c], dst[c]);
  }
}

__global__ __launch_bounds__(256) void k_tendency_reset_add(uint32_t* M, KArg a) { tendency_reset_add_body(M, a, te_block(a)); }

__global__ __launch_bounds__(256) void k_copy_fields(uint32_t* M, KArg a) { copy_fields_body(M, a, te_block(a)); }

// ---- acoustic substep
// acoustic_pp (acoustic_pp.wgsl:131-167) at interior points, then
// acoustic_accumulate (acoustic_accumulate.wgsl:129-158) at every point of
// the whole grid.  Neither reads what the other writes, so one pass does
// both.  p: 0 dims, 1 acoustic, 2 w, 3 pk1, 4 pk2, 5 qk, 6 fpk, 7 pp3d, 8 ppd,
// 9 ppx, 10 -> saveX, 11 u, 12 v, 13 rru, 14 rrv, 15 rrw, 16 -> tavg, 17-19
// (if bound) the fields the accumulated rru, rrv, rrw go to instead.
__global__ __launch_bounds__(256) void k_ac_pp_accumulate(uint32_t* M, KArg a) {
  TE_TID3
  Dims g = dims(a.q[0], 0);
  int i = gx - 3, j = gy - 3, k = gz;
  if (i > g.nx + 3 || j > g.ny + 3 || k > g.nz) return;
  Acoustic ac = acoustic(a.q[1], 0);
  const float* w = fq(a.q[2]);
  const int64_t sk = g.sk(), c = g.idx(i, j, k);
  const float wc = w[c];
  if (i >= 0 && i < g.nx && j >= 0 && j < g.ny && k < g.nz) {
    const float *pk1 = fq(a.q[3]), *pk2 = fq(a.q[4]), *qk = fq(a.q[5]), *fpk = fq(a.q[6]);
    float *pp3d = fq(a.q[7]), *ppd = fq(a.q[8]), *ppx = fq(a.q[9]);
    const float prev = pp3d[c];
    float p = fma_(ac.alph, fma_(wc, pk1[c] + qk[c], w[c + sk] * (pk2[c] - qk[c])), prev + fpk[c]);
    if (ab(p) < ac.smeps) p = 0.0f;
    pp3d[c] = p;
    const float dum1 = ac.kdiv * (p - prev);
    ppd[c] = p + dum1;
    if (ldi(a.q[10], 0) != 0) ppx[c] = dum1;
  }
  const float *u = fq(a.q[11]), *v = fq(a.q[12]);
  const float *rru = fq(a.q[13]), *rrv = fq(a.q[14]), *rrw = fq(a.q[15]);
  auto out = [&](int q, int in) { return fq(a.p[q] != 0 ? a.q[q] : a.q[in]); };
  float *ru = out(17, 13), *rv = out(18, 14), *rw = out(19, 15);
  const float tavg = ldf(a.q[16], 0);
  if (tavg > 0.0f) {
    ru[c] = (rru[c] + u[c]) * tavg;
    rv[c] = (rrv[c] + v[c]) * tavg;
    rw[c] = fma_(wc, ac.alph, rrw[c]) * tavg;
  } else {
    ru[c] = rru[c] + u[c];
    rv[c] = rrv[c] + v[c];
    rw[c] = rrw[c] + wc;
  }
}

}  // namespace te

namespace te {

// One acoustic substep's accumulation of u and v over the whole grid
// (acoustic_accumulate's rru, rrv) and the halo fill of u and v, by workgroups of their own in the same
// launch: none of it waits for the column sweep, whose workgroups leave the
// memory idle while they pass it on.  A wave takes AC_UV_UNITS (row, 64
// columns) pairs, all loads before the first store (4: 2, 8 and 16 were slower
// from 160 x 160 x 40 on, by up to 3, 1 and 7% of a step); the pairs are
// numbered level by level within a row j, so that an XCD takes the rows its
// column workgroups read.  u at (nx, j) and v at (i, ny) of interior rows /
// columns belong to the column workgroups, which read them.
// OPEN: a side is open (p38); a halo cell's image is then found per field and
// axis as by bc_open_xy, and u at (nx, j), v at (i, ny) of an open axis are
// faces like the others.
template <bool OPEN>
TE_DEV void ac_accumulate_uv(uint32_t* M, const KArg& a, const Dims& g, uint32_t wg, int wave, int lane) {
  const uint32_t n = a.n[2], q8 = n >> 3, r8 = n & 7u, xcd = wg & 7u;  // a.n[2]: workgroups of this kind
  const uint32_t l = xcd * q8 + min(xcd, r8) + (wg >> 3);
  const int nc = (g.sJ + 63) / 64, nl = g.nz + 1, units = g.sK * nl * nc;
  auto F = [&](int q) { return FieldB(reinterpret_cast<float*>(M) + a.p[q]); };
  const FieldB u = F(2), v = F(3), rru = F(13), rrv = F(14);
  const FieldB rruO = a.p[35] != 0 ? F(35) : rru, rrvO = a.p[36] != 0 ? F(36) : rrv;
  const bool openx = OPEN && ldi(a.q[38], 0) != 0, openy = OPEN && ldi(a.q[38], 1) != 0;
  auto source = [](int q, int cells, bool open, int last) {
    if (!open) return q < 0 ? q + cells : q >= cells ? q - cells : q;
    return q < 0 ? 0 : (q > last && q <= last + 3 ? last : q);
  };
  const bool first = ldi(a.q[33], 0) != 0;
  const float tavg = ldf(a.q[17], 0), tv = tavg > 0.0f ? tavg : 1.0f;
  const uint32_t sjb = 4u * (uint32_t)g.sJ, skb = sjb * (uint32_t)g.sK;
  const int u0 = (int)(l * AC_WAVES + (uint32_t)wave) * AC_UV_UNITS;
  uint32_t h[AC_UV_UNITS];
  int todo[AC_UV_UNITS];  // 1 rru, 2 rrv, 4 a halo cell, 8 u and 16 v from its image
  float uo[AC_UV_UNITS], vo[AC_UV_UNITS], ru[AC_UV_UNITS], rv[AC_UV_UNITS], us[AC_UV_UNITS], vs[AC_UV_UNITS];
#pragma unroll
  for (int d = 0; d < AC_UV_UNITS; ++d) {
    const int id = u0 + d;
    todo[d] = 0;
    if (id >= units) continue;
    const int row = id / nc, c = id - row * nc, jr = row / nl, k = row - jr * nl;
    const int i = c * 64 + lane - 3, j = jr - 3;
    if (i > g.nx + 3) continue;
    const bool hx = i < 0 || i >= g.nx, hy = j < 0 || j >= g.ny;
    const uint32_t lv = skb * (uint32_t)k;
    h[d] = lv + 4u * (uint32_t)(i + 3) + sjb * (uint32_t)jr;
    todo[d] = (!openx && !hy && i == g.nx ? 0 : 1) | (!openy && !hx && j == g.ny ? 0 : 2) | (hx || hy ? 4 : 0);
    uo[d] = u(h[d]);
    vo[d] = v(h[d]);
    ru[d] = rv[d] = 0.0f;
    if (!first) {
      ru[d] = rru(h[d]);
      rv[d] = rrv(h[d]);
    }
    if (OPEN && (todo[d] & 4)) {
      const int su = source(i, g.nx, openx, g.nx), ju = source(j, g.ny, openy, g.ny - 1);
      const int sv = source(i, g.nx, openx, g.nx - 1), jv = source(j, g.ny, openy, g.ny);
      us[d] = u(lv + 4u * (uint32_t)(su + 3) + sjb * (uint32_t)(ju + 3));
      vs[d] = v(lv + 4u * (uint32_t)(sv + 3) + sjb * (uint32_t)(jv + 3));
      if (su != i || ju != j) todo[d] |= 8;
      if (sv != i || jv != j) todo[d] |= 16;
    } else if (todo[d] & 4) {
      const int si = i < 0 ? i + g.nx : i >= g.nx ? i - g.nx : i, sj = j < 0 ? j + g.ny : j >= g.ny ? j - g.ny : j;
      const uint32_t src = lv + 4u * (uint32_t)(si + 3) + sjb * (uint32_t)(sj + 3);
      us[d] = u(src);
      vs[d] = v(src);
      todo[d] |= 24;
    }
  }
#pragma unroll
  for (int d = 0; d < AC_UV_UNITS; ++d) {
    if (todo[d] & 1) rruO.put(h[d], (ru[d] + uo[d]) * tv);
    if (todo[d] & 2) rrvO.put(h[d], (rv[d] + vo[d]) * tv);
    if ((todo[d] & 9) == 9) u.put(h[d], us[d]);
    if ((todo[d] & 18) == 18) v.put(h[d], vs[d]);
  }
}

// One acoustic substep after acoustic_uv, in one launch:
// acoustic_fpk, acoustic_w_solve, acoustic_pp and acoustic_accumulate, then
// the periodic halo fill of ppd, u, v and w, and on the stage's last substep
// the one of pp3d that follows the substeps (timestep.js:2023-2054,
// acoustic_fpk.wgsl:167-207, acoustic_w_solve.wgsl:124-212,
// acoustic_pp.wgsl:131-167, acoustic_accumulate.wgsl:129-158); on the first
// substep of a stage also acoustic_begin (acoustic_begin.wgsl:129-149).
// acoustic_prepare's qk, pk1, pk2 and mm (acoustic_prepare.wgsl:131-184) are
// formed per level from ppterm, piadv and thv with its operations, instead of
// being stored once per stage and read on every substep.
//
// A workgroup owns 64 columns of one row (lanes along i) and all levels:
// AC_WAVES waves each take a contiguous range of levels for the pointwise
// parts, and the tridiagonal sweep is passed from wave to wave (forward
// elimination upwards, back substitution downwards), each wave keeping its
// levels' coefficients in registers.  Values of the sweep are the reference's
// sequential Thomas recurrence, level by level.
//
// The nz levels are dealt nz / AC_WAVES or one more to each wave, so only the
// last of a wave's L rows is conditional; lanes past nx follow column nx - 1
// and store nothing.  The elimination forms a row's coefficients while the
// pivot before it is inverted, and takes the division only where a wave meets a
// pivot outside the refined reciprocal's range (one uniform branch per row).
//
// OPEN (a side is open, p38): the halo of w, ppd and rrw is left to
// ac_halo_open, since an open side's cells have up to 15 copies each; of a
// periodic axis u at (nx, j) or v at (i, ny) stay here.  us per substep at
// 120 x 120 x 40 with 7 species: 43 in six launches (edges, uv, fpk, w, pp with
// the accumulation, halos) and 27 in three.
// Halo cells (every halo cell of ppd, u, v, w is the image of interior cell
// (i mod nx, j mod ny), as the halo fill leaves it), each updated by the
// workgroup of its interior cell, at each level by the wave that owns it:
//  * w and ppd: rrw accumulates the image's old w (the accumulate runs
//    before the fill), then the new values are copied in.
//  * u and v: rru, rrv accumulate the value there (acoustic_uv's at i = nx or
//    j = ny, else the old image), then the image is copied in.  u at
//    (nx, j) and v at (i, ny) are updated by the workgroup of column nx-1 /
//    row ny-1, the only one that reads them (acoustic_fpk), after its reads;
//    all the others, with the accumulation at interior points, by
//    ac_accumulate_uv's workgroups.
// Only the new w, ppd and pp3d wait for the sweep.  The rest (`early`) is done
// where the wave would wait for the sweep: before the elimination in the upper
// waves, before the back substitution in the lower ones.  What follows the
// sweep then holds stores only.  (gfx950 retires a wave's loads and stores in
// order, so a load behind stores waits for their acknowledgement: 2-4 k cycles
// with the grid's traffic, and every turn from stores to loads costs that.)
// What bounds it: below about 256 workgroups the chain of one workgroup's
// phases, above them the memory (212 MB of fields at 192 x 192 x 80).  Clock
// stamps of the form before (a branch around each reciprocal, loads and stores
// in turn after the sweep, halos last): 300 cycles to eliminate a row and 150 to
// substitute it back, 45 k cycles in a row without y images and 60 k in one
// with them at 64 x 64 x 40, 125 k and 180 k at 192 x 192 x 80; now 120 and 60
// per row, 26 k and 32 k, 105 k and 145 k.  us per launch within a step, before
// and now: 64 x 64 x 40 24.3 and 13.9, 192 x 192 x 80 69 and 56, 256 x 256 x 120
// 203 and 165.  A reload of a spilled register behind stores waits for them, so 9
// to 12 levels per wave have 1 level of loads in flight: these instances still
// spill 3 to 12 VGPRs (open sides: 0 to 2), with 2 levels more (7 us longer a
// launch at 192 x 192 x 80).
// p: 0 dims, 1 acoustic, 2 u, 3 v, 4 w, 5 piadv, 6 ppten, 7 ppterm, 8 thv,
//    9 wten, 10 pp3d, 11 ppd, 12 ppx, 13 rru, 14 rrv, 15 rrw, 16 -> save ppx,
//    17 -> tavg, 18 rr0, 19 rf0, 20 mh, 21 mf, 22 c1, 23 c2, 30 metric,
//    33 -> first substep of the stage, 34 -> (if bound) fill pp3d's halo
//    too (with ppd's, group 4 below); the fields the replaced dispatches
//    write as scratch (for expansions of this launch into them): 24 qk,
//    25 pk1, 26 pk2, 27 mm, 28 fpk, 29 cA, 31 cB, and 32 rho0; 35-37 (if
//    bound) the fields the accumulated rru, rrv, rrw go to instead, every word
//    (OPEN: but the halo of rrw); 38 -> open x, open y (OPEN only).
// Grid: 64 x AC_WAVES threads per workgroup, ceil(nx / 64) * ny workgroups of
// columns (padded to a multiple of 8), then a.n[2] of ac_accumulate_uv.
// Needs nx, ny >= 4, 4 <= nz <= AC_WAVES * 16, and fields below 2^32 bytes
// (word offsets into M are 32 bits and a program's fields share that range).
#define AC_HALO_CELLS 40  // per workgroup: at most 7 x-images, 1 (nx, j) cell, 14 corners
template <int L, bool OPEN>
__device__ __forceinline__ void ac_column(uint32_t* M, const KArg& a) {
  // Few levels per wave: the later phases' operands are kept or loaded ahead
  // of the sweep (registers to spare); many: the w rows wait in LDS and the
  // loads come in chunks, so that three workgroups stay resident per CU.
  constexpr bool AHEAD = L <= 6;
  constexpr int CH = AHEAD ? L : L >= 9 && L <= 12 ? 1 : 2;  // levels of loads in flight, pointwise part
  __shared__ float xa[AC_WAVES][3][64];  // pk1+qk, pk2-qk, pp3d+fpk at each wave's last level
  __shared__ float xb[2][64];            // elimination carry between waves
  __shared__ float xw[64];               // new w at the first level of the wave above
  __shared__ int fwd_done, back_next;    // the sweep's hand-offs between waves
  __shared__ int hcnt;
  __shared__ uint32_t hcell[AC_HALO_CELLS];
  // acoustic_prepare's per-level factors tem, r1, r2, tem1, c1, c2: scalar
  // loads where a wave has few levels, else a table
  __shared__ float lv[AHEAD ? 1 : 6][AHEAD ? 1 : AC_WAVES * 16 + 1];
  // dynamic (L > 6): per level and lane mm and the w row's right-hand side
  // part, then the elimination coefficients
  float* me0 = te_lds;
  const int lane = (int)threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.y);  // one wave per threadIdx.y
  const Dims g = dims(a.q[0], 0);
  const uint32_t solvers = (a.lg[9] + 7u) & ~7u;  // workgroups of columns, padded to the XCDs
  if (blockIdx.x >= solvers) {
    ac_accumulate_uv<OPEN>(M, a, g, blockIdx.x - solvers, wave, lane);
    return;
  }
  if (blockIdx.x >= a.lg[9]) return;
  const Blk blk = te_block(a);
  const int i = blk.x * 64 + lane, j = blk.y, nx = g.nx, ny = g.ny, nz = g.nz;
  float* me1 = te_lds + nz * 64;
  const bool active = i < nx;
  const int ic = min(i, nx - 1);
  const int base = nz / AC_WAVES, rem = nz % AC_WAVES;
  const int Lq = base + (wave < rem ? 1 : 0), k0 = wave * base + min(wave, rem);
  const bool full = Lq == L;  // else Lq == L - 1
  const bool top = Lq > 0 && k0 + Lq == nz;
  const Acoustic ac = acoustic(a.q[1], 0);
  auto F = [&](int q) { return FieldB(reinterpret_cast<float*>(M) + a.p[q]); };
  auto prof = [&](int q, int k) { return (reinterpret_cast<const float*>(M) + a.p[q])[k]; };
  const bool saveX = ldi(a.q[16], 0) != 0, first = ldi(a.q[33], 0) != 0;
  const bool imgP = a.p[34] != 0 && ldi(a.q[34], 0) != 0;
  const float tavg = ldf(a.q[17], 0);
  if (threadIdx.x == 0 && threadIdx.y == 0) {
    fwd_done = 0;
    back_next = AC_WAVES - 1;
    hcnt = 0;
  }
  // Halo cells of the x-images and corners of this workgroup's columns, and
  // (nx, j) (low bit set): byte offsets within a level
  const bool openx = OPEN && ldi(a.q[38], 0) != 0, openy = OPEN && ldi(a.q[38], 1) != 0;
  const int ys[2] = {j >= ny - 3 ? j - ny : j, j <= 3 ? j + ny : j};
  const uint32_t sjb = 4u * (uint32_t)g.sJ, skb = sjb * (uint32_t)g.sK;
  auto cell = [&](int x, int y) { return 4u * (uint32_t)(x + 3) + sjb * (uint32_t)(y + 3); };
  if (OPEN) {
    if (active && wave == 0 && i == nx - 1 && !openx) {
      hcell[0] = cell(nx, j) | 1u;
      hcnt = 1;
    }
  } else if (active && wave == 0) {  // (one wave: its LDS operations keep their order)
    const int xs[2] = {i >= nx - 3 ? i - nx : i, i <= 3 ? i + nx : i};
    const int nxi = (i >= nx - 3) + (i <= 3), nyi = (j >= ny - 3) + (j <= 3);
    const int n = nxi * (1 + nyi) + (i == nx - 1);
    if (n > 0) {
      int q = atomicAdd(&hcnt, n);
      for (int by = 0; by < 3; ++by)
        for (int bx = 0; bx < 2; ++bx) {
          const int hx = xs[bx], hy = by == 0 ? j : ys[by - 1];
          if (hx == i || (by > 0 && hy == j)) continue;
          hcell[q++] = cell(hx, hy);
        }
      if (i == nx - 1) hcell[q] = cell(nx, j) | 1u;
    }
  }
  auto prep = [&](int k, float f[6]) {
    const int kp = min(k + 1, nz);
    const float tem = (ac.dts * g.rdz) * prof(20, k), rr0k = prof(18, k);
    f[0] = tem;
    f[1] = (tem * rr0k) * prof(19, k);
    f[2] = (tem * rr0k) * prof(19, kp);
    f[3] = ((ac.dts * g.rdz) * CP) * prof(21, k);
    f[4] = prof(22, k);
    f[5] = prof(23, k);
  };
  if constexpr (!AHEAD) {
    for (int k = (int)(threadIdx.y * 64 + threadIdx.x); k <= nz; k += 64 * AC_WAVES) {
      float f[6];
      prep(k, f);
      for (int q = 0; q < 6; ++q) lv[q][k] = f[q];
    }
    __syncthreads();
  }
  const FieldB u = F(2), v = F(3), w = F(4), piadv = F(5), ppten = F(6), ppterm = F(7), thv = F(8), wten = F(9),
               pp3d = F(10), ppd = F(11), ppx = F(12), rru = F(13), rrv = F(14), rrw = F(15);
  const FieldB rruO = a.p[35] != 0 ? F(35) : rru, rrvO = a.p[36] != 0 ? F(36) : rrv, rrwO = a.p[37] != 0 ? F(37) : rrw;
  // byte offset of this lane's column at level k (the same in every field)
  const uint32_t o00 = cell(ic, j);
  auto at = [&](int k) { return o00 + skb * (uint32_t)k; };
  const float asq = ac.alph * ac.alph;
  const float temx = (ac.dts * 0.5f) * g.rdx, temy = (ac.dts * 0.5f) * g.rdy;
  const bool vec_v = nx > 3 && i < (nx / 4) * 4;
  // the accumulation, scaled on the last substep; before it the factors are 1
  // (exact in both operations)
  const float tv = tavg > 0.0f ? tavg : 1.0f, al = tavg > 0.0f ? ac.alph : 1.0f;
  auto acc = [&](float b, float x) { return (b + x) * tv; };
  auto accw = [&](float b, float x) { return fma_(x, al, b) * tv; };
#define ROW(t) ((t) < L - 1 || full)
  float PQ[L], P2Q[L], PF[L], ME[L], EE[L];
  // ---- pointwise: acoustic_prepare's terms, acoustic_fpk, the w row's
  // right-hand side.  Row L - 1 of a wave with L - 1 levels is formed from
  // the level above (or level nz) and not used.
  float PP[L];  // pp3d before the substep
  {
    const float* hm = reinterpret_cast<const float*>(M) + a.p[30];
    const float uh = hm_uh(hm, g, ic), vh = hm_vh(hm, g, j);
    const uint32_t om = at(max(k0 - 1, 0));  // level -1 is not used
    float pam = piadv(om), thm0 = thv(om), ppm = pp3d(om);
#pragma unroll
    for (int t0 = 0; t0 < L; t0 += CH) {
      float U[CH], UP[CH], V[CH], VP[CH], W[CH + 1], PA[CH + 1], XM[CH], XP[CH], YM[CH], YP[CH], PT[CH], PN[CH], TH[CH],
          WT[CH];
#pragma unroll
      for (int d = 0; d < CH; ++d)
        if (t0 + d < L) {
          const uint32_t o = at(min(k0 + t0 + d, nz));
          U[d] = u(o); UP[d] = u(o + 4u); V[d] = v(o); VP[d] = v(o + sjb);
          W[d] = w(o); PA[d] = piadv(o);
          XM[d] = piadv(o - 4u); XP[d] = piadv(o + 4u); YM[d] = piadv(o - sjb); YP[d] = piadv(o + sjb);
          PT[d] = ppterm(o); PN[d] = ppten(o); PP[t0 + d] = pp3d(o); TH[d] = thv(o); WT[d] = wten(o);
        }
      {
        const int n = t0 + CH < L ? CH : L - t0;  // rows of this chunk; the level above its last
        const uint32_t o = at(min(k0 + t0 + n, nz));
        W[n] = w(o);
        PA[n] = piadv(o);
      }
      // AHEAD: the workgroup meets here, every load on its way, rather than
      // before them (what the barrier guards lies in LDS: the counters and the
      // list above)
      if constexpr (AHEAD) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
#pragma unroll
      for (int d = 0; d < CH; ++d)
        if (t0 + d < L) {
          const int t = t0 + d, k = min(k0 + t, nz), kp = min(k + 1, nz);
          const float pa0 = PA[d];
          const bool bot = k == 0, ktop = k == nz - 1;
          const float pzp = ktop ? 0.0f : PA[d + 1], pzm = bot ? 0.0f : pam, thm = bot ? TH[d] : thm0;
          float f[6];
          if constexpr (AHEAD) {
            prep(k, f);
          } else {
            for (int q = 0; q < 6; ++q) f[q] = lv[q][k];
          }
          const float tem = f[0], r1 = f[1], r2 = f[2], tem1 = f[3], c1a = f[4], c2a = f[5];
          const float c1b = AHEAD ? prof(22, kp) : lv[AHEAD ? 0 : 4][AHEAD ? 0 : kp], c2b = AHEAD ? prof(23, kp) : lv[AHEAD ? 0 : 5][AHEAD ? 0 : kp];
          const float qk = tem * PT[d];
          const float p2 = ktop ? 0.0f : (vec_v ? fma_(-c2b, pzp, (1.0f - c1b) * pa0) : fma_(1.0f - c1b, pa0, -(c2b * pzp)));
          const float p1 = bot ? 0.0f : (vec_v ? fma_(c2a - 1.0f, pa0, c1a * pzm) : fma_(c1a, pzm, (c2a - 1.0f) * pa0));
          const float pk2 = ktop ? 0.0f : r2 * p2;
          const float pk1 = bot ? 0.0f : r1 * p1;
          const float mm = tem1 * fma_(c2a, TH[d], c1a * thm);
          float div = fma_((UP[d] - U[d]) * g.rdx, uh, ((VP[d] - V[d]) * g.rdy) * vh);
          if (ab(div) < ac.smeps) div = 0.0f;
          const float Au = fma_(U[d], pa0 - XM[d], UP[d] * (XP[d] - pa0));
          const float Av = fma_(V[d], pa0 - YM[d], VP[d] * (YP[d] - pa0));
          const float advPi = fma_((-Au) * temx, uh, -((Av * temy) * vh));
          const float fpk = fma_(ac.beta, fma_(W[d], pk1 + qk, W[d + 1] * (pk2 - qk)),
                                 fma_(ac.dts, fma_(-PT[d], div, PN[d]), advPi));
          PQ[t] = pk1 + qk;
          P2Q[t] = pk2 - qk;
          PF[t] = PP[t] + fpk;
          ME[t] = mm;
          EE[t] = bot ? 0.0f : W[d] + fma_(ac.dts, WT[d], ac.beta * ((-mm) * (PP[t] - ppm)));
          te_pin(PQ[t]); te_pin(P2Q[t]); te_pin(PF[t]); te_pin(ME[t]); te_pin(EE[t]);
          if constexpr (!AHEAD)
            if (ROW(t)) {
              me0[k * 64 + lane] = ME[t];
              me1[k * 64 + lane] = EE[t];
            }
          ppm = PP[t];
          pam = pa0;
          thm0 = TH[d];
        }
    }
    if (Lq > 0) {
      xa[wave][0][lane] = full ? PQ[L - 1] : PQ[L > 1 ? L - 2 : 0];
      xa[wave][1][lane] = full ? P2Q[L - 1] : P2Q[L > 1 ? L - 2 : 0];
      xa[wave][2][lane] = full ? PF[L - 1] : PF[L > 1 ? L - 2 : 0];
    }
  }
  float RW[L], ppdz = 0.0f, ppz = 0.0f;  // rrw before the substep; ppd, pp3d of level nz
  // What does not wait for the sweep (see above).  Level nz goes with the top
  // wave: w stays 0 there (acoustic_w_solve clears it), ppd is not updated.
  auto early = [&]() {
    const int nl = Lq + (top ? 1 : 0);
    if (top) {
      const uint32_t o = at(nz);
      const float rw = first ? w(o) * ac.beta : rrw(o);
      ppdz = ppd(o);
      ppz = pp3d(o);
      if (active) {
        rrwO.put(o, accw(rw, 0.0f));
        w.put(o, 0.0f);
      }
    }
    // a halo cell's rrw accumulates the old w there; u at (nx, j) and v at
    // (i, ny) are accumulated, then replaced by their images
    struct Item {
      uint32_t h;
      int m;
      float x, y, z;
    };
    // the x-images, the corners and (nx, j): the list, a (cell, level) pair per
    // lane, the first 64 pairs loaded before the first store
    const int nc = hcnt, items = nc * nl;
    auto item = [&](int it) {
      Item c = {0u, 0, 0.0f, 0.0f, 0.0f};
      if (it < items) {
        const int kk = it / nc;
        const uint32_t e = hcell[it - kk * nc], lv = skb * (uint32_t)(k0 + kk);
        c.m = e & 1u ? 1 : 4;
        c.h = lv + (e & ~3u);
        if (c.m == 4) {
          c.x = w(c.h);
          c.y = first ? c.x * ac.beta : rrw(c.h);
        } else {
          c.x = u(c.h);
          c.y = first ? 0.0f : rru(c.h);
          c.z = u(lv + cell(0, j));
        }
      }
      return c;
    };
    auto store = [&](const Item& c) {
      if (c.m == 4) {
        rrwO.put(c.h, accw(c.y, c.x));
      } else if (c.m != 0) {
        rruO.put(c.h, acc(c.y, c.x));
        u.put(c.h, c.z);
      }
    };
    const Item ia = item(lane);
    Item ib = {0u, 0, 0.0f, 0.0f, 0.0f};  // (rows with y images: more than 64 pairs)
    if (AHEAD && items > 64) ib = item(lane + 64);
    // the row's own images, lane = column: rows t0 .. t0 + CI - 1 of the wave
    // (and level nz as row Lq), loads without a branch between them
    constexpr int CI = AHEAD ? L : 5;
    auto batch = [&](int t0, auto&& f) {
#pragma unroll
      for (int d = 0; d < CI; ++d)
        if (t0 + d < L && ROW(t0 + d)) f(d, at(k0 + t0 + d));
    };
#pragma unroll 1
    for (int r = 0; r < (OPEN ? 0 : 2); ++r) {
      const int hy = ys[r];
      if (hy == j) continue;
      const uint32_t off = sjb * (uint32_t)(hy - j);
#pragma unroll
      for (int t0 = 0; t0 < L; t0 += CI) {
        float x[CI], y[CI], xz = 0.0f, yz = 0.0f;
        const bool z = top && t0 + CI >= L;
        batch(t0, [&](int d, uint32_t o) { x[d] = w(o + off); });
        if (z) xz = w(at(nz) + off);
        if (first) {
          batch(t0, [&](int d, uint32_t) { y[d] = x[d] * ac.beta; });
          yz = xz * ac.beta;
        } else {
          batch(t0, [&](int d, uint32_t o) { y[d] = rrw(o + off); });
          if (z) yz = rrw(at(nz) + off);
        }
        if (active) {
          batch(t0, [&](int d, uint32_t o) { rrwO.put(o + off, accw(y[d], x[d])); });
          if (z) rrwO.put(at(nz) + off, accw(yz, xz));
        }
      }
    }
    store(ia);
    if (AHEAD) store(ib);
#pragma unroll 1
    for (int it = lane + (AHEAD ? 128 : 64); it < items; it += 64) store(item(it));
    if (j == ny - 1 && !openy) {  // v at (i, ny)
      const uint32_t src = sjb * (uint32_t)(-j);
#pragma unroll
      for (int t0 = 0; t0 < L; t0 += CI) {
        float x[CI], y[CI], s[CI], xz = 0.0f, yz = 0.0f, sz = 0.0f;
        const bool z = top && t0 + CI >= L;
        batch(t0, [&](int d, uint32_t o) { x[d] = v(o + sjb); s[d] = v(o + src); y[d] = 0.0f; });
        if (!first) batch(t0, [&](int d, uint32_t o) { y[d] = rrv(o + sjb); });
        if (z) {
          const uint32_t o = at(nz);
          xz = v(o + sjb);
          sz = v(o + src);
          yz = first ? 0.0f : rrv(o + sjb);
        }
        if (active) {
          batch(t0, [&](int d, uint32_t o) {
            rrvO.put(o + sjb, acc(y[d], x[d]));
            v.put(o + sjb, s[d]);
          });
          if (z) {
            rrvO.put(at(nz) + sjb, acc(yz, xz));
            v.put(at(nz) + sjb, sz);
          }
        }
      }
    }
  };
  const FieldB rw0 = first ? w : rrw;  // acoustic_begin's rrw is w * beta
  const float bf = first ? ac.beta : 1.0f;
  auto load_rrw = [&]() {
#pragma unroll
    for (int t = 0; t < L; ++t) {
      RW[t] = 0.0f;
      if (ROW(t)) RW[t] = rw0(at(k0 + t));
    }
  };
  const bool upper = wave >= AC_WAVES / 2;
  // The sweep passes from wave to wave through LDS counters instead of
  // workgroup barriers, so a wave's share of the serial recurrence overlaps
  // the loads of the waves above it (forward) and the stores of the waves
  // that finished (backward).  Every wave passes every hand-off, in wave
  // order: wave w waits for fwd_done == w (set by wave w-1 after its
  // elimination) and for back_next == w (set by wave w+1 after its back
  // substitution; the top wave is the last of the forward chain), so each
  // wait ends once the waves below / above it have run.  The waits are
  // bounded (2^22 polls) all the same.  What is handed over lies in LDS, which
  // executes a wave's operations in the order it issues them: data written
  // before the flag is there when the flag is, and data read after the flag,
  // in the same poll, is valid when the flag was set.  So a hand-off waits for
  // no counter and reads nothing after the flag; a wave whose turn is next
  // polls without sleeping.  (450 cycles a hand-off with the flag behind a
  // wait, the data read after it and a sleep in every poll, 16 of them a
  // launch; a release of the wave's global accesses cost 43 k cycles at
  // 192 x 192 x 80.)
  auto wait_for = [&](int* flag, int want, auto&& read) {
    for (int s = 0; s < (1 << 22); ++s) {
      const int f0 = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      asm volatile("" ::: "memory");
      read();
      const int f = __builtin_amdgcn_readfirstlane(f0);
      if (f == want) break;
      if (f < want - 1 || f > want + 1) __builtin_amdgcn_s_sleep(1);
    }
    asm volatile("" ::: "memory");
  };
  auto pass = [&](int* flag, int f) {
    asm volatile("" ::: "memory");
    __hip_atomic_store(flag, f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  // ---- forward elimination, wave after wave: (mm, right-hand side) of a row
  // become its elimination coefficients (the top row's leave w at nz-1).
  // Row k = 1 has no row below it (row 1 of wave 0, or row 0 of wave 1 when
  // waves hold one level); level 0 is no row.
  float CA[L], CB[L];
  struct Row {
    float aa, cc, bb, dd;
  };
  // row t from PQ, P2Q and PF of its own level and of the one below
  auto row = [&](int t, float pq_m, float p2q_m, float ppf_m) {
    const float m = AHEAD ? ME[t] : me0[(k0 + t) * 64 + lane], e = AHEAD ? EE[t] : me1[(k0 + t) * 64 + lane];
    Row r = {(-asq) * (m * pq_m), (-asq) * ((-m) * P2Q[t]), fma_(-asq, m * ((-PQ[t]) + p2q_m), 1.0f),
             fma_(ac.alph, (-m) * (PF[t] - ppf_m), e)};
    te_pin(r.aa); te_pin(r.cc); te_pin(r.bb); te_pin(r.dd);
    return r;
  };
  // AHEAD: every row but the first (which waits for the wave below's last
  // level) before the wait; else row t + 1 between row t's pivot and the test
  // that waits for its reciprocal
  Row R[AHEAD ? L : 2];
  if constexpr (AHEAD) {
#pragma unroll
    for (int t = 1; t < L; ++t) R[t] = row(t, PQ[t - 1], P2Q[t - 1], PF[t - 1]);
  }
  if (upper && Lq > 0) early();
  float pa = 0.0f, pb = 0.0f, x0 = 0.0f, x1 = 0.0f, x2 = 0.0f;
  const int below = max(wave - 1, 0);
  wait_for(&fwd_done, wave, [&]() {
    pa = xb[0][lane];
    pb = xb[1][lane];
    x0 = xa[below][0][lane];
    x1 = xa[below][1][lane];
    x2 = xa[below][2][lane];
  });
  if (Lq > 0) {
    if (wave > 0) R[0] = row(0, x0, x1, x2);
    else pa = pb = 0.0f;
#pragma unroll
    for (int t = 0; t < L; ++t) {
      const bool first_row = t == (L > 1 ? 1 : 0) && k0 + t == 1;
      const Row& r = R[AHEAD ? t : t % 2];
      if (t == 0 ? (wave > 0 && ROW(0)) : ROW(t)) {
        const float x = first_row ? r.bb : fma_(r.aa, pa, r.bb);
        float y = recip_refined(x);
        if constexpr (!AHEAD)
          if (t + 1 < L) R[(t + 1) % 2] = row(t + 1, PQ[t], P2Q[t], PF[t]);
        if (__builtin_expect(__any(recip_far(x) > kRecipRange), 0)) y = recip(x);
        pb = (first_row ? r.dd : fma_(-r.aa, pb, r.dd)) * y;
        pa = (-r.cc) * y;
        if constexpr (AHEAD) {
          CA[t] = pa;  // not read for the top row (w there is pb)
          CB[t] = pb;
        } else {
          me0[(k0 + t) * 64 + lane] = pa;
          me1[(k0 + t) * 64 + lane] = pb;
        }
      } else if constexpr (!AHEAD) {
        if (t + 1 < L) R[(t + 1) % 2] = row(t + 1, PQ[t], P2Q[t], PF[t]);
      }
    }
    xb[0][lane] = pa;
    xb[1][lane] = pb;
  }
  pass(&fwd_done, wave + 1);
  if (!upper && Lq > 0) early();
  if (Lq > 0) load_rrw();
  // ---- back substitution, wave after wave downwards: CA becomes the new w
  float wnext = 0.0f;
  wait_for(&back_next, wave, [&]() { wnext = xw[lane]; });
  if (Lq > 0) {
    if (top) wnext = 0.0f;
    float wn = wnext;
#pragma unroll
    for (int t = L - 1; t >= 0; --t)
      if (ROW(t)) {
        const float ca = AHEAD ? CA[t] : me0[(k0 + t) * 64 + lane], cb = AHEAD ? CB[t] : me1[(k0 + t) * 64 + lane];
        wn = t >= L - 2 && k0 + t == nz - 1 ? cb : fma_(ca, wn, cb);
        if (t == 0 && wave == 0) wn = 0.0f;  // level 0
        CA[t] = wn;
        // (the coefficients of a few rows in registers at a time)
        if constexpr (!AHEAD)
          if (t % 4 == 0) __builtin_amdgcn_sched_barrier(0);
      }
    xw[lane] = wn;
  }
  pass(&back_next, wave - 1);
  // ---- acoustic_pp, the rrw accumulation, new w; CB keeps ppd, PF pp3d
#pragma unroll
  for (int t = 0; t < L; ++t)
    if (ROW(t)) {
      const uint32_t o = at(k0 + t);
      const float w0 = CA[t];
      const float w1 = t == L - 1 || (t == L - 2 && !full) ? wnext : CA[t + 1 < L ? t + 1 : t];
      float p = fma_(ac.alph, fma_(w0, PQ[t], w1 * P2Q[t]), PF[t]);
      if (ab(p) < ac.smeps) p = 0.0f;
      const float dum1 = ac.kdiv * (p - PP[t]);
      PF[t] = p;
      CB[t] = p + dum1;
      if (active) {
        pp3d.put(o, p);
        ppd.put(o, CB[t]);
        if (saveX) ppx.put(o, dum1);
        w.put(o, w0);
        rrwO.put(o, accw(RW[t] * bf, w0));
      }
    }
  // ---- the halo cells' w, ppd and pp3d, lane = column: images of the row in
  // y (dy rows away), of the column in x (dx columns), and both
  const bool lo = i >= nx - 3, hi = i <= 3;
#pragma unroll 1
  for (int q = 1; q < (OPEN ? 0 : 9); ++q) {
    const int xi = q % 3, yi = q / 3;
    const int dy = yi == 0 ? 0 : yi == 1 ? (j >= ny - 3 ? -ny : 0) : (j <= 3 ? ny : 0);
    if (yi > 0 && dy == 0) continue;
    const int dx = xi == 0 ? 0 : xi == 1 ? (lo ? -nx : hi ? nx : 0) : (lo && hi ? nx : 0);
    if (!active || (xi > 0 && dx == 0)) continue;
    const uint32_t h0 = at(k0) + (uint32_t)(4 * dx) + sjb * (uint32_t)dy;
#pragma unroll
    for (int t = 0; t < L; ++t)
      if (ROW(t)) {
        const uint32_t h = h0 + skb * (uint32_t)t;
        w.put(h, CA[t]);
        ppd.put(h, CB[t]);
        if (imgP) pp3d.put(h, PF[t]);
      }
    if (top) {
      const uint32_t h = h0 + skb * (uint32_t)Lq;
      w.put(h, 0.0f);
      ppd.put(h, ppdz);
      if (imgP) pp3d.put(h, ppz);
    }
  }
#undef ROW
}
// instantiations by levels per wave: the runtime picks the one with
// ceil(nz / AC_WAVES) levels (k_ac_column: 16)
#define AC_INST(L, name, waves) \
  __global__ __launch_bounds__(64 * AC_WAVES) __attribute__((amdgpu_waves_per_eu(waves))) void name(uint32_t* M, KArg a) { ac_column<L, false>(M, a); } \
  __global__ __launch_bounds__(64 * AC_WAVES) __attribute__((amdgpu_waves_per_eu(waves))) void name##_open(uint32_t* M, KArg a) { ac_column<L, true>(M, a); }
AC_INST(1, k_ac_column1, 4) AC_INST(2, k_ac_column2, 4) AC_INST(3, k_ac_column3, 4) AC_INST(4, k_ac_column4, 4)
AC_INST(5, k_ac_column5, 4) AC_INST(6, k_ac_column6, 4) AC_INST(7, k_ac_column7, 6) AC_INST(8, k_ac_column8, 6)
AC_INST(9, k_ac_column9, 6) AC_INST(10, k_ac_column10, 6) AC_INST(11, k_ac_column11, 6) AC_INST(12, k_ac_column12, 6)
AC_INST(13, k_ac_column13, 4) AC_INST(14, k_ac_column14, 4) AC_INST(15, k_ac_column15, 4) AC_INST(16, k_ac_column, 4)
#undef AC_INST

const void* ac_column_kernel(int levels_per_wave, bool open) {
#define E(n) {(const void*)&n, (const void*)&n##_open}
  static const void* const fns[17][2] = {{nullptr, nullptr}, E(k_ac_column1), E(k_ac_column2), E(k_ac_column3),
                                         E(k_ac_column4), E(k_ac_column5), E(k_ac_column6), E(k_ac_column7),
                                         E(k_ac_column8), E(k_ac_column9), E(k_ac_column10), E(k_ac_column11),
                                         E(k_ac_column12), E(k_ac_column13), E(k_ac_column14), E(k_ac_column15),
                                         E(k_ac_column)};
#undef E
  return levels_per_wave >= 1 && levels_per_wave <= 16 ? fns[levels_per_wave][open] : nullptr;
}

// The halo of w, ppd, rrw and, if asked for, pp3d after a substep of a domain
// with an open side: rrw accumulates the old w there (the accumulation runs
// before the fill), then w and ppd take their sources' values (k_bc_open_xy).
// p: 1 acoustic, 2 w, 3 ppd, 4 rrw, 5 the accumulated rrw, 6 pp3d, 7 -> tavg,
// 8 -> first substep of the stage (rrw starts as w * beta), 9 -> fill pp3d,
// 10 -> open x, open y.  Grid as k_bc_open_xy.
__global__ __launch_bounds__(256) void k_ac_halo_open(uint32_t* M, KArg a) {
  TE_TID3
  const Dims g = dims(a.q[0], 0);
  const int k = gy;
  if (k > g.nz) return;
  int i, j;
  if (!halo_cell_at(g, gx, i, j)) return;
  const Acoustic ac = acoustic(a.q[1], 0);
  const bool openx = ldi(a.q[10], 0) != 0, openy = ldi(a.q[10], 1) != 0, first = ldi(a.q[8], 0) != 0;
  const bool fillP = ldi(a.q[9], 0) != 0;
  const float tavg = ldf(a.q[7], 0);
  const int64_t dst = g.idx(i, j, k);
  const int64_t src = g.idx(halo_source(i, g.nx, openx, g.nx - 1), halo_source(j, g.ny, openy, g.ny - 1), k);
  float *w = fq(a.q[2]), *ppd = fq(a.q[3]), *pp3d = fq(a.q[6]);
  const float x = w[dst], y = first ? x * ac.beta : fq(a.q[4])[dst];
  const float ws = w[src], ps = ppd[src], qs = fillP ? pp3d[src] : 0.0f;
  fq(a.q[5])[dst] = tavg > 0.0f ? fma_(x, ac.alph, y) * tavg : y + x;
  if (src != dst) {
    w[dst] = ws;
    ppd[dst] = ps;
    if (fillP) pp3d[dst] = qs;
  }
}

}  // namespace te
