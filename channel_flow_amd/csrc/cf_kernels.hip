// HIP kernels of the channel-flow dual-time inner iteration (gfx950, FP64).
//
// One kernel per reference stage: ghost cells, MUSCL5+Roe fluxes per
// direction, viscous face fluxes + divergence, BDF2 right-hand side with the
// preconditioned transform, hyperplane LU-SGS sweeps, primitive update with a
// deterministic two-pass residual reduction.  Fields use the reference
// [X_np][Y_m][Z_m] indexing with a padded k pitch (Geo), metrics are
// j-profiles (they vary only with j, Jacobian*.cpp).
#include "cf_kernels.hpp"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace cf {

// ---------------------------------------------------------------------------
// ghost cells: main.cpp:203-240 (x), Y_boundary_condition.cpp:48-120 (walls),
// Z_boundary_condition.cpp:48-66 (periodic z)
// ---------------------------------------------------------------------------
// The wall ghost of the cell (is, ja, k): rho, velocities and energy of the
// mirrored state at the wall temperature, over Jb
__device__ __forceinline__ void wall_ghost(const double* __restrict__ U, const double* __restrict__ prof, const Geo& g,
                                           int is, int top, int k, double o[5]) {
  const int ja = top ? g.ny : 2, jb = top ? g.ny + 1 : 1;
  const long a = at(g, is, ja, k);
  const double Ja = pf(prof, g.Ym, SET_C, 0, ja), Jb = pf(prof, g.Ym, SET_C, 0, jb);
  const double U1 = U[a], U2 = U[g.nf + a], U3 = U[2 * g.nf + a], U4 = U[3 * g.nf + a], U5 = U[4 * g.nf + a];
  double rho = U1 * Ja;
  const double Uu = U2 / U1, V = U3 / U1, W = U4 / U1;
  const double VV = Uu * Uu + V * V + W * W;
  const double P = (U5 * Ja - 0.5 * rho * VV) * (KG - 1);
  const double temp = P / rho / RG;
  const double T = T_WALL2 - temp;
  rho = P / RG / T;
  o[0] = P / RG / T / Jb;
  o[1] = -P / RG / T * Uu / Jb;
  o[2] = -P / RG / T * V / Jb;
  o[3] = -P / RG / T * W / Jb;
  o[4] = (rho * RG * T / (KG - 1) + 0.5 * P / RG / T * VV) / Jb;
}

// All ghost cells in one launch.  The reference copies the x ghost planes,
// then forms the walls' ghosts (the x ghost planes' too), then copies the
// periodic z ghosts (the walls' too); every one of them follows from cells
// that stay as they are: plane is = src_lo, src_hi or i, column k' = nz, 2 or
// k, and at j = 1, ny + 1 the wall's mirror of (is, ., k').  Threads: the two
// x ghost planes, then the wall rows, then the z columns of the others.
// In place of three launches: 35 -> 29 us at 256x192x256, 12 -> 8 us at
// 16x12x16.
__global__ void __launch_bounds__(256) k_ghosts(double* __restrict__ U, const double* __restrict__ prof, Geo g,
                                                int src_lo, int src_hi) {
  const int Z = g.nz - 1, X = g.gend - 2;
  const long nx = 2 * g.plane, nw = (long)X * 2 * Z, nc = (long)X * (g.ny + 3) * 2;
  long t = (long)blockIdx.x * 256 + threadIdx.x;
  int i, j, k, is;
  if (t < nx) {
    const int hi = t >= g.plane;
    const long e = t - (hi ? g.plane : 0);
    i = hi ? g.gend + 1 : 2;
    is = hi ? src_hi : src_lo;
    j = (int)(e / g.Zp);
    k = (int)(e - (long)j * g.Zp);
  } else if ((t -= nx) < nw) {
    const long r = t / Z;
    k = 2 + (int)(t - r * Z);
    j = r & 1 ? g.ny + 1 : 1;
    i = is = 3 + (int)(r >> 1);
  } else if ((t -= nw) < nc) {
    const long r = t >> 1;
    k = t & 1 ? g.nz + 1 : 1;
    i = (int)(r / (g.ny + 3));
    j = (int)(r - (long)i * (g.ny + 3));
    i = is = 3 + i;
  } else {
    return;
  }
  const int ks = k == 1 ? g.nz : k == g.nz + 1 ? 2 : k;
  double o[5];
  if ((j == 1 || j == g.ny + 1) && ks >= 2 && ks <= g.nz) {
    wall_ghost(U, prof, g, is, j != 1, ks, o);
  } else {
    const long a = at(g, is, j, ks);
#pragma unroll
    for (int v = 0; v < 5; v++) o[v] = U[v * g.nf + a];
  }
  const long b = at(g, i, j, k);
#pragma unroll
  for (int v = 0; v < 5; v++) U[v * g.nf + b] = o[v];
}

// ---------------------------------------------------------------------------
// MUSCL5 + Roe fluxes
// ---------------------------------------------------------------------------
// Face f along DIR of the column (i, j, k) (the cell f along the direction):
// u[v][t] holds U_ of cells f-2 .. f+3 (t = cell - f + 2); each recipe reads
// only its own cells.  Returns the sum of the five outputs, which is NaN where
// one of them is; PLAIN as in roe_flux.
template <int DIR, bool PLAIN>
__device__ __forceinline__ double flux_face(const double (&u)[5][6], int f, int i, int j, int k,
                                            const double* __restrict__ prof, double* __restrict__ F, const Geo& g) {
  int rl = recipe_left(DIR, f, g.gend, g.ny, g.nz);
  int rr = recipe_right(DIR, f, g.gend, g.ny, g.nz);
  // 1/sum(w/J) varies with j only: with the cell's j along x and z, with the
  // face index along y
  const int rj = DIR == 1 ? f : j;
  double L[5], R[5], out[5];
  reconstruct_t(rl, u, prow(prof, g.Ym, FT_REC + 7 * DIR + rl, rj), L);
  reconstruct_t(rr, u, prow(prof, g.Ym, FT_REC + 7 * DIR + rr, rj), R);
  long o;
  int set, jp;
  if (DIR == 0) { o = at(g, f, j - 1, k - 1); set = SET_U; jp = j - 1; }
  else if (DIR == 1) { o = at(g, i - 1, f, k - 1); set = SET_V; jp = f; }
  else { o = at(g, i - 1, j - 1, f); set = SET_W; jp = j - 1; }
  double n[3] = {pf(prof, g.Ym, set, 1 + 3 * DIR, jp), pf(prof, g.Ym, set, 2 + 3 * DIR, jp),
                 pf(prof, g.Ym, set, 3 + 3 * DIR, jp)};
  double nt[4];
#pragma unroll
  for (int c = 0; c < 4; c++) nt[c] = prow(prof, g.Ym, FT_NRM + 4 * DIR + c, jp);
  double Jf = pf(prof, g.Ym, set, 0, jp);
  bool wall = DIR == 1 && (f == 1 || f == g.ny);
  const double rJf = prow(prof, g.Ym, FT_RCP + 2 * DIR, jp), rin = prow(prof, g.Ym, FT_RCP + 2 * DIR + 1, jp);
  roe_flux<PLAIN>(L, R, n, nt, Jf, rJf, rin, DIR == 1, wall, out);
#pragma unroll
  for (int v = 0; v < 5; v++) F[v * g.nf + o] = out[v];
  return out[0] + out[1] + out[2] + out[3] + out[4];
}

// v, as a value the compiler knows nothing of (uniform; per lane): what a rare
// path forms from it is not kept in registers along the usual one (Flux_X 127
// VGPRs and four waves per SIMD, 132 and three without this)
template <class T>
__device__ __forceinline__ T anew_s(T v) {
  asm volatile("" : "+s"(v));
  return v;
}
template <class T>
__device__ __forceinline__ T anew_v(T v) {
  asm volatile("" : "+v"(v));
  return v;
}

// threadIdx.y of a block 64 threads wide: one wave per row, so the value is
// uniform across the wave, and what depends on it alone (j, the grid
// profiles at j) is held in scalar registers and read with scalar loads
__device__ __forceinline__ int wave_row() { return __builtin_amdgcn_readfirstlane(threadIdx.y); }

// Flux_Z: a block of 64 faces (lanes, along k) by 4 rows j stages each row's
// cells f0-2 .. f0+66 in LDS once, and each thread reads its six stencil
// cells from there (cells beyond the row, next to the periodic seam, are
// clamped onto it; no recipe of those faces reads them)
template <int DIR>
__global__ void __launch_bounds__(256) k_flux_zs(const double* __restrict__ U, const double* __restrict__ prof,
                                                 double* __restrict__ F, Geo g) {
  static_assert(DIR == 2, "faces along k");
  __shared__ double S[4][5][72];
  const int tx = threadIdx.x, ty = wave_row();  // j's profiles in scalar registers: 80 VGPRs, six waves per SIMD
  const int f0 = 1 + blockIdx.x * 64;
  const int j = 2 + blockIdx.y * 4 + ty, i = 3 + blockIdx.z;
  const bool row = j <= g.ny;
  for (int c = tx; c < 69; c += 64) {
    const int kc = min(max(f0 - 2 + c, 0), g.Zm - 1);
    if (row) {
      const long p = at(g, i, j, kc);
#pragma unroll
      for (int v = 0; v < 5; v++) S[ty][v][c] = U[v * g.nf + p];
    }
  }
  __syncthreads();
  const int f = f0 + tx;
  if (!row || f > g.nz) return;
  double u[5][6];
  auto cells = [&](int x) {
#pragma unroll
    for (int t = 0; t < 6; t++)
#pragma unroll
      for (int v = 0; v < 5; v++) u[v][t] = S[ty][v][x + t];
  };
  cells(tx);
  const double s = flux_face<DIR, false>(u, f, i, j, f, prof, F, g);
  if (__builtin_expect(s != s, 0)) {  // with plain divisions, from the cells again
    const double* const pr = anew_s(prof);
    const int x = anew_v(tx);
    cells(x);
    flux_face<DIR, true>(u, f0 + x, i, j, f0 + x, pr, anew_s(F), g);
  }
}

// Flux_X and Flux_Y with one thread per column of faces: lanes run along k
// and each thread walks fc <= FC consecutive faces along the direction with cells
// f-2 .. f+3 in registers, loading one new cell per face (and that one a
// face ahead) where a thread per face loads up to six.  16 faces per
// thread measured faster than 8 and equal to 32 at 256x192x256.
constexpr int FC = 16;
// at least 3 waves per SIMD: x takes 127 VGPRs (4 waves), y 132 (forcing 4
// took y from 318 to 350 us)
constexpr int FLUX_COL_WAVES = 3;

template <int DIR>
__global__ void __launch_bounds__(256, FLUX_COL_WAVES) k_flux_col(const double* __restrict__ U, const double* __restrict__ prof,
                                                  double* __restrict__ F, Geo g, int fc) {
  static_assert(DIR == 0 || DIR == 1, "columns along x or y");
  // DIR 0: f in [2,gend] (i), a = j in [2,ny]; DIR 1: f in [1,ny] (j), a = i in [3,gend]
  const int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  // x: the row is j, whose profiles every face reads (a wave-uniform row
  // took the kernel from 168 to 126 VGPRs and 0.398 to 0.318 ms); y: the
  // row is i, and a uniform i measured 2% slower
  const int a = blockIdx.y * blockDim.y + (DIR == 0 ? wave_row() : (int)threadIdx.y);
  const int i = DIR == 0 ? 0 : 3 + a, j = DIR == 0 ? 2 + a : 0;
  if (k > g.nz || (DIR == 0 ? j > g.ny : i > g.gend)) return;
  const int fmin = DIR == 0 ? 2 : 1, fmax = DIR == 0 ? g.gend : g.ny;
  const int f0 = fmin + blockIdx.z * fc, f1 = min(f0 + fc - 1, fmax);
  // cells outside the array (j = -1 and j = ny + 3 next to the walls) are
  // clamped onto it; no recipe of those faces reads them
  const int cmax = DIR == 0 ? g.Xnp - 1 : g.Ym - 1;
  auto cell = [&](int c) -> long {
    c = min(max(c, 0), cmax);
    return DIR == 0 ? at(g, c, j, k) : at(g, i, c, k);
  };
  double u[5][6];
  auto cells = [&](int f) {
#pragma unroll
    for (int t = 0; t < 6; t++) {
      const long p = cell(f - 2 + t);
#pragma unroll
      for (int v = 0; v < 5; v++) u[v][t] = U[v * g.nf + p];
    }
  };
  bool again = false;
  cells(f0);
  for (int f = f0; f <= f1; f++) {
    double nx[5];
    const long p = cell(f + 4);
#pragma unroll
    for (int v = 0; v < 5; v++) nx[v] = U[v * g.nf + p];
    const double s = flux_face<DIR, false>(u, f, DIR == 0 ? f : i, DIR == 0 ? j : f, k, prof, F, g);
    again |= s != s;
#pragma unroll
    for (int v = 0; v < 5; v++) {
#pragma unroll
      for (int t = 0; t < 5; t++) u[v][t] = u[v][t + 1];
      u[v][5] = nx[v];
    }
  }
  // a NaN among the run's outputs: all of them again with plain divisions,
  // after the run, where nothing else is held in registers
  if (__builtin_expect(again, 0)) {
    const double* const pr = anew_s(prof);
    const int kk = anew_v(k);
    for (int f = f0; f <= f1; f++) {
      cells(f);
      flux_face<DIR, true>(u, f, DIR == 0 ? f : i, DIR == 0 ? j : f, kk, pr, F, g);
    }
  }
}

// ---------------------------------------------------------------------------
// limiter fluxes, one thread per face (Flux_X_limiter.cpp:104-547,
// Flux_Y_limiter.cpp:106-685, Flux_Z_limiter.cpp:113-710)
// ---------------------------------------------------------------------------
// the limiter face flux of face f along DIR of the column (i, j, k) from the
// cells f-2 .. f+3 (u, with zero outside the array) and their J (jj)
template <int DIR>
__device__ __forceinline__ void lim_face(const double (&u)[5][6], const double (&jj)[6], int f, int i, int j, int k,
                                         const double* __restrict__ Ep, const double* __restrict__ prof,
                                         double* __restrict__ F, const Geo& g) {
  long o;
  int set, jp;
  if (DIR == 0) { o = at(g, f, j - 1, k - 1); set = SET_U; jp = j - 1; }
  else if (DIR == 1) { o = at(g, i - 1, f, k - 1); set = SET_V; jp = f; }
  else { o = at(g, i - 1, j - 1, f); set = SET_W; jp = j - 1; }
  const double Jf = pf(prof, g.Ym, set, 0, jp);
  double L[5], R[5];
  if (DIR == 0) {
    // 3-point within two cells of the x ends (Flux_X_limiter.cpp:133)
    const bool l3 = f <= 3 || f >= g.gend, r3 = f + 1 <= 3 || f + 1 >= g.gend;
#pragma unroll
    for (int v = 0; v < 5; v++) {
      L[v] = (l3 ? lim3_up<1>(u[v][1], u[v][2], u[v][3]) : lim5_up<1>(u[v][0], u[v][1], u[v][2], u[v][3], u[v][4])) * Jf;
      R[v] = (r3 ? lim3_dn(u[v][2], u[v][3], u[v][4]) : lim5_dn(u[v][1], u[v][2], u[v][3], u[v][4], u[v][5])) * Jf;
    }
  } else if (DIR == 1) {
    // near-wall cells j <= 2, j >= ny-1 (Flux_Y_limiter.cpp:126); the face J
    // of the interior branch also scales ML/MR 2..5 there (the reference
    // leaves it unassigned); wall faces take J-weighted averages (:368-440)
    const bool lw = f <= 2 || f >= g.ny - 1, rw = f + 1 <= 2 || f + 1 >= g.ny - 1;
#pragma unroll
    for (int v = 0; v < 5; v++) {
      if (f == 1) {
        const double temp = 1. / (1 / jj[2] + 1 / jj[3]);
        L[v] = temp * (u[v][2] + u[v][3]);
      } else if (lw) {
        L[v] = v == 0 ? lim3y_up(u[v][1], u[v][2], u[v][3], jj[2]) : lim3_up<1>(u[v][1], u[v][2], u[v][3]) * Jf;
      } else {
        L[v] = lim5_up<1>(u[v][0], u[v][1], u[v][2], u[v][3], u[v][4]) * Jf;
      }
      if (f == g.ny) {
        const double temp = 1. / (1 / jj[2] + 1 / jj[3]);
        R[v] = temp * (u[v][2] + u[v][3]);
      } else if (rw) {
        R[v] = v == 0 ? lim3y_dn(u[v][2], u[v][3], u[v][4], jj[3]) : lim3_dn(u[v][2], u[v][3], u[v][4]) * Jf;
      } else {
        R[v] = lim5_dn(u[v][1], u[v][2], u[v][3], u[v][4], u[v][5]) * Jf;
      }
    }
  } else {
    // seam recipes (as Flux_Z.cpp) at k = 1, 2, nz; MUSCL cells k in
    // [3, nz-1] with the 3-point branch for k >= ny (Flux_Z_limiter.cpp:130,
    // B9), left state u - 0.5 phi du, face weights 1/sum(w/J) unnormalised
    const int nz = g.nz;
    if (f == 1) reconstruct(AVG, u, jj, L);
    else if (f == 2 || f == nz) reconstruct(O3L, u, jj, L);
    else {
      const int c = f;
      const bool o3 = c <= 2 || c >= g.ny;
      const double jw = o3 ? 1. / (-1 / jj[1] + 5 / jj[2] + 2 / jj[3])
                           : 1. / (2 / jj[0] - 13 / jj[1] + 47 / jj[2] + 27 / jj[3] - 3 / jj[4]);
#pragma unroll
      for (int v = 0; v < 5; v++)
        L[v] = (o3 ? lim3_up<-1>(u[v][1], u[v][2], u[v][3]) : lim5_up<-1>(u[v][0], u[v][1], u[v][2], u[v][3], u[v][4])) * jw;
    }
    if (f == 1 || f == nz - 1) reconstruct(O3R, u, jj, R);
    else if (f == nz) reconstruct(AVG, u, jj, R);
    else {
      const int c = f + 1;
      const bool o3 = c <= 2 || c >= g.ny;
      const double jw = o3 ? 1. / (2 / jj[2] + 5 / jj[3] - 1 / jj[4])
                           : 1. / (-3 / jj[1] + 27 / jj[2] + 47 / jj[3] - 13 / jj[4] + 2 / jj[5]);
#pragma unroll
      for (int v = 0; v < 5; v++)
        R[v] = (o3 ? lim3_dn(u[v][2], u[v][3], u[v][4]) : lim5_dn(u[v][1], u[v][2], u[v][3], u[v][4], u[v][5])) * jw;
    }
  }
  const double n[3] = {pf(prof, g.Ym, set, 1 + 3 * DIR, jp), pf(prof, g.Ym, set, 2 + 3 * DIR, jp),
                       pf(prof, g.Ym, set, 3 + 3 * DIR, jp)};
  const double e = Ep[o];
  double out[5], fav3, psum;
  limiter_face_flux(L, R, n, Jf, e, out, &fav3, &psum);
  if (DIR == 1 && (f == 1 || f == g.ny)) {
    // wall faces (Flux_Y_limiter.cpp:658-666)
    out[0] = 0;
    out[1] = 0;
    out[2] = 0.5 * (n[1] * psum - e * fav3) / Jf;
    out[3] = 0;
    out[4] = 0;
  }
#pragma unroll
  for (int v = 0; v < 5; v++) F[v * g.nf + o] = out[v];
}


template <int DIR>
__global__ void __launch_bounds__(256) k_flux_lim(const double* __restrict__ U, const double* __restrict__ Ep,
                                                  const double* __restrict__ prof, double* __restrict__ F, Geo g) {
  // one thread per face.  DIR 0: f in [2,gend] (i), j in [2,ny], k in
  // [2,nz]; DIR 1: f in [1,ny] (j), i in [3,gend], k in [2,nz]; DIR 2: f in
  // [1,nz] (k), i in [3,gend], j in [2,ny] (the lanes run along k, for
  // Flux_Z the direction itself)
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int y = blockIdx.y * blockDim.y + threadIdx.y;
  int z = blockIdx.z;
  int f, i, j, k;
  if (DIR == 0) { k = 2 + x; j = 2 + y; f = 2 + z; i = f; if (k > g.nz || j > g.ny) return; }
  else if (DIR == 1) { k = 2 + x; f = 1 + y; i = 3 + z; j = f; if (k > g.nz || f > g.ny) return; }
  else { f = 1 + x; j = 2 + y; i = 3 + z; k = f; if (f > g.nz || j > g.ny) return; }
  const long stride = DIR == 0 ? g.plane : (DIR == 1 ? (long)g.Zp : 1L);
  const long base = at(g, i, j, k);  // cell f along the direction
  // cells f-2 .. f+3 (t = 0..5); ghosts the reference never fills are zero
  double u[5][6], jj[6];
#pragma unroll
  for (int t = 0; t < 6; t++) {
    const int c = f + t - 2;
    const bool in = DIR == 0 ? (c >= 0 && c < g.Xnp) : (DIR == 1 ? (c >= 0 && c < g.Ym) : (c >= 0 && c < g.Zm));
    const long p = base + (long)(t - 2) * stride;
    jj[t] = pf(prof, g.Ym, SET_C, 0, DIR == 1 ? min(max(c, 0), g.Ym - 1) : j);
#pragma unroll
    for (int v = 0; v < 5; v++) u[v][t] = in ? U[v * g.nf + p] : 0.0;
  }
  lim_face<DIR>(u, jj, f, i, j, k, Ep, prof, F, g);
}

// cell c along DIR of the column as the limiter fluxes read it: U_, or zero
// outside the array (ghosts the reference never fills), and its J
template <int DIR>
__device__ __forceinline__ void lim_cell(const double* __restrict__ U, const double* __restrict__ prof, const Geo& g,
                                         int c, int i, int j, int k, double (&u)[5][6], double (&jj)[6], int t) {
  const bool in = DIR == 0 ? (c >= 0 && c < g.Xnp) : (DIR == 1 ? (c >= 0 && c < g.Ym) : (c >= 0 && c < g.Zm));
  const int cc = DIR == 0 ? min(max(c, 0), g.Xnp - 1) : (DIR == 1 ? min(max(c, 0), g.Ym - 1) : min(max(c, 0), g.Zm - 1));
  const long p = DIR == 0 ? at(g, cc, j, k) : (DIR == 1 ? at(g, i, cc, k) : at(g, i, j, cc));
  jj[t] = pf(prof, g.Ym, SET_C, 0, DIR == 1 ? cc : j);
#pragma unroll
  for (int v = 0; v < 5; v++) u[v][t] = in ? U[v * g.nf + p] : 0.0;
}

// Flux_X/Y_limiter by columns of FC faces, as k_flux_col (2 waves per SIMD:
// the limiter face needs more registers than the Roe face)
template <int DIR>
__global__ void __launch_bounds__(256, 2) k_flux_lim_col(const double* __restrict__ U,
                                                                         const double* __restrict__ Ep,
                                                                         const double* __restrict__ prof,
                                                                         double* __restrict__ F, Geo g, int fc) {
  static_assert(DIR == 0 || DIR == 1, "columns along x or y");
  const int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  const int a = blockIdx.y * blockDim.y + (DIR == 0 ? wave_row() : (int)threadIdx.y);
  const int i = DIR == 0 ? 0 : 3 + a, j = DIR == 0 ? 2 + a : 0;
  if (k > g.nz || (DIR == 0 ? j > g.ny : i > g.gend)) return;
  const int fmin = DIR == 0 ? 2 : 1, fmax = DIR == 0 ? g.gend : g.ny;
  const int f0 = fmin + blockIdx.z * fc, f1 = min(f0 + fc - 1, fmax);
  double u[5][6], jj[6];
#pragma unroll
  for (int t = 0; t < 6; t++) lim_cell<DIR>(U, prof, g, f0 - 2 + t, i, j, k, u, jj, t);
  for (int f = f0; f <= f1; f++) {
    double nu[5][6], nj[6];
    lim_cell<DIR>(U, prof, g, f + 4, i, j, k, nu, nj, 0);
    lim_face<DIR>(u, jj, f, DIR == 0 ? f : i, DIR == 0 ? j : f, k, Ep, prof, F, g);
#pragma unroll
    for (int t = 0; t < 5; t++) {
      jj[t] = jj[t + 1];
#pragma unroll
      for (int v = 0; v < 5; v++) u[v][t] = u[v][t + 1];
    }
    jj[5] = nj[0];
#pragma unroll
    for (int v = 0; v < 5; v++) u[v][5] = nu[v][0];
  }
}

// ---------------------------------------------------------------------------
// ADM sensor (Filter.cpp:12-1720): two chains (h, 2h) of six separable
// 3-point filter passes over the interior box on rho and the momenta; every
// value read outside the box is U_'s own (the reference's work arrays start
// as copies of U_ and no pass writes outside the box).
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool in_box(const Geo& g, int i, int j, int k) {
  return i >= 3 && i <= g.gend && j >= 2 && j <= g.ny && k >= 2 && k <= g.nz;
}

// One filter pass (x, then y, then z, Filter.cpp:218-775) in one kernel: a
// block owns an 8 (j) x 32 (k) tile and marches through FI planes i.  Each
// thread keeps its (at most two) tile-and-rim positions' values at planes
// i-1, i, i+1 in registers and loads plane i+2 while plane i is filtered,
// so every plane is read once per block.  Gx of the tile and of a one-cell
// rim, and Gy of the tile rows and rim columns, stay in LDS; a rim position
// outside the filter box holds U_'s own value there, and the x filter reads
// U_'s planes next to the box, as the reference's passes read them (their
// work arrays start as copies of U_ and no pass writes outside the box).
// Each 1-D filter keeps the reference's operands and order, so the three
// fused passes give the same bits.  Passes 1-5 store their result G_p.  The
// sixth forms the filtered state 6 G1 - 15 G2 + 20 G3 - 15 G4 + 6 G5 - G6
// from the stored ones, accumulated in the reference's order
// (Filter.cpp:222-775), and from it the energy E = |u - u_f|^2
// (Filter.cpp:790-800, 1465-1475).
// 8 planes per block measured fastest (1, 4, 16, 32: 5.28, 4.55, 4.78,
// 5.35 ms against 4.53 ms for the whole Filter at 256x192x256)
constexpr int FJ = 8, FK = 32, FI = 8;  // FI planes per block
constexpr int FNP = (FJ + 2) * (FK + 2);  // tile and rim positions of a plane
static_assert(FNP <= 512 && FJ * FK == 256, "two rim positions per thread, one tile cell per thread");

struct FiltHist {
  const double* G[5];  // G1..G5, 4 fields each
};

// field v at plane ii of a rim position (offset pp within a plane) as the x
// filter reads it: the pass input inside the box, U_ outside it
__device__ __forceinline__ double filt_x_in(const double* __restrict__ src, const double* __restrict__ U, bool box,
                                            long pp, int ii, int v, const Geo& g) {
  const double* base = (box && ii >= 3 && ii <= g.gend) ? src : U;
  return base[v * g.nf + (long)ii * g.plane + pp];
}

template <int WIDE, bool LAST>
__global__ void __launch_bounds__(256) k_filt_pass(const double* __restrict__ src, const double* __restrict__ U,
                                                   const double* __restrict__ prof, const double* __restrict__ Yp,
                                                   double* __restrict__ G, FiltHist hist, double* __restrict__ E,
                                                   Geo g) {
  __shared__ double Lx[4][FJ + 2][FK + 2];  // rows j0-1 .. j0+FJ, columns k0-1 .. k0+FK
  __shared__ double Ly[4][FJ][FK + 2];      // rows j0 .. j0+FJ-1
  const int k0 = 2 + blockIdx.x * FK, j0 = 2 + blockIdx.y * FJ;
  const int i0 = 3 + blockIdx.z * FI, i1 = min(i0 + FI, g.gend + 1);  // planes i0 .. i1-1
  const int tid = threadIdx.x;
  const long nf = g.nf;
  // this thread's rim positions: row, column, offset within a plane, whether
  // the position exists and whether it is inside the box (in j and k; every
  // plane of the block is inside in i)
  int pr[2], pc[2];
  long pp[2];
  bool pv[2], pb[2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const int idx = tid + 256 * q;
    pr[q] = idx / (FK + 2);
    pc[q] = idx - pr[q] * (FK + 2);
    const int j = j0 - 1 + pr[q], k = k0 - 1 + pc[q];
    pv[q] = idx < FNP && j <= g.ny + 1 && k <= g.nz + 1;
    pb[q] = pv[q] && j >= 2 && j <= g.ny && k >= 2 && k <= g.nz;
    pp[q] = pv[q] ? at(g, 0, j, k) : 0;
  }
  double w[2][3][4];  // planes i-1, i, i+1
#pragma unroll
  for (int q = 0; q < 2; q++)
    if (pv[q])
#pragma unroll
      for (int s = 0; s < 3; s++)
#pragma unroll
        for (int v = 0; v < 4; v++) w[q][s][v] = filt_x_in(src, U, pb[q], pp[q], i0 - 1 + s, v, g);
  for (int i = i0; i < i1; i++) {
    // plane i+2 for the next plane's x filter, in flight during this one
    double nx[2][4];
    const bool more = i + 1 < i1;
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int v = 0; v < 4; v++) nx[q][v] = (pv[q] && more) ? filt_x_in(src, U, pb[q], pp[q], i + 2, v, g) : 0.0;
#pragma unroll
    for (int q = 0; q < 2; q++) {
      if (!pv[q]) continue;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const double a = w[q][0][v], b = w[q][1][v], cc = w[q][2][v];
        Lx[v][pr[q]][pc[q]] = !pb[q] ? b : (WIDE ? 0.25 * (a + 2 * b + cc) : 0.125 * (a + 6 * b + cc));
      }
    }
    __syncthreads();
    for (int idx = tid; idx < FJ * (FK + 2); idx += 256) {
      const int r = idx / (FK + 2), c = idx - r * (FK + 2);
      const int j = j0 + r, k = k0 - 1 + c;
      if (j > g.ny + 1 || k > g.nz + 1) continue;
      if (in_box(g, i, j, k)) {
        const double A = Yp[j + 1] - Yp[j - 1];  // H_L + H_R
        const double B = Yp[j + 1] - Yp[j];      // H_R
        const double C = Yp[j] - Yp[j - 1];      // H_L
        const double Jm = pf(prof, g.Ym, SET_C, 0, j - 1), J0 = pf(prof, g.Ym, SET_C, 0, j),
                     Jp = pf(prof, g.Ym, SET_C, 0, j + 1);
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const double gm = Lx[v][r][c], gx = Lx[v][r + 1][c], gp = Lx[v][r + 2][c];
          Ly[v][r][c] = WIDE ? 0.5 * (B / A * gm * Jm + gx * J0 + C / A * gp * Jp) / J0
                             : 0.125 * (2 * B / A * gm * Jm + 6 * gx * J0 + 2 * C / A * gp * Jp) / J0;
        }
      } else {
        // outside the box: U_'s own value, which the x step left in Lx
#pragma unroll
        for (int v = 0; v < 4; v++) Ly[v][r][c] = Lx[v][r + 1][c];
      }
    }
    __syncthreads();
    {
      const int r = tid / FK, c = tid - r * FK;  // 256 threads = the FJ x FK tile
      const int j = j0 + r, k = k0 + c;
      if (j <= g.ny && k <= g.nz) {
        const long p = at(g, i, j, k);
        double f[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const double a = Ly[v][r][c], y = Ly[v][r][c + 1], cc = Ly[v][r][c + 2];
          const double t = WIDE ? 0.25 * (a + 2 * y + cc) : 0.125 * (a + 6 * y + cc);
          if (LAST) {
            const long o = v * nf + p;
            double s = 6 * hist.G[0][o];
            s = s - 15 * hist.G[1][o];
            s = s + 20 * hist.G[2][o];
            s = s - 15 * hist.G[3][o];
            s = s + 6 * hist.G[4][o];
            f[v] = s - t;
          } else {
            G[v * nf + p] = t;
          }
        }
        if (LAST) {
          const double Ue = U[nf + p] / U[p] - f[1] / f[0];
          const double Ve = U[2 * nf + p] / U[p] - f[2] / f[0];
          const double We = U[3 * nf + p] / U[p] - f[3] / f[0];
          E[p] = Ue * Ue + Ve * Ve + We * We;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        w[q][0][v] = w[q][1][v];
        w[q][1][v] = w[q][2][v];
        w[q][2][v] = nx[q][v];
      }
  }
}

// E at a cell of the sensor stencils: the planes next to the box copy the
// box's first/last cells (Filter.cpp:1490-1540)
__device__ __forceinline__ double e_at(const double* __restrict__ E, const Geo& g, int i, int j, int k) {
  i = min(max(i, 3), g.gend);
  j = min(max(j, 2), g.ny);
  k = min(max(k, 2), g.nz);
  return E[at(g, i, j, k)];
}

// sensors on the face layouts (Filter.cpp:1550-1645); a 0/0 ratio compares
// false and gives E_low
template <int DIR>
__global__ void __launch_bounds__(256) k_filt_sensor(const double* __restrict__ Eh, const double* __restrict__ E2h,
                                                     double crit, double E_high, double E_low,
                                                     double* __restrict__ Ep, Geo g) {
  const int k = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  const int i = 2 + blockIdx.z;
  if (DIR == 0 && (k >= g.nz || j >= g.ny || i > g.gend)) return;
  if (DIR == 1 && (k >= g.nz || j > g.ny || i > g.gend - 1)) return;
  if (DIR == 2 && (k > g.nz || j >= g.ny || i > g.gend - 1)) return;
  double r;
  if (DIR == 0)
    r = (e_at(Eh, g, i, j + 1, k + 1) + e_at(Eh, g, i + 1, j + 1, k + 1)) /
        (e_at(E2h, g, i, j + 1, k + 1) + e_at(E2h, g, i + 1, j + 1, k + 1));
  else if (DIR == 1)
    r = (e_at(Eh, g, i + 1, j, k + 1) + e_at(Eh, g, i + 1, j + 1, k + 1)) /
        (e_at(E2h, g, i + 1, j, k + 1) + e_at(E2h, g, i + 1, j + 1, k + 1));
  else
    r = (e_at(Eh, g, i + 1, j + 1, k) + e_at(Eh, g, i + 1, j + 1, k + 1)) /
        (e_at(E2h, g, i + 1, j + 1, k) + e_at(E2h, g, i + 1, j + 1, k + 1));
  Ep[at(g, i, j, k)] = r >= crit ? E_high : E_low;
}

// ---------------------------------------------------------------------------
// viscous terms: primitives on the stencil box, face fluxes, divergence
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_visc_prim(const double* __restrict__ U, const double* __restrict__ prof,
                                                   double* __restrict__ Pr, Geo g) {
  // box i in [2,gend+1], j in [1,ny+1], k in [1,nz+1]
  int k = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  int j = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  int i = 2 + blockIdx.z;
  if (k > g.nz + 1 || j > g.ny + 1) return;
  long p = at(g, i, j, k);
  Prim q = prim_visc(U[p], U[g.nf + p], U[2 * g.nf + p], U[3 * g.nf + p], U[4 * g.nf + p],
                     pf(prof, g.Ym, SET_C, 0, j));
  Pr[p] = q.U;
  Pr[g.nf + p] = q.V;
  Pr[2 * g.nf + p] = q.W;
  Pr[3 * g.nf + p] = q.T;
}

__device__ __forceinline__ Prim ldp(const double* __restrict__ Pr, long nf, long p) {
  Prim q;
  q.U = Pr[p];
  q.V = Pr[nf + p];
  q.W = Pr[2 * nf + p];
  q.T = Pr[3 * nf + p];
  return q;
}

__device__ __forceinline__ void face_metric(const double* __restrict__ prof, int Ym, int set, int j, double m[9]) {
#pragma unroll
  for (int c = 0; c < 9; c++) m[c] = pf(prof, Ym, set, 1 + c, j);
}

__global__ void __launch_bounds__(256) k_visc_faces(const double* __restrict__ Pr, const double* __restrict__ prof,
                                                    double* __restrict__ VS, Geo g, double invXI, double invET,
                                                    double invZT, double inv4XI, double inv4ET, double inv4ZT) {
  // cell (i,j,k) owns the x face (i-1,i), y face (j-1,j), z face (k-1,k);
  // i in [3,gend+1], j in [2,ny+1], k in [2,nz+1]
  int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  int j = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  int i = 3 + blockIdx.z;
  if (k > g.nz + 1 || j > g.ny + 1) return;
  const long nf = g.nf, sI = g.plane, sJ = g.Zp;
  long c = at(g, i, j, k);
  Prim P0 = ldp(Pr, nf, c);
  double m[9], o[4];
  Coef q;
  if (j <= g.ny && k <= g.nz) {
    Prim iP = ldp(Pr, nf, c - sI);
    DSet dx = d_two(P0, iP, invXI);
    DSet dy = d_four(ldp(Pr, nf, c + sJ), ldp(Pr, nf, c - sI + sJ), ldp(Pr, nf, c - sJ), ldp(Pr, nf, c - sI - sJ), inv4ET);
    DSet dz = d_four(ldp(Pr, nf, c + 1), ldp(Pr, nf, c - sI + 1), ldp(Pr, nf, c - 1), ldp(Pr, nf, c - sI - 1), inv4ZT);
    face_metric(prof, g.Ym, SET_U, j - 1, m);
    coefs(m, q);
    visc_flux_x(q, dx, dy, dz, 0.5 * (P0.U + iP.U), 0.5 * (P0.V + iP.V), 0.5 * (P0.W + iP.W),
                pf(prof, g.Ym, SET_U, 0, j - 1), o);
#pragma unroll
    for (int v = 0; v < 4; v++) VS[v * nf + c] = o[v];
  }
  if (i <= g.gend && k <= g.nz) {
    Prim jP = ldp(Pr, nf, c - sJ);
    DSet dx = d_four(ldp(Pr, nf, c + sI), ldp(Pr, nf, c + sI - sJ), ldp(Pr, nf, c - sI), ldp(Pr, nf, c - sI - sJ), inv4XI);
    DSet dy = d_two(P0, jP, invET);
    DSet dz = d_four(ldp(Pr, nf, c + 1), ldp(Pr, nf, c - sJ + 1), ldp(Pr, nf, c - 1), ldp(Pr, nf, c - sJ - 1), inv4ZT);
    face_metric(prof, g.Ym, SET_V, j - 1, m);
    coefs(m, q);
    visc_flux_y(q, dx, dy, dz, 0.5 * (P0.U + jP.U), 0.5 * (P0.V + jP.V), 0.5 * (P0.W + jP.W),
                pf(prof, g.Ym, SET_V, 0, j - 1), o);
#pragma unroll
    for (int v = 0; v < 4; v++) VS[(4 + v) * nf + c] = o[v];
  }
  if (i <= g.gend && j <= g.ny) {
    Prim kP = ldp(Pr, nf, c - 1);
    Prim Pj = ldp(Pr, nf, c + sJ), kPj = ldp(Pr, nf, c + sJ - 1), jP = ldp(Pr, nf, c - sJ),
         jkP = ldp(Pr, nf, c - sJ - 1), iPj = ldp(Pr, nf, c - sI + sJ);
    DSet dx = d_four(ldp(Pr, nf, c + sI), ldp(Pr, nf, c + sI - 1), ldp(Pr, nf, c - sI), ldp(Pr, nf, c - sI - 1), inv4XI);
    DSet dy = d_four(Pj, kPj, jP, jkP, inv4ET);
    // Viscous_terms.cpp:728-730: the second uv/vw/uw product takes V or W of (i-1,j+1)
    dy.uv = (Pj.U * Pj.V + kPj.U * iPj.V - jP.U * jP.V - jkP.U * jkP.V) * inv4ET;
    dy.vw = (Pj.V * Pj.W + kPj.V * iPj.W - jP.V * jP.W - jkP.V * jkP.W) * inv4ET;
    dy.uw = (Pj.U * Pj.W + kPj.U * iPj.W - jP.U * jP.W - jkP.U * jkP.W) * inv4ET;
    DSet dz = d_two(P0, kP, invZT);
    face_metric(prof, g.Ym, SET_W, j - 1, m);
    coefs(m, q);
    visc_flux_z(q, dx, dy, dz, 0.5 * (P0.U + kP.U), 0.5 * (P0.V + kP.V), 0.5 * (P0.W + kP.W),
                pf(prof, g.Ym, SET_W, 0, j - 1), o);
#pragma unroll
    for (int v = 0; v < 4; v++) VS[(8 + v) * nf + c] = o[v];
  }
}

__global__ void __launch_bounds__(256) k_visc_div(const double* __restrict__ VS, double* __restrict__ vF, Geo g,
                                                  double invXI, double invET, double invZT) {
  int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  int j = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  int i = 3 + blockIdx.z;
  if (k > g.nz || j > g.ny) return;
  const long nf = g.nf;
  long c = at(g, i, j, k);
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const double* LL = VS + v * nf;
    const double* ML = VS + (4 + v) * nf;
    const double* NL = VS + (8 + v) * nf;
    vF[v * nf + c] = (LL[c + g.plane] - LL[c]) * invXI + (ML[c + g.Zp] - ML[c]) * invET + (NL[c + 1] - NL[c]) * invZT;
  }
}

// Fused viscous terms for diagonal metrics.  One block owns a VJ (j) x VK (k) tile of cells and a
// run of vc planes in i (at most VC).  The primitives of three consecutive planes, with a
// one-cell rim in j and k, live in LDS.  Each of the VJ*VK main threads
// computes the x face above its cell and the y and z faces below it; a
// fifth wave computes the tile's extra y-face row (j0+VJ) and z-face column
// (k0+VK).  The x face below a cell is the one computed at the previous
// plane.  The face arithmetic and the divergence are those of k_visc_faces
// and k_visc_div, operand for operand, so vF is unchanged bit for bit while
// the primitives and the twelve face-flux fields never reach HBM.  Each
// thread holds the raw U_ of plane i+1 in registers while plane i's faces are
// formed (0.638 -> 0.55 ms at 256x192x256; at 166 VGPRs before the face
// metrics moved to LDS it cost a block per CU and gained nothing).
constexpr int VJ = 8, VK = 32, VC = 16, VR = VJ + 2, VKK = VK + 2, VTHREADS = VJ * VK + 64;

struct VLds {
  double P[3][4][VR][VKK];
  double ML[4][VJ + 1][VK];
  double NL[4][VJ][VK + 1];
  double PJ[3][5][VJ + 1];  // face sets U, V, W: xidx, etdy, ztdz, J and 1 / J at j - 1, row j - j0
};

__device__ __forceinline__ Prim vp(const VLds& L, int s, int r, int c) {
  Prim q;
  q.U = L.P[s][0][r][c];
  q.V = L.P[s][1][r][c];
  q.W = L.P[s][2][r][c];
  q.T = L.P[s][3][r][c];
  return q;
}

// raw U_ and J of the rim tile's cells tid and tid + VTHREADS of one plane
// (VR * VKK <= 2 * VTHREADS), fetched a plane ahead so that the loads are in
// flight while the faces of the current plane are formed
static_assert(VR * VKK <= 2 * VTHREADS, "two rim cells per thread");
struct VRaw {
  double u[2][5];
  double J[2];
};

__device__ __forceinline__ void vfetch(VRaw& R, const double* __restrict__ U, const double* __restrict__ prof,
                                       const Geo& g, int ip, int j0, int k0, int tid) {
#pragma unroll
  for (int m = 0; m < 2; m++) {
    const int idx = tid + m * VTHREADS;
    if (idx >= VR * VKK) continue;
    const int r = idx / VKK, c = idx - r * VKK;
    const int jj = j0 - 1 + r, kk = k0 - 1 + c;
    if (jj <= g.ny + 1 && kk <= g.nz + 1) {
      const long p = at(g, ip, jj, kk);
#pragma unroll
      for (int v = 0; v < 5; v++) R.u[m][v] = U[v * g.nf + p];
      R.J[m] = pf(prof, g.Ym, SET_C, 0, jj);
    }
  }
}

__device__ __forceinline__ void vstore(VLds& L, const VRaw& R, const Geo& g, int s, int j0, int k0, int tid) {
#pragma unroll
  for (int m = 0; m < 2; m++) {
    const int idx = tid + m * VTHREADS;
    if (idx >= VR * VKK) continue;
    const int r = idx / VKK, c = idx - r * VKK;
    const int jj = j0 - 1 + r, kk = k0 - 1 + c;
    Prim q{0., 0., 0., 0.};
    if (jj <= g.ny + 1 && kk <= g.nz + 1) q = prim_visc(R.u[m][0], R.u[m][1], R.u[m][2], R.u[m][3], R.u[m][4], R.J[m]);
    L.P[s][0][r][c] = q.U;
    L.P[s][1][r][c] = q.V;
    L.P[s][2][r][c] = q.W;
    L.P[s][3][r][c] = q.T;
  }
}

// The three faces for diagonal metrics (xidy = xidz = etdx = etdz = ztdx =
// ztdy = 0 in every face set).  Of the coefficient groups a..f of
// Viscous_terms.cpp:471-526 only a1..a4, b1..b4, c1..c4, d5, d7, e6, e9, f8
// and f10 are then non-zero; the fluxes of Viscous_terms.cpp:533-547,
// 681-695 and 827-841 keep their remaining terms in the reference's order, so
// each result differs from the full sum at most in the sign of a zero.  Each
// face needs only the tangential derivatives that meet a non-zero
// coefficient, which is also why the B6 typo (it alters dy.uv, dy.vw, dy.uw
// of the z face) does not reach the z-face fluxes.
struct DiagCoef {
  double X, E, Z;  // xidx, etdy, ztdz of the face set
};

__device__ __forceinline__ double lp(const VLds& L, int s, int f, int r, int c) { return L.P[s][f][r][c]; }

// the four fluxes of a face over its J (rJ = RN(1/Jf)); where one is NaN, by
// plain divisions: div_rn's bits end where an operand is infinite or zero.
// (The check takes the kernel from 467 to 481 us at 256x192x256; one check a
// plane, with the faces formed again by a second copy of their code, 529.)
__device__ __forceinline__ void over_face_J(double o[4], double Jf, double rJ) {
  double q[4], s = 0.0;
#pragma unroll
  for (int v = 0; v < 4; v++) s += q[v] = div_rn(o[v], Jf, rJ);
  if (__builtin_expect(s != s, 0)) {
#pragma unroll
    for (int v = 0; v < 4; v++) q[v] = o[v] / Jf;
  }
#pragma unroll
  for (int v = 0; v < 4; v++) o[v] = q[v];
}

// x face between planes (slot sm) and (slot s0) at LDS cell (r, c); the
// face metrics of LDS row r are L.PJ[.][.][r - 1]
__device__ __forceinline__ void vface_x(const VLds& L, int s0, int sm, int r, int c, double invXI, double inv4ET,
                                        double inv4ZT, double o[4]) {
  const Prim P0 = vp(L, s0, r, c), iP = vp(L, sm, r, c);
  const DSet dx = d_two(P0, iP, invXI);
  const double dyu = (lp(L, s0, 0, r + 1, c) + lp(L, sm, 0, r + 1, c) - lp(L, s0, 0, r - 1, c) - lp(L, sm, 0, r - 1, c)) * inv4ET;
  const double dyv = (lp(L, s0, 1, r + 1, c) + lp(L, sm, 1, r + 1, c) - lp(L, s0, 1, r - 1, c) - lp(L, sm, 1, r - 1, c)) * inv4ET;
  const double dzu = (lp(L, s0, 0, r, c + 1) + lp(L, sm, 0, r, c + 1) - lp(L, s0, 0, r, c - 1) - lp(L, sm, 0, r, c - 1)) * inv4ZT;
  const double dzw = (lp(L, s0, 2, r, c + 1) + lp(L, sm, 2, r, c + 1) - lp(L, s0, 2, r, c - 1) - lp(L, sm, 2, r, c - 1)) * inv4ZT;
  const DiagCoef m{L.PJ[0][0][r - 1], L.PJ[0][1][r - 1], L.PJ[0][2][r - 1]};
  const double Jf = L.PJ[0][3][r - 1], rJ = L.PJ[0][4][r - 1];
  const double a1 = (4. / 3) * m.X * m.X, a2 = m.X * m.X, a3 = m.X * m.X, a4 = m.X * m.X;
  const double d5 = m.X * m.E, d7 = -((2. / 3) * m.X * m.E);
  const double e6 = m.X * m.Z, e9 = -((2. / 3) * m.X * m.Z);
  const double Ux = 0.5 * (P0.U + iP.U), Vx = 0.5 * (P0.V + iP.V), Wx = 0.5 * (P0.W + iP.W);
  o[0] = MU_L * (a1 * dx.u + d7 * dyv + e9 * dzw);
  o[1] = MU_L * (a2 * dx.v + d5 * dyu);
  o[2] = MU_L * (a3 * dx.w + e6 * dzu);
  o[3] = MU_L * (0.5 * a1 * dx.uu + 0.5 * a2 * dx.vv + 0.5 * a3 * dx.ww + CF_CVK_PR(a4, dx.T) + d5 * Vx * dyu +
                 d7 * Ux * dyv + e6 * Wx * dzu + e9 * Ux * dzw);
  over_face_J(o, Jf, rJ);
}

// y face between rows r-1 and r of plane slot s0
__device__ __forceinline__ void vface_y(const VLds& L, int sp, int s0, int sm, int r, int c, double invET,
                                        double inv4XI, double inv4ZT, double o[4]) {
  const Prim P0 = vp(L, s0, r, c), jP = vp(L, s0, r - 1, c);
  const DSet dy = d_two(P0, jP, invET);
  const double dxu = (lp(L, sp, 0, r, c) + lp(L, sp, 0, r - 1, c) - lp(L, sm, 0, r, c) - lp(L, sm, 0, r - 1, c)) * inv4XI;
  const double dxv = (lp(L, sp, 1, r, c) + lp(L, sp, 1, r - 1, c) - lp(L, sm, 1, r, c) - lp(L, sm, 1, r - 1, c)) * inv4XI;
  const double dzv = (lp(L, s0, 1, r, c + 1) + lp(L, s0, 1, r - 1, c + 1) - lp(L, s0, 1, r, c - 1) - lp(L, s0, 1, r - 1, c - 1)) * inv4ZT;
  const double dzw = (lp(L, s0, 2, r, c + 1) + lp(L, s0, 2, r - 1, c + 1) - lp(L, s0, 2, r, c - 1) - lp(L, s0, 2, r - 1, c - 1)) * inv4ZT;
  const DiagCoef m{L.PJ[1][0][r - 1], L.PJ[1][1][r - 1], L.PJ[1][2][r - 1]};
  const double Jf = L.PJ[1][3][r - 1], rJ = L.PJ[1][4][r - 1];
  const double b1 = m.E * m.E, b2 = (4. / 3) * m.E * m.E, b3 = m.E * m.E, b4 = m.E * m.E;
  const double d5 = m.X * m.E, d7 = -((2. / 3) * m.X * m.E);
  const double f8 = m.E * m.Z, f10 = -((2. / 3) * m.E * m.Z);
  const double Uy = 0.5 * (P0.U + jP.U), Vy = 0.5 * (P0.V + jP.V), Wy = 0.5 * (P0.W + jP.W);
  o[0] = MU_L * (d5 * dxv + b1 * dy.u);
  o[1] = MU_L * (d7 * dxu + b2 * dy.v + f10 * dzw);
  o[2] = MU_L * (b3 * dy.w + f8 * dzv);
  o[3] = MU_L * (0.5 * b1 * dy.uu + 0.5 * b2 * dy.vv + 0.5 * b3 * dy.ww + CF_CVK_PR(b4, dy.T) + d5 * Uy * dxv +
                 d7 * Vy * dxu + f8 * Wy * dzv + f10 * Vy * dzw);
  over_face_J(o, Jf, rJ);
}

// z face between columns c-1 and c of plane slot s0
__device__ __forceinline__ void vface_z(const VLds& L, int sp, int s0, int sm, int r, int c, double invZT,
                                        double inv4XI, double inv4ET, double o[4]) {
  const Prim P0 = vp(L, s0, r, c), kP = vp(L, s0, r, c - 1);
  const DSet dz = d_two(P0, kP, invZT);
  const double dxu = (lp(L, sp, 0, r, c) + lp(L, sp, 0, r, c - 1) - lp(L, sm, 0, r, c) - lp(L, sm, 0, r, c - 1)) * inv4XI;
  const double dxw = (lp(L, sp, 2, r, c) + lp(L, sp, 2, r, c - 1) - lp(L, sm, 2, r, c) - lp(L, sm, 2, r, c - 1)) * inv4XI;
  const double dyv = (lp(L, s0, 1, r + 1, c) + lp(L, s0, 1, r + 1, c - 1) - lp(L, s0, 1, r - 1, c) - lp(L, s0, 1, r - 1, c - 1)) * inv4ET;
  const double dyw = (lp(L, s0, 2, r + 1, c) + lp(L, s0, 2, r + 1, c - 1) - lp(L, s0, 2, r - 1, c) - lp(L, s0, 2, r - 1, c - 1)) * inv4ET;
  const DiagCoef m{L.PJ[2][0][r - 1], L.PJ[2][1][r - 1], L.PJ[2][2][r - 1]};
  const double Jf = L.PJ[2][3][r - 1], rJ = L.PJ[2][4][r - 1];
  const double c1 = m.Z * m.Z, c2 = m.Z * m.Z, c3 = (4. / 3) * m.Z * m.Z, c4 = m.Z * m.Z;
  const double e6 = m.X * m.Z, e9 = -((2. / 3) * m.X * m.Z);
  const double f8 = m.E * m.Z, f10 = -((2. / 3) * m.E * m.Z);
  const double Uz = 0.5 * (P0.U + kP.U), Vz = 0.5 * (P0.V + kP.V), Wz = 0.5 * (P0.W + kP.W);
  o[0] = MU_L * (e6 * dxw + c1 * dz.u);
  o[1] = MU_L * (f8 * dyw + c2 * dz.v);
  o[2] = MU_L * (e9 * dxu + f10 * dyv + c3 * dz.w);
  o[3] = MU_L * (0.5 * c1 * dz.uu + 0.5 * c2 * dz.vv + 0.5 * c3 * dz.ww + CF_CVK_PR(c4, dz.T) + e6 * Uz * dxw +
                 e9 * Wz * dxu + f8 * Vz * dyw + f10 * Wz * dyv);
  over_face_J(o, Jf, rJ);
}

__global__ void __launch_bounds__(VTHREADS) k_visc_fused(const double* __restrict__ U,
                                                         const double* __restrict__ prof, double* __restrict__ vF,
                                                         Geo g, int vc, double invXI, double invET, double invZT,
                                                         double inv4XI, double inv4ET, double inv4ZT) {
  __shared__ VLds L;
  const int tid = threadIdx.x;
  const int k0 = 2 + blockIdx.x * VK, j0 = 2 + blockIdx.y * VJ;
  const int ib = 3 + blockIdx.z * vc, ie = min(ib + vc - 1, g.gend);
  const bool main_t = tid < VJ * VK;
  const int ty = main_t ? tid / VK : 0, tx = main_t ? tid % VK : 0;
  const int j = j0 + ty, k = k0 + tx;
  const bool cell = main_t && j <= g.ny && k <= g.nz;
  const bool doML = main_t && j <= g.ny + 1 && k <= g.nz;
  const bool doNL = main_t && j <= g.ny && k <= g.nz + 1;
  // the fifth wave: lanes [0,VK) the y faces of row j0+VJ, lanes [VK,VK+VJ)
  // the z faces of column k0+VK
  const int e = tid - VJ * VK;
  const bool exML = !main_t && e < VK && j0 + VJ <= g.ny + 1 && k0 + e <= g.nz;
  const bool exNL = !main_t && e >= VK && e < VK + VJ && j0 + (e - VK) <= g.ny && k0 + VK <= g.nz + 1;
  const long nf = g.nf;

  // the face metrics of the tile's rows, read once: a wave spans two rows j,
  // so reading them per face from global memory takes vector loads and
  // registers (128 -> 98 VGPRs, 0.69 -> 0.654 ms at 256x192x256)
  for (int idx = tid; idx < 3 * (VJ + 1); idx += VTHREADS) {
    const int set = idx / (VJ + 1), r = idx - set * (VJ + 1), jp = j0 + r - 1;
    const int sid = set == 0 ? SET_U : set == 1 ? SET_V : SET_W;
    const bool in = jp < g.Ym;
    L.PJ[set][0][r] = in ? pf(prof, g.Ym, sid, 1, jp) : 0.;
    L.PJ[set][1][r] = in ? pf(prof, g.Ym, sid, 5, jp) : 0.;
    L.PJ[set][2][r] = in ? pf(prof, g.Ym, sid, 9, jp) : 0.;
    const double Jf = in ? pf(prof, g.Ym, sid, 0, jp) : 0.;
    L.PJ[set][3][r] = Jf;
    L.PJ[set][4][r] = 1.0 / Jf;
  }
  VRaw R;
  vfetch(R, U, prof, g, ib - 1, j0, k0, tid);
  vstore(L, R, g, (ib - 1) % 3, j0, k0, tid);
  vfetch(R, U, prof, g, ib, j0, k0, tid);
  vstore(L, R, g, ib % 3, j0, k0, tid);
  vfetch(R, U, prof, g, ib + 1, j0, k0, tid);
  __syncthreads();
  double LLc[4] = {0., 0., 0., 0.};
  if (cell) vface_x(L, ib % 3, (ib - 1) % 3, ty + 1, tx + 1, invXI, inv4ET, inv4ZT, LLc);
  for (int i = ib; i <= ie; i++) {
    const int sm = (i - 1) % 3, s0 = i % 3, sp = (i + 1) % 3;
    vstore(L, R, g, sp, j0, k0, tid);
    if (i + 1 <= ie) vfetch(R, U, prof, g, i + 2, j0, k0, tid);
    __syncthreads();
    double LLn[4] = {0., 0., 0., 0.}, o[4];
    if (cell) vface_x(L, sp, s0, ty + 1, tx + 1, invXI, inv4ET, inv4ZT, LLn);
    if (doML) {
      vface_y(L, sp, s0, sm, ty + 1, tx + 1, invET, inv4XI, inv4ZT, o);
#pragma unroll
      for (int v = 0; v < 4; v++) L.ML[v][ty][tx] = o[v];
    }
    if (doNL) {
      vface_z(L, sp, s0, sm, ty + 1, tx + 1, invZT, inv4XI, inv4ET, o);
#pragma unroll
      for (int v = 0; v < 4; v++) L.NL[v][ty][tx] = o[v];
    }
    if (exML) {
      vface_y(L, sp, s0, sm, VJ + 1, e + 1, invET, inv4XI, inv4ZT, o);
#pragma unroll
      for (int v = 0; v < 4; v++) L.ML[v][VJ][e] = o[v];
    }
    if (exNL) {
      const int r = e - VK;
      vface_z(L, sp, s0, sm, r + 1, VK + 1, invZT, inv4XI, inv4ET, o);
#pragma unroll
      for (int v = 0; v < 4; v++) L.NL[v][r][VK] = o[v];
    }
    __syncthreads();
    if (cell) {
      const long c = at(g, i, j, k);
#pragma unroll
      for (int v = 0; v < 4; v++) {
        vF[v * nf + c] = (LLn[v] - LLc[v]) * invXI + (L.ML[v][ty + 1][tx] - L.ML[v][ty][tx]) * invET +
                         (L.NL[v][ty][tx + 1] - L.NL[v][ty][tx]) * invZT;
        LLc[v] = LLn[v];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// right-hand side: Dual_time_stepping.cpp:338-507
// ---------------------------------------------------------------------------
__device__ __forceinline__ void cell_metric(const double* __restrict__ prof, int Ym, int j, double m9[9]) {
#pragma unroll
  for (int c = 0; c < 9; c++) m9[c] = pf(prof, Ym, SET_C, 1 + c, j);
}

// MR = Gamma^-1 Rk of interior cell (i, j, k) (Dual_time_stepping.cpp:
// 338-436); s receives the cell's primitive state and u5 its U_
__device__ __forceinline__ void rhs_cell(const double* __restrict__ Ui, const double* __restrict__ Un,
                                         const double* __restrict__ Uq, const double* __restrict__ Fx,
                                         const double* __restrict__ Fy, const double* __restrict__ Fz,
                                         const double* __restrict__ vF, const double* __restrict__ prof,
                                         const Geo& g, double deltaT, double f_drive, int i, int j, int k,
                                         double M[5], PState& s, double u5[5]) {
  const long nf = g.nf;
  long c = at(g, i, j, k);
  long fx = at(g, i, j - 1, k - 1), fxm = fx - g.plane;
  long fy = at(g, i - 1, j, k - 1), fym = fy - g.Zp;
  long fz = at(g, i - 1, j - 1, k), fzm = fz - 1;
  double J = pf(prof, g.Ym, SET_C, 0, j);
#pragma unroll
  for (int v = 0; v < 5; v++) u5[v] = Ui[v * nf + c];
  s = prim_dt(u5[0], u5[1], u5[2], u5[3], u5[4], J);
  double beta = s.beta, rho = s.rho, u = s.u, v = s.v, w = s.w, VV = s.VV, T = s.T, H = s.H;
  double temp = rho * KG;
  double d11 = -(H * (KG - 1) + VV - KG * (T + VV)) * beta;
  double d12 = -(KG - 1) * u * beta, d13 = -(KG - 1) * v * beta, d14 = -(KG - 1) * w * beta;
  double d15 = (KG - 1) * beta;
  double d21 = -u / rho, d22 = 1 / rho, d31 = -v / rho, d41 = -w / rho;
  double d51 = (KG - 1) * (VV + KG * T * beta + (KG - 1) * VV * beta + H * (-1 + beta - KG * beta)) / temp;
  double d52 = -(KG - 1) * u * (1 + (KG - 1) * beta) / temp;
  double d53 = -(KG - 1) * v * (1 + (KG - 1) * beta) / temp;
  double d54 = -(KG - 1) * w * (1 + (KG - 1) * beta) / temp;
  double d55 = (KG - 1) * (1 + (KG - 1) * beta) / temp;
  double Rk[5];
#pragma unroll
  for (int q = 0; q < 5; q++) {
    double Rp = -(3 * u5[q] - 4 * Un[q * nf + c] + Uq[q * nf + c]) / (2 * deltaT);
    double Rf = -((Fx[q * nf + fx] - Fx[q * nf + fxm]) / g.dXI + (Fy[q * nf + fy] - Fy[q * nf + fym]) / g.dET +
                  (Fz[q * nf + fz] - Fz[q * nf + fzm]) / g.dZT);
    Rk[q] = Rp + Rf;
  }
  Rk[1] = Rk[1] + vF[c] + f_drive / J;
  Rk[2] = Rk[2] + vF[nf + c];
  Rk[3] = Rk[3] + vF[2 * nf + c];
  Rk[4] = Rk[4] + vF[3 * nf + c] + f_drive * u / J;
  M[0] = (d11 * Rk[0] + d12 * Rk[1] + d13 * Rk[2] + d14 * Rk[3] + d15 * Rk[4]);
  M[1] = (d21 * Rk[0] + d22 * Rk[1] + 0 * Rk[2] + 0 * Rk[3] + 0 * Rk[4]);
  M[2] = (d31 * Rk[0] + 0 * Rk[1] + d22 * Rk[2] + 0 * Rk[3] + 0 * Rk[4]);
  M[3] = (d41 * Rk[0] + 0 * Rk[1] + 0 * Rk[2] + d22 * Rk[3] + 0 * Rk[4]);
  M[4] = (d51 * Rk[0] + d52 * Rk[1] + d53 * Rk[2] + d54 * Rk[3] + d55 * Rk[4]);
}

__global__ void __launch_bounds__(256) k_rhs(const double* __restrict__ Ui, const double* __restrict__ Un,
                                             const double* __restrict__ Uq, const double* __restrict__ Fx,
                                             const double* __restrict__ Fy, const double* __restrict__ Fz,
                                             const double* __restrict__ vF, const double* __restrict__ prof,
                                             double* __restrict__ MR, double* __restrict__ NL, Geo g, double deltaT,
                                             double f_drive) {
  int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  int j = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  int i = 3 + blockIdx.z;
  if (k > g.nz || j > g.ny) return;
  const long nf = g.nf;
  const long c = at(g, i, j, k);
  double M[5], u5[5];
  PState s;
  rhs_cell(Ui, Un, Uq, Fx, Fy, Fz, vF, prof, g, deltaT, f_drive, i, j, k, M, s, u5);
#pragma unroll
  for (int q = 0; q < 5; q++) MR[q * nf + c] = M[q];
  if (NL) {
    double m9[9], e11, e22, e51;
    cell_metric(prof, g.Ym, j, m9);
    dinv(s, m9, g.dXI, g.dET, g.dZT, deltaT, &e11, &e22, &e51);
    NL[c] = e11 * M[0];
    NL[nf + c] = e22 * M[1];
    NL[2 * nf + c] = e22 * M[2];
    NL[3 * nf + c] = e22 * M[3];
    NL[4 * nf + c] = e51 * M[0] + e22 * M[4];
  }
}

// ---------------------------------------------------------------------------
// LU-SGS sweeps, one hyperplane i+j+k = m per launch
// (Dual_time_stepping.cpp:563-881 forward, :890-1250 backward)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void ld5(const double* __restrict__ A, long nf, long p, double o[5]) {
#pragma unroll
  for (int v = 0; v < 5; v++) o[v] = A[v * nf + p];
}

__global__ void __launch_bounds__(256) k_sweep_fwd(const double* __restrict__ Ui, const double* __restrict__ MR,
                                                   double* __restrict__ NL, const double* __restrict__ prof, Geo g,
                                                   double deltaT, int m, int ilo) {
  int j = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  int i = ilo + blockIdx.y;
  int k = m - i - j;
  if (j > g.ny || k < 2 || k > g.nz) return;
  const long nf = g.nf;
  long c = at(g, i, j, k);
  const long nb[3] = {c - g.plane, c - (long)g.Zp, c - 1};
  const bool inside[3] = {i - 1 >= 3, j - 1 >= 2, k - 1 >= 2};
  const int jn[3] = {j, j - 1, j};
  const double dd[3] = {g.dXI, g.dET, g.dZT};
  double LL[5];
  double acc[3][5];
#pragma unroll
  for (int dir = 0; dir < 3; dir++) {
    if (!inside[dir]) {
#pragma unroll
      for (int v = 0; v < 5; v++) acc[dir][v] = 0.0;
      continue;
    }
    double u5[5], N[5];
    ld5(Ui, nf, nb[dir], u5);
    ld5(NL, nf, nb[dir], N);
    PState s = prim_dt(u5[0], u5[1], u5[2], u5[3], u5[4], pf(prof, g.Ym, SET_C, 0, jn[dir]));
    Split a = split_jac(s, pf(prof, g.Ym, SET_C, 1 + 3 * dir, jn[dir]), pf(prof, g.Ym, SET_C, 2 + 3 * dir, jn[dir]),
                        pf(prof, g.Ym, SET_C, 3 + 3 * dir, jn[dir]), dir);
    lower_sum(a, N, acc[dir]);
  }
#pragma unroll
  for (int v = 0; v < 5; v++) LL[v] = acc[0][v] / dd[0] + acc[1][v] / dd[1] + acc[2][v] / dd[2];
  double u5[5], m9[9], d11, d22, d51;
  ld5(Ui, nf, c, u5);
  PState s0 = prim_dt(u5[0], u5[1], u5[2], u5[3], u5[4], pf(prof, g.Ym, SET_C, 0, j));
  cell_metric(prof, g.Ym, j, m9);
  dinv(s0, m9, g.dXI, g.dET, g.dZT, deltaT, &d11, &d22, &d51);
  double M[5];
  ld5(MR, nf, c, M);
  NL[c] = d11 * (M[0] - LL[0]);
  NL[nf + c] = d22 * (M[1] - LL[1]);
  NL[2 * nf + c] = d22 * (M[2] - LL[2]);
  NL[3 * nf + c] = d22 * (M[3] - LL[3]);
  NL[4 * nf + c] = d51 * (M[0] - LL[0]) + d22 * (M[4] - LL[4]);
}

__global__ void __launch_bounds__(256) k_sweep_bwd(const double* __restrict__ Ui, const double* __restrict__ NL,
                                                   double* __restrict__ NR, const double* __restrict__ prof, Geo g,
                                                   double deltaT, int m, int ilo) {
  int j = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  int i = ilo + blockIdx.y;
  int k = m - i - j;
  if (j > g.ny || k < 2 || k > g.nz) return;
  const long nf = g.nf;
  long c = at(g, i, j, k);
  const long nb[3] = {c + g.plane, c + (long)g.Zp, c + 1};
  const bool inside[3] = {i + 1 <= g.gend, j + 1 <= g.ny, k + 1 <= g.nz};
  const int jn[3] = {j, j + 1, j};
  const double dd[3] = {g.dXI, g.dET, g.dZT};
  double UU[5];
  double acc[3][5];
#pragma unroll
  for (int dir = 0; dir < 3; dir++) {
    if (!inside[dir]) {
#pragma unroll
      for (int v = 0; v < 5; v++) acc[dir][v] = 0.0;
      continue;
    }
    double u5[5], N[5];
    ld5(Ui, nf, nb[dir], u5);
    ld5(NR, nf, nb[dir], N);
    PState s = prim_dt(u5[0], u5[1], u5[2], u5[3], u5[4], pf(prof, g.Ym, SET_C, 0, jn[dir]));
    Split a = split_jac(s, pf(prof, g.Ym, SET_C, 1 + 3 * dir, jn[dir]), pf(prof, g.Ym, SET_C, 2 + 3 * dir, jn[dir]),
                        pf(prof, g.Ym, SET_C, 3 + 3 * dir, jn[dir]), dir);
    upper_sum(a, N, acc[dir]);
  }
#pragma unroll
  for (int v = 0; v < 5; v++) UU[v] = acc[0][v] / dd[0] + acc[1][v] / dd[1] + acc[2][v] / dd[2];
  double u5[5], m9[9], d11, d22, d51;
  ld5(Ui, nf, c, u5);
  PState s0 = prim_dt(u5[0], u5[1], u5[2], u5[3], u5[4], pf(prof, g.Ym, SET_C, 0, j));
  cell_metric(prof, g.Ym, j, m9);
  dinv(s0, m9, g.dXI, g.dET, g.dZT, deltaT, &d11, &d22, &d51);
  double N0[5];
  ld5(NL, nf, c, N0);
  NR[c] = N0[0] - d11 * UU[0];
  NR[nf + c] = N0[1] - d22 * UU[1];
  NR[2 * nf + c] = N0[2] - d22 * UU[2];
  NR[3 * nf + c] = N0[3] - d22 * UU[3];
  NR[4 * nf + c] = N0[4] - (d51 * UU[0] + d22 * UU[4]);
}

// ---------------------------------------------------------------------------
// LU-SGS sweeps as one persistent launch per direction.
//
// The sweep result depends only on the dependency DAG (each cell needs its
// three upstream neighbours), so any topological visiting order reproduces
// the hyperplane order of Dual_time_stepping.cpp:563-1250 bit for bit.  Here
// one 64-lane wave owns an 8x8 tile of (i,j) columns and walks k: lane (a,b)
// handles k = kmin + tau - a - b at step tau (a hyperplane inside the tile).
// Neighbours inside the tile come through double-buffered LDS, the previous
// cell of the column stays in registers, and results of the two upstream
// tiles are read from global memory.
//
// Cross-tile hand-off: before a sweep direction starts, the cells whose
// result another tile reads are filled with a NaN-payload sentinel that no
// arithmetic produces.  The producer writes its results with agent-scope
// relaxed atomic stores (coherent at device scope, no L2 write-back needed)
// and the consumer reads them with agent-scope relaxed atomic loads, re-
// reading while it still sees the sentinel.  The data carries its own
// readiness, so there is no flag, no fence and no store-completion wait;
// each step's loads are issued one step ahead to overlap their latency.
// Tiles take tickets in dependency order, so a wave only ever waits on tiles
// that are already running; every wait is bounded and reports
// CF_ERR_TIMEOUT.
// ---------------------------------------------------------------------------
constexpr int TI = 8, TJ = 8;
constexpr unsigned long long SENTINEL = 0x7FF4C0FFEE5EED01ULL;

__device__ __forceinline__ bool is_sentinel(double v) {
  return (unsigned long long)__double_as_longlong(v) == SENTINEL;
}

// the FP32 sweep's hand-off slots: a signalling-NaN payload that no
// arithmetic produces (loads, stores and cross-lane moves keep the bits)
constexpr unsigned SENTINEL32 = 0x7FA5EED1u;

__device__ __forceinline__ bool is_sentinel(float v) { return __float_as_uint(v) == SENTINEL32; }

template <class T>
__device__ __forceinline__ T sentinel_value();
template <>
__device__ __forceinline__ double sentinel_value<double>() {
  return __longlong_as_double((long long)SENTINEL);
}
template <>
__device__ __forceinline__ float sentinel_value<float>() {
  return __uint_as_float(SENTINEL32);
}

// Sweep-order layout: element (tile, s, lane) with lane = a + 8b and
// s = (k-2) + a + b, i.e. the step at which the forward walk visits the cell;
// the backward walk visits it at step nsteps-1-s.  At every step the 64 lanes
// of a tile touch one contiguous 512-byte row of each field.
struct Sk {
  int nTI, nTJ, ntiles, Nz, nsteps;
  long nsk;  // elements per field
};

__device__ __forceinline__ long sk_at(const Sk& q, int tile, int s, int lane) {
  return ((long)tile * q.nsteps + s) * 64 + lane;
}

// Slots of 5 x 8 values per tile, edge and step, each in cache lines of its
// own: the hand-off of the pipelined sweeps (edge 0 x, 1 y) and the compact
// copy of the summary along x (edge 0: a = 7, edge 1: a = 0; P, beta, rho, U_x
// and lambda_x by b), whose lanes are 64 bytes apart in the rows
constexpr int HO_SLOT = 64;  // elements per slot (40 used)
__host__ __device__ __forceinline__ long ho_at(const Sk& q, int tile, int edge, int s) {
  return (((long)tile * 2 + edge) * q.nsteps + s) * HO_SLOT;
}

// thread (s, lane) of a block of 16 steps x 64 lanes -> cell; false if the
// slot holds no interior cell
__device__ __forceinline__ bool sk_cell(const Sk& q, const Geo& g, int tile, int s, int lane, int* i, int* j,
                                        int* k) {
  const int a = lane & 7, b = lane >> 3;
  const int kk = s - a - b;
  *i = 3 + (tile % q.nTI) * TI + a;
  *j = 2 + (tile / q.nTI) * TJ + b;
  *k = 2 + kk;
  return s < q.nsteps && kk >= 0 && kk < q.Nz && *i <= g.gend && *j <= g.ny;
}

// diagonal-metric summary (DiagField) of one cell (Dual_time_stepping.cpp:
// 343-372 primitives, 751-811 split-Jacobian ingredients)
__device__ __forceinline__ void prep_summary(const double u5[5], const double* __restrict__ prof, const Geo& g, int j,
                                             double v[G_N]) {
  PState st = prim_dt(u5[0], u5[1], u5[2], u5[3], u5[4], pf(prof, g.Ym, SET_C, 0, j));
  double m9[9];
#pragma unroll
  for (int r = 0; r < 9; r++) m9[r] = pf(prof, g.Ym, SET_C, 1 + r, j);
  double U3[3], L3[3];
  L3[0] = lambda_dir(st, m9[0], m9[1], m9[2], &U3[0]);
  L3[1] = lambda_dir(st, m9[3], m9[4], m9[5], &U3[1]);
  L3[2] = lambda_dir(st, m9[6], m9[7], m9[8], &U3[2]);
  v[G_P] = st.P;
  v[G_BETA] = st.beta;
  v[G_RHO] = st.rho;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    v[G_UX + 2 * d] = U3[d];
    v[G_LX + 2 * d] = L3[d];
  }
}

// the summary row, and the x edges' compact copy
template <class T>
__device__ __forceinline__ void store_summary(T* __restrict__ S, T* __restrict__ E, const Sk& q, int tile, int s,
                                              int lane, const double v[G_N]) {
  const long o = sk_at(q, tile, s, lane);
#pragma unroll
  for (int r = 0; r < G_N; r++) S[r * q.nsk + o] = T(v[r]);
  const int a = lane & 7;
  if (a == 0 || a == TI - 1) {
    T* e = E + ho_at(q, tile, a == 0, s) + (lane >> 3);
    constexpr int f[5] = {G_P, G_BETA, G_RHO, G_UX, G_LX};
#pragma unroll
    for (int r = 0; r < 5; r++) e[8 * r] = T(v[f[r]]);
  }
}

// tickets, error flags and progress of both sweep directions back to zero: by
// the pre-pass's first block for the first sweep pair, by k_sweep_reset before
// each later one
__device__ __forceinline__ void sweep_reset(int* __restrict__ sync, int n) {
  if (blockIdx.x == 0 && blockIdx.y == 0)
    for (int t = threadIdx.x; t < n; t += blockDim.x) sync[t] = 0;
}

__global__ void __launch_bounds__(256) k_sweep_reset(int* __restrict__ sync, int n) { sweep_reset(sync, n); }

// A prep block covers PC steps of one tile.  Column (a, b) of the tile meets
// cells k-2 = s - a - b at steps s0 .. s0+PC-1: one run of PC consecutive k,
// which the block stages in LDS with coalesced loads; slot (s, lane) then
// reads its cell at LDS index s - s0 whatever the column.
// 16 steps (53 KB of LDS with the update's reduction buffer, three blocks
// per CU) measured fastest for the
// update pass at 256x192x256: 0.327 ms against 0.342 / 0.358 / 0.361 ms for
// 12 / 24 / 8 steps (FP64 NR), 0.286 against 0.310 / 0.334 / 0.325 ms (float)
constexpr int PC = 16, PCP = PC + 1;  // steps per block; LDS column stride

__device__ __forceinline__ void prep_stage(double (*L)[64][PCP], const double* __restrict__ src, const Geo& g,
                                           const Sk& q, int tile, int s0) {
  const int TX = tile % q.nTI, TY = tile / q.nTI;
  for (int idx = threadIdx.x; idx < 64 * PC; idx += blockDim.x) {
    const int col = idx / PC, t = idx - col * PC;
    const int a = col & 7, b = col >> 3;
    const int i = 3 + TX * TI + a, j = 2 + TY * TJ + b, kk = s0 - a - b + t;
    if (i > g.gend || j > g.ny || kk < 0 || kk >= q.Nz) continue;
    const long c = at(g, i, j, 2 + kk);
#pragma unroll
    for (int f = 0; f < 5; f++) L[f][col][t] = src[f * g.nf + c];
  }
}

// the summary and MR in sweep order; each wave writes whole 512-byte rows
template <class T>
__global__ void __launch_bounds__(256) k_sweep_prep(const double* __restrict__ Ui, const double* __restrict__ MR,
                                                    const double* __restrict__ prof, T* __restrict__ S,
                                                    T* __restrict__ MRs, T* __restrict__ E, Geo g, Sk q,
                                                    int* __restrict__ sync) {
  __shared__ double L[5][64][PCP];
  sweep_reset(sync, 2 * q.ntiles + 4);
  int bx, by, bz;
  xcd_block3(&bx, &by, &bz);
  const int tile = by, s0 = bx * PC;
  prep_stage(L, Ui, g, q, tile, s0);
  __syncthreads();
  for (int idx = threadIdx.x; idx < PC * 64; idx += blockDim.x) {
    const int t = idx >> 6, lane = idx & 63, s = s0 + t;
    int i, j, k;
    if (!sk_cell(q, g, tile, s, lane, &i, &j, &k)) continue;
    const long o = sk_at(q, tile, s, lane);
    double u5[5], v[G_N];
#pragma unroll
    for (int f = 0; f < 5; f++) u5[f] = L[f][lane][t];
    prep_summary(u5, prof, g, j, v);
    store_summary(S, E, q, tile, s, lane, v);
  }
  __syncthreads();
  prep_stage(L, MR, g, q, tile, s0);
  __syncthreads();
  for (int idx = threadIdx.x; idx < PC * 64; idx += blockDim.x) {
    const int t = idx >> 6, lane = idx & 63, s = s0 + t;
    int i, j, k;
    if (!sk_cell(q, g, tile, s, lane, &i, &j, &k)) continue;
    const long o = sk_at(q, tile, s, lane);
#pragma unroll
    for (int r = 0; r < 5; r++) MRs[r * q.nsk + o] = T(L[r][lane][t]);
  }
}

// k_rhs and k_sweep_prep in one pass.  A block covers PR steps of one tile
// (as k_sweep_prep does) in two rounds through one 5-field LDS tile: it walks
// each column's run of PR consecutive k in the natural layout (coalesced),
// forms MR of each cell with rhs_cell and writes whole 512-byte sweep-order
// rows of MR; then it stages the runs of U_ and writes the rows of the
// summary.  MR never goes to HBM in the natural layout.  The single 5-field
// tile (43 KB) lets three blocks share a CU; ten fields staged at once
// (PR = 12, 66 KB, two blocks) took 3.4% longer in FP64 and 5.5% in float.
// Each thread keeps the U_ of its PR / 4 cells in registers from the first
// round to the second: a block's first round outlasts the L2's turnover, so
// reading U_ again would fetch it from HBM a second time.
constexpr int PR = 16, PRP = PR + 1, PR_THREADS = 256, PR_CELLS = 64 * PR / PR_THREADS;
static_assert(64 * PR % PR_THREADS == 0, "whole cells per thread");

template <class T>
__global__ void __launch_bounds__(PR_THREADS) k_sweep_prep_rhs(const double* __restrict__ Ui, RhsIn rin,
                                                               const double* __restrict__ prof, T* __restrict__ S,
                                                               T* __restrict__ MRs, T* __restrict__ E, Geo g, Sk q,
                                                               double deltaT, int* __restrict__ sync) {
  sweep_reset(sync, 2 * q.ntiles + 4);
  __shared__ double L[5][64][PRP];
  int bx, by, bz;
  xcd_block3(&bx, &by, &bz);
  const int tile = by, s0 = bx * PR;
  const int TX = tile % q.nTI, TY = tile / q.nTI;
  double keep[PR_CELLS][5];
#pragma unroll
  for (int m = 0; m < PR_CELLS; m++) {
    const int idx = threadIdx.x + m * PR_THREADS;
    const int col = idx / PR, t = idx - col * PR;
    const int a = col & 7, b = col >> 3;
    const int i = 3 + TX * TI + a, j = 2 + TY * TJ + b, kk = s0 - a - b + t;
    if (i > g.gend || j > g.ny || kk < 0 || kk >= q.Nz) continue;
    double M[5];
    PState st;
    rhs_cell(Ui, rin.Un, rin.Uq, rin.Fx, rin.Fy, rin.Fz, rin.vF, prof, g, deltaT, rin.f_drive, i, j, 2 + kk, M, st,
             keep[m]);
#pragma unroll
    for (int f = 0; f < 5; f++) L[f][col][t] = M[f];
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < PR * 64; idx += blockDim.x) {
    const int t = idx >> 6, lane = idx & 63, s = s0 + t;
    int i, j, k;
    if (!sk_cell(q, g, tile, s, lane, &i, &j, &k)) continue;
    const long o = sk_at(q, tile, s, lane);
#pragma unroll
    for (int r = 0; r < 5; r++) MRs[r * q.nsk + o] = T(L[r][lane][t]);
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < PR_CELLS; m++) {
    const int idx = threadIdx.x + m * PR_THREADS;
    const int col = idx / PR, t = idx - col * PR;
    const int a = col & 7, b = col >> 3;
    const int i = 3 + TX * TI + a, j = 2 + TY * TJ + b, kk = s0 - a - b + t;
    if (i > g.gend || j > g.ny || kk < 0 || kk >= q.Nz) continue;
#pragma unroll
    for (int f = 0; f < 5; f++) L[f][col][t] = keep[m][f];
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < PR * 64; idx += blockDim.x) {
    const int t = idx >> 6, lane = idx & 63, s = s0 + t;
    int i, j, k;
    if (!sk_cell(q, g, tile, s, lane, &i, &j, &k)) continue;
    const long o = sk_at(q, tile, s, lane);
    double u5[5], v[G_N];
#pragma unroll
    for (int f = 0; f < 5; f++) u5[f] = L[f][lane][t];
    prep_summary(u5, prof, g, j, v);
    store_summary(S, E, q, tile, s, lane, v);
  }
}

// sweep-order field(s) back to the natural layout
template <class T>
__global__ void __launch_bounds__(1024) k_sk_to_natural(const T* __restrict__ src, double* __restrict__ dst,
                                                        Geo g, Sk q, int nfields) {
  const int lane = threadIdx.x & 63;
  const int s = blockIdx.x * 16 + (threadIdx.x >> 6);
  const int tile = blockIdx.y;
  int i, j, k;
  if (!sk_cell(q, g, tile, s, lane, &i, &j, &k)) return;
  const long c = at(g, i, j, k), o = sk_at(q, tile, s, lane);
  for (int v = 0; v < nfields; v++) dst[v * g.nf + c] = double(src[v * q.nsk + o]);
}

// The NL slots that k_sweep_tiles' forward sweep hands across tiles (lanes on
// a tile's high x or y edge, every step) set to the sentinel.  Its backward
// sweep sets every such slot it has read back to the sentinel, so this runs
// only when the slots may hold anything else: a new buffer, after a sweep
// that gave up, or after pipelined sweeps, which fill NL.
__global__ void __launch_bounds__(256) k_seed_tiles(double* __restrict__ NLs, Sk q) {
  const int lane = threadIdx.x & 63, s = blockIdx.x * 4 + (threadIdx.x >> 6), tile = blockIdx.y;
  if (s >= q.nsteps || ((lane & 7) != TI - 1 && (lane >> 3) != TJ - 1)) return;
  const long o = sk_at(q, tile, s, lane);
  const double sv = sentinel_value<double>();
#pragma unroll
  for (int v = 0; v < 5; v++) NLs[v * q.nsk + o] = sv;
}

__device__ __forceinline__ double ld_coherent(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void st_coherent(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ float ld_coherent(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void st_coherent(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// one step's global inputs of a lane
struct StepIn {
  double own[G_N];   // summary of the lane's cell
  double src[5];     // MR (forward) or NL (backward) of the lane's cell
  double xN[5], yN[5];
  DNb xc, yc;        // remote neighbours along x and y
};

// LDS slot of one lane: N(5), P, T, beta, x: U, lam, pd, p51, y: U, lam, pd, p51
constexpr int LDS_F = 16;

// neighbour p along direction d; n: the diagonal metric entry at its j
__device__ __forceinline__ DNb dnb_at(const double* __restrict__ S, long nsk, long p, int d, double n) {
  DNb c;
  const double rho = S[G_RHO * nsk + p];
  const double rr = rcp_rho(rho);
  c.P = S[G_P * nsk + p];
  c.T = over_rho(c.P, rho, rr);
  c.beta = S[G_BETA * nsk + p];
  c.U = S[(G_UX + 2 * d) * nsk + p];
  c.lam = S[(G_LX + 2 * d) * nsk + p];
  split_pd_p51(n, c.U, c.beta, rho, rr, &c.pd, &c.p51);
  return c;
}

template <bool FWD>
__global__ void __launch_bounds__(64) k_sweep_tiles(const double* __restrict__ S, double* __restrict__ SRC,
                                                    double* __restrict__ DST, double* __restrict__ AUX,
                                                    const double* __restrict__ prof, Geo g, Sk q,
                                                    const int* __restrict__ order, int* __restrict__ sync,
                                                    long spin_limit, double deltaT) {
  // all arrays in sweep order (Sk); S holds the DiagField summary
  // FWD: SRC = MR, DST = NL   (NL = D^-1 (MR - L)); seeds the NR (AUX) sentinels
  // BWD: SRC = NL, DST = NR   (NR = NL - D^-1 U); re-seeds the NL sentinels
  const int nTI = q.nTI;
  __shared__ double lds[2][LDS_F][64];
  __shared__ int s_ticket;
  const int ntiles = q.ntiles;
  int* ticket = sync;
  int* err = sync + 1;
  const int lane = threadIdx.x;
  const int a = lane & 7, b = lane >> 3;
  if (lane == 0) s_ticket = atomicAdd(ticket, 1);
  __syncthreads();
  const int t = s_ticket;
  if (t >= ntiles) return;
  const int tile = order[FWD ? t : ntiles - 1 - t];
  const int TX = tile % nTI, TY = tile / nTI;
  const int i = 3 + TX * TI + a, j = 2 + TY * TJ + b;
  const bool col = i <= g.gend && j <= g.ny;
  const int Nz = q.Nz;
  const int nsteps = q.nsteps;
  const int off = FWD ? a + b : (TI - 1 - a) + (TJ - 1 - b);
  const int ax_lane = FWD ? lane - 1 : lane + 1;   // (a-1,b) or (a+1,b)
  const int ay_lane = FWD ? lane - 8 : lane + 8;   // (a,b-1) or (a,b+1)
  const bool x_in_tile = FWD ? a > 0 : a < TI - 1;
  const bool y_in_tile = FWD ? b > 0 : b < TJ - 1;
  const bool x_dom = FWD ? i - 1 >= 3 : i + 1 <= g.gend;
  const bool y_dom = FWD ? j - 1 >= 2 : j + 1 <= g.ny;
  const bool x_remote = col && x_dom && !x_in_tile;
  const bool y_remote = col && y_dom && !y_in_tile;
  const int jy = FWD ? j - 1 : j + 1;
  const long nf = q.nsk;
  // remote neighbours: same k, lane (7,b)/(a,7) of the upstream tile (forward)
  // or (0,b)/(a,0) of the downstream tile (backward), 7 steps apart
  const long sx = FWD ? (-(long)q.nsteps * 64 + 7 * 64 + 7) : ((long)q.nsteps * 64 - 7 * 64 - 7);
  const long sy = FWD ? (-(long)nTI * q.nsteps * 64 + 7 * 64 + 56) : ((long)nTI * q.nsteps * 64 - 7 * 64 - 56);
  // diagonal metric entries of the neighbours (functions of j)
  const double nx = pf(prof, g.Ym, SET_C, 1, j), ny_ = pf(prof, g.Ym, SET_C, 5, jy), nz_ = pf(prof, g.Ym, SET_C, 9, j);
  const double nyo = pf(prof, g.Ym, SET_C, 5, j);  // at the lane's own j, for the entries it hands on

  auto cell_of = [&](int tau) -> long { return sk_at(q, tile, FWD ? tau : q.nsteps - 1 - tau, lane); };
  auto active = [&](int tau) -> bool {
    const int kk = tau - off;
    return col && kk >= 0 && kk < Nz;
  };
  auto load_step = [&](int tau, StepIn& in) {
    if (!active(tau)) return;
    const long c = cell_of(tau);
#pragma unroll
    for (int r = 0; r < G_N; r++) in.own[r] = S[r * nf + c];
#pragma unroll
    for (int v = 0; v < 5; v++) in.src[v] = SRC[v * nf + c];
    if (x_remote) {
      const long p = c + sx;
#pragma unroll
      for (int v = 0; v < 5; v++) in.xN[v] = ld_coherent(DST + v * nf + p);
      in.xc = dnb_at(S, nf, p, 0, nx);
    }
    if (y_remote) {
      const long p = c + sy;
#pragma unroll
      for (int v = 0; v < 5; v++) in.yN[v] = ld_coherent(DST + v * nf + p);
      in.yc = dnb_at(S, nf, p, 1, ny_);
    }
  };
  // re-reads remote values that were not ready when first loaded
  auto settle = [&](double (&N)[5], long p) {
    long n = 0;
    bool pending = true;
    while (pending) {
      pending = false;
#pragma unroll
      for (int v = 0; v < 5; v++) pending |= is_sentinel(N[v]);
      if (!pending) break;
      if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 || ++n > spin_limit) {
        __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
#pragma unroll
      for (int v = 0; v < 5; v++) N[v] = ld_coherent(DST + v * nf + p);
    }
  };
  const bool edge_fwd = a == TI - 1 || b == TJ - 1;   // slots read across tiles by a forward sweep
  const bool edge_bwd = a == 0 || b == 0;             // ... by a backward sweep
  const double sv = __longlong_as_double((long long)SENTINEL);
  auto lds_nb = [&](int pb, int src_lane, int d, DNb& c, double (&N)[5]) {
#pragma unroll
    for (int v = 0; v < 5; v++) N[v] = lds[pb][v][src_lane];
    c.P = lds[pb][5][src_lane];
    c.T = lds[pb][6][src_lane];
    c.beta = lds[pb][7][src_lane];
    c.U = lds[pb][8 + 4 * d][src_lane];
    c.lam = lds[pb][9 + 4 * d][src_lane];
    c.pd = lds[pb][10 + 4 * d][src_lane];
    c.p51 = lds[pb][11 + 4 * d][src_lane];
  };

  double zN[5] = {0, 0, 0, 0, 0};
  DNb zc = {0, 0, 0, 0, 0, 0, 0};
  StepIn nxt;
  load_step(0, nxt);
  for (int tau = 0; tau < nsteps; tau++) {
    StepIn cur = nxt;
    if (tau + 1 < nsteps) load_step(tau + 1, nxt);
    const bool act = active(tau);
    const int kk = tau - off;
    const int pb = (tau + 1) & 1, cb = tau & 1;
    if (act) {
      const long c = cell_of(tau);
      if (x_remote) settle(cur.xN, c + sx);
      if (y_remote) settle(cur.yN, c + sy);
      double acc[3][5];
      if (x_dom) {
        DNb nc;
        double N[5];
        if (x_in_tile) {
          lds_nb(pb, ax_lane, 0, nc, N);
        } else {
          nc = cur.xc;
#pragma unroll
          for (int v = 0; v < 5; v++) N[v] = cur.xN[v];
        }
        if (FWD) lower_diag<0>(nc, nx, N, acc[0]); else upper_diag<0>(nc, nx, N, acc[0]);
      } else {
#pragma unroll
        for (int v = 0; v < 5; v++) acc[0][v] = 0.0;
      }
      if (y_dom) {
        DNb nc;
        double N[5];
        if (y_in_tile) {
          lds_nb(pb, ay_lane, 1, nc, N);
        } else {
          nc = cur.yc;
#pragma unroll
          for (int v = 0; v < 5; v++) N[v] = cur.yN[v];
        }
        if (FWD) lower_diag<1>(nc, ny_, N, acc[1]); else upper_diag<1>(nc, ny_, N, acc[1]);
      } else {
#pragma unroll
        for (int v = 0; v < 5; v++) acc[1][v] = 0.0;
      }
      if (kk > 0) {
        if (FWD) lower_diag<2>(zc, nz_, zN, acc[2]); else upper_diag<2>(zc, nz_, zN, acc[2]);
      } else {
#pragma unroll
        for (int v = 0; v < 5; v++) acc[2][v] = 0.0;
      }
      double L[5];
#pragma unroll
      for (int v = 0; v < 5; v++)
        L[v] = div_rn(acc[0][v], g.dXI, g.rXI) + div_rn(acc[1][v], g.dET, g.rET) + div_rn(acc[2][v], g.dZT, g.rZT);
      double d11, d22, d51;
      diag_dinv<false>(cur.own[G_BETA], cur.own[G_RHO], cur.own[G_LX], cur.own[G_LY], cur.own[G_LZ], g, deltaT, &d11,
                       &d22, &d51);
      const double* M = cur.src;
      double out[5];
      if (FWD) {
        out[0] = d11 * (M[0] - L[0]);
        out[1] = d22 * (M[1] - L[1]);
        out[2] = d22 * (M[2] - L[2]);
        out[3] = d22 * (M[3] - L[3]);
        out[4] = d51 * (M[0] - L[0]) + d22 * (M[4] - L[4]);
      } else {
        out[0] = M[0] - d11 * L[0];
        out[1] = M[1] - d22 * L[1];
        out[2] = M[2] - d22 * L[2];
        out[3] = M[3] - d22 * L[3];
        out[4] = M[4] - (d51 * L[0] + d22 * L[4]);
      }
#pragma unroll
      for (int v = 0; v < 5; v++) st_coherent(DST + v * nf + c, out[v]);
      if (FWD && edge_bwd) {
        // the backward sweep that follows hands these NR slots across tiles
#pragma unroll
        for (int v = 0; v < 5; v++) AUX[v * nf + c] = sv;
      }
      if (!FWD && edge_fwd) {
        // this NL slot has been consumed; the next forward sweep hands it on
#pragma unroll
        for (int v = 0; v < 5; v++) SRC[v * nf + c] = sv;
      }
#pragma unroll
      for (int v = 0; v < 5; v++) {
        lds[cb][v][lane] = out[v];
        zN[v] = out[v];
      }
      const double Tc = cur.own[G_P] / cur.own[G_RHO];
      lds[cb][5][lane] = cur.own[G_P];
      lds[cb][6][lane] = Tc;
      lds[cb][7][lane] = cur.own[G_BETA];
      const double dn[3] = {nx, nyo, nz_};
#pragma unroll
      for (int d = 0; d < 2; d++) {
        double pd, p51;
        split_pd_p51(dn[d], cur.own[G_UX + 2 * d], cur.own[G_BETA], cur.own[G_RHO], rcp_rho(cur.own[G_RHO]), &pd, &p51);
        lds[cb][8 + 4 * d][lane] = cur.own[G_UX + 2 * d];
        lds[cb][9 + 4 * d][lane] = cur.own[G_LX + 2 * d];
        lds[cb][10 + 4 * d][lane] = pd;
        lds[cb][11 + 4 * d][lane] = p51;
      }
      zc.P = cur.own[G_P];
      zc.T = Tc;
      zc.beta = cur.own[G_BETA];
      zc.U = cur.own[G_UZ];
      zc.lam = cur.own[G_LZ];
      split_pd_p51(dn[2], zc.U, zc.beta, cur.own[G_RHO], rcp_rho(cur.own[G_RHO]), &zc.pd, &zc.p51);
    }
    // one wave per block: LDS writes of this step are complete and ordered
    // before the next step's reads
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// ---------------------------------------------------------------------------
// Pipelined tiled sweep: the same tiles, steps and arithmetic as
// k_sweep_tiles, spread over the ten waves of a block that meet at one
// LDS-only barrier per step (loads stay in flight across steps).  The sweep
// is a chain of dependent steps, so its time is the number of steps on the
// longest path times the work of the busiest wave (and SIMD) per step; every
// wave does one short job:
//   waves 0-3   load the rows of every fourth step and form, over four steps'
//               time, D^-1 and the split-Jacobian entries (SplitCoef,
//               diag_coef) that the cells' downstream neighbours use;
//   waves 4, 5  compute one cell per lane and step from LDS only, wave 4 the
//               components P and T (0, 4), wave 5 the velocities (1, 2, 3):
//               each component reads at most two others of a neighbour, and
//               those cross between the two waves with the neighbours' values;
//   waves 6, 7  poll the cross-tile neighbours' outputs of the even (odd) steps;
//   wave 8      writes the outputs to their rows;
//   wave 9      the split-Jacobian entries of the cross-tile neighbours, four
//               steps at a time (16 cells a step).
// Waves w, w + 4 and w + 8 share a SIMD.  What bounds it: at 64^3 the step, at
// 256x192x256 (FP64) also the 2.2 GB a sweep moves.  Measured, forward /
// backward, against four waves per block (one computing all five components,
// two loading, one polling two steps ahead; hand-off through the NL and NR
// rows): 64^3 FP64 156 / 151 -> 105 / 107 us, FP32 128 / 124 -> 83 / 84 us;
// 97x75x130 341 / 328 -> 184 / 179 and 205 / 195 -> 142 / 135 us; 256x192x256
// 915 / 838 -> 639 / 635 and 655 / 640 -> 485 / 475 us.  Steps that did not
// pay: two loader waves of every second step (64^3 144 us: each then takes
// longer than the compute waves), a wave per direction and one for D^-1 (131
// us), polling 4 or 8 steps ahead (120, 141 us), one polling wave (104 us at
// 64^3, but 795 us at 256x192x256), two tiles per CU (no change).
// LDS holds four step slots of per-lane data; slot s-1 carries the neighbour
// entries of step s, with the halo in columns 64..71 (x: by b, y: by a) so
// that every lane reads its neighbours at fixed offsets.
//
// Hand-off between tiles: slot s of a tile's x (or y) edge holds the 5 x 8
// outputs its downstream tile needs from step s, contiguous, in a buffer of
// its own.  The compute waves write a slot with agent-scope relaxed stores as
// soon as they have the values; the consumer's wave 6 or 7 re-reads it until no
// value is the sentinel, then its wave 8 sets it back to the sentinel.  So
// the buffer holds sentinels only between sweeps, whatever their direction,
// and the output rows themselves are ordinary stores.  A slot has 64
// elements, so no cache line holds values of two steps.
// ---------------------------------------------------------------------------
constexpr int PIPE_THREADS = 640;
constexpr int PIPE_SLOTS = 4;  // step slots in LDS
constexpr int PO_D11 = 0, PO_D22 = 1, PO_D51 = 2, PO_M = 3, PO_Z = 8, PO_N = 14;  // rows of PipeLds::own

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// f(0), f(1), .. f(N-1) in turn, again and again, until one returns false;
// the argument is an integral_constant, so that every register and LDS slot
// index is a constant.  for_each calls each once.
template <class F, int... K>
__device__ __forceinline__ void cycle_seq(F f, std::integer_sequence<int, K...>) {
  while ((f(std::integral_constant<int, K>{}) && ...)) {
  }
}
template <int N, class F>
__device__ __forceinline__ void cycle(F f) {
  cycle_seq(f, std::make_integer_sequence<int, N>{});
}
template <class F, int... K>
__device__ __forceinline__ void each_seq(F f, std::integer_sequence<int, K...>) {
  (f(std::integral_constant<int, K>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void for_each(F f) {
  each_seq(f, std::make_integer_sequence<int, N>{});
}
template <int N>
using Int = std::integral_constant<int, N>;

// an ordinary load that the compiler leaves where it is written: without
// this it sinks a load of a later step to the step that uses it
template <class T>
__device__ __forceinline__ T ld_here(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// T: the sweep's arithmetic and storage type (double, or float for the FP32
// inner solve)
template <class T>
struct PipeLds {
  T own[PIPE_SLOTS][PO_N][64];  // D11 D22 D51, MR or NL (5), z SplitCoef (6) of the lane cells
  T xc[PIPE_SLOTS][6][72];      // x SplitCoef: lanes, then the x halo by b
  T yc[PIPE_SLOTS][6][72];      // y SplitCoef: lanes, then the y halo by a
  T N[2][5][80];                // outputs of the previous step: lanes, x halo by b (64+), y halo by a (72+)
  int ticket;
};

template <class T, int W>
__device__ __forceinline__ void coef_store(T (*row)[W], int col, const SplitCoefT<T>& c) {
  row[0][col] = c.c11;
  row[1][col] = c.c1q;
  row[2][col] = c.c22;
  row[3][col] = c.c5q;
  row[4][col] = c.pd;
  row[5][col] = c.p51;
}

// A neighbour's contribution to the components a compute wave owns: those of
// diag_apply, expression by expression.  PT: components 0 and 4 (o[0], o[1]);
// otherwise components 1, 2, 3.
template <int D, bool FWD, bool PT, int W, class T>
__device__ __forceinline__ void apply_part(T (*c)[W], int col, const T N[5], T o[3]) {
  constexpr int q = D + 1;
  const T c22 = c[2][col];
  if constexpr (PT) {
    const T c11 = c[0][col], c1q = c[1][col], c5q = c[3][col], p51 = c[5][col];
    if (FWD) {
      o[0] = -c11 * N[0] - c1q * N[q];
      o[1] = -p51 * N[0] - c5q * N[q] - c22 * N[4];
    } else {
      o[0] = +c11 * N[0] + c1q * N[q];
      o[1] = +p51 * N[0] + c5q * N[q] + c22 * N[4];
    }
  } else {
    const T pd = c[4][col];
#pragma unroll
    for (int m = 1; m <= 3; m++) {
      if (FWD)
        o[m - 1] = m == q ? -pd * N[0] - c22 * N[m] : -(c22 * N[m]);
      else
        o[m - 1] = m == q ? +pd * N[0] + c22 * N[m] : c22 * N[m];
    }
  }
}

// waves 4 and 5: one cell per lane and step, inputs from LDS only.  In FP32
// the divisions by the spacings become products with their float reciprocals.
template <bool FWD, bool FD, bool PT, class T>
__device__ __forceinline__ void pipe_compute(PipeLds<T>& L, T* __restrict__ H, const Geo& g, const Sk& q, int tile,
                                             int TX, int TY) {
  constexpr bool F64 = std::is_same<T, double>::value;
  constexpr int NC = PT ? 2 : 3;
  constexpr int comp[3] = {PT ? 0 : 1, PT ? 4 : 2, 3};
  const int lane = threadIdx.x & 63;
  const int a = lane & 7, b = lane >> 3;
  const int i = 3 + TX * TI + a, j = 2 + TY * TJ + b;
  const bool col = i <= g.gend && j <= g.ny;
  const int Nz = q.Nz, nsteps = q.nsteps;
  const int off = FWD ? a + b : (TI - 1 - a) + (TJ - 1 - b);
  const bool x_dom = FWD ? i - 1 >= 3 : i + 1 <= g.gend;
  const bool y_dom = FWD ? j - 1 >= 2 : j + 1 <= g.ny;
  const bool x_in = FWD ? a > 0 : a < TI - 1;
  const bool y_in = FWD ? b > 0 : b < TJ - 1;
  // some cell of the tile has no x (y) neighbour: the same for all lanes
  const bool rim = FWD ? TX == 0 || TY == 0 : TX + 1 == q.nTI || tile + q.nTI >= q.ntiles;
  // neighbour columns: in-tile lanes or the halo
  const int xi = x_in ? (FWD ? lane - 1 : lane + 1) : 64 + b;
  const int yi = y_in ? (FWD ? lane - 8 : lane + 8) : 64 + a;
  const int yiN = y_in ? yi : 72 + a;
  // lanes whose outputs the downstream tiles read
  const bool hx = FWD ? a == TI - 1 && TX + 1 < q.nTI : a == 0 && TX > 0;
  const bool hy = FWD ? b == TJ - 1 && tile + q.nTI < q.ntiles : b == 0 && TY > 0;
  T* Hx = H + ho_at(q, tile, 0, 0) + b;
  T* Hy = H + ho_at(q, tile, 1, 0) + a;
  const float fXI = float(1.0 / g.dXI), fET = float(1.0 / g.dET), fZT = float(1.0 / g.dZT);
  T zN[5] = {0, 0, 0, 0, 0};
  int tau = 0;
  lds_barrier();  // step 0 inputs are in LDS
  cycle<PIPE_SLOTS>([&](auto k) -> bool {
    constexpr int cs = decltype(k)::value, ps = (cs + PIPE_SLOTS - 1) % PIPE_SLOTS, nw = cs & 1, nr = nw ^ 1;
    const int kk = tau - off;
    if (col && kk >= 0 && kk < Nz) {
      const T d22 = L.own[cs][PO_D22][lane];
      T d11 = 0, d51 = 0;
      if constexpr (PT) {
        d11 = L.own[cs][PO_D11][lane];
        d51 = L.own[cs][PO_D51][lane];
      }
      T M[NC];
#pragma unroll
      for (int v = 0; v < NC; v++) M[v] = L.own[cs][PO_M + comp[v]][lane];
      // both neighbours' inputs are read unconditionally (the indices are
      // inside the LDS rows for every lane), so the x and y reads share one
      // LDS round trip; a neighbour outside the domain contributes zero.
      // Components that apply_part does not use are not read.
      T Nx[5], Ny[5];
#pragma unroll
      for (int v = 0; v < 5; v++) {
        Nx[v] = L.N[nr][v][xi];
        Ny[v] = L.N[nr][v][yiN];
      }
      // the z neighbour is this lane's cell of the previous step: the
      // component of the other compute wave comes through LDS, and its split
      // Jacobian is still in that step's own slot (the loaders fill others)
      if constexpr (PT)
        zN[3] = L.N[nr][3][lane];
      else
        zN[0] = L.N[nr][0][lane];
      T ax[3], ay[3], az[3];
      apply_part<0, FWD, PT>(L.xc[ps], xi, Nx, ax);
      apply_part<1, FWD, PT>(L.yc[ps], yi, Ny, ay);
      apply_part<2, FWD, PT>(&L.own[ps][PO_Z], lane, zN, az);
      if (rim) {
#pragma unroll
        for (int v = 0; v < NC; v++) {
          ax[v] = x_dom ? ax[v] : T(0);
          ay[v] = y_dom ? ay[v] : T(0);
        }
      }
      if (tau < TI + TJ - 1) {  // a lane's first cell is at step off < TI + TJ - 1
#pragma unroll
        for (int v = 0; v < NC; v++) az[v] = kk > 0 ? az[v] : T(0);
      }
      T Lv[NC];
#pragma unroll
      for (int v = 0; v < NC; v++) {
        if constexpr (F64)
          Lv[v] = div_sp<FD>(ax[v], g.dXI, g.rXI) + div_sp<FD>(ay[v], g.dET, g.rET) + div_sp<FD>(az[v], g.dZT, g.rZT);
        else
          Lv[v] = ax[v] * fXI + ay[v] * fET + az[v] * fZT;
      }
      T out[NC];
      if constexpr (PT) {
        if (FWD) {
          out[0] = d11 * (M[0] - Lv[0]);
          out[1] = d51 * (M[0] - Lv[0]) + d22 * (M[1] - Lv[1]);
        } else {
          out[0] = M[0] - d11 * Lv[0];
          out[1] = M[1] - (d51 * Lv[0] + d22 * Lv[1]);
        }
      } else {
#pragma unroll
        for (int v = 0; v < NC; v++) out[v] = FWD ? d22 * (M[v] - Lv[v]) : M[v] - d22 * Lv[v];
      }
      // downstream tiles first: they are waiting
      if (hx) {
#pragma unroll
        for (int v = 0; v < NC; v++) st_coherent(Hx + comp[v] * 8, out[v]);
      }
      if (hy) {
#pragma unroll
        for (int v = 0; v < NC; v++) st_coherent(Hy + comp[v] * 8, out[v]);
      }
#pragma unroll
      for (int v = 0; v < NC; v++) {
        L.N[nw][comp[v]][lane] = out[v];
        zN[comp[v]] = out[v];
      }
    }
    Hx += HO_SLOT;
    Hy += HO_SLOT;
    lds_barrier();
    return ++tau < nsteps;
  });
}

// the split-Jacobian entries of one cell along x (along_x) or y, z from its
// summary; rr = rcp_rho(rho), T = P / rho
template <bool FWD, class T>
__device__ __forceinline__ SplitCoefT<T> coef_of(T P, T beta, T rho, T rr, T Tc, T U, T lam, T n, bool along_x) {
  T pd, p51;
  split_pd_p51(n, U, beta, rho, rr, &pd, &p51);
  SplitCoefT<T> c = diag_coef<1, FWD>(P, Tc, beta, U, lam, pd, p51, n);
  if (along_x) c.c5q = diag_coef<0, FWD>(P, Tc, beta, U, lam, pd, p51, n).c5q;
  return c;
}

// waves 0 .. 3 (r): the steps s = r (mod 4), each over four steps' time: D^-1
// at step s - 4 and to LDS with MR (forward) or NL (backward) at step s - 3,
// the x and y split-Jacobian entries at step s - 2, the z ones at step s - 1;
// then the loads of step s + 8.  A slot's D^-1 and M rows are last read at
// step s - 4, its entries at step s - 3.  Every turn issues the same loads
// (the step is clamped), so the compiler counts the loads in flight exactly
// and waits only for the oldest.
template <bool FWD, bool FD, class T>
__device__ __forceinline__ void pipe_loader(PipeLds<T>& L, const T* __restrict__ S, const T* __restrict__ SRC,
                                            const double* __restrict__ prof, const Geo& g, const Sk& q, int tile,
                                            int TY, int r, double deltaT) {
  static_assert(PIPE_SLOTS == 4, "one loader wave per slot");
  constexpr int NF = 5 + G_N, F = 5;  // SRC0..4, then the summary
  const int lane = threadIdx.x & 63;
  const int nsteps = q.nsteps;
  const long nf = q.nsk, row0 = (long)tile * nsteps * 64;
  // metric of the lane's j (clamped for columns outside the domain)
  const int j = min(2 + TY * TJ + (lane >> 3), g.ny);
  const T nx = T(pf(prof, g.Ym, SET_C, 1, j)), ny = T(pf(prof, g.Ym, SET_C, 5, j)),
          nz = T(pf(prof, g.Ym, SET_C, 9, j));
  T(*own)[64] = L.own[r];
  T buf[2][NF];
  T d11 = 0, d22 = 0, d51 = 0, rr = 0, Tc = 0;
  auto issue = [&](int s, auto sl) {
    const int sc = min(s, nsteps - 1);
    const long c = row0 + (long)(FWD ? sc : nsteps - 1 - sc) * 64;
#pragma unroll
    for (int f = 0; f < NF; f++) buf[sl][f] = ld_here((f < F ? SRC + c + (long)f * nf : S + c + (long)(f - F) * nf) + lane);
  };
  auto part = [&](auto which, auto sl) {
    constexpr int W = decltype(which)::value;
    const T(&d)[NF] = buf[sl];
    const T P = d[F + G_P], be = d[F + G_BETA], rho = d[F + G_RHO];
    if constexpr (W == 0) {
      diag_dinv<FD>(be, rho, d[F + G_LX], d[F + G_LY], d[F + G_LZ], g, deltaT, &d11, &d22, &d51);
    } else if constexpr (W == 1) {
      own[PO_D11][lane] = d11;
      own[PO_D22][lane] = d22;
      own[PO_D51][lane] = d51;
#pragma unroll
      for (int f = 0; f < F; f++) own[PO_M + f][lane] = d[f];
      rr = rcp_rho(rho);
      Tc = over_rho(P, rho, rr);
    } else if constexpr (W == 2) {
      coef_store(L.xc[r], lane, coef_of<FWD>(P, be, rho, rr, Tc, d[F + G_UX], d[F + G_LX], nx, true));
      coef_store(L.yc[r], lane, coef_of<FWD>(P, be, rho, rr, Tc, d[F + G_UY], d[F + G_LY], ny, false));
    } else {
      coef_store(&own[PO_Z], lane, coef_of<FWD>(P, be, rho, rr, Tc, d[F + G_UZ], d[F + G_LZ], nz, false));
    }
  };
  issue(r, Int<0>{});
  issue(r + 4, Int<1>{});
  for_each<4>([&](auto k) { part(k, Int<0>{}); });
  issue(r + 8, Int<0>{});
  lds_barrier();
  int tau = 0;
  for (; tau < r; tau++) lds_barrier();  // nsteps > 3 in every grid
  cycle<8>([&](auto k) -> bool {
    constexpr int W = decltype(k)::value % 4;
    const Int<1 - decltype(k)::value / 4> sl;
    part(Int<W>{}, sl);
    if constexpr (W == 3) issue(tau + 9, sl);  // the step at hand is tau + 1
    lds_barrier();
    return ++tau < nsteps;
  });
}

// The halo has 16 consumer lanes of the compute waves: 0..7 on the x edge
// (b = c) and 8..15 on the y edge (a = c - 8).
template <bool FWD>
struct HaloLane {
  int dir, idx, a, b, off;
  bool ok;  // the consumer is a cell of the domain and has this neighbour
  __device__ __forceinline__ HaloLane(int dir_, int idx_, const Geo& g, int TX, int TY) : dir(dir_), idx(idx_) {
    a = dir == 0 ? (FWD ? 0 : TI - 1) : idx;
    b = dir == 0 ? idx : (FWD ? 0 : TJ - 1);
    const int i = 3 + TX * TI + a, j = 2 + TY * TJ + b;
    const bool dom = dir == 0 ? (FWD ? i - 1 >= 3 : i + 1 <= g.gend) : (FWD ? j - 1 >= 2 : j + 1 <= g.ny);
    ok = i <= g.gend && j <= g.ny && dom;
    off = FWD ? a + b : (TI - 1 - a) + (TJ - 1 - b);
  }
  __device__ __forceinline__ bool live(int sig, const Sk& q) const {
    const int kk = sig - off;
    return ok && kk >= 0 && kk < q.Nz;
  }
};

// wave 9: the split-Jacobian entries of the cross-tile neighbours, from their
// summaries (along x the compact edge copy, along y the neighbour tile's row), into the halo columns of slot sig - 1.
// Lane 16 d + c serves consumer c at step 4 m + d.  The entries of steps
// 4 m .. 4 m + 2 go to LDS during step 4 m - 1, those of step 4 m + 3, whose
// slot is still being read then, during step 4 m.
template <bool FWD, class T>
__device__ __forceinline__ void pipe_halo_coef(PipeLds<T>& L, const T* __restrict__ S, const T* __restrict__ E,
                                               const double* __restrict__ prof, const Geo& g, const Sk& q, int tile,
                                               int TX, int TY) {
  static_assert(PIPE_SLOTS == 4, "four steps of 16 lanes");
  const int lane = threadIdx.x & 63, c = lane & 15, d4 = lane >> 4;
  const HaloLane<FWD> h(c >> 3, c & 7, g, TX, TY);
  const int nsteps = q.nsteps;
  const long nf = q.nsk;
  static_assert(HO_SLOT == 64, "a step is 64 elements on in the edge copy and in the rows");
  // metric at the remote cell's j
  const int j = 2 + TY * TJ + h.b;
  const int jr = h.dir == 0 ? j : (FWD ? j - 1 : j + 1);
  const T n = T(pf(prof, g.Ym, SET_C, h.dir == 0 ? 1 : 5, min(max(jr, 0), g.Ym - 1)));
  // field f of the neighbour at its (forward) step p: fld[f] + p * 64; a
  // consumer without a neighbour reads its own tile's
  const int px = h.ok ? (FWD ? tile - 1 : tile + 1) : tile, py = h.ok ? (FWD ? tile - q.nTI : tile + q.nTI) : tile;
  const T* fld[5];
#pragma unroll
  for (int f = 0; f < 5; f++)
    fld[f] = h.dir == 0 ? E + ho_at(q, px, FWD ? 0 : 1, 0) + 8 * f + h.idx
                        : S + (long)(f < 3 ? G_P + f : G_UY + f - 3) * nf + sk_at(q, py, 0, (FWD ? 56 : 0) + h.idx);
  T(*row)[72] = (h.dir == 0 ? L.xc : L.yc)[(d4 + 3) % PIPE_SLOTS];
  T buf[2][5];
  auto issue = [&](int s0, auto sl) {
    // the consumer's step sig uses what the neighbour's walk has at sig + 7
    const int sc = min(s0 + d4 + 7, nsteps - 1);
    const long o = (long)(FWD ? sc : nsteps - 1 - sc) * 64;
#pragma unroll
    for (int f = 0; f < 5; f++) buf[sl][f] = ld_here(fld[f] + o);
  };
  SplitCoefT<T> cf;
  auto form = [&](auto sl) {
    const T(&d)[5] = buf[sl];
    const T rr = rcp_rho(d[2]);
    cf = coef_of<FWD>(d[0], d[1], d[2], rr, over_rho(d[0], d[2], rr), d[3], d[4], n, h.dir == 0);
  };
  issue(0, Int<0>{});
  issue(4, Int<1>{});
  form(Int<0>{});
  if (d4 < 3) coef_store(row, 64 + h.idx, cf);
  lds_barrier();
  int tau = 0;
  cycle<8>([&](auto k) -> bool {
    constexpr int K = decltype(k)::value % 4, B = decltype(k)::value / 4;
    if constexpr (K == 0) {
      if (d4 == 3) coef_store(row, 64 + h.idx, cf);
      issue(tau + 8, Int<B>{});
    } else if constexpr (K == 3) {
      form(Int<1 - B>{});
      if (d4 < 3) coef_store(row, 64 + h.idx, cf);
    }
    lds_barrier();
    return ++tau < nsteps;
  });
}

// The 80 values a tile takes over per step (x edge, then y edge: 5 components
// x 8 cells each): lane l has values l and, below lane 16, 64 + l.  p0, p1:
// their producers' slots of step 0.
template <bool FWD, class T>
struct HaloValues {
  int r0, r1;
  bool two;
  HaloLane<FWD> h0, h1;
  T *p0, *p1;
  __device__ __forceinline__ HaloValues(T* __restrict__ H, const Geo& g, const Sk& q, int tile, int TX, int TY, int lane)
      : r0(lane < 40 ? lane : lane - 40),
        r1(lane + 24),
        two(lane < 16),
        h0(lane < 40 ? 0 : 1, r0 & 7, g, TX, TY),
        h1(1, r1 & 7, g, TX, TY) {
    const int px = FWD ? tile - 1 : tile + 1, py = FWD ? tile - q.nTI : tile + q.nTI;
    p0 = H + ho_at(q, h0.ok ? (h0.dir == 0 ? px : py) : tile, h0.dir, 0) + r0;
    p1 = two ? H + ho_at(q, h1.ok ? py : tile, 1, 0) + r1 : p0;
  }
  __device__ __forceinline__ bool live0(int sig, const Sk& q) const { return h0.live(sig, q); }
  __device__ __forceinline__ bool live1(int sig, const Sk& q) const { return two && h1.live(sig, q); }
  // the consumer's step sig reads what the producer formed at its step sig + 7
  __device__ __forceinline__ static long slot(int sig, const Sk& q) {
    return (long)min(sig + 7, q.nsteps - 1) * HO_SLOT;
  }
};

// waves 6 and 7 (odd): the cross-tile neighbours' outputs of every second
// step, polled.  A coherent load takes about a microsecond, two steps' time,
// so each wave has its next step's load in flight while the other takes its
// own over.  Looking further ahead lengthens every hop instead: a tile that
// finds a value missing waits, and so falls behind its upstream tiles until
// its loads, issued that much earlier, succeed.
template <bool FWD, class T>
__device__ __forceinline__ void pipe_halo_poll(PipeLds<T>& L, T* __restrict__ H, const Geo& g, const Sk& q, int tile,
                                               int TX, int TY, int odd, int* err, long spin_limit) {
  const int lane = threadIdx.x & 63;
  const int nsteps = q.nsteps;
  const HaloValues<FWD, T> hv(H, g, q, tile, TX, TY, lane);
  T *p0 = hv.p0, *p1 = hv.p1;
  // step sig's values go to the half of N that step sig - 1 fills
  T* l0 = &L.N[odd ^ 1][min(hv.r0 >> 3, 4)][(hv.h0.dir == 0 ? 64 : 72) + hv.h0.idx];
  T* l1 = &L.N[odd ^ 1][min(hv.r1 >> 3, 4)][72 + hv.h1.idx];
  T v0, v1;
  auto issue = [&](int sig) {
    const long s = hv.slot(sig, q);
    v0 = ld_coherent(p0 + s);
    v1 = ld_coherent(p1 + s);  // a lane without a second value reads its first again
  };
  auto consume = [&](int sig) {
    const bool lv0 = hv.live0(sig, q), lv1 = hv.live1(sig, q);
    bool pend = (lv0 && is_sentinel(v0)) || (lv1 && is_sentinel(v1));
    long cnt = 0;
    while (__any(pend)) {
      // one memory round trip per poll: the pending outputs and the error
      // flag (set by a tile that gave up) are loaded together
      const int e = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      issue(sig);
      pend = (lv0 && is_sentinel(v0)) || (lv1 && is_sentinel(v1));
      if (__builtin_amdgcn_readfirstlane(e) != 0 || ++cnt > spin_limit) {
        if (lane == 0) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    if (lv0) *l0 = v0;
    if (lv1) *l1 = v1;
  };
  issue(odd);
  // step sig is taken over during step sig - 1 (step 0 before the first);
  // `left` barriers remain of the nsteps + 1 every wave passes
  int left = nsteps + 1, sig = odd;
  if (odd) {
    lds_barrier();
    left--;
  }
  for (;;) {
    consume(sig);  // past the last step no value is live
    sig += 2;
    issue(sig);
    lds_barrier();
    if (--left == 0) break;
    lds_barrier();
    if (--left == 0) break;
  }
}

// wave 8: writes the outputs of the step before the one being computed to
// their rows of DST (from the LDS half that the compute waves fill again only
// after the next barrier) and sets the hand-off slots that waves 6, 7 have read
// back to the sentinel.  It waits for no load, so these stores delay nobody:
// stores and loads share one counter, and a wave that waits for a load waits
// for its earlier stores too.
template <bool FWD, class T>
__device__ __forceinline__ void pipe_writer(PipeLds<T>& L, T* __restrict__ DST, T* __restrict__ H, const Geo& g,
                                            const Sk& q, int tile, int TX, int TY) {
  const int lane = threadIdx.x & 63;
  const int a = lane & 7, b = lane >> 3;
  const int nsteps = q.nsteps;
  const long nf = q.nsk, row0 = (long)tile * nsteps * 64;
  const bool col = 3 + TX * TI + a <= g.gend && 2 + TY * TJ + b <= g.ny;
  const int off = FWD ? a + b : (TI - 1 - a) + (TJ - 1 - b);
  const T sv = sentinel_value<T>();
  const HaloValues<FWD, T> hv(H, g, q, tile, TX, TY, lane);
  auto store_out = [&](int s, auto half) {
    const int kk = s - off;
    if (col && kk >= 0 && kk < q.Nz) {
      T* r = DST + row0 + (long)(FWD ? s : nsteps - 1 - s) * 64;
#pragma unroll
      for (int v = 0; v < 5; v++) (r + (long)v * nf)[lane] = L.N[half][v][lane];
    }
  };
  lds_barrier();
  int tau = 0;
  cycle<2>([&](auto k) -> bool {
    store_out(tau - 1, Int<1 - decltype(k)::value>{});
    const long s = hv.slot(tau, q);
    if (hv.live0(tau, q)) st_coherent(hv.p0 + s, sv);
    if (hv.live1(tau, q)) st_coherent(hv.p1 + s, sv);
    lds_barrier();
    return ++tau < nsteps;
  });
  if (nsteps & 1)
    store_out(nsteps - 1, Int<0>{});
  else
    store_out(nsteps - 1, Int<1>{});
}

template <bool FWD, bool FD, class T>
__device__ __forceinline__ void pipe_tile(PipeLds<T>& L, const T* __restrict__ S, const T* __restrict__ SRC,
                                          T* __restrict__ DST, T* __restrict__ H, const T* __restrict__ E,
                                          const double* __restrict__ prof, const Geo& g, const Sk& q, int tile,
                                          int* err, long spin_limit, double deltaT) {
  const int TX = tile % q.nTI, TY = tile / q.nTI;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  switch (wave) {
    case 4:
      __builtin_amdgcn_s_setprio(3);  // the step waits for these four
      pipe_compute<FWD, FD, true>(L, H, g, q, tile, TX, TY);
      break;
    case 5:
      __builtin_amdgcn_s_setprio(3);
      pipe_compute<FWD, FD, false>(L, H, g, q, tile, TX, TY);
      break;
    case 6:
    case 7:
      __builtin_amdgcn_s_setprio(3);
      pipe_halo_poll<FWD>(L, H, g, q, tile, TX, TY, wave - 6, err, spin_limit);
      break;
    case 8: pipe_writer<FWD>(L, DST, H, g, q, tile, TX, TY); break;
    case 9: pipe_halo_coef<FWD>(L, S, E, prof, g, q, tile, TX, TY); break;
    default: pipe_loader<FWD, FD>(L, S, SRC, prof, g, q, tile, TY, wave, deltaT); break;
  }
}

template <bool FWD, class T>
__global__ void __launch_bounds__(PIPE_THREADS) k_sweep_pipe(const T* __restrict__ S, const T* __restrict__ SRC,
                                                             T* __restrict__ DST, T* __restrict__ H,
                                                             const T* __restrict__ E,
                                                             const double* __restrict__ prof, Geo g, Sk q,
                                                             const int* __restrict__ order, int* __restrict__ sync,
                                                             long spin_limit, double deltaT) {
  // arrays in sweep order (Sk); S holds the DiagField summary, E its copy of
  // the x edges, H the hand-off slots
  // FWD: SRC = MR, DST = NL   (NL = D^-1 (MR - L))
  // BWD: SRC = NL, DST = NR   (NR = NL - D^-1 U); the two may be the same rows,
  // since a thread reads the one or writes the other (without __restrict__ the
  // FP32 sweeps took 514 / 490 us at 256x192x256 for 494 / 473)
  __shared__ PipeLds<T> L;
  if (threadIdx.x == 0) L.ticket = atomicAdd(sync, 1);
  __syncthreads();
  // the ticket is the same for all lanes: rows and slots get scalar addresses
  const int t = __builtin_amdgcn_readfirstlane(L.ticket);
  if (t >= q.ntiles) return;
  const int tile = order[FWD ? t : q.ntiles - 1 - t];
  // the kernel arguments make this choice uniform: one scalar branch
  if constexpr (std::is_same<T, double>::value) {
    if (g.fast_div) {
      pipe_tile<FWD, true>(L, S, SRC, DST, H, E, prof, g, q, tile, sync + 1, spin_limit, deltaT);
      return;
    }
  }
  pipe_tile<FWD, false>(L, S, SRC, DST, H, E, prof, g, q, tile, sync + 1, spin_limit, deltaT);
}

// every hand-off slot set to the sentinel: a new buffer, or after a sweep that
// gave up (a sweep that ends leaves them so); two steps of a tile per block
template <class T>
__global__ void __launch_bounds__(256) k_seed_hand_off(T* __restrict__ H, Sk q) {
  const int dir = (threadIdx.x >> 6) & 1, s = blockIdx.x * 2 + (threadIdx.x >> 7);
  if (s < q.nsteps) H[ho_at(q, blockIdx.y, dir, s) + (threadIdx.x & 63)] = sentinel_value<T>();
}

// ---------------------------------------------------------------------------
// DPLUSGS (DPLUSGS.cpp:488-1140): point-Jacobi sweeps over all interior
// cells at once, NR = D^-1 (MR - L NL - U NL) with the split Jacobians of
// the neighbours; the upper neighbours' NL is read at j+1, k+1 (where the
// reference reads their states; its NL indices j_, k_ are never assigned)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_jacobi(const double* __restrict__ Ui, const double* __restrict__ MR,
                                                const double* __restrict__ NLin, double* __restrict__ NRout,
                                                const double* __restrict__ prof, Geo g, double deltaT) {
  const int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  const int i = 3 + blockIdx.z;
  if (k > g.nz || j > g.ny) return;
  const long nf = g.nf;
  const long c = at(g, i, j, k);
  const double dd[3] = {g.dXI, g.dET, g.dZT};
  double lo[3][5], hi[3][5];
#pragma unroll
  for (int side = 0; side < 2; side++) {
#pragma unroll
    for (int dir = 0; dir < 3; dir++) {
      double(&acc)[5] = side == 0 ? lo[dir] : hi[dir];
      const long st = dir == 0 ? g.plane : (dir == 1 ? (long)g.Zp : 1L);
      const long nb = side == 0 ? c - st : c + st;
      const bool inside = side == 0 ? (dir == 0 ? i - 1 >= 3 : dir == 1 ? j - 1 >= 2 : k - 1 >= 2)
                                    : (dir == 0 ? i + 1 <= g.gend : dir == 1 ? j + 1 <= g.ny : k + 1 <= g.nz);
      if (!inside) {
        // ghost neighbours: NL is zero there
#pragma unroll
        for (int v = 0; v < 5; v++) acc[v] = 0.0;
        continue;
      }
      const int jn = dir == 1 ? (side == 0 ? j - 1 : j + 1) : j;
      double u5[5], N[5];
      ld5(Ui, nf, nb, u5);
      ld5(NLin, nf, nb, N);
      PState s = prim_dt(u5[0], u5[1], u5[2], u5[3], u5[4], pf(prof, g.Ym, SET_C, 0, jn));
      Split a = split_jac(s, pf(prof, g.Ym, SET_C, 1 + 3 * dir, jn), pf(prof, g.Ym, SET_C, 2 + 3 * dir, jn),
                          pf(prof, g.Ym, SET_C, 3 + 3 * dir, jn), dir);
      if (side == 0) lower_sum(a, N, acc); else upper_sum(a, N, acc);
    }
  }
  double LL[5], UU[5];
#pragma unroll
  for (int v = 0; v < 5; v++) {
    LL[v] = lo[0][v] / dd[0] + lo[1][v] / dd[1] + lo[2][v] / dd[2];
    UU[v] = hi[0][v] / dd[0] + hi[1][v] / dd[1] + hi[2][v] / dd[2];
  }
  double u5[5], m9[9], d11, d22, d51;
  ld5(Ui, nf, c, u5);
  PState s0 = prim_dt(u5[0], u5[1], u5[2], u5[3], u5[4], pf(prof, g.Ym, SET_C, 0, j));
  cell_metric(prof, g.Ym, j, m9);
  dinv(s0, m9, g.dXI, g.dET, g.dZT, deltaT, &d11, &d22, &d51);
  double M[5];
  ld5(MR, nf, c, M);
  NRout[c] = d11 * (M[0] - LL[0] - UU[0]);
  NRout[nf + c] = d22 * (M[1] - LL[1] - UU[1]);
  NRout[2 * nf + c] = d22 * (M[2] - LL[2] - UU[2]);
  NRout[3 * nf + c] = d22 * (M[3] - LL[3] - UU[3]);
  NRout[4 * nf + c] = d51 * (M[0] - LL[0] - UU[0]) + d22 * (M[4] - LL[4] - UU[4]);
}

// The same sweep for diagonal metrics from a summary of every interior cell,
// formed once for the four sweeps: P, beta, rho and the three contravariant
// velocities.  A neighbour is then nine loads, one division and one square root
// in place of its primitives and split Jacobian with a dozen divisions, six
// times per cell and sweep.  Bound by memory: the six neighbours' fields miss
// the L2 by half, so stored spectral radii (nine fields) cost more than their
// roots, 106 us a sweep.  128x96x128: 154 -> 100 us a sweep, and 34 for the
// summary.  S: jacobi_summary_elems doubles.
__global__ void __launch_bounds__(256) k_jacobi_summary(const double* __restrict__ Ui, const double* __restrict__ prof,
                                                        double* __restrict__ S, Geo g) {
  const int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  const int i = 3 + blockIdx.z;
  if (k > g.nz || j > g.ny) return;
  const long c = at(g, i, j, k);
  double u5[5], v[G_N];
  ld5(Ui, g.nf, c, u5);
  prep_summary(u5, prof, g, j, v);
  S[c] = v[G_P];
  S[g.nf + c] = v[G_BETA];
  S[2 * g.nf + c] = v[G_RHO];
#pragma unroll
  for (int d = 0; d < 3; d++) S[(3 + d) * g.nf + c] = v[G_UX + 2 * d];
}

// neighbour p along direction d from that summary; n: the diagonal metric entry at its j
__device__ __forceinline__ DNb jacobi_nb(const double* __restrict__ S, long nf, long p, int d, double n) {
  DNb c;
  const double rho = S[2 * nf + p];
  const double rr = rcp_rho(rho);
  c.P = S[p];
  c.T = over_rho(c.P, rho, rr);
  c.beta = S[nf + p];
  c.U = S[(3 + d) * nf + p];
  c.lam = lambda_of(c.U, c.beta, over_rho(KG * c.P, rho, rr), n * n);
  split_pd_p51(n, c.U, c.beta, rho, rr, &c.pd, &c.p51);
  return c;
}

constexpr int JAC_JG = 4;  // blocks along j that a walk along i takes with it

__global__ void __launch_bounds__(256) k_jacobi_diag(const double* __restrict__ S, const double* __restrict__ MR,
                                                     const double* __restrict__ NLin, double* __restrict__ NRout,
                                                     const double* __restrict__ prof, Geo g, double deltaT) {
  int bx, by, bz;
  xcd_block3(&bx, &by, &bz);
  // grid (k blocks x JAC_JG, i, groups along j): consecutive blocks walk i, so
  // that the i neighbours' planes of a group are still in the L2 (256x192x256:
  // 3% of an iteration against whole planes, 1 to 8 blocks within 2%)
  const int nkb = gridDim.x / JAC_JG;
  const int k = 2 + (bx % nkb) * blockDim.x + threadIdx.x;
  const int j = 2 + (bz * JAC_JG + bx / nkb) * blockDim.y + threadIdx.y;
  const int i = 3 + by;
  if (k > g.nz || j > g.ny) return;
  const long nf = g.nf;
  const long c = at(g, i, j, k);
  double lo[3][5], hi[3][5];
  for_each<3>([&](auto d) {
    constexpr int D = decltype(d)::value;
    const long st = D == 0 ? g.plane : (D == 1 ? (long)g.Zp : 1L);
    const bool in_lo = D == 0 ? i - 1 >= 3 : D == 1 ? j - 1 >= 2 : k - 1 >= 2;
    const bool in_hi = D == 0 ? i + 1 <= g.gend : D == 1 ? j + 1 <= g.ny : k + 1 <= g.nz;
#pragma unroll
    for (int v = 0; v < 5; v++) lo[D][v] = hi[D][v] = 0.0;  // ghost neighbours: NL is zero there
    double N[5];
    if (in_lo) {
      const double n = pf(prof, g.Ym, SET_C, 1 + 4 * D, D == 1 ? j - 1 : j);
      ld5(NLin, nf, c - st, N);
      lower_diag<D>(jacobi_nb(S, nf, c - st, D, n), n, N, lo[D]);
    }
    if (in_hi) {
      const double n = pf(prof, g.Ym, SET_C, 1 + 4 * D, D == 1 ? j + 1 : j);
      ld5(NLin, nf, c + st, N);
      upper_diag<D>(jacobi_nb(S, nf, c + st, D, n), n, N, hi[D]);
    }
  });
  double LL[5], UU[5];
#pragma unroll
  for (int v = 0; v < 5; v++) {
    LL[v] = div_rn(lo[0][v], g.dXI, g.rXI) + div_rn(lo[1][v], g.dET, g.rET) + div_rn(lo[2][v], g.dZT, g.rZT);
    UU[v] = div_rn(hi[0][v], g.dXI, g.rXI) + div_rn(hi[1][v], g.dET, g.rET) + div_rn(hi[2][v], g.dZT, g.rZT);
  }
  double d11, d22, d51;
  const double beta = S[nf + c], rho = S[2 * nf + c], C = over_rho(KG * S[c], rho, rcp_rho(rho));
  double lam[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const double n = pf(prof, g.Ym, SET_C, 1 + 4 * d, j);
    lam[d] = lambda_of(S[(3 + d) * nf + c], beta, C, n * n);
  }
  diag_dinv<false>(beta, rho, lam[0], lam[1], lam[2], g, deltaT, &d11, &d22, &d51);
  double M[5];
  ld5(MR, nf, c, M);
  NRout[c] = d11 * (M[0] - LL[0] - UU[0]);
  NRout[nf + c] = d22 * (M[1] - LL[1] - UU[1]);
  NRout[2 * nf + c] = d22 * (M[2] - LL[2] - UU[2]);
  NRout[3 * nf + c] = d22 * (M[3] - LL[3] - UU[3]);
  NRout[4 * nf + c] = d51 * (M[0] - LL[0] - UU[0]) + d22 * (M[4] - LL[4] - UU[4]);
}

// Initial iterate of a physical step from the time levels, on the interior:
// order 1: 2 U^n - U^{n-1}; order 2: 3 U^n - 3 U^{n-1} + U^{n-2}; order 3:
// 4 U^n - 6 U^{n-1} + 4 U^{n-2} - U^{n-3}.  The reference starts every
// physical step at U^n (main.cpp:444-464).
__global__ void k_extrapolate(double* __restrict__ Ui, const double* __restrict__ Un, const double* __restrict__ Uq,
                              const double* __restrict__ Uqq, const double* __restrict__ U3, Geo g, int order) {
  const int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  const int i = 3 + blockIdx.z;
  if (k > g.nz || j > g.ny) return;
  const long c = at(g, i, j, k);
#pragma unroll
  for (int v = 0; v < 5; v++) {
    const long o = v * g.nf + c;
    Ui[o] = order == 3   ? 4 * Un[o] - 6 * Uq[o] + 4 * Uqq[o] - U3[o]
            : order == 2 ? 3 * Un[o] - 3 * Uq[o] + Uqq[o]
                         : 2 * Un[o] - Uq[o];
  }
}

__global__ void k_copy_interior(const double* __restrict__ src, double* __restrict__ dst, Geo g) {
  int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  int j = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  int i = 3 + blockIdx.z;
  if (k > g.nz || j > g.ny) return;
  long c = at(g, i, j, k);
#pragma unroll
  for (int v = 0; v < 5; v++) dst[v * g.nf + c] = src[v * g.nf + c];
}

// ---------------------------------------------------------------------------
// update + residual norms: Dual_time_stepping.cpp:1290-1352.  Pass 1 writes
// one partial sum of dq^4 per block and component (fixed tree order); pass 2
// adds the partials in index order, so repeated runs give identical bits.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_update(double* __restrict__ Ui, const double* __restrict__ NR,
                                                const double* __restrict__ prof, double* __restrict__ partial, Geo g) {
  __shared__ double red[5][256];
  int tid = threadIdx.y * blockDim.x + threadIdx.x;
  int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  int j = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  int i = 3 + blockIdx.z;
  double r[5] = {0, 0, 0, 0, 0};
  if (k <= g.nz && j <= g.ny) {
    const long nf = g.nf;
    long c = at(g, i, j, k);
    double J = pf(prof, g.Ym, SET_C, 0, j);
    double U1 = Ui[c], U2 = Ui[nf + c], U3 = Ui[2 * nf + c], U4 = Ui[3 * nf + c], U5 = Ui[4 * nf + c];
    double rhoold = U1 * J;
    double Uold = U2 / U1, Vold = U3 / U1, Wold = U4 / U1;
    double VVold = Uold * Uold + Vold * Vold + Wold * Wold;
    double Pold = (U5 * J - 0.5 * rhoold * VVold) * (KG - 1);
    double Told = Pold / rhoold;
    double P = Pold + NR[c] * J;
    double Uu = Uold + NR[nf + c] * J;
    double V = Vold + NR[2 * nf + c] * J;
    double W = Wold + NR[3 * nf + c] * J;
    double T = Told + NR[4 * nf + c] * J;
    double rho = P / T;
    Ui[c] = rho / J;
    Ui[nf + c] = rho * Uu / J;
    Ui[2 * nf + c] = rho * V / J;
    Ui[3 * nf + c] = rho * W / J;
    Ui[4 * nf + c] = (P / (KG - 1) + 0.5 * rho * (Uu * Uu + V * V + W * W)) / J;
    double q[5] = {(P - Pold) * (P - Pold), (Uu - Uold) * (Uu - Uold), (V - Vold) * (V - Vold),
                   (W - Wold) * (W - Wold), (T - Told) * (T - Told)};
#pragma unroll
    for (int v = 0; v < 5; v++) r[v] = q[v] * q[v];
  }
#pragma unroll
  for (int v = 0; v < 5; v++) red[v][tid] = r[v];
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s)
#pragma unroll
      for (int v = 0; v < 5; v++) red[v][tid] += red[v][tid + s];
    __syncthreads();
  }
  if (tid == 0) {
    long b = ((long)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
#pragma unroll
    for (int v = 0; v < 5; v++) partial[b * 5 + v] = red[v][0];
  }
}

// The primitive update (Dual_time_stepping.cpp:1290-1352) with NR read from
// the sweep order through LDS: a block
// covers PC steps of one tile (as k_sweep_prep does), loads those NR rows
// coalesced, then walks each column's run of PC consecutive k in the natural
// layout.  Per-block partial sums of the residuals, in a fixed order.
template <class R>
__global__ void __launch_bounds__(256) k_update_sk(double* __restrict__ Ui, const R* __restrict__ NR,
                                                   const double* __restrict__ prof, double* __restrict__ partial,
                                                   Geo g, Sk q) {
  __shared__ double L[5][64][PCP];
  __shared__ double red[5][256];
  const int tid = threadIdx.x;
  int bx, by, bz;
  xcd_block3(&bx, &by, &bz);
  const int tile = by, s0 = bx * PC;
  const int TX = tile % q.nTI, TY = tile / q.nTI;
  for (int idx = tid; idx < PC * 64; idx += blockDim.x) {
    const int t = idx >> 6, lane = idx & 63, s = s0 + t;
    if (s >= q.nsteps) continue;
    const long o = sk_at(q, tile, s, lane);
#pragma unroll
    for (int f = 0; f < 5; f++) L[f][lane][t] = double(NR[f * q.nsk + o]);
  }
  __syncthreads();
  double r[5] = {0, 0, 0, 0, 0};
  const long nf = g.nf;
  for (int idx = tid; idx < 64 * PC; idx += blockDim.x) {
    const int col = idx / PC, t = idx - col * PC;
    const int a = col & 7, b = col >> 3;
    const int i = 3 + TX * TI + a, j = 2 + TY * TJ + b, kk = s0 - a - b + t;
    if (i > g.gend || j > g.ny || kk < 0 || kk >= q.Nz) continue;
    const long c = at(g, i, j, 2 + kk);
    const double J = pf(prof, g.Ym, SET_C, 0, j);
    const double U1 = Ui[c], U2 = Ui[nf + c], U3 = Ui[2 * nf + c], U4 = Ui[3 * nf + c], U5 = Ui[4 * nf + c];
    const double rhoold = U1 * J;
    const double Uold = U2 / U1, Vold = U3 / U1, Wold = U4 / U1;
    const double VVold = Uold * Uold + Vold * Vold + Wold * Wold;
    const double Pold = (U5 * J - 0.5 * rhoold * VVold) * (KG - 1);
    const double Told = Pold / rhoold;
    const double P = Pold + L[0][col][t] * J;
    const double Uu = Uold + L[1][col][t] * J;
    const double V = Vold + L[2][col][t] * J;
    const double W = Wold + L[3][col][t] * J;
    const double T = Told + L[4][col][t] * J;
    const double rho = P / T;
    Ui[c] = rho / J;
    Ui[nf + c] = rho * Uu / J;
    Ui[2 * nf + c] = rho * V / J;
    Ui[3 * nf + c] = rho * W / J;
    Ui[4 * nf + c] = (P / (KG - 1) + 0.5 * rho * (Uu * Uu + V * V + W * W)) / J;
    const double d[5] = {(P - Pold) * (P - Pold), (Uu - Uold) * (Uu - Uold), (V - Vold) * (V - Vold),
                         (W - Wold) * (W - Wold), (T - Told) * (T - Told)};
#pragma unroll
    for (int v = 0; v < 5; v++) r[v] += d[v] * d[v];
  }
#pragma unroll
  for (int v = 0; v < 5; v++) red[v][tid] = r[v];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (tid < h)
#pragma unroll
      for (int v = 0; v < 5; v++) red[v][tid] += red[v][tid + h];
    __syncthreads();
  }
  if (tid == 0) {
    const long blk = (long)by * gridDim.x + bx;
#pragma unroll
    for (int v = 0; v < 5; v++) partial[blk * 5 + v] = red[v][0];
  }
}

// out[0..4]: the norms; out[5], out[6]: the forward and backward tiled
// sweeps' error flags (0 without them), so that one copy brings back both
__global__ void __launch_bounds__(1024) k_reduce_partials(const double* __restrict__ partial, long nblocks,
                                                          double* __restrict__ out, double DN,
                                                          const int* __restrict__ fa, const int* __restrict__ fb) {
  __shared__ double red[5][1024];
  int tid = threadIdx.x;
  double s[5] = {0, 0, 0, 0, 0};
  for (long b = tid; b < nblocks; b += 1024)
#pragma unroll
    for (int v = 0; v < 5; v++) s[v] += partial[b * 5 + v];
#pragma unroll
  for (int v = 0; v < 5; v++) red[v][tid] = s[v];
  __syncthreads();
  for (int st = 512; st > 0; st >>= 1) {
    if (tid < st)
#pragma unroll
      for (int v = 0; v < 5; v++) red[v][tid] += red[v][tid + st];
    __syncthreads();
  }
  if (tid < 5) out[tid] = sqrt(red[tid][0]) * DN;
  else if (tid == 5) out[5] = fa ? double(*fa) : 0.;
  else if (tid == 6) out[6] = fb ? double(*fb) : 0.;
}

// ---------------------------------------------------------------------------
// host arrays <-> device fields through a contiguous staging copy.  A copy
// between the host and rows of another pitch moves one row (Zm doubles) at a
// time, about 0.15 ms each here; a contiguous copy runs at the link's rate
// (18-30 GB/s from pageable memory) and these passes at HBM's.
// ---------------------------------------------------------------------------
// reference layout (rows of Zm) -> device rows of Zp, blockIdx.y the field;
// the padding is left alone
__global__ void __launch_bounds__(256) k_rows_in(const double* __restrict__ src, double* __restrict__ dst, Geo g,
                                                 unsigned n) {
  for (unsigned e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
    const unsigned row = e / (unsigned)g.Zm, k = e - row * (unsigned)g.Zm;
    dst[blockIdx.y * g.nf + (long)row * g.Zp + k] = src[(long)blockIdx.y * n + e];
  }
}

__global__ void __launch_bounds__(256) k_rows_out(const double* __restrict__ src, double* __restrict__ dst, Geo g,
                                                  unsigned n) {
  for (unsigned e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
    const unsigned row = e / (unsigned)g.Zm, k = e - row * (unsigned)g.Zm;
    dst[(long)blockIdx.y * n + e] = src[blockIdx.y * g.nf + (long)row * g.Zp + k];
  }
}

// interior Q [X][Y][Z] -> U = Q / J in the device layout, zero elsewhere
__global__ void __launch_bounds__(256) k_q_in(const double* __restrict__ Q, const double* __restrict__ J,
                                              double* __restrict__ U, Geo g) {
  const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, i = blockIdx.z;
  if (k >= g.Zp || j >= g.Ym) return;
  const int X = g.gend - 2, Y = g.ny - 1, Z = g.nz - 1;
  const bool in = i >= 3 && i <= g.gend && j >= 2 && j <= g.ny && k >= 2 && k <= g.nz;
  const long c = at(g, i, j, k), e = ((long)(i - 3) * Y + (j - 2)) * Z + (k - 2), n = (long)X * Y * Z;
#pragma unroll
  for (int v = 0; v < 5; v++) U[v * g.nf + c] = in ? Q[v * n + e] / J[j] : 0.0;
}

// Q = U J of the interior, [X][Y][Z]
__global__ void __launch_bounds__(256) k_q_out(const double* __restrict__ U, const double* __restrict__ J,
                                               double* __restrict__ Q, Geo g) {
  const int k = 2 + blockIdx.x * 64 + threadIdx.x, j = 2 + blockIdx.y * 4 + threadIdx.y, i = 3 + blockIdx.z;
  if (k > g.nz || j > g.ny) return;
  const int X = g.gend - 2, Y = g.ny - 1, Z = g.nz - 1;
  const long c = at(g, i, j, k), e = ((long)(i - 3) * Y + (j - 2)) * Z + (k - 2), n = (long)X * Y * Z;
#pragma unroll
  for (int v = 0; v < 5; v++) Q[v * n + e] = U[v * g.nf + c] * J[j];
}

// ---------------------------------------------------------------------------
// host-side launchers
// ---------------------------------------------------------------------------
static inline dim3 box_grid(int nk, int nj, int ni, dim3 blk) {
  return dim3((nk + blk.x - 1) / blk.x, (nj + blk.y - 1) / blk.y, ni);
}

static dim3 row_grid(long n, int fields) { return dim3((unsigned)std::min((n + 255) / 256, 4096L), fields); }

void launch_rows_in(hipStream_t st, const double* src, double* dst, int fields, const Geo& g) {
  const long n = (long)g.Xnp * g.Ym * g.Zm;
  hipLaunchKernelGGL(k_rows_in, row_grid(n, fields), dim3(256), 0, st, src, dst, g, (unsigned)n);
}

void launch_rows_out(hipStream_t st, const double* src, double* dst, int fields, const Geo& g) {
  const long n = (long)g.Xnp * g.Ym * g.Zm;
  hipLaunchKernelGGL(k_rows_out, row_grid(n, fields), dim3(256), 0, st, src, dst, g, (unsigned)n);
}

void launch_q_in(hipStream_t st, const double* Q, const double* J, double* U, const Geo& g) {
  dim3 blk(64, 4);
  hipLaunchKernelGGL(k_q_in, box_grid(g.Zp, g.Ym, g.Xnp, blk), blk, 0, st, Q, J, U, g);
}

void launch_q_out(hipStream_t st, const double* U, const double* J, double* Q, const Geo& g) {
  dim3 blk(64, 4);
  hipLaunchKernelGGL(k_q_out, box_grid(g.nz - 1, g.ny - 1, g.gend - 2, blk), blk, 0, st, U, J, Q, g);
}

void launch_halo_bc(hipStream_t st, double* U, const double* prof, const Geo& g, int x_periodic) {
  int src_lo = x_periodic ? g.gend : 3, src_hi = x_periodic ? 3 : g.gend;
  const long n = 2 * g.plane + (long)(g.gend - 2) * (2 * (g.nz - 1) + 2 * (g.ny + 3));
  hipLaunchKernelGGL(k_ghosts, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, U, prof, g, src_lo, src_hi);
}

// derived profile rows for the fluxes, recomputed whenever the metric rows
// change: FT_REC + 7 d + r holds 1/sum(w/J) of recipe r in direction d (at
// the cell's j along x and z, at face j along y; stencil J clamped to the
// array for recipes a face does not use), FT_NRM + 4 d the face normal's
// (insqr, N0, N1, N2) at the face row the fluxes read, FT_RCP + 2 d the
// reciprocals of that row's face J and insqr
__global__ void k_flux_tables(double* __restrict__ prof, Geo g) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= 24 * g.Ym) return;
  const int row = idx / g.Ym, j = idx - row * g.Ym;
  if (row < 21) {
    const int d = row / 7, r = row % 7;
    double jj[6];
#pragma unroll
    for (int t = 0; t < 6; t++) jj[t] = pf(prof, g.Ym, SET_C, 0, d == 1 ? min(max(j + t - 2, 0), g.Ym - 1) : j);
    prof[(long)(FT_REC + row) * g.Ym + j] = rec_temp(r, jj);
  } else {
    const int d = row - 21, set = SET_U + d;
    const double n0 = pf(prof, g.Ym, set, 1 + 3 * d, j), n1 = pf(prof, g.Ym, set, 2 + 3 * d, j),
                 n2 = pf(prof, g.Ym, set, 3 + 3 * d, j);
    const double insqr = 1.0 / sqrt(n0 * n0 + n1 * n1 + n2 * n2);
    prof[(long)(FT_NRM + 4 * d) * g.Ym + j] = insqr;
    prof[(long)(FT_NRM + 4 * d + 1) * g.Ym + j] = n0 * insqr;
    prof[(long)(FT_NRM + 4 * d + 2) * g.Ym + j] = n1 * insqr;
    prof[(long)(FT_NRM + 4 * d + 3) * g.Ym + j] = n2 * insqr;
    prof[(long)(FT_RCP + 2 * d) * g.Ym + j] = 1.0 / pf(prof, g.Ym, set, 0, j);
    prof[(long)(FT_RCP + 2 * d + 1) * g.Ym + j] = 1.0 / insqr;
  }
}

void launch_flux_tables(hipStream_t st, double* prof, const Geo& g) {
  hipLaunchKernelGGL(k_flux_tables, dim3((24 * g.Ym + 127) / 128), dim3(128), 0, st, prof, g);
}

// Faces per thread of the column kernels: FC, halved until `rows` waves times
// the runs of a column of nf faces fill the chip's 1024 SIMDs with six waves
// each.  A run loads six cells before its first face, but with few waves the
// time is that of one run, face after face.  Flux_X / Flux_Y: 64^3 38 / 38 us
// with 16 faces, 16 / 16 with 1 (4160 waves); 128x96x128 62 / 60 us with 16,
// 48 / 50 with 4 (6336); 256x192x256 438 / 434 us with 1, 322 / 329 with 16
// (13056).  The limiter fluxes, x / y, with 16 faces and with this rule: 64^3
// 67 / 79 and 25 / 27 us, 128x96x128 118 / 135 and 96 / 107, 192x144x192
// 333 / 379 and 311 / 350.
static int flux_run(long rows, int nf) {
  int fc = FC;
  while (fc > 1 && rows * ((nf + fc - 1) / fc) < 6144) fc /= 2;
  return fc;
}

void launch_flux(hipStream_t st, int dir, const double* U, const double* prof, double* F, const Geo& g) {
  dim3 blk(64, 4);
  if (dir == 2) {
    hipLaunchKernelGGL(k_flux_zs<2>, box_grid(g.nz, g.ny - 1, g.gend - 2, blk), blk, 0, st, U, prof, F, g);
    return;
  }
  const int nr = dir == 0 ? g.ny - 1 : g.gend - 2, nf = dir == 0 ? g.gend - 1 : g.ny;
  const int fc = flux_run((long)((g.nz - 1 + 63) / 64) * nr, nf);
  const dim3 gr = box_grid(g.nz - 1, nr, (nf + fc - 1) / fc, blk);
  if (dir == 0)
    hipLaunchKernelGGL(k_flux_col<0>, gr, blk, 0, st, U, prof, F, g, fc);
  else
    hipLaunchKernelGGL(k_flux_col<1>, gr, blk, 0, st, U, prof, F, g, fc);
}

void launch_flux_limiter(hipStream_t st, int dir, const double* U, const double* Ep, const double* prof, double* F,
                         const Geo& g) {
  dim3 blk(64, 4);
  if (dir == 2) {
    hipLaunchKernelGGL(k_flux_lim<2>, box_grid(g.nz, g.ny - 1, g.gend - 2, blk), blk, 0, st, U, Ep, prof, F, g);
    return;
  }
  const int nr = dir == 0 ? g.ny - 1 : g.gend - 2, nf = dir == 0 ? g.gend - 1 : g.ny;
  const int fc = flux_run((long)((g.nz - 1 + 63) / 64) * nr, nf);
  const dim3 gr = box_grid(g.nz - 1, nr, (nf + fc - 1) / fc, blk);
  if (dir == 0)
    hipLaunchKernelGGL(k_flux_lim_col<0>, gr, blk, 0, st, U, Ep, prof, F, g, fc);
  else
    hipLaunchKernelGGL(k_flux_lim_col<1>, gr, blk, 0, st, U, Ep, prof, F, g, fc);
}

void launch_filter(hipStream_t st, const double* U, const double* prof, const double* Yp, double* W, double crit,
                   double E_high, double E_low, double* EpX, double* EpY, double* EpZ, const Geo& g) {
  // W: 22 fields = G1..G5 (4 each) E_h E_2h (the passes' Gx, Gy stay in LDS)
  const long n = g.nf;
  FiltHist hist;
  double* Gp[5];
  for (int q = 0; q < 5; q++) hist.G[q] = Gp[q] = W + 4 * q * n;
  double *Eh = W + 20 * n, *E2h = W + 21 * n;
  dim3 blk(64, 4);
  const dim3 gp((g.nz - 1 + FK - 1) / FK, (g.ny - 1 + FJ - 1) / FJ, (g.gend - 2 + FI - 1) / FI);
  for (int wide = 0; wide < 2; wide++) {
    double* E = wide ? E2h : Eh;
    for (int pass = 0; pass < 6; pass++) {
      const double* src = pass == 0 ? U : Gp[pass - 1];
      double* out = pass < 5 ? Gp[pass] : nullptr;
      if (wide) {
        if (pass < 5)
          hipLaunchKernelGGL((k_filt_pass<1, false>), gp, dim3(256), 0, st, src, U, prof, Yp, out, hist, E, g);
        else
          hipLaunchKernelGGL((k_filt_pass<1, true>), gp, dim3(256), 0, st, src, U, prof, Yp, out, hist, E, g);
      } else {
        if (pass < 5)
          hipLaunchKernelGGL((k_filt_pass<0, false>), gp, dim3(256), 0, st, src, U, prof, Yp, out, hist, E, g);
        else
          hipLaunchKernelGGL((k_filt_pass<0, true>), gp, dim3(256), 0, st, src, U, prof, Yp, out, hist, E, g);
      }
    }
  }
  hipLaunchKernelGGL(k_filt_sensor<0>, box_grid(g.nz - 1, g.ny - 1, g.gend - 1, blk), blk, 0, st, Eh, E2h, crit,
                     E_high, E_low, EpX, g);
  hipLaunchKernelGGL(k_filt_sensor<1>, box_grid(g.nz - 1, g.ny, g.gend - 2, blk), blk, 0, st, Eh, E2h, crit, E_high,
                     E_low, EpY, g);
  hipLaunchKernelGGL(k_filt_sensor<2>, box_grid(g.nz, g.ny - 1, g.gend - 2, blk), blk, 0, st, Eh, E2h, crit, E_high,
                     E_low, EpZ, g);
}

void launch_viscous(hipStream_t st, const double* U, const double* prof, double* Pr, double* VS, double* vF,
                    const Geo& g, bool fused_viscous) {
  dim3 blk(64, 4);
  double invXI = 1. / (g.dXI), invET = 1. / (g.dET), invZT = 1. / (g.dZT);
  double inv4XI = 1. / (4 * g.dXI), inv4ET = 1. / (4 * g.dET), inv4ZT = 1. / (4 * g.dZT);
  if (fused_viscous) {
    // planes per block: VC, halved until two blocks per CU are there.  64^3: 53
    // us with 16 planes, 21 with 2 (512 blocks); 16x12x16: 48 and 10 (1 plane);
    // 128x96x128: 85 with 16, 72 with 8 (768 blocks), 88 with 4; 256x192x256:
    // 542 with 16, 605 with 4.
    const long tiles = (long)((g.nz - 1 + VK - 1) / VK) * ((g.ny - 1 + VJ - 1) / VJ);
    int vc = VC;
    while (vc > 1 && tiles * ((g.gend - 2 + vc - 1) / vc) < 512) vc /= 2;
    dim3 gr((g.nz - 1 + VK - 1) / VK, (g.ny - 1 + VJ - 1) / VJ, (g.gend - 2 + vc - 1) / vc);
    hipLaunchKernelGGL(k_visc_fused, gr, dim3(VTHREADS), 0, st, U, prof, vF, g, vc, invXI, invET, invZT, inv4XI, inv4ET,
                       inv4ZT);
    return;
  }
  hipLaunchKernelGGL(k_visc_prim, box_grid(g.nz + 1, g.ny + 1, g.gend, blk), blk, 0, st, U, prof, Pr, g);
  hipLaunchKernelGGL(k_visc_faces, box_grid(g.nz, g.ny, g.gend - 1, blk), blk, 0, st, Pr, prof, VS, g, invXI, invET,
                     invZT, inv4XI, inv4ET, inv4ZT);
  hipLaunchKernelGGL(k_visc_div, box_grid(g.nz - 1, g.ny - 1, g.gend - 2, blk), blk, 0, st, VS, vF, g, invXI, invET,
                     invZT);
}

// RK3NODT.cpp:115-183: one stage of the explicit three-stage update on the
// interior, U_ <- c1 U + c2 U_ + c3 (dt Rk), in place (each cell reads its
// own U_ before writing it; the fluxes are separate arrays).  vF may be null:
// the terms are then +0, as for the never-assigned (zero) vF arrays of a
// reference build that skips Viscous_terms.
__global__ void __launch_bounds__(256) k_rk3(double* __restrict__ Ui, const double* __restrict__ Un,
                                             const double* __restrict__ Fx, const double* __restrict__ Fy,
                                             const double* __restrict__ Fz, const double* __restrict__ vF,
                                             const double* __restrict__ prof, double* __restrict__ MR, Geo g,
                                             double deltaT, double f_drive, double c1, double c2, double c3) {
  const int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  const int i = 3 + blockIdx.z;
  if (k > g.nz || j > g.ny) return;
  const long nf = g.nf;
  const long c = at(g, i, j, k);
  const long fx = at(g, i, j - 1, k - 1), fxm = fx - g.plane;
  const long fy = at(g, i - 1, j, k - 1), fym = fy - g.Zp;
  const long fz = at(g, i - 1, j - 1, k), fzm = fz - 1;
  const double J = pf(prof, g.Ym, SET_C, 0, j);
  const double tmp = Ui[nf + c] / Ui[c];
  double Rk[5];
#pragma unroll
  for (int q = 0; q < 5; q++)
    Rk[q] = -((Fx[q * nf + fx] - Fx[q * nf + fxm]) / g.dXI + (Fy[q * nf + fy] - Fy[q * nf + fym]) / g.dET +
              (Fz[q * nf + fz] - Fz[q * nf + fzm]) / g.dZT);
  const double v2 = vF ? vF[c] : 0.0, v3 = vF ? vF[nf + c] : 0.0, v4 = vF ? vF[2 * nf + c] : 0.0,
               v5 = vF ? vF[3 * nf + c] : 0.0;
  Rk[1] = Rk[1] + v2 + f_drive / J;
  Rk[2] = Rk[2] + v3;
  Rk[3] = Rk[3] + v4;
  Rk[4] = Rk[4] + v5 + f_drive * tmp / J;
#pragma unroll
  for (int q = 0; q < 5; q++) {
    const double m = deltaT * Rk[q];
    if (MR) MR[q * nf + c] = m;
    Ui[q * nf + c] = c1 * Un[q * nf + c] + c2 * Ui[q * nf + c] + c3 * m;
  }
}

void launch_rk3(hipStream_t st, int RK, double* Ui, const double* Un, const double* Fx, const double* Fy,
                const double* Fz, const double* vF, const double* prof, double* MR, const Geo& g, double deltaT,
                double f_drive) {
  // RK3NODT.cpp:112-114
  const double c1[3] = {1.0, 0.75, 1.0 / 3.0};
  const double c2[3] = {0.0, 0.25, 2.0 / 3.0};
  const double c3[3] = {1.0, 0.25, 2.0 / 3.0};
  dim3 blk(64, 4);
  hipLaunchKernelGGL(k_rk3, box_grid(g.nz - 1, g.ny - 1, g.gend - 2, blk), blk, 0, st, Ui, Un, Fx, Fy, Fz, vF, prof,
                     MR, g, deltaT, f_drive, c1[RK - 1], c2[RK - 1], c3[RK - 1]);
}

// Statistic.cpp:1043-1071: one block per j adds the state's sums over i and
// k of U, V, W, UU, VV, WW, UV to sums[q * Ym + j].  Each thread sums its
// cells in (i, k) order, then the block combines the 256 partial sums in a
// fixed tree, so repeated runs give the same bits (the reference's single
// running sum is matched to rounding, not bit for bit).
__global__ void __launch_bounds__(256) k_stat(const double* __restrict__ U, double* __restrict__ sums, Geo g) {
  __shared__ double red[7][256];
  const int j = 2 + blockIdx.x;
  const int t = threadIdx.x;
  const int X = g.gend - 2, Z = g.nz - 1;
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  for (long c = t; c < (long)X * Z; c += 256) {
    const int i = 3 + (int)(c / Z), k = 2 + (int)(c % Z);
    const long p = at(g, i, j, k);
    const double r = U[p];
    const double u = U[g.nf + p] / r, v = U[2 * g.nf + p] / r, w = U[3 * g.nf + p] / r;
    acc[0] += u;
    acc[1] += v;
    acc[2] += w;
    acc[3] += u * u;
    acc[4] += v * v;
    acc[5] += w * w;
    acc[6] += u * v;
  }
#pragma unroll
  for (int q = 0; q < 7; q++) red[q][t] = acc[q];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h)
#pragma unroll
      for (int q = 0; q < 7; q++) red[q][t] += red[q][t + h];
    __syncthreads();
  }
  if (t < 7) sums[t * g.Ym + j] += red[t][0];
}

void launch_stat(hipStream_t st, const double* U, double* sums, const Geo& g) {
  hipLaunchKernelGGL(k_stat, dim3(g.ny - 1), dim3(256), 0, st, U, sums, g);
}

// Driven_force.cpp:49-61: one block per i-plane sums ((U2_ J) 1) / J / Jsum
// over (j, k) (per thread in order, then a fixed tree) into part[i - 3]
__global__ void __launch_bounds__(256) k_bulk_flux(const double* __restrict__ U2, const double* __restrict__ prof,
                                                   double Jsum, double* __restrict__ part, Geo g) {
  __shared__ double red[256];
  const int i = 3 + blockIdx.x, t = threadIdx.x;
  const int Y = g.ny - 1, Z = g.nz - 1;
  double acc = 0;
  for (long c = t; c < (long)Y * Z; c += 256) {
    const int j = 2 + (int)(c / Z), k = 2 + (int)(c % Z);
    const double J = pf(prof, g.Ym, SET_C, 0, j);
    acc += (U2[at(g, i, j, k)] * J) * 1. / J / Jsum;
  }
  red[t] = acc;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h) red[t] += red[t + h];
    __syncthreads();
  }
  if (t == 0) part[blockIdx.x] = red[0];
}

void launch_bulk_flux(hipStream_t st, const double* U2, const double* prof, double Jsum, double* part,
                      const Geo& g) {
  hipLaunchKernelGGL(k_bulk_flux, dim3(g.gend - 2), dim3(256), 0, st, U2, prof, Jsum, part, g);
}

// Statistic.cpp:552-828, the part behind Shear_stress.dat: the y-face
// viscous flux of x-momentum ML2 (:818-824) at the bottom wall face (j = 2,
// SXYm[1]) and the top one (j = ny + 1, SXYm[ny]) for i = 3..gend and
// k = 2..nz, into out[(w * X_out + i - 3) * Z_out + k - 2], with the
// reference's velocities, 4-point x/z and 2-point y derivatives (:734-786)
// and y-face metrics at j - 1 (:716-724), in its order of operations
__global__ void k_wall_shear(const double* __restrict__ U, const double* __restrict__ prof, Geo g,
                             double* __restrict__ out) {
  const int k = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  const int i = 3 + blockIdx.y, w = blockIdx.z;
  if (k > g.nz) return;
  const int j = w == 0 ? 2 : g.ny + 1;
  const double inv4XI = 1. / (4 * g.dXI), invET = 1. / (g.dET), inv4ZT = 1. / (4 * g.dZT);
  double u[10], v[10], ww[10];
  const int off[10][3] = {{0, 0, 0},  {-1, 0, 0}, {1, 0, 0},  {0, -1, 0}, {-1, -1, 0},
                          {1, -1, 0}, {0, 0, 1},  {0, 0, -1}, {0, -1, 1}, {0, -1, -1}};
#pragma unroll
  for (int q = 0; q < 10; q++) {
    const long c = at(g, i + off[q][0], j + off[q][1], k + off[q][2]);
    const double rho = U[c];
    u[q] = U[g.nf + c] / rho;
    v[q] = U[2 * g.nf + c] / rho;
    ww[q] = U[3 * g.nf + c] / rho;
  }
  // q: 0 (0,0,0) 1 (-1,0,0) 2 (1,0,0) 3 (0,-1,0) 4 (-1,-1,0) 5 (1,-1,0)
  //    6 (0,0,1) 7 (0,0,-1) 8 (0,-1,1) 9 (0,-1,-1)
  const double du_dx = (u[2] + u[5] - u[1] - u[4]) * inv4XI;
  const double dv_dx = (v[2] + v[5] - v[1] - v[4]) * inv4XI;
  const double dw_dx = (ww[2] + ww[5] - ww[1] - ww[4]) * inv4XI;
  const double du_dy = (u[0] - u[3]) * invET;
  const double dv_dy = (v[0] - v[3]) * invET;
  const double dw_dy = (ww[0] - ww[3]) * invET;
  const double du_dz = (u[6] + u[8] - u[7] - u[9]) * inv4ZT;
  const double dv_dz = (v[6] + v[8] - v[7] - v[9]) * inv4ZT;
  const double dw_dz = (ww[6] + ww[8] - ww[7] - ww[9]) * inv4ZT;
  const int jf = j - 1;
  const double xix = pf(prof, g.Ym, SET_V, 1, jf), xiy = pf(prof, g.Ym, SET_V, 2, jf),
               xiz = pf(prof, g.Ym, SET_V, 3, jf), etx = pf(prof, g.Ym, SET_V, 4, jf),
               ety = pf(prof, g.Ym, SET_V, 5, jf), etz = pf(prof, g.Ym, SET_V, 6, jf),
               ztx = pf(prof, g.Ym, SET_V, 7, jf), zty = pf(prof, g.Ym, SET_V, 8, jf),
               ztz = pf(prof, g.Ym, SET_V, 9, jf);
  const double b1 = (4. / 3) * etx * etx + ety * ety + etz * etz;
  const double b5 = (1. / 3) * etx * ety;
  const double b7 = (1. / 3) * etx * etz;
  const double d1 = (4. / 3) * xix * etx + xiy * ety + xiz * etz;
  const double d5 = xix * ety - (2. / 3) * xiy * etx;
  const double d6 = xix * etz - (2. / 3) * xiz * etx;
  const double f1 = (4. / 3) * etx * ztx + ety * zty + etz * ztz;
  const double f7 = ety * ztx - (2. / 3) * etx * zty;
  const double f9 = etz * ztx - (2. / 3) * etx * ztz;
  const int X = g.gend - 2, Z = g.nz - 1;
  out[((long)w * X + i - 3) * Z + k - 2] =
      MU_L * (d1 * du_dx + d5 * dv_dx + d6 * dw_dx + b1 * du_dy + b5 * dv_dy + b7 * dw_dy + f1 * du_dz + f7 * dv_dz +
              f9 * dw_dz) / pf(prof, g.Ym, SET_V, 0, jf);
}

void launch_wall_shear(hipStream_t st, const double* U, const double* prof, const Geo& g, double* out) {
  hipLaunchKernelGGL(k_wall_shear, dim3((g.nz - 1 + 63) / 64, g.gend - 2, 2), dim3(64), 0, st, U, prof, g, out);
}

// out[0] = ((0 + a[0]) + a[1]) + ... + a[n-1], one thread: the order of a host loop
__global__ void k_sum_in_order(const double* __restrict__ a, int n, double* __restrict__ out) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double s = 0;
  for (int i = 0; i < n; i++) s = s + a[i];
  out[0] = s;
}

void launch_sum_in_order(hipStream_t st, const double* a, int n, double* out) {
  hipLaunchKernelGGL(k_sum_in_order, dim3(1), dim3(64), 0, st, a, n, out);
}

void launch_rhs(hipStream_t st, const double* Ui, const double* Un, const double* Uq, const double* Fx,
                const double* Fy, const double* Fz, const double* vF, const double* prof, double* MR, double* NL,
                const Geo& g, double deltaT, double f_drive) {
  dim3 blk(64, 4);
  hipLaunchKernelGGL(k_rhs, box_grid(g.nz - 1, g.ny - 1, g.gend - 2, blk), blk, 0, st, Ui, Un, Uq, Fx, Fy, Fz, vF, prof,
                     MR, NL, g, deltaT, f_drive);
}

Sk sweep_layout(const Geo& g) {
  Sk q;
  q.nTI = (g.gend - 2 + TI - 1) / TI;
  q.nTJ = (g.ny - 1 + TJ - 1) / TJ;
  q.ntiles = q.nTI * q.nTJ;
  q.Nz = g.nz - 1;
  q.nsteps = q.Nz + (TI - 1) + (TJ - 1);
  q.nsk = (long)q.ntiles * q.nsteps * 64;
  return q;
}

int sweep_tiles(const Geo& g, int* nTI, int* nTJ) {
  Sk q = sweep_layout(g);
  *nTI = q.nTI;
  *nTJ = q.nTJ;
  return q.ntiles;
}

long sweep_field_elems(const Geo& g) { return sweep_layout(g).nsk; }

// (S + MR: rewritten by every sweep's pre-pass and read by no one after it; a
// float layout has half the bytes, and what follows it is kept)
long sweep_scratch_elems(const Geo& g, bool fp32) { return (G_N + 5) * sweep_layout(g).nsk / (fp32 ? 2 : 1); }

long jacobi_summary_elems(const Geo& g) { return 6 * g.nf; }

long sweep_buffer_elems(const Geo& g) { return (G_N + 15) * sweep_layout(g).nsk; }

long sweep_update_blocks(const Geo& g) {
  Sk q = sweep_layout(g);
  return (long)((q.nsteps + 3) / 4) * q.ntiles;
}

// Sbuf holds G_N summary fields, MR and NL (5 each) in sweep order, then room
// for five more: the single-wave tiles' NR or, with the pipelined sweeps, the
// hand-off slots and the x edges' summary (two fields each).  Those put the
// last pair's NR into MR's rows, which no one reads any more, and an earlier
// pair's, which no one reads at all, into NL's (a row is read steps before it
// is written).  A float layout uses the first half of the buffer.
template <class T>
struct SweepBuf {
  T *S, *MR, *NL, *NR, *H, *E;
  SweepBuf(double* Sbuf, const Sk& q, bool pipelined) {
    S = reinterpret_cast<T*>(Sbuf);
    MR = S + (long)G_N * q.nsk;
    NL = MR + 5 * q.nsk;
    H = NL + 5 * q.nsk;
    E = H + ho_at(q, q.ntiles, 0, 0);
    NR = pipelined ? MR : H;
  }
};
static_assert(4 * HO_SLOT <= 5 * 64, "the hand-off slots and the edge copy fit in five fields");

template <class T>
static void sweeps_t(hipStream_t st, double* Ui, const double* MR, double* Sbuf, const double* prof, const Geo& g,
                     double deltaT, int n_sweeps, const int* order, int* sync, double* partial, double* er_dev,
                     double DN, long spin_limit, const hipEvent_t* marks, bool pipelined, const RhsIn* rin) {
  Sk q = sweep_layout(g);
  const SweepBuf<T> b(Sbuf, q, pipelined);
  T *S = b.S, *MRs = b.MR, *NLs = b.NL, *NRs = b.NR, *H = b.H, *E = b.E;
  if (rin)
    hipLaunchKernelGGL(k_sweep_prep_rhs<T>, dim3((q.nsteps + PR - 1) / PR, q.ntiles), dim3(PR_THREADS), 0, st, Ui, *rin,
                       prof, S, MRs, E, g, q, deltaT, sync);
  else
    hipLaunchKernelGGL(k_sweep_prep<T>, dim3((q.nsteps + PC - 1) / PC, q.ntiles), dim3(256), 0, st, Ui, MR, prof, S,
                       MRs, E, g, q, sync);
  if (marks) (void)hipEventRecord(marks[0], st);
  const int nt = q.ntiles;
  for (int sweep = 0; sweep < n_sweeps; sweep++) {
    if (sweep > 0) hipLaunchKernelGGL(k_sweep_reset, dim3(1), dim3(256), 0, st, sync, 2 * nt + 4);
    if (marks) (void)hipEventRecord(marks[1 + 3 * sweep], st);
    if constexpr (std::is_same<T, double>::value) {
      if (!pipelined)
        hipLaunchKernelGGL(k_sweep_tiles<true>, dim3(nt), dim3(64), 0, st, S, MRs, NLs, NRs, prof, g, q, order, sync,
                           spin_limit, deltaT);
    }
    if (pipelined)
      hipLaunchKernelGGL((k_sweep_pipe<true, T>), dim3(nt), dim3(PIPE_THREADS), 0, st, S, MRs, NLs, H,
                         E, prof, g, q, order, sync, spin_limit, deltaT);
    if (marks) (void)hipEventRecord(marks[2 + 3 * sweep], st);
    if constexpr (std::is_same<T, double>::value) {
      if (!pipelined)
        hipLaunchKernelGGL(k_sweep_tiles<false>, dim3(nt), dim3(64), 0, st, S, NLs, NRs, NRs, prof, g, q, order,
                           sync + nt + 2, spin_limit, deltaT);
    }
    if (pipelined)
      hipLaunchKernelGGL((k_sweep_pipe<false, T>), dim3(nt), dim3(PIPE_THREADS), 0, st, S, NLs,
                         sweep + 1 < n_sweeps ? NLs : NRs, H, E, prof, g, q, order, sync + nt + 2, spin_limit, deltaT);
    if (marks) (void)hipEventRecord(marks[3 + 3 * sweep], st);
  }
  // primitive update reading NR from the sweep order
  dim3 gr((q.nsteps + PC - 1) / PC, q.ntiles);
  hipLaunchKernelGGL(k_update_sk<T>, gr, dim3(256), 0, st, Ui, NRs, prof, partial, g, q);
  hipLaunchKernelGGL(k_reduce_partials, dim3(1), dim3(1024), 0, st, partial, (long)gr.x * gr.y, er_dev, DN, sync + 1,
                     sync + nt + 3);
}

template <class T>
static void seed_hand_off_t(hipStream_t st, double* Sbuf, const Geo& g) {
  Sk q = sweep_layout(g);
  hipLaunchKernelGGL(k_seed_hand_off<T>, dim3((q.nsteps + 1) / 2, q.ntiles), dim3(256), 0, st,
                     SweepBuf<T>(Sbuf, q, true).H, q);
}

void launch_seed_hand_off(hipStream_t st, double* Sbuf, const Geo& g, bool fp32) {
  if (fp32)
    seed_hand_off_t<float>(st, Sbuf, g);
  else
    seed_hand_off_t<double>(st, Sbuf, g);
}

void launch_seed_tiles(hipStream_t st, double* Sbuf, const Geo& g) {
  Sk q = sweep_layout(g);
  hipLaunchKernelGGL(k_seed_tiles, dim3((q.nsteps + 3) / 4, q.ntiles), dim3(256), 0, st,
                     SweepBuf<double>(Sbuf, q, false).NL, q);
}

void launch_sweeps(hipStream_t st, double* Ui, const double* MR, double* Sbuf, const double* prof, const Geo& g,
                   double deltaT, int n_sweeps, const int* order, int* sync, double* partial, double* er_dev,
                   double DN, long spin_limit, const hipEvent_t* marks, bool pipelined, const RhsIn* rin, bool fp32) {
  if (fp32)
    sweeps_t<float>(st, Ui, MR, Sbuf, prof, g, deltaT, n_sweeps, order, sync, partial, er_dev, DN, spin_limit, marks,
                    true, rin);
  else
    sweeps_t<double>(st, Ui, MR, Sbuf, prof, g, deltaT, n_sweeps, order, sync, partial, er_dev, DN, spin_limit,
                     marks, pipelined, rin);
}

template <class T>
static void sweep_outputs_t(hipStream_t st, double* Sbuf, double* NL, double* NR, const Geo& g, bool pipelined) {
  Sk q = sweep_layout(g);
  const SweepBuf<T> b(Sbuf, q, pipelined);
  const dim3 gr((q.nsteps + 15) / 16, q.ntiles);
  hipLaunchKernelGGL(k_sk_to_natural<T>, gr, dim3(1024), 0, st, b.NL, NL, g, q, 5);
  hipLaunchKernelGGL(k_sk_to_natural<T>, gr, dim3(1024), 0, st, b.NR, NR, g, q, 5);
}

void launch_sweep_outputs(hipStream_t st, double* Sbuf, double* NL, double* NR, const Geo& g, bool pipelined, bool fp32) {
  if (fp32)
    sweep_outputs_t<float>(st, Sbuf, NL, NR, g, pipelined);
  else
    sweep_outputs_t<double>(st, Sbuf, NL, NR, g, pipelined);
}

void launch_sweeps_planes(hipStream_t st, const double* Ui, const double* MR, double* NL, double* NR,
                          const double* prof, const Geo& g, double deltaT, int n_sweeps, const hipEvent_t* marks) {
  int mmin = 7, mmax = g.gend + g.ny + g.nz;
  int nj = g.ny - 1;
  dim3 blk(64);
  if (marks) (void)hipEventRecord(marks[0], st);
  for (int sweep = 0; sweep < n_sweeps; sweep++) {
    if (marks) (void)hipEventRecord(marks[1 + 3 * sweep], st);
    for (int m = mmin; m <= mmax; m++) {
      int ilo = max(3, m - g.ny - g.nz), ihi = min(g.gend, m - 4);
      hipLaunchKernelGGL(k_sweep_fwd, dim3((nj + 63) / 64, ihi - ilo + 1), blk, 0, st, Ui, MR, NL, prof, g, deltaT, m,
                         ilo);
    }
    for (int m = mmax; m >= mmin; m--) {
      int ilo = max(3, m - g.ny - g.nz), ihi = min(g.gend, m - 4);
      if (m == mmax && marks) (void)hipEventRecord(marks[2 + 3 * sweep], st);
      hipLaunchKernelGGL(k_sweep_bwd, dim3((nj + 63) / 64, ihi - ilo + 1), blk, 0, st, Ui, NL, NR, prof, g, deltaT, m,
                         ilo);
    }
    if (marks) (void)hipEventRecord(marks[3 + 3 * sweep], st);
  }
}

void launch_extrapolate(hipStream_t st, double* Ui, const double* Un, const double* Uq, const double* Uqq,
                        const double* U3, const Geo& g, int order) {
  dim3 blk(64, 4);
  hipLaunchKernelGGL(k_extrapolate, box_grid(g.nz - 1, g.ny - 1, g.gend - 2, blk), blk, 0, st, Ui, Un, Uq, Uqq, U3, g,
                     order);
}

void launch_copy_interior(hipStream_t st, const double* src, double* dst, const Geo& g) {
  dim3 blk(64, 4);
  hipLaunchKernelGGL(k_copy_interior, box_grid(g.nz - 1, g.ny - 1, g.gend - 2, blk), blk, 0, st, src, dst, g);
}

void launch_dplusgs(hipStream_t st, const double* Ui, const double* MR, double* NL, double* NR, const double* prof,
                    const Geo& g, double deltaT, double* S) {
  dim3 blk(64, 4);
  dim3 gr = box_grid(g.nz - 1, g.ny - 1, g.gend - 2, blk);
  if (S) hipLaunchKernelGGL(k_jacobi_summary, gr, blk, 0, st, Ui, prof, S, g);
  // four sweeps, ping-pong NL -> NR -> NL -> NR -> NL; both end with the last
  for (int sweep = 0; sweep < 4; sweep++) {
    const double* in = (sweep & 1) ? NR : NL;
    double* out = (sweep & 1) ? NL : NR;
    if (S)
      hipLaunchKernelGGL(k_jacobi_diag, dim3(gr.x * JAC_JG, gr.z, (gr.y + JAC_JG - 1) / JAC_JG), blk, 0, st, S, MR, in, out, prof, g, deltaT);
    else
      hipLaunchKernelGGL(k_jacobi, gr, blk, 0, st, Ui, MR, in, out, prof, g, deltaT);
  }
  launch_copy_interior(st, NL, NR, g);
}

long update_blocks(const Geo& g) {
  dim3 blk(64, 4);
  dim3 gr = box_grid(g.nz - 1, g.ny - 1, g.gend - 2, blk);
  return (long)gr.x * gr.y * gr.z;
}

void launch_update(hipStream_t st, double* Ui, const double* NR, const double* prof, double* partial, double* er_dev,
                   const Geo& g, double DN) {
  dim3 blk(64, 4);
  dim3 gr = box_grid(g.nz - 1, g.ny - 1, g.gend - 2, blk);
  hipLaunchKernelGGL(k_update, gr, blk, 0, st, Ui, NR, prof, partial, g);
  hipLaunchKernelGGL(k_reduce_partials, dim3(1), dim3(1024), 0, st, partial, update_blocks(g), er_dev, DN, nullptr,
                     nullptr);
}

}  // namespace cf
