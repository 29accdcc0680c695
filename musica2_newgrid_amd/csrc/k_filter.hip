// Numerical dissipation applied once per step after the last RK stage,
// fused with update_varn (src/Time/update.f90:538-565):
//   selective filter   filtering_11pts  src/Num_dissipation/mod_filtering.f90:992-1034,
//                      1192-1233, 1382-1423 (coefficients :63-68, scaled :189-203)
//   shock filter       filter_o10_shock src/Num_dissipation/mod_filtering_shock.f90:
//                      pressure sensor :243-260, face dissipation :419-440,
//                      increment :690-700 (and the j, k repeats)
//   artificial viscosity artvisc_o9 mod_artvisc.f90:82-874 (coefficients :16-79),
//                      with update_varn_artvisc (update.f90:568-608): the
//                      shock filter's face dissipation without the sensor,
//                      weighted by the spectral radius |u_d| + c of U^n
//                      averaged to the faces, times the metric, U += deltat*K
// Interior rows of periodic faces and 1-to-1 interfaces; next to boundary
// faces on i or j (walls, characteristic outflow, supersonic inlet) the
// selective filter leaves rows 1,2 (n-1,n) unfiltered along that axis and
// uses the 5/7/9-pt filters on rows 3,4,5 (mod_filtering.f90:900-988,
// 1116-1190); along k every row is filtered.
//
// 2.5-D layout: the state of the tile + 5-cell halos of the current k plane
// sits in LDS for the i/j stencils, the own column keeps an 11-deep register
// queue for k.  The shock filter also stages p(U^n) and computes each
// pressure sensor once per plane in LDS.  Halo cells are statically assigned
// to lanes so that all global loads of a plane are issued in one batch.
// k_shock is the shock filter alone; k_filter_shock takes it with the Edoh
// switch, and the artificial viscosities.
#include <type_traits>

#include "mgpu_internal.h"

namespace mgpu {

namespace {

constexpr int FX = 32, FY = 16, FT = FX * FY;
constexpr int NHX = 10 * FY, NH = NHX + 10 * FX, NS = (NH + FT - 1) / FT;  // state halo cells
constexpr int NPX = FY * (FX + 4), NPY = (FY + 4) * FX;                  // p cells along i / j
constexpr int NSP = (NPX + NPY + FT - 1) / FT;

// Block and tile of this workgroup in a batched launch.
__device__ __forceinline__ const FilterArgs &tile_of(const Batch<FilterArgs> *__restrict__ tab, int nb, int ntiles,
                                                     int &i0, int &j0, int &kbeg, int &kend) {
  const int w = xcd_remap(blockIdx.x, ntiles);
  const Batch<FilterArgs> &e = batch_find(tab, nb, w);
  int tile_x, tile_y, chunk;
  tile_coords(e.t, w, tile_x, tile_y, chunk);
  i0 = tile_x * FX + 1;
  j0 = tile_y * FY + 1;
  kbeg = chunk * e.t.kchunk + 1;
  kend = min(kbeg + e.t.kchunk - 1, e.a.g.nz);
  return e.a;
}

// Static assignment of the 5-cell state halo of a plane to the lanes.
struct Halo {
  idx_t off[NS];
  int r[NS], c[NS];
  bool on[NS], xdir[NS];
};

__device__ __forceinline__ void halo_setup(const Geom &g, int i0, int j0, Halo &h) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const int t = tid + s * FT;
    h.on[s] = false;
    h.xdir[s] = true;
    h.r[s] = h.c[s] = 0;
    h.off[s] = 0;
    if (t < NHX) {
      const int r = t / 10, c = t % 10;
      const int li = c < 5 ? c : FX + c;
      const int gi = i0 - 5 + li, gj = j0 + r;
      h.on[s] = gj <= g.ny && gi <= g.nx + 5;
      h.r[s] = r;
      h.c[s] = li;
      h.off[s] = lin_w(g, gi, gj);
    } else if (t < NH) {
      const int tt = t - NHX;
      const int r = tt / FX, c = tt % FX;
      const int lj = r < 5 ? r : FY + r;
      const int gi = i0 + c, gj = j0 - 5 + lj;
      h.on[s] = gi <= g.nx && gj <= g.ny + 5;
      h.xdir[s] = false;
      h.r[s] = lj;
      h.c[s] = c;
      h.off[s] = lin_w(g, gi, gj);
    }
  }
}

__device__ __forceinline__ void ld5(const CState &U, idx_t p, double o[5]) {
#pragma unroll
  for (int v = 0; v < 5; v++) o[v] = ldg(U.v[v], p);
}

// State at element p.  The filters run in FP64 in both precisions: they read
// and write FP64 states (the last stage's output and U^{n+1}), so FP32
// arithmetic saved no time (0.93 ms per launch either way on the 512x256x128
// channel), while rounding the state's difference with the reference state
// to FP32 before the stencil was the largest error of the mixed path
// (density 2.4e-6 after 1000 steps there, 4.7e-8 with FP64 filters).
__device__ __forceinline__ void ldr(const CState &U, idx_t p, double o[5]) {
#pragma unroll
  for (int v = 0; v < 5; v++) o[v] = ldg(U.v[v], p);
}

// Filter increment along j of rows next to a wall: nothing on the first two,
// the 5/7/9-pt filters (times -chi) on the next three; y points at the row
// with stride s.  Reads nothing beyond the wall.
template <class R>
__device__ __forceinline__ R fwall(const R *y, int s, int hw, double chi) {
  const R c = R(-chi);
  switch (hw) {
    case 2: return c * (R(D5_0) * y[0] + R(D5_1) * (y[s] + y[-s]) + R(D5_2) * (y[2 * s] + y[-2 * s]));
    case 3:
      return c * (R(D7_0) * y[0] + R(D7_1) * (y[s] + y[-s]) + R(D7_2) * (y[2 * s] + y[-2 * s]) +
                  R(D7_3) * (y[3 * s] + y[-3 * s]));
    case 4:
      return c * (R(D9_0) * y[0] + R(D9_1) * (y[s] + y[-s]) + R(D9_2) * (y[2 * s] + y[-2 * s]) +
                  R(D9_3) * (y[3 * s] + y[-3 * s]) + R(D9_4) * (y[4 * s] + y[-4 * s]));
    default: return R(0);
  }
}

// A plane of the tile and its 5-cell halos in LDS: a cross of rows (j0-5..)
// and columns (i0-5..) whose corners are neither written nor read; every cell
// of the tile once, for the i- and the j-stencils alike.
constexpr int SW = FX + 10, SH = FY + 10;
static_assert(NS == 1, "one halo cell per lane");

// k_filter_sf and k_shock march along k with one barrier per plane: while the
// stencils of plane k run from one LDS buffer, plane k+1 is written to the
// other and the loads of plane k+2 are in flight.  One workgroup of 8 waves
// per CU (its register queue), so nothing else hides what a wave waits for.
// k_filter_sf, against two barriers and the plane staged twice: 192^3 268 us,
// now 239 (its 10 words per cell take 113 us), 384x192x96 with walls 292,
// now 273.
template <bool WALL>
__global__ __launch_bounds__(FT, 2) void k_filter_sf(const Batch<FilterArgs> *__restrict__ tab, int nb, int ntiles) {
  using R = double;
  __shared__ R su[2][5][SH][SW];
  int i0, j0, kbeg, kend;
  const FilterArgs &a = tile_of(tab, nb, ntiles, i0, j0, kbeg, kend);
  // the block's array pointers, read once from the table into registers
  const CState uinp = a.uin;
  const State uoutp = a.uout;
  const Geom &g = a.g;
  const int tx = threadIdx.x % FX, ty = threadIdx.x / FX;
  const int i = i0 + tx, j = j0 + ty;
  const bool own = i <= g.nx && j <= g.ny;
  // points past the end of a partial tile that its stencils reach
  const bool past = !own && ((i <= g.nx + 5 && j <= g.ny) || (i <= g.nx && j <= g.ny + 5));
  const idx_t sz = g.sy, own_off = lin_w(g, i, j);
  Halo hl;
  halo_setup(g, i0, j0, hl);
  const int hr = hl.xdir[0] ? hl.r[0] + 5 : hl.r[0], hc = hl.xdir[0] ? hl.c[0] : hl.c[0] + 5;
  const int hw = WALL ? jhalf(g, j) : 5;
  const int hwi = WALL ? ihalf(g, i) : 5;
  R dd[6];
#pragma unroll
  for (int l = 0; l < 6; l++) dd[l] = (R)a.dd[l];

  // own column: planes k-5..k+5, plane k+6 in flight; a point past the end
  // has its plane k+1 there instead
  R q[11][5], qn[5], uh[5];
  if (own) {
#pragma unroll
    for (int l = 0; l < 10; l++) ldr(uinp, own_off + (idx_t)wrap_k(g, kbeg - 5 + l) * sz, q[l]);
  }
  if (past) ldr(uinp, own_off + (idx_t)kbeg * sz, qn);
  if (hl.on[0]) ldr(uinp, hl.off[0] + (idx_t)kbeg * sz, uh);
  auto stage = [&](int b, const R c[5]) __attribute__((always_inline)) {
    if (own || past) {
#pragma unroll
      for (int v = 0; v < 5; v++) su[b][v][ty + 5][tx + 5] = c[v];
    }
    if (hl.on[0]) {
#pragma unroll
      for (int v = 0; v < 5; v++) su[b][v][hr][hc] = uh[v];
    }
  };
  {
    R c[5];
#pragma unroll
    for (int v = 0; v < 5; v++) c[v] = own ? q[5][v] : qn[v];
    stage(kbeg & 1, c);
  }
  if (own) ldr(uinp, own_off + (idx_t)wrap_k(g, kbeg + 5) * sz, qn);
  if (kbeg < kend) {
    if (past) ldr(uinp, own_off + (idx_t)(kbeg + 1) * sz, qn);
    if (hl.on[0]) ldr(uinp, hl.off[0] + (idx_t)(kbeg + 1) * sz, uh);
  }
  __syncthreads();

  for (int k = kbeg; k <= kend; k++) {
    const idx_t pk = own_off + (idx_t)k * sz;
    const int b = k & 1;
    if (own) {
#pragma unroll
      for (int v = 0; v < 5; v++) q[10][v] = qn[v];
    }
    if (k < kend) {
      R c[5];
#pragma unroll
      for (int v = 0; v < 5; v++) c[v] = own ? q[6][v] : qn[v];
      stage(b ^ 1, c);
      if (own) ldr(uinp, own_off + (idx_t)wrap_k(g, k + 6) * sz, qn);
      if (k + 2 <= kend) {
        if (past) ldr(uinp, pk + 2 * sz, qn);
        if (hl.on[0]) ldr(uinp, hl.off[0] + (idx_t)(k + 2) * sz, uh);
      }
    }
    if (own) {
#pragma unroll
      for (int v = 0; v < 5; v++) {
        const R *x = &su[b][v][ty + 5][tx + 5];
        R K;
        if (!WALL || hwi == 5) {
          K = dd[0] * x[0] + dd[1] * (x[1] + x[-1]) + dd[2] * (x[2] + x[-2]) + dd[3] * (x[3] + x[-3]) +
              dd[4] * (x[4] + x[-4]) + dd[5] * (x[5] + x[-5]);
        } else {
          K = R(0);
          if constexpr (WALL) K = fwall<R>(x, 1, hwi, a.chi);
        }
        if (!WALL || hw == 5) {
          K = K + dd[0] * x[0] + dd[1] * (x[SW] + x[-SW]) + dd[2] * (x[2 * SW] + x[-2 * SW]) +
              dd[3] * (x[3 * SW] + x[-3 * SW]) + dd[4] * (x[4 * SW] + x[-4 * SW]) +
              dd[5] * (x[5 * SW] + x[-5 * SW]);
        } else {
          if constexpr (WALL) K = K + fwall<R>(x, SW, hw, a.chi);
        }
        K = K + dd[0] * q[5][v] + dd[1] * (q[6][v] + q[4][v]) + dd[2] * (q[7][v] + q[3][v]) +
            dd[3] * (q[8][v] + q[2][v]) + dd[4] * (q[9][v] + q[1][v]) + dd[5] * (q[10][v] + q[0][v]);
        stg_nt(uoutp.v[v], pk, q[5][v] + K);
      }
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < 10; l++)
#pragma unroll
      for (int v = 0; v < 5; v++) q[l][v] = q[l + 1][v];
  }
}

// pressure sensor (mod_filtering_shock.f90:252-257) from p at m-1, m, m+1
__device__ __forceinline__ double psens3(double pm, double p0, double pp, double sn, double cs) {
  const double ptrad = pm + 2.0 * p0 + pp;
  const double ptvd = fabs(pp - p0) + fabs(p0 - pm);
  return sn * fabs(pm - 2.0 * p0 + pp) / (cs * ptrad + (1.0 - cs) * ptvd);
}

// D_{m+1/2} from u at m-4..m+5 given as x[-4..5] with stride s
template <class R>
__device__ __forceinline__ R dface(const R *x, int s, R xk0, R xk10) {
  return (x[s] - x[0]) * xk0 +
         (R(D10_1) * (x[s] - x[0]) + R(D10_2) * (x[2 * s] - x[-s]) + R(D10_3) * (x[3 * s] - x[-2 * s]) +
          R(D10_4) * (x[4 * s] - x[-3 * s]) + R(D10_5) * (x[5 * s] - x[-4 * s])) *
             xk10;
}

// 10th difference of the face dissipation (without its amplitude)
template <class R>
__device__ __forceinline__ R d10face(const R *x, int s) {
  return R(D10_1) * (x[s] - x[0]) + R(D10_2) * (x[2 * s] - x[-s]) + R(D10_3) * (x[3 * s] - x[-2 * s]) +
         R(D10_4) * (x[4 * s] - x[-3 * s]) + R(D10_5) * (x[5 * s] - x[-4 * s]);
}

// Half-width of the shock filter's face m+1/2 (between rows m and m+1) along
// an axis of n rows with bounded faces bnd: the d2/d4/d6/d8 faces are the
// first four from a boundary, the boundary face with a tenth of the sensor
// term (filter_o10_shock, mod_filtering_shock.f90:266-466 i, :724-1057 j),
// d10 inside; <= 0: no face (the boundary rows get no increment along that
// axis, :1128-1140 runs over ndy_d..nfy_d).
__device__ __forceinline__ int face_half_n(int bnd, int n, int m) {
  int h = 5;
  if ((bnd & 1) && m < h) h = m;
  if ((bnd & 2) && n - m < h) h = n - m;
  return h;
}
__device__ __forceinline__ int face_half(const Geom &g, int m) { return face_half_n(g.jbnd, g.ny, m); }

// Edoh switch factor of direction d at element p (position r along d):
// min(1, CFL/chi) with CFL = sr_d deltat, times idx_d(r) on Cartesian blocks
// (mod_filtering_shock.f90:668-676 and the j, k repeats; c3 :627-632).
// Metric factor of direction d at position r: idx_d(r) on Cartesian
// directions, 1 where the spectral radius carries the metric (null array).
__device__ __forceinline__ double met_at(const double *met, int r) {
  return met ? ldg(met, (idx_t)(r - 1 + G)) : 1.0;
}

__device__ __forceinline__ double edoh_mul(const FilterArgs &a, int d, idx_t p, int r) {
  const double *met = d == 0 ? a.idx : (d == 1 ? a.idy : a.idz);
  double cfl = ldg(a.sr[d], p) * a.dt;
  if (met) cfl = cfl * ldg(met, (idx_t)(r - 1 + G));
  return fmin(1.0, cfl / a.chi);
}

// The shock filter (without the Edoh switch).  Sensors run one plane ahead of
// the stencils, p two.  Along k the face k+1/2 of a plane is the face k-1/2 of
// the next and is computed once, as is its pressure sensor.  With three
// barriers per plane, the plane staged twice (for i and for j) and both k
// faces of every point: 512x256x128 c3 with walls 876 us, 2.5-D 862 us,
// 113x75x51 38 us; now 645, 683 and 33 us.  On the first it moves 2.57 GB
// (1.6 times its words; halo reads), 510 us at the rate of a large copy; waves
// wait for 38 % of their cycles and 27 % more for an issue slot, vector
// instructions take 25 %.
// WALL: blocks with boundary faces on i or j; rows 1..5 and n-4..n of a
// bounded axis get no increment along it here (k_shock_wall adds it with the
// reduced faces of the boundary closure).
template <bool WALL>
__global__ __launch_bounds__(FT, 2) void k_shock(const Batch<FilterArgs> *__restrict__ tab, int nb, int ntiles) {
  using R = double;
  __shared__ R su[2][5][SH][SW];
  __shared__ double spr[2][FY + 4][FX + 4];  // p from (i0-2, j0-2)
  __shared__ double psx[2][FY][FX + 2];      // psens_x at i0-1 .. i0+FX
  __shared__ double psy[2][FY + 2][FX];      // psens_y at j0-1 .. j0+FY

  int i0, j0, kbeg, kend;
  const FilterArgs &a = tile_of(tab, nb, ntiles, i0, j0, kbeg, kend);
  // the block's array pointers, read once from the table into registers
  const CState uinp = a.uin;
  const State uoutp = a.uout;
  const double *const prsp = a.prs, *const sensp = a.sens;
  const Geom &g = a.g;
  const int tid = threadIdx.x, tx = tid % FX, ty = tid / FX;
  const int i = i0 + tx, j = j0 + ty;
  const bool own = i <= g.nx && j <= g.ny;
  // points past the end of a partial tile: state, p and sensor that it reads
  const bool past = !own && ((i <= g.nx + 5 && j <= g.ny) || (i <= g.nx && j <= g.ny + 5));
  const bool pon = (i <= g.nx + 2 && j <= g.ny) || (i <= g.nx && j <= g.ny + 2);
  const bool sxon = i <= g.nx + 1 && j <= g.ny, syon = i <= g.nx && j <= g.ny + 1;
  const bool duc = sensp != nullptr;
  const double cs = a.csens;
  const idx_t sz = g.sy, own_off = lin_w(g, i, j);
  Halo hl;
  halo_setup(g, i0, j0, hl);
  const bool hon = hl.on[0], hx = hl.xdir[0];
  const int hr = hx ? hl.r[0] + 5 : hl.r[0], hc = hx ? hl.c[0] : hl.c[0] + 5;
  const idx_t h_off = hl.off[0];
  // halo cells whose p (two rows) and sensor (one row) are needed
  const int hn = hx ? hc - 5 : hr - 5, hm = hx ? FX : FY;
  const bool hpon = hon && hn >= -2 && hn <= hm + 1 && (hx ? i0 + hn <= g.nx + 2 : j0 + hn <= g.ny + 2);
  const bool hson = hon && hn >= -1 && hn <= hm && (hx ? i0 + hn <= g.nx + 1 : j0 + hn <= g.ny + 1);

  R q[11][5], qn[5], uh[5];  // as k_filter_sf
  double qp[5];              // p at k-2..k+2
  double qpn = 0.0, ph = 0.0, sc = 1.0, scn = 1.0, sh = 1.0;
  auto put_u = [&](int b, const R c[5]) __attribute__((always_inline)) {
    if (own || past) {
#pragma unroll
      for (int v = 0; v < 5; v++) su[b][v][ty + 5][tx + 5] = c[v];
    }
    if (hon) {
#pragma unroll
      for (int v = 0; v < 5; v++) su[b][v][hr][hc] = uh[v];
    }
  };
  auto put_p = [&](int b, double pc) __attribute__((always_inline)) {
    if (pon) spr[b][ty + 2][tx + 2] = pc;
    if (hpon) spr[b][hr - 3][hc - 3] = ph;
  };
  // pressure sensors of a plane, from sc (own cell) and sh (halo cell)
  auto sensors = [&](int b) __attribute__((always_inline)) {
    const double *c = &spr[b][ty + 2][tx + 2];
    constexpr int W = FX + 4;
    if (sxon) psx[b][ty][tx + 1] = psens3(c[-1], c[0], c[1], sc, cs);
    if (syon) psy[b][ty + 1][tx] = psens3(c[-W], c[0], c[W], sc, cs);
    if (hson) {
      const double *h = &spr[b][hr - 3][hc - 3];
      const int d = hx ? 1 : W;
      const double e = psens3(h[-d], h[0], h[d], sh, cs);
      if (hx) psx[b][hr - 5][hc - 4] = e;
      else psy[b][hr - 4][hc - 5] = e;
    }
  };

  // ---- planes kbeg (state, p, sensors) and kbeg+1 (p) ----
  R dlo[5];        // D at the face k-1/2
  double ps0 = 0;  // pressure sensor along k at k
#pragma unroll
  for (int v = 0; v < 5; v++) dlo[v] = R(0);
  if (own) {
#pragma unroll
    for (int l = 0; l < 10; l++) ldr(uinp, own_off + (idx_t)wrap_k(g, kbeg - 5 + l) * sz, q[l]);
#pragma unroll
    for (int l = 0; l < 2; l++) qp[l] = ldg(prsp, own_off + (idx_t)wrap_k(g, kbeg - 2 + l) * sz);
  }
  if (pon) {
#pragma unroll
    for (int l = 2; l < 4; l++) qp[l] = ldg(prsp, own_off + (idx_t)wrap_k(g, kbeg - 2 + l) * sz);
  }
  if (duc && (sxon || syon)) sc = ldg(sensp, own_off + (idx_t)kbeg * sz);
  if (past) ldr(uinp, own_off + (idx_t)kbeg * sz, qn);
  if (hon) ldr(uinp, h_off + (idx_t)kbeg * sz, uh);
  if (hpon) ph = ldg(prsp, h_off + (idx_t)kbeg * sz);
  if (duc && hson) sh = ldg(sensp, h_off + (idx_t)kbeg * sz);
  {
    R c[5];
#pragma unroll
    for (int v = 0; v < 5; v++) c[v] = own ? q[5][v] : qn[v];
    put_u(kbeg & 1, c);
  }
  put_p(kbeg & 1, qp[2]);
  if (kbeg < kend) {
    if (hpon) ph = ldg(prsp, h_off + (idx_t)(kbeg + 1) * sz);
    put_p((kbeg & 1) ^ 1, qp[3]);
  }
  __syncthreads();
  sensors(kbeg & 1);
  if (own) {
    const double sm = duc ? ldg(sensp, own_off + (idx_t)wrap_k(g, kbeg - 1) * sz) : 1.0;
    const double pm = psens3(qp[0], qp[1], qp[2], sm, cs);
    ps0 = psens3(qp[1], qp[2], qp[3], sc, cs);
    const double xk0m = a.xnu0 * fmax(ps0, pm), xk10m = fmax(0.0, a.xnu10 + xk0m / 105.0);
#pragma unroll
    for (int v = 0; v < 5; v++) {
      dlo[v] = (q[5][v] - q[4][v]) * (R)xk0m +
               (R(D10_1) * (q[5][v] - q[4][v]) + R(D10_2) * (q[6][v] - q[3][v]) + R(D10_3) * (q[7][v] - q[2][v]) +
                R(D10_4) * (q[8][v] - q[1][v]) + R(D10_5) * (q[9][v] - q[0][v])) *
                   (R)xk10m;
    }
  }
  // in flight for plane kk = k+1 of the march: the state of the halo and of
  // points past the end at kk, the queue's kk+4 (and kk+5 from then on), p at
  // kk+1 and the sensors at kk
  auto load_ps = [&](int kk) __attribute__((always_inline)) {
    if (pon) qpn = ldg(prsp, own_off + (idx_t)wrap_k(g, kk + 1) * sz);
    if (duc && (sxon || syon)) scn = ldg(sensp, own_off + (idx_t)wrap_k(g, kk) * sz);
    if (kk + 1 <= kend && hpon) ph = ldg(prsp, h_off + (idx_t)(kk + 1) * sz);
    if (kk <= kend && duc && hson) sh = ldg(sensp, h_off + (idx_t)kk * sz);
  };
  if (own) ldr(uinp, own_off + (idx_t)wrap_k(g, kbeg + 5) * sz, qn);
  if (kbeg < kend) {
    if (past) ldr(uinp, own_off + (idx_t)(kbeg + 1) * sz, qn);
    if (hon) ldr(uinp, h_off + (idx_t)(kbeg + 1) * sz, uh);
  }
  load_ps(kbeg + 1);
  __syncthreads();

  for (int k = kbeg; k <= kend; k++) {
    const idx_t pk = own_off + (idx_t)k * sz;
    const int b = k & 1;
    if (own) {
#pragma unroll
      for (int v = 0; v < 5; v++) q[10][v] = qn[v];
    }
    qp[4] = qpn;
    sc = scn;
    if (k < kend) {
      R c[5];
#pragma unroll
      for (int v = 0; v < 5; v++) c[v] = own ? q[6][v] : qn[v];
      put_u(b ^ 1, c);
      if (k + 2 <= kend) put_p(b, qp[4]);
      sensors(b ^ 1);
      if (own) ldr(uinp, own_off + (idx_t)wrap_k(g, k + 6) * sz, qn);
      if (k + 2 <= kend) {
        if (past) ldr(uinp, pk + 2 * sz, qn);
        if (hon) ldr(uinp, h_off + (idx_t)(k + 2) * sz, uh);
      }
      load_ps(k + 2);
    }
    if (own) {
      R K[5];
      // i faces i-1/2 and i+1/2 (bounded i: rows 1..5 and nx-4..nx take theirs from k_shock_wall)
      if (WALL && (face_half_n(g.ibnd, g.nx, i - 1) < 5 || face_half_n(g.ibnd, g.nx, i) < 5)) {
#pragma unroll
        for (int v = 0; v < 5; v++) K[v] = R(0);
      } else {
        const double pm = psx[b][ty][tx], p0 = psx[b][ty][tx + 1], pp = psx[b][ty][tx + 2];
        const double xk0m = a.xnu0 * fmax(p0, pm), xk10m = fmax(0.0, a.xnu10 + xk0m / 105.0);
        const double xk0p = a.xnu0 * fmax(pp, p0), xk10p = fmax(0.0, a.xnu10 + xk0p / 105.0);
#pragma unroll
        for (int v = 0; v < 5; v++) {
          const R *x = &su[b][v][ty + 5][tx + 5];
          K[v] = dface<R>(x - 1, 1, (R)xk0m, (R)xk10m) - dface<R>(x, 1, (R)xk0p, (R)xk10p);
        }
      }
      // j faces (walls: rows 1..5 and ny-4..ny take theirs from k_shock_wall)
      if (!WALL || (face_half(g, j - 1) >= 5 && face_half(g, j) >= 5)) {
        const double pm = psy[b][ty][tx], p0 = psy[b][ty + 1][tx], pp = psy[b][ty + 2][tx];
        const double xk0m = a.xnu0 * fmax(p0, pm), xk10m = fmax(0.0, a.xnu10 + xk0m / 105.0);
        const double xk0p = a.xnu0 * fmax(pp, p0), xk10p = fmax(0.0, a.xnu10 + xk0p / 105.0);
#pragma unroll
        for (int v = 0; v < 5; v++) {
          const R *y = &su[b][v][ty + 5][tx + 5];
          K[v] = K[v] + dface<R>(y - SW, SW, (R)xk0m, (R)xk10m) - dface<R>(y, SW, (R)xk0p, (R)xk10p);
        }
      }
      // k face k+1/2 from the register queues
      {
        const double pp = psens3(qp[2], qp[3], qp[4], sc, cs);
        const double xk0p = a.xnu0 * fmax(pp, ps0), xk10p = fmax(0.0, a.xnu10 + xk0p / 105.0);
        ps0 = pp;
#pragma unroll
        for (int v = 0; v < 5; v++) {
          const R dhi = (q[6][v] - q[5][v]) * (R)xk0p +
                        (R(D10_1) * (q[6][v] - q[5][v]) + R(D10_2) * (q[7][v] - q[4][v]) +
                         R(D10_3) * (q[8][v] - q[3][v]) + R(D10_4) * (q[9][v] - q[2][v]) +
                         R(D10_5) * (q[10][v] - q[1][v])) * (R)xk10p;
          K[v] = K[v] + dlo[v] - dhi;
          dlo[v] = dhi;
        }
      }
#pragma unroll
      for (int v = 0; v < 5; v++) stg_nt(uoutp.v[v], pk, q[5][v] + K[v]);
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < 10; l++)
#pragma unroll
      for (int v = 0; v < 5; v++) q[l][v] = q[l + 1][v];
#pragma unroll
    for (int l = 0; l < 4; l++) qp[l] = qp[l + 1];
  }
}

// ARTV: the artificial viscosity.  The LDS "pressure" pencils then hold the
// spectral radii sr_x (i-pencil) and sr_y (j-pencil), the k queue sr_z.
// AVS: the artificial viscosity with shock capturing (artvisc_o9_shock,
// mod_artvisc_shock.f90:113-1287): the shock filter's faces D, each
// direction's K = (sr_{-1/2} D_{-1/2} - sr_{+1/2} D_{+1/2}) * metric with the
// spectral radius of U^n averaged to the faces (:480-550 i, :866-935 j,
// :1243-1283 k), U_n += deltat*K (update_varn_artvisc).
// WALL: blocks with boundary faces on i or j; rows 1..5 and n-4..n of a
// bounded axis get no increment along it here (k_shock_wall adds it with the
// reduced faces of the boundary closure).
// EDOH: the shock filter's Edoh switch, each direction's increment times
// min(1, CFL_d / chi) with the local CFL_d = sr_d deltat (idx_d on Cartesian
// blocks) (mod_filtering_shock.f90:620-700, :1059-1140, :1450-1496).
template <bool ARTV, bool WALL, bool EDOH, bool AVS>
__global__ __launch_bounds__(FT, 2) void k_filter_shock(const Batch<FilterArgs> *__restrict__ tab, int nb,
                                                        int ntiles) {
  static_assert(ARTV || EDOH || AVS, "the shock filter alone is k_shock");
  static_assert(!(WALL && ARTV), "walls: not with artvisc_o9");
  static_assert(!(EDOH && (ARTV || AVS)), "the Edoh switch belongs to the shock filter");
  static_assert(!(AVS && ARTV), "one artificial viscosity at a time");
  using R = double;
  __shared__ R sux[5][FY][FX + 10];
  __shared__ R suy[5][FY + 10][FX];
  __shared__ double spx[FY][FX + 4];    // p at i0-2 .. i0+FX+1
  __shared__ double spy[FY + 4][FX];    // p at j0-2 .. j0+FY+1
  __shared__ double ssx[FY][FX + 4];    // sensor at i0-2 .. i0+FX+1 (ends unused)
  __shared__ double ssy[FY + 4][FX];    // sensor at j0-2 .. j0+FY+1 (ends unused)
  __shared__ double psx[FY][FX + 2];    // psens_x at i0-1 .. i0+FX
  __shared__ double psy[FY + 2][FX];    // psens_y at j0-1 .. j0+FY
  // Edoh factors of the plane's own points (AVS: the face spectral radii
  // sr_{-1/2}, sr_{+1/2} of the three directions, then their metrics; ARTV:
  // the metrics)
  __shared__ double smul[EDOH || ARTV ? 3 : (AVS ? 9 : 1)][FY][FX];

  int i0, j0, kbeg, kend;
  const FilterArgs &a = tile_of(tab, nb, ntiles, i0, j0, kbeg, kend);
  // the block's array pointers, read once from the table into registers
  const CState uinp = a.uin;
  const State uoutp = a.uout;
  const double *const prsp = ARTV ? a.sr[2] : a.prs, *const sensp = a.sens;
  const double *const px = ARTV ? a.sr[0] : a.prs, *const py = ARTV ? a.sr[1] : a.prs;
  const Geom &g = a.g;
  const int tid = threadIdx.x, tx = tid % FX, ty = tid / FX;
  const int i = i0 + tx, j = j0 + ty;
  const bool own = i <= g.nx && j <= g.ny;
  const bool needx = i <= g.nx + 5 && j <= g.ny, needy = i <= g.nx && j <= g.ny + 5;
  const bool duc = !ARTV && a.sens != nullptr;
  const double cs = a.csens;
  const idx_t sz = g.sy, own_off = lin_w(g, i, j);
  Halo hl;
  halo_setup(g, i0, j0, hl);
  // p / sensor cells of this thread: rows of spx (i-direction) then of spy
  idx_t pp_off[NSP];
  int pp_r[NSP], pp_c[NSP];
  bool pp_on[NSP], pp_x[NSP], pp_s[NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) {
    const int t = tid + s * FT;
    pp_on[s] = false;
    pp_x[s] = true;
    pp_s[s] = false;
    pp_r[s] = pp_c[s] = 0;
    pp_off[s] = 0;
    if (t < NPX) {
      const int r = t / (FX + 4), c = t % (FX + 4);
      const int gi = i0 - 2 + c, gj = j0 + r;
      pp_on[s] = gj <= g.ny && gi <= g.nx + 2;
      pp_s[s] = c >= 1 && c <= FX + 2 && gi <= g.nx + 1;  // sensor needed at i0-1..i0+FX
      pp_r[s] = r;
      pp_c[s] = c;
      pp_off[s] = lin_w(g, gi, gj);
    } else if (t < NPX + NPY) {
      const int tt = t - NPX;
      const int r = tt / FX, c = tt % FX;
      const int gi = i0 + c, gj = j0 - 2 + r;
      pp_on[s] = gi <= g.nx && gj <= g.ny + 2;
      pp_s[s] = r >= 1 && r <= FY + 2 && gj <= g.ny + 1;
      pp_x[s] = false;
      pp_r[s] = r;
      pp_c[s] = c;
      pp_off[s] = lin_w(g, gi, gj);
    }
  }

  R q[11][5];        // U at k-5..k+5
  double qp[5];      // p at k-2..k+2 (ARTV: |w|+c at k-1..k+1 in qp[0..2])
  double qs[3];      // sensor at k-1..k+1
  if (own) {
#pragma unroll
    for (int l = 0; l < 10; l++) ldr(uinp, own_off + (idx_t)wrap_k(g, kbeg - 5 + l) * sz, q[l]);
    if constexpr (ARTV) {
#pragma unroll
      for (int l = 0; l < 2; l++) qp[l] = ldg(prsp, own_off + (idx_t)wrap_k(g, kbeg - 1 + l) * sz);
    } else {
#pragma unroll
      for (int l = 0; l < 4; l++) qp[l] = ldg(prsp, own_off + (idx_t)wrap_k(g, kbeg - 2 + l) * sz);
    }
#pragma unroll
    for (int l = 0; l < 2; l++) qs[l] = duc ? ldg(sensp, own_off + (idx_t)wrap_k(g, kbeg - 1 + l) * sz) : 1.0;
  }

  // every global load of a plane is issued one plane ahead, during the
  // previous plane's stencils: queue points, pencil cell, halo cells, p/sensor
  R qn[5], uc[5], uh[NS][5];
  double qpn = 0.0, qsn = 1.0, pv[NSP], sv[NSP];
  auto load_plane = [&](int kk) {
    const idx_t pkk = own_off + (idx_t)kk * sz;
    if (own) {
      const idx_t p1 = own_off + (idx_t)wrap_k(g, kk + 1) * sz;
      ldr(uinp, own_off + (idx_t)wrap_k(g, kk + 5) * sz, qn);
      qpn = ARTV ? ldg(prsp, p1) : ldg(prsp, own_off + (idx_t)wrap_k(g, kk + 2) * sz);
      qsn = duc ? ldg(sensp, p1) : 1.0;
    }
    if (!own && (needx || needy)) ldr(uinp, pkk, uc);
#pragma unroll
    for (int s = 0; s < NS; s++)
      if (hl.on[s]) ldr(uinp, hl.off[s] + (idx_t)kk * sz, uh[s]);
#pragma unroll
    for (int s = 0; s < NSP; s++) {
      if (pp_on[s]) {
        pv[s] = ldg(pp_x[s] ? px : py, pp_off[s] + (idx_t)kk * sz);
        sv[s] = (duc && pp_s[s]) ? ldg(sensp, pp_off[s] + (idx_t)kk * sz) : 1.0;
      }
    }
  };
  load_plane(kbeg);

  for (int k = kbeg; k <= kend; k++) {
    const idx_t pk = own_off + (idx_t)k * sz;
    if (own) {
#pragma unroll
      for (int v = 0; v < 5; v++) q[10][v] = qn[v];
      if constexpr (ARTV) qp[2] = qpn;
      else qp[4] = qpn;
      qs[2] = qsn;
    }
    // ---- stage the plane in LDS ----
    if (needx || needy) {
#pragma unroll
      for (int v = 0; v < 5; v++) {
        const R x = own ? q[5][v] : uc[v];
        if (needx) sux[v][ty][tx + 5] = x;
        if (needy) suy[v][ty + 5][tx] = x;
      }
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
      if (hl.on[s]) {
#pragma unroll
        for (int v = 0; v < 5; v++) {
          if (hl.xdir[s]) sux[v][hl.r[s]][hl.c[s]] = uh[s][v];
          else suy[v][hl.r[s]][hl.c[s]] = uh[s][v];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < NSP; s++) {
      if (pp_on[s]) {
        if (pp_x[s]) {
          spx[pp_r[s]][pp_c[s]] = pv[s];
          ssx[pp_r[s]][pp_c[s]] = sv[s];
        } else {
          spy[pp_r[s]][pp_c[s]] = pv[s];
          ssy[pp_r[s]][pp_c[s]] = sv[s];
        }
      }
    }
    if constexpr (EDOH) {
      // computed here and kept in LDS, so that nothing of them stays in
      // registers through the stencils
      if (own) {
        smul[0][ty][tx] = edoh_mul(a, 0, pk, i);
        smul[1][ty][tx] = edoh_mul(a, 1, pk, j);
        smul[2][ty][tx] = edoh_mul(a, 2, pk, k);
      }
    }
    if constexpr (AVS) {
      if (own) {
        double s0 = ldg(a.sr[0], pk);
        smul[0][ty][tx] = 0.5 * (ldg(a.sr[0], pk - 1) + s0);
        smul[1][ty][tx] = 0.5 * (ldg(a.sr[0], pk + 1) + s0);
        s0 = ldg(a.sr[1], pk);
        smul[2][ty][tx] = 0.5 * (ldg(a.sr[1], pk - g.sx) + s0);
        smul[3][ty][tx] = 0.5 * (ldg(a.sr[1], pk + g.sx) + s0);
        s0 = ldg(a.sr[2], pk);
        smul[4][ty][tx] = 0.5 * (ldg(a.sr[2], pk - sz) + s0);
        smul[5][ty][tx] = 0.5 * (ldg(a.sr[2], pk + sz) + s0);
        smul[6][ty][tx] = met_at(a.idx, i);
        smul[7][ty][tx] = met_at(a.idy, j);
        smul[8][ty][tx] = met_at(a.idz, k);
      }
    }
    if constexpr (ARTV) {
      if (own) {
        smul[0][ty][tx] = met_at(a.idx, i);
        smul[1][ty][tx] = met_at(a.idy, j);
        smul[2][ty][tx] = met_at(a.idz, k);
      }
    }
    __syncthreads();
    if (k < kend) load_plane(k + 1);
    // pressure sensors of the plane
    for (int t = tid; t < (ARTV ? 0 : FY * (FX + 2)); t += FT) {
      const int r = t / (FX + 2), c = t % (FX + 2);
      const int gi = i0 - 1 + c, gj = j0 + r;
      if (gj <= g.ny && gi <= g.nx + 1)
        psx[r][c] = psens3(spx[r][c], spx[r][c + 1], spx[r][c + 2], ssx[r][c + 1], cs);
    }
    for (int t = tid; t < (ARTV ? 0 : (FY + 2) * FX); t += FT) {
      const int r = t / FX, c = t % FX;
      const int gi = i0 + c, gj = j0 - 1 + r;
      if (gi <= g.nx && gj <= g.ny + 1)
        psy[r][c] = psens3(spy[r][c], spy[r + 1][c], spy[r + 2][c], ssy[r + 1][c], cs);
    }
    __syncthreads();

    if (ARTV && own) {
      // K_d = (sr_{+1/2} D_{+1/2} - sr_{-1/2} D_{-1/2}) * metric with D = -x10 * d10face
      const double x10 = a.xnu10;
      double K[5];
      {
        const double s0 = spx[ty][tx + 2], srp = 0.5 * (spx[ty][tx + 3] + s0), srm = 0.5 * (spx[ty][tx + 1] + s0);
        const double m = smul[0][ty][tx];
#pragma unroll
        for (int v = 0; v < 5; v++) {
          const R *x = &sux[v][ty][tx + 5];
          K[v] = (srm * (x10 * (double)d10face<R>(x - 1, 1)) - srp * (x10 * (double)d10face<R>(x, 1))) * m;
        }
      }
      {
        const double s0 = spy[ty + 2][tx], srp = 0.5 * (spy[ty + 3][tx] + s0), srm = 0.5 * (spy[ty + 1][tx] + s0);
        const double m = smul[1][ty][tx];
#pragma unroll
        for (int v = 0; v < 5; v++) {
          const R *y = &suy[v][ty + 5][tx];
          K[v] = K[v] + (srm * (x10 * (double)d10face<R>(y - FX, FX)) - srp * (x10 * (double)d10face<R>(y, FX))) * m;
        }
      }
      {
        const double s0 = qp[1], srp = 0.5 * (qp[2] + s0), srm = 0.5 * (qp[0] + s0);
        const double m = smul[2][ty][tx];
#pragma unroll
        for (int v = 0; v < 5; v++) {
          const double dlo = R(D10_1) * (q[5][v] - q[4][v]) + R(D10_2) * (q[6][v] - q[3][v]) +
                             R(D10_3) * (q[7][v] - q[2][v]) + R(D10_4) * (q[8][v] - q[1][v]) +
                             R(D10_5) * (q[9][v] - q[0][v]);
          const double dhi = R(D10_1) * (q[6][v] - q[5][v]) + R(D10_2) * (q[7][v] - q[4][v]) +
                             R(D10_3) * (q[8][v] - q[3][v]) + R(D10_4) * (q[9][v] - q[2][v]) +
                             R(D10_5) * (q[10][v] - q[1][v]);
          K[v] = K[v] + (srm * (x10 * dlo) - srp * (x10 * dhi)) * m;
        }
      }
#pragma unroll
      for (int v = 0; v < 5; v++) {
        stg_nt(uoutp.v[v], pk, q[5][v] + a.dt * K[v]);
      }
    }
    if (!ARTV && own) {
      R K[5];
      // i faces i-1/2 and i+1/2 (bounded i: rows 1..5 and nx-4..nx take theirs from k_shock_wall)
      if (WALL && (face_half_n(g.ibnd, g.nx, i - 1) < 5 || face_half_n(g.ibnd, g.nx, i) < 5)) {
#pragma unroll
        for (int v = 0; v < 5; v++) K[v] = R(0);
      } else {
        const double pm = psx[ty][tx], p0 = psx[ty][tx + 1], pp = psx[ty][tx + 2];
        const double xk0m = a.xnu0 * fmax(p0, pm), xk10m = fmax(0.0, a.xnu10 + xk0m / 105.0);
        const double xk0p = a.xnu0 * fmax(pp, p0), xk10p = fmax(0.0, a.xnu10 + xk0p / 105.0);
        const R mul = EDOH ? (R)smul[0][ty][tx] : R(1);
        double srm = 0.0, srp = 0.0, m = 1.0;
        if constexpr (AVS) {
          srm = smul[0][ty][tx];
          srp = smul[1][ty][tx];
          m = smul[6][ty][tx];
        }
#pragma unroll
        for (int v = 0; v < 5; v++) {
          const R *x = &sux[v][ty][tx + 5];
          if constexpr (AVS)
            K[v] = (srm * dface<R>(x - 1, 1, (R)xk0m, (R)xk10m) - srp * dface<R>(x, 1, (R)xk0p, (R)xk10p)) * m;
          else K[v] = mul * (dface<R>(x - 1, 1, (R)xk0m, (R)xk10m) - dface<R>(x, 1, (R)xk0p, (R)xk10p));
        }
      }
      // j faces (walls: rows 1..5 and ny-4..ny take theirs from k_shock_wall)
      if (!WALL || (face_half(g, j - 1) >= 5 && face_half(g, j) >= 5)) {
        const double pm = psy[ty][tx], p0 = psy[ty + 1][tx], pp = psy[ty + 2][tx];
        const double xk0m = a.xnu0 * fmax(p0, pm), xk10m = fmax(0.0, a.xnu10 + xk0m / 105.0);
        const double xk0p = a.xnu0 * fmax(pp, p0), xk10p = fmax(0.0, a.xnu10 + xk0p / 105.0);
        const R mul = EDOH ? (R)smul[1][ty][tx] : R(1);
        double srm = 0.0, srp = 0.0, m = 1.0;
        if constexpr (AVS) {
          srm = smul[2][ty][tx];
          srp = smul[3][ty][tx];
          m = smul[7][ty][tx];
        }
#pragma unroll
        for (int v = 0; v < 5; v++) {
          const R *y = &suy[v][ty + 5][tx];
          if constexpr (AVS)
            K[v] = K[v] +
                   (srm * dface<R>(y - FX, FX, (R)xk0m, (R)xk10m) - srp * dface<R>(y, FX, (R)xk0p, (R)xk10p)) * m;
          else K[v] = K[v] + mul * (dface<R>(y - FX, FX, (R)xk0m, (R)xk10m) - dface<R>(y, FX, (R)xk0p, (R)xk10p));
        }
      }
      // k faces from the register queues
      {
        const double pm = psens3(qp[0], qp[1], qp[2], qs[0], cs);
        const double p0 = psens3(qp[1], qp[2], qp[3], qs[1], cs);
        const double pp = psens3(qp[2], qp[3], qp[4], qs[2], cs);
        const double xk0m = a.xnu0 * fmax(p0, pm), xk10m = fmax(0.0, a.xnu10 + xk0m / 105.0);
        const double xk0p = a.xnu0 * fmax(pp, p0), xk10p = fmax(0.0, a.xnu10 + xk0p / 105.0);
        const R mul = EDOH ? (R)smul[2][ty][tx] : R(1);
        double srm = 0.0, srp = 0.0, m = 1.0;
        if constexpr (AVS) {
          srm = smul[4][ty][tx];
          srp = smul[5][ty][tx];
          m = smul[8][ty][tx];
        }
#pragma unroll
        for (int v = 0; v < 5; v++) {
          const R dlo = (q[5][v] - q[4][v]) * (R)xk0m +
                        (R(D10_1) * (q[5][v] - q[4][v]) + R(D10_2) * (q[6][v] - q[3][v]) +
                         R(D10_3) * (q[7][v] - q[2][v]) + R(D10_4) * (q[8][v] - q[1][v]) +
                         R(D10_5) * (q[9][v] - q[0][v])) * (R)xk10m;
          const R dhi = (q[6][v] - q[5][v]) * (R)xk0p +
                        (R(D10_1) * (q[6][v] - q[5][v]) + R(D10_2) * (q[7][v] - q[4][v]) +
                         R(D10_3) * (q[8][v] - q[3][v]) + R(D10_4) * (q[9][v] - q[2][v]) +
                         R(D10_5) * (q[10][v] - q[1][v])) * (R)xk10p;
          if constexpr (AVS) K[v] = K[v] + (srm * dlo - srp * dhi) * m;
          else K[v] = K[v] + mul * (dlo - dhi);
        }
      }
#pragma unroll
      for (int v = 0; v < 5; v++) {
        if constexpr (AVS) stg_nt(uoutp.v[v], pk, q[5][v] + a.dt * K[v]);
        else stg_nt(uoutp.v[v], pk, q[5][v] + K[v]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < 10; l++)
#pragma unroll
      for (int v = 0; v < 5; v++) q[l][v] = q[l + 1][v];
    if constexpr (ARTV) {
      qp[0] = qp[1];
      qp[1] = qp[2];
    } else {
#pragma unroll
      for (int l = 0; l < 4; l++) qp[l] = qp[l + 1];
    }
    qs[0] = qs[1];
    qs[1] = qs[2];
  }
}

// Differences d2, d4, d6, d8, d10 of the face dissipation by half-width
// (init_filter_shock with iSF = 0, mod_filtering_shock.f90:75-107).
__constant__ double kShockD[6][5] = {{0.0, 0.0, 0.0, 0.0, 0.0},     {-1.0, 0.0, 0.0, 0.0, 0.0},
                                     {-3.0, 1.0, 0.0, 0.0, 0.0},    {-10.0, 5.0, -1.0, 0.0, 0.0},
                                     {-35.0, 21.0, -7.0, 1.0, 0.0}, {D10_1, D10_2, D10_3, D10_4, D10_5}};

constexpr int kShockWallThreads = 256;

// Shock filter increment along axis ax (0: i, 1: j) of the rows next to the
// bounded faces of that axis, added to the output of the WALL kernels above
// (which leaves rows 1..5 and n-4..n of a bounded axis without one): faces
// 1..4 from a boundary use d2/d4/d6/d8 with amplitude max(0, xnu + xk0), the
// boundary face a tenth of the sensor term (filter_o10_shock,
// mod_filtering_shock.f90:266-466 i, :724-870 jmin, :915-1057 jmax); the
// boundary rows get none (:1128-1140 over ndy_d..nfy_d).  The pressure
// sensor of row 1 (n) reads p one row beyond the face.  One thread per point
// of rows 2..5 and n-4..n-1 of each bounded side; nothing beyond a face is
// read but p.
// a.avs: artvisc_o9_shock (j only), whose faces 3 and 4 from a wall take
// xk0/5 and 3/70 xk0 (mod_artvisc_shock.f90:577-695 jmin, :744-862 jmax) and
// whose increment is deltat (sr_{-1/2} D_{-1/2} - sr_{+1/2} D_{+1/2}) idy(j).
__global__ __launch_bounds__(kShockWallThreads) void k_shock_wall(FilterArgs a, int ax) {
  const Geom &g = a.g;
  const int bnd = ax ? g.jbnd : g.ibnd, n = ax ? g.ny : g.nx;
  const int n1 = ax ? g.nx : g.ny;  // the other in-plane axis
  const long nface = (long)n1 * g.nz;
  const long t = (long)blockIdx.x * kShockWallThreads + threadIdx.x;
  if (t >= 8 * nface) return;
  const int q = (int)(t / nface);
  const int side = q >> 2;
  if (!((bnd >> side) & 1)) return;
  const long r = t - q * nface;
  const int a1 = 1 + (int)(r % n1), k = 1 + (int)(r / n1);
  const int m0 = side ? n - 4 + (q & 3) : 2 + (q & 3);  // row along ax
  const idx_t sj = ax ? (idx_t)g.sx : (idx_t)1;
  const idx_t pj = ax ? lin(g, a1, m0, k) : lin(g, m0, a1, k);
  // pressure sensors of rows m0-1, m0, m0+1 (faces m0-1/2, m0+1/2)
  double ps[3];
#pragma unroll
  for (int l = 0; l < 3; l++) {
    const idx_t pm = pj + (l - 1) * sj;
    const double sn = a.sens ? ldg(a.sens, pm) : 1.0;
    ps[l] = psens3(ldg(a.prs, pm - sj), ldg(a.prs, pm), ldg(a.prs, pm + sj), sn, a.csens);
  }
  double D[2][5];
#pragma unroll
  for (int f = 0; f < 2; f++) {
    const int m = m0 - 1 + f;
    const int hf = face_half_n(bnd, n, m);
    // no sensor term (artvisc_o9): p beyond the wall is not read into it
    double xk0 = a.xnu0 == 0.0 ? 0.0 : a.xnu0 * fmax(ps[f + 1], ps[f]);
    if (hf == 1) xk0 = xk0 / 10.0;
    double xkh;
    switch (hf) {
      case 1: xkh = fmax(0.0, 0.0 + xk0); break;
      case 2: xkh = fmax(0.0, a.chi / 12.0 + xk0); break;
      case 3: xkh = fmax(0.0, a.chi / 60.0 + (a.avs ? xk0 / 5.0 : xk0)); break;
      case 4: xkh = fmax(0.0, a.chi / 280.0 + (a.avs ? 3.0 / 70.0 * xk0 : xk0)); break;
      default: xkh = fmax(0.0, a.xnu10 + xk0 / 105.0);
    }
    const idx_t pf = pj + (f - 1) * sj;  // row m
#pragma unroll
    for (int v = 0; v < 5; v++) {
      const double *u = a.uin.v[v];
      const double d1 = ldg(u, pf + sj) - ldg(u, pf);
      double dd = 0.0;
      for (int l = 1; l <= hf; l++) dd = dd + kShockD[hf][l - 1] * (ldg(u, pf + l * sj) - ldg(u, pf + (1 - l) * sj));
      D[f][v] = d1 * xk0 + dd * xkh;
    }
  }
  if (a.avs) {
    const double s0 = ldg(a.sr[1], pj);
    const double srp = 0.5 * (ldg(a.sr[1], pj + sj) + s0), srm = 0.5 * (ldg(a.sr[1], pj - sj) + s0);
    const double m = met_at(a.idy, m0);
#pragma unroll
    for (int v = 0; v < 5; v++)
      stg(a.uout.v[v], pj, ldg(a.uout.v[v], pj) + a.dt * ((srm * D[0][v] - srp * D[1][v]) * m));
    return;
  }
  const double mul = a.edoh ? edoh_mul(a, ax, pj, m0) : 1.0;
#pragma unroll
  for (int v = 0; v < 5; v++) {
    const double kd = a.edoh ? mul * (D[0][v] - D[1][v]) : D[0][v] - D[1][v];
    stg(a.uout.v[v], pj, ldg(a.uout.v[v], pj) + kd);
  }
}

}  // namespace

hipError_t launch_shock_wall(const FilterArgs &a, int axis, hipStream_t s) {
  if (axis == 0 && a.avs) return hipErrorInvalidValue;  // artvisc_o9_shock: j-walls only
  const long n = 8L * (axis ? a.g.nx : a.g.ny) * a.g.nz;
  hipLaunchKernelGGL(k_shock_wall, dim3((unsigned)((n + kShockWallThreads - 1) / kShockWallThreads)),
                     dim3(kShockWallThreads), 0, s, a, axis);
  return hipGetLastError();
}

// Tiles of the filters: 32x16, chunks of kc planes.
TileRange filter_tiles(const Geom &g, int kc) {
  TileRange t{};
  t.tiles_x = (g.nx + FX - 1) / FX;
  t.tiles_y = (g.ny + FY - 1) / FY;
  t.kchunk = kc < 1 ? 1 : (kc > g.nz ? g.nz : kc);
  return t;
}

hipError_t launch_filter_sf(const Batch<FilterArgs> *tab, int nb, int nt, bool wall, hipStream_t s) {
  if (nt <= 0) return hipSuccess;
  if (wall) hipLaunchKernelGGL((k_filter_sf<true>), dim3(nt), dim3(FT), 0, s, tab, nb, nt);
  else hipLaunchKernelGGL((k_filter_sf<false>), dim3(nt), dim3(FT), 0, s, tab, nb, nt);
  return hipGetLastError();
}

hipError_t launch_filter_shock(const Batch<FilterArgs> *tab, int nb, int nt, DissipKind kind, bool wall, bool edoh,
                               hipStream_t s) {
  if (nt <= 0) return hipSuccess;
  if (kind == kDissipArtvisc) {
    if (wall || edoh) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_filter_shock<true, false, false, false>), dim3(nt), dim3(FT), 0, s, tab, nb, nt);
  } else if (kind == kDissipArtviscShock) {
    if (edoh) return hipErrorInvalidValue;
    if (wall) hipLaunchKernelGGL((k_filter_shock<false, true, false, true>), dim3(nt), dim3(FT), 0, s, tab, nb, nt);
    else hipLaunchKernelGGL((k_filter_shock<false, false, false, true>), dim3(nt), dim3(FT), 0, s, tab, nb, nt);
  } else if (edoh) {
    if (wall) hipLaunchKernelGGL((k_filter_shock<false, true, true, false>), dim3(nt), dim3(FT), 0, s, tab, nb, nt);
    else hipLaunchKernelGGL((k_filter_shock<false, false, true, false>), dim3(nt), dim3(FT), 0, s, tab, nb, nt);
  } else {
    if (wall) hipLaunchKernelGGL((k_shock<true>), dim3(nt), dim3(FT), 0, s, tab, nb, nt);
    else hipLaunchKernelGGL((k_shock<false>), dim3(nt), dim3(FT), 0, s, tab, nb, nt);
  }
  return hipGetLastError();
}

}  // namespace mgpu
