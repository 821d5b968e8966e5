// k_multigrid.hip - geometric multigrid solve of the pressure equation
// (poisson_solver = ELMM_POISSON_MG), the role of PoissMG
// (src/multigrid.f90:1047-1172: V-cycle MG_CGC 994-1044, smoother MG_GS
// 786-910, residual MG_res 912-977, Restrict 114-165, Prolongate 58-111).
//
// The operator is the cell-centred one of Residue_variable_z
// (src/poisson.f90:23-60) that the spectral solver inverts: periodic x and
// y, staggered Neumann walls in z, stretched z.  Levels coarsen x and y by 2
// and keep every z level, so the z coefficients are the same on all of them
// and a z-line smoother handles the strong vertical coupling of stretched
// grids.  Arrays of a level are dense, nx x ny x nz doubles, x fastest.
//
// Operation order (shared with the oracle, so the two agree bit for bit):
//   sweep (one colour, (i + j) & 1): per column, h_k = ax (P_w + P_e) +
//     ay (P_s + P_n), g_k = ((h_k - rhs_k) + az_k g_{k-1}) / den_k, then
//     P_k = g_k + e_k P_{k+1} from the top; den_k, e_k are host tables;
//   residual r = rhs - s, s = ((P_w - P) + (P_e - P)) ax + ((P_s - P) +
//     (P_n - P)) ay [+ az_k (P_b - P)] [+ cz_k (P_t - P)];
//   restriction rhs_c = ((r1 + r2) + (r3 + r4)) * 0.25 (children in x
//     pairs, lower y first), P_c = 0;
//   prolongation P += 0.75 (0.75 c + 0.25 c_x) + 0.25 (0.75 c_y + 0.25 c_xy);
//   coarsest level: exact, by discrete Fourier sums in x and y and a
//     tridiagonal elimination in z per mode (k_mg_coarse).
#include <cmath>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace elmm {

namespace {

inline unsigned nblk(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

__device__ inline int wrap_lo(int i, int n) { return i > 1 ? i - 1 : n; }
__device__ inline int wrap_hi(int i, int n) { return i < n ? i + 1 : 1; }

// residual of cell (i, j, k) (1-based) of a level
__device__ inline double mg_res(const MgLevel &L, const double *__restrict__ az, const double *__restrict__ cz, int i,
                                int j, int k) {
  const int nx = L.nx, ny = L.ny;
  const long plane = (long)nx * ny, o = (long)(k - 1) * plane;
  const double *P = L.phi;
  const long c = (i - 1) + (long)(j - 1) * nx + o;
  const double p = P[c];
  double s = ((P[(wrap_lo(i, nx) - 1) + (long)(j - 1) * nx + o] - p) + (P[(wrap_hi(i, nx) - 1) + (long)(j - 1) * nx + o] - p)) *
                 L.ax +
             ((P[(i - 1) + (long)(wrap_lo(j, ny) - 1) * nx + o] - p) + (P[(i - 1) + (long)(wrap_hi(j, ny) - 1) * nx + o] - p)) *
                 L.ay;
  if (k > 1) s = s + az[k - 1] * (P[c - plane] - p);
  if (k < L.nz) s = s + cz[k - 1] * (P[c + plane] - p);
  return L.rhs[c] - s;
}

}  // namespace

// Right-hand side of the pressure equation (PrePoisson, src/pressure.f90:
// 657-717): ((U_i - U_{i-1})/dx + (V_j - V_{j-1})/dy + (W_k - W_{k-1})/dz
// - Q) / coef, into the dense level-0 array and the ghosted RHS.
template <typename T>
__global__ void __launch_bounds__(256) k_mg_rhs(Geo g, const T *__restrict__ U, const T *__restrict__ V,
                                                const T *__restrict__ W, const double *__restrict__ Q, double dt2_rec,
                                                double *__restrict__ rhs0, double *__restrict__ RHS) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)g.nx * g.ny * g.nz) return;
  const int i = (int)(t % g.nx) + 1, j = (int)((t / g.nx) % g.ny) + 1, k = (int)(t / ((long)g.nx * g.ny)) + 1;
  const long p = gix(g, i, j, k);
  const double dz = g.variable_z ? g.dzPr[k] : g.dzmin;
  // U(0) and V(0) by index wrap (periodic x and y), W = 0 on the walls (see
  // k_fft_x_fwd)
  const long pw = i > 1 ? p - 1 : p - 1 + g.nx, ps = j > 1 ? p - g.sy : p - g.sy + (long)g.ny * g.sy;
  const double wt = (double)W[p], wb = (double)W[p - g.sz];
  double r = ((double)U[p] - (double)U[pw]) / g.dxmin + ((double)V[p] - (double)V[ps]) / g.dymin +
             ((k < g.nz ? wt : 0.0) - (k > 1 ? wb : 0.0)) / dz;
  if (Q) r = r - Q[p];
  r = r * dt2_rec;
  rhs0[t] = r;
  RHS[p] = r;
}

// Level-0 solution into the ghosted Phi interior.
__global__ void __launch_bounds__(256) k_mg_to_phi(Geo g, const double *__restrict__ phi0, double *__restrict__ Phi) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)g.nx * g.ny * g.nz) return;
  const int i = (int)(t % g.nx) + 1, j = (int)((t / g.nx) % g.ny) + 1, k = (int)(t / ((long)g.nx * g.ny)) + 1;
  Phi[gix(g, i, j, k)] = phi0[t];
}

__global__ void __launch_bounds__(256) k_mg_zero(double *__restrict__ a, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) a[t] = 0.0;
}

// Line Gauss-Seidel sweep of one colour: Thomas elimination up every column
// with (i + j) & 1 == color (the same colour's columns are not neighbours),
// then back down.  The serial part is one product-sum-quotient per level; its
// inputs h - rhs need only the other colour, so a block first forms them for
// COLS columns and all levels with every load in flight, keeps the columns in
// LDS for the two passes, and writes them back.  (One thread per column
// loading as it went: 30 us a sweep of 128x64 columns of 64 levels, bound by
// a memory round trip per four levels; staged about 9.)
// Levels are padded to whole groups of ZB, so the chain carries no conditions
// and a group's operands are fetched while the previous group is worked
// through.
constexpr int kMgCols = 16, kMgThreads = 256, ZB = 4;
__host__ __device__ constexpr int mg_pad(int nz) { return (nz + ZB - 1) / ZB * ZB; }
// the columns of a block and the tables of MgTab: up to 1024 levels fit a CU
constexpr size_t mg_sweep_lds(int nz) { return (size_t)mg_pad(nz) * (kMgCols + 4) * sizeof(double); }
static_assert(mg_sweep_lds(1024) <= 160 * 1024 && mg_sweep_lds(1025) > 160 * 1024, "k_mg_sweep's tallest column");
// Tables of a sweep in LDS: az, den, RN(1/den) and e of each level.
struct MgTab {
  double *az, *den, *rden, *e;
};
__device__ inline MgTab mg_tab_at(double *p, int np) { return MgTab{p, p + np, p + 2 * np, p + 3 * np}; }
template <int TH>
__device__ inline void mg_tab_fill(MgTab t, const double *__restrict__ az, const double *__restrict__ den,
                                   const double *__restrict__ e, int nz, int np) {
  for (int k = threadIdx.x; k < np; k += TH) {
    const int kc = min(k, nz - 1);
    const double a = az[kc], d = den[kc], ek = e[kc];
    t.az[k] = k < nz ? a : 0.0;
    t.den[k] = k < nz ? d : 1.0;
    t.rden[k] = k < nz ? (fabs(d) >= 0x1p-200 && fabs(d) <= 0x1p200 ? 1.0 / d : 0.0) : 1.0;
    t.e[k] = k < nz ? ek : 0.0;
  }
}

// Thomas elimination up a column of np levels at x[k * S] (h - rhs on entry,
// 1 above level nz; P on return) and back down.
// A column is one lane of one wave, whose time is its instructions one after
// another.  The quotient is formed from r = RN(1/d) in 5 instead of 11: q0 =
// RN(x r) is within two ulp of x/d, one Newton step gives a q1 within one
// ulp, and then RN(q1 + (x - q1 d) r) is the correctly rounded quotient (P.
// Markstein, IBM J. Res. Dev. 34, 1990), as long as no remainder underflows:
// a group of levels with a quotient outside 2^-700..2^700 (zeros too: their
// sign; r = 0 marks a d outside 2^-200..2^200) is done again with divisions.
template <int S>
__device__ inline void mg_column(double *x, MgTab tb, int nz, int np) {
  double xc[ZB], ac[ZB], dc[ZB], rc[ZB];
  double gv = 0;
  // 2^-700 <= |v| < 2^700 as one unsigned range of the upper word
  constexpr unsigned lo = (1023u - 700) << 20, range = 1400u << 20;
  auto fetch = [&](int k0, const double *p, double *xo, double *ao) {
#pragma unroll
    for (int b = 0; b < ZB; b++) {
      xo[b] = x[(k0 + b) * S];
      ao[b] = p[k0 + b];
    }
  };
  auto fetch_d = [&](int k0, double *dd, double *rr) {
#pragma unroll
    for (int b = 0; b < ZB; b++) {
      dd[b] = tb.den[k0 + b];
      rr[b] = tb.rden[k0 + b];
    }
  };
  fetch(0, tb.az, xc, ac);
  fetch_d(0, dc, rc);
#pragma unroll 2
  for (int k0 = 0; k0 < np; k0 += ZB) {
    double xn[ZB], an[ZB], dn[ZB], rn[ZB], g[ZB];
    const int kn = min(k0 + ZB, np - ZB);
    fetch(kn, tb.az, xn, an);
    fetch_d(kn, dn, rn);
    const double g0 = gv;
    unsigned far = 0;
#pragma unroll
    for (int b = 0; b < ZB; b++) {
      const double t = xc[b] + ac[b] * gv;
      const double q0 = t * rc[b], q1 = fma(fma(-q0, dc[b], t), rc[b], q0);
      gv = fma(fma(-q1, dc[b], t), rc[b], q1);
      far = max(far, ((unsigned)__double2hiint(gv) & 0x7fffffffu) - lo);
      g[b] = gv;
    }
    if (far >= range) {
      gv = g0;
#pragma unroll
      for (int b = 0; b < ZB; b++) {
        gv = (xc[b] + ac[b] * gv) / dc[b];
        g[b] = gv;
      }
    }
#pragma unroll
    for (int b = 0; b < ZB; b++) {
      x[(k0 + b) * S] = g[b];
      xc[b] = xn[b];
      ac[b] = an[b];
      dc[b] = dn[b];
      rc[b] = rn[b];
    }
  }
  // P of the top level is its g: e is 0 there, and v = -0 above it leaves
  // any sum unchanged
  for (int k = nz; k < np; k++) x[k * S] = -0.0;
  double v = -0.0;
  fetch(np - ZB, tb.e, xc, ac);
#pragma unroll 2
  for (int k0 = np - ZB; k0 >= 0; k0 -= ZB) {
    double xn[ZB], an[ZB];
    fetch(max(k0 - ZB, 0), tb.e, xn, an);
#pragma unroll
    for (int b = ZB - 1; b >= 0; b--) {
      v = xc[b] + ac[b] * v;
      x[(k0 + b) * S] = v;
    }
#pragma unroll
    for (int b = 0; b < ZB; b++) {
      xc[b] = xn[b];
      ac[b] = an[b];
    }
  }
}

__global__ void __launch_bounds__(kMgThreads) k_mg_sweep(MgLevel L, const double *__restrict__ az,
                                                         const double *__restrict__ den,
                                                         const double *__restrict__ e, int color) {
  extern __shared__ double hs[];  // [np][kMgCols], then the tables
  const int half = L.nx / 2, ncol = half * L.ny, nx = L.nx, nz = L.nz, np = mg_pad(nz);
  const MgTab tb = mg_tab_at(hs + np * kMgCols, np);
  const int l = threadIdx.x % kMgCols, t = blockIdx.x * kMgCols + l;
  const int tc = min(t, ncol - 1);
  const int j = tc / half + 1, ii = tc - (j - 1) * half;
  const int i = 2 * ii + (((j + color) & 1) ? 1 : 2);
  const long plane = (long)nx * L.ny;
  const long c = (i - 1) + (long)(j - 1) * nx;
  double *P = L.phi;
  {
    const double *R = L.rhs + c;
    const double *W = P + (wrap_lo(i, nx) - 1) + (long)(j - 1) * nx, *E = P + (wrap_hi(i, nx) - 1) + (long)(j - 1) * nx;
    const double *S = P + (i - 1) + (long)(wrap_lo(j, L.ny) - 1) * nx, *N = P + (i - 1) + (long)(wrap_hi(j, L.ny) - 1) * nx;
    // the loads in batches without conditions (levels clamped into the
    // column), so that a batch is in flight together
    constexpr int SK = kMgThreads / kMgCols, NK = 4;
    for (int k0 = threadIdx.x / kMgCols; k0 < np; k0 += SK * NK) {
      double w[NK], ea[NK], so[NK], no[NK], r[NK];
#pragma unroll
      for (int u = 0; u < NK; u++) {
        const long o = (long)min(k0 + u * SK, nz - 1) * plane;
        w[u] = W[o];
        ea[u] = E[o];
        so[u] = S[o];
        no[u] = N[o];
        r[u] = R[o];
      }
#pragma unroll
      for (int u = 0; u < NK; u++) {
        const int k = k0 + u * SK;
        const double h = L.ax * (w[u] + ea[u]) + L.ay * (so[u] + no[u]);
        if (k < np) hs[k * kMgCols + l] = k < nz ? h - r[u] : 1.0;
      }
    }
    mg_tab_fill<kMgThreads>(tb, az, den, e, nz, np);
  }
  __syncthreads();
  if (threadIdx.x < kMgCols) mg_column<kMgCols>(hs + l, tb, nz, np);
  __syncthreads();
  if (t < ncol) {
#pragma unroll 4
    for (int k = threadIdx.x / kMgCols; k < nz; k += kMgThreads / kMgCols) P[c + (long)k * plane] = hs[k * kMgCols + l];
  }
}

// The sweep of columns too tall for LDS, any number of levels: one thread per
// column, the forward values stored in place.  Same operations as
// k_mg_sweep, whose quotients are the divisions' bits.
__global__ void __launch_bounds__(256) k_mg_sweep_tall(MgLevel L, const double *__restrict__ az,
                                                       const double *__restrict__ den, const double *__restrict__ e,
                                                       int color) {
  const int half = L.nx / 2;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= half * L.ny) return;
  const int j = t / half + 1, ii = t - (j - 1) * half;
  const int i = 2 * ii + (((j + color) & 1) ? 1 : 2);
  const int nx = L.nx, nz = L.nz;
  const long plane = (long)nx * L.ny;
  const long c = (i - 1) + (long)(j - 1) * nx;
  const long w = (wrap_lo(i, nx) - 1) + (long)(j - 1) * nx, ea = (wrap_hi(i, nx) - 1) + (long)(j - 1) * nx;
  const long so = (i - 1) + (long)(wrap_lo(j, L.ny) - 1) * nx, no = (i - 1) + (long)(wrap_hi(j, L.ny) - 1) * nx;
  double *P = L.phi;
  const double *R = L.rhs;
  double gv = 0;
#pragma unroll 4
  for (int k = 1; k <= nz; k++) {
    const long o = (long)(k - 1) * plane;
    const double h = L.ax * (P[w + o] + P[ea + o]) + L.ay * (P[so + o] + P[no + o]);
    gv = ((h - R[c + o]) + az[k - 1] * gv) / den[k - 1];
    P[c + o] = gv;
  }
  double x = gv;
#pragma unroll 4
  for (int k = nz - 1; k >= 1; k--) {
    const long o = (long)(k - 1) * plane;
    x = P[c + o] + e[k - 1] * x;
    P[c + o] = x;
  }
}

// Both colours' sweeps twice over, a whole smoothing, in one launch: a block
// owns a tile of kMgTile x kMgTile columns, holds it with a ring of 4 columns
// in LDS and sweeps everything within 3 columns of the tile.  What a sweep
// leaves right shrinks by one ring per colour: after the first it reaches 3
// columns out, after the fourth it is the tile, which the block writes to the
// level's other array (its neighbours still read this one).  Columns of
// colour 0 are written before they are read, so only colour 1 is loaded; with
// PRO the coarse correction is added in that load (see k_mg_prolong).
// The columns of a colour are solved in place: a column's own values are not
// read by its sweep.  (Columns of the outer rings take unset or outdated
// neighbours in; what comes of that stays out of the tile.)
// 128x64 / 64x32 / 16x8 columns of 64 levels: four sweeps and the prolongation
// 45 us in five launches, 50 / 33 / 31 here, of which 10 are loads and stores,
// 5 the sums and 16 the four columns' chains.
constexpr int kMgTile = 4, kMgReg = kMgTile + 8, kMgRegCols = kMgReg * kMgReg;
constexpr int kMgHalf = (kMgTile + 6) * (kMgTile + 6) / 2;  // swept columns of a colour
constexpr int kMgSmoothThreads = 512;
constexpr size_t mg_smooth_lds(int nz) { return (size_t)mg_pad(nz) * (kMgRegCols + 4) * sizeof(double); }
// Where: two blocks in a CU's LDS (nz <= 68) and at most two per CU (512).
// ms a step of the channel, smoothings whole on levels up to 0 / 128 / 512 /
// 2048 tiles: 128x128x32 16.2 / 14.6 / 13.7 / 14.2, 128x64x64 12.2 / 11.7 /
// 11.8 / 11.8, 256x128x64 18.3 / 17.6 / 17.8 / 23.5; with one block per CU
// 128x64x128 19.8 / 19.8 / 22.5 / 22.5.
constexpr long kMgSmoothMaxTiles = 512;
constexpr int kMgMaxNr = 7;
static_assert(2 * mg_smooth_lds(68) <= 160 * 1024 && 2 * mg_smooth_lds(69) > 160 * 1024 &&
                  kMgHalf * 68 <= kMgMaxNr * kMgSmoothThreads,
              "values of a colour per thread at the largest nz");
// NR: right-hand-side values of a colour per thread
template <int NR, bool PRO>
__global__ void __launch_bounds__(kMgSmoothThreads, 4)
    k_mg_smooth(MgLevel L, MgLevel Cs, const double *__restrict__ az, const double *__restrict__ den,
                const double *__restrict__ e) {
  extern __shared__ double hs[];  // [np][kMgRegCols], then the tables
  constexpr int S = kMgRegCols, TH = kMgSmoothThreads;
  const int nx = L.nx, ny = L.ny, nz = L.nz, np = mg_pad(nz), tid = threadIdx.x;
  const MgTab tb = mg_tab_at(hs + np * S, np);
  const int tx = blockIdx.x % (nx / kMgTile), ty = blockIdx.x / (nx / kMgTile);
  const int i0 = tx * kMgTile - 4, j0 = ty * kMgTile - 4;  // level column of the region's column (0, 0)
  const long plane = (long)nx * ny;
  // nx, ny are multiples of 4 and at least 8: one wrap suffices
  const auto wrapi = [&](int i) { return i < 0 ? i + nx : i >= nx ? i - nx : i; };
  const auto wrapj = [&](int j) { return j < 0 ? j + ny : j >= ny ? j - ny : j; };
  // swept column c of a colour: region coordinates
  const auto ycol = [](int c) { return 1 + c / (kMgReg / 2 - 1); };
  const auto xcol = [&](int c, int y, int color) { return 1 + 2 * (c % (kMgReg / 2 - 1)) + ((1 + y + color) & 1); };
  double r[2][NR];
#pragma unroll
  for (int color = 0; color < 2; color++)
#pragma unroll
    for (int u = 0; u < NR; u++) {
      const int q = tid + u * TH, k = min(q / kMgHalf, nz - 1), c = q % kMgHalf, y = ycol(c);
      r[color][u] = L.rhs[wrapi(i0 + xcol(c, y, color)) + (long)wrapj(j0 + y) * nx + k * plane];
    }
  {
    constexpr int NK = 4, H = S / 2;
    for (int q0 = tid; q0 < H * nz; q0 += TH * NK) {
      double v[NK];
#pragma unroll
      for (int u = 0; u < NK; u++) {
        const int q = min(q0 + u * TH, H * nz - 1), k = q / H, c = q % H, y = c / (kMgReg / 2);
        const int i = wrapi(i0 + 2 * (c % (kMgReg / 2)) + ((y + 1) & 1)), j = wrapj(j0 + y);
        v[u] = L.phi[i + (long)j * nx + k * plane];
        if (PRO) {
          const int I = i / 2, J = j / 2, cx = Cs.nx, cy = Cs.ny;
          const int Ix = (i & 1) ? (I + 1 < cx ? I + 1 : 0) : (I > 0 ? I - 1 : cx - 1);
          const int Jy = (j & 1) ? (J + 1 < cy ? J + 1 : 0) : (J > 0 ? J - 1 : cy - 1);
          const double *E = Cs.phi + (long)k * cx * cy;
          const double c00 = E[I + (long)J * cx], c10 = E[Ix + (long)J * cx];
          const double c01 = E[I + (long)Jy * cx], c11 = E[Ix + (long)Jy * cx];
          const double ex0 = 0.75 * c00 + 0.25 * c10, ex1 = 0.75 * c01 + 0.25 * c11;
          v[u] = v[u] + (0.75 * ex0 + 0.25 * ex1);
        }
      }
#pragma unroll
      for (int u = 0; u < NK; u++) {
        const int q = q0 + u * TH, k = q / H, c = q % H, y = c / (kMgReg / 2);
        if (q < H * nz) hs[k * S + y * kMgReg + 2 * (c % (kMgReg / 2)) + ((y + 1) & 1)] = v[u];
      }
    }
    mg_tab_fill<TH>(tb, az, den, e, nz, np);
  }
#pragma unroll 1
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int color = 0; color < 2; color++) {
      __syncthreads();
#pragma unroll
      for (int u = 0; u < NR; u++) {
        const int q = tid + u * TH, k = q / kMgHalf, c = q % kMgHalf, y = ycol(c);
        if (k < np) {
          double *x = hs + k * S + y * kMgReg + xcol(c, y, color);
          const double hv = L.ax * (x[-1] + x[1]) + L.ay * (x[-kMgReg] + x[kMgReg]);
          *x = k < nz ? hv - r[color][u] : 1.0;
        }
      }
      __syncthreads();
      if (tid < kMgHalf) mg_column<S>(hs + ycol(tid) * kMgReg + xcol(tid, ycol(tid), color), tb, nz, np);
    }
  __syncthreads();
  for (int q = tid; q < kMgTile * kMgTile * nz; q += TH) {
    const int k = q / (kMgTile * kMgTile), c = q % (kMgTile * kMgTile), y = 4 + c / kMgTile, x = 4 + c % kMgTile;
    L.phi2[(i0 + x) + (long)(j0 + y) * nx + k * plane] = hs[k * S + y * kMgReg + x];
  }
}

// Maximum |residual| of a level: block maxima (a NaN counts as +inf).
__global__ void __launch_bounds__(256) k_mg_resmax(MgLevel L, const double *__restrict__ az,
                                                   const double *__restrict__ cz, double *__restrict__ partial) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  double v = 0;
  if (t < (long)L.nx * L.ny * L.nz) {
    const int i = (int)(t % L.nx) + 1, j = (int)((t / L.nx) % L.ny) + 1, k = (int)(t / ((long)L.nx * L.ny)) + 1;
    v = fabs(mg_res(L, az, cz, i, j, k));
    if (v != v) v = INFINITY;
  }
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = red[0];
    for (int q = 1; q < 4; q++) m = fmax(m, red[q]);
    partial[blockIdx.x] = m;
  }
}

// Residual of the fine level restricted to the coarse one (coarse P = 0).
__global__ void __launch_bounds__(256) k_mg_restrict(MgLevel F, MgLevel Cs, const double *__restrict__ az,
                                                     const double *__restrict__ cz) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)Cs.nx * Cs.ny * Cs.nz) return;
  const int I = (int)(t % Cs.nx) + 1, J = (int)((t / Cs.nx) % Cs.ny) + 1, k = (int)(t / ((long)Cs.nx * Cs.ny)) + 1;
  const double r1 = mg_res(F, az, cz, 2 * I - 1, 2 * J - 1, k);
  const double r2 = mg_res(F, az, cz, 2 * I, 2 * J - 1, k);
  const double r3 = mg_res(F, az, cz, 2 * I - 1, 2 * J, k);
  const double r4 = mg_res(F, az, cz, 2 * I, 2 * J, k);
  Cs.rhs[t] = ((r1 + r2) + (r3 + r4)) * 0.25;
  Cs.phi[t] = 0.0;
}

// Bilinear (x, y) prolongation of the coarse correction, added to the fine P.
__global__ void __launch_bounds__(256) k_mg_prolong(MgLevel Cs, MgLevel F) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)F.nx * F.ny * F.nz) return;
  const int i = (int)(t % F.nx) + 1, j = (int)((t / F.nx) % F.ny) + 1, k = (int)(t / ((long)F.nx * F.ny)) + 1;
  const int I = (i + 1) / 2, J = (j + 1) / 2;
  const int Ix = (i & 1) ? wrap_lo(I, Cs.nx) : wrap_hi(I, Cs.nx);
  const int Jy = (j & 1) ? wrap_lo(J, Cs.ny) : wrap_hi(J, Cs.ny);
  const double *E = Cs.phi + (long)(k - 1) * Cs.nx * Cs.ny;
  const double c00 = E[(I - 1) + (long)(J - 1) * Cs.nx], c10 = E[(Ix - 1) + (long)(J - 1) * Cs.nx];
  const double c01 = E[(I - 1) + (long)(Jy - 1) * Cs.nx], c11 = E[(Ix - 1) + (long)(Jy - 1) * Cs.nx];
  const double ex0 = 0.75 * c00 + 0.25 * c10, ex1 = 0.75 * c01 + 0.25 * c11;
  F.phi[t] = F.phi[t] + (0.75 * ex0 + 0.25 * ex1);
}

// Exact solve of the coarsest level (P = 0 on entry) by one block: discrete
// Fourier sums in x, then y (twiddles w(q) = (cos 2 pi q/N, -sin 2 pi q/N)),
// a tridiagonal elimination in z per mode (the (0, 0) mode integrated as the
// singular Neumann problem with x_1 = 0), conjugate sums over y, then x.
// The right-hand side, the work arrays Y, X (complex, nx ny nz) and cp (nx ny
// nz, which takes the right-hand side's place) and the tables are held in LDS
// where they fit (SH), else in global memory: the sums and the elimination
// are chains of dependent reads, 8x4x64 100 us from global memory by 256
// threads, 34 us from LDS by 1024.
constexpr int kMgCoarseThreads = 1024;
constexpr size_t mg_coarse_lds(long n, int nx, int ny, int nz) {
  return (size_t)(n * 5 + 2 * (nx + ny) + 2 * nz) * sizeof(double);
}
template <bool SH>
__global__ void __launch_bounds__(SH ? kMgCoarseThreads : 256)
    k_mg_coarse(MgLevel L, MgCoarse C, const double *__restrict__ gaz, const double *__restrict__ gcz,
                const double *__restrict__ dzPr, const double *__restrict__ dzW) {
  extern __shared__ __align__(16) double sm[];
  const int nx = L.nx, ny = L.ny, nz = L.nz;
  const int plane = nx * ny, n = plane * nz;
  double2 *Y = SH ? reinterpret_cast<double2 *>(sm) : C.Y, *X = SH ? Y + n : C.X;
  double *cp = SH ? sm + 4 * (long)n : C.cp;
  double *tab = sm + 5 * (long)n;
  const double *rhs = SH ? cp : L.rhs;
  const double *cx = SH ? tab : C.cx, *sx = SH ? cx + nx : C.sx;
  const double *cy = SH ? sx + nx : C.cy, *sy = SH ? cy + ny : C.sy;
  const double *az = SH ? sy + ny : gaz, *cz = SH ? az + nz : gcz;
  if (SH) {
    for (int q = threadIdx.x; q < n; q += blockDim.x) cp[q] = L.rhs[q];
    for (int q = threadIdx.x; q < nx; q += blockDim.x) {
      tab[q] = C.cx[q];
      tab[nx + q] = C.sx[q];
    }
    for (int q = threadIdx.x; q < ny; q += blockDim.x) {
      tab[2 * nx + q] = C.cy[q];
      tab[2 * nx + ny + q] = C.sy[q];
    }
    for (int q = threadIdx.x; q < nz; q += blockDim.x) {
      tab[2 * (nx + ny) + q] = gaz[q];
      tab[2 * (nx + ny) + nz + q] = gcz[q];
    }
    __syncthreads();
  }
  // tq = (m i) mod nx by steps
  const auto next = [](int tq, int m, int len) { return tq + m >= len ? tq + m - len : tq + m; };
  for (int q = threadIdx.x; q < n; q += blockDim.x) {
    const int row = q / nx, m = q - row * nx;
    double ar = 0, ai = 0;
    for (int i = 0, tq = 0; i < nx; i++, tq = next(tq, m, nx)) {
      const double r = rhs[i + row * nx];
      const double pr = r * cx[tq] - 0.0 * sx[tq], pi = r * sx[tq] + 0.0 * cx[tq];
      ar = ar + pr;
      ai = ai + pi;
    }
    Y[q] = make_double2(ar, ai);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < n; q += blockDim.x) {
    const int row = q / nx, m = q - row * nx, k = row / ny, nn = row - k * ny;
    double ar = 0, ai = 0;
    for (int j = 0, tq = 0; j < ny; j++, tq = next(tq, nn, ny)) {
      const double2 y = Y[m + j * nx + k * plane];
      const double pr = y.x * cy[tq] - y.y * sy[tq], pi = y.x * sy[tq] + y.y * cy[tq];
      ar = ar + pr;
      ai = ai + pi;
    }
    X[q] = make_double2(ar, ai);
  }
  __syncthreads();
  for (int mode = threadIdx.x; mode < plane; mode += blockDim.x) {
    const int m = mode % nx, nn = mode / nx;
    double2 *col = X + mode;
    if (m == 0 && nn == 0) {
      double Gr = 0, Gi = 0, xr = 0, xi = 0;
      for (int k = 1; k <= nz; k++) {
        const double2 d = col[(k - 1) * plane];
        col[(k - 1) * plane] = make_double2(xr, xi);
        if (k < nz) {
          Gr = Gr + d.x * dzPr[k];
          Gi = Gi + d.y * dzPr[k];
          xr = xr + Gr * dzW[k];
          xi = xi + Gi * dzW[k];
        }
      }
      continue;
    }
    const double lam = C.lam[mode];  // host table (the host's sin)
    double cprev = 0, dr = 0, di = 0;
    double2 d = col[0];
    double a = az[0], c = cz[0];
    for (int k = 0; k < nz; k++) {
      // the next level's inputs before this level's chain
      const int kn = min(k + 1, nz - 1);
      const double2 dn = col[kn * plane];
      const double an = az[kn], cn = cz[kn];
      const double b = (lam - a) - c;
      const double den = b - a * cprev;
      const double cpk = c / den;
      dr = (d.x - a * dr) / den;
      di = (d.y - a * di) / den;
      cp[mode + k * plane] = cpk;
      col[k * plane] = make_double2(dr, di);
      cprev = cpk;
      d = dn;
      a = an;
      c = cn;
    }
    double xr = dr, xi = di;
    for (int k = nz - 2; k >= 0; k--) {
      const double2 dp = col[k * plane];
      const double cpk = cp[mode + k * plane];
      xr = dp.x - cpk * xr;
      xi = dp.y - cpk * xi;
      col[k * plane] = make_double2(xr, xi);
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < n; q += blockDim.x) {
    const int row = q / nx, m = q - row * nx, k = row / ny, j = row - k * ny;
    double ar = 0, ai = 0;
    for (int nn = 0, tq = 0; nn < ny; nn++, tq = next(tq, j, ny)) {
      const double2 x = X[m + nn * nx + k * plane];
      const double wr = cy[tq], wi = -sy[tq];
      const double pr = x.x * wr - x.y * wi, pi = x.x * wi + x.y * wr;
      ar = ar + pr;
      ai = ai + pi;
    }
    Y[q] = make_double2(ar, ai);
  }
  __syncthreads();
  const double scale = 1.0 / (double)plane;
  for (int q = threadIdx.x; q < n; q += blockDim.x) {
    const int row = q / nx, i = q - row * nx;
    double acc = 0;
    for (int m = 0, tq = 0; m < nx; m++, tq = next(tq, i, nx)) {
      const double2 y = Y[m + row * nx];
      const double wr = cx[tq], wi = -sx[tq];
      acc = acc + (y.x * wr - y.y * wi);
    }
    L.phi[q] = acc * scale;
  }
}

template <typename T>
void launch_mg_rhs(const Geo &g, const T *U, const T *V, const T *W, const double *Q, double dt2_rec, double *rhs0,
                   double *RHS, hipStream_t st) {
  const long n = (long)g.nx * g.ny * g.nz;
  hipLaunchKernelGGL(k_mg_rhs<T>, dim3(nblk(n, 256)), dim3(256), 0, st, g, U, V, W, Q, dt2_rec, rhs0, RHS);
}

void launch_mg_to_phi(const Geo &g, const double *phi0, double *Phi, hipStream_t st) {
  const long n = (long)g.nx * g.ny * g.nz;
  hipLaunchKernelGGL(k_mg_to_phi, dim3(nblk(n, 256)), dim3(256), 0, st, g, phi0, Phi);
}

void launch_mg_zero(double *a, long n, hipStream_t st) {
  hipLaunchKernelGGL(k_mg_zero, dim3(nblk(n, 256)), dim3(256), 0, st, a, n);
}

void launch_mg_sweep(const MgLevel &L, const double *az, const double *den, const double *e, int color,
                     hipStream_t st) {
  const long cols = (long)(L.nx / 2) * L.ny;
  const size_t sh = mg_sweep_lds(L.nz);
  if (sh > 160 * 1024) {
    hipLaunchKernelGGL(k_mg_sweep_tall, dim3(nblk(cols, 256)), dim3(256), 0, st, L, az, den, e, color);
    return;
  }
  if (sh > 65536) (void)lds_limit_raise((const void *)k_mg_sweep, sh);
  hipLaunchKernelGGL(k_mg_sweep, dim3(nblk(cols, kMgCols)), dim3(kMgThreads), sh, st, L, az, den, e, color);
}

// A smoothing of level L from phi to phi2; coarse: the level whose correction
// is added first (or null).
bool mg_smooth_wanted(const MgLevel &L) {
  return 2 * mg_smooth_lds(L.nz) <= 160 * 1024 && (long)L.nx * L.ny / (kMgTile * kMgTile) <= kMgSmoothMaxTiles;
}

void launch_mg_smooth(const MgLevel &L, const MgLevel *coarse, const double *az, const double *den, const double *e,
                      hipStream_t st) {
  const size_t sh = mg_smooth_lds(L.nz);
  const MgLevel Cs = coarse ? *coarse : MgLevel{};
  const auto run = [&](auto nr, auto pro) {
    constexpr int NR = decltype(nr)::value;
    constexpr bool PRO = decltype(pro)::value;
    if (sh > 65536) (void)lds_limit_raise((const void *)k_mg_smooth<NR, PRO>, sh);
    hipLaunchKernelGGL((k_mg_smooth<NR, PRO>), dim3(L.nx * L.ny / (kMgTile * kMgTile)), dim3(kMgSmoothThreads), sh, st,
                       L, Cs, az, den, e);
  };
  // values of a colour: swept columns times padded levels, over the threads
  const int need = (kMgHalf * mg_pad(L.nz) + kMgSmoothThreads - 1) / kMgSmoothThreads;
  const auto pro = [&](auto nr) { coarse ? run(nr, std::true_type{}) : run(nr, std::false_type{}); };
  if (need <= 4)
    pro(std::integral_constant<int, 4>{});
  else
    pro(std::integral_constant<int, kMgMaxNr>{});
}

int mg_resmax_blocks(const MgLevel &L) { return (int)nblk((long)L.nx * L.ny * L.nz, 256); }

void launch_mg_resmax(const MgLevel &L, const double *az, const double *cz, double *partial, hipStream_t st) {
  hipLaunchKernelGGL(k_mg_resmax, dim3(mg_resmax_blocks(L)), dim3(256), 0, st, L, az, cz, partial);
}

void launch_mg_restrict(const MgLevel &F, const MgLevel &Cs, const double *az, const double *cz, hipStream_t st) {
  const long n = (long)Cs.nx * Cs.ny * Cs.nz;
  hipLaunchKernelGGL(k_mg_restrict, dim3(nblk(n, 256)), dim3(256), 0, st, F, Cs, az, cz);
}

void launch_mg_prolong(const MgLevel &Cs, const MgLevel &F, hipStream_t st) {
  const long n = (long)F.nx * F.ny * F.nz;
  hipLaunchKernelGGL(k_mg_prolong, dim3(nblk(n, 256)), dim3(256), 0, st, Cs, F);
}

void launch_mg_coarse(const MgLevel &L, const MgCoarse &C, const double *az, const double *cz, const double *dzPr,
                      const double *dzW, hipStream_t st) {
  const size_t sh = mg_coarse_lds((long)L.nx * L.ny * L.nz, L.nx, L.ny, L.nz);
  if (sh <= 160 * 1024) {
    if (sh > 65536) (void)lds_limit_raise((const void *)k_mg_coarse<true>, sh);
    hipLaunchKernelGGL(k_mg_coarse<true>, dim3(1), dim3(kMgCoarseThreads), sh, st, L, C, az, cz, dzPr, dzW);
  } else {
    hipLaunchKernelGGL(k_mg_coarse<false>, dim3(1), dim3(256), 0, st, L, C, az, cz, dzPr, dzW);
  }
}

template void launch_mg_rhs<double>(const Geo &, const double *, const double *, const double *, const double *,
                                    double, double *, double *, hipStream_t);
template void launch_mg_rhs<float>(const Geo &, const float *, const float *, const float *, const double *, double,
                                   double *, double *, hipStream_t);

}  // namespace elmm
