// k_fft_mr.hip - transform passes of the spectral Poisson solve for line
// lengths n = 2^a 3^b that are not powers of two (the batched-ensemble grids
// such as 96, 144 or 192 cells).
//
// The lines are transformed in LDS by a self-sorting (Stockham) mixed-radix
// FFT: radix-3 stages first, then radix-2 stages; stage s with radix r and
// span Ns (the product of the earlier radices) maps element j + q n/r
// (q < r) of the source, multiplied by w^(k q n/(Ns r)) with k = j mod Ns and
// w = exp(-2 pi i/n) (conjugate for the inverse), through an r-point DFT to
// element (j div Ns) Ns r + k + q Ns of the destination.  Every operation
// is stated so the oracle can repeat it bit for bit: complex products
// (a.x w.x - a.y w.y, a.x w.y + a.y w.x), no product when k q = 0, and the
// 3-point DFT  s = b + c, d = b - c, y0 = a + s, m = a - s/2,
// t = (s3 d.y, -s3 d.x) (forward) or (-s3 d.y, s3 d.x) (inverse) with
// s3 = sin(pi/3), y1 = m + t, y2 = m - t.  Which stages share a pass over LDS
// changes none of that.
// The passes have the same inputs and outputs as the power-of-two kernels
// in k_pressure.hip (divergence -> x FFT, y FFT, inverse y, inverse x ->
// Phi), with rows mapped by division since ny need not be a power of two.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace elmm {

namespace {

inline unsigned nblk(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

__device__ inline double2 mk2(double x, double y) { return make_double2(x, y); }
__device__ inline float2 mk2(float x, float y) { return make_float2(x, y); }
template <typename V>
__device__ inline V cmul(V a, V b) {
  return mk2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Bound by latency at the batched grids (144x144x64: 640 blocks of the y pass,
// all resident at once): the loads and stores alone take 2/3 of each pass.
// So: loads in batches, no division per element, and the stages in groups
// that a thread runs in registers, 144 = 9 4 4 instead of 3 3 2 2 2 2, which
// divides the LDS round trips and barriers by two.  Groups up to 16 cost
// 142 registers and with them half of the waves.  144x144x64 in FP64, us,
// one stage per barrier with the lines contiguous -> here: forward x 26.8 ->
// 20.6, y 20.4 -> 12.0 (mean of both directions), inverse x 22.8 -> 14.8;
// with 128 threads or x blocks of 512 or 1536 elements 10 to 60 % slower.
constexpr int kMrThreads = 256;
constexpr int kMrElemsX = 1024;  // line elements per block and buffer of the x passes
// y pass: 8 modes of a row are one or two whole cache lines; 144-point lines
// with 4 modes instead take 14.7 us
constexpr int kMrElemsY = 2048, kMrColsY = 8;
constexpr int kMrLinesX = 64;
constexpr int kMrMaxRadix = 9;
constexpr int kMrMaxStages = 12;
constexpr int kMrBatch = 4;  // global loads of a thread in flight (per array)

// q / d for q * d < 2^32, d > 1: m = floor(2^32 / d) + 1 exceeds 2^32 / d by
// at most 1, so the product is high by less than q / 2^32 < 1 / d.
struct MrDiv {
  unsigned d, m;
};
__device__ __host__ inline MrDiv mr_div(unsigned d) {
  return MrDiv{d, d > 1 ? (unsigned)(0x100000000ull / d + 1) : 0};
}
__device__ inline int mr_quot(int q, MrDiv d) { return d.d > 1 ? (int)__umulhi((unsigned)q, d.m) : q; }

// Groups of consecutive stages that one thread runs in registers: `radix` is
// the product of the group's radices, ns its span, nb = n / radix its
// butterflies per line, t0 = n / (ns radix) the twiddle stride of its last
// stage.
struct MrStage {
  int radix, nb, t0;
  MrDiv ns;
};
struct MrPlan {
  int n, nst, lines, llog, pitch;  // line l, element j at j * pitch + l
  MrDiv dn, dny, dm;               // by n, ny and M
  MrStage st[kMrMaxStages];
};

template <typename R>
__device__ inline R sin60() {
  return (R)0.86602540378443864676;
}

// Stage of radix RAD and span NS within a group of N elements held in v (the
// group's own Stockham order: the element p of the group is element
// j0 + p nb of the line before the group and (j0 div ns) ns N + k + p ns
// after it).  k: the butterfly's position within the group's span.
template <typename R, int N, int RAD, int NS, bool FIRST, bool INV>
__device__ inline void mr_micro(C2<R> *v, int k, int t0, const C2<R> *tw, int ns) {
  using V = C2<R>;
  V o[N];
  constexpr int nb = N / RAD, tmul = N / (NS * RAD);
#pragma unroll
  for (int j = 0; j < nb; j++) {
    const int kl = j % NS;
    V x[RAD];
#pragma unroll
    for (int r = 0; r < RAD; r++) {
      x[r] = v[j + r * nb];
      if (r > 0 && (kl > 0 || !FIRST)) {
        const int kk = k + kl * ns;
        V w = tw[kk * r * (t0 * tmul)];
        if (INV) w.y = -w.y;
        const V m = cmul(x[r], w);
        if (kl > 0 || kk > 0) x[r] = m;
      }
    }
    const int d = (j / NS) * NS * RAD + kl;
    if (RAD == 2) {
      o[d] = mk2(x[0].x + x[1].x, x[0].y + x[1].y);
      o[d + NS] = mk2(x[0].x - x[1].x, x[0].y - x[1].y);
    } else {
      const R s3 = sin60<R>(), h = (R)0.5;
      const V sm = mk2(x[1].x + x[2 % RAD].x, x[1].y + x[2 % RAD].y);
      const V df = mk2(x[1].x - x[2 % RAD].x, x[1].y - x[2 % RAD].y);
      const V m = mk2(x[0].x - h * sm.x, x[0].y - h * sm.y);
      const V t = INV ? mk2(-(s3 * df.y), s3 * df.x) : mk2(s3 * df.y, -(s3 * df.x));
      o[d] = mk2(x[0].x + sm.x, x[0].y + sm.y);
      o[d + NS] = mk2(m.x + t.x, m.y + t.y);
      o[d + 2 % RAD * NS] = mk2(m.x - t.x, m.y - t.y);
    }
  }
#pragma unroll
  for (int p = 0; p < N; p++) v[p] = o[p];
}

template <typename R, int N, int NS, bool FIRST, bool INV>
__device__ inline void mr_micros(C2<R> *v, int k, int t0, const C2<R> *tw, int ns) {
  if constexpr (NS < N) {
    constexpr int RAD = (N / NS) % 3 == 0 ? 3 : 2;
    mr_micro<R, N, RAD, NS, FIRST, INV>(v, k, t0, tw, ns);
    mr_micros<R, N, NS * RAD, FIRST, INV>(v, k, t0, tw, ns);
  }
}

template <typename R, int N, bool FIRST, bool INV>
__device__ inline void mr_group(const C2<R> *src, C2<R> *dst, const MrPlan &mp, const MrStage &s, const C2<R> *tw) {
  const int ns = FIRST ? 1 : (int)s.ns.d;
  for (int q = threadIdx.x; q < s.nb << mp.llog; q += kMrThreads) {
    const int l = q & (mp.lines - 1), j = q >> mp.llog;
    const int jq = FIRST ? j : mr_quot(j, s.ns), k = FIRST ? 0 : j - jq * ns;
    C2<R> v[N];
#pragma unroll
    for (int p = 0; p < N; p++) v[p] = src[(j + p * s.nb) * mp.pitch + l];
    mr_micros<R, N, 1, FIRST, INV>(v, k, s.t0, tw, ns);
    const int base = jq * ns * N + k;
#pragma unroll
    for (int p = 0; p < N; p++) dst[(base + p * ns) * mp.pitch + l] = v[p];
  }
}

template <typename R, bool FIRST, bool INV>
__device__ inline void mr_stage(const C2<R> *src, C2<R> *dst, const MrPlan &mp, const MrStage &s, const C2<R> *tw) {
  switch (s.radix) {
    case 2: mr_group<R, 2, FIRST, INV>(src, dst, mp, s, tw); break;
    case 3: mr_group<R, 3, FIRST, INV>(src, dst, mp, s, tw); break;
    case 4: mr_group<R, 4, FIRST, INV>(src, dst, mp, s, tw); break;
    case 6: mr_group<R, 6, FIRST, INV>(src, dst, mp, s, tw); break;
    case 8: mr_group<R, 8, FIRST, INV>(src, dst, mp, s, tw); break;
    case 9: mr_group<R, 9, FIRST, INV>(src, dst, mp, s, tw); break;
  }
}

// Transforms the block's lines held in a (natural order); returns the buffer
// (a or b) that holds the result.
template <typename R, bool INV>
__device__ inline C2<R> *mr_fft(C2<R> *a, C2<R> *b, const MrPlan &mp, const C2<R> *tw) {
  for (int s = 0; s < mp.nst; s++) {
    __syncthreads();
    if (s == 0)
      mr_stage<R, true, INV>(a, b, mp, mp.st[0], tw);
    else
      mr_stage<R, false, INV>(a, b, mp, mp.st[s], tw);
    C2<R> *t = a;
    a = b;
    b = t;
  }
  __syncthreads();
  return a;
}

template <typename R>
__device__ inline void mr_twiddles(C2<R> *dst, const C2<R> *__restrict__ src, int n) {
  for (int t = threadIdx.x; t < n; t += kMrThreads) dst[t] = src[t];
}

// The groups of n's stages: as few as products up to kMrMaxRadix allow, and
// of those the split with the smallest largest product.
MrPlan mr_plan(int n, int lines, bool odd_pitch, int ny, int M) {
  MrPlan mp{};
  mp.n = n;
  mp.lines = lines;
  while ((1 << mp.llog) < lines) mp.llog++;
  mp.pitch = odd_pitch ? lines | 1 : lines;
  mp.dn = mr_div(n);
  mp.dny = mr_div(ny);
  mp.dm = mr_div(M);
  int rad[32], nr = 0;
  for (int rest = n; rest > 1; rest /= rad[nr - 1]) rad[nr++] = rest % 3 == 0 ? 3 : 2;
  int cost[33], from[33];
  cost[0] = 0;
  for (int e = 1; e <= nr; e++) {
    cost[e] = 1 << 30;
    int prod = 1;
    for (int b = e - 1; b >= 0; b--) {
      prod *= rad[b];
      if (prod > kMrMaxRadix) break;
      const int c = std::max(cost[b] & 63, prod) + (cost[b] & ~63) + 64;  // groups, then the largest product
      if (c < cost[e]) {
        cost[e] = c;
        from[e] = b;
      }
    }
  }
  int cut[33], nc = 0;
  for (int e = nr; e > 0; e = from[e]) cut[nc++] = e;
  int ns = 1;
  for (int c = nc - 1, b = 0; c >= 0; b = cut[c--]) {
    int prod = 1;
    for (int i = b; i < cut[c]; i++) prod *= rad[i];
    mp.st[mp.nst++] = MrStage{prod, n / prod, n / (ns * prod), mr_div(ns)};
    ns *= prod;
  }
  return mp;
}

}  // namespace

// Pass 1 (or a refinement sweep's first pass): right-hand side of `rows`
// (j, k) rows per block, x FFT, modes 0..M-1 to the spectral array.
// mode: kMrDiv (divergence of U, V, W, minus Q where qmask says so, over
// coef; stored to rhs_out when given), kMrIn (rhs_in), kMrResid (rhs_in - A
// phi).
enum { kMrDiv = 0, kMrIn = 1, kMrResid = 2 };

template <typename T, typename R, int MODE>
__global__ void __launch_bounds__(kMrThreads)
    k_fft_x_fwd_mr(Geo g, PoissonPlan<R> pp, MrPlan mp, const T *__restrict__ U, const T *__restrict__ V,
                   const T *__restrict__ W, const double *__restrict__ Q, const uint32_t *__restrict__ qmask,
                   const double *__restrict__ rhs_in, const double *__restrict__ phi, double dt2_rec,
                   double *__restrict__ rhs_out) {
  using C = C2<R>;
  extern __shared__ __align__(16) unsigned char sh_raw[];
  const int n = mp.n;
  C *tw = reinterpret_cast<C *>(sh_raw);
  C *a = tw + n, *b = a + mp.pitch * n;
  mr_twiddles<R>(tw, pp.twx, n);
  const int nrows = pp.ny * pp.nz, row0 = blockIdx.x * mp.lines;
  const int nl = min(mp.lines, nrows - row0), total = nl * n;
  const int kb = row0 / pp.ny, jb = row0 - kb * pp.ny;
  for (int e0 = threadIdx.x; e0 < total; e0 += kMrThreads * kMrBatch) {
    double r[kMrBatch];
    int at[kMrBatch];
#pragma unroll
    for (int c = 0; c < kMrBatch; c++) {
      const int e = min(e0 + c * kMrThreads, total - 1);
      const int l = mr_quot(e, mp.dn), i = e - l * n;
      const int kk = mr_quot(jb + l, mp.dny);
      const int j = jb + l - kk * pp.ny + 1, k = kb + kk + 1;
      const long p = gix(g, i + 1, j, k);
      at[c] = i * mp.pitch + l;
      if (MODE == kMrResid) {
        const double rx = 1 / (g.dxmin * g.dxmin), ry = 1 / (g.dymin * g.dymin);
        const double ph = phi[p];
        const double pw = phi[i + 1 > 1 ? p - 1 : p - 1 + g.nx], pe = phi[i + 1 < g.nx ? p + 1 : p + 1 - g.nx];
        const double ps = phi[j > 1 ? p - g.sy : p - g.sy + (long)g.ny * g.sy];
        const double pn = phi[j < g.ny ? p + g.sy : p + g.sy - (long)g.ny * g.sy];
        double s = ((pw - ph) + (pe - ph)) * rx + ((ps - ph) + (pn - ph)) * ry;
        if (k > 1) s = s + pp.az[k - 1] * (phi[p - g.sz] - ph);
        if (k < g.nz) s = s + pp.cz[k - 1] * (phi[p + g.sz] - ph);
        r[c] = rhs_in[p] - s;
      } else if (MODE == kMrIn) {
        r[c] = rhs_in[p];
      } else {
        // U(0) and V(0) by index wrap, W = 0 on the walls, as in k_fft_x_fwd
        const double du = (double)U[p] - (double)U[i > 0 ? p - 1 : p - 1 + g.nx];
        const double dv = (double)V[p] - (double)V[j > 1 ? p - g.sy : p - g.sy + (long)g.ny * g.sy];
        const double wt = (double)W[p], wb = (double)W[p - g.sz];
        const double dw = (k < g.nz ? wt : 0.0) - (k > 1 ? wb : 0.0);
        r[c] = div_rn(du, g.dxmin, g.rdx) + div_rn(dv, g.dymin, g.rdy) +
               (g.variable_z ? dw / g.dzPr[k] : div_rn(dw, g.dzmin, g.rdz));
      }
    }
    if (MODE == kMrDiv) {
#pragma unroll
      for (int c = 0; c < kMrBatch; c++) {
        const int e = e0 + c * kMrThreads;
        if (e < total) {
          const int l = mr_quot(e, mp.dn), i = e - l * n;
          const int kk = mr_quot(jb + l, mp.dny);
          const long p = gix(g, i + 1, jb + l - kk * pp.ny + 1, kb + kk + 1);
          if (Q && ((qmask[row0 + l] >> (i >> 6)) & 1u)) r[c] = r[c] - Q[p];
          r[c] = r[c] * dt2_rec;
          if (rhs_out) rhs_out[p] = r[c];
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kMrBatch; c++)
      if (e0 + c * kMrThreads < total) a[at[c]] = mk2((R)r[c], (R)0);
  }
  const C *res = mr_fft<R, false>(a, b, mp, tw);
  for (int e = threadIdx.x; e < nl * pp.M; e += kMrThreads) {
    const int l = mr_quot(e, mp.dm), m = e - l * pp.M;
    pp.X[(long)(row0 + l) * pp.Mp + m] = res[m * mp.pitch + l];
  }
}

// Passes 2 and 4: y FFT of `lines` consecutive x-modes of one z-plane.
template <typename R, bool INV>
__global__ void __launch_bounds__(kMrThreads) k_fft_y_mr(PoissonPlan<R> pp, MrPlan mp) {
  using C = C2<R>;
  extern __shared__ __align__(16) unsigned char sh_raw[];
  const int n = mp.n, cols = mp.lines;
  C *tw = reinterpret_cast<C *>(sh_raw);
  C *a = tw + n, *b = a + cols * n;
  mr_twiddles<R>(tw, pp.twy, n);
  const int m0 = blockIdx.x * cols, k = blockIdx.y, total = cols * n;
  C *X = pp.X + (long)k * n * pp.Mp;
  // consecutive threads: consecutive modes of one row; columns past the last
  // mode hold it again and are not stored
  for (int e0 = threadIdx.x; e0 < total; e0 += kMrThreads * 2 * kMrBatch) {
    C v[2 * kMrBatch];
#pragma unroll
    for (int c = 0; c < 2 * kMrBatch; c++) {
      const int e = min(e0 + c * kMrThreads, total - 1);
      v[c] = X[(long)(e >> mp.llog) * pp.Mp + min(m0 + (e & (cols - 1)), pp.M - 1)];
    }
#pragma unroll
    for (int c = 0; c < 2 * kMrBatch; c++)
      if (e0 + c * kMrThreads < total) a[e0 + c * kMrThreads] = v[c];
  }
  const C *res = mr_fft<R, INV>(a, b, mp, tw);
  for (int e = threadIdx.x; e < total; e += kMrThreads) {
    const int m = m0 + (e & (cols - 1));
    if (m < pp.M) X[(long)(e >> mp.llog) * pp.Mp + m] = res[e];
  }
}

// Pass 5: inverse x FFT of the half spectrum (Hermitian fill), real part
// scaled by 1/(nx ny) to Phi (added with accumulate).
template <typename R>
__global__ void __launch_bounds__(kMrThreads)
    k_fft_x_inv_mr(Geo g, PoissonPlan<R> pp, MrPlan mp, double *__restrict__ Phi, int accumulate) {
  using C = C2<R>;
  extern __shared__ __align__(16) unsigned char sh_raw[];
  const int n = mp.n;
  C *tw = reinterpret_cast<C *>(sh_raw);
  C *a = tw + n, *b = a + mp.pitch * n;
  mr_twiddles<R>(tw, pp.twx, n);
  const int nrows = pp.ny * pp.nz, row0 = blockIdx.x * mp.lines, M = pp.M;
  const int nl = min(mp.lines, nrows - row0), total = nl * M;
  for (int e0 = threadIdx.x; e0 < total; e0 += kMrThreads * kMrBatch) {
    C v[kMrBatch];
#pragma unroll
    for (int c = 0; c < kMrBatch; c++) {
      const int e = min(e0 + c * kMrThreads, total - 1);
      const int l = mr_quot(e, mp.dm), m = e - l * M;
      v[c] = pp.X[(long)(row0 + l) * pp.Mp + m];
    }
#pragma unroll
    for (int c = 0; c < kMrBatch; c++) {
      const int e = e0 + c * kMrThreads;
      if (e < total) {
        const int l = mr_quot(e, mp.dm), m = e - l * M;
        a[m * mp.pitch + l] = v[c];
        if (m > 0 && n - m >= M) a[(n - m) * mp.pitch + l] = mk2(v[c].x, -v[c].y);
      }
    }
  }
  const C *res = mr_fft<R, true>(a, b, mp, tw);
  const R scale = (R)1.0 / ((R)n * pp.ny);
  const int kb = row0 / pp.ny, jb = row0 - kb * pp.ny;
  for (int e = threadIdx.x; e < nl * n; e += kMrThreads) {
    const int l = mr_quot(e, mp.dn), i = e - l * n;
    const int kk = mr_quot(jb + l, mp.dny);
    const long q = gix(g, i + 1, jb + l - kk * pp.ny + 1, kb + kk + 1);
    const double val = (double)(res[i * mp.pitch + l].x * scale);
    Phi[q] = accumulate ? Phi[q] + val : val;
  }
}

// Lines per block: the largest power of two within both limits, at least 1.
static int mr_lines(int n, int most, int elems) {
  int l = 1;
  while (2 * l <= most && 2 * l * n <= elems) l *= 2;
  return l;
}

template <typename R>
static size_t mr_lds(const MrPlan &mp) {
  return ((size_t)mp.n + 2 * (size_t)mp.pitch * mp.n) * sizeof(C2<R>);
}

template <typename T, typename R>
void launch_fft_x_fwd_mr(const Geo &g, const PoissonPlan<R> &pp, const T *U, const T *V, const T *W, const double *Q,
                         const uint32_t *qmask, const double *rhs, const double *phi, double dt2_rec,
                         double *rhs_out, hipStream_t st) {
  const MrPlan mp = mr_plan(pp.nx, mr_lines(pp.nx, kMrLinesX, kMrElemsX), true, pp.ny, pp.M);
  const dim3 gr(nblk((long)pp.ny * pp.nz, mp.lines)), bl(kMrThreads);
  const size_t sh = mr_lds<R>(mp);
  const auto run = [&](auto mode) {
    constexpr int MODE = decltype(mode)::value;
    if (sh > 65536) (void)lds_limit_raise((const void *)k_fft_x_fwd_mr<T, R, MODE>, sh);
    hipLaunchKernelGGL((k_fft_x_fwd_mr<T, R, MODE>), gr, bl, sh, st, g, pp, mp, U, V, W, Q, qmask, rhs, phi, dt2_rec,
                       rhs_out);
  };
  if (phi)
    run(std::integral_constant<int, kMrResid>{});
  else if (rhs)
    run(std::integral_constant<int, kMrIn>{});
  else
    run(std::integral_constant<int, kMrDiv>{});
}

template <typename R>
void launch_fft_y_mr(const PoissonPlan<R> &pp, int inverse, hipStream_t st) {
  const MrPlan mp = mr_plan(pp.ny, mr_lines(pp.ny, kMrColsY, kMrElemsY), false, pp.ny, pp.M);
  const dim3 gr(nblk(pp.M, mp.lines), pp.nz), bl(kMrThreads);
  const size_t sh = mr_lds<R>(mp);
  if (inverse) {
    if (sh > 65536) (void)lds_limit_raise((const void *)k_fft_y_mr<R, true>, sh);
    hipLaunchKernelGGL((k_fft_y_mr<R, true>), gr, bl, sh, st, pp, mp);
  } else {
    if (sh > 65536) (void)lds_limit_raise((const void *)k_fft_y_mr<R, false>, sh);
    hipLaunchKernelGGL((k_fft_y_mr<R, false>), gr, bl, sh, st, pp, mp);
  }
}

template <typename R>
void launch_fft_x_inv_mr(const Geo &g, const PoissonPlan<R> &pp, double *Phi, int accumulate, hipStream_t st) {
  const MrPlan mp = mr_plan(pp.nx, mr_lines(pp.nx, kMrLinesX, kMrElemsX), true, pp.ny, pp.M);
  const size_t sh = mr_lds<R>(mp);
  if (sh > 65536) (void)lds_limit_raise((const void *)k_fft_x_inv_mr<R>, sh);
  hipLaunchKernelGGL((k_fft_x_inv_mr<R>), dim3(nblk((long)pp.ny * pp.nz, mp.lines)), dim3(kMrThreads), sh, st, g, pp,
                     mp, Phi, accumulate);
}

#define ELMM_INST_MR_R(R)                                                                                          \
  template void launch_fft_y_mr<R>(const PoissonPlan<R> &, int, hipStream_t);                                     \
  template void launch_fft_x_inv_mr<R>(const Geo &, const PoissonPlan<R> &, double *, int, hipStream_t);
ELMM_INST_MR_R(double)
ELMM_INST_MR_R(float)
#define ELMM_INST_MR_TR(T, R)                                                                                      \
  template void launch_fft_x_fwd_mr<T, R>(const Geo &, const PoissonPlan<R> &, const T *, const T *, const T *,     \
                                          const double *, const uint32_t *, const double *, const double *, double,  \
                                          double *, hipStream_t);
ELMM_INST_MR_TR(double, double)
ELMM_INST_MR_TR(float, double)
ELMM_INST_MR_TR(float, float)

}  // namespace elmm
