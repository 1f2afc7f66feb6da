// FP64 construction of every spectral table on the GPU.
//
//   kx      = 2 pi fftfreq(Nx, dx)                     (transformer.py:38)
//   kr_m    = j_{m,k} / R_period, k = 1..Nr-1, m = 0..M+1 (transformer.py:40-45)
//             Bessel roots: McMahon's asymptotic start, then Newton on J_m.
//   DHT_inv = J_m(r_i kr_{m,k}), r_i = Rgrid[1:]      (transformer.py:77-82)
//   DHT     = DHT_inv^{-1} (blocked Gauss-Jordan, partial pivoting; the reference's
//             pinv equals the inverse for these full-rank matrices)
//   dDHT+-  = DHT @ [kr_{m+-1}/2 J_m(r_i kr_{m+-1,k})] (transformer.py:89-92)
//   w, Poisson 1/w^2, smoothing filter                 (transformer.py:47-57)
//   cos(w dt), w sin(w dt), 1/w^2                      (solver.py:41-52)
//   phase exp(-+ i kx Xmin)                            (transformer_generic.cl:28-55)
//   damping profile                                    (solver_methods_cl.py:32-41)
//   FFT twiddles exp(-2 pi i t / Nx)
#include "gemm.h"

#define PI_D 3.14159265358979323846

// J_n(x), n >= 0, x >= 0: power series below x = 2, forward recurrence from
// J_0, J_1 above (stable there for the small orders used here).
__device__ double bessel_jn(int n, double x) {
  if (x < 2.0) {
    double h = 0.5 * x, h2 = h * h;
    double t = 1.0;
    for (int k = 1; k <= n; k++) t *= h / (double)k;
    double s = t;
    for (int k = 1; k < 40; k++) {
      t *= -h2 / ((double)k * (double)(k + n));
      s += t;
      if (fabs(t) < 1e-18 * fabs(s)) break;
    }
    return s;
  }
  double j0v = j0(x);
  if (n == 0) return j0v;
  double j1v = j1(x);
  for (int i = 1; i < n; i++) {
    double j2 = (2.0 * i) / x * j1v - j0v;
    j0v = j1v;
    j1v = j2;
  }
  return j1v;
}

// k-th positive root (k >= 1) of J_m.
__device__ double bessel_root(int m, int k) {
  double mu = 4.0 * m * m;
  double b = (k + 0.5 * m - 0.25) * PI_D;
  double e = 8.0 * b;
  double x = b - (mu - 1) / e - 4 * (mu - 1) * (7 * mu - 31) / (3 * e * e * e) -
             32 * (mu - 1) * (83 * mu * mu - 982 * mu + 3779) / (15 * e * e * e * e * e);
  // 50 steps unless a correction falls below 1e-16 x.  Most roots do not get
  // there (it is less than an ulp): they come to stand or to alternate
  // between two values.  Then the value that step 50 would leave is known.
  double x1 = -1.0, x2 = -1.0;  // one and two steps before
  for (int it = 0; it < 50; it++) {
    double f = bessel_jn(m, x);
    double fp = (m == 0) ? -bessel_jn(1, x) : (bessel_jn(m - 1, x) - (double)m / x * f);
    double dx = f / fp;
    x2 = x1;
    x1 = x;
    x -= dx;
    if (fabs(dx) < 1e-16 * x || x == x1) break;
    if (x == x2) {
      if ((49 - it) & 1) x = x1;
      break;
    }
  }
  return x;
}

__global__ void k_kx(double *kx, int Nx, double dx) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= Nx) return;
  // numpy.fft.fftfreq: integers [0..(n-1)/2, -(n/2)..-1] times 1/(n d)
  int half = (Nx - 1) / 2 + 1;
  double fi = i < half ? (double)i : (double)(i - Nx);
  double val = 1.0 / ((double)Nx * dx);
  kx[i] = (2.0 * PI_D) * (fi * val);
}

__global__ void k_roots(double *kr, int nm, int Nk, double R_period) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nm * Nk) return;
  int m = e / Nk, k = e % Nk;
  kr[e] = bessel_root(m, k + 1) / R_period;
}

// out[i][k] = J_m(r_i kr[k]), times kr[k] / 2 where half is set
struct JmatSet {
  double *out[3 * (CHM_MAXM + 1)];
  const double *kr[3 * (CHM_MAXM + 1)];
  int m[3 * (CHM_MAXM + 1)], half[3 * (CHM_MAXM + 1)];
};
__global__ void k_jmat(JmatSet js, int Nk, double rmin, double dr) {
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)Nk * Nk) return;
  const int s = blockIdx.y;
  const double *kr = js.kr[s];
  int i = (int)(e / Nk), k = (int)(e % Nk);
  double r = rmin + dr * (double)(i + 1);
  double v = bessel_jn(js.m[s], r * kr[k]);
  js.out[s][e] = js.half[s] ? (0.5 * kr[k]) * v : v;
}

// Inverse of an n x n matrix by in-place Gauss-Jordan elimination with partial
// pivoting, NB columns at a time, all modes of a solver in the same launches
// (blockIdx.z = mode).  Every element sees the eliminations of the plain
// column-by-column algorithm, in its order and with its roundings (a product
// and a difference each, pivot rows divided by the pivot), so the blocking
// does not show in the result.  Per panel of NB columns two launches:
//   k_gj_panel   one workgroup: the panel's unfinished rows, one row per
//                thread in registers (RPT rows where n > 1024), column by
//                column (largest remaining element as the pivot, ties to the
//                lowest row).  Leaves the rows' factors F, the scaled pivot
//                rows PR and the pivots D of the panel, and the row order that
//                brings the pivot rows to the panel's place.
//   k_gj_update  the whole matrix, 32 x 32 tiles: the panel's eliminations, in
//                order, on the reordered source.  Source and destination
//                alternate, so the reorder costs nothing; the last panel
//                writes the inverse with its columns put back in the original
//                row order.
// Bound by the chain of pivots: 2 launches per NB columns instead of a
// workgroup that walks the augmented matrix once per column (n = 255, two
// modes: 23.8 -> 0.70 ms; a 1024 x 256 mixed solver with its laser 50.7 ->
// 2.2 ms, with the pulse built from the solver's own tables).
// (k_gj_update deals a panel to eight lanes: NB >= 8)
template <int RPT> struct GjCfg { static constexpr int NB = RPT < 4 ? 32 / RPT : 8; };
#define GJ_T 32  // tile of k_gj_update

struct GjModes {
  const double *src[CHM_MAXM + 1];
  double *dst[CHM_MAXM + 1];
  double *F[CHM_MAXM + 1];   // [n][NB] factors of the rows from the panel on
  double *PR[CHM_MAXM + 1];  // [NB][NB] scaled pivot rows, [NB] pivots
  int *map[CHM_MAXM + 1];    // [n] source row of each destination row
  int *perm[CHM_MAXM + 1];   // [n] original row at each position
};

template <int RPT>
__global__ void __launch_bounds__(1024) k_gj_panel(GjModes g, int n, int p0) {
  constexpr int NB = GjCfg<RPT>::NB;
  __shared__ double raw[NB], prow[2][NB];
  __shared__ double wv[16];
  __shared__ int wi[16];
  __shared__ int piv[NB];
  __shared__ int at[1024 * RPT], pos[1024 * RPT];  // row at a position, position of a row
  const int z = blockIdx.z, t = threadIdx.x, nt = blockDim.x, nw = nt >> 6;
  const int nb = n - p0 < NB ? n - p0 : NB, rows = n - p0;
  const double *S = g.src[z];
  double *F = g.F[z], *PR = g.PR[z];
  double a[RPT][NB];
  int done[RPT];
#pragma unroll
  for (int q = 0; q < RPT; q++) {
    const int r = t + q * nt;
    done[q] = r >= rows;
#pragma unroll
    for (int c = 0; c < NB; c++)
      a[q][c] = (!done[q] && c < nb) ? S[(int64_t)(p0 + r) * n + p0 + c] : 0.0;
    if (r < rows) at[r] = pos[r] = r;
  }
  // The registers shift: a[][0] is always the current column (a loop that
  // names every column is 32 copies of its body, each fetched once: 103
  // us a panel instead of 66, n = 255).
#pragma unroll 1
  for (int c = 0; c < nb; c++) {
    // largest |a[c]| of the rows without a pivot
    double v = -1.0;
    int vi = 0x7fffffff;
#pragma unroll
    for (int q = 0; q < RPT; q++) {
      const double w = fabs(a[q][0]);
      if (!done[q] && w > v) {
        v = w;
        vi = t + q * nt;
      }
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
      const double o = __shfl_xor(v, d);
      const int oi = __shfl_xor(vi, d);
      if (o > v || (o == v && oi < vi)) {
        v = o;
        vi = oi;
      }
    }
    if ((t & 63) == 0) {
      wv[t >> 6] = v;
      wi[t >> 6] = vi;
    }
    __syncthreads();
    v = wv[0];
    vi = wi[0];
    for (int w = 1; w < nw; w++)
      if (wv[w] > v || (wv[w] == v && wi[w] < vi)) {
        v = wv[w];
        vi = wi[w];
      }
    // a column of NaN leaves no candidate: take the lowest row left, so
    // that every index stays in range (the result is NaN, as it must be)
    if (vi >= rows) {
      vi = 0;
      for (int i = 0; i < c; i++)
        for (int k = 0; k < c; k++) vi = piv[k] == vi ? vi + 1 : vi;
    }
#pragma unroll
    for (int q = 0; q < RPT; q++)
      if (t + q * nt == vi) {
#pragma unroll
        for (int k = 0; k < NB; k++) raw[k] = a[q][k];
        done[q] = 1;
        piv[c] = vi;
      }
    __syncthreads();
    double *pr = prow[c & 1];
    if (t < NB) {
      const double d = raw[0], r = t == 0 ? 1.0 : raw[t] / d;
      pr[t] = r;
      PR[c * NB + (c + t) % NB] = r;
      if (t == 0) PR[NB * NB + c] = d;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RPT; q++) {
      const int r = t + q * nt;
      const bool own = r == vi;
      const double f = own ? 0.0 : a[q][0];
      if (r < rows) F[(int64_t)r * NB + c] = f;
#pragma unroll
      for (int k = 1; k < NB; k++) a[q][k - 1] = own ? pr[k] : a[q][k] - f * pr[k];
      a[q][NB - 1] = 0.0;
    }
  }
  if (t == 0)
    for (int c = 0; c < nb; c++) {
      const int from = pos[piv[c]], r = at[c];
      at[c] = piv[c];
      at[from] = r;
      pos[piv[c]] = c;
      pos[r] = from;
    }
  __syncthreads();
  // row order of the whole matrix, and the accumulated one
  int pm[RPT];
#pragma unroll
  for (int q = 0; q < RPT; q++) {
    const int r = t + q * nt;
    pm[q] = r < rows ? g.perm[z][p0 + at[r]] : 0;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < RPT; q++) {
    const int r = t + q * nt;
    if (r < rows) {
      g.map[z][p0 + r] = p0 + at[r];
      g.perm[z][p0 + r] = pm[q];
    }
  }
}

// The panel of more rows than k_gj_panel holds in registers and LDS: the same
// steps on a copy of the panel and on row lists in the mode's scratch (rows
// [n][NB] of F's unused part, lists behind them).
#define GJ_ROWS (1024 * 16)
__global__ void __launch_bounds__(1024) k_gj_panel_mem(GjModes g, int n, int p0) {
  constexpr int NB = GjCfg<16>::NB;
  __shared__ double raw[NB], prow[NB];
  __shared__ double wv[16];
  __shared__ int wi[16];
  __shared__ int piv[NB];
  const int z = blockIdx.z, t = threadIdx.x, nt = blockDim.x, nw = nt >> 6;
  const int nb = n - p0 < NB ? n - p0 : NB, rows = n - p0;
  const double *S = g.src[z];
  double *F = g.F[z], *PR = g.PR[z], *a = F + (int64_t)n * NB;
  int *at = (int *)(a + (int64_t)n * NB), *pos = at + n, *done = pos + n, *tmp = done + n;
  for (int r = t; r < rows; r += nt) {
    for (int c = 0; c < NB; c++)
      a[(int64_t)r * NB + c] = c < nb ? S[(int64_t)(p0 + r) * n + p0 + c] : 0.0;
    at[r] = pos[r] = r;
    done[r] = 0;
  }
  __syncthreads();
  for (int c = 0; c < nb; c++) {
    double v = -1.0;
    int vi = 0x7fffffff;
    for (int r = t; r < rows; r += nt) {
      const double w = fabs(a[(int64_t)r * NB + c]);
      if (!done[r] && w > v) {
        v = w;
        vi = r;
      }
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
      const double o = __shfl_xor(v, d);
      const int oi = __shfl_xor(vi, d);
      if (o > v || (o == v && oi < vi)) {
        v = o;
        vi = oi;
      }
    }
    if ((t & 63) == 0) {
      wv[t >> 6] = v;
      wi[t >> 6] = vi;
    }
    __syncthreads();
    v = wv[0];
    vi = wi[0];
    for (int w = 1; w < nw; w++)
      if (wv[w] > v || (wv[w] == v && wi[w] < vi)) {
        v = wv[w];
        vi = wi[w];
      }
    if (vi >= rows) {  // a column of NaN, as in k_gj_panel
      vi = 0;
      for (int i = 0; i < c; i++)
        for (int k = 0; k < c; k++) vi = piv[k] == vi ? vi + 1 : vi;
    }
    if (t < NB) raw[t] = t < c ? 0.0 : a[(int64_t)vi * NB + t];
    if (t == 0) {
      done[vi] = 1;
      piv[c] = vi;
    }
    __syncthreads();
    if (t < NB) {
      const double d = raw[c], r = t == c ? 1.0 : raw[t] / d;
      prow[t] = r;
      PR[c * NB + t] = r;
      if (t == 0) PR[NB * NB + c] = d;
    }
    __syncthreads();
    for (int r = t; r < rows; r += nt) {
      double *ar = a + (int64_t)r * NB;
      const bool own = r == vi;
      const double f = own ? 0.0 : ar[c];
      F[(int64_t)r * NB + c] = f;
      for (int k = c + 1; k < NB; k++) ar[k] = own ? prow[k] : ar[k] - f * prow[k];
    }
    __syncthreads();
  }
  if (t == 0)
    for (int c = 0; c < nb; c++) {
      const int from = pos[piv[c]], r = at[c];
      at[c] = piv[c];
      at[from] = r;
      pos[piv[c]] = c;
      pos[r] = from;
    }
  __syncthreads();
  for (int r = t; r < rows; r += nt) tmp[r] = g.perm[z][p0 + at[r]];
  __syncthreads();
  for (int r = t; r < rows; r += nt) {
    g.map[z][p0 + r] = p0 + at[r];
    g.perm[z][p0 + r] = tmp[r];
  }
}

template <int RPT>
__global__ void __launch_bounds__(256) k_gj_update(GjModes g, int n, int p0, int last) {
  constexpr int NB = GjCfg<RPT>::NB;
  constexpr int PER = NB / 8;  // panel rows (columns) of each of 8 lanes
  __shared__ double Fs[GJ_T][NB + 1], Y[NB][GJ_T + 1], Z[NB][GJ_T + 1], Fp[NB][NB + 1], P[NB][NB + 1];
  const int z = blockIdx.z, t = threadIdx.x, j0 = blockIdx.x * GJ_T, i0 = blockIdx.y * GJ_T;
  const int nb = n - p0 < NB ? n - p0 : NB;
  const double *S = g.src[z], *F = g.F[z], *PR = g.PR[z];
  const int *map = g.map[z];
  auto row = [&](int i) { return i < p0 ? i : map[i]; };
  auto in = [&](int i) { return i >= p0 && i < p0 + nb; };
  // factors of the pivot rows, scaled pivot rows within the panel
  for (int e = t; e < NB * NB; e += 256) {
    const int q = e / NB, k = e % NB;
    Fp[q][k] = q < nb && k < nb ? F[(int64_t)(map[p0 + q] - p0) * NB + k] : 0.0;
    P[q][k] = q < nb && k < nb ? PR[e] : 0.0;
  }
  __syncthreads();
  const int g8 = t >> 3, l8 = t & 7, base = (t & 63) & ~7;
  // Y[q] = pivot row q as the others see it, Z[q] = pivot row q in the end;
  // eight lanes share a column
  {
    const int j = j0 + g8, jq = j - p0;
    double v[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int q = l8 * PER + u;
      v[u] = q < nb && j < n ? S[(int64_t)map[p0 + q] * n + j] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < NB; q++) {
      if (q < nb) {
        const double x = __shfl(v[q % PER], base + q / PER), d = PR[NB * NB + q];
        const double s = jq == q ? 1.0 / d : x / d;
        if (l8 == 0) Y[q][g8] = s;
#pragma unroll
        for (int u = 0; u < PER; u++) {
          const int r = l8 * PER + u;
          const double o = jq == q ? 0.0 : v[u];
          v[u] = r == q ? s : o - Fp[r][q] * s;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < PER; u++) Z[l8 * PER + u][g8] = v[u];
  }
  // factors of the tile's rows: from the panel on they are known, above it
  // the row's panel columns are taken through the eliminations
  {
    const int i = i0 + g8;
    if (i0 + GJ_T > p0) {
#pragma unroll
      for (int u = 0; u < PER; u++) {
        const int k = l8 * PER + u;
        if (i >= p0) Fs[g8][k] = i < n && k < nb ? F[(int64_t)(map[i] - p0) * NB + k] : 0.0;
      }
    }
    if (i0 < p0) {
      double v[PER];
#pragma unroll
      for (int u = 0; u < PER; u++) {
        const int k = l8 * PER + u;
        v[u] = i < n && k < nb ? S[(int64_t)row(i) * n + p0 + k] : 0.0;
      }
#pragma unroll
      for (int q = 0; q < NB; q++) {
        if (q < nb) {
          const double f = __shfl(v[q % PER], base + q / PER);
          if (l8 == 0 && i < p0) Fs[g8][q] = f;
#pragma unroll
          for (int u = 0; u < PER; u++) v[u] = v[u] - f * P[q][l8 * PER + u];
        }
      }
    }
  }
  __syncthreads();
  const int tx = t & 15, ty = t >> 4;
  double acc[2][2];
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++) {
      const int i = i0 + ty + 16 * u, j = j0 + tx + 16 * v;
      acc[u][v] = i < n && j < n && !in(i) ? S[(int64_t)row(i) * n + j] : 0.0;
    }
  for (int q = 0; q < nb; q++) {
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int v = 0; v < 2; v++) {
        const int j = j0 + tx + 16 * v;
        const double o = j - p0 == q ? 0.0 : acc[u][v];
        acc[u][v] = o - Fs[ty + 16 * u][q] * Y[q][tx + 16 * v];
      }
  }
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++) {
      const int i = i0 + ty + 16 * u, j = j0 + tx + 16 * v;
      if (i >= n || j >= n) continue;
      const double r = in(i) ? Z[i - p0][tx + 16 * v] : acc[u][v];
      g.dst[z][(int64_t)i * n + (last ? g.perm[z][j] : j)] = r;
    }
}

__global__ void k_gj_iota(GjModes g, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) g.perm[blockIdx.z][i] = i;
}

// Scratch of one mode: two n x n buffers (the panels alternate between them;
// the first panel reads the input itself), F, PR and D, map and perm.
static size_t gj_pr_bytes() { return chm_align((32 * 32 + 32) * 8); }
static size_t gj_bytes(int n) {
  return 2 * chm_align((size_t)n * n * 8) + chm_align((size_t)n * 32 * 8) + gj_pr_bytes() +
         2 * chm_align((size_t)n * 4);
}

template <int RPT>
static void gj_inverse(const double *const *a, double *const *inv, int nmode, int n, char *ws,
                       hipStream_t st) {
  constexpr int NB = GjCfg<RPT>::NB;
  GjModes g = {};
  double *buf[CHM_MAXM + 1][2];
  const size_t mat = chm_align((size_t)n * n * 8);
  for (int m = 0; m < nmode; m++) {
    char *b = ws + (size_t)m * gj_bytes(n);
    buf[m][0] = (double *)b;
    buf[m][1] = (double *)(b + mat);
    b += 2 * mat;
    g.F[m] = (double *)b;
    b += chm_align((size_t)n * 32 * 8);
    g.PR[m] = (double *)b;
    b += gj_pr_bytes();
    g.map[m] = (int *)b;
    g.perm[m] = (int *)(b + chm_align((size_t)n * 4));
    g.src[m] = a[m];
  }
  k_gj_iota<<<dim3(chm_blocks(n, 256), 1, nmode), 256, 0, st>>>(g, n);
  const dim3 tiles((n + GJ_T - 1) / GJ_T, (n + GJ_T - 1) / GJ_T, nmode);
  for (int p0 = 0, s = 0; p0 < n; p0 += NB, s ^= 1) {
    const int last = p0 + NB >= n;
    for (int m = 0; m < nmode; m++) g.dst[m] = last ? inv[m] : buf[m][s];
    if (n - p0 > GJ_ROWS) {
      k_gj_panel_mem<<<dim3(1, 1, nmode), 1024, 0, st>>>(g, n, p0);
    } else {
      int nt = (n - p0 + RPT - 1) / RPT;
      nt = (nt + 63) / 64 * 64;
      k_gj_panel<RPT><<<dim3(1, 1, nmode), nt, 0, st>>>(g, n, p0);
    }
    k_gj_update<RPT><<<tiles, 256, 0, st>>>(g, n, p0, last);
    for (int m = 0; m < nmode; m++) g.src[m] = g.dst[m];
  }
}

__global__ void k_wtables(chm_tables_out_t o, int Nx, int Nk, double dt) {
  const int m = blockIdx.y;
  const double *kx = o.kx, *kr = o.kr + (int64_t)m * Nk;
  double *w = o.w[m], *c1 = o.c1[m], *c2 = o.c2[m], *c3 = o.c3[m], *smooth = o.smooth[m];
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)Nk * Nx) return;
  int i = (int)(e / Nx), j = (int)(e % Nx);
  double kxv = kx[j], krv = kr[i];
  double ww = sqrt(kxv * kxv + krv * krv);
  w[e] = ww;
  c1[e] = cos(ww * dt);
  c2[e] = sin(ww * dt) * ww;
  c3[e] = 1. / (ww * ww);
  // kx.max() of fftfreq order is kx[(Nx-1)/2]; kr.max() is the last root
  double kxmax = kx[(Nx - 1) / 2], krmax = kr[Nk - 1];
  double sx = sin(0.5 * PI_D * kxv / kxmax), sr = sin(0.5 * PI_D * krv / krmax);
  smooth[e] = (1 - sx * sx) * (1 - sr * sr);
}

__global__ void k_phase_tw(const double *kx, int Nx, double xmin, double2 *pm, double2 *pp, double2 *tw) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= Nx) return;
  double a = xmin * kx[i];
  double c = cos(a), s = sin(a);
  pm[i] = make_double2(c, -s);
  pp[i] = make_double2(c, s);
  double sn, cs;
  sincospi(2.0 * (double)i / (double)Nx, &sn, &cs);
  tw[i] = make_double2(cs, -sn);
}

__global__ void k_damp_profile(double *f, int N) {
  int z = blockIdx.x * blockDim.x + threadIdx.x;
  if (z >= 2 * N) return;
  double zs = 3. * (z - N + 1) / (N + 1);
  double s = sin(0.5 * PI_D * zs);
  double v = ((z < 4. * N / 3) && (z >= N)) ? s * s : 0.0;
  if (z >= 4. * N / 3) v += 1.0;
  f[z] = v;
}

// Per mode: the scratch of the inverse, J_{m+1} and J_{m-1} matrices and the
// padded DHT the products read.
static size_t tables_mode_bytes(int Nk) {
  return gj_bytes(Nk) + 2 * chm_align((size_t)Nk * Nk * 8) +
         chm_align(chm_dht_table_elems(Nk, Nk) * 8);
}
extern "C" size_t chm_tables_workspace_bytes(int32_t Nx, int32_t Nr, int32_t M) {
  return (size_t)(M + 1) * tables_mode_bytes(Nr - 1);
}

// Every matrix of every mode goes through the same launches: the set-up of a
// small grid is bound by the number of launches, that of a large one by the
// pivots of the inverse, and neither grows with the number of modes.
extern "C" int chm_build_tables_f64(int32_t Nx, int32_t Nr, int32_t M, double dx, double dr, double dt,
                                    double xmin, int32_t damp_cells, const chm_tables_out_t *out, void *ws,
                                    size_t ws_bytes, void *stream) {
  if (!out || Nx < 2 || Nr < 3 || M < 0 || M > CHM_MAXM) return CHM_EINVAL;
  if (chm_tables_workspace_bytes(Nx, Nr, M) > ws_bytes || !ws) return CHM_EWORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  const int Nk = Nr - 1;
  const double rmin = -0.5 * dr;
  const double R_period = (rmin + dr * (double)(Nr - 1)) + 0.5 * dr;
  const size_t mat = chm_align((size_t)Nk * Nk * 8);
  char *b = (char *)ws + (size_t)(M + 1) * gj_bytes(Nk);
  const size_t pad = chm_align(chm_dht_table_elems(Nk, Nk) * 8);
  k_kx<<<chm_blocks(Nx, 256), 256, 0, st>>>(out->kx, Nx, dx);
  k_roots<<<chm_blocks((M + 2) * Nk, 64), 64, 0, st>>>(out->kr, M + 2, Nk, R_period);
  int64_t nn = (int64_t)Nk * Nk;
  JmatSet js = {};
  GemmBatch gb = {};
  gb.M = gb.K = Nk;
  gb.lda = gemm_lda(Nk);
  const double *jm[CHM_MAXM + 1];
  double *dht[CHM_MAXM + 1];
  for (int m = 0; m <= M; m++) {
    double *Jp = (double *)(b + (size_t)m * (2 * mat + pad)), *Jm = Jp + mat / 8, *Dpad = Jm + mat / 8;
    jm[m] = out->DHT_inv[m];
    dht[m] = out->DHT[m];
    double *const o[3] = {out->DHT_inv[m], Jp, Jm};
    const int of[3] = {m, m + 1, m > 0 ? m - 1 : 1};
    for (int q = 0; q < 3; q++) {
      js.out[3 * m + q] = o[q];
      js.kr[3 * m + q] = out->kr + (size_t)of[q] * Nk;
      js.m[3 * m + q] = m;
      js.half[3 * m + q] = q > 0;
    }
    for (int q = 0; q < 2; q++) {
      GemmItem &it = gb.it[2 * m + q];
      it.A = Dpad;
      it.X = q ? Jm : Jp;
      it.C = q ? out->dDm[m] : out->dDp[m];
      it.N = Nk;
    }
  }
  k_jmat<<<dim3(chm_blocks(nn, 256), 3 * (M + 1)), 256, 0, st>>>(js, Nk, rmin, dr);
  if (Nk <= 1024) gj_inverse<1>(jm, dht, M + 1, Nk, (char *)ws, st);
  else if (Nk <= 4096) gj_inverse<4>(jm, dht, M + 1, Nk, (char *)ws, st);
  else gj_inverse<16>(jm, dht, M + 1, Nk, (char *)ws, st);  // (rows partly, above GJ_ROWS all in scratch memory)
  for (int m = 0; m <= M; m++) {
    int rc = chm_pad_table(dht[m], Nk, Nk, (double *)gb.it[2 * m].A, nullptr, nullptr, nullptr, stream);
    if (rc) return rc;
  }
  int rc = chm_gemm_launch(gb, 2 * (M + 1), GEMM_F64, st);
  if (rc) return rc;
  k_wtables<<<dim3(chm_blocks((int64_t)Nk * Nx, 256), M + 1), 256, 0, st>>>(*out, Nx, Nk, dt);
  k_phase_tw<<<chm_blocks(Nx, 256), 256, 0, st>>>(out->kx, Nx, xmin, (double2 *)out->phase_minus,
                                                  (double2 *)out->phase_plus, (double2 *)out->twiddle);
  if (damp_cells > 0 && out->damp)
    k_damp_profile<<<chm_blocks(2 * damp_cells, 256), 256, 0, st>>>(out->damp, damp_cells);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

// ---------------------------------------------------------------- conversions
__global__ void k_convert(const double *src, int64_t n, float *f32, uint16_t *hi, uint16_t *lo) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double v = src[i];
  if (f32) f32[i] = (float)v;
  if (hi) {
    __bf16 h = (__bf16)(float)v;
    __bf16 l = (__bf16)(float)(v - (double)(float)h);
    hi[i] = __builtin_bit_cast(uint16_t, h);
    lo[i] = __builtin_bit_cast(uint16_t, l);
  }
}

extern "C" int chm_convert_table(const double *src, int64_t n, float *f32, uint16_t *bf16_hi,
                                 uint16_t *bf16_lo, void *stream) {
  if (!src || n < 0 || ((bf16_hi == nullptr) != (bf16_lo == nullptr))) return CHM_EINVAL;
  if (n == 0) return CHM_OK;
  k_convert<<<chm_blocks(n, 256), 256, 0, (hipStream_t)stream>>>(src, n, f32, bf16_hi, bf16_lo);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

// ---------------------------------------------------------------- frame
// get_phase_minus / get_phase_plus (transformer_generic.cl:28-55) for a new
// window origin xmin (moving window, frame.py:22-30).
__global__ void k_phases(const double *kx, int Nx, double xmin, double2 *pm, double2 *pp) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= Nx) return;
  double a = xmin * kx[i];
  double c = cos(a), s = sin(a);
  pm[i] = make_double2(c, -s);
  pp[i] = make_double2(c, s);
}

extern "C" int chm_phase_tables_f64(const double *kx, int32_t Nx, double xmin, void *phase_minus,
                                    void *phase_plus, void *stream) {
  if (!kx || !phase_minus || !phase_plus || Nx < 1) return CHM_EINVAL;
  k_phases<<<chm_blocks(Nx, 256), 256, 0, (hipStream_t)stream>>>(kx, Nx, xmin, (double2 *)phase_minus,
                                                                 (double2 *)phase_plus);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}
