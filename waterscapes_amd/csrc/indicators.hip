// A-posteriori error indicators of the two-field MPET step
// (AdaptiveMPETSolver.__init_error_estimators / estimate_error_at_t,
// mpet/adaptivempetsolver.py:82-185), per cell (DG0):
//
//   zeta_p(K)    = sum_j  h_K^2 ||RK_p,j||_K^2 + sum_F avg(h) avg(w) ||RE_p,j||_F^2
//   zeta_u(K)    =        h_K^2 ||RK_u||_K^2   + sum_F avg(h) avg(w) ||RE_u||_F^2
//   zeta_udt(K)  = the same with (RK_u - RK_u^-)/dt and (RE_u - RE_u^-)/dt
//   r4(K)        = the cell part of R4p (:146-153)
//
//   RK_u   = f + div sigma(u) - sum_i alpha_i grad p_i        (:121)
//   RE_u   = sum_i jump(alpha_i p_i, n) - jump(sigma(u), n)     (:122)
//   RK_p,j = -g_j - c_j (p_j - p_j^-)/dt - alpha_j div(u - u^-)/dt
//            + K_j div grad p_j - sum_i S_ij (p_j - p_i)        (:130-132)
//   RE_p,j = -K_j jump(grad p_j, n)                             (:133)
//   sigma(u) = 2 mu eps(u) + lambda div u I, h = cell diameter (longest
//   edge), the facet sums over interior facets (dS) with avg(w) = 1/2 for
//   each of the two cells.
//
// u is P2 (div sigma(u) is constant per cell), p_j P1 (div grad p_j = 0).
// Cell integrals use a Grundmann-Moeller rule exact for the integrand
// degree, facet integrals the 3-point edge-midpoint rule (exact for the
// quadratic |RE_u|^2).  One thread per cell / per interior facet; the facet
// values are summed into the cells by a gather kernel (deterministic).
#include "mpet_ops.h"
#include <mutex>
#include <stdio.h>

namespace mpet {

struct IGeom {
  double g[4][3];   // grad lambda_k
  double vol, h;
};

// Local vertices may be taken in any order p of the cell's own (a facet's
// first, see ind_facet_kernel): vertex i is the cell's p[i], and the edge node
// of i and j is found from the cell's own numbering (edges (2,3), (1,3),
// (1,2), (0,3), (0,2), (0,1) after the four vertices).
__device__ __forceinline__ int p2_edge(int i, int j) {
  const int lo = i < j ? i : j, hi = i < j ? j : i;
  return 4 + (lo == 0 ? 6 - hi : (lo == 1 ? 4 - hi : 0));
}

// Geometry from four vertices: gradients of the barycentric coordinates,
// volume and diameter (longest edge).
__device__ __forceinline__ void igeom(const double v[4][3], IGeom& G) {
  double J[3][3];
  for (int d = 0; d < 3; ++d)
    for (int k = 0; k < 3; ++k) J[d][k] = v[k + 1][d] - v[0][d];
  const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
  const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
  const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
  const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
  const double id = 1.0 / det;
  // rows of J^-1 = grad lambda_1..3
  double Ji[3][3];
  Ji[0][0] = c00 * id;
  Ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
  Ji[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
  Ji[1][0] = c01 * id;
  Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
  Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
  Ji[2][0] = c02 * id;
  Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
  Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
  for (int m = 0; m < 3; ++m) {
    G.g[1][m] = Ji[0][m];
    G.g[2][m] = Ji[1][m];
    G.g[3][m] = Ji[2][m];
    G.g[0][m] = -(Ji[0][m] + Ji[1][m] + Ji[2][m]);
  }
  G.vol = fabs(det) / 6.0;
  double h2 = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = i + 1; j < 4; ++j) {
      double s = 0.0;
      for (int d = 0; d < 3; ++d) s += (v[i][d] - v[j][d]) * (v[i][d] - v[j][d]);
      h2 = fmax(h2, s);
    }
  G.h = sqrt(h2);
}

// A P2 gradient is linear on the cell, so everything the indicators need of
// u follows from grad u at the vertices,
//   (grad u)_n = 4 u_n G_n - sum_j u_j G_j + 4 sum_{k != n} u_{nk} G_k
// (G_j = grad lambda_j): div sigma = sum_n sigma_n G_n, the divergence by its
// vertex values, a facet's tractions at its vertices and their means at the
// edge midpoints.  (Summing basis gradients and Hessians node by node at
// every point, and the facets' geometry at every point, took 5 times the
// arithmetic: see the figures at the kernels.)
// nd: the cell's ten node numbers in the local order; visit(n, g) with g[i][j]
// = d_j u_i at vertex n, for the first NV vertices.
template <int NV, typename V>
__device__ __forceinline__ void vertex_gradients(const IGeom& G, const double* __restrict__ x,
                                                 const int nd[10], V visit) {
  double u[10][3];
#pragma unroll
  for (int a = 0; a < 10; ++a)
    for (int i = 0; i < 3; ++i) u[a][i] = x[3ll * nd[a] + i];
  double U[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      U[i][j] = (u[0][i] * G.g[0][j] + u[1][i] * G.g[1][j]) +
                (u[2][i] * G.g[2][j] + u[3][i] * G.g[3][j]);
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    double g[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        double t = u[n][i] * G.g[n][j];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k != n) t += u[p2_edge(n, k)][i] * G.g[k][j];
        g[i][j] = 4.0 * t - U[i][j];
      }
    visit(n, g);
  }
}

// One thread per cell; the network count is a template argument so that the
// pressure loops hold exactly A fields.  Bound by the FP64 arithmetic and the
// registers it holds (two waves a SIMD): 24 us at 32^3 x 6 tets, A = 2 (both
// kernels and the gather 79 us of a call's 367, the rest brings 6.3 MB to the
// host; the call took 880 us with per-point gradients and Hessians and a
// pageable copy).
// The sources' nodal values are 3 nkf (f, f^-) and A nkg (g) consecutive
// doubles a cell, read again at every quadrature point.  A thread reading its
// own cell's has 64 lines a load: 398 us at degree 2 with 15 points, 32^3 x 6
// tets.  STAGE brings a block's into LDS first (one run in memory; rows of odd
// length, so that a wave's reads spread over the banks): 128 us there.  Up to
// 64 KB a block: degree 3 for both f and f^- takes 62,464 bytes (two waves a CU,
// and still the faster: a call 0.89 against 2.57 ms read directly at 32^3, 117
// against 223 us at 8^3); rows past 127 doubles, such as those with a g beside
// them, are read directly.
static inline __host__ __device__ int ind_row(const double* p, int w) { return p ? w | 1 : 0; }
constexpr int IND_STAGE_ROW = 127;   // doubles a cell: at most 64 KB per 64 cells
template <int A, bool STAGE>
__global__ void __launch_bounds__(STAGE ? 64 : 128)
ind_cell_kernel(MpetIndDesc d, const double* __restrict__ x, const double* __restrict__ xp,
                double* __restrict__ out) {
  constexpr int NTI = STAGE ? 64 : 128;
  extern __shared__ double ind_lds[];
  const int e = blockIdx.x * NTI + threadIdx.x;
  const int wf = 3 * d.nkf, wg = A * d.nkg;
  const int Wf = ind_row(d.f, wf), Wp = ind_row(d.fp, wf), Wg = ind_row(d.g, wg);
  const double* sf = ind_lds;
  const double* sp = ind_lds + NTI * Wf;
  const double* sg = ind_lds + NTI * (Wf + Wp);
  if constexpr (STAGE) {
    const int first = blockIdx.x * NTI;
    const int cnt = d.nC - first < NTI ? d.nC - first : NTI;
    auto bring = [&](const double* __restrict__ src, int w, int W, double* dst) {
      if (!src) return;
      const double* __restrict__ p = src + (long long)first * w;
      int row = threadIdx.x / w, col = threadIdx.x % w;
      for (int i = threadIdx.x; i < cnt * w; i += NTI) {
        dst[row * W + col] = p[i];
        col += NTI % w;
        row += NTI / w;
        if (col >= w) {
          col -= w;
          ++row;
        }
      }
    };
    bring(d.f, wf, Wf, ind_lds);
    bring(d.fp, wf, Wp, ind_lds + NTI * Wf);
    bring(d.g, wg, Wg, ind_lds + NTI * (Wf + Wp));
    __syncthreads();
  }
  if (e >= d.nC) return;
  auto f_at = [&](int k) { return STAGE ? sf[threadIdx.x * Wf + k] : d.f[(long long)e * wf + k]; };
  auto fp_at = [&](int k) {
    return STAGE ? sp[threadIdx.x * Wp + k] : d.fp[(long long)e * wf + k];
  };
  auto g_at = [&](int k) { return STAGE ? sg[threadIdx.x * Wg + k] : d.g[(long long)e * wg + k]; };
  const long long nu = 3ll * d.nP2;
  IGeom G;
  int p2[10], v[4];
  for (int k = 0; k < 4; ++k) v[k] = d.cells[4 * e + k];
  for (int a = 0; a < 10; ++a) p2[a] = d.cell_p2[10 * e + a];
  {
    double X[4][3];
    for (int k = 0; k < 4; ++k)
      for (int m = 0; m < 3; ++m) X[k][m] = d.coords[3ll * v[k] + m];
    igeom(X, G);
  }
  // constant parts of RK_u, RK_u^-: div sigma(u) - sum_i alpha_i grad p_i;
  // div(u - u^-) at the vertices
  double cu[3], cup[3] = {0, 0, 0}, dv[4] = {0, 0, 0, 0};
  const double mu = d.mu, lm = d.lmbda;
  auto add = [&](int n, const double g[3][3], double c[3]) {
    const double tr = g[0][0] + g[1][1] + g[2][2];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      double s = lm * tr * G.g[n][i];
#pragma unroll
      for (int j = 0; j < 3; ++j) s += mu * (g[i][j] + g[j][i]) * G.g[n][j];
      c[i] += s;
    }
    return tr;
  };
#pragma unroll 1
  for (int k = 0; k < 2; ++k) {                // one state's values live at a time
    for (int i = 0; i < 3; ++i) {
      cu[i] = cup[i];
      cup[i] = 0.0;
    }
    vertex_gradients<4>(G, k ? xp : x, p2, [&](int n, const double g[3][3]) {
      const double tr = add(n, g, cup);
      dv[n] = k ? dv[n] - tr : tr;
    });
  }
  double r4 = 0.0;
#pragma unroll
  for (int j = 0; j < A; ++j) {
    double gp[3] = {0, 0, 0}, gpp[3] = {0, 0, 0};
    for (int k = 0; k < 4; ++k) {
      const long long q = nu + (long long)A * v[k] + j;
      for (int m = 0; m < 3; ++m) {
        gp[m] += x[q] * G.g[k][m];
        gpp[m] += xp[q] * G.g[k][m];
      }
    }
    for (int m = 0; m < 3; ++m) {
      cu[m] -= d.alpha[j] * gp[m];
      cup[m] -= d.alpha[j] * gpp[m];
      r4 += d.K[j] * (gp[m] - gpp[m]) * (gp[m] - gpp[m]) * G.vol;
    }
  }
  const double idt = 1.0 / d.dt;
  double zu = 0.0, zudt = 0.0, zp = 0.0, r4s = 0.0;
#pragma unroll 1
  for (int q = 0; q < d.nq; ++q) {
    const double* l = d.qbary + 4 * q;
    const double w = d.qw[q];
    double fq[3] = {0, 0, 0}, fpq[3] = {0, 0, 0};
    if (d.f)
      for (int m = 0; m < d.nkf; ++m) {
        const double L = d.Lf[q * d.nkf + m];
        for (int i = 0; i < 3; ++i) fq[i] += L * f_at(3 * m + i);
      }
    if (d.fp)
      for (int m = 0; m < d.nkf; ++m) {
        const double L = d.Lf[q * d.nkf + m];
        for (int i = 0; i < 3; ++i) fpq[i] += L * fp_at(3 * m + i);
      }
    double ru2 = 0.0, rd2 = 0.0;
    for (int i = 0; i < 3; ++i) {
      const double r = fq[i] + cu[i], rp = fpq[i] + cup[i];
      ru2 += r * r;
      rd2 += (r - rp) * idt * (r - rp) * idt;
    }
    zu += w * ru2;
    zudt += w * rd2;
    // div(u - u^-) at the point (linear on the cell)
    const double du = l[0] * dv[0] + l[1] * dv[1] + l[2] * dv[2] + l[3] * dv[3];
    double pj[A], ppj[A];
#pragma unroll
    for (int j = 0; j < A; ++j) {
      pj[j] = ppj[j] = 0.0;
      for (int k = 0; k < 4; ++k) {
        const long long qq = nu + (long long)A * v[k] + j;
        pj[j] += l[k] * x[qq];
        ppj[j] += l[k] * xp[qq];
      }
    }
#pragma unroll
    for (int j = 0; j < A; ++j) {
      double gj = 0.0;
      if (d.g)
        for (int m = 0; m < d.nkg; ++m)
          gj += d.Lg[q * d.nkg + m] * g_at(m * A + j);
      double r = -gj - d.c[j] * (pj[j] - ppj[j]) * idt - d.alpha[j] * du * idt;
#pragma unroll
      for (int i = 0; i < A; ++i) r -= d.S[i * MPET_MAXF + j] * (pj[j] - pj[i]);
      zp += w * r * r;
#pragma unroll
      for (int i = 0; i < A; ++i)
        if (d.S[i * MPET_MAXF + j] > 3.0e-16)
          r4s += w * d.S[i * MPET_MAXF + j] * ((pj[j] - ppj[j]) - (pj[i] - ppj[i])) *
                 (pj[j] - ppj[j]);
    }
  }
  const double h2v = G.h * G.h * G.vol;
  out[e] = zp * h2v;
  out[(long long)d.nC + e] = zu * h2v;
  out[2ll * d.nC + e] = zudt * h2v;
  out[3ll * d.nC + e] = r4 + r4s * G.vol;
}

// One interior facet: fac = (cell a, local face a, cell b, local face b).
// out_f[0..2][t] = avg(h) int_F |RE_p|^2 (sum over j), |RE_u|^2, |RE_u,dt|^2.
// Each cell's vertices are taken facet first (the three shared ones in cell
// a's order, found in cell b by their numbers), the opposite one last, so
// that the tractions at the facet's vertices are the first three of
// vertex_gradients and every register index is static.  The pressures are
// continuous: their jump alpha_i (p_i^a - p_i^b) n is zero.  RE_u is linear on
// the facet; the edge-midpoint rule takes the means of its vertex values.
// Bound as the cell kernel: 48 us for the 32^3 mesh's 390,000 facets.
template <int A>
__global__ void __launch_bounds__(128)
ind_facet_kernel(MpetIndDesc d, const double* __restrict__ x, const double* __restrict__ xp,
                 const int* __restrict__ fac, int nF, double* __restrict__ out_f) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nF) return;
  const int la = fac[4 * t + 1], lb = fac[4 * t + 3];
  const long long nu = 3ll * d.nP2;
  double re[3][3], rp[3][3], jn[A];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int i = 0; i < 3; ++i) re[k][i] = rp[k][i] = 0.0;
#pragma unroll
  for (int j = 0; j < A; ++j) jn[j] = 0.0;
  double nrm[3] = {0.0, 0.0, 0.0}, area = 0.0, hsum = 0.0;
  int fv[3] = {0, 0, 0};
#pragma unroll 1
  for (int side = 0; side < 2; ++side) {       // one cell's geometry live at a time
    const int cell = fac[4 * t + 2 * side], opp = side ? lb : la;
    const int* __restrict__ cv = d.cells + 4ll * cell;
    const int* __restrict__ c2 = d.cell_p2 + 10ll * cell;
    // local order: facet vertices, then the opposite one
    int p[4];
    p[0] = opp == 0 ? 1 : 0;
    p[1] = opp <= 1 ? 2 : 1;
    p[2] = opp <= 2 ? 3 : 2;
    p[3] = opp;
    int g4[4];
    for (int k = 0; k < 4; ++k) g4[k] = cv[p[k]];
    if (side) {                                 // cell a's order of the shared three
      int q[3];
#pragma unroll
      for (int k = 0; k < 3; ++k)
        q[k] = g4[0] == fv[k] ? p[0] : (g4[1] == fv[k] ? p[1] : p[2]);
      p[0] = q[0]; p[1] = q[1]; p[2] = q[2];
      g4[0] = fv[0]; g4[1] = fv[1]; g4[2] = fv[2];
    } else {
      fv[0] = g4[0]; fv[1] = g4[1]; fv[2] = g4[2];
    }
    int nd[10];
#pragma unroll
    for (int k = 0; k < 4; ++k) nd[k] = c2[p[k]];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = i + 1; j < 4; ++j) nd[p2_edge(i, j)] = c2[p2_edge(p[i], p[j])];
    IGeom G;
    {
      double X[4][3];
      for (int k = 0; k < 4; ++k)
        for (int m = 0; m < 3; ++m) X[k][m] = d.coords[3ll * g4[k] + m];
      igeom(X, G);
      if (side == 0) {
        // outward normal of cell a: -grad lambda of the opposite vertex
        const double n = sqrt(G.g[3][0] * G.g[3][0] + G.g[3][1] * G.g[3][1] +
                              G.g[3][2] * G.g[3][2]);
        for (int m = 0; m < 3; ++m) nrm[m] = -G.g[3][m] / n;
        area = 3.0 * G.vol * n;                 // |F| = 3 |K| |grad lambda_opp|
      }
    }
    hsum += G.h;
    const double sg = side ? 1.0 : -1.0;        // RE_u = -(sigma_a - sigma_b) n
#pragma unroll
    for (int j = 0; j < A; ++j) {
      double s = 0.0;
      for (int k = 0; k < 4; ++k) {
        const double gn = G.g[k][0] * nrm[0] + G.g[k][1] * nrm[1] + G.g[k][2] * nrm[2];
        s += x[nu + (long long)A * g4[k] + j] * gn;
      }
      jn[j] -= sg * s;
    }
    auto traction = [&](const double g[3][3], double (&r)[3]) {
      const double tr = g[0][0] + g[1][1] + g[2][2];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        double s = d.lmbda * tr * nrm[i];
#pragma unroll
        for (int j = 0; j < 3; ++j) s += d.mu * (g[i][j] + g[j][i]) * nrm[j];
        r[i] += sg * s;
      }
    };
    vertex_gradients<3>(G, x, nd, [&](int n, const double g[3][3]) { traction(g, re[n]); });
    vertex_gradients<3>(G, xp, nd, [&](int n, const double g[3][3]) { traction(g, rp[n]); });
  }
  const double havg = 0.5 * hsum, idt = 1.0 / d.dt;
  double fp = 0.0;
#pragma unroll
  for (int j = 0; j < A; ++j) fp += d.K[j] * jn[j] * d.K[j] * jn[j];
  fp *= area;
  double fu = 0.0, fud = 0.0;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int o = q == 2 ? 0 : q + 1;
    double a2 = 0.0, d2 = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double m = 0.5 * (re[q][i] + re[o][i]);
      const double r = (m - 0.5 * (rp[q][i] + rp[o][i])) * idt;
      a2 += m * m;
      d2 += r * r;
    }
    fu += a2 * (area / 3.0);
    fud += d2 * (area / 3.0);
  }
  out_f[t] = havg * fp;
  out_f[(long long)nF + t] = havg * fu;
  out_f[2ll * nF + t] = havg * fud;
}

// out[k][e] += 1/2 sum over the interior facets of cell e of out_f[k].
__global__ void __launch_bounds__(256)
ind_gather_kernel(int nC, const int* __restrict__ cell_f, const double* __restrict__ out_f,
                  int nF, double* __restrict__ out) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nC) return;
  for (int k = 0; k < 3; ++k) {
    double s = 0.0;
    for (int l = 0; l < 4; ++l) {
      const int f = cell_f[4 * e + l];
      if (f >= 0) s += out_f[(long long)k * nF + f];
    }
    out[(long long)k * nC + e] += 0.5 * s;
  }
}

}  // namespace mpet

using namespace mpet;

static int launch_indicators(const MpetIndDesc* d, const double* x, const double* xp,
                             const int* fac, int nF, const int* cell_f, double* tmp,
                             double* out, hipStream_t stream, const char* who) {
  const int row = ind_row(d->f, 3 * d->nkf) + ind_row(d->fp, 3 * d->nkf) +
                  ind_row(d->g, d->A * d->nkg);
  const bool stage = row > 0 && row <= IND_STAGE_ROW;
#define IND_CASE(N)                                                                            \
  case N:                                                                                      \
    if (stage)                                                                                 \
      hipLaunchKernelGGL((ind_cell_kernel<N, true>), dim3((d->nC + 63) / 64), dim3(64),        \
                         64 * row * sizeof(double), stream, *d, x, xp, out);                   \
    else                                                                                       \
      hipLaunchKernelGGL((ind_cell_kernel<N, false>), dim3((d->nC + 127) / 128), dim3(128), 0, \
                         stream, *d, x, xp, out);                                              \
    if (nF > 0)                                                                                \
      hipLaunchKernelGGL((ind_facet_kernel<N>), dim3((nF + 127) / 128), dim3(128), 0, stream,  \
                         *d, x, xp, fac, nF, tmp);                                             \
    break;
  switch (d->A) {
    IND_CASE(1) IND_CASE(2) IND_CASE(3) IND_CASE(4) IND_CASE(5) IND_CASE(6) IND_CASE(7)
    IND_CASE(8)
    default: break;
  }
#undef IND_CASE
  if (nF > 0) {
    hipLaunchKernelGGL(ind_gather_kernel, dim3((d->nC + 255) / 256), dim3(256), 0, stream,
                       d->nC, cell_f, (const double*)tmp, nF, out);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    char m[300];
    snprintf(m, sizeof(m), "%s: %s", who, hipGetErrorString(e));
    mpet_set_error(m);
    return ERR_HIP;
  }
  return OK;
}

static bool indicators_args_ok(const MpetIndDesc* d, const double* x, const double* xp,
                               const double* out, const int* fac, int nF, const int* cell_f) {
  return d && x && xp && out && d->coords && d->cells && d->cell_p2 && d->nC >= 1 &&
         d->A >= 1 && d->A <= MPET_MAXF && d->nq >= 1 && d->qbary && d->qw && d->dt > 0.0 &&
         !((d->f || d->fp) && (!d->Lf || d->nkf < 1)) && !(d->g && (!d->Lg || d->nkg < 1)) &&
         nF >= 0 && !(nF > 0 && (!fac || !cell_f));
}

extern "C" int mpet_error_indicators(const MpetIndDesc* d, const double* x, const double* xp,
                                     const int* fac, int nF, const int* cell_f, double* tmp,
                                     double* out, hipStream_t stream) {
  if (!indicators_args_ok(d, x, xp, out, fac, nF, cell_f) || (nF > 0 && !tmp)) {
    mpet_set_error("mpet_error_indicators: invalid argument");
    return ERR_INVALID;
  }
  return launch_indicators(d, x, xp, fac, nF, cell_f, tmp, out, stream,
                           "mpet_error_indicators");
}

// ---------------------------------------------------------------------------
// Allocation-free variant: the facet values (3 doubles per interior facet,
// the tmp workspace above) live in a file-scope device array, one copy per
// GPU for the life of the process.  Every facet value is written by the facet
// kernel before the gather reads it, so nothing needs clearing between
// calls; calls that overlap on one GPU share the array and race.
// ---------------------------------------------------------------------------
static __device__ __align__(256) double scratch[3ll * MPET_NOALLOC_MAX_FACETS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch[kMaxDevices] = {};
}  // namespace

// Device address of this GPU's copy of scratch, looked up once per device
// (with that device current) and kept.  The array's name is a host-side
// stand-in; only this address may be passed to kernels.
static int scratch_address(double** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    mpet_set_error("mpet_error_indicators_noalloc: no current device");
    return ERR_HIP;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      char m[300];
      snprintf(m, sizeof(m), "mpet_error_indicators_noalloc: hipGetSymbolAddress: %s",
               hipGetErrorString(e));
      mpet_set_error(m);
      return ERR_HIP;
    }
    g_scratch[dev] = (double*)p;
  }
  *out = g_scratch[dev];
  return OK;
}

extern "C" int mpet_error_indicators_noalloc(const MpetIndDesc* d, const double* x,
                                             const double* xp, const int* fac, int nF,
                                             const int* cell_f, double* out,
                                             hipStream_t stream) {
  if (!indicators_args_ok(d, x, xp, out, fac, nF, cell_f)) {
    mpet_set_error("mpet_error_indicators_noalloc: invalid argument");
    return ERR_INVALID;
  }
  if (nF > MPET_NOALLOC_MAX_FACETS) {
    char m[200];
    snprintf(m, sizeof(m),
             "mpet_error_indicators_noalloc: %d interior facets exceed the maximum %d "
             "(use mpet_error_indicators with a workspace)",
             nF, (int)MPET_NOALLOC_MAX_FACETS);
    mpet_set_error(m);
    return ERR_INVALID;
  }
  double* tmp = nullptr;
  if (nF > 0) {
    const int rc = scratch_address(&tmp);
    if (rc) return rc;
  }
  return launch_indicators(d, x, xp, fac, nF, cell_f, tmp, out, stream,
                           "mpet_error_indicators_noalloc");
}
