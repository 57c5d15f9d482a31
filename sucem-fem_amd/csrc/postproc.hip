// Post-processing of a solved field on the device: the power flux through the
// mesh boundary and the near-to-far-field transform (NTFF), replacing the DOLFIN
// functionals of PostProcessing/power_flux.py:52-133,
// PostProcessing/surface_ntff.py:36-155 and PostProcessing/variational_ntff.py:64-131.
//
// Surface terms: one thread per (boundary face, quadrature point) evaluates E and
// curl E from the DOF vector (covariant Piola map of the reference basis) and
// stores the sample; the flux and the far-field potentials are then block sums
// over the samples, one grid row per direction.  Partial sums go to the host in
// block order, so every result is deterministic.
//
// Variational terms: the free-space functional <curl E, curl g> - k0^2 <E, g> over
// the cells that touch the boundary through an edge, with g supported on the
// boundary DOFs.  W_c = (S_e - k0^2 T_e) E_c is formed once per marked cell; each
// direction then needs only g at the boundary DOFs (nodal functionals of the
// testing field evaluated at the DOF points).
#include <cmath>
#include <vector>

#include "geom.hpp"
#include "internal.hpp"
#include "kernels.hpp"

namespace sucem {
namespace {

constexpr int TB = 256;
constexpr int QN = 5;            // collapsed Gauss rule, QN^2 points per face
constexpr int NQ = QN * QN;

__constant__ int c_pfaces[4][3] = {{1, 2, 3}, {0, 2, 3}, {0, 1, 3}, {0, 1, 2}};
__constant__ int c_pedges[6][2] = {{2, 3}, {1, 3}, {1, 2}, {0, 3}, {0, 2}, {0, 1}};
__constant__ int c_face_edges[4][3] = {{0, 1, 2}, {0, 3, 4}, {1, 3, 5}, {2, 4, 5}};
__constant__ int c_psym[6][2] = {{0, 0}, {1, 1}, {2, 2}, {0, 1}, {0, 2}, {1, 2}};

struct Sample {
  double w;          // quadrature weight x 2 x face area
  double p[3];       // physical point
  double n[3];       // outward unit normal
  double2 E[3];      // field
  double2 H[3];      // curl E (divided by mu_r when requested)
};

// Gauss-Legendre nodes and weights on [0, 1] (Newton on P_n).
void gauss01(int n, double* x, double* w) {
  for (int i = 0; i < n; ++i) {
    double z = std::cos(M_PI * (i + 0.75) / (n + 0.5));
    double dp = 1.0;
    for (int it = 0; it < 100; ++it) {
      double p0 = 1.0, p1 = z;
      for (int k = 2; k <= n; ++k) {
        double p2 = ((2.0 * k - 1.0) * z * p1 - (k - 1.0) * p0) / k;
        p0 = p1;
        p1 = p2;
      }
      dp = n * (z * p1 - p0) / (z * z - 1.0);
      double dz = p1 / dp;
      z -= dz;
      if (std::fabs(dz) < 1e-16) break;
    }
    x[i] = (1.0 - z) / 2.0;
    w[i] = 1.0 / ((1.0 - z * z) * dp * dp);   // 2/((1-z^2)P'^2) on [-1,1], halved
  }
}

// (s, t, w) of the collapsed rule on the reference triangle (weights sum to 1/2).
std::vector<double> triangle_rule() {
  double x[QN], w[QN];
  gauss01(QN, x, w);
  std::vector<double> r;
  for (int i = 0; i < QN; ++i)
    for (int j = 0; j < QN; ++j) {
      r.push_back(x[i] * (1.0 - x[j]));
      r.push_back(x[j]);
      r.push_back(w[i] * w[j] * (1.0 - x[j]));
    }
  return r;
}

__global__ void k_samples(int64_t nbf, const double* xyz, const int32_t* cells,
                          const int32_t* bf_cell, const int32_t* bf_local,
                          const int32_t* cell_dofs, const double* ref_basis, int nloc,
                          const double* rule, const double2* x, const double* inv_mu,
                          Sample* out) {
  __shared__ double rb[2 * 20 * 30];   // every sample reads all of the basis and its curl
  for (int k = threadIdx.x; k < 2 * nloc * 30; k += blockDim.x) rb[k] = ref_basis[k];
  __syncthreads();
  const int64_t total = nbf * NQ;
  for (int64_t id = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; id < total;
       id += (int64_t)gridDim.x * blockDim.x) {
    const int64_t f = id / NQ;
    const int q = (int)(id % NQ);
    const int64_t c = bf_cell[f];
    const int lf = bf_local[f];
    const int32_t* cell = cells + 4 * c;
    double J[3][3], Ji[3][3], det;
    cell_jacobian(xyz, cell, J, det, Ji);
    const double* P = xyz + 3 * (int64_t)cell[c_pfaces[lf][0]];
    const double* Q = xyz + 3 * (int64_t)cell[c_pfaces[lf][1]];
    const double* R = xyz + 3 * (int64_t)cell[c_pfaces[lf][2]];
    const double* O = xyz + 3 * (int64_t)cell[lf];   // the vertex opposite the face
    double e1[3], e2[3], n[3];
    for (int k = 0; k < 3; ++k) { e1[k] = Q[k] - P[k]; e2[k] = R[k] - P[k]; }
    n[0] = e1[1] * e2[2] - e1[2] * e2[1];
    n[1] = e1[2] * e2[0] - e1[0] * e2[2];
    n[2] = e1[0] * e2[1] - e1[1] * e2[0];
    const double a2 = sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    for (int k = 0; k < 3; ++k) n[k] /= a2;
    if (n[0] * (O[0] - P[0]) + n[1] * (O[1] - P[1]) + n[2] * (O[2] - P[2]) > 0)
      for (int k = 0; k < 3; ++k) n[k] = -n[k];
    const double s = rule[3 * q], t = rule[3 * q + 1];
    Sample smp;
    smp.w = rule[3 * q + 2] * a2;
    for (int k = 0; k < 3; ++k) {
      smp.p[k] = P[k] + s * e1[k] + t * e2[k];
      smp.n[k] = n[k];
    }
    const double* x0 = xyz + 3 * (int64_t)cell[0];
    double d[3] = {smp.p[0] - x0[0], smp.p[1] - x0[1], smp.p[2] - x0[2]};
    double xh[3];
    for (int a = 0; a < 3; ++a) xh[a] = Ji[a][0] * d[0] + Ji[a][1] * d[1] + Ji[a][2] * d[2];
    const double mono[10] = {1.0,           xh[0],         xh[1],         xh[2],
                             xh[0] * xh[0], xh[0] * xh[1], xh[0] * xh[2], xh[1] * xh[1],
                             xh[1] * xh[2], xh[2] * xh[2]};
    double2 Eh[3], Ch[3];
    for (int k = 0; k < 3; ++k) { Eh[k] = make_double2(0, 0); Ch[k] = make_double2(0, 0); }
    const double* rcurl = rb + nloc * 30;
    for (int i = 0; i < nloc; ++i) {
      const double2 xi = x[cell_dofs[c * nloc + i]];
      for (int dd = 0; dd < 3; ++dd) {
        double bv = 0, cv = 0;
        for (int m = 0; m < 10; ++m) {
          bv += rb[(i * 3 + dd) * 10 + m] * mono[m];
          cv += rcurl[(i * 3 + dd) * 10 + m] * mono[m];
        }
        Eh[dd].x += bv * xi.x; Eh[dd].y += bv * xi.y;
        Ch[dd].x += cv * xi.x; Ch[dd].y += cv * xi.y;
      }
    }
    const double hs = (inv_mu ? inv_mu[c] : 1.0) / det;
    for (int a = 0; a < 3; ++a) {
      // E = J^-T E^, curl E = J C^ / det J
      smp.E[a] = make_double2(Ji[0][a] * Eh[0].x + Ji[1][a] * Eh[1].x + Ji[2][a] * Eh[2].x,
                              Ji[0][a] * Eh[0].y + Ji[1][a] * Eh[1].y + Ji[2][a] * Eh[2].y);
      smp.H[a] = make_double2(hs * (J[a][0] * Ch[0].x + J[a][1] * Ch[1].x + J[a][2] * Ch[2].x),
                              hs * (J[a][0] * Ch[0].y + J[a][1] * Ch[1].y + J[a][2] * Ch[2].y));
    }
    out[id] = smp;
  }
}

// w n . (E_r x (-H_i) + E_i x H_r), summed per block
__global__ __launch_bounds__(TB) void k_flux(int64_t ns, const Sample* smp, double* part) {
  double acc = 0;
  for (int64_t i = blockIdx.x * (int64_t)TB + threadIdx.x; i < ns; i += (int64_t)gridDim.x * TB) {
    const Sample& s = smp[i];
    double a[3] = {s.E[0].x, s.E[1].x, s.E[2].x}, b[3] = {-s.H[0].y, -s.H[1].y, -s.H[2].y};
    double c[3] = {s.E[0].y, s.E[1].y, s.E[2].y}, d[3] = {s.H[0].x, s.H[1].x, s.H[2].x};
    double v = 0;
    for (int k = 0; k < 3; ++k) {
      const int k1 = (k + 1) % 3, k2 = (k + 2) % 3;
      v += s.n[k] * (a[k1] * b[k2] - a[k2] * b[k1] + c[k1] * d[k2] - c[k2] * d[k1]);
    }
    acc += s.w * v;
  }
  const double2 r = block_sum<TB>(make_double2(acc, 0.0));
  if (threadIdx.x == 0) part[blockIdx.x] = r.x;
}

__device__ inline void cross_c(const double n[3], const double2 v[3], double2 out[3]) {
  for (int k = 0; k < 3; ++k) {
    const int k1 = (k + 1) % 3, k2 = (k + 2) % 3;
    out[k] = make_double2(n[k1] * v[k2].x - n[k2] * v[k1].x, n[k1] * v[k2].y - n[k2] * v[k1].y);
  }
}

// Far-field sums S_d = sum_i v_i exp(j k0 p_i . r_d) of NC complex components v over points
// p_i, for every direction r_d (the projections on theta_hat and phi_hat are linear and
// taken from the sums afterwards).  A thread owns one direction and adds its share of the
// points, which the block stages in LDS, so a point is read once per 64 directions instead
// of once per direction, and what is left is the sincos and 4 NC FMAs per point and
// direction, bound by FP64 arithmetic.  The points go in P chunks, a chunk in four shares
// (i mod 4, one wave each: a wave reads one point, a broadcast); k_ff_few, for few
// directions, where most lanes of a wave would idle, has one thread per direction, chunk and
// share and the same sums in the same order, so that a direction's result does not depend
// on how many are asked for.  part[(q nd + d) 2 NC + k]: the sums of chunk q.
// 264,000 points, 181 directions: 597 us (one block row per direction) -> 110 us; the
// boundary DOFs' sums of the variational form, which ran over all cells, 783 -> 39 us.
// FF_FEW: a surface transform (79,200 points) of 4 / 16 / 17 / 32 / 48 / 181 directions takes
// 120 / 123 / 137 / 139 / 159 / 328 us with k_ff_few and 134 / 136 / 137 / 136 / 138 / 209 us
// with k_ff_sums.
constexpr int FF_TILE = 64, FF_SL = 4, FF_DL = TB / FF_SL, FF_CHUNKS = 1024, FF_FEW = 16;

// NC = 6: w (n x H), w (n x E) of the boundary samples
struct SurfacePoints {
  static constexpr int NC = 6;
  const Sample* smp;
  __device__ void load(int64_t i, double p[3], double2 v[NC]) const {
    const Sample& s = smp[i];
    double2 h[3], e[3];
    cross_c(s.n, s.H, h);
    cross_c(s.n, s.E, e);
    for (int k = 0; k < 3; ++k) {
      p[k] = s.p[k];
      v[k] = make_double2(s.w * h[k].x, s.w * h[k].y);
      v[3 + k] = make_double2(s.w * e[k].x, s.w * e[k].y);
    }
  }
};

// NC = 3: t W of the boundary DOFs of the cells at the boundary (dual point p, tangent t)
struct SkinEntry {
  double p[3], t[3];
  double2 w;
  int64_t dof;
};
struct SkinPoints {
  static constexpr int NC = 3;
  const SkinEntry* ent;
  __device__ void load(int64_t i, double p[3], double2 v[NC]) const {
    const SkinEntry& s = ent[i];
    for (int k = 0; k < 3; ++k) {
      p[k] = s.p[k];
      v[k] = make_double2(s.t[k] * s.w.x, s.t[k] * s.w.y);
    }
  }
};

template <typename PTS>
__global__ __launch_bounds__(TB) void k_ff_sums(int64_t np, PTS pts, int64_t nd, int P,
                                                const double* __restrict__ dirs, double k0,
                                                double* __restrict__ part) {
  constexpr int NC = PTS::NC;
  __shared__ double sp[3][FF_TILE];
  __shared__ double2 sv[NC][FF_TILE];
  __shared__ double2 red[TB];
  const int64_t group = blockIdx.x / P;
  const int q = (int)(blockIdx.x % P);
  const int dl = threadIdx.x % FF_DL, slice = threadIdx.x / FF_DL;
  const int64_t d = group * FF_DL + dl;
  const double* dr = dirs + 9 * (d < nd ? d : nd - 1);
  const double rx = k0 * dr[0], ry = k0 * dr[1], rz = k0 * dr[2];
  double2 acc[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) acc[k] = make_double2(0, 0);
  const int64_t chunk = (np + P - 1) / P;
  const int64_t i0 = q * chunk, i1 = i0 + chunk < np ? i0 + chunk : np;
  for (int64_t t0 = i0; t0 < i1; t0 += FF_TILE) {
    const int cnt = (int)(i1 - t0 < FF_TILE ? i1 - t0 : FF_TILE);
    __syncthreads();
    if (threadIdx.x < cnt) {
      double p[3];
      double2 v[NC];
      pts.load(t0 + threadIdx.x, p, v);
      for (int k = 0; k < 3; ++k) sp[k][threadIdx.x] = p[k];
      for (int k = 0; k < NC; ++k) sv[k][threadIdx.x] = v[k];
    }
    __syncthreads();
    for (int i = slice; i < cnt; i += FF_SL) {
      double sn, cs;
      sincos(rx * sp[0][i] + ry * sp[1][i] + rz * sp[2][i], &sn, &cs);
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        const double2 v = sv[k][i];
        acc[k].x += cs * v.x - sn * v.y;
        acc[k].y += cs * v.y + sn * v.x;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NC; ++k) {   // the shares, in order
    __syncthreads();
    red[threadIdx.x] = acc[k];
    __syncthreads();
    if (threadIdx.x < FF_DL && d < nd) {
      double2 s = red[threadIdx.x];
      for (int j = 1; j < FF_SL; ++j) {
        s.x += red[j * FF_DL + threadIdx.x].x;
        s.y += red[j * FF_DL + threadIdx.x].y;
      }
      double* out = part + ((q * nd + d) * NC + k) * 2;
      out[0] = s.x;
      out[1] = s.y;
    }
  }
}

template <typename PTS>
__global__ __launch_bounds__(TB) void k_ff_few(int64_t np, PTS pts, int nd, int P,
                                               const double* __restrict__ dirs, double k0,
                                               double* __restrict__ part) {
  constexpr int NC = PTS::NC;
  const int64_t t = blockIdx.x * (int64_t)TB + threadIdx.x;
  const int slice = (int)(t % FF_SL);
  const int64_t dq = t / FF_SL;
  const int d = (int)(dq % nd);
  const int64_t q = dq / nd;
  const bool live = q < P;
  const double* dr = dirs + 9 * d;
  const double rx = k0 * dr[0], ry = k0 * dr[1], rz = k0 * dr[2];
  double2 acc[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) acc[k] = make_double2(0, 0);
  const int64_t chunk = (np + P - 1) / P;
  const int64_t i0 = q * chunk, i1 = !live ? i0 : (i0 + chunk < np ? i0 + chunk : np);
  for (int64_t i = i0 + slice; i < i1; i += FF_SL) {
    double p[3];
    double2 v[NC];
    pts.load(i, p, v);
    double sn, cs;
    sincos(rx * p[0] + ry * p[1] + rz * p[2], &sn, &cs);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      acc[k].x += cs * v[k].x - sn * v[k].y;
      acc[k].y += cs * v[k].y + sn * v[k].x;
    }
  }
  const int lane0 = (threadIdx.x & 63) - slice;   // the four shares are neighbouring lanes
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    double2 s = make_double2(__shfl(acc[k].x, lane0), __shfl(acc[k].y, lane0));
    for (int j = 1; j < FF_SL; ++j) {
      s.x += __shfl(acc[k].x, lane0 + j);
      s.y += __shfl(acc[k].y, lane0 + j);
    }
    if (live && slice == 0) {
      double* out = part + ((q * nd + d) * NC + k) * 2;
      out[0] = s.x;
      out[1] = s.y;
    }
  }
}

// out[i] = sum over the P chunks of part[q m + i], in order
__global__ __launch_bounds__(64) void k_ff_total(int64_t m, int P, const double* __restrict__ part,
                                                 double* __restrict__ out) {
  const int64_t i = blockIdx.x * (int64_t)64 + threadIdx.x;
  if (i >= m) return;
  double s = 0;
  int q = 0;
  constexpr int U = 32;
  for (; q + U <= P; q += U) {   // U loads in flight
    double v[U];
#pragma unroll
    for (int j = 0; j < U; ++j) v[j] = part[(q + j) * m + i];
#pragma unroll
    for (int j = 0; j < U; ++j) s += v[j];
  }
  for (; q < P; ++q) s += part[q * m + i];
  out[i] = s;
}

__global__ void k_mark_edges(int64_t nbf, const int32_t* bf_cell, const int32_t* bf_local,
                             const int32_t* cell_edges, uint8_t* edge_on_b) {
  for (int64_t f = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; f < nbf;
       f += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = bf_cell[f];
    for (int k = 0; k < 3; ++k) edge_on_b[cell_edges[6 * c + c_face_edges[bf_local[f]][k]]] = 1;
  }
}

__global__ void k_mark_cells(int64_t nc, const int32_t* cell_edges, const uint8_t* edge_on_b,
                             uint8_t* cell_on_b) {
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < nc;
       c += (int64_t)gridDim.x * blockDim.x) {
    uint8_t m = 0;
    for (int k = 0; k < 6; ++k) m |= edge_on_b[cell_edges[6 * c + k]];
    cell_on_b[c] = m;
  }
}

// Nodal functional of local DOF i: point and (unnormalised) tangent from the cell vertices.
__device__ inline void dof_point(const double* xyz, const int32_t* cell, int order, int i,
                                 double p[3], double t[3]) {
  if (order == 1 || i < 12) {
    const int l = order == 1 ? i : i / 2;
    const double s = order == 1 ? 0.5 : ((i & 1) ? 2.0 / 3.0 : 1.0 / 3.0);
    const double* A = xyz + 3 * (int64_t)cell[c_pedges[l][0]];
    const double* B = xyz + 3 * (int64_t)cell[c_pedges[l][1]];
    for (int k = 0; k < 3; ++k) { t[k] = B[k] - A[k]; p[k] = A[k] + s * t[k]; }
  } else {
    const int f = (i - 12) / 2;
    const double* P = xyz + 3 * (int64_t)cell[c_pfaces[f][0]];
    const double* Q = xyz + 3 * (int64_t)cell[c_pfaces[f][1]];
    const double* R = xyz + 3 * (int64_t)cell[c_pfaces[f][2]];
    const double* T = (i & 1) ? R : Q;
    for (int k = 0; k < 3; ++k) { p[k] = (P[k] + Q[k] + R[k]) / 3.0; t[k] = T[k] - P[k]; }
  }
}

// flag[c nloc + i] = 1 for the boundary DOFs of the marked cells
__global__ void k_skin_flags(int64_t nc, int nloc, const uint8_t* cell_on_b,
                             const int32_t* cell_dofs, const uint8_t* bdof, int32_t* flag) {
  for (int64_t id = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; id < nc * nloc;
       id += (int64_t)gridDim.x * blockDim.x)
    flag[id] = cell_on_b[id / nloc] && bdof[cell_dofs[id]] ? 1 : 0;
}

__global__ void k_skin_ids(int64_t n, const int32_t* flag, const int32_t* pos, int32_t* ids) {
  for (int64_t id = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; id < n;
       id += (int64_t)gridDim.x * blockDim.x)
    if (flag[id]) ids[pos[id]] = (int32_t)id;
}

// Entry of (cell c, local DOF i): W = sum_j (S_e - k0^2 T_e)_ij x_j with eps_r = mu_r = 1, the
// DOF's dual point and tangent.
__global__ void k_skin_entries(int64_t ne, const int32_t* ids, const double* xyz,
                               const int32_t* cells, const int32_t* cell_dofs,
                               const double* ref_mass, const double* ref_stiff, int nloc,
                               int order, double k0, const double2* x, SkinEntry* out) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < ne;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = ids[e] / nloc;
    const int i = ids[e] % nloc;
    double J[3][3], Ji[3][3], det;
    cell_jacobian(xyz, cells + 4 * c, J, det, Ji);
    const double adet = fabs(det);
    double ct[6], cs[6];
    for (int k = 0; k < 6; ++k) {
      const int a = c_psym[k][0], b = c_psym[k][1];
      ct[k] = -k0 * k0 * adet * (Ji[a][0] * Ji[b][0] + Ji[a][1] * Ji[b][1] + Ji[a][2] * Ji[b][2]);
      cs[k] = (J[0][a] * J[0][b] + J[1][a] * J[1][b] + J[2][a] * J[2][b]) / adet;
    }
    double2 acc = make_double2(0, 0);
    for (int j = 0; j < nloc; ++j) {
      double kij = 0;
      for (int k = 0; k < 6; ++k)
        kij += cs[k] * ref_stiff[(k * nloc + i) * nloc + j] + ct[k] * ref_mass[(k * nloc + i) * nloc + j];
      const double2 xj = x[cell_dofs[c * nloc + j]];
      acc.x += kij * xj.x;
      acc.y += kij * xj.y;
    }
    SkinEntry s;
    dof_point(xyz, cells + 4 * c, order, i, s.p, s.t);
    s.w = acc;
    s.dof = cell_dofs[ids[e]];
    out[e] = s;
  }
}

// sum over the entries of conj(x_i) W
__global__ __launch_bounds__(TB) void k_flux_variational(int64_t ne, const SkinEntry* ent,
                                                         const double2* x, double* part) {
  double2 acc = make_double2(0, 0);
  for (int64_t e = blockIdx.x * (int64_t)TB + threadIdx.x; e < ne; e += (int64_t)gridDim.x * TB) {
    const double2 xi = x[ent[e].dof], w = ent[e].w;
    const double2 g = make_double2(xi.x, -xi.y);
    acc.x += g.x * w.x - g.y * w.y;
    acc.y += g.x * w.y + g.y * w.x;
  }
  const double2 r = block_sum<TB>(acc);
  if (threadIdx.x == 0) { part[2 * blockIdx.x] = r.x; part[2 * blockIdx.x + 1] = r.y; }
}

void directions(int64_t n, const double* theta, const double* phi, std::vector<double>& d) {
  d.resize(9 * n);
  for (int64_t i = 0; i < n; ++i) {
    const double st = std::sin(theta[i]), ct = std::cos(theta[i]);
    const double sp = std::sin(phi[i]), cp = std::cos(phi[i]);
    const double v[9] = {st * cp, st * sp, ct, ct * cp, ct * sp, -st, -sp, cp, 0.0};
    for (int k = 0; k < 9; ++k) d[9 * i + k] = v[k];
  }
}

void make_samples(Context* c, const Space* s, const void* x, bool use_mu, DBuf<Sample>& smp) {
  const std::vector<double> rule = triangle_rule();
  DBuf<double> drule(rule.size());
  h2d(c, drule.p, rule.data(), rule.size());
  smp.alloc((size_t)s->nbf * NQ);
  const Mesh* m = s->mesh;
  SUCEM_LAUNCH(k_samples, grid_for(s->nbf * NQ, TB, 4096), TB, 0, c->stream, s->nbf,
               m->xyz.p, m->cells.p, s->bf_cell.p, s->bf_local.p, s->cell_dofs.p,
               s->ref_basis.p, s->nloc, drule.p, (const double2*)x,
               use_mu ? m->inv_mu_r.p : nullptr, smp.p);
  c->sync();   // drule is released on return
}

// The boundary DOFs of the cells that touch the boundary through an edge, with their W.
struct Skin {
  int64_t n = 0;
  DBuf<SkinEntry> ent;
};

void make_skin(Context* c, const Space* s, const void* x, double k0, Skin& sk) {
  const Mesh* m = s->mesh;
  const int64_t total = m->nc * s->nloc;
  DBuf<uint8_t> edge_on_b(s->nE), cell_on_b(m->nc);
  DBuf<int32_t> flag(total), pos(total);
  SUCEM_HIP(hipMemsetAsync(edge_on_b.p, 0, s->nE, c->stream));
  SUCEM_LAUNCH(k_mark_edges, grid_for(s->nbf, TB, 4096), TB, 0, c->stream, s->nbf, s->bf_cell.p,
               s->bf_local.p, s->cell_edges.p, edge_on_b.p);
  SUCEM_LAUNCH(k_mark_cells, grid_for(m->nc, TB, 4096), TB, 0, c->stream, m->nc, s->cell_edges.p,
               edge_on_b.p, cell_on_b.p);
  SUCEM_LAUNCH(k_skin_flags, grid_for(total, TB, 8192), TB, 0, c->stream, m->nc, s->nloc,
               cell_on_b.p, s->cell_dofs.p, s->bdof.p, flag.p);
  exclusive_scan_i32(c, flag.p, pos.p, (size_t)total);
  int32_t last[2] = {0, 0};
  d2h(c, &last[0], pos.p + (total - 1), 1);
  d2h(c, &last[1], flag.p + (total - 1), 1);
  c->sync();
  sk.n = (int64_t)last[0] + last[1];
  if (sk.n == 0) return;
  DBuf<int32_t> ids(sk.n);
  SUCEM_LAUNCH(k_skin_ids, grid_for(total, TB, 8192), TB, 0, c->stream, total, flag.p, pos.p,
               ids.p);
  sk.ent.alloc(sk.n);
  SUCEM_LAUNCH(k_skin_entries, grid_for(sk.n, TB, 8192), TB, 0, c->stream, sk.n, ids.p, m->xyz.p,
               m->cells.p, s->cell_dofs.p, s->ref_mass.p, s->ref_stiff.p, s->nloc, s->order, k0,
               (const double2*)x, sk.ent.p);
}

// The far-field sums of every direction: out[d][2 NC] on the host (valid after the stream has
// been synchronised).  Directions go in groups whose chunk sums take at most 256 MB.
template <typename PTS>
void ff_sums(Context* c, int64_t np, PTS pts, int64_t nd, const double* dirs_d, double k0,
             std::vector<double>& out) {
  constexpr int NC = PTS::NC;
  out.assign((size_t)nd * 2 * NC, 0.0);
  if (np == 0) return;
  const int P = (int)std::min<int64_t>(FF_CHUNKS, (np + FF_TILE - 1) / FF_TILE);
  const int64_t most = (int64_t(256) << 20) / (int64_t)(P * 2 * NC * sizeof(double));
  DBuf<double> part((size_t)(std::min(nd, most) * P * 2 * NC)), tot((size_t)nd * 2 * NC);
  for (int64_t d0 = 0; d0 < nd; d0 += most) {
    const int64_t n = std::min(most, nd - d0), m = n * 2 * NC;
    if (n <= FF_FEW)
      SUCEM_LAUNCH((k_ff_few<PTS>), (unsigned)((n * P * FF_SL + TB - 1) / TB), TB, 0, c->stream,
                   np, pts, (int)n, P, dirs_d + 9 * d0, k0, part.p);
    else
      SUCEM_LAUNCH((k_ff_sums<PTS>), (unsigned)((n + FF_DL - 1) / FF_DL * P), TB, 0, c->stream,
                   np, pts, n, P, dirs_d + 9 * d0, k0, part.p);
    SUCEM_LAUNCH(k_ff_total, (unsigned)((m + 63) / 64), 64, 0, c->stream, m, P, part.p,
                 tot.p + d0 * 2 * NC);
  }
  d2h(c, out.data(), tot.p, out.size());
}

}  // namespace

double surface_flux(Context* c, const Space* s, const void* x, double k0, bool use_mu) {
  DBuf<Sample> smp;
  make_samples(c, s, x, use_mu, smp);
  const int64_t ns = s->nbf * NQ;
  const unsigned G = grid_for(ns, TB, 1024);
  DBuf<double> part(G);
  SUCEM_LAUNCH(k_flux, G, TB, 0, c->stream, ns, smp.p, part.p);
  std::vector<double> h(G);
  d2h(c, h.data(), part.p, G);
  c->sync();
  double sum = 0;
  for (unsigned i = 0; i < G; ++i) sum += h[i];
  return sum / k0 / kZ0;
}

void variational_flux(Context* c, const Space* s, const void* x, double k0, double out[2]) {
  Skin sk;
  make_skin(c, s, x, k0, sk);
  if (sk.n == 0) {
    out[0] = out[1] = 0.0;
    return;
  }
  const unsigned G = grid_for(sk.n, TB, 1024);
  DBuf<double> part(2 * (size_t)G);
  SUCEM_LAUNCH(k_flux_variational, G, TB, 0, c->stream, sk.n, sk.ent.p, (const double2*)x, part.p);
  std::vector<double> h(2 * (size_t)G);
  d2h(c, h.data(), part.p, h.size());
  c->sync();
  double sr = 0, si = 0;
  for (unsigned i = 0; i < G; ++i) { sr += h[2 * i]; si += h[2 * i + 1]; }
  // F = sum g W with g = j conj(x) / (k0 Z0); the flux is conj(F)
  const double fr = -si / (k0 * kZ0), fi = sr / (k0 * kZ0);
  out[0] = fr;
  out[1] = -fi;
}

void ntff(Context* c, const Space* s, const void* x, double k0, bool variational, int64_t n,
          const double* theta, const double* phi, double* E_ff) {
  std::vector<double> dirs;
  directions(n, theta, phi, dirs);
  DBuf<double> ddirs(dirs.size());
  h2d(c, ddirs.p, dirs.data(), dirs.size());
  DBuf<Sample> smp;
  make_samples(c, s, x, false, smp);
  const int64_t ns = s->nbf * NQ;
  std::vector<double> hs, hv;
  ff_sums(c, ns, SurfacePoints{smp.p}, n, ddirs.p, k0, hs);
  Skin sk;
  if (variational) {
    make_skin(c, s, x, k0, sk);
    ff_sums(c, sk.n, SkinPoints{sk.ent.p}, n, ddirs.p, k0, hv);
  }
  c->sync();
  // far-field factor j k0 exp(-j k0) / (4 pi)
  const double fr = k0 * std::sin(k0) / (4 * M_PI), fi = k0 * std::cos(k0) / (4 * M_PI);
  auto mul = [](double ar, double ai, double br, double bi, double& cr, double& ci) {
    cr = ar * br - ai * bi;
    ci = ar * bi + ai * br;
  };
  for (int64_t a = 0; a < n; ++a) {
    // (A.th, A.ph, B.th, B.ph) as complex pairs from the sums A = int e n x curl E and
    // B = int e n x E
    const double* dr = &dirs[9 * a];
    double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int ab = 0; ab < 2; ++ab)
      for (int v = 0; v < 2; ++v)
        for (int k = 0; k < 3; ++k)
          for (int z = 0; z < 2; ++z)
            acc[4 * ab + 2 * v + z] += dr[3 + 3 * v + k] * hs[((size_t)a * 6 + 3 * ab + k) * 2 + z];
    // N = j/(k0 Z0) A, L = -B (A = int e n x curl E, B = int e n x E)
    const double sN = 1.0 / (k0 * kZ0);
    const double Nth_r = -sN * acc[1], Nth_i = sN * acc[0];
    const double Nph_r = -sN * acc[3], Nph_i = sN * acc[2];
    const double Lth_r = -acc[4], Lth_i = -acc[5], Lph_r = -acc[6], Lph_i = -acc[7];
    double t_r, t_i, p_r, p_i;
    if (!variational) {
      // E_theta = -f (L_phi + Z0 N_theta), E_phi = f (L_theta - Z0 N_phi)
      mul(fr, fi, -(Lph_r + kZ0 * Nth_r), -(Lph_i + kZ0 * Nth_i), t_r, t_i);
      mul(fr, fi, Lth_r - kZ0 * Nph_r, Lth_i - kZ0 * Nph_i, p_r, p_i);
    } else {
      // sum of g_a W for the testing fields g_a = (j/k0) r x (a x r) exp(j k0 r.x),
      // a = theta_hat, phi_hat: r x (a x r) = a for unit r and a normal to it
      double v[4] = {0, 0, 0, 0};
      for (int q = 0; q < 2; ++q) {
        double sr = 0, si = 0;
        for (int k = 0; k < 3; ++k) {
          sr += dr[3 + 3 * q + k] * hv[((size_t)a * 3 + k) * 2];
          si += dr[3 + 3 * q + k] * hv[((size_t)a * 3 + k) * 2 + 1];
        }
        v[2 * q] = -si / k0;
        v[2 * q + 1] = sr / k0;
      }
      // E_theta = f (-L_phi + E_H_theta), E_phi = f (L_theta + E_H_phi)
      mul(fr, fi, -Lph_r + v[0], -Lph_i + v[1], t_r, t_i);
      mul(fr, fi, Lth_r + v[2], Lth_i + v[3], p_r, p_i);
    }
    E_ff[4 * a] = t_r;
    E_ff[4 * a + 1] = t_i;
    E_ff[4 * a + 2] = p_r;
    E_ff[4 * a + 3] = p_i;
  }
}

}  // namespace sucem
