// coeff.hip -- what a change of the coefficients costs: the power-law viscosity
// at the quadrature points and the diagonal of A11, any mesh, one lane per
// element (see lane.h).
#include "lane_geom.h"

namespace ptmf {
namespace {

// ---------------------------------------------------------------------------
// diag(A11): d[3n+c] = sum_q w detJ eta (|grad N_n|^2 + (d_c N_n)^2), Dirichlet
// rows 1 (MFStokesWrapper_diagA11, stokes_operators_mf.c:67-131 with
// MatMultMF_Stokes_MixedFEM3d_diagB11, stokes_q2p1_mf_operators_diag_def.c:120-205).
//
// With T_c = sum_q w detJ eta (d_c N_n)^2 the entry is T_c + T_0 + T_1 + T_2.
// d_c N_n is a combination of the three reference derivatives, so T_c is the
// sum of six products of 1-D tables (squares of B and D and their product)
// contracted with h A[c][i] A[c][j], h = w eta / detJ, A the adjugate: 2,700
// operations an element by sum factorisation where 27 x 27 gradients take
// 20,000.  Bound by instruction issue at one wave per SIMD (6,500 FP64
// instructions a layer, 3,500 of them the geometry): 48^3 in 56 us and 9 us of
// faces, and no fill or Dirichlet pass; eight passes over element classes, 27
// lanes per element, took 230 us.
// ---------------------------------------------------------------------------
struct DiagTabs {
  double t[3][3][3];  // [BB, DD, DB][point][node]
  constexpr DiagTabs() : t{} {
    for (int a = 0; a < 3; a++)
      for (int i = 0; i < 3; i++) {
        t[0][a][i] = kB[a][i] * kB[a][i];
        t[1][a][i] = kD[a][i] * kD[a][i];
        t[2][a][i] = 2.0 * kD[a][i] * kB[a][i];
      }
  }
};
constexpr DiagTabs kDiag;
// tables of the products (0,0) (1,1) (2,2) (0,1) (0,2) (1,2) per direction; the
// factor 2 of a mixed product sits in the second of its DB tables
constexpr int kDiagTab[3][6] = {{1, 0, 0, 2, 2, 0}, {0, 1, 0, 2, 0, 2}, {0, 0, 1, 0, 2, 2}};

struct DiagOp {
  static constexpr LaneBC kBC = kLaneOne;
  const double *eta;  // [27][nel]
  const double *ek_;  // of the layer's first element in the tile
  long nel;
  unsigned oe;
  bool live;
  double et[9];

  __device__ __forceinline__ void begin(const TileArgs &a, const LaneTile &q, int ek) {
    ek_ = eta + q.tb.x0 + (long)a.mx * (q.tb.y0 + (long)a.my * ek);
    oe = q.cx + (unsigned)a.mx * q.cy;
    live = q.live;
  }
  __device__ __forceinline__ void frame(const double *, const double *, const double *) const {}
  template <int c>
  __device__ __forceinline__ void load() {
#pragma unroll
    for (int p = 0; p < 9; p++) et[p] = (ek_ + (9 * c + p) * nel)[oe];
  }
  template <int c>
  __device__ __forceinline__ void plane(double X[3][9], double Z[3][9], double out[3][3][9]) {
#pragma unroll
    for (int p = 0; p < 9; p++) et[p] = live ? et[p] : 0.0;
#pragma unroll
    for (int l = 0; l < 3; l++) {
      // the geometry is formed again for each component: 54 positions and
      // derivatives are kept in place of 162 metric terms
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int p = 0; p < 9; p++) {
          asm volatile("" : "+v"(X[d][p]));
          asm volatile("" : "+v"(Z[d][p]));
        }
      double g[3][9];  // contracted in x and y, by z table
#pragma unroll
      for (int t = 0; t < 3; t++)
#pragma unroll
        for (int n = 0; n < 9; n++) g[t][n] = 0.0;
#pragma unroll
      for (int b = 0; b < 3; b++) {
        double H[6][3];  // contracted in x
#pragma unroll
        for (int f = 0; f < 6; f++)
#pragma unroll
          for (int i = 0; i < 3; i++) H[f][i] = 0.0;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const int p = 3 * b + a;
          double A[3][3], m[6];
          plane_adjugate(a, b, X, Z, A);
          // detJ along the component's own row of the adjugate
          const double det = A[l][0] * cdot<double>(a, X[l][3 * b], X[l][3 * b + 1], X[l][3 * b + 2]) +
                             A[l][1] * cdot<double>(b, X[l][a], X[l][3 + a], X[l][6 + a]) + A[l][2] * Z[l][p];
          const double h = et[p] * (kW[a] * kW[b] * kW[c]) * recip<double>(det);
          const double h0 = h * A[l][0], h1 = h * A[l][1];
          m[0] = h0 * A[l][0];
          m[1] = h1 * A[l][1];
          m[2] = h * A[l][2] * A[l][2];
          m[3] = h0 * A[l][1];
          m[4] = h0 * A[l][2];
          m[5] = h1 * A[l][2];
#pragma unroll
          for (int f = 0; f < 6; f++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
              constexpr double half = 0.5;
              const double w = (f == 3 || f == 4 ? half : 1.0) * kDiag.t[kDiagTab[0][f]][a][i];
              if (w != 0.0) H[f][i] += w * m[f];
            }
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int f = 0; f < 6; f++)
#pragma unroll
          for (int j = 0; j < 3; j++) {
            const double w = (f == 5 ? 0.5 : 1.0) * kDiag.t[kDiagTab[1][f]][b][j];
            if (w == 0.0) continue;
#pragma unroll
            for (int i = 0; i < 3; i++) g[kDiagTab[2][f]][3 * j + i] += w * H[f][i];
          }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int t = 0; t < 3; t++) {
          if (kDiag.t[t][c][k] == 0.0) continue;
#pragma unroll
          for (int n = 0; n < 9; n++) out[k][l][n] += kDiag.t[t][c][k] * g[t][n];
        }
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int n = 0; n < 9; n++) asm volatile("" : "+v"(out[k][l][n]));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // T_c -> T_c + T_0 + T_1 + T_2
  __device__ __forceinline__ void finish(double o[3][9]) const {
#pragma unroll
    for (int n = 0; n < 9; n++) {
      const double t = o[0][n] + o[1][n] + o[2][n];
#pragma unroll
      for (int l = 0; l < 3; l++) o[l][n] += t;
    }
  }
};

// ---------------------------------------------------------------------------
// Strain-rate-dependent viscosity at the quadrature points:
// eta = clip(B * max(eII, 1e-17)^(1/n - 1)), eII = sqrt(0.5 D:D), D = sym(grad u)
// (ComputeStrainRate3d / ComputeSecondInvariant3d, stokes_rheology_vp_std.c:85-148;
// the VISCOUS_ARRHENIUS_2 power law, stokes_rheology_vp_std.c:437-461, with the
// prefactor B per quadrature point).  Element-major input B and output eta.
//
// The A21 kernel's march (see couple.hip).  The invariants of the 27 points
// stay in registers; B comes in, and eta goes out, in memory order through the
// one plane slot that is free by then.  Bound by instruction issue, half of it
// in pow: 48^3 in 75 us, 27 lanes per element took 178 us.
// ---------------------------------------------------------------------------
template <int c>
__device__ __forceinline__ void strain_plane(const double X[3][9], const double XZ[3][9], const double U[3][9],
                                             const double UZ[3][9], double e2[9]) {
#pragma unroll
  for (int b = 0; b < 3; b++)
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int p = 3 * b + a;
      double A[3][3], L[3][3];  // L[l][k] = detJ d u_l / d x_k
      plane_adjugate(a, b, X, XZ, A);
      const double det = A[0][0] * cdot<double>(a, X[0][3 * b], X[0][3 * b + 1], X[0][3 * b + 2]) +
                         A[0][1] * cdot<double>(b, X[0][a], X[0][3 + a], X[0][6 + a]) + A[0][2] * XZ[0][p];
#pragma unroll
      for (int l = 0; l < 3; l++) {
        const double g0 = cdot<double>(a, U[l][3 * b], U[l][3 * b + 1], U[l][3 * b + 2]),
                     g1 = cdot<double>(b, U[l][a], U[l][3 + a], U[l][6 + a]), g2 = UZ[l][p];
#pragma unroll
        for (int k = 0; k < 3; k++) L[l][k] = A[k][0] * g0 + A[k][1] * g1 + A[k][2] * g2;
      }
      const double r = recip<double>(det);
      const double d0 = r * L[0][0], d1 = r * L[1][1], d2 = r * L[2][2], s01 = r * (L[0][1] + L[1][0]),
                   s02 = r * (L[0][2] + L[2][0]), s12 = r * (L[1][2] + L[2][1]);
      e2[p] = 0.5 * (d0 * d0 + d1 * d1 + d2 * d2) + 0.25 * (s01 * s01 + s02 * s02 + s12 * s12);
      asm volatile("" : "+v"(e2[p]));
      __builtin_amdgcn_sched_barrier(0);
    }
}

__global__ void __launch_bounds__(64)
    powerlaw_lane_kernel(TileArgs a, const double *__restrict__ xc, const double *__restrict__ u,
                         const double *__restrict__ B, double half_exp, double eta_min, double eta_max,
                         double *__restrict__ eta) {
  __shared__ double sm[2 * 6 * kLPlane + 6 * kOdd];
  static_assert(27 * 64 <= 6 * kLPlane, "an element tile's points fit a plane slot");
  const LaneTile q = lane_tile(a, (unsigned)xcd_tile(blockIdx.x, a.ntiles));
  const TileBox &tb = q.tb;
  double *const s1 = sm + 2 * 6 * kLPlane;
  const double org = lane_origin(a, q, xc);
  const double *const first = xc + 3 * lane_node(a, tb, 2 * tb.z0);
  PlaneRows r1, r2;
  {
    const long n = lane_node(a, tb, 2 * tb.z0);
    r2.load(q, a.X, xc + 3 * n, u + 3 * n);
    r2.store<kLPlane>(q, sm, org);
  }
  for (int kz = 0; kz < tb.nzt; kz++) {
    const int ek = tb.z0 + kz;
    double *const s0 = sm + (kz & 1) * 6 * kLPlane, *const s2 = sm + ((kz & 1) ^ 1) * 6 * kLPlane;
    const long n1 = lane_node(a, tb, 2 * ek + 1), n2 = n1 + a.XY;
    const long nc = n1 + a.X * (2 * q.cy + 1) + 2 * q.cx + 1;  // the element's centre
    double ctr[6];
    r1.load(q, a.X, xc + 3 * n1, u + 3 * n1);
    r2.load(q, a.X, xc + 3 * n2, u + 3 * n2);
#pragma unroll
    for (int f = 0; f < 3; f++) {
      ctr[f] = xc[3 * nc + f] - first[f];
      ctr[3 + f] = u[3 * nc + f];
    }
    r1.store<kOdd>(q, s1, org);
    r2.store<kLPlane>(q, s2, org);
    __syncthreads();
    double X[3][9], XZ[3][9], U[3][9], UZ[3][9], e2[3][9];
    int lq = q.li;
    auto part = [&](auto c) {
      constexpr int C = decltype(c)::value;
      asm volatile("" : "+v"(lq));
      plane_fields<C, kOdd>(s0 + lq, s1 + lq, s2 + lq, X, XZ, ctr);
      plane_fields<C, kOdd>(s0 + lq + 3 * kLPlane, s1 + lq + 3 * kOdd, s2 + lq + 3 * kLPlane, U, UZ, ctr + 3);
      strain_plane<C>(X, XZ, U, UZ, e2[C]);
    };
    part(std::integral_constant<int, 0>());
    part(std::integral_constant<int, 1>());
    part(std::integral_constant<int, 2>());
    __syncthreads();
    double *const se = s0 + 27 * q.lane;
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int p = 0; p < 9; p++) se[9 * c + p] = e2[c][p];
    // the tile's rows of 8 elements: 216 consecutive values each
    const long e0 = 27 * (tb.x0 + (long)a.mx * (tb.y0 + (long)a.my * ek));
    const unsigned w = 27u * (unsigned)tb.nxt, rs = 27u * (unsigned)a.mx;
    auto at = [&](int i, unsigned &o) {  // value 64 i + lane of the tile: its place, and whether there is one
      const unsigned t = 64u * i + q.lane, row = t / 216u, col = t - 216u * row;
      o = rs * row + col;
      return col < w && (int)row < tb.nyt;
    };
    double v[27];  // in flight during the powers
#pragma unroll
    for (int i = 0; i < 27; i++) {
      unsigned o;
      const bool in = at(i, o);
      v[i] = (B + e0)[in ? o : 0u];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 3
    for (int p = 0; p < 27; p++) {
      double s = se[p];
      if (s < 1.0e-34) s = 1.0e-34;  // e_II >= 1e-17
      se[p] = pow(s, half_exp);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 27; i++) {
      unsigned o;
      const double t = v[i] * s0[64 * i + q.lane];
      if (at(i, o)) (eta + e0)[o] = fmin(fmax(t, eta_min), eta_max);
    }
    __syncthreads();
  }
}

}  // namespace

// Measured, 27 lanes and one lane: one element 22 and 35 us, 2^3 76 and 37, 48^3 233
// and 70; 1 x 1 x 5000 37 and 117, 256 x 1 x 256 143 and 178, 128 x 1 x 128 67 and
// 61, 512 x 2 x 64 163 and 104.
static bool diag_lane(const Box &b, TileArgs &a) { return node_lane_plan(b, 14.0, 8.0, 1.5, 8.5, 19.6, a); }

bool a11_diag_lane(const Box &b) {
  TileArgs a;
  return diag_lane(b, a);
}

int launch_a11_diag(const ptmf_op_s *op, double *d) {
  TileArgs a;
  if (!diag_lane(op->box, a)) return launch_a11_diag_elems(op, d);
  DiagOp g{};
  g.eta = op->d64.eta;
  g.nel = op->box.nel;
  return launch_node_lane(op, a, g, d);
}

int launch_powerlaw(const ptmf_op_s *op, const double *u, const double *B, double nexp, double eta_min,
                    double eta_max, double *eta) {
  const double half_exp = 0.5 * (1.0 / nexp - 1.0);
  double layers;
  const TileArgs a = lane_args(op->box, 1024, 0.2, &layers);
  // In microseconds, 27 lanes per element take 14.5 and 1.33 per thousand elements,
  // the lane kernel 8 and 27.3 per layer that a wave marches through, however
  // much of its 8 x 8 tile the box fills.  Measured, 27 lanes and one lane:
  // 8^3 17 and 40, 24^3 33 and 41, 32^3 57 and 43, 48^3 160 and 77; 256 x 1 x 256
  // 100 and 234, 512 x 2 x 64 101 and 127, 17 x 17 x 300 129 and 101.
  const bool lane = 8.0 + 27.3 * layers < 14.5 + 1.33e-3 * (double)op->box.nel;
  if (!lane || a.ntiles >= (1L << 31) || !lane_fits(op->box))
    return launch_powerlaw_elems(op, u, B, half_exp, eta_min, eta_max, eta);
  powerlaw_lane_kernel<<<dim3((unsigned)a.ntiles), dim3(64), 0, op->stream>>>(a, op->d64.coords, u, B, half_exp,
                                                                             eta_min, eta_max, eta);
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

}  // namespace ptmf
