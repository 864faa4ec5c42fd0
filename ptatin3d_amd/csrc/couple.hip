// couple.hip -- the pressure-velocity couplings B (A12) and B^T (A21) of the
// Q2-P1disc element, any mesh, one lane per element (see lane.h).
//
// Both need no division: with A = det(J) J^-1 the adjugate, w det(J) d_k N_n is
// w sum_j A[k][j] (dN_n / d xi_j) and w det(J) div u is w sum_jk A[k][j] (du_k /
// d xi_j).
#include <algorithm>

#include "lane_geom.h"

namespace ptmf {
namespace {

// The element's frame of the P1GRel pressure basis {1, (x - xb)_d / L_d}
// (element_utils_q2.c:183-224): the mean of its nodes and the lengths x14 -
// x12, y16 - y10, z22 - z4.  s0, s1, s2: node (0, 0) of the three planes.
// kP1: component stride of the middle plane; centre: its element centres, when
// they are not in the slot (kP1 < kLPlane)
template <int kP1 = kLPlane>
__device__ __forceinline__ void pressure_frame(const double *s0, const double *s1, const double *s2, double xb[3],
                                               double L[3], const double *centre = nullptr) {
#pragma unroll
  for (int d = 0; d < 3; d++) {
    double s = 0.0;
#pragma unroll
    for (int n = 0; n < 9; n++) {
      const int o = lane_off(n % 3, n / 3);
      s += s0[d * kLPlane + o] + (kP1 < kLPlane && n == 4 ? centre[d] : s1[d * kP1 + o]) + s2[d * kLPlane + o];
    }
    xb[d] = s * (1.0 / 27.0);
    __builtin_amdgcn_sched_barrier(0);
  }
  L[0] = s1[lane_off(2, 1)] - s1[lane_off(0, 1)];
  L[1] = s1[kP1 + lane_off(1, 2)] - s1[kP1 + lane_off(1, 0)];
  L[2] = s2[2 * kLPlane + lane_off(1, 1)] - s0[2 * kLPlane + lane_off(1, 1)];
  // finished here, not where they are first used
#pragma unroll
  for (int d = 0; d < 3; d++) {
    asm volatile("" : "+v"(xb[d]));
    asm volatile("" : "+v"(L[d]));
  }
}

// ---------------------------------------------------------------------------
// B p: yu[3n+c] = sum_q -w detJ (d_c N_n) p_h(x_q) (MFStokesWrapper_A12,
// stokes_operators_mf.c:788-856 with MatMultMF_Stokes_MixedFEM3d_A12,
// stokes_q2p1_mf_operators_def.c:423-516), Dirichlet velocity rows zero.
//
// Bound by instruction issue at one wave
// per SIMD (4,100 FP64 instructions a layer of 64 elements, two thirds of the
// kernel's): 64 x 48 x 40 in 44 us and 9 us of faces; eight passes over element
// classes, 27 lanes per element, took 290 us.
// ---------------------------------------------------------------------------
struct A12Op {
  static constexpr LaneBC kBC = kLaneZero;
  const double *p;
  double pc[4], xb[3], L[3];
  bool live;

  __device__ __forceinline__ void begin(const TileArgs &a, const LaneTile &q, int ek) {
    const double *pe = p + 4 * (q.tb.x0 + (long)a.mx * (q.tb.y0 + (long)a.my * ek)) + 4 * (q.cx + a.mx * q.cy);
#pragma unroll
    for (int i = 0; i < 4; i++) pc[i] = pe[i];
    live = q.live;
  }
  __device__ __forceinline__ void frame(const double *s0, const double *s1, const double *s2) {
    pressure_frame(s0, s1, s2, xb, L);
  }
  template <int c>
  __device__ __forceinline__ void load() {}
  __device__ __forceinline__ void finish(double (*)[9]) const {}
  template <int c>
  __device__ __forceinline__ void plane(const double X[3][9], double Z[3][9], double out[3][3][9]) {
    if (c == 0) {
      // (a lane past a partial tile must sum zeros)
      pc[0] = live ? pc[0] : 0.0;
#pragma unroll
      for (int d = 0; d < 3; d++) pc[1 + d] = live ? pc[1 + d] / L[d] : 0.0;
    }
    double W[3][9];
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int p = 0; p < 9; p++) W[l][p] = 0.0;
#pragma unroll
    for (int b = 0; b < 3; b++)
#pragma unroll
      for (int a = 0; a < 3; a++) {
        const int p = 3 * b + a;
        double A[3][3];
        plane_adjugate(a, b, X, Z, A);
        const double ph = pc[0] + pc[1] * (X[0][p] - xb[0]) + pc[2] * (X[1][p] - xb[1]) + pc[3] * (X[2][p] - xb[2]);
        const double t = -(kW[a] * kW[b] * kW[c]) * ph;
#pragma unroll
        for (int l = 0; l < 3; l++) {
          const double dv0 = t * A[l][0], dv1 = t * A[l][1];
          Z[l][p] = t * A[l][2];
#pragma unroll
          for (int r = 0; r < 3; r++) {
            if (a != 1 || r != 1) W[l][3 * b + r] += kC[a][r] * dv0;
            if (b != 1 || r != 1) W[l][3 * r + a] += kC[b][r] * dv1;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int l = 0; l < 3; l++)
      lane_field_t<double, c>(W[l], Z[l], kD[c][0], kD[c][1], kD[c][2], out[0][l], out[1][l], out[2][l]);
  }
};

// ---------------------------------------------------------------------------
// B^T u: yp[4e+i] = sum_q -w detJ NIp_i div u_h(x_q), u Dirichlet-masked
// (MFStokesWrapper_A21, stokes_operators_mf.c:858-933 with
// MatMultMF_Stokes_MixedFEM3d_A21, stokes_q2p1_mf_operators_def.c:517-538).
//
// No sums leave the element, so there are no windows and no faces.  Three
// plane slots of coordinates and velocity each, the middle plane's without the
// element centres (a lane loads its own), so that a wave's 40,608 B let four
// waves live on a CU.  A layer's rows are all in flight before the first is
// stored: one exposed latency a layer, in place of five slots that would leave
// two waves a CU.  Bound by instruction issue: 64 x 48 x 40 in 40 us (53 us at
// three waves a CU with the centres in the slots); 27 lanes per element with a
// reduction over them took 330 us.
// ---------------------------------------------------------------------------
template <int c>
__device__ __forceinline__ void a21_plane(const double X[3][9], const double XZ[3][9], const double U[3][9],
                                          const double UZ[3][9], const double xb[3], double acc[4]) {
#pragma unroll
  for (int b = 0; b < 3; b++)
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int p = 3 * b + a;
      double A[3][3];
      plane_adjugate(a, b, X, XZ, A);
      double div = 0.0;
#pragma unroll
      for (int k = 0; k < 3; k++)
        div += cdot<double>(a, U[k][3 * b], U[k][3 * b + 1], U[k][3 * b + 2]) * A[k][0] +
               cdot<double>(b, U[k][a], U[k][3 + a], U[k][6 + a]) * A[k][1] + UZ[k][p] * A[k][2];
      const double t = -(kW[a] * kW[b] * kW[c]) * div;
      acc[0] += t;
#pragma unroll
      for (int d = 0; d < 3; d++) acc[1 + d] += t * (X[d][p] - xb[d]);
      __builtin_amdgcn_sched_barrier(0);
    }
}

__global__ void __launch_bounds__(64)
    a21_lane_kernel(TileArgs a, const double *__restrict__ xc, const unsigned *__restrict__ bcw,
                    const double *__restrict__ u, double *__restrict__ yp) {
  __shared__ double sm[2 * 6 * kLPlane + 6 * kOdd];
  const LaneTile q = lane_tile(a, (unsigned)xcd_tile(blockIdx.x, a.ntiles));
  const TileBox &tb = q.tb;
  double *const s1 = sm + 2 * 6 * kLPlane;
  const double org = lane_origin(a, q, xc);
  const double *const first = xc + 3 * lane_node(a, tb, 2 * tb.z0);
  PlaneRows r1, r2;
  {
    const long n = lane_node(a, tb, 2 * tb.z0);
    r2.load(q, a.X, xc + 3 * n, u + 3 * n);
    r2.mask(lane_bc_word(a, q, bcw, 2 * tb.z0));
    r2.store<kLPlane>(q, sm, org);
  }
  for (int kz = 0; kz < tb.nzt; kz++) {
    const int ek = tb.z0 + kz;
    double *const s0 = sm + (kz & 1) * 6 * kLPlane, *const s2 = sm + ((kz & 1) ^ 1) * 6 * kLPlane;
    const long n1 = lane_node(a, tb, 2 * ek + 1), n2 = n1 + a.XY;
    const long nc = n1 + a.X * (2 * q.cy + 1) + 2 * q.cx + 1;  // the element's centre
    double ctr[6];
    const unsigned m1 = lane_bc_word(a, q, bcw, 2 * ek + 1), m2 = lane_bc_word(a, q, bcw, 2 * ek + 2);
    r1.load(q, a.X, xc + 3 * n1, u + 3 * n1);
    r2.load(q, a.X, xc + 3 * n2, u + 3 * n2);
#pragma unroll
    for (int f = 0; f < 3; f++) {
      ctr[f] = xc[3 * nc + f] - first[f];
      ctr[3 + f] = u[3 * nc + f];
    }
    r1.mask(m1);
    if (__ballot(m1 != 0u) != 0) {
#pragma unroll
      for (int f = 0; f < 3; f++)  // the lane that holds the centre's entry of its row knows
        ctr[3 + f] = ((__shfl(m1, 3 * (2 * q.cx + 1) + f) >> (2 * q.cy + 1)) & 1u) ? 0.0 : ctr[3 + f];
    }
    r2.mask(m2);
    r1.store<kOdd>(q, s1, org);
    r2.store<kLPlane>(q, s2, org);
    __syncthreads();
    double xb[3], L[3], X[3][9], XZ[3][9], U[3][9], UZ[3][9], acc[4] = {0.0, 0.0, 0.0, 0.0};
    int lq = q.li;
    pressure_frame<kOdd>(s0 + lq, s1 + lq, s2 + lq, xb, L, ctr);
    auto part = [&](auto c) {
      constexpr int C = decltype(c)::value;
      asm volatile("" : "+v"(lq));
      plane_fields<C, kOdd>(s0 + lq, s1 + lq, s2 + lq, X, XZ, ctr);
      plane_fields<C, kOdd>(s0 + lq + 3 * kLPlane, s1 + lq + 3 * kOdd, s2 + lq + 3 * kLPlane, U, UZ, ctr + 3);
      a21_plane<C>(X, XZ, U, UZ, xb, acc);
#pragma unroll
      for (int i = 0; i < 4; i++) asm volatile("" : "+v"(acc[i]));
    };
    part(std::integral_constant<int, 0>());
    part(std::integral_constant<int, 1>());
    part(std::integral_constant<int, 2>());
    if (q.live) {
      double *ye = yp + 4 * (tb.x0 + (long)a.mx * (tb.y0 + (long)a.my * ek)) + 4 * (q.cx + a.mx * q.cy);
      ye[0] = acc[0];
#pragma unroll
      for (int d = 0; d < 3; d++) ye[1 + d] = acc[1 + d] / L[d];
    }
    __syncthreads();
  }
}

}  // namespace

// Measured, 27 lanes and one lane: one element 21 and 30 us, 2^3 63 and 31, 48^3 252
// and 58; 1 x 1 x 5000 36 and 91, 2 x 2 x 20000 197 and 302, 256 x 1 x 256 154 and
// 136.
static bool a12_lane(const Box &b, TileArgs &a) { return node_lane_plan(b, 14.3, 6.4, 1.7, 9.0, 14.6, a); }

long node_face_doubles(const Box &b) {
  TileArgs a;
  // (the diagonal's decomposition is the same)
  return a12_lane(b, a) || a11_diag_lane(b) ? face_buffer_doubles(kLT, kLT, a.ZC, a.ntiles) : 0;
}

int launch_a12(const ptmf_op_s *op, const double *p, double *yu) {
  TileArgs a;
  if (!a12_lane(op->box, a)) return launch_a12_elems(op, p, yu);
  A12Op b{};
  b.p = p;
  return launch_node_lane(op, a, b, yu);
}

int launch_a21(const ptmf_op_s *op, const double *u, double *yp) {
  double layers;
  const TileArgs a = lane_args(op->box, 1024, 0.2, &layers);
  // In microseconds, 27 lanes per element take 17.5, or 11 and 2.85 per thousand
  // elements, the lane kernel 9 and 14.2 per layer that a wave marches through,
  // however much of its 8 x 8 tile the box fills.  Measured, 27 lanes and one lane:
  // 8^3 18 and 26, 16^3 23 and 26, 20^3 34 and 26, 48^3 324 and 47; 2 x 2 x 20000
  // 238 and 287, 256 x 1 x 256 196 and 127.
  const bool lane = 9.0 + 14.2 * layers < std::max(17.5, 11.0 + 2.85e-3 * (double)op->box.nel);
  if (!lane || a.ntiles >= (1L << 31) || !lane_fits(op->box)) return launch_a21_elems(op, u, yp);
  a21_lane_kernel<<<dim3((unsigned)a.ntiles), dim3(64), 0, op->stream>>>(a, op->d64.coords, op->bcword, u, yp);
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

}  // namespace ptmf
