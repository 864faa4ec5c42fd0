// couple.hip -- the pressure-velocity couplings B (A12) and B^T (A21) of the
// Q2-P1disc element, any mesh, one lane per element (see lane.h).
//
// Both need no division: with A = det(J) J^-1 the adjugate, w det(J) d_k N_n is
// w sum_j A[k][j] (dN_n / d xi_j) and w det(J) div u is w sum_jk A[k][j] (du_k /
// d xi_j).
#include <type_traits>

#include "lane.h"

namespace ptmf {
namespace {

// adjugate A[k][j] = det(J) d xi_j / d x_k at point (a, b) of a quadrature
// plane from the positions X and their zeta derivatives Z there
__device__ __forceinline__ void plane_adjugate(int a, int b, const double X[3][9], const double Z[3][9],
                                               double A[3][3]) {
  double M[3][3];  // M[j][d] = d x_d / d xi_j
#pragma unroll
  for (int d = 0; d < 3; d++) {
    M[0][d] = cdot<double>(a, X[d][3 * b], X[d][3 * b + 1], X[d][3 * b + 2]);
    M[1][d] = cdot<double>(b, X[d][a], X[d][3 + a], X[d][6 + a]);
    M[2][d] = Z[d][3 * b + a];
  }
  A[0][0] = M[1][1] * M[2][2] - M[2][1] * M[1][2];
  A[0][1] = M[2][1] * M[0][2] - M[0][1] * M[2][2];
  A[0][2] = M[0][1] * M[1][2] - M[1][1] * M[0][2];
  A[1][0] = M[2][0] * M[1][2] - M[1][0] * M[2][2];
  A[1][1] = M[0][0] * M[2][2] - M[2][0] * M[0][2];
  A[1][2] = M[1][0] * M[0][2] - M[0][0] * M[1][2];
  A[2][0] = M[1][0] * M[2][1] - M[2][0] * M[1][1];
  A[2][1] = M[2][0] * M[0][1] - M[0][0] * M[2][1];
  A[2][2] = M[0][0] * M[1][1] - M[1][0] * M[0][1];
}

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

template <int c, int kP1 = kLPlane>
__device__ __forceinline__ void plane_fields(const double *s0, const double *s1, const double *s2, double V[3][9],
                                             double Z[3][9], const double *centre = nullptr) {
#pragma unroll
  for (int f = 0; f < 3; f++)
    lane_field<double, c, (kP1 < kLPlane)>(s0 + f * kLPlane, s1 + f * kP1, s2 + f * kLPlane, kD[c][0], kD[c][1],
                                           kD[c][2], V[f], Z[f], kP1 < kLPlane ? centre[f] : 0.0);
}

// ---------------------------------------------------------------------------
// B p: yu[3n+c] = sum_q -w detJ (d_c N_n) p_h(x_q) (MFStokesWrapper_A12,
// stokes_operators_mf.c:788-856 with MatMultMF_Stokes_MixedFEM3d_A12,
// stokes_q2p1_mf_operators_def.c:423-516), Dirichlet velocity rows zero.
//
// The coordinate planes take the place of the velocity's in the A11 lane
// kernel, and so do the transfers (five plane slots, the next layer's planes
// loaded behind the forward stages).  Bound by instruction issue at one wave
// per SIMD (4,100 FP64 instructions a layer of 64 elements, two thirds of the
// kernel's): 64 x 48 x 40 in 57 us and 5 us of faces; one 27-lane group per
// element with atomic adds to y took 290 us.
// ---------------------------------------------------------------------------
template <int c>
__device__ __forceinline__ void a12_plane(const double X[3][9], double Z[3][9], const double pc[4],
                                          const double xb[3], double out[3][3][9]) {
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

__global__ void __launch_bounds__(64)
    a12_lane_kernel(TileArgs a, const double *__restrict__ xc, const double *__restrict__ p,
                    const uint8_t *__restrict__ bcn, const uint8_t *__restrict__ bcp, double *__restrict__ y,
                    double *__restrict__ fbx, double *__restrict__ fby, double *__restrict__ fbz) {
  __shared__ double sm[5 * kLSlot];
  const LaneTile q = lane_tile(a, (unsigned)xcd_tile(blockIdx.x, a.ntiles));
  const TileBox &tb = q.tb;
  const unsigned long long bits = lane_bc_bits(a, q, bcp);
  auto plane = [&](int P) { return LaneBuf<double>(xc + 3 * lane_node(a, tb, P)); };
  {
    const LaneBuf<double> v0 = plane(2 * tb.z0), v1 = plane(2 * tb.z0 + 1), v2 = plane(2 * tb.z0 + 2);
    double r0[kLBatch], r1[kLBatch], r2[kLBatch];
    lane_rows_load<double, 0>(r0, q, a.X, v0, v1);
    lane_rows_load<double, 1>(r1, q, a.X, v0, v1);
    lane_rows_store<double, 0>(r0, q, sm, sm + kLSlot);
    lane_rows_load<double, 2>(r2, q, a.X, v0, v1);
    lane_rows_store<double, 1>(r1, q, sm, sm + kLSlot);
    lane_rows_load<double, 0, kLRows>(r0, q, a.X, v2, v2);
    lane_rows_load<double, 1, kLRows>(r1, q, a.X, v2, v2);
    lane_rows_store<double, 2>(r2, q, sm, sm + kLSlot);
    lane_rows_store<double, 0, kLRows>(r0, q, sm + 2 * kLSlot, nullptr);
    lane_rows_store<double, 1, kLRows>(r1, q, sm + 2 * kLSlot, nullptr);
  }
  double out[3][3][9];
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int n = 0; n < 9; n++) out[2][l][n] = 0.0;

  int slot = 0;  // of plane 2 ek; its successors follow modulo 5
  for (int kz = 0; kz < tb.nzt; kz++) {
    const int ek = tb.z0 + kz;
    auto place = [&](int k) { return sm + kLSlot * (slot + k >= 5 ? slot + k - 5 : slot + k); };
    double *const s0 = place(0), *const s1 = place(1), *const s2 = place(2), *const s3 = place(3),
                 *const s4 = place(4);
    // (the last layer of the chunk loads its own planes again, into free slots)
    const int nn = kz + 1 < tb.nzt ? 2 * ek + 3 : 2 * ek + 1;
    const LaneBuf<double> v1 = plane(nn), v2 = plane(nn + 1);
    const double *pe = p + 4 * (tb.x0 + (long)a.mx * (tb.y0 + (long)a.my * ek)) + 4 * (q.cx + a.mx * q.cy);
    double pc[4], xb[3], L[3], X[3][9], Z[3][9], r[kLBatch];
#pragma unroll
    for (int i = 0; i < 4; i++) pc[i] = pe[i];
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int n = 0; n < 9; n++) {
        out[0][l][n] = out[2][l][n];
        out[1][l][n] = out[2][l][n] = 0.0;
      }
    __syncthreads();
    int lq = q.li;
    pressure_frame(s0 + lq, s1 + lq, s2 + lq, xb, L);
    asm volatile("" : "+v"(lq));
    lane_rows_load<double, 0>(r, q, a.X, v1, v2);
    plane_fields<0>(s0 + lq, s1 + lq, s2 + lq, X, Z);
    lane_rows_store<double, 0>(r, q, s3, s4);
    // (a lane past a partial tile must sum zeros)
    pc[0] = q.live ? pc[0] : 0.0;
#pragma unroll
    for (int d = 0; d < 3; d++) pc[1 + d] = q.live ? pc[1 + d] / L[d] : 0.0;
    a12_plane<0>(X, Z, pc, xb, out);
    lane_pin<double>(out);
    asm volatile("" : "+v"(lq));
    lane_rows_load<double, 1>(r, q, a.X, v1, v2);
    plane_fields<1>(s0 + lq, s1 + lq, s2 + lq, X, Z);
    lane_rows_store<double, 1>(r, q, s3, s4);
    a12_plane<1>(X, Z, pc, xb, out);
    lane_pin<double>(out);
    asm volatile("" : "+v"(lq));
    lane_rows_load<double, 2>(r, q, a.X, v1, v2);
    plane_fields<2>(s0 + lq, s1 + lq, s2 + lq, X, Z);
    lane_rows_store<double, 2>(r, q, s3, s4);
    a12_plane<2>(X, Z, pc, xb, out);
    lane_pin<double>(out);
    __syncthreads();
    lane_window<double>(s0 + q.lw, q.moreX, q.moreY, out[0]);
    lane_window<double>(s1 + q.lw, q.moreX, q.moreY, out[1]);
    __syncthreads();
    lane_flush<double, kLaneZero, false>(a, q, 2 * ek, s0, (bits >> (2 * kz)) & 1, nullptr, bcn, y, fbx, fby, fbz);
    lane_flush<double, kLaneZero, false>(a, q, 2 * ek + 1, s1, (bits >> (2 * kz + 1)) & 1, nullptr, bcn, y, fbx, fby,
                                         fbz);
    __syncthreads();
    slot = slot + 2 >= 5 ? slot - 3 : slot + 2;
  }
  double *const top = sm + kLSlot * slot;
  lane_window<double>(top + q.lw, q.moreX, q.moreY, out[2]);
  __syncthreads();
  lane_flush<double, kLaneZero, true>(a, q, 2 * (tb.z0 + tb.nzt), top, (bits >> (2 * tb.nzt)) & 1, nullptr, bcn, y, fbx,
                                      fby, fbz);
}

constexpr int kFaceThreads = 256;

__global__ void __launch_bounds__(kFaceThreads)
    a12_face_kernel(TileArgs a, const double *__restrict__ fbx, const double *__restrict__ fby,
                    const double *__restrict__ fbz, double *__restrict__ y, const uint8_t *__restrict__ bcn) {
  face_sum<double, true>(a, xcd_tile(blockIdx.x, a.ntiles), fbx, fby, fbz, y, bcn);
}

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
// two waves a CU.  Bound by instruction issue: 64 x 48 x 40 in 35 us (53 us at
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

constexpr int kOdd = 234;  // nodes of a plane slot without the element centres

// One node plane of the tile on its way to its slot: the rows of its
// coordinates and velocity; all of a layer's are in flight together.
struct PlaneRows {
  double x[kLRows], u[kLRows];
  __device__ __forceinline__ void load(const LaneTile &q, long X, const double *xc, const double *u_) {
    const LaneBuf<double> bx(xc), bu(u_);
#pragma unroll
    for (int j = 0; j < kLRows; j++) {
      const unsigned row = 24u * (unsigned)X * (unsigned)min(j, q.last);
      x[j] = bx.load(8u * q.t, row);
      u[j] = bu.load(8u * q.t, row);
    }
  }
  // S: component stride of the slot
  template <int S>
  __device__ __forceinline__ void store(const LaneTile &q, double *p) const {
    const int ev = S * q.d + kLCls[q.il & 1] + (q.il >> 1);
    // (without centres their entries of the odd rows go to the rows' padding)
    const int od = S * q.d + (S == kLPlane ? kLCls[2 + (q.il & 1)] + (q.il >> 1)
                                           : ((q.il & 1) ? kLCls[1] + 8 : kLCls[2] + (q.il >> 1)));
#pragma unroll
    for (int j = 0; j < kLRows; j++) {
      p[(j & 1 ? od : ev) + kLRow * (j >> 1)] = x[j];
      p[(j & 1 ? od : ev) + kLRow * (j >> 1) + 3 * S] = u[j];
    }
  }
  __device__ __forceinline__ void mask(const LaneTile &q, long X, const uint8_t *bcn) {
    const LaneBuf<uint8_t> b(bcn);
    unsigned m[kLRows];
#pragma unroll
    for (int j = 0; j < kLRows; j++) m[j] = b.load(q.tn, (unsigned)X * (unsigned)min(j, q.last));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kLRows; j++) u[j] = ((m[j] >> q.d) & 1u) ? 0.0 : u[j];
  }
};

__global__ void __launch_bounds__(64)
    a21_lane_kernel(TileArgs a, const double *__restrict__ xc, const uint8_t *__restrict__ bcn,
                    const uint8_t *__restrict__ bcp, const double *__restrict__ u, double *__restrict__ yp) {
  __shared__ double sm[2 * 6 * kLPlane + 6 * kOdd];
  const LaneTile q = lane_tile(a, (unsigned)xcd_tile(blockIdx.x, a.ntiles));
  const TileBox &tb = q.tb;
  const unsigned long long bits = lane_bc_bits(a, q, bcp);
  double *const s1 = sm + 2 * 6 * kLPlane;
  PlaneRows r1, r2;
  {
    const long n = lane_node(a, tb, 2 * tb.z0);
    r2.load(q, a.X, xc + 3 * n, u + 3 * n);
    if (bits & 1) r2.mask(q, a.X, bcn + n);
    r2.store<kLPlane>(q, sm);
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
      ctr[f] = xc[3 * nc + f];
      ctr[3 + f] = u[3 * nc + f];
    }
    if ((bits >> (2 * kz + 1)) & 1) {
      const unsigned m = bcn[nc];
      r1.mask(q, a.X, bcn + n1);
#pragma unroll
      for (int f = 0; f < 3; f++) ctr[3 + f] = ((m >> f) & 1u) ? 0.0 : ctr[3 + f];
    }
    if ((bits >> (2 * kz + 2)) & 1) r2.mask(q, a.X, bcn + n2);
    r1.store<kOdd>(q, s1);
    r2.store<kLPlane>(q, s2);
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

long couple_face_doubles(const Box &b) {
  const TileArgs a = lane_args(b, 1024, 0.45);
  return face_buffer_doubles(kLT, kLT, a.ZC, a.ntiles);
}

int launch_a12(const ptmf_op_s *op, const double *p, double *yu) {
  const TileArgs a = lane_args(op->box, 1024, 0.45);
  PTMF_CHECK(face_buffer_doubles(kLT, kLT, a.ZC, a.ntiles) <= op->faces_doubles && a.ntiles < (1L << 31),
             PTMF_ERR_ARG, "a12: mesh too large (%ld tiles)", a.ntiles);
  double *fbx = (double *)op->faces, *fby = fbx + 3 * a.fbx_n * a.ntiles, *fbz = fby + 3 * a.fby_n * a.ntiles;
  a12_lane_kernel<<<dim3((unsigned)a.ntiles), dim3(64), 0, op->stream>>>(a, op->d64.coords, p, op->bcnode, op->bcplane,
                                                                         yu, fbx, fby, fbz);
  PTMF_HIP(hipGetLastError());
  a12_face_kernel<<<dim3((unsigned)a.ntiles), dim3(kFaceThreads), 0, op->stream>>>(a, fbx, fby, fbz, yu, op->bcnode);
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

int launch_a21(const ptmf_op_s *op, const double *u, double *yp) {
  const TileArgs a = lane_args(op->box, 1024, 0.2);
  PTMF_CHECK(a.ntiles < (1L << 31), PTMF_ERR_ARG, "a21: mesh too large (%ld tiles)", a.ntiles);
  a21_lane_kernel<<<dim3((unsigned)a.ntiles), dim3(64), 0, op->stream>>>(a, op->d64.coords, op->bcnode, op->bcplane, u,
                                                                         yp);
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

}  // namespace ptmf
