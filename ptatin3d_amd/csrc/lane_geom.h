// lane_geom.h -- lane kernels (see lane.h) of general meshes: the geometry of a
// lane's element from the node planes in LDS, and the march of the kernels that
// sum nodal values from the coordinates and per-element data alone.
#pragma once

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

template <int c, int kP1 = kLPlane>
__device__ __forceinline__ void plane_fields(const double *s0, const double *s1, const double *s2, double V[3][9],
                                             double Z[3][9], const double *centre = nullptr) {
#pragma unroll
  for (int f = 0; f < 3; f++)
    lane_field<double, c, (kP1 < kLPlane)>(s0 + f * kLPlane, s1 + f * kP1, s2 + f * kLPlane, kD[c][0], kD[c][1],
                                           kD[c][2], V[f], Z[f], kP1 < kLPlane ? centre[f] : 0.0);
}

// the first node of the tile's chunk, the coordinate of the lane's rows
__device__ __forceinline__ double lane_origin(const TileArgs &a, const LaneTile &q, const double *__restrict__ xc) {
  return xc[3 * lane_node(a, q.tb, 2 * q.tb.z0) + q.d];
}

// Middle node planes may lack the element centres, which a lane then holds
// itself: a smaller slot.
constexpr int kOdd = 234;  // nodes of a plane slot without the element centres

// One node plane of the tile on its way to its slot: the rows of its
// coordinates and velocity; all of a layer's are in flight together.
// Positions are kept from the tile's first node: an element's differences then
// lose no digits to its distance from the origin.  org: lane_origin.
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
  __device__ __forceinline__ void store(const LaneTile &q, double *p, double org) const {
    const int ev = S * q.d + kLCls[q.il & 1] + (q.il >> 1);
    // (without centres their entries of the odd rows go to the rows' padding)
    const int od = S * q.d + (S == kLPlane ? kLCls[2 + (q.il & 1)] + (q.il >> 1)
                                           : ((q.il & 1) ? kLCls[1] + 8 : kLCls[2] + (q.il >> 1)));
#pragma unroll
    for (int j = 0; j < kLRows; j++) {
      p[(j & 1 ? od : ev) + kLRow * (j >> 1)] = x[j] - org;
      p[(j & 1 ? od : ev) + kLRow * (j >> 1) + 3 * S] = u[j];
    }
  }
  __device__ __forceinline__ void mask(unsigned m) {  // the plane's lane_bc_word
    if (__ballot(m != 0u) == 0) return;
#pragma unroll
    for (int j = 0; j < kLRows; j++) u[j] = ((m >> j) & 1u) ? 0.0 : u[j];
  }
};

// y = sums over the elements of nodal values that op forms from its element's
// geometry:
//   op.begin(a, q, ek)          issues the layer's loads
//   op.frame(s0, s1, s2)        the element's nodes are in LDS
//   op.load<c>()                issues loads for quadrature plane c
//   op.plane<c>(X, Z, out)      out += the plane's part; X, Z are free to use
//   op.finish(o)                one complete node plane of sums
// The planes' coordinates take the place of the velocity's in the A11 lane
// kernel, and so do the transfers: five plane slots, the next layer's planes
// loaded behind the forward stages.
template <typename Op>
__global__ void __launch_bounds__(64)
    node_lane_kernel(TileArgs a, Op op, const double *__restrict__ xc, const unsigned *__restrict__ bcw,
                     double *__restrict__ y, double *__restrict__ fbx,
                     double *__restrict__ fby, double *__restrict__ fbz) {
  __shared__ double sm[5 * kLSlot];
  const LaneTile q = lane_tile(a, (unsigned)xcd_tile(blockIdx.x, a.ntiles));
  const TileBox &tb = q.tb;
  auto plane = [&](int P) { return LaneBuf<double>(xc + 3 * lane_node(a, tb, P)); };
  const double org = lane_origin(a, q, xc);
  auto shift = [&](double r[kLBatch]) {
#pragma unroll
    for (int k = 0; k < kLBatch; k++) r[k] -= org;
  };
  {
    const LaneBuf<double> v0 = plane(2 * tb.z0), v1 = plane(2 * tb.z0 + 1), v2 = plane(2 * tb.z0 + 2);
    double r0[kLBatch], r1[kLBatch], r2[kLBatch];
    lane_rows_load<double, 0>(r0, q, a.X, v0, v1);
    lane_rows_load<double, 1>(r1, q, a.X, v0, v1);
    shift(r0);
    lane_rows_store<double, 0>(r0, q, sm, sm + kLSlot);
    lane_rows_load<double, 2>(r2, q, a.X, v0, v1);
    shift(r1);
    lane_rows_store<double, 1>(r1, q, sm, sm + kLSlot);
    lane_rows_load<double, 0, kLRows>(r0, q, a.X, v2, v2);
    lane_rows_load<double, 1, kLRows>(r1, q, a.X, v2, v2);
    shift(r2);
    lane_rows_store<double, 2>(r2, q, sm, sm + kLSlot);
    shift(r0);
    lane_rows_store<double, 0, kLRows>(r0, q, sm + 2 * kLSlot, nullptr);
    shift(r1);
    lane_rows_store<double, 1, kLRows>(r1, q, sm + 2 * kLSlot, nullptr);
  }
  double out[3][3][9];
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int n = 0; n < 9; n++) out[2][l][n] = 0.0;

  unsigned m0 = 0, m1 = 0, m2 = 0;
  int slot = 0;  // of plane 2 ek; its successors follow modulo 5
  for (int kz = 0; kz < tb.nzt; kz++) {
    const int ek = tb.z0 + kz;
    auto place = [&](int k) { return sm + kLSlot * (slot + k >= 5 ? slot + k - 5 : slot + k); };
    double *const s0 = place(0), *const s1 = place(1), *const s2 = place(2), *const s3 = place(3),
                 *const s4 = place(4);
    // (the last layer of the chunk loads its own planes again, into free slots)
    const int nn = kz + 1 < tb.nzt ? 2 * ek + 3 : 2 * ek + 1;
    const LaneBuf<double> v1 = plane(nn), v2 = plane(nn + 1);
    double X[3][9], Z[3][9], r[kLBatch];
    op.begin(a, q, ek);
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int n = 0; n < 9; n++) {
        out[0][l][n] = out[2][l][n];
        out[1][l][n] = out[2][l][n] = 0.0;
      }
    __syncthreads();
    int lq = q.li;
    op.frame(s0 + lq, s1 + lq, s2 + lq);
    asm volatile("" : "+v"(lq));
    op.template load<0>();
    lane_rows_load<double, 0>(r, q, a.X, v1, v2);
    plane_fields<0>(s0 + lq, s1 + lq, s2 + lq, X, Z);
    shift(r);
    lane_rows_store<double, 0>(r, q, s3, s4);
    op.template plane<0>(X, Z, out);
    lane_pin<double>(out);
    asm volatile("" : "+v"(lq));
    op.template load<1>();
    lane_rows_load<double, 1>(r, q, a.X, v1, v2);
    plane_fields<1>(s0 + lq, s1 + lq, s2 + lq, X, Z);
    shift(r);
    lane_rows_store<double, 1>(r, q, s3, s4);
    op.template plane<1>(X, Z, out);
    lane_pin<double>(out);
    asm volatile("" : "+v"(lq));
    op.template load<2>();
    m0 = lane_bc_word(a, q, bcw, 2 * ek);
    m1 = lane_bc_word(a, q, bcw, 2 * ek + 1);
    m2 = lane_bc_word(a, q, bcw, 2 * ek + 2);
    lane_rows_load<double, 2>(r, q, a.X, v1, v2);
    plane_fields<2>(s0 + lq, s1 + lq, s2 + lq, X, Z);
    shift(r);
    lane_rows_store<double, 2>(r, q, s3, s4);
    asm volatile("" : "+v"(m0), "+v"(m1), "+v"(m2));
    op.template plane<2>(X, Z, out);
    lane_pin<double>(out);
    op.finish(out[0]);
    op.finish(out[1]);
    __syncthreads();
    lane_window<double>(s0 + q.lw, q.moreX, q.moreY, out[0]);
    lane_window<double>(s1 + q.lw, q.moreX, q.moreY, out[1]);
    __syncthreads();
    lane_flush<double, Op::kBC, false>(a, q, 2 * ek, s0, m0, y, fbx, fby, fbz);
    lane_flush<double, Op::kBC, false>(a, q, 2 * ek + 1, s1, m1, y, fbx, fby,
                                         fbz);
    __syncthreads();
    slot = slot + 2 >= 5 ? slot - 3 : slot + 2;
  }
  double *const top = sm + kLSlot * slot;
  op.finish(out[2]);
  lane_window<double>(top + q.lw, q.moreX, q.moreY, out[2]);
  __syncthreads();
  lane_flush<double, Op::kBC, true>(a, q, 2 * (tb.z0 + tb.nzt), top, m2, y, fbx,
                                      fby, fbz);
}

constexpr int kFaceThreads = 256;

__global__ void __launch_bounds__(kFaceThreads)
    node_face_kernel(TileArgs a, const double *__restrict__ fbx, const double *__restrict__ fby,
                    const double *__restrict__ fbz, double *__restrict__ y, const uint8_t *__restrict__ bcn) {
  face_sum<double, true>(a, xcd_tile(blockIdx.x, a.ntiles), fbx, fby, fbz, y, bcn);
}

// The decomposition of box b; false where 27 lanes per element are faster: in
// microseconds these take `few` and `launch` for each parity class that has
// elements and `elem` per thousand elements, the lane kernel `first` and `layer`
// per layer that a wave marches through, however much of its 8 x 8 tile the box
// fills.  (They also have the boxes past the lane kernel's 32-bit offsets.)
inline bool node_lane_plan(const Box &b, double few, double launch, double elem, double first, double layer,
                           TileArgs &a) {
  double layers;
  a = lane_args(b, 1024, 0.45, &layers);
  int classes = 0;
  for (int color = 0; color < 8; color++) classes += class_count(b, color) > 0;
  return first + layer * layers < few + launch * classes + 1e-3 * elem * (double)b.nel && a.ntiles < (1L << 31) &&
         lane_fits(b);
}

// the kernel and its faces
template <typename Op>
int launch_node_lane(const ptmf_op_s *op, const TileArgs &a, const Op &nodal, double *y) {
  PTMF_CHECK(face_buffer_doubles(kLT, kLT, a.ZC, a.ntiles) <= op->node_faces_doubles, PTMF_ERR_NOT_SETUP,
             "face buffers not allocated");
  std::lock_guard<std::mutex> lock(op->node_faces_mu);
  double *fbx = op->node_faces, *fby = fbx + 3 * a.fbx_n * a.ntiles, *fbz = fby + 3 * a.fby_n * a.ntiles;
  node_lane_kernel<Op><<<dim3((unsigned)a.ntiles), dim3(64), 0, op->stream>>>(a, nodal, op->d64.coords, op->bcword, y,
                                                                              fbx, fby, fbz);
  PTMF_HIP(hipGetLastError());
  node_face_kernel<<<dim3((unsigned)a.ntiles), dim3(kFaceThreads), 0, op->stream>>>(a, fbx, fby, fbz, y, op->bcnode);
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

}  // namespace
}  // namespace ptmf
