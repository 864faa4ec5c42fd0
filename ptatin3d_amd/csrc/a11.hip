// a11.hip -- matrix-free Q2 viscous block (A11) apply for gfx950.
//
// Computes A11_local u for all elements of a structured Q2 box, the operator
// of MFStokesWrapper_A11_Tensor (stokes_operators_tensor.c:181-288): per
// element and quadrature point, grad u and the Jacobian from the 27 nodal
// values, then w*detJ*(2 eta sym(grad u)) G^T, then the transposed gradient
// back to the nodes.
//
// Element work decomposition (MI355X-first, not one-warp-per-element):
//   * 3 lanes per element, lane c owns quadrature plane zeta_c (9 qps) and,
//     on input/output, node plane k = c of the element; 21 elements per
//     64-lane wave, one wave per work-group (no cross-wave barriers).
//   * Collocated sum factorisation: nodal -> quadrature-grid interpolation
//     (B x B x B), then the three reference derivatives on the quadrature
//     grid with the 3x3 collocation matrix C = D B^-1.  The xi/eta stages
//     are in registers; only the zeta stage crosses lanes, through LDS.
//   * The 1/detJ of the inverse Jacobian is folded into one scalar per qp
//     (adjugate form): one division per qp.
//   * Viscosity is stored quadrature-point-major (eta[q*nel + e]) so the
//     lanes of a wave read consecutive elements.
//
// Scatter (MatMult path, a11_tile_kernel + a11_face_copy_kernel):
//   * A wave owns a TX x TY tile of elements in x-y (TX*TY <= 21) and marches
//     through a chunk of ZC element layers in z.  Element outputs are summed
//     into an LDS window of three node planes (ordered plain read-add-write,
//     LDS float atomics are slow here); after each layer the two completed
//     node planes are flushed with plain stores.
//   * A tile owns its node range [2x0,2x1) x [2y0,2y1) x [2z0,2z1) (plus the
//     closing planes at the domain's upper boundary).  Contributions to the
//     tile's upper faces go to per-tile face buffers (x face first, then y,
//     then z), and a11_face_copy_kernel adds them into the owning tile's lower
//     faces.  No global atomics, no clearing of y, deterministic sums.
//   * Dirichlet rows (y = x) are written by work-groups of the same launch,
//     over the compact list of Dirichlet dofs.
// This tile kernel has the large deformed meshes and the tilings and variants of
// the caller's choice; rectilinear meshes take a11_lane.h and small boxes
// a11_col.h (lane_plan and col_box below).
// The spmv path (y += A u, no boundary handling) keeps a one-pass kernel with
// global atomic adds; it serves the host-array PETSc adapter contract.
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "ptmf_internal.h"
#include "lane.h"

namespace ptmf {
namespace {

constexpr int kEPW = 21;  // elements per wave (3 lanes each; lane 63 idle)
constexpr int kSlots = 54;
// Exchange-buffer columns: the 21 element slots, plus (FP32) one for the
// idle lane 63, which then reads and writes a column of its own and needs
// no write guards.  Measured on the 64^3 MatMult: the FP32 kernel is 3-4 %
// faster with the spare column, the FP64 kernel 2.5 % slower, so FP64 keeps
// 21 columns and guards its writes.
template <typename T>
constexpr int sh_cols() { return sizeof(T) == 4 ? kEPW + 1 : kEPW; }
constexpr int kWinNodes = 130;  // >= (2TX+1)(2TY+1) for every TX*TY <= 21

// Barrier of one element tile's lanes.  A work-group holds kW waves, each
// marching through its own tile with its own LDS buffers, so with kW > 1 the
// waves never wait for each other (their tiles may have different numbers
// of layers): the barrier is the wave's own (LDS operations of one wave
// execute in order; the fences keep the compiler from moving them across).
template <int kWaves>
__device__ __forceinline__ void tsync() {
  if constexpr (kWaves == 1) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// lane of the calling thread within its wave
template <int kWaves>
__device__ __forceinline__ int wave_lane() {
  if constexpr (kWaves == 1) return (int)threadIdx.x;
  else return (int)(threadIdx.x & 63);
}

// Raw input of one lane's node plane: coordinates and velocity of the 9
// nodes (i, j) of plane k = cp, their Dirichlet bits, and the viscosity at
// the lane's 9 quadrature points.  Kept unmodified in registers between the
// load and the forward stage so the loads can be issued a layer ahead.
template <typename T>
struct PlaneRaw {
  T x[3][9];  // [d][3j+i]
  T u[3][9];
  unsigned m[9];
  T eta[9];
};

template <typename T, bool kMask>
__device__ __forceinline__ void load_plane_nodes(PlaneRaw<T> &r, const T *__restrict__ xc,
                                                 const T *__restrict__ u,
                                                 const uint8_t *__restrict__ bcn, long base, long X) {
#pragma unroll
  for (int j = 0; j < 3; j++)
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const long node = base + i + X * j;
      r.m[3 * j + i] = kMask ? (unsigned)bcn[node] : 0u;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        r.x[d][3 * j + i] = xc[3 * node + d];
        r.u[d][3 * j + i] = u[3 * node + d];
      }
    }
}

template <typename T>
__device__ __forceinline__ void load_plane_eta(PlaneRaw<T> &r, const T *__restrict__ etap, long stride) {
#pragma unroll
  for (int p = 0; p < 9; p++) r.eta[p] = etap[(long)p * stride];
}

// in-plane interpolation of a 3x3 node plane to the 3x3 quadrature grid:
// V[d][3b+a] = sum_{i,j} B[a][i] B[b][j] g[d][3j+i]
template <typename T>
__device__ __forceinline__ void interp_plane(const T g[3][9], T V[3][9]) {
#pragma unroll
  for (int d = 0; d < 3; d++) {
    T t[3][3];  // [j][a]
#pragma unroll
    for (int j = 0; j < 3; j++) interp3<T>(g[d][3 * j], g[d][3 * j + 1], g[d][3 * j + 2], t[j][0], t[j][1], t[j][2]);
#pragma unroll
    for (int a = 0; a < 3; a++) interp3<T>(t[0][a], t[1][a], t[2][a], V[d][a], V[d][3 + a], V[d][6 + a]);
  }
}

// Forward stage: in-plane interpolation of the lane's node plane, exchange
// through the LDS buffer (slots 0..26 coordinates, 27..53 masked velocity),
// zeta interpolation to the lane's quadrature plane.
template <typename T, bool kMask, int kWaves = 1>
__device__ __forceinline__ void plane_forward(int cp, int le, bool writer, const PlaneRaw<T> &r,
                                              T (*sh)[kSlots][sh_cols<T>()], T Xq[3][9], T Uq[3][9]) {
  T bz[3];
#pragma unroll
  for (int k = 0; k < 3; k++) bz[k] = sel3<T>(cp, kB[0][k], kB[1][k], kB[2][k]);
  {
    T V[3][9];
    interp_plane<T>(r.x, V);
    if (writer) {
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int p = 0; p < 9; p++) sh[cp][9 * d + p][le] = V[d][p];
    }
  }
  {
    T g[3][9], V[3][9];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
      for (int n = 0; n < 9; n++) g[d][n] = ((r.m[n] >> d) & 1u) ? T(0) : r.u[d][n];
    interp_plane<T>(g, V);
    if (writer) {
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int p = 0; p < 9; p++) sh[cp][27 + 9 * d + p][le] = V[d][p];
    }
  }
  tsync<kWaves>();
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int p = 0; p < 9; p++) {
      Xq[d][p] = bz[0] * sh[0][9 * d + p][le] + bz[1] * sh[1][9 * d + p][le] +
                 bz[2] * sh[2][9 * d + p][le];
      Uq[d][p] = bz[0] * sh[0][27 + 9 * d + p][le] + bz[1] * sh[1][27 + 9 * d + p][le] +
                 bz[2] * sh[2][27 + 9 * d + p][le];
    }
}

// Pointwise stage on the 9 quadrature points of the lane's plane: Jacobian
// (adjugate form, one division per point), symmetric gradient, viscous
// stress, and the transposed derivatives.  The xi/eta parts are accumulated
// in W and exchanged with the zeta parts through the LDS buffer: on return,
// slots 9l+p hold the zeta components and slots 27+9l+p the xi/eta
// accumulations of every plane.
//
// A work-group is a single wave, so the LDS operations of all lanes execute
// in program order: a slot read by every lane at qp p is overwritten only
// after those reads.
// Per-lane data of the pressure coupling in the fused saddle-point MatMult:
// the element centroid xb, the pressure coefficients with the element
// lengths divided out, p_h(x) = pc0 + sum_d pc[1+d] (x_d - xb_d) (the P1GRel
// basis, element_utils_q2.c:183-224), and the lane's partial sums of
// B^T u against {1, x - xb, y - yb, z - zb}.
template <typename T>
struct PCoupling {
  T xb[3];
  T pc[4];
  T acc[4];
};

template <typename T, bool kStokes = false, int kWaves = 1>
__device__ __forceinline__ void plane_qp(int cp, int le, bool writer, const T Xq[3][9],
                                         const T Uq[3][9], const T etq9[9],
                                         T (*sh)[kSlots][sh_cols<T>()], PCoupling<T> *pcp = nullptr) {
  T dz[3];
#pragma unroll
  for (int k = 0; k < 3; k++) dz[k] = sel3<T>(cp, kD[0][k], kD[1][k], kD[2][k]);
  const T wz = sel3<T>(cp, kW[0], kW[1], kW[2]);
  T W[3][9];  // in-plane transposed xi/eta derivatives, accumulated
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int p = 0; p < 9; p++) W[l][p] = T(0);

  // zeta-plane values of the next point are read before this point's zeta
  // part is written (point p writes slots p, 9+p, 18+p; point p+1 reads
  // slots p+1, 9+p+1, ... only)
  T Z[2][2][3][3];
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int k = 0; k < 3; k++) {
      Z[0][0][d][k] = sh[k][9 * d][le];
      Z[0][1][d][k] = sh[k][27 + 9 * d][le];
    }
#pragma unroll
  for (int b = 0; b < 3; b++)
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int p = 3 * b + a;
      if (p < 8) {
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
          for (int k = 0; k < 3; k++) {
            Z[(p + 1) & 1][0][d][k] = sh[k][9 * d + p + 1][le];
            Z[(p + 1) & 1][1][d][k] = sh[k][27 + 9 * d + p + 1][le];
          }
      }
      const T etq = etq9[p];
      // M[j][d] = d x_d / d xi_j, Gu[j][l] = d u_l / d xi_j
      T M[3][3], Gu[3][3];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        M[0][d] = cdot<T>(a, Xq[d][3 * b], Xq[d][3 * b + 1], Xq[d][3 * b + 2]);
        M[1][d] = cdot<T>(b, Xq[d][a], Xq[d][3 + a], Xq[d][6 + a]);
        M[2][d] = dz[0] * Z[p & 1][0][d][0] + dz[1] * Z[p & 1][0][d][1] + dz[2] * Z[p & 1][0][d][2];
        Gu[0][d] = cdot<T>(a, Uq[d][3 * b], Uq[d][3 * b + 1], Uq[d][3 * b + 2]);
        Gu[1][d] = cdot<T>(b, Uq[d][a], Uq[d][3 + a], Uq[d][6 + a]);
        Gu[2][d] = dz[0] * Z[p & 1][1][d][0] + dz[1] * Z[p & 1][1][d][1] + dz[2] * Z[p & 1][1][d][2];
      }
      // adjugate A = det * M^-1 (A[k][j] = det * d xi_j / d x_k)
      T A[3][3];
      A[0][0] = M[1][1] * M[2][2] - M[2][1] * M[1][2];
      A[0][1] = M[2][1] * M[0][2] - M[0][1] * M[2][2];
      A[0][2] = M[0][1] * M[1][2] - M[1][1] * M[0][2];
      A[1][0] = M[2][0] * M[1][2] - M[1][0] * M[2][2];
      A[1][1] = M[0][0] * M[2][2] - M[2][0] * M[0][2];
      A[1][2] = M[1][0] * M[0][2] - M[0][0] * M[1][2];
      A[2][0] = M[1][0] * M[2][1] - M[2][0] * M[1][1];
      A[2][1] = M[2][0] * M[0][1] - M[0][0] * M[2][1];
      A[2][2] = M[0][0] * M[1][1] - M[1][0] * M[0][1];
      const T det = M[0][0] * A[0][0] + M[0][1] * A[1][0] + M[0][2] * A[2][0];
      const T wq = (T)(kW[a] * kW[b]) * wz;
      const T s = (T(2) * wq * etq) * recip<T>(det);
      // gh[k][l] = det * d u_l / d x_k
      T gh[3][3];
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int l = 0; l < 3; l++)
          gh[k][l] = Gu[0][l] * A[k][0] + Gu[1][l] * A[k][1] + Gu[2][l] * A[k][2];
      // sigma = 2 eta sym(grad u) * w * detJ / det^2 (scaled so that the
      // adjugate can stand in for detJ * G)
      const T hs = T(0.5) * s;
      T sg[3][3];
      sg[0][0] = s * gh[0][0];
      sg[1][1] = s * gh[1][1];
      sg[2][2] = s * gh[2][2];
      sg[0][1] = sg[1][0] = hs * (gh[0][1] + gh[1][0]);
      sg[0][2] = sg[2][0] = hs * (gh[0][2] + gh[2][0]);
      sg[1][2] = sg[2][1] = hs * (gh[1][2] + gh[2][1]);
      if constexpr (kStokes) {
        // A12: the pressure enters the stress as -p_h I; A21: the lane's
        // share of -sum_q w detJ NIp_i div u (w detJ div u = w tr(gh))
        const T d0 = Xq[0][p] - pcp->xb[0], d1 = Xq[1][p] - pcp->xb[1], d2 = Xq[2][p] - pcp->xb[2];
        const T wp = wq * (pcp->pc[0] + pcp->pc[1] * d0 + pcp->pc[2] * d1 + pcp->pc[3] * d2);
        sg[0][0] -= wp;
        sg[1][1] -= wp;
        sg[2][2] -= wp;
        const T dv = -wq * (gh[0][0] + gh[1][1] + gh[2][2]);
        pcp->acc[0] += dv;
        pcp->acc[1] += dv * d0;
        pcp->acc[2] += dv * d1;
        pcp->acc[3] += dv * d2;
      }
      // every lane has read slot p of all planes; reuse it for the zeta data
      __builtin_amdgcn_wave_barrier();
      // dv[j][l] = w detJ sum_m sigma[m][l] d xi_j / d x_m
#pragma unroll
      for (int l = 0; l < 3; l++) {
        const T dv0 = sg[0][l] * A[0][0] + sg[1][l] * A[1][0] + sg[2][l] * A[2][0];
        const T dv1 = sg[0][l] * A[0][1] + sg[1][l] * A[1][1] + sg[2][l] * A[2][1];
        const T dv2 = sg[0][l] * A[0][2] + sg[1][l] * A[1][2] + sg[2][l] * A[2][2];
#pragma unroll
        for (int r = 0; r < 3; r++) {
          if (a != 1 || r != 1) W[l][3 * b + r] += (T)kC[a][r] * dv0;
          if (b != 1 || r != 1) W[l][3 * r + a] += (T)kC[b][r] * dv1;
        }
        if (writer) sh[cp][9 * l + p][le] = dv2;  // zeta component, exchanged below
      }
      __builtin_amdgcn_wave_barrier();
    }
  tsync<kWaves>();
  if (writer) {
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int p = 0; p < 9; p++) sh[cp][27 + 9 * l + p][le] = W[l][p];
  }
  tsync<kWaves>();
}

// Backward stage: node plane k = cp gathers the three quadrature planes
// (zeta), then the transposed in-plane interpolation; out[l][3j+i] is the
// element result at node (i, j, k = cp), component l.  Ends with a barrier:
// the exchange buffer is free again on return.
template <typename T, int kWaves = 1>
__device__ __forceinline__ void plane_backward(int cp, int le, T (*sh)[kSlots][sh_cols<T>()], T out[3][9]) {
  T bt[3], dt[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    bt[k] = sel3<T>(cp, kB[k][0], kB[k][1], kB[k][2]);
    dt[k] = sel3<T>(cp, kD[k][0], kD[k][1], kD[k][2]);
  }
  T Y[3][9];
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int p = 0; p < 9; p++) {
      const T z0 = sh[0][9 * l + p][le], z1 = sh[1][9 * l + p][le], z2 = sh[2][9 * l + p][le];
      const T w0 = sh[0][27 + 9 * l + p][le], w1 = sh[1][27 + 9 * l + p][le],
              w2 = sh[2][27 + 9 * l + p][le];
      Y[l][p] = bt[0] * w0 + bt[1] * w1 + bt[2] * w2 + dt[0] * z0 + dt[1] * z1 + dt[2] * z2;
    }
  tsync<kWaves>();
#pragma unroll
  for (int l = 0; l < 3; l++) interp_plane_t<T>(Y[l], out[l]);
}

// The element computation of one lane: element e (node plane origin `base`,
// lane plane cp), result out[l][3j+i] = (A11_e u)(node (i,j,k=cp), comp l).
// Every lane of the wave must call it (it contains wave-wide barriers); lanes
// with writer == false (lane 63) never write the exchange buffer.
template <typename T, bool kMask, int kWaves = 1>
__device__ __forceinline__ void element_plane_apply(int cp, int le, bool writer, const T *__restrict__ etap,
                                                    long estride, long base, long X,
                                                    const T *__restrict__ xc,
                                                    const uint8_t *__restrict__ bcn,
                                                    const T *__restrict__ u,
                                                    T (*sh)[kSlots][sh_cols<T>()], T out[3][9]) {
  PlaneRaw<T> r;
  load_plane_nodes<T, kMask>(r, xc, u, bcn, base, X);
  load_plane_eta<T>(r, etap, estride);
  T Xq[3][9], Uq[3][9];
  plane_forward<T, kMask, kWaves>(cp, le, writer, r, sh, Xq, Uq);
  plane_qp<T, false, kWaves>(cp, le, writer, Xq, Uq, r.eta, sh);
  plane_backward<T, kWaves>(cp, le, sh, out);
}

// The same element computation for the saddle-point operator
// [A11 A12; A21 0] (MatMult_MFStokes_A, stokes_operators.c:884-967): the
// element's pressure pe[0..3] enters the stress, and B^T of the masked
// velocity is written to ype[0..3] by the lane of plane 0 (live lanes only).
// sL holds the element lengths between the first and last stage.
template <typename T>
__device__ __forceinline__ void element_plane_apply_stokes(int cp, int le, bool writer, bool live,
                                                           const T *__restrict__ etap, long estride, long base,
                                                           long X, const T *__restrict__ xc,
                                                           const uint8_t *__restrict__ bcn,
                                                           const T *__restrict__ u, const T *__restrict__ pe,
                                                           T *__restrict__ ype, T (*sh)[kSlots][sh_cols<T>()],
                                                           T (*sL)[kEPW], T out[3][9]) {
  PlaneRaw<T> r;
  load_plane_nodes<T, true>(r, xc, u, bcn, base, X);
  load_plane_eta<T>(r, etap, estride);
  PCoupling<T> pcp;
  // centroid and lengths: x14 - x12 and y16 - y10 lie in plane 1, z22 - z4
  // joins the centre nodes of planes 2 and 0
  if (writer) {
#pragma unroll
    for (int d = 0; d < 3; d++) {
      T sum = T(0);
#pragma unroll
      for (int n = 0; n < 9; n++) sum += r.x[d][n];
      sh[cp][d][le] = sum;
    }
    sh[cp][3][le] = r.x[2][4];
    sh[cp][4][le] = r.x[0][5] - r.x[0][3];
    sh[cp][5][le] = r.x[1][7] - r.x[1][1];
  }
  __syncthreads();
  const T Lx = sh[1][4][le], Ly = sh[1][5][le], Lz = sh[2][3][le] - sh[0][3][le];
#pragma unroll
  for (int d = 0; d < 3; d++) pcp.xb[d] = (sh[0][d][le] + sh[1][d][le] + sh[2][d][le]) * T(1.0 / 27.0);
  if (writer && cp == 0) {
    sL[0][le] = Lx;
    sL[1][le] = Ly;
    sL[2][le] = Lz;
  }
  pcp.pc[0] = pe[0];
  pcp.pc[1] = pe[1] / Lx;
  pcp.pc[2] = pe[2] / Ly;
  pcp.pc[3] = pe[3] / Lz;
#pragma unroll
  for (int i = 0; i < 4; i++) pcp.acc[i] = T(0);
  __syncthreads();
  T Xq[3][9], Uq[3][9];
  plane_forward<T, true>(cp, le, writer, r, sh, Xq, Uq);
  plane_qp<T, true>(cp, le, writer, Xq, Uq, r.eta, sh, &pcp);
  plane_backward<T>(cp, le, sh, out);
  if (writer) {
#pragma unroll
    for (int i = 0; i < 4; i++) sh[cp][i][le] = pcp.acc[i];
  }
  __syncthreads();
  if (live && cp == 0) {
    ype[0] = sh[0][0][le] + sh[1][0][le] + sh[2][0][le];
#pragma unroll
    for (int i = 1; i < 4; i++) ype[i] = (sh[0][i][le] + sh[1][i][le] + sh[2][i][le]) / sL[i - 1][le];
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// spmv: y += A11_local u with global atomic adds (no boundary handling)
// ---------------------------------------------------------------------------
template <typename T, bool kMask>
__global__ void __launch_bounds__(64)
    a11_atomic_kernel(int mx, int my, long nel, long X, long XY, const T *__restrict__ xc,
                      const T *__restrict__ eta, const uint8_t *__restrict__ bcn,
                      const T *__restrict__ u, T *__restrict__ y) {
  __shared__ T sh[3][kSlots][sh_cols<T>()];
  const int lane = threadIdx.x;
  const int c = lane / kEPW;  // quadrature / node plane; 3 marks the idle lane
  const int le = lane - c * kEPW;
  const int cp = c < 3 ? c : 2;
  long e = (long)blockIdx.x * kEPW + le;
  const bool live = (c < 3) && (e < nel);
  if (e >= nel) e = nel - 1;
  const long ei = e % mx, er = e / mx, ej = er % my, ek = er / my;
  const long base = 2 * ei + X * (2 * ej) + XY * (2 * ek + cp);
  T out[3][9];
  element_plane_apply<T, kMask>(cp, le, c < 3, eta + (long)(9 * cp) * nel + e, nel, base, X, xc, bcn,
                                u, sh, out);
  if (live) {
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int j = 0; j < 3; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) atomicAdd(&y[3 * (base + i + X * j) + l], out[l][3 * j + i]);
  }
}

// ---------------------------------------------------------------------------
// MatMult with a coloured scatter (kernel variant 3): one launch per element
// parity class, 21 elements of the class per wave, each lane adding its
// node plane's sums into y with plain read-add-write (no two elements of a
// class share a node).  y is cleared first; viscosity read quadrature-point
// major (eta[q * nel + e]).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(64)
    a11_colour_kernel(int mx, int my, int mz, long nel, long X, long XY, int color, const T *__restrict__ xc,
                      const T *__restrict__ eta, const uint8_t *__restrict__ bcn, const T *__restrict__ u,
                      T *__restrict__ y) {
  __shared__ T sh[3][kSlots][sh_cols<T>()];
  const int lane = threadIdx.x;
  const int c = lane / kEPW;  // quadrature / node plane; 3 marks the idle lane
  const int le = lane - c * kEPW;
  const int cp = c < 3 ? c : 2;
  bool in_class;
  const long e = class_element(mx, my, mz, color, (long)blockIdx.x * kEPW + le, in_class);
  const bool live = (c < 3) && in_class;
  const long ei = e % mx, er = e / mx, ej = er % my, ek = er / my;
  const long base = 2 * ei + X * (2 * ej) + XY * (2 * ek + cp);
  T out[3][9];
  element_plane_apply<T, true>(cp, le, c < 3, eta + (long)(9 * cp) * nel + e, nel, base, X, xc, bcn, u, sh, out);
  if (live) {
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int l = 0; l < 3; l++) {
          T *q = y + 3 * (base + i + X * j) + l;
          *q += out[l][3 * j + i];
        }
  }
}

// ---------------------------------------------------------------------------
// MatMult: tiled z-march with an LDS node-plane window and face buffers
// ---------------------------------------------------------------------------
// Tile-ordered quadrature-point data (viscosity for variants 0/1): for tile
// t, layer kz of its z-chunk, quadrature point q and element slot le of the
// wave, index ((t * ZC + kz) * 27 + q) * 21 + le, so the lanes of a plane read
// 21 consecutive values.  Slots beyond a partial tile repeat the clamped
// element, as the MatMult kernels do.
__device__ __forceinline__ long tq_index(long tile, int ZC, int kz, int q, int le) {
  return ((tile * ZC + kz) * 27 + q) * (long)kEPW + le;
}

// One thread per place in a tile layer, so that it is worked out once for the
// 27 points (48^3 11.2 us; per value 25.8 us).
template <typename T>
__global__ void __launch_bounds__(256)
    eta_tile_kernel(TileArgs a, const double *__restrict__ eta, T *__restrict__ et) {
  const long nslots = a.ntiles * a.ZC * kEPW, step = 256L * gridDim.x;
  for (long t = xcd_tile(blockIdx.x, gridDim.x) * 256L + threadIdx.x; t < nslots; t += step) {
    const long layer = t / kEPW, tile = layer / a.ZC;
    const int le = (int)(t - kEPW * layer), kz = (int)(layer - a.ZC * tile);
    const TileBox tb = tile_box(a, tile);
    if (kz >= tb.nzt) continue;
    const int ly = le / a.TX, lx = le - a.TX * ly;
    const int ex = tb.x0 + min(lx, tb.nxt - 1), ey = tb.y0 + min(ly, tb.nyt - 1);
    const double *src = eta + ex + (long)a.mx * (ey + (long)a.my * (tb.z0 + kz));
    T *dst = et + tq_index(tile, a.ZC, kz, 0, le);
    double v[27];
#pragma unroll
    for (int q = 0; q < 27; q++) v[q] = src[q * a.nel];
#pragma unroll
    for (int q = 0; q < 27; q++) dst[q * kEPW] = (T)v[q];
  }
}

// Write the completed node plane P of the window: owned nodes to y, the
// tile's upper-face nodes to the face buffers (the x face column, corner
// included, then the y face row, then on the tile's top plane the z face).
// Pure LDS reads and global stores; clears the window entries it reads.
// Three loops, one destination each (no divergent stores): the owned block
// (node columns il < nxo, rows jl < nyo), the upper x face column and the
// upper y face row.
template <typename T, int kWaves = 1>
__device__ __forceinline__ void flush_plane(const TileArgs &a, long tile, const TileBox &tb, int P,
                                            T *__restrict__ win, T *__restrict__ y,
                                            T *__restrict__ fbx, T *__restrict__ fby,
                                            T *__restrict__ fbz) {
  const int wX = 2 * tb.nxt + 1, wY = 2 * tb.nyt + 1;
  const int W3 = 3 * wX;
  const int kl = P - 2 * tb.z0;
  const int nxo = tb.xend ? wX : 2 * tb.nxt;  // owned node columns
  const int nyo = tb.yend ? wY : 2 * tb.nyt;  // owned node rows
  const int R3 = 3 * nxo;
  const int lane = wave_lane<kWaves>();
  {
    // owned block: entry t = jl * R3 + r (r = 3 il + l) is window entry jl * W3 + r
    const bool zface = kl >= 2 * tb.nzt && !tb.zend;
    T *const dst = zface ? fbz : y;
    const long off = zface ? 3 * tile * a.fbz_n
                           : 3 * ((long)(2 * tb.x0) + a.XY * (long)P + a.X * (long)(2 * tb.y0));
    const long rs = zface ? 3L * (2 * a.TX + 1) : 3 * a.X;
    const float inv = 1.0f / (float)R3;
    for (int t = lane; t < R3 * nyo; t += 64) {
      int jl = (int)((float)t * inv);
      if (jl * R3 > t) jl--;
      if ((jl + 1) * R3 <= t) jl++;
      const int r = t - jl * R3;
      const int w = jl * W3 + r;
      const T v = win[w];
      win[w] = T(0);
      dst[off + rs * jl + r] = v;
    }
  }
  if (!tb.xend) {
    // upper x face: node column il = 2 nxt of every row, t = 3 jl + l
    const long off = 3 * (tile * a.fbx_n + (long)(2 * a.TY + 1) * kl);
    for (int t = lane; t < 3 * wY; t += 64) {
      const int jl = t / 3;
      const int w = jl * W3 + 6 * tb.nxt + (t - 3 * jl);
      const T v = win[w];
      win[w] = T(0);
      fbx[off + t] = v;
    }
  }
  if (!tb.yend) {
    // upper y face: node row jl = 2 nyt without the x face corner, t = 3 il + l
    const long off = 3 * (tile * a.fby_n + (long)(2 * a.TX + 1) * kl);
    for (int t = lane; t < R3; t += 64) {
      const int w = 2 * tb.nyt * W3 + t;
      const T v = win[w];
      win[w] = T(0);
      fby[off + t] = v;
    }
  }
}

// One tile's z-march (the work of one wave); shared by the single-box and
// the batched MatMult kernels.
template <typename T, bool kMask, bool kStokes = false, int kWaves = 1>
__device__ __forceinline__ void tile_march(const TileArgs &a, long tile, const T *__restrict__ xc,
                                           const T *__restrict__ eta, const uint8_t *__restrict__ bcn,
                                           const T *__restrict__ u, T *__restrict__ y, T *__restrict__ fbx,
                                           T *__restrict__ fby, T *__restrict__ fbz,
                                           T (*sh)[kSlots][sh_cols<T>()], T (*win)[3 * kWinNodes],
                                           const T *__restrict__ p = nullptr, T *__restrict__ yp = nullptr,
                                           T (*sL)[kEPW] = nullptr) {
  const TileBox tb = tile_box(a, tile);
  const int lane = wave_lane<kWaves>();
  const int c = lane / kEPW;
  const int le = lane - c * kEPW;
  const int cp = c < 3 ? c : 2;
  const int lx = le % a.TX, ly = le / a.TX;
  const bool live = (c < 3) && (le < a.TX * a.TY) && (lx < tb.nxt) && (ly < tb.nyt);
  const int ex = tb.x0 + min(lx, tb.nxt - 1), ey = tb.y0 + min(ly, tb.nyt - 1);
  const int wX = 2 * tb.nxt + 1;
  // exchange-buffer column and write permission: with the spare column
  // (FP32) the idle lane computes on element slot 0 but uses a column of its
  // own, so every lane may write
  constexpr bool kSpare = sh_cols<T>() > kEPW;
  const int lc = (c < 3 || !kSpare) ? le : kEPW;
  const bool wr = kSpare || c < 3;

  for (int t = lane; t < 9 * kWinNodes; t += 64) (&win[0][0])[t] = T(0);
  tsync<kWaves>();

  for (int kz = 0; kz < tb.nzt; kz++) {
    const long ek = tb.z0 + kz;
    const long base = 2L * ex + a.X * (2L * ey) + a.XY * (2 * ek + cp);
    T out[3][9];
    if constexpr (kStokes) {
      const long e = ex + (long)a.mx * (ey + (long)a.my * ek);
      element_plane_apply_stokes<T>(cp, le, c < 3, live, eta + tq_index(tile, a.ZC, kz, 9 * cp, le), kEPW, base,
                                    a.X, xc, bcn, u, p + 4 * e, yp + 4 * e, sh, sL, out);
    } else {
      element_plane_apply<T, kMask, kWaves>(cp, lc, wr, eta + tq_index(tile, a.ZC, kz, 9 * cp, le), kEPW, base,
                                            a.X, xc, bcn, u, sh, out);
    }
    // Sum into the window with plain read-add-write.  Element (lx, ly)
    // touches nodes (2lx + i, 2ly + j); only slots i = 2 / j = 2 meet the
    // slots i = 0 / j = 0 of the next element, so the nine slots go in four
    // groups, within which no two lanes touch the same entry: {i, j < 2},
    // {i = 2, j < 2}, {i < 2, j = 2}, {(2, 2)}.  The wave executes LDS
    // operations in order; the barriers between groups keep the compiler
    // from interleaving them.
    {
      T *w = win[(2 * kz + cp) % 3] + 3 * ((2 * ly) * wX + 2 * lx);
#pragma unroll
      for (int g = 0; g < 4; g++) {
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
          for (int i = 0; i < 3; i++) {
            if ((i == 2 ? 1 : 0) + (j == 2 ? 2 : 0) != g) continue;
            if (live) {
              T *q = w + 3 * (j * wX + i);
              const T q0 = q[0], q1 = q[1], q2 = q[2];
              q[0] = q0 + out[0][3 * j + i];
              q[1] = q1 + out[1][3 * j + i];
              q[2] = q2 + out[2][3 * j + i];
            }
          }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
    tsync<kWaves>();
    flush_plane<T, kWaves>(a, tile, tb, (int)(2 * ek), win[(2 * kz) % 3], y, fbx, fby, fbz);
    flush_plane<T, kWaves>(a, tile, tb, (int)(2 * ek + 1), win[(2 * kz + 1) % 3], y, fbx, fby, fbz);
    tsync<kWaves>();
  }
  flush_plane<T, kWaves>(a, tile, tb, 2 * (tb.z0 + tb.nzt), win[(2 * tb.nzt) % 3], y, fbx, fby, fbz);
}

template <typename T, bool kMask>
__global__ void __launch_bounds__(64)
    a11_tile_kernel(TileArgs a, const T *__restrict__ xc, const T *__restrict__ eta,
                    const uint8_t *__restrict__ bcn, const T *__restrict__ u, T *__restrict__ y,
                    T *__restrict__ fbx, T *__restrict__ fby, T *__restrict__ fbz) {
  __shared__ T sh[3][kSlots][sh_cols<T>()];
  __shared__ T win[3][3 * kWinNodes];
  tile_march<T, kMask>(a, xcd_tile(blockIdx.x, a.ntiles), xc, eta, bcn, u, y, fbx, fby, fbz, sh, win);
}

// The same z-march with kW tiles per work-group (one wave each, own LDS
// buffers): work-group g takes tiles kW g .. kW g + kW - 1 of the x-fastest
// order, work-groups mapped to XCDs as above.  A wave past the last tile
// returns at once; no barrier spans waves.
template <typename T, bool kMask, int kWaves>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 2 : 1)))
    a11_tile_wg_kernel(TileArgs a, long nwg, const T *__restrict__ xc, const T *__restrict__ eta,
                       const uint8_t *__restrict__ bcn, const T *__restrict__ u, T *__restrict__ y,
                       T *__restrict__ fbx, T *__restrict__ fby, T *__restrict__ fbz) {
  __shared__ T sh[kWaves][3][kSlots][sh_cols<T>()];
  __shared__ T win[kWaves][3][3 * kWinNodes];
  const int w = (int)(threadIdx.x >> 6);
  const long tile = xcd_tile(blockIdx.x, nwg) * kWaves + w;
  if (tile >= a.ntiles) return;
  tile_march<T, kMask, false, kWaves>(a, tile, xc, eta, bcn, u, y, fbx, fby, fbz, sh[w], win[w]);
}

// Saddle-point MatMult: the A11 z-march with the pressure coupling; y holds
// the velocity part, yp the pressure part (4 per element, written once).
template <typename T>
__global__ void __launch_bounds__(64)
    stokes_tile_kernel(TileArgs a, const T *__restrict__ xc, const T *__restrict__ eta,
                       const uint8_t *__restrict__ bcn, const T *__restrict__ u, const T *__restrict__ p,
                       T *__restrict__ y, T *__restrict__ yp, T *__restrict__ fbx, T *__restrict__ fby,
                       T *__restrict__ fbz) {
  __shared__ T sh[3][kSlots][sh_cols<T>()];
  __shared__ T win[3][3 * kWinNodes];
  __shared__ T sL[3][kEPW];
  tile_march<T, true, true>(a, xcd_tile(blockIdx.x, a.ntiles), xc, eta, bcn, u, y, fbx, fby, fbz, sh, win, p, yp,
                            sL);
}

// The same z-march, software-pipelined across layers: the raw node plane of
// layer k+1 is loaded while layer k's backward stage runs, its viscosity
// while layer k's window sums run, and layer k's completed node planes are
// flushed after layer k+1's forward stage, so no global load is waited on
// right after it is issued.
template <typename T, bool kMask>
__global__ void __launch_bounds__(64)
    a11_tile_pf_kernel(TileArgs a, const T *__restrict__ xc, const T *__restrict__ eta,
                       const uint8_t *__restrict__ bcn, const T *__restrict__ u, T *__restrict__ y,
                       T *__restrict__ fbx, T *__restrict__ fby, T *__restrict__ fbz) {
  __shared__ T sh[3][kSlots][sh_cols<T>()];
  __shared__ T win[3][3 * kWinNodes];
  const long tile = xcd_tile(blockIdx.x, a.ntiles);
  const TileBox tb = tile_box(a, tile);
  const int lane = threadIdx.x;
  const int c = lane / kEPW;
  const int le = lane - c * kEPW;
  const int cp = c < 3 ? c : 2;
  const bool writer = c < 3;
  const int lx = le % a.TX, ly = le / a.TX;
  const bool live = writer && (le < a.TX * a.TY) && (lx < tb.nxt) && (ly < tb.nyt);
  const int ex = tb.x0 + min(lx, tb.nxt - 1), ey = tb.y0 + min(ly, tb.nyt - 1);
  const int wX = 2 * tb.nxt + 1;
  const long ncol = 2L * ex + a.X * (2L * ey);  // node (0, 0, 0) of element (ex, ey, 0)

  PlaneRaw<T> r;
  load_plane_nodes<T, kMask>(r, xc, u, bcn, ncol + a.XY * (2L * tb.z0 + cp), a.X);
  load_plane_eta<T>(r, eta + tq_index(tile, a.ZC, 0, 9 * cp, le), kEPW);
  for (int t = lane; t < 9 * kWinNodes; t += 64) (&win[0][0])[t] = T(0);
  __syncthreads();

  for (int kz = 0; kz < tb.nzt; kz++) {
    const long ek = tb.z0 + kz;
    T out[3][9];
    {
      T Xq[3][9], Uq[3][9];
      plane_forward<T, kMask>(cp, le, writer, r, sh, Xq, Uq);
      plane_qp<T>(cp, le, writer, Xq, Uq, r.eta, sh);
    }
    plane_backward<T>(cp, le, sh, out);
    // next layer's loads: in flight during the window sums and the flush
    __builtin_amdgcn_sched_barrier(0);
    if (kz + 1 < tb.nzt) {
      load_plane_nodes<T, kMask>(r, xc, u, bcn, ncol + a.XY * (2 * ek + 2 + cp), a.X);
      load_plane_eta<T>(r, eta + tq_index(tile, a.ZC, kz + 1, 9 * cp, le), kEPW);
    }
    __builtin_amdgcn_sched_barrier(0);
    // window sums, as in a11_tile_kernel
    {
      T *w = win[(2 * kz + cp) % 3] + 3 * ((2 * ly) * wX + 2 * lx);
#pragma unroll
      for (int j = 0; j < 3; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) {
          if (live) {
            T *q = w + 3 * (j * wX + i);
            const T q0 = q[0], q1 = q[1], q2 = q[2];
            q[0] = q0 + out[0][3 * j + i];
            q[1] = q1 + out[1][3 * j + i];
            q[2] = q2 + out[2][3 * j + i];
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();
    flush_plane<T>(a, tile, tb, (int)(2 * ek), win[(2 * kz) % 3], y, fbx, fby, fbz);
    flush_plane<T>(a, tile, tb, (int)(2 * ek + 1), win[(2 * kz + 1) % 3], y, fbx, fby, fbz);
    __syncthreads();
  }
  flush_plane<T>(a, tile, tb, 2 * (tb.z0 + tb.nzt), win[(2 * tb.nzt) % 3], y, fbx, fby, fbz);
}

// ---------------------------------------------------------------------------
// Partial assembly (kernel variant 2): per quadrature point the 9 entries of
// Ah = sqrt(2 w eta / det) * adj(J) (adj(J) = det * J^-1, rows k: d xi / d x_k
// scaled), stored once per coefficient/tiling change.  The pointwise action
// of MFStokesWrapper_A11_Tensor (QuadratureAction, tensor.c:127-179) is then
//   dv = sym(Gu Ah^T) Ah,   Gu[j][l] = d u_l / d xi_j,
// which equals w detJ (2 eta sym(grad u)) G^T with G = J^-1.  Layout follows
// the MatMult tiles so a lane group reads 21 consecutive values:
//   pa[((((tile * ZC + kz) * 27 + q) * 9 + m) * 21) + le].
// ---------------------------------------------------------------------------
__device__ __forceinline__ long pa_index(long tile, int ZC, int kz, int q, int m, int le) {
  return ((((tile * ZC + kz) * 27 + q) * 9 + m) * (long)kEPW) + le;
}

template <typename T>
__global__ void __launch_bounds__(256)
    pa_build_kernel(TileArgs a, long ntiles, const double *__restrict__ xc,
                    const double *__restrict__ eta, T *__restrict__ pa, int *__restrict__ bad) {
  const long total = ntiles * a.ZC * 27L * kEPW;
  for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
    const int le = (int)(t % kEPW);
    const int q = (int)((t / kEPW) % 27);
    const int kz = (int)((t / (27L * kEPW)) % a.ZC);
    const long tile = t / (27L * kEPW * a.ZC);
    const TileBox tb = tile_box(a, tile);
    if (kz >= tb.nzt) continue;
    const int lx = le % a.TX, ly = le / a.TX;
    const int ex = tb.x0 + min(lx, tb.nxt - 1), ey = tb.y0 + min(ly, tb.nyt - 1);
    const long ek = tb.z0 + kz;
    const long e = ex + (long)a.mx * (ey + (long)a.my * ek);
    const int qa = q % 3, qb = (q / 3) % 3, qc = q / 9;
    // M[j][d] = d x_d / d xi_j at the quadrature point
    double M[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    const long base = 2L * ex + a.X * (2L * ey) + a.XY * (2L * ek);
    for (int k = 0; k < 3; k++)
      for (int j = 0; j < 3; j++)
        for (int i = 0; i < 3; i++) {
          const long n = base + i + a.X * j + a.XY * k;
          const double g0 = kD[qa][i] * kB[qb][j] * kB[qc][k];
          const double g1 = kB[qa][i] * kD[qb][j] * kB[qc][k];
          const double g2 = kB[qa][i] * kB[qb][j] * kD[qc][k];
          for (int d = 0; d < 3; d++) {
            const double x = xc[3 * n + d];
            M[0][d] += g0 * x;
            M[1][d] += g1 * x;
            M[2][d] += g2 * x;
          }
        }
    double A[3][3];
    A[0][0] = M[1][1] * M[2][2] - M[2][1] * M[1][2];
    A[0][1] = M[2][1] * M[0][2] - M[0][1] * M[2][2];
    A[0][2] = M[0][1] * M[1][2] - M[1][1] * M[0][2];
    A[1][0] = M[2][0] * M[1][2] - M[1][0] * M[2][2];
    A[1][1] = M[0][0] * M[2][2] - M[2][0] * M[0][2];
    A[1][2] = M[1][0] * M[0][2] - M[0][0] * M[1][2];
    A[2][0] = M[1][0] * M[2][1] - M[2][0] * M[1][1];
    A[2][1] = M[2][0] * M[0][1] - M[0][0] * M[2][1];
    A[2][2] = M[0][0] * M[1][1] - M[1][0] * M[0][1];
    const double det = M[0][0] * A[0][0] + M[0][1] * A[1][0] + M[0][2] * A[2][0];
    const double s = 2.0 * kW[qa] * kW[qb] * kW[qc] * eta[(long)q * a.nel + e] / det;
    if (!(s > 0.0) || !isfinite(s)) *bad = 1;
    const double r = sqrt(fabs(s));
    for (int k = 0; k < 3; k++)
      for (int j = 0; j < 3; j++) pa[pa_index(tile, a.ZC, kz, q, 3 * k + j, le)] = (T)(r * A[k][j]);
  }
}

// Pointwise stage with stored geometry (see above); same exchange protocol
// as plane_qp with the velocity in slots 0..26 of a 27-slot buffer: on
// return slots 9l+p hold the zeta components, W the xi/eta accumulations.
template <typename T>
__device__ __forceinline__ void plane_qp_pa(int cp, int le, bool writer, const T Uq[3][9],
                                            const T *__restrict__ pal, T (*sh)[27][kEPW],
                                            T W[3][9]) {
  T dz[3];
#pragma unroll
  for (int k = 0; k < 3; k++) dz[k] = sel3<T>(cp, kD[0][k], kD[1][k], kD[2][k]);
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int p = 0; p < 9; p++) W[l][p] = T(0);
  T An[9];
#pragma unroll
  for (int m = 0; m < 9; m++) An[m] = pal[m * kEPW];
#pragma unroll
  for (int b = 0; b < 3; b++)
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int p = 3 * b + a;
      T Ah[9];
#pragma unroll
      for (int m = 0; m < 9; m++) Ah[m] = An[m];
      if (p < 8) {
#pragma unroll
        for (int m = 0; m < 9; m++) An[m] = pal[((p + 1) * 9 + m) * kEPW];
      }
      T Gu[3][3];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        Gu[0][d] = cdot<T>(a, Uq[d][3 * b], Uq[d][3 * b + 1], Uq[d][3 * b + 2]);
        Gu[1][d] = cdot<T>(b, Uq[d][a], Uq[d][3 + a], Uq[d][6 + a]);
        Gu[2][d] = dz[0] * sh[0][9 * d + p][le] + dz[1] * sh[1][9 * d + p][le] +
                   dz[2] * sh[2][9 * d + p][le];
      }
      // gh[k][l] = sum_j Gu[j][l] Ah[k][j]; sg = sym(gh)
      T gh[3][3];
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int l = 0; l < 3; l++)
          gh[k][l] = Gu[0][l] * Ah[3 * k] + Gu[1][l] * Ah[3 * k + 1] + Gu[2][l] * Ah[3 * k + 2];
      T sg[3][3];
      sg[0][0] = gh[0][0];
      sg[1][1] = gh[1][1];
      sg[2][2] = gh[2][2];
      sg[0][1] = sg[1][0] = T(0.5) * (gh[0][1] + gh[1][0]);
      sg[0][2] = sg[2][0] = T(0.5) * (gh[0][2] + gh[2][0]);
      sg[1][2] = sg[2][1] = T(0.5) * (gh[1][2] + gh[2][1]);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int l = 0; l < 3; l++) {
        const T dv0 = sg[0][l] * Ah[0] + sg[1][l] * Ah[3] + sg[2][l] * Ah[6];
        const T dv1 = sg[0][l] * Ah[1] + sg[1][l] * Ah[4] + sg[2][l] * Ah[7];
        const T dv2 = sg[0][l] * Ah[2] + sg[1][l] * Ah[5] + sg[2][l] * Ah[8];
#pragma unroll
        for (int r = 0; r < 3; r++) {
          if (a != 1 || r != 1) W[l][3 * b + r] += (T)kC[a][r] * dv0;
          if (b != 1 || r != 1) W[l][3 * r + a] += (T)kC[b][r] * dv1;
        }
        if (writer) sh[cp][9 * l + p][le] = dv2;
      }
      __builtin_amdgcn_wave_barrier();
    }
  __syncthreads();
}

// MatMult with stored geometry: the z-march of a11_tile_kernel with only the
// velocity exchanged (27 LDS slots) and the backward zeta stage in two
// passes over the same slots.
template <typename T, bool kMask>
__global__ void __launch_bounds__(64)
    a11_tile_pa_kernel(TileArgs a, const T *__restrict__ pa, const uint8_t *__restrict__ bcn,
                       const T *__restrict__ u, T *__restrict__ y, T *__restrict__ fbx,
                       T *__restrict__ fby, T *__restrict__ fbz) {
  __shared__ T sh[3][27][kEPW];
  __shared__ T win[3][3 * kWinNodes];
  const long tile = xcd_tile(blockIdx.x, a.ntiles);
  const TileBox tb = tile_box(a, tile);
  const int lane = threadIdx.x;
  const int c = lane / kEPW;
  const int le = lane - c * kEPW;
  const int cp = c < 3 ? c : 2;
  const bool writer = c < 3;
  const int lx = le % a.TX, ly = le / a.TX;
  const bool live = writer && (le < a.TX * a.TY) && (lx < tb.nxt) && (ly < tb.nyt);
  const int ex = tb.x0 + min(lx, tb.nxt - 1), ey = tb.y0 + min(ly, tb.nyt - 1);
  const int wX = 2 * tb.nxt + 1;
  const long ncol = 2L * ex + a.X * (2L * ey);

  for (int t = lane; t < 9 * kWinNodes; t += 64) (&win[0][0])[t] = T(0);
  __syncthreads();

  T bz[3], bt[3], dt[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    bz[k] = sel3<T>(cp, kB[0][k], kB[1][k], kB[2][k]);
    bt[k] = sel3<T>(cp, kB[k][0], kB[k][1], kB[k][2]);
    dt[k] = sel3<T>(cp, kD[k][0], kD[k][1], kD[k][2]);
  }

  for (int kz = 0; kz < tb.nzt; kz++) {
    const long ek = tb.z0 + kz;
    const long base = ncol + a.XY * (2 * ek + cp);
    const T *pal = pa + pa_index(tile, a.ZC, kz, 9 * cp, 0, le);
    // forward: masked velocity plane, in-plane interpolation, zeta exchange
    T Uq[3][9];
    {
      T g[3][9];
#pragma unroll
      for (int j = 0; j < 3; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) {
          const long node = base + i + a.X * j;
          const unsigned m = kMask ? (unsigned)bcn[node] : 0u;
#pragma unroll
          for (int d = 0; d < 3; d++) {
            const T v = u[3 * node + d];
            g[d][3 * j + i] = ((m >> d) & 1u) ? T(0) : v;
          }
        }
      T V[3][9];
      interp_plane<T>(g, V);
      if (writer) {
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
          for (int p = 0; p < 9; p++) sh[cp][9 * d + p][le] = V[d][p];
      }
    }
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
      for (int p = 0; p < 9; p++)
        Uq[d][p] = bz[0] * sh[0][9 * d + p][le] + bz[1] * sh[1][9 * d + p][le] +
                   bz[2] * sh[2][9 * d + p][le];
    T W[3][9];
    plane_qp_pa<T>(cp, le, writer, Uq, pal, sh, W);
    // backward zeta stage, pass 1: the zeta components
    T Y[3][9];
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int p = 0; p < 9; p++)
        Y[l][p] = dt[0] * sh[0][9 * l + p][le] + dt[1] * sh[1][9 * l + p][le] +
                  dt[2] * sh[2][9 * l + p][le];
    __syncthreads();
    if (writer) {
#pragma unroll
      for (int l = 0; l < 3; l++)
#pragma unroll
        for (int p = 0; p < 9; p++) sh[cp][9 * l + p][le] = W[l][p];
    }
    __syncthreads();
    // pass 2: the xi/eta accumulations
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int p = 0; p < 9; p++)
        Y[l][p] += bt[0] * sh[0][9 * l + p][le] + bt[1] * sh[1][9 * l + p][le] +
                   bt[2] * sh[2][9 * l + p][le];
    __syncthreads();
    T out[3][9];
#pragma unroll
    for (int l = 0; l < 3; l++) interp_plane_t<T>(Y[l], out[l]);
    {
      T *w = win[(2 * kz + cp) % 3] + 3 * ((2 * ly) * wX + 2 * lx);
#pragma unroll
      for (int j = 0; j < 3; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) {
          if (live) {
            T *q = w + 3 * (j * wX + i);
            const T q0 = q[0], q1 = q[1], q2 = q[2];
            q[0] = q0 + out[0][3 * j + i];
            q[1] = q1 + out[1][3 * j + i];
            q[2] = q2 + out[2][3 * j + i];
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();
    flush_plane<T>(a, tile, tb, (int)(2 * ek), win[(2 * kz) % 3], y, fbx, fby, fbz);
    flush_plane<T>(a, tile, tb, (int)(2 * ek + 1), win[(2 * kz + 1) % 3], y, fbx, fby, fbz);
    __syncthreads();
  }
  flush_plane<T>(a, tile, tb, 2 * (tb.z0 + tb.nzt), win[(2 * tb.nzt) % 3], y, fbx, fby, fbz);
}

// One tile per work-group of kFaceThreads, one face node per thread: the
// tall tiles of long z-chunks have 400-800 lower-face nodes, which a single
// wave would walk one dependent load/store round after another.
constexpr int kFaceThreads = 256;

// It adds the face sums and copies the Dirichlet rows y = x
// (BCListInsertDirichlet_MatMult with scale 1), which the face sums leave alone,
// in work-groups of their own: beside the sums and not after them (64^3: 13 us for
// both, apart 5 us more; copied by the lane kernel as it writes the other rows
// 16 us more).
constexpr int kCopyGroup = 4 * kFaceThreads;  // rows per work-group
template <typename T>
__global__ void __launch_bounds__(kFaceThreads)
    a11_face_copy_kernel(TileArgs a, const T *__restrict__ fbx, const T *__restrict__ fby, const T *__restrict__ fbz,
                         T *__restrict__ y, const uint8_t *__restrict__ bcn, const long *__restrict__ bcidx, long nbc,
                         const T *__restrict__ x) {
  // (the copies first: they are short, and the face sums fill up behind them)
  const long g = (long)blockIdx.x - ((long)gridDim.x - a.ntiles);
  if (g >= 0) {
    face_sum<T, true>(a, xcd_tile(g, a.ntiles), fbx, fby, fbz, y, bcn);
    return;
  }
  constexpr int kN = kCopyGroup / kFaceThreads;
  const long i0 = (long)kCopyGroup * blockIdx.x + threadIdx.x;
  long idx[kN];
  T v[kN];
#pragma unroll
  for (int k = 0; k < kN; k++) idx[k] = bcidx[min(i0 + kFaceThreads * k, nbc - 1)];
#pragma unroll
  for (int k = 0; k < kN; k++) v[k] = x[idx[k]];
#pragma unroll
  for (int k = 0; k < kN; k++) y[idx[k]] = v[k];
}

// RowUpdates by what they read besides b: nothing (a residual), dinv, or dinv
// and prev
enum UpdateKind { kUpResidual, kUpFirst, kUpStep };

// One row: all it reads is requested before any of it is used (out may be prev
// or the element sums, the same row of them).
template <typename T, UpdateKind kUp>
struct UpdateRow {
  T b, x, dinv, prev;
  unsigned m;
  __device__ __forceinline__ void load(const RowUpdate<T> &up, long i, const T *__restrict__ x_, unsigned bits) {
    m = bits;
    b = up.b[i];
    x = x_[i];
    if (kUp != kUpResidual) dinv = up.dinv[i];
    if (kUp == kUpStep) prev = up.prev[i];
  }
  __device__ __forceinline__ void store(const RowUpdate<T> &up, long i, unsigned d, T sum) const {
    T o = b - (((m >> d) & 1u) ? x : sum);
    if (kUp != kUpResidual) o = up.os * (o * dinv);
    if (kUp == kUpStep) o += up.om1 * prev;
    if (kUp != kUpResidual) o += up.om * x;
    if (up.out64) ((double *)up.out)[i] = (double)o;
    else ((T *)up.out)[i] = o;
  }
};

// A RowUpdate with the face sums added on the way: one pass over the vectors in
// place of the face pass and the update (FP64 32^3: 8.0 us, apart 14.2 us; 48 x
// 48 x 32 FP32 10.0 and 16 us; 64^3 47 us, apart 44 us but one launch more).
// Bound by memory: up to five vectors in and one out.  A thread takes one row of
// the two node planes 2 ek and 2 ek + 1 of an element layer (of the top layer:
// three): its place in the tiles is worked out once, and all loads of both are
// in flight together (all planes of a tile layer two at a time: 56 us).  Each
// XCD has a slab of its own, as in the element kernel (52 us without).  r: the
// element kernel's sums.
template <typename T, UpdateKind kUp>
__global__ void __launch_bounds__(256)
    a11_update_kernel(TileArgs a, unsigned gx, const T *__restrict__ fbx, const T *__restrict__ fby,
                      const T *__restrict__ fbz, const T *r, const uint8_t *__restrict__ bcn, const T *__restrict__ x,
                      RowUpdate<T> up) {
  const unsigned blk = (unsigned)xcd_tile(blockIdx.x, gridDim.x), ek = blk / gx;
  const unsigned t = (blk - ek * gx) * 256u + threadIdx.x, X = (unsigned)a.X;
  if (t >= 3u * (unsigned)a.XY) return;
  const unsigned m = t / 3u, d = t - 3u * m, J = m / X, I = m - J * X;
  const int tx = min((int)(I / (2u * a.TX)), a.ntx - 1), ty = min((int)(J / (2u * a.TY)), a.nty - 1);
  const int il = (int)I - 2 * a.TX * tx, jl = (int)J - 2 * a.TY * ty;
  const bool hx = tx > 0 && il == 0, hy = ty > 0 && jl == 0;
  const int tz = (int)ek / a.ZC, k0 = 2 * ((int)ek - a.ZC * tz);
  const int sx = 3 * (2 * a.TY + 1), sy = 3 * (2 * a.TX + 1);
  const long tile = tx + (long)a.ntx * (ty + (long)a.nty * tz), below = (long)a.ntx * a.nty;
  // the neighbours' upper faces at this row, in the order of face_sum
  const T *const p0 = fbx + 3 * ((tile - 1 - a.ntx) * a.fbx_n + 2 * a.TY) + d,
                 *const p1 = fby + 3 * ((tile - a.ntx) * a.fby_n + il) + d,
                 *const p2 = fbx + 3 * ((tile - 1) * a.fbx_n + jl) + d;
  auto faces = [&](long kx, long ky) {
    const T v0 = hx && hy ? p0[kx] : T(0), v1 = hy ? p1[ky] : T(0), v2 = hx ? p2[kx] : T(0);
    return v0 + v1 + v2;
  };
  const long n0 = m + a.XY * (2L * ek);
  auto planes = [&](auto first, auto count) {
    constexpr int kF = decltype(first)::value, kN = decltype(count)::value;
    UpdateRow<T, kUp> u[kN];
    T s[kN], f[kN];
#pragma unroll
    for (int p = 0; p < kN; p++) {
      const long n = n0 + a.XY * (kF + p);
      s[p] = r[3 * n + d];
      u[p].load(up, 3 * n + d, x, bcn[n]);
      f[p] = T(0);
    }
    if (kF == 0 && k0 == 0 && tz > 0)  // the tiles below
      f[0] = faces(2L * a.ZC * sx - 3 * below * a.fbx_n, 2L * a.ZC * sy - 3 * below * a.fby_n) +
             fbz[3 * ((tile - below) * a.fbz_n + il + (long)(2 * a.TX + 1) * jl) + d];
    if (hx || hy) {
#pragma unroll
      for (int p = 0; p < kN; p++) f[p] += faces((long)sx * (k0 + kF + p), (long)sy * (k0 + kF + p));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < kN; p++) u[p].store(up, 3 * (n0 + a.XY * (kF + p)) + d, d, s[p] + f[p]);
  };
  planes(std::integral_constant<int, 0>(), std::integral_constant<int, 2>());
  if ((int)ek == a.mz - 1) planes(std::integral_constant<int, 2>(), std::integral_constant<int, 1>());
}

#include "a11_col.h"

// ---------------------------------------------------------------------------
// Batched MatMult: many independent boxes in one launch per stage.  Every box
// takes the column kernel or, too large for it or tiled by the caller, the tile
// kernel.  A work item is (box, tile), or (box, wave) and then (box, 256 nodes);
// every box has its own sizes, coefficients, Dirichlet data and buffers
// (BoxDesc, in device memory).
// ---------------------------------------------------------------------------
struct BoxDesc {
  TileArgs a;
  ColArgs c;
  const void *xc, *eta;  // coordinates; viscosity, tile-ordered for the tile kernel
  const uint8_t *bcn;
  const long *bcidx;
  long nbc;              // 0 for the column kernel, whose sums copy the Dirichlet rows
  void *fbx, *fby, *fbz; // fbx: the element sums of the column kernel
};

template <typename T>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
    a11_col_batch_kernel(const BoxDesc *__restrict__ boxes, const int2 *__restrict__ work, long nwork,
                         const T *const *__restrict__ xs, const int *__restrict__ active) {
  __shared__ T sm[18][64];
  const int2 w = work[xcd_tile(blockIdx.x, nwork)];
  if (active && !active[w.x]) return;  // whole work-group: the box is idle
  const BoxDesc &d = boxes[w.x];
  col_wave<T>(d.c, (unsigned)w.y, (const T *)d.xc, (const T *)d.eta, d.bcn, xs[w.x], (T *)d.fbx, sm);
}

template <typename T>
__global__ void __launch_bounds__(kColSumThreads)
    col_sum_batch_kernel(const BoxDesc *__restrict__ boxes, const int2 *__restrict__ work, long nwork,
                         const T *const *__restrict__ xs, T *const *__restrict__ ys, const int *__restrict__ active) {
  const int2 w = work[xcd_tile(blockIdx.x, nwork)];
  if (active && !active[w.x]) return;
  const BoxDesc &d = boxes[w.x];
  col_node<T>(d.c, (unsigned)(w.y * kColSumThreads) + threadIdx.x, (const T *)d.fbx, ys[w.x], d.bcn, xs[w.x]);
}

template <typename T>
__global__ void __launch_bounds__(64)
    a11_tile_batch_kernel(const BoxDesc *__restrict__ boxes, const int2 *__restrict__ work, long nwork,
                          const T *const *__restrict__ xs, T *const *__restrict__ ys,
                          const int *__restrict__ active) {
  __shared__ T sh[3][kSlots][sh_cols<T>()];
  __shared__ T win[3][3 * kWinNodes];
  const int2 w = work[xcd_tile(blockIdx.x, nwork)];
  if (active && !active[w.x]) return;  // whole work-group: the box is idle
  const BoxDesc &d = boxes[w.x];
  tile_march<T, true>(d.a, w.y, (const T *)d.xc, (const T *)d.eta, d.bcn, xs[w.x], ys[w.x], (T *)d.fbx,
                      (T *)d.fby, (T *)d.fbz, sh, win);
}

template <typename T>
__global__ void __launch_bounds__(64)
    a11_face_batch_kernel(const BoxDesc *__restrict__ boxes, const int2 *__restrict__ work, long nwork,
                          T *const *__restrict__ ys, const int *__restrict__ active) {
  const int2 w = work[xcd_tile(blockIdx.x, nwork)];
  if (active && !active[w.x]) return;
  const BoxDesc &d = boxes[w.x];
  face_sum<T>(d.a, w.y, (const T *)d.fbx, (const T *)d.fby, (const T *)d.fbz, ys[w.x]);
}

// Dirichlet rows y = x of every box (blockIdx.y = box)
template <typename T>
__global__ void bc_copy_batch_kernel(const BoxDesc *__restrict__ boxes, const T *const *__restrict__ xs,
                                     T *const *__restrict__ ys, const int *__restrict__ active) {
  if (active && !active[blockIdx.y]) return;
  const BoxDesc &d = boxes[blockIdx.y];
  const T *x = xs[blockIdx.y];
  T *y = ys[blockIdx.y];
  for (long k = blockIdx.x * (long)blockDim.x + threadIdx.x; k < d.nbc; k += (long)gridDim.x * blockDim.x) {
    const long g = d.bcidx[k];
    y[g] = x[g];
  }
}

#include "a11_lane.h"

TileArgs tile_args(const ptmf_op_s *op) {
  const Box &b = op->box;
  TileArgs a;
  a.mx = b.mx; a.my = b.my; a.mz = b.mz;
  a.X = b.X; a.XY = b.X * b.Y; a.nel = b.nel;
  a.TX = op->tiling.TX; a.TY = op->tiling.TY; a.ZC = op->tiling.ZC;
  a.ntx = op->tiling.ntx; a.nty = op->tiling.nty;
  a.ntiles = op->tiling.ntiles;
  a.fbx_n = (long)(2 * a.TY + 1) * (2 * a.ZC + 1);
  a.fby_n = (long)(2 * a.TX + 1) * (2 * a.ZC + 1);
  a.fbz_n = (long)(2 * a.TX + 1) * (2 * a.TY + 1);
  return a;
}

// The lane kernel's decomposition of box b in precision T; false where the tile
// kernel runs instead (as it does on a mesh that is not rectilinear, or with a
// tiling, variant or tiles per work-group of the caller's choice): with arrays
// past the 32-bit offsets of the lane kernel, in FP32 with more than 64 elements in
// a direction, and where the tile kernel is faster.  The FP32 line is no choice by
// speed or accuracy: larger boxes keep the tile kernel's results, which err by its
// FP32 interpolation of the coordinates (1.9e-5 of the largest at 64^3, 2.4e-5 at
// 65^3, 5.1e-5 at 128^3; this kernel 2.3e-7 at each) and take 105 us at 65^3 and
// 746 us at 128^3 where this kernel takes 56 and 323 us.
// The costs are microseconds per round of one wave on each of the 1024 SIMDs,
// times the layers a wave marches through.  Measured on boxes from 8^3 to
// 96 x 96 x 48, FP64: 14 us per layer of 64 elements (lane) and 14.6 us per
// layer of 20 (tile); FP32, two waves per SIMD: 14.2 and 15.7 us for both, 10 and
// 10.5 us with one; the lane kernel's first and last planes add 0.57 (0.45) of a
// layer.  So the tile kernel keeps the boxes that it takes in one round (16^3: 13.1
// us against 14.9 us; 20^3: 14.7 and 15.0 us; this concerns the saddle point, the
// MatMult having the column kernel there), and the lane kernel has the rest (28^3:
// 16.5 us against 28.6 us, FP32 13.2 and 13.7 us; 48 x 48 x 32: 29 and 61 us, FP32
// 17 and 27 us; 64^3: 56 and 175 us, FP32 31 and 77 us).
//
// The column kernel (a11_col.h) has the boxes of up to 100,000 elements, whose
// element sums fit 64 MiB, on meshes that are not rectilinear (MatMult against
// the tile kernel's: 8^3 7.8 and 16.5 us, 24^3 15 and 21 us, 45 x 37 x 29 40 and
// 61 us, 48 x 48 x 32 57 and 71 us, FP32 34 and 36 us), and the small rectilinear
// ones: its MatMult takes 6.6 + E / 1390 us (FP32 6.9 + E / 2670), the lane kernel's
// that of its kernel above and in FP32 3.7 us (in FP64 the kernel's time falls
// short of the model by its face pass): 27^3 19.6 against 21.8 us, 28^3 22.4 and
// 21.7 us, 30^3 24 and 22 us, 32^3 30 and 23 us; FP32 28^3 15 and 18 us, 31^3 17.7
// and 18.4 us, 32^3 20 and 18 us.
constexpr long kColDoubles = 8L << 20;

template <typename T>
double col_cost(long nel) {
  return sizeof(T) == 8 ? 6.6 + 0.72e-3 * (double)nel : 6.9 + 0.375e-3 * (double)nel;
}

template <typename T>
double lane_rounds(long waves, double one, double two) {
  const long r = (waves + 1023) / 1024;
  return sizeof(T) == 8 ? one * (double)r : two * (double)(r / 2) + one * (double)(r % 2);
}

// kernel: the one the lane kernel would take the place of
enum LaneOther { kOtherTile, kOtherCol };

template <typename T>
bool lane_plan(const Box &b, const Tiling &t, LaneOther other, TileArgs &a) {
  constexpr bool f64 = sizeof(T) == 8;
  if (!f64 && std::max(b.mx, std::max(b.my, b.mz)) > 64) return false;
  a.mx = b.mx; a.my = b.my; a.mz = b.mz;
  a.X = b.X; a.XY = b.X * b.Y; a.nel = b.nel;
  a.TX = a.TY = kLT;
  a.ntx = (b.mx + kLT - 1) / kLT;
  a.nty = (b.my + kLT - 1) / kLT;
  const long txy = (long)a.ntx * a.nty;
  double best = 1e300;
  for (int zc = 1; zc <= b.mz && zc <= kLMaxZ; zc++) {
    const long nt = txy * ((b.mz + zc - 1) / zc);
    const double cost = (zc + (f64 ? 0.57 : 0.45)) * lane_rounds<T>(nt, f64 ? 14.0 : 10.0, 14.2);
    if (cost < best) {
      best = cost;
      a.ZC = zc;
      a.ntiles = nt;
    }
  }
  if (other == kOtherTile && best >= t.ZC * lane_rounds<T>(t.ntiles, f64 ? 14.6 : 10.5, 15.7)) return false;
  if (other == kOtherCol && best + (f64 ? 0.0 : 3.7) >= col_cost<T>(b.nel)) return false;
  a.fbx_n = a.fby_n = (long)kLRows * (2 * a.ZC + 1);
  a.fbz_n = kLRows * kLRows;
  // byte offsets of the 27 quadrature points' viscosities and of 17 node rows
  return 8 * 27 * b.nel < (1L << 32) && lane_fits(b) && a.ntiles < (1L << 31);
}

// the same for an operator with face buffers of fb_doubles
template <typename T>
bool lane_tiles(const ptmf_op_s *op, long fb_doubles, LaneOther other, TileArgs &a) {
  return op->rect && op->tiling_default && op->wg_tiles == 1 && lane_plan<T>(op->box, op->tiling, other, a) &&
         face_buffer_doubles(kLT, kLT, a.ZC, a.ntiles) <= fb_doubles;
}

long col_doubles(const Box &b) { return 81 * b.nel <= kColDoubles ? 81 * b.nel : 0; }

ColArgs col_args(const Box &b) {
  const unsigned ne = (unsigned)b.nel;
  return ColArgs{(unsigned)b.mx, (unsigned)b.my, (unsigned)b.mz, ne, (ne + kColElems - 1) / kColElems};
}

// the column kernel, with a buffer of fb_doubles, where the lane kernel is not chosen
bool col_box(const ptmf_op_s *op, long fb_doubles) {
  return op->tiling_default && op->wg_tiles == 1 && col_doubles(op->box) > 0 && col_doubles(op->box) <= fb_doubles;
}

// Is the mesh rectilinear?  Axis lines of the three directions first (mid
// nodes halfway between their neighbours, 2 m / h per element), then every
// node against the lines.  "Equal" is to 4 units of rounding of the largest
// coordinate of the direction: what a mesh generator's own rounding leaves,
// and what the general kernel's interpolation of the coordinates rounds off
// anyway.  *bad is cleared, and set when a check fails.
__global__ void __launch_bounds__(256)
    rect_axes_kernel(int mx, int my, int mz, long X, long XY, const double *__restrict__ xc, double *__restrict__ a64,
                     float *__restrict__ a32, double *__restrict__ tol, int *__restrict__ bad) {
  __shared__ double red[256];
  const int m[3] = {mx, my, mz};
  const long stride[3] = {3, 3 * X, 3 * XY};
  const double unit = ldexp(1.0, ilogb(xc[6] - xc[0]));  // m of a11_lane.h
  if (threadIdx.x == 0) {
    *bad = 0;
    a64[mx + my + mz] = unit;
    a32[mx + my + mz] = (float)unit;
  }
  for (int d = 0, first = 0; d < 3; first += m[d], d++) {
    double big = 0.0;
    for (int i = threadIdx.x; i <= 2 * m[d]; i += 256) big = fmax(big, fabs(xc[stride[d] * i + d]));
    red[threadIdx.x] = big;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
      __syncthreads();
    }
    const double t = 4.0 * 2.220446049250313e-16 * red[0];
    __syncthreads();
    if (threadIdx.x == 0) tol[d] = t;
    for (int e = threadIdx.x; e < m[d]; e += 256) {
      const double *x = xc + stride[d] * (2 * e) + d;
      const double x0 = x[0], x1 = x[stride[d]], x2 = x[2 * stride[d]], h = x2 - x0;
      if (!(fabs(x1 - 0.5 * (x0 + x2)) <= t) || !(fabs(h) > 64.0 * t) || !isfinite(h)) *bad = 1;
      a64[first + e] = 2.0 * unit / h;
      a32[first + e] = (float)(2.0 * unit / h);
    }
  }
}

__global__ void __launch_bounds__(256)
    rect_check_kernel(long n, int X, int Y, const double *__restrict__ xc, const double *__restrict__ tol,
                      int *__restrict__ bad) {
  const double t0 = tol[0], t1 = tol[1], t2 = tol[2];
  bool off = false;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += 256L * gridDim.x) {
    const int r = (int)(i / X), I = (int)(i - (long)r * X), K = r / Y, J = r - K * Y;
    const double *x = xc + 3 * i;
    off |= !(fabs(x[0] - xc[3L * I]) <= t0) || !(fabs(x[1] - xc[3L * X * J + 1]) <= t1) ||
           !(fabs(x[2] - xc[3L * X * Y * K + 2]) <= t2);
  }
  if (__any(off) && (threadIdx.x & 63) == 0) *bad = 1;
}

// lane_bc_word of every tile column of the lane kernels and node plane
__global__ void __launch_bounds__(64)
    bc_word_kernel(int mx, int my, int ntx, long X, long XY, long Z, const uint8_t *__restrict__ bcn,
                   unsigned *__restrict__ words) {
  const long col = blockIdx.x / Z, P = blockIdx.x - col * Z;
  const int tx = (int)(col % ntx), ty = (int)(col / ntx);
  const int x0 = kLT * tx, y0 = kLT * ty, wX = 2 * min(kLT, mx - x0) + 1, wY = 2 * min(kLT, my - y0) + 1;
  const int il = threadIdx.x / 3, d = threadIdx.x - 3 * il;
  unsigned w = 0;
  if (il < wX)
    for (int j = 0; j < wY; j++) w |= ((bcn[2 * x0 + il + X * (2 * y0 + j) + XY * P] >> d) & 1u) << j;
  words[64L * blockIdx.x + threadIdx.x] = w;
}

}  // namespace

int alloc_lane_data(ptmf_op_s *op) {
  // one allocation: the face buffers of A12 and the diagonal, 2 m / h and m in FP64
  // (and three tolerances) and in FP32, the classification's flag, the Dirichlet words
  const Box &b = op->box;
  const long na = b.mx + b.my + b.mz;
  const long planes = (long)((b.mx + kLT - 1) / kLT) * ((b.my + kLT - 1) / kLT) * b.Z;
  const long nf = node_face_doubles(b);
  PTMF_TRY(ptmf_malloc((void **)&op->lane_data, sizeof(double) * (nf + na + 4) + sizeof(float) * (na + 1) + sizeof(int) +
                                                    64 * sizeof(unsigned) * planes));
  op->node_faces = op->lane_data;
  op->node_faces_doubles = nf;
  op->ax64 = op->lane_data + nf;
  op->ax32 = (float *)(op->ax64 + na + 4);
  op->rect_bad = (int *)(op->ax32 + na + 1);
  op->bcword = (unsigned *)(op->rect_bad + 1);
  return PTMF_OK;
}

int mark_dirichlet_planes(ptmf_op_s *op) {
  const Box &b = op->box;
  const int ntx = (b.mx + kLT - 1) / kLT, nty = (b.my + kLT - 1) / kLT;
  const long n = (long)ntx * nty * b.Z;
  PTMF_CHECK(n < (1L << 31), PTMF_ERR_ARG, "set_dirichlet: mesh too large");
  bc_word_kernel<<<dim3((unsigned)n), 64, 0, op->stream>>>(b.mx, b.my, ntx, b.X, b.X * b.Y, b.Z, op->bcnode, op->bcword);
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

int classify_mesh(ptmf_op_s *op) {
  const Box &b = op->box;
  const long na = b.mx + b.my + b.mz;
  op->rect = 0;
  rect_axes_kernel<<<1, 256, 0, op->stream>>>(b.mx, b.my, b.mz, b.X, b.X * b.Y, op->d64.coords, op->ax64, op->ax32,
                                              op->ax64 + na + 1, op->rect_bad);
  long nb = (b.nnodes + 255) / 256;
  if (nb > 8192) nb = 8192;
  rect_check_kernel<<<dim3((unsigned)nb), 256, 0, op->stream>>>(b.nnodes, (int)b.X, (int)b.Y, op->d64.coords,
                                                               op->ax64 + na + 1, op->rect_bad);
  PTMF_HIP(hipGetLastError());
  int bad = 1;
  PTMF_HIP(hipMemcpyAsync(&bad, op->rect_bad, sizeof(int), hipMemcpyDeviceToHost, op->stream));
  PTMF_HIP(hipStreamSynchronize(op->stream));
  op->rect = !bad;
  return PTMF_OK;
}

long lane_face_doubles(const Box &b, const Tiling &t) {
  TileArgs a;
  long n = 0;
  if (lane_plan<double>(b, t, kOtherTile, a)) n = face_buffer_doubles(kLT, kLT, a.ZC, a.ntiles);
  if (lane_plan<float>(b, t, kOtherTile, a)) n = std::max(n, face_buffer_doubles(kLT, kLT, a.ZC, a.ntiles));
  return std::max(n, col_doubles(b));
}

long face_buffer_doubles(int TX, int TY, int ZC, long ntiles) {
  const long per = (long)(2 * TY + 1) * (2 * ZC + 1) + (long)(2 * TX + 1) * (2 * ZC + 1) +
                   (long)(2 * TX + 1) * (2 * TY + 1);
  return 3 * per * ntiles;
}

template <typename T>
int launch_a11(const ptmf_op_s *op, const T *u, T *y, bool mask_columns) {
  const Box &b = op->box;
  const OpData<T> &d = *(const OpData<T> *)(sizeof(T) == 8 ? (const void *)&op->d64
                                                           : (const void *)&op->d32);
  const long nblk = (b.nel + kEPW - 1) / kEPW;
  PTMF_CHECK(nblk < (1L << 31), PTMF_ERR_ARG, "a11: mesh too large (%ld blocks)", nblk);
  if (mask_columns)
    a11_atomic_kernel<T, true><<<dim3((unsigned)nblk), dim3(64), 0, op->stream>>>(
        b.mx, b.my, b.nel, b.X, b.X * b.Y, d.coords, d.eta, op->bcnode, u, y);
  else
    a11_atomic_kernel<T, false><<<dim3((unsigned)nblk), dim3(64), 0, op->stream>>>(
        b.mx, b.my, b.nel, b.X, b.X * b.Y, d.coords, d.eta, nullptr, u, y);
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

// (Re)build the tile-ordered viscosity for precision T when the coefficients
// or the tiling changed since the last build.
template <typename T>
int ensure_eta_tiled(ptmf_op_s *op) {
  const int ip = sizeof(T) == 8 ? 0 : 1;
  const Tiling &tl = op->tiling;
  if (op->et_state[ip] == op->state && op->et_tiling[ip][0] == tl.TX &&
      op->et_tiling[ip][1] == tl.TY && op->et_tiling[ip][2] == tl.ZC)
    return PTMF_OK;
  const long len = tl.ntiles * tl.ZC * 27L * kEPW;
  if (len > op->et_len) {
    PTMF_HIP(hipStreamSynchronize(op->stream));
    (void)hipFree(op->et64);
    (void)hipFree(op->et32);
    op->et64 = nullptr;
    op->et32 = nullptr;
    op->et_state[0] = op->et_state[1] = ~0UL;
    op->et_len = len;
  }
  T **dst = (T **)(sizeof(T) == 8 ? (void *)&op->et64 : (void *)&op->et32);
  if (!*dst) PTMF_HIP(hipMalloc((void **)dst, sizeof(T) * op->et_len));
  const TileArgs a = tile_args(op);
  const long nb = std::min<long>((len / 27 + 255) / 256, 65536);
  eta_tile_kernel<T><<<dim3((unsigned)nb), dim3(256), 0, op->stream>>>(a, op->d64.eta, *dst);
  PTMF_HIP(hipGetLastError());
  op->et_state[ip] = op->state;
  op->et_tiling[ip][0] = tl.TX;
  op->et_tiling[ip][1] = tl.TY;
  op->et_tiling[ip][2] = tl.ZC;
  return PTMF_OK;
}

// (Re)build the stored geometry of variant 2 for precision T when the
// coefficients or the tiling changed since the last build.
template <typename T>
int ensure_pa(ptmf_op_s *op) {
  const int ip = sizeof(T) == 8 ? 0 : 1;
  const Tiling &tl = op->tiling;
  if (op->pa_state[ip] == op->state && op->pa_tiling[ip][0] == tl.TX &&
      op->pa_tiling[ip][1] == tl.TY && op->pa_tiling[ip][2] == tl.ZC)
    return PTMF_OK;
  const long len = tl.ntiles * tl.ZC * 27L * 9L * kEPW;
  if (len > op->pa_len) {
    PTMF_HIP(hipStreamSynchronize(op->stream));
    (void)hipFree(op->pa64);
    (void)hipFree(op->pa32);
    op->pa64 = nullptr;
    op->pa32 = nullptr;
    op->pa_state[0] = op->pa_state[1] = ~0UL;
    op->pa_len = len;
  }
  T **dst = (T **)(sizeof(T) == 8 ? (void *)&op->pa64 : (void *)&op->pa32);
  if (!*dst) PTMF_HIP(hipMalloc((void **)dst, sizeof(T) * op->pa_len));
  if (!op->pa_bad) PTMF_HIP(hipMalloc((void **)&op->pa_bad, sizeof(int)));
  PTMF_TRY(launch_fill<int>(op->pa_bad, 0, 1, op->stream));
  const TileArgs a = tile_args(op);
  const long total = tl.ntiles * tl.ZC * 27L * kEPW;
  long nb = (total + 255) / 256;
  if (nb > 65536) nb = 65536;
  pa_build_kernel<T><<<dim3((unsigned)nb), dim3(256), 0, op->stream>>>(a, tl.ntiles, op->d64.coords,
                                                                      op->d64.eta, *dst, op->pa_bad);
  PTMF_HIP(hipGetLastError());
  int bad = 0;
  PTMF_HIP(hipMemcpyAsync(&bad, op->pa_bad, sizeof(int), hipMemcpyDeviceToHost, op->stream));
  PTMF_HIP(hipStreamSynchronize(op->stream));
  PTMF_CHECK(!bad, PTMF_ERR_ARG,
             "a11 (stored geometry): non-positive or non-finite 2 w eta / det at some quadrature "
             "point (inverted element or eta <= 0)");
  op->pa_state[ip] = op->state;
  op->pa_tiling[ip][0] = tl.TX;
  op->pa_tiling[ip][1] = tl.TY;
  op->pa_tiling[ip][2] = tl.ZC;
  return PTMF_OK;
}

// The tile-ordered viscosity for precision T rebuilt, when stale, into the
// buffer the operator already holds (kernel only, no allocation); an error
// when that buffer does not exist or is too short for the current tiling.
template <typename T>
int eta_tiled_in_place(ptmf_op_s *op) {
  const int ip = sizeof(T) == 8 ? 0 : 1;
  const Tiling &tl = op->tiling;
  if (op->et_state[ip] == op->state && op->et_tiling[ip][0] == tl.TX && op->et_tiling[ip][1] == tl.TY &&
      op->et_tiling[ip][2] == tl.ZC)
    return PTMF_OK;
  const long len = tl.ntiles * tl.ZC * 27L * kEPW;
  T *dst = (T *)(sizeof(T) == 8 ? (void *)op->et64 : (void *)op->et32);
  PTMF_CHECK(dst && len <= op->et_len, PTMF_ERR_NOT_SETUP,
             "a11_mult_noalloc: the tile-ordered viscosity of the current tiling is not allocated "
             "(ptmf_op_set_viscosity and ptmf_op_set_tiling build it; a hierarchy's level operator "
             "gets it from its first ptmf_a11_mult)");
  const TileArgs a = tile_args(op);
  const long nb = std::min<long>((len / 27 + 255) / 256, 65536);
  eta_tile_kernel<T><<<dim3((unsigned)nb), dim3(256), 0, op->stream>>>(a, op->d64.eta, dst);
  PTMF_HIP(hipGetLastError());
  op->et_state[ip] = op->state;
  op->et_tiling[ip][0] = tl.TX;
  op->et_tiling[ip][1] = tl.TY;
  op->et_tiling[ip][2] = tl.ZC;
  return PTMF_OK;
}

// the face sums and the Dirichlet rows
template <typename T>
int launch_face_copy(const ptmf_op_s *op, const TileArgs &a, const T *fbx, const T *fby, const T *fbz, const T *x,
                     T *y) {
  // (whole rounds of the XCDs, so that each keeps its own tiles; a row copied twice is the same)
  const long copies = 8 * ((op->nbc + 8 * kCopyGroup - 1) / (8 * kCopyGroup)), groups = a.ntiles + copies;
  PTMF_CHECK(groups < (1L << 31), PTMF_ERR_ARG, "a11: mesh too large (%ld work-groups)", groups);
  if (groups == 0) return PTMF_OK;  // (no faces, no Dirichlet dofs: the coloured variant on a free box)
  a11_face_copy_kernel<T><<<dim3((unsigned)groups), dim3(kFaceThreads), 0, op->stream>>>(
      a, fbx, fby, fbz, y, op->bcnode, op->bcidx, op->nbc, x);
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

template <typename T, typename F>
void with_kind(const RowUpdate<T> &up, F &&f) {
  if (!up.dinv) f(std::integral_constant<UpdateKind, kUpResidual>());
  else if (!up.prev) f(std::integral_constant<UpdateKind, kUpFirst>());
  else f(std::integral_constant<UpdateKind, kUpStep>());
}

// what follows the element kernel: nothing (its timing alone), the MatMult's face
// sums and Dirichlet rows, or a RowUpdate
enum Finish { kFinNone, kFinMult, kFinUpdate };

template <typename T>
int finish_rows(const ptmf_op_s *op, const TileArgs &a, Finish fin, const RowUpdate<T> *up, const T *fbx, const T *fby,
                const T *fbz, const T *x, T *y) {
  if (fin == kFinNone) return PTMF_OK;
  if (fin == kFinMult) return launch_face_copy<T>(op, a, fbx, fby, fbz, x, y);
  PTMF_CHECK(3 * a.XY < (1L << 32) - 256, PTMF_ERR_ARG, "a11: mesh too large (%ld nodes in a plane)", a.XY);
  const long gx = (3 * a.XY + 255) / 256;
  PTMF_CHECK(gx * a.mz < (1L << 31), PTMF_ERR_ARG, "a11: mesh too large (%ld work-groups)", gx * a.mz);
  with_kind(*up, [&](auto k) {
    a11_update_kernel<T, decltype(k)::value><<<dim3((unsigned)(gx * a.mz)), dim3(256), 0, op->stream>>>(
        a, (unsigned)gx, fbx, fby, fbz, y, op->bcnode, x, *up);
  });
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

// the lane kernel (lane_tiles must hold) and what follows
template <typename T, bool kP>
int launch_lane(const ptmf_op_s *op, const TileArgs &a, Finish fin, const RowUpdate<T> *up, const T *x, const T *p, T *y,
                T *yp, T *fb) {
  const T *ax = sizeof(T) == 8 ? (const T *)op->ax64 : (const T *)op->ax32;
  const T *eta = sizeof(T) == 8 ? (const T *)op->d64.eta : (const T *)op->d32.eta;
  T *fbx = fb, *fby = fbx + 3 * a.fbx_n * a.ntiles, *fbz = fby + 3 * a.fby_n * a.ntiles;
  a11_lane_kernel<T, kP><<<dim3((unsigned)a.ntiles), dim3(64), 0, op->stream>>>(a, ax, eta, op->bcword, x, p, y, yp, fbx,
                                                                               fby, fbz);
  PTMF_HIP(hipGetLastError());
  return finish_rows<T>(op, a, fin, up, fbx, fby, fbz, x, y);
}

template <typename T>
int launch_col(const ptmf_op_s *op, Finish fin, const RowUpdate<T> *up, const T *x, T *y, T *es) {
  const Box &b = op->box;
  const OpData<T> &d = *(const OpData<T> *)(sizeof(T) == 8 ? (const void *)&op->d64 : (const void *)&op->d32);
  const ColArgs a = col_args(b);
  a11_col_kernel<T><<<dim3(a.nwaves), dim3(64), 0, op->stream>>>(a, d.coords, d.eta, op->bcnode, x, es);
  PTMF_HIP(hipGetLastError());
  if (fin == kFinNone) return PTMF_OK;
  const long groups = (b.nnodes + kColSumThreads - 1) / kColSumThreads;
  if (fin == kFinMult)
    col_sum_kernel<T><<<dim3((unsigned)groups), dim3(kColSumThreads), 0, op->stream>>>(a, es, y, op->bcnode, x);
  else
    with_kind(*up, [&](auto k) {
      col_update_kernel<T, decltype(k)::value>
          <<<dim3((unsigned)groups), dim3(kColSumThreads), 0, op->stream>>>(a, es, op->bcnode, x, *up);
    });
  PTMF_HIP(hipGetLastError());
  return PTMF_OK;
}

// The element kernel of a MatMult with face buffers of fb_doubles; la: the
// decomposition of the lane kernel.  noalloc: as in launch_a11_mult_fb.
enum MultKernel { kMultTile, kMultPipelined, kMultStored, kMultColoured, kMultLane, kMultColumn };  // (variants first)

template <typename T>
MultKernel mult_kernel(const ptmf_op_s *op, long fb_doubles, bool noalloc, TileArgs &la) {
  if (op->variant != 0 && !(noalloc && op->variant >= 2)) return (MultKernel)op->variant;
  const bool col = col_box(op, fb_doubles);
  if (lane_tiles<T>(op, fb_doubles, col ? kOtherCol : kOtherTile, la)) return kMultLane;
  return col ? kMultColumn : kMultTile;
}

// The MatMult's kernels with the operator's own face buffers or those at
// `scratch`, of the allocation-free entry point.  With these nothing is
// allocated on the way (the stored-geometry and coloured variants, which build
// tables of their own or need no face buffers, give way to the z-march).
template <typename T>
int launch_a11_mult_fb(ptmf_op_s *op, Finish fin, const RowUpdate<T> *up, const T *x, T *y, double *scratch = nullptr,
                       long scratch_doubles = 0) {
  const OpData<T> &d = *(const OpData<T> *)(sizeof(T) == 8 ? (const void *)&op->d64
                                                           : (const void *)&op->d32);
  const Tiling &tl = op->tiling;
  PTMF_CHECK(tl.TX * tl.TY <= kEPW && (2 * tl.TX + 1) * (2 * tl.TY + 1) <= kWinNodes && tl.ZC > 0,
             PTMF_ERR_ARG, "a11: invalid tiling %d x %d x %d", tl.TX, tl.TY, tl.ZC);
  std::lock_guard<std::mutex> lock(op->faces_mu);
  const bool noalloc = scratch != nullptr;
  T *const fb = (T *)(noalloc ? scratch : op->faces);
  const long fb_doubles = noalloc ? scratch_doubles : op->faces_doubles;
  PTMF_CHECK(fb != nullptr, PTMF_ERR_NOT_SETUP, "a11: face buffers not allocated");
  TileArgs la;
  const MultKernel kernel = mult_kernel<T>(op, fb_doubles, noalloc, la);
  if (kernel == kMultColoured) {
    // coloured scatter: no tiles, no face buffers
    const Box &b = op->box;
    PTMF_TRY(launch_fill<T>(y, T(0), 3 * b.nnodes, op->stream));
    for (int color = 0; color < 8; color++) {
      const long nb = (class_count(b, color) + kEPW - 1) / kEPW;
      if (nb == 0) continue;
      a11_colour_kernel<T><<<dim3((unsigned)nb), dim3(64), 0, op->stream>>>(
          b.mx, b.my, b.mz, b.nel, b.X, b.X * b.Y, color, d.coords, d.eta, op->bcnode, x, y);
    }
    PTMF_HIP(hipGetLastError());
    TileArgs one = tile_args(op);  // (a single tile: no faces)
    one.TX = b.mx; one.TY = b.my; one.ZC = b.mz;
    one.ntx = one.nty = 1;
    one.ntiles = 0;
    return finish_rows<T>(op, one, fin, up, nullptr, nullptr, nullptr, x, y);
  }
  if (kernel == kMultLane) return launch_lane<T, false>(op, la, fin, up, x, nullptr, y, nullptr, fb);
  if (kernel == kMultColumn) return launch_col<T>(op, fin, up, x, y, fb);
  const TileArgs a = tile_args(op);
  const long ntiles = tl.ntiles;
  T *fbx = fb, *fby = fbx + 3 * a.fbx_n * ntiles, *fbz = fby + 3 * a.fby_n * ntiles;
  if (kernel == kMultStored) {
    PTMF_TRY(ensure_pa<T>(op));
    const T *pa = sizeof(T) == 8 ? (const T *)op->pa64 : (const T *)op->pa32;
    a11_tile_pa_kernel<T, true><<<dim3((unsigned)ntiles), dim3(64), 0, op->stream>>>(
        a, pa, op->bcnode, x, y, fbx, fby, fbz);
  } else {
    PTMF_TRY(noalloc ? eta_tiled_in_place<T>(op) : ensure_eta_tiled<T>(op));
    const T *et = sizeof(T) == 8 ? (const T *)op->et64 : (const T *)op->et32;
    const int kw = op->wg_tiles;
    const long nwg = (ntiles + kw - 1) / kw;
    if (kernel == kMultPipelined)
      a11_tile_pf_kernel<T, true><<<dim3((unsigned)ntiles), dim3(64), 0, op->stream>>>(
          a, d.coords, et, op->bcnode, x, y, fbx, fby, fbz);
    else if (kw == 2)
      a11_tile_wg_kernel<T, true, 2><<<dim3((unsigned)nwg), dim3(128), 0, op->stream>>>(
          a, nwg, d.coords, et, op->bcnode, x, y, fbx, fby, fbz);
    else if (kw == 4)
      a11_tile_wg_kernel<T, true, 4><<<dim3((unsigned)nwg), dim3(256), 0, op->stream>>>(
          a, nwg, d.coords, et, op->bcnode, x, y, fbx, fby, fbz);
    else
      a11_tile_kernel<T, true><<<dim3((unsigned)ntiles), dim3(64), 0, op->stream>>>(
          a, d.coords, et, op->bcnode, x, y, fbx, fby, fbz);
  }
  PTMF_HIP(hipGetLastError());
  return finish_rows<T>(op, a, fin, up, fbx, fby, fbz, x, y);
}

template <typename T>
int launch_a11_mult(ptmf_op_s *op, const T *x, T *y, bool whole) {
  return launch_a11_mult_fb<T>(op, whole ? kFinMult : kFinNone, nullptr, x, y);
}

template <typename T>
int launch_a11_update(ptmf_op_s *op, const T *x, T *r, const RowUpdate<T> &up) {
  return launch_a11_mult_fb<T>(op, kFinUpdate, &up, x, r);
}

template <typename T>
int launch_stokes_mult_t(ptmf_op_s *op, const T *x, T *y) {
  const OpData<T> &d = *(const OpData<T> *)(sizeof(T) == 8 ? (const void *)&op->d64
                                                           : (const void *)&op->d32);
  const Tiling &tl = op->tiling;
  PTMF_CHECK(tl.TX * tl.TY <= kEPW && (2 * tl.TX + 1) * (2 * tl.TY + 1) <= kWinNodes && tl.ZC > 0,
             PTMF_ERR_ARG, "stokes: invalid tiling %d x %d x %d", tl.TX, tl.TY, tl.ZC);
  std::lock_guard<std::mutex> lock(op->faces_mu);
  PTMF_CHECK(op->faces != nullptr, PTMF_ERR_NOT_SETUP, "stokes: face buffers not allocated");
  const long nu = 3 * op->box.nnodes;
  // (by lane_plan's rule: at 24^3, with the tile kernel, 37 us; at 28^3 the lane
  // kernel takes 33 us and the tile kernel 56 us, and further apart above)
  TileArgs la;
  if (lane_tiles<T>(op, op->faces_doubles, kOtherTile, la))
    return launch_lane<T, true>(op, la, kFinMult, nullptr, x, x + nu, y, y + nu, (T *)op->faces);
  PTMF_TRY(ensure_eta_tiled<T>(op));
  const T *et = sizeof(T) == 8 ? (const T *)op->et64 : (const T *)op->et32;
  const TileArgs a = tile_args(op);
  const long ntiles = tl.ntiles;
  T *fbx = (T *)op->faces, *fby = fbx + 3 * a.fbx_n * ntiles, *fbz = fby + 3 * a.fby_n * ntiles;
  stokes_tile_kernel<T><<<dim3((unsigned)ntiles), dim3(64), 0, op->stream>>>(
      a, d.coords, et, op->bcnode, x, x + nu, y, y + nu, fbx, fby, fbz);
  PTMF_HIP(hipGetLastError());
  return launch_face_copy<T>(op, a, fbx, fby, fbz, x, y);
}

int launch_stokes_mult(ptmf_op_s *op, const double *x, double *y) { return launch_stokes_mult_t<double>(op, x, y); }

// FP32 saddle-point MatMult (FP32 coordinates, viscosity and accumulation):
// the preconditioner's A12 product of an FP32 velocity V-cycle.
int launch_stokes_mult_f32(ptmf_op_s *op, const float *x, float *y) { return launch_stokes_mult_t<float>(op, x, y); }

int a11_mult_kernel(const ptmf_op_s *op, int precision) {
  TileArgs la;
  return precision == 64 ? mult_kernel<double>(op, op->faces_doubles, false, la)
                         : mult_kernel<float>(op, op->faces_doubles, false, la);
}

int prepare_eta_tiled(ptmf_op_s *op) { return ensure_eta_tiled<double>(op); }

template int launch_a11<double>(const ptmf_op_s *, const double *, double *, bool);
template int launch_a11<float>(const ptmf_op_s *, const float *, float *, bool);
template int launch_a11_mult<double>(ptmf_op_s *, const double *, double *, bool);
template int launch_a11_mult<float>(ptmf_op_s *, const float *, float *, bool);
template int launch_a11_update<double>(ptmf_op_s *, const double *, double *, const RowUpdate<double> &);
template int launch_a11_update<float>(ptmf_op_s *, const float *, float *, const RowUpdate<float> &);

}  // namespace ptmf

// ---------------------------------------------------------------------------
// Batched MatMult object (C-ABI)
// ---------------------------------------------------------------------------
struct ptmf_batch_s {
  std::vector<ptmf_op> ops;
  std::vector<ptmf_op> distinct;  // the same, for FacesLock
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  // device data, rebuilt when the operators' tilings or buffers change
  ptmf::BoxDesc *dbox[2] = {nullptr, nullptr};
  std::vector<unsigned char> hbox[2];
  // (box, tile) of the tile kernel, then (box, wave) and (box, node block) of
  // the column kernel
  int2 *dwork = nullptr;
  long nwork = 0, ncol = 0, nsum = 0;
  std::vector<int> key;  // TX, TY, ZC, ntiles, column kernel per operator of the current work list
  void **dxy[2] = {nullptr, nullptr};  // device arrays of x and y pointers, per precision
  std::vector<const void *> hxy[2];
  long maxnbc = 0;
};

namespace {

// work list and per-box descriptors of precision T (no vectors)
template <typename T>
int batch_prepare_boxes(ptmf_batch_s *b) {
  const int ip = sizeof(T) == 8 ? 0 : 1;
  const int n = (int)b->ops.size();
  // work lists
  auto col = [](const ptmf_op_s *op) { return op->variant == 0 && ptmf::col_box(op, op->faces_doubles); };
  std::vector<int> key;
  for (ptmf_op op : b->ops) {
    const ptmf::Tiling &t = op->tiling;
    key.insert(key.end(), {t.TX, t.TY, t.ZC, (int)t.ntiles, col(op) ? 1 : 0});
  }
  if (key != b->key) {
    std::vector<int2> work;
    auto add = [&](bool column, auto &&count) {
      const size_t first = work.size();
      for (int i = 0; i < n; i++)
        if (col(b->ops[i]) == column)
          for (long t = 0, m = count(b->ops[i]); t < m; t++) work.push_back(make_int2(i, (int)t));
      return (long)(work.size() - first);
    };
    b->nwork = add(false, [](ptmf_op op) { return op->tiling.ntiles; });
    b->ncol = add(true, [](ptmf_op op) { return (op->box.nel + ptmf::kColElems - 1) / ptmf::kColElems; });
    b->nsum = add(true, [](ptmf_op op) { return (op->box.nnodes + ptmf::kColSumThreads - 1) / ptmf::kColSumThreads; });
    PTMF_CHECK(!work.empty() && work.size() < (1UL << 31), PTMF_ERR_ARG, "batch: %zu work items", work.size());
    (void)hipFree(b->dwork);
    b->dwork = nullptr;
    PTMF_HIP(hipMalloc((void **)&b->dwork, sizeof(int2) * work.size()));
    PTMF_HIP(hipMemcpy(b->dwork, work.data(), sizeof(int2) * work.size(), hipMemcpyHostToDevice));
    b->key = key;
  }
  // per-box descriptors of this precision
  std::vector<ptmf::BoxDesc> box(n);
  b->maxnbc = 0;
  for (int i = 0; i < n; i++) {
    ptmf_op op = b->ops[i];
    PTMF_CHECK(op->has_coords && op->has_eta && op->has_bc, PTMF_ERR_NOT_SETUP,
               "batch: operator %d: MF operator not setup", i);
    ptmf::BoxDesc &d = box[i];
    memset((void *)&d, 0, sizeof(d));  // (compared bytewise)
    if (!col(op)) {
      PTMF_TRY(ptmf::ensure_eta_tiled<T>(op));
      PTMF_HIP(hipStreamSynchronize(op->stream));  // (built on the operator's own stream)
    }
    d.a = ptmf::tile_args(op);
    const ptmf::OpData<T> &od = *(const ptmf::OpData<T> *)(ip == 0 ? (const void *)&op->d64 : (const void *)&op->d32);
    d.xc = od.coords;
    d.eta = ip == 0 ? (const void *)op->et64 : (const void *)op->et32;
    d.bcn = op->bcnode;
    d.bcidx = op->bcidx;
    d.nbc = op->nbc;
    T *fb = (T *)op->faces;
    d.fbx = fb;
    d.fby = fb + 3 * d.a.fbx_n * d.a.ntiles;
    d.fbz = (T *)d.fby + 3 * d.a.fby_n * d.a.ntiles;
    if (col(op)) {
      d.c = ptmf::col_args(op->box);
      d.eta = od.eta;
      d.nbc = 0;
    }
    if (d.nbc > b->maxnbc) b->maxnbc = d.nbc;
  }
  const size_t bytes = sizeof(ptmf::BoxDesc) * n;
  if (!b->dbox[ip]) PTMF_HIP(hipMalloc((void **)&b->dbox[ip], bytes));
  const unsigned char *raw = (const unsigned char *)box.data();
  if (b->hbox[ip].size() != bytes || memcmp(b->hbox[ip].data(), raw, bytes) != 0) {
    b->hbox[ip].assign(raw, raw + bytes);
    PTMF_HIP(hipMemcpyAsync(b->dbox[ip], b->hbox[ip].data(), bytes, hipMemcpyHostToDevice, b->stream));
  }
  return PTMF_OK;
}

template <typename T>
int batch_prepare(ptmf_batch_s *b, const void *const *x, void *const *y) {
  const int ip = sizeof(T) == 8 ? 0 : 1;
  const int n = (int)b->ops.size();
  PTMF_TRY(batch_prepare_boxes<T>(b));
  // x and y pointer arrays
  std::vector<const void *> xy(2 * n);
  for (int i = 0; i < n; i++) {
    PTMF_CHECK(x[i] && y[i] && x[i] != y[i], PTMF_ERR_ARG, "batch: vectors of box %d", i);
    xy[i] = x[i];
    xy[n + i] = y[i];
  }
  if (!b->dxy[ip]) PTMF_HIP(hipMalloc((void **)&b->dxy[ip], sizeof(void *) * 2 * n));
  if (b->hxy[ip] != xy) {
    b->hxy[ip] = xy;
    PTMF_HIP(hipMemcpyAsync(b->dxy[ip], b->hxy[ip].data(), sizeof(void *) * 2 * n, hipMemcpyHostToDevice,
                            b->stream));
  }
  return PTMF_OK;
}

// the batched stages on device tables of x and y pointers
template <typename T>
int batch_launch_tables(ptmf_batch_s *b, const T *const *xs, T *const *ys, hipStream_t s,
                        const int *active = nullptr) {
  const int ip = sizeof(T) == 8 ? 0 : 1;
  const int n = (int)b->ops.size();
  if (b->ncol > 0) {
    const int2 *work = b->dwork + b->nwork;
    ptmf::a11_col_batch_kernel<T><<<dim3((unsigned)b->ncol), dim3(64), 0, s>>>(b->dbox[ip], work, b->ncol, xs, active);
    PTMF_HIP(hipGetLastError());
    ptmf::col_sum_batch_kernel<T><<<dim3((unsigned)b->nsum), dim3(ptmf::kColSumThreads), 0, s>>>(
        b->dbox[ip], work + b->ncol, b->nsum, xs, ys, active);
    PTMF_HIP(hipGetLastError());
  }
  if (b->nwork == 0) return PTMF_OK;
  ptmf::a11_tile_batch_kernel<T><<<dim3((unsigned)b->nwork), dim3(64), 0, s>>>(b->dbox[ip], b->dwork, b->nwork, xs,
                                                                              ys, active);
  PTMF_HIP(hipGetLastError());
  ptmf::a11_face_batch_kernel<T><<<dim3((unsigned)b->nwork), dim3(64), 0, s>>>(b->dbox[ip], b->dwork, b->nwork, ys,
                                                                              active);
  PTMF_HIP(hipGetLastError());
  if (b->maxnbc > 0) {
    long gx = (b->maxnbc + 255) / 256;
    if (gx > 1024) gx = 1024;
    ptmf::bc_copy_batch_kernel<T><<<dim3((unsigned)gx, (unsigned)n), dim3(256), 0, s>>>(b->dbox[ip], xs, ys,
                                                                                        active);
    PTMF_HIP(hipGetLastError());
  }
  return PTMF_OK;
}

template <typename T>
int batch_launch(ptmf_batch_s *b) {
  const int ip = sizeof(T) == 8 ? 0 : 1;
  const int n = (int)b->ops.size();
  return batch_launch_tables<T>(b, (const T *const *)b->dxy[ip], (T *const *)(b->dxy[ip] + n), b->stream);
}

}  // namespace

namespace ptmf {
int batch_bind(ptmf_batch_s *b, int precision) {
  for (ptmf_op op : b->ops) PTMF_HIP(hipStreamSynchronize(op->stream));
  if (precision == 64) PTMF_TRY(batch_prepare_boxes<double>(b));
  else PTMF_TRY(batch_prepare_boxes<float>(b));
  PTMF_HIP(hipStreamSynchronize(b->stream));
  return PTMF_OK;
}

int batch_apply(ptmf_batch_s *b, int precision, const void *const *xs, void *const *ys, hipStream_t s,
                const int *active) {
  if (precision == 64)
    return batch_launch_tables<double>(b, (const double *const *)xs, (double *const *)ys, s, active);
  return batch_launch_tables<float>(b, (const float *const *)xs, (float *const *)ys, s, active);
}
}  // namespace ptmf

extern "C" {

int ptmf_batch_create(const ptmf_op *ops, int nops, ptmf_batch *out) {
  PTMF_CHECK(ops && out && nops > 0 && nops <= 65535, PTMF_ERR_ARG, "batch_create: bad arguments");
  for (int i = 0; i < nops; i++) PTMF_CHECK(ops[i], PTMF_ERR_ARG, "batch_create: null operator %d", i);
  ptmf_batch_s *b = new ptmf_batch_s;
  b->ops.assign(ops, ops + nops);
  b->distinct = b->ops;
  std::sort(b->distinct.begin(), b->distinct.end());
  b->distinct.erase(std::unique(b->distinct.begin(), b->distinct.end()), b->distinct.end());
  hipError_t e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreate(&b->ev0);
  if (e == hipSuccess) e = hipEventCreate(&b->ev1);
  if (e != hipSuccess) {
    ptmf_batch tmp = b;
    ptmf_batch_destroy(&tmp);
    return ptmf_set_error(PTMF_ERR_DEVICE, "batch_create: %s", hipGetErrorString(e));
  }
  *out = b;
  return PTMF_OK;
}

int ptmf_batch_destroy(ptmf_batch *pb) {
  if (!pb || !*pb) return PTMF_OK;
  ptmf_batch_s *b = *pb;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  for (int i = 0; i < 2; i++) {
    (void)hipFree(b->dbox[i]);
    (void)hipFree(b->dxy[i]);
  }
  (void)hipFree(b->dwork);
  if (b->ev0) (void)hipEventDestroy(b->ev0);
  if (b->ev1) (void)hipEventDestroy(b->ev1);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
  *pb = nullptr;
  return PTMF_OK;
}

namespace {
// the batched MatMult, with the FacesLock held
int batch_mult_locked(ptmf_batch b, int precision, const void *const *x, void *const *y) {
  for (ptmf_op op : b->ops) PTMF_HIP(hipStreamSynchronize(op->stream));
  if (precision == 64) {
    PTMF_TRY(batch_prepare<double>(b, x, y));
    PTMF_TRY(batch_launch<double>(b));
  } else {
    PTMF_TRY(batch_prepare<float>(b, x, y));
    PTMF_TRY(batch_launch<float>(b));
  }
  PTMF_HIP(hipStreamSynchronize(b->stream));
  return PTMF_OK;
}
}  // namespace

int ptmf_batch_mult(ptmf_batch b, int precision, const void *const *x, void *const *y) {
  PTMF_CHECK(b && x && y, PTMF_ERR_ARG, "batch_mult: null argument");
  PTMF_CHECK(precision == 64 || precision == 32, PTMF_ERR_UNSUPPORTED, "batch_mult: precision %d", precision);
  ptmf::FacesLock lock(b->distinct);
  return batch_mult_locked(b, precision, x, y);
}

int ptmf_batch_time(ptmf_batch b, int precision, const void *const *x, void *const *y, int reps, double *ms) {
  PTMF_CHECK(b && x && y && reps > 0 && ms, PTMF_ERR_ARG, "batch_time: bad arguments");
  PTMF_CHECK(precision == 64 || precision == 32, PTMF_ERR_UNSUPPORTED, "batch_mult: precision %d", precision);
  ptmf::FacesLock lock(b->distinct);
  PTMF_TRY(batch_mult_locked(b, precision, x, y));  // prepares and warms up
  PTMF_HIP(hipEventRecord(b->ev0, b->stream));
  for (int r = 0; r < reps; r++) {
    if (precision == 64) PTMF_TRY(batch_launch<double>(b));
    else PTMF_TRY(batch_launch<float>(b));
  }
  PTMF_HIP(hipEventRecord(b->ev1, b->stream));
  PTMF_HIP(hipEventSynchronize(b->ev1));
  float t = 0.0f;
  PTMF_HIP(hipEventElapsedTime(&t, b->ev0, b->ev1));
  *ms = (double)t / reps;
  return PTMF_OK;
}

}  // extern "C"


// ---------------------------------------------------------------------------
// Allocation-free MatMult (ptmf_a11_mult_noalloc): the FP64 MatMult of
// ptmf_a11_mult with the z-march's face buffers in `scratch`, a file-scope
// device array of kScratchDoubles doubles (64 MiB) that every GPU the library
// runs on holds until the process ends, instead of the operator's own
// allocation.  In host code `scratch` names a host-side stand-in, not device
// memory: the device address comes from hipGetSymbolAddress, once per
// device, with that device current, and only that address reaches kernels.
// Every call on one GPU shares its array (the tile kernel writes every face
// entry the face kernel reads, so nothing needs clearing): calls that overlap
// on one GPU race.
// ---------------------------------------------------------------------------
#include <mutex>

namespace {
constexpr long kScratchDoubles = 8L << 20;
constexpr int kScratchDevices = 64;
}  // namespace

static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {
std::mutex scratch_mu;
double *scratch_at[kScratchDevices];

// device address of `scratch` on device dev (the current device)
int scratch_address(int dev, double **out) {
  PTMF_CHECK(dev >= 0 && dev < kScratchDevices, PTMF_ERR_DEVICE, "a11_mult_noalloc: device %d", dev);
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_at[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    PTMF_CHECK(e == hipSuccess && p, PTMF_ERR_DEVICE, "a11_mult_noalloc: hipGetSymbolAddress(scratch): %s",
               hipGetErrorString(e));
    scratch_at[dev] = (double *)p;
  }
  *out = scratch_at[dev];
  return PTMF_OK;
}
}  // namespace

extern "C" int ptmf_a11_mult_noalloc(ptmf_op op, const double *x, double *y) {
  PTMF_CHECK(op, PTMF_ERR_ARG, "a11_mult_noalloc: null operator");
  PTMF_CHECK(op->has_coords && op->has_eta && op->has_bc, PTMF_ERR_NOT_SETUP, "MF operator not setup");
  PTMF_CHECK(x && y && (const void *)x != (const void *)y, PTMF_ERR_ARG,
             "a11_mult_noalloc: x and y must be distinct device arrays");
  int dev = -1;
  PTMF_HIP(hipGetDevice(&dev));
  PTMF_CHECK(dev == op->device, PTMF_ERR_ARG,
             "a11_mult_noalloc: the operator lives on device %d but device %d is current", op->device, dev);
  const ptmf::Tiling &tl = op->tiling;
  const long need = ptmf::face_buffer_doubles(tl.TX, tl.TY, tl.ZC, tl.ntiles);
  PTMF_CHECK(need <= kScratchDoubles, PTMF_ERR_UNSUPPORTED,
             "a11_mult_noalloc: the face buffers of this box and tiling take %ld doubles, the static scratch "
             "holds %ld (64 MiB); use ptmf_a11_mult",
             need, kScratchDoubles);
  double *fb = nullptr;
  PTMF_TRY(scratch_address(dev, &fb));
  return ptmf::launch_a11_mult_fb<double>(op, ptmf::kFinMult, nullptr, x, y, fb, kScratchDoubles);
}
