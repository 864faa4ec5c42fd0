// tile.h -- device code shared by the tiled element kernels: the 1-D operators
// of the Q2 element, the tile decomposition of a box with its XCD-aware order,
// and the sums over tile faces.
#pragma once

#include "ptmf_internal.h"

namespace ptmf {
namespace {

template <typename T>
__device__ __forceinline__ T sel3(int c, double a0, double a1, double a2) {
  return (T)(c == 0 ? a0 : (c == 1 ? a1 : a2));
}

// 1-D operators written with the exact structure of the Gauss tables (the
// compiler may not drop multiplications by exact zeros or ones under IEEE
// rules): B = [[a, m, b], [0, 1, 0], [b, m, a]] with a, b = e +- o, e = 0.3,
// o = sqrt(3/5)/2, m = 0.4.  interp3: y = B x, in 5 operations; interp3t: y =
// B^T x, in even/odd form in 6.
constexpr double kBe = 0.5 * (kB[0][0] + kB[0][2]);
constexpr double kBo = 0.5 * (kB[0][0] - kB[0][2]);

template <typename T>
__device__ __forceinline__ void interp3(T x0, T x1, T x2, T &y0, T &y1, T &y2) {
  const T p = (T)kB[0][1] * x1, u = p + (T)kB[0][2] * x2, v = p + (T)kB[2][2] * x2;
  y0 = u + (T)kB[0][0] * x0;
  y1 = x1;
  y2 = v + (T)kB[2][0] * x0;
}

template <typename T>
__device__ __forceinline__ void interp3t(T x0, T x1, T x2, T &y0, T &y1, T &y2) {
  const T sm = x0 + x2, df = x0 - x2;
  const T t = (T)kBe * sm;
  y0 = t + (T)kBo * df;
  y1 = x1 + (T)kB[0][1] * sm;
  y2 = t - (T)kBo * df;
}

// collocated derivative at quadrature point a of a 3-point line,
// sum_r C[a][r] x_r, with the zero of the middle row skipped
template <typename T>
__device__ __forceinline__ T cdot(int a, T x0, T x1, T x2) {
  if (a == 1) return (T)kC[1][2] * (x2 - x0);
  return (T)kC[a][0] * x0 + (T)kC[a][1] * x1 + (T)kC[a][2] * x2;
}

// 1/x by the hardware reciprocal estimate refined with Newton-Raphson steps
// r <- r + r (1 - x r) (two for double, one for float)
template <typename T>
__device__ __forceinline__ T recip(T x);
template <>
__device__ __forceinline__ double recip<double>(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = fma(-x, r, 1.0);
  r = fma(r, e, r);
  e = fma(-x, r, 1.0);
  return fma(r, e, r);
}
template <>
__device__ __forceinline__ float recip<float>(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  const float e = fmaf(-x, r, 1.0f);
  return fmaf(r, e, r);
}

// transposed in-plane interpolation: out[3j+i] = sum_{a,b} B[a][i] B[b][j] Y[3b+a]
template <typename T>
__device__ __forceinline__ void interp_plane_t(const T Y[9], T out[9]) {
  T t[3][3];  // [b][i]
#pragma unroll
  for (int b = 0; b < 3; b++) interp3t<T>(Y[3 * b], Y[3 * b + 1], Y[3 * b + 2], t[b][0], t[b][1], t[b][2]);
#pragma unroll
  for (int i = 0; i < 3; i++) interp3t<T>(t[0][i], t[1][i], t[2][i], out[i], out[3 + i], out[6 + i]);
}

// Work decomposition of a tiled kernel: TX x TY elements in x-y, ZC layers in
// z, and the sizes of a tile's face buffers (nodes)
struct TileArgs {
  int mx, my, mz;
  long X, XY, nel;
  int TX, TY, ZC, ntx, nty;
  long ntiles;
  long fbx_n, fby_n, fbz_n;  // per-tile face buffer sizes in nodes
};

// Work-groups are dispatched round-robin over the 8 XCDs (each with its own
// L2); give every XCD a contiguous run of tiles (x fastest), so tiles that
// share halo nodes and viscosity cache lines share an L2.
__device__ __forceinline__ long xcd_tile(long b, long ntiles) {
  const long per = ntiles / 8, rem = ntiles % 8;
  const long x = b % 8, slot = b / 8;
  return x * per + (x < rem ? x : rem) + slot;
}

struct TileBox {
  int tx, ty, tz, x0, y0, z0, nxt, nyt, nzt;
  bool xend, yend, zend;
};

__device__ __forceinline__ TileBox tile_box(const TileArgs &a, long tile) {
  TileBox t;
  t.tx = (int)(tile % a.ntx);
  t.ty = (int)((tile / a.ntx) % a.nty);
  t.tz = (int)(tile / ((long)a.ntx * a.nty));
  t.x0 = t.tx * a.TX;
  t.y0 = t.ty * a.TY;
  t.z0 = t.tz * a.ZC;
  t.nxt = min(a.TX, a.mx - t.x0);
  t.nyt = min(a.TY, a.my - t.y0);
  t.nzt = min(a.ZC, a.mz - t.z0);
  t.xend = t.x0 + t.nxt == a.mx;
  t.yend = t.y0 + t.nyt == a.my;
  t.zend = t.z0 + t.nzt == a.mz;
  return t;
}

// Adds the neighbours' face-buffer contributions into the nodes on the lower
// faces of each tile (the work-group's threads take one node each in turn;
// every node's sum has one thread and a fixed order).
// kSkip: the Dirichlet dofs (bcn) are left alone, their rows are already y = x.
template <typename T, bool kSkip = false>
__device__ __forceinline__ void face_sum(const TileArgs &a, long tile, const T *__restrict__ fbx,
                                         const T *__restrict__ fby, const T *__restrict__ fbz,
                                         T *__restrict__ y, const uint8_t *__restrict__ bcn = nullptr) {
  const TileBox tb = tile_box(a, tile);
  const int oX = 2 * tb.nxt + (tb.xend ? 1 : 0);
  const int oY = 2 * tb.nyt + (tb.yend ? 1 : 0);
  const int oZ = 2 * tb.nzt + (tb.zend ? 1 : 0);
  const bool hx = tb.tx > 0, hy = tb.ty > 0, hz = tb.tz > 0;
  const int nX = hx ? oY * oZ : 0;
  const int iy0 = hx ? 1 : 0, jz0 = hy ? 1 : 0, iz0 = hx ? 1 : 0;
  const int nY = hy ? (oX - iy0) * oZ : 0;
  const int nZ = hz ? (oX - iz0) * (oY - jz0) : 0;
  for (int t = threadIdx.x; t < nX + nY + nZ; t += blockDim.x) {
    int il, jl, kl;
    if (t < nX) {
      il = 0; jl = t % oY; kl = t / oY;
    } else if (t < nX + nY) {
      const int r = t - nX, w = oX - iy0;
      il = iy0 + r % w; jl = 0; kl = r / w;
    } else {
      const int r = t - nX - nY, w = oX - iz0;
      il = iz0 + r % w; jl = jz0 + r / w; kl = 0;
    }
    const int I = 2 * tb.x0 + il, J = 2 * tb.y0 + jl, K = 2 * tb.z0 + kl;
    const long n = (long)I + a.X * (long)J + a.XY * (long)K;
    // all that the row needs is requested before any of it is used
    const unsigned m = kSkip ? (unsigned)bcn[n] : 0u;
    T row[3], v[7][3];
#pragma unroll
    for (int l = 0; l < 3; l++) row[l] = y[3 * n + l];
#pragma unroll
    for (int s = 0; s < 7; s++) {  // the neighbours one tile on in x, y, z; lowest first
      const int dx = s & 1 ? 0 : -1, dy = s & 2 ? 0 : -1, dz = s & 4 ? 0 : -1;
      const bool has = (dx == 0 || (hx && il == 0)) && (dy == 0 || (hy && jl == 0)) && (dz == 0 || (hz && kl == 0));
#pragma unroll
      for (int l = 0; l < 3; l++) v[s][l] = T(0);
      if (!has) continue;
      const long tp = (tb.tx + dx) + (long)a.ntx * ((tb.ty + dy) + (long)a.nty * (tb.tz + dz));
      const int ilp = I - 2 * (tb.tx + dx) * a.TX, jlp = J - 2 * (tb.ty + dy) * a.TY,
                klp = K - 2 * (tb.tz + dz) * a.ZC;
      const T *src;
      if (dx == -1)
        src = fbx + 3 * (tp * a.fbx_n + jlp + (long)(2 * a.TY + 1) * klp);
      else if (dy == -1)
        src = fby + 3 * (tp * a.fby_n + ilp + (long)(2 * a.TX + 1) * klp);
      else
        src = fbz + 3 * (tp * a.fbz_n + ilp + (long)(2 * a.TX + 1) * jlp);
#pragma unroll
      for (int l = 0; l < 3; l++) v[s][l] = src[l];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int l = 0; l < 3; l++) {
      T acc = v[0][l];
#pragma unroll
      for (int s = 1; s < 7; s++) acc += v[s][l];
      if (!kSkip || !((m >> l) & 1u)) y[3 * n + l] = row[l] + acc;
    }
  }
}

}  // namespace
}  // namespace ptmf
