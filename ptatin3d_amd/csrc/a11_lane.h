// a11_lane.h -- the A11 MatMult of a rectilinear mesh, one lane per element
// (included by a11.hip, inside its anonymous namespace).
//
// A wave owns an 8 x 8 tile of elements in x-y, one element per lane, and
// marches through a chunk of element layers in z.  On a rectilinear mesh (all
// element faces normal to the axes) the Jacobian is diag(hx, hy, hz) / 2, so
// an element's state is its velocity alone and one lane can hold all of it:
// nothing is exchanged between lanes but the node values, which neighbouring
// elements share through LDS.  Per layer a lane reads its 27 nodes once per
// quadrature plane (243 LDS reads for 64 elements; the tile kernel of a11.hip
// needs about 590 for 21), and the arithmetic is half of the general
// element's: no Jacobian, adjugate or division per point.
//
// What bounds it: instruction issue of the one (FP64) or two (FP32) waves per
// SIMD that the registers allow.  FP64: 256 VGPRs + 150 AGPRs, about 4,900
// vector instructions per layer of which 3,340 are FP64 arithmetic, VALU busy
// 44 % of the wave's cycles.  64^3, MI355X: 79.6 us in FP64 (tile kernel 178
// us), 48 us in FP32 (82 us).  The loads are the delicate part: a value that
// is still in flight when the registers run short is waited for at once, to
// be moved to an accumulation register or to scratch, one round trip each (the
// same kernel with its loads in flight across the stress stage took 130 us,
// with 40 scratch moves 156 us).  So every load is issued before a forward
// stage and used up at its end, where few registers are live.
constexpr int kLT = 8;     // elements per tile side
constexpr int kLRow = 9;   // row stride of a node class
constexpr int kLRows = 17; // node rows and columns of a tile
constexpr int kLMaxZ = 31; // element layers of a chunk (63 node planes: one bit each of a 64-bit mask)
// The nodes of a tile plane are stored by the parity of their indices, so a
// lane's node (i, j) lies at a constant offset from the lane's own index and
// neighbouring lanes read neighbouring words: class (i & 1) + 2 (j & 1).
constexpr int kLCls[4] = {0, 81, 162, 234};
constexpr int kLPlane = 306;         // nodes of a plane in this layout
constexpr int kLSlot = 3 * kLPlane;  // a plane's three components

__device__ __forceinline__ constexpr int lane_off(int i, int j) {
  return kLCls[(i & 1) + 2 * (j & 1)] + (i >> 1) + kLRow * (j >> 1);
}

// Device arrays as buffer resources: one 32-bit lane offset and one scalar
// row offset address an entry (64-bit pointers per row would cost two scalar
// additions each, and a single wave issues those in place of arithmetic).
// Offsets are in bytes; the host checks that every array is below 4 GiB.
template <typename T>
struct LaneBuf {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ explicit LaneBuf(const T *p, unsigned bytes = 0xffffffffu)
      : r(__builtin_amdgcn_make_buffer_rsrc((void *)p, 0, bytes, 0x00027000)) {}
  __device__ __forceinline__ T load(unsigned lane, unsigned row) const {
    if constexpr (sizeof(T) == 8)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, (int)lane, (int)row, 0));
    else if constexpr (sizeof(T) == 4)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, (int)lane, (int)row, 0));
    else
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b8(r, (int)lane, (int)row, 0));
  }
  __device__ __forceinline__ void store(T v, unsigned lane, unsigned row) const {
    if constexpr (sizeof(T) == 8) {
      using V = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0));
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V, v), r, (int)lane, (int)row, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)lane, (int)row, 0);
    }
  }
};

// The next layer's two node planes (34 rows of 17 nodes) travel from memory
// to LDS in three batches, one per quadrature plane of the current layer:
// loaded at its start, stored at its end.  Lane t holds entry t (node t / 3,
// component t % 3) of a row; rows past a partial tile repeat its last one.
constexpr int kLBatch = 12;

// n1: the first plane's first node of the tile; t: the lane's entry; kN: rows
// in all (17 for a single plane)
template <typename T, int kB, int kN = 2 * kLRows>
__device__ __forceinline__ void lane_rows_load(T r[kLBatch], const TileArgs &a, int last, unsigned n1, unsigned t,
                                               const LaneBuf<T> &u) {
  const unsigned X = (unsigned)a.X, XY = (unsigned)a.XY;
#pragma unroll
  for (int q = 0; q < kLBatch; q++) {
    const int h = kB * kLBatch + q, j = h % kLRows;
    if (h >= kN) continue;
    const unsigned n = n1 + (h >= kLRows ? XY : 0u);
    r[q] = u.load((unsigned)sizeof(T) * (3 * n + t), 3 * (unsigned)sizeof(T) * X * (unsigned)min(j, last));
  }
}

// ev, od: the lane's place in the even and odd node rows of a plane
template <typename T, int kB, int kN = 2 * kLRows>
__device__ __forceinline__ void lane_rows_store(const T r[kLBatch], T *p1, T *p2, int ev, int od) {
#pragma unroll
  for (int q = 0; q < kLBatch; q++) {
    const int h = kB * kLBatch + q, j = h % kLRows;
    if (h >= kN) continue;
    (h >= kLRows ? p2 : p1)[(j & 1 ? od : ev) + kLRow * (j >> 1)] = r[q];
  }
}

// zeroes the Dirichlet dofs of a stored plane (n1: its first node of the tile;
// tn: the lane's node)
template <typename T>
__device__ __forceinline__ void lane_rows_mask(T *p, const TileArgs &a, int last, unsigned n1, unsigned tn, int ev,
                                               int od, int d, const LaneBuf<uint8_t> &bcn) {
  unsigned m[kLRows];
#pragma unroll
  for (int j = 0; j < kLRows; j++) m[j] = bcn.load(n1 + tn, (unsigned)a.X * (unsigned)min(j, last));
#pragma unroll
  for (int j = 0; j < kLRows; j++)
    if ((m[j] >> d) & 1u) p[(j & 1 ? od : ev) + kLRow * (j >> 1)] = T(0);
}

// per-lane constants of a rectilinear element: the collocation coefficients
// of the two in-plane directions scaled by 2 / h, and the Jacobian determinant
template <typename T>
struct LaneGeom {
  T cx[3], cy[3];  // (5/2, 10/3, 5/6) s times 2 / hx, 2 / hy
  T az, vol;       // 2 / hz, hx hy hz / 8
};

// collocated derivative at point a of a line with the scaled coefficients
template <typename T>
__device__ __forceinline__ T ldot(int a, const T c[3], T x0, T x1, T x2) {
  if (a == 0) return c[1] * x1 - c[0] * x0 - c[2] * x2;
  if (a == 1) return c[2] * (x2 - x0);
  return c[2] * x0 + c[0] * x2 - c[1] * x1;
}

// its transpose: y += C[a][.] v
template <typename T>
__device__ __forceinline__ void ldot_t(int a, const T c[3], T v, T &y0, T &y1, T &y2) {
  if (a == 0) {
    y0 -= c[0] * v;
    y1 += c[1] * v;
    y2 -= c[2] * v;
  } else if (a == 1) {
    const T t = c[2] * v;
    y0 -= t;
    y2 += t;
  } else {
    y0 += c[2] * v;
    y1 -= c[1] * v;
    y2 += c[0] * v;
  }
}

// Velocity of one element at quadrature plane c: U at its 9 points, Z the
// derivative along z there
template <typename T, int c>
__device__ __forceinline__ void lane_forward(const T *s0, const T *s1, const T *s2, const LaneGeom<T> &g, T U[3][9],
                                             T Z[3][9]) {
  const T d0 = (T)kD[c][0] * g.az, d1 = (T)kD[c][1] * g.az, d2 = (T)kD[c][2] * g.az;
#pragma unroll
  for (int f = 0; f < 3; f++) {
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const int o = f * kLPlane + lane_off(i, j);
        const T n0 = s0[o], n1 = s1[o], n2 = s2[o];
        if (c == 1) {
          U[f][3 * j + i] = n1;
          Z[f][3 * j + i] = d2 * (n2 - n0);
        } else {
          U[f][3 * j + i] = (T)kB[c][0] * n0 + (T)kB[c][1] * n1 + (T)kB[c][2] * n2;
          Z[f][3 * j + i] = d0 * n0 + d1 * n1 + d2 * n2;
        }
      }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      T *v = h ? Z[f] : U[f];
#pragma unroll
      for (int j = 0; j < 3; j++)
        interp3<T>(v[3 * j], v[3 * j + 1], v[3 * j + 2], v[3 * j], v[3 * j + 1], v[3 * j + 2]);
#pragma unroll
      for (int i = 0; i < 3; i++) interp3<T>(v[i], v[3 + i], v[6 + i], v[i], v[3 + i], v[6 + i]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Stress at the plane's points and its transposed derivatives:
// out[k][l][3j+i] += the plane's part of (A11_e u)(node (i, j, k), component l)
template <typename T, int c>
__device__ __forceinline__ void lane_stress(const T U[3][9], T Z[3][9], const LaneGeom<T> &g, const T et[9],
                                            T out[3][3][9]) {
  const T d0 = (T)kD[c][0] * g.az, d1 = (T)kD[c][1] * g.az, d2 = (T)kD[c][2] * g.az;
  T W[3][9];
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int p = 0; p < 9; p++) W[l][p] = T(0);
#pragma unroll
  for (int b = 0; b < 3; b++)
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int p = 3 * b + a;
      T G[3][3];  // G[k][l] = d u_l / d x_k
#pragma unroll
      for (int l = 0; l < 3; l++) {
        G[0][l] = ldot<T>(a, g.cx, U[l][3 * b], U[l][3 * b + 1], U[l][3 * b + 2]);
        G[1][l] = ldot<T>(b, g.cy, U[l][a], U[l][3 + a], U[l][6 + a]);
        G[2][l] = Z[l][p];
      }
      const T t = et[p] * ((T)(kW[a] * kW[b] * kW[c]) * g.vol), t2 = t + t;
      T sg[3][3];
      sg[0][0] = t2 * G[0][0];
      sg[1][1] = t2 * G[1][1];
      sg[2][2] = t2 * G[2][2];
      sg[0][1] = sg[1][0] = t * (G[0][1] + G[1][0]);
      sg[0][2] = sg[2][0] = t * (G[0][2] + G[2][0]);
      sg[1][2] = sg[2][1] = t * (G[1][2] + G[2][1]);
#pragma unroll
      for (int l = 0; l < 3; l++) {
        ldot_t<T>(a, g.cx, sg[0][l], W[l][3 * b], W[l][3 * b + 1], W[l][3 * b + 2]);
        ldot_t<T>(b, g.cy, sg[1][l], W[l][a], W[l][3 + a], W[l][6 + a]);
        Z[l][p] = sg[2][l];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
  for (int l = 0; l < 3; l++) {
    T Wn[9], Zn[9];
    interp_plane_t<T>(W[l], Wn);
    interp_plane_t<T>(Z[l], Zn);
#pragma unroll
    for (int n = 0; n < 9; n++) {
      if (c == 1) {
        const T z = d2 * Zn[n];
        out[0][l][n] -= z;
        out[1][l][n] += Wn[n];
        out[2][l][n] += z;
      } else {
        out[0][l][n] += (T)kB[c][0] * Wn[n] + d0 * Zn[n];
        out[1][l][n] += (T)kB[c][1] * Wn[n] + d1 * Zn[n];
        out[2][l][n] += (T)kB[c][2] * Wn[n] + d2 * Zn[n];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The sums are finished here: left alone, the compiler sinks the arithmetic
// past the next branch and keeps the node values alive in its place.
template <typename T>
__device__ __forceinline__ void lane_pin(T out[3][3][9]) {
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int n = 0; n < 9; n++) asm volatile("" : "+v"(out[k][l][n]));
}

// Node sums of one plane over the tile's elements, into the plane's window
// (component stride kLPlane).  Four ordered groups without a shared node
// within a group; the first writer of a node stores, later ones add.  w: the
// lane's own place in the window (lanes past a partial tile write to a spare
// one, so that no branch splits the sums).
template <typename T>
__device__ __forceinline__ void lane_window(T *w, bool moreX, bool moreY, const T o[3][9]) {
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const bool add = g == 1 ? moreX : (g == 2 ? moreY : (moreX || moreY));
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) {
        if ((i == 2 ? 1 : 0) + (j == 2 ? 2 : 0) != g) continue;
#pragma unroll
        for (int l = 0; l < 3; l++) {
          T *q = w + l * kLPlane + lane_off(i, j);
          if (g == 0) *q = o[l][3 * j + i];
          else {
            const T old = *q;
            *q = (add ? old : T(0)) + o[l][3 * j + i];
          }
        }
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// Writes a completed node plane: the tile's own nodes to y (or, on the
// tile's top plane, to the z face), the upper x face column and y face row.
// dirichlet: the plane holds Dirichlet dofs, whose rows are y = x.  kTop: P is
// the tile's top plane.
template <typename T, bool kBC, bool kTop>
__device__ __forceinline__ void lane_flush(const TileArgs &a, unsigned tile, const TileBox &tb, int P, const T *win,
                                           int lane, bool dirichlet, const LaneBuf<T> &x,
                                           const LaneBuf<uint8_t> &bcn, const LaneBuf<T> &y, const LaneBuf<T> &fbx,
                                           const LaneBuf<T> &fby, const LaneBuf<T> &fbz) {
  constexpr unsigned S = sizeof(T);
  const unsigned kl = (unsigned)(P - 2 * tb.z0);
  const int nyo = tb.yend ? 2 * tb.nyt + 1 : 2 * tb.nyt;
  const int R3 = 3 * (tb.xend ? 2 * tb.nxt + 1 : 2 * tb.nxt);
  const int il = lane / 3, d = lane - 3 * il;
  const bool zface = kTop && !tb.zend;
  const T *const even = win + kLPlane * d + kLCls[il & 1] + (il >> 1);
  const T *const odd = win + kLPlane * d + kLCls[2 + (il & 1)] + (il >> 1);
  const unsigned X = (unsigned)a.X, n0 = 2u * tb.x0 + (unsigned)a.XY * P + X * 2u * tb.y0;
  if (lane < R3) {
    T v[kLRows];
#pragma unroll
    for (int j = 0; j < kLRows; j++) v[j] = (j & 1) ? odd[kLRow * (j >> 1)] : even[kLRow * (j >> 1)];
    if (kBC && dirichlet && !zface) {
      unsigned m[kLRows];
      T xv[kLRows];
#pragma unroll
      for (int j = 0; j < kLRows; j++) {
        const unsigned row = X * (unsigned)min(j, nyo - 1);
        m[j] = bcn.load(n0 + (unsigned)il, row);
        xv[j] = x.load(S * (3 * n0 + (unsigned)lane), 3 * S * row);
      }
#pragma unroll
      for (int j = 0; j < kLRows; j++) v[j] = ((m[j] >> d) & 1u) ? xv[j] : v[j];
    }
    auto rows = [&](const LaneBuf<T> &q, unsigned o, unsigned rs) {
      if (nyo >= 2 * kLT) {
#pragma unroll
        for (int j = 0; j < 2 * kLT; j++) q.store(v[j], o, rs * j);
        if (nyo > 2 * kLT) q.store(v[2 * kLT], o, rs * 2 * kLT);
      } else {
#pragma unroll
        for (int j = 0; j < 2 * kLT - 1; j++)
          if (j < nyo) q.store(v[j], o, rs * j);
      }
    };
    if (zface) rows(fbz, S * (3 * tile * (unsigned)a.fbz_n + (unsigned)lane), 3 * S * kLRows);
    else rows(y, S * (3 * n0 + (unsigned)lane), 3 * S * X);
  }
  if (!tb.xend && lane < 3 * (2 * tb.nyt + 1)) {
    // lane = 3 jl + l: node (2 nxt, jl)
    const T *q = win + kLPlane * d + kLCls[2 * (il & 1)] + tb.nxt + kLRow * (il >> 1);
    fbx.store(*q, S * (3 * (tile * (unsigned)a.fbx_n + kLRows * kl) + (unsigned)lane), 0);
  }
  if (!tb.yend && lane < R3)
    fby.store(even[kLRow * tb.nyt], S * (3 * (tile * (unsigned)a.fby_n + kLRows * kl) + (unsigned)lane), 0);
}

// kBC: Dirichlet rows are written y = x (the face pass leaves them alone);
// otherwise they are left as the element sums.  bcp: per tile column and node
// plane, whether the tile's nodes there have a Dirichlet dof.  ax: 2 / h of the mx element
// columns, the my rows and the mz layers.
template <typename T, bool kBC>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 2 : 1)))
    a11_lane_kernel(TileArgs a, const T *__restrict__ ax, const T *__restrict__ eta_,
                    const uint8_t *__restrict__ bcn_, const uint8_t *__restrict__ bcp, const T *__restrict__ u_, T *__restrict__ y_,
                    T *__restrict__ fbx_, T *__restrict__ fby_, T *__restrict__ fbz_) {
  // five plane slots: the layer's three planes and the next layer's two
  __shared__ T sm[5 * kLSlot];
  const unsigned tile = (unsigned)xcd_tile(blockIdx.x, a.ntiles);
  const TileBox tb = tile_box(a, tile);
  const LaneBuf<T> eta(eta_), u(u_), y(y_), fbx(fbx_), fby(fby_), fbz(fbz_);
  const LaneBuf<uint8_t> bcn(bcn_);
  const int lane = threadIdx.x;
  const int lx = lane % kLT, ly = lane / kLT;
  const bool live = lx < tb.nxt && ly < tb.nyt;
  // lanes past a partial tile compute its last element with a zero
  // determinant; their zero sums fall on nodes that are stored or added to
  // by the tile's own elements afterwards
  const int cx = min(lx, tb.nxt - 1), cy = min(ly, tb.nyt - 1);
  const int li = cx + kLRow * cy, lw = lx + kLRow * ly;
  const bool moreX = lx + 1 < tb.nxt, moreY = ly + 1 < tb.nyt;
  // entry of the row loads (clamped to the tile's nodes), its node, and its
  // places in the slots (lanes past entry 50 write to a row's padding)
  const unsigned t = min(lane, 3 * (2 * tb.nxt + 1) - 1), tn = t / 3;
  const int d = lane % 3, il = min(lane / 3, kLRows);
  const int ev = kLPlane * d + kLCls[il & 1] + (il >> 1), od = kLPlane * d + kLCls[2 + (il & 1)] + (il >> 1);
  const int last = 2 * tb.nyt;
  const unsigned XY = (unsigned)a.XY;
  unsigned np = 2u * tb.x0 + (unsigned)a.X * 2u * tb.y0 + XY * 2u * tb.z0;  // first node of the tile in plane 2 ek
  // bit P - 2 z0: Dirichlet dofs in the tile's plane P (one vector load for
  // the whole chunk, at most 63 planes; a byte load per plane would be waited
  // for together with every store in flight)
  const uint8_t *fl = bcp + (2L * a.mz + 1) * (tb.tx + (long)a.ntx * tb.ty) + 2 * tb.z0;
  const unsigned long long bits = __ballot(fl[min(lane, 2 * tb.nzt)] != 0);
  // 2 / hz of the chunk's layers, one per lane
  const T szs = ax[a.mx + a.my + tb.z0 + min(lane, tb.nzt - 1)];

  LaneGeom<T> g;
  const T sx = ax[tb.x0 + cx], sy = ax[a.mx + tb.y0 + cy];
  g.cx[0] = (T)(2.5 * kS) * sx;
  g.cx[1] = (T)(10.0 / 3.0 * kS) * sx;
  g.cx[2] = (T)(5.0 / 6.0 * kS) * sx;
  g.cy[0] = (T)(2.5 * kS) * sy;
  g.cy[1] = (T)(10.0 / 3.0 * kS) * sy;
  g.cy[2] = (T)(5.0 / 6.0 * kS) * sy;

  {
    // planes 2 z0 .. 2 z0 + 2
    T r0[kLBatch], r1[kLBatch], r2[kLBatch];
    lane_rows_load<T, 0>(r0, a, last, np, t, u);
    lane_rows_load<T, 1>(r1, a, last, np, t, u);
    lane_rows_store<T, 0>(r0, sm, sm + kLSlot, ev, od);
    lane_rows_load<T, 2>(r2, a, last, np, t, u);
    lane_rows_store<T, 1>(r1, sm, sm + kLSlot, ev, od);
    lane_rows_load<T, 0, kLRows>(r0, a, last, np + 2 * XY, t, u);
    lane_rows_load<T, 1, kLRows>(r1, a, last, np + 2 * XY, t, u);
    lane_rows_store<T, 2>(r2, sm, sm + kLSlot, ev, od);
    lane_rows_store<T, 0, kLRows>(r0, sm + 2 * kLSlot, nullptr, ev, od);
    lane_rows_store<T, 1, kLRows>(r1, sm + 2 * kLSlot, nullptr, ev, od);
    for (int k = 0; k < 3; k++)
      if ((bits >> k) & 1) lane_rows_mask<T>(sm + k * kLSlot, a, last, np + k * XY, tn, ev, od, d, bcn);
  }
  T out[3][3][9];
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int n = 0; n < 9; n++) out[2][l][n] = T(0);

  unsigned oe = (unsigned)sizeof(T) * (tb.x0 + cx + (unsigned)a.mx * (tb.y0 + cy + (unsigned)a.my * tb.z0));
  const unsigned qs = (unsigned)sizeof(T) * (unsigned)a.nel;
  int slot = 0;  // of plane 2 ek; its successors follow modulo 5
  for (int kz = 0; kz < tb.nzt; kz++) {
    const int ek = tb.z0 + kz;
    auto place = [&](int k) { return sm + kLSlot * (slot + k >= 5 ? slot + k - 5 : slot + k); };
    T *const s0 = place(0), *const s1 = place(1), *const s2 = place(2), *const s3 = place(3), *const s4 = place(4);
    const bool more = kz + 1 < tb.nzt;
    // (the last layer of the chunk loads its own planes again, into free slots)
    const unsigned nn = more ? np + 3 * XY : np + XY;
    const T sz = __shfl(szs, kz);
    g.az = sz;
    g.vol = live ? T(1) / (sx * sy * sz) : T(0);
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int n = 0; n < 9; n++) {
        out[0][l][n] = out[2][l][n];  // the lower element's share of the common plane
        out[1][l][n] = out[2][l][n] = T(0);
      }
    __syncthreads();
    // The loads of a plane are in flight during its forward stage only: held
    // through the stress stage, the compiler would wait for each of them at
    // once to move it out of the registers that stage needs.
    T et[9], r[kLBatch], U[3][9], Z[3][9];
    int lq = li;
#pragma unroll
    for (int p = 0; p < 9; p++) et[p] = eta.load(oe, qs * (0 + p));
    lane_rows_load<T, 0>(r, a, last, nn, t, u);
    lane_forward<T, 0>(s0 + lq, s1 + lq, s2 + lq, g, U, Z);
    lane_rows_store<T, 0>(r, s3, s4, ev, od);
    lane_stress<T, 0>(U, Z, g, et, out);
    lane_pin<T>(out);
    // the node values are read again per quadrature plane, not held: an
    // index the compiler knows nothing about keeps it from merging the reads
    asm volatile("" : "+v"(lq));
#pragma unroll
    for (int p = 0; p < 9; p++) et[p] = eta.load(oe, qs * (9 + p));
    lane_rows_load<T, 1>(r, a, last, nn, t, u);
    lane_forward<T, 1>(s0 + lq, s1 + lq, s2 + lq, g, U, Z);
    lane_rows_store<T, 1>(r, s3, s4, ev, od);
    lane_stress<T, 1>(U, Z, g, et, out);
    lane_pin<T>(out);
    asm volatile("" : "+v"(lq));
#pragma unroll
    for (int p = 0; p < 9; p++) et[p] = eta.load(oe, qs * (18 + p));
    lane_rows_load<T, 2>(r, a, last, nn, t, u);
    lane_forward<T, 2>(s0 + lq, s1 + lq, s2 + lq, g, U, Z);
    lane_rows_store<T, 2>(r, s3, s4, ev, od);
    lane_stress<T, 2>(U, Z, g, et, out);
    lane_pin<T>(out);
    if (more && ((bits >> (2 * kz + 3)) & 1)) lane_rows_mask<T>(s3, a, last, nn, tn, ev, od, d, bcn);
    if (more && ((bits >> (2 * kz + 4)) & 1)) lane_rows_mask<T>(s4, a, last, nn + XY, tn, ev, od, d, bcn);
    __syncthreads();
    // the planes 2 ek and 2 ek + 1 are complete: their slots become windows
    lane_window<T>(s0 + lw, moreX, moreY, out[0]);
    lane_window<T>(s1 + lw, moreX, moreY, out[1]);
    __syncthreads();
    lane_flush<T, kBC, false>(a, tile, tb, 2 * ek, s0, lane, (bits >> (2 * kz)) & 1, u, bcn, y, fbx, fby, fbz);
    lane_flush<T, kBC, false>(a, tile, tb, 2 * ek + 1, s1, lane, (bits >> (2 * kz + 1)) & 1, u, bcn, y, fbx, fby, fbz);
    __syncthreads();
    np += 2 * XY;
    oe += (unsigned)sizeof(T) * (unsigned)(a.mx * a.my);
    slot = slot + 2 >= 5 ? slot - 3 : slot + 2;
  }
  T *const top = sm + kLSlot * slot;
  lane_window<T>(top + lw, moreX, moreY, out[2]);
  __syncthreads();
  lane_flush<T, kBC, true>(a, tile, tb, 2 * (tb.z0 + tb.nzt), top, lane, (bits >> (2 * tb.nzt)) & 1, u, bcn, y, fbx,
                          fby, fbz);
}
