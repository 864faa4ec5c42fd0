// lane.h -- device code shared by the kernels that give an element one lane.
//
// A wave owns an 8 x 8 tile of elements in x-y, one element per lane, and
// marches through a chunk of element layers in z.  The tile's node planes lie
// in LDS, where neighbouring elements share them; everything else of an
// element stays in its lane's registers.  Output sums go through LDS too, one
// node plane at a time (the slot of a plane that is no longer read), and from
// there to memory in whole node rows.  Node sums on a tile's upper faces go to
// face buffers, as in the tile kernels.
#pragma once

#include "tile.h"

namespace ptmf {
namespace {

constexpr int kLT = 8;     // elements per tile side
constexpr int kLRow = 9;   // row stride of a node class
constexpr int kLRows = 17; // node rows and columns of a tile
constexpr int kLMaxZ = 31; // element layers of a chunk, at most
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
// Offsets are in bytes from the pointer given, which is a node plane's or an
// element layer's first entry of the tile: any array size will do.
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

// a tile's node rows lie within the 32-bit row offset
inline bool lane_fits(const Box &b) { return 8 * 3 * (b.Y < kLRows ? b.Y : kLRows) * b.X < (1L << 32); }

// Work decomposition of a lane kernel that runs `waves` waves at a time, each
// spending `ends` of a layer's time on its first and last planes.  layers: the
// time it takes, in those of a layer.
inline TileArgs lane_args(const Box &b, long waves, double ends, double *layers = nullptr) {
  TileArgs a;
  a.mx = b.mx; a.my = b.my; a.mz = b.mz;
  a.X = b.X; a.XY = b.X * b.Y; a.nel = b.nel;
  a.TX = a.TY = kLT;
  a.ntx = (b.mx + kLT - 1) / kLT;
  a.nty = (b.my + kLT - 1) / kLT;
  double best = 1e300;
  for (int zc = 1; zc <= b.mz && zc <= kLMaxZ; zc++) {
    const long nt = (long)a.ntx * a.nty * ((b.mz + zc - 1) / zc);
    const double cost = (double)((nt + waves - 1) / waves) * (zc + ends);
    if (cost < best) {
      best = cost;
      a.ZC = zc;
      a.ntiles = nt;
    }
  }
  a.fbx_n = a.fby_n = (long)kLRows * (2 * a.ZC + 1);
  a.fbz_n = kLRows * kLRows;
  if (layers) *layers = best;
  return a;
}

// What a lane is to its tile.
struct LaneTile {
  unsigned tile;
  TileBox tb;
  int lane, lx, ly;
  // lanes past a partial tile compute its last element (cx, cy) again; what
  // they sum must come out zero: it falls on nodes that the tile's own
  // elements store or add to afterwards
  bool live;
  int cx, cy;
  int li, lw;         // place of the element's node (0, 0) in a slot, for reading and for the sums
  bool moreX, moreY;  // another element of the tile follows
  // row transfers: entry t (clamped to the tile's nodes) and node tn of a row,
  // component d; places in the even and odd rows of a slot (lanes past entry
  // 50 write to a row's padding); the tile's last row
  unsigned t, tn;
  int d, il, ev, od, last;
};

__device__ __forceinline__ LaneTile lane_tile(const TileArgs &a, unsigned tile) {
  LaneTile q;
  q.tile = tile;
  q.tb = tile_box(a, tile);
  q.lane = threadIdx.x;
  q.lx = q.lane % kLT;
  q.ly = q.lane / kLT;
  q.live = q.lx < q.tb.nxt && q.ly < q.tb.nyt;
  q.cx = min(q.lx, q.tb.nxt - 1);
  q.cy = min(q.ly, q.tb.nyt - 1);
  q.li = q.cx + kLRow * q.cy;
  q.lw = q.lx + kLRow * q.ly;
  q.moreX = q.lx + 1 < q.tb.nxt;
  q.moreY = q.ly + 1 < q.tb.nyt;
  q.t = min(q.lane, 3 * (2 * q.tb.nxt + 1) - 1);
  q.tn = q.t / 3;
  q.d = q.lane % 3;
  q.il = min(q.lane / 3, kLRows);
  q.ev = kLPlane * q.d + kLCls[q.il & 1] + (q.il >> 1);
  q.od = kLPlane * q.d + kLCls[2 + (q.il & 1)] + (q.il >> 1);
  q.last = 2 * q.tb.nyt;
  return q;
}

// first node of the tile in node plane P
__device__ __forceinline__ long lane_node(const TileArgs &a, const TileBox &tb, int P) {
  return 2L * tb.x0 + a.X * (2L * tb.y0) + a.XY * (long)P;
}

// One or two node planes (17 rows of 17 nodes each) travel from memory to LDS
// in batches of 12 rows: rows 12 kB .. of kN in all.  Lane t holds entry t
// (node t / 3, component t % 3) of a row; rows past a partial tile repeat its
// last one.  v1, v2: the planes' first nodes of the tile.
constexpr int kLBatch = 12;

template <typename T, int kB, int kN = 2 * kLRows>
__device__ __forceinline__ void lane_rows_load(T r[kLBatch], const LaneTile &q, long X, const LaneBuf<T> &v1,
                                               const LaneBuf<T> &v2) {
#pragma unroll
  for (int k = 0; k < kLBatch; k++) {
    const int h = kB * kLBatch + k, j = h % kLRows;
    if (h >= kN) continue;
    r[k] = (h >= kLRows ? v2 : v1)
               .load((unsigned)sizeof(T) * q.t, 3 * (unsigned)sizeof(T) * (unsigned)X * (unsigned)min(j, q.last));
  }
}

template <typename T, int kB, int kN = 2 * kLRows>
__device__ __forceinline__ void lane_rows_store(const T r[kLBatch], const LaneTile &q, T *p1, T *p2) {
#pragma unroll
  for (int k = 0; k < kLBatch; k++) {
    const int h = kB * kLBatch + k, j = h % kLRows;
    if (h >= kN) continue;
    (h >= kLRows ? p2 : p1)[(j & 1 ? q.od : q.ev) + kLRow * (j >> 1)] = r[k];
  }
}

// Dirichlet dofs of the tile's node plane P as the lane that holds entry t of
// its rows sees them: bit j for row j, none for lanes past the rows' entries.
// One word a plane: a byte per node would be 17 loads, waited for behind every
// store in flight.
__device__ __forceinline__ unsigned lane_bc_word(const TileArgs &a, const LaneTile &q, const unsigned *__restrict__ bcw,
                                                 int P) {
  return (bcw + 64 * ((2L * a.mz + 1) * (q.tb.tx + (long)a.ntx * q.tb.ty) + P))[q.lane];
}

// the Dirichlet dofs of a batch of rows to zero (m1, m2: the planes' words)
template <typename T, int kB, int kN = 2 * kLRows>
__device__ __forceinline__ void lane_rows_mask(T r[kLBatch], unsigned m1, unsigned m2) {
  if (__ballot((m1 | m2) != 0u) == 0) return;
#pragma unroll
  for (int k = 0; k < kLBatch; k++) {
    const int h = kB * kLBatch + k, j = h % kLRows;
    if (h >= kN) continue;
    r[k] = (((h >= kLRows ? m2 : m1) >> j) & 1u) ? T(0) : r[k];
  }
}

// One component at quadrature plane c of an element: V at the plane's 9 points
// and Z, its zeta derivative times d2 / kD[1][2]; s0, s1, s2: the element's
// node (0, 0) in the three planes (kCentre: the middle plane's centre node is
// `centre`, not in its slot)
template <typename T, int c, bool kCentre = false>
__device__ __forceinline__ void lane_field(const T *s0, const T *s1, const T *s2, T d0, T d1, T d2, T V[9], T Z[9],
                                           T centre = T(0)) {
#pragma unroll
  for (int j = 0; j < 3; j++)
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int o = lane_off(i, j);
      const T n0 = s0[o], n1 = kCentre && i == 1 && j == 1 ? centre : s1[o], n2 = s2[o];
      if (c == 1) {
        V[3 * j + i] = n1;
        Z[3 * j + i] = d2 * (n2 - n0);
      } else {
        V[3 * j + i] = (T)kB[c][0] * n0 + (T)kB[c][1] * n1 + (T)kB[c][2] * n2;
        Z[3 * j + i] = d0 * n0 + d1 * n1 + d2 * n2;
      }
    }
#pragma unroll
  for (int h = 0; h < 2; h++) {
    T *v = h ? Z : V;
#pragma unroll
    for (int j = 0; j < 3; j++)
      interp3<T>(v[3 * j], v[3 * j + 1], v[3 * j + 2], v[3 * j], v[3 * j + 1], v[3 * j + 2]);
#pragma unroll
    for (int i = 0; i < 3; i++) interp3<T>(v[i], v[3 + i], v[6 + i], v[i], v[3 + i], v[6 + i]);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// The transpose: out[k][n] += the plane's in-plane fluxes W and zeta fluxes Z
template <typename T, int c>
__device__ __forceinline__ void lane_field_t(const T W[9], const T Z[9], T d0, T d1, T d2, T o0[9], T o1[9],
                                             T o2[9]) {
  T Wn[9], Zn[9];
  interp_plane_t<T>(W, Wn);
  interp_plane_t<T>(Z, Zn);
#pragma unroll
  for (int n = 0; n < 9; n++) {
    // (each term an addition to the sum: one operation apiece)
    if (c == 1) {
      o0[n] -= d2 * Zn[n];
      o1[n] += Wn[n];
      o2[n] += d2 * Zn[n];
    } else {
      o0[n] += (T)kB[c][0] * Wn[n];
      o0[n] += d0 * Zn[n];
      o1[n] += (T)kB[c][1] * Wn[n];
      o1[n] += d1 * Zn[n];
      o2[n] += (T)kB[c][2] * Wn[n];
      o2[n] += d2 * Zn[n];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
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

// Dirichlet rows of a flushed plane
enum LaneBC {
  kLaneSums,  // left as the element sums
  kLaneZero,  // y = 0
  kLaneOne    // y = 1
};

// Writes a completed node plane P: the tile's own nodes to y (or, on the
// tile's top plane, kTop, to the z face), the upper x face column and y face
// row.  m: the plane's lane_bc_word.
template <typename T, LaneBC kBC, bool kTop>
__device__ __forceinline__ void lane_flush(const TileArgs &a, const LaneTile &q, int P, const T *win, unsigned m,
                                           T *__restrict__ y, T *__restrict__ fbx, T *__restrict__ fby,
                                           T *__restrict__ fbz) {
  constexpr unsigned S = sizeof(T);
  const TileBox &tb = q.tb;
  const int lane = q.lane;
  const unsigned kl = (unsigned)(P - 2 * tb.z0);
  const int nyo = tb.yend ? 2 * tb.nyt + 1 : 2 * tb.nyt;
  const int R3 = 3 * (tb.xend ? 2 * tb.nxt + 1 : 2 * tb.nxt);
  const int il = lane / 3;  // not q.il: lanes past the row's entries do not store
  const bool zface = kTop && !tb.zend;
  const T *const even = win + q.ev, *const odd = win + q.od;
  const unsigned X = (unsigned)a.X;
  const long n0 = lane_node(a, tb, P);
  if (lane < R3) {
    T v[kLRows];
#pragma unroll
    for (int j = 0; j < kLRows; j++) v[j] = (j & 1) ? odd[kLRow * (j >> 1)] : even[kLRow * (j >> 1)];
    if (kBC != kLaneSums && !zface && __ballot(m != 0u) != 0) {
#pragma unroll
      for (int j = 0; j < kLRows; j++) v[j] = ((m >> j) & 1u) ? T(kBC == kLaneOne ? 1 : 0) : v[j];
    }
    auto rows = [&](const LaneBuf<T> &w, unsigned rs) {
      const unsigned o = S * (unsigned)lane;
      if (nyo >= 2 * kLT) {
#pragma unroll
        for (int j = 0; j < 2 * kLT; j++) w.store(v[j], o, rs * j);
        if (nyo > 2 * kLT) w.store(v[2 * kLT], o, rs * 2 * kLT);
      } else {
#pragma unroll
        for (int j = 0; j < 2 * kLT - 1; j++)
          if (j < nyo) w.store(v[j], o, rs * j);
      }
    };
    if (zface) rows(LaneBuf<T>(fbz + 3 * q.tile * a.fbz_n), 3 * S * kLRows);
    else rows(LaneBuf<T>(y + 3 * n0), 3 * S * X);
  }
  if (!tb.xend && lane < 3 * (2 * tb.nyt + 1)) {
    // lane = 3 jl + l: node (2 nxt, jl)
    const T *p = win + kLPlane * q.d + kLCls[2 * (il & 1)] + tb.nxt + kLRow * (il >> 1);
    fbx[3 * (q.tile * a.fbx_n + (long)kLRows * kl) + lane] = *p;
  }
  if (!tb.yend && lane < R3) fby[3 * (q.tile * a.fby_n + (long)kLRows * kl) + lane] = even[kLRow * tb.nyt];
}

}  // namespace
}  // namespace ptmf
