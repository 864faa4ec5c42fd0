// a11_col.h -- the A11 MatMult of a small box, any mesh, with one lane per node
// column of an element (included by a11.hip, inside its anonymous namespace).
//
// Nine lanes hold an element, one each of its 3 x 3 node columns in z, and a
// wave five elements, in index order: a box of any shape fills the waves.  The
// z direction of every contraction happens in a lane's registers, x between the
// lanes of a quad, y through LDS.  The element's 81 sums go to memory; a second
// pass adds up each node's up to eight elements in a fixed order.
//
// What bounds it: on small boxes one wave's latency, less than half of the tile
// kernel's, whose lanes do the work of three of these (16^3, kernel and what
// follows it in one launch after the other: 6.0 us and 3.3 us for the sums, the
// tile kernel 13.1 and 3.8 us).  On larger ones instruction issue, at three waves
// per SIMD (1,210 vector instructions for five elements, 730 of them FP64; VALU
// busy 87 %), and the 650 bytes of sums per element: 45 x 37 x 29 in 31 and 9 us
// (tile kernel 55 and 6 us).  With x in LDS too, seven elements to a wave, bank
// conflicts bound it (16^3 6.9 us).

constexpr int kColElems = 5;  // elements of a wave

// a lane's rows and columns of the 1-D tables: entry k couples it to the lane
// k places on (modulo 3) in the direction
template <typename T>
struct ColRow {
  T b[3], bt[3], c[3], ct[3];  // B[r][.], B[.][r], C[r][.], C[.][r]
  __device__ __forceinline__ explicit ColRow(int r) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      b[k] = sel3<T>(r, kB[0][k], kB[1][(1 + k) % 3], kB[2][(2 + k) % 3]);
      bt[k] = sel3<T>(r, kB[k][0], kB[(1 + k) % 3][1], kB[(2 + k) % 3][2]);
      c[k] = sel3<T>(r, kC[0][k], kC[1][(1 + k) % 3], kC[2][(2 + k) % 3]);
      ct[k] = sel3<T>(r, kC[k][0], kC[(1 + k) % 3][1], kC[(2 + k) % 3][2]);
    }
  }
};

// the value of the lane k places on in x: the columns of a row are lanes 0, 1
// and 2 of a quad (lane 3 does as lane 2)
template <int k, typename T>
__device__ __forceinline__ T col_x(T v) {
  constexpr int ctrl = k == 1 ? (1 | 2 << 2 | 0 << 4 | 0 << 6) : (2 | 0 << 2 | 1 << 4 | 1 << 6);
  if constexpr (sizeof(T) == 8) {
    struct Pair { int a, b; } p = __builtin_bit_cast(Pair, v);
    p.a = __builtin_amdgcn_mov_dpp(p.a, ctrl, 0xf, 0xf, true);
    p.b = __builtin_amdgcn_mov_dpp(p.b, ctrl, 0xf, 0xf, true);
    return __builtin_bit_cast(T, p);
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), ctrl, 0xf, 0xf, true));
  }
}

template <typename T>
__device__ __forceinline__ T col_mix_x(T v, const T m[3]) {
  return m[0] * v + m[1] * col_x<1>(v) + m[2] * col_x<2>(v);
}

__device__ __forceinline__ void col_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// the same in y through LDS, for kN values; n1, n2: the lanes one and two on
template <typename T, int kN>
__device__ __forceinline__ void col_mix_y(T (*sm)[64], int lane, T *v, const T m[3], int n1, int n2) {
#pragma unroll
  for (int f = 0; f < kN; f++) sm[f][lane] = v[f];
  col_fence();
#pragma unroll
  for (int f = 0; f < kN; f++) v[f] = m[0] * v[f] + m[1] * sm[f][n1] + m[2] * sm[f][n2];
  col_fence();
}

struct ColArgs {
  unsigned mx, my, mz, ne, nwaves;
};

// the element sums es of wave `wave`'s elements
template <typename T>
__device__ __forceinline__ void col_wave(const ColArgs &a, unsigned wave, const T *__restrict__ xc,
                                         const T *__restrict__ eta, const uint8_t *__restrict__ bcn,
                                         const T *__restrict__ u, T *__restrict__ es, T (*sm)[64]) {
  // quad 5 j + s holds row j of element s (the last quad repeats its neighbour):
  // rows that exchange values lie in different LDS banks
  const int lane = threadIdx.x, quad = min(lane >> 2, 3 * kColElems - 1), j = quad / kColElems,
            s = quad - kColElems * j, i = min(lane & 3, 2);
  const unsigned el = (unsigned)kColElems * wave + (unsigned)s;
  const bool live = (lane & 3) < 3 && lane < 12 * kColElems && el < a.ne;
  const unsigned e = min(el, a.ne - 1u), X = 2 * a.mx + 1, XY = X * (2 * a.my + 1);
  const unsigned r = e / a.mx, ex = e - r * a.mx, ez = r / a.my, ey = r - ez * a.my;
  const unsigned node = 2 * ex + i + X * (2 * ey + j) + XY * (2 * ez);
  const ColRow<T> rx(i), ry(j);
  const int n1 = 4 * (kColElems * (j == 2 ? 0 : j + 1) + s) + i, n2 = 4 * (kColElems * (j == 0 ? 2 : j - 1) + s) + i;

  T v[18], et[3];  // [x, y, z, u_x, u_y, u_z][z index]
  unsigned m[3];
  T org[3];
#pragma unroll
  for (int d = 0; d < 3; d++) org[d] = xc[3 * (node - i - X * j) + d];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const unsigned n = node + XY * k;
    m[k] = bcn[n];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      v[3 * d + k] = xc[3 * n + d];
      v[9 + 3 * d + k] = u[3 * n + d];
    }
    et[k] = eta[(i + 3 * j + 9 * k) * a.ne + e];
  }
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int d = 0; d < 3; d++) v[9 + 3 * d + k] = ((m[k] >> d) & 1u) ? T(0) : v[9 + 3 * d + k];
  // positions from the element's first node: no digits are lost to the
  // element's distance from the origin
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int k = 0; k < 3; k++) v[3 * d + k] -= org[d];
#pragma unroll
  for (int f = 0; f < 6; f++) interp3<T>(v[3 * f], v[3 * f + 1], v[3 * f + 2], v[3 * f], v[3 * f + 1], v[3 * f + 2]);
#pragma unroll
  for (int f = 0; f < 18; f++) v[f] = col_mix_x<T>(v[f], rx.b);
  col_mix_y<T, 18>(sm, lane, v, ry.b, n1, n2);
#pragma unroll
  for (int f = 0; f < 18; f++) sm[f][lane] = v[f];
  col_fence();

  T w[9];  // [component][z index]
#pragma unroll
  for (int f = 0; f < 9; f++) w[f] = T(0);
  const T wxy = sel3<T>(i, kW[0], kW[1], kW[2]) * sel3<T>(j, kW[0], kW[1], kW[2]);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    T M[3][3], G[3][3];  // d x_d / d xi_j, d u_l / d xi_j
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const int fx = 3 * d + k, fu = 9 + 3 * d + k;
      M[0][d] = col_mix_x<T>(v[fx], rx.c);
      M[1][d] = ry.c[0] * v[fx] + ry.c[1] * sm[fx][n1] + ry.c[2] * sm[fx][n2];
      M[2][d] = cdot<T>(k, v[3 * d], v[3 * d + 1], v[3 * d + 2]);
      G[0][d] = col_mix_x<T>(v[fu], rx.c);
      G[1][d] = ry.c[0] * v[fu] + ry.c[1] * sm[fu][n1] + ry.c[2] * sm[fu][n2];
      G[2][d] = cdot<T>(k, v[9 + 3 * d], v[9 + 3 * d + 1], v[9 + 3 * d + 2]);
    }
    col_fence();
    T A[3][3];  // detJ d xi_j / d x_k
    A[0][0] = M[1][1] * M[2][2] - M[2][1] * M[1][2];
    A[0][1] = M[2][1] * M[0][2] - M[0][1] * M[2][2];
    A[0][2] = M[0][1] * M[1][2] - M[1][1] * M[0][2];
    A[1][0] = M[2][0] * M[1][2] - M[1][0] * M[2][2];
    A[1][1] = M[0][0] * M[2][2] - M[2][0] * M[0][2];
    A[1][2] = M[1][0] * M[0][2] - M[0][0] * M[1][2];
    A[2][0] = M[1][0] * M[2][1] - M[2][0] * M[1][1];
    A[2][1] = M[2][0] * M[0][1] - M[0][0] * M[2][1];
    A[2][2] = M[0][0] * M[1][1] - M[1][0] * M[0][1];
    const T t = et[k] * (wxy * (T)kW[k]) * recip<T>(M[0][0] * A[0][0] + M[1][0] * A[0][1] + M[2][0] * A[0][2]);
    T H[3][3];  // detJ d u_l / d x_k
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
      for (int l = 0; l < 3; l++) H[q][l] = A[q][0] * G[0][l] + A[q][1] * G[1][l] + A[q][2] * G[2][l];
    T S[3][3];
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
      for (int l = 0; l <= q; l++) S[q][l] = S[l][q] = t * (H[q][l] + H[l][q]);
#pragma unroll
    for (int l = 0; l < 3; l++) {
      const T f0 = A[0][0] * S[0][l] + A[1][0] * S[1][l] + A[2][0] * S[2][l];
      const T f1 = A[0][1] * S[0][l] + A[1][1] * S[1][l] + A[2][1] * S[2][l];
      const T f2 = A[0][2] * S[0][l] + A[1][2] * S[1][l] + A[2][2] * S[2][l];
      // the level's slots of the forward fields are read by now
      sm[3 * l + k][lane] = f1;
      w[3 * l + k] += rx.ct[0] * f0;
      w[3 * l + k] += rx.ct[1] * col_x<1>(f0);
      w[3 * l + k] += rx.ct[2] * col_x<2>(f0);
      w[3 * l + k] += ry.ct[0] * f1;
#pragma unroll
      for (int q = 0; q < 3; q++)
        if (k != 1 || q != 1) w[3 * l + q] += (T)kC[k][q] * f2;
    }
    col_fence();
#pragma unroll
    for (int l = 0; l < 3; l++) {
      w[3 * l + k] += ry.ct[1] * sm[3 * l + k][n1];
      w[3 * l + k] += ry.ct[2] * sm[3 * l + k][n2];
    }
    col_fence();
  }
#pragma unroll
  for (int l = 0; l < 3; l++)
    interp3t<T>(w[3 * l], w[3 * l + 1], w[3 * l + 2], w[3 * l], w[3 * l + 1], w[3 * l + 2]);
#pragma unroll
  for (int f = 0; f < 9; f++) w[f] = col_mix_x<T>(w[f], rx.bt);
  col_mix_y<T, 9>(sm, lane, w, ry.bt, n1, n2);
  if (live) {
    // entry 3 e + i of row 3 (3 k + l) + j: component l of local node (i, j, k)
    const unsigned o = 3 * (a.ne * j + el) + i;
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int l = 0; l < 3; l++) (es + 9 * (3 * k + l) * (long)a.ne)[o] = w[3 * l + k];
  }
}

template <typename T>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
    a11_col_kernel(ColArgs a, const T *__restrict__ xc, const T *__restrict__ eta, const uint8_t *__restrict__ bcn,
                   const T *__restrict__ u, T *__restrict__ es) {
  __shared__ T sm[18][64];
  col_wave<T>(a, (unsigned)xcd_tile(blockIdx.x, a.nwaves), xc, eta, bcn, u, es, sm);
}

// Sums of node (I, J, K) over its elements, lowest first
template <typename T>
__device__ __forceinline__ void col_sum(const ColArgs &a, unsigned I, unsigned J, unsigned K, const T *__restrict__ es,
                                        T sum[3]) {
  T v[8][3];
#pragma unroll
  for (int s = 0; s < 8; s++) {  // all in flight together
    const bool dx = s & 1, dy = s & 2, dz = s & 4;
    const int x = (int)(I >> 1) - (dx ? 0 : 1), y = (int)(J >> 1) - (dy ? 0 : 1), z = (int)(K >> 1) - (dz ? 0 : 1);
    const bool has = (dx ? x < (int)a.mx : !(I & 1) && x >= 0) && (dy ? y < (int)a.my : !(J & 1) && y >= 0) &&
                     (dz ? z < (int)a.mz : !(K & 1) && z >= 0);
#pragma unroll
    for (int l = 0; l < 3; l++) v[s][l] = T(0);
    if (!has) continue;
    const int i = (int)I - 2 * x, j = (int)J - 2 * y, k = (int)K - 2 * z;
    const T *p = es + 3 * ((9 * k + j) * (long)a.ne + x + (long)a.mx * (y + (long)a.my * z)) + i;
#pragma unroll
    for (int l = 0; l < 3; l++) v[s][l] = p[9 * l * (long)a.ne];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int l = 0; l < 3; l++) {
    sum[l] = v[0][l];
#pragma unroll
    for (int s = 1; s < 8; s++) sum[l] += v[s][l];
  }
}

// node n of y from the element sums, Dirichlet rows y = x
constexpr int kColSumThreads = 256;
template <typename T>
__device__ __forceinline__ void col_node(const ColArgs &a, unsigned n, const T *__restrict__ es, T *__restrict__ y,
                                         const uint8_t *__restrict__ bcn, const T *__restrict__ x) {
  const unsigned X = 2 * a.mx + 1, Y = 2 * a.my + 1;
  const unsigned r = n / X, I = n - r * X, K = r / Y, J = r - K * Y;
  if (K > 2 * a.mz) return;
  T sum[3];
  col_sum<T>(a, I, J, K, es, sum);
  const unsigned m = bcn[n];
#pragma unroll
  for (int l = 0; l < 3; l++) y[3 * (long)n + l] = ((m >> l) & 1u) ? x[3 * (long)n + l] : sum[l];
}

template <typename T>
__global__ void __launch_bounds__(kColSumThreads)
    col_sum_kernel(ColArgs a, const T *__restrict__ es, T *__restrict__ y, const uint8_t *__restrict__ bcn,
                   const T *__restrict__ x) {
  col_node<T>(a, (unsigned)xcd_tile(blockIdx.x, gridDim.x) * kColSumThreads + threadIdx.x, es, y, bcn, x);
}

// the same with a RowUpdate of the row
template <typename T, UpdateKind kUp>
__global__ void __launch_bounds__(kColSumThreads)
    col_update_kernel(ColArgs a, const T *__restrict__ es, const uint8_t *__restrict__ bcn, const T *__restrict__ x,
                      RowUpdate<T> up) {
  const unsigned n = (unsigned)xcd_tile(blockIdx.x, gridDim.x) * kColSumThreads + threadIdx.x;
  const unsigned X = 2 * a.mx + 1, Y = 2 * a.my + 1;
  const unsigned r = n / X, I = n - r * X, K = r / Y, J = r - K * Y;
  if (K > 2 * a.mz) return;
  UpdateRow<T, kUp> u[3];
#pragma unroll
  for (int l = 0; l < 3; l++) u[l].load(up, 3 * (long)n + l, x, bcn[n]);
  T sum[3];
  col_sum<T>(a, I, J, K, es, sum);
#pragma unroll
  for (int l = 0; l < 3; l++) u[l].store(up, 3 * (long)n + l, l, sum[l]);
}
