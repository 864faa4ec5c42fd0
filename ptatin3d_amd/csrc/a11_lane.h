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
// SIMD that the registers allow.  FP64: 256 VGPRs + 168 AGPRs, about 4,200
// vector instructions per layer of which 3,050 are FP64 arithmetic, VALU busy
// 57 % of the wave's cycles, waiting 20 %.  64^3, MI355X: 54 us in FP64 (tile
// kernel 175 us), 32 us in FP32 (77 us).  The loads are the delicate part: a value that
// is still in flight when the registers run short is waited for at once, to
// be moved to an accumulation register or to scratch, one round trip each (the
// same kernel with its loads in flight across the stress stage took 130 us,
// with 40 scratch moves 156 us).  So every load is issued before a forward
// stage and used up at its end, where few registers are live.
//
// The saddle-point product runs the same way: the couplings add some 10
// instructions a point, the pressure basis being that of the unit cube, and 38
// AGPRs (96 x 96 x 48 MatMult 143 us, the tile kernel's 485 us before its face
// pass became faster; 28^3 33 and 56 us, 48^3 53 and 145 us).

// Per-lane constants of a rectilinear element: the collocation coefficients of
// the in-plane directions scaled by 2 m / h, and the weights.  m is a power of two
// of about an element's length, one for the mesh: derivatives in space times m
// are about those in the element, and the weights hold the lengths they lack, so
// that no product on the way is larger than the terms of the result but for the
// ratios of the lengths (with weights of det J, eta h^3 overflows FP32 at 3e39: SI
// units, 100 km elements).  A power of two changes no rounding.
template <typename T>
struct LaneGeom {
  T cx[3], cy[3];  // (5/2, 10/3, 5/6) s times 2 m / hx, 2 m / hy
  T az;            // 2 m / hz
  T vol;           // det J / m^2
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
    y0 -= c[2] * v;
    y2 += c[2] * v;
  } else {
    y0 += c[2] * v;
    y1 -= c[1] * v;
    y2 += c[0] * v;
  }
}

// Stress at the plane's points and its transposed derivatives:
// out[k][l][3j+i] += the plane's part of (A11_e u)(node (i, j, k), component l)
// kP: of the saddle-point product.  The pressure basis of a rectilinear element
// is {1, xi / 2, eta / 2, zeta / 2}; pc: its coefficients times m, the last three
// times s / 2 too; acc += the plane's part of (A21_e u), over the same factors.
template <typename T, int c, bool kP>
__device__ __forceinline__ void lane_stress(const T U[3][9], T Z[3][9], const LaneGeom<T> &g, const T et[9],
                                            T out[3][3][9], const T pc[4], T acc[4]) {
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
      T G[3][3];  // G[k][l] = m d u_l / d x_k
#pragma unroll
      for (int l = 0; l < 3; l++) {
        G[0][l] = ldot<T>(a, g.cx, U[l][3 * b], U[l][3 * b + 1], U[l][3 * b + 2]);
        G[1][l] = ldot<T>(b, g.cy, U[l][a], U[l][3 + a], U[l][6 + a]);
        G[2][l] = Z[l][p];
      }
      const T wv = (T)(kW[a] * kW[b] * kW[c]) * g.vol, t = et[p] * wv, t2 = t + t;
      T sg[3][3];
      if constexpr (kP) {
        T pq = pc[0];
        if (a != 1) pq += a == 0 ? -pc[1] : pc[1];
        if (b != 1) pq += b == 0 ? -pc[2] : pc[2];
        if (c != 1) pq += c == 0 ? -pc[3] : pc[3];
        const T wp = wv * pq, wd = wv * (G[0][0] + G[1][1] + G[2][2]);
        acc[0] -= wd;
        if (a != 1) acc[1] += a == 0 ? wd : -wd;
        if (b != 1) acc[2] += b == 0 ? wd : -wd;
        if (c != 1) acc[3] += c == 0 ? wd : -wd;
#pragma unroll
        for (int i = 0; i < 4; i++) asm volatile("" : "+v"(acc[i]));
        sg[0][0] = t2 * G[0][0] - wp;
        sg[1][1] = t2 * G[1][1] - wp;
        sg[2][2] = t2 * G[2][2] - wp;
      } else {
        sg[0][0] = t2 * G[0][0];
        sg[1][1] = t2 * G[1][1];
        sg[2][2] = t2 * G[2][2];
      }
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
  for (int l = 0; l < 3; l++)
    lane_field_t<T, c>(W[l], Z[l], d0, d1, d2, out[0][l], out[1][l], out[2][l]);
}

// Dirichlet rows are left as the element sums.  bcw: lane_bc_word's.  ax: 2 m / h
// of the mx element columns, the my rows and the mz layers, then m.
// kP: the saddle-point product with p, yp the pressures (4 per element).
template <typename T, bool kP>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 2 : 1)))
    a11_lane_kernel(TileArgs a, const T *__restrict__ ax, const T *__restrict__ eta,
                    const unsigned *__restrict__ bcw, const T *__restrict__ u, const T *__restrict__ p,
                    T *__restrict__ y, T *__restrict__ yp, T *__restrict__ fbx,
                    T *__restrict__ fby, T *__restrict__ fbz) {
  // five plane slots: the layer's three planes and the next layer's two
  __shared__ T sm[5 * kLSlot];
  const LaneTile q = lane_tile(a, (unsigned)xcd_tile(blockIdx.x, a.ntiles));
  const TileBox &tb = q.tb;
  // 2 m / hz of the chunk's layers, one per lane
  const T szs = ax[a.mx + a.my + tb.z0 + min(q.lane, tb.nzt - 1)];
  auto plane = [&](int P) { return LaneBuf<T>(u + 3 * lane_node(a, tb, P)); };

  LaneGeom<T> g;
  const T sx = ax[tb.x0 + q.cx], sy = ax[a.mx + tb.y0 + q.cy], m = ax[a.mx + a.my + a.mz];
  g.cx[0] = (T)(2.5 * kS) * sx;
  g.cx[1] = (T)(10.0 / 3.0 * kS) * sx;
  g.cx[2] = (T)(5.0 / 6.0 * kS) * sx;
  g.cy[0] = (T)(2.5 * kS) * sy;
  g.cy[1] = (T)(10.0 / 3.0 * kS) * sy;
  g.cy[2] = (T)(5.0 / 6.0 * kS) * sy;

  {
    const LaneBuf<T> v0 = plane(2 * tb.z0), v1 = plane(2 * tb.z0 + 1), v2 = plane(2 * tb.z0 + 2);
    T r0[kLBatch], r1[kLBatch], r2[kLBatch];
    const unsigned m0 = lane_bc_word(a, q, bcw, 2 * tb.z0), m1 = lane_bc_word(a, q, bcw, 2 * tb.z0 + 1),
                   m2 = lane_bc_word(a, q, bcw, 2 * tb.z0 + 2);
    lane_rows_load<T, 0>(r0, q, a.X, v0, v1);
    lane_rows_load<T, 1>(r1, q, a.X, v0, v1);
    lane_rows_mask<T, 0>(r0, m0, m1);
    lane_rows_store<T, 0>(r0, q, sm, sm + kLSlot);
    lane_rows_load<T, 2>(r2, q, a.X, v0, v1);
    lane_rows_mask<T, 1>(r1, m0, m1);
    lane_rows_store<T, 1>(r1, q, sm, sm + kLSlot);
    lane_rows_load<T, 0, kLRows>(r0, q, a.X, v2, v2);
    lane_rows_load<T, 1, kLRows>(r1, q, a.X, v2, v2);
    lane_rows_mask<T, 2>(r2, m0, m1);
    lane_rows_store<T, 2>(r2, q, sm, sm + kLSlot);
    lane_rows_mask<T, 0, kLRows>(r0, m2, 0u);
    lane_rows_store<T, 0, kLRows>(r0, q, sm + 2 * kLSlot, nullptr);
    lane_rows_mask<T, 1, kLRows>(r1, m2, 0u);
    lane_rows_store<T, 1, kLRows>(r1, q, sm + 2 * kLSlot, nullptr);
  }
  T out[3][3][9];
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int n = 0; n < 9; n++) out[2][l][n] = T(0);

  const unsigned oe = (unsigned)sizeof(T) * (q.cx + (unsigned)a.mx * q.cy);
  const unsigned qs = (unsigned)sizeof(T) * (unsigned)a.nel;
  int slot = 0;  // of plane 2 ek; its successors follow modulo 5
  for (int kz = 0; kz < tb.nzt; kz++) {
    const int ek = tb.z0 + kz;
    auto place = [&](int k) { return sm + kLSlot * (slot + k >= 5 ? slot + k - 5 : slot + k); };
    T *const s0 = place(0), *const s1 = place(1), *const s2 = place(2), *const s3 = place(3), *const s4 = place(4);
    // (the last layer of the chunk loads its own planes again, into free slots)
    const int nn = kz + 1 < tb.nzt ? 2 * ek + 3 : 2 * ek + 1;
    const LaneBuf<T> v1 = plane(nn), v2 = plane(nn + 1);
    const LaneBuf<T> eta_k(eta + tb.x0 + (long)a.mx * (tb.y0 + (long)a.my * ek));
    const T sz = __shfl(szs, kz);
    g.az = sz;
    g.vol = q.live ? m * (T(1) / (sx * sy * sz)) : T(0);
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
    T et[9], r[kLBatch], U[3][9], Z[3][9], pc[4], acc[4] = {T(0), T(0), T(0), T(0)};
    const long e4 = 4 * (tb.x0 + (long)a.mx * (tb.y0 + (long)a.my * ek)) + 4 * (q.cx + a.mx * q.cy);
    if constexpr (kP) {
#pragma unroll
      for (int i = 0; i < 4; i++) pc[i] = p[e4 + i];
    }
    int lq = q.li;
    auto forward = [&](auto c) {
      constexpr int C = decltype(c)::value;
      const T d0 = (T)kD[C][0] * g.az, d1 = (T)kD[C][1] * g.az, d2 = (T)kD[C][2] * g.az;
#pragma unroll
      for (int f = 0; f < 3; f++)
        lane_field<T, C>(s0 + lq + f * kLPlane, s1 + lq + f * kLPlane, s2 + lq + f * kLPlane, d0, d1, d2, U[f], Z[f]);
    };
#pragma unroll
    for (int p = 0; p < 9; p++) et[p] = eta_k.load(oe, qs * p);
    const unsigned m3 = lane_bc_word(a, q, bcw, nn), m4 = lane_bc_word(a, q, bcw, nn + 1);
    lane_rows_load<T, 0>(r, q, a.X, v1, v2);
    forward(std::integral_constant<int, 0>());
    lane_rows_mask<T, 0>(r, m3, m4);
    lane_rows_store<T, 0>(r, q, s3, s4);
    if constexpr (kP) {
#pragma unroll
      for (int i = 0; i < 4; i++) pc[i] *= i ? (T)(0.5 * kS) * m : m;
    }
    lane_stress<T, 0, kP>(U, Z, g, et, out, pc, acc);
    lane_pin<T>(out);
    // the node values are read again per quadrature plane, not held: an
    // index the compiler knows nothing about keeps it from merging the reads
    asm volatile("" : "+v"(lq));
#pragma unroll
    for (int p = 0; p < 9; p++) et[p] = eta_k.load(oe, qs * (9 + p));
    lane_rows_load<T, 1>(r, q, a.X, v1, v2);
    forward(std::integral_constant<int, 1>());
    lane_rows_mask<T, 1>(r, m3, m4);
    lane_rows_store<T, 1>(r, q, s3, s4);
    lane_stress<T, 1, kP>(U, Z, g, et, out, pc, acc);
    lane_pin<T>(out);
    asm volatile("" : "+v"(lq));
#pragma unroll
    for (int p = 0; p < 9; p++) et[p] = eta_k.load(oe, qs * (18 + p));
    lane_rows_load<T, 2>(r, q, a.X, v1, v2);
    forward(std::integral_constant<int, 2>());
    lane_rows_mask<T, 2>(r, m3, m4);
    lane_rows_store<T, 2>(r, q, s3, s4);
    lane_stress<T, 2, kP>(U, Z, g, et, out, pc, acc);
    lane_pin<T>(out);
    if constexpr (kP) {
      if (q.live) {
#pragma unroll
        for (int i = 0; i < 4; i++) yp[e4 + i] = (i ? (T)(0.5 * kS) * m : m) * acc[i];
      }
    }
    __syncthreads();
    // the planes 2 ek and 2 ek + 1 are complete: their slots become windows
    lane_window<T>(s0 + q.lw, q.moreX, q.moreY, out[0]);
    lane_window<T>(s1 + q.lw, q.moreX, q.moreY, out[1]);
    __syncthreads();
    lane_flush<T, kLaneSums, false>(a, q, 2 * ek, s0, 0u, y, fbx, fby, fbz);
    lane_flush<T, kLaneSums, false>(a, q, 2 * ek + 1, s1, 0u, y, fbx, fby, fbz);
    __syncthreads();
    slot = slot + 2 >= 5 ? slot - 3 : slot + 2;
  }
  T *const top = sm + kLSlot * slot;
  lane_window<T>(top + q.lw, q.moreX, q.moreY, out[2]);
  __syncthreads();
  lane_flush<T, kLaneSums, true>(a, q, 2 * (tb.z0 + tb.nzt), top, 0u, y, fbx, fby, fbz);
}
