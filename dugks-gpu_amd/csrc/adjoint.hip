// Discrete adjoint of one DUGKS step (no counterpart in the reference).
//
// Forward stages of a step (src/dugks.cu:322-391 of the reference):
//   S1 centre    fb_c = bw1 f_c + (bw2 + bw0 T_i) feq_i(rho, u), u = j/rho + h F_c
//   S2 ghosts    periodic copy / wall extrapolation (linear)
//   S3 faces     trilinear reconstruction of fb (linear) + wall bounce-back
//   S4 collide   ft = fw1 fbar + (fw2 + fw0 T'_i) feq_i(rho_f, u_f), u_f = j_f/rho_f + (h/2) F
//   S5 update    f' = 4/3 fb_c - 1/3 f_c - sum_a (dt/dx_a) c_a (ft_a+ - ft_a-)
// Given lam' = dJ/df', the adjoint returns lam = (df'/df)^T lam' and
// accumulates dJ/dF_c.  Work split:
//   1. f-bar+ with ghosts is recomputed (the two-pass kernels);
//   2. k_adj_faces: every face once: S3 forward, S4^T driven by the face's
//      cotangent lam_ft_q = c_qa (dt/dx_R lam'_q(R) - dt/dx_L lam'_q(L)) of
//      its crossing populations.  The collision cotangent of every population
//      is lam_fbar_q = fw1 lam_ft_q + A + B.c_q; after the transpose of the
//      wall bounce-back the face stores the cotangent of its 19
//      reconstructed values (in the arithmetic type);
//   3. the gather: S3^T of those values over the faces whose stencil
//      contains each cell (the wall ghost extrapolation folded in), then S5^T
//      and S1^T.  k_adj_cells_z
//      stages each plane of face cotangents in LDS and marches along z (its
//      faces come from the fused pass as records of A and B alone, and it
//      forms lam_ft from lam' itself);
//      k_adj_cells (every other case) runs one thread per cell over face
//      arrays with periodic ghost copies (k_face_ghosts).
// Deterministic (no atomics).  At most one wall axis.
#include "device_common.h"

namespace dugks {

namespace {

#include "fused_common.h"

__device__ __forceinline__ long long ext_index(const KParams& P, int m0, int m1, int m2) {
  return ((long long)m2 * P.e[1] + m1) * P.e[0] + m0;
}

// Wrap a ghost-inclusive index of a periodic axis into 1..n.
__device__ __forceinline__ int wrap(const KParams& P, int a, int m) {
  if (!P.periodic[a]) return m;
  const int n = P.n[a];
  return m < 1 ? m + n : (m > n ? m - n : m);
}

// lam' of population ip at a ghost-inclusive position (0 outside the domain).
__device__ __forceinline__ double lam_at(const KParams& P, const double* lam, int ip, int m0, int m1, int m2) {
  int m[3] = {wrap(P, 0, m0), wrap(P, 1, m1), wrap(P, 2, m2)};
  for (int a = 0; a < 3; a++)
    if (m[a] < 1 || m[a] > P.n[a]) return 0.0;
  const long long c = ((long long)(m[2] - 1) * P.n[1] + (m[1] - 1)) * P.n[0] + (m[0] - 1);
  return lam[ip * P.N + c];
}

// ---- kernel 2: one thread per face of axis A ----
template <class Real, int A>
__global__ void __launch_bounds__(256) k_adj_faces(KParams P, const Real* __restrict__ fbx,
                                                   const double* __restrict__ lam, Real* __restrict__ faces) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= P.eN) return;
  int m[3];
  m[0] = (int)(e % P.e[0]);
  m[1] = (int)((e / P.e[0]) % P.e[1]);
  m[2] = (int)(e / ((long long)P.e[0] * P.e[1]));
  for (int b = 0; b < 3; b++) {
    if (b == A) continue;
    if (m[b] < 1 || m[b] > P.n[b]) return;
  }
  const int nA = P.n[A];
  if (P.periodic[A] ? (m[A] < 1 || m[A] > nA) : (m[A] < 0 || m[A] > nA)) return;
  const long long st[3] = {1, P.e[0], (long long)P.e[0] * P.e[1]};
  const double* tab = P.tab[A] + m[A] * 9;
  // S3: reconstruction as the +A face of the left cell
  Real ft[Q];
  ft[0] = Real(0.5) * (fbx[e] + fbx[e + st[A]]);
  static_for<Q - 1>([&](auto I) {
    constexpr int ip = decltype(I)::value + 1;
    constexpr int c[3] = {CX[ip], CY[ip], CZ[ip]};
    const Real* p = fbx + ip * P.eN + e;
    long long off[3];
    Real w[3];
#pragma unroll
    for (int b = 0; b < 3; b++) {
      if (b == A) {
        off[b] = st[b];
        w[b] = (Real)tab[c[b] + 1];
      } else {
        off[b] = -c[b] * st[b];
        w[b] = c[b] == 0 ? Real(0) : (Real)P.tab[b][m[b] * 9 + (c[b] < 0 ? 6 : 7)];
      }
    }
    Real r = 0;
#pragma unroll
    for (int corner = 0; corner < 8; corner++) {
      const int bx = corner & 1, by = (corner >> 1) & 1, bz = (corner >> 2) & 1;
      const Real wt = (bx ? w[0] : Real(1) - w[0]) * (by ? w[1] : Real(1) - w[1]) * (bz ? w[2] : Real(1) - w[2]);
      if (wt != Real(0)) r += wt * p[bx * off[0] + by * off[1] + bz * off[2]];
    }
    ft[ip] = r;
  });
  // wall bounce-back (src/dugks.cu:807-823)
  const bool low = !P.periodic[A] && m[A] == 0, high = !P.periodic[A] && m[A] == nA;
  if (low || high) {
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      if constexpr (cv(A, ip) != 0) {
        if ((low && cv(A, ip) > 0) || (high && cv(A, ip) < 0)) ft[ip] = ft[OPP[ip]];
      }
    });
  }
  Real rho = 0, j[3] = {0, 0, 0};
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    rho += ft[ip];
    j[0] += Real(CX[ip]) * ft[ip];
    j[1] += Real(CY[ip]) * ft[ip];
    j[2] += Real(CZ[ip]) * ft[ip];
  });
  Real F[3], u[3], ut[3];
  for (int a = 0; a < 3; a++) {
    F[a] = (Real)P.famb_dev[a];
    ut[a] = j[a] / rho;
    u[a] = ut[a] + Real(0.5) * (Real)P.hdt * F[a];
  }
  // cotangent of the crossing populations (S5^T)
  int mR[3] = {m[0], m[1], m[2]};
  mR[A] += 1;
  const Real updL = (Real)tab[8], updR = (Real)P.tab[A][(m[A] + 1) * 9 + 8];
  Real lft[Q];
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    if constexpr (cv(A, ip) != 0) {
      const Real lL = (Real)lam_at(P, lam, ip, m[0], m[1], m[2]);
      const Real lR = (Real)lam_at(P, lam, ip, mR[0], mR[1], mR[2]);
      lft[ip] = Real(cv(A, ip)) * (updR * lR - updL * lL);
    } else {
      lft[ip] = 0;
    }
  });
  Real g_rho, g_u[3], g_F[3];
  feq_adjoint<Real>(lft, (Real)P.fw2, (Real)P.fw0, rho, u, F, g_rho, g_u, g_F, Crossing<A>{});
  const Real invr = Real(1) / rho;
  const Real Acoef = g_rho - (g_u[0] * ut[0] + g_u[1] * ut[1] + g_u[2] * ut[2]) * invr;
  const Real Bx = g_u[0] * invr, By = g_u[1] * invr, Bz = g_u[2] * invr;
  // collision cotangent of each (post-bounce) face value
  Real lpost[Q];
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    lpost[ip] = (Real)P.fw1 * lft[ip] + Acoef + Bx * Real(CX[ip]) + By * Real(CY[ip]) + Bz * Real(CZ[ip]);
  });
  // transpose of the bounce-back: an incoming population took its
  // opposite's reconstructed value
  Real* out = faces + (long long)A * Q * P.eN + e;
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    Real v = lpost[ip];
    if constexpr (cv(A, ip) != 0) {
      if (low || high) {
        const bool in = (low && cv(A, ip) > 0) || (high && cv(A, ip) < 0);
        v = in ? Real(0) : v + lpost[OPP[ip]];
      }
    }
    out[(long long)ip * P.eN] = v;
  });
}

// Face-slot index of a periodic axis' ghost position in the weight table
// (the table rows of ghost positions are only used for wall axes).
__device__ __forceinline__ int table_slot(const KParams& P, int a, int m) {
  if (!P.periodic[a]) return m;
  return m == 0 ? P.n[a] : (m == P.n[a] + 1 ? 1 : m);
}

// S3^T at ghost-inclusive position t (linear index et) for population ip: the
// sum over the faces of axis A whose reconstruction stencil contains t of
// the face cotangent times the stencil weight.  Face arrays hold periodic
// ghost copies (k_face_ghosts) and zeros at the ghost rows of wall axes, so
// every stencil face of an interior position is a plain offset from et.  A
// wall ghost position (GHOST) can reach outside the array and is checked.
template <class Real, int A, int ip, bool GHOST>
__device__ __forceinline__ Real gather_axis(const KParams& P, const Real* faces, const int t[3], long long et) {
  constexpr int c[3] = {CX[ip], CY[ip], CZ[ip]};
  constexpr int B1 = (A + 1) % 3, B2 = (A + 2) % 3;
  const long long st[3] = {1, P.e[0], (long long)P.e[0] * P.e[1]};
  const Real* fa = faces + ((long long)A * Q + ip) * P.eN + et;
  Real acc = 0;
  // normal: t is the left cell of the face in slot t_A, the right cell of slot t_A - 1
#pragma unroll
  for (int side = 0; side < 2; side++) {
    const int sl = t[A] - side;
    if (GHOST && (sl < 0 || sl > P.n[A])) continue;
    Real wn;
    if constexpr (ip == 0) {
      wn = Real(0.5);
    } else {
      const Real wR = tabv<Real>(P, A, table_slot(P, A, sl) * 9 + c[A] + 1);  // toward the right cell
      wn = side == 0 ? Real(1) - wR : wR;
    }
#pragma unroll
    for (int s1 = 0; s1 < 2; s1++) {
      if (s1 == 1 && (c[B1] == 0 || ip == 0)) continue;
      const int f1 = t[B1] + s1 * c[B1];
      if (GHOST && (f1 < 0 || f1 > P.n[B1] + 1)) continue;
      Real w1 = 1;
      if (c[B1] != 0 && ip != 0) {
        const Real m = tabv<Real>(P, B1, table_slot(P, B1, f1) * 9 + (c[B1] < 0 ? 6 : 7));
        w1 = s1 ? m : Real(1) - m;
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; s2++) {
        if (s2 == 1 && (c[B2] == 0 || ip == 0)) continue;
        const int f2 = t[B2] + s2 * c[B2];
        if (GHOST && (f2 < 0 || f2 > P.n[B2] + 1)) continue;
        Real w2 = 1;
        if (c[B2] != 0 && ip != 0) {
          const Real m = tabv<Real>(P, B2, table_slot(P, B2, f2) * 9 + (c[B2] < 0 ? 6 : 7));
          w2 = s2 ? m : Real(1) - m;
        }
        const long long off = -side * st[A] + s1 * c[B1] * st[B1] + s2 * c[B2] * st[B2];
        acc += wn * w1 * w2 * fa[off];
      }
    }
  }
  return acc;
}

template <class Real, int ip, bool GHOST>
__device__ __forceinline__ Real gather(const KParams& P, const Real* faces, const int t[3]) {
  const long long et = ext_index(P, t[0], t[1], t[2]);
  return gather_axis<Real, 0, ip, GHOST>(P, faces, t, et) + gather_axis<Real, 1, ip, GHOST>(P, faces, t, et) +
         gather_axis<Real, 2, ip, GHOST>(P, faces, t, et);
}

// Periodic ghost copies of the face arrays along axis b (slot 0 <- n,
// n+1 <- 1), for all three face axes and 19 populations; axes in the order
// x, y, z so that edges and corners are consistent.
template <class Real>
__global__ void __launch_bounds__(256) k_face_ghosts(KParams P, Real* __restrict__ faces, int b) {
  const int b1 = (b + 1) % 3, b2 = (b + 2) % 3;
  const long long plane = (long long)P.e[b1] * P.e[b2];
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= plane * 3 * Q) return;
  const long long arr = id / plane, pos = id % plane;
  int m[3];
  m[b1] = (int)(pos % P.e[b1]);
  m[b2] = (int)(pos / P.e[b1]);
  Real* fa = faces + arr * P.eN;
  const int n = P.n[b];
  m[b] = n;
  const Real vn = fa[ext_index(P, m[0], m[1], m[2])];
  m[b] = 1;
  const Real v1 = fa[ext_index(P, m[0], m[1], m[2])];
  m[b] = 0;
  fa[ext_index(P, m[0], m[1], m[2])] = vn;
  m[b] = n + 1;
  fa[ext_index(P, m[0], m[1], m[2])] = v1;
}

// ---- kernel 3: one thread per interior cell ----
constexpr int kCX = 32, kCY = 8, kCZ = 1;  // cell tile of a 256-thread block
template <class Real, class Store>
__global__ void __launch_bounds__(256) k_adj_cells(KParams P, const Store* __restrict__ f,
                                                   const double* __restrict__ lam, const Real* __restrict__ faces,
                                                   double* __restrict__ lam_prev, double* __restrict__ grad,
                                                   int wall_axis) {
  // kCX x kCY x kCZ cell tiles, dealt to the XCDs in contiguous runs of
  // tiles (x fastest) so that neighbouring tiles share an L2: each face
  // value is gathered by cells of up to eight tiles
  const int gx = (P.n[0] + kCX - 1) / kCX, gy = (P.n[1] + kCY - 1) / kCY, gz = (P.n[2] + kCZ - 1) / kCZ;
  const int ntiles = gx * gy * gz;
  const int b = blockIdx.x;
  const int tt = (ntiles % 8 == 0) ? (b % 8) * (ntiles / 8) + b / 8 : b;
  const int ci = (tt % gx) * kCX + (int)threadIdx.x % kCX;
  const int cj = ((tt / gx) % gy) * kCY + ((int)threadIdx.x / kCX) % kCY;
  const int ck = (tt / (gx * gy)) * kCZ + (int)threadIdx.x / (kCX * kCY);
  if (ci >= P.n[0] || cj >= P.n[1] || ck >= P.n[2]) return;
  const long long c = ((long long)ck * P.n[1] + cj) * P.n[0] + ci;
  const int t[3] = {ci + 1, cj + 1, ck + 1};
  Real lfb[Q];
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    Real v = Real(4.0 / 3.0) * (Real)lam[ip * P.N + c] + gather<Real, ip, false>(P, faces, t);
    if (wall_axis >= 0) {
      // S2^T: the wall ghost g = q f(1) + (1-q) f(2) (and mirrored at the top)
      const int W = wall_axis, n = P.n[W];
      int g[3] = {t[0], t[1], t[2]};
      if (t[W] == 1 || t[W] == 2) {
        g[W] = 0;
        const Real q = (Real)P.qlo[W];
        v += (t[W] == 1 ? q : Real(1) - q) * gather<Real, ip, true>(P, faces, g);
      }
      if (t[W] == n || t[W] == n - 1) {
        g[W] = n + 1;
        const Real q = (Real)P.qhi[W];
        v += (t[W] == n ? q : Real(1) - q) * gather<Real, ip, true>(P, faces, g);
      }
    }
    lfb[ip] = v;
  });
  // S1^T
  Real ff[Q];
  load_cell<Real, Store>(f, c, P, ff);
  Real rho = 0, j[3] = {0, 0, 0};
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    rho += ff[ip];
    j[0] += Real(CX[ip]) * ff[ip];
    j[1] += Real(CY[ip]) * ff[ip];
    j[2] += Real(CZ[ip]) * ff[ip];
  });
  Real F[3], u[3], ut[3];
  for (int a = 0; a < 3; a++) {
    F[a] = (Real)P.famb_dev[a];
    if (P.fcell) F[a] += (Real)P.fcell[a * P.N + c];
    ut[a] = j[a] / rho;
    u[a] = ut[a] + (Real)P.hdt * F[a];
  }
  Real g_rho, g_u[3], g_F[3];
  feq_adjoint<Real>(lfb, (Real)P.bw2, (Real)P.bw0, rho, u, F, g_rho, g_u, g_F, AllPops{});
  const Real invr = Real(1) / rho;
  const Real Acoef = g_rho - (g_u[0] * ut[0] + g_u[1] * ut[1] + g_u[2] * ut[2]) * invr;
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    const Real v = -(Real)lam[ip * P.N + c] * Real(1.0 / 3.0) + (Real)P.bw1 * lfb[ip] + Acoef +
                   (g_u[0] * Real(CX[ip]) + g_u[1] * Real(CY[ip]) + g_u[2] * Real(CZ[ip])) * invr;
    lam_prev[ip * P.N + c] = (double)v;
  });
  if (grad) {
    for (int a = 0; a < 3; a++) grad[a * P.N + c] += (double)(g_F[a] + (Real)P.hdt * g_u[a]);
  }
}

// ---- kernel 3, z-marching form ----
// A workgroup owns a tile of cell columns (32 x 12 with FP32 arithmetic, 16 x
// 12 with FP64) and marches along z over a chunk of planes.  A lane stages one
// position of the tile or of its one-deep ring (periodic indices wrapped, so no
// ghost copies are needed).  Per plane p:
//   - lam'(p) of every position goes to LDS;
//   - each position's x- and y-face of plane p and z-face p-1/2 are expanded to
//     their 19 reconstructed-value cotangents in LDS, from the face's record
//     (Ac, B) and the lam' on both of its sides;
//   - each cell gathers its transposed in-plane lerps from LDS.  The transposed
//     z-lerps are pushed into the f-bar+ cotangents of planes p-1, p and p+1
//     held in registers: the x- and y-faces of plane p (z-lerped toward p - c_z
//     in the step) and the z-face p-1/2 (normal lerp between p-1 and p).  Plane
//     p-1 is then complete and goes through the centre stage's adjoint.
// Wall ghosts are folded at the in-plane level: a cell beside a wall adds q (or
// 1 - q) times the in-plane gather at the ghost position, which takes the same
// z transposes as its own.  The centre stage needs only rho and j of the state:
// with the state stored in the arithmetic type it reads them from the face pass
// (16 or 32 bytes a cell) rather than the 19 values of f.
//
// What bounds it: issue in FP32 (two waves per SIMD, VALU 61 % busy, 1795
// lane-instructions a cell; 3.4 GB of HBM traffic on 256x192x256 at 3.7 TB/s, where
// a large copy runs at 4.9) and latency in FP64 (a column's registers leave one
// wave per SIMD, VALU 30 % busy).  A cell reads lam' (19 values), three face
// records (4 each, in one 16-byte access with FP32) and rho, j, and writes lam; the
// records held the ten crossing values as well (13 each) before, so that the two
// passes moved 174 values a cell, now 120.  The next plane's loads go out during the
// gather, a plane ahead of their use, without branches (accesses that are not
// wanted go out of range), so that every wait counts exactly.  Ring lanes run
// the gather and the centre stage on clamped positions and store nothing: they
// share SIMDs with one wave of cells where the others hold two.  The FP64 form
// without FLOW and the 8-row FP16 form with FP64 lam spill two and seven registers.
// 256x192x256 FP32: 0.94 ms, before 1.23 (the face pass beside it 0.84, before 1.41).
// lanes of a workgroup, and LDS positions (the last ones idle)
constexpr int gather_lanes(bool fp64, int rows) { return ((rows + 2) * (fp64 ? 18 : 34) + 63) / 64 * 64; }
template <class Real, int ROWS>
struct GatherTile {
  static constexpr int TX = sizeof(Real) == 8 ? 16 : 32, TY = ROWS;
  static constexpr int AC = TX + 2, NP = (TY + 2) * AC;
  static constexpr int NT = gather_lanes(sizeof(Real) == 8, ROWS);
  static_assert(NT > NP, "an idle position, whose face cotangents are zeros");
};

// mom: the region of rho, j behind the face records that holds fin's
// (storage in the arithmetic type).  FLOW (such storage, with FP32 lam and
// arithmetic or FP64 throughout; a sweep through the flow-rate
// controller): lam' still lacks the bulk velocity's cotangent ubar (dV/V)
// (c_ia - u_a)/rho of f(n+1), whose rho, j the previous pass left in the
// other region; it is added as lam' is used.
// PLANES 1 or 2: the grid has that many planes, in one chunk, and each is taken
// once: on one plane p-1, p and p+1 are the same, on two p-1 and p+1 are, so that
// what a plane gives to either goes to the other one.  (PLANES 0 takes the two
// planes beside a chunk too.  FP32 with FP64 lam, us an adjoint step: 512x768x1 98,
// with the same plane taken three times 144; 64x64x1 18 and 29.  FP64, 192x288x2
// with walls 90 and 105, 512x256x2 143 and 158.  With FP32 arithmetic the two-plane
// form spills 34 to 96 registers and was slower, 100 and 89 us on 512x256x2.)
template <class Real, class Store, class Lam, int ROWS, bool FLOW, int PLANES>
__global__ void __launch_bounds__(gather_lanes(sizeof(Real) == 8, ROWS), sizeof(Real) == 4 ? 2 : 1)
    k_adj_cells_z(KParams P, const Store* __restrict__ fin, const Lam* __restrict__ lam,
                  const Real* __restrict__ faces, Lam* __restrict__ lam_prev, double* __restrict__ grad, int nchunk,
                  int mom, const double* __restrict__ ubar, double inv_vol) {
  using T = GatherTile<Real, ROWS>;
  constexpr int TX = T::TX, TY = T::TY, AC = T::AC, NT = T::NT;
  __shared__ Real S[3][Q][NT];   // face cotangents: x-faces and y-faces of plane p, z-faces p-1/2
  __shared__ Real L[Q][NT];      // lam'(p) (populations with c_x or c_y)
  __shared__ Real WXs[6][AC];    // per staged column: wR for c = -1, 0, +1, the shift weights, dt/dx
  __shared__ Real WYs[6][TY + 2];  // per staged row

  const int nx = P.n[0], ny = P.n[1], nz = P.n[2];
  const int t = threadIdx.x;
  // XCD-aware tile order (workgroup b runs on XCD b % 8)
  const int gxn = nx / TX, gyn = (ny + TY - 1) / TY;
  const int nblocks = gxn * gyn * nchunk, b = blockIdx.x, xcd = b % 8;
  const int tt = xcd * (nblocks / 8) + min(xcd, nblocks % 8) + b / 8;
  const int bx = tt % gxn, by = (tt / gxn) % gyn, bz = tt / (gxn * gyn);
  // the last row of tiles starts early where TY does not divide ny; its first
  // ry0 rows are the other tile's to store
  const int th = min(TY, ny);
  const int i0 = bx * TX, j0 = min(by * TY, ny - th), ry0 = by * TY - j0;
  const int z0 = (int)((long long)bz * nz / nchunk), zend = (int)((long long)(bz + 1) * nz / nchunk);
  const int ex = P.e[0], ey = P.e[1];

  // the lane's staged position (R, C), ghost-inclusive and tile-local: the
  // cells first, then the rows above and below, then the columns beside
  int R, C;
  if (t < TX * TY) {
    R = t / TX + 1;
    C = t % TX + 1;
  } else if (t < TX * TY + 2 * AC) {
    const int v = t - TX * TY;
    R = v < AC ? 0 : th + 1;
    C = v % AC;
  } else {
    const int v = t - TX * TY - 2 * AC;
    R = v % TY + 1;
    C = v < TY ? 0 : TX + 1;
  }
  const bool staged = t < T::NP && (R <= th || (R == th + 1 && t >= TX * TY));
  const bool cell_lane = staged && t < TX * TY;
  const int pos0 = staged ? R * AC + C : T::NP;  // the others: the idle position
  const bool stored = cell_lane && R > ry0;
  // where the lane gathers (cells: their own position)
  const int Rg0 = min(max(R, 1), th), Cg0 = min(max(C, 1), TX);

  // weights of the staged columns and rows (table_slot maps the periodic ghosts)
  for (int u = t; u < 6 * AC + 6 * (TY + 2); u += NT) {
    const bool isx = u < 6 * AC;
    const int v = isx ? u : u - 6 * AC;
    const int n = isx ? AC : TY + 2;
    const int k = v / n, q = v % n;
    const int a = isx ? 0 : 1;
    const int slot = table_slot(P, a, min((isx ? i0 : j0) + q, (isx ? nx : ny) + 1));
    const Real w = tabv<Real>(P, a, slot * 9 + (k < 3 ? k : k + 3));
    if (isx)
      WXs[k][q] = w;
    else
      WYs[k][q] = w;
  }
  // z is periodic and uniform
  const Real mz6 = tabv<Real>(P, 2, 9 + 6), mz7 = tabv<Real>(P, 2, 9 + 7), updz = tabv<Real>(P, 2, 9 + 8);
  const Real wRz[3] = {tabv<Real>(P, 2, 9 + 0), tabv<Real>(P, 2, 9 + 1), tabv<Real>(P, 2, 9 + 2)};

  Real Famb[3];
  Famb[0] = (Real)P.famb_dev[0];
  Famb[1] = (Real)P.famb_dev[1];
  Famb[2] = (Real)P.famb_dev[2];
  const Real hdt = (Real)P.hdt, bw0 = (Real)P.bw0, bw1 = (Real)P.bw1, bw2 = (Real)P.bw2, fw1 = (Real)P.fw1;

  // the staged position's face slot and cell, the faces it has, and which are at walls
  int x = i0 + C, y = j0 + R;
  const bool wlx = !P.periodic[0] && x == 0, whx = !P.periodic[0] && x == nx;
  const bool wly = !P.periodic[1] && y == 0, why = !P.periodic[1] && y == ny;
  if (P.periodic[0]) x = x == 0 ? nx : (x == nx + 1 ? 1 : x);
  if (P.periodic[1]) y = y == 0 ? ny : (y == ny + 1 ? 1 : y);
  const unsigned exy = (unsigned)y * (unsigned)ex + (unsigned)x;
  const bool has_cell = staged && x >= 1 && x <= nx && y >= 1 && y <= ny;
  const bool okx = staged && C <= TX, oky = staged && R <= th;
  const unsigned plane = (unsigned)nx * (unsigned)ny;
  const unsigned column = has_cell ? (unsigned)(y - 1) * (unsigned)nx + (unsigned)(x - 1) : 0u;

  const RawBuf recs[3] = {face_records<Real>(faces, 0, P.eN), face_records<Real>(faces, 1, P.eN),
                          face_records<Real>(faces, 2, P.eN)};
  const RawBuf lamb(lam, (unsigned)(Q * P.N * sizeof(Lam))), outb(lam_prev, (unsigned)(Q * P.N * sizeof(Lam)));
  const unsigned lam_pop = (unsigned)(P.N * sizeof(Lam));
  // the cell force and the gradient; absent ones read as 0 and take no stores
  const RawBuf fcb(P.fcell, P.fcell ? (unsigned)(3 * P.N * 8) : 0u), gradb(grad, grad ? (unsigned)(3 * P.N * 8) : 0u);
  const unsigned vec_pop = (unsigned)(P.N * 8);
  const StateBuf<Store> bin(fin, Q * (unsigned)(P.N * (long long)sizeof(Store)));
  constexpr bool kMoments = std::is_same<Store, Real>::value;
  const RawBuf mb = cell_records<Real>(faces, mom, P.eN, P.N);
  // FLOW: rho and j_a of f(n+1) at the staged cell, and s0 = ubar dV / V
  static_assert(!FLOW || kMoments, "the controller term needs the moments of f(n+1)");
  const RawBuf mbn = cell_records<Real>(faces, 1 - mom, P.eN, P.N);
  const int fa = P.flow_axis;
  Real s0 = Real(0), rn = Real(0), jn = Real(0);
  if constexpr (FLOW)
    if (has_cell) s0 = (Real)(ubar[0] * P.wd[0][x] * P.wd[1][y] * P.wd[2][1] * inv_vol);

  // lam' of planes p-1 and p at the staged position, and of p+1 as loaded; the
  // records of the position's faces
  Real lamP[Q], lamC[Q];
  Lam lraw[Q];
  Real rec[3][kCompact];
  auto load_lam = [&](auto A, auto B, int k, bool want) {
    const unsigned vb = want && has_cell ? ((unsigned)k * plane + column) * (unsigned)sizeof(Lam) : kOutOfRange;
    static_for<decltype(B)::value - decltype(A)::value>([&](auto I) {
      constexpr int ip = decltype(A)::value + decltype(I)::value;
      lraw[ip] = lamb.ld<Lam>(vb, ip * lam_pop);
    });
    if constexpr (FLOW && decltype(A)::value == 0) {
      const unsigned vm = want && has_cell ? ((unsigned)k * plane + column) * (unsigned)(4 * sizeof(Real)) : kOutOfRange;
      rn = mbn.ld<Real>(vm, 0);
      jn = mbn.ld<Real>(vm, (unsigned)(1 + fa) * (unsigned)sizeof(Real));
    }
  };
  // the x- and y-face records of plane k (0-based; z slot k + 1) and the z-face's of k - 1/2 (z slot kl + 1, kl = k - 1 wrapped)
  auto load_recs = [&](int k, bool want) {
    const int kl = k == 0 ? nz - 1 : k - 1;
    const unsigned ez = (unsigned)ey * (unsigned)ex, size = (unsigned)(kCompact * sizeof(Real));
    const unsigned v = ((unsigned)(k + 1) * ez + exy) * size, vz = ((unsigned)(kl + 1) * ez + exy) * size;
    recs[0].ld4(want && okx ? v : kOutOfRange, rec[0]);
    recs[1].ld4(want && oky ? v : kOutOfRange, rec[1]);
    recs[2].ld4(want && staged ? vz : kOutOfRange, rec[2]);
  };
  using I0 = std::integral_constant<int, 0>;
  using I10 = std::integral_constant<int, 10>;
  using IQ = std::integral_constant<int, Q>;
  auto wrap = [&](int k) { return k < 0 ? k + nz : (k >= nz ? k - nz : k); };

  // the 19 reconstructed-value cotangents of the lane's A-face into LDS, from mu
  auto expand = [&](auto AI, int pos, const Real (&mu)[10], bool ok, bool lo, bool hi) {
    constexpr int A = decltype(AI)::value;
    Real v[Q];
    const Real B[3] = {rec[A][1], rec[A][2], rec[A][3]};
    expand_cotangents<Real, A>(mu, rec[A][0], B, fw1, lo, hi, v);
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      S[A][ip][pos] = ok ? v[ip] : Real(0);
    });
  };

  // In-plane transposed lerps at a position for population ip: the cotangent
  // of Z(p) (x- and y-faces) and of Zn (z-faces).  at(A, ip, dr, dc): the A-face
  // cotangent dr rows and dc columns from the position; WX(k, dc), WY(k, dr):
  // the weights there.
  auto inplane = [&](auto I, auto at, auto WX, auto WY, Real& hz_out) -> Real {
    constexpr int ip = decltype(I)::value;
    constexpr int cx = CX[ip], cy = CY[ip];
    if constexpr (ip == 0) {
      hz_out = at(2, 0, 0, 0);
      return Real(0.5) * (at(0, 0, 0, 0) + at(0, 0, 0, -1)) + Real(0.5) * (at(1, 0, 0, 0) + at(1, 0, -1, 0));
    } else {
      // x-faces: this column is the left cell of its own slot, the right cell
      // of the slot before; rows 0 and c_y
      const Real a0 = Real(1) - WX(cx + 1, 0), a1 = WX(cx + 1, -1);
      Real hx = a0 * at(0, ip, 0, 0) + a1 * at(0, ip, 0, -1);
      if constexpr (cy != 0) {
        const Real m0 = Real(1) - WY(cy < 0 ? 3 : 4, 0), m1 = WY(cy < 0 ? 3 : 4, cy);
        hx = m0 * hx + m1 * (a0 * at(0, ip, cy, 0) + a1 * at(0, ip, cy, -1));
      }
      // y-faces: this row is the lower cell of its own slot, the upper cell of
      // the slot before; columns 0 and c_x
      const Real b0 = Real(1) - WY(cy + 1, 0), b1 = WY(cy + 1, -1);
      Real hy = b0 * at(1, ip, 0, 0) + b1 * at(1, ip, -1, 0);
      if constexpr (cx != 0) {
        const Real m0 = Real(1) - WX(cx < 0 ? 3 : 4, 0), m1 = WX(cx < 0 ? 3 : 4, cx);
        hy = m0 * hy + m1 * (b0 * at(1, ip, 0, cx) + b1 * at(1, ip, -1, cx));
      }
      // z-face: columns 0, c_x; rows 0, c_y
      Real hz = at(2, ip, 0, 0);
      Real hz2 = Real(0);
      if constexpr (cy != 0) hz2 = at(2, ip, cy, 0);
      if constexpr (cx != 0) {
        const Real m0 = Real(1) - WX(cx < 0 ? 3 : 4, 0), m1 = WX(cx < 0 ? 3 : 4, cx);
        hz = m0 * hz + m1 * at(2, ip, 0, cx);
        if constexpr (cy != 0) hz2 = m0 * hz2 + m1 * at(2, ip, cy, cx);
      }
      if constexpr (cy != 0) {
        const Real m0 = Real(1) - WY(cy < 0 ? 3 : 4, 0), m1 = WY(cy < 0 ? 3 : 4, cy);
        hz = m0 * hz + m1 * hz2;
      }
      hz_out = hz;
      return hx + hy;
    }
  };

  // wall ghost folded into this cell: position and weight (at most one wall axis)
  int gR0 = -1, gC0 = -1;
  Real gq = Real(0);
  if (cell_lane && !P.periodic[1]) {
    if (j0 == 0 && R <= 2) {
      gR0 = 0, gC0 = C, gq = R == 1 ? (Real)P.qlo[1] : Real(1) - (Real)P.qlo[1];
    } else if (j0 + th == ny && R >= th - 1) {
      gR0 = th + 1, gC0 = C, gq = R == th ? (Real)P.qhi[1] : Real(1) - (Real)P.qhi[1];
    }
  } else if (cell_lane && !P.periodic[0]) {
    if (i0 == 0 && C <= 2) {
      gR0 = R, gC0 = 0, gq = C == 1 ? (Real)P.qlo[0] : Real(1) - (Real)P.qlo[0];
    } else if (i0 + TX == nx && C >= TX - 1) {
      gR0 = R, gC0 = TX + 1, gq = C == TX ? (Real)P.qhi[0] : Real(1) - (Real)P.qhi[0];
    }
  }
  const bool ghost = gR0 >= 0;

  Real accP[Q], accC[Q], accN[Q];
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    accP[ip] = Real(0);
    accC[ip] = Real(0);
    lamC[ip] = Real(0);
  });
  load_lam(I0{}, IQ{}, wrap(z0 - 1), true);
  load_recs(wrap(z0 - 1), true);

  for (int p = PLANES == 1 ? z0 : z0 - 1; p <= (PLANES == 1 ? z0 : zend); p++) {
    const int pos = here(pos0), Rg = here(Rg0), Cg = here(Cg0);  // (addresses formed anew each plane)
    // lam'(p), complete
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      lamP[ip] = lamC[ip];
      lamC[ip] = (Real)lraw[ip];
    });
    if constexpr (FLOW) {
      // rn is 0 where nothing was loaded (s0 or lam' is unused there)
      const Real inv = Real(1) / (rn != Real(0) ? rn : Real(1)), sc = s0 * inv, t0 = -sc * (jn * inv);
      const Real ax = fa == 0 ? Real(1) : Real(0), ay = fa == 1 ? Real(1) : Real(0), az = fa == 2 ? Real(1) : Real(0);
      static_for<Q>([&](auto I) {
        constexpr int ip = decltype(I)::value;
        lamC[ip] += fma_rn(Real(CX[ip]) * ax + Real(CY[ip]) * ay + Real(CZ[ip]) * az, sc, t0);
      });
    }
    if constexpr (PLANES == 1)
      for (int ip = 0; ip < Q; ip++) lamP[ip] = lamC[ip];
    // two planes: p = -1 gives lam' only, p = 2 takes plane 1 through the centre stage only
    if (PLANES == 2 && p < z0) {
      load_lam(I0{}, IQ{}, z0, true);
      load_recs(z0, true);
      continue;
    }
    const bool faces = PLANES != 2 || p < zend;
    if (faces) {
    __syncthreads();  // the previous plane's gather is done with S
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      if constexpr (CX[ip] != 0 || CY[ip] != 0) L[ip][pos] = lamC[ip];
    });
    __syncthreads();
    {
      // mu of a face: c_A (dt/dA lam' of the upper cell - dt/dA lam' of the lower)
      Real mu[10];
      const int posx = okx ? pos + 1 : pos, posy = oky ? pos + AC : pos;
      const Real ul = WXs[5][C], ur = WXs[5][min(C + 1, AC - 1)];
      static_for<10>([&](auto K) {
        constexpr int ip = XD[decltype(K)::value];
        mu[decltype(K)::value] = Real(CX[ip]) * (ur * L[ip][posx] - ul * lamC[ip]);
      });
      expand(std::integral_constant<int, 0>{}, pos, mu, okx, wlx, whx);
      const Real vl = WYs[5][R], vr = WYs[5][min(R + 1, TY + 1)];
      static_for<10>([&](auto K) {
        constexpr int ip = YD[decltype(K)::value];
        mu[decltype(K)::value] = Real(CY[ip]) * (vr * L[ip][posy] - vl * lamC[ip]);
      });
      expand(std::integral_constant<int, 1>{}, pos, mu, oky, wly, why);
      static_for<10>([&](auto K) {
        constexpr int ip = ZD[decltype(K)::value];
        mu[decltype(K)::value] = Real(CZ[ip]) * updz * (lamC[ip] - lamP[ip]);
      });
      expand(std::integral_constant<int, 2>{}, pos, mu, p >= z0, false, false);
    }
    }
    // The centre stage's inputs of plane p-1 first, then, in groups, what the
    // next plane needs
    const bool centre = stored && (PLANES == 1 || p - 1 >= z0);
    const bool more = PLANES == 0 ? p < zend : (PLANES == 2 && p + 1 < zend);
    const unsigned cell = centre ? (PLANES == 1 ? 0u : (unsigned)(p - 1) * plane) + column : 0u;
    const unsigned v8 = centre ? cell * 8u : kOutOfRange;
    Real m4[4] = {Real(1), Real(0), Real(0), Real(0)};
    RawCell<Real, Store> fraw;
    double fc[3], g0[3];
    if constexpr (kMoments)
      mb.ld4(centre ? cell * (unsigned)(4 * sizeof(Real)) : kOutOfRange, m4);
    else
      fraw.load(bin, cell, (unsigned)P.N);
    for (int a = 0; a < 3; a++) fc[a] = fcb.ld<double>(v8, a * vec_pop);
    for (int a = 0; a < 3; a++) g0[a] = gradb.ld<double>(v8, a * vec_pop);
    if (faces) {
    __syncthreads();
    // transposed reconstruction: a position's in-plane lerps through the
    // transposed z-lerps
    auto push = [&](auto I, Real hzr, Real hz) {
      constexpr int ip = decltype(I)::value;
      constexpr int cz = CZ[ip];
      if constexpr (cz == 0) {
        accC[ip] += hzr;
      } else if constexpr (cz > 0) {
        accC[ip] += (Real(1) - mz7) * hzr;
        accP[ip] += mz7 * hzr;
      } else {
        accC[ip] += (Real(1) - mz6) * hzr;
        accN[ip] += mz6 * hzr;
      }
      const Real wn = ip == 0 ? Real(0.5) : wRz[cz + 1];
      accP[ip] += (Real(1) - wn) * hz;
      accC[ip] += wn * hz;
    };
    const int gat = Rg * AC + Cg;
    auto cell_at = [&](int A, int ip, int dr, int dc) -> Real { return S[A][ip][gat + dr * AC + dc]; };
    auto cell_wx = [&](int k, int dc) -> Real { return WXs[k][Cg + dc]; };
    auto cell_wy = [&](int k, int dr) -> Real { return WYs[k][Rg + dr]; };
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      if constexpr (ip == 1) load_lam(I0{}, I10{}, wrap(p + 1), more);
      if constexpr (ip == 7) load_lam(I10{}, IQ{}, wrap(p + 1), more);
      if constexpr (ip == 13) load_recs(wrap(p + 1), more);
      Real hz;
      const Real hzr = inplane(I, cell_at, cell_wx, cell_wy, hz);
      accN[ip] = Real(0);
      push(I, hzr, hz);
    });
    if (ghost) {
      // The same at the ghost position, whose stencil reaches outside the
      // staged region: nothing is there, and the idle position holds zeros.
      // (One branch for all populations and no condition per value: with a
      // branch each, the tiles at a wall took twice the time.)  The weights
      // there only multiply zeros; their index is clamped.
      const int gR = here(gR0), gC = here(gC0);
      int gi[3][3], gx[3], gy[3];
      for (int q = -1; q <= 1; q++) {
        gx[q + 1] = min(max(gC + q, 0), AC - 1);
        gy[q + 1] = min(max(gR + q, 0), TY + 1);
        for (int v = -1; v <= 1; v++) {
          const bool in = gR + q >= 0 && gR + q <= th + 1 && gC + v >= 0 && gC + v <= TX + 1;
          gi[q + 1][v + 1] = in ? (gR + q) * AC + gC + v : T::NP;
        }
      }
      auto ghost_at = [&](int A, int ip, int dr, int dc) -> Real { return S[A][ip][gi[dr + 1][dc + 1]]; };
      auto ghost_wx = [&](int k, int dc) -> Real { return WXs[k][gx[dc + 1]]; };
      auto ghost_wy = [&](int k, int dr) -> Real { return WYs[k][gy[dr + 1]]; };
      static_for<Q>([&](auto I) {
        Real hz;
        const Real hzr = inplane(I, ghost_at, ghost_wx, ghost_wy, hz);
        push(I, gq * hzr, gq * hz);
      });
    }
    if constexpr (PLANES == 1)
      for (int ip = 0; ip < Q; ip++) accP[ip] += accC[ip] + accN[ip];
    if constexpr (PLANES == 2) {
      const bool low = p == z0;  // plane -1 is plane 1, plane 2 plane 0
      for (int ip = 0; ip < Q; ip++) {
        const Real v = accP[ip] + accN[ip];
        if (low) accN[ip] = v; else accP[ip] = v;
      }
    }
    }
    // centre-stage adjoint of plane p-1 (as k_adj_cells)
    Real rho = m4[0], j[3] = {m4[1], m4[2], m4[3]};
    if constexpr (!kMoments) {
      Real ff[Q], u0[3];
      fraw.decode(P, ff, rho, u0);
      cell_moments<Real>(ff, rho, j);
    }
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      accP[ip] += Real(4.0 / 3.0) * lamP[ip];
    });
    Real F[3], u[3], ut[3];
    const Real invr = Real(1) / rho;
    for (int a = 0; a < 3; a++) {
      F[a] = Famb[a] + (Real)fc[a];
      ut[a] = j[a] * invr;
      u[a] = ut[a] + hdt * F[a];
    }
    Real g_rho, g_u[3], g_F[3];
    feq_adjoint<Real>(accP, bw2, bw0, rho, u, F, g_rho, g_u, g_F, AllPops{});
    const Real Acoef = g_rho - (g_u[0] * ut[0] + g_u[1] * ut[1] + g_u[2] * ut[2]) * invr;
    const unsigned vl = centre ? cell * (unsigned)sizeof(Lam) : kOutOfRange;
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      const Real v = -lamP[ip] * Real(1.0 / 3.0) + bw1 * accP[ip] + Acoef +
                     (g_u[0] * Real(CX[ip]) + g_u[1] * Real(CY[ip]) + g_u[2] * Real(CZ[ip])) * invr;
      outb.st((Lam)v, vl, ip * lam_pop);
    });
    for (int a = 0; a < 3; a++) gradb.st(g0[a] + (double)(g_F[a] + hdt * g_u[a]), v8, a * vec_pop);
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      accP[ip] = accC[ip];
      accC[ip] = accN[ip];
    });
  }
}

// The z-marching gather covers FP32 and FP64 arithmetic on grids of whole 32 x
// 8 columns with z periodic and uniform, at most one wall axis (x or y), and
// face arrays and lam' that 32-bit buffer offsets reach.
bool gather_z_supported(const Ctx& c) {
  const Setup& s = c.s;
  if (c.kernel == 0) return false;
  if (s.n[0] % 32 != 0 || s.n[1] % 8 != 0 || !s.periodic[2] || !s.uniform[2]) return false;
  if (!s.periodic[0] && !s.periodic[1]) return false;
  if (!s.periodic[0] && s.n[0] < 3) return false;
  if (!s.periodic[1] && s.n[1] < 3) return false;
  const double rb = c.precision == 0 ? 8.0 : 4.0;
  if ((double)Q * c.kp.eN * rb >= 2147483648.0 || (double)Q * c.kp.N * 8.0 >= 2147483648.0) return false;
  return true;
}

}  // namespace

// Tile height (12 or 8 rows) and z-chunks of the gather, one workgroup per CU;
// a chunk gathers the two planes beside it too.  A plane of an 8-row tile takes
// 0.8 of the time, so they go where they fill more CUs (64x64x32: FP32 adjoint
// step 58 us against 62 with 12 rows, FP64 gather 56.5 against 58).
GatherPlan gather_plan(const Setup& s, bool fp64) {
  GatherPlan best{};
  double least = 0;
  for (const int rows : {12, 8}) {
    const long long tiles = (long long)(s.n[0] / (fp64 ? 16 : 32)) * ((s.n[1] + rows - 1) / rows);
    const int nz = s.n[2], nc = plan_z_chunks(tiles, nz, 256, 2.0);
    const double cost = (rows == 12 ? 1.0 : 0.8) * (double)((tiles * nc + 255) / 256) * ((nz + nc - 1) / nc + 2.0);
    if (rows == 12 || cost < 0.97 * least) {
      best = {rows, nc, tiles * nc};
      least = cost;
    }
  }
  return best;
}

namespace {

template <class Real, class Store, class Lam, int ROWS, bool FLOW, int PLANES>
void launch_gather(const Ctx& cx, const GatherPlan& g, const void* f, const Lam* lam_next, Lam* lam_prev,
                   double* grad, int mom, const double* ubar) {
  const double inv_vol = 1.0 / (cx.s.width[0] * cx.s.width[1] * cx.s.width[2]);
  hipLaunchKernelGGL((k_adj_cells_z<Real, Store, Lam, ROWS, FLOW, PLANES>), dim3((unsigned)g.nblocks),
                     dim3(GatherTile<Real, ROWS>::NT), 0, cx.stream, cx.kp, static_cast<const Store*>(f), lam_next,
                     static_cast<const Real*>(cx.adj_faces), lam_prev, grad, g.nchunk, mom, FLOW ? ubar : nullptr,
                     inv_vol);
}
template <class Real, class Store, class Lam, bool FLOW>
void launch_gather(const Ctx& cx, const void* f, const Lam* lam_next, Lam* lam_prev, double* grad, int mom,
                   const double* ubar) {
  const GatherPlan g = gather_plan(cx.s, sizeof(Real) == 8);
  const bool tall = g.rows == 12;
  if (cx.s.n[2] == 1)
    return tall ? launch_gather<Real, Store, Lam, 12, FLOW, 1>(cx, g, f, lam_next, lam_prev, grad, mom, ubar)
                : launch_gather<Real, Store, Lam, 8, FLOW, 1>(cx, g, f, lam_next, lam_prev, grad, mom, ubar);
  if constexpr (sizeof(Real) == 8) {
    if (cx.s.n[2] == 2 && g.nchunk == 1)
      return tall ? launch_gather<Real, Store, Lam, 12, FLOW, 2>(cx, g, f, lam_next, lam_prev, grad, mom, ubar)
                  : launch_gather<Real, Store, Lam, 8, FLOW, 2>(cx, g, f, lam_next, lam_prev, grad, mom, ubar);
  }
  return tall ? launch_gather<Real, Store, Lam, 12, FLOW, 0>(cx, g, f, lam_next, lam_prev, grad, mom, ubar)
              : launch_gather<Real, Store, Lam, 8, FLOW, 0>(cx, g, f, lam_next, lam_prev, grad, mom, ubar);
}

// One adjoint step.  Lam = double: every configuration; Lam = float (FP32
// arithmetic with the z-marching gather only): lam' and lam in FP32.
template <class Real, class Store, class Lam>
hipError_t run_adjoint(Ctx& cx, const void* f, const Lam* lam_next, Lam* lam_prev, double* grad, int wall,
                       double* fpart, long long fpart_len, long long* nparts, int mom, const double* ubar) {
  const KParams& P = cx.kp;
  Real* faces = static_cast<Real*>(cx.adj_faces);
  constexpr bool kLam32 = std::is_same<Lam, float>::value;
  bool handled = false;
  // With the z-marching gather the fused adjoint-face pass writes the
  // compact face records, which the gather expands
  const int format = adjoint_record_format(cx, kLam32);
  const bool compact = format != kFacesFull;
  if (kLam32 && !compact) return hipErrorNotSupported;
  // Each format leaves some slots unwritten (ghost rows, missing faces) that
  // must read as 0: clear the arrays when the format changes.
  const int fmt = compact ? 1 : 0;
  if (cx.adj_faces_format != fmt) {
    hipError_t e0 = hipMemsetAsync(cx.adj_faces, 0, (size_t)P.eN * 3 * Q * sizeof(Real), cx.stream);
    if (e0 != hipSuccess) return e0;
    cx.adj_faces_format = fmt;
  }
  // the controller term rides on lam' where the face pass hands rho and j to
  // the gather (storage in the arithmetic type) and lam' is the sweep's:
  // FP32 with FP32 arithmetic, FP64 with FP64
  constexpr bool kFuse = std::is_same<Store, Real>::value && (kLam32 || std::is_same<Real, double>::value);
  if (ubar && !kFuse) return hipErrorNotSupported;
  hipError_t e = launch_adjoint_faces_fused(cx, f, lam_next, faces, format, &handled, fpart, fpart_len, nparts, mom,
                                            ubar);
  if (e != hipSuccess) return e;
  // the force cotangent of the face collisions comes from the fused pass only
  if (fpart && !handled) return hipErrorNotSupported;
  {
    if (compact) {
      bool flow = false;
      if constexpr (kFuse) {
        flow = ubar != nullptr;
        if (flow) launch_gather<Real, Store, Lam, true>(cx, f, lam_next, lam_prev, grad, mom, ubar);
      }
      if (!flow) launch_gather<Real, Store, Lam, false>(cx, f, lam_next, lam_prev, grad, mom, ubar);
      return hipGetLastError();
    }
  }
  if constexpr (!kLam32) {
    if (!handled) {
      if (!cx.fbx) {
        e = cx.alloc(&cx.fbx, (size_t)P.eN * Q * sizeof(Real));
        if (e != hipSuccess) return e;
      }
      e = launch_fbar_ghosts(cx, f, cx.fbx);
      if (e != hipSuccess) return e;
      const unsigned nbe = (unsigned)((P.eN + 255) / 256);
      const Real* fbx = static_cast<const Real*>(cx.fbx);
      hipLaunchKernelGGL((k_adj_faces<Real, 0>), dim3(nbe), dim3(256), 0, cx.stream, P, fbx, lam_next, faces);
      hipLaunchKernelGGL((k_adj_faces<Real, 1>), dim3(nbe), dim3(256), 0, cx.stream, P, fbx, lam_next, faces);
      hipLaunchKernelGGL((k_adj_faces<Real, 2>), dim3(nbe), dim3(256), 0, cx.stream, P, fbx, lam_next, faces);
    }
    for (int b = 0; b < 3; b++) {
      if (!P.periodic[b]) continue;
      const long long cnt = (long long)P.e[(b + 1) % 3] * P.e[(b + 2) % 3] * 3 * Q;
      hipLaunchKernelGGL((k_face_ghosts<Real>), dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, cx.stream, P,
                         faces, b);
    }
    const unsigned nbc = (unsigned)((P.n[0] + kCX - 1) / kCX * ((P.n[1] + kCY - 1) / kCY) *
                                    ((P.n[2] + kCZ - 1) / kCZ));
    hipLaunchKernelGGL((k_adj_cells<Real, Store>), dim3(nbc), dim3(256), 0, cx.stream, P,
                       static_cast<const Store*>(f), lam_next, static_cast<const Real*>(cx.adj_faces), lam_prev, grad,
                       wall);
    return hipGetLastError();
  }
  return hipErrorNotSupported;
}

}  // namespace

namespace {

template <class Lam>
hipError_t adjoint_step(Ctx& c, const void* f, const Lam* lam_next, Lam* lam_prev, double* grad_force,
                        double* fpart, long long fpart_len, long long* nparts, int mom, const double* ubar) {
  const Setup& s = c.s;
  if (s.recon != 0) return hipErrorNotSupported;
  int walls = 0, wall = -1;
  for (int a = 0; a < 3; a++)
    if (!s.periodic[a]) {
      walls++;
      wall = a;
    }
  if (walls > 1) return hipErrorNotSupported;
  // FP16 non-equilibrium storage has no adjoint
  if (c.precision == 3) return hipErrorNotSupported;
  if constexpr (!std::is_same<Lam, double>::value) {
    if (c.precision == 0) return hipErrorNotSupported;
  }
  const size_t rb = c.precision == 0 ? 8 : 4;
  if (!c.adj_faces) {
    const size_t bytes = (size_t)c.kp.eN * 3 * Q * rb;
    hipError_t e = c.alloc(&c.adj_faces, bytes);
    if (e != hipSuccess) return e;
    c.adj_faces_format = -1;  // cleared before first use (run_adjoint)
  }
  switch (c.precision) {
    case 0:
      if constexpr (std::is_same<Lam, double>::value)
        return run_adjoint<double, double, Lam>(c, f, lam_next, lam_prev, grad_force, wall, fpart, fpart_len,
                                                nparts, mom, ubar);
      else
        return hipErrorNotSupported;
    case 1:
      return run_adjoint<float, float, Lam>(c, f, lam_next, lam_prev, grad_force, wall, fpart, fpart_len, nparts,
                                            mom, ubar);
    default:
      return run_adjoint<float, __half, Lam>(c, f, lam_next, lam_prev, grad_force, wall, fpart, fpart_len, nparts,
                                             mom, ubar);
  }
}

}  // namespace

hipError_t launch_adjoint(Ctx& c, const void* f, const double* lam_next, double* lam_prev, double* grad_force,
                          double* fpart, long long fpart_len, long long* nparts, int mom, const double* ubar) {
  return adjoint_step<double>(c, f, lam_next, lam_prev, grad_force, fpart, fpart_len, nparts, mom, ubar);
}

hipError_t launch_adjoint_lam32(Ctx& c, const void* f, const float* lam_next, float* lam_prev, double* grad_force,
                                double* fpart, long long fpart_len, long long* nparts, int mom,
                                const double* ubar) {
  return adjoint_step<float>(c, f, lam_next, lam_prev, grad_force, fpart, fpart_len, nparts, mom, ubar);
}

// The face-record format of an adjoint step: compact records for the
// z-marching gather wherever it and the fused face pass run (lam' in FP32
// with lam32), else the 19 cotangents of every face.
int adjoint_record_format(const Ctx& c, bool lam32) {
  if (!gather_z_supported(c) || !adjoint_faces_fused_covers(c)) return kFacesFull;
  return lam32 ? kFacesCompactLam32 : kFacesCompact;
}

bool adjoint_flow_fused(const Ctx& c) {
  if (c.precision == 0) return adjoint_record_format(c, false) == kFacesCompact;
  return c.precision == 1 && adjoint_lam32_supported(c);
}

bool adjoint_lam32_supported(const Ctx& c) {
  if (c.precision == 0 || c.precision == 3 || c.s.recon != 0) return false;
  return gather_z_supported(c) && adjoint_faces_fused_covers(c);
}

// The sweep's adjoint step: FP64 on the fused face pass (full records), or
// FP32 arithmetic with lam in FP32 (compact records); the forms
// launch_adjoint_faces_fused gives the force cotangent for.
bool adjoint_flow_supported(const Ctx& c) {
  if (c.s.recon != 0) return false;
  int walls = 0;
  for (int a = 0; a < 3; a++) walls += !c.s.periodic[a];
  if (walls > 1) return false;
  if (c.precision == 0) return adjoint_faces_fused_covers(c);
  return adjoint_lam32_supported(c);
}

}  // namespace dugks
