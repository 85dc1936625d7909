// Fused DUGKS step: one kernel per time step, f read once and written once;
// and the adjoint-face pass.
//
// Decomposition of the step (step_kernel.h).  A workgroup owns a TX x TY tile
// of (x, y) columns and marches along z over a chunk of planes.  Its lanes
// hold the tile's columns, the two y-halo rows and the two x-halo columns; a
// column is a lane's with FP32 arithmetic and a pair of lanes' with FP64
// (step_common.h).  Each plane it:
//   - computes f-bar+ of its columns at plane p+1 (calc_fb1 of the reference,
//     src/dugks.cu:1131-1196) from the f it loaded a plane ahead; halo columns
//     recompute it, wall ghost columns extrapolate it
//     (src/dugks.cu:1234-1251 and the stretched form,
//     src/fortran/channel/src/dugks.cuf:365-374);
//   - reconstructs every face once (the reference computes each interior face
//     twice): the trilinear interpolation of src/dugks.cu:756-906 is
//     evaluated z-lerp first, so the x- and y-faces of plane p read a single
//     LDS plane Z(p) and the z-face between p and p+1 reads Zn(p+1/2);
//   - applies wall bounce-back and the face collision (f2ruvwh + feq_s,
//     src/dugks.cu:675-709, 1201-1207) and keeps only the populations that
//     cross the face;
//   - updates plane p (src/dugks.cu:945-956) into the other f buffer.
// Two barriers per plane: [f-bar(p+1); write Z(p), Zn(p+1/2)] | [faces] |
// [update], the update of one plane overlapping the next plane's f-bar.
// z must be periodic; x and y may be periodic or walls, uniform or stretched.
// GRAD: the gradient reconstruction instead (calc_fx, src/dugks.cu:421-583:
// the mean of the two cells beside the face less h c.g, with the normal
// derivative from those two cells and the tangential ones by central
// differences of the two-cell means), on uniform axes; the LDS then holds a
// ring of the f-bar+ planes p-1, p and p+1, written as each is computed.
// Other configurations use the two-pass kernels.
//
// What bounds it.  The step moves 38 values per cell (f in, f out; halos come
// from L2) and issues about 1450 VALU lane-instructions per cell in FP32 and 2360
// in FP64.  On 256x192x256 with one
// MI355X (a large copy runs at 4.9 TB/s) the traffic alone takes 0.39 ms in
// FP32 and 0.78 ms in FP64, the arithmetic with the memory accesses taken out
// 0.55 and 1.13 ms: the kernel is bound by issue.  Two waves per SIMD fit, so
// what counts is that a wave never waits: the loads of the next plane go out
// in three groups between the phases (issued in one burst they fill the
// memory pipeline and the wave stalls at issue: 0.83 against 0.68 ms in FP32,
// 1.54 against 1.19 ms in FP64), loads and stores run without branches so
// that a wait counts exactly, and the halo waves take their share of the
// y-faces.  Measured per step, 256x192x256 periodic / channel with a
// flow-rate controller (before: a lane per column with planes of single
// values in LDS, one wave per SIMD in FP64, whole-plane loads at once):
//   FP32          0.623 / 0.685 ms  (0.719 / 0.751)
//   FP64          1.185 / 1.329     (1.88  / 1.92)
//   FP16 dev.     0.649 / 0.710     (0.729 / 0.797)
//   FP16 non-eq.  0.717 / 0.772     (0.966 / 0.964)
#include <algorithm>
#include "device_common.h"

namespace dugks {

namespace {

#include "fused_common.h"
#include "step_common.h"

constexpr int kXcds = 8;  // accelerator complex dies of an MI355X

// threads of a TX x TY tile's workgroup (Tile<TX, TY>::NT)
constexpr int Tile_nt(int TX, int TY) { return ((TY + 2) * TX + 2 * (TY + 2) + 63) / 64 * 64; }

template <int TX, int TY>
struct Tile {
  static constexpr int NROW = (TY + 2) * TX;    // the tile rows and the two y-halo rows
  static constexpr int NHALO = 2 * (TY + 2);     // the two x-halo columns
  static constexpr int NT = (NROW + NHALO + 63) / 64 * 64;
  static constexpr int AC = TX + 2;
  static_assert(TX % 16 == 0 && TX <= 64, "rows of 16, 32, 48 or 64 lanes");
};

// Inputs and outputs of the adjoint-face mode of the fused kernel.
struct AdjFaceIO {
  const void* lam;    // lam' = dJ/df(n+1), SoA [19][nz][ny][nx], FP64 or (LamT = float) FP32
  void* faces;        // out: [3][19][ghost-inclusive face slot], arithmetic type; COMPACT:
                      // [3][slot][kCompact], then (storage in the arithmetic type) two
                      // [N][4] regions of rho, j of every cell
  int mom = 0;        // COMPACT, such storage: the region the pass writes rho, j of fin into
  // sweep through the flow-rate controller: lam' still lacks the bulk
  // velocity's cotangent ubar (dV/V) (c_ia - u_a)/rho of f(n+1), whose rho, j
  // the previous pass left in the other region; added as lam' is loaded
  // (nullptr: lam' is complete)
  const double* ubar = nullptr;
  double inv_vol = 0;  // 1 / V
};

// Gradient reconstruction of one population at a face's foot point: the
// mean m of the two cells beside the face less h c.g (calc_fx,
// src/dugks.cu:421-583); the terms of the components c_a = 0 are left out
// (they add zero).  dx, dy, dz are differences of values, kx, ky, kz what turns
// them into h times the derivative.
template <int cx, int cy, int cz, class Real>
__device__ __forceinline__ Real grad_foot(Real m, Real kx, Real dx, Real ky, Real dy, Real kz, Real dz) {
  if constexpr (cx != 0) m = fma_rn(Real(-cx) * kx, dx, m);
  if constexpr (cy != 0) m = fma_rn(Real(-cy) * ky, dy, m);
  if constexpr (cz != 0) m = fma_rn(Real(-cz) * kz, dz, m);
  return m;
}

// The adjoint-face pass of the step taken from fin: every face is
// reconstructed and its collision linearised as in the step (trilinear
// reconstruction), and the cotangents of its 19 reconstructed values, driven
// by lam' (adj.lam), are written to adj.faces; nothing else is written.  FADJ:
// also the cotangent of the ambient force along the flow axis through the
// face collisions, summed per block into partial[tile] (fixed order).
//
// What bounds it: with compact records the 38 loads and 4 wide stores of a
// plane at issue, then the faces' arithmetic.  So the loads go out in three
// groups (lam' after f-bar+, f of the plane after next between the faces), and
// wall ghosts are extrapolated in LDS (the lanes of a ghost column formed f-bar+
// of two columns from memory before, alone and waiting).  256x192x256 channel,
// FP32: 0.86 ms, before 1.09; 64x64x32 FP64: 35 us, before 47.
template <class Real, class Store, int TX, int TY, bool COMPACT = false, class LamT = double, bool FADJ = false>
// FP32 arithmetic: two blocks per CU (at most 256 registers per lane)
__global__ void __launch_bounds__(((TY + 2) * TX + 2 * (TY + 2) + 63) / 64 * 64, sizeof(Real) == 4 ? 2 : 1)
    k_adj_tile_faces(KParams P, const Store* __restrict__ fin, int TZ, double* __restrict__ partial, AdjFaceIO adj) {
  using T = Tile<TX, TY>;
  constexpr int AC = T::AC;
  // LDS planes indexed (row, column).  16-wide rows put four rows in a wave:
  // column-major planes (column stride TY + 2, even) then keep the lanes of
  // a ds_read on distinct banks; 32-wide rows are conflict-free row-major.
  constexpr bool CM = TX == 16;
  auto ia = [](int rr, int cc) { return CM ? cc * (TY + 2) + rr : rr * AC + cc; };       // A, An, Lam
  __shared__ Real A[Q][(TY + 2) * AC];    // Z(p): tangential z-lerp of f-bar(p)
  __shared__ Real An[Q][(TY + 2) * AC];   // Zn(p+1/2): normal z-lerp between p and p+1
  __shared__ Real Lam[Q][(TY + 2) * AC];  // lam'(p) of the tile and halo
  __shared__ Real WX[6][TX + 2];           // weights per tile column
  __shared__ Real WY[6][TY + 2];           // weights per tile row

  const int nx = P.n[0], ny = P.n[1], nz = P.n[2];
  const int t = threadIdx.x;
  // XCD-aware tile order.  Workgroups are dealt round-robin to the 8 XCDs
  // (workgroup b runs on XCD b % 8), each with its own L2.  Every XCD gets a
  // contiguous run of tiles (x fastest), so the tiles whose halos overlap share
  // one L2 and run at about the same time; the plain order would put
  // x-neighbours on different XCDs and every x-halo line would come from HBM
  // (96x36x128 FP32, full records, 468 tiles: 178 us an adjoint step, in plain
  // order 219).
  const int gx = nx / TX, gy = ny / TY;
  const int ntiles = gx * gy * (int)gridDim.z;
  const int b = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), xcd = b % kXcds;
  const int tt = xcd * (ntiles / kXcds) + min(xcd, ntiles % kXcds) + b / kXcds;
  const int bx = tt % gx, by = (tt / gx) % gy, bz = tt / (gx * gy);
  const int i0 = bx * TX, j0 = by * TY;
  const int z0 = bz * TZ;
  const int zend = min(z0 + TZ, nz);
  const unsigned span = (unsigned)state_bytes<Store>((unsigned long long)P.N);
  const StateBuf<Store> bin(fin, span);

  // column of this thread in tile coordinates: r = 0..TY+1 (y = j0-1+r),
  // c = -1..TX (x = i0+c).  Lanes: the TY interior rows first (whole waves
  // when TY*TX is a multiple of 64, so the interior-only phases run on as few
  // waves as possible), then the two y-halo rows, then the two x-halo columns
  // packed behind them; lanes past those idle.
  int r = 0, c = 0;
  bool active = true;
  if (t < TY * TX) {
    r = t / TX + 1;
    c = t % TX;
  } else if (t < T::NROW) {
    const int u = t - TY * TX;
    r = u < TX ? 0 : TY + 1;
    c = u % TX;
  } else if (t < T::NROW + T::NHALO) {
    const int u = t - T::NROW;
    r = u % (TY + 2);
    c = u < TY + 2 ? -1 : TX;
  } else {
    active = false;
  }
  const bool interior = t < T::NROW && r >= 1 && r <= TY;
  int gi = i0 + c, gj = j0 - 1 + r;
  if (P.periodic[0]) gi = (gi + nx) % nx;
  if (P.periodic[1]) gj = (gj + ny) % ny;
  // ghost-inclusive table indices of the column
  const int mi = gi + 1, mj = gj + 1;
  // weight tables in the arithmetic type (layout documented on KParams)
  auto tx = [&](int idx) { return tabv<Real>(P, 0, idx); };
  auto ty = [&](int idx) { return tabv<Real>(P, 1, idx); };
  auto tz = [&](int idx) { return tabv<Real>(P, 2, idx); };

  Real Famb[3];
  ambient_force<Real>(P, Famb);
  const Real hdt = (Real)P.hdt, fw0 = (Real)P.fw0, fw1 = (Real)P.fw1, fw2 = (Real)P.fw2;
  // uniform z weights (z is periodic and uniform here)
  const Real wzt_m = tz(9 + 6);  // tangential, toward p+1 (c_z = -1)
  const Real wzt_p = tz(9 + 7);  // tangential, toward p-1 (c_z = +1)
  const Real wzn[3] = {tz(9 + 0), tz(9 + 1), tz(9 + 2)};  // normal, toward p+1
  const Real updz = tz(9 + 8);
  // Per-column and per-row weights of the tile, copied once into LDS: the
  // tables are not written by this kernel, but the compiler cannot prove that
  // against the f stores and would reload them (or hold them in registers)
  // across the plane loop.  Row k of WX/WY: 0-2 the -face normal weight
  // toward the upper cell for c = -1, 0, +1; 3-4 the tangential shift
  // weights for c < 0 and c > 0; 5 dt/d.  The -face index is clamped for the
  // ghost column/row, which never owns a -face.
  for (int u = t; u < 6 * (TX + 2) + 6 * (TY + 2); u += T::NT) {
    const bool isx = u < 6 * (TX + 2);
    const int v = isx ? u : u - 6 * (TX + 2);
    const int n = isx ? TX + 2 : TY + 2;
    const int k = v / n, q = v % n;
    int g = isx ? i0 - 1 + q : j0 - 1 + q;
    const int na = isx ? nx : ny;
    if (P.periodic[isx ? 0 : 1]) g = (g + na) % na;
    const int m = g + 1;
    const int idx = k < 3 ? max(m - 1, 0) * 9 + k : m * 9 + (k + 3);
    (isx ? WX[k][q] : WY[k][q]) = isx ? tx(idx) : ty(idx);
  }
  auto xn = [&](int k) { return WX[k][c + 1]; };
  auto xt = [&](int s) { return WX[3 + s][c + 1]; };
  auto yn = [&](int k) { return WY[k][r]; };
  auto yt = [&](int s) { return WY[3 + s][r]; };

  Real fbm[5], fbc[Q], fbn[Q];
  const int as = P.flow_axis;
  // FADJ: the face collisions' force cotangents of this thread's faces
  double fsum[3] = {0, 0, 0};

  // +z face of an interior column from Zn in A: bilinear over the upwind
  // tangential neighbours, then collision; out = crossing populations
  auto zface_rec = [&](Face<Real, 2>& fc) {
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      constexpr int cx = CX[ip], cy = CY[ip];
      Real v = An[ip][ia(r, c + 1)];
      if constexpr (cx != 0) {
        const Real w = xt(cx < 0 ? 0 : 1);
        v = lerp_(v, An[ip][ia(r, c + 1 - cx)], w);
        if constexpr (cy != 0) {
          const Real wy = yt(cy < 0 ? 0 : 1);
          const Real v2 = lerp_(An[ip][ia(r - cy, c + 1)], An[ip][ia(r - cy, c + 1 - cx)], w);
          v = lerp_(v, v2, wy);
        }
      } else if constexpr (cy != 0) {
        const Real wy = yt(cy < 0 ? 0 : 1);
        v = lerp_(v, An[ip][ia(r - cy, c + 1)], wy);
      }
      fc.template put<ip>(v);
    });
  };
  // adjoint-face mode: lam' of population ip at an interior cell (0 for a
  // ghost, cell < 0) and the store of a face's cotangents
  // (both arrays are < 2 GiB, checked at launch: 32-bit buffer offsets)
  constexpr unsigned kLamBytes = sizeof(LamT);
  const RawBuf lamb(adj.lam, (unsigned)(Q * P.N * kLamBytes));
  const unsigned lam_pop = (unsigned)(P.N * kLamBytes);         // bytes per population
  const unsigned face_pop = (unsigned)(P.eN * sizeof(Real));    // bytes per population
  // lam' of the thread's own column at plane k (0 for a wall ghost column).
  // The pass computes the -x and -y faces of its cells (and a wall's +x, +y
  // face, whose outside column is a ghost), so the right halo column, the top
  // halo row and the bottom-left corner never need lam' and load none.
  const bool lam_cell = active && gi >= 0 && gi < nx && gj >= 0 && gj < ny && c < TX && r <= TY &&
                        !(c < 0 && r == 0);
  auto load_lam = [&](int k, Real (&l)[Q]) {
    const unsigned vb = lam_cell ? (unsigned)(((long long)k * ny + gj) * nx + gi) * kLamBytes : kOutOfRange;
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      if constexpr (ip != 0) l[ip] = (Real)lamb.ld<LamT>(vb, ip * lam_pop);
    });
  };
  // the flow-rate controller's term of lam' (AdjFaceIO::ubar): rho and j_a
  // of f(n+1) at the column's cell of plane k, loaded with lam', added before
  // lam' is used: lam'_i += s (c_ia - u_a), s = ubar (dV/V) / rho
  constexpr bool kFlowFuse = FADJ && COMPACT && std::is_same<Store, Real>::value;
  const bool fuse = kFlowFuse && adj.ubar != nullptr;
  const RawBuf momn = cell_records<Real>(adj.faces, 1 - adj.mom, P.eN, P.N);
  Real s0 = Real(0), ex = Real(0), ey = Real(0), ez = Real(0);
  if constexpr (kFlowFuse) {
    if (fuse && lam_cell)
      s0 = (Real)(adj.ubar[0] * P.wd[0][mi] * P.wd[1][mj] * P.wd[2][1] * adj.inv_vol);
    ex = as == 0 ? Real(1) : Real(0);
    ey = as == 1 ? Real(1) : Real(0);
    ez = as == 2 ? Real(1) : Real(0);
  }
  auto load_flow = [&](int k, Real& rn, Real& jn) {
    if constexpr (kFlowFuse) {
      const unsigned vb = fuse && lam_cell ? (unsigned)(((long long)k * ny + gj) * nx + gi) * 4u * sizeof(Real)
                                           : kOutOfRange;
      rn = momn.ld<Real>(vb, 0);
      jn = momn.ld<Real>(vb, (unsigned)(1 + as) * (unsigned)sizeof(Real));
    }
  };
  auto add_flow = [&](Real (&l)[Q], Real rn, Real jn) {
    if constexpr (kFlowFuse) {
      // rn is 0 where nothing was loaded (s0 is 0 there)
      const Real inv = Real(1) / (rn != Real(0) ? rn : Real(1));
      const Real s = s0 * inv, t0 = -s * (jn * inv);
      static_for<Q>([&](auto I) {
        constexpr int ip = decltype(I)::value;
        if constexpr (ip != 0) l[ip] += fma_rn(Real(CX[ip]) * ex + Real(CY[ip]) * ey + Real(CZ[ip]) * ez, s, t0);
      });
    }
  };
  Real lamc[Q], lamn[Q], rnn = Real(0), jnn = Real(0);
  load_lam(z0, lamc);
  if constexpr (kFlowFuse) {
    Real rn = Real(0), jn = Real(0);
    load_flow(z0, rn, jn);
    add_flow(lamc, rn, jn);
  }
  // compact form (COMPACT): Ac and B of a face
  auto store_compact = [&](int a, long long slot, Real Ac, const Real (&B)[3], bool ok = true) {
    const Real rec[kCompact] = {Ac, B[0], B[1], B[2]};
    face_records<Real>(adj.faces, a, P.eN)
        .st4(rec, ok ? (unsigned)slot * (unsigned)(kCompact * sizeof(Real)) : kOutOfRange);
  };
  auto store_face = [&](int a, long long slot, const Real (&lam)[Q]) {
    const RawBuf fb(static_cast<Real*>(adj.faces) + (long long)a * Q * P.eN, Q * face_pop);
    const unsigned vb = (unsigned)slot * (unsigned)sizeof(Real);
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      fb.st(lam[ip], vb, ip * face_pop);
    });
  };
  const long long e0 = P.e[0], e1 = P.e[1];

  // Columns inside the domain (tile and periodic halo) compute f-bar+ from f
  // of their own column; wall ghost columns are extrapolated in LDS.
  const bool own = active && gi >= 0 && gi < nx && gj >= 0 && gj < ny;
  // body force at plane k of the own column
  auto force_own = [&](int k, Real (&F)[3]) {
    F[0] = Famb[0];
    F[1] = Famb[1];
    F[2] = Famb[2];
    if (P.fcell && own) {
      const unsigned cc = ((unsigned)k * ny + gj) * nx + gi;
      F[0] += (Real)P.fcell[cc];
      F[1] += (Real)P.fcell[P.N + cc];
      F[2] += (Real)P.fcell[2 * P.N + cc];
    }
  };
  // f of the own column (other lanes load zeros) one plane ahead of its f-bar.
  // The loads go out in two groups between the faces: in one burst with those
  // of lam' they fill the memory pipeline and the wave stalls at issue.
  using Raw = RawLane<false, Real, Store>;
  const unsigned column = (unsigned)(gj * nx + gi), nxy = (unsigned)nx * (unsigned)ny;
  auto load_part = [&](auto X, auto Y, int k, Raw& raw) {
    raw.template load<decltype(X)::value, decltype(Y)::value>(
        bin, LaneOffsets<false, Store>(column, (unsigned)P.N, 0).where(own, true, span), (unsigned)k * nxy,
        (unsigned)P.N);
  };
  using L0 = std::integral_constant<int, 0>;
  using L1 = std::integral_constant<int, 10>;
  using L2 = std::integral_constant<int, Q>;
  Raw fpre;
  load_part(L0{}, L2{}, (z0 + 1) % nz, fpre);

  // ---- pre-loop: f-bar at z0-1 and z0 ----
  {
    Raw lo, hi;
    const int km = (z0 - 1 + nz) % nz;
    load_part(L0{}, L2{}, km, lo);
    load_part(L0{}, L2{}, z0, hi);
    Real F[3], ff[Q], rho, u0[3];
    force_own(km, F);
    lo.template decode<false>(P, Real(1), ff, rho, u0);
    centre_fbar<Real>(ff, rho, u0, F, hdt, (Real)P.bw0, (Real)P.bw2, fbn);
    force_own(z0, F);
    hi.template decode<false>(P, Real(1), ff, rho, u0);
    centre_fbar<Real>(ff, rho, u0, F, hdt, (Real)P.bw0, (Real)P.bw2, fbc);
    static_for<5>([&](auto K) {
      constexpr int k = decltype(K)::value;
      fbm[k] = fbn[ZP[k]];
    });
  }

  // The wall ghost that the lane's column extrapolates (the column at the wall
  // does, from itself and the next one, which is in the same wave: rows in
  // pairs, halo columns in one wave), as q f(1) + (1 - q) f(2) taken as f(2) +
  // q (f(1) - f(2)).  Z and Zn are linear in f-bar+ with weights shared by the
  // columns, so their ghosts extrapolate as f-bar+ does.  At most one wall axis.
  static_assert(TX * TY % 64 == 0 && 64 / TX % 2 == 0 && T::NROW % 64 + T::NHALO <= 64, "columns of a wave");
  const bool xin = own && !P.periodic[0] && c >= 0 && c < TX, yin = own && !P.periodic[1] && r >= 1 && r <= TY;
  const int gdx = !xin ? 0 : (gi == 0 ? -1 : (gi == nx - 1 ? 1 : 0));
  const int gdy = !yin ? 0 : (gj == 0 ? -1 : (gj == ny - 1 ? 1 : 0));
  const Real gqx = gdx < 0 ? uniform((Real)P.qlo[0]) : uniform((Real)P.qhi[0]);
  const Real gqy = gdy < 0 ? uniform((Real)P.qlo[1]) : uniform((Real)P.qhi[1]);

  // compact adjoint-face records with the state stored in the arithmetic
  // type (FP32 or FP64): rho and j of every cell
  // for the gather, written by the interior lanes from the prefetched f.
  // A chunk writes its planes z0+1 .. zend (mod nz), so the chunks cover
  // every plane once.
  auto store_moments = [&](int k, Real rho, const Real (&jm)[3]) {
    const Real rec[4] = {rho, jm[0], jm[1], jm[2]};
    cell_records<Real>(adj.faces, adj.mom, P.eN, P.N)
        .st4(rec, (unsigned)(((long long)k * ny + gj) * nx + gi) * (unsigned)(4 * sizeof(Real)));
  };
  // One plane p: fbc / lamc hold f-bar+ and lam' of plane p, and the plane
  // computes those of p + 1 into fbn / lamn.
  // (Parameters, not captures: captured arrays that the loop also copies stay
  // in scratch memory, 3.8 against 2.7 ms an adjoint step on 256x192x256.)
  auto plane = [&](int p, Real (&fbc)[Q], Real (&fbn)[Q], Real (&lamc)[Q], Real (&lamn)[Q]) {
    const int kn = (p + 1) % nz;
    {
      Real F[3];
      force_own(kn, F);
      Real ff[Q], rho, u0[3];
      fpre.template decode<false>(P, Real(1), ff, rho, u0);
      if constexpr (COMPACT && std::is_same<Store, Real>::value) {
        if (interior) {
          Real jm[3];
          cell_moments<Real>(ff, rho, jm);
          store_moments(kn, rho, jm);
        }
      }
      centre_fbar<Real>(ff, rho, u0, F, hdt, (Real)P.bw0, (Real)P.bw2, fbn);
    }
    load_lam(kn, lamn);
    load_flow(kn, rnn, jnn);
    // ---- phase 1: Z(p) (tangential z-lerp of f-bar(p)) and Zn(p+1/2) ----
    Real zt[Q], zn[Q];
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      constexpr int cz = CZ[ip];
      if constexpr (cz == 0) {
        zt[ip] = fbc[ip];
      } else if constexpr (cz > 0) {
        constexpr int zk = ip == 5 ? 0 : (ip == 11 ? 1 : (ip == 12 ? 2 : (ip == 15 ? 3 : 4)));
        zt[ip] = lerp_(fbc[ip], fbm[zk], wzt_p);
      } else {
        zt[ip] = lerp_(fbc[ip], fbn[ip], wzt_m);
      }
      if constexpr (ip == 0)
        zn[0] = Real(0.5) * (fbc[0] + fbn[0]);
      else
        zn[ip] = lerp_(fbc[ip], fbn[ip], wzn[cz + 1]);
    });
    if (own) {
      static_for<Q>([&](auto I) {
        constexpr int ip = decltype(I)::value;
        A[ip][ia(r, c + 1)] = zt[ip];
        An[ip][ia(r, c + 1)] = zn[ip];
      });
    }
    if (gdx != 0 || gdy != 0) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const int g = ia(r + gdy, c + 1 + gdx), i2 = ia(r - gdy, c + 1 - gdx);
      const Real q = gdx != 0 ? gqx : gqy;
      static_for<Q>([&](auto I) {
        constexpr int ip = decltype(I)::value;
        const Real a2 = A[ip][i2], n2 = An[ip][i2];
        A[ip][g] = fma_rn(q, zt[ip] - a2, a2);
        An[ip][g] = fma_rn(q, zn[ip] - n2, n2);
      });
    }
    if (active) {
      static_for<Q>([&](auto I) {
        constexpr int ip = decltype(I)::value;
        if constexpr (ip != 0) Lam[ip][ia(r, c + 1)] = lamc[ip];
      });
    }
    __syncthreads();
    // ---- phase 2: the faces of plane p (-x, -y from Z; +z from Zn) ----
    // the tile's right and top boundary faces are the next tile's, except at a wall
    const bool xhalo = active && t >= T::NROW && c == TX && r >= 1 && r <= TY;
    const bool do_x = interior || (xhalo && !P.periodic[0] && gi == nx);
    const bool do_y = t < T::NROW && r >= 1 && (r <= TY || (!P.periodic[1] && gj == ny));
    if (do_x) {
      // face between x-columns gi-1 (left, ghost-inclusive index mi-1) and gi
      Face<Real, 0> fc;
      static_for<Q>([&](auto I) {
        constexpr int ip = decltype(I)::value;
        constexpr int cx = CX[ip], cy = CY[ip];
        if constexpr (ip == 0) {
          fc.template put<0>(Real(0.5) * (A[0][ia(r, c)] + A[0][ia(r, c + 1)]));
        } else {
          const Real w = xn(cx + 1);  // fraction toward the right cell
          Real v = lerp_(A[ip][ia(r, c)], A[ip][ia(r, c + 1)], w);
          if constexpr (cy != 0) {
            const Real wy = yt(cy < 0 ? 0 : 1);
            const Real v2 = lerp_(A[ip][ia(r - cy, c)], A[ip][ia(r - cy, c + 1)], w);
            v = lerp_(v, v2, wy);
          }
          fc.template put<ip>(v);
        }
      });
      const bool lw = !P.periodic[0] && gi == 0, hw = !P.periodic[0] && gi == nx;
      if (!P.periodic[0]) fc.bounce(lw, hw);
      const Real uL = WX[5][c], uR = WX[5][c + 1];
      Real mu[10], lam[Q];
      static_for<10>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = XD[k];
        mu[k] = Real(CX[ip]) * (uR * Lam[ip][ia(r, c + 1)] - uL * Lam[ip][ia(r, c)]);
      });
      // (no "cond ? nx : gi": the optimiser turns a select between two
      // captured variables into a select between their addresses, which
      // keeps them in scratch memory)
      const int slot = gi + ((gi == 0 && P.periodic[0]) ? nx : 0);
      const long long fs = ((long long)(p + 1) * e1 + (gj + 1)) * e0 + slot;
      if constexpr (COMPACT) {
        Real Ac, B[3];
        fc.template adjoint_coeffs<FADJ>(Famb, hdt, fw0, fw2, mu, Ac, B, fsum);
        store_compact(0, fs, Ac, B);
      } else {
        fc.template adjoint<FADJ>(Famb, hdt, fw0, fw1, fw2, mu, lw, hw, lam, fsum);
        store_face(0, fs, lam);
      }
    }
    const int kp = (p + 2) % nz;
    load_part(L0{}, L1{}, kp, fpre);
    if (do_y) {
      // face between y-rows gj-1 (below) and gj
      Face<Real, 1> fc;
      static_for<Q>([&](auto I) {
        constexpr int ip = decltype(I)::value;
        constexpr int cx = CX[ip], cy = CY[ip];
        if constexpr (ip == 0) {
          fc.template put<0>(Real(0.5) * (A[0][ia(r - 1, c + 1)] + A[0][ia(r, c + 1)]));
        } else {
          const Real w = yn(cy + 1);  // fraction toward the upper cell
          Real lo = A[ip][ia(r - 1, c + 1)], hi = A[ip][ia(r, c + 1)];
          if constexpr (cx != 0) {
            const Real wx = xt(cx < 0 ? 0 : 1);
            lo = lerp_(lo, A[ip][ia(r - 1, c + 1 - cx)], wx);
            hi = lerp_(hi, A[ip][ia(r, c + 1 - cx)], wx);
          }
          fc.template put<ip>(lerp_(lo, hi, w));
        }
      });
      const bool lw = !P.periodic[1] && gj == 0, hw = !P.periodic[1] && gj == ny;
      if (!P.periodic[1]) fc.bounce(lw, hw);
      const Real uL = WY[5][r - 1], uR = WY[5][r];
      Real mu[10], lam[Q];
      static_for<10>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = YD[k];
        mu[k] = Real(CY[ip]) * (uR * Lam[ip][ia(r, c + 1)] - uL * Lam[ip][ia(r - 1, c + 1)]);
      });
      const int slot = gj + ((gj == 0 && P.periodic[1]) ? ny : 0);
      const long long fs = ((long long)(p + 1) * e1 + slot) * e0 + (gi + 1);
      if constexpr (COMPACT) {
        Real Ac, B[3];
        fc.template adjoint_coeffs<FADJ>(Famb, hdt, fw0, fw2, mu, Ac, B, fsum);
        store_compact(1, fs, Ac, B);
      } else {
        fc.template adjoint<FADJ>(Famb, hdt, fw0, fw1, fw2, mu, lw, hw, lam, fsum);
        store_face(1, fs, lam);
      }
    }
    load_part(L1{}, L2{}, kp, fpre);
    // lam' of plane p+1 complete (its loads were issued in phase 1)
    if constexpr (kFlowFuse) add_flow(lamn, rnn, jnn);
    Real zA = Real(0), zB[3] = {Real(0), Real(0), Real(0)};
    const long long zs = ((long long)(p + 1) * e1 + (gj + 1)) * e0 + (gi + 1);
    if (interior) {
      // +z face of the cell: between planes p and p+1 (z is periodic)
      Face<Real, 2> fc;
      zface_rec(fc);
      Real mu[10], lam[Q];
      static_for<10>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = ZD[k];
        mu[k] = Real(CZ[ip]) * updz * (lamn[ip] - lamc[ip]);
      });
      if constexpr (COMPACT) {
        fc.template adjoint_coeffs<FADJ>(Famb, hdt, fw0, fw2, mu, zA, zB, fsum);
      } else {
        fc.template adjoint<FADJ>(Famb, hdt, fw0, fw1, fw2, mu, false, false, lam, fsum);
        store_face(2, zs, lam);
      }
    }
    // without a branch: the next plane's wait for the loads above does not cover it
    if constexpr (COMPACT) store_compact(2, zs, zA, zB, interior);
    __syncthreads();
    static_for<5>([&](auto K) {
      constexpr int k = decltype(K)::value;
      fbm[k] = fbc[ZP[k]];
    });
  };
  for (int p = z0; p < zend; p++) {
    plane(p, fbc, fbn, lamc, lamn);
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      fbc[ip] = fbn[ip];
      if constexpr (ip != 0) lamc[ip] = lamn[ip];
    });
  }

  if constexpr (FADJ) {
    // the flow-axis component (assigned, not selected as an lvalue: a select
    // between array elements can keep the array in scratch memory)
    double v[1] = {fsum[0]};
    if (as == 1) v[0] = fsum[1];
    if (as == 2) v[0] = fsum[2];
    constexpr int kSum[1] = {0};
    block_reduce<1, T::NT>(v, kSum);
    if (t == 0) partial[tt] = v[0];
  }
}

#include "step_kernel.h"

// z-chunk length of the adjoint-face pass (plan_z_chunks; a chunk recomputes
// f-bar+ of the two planes before it, about as long as one plane).  At most
// 32 planes: several rounds even out the finish (256x192x256 FP32: 128 planes
// 0.3 % slower).  On 64x64x32 FP64 (32 tiles, one workgroup per CU) 4-plane
// chunks took 51 us where 8-plane ones took 86.
int blocks_per_cu(bool fp64, int TX, int TY) { return fp64 || Tile_nt(TX, TY) > 256 ? 1 : 2; }
int z_chunk(const Ctx& cx, int TX, int TY) {
  const long long cols = (long long)(cx.kp.n[0] / TX) * (cx.kp.n[1] / TY);
  const int nz = cx.kp.n[2], nc = plan_z_chunks(cols, nz, 256 * blocks_per_cu(cx.precision == 0, TX, TY), 1.2,
                                                  (cx.kp.n[2] + 31) / 32);
  return (nz + nc - 1) / nc;
}

}  // namespace

// Tiles of 32 x 12 cells with FP32 arithmetic and 16 x 12 with FP64 are the
// tallest whose two LDS planes and face values fit 160 KB: one workgroup of
// eight waves per CU, f-bar+ formed on 1.24 and 1.31 times the cells.  (FP32
// on 16 x 12, two workgroups per CU: 0.80 against 0.68 ms on the 256x192x256
// channel.)
// A plane takes the same time whatever the grid, and the start of a tile or
// chunk about 2.2 planes' time (f-bar+ of two planes and one face).  So a
// round of 256 workgroups costs the planes of the longest one + 2.2, and the
// plan is the cheapest of these (times are those of a run of steps over their
// number; event pairs around a launch read about 2.5 us more):
//  - z-chunks of every tile (plan_z_chunks).  64x64x32 FP64 (24 tiles): 8
//    chunks 30.5 us, 16 36.6, 32 39.4; 64x72x32 FP32 (12 tiles): 8 chunks
//    28.0 us, 16 20.3, 32 24.3;
//  - the same with lower tiles, whose plane takes 0.88 (8 rows) or 0.62 to
//    0.66 (4 rows) of the time: 8 rows where they fill more CUs (64x64x32 FP64
//    25.2 us against 28.0), 4 rows where a workgroup has a single plane
//    (8x64x8 FP64 10.0 against 12.7 us, 20x20x20 FP64 9.5 against 12.5);
//    elsewhere they lose (90x50x121 FP64 88.7, 96.9 and 131 us);
//  - full chunks and runs over what they leave, in one round, where no chunk
//    count fills the last round: 128^3 FP64 (88 tiles: 2 chunks of 46 planes
//    each, and 80 workgroups with 39 or 40 planes of the rest, against 3 rounds
//    of 16 planes) 242 us against 251, FP32 (44 tiles: 5 chunks of 23, 36
//    workgroups with 16, against 26 planes) 115 against 123, FP16
//    non-equilibrium storage 142 against 158.  (Runs over all planes put
//    neighbouring tiles out of step, so that their halos miss L2: 263 us in
//    FP64 and 137 in FP32.)  Only where the model gives 7 %: at 5 % a
//    150x97x83 FP32 channel gained 2 % and a 90x50x121 FP64 duct lost 3.
// Gradient reconstruction takes the first two forms (its kernel has no registers
// left for the runs).  Periodic, us a step with 12, 8 and 4 rows: 64x32x2 FP32
// 13.8, 12.5 and 10.4; 64x64x32 FP32 21.6, 19.5 and 22.6, FP64 31.3, 26.6 and 31.8;
// 96x96x16 FP32 22.9, 23.9 and 28.7.
StepPlan step_plan(const Setup& s, int precision) {
  const int tx = precision == 0 ? 16 : 32, nz = s.n[2];
  const double start = 2.2;
  StepPlan best{};
  double least = 0;
  for (const int rows : {12, 8, 4}) {
    const double plane = rows == 12 ? 1.0 : (rows == 8 ? 0.88 : (precision == 0 ? 0.62 : 0.66));
    const long long tiles = (long long)((s.n[0] + tx - 1) / tx) * ((s.n[1] + rows - 1) / rows);
    const int nc = plan_z_chunks(tiles, nz, 256, start);
    const double cost = plane * (double)((tiles * nc + 255) / 256) * ((nz + nc - 1) / nc + start);
    if (rows == 12 || cost < 0.97 * least) {
      best = {rows, nc, 0, tiles * nc};
      least = cost;
    }
    if (rows != 12 || s.recon != 0) continue;
    const double chunks = 0.93 * least;
    for (int m = 1; m * tiles < 256; m++)
      for (int len = 1; m * len < nz && len + start < chunks; len++) {
        const int rest = nz - m * len;
        const long long nb = 256 - m * tiles, run = (rest * tiles + nb - 1) / nb;
        const double cost_runs = std::max(len + start, run + start * ((run + rest - 2) / rest + 1));
        // (at a tie more chunks, which keep neighbouring tiles in step)
        if (cost_runs < chunks && (cost_runs < least || (best.len > 0 && cost_runs <= least))) {
          best = {12, m, len, 256};
          least = cost_runs;
        }
      }
  }
  return best;
}

namespace {

template <class Real, class Store, int TX, int TY, bool GRAD, bool RUNS, bool FLAT>
hipError_t run_step(Ctx& cx, const void* fin, void* fout, const StepPlan& plan) {
  using T = StepTile<Real, TX, TY, GRAD>;
  FlowLaw law{};
  if (cx.s.flow_rate != 0 && !cx.flow_frozen) {
    const Setup& s = cx.s;
    if ((size_t)plan.nblocks > cx.flow_partial_len) return hipErrorInvalidValue;
    law = {cx.flow_partial, reinterpret_cast<unsigned*>(cx.famb_dev + kFambArrived), cx.famb_dev,
           s.width[0] * s.width[1] * s.width[2], s.flow_rate, s.flow_gain, s.dt};
  }
  if (cx.timing) hipEventRecord(cx.tev[0], cx.stream);
  hipLaunchKernelGGL((k_step<Real, Store, TX, TY, GRAD, RUNS, FLAT>), dim3((unsigned)plan.nblocks), dim3(T::NT), 0, cx.stream,
                     cx.kp, static_cast<const Store*>(fin), static_cast<Store*>(fout), plan.nchunk, plan.len, law);
  if (cx.timing) hipEventRecord(cx.tev[1], cx.stream);
  cx.launches_per_step = 1;
  return hipGetLastError();
}

template <int TX, int TY>
dim3 adj_faces_grid(const Ctx& cx, int* TZ) {
  const KParams& P = cx.kp;
  *TZ = z_chunk(cx, TX, TY);
  return dim3(P.n[0] / TX, P.n[1] / TY, (P.n[2] + *TZ - 1) / *TZ);
}

// FADJ: also the per-block force partials into fpart (nparts of them).
template <class Real, class Store, int TX, int TY, bool COMPACT = false, class LamT = double, bool FADJ = false>
hipError_t run_adj_faces(Ctx& cx, const void* f, const void* lam, void* faces, double* fpart = nullptr,
                         long long fpart_len = 0, long long* nparts = nullptr, int mom = 0,
                         const double* ubar = nullptr) {
  const KParams& P = cx.kp;
  using T = Tile<TX, TY>;
  int TZ = 0;
  const dim3 grid = adj_faces_grid<TX, TY>(cx, &TZ);
  if constexpr (FADJ) {
    const long long nb = (long long)grid.x * grid.y * grid.z;
    if (nb > fpart_len) return hipErrorInvalidValue;
    *nparts = nb;
  }
  hipLaunchKernelGGL((k_adj_tile_faces<Real, Store, TX, TY, COMPACT, LamT, FADJ>), grid, dim3(T::NT), 0, cx.stream, P,
                     static_cast<const Store*>(f), TZ, FADJ ? fpart : nullptr,
                     AdjFaceIO{lam, faces, mom, ubar, 1.0 / (cx.s.width[0] * cx.s.width[1] * cx.s.width[2])});
  return hipGetLastError();
}

}  // namespace

namespace {
// What the tile kernels need of the grid, whatever its size.  Either
// reconstruction (gradient reconstruction needs uniform axes, which the
// configuration enforces).
bool tiles_cover(const Ctx& c) {
  const Setup& s = c.s;
  if (!s.periodic[2] || !s.uniform[2]) return false;
  // buffer offsets are 32-bit: one state array must span < 4 GiB
  if ((double)c.state_bytes >= 4294967296.0) return false;
  // a wall axis needs two interior cells per side of the extrapolation
  return (s.periodic[0] || s.n[0] >= 3) && (s.periodic[1] || s.n[1] >= 3);
}
}  // namespace

// Grids of whole tiles: what DUGKS_KERNEL_FUSED asks for and the adjoint-face
// pass needs (trilinear reconstruction there).
bool fused_supported(const Ctx& c, int* tx, int* ty) {
  const Setup& s = c.s;
  // Tiles of the adjoint-face pass, 4 waves: 16 x 12 cells when the grid
  // divides (1.31 f-bar evaluations per cell, the x-halo lanes packed behind
  // the rows), else 32 x 4 (1.59 per cell, the last wave holding only the 12
  // x-halo lanes).  Four waves per block keep FP64 at one wave per SIMD
  // without spills and fit two FP32 blocks (at most 256 registers per lane)
  // on a CU.
  if (s.n[0] % 16 == 0 && s.n[1] % 12 == 0) {
    *tx = 16;
    *ty = 12;
  } else {
    *tx = 32;
    *ty = 4;
  }
  return s.n[0] % *tx == 0 && s.n[1] % *ty == 0 && tiles_cover(c);
}

namespace {
// The step kernel takes any nx and ny (the last tile of an axis overlaps the
// one before it), and the automatic choice uses it wherever it can: on 90x50x121
// FP64 in a duct 89 us a step against 525 with the two-pass kernels, on a
// 150x97x83 FP32 channel 90 against 301, on 8x64x8 FP64 12.7 against 89, on
// 20x20x20 FP64 12.5 against 100.  Below 512 cells, grids that are not whole
// tiles keep the two-pass kernels although these are slower there too
// (13x6x5 FP64: 69 against 10.5 us): that choice is part of the tested
// interface, and no run of use is that small.
bool step_covers(const Ctx& c) {
  int tx, ty;
  if (fused_supported(c, &tx, &ty)) return true;
  return c.kernel != 1 /* DUGKS_KERNEL_FUSED */ && tiles_cover(c) && c.kp.N >= 512;
}

template <class Real, class Store, bool GRAD, bool FLAT>
hipError_t run_step_rows(Ctx& c, const void* fin, void* fout) {
  constexpr int TX = sizeof(Real) == 8 ? 16 : 32;
  if (c.plan.rows == 12) return run_step<Real, Store, TX, 12, GRAD, false, FLAT>(c, fin, fout, c.plan);
  if (c.plan.rows == 8) return run_step<Real, Store, TX, 8, GRAD, false, FLAT>(c, fin, fout, c.plan);
  return run_step<Real, Store, TX, 4, GRAD, false, FLAT>(c, fin, fout, c.plan);
}

template <class Real, class Store>
hipError_t launch_step_mode(Ctx& c, const void* fin, void* fout) {
  constexpr int TX = sizeof(Real) == 8 ? 16 : 32;
  if (c.s.recon != 0)
    return c.s.n[2] == 1 ? run_step_rows<Real, Store, true, true>(c, fin, fout)
                         : run_step_rows<Real, Store, true, false>(c, fin, fout);
  if (c.plan.len > 0) return run_step<Real, Store, TX, 12, false, true, false>(c, fin, fout, c.plan);
  return run_step_rows<Real, Store, false, false>(c, fin, fout);
}
}  // namespace

hipError_t launch_step_fused(Ctx& c, const void* fin, void* fout, bool* handled) {
  *handled = step_covers(c);
  if (!*handled) return hipSuccess;
  switch (c.precision) {
    case 0:
      return launch_step_mode<double, double>(c, fin, fout);
    case 1:
      return launch_step_mode<float, float>(c, fin, fout);
    case 2:
      return launch_step_mode<float, __half>(c, fin, fout);
    default:
      return launch_step_mode<float, NeqHalf>(c, fin, fout);
  }
}

bool adjoint_faces_fused_covers(const Ctx& c) {
  int tx = 32, ty = 4;
  // the adjoint does not cover FP16 non-equilibrium storage or the gradient
  // reconstruction
  if (c.kernel == 0 || c.precision == 3 || c.s.recon != 0 || !fused_supported(c, &tx, &ty)) return false;
  // lam' and each face array are addressed with 32-bit buffer offsets
  const double rb = c.precision == 0 ? 8.0 : 4.0;
  return (double)Q * c.kp.N * 8.0 < 2147483648.0 && (double)Q * c.kp.eN * rb < 2147483648.0;
}

namespace {
// Tiles of the adjoint-face pass: 0 = 32 x 4, 1 = 16 x 12, 2 = 32 x 12.
// Compact records go with the z-marching gather (nx % 32 == 0).  With FP32
// arithmetic their rows must be whole 128-byte lines, so 32-wide: 16 x 12
// tiles (half-line stores) took the adjoint step with FP32 lam to 2.92 ms on
// the 256x192x256 channel against 2.76 on 32 x 4, and 32 x 12 tiles (one
// workgroup of 8 waves per CU, f-bar+ on 1.24x the cells instead of 1.59x,
// 93 % of the lanes busy) bring it to 2.60 where ny % 12 == 0.  Both lam
// forms take the same tiles, so the same kernel code gives the same bits
// for a lam' that FP32 holds exactly.  With FP64 arithmetic 16 doubles are a
// whole line, and 16 x 12 tiles serve every format where the grid divides
// (FP64 adjoint step 5.88 against 6.61 ms on 32 x 4).  FP32 full records
// take the step's tiles.
int adj_tile(const Ctx& c, int format, int tx) {
  const bool compact32 = c.precision != 0 && format != kFacesFull;
  if (compact32) return c.kp.n[1] % 12 == 0 ? 2 : 0;
  return tx == 16 ? 1 : 0;
}
}  // namespace

hipError_t launch_adjoint_faces_fused(Ctx& c, const void* f, const void* lam, void* faces, int format,
                                      bool* handled, double* fpart, long long fpart_len, long long* nparts, int mom,
                                      const double* ubar) {
  int tx = 32, ty = 4;
  *handled = false;
  if (!adjoint_faces_fused_covers(c) || (format == kFacesCompactLam32 && c.precision == 0)) return hipSuccess;
  fused_supported(c, &tx, &ty);
  *handled = true;
  const int tile = adj_tile(c, format, tx);
  const bool tall = tile == 1, wide = tile == 2;
  if (fpart) {
    // with the ambient-force cotangent: the formats of the forward-adjoint
    // sweep (FP64, and FP32 arithmetic with lam in FP32)
    if (c.precision == 0 && format == kFacesFull)
      return tall ? run_adj_faces<double, double, 16, 12, false, double, true>(c, f, lam, faces, fpart, fpart_len,
                                                                                nparts)
                  : run_adj_faces<double, double, 32, 4, false, double, true>(c, f, lam, faces, fpart, fpart_len,
                                                                               nparts);
    if (c.precision == 0 && format == kFacesCompact)
      return tall ? run_adj_faces<double, double, 16, 12, true, double, true>(c, f, lam, faces, fpart, fpart_len,
                                                                               nparts, mom, ubar)
                  : run_adj_faces<double, double, 32, 4, true, double, true>(c, f, lam, faces, fpart, fpart_len,
                                                                              nparts, mom, ubar);
    if (c.precision == 1 && format == kFacesCompactLam32)
      return wide ? run_adj_faces<float, float, 32, 12, true, float, true>(c, f, lam, faces, fpart, fpart_len,
                                                                            nparts, mom, ubar)
                  : run_adj_faces<float, float, 32, 4, true, float, true>(c, f, lam, faces, fpart, fpart_len,
                                                                           nparts, mom, ubar);
    if (c.precision == 2 && format == kFacesCompactLam32)
      return wide ? run_adj_faces<float, __half, 32, 12, true, float, true>(c, f, lam, faces, fpart, fpart_len,
                                                                             nparts)
                  : run_adj_faces<float, __half, 32, 4, true, float, true>(c, f, lam, faces, fpart, fpart_len,
                                                                            nparts);
    return hipErrorNotSupported;
  }
  switch (c.precision) {
    case 0:
      if (format == kFacesCompact)
        return tall ? run_adj_faces<double, double, 16, 12, true>(c, f, lam, faces, nullptr, 0, nullptr, mom)
                    : run_adj_faces<double, double, 32, 4, true>(c, f, lam, faces, nullptr, 0, nullptr, mom);
      return tall ? run_adj_faces<double, double, 16, 12>(c, f, lam, faces)
                  : run_adj_faces<double, double, 32, 4>(c, f, lam, faces);
    case 1:
      if (format == kFacesCompactLam32)
        return wide ? run_adj_faces<float, float, 32, 12, true, float>(c, f, lam, faces, nullptr, 0, nullptr, mom)
                    : run_adj_faces<float, float, 32, 4, true, float>(c, f, lam, faces, nullptr, 0, nullptr, mom);
      if (format == kFacesCompact)
        return wide ? run_adj_faces<float, float, 32, 12, true>(c, f, lam, faces, nullptr, 0, nullptr, mom)
                    : run_adj_faces<float, float, 32, 4, true>(c, f, lam, faces, nullptr, 0, nullptr, mom);
      return tall ? run_adj_faces<float, float, 16, 12>(c, f, lam, faces)
                  : run_adj_faces<float, float, 32, 4>(c, f, lam, faces);
    default:
      if (format == kFacesCompactLam32)
        return wide ? run_adj_faces<float, __half, 32, 12, true, float>(c, f, lam, faces)
                    : run_adj_faces<float, __half, 32, 4, true, float>(c, f, lam, faces);
      if (format == kFacesCompact)
        return wide ? run_adj_faces<float, __half, 32, 12, true>(c, f, lam, faces)
                    : run_adj_faces<float, __half, 32, 4, true>(c, f, lam, faces);
      return tall ? run_adj_faces<float, __half, 16, 12>(c, f, lam, faces)
                  : run_adj_faces<float, __half, 32, 4>(c, f, lam, faces);
  }
}

long long adjoint_faces_fused_blocks(const Ctx& c, int format) {
  int tx = 32, ty = 4, TZ = 0;
  if (!fused_supported(c, &tx, &ty)) return 0;
  const int tile = adj_tile(c, format, tx);
  const dim3 g = tile == 1 ? adj_faces_grid<16, 12>(c, &TZ)
                           : (tile == 2 ? adj_faces_grid<32, 12>(c, &TZ) : adj_faces_grid<32, 4>(c, &TZ));
  return (long long)g.x * g.y * g.z;
}

}  // namespace dugks
