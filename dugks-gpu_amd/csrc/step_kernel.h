// The step kernel.  Included by step_fused.hip inside namespace
// dugks { namespace { ... } }, after step_common.h.
#pragma once

// Columns of a tile (with its halo) a wave holds, waves and threads of its workgroup.
constexpr int step_unit(bool pair) { return pair ? 32 : 64; }
constexpr int step_nw(bool pair, int TX, int TY) {
  return ((TY + 2) * (TX + 2) + step_unit(pair) - 1) / step_unit(pair);
}

// The flow-rate controller: where the workgroups leave their parts of the sum
// over cells of u dV of the new state (nullptr: no controller), and how many
// have; the force and the controller's state (flow_update), and its constants.
struct FlowLaw {
  double* partial;
  unsigned* arrived;
  double* famb;
  double volume, target, gain, dt;
};
template <class Real, int TX, int TY, bool GRAD>
struct StepTile {
  static constexpr bool PAIR = sizeof(Real) == 8;
  static constexpr int NQ = lane_slots(PAIR), NX = lane_crossings(PAIR);
  static constexpr int AC = TX + 2;
  static constexpr int NROW = (TY + 2) * TX;         // the tile rows and the two y-halo rows
  static constexpr int NSLOT = NROW + 2 * (TY + 2);  // and the two x-halo columns
  static constexpr int UNIT = step_unit(PAIR);
  static constexpr int NW = step_nw(PAIR, TX, TY), NT = NW * 64;
  static constexpr int NWI = TX * TY / UNIT;         // waves that hold the tile's own columns
  static_assert(TX * TY % UNIT == 0 && UNIT % TX == 0, "whole rows in a wave");
  // LDS of one lane half: NPL planes of positions (GRAD: the ring of f-bar+
  // at p-1, p, p+1; else Z(p) and Zn(p+1/2)), then the crossing populations
  // of the -x and -y faces (position of the cell above the face)
  static constexpr int STR = lds_stride(PAIR);
  static constexpr int FS = PAIR ? (GRAD ? 5 : 6) : 12;
  static constexpr int AP = (TY + 2) * AC * STR;
  static constexpr int NPL = GRAD ? 3 : 2;
  static constexpr int OX = NPL * AP - AC * FS;       // -x faces: rows 1..TY
  static constexpr int OY = OX + TY * AC * FS;        // -y faces: rows 1..TY+1
  static constexpr int REG = (OY + (TY + 2) * AC * FS + 3) / 4 * 4;
  static constexpr int NH = PAIR ? 2 : 1;
  static constexpr int kW = 6;                        // weights per tile column and row
};

// One DUGKS step fin -> fout (see the top of step_fused.hip).  The grid is
// one-dimensional: nchunk z-chunks of gx gy tiles.  RUNS: chunks of `len`
// planes, which leave the last nz - nchunk len planes of every tile; these, one
// tile after the other, are dealt in equal runs to the workgroups behind, and
// such a workgroup goes from the planes of one tile to those of the next.  (A
// template argument: the loop over the runs costs registers.)  FLAT: the grid has
// one plane, so a cell's two z-faces have the same flux, whose difference the
// update would take; neither is formed.  (Gradient reconstruction, 1024x768x1
// FP32: 94 us a step, before 107, the kernel before that 96.)
template <class Real, class Store, int TX, int TY, bool GRAD, bool RUNS, bool FLAT>
__global__ void __launch_bounds__(step_nw(sizeof(Real) == 8, TX, TY) * 64, 2)
    k_step(KParams P, const Store* __restrict__ fin, Store* __restrict__ fout, int nchunk,
           int len, FlowLaw law) {
  using T = StepTile<Real, TX, TY, GRAD>;
  constexpr bool PAIR = T::PAIR;
  constexpr int NQ = T::NQ, NX = T::NX, AC = T::AC, STR = T::STR, FS = T::FS, UNIT = T::UNIT;
  // FP16 non-equilibrium storage steps the shifted populations h = f - w
  // (EqShift), decoded from and encoded to the stored rho - 1, u and
  // non-equilibrium part without forming f
  constexpr bool kNeq = std::is_same<Store, NeqHalf>::value;
  constexpr bool kShift = kNeq;
  __shared__ __align__(16) Real S[T::NH * T::REG];
  __shared__ Real WX[T::NH][T::kW][TX + 2];
  __shared__ Real WY[T::NH][T::kW][TY + 2];

  const int nx = P.n[0], ny = P.n[1], nz = P.n[2];
  const int t = threadIdx.x;
  // XCD-aware tile order: workgroup b runs on XCD b % 8; each XCD gets a
  // contiguous run of tiles (x fastest), so that tiles whose halos overlap
  // share an L2 and run at about the same time
  const int gx = (nx + TX - 1) / TX, gy = (ny + TY - 1) / TY;
  const int nblocks = (int)gridDim.x, b = blockIdx.x, xcd = b % kXcds;
  const int tt = xcd * (nblocks / kXcds) + min(xcd, nblocks % kXcds) + b / kXcds;
  // the workgroup's planes q0..q1-1, plane zb + z of tile k counted as k per + z
  int q0, q1, per = nz, zb = 0;
  const int tiles = gx * gy;
  if (!RUNS || tt < tiles * nchunk) {
    const int tile = tt % tiles, bz = tt / tiles;
    q0 = tile * nz + (RUNS ? bz * len : (int)((long long)bz * nz / nchunk));
    q1 = RUNS ? q0 + len : tile * nz + (int)((long long)(bz + 1) * nz / nchunk);
  } else {
    zb = nchunk * len;
    per = nz - zb;
    const long long k = tt - tiles * nchunk, nk = nblocks - tiles * nchunk, planes = (long long)tiles * per;
    q0 = (int)(k * planes / nk);
    q1 = (int)((k + 1) * planes / nk);
  }
  const unsigned N = (unsigned)P.N, nxy = (unsigned)nx * (unsigned)ny;
  const unsigned span = (unsigned)state_bytes<Store>((unsigned long long)P.N);
  const StateBuf<Store> bin(fin, span), bout(fout, span);

  // the lane's column in tile coordinates: r = 0..TY+1 (y = j0-1+r), c = -1..TX
  // (x = i0+c): the TY tile rows first (whole waves), then the two y-halo
  // rows, then the two x-halo columns
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lane = PAIR ? ((t >> 4) & 3) * 8 + (t & 7) : t & 63;  // column within the wave
  const int u = wave * UNIT + lane;
  int r, c;
  if (u < TY * TX) {
    r = u / TX + 1;
    c = u % TX;
  } else if (u < T::NROW) {
    const int v = u - TY * TX;
    r = v < TX ? 0 : TY + 1;
    c = v % TX;
  } else {
    const int v = u - T::NROW;
    r = v % (TY + 2);
    c = v < TY + 2 ? -1 : TX;
  }
  const int tw = min(TX, nx), th = min(TY, ny);  // columns and rows of a tile
  // on an axis shorter than the tile the far halo is at c = tw, r = th + 1
  const bool active = u < T::NSLOT && c <= tw && r <= th + 1;
  const bool interior = active && r >= 1 && r <= th && c >= 0 && c < tw;
  auto sign = [](int half) { return half ? Real(-1) : Real(1); };

  // uniform parameters in scalar registers; the lane's frame turns the sign
  // of the force terms, of the c_z = +1 slots' z weights and of c dt/d
  Real F0[3];
  ambient_force<Real>(P, F0);
  const Real F[3] = {uniform(F0[0]), uniform(F0[1]), uniform(F0[2])};
  const Real fw1 = uniform((Real)P.fw1), fw2 = uniform((Real)P.fw2), bw2 = uniform((Real)P.bw2);
  const Real hdt = uniform((Real)P.hdt), hh = uniform(Real(0.5) * (Real)P.hdt), fw0 = uniform((Real)P.fw0),
             bw0 = uniform((Real)P.bw0);
  auto tz = [&](int idx) { return tabv<Real>(P, 2, idx); };
  // z weights (uniform axis): tangential (toward p-1 for c_z > 0, p+1 for
  // c_z < 0: the same), normal toward p+1 for c_z = 0, +1, -1
  const Real wzt = uniform(tz(9 + 6)), wzn0 = uniform(tz(9 + 1));
  const Real wznp = uniform(tz(9 + 2)), wznm = uniform(tz(9 + 0)), updz = uniform(tz(9 + 8));
  // GRAD: h / d of the difference across a face, h / 4d of the difference of
  // the two-cell sums two rows apart
  Real gin[3] = {Real(0), Real(0), Real(0)}, gtn[3] = {Real(0), Real(0), Real(0)};
  if constexpr (GRAD) {
    for (int a = 0; a < 3; a++) {
      gin[a] = uniform((Real)(P.hdt / P.du[a]));
      gtn[a] = uniform((Real)(0.25 * P.hdt / P.du[a]));
    }
  }
  double flow = 0;
  const int as = P.flow_axis;

  for (int q = q0; q < q1;) {  // (the body is one run, not indented)
  const int tile = q / per, z0 = zb + q - tile * per, zend = RUNS ? min(zb + per, z0 + q1 - q) : z0 + q1 - q0;
  // the next run's first barrier: this run's last plane still reads the weights
  if (RUNS && q != q0) __syncthreads();
  q += zend - z0;
  const int bx = tile % gx, by = tile / gx;
  // the last tile of an axis that TX or TY does not divide starts early and
  // overlaps the one before it; the first cx0 columns and ry0 rows of it are
  // the other tile's to store
  const int i0 = min(bx * TX, nx - tw), j0 = min(by * TY, ny - th);
  const int cx0 = bx * TX - i0, ry0 = by * TY - j0;
  const bool stored = interior && c >= cx0 && r > ry0;
  int gi = i0 + c, gj = j0 - 1 + r;
  if (P.periodic[0]) gi = (gi + nx) % nx;
  if (P.periodic[1]) gj = (gj + ny) % ny;
  const bool own = active && gi >= 0 && gi < nx && gj >= 0 && gj < ny;
  // tiles beside a wall extrapolate the ghost columns behind it (fill_ghosts)
  const bool wall_tile = (!P.periodic[0] && (i0 == 0 || i0 + tw == nx)) ||
                         (!P.periodic[1] && (j0 == 0 || j0 + th == ny));
  // A lane's place in the tile, made opaque where it is used (`here`): the
  // addresses formed from it then do not live in registers across the plane
  // loop, where the compiler would otherwise keep several dozen
  const int half0 = PAIR ? (t >> 3) & 1 : 0, pos0 = r * AC + (c + 1);
  const int base0 = (half0 ? T::REG : 0) + pos0 * STR, fbase0 = (half0 ? T::REG : 0) + pos0 * FS;
  struct Place {
    int half, r, c, at, fat;  // at, fat: LDS index of the column's slots, of its -x and -y fluxes
  };
  auto place = [&]() {
    Place q;
    q.half = PAIR ? (here(t) >> 3) & 1 : 0;
    q.r = here(r);
    q.c = here(c);
    q.at = here(base0);
    q.fat = here(fbase0);
    return q;
  };
  // Weights of the tile's columns and rows, copied once into LDS, in each
  // half's frame.  Value k: 0-2 the -face normal weight toward the upper cell
  // of the slots with c = -1, 0, +1; 3-4 the tangential shift weights for c =
  // -1 and +1; 5 s dt/d.
  for (int v = t; v < T::NH * T::kW * (TX + 2 + TY + 2); v += T::NT) {
    const bool isx = v < T::NH * T::kW * (TX + 2);
    const int q0 = isx ? v : v - T::NH * T::kW * (TX + 2);
    const int n = isx ? TX + 2 : TY + 2;
    const int hf = q0 / (T::kW * n), k = q0 / n % T::kW, q = q0 % n;
    int g = isx ? i0 - 1 + q : j0 - 1 + q;
    const int na = isx ? nx : ny;
    if (P.periodic[isx ? 0 : 1]) g = (g + na) % na;
    const int m = min(g + 1, na + 1);
    // the table row's entry for this half: the minus lanes' velocities are -c
    const int e = k < 3 ? (hf ? 2 - k : k) : (k < 5 ? 6 + (hf ? 4 - k : k - 3) : 8);
    Real w = tabv<Real>(P, isx ? 0 : 1, (k < 3 ? max(m - 1, 0) : m) * 9 + e);
    if (k == 5 && hf) w = -w;
    (isx ? WX[hf][k][q] : WY[hf][k][q]) = w;
  }
  auto xw = [&](int half, int k, int c) { return WX[half][k][c + 1]; };
  auto yw = [&](int half, int k, int r) { return WY[half][k][r]; };

  // LDS position of a column (r, c), and of its -x and -y faces; in the lane's
  // frame the column upwind of c_x = +1 lies at -sx, the row at -sy
  auto at = [](int half, int pos) { return (half ? T::REG : 0) + pos * STR; };
  auto fat = [](int half, int pos) { return (half ? T::REG : 0) + pos * FS; };
  auto up_x = [](int half) { return half ? -STR : STR; };
  auto up_y = [](int half) { return half ? -AC * STR : AC * STR; };
  constexpr int AN = T::AP;  // from Z(p) to Zn(p+1/2)
  auto rslot = [](int k) { return ((k + 3) % 3) * T::AP; };  // GRAD: ring offset of plane k >= -1
  constexpr unsigned kAll = all_slots(PAIR);
  // Wall ghost columns of a plane from the two columns beside the wall,
  // q f(1) + (1 - q) f(2) taken as f(2) + q (f(1) - f(2)) (exact for
  // constants), by the lane of the column at the wall; a corner of two walls
  // extrapolates the ghosts.  Z and Zn are linear in f-bar+ with weights
  // shared by the columns, so their ghosts extrapolate as f-bar+ does
  // (src/dugks.cu:1234-1251 and the stretched form,
  // src/fortran/channel/src/dugks.cuf:365-374).  The second column's lane is
  // in the same wave (rows in pairs from row 1, x-halo columns in one wave),
  // whose LDS accesses are in order, so no barrier is needed, except above
  // an odd number of rows (ny < TY): split_y.  (A barrier and a pass of the
  // ghost lanes instead: 0.828 against 0.763 ms without walls on
  // 256x192x256 in FP32.)
  const bool split_y = !P.periodic[1] && j0 + th == ny && (th * TX) % UNIT != 0;
  auto wave_order = []() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  // the ghosts of one plane (two with TWO), fa and fb the column's own values there
  auto fill_ghosts = [&](auto TWO, int plane_a, const Real (&fa)[NQ], int plane_b, const Real (&fb)[NQ])
                         __attribute__((always_inline)) {
    wave_order();
    const Place w = place();
    const int gi = i0 + w.c, gj = j0 - 1 + w.r;
    // side of the column's ghost along x and y: -1, +1, or none (a halo column
    // at the wall, beside an overlapping tile, has its ghost outside the tile,
    // where nothing reads it)
    const bool xin = own && !P.periodic[0] && w.c >= 0 && w.c < tw, yin = own && !P.periodic[1] && w.r >= 1 && w.r <= th;
    const int dx = !xin ? 0 : (gi == 0 ? -1 : (gi == nx - 1 ? 1 : 0));
    const int dy = !yin ? 0 : (gj == 0 ? -1 : (gj == ny - 1 ? 1 : 0));
    Real *xa = S + plane_a + w.at, *xb = xa + (plane_b - plane_a);
    const int ox = dx * STR, oy = dy * AC * STR;
    constexpr bool two = decltype(TWO)::value;
    // (scalar loads; a select between the two would be a load per lane)
    const Real qxl = uniform((Real)P.qlo[0]), qxh = uniform((Real)P.qhi[0]), qyl = uniform((Real)P.qlo[1]),
               qyh = uniform((Real)P.qhi[1]);
    const Real qx = dx < 0 ? qxl : qxh, qy = dy < 0 ? qyl : qyh;
    if (dx != 0) ghost_line<PAIR, two>(xa, xb, ox, qx, fa, fb);
    if (split_y) __syncthreads();
    if (dy != 0) ghost_line<PAIR, two>(xa, xb, oy, qy, fa, fb);
    if (dx != 0 && dy != 0) {  // a corner: its x ghosts, extrapolated along y
      wave_order();
      Real ca[NQ], cb[NQ];
      lds_get<PAIR, all_slots(PAIR)>(xa + ox, ca);
      if constexpr (two) lds_get<PAIR, all_slots(PAIR)>(xb + ox, cb);
      ghost_line<PAIR, two>(xa + ox, xb + ox, oy, qy, ca, cb);
    }
  };
  using Two = std::true_type;
  using One = std::false_type;

  // ---- faces: reconstruction from LDS and collision ----
  // The trilinear interpolation of src/dugks.cu:756-906; GRAD: calc_fx,
  // src/dugks.cu:421-583.  A face's arithmetic does not need the lane that
  // owns its cells: any lane can take any x- or y-face.
  constexpr unsigned kXp = slot_mask<PAIR>(0, 1), kXm = slot_mask<PAIR>(0, -1), kYp = slot_mask<PAIR>(1, 1),
                     kYm = slot_mask<PAIR>(1, -1), kX = kXp | kXm, kY = kYp | kYm, kZ = slot_mask<PAIR>(2, 2);
  // values upwind along an axis of every slot that moves along it: up from
  // the neighbour of c = +1, dn from that of c = -1
  auto get_upwind = [&](auto MP, auto MM, const Real* up, const Real* dn, Real (&v)[NQ]) {
    lds_get<PAIR, decltype(MP)::value>(up, v);
    lds_get<PAIR, decltype(MM)::value>(dn, v);
  };
  using MXp = std::integral_constant<unsigned, kXp>;
  using MXm = std::integral_constant<unsigned, kXm>;
  using MYp = std::integral_constant<unsigned, kYp>;
  using MYm = std::integral_constant<unsigned, kYm>;
  // the z-face above plane p (Zn; GRAD: between ring slots q0 and qp) of the lane's column
  auto zface = [&](Real (&out)[NX], int q0, int qp) {
    LaneFace<PAIR, Real, 2> fc;
    const Place w = place();
    const Real sh = sign(w.half);
    if constexpr (GRAD) {
      const Real *a = S + q0 + w.at, *d = a + (qp - q0);
      Real fl[NQ], fr[NQ], gx[NQ] = {}, gy[NQ] = {};
      lds_diff<PAIR, kX>(a + STR, d + STR, a - STR, d - STR, gx);
      lds_diff<PAIR, kY>(a + AC * STR, d + AC * STR, a - AC * STR, d - AC * STR, gy);
      lds_get<PAIR, kAll>(a, fl);
      lds_get<PAIR, kAll>(d, fr);
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = slot_pop(PAIR, k), cx = CX[ip], cy = CY[ip], cz = CZ[ip];
        fc.template put<k>(grad_foot<cx, cy, cz>(Real(0.5) * (fr[k] + fl[k]), sh * gtn[0], gx[k], sh * gtn[1], gy[k],
                                                 sh * gin[2], fr[k] - fl[k]));
      });
    } else {
      const Real* a = S + AN + w.at;
      const int sx = up_x(w.half), sy = up_y(w.half);
      const Real xt[2] = {xw(w.half, 3, w.c), xw(w.half, 4, w.c)}, yt[2] = {yw(w.half, 3, w.r), yw(w.half, 4, w.r)};
      Real v[NQ], vx[NQ], vy[NQ], vd[NQ];
      lds_get<PAIR, kAll>(a, v);
      get_upwind(MXp{}, MXm{}, a - sx, a + sx, vx);
      get_upwind(MYp{}, MYm{}, a - sy, a + sy, vy);
      lds_get<PAIR, kXp & kYp>(a - sx - sy, vd);
      lds_get<PAIR, kXm & kYp>(a + sx - sy, vd);
      lds_get<PAIR, kXp & kYm>(a - sx + sy, vd);
      lds_get<PAIR, kXm & kYm>(a + sx + sy, vd);
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = slot_pop(PAIR, k), cx = CX[ip], cy = CY[ip];
        Real w = v[k];
        if constexpr (cx != 0) w = lerp_(w, vx[k], xt[cx > 0]);
        if constexpr (cy != 0) {
          Real w2 = vy[k];
          if constexpr (cx != 0) w2 = lerp_(w2, vd[k], xt[cx > 0]);
          w = lerp_(w, w2, yt[cy > 0]);
        }
        fc.template put<k>(w);
      });
    }
    fc.template collide<kShift>(F, sh * hh, sh * fw0, fw1, fw2, out);
  };
  // the x-face between tile columns c-1 and c of row r
  auto xface = [&](int half, int r, int c, int qm, int q0, int qp) {
    LaneFace<PAIR, Real, 0> fc;
    const Real sh = sign(half);
    const int pos = r * AC + c + 1;
    if constexpr (GRAD) {
      const Real *a = S + q0 + at(half, pos), *m = a + (qm - q0), *d = a + (qp - q0);
      Real fl[NQ], fr[NQ], gy[NQ] = {}, gz[NQ] = {};
      lds_diff<PAIR, kY>(a + AC * STR - STR, a + AC * STR, a - AC * STR - STR, a - AC * STR, gy);
      lds_diff<PAIR, kZ>(d - STR, d, m - STR, m, gz);
      lds_get<PAIR, kAll>(a - STR, fl);
      lds_get<PAIR, kAll>(a, fr);
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = slot_pop(PAIR, k), cx = CX[ip], cy = CY[ip], cz = CZ[ip];
        fc.template put<k>(grad_foot<cx, cy, cz>(Real(0.5) * (fr[k] + fl[k]), sh * gin[0], fr[k] - fl[k], sh * gtn[1],
                                                 gy[k], sh * gtn[2], gz[k]));
      });
    } else {
      const Real* a = S + at(half, pos);
      const int sy = up_y(half);
      const Real xn[3] = {xw(half, 0, c), xw(half, 1, c), xw(half, 2, c)}, yt[2] = {yw(half, 3, r), yw(half, 4, r)};
      Real lo[NQ], hi[NQ], lt[NQ], ht[NQ];
      lds_get<PAIR, kAll>(a - STR, lo);
      lds_get<PAIR, kAll>(a, hi);
      get_upwind(MYp{}, MYm{}, a - STR - sy, a - STR + sy, lt);
      get_upwind(MYp{}, MYm{}, a - sy, a + sy, ht);
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = slot_pop(PAIR, k), cx = CX[ip], cy = CY[ip];
        if constexpr (k == 0) {
          fc.template put<0>(Real(0.5) * (lo[0] + hi[0]));
        } else {
          Real v = lerp_(lo[k], hi[k], xn[cx + 1]);
          if constexpr (cy != 0) v = lerp_(v, lerp_(lt[k], ht[k], xn[cx + 1]), yt[cy > 0]);
          fc.template put<k>(v);
        }
      });
    }
    if (!P.periodic[0]) fc.bounce(i0 + c == 0, i0 + c == nx, half);
    Real out[NX];
    fc.template collide<kShift>(F, sh * hh, sh * fw0, fw1, fw2, out);
    flux_put<NX, FS>(S + T::OX + fat(half, pos), out);
  };
  // the y-face between tile rows r-1 and r of column c
  auto yface = [&](int half, int r, int c, int qm, int q0, int qp) {
    LaneFace<PAIR, Real, 1> fc;
    const Real sh = sign(half);
    const int pos = r * AC + c + 1;
    if constexpr (GRAD) {
      const Real *a = S + q0 + at(half, pos), *m = a + (qm - q0), *d = a + (qp - q0);
      Real fl[NQ], fr[NQ], gx[NQ] = {}, gz[NQ] = {};
      lds_diff<PAIR, kX>(a - AC * STR + STR, a + STR, a - AC * STR - STR, a - STR, gx);
      lds_diff<PAIR, kZ>(d - AC * STR, d, m - AC * STR, m, gz);
      lds_get<PAIR, kAll>(a - AC * STR, fl);
      lds_get<PAIR, kAll>(a, fr);
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = slot_pop(PAIR, k), cx = CX[ip], cy = CY[ip], cz = CZ[ip];
        fc.template put<k>(grad_foot<cx, cy, cz>(Real(0.5) * (fr[k] + fl[k]), sh * gtn[0], gx[k], sh * gin[1],
                                                 fr[k] - fl[k], sh * gtn[2], gz[k]));
      });
    } else {
      const Real* a = S + at(half, pos);
      const int sx = up_x(half);
      const Real yn[3] = {yw(half, 0, r), yw(half, 1, r), yw(half, 2, r)}, xt[2] = {xw(half, 3, c), xw(half, 4, c)};
      Real lo[NQ], hi[NQ], lt[NQ], ht[NQ];
      lds_get<PAIR, kAll>(a - AC * STR, lo);
      lds_get<PAIR, kAll>(a, hi);
      get_upwind(MXp{}, MXm{}, a - AC * STR - sx, a - AC * STR + sx, lt);
      get_upwind(MXp{}, MXm{}, a - sx, a + sx, ht);
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = slot_pop(PAIR, k), cx = CX[ip], cy = CY[ip];
        if constexpr (k == 0) {
          fc.template put<0>(Real(0.5) * (lo[0] + hi[0]));
        } else {
          Real l = lo[k], h = hi[k];
          if constexpr (cx != 0) {
            l = lerp_(l, lt[k], xt[cx > 0]);
            h = lerp_(h, ht[k], xt[cx > 0]);
          }
          fc.template put<k>(lerp_(l, h, yn[cy + 1]));
        }
      });
    }
    if (!P.periodic[1]) fc.bounce(j0 - 1 + r == 0, j0 - 1 + r == ny, half);
    Real out[NX];
    fc.template collide<kShift>(F, sh * hh, sh * fw0, fw1, fw2, out);
    flux_put<NX, FS>(S + T::OY + fat(half, pos), out);
  };

  // The faces each wave takes.  An interior wave takes the z- and x-faces of
  // its own columns; the y-faces, in units of the interior waves' columns,
  // go mostly to the waves of the halo columns, which have no z-faces and no
  // update: on 32 x 12 tiles the halo waves 6 and 7 take two units each and
  // the top row of y-faces or the right column of x-faces, waves 0 and 1 one
  // unit each, which evens the SIMDs out (wave w runs on SIMD w % 4, so two
  // SIMDs hold two interior waves and two hold one).
  constexpr int kMore = T::NWI >= 6 ? 2 : 1;
  constexpr int kGive = 2 * kMore;  // y units the halo waves take
  static_assert(T::NW - T::NWI == 2 && kGive <= T::NWI, "two waves of halo columns");
  const bool top_wave = wave == T::NW - 2, right_wave = wave == T::NW - 1;
  const int ya = top_wave ? T::NWI - kMore : (right_wave ? T::NWI - 2 * kMore : (wave < T::NWI - kGive ? wave : 0));
  const int yb = top_wave ? T::NWI : (right_wave ? T::NWI - kMore : (wave < T::NWI - kGive ? wave + 1 : 0));
  const bool do_x = right_wave ? lane < th : interior;

  // ---- the column's f-bar+ ----
  using Raw = RawLane<PAIR, Real, Store>;
  // lanes without a column of their own load zeros (and compute on them)
  const unsigned column = (unsigned)(gj * nx + gi);
  auto load_part = [&](auto A, auto B, int k, Raw& raw) {
    raw.template load<decltype(A)::value, decltype(B)::value>(
        bin, LaneOffsets<PAIR, Store>(here(column), N, place().half).where(own, true, span),
        (unsigned)k * nxy, N);
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, NQ / 3>;
  using B2 = std::integral_constant<int, NQ * 2 / 3>;
  using B3 = std::integral_constant<int, NQ>;
  auto load_own = [&](int k, Raw& raw) { load_part(B0{}, B3{}, k, raw); };
  // f-bar+ of plane k from its stored values, and g = f-bar+ + (f-bar+ - f)/3,
  // the part of the update that needs f: 4/3 f-bar+ - 1/3 f written so that
  // the rounding of 1/3 biases nothing (the two terms of the difference
  // carry the same mass)
  auto centre = [&](const Raw& raw, int k, Real (&fb)[NQ], Real (&g)[NQ]) {
    Real Fc[3] = {F[0], F[1], F[2]};
    if (P.fcell && own) {
      const unsigned cc = (unsigned)k * nxy + column;
      for (int a = 0; a < 3; a++) Fc[a] += (Real)P.fcell[a * P.N + cc];
    }
    const Real sh = sign(place().half);
    Real ff[NQ], rho, us0[3];
    raw.template decode<kShift>(P, sh, ff, rho, us0);
    lane_fbar<PAIR, kShift, Real>(ff, rho, us0, Fc, sh * hdt, sh * bw0, bw2, fb);
    for (int q = 0; q < NQ; q++) g[q] = fb[q] + (fb[q] - ff[q]) * Real(1.0 / 3.0);
  };
  // Zn(p+1/2) of this column
  auto form_zn = [&](const Real (&lo)[NQ], const Real (&hi)[NQ], int half, Real (&v)[NQ]) {
    const Real wp = PAIR && half ? wznm : wznp;
    static_for<NQ>([&](auto K) {
      constexpr int k = decltype(K)::value;
      constexpr int cz = CZ[slot_pop(PAIR, k)];
      if constexpr (k == 0)
        v[0] = Real(0.5) * (lo[0] + hi[0]);
      else
        v[k] = lerp_(lo[k], hi[k], cz == 0 ? wzn0 : (cz > 0 ? wp : wznm));
    });
  };

  // f-bar+(p-1) of the slots with c_z = +1 (pair: those that move along z)
  constexpr int NM = 5;
  auto zp_slot = [](int n) {
    int m = 0;
    for (int k = 0; k < NQ; k++)
      if (CZ[slot_pop(PAIR, k)] > 0 && m++ == n) return k;
    return 0;
  };
  Real fbm[NM], fbc[NQ], fbn[NQ], gc[NQ], gn[NQ], zm[NX];
  double run_flow = 0;
  // f of the own column one plane ahead of its f-bar+
  Raw fpre;
  load_own((z0 + 1) % nz, fpre);

  // ---- pre-loop: f-bar+ at z0-1 and z0, and the -z face of plane z0 ----
  {
    Raw lo, hi;
    const int km = (z0 - 1 + nz) % nz;
    load_own(km, lo);
    load_own(z0, hi);
    centre(lo, km, fbn, gn);
    centre(hi, z0, fbc, gc);
    static_for<NM>([&](auto M) {
      constexpr int n = decltype(M)::value;
      constexpr int k = zp_slot(n);
      fbm[n] = fbn[k];
    });
    const Place w = place();
    if constexpr (GRAD) {
      if (own) {
        lds_put<PAIR>(S + rslot(z0 - 1) + w.at, fbn);
        lds_put<PAIR>(S + rslot(z0) + w.at, fbc);
      }
      if (wall_tile) fill_ghosts(Two{}, rslot(z0 - 1), fbn, rslot(z0), fbc);
    } else {
      Real v[NQ];
      form_zn(fbn, fbc, w.half, v);
      if (own) lds_put<PAIR>(S + AN + w.at, v);
      if (wall_tile) fill_ghosts(One{}, AN, v, AN, v);
    }
    __syncthreads();
    if (interior && !FLAT) zface(zm, rslot(z0 - 1), rslot(z0));
    __syncthreads();
  }

  // One plane p: fbc / gc hold f-bar+ and g of plane p, and the plane computes
  // those of p + 1 into fbn / gn.  The loop runs planes in pairs with the two
  // register sets swapped, so that no copy moves them.
  auto plane = [&](int p, Real (&fbc)[NQ], Real (&fbn)[NQ], Real (&gc)[NQ], Real (&gn)[NQ]) {
    const int qm = rslot(p - 1), q0 = rslot(p), qp = rslot(p + 1);
    // ---- phase 1: f-bar+(p+1); Z(p) and Zn(p+1/2) (GRAD: its ring slot) ----
    const int kn = p + 1 < nz ? p + 1 : 0;
    centre(fpre, kn, fbn, gn);
    const int kp = kn + 1 < nz ? kn + 1 : 0;
    load_part(B0{}, B1{}, kp, fpre);
    if constexpr (GRAD) {
      const Place w = place();
      if (own) lds_put<PAIR>(S + qp + w.at, fbn);
      if (wall_tile) fill_ghosts(One{}, qp, fbn, qp, fbn);
    } else {
      const Place w = place();
      Real v[NQ], vn[NQ];
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int cz = CZ[slot_pop(PAIR, k)];
        v[k] = fbc[k];
        if constexpr (cz < 0) v[k] = lerp_(fbc[k], fbn[k], wzt);
      });
      static_for<NM>([&](auto M) {
        constexpr int n = decltype(M)::value;
        constexpr int k = zp_slot(n);
        v[k] = lerp_(fbc[k], PAIR && w.half ? fbn[k] : fbm[n], wzt);
      });
      form_zn(fbc, fbn, w.half, vn);
      if (own) {
        lds_put<PAIR>(S + w.at, v);
        lds_put<PAIR>(S + AN + w.at, vn);
      }
      if (wall_tile) fill_ghosts(Two{}, 0, v, AN, vn);
    }
    __syncthreads();
    // ---- phase 2: the faces of plane p (-x, -y from Z; +z from Zn) ----
    {
      const Place w = place();
      if (do_x) xface(w.half, right_wave ? lane + 1 : w.r, right_wave ? tw : w.c, qm, q0, qp);
    }
    load_part(B1{}, B2{}, kp, fpre);
    for (int q = ya; q < yb + (top_wave ? 1 : 0); q++) {
      const int h = place().half, l = PAIR ? ((here(t) >> 4) & 3) * 8 + (t & 7) : here(t) & 63;
      const int v = q * UNIT + l;
      const bool top = q == yb;
      const int yr = top ? th + 1 : v / TX + 1, yc = top ? l : v % TX;
      if ((top || yr <= th) && yc < tw) yface(h, yr, yc, qm, q0, qp);
    }
    load_part(B2{}, B3{}, kp, fpre);
    Real zp[NX];
    if (interior && !FLAT) zface(zp, q0, qp);
    __syncthreads();
    // ---- phase 3: update of plane p ----
    Real fnew[NQ], rr = Real(0), un[3] = {Real(0), Real(0), Real(0)};  // kNeq: drho and u of the new state
    if (interior) {
      const Place w = place();
      const Real updx = xw(w.half, 5, w.c), updy = yw(w.half, 5, w.r), uz = sign(w.half) * updz;
      const Real *X = S + T::OX + w.fat, *Y = S + T::OY + w.fat;
      Real xl[NX], xh[NX], yl[NX], yh[NX];
      flux_get<NX, FS>(X, xl);
      flux_get<NX, FS>(X + FS, xh);
      flux_get<NX, FS>(Y, yl);
      flux_get<NX, FS>(Y + AC * FS, yh);
      // f~(p+1) = 4/3 f-bar+ - 1/3 f~ - sum_a (dt/dx_a) c_a (F_a+ - F_a-)
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = slot_pop(PAIR, k);
        constexpr int kx = lane_cross<PAIR, 0>(k), ky = lane_cross<PAIR, 1>(k), kz = lane_cross<PAIR, 2>(k);
        Real v = gc[k];
        if constexpr (kx >= 0) v -= Real(CX[ip]) * updx * (xh[kx] - xl[kx]);
        if constexpr (ky >= 0) v -= Real(CY[ip]) * updy * (yh[ky] - yl[ky]);
        if constexpr (kz >= 0 && !FLAT) {
          v -= Real(CZ[ip]) * uz * (zp[kz] - zm[kz]);
          zm[kz] = zp[kz];
        }
        fnew[k] = v;
      });
      if constexpr (kNeq) {
        lane_rho_u<PAIR, Real>(fnew, rr, un, true);
        // (the velocity as it is stored)
        if (law.partial && stored) run_flow += (double)(as == 0 ? un[0] : (as == 1 ? un[1] : un[2]));
      } else if (law.partial) {
        // bulk velocity of the new state for the flow-rate controller
        const double u = lane_velocity<PAIR, Real>(fnew, as);
        if (stored) run_flow += u;
      }
    }
    // Stores without a branch (lanes that store nothing address the end of
    // the array): the compiler then knows how many stores follow the loads
    // issued in phase 1, and the next plane's decode waits for those loads
    // alone.  (The vector-memory counter counts loads and stores in issue
    // order; behind a branch the wait would cover the stores too.)
    {
      using O = LaneOffsets<PAIR, Store>;
      const unsigned cell = (unsigned)p * nxy;
      const int h = place().half;
      const O so = O(here(column), N, h).where(stored, !h, span);
      if constexpr (kNeq) {
        // FP16 non-equilibrium encoding: rho - 1, u and
        // s_i = (h_i / w_i - drho - rho eps_i) kNeqScale
        static_assert(!PAIR, "FP16 storage steps whole cells");
        const NeqEq<Real> eq(rr, un);
        bout.putf((float)rr, so.mom, cell * 4u);
        for (int q = 0; q < 3; q++) bout.putf((float)un[q], so.mom, cell * 4u + (q + 1) * 4u * N);
        static_for<NQ>([&](auto K) {
          constexpr int k = decltype(K)::value;
          const Real n = (fnew[k] - eq.template eq<k>()) * Real((double)kNeqScale / wgt(k));
          bout.put(__float2half((float)n), so.template at<k>(), O::template scalar<k>(cell, N));
        });
      } else {
        static_for<NQ>([&](auto K) {
          constexpr int k = decltype(K)::value;
          st_state<Real, Store>(bout, so.template at<k>(), O::template scalar<k>(cell, N), fnew[k], P,
                                slot_pop(PAIR, k));
        });
      }
    }
    static_for<NM>([&](auto M) {
      constexpr int n = decltype(M)::value;
      constexpr int k = zp_slot(n);
      fbm[n] = fbc[k];
    });
    // no barrier: the next phase 1 writes the planes (GRAD: the ring slot of
    // p-1, last read in this plane's phase 2), which phase 3 does not read,
    // and the next phase 2 writes the fluxes only after the next phase-1 barrier
  };
  if constexpr (GRAD) {
    // (g alone moves, and the pair's second copy of the code would spill)
    for (int p = z0; p < zend; p++) {
      plane(p, fbc, fbn, gc, gn);
      for (int k = 0; k < NQ; k++) gc[k] = gn[k];
    }
  } else {
    for (int p = z0; p < zend; p += 2) {
      plane(p, fbc, fbn, gc, gn);
      if (p + 1 < zend) plane(p + 1, fbn, fbc, gn, gc);
    }
  }

  if (law.partial) {
    // every column of the tile has the same z width (z is uniform here)
    const Place w = place();
    if (stored && !w.half) flow += run_flow * (P.wd[0][i0 + w.c + 1] * P.wd[1][j0 + w.r] * P.wd[2][1]);
  }
  if constexpr (!RUNS) break;
  }

  if (law.partial) {
    // fixed-order block reduction of the flow sums; the last workgroup to get
    // here adds them all up, in order, and moves the force (every workgroup
    // read it at its start).  A launch of its own for that took 8 us a step.
    double v[1] = {flow};
    constexpr int kSum[1] = {0};
    block_reduce<1, T::NT>(v, kSum);
    __shared__ unsigned arrived;
    if (t == 0) {
      __hip_atomic_store(&law.partial[tt], v[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      arrived = __hip_atomic_fetch_add(law.arrived, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (arrived == gridDim.x - 1) {
      double sum[1] = {0.0};
      for (int k = t; k < (int)gridDim.x; k += T::NT)
        sum[0] += __hip_atomic_load(&law.partial[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      block_reduce<1, T::NT>(sum, kSum);
      if (t == 0) {
        flow_update(law.famb, as, sum[0] / law.volume, law.target, law.gain, law.dt);
        *law.arrived = 0;  // for the next launch
      }
    }
  }
}
