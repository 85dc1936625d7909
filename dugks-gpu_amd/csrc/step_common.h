// Building blocks of the step kernel (step_kernel.h): what one lane holds of
// a cell, its loads, its half or whole faces.
//
// With FP32 arithmetic a lane holds a whole cell (19 slots).  With FP64 a
// pair of lanes shares a cell (10 slots each): one holds the rest population
// and nine moving ones, the other the rest population and the nine opposite
// ones.  A whole cell in FP64 took 393 registers, one wave per SIMD, and the
// step waited on latency 70 % of the time; half a cell leaves room for two.
//
// The lanes of a pair are eight apart in a row of sixteen (DPP row_ror:8
// exchanges them within a VALU instruction).  The minus lane sees the lattice
// mirrored through the origin: with s = +1 on plus lanes and -1 on minus
// lanes, us = s u, the velocity of the population in slot k is s c_k (c_k the
// plus lane's), so c.u = c_k.us and c.F = s c_k.F, and both lanes run the same
// instructions.  Sums over the lattice add the two lanes' partial sums; sums
// weighted by c take the difference own - other, which is s j.  For a whole
// cell s is 1 and the sums are the lane's own.
// Included inside namespace dugks { namespace { ... } }.
#pragma once

constexpr int kPairPops[10] = {0, 1, 3, 5, 7, 8, 11, 12, 15, 16};
constexpr int lane_slots(bool pair) { return pair ? 10 : Q; }
// population of slot k (pair: of the plus lane; the minus lane's is its opposite)
__host__ __device__ constexpr int slot_pop(bool pair, int k) { return pair ? kPairPops[k] : k; }

// Index of slot k among those that cross a face normal to axis A (-1: does
// not cross), the slot of crossing index n, and the number of them.
template <bool PAIR, int A>
__host__ __device__ constexpr int lane_cross(int k) {
  int n = 0;
  for (int q = 0; q < lane_slots(PAIR); q++) {
    if (cv(A, slot_pop(PAIR, q)) == 0) continue;
    if (q == k) return n;
    n++;
  }
  return -1;
}
template <bool PAIR, int A>
__host__ __device__ constexpr int cross_slot(int n) {
  for (int q = 0; q < lane_slots(PAIR); q++)
    if (lane_cross<PAIR, A>(q) == n) return q;
  return -1;
}
constexpr int lane_crossings(bool pair) { return pair ? 5 : 10; }
// First moving slot (that does not cross axis A) with a component b (b < 0:
// any): partial sums start from their first term.
template <bool PAIR>
__host__ __device__ constexpr int first_slot(int b, int A = -1) {
  for (int q = 1; q < lane_slots(PAIR); q++) {
    const int ip = slot_pop(PAIR, q);
    if (A >= 0 && cv(A, ip) != 0) continue;
    if (b < 0 || cv(b, ip) != 0) return q;
  }
  return -1;
}

// x of the pair's other lane.
__device__ __forceinline__ float pair_other(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x128, 0xf, 0xf, true));
}
__device__ __forceinline__ double pair_other(double x) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)b, 0x128, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), 0x128, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (unsigned long long)(unsigned)lo | (unsigned long long)(unsigned)hi << 32);
}
// a cell's sum over the lattice, and s times its c-weighted sum, from the lane's part
template <bool PAIR, class T>
__device__ __forceinline__ T cell_sum(T x) {
  if constexpr (PAIR) return x + pair_other(x); else return x;
}
template <bool PAIR, class T>
__device__ __forceinline__ T cell_diff(T x) {
  if constexpr (PAIR) return x - pair_other(x); else return x;
}

// A value that is the same in every lane, held in scalar registers.
__device__ __forceinline__ float uniform(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}
__device__ __forceinline__ double uniform(double x) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b);
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32));
  return __builtin_bit_cast(double, (unsigned long long)lo | (unsigned long long)hi << 32);
}
// v as a value of its own: keeps the optimiser from widening the load of an
// array element that starts a vector into a load of the array's memory, which
// would put the array into scratch.
template <class T>
__device__ __forceinline__ T scalar(T v) {
  asm("" : "+v"(v));
  return v;
}

// Partial sums over the lane's moving slots: r = sum v, j = sum c_k v.
template <bool PAIR, class T, class V>
__device__ __forceinline__ void lane_moments(const V (&v)[lane_slots(PAIR)], T& r, T (&j)[3]) {
  static_for<lane_slots(PAIR) - 1>([&](auto K) {
    constexpr int k = decltype(K)::value + 1;
    constexpr int ip = slot_pop(PAIR, k);
    const T x = (T)v[k];
    if constexpr (k == 1) r = x; else r += x;
    static_for<3>([&](auto B) {
      constexpr int b = decltype(B)::value;
      if constexpr (cv(b, ip) != 0) {
        const T y = cv(b, ip) > 0 ? x : -x;
        if constexpr (k == first_slot<PAIR>(b)) j[b] = y; else j[b] += y;
      }
    });
  });
}

// rho and us0 = s u0, u0 = j / rho, of the cell (cell_rho_u: FP32 populations
// are summed in FP64 and rounded once); with `shifted` the values are
// h = f - w and rho is drho = rho - 1.
template <bool PAIR, class Real>
__device__ __forceinline__ void lane_rho_u(const Real (&v)[lane_slots(PAIR)], Real& rho_out, Real (&us0)[3],
                                           bool shifted = false) {
  if constexpr (sizeof(Real) == 4) {
    double r, j[3];
    lane_moments<PAIR, double>(v, r, j);
    r = cell_sum<PAIR>(r) + (double)v[0];
    rho_out = (Real)r;
    const double rho = shifted ? 1.0 + r : r;
    // 1/rho: the hardware reciprocal and one Newton step (error ~1e-14)
    double x = __builtin_amdgcn_rcp(rho);
    x = __builtin_fma(x, __builtin_fma(-rho, x, 1.0), x);
    for (int a = 0; a < 3; a++) us0[a] = (Real)(cell_diff<PAIR>(j[a]) * x);
  } else {
    Real r, j[3];
    lane_moments<PAIR, Real>(v, r, j);
    rho_out = cell_sum<PAIR>(r) + v[0];
    const Real inv = rcp_real(shifted ? Real(1) + rho_out : rho_out);
    for (int a = 0; a < 3; a++) us0[a] = cell_diff<PAIR>(j[a]) * inv;
  }
}

// s u_axis of the cell for the flow-rate controller, summed in FP64 whatever the
// arithmetic.  The controller divides the change of the bulk velocity by dt, so
// it reads what the state holds, as the two-pass kernels' reduction over the
// state does (FP32 sums left the reading of a 16x12x1 channel 8e-12 off, these
// leave it within 5e-15).  128^3 channel with FP16 deviations 168 us a step, with
// FP32 sums 166; FP32 channels 150x97x83 and 256x192x256 the same.
template <bool PAIR, class Real>
__device__ __forceinline__ double lane_velocity(const Real (&v)[lane_slots(PAIR)], int axis) {
  double r, j[3];
  lane_moments<PAIR, double>(v, r, j);
  r = cell_sum<PAIR>(r) + (double)v[0];
  const double ja = cell_diff<PAIR>(axis == 0 ? j[0] : (axis == 1 ? j[1] : j[2]));
  if constexpr (sizeof(Real) == 8) {
    return ja * rcp_real(r);
  } else {
    // 1/rho: the hardware reciprocal and two Newton steps
    double x = __builtin_amdgcn_rcp(r);
    x = __builtin_fma(x, __builtin_fma(-r, x, 1.0), x);
    x = __builtin_fma(x, __builtin_fma(-r, x, 1.0), x);
    return ja * x;
  }
}

// centre_fbar of the lane's slots (SHIFT: in shifted populations, hb = f-bar+
// - w from h, drho and u0; see EqShift).  shdt = s h and
// sbw0 = s bw0 carry the mirrored frame's sign of the force terms: h F enters
// us as s h F, and bw0 (c - u).F = s bw0 (c_k - us).F.
template <bool PAIR, bool SHIFT, class Real>
__device__ __forceinline__ void lane_fbar(const Real (&f)[lane_slots(PAIR)], Real rho, const Real (&us0)[3],
                                          const Real F[3], Real shdt, Real sbw0, Real bw2,
                                          Real (&fb)[lane_slots(PAIR)]) {
  constexpr int NQ = lane_slots(PAIR);
  const Real ux = us0[0] + shdt * F[0], uy = us0[1] + shdt * F[1], uz = us0[2] + shdt * F[2];
  if constexpr (SHIFT) {
    const EqShift<Real> eq(ExactProducts{}, rho, ux, uy, uz, F, bw2, sbw0);
    static_for<NQ>([&](auto K) {
      constexpr int ip = slot_pop(PAIR, decltype(K)::value);
      fb[decltype(K)::value] =
          eq.template relax<ip>(-bw2, f[decltype(K)::value], cdot<ip>(F[0], F[1], F[2]));
    });
  } else {
    const EqTerm<Real> eq(ExactProducts{}, rho, ux, uy, uz, F, bw2, sbw0);
    static_for<NQ>([&](auto K) {
      constexpr int k = decltype(K)::value;
      constexpr int ip = slot_pop(PAIR, k);
      if constexpr (k != 0 || sizeof(Real) != 4)
        fb[k] = eq.template relax_keep<ip>(-bw2, f[k], cdot<ip>(F[0], F[1], F[2]));
    });
    if constexpr (sizeof(Real) == 4) {
      Real moving = fb[1];
      for (int k = 2; k < NQ; k++) moving += fb[k];
      fb[0] = rho - cell_sum<PAIR>(moving);
    }
  }
}

// Byte offsets of a column's values in a state array.  Pair: population
// kPairPops[k] on plus lanes and its opposite on minus lanes, which lies one
// population further, or three for the slots whose opposite is the fourth of
// its edge group.  The plane and the slot go into the scalar offset.
template <bool PAIR, class Store>
struct LaneOffsets {
  static constexpr bool kNeq = std::is_same<Store, NeqHalf>::value;
  static constexpr unsigned kSize = kNeq ? 2u : (unsigned)sizeof(Store);
  unsigned rest, one, three;  // rest slot; slots with gap 1, gap 3
  unsigned mom;               // NeqHalf: of the first FP32 value
  __device__ __forceinline__ LaneOffsets(unsigned column, unsigned N, int half) {
    rest = column * kSize;
    one = rest + (PAIR && half ? N * kSize : 0u);
    three = rest + (PAIR && half ? 3u * N * kSize : 0u);
    mom = column * 4u;
  }
  // these offsets, or (where a condition fails) the end of the array, where
  // loads return 0 and stores are dropped: the accesses then need no branch
  __device__ __forceinline__ LaneOffsets where(bool all, bool also_rest, unsigned end) const {
    LaneOffsets o = *this;
    o.rest = all && also_rest ? rest : end;
    o.one = all ? one : end;
    o.three = all ? three : end;
    o.mom = all ? mom : end;
    return o;
  }
  template <int k>
  __device__ __forceinline__ unsigned at() const {
    if constexpr (!PAIR || k == 0) {
      return rest;
    } else {
      constexpr int gap = OPP[slot_pop(PAIR, k)] - slot_pop(PAIR, k);
      static_assert(gap == 1 || gap == 3, "lattice order");
      return gap == 3 ? three : one;
    }
  }
  // scalar offset of slot k in the plane whose first cell is `cell`
  template <int k>
  __device__ __forceinline__ static unsigned scalar(unsigned cell, unsigned N) {
    return (kNeq ? 16u * N : 0u) + slot_pop(PAIR, k) * kSize * N + cell * kSize;
  }
};

// The lane's part of a cell as loaded through a StateBuf (see RawCell: loads
// issued ahead, decoded at use, FP16 values held in 32-bit slots).
template <bool PAIR, class Real, class Store>
struct RawLane {
  static constexpr int NQ = lane_slots(PAIR);
  static constexpr bool kNeq = std::is_same<Store, NeqHalf>::value;
  static constexpr bool kHalf = kNeq || std::is_same<Store, __half>::value;
  using Slot = typename std::conditional<kHalf, unsigned, Store>::type;
  Slot v[NQ];
  float m[kNeq ? 4 : 1];
  // slots A..B-1 of the column in the plane whose first cell is `cell`
  // (uniform); slot 0 comes with the NeqHalf moments
  template <int A = 0, int B = NQ>
  __device__ __forceinline__ void load(const StateBuf<Store>& b, const LaneOffsets<PAIR, Store>& o, unsigned cell,
                                       unsigned N) {
    using O = LaneOffsets<PAIR, Store>;
    if constexpr (kNeq && A == 0)
      for (int q = 0; q < 4; q++) m[q] = b.rawf(o.mom, cell * 4u + q * 4u * N);
    static_for<B - A>([&](auto K) {
      constexpr int k = decltype(K)::value + A;
      if constexpr (kHalf)
        v[k] = raw_b16_32(b.r, o.template at<k>(), O::template scalar<k>(cell, N));
      else
        v[k] = b.raw(o.template at<k>(), O::template scalar<k>(cell, N));
    });
  }
  // The lane's populations (SHIFT: less their weights), rho (SHIFT: drho) and
  // us0 = s u0.
  template <bool SHIFT>
  __device__ __forceinline__ void decode(const KParams& P, Real s, Real (&f)[NQ], Real& rho, Real (&us0)[3]) const {
    if constexpr (kNeq) {
      // h_i = f_i - w_i = w_i rho eps_i + w_i drho + w_i s_i / kNeqScale straight
      // from the stored drho, u and s (see EqShift), with the per-class products
      // w rho and w drho rounded once (NeqEq; as in the centre stage, products
      // rounded twice bias the flow's dissipation.  On the Re = 1600
      // Taylor-Green vortex, against FP64: this decode and the centre stage's
      // EqShift products both rounded twice, 0.67 % less dissipation; only
      // EqShift's once, 0.54 % more; only the decode's once, 1.2 % less; both
      // once, 0.01 %)
      static_assert(SHIFT, "FP16 non-equilibrium storage steps shifted populations");
      rho = (Real)m[0];
      for (int a = 0; a < 3; a++) us0[a] = s * (Real)m[1 + a];
      const NeqEq<Real> eq(rho, us0);
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        const Real sv = (Real)__half2float(__ushort_as_half((unsigned short)v[k]));
        f[k] = eq.template shift_of<slot_pop(PAIR, k)>(sv);
      });
    } else {
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = slot_pop(PAIR, k);
        if constexpr (kHalf)
          f[k] = (Real)((float)wgt(ip) * (P.rho0f + __half2float(__ushort_as_half((unsigned short)v[k]))));
        else
          f[k] = (Real)v[k];
      });
      lane_rho_u<PAIR, Real>(f, rho, us0);
    }
  }
};

// The lane's part of a face normal to axis A (Face): the crossing values, the
// rest value, and the partial moments of the others.
template <bool PAIR, class Real, int A>
struct LaneFace {
  static constexpr int NX = lane_crossings(PAIR);
  Real cross[NX], rest, rho, j[3];
  template <int k>
  __device__ __forceinline__ void put(Real v) {
    constexpr int n = lane_cross<PAIR, A>(k);
    constexpr int ip = slot_pop(PAIR, k);
    if constexpr (k == 0) {
      rest = v;
    } else if constexpr (n >= 0) {
      cross[n] = v;
    } else {
      if constexpr (k == first_slot<PAIR>(-1, A)) rho = v; else rho += v;
      static_for<3>([&](auto B) {
        constexpr int b = decltype(B)::value;
        if constexpr (b != A && cv(b, ip) != 0) {
          const Real y = cv(b, ip) > 0 ? v : -v;
          if constexpr (k == first_slot<PAIR>(b, A)) j[b] = y; else j[b] += y;
        }
      });
    }
  }
  // Half-way bounce-back (src/dugks.cu:807-823): populations entering through
  // a wall take the value of their opposite, which a pair's other lane holds.
  __device__ __forceinline__ void bounce(bool low_wall, bool high_wall, int half) {
    Real was[NX];
    for (int n = 0; n < NX; n++) was[n] = cross[n];
    static_for<NX>([&](auto M) {
      constexpr int n = decltype(M)::value;
      constexpr int ip = slot_pop(PAIR, cross_slot<PAIR, A>(n));
      if constexpr (PAIR) {
        const Real o = pair_other(was[n]);
        const bool up = (cv(A, ip) > 0) != (half != 0);  // moves toward +A
        cross[n] = (up ? low_wall : high_wall) ? o : was[n];
      } else {
        cross[n] = (cv(A, ip) > 0 ? low_wall : high_wall) ? was[lane_cross<PAIR, A>(OPP[ip])] : was[n];
      }
    });
  }
  // rho (or drho) of the face and s j.
  __device__ __forceinline__ void moments() {
    static_for<NX>([&](auto M) {
      constexpr int n = decltype(M)::value;
      constexpr int ip = slot_pop(PAIR, cross_slot<PAIR, A>(n));
      const Real v = cross[n];
      rho += v;
      static_for<3>([&](auto B) {
        constexpr int b = decltype(B)::value;
        if constexpr (cv(b, ip) != 0) {
          const Real y = cv(b, ip) > 0 ? v : -v;
          if constexpr (b == A && n == 0) j[b] = y; else j[b] += y;
        }
      });
    });
    rho = cell_sum<PAIR>(rho) + rest;
    for (int a = 0; a < 3; a++) j[a] = cell_diff<PAIR>(j[a]);
  }
  // Face collision (f2ruvwh + feq_s, src/dugks.cu:675-709, 1201-1207):
  // rho = sum fbar, u = j/rho + (h/2) F, out = fw1 fbar + (fw2 + fw0 (c-u).F/RT) feq
  // of the lane's crossing populations (SHIFT: the same less their weights,
  // see EqShift); shh = s h/2 and sfw0 = s fw0 (see lane_fbar).
  template <bool SHIFT>
  __device__ __forceinline__ void collide(const Real F[3], Real shh, Real sfw0, Real fw1, Real fw2,
                                          Real (&out)[NX]) {
    moments();
    const Real inv = rcp_real(SHIFT ? Real(1) + rho : rho);
    const Real ux = j[0] * inv + shh * F[0], uy = j[1] * inv + shh * F[1], uz = j[2] * inv + shh * F[2];
    if constexpr (SHIFT) {
      const EqShift<Real> eq(rho, ux, uy, uz, F, fw2, sfw0);
      static_for<NX>([&](auto M) {
        constexpr int n = decltype(M)::value;
        constexpr int ip = slot_pop(PAIR, cross_slot<PAIR, A>(n));
        out[n] = eq.template relax<ip>(-fw2, cross[n], cdot<ip>(F[0], F[1], F[2]));
      });
    } else {
      const EqTerm<Real> eq(rho, ux, uy, uz, F, fw2, sfw0);
      static_for<NX>([&](auto M) {
        constexpr int n = decltype(M)::value;
        constexpr int ip = slot_pop(PAIR, cross_slot<PAIR, A>(n));
        out[n] = eq.template relax<ip>(fw1, cross[n], cdot<ip>(F[0], F[1], F[2]));
      });
    }
  }
};

// ---- a lane's values of a position in LDS ----
// A position holds its slots side by side, STRIDE values apart from the next,
// so that 16-byte accesses move four FP32 or two FP64 values and one address
// register with immediate offsets reaches every neighbour.  STRIDE is an odd
// number of 16-byte units: the eight lanes of a 16-byte pass then start on
// different banks.  (Conflicts remain, 1.1 cycles an LDS instruction in FP32 and
// 2.9 in FP64; candidates are the groups that end in a single value, read 4 or 8
// bytes wide at this stride, and the two halves that share a pass in FP64.)  The
// order keeps the five slots with one sign of c_x or c_y, which
// the reconstruction reads from an upwind neighbour, within two 16-byte
// units (FP32: one unit and one value of the next).
template <bool PAIR>
__host__ __device__ constexpr int lds_index(int k) {
  constexpr int whole[Q] = {16, 0, 9, 5, 13, 17, 18, 4, 8, 3, 12, 1, 10, 2, 11, 6, 14, 7, 15};
  constexpr int pair[10] = {8, 0, 4, 9, 2, 3, 1, 6, 5, 7};
  return PAIR ? pair[k < 10 ? k : 0] : whole[k];
}
constexpr int lds_stride(bool pair) { return pair ? 10 : 20; }

// Slots whose velocity component along axis b is c (c = 2: any non-zero).
template <bool PAIR>
__host__ __device__ constexpr unsigned slot_mask(int b, int c) {
  unsigned m = 0;
  for (int k = 0; k < lane_slots(PAIR); k++) {
    const int v = cv(b, slot_pop(PAIR, k));
    if (c == 2 ? v != 0 : v == c) m |= 1u << k;
  }
  return m;
}

constexpr unsigned all_slots(bool pair) { return (1u << lane_slots(pair)) - 1; }

// Loads the slots of MASK from a position into v (16-byte accesses where two
// or more of a unit's values are wanted).
template <bool PAIR, unsigned MASK, class Real>
__device__ __forceinline__ void lds_get(const Real* p, Real (&v)[lane_slots(PAIR)]) {
  constexpr int VB = 16 / sizeof(Real), NQ = lane_slots(PAIR);
  typedef Real vec __attribute__((ext_vector_type(VB)));
  static_for<lds_stride(PAIR) / VB>([&](auto B) {
    constexpr int b = decltype(B)::value;
    constexpr auto count = [](unsigned mask) {
      int n = 0;
      for (int k = 0; k < lane_slots(PAIR); k++)
        if ((mask >> k & 1) && lds_index<PAIR>(k) / VB == b) n++;
      return n;
    };
    if constexpr (count(MASK) >= 2) {
      const vec x = *reinterpret_cast<const vec*>(p + b * VB);
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        if constexpr ((MASK >> k & 1) && lds_index<PAIR>(k) / VB == b) v[k] = x[lds_index<PAIR>(k) % VB];
      });
    } else if constexpr (count(MASK) == 1) {
      static_for<NQ>([&](auto K) {
        constexpr int k = decltype(K)::value;
        if constexpr ((MASK >> k & 1) && lds_index<PAIR>(k) / VB == b) v[k] = p[lds_index<PAIR>(k)];
      });
    }
  });
}
// Stores all slots of a position.
template <bool PAIR, class Real>
__device__ __forceinline__ void lds_put(Real* p, const Real (&v)[lane_slots(PAIR)]) {
  constexpr int VB = 16 / sizeof(Real), NQ = lane_slots(PAIR);
  typedef Real vec __attribute__((ext_vector_type(VB)));
  static_for<lds_stride(PAIR) / VB>([&](auto B) {
    constexpr int b = decltype(B)::value;
    vec x = {};
    static_for<NQ>([&](auto K) {
      constexpr int k = decltype(K)::value;
      if constexpr (lds_index<PAIR>(k) / VB == b) x[lds_index<PAIR>(k) % VB] = scalar(v[k]);
    });
    *reinterpret_cast<vec*>(p + b * VB) = x;
  });
}
// x[o] = the extrapolation q f(1) + (1 - q) f(2) of f(1) = x[0] (given) and
// f(2) = x[-o], in one plane or two (TWO; both planes' reads first, so that
// their latencies overlap).
template <bool PAIR, bool TWO, class Real>
__device__ __forceinline__ void ghost_line(Real* xa, Real* xb, int o, Real q, const Real (&fa)[lane_slots(PAIR)],
                                           const Real (&fb)[lane_slots(PAIR)]) {
  constexpr int NQ = lane_slots(PAIR);
  Real ga[NQ], gb[NQ], ea[NQ], eb[NQ];
  lds_get<PAIR, all_slots(PAIR)>(xa - o, ga);
  if constexpr (TWO) lds_get<PAIR, all_slots(PAIR)>(xb - o, gb);
  static_for<NQ>([&](auto K) {
    constexpr int k = decltype(K)::value;
    ea[k] = fma_rn(q, fa[k] - ga[k], ga[k]);
  });
  lds_put<PAIR>(xa + o, ea);
  if constexpr (TWO) {
    static_for<NQ>([&](auto K) {
      constexpr int k = decltype(K)::value;
      eb[k] = fma_rn(q, fb[k] - gb[k], gb[k]);
    });
    lds_put<PAIR>(xb + o, eb);
  }
}
// The difference of two-cell sums, (a1 + a2) - (b1 + b2), of the slots of MASK
// (gradient reconstruction; the factor 1/2 of the means is in the coefficients).
// The gradient form is bound by LDS, about 126 16-byte reads a cell and plane.
// 128x96x128 FP32: 104.5 us a step, before 107.3 with the means, the spacing and
// h multiplied in one after the other and the reads in fixed order.
template <bool PAIR, unsigned MASK, class Real>
__device__ __forceinline__ void lds_diff(const Real* a1, const Real* a2, const Real* b1, const Real* b2,
                                         Real (&g)[lane_slots(PAIR)]) {
  constexpr int NQ = lane_slots(PAIR);
  Real x[NQ], y[NQ], z[NQ], w[NQ];
  lds_get<PAIR, MASK>(a1, x);
  lds_get<PAIR, MASK>(a2, y);
  static_for<NQ>([&](auto K) {
    constexpr int k = decltype(K)::value;
    if constexpr (MASK >> k & 1) g[k] = x[k] + y[k];
  });
  lds_get<PAIR, MASK>(b1, z);
  lds_get<PAIR, MASK>(b2, w);
  static_for<NQ>([&](auto K) {
    constexpr int k = decltype(K)::value;
    if constexpr (MASK >> k & 1) g[k] -= z[k] + w[k];
  });
}
// The crossing values of a face, FS values apart from the next face's (an odd
// number of 16-byte units, or with FS not a multiple of one, single values).
template <int NX, int FS, class Real>
__device__ __forceinline__ void flux_get(const Real* p, Real (&v)[NX]) {
  constexpr int VB = 16 / sizeof(Real);
  typedef Real vec __attribute__((ext_vector_type(VB)));
  if constexpr (FS % VB == 0) {
    static_for<(NX + VB - 1) / VB>([&](auto B) {
      constexpr int b = decltype(B)::value;
      const vec x = *reinterpret_cast<const vec*>(p + b * VB);
      for (int q = 0; q < VB; q++)
        if (b * VB + q < NX) v[b * VB + q] = x[q];
    });
  } else {
    for (int n = 0; n < NX; n++) v[n] = p[n];
  }
}
template <int NX, int FS, class Real>
__device__ __forceinline__ void flux_put(Real* p, const Real (&v)[NX]) {
  constexpr int VB = 16 / sizeof(Real);
  typedef Real vec __attribute__((ext_vector_type(VB)));
  if constexpr (FS % VB == 0) {
    static_for<(NX + VB - 1) / VB>([&](auto B) {
      constexpr int b = decltype(B)::value;
      vec x = {};
      for (int q = 0; q < VB; q++)
        if (b * VB + q < NX) x[q] = scalar(v[b * VB + q]);
      *reinterpret_cast<vec*>(p + b * VB) = x;
    });
  } else {
    for (int n = 0; n < NX; n++) p[n] = v[n];
  }
}
