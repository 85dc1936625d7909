// Building blocks of the fused step kernel and the adjoint passes: per-axis
// direction sets, and a face's reconstruction record with the transpose of its
// collision.  Included inside namespace dugks { namespace { ... } } of the
// kernel files.
#pragma once

// populations with a non-zero component along each axis
constexpr int XD[10] = {1, 2, 7, 8, 9, 10, 11, 12, 13, 14};
constexpr int YD[10] = {3, 4, 7, 8, 9, 10, 15, 16, 17, 18};
constexpr int ZD[10] = {5, 6, 11, 12, 13, 14, 15, 16, 17, 18};
constexpr int ZP[5] = {5, 11, 12, 15, 16};  // c_z = +1

template <int A>
__device__ constexpr int dirs(int k) {
  return A == 0 ? XD[k] : (A == 1 ? YD[k] : ZD[k]);
}

// v, opaque to the optimiser: what is formed from it is formed at its use and
// does not live in registers across the plane loop.
template <class T>
__device__ __forceinline__ T here(T v) {
  asm volatile("" : "+v"(v));
  return v;
}

// (1 - m) a + m b, evaluated as a + m (b - a): a constant stays exactly
// constant whatever the rounding of m.  In FP32, (1 - m) and m rounded apart
// do not sum to 1, which on a stretched axis biases every face value by a
// fixed fraction of its size; the flux divergence turns that into a steady
// source that shifts the mean flow (the 10^4-step channel's FP32 profiles
// drift by up to 3e-3 in the other form).
template <class Real>
__device__ __forceinline__ Real lerp_(Real a, Real b, Real m) {
  return fma_rn(m, b - a, a);
}

template <class Real>
__device__ __forceinline__ void ambient_force(const KParams& P, Real F[3]) {
  F[0] = (Real)P.famb_dev[0];
  F[1] = (Real)P.famb_dev[1];
  F[2] = (Real)P.famb_dev[2];
}

// Index of population ip in the crossing set of axis A (-1 if it does not
// cross a face normal to A).
template <int A>
__device__ constexpr int cross_index(int ip) {
  for (int k = 0; k < 10; k++)
    if (dirs<A>(k) == ip) return k;
  return -1;
}

// Transpose of the wall bounce-back: a population that entered through a
// wall took its opposite's value, so its cotangent moves to that opposite.
template <class Real, int A>
__device__ __forceinline__ void bounce_transpose(const Real (&post)[Q], bool low_wall, bool high_wall,
                                                 Real (&lam)[Q]) {
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    Real v = post[ip];
    if constexpr (cv(A, ip) != 0) {
      const bool in = (low_wall && cv(A, ip) > 0) || (high_wall && cv(A, ip) < 0);
      const bool opp_in = (low_wall && cv(A, ip) < 0) || (high_wall && cv(A, ip) > 0);
      if (in) v = Real(0);
      if (opp_in) v += post[OPP[ip]];
    }
    lam[ip] = v;
  });
}

// Cotangents of the 19 reconstructed values of a face normal to axis A from
// the transposed collision's coefficients: fw1 mu_p + Ac + B.c_p, then the
// transposed bounce-back.
template <class Real, int A>
__device__ __forceinline__ void expand_cotangents(const Real (&mu)[10], Real Ac, const Real (&B)[3], Real fw1,
                                                  bool low_wall, bool high_wall, Real (&lam)[Q]) {
  Real post[Q];
  static_for<Q>([&](auto I) {
    constexpr int ip = decltype(I)::value;
    constexpr int k = cross_index<A>(ip);
    Real v = plus_cdot<ip>(Ac, B[0], B[1], B[2]);
    if constexpr (k >= 0) v += fw1 * mu[k];
    post[ip] = v;
  });
  bounce_transpose<Real, A>(post, low_wall, high_wall, lam);
}

// The compact form of the adjoint's face data.  The cotangent of a
// reconstructed value of a face is fw1 mu_p + Ac + B.c_p, and mu (of the
// crossing populations) is a difference of lam' between the two cells beside
// the face; so a face record is (Ac, B), four values side by side, one array
// per axis ([3][slot][4]), and the gather forms mu from the lam' it reads
// anyway.  Behind the records (storage in the arithmetic type) lie two regions
// of (rho, j) of every cell ([2][N][4]).
template <class Real>
__device__ __forceinline__ RawBuf face_records(const void* faces, int axis, long long eN) {
  return RawBuf(static_cast<const Real*>(faces) + axis * kCompact * eN,
                (unsigned)(kCompact * eN * (long long)sizeof(Real)));
}
template <class Real>
__device__ __forceinline__ RawBuf cell_records(const void* faces, int region, long long eN, long long N) {
  return RawBuf(static_cast<const Real*>(faces) + 3 * kCompact * eN + region * 4 * N,
                (unsigned)(4 * N * (long long)sizeof(Real)));
}

// First population that does not cross a face normal to axis A and has a
// non-zero component b (b != A); the moments of a face start from it.
template <int A>
__device__ constexpr int first_tangential(int b) {
  for (int ip = 0; ip < Q; ip++)
    if (cv(A, ip) == 0 && cv(b, ip) != 0) return ip;
  return -1;
}

// Reconstructed populations of one face normal to axis A, held as the ten
// values that cross the face plus the partial moments of the nine that do
// not (those only enter rho and j of the face collision).  The populations
// are put in order 0..18 (the rest population first); every moment starts
// from its first term, so no sum adds to a zero.
template <class Real, int A>
struct Face {
  Real cross[10];
  Real rho, j[3];
  template <int ip>
  __device__ __forceinline__ void put(Real v) {
    constexpr int k = cross_index<A>(ip);
    if constexpr (k >= 0) {
      cross[k] = v;
    } else {
      if constexpr (ip == 0) rho = v; else rho += v;
      static_for<3>([&](auto B) {
        constexpr int b = decltype(B)::value;
        if constexpr (b != A && cv(b, ip) != 0) {
          const Real s = cv(b, ip) > 0 ? v : -v;
          if constexpr (ip == first_tangential<A>(b)) j[b] = s; else j[b] += s;
        }
      });
    }
  }
  // rho and j of the face: the partial moments plus the crossing populations
  // (j_A starts from the first crossing population, c_A = +1)
  __device__ __forceinline__ void moments() {
    static_for<10>([&](auto K) {
      constexpr int k = decltype(K)::value;
      constexpr int ip = dirs<A>(k);
      const Real v = cross[k];
      rho += v;
      static_for<3>([&](auto B) {
        constexpr int b = decltype(B)::value;
        if constexpr (cv(b, ip) != 0) {
          const Real s = cv(b, ip) > 0 ? v : -v;
          if constexpr (b == A && k == 0) j[b] = s; else j[b] += s;
        }
      });
    });
  }
  // Half-way bounce-back: populations entering the domain through a wall
  // take the value of their opposite (src/dugks.cu:807-823).
  __device__ __forceinline__ void bounce(bool low_wall, bool high_wall) {
    if (low_wall) {
      static_for<10>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = dirs<A>(k);
        if constexpr (cv(A, ip) > 0) cross[k] = cross[cross_index<A>(OPP[ip])];
      });
    }
    if (high_wall) {
      static_for<10>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ip = dirs<A>(k);
        if constexpr (cv(A, ip) < 0) cross[k] = cross[cross_index<A>(OPP[ip])];
      });
    }
  }
  // The transposed collision up to its equilibrium coefficients: the
  // cotangent of reconstructed value p is fw1 mu_p + Ac + B.c_p (mu_p = 0
  // for the populations that do not cross), before the bounce transpose.
  // FORCE: also adds the cotangent of the face's force F to gF[0..2]
  // (through the equilibrium's explicit F and through u = j/rho + (h/2) F).
  template <bool FORCE = false>
  __device__ __forceinline__ void adjoint_coeffs(const Real F[3], Real hdt, Real fw0, Real fw2,
                                                 const Real (&mu)[10], Real& Ac, Real (&B)[3],
                                                 double* gF = nullptr) {
    moments();
    const Real inv = rcp_real(rho);
    const Real hh = Real(0.5) * hdt;
    const Real ut[3] = {j[0] * inv, j[1] * inv, j[2] * inv};
    const Real u[3] = {ut[0] + hh * F[0], ut[1] + hh * F[1], ut[2] + hh * F[2]};
    Real lq[Q];
    static_for<Q>([&](auto I) {
      constexpr int ip = decltype(I)::value;
      constexpr int k = cross_index<A>(ip);
      if constexpr (k >= 0) lq[ip] = mu[k]; else lq[ip] = Real(0);
    });
    Real g_rho, g_u[3], g_F[3];
    feq_adjoint<Real>(lq, fw2, fw0, rho, u, F, g_rho, g_u, g_F, Crossing<A>{});
    Ac = g_rho - (g_u[0] * ut[0] + g_u[1] * ut[1] + g_u[2] * ut[2]) * inv;
    B[0] = g_u[0] * inv;
    B[1] = g_u[1] * inv;
    B[2] = g_u[2] * inv;
    if constexpr (FORCE) {
      gF[0] += (double)(g_F[0] + hh * g_u[0]);
      gF[1] += (double)(g_F[1] + hh * g_u[1]);
      gF[2] += (double)(g_F[2] + hh * g_u[2]);
    }
  }
  // Transpose of collide (after bounce) and bounce: given the cotangent mu
  // of the ten outputs, the cotangent of the 19 reconstructed values before
  // bounce-back.  d out_q / d fbar_p = fw1 delta_qp + (d/d rho + c_p.d/d j)
  // of the equilibrium term, so lam_p = fw1 mu_p + A + B.c_p; a population
  // that entered through a wall took its opposite's value, so its cotangent
  // moves to that opposite.
  template <bool FORCE = false>
  __device__ __forceinline__ void adjoint(const Real F[3], Real hdt, Real fw0, Real fw1, Real fw2,
                                          const Real (&mu)[10], bool low_wall, bool high_wall, Real (&lam)[Q],
                                          double* gF = nullptr) {
    Real Ac, B[3];
    adjoint_coeffs<FORCE>(F, hdt, fw0, fw2, mu, Ac, B, gF);
    expand_cotangents<Real, A>(mu, Ac, B, fw1, low_wall, high_wall, lam);
  }
};

