// Face numerics, included into alpaca::exact and alpaca::fast (see
// fv_device.h).  Real type R is double (FP64) or float (mixed form).  For
// R = double every expression keeps the reference's operation order, so the
// exact namespace reproduces it bit for bit.  Citations name the reference
// file:line each function follows.

template <typename R> __device__ __forceinline__ R smin(R a, R b) { return (b < a) ? b : a; }
template <typename R> __device__ __forceinline__ R smax(R a, R b) { return (a < b) ? b : a; }

// FP64 division a/b by Newton-Raphson on the hardware reciprocal: two
// iterations on r ~ 1/b (r += r(1 - b r)), then one residual correction of
// the quotient (q += r(a - b q)); each residual is exact in an FMA, so the
// result is within 1 ulp of a/b for normal operands.
__device__ __forceinline__ double nr_div64(double a, double b) {
  double r = __builtin_amdgcn_rcp(b);
  double e = __builtin_fma(-b, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-b, r, 1.0);
  r = __builtin_fma(r, e, r);
  double const q = a * r;
  double const rem = __builtin_fma(-b, q, a);
  return __builtin_fma(rem, r, q);
}

// FP64 division of the fast namespace: one Newton step on the hardware
// reciprocal, then the residual correction of the quotient.  v_rcp_f64 is
// within 2^-24 of 1/b (largest relative error 2^-24.4 over 16.7 M operands of
// exponents -200..200, including divisors just below a power of two), the
// step leaves at most about 2^-48, and the correction (residual exact in an
// FMA) squares that again, so the result is within 1 ulp of a/b for normal
// operands.  Random pairs come out correctly rounded (all 16.7 M of them);
// quotients within about 2^-90 of a rounding midpoint can round the other
// way.
__device__ __forceinline__ double fast_div64(double a, double b) {
  double r = __builtin_amdgcn_rcp(b);
  double const e = __builtin_fma(-b, r, 1.0);
  r = __builtin_fma(r, e, r);
  double const q = a * r;
  double const rem = __builtin_fma(-b, q, a);
  return __builtin_fma(rem, r, q);
}

// FP64 square root by the coupled Newton iteration for g ~ sqrt(x) and
// h ~ 1/(2 sqrt(x)) from the hardware reciprocal square root, with a final
// residual correction (x - g^2 exact in an FMA).  sqrt(0) = 0.
__device__ __forceinline__ double nr_sqrt64(double x) {
  double const r = __builtin_amdgcn_rsq(x);
  double g = x * r;
  double h = 0.5 * r;
  double const e = __builtin_fma(-g, h, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  double const d = __builtin_fma(-g, g, x);
  g = __builtin_fma(d, h, g);
  return x == 0.0 ? 0.0 : g;
}

// Divisors whose reciprocal lies within about 2^-100 (relative) of a rounding
// midpoint: b = 2^e (2 - k 2^-52) for small odd k, whose significand has its
// top 20 bits set (a density just below a power of two after round-off is
// one; so are the Roe-averaged density and sqrt(rho_i) + sqrt(rho_n) of two
// such cells).  For them the two Newton steps of the hardware division sequence can
// leave the reciprocal one ulp from RN(1/b), and a quotient that also lies
// within about 2^-105 of a midpoint then rounds the wrong way (0x1.6666666666663p-2
// / 0x1.ffffffffffffbp-4 gives 2.8 instead of x86's 2.8000000000000003).
// Other divisors' reciprocals come out of the sequence correctly rounded, and
// with a correctly rounded reciprocal its final residual correction rounds the
// quotient correctly.
__device__ __forceinline__ bool recip_hard(double b) {
  return ((unsigned)((unsigned long long)__double_as_longlong(b) >> 32) & 0xFFFFFu) == 0xFFFFFu;
}

// The correctly rounded quotient from q, a quotient within one ulp of a/b:
// of q and its neighbour toward a/b, the one whose residual a - b q' is
// smaller (both residuals are exact in an FMA when |a| >= 2^-960; the distance
// to a/b is |residual| / |b| for both).  A tie cannot occur: no quotient of
// two doubles lies exactly on a midpoint.
__device__ __forceinline__ double div_round(double a, double b, double q) {
  if (!(__builtin_fabs(q) <= 1.7976931348623157e308) || q == 0.0 ||
      !(__builtin_fabs(a) >= 0x1p-960))
    return q;
  double const r = __builtin_fma(-b, q, a);
  if (r == 0.0) return q;
  bool const above = (r > 0.0) == (b > 0.0);  // a/b > q
  long long const qi = __double_as_longlong(q);
  double const q2 = __longlong_as_double(above == (q > 0.0) ? qi + 1 : qi - 1);
  double const r2 = __builtin_fma(-b, q2, a);
  return __builtin_fabs(r2) < __builtin_fabs(r) ? q2 : q;
}

// The WENO5 weight divisions c / x in the exact form: x = (s + 1e-6)^2 in
// [1e-12, 2^700) and c in {0.1, 0.6, 0.3} (and 1 / (a1 + a2 + a3) >= 2^-704),
// where the hardware division sequence scales nothing and fixes up nothing,
// so it is exactly its core nr_div64.  These 40 divisions per face take no
// hard-reciprocal check (it would cost about 3% of the exact stage kernel's time): their
// divisors are smoothness indicators, not state values, and one of them would
// have to lie within 2^-48 below a power of two, with the quotient within
// about 2^-105 of a midpoint, to round differently from x86.
__device__ __forceinline__ double weno_div(double c, double x) { return nr_div64(c, x); }

// Division and square root: the compiler's FP64 sequences (what a/b and
// sqrt(x) compile to) in the exact namespace; Newton-Raphson FP64 in the fast
// namespace; hardware reciprocal and square root (about 1 ulp) for the FP32
// part of the mixed form.
template <typename R> __device__ __forceinline__ R fdiv(R a, R b) {
  if constexpr (std::is_same<R, float>::value)
    return a * __builtin_amdgcn_rcpf(b);
  else if constexpr (kFastArith)
    return fast_div64(a, b);
  else {
    // The compiler's sequence, correctly rounded also for the divisors with a
    // hard reciprocal.
    double const q = a / b;
    return __builtin_expect(recip_hard(b), 0) ? div_round(a, b, q) : q;
  }
}
template <typename R> __device__ __forceinline__ R dsqrt(R x) {
  if constexpr (std::is_same<R, float>::value) {
    return __builtin_amdgcn_sqrtf(x);
  } else if constexpr (kFastArith) {
    return nr_sqrt64(x);
  } else {
    // The compiler's square root.  For finite x >= 2^-767 (high word in
    // [0x10000000, 0x7FF00000)) the hardware sequence scales nothing and its
    // zero/infinity select passes the iterate through, so it reduces to this
    // core (v_rsq, then Goldschmidt refinement of g ~ sqrt(x) and
    // h ~ 1/(2 sqrt(x)) with two residual corrections): the same bits with 8
    // fewer instructions.  Other arguments (0, tiny, negative, inf, NaN) take
    // the full sequence.
    unsigned const hw = (unsigned)((unsigned long long)__double_as_longlong(x) >> 32);
    if (__builtin_expect(hw - 0x10000000u < 0x6FF00000u, 1)) {
      double const r = __builtin_amdgcn_rsq(x);
      double g = x * r;
      double h = r * 0.5;
      double const e = __builtin_fma(-h, g, 0.5);
      g = __builtin_fma(g, e, g);
      double d = __builtin_fma(-g, g, x);
      h = __builtin_fma(h, e, h);
      g = __builtin_fma(d, h, g);
      d = __builtin_fma(-g, g, x);
      return __builtin_fma(d, h, g);
    }
    return __builtin_sqrt(x);
  }
}

// ConsistencyManagedSum, full symmetry (mathematical_functions.h:79-91).
// For finite a, b, c the three orderings are never NaN (two roundings cannot
// meet an opposite infinity) and are -0 all together or not at all (a rounded
// sum is -0 only when both addends are -0), so the hardware minimum/maximum
// (one instruction each) pick exactly what std::min/std::max pick.
template <typename R> __device__ __forceinline__ R cms3(R a, R b, R c) {
  R const s1 = (a + b) + c;
  R const s2 = (a + c) + b;
  R const s3 = (b + c) + a;
  R mn, mx;
  if constexpr (std::is_same<R, float>::value) {
    mn = __builtin_fminf(__builtin_fminf(s1, s2), s3);
    mx = __builtin_fmaxf(__builtin_fmaxf(s1, s2), s3);
  } else {
    mn = __builtin_fmin(__builtin_fmin(s1, s2), s3);
    mx = __builtin_fmax(__builtin_fmax(s1, s2), s3);
  }
  return R(0.5) * (mn + mx);
}

// DimensionAwareConsistencyManagedSum (mathematical_functions.h:100-108).
template <int DIM, typename R> __device__ __forceinline__ R dams(R a, R b, R c) {
  if constexpr (DIM == 2) {
    (void)c;
    return a + b;
  } else {
    return cms3(a, b, c);
  }
}

// CalculatePressure<false> (generic_stiffened_gas.h:40-58).  The recovery
// p = -gamma*B + (gamma-1)(E - |m|^2/(2 rho)) always runs in FP64: the
// difference cancels at high Mach number.
template <int DIM>
__device__ __forceinline__ double eos_pressure64(double gamma, double b, double rho, double mx,
                                                 double my, double mz, double e) {
  double const q = 0.5 * dams<DIM>(mx * mx, my * my, mz * mz);
  return -gamma * b + (gamma - 1.0) * (e - fdiv(q, rho));
}
template <int DIM, typename R>
__device__ __forceinline__ R eos_pressure(R gamma, R b, R rho, R mx, R my, R mz, R e) {
  return R(eos_pressure64<DIM>(double(gamma), double(b), double(rho), double(mx), double(my),
                               double(mz), double(e)));
}

// CalculateSpeedOfSound<false> (generic_stiffened_gas.h:84-97).
template <typename R> __device__ __forceinline__ R eos_sos(R gamma, R b, R rho, R p) {
  return dsqrt(fdiv(gamma * (p + b), rho));
}

// ComputePsi (stiffened_gas.cpp:127-130).
template <typename R> __device__ __forceinline__ R eos_psi(R gamma, R b, R p, R one_rho) {
  return (p + gamma * b) * one_rho;
}

template <typename R> struct Prim {
  R rho, p, vel[3];
};

// ConservativesToPrimeStates (prime_state_handler.h:279-370).
template <int DIM, typename R>
__device__ __forceinline__ void cons_to_prim(R gamma, R b, const R *c, Prim<R> &o) {
  o.rho = c[kMass];
  R const one_density = fdiv(R(1.0), c[kMass]);
  o.vel[0] = c[kMomX] * one_density;
  o.vel[1] = c[kMomX + 1] * one_density;
  if constexpr (DIM == 3)
    o.vel[2] = c[kMomX + 2] * one_density;
  else
    o.vel[2] = R(0.0);
  R const mz = DIM == 3 ? c[kMomX + DIM - 1] : R(0.0);
  o.p = eos_pressure<DIM>(gamma, b, c[kMass], c[kMomX], c[kMomX + 1], mz, c[kEnergy]);
}

// Per-cell quantities the Roe average needs, from the cell's FP64
// conservatives: 1/rho, prime velocities and pressure
// (prime_state_handler.h:279-370), psi (stiffened_gas.cpp:127-130) and the
// enthalpy with its EOS-recomputed pressure (stiffened_gas.cpp:80-87), as
// eigendecomposition.h:266-283 reads them.
template <typename R> struct CellQ {
  R rho, one_rho, vel[3], p, psi, H;
};

template <int DIM, typename R>
__device__ __forceinline__ void cell_quantities(double gamma, double b, const double *c,
                                                CellQ<R> &q) {
  Prim<double> p;
  cons_to_prim<DIM, double>(gamma, b, c, p);
  double const one_rho = fdiv(1.0, c[kMass]);
  double const mz = DIM == 3 ? c[kMomX + DIM - 1] : 0.0;
  double const H = fdiv(c[kEnergy] + eos_pressure64<DIM>(gamma, b, c[kMass], c[kMomX],
                                                         c[kMomX + 1], mz, c[kEnergy]),
                        c[kMass]);
  q.rho = R(c[kMass]);
  q.one_rho = R(one_rho);
  q.vel[0] = R(p.vel[0]);
  q.vel[1] = R(p.vel[1]);
  q.vel[2] = R(p.vel[2]);
  q.p = R(p.p);
  q.psi = R(eos_psi<double>(gamma, b, p.p, one_rho));
  q.H = R(H);
}

// What the Roe average takes from a cell (eigendecomposition.h:266-283): the
// square root of the density, the velocities, psi, the enthalpy and p / rho.
// A face needs them of its two inner cells, so a cell's are used by six
// faces: the plane-marching kernels form them once per cell and keep them in
// LDS (PackedQ), the tile kernels form them per face.  The same operations on
// the same values either way.
template <typename R> struct FaceQ {
  R rho, sq, vel[3], psi, H, pod;
};

template <int DIM, typename R>
__device__ __forceinline__ FaceQ<R> face_quantities(double gamma, double b, const double *c) {
  CellQ<R> q;
  cell_quantities<DIM, R>(gamma, b, c, q);
  FaceQ<R> f;
  f.rho = q.rho;
  f.sq = dsqrt(q.rho);
  f.vel[0] = q.vel[0];
  f.vel[1] = q.vel[1];
  f.vel[2] = q.vel[2];
  f.psi = q.psi;
  f.H = q.H;
  f.pod = q.p * q.one_rho;
  return f;
}

// A cell's FP64 FaceQ as kPackedQ values: 1/rho is kept and the velocities are formed from the
// stencil's momenta again (one exact repetition of a product each).
constexpr int kPackedQ = 5;

// Writes the FaceQ of the cell with conservatives c to q[0], q[STRIDE], ...
template <int DIM, int STRIDE>
__device__ __forceinline__ void store_packed(double gamma, double b, const double *c, double *q) {
  CellQ<double> w;
  cell_quantities<DIM, double>(gamma, b, c, w);
  q[0] = dsqrt(w.rho);
  q[STRIDE] = w.one_rho;
  q[2 * STRIDE] = w.psi;
  q[3 * STRIDE] = w.H;
  q[4 * STRIDE] = w.p * w.one_rho;
}

template <int DIM, int STRIDE>
__device__ __forceinline__ FaceQ<double> load_packed(const double *q, const double *c) {
  FaceQ<double> f;
  double const one_rho = q[STRIDE];
  f.rho = c[kMass];
  f.sq = q[0];
  f.vel[0] = c[kMomX] * one_rho;
  f.vel[1] = c[kMomX + 1] * one_rho;
  f.vel[2] = DIM == 3 ? c[kMomX + DIM - 1] * one_rho : 0.0;
  f.psi = q[2 * STRIDE];
  f.H = q[3 * STRIDE];
  f.pod = q[4 * STRIDE];
  return f;
}

// The FP64-with-FMA form takes its own expressions for the reconstruction and
// the Riemann problem (fewer operations, no bit parity).
template <typename R> constexpr bool kLean = kFastArith && std::is_same<R, double>::value;
// The exact FP64 form.
template <typename R> constexpr bool kExact = !kFastArith && std::is_same<R, double>::value;

// WENO5::ApplyImplementation (weno5.h:88-158) on ordered v1..v5, mixed form.
template <typename R> __device__ __forceinline__ R weno5(R v1, R v2, R v3, R v4, R v5) {
  R const c_s1 = R(13.0 / 12.0), c_s2 = R(0.25), eps = R(1.0e-6);
  R const s11 = R(1.0) * v1 + R(-2.0) * v2 + R(1.0) * v3;
  R const s12 = R(1.0) * v1 + R(-4.0) * v2 + R(3.0) * v3;
  R const s1 = c_s1 * s11 * s11 + c_s2 * s12 * s12;
  R const s21 = R(1.0) * v2 + R(-2.0) * v3 + R(1.0) * v4;
  R const s22 = R(1.0) * v2 + R(-1.0) * v4;
  R const s2 = c_s1 * s21 * s21 + c_s2 * s22 * s22;
  R const s31 = R(1.0) * v3 + R(-2.0) * v4 + R(1.0) * v5;
  R const s32 = R(3.0) * v3 + R(-4.0) * v4 + R(1.0) * v5;
  R const s3 = c_s1 * s31 * s31 + c_s2 * s32 * s32;
  R const x1 = (s1 + eps) * (s1 + eps);
  R const x2 = (s2 + eps) * (s2 + eps);
  R const x3 = (s3 + eps) * (s3 + eps);
  R const p1 = R(2.0 / 6.0) * v1 + R(-7.0 / 6.0) * v2 + R(11.0 / 6.0) * v3;
  R const p2 = R(-1.0 / 6.0) * v2 + R(5.0 / 6.0) * v3 + R(2.0 / 6.0) * v4;
  R const p3 = R(2.0 / 6.0) * v3 + R(5.0 / 6.0) * v4 + R(-1.0 / 6.0) * v5;
  R const a1 = fdiv(R(0.1), x1);
  R const a2 = fdiv(R(0.6), x2);
  R const a3 = fdiv(R(0.3), x3);
  R const one_a_sum = fdiv(R(1.0), a1 + a2 + a3);
  R const w1 = a1 * one_a_sum;
  R const w2 = a2 * one_a_sum;
  R const w3 = a3 * one_a_sum;
  return w1 * p1 + w2 * p2 + w3 * p3;
}

// weno5 in the exact FP64 form, in two halves: the smoothness indicators and
// polynomials, then the weights.  Two products of the reference are fused
// where a power of two makes the fused form round the same: v1 + (-2 v2) and
// v1 + (-4 v2) (the product is exact) and t + 0.25 (s s) for (0.25 s) s
// (scaling by 0.25 changes no significand, and the sum only enters s + 1e-6).
// 13 fewer instructions per pair of reconstructions; the same bits for
// |v| < 2^1022.
struct Weno5 {
  double x[3], p[3];
  __device__ __forceinline__ Weno5(double v1, double v2, double v3, double v4, double v5) {
    double const c_s1 = 13.0 / 12.0, eps = 1.0e-6;
    double const t3 = 3.0 * v3;
    double const s11 = __builtin_fma(-2.0, v2, v1) + v3;
    double const s12 = __builtin_fma(-4.0, v2, v1) + t3;
    double const s1 = __builtin_fma(0.25, s12 * s12, c_s1 * s11 * s11);
    double const s21 = __builtin_fma(-2.0, v3, v2) + v4;
    double const s22 = v2 - v4;
    double const s2 = __builtin_fma(0.25, s22 * s22, c_s1 * s21 * s21);
    double const s31 = __builtin_fma(-2.0, v4, v3) + v5;
    double const s32 = __builtin_fma(-4.0, v4, t3) + v5;
    double const s3 = __builtin_fma(0.25, s32 * s32, c_s1 * s31 * s31);
    x[0] = (s1 + eps) * (s1 + eps);
    x[1] = (s2 + eps) * (s2 + eps);
    x[2] = (s3 + eps) * (s3 + eps);
    p[0] = (2.0 / 6.0) * v1 + (-7.0 / 6.0) * v2 + (11.0 / 6.0) * v3;
    p[1] = (-1.0 / 6.0) * v2 + (5.0 / 6.0) * v3 + (2.0 / 6.0) * v4;
    p[2] = (2.0 / 6.0) * v3 + (5.0 / 6.0) * v4 + (-1.0 / 6.0) * v5;
  }
  // x_k = (s_k + 1e-6)^2 >= 1e-12 (s_k >= 0 or NaN).  The positive x_k order
  // like the high words of their bit patterns; NaN and infinity lie above.
  __device__ __forceinline__ unsigned top() const {
    auto hi = [](double v) { return (unsigned)((unsigned long long)__double_as_longlong(v) >> 32); };
    return __builtin_elementwise_max(__builtin_elementwise_max(hi(x[0]), hi(x[1])), hi(x[2]));
  }
  // CORE: every x_k is below 2^700.  The hardware's correctly rounded division
  // of 0.1, 0.6, 0.3 by x_k and of 1 by a1 + a2 + a3 (>= 2^-704) then scales
  // nothing and fixes up nothing, so it is exactly its Newton-Raphson core
  // nr_div64 (v_rcp, two refinements, quotient, one residual correction):
  // same bits, 3 fewer instructions per division.
  template <bool CORE> __device__ __forceinline__ double value() const {
    auto div = [](double a, double b) { return CORE ? weno_div(a, b) : fdiv(a, b); };
    double const a1 = div(0.1, x[0]);
    double const a2 = div(0.6, x[1]);
    double const a3 = div(0.3, x[2]);
    double const one_a_sum = div(1.0, a1 + a2 + a3);
    double const w1 = a1 * one_a_sum;
    double const w2 = a2 * one_a_sum;
    double const w3 = a3 * one_a_sum;
    return w1 * p[0] + w2 * p[1] + w3 * p[2];
  }
};

// UpwindLeft {0,+1} of l and UpwindRight {1,-1} of r (apply_wrapper.h:48-58) in
// the exact form.  Returns whether every x_k was in the core's range; l[0..4]
// and r[1..5] are then finite.  PAIRED: one range check for both; otherwise
// one after the other.  The split decides what the register allocator holds
// at once (the finite-volume face, with one projection per field, takes 241 VGPRs
// paired and 224 in sequence).
template <bool PAIRED>
__device__ __forceinline__ bool weno_pair_exact(const double *l, const double *r, double &left,
                                                double &right) {
  auto in_core = [](unsigned top) { return top < 0x6BB00000u; };  // 2^700
  if constexpr (PAIRED) {
    Weno5 const a(l[0], l[1], l[2], l[3], l[4]), b(r[5], r[4], r[3], r[2], r[1]);
    bool const core = in_core(__builtin_elementwise_max(a.top(), b.top()));
    if (__builtin_expect(core, 1)) {
      left = a.template value<true>();
      right = b.template value<true>();
    } else {
      left = a.template value<false>();
      right = b.template value<false>();
    }
    return core;
  } else {
    auto one = [&](Weno5 const &a, double &v) {
      bool const core = in_core(a.top());
      if (__builtin_expect(core, 1))
        v = a.template value<true>();
      else
        v = a.template value<false>();
      return core;
    };
    bool const cl = one(Weno5(l[0], l[1], l[2], l[3], l[4]), left);
    bool const cr = one(Weno5(r[5], r[4], r[3], r[2], r[1]), right);
    return cl && cr;
  }
}

// WENO5 in the FP64-with-FMA form, from the first differences d1..d4 and the
// second differences D1..D3 of the five values, relative to the middle value:
//   4 s_k = 13/3 D_k^2 + m_k^2, m = (3 d2 - d1, d2 + d3, 3 d3 - d4),
//   6 (p_k - v3) = e_k = (5 d2 - 2 d1, d2 + 2 d3, 4 d3 - d4),
// and the weights w_k = d_k / x_k, x_k = (s_k + 1e-6)^2, over the common
// denominator x1 x2 x3, so that one division serves all:
//   v = v3 + 1/6 (z1 e1 + 6 z2 e2 + 3 z3 e3) / (z1 + 6 z2 + 3 z3),
// z1 = x2 x3, z2 = x1 x3, z3 = x1 x2.  The four times scaled s_k + 1e-6 are
// scaled by a power of two r (which changes no significand) so that the
// largest lies in [1/8, 1]; er = 4e-6 r is kept at least 2^-250, so the x_k
// stay in [2^-500, 1] and the z_k normal.  An infinite s_k is clamped to 1 (its
// stencil gets a weight 2^-500 of the others', as its d_k / x_k = 0 would); a
// NaN still makes the result NaN through its e_k.
// The left and right reconstructions of one array share the differences, the
// D terms and the scale: 96 instructions for both, against 133 with the
// candidate polynomials and indicators formed from the values.
struct WenoScale {
  double r, er;
  __device__ __forceinline__ explicit WenoScale(double smax) {
    unsigned h = (unsigned)((unsigned long long)__double_as_longlong(smax) >> 32);
    h = __builtin_elementwise_min(__builtin_elementwise_max(h, 0x3EE00000u), 0x7FB00000u);
    r = __longlong_as_double((long long)((unsigned long long)(0x7FC00000u - (h & 0x7FF00000u)) << 32));
    er = __builtin_fmax(4.0e-6 * r, 0x1p-250);
  }
};
__device__ __forceinline__ double max3(double a, double b, double c) {
  return __builtin_fmax(__builtin_fmax(a, b), c);
}
// 6 (v - v3): indicators s_k (times four), differences d1..d4.
__device__ __forceinline__ double weno_lean(const WenoScale &w, double s1, double s2, double s3,
                                            double d1, double d2, double d3, double d4) {
  auto x = [&w](double s) {
    double const t = __builtin_fmin(__builtin_fmax(s * w.r + w.er, 0.0), 1.0);
    return t * t;
  };
  double const x1 = x(s1), x2 = x(s2), x3 = x(s3);
  double const z1 = x2 * x3, z2 = 6.0 * (x1 * x3), z3 = 3.0 * (x1 * x2);
  double const num = z1 * (5.0 * d2 - 2.0 * d1) + z2 * (d2 + 2.0 * d3) + z3 * (4.0 * d3 - d4);
  return fast_div64(num, z1 + z2 + z3);
}
__device__ __forceinline__ void weno_pair_lean(const double *a, double &left, double &right) {
  double const d0 = a[1] - a[0], d1 = a[2] - a[1], d2 = a[3] - a[2], d3 = a[4] - a[3],
               d4 = a[5] - a[4];
  double const c = 13.0 / 3.0;
  double const D0 = d1 - d0, D1 = d2 - d1, D2 = d3 - d2, D3 = d4 - d3;
  double const C0 = c * D0, C1 = c * D1, C2 = c * D2, C3 = c * D3;
  auto ind = [](double D, double C, double m) { return D * C + m * m; };
  double const l1 = ind(D0, C0, 3.0 * d1 - d0), l2 = ind(D1, C1, d1 + d2), l3 = ind(D2, C2, 3.0 * d2 - d3);
  double const r1 = ind(D3, C3, 3.0 * d3 - d4), r2 = ind(D2, C2, d3 + d2), r3 = ind(D1, C1, 3.0 * d2 - d1);
  WenoScale const w(__builtin_fmax(max3(l1, l2, l3), max3(r1, r2, r3)));
  left = a[2] + (1.0 / 6.0) * weno_lean(w, l1, l2, l3, d0, d1, d2, d3);
  right = a[3] - (1.0 / 6.0) * weno_lean(w, r1, r2, r3, d4, d3, d2, d1);
}
__device__ __forceinline__ double weno_one_lean(double v1, double v2, double v3, double v4, double v5) {
  double const d1 = v2 - v1, d2 = v3 - v2, d3 = v4 - v3, d4 = v5 - v4;
  double const c = 13.0 / 3.0;
  double const D1 = d2 - d1, D2 = d3 - d2, D3 = d4 - d3;
  auto ind = [c](double D, double m) { return D * (c * D) + m * m; };
  double const s1 = ind(D1, 3.0 * d2 - d1), s2 = ind(D2, d2 + d3), s3 = ind(D3, 3.0 * d3 - d4);
  WenoScale const w(max3(s1, s2, s3));
  return v3 + (1.0 / 6.0) * weno_lean(w, s1, s2, s3, d1, d2, d3, d4);
}

// The left reconstruction of l and the right one of r (apply_wrapper.h:48-58) in the
// contracting forms.
template <typename R>
__device__ __forceinline__ void weno_pair(const R *l, const R *r, R &left, R &right) {
  if constexpr (kLean<R>) {
    left = weno_one_lean(l[0], l[1], l[2], l[3], l[4]);
    right = weno_one_lean(r[5], r[4], r[3], r[2], r[1]);
  } else {
    left = weno5<R>(l[0], l[1], l[2], l[3], l[4]);
    right = weno5<R>(r[5], r[4], r[3], r[2], r[1]);
  }
}

template <int NE, typename R> struct Eig {
  R L[NE][NE];
  R Rm[NE][NE];
  R lam[NE];
  // Roe averages the right eigenvectors are built from when they are built
  // late (kDeferRight below).
  R u, v, w, c, H, g, rho_roe;
  bool ok;
};

// Structural zeros of the left Roe eigenvectors (eigendecomposition.h:238-466):
// rows 1 and 2 (the shear waves) hold only the mass and their own transverse
// momentum.  The exact form leaves these products out where the stencil is
// finite; the mixed form keeps its measured accuracy by forming them.
template <int DIM, int DIR> __device__ __forceinline__ constexpr bool left_zero(int n, int c) {
  constexpr int M1 = kMomX + Minor<DIR>::m1, M2 = kMomX + Minor<DIR>::m2;
  if (n == 1) return c != kMass && c != M1;
  if (DIM == 3 && n == 2) return c != kMass && c != M2;
  return false;
}
// The exact FP64 finite-volume (HLLC) kernels build the right eigenvectors
// only once the characteristic values are formed, so the 19 entries are not
// held in registers meanwhile (it saves 20 VGPRs in 3D); without contraction
// the position changes no bit.  (Flux splitting builds them with the left
// ones: deferring them there made the exact kernel slower.)  The contracting kernels build them beside
// the left eigenvectors: there the basic block they sit in decides which
// products fuse, and the mixed form's accuracy was measured that way.
template <typename R>
constexpr bool kDeferRight = std::is_same<R, double>::value && !kFastArith;

template <int DIM, int DIR, typename R>
__device__ __forceinline__ void set_right_eigenvectors(Eig<DIM + 2, R> &ev, R u, R v, R w, R c,
                                                       R H, R g, R rho_roe) {
  constexpr int NE = DIM + 2;
  constexpr int m1 = Minor<DIR>::m1, m2 = Minor<DIR>::m2;
  constexpr int evp = DIM;
  constexpr int Mp = kMomX + DIR, M1 = kMomX + m1, M2 = kMomX + m2;
  (void)m2;
  (void)M2;
  (void)w;
  ev.Rm[kMass][0] = R(1.0);
  ev.Rm[kMass][evp] = g;
  ev.Rm[kMass][NE - 1] = R(1.0);

  ev.Rm[Mp][0] = u - c;
  ev.Rm[Mp][evp] = g * u;
  ev.Rm[Mp][NE - 1] = u + c;

  ev.Rm[M1][0] = v;
  ev.Rm[M1][1] = -rho_roe;
  ev.Rm[M1][evp] = g * v;
  ev.Rm[M1][NE - 1] = v;

  if constexpr (DIM == 3) {
    ev.Rm[M2][0] = w;
    ev.Rm[M2][2] = rho_roe;
    ev.Rm[M2][evp] = g * w;
    ev.Rm[M2][NE - 1] = w;
  }

  ev.Rm[kEnergy][0] = H - u * c;
  ev.Rm[kEnergy][1] = -v * rho_roe;
  if constexpr (DIM == 3) ev.Rm[kEnergy][2] = rho_roe * w;
  ev.Rm[kEnergy][evp] = g * H - c * c;
  ev.Rm[kEnergy][NE - 1] = H + u * c;
}

// The right eigenvectors of a roe_eigensystem call that deferred them.
template <int DIM, int DIR, typename R, bool kDefer = kDeferRight<R>>
__device__ __forceinline__ void roe_right_eigenvectors(Eig<DIM + 2, R> &ev) {
  if constexpr (kDefer) {
    if (ev.ok) set_right_eigenvectors<DIM, DIR>(ev, ev.u, ev.v, ev.w, ev.c, ev.H, ev.g, ev.rho_roe);
  }
}

// ComputeRoeEigendecomposition for one face (eigendecomposition.h:238-466).
// t = cell i, n = cell i+1 along DIR.  Returns false (all zero) when a
// density is not positive.
template <int DIM, int DIR, typename R, bool kDefer = kDeferRight<R>>
__device__ __forceinline__ bool roe_eigensystem(R gamma, const FaceQ<R> &t, const FaceQ<R> &n,
                                                Eig<DIM + 2, R> &ev) {
  constexpr int NE = DIM + 2;
  constexpr int m1 = Minor<DIR>::m1, m2 = Minor<DIR>::m2;
  constexpr int evp = DIM;
  constexpr int Mp = kMomX + DIR, M1 = kMomX + m1, M2 = kMomX + m2;
#pragma unroll
  for (int r = 0; r < NE; ++r) {
#pragma unroll
    for (int c = 0; c < NE; ++c) {
      ev.L[r][c] = R(0.0);
      ev.Rm[r][c] = R(0.0);
    }
    ev.lam[r] = R(0.0);
  }
  ev.ok = false;
  if (t.rho <= R(0.0) || n.rho <= R(0.0)) return false;
  ev.ok = true;

  R const u_t = t.vel[DIR];
  R const v_t = t.vel[m1];
  R const w_t = DIM == 3 ? t.vel[m2] : R(0.0);
  R const u_n = n.vel[DIR];
  R const v_n = n.vel[m1];
  R const w_n = DIM == 3 ? n.vel[m2] : R(0.0);

  R const sq_t = t.sq;
  R const sq_n = n.sq;
  R const rho_div = fdiv(R(1.0), sq_t + sq_n);
  R const rho_roe = sq_t * sq_n;
  R const one_rho_roe = fdiv(R(1.0), rho_roe);

  R const u = ((u_t * sq_t) + (u_n * sq_n)) * rho_div;
  R const v = ((v_t * sq_t) + (v_n * sq_n)) * rho_div;
  R const w = ((w_t * sq_t) + (w_n * sq_n)) * rho_div;
  R const psi = ((t.psi * sq_t) + (n.psi * sq_n)) * rho_div;
  R const g = gamma - R(1.0);
  R const H = (t.H * sq_t + n.H * sq_n) * rho_div;

  R const q2 = dams<DIM>(u * u, v * v, w * w);
  R const tmp = dams<DIM>((u_t - u_n) * (u_t - u_n), (v_t - v_n) * (v_t - v_n),
                          (w_t - w_n) * (w_t - w_n));
  R const pod = (t.pod * sq_t + n.pod * sq_n) * rho_div +
                R(0.5) * rho_roe * (rho_div * rho_div) * tmp;
  R const cc = psi + g * pod;
  R const one_cc = fdiv(R(1.0), cc);
  R const c = dsqrt(cc);

  ev.L[0][kMass] = R(0.5) * one_cc * (g * q2 - g * H + (u + c) * c);
  ev.L[0][Mp] = R(0.5) * one_cc * (-u * g - c);
  ev.L[0][M1] = R(0.5) * one_cc * (-v * g);
  if constexpr (DIM == 3) ev.L[0][M2] = R(0.5) * one_cc * (-w * g);
  ev.L[0][kEnergy] = R(0.5) * one_cc * g;

  ev.L[1][kMass] = v * one_rho_roe;
  ev.L[1][M1] = -one_rho_roe;

  if constexpr (DIM == 3) {
    ev.L[2][kMass] = -w * one_rho_roe;
    ev.L[2][M2] = one_rho_roe;
  }

  ev.L[evp][kMass] = one_cc * (H - q2);
  ev.L[evp][Mp] = one_cc * u;
  ev.L[evp][M1] = one_cc * v;
  if constexpr (DIM == 3) ev.L[evp][M2] = one_cc * w;
  ev.L[evp][kEnergy] = -one_cc;

  ev.L[NE - 1][kMass] = R(0.5) * one_cc * (g * q2 - g * H - (u - c) * c);
  ev.L[NE - 1][Mp] = R(0.5) * one_cc * (-u * g + c);
  ev.L[NE - 1][M1] = R(0.5) * one_cc * (-v * g);
  if constexpr (DIM == 3) ev.L[NE - 1][M2] = R(0.5) * one_cc * (-w * g);
  ev.L[NE - 1][kEnergy] = R(0.5) * one_cc * g;

  if constexpr (kDefer) {
    ev.u = u;
    ev.v = v;
    ev.w = w;
    ev.c = c;
    ev.H = H;
    ev.g = g;
    ev.rho_roe = rho_roe;
  } else {
    set_right_eigenvectors<DIM, DIR>(ev, u, v, w, c, H, g, rho_roe);
  }

  ev.lam[0] = __builtin_fabs(u - c);
  ev.lam[NE - 1] = __builtin_fabs(u + c);
#pragma unroll
  for (int l = 1; l < NE - 1; ++l) ev.lam[l] = __builtin_fabs(u);
  return true;
}

// TransformToPhysicalSpace (eigendecomposition.h:144-165).  Every product is
// formed, the zero entries' too: 0 * x is NaN for a non-finite x, as in the
// reference.
template <int DIM, int DIR, typename R>
__device__ __forceinline__ void to_physical(const R *ch, const R (&Rm)[DIM + 2][DIM + 2], R *out) {
  constexpr int NE = DIM + 2;
#pragma unroll
  for (int l = 0; l < NE; ++l) {
    R s = R(0.0);
#pragma unroll
    for (int n = 1; n < NE - 1; ++n)
      s += ch[n] * Rm[l][n];
    s += (ch[0] * Rm[l][0] + ch[NE - 1] * Rm[l][NE - 1]);
    out[l] = s;
  }
}

// CalculateSignalSpeed, Einfeldt (hll_signal_speed_calculator.h:77-101).
template <typename R>
__device__ __forceinline__ void einfeldt(R rl, R rr, R ul, R ur, R cl, R cr, R &sl, R &sr) {
  R const sql = dsqrt(rl);
  R const sqr = dsqrt(rr);
  R const rho_div = fdiv(R(1.0), sql + sqr);
  R const u_roe = ((ul * sql) + (ur * sqr)) * rho_div;
  R const c_e = dsqrt(((cl * cl * sql) + (cr * cr * sqr)) * rho_div +
                      (R(0.5) * sql * sqr * rho_div * rho_div) * (ur - ul) * (ur - ul));
  sl = smin(u_roe - c_e, ul - cl);
  sr = smax(u_roe + c_e, ur + cr);
}

// HllcRiemannSolver::SolveRiemannProblemImplementation (hllc_riemann_solver.h:
// 52-198), including the clamped wave speeds in the energy star states.
template <int DIM, int DIR, typename R>
__device__ __forceinline__ void hllc(R gamma, R b, const R *cl, const R *cr, const Prim<R> &pl,
                                     const Prim<R> &pr, R *f) {
  constexpr int NE = DIM + 2;
  constexpr int Mp = kMomX + DIR;
  R qsl[NE], qsr[NE], fl[NE], fr[NE];
  R const p_l = pl.p, p_r = pr.p;
  R const one_rho_l = fdiv(R(1.0), cl[kMass]);
  R const one_rho_r = fdiv(R(1.0), cr[kMass]);
  R const u_l = pl.vel[DIR], u_r = pr.vel[DIR];
  R const c_l = eos_sos(gamma, b, cl[kMass], p_l);
  R const c_r = eos_sos(gamma, b, cr[kMass], p_r);
  R sls, srs;
  einfeldt(cl[kMass], cr[kMass], u_l, u_r, c_l, c_r, sls, srs);
  R const sc = fdiv((p_r - p_l) + (cl[Mp] * (sls - u_l) - cr[Mp] * (srs - u_r)),
                    cl[kMass] * (sls - u_l) - cr[kMass] * (srs - u_r));
  R const sl = smin(sls, R(0.0));
  R const sr = smax(srs, R(0.0));
  R const chi_l = fdiv(sls - u_l, sls - sc);
  R const chi_r = fdiv(srs - u_r, srs - sc);

  qsl[kMass] = cl[kMass] * chi_l;
  qsl[Mp] = cl[kMass] * chi_l * sc;
  qsl[kEnergy] = cl[kMass] * chi_l *
                 (cl[kEnergy] * one_rho_l + (sc - u_l) * (sc + fdiv(p_l, cl[kMass] * (sl - u_l))));
  qsr[kMass] = cr[kMass] * chi_r;
  qsr[Mp] = cr[kMass] * chi_r * sc;
  qsr[kEnergy] = cr[kMass] * chi_r *
                 (cr[kEnergy] * one_rho_r + (sc - u_r) * (sc + fdiv(p_r, cr[kMass] * (sr - u_r))));

  fl[kMass] = cl[Mp];
  fl[Mp] = ((cl[Mp] * cl[Mp]) * one_rho_l) + p_l;
  fl[kEnergy] = u_l * (cl[kEnergy] + p_l);
  fr[kMass] = cr[Mp];
  fr[Mp] = ((cr[Mp] * cr[Mp]) * one_rho_r) + p_r;
  fr[kEnergy] = u_r * (cr[kEnergy] + p_r);

#pragma unroll
  for (int d = 0; d < DIM - 1; ++d) {
    int const Mm = kMomX + (d == 0 ? Minor<DIR>::m1 : Minor<DIR>::m2);
    qsl[Mm] = chi_l * cl[Mm];
    qsr[Mm] = chi_r * cr[Mm];
    fl[Mm] = u_l * cl[Mm];
    fr[Mm] = u_r * cr[Mm];
  }
  int const sg = (R(0.0) < sc) - (sc < R(0.0));
  R const wl = R(0.5) * (R(1.0) + R(sg));
  R const wr = R(0.5) * (R(1.0) - R(sg));
#pragma unroll
  for (int n = 0; n < NE; ++n) {
    R const fsl = fl[n] + (sl * (qsl[n] - cl[n]));
    R const fsr = fr[n] + (sr * (qsr[n] - cr[n]));
    f[n] = (wl * fsl + wr * fsr);
  }
}

// ComputeAdvection (flux_splitting_scheme.cpp:42-76) of one cell in FP64.
template <int DIM, int DIR>
__device__ __forceinline__ void advection(const double *c, const Prim<double> &pd, double *a) {
  double const ud = pd.vel[DIR];
  a[kMass] = pd.rho * ud;
  a[kEnergy] = (c[kEnergy] + pd.p) * ud;
#pragma unroll
  for (int d = 0; d < DIM; ++d) a[kMomX + d] = pd.rho * (ud * pd.vel[d]);
  a[kMomX + DIR] += pd.p;
}

// FluxSplittingScheme::ComputeFluxes + ComputeAdvection for one face in the
// exact FP64 form (flux_splitting_scheme.cpp:42-76, 185-315), added into f.
// Every value is formed by the reference's operations in the reference's
// order; only the time at which each is formed differs, which without
// contraction changes no bit.  The eigensystem of cells i and i+1, then the stencil
// cell by cell: its conservatives (read one cell ahead, through a buffer
// resource: no address arithmetic), its advection and its projections onto every
// field, then WENO5 field by field.  The projections are what is held, 60 doubles in
// 3D, beside L; empty asm statements make each cell's be formed before the next
// cell's and each field's reconstruction before the next field's, so that two
// wavefronts per SIMD fit (left to itself the compiler forms the products of all
// cells at once).  Field by field, with the stencil read again for each
// field, a face had 220 reads instead of 40 and waited for them 29% of the
// time: 128^3, one step, 2778 -> 1892 us; 24 blocks, two steps, 338 -> 262 us.
// The shear rows of L leave their structural zeros out: a sum that starts at 0.0 is
// never -0, so a zero product changes it only where a stencil value is not
// finite (0 * x is then NaN).  Row 0 is dense, so if its reconstruction stayed in the
// core's range, every value is finite; otherwise the zero products are added.
template <int DIM, int DIR, typename QS>
__device__ __forceinline__ void roe_split_flux_exact(double gamma, double b,
                                                     const double *__restrict__ blk, int off,
                                                     const QS &qs, double *f) {
  constexpr int NE = DIM + 2;
  constexpr int S = axis_stride<DIM, DIR>();
  BlockReader<DIM> const rd(blk);
  // Byte offset of stencil cell 0 (cell i-2, inside the haloed block).
  int const off0 = (off - 2 * S) * (int)sizeof(double);
  auto read = [&rd](int o, int m, double *c) {
#pragma unroll
    for (int e = 0; e < NE; ++e) c[e] = rd(o, (e * Dims<DIM>::FIELD + m * S) * (int)sizeof(double));
  };
  Eig<NE, double> ev;
  {
    double Ui[NE], Un[NE];
    read(off0, 2, Ui);
    read(off0, 3, Un);
    roe_eigensystem<DIM, DIR, double, true>(gamma, qs.left(Ui), qs.right(Un), ev);
  }
  double pos[NE][6], neg[NE][6];
  double dep = ev.lam[0], U[NE], ahead[NE];
  {
    int o = off0;
    asm volatile("" : "+v"(o) : "v"(dep));
    read(o, 0, ahead);
  }
#pragma unroll
  for (int m = 0; m < 6; ++m) {
#pragma unroll
    for (int e = 0; e < NE; ++e) U[e] = ahead[e];
    if (m < 5) {
      int o = off0;
      asm volatile("" : "+v"(o) : "v"(dep));
      read(o, m + 1, ahead);
    }
    Prim<double> P;
    cons_to_prim<DIM, double>(gamma, b, U, P);
    double adv[NE];
    advection<DIM, DIR>(U, P, adv);
#pragma unroll
    for (int n = 0; n < NE; ++n) {
      double sp = 0.0, sn = 0.0;
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        int const l = seq<DIM, DIR>(q);
        if (left_zero<DIM, DIR>(n, l)) continue;
        double const uct = U[l] * ev.L[n][l];
        double const act = adv[l] * ev.L[n][l];
        sp += (act + ev.lam[n] * uct);
        sn += (act - ev.lam[n] * uct);
      }
      pos[n][m] = sp;
      neg[n][m] = sn;
    }
#pragma unroll
    for (int n = 0; n < NE; ++n) asm volatile("" : "+v"(pos[n][m]), "+v"(neg[n][m]));
    dep = neg[NE - 1][m];
  }
  double chf[NE];
#pragma unroll
  for (int n = 0; n < NE; ++n) {
    double wl, wr;
    bool const core = weno_pair_exact<true>(pos[n], neg[n], wl, wr);
    chf[n] = 0.5 * (wl + wr);
    if (n == 0 && __builtin_expect(!core, 0)) {
#pragma unroll 1
      for (int m = 0; m < 6; ++m) {
        int o = off0 + m * S * (int)sizeof(double);
        double c[NE], adv[NE];
        read(o, 0, c);
        Prim<double> P;
        cons_to_prim<DIM, double>(gamma, b, c, P);
        advection<DIM, DIR>(c, P, adv);
#pragma unroll
        for (int k = 1; k < DIM; ++k) {
          double z = 0.0;
#pragma unroll
          for (int l = 0; l < NE; ++l)
            if (left_zero<DIM, DIR>(k, l)) z += adv[l] * 0.0 + ev.lam[k] * (c[l] * 0.0);
#pragma unroll
          for (int i = 0; i < 6; ++i) {
            pos[k][i] += i == m ? z : 0.0;
            neg[k][i] += i == m ? z : 0.0;
          }
        }
      }
    }
    if (n + 1 < NE) {
#pragma unroll
      for (int m = 0; m < 6; ++m)
        asm volatile("" : "+v"(pos[n + 1][m]), "+v"(neg[n + 1][m]) : "v"(chf[n]));
    }
  }
  roe_right_eigenvectors<DIM, DIR, double, true>(ev);
  double phys[NE];
  to_physical<DIM, DIR>(chf, ev.Rm, phys);
#pragma unroll
  for (int e = 0; e < NE; ++e) f[e] += phys[e];
}

// FluxSplittingScheme::ComputeFluxes + ComputeAdvection for one face
// (flux_splitting_scheme.cpp:42-76, 185-315), added into f, in the mixed form.
// The stencil is walked cell by cell -- load, advection, projection onto every
// field -- which keeps few values live: 3 waves per SIMD.  Each projection is
// the expression of the exact form.  The stencil is read through a buffer resource: with
// 64-bit addresses 512 3D blocks took 1212 us a step, 1165 so, 4900 2D blocks 357 and 344.
template <int DIM, int DIR, typename QS>
__device__ __forceinline__ void roe_split_flux(double gamma64, double b64,
                                               const double *__restrict__ blk, int off, const QS &qs,
                                               float *f) {
  using R = float;
  constexpr int NE = DIM + 2;
  R const gamma = R(gamma64);
  constexpr int S = axis_stride<DIM, DIR>();
  BlockReader<DIM> const rd(blk);
  int const off0 = (off - 2 * S) * (int)sizeof(double);
  auto load = [&](int m, double *c) {
#pragma unroll
    for (int e = 0; e < NE; ++e)
      c[e] = rd(off0, (e * Dims<DIM>::FIELD + m * S) * (int)sizeof(double));
  };
  Eig<NE, R> ev;
  double adv2[NE];  // advection of cell i (FP64)
  R chf[NE];
  {
    double Ui[NE], Un[NE];
    load(2, Ui);
    load(3, Un);
    roe_eigensystem<DIM, DIR, R, false>(gamma, qs.left(Ui), qs.right(Un), ev);
    {
      Prim<double> pd;
      cons_to_prim<DIM, double>(gamma64, b64, Ui, pd);
      advection<DIM, DIR>(Ui, pd, adv2);
    }
    R pos[NE][6], neg[NE][6];
#pragma unroll
    for (int m = 0; m < 6; ++m) {
      double Um[NE];
      load(m, Um);
      R Uc[NE];
#pragma unroll
      for (int e = 0; e < NE; ++e) Uc[e] = R(Um[e] - Ui[e]);
      R adv[NE];
      Prim<double> pd;
      cons_to_prim<DIM, double>(gamma64, b64, Um, pd);
      // ComputeAdvection in FP64, then the difference from cell i into FP32
      // (see face_flux).
      double a64[NE];
      advection<DIM, DIR>(Um, pd, a64);
#pragma unroll
      for (int e = 0; e < NE; ++e) adv[e] = R(a64[e] - adv2[e]);
#pragma unroll
      for (int n = 0; n < NE; ++n) {
        R sp = R(0.0), sn = R(0.0);
#pragma unroll
        for (int q = 0; q < NE; ++q) {
          int const l = seq<DIM, DIR>(q);
          R const uct = Uc[l] * ev.L[n][l];
          R const act = adv[l] * ev.L[n][l];
          sp += (act + ev.lam[n] * uct);
          sn += (act - ev.lam[n] * uct);
        }
        pos[n][m] = sp;
        neg[n][m] = sn;
      }
    }
#pragma unroll
    for (int n = 0; n < NE; ++n) {
      R wl, wr;
      weno_pair<R>(pos[n], neg[n], wl, wr);
      chf[n] = R(0.5) * (wl + wr);
    }
  }
  R phys[NE];
  to_physical<DIM, DIR>(chf, ev.Rm, phys);
  // R L (adv of cell i) = adv of cell i: the half sums of the shifts.
#pragma unroll
  for (int e = 0; e < NE; ++e) f[e] += R(double(phys[e]) + adv2[e]);
}

// The reconstruction of the FP64-with-FMA form: the products with the Roe
// eigenvectors factored through the quantities they share.  With
//   Y = E - u m_n - v m_1 - w m_2 + (q^2 - H) rho,
//   A = g/(2c^2) Y + rho/2,  B = (u rho - m_n) / (2c)
// the amplitudes of the waves u-c, u+c and of the entropy wave are A + B, A - B
// and -Y/c^2 (15 instructions per cell for all five, against 19 row by row),
// and back, with a = the five reconstructed amplitudes,
//   rho = a_- + a_+ + g a_e,  d = c (a_+ - a_-),  m_n = u rho + d, ...
// The stencil is dead once Y, A, B and the shear amplitudes are formed, and no
// eigenvector matrix is held.
template <int DIM, int DIR> struct LeanEig {
  static constexpr int m1 = Minor<DIR>::m1, m2 = Minor<DIR>::m2;
  static constexpr int Mp = kMomX + DIR, M1 = kMomX + m1, M2 = kMomX + m2;
  double g, u, v, w, H, c, cc, one_cc, rho_roe, one_rho, kY, kA, kB, kBu, kv, kw;
  // Returns false where a density is not positive: no eigensystem.
  __device__ __forceinline__ bool form(double gamma, const FaceQ<double> &t, const FaceQ<double> &n) {
    if (!(t.rho > 0.0) || !(n.rho > 0.0)) {
      if (t.rho <= 0.0 || n.rho <= 0.0) return false;
    }
    double const rho_div = fdiv(1.0, t.sq + n.sq);
    rho_roe = t.sq * n.sq;
    one_rho = fdiv(1.0, rho_roe);
    auto mean = [&](double a, double b) { return (a * t.sq + b * n.sq) * rho_div; };
    u = mean(t.vel[DIR], n.vel[DIR]);
    v = mean(t.vel[m1], n.vel[m1]);
    w = DIM == 3 ? mean(t.vel[m2], n.vel[m2]) : 0.0;
    g = gamma - 1.0;
    H = mean(t.H, n.H);
    double const du = t.vel[DIR] - n.vel[DIR], dv = t.vel[m1] - n.vel[m1];
    double q2 = u * u + v * v, dq = du * du + dv * dv;
    if constexpr (DIM == 3) {
      double const dw = t.vel[m2] - n.vel[m2];
      q2 += w * w;
      dq += dw * dw;
    }
    cc = mean(t.psi + g * t.pod, n.psi + g * n.pod) + g * (0.5 * rho_roe * (rho_div * rho_div) * dq);
    one_cc = fdiv(1.0, cc);
    c = dsqrt(cc);
    kY = q2 - H;
    kA = 0.5 * g * one_cc;
    kB = 0.5 * one_cc * c;
    kBu = kB * u;
    kv = v * one_rho;
    kw = w * one_rho;
    return true;
  }
  // Y, B and the shear amplitudes of a vector of conservatives.
  __device__ __forceinline__ void parts(const double *U, double &Y, double &B, double &s1,
                                        double &s2) const {
    s1 = kv * U[kMass] - one_rho * U[M1];
    Y = U[kEnergy] - u * U[Mp] - v * U[M1] + kY * U[kMass];
    B = kBu * U[kMass] - kB * U[Mp];
    if constexpr (DIM == 3) {
      s2 = one_rho * U[M2] - kw * U[kMass];
      Y -= w * U[M2];
    }
  }
  // Conservatives from the amplitudes.
  __device__ __forceinline__ void back(const double *a, double *o) const {
    double const rho = a[0] + a[DIM + 1] + g * a[DIM];
    double const d = c * (a[DIM + 1] - a[0]);
    double const t1 = rho_roe * a[1];
    double e = H * rho + u * d - cc * a[DIM] - v * t1;
    o[kMass] = rho;
    o[Mp] = u * rho + d;
    o[M1] = v * rho - t1;
    if constexpr (DIM == 3) {
      double const t2 = rho_roe * a[2];
      o[M2] = w * rho + t2;
      e += w * t2;
    }
    o[kEnergy] = e;
  }
};

template <int DIM, int DIR, typename QS>
__device__ __forceinline__ void fv_reconstruct_lean(double gamma, const double (&U)[6][DIM + 2],
                                                    const QS &qs, double *cl, double *cr,
                                                    double &skipped) {
  LeanEig<DIM, DIR> ev;
  if (!ev.form(gamma, qs.left(U[2]), qs.right(U[3]))) {
    // Zero eigenvectors: zero states, whose face is skipped, or NaN where a value of a
    // state's five cells is not finite (as their products with zeros are), and a flux
    // of NaN where both states are.
    double l = 0.0, r = 0.0;
#pragma unroll
    for (int e = 0; e < DIM + 2; ++e) {
      cl[e] = cr[e] = 0.0;
      l += 0.0 * U[0][e];
      r += 0.0 * U[5][e];
#pragma unroll
      for (int m = 1; m < 5; ++m) {
        l += 0.0 * U[m][e];
        r += 0.0 * U[m][e];
      }
    }
    skipped = l == l ? 0.0 : r;
    return;
  }
  double Y[6], B[6], lo[DIM + 2], hi[DIM + 2];
  {
    double s1[6], s2[6];
#pragma unroll
    for (int m = 0; m < 6; ++m) {
      ev.parts(U[m], Y[m], B[m], s1[m], s2[m]);
    }
    weno_pair_lean(s1, lo[1], hi[1]);
    if constexpr (DIM == 3) weno_pair_lean(s2, lo[2], hi[2]);
  }
  double A[6], x[6];
#pragma unroll
  for (int m = 0; m < 6; ++m) {
    A[m] = ev.kA * Y[m] + 0.5 * U[m][kMass];
    x[m] = -ev.one_cc * Y[m];
  }
  weno_pair_lean(x, lo[DIM], hi[DIM]);
#pragma unroll
  for (int m = 0; m < 6; ++m) x[m] = A[m] + B[m];
  weno_pair_lean(x, lo[0], hi[0]);
#pragma unroll
  for (int m = 0; m < 6; ++m) x[m] = A[m] - B[m];
  weno_pair_lean(x, lo[DIM + 1], hi[DIM + 1]);
  ev.back(lo, cl);
  ev.back(hi, cr);
}

// Flux splitting in the FP64-with-FMA form (roe_split_flux below): the conservatives
// and the advection of a stencil cell are projected by the factored products, 40
// instructions a cell with the sums and differences against 114 row by row.
template <int DIM, int DIR, typename QS>
__device__ __forceinline__ void roe_split_flux_lean(double gamma, double b,
                                                    const double *__restrict__ base, const QS &qs,
                                                    double *f) {
  constexpr int NE = DIM + 2;
  using E = LeanEig<DIM, DIR>;
  auto load = [base](int m, double *c) {
#pragma unroll
    for (int e = 0; e < NE; ++e)
      c[e] = base[e * Dims<DIM>::FIELD + (m - 2) * axis_stride<DIM, DIR>()];
  };
  // A stencil cell's conservatives and advection.
  auto cell = [&](int m, double *U, double *adv) {
    load(m, U);
    double const one = fdiv(1.0, U[kMass]), ud = U[E::Mp] * one;
    double k = U[E::Mp] * ud + U[E::M1] * (U[E::M1] * one);
    if constexpr (DIM == 3) k += U[E::M2] * (U[E::M2] * one);
    double const p = (gamma - 1.0) * (U[kEnergy] - 0.5 * k) - gamma * b;
    adv[kMass] = U[E::Mp];
    adv[kEnergy] = (U[kEnergy] + p) * ud;
    adv[E::Mp] = U[E::Mp] * ud + p;
    adv[E::M1] = U[E::M1] * ud;
    if constexpr (DIM == 3) adv[E::M2] = U[E::M2] * ud;
  };
  E ev;
  {
    double Ui[NE], Un[NE];
    load(2, Ui);
    load(3, Un);
    if (!ev.form(gamma, qs.left(Ui), qs.right(Un))) {
      // Zero eigenvectors: no flux, or NaN where a value of the six cells is not finite
      // (as their products with zeros are).
      double z = 0.0;
#pragma unroll 1
      for (int m = 0; m < 6; ++m) {
        double U[NE], adv[NE];
        cell(m, U, adv);
#pragma unroll
        for (int e = 0; e < NE; ++e) z += 0.0 * U[e] + 0.0 * adv[e];
      }
#pragma unroll
      for (int e = 0; e < NE; ++e) f[e] += z;
      return;
    }
  }
  double const lam = __builtin_fabs(ev.u), lam_lo = __builtin_fabs(ev.u - ev.c),
               lam_hi = __builtin_fabs(ev.u + ev.c);
  double pos[NE][6], neg[NE][6];
#pragma unroll
  for (int m = 0; m < 6; ++m) {
    double U[NE], adv[NE];
    cell(m, U, adv);
    double uY, uB, u1, u2, aY, aB, a1, a2;
    ev.parts(U, uY, uB, u1, u2);
    ev.parts(adv, aY, aB, a1, a2);
    auto put = [&](int n, double a, double lu) {
      pos[n][m] = a + lu;
      neg[n][m] = a - lu;
    };
    double const uA = ev.kA * uY + 0.5 * U[kMass], aA = ev.kA * aY + 0.5 * adv[kMass];
    put(0, aA + aB, lam_lo * (uA + uB));
    put(1, a1, lam * u1);
    if constexpr (DIM == 3) put(2, a2, lam * u2);
    put(DIM, -ev.one_cc * aY, -ev.one_cc * (lam * uY));
    put(DIM + 1, aA - aB, lam_hi * (uA - uB));
  }
  double chf[NE], phys[NE];
#pragma unroll
  for (int n = 0; n < NE; ++n) {
    double wl, wr;
    weno_pair<double>(pos[n], neg[n], wl, wr);
    chf[n] = 0.5 * (wl + wr);
  }
  ev.back(chf, phys);
#pragma unroll
  for (int e = 0; e < NE; ++e) f[e] += phys[e];
}

// FP64 square root of a positive argument: nr_sqrt64 without its zero case.
__device__ __forceinline__ double nr_sqrt64_pos(double x) {
  double const r = __builtin_amdgcn_rsq(x);
  double g = x * r;
  double h = 0.5 * r;
  double const e = __builtin_fma(-g, h, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// The Riemann problem of the FP64-with-FMA form (hllc and einfeldt below): the
// side of the contact the face lies on is selected before its star state is
// formed, and that state takes one division: with i = 1 / (S - S*),
// chi = (S - u) i and p / (rho (S - u)) rho chi = p i.  (The reference's
// clamped speed differs from S only where it is zero, and it then multiplies
// the star state by zero.)  1/rho serves the velocities, the pressure and the
// sound speed.  Five divisions per face instead of twelve.
template <int DIM, int DIR>
__device__ __forceinline__ void fv_riemann_lean(double gamma, double b, const double *cl,
                                                const double *cr, double skipped, double *f) {
  constexpr int NE = DIM + 2;
  constexpr int Mp = kMomX + DIR, M1 = kMomX + Minor<DIR>::m1, M2 = kMomX + Minor<DIR>::m2;
#pragma unroll
  for (int e = 0; e < NE; ++e) f[e] = skipped;
  double const eps = 2.220446049250313080847263336181640625e-16;  // DBL_EPSILON
  if (cl[kMass] <= eps || cr[kMass] <= eps) return;
  auto pressure = [&](const double *c, double one_rho, double &u) {
    u = c[Mp] * one_rho;
    double k = c[Mp] * u + c[M1] * (c[M1] * one_rho);
    if constexpr (DIM == 3) k += c[M2] * (c[M2] * one_rho);
    return (gamma - 1.0) * (c[kEnergy] - 0.5 * k) - gamma * b;
  };
  double const il = fdiv(1.0, cl[kMass]), ir = fdiv(1.0, cr[kMass]);
  double ul, ur;
  double const pl = pressure(cl, il, ul), pr = pressure(cr, ir, ur);
  if (pl <= -b || pr <= -b) return;
  double const ccl = gamma * (pl + b) * il, ccr = gamma * (pr + b) * ir;
  double const al = nr_sqrt64_pos(ccl), ar = nr_sqrt64_pos(ccr);
  double const sql = nr_sqrt64_pos(cl[kMass]), sqr = nr_sqrt64_pos(cr[kMass]);
  double const rd = fdiv(1.0, sql + sqr);
  double const um = (ul * sql + ur * sqr) * rd;
  double const du = ur - ul;
  double const ce = nr_sqrt64_pos((ccl * sql + ccr * sqr) * rd + 0.5 * (sql * rd) * (sqr * rd) * (du * du));
  double const sl = __builtin_fmin(um - ce, ul - al), sr = __builtin_fmax(um + ce, ur + ar);
  double const dl = sl - ul, dr = sr - ur;
  double const sc = fdiv((pr - pl) + (cl[Mp] * dl - cr[Mp] * dr), cl[kMass] * dl - cr[kMass] * dr);
  bool const left = sc >= 0.0;
  double c[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) c[e] = left ? cl[e] : cr[e];
  double const p = left ? pl : pr, u = left ? ul : ur, d = left ? dl : dr, s = left ? sl : sr;
  double const sk = left ? __builtin_fmin(sl, 0.0) : __builtin_fmax(sr, 0.0);
  double const i = fdiv(1.0, s - sc);
  double const chi = d * i, rchi = c[kMass] * chi;
  double const n = rchi * sc, chi1 = chi - 1.0;
  f[kMass] = c[Mp] + sk * (rchi - c[kMass]);
  f[Mp] = (c[Mp] * u + p) + sk * (n - c[Mp]);
  f[kEnergy] = u * (c[kEnergy] + p) + sk * (chi1 * c[kEnergy] + (sc - u) * (n + p * i));
  f[M1] = c[M1] * (u + sk * chi1);
  if constexpr (DIM == 3) f[M2] = c[M2] * (u + sk * chi1);
}

// The finite-volume face (FiniteVolumeScheme::ComputeFluxes,
// finite_volume_scheme.cpp:160-251, with CharacteristicStateReconstruction,
// characteristic_state_reconstruction.h:60-134) in two parts: fv_reconstruct
// forms the states cl and cr left and right of the face from its stencil Ud
// (FP64 conservatives of cells i-2..i+3 along DIR), fv_riemann the flux.  `skipped`
// passes the flux of a face without an eigensystem.
template <int DIM, int DIR, typename R, typename QS>
__device__ __forceinline__ void fv_reconstruct(double gamma64, const double (&Ud)[6][DIM + 2],
                                               const QS &qs, R *cl, R *cr, R &skipped) {
  skipped = R(0.0);
  if constexpr (kLean<R>) {
    fv_reconstruct_lean<DIM, DIR>(gamma64, Ud, qs, cl, cr, skipped);
    return;
  }
  R const gamma = R(gamma64);
  constexpr int NE = DIM + 2;
  // Mixed form: the stencil enters the FP32 reconstruction as differences
  // from cell i (taken in FP64), and cell i is added back in FP64 after the
  // back-transform.  Exact arithmetic gives the same flux: the WENO5
  // smoothness indicators see only differences and its candidate stencils
  // sum to one, so WENO(v - c) = WENO(v) - c, and R L = I.  In FP32 it keeps
  // the rounding error proportional to the local variation instead of the
  // state's magnitude.
  constexpr bool kShift = std::is_same<R, float>::value;
  Eig<NE, R> ev;
  R U[6][NE];
#pragma unroll
  for (int m = 0; m < 6; ++m)
#pragma unroll
    for (int e = 0; e < NE; ++e) U[m][e] = kShift ? R(Ud[m][e] - Ud[2][e]) : R(Ud[m][e]);
  roe_eigensystem<DIM, DIR>(gamma, qs.left(Ud[2]), qs.right(Ud[3]), ev);
  R minus[NE], plus[NE];
  // Row n of L times the stencil; SKIP leaves out the row's structural zeros.
  // The reference's sum starts at 0.0; the exact form starts at the first
  // product, which can differ in the sign of a zero only, and no zero's sign
  // passes the back-transform's sum, which does start at 0.0.
  auto project = [&](int n, auto skip, R *uc) {
#pragma unroll
    for (int m = 0; m < 6; ++m) {
      R s = R(0.0);
      bool first = kExact<R>;
#pragma unroll
      for (int q = 0; q < NE; ++q) {
        int const l = seq<DIM, DIR>(q);
        if (decltype(skip)::value && left_zero<DIM, DIR>(n, l)) continue;
        s = first ? ev.L[n][l] * U[m][l] : s + ev.L[n][l] * U[m][l];
        first = false;
      }
      uc[m] = s;
    }
  };
  // In the exact form a zero entry's product matters only where a stencil
  // value is not finite (0 * x is then NaN, as in the reference).  Field 0's
  // row is dense: if its reconstruction stayed in the core's range, every
  // stencil value is finite, and the shear rows leave their zeros out.
  bool finite = true;
#pragma unroll
  for (int n = 0; n < NE; ++n) {
    R uc[6];
    if constexpr (kExact<R>) {
      if (n >= 1 && n < DIM) {
        project(n, std::true_type{}, uc);
        if (__builtin_expect(!finite, 0)) project(n, std::false_type{}, uc);
      } else {
        project(n, std::false_type{}, uc);
      }
      bool const core = weno_pair_exact<false>(uc, uc, minus[n], plus[n]);
      if (n == 0) finite = core;
    } else {
      project(n, std::false_type{}, uc);
      weno_pair<R>(uc, uc, minus[n], plus[n]);
    }
  }
  roe_right_eigenvectors<DIM, DIR>(ev);
  to_physical<DIM, DIR>(minus, ev.Rm, cl);
  to_physical<DIM, DIR>(plus, ev.Rm, cr);
  if constexpr (kShift) {
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      cl[e] = R(double(cl[e]) + Ud[2][e]);
      cr[e] = R(double(cr[e]) + Ud[2][e]);
    }
  }
}

// The six-cell stencil of a face: cells off + (m - 2) * stride, m = 0..5,
// through the block's buffer resource (one 32-bit byte offset per cell, the
// field as a scalar offset).
template <int DIM>
__device__ __forceinline__ void load_stencil(const BlockReader<DIM> &rd, int off, int stride,
                                             double (&Ud)[6][DIM + 2]) {
#pragma unroll
  for (int m = 0; m < 6; ++m)
#pragma unroll
    for (int e = 0; e < DIM + 2; ++e)
      Ud[m][e] = rd((off + (m - 2) * stride) * (int)sizeof(double),
                    e * Dims<DIM>::FIELD * (int)sizeof(double));
}

// Writes f (zero when the reference skips the face).
template <int DIM, int DIR, typename R>
__device__ __forceinline__ void fv_riemann(double gamma64, double b64, const R *cl, const R *cr,
                                           R skipped, R *f) {
  if constexpr (kLean<R>) {
    fv_riemann_lean<DIM, DIR>(gamma64, b64, cl, cr, skipped, f);
    return;
  }
  constexpr int NE = DIM + 2;
  R const gamma = R(gamma64), b = R(b64);
#pragma unroll
  for (int e = 0; e < NE; ++e) f[e] = R(0.0);
  R const eps = R(2.220446049250313080847263336181640625e-16);  // DBL_EPSILON
  if (cl[kMass] <= eps || cr[kMass] <= eps) return;
  Prim<R> pl, pr;
  cons_to_prim<DIM>(gamma, b, cl, pl);
  cons_to_prim<DIM>(gamma, b, cr, pr);
  if (pl.p <= -b || pr.p <= -b) return;
  R hf[NE];
  hllc<DIM, DIR>(gamma, b, cl, cr, pl, pr, hf);
#pragma unroll
  for (int e = 0; e < NE; ++e) f[e] += hf[e];
}

template <int DIM, int DIR, typename R, typename QS>
__device__ __forceinline__ void fv_face(double gamma64, double b64, const double *blk, int off,
                                        const QS &qs, R *f) {
  BlockReader<DIM> const rd(blk);
  double Ud[6][DIM + 2];
  load_stencil<DIM>(rd, off, axis_stride<DIM, DIR>(), Ud);
  R cl[DIM + 2], cr[DIM + 2], skipped;
  fv_reconstruct<DIM, DIR, R>(gamma64, Ud, qs, cl, cr, skipped);
  fv_riemann<DIM, DIR, R>(gamma64, b64, cl, cr, skipped, f);
}

// The conservatives of one cell.
template <int DIM>
__device__ __forceinline__ void load_cell(const BlockReader<DIM> &rd, int off, double (&c)[DIM + 2]) {
#pragma unroll
  for (int e = 0; e < DIM + 2; ++e)
    c[e] = rd(off * (int)sizeof(double), e * Dims<DIM>::FIELD * (int)sizeof(double));
}

// One face flux from the six-cell stencil Ud[m] (FP64 conservatives of cells
// i-2..i+3 along DIR); reconstruction and Riemann arithmetic in R.
// FV:  FiniteVolumeScheme::ComputeFluxes (finite_volume_scheme.cpp:160-251)
//      + CharacteristicStateReconstruction (characteristic_state_reconstruction.h:60-134).
// Roe: FluxSplittingScheme::ComputeFluxes + ComputeAdvection
//      (flux_splitting_scheme.cpp:42-76, 185-315).
// Writes f (zero when the reference skips the face).  qs gives the FaceQ of
// the cells left and right of the face.
template <int DIM, int DIR, int FLUX, typename R, typename QS>
__device__ __forceinline__ void face_flux(double gamma64, double b64,
                                          const double *__restrict__ blk, int off, const QS &qs,
                                          R *f) {
  constexpr int NE = DIM + 2;
  const double *__restrict__ base = blk + off;
#pragma unroll
  for (int e = 0; e < NE; ++e) f[e] = R(0.0);
  if constexpr (FLUX == 0) {
    fv_face<DIM, DIR, R>(gamma64, b64, blk, off, qs, f);
  } else if constexpr (std::is_same<R, double>::value && !kFastArith) {
    roe_split_flux_exact<DIM, DIR>(gamma64, b64, blk, off, qs, f);
  } else if constexpr (kLean<R>) {
    roe_split_flux_lean<DIM, DIR>(gamma64, b64, base, qs, f);
  } else {
    roe_split_flux<DIM, DIR>(gamma64, b64, blk, off, qs, f);
  }
}

// FaceQ sources of a face.  Formed: from the cell's conservatives.  Kept: of
// both cells from LDS.  KeptThenFormed: the left cell's from LDS, the right
// cell's formed and written to LDS for the next plane.
template <int DIM, typename R> struct FormedQ {
  double gamma, b;
  __device__ __forceinline__ FaceQ<R> left(const double *c) const {
    return face_quantities<DIM, R>(gamma, b, c);
  }
  __device__ __forceinline__ FaceQ<R> right(const double *c) const {
    return face_quantities<DIM, R>(gamma, b, c);
  }
};
template <int DIM, int STRIDE> struct KeptQ {
  const double *l, *r;
  __device__ __forceinline__ FaceQ<double> left(const double *c) const {
    return load_packed<DIM, STRIDE>(l, c);
  }
  __device__ __forceinline__ FaceQ<double> right(const double *c) const {
    return load_packed<DIM, STRIDE>(r, c);
  }
};
template <int DIM, int STRIDE> struct KeptThenFormedQ {
  double gamma, b;
  const double *l;
  double *r;
  __device__ __forceinline__ FaceQ<double> left(const double *c) const {
    return load_packed<DIM, STRIDE>(l, c);
  }
  __device__ __forceinline__ FaceQ<double> right(const double *c) const {
    store_packed<DIM, STRIDE>(gamma, b, c, r);
    return load_packed<DIM, STRIDE>(r, c);
  }
};

// Loads the six-cell stencil around the face (i,j,k)+1/2 along DIR (halo
// indices of the cell left of the face) and computes its flux.
template <int DIM, int DIR, int FLUX, typename R>
__device__ __forceinline__ void stencil_flux(const double *__restrict__ blk, int i, int j, int k,
                                             double gamma, double b, R *f) {
  using D = Dims<DIM>;
  face_flux<DIM, DIR, FLUX, R>(gamma, b, blk, i * D::SX + j * D::SY + k, FormedQ<DIM, R>{gamma, b}, f);
}
