// trace_fast.h — the persistent tracing kernel for the common decks: Boris
// mover, analytic dipole, legacy step selector with the adaptive gyro budget.
// Included by trace.hip.
//
// What bounds it.  A FP64 Boris step is arithmetic in registers; the general
// stepper (Fp64Stepper) issues about 1,170 vector instructions a step: 15
// divisions and 6 square roots as IEEE sequences with operand scaling and
// special-case fix-up, and some 600 reloads of spilled scalar registers that
// its run-time modes cost; a full map of 786,432 trajectories took 0.44 s
// (0.16 s in FP32), 0.142 s (0.095 s) now.  Here a step is about 270: the work modes, the
// outer boundary and the limiter are template parameters, divisions by one
// denominator share its refined reciprocal (the gyro factor's and the
// momentum's are carried from the end of one step to the start of the next),
// the scaling and fix-up are left out where the operands' range makes them
// the identity, and the inner-sphere chord test runs only for chords that can
// reach the sphere.
//
// Same bits.  div() and root() are the instruction sequences that the
// compiler emits for a / b and sqrt(x) less v_div_scale, v_div_fixup, ldexp
// and the class tests, which are the identity for finite operands well inside
// the exponent range (quotient, operands and reciprocal within 2^+-700; a zero
// quotient comes out as +0, equal to the -0 that a / b may give).  The
// host admits only launches whose constants keep every operand in that range
// (fast64_view); what depends on the trajectory is checked in the step: a
// step with an operand outside is made again with the compiler's own
// operations (IEEE = true), before anything is committed, and a trajectory
// that starts outside is traced with them throughout.
#pragma once

namespace {

template <bool IEEE>
struct Arith {
  static __device__ __forceinline__ double rcp(double b) { return IEEE ? 0.0 : rcp_full(b); }
  // a / b, r = rcp(b)
  static __device__ __forceinline__ double div(double a, double b, double r) {
    if constexpr (IEEE) return a / b;
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
  }
  static __device__ __forceinline__ double root(double x) {
    if constexpr (IEEE) return sqrt(x);
    const double y = __builtin_amdgcn_rsq(x);
    const double h0 = 0.5 * y, s0 = x * y;
    const double e = fma(-h0, s0, 0.5);
    const double h1 = fma(h0, e, h0), s1 = fma(s0, e, s0);
    const double s2 = fma(fma(-s1, s1, x), h1, s1);
    return fma(fma(-s2, s2, x), h1, s2);
  }
};

struct Fast64View {
  double mc2, m0, q, qabs, dphi;
  double M[3];     // moment times its direction
  double Bext[3];  // uniform field
  double rin, rin2, rin_far, rout2;
  double box_min[3], box_max[3];
  double dt_trace, dt_trace1, max_time, max_time1;  // of the first attempt and of the retry
  double maxdist, maxdist_eff;  // as given (off: <= 0); infinite when off
  int max_steps, max_steps1;
};

struct Fast64Lane {
  double x[3], p[3], t, s, dtTrace, maxTime;
  double r2, gm, rgm, iv;  // |x|^2; gamma m0, its refined reciprocal and 1 / it
  int n, maxSteps, retry;
  bool ieee;               // traced with IEEE operations throughout
};

// |v| within 2^-400 .. 2^400, or zero
__device__ __forceinline__ bool usual(double v) {
  const double a = fabs(v);
  return a == 0.0 || (a > 0x1p-400 && a < 0x1p+400);
}

// SPHERE: outer sphere, else the box.  LIM: the distance limiter and the
// floor (switched by the parameters) are compiled in.
template <bool SPHERE, bool LIM>
struct Fast64 {
  struct View {
    Fast64View f;
    amps_trace_params P;  // LIM only reads it in the step
  };
  using Lane = Fast64Lane;

  // what the step carries, for the state in L
  static __device__ __forceinline__ void derive(const Fast64View& V, Lane& L) {
    L.r2 = dot3(L.x, L.x);
    const double gam = sqrt(1.0 + dot3(L.p, L.p) / V.mc2);
    L.gm = gam * V.m0;
    L.rgm = rcp_full(L.gm);
    L.iv = 1.0 / L.gm;
  }

  static __device__ __forceinline__ void init(const View& v, Lane& L, const double* x0, const double* dir, double R,
                                              int attempt) {
    const Fast64View& V = v.f;
    const double pMag = (R * 1.0e9 * V.qabs) / C_LIGHT;
    const double v0[3] = {-1.0 * dir[0], -1.0 * dir[1], -1.0 * dir[2]};
#pragma unroll
    for (int d = 0; d < 3; d++) {
      L.p[d] = pMag * v0[d];
      L.x[d] = x0[d];
    }
    L.t = 0.0;
    L.s = 0.0;
    L.n = 0;
    L.retry = attempt;
    L.dtTrace = attempt ? V.dt_trace1 : V.dt_trace;
    L.maxTime = attempt ? V.max_time1 : V.max_time;
    L.maxSteps = attempt ? V.max_steps1 : V.max_steps;
    derive(V, L);
    const double p2 = dot3(L.p, L.p);
    // |p| is conserved to rounding, so the momentum's range holds for the
    // whole trajectory; so does the position's lower end (r > r_inner)
    L.ieee = !(p2 > 0x1p-400 && p2 < 0x1p+400 && p2 / V.mc2 < 0x1p+100 && L.r2 < 0x1p+160);
#pragma unroll
    for (int d = 0; d < 3; d++) L.ieee = L.ieee || !usual(L.x[d]) || !usual(L.p[d]);
  }

  // One iteration of the trace loop with the compiler's own operations: a
  // termination code or -1.
  static __device__ __forceinline__ int step_ieee(const View& v, Lane& L) {
    const Fast64View& V = v.f;
    if (!(L.n < L.maxSteps && L.t < L.maxTime && (V.maxdist <= 0.0 || L.s < V.maxdist))) {
      if (L.n >= L.maxSteps) return 4;
      if (V.maxdist > 0.0 && L.s >= V.maxdist) return 5;
      if (L.t >= L.maxTime) return 3;
      return 8;
    }
    if (!fin3(L.x) || !fin3(L.p)) return 8;
    if (L.r2 <= V.rin2) return 1;
    if (!inside(V, L)) return 0;
    return advance<true>(v, L);
  }
  static __device__ __forceinline__ bool inside(const Fast64View& V, const Lane& L) {
    if (SPHERE) return L.r2 <= V.rout2;
    const double* x = L.x;
    return (x[0] >= V.box_min[0]) & (x[0] <= V.box_max[0]) & (x[1] >= V.box_min[1]) & (x[1] <= V.box_max[1]) &
           (x[2] >= V.box_min[2]) & (x[2] <= V.box_max[2]);
  }

  // The same; whatever is out of the ordinary (an end of the trajectory, an
  // operand out of range) is left to step_ieee, so that the common step has
  // one branch at its start, one before its state is committed and one for
  // chords near the inner sphere.
  static __device__ __forceinline__ int step(const View& v, Lane& L) {
    const Fast64View& V = v.f;
    int term = -2;
    if ((L.n < L.maxSteps) & (L.t < L.maxTime) & (L.s < V.maxdist_eff) & (L.r2 > V.rin2) & inside(V, L) & !L.ieee)
      term = advance<false>(v, L);
    if (term == -2) term = step_ieee(v, L);
    return term;
  }

  // the step itself, from a state that passed those checks; IEEE false: -2
  // with nothing committed where an operand is out of range
  template <bool IEEE>
  static __device__ __forceinline__ int advance(const View& v, Lane& L) {
    using A = Arith<IEEE>;
    const Fast64View& V = v.f;
    double* x = L.x;
    double* p = L.p;
    // the dipole and the uniform field (dipole64)
    const double r = A::root(L.r2), r3 = L.r2 * r, r5 = r3 * L.r2;
    const double i3 = A::rcp(r3), i5 = A::rcp(r5);
    const double mdotr = V.M[0] * x[0] + V.M[1] * x[1] + V.M[2] * x[2];
    double B[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
      B[d] = 1.0e-7 * (A::div(3.0 * x[d] * mdotr, r5, i5) - A::div(V.M[d], r3, i3)) + V.Bext[d];
    // the step selector (select_dt64)
    const double trem = L.maxTime - L.t;
    double dt = L.dtTrace;
    if (trem < dt) dt = trem;
    const double B2 = dot3(B, B);
    const double Bmag = A::root(B2);
    const double qB = V.qabs * Bmag;
    if (!IEEE || Bmag > 0.0) {
      const double omega = A::div(qB, L.gm, L.rgm);
      if (!IEEE || omega > 0.0) dt = dmin(dt, A::div(V.dphi, omega, A::rcp(omega)));
    }
    if (LIM) dt = limit(v, L, dt);
    if (trem > 0.0) dt = dmin(dt, trem);
    bool ok = B2 > 0x1p-240;
    if (LIM || IEEE) {
      if (!(dt > 0.0) || !isfinite(dt)) return IEEE || ok ? 6 : -2;
      ok = ok & (dt > 0x1p-400);
    }
    // half drift, rotation, half drift (boris64)
    const double h = 0.5 * dt;
    double xn[3], pn[3];
#pragma unroll
    for (int d = 0; d < 3; d++) xn[d] = x[d] + h * (L.iv * p[d]);
    // (q dt) / (2 gamma m0): the factor 2 is exact on either side
    const double tc = IEEE ? (V.q * dt) / (2.0 * L.gm) : 0.5 * A::div(V.q * dt, L.gm, L.rgm);
    const double t[3] = {tc * B[0], tc * B[1], tc * B[2]};
    const double t2 = dot3(t, t);
    const double o2 = 1.0 + t2;
    const double sc = A::div(2.0, o2, A::rcp(o2));
    const double s[3] = {sc * t[0], sc * t[1], sc * t[2]};
    const double pp[3] = {p[0] + (p[1] * t[2] - p[2] * t[1]), p[1] + (p[2] * t[0] - p[0] * t[2]),
                          p[2] + (p[0] * t[1] - p[1] * t[0])};
    pn[0] = p[0] + (pp[1] * s[2] - pp[2] * s[1]);
    pn[1] = p[1] + (pp[2] * s[0] - pp[0] * s[2]);
    pn[2] = p[2] + (pp[0] * s[1] - pp[1] * s[0]);
    const double p2 = dot3(pn, pn);
    const double gam = A::root(1.0 + A::div(p2, V.mc2, A::rcp(V.mc2)));
    const double gm = gam * V.m0;
    const double rgm = rcp_full(gm);
    const double iv = A::div(1.0, gm, rgm);
#pragma unroll
    for (int d = 0; d < 3; d++) xn[d] = xn[d] + h * (iv * pn[d]);
    const double dd[3] = {xn[0] - x[0], xn[1] - x[1], xn[2] - x[2]};
    const double d2 = dot3(dd, dd);
    const double seg = A::root(d2);
    const double r2n = dot3(xn, xn);
    if (!IEEE) {
      // the operands of this step that no launch or trajectory check covers;
      // r2n and p2 finite: so are x and p (a NaN fails every comparison)
      ok = ok & (d2 > 0x1p-300) & (r2n < 0x1p+160) & (p2 < 0x1p+400);
      if (LIM) ok = ok & (t2 < 0x1p+400);
      if (!ok) return -2;
    }
    // the chord can reach (or end inside) the inner sphere only if it starts
    // within its length of it
    const bool hit = (IEEE || r - seg <= V.rin_far) && (seg_hits(x, xn, V.rin) || inside_inner_m(xn, V.rin));
#pragma unroll
    for (int d = 0; d < 3; d++) x[d] = xn[d], p[d] = pn[d];
    L.r2 = r2n;
    L.gm = gm;
    L.rgm = rgm;
    L.iv = iv;
    if (hit) return 1;
    if (IEEE) {
      if (!fin3(x) || !fin3(p)) return 8;
      L.s += isfinite(seg) ? seg : 0.0;
    } else {
      L.s += seg;
    }
    L.t += dt;
    ++L.n;
    return -1;
  }

  // the distance limiter and the floor of select_dt64
  static __device__ __forceinline__ double limit(const View& v, const Lane& L, double dt) {
    const amps_trace_params& P = v.P;
    const double* x = L.x;
    const double pMag = sqrt(dmax(0.0, dot3(L.p, L.p)));
    const double vFor = (L.gm > 0.0) ? pMag / L.gm : 0.0;
    if (P.dist_limiter) {
      const double Re = P.earth_radius_m;
      const double xRe[3] = {x[0] / Re, x[1] / Re, x[2] / Re};
      const double rRe = sqrt(xRe[0] * xRe[0] + xRe[1] * xRe[1] + xRe[2] * xRe[2]);
      double dInner = 1.0e300;
      if (rRe > P.r_inner_Re) dInner = (rRe - P.r_inner_Re) * Re;
      double dBox = 1.0e300;
      if (SPHERE) {
        if (rRe < P.r_outer_Re) dBox = (P.r_outer_Re - rRe) * Re;
      } else if (xRe[0] >= P.box_min_Re[0] && xRe[0] <= P.box_max_Re[0] && xRe[1] >= P.box_min_Re[1] &&
                 xRe[1] <= P.box_max_Re[1] && xRe[2] >= P.box_min_Re[2] && xRe[2] <= P.box_max_Re[2]) {
        const double dxp = (P.box_max_Re[0] - xRe[0]) * Re, dxm = (xRe[0] - P.box_min_Re[0]) * Re;
        const double dyp = (P.box_max_Re[1] - xRe[1]) * Re, dym = (xRe[1] - P.box_min_Re[1]) * Re;
        const double dzp = (P.box_max_Re[2] - xRe[2]) * Re, dzm = (xRe[2] - P.box_min_Re[2]) * Re;
        dBox = dmin(dmin(dmin(dxp, dxm), dmin(dyp, dym)), dmin(dzp, dzm));
      }
      const double dNear = dmin(dInner, dBox);
      if (vFor > 0.0 && dNear < 1.0e299) dt = dmin(dt, 0.20 * dNear / vFor);
    }
    if (P.dt_floor) {
      const double safeSpeed = dmax(vFor, 1.0e-12);
      const double dtFloor = dmax(dmax(1.0e-12, 1.0e-9 * dmax(L.dtTrace, 1.0)), 100.0e3 / safeSpeed);
      dt = dmax(dtFloor, dt);
    }
    return dt;
  }

  static __device__ __forceinline__ int steps_of(const Lane& L) { return L.n; }
  static __device__ __forceinline__ void result(const View&, const Lane& L, int term, amps_trace_result& r) {
    r.termination = term;
    r.retry_count = L.retry;
    r.steps = L.n;
    r.time_s = L.t;
    r.distance_m = L.s;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      r.x[d] = L.x[d];
      r.p[d] = L.p[d];
    }
  }
};

// The FP32 Boris step (Fp32Stepper<MV_BORIS>) with the same template
// parameters.  Its fused multiply-adds are written out: those that the
// compiler's contraction chose in the general kernel, so that every mode's
// kernel and the general one trace the same bits.
struct Fast32View {
  // rin2_eff, maxdist_eff: below every square, infinite where the limit is off
  double len, rin, rin2_eff, rout2, rout, maxdist_eff, floor_abs, floor_rel, floor_dist;
  double dt_trace, dt_trace1, max_time, max_time1;  // of the first attempt and of the retry, units of len / c
  double box_min[3], box_max[3];
  double m0, qabs;
  float cb, mhat[3], bext[3], dphi, rin_c;
  int max_steps, max_steps1, adaptive, dist_limiter, dt_floor;
};

struct Fast32Lane {
  double x[3], t, s, dtTrace, maxTime, r2;
  float u[3];
  int n, maxSteps, retry;
  bool bad;  // starts with a not-finite state
};

// a a + b b + c c, contracted as below: the first square rounded
__device__ __forceinline__ float sumsq(float a, float b, float c) { return fmaf(c, c, fmaf(b, b, a * a)); }

template <bool SPHERE, bool LIM>
struct Fast32 {
  using View = Fast32View;
  using Lane = Fast32Lane;
  static __device__ __forceinline__ void init(const View& V, Lane& L, const double* x0, const double* dir, double R,
                                              int attempt) {
    // |u| = p/(m0 c) with p = R*1e9*|q|/c
    const double umag = (R * 1.0e9 * V.qabs) / C_LIGHT / (V.m0 * C_LIGHT);
#pragma unroll
    for (int d = 0; d < 3; d++) {
      L.u[d] = (float)(umag * (-1.0 * dir[d]));
      L.x[d] = x0[d] / V.len;
    }
    L.t = 0.0;
    L.s = 0.0;
    L.n = 0;
    L.retry = attempt;
    L.dtTrace = attempt ? V.dt_trace1 : V.dt_trace;
    L.maxTime = attempt ? V.max_time1 : V.max_time;
    L.maxSteps = attempt ? V.max_steps1 : V.max_steps;
    L.r2 = dot3(L.x, L.x);
    L.bad = !fin3(L.x) || !isfinite(L.u[0]) || !isfinite(L.u[1]) || !isfinite(L.u[2]);
  }
  static __device__ __forceinline__ int step(const View& V, Lane& L) {
    double* x = L.x;
    float* u = L.u;
    bool inside;
    if (SPHERE)
      inside = L.r2 <= V.rout2;
    else
      inside = (x[0] >= V.box_min[0]) & (x[0] <= V.box_max[0]) & (x[1] >= V.box_min[1]) & (x[1] <= V.box_max[1]) &
               (x[2] >= V.box_min[2]) & (x[2] <= V.box_max[2]);
    // the checks of a step's start as one branch
    if (!((L.n < L.maxSteps) & (L.t < L.maxTime) & (L.s < V.maxdist_eff) & !(L.r2 <= V.rin2_eff) & inside & !L.bad)) {
      if (L.n >= L.maxSteps) return 4;
      if (!(L.s < V.maxdist_eff) && L.s >= V.maxdist_eff) return 5;
      if (L.t >= L.maxTime) return 3;
      if (!(L.t < L.maxTime && L.s < V.maxdist_eff) || L.bad) return 8;
      return L.r2 <= V.rin2_eff ? 1 : 0;
    }
    const float u2 = sumsq(u[1], u[0], u[2]);
    const float w = 1.0f + u2;
    const float igam = rsqrtf(w);
    // the field (bfield32)
    const float xf[3] = {(float)x[0], (float)x[1], (float)x[2]};
    const float ir = rsqrtf(sumsq(xf[0], xf[1], xf[2]));
    const float ir2 = ir * ir, ir3 = ir2 * ir;
    const float mdr = fmaf(V.mhat[2], xf[2], fmaf(V.mhat[1], xf[1], V.mhat[0] * xf[0]));
    const float k5 = 3.0f * mdr * ir3 * ir2;
    float b[3];
#pragma unroll
    for (int d = 0; d < 3; d++) b[d] = fmaf(V.cb, fmaf(k5, xf[d], -(V.mhat[d] * ir3)), V.bext[d]);
    // time step (normalized)
    double dt = L.dtTrace;
    const double trem = L.maxTime - L.t;
    if (trem < dt) dt = trem;
    if (V.adaptive) {
      const float bm2 = sumsq(b[1], b[0], b[2]);
      // dphi / omega with omega = |B| / gamma, gamma = (1 + u^2) / sqrt(1 + u^2)
      if (bm2 > 0.0f) dt = dmin(dt, (double)(V.dphi * (w * igam) * rsqrtf(bm2)));
      if (LIM) {
        const float vmag = sqrtf(u2) * igam;
        if (V.dist_limiter) {
          const double r = sqrt(L.r2);
          double dIn = 1.0e300, dOut = 1.0e300;
          if (r > V.rin) dIn = r - V.rin;
          if (SPHERE) {
            if (r < V.rout) dOut = V.rout - r;
          } else {
            dOut = dmin(dmin(dmin(V.box_max[0] - x[0], x[0] - V.box_min[0]), dmin(V.box_max[1] - x[1], x[1] - V.box_min[1])),
                        dmin(V.box_max[2] - x[2], x[2] - V.box_min[2]));
          }
          const double dn = dmin(dIn, dOut);
          if (vmag > 0.0f && dn < 1.0e299) dt = dmin(dt, 0.20 * dn / (double)vmag);
        }
        if (V.dt_floor) {
          const double sv = dmax((double)vmag, 1.0e-12 / C_LIGHT);
          const double fl = dmax(dmax(V.floor_abs, V.floor_rel), V.floor_dist / sv);
          dt = dmax(fl, dt);
        }
      }
      if (trem > 0.0) dt = dmin(dt, trem);
    }
    if (!(dt > 0.0) || !isfinite(dt)) return 6;
    // drift - kick - drift (rotate32 between two half drifts)
    const float hf = 0.5f * (float)dt;
    const double xb[3] = {x[0], x[1], x[2]};
#pragma unroll
    for (int d = 0; d < 3; d++) x[d] += (double)(hf * (u[d] * igam));
    const float tc = hf * igam;
    const float t[3] = {tc * b[0], tc * b[1], tc * b[2]};
    const float sc = 2.0f * __builtin_amdgcn_rcpf(1.0f + sumsq(t[1], t[0], t[2]));
    const float s[3] = {sc * t[0], sc * t[1], sc * t[2]};
    const float pp[3] = {u[0] + fmaf(u[1], t[2], -(u[2] * t[1])), u[1] + fmaf(u[2], t[0], -(u[0] * t[2])),
                         u[2] + fmaf(u[0], t[1], -(u[1] * t[0]))};
    u[0] = u[0] + fmaf(pp[1], s[2], -(pp[2] * s[1]));
    u[1] = u[1] + fmaf(pp[2], s[0], -(pp[0] * s[2]));
    u[2] = u[2] + fmaf(pp[0], s[1], -(pp[1] * s[0]));
    const float w2 = fmaf(u[2], u[2], fmaf(u[1], u[1], fmaf(u[0], u[0], 1.0f)));
    const float igam2 = rsqrtf(w2);
#pragma unroll
    for (int d = 0; d < 3; d++) x[d] += (double)(hf * (u[d] * igam2));
    const float dd[3] = {(float)(x[0] - xb[0]), (float)(x[1] - xb[1]), (float)(x[2] - xb[2])};
    const float seg = sqrtf(sumsq(dd[1], dd[0], dd[2]));
    // the chord can reach the inner sphere only if it starts within its
    // length of the sphere (rin_c: 1e-4 of slack for the FP32 lengths); the
    // exact FP64 test runs only then
    const float reach = seg + V.rin_c;
    if (V.rin > 0.0 && !((float)L.r2 > reach * reach))
      if (seg_hits(xb, x, V.rin) || inside_inner_m(x, V.rin)) return 1;
    const double r2n = dot3(x, x);
    // a finite sum of squares: every component is finite
    if (!isfinite(r2n) || !isfinite(w2))
      if (!fin3(x) || !isfinite(u[0]) || !isfinite(u[1]) || !isfinite(u[2])) return 8;
    L.r2 = r2n;
    L.s += isfinite(seg) ? (double)seg : 0.0;
    L.t += dt;
    ++L.n;
    return -1;
  }
  static __device__ __forceinline__ int steps_of(const Lane& L) { return L.n; }
  static __device__ __forceinline__ void result(const View& V, const Lane& L, int term, amps_trace_result& r) {
    const double T = V.len / C_LIGHT;
    const double pu = V.m0 * C_LIGHT;
    r.termination = term;
    r.retry_count = L.retry;
    r.steps = L.n;
    r.time_s = L.t * T;
    r.distance_m = L.s * V.len;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      r.x[d] = L.x[d] * V.len;
      r.p[d] = (double)L.u[d] * pu;
    }
  }
};

// The work of a launch (TraceView's, without the physics).
struct ScanWork {
  int chunk, nR, W, retry;
  int64_t nitems, nloc;
  double inv_nloc;
  unsigned long long *queue, *steps_total;
  const double *x0, *dir, *R, *grid;
  const int *lo, *hi;
  amps_trace_result* out;
  int8_t* states;
  int *cutoff, *pend, *status;
  // BRACKET: the locations whose rescan has opened, in order of opening (-1:
  // not yet stored), their number, the tickets drawn for rescan items, and
  // the bracket items not yet retired
  int* open_list;
  unsigned long long *n_open, *tickets, *bracket_left;
  int* stop;              // UPPER: highest non-allowed bin found so far, -1 none
  uint32_t* item_steps;   // UPPER: [nloc][nR] steps of each traced bin
};

__device__ __forceinline__ unsigned long long load_count(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// a location's rescan opens: its other bins become items
__device__ __forceinline__ void open_rescan(const ScanWork& a, int loc) {
  store_status(a.status + loc, 2);
  const unsigned long long i = atomicAdd(a.n_open, 1ull);
  __hip_atomic_store(a.open_list + i, loc, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

// k_trace_persistent with the mode as a template parameter (LIST and FULL as
// there).
//
// BRACKET traces the same bins and reads them off the same way, but a lane
// that finds no bracket item left takes a ticket for the i-th rescan item
// instead of drawing (and mostly skipping) every location's other bins: the
// item is bin i % (nR - W) of the other bins of the i / (nR - W)-th location
// to open.  A location's rescan therefore fills neighbouring lanes of one or
// two wavefronts, where holding one bin of each unresolved location a lane
// spread every rescan over the whole grid, one active lane a wavefront
// (32,768 pairs, one set of directions: 310 against 210 ms with two wavefronts
// per SIMD, 152 against 145 with one; eight other sets take 147 to 190 with one;
// the longest trajectory alone takes 75).  A lane whose item has not opened waits; every bracket item
// has been drawn and is being traced by then, and when the last of them
// retires no further rescan opens, so every wait ends.
//
// UPPER: instead of one lane walking a location's
// bins downward one after the other (the longest walk of 48 trajectories
// bounded the launch: 0.59 s at 131,738 locations in FP32, 0.147 s now),
// every (location, bin) is an item of its own, the top bins of all locations
// first.  An item below a bin already found not allowed is skipped, or
// dropped when its lane next looks; every bin down to the first not-allowed
// one is always traced.  k_upper_read then walks each location's samples as
// the sequential scan would, counts the steps of the bins that scan visits
// and unmarks the others.
template <class S, int MODE>
__global__ __launch_bounds__(256) void k_trace_mode(typename S::View v, ScanWork a) {
  typename S::Lane L;
  int64_t item = -1;
  int loc = 0, bin = 0, attempt = 0;
  bool has = false, done = false, wait = false;
  int64_t my_steps = 0;
  int64_t failed_steps = 0;  // UPPER: of the item's first attempt
  const int lane = __lane_id();
  constexpr bool BRK = MODE == TRACE_MODE_BRACKET, UPPER = MODE == TRACE_MODE_UPPER;
  constexpr int ROUNDS = UPPER ? 8 : 1;
  for (;;) {
    if (BRK && wait) {
      // the count of bracket items before the count of opened locations: no
      // opening is missed when the former is zero
      const bool last = load_count(a.bracket_left) == 0;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      const int64_t nother = a.nR - a.W;
      if (item < (int64_t)load_count(a.n_open) * nother) {
        const int64_t i = item / nother;
        const int l = load_status(a.open_list + i);
        if (l >= 0) {
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
          wait = false;
          loc = l;
          const int k2 = (int)(item - i * nother), lo = a.lo[loc];
          bin = k2 < lo ? k2 : k2 + a.W;
          S::init(v, L, a.x0 + 3 * (int64_t)loc, a.dir + 3 * (int64_t)loc, a.grid[bin], 0);
        }
      } else if (last) {
        wait = false;
        has = false;
        done = true;
      }
    }
    if (UPPER && has && load_status(a.stop + loc) > bin) has = false;
    for (int round = 0; round < ROUNDS; round++) {
      const bool need = !has && !done;
      const uint64_t mask = __ballot(need);
      if (!mask) break;
      const int leader = __ffsll((long long)mask) - 1;
      unsigned long long base = 0;
      if (lane == leader) base = atomicAdd(a.queue, (unsigned long long)__popcll(mask));
      base = __shfl(base, leader);
      if (need) {
        const uint64_t below = (lane == 0) ? 0ull : (mask & ((1ull << lane) - 1ull));
        const int64_t my = (int64_t)(base + (unsigned long long)__popcll(below));
        if (my < a.nitems) {
          item = my;
          attempt = 0;
          has = true;
          failed_steps = 0;
          double R;
          if constexpr (MODE == TRACE_MODE_LIST) {
            loc = (int)item;
            R = a.R[item];
          } else {
            // item = level * nloc + loc (items below 2^41: exact in double)
            int64_t kk = (int64_t)((double)item * a.inv_nloc), rem = item - kk * a.nloc;
            if (rem < 0) kk--, rem += a.nloc;
            if (rem >= a.nloc) kk++, rem -= a.nloc;
            loc = (int)rem;
            const int lo = a.lo ? a.lo[loc] : 0;
            if constexpr (MODE == TRACE_MODE_FULL) {
              // every location's lowest rigidities first: the longest
              // trajectories (quasi-trapped, up to the step cap) start first
              bin = lo + (int)kk;
            } else if constexpr (UPPER) {
              bin = (a.hi ? a.hi[loc] : a.nR - 1) - (int)kk;
              if (bin < lo || load_status(a.stop + loc) > bin) has = false;
            } else {
              // the bins just below the bracket's centre first, where the
              // quasi-trapped (longest) trajectories are
              const int half = a.W / 2, k = (int)kk;
              bin = lo + (k < half ? half - 1 - k : k);
            }
            R = has ? a.grid[bin] : 0.0;
          }
          if (has) S::init(v, L, a.x0 + 3 * (int64_t)loc, a.dir + 3 * (int64_t)loc, R, 0);
        } else if (BRK && a.nR > a.W) {
          item = (int64_t)atomicAdd(a.tickets, 1ull);  // the wavefront's lanes: consecutive tickets
          attempt = 0;
          has = wait = true;
        } else {
          done = true;
        }
      }
    }
    if (__ballot(has) == 0ull) {
      if (__ballot(!done) == 0ull) break;
      continue;  // every draw of these rounds was skipped
    }
    // a wavefront whose lanes all wait for bracket results yields its issue slots
    if (BRK && __ballot(has && !wait) == 0ull) __builtin_amdgcn_s_sleep(64);
    for (int k = 0; k < a.chunk && has && !wait; k++) {
      const int term = S::step(v, L);
      if (term < 0) continue;
      if (a.retry && attempt == 0 && retryable(a.retry, term)) {
        attempt = 1;
        if (UPPER) failed_steps = S::steps_of(L);
        else my_steps += S::steps_of(L);
        S::init(v, L, a.x0 + 3 * (int64_t)loc, a.dir + 3 * (int64_t)loc,
                MODE == TRACE_MODE_LIST ? a.R[item] : a.grid[bin], 1);
        continue;
      }
      if (!UPPER) my_steps += S::steps_of(L);
      has = false;
      if constexpr (MODE == TRACE_MODE_LIST) {
        amps_trace_result r;
        S::result(v, L, term, r);
        a.out[item] = r;
      } else if constexpr (MODE == TRACE_MODE_FULL) {
        a.states[(int64_t)loc * a.nR + bin] = state_of(term);
      } else if constexpr (UPPER) {
        const int8_t sv = state_of(term);
        a.states[(int64_t)loc * a.nR + bin] = sv;
        a.item_steps[(int64_t)loc * a.nR + bin] = (uint32_t)(failed_steps + S::steps_of(L));
        if (sv != 1) atomicMax(a.stop + loc, bin);
      } else {
        int8_t* s = a.states + (int64_t)loc * a.nR;
        const int8_t sv = state_of(term);
        s[bin] = sv;
        const int top = a.lo[loc] + a.W - 1;
        const bool in_bracket = bin >= a.lo[loc] && bin <= top;
        if (bin == top && sv != 1 && top < a.nR - 1 && load_status(a.status + loc) == 0) {
          // the bracket's top is not allowed below the grid's top: the
          // transition lies above the bracket, whatever its other bins give,
          // so the rescan starts now (counted before this bin is retired)
          atomicAdd(a.pend + loc, a.nR - a.W);
          open_rescan(a, loc);
        }
        // the sample (and any rescan count and phase) before this item retires
        __threadfence();
        if (atomicSub(a.pend + loc, 1) == 1) {
          // this location's phase is complete: every sample of it is visible
          __threadfence();
          const int phase = load_status(a.status + loc);
          const int lo = phase == 0 ? a.lo[loc] : 0;
          const int hi = phase == 0 ? lo + a.W - 1 : a.nR - 1;
          int b;
          if (bin_from_samples(s, lo, hi, a.nR, b)) {
            a.cutoff[loc] = b;
            if (phase == 0) store_status(a.status + loc, 1);
          } else {
            // allowed down to a bottom above Rmin: the other bins, then the whole grid
            __hip_atomic_store(a.pend + loc, a.nR - a.W, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            open_rescan(a, loc);
          }
        }
        if (in_bracket) {
          __threadfence();  // any opening before this item is counted off
          atomicSub(a.bracket_left, 1ull);
        }
      }
    }
  }
  if (UPPER) return;  // counted by k_upper_read
  unsigned long long tot = (unsigned long long)my_steps;
  for (int off = 32; off > 0; off >>= 1) tot += __shfl_down(tot, off);
  if (lane == 0 && a.steps_total) atomicAdd(a.steps_total, tot);
}

// The downward scan read off the samples (UPPER): the visited bins' steps,
// the cutoff as the sequential scan leaves it, -1 for the bins below.
__global__ __launch_bounds__(256) void k_upper_read(ScanWork a) {
  const int64_t loc = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  unsigned long long tot = 0;
  if (loc < a.nloc) {
    int8_t* s = a.states + loc * a.nR;
    const uint32_t* st = a.item_steps + loc * a.nR;
    const int lo = a.lo ? a.lo[loc] : 0;
    int bin = a.hi ? a.hi[loc] : a.nR - 1;
    for (;; bin--) {
      tot += st[bin];
      if (s[bin] != 1 || bin == lo) break;
    }
    a.cutoff[loc] = s[bin] == 1 ? bin : bin + 1;
    for (int k = bin - 1; k >= lo; k--) s[k] = -1;
  }
  for (int off = 32; off > 0; off >>= 1) tot += __shfl_down(tot, off);
  if ((threadIdx.x & 63) == 0 && a.steps_total) atomicAdd(a.steps_total, tot);
}

// ---------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------
// Workgroups per CU of a launch (one: a wavefront per SIMD).  Two keep the
// arithmetic units fed; more only slow each of the longest trajectories,
// which end a launch (full FP64 map: 177, 142, 175, 220 ms with 1, 2, 3, 4;
// FP32: 152, 95, 106, 128 ms).  One where trajectories follow one another or
// are traced ahead of need, so that the longest come late: the bracketed mode
// (32,768 pairs, one set of directions: 145, 210, 260, 260 ms) and FP64 downward scans of fewer
// locations than two wavefronts per SIMD have lanes (16,384: 91, 170, 215,
// 220 ms; FP32, 131,738: 195, 147, 158, 181 ms).
int fast_wgs_per_cu(int mode, int precision, int64_t nloc, int n_cu) {
  if (mode == TRACE_MODE_BRACKET) return 1;
  if (mode == TRACE_MODE_UPPER && precision == AMPS_FP64 && nloc < (int64_t)n_cu * 512) return 1;
  return 2;
}

bool in_range(double v, double lo, double hi) { return v >= lo && v <= hi; }  // false for NaN

// The constants of a fast FP64 launch; false when the launch is outside what
// the fast step covers (another mover, field, selector or policy, no gyro
// budget, no inner sphere, or constants that could take an operand of the
// step out of the range in which its arithmetic is the IEEE operations').
bool fast64_view(const TraceView& a, Fast64View& V) {
  const amps_trace_params& P = a.P;
  if (P.mover != MV_BORIS || P.field_model != 0 || P.dt_selector != 0 || P.policy != 0 || P.trap || !P.adaptive)
    return false;
  if (P.max_steps > ((int64_t)1 << 29)) return false;
  const double mc = P.m0_kg * C_LIGHT;
  V.mc2 = mc * mc;
  V.m0 = P.m0_kg;
  V.q = P.q_C;
  V.qabs = std::fabs(P.q_C);
  V.dphi = P.dphi_max;
  bool ok = in_range(V.m0, 0x1p-160, 0x1p+40) && in_range(V.qabs, 0x1p-120, 0x1p+40) &&
            in_range(P.qabs_C, 0x1p-120, 0x1p+40) && P.qabs_C == V.qabs && in_range(V.dphi, 0x1p-60, 0x1p+30);
  for (int d = 0; d < 3; d++) {
    V.M[d] = P.moment_Am2 * P.m_hat[d];
    V.Bext[d] = P.B_ext_T[d];
    ok = ok && (V.M[d] == 0.0 || in_range(std::fabs(V.M[d]), 0x1p-100, 0x1p+120)) &&
         (V.Bext[d] == 0.0 || in_range(std::fabs(V.Bext[d]), 0x1p-100, 0x1p+60));
    V.box_min[d] = a.box_min_m[d];
    V.box_max[d] = a.box_max_m[d];
  }
  V.rin = a.r_inner_m;
  V.rin2 = V.rin * V.rin;
  V.rin_far = 1.0001 * V.rin;
  V.rout2 = a.r_outer_m * a.r_outer_m;
  ok = ok && in_range(V.rin, 0x1p-20, 0x1p+70);
  V.dt_trace = P.dt_trace_s;
  V.dt_trace1 = std::max(1.0e-12, 0.5 * P.dt_trace_s);
  V.max_time = P.max_time_s;
  V.max_time1 = 2.0 * P.max_time_s;
  ok = ok && V.dt_trace >= 0x1p-200 && V.max_time >= 0x1p-100;
  V.maxdist = P.max_distance_m;
  V.maxdist_eff = V.maxdist <= 0.0 ? HUGE_VAL : V.maxdist;
  V.max_steps = (int)P.max_steps;
  V.max_steps1 = (int)(2 * P.max_steps);
  return ok;
}

// The constants of an FP32 launch; false for the steps and movers that only
// the general kernel runs.
bool fast32_view(const TraceView& a, Fast32View& V) {
  const amps_trace_params& P = a.P;
  if (P.mover != MV_BORIS || P.max_steps > ((int64_t)1 << 29)) return false;
  const double T = a.len / C_LIGHT;
  V.len = a.len;
  V.rin = a.rin_n, V.rin2_eff = a.rin_n > 0.0 ? a.rin_n * a.rin_n : -1.0;
  V.rout = a.rout_n, V.rout2 = a.rout_n * a.rout_n;
  V.maxdist_eff = a.maxdist_n <= 0.0 ? HUGE_VAL : a.maxdist_n;
  V.floor_abs = a.floor_abs_n, V.floor_rel = a.floor_rel_n, V.floor_dist = a.floor_dist_n;
  V.dt_trace = P.dt_trace_s / T;
  V.dt_trace1 = std::max(1.0e-12, 0.5 * P.dt_trace_s) / T;
  V.max_time = P.max_time_s / T;
  V.max_time1 = 2.0 * P.max_time_s / T;
  V.m0 = P.m0_kg, V.qabs = P.qabs_C;
  V.cb = a.f_cb, V.dphi = a.f_dphi, V.rin_c = (float)a.rin_n * 1.0001f;
  for (int d = 0; d < 3; d++) {
    V.mhat[d] = a.f_mhat[d], V.bext[d] = a.f_bext[d];
    V.box_min[d] = P.box_min_Re[d], V.box_max[d] = P.box_max_Re[d];
  }
  V.max_steps = (int)P.max_steps;
  V.max_steps1 = (int)(2 * P.max_steps);
  V.adaptive = P.adaptive, V.dist_limiter = P.dist_limiter, V.dt_floor = P.dt_floor;
  return true;
}

template <class S>
void launch_mode(amps_ctx* c, const typename S::View& v, const ScanWork& w, int mode, dim3 g) {
  switch (mode) {
    case TRACE_MODE_LIST: hipLaunchKernelGGL((k_trace_mode<S, TRACE_MODE_LIST>), g, dim3(256), 0, c->stream, v, w); break;
    case TRACE_MODE_FULL: hipLaunchKernelGGL((k_trace_mode<S, TRACE_MODE_FULL>), g, dim3(256), 0, c->stream, v, w); break;
    case TRACE_MODE_UPPER: hipLaunchKernelGGL((k_trace_mode<S, TRACE_MODE_UPPER>), g, dim3(256), 0, c->stream, v, w); break;
    default: hipLaunchKernelGGL((k_trace_mode<S, TRACE_MODE_BRACKET>), g, dim3(256), 0, c->stream, v, w); break;
  }
}

}  // namespace
