// Device-side skeleton of the generated right-hand-side kernels.
//
// This header is not compiled with the library: its text is embedded into libmolgpu.so and
// handed to hiprtc together with the source that mol_jit.cpp generates for one PDE system.
// The generated source defines MOL_T (double or float) before including this header, then a
// struct `Geo` with the tile geometry as constants and the per-node right-hand side
// `Geo::node`, whose operator weights, constants and programs are folded into straight-line
// code.  The tile kernel below stages the tile plus halo into LDS with periodic wrap and runs
// the node function with the fused Runge-Kutta stage epilogue.
#pragma once

typedef MOL_T T;
typedef long long i64;

// Layout identical to mol::Epi<T> of the library (passed by value as a kernel argument).
struct Epi {
  int mode;
  int subA;
  T* out;
  const T* A;
  const T* B;
  T* acc;
  T* comp;
  double ca, cb, cf, acc_keep, acc_f;
  const double* tnow;
  double tofs;
  const T* p;
  double* tnext;   // last stage of a step: *tnext = *tnow + tadv (double-buffered device clock)
  double tadv;
};

__device__ __forceinline__ void mol_advance_clock(const Epi& ep) {
  if (ep.tnext && blockIdx.x == 0 && threadIdx.x == 0) ep.tnext[0] = ep.tnow[0] + ep.tadv;
}

// Constant memory (tables, coordinates, instance headers: no kernel that reads through this type
// writes them): loads are hoisted out of loops, and are scalar where the address is uniform.
#ifdef __AMDGCN__
typedef const __attribute__((address_space(4))) double* MolRow;
#else
typedef const double* MolRow;
#endif

#ifdef __AMDGCN__
typedef const __attribute__((address_space(4))) T* MolPar;
#else
typedef const T* MolPar;
#endif

// Node coordinates and auxiliary grid arrays (layout identical to mol::JitPtrs<T>).
struct JPtrs {
  const double* coord[3];
  const T* aux[8];
  const double* pool;      // weight pool: per-node rows of nonuniform axes
  const double* wtab[3];   // per axis: nonuniform WENO5 coefficient rows (MOL_NU_NC per node)
};

// Fused epilogue of one Runge-Kutta stage:
//   mode 0:  out = f
//   mode 1:  out = ca*A + cb*B + cf*f ;  acc = acc_keep*acc + acc_f*f  (if acc)
//   mode 2:  compensated update  out = A (+) [cb*(B - subA*A) + cf*f]  with Kahan term comp
template <class I>
__device__ __forceinline__ void mol_epilogue(const Epi& ep, const I idx, T f) {
  if (ep.mode == 0) {
    ep.out[idx] = f;
    return;
  }
  if (ep.mode == 1) {
    T v = (T)ep.cf * f;
    if (ep.A) v += (T)ep.ca * ep.A[idx];
    if (ep.B) v += (T)ep.cb * ep.B[idx];
    if (ep.acc) {
      T a = (T)ep.acc_f * f;
      if (ep.acc_keep != 0.0) a += (T)ep.acc_keep * ep.acc[idx];
      ep.acc[idx] = a;
    }
    ep.out[idx] = v;
    return;
  }
  const T a = ep.A[idx];
  T incr = (T)ep.cf * f;
  if (ep.B) incr += (T)ep.cb * (ep.subA ? (ep.B[idx] - a) : ep.B[idx]);
  const T y = incr - ep.comp[idx];
  const T s = a + y;
  ep.comp[idx] = (s - a) - y;
  ep.out[idx] = s;
}

// The epilogue of CH nodes at once (ok[k]: node k exists; out[k][f] at index idx[k] + dv[f]):
// every operand load of the CH nodes is issued before the first store, so one memory latency
// is exposed per chunk instead of one per node.
template <int CH, int NF>
__device__ __forceinline__ void mol_epilogue_chunk(const Epi& ep, const i64 (&idx)[CH], const bool (&ok)[CH],
                                                   const i64 (&dv)[NF], const T (&out)[CH][NF]) {
  if (ep.mode == 0) {
#pragma unroll
    for (int k = 0; k < CH; ++k)
      if (ok[k])
#pragma unroll
        for (int f = 0; f < NF; ++f) ep.out[idx[k] + dv[f]] = out[k][f];
    return;
  }
  T a[CH][NF], b[CH][NF], c[CH][NF];
  const bool keep = ep.mode == 1 && ep.acc && ep.acc_keep != 0.0;
#pragma unroll
  for (int k = 0; k < CH; ++k)
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const i64 i = idx[k] + dv[f];
      a[k][f] = ok[k] && ep.A ? ep.A[i] : T(0);
      b[k][f] = ok[k] && ep.B ? ep.B[i] : T(0);
      c[k][f] = ok[k] && (ep.mode == 2 || keep) ? (ep.mode == 2 ? ep.comp[i] : ep.acc[i]) : T(0);
    }
#pragma unroll
  for (int k = 0; k < CH; ++k) {
    if (!ok[k]) continue;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const i64 i = idx[k] + dv[f];
      const T fv = out[k][f];
      if (ep.mode == 1) {
        T v = (T)ep.cf * fv;
        if (ep.A) v += (T)ep.ca * a[k][f];
        if (ep.B) v += (T)ep.cb * b[k][f];
        if (ep.acc) {
          T ac = (T)ep.acc_f * fv;
          if (ep.acc_keep != 0.0) ac += (T)ep.acc_keep * c[k][f];
          ep.acc[i] = ac;
        }
        ep.out[i] = v;
      } else {
        T incr = (T)ep.cf * fv;
        if (ep.B) incr += (T)ep.cb * (ep.subA ? (b[k][f] - a[k][f]) : b[k][f]);
        const T y = incr - c[k][f];
        const T sm = a[k][f] + y;
        ep.comp[i] = (sm - a[k][f]) - y;
        ep.out[i] = sm;
      }
    }
  }
}

// Single periodic wrap of a node index onto the ring 2..n (node 1 is the image of node n).
__device__ __forceinline__ int mol_wrap(int k, int n) {
  return k <= 1 ? k + (n - 1) : (k > n ? k - (n - 1) : k);
}

__device__ __forceinline__ T mol_sign(T a) { return a > T(0) ? T(1) : (a < T(0) ? T(-1) : T(0)); }
__device__ __forceinline__ T mol_heaviside(T a) { return a > T(0) ? T(1) : (a < T(0) ? T(0) : T(0.5)); }

// x^e for |e| > 3 by repeated squaring (small exponents are expanded by the generator).
__device__ __noinline__ T mol_powi(T x, int e) {
  const bool neg = e < 0;
  unsigned m = neg ? (unsigned)(-e) : (unsigned)e;
  T r = T(1), base = x;
  while (m) {
    if (m & 1u) r *= base;
    base *= base;
    m >>= 1;
  }
  return neg ? T(1) / r : r;
}

// FP64 quotient n / d for the WENO5 weights: the hardware reciprocal (v_rcp_f64, about 23 good
// bits) refined by one Newton step (46 bits) and the quotient corrected by its residual
// (Markstein; the correction's relative error is the square of the reciprocal's): 6 instructions
// against about 11 for the IEEE division sequence, within an ulp of the IEEE quotient.
// d is a positive normal number here (a product of sums of squares offset by eps).
__device__ __forceinline__ double mol_quot(const double n, const double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  const double q = n * r;
  return fma(r, fma(-d, q, n), q);
}

// What both forms of the Jiang-Shu WENO5 node derivative (u^-_{i+1/2} - u^+_{i-1/2}) / dx share,
// from the five values u(i-2) .. u(i+2).  Every candidate reconstruction is the central one plus
// a multiple of a third difference: with E = D2_{i+1} - D2_i, F = D2_i - D2_{i-1} and weights
// proportional to g_k w_k (w_k = 1 / (eps + beta_k)^2 up to one common factor),
//   6 (u^- - u^+) = 3 (u_{i+1} - u_{i-1}) - (3 X + 2 Y) / Dp - (2 X + 3 Y) / Dm,
//   X = w_1 E,  Y = w_3 F,  Dp = 3 w_1 + 6 w_2 + w_3,  Dm = w_1 + 6 w_2 + 3 w_3
// (w_1: the stencil i .. i+2).  The smoothness sums are formed as 4 (eps + beta_k) = 13/3 D2^2 +
// a^2 + 4 eps.  Sums that the neighbouring node along the axis shares (differences, D2, the
// 13/3 D2^2 terms) are written as expressions of their own.
template <class U>
struct MolWeno5 {
  U a2, E, F, b1, b2, b3;
  __device__ __forceinline__ MolWeno5(U um2, U um1, U u0, U up1, U up2, T eps) {
    const U dmm = um1 - um2, dm = u0 - um1, dp = up1 - u0, dpp = up2 - up1;
    const U D2m = dm - dmm, D20 = dp - dm, D2p = dpp - dp;
    const U a1 = T(-2) * dp + D2p, a3 = T(2) * dm + D2m;
    a2 = dm + dp;
    E = D2p - D20;
    F = D20 - D2m;
    const T eps4 = T(4) * eps;
    b1 = a1 * a1 + ((T(13.0 / 3.0) * D2p) * D2p + eps4);
    b2 = a2 * a2 + ((T(13.0 / 3.0) * D20) * D20 + eps4);
    b3 = a3 * a3 + ((T(13.0 / 3.0) * D2m) * D2m + eps4);
  }
  // the derivative from the weights
  __device__ __forceinline__ U apply(const U w1, const U w2, const U w3, const T inv_dx) const {
    const U X = w1 * E, Y = w3 * F;
    const U Dp = T(3) * w1 + (T(6) * w2 + w3), Dm = T(3) * w3 + (T(6) * w2 + w1);
    const U Np = T(3) * X + T(2) * Y, Nm = T(2) * X + T(3) * Y;
    return (T(0.5) * inv_dx) * a2 - (inv_dx * T(1.0 / 6.0)) * mol_quot(Np * Dm + Nm * Dp, Dp * Dm);
  }
};

// FP64: w_k cleared to the product of the other two (4 (eps + beta_j))^2, so the derivative has
// one quotient.  48 instructions per derivative (61 with the candidate values and both normalised
// weight sets formed separately): Burgers right-hand side at 4096^2 103 -> 92 us.
template <class U>
__device__ __forceinline__ U mol_weno5_t(U um2, U um1, U u0, U up1, U up2, T eps, T inv_dx) {
  const MolWeno5<U> s(um2, um1, u0, up1, up2, eps);
  const U q1 = s.b1 * s.b1, q2 = s.b2 * s.b2, q3 = s.b3 * s.b3;
  return s.apply(q2 * q3, q1 * q3, q1 * q2, inv_dx);
}

// Reciprocal and quotient for the FP32 WENO5 weights: the hardware reciprocal (v_rcp_f32,
// within 1 ulp) refined by one Newton step, and the quotient corrected by its residual
// (Markstein), which is the correctly rounded result but for rare ties, in 3 and 5
// instructions against about 10 for the IEEE division sequence.  FP64: plain divisions.
__device__ __forceinline__ float mol_rcp(const float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(r, fmaf(-x, r, 1.0f), r);
}
__device__ __forceinline__ double mol_rcp(const double x) { return 1.0 / x; }
__device__ __forceinline__ float mol_quot(const float n, const float d) {
  const float r = mol_rcp(d);
  const float q = n * r;
  return fmaf(fmaf(-d, q, n), r, q);
}

__device__ __forceinline__ double mol_val(double v) { return v; }
__device__ __forceinline__ float mol_val(float v) { return v; }

// FP32, where products of four squared smoothness sums (~eps^8) underflow: w_k = (b / b_k)^2 with
// b the smallest of the three sums, so every weight lies in (0, 1], at least one is 1, and
// neither the sums nor the quotient leave the FP32 range whatever eps and the state's scale.
// One quotient instead of two and no cancellation of the two face values (SSPRK3 step of the
// FP32 + Kahan Burgers system at 1447^2: 67 -> 50 us).
template <class U>
__device__ __forceinline__ U mol_weno5_ref_t(U um2, U um1, U u0, U up1, U up2, T eps, T inv_dx) {
  const MolWeno5<U> s(um2, um1, u0, up1, up2, eps);
  const T b = fmin(fmin(mol_val(s.b1), mol_val(s.b2)), mol_val(s.b3));
  const U r1 = b * mol_rcp(s.b1), r2 = b * mol_rcp(s.b2), r3 = b * mol_rcp(s.b3);
  return s.apply(r1 * r1, r2 * r2, r3 * r3, inv_dx);
}

__device__ __forceinline__ T mol_weno5(T um2, T um1, T u0, T up1, T up2, T eps, T inv_dx) {
  return mol_weno5_t<T>(um2, um1, u0, up1, up2, eps, inv_dx);
}
__device__ __forceinline__ T mol_weno5_ref(T um2, T um1, T u0, T up1, T up2, T eps, T inv_dx) {
  return mol_weno5_ref_t<T>(um2, um1, u0, up1, up2, eps, inv_dx);
}

// Forward-mode dual number (value, derivative) for the gradient of the WENO reconstruction.
struct MolDual {
  T v, d;
};
__device__ __forceinline__ MolDual operator+(MolDual a, MolDual b) { return {a.v + b.v, a.d + b.d}; }
__device__ __forceinline__ MolDual operator-(MolDual a, MolDual b) { return {a.v - b.v, a.d - b.d}; }
__device__ __forceinline__ MolDual operator*(MolDual a, MolDual b) { return {a.v * b.v, a.d * b.v + a.v * b.d}; }
__device__ __forceinline__ MolDual operator/(MolDual a, MolDual b) {
  const T q = a.v / b.v;
  return {q, (a.d - q * b.d) / b.v};
}
__device__ __forceinline__ MolDual operator+(MolDual a, T b) { return {a.v + b, a.d}; }
__device__ __forceinline__ MolDual operator+(T a, MolDual b) { return {a + b.v, b.d}; }
__device__ __forceinline__ MolDual operator*(T a, MolDual b) { return {a * b.v, a * b.d}; }
__device__ __forceinline__ MolDual operator*(MolDual a, T b) { return {a.v * b, a.d * b}; }
__device__ __forceinline__ MolDual operator/(MolDual a, T b) { return {a.v / b, a.d / b}; }
__device__ __forceinline__ MolDual operator/(T a, MolDual b) {
  const T q = a / b.v;
  return {q, -q * b.d / b.v};
}
__device__ __forceinline__ MolDual mol_rcp(const MolDual x) {
  const T r = mol_rcp(x.v);
  return {r, -(x.d * r) * r};
}
__device__ __forceinline__ MolDual mol_quot(const MolDual n, const MolDual d) { return n / d; }

__device__ __forceinline__ T mol_val(MolDual v) { return v.v; }

// Gradient of the WENO5 node derivative with respect to its five inputs.
__device__ __noinline__ void mol_weno5_grad(T um2, T um1, T u0, T up1, T up2, T eps, T inv_dx, T* g, bool cleared) {
  const T x[5] = {um2, um1, u0, up1, up2};
  for (int k = 0; k < 5; ++k) {
    MolDual d[5];
    for (int j = 0; j < 5; ++j) d[j] = MolDual{x[j], j == k ? T(1) : T(0)};
    const MolDual r = cleared ? mol_weno5_t<MolDual>(d[0], d[1], d[2], d[3], d[4], eps, inv_dx)
                              : mol_weno5_ref_t<MolDual>(d[0], d[1], d[2], d[3], d[4], eps, inv_dx);
    g[k] = r.d;
  }
}

// ---- node-centred WENO5 on nonuniform coordinates (weno_f_nonuniform,
//      src/discretization/schemes/WENO/nonuniform_weno.jl): Fornberg 3-point sub-stencil weights
//      (:5-46), Simpson smoothness indicators (:54-73), target geometry (:76-82), closed-form
//      ideal weights (:85-118), Shi-Hu-Shu splitting with theta = 3 (:120-163).  Coordinates and
//      weights in FP64, values in U (T, or MolDual for the gradient).
__device__ __forceinline__ void mol_fornberg3(const double a0, const double a1, const double a2, const double xt,
                                              double* m0, double* m1, double* m2) {
  double n1m0 = 1.0, n1m1 = 0.0, n1m2 = 0.0, c1 = 1.0;
  double c2 = a1 - a0;
  const double r1 = c1 / c2;
  const double tA = a1 - xt;
  const double a1m0 = (tA * n1m0) / c2, a1m1 = (tA * n1m1 - n1m0) / c2, a1m2 = (tA * n1m2 - 2.0 * n1m1) / c2;
  const double sB = a0 - xt;
  const double a2m0 = r1 * (-(sB)*n1m0), a2m1 = r1 * (n1m0 - sB * n1m1), a2m2 = r1 * (2.0 * n1m1 - sB * n1m2);
  c1 = c2;
  n1m0 = a1m0;
  n1m1 = a1m1;
  n1m2 = a1m2;
  c2 = (a2 - a0) * (a2 - a1);
  const double r2 = c1 / c2;
  const double c3a = a2 - a0, c3b = a2 - a1, tA2 = a2 - xt;
  m0[0] = (tA2 * n1m0) / c3a;
  m1[0] = (tA2 * n1m1 - n1m0) / c3a;
  m2[0] = (tA2 * n1m2 - 2.0 * n1m1) / c3a;
  m0[1] = (tA2 * a2m0) / c3b;
  m1[1] = (tA2 * a2m1 - a2m0) / c3b;
  m2[1] = (tA2 * a2m2 - 2.0 * a2m1) / c3b;
  const double sB2 = a1 - xt;
  m0[2] = r2 * (-(sB2)*a2m0);
  m1[2] = r2 * (a2m0 - sB2 * a2m1);
  m2[2] = r2 * (2.0 * a2m1 - sB2 * a2m2);
}

template <class U>
__device__ __forceinline__ U mol_dot3(const double* w, U a, U b, U c) {
  return (T)w[0] * a + (T)w[1] * b + (T)w[2] * c;
}

// Centred target (node 3 of the stencil: every node but the two next to a non-periodic end).
// Here the ideal weights d_k are positive on any nodes (the denominators of 1 - d_0 - d_2 add up
// to sums of products of spacings), so the split weights are 2 d_k and d_k, both normalised sets
// are equal and the derivative is the single sum  sum_k w_k r_k, w_k ~ d_k / (eps + beta_k)^2.
// The quadratic p_k has p_k'(x) = pM + (x - xM) pp, so Simpson's rule of the smoothness indicator
// is exact: beta_k = (dx pM)^2 + 13/12 (dx^2 pp)^2 and r_k = (g_k + gamma c_k) / dx with
// g_k = dx pM, c_k = sqrt(13/12) dx^2 pp, each a combination of two differences of u.
// MOL_NU3 coefficients: per k the factors of the differences in g_k and c_k, then gamma, 1/dx,
// d_0, d_1, d_2.
constexpr int MOL_NU3 = 17;
constexpr int MOL_NU_NC = 56;   // row stride of the axis tables

__device__ __forceinline__ void mol_weno5_nu3_coefs(const double* x, double* c) {
  const double xL = (x[1] + x[2]) / 2, xph = (x[2] + x[3]) / 2, dx = xph - xL, xM = (xL + xph) / 2;
  const double s = 1.0408329997330663;   // sqrt(13/12)
  for (int k = 0; k < 3; ++k) {
    double m0[3], m1[3], m2[3];
    mol_fornberg3(x[k], x[k + 1], x[k + 2], xM, m0, m1, m2);
    c[4 * k + 0] = -dx * m1[0];
    c[4 * k + 1] = dx * m1[2];
    c[4 * k + 2] = -s * dx * dx * m2[0];
    c[4 * k + 3] = s * dx * dx * m2[2];
  }
  c[12] = (x[2] - xM) / (dx * s);
  c[13] = 1.0 / dx;
  c[14] = ((x[2] - x[3]) * (x[2] - x[4])) / ((x[0] - x[3]) * (x[0] - x[4]));
  c[16] = ((x[2] - x[0]) * (x[2] - x[1])) / ((x[4] - x[0]) * (x[4] - x[1]));
  c[15] = 1.0 - c[14] - c[16];
}

// The derivative from the coefficients (C: a row, or a column of the tile's table in LDS).  The
// weights are cleared to products in FP64 and scaled by the smallest sum in FP32, as on uniform
// nodes: one quotient.  17 coefficients and 46 operations against 56 and about 140 of the split
// form: the FP64 Burgers right-hand side on 1024^2 stretched nodes 116 -> 9.7 us, with the
// coefficients along x read from the tile's columns in LDS and those along y by scalar loads.
template <class U, class C>
__device__ __forceinline__ U mol_weno5_nu3_t(U u1, U u2, U u3, U u4, U u5, const C& c, const T eps) {
  const U d[4] = {u2 - u1, u3 - u2, u4 - u3, u5 - u4};
  U e[3], r[3], w[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const U g = (T)c[4 * k] * d[k] + (T)c[4 * k + 1] * d[k + 1];
    const U h = (T)c[4 * k + 2] * d[k] + (T)c[4 * k + 3] * d[k + 1];
    e[k] = h * h + (g * g + eps);
    r[k] = g + (T)c[12] * h;
  }
  if constexpr (sizeof(T) == 8) {
    const U q0 = e[0] * e[0], q1 = e[1] * e[1], q2 = e[2] * e[2];
    w[0] = q1 * q2;
    w[1] = q0 * q2;
    w[2] = q0 * q1;
  } else {
    const T b = fmin(fmin(mol_val(e[0]), mol_val(e[1])), mol_val(e[2]));
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const U v = b * mol_rcp(e[k]);
      w[k] = v * v;
    }
  }
  w[0] = (T)c[14] * w[0];
  w[1] = (T)c[15] * w[1];
  w[2] = (T)c[16] * w[2];
  return (T)c[13] * mol_quot(w[0] * r[0] + (w[1] * r[1] + w[2] * r[2]), w[0] + (w[1] + w[2]));
}

template <class C>
__device__ __forceinline__ T mol_weno5_nu3(T u1, T u2, T u3, T u4, T u5, const C& c, T eps) {
  return mol_weno5_nu3_t<T>(u1, u2, u3, u4, u5, c, eps);
}

// The gradient with respect to the five values.
__device__ __noinline__ void mol_weno5_nu3_grad(T u1, T u2, T u3, T u4, T u5, const double* c, T eps, T* g) {
  const T x[5] = {u1, u2, u3, u4, u5};
  for (int k = 0; k < 5; ++k) {
    MolDual d[5];
    for (int j = 0; j < 5; ++j) d[j] = MolDual{x[j], j == k ? T(1) : T(0)};
    g[k] = mol_weno5_nu3_t<MolDual>(d[0], d[1], d[2], d[3], d[4], c, eps).d;
  }
}

// Column of the tile's table of centred-target coefficients along x (G::nux: MOL_NU3 rows of
// NUP = TX + 1 values, so that both the copy below and the nodes' reads are free of bank
// conflicts).  The 17 values of a node lie 448 bytes from its neighbour's in the axis table:
// read per lane they cost the L1 64 lines per load.
template <int NUP>
struct MolCol {
  const T* p;
  __device__ __forceinline__ T operator[](const int k) const { return p[k * NUP]; }
};
template <class G>
__device__ __forceinline__ void mol_stage_nux(const int o0, const JPtrs& jp) {
  if constexpr (G::NUP > 0)
    for (int e = (int)threadIdx.x; e < G::TX * MOL_NU3; e += G::NTHR) {
      const int x = e / MOL_NU3, k = e - x * MOL_NU3;
      G::nux()[k * G::NUP + x] = (T)jp.wtab[0][(i64)MOL_NU_NC * (min(o0 + x, (int)G::UHI0) - 1) + k];
    }
}

// One-sided targets (TG = 1, 2, 4, 5 of the stencil x1..x5).  The coordinate-only part of the
// derivative, MOL_NU_NC values: for each sub-stencil k = 0, 1, 2 the weights of r_k
// (derivative at the target) and of the interval values pL, pM, pR (first derivative at the left
// end, midpoint and right end) and pp (second derivative), 15 per sub-stencil; then dx/6, dx,
// dx^3 of the Simpson smoothness indicator, the split ideal weights dp_k/sgp and dm_k/sgm, and
// sgp, sgm.  mol_weno5_nu_apply turns them and the five values into the derivative.
__device__ __forceinline__ void mol_nu_sub(const double a0, const double a1, const double a2, const double xi,
                                           const double xL, const double xM, const double xph, double* c) {
  double m0[3], t2[3];
  mol_fornberg3(a0, a1, a2, xi, m0, c + 0, t2);
  mol_fornberg3(a0, a1, a2, xL, m0, c + 3, t2);
  mol_fornberg3(a0, a1, a2, xM, m0, c + 6, c + 12);
  mol_fornberg3(a0, a1, a2, xph, m0, c + 9, t2);
}

template <int TG>
__device__ __forceinline__ void mol_weno5_nu_coefs(const double x1, const double x2, const double x3, const double x4,
                                                   const double x5, double* c) {
  double xi, xL, xph, d0, d2;
  if (TG == 1) { xi = x1; xL = x1; xph = (x1 + x2) / 2; }
  else if (TG == 2) { xi = x2; xL = (x1 + x2) / 2; xph = (x2 + x3) / 2; }
  else if (TG == 4) { xi = x4; xL = (x3 + x4) / 2; xph = (x4 + x5) / 2; }
  else { xi = x5; xL = (x4 + x5) / 2; xph = x5; }
  if (TG == 1) {
    d0 = ((2 * x1 - x2 - x3) * (x1 - x4) * (x1 - x5) + (x1 - x3) * (x1 - x5) * (x1 - x2) +
          (x1 - x3) * (x1 - x4) * (x1 - x2)) / ((2 * x1 - x2 - x3) * (x1 - x4) * (x1 - x5));
    d2 = ((x1 - x3) * (x1 - x4) * (x1 - x2)) / ((-x1 + x5) * (2 * x1 - x3 - x4) * (-x2 + x5));
  } else if (TG == 2) {
    d0 = ((x2 - x4) * (x2 - x5)) / ((x1 - x4) * (x1 - x5));
    d2 = ((-x1 + x2) * (x2 - x3) * (x2 - x4)) / ((-x1 + x5) * (2 * x2 - x3 - x4) * (-x2 + x5));
  } else if (TG == 4) {
    d0 = ((-x2 + x4) * (-x3 + x4) * (x4 - x5)) / ((x1 - x4) * (x1 - x5) * (-x2 - x3 + 2 * x4));
    d2 = ((-x1 + x4) * (-x2 + x4)) / ((-x1 + x5) * (-x2 + x5));
  } else {
    d0 = ((-x2 + x5) * (-x3 + x5) * (-x4 + x5)) / ((x1 - x4) * (x1 - x5) * (-x2 - x3 + 2 * x5));
    d2 = ((-x1 - x4 + 2 * x5) * (-x2 + x5) * (-x3 + x5) + (-x1 + x5) * (-x2 - x3 + 2 * x5) * (-x4 + x5)) /
         ((-x1 + x5) * (-x2 + x5) * (-x3 - x4 + 2 * x5));
  }
  const double dx = xph - xL, xM = (xL + xph) / 2;
  mol_nu_sub(x1, x2, x3, xi, xL, xM, xph, c + 0);
  mol_nu_sub(x2, x3, x4, xi, xL, xM, xph, c + 15);
  mol_nu_sub(x3, x4, x5, xi, xL, xM, xph, c + 30);
  c[45] = dx / 6;
  c[46] = dx;
  c[47] = dx * dx * dx;
  const double d1 = 1.0 - d0 - d2, th = 3.0, half = 0.5;
  const double dp0 = half * (d0 + th * fabs(d0)), dp1 = half * (d1 + th * fabs(d1)), dp2 = half * (d2 + th * fabs(d2));
  const double dm0 = dp0 - d0, dm1 = dp1 - d1, dm2 = dp2 - d2;
  const double sgp = dp0 + dp1 + dp2, sgm = dm0 + dm1 + dm2;
  c[48] = dp0 / sgp;
  c[49] = dp1 / sgp;
  c[50] = dp2 / sgp;
  c[51] = dm0 / sgm;
  c[52] = dm1 / sgm;
  c[53] = dm2 / sgm;
  c[54] = sgp;
  c[55] = sgm;
}

template <class U>
__device__ __forceinline__ void mol_nu_beta_r(const double* c, const double* k, U ua, U ub, U uc, U& beta, U& r) {
  r = mol_dot3(c + 0, ua, ub, uc);
  const U pL = mol_dot3(c + 3, ua, ub, uc), pM = mol_dot3(c + 6, ua, ub, uc), pR = mol_dot3(c + 9, ua, ub, uc);
  const U pp = mol_dot3(c + 12, ua, ub, uc);
  const U I1 = (T)k[0] * (pL * pL + T(4) * (pM * pM) + pR * pR);
  const U I2 = (T)k[1] * (pp * pp);
  const U v = (T)k[1] * I1 + (T)k[2] * I2;
  beta = mol_val(v) > T(0) ? v : U{T(0)};
}

template <class U>
__device__ __forceinline__ U mol_weno5_nu_apply(U u1, U u2, U u3, U u4, U u5, const double* c, const T eps) {
  U b0, b1, b2, r0, r1, r2;
  mol_nu_beta_r(c + 0, c + 45, u1, u2, u3, b0, r0);
  mol_nu_beta_r(c + 15, c + 45, u2, u3, u4, b1, r1);
  mol_nu_beta_r(c + 30, c + 45, u3, u4, u5, b2, r2);
  const U e0 = eps + b0, e1 = eps + b1, e2 = eps + b2;
  const U q0 = e0 * e0, q1 = e1 * e1, q2 = e2 * e2;
  const U ap0 = (T)c[48] / q0, ap1 = (T)c[49] / q1, ap2 = (T)c[50] / q2;
  const U sp = ap0 + ap1 + ap2;
  const U am0 = (T)c[51] / q0, am1 = (T)c[52] / q1, am2 = (T)c[53] / q2;
  const U sm = am0 + am1 + am2;
  const U Rp = (ap0 / sp) * r0 + (ap1 / sp) * r1 + (ap2 / sp) * r2;
  const U Rm = (am0 / sm) * r0 + (am1 / sm) * r1 + (am2 / sm) * r2;
  return (T)c[54] * Rp - (T)c[55] * Rm;
}

// The FP64 derivative from the coefficients with the normalised nonlinear weights cleared, as
// in the uniform case: alpha_k / sum_j alpha_j = g_k P_k / sum_j g_j P_j with P_k the product of
// the other two q_j, so sgp Rp - sgm Rm = (sgp Np Dm - sgm Nm Dp) / (Dp Dm) costs one quotient
// (mol_quot) instead of twelve divisions.  The q_j are at least eps^2, so the products of four
// stay far above the FP64 underflow threshold (FP32 keeps the normalised form).
__device__ __forceinline__ double mol_weno5_nu_cleared(double u1, double u2, double u3, double u4, double u5,
                                                       const double* c, double eps) {
  double b0, b1, b2, r0, r1, r2;
  mol_nu_beta_r<double>(c + 0, c + 45, u1, u2, u3, b0, r0);
  mol_nu_beta_r<double>(c + 15, c + 45, u2, u3, u4, b1, r1);
  mol_nu_beta_r<double>(c + 30, c + 45, u3, u4, u5, b2, r2);
  const double e0 = eps + b0, e1 = eps + b1, e2 = eps + b2;
  const double q0 = e0 * e0, q1 = e1 * e1, q2 = e2 * e2;
  const double P0 = q1 * q2, P1 = q0 * q2, P2 = q0 * q1;
  const double A0 = c[48] * P0, A1 = c[49] * P1, A2 = c[50] * P2;
  const double B0 = c[51] * P0, B1 = c[52] * P1, B2 = c[53] * P2;
  const double Dp = A0 + A1 + A2, Dm = B0 + B1 + B2;
  const double Np = A0 * r0 + A1 * r1 + A2 * r2, Nm = B0 * r0 + B1 * r1 + B2 * r2;
  return mol_quot(c[54] * Np * Dm - c[55] * Nm * Dp, Dp * Dm);
}

// The same derivative from a node's row of precomputed coefficients (mol_weno_nu_table).
__device__ __forceinline__ T mol_weno5_nu_tab(T u1, T u2, T u3, T u4, T u5, const double* c, T eps) {
  if constexpr (sizeof(T) == 8) return (T)mol_weno5_nu_cleared(u1, u2, u3, u4, u5, c, eps);
  else return mol_weno5_nu_apply<T>(u1, u2, u3, u4, u5, c, eps);
}

// Distance of (unwrapped) node k of an axis from node i: past an end of a periodic axis the image's,
// continued by the period x[n] - x[1] (bcoord, src/discretization/interface_boundary.jl:120-151) and
// summed from differences on either side of the end.
__device__ __forceinline__ double mol_offset(const double* x, const int k, const int i, const int n) {
  if (k < 1) return (x[k + n - 2] - x[n - 1]) - (x[i - 1] - x[0]);
  if (k > n) return (x[n - 1] - x[i - 1]) + (x[k - n] - x[0]);
  return x[k - 1] - x[i - 1];
}

// The gradient from a node's row of precomputed coefficients.
__device__ __noinline__ void mol_weno5_nu_tab_grad(T u1, T u2, T u3, T u4, T u5, const double* c, T eps, T* g) {
  const T x[5] = {u1, u2, u3, u4, u5};
  for (int k = 0; k < 5; ++k) {
    MolDual d[5];
    for (int j = 0; j < 5; ++j) d[j] = MolDual{x[j], j == k ? T(1) : T(0)};
    g[k] = mol_weno5_nu_apply<MolDual>(d[0], d[1], d[2], d[3], d[4], c, eps).d;
  }
}

// Row of coefficients (MOL_NU3 or MOL_NU_NC values) of node i = 1..n of an axis with coordinates x: the
// stencil and target of the generated code (one-sided at nodes 1, 2, n-1, n of a non-periodic
// axis, centred elsewhere).  They depend on differences of coordinates only and are made from the
// stencil's distances to the node: half points of whole coordinates carry their rounding, eps / h of
// a spacing h (705 nodes, largest error of the derivative of random values 6.1e-11 -> 1e-12).
__device__ __forceinline__ void mol_weno_nu_row(const double* x, const int n, const bool periodic, const int i,
                                                double* c) {
  int first = -2, target = 3;
  if (!periodic) {
    if (i <= 2) {
      target = i;
      first = 1 - i;
    } else if (i >= n - 1) {
      target = 5 - (n - i);
      first = n - 4 - i;
    }
  }
  double xs[5];
  for (int q = 0; q < 5; ++q) {
    const int k = i + first + q;
    xs[q] = mol_offset(x, k, i, n);
  }
  switch (target) {
    case 1: mol_weno5_nu_coefs<1>(xs[0], xs[1], xs[2], xs[3], xs[4], c); break;
    case 2: mol_weno5_nu_coefs<2>(xs[0], xs[1], xs[2], xs[3], xs[4], c); break;
    case 4: mol_weno5_nu_coefs<4>(xs[0], xs[1], xs[2], xs[3], xs[4], c); break;
    case 5: mol_weno5_nu_coefs<5>(xs[0], xs[1], xs[2], xs[3], xs[4], c); break;
    default: mol_weno5_nu3_coefs(xs, c); break;
  }
}

// Hardware floating-point atomic add on global memory.
__device__ __forceinline__ void mol_atomic_add(T* p, T v) { unsafeAtomicAdd(p, v); }
__device__ __forceinline__ void mol_atomic_add_f64(double* p, double v) { unsafeAtomicAdd(p, v); }

// Work-groups are dealt to the 8 XCDs round-robin; remap so that each XCD runs one contiguous
// range of tiles (neighbouring tiles share halo lines in that XCD's L2).
template <int NBLK>
__device__ __forceinline__ int mol_xcd_tile(int b) {
  constexpr int NX = 8;
  if (NBLK < 2 * NX) return b;
  constexpr int q = NBLK / NX, rem = NBLK % NX;
  const int x = b % NX, i = b / NX;
  return x * q + (x < rem ? x : rem) + i;
}

// Coordinates (x, y, z) of position q of an EX x EY x ... box, advanced by a fixed stride
// without divisions (the staging loops visit q, q + S, q + 2S, ...).
template <int EX, int EY, int S>
struct MolWalk {
  int x, y, z;
  __device__ __forceinline__ explicit MolWalk(const int q) {
    z = q / (EX * EY);
    const int r = q - z * (EX * EY);
    y = r / EX;
    x = r - y * EX;
  }
  __device__ __forceinline__ void step() {
    constexpr int DZ = S / (EX * EY), R = S % (EX * EY), DY = R / EX, DX = R % EX;
    x += DX;
    y += DY;
    z += DZ;
    if (x >= EX) { x -= EX; ++y; }
    if (y >= EY) { y -= EY; ++z; }
  }
};

// Staging mode of a tile in variant G: 0 plain loads, 1 plain loads after the periodic wrap,
// 2 through the ghost-node closures (tile + halo leaves a variable's unknown box).
template <class G>
__device__ __forceinline__ int mol_stage_mode(const int tx, const int ty, const int tz) {
  if (tx >= G::FLO0 && tx <= G::FHI0 && ty >= G::FLO1 && ty <= G::FHI1 && tz >= G::FLO2 && tz <= G::FHI2) return 0;
  if (tx >= G::SLO0 && tx <= G::SHI0 && ty >= G::SLO1 && ty <= G::SHI1 && tz >= G::SLO2 && tz <= G::SHI2) return 1;
  return 2;
}

// Position (x, y, z) of the tile + halo box lies outside the tile along two or more axes and
// variant G reads no such position (G::CROSS): it is not staged.
template <class G>
__device__ __forceinline__ bool mol_unread(const int x, const int y, const int z) {
  if (!G::CROSS) return false;
  return (int)(x < G::HX || x >= G::HX + G::TX) + (int)(y < G::HY || y >= G::HY + G::TY) +
             (int)(z < G::HZ || z >= G::HZ + G::TZ) >= 2;
}

// Tile + halo of the staged arrays into LDS.
template <class G>
__device__ __forceinline__ void mol_stage_tile(T* L, const int o0, const int o1, const int o2, const int mode,
                                               const double t, const T* __restrict__ P, const T* __restrict__ u,
                                               const JPtrs& jp) {
  constexpr int IT = (G::VOL + G::NTHR - 1) / G::NTHR;   // positions per thread
  MolWalk<G::EX, G::EY, G::NTHR> w((int)threadIdx.x);
  if constexpr (G::NST > 0 && IT * G::NST <= 16) {
    // every load of the thread is issued before its first LDS store: one exposed memory
    // latency per tile instead of one per position
    T v[IT][G::NST];
    bool ok[IT];
#pragma unroll
    for (int k = 0; k < IT; ++k, w.step()) {
      const int q = (int)threadIdx.x + k * G::NTHR;
      ok[k] = (G::VOL % G::NTHR == 0 || q < G::VOL) && !mol_unread<G>(w.x, w.y, w.z);
      if (ok[k]) G::stage_vals(v[k], o0 + w.x - G::HX, o1 + w.y - G::HY, o2 + w.z - G::HZ, mode, t, P, u, jp);
    }
#pragma unroll
    for (int k = 0; k < IT; ++k) {
      const int q = (int)threadIdx.x + k * G::NTHR;
      if (ok[k])
#pragma unroll
        for (int s = 0; s < G::NST; ++s) L[s * G::VOL + q] = v[k][s];
    }
  } else {
    for (int q = threadIdx.x; q < G::VOL; q += G::NTHR, w.step())
      if (!mol_unread<G>(w.x, w.y, w.z))
        G::stage_pos(L, q, o0 + w.x - G::HX, o1 + w.y - G::HY, o2 + w.z - G::HZ, mode, t, P, u, jp);
  }
}

// The value of the wave's first lane in every lane (v is the same in all of them): index
// arithmetic and table reads along rows become scalar.
__device__ __forceinline__ int mol_uniform(const int v) {
#ifdef __AMDGCN__
  return __builtin_amdgcn_readfirstlane(v);
#else
  return v;
#endif
}

// Node phase of one staged tile in variant G: each thread runs G::RB consecutive nodes along
// axis G::BA; their node functions see the same LDS tile at offsets that differ by a constant,
// so shared taps and subexpressions are loaded and computed once.  Nodes of a ragged tile past
// the unknown box run at the last node of the box (every load stays inside the tile + halo
// and the arrays) and store nothing.
template <class G>
__device__ __forceinline__ void mol_tile_nodes(const T* L, const int tx, const int ty, const int tz,
                                               const T* __restrict__ u, const Epi& ep, const JPtrs& jp,
                                               const double t) {
  const int o0 = G::ULO0 + tx * G::TX, o1 = G::ULO1 + ty * G::TY, o2 = G::ULO2 + tz * G::TZ;
  constexpr int RB = G::RB;
  constexpr int PX = G::TX, PY = G::BA == 1 ? G::TY / RB : G::TY, PZ = G::BA == 2 ? G::TZ / RB : G::TZ;
  constexpr int PXY = PX * PY, PV = PXY * PZ;
  constexpr int STEP = G::BA == 1 ? G::EX : (G::BA == 2 ? G::EX * G::EY : 1);
#pragma unroll
  for (int r = 0; r < (PV + G::NTHR - 1) / G::NTHR; ++r) {
    const int q = (int)threadIdx.x + r * G::NTHR;
    if (PV % G::NTHR != 0 && q >= PV) break;
    int lz0 = q / PXY;
    const int rr = q - lz0 * PXY;
    int ly0 = rr / PX;
    const int lx = rr - ly0 * PX;
    if constexpr (PX % 64 == 0 && G::NUP > 0) {   // a wave's nodes lie in one row: scalar table reads
      ly0 = mol_uniform(ly0);
      lz0 = mol_uniform(lz0);
    }
    const int ly = G::BA == 1 ? ly0 * RB : ly0, lz = G::BA == 2 ? lz0 * RB : lz0;
    const int base = (lx + G::HX) + G::EX * (ly + G::HY) + G::EX * G::EY * (lz + G::HZ);
    T out[RB][G::NF];
    int J[RB][3];
#pragma unroll
    for (int k = 0; k < RB; ++k) {
      J[k][0] = o0 + lx;
      J[k][1] = o1 + ly + (G::BA == 1 ? k : 0);
      J[k][2] = o2 + lz + (G::BA == 2 ? k : 0);
      G::node(L, base + k * STEP, min(J[k][0], (int)G::UHI0), min(J[k][1], (int)G::UHI1), min(J[k][2], (int)G::UHI2), t,
              ep.p, u, jp, out[k]);
    }
#pragma unroll
    for (int k = 0; k < RB; ++k) {
      if (J[k][0] > G::UHI0 || J[k][1] > G::UHI1 || J[k][2] > G::UHI2) continue;
#pragma unroll
      for (int f = 0; f < G::NF; ++f)
        if (G::inbox(f, J[k][0], J[k][1], J[k][2])) mol_epilogue(ep, G::uidx(f, J[k][0], J[k][1], J[k][2]), out[k][f]);
    }
  }
}

// Loads of the tile + halo of variant G into registers R[i][slot] (position threadIdx.x + i *
// NTHR): issued for the next tile while the current one runs its node phase.
template <class G, int NPF, int NSR>
__device__ __forceinline__ void mol_fetch(T (&R)[NPF][NSR], const int tx, const int ty, const int tz, const double t,
                                          const T* __restrict__ P, const T* __restrict__ u, const JPtrs& jp) {
  const int o0 = G::ULO0 + tx * G::TX, o1 = G::ULO1 + ty * G::TY, o2 = G::ULO2 + tz * G::TZ;
  const int mode = mol_stage_mode<G>(tx, ty, tz);
  MolWalk<G::EX, G::EY, G::NTHR> w((int)threadIdx.x);
#pragma unroll
  for (int i = 0; i < NPF; ++i) {
    if (i * G::NTHR >= G::VOL) break;
    if ((int)threadIdx.x + i * G::NTHR < G::VOL) {
      if (mol_unread<G>(w.x, w.y, w.z)) {
#pragma unroll
        for (int s = 0; s < NSR; ++s) R[i][s] = T(0);
      } else {
        G::stage_vals(R[i], o0 + w.x - G::HX, o1 + w.y - G::HY, o2 + w.z - G::HZ, mode, t, P, u, jp);
      }
    }
    w.step();
  }
}

template <class G, int NPF, int NSR>
__device__ __forceinline__ void mol_put(T* L, const T (&R)[NPF][NSR]) {
#pragma unroll
  for (int i = 0; i < NPF; ++i) {
    const int q = (int)threadIdx.x + i * G::NTHR;
    if (i * G::NTHR >= G::VOL) break;
    if (q < G::VOL)
#pragma unroll
      for (int s = 0; s < G::NST; ++s) L[s * G::VOL + q] = R[i][s];
  }
}

// One tile of the union unknown box, in the tile variant G (interior-rows core variant or the
// boundary variant, each with its own halo): stage (mol_stage_tile), then the node phase.
template <class G>
__device__ __forceinline__ void mol_full_tile(T* L, const int tx, const int ty, const int tz, const T* __restrict__ u,
                                              const Epi& ep, const JPtrs& jp, const double t) {
  if (G::NST > 0) {
    const int o0 = G::ULO0 + tx * G::TX, o1 = G::ULO1 + ty * G::TY, o2 = G::ULO2 + tz * G::TZ;
    mol_stage_tile<G>(L, o0, o1, o2, mol_stage_mode<G>(tx, ty, tz), t, ep.p, u, jp);
    mol_stage_nux<G>(o0, jp);
    __syncthreads();
  }
  mol_tile_nodes<G>(L, tx, ty, tz, u, ep, jp, t);
}

// Persistent loop over the tiles of a launch of gridDim.x work-groups (a multiple of 8 when
// smaller than the tile count, so that tile k + gridDim.x stays on the XCD of tile k): the
// staging loads of the next tile are in flight while the current tile runs its node phase.
// GC: interior-rows variant (used when HASC and the tile is a core tile), GB: boundary variant;
// both stage the same arrays.
template <class GC, class GB, bool HASC, int NPF>
__device__ __forceinline__ void mol_tiles_persistent(T* L, const T* __restrict__ u, const Epi& ep, const JPtrs& jp,
                                                     const double t) {
  constexpr int NSR = GB::NST > 0 ? GB::NST : 1;
  constexpr int NBLK = GB::NBLK;
  int k = (int)blockIdx.x;
  if (k >= NBLK) return;
  auto decode = [](const int lin, int& x, int& y, int& z) {
    int b = mol_xcd_tile<NBLK>(lin);
    x = b % GB::NT0;
    b /= GB::NT0;
    y = b % GB::NT1;
    z = b / GB::NT1;
  };
  // more than 16 staging values per thread would cost occupancy: stage each tile in turn
  if (NPF * NSR > 16) {
    for (; k < NBLK; k += (int)gridDim.x) {
      int tx, ty, tz;
      decode(k, tx, ty, tz);
      if (HASC && GB::is_core(tx, ty, tz)) mol_full_tile<GC>(L, tx, ty, tz, u, ep, jp, t);
      else mol_full_tile<GB>(L, tx, ty, tz, u, ep, jp, t);
      if (GB::NST > 0 && k + (int)gridDim.x < NBLK) __syncthreads();
    }
    return;
  }
  T R[NPF][NSR];
  int tx, ty, tz;
  decode(k, tx, ty, tz);
  bool core = HASC && GB::is_core(tx, ty, tz);
  if (GB::NST > 0) {
    if (HASC && core) mol_fetch<GC, NPF, NSR>(R, tx, ty, tz, t, ep.p, u, jp);
    else mol_fetch<GB, NPF, NSR>(R, tx, ty, tz, t, ep.p, u, jp);
  }
  while (true) {
    if (GB::NST > 0) {
      if (HASC && core) mol_put<GC, NPF, NSR>(L, R);
      else mol_put<GB, NPF, NSR>(L, R);
      mol_stage_nux<GB>(GB::ULO0 + tx * GB::TX, jp);
      __syncthreads();
    }
    const int kn = k + (int)gridDim.x;
    int nx = 0, ny = 0, nz = 0;
    bool ncore = false;
    if (kn < NBLK) {
      decode(kn, nx, ny, nz);
      ncore = HASC && GB::is_core(nx, ny, nz);
      if (GB::NST > 0) {
        if (HASC && ncore) mol_fetch<GC, NPF, NSR>(R, nx, ny, nz, t, ep.p, u, jp);
        else mol_fetch<GB, NPF, NSR>(R, nx, ny, nz, t, ep.p, u, jp);
      }
    }
    if (HASC && core) mol_tile_nodes<GC>(L, tx, ty, tz, u, ep, jp, t);
    else mol_tile_nodes<GB>(L, tx, ty, tz, u, ep, jp, t);
    if (kn >= NBLK) break;
    if (GB::NST > 0) __syncthreads();
    k = kn;
    tx = nx;
    ty = ny;
    tz = nz;
    core = ncore;
  }
}

// ---------------------------------------------------------------------------------------
// Fused classic RK4 step: stage S of tile (o0, o1, o2) on the tile grown by (4 - S) reach per
// axis.  The items of a stage are the tile's nodes (0 .. TVOL-1) and then the frame of the
// grown region; item q belongs to thread q mod NTHR, so every tile node keeps its thread across
// the four stages and its step-initial value Ur and running sum Ar = k1 + 2 k2 + 2 k3 stay in
// that thread's registers.  Lin holds the stage input (u, y1, y2, y3), Lout receives
// y_S = u + c_S dt k_S; stage 4 writes u + dt/6 k4 + dt/6 Ar.  The arithmetic is that of the
// stage kernels' epilogue (mode 1 with ca = 1, acc_f = 1 or 2, acc_keep = 0 or 1), so a fused
// step equals four stage launches.
template <class G>
struct MolFusedItems {
  static constexpr int TVOL = G::TX * G::TY * G::TZ;
  static constexpr int NJ = (TVOL + G::NTHR - 1) / G::NTHR;   // tile nodes per thread, NTHR apart
  static __device__ __forceinline__ void pos(const int j, int& lx, int& ly) {
    const int q = (int)threadIdx.x + j * G::NTHR;
    ly = q / G::TX;
    lx = q - ly * G::TX;
  }
  static __device__ __forceinline__ bool valid(const int j) {
    return TVOL % G::NTHR == 0 || (int)threadIdx.x + j * G::NTHR < TVOL;
  }
};

// Frame items of the region grown by M: the square (tile + M reach per axis) less the tile,
// or, for 2D cross-shaped stencils of reach one on periodic axes (G::DIAM), the positions
// within M steps of the tile along the axes (L1 distance), which are all that the remaining
// stages read: 2 M (TX + TY) + 2 M (M - 1) items instead of 2 M (TX + TY) + 4 M^2.
template <class G, int M>
struct MolFrame2 {
  static constexpr int N = G::DIAM ? 2 * M * (G::TX + G::TY) + 2 * M * (M - 1)
                                   : (G::TX + 2 * M * G::RX) * (G::TY + 2 * M * G::RY) - G::TX * G::TY;
};

// Position (tile-relative) of frame item h of the region grown by M (2D / 1D: RZ = 0).
template <class G, int M>
__device__ __forceinline__ void mol_frame_pos(const int h, int& lx, int& ly) {
  if constexpr (G::DIAM) {
    // rows above the tile from the outermost (ly = -M, TX wide) inwards (ly = -d spans
    // TX + 2 (M - d) positions centred on the tile), the same rows below, then M positions on
    // either side of each tile row
    constexpr int TOP = M * G::TX + M * (M - 1);
    if (h < 2 * TOP) {
      const bool below = h >= TOP;
      int r = below ? h - TOP : h;
      int d = M;
#pragma unroll
      for (int k = M; k > 1; --k) {
        const int w = G::TX + 2 * (M - k);
        if (d == k && r >= w) {
          r -= w;
          d = k - 1;
        }
      }
      ly = below ? G::TY - 1 + d : -d;
      lx = -(M - d) + r;
    } else {
      const int h3 = h - 2 * TOP;
      const int c = h3 % (2 * M);
      ly = h3 / (2 * M);
      lx = c < M ? -M + c : G::TX + (c - M);
    }
    return;
  }
  constexpr int MR0 = M * G::RX, MR1 = M * G::RY, W0 = G::TX + 2 * MR0;
  if (h < MR1 * W0) {
    ly = -MR1 + h / W0;
    lx = -MR0 + h % W0;
  } else if (h < 2 * MR1 * W0) {
    const int h2 = h - MR1 * W0;
    ly = G::TY + h2 / W0;
    lx = -MR0 + h2 % W0;
  } else {
    const int h3 = h - 2 * MR1 * W0;
    const int c = h3 % (2 * MR0);
    ly = h3 / (2 * MR0);
    lx = c < MR0 ? -MR0 + c : G::TX + (c - MR0);
  }
}

// Node-invariant values of the tile nodes (G::NINV per node: what depends only on constants,
// parameters and coordinates), computed once per launch and read by G::node_h in every stage.
template <class G>
struct MolFusedInv {
  static constexpr int NI = G::NINV > 0 ? G::NINV : 1;
  T v[MolFusedItems<G>::NJ][NI];
  __device__ __forceinline__ void init(const int o0, const int o1, const int o2, const T* __restrict__ P,
                                       const JPtrs& jp) {
    if constexpr (G::NINV > 0) {
#pragma unroll
      for (int j = 0; j < MolFusedItems<G>::NJ; ++j) {
        int lx, ly;
        MolFusedItems<G>::pos(j, lx, ly);
        if (MolFusedItems<G>::valid(j)) G::node_inv(o0 + lx, o1 + ly, o2, P, jp, v[j]);
      }
    }
  }
};

template <class G, int S, int M = 4 - S, int ME = 0>
__device__ __forceinline__ void mol_rk4_stage(const T* Lin, T* Lout, T* U, T (&Ur)[MolFusedItems<G>::NJ][G::NF],
                                              T (&Ar)[MolFusedItems<G>::NJ][G::NF], const MolFusedInv<G>& Iv,
                                              const int o0, const int o1,
                                              const int o2, const T* __restrict__ u, T* __restrict__ unew,
                                              const Epi& ep, const JPtrs& jp, const double t, const double dt,
                                              T* Ac) {
  // M: the stage region is the tile grown by M reach per axis.  ME: the step's result is
  // wanted on the tile grown by ME (ME > 0: the first of two steps in one launch, whose result
  // is the next step's tile + halo); the frame positions inside it keep their running sum in
  // Ac, and stage 4 (M == ME) leaves the new state in U, in place, at every position of its
  // region and in Ur for the tile nodes.
  static_assert(S < 4 ? M == ME + 4 - S : M == ME, "stage regions shrink by one reach per stage");
  constexpr int TVOL = MolFusedItems<G>::TVOL, NJ = MolFusedItems<G>::NJ;
  constexpr int FR = MolFrame2<G, M>::N;
  static_assert(G::TZ == 1 && G::RZ == 0, "fused RK4 steps are 1D / 2D");
  static_assert(!G::DIAM || (G::RX == 1 && G::RY == 1 && !G::FIX), "L1 stage regions: reach one, periodic");
  const double ts = t + (S == 1 ? 0.0 : (S == 4 ? dt : dt / 2));
  const double cf = S == 1 || S == 2 ? dt / 2 : (S == 3 ? dt : dt / 6);
  // tile nodes: registers carry u and the running sum
  T out[NJ][G::NF];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    if (!MolFusedItems<G>::valid(j)) break;
    int lx, ly;
    MolFusedItems<G>::pos(j, lx, ly);
    if constexpr (G::NINV > 0)
      G::node_h(Lin, (lx + G::HX) + G::EX * (ly + G::HY), o0 + lx, o1 + ly, o2, ts, ep.p, u, jp, Iv.v[j], out[j]);
    else
      G::node(Lin, (lx + G::HX) + G::EX * (ly + G::HY), o0 + lx, o1 + ly, o2, ts, ep.p, u, jp, out[j]);
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    if (!MolFusedItems<G>::valid(j)) break;
    int lx, ly;
    MolFusedItems<G>::pos(j, lx, ly);
    const int b = (lx + G::HX) + G::EX * (ly + G::HY);
    const int I0 = o0 + lx, I1 = o1 + ly, I2 = o2;
#pragma unroll
    for (int f = 0; f < G::NF; ++f) {
      T v = (T)cf * out[j][f];
      v += Ur[j][f];
      if (S < 4) {
        Lout[f * G::VOL + b] = v;
        T a = (S == 1 ? T(1) : T(2)) * out[j][f];
        if (S > 1) a += Ar[j][f];
        Ar[j][f] = a;
      } else {
        v += (T)cf * Ar[j][f];
        if (ME == 0 && I0 <= G::UHI0 && I1 <= G::UHI1 && I2 <= G::UHI2) unew[G::uidx(f, I0, I1, I2)] = v;
        if (ME > 0) {
          U[f * G::VOL + b] = v;
          Ur[j][f] = v;
          Ar[j][f] = T(0);
        }
      }
    }
  }
  // frame of the grown region: u from LDS, and inside the step's result region the running
  // sum from Ac
  if (M > 0) {
    for (int q = (int)threadIdx.x; q < TVOL + FR; q += G::NTHR) {
      if (q < TVOL) continue;
      int lx, ly;
      mol_frame_pos<G, M>(q - TVOL, lx, ly);
      const int b = (lx + G::HX) + G::EX * (ly + G::HY);
      T out[G::NF];
      G::node(Lin, b, o0 + lx, o1 + ly, o2, ts, ep.p, u, jp, out);
      const bool keep = ME > 0 && lx >= -ME * G::RX && lx < G::TX + ME * G::RX && ly >= -ME * G::RY &&
                        ly < G::TY + ME * G::RY;
#pragma unroll
      for (int f = 0; f < G::NF; ++f) {
        T v = (T)cf * out[f];
        v += U[f * G::VOL + b];
        if (S < 4) {
          Lout[f * G::VOL + b] = v;
          if (keep) {
            T a = (S == 1 ? T(1) : T(2)) * out[f];
            if (S > 1) a += Ac[f * G::VOL + b];
            Ac[f * G::VOL + b] = a;
          }
        } else {
          v += (T)cf * Ac[f * G::VOL + b];
          U[f * G::VOL + b] = v;
        }
      }
    }
  }
}

// After a stage of a fused step on a non-periodic system: the positions of the stage region
// (tile + M reach) outside the unknown box along a non-periodic axis get the value of their
// boundary equations from the stage values just written, at the next stage's time (what
// staging does for each stage launch of the unfused path).  Returns whether it wrote.
template <class G, int M>
__device__ __forceinline__ bool mol_rk4_fix_ghosts(T* L, const int o0, const int o1, const int o2, const double tn,
                                                   const T* __restrict__ P, const JPtrs& jp) {
  constexpr int W0 = G::TX + 2 * M * G::RX, W1 = G::TY + 2 * M * G::RY, W2 = G::TZ + 2 * M * G::RZ;
  constexpr int NV = W0 * W1 * W2;
  // the whole work-group takes the same branch: the region reaches outside the box or not
  const bool out0 = !G::PER0 && (o0 - M * G::RX < (int)G::ULO0 || o0 + G::TX - 1 + M * G::RX > (int)G::UHI0);
  const bool out1 = !G::PER1 && G::RY > 0 && (o1 - M * G::RY < (int)G::ULO1 || o1 + G::TY - 1 + M * G::RY > (int)G::UHI1);
  if (!out0 && !out1) return false;
  for (int q = threadIdx.x; q < NV; q += G::NTHR) {
    const int z = q / (W0 * W1);
    const int r = q - z * (W0 * W1);
    const int y = r / W0;
    const int x = r - y * W0;
    const int lx = x - M * G::RX, ly = y - M * G::RY, lz = z - M * G::RZ;
    const int p0 = o0 + lx, p1 = o1 + ly, p2 = o2 + lz;
    const bool ghost = (!G::PER0 && (p0 < (int)G::ULO0 || p0 > (int)G::UHI0)) ||
                       (!G::PER1 && G::RY > 0 && (p1 < (int)G::ULO1 || p1 > (int)G::UHI1));
    if (!ghost) continue;
    const int b = (lx + G::HX) + G::EX * ((ly + G::HY) + G::EY * (lz + G::HZ));
    T v[G::NF];
#pragma unroll
    for (int f = 0; f < G::NF; ++f) v[f] = G::stage_lds(f, p0, p1, p2, tn, P, L, o0 - G::HX, o1 - G::HY, o2 - G::HZ, jp);
#pragma unroll
    for (int f = 0; f < G::NF; ++f) L[f * G::VOL + b] = v[f];
  }
  return true;
}

// One RK4 step of a fused launch from U (tile + halo) at time t: stage regions of margin
// ME + 3 .. ME; ME = 4: the first of two steps, whose result (tile + 4 reach) stays in U with its
// ghosts refilled at t + dt; ME = 0: the last step, stored to unew.
template <class G, int ME>
__device__ __forceinline__ void mol_rk4_step(T* U, T* Ya, T* Yb, T* Ac, T (&Ur)[MolFusedItems<G>::NJ][G::NF],
                                             T (&Ar)[MolFusedItems<G>::NJ][G::NF], const MolFusedInv<G>& Iv,
                                             const int o0, const int o1, const int o2, const T* __restrict__ u,
                                             T* __restrict__ unew, const Epi& ep, const JPtrs& jp, const double t,
                                             const double dt) {
  mol_rk4_stage<G, 1, ME + 3, ME>(U, Ya, U, Ur, Ar, Iv, o0, o1, o2, u, unew, ep, jp, t, dt, Ac);
  __syncthreads();
  if constexpr (G::FIX) {
    if (mol_rk4_fix_ghosts<G, ME + 3>(Ya, o0, o1, o2, t + dt / 2, ep.p, jp)) __syncthreads();
  }
  mol_rk4_stage<G, 2, ME + 2, ME>(Ya, Yb, U, Ur, Ar, Iv, o0, o1, o2, u, unew, ep, jp, t, dt, Ac);
  __syncthreads();
  if constexpr (G::FIX) {
    if (mol_rk4_fix_ghosts<G, ME + 2>(Yb, o0, o1, o2, t + dt / 2, ep.p, jp)) __syncthreads();
  }
  mol_rk4_stage<G, 3, ME + 1, ME>(Yb, Ya, U, Ur, Ar, Iv, o0, o1, o2, u, unew, ep, jp, t, dt, Ac);
  __syncthreads();
  if constexpr (G::FIX) {
    if (mol_rk4_fix_ghosts<G, ME + 1>(Ya, o0, o1, o2, t + dt, ep.p, jp)) __syncthreads();
  }
  mol_rk4_stage<G, 4, ME, ME>(Ya, nullptr, U, Ur, Ar, Iv, o0, o1, o2, u, unew, ep, jp, t, dt, Ac);
  if constexpr (ME > 0) {
    __syncthreads();
    if constexpr (G::FIX) {
      if (mol_rk4_fix_ghosts<G, ME>(U, o0, o1, o2, t + dt, ep.p, jp)) __syncthreads();
    }
  }
}

// A fused launch of nsteps (1, or 2 when the halo is 8 reach wide) RK4 steps on one tile.  The
// second step starts at t + dt, the device clock's next value.
template <class G>
__device__ __forceinline__ void mol_rk4_fused_tile(T* U, T* Ya, T* Yb, T* Ac, double* fc, const int fcs, int* fo,
                                                   const int tx, const int ty, const int tz, const T* __restrict__ u,
                                                   T* __restrict__ unew, const Epi& ep, const JPtrs& jp,
                                                   const double t, const int nsteps) {
  const int o0 = G::ULO0 + tx * G::TX, o1 = G::ULO1 + ty * G::TY, o2 = G::ULO2 + tz * G::TZ;
  const double dt = ep.tadv;
  // coordinates of the tile + halo positions (periodic images wrapped), per axis: position c of
  // the concatenated extents EX, EY, EZ; loaded before the staging loads are awaited, so both
  // are in flight together
  constexpr int NCP = G::EX + G::EY + G::EZ, NCI = (NCP + G::NTHR - 1) / G::NTHR;
  double cv[NCI];
  int cdst[NCI];
#pragma unroll
  for (int k = 0; k < NCI; ++k) {
    const int c = (int)threadIdx.x + k * G::NTHR;
    const int a = c < G::EX ? 0 : (c < G::EX + G::EY ? 1 : 2);
    const int e = c - (a == 0 ? 0 : (a == 1 ? G::EX : G::EX + G::EY));
    const int org = a == 0 ? o0 - G::HX : (a == 1 ? o1 - G::HY : o2 - G::HZ);
    const int nn = a == 0 ? G::N0 : (a == 1 ? G::N1 : G::N2);
    const bool per = a == 0 ? G::PER0 != 0 : (a == 1 ? G::PER1 != 0 : G::PER2 != 0);
    cdst[k] = -1;
    cv[k] = 0.0;
    if (c < NCP && jp.coord[a]) {
      int p = org + e;
      if (per) p = mol_wrap(mol_wrap(p, nn), nn);
      cv[k] = jp.coord[a][min(max(p, 1), nn) - 1];
      cdst[k] = a * fcs + e;
    }
  }
  for (int a = (int)threadIdx.x; a < 3; a += G::NTHR) fo[a] = a == 0 ? o0 - G::HX : (a == 1 ? o1 - G::HY : o2 - G::HZ);
  mol_stage_tile<G>(U, o0, o1, o2, mol_stage_mode<G>(tx, ty, tz), t, ep.p, u, jp);
#pragma unroll
  for (int k = 0; k < NCI; ++k)
    if (cdst[k] >= 0) fc[cdst[k]] = cv[k];
  __syncthreads();
  constexpr int NJ = MolFusedItems<G>::NJ;
  T Ur[NJ][G::NF], Ar[NJ][G::NF];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    int lx, ly;
    MolFusedItems<G>::pos(j, lx, ly);
    const bool ok = MolFusedItems<G>::valid(j);
    const int b = ok ? (lx + G::HX) + G::EX * (ly + G::HY) : 0;
#pragma unroll
    for (int f = 0; f < G::NF; ++f) {
      Ur[j][f] = ok ? U[f * G::VOL + b] : T(0);
      Ar[j][f] = T(0);
    }
  }
  MolFusedInv<G> Iv;
  Iv.init(o0, o1, o2, ep.p, jp);
  if constexpr (G::HX >= 8 * G::RX && G::HY >= 8 * G::RY) {
    if (nsteps == 2) {
      mol_rk4_step<G, 4>(U, Ya, Yb, Ac, Ur, Ar, Iv, o0, o1, o2, u, unew, ep, jp, t, dt);
      mol_rk4_step<G, 0>(U, Ya, Yb, Ac, Ur, Ar, Iv, o0, o1, o2, u, unew, ep, jp, t + dt, dt);
      return;
    }
  }
  mol_rk4_step<G, 0>(U, Ya, Yb, Ac, Ur, Ar, Iv, o0, o1, o2, u, unew, ep, jp, t, dt);
}

// Value of the neighbouring lane (lane - 1, lane + 1) of the wave, 0 past its ends: DPP wave
// shifts, no LDS access.  mol_lane(x, l): lane l's value in every lane (l: the same in every
// lane).  Off the GPU a wave is one lane.
#ifdef __AMDGCN__
constexpr int MOL_WAVE = 64;
template <int CTRL, class U>
__device__ __forceinline__ U mol_dpp(const U x) {
  constexpr int N = sizeof(U) / 4;
  int w[N];
  __builtin_memcpy(w, &x, sizeof(U));
#pragma unroll
  for (int k = 0; k < N; ++k) w[k] = __builtin_amdgcn_update_dpp(0, w[k], CTRL, 0xf, 0xf, true);
  U r;
  __builtin_memcpy(&r, w, sizeof(U));
  return r;
}
template <class U>
__device__ __forceinline__ U mol_lane_below(const U x) { return mol_dpp<0x138>(x); }   // wave_shr:1
template <class U>
__device__ __forceinline__ U mol_lane_above(const U x) { return mol_dpp<0x130>(x); }   // wave_shl:1
template <class U>
__device__ __forceinline__ U mol_lane(const U x, const int l) {
  constexpr int N = sizeof(U) / 4;
  int w[N];
  __builtin_memcpy(w, &x, sizeof(U));
#pragma unroll
  for (int k = 0; k < N; ++k) w[k] = __builtin_amdgcn_readlane(w[k], l);
  U r;
  __builtin_memcpy(&r, w, sizeof(U));
  return r;
}
#else
constexpr int MOL_WAVE = 1;
template <class U>
inline U mol_lane_below(const U) { return U(0); }
template <class U>
inline U mol_lane_above(const U) { return U(0); }
template <class U>
inline U mol_lane(const U x, const int) { return x; }
#endif

// Resident steps of a 1D system held by a single work-group, the state in registers.  A lane
// holds NJ consecutive nodes; the taps of its end nodes come from the neighbouring lanes by DPP,
// so a stage has no LDS access and no barrier.  One wave holds a non-periodic system whole.
// Otherwise (several waves, or a periodic ring) a wave holds S nodes and, evaluated redundantly,
// the HL = 4 reach nodes past either end: a whole step needs no other wave, and the end nodes
// are exchanged once per step through LDS (two buffers in turn, one barrier).
// What bounds it is the serial chain of a stage (the 101-node FP64 heat equation: 71 VALU instructions
// and 341 cycles per step, 0.142 us, against 0.88 us for the stages on an LDS tile with two
// barriers each).
template <class G>
struct MolRing {
  static constexpr int LN = G::NTHR < MOL_WAVE ? G::NTHR : MOL_WAVE;   // lanes per wave
  static constexpr int W = G::NTHR / LN;                               // waves
  static constexpr int R = G::RX, TN = G::TX;                          // reach, nodes
  static constexpr bool PER = G::PER0 != 0, ONE = W == 1 && !PER;
  static constexpr int HL = ONE ? 0 : 4 * R;
  static constexpr int S = (TN + W - 1) / W;                           // nodes of a wave
  static constexpr int NJ0 = (S + 2 * HL + LN - 1) / LN, NJ = NJ0 > R ? NJ0 : (R > 0 ? R : 1);
  static constexpr int SL = TN - (W - 1) * S;                          // nodes of the last wave
  static constexpr int XN = ONE ? 1 : 2 * G::NF * TN;                  // exchange buffers (values)
  // the ghosts of an end are needed by the wave that holds it only: the waves next to it do not
  // reach past its own nodes
  static_assert(W == 1 || (S >= HL + G::KMAX && SL >= HL + G::KMAX), "a wave holds too few nodes");
  static_assert(NJ + 2 * R <= G::VOL, "register window larger than the printed geometry");
};

template <class G>
__device__ __forceinline__ void mol_rk4_ring(T* X, double* fc, int* fo, const T* u, T* unew, const Epi& ep,
                                             const JPtrs& jp, const double t0, const int nsub) {
  // u and unew may be the same array
  using Q = MolRing<G>;
  static_assert(G::NBLK == 1 && G::RY == 0 && G::TY == 1 && (Q::PER || G::RX <= 1), "resident steps: one 1D tile");
  constexpr int R = Q::R, NJ = Q::NJ, NF = G::NF, NI = G::NINV > 0 ? G::NINV : 1;
  const int o0 = G::ULO0, o1 = G::ULO1, o2 = G::ULO2;
  const double dt = ep.tadv;
  // coordinates of the tile + halo (periodic images wrapped)
  if (threadIdx.x == 0) fo[0] = o0 - G::HX;
  if (jp.coord[0])
    for (int e = (int)threadIdx.x; e < G::EX; e += G::NTHR) {
      int p = o0 - G::HX + e;
      if (Q::PER) p = mol_wrap(mol_wrap(p, G::N0), G::N0);
      fc[e] = jp.coord[0][min(max(p, 1), (int)G::N0) - 1];
    }
  __syncthreads();
  const int wv = (int)threadIdx.x / Q::LN, lane = (int)threadIdx.x % Q::LN;
  const int i0 = wv * Q::S - Q::HL + lane * NJ;   // node (from 0) of the lane's first slot
  // node held by slot j: its image on a periodic axis, the end node past a non-periodic end
  // (such slots are evaluated, their values never reach a node)
  auto at = [&](const int j) {
    int i = i0 + j;
    if (Q::PER) {
      if (i < 0) i += Q::TN;
      else if (i >= Q::TN) i -= Q::TN;
    }
    return min(max(i, 0), Q::TN - 1);
  };
  auto own = [&](const int j) {
    const int r = lane * NJ + j - Q::HL;
    return r >= 0 && r < Q::S && wv * Q::S + r < Q::TN;
  };
  T U[NJ][NF], A[NJ][NF], y[NJ][NF], Iv[NJ][NI];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      U[j][f] = y[j][f] = u[G::uidx(f, o0 + at(j), o1, o2)];
      A[j][f] = T(0);
    }
    if constexpr (G::NINV > 0) G::node_inv(o0 + at(j), o1, o2, ep.p, jp, Iv[j]);
  }
  if (!Q::ONE) __syncthreads();   // every wave has read its overlaps before one writes
  // slot of the first and last node (compile time) and the lane holding it in this wave, or -1
  constexpr int QL = Q::HL, QH = Q::HL + Q::SL - 1;
  const bool low = !Q::PER && wv == 0 && lane == QL / NJ, high = !Q::PER && wv == Q::W - 1 && lane == QH / NJ;
  double t = t0;
  // one stage: w holds the lane's nodes and R taps on either side
  auto stage = [&](const int s) {
    const double ts = t + (s == 1 ? 0.0 : (s == 4 ? dt : dt / 2));
    const double cf = s <= 2 ? dt / 2 : (s == 3 ? dt : dt / 6);
    T w[NF * G::VOL];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) w[f * G::VOL + R + j] = y[j][f];
#pragma unroll
      for (int q = 1; q <= R; ++q) {
        w[f * G::VOL + R - q] = mol_lane_below(y[NJ - q][f]);
        w[f * G::VOL + R + NJ - 1 + q] = mol_lane_above(y[q - 1][f]);
      }
    }
    if constexpr (G::FIX && R > 0) {
      // ghosts of the boundary equations from the KMAX nodes next to each end
      T el[NF * G::VOL], eh[NF * G::VOL];
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int m = 0; m < G::KMAX; ++m) {
          el[f * G::VOL + m] = mol_lane(y[(QL + m) % NJ][f], (QL + m) / NJ);
          eh[f * G::VOL + G::KMAX - 1 - m] = mol_lane(y[(QH - m) % NJ][f], (QH - m) / NJ);
        }
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const T gl = G::stage_lds(f, (int)G::ULO0 - 1, o1, o2, ts, ep.p, el, (int)G::ULO0, o1, o2, jp);
        const T gh = G::stage_lds(f, (int)G::UHI0 + 1, o1, o2, ts, ep.p, eh, (int)G::UHI0 - (G::KMAX - 1), o1, o2, jp);
        T& wl = w[f * G::VOL + R + QL % NJ - 1];
        wl = low ? gl : wl;
        T& wh = w[f * G::VOL + R + QH % NJ + 1];
        wh = high ? gh : wh;
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      T out[NF];
      if constexpr (G::NINV > 0) G::node_h(w, R + j, o0 + at(j), o1, o2, ts, ep.p, u, jp, Iv[j], out);
      else G::node(w, R + j, o0 + at(j), o1, o2, ts, ep.p, u, jp, out);
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        T v = (T)cf * out[f];
        v += U[j][f];
        if (s < 4) {
          T a = (s == 1 ? T(1) : T(2)) * out[f];
          if (s > 1) a += A[j][f];
          A[j][f] = a;
        } else {
          v += (T)cf * A[j][f];
          U[j][f] = v;
        }
        y[j][f] = v;
      }
    }
  };
  for (int k = 0; k < nsub; ++k) {
    stage(1);
    stage(2);
    stage(3);
    stage(4);
    t = t + dt;
    if (!Q::ONE && k + 1 < nsub) {
      T* const B = X + (k & 1) * (NF * Q::TN);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int f = 0; f < NF; ++f)
          if (own(j)) B[f * Q::TN + at(j)] = U[j][f];
      __syncthreads();
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int f = 0; f < NF; ++f)
          if (!own(j)) U[j][f] = y[j][f] = B[f * Q::TN + at(j)];
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int f = 0; f < NF; ++f)
      if (own(j)) unew[G::uidx(f, o0 + at(j), o1, o2)] = U[j][f];
  if (ep.tnext && threadIdx.x == 0) ep.tnext[0] = t;
}

// ---------------------------------------------------------------------------------------
// One RK4 step of a 2D system of reach one (cross-shaped stencils) swept along y in registers.
//
// A wave owns a window of columns, one per lane (CX per lane: off the GPU a lane holds whole rows;
// on it two or four FP32 columns per lane halve the DPP moves but not the time), and a strip of rows, and walks up the strip a row per iteration: iteration r takes row r of u, and stage s
// evaluates row r - s from the three newest rows of its input, so the four stages run one row
// apart and every stage value lives in registers for three iterations.  Neighbours along x come
// from the adjacent lanes by DPP, ghosts along a non-periodic axis from the two nodes next to the
// side: no LDS, no barrier, one read and one write of the state per step.  Windows overlap by
// four columns (none where one window holds whole rows), strips by four rows on either side;
// what is evaluated past the needed region never reaches an owned node.  A strip starts at row 0
// of a non-periodic axis or at row 4 or above.
//
// What bounds it is VALU issue: the tile kernel above spends 74 instructions per node and stage of
// the FP64 Brusselator (frame positions, index arithmetic, LDS addresses) where the arithmetic is
// 23; the sweep spends 33, eight of them DPP moves.  Measured, us per step, tile kernel or stage
// launches against the sweep: Brusselator FP64 1501^2 33 / 20, 1024^2 16.7 / 12.3, 400^2 6.8 / 5.6;
// diffusion-reaction FP32 + Kahan 1500^2 57 / 13; 512 FP32 + Kahan instances 266 / 63 (3.2 TB/s).
template <int V>
struct MolInt {
  static constexpr int v = V;
};
struct MolNoHdr {};   // header of a specialised system (all numbers are literals)

// What a batched instance's generated code reads, loaded once per wave.
template <int NF>
struct MolSHdr {
  int n[3];
  MolRow W, K;
  T g[NF][4][3];   // per side (x low, x high, y low, y high): factors of the two nodes next to it, of G
};

// Geometry of one sweep: unknowns nx x ny whose first node is (lo0, lo1), variable f at fofs[f];
// window columns xb .., owned columns [x0, x1) and rows [y0, y1).
template <int NF>
struct MolSweep {
  int nx, ny, lo0, lo1, lo2, xb, x0, x1, y0, y1;
  i64 fofs[NF];
};

// Windows along an axis of n columns: their number, and window w's first and owned columns.
template <bool PER, int CX>
__device__ __forceinline__ constexpr int mol_sweep_windows(const int n) {
  constexpr int WC = MOL_WAVE * CX, S = WC - 8;
  return PER ? (n + S - 1) / S : (n <= WC ? 1 : (n - 8 + S - 1) / S);
}
template <bool PER, int CX, class Q>
__device__ __forceinline__ void mol_sweep_window(Q& g, const int w) {
  constexpr int WC = MOL_WAVE * CX, S = WC - 8;
  const int nw = mol_sweep_windows<PER, CX>(g.nx);
  g.xb = w * S - (PER ? 4 : 0);
  g.x0 = PER ? w * S : (w == 0 ? 0 : g.xb + 4);
  g.x1 = PER ? min(g.nx, (w + 1) * S) : (w == nw - 1 ? g.nx : g.xb + WC - 4);
}

template <class G, bool KAHAN, class HD>
__device__ __forceinline__ void mol_rk4_sweep(const HD& hd, const MolSweep<G::NF>& g, const T* __restrict__ u,
                                              T* __restrict__ unew, const Epi& ep, const JPtrs& jp, const double t) {
  constexpr int NF = G::NF, CX = G::CX, NI = G::NINV > 0 ? G::NINV : 1, PF = 3;
  constexpr bool PX = G::PER0 != 0, PY = G::PER1 != 0;
  typedef T Row[CX][NF];
  const double dt = ep.tadv;
  const int lane = (int)threadIdx.x % MOL_WAVE, nx = g.nx, ny = g.ny, cb = g.xb + lane * CX;
  // node index of each slot (its image on a periodic axis; the last node past the end, where the
  // slot's values are never used)
  int I0[CX];
  unsigned co[CX];
  bool own[CX];
#pragma unroll
  for (int c = 0; c < CX; ++c) {
    int k = cb + c;
    own[c] = k >= g.x0 && k < g.x1;
    if (PX) {
      k = min(k, nx + 3);
      k = k < 0 ? k + nx : (k >= nx ? k - nx : k);
    } else {
      k = min(k, nx - 1);
    }
    I0[c] = g.lo0 + k;
    co[c] = (unsigned)k * (unsigned)sizeof(T);
  }
  auto row_of = [&](int r) {
    if (PY) return r < 0 ? r + ny : (r >= ny ? r - ny : r);
    return min(max(r, 0), ny - 1);
  };
  // row at element offset o of each variable
  auto load = [&](Row& v, const T* __restrict__ src, const i64 o) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const char* const p = (const char*)(src + g.fofs[f] + o);
#pragma unroll
      for (int c = 0; c < CX; ++c) v[c][f] = *(const T*)(p + co[c]);
    }
  };
  auto store = [&](T* __restrict__ dst, const Row& v, const i64 o) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      char* const p = (char*)(dst + g.fofs[f] + o);
#pragma unroll
      for (int c = 0; c < CX; ++c)
        if (own[c]) *(T*)(p + co[c]) = v[c][f];
    }
  };
  // k = f at row q from rows up, ctr, dn of the stage input
  auto eval = [&](const Row& up, const Row& ctr, const Row& dn, const int q, const double ts, const T (&iv)[CX][NI],
                  Row& k) {
    T w[NF * G::VOL];
    const int I1 = g.lo1 + row_of(q);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      T* const L = w + f * G::VOL;
#pragma unroll
      for (int c = 0; c < CX; ++c) {
        L[1 + c] = up[c][f];
        L[1 + c + G::EX] = ctr[c][f];
        L[1 + c + 2 * G::EX] = dn[c][f];
      }
      L[G::EX] = mol_lane_below(ctr[CX - 1][f]);
      L[G::EX + CX + 1] = mol_lane_above(ctr[0][f]);
      if constexpr (!PX) {
        // window 0 starts at column 0
        const T gl = G::ghost(hd, f, 0, L[G::EX + 1], L[G::EX + 2], g.lo0 - 1, I1, g.lo2, ts, ep.p, jp);
        T gh[CX];
#pragma unroll
        for (int c = 0; c < CX; ++c)
          gh[c] = G::ghost(hd, f, 1, L[G::EX + 1 + c], L[G::EX + c], g.lo0 + nx, I1, g.lo2, ts, ep.p, jp);
        L[G::EX] = cb == 0 ? gl : L[G::EX];
#pragma unroll
        for (int c = 0; c < CX; ++c) L[G::EX + 2 + c] = cb + c == nx - 1 ? gh[c] : L[G::EX + 2 + c];
      }
      if constexpr (!PY) {
        if (q == 0)
#pragma unroll
          for (int c = 0; c < CX; ++c)
            L[1 + c] = G::ghost(hd, f, 2, ctr[c][f], dn[c][f], I0[c], g.lo1 - 1, g.lo2, ts, ep.p, jp);
        if (q == ny - 1)
#pragma unroll
          for (int c = 0; c < CX; ++c)
            L[1 + c + 2 * G::EX] = G::ghost(hd, f, 3, ctr[c][f], up[c][f], I0[c], g.lo1 + ny, g.lo2, ts, ep.p, jp);
      }
    }
#pragma unroll
    for (int c = 0; c < CX; ++c) G::node(hd, w, 1 + c + G::EX, I0[c], I1, g.lo2, ts, ep.p, jp, iv[c], k[c]);
  };
  // Rings indexed by the row modulo their length: with six iterations unrolled every index is a
  // constant and no value moves between registers.
  constexpr int UN = 6;
  Row U[UN], Y1[3], Y2[3], Y3[3], A1[2], A2[2], A3[2], pre[PF], cp[UN];
  T iv[UN][CX][NI];
#pragma unroll
  for (int c = 0; c < CX; ++c)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int i = 0; i < UN; ++i) {
        U[i][c][f] = T(0);
        Y1[i % 3][c][f] = Y2[i % 3][c][f] = Y3[i % 3][c][f] = T(0);
        A1[i % 2][c][f] = A2[i % 2][c][f] = A3[i % 2][c][f] = cp[i][c][f] = T(0);
      }
#pragma unroll
  for (int c = 0; c < CX; ++c)
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < UN; ++j) iv[j][c][i] = T(0);
  // r: the row taken by the running iteration; lr: the row being loaded, PF rows ahead (past a
  // non-periodic end the last row again: its values are not used); offsets advance row by row
  const bool cut = !PY && g.y0 == 0;   // no rows below the strip
  int r = cut ? 0 : g.y0 - 4, lr = row_of(r);
  const int rend = g.y1 + 4;
  i64 lo = (i64)lr * nx, so = (i64)g.y0 * nx, ko = so;
  const i64 ke = (i64)g.y1 * nx;
  auto next = [&]() {
    if (PY) {
      if (++lr == ny) {
        lr = 0;
        lo = 0;
      } else {
        lo += nx;
      }
    } else if (lr < ny - 1) {
      ++lr;
      lo += nx;
    }
  };
  const bool comp0 = KAHAN && ep.subA == 0;   // the compensation is read (else it is zero)
  auto load_comp = [&](auto XC) {
    if (KAHAN && comp0 && ko < ke) {
      load(cp[decltype(XC)::v % UN], ep.comp, ko);
      ko += nx;
    }
  };
  // One iteration at ring position X (r modulo 6 from the strip's start) with its first NS stages.
  auto step = [&](auto XC, auto NC) {
    constexpr int x = decltype(XC)::v % 6, NS = decltype(NC)::v;
    Row &u0 = U[x], &u1 = U[(x + 5) % 6], &u2 = U[(x + 4) % 6], &u3 = U[(x + 3) % 6], &u4 = U[(x + 2) % 6];
#pragma unroll
    for (int c = 0; c < CX; ++c)
#pragma unroll
      for (int f = 0; f < NF; ++f) u0[c][f] = pre[x % PF][c][f];
    load(pre[x % PF], u, lo);
    next();
    Row k;
    if constexpr (NS >= 1) {
      auto& iw = iv[(x + 5) % 6];
      if constexpr (G::NINV > 0)
#pragma unroll
        for (int c = 0; c < CX; ++c) G::node_inv(hd, I0[c], g.lo1 + row_of(r - 1), g.lo2, ep.p, jp, iw[c]);
      // u0 .. u4: rows r .. r - 4; stage s evaluates row r - s
      eval(u2, u1, u0, r - 1, t, iw, k);
      Row &a1 = A1[x % 2], &y1 = Y1[x % 3];
#pragma unroll
      for (int c = 0; c < CX; ++c)
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          T v = (T)(dt / 2) * k[c][f];
          v += u1[c][f];
          y1[c][f] = v;
          a1[c][f] = k[c][f];
        }
    }
    if constexpr (NS >= 2) {
      eval(Y1[(x + 1) % 3], Y1[(x + 2) % 3], Y1[x % 3], r - 2, t + dt / 2, iv[(x + 4) % 6], k);
      Row &a2 = A2[x % 2], &b1 = A1[(x + 1) % 2], &y2 = Y2[x % 3];
#pragma unroll
      for (int c = 0; c < CX; ++c)
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          T v = (T)(dt / 2) * k[c][f];
          v += u2[c][f];
          y2[c][f] = v;
          const T a = T(2) * k[c][f];
          a2[c][f] = a + b1[c][f];
        }
    }
    if constexpr (NS >= 3) {
      eval(Y2[(x + 1) % 3], Y2[(x + 2) % 3], Y2[x % 3], r - 3, t + dt / 2, iv[(x + 3) % 6], k);
      Row &a3 = A3[x % 2], &b2 = A2[(x + 1) % 2], &y3 = Y3[x % 3];
#pragma unroll
      for (int c = 0; c < CX; ++c)
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          T v = (T)dt * k[c][f];
          v += u3[c][f];
          y3[c][f] = v;
          const T a = T(2) * k[c][f];
          a3[c][f] = a + b2[c][f];
        }
    }
    if constexpr (NS >= 4) {
      eval(Y3[(x + 1) % 3], Y3[(x + 2) % 3], Y3[x % 3], r - 4, t + dt, iv[(x + 2) % 6], k);
      Row out;
      const Row &cx = cp[(x + 2) % UN], &b3 = A3[(x + 1) % 2];
#pragma unroll
      for (int c = 0; c < CX; ++c)
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          if (KAHAN) {
            T incr = (T)(dt / 6) * k[c][f];
            incr += (T)(dt / 6) * b3[c][f];
            const T y = incr - cx[c][f];
            const T sm = u4[c][f] + y;
            k[c][f] = (sm - u4[c][f]) - y;
            out[c][f] = sm;
          } else {
            T v = (T)(dt / 6) * k[c][f];
            v += u4[c][f];
            v += (T)(dt / 6) * b3[c][f];
            out[c][f] = v;
          }
        }
      store(unew, out, so);
      if (KAHAN) store(ep.comp, k, so);
      so += nx;
    }
    // row r + 2 of the compensation, wanted six iterations later (its slot held row r - 4's)
    if constexpr (NS >= 1) load_comp(MolInt<x + 2>{});
    ++r;
  };
  // Rows y0 - 4 .. y0 + 3 start the stages two rows apart (a strip at a non-periodic end starts at
  // its first row); from row y0 + 4 on every iteration finishes one row.
#define MOL_STEP(X, N) step(MolInt<X>{}, MolInt<N>{})
  auto fill = [&](auto XC) {   // the first PF rows, the strip's first one at ring position X
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      load(pre[(decltype(XC)::v + i) % PF], u, lo);
      next();
    }
  };
  if (!cut) {
    fill(MolInt<0>{});
    MOL_STEP(0, 0); MOL_STEP(1, 0); MOL_STEP(2, 1); MOL_STEP(3, 1);
  } else {
    fill(MolInt<4>{});
    load_comp(MolInt<4>{});
    load_comp(MolInt<5>{});
  }
  MOL_STEP(4, 2); MOL_STEP(5, 2); MOL_STEP(6, 3); MOL_STEP(7, 3);
  while (true) {
    MOL_STEP(8, 4);
    if (r >= rend) break;
    MOL_STEP(9, 4);
    if (r >= rend) break;
    MOL_STEP(10, 4);
    if (r >= rend) break;
    MOL_STEP(11, 4);
    if (r >= rend) break;
    MOL_STEP(12, 4);
    if (r >= rend) break;
    MOL_STEP(13, 4);
    if (r >= rend) break;
  }
#undef MOL_STEP
}

// Arguments of the generated vector-Jacobian product (layout identical to mol::VArgs<T>).
// The seed is lam = c1*s1 + c2*s2 (s2 may be null); out receives (df/du)^T lam and g_aux the
// FP64 auxiliary-array gradients (may be null); both are accumulated, not overwritten.  bf and
// ba hold each tile's tile + halo adjoints of the staged variables and grid fields between the
// tile kernel and the gather kernel.
struct VArgs {
  const T* u;
  const T* s1;
  const T* s2;
  double c1, c2;
  T* out;
  double* g_aux;
  const T* p;
  const double* tnow;
  double tofs;
  T* bf;
  double* ba;
  int mode;   // 1: gather the variables, 2: gather the grid fields, 4: add the tile kernel's
              // grid-field adjoints to the buffers instead of storing them, 8: the gather ends
              // an RK4 step of the adjoint sweep: lam = lam + y0 + y1 + y2 + (this gather)
  T* lam;
  const T* y0;
  const T* y1;
  const T* y2;
};

// Floor of a / b for b > 0.
__device__ __forceinline__ int mol_floordiv(const int a, const int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }

// Tiles along one axis whose tile + halo (halo H, the larger of the two variants) contains
// position p or, on a periodic axis with period P, one of its images p + kP: tile indices and
// the position relative to each tile's origin.  At most 10 entries.
template <int TL, int H, int NT, int ULO, bool PER, int P>
__device__ __forceinline__ int mol_cover(const int p, int* ts, int* ls) {
  int n = 0;
  if (!PER && H <= TL) {
    // own tile and at most one neighbour on each side
    const int r = p - ULO, t = mol_floordiv(r, TL), l = r - t * TL;
    if (l < H && t - 1 >= 0 && t - 1 < NT) { ts[n] = t - 1; ls[n] = l + TL; ++n; }
    if (t >= 0 && t < NT) { ts[n] = t; ls[n] = l; ++n; }
    if (l >= TL - H && t + 1 >= 0 && t + 1 < NT) { ts[n] = t + 1; ls[n] = l - TL; ++n; }
    return n;
  }
#pragma unroll
  for (int k = PER ? -2 : 0; k <= (PER ? 2 : 0); ++k) {
    const int pp = p + k * P;
    const int tlo = max(0, -mol_floordiv(-(pp - ULO - TL + 1 - H), TL));
    const int thi = min(NT - 1, mol_floordiv(pp - ULO + H, TL));
    for (int t = tlo; t <= thi && n < 10; ++t) {
      ts[n] = t;
      ls[n] = pp - (ULO + t * TL);
      ++n;
    }
  }
  return n;
}

// The (at most) three tiles along one axis whose tile + halo H contains position p: the left
// neighbour, the own tile and the right neighbour (slots 0, 1, 2), with p relative to each
// tile's origin; on a periodic axis of period P the neighbours across the ends hold the images
// p + P and p - P.  Exact when H <= TL and, on a periodic axis, the last tile is at least H wide.
struct MolCov {
  int t[3], l[3];
  bool v[3];
};
template <int TL, int H, int NT, int ULO, bool PER, int P>
__device__ __forceinline__ MolCov mol_cover3(const int p) {
  MolCov c;
  const int r = p - ULO, t = mol_floordiv(r, TL), l = r - t * TL;
  c.t[1] = t;
  c.l[1] = l;
  c.v[1] = t >= 0 && t < NT;
  if (t - 1 >= 0 || !PER) {
    c.t[0] = t - 1;
    c.l[0] = l + TL;
    c.v[0] = l < H && t - 1 >= 0 && t - 1 < NT;
  } else {
    c.t[0] = NT - 1;
    c.l[0] = r + P - (NT - 1) * TL;
    c.v[0] = c.l[0] < TL + H;
  }
  if (t + 1 < NT || !PER) {
    c.t[2] = t + 1;
    c.l[2] = l - TL;
    c.v[2] = l >= TL - H && t + 1 >= 0 && t + 1 < NT;
  } else {
    c.t[2] = 0;
    c.l[2] = r - P;
    c.v[2] = c.l[2] >= -H;
  }
  return c;
}

template <class G, int A>
struct MolAxis {
  static constexpr int TL = A == 0 ? G::TX : (A == 1 ? G::TY : G::TZ);
  static constexpr int H = A == 0 ? G::HX : (A == 1 ? G::HY : G::HZ);
  static constexpr int NT = A == 0 ? G::NT0 : (A == 1 ? G::NT1 : G::NT2);
  static constexpr int ULO = A == 0 ? G::ULO0 : (A == 1 ? G::ULO1 : G::ULO2);
  static constexpr int UHI = A == 0 ? G::UHI0 : (A == 1 ? G::UHI1 : G::UHI2);
  static constexpr bool PER = (A == 0 ? G::PER0 : (A == 1 ? G::PER1 : G::PER2)) != 0;
  static constexpr int P = (A == 0 ? G::N0 : (A == 1 ? G::N1 : G::N2)) - 1;
  static constexpr bool FAST = H <= TL && (!PER || (UHI - ULO + 1) - (NT - 1) * TL >= H);
};

// Adjoint-buffer value of slot s at tile-relative position (l0, l1, l2) of tile (t0, t1, t2), in
// the tile's own variant layout, or 0 outside that variant's tile + halo.
template <class GC, class GB, bool HASC, int VOLX, int NS, typename B>
__device__ __forceinline__ double mol_tile_buf(const B* __restrict__ base, const int s, const int t0, const int t1,
                                               const int t2, const int l0, const int l1, const int l2) {
  // cross-shaped staging: positions outside the tile along two or more axes hold no adjoint
  // (no diagonal taps) and the tile kernel leaves their buffer entries unwritten
  if (GB::CROSS && (int)(l0 < 0 || l0 >= GB::TX) + (int)(l1 < 0 || l1 >= GB::TY) + (int)(l2 < 0 || l2 >= GB::TZ) >= 2)
    return 0.0;
  const int tl = t0 + GB::NT0 * (t1 + GB::NT1 * t2);
  int q;
  if (HASC && GB::is_core(t0, t1, t2)) {
    if (l0 < -GC::HX || l0 >= GC::TX + GC::HX || l1 < -GC::HY || l1 >= GC::TY + GC::HY || l2 < -GC::HZ ||
        l2 >= GC::TZ + GC::HZ)
      return 0.0;
    q = (l0 + GC::HX) + GC::EX * ((l1 + GC::HY) + GC::EY * (l2 + GC::HZ));
  } else {
    if (l0 < -GB::HX || l0 >= GB::TX + GB::HX || l1 < -GB::HY || l1 >= GB::TY + GB::HY || l2 < -GB::HZ ||
        l2 >= GB::TZ + GB::HZ)
      return 0.0;
    q = (l0 + GB::HX) + GB::EX * ((l1 + GB::HY) + GB::EY * (l2 + GB::HZ));
  }
  return (double)base[(i64)tl * (NS * VOLX) + (i64)s * VOLX + q];
}

// Sum over the tiles covering position (p0, p1, p2) of slot s of their adjoint buffers (base:
// buffer of tile 0, stride NS * VOLX per tile), in a fixed order: each tile in its own
// variant's layout.
template <class GC, class GB, bool HASC, int VOLX, int NS, typename B>
__device__ __forceinline__ double mol_gather_pos(const B* __restrict__ base, const int s, const int p0, const int p1,
                                                 const int p2) {
  using A0 = MolAxis<GB, 0>;
  using A1 = MolAxis<GB, 1>;
  using A2 = MolAxis<GB, 2>;
  double sum = 0.0;
  if (A0::FAST && A1::FAST && A2::FAST) {
    const MolCov c0 = mol_cover3<A0::TL, A0::H, A0::NT, A0::ULO, A0::PER, A0::P>(p0);
    const MolCov c1 = mol_cover3<A1::TL, A1::H, A1::NT, A1::ULO, A1::PER, A1::P>(p1);
    const MolCov c2 = mol_cover3<A2::TL, A2::H, A2::NT, A2::ULO, A2::PER, A2::P>(p2);
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          // slot 1 is the tile owning the position along that axis; with cross-shaped staging a
          // neighbour along two or more axes holds the position outside its tile along those
          // axes, where its buffer is never written: those combinations drop out at compile time
          if (GB::CROSS && (int)(a != 1) + (int)(b != 1) + (int)(c != 1) >= 2) continue;
          if (c0.v[a] && c1.v[b] && c2.v[c])
            sum += mol_tile_buf<GC, GB, HASC, VOLX, NS>(base, s, c0.t[a], c1.t[b], c2.t[c], c0.l[a], c1.l[b], c2.l[c]);
        }
    return sum;
  }
  int t0[10], l0[10], t1[10], l1[10], t2[10], l2[10];
  const int n0 = mol_cover<GB::TX, GB::HX, GB::NT0, GB::ULO0, GB::PER0 != 0, GB::N0 - 1>(p0, t0, l0);
  const int n1 = mol_cover<GB::TY, GB::HY, GB::NT1, GB::ULO1, GB::PER1 != 0, GB::N1 - 1>(p1, t1, l1);
  const int n2 = mol_cover<GB::TZ, GB::HZ, GB::NT2, GB::ULO2, GB::PER2 != 0, GB::N2 - 1>(p2, t2, l2);
  for (int c = 0; c < n2; ++c)
    for (int b = 0; b < n1; ++b)
      for (int a = 0; a < n0; ++a)
        sum += mol_tile_buf<GC, GB, HASC, VOLX, NS>(base, s, t0[a], t1[b], t2[c], l0[a], l1[b], l2[c]);
  return sum;
}

// One tile of the reverse-mode sweep in tile variant G: stage as the forward kernel, run each
// node's adjoint (tap adjoints summed in FP64 in LDS with LDS atomics, whatever the state's
// type; arrays read only at the node go
// straight to global memory), then add the LDS adjoints of tile + halo to the unknowns (through
// the transposed ghost closures) and to the grid-field gradients.
template <class G, int VOLX>
__device__ __forceinline__ void mol_vjp_tile(T* L, double* Ab, double* Aa, const int tx, const int ty, const int tz,
                                             const VArgs& va, const JPtrs& jp, const double t) {
  const int o0 = G::ULO0 + tx * G::TX, o1 = G::ULO1 + ty * G::TY, o2 = G::ULO2 + tz * G::TZ;
  constexpr int EXY = G::EX * G::EY;
  {
    const int mode = mol_stage_mode<G>(tx, ty, tz);
    MolWalk<G::EX, G::EY, G::NTHR> w((int)threadIdx.x);
    for (int q = threadIdx.x; q < G::VOL; q += G::NTHR, w.step()) {
      if (!mol_unread<G>(w.x, w.y, w.z)) {
        G::stage_pos(L, q, o0 + w.x - G::HX, o1 + w.y - G::HY, o2 + w.z - G::HZ, mode, t, va.p, va.u, jp);
        G::zero_pos(Ab, Aa, q);
      }
    }
  }
  __syncthreads();
  constexpr int TXY = G::TX * G::TY, TVOL = TXY * G::TZ;
  for (int q = threadIdx.x; q < TVOL; q += G::NTHR) {
    const int lz = q / TXY;
    const int rr = q - lz * TXY;
    const int ly = rr / G::TX;
    const int lx = rr - ly * G::TX;
    const int I0 = o0 + lx, I1 = o1 + ly, I2 = o2 + lz;
    if (I0 > G::UHI0 || I1 > G::UHI1 || I2 > G::UHI2) continue;
    T lam[G::NF];
    bool any = false;
#pragma unroll
    for (int f = 0; f < G::NF; ++f) {
      T s = T(0);
      if (G::inbox(f, I0, I1, I2)) {
        const auto k = G::uidx(f, I0, I1, I2);
        s = (T)va.c1 * va.s1[k];
        if (va.s2) s += (T)va.c2 * va.s2[k];
      }
      lam[f] = s;
      any = any || s != T(0);
    }
    if (!any) continue;
    const int base = (lx + G::HX) + G::EX * (ly + G::HY) + EXY * (lz + G::HZ);
    G::vjp(L, Ab, Aa, base, I0, I1, I2, t, va.p, va.u, jp, lam, va.out, va.g_aux);
  }
  __syncthreads();
  // tile + halo adjoints to this tile's buffers (plain stores; the gather kernel sums the
  // buffers of the tiles covering each position), ghost positions through the closures
  const i64 tl = tx + (i64)G::NT0 * (ty + (i64)G::NT1 * tz);
  T* bft = va.bf + tl * (G::NSTF * VOLX);
  double* bat = va.g_aux ? va.ba + tl * (G::NSTA * VOLX) : nullptr;
  const bool acc = (va.mode & 4) != 0;
  MolWalk<G::EX, G::EY, G::NTHR> w((int)threadIdx.x);
  for (int q = threadIdx.x; q < G::VOL; q += G::NTHR, w.step())
    if (!mol_unread<G>(w.x, w.y, w.z))
      G::flush_pos(Ab, Aa, q, o0 + w.x - G::HX, o1 + w.y - G::HY, o2 + w.z - G::HZ, va.out, bft, bat, VOLX, acc);
}

// ---------------------------------------------------------------------------------------
// 3D divergence form  u_t = r(u, aux) + sum over the axes of  d/dx (a(u, aux) du/dx)  marched
// along z: the right-hand side (or one Runge-Kutta stage) and its reverse mode.
//
// The reference evaluates the half-point flux a(...) du/dx on either side of a node; the flux on
// a node's upper side is the one on the lower side of its neighbour.  A work-group owns TX x TY
// columns and walks up a chunk of planes: along z a thread keeps the last planes and the last flux in
// registers, along x and y the plane lies in LDS with its halo, every thread evaluates the fluxes
// on its upper sides and leaves them in LDS for the neighbours.  So a node costs three fluxes
// instead of six, and the state is read once per plane and tile (with the halo columns) instead
// of 2.25 times.  The one-sided interpolation next to a side equals the interior row with one
// more node past the boundary node, extrapolated from the four nodes next to it (G::ext): with
// that node all half points have one formula.  Every load of a plane is without a branch (columns
// outside are clamped) and one plane ahead; boundary and extrapolated nodes are made from the
// staged plane, along z from the planes in registers.
// Bound: forward FP64 by memory (126^3: 22 us per stage for about 105 MB, 31 us with tiles that stage
// 2.25 positions per node), FP32 and small grids by the serial chain of a plane (LDS, fluxes, LDS:
// 0.9 us).  Reverse mode 47 us instead of 105 (tile kernel and gather) at 126^3, 15 instead of 33
// at 73^3 FP32: about 620 instructions and three barriers per plane.
//
// Positions are counted from the first unknown: 0 .. M-1 unknowns, -1 and M boundary nodes, -2 and
// M + 1 the extrapolated ones.  Staged arrays: 0 the state, 1 .. NAH the grid fields of a().

// Launch bounds with a number of waves per SIMD unit that the registers have to allow.
#ifdef __AMDGCN__
#define MOL_BOUNDS(threads, waves) __launch_bounds__(threads, waves)
#else
#define MOL_BOUNDS(threads, waves)
#endif

// Offsets in bytes of a column in a plane of the state and of a grid field; columns outside give the
// nearest one.  (The plane is added to the pointer, which is the same for all threads.)
template <class G>
struct MolFluxCol {
  unsigned u, a;
  __device__ __forceinline__ void at(const int x, const int y) {
    u = (unsigned)(min(max(x, 0), G::M0 - 1) + G::M0 * min(max(y, 0), G::M1 - 1)) * (unsigned)sizeof(T);
    a = (unsigned)((min(max(x, -1), (int)G::M0) + 1) + G::N0 * (min(max(y, -1), (int)G::M1) + 1)) * (unsigned)sizeof(T);
  }
};
template <typename V>
__device__ __forceinline__ V& mol_at(V* const p, const unsigned bytes) {
  return *(V*)((char*)p + bytes);
}
template <typename V>
__device__ __forceinline__ const V& mol_at(const V* const p, const unsigned bytes) {
  return *(const V*)((const char*)p + bytes);
}

// The same with the pointer kept in scalar registers.  Left to itself the compiler holds pointer +
// offset of every array over the loop, two vector registers each: the reverse mode takes 166
// registers instead of 141 (FP64) and 1.1 to 1.4 times as long in FP32, the right-hand side, which
// has registers to spare, gets slower by a few per cent.
#ifdef __AMDGCN__
template <typename V>
using MolGlobal = __attribute__((address_space(1))) V;
__device__ __forceinline__ MolGlobal<char>* mol_scalar(const void* const p) {
  const unsigned long long v = (unsigned long long)p;   // (an "s" operand has to be in scalar registers)
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
  return (MolGlobal<char>*)(((unsigned long long)hi << 32) | lo);
}
template <typename V>
__device__ __forceinline__ MolGlobal<V>& mol_at_s(V* const p, unsigned bytes) {
  MolGlobal<char>* q = mol_scalar(p);
  asm("" : "+s"(q), "+v"(bytes));
  return *(MolGlobal<V>*)(q + bytes);
}
template <typename V>
__device__ __forceinline__ const MolGlobal<V>& mol_at_s(const V* const p, unsigned bytes) {
  MolGlobal<char>* q = mol_scalar(p);
  asm("" : "+s"(q), "+v"(bytes));
  return *(const MolGlobal<V>*)(q + bytes);
}
#else
template <typename V>
inline V& mol_at_s(V* const p, const unsigned bytes) {
  return mol_at(p, bytes);
}
#endif

// Staged arrays of a column at plane z (state at the nearest unknown); SC: scalar pointers.
template <class G, bool SC>
__device__ __forceinline__ void mol_flux_load(T (&v)[1 + G::NAH], const MolFluxCol<G>& c, const T* __restrict__ u,
                                              const JPtrs& jp, const int z) {
  int zu = min(max(z, 0), G::M2 - 1), za = min(max(z, -1), (int)G::M2) + 1;
  if constexpr (SC) {
    zu = mol_uniform(zu);
    za = mol_uniform(za);
  }
  const T* const p = u + (i64)G::M0 * G::M1 * zu;
  v[0] = SC ? mol_at_s(p, c.u) : mol_at(p, c.u);
#pragma unroll
  for (int a = 0; a < G::NAH; ++a) {
    const T* const q = jp.aux[G::AH[a]] + (i64)G::N0 * G::N1 * za;
    v[1 + a] = SC ? mol_at_s(q, c.a) : mol_at(q, c.a);
  }
}

// State at the boundary (g = 0) or extrapolated (g = 1) node of a side from the three unknowns
// next to it.
template <class G>
__device__ __forceinline__ T mol_flux_ghost(const int ax, const int side, const int g, const T n0, const T n1, const T n2,
                                            const T bv) {
  T s = G::closure(ax, side, g, 0) * n0;
  s += G::closure(ax, side, g, 1) * n1;
  s += G::closure(ax, side, g, 2) * n2;
  if constexpr (G::BV) s += G::closure(ax, side, g, 3) * bv;
  return s;
}

// Plane M2 (g = 0) or M2 + 1 (g = 1) of a column from the four planes before it, the last in r3;
// v holds the loaded grid fields.
template <class G>
__device__ __forceinline__ void mol_flux_above(T (&v)[1 + G::NAH], const T (&r0)[1 + G::NAH], const T (&r1)[1 + G::NAH],
                                               const T (&r2)[1 + G::NAH], const T (&r3)[1 + G::NAH], const int g,
                                               const T bv) {
  if (g == 0) {
    v[0] = mol_flux_ghost<G>(2, 1, 0, r3[0], r2[0], r1[0], bv);
  } else {
    v[0] = mol_flux_ghost<G>(2, 1, 1, r2[0], r1[0], r0[0], bv);
#pragma unroll
    for (int a = 1; a <= G::NAH; ++a)
      v[a] = G::ext(2, 1, 0) * r3[a] + G::ext(2, 1, 1) * r2[a] + G::ext(2, 1, 2) * r1[a] + G::ext(2, 1, 3) * r0[a];
  }
}

// Value of the boundary program of a side at a position (coordinates outside the grid: the nearest).
template <class G>
__device__ __forceinline__ T mol_flux_bval(const int ax, const int side, const int x, const int y, const int z,
                                           const double t, const T* __restrict__ P, const JPtrs& jp) {
  if constexpr (!G::BV) return T(0);
  else
    return G::bval(ax, side, min(max(x, -1), (int)G::M0) + 2, min(max(y, -1), (int)G::M1) + 2,
                   min(max(z, -1), (int)G::M2) + 2, t, P, jp);
}

// NP planes z0 - B .. of a column: loaded, then those past a side along z.
template <class G, int NP, int B, bool SC>
__device__ __forceinline__ void mol_flux_planes(T (&q)[NP][1 + G::NAH], const MolFluxCol<G>& col, const int x, const int y,
                                                const int z0, const T* __restrict__ u, const JPtrs& jp, const double t,
                                                const T* __restrict__ P) {
#pragma unroll
  for (int i = 0; i < NP; ++i) mol_flux_load<G, SC>(q[i], col, u, jp, z0 - B + i);
  if (z0 == 0) {
    const T bv = mol_flux_bval<G>(2, 0, x, y, -1, t, P, jp);
    q[B - 1][0] = mol_flux_ghost<G>(2, 0, 0, q[B][0], q[B + 1][0], q[B + 2][0], bv);
    q[B - 2][0] = mol_flux_ghost<G>(2, 0, 1, q[B][0], q[B + 1][0], q[B + 2][0], bv);
#pragma unroll
    for (int a = 1; a <= G::NAH; ++a)
      q[B - 2][a] = G::ext(2, 0, 0) * q[B - 1][a] + G::ext(2, 0, 1) * q[B][a] + G::ext(2, 0, 2) * q[B + 1][a] +
                    G::ext(2, 0, 3) * q[B + 2][a];
  }
  if (z0 - B + NP > G::M2)   // (the last chunk has three planes or more: plane M2 only, the last)
    mol_flux_above<G>(q[NP - 1], q[0], q[NP - 4], q[NP - 3], q[NP - 2], 0, mol_flux_bval<G>(2, 1, x, y, G::M2, t, P, jp));
}

// First plane of chunk i: NT2 chunks that differ by one plane at most (three planes or more).
template <class G>
__device__ __forceinline__ int mol_flux_chunk(const int i) {
  return (int)((i64)G::M2 * i / G::NT2);
}

// Halo position q of a TX x TY tile with HL positions before and HH past it along either axis
// (no corners), relative to the tile.
template <class G, int HL, int HH>
__device__ __forceinline__ void mol_flux_halo(const int q, int& x, int& y) {
  constexpr int H = HL + HH;
  const int r = q - H * G::TY;
  const bool ax = r < 0;
  const int y0 = q / H, x0 = q - y0 * H, y1 = r / G::TX, x1 = r - y1 * G::TX;
  x = ax ? (x0 < HL ? x0 - HL : G::TX + (x0 - HL)) : x1;
  y = ax ? y0 : (y1 < HL ? y1 - HL : G::TY + (y1 - HL));
}

// Boundary and extrapolated nodes of one side in the staged plane (halo HL, HH, rows of LX).
template <class G, int AX, int SIDE, int HL, int HH, int LX>
__device__ __forceinline__ void mol_flux_side(T* const L, const int LN, const int X0, const int Y0, const int c,
                                              const double t, const T* __restrict__ P, const JPtrs& jp) {
  constexpr int M = AX == 0 ? G::M0 : G::M1, TA = AX == 0 ? G::TX : G::TY, TB = AX == 0 ? G::TY : G::TX;
  const int b = (SIDE == 0 ? -1 : M) - (AX == 0 ? X0 : Y0);   // the boundary node, relative to the tile
  if (SIDE == 0 ? b != -1 : b >= TA + HH) return;
  const bool two = SIDE == 0 || b + 1 < TA + HH;
  constexpr int st = AX == 0 ? 1 : LX, d = SIDE == 0 ? st : -st;
  for (int r = (int)threadIdx.x; r < TB; r += G::NTHR) {
    const int o = AX == 0 ? (b + HL) + LX * (r + HL) : (r + HL) + LX * (b + HL);
    const T bv = AX == 0 ? mol_flux_bval<G>(0, SIDE, X0 + b, Y0 + r, c, t, P, jp)
                         : mol_flux_bval<G>(1, SIDE, X0 + r, Y0 + b, c, t, P, jp);
    const T n0 = L[o + d], n1 = L[o + 2 * d], n2 = L[o + 3 * d];
    L[o] = mol_flux_ghost<G>(AX, SIDE, 0, n0, n1, n2, bv);
    if (two) {
      L[o - d] = mol_flux_ghost<G>(AX, SIDE, 1, n0, n1, n2, bv);
#pragma unroll
      for (int a = 1; a <= G::NAH; ++a) {
        const T* const A = L + a * LN + o;
        L[a * LN + o - d] = G::ext(AX, SIDE, 0) * A[0] + G::ext(AX, SIDE, 1) * A[d] + G::ext(AX, SIDE, 2) * A[2 * d] +
                            G::ext(AX, SIDE, 3) * A[3 * d];
      }
    }
  }
}

// All four sides of a staged plane, and the barrier after it (a tile that touches no side has none).
template <class G, int HL, int HH, int LX>
__device__ __forceinline__ void mol_flux_sides(T* const L, const int LN, const int X0, const int Y0, const int c,
                                               const double t, const T* __restrict__ P, const JPtrs& jp) {
  if (X0 > 0 && Y0 > 0 && X0 + G::TX + HH <= G::M0 && Y0 + G::TY + HH <= G::M1) return;
  mol_flux_side<G, 0, 0, HL, HH, LX>(L, LN, X0, Y0, c, t, P, jp);
  mol_flux_side<G, 0, 1, HL, HH, LX>(L, LN, X0, Y0, c, t, P, jp);
  mol_flux_side<G, 1, 0, HL, HH, LX>(L, LN, X0, Y0, c, t, P, jp);
  mol_flux_side<G, 1, 1, HL, HH, LX>(L, LN, X0, Y0, c, t, P, jp);
  __syncthreads();
}

// Interpolated values and inner derivative at a half point from four consecutive positions.
template <class G>
__device__ __forceinline__ void mol_flux_half(const int ax, const T (&w)[4][1 + G::NAH], T (&h)[1 + G::NAH], T& d) {
#pragma unroll
  for (int a = 0; a <= G::NAH; ++a) {
    T s = G::wi(ax, 0) * w[0][a];
    s += G::wi(ax, 1) * w[1][a];
    s += G::wi(ax, 2) * w[2][a];
    s += G::wi(ax, 3) * w[3][a];
    h[a] = s;
  }
  d = G::wd(ax, 0) * w[1][0];
  d += G::wd(ax, 1) * w[2][0];
}

template <class G, int AX>
__device__ __forceinline__ T mol_flux_at(const T (&w)[4][1 + G::NAH], const double t, const T* __restrict__ P) {
  T h[1 + G::NAH], d;
  mol_flux_half<G>(AX, w, h, d);
  return G::template flux<AX>(h, d, t, P);
}

// Right-hand side or one stage.  L: plane with a halo of two, FX, FY: fluxes on the upper sides of
// columns -1 .. and rows -1 ..
template <class G>
struct MolFluxLds {
  static constexpr int LX = G::TX + 4, LY = G::TY + 4, NA = 1 + G::NAH, NC = G::TX * G::TY;
  T L[NA][LX * LY];
  T FX[(G::TX + 1) * G::TY], FY[G::TX * (G::TY + 1)];
};

template <class G>
__device__ __forceinline__ void mol_flux_rhs(MolFluxLds<G>& S, const T* __restrict__ u, const Epi& ep, const JPtrs& jp,
                                             const double t) {
  typedef MolFluxLds<G> Q;
  constexpr int TX = G::TX, TY = G::TY, NA = Q::NA, NI = Q::NC / G::NTHR, NH = 4 * (TX + TY);
  constexpr int NHI = (NH + G::NTHR - 1) / G::NTHR, NQ = G::NAU > 0 ? G::NAU : 1;
  constexpr i64 PU = (i64)G::M0 * G::M1, PA = (i64)G::N0 * G::N1;
  const int b = mol_xcd_tile<G::NBLK>((int)blockIdx.x);
  const int X0 = (b % G::NT0) * TX, Y0 = (b / G::NT0 % G::NT1) * TY, zc = b / (G::NT0 * G::NT1);
  const int z0 = mol_flux_chunk<G>(zc), z1 = mol_flux_chunk<G>(zc + 1);
  const T* const P = ep.p;
  T R[NI][4][NA], Fz[NI], hv[NHI][NA];   // planes c-1 .. c+2 of a column, flux below plane c, halo of plane c
  int cx[NI], cy[NI], ho[NHI];           // ho: the halo position's place in L
  MolFluxCol<G> col[NI], hc[NHI];
#pragma unroll
  for (int i = 0; i < NHI; ++i) {
    int x, y;
    mol_flux_halo<G, 2, 2>(min((int)threadIdx.x + i * G::NTHR, NH - 1), x, y);   // (past the last: it again)
    hc[i].at(X0 + x, Y0 + y);
    ho[i] = (x + 2) + Q::LX * (y + 2);
    mol_flux_load<G, false>(hv[i], hc[i], u, jp, z0);
  }
#pragma unroll
  for (int k = 0; k < NI; ++k) {
    const int q = (int)threadIdx.x + k * G::NTHR;
    cy[k] = q / TX;
    cx[k] = q - cy[k] * TX;
    col[k].at(X0 + cx[k], Y0 + cy[k]);
    T v[5][NA], w[4][NA];
    mol_flux_planes<G, 5, 2, false>(v, col[k], X0 + cx[k], Y0 + cy[k], z0, u, jp, t, P);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        w[i][a] = v[i][a];
        R[k][i][a] = v[i + 1][a];
      }
    Fz[k] = mol_flux_at<G, 2>(w, t, P);
  }
  for (int c = z0; c < z1; ++c) {
    // the plane into LDS
#pragma unroll
    for (int k = 0; k < NI; ++k)
#pragma unroll
      for (int a = 0; a < NA; ++a) S.L[a][(cx[k] + 2) + Q::LX * (cy[k] + 2)] = R[k][1][a];
#pragma unroll
    for (int i = 0; i < NHI; ++i)
#pragma unroll
      for (int a = 0; a < NA; ++a) S.L[a][ho[i]] = hv[i][a];
    // what the next plane and this plane's node program and update read, in flight during the fluxes
    T nxt[NI][NA], av[NI][NQ], ea[NI], eb[NI], ec[NI];
#pragma unroll
    for (int i = 0; i < NHI; ++i) mol_flux_load<G, false>(hv[i], hc[i], u, jp, c + 1);
    const i64 pu = PU * c, pa = PA * (c + 1);
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      mol_flux_load<G, false>(nxt[k], col[k], u, jp, c + 3);
#pragma unroll
      for (int a = 0; a < G::NAU; ++a) av[k][a] = mol_at(jp.aux[G::AN[a]] + pa, col[k].a);
      ea[k] = eb[k] = ec[k] = T(0);
      if (ep.mode != 0) {
        if (ep.A) ea[k] = mol_at(ep.A + pu, col[k].u);
        if (ep.B) eb[k] = mol_at(ep.B + pu, col[k].u);
        if (ep.mode == 2) ec[k] = mol_at(ep.comp + pu, col[k].u);
        else if (ep.acc && ep.acc_keep != 0.0) ec[k] = mol_at(ep.acc + pu, col[k].u);
      }
    }
    __syncthreads();
    mol_flux_sides<G, 2, 2, Q::LX>(&S.L[0][0], Q::LX * Q::LY, X0, Y0, c, t, P, jp);
    T fx[NI], fy[NI], fz[NI];
    auto face = [&](const int ax, const int x, const int y) {
      const int o = (x + 2) + Q::LX * (y + 2), st = ax == 0 ? 1 : Q::LX;
      T w[4][NA];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int a = 0; a < NA; ++a) w[i][a] = S.L[a][o + (i - 1) * st];
      return ax == 0 ? mol_flux_at<G, 0>(w, t, P) : mol_flux_at<G, 1>(w, t, P);
    };
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      fx[k] = face(0, cx[k], cy[k]);
      fy[k] = face(1, cx[k], cy[k]);
      fz[k] = mol_flux_at<G, 2>(R[k], t, P);
      S.FX[(cx[k] + 1) + (TX + 1) * cy[k]] = fx[k];
      S.FY[cx[k] + TX * (cy[k] + 1)] = fy[k];
    }
    for (int q = (int)threadIdx.x; q < TX + TY; q += G::NTHR) {   // the lower sides of the tile
      if (q < TY) S.FX[(TX + 1) * q] = face(0, -1, q);
      else S.FY[q - TY] = face(1, q - TY, -1);
    }
    __syncthreads();
    const int g = c + 3 - G::M2;
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      const int x = X0 + cx[k], y = Y0 + cy[k];
      T sv[3], out;
      sv[0] = G::wo(0, 0) * S.FX[cx[k] + (TX + 1) * cy[k]] + G::wo(0, 1) * fx[k];
      sv[1] = G::wo(1, 0) * S.FY[cx[k] + TX * cy[k]] + G::wo(1, 1) * fy[k];
      sv[2] = G::wo(2, 0) * Fz[k] + G::wo(2, 1) * fz[k];
      Fz[k] = fz[k];
      if (x < G::M0 && y < G::M1) {
        G::node(R[k][1][0], sv, av[k], x + 2, y + 2, c + 2, t, P, jp, out);
        const unsigned i = col[k].u;
        if (ep.mode == 0) {
          mol_at(ep.out + pu, i) = out;
        } else if (ep.mode == 1) {
          T v = (T)ep.cf * out;
          if (ep.A) v += (T)ep.ca * ea[k];
          if (ep.B) v += (T)ep.cb * eb[k];
          if (ep.acc) {
            T a = (T)ep.acc_f * out;
            if (ep.acc_keep != 0.0) a += (T)ep.acc_keep * ec[k];
            mol_at(ep.acc + pu, i) = a;
          }
          mol_at(ep.out + pu, i) = v;
        } else {
          T incr = (T)ep.cf * out;
          if (ep.B) incr += (T)ep.cb * (ep.subA ? (eb[k] - ea[k]) : eb[k]);
          const T yk = incr - ec[k];
          const T s = ea[k] + yk;
          mol_at(ep.comp + pu, i) = (s - ea[k]) - yk;
          mol_at(ep.out + pu, i) = s;
        }
      }
      if (g == 0 || g == 1) {
        const T bv = mol_flux_bval<G>(2, 1, x, y, G::M2, t, P, jp);
        mol_flux_above<G>(nxt[k], R[k][0], R[k][1], R[k][2], R[k][3], g, bv);
      }
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        R[k][0][a] = R[k][1][a];
        R[k][1][a] = R[k][2][a];
        R[k][2][a] = R[k][3][a];
        R[k][3][a] = nxt[k][a];
      }
    }
  }
}

// Reverse mode of the march: lam_dot = (df/du)^T lam and the gradients of the grid fields, each
// node's sum complete in one thread (no atomics, no per-tile buffers, no gather).  With
// phi = wo1 lam(h) + wo0 lam(h+1) the adjoint of the flux at half point h (lam = 0 outside the
// unknowns), a half point leaves p = phi dF/d(u_h), q = phi dF/d(inner derivative) and
// r_a = phi dF/d(aux_h); a position's adjoint is the transposed interpolation and difference of the
// half points around it, and what the boundary and extrapolated positions get goes back to the
// nodes they are made of.  Columns within three of a side see its half points: faces -2 .. TX + 1
// of the tile are evaluated, from a halo of three positions below and four above.  Along z a half
// point adds to the sums of its four planes, which a thread holds open: plane c is finished when
// half point c + 1 is in.  Sums in FP64.
template <class G>
struct MolFluxAdj {   // what a half point leaves
  T p, q, r[G::NAH > 0 ? G::NAH : 1];
};
template <class G>
struct MolFluxVLds {
  static constexpr int LX = G::TX + 7, LY = G::TY + 7, NA = 1 + G::NAH, NC = G::TX * G::TY;
  static constexpr int FXN = (G::TX + 4) * G::TY, FYN = G::TX * (G::TY + 4), NR = 2 + G::NAH;
  T L[NA + 1][LX * LY];   // staged arrays, then the seed
  T FX[NR][FXN], FY[NR][FYN];
};

template <class G, int AX>
__device__ __forceinline__ MolFluxAdj<G> mol_flux_rev(const T (&w)[4][1 + G::NAH], const T l0, const T l1,
                                                      const double t, const T* __restrict__ P) {
  T h[1 + G::NAH], d;
  mol_flux_half<G>(AX, w, h, d);
  T phi = G::wo(AX, 1) * l0;
  phi += G::wo(AX, 0) * l1;
  MolFluxAdj<G> o;
  G::template dflux<AX>(h, d, phi * G::ws(AX), t, P, o.p, o.r, o.q);
  return o;
}

// Adjoint of position j along an axis from the half points j - 2 .. j + 1 (f[0] .. f[3]): of the
// state (R < 0) or of grid field R.
template <class G, int R>
__device__ __forceinline__ double mol_flux_tr(const int ax, const MolFluxAdj<G> (&f)[4]) {
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i) s += (double)G::wi(ax, 3 - i) * (double)(R < 0 ? f[i].p : f[i].r[R < 0 ? 0 : R]);
  if (R < 0) {
    s += (double)G::wd(ax, 0) * (double)f[2].q;
    s += (double)G::wd(ax, 1) * (double)f[1].q;
  }
  return s;
}

// One side's part of a node at distance m (0 .. 2) from it: e0, e1 the side's own half point and the
// next one inside; edge(a, value): the gradient of a grid field at the boundary node.
template <class G, int AX, int SIDE, class EDGE>
__device__ __forceinline__ void mol_flux_back(const int m, const MolFluxAdj<G>& e0, const MolFluxAdj<G>& e1, double& ub,
                                              double (&da)[G::NAH > 0 ? G::NAH : 1], const bool ga, const EDGE& edge) {
  MolFluxAdj<G> f[4] = {};
  f[SIDE == 0 ? 2 : 1] = e0;
  f[SIDE == 0 ? 3 : 0] = e1;
  const double we = (double)G::wi(AX, SIDE == 0 ? 0 : 3);
  auto pick = [&](const T a, const T b, const T c) { return (double)(m == 0 ? a : (m == 1 ? b : c)); };
  ub += pick(G::closure(AX, SIDE, 0, 0), G::closure(AX, SIDE, 0, 1), G::closure(AX, SIDE, 0, 2)) * mol_flux_tr<G, -1>(AX, f) +
        pick(G::closure(AX, SIDE, 1, 0), G::closure(AX, SIDE, 1, 1), G::closure(AX, SIDE, 1, 2)) * (we * (double)e0.p);
  if (ga) {
    const double ex = pick(G::ext(AX, SIDE, 1), G::ext(AX, SIDE, 2), G::ext(AX, SIDE, 3));
    if constexpr (G::NAH > 0) {
      const double v = we * (double)e0.r[0];
      da[0] += ex * v;
      if (m == 0) edge(0, mol_flux_tr<G, 0>(AX, f) + (double)G::ext(AX, SIDE, 0) * v);
    }
    if constexpr (G::NAH > 1) {
      const double v = we * (double)e0.r[1];
      da[1] += ex * v;
      if (m == 0) edge(1, mol_flux_tr<G, 1>(AX, f) + (double)G::ext(AX, SIDE, 0) * v);
    }
  }
}

// The part of the x or y axis of a node at coordinate v of M: at(i) returns half point v + i, -2 <= i <= 2
// (zero outside -1 .. M-1); edge(side, a, value): the gradient of a grid field at a boundary node.
template <class G, int AX, class AT, class EDGE>
__device__ __forceinline__ void mol_flux_axis(const int v, const AT& at, double& ub,
                                              double (&da)[G::NAH > 0 ? G::NAH : 1], const bool ga, const EDGE& edge) {
  constexpr int M = AX == 0 ? G::M0 : G::M1;
  {
    const MolFluxAdj<G> f[4] = {at(-2), at(-1), at(0), at(1)};
    ub += mol_flux_tr<G, -1>(AX, f);
    if (ga) {
      if constexpr (G::NAH > 0) da[0] += mol_flux_tr<G, 0>(AX, f);
      if constexpr (G::NAH > 1) da[1] += mol_flux_tr<G, 1>(AX, f);
    }
  }
  if (v <= 2)
    mol_flux_back<G, AX, 0>(v, at(-1 - v), at(-v), ub, da, ga, [&](const int a, const double x) { edge(0, a, x); });
  if (M - 1 - v <= 2)
    mol_flux_back<G, AX, 1>(M - 1 - v, at(M - 1 - v), at(M - 2 - v), ub, da, ga,
                            [&](const int a, const double x) { edge(1, a, x); });
}

template <class G>
__device__ __forceinline__ void mol_flux_vjp(MolFluxVLds<G>& S, const VArgs& va, const JPtrs& jp, const double t) {
  typedef MolFluxVLds<G> Q;
  typedef MolFluxAdj<G> F;
  constexpr int TX = G::TX, TY = G::TY, NA = Q::NA, NI = Q::NC / G::NTHR, NH = 7 * (TX + TY);
  constexpr int NHI = (NH + G::NTHR - 1) / G::NTHR, NAD = G::NAH > 0 ? G::NAH : 1, NQ = G::NAU > 0 ? G::NAU : 1;
  constexpr int NAG = G::NAG > 0 ? G::NAG : 1;
  constexpr i64 PU = (i64)G::M0 * G::M1, PA = (i64)G::N0 * G::N1;
  const int b = mol_xcd_tile<G::NBLK>((int)blockIdx.x);
  const int X0 = (b % G::NT0) * TX, Y0 = (b / G::NT0 % G::NT1) * TY, zc = b / (G::NT0 * G::NT1);
  const int z0 = mol_flux_chunk<G>(zc), z1 = mol_flux_chunk<G>(zc + 1);
  const T* const P = va.p;
  const T* const u = va.u;
  const bool ga = va.g_aux != nullptr, sum = (va.mode & 8) != 0;
  // seed at plane z: its two parts as loaded, then put together (0 outside)
  const T* const s2 = va.s2 ? va.s2 : va.s1;
  auto raw = [&](T (&v)[2], const MolFluxCol<G>& c, const int z) {
    const i64 o = PU * mol_uniform(min(max(z, 0), G::M2 - 1));
    v[0] = mol_at_s(va.s1 + o, c.u);
    v[1] = mol_at_s(s2 + o, c.u);
  };
  auto seed = [&](const T (&v)[2], const bool in, const int z) {
    const T a = (T)va.c1 * v[0], b = a + (T)va.c2 * v[1];
    return in && z >= 0 && z < G::M2 ? (va.s2 ? b : a) : T(0);
  };
  // a column's planes c .. c+3, seeds and open sums c .. c+2 (and c+3 with half point c+1); the halo
  // of plane c
  T R[NI][4][NA], Ls[NI][3], hv[NHI][NA], hs[NHI][2];
  double ub[NI][4], da[NI][4][NAD];
  int cx[NI], cy[NI], ho[NHI];
  MolFluxCol<G> col[NI], hc[NHI];
  bool in[NI], hin[NHI];
  auto halo = [&](const int c) {
#pragma unroll
    for (int i = 0; i < NHI; ++i) {
      mol_flux_load<G, true>(hv[i], hc[i], u, jp, c);
      raw(hs[i], hc[i], c);
    }
  };
#pragma unroll
  for (int i = 0; i < NHI; ++i) {
    int x, y;
    mol_flux_halo<G, 3, 4>(min((int)threadIdx.x + i * G::NTHR, NH - 1), x, y);
    hc[i].at(X0 + x, Y0 + y);
    ho[i] = (x + 3) + Q::LX * (y + 3);
    hin[i] = X0 + x >= 0 && X0 + x < G::M0 && Y0 + y >= 0 && Y0 + y < G::M1;
  }
  halo(z0);
  // adds to the gradient of the a-th interpolated field at a boundary node
  auto edge = [&](const int a, const int px, const int py, const int pz, const double v) {
    va.g_aux[G::AH[a] * G::NGRID + (i64)(px + 1) + (i64)G::N0 * ((py + 1) + (i64)G::N1 * (pz + 1))] += v;
  };
  // half point between open planes J + 1 and J + 2 along z into the sums J .. J + 3 (those there are)
  auto push = [&](const int k, const F& f, const int J) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (J + i < 0) continue;
      ub[k][J + i] += (double)G::wi(2, i) * (double)f.p;
      if (i == 1 || i == 2) ub[k][J + i] += (double)G::wd(2, i - 1) * (double)f.q;
#pragma unroll
      for (int a = 0; a < G::NAH; ++a) da[k][J + i][a] += (double)G::wi(2, i) * (double)f.r[a];
    }
  };
#pragma unroll
  for (int k = 0; k < NI; ++k) {
    const int q = (int)threadIdx.x + k * G::NTHR;
    cy[k] = q / TX;
    cx[k] = q - cy[k] * TX;
    const int x = X0 + cx[k], y = Y0 + cy[k];
    in[k] = x < G::M0 && y < G::M1;
    col[k].at(x, y);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ub[k][i] = 0.0;
#pragma unroll
      for (int a = 0; a < NAD; ++a) da[k][i][a] = 0.0;
    }
    // planes z0-3 .. z0+3, half points z0-2 .. z0
    T v[7][NA], lr[5][2], l[5];
    F f[3];
#pragma unroll
    for (int i = 0; i < 5; ++i) raw(lr[i], col[k], z0 - 2 + i);
    mol_flux_planes<G, 7, 3, true>(v, col[k], x, y, z0, u, jp, t, P);
#pragma unroll
    for (int i = 0; i < 5; ++i) l[i] = seed(lr[i], in[k], z0 - 2 + i);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      T w[4][NA];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int a = 0; a < NA; ++a) w[j][a] = v[i + j][a];
      f[i] = mol_flux_rev<G, 2>(w, l[i], l[i + 1], t, P);
      if (i == 0 && z0 == 0) f[i] = F{};   // (outside)
      push(k, f[i], i - 3);
      Ls[k][i] = l[2 + i];
    }
    if (z0 == 0 && in[k])
#pragma unroll
      for (int m = 0; m < 3; ++m)
        mol_flux_back<G, 2, 0>(m, f[1], f[2], ub[k][m], da[k][m], ga,
                               [&](const int a, const double e) { edge(a, x, y, -1, e); });
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int a = 0; a < NA; ++a) R[k][i][a] = v[3 + i][a];
  }
  // plane c into LDS: the columns' plane R[.][I] and the halo that was loaded
  auto stage = [&](const int I, const int c) {
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      const int o = (cx[k] + 3) + Q::LX * (cy[k] + 3);
#pragma unroll
      for (int a = 0; a < NA; ++a) S.L[a][o] = R[k][I][a];
      S.L[NA][o] = Ls[k][I];
    }
#pragma unroll
    for (int i = 0; i < NHI; ++i) {
#pragma unroll
      for (int a = 0; a < NA; ++a) S.L[a][ho[i]] = hv[i][a];
      S.L[NA][ho[i]] = seed(hs[i], hin[i], c);
    }
  };
  auto ag = [&](const int k) { return col[k].a * (unsigned)(sizeof(double) / sizeof(T)); };
  stage(0, z0);
  // (four planes in a row: the open sums and planes change names instead of registers; 198^3 197 ->
  // 191 us, 98^3 32.0 -> 30.1, 48^3 14.2 -> 13.2, 126^3 even)
#pragma unroll 4
  for (int c = z0; c < z1; ++c) {
    // in flight during the half points: the next plane, the node's fields, the sums to add to
    T nxt[NI][NA], nl[NI][2], av[NI][NQ], ys[NI][4];
    double gv[NI][NAG];
    const i64 pu = PU * mol_uniform(c), pa = PA * mol_uniform(c + 1);
    halo(c + 1);
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      mol_flux_load<G, true>(nxt[k], col[k], u, jp, c + 4);
      raw(nl[k], col[k], c + 3);
#pragma unroll
      for (int a = 0; a < G::NAU; ++a) av[k][a] = mol_at_s(jp.aux[G::AN[a]] + pa, col[k].a);
      if (sum) {
        ys[k][0] = mol_at_s((const T*)va.lam + pu, col[k].u);
        ys[k][1] = mol_at_s(va.y0 + pu, col[k].u);
        ys[k][2] = mol_at_s(va.y1 + pu, col[k].u);
        ys[k][3] = mol_at_s(va.y2 + pu, col[k].u);
      }
      if (ga) {
#pragma unroll
        for (int a = 0; a < G::NAG; ++a) gv[k][a] = mol_at_s((const double*)va.g_aux + G::AG[a] * G::NGRID + pa, ag(k));
      }
    }
    __syncthreads();
    mol_flux_sides<G, 3, 4, Q::LX>(&S.L[0][0], Q::LX * Q::LY, X0, Y0, c, t, P, jp);
    // half points of the plane along x and y: every column's upper sides, and faces -2, -1, TX,
    // TX + 1 of the tile's rows and columns
    auto face = [&](const int ax, const int x, const int y) {
      const int o = (x + 3) + Q::LX * (y + 3), st = ax == 0 ? 1 : Q::LX;
      const int h = ax == 0 ? X0 + x : Y0 + y;
      T w[4][NA];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int a = 0; a < NA; ++a) w[i][a] = S.L[a][o + (i - 1) * st];
      F f = ax == 0 ? mol_flux_rev<G, 0>(w, S.L[NA][o], S.L[NA][o + st], t, P)
                    : mol_flux_rev<G, 1>(w, S.L[NA][o], S.L[NA][o + st], t, P);
      if (h < -1 || h >= (ax == 0 ? G::M0 : G::M1)) f = F{};
      T* const B = ax == 0 ? &S.FX[0][(x + 2) + (TX + 4) * y] : &S.FY[0][x + TX * (y + 2)];
      const int N = ax == 0 ? Q::FXN : Q::FYN;
      B[0] = f.p;
      B[N] = f.q;
#pragma unroll
      for (int a = 0; a < G::NAH; ++a) B[(2 + a) * N] = f.r[a];
    };
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      face(0, cx[k], cy[k]);
      face(1, cx[k], cy[k]);
    }
    for (int q = (int)threadIdx.x; q < 4 * (TX + TY); q += G::NTHR) {
      int x, y;
      mol_flux_halo<G, 2, 2>(q, x, y);
      if (q < 4 * TY) face(0, x, y);
      else face(1, x, y);
    }
    __syncthreads();
    stage(1, c + 1);   // (before this plane's stores: the wait for its halo is not one for them)
    const int g = c + 4 - G::M2;
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      const int x = X0 + cx[k], y = Y0 + cy[k];
      if (g == 0 || g == 1) {
        const T bv = mol_flux_bval<G>(2, 1, x, y, G::M2, t, P, jp);
        mol_flux_above<G>(nxt[k], R[k][0], R[k][1], R[k][2], R[k][3], g, bv);
      }
      // along z: half point c + 1; before plane M2 - 3 is finished what its side gives back
      if (c + 1 < G::M2) {
        const F f = mol_flux_rev<G, 2>(R[k], Ls[k][1], Ls[k][2], t, P);
        push(k, f, 0);
        if (c == G::M2 - 3 && in[k]) {
          T w[4][NA];
#pragma unroll
          for (int a = 0; a < NA; ++a) {
            w[0][a] = R[k][1][a];
            w[1][a] = R[k][2][a];
            w[2][a] = R[k][3][a];
            w[3][a] = nxt[k][a];
          }
          const F e = mol_flux_rev<G, 2>(w, Ls[k][2], T(0), t, P);
#pragma unroll
          for (int m = 0; m < 3; ++m)
            mol_flux_back<G, 2, 1>(m, e, f, ub[k][2 - m], da[k][2 - m], ga,
                                   [&](const int a, const double v) { edge(a, x, y, G::M2, v); });
        }
      }
      if (in[k]) {
        double dg[NAG] = {};
        auto from = [&](const T* const B, const int N) {
          F f;
          f.p = B[0];
          f.q = B[N];
#pragma unroll
          for (int a = 0; a < NAD; ++a) f.r[a] = a < G::NAH ? B[(2 + a) * N] : T(0);
          return f;
        };
        mol_flux_axis<G, 0>(x, [&](const int i) { return from(&S.FX[0][cx[k] + 2 + i + (TX + 4) * cy[k]], Q::FXN); },
                            ub[k][0], da[k][0], ga,
                            [&](const int side, const int a, const double v) { edge(a, side ? G::M0 : -1, y, c, v); });
        mol_flux_axis<G, 1>(y, [&](const int i) { return from(&S.FY[0][cx[k] + TX * (cy[k] + 2 + i)], Q::FYN); },
                            ub[k][0], da[k][0], ga,
                            [&](const int side, const int a, const double v) { edge(a, x, side ? G::M1 : -1, c, v); });
        // the node's own terms
        G::dnode(R[k][0][0], Ls[k][0], av[k], x + 2, y + 2, c + 2, t, P, jp, ub[k][0], dg);
        if (ga) {
#pragma unroll
          for (int a = 0; a < G::NAH; ++a) dg[G::HG[a]] += da[k][0][a];
#pragma unroll
          for (int a = 0; a < G::NAG; ++a)
            mol_at_s(va.g_aux + G::AG[a] * G::NGRID + pa, ag(k)) = gv[k][a] + dg[a];
        }
        mol_at_s(va.out + pu, col[k].u) = sum ? (((ys[k][0] + ys[k][1]) + ys[k][2]) + ys[k][3]) + (T)ub[k][0] : (T)ub[k][0];
      }
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        R[k][0][a] = R[k][1][a];
        R[k][1][a] = R[k][2][a];
        R[k][2][a] = R[k][3][a];
        R[k][3][a] = nxt[k][a];
      }
      Ls[k][0] = Ls[k][1];
      Ls[k][1] = Ls[k][2];
      Ls[k][2] = seed(nl[k], in[k], c + 3);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ub[k][i] = i < 3 ? ub[k][i < 3 ? i + 1 : 0] : 0.0;
#pragma unroll
        for (int a = 0; a < NAD; ++a) da[k][i][a] = i < 3 ? da[k][i < 3 ? i + 1 : 0][a] : 0.0;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------
// Batched instances.  Each instance of a batch has a header with its grid sizes, unknown
// boxes (offsets into the batch state vector), tile counts and tile classes, and pointers to
// its weight pool W (the descriptor's pool), constants K (the constant pool, then eps and
// 1/dx of every slot) and coordinates.  Instances of one structure share a class body
// (struct with the node function); a persistent kernel walks the work list of (instance, tile)
// items and dispatches on the class.  Layout identical to mol::BInst.
struct BInst {
  int n[3];
  int lo[8][3];
  int hi[8][3];
  i64 fofs[8];
  int ulo[3], uhi[3], nt[3];
  int slo[3], shi[3], clo[3], chi[3];
  int ilo[3], ihi[3];   // nodes where the interior-rows code applies
  int cls, first;
  const double* coord[3];
  const double* W;
  const double* K;
  double g[8][4][3];    // per variable and side of the first two axes (x low, x high, y low, y high): the ghost
                        // next to the box as factors of the two nodes next to the side and of G
};

// Index of node (p0, p1, p2) of variable f in the batch state: the instance's offset plus a
// 32-bit offset inside the variable's box (each box holds fewer than 2^31 unknowns).
__device__ __forceinline__ i64 mol_b_uidx(const BInst& hd, const int f, const int p0, const int p1, const int p2) {
  return hd.fofs[f] + (i64)((p0 - hd.lo[f][0]) +
                            (hd.hi[f][0] - hd.lo[f][0] + 1) *
                                ((p1 - hd.lo[f][1]) + (hd.hi[f][1] - hd.lo[f][1] + 1) * (p2 - hd.lo[f][2])));
}

__device__ __forceinline__ bool mol_b_inbox(const BInst& hd, const int f, const int I0, const int I1, const int I2) {
  return I0 >= hd.lo[f][0] && I0 <= hd.hi[f][0] && I1 >= hd.lo[f][1] && I1 <= hd.hi[f][1] && I2 >= hd.lo[f][2] &&
         I2 <= hd.hi[f][2];
}

// Position walker over a box of run-time extents (x fastest), advanced by the work-group's
// thread count: one division per axis when a tile starts, none per position.
// Positions of a box of run-time extents (x fastest), visited by the threads of a work-group
// with stride NTHR: one division per axis when a walk starts, none per position.  Z: the box
// has more than one plane.
template <bool Z>
struct MolRtWalk {
  int x, y, z, dx, dy, dz, ex, ey;
  __device__ __forceinline__ MolRtWalk(const int q, const int ex_, const int ey_, const int stride) : ex(ex_), ey(ey_) {
    if constexpr (Z) {
      const int exy = ex * ey;
      z = q / exy;
      const int r = q - z * exy;
      y = r / ex;
      x = r - y * ex;
      dz = stride / exy;
      const int rs = stride - dz * exy;
      dy = rs / ex;
      dx = rs - dy * ex;
    } else {
      z = dz = 0;
      y = q / ex;
      x = q - y * ex;
      dy = stride / ex;
      dx = stride - dy * ex;
    }
  }
  __device__ __forceinline__ void step() {
    x += dx;
    y += dy;
    if (x >= ex) { x -= ex; ++y; }
    if constexpr (Z) {
      z += dz;
      if (y >= ey) { y -= ey; ++z; }
    }
  }
};

// Inclusive integer box.
struct MolBox {
  int lo[3], hi[3];
  __device__ __forceinline__ bool empty() const { return hi[0] < lo[0] || hi[1] < lo[1] || hi[2] < lo[2]; }
  __device__ __forceinline__ int ext(const int a) const { return hi[a] - lo[a] + 1; }
  __device__ __forceinline__ int vol() const { return ext(0) * ext(1) * ext(2); }
  __device__ __forceinline__ MolBox meet(const MolBox& o) const {
    MolBox m;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      m.lo[a] = max(lo[a], o.lo[a]);
      m.hi[a] = min(hi[a], o.hi[a]);
    }
    return m;
  }
};

// The positions of box B outside its sub-box A (A non-empty), as up to six slabs: below and
// above A along z (whole planes of B), then along y (within A's planes), then along x (within
// A's rows).  count(): their number; at(k): the k-th position.
struct MolFrame {
  MolBox B, A;
  int n[6];
  __device__ __forceinline__ MolFrame(const MolBox& b, const MolBox& a) : B(b), A(a) {
    const int ex = B.ext(0), ey = B.ext(1), ay = A.ext(1), az = A.ext(2);
    n[0] = (A.lo[2] - B.lo[2]) * ex * ey;
    n[1] = (B.hi[2] - A.hi[2]) * ex * ey;
    n[2] = (A.lo[1] - B.lo[1]) * ex * az;
    n[3] = (B.hi[1] - A.hi[1]) * ex * az;
    n[4] = (A.lo[0] - B.lo[0]) * ay * az;
    n[5] = (B.hi[0] - A.hi[0]) * ay * az;
  }
  __device__ __forceinline__ int count() const { return n[0] + n[1] + n[2] + n[3] + n[4] + n[5]; }
  __device__ __forceinline__ void at(int k, int& p0, int& p1, int& p2) const {
    const int ex = B.ext(0), ey = B.ext(1);
    int s = 0;
    while (s < 5 && k >= n[s]) k -= n[s++];
    if (s < 2) {   // planes of B
      const int exy = ex * ey, pz = k / exy, r = k - pz * exy, py = r / ex;
      p2 = (s == 0 ? B.lo[2] : A.hi[2] + 1) + pz;
      p1 = B.lo[1] + py;
      p0 = B.lo[0] + (r - py * ex);
    } else if (s < 4) {   // rows of B within A's planes
      const int w = (s == 2 ? A.lo[1] - B.lo[1] : B.hi[1] - A.hi[1]);
      const int pz = k / (ex * w), r = k - pz * ex * w, py = r / ex;
      p2 = A.lo[2] + pz;
      p1 = (s == 2 ? B.lo[1] : A.hi[1] + 1) + py;
      p0 = B.lo[0] + (r - py * ex);
    } else {   // columns within A's rows
      const int w = (s == 4 ? A.lo[0] - B.lo[0] : B.hi[0] - A.hi[0]), ay = A.ext(1);
      const int pz = k / (w * ay), r = k - pz * w * ay, py = r / w;
      p2 = A.lo[2] + pz;
      p1 = A.lo[1] + py;
      p0 = (s == 4 ? B.lo[0] : A.hi[0] + 1) + (r - py * w);
    }
  }
};

// Position inside every variable's unknown box.
template <int NF>
__device__ __forceinline__ bool mol_b_inall(const BInst& hd, const int p0, const int p1, const int p2) {
  bool in = true;
#pragma unroll
  for (int f = 0; f < NF; ++f) in = in && mol_b_inbox(hd, f, p0, p1, p2);
  return in;
}

// One node of a batched tile whose LDS box starts at (s0, s1, s2), and its stage epilogue.
// INTERIOR: the interior-rows code, at a node inside every variable's box.
template <class G, bool INTERIOR>
__device__ __forceinline__ void mol_batch_node(const T* L, const BInst& hd, const int I0, const int I1, const int I2,
                                               const int s0, const int s1, const int s2, const T* __restrict__ u,
                                               const Epi& ep, const JPtrs& jp, const double t) {
  const int base = (I0 - s0) + G::EX * ((I1 - s1) + G::EY * (I2 - s2));
  T out[G::NF];
  G::template node<INTERIOR>(hd, L, base, I0, I1, I2, t, nullptr, u, jp, out);
#pragma unroll
  for (int f = 0; f < G::NF; ++f)
    if (INTERIOR || mol_b_inbox(hd, f, I0, I1, I2)) mol_epilogue(ep, mol_b_uidx(hd, f, I0, I1, I2), out[f]);
}

// One tile of one instance (L: the kernel's LDS tile, sized for the largest class).  Only the
// part of the tile inside the instance's union box is staged and evaluated, so tiles at least
// as wide as an instance cover whole rows of it (contiguous in memory: staging loads and the
// epilogue touch no cache line of another row) and narrow instances leave no idle lanes in a
// wide tile.  Staging: plain loads where the tile + halo lies inside every variable's box,
// the ghost closures (and periodic images) on the frame around it.  Nodes: the interior-rows
// code inside the instance's interior node range, the boundary-rows code on the frame around it.
template <class G>
__device__ __forceinline__ void mol_batch_tile(T* L, const BInst& hd, const int tile, const T* __restrict__ u,
                                               const Epi& ep, const double t) {
  constexpr bool Z = G::TZ > 1 || G::HZ > 0;
  const int tx = tile % hd.nt[0];
  const int r1 = tile / hd.nt[0];
  const int ty = r1 % hd.nt[1];
  const int tz = r1 / hd.nt[1];
  MolBox N;   // the tile's nodes inside the union box
  N.lo[0] = hd.ulo[0] + tx * G::TX;
  N.lo[1] = hd.ulo[1] + ty * G::TY;
  N.lo[2] = hd.ulo[2] + tz * G::TZ;
  N.hi[0] = min(N.lo[0] + G::TX - 1, hd.uhi[0]);
  N.hi[1] = min(N.lo[1] + G::TY - 1, hd.uhi[1]);
  N.hi[2] = min(N.lo[2] + G::TZ - 1, hd.uhi[2]);
  MolBox S = N;   // with the halo: the LDS box
  S.lo[0] -= G::HX; S.hi[0] += G::HX;
  S.lo[1] -= G::HY; S.hi[1] += G::HY;
  S.lo[2] -= G::HZ; S.hi[2] += G::HZ;
  JPtrs jp;
  jp.coord[0] = hd.coord[0];
  jp.coord[1] = hd.coord[1];
  jp.coord[2] = hd.coord[2];
  if constexpr (G::NST > 0) {
    MolBox V = S;   // inside every variable's box: plain loads
#pragma unroll
    for (int f = 0; f < G::NF; ++f) {
      MolBox bf;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        bf.lo[a] = hd.lo[f][a];
        bf.hi[a] = hd.hi[f][a];
      }
      V = V.meet(bf);
    }
    constexpr int IT = (G::VOL + G::NTHR - 1) / G::NTHR;
    constexpr int NS = G::NST > 0 ? G::NST : 1;
    if (!V.empty()) {
      // variable boxes and the first plain position, per staged slot
      i64 vb[NS];
      int sx[NS], sxy[NS];
#pragma unroll
      for (int s = 0; s < G::NST; ++s) {
        const int f = G::SF[s];
        sx[s] = hd.hi[f][0] - hd.lo[f][0] + 1;
        sxy[s] = sx[s] * (hd.hi[f][1] - hd.lo[f][1] + 1);
        vb[s] = mol_b_uidx(hd, f, V.lo[0], V.lo[1], V.lo[2]);
      }
      const int nv = V.vol();
      const int lofs = (V.lo[0] - S.lo[0]) + G::EX * ((V.lo[1] - S.lo[1]) + G::EY * (V.lo[2] - S.lo[2]));
      MolRtWalk<Z> w((int)threadIdx.x, V.ext(0), V.ext(1), G::NTHR);
      // chunks of CH positions per thread: all loads of a chunk are issued before its LDS
      // stores (one exposed memory latency per chunk, not per position)
      constexpr int CH = IT * G::NST <= 16 ? IT : (16 / G::NST > 0 ? 16 / G::NST : 1);
      for (int q0 = (int)threadIdx.x; q0 < nv; q0 += CH * G::NTHR) {
        T v[CH][NS];
        int dst[CH];
#pragma unroll
        for (int k = 0; k < CH; ++k, w.step()) {
          dst[k] = q0 + k * G::NTHR < nv ? lofs + w.x + G::EX * (w.y + G::EY * w.z) : -1;
          if (dst[k] >= 0)
#pragma unroll
            for (int s = 0; s < G::NST; ++s) v[k][s] = u[vb[s] + (w.x + sx[s] * w.y + sxy[s] * w.z)];
        }
#pragma unroll
        for (int k = 0; k < CH; ++k)
          if (dst[k] >= 0)
#pragma unroll
            for (int s = 0; s < G::NST; ++s) L[s * G::VOL + dst[k]] = v[k][s];
      }
    }
    // the frame of ghost positions and periodic images (everything when nothing is plain)
    const MolFrame F(S, V.empty() ? S : V);
    const int nf = V.empty() ? S.vol() : F.count();
    for (int q = threadIdx.x; q < nf; q += G::NTHR) {
      int p0, p1, p2;
      if (V.empty()) {
        const int e0 = S.ext(0), e1 = S.ext(1), pz = q / (e0 * e1), r = q - pz * e0 * e1, py = r / e0;
        p0 = S.lo[0] + (r - py * e0);
        p1 = S.lo[1] + py;
        p2 = S.lo[2] + pz;
      } else {
        F.at(q, p0, p1, p2);
      }
      T v[NS];
      G::stage_vals(hd, v, p0, p1, p2, false, t, nullptr, u, jp);
      const int d = (p0 - S.lo[0]) + G::EX * ((p1 - S.lo[1]) + G::EY * (p2 - S.lo[2]));
#pragma unroll
      for (int s = 0; s < G::NST; ++s) L[s * G::VOL + d] = v[s];
    }
    __syncthreads();
  }
  MolBox I;   // nodes where the interior-rows code applies
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    I.lo[a] = hd.ilo[a];
    I.hi[a] = hd.ihi[a];
  }
  I = I.meet(N);
  if (!I.empty()) {
    // interior nodes lie in every variable's box (the interior range is empty otherwise), so
    // the variables' indices differ by their offsets only; chunks of CN nodes per thread share
    // one exposed latency of the epilogue's loads
    constexpr int CN = 4;
    i64 dv[G::NF];
#pragma unroll
    for (int f = 0; f < G::NF; ++f) dv[f] = hd.fofs[f] - hd.fofs[0];
    const int ni = I.vol();
    MolRtWalk<Z> w((int)threadIdx.x, I.ext(0), I.ext(1), G::NTHR);
    for (int q0 = (int)threadIdx.x; q0 < ni; q0 += CN * G::NTHR) {
      T out[CN][G::NF];
      i64 idx[CN];
      bool ok[CN];
#pragma unroll
      for (int k = 0; k < CN; ++k, w.step()) {
        ok[k] = q0 + k * G::NTHR < ni;
        idx[k] = 0;
        if (!ok[k]) continue;
        const int I0 = I.lo[0] + w.x, I1 = I.lo[1] + w.y, I2 = I.lo[2] + w.z;
        const int base = (I0 - S.lo[0]) + G::EX * ((I1 - S.lo[1]) + G::EY * (I2 - S.lo[2]));
        G::template node<true>(hd, L, base, I0, I1, I2, t, nullptr, u, jp, out[k]);
        idx[k] = mol_b_uidx(hd, 0, I0, I1, I2);
      }
      mol_epilogue_chunk<CN, G::NF>(ep, idx, ok, dv, out);
    }
    const MolFrame F(N, I);
    const int nf = F.count();
    for (int q = threadIdx.x; q < nf; q += G::NTHR) {
      int p0, p1, p2;
      F.at(q, p0, p1, p2);
      mol_batch_node<G, false>(L, hd, p0, p1, p2, S.lo[0], S.lo[1], S.lo[2], u, ep, jp, t);
    }
  } else {
    const int nn = N.vol();
    MolRtWalk<Z> w((int)threadIdx.x, N.ext(0), N.ext(1), G::NTHR);
    for (int q = threadIdx.x; q < nn; q += G::NTHR, w.step())
      mol_batch_node<G, false>(L, hd, N.lo[0] + w.x, N.lo[1] + w.y, N.lo[2] + w.z, S.lo[0], S.lo[1], S.lo[2], u,
                               ep, jp, t);
  }
  __syncthreads();
}
