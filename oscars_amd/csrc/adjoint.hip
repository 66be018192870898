// Reverse pass (adjoint) of frozen-level flux values with respect to the
// samples of one grid field and the particle's initial position and velocity.
//
// Forward chain, restated from the reference (paths relative to its root):
//   flux  F = C2 |C0 dt_L S|^2,  S = sum_j A_j exp(i phi_j)      src/OSCARSSR.cc:4179-4245 (fixed level L)
//   level samples s_j = spline(t_j)                              include/TOMATH.h:92-126
//   spline second derivatives from the knots                     include/TOMATH.h:141-203
//   knots = RK4 states, acceleration stored one step late        src/OSCARSSR.cc:910-1009, 1321-1386
//   field = linear interpolation of grid samples                 src/TField3D_Grid.cc:153-278
// Each kernel below applies the transpose of the derivative of one stage.
//
// RK4 reverse with checkpoints: the forward keeps the state every K = ceil(sqrt(N))
// steps.  The adjoint state obeys the affine recurrence
//   lambda_i = J_i^T lambda_{i+1} + c_i
// (J_i the Jacobian of step i, c_i the direct knot terms).  Segments of K steps
// are independent given their checkpoint, so
//   A: each segment recomputes its states and composes its own affine map
//      lambda_{i0} = M lambda_{i1} + b (tangents through the four RK4 stages),
//   B: one thread chains the sqrt(N) segment maps from the end,
//   C: each segment recomputes its states again and sweeps back from its
//      lambda_{i1}, writing each field evaluation's grid-sample gradient as
//      records in fixed slots; the records are sorted stably by sample and
//      summed per sample in record order (bit-for-bit reproducible).
// The sequential depth is about 3 K steps instead of 3 N.
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/iterator/counting_iterator.hpp>

#include "adj_types.h"
#include "lw_common.h"
#include "rk4_common.h"

namespace om {

// ---------------------------------------------------------------- checkpoints
// Raw knots (before the division of velocity and acceleration by c) hold the
// RK4 state of every forward step; keep every K-th one in state order.
__global__ void __launch_bounds__(256) adj_ckpt_kernel(const double* __restrict__ p_raw, long K, long nseg,
                                                       double* __restrict__ ckpt) {
  long s = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg) return;
  const double* o = p_raw + 9 * (s * K);
  double* c = ckpt + 6 * s;
  c[0] = o[0]; c[1] = o[3];
  c[2] = o[1]; c[3] = o[4];
  c[4] = o[2]; c[5] = o[5];
}

// ---------------------------------------------------------------- LW sum
__device__ __forceinline__ V3 vscale(V3 a, double s) { return v3(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ V3 vadd(V3 a, V3 b) { return v3(a.x + b.x, a.y + b.y, a.z + b.z); }

// One thread per trajectory sample, a chunk of observation points per
// workgroup row.  With S_k += A_k (cos phi + i sin phi), phi = -w tau, the
// energy loop of one point accumulates
//   P_k = sum_w (gr_k cos phi + gi_k sin phi)              = dLoss/dA_k
//   Q   = sum_w (-w) sum_k A_k (gi_k cos phi - gr_k sin phi) = dLoss/dtau
// and the amplitude A(x, beta, a) and tau = t + D/c are then differentiated by hand.
// Bound by FP64 issue.  The phase, N, W and k are formed as the forward forms
// them; the divisors D and k are inverted once (15 divisions a point and sample
// were 7 too many), and four energies' sines and cosines go side by side.
// 8191 samples, 2601 points, 4 energies: 749 -> 396 us.
__global__ void __launch_bounds__(256) adj_lw_kernel(AdjLwArgs A) {
  long j = (long) blockIdx.x * blockDim.x + threadIdx.x;
  long o0 = (long) blockIdx.y * A.obs_per_chunk;
  long o1 = o0 + A.obs_per_chunk < A.n_obs ? o0 + A.obs_per_chunk : A.n_obs;
  bool valid = j < A.ns;
  const double* s = A.rows + 10 * (valid ? j : A.ns - 1);
  double t = s[0];
  V3 X = v3(s[1], s[2], s[3]);
  V3 Bt = v3(s[4], s[5], s[6]);
  V3 Ac = v3(s[7], s[8], s[9]);
  double b2 = mag2(Bt);
  double gx[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (long o = o0; o < o1; ++o) {
    V3 ob = v3(A.obs[3 * o], A.obs[3 * o + 1], A.obs[3 * o + 2]);
    V3 R = sub(ob, X);
    double D = sqrt(mag2(R));
    V3 N = v3(R.x / D, R.y / D, R.z / D);
    V3 W = sub(N, Bt);
    double k = 1 - dot(N, Bt);
    // reciprocals of D and k: d1 = D^2 k^2, d2 = D k^2 of the integrand
    const double iD = 1.0 / D, ik = 1.0 / k;
    const double i2 = iD * ik * ik, i1 = i2 * iD;
    V3 Y = cross(W, Ac);
    V3 NY = cross(N, Y);
    V3 Am = vadd(vscale(W, (1 - b2) * i1), vscale(NY, i2));
    double tau = t + D / kC;
    V3 P = v3(0, 0, 0);
    double Q = 0;
    const double* go = A.g + 6 * A.n_e * o;
    auto add = [&](const double* ge, double w, double sn, double cs) {
      P.x = __builtin_fma(ge[0], cs, __builtin_fma(ge[1], sn, P.x));
      P.y = __builtin_fma(ge[2], cs, __builtin_fma(ge[3], sn, P.y));
      P.z = __builtin_fma(ge[4], cs, __builtin_fma(ge[5], sn, P.z));
      const double gi = __builtin_fma(Am.x, ge[1], __builtin_fma(Am.y, ge[3], Am.z * ge[5]));
      const double gr = __builtin_fma(Am.x, ge[0], __builtin_fma(Am.y, ge[2], Am.z * ge[4]));
      Q = __builtin_fma(-w, __builtin_fma(gi, cs, -(gr * sn)), Q);
    };
    long e = 0;
    for (; e + 4 <= A.n_e; e += 4) {
      double phi[4], sn[4], cs[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) phi[u] = (-A.omega[e + u]) * tau;
      sincos_n<false, 4>(phi, sn, cs);
#pragma unroll
      for (int u = 0; u < 4; ++u) add(go + 6 * (e + u), A.omega[e + u], sn[u], cs[u]);
    }
    for (; e < A.n_e; ++e) {
      double sn, cs;
      sincos_huge64((-A.omega[e]) * tau, &sn, &cs);
      add(go + 6 * e, A.omega[e], sn, cs);
    }
    // s = P . A(x, beta, a), dLoss/dtau = Q
    double pw = dot(P, W);
    double b2b = -pw * i1;
    double s1 = (b2 - 1) * b2b;
    V3 PxN = cross(P, N);
    double s2 = dot(P, NY) * i2;
    V3 Wb = vadd(vscale(P, (1 - b2) * i1), vscale(cross(Ac, PxN), i2));
    V3 ab = vscale(cross(PxN, W), i2);
    V3 Nb = vscale(cross(Y, P), i2);
    double kb = -2 * (s1 + s2) * ik;
    double Db = Q * (1.0 / kC) - (2 * s1 + s2) * iD;
    Nb = vadd(vadd(Nb, Wb), vscale(Bt, -kb));
    V3 bb = vadd(vadd(vscale(Wb, -1.0), vscale(N, -kb)), vscale(Bt, 2 * b2b));
    double nbn = dot(Nb, N);
    V3 Rb = vadd(vscale(Nb, iD), vscale(N, Db - nbn * iD));
    gx[0] -= Rb.x; gx[1] -= Rb.y; gx[2] -= Rb.z;
    gx[3] += bb.x; gx[4] += bb.y; gx[5] += bb.z;
    gx[6] += ab.x; gx[7] += ab.y; gx[8] += ab.z;
  }
  if (!valid) return;
  double* out = A.partial + 9 * ((long) blockIdx.y * A.ns + j);
#pragma unroll
  for (int c = 0; c < 9; ++c) out[c] = gx[c];
}

// Sum of the per-chunk partials in a fixed order (deterministic).
__global__ void __launch_bounds__(256) adj_chunk_sum_kernel(const double* __restrict__ partial, long ns, int nchunks,
                                                            double* __restrict__ out) {
  long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 9 * ns) return;
  double s = 0;
  for (int c = 0; c < nchunks; ++c) s += partial[(long) c * 9 * ns + i];
  out[i] = s;
}

// ---------------------------------------------------------------- spline evaluation
__global__ void __launch_bounds__(256) adj_klo_kernel(const double* __restrict__ rows, long ns,
                                                      const double* __restrict__ X, long n, int* __restrict__ klo) {
  long j = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= ns) return;
  klo[j] = (int) spline_interval(X, n, rows[10 * j]);
}

// First index in klo[0..cnt) with klo[i] >= k (klo is non-decreasing within a level).
__device__ __forceinline__ long lower_bound_int(const int* __restrict__ a, long cnt, int k) {
  long lo = 0, hi = cnt;
  while (lo < hi) {
    long mid = (lo + hi) >> 1;
    if (a[mid] < k) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// Transpose of s_j = a Y_lo + b Y_hi + (ca Y''_lo + cb Y''_hi) h^2/6, gathered
// per knot (no atomics): knot k collects the samples whose interval starts at
// k (coefficients a, ca) and at k-1 (coefficients b, cb), level by level.
__global__ void __launch_bounds__(256) adj_knot_gather_kernel(const double* __restrict__ rows,
                                                              const double* __restrict__ sb, const int* __restrict__ klo,
                                                              int L, const double* __restrict__ X, long n,
                                                              double* __restrict__ yb, double* __restrict__ yppb) {
  long k = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  double ay[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  double ap[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int lev = 0; lev <= L; ++lev) {
    long off = (1L << lev) - 1, cnt = 1L << lev;
    const int* kl = klo + off;
    for (int side = 0; side < 2; ++side) {
      int want = (int) k - side;  // side 0: sample interval starts at k; side 1: at k-1
      if (want < 0 || want > n - 2) continue;
      long i = lower_bound_int(kl, cnt, want);
      for (; i < cnt && kl[i] == want; ++i) {
        long js = off + i;
        double x = rows[10 * js];
        long lo = want, hi = want + 1;
        double h = X[hi] - X[lo];
        double a = (X[hi] - x) / h;
        double b = (x - X[lo]) / h;
        double cy = side == 0 ? a : b;
        double cc = side == 0 ? (a * a * a - a) : (b * b * b - b);
        double cp = cc * (h * h) / 6.;
        const double* g = sb + 9 * js;
#pragma unroll
        for (int c = 0; c < 9; ++c) {
          ay[c] += cy * g[c];
          ap[c] += cp * g[c];
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 9; ++c) {
    yb[9 * k + c] = ay[c];
    yppb[9 * k + c] = ap[c];
  }
}

// Transpose of the spline build (include/TOMATH.h:141-203 with the end slopes
// equal to the end secants, so u[0] = un = 0 identically):
//   p_i = sig_i P_{i-1} + 2, P_i = (sig_i - 1)/p_i, U_i = (w_i - sig_i U_{i-1})/p_i,
//   Y''_{N-1} = -U_{N-2}/(P_{N-2} + 2), Y''_k = P_k Y''_{k+1} + U_k,
//   w_i = ((Y_{i+1}-Y_i)/h_i - (Y_i-Y_{i-1})/h_{i-1}) 6/(t_{i+1}-t_{i-1}).
// All three recurrences are contractions on a near-uniform knot grid
// (|dP_i/dP_{i-1}| ~ 0.07, |P| ~ 0.27, |sig/p| ~ 0.14), so each value is a
// geometric sum whose terms beyond kWin = 64 steps are below 1e-36 of the
// first: every knot evaluates its own window in parallel instead of one lane
// walking the N knots.  (The forward spline keeps the reference's sequential
// order; the reverse pass only needs the derivative's value.)
constexpr long kWin = 64;

// P_i, p_i and sig_i (they depend on the knot times only); P_0 = -0.5.
__global__ void __launch_bounds__(256) adj_spline_p_kernel(const double* __restrict__ X, long n,
                                                           double* __restrict__ Pw, double* __restrict__ ppw,
                                                           double* __restrict__ sgw) {
  long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n - 1) return;
  if (i == 0) {
    Pw[0] = -0.5;
    ppw[0] = 1;
    sgw[0] = 0;
    return;
  }
  long j0 = i - kWin > 1 ? i - kWin : 1;
  // start at P_0 exactly, or at the recurrence's fixed point for sig = 1/2 (sqrt(3) - 2)
  double P = j0 == 1 ? -0.5 : -0.26794919243112270;
  double pp = 1, sig = 0;
  for (long j = j0; j <= i; ++j) {
    sig = (X[j] - X[j - 1]) / (X[j + 1] - X[j - 1]);
    pp = sig * P + 2.0;
    P = (sig - 1.0) / pp;
  }
  Pw[i] = P;
  ppw[i] = pp;
  sgw[i] = sig;
}

// Back substitution transposed: T_k = Y''bar_k + P_{k-1} T_{k-1}, T_0 = Y''bar_0;
// Ubar_k = T_k (k <= N-2), and T_{N-1} feeds U_{N-2} through Y''_{N-1}.
__global__ void __launch_bounds__(256) adj_spline_t_kernel(long n, const double* __restrict__ yppb,
                                                           const double* __restrict__ Pw, double* __restrict__ tb) {
  long g = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= 9 * n) return;
  long k = g / 9;
  int c = (int) (g - 9 * k);
  long j0 = k - kWin > 0 ? k - kWin : 0;
  double acc = 0;
  for (long j = j0; j <= k; ++j) acc = yppb[9 * j + c] + (j > 0 ? Pw[j - 1] : 0.0) * acc;
  tb[9 * k + c] = acc;
}

// U recurrence transposed: V_{N-2} = T_{N-2} + alpha T_{N-1}, V_i = T_i - (sig_{i+1}/p_{i+1}) V_{i+1};
// then cc_i = V_i / p_i * 6 / (t_{i+1} - t_{i-1}) for i = 1..N-2.
__global__ void __launch_bounds__(256) adj_spline_v_kernel(const double* __restrict__ X, long n,
                                                           const double* __restrict__ tb, const double* __restrict__ Pw,
                                                           const double* __restrict__ ppw,
                                                           const double* __restrict__ sgw, double* __restrict__ cc) {
  long g = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= 9 * n) return;
  long i = g / 9;
  int c = (int) (g - 9 * i);
  if (i < 1 || i > n - 2) {
    cc[9 * i + c] = 0;
    return;
  }
  long j1 = i + kWin < n - 2 ? i + kWin : n - 2;
  double alpha = -0.5 / (0.5 * Pw[n - 2] + 1.);
  double v = 0;
  for (long j = j1; j >= i; --j) {
    double t = tb[9 * j + c];
    if (j == n - 2) t += alpha * tb[9 * (n - 1) + c];
    v = t + (j < n - 2 ? -sgw[j + 1] / ppw[j + 1] : 0.0) * v;
  }
  cc[9 * i + c] = v / ppw[i] * 6. / (X[i + 1] - X[i - 1]);
}

// Y_bar_k += cc_{k-1}/h_{k-1} - cc_k (1/h_k + 1/h_{k-1}) + cc_{k+1}/h_k (h_k = t_{k+1} - t_k),
// each term present when its index lies in 1..N-2 (cc is zero outside).
__global__ void __launch_bounds__(256) adj_spline_gather_kernel(const double* __restrict__ X, long n,
                                                                const double* __restrict__ cc,
                                                                double* __restrict__ yb) {
  long g = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= 9 * n) return;
  long k = g / 9;
  int c = (int) (g - 9 * k);
  double add = 0;
  if (k >= 2) add += cc[9 * (k - 1) + c] / (X[k] - X[k - 1]);
  if (k >= 1 && k <= n - 2) add += -cc[9 * k + c] / (X[k + 1] - X[k]) - cc[9 * k + c] / (X[k] - X[k - 1]);
  if (k + 1 <= n - 2) add += cc[9 * (k + 1) + c] / (X[k + 1] - X[k]);
  yb[9 * k + c] += add;
}

// ---------------------------------------------------------------- field derivatives
// Field, its Jacobian dB_i/dx_j, and for the differentiated grid the lower
// sample index and the interpolation weight of the upper sample.
struct FieldD {
  double B[3];
  double J[3][3];
  long n0;  // -1: outside the differentiated grid
  double w;
};

__device__ __forceinline__ void und_part_grad(const FieldDev& f, double D, double PS, const double* a, double tc,
                                              double B[3], double dBdD[3]) {
  double L = f.und_length, PL = f.period_length;
  if (D > L / 2. + PS || D < -L / 2. + PS) return;
  double scale = 1;
  if (D < -L / 2. + PS + PL || D > L / 2. + PS - PL)
    scale = (D < -L / 2. + PS + PL / 2. || D > L / 2. + PS - PL / 2.) ? 0.25 : 0.75;
  double sn, cs;
  sincos_huge64(div_by(2.0 * kPi * (D - PS), PL, f.inv_period_length), &sn, &cs);
  double k = 2.0 * kPi / PL;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    B[i] += a[i] * scale * sn * tc;
    dBdD[i] += a[i] * scale * (cs * k * tc + sn * f.taper);
  }
}

__device__ __forceinline__ void field_grad(const FieldDev* __restrict__ F, int nf, int gfield, const double* y,
                                           FieldD& r) {
  double x = y[0], yy = y[2], z = y[4];
  for (int i = 0; i < 3; ++i) {
    r.B[i] = 0;
    for (int j = 0; j < 3; ++j) r.J[i][j] = 0;
  }
  r.n0 = -1;
  r.w = 0;
  for (int fi = 0; fi < nf; ++fi) {
    const FieldDev& f = F[fi];
    if (f.type == kUndulator || f.type == kEPU) {
      double D = (x - f.center[0]) * f.unit[0] + (yy - f.center[1]) * f.unit[1] + (z - f.center[2]) * f.unit[2];
      double tc = 1 + D * f.taper;
      double B[3] = {0, 0, 0}, dB[3] = {0, 0, 0};
      und_part_grad(f, D, f.phase_shift_a, f.field, tc, B, dB);
      if (f.type == kEPU) und_part_grad(f, D, f.phase_shift_b, f.fieldB, tc, B, dB);
      for (int i = 0; i < 3; ++i) {
        r.B[i] += B[i];
        for (int j = 0; j < 3; ++j) r.J[i][j] += dB[i] * f.unit[j];
      }
      continue;
    }
    // grid without rotation (the host rejects rotated grids for the reverse pass).
    // The axis is a run-time value: everything it selects is picked with
    // selects, so no local array is indexed at run time (that would put the
    // arrays, and the field derivatives with them, in scratch memory).
    double X0 = x - f.trans[0], X1 = yy - f.trans[1], X2 = z - f.trans[2];
    if (f.n[0] > 1 && (X0 <= f.start[0] || X0 >= f.stop[0])) continue;
    if (f.n[1] > 1 && (X1 <= f.start[1] || X1 >= f.stop[1])) continue;
    if (f.n[2] > 1 && (X2 <= f.start[2] || X2 >= f.stop[2])) continue;
    int a = f.axis;
    double coord = a == 0 ? X0 : (a == 1 ? X1 : X2);
    double start = a == 0 ? f.start[0] : (a == 1 ? f.start[1] : f.start[2]);
    double step = a == 0 ? f.step[0] : (a == 1 ? f.step[1] : f.step[2]);
    double istep = a == 0 ? f.inv_step[0] : (a == 1 ? f.inv_step[1] : f.inv_step[2]);
    long na = a == 0 ? f.n[0] : (a == 1 ? f.n[1] : f.n[2]);
    int n0 = cell_of(div_by(coord - start, step, istep));
    if (n0 > na - 2) n0 = (int) (na - 2);
    double dd = (coord - start) - (double) n0 * step;
    const double* lo = f.data + 3 * n0;
    for (int i = 0; i < 3; ++i) {
      r.B[i] += lo[i] + div_by((lo[3 + i] - lo[i]) * dd, step, istep);
      double g = div_by(lo[3 + i] - lo[i], step, istep);  // the IEEE quotient
      r.J[i][0] = a == 0 ? r.J[i][0] + g : r.J[i][0];
      r.J[i][1] = a == 1 ? r.J[i][1] + g : r.J[i][1];
      r.J[i][2] = a == 2 ? r.J[i][2] + g : r.J[i][2];
    }
    if (fi == gfield) {
      r.n0 = n0;
      r.w = div_by(dd, step, istep);
    }
  }
}

// The forward's field sum (get_b / field_eval, rk4_common.h) for the fields
// the reverse pass takes: undulators and EPUs, and one-dimensional grids
// without rotation or time dependence.  Same operations in the same order
// (the zero rotation is applied as field_eval applies it), without the other
// models' branches and the out-of-line multi-dimensional grid call, which
// would cost register traffic on every step of the segment kernels.
__device__ __forceinline__ void adj_get_b(const FieldDev* __restrict__ F, int nf, double x, double y, double z,
                                          double B[3]) {
  double s0 = 0, s1 = 0, s2 = 0;
  for (int i = 0; i < nf; ++i) {
    const FieldDev& f = F[i];
    double v[3] = {0, 0, 0};
    if (f.type == kUndulator || f.type == kEPU) {
      double D = (x - f.center[0]) * f.unit[0] + (y - f.center[1]) * f.unit[1] + (z - f.center[2]) * f.unit[2];
      double tc = 1 + D * f.taper;
      undulator_part(f, D, f.phase_shift_a, f.field[0], f.field[1], f.field[2], tc, v, false);
      if (f.type == kEPU) undulator_part(f, D, f.phase_shift_b, f.fieldB[0], f.fieldB[1], f.fieldB[2], tc, v, true);
    } else {
      double X[3] = {x, y, z};
      rot_xyz(X, f);
      X[0] -= f.trans[0]; X[1] -= f.trans[1]; X[2] -= f.trans[2];
      bool out = (f.n[0] > 1 && (X[0] <= f.start[0] || X[0] >= f.stop[0])) ||
                 (f.n[1] > 1 && (X[1] <= f.start[1] || X[1] >= f.stop[1])) ||
                 (f.n[2] > 1 && (X[2] <= f.start[2] || X[2] >= f.stop[2]));
      if (!out) {
        int a = f.axis;
        double coord = a == 0 ? X[0] : (a == 1 ? X[1] : X[2]);
        double start = a == 0 ? f.start[0] : (a == 1 ? f.start[1] : f.start[2]);
        double step = a == 0 ? f.step[0] : (a == 1 ? f.step[1] : f.step[2]);
        double istep = a == 0 ? f.inv_step[0] : (a == 1 ? f.inv_step[1] : f.inv_step[2]);
        long na = a == 0 ? f.n[0] : (a == 1 ? f.n[1] : f.n[2]);
        int n0 = cell_of(div_by(coord - start, step, istep));
        if (n0 > na - 2) n0 = (int) (na - 2);
        double dd = (coord - start) - (double) n0 * step;
        const double* lo = f.data + 3 * n0;
        v[0] = (lo[0] + div_by((lo[3] - lo[0]) * dd, step, istep)) * 1.0;
        v[1] = (lo[1] + div_by((lo[4] - lo[1]) * dd, step, istep)) * 1.0;
        v[2] = (lo[2] + div_by((lo[5] - lo[2]) * dd, step, istep)) * 1.0;
      }
    }
    s0 += v[0]; s1 += v[1]; s2 += v[2];
  }
  B[0] = s0; B[1] = s1; B[2] = s2;
}

// The forward's equations of motion and RK4 step (derivs<kFieldsGeneric>,
// rk4_try, rk4_common.h) over adj_get_b.  The forward refuses trajectories
// whose steps were halved, so the plain step is the forward's.
__device__ __forceinline__ void adj_derivs(const FieldDev* __restrict__ F, int nf, double qomg, const double* x,
                                           double* d) {
  double B[3];
  adj_get_b(F, nf, x[0], x[2], x[4], B);
  d[0] = x[1];
  d[1] = qomg * (-x[5] * B[1] + x[3] * B[2]);
  d[2] = x[3];
  d[3] = qomg * (x[5] * B[0] - x[1] * B[2]);
  d[4] = x[5];
  d[5] = qomg * (x[1] * B[1] - x[3] * B[0]);
}

__device__ __forceinline__ void adj_step(const FieldDev* __restrict__ F, int nf, double qomg, double h, double* y) {
  double dydx[6], dym[6], dyt[6], yt[6];
  adj_derivs(F, nf, qomg, y, dydx);
  double hh = h * 0.5;
  double h6 = h / 6.0;
  for (int i = 0; i < 6; ++i) yt[i] = y[i] + hh * dydx[i];
  adj_derivs(F, nf, qomg, yt, dyt);
  for (int i = 0; i < 6; ++i) yt[i] = y[i] + hh * dyt[i];
  adj_derivs(F, nf, qomg, yt, dym);
  for (int i = 0; i < 6; ++i) {
    yt[i] = y[i] + h * dym[i];
    dym[i] += dyt[i];
  }
  adj_derivs(F, nf, qomg, yt, dyt);
  for (int i = 0; i < 6; ++i) y[i] = y[i] + h6 * (dydx[i] + dyt[i] + 2.0 * dym[i]);
}

// f(y) = (v, qomg v x B(x)) in state order (x, vx, y, vy, z, vz)
__device__ __forceinline__ void fval(const FieldD& fd, double qomg, const double* y, double* d) {
  d[0] = y[1];
  d[1] = qomg * (-y[5] * fd.B[1] + y[3] * fd.B[2]);
  d[2] = y[3];
  d[3] = qomg * (y[5] * fd.B[0] - y[1] * fd.B[2]);
  d[4] = y[5];
  d[5] = qomg * (y[1] * fd.B[1] - y[3] * fd.B[0]);
}

// tangent: out = Jf(y) . t
__device__ __forceinline__ void fjac_vec(const FieldD& fd, double qomg, const double* y, const double* t, double* out) {
  double dx[3] = {t[0], t[2], t[4]};
  double dv[3] = {t[1], t[3], t[5]};
  double v[3] = {y[1], y[3], y[5]};
  double dB[3];
  for (int i = 0; i < 3; ++i) dB[i] = fd.J[i][0] * dx[0] + fd.J[i][1] * dx[1] + fd.J[i][2] * dx[2];
  // d(v x B) = dv x B + v x dB
  out[0] = dv[0];
  out[2] = dv[1];
  out[4] = dv[2];
  out[1] = qomg * ((dv[1] * fd.B[2] - dv[2] * fd.B[1]) + (v[1] * dB[2] - v[2] * dB[1]));
  out[3] = qomg * ((dv[2] * fd.B[0] - dv[0] * fd.B[2]) + (v[2] * dB[0] - v[0] * dB[2]));
  out[5] = qomg * ((dv[0] * fd.B[1] - dv[1] * fd.B[0]) + (v[0] * dB[1] - v[1] * dB[0]));
}

// adjoint: ybar += Jf(y)^T w, and the grid-sample gradient of w . f(y) as the
// two records rec, rec + 1 (the samples either side of the point; ngrid marks
// no contribution)
__device__ __forceinline__ void fjac_tvec(const FieldD& fd, double qomg, const double* y, const double* w,
                                          double* ybar, const AdjRkArgs& A, long rec) {
  double wa[3] = {w[1], w[3], w[5]};
  double v[3] = {y[1], y[3], y[5]};
  // v-bar = w_pos + qomg (B x w_a);  B-bar = qomg (w_a x v)
  ybar[1] += w[0] + qomg * (fd.B[1] * wa[2] - fd.B[2] * wa[1]);
  ybar[3] += w[2] + qomg * (fd.B[2] * wa[0] - fd.B[0] * wa[2]);
  ybar[5] += w[4] + qomg * (fd.B[0] * wa[1] - fd.B[1] * wa[0]);
  double Bb[3] = {qomg * (wa[1] * v[2] - wa[2] * v[1]), qomg * (wa[2] * v[0] - wa[0] * v[2]),
                  qomg * (wa[0] * v[1] - wa[1] * v[0])};
  for (int j = 0; j < 3; ++j) ybar[2 * j] += Bb[0] * fd.J[0][j] + Bb[1] * fd.J[1][j] + Bb[2] * fd.J[2][j];
  if (A.grec_key && rec >= 0) {
    const bool on = fd.n0 >= 0;
    A.grec_key[rec] = on ? fd.n0 : A.ngrid;
    A.grec_key[rec + 1] = on ? fd.n0 + 1 : A.ngrid;
    for (int i = 0; i < 3; ++i) {
      A.grec_val[3 * rec + i] = on ? (1 - fd.w) * Bb[i] : 0.0;
      A.grec_val[3 * (rec + 1) + i] = on ? fd.w * Bb[i] : 0.0;
    }
  }
}

// c_i: direct knot terms and the late-stored acceleration terms of state i.
// Acceleration knot a_{i+1} = f_a(y_i)/c, and a_0 = f_a(y_0)/c.
// k: knot i's row of kb, k1: knot i+1's (read ahead by the segment kernels, so
// the loads are in flight a step before their use).
__device__ __forceinline__ void direct_terms(const AdjRkArgs& A, long i, const double* k, const double* k1,
                                             const FieldD& fd, const double* y, double* c, long rec) {
  for (int r = 0; r < 6; ++r) c[r] = 0;
  c[0] = k[0]; c[2] = k[1]; c[4] = k[2];
  c[1] = k[3] / kC; c[3] = k[4] / kC; c[5] = k[5] / kC;
  double w[6] = {0, 0, 0, 0, 0, 0};
  bool any = false;
  if (i + 1 < A.nf) {
    w[1] += k1[6] / kC; w[3] += k1[7] / kC; w[5] += k1[8] / kC;
    any = true;
  }
  if (i == 0) {
    w[1] += k[6] / kC; w[3] += k[7] / kC; w[5] += k[8] / kC;
    any = true;
  }
  if (any) fjac_tvec(fd, A.qomg, y, w, c, A, rec);
}

// The segment kernels evaluate the fields at every stage of every step on
// one lane's serial chain: the field descriptions and the grid samples are
// copied into LDS first when they fit (a 4001-sample map takes 96 KB), so the
// chain waits on LDS instead of L2.  The copies are bit for bit; returns the
// descriptions to use (the global ones when they do not fit).
extern __shared__ double adj_lds[];

__device__ const FieldDev* stage_fields(const FieldDev* __restrict__ F, int nf, long cap) {
  constexpr long kWords = (long) (sizeof(FieldDev) / sizeof(double));
  long need = nf * kWords;
  for (int i = 0; i < nf; ++i)
    if (F[i].type == kGrid) need += 3 * F[i].n[0] * F[i].n[1] * F[i].n[2];
  if (need > cap) return F;
  const double* src = reinterpret_cast<const double*>(F);
  for (long k = threadIdx.x; k < nf * kWords; k += blockDim.x) adj_lds[k] = src[k];
  long off = nf * kWords;
  for (int i = 0; i < nf; ++i) {
    if (F[i].type != kGrid) continue;
    long n = 3 * F[i].n[0] * F[i].n[1] * F[i].n[2];
    const double* __restrict__ d = F[i].data;
    long k = threadIdx.x;
    for (; k + 15L * blockDim.x < n; k += 16L * blockDim.x) {
      double v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = d[k + (long) u * blockDim.x];
#pragma unroll
      for (int u = 0; u < 16; ++u) adj_lds[off + k + (long) u * blockDim.x] = v[u];
    }
    for (; k < n; k += blockDim.x) adj_lds[off + k] = d[k];
    off += n;
  }
  __syncthreads();
  FieldDev* Fl = reinterpret_cast<FieldDev*>(adj_lds);
  if (threadIdx.x == 0) {
    long o = nf * kWords;
    for (int i = 0; i < nf; ++i) {
      if (Fl[i].type != kGrid) continue;
      Fl[i].data = adj_lds + o;
      o += 3 * Fl[i].n[0] * Fl[i].n[1] * Fl[i].n[2];
    }
  }
  __syncthreads();
  return Fl;
}

// Phase A: per segment, lambda_{i0} = M lambda_{i1} + b with
// M = J_{i0}^T J_{i0+1}^T ... J_{i1-1}^T (J_i the RK4 step's Jacobian) and
// b = sum_i (J_{i0}^T ... J_{i-1}^T) c_i (c_i the knot's direct terms).  Row q of
// M is then the tangent e_q carried forward through the segment's steps:
// row q <- J_i row q.  Eight lanes per segment: every lane of the group
// integrates the same states and field derivatives, and lane q < 6 carries row
// q of M through each step's four stages and adds its share of b, so nothing
// passes between the lanes.
constexpr int kSegLanes = 8;

__global__ void __launch_bounds__(64) adj_seg_map_kernel(AdjRkArgs A) {
  const int grp = threadIdx.x / kSegLanes;
  const int q = threadIdx.x % kSegLanes;
  const int row = q < 6 ? q : 5;  // lanes 6 and 7 repeat row 5 and write nothing
  const long s = (long) blockIdx.x * (64 / kSegLanes) + grp;
  const bool live = s < A.nseg;
  const long ss = live ? s : A.nseg - 1;
  const FieldDev* __restrict__ F = stage_fields(A.F, A.nfields, A.lds_cap);
  // With grid fields only, the fields at the four stages (field_grad) are the
  // ones adj_step would evaluate again, to the bit (the same interpolation,
  // summed from zero in field order), so the next state is formed from them.
  bool all_grid = true;
  for (int fi = 0; fi < A.nfields; ++fi) all_grid = all_grid && F[fi].type == kGrid;
  long i0 = ss * A.K, i1 = i0 + A.K < A.nf ? i0 + A.K : A.nf;
  double y[6];
  for (int r = 0; r < 6; ++r) y[r] = A.ckpt[6 * ss + r];
  double t[6];  // row `row` of M
  for (int r = 0; r < 6; ++r) t[r] = r == row ? 1.0 : 0.0;
  double bq = 0;  // b[row]
  double h = A.dt, hh = h * 0.5, h6 = h / 6.0;
  // kb rows of knots i and i + 1, read one step ahead
  double kc[9], kn[9];
  for (int r = 0; r < 9; ++r) {
    kc[r] = A.kb[9 * i0 + r];
    kn[r] = i0 + 1 < A.nf ? A.kb[9 * (i0 + 1) + r] : 0.0;
  }
  for (long i = i0; i < i1; ++i) {
    double kf[9];
    for (int r = 0; r < 9; ++r) kf[r] = i + 2 < A.nf ? A.kb[9 * (i + 2) + r] : 0.0;
    // the recomputed state, for the reverse sweep
    if (live && q == 0)
      for (int r = 0; r < 6; ++r) A.ybuf[6 * i + r] = y[r];
    FieldD f0;
    field_grad(F, A.nfields, A.gfield, y, f0);
    double c[6];
    direct_terms(A, i, kc, kn, f0, y, c, -1);
    for (int r = 0; r < 9; ++r) {
      kc[r] = kn[r];
      kn[r] = kf[r];
    }
    {
      double acc = bq;
#pragma unroll
      for (int m = 0; m < 6; ++m) acc += t[m] * c[m];
      bq = acc;
    }
    if (i == A.nf - 1) break;
    // stage states and their field derivatives
    double k1[6], y1[6], k2[6], y2[6], k3[6], y3[6];
    fval(f0, A.qomg, y, k1);
    for (int r = 0; r < 6; ++r) y1[r] = y[r] + hh * k1[r];
    FieldD f1;
    field_grad(F, A.nfields, A.gfield, y1, f1);
    fval(f1, A.qomg, y1, k2);
    for (int r = 0; r < 6; ++r) y2[r] = y[r] + hh * k2[r];
    FieldD f2;
    field_grad(F, A.nfields, A.gfield, y2, f2);
    fval(f2, A.qomg, y2, k3);
    for (int r = 0; r < 6; ++r) y3[r] = y[r] + h * k3[r];
    FieldD f3;
    field_grad(F, A.nfields, A.gfield, y3, f3);
    {  // row <- J row, through the four stages
      double d1[6], d2[6], d3[6], d4[6], u[6];
      fjac_vec(f0, A.qomg, y, t, d1);
      for (int r = 0; r < 6; ++r) u[r] = t[r] + hh * d1[r];
      fjac_vec(f1, A.qomg, y1, u, d2);
      for (int r = 0; r < 6; ++r) u[r] = t[r] + hh * d2[r];
      fjac_vec(f2, A.qomg, y2, u, d3);
      for (int r = 0; r < 6; ++r) u[r] = t[r] + h * d3[r];
      fjac_vec(f3, A.qomg, y3, u, d4);
      for (int r = 0; r < 6; ++r) t[r] = t[r] + h6 * (d1[r] + d4[r] + 2.0 * (d2[r] + d3[r]));
    }
    // the next state, as the forward computes it
    if (all_grid) {
      double k4[6];
      fval(f3, A.qomg, y3, k4);
      for (int r = 0; r < 6; ++r) y[r] = y[r] + h6 * (k1[r] + k4[r] + 2.0 * (k3[r] + k2[r]));
    } else {
      adj_step(F, A.nfields, A.qomg, A.dt, y);
    }
  }
  if (!live || q >= 6) return;
  double* o = A.segmap + 42 * s;
  for (int m = 0; m < 6; ++m) o[6 * q + m] = t[m];
  o[36 + q] = bq;
}

// Phase B: lambda at the segment starts, from the end (it is 0 after the last
// knot).  One workgroup of kChainGroups groups of eight lanes, each with a run of
// segments: the run's map is composed (lane q carries row q, as above), the
// groups' maps are chained, and each group goes back through its run with its
// own lambda (lane r component r).  A segment's map is read a step ahead: in
// order on one lane a segment takes 0.55 us, 1.1 ms for 2000 of them; here 2000
// take 59 us.
constexpr int kChainGroups = 32;

__global__ void __launch_bounds__(kChainGroups * kSegLanes) adj_chain_kernel(AdjRkArgs A) {
  __shared__ double gmap[kChainGroups][42];
  __shared__ double glam[kChainGroups + 1][6];
  const int g = threadIdx.x / kSegLanes, q = threadIdx.x % kSegLanes;
  const int row = q < 6 ? q : 5;
  const long per = (A.nseg + kChainGroups - 1) / kChainGroups;
  const long a = g * per < A.nseg ? g * per : A.nseg;
  const long b = a + per < A.nseg ? a + per : A.nseg;
  {
    double t[6], bq = 0, m[42];
#pragma unroll
    for (int r = 0; r < 6; ++r) t[r] = r == row ? 1.0 : 0.0;
#pragma unroll
    for (int r = 0; r < 42; ++r) m[r] = a < b ? A.segmap[42 * a + r] : 0.0;
    for (long s = a; s < b; ++s) {
      double mn[42], u[6];
      const double* o = A.segmap + 42 * (s + 1 < b ? s + 1 : s);
#pragma unroll
      for (int r = 0; r < 42; ++r) mn[r] = o[r];
#pragma unroll
      for (int r = 0; r < 6; ++r) u[r] = t[0] * m[r];
#pragma unroll
      for (int k = 0; k < 6; ++k) bq = __builtin_fma(t[k], m[36 + k], bq);
#pragma unroll
      for (int k = 1; k < 6; ++k)
#pragma unroll
        for (int r = 0; r < 6; ++r) u[r] = __builtin_fma(t[k], m[6 * k + r], u[r]);
#pragma unroll
      for (int r = 0; r < 6; ++r) t[r] = u[r];
#pragma unroll
      for (int r = 0; r < 42; ++r) m[r] = mn[r];
    }
    if (q < 6) {
#pragma unroll
      for (int r = 0; r < 6; ++r) gmap[g][6 * q + r] = t[r];
      gmap[g][36 + q] = bq;
    }
  }
  __syncthreads();
  if (g == 0) {
    double l = 0;
    if (q < 6) glam[kChainGroups][q] = 0;
    for (int k = kChainGroups - 1; k >= 0; --k) {
      double n = gmap[k][36 + row];
#pragma unroll
      for (int c = 0; c < 6; ++c) n = __builtin_fma(gmap[k][6 * row + c], __shfl(l, c, kSegLanes), n);
      l = n;
      if (q < 6) glam[k][q] = l;
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) A.lam[6 * A.nseg + threadIdx.x] = 0;
  double l = glam[g + 1][row], m[7];
#pragma unroll
  for (int c = 0; c < 7; ++c) m[c] = a < b ? A.segmap[42 * (b - 1) + (c < 6 ? 6 * row + c : 36 + row)] : 0.0;
  for (long s = b - 1; s >= a; --s) {
    double mn[7];
    const double* o = A.segmap + 42 * (s > a ? s - 1 : s);
#pragma unroll
    for (int c = 0; c < 7; ++c) mn[c] = o[c < 6 ? 6 * row + c : 36 + row];
    double n = m[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) n = __builtin_fma(m[c], __shfl(l, c, kSegLanes), n);
    l = n;
    if (q < 6) A.lam[6 * s + q] = l;
#pragma unroll
    for (int c = 0; c < 7; ++c) m[c] = mn[c];
  }
}

// Phase C: per segment, recompute the states and sweep back from lambda_{i1},
// scattering the grid-sample gradients.
__global__ void __launch_bounds__(64) adj_seg_reverse_kernel(AdjRkArgs A) {
  const FieldDev* __restrict__ F = stage_fields(A.F, A.nfields, A.lds_cap);
  long s = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= A.nseg) return;
  long i0 = s * A.K, i1 = i0 + A.K < A.nf ? i0 + A.K : A.nf;
  double y[6];
  // the segment's states, recomputed from its checkpoint by adj_seg_map_kernel
  double lam[6];
  for (int r = 0; r < 6; ++r) lam[r] = A.lam[6 * (s + 1) + r];
  double h = A.dt, hh = h * 0.5, h6 = h / 6.0;
  // kb rows of knots i and i + 1, the next one down read one step ahead
  double kc[9], kn[9];
  for (int r = 0; r < 9; ++r) {
    kc[r] = A.kb[9 * (i1 - 1) + r];
    kn[r] = i1 < A.nf ? A.kb[9 * i1 + r] : 0.0;
  }
  for (long i = i1 - 1; i >= i0; --i) {
    double kf[9];
    for (int r = 0; r < 9; ++r) kf[r] = i > i0 ? A.kb[9 * (i - 1) + r] : 0.0;
    for (int r = 0; r < 6; ++r) y[r] = A.ybuf[6 * i + r];
    FieldD f0;
    field_grad(F, A.nfields, A.gfield, y, f0);
    double yb[6] = {0, 0, 0, 0, 0, 0};
    if (i < A.nf - 1) {
      double k1[6], y1[6], k2[6], y2[6], k3[6], y3[6];
      fval(f0, A.qomg, y, k1);
      for (int r = 0; r < 6; ++r) y1[r] = y[r] + hh * k1[r];
      FieldD f1;
      field_grad(F, A.nfields, A.gfield, y1, f1);
      fval(f1, A.qomg, y1, k2);
      for (int r = 0; r < 6; ++r) y2[r] = y[r] + hh * k2[r];
      FieldD f2;
      field_grad(F, A.nfields, A.gfield, y2, f2);
      fval(f2, A.qomg, y2, k3);
      for (int r = 0; r < 6; ++r) y3[r] = y[r] + h * k3[r];
      FieldD f3;
      field_grad(F, A.nfields, A.gfield, y3, f3);
      // yo = y + h6 (k1 + k4 + 2 (k2 + k3))
      double k1b[6], k2b[6], k3b[6], k4b[6];
      for (int r = 0; r < 6; ++r) {
        yb[r] = lam[r];
        k1b[r] = h6 * lam[r];
        k4b[r] = h6 * lam[r];
        k2b[r] = 2.0 * h6 * lam[r];
        k3b[r] = 2.0 * h6 * lam[r];
      }
      double sb[6];
      for (int r = 0; r < 6; ++r) sb[r] = 0;
      fjac_tvec(f3, A.qomg, y3, k4b, sb, A, 10 * i);      // k4 = f(y3), y3 = y + h k3
      for (int r = 0; r < 6; ++r) {
        yb[r] += sb[r];
        k3b[r] += h * sb[r];
        sb[r] = 0;
      }
      fjac_tvec(f2, A.qomg, y2, k3b, sb, A, 10 * i + 2);  // k3 = f(y2), y2 = y + hh k2
      for (int r = 0; r < 6; ++r) {
        yb[r] += sb[r];
        k2b[r] += hh * sb[r];
        sb[r] = 0;
      }
      fjac_tvec(f1, A.qomg, y1, k2b, sb, A, 10 * i + 4);  // k2 = f(y1), y1 = y + hh k1
      for (int r = 0; r < 6; ++r) {
        yb[r] += sb[r];
        k1b[r] += hh * sb[r];
      }
      fjac_tvec(f0, A.qomg, y, k1b, yb, A, 10 * i + 6);   // k1 = f(y)
    }
    double c[6];
    direct_terms(A, i, kc, kn, f0, y, c, 10 * i + 8);
    for (int r = 0; r < 6; ++r) {
      lam[r] = yb[r] + c[r];
    }
    for (int r = 0; r < 9; ++r) {
      kn[r] = kc[r];
      kc[r] = kf[r];
    }
  }
  if (s == 0) {
    for (int r = 0; r < 6; ++r) A.lam[r] = lam[r];
  }
}

__global__ void __launch_bounds__(256) adj_fill_kernel(double* __restrict__ p, long n) {
  long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0;
}

// dLoss/dS from dLoss/dF, F = C2 |E|^2 with E = C0 dt_L S:
// g[6p + k] = (dl[p] f) E[6p + k], f = 2 C2 C0 dt_L.
__global__ void __launch_bounds__(256) adj_dloss_kernel(const double* __restrict__ dl, const double* __restrict__ E,
                                                        double f, double* __restrict__ g, long npts) {
  long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 6 * npts) g[i] = dl[i / 6] * f * E[i];
}

// Gradients with respect to the initial position and beta from the adjoint
// state at t0 (state velocity v = beta c); null outputs are skipped.
__global__ void __launch_bounds__(64) adj_lam_out_kernel(const double* __restrict__ lam, double* __restrict__ gx0,
                                                         double* __restrict__ gb0, double c) {
  int k = threadIdx.x;
  if (k >= 3) return;
  if (gx0) gx0[k] = lam[2 * k];
  if (gb0) gb0[k] = lam[2 * k + 1] * c;
}

// Record keys start at `v` (no contribution).
__global__ void __launch_bounds__(256) adj_key_fill_kernel(int* __restrict__ k, long n, int v) {
  long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) k[i] = v;
}

// gbar[3g + c]: the sum over the records of grid sample g, in record order (the
// records sorted stably by sample; the first of sample g found by bisection).
__global__ void __launch_bounds__(256) adj_grad_gather_kernel(const int* __restrict__ skey,
                                                              const int* __restrict__ sidx, long n,
                                                              const double* __restrict__ val, int ngrid,
                                                              double* __restrict__ gbar) {
  long g = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ngrid) return;
  long lo = 0, hi = n;
  while (lo < hi) {
    long mid = (lo + hi) >> 1;
    if (skey[mid] < g) lo = mid + 1; else hi = mid;
  }
  double s0 = 0, s1 = 0, s2 = 0;
  for (long r = lo; r < n && skey[r] == g; ++r) {
    const long k = sidx[r];
    s0 += val[3 * k];
    s1 += val[3 * k + 1];
    s2 += val[3 * k + 2];
  }
  gbar[3 * g] = s0;
  gbar[3 * g + 1] = s1;
  gbar[3 * g + 2] = s2;
}

}  // namespace om

// ---------------------------------------------------------------- launchers (host)
extern "C" hipError_t om_launch_adj_ckpt(const double* p_raw, long K, long nseg, double* ckpt, hipStream_t s) {
  long blocks = (nseg + 255) / 256;
  hipLaunchKernelGGL(om::adj_ckpt_kernel, dim3((unsigned) blocks), dim3(256), 0, s, p_raw, K, nseg, ckpt);
  return hipGetLastError();
}

extern "C" hipError_t om_launch_adj_lw(const om::AdjLwArgs* A, int nchunks, hipStream_t s) {
  long bx = (A->ns + 255) / 256;
  hipLaunchKernelGGL(om::adj_lw_kernel, dim3((unsigned) bx, (unsigned) nchunks), dim3(256), 0, s, *A);
  return hipGetLastError();
}

extern "C" hipError_t om_launch_adj_chunk_sum(const double* partial, long ns, int nchunks, double* out,
                                              hipStream_t s) {
  long blocks = (9 * ns + 255) / 256;
  hipLaunchKernelGGL(om::adj_chunk_sum_kernel, dim3((unsigned) blocks), dim3(256), 0, s, partial, ns, nchunks, out);
  return hipGetLastError();
}

// scratch: Pw, ppw, sgw (n each), tb and cc (9 n each)
extern "C" hipError_t om_launch_adj_spline(const double* rows, long ns, const double* sb, int L, const double* X,
                                           long n, int* klo, double* yb, double* yppb, double* Pw, double* ppw,
                                           double* sgw, double* tb, double* cc, hipStream_t s) {
  hipLaunchKernelGGL(om::adj_klo_kernel, dim3((unsigned) ((ns + 255) / 256)), dim3(256), 0, s, rows, ns, X, n, klo);
  hipLaunchKernelGGL(om::adj_knot_gather_kernel, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, rows, sb, klo,
                     L, X, n, yb, yppb);
  unsigned b1 = (unsigned) ((n + 255) / 256), b9 = (unsigned) ((9 * n + 255) / 256);
  hipLaunchKernelGGL(om::adj_spline_p_kernel, dim3(b1), dim3(256), 0, s, X, n, Pw, ppw, sgw);
  hipLaunchKernelGGL(om::adj_spline_t_kernel, dim3(b9), dim3(256), 0, s, n, yppb, Pw, tb);
  hipLaunchKernelGGL(om::adj_spline_v_kernel, dim3(b9), dim3(256), 0, s, X, n, tb, Pw, ppw, sgw, cc);
  hipLaunchKernelGGL(om::adj_spline_gather_kernel, dim3(b9), dim3(256), 0, s, X, n, cc, yb);
  return hipGetLastError();
}

extern "C" hipError_t om_launch_adj_rk4(const om::AdjRkArgs* A, hipStream_t s) {
  long blocks = (A->nseg + 63) / 64;
  long map_blocks = (A->nseg + 64 / om::kSegLanes - 1) / (64 / om::kSegLanes);
  // dynamic LDS for the staged fields: what the 160 KB of a CU leaves beside
  // the static arrays (one workgroup per CU; these kernels run few waves)
  constexpr size_t kMapBytes = 160 * 1024 - 1024;
  constexpr size_t kRevBytes = 160 * 1024 - 1024;
  om::AdjRkArgs R = *A;
  size_t map_bytes = kMapBytes, rev_bytes = kRevBytes;
  if (hipFuncSetAttribute((const void*) om::adj_seg_map_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int) map_bytes) != hipSuccess)
    map_bytes = 0;
  if (hipFuncSetAttribute((const void*) om::adj_seg_reverse_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int) rev_bytes) != hipSuccess)
    rev_bytes = 0;
  (void) hipGetLastError();  // a refused attribute leaves the fields in global memory
  R.lds_cap = (long) (map_bytes / sizeof(double));
  hipLaunchKernelGGL(om::adj_seg_map_kernel, dim3((unsigned) map_blocks), dim3(64), map_bytes, s, R);
  hipLaunchKernelGGL(om::adj_chain_kernel, dim3(1), dim3(om::kChainGroups * om::kSegLanes), 0, s, R);
  R.lds_cap = (long) (rev_bytes / sizeof(double));
  hipLaunchKernelGGL(om::adj_seg_reverse_kernel, dim3((unsigned) blocks), dim3(64), rev_bytes, s, R);
  return hipGetLastError();
}

extern "C" hipError_t om_launch_adj_fill(double* p, long n, hipStream_t s) {
  long blocks = (n + 255) / 256;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(om::adj_fill_kernel, dim3((unsigned) blocks), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

extern "C" hipError_t om_launch_adj_dloss(const double* dl, const double* E, double f, double* g, long npts,
                                          hipStream_t s) {
  long blocks = (6 * npts + 255) / 256;
  hipLaunchKernelGGL(om::adj_dloss_kernel, dim3((unsigned) blocks), dim3(256), 0, s, dl, E, f, g, npts);
  return hipGetLastError();
}

extern "C" hipError_t om_launch_adj_lam_out(const double* lam, double* gx0, double* gb0, double c, hipStream_t s) {
  hipLaunchKernelGGL(om::adj_lam_out_kernel, dim3(1), dim3(64), 0, s, lam, gx0, gb0, c);
  return hipGetLastError();
}

extern "C" hipError_t om_launch_adj_key_fill(int* k, long n, int v, hipStream_t s) {
  long blocks = (n + 255) / 256;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(om::adj_key_fill_kernel, dim3((unsigned) blocks), dim3(256), 0, s, k, n, v);
  return hipGetLastError();
}

// Bytes of temporary storage the stable sort of n records (keys below 2^end_bit) takes.
extern "C" hipError_t om_adj_grad_sort_bytes(long n, int end_bit, size_t* bytes) {
  return rocprim::radix_sort_pairs(nullptr, *bytes, (const int*) nullptr, (int*) nullptr,
                                   rocprim::counting_iterator<int>(0), (int*) nullptr, (unsigned) n, 0,
                                   (unsigned) end_bit);
}

// The records sorted stably by grid sample (rocPRIM's radix sort: records of
// one sample keep their order), then summed per sample into gbar.
extern "C" hipError_t om_launch_adj_grad_gather(const int* key, int* skey, int* sidx, const double* val, long n,
                                                int ngrid, int end_bit, void* temp, size_t temp_bytes, double* gbar,
                                                hipStream_t s) {
  size_t bytes = temp_bytes;
  hipError_t e = rocprim::radix_sort_pairs(temp, bytes, key, skey, rocprim::counting_iterator<int>(0), sidx,
                                           (unsigned) n, 0, (unsigned) end_bit, s);
  if (e != hipSuccess) return e;
  long blocks = (ngrid + 255) / 256;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(om::adj_grad_gather_kernel, dim3((unsigned) blocks), dim3(256), 0, s, skey, sidx, n, val, ngrid,
                     gbar);
  return hipGetLastError();
}
