// Batched multi-particle Lienard-Wiechert sums in one persistent launch.
//
// Every particle of the resident trajectory set contributes weight * flux to
// one request (an observation grid x an energy list); requests may differ in
// grid size and energy count, and particles in trajectory length.  The work
// unit is (particle, observation point, block of up to kBatchEB energies); a
// persistent grid of single-wave workgroups pulls units from a device counter
// (a vector atomic on global memory), runs the reference's level loop for the
// block's energies, re-packing the still-active ones into full waves at every
// level, and adds the weighted flux into the request's output with FP64
// atomics (an incoherent sum over particles; the summation order, and so the
// last bits, depend on scheduling).
//
// Reference behaviour restated (paths relative to the reference root):
//   multi-particle loop with weight 1/N   src/OSCARSSR.cc:4016-4063, 1778-1818
//   level loop and convergence           src/OSCARSSR.cc:4179-4245
//   level sample times                   src/TParticleTrajectoryInterpolated.cc:124-161, 264-270
//
// Level samples of all particles live in one block: particle p, level L starts
// at row p*stride + 2^L - 1 (stride = 2^(Lcap+1) - 1 rows of 10 doubles).
// Deeper levels (rare: slowly converging points) are interpolated from the
// spline inside the sum kernel with the same expressions, so a batch follows
// the same level rule as the single-particle path up to max_level.
#include "lw_common.h"
#include "rk4_common.h"

namespace om {


__global__ void __launch_bounds__(256) level_batch_kernel(LevelJobBatch J) {
  long g = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (long) J.np * J.stride) return;
  int ip = (int) (g / J.stride);
  long s = g - (long) ip * J.stride;
  int L = 63 - __clzll((unsigned long long) (s + 1));  // s in [2^L - 1, 2^(L+1) - 1)
  long i = s - ((1L << L) - 1);
  double ts = J.tspan[2 * ip], te = J.tspan[2 * ip + 1];
  // src/TParticleTrajectoryInterpolated.cc:138-147, 264-270 and
  // src/TParticleTrajectoryInterpolatedPoints.cc:33-37 (same operations as the host)
  double p2L = (double) (1L << L);
  double spacing = L > J.stop_mem ? (te - ts) / (p2L - 1) : (te - ts) / p2L;
  double tt = ts + (te - ts) / (2.0 * p2L) + spacing * (double) i;
  TrajDesc D = J.desc[ip];
  double v[9];
  spline_value(J.t + D.knot_offset, J.p + 9 * D.knot_offset, J.ypp + 9 * D.knot_offset, D.n, tt, v);
  double* o = J.rows + 10 * g;
  o[0] = tt;
#pragma unroll
  for (int c = 0; c < 9; ++c) o[1 + c] = v[c];
}



// Amplitude of a sample interpolated from the spline at time tt (levels above
// the stored rows; rare).
__device__ __forceinline__ Amp interpolated_amplitude(const BatchArgs& A, const TrajDesc& D, V3 obs,
                                                                double tt) {
  double srow[10];
  srow[0] = tt;
  spline_value(A.t + D.knot_offset, A.p + 9 * D.knot_offset, A.ypp + 9 * D.knot_offset, D.n, tt, srow + 1);
  return amplitude(obs, srow);
}

// Lane 0's value as a wave-uniform scalar (two 32-bit readfirstlane moves).
__device__ __forceinline__ unsigned long long uniform_u64(unsigned long long v) {
  unsigned lo = (unsigned) __builtin_amdgcn_readfirstlane((int) (unsigned) v);
  unsigned hi = (unsigned) __builtin_amdgcn_readfirstlane((int) (unsigned) (v >> 32));
  return ((unsigned long long) hi << 32) | lo;
}

// LDS of one persistent wave: the amplitudes of the current super-block and the
// active list.
struct BatchLds : AmpLds {
  unsigned short list[kBatchEB];
};

// One atomic for the wave, by lane 0, its old value in every lane.  (An atomic
// executed by all lanes with zeros but in lane 0 is 64 operations on one
// address, one after the other.)
__device__ __forceinline__ unsigned long long wave_add(unsigned long long* p, int lane, unsigned long long v) {
  unsigned long long old = 0;
  if (lane == 0) old = atomicAdd(p, v);
  return uniform_u64(old);
}

// One work unit (particle ip, observation point io, energies e0 .. e0+n_eb-1).
struct Unit {
  long item;
  int ip;
  long io, e0;
  int n_eb;
  V3 obs;
  double ts, te, T;
  const double* prow;
  TrajDesc D;
  ReqDev R;
};

__device__ __forceinline__ Unit unit_of(const BatchArgs& A, long item) {
  Unit U;
  U.item = item;
  // particle of this work unit: last p with item_prefix[p] <= item
  int lo = 0, hi = A.np;
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (A.item_prefix[mid] <= item) lo = mid; else hi = mid;
  }
  U.ip = lo;
  const long local = item - A.item_prefix[U.ip];
  U.R = A.req[A.req_of[U.ip]];
  U.io = local / U.R.n_blocks_e;
  U.e0 = (local - U.io * U.R.n_blocks_e) * kBatchEB;
  U.n_eb = (int) (U.R.n_e - U.e0 < kBatchEB ? U.R.n_e - U.e0 : kBatchEB);
  U.obs = v3(U.R.obs[3 * U.io], U.R.obs[3 * U.io + 1], U.R.obs[3 * U.io + 2]);
  U.ts = A.tspan[2 * U.ip];
  U.te = A.tspan[2 * U.ip + 1];
  U.T = U.te - U.ts;
  U.prow = A.rows + 10 * (long) U.ip * A.stride;
  U.D = A.desc[U.ip];
  return U;
}

// End of level L for one energy: the level's sum ps added, then the convergence
// test of src/OSCARSSR.cc:4227-4239.  SC32: anl is the level's sum of |V|_1, and
// border is set where the decision lay within the sin/cos error bound.
template <bool SC32>
__device__ __forceinline__ bool batch_level_end(const BatchArgs& A, int L, double dt, const double ps[6], double maxd,
                                                double anl, double sum[6], double& lastmag, double& prec,
                                                double& an_run, double& dm_last, bool& border) {
#pragma unroll
  for (int c = 0; c < 6; ++c) sum[c] += ps[c];
  double E[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) E[c] = sum[c] * dt;
  if (A.use_pol) pol_project(E, A.pol);
  const double mag = cmag2(E);
  const double mag_prev = lastmag;
  prec = fabs(mag - mag_prev) / mag_prev;
  if (SC32) {
    an_run += anl;
    if (level_borderline(L, dt, A.precision, mag_prev, mag, prec, maxd, an_run, dm_last)) border = true;
  }
  lastmag = mag;
  return (L > 8 && prec < A.precision && maxd < kPi) || (L > 8 && maxd < kPi && mag == mag_prev);
}

// Adds a finished energy of a unit to its request, and its counts.
__device__ __forceinline__ void batch_add_point(const BatchArgs& A, const Unit& U, int e, int lev, const double sum[6],
                                                bool converged) {
  double f = A.C0 * (U.T / (2.0 * (double) (1L << lev) - 1));
  double E[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) E[k] = sum[k] * f;
  if (A.use_pol) pol_project(E, A.pol);
  atomicAdd(&U.R.out[U.io * U.R.n_e + U.e0 + e], A.C2 * cmag2(E) * A.weight[U.ip]);
  if (!converged) atomicAdd(A.n_unconverged, 1ULL);
  atomicAdd(A.evals, (unsigned long long) ((2L << lev) - 1));
}

// Flags of an energy in the wave's scratch.
constexpr int kFConverged = 1;
constexpr int kFBorderline = 2;  // mixed pass: a stop decision lay within the sin/cos error bound
constexpr int kFHanded = 4;      // handed to lw_batch_level_kernel
constexpr int kFRecheck = 8;     // recomputed in FP64 inside the unit
constexpr int kFIdle = 16;       // not part of the FP64 recheck pass

// The reference's level loop for the energies of a unit whose flags carry none
// of the bits in `skip`.  SC32: reduced-accuracy sin/cos (sincos_fast64) with
// the borderline test, else full-accuracy sin/cos.  Level by level, the still
// active energies are packed into groups: 64 energies, one per lane, and for
// the last r < 64 of a level, m = 64 / r replicas of the r energies, replica q
// walking the q-th contiguous part of every super-block.  The level's samples
// go in super-blocks of kSuper: the lanes compute their amplitudes into LDS
// once, then every group walks the super-block at its energies (a group's
// partial sums wait in the wave's scratch while the others walk), so a
// sample's amplitude is computed once per level whatever the number of
// groups.  The replicas' partial sums are added in a fixed tree order.  The
// largest phase step takes the sample before each part from LDS (or from the
// previous super-block), so it is the same maximum over the same consecutive
// pairs as a sequential walk.  Energies still active at level Ldeep leave the
// unit in groups for lw_batch_level_kernel (while there are groups to be had).
template <bool SC32>
__device__ __forceinline__ void unit_levels(const BatchArgs& A, const Unit& U, int lane, double* __restrict__ ws,
                                            int* __restrict__ wsi, BatchLds& S, int skip, unsigned long long& n_amp,
                                            unsigned long long& n_ev, unsigned long long& n_slot) {
  double* w_sum = ws;                    // 6 x kBatchEB
  double* w_lastmag = ws + 6 * kBatchEB;
  double* w_prec = ws + 7 * kBatchEB;
  double* w_an = ws + 8 * kBatchEB;      // mixed: sum of |V|_1 over the samples so far
  double* w_dm = ws + 9 * kBatchEB;      // mixed: error bound of lastmag
  double* w_grp = ws + kBatchWsD * kBatchEB;  // partial sums of the groups between super-blocks
  int* w_level = wsi;
  int* w_flags = wsi + kBatchEB;
  const int n_eb = U.n_eb;
  for (int L = 0; L <= A.Lmax; ++L) {
    // pack the energies still active
    int n_act = 0;
    for (int t = 0; t < n_eb; t += 64) {
      int e = t + lane;
      bool a = e < n_eb && (w_flags[e < n_eb ? e : 0] & skip) == 0;
      unsigned long long m = __ballot(a);
      if (a) S.list[n_act + __popcll(m & ((1ULL << lane) - 1ULL))] = e;
      n_act += __popcll(m);
    }
    __syncthreads();
    if (n_act == 0) break;
    if (L == A.Ldeep) {
      const int ng = (n_act + 63) >> 6;
      const unsigned long long g0 =
          wave_add(A.n_group, lane, (unsigned long long) ng);
      if (g0 + (unsigned long long) ng <= (unsigned long long) A.group_cap) {
        constexpr int kind = SC32 ? 0 : 1;
        for (int g = 0; g < ng; ++g) {
          const long id = (long) g0 + g;
          const int W = n_act - 64 * g < 64 ? n_act - 64 * g : 64;
          if (lane < W) {
            const int e = S.list[64 * g + lane];
            double* st = A.group_state + id * (kBatchGroupD * 64) + lane;
            A.group_e[64 * id + lane] = (unsigned short) e;
#pragma unroll
            for (int k = 0; k < 6; ++k) st[64 * k] = w_sum[k * kBatchEB + e];
            st[64 * 6] = w_lastmag[e];
            st[64 * 7] = w_an[e];
            st[64 * 8] = w_dm[e];
            w_flags[e] |= kFHanded;
          }
          if (lane == 0) {
            A.group_item[id] = U.item;
            A.group_n[id] = W;
            const unsigned long long j = atomicAdd(&A.n_list[kind * kBatchLevels + L], 1ULL);
            A.group_list[(2 * kind + (L & 1)) * A.group_cap + (long) j] = (int) id;
          }
        }
        if (lane == 0) atomicAdd(A.n_deep, (unsigned long long) n_act);
        __syncthreads();
        break;
      }
    }
    const double* __restrict__ rows = U.prow + 10 * ((1L << L) - 1);
    const long ns = 1L << L;
    // sample times of level L (the expressions of level_batch_kernel)
    const double p2L = (double) (1L << L);
    const double spacing = L > A.stop_mem ? (U.te - U.ts) / (p2L - 1) : (U.te - U.ts) / p2L;
    const double tfirst = U.ts + (U.te - U.ts) / (2.0 * p2L);
    const bool stored = L <= A.Lb;
    const double dt = U.T / (2.0 * (double) (1L << L) - 1);
    const int n_groups = (n_act + 63) >> 6;  // 64 energies each, the last one r <= 64
    const long n_sb = (ns + kSuper - 1) / kSuper;
    n_amp += (unsigned long long) ns;
    double anl = 0;   // mixed: sum of |V|_1 over the samples this lane computed
    double tprev = 0; // tau of the last sample of the previous super-block
    double ps[6] = {0, 0, 0, 0, 0, 0};
    double maxd = 0;
    for (long sb = 0; sb < n_sb; ++sb) {
      const long base = sb * kSuper;
      const int cnt = (int) ((ns - base) < kSuper ? (ns - base) : kSuper);
#pragma unroll 1
      for (int h = 0; h < kSuper; h += 64) {
        const long si = base + h + lane;
        if (si < ns) {
          Amp a;
          if (stored) {
            a = amplitude(U.obs, rows + 10 * si);
          } else {
            a = interpolated_amplitude(A, U.D, U.obs, tfirst + spacing * (double) si);
          }
          S.tau[blk(h + lane)] = a.tau;
          S.vx[blk(h + lane)] = a.V.x;
          S.vy[blk(h + lane)] = a.V.y;
          S.vz[blk(h + lane)] = a.V.z;
          if (SC32) anl += fabs(a.V.x) + fabs(a.V.y) + fabs(a.V.z);
        }
      }
      wave_sync();
      const bool last_sb = sb == n_sb - 1;
      if (SC32 && last_sb) {
        // every sample of the level was computed by one lane: the |V|_1 sum is wave-uniform
        for (int off = 32; off > 0; off >>= 1) anl += __shfl_xor(anl, off);
      }
      for (int grp = 0; grp < n_groups; ++grp) {
        const int g = grp << 6;
        const int W = n_act - g < 64 ? n_act - g : 64;  // energies in this group
        const int m = 64 / W;                            // replicas of each
        const int q = lane / W;                          // this lane's replica (q >= m: idle)
        const int j = lane - q * W;
        const bool act = q < m;
        const int e = S.list[g + (act ? j : 0)];  // idle lanes shadow the group's first energy
        const double negw = -U.R.omega[U.e0 + e];
        if (sb == 0) {
          n_ev += (unsigned long long) ns * (unsigned long long) W;
          const long full = ns >> 6, part = ns & 63;
          n_slot += 64ULL * ((unsigned long long) full * (unsigned long long) ((64 + m - 1) / m) +
                             (unsigned long long) ((part + m - 1) / m));
        }
        if (n_groups > 1) {
          // this group's partial sums from the previous super-block (lane-private)
          double* gp = w_grp + grp * 7 * 64 + lane;
          if (sb == 0) {
#pragma unroll
            for (int c = 0; c < 6; ++c) ps[c] = 0;
            maxd = 0;
          } else {
#pragma unroll
            for (int c = 0; c < 6; ++c) ps[c] = gp[c * 64];
            maxd = gp[6 * 64];
          }
        }
        double lastphase;  // phase of the sample before the part being walked
        auto walk = [&](int k0, int k1) {
          int k = k0;
          for (; k + 4 <= k1; k += 4) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const int b = blk(k + u);
              double phi = negw * S.tau[b];
              maxd = fmax(maxd, fabs(phi - lastphase));
              lastphase = phi;
              double sn, cs;
              sincos_mode(SC32, phi, sn, cs);
              double vx = S.vx[b], vy = S.vy[b], vz = S.vz[b];
              ps[0] = __builtin_fma(vx, cs, ps[0]); ps[1] = __builtin_fma(vx, sn, ps[1]);
              ps[2] = __builtin_fma(vy, cs, ps[2]); ps[3] = __builtin_fma(vy, sn, ps[3]);
              ps[4] = __builtin_fma(vz, cs, ps[4]); ps[5] = __builtin_fma(vz, sn, ps[5]);
            }
          }
          for (; k < k1; ++k) {
            const int b = blk(k);
            double phi = negw * S.tau[b];
            maxd = fmax(maxd, fabs(phi - lastphase));
            lastphase = phi;
            double sn, cs;
            sincos_mode(SC32, phi, sn, cs);
            double vx = S.vx[b], vy = S.vy[b], vz = S.vz[b];
            ps[0] = __builtin_fma(vx, cs, ps[0]); ps[1] = __builtin_fma(vx, sn, ps[1]);
            ps[2] = __builtin_fma(vy, cs, ps[2]); ps[3] = __builtin_fma(vy, sn, ps[3]);
            ps[4] = __builtin_fma(vz, cs, ps[4]); ps[5] = __builtin_fma(vz, sn, ps[5]);
          }
        };
        if (m == 1) {  // one energy per lane: the whole super-block, wave-uniform bounds
          lastphase = negw * (base > 0 ? tprev : S.tau[0]);
          walk(0, cnt);
        } else {
          const int k0 = act ? (q * cnt) / m : 0;
          const int k1 = act ? ((q + 1) * cnt) / m : 0;
          lastphase = negw * (k0 > 0 ? S.tau[blk(k0 - 1)] : (base > 0 ? tprev : S.tau[0]));
          walk(k0, k1);
        }
        if (!last_sb) {
          if (n_groups > 1) {
            double* gp = w_grp + grp * 7 * 64 + lane;
#pragma unroll
            for (int c = 0; c < 6; ++c) gp[c * 64] = ps[c];
            gp[6 * 64] = maxd;
          }
          continue;
        }
        // the level is complete for this group
        if (m > 1) {
          double none = 0;
          add_replicas(ps, maxd, none, lane, W, m, q, act);
        }
        if (q == 0) {
          double sum[6], lastmag = w_lastmag[e], prec, an_run = 0, dm_last = 0;
          bool border = false;
#pragma unroll
          for (int c = 0; c < 6; ++c) sum[c] = w_sum[c * kBatchEB + e];
          if (SC32) {
            an_run = w_an[e];
            dm_last = w_dm[e];
          }
          const bool c =
              batch_level_end<SC32>(A, L, dt, ps, maxd, anl, sum, lastmag, prec, an_run, dm_last, border);
          if (SC32) {
            w_an[e] = an_run;
            w_dm[e] = dm_last;
          }
#pragma unroll
          for (int k = 0; k < 6; ++k) w_sum[k * kBatchEB + e] = sum[k];
          w_lastmag[e] = lastmag;
          w_prec[e] = prec;
          w_level[e] = L;
          w_flags[e] = w_flags[e] | (c ? kFConverged : 0) | (border ? kFBorderline : 0);
        }
      }
      tprev = S.tau[blk(cnt - 1)];
      wave_sync();  // the next super-block overwrites the amplitudes
    }
    __syncthreads();  // this level's state is read by other lanes at the next one
  }
}

// One work unit: the level loop for the block's energies, weighted flux added
// into the request's output with FP64 atomics.  MIXED: a first pass with the
// reduced-accuracy sin/cos; the energies whose stop decision lay within its error bound are
// then recomputed from level 0 with FP64 sin/cos in a second pass of the same
// unit (their amplitudes shared, the rows still in cache), so every energy
// stops where the FP64 path stops.  The per-energy state lives in the wave's
// scratch (ws, wsi) between levels.
template <bool MIXED>
__device__ __forceinline__ void batch_unit(const BatchArgs& A, long item, int lane, double* __restrict__ ws,
                                           int* __restrict__ wsi, BatchLds& S) {
  const Unit U = unit_of(A, item);
  const int n_eb = U.n_eb;
  double* w_sum = ws;
  double* w_lastmag = ws + 6 * kBatchEB;
  double* w_prec = ws + 7 * kBatchEB;
  double* w_an = ws + 8 * kBatchEB;
  double* w_dm = ws + 9 * kBatchEB;
  int* w_level = wsi;
  int* w_flags = wsi + kBatchEB;
  for (int e = lane; e < n_eb; e += 64) {
#pragma unroll
    for (int k = 0; k < 6; ++k) w_sum[k * kBatchEB + e] = 0;
    w_lastmag[e] = -1;
    w_prec[e] = -1;
    w_an[e] = 0;
    w_dm[e] = 0;
    w_level[e] = -1;
    w_flags[e] = 0;
  }
  __syncthreads();  // the state written above is read by other lanes
  unsigned long long n_amp = 0, n_ev = 0, n_slot = 0;  // wave-uniform work counts of this unit
  unit_levels<MIXED>(A, U, lane, ws, wsi, S, kFConverged | kFBorderline | kFHanded, n_amp, n_ev, n_slot);
  if (MIXED) {
    // FP64 recheck: reset the borderline energies (the first pass left them
    // where they were met), park the others
    int n_re = 0;
    for (int t = 0; t < n_eb; t += 64) {
      const int e = t + lane;
      const int ec = e < n_eb ? e : 0;
      const int flags = w_flags[ec];
      const bool want = e < n_eb && (flags & (kFBorderline | kFHanded)) == kFBorderline;
      n_re += __popcll(__ballot(want));
      if (want) {
#pragma unroll
        for (int k = 0; k < 6; ++k) w_sum[k * kBatchEB + e] = 0;
        w_lastmag[e] = -1;
        w_prec[e] = -1;
        w_level[e] = -1;
        w_flags[e] = kFRecheck;
        w_an[e] = 0;
        w_dm[e] = 0;
      } else if (e < n_eb) {
        w_flags[e] = flags | kFIdle;
      }
    }
    __syncthreads();
    if (n_re > 0) {
      unit_levels<false>(A, U, lane, ws, wsi, S, kFConverged | kFHanded | kFIdle, n_amp, n_ev, n_slot);
    }
    if (lane == 0 && n_re > 0) atomicAdd(A.n_recheck, (unsigned long long) n_re);
  }
  // outputs and bookkeeping for the block's energies
  unsigned long long n_unc = 0, n_evals = 0;  // lane 0's
  for (int t = 0; t < n_eb; t += 64) {
    const int e = t + lane;
    const int ec = e < n_eb ? e : 0;
    const int lev = w_level[ec];
    const int flags = w_flags[ec];
    const bool v = e < n_eb && (flags & kFHanded) == 0;  // handed-over energies finish in the deep kernel
    if (v) {
      double f = A.C0 * (U.T / (2.0 * (double) (1L << lev) - 1));
      double E[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) E[k] = w_sum[k * kBatchEB + e] * f;
      if (A.use_pol) pol_project(E, A.pol);
      atomicAdd(&U.R.out[U.io * U.R.n_e + U.e0 + e], A.C2 * cmag2(E) * A.weight[U.ip]);
    }
    unsigned long long nc = __ballot(v && !(flags & kFConverged));
    unsigned long long ev = v ? (unsigned long long) ((2L << lev) - 1) : 0ULL;
    for (int off = 32; off > 0; off >>= 1) ev += __shfl_down(ev, off);
    n_unc += (unsigned long long) __popcll(nc);
    n_evals += ev;
  }
  if (lane == 0) {
    if (n_unc) atomicAdd(A.n_unconverged, n_unc);
    atomicAdd(A.evals, n_evals);
    atomicAdd(A.main_amps, n_amp);
    atomicAdd(A.main_evals, n_ev);
    atomicAdd(A.main_slots, n_slot);
  }
  __syncthreads();  // the next unit overwrites the scratch
}

// Four waves per SIMD: the register budget is set for the hot stored-row path;
// the rare interpolation path may spill.
template <bool MIXED>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) lw_batch_kernel(BatchArgs A) {
  __shared__ BatchLds S;
  int lane = threadIdx.x;
  double* ws = A.ws + (long) blockIdx.x * kBatchWsTotal;
  int* wsi = A.wsi + (long) blockIdx.x * kBatchWsI * kBatchEB;
  while (true) {
    // Next work unit: the index is taken from lane 0 with readfirstlane, so it is
    // a scalar and the loop exit a uniform branch.
    const long item = (long) wave_add(A.counter, lane, 1ULL);
    if (item >= A.total_items) break;
    batch_unit<MIXED>(A, item, lane, ws, wsi, S);
  }
}

// ---------------------------------------------------------------- deep levels
// One level of the groups handed over.  A unit whose energies converge slowly
// has level after level of 2^L samples: left to its one wave, a single energy
// at level 25 takes 0.2 s, most of a batch of 64 particles (182 ms of which the
// chip's work was 26).  Here the level's samples are cut into slices, enough to
// occupy every wave (one each when there are many groups), a wave computes a
// slice's amplitudes super-block by super-block as unit_levels does and walks
// them with the group's energies, and the wave that completes a group adds the
// slices' partial sums in order, takes the decisions and lists the group, its
// energies packed again, for the next level.
// Measured, 64 particles (13664 units): 182 ms and 324 ms (two seeds) with every
// energy left to its unit, 40 ms and 38 ms handed over at level 12; 2048
// particles (1.76 M units) 5.10 -> 4.85 s at level 17.
constexpr int kLevelWaves = 4;  // independent waves per workgroup
template <bool SC32>
__global__ void __launch_bounds__(64 * kLevelWaves) __attribute__((amdgpu_waves_per_eu(4)))
lw_batch_level_kernel(BatchArgs A, int L) {
  __shared__ BatchLds lds[kLevelWaves];
  constexpr int kind = SC32 ? 0 : 1;
  BatchLds& S = lds[threadIdx.x >> 6];
  const int lane = threadIdx.x & 63;
  const long n = (long) A.n_list[kind * kBatchLevels + L];
  if (n == 0) return;
  const long ns = 1L << L;
  // slices of at least 512 samples, at most 256 to a group, in all at most what
  // there is room for (16 for each of the 4096 waves; their cost depends on the
  // group's energies, so they are taken from a counter)
  long nsl = kBatchParts / n;
  nsl = nsl < 1 ? 1 : (nsl > kBatchGroupSlices ? kBatchGroupSlices : nsl);
  nsl = nsl > ns / 512 ? ns / 512 : nsl;
  const int* __restrict__ ids = A.group_list + (2 * kind + (L & 1)) * A.group_cap;
  while (true) {
    const long job = (long) wave_add(&A.n_job[kind * kBatchLevels + L], lane, 1ULL);
    if (job >= n * nsl) break;
    const long gi = job / nsl, sl = job - gi * nsl;
    const long id = ids[gi];
    const Unit U = unit_of(A, A.group_item[id]);
    const int W = A.group_n[id];
    const int m = 64 / W;      // replicas of each energy
    const int q = lane / W;    // this lane's (q >= m: idle)
    const int j = lane - q * W;
    const bool act = q < m;
    const int slot = act ? j : 0;
    const int e = A.group_e[64 * id + slot];
    const double negw = -U.R.omega[U.e0 + e];
    const double* __restrict__ rows = U.prow + 10 * (ns - 1);
    const double p2L = (double) ns;
    const double spacing = L > A.stop_mem ? (U.te - U.ts) / (p2L - 1) : (U.te - U.ts) / p2L;
    const double tfirst = U.ts + (U.te - U.ts) / (2.0 * p2L);
    const bool stored = L <= A.Lb;
    auto amp_at = [&](long i) {
      return stored ? amplitude(U.obs, rows + 10 * i)
                    : interpolated_amplitude(A, U.D, U.obs, tfirst + spacing * (double) i);
    };
    const long i0 = ns * sl / nsl, i1 = ns * (sl + 1) / nsl;
    double ps[6], maxd, anl;
    walk_slice<SC32>(amp_at, i0, i1, negw, lane, m, q, act, S, ps, maxd, anl);
    double none = 0;
    add_replicas(ps, maxd, none, lane, W, m, q, act);
    const bool mine = lane < W;  // replica 0
    if (nsl > 1) {
      part_publish(A.part + (gi * nsl + sl) * (8 * 64), lane, mine, ps, maxd, anl);
      if (part_arrive(&A.group_arrived[id], lane) + 1 < (unsigned) nsl) continue;
      if (lane == 0) A.group_arrived[id] = 0;
      part_gather(A.part + gi * nsl * (8 * 64), nsl, lane, W, m, q, act, ps, maxd, anl);
    }
    // decisions, one energy per lane; the others' lanes hold none
    double* gs = A.group_state + id * (kBatchGroupD * 64);
    double sum[6], lastmag = 0, prec, an_run = 0, dm_last = 0;
    bool border = false, go_on = false;
    if (mine) {
#pragma unroll
      for (int k = 0; k < 6; ++k) sum[k] = gs[64 * k + lane];
      lastmag = gs[64 * 6 + lane];
      if (SC32) {
        an_run = gs[64 * 7 + lane];
        dm_last = gs[64 * 8 + lane];
      }
      // (a decision that lay within the error bound at an earlier level went to
      // the recomputation list there)
      const bool c = batch_level_end<SC32>(A, L, U.T / (2.0 * (double) ns - 1), ps, maxd, anl, sum, lastmag, prec,
                                           an_run, dm_last, border);
      bool listed = false;
      if (SC32 && border) {
        const unsigned long long k = atomicAdd(A.n_fix, 1ULL);
        if (k < (unsigned long long) A.fix_cap) {
          A.fix_list[k] = (unsigned long long) U.item * kBatchEB + (unsigned long long) e;
          listed = true;
        }
      }
      go_on = !listed && !c && L < A.Lmax;
      if (!listed && !go_on) batch_add_point(A, U, e, L, sum, c);
    }
    const unsigned long long live = __ballot(go_on);
    if (live) {
      const int at = __popcll(live & ((1ULL << lane) - 1ULL));
      if (go_on) {
        A.group_e[64 * id + at] = (unsigned short) e;
#pragma unroll
        for (int k = 0; k < 6; ++k) gs[64 * k + at] = sum[k];
        gs[64 * 6 + at] = lastmag;
        if (SC32) {
          gs[64 * 7 + at] = an_run;
          gs[64 * 8 + at] = dm_last;
        }
      }
      if (lane == 0) {
        A.group_n[id] = __popcll(live);
        const unsigned long long k = atomicAdd(&A.n_list[kind * kBatchLevels + L + 1], 1ULL);
        A.group_list[(2 * kind + ((L + 1) & 1)) * A.group_cap + (long) k] = (int) id;
      }
    }
  }
}

// FP64 recomputation of the points the mixed kernels listed, from level 0, so
// their levels and values are the FP64 path's.  One wave per point, its lanes
// splitting each level's samples, up to level Ldeep - 1; a point active there
// becomes a group of its own for lw_batch_level_kernel<false> (or, with no
// group left, goes on here).  Four waves per workgroup; the waves stride over
// the list independently.
__global__ void __launch_bounds__(256) lw_batch_fix_kernel(BatchArgs A) {
  const int lane = threadIdx.x & 63;
  const long wave = (long) blockIdx.x * 4 + (threadIdx.x >> 6);
  const long n_waves = (long) gridDim.x * 4;
  long n = (long) *A.n_fix;
  if (n > A.fix_cap) n = A.fix_cap;
  for (long k = wave; k < n; k += n_waves) {
    const unsigned long long code = A.fix_list[k];
    const Unit U = unit_of(A, (long) (code / kBatchEB));
    const int e = (int) (code - (unsigned long long) U.item * kBatchEB);
    const double negw = -U.R.omega[U.e0 + e];
    double sum[6] = {0, 0, 0, 0, 0, 0};
    double lastmag = -1, prec, an_run = 0, dm_last = 0;
    int lev = -1;
    bool c = false, border = false, handed = false;
    for (int L = 0; L <= A.Lmax && !c; ++L) {
      if (L == A.Ldeep) {
        const unsigned long long id = wave_add(A.n_group, lane, 1ULL);
        if (id < (unsigned long long) A.group_cap) {
          if (lane == 0) {
            double* st = A.group_state + (long) id * (kBatchGroupD * 64);
#pragma unroll
            for (int q = 0; q < 6; ++q) st[64 * q] = sum[q];
            st[64 * 6] = lastmag;
            A.group_e[64 * id] = (unsigned short) e;
            A.group_item[id] = U.item;
            A.group_n[id] = 1;
            const unsigned long long j = atomicAdd(&A.n_list[kBatchLevels + L], 1ULL);
            A.group_list[(2 + (L & 1)) * A.group_cap + (long) j] = (int) id;
          }
          handed = true;
          break;
        }
      }
      const long ns = 1L << L;
      const double p2L = (double) ns;
      double tot[6], maxd, an;
      if (L <= A.Lb) {
        slice_level_sum_rows<false>(U.prow + 10 * (ns - 1), 0, ns, U.obs, negw, lane, tot, maxd, an);
      } else {
        const double spacing = L > A.stop_mem ? (U.te - U.ts) / (p2L - 1) : (U.te - U.ts) / p2L;
        const double tfirst = U.ts + (U.te - U.ts) / (2.0 * p2L);
        slice_level_sum<false>(
            0, ns, negw, lane,
            [&](long i) { return interpolated_amplitude(A, U.D, U.obs, tfirst + spacing * (double) i); }, tot, maxd,
            an);
      }
      lev = L;
      c = batch_level_end<false>(A, L, U.T / (2.0 * p2L - 1), tot, maxd, 0.0, sum, lastmag, prec, an_run, dm_last,
                                 border);
    }
    // every lane holds the same totals (butterfly sums): lane 0 adds the point
    if (lane == 0 && !handed) batch_add_point(A, U, e, lev, sum, c);
  }
}

// Clears n doubles (outputs) and the counters without a memset node, so the
// sequence can be captured in a HIP graph and replayed.
__global__ void __launch_bounds__(256) batch_clear_kernel(double* __restrict__ out, long n,
                                                          unsigned long long* __restrict__ counters, int nc) {
  long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = 0.0;
  if (i < nc) counters[i] = 0ULL;
}

}  // namespace om

extern "C" hipError_t om_launch_level_batch(const om::LevelJobBatch* J, hipStream_t s) {
  long total = (long) J->np * J->stride;
  long blocks = (total + 255) / 256;
  hipLaunchKernelGGL(om::level_batch_kernel, dim3((unsigned) blocks), dim3(256), 0, s, *J);
  return hipGetLastError();
}

extern "C" hipError_t om_launch_batch_clear(double* out, long n, unsigned long long* counters, int nc,
                                            hipStream_t s) {
  long m = n > nc ? n : nc;
  long blocks = (m + 255) / 256;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(om::batch_clear_kernel, dim3((unsigned) blocks), dim3(256), 0, s, out, n, counters, nc);
  return hipGetLastError();
}

// The batch: the persistent kernel (stage bit 0), the levels of the energies it
// handed over (bit 1) and, mixed, the FP64 recomputation of borderline points
// (bit 2); stages = 7 launches all three in order.  A launch per level: one with
// nothing listed returns at once (about 5 us in a graph).
extern "C" hipError_t om_launch_lw_batch_stages(const om::BatchArgs* A, int mixed, int n_groups, int stages,
                                                hipStream_t s) {
  if (stages & 1) {
    if (mixed) hipLaunchKernelGGL(om::lw_batch_kernel<true>, dim3(n_groups), dim3(64), 0, s, *A);
    else hipLaunchKernelGGL(om::lw_batch_kernel<false>, dim3(n_groups), dim3(64), 0, s, *A);
  }
  const unsigned waves = 4096;  // 16 per CU
  const dim3 grid(waves / om::kLevelWaves), block(64 * om::kLevelWaves);
  if (stages & 2)
    for (int L = A->Ldeep; L <= A->Lmax; ++L) {
      if (mixed) hipLaunchKernelGGL(om::lw_batch_level_kernel<true>, grid, block, 0, s, *A, L);
      else hipLaunchKernelGGL(om::lw_batch_level_kernel<false>, grid, block, 0, s, *A, L);
    }
  if (mixed && (stages & 4) && A->Ldeep <= A->Lmax) {
    hipLaunchKernelGGL(om::lw_batch_fix_kernel, dim3(waves / 4), dim3(256), 0, s, *A);
    for (int L = A->Ldeep; L <= A->Lmax; ++L)
      hipLaunchKernelGGL(om::lw_batch_level_kernel<false>, grid, block, 0, s, *A, L);
  }
  return hipGetLastError();
}

extern "C" hipError_t om_launch_lw_batch(const om::BatchArgs* A, int mixed, int n_groups, hipStream_t s) {
  return om_launch_lw_batch_stages(A, mixed, n_groups, 7, s);
}
