// Trajectory integration in parallel segments (multiple shooting) for gfx950.
//
// What bounds it: the RK4 recurrence of src/OSCARSSR.cc:910-1009 is one serial
// chain; stepped in order (rk4_kernel, traj.hip) a 20001-point planar
// trajectory keeps one wave of the chip busy for 12 ms (0.62 us a step, bound by
// the step's dependent instructions), an EPU's 40001 points for 36 ms.  Here a
// chain of steps is cut into segments that run at once, each from an estimate of
// its start state, and the estimates are corrected until the segments join.
// With F_s the map of segment s and U_s its start estimate,
//   r_{s+1} = F_s(U_s) - U_{s+1}             (the mismatch at a join)
//   d_{s+1} = J_s d_s + r_{s+1},  d_0 = 0    (Newton, J_s the Jacobian of F_s)
//   U_s <- U_s + d_s
// The first estimate is a straight line.  The fields move the states a little
// at a time, so the mismatches fall from 1e-6 m to 1e-13, 1e-16 and then to the
// last bits.  The corrections are exact there (r is the exact difference of
// two close doubles, so a segment whose start stops changing repeats its bits),
// and a chain is accepted when no join differs by more than a small fraction of
// the last bit of the position and velocity along the trajectory (kShootPos,
// kShootVelAlong): the knots are then those of the integration in order, apart
// from the last bits of the small transverse components.  On the undulators,
// EPUs, maps and field pairs tried: 12 rounds, 25 at most, z and beta_z equal in every
// bit, x and y within 2.1e-16 m (8e-18 m in all but four settings).
//
// Every step is the reference's, in the operation order of rk4_kernel (derivs
// and rk4_try of rk4_common.h).  A segment in which |beta| >= 1 is met is never
// accepted (its steps would have to be halved), nor is a chain whose joins
// still differ after its rounds: rk4_kernel then integrates that
// particle in order, as it does for short chains.
//
// Layout: one wave holds eight segments of eight lanes.  Lane 0 of a segment
// steps its start state; lanes 1..6 step the same state moved along one of the
// six coordinates, which gives J_s as differences at no further cost in time
// (the wave issues the same instructions).  A workgroup is four waves, one per
// SIMD (a wave's steps fill its SIMD's issue slots), with its 32 segments' maps
// d -> J d + r in LDS and their composition, 42 doubles, in memory; the
// workgroups of a chain wait for each other once a round, and each walks the
// compositions before its own.  One launch for everything (as two launches a
// round, segments and walk, the 20001-point planar chain took 0.30 ms of kernels
// and 36 launches).  Measured, by the rounds an electron takes: planar 20001 points
// 12.4 -> 0.16 to 0.24 ms, EPU 40001 points 37.5 -> 0.39 to 0.55 ms, 1-D map 20001
// points 18.1 -> 0.40 to 0.57 ms, undulator and Gaussian 8001 points 23.7 -> 0.4 to
// 1.05 ms (8 to 24 rounds).
//
// The wait is bounded: if the workgroups of a chain cannot all be resident,
// because other work fills the GPU, the first whose wait runs out gives the chain
// up for all (the count of arrivals turns negative), and it is integrated in
// order.  It runs out after a poll (0.4 us) per step, about half the time in
// order takes with one magnet and far more than a round's.  300 calls beside a
// batch of 8 / 12 waves per CU: 20001 planar points 4 / 15 given up (16 to 21 ms
// each), mean 1.9 / 4.9 ms; 40001 EPU points 9 / 29 (42 to 55 ms, 107 for a few
// that found no place to run), mean 4.6 / 9.3 ms; every call in order takes 13 and
// 36 ms.  A quarter of the wait: 5 / 46 and 8 / 33 given up; three times: 4 / 8 and
// 10 / 8, of 25 to 32 and 52 to 64 ms.
#include "om_device.h"
#include "launch_types.h"
#include "om_types.h"
#include "rk4_common.h"
#include "rk4_variant.h"

namespace om {

// Accepted mismatch at a join, relative to the trajectory's length (c dt n) for
// the position and to the speed for the velocity.  Along the trajectory none is
// left but next to z = 0, where the last bit is smaller: a photon's phase, 1e11
// rad, is sensitive to the last bit of z, and a join off by less than a bit
// there is off by one further on.  Across, two units of the coordinate's own last
// place: the joins' mismatches add up along the chain.  The random walk of the
// last bits can keep a chain from settling for long: 1920 electrons of 3 GeV
// through five settings of fields with 3001 to 40001 points took 12 rounds at the
// median, 25 at most, and z and beta_z were those of the integration in order in
// every bit.  Strong fields take longer: 100 MeV in 0.3 T, 8001 points, 85; 3 GeV
// in a 10 T wiggler, 60001 points, 60.  So there are kShootRounds rounds, and up
// to kShootRoundsMax where a chain is long: one for 128 steps, about a quarter of
// the time in order takes, which is what a chain that does not settle loses (steps
// of 7 cm, 3001 points: 3.3 -> 4.1 ms; 100 MeV in 0.3 T, 2001 points: 1.4 -> 2.1;
// the 10 T wiggler, settled, 39 -> 3.1 ms).
constexpr double kShootPos = 1.3552527156068805e-20;      // 2^-66
constexpr double kShootVelAlong = 5.551115123125783e-17;  // 2^-54
constexpr double kShootVel = 2.168404344971009e-19;       // 2^-62
constexpr double kShootUlps = 4.440892098500626e-16;      // 2^-51 of the component itself
constexpr int kShootGivenUp = -(1 << 30);  // arrivals of a chain given up, plus those since

// d <- J d + r, d in every lane; lane r < 6 holds row r of J and r_r (lanes
// beyond compute copies of row 5).
__device__ __forceinline__ void shoot_advance(double d[6], const double row[7]) {
  double a = row[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) a = __builtin_fma(row[q], d[q], a);
  const long long b = __builtin_bit_cast(long long, a);
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const unsigned lo = __builtin_amdgcn_readlane((int) (b & 0xffffffff), q);
    const unsigned hi = __builtin_amdgcn_readlane((int) (b >> 32), q);
    d[q] = __builtin_bit_cast(double, ((unsigned long long) hi << 32) | lo);
  }
}

// d through the n maps at m (42 doubles each, by rows); at(s) is called with
// the index of each map before d passes it, after(s) after.
template <class At, class After>
__device__ __forceinline__ void shoot_walk(double d[6], const double* m, int n, int row, At at, After after) {
  double cur[7], nxt[7];
#pragma unroll
  for (int k = 0; k < 7; ++k) nxt[k] = n > 0 ? m[7 * row + k] : 0.0;
#pragma unroll 1
  for (int s = 0; s < n; ++s) {
#pragma unroll
    for (int k = 0; k < 7; ++k) cur[k] = nxt[k];
    const double* p = m + 42 * (s + 1 < n ? s + 1 : s) + 7 * row;
#pragma unroll
    for (int k = 0; k < 7; ++k) nxt[k] = p[k];
    at(s);
    shoot_advance(d, cur);
    after(s);
  }
}

// The n maps at m composed into out, in lanes 0..6: lane q < 6 holds column q
// of the product of the J, lane 6 the offset.
__device__ __forceinline__ void shoot_compose(const double* m, int n, int stride, int lane, double v[6]) {
#pragma unroll
  for (int k = 0; k < 6; ++k) v[k] = lane == k ? 1.0 : 0.0;
#pragma unroll 1
  for (int s = 0; s < n; ++s, m += stride) {
    double nv[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      double a = lane == 6 ? m[7 * k + 6] : 0.0;
#pragma unroll
      for (int j = 0; j < 6; ++j) a = __builtin_fma(m[7 * k + j], v[j], a);
      nv[k] = a;
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] = nv[k];
  }
}

// Wave-scope ordering of LDS accesses exchanged inside one wave.
__device__ __forceinline__ void shoot_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int M>
__global__ void __launch_bounds__(64 * kShootWaves) shoot_kernel(const ShootArgs A, const UndParams f_arg, const GridZ g) {
  __shared__ double sSeg[kShootWaves][8][42];  // the segments' maps, by rows (six coefficients and the offset)
  __shared__ double sWave[kShootWaves][42];    // composed per wave
  __shared__ double sWalk[kShootWalk][42];     // other workgroups' maps
  __shared__ double sD[12];  // corrections at this workgroup's start and at the next one's
  __shared__ int sOk[kShootWaves];
  __shared__ int sWait;
  const int ib = blockIdx.x;
  const ShootChain C = A.chain[A.block_chain[ib]];
  const int me = ib - C.block0;  // this workgroup's place in its chain
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, grp = lane >> 3, q = lane & 7;
  const int row = lane < 6 ? lane : 5;
  const TrajDesc* D = A.desc + C.ip;
  const double h = C.dir ? -D->dt : D->dt;
  const double t0 = D->t0_over_c;
  const long n = C.n;                                                          // steps of the chain
  const long i0 = (((long) me * kShootWaves + wv) * 8 + grp) * C.steps;  // first step of this segment
  const long left = n - i0;
  const int ns = left < 0 ? 0 : (left < C.steps ? (int) left : C.steps);
  const bool last = i0 + C.steps >= n;
  double U[6], Un[6];  // this segment's start and the next one's: a straight line
  double speed;
  {
    double x0[6];
    x0[0] = D->x0[0]; x0[1] = D->b0[0] * kC;
    x0[2] = D->x0[1]; x0[3] = D->b0[1] * kC;
    x0[4] = D->x0[2]; x0[5] = D->b0[2] * kC;
    speed = sqrt(x0[1] * x0[1] + x0[3] * x0[3] + x0[5] * x0[5]);
    const double ta = h * (double) i0, tb = h * (double) (i0 + C.steps);
#pragma unroll
    for (int k = 0; k < 6; k += 2) {
      U[k] = x0[k] + x0[k + 1] * ta;
      Un[k] = x0[k] + x0[k + 1] * tb;
      U[k + 1] = Un[k + 1] = x0[k + 1];
    }
  }
  const double length = kC * D->dt * (double) D->n;
  const UndParams f0 = (M == kOneUndulator || (M >= kAxisUndX && M <= kAxisUndZ) || M == kUndZ) ? und_in_vgpr(f_arg)
                                                                                              : f_arg;
  RkCtx c{A.F, A.nf, D->qomg, 0, g, 0, D->qom, 0};
  double* tk = A.t + D->knot_offset;
  double* pk = A.p + 9 * D->knot_offset;
  const long nb = D->nb;
  for (int round = 0; round < A.rounds; ++round) {
    // lanes 1..6: the start moved along coordinate q - 1, by 2^-26 m or 2^-24 c
    // (any step between the roundings and the fields' scale serves: the
    // differences only steer the corrections)
    double y[6], eps = 1.0;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      y[k] = U[k];
      if (q == k + 1) {
        y[k] += (k & 1) ? kC * 5.9604644775390625e-08 : 1.4901161193847656e-08;
        eps = y[k] - U[k];
      }
    }
    bool bad = false;
    double dxdt[6];
    if (C.dir == 0 && i0 == 0) {  // the initial knot
      derivs<M>(c, f0, t0 + h * 0.0, y, dxdt);
      if (q == 0) store_knot(tk, pk, nb, t0 + h * 0.0, y, dxdt);
    }
#pragma unroll 1
    for (int i = 0; i < ns; ++i) {
      const long k = i0 + i;
      const double t1 = t0 + h * (double) k;
      double yo[6];
      c.err = 0;
      derivs<M>(c, f0, t1, y, dxdt);
      bad = rk4_try<M>(c, f0, y, dxdt, t1, h, yo) || bad;
#pragma unroll
      for (int j = 0; j < 6; ++j) y[j] = yo[j];
      // the forward chain's last step is taken and not stored, as in rk4_kernel
      if (q == 0 && (C.dir || k < n - 1))
        store_knot(tk, pk, C.dir ? nb - 1 - k : nb + 1 + k, t0 + h * (double) (k + 1), y, dxdt);
    }
    // the segment's map: Jacobian columns from the moved starts, and the
    // mismatch with the next segment's start (none after the last one)
    double r[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const double yb = __shfl(y[k], lane & 56);
      r[k] = last ? 0.0 : yb - Un[k];
      const double v = q == 0 ? r[k] : (y[k] - yb) / eps;
      if (q < 7) sSeg[wv][grp][7 * k + (q == 0 ? 6 : q - 1)] = v;
    }
    {
      const double tol_x = kShootPos * length, tol_v = kShootVel * speed;
      bool ok = !bad && fabs(U[1] * r[0] + U[3] * r[2] + U[5] * r[4]) <= tol_x * speed &&
                fabs(U[1] * r[1] + U[3] * r[3] + U[5] * r[5]) <= kShootVelAlong * speed * speed;
#pragma unroll
      for (int k = 0; k < 6; ++k)  // (a NaN is not accepted)
        ok = ok && fabs(r[k]) <= fmax((k & 1) ? tol_v : tol_x, kShootUlps * fabs(U[k]));
      const bool all_ok = __all(ok || q != 0);
      if (lane == 0) sOk[wv] = all_ok ? 1 : 0;
    }
    shoot_wave_sync();
    double v[6];
    if (lane < 7) {
      shoot_compose(&sSeg[wv][0][0], 8, 42, lane, v);
#pragma unroll
      for (int k = 0; k < 6; ++k) sWave[wv][7 * k + lane] = v[k];
    }
    __syncthreads();
    bool done = sOk[0] && sOk[1] && sOk[2] && sOk[3];
    static_assert(kShootWaves == 4, "flags of the waves");
    if (C.nblock > 1) {
      // the workgroup's map to the others, in the buffer of the round's parity:
      // a workgroup writes this one again only after all have read it
      double* Mb = A.Mb + 42L * A.nblocks * (round & 1);
      int* okb = A.block_ok + A.nblocks * (round & 1);
      if (wv == 0) {
        if (lane < 7) {
          shoot_compose(&sWave[0][0], kShootWaves, 42, lane, v);
#pragma unroll
          for (int k = 0; k < 6; ++k)
            __hip_atomic_store(Mb + 42L * ib + 7 * k + lane, v[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0) __hip_atomic_store(okb + ib, done ? 1 : 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // The map and the flag are past the caches before the arrival is.  This rests
        // on gfx950, not on the language's memory model, in which the relaxed stores
        // are not ordered before the relaxed arrival: stores at agent scope are
        // written through to what the XCDs share, vmcnt(0) waits until they are there,
        // the arrival is a later instruction of the same wave, and the readers drop
        // their caches' copies (the acquire fence below) after they have seen it.  A
        // release fence here would write the knots back from L2 in every round.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (lane == 0) {
          int* cnt = A.arrived + A.block_chain[ib];
          const int target = C.nblock * (round + 1);
          int now = atomicAdd(cnt, 1) + 1;
          for (long polls = A.polls >= 0 ? A.polls : n; now >= 0 && now < target && polls > 0; --polls) {
            __builtin_amdgcn_s_sleep(1);
            now = __hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
          if (now < target) atomicMin(cnt, kShootGivenUp);
          sWait = now < target ? 0 : 1;
        }
      }
      __syncthreads();
      if (!sWait) return;  // given up: the chain is not marked done
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      bool ok = true;
      for (int b = lane; b < C.nblock; b += 64) ok = ok && okb[C.block0 + b] != 0;
      done = __all(ok);
    }
    if (done) {
      if (me == 0 && threadIdx.x == 0) A.done[A.block_chain[ib]] = round + 1;
      return;
    }
    // The corrections.  Un must stay the very double the next segment's lanes
    // hold, so a correction used on both sides of a wave's or a workgroup's edge
    // is formed the same way on both: through the compositions of the waves
    // (workgroups) before it.
    double d[6] = {0, 0, 0, 0, 0, 0}, dn[6] = {0, 0, 0, 0, 0, 0};
    if (C.nblock > 1) {
      const double* Mb = A.Mb + 42L * A.nblocks * (round & 1) + 42L * C.block0;
      for (int b0 = 0; b0 <= me; b0 += kShootWalk) {  // this workgroup's own map last
        const int nw = me + 1 - b0 < kShootWalk ? me + 1 - b0 : kShootWalk;
        for (int k = threadIdx.x; k < 42 * nw; k += 64 * kShootWaves) (&sWalk[0][0])[k] = Mb[42L * b0 + k];
        __syncthreads();
        if (wv == 0)
          shoot_walk(
              dn, &sWalk[0][0], nw, row,
              [&](int s) {
#pragma unroll
                for (int k = 0; k < 6; ++k) d[k] = b0 + s == me ? dn[k] : d[k];
              },
              [](int) {});
        __syncthreads();
      }
      if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          sD[k] = d[k];
          sD[6 + k] = dn[k];
        }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 6; ++k) d[k] = sD[k];
    }
    shoot_walk(d, &sWave[0][0], wv, row, [](int) {}, [](int) {});
    if (wv < kShootWaves - 1) {
#pragma unroll
      for (int k = 0; k < 6; ++k) dn[k] = d[k];
      shoot_walk(dn, &sWave[wv][0], 1, row, [](int) {}, [](int) {});
    } else if (C.nblock > 1) {
#pragma unroll
      for (int k = 0; k < 6; ++k) dn[k] = sD[6 + k];
    }
    shoot_walk(
        d, &sSeg[wv][0][0], 8, row,
        [&](int s) {
#pragma unroll
          for (int k = 0; k < 6; ++k) U[k] = s == grp ? U[k] + d[k] : U[k];
        },
        [&](int s) {
#pragma unroll
          for (int k = 0; k < 6; ++k) Un[k] = s == grp ? Un[k] + (s < 7 ? d[k] : dn[k]) : Un[k];
        });
    __syncthreads();  // the maps are rewritten by the next round
  }
}

}  // namespace om

// ---------------------------------------------------------------- launchers (host)
namespace {
template <int M>
void launch_shoot(const om::Rk4Variant& v, const om::ShootArgs& A, hipStream_t s) {
  hipLaunchKernelGGL(om::shoot_kernel<M>, dim3((unsigned) A.nblocks), dim3(64 * om::kShootWaves), 0, s, A, v.und,
                     v.grid);
}
}  // namespace

// Steps a segment should have at least: a round costs some 14 us beside its steps
// (composition, wait, walk), a step 0.45 us with one magnet and 3 to 5 us with
// several field models.  Measured, om_trajectories with 4 / 8 / 12 / 16 / 24 steps:
// planar 20001 points 607 / 389 / 356 / 365 / 375 us, EPU 40001 points 874 / 673 /
// 634 / 607 / 739, two field models 20001 points 728 / 844 / 937 / 1121 / 1779.
extern "C" int om_shoot_steps(const om::FieldDev* F0_host, int nfields) {
  return om::rk4_variant(*F0_host, nfields, 0).m == om::kFieldsGeneric ? 4 : 12;
}

// The two-part variant of rk4_kernel for an EPU along z has no use here (a
// segment has its lanes taken): und_eval gives the same doubles.
extern "C" hipError_t om_launch_shoot(const om::ShootArgs* A, const om::FieldDev* F0_host, hipStream_t s) {
  const om::Rk4Variant v = om::rk4_variant(*F0_host, A->nf, 0);
  switch (v.m) {
    case om::kGridZ: launch_shoot<om::kGridZ>(v, *A, s); break;
    case om::kAxisUndX: launch_shoot<om::kAxisUndX>(v, *A, s); break;
    case om::kAxisUndY: launch_shoot<om::kAxisUndY>(v, *A, s); break;
    case om::kAxisUndZ: launch_shoot<om::kAxisUndZ>(v, *A, s); break;
    case om::kUndZ: launch_shoot<om::kUndZ>(v, *A, s); break;
    case om::kEpuZ:
    case om::kOneUndulator: launch_shoot<om::kOneUndulator>(v, *A, s); break;
    default: launch_shoot<om::kFieldsGeneric>(v, *A, s); break;
  }
  return hipGetLastError();
}
