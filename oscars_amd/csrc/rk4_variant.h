// Host side: which variant of the equations of motion (rk4_common.h) a set of
// fields takes, with the compact parameters the specialised ones are passed by
// value.  Used by the launchers of the step-by-step and of the segmented
// integration (traj.hip, shoot.hip), which therefore agree on it.
#pragma once

#include <string.h>

#include "rk4_common.h"

namespace om {

struct Rk4Variant {
  int m;             // kFieldsGeneric ... kEpuZ
  UndParams und;     // a single undulator or EPU
  GridZ grid;        // kGridZ (samples in device memory)
  size_t grid_bytes;  // kGridZ: LDS the staged samples take
};

// f: the first magnetic field (host copy; its data pointer is a device one).
inline Rk4Variant rk4_variant(const FieldDev& f, int nfields, int nefields) {
  Rk4Variant v;
  memset(&v, 0, sizeof(v));
  v.m = nefields > 0 ? kFieldsEB : kFieldsGeneric;
  // the specialised variants hold time-independent magnetic fields only
  if (nefields > 0 || nfields != 1 || f.td) return v;
  // one z grid without rotation whose samples fit in LDS: the staged-grid variant
  const size_t grid_bytes = (size_t) 3 * f.n[2] * sizeof(double);
  if (f.type == kGrid && f.axis == 2 && f.rot_sin[0] == 0 && f.rot_sin[1] == 0 && f.rot_sin[2] == 0 &&
      f.rot_cos[0] == 1 && f.rot_cos[1] == 1 && f.rot_cos[2] == 1 && grid_bytes <= 160 * 1024) {
    v.m = kGridZ;
    v.grid_bytes = grid_bytes;
    v.grid.data = f.data;
    v.grid.n = f.n[2];
    v.grid.start = f.start[2];
    v.grid.stop = f.stop[2];
    v.grid.step = f.step[2];
    v.grid.inv_step = f.inv_step[2];
    v.grid.trans = f.trans[2];
    return v;
  }
  if (f.type != kUndulator && f.type != kEPU) return v;
  UndParams& u = v.und;
  u.c0 = f.center[0]; u.c1 = f.center[1]; u.c2 = f.center[2];
  u.u0 = f.unit[0]; u.u1 = f.unit[1]; u.u2 = f.unit[2];
  u.taper = f.taper;
  u.half_len = f.und_length / 2.;
  u.PL = f.period_length;
  u.inv_PL = f.inv_period_length;
  u.half_PL = f.period_length / 2.;
  u.psA = f.phase_shift_a;
  u.psB = f.phase_shift_b;
  u.a0 = f.field[0]; u.a1 = f.field[1]; u.a2 = f.field[2];
  u.b0 = f.fieldB[0]; u.b1 = f.fieldB[1]; u.b2 = f.fieldB[2];
  u.epu = f.type == kEPU;
  for (int k = 0; k < 2; ++k) {
    double ps = k == 0 ? u.psA : u.psB;
    double* th = k == 0 ? u.thA : u.thB;
    th[0] = -u.half_len + ps;
    th[1] = u.half_len + ps;
    th[2] = -u.half_len + ps + u.PL;
    th[3] = u.half_len + ps - u.PL;
    th[4] = -u.half_len + ps + u.half_PL;
    th[5] = u.half_len + ps - u.half_PL;
  }
  v.m = kOneUndulator;
  if (f.unit[0] != 0 || f.unit[1] != 0 || f.unit[2] != 1 || f.taper != 0) return v;
  // period along z, untapered: the EPU's pair variant, and for an undulator
  // the reduced equations when its field lies along one axis
  int nz = (f.field[0] != 0) + (f.field[1] != 0) + (f.field[2] != 0);
  if (f.type == kEPU) v.m = kEpuZ;
  else if (nz == 1) v.m = f.field[0] != 0 ? kAxisUndX : (f.field[1] != 0 ? kAxisUndY : kAxisUndZ);
  else v.m = kUndZ;
  return v;
}

}  // namespace om
