// launch.h -- launch shapes of the sweeps: workgroups, lanes and LDS.  Plain
// C++ (no HIP): the kernels, the host side and its CPU test share it.
#pragma once

#include <cstddef>

namespace amun_dev {

// LDS, in elements of T: the pencils' primitive state with R + 1 cells beyond
// each end, then in its place the upper face states, then the fluxes.  The
// width of a pencil's row is the smallest that spreads the lanes of a wave
// over all banks: four cells by four pencils (x), four pencils by sixteen
// cells (y), one cell each (z).
constexpr int row_width(int n, int dir) {
  return dir == 0 ? (n + 3) / 8 * 8 + 4 : (dir == 1 ? (n + 7) / 16 * 16 + 8 : n | 1);
}
constexpr int tile_width(int nc, int R, int dir) {
  return row_width(nc + 2 * (R + 1), dir);
}
constexpr int face_width(int nc, int dir) { return row_width(nc + 1, dir); }
// Whether the solver leaves registers for the cell's increment and states
// (HD, and every FP32 system but the relativistic: at most 10 words a state);
// where not, the increment of the directions before waits in LDS: read at the
// update instead, it cost 0.5 ms of a 256^3 FP64 MHD step, and early in
// registers it spilled.
constexpr bool sweep_loads_early(int nv, int es, bool sr) {
  return nv * es <= 40 && !sr;
}
constexpr bool sweep_inc_lds(int nv, int es, bool sr, int R, int dir) {
  return R > 0 && dir > 0 && !sweep_loads_early(nv, es, sr);
}
constexpr size_t sweep_lds_elems(int nv, int es, bool sr, int R, int nc, int np, int dir) {
  const int w = R ? tile_width(nc, R, dir) : face_width(nc, dir);
  return (size_t)nv * np * (w + (sweep_inc_lds(nv, es, sr, R, dir) ? nc : 0));
}

// what the shape of a sweep depends on
struct SweepCfg {
  int nv, es;          // variables, bytes of an element
  bool sr;             // relativistic
  int R;               // half width of the reconstruction's window
  int nd, nc, nblk;
};

// np pencils of nc + 2 lanes each per workgroup, the lanes, the workgroups and
// the LDS in bytes
struct SweepShape {
  int np, lanes;
  unsigned grid;
  size_t lds;
};

// Of the even np with at most wg lanes (at least two pencils), the one that
// leaves the fewest lanes idle: 14 pencils on 252 of 256 lanes at nc = 16.
constexpr SweepShape sweep_shape(const SweepCfg& c, int dir, int wg) {
  const long long total = (long long)c.nblk * (c.nd == 3 ? c.nc * c.nc : c.nc);
  const auto lanes = [&](int np) { return (np * (c.nc + 2) + 63) / 64 * 64; };
  SweepShape s{2, 0, 0, 0};
  for (int np = 2; lanes(np) <= wg; np += 2)
    if ((long long)np * lanes(s.np) >= (long long)s.np * lanes(np)) s.np = np;
  s.lanes = lanes(s.np);
  s.grid = (unsigned)((total + s.np - 1) / s.np);
  s.lds = sweep_lds_elems(c.nv, c.es, c.sr, c.R, c.nc, s.np, dir) * (size_t)c.es;
  return s;
}

// The shape that a sweep is launched with.  A workgroup size that was chosen
// (amun_dev_set_launch, amun_dev_autotune) holds.  wg = 0, the default: 256,
// and on a grid that leaves CUs idle with it 128, then 64, until every CU has
// a workgroup (us a step replayed from graphs with 256, 128, 64 lanes: 128^2
// HD 36.7, 34.9, 33.8; with 128 and 64: 64^2 HD 34.6, 32.5, 64^2 MHD 60.9,
// 57.1, 16^3 MHD WENO5-Z 76.6, 72.1).  With more workgroups than CUs the
// larger ones waste fewer lanes: 512^2 SRMHD y sweep 75 us with 256, 83 with
// 128, 106 with 64.
constexpr unsigned kComputeUnits = 256;
constexpr SweepShape launch_shape(const SweepCfg& c, int dir, int wg) {
  if (wg) return sweep_shape(c, dir, wg);
  SweepShape s = sweep_shape(c, dir, 256);
  for (int w = 128; w >= 64 && s.grid < kComputeUnits; w /= 2) s = sweep_shape(c, dir, w);
  return s;
}

// The largest LDS of any launch of a sweep kernel, over the block sizes that a
// context may have and the three workgroup sizes.  The limit of dynamic LDS
// belongs to the kernel, which all contexts of a process share: set to one
// context's own need it fell below another's (FP64 MHD WENO5-Z along y: 83 KB
// at 4 cells a block, 39 KB at 16).
constexpr int kMinCells = 4, kMaxCells = 64;
constexpr size_t sweep_lds_limit(SweepCfg c, int dir) {
  size_t most = 0;
  for (c.nc = kMinCells; c.nc <= kMaxCells; c.nc += 4)
    for (int wg = 64; wg <= 256; wg *= 2) {
      const size_t lds = sweep_shape(c, dir, wg).lds;
      if (lds > most) most = lds;
    }
  return most;
}

}  // namespace amun_dev
