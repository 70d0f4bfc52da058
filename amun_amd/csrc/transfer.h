// transfer.h -- the state between the block pool and the host's layouts.
//
// The host hands over and takes global arrays U[nv][nz][ny][nx], block arrays
// u(nv, im, jm, km) with ghost layers, or block interiors.  These kernels
// convert between them and the pool's bricks in a device buffer, so that the
// copy over the bus is one contiguous block straight into the caller's
// memory.  Bound by the bus (the conversion of 1.2 GB takes 1 ms); the same
// conversion by a host loop over a host copy took 0.37 s of the 0.49 s of a
// 256^3 MHD download.
#pragma once

namespace amun_dev {

// block range and grid of one run: blocks b0 .. of ir x jr x kr blocks, in x,
// y, z order
struct GridShape {
  int b0, ir, jr, kr;
};

// x in the pool's element type TX to and from the global array of one run,
// one thread per cell of the global array and variable (blockIdx.y)
template <typename TX, bool kToPool>
static __global__ __launch_bounds__(256) void k_grid_transfer(
    std::conditional_t<kToPool, TX, const TX>* __restrict__ X,
    std::conditional_t<kToPool, const double, double>* __restrict__ G, GridShape s, RunConst rc,
    int nv) {
  const int nc = rc.nc, nx = s.ir * nc, ny = s.jr * nc, v = blockIdx.y;
  const long long n = (long long)nx * ny * (rc.nd == 3 ? s.kr * nc : 1);
  for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < n;
       g += (long long)gridDim.x * blockDim.x) {
    const int x = (int)(g % nx);
    const long long r = g / nx;
    const int y = (int)(r % ny), z = (int)(r / ny);
    const int bx = x / nc, by = y / nc, bz = z / nc;
    const size_t b = (size_t)s.b0 + ((size_t)bz * s.jr + by) * s.ir + bx;
    const size_t o = (b * nv + v) * (size_t)rc.ncell +
                     lidx<sizeof(TX)>(nc, rc.nd, x - bx * nc, y - by * nc, z - bz * nc);
    if constexpr (kToPool) X[o] = TX(G[(size_t)v * n + g]);
    else G[(size_t)v * n + g] = double(X[o]);
  }
}

// a run's blocks at h, a host copy of its part of the pool, into its global
// array u (small runs, see kHostBytes)
template <typename T>
static void blocks_to_grid(const GridShape& s, const RunConst& rc, int nv, const T* h, double* u) {
  const int nc = rc.nc, kn = rc.nd == 3 ? nc : 1;
  const size_t nx = (size_t)s.ir * nc, ny = (size_t)s.jr * nc, nz = (size_t)s.kr * kn;
  for (int b = 0; b < s.ir * s.jr * s.kr; b++) {
    const size_t x0 = (size_t)(b % s.ir) * nc, y0 = (size_t)(b / s.ir % s.jr) * nc;
    const size_t z0 = (size_t)(b / (s.ir * s.jr)) * kn;
    for (int v = 0; v < nv; v++, h += rc.ncell)
      for (int k = 0; k < kn; k++)
        for (int j = 0; j < nc; j++) {
          double* row = u + ((v * nz + z0 + k) * ny + y0 + j) * nx + x0;
          for (int i = 0; i < nc; i++) row[i] = double(h[lidx<sizeof(T)>(nc, rc.nd, i, j, k)]);
        }
  }
}

// the interiors h of nblk host blocks u with ng ghost layers, variables
// fastest: a row of cells is contiguous in both
static void interiors_of(const RunConst& rc, int nv, int ng, int nblk, const double* u,
                         double* h) {
  const int nc = rc.nc, m = nc + 2 * ng;
  const int kn = rc.nd == 3 ? nc : 1, km = rc.nd == 3 ? m : 1, kg = rc.nd == 3 ? ng : 0;
  const size_t row = (size_t)nc * nv;
  for (int b = 0; b < nblk; b++)
    for (int k = 0; k < kn; k++)
      for (int j = 0; j < nc; j++, h += row)
        std::memcpy(h, u + ((((size_t)b * km + (k + kg)) * m + (j + ng)) * m + ng) * nv,
                    row * sizeof(double));
}

// conserved state of blocks b0 .. b0 + nb - 1 to and from arrays of m^d cells
// a block, variables fastest, of which the first ng along each axis lie
// before the interior (ng = 0 and m = nc: interiors); to the pool, the ghost
// cells are skipped
template <bool kToPool>
static __global__ __launch_bounds__(256) void k_block_transfer(
    std::conditional_t<kToPool, double, const double>* __restrict__ U,
    std::conditional_t<kToPool, const double, double>* __restrict__ B, int b0, int nb, int m,
    int ng, RunConst rc, int nv) {
  const int nc = rc.nc, kg = rc.nd == 3 ? ng : 0, km = rc.nd == 3 ? m : 1;
  const int kn = rc.nd == 3 ? nc : 1;
  const long long per = (long long)nc * nc * kn * nv, n = per * nb;
  for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < n;
       g += (long long)gridDim.x * blockDim.x) {
    const int b = (int)(g / per), q = (int)(g - (long long)b * per);
    const int v = q % nv, cell = q / nv;
    const int i = cell % nc, j = (cell / nc) % nc, k = cell / (nc * nc);
    const size_t o = ((size_t)(b0 + b) * nv + v) * rc.ncell + lidx<8>(nc, rc.nd, i, j, k);
    const size_t h = ((((size_t)b * km + (k + kg)) * m + (j + ng)) * m + (i + ng)) * nv + v;
    if constexpr (kToPool) U[o] = B[h];
    else B[h] = U[o];
  }
}

// blocks b0 .. b0 + nb - 1 with their ghost layers from the filled primitive
// pool Q: the primitives, or (U given) the conserved state, in the interior
// U itself and in the ghost cells prim2cons of the primitives
// (update_ghost_cells, boundaries.F90:6633-6736; equations.F90:1360, 1762,
// 2220, 2815), rounded as the reference rounds it
template <class P, typename TQ>
static __global__ __launch_bounds__(256) void k_blocks_ghosts(
    const TQ* __restrict__ Q, const double* __restrict__ U, double* __restrict__ out,
    const int* __restrict__ nbr, RunConst rc, int ng, int b0, int nb) {
#pragma clang fp contract(off)
  constexpr int NV = P::nv;
  const int nc = rc.nc, im = nc + 2 * ng, km = rc.nd == 3 ? im : 1, kg = rc.nd == 3 ? ng : 0;
  const long long per = (long long)im * im * km, n = per * nb;
  for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < n;
       g += (long long)gridDim.x * blockDim.x) {
    const int b = b0 + (int)(g / per);
    const int r = (int)(g % per);
    const int i = r % im - ng, j = (r / im) % im - ng, k = r / (im * im) - kg;
    double* o = out + (size_t)g * NV;
    if (U && i >= 0 && i < nc && j >= 0 && j < nc && k >= 0 && k < (rc.nd == 3 ? nc : 1)) {
      const size_t at = (size_t)b * NV * rc.ncell + lidx<8>(nc, rc.nd, i, j, k);
      for (int v = 0; v < NV; v++) o[v] = U[at + (size_t)v * rc.ncell];
      continue;
    }
    const size_t pk = cell_index<sizeof(TQ)>(nbr, rc, b, i, j, k);
    double q[NV];
    for (int v = 0; v < NV; v++) q[v] = double(Q[var_index<NV>(rc, pk, v)]);
    if (!U) {
      for (int v = 0; v < NV; v++) o[v] = q[v];
      continue;
    }
    const double mx = q[0] * q[1], my = q[0] * q[2], mz = q[0] * q[3];
    o[0] = q[0];
    o[1] = mx;
    o[2] = my;
    o[3] = mz;
    if constexpr (P::iso) {
      for (int v = 4; v < NV; v++) o[v] = q[v];
    } else {
      const double ek = 0.5 * ((mx * q[1] + my * q[2]) + mz * q[3]);
      const double ei = q[NV - 1] / rc.gammam1;
      if constexpr (P::mhd) {
        for (int v = 4; v < 8; v++) o[v] = q[v];
        const double em = 0.5 * ((q[4] * q[4] + q[5] * q[5]) + q[6] * q[6]);
        o[8] = (ei + ek) + em;
      } else {
        o[4] = ei + ek;
      }
    }
  }
}

}  // namespace amun_dev
