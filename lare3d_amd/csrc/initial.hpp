// initial.hpp -- potential_field (initial_conditions.f90:114-296) on the
// device: red-black SOR for the potential phi of a current-free field,
// B = -grad phi, scaled by the largest bz on the lower z boundary.
//
// The reference's colouring depends on (ix + iy) only: x1 restarts at z1
// for every iz (:141-160), so the two passes are checkerboards in x-y and
// each z column of a colour is relaxed from iz = 1 upwards, the point below
// already updated in the same pass.  One thread per column of the colour
// does exactly that; the x and y neighbours belong to the other colour and
// do not change during the pass, so the result is that of the reference's
// sequential loops, bit for bit.  Iterations run in batches without a host
// synchronisation; a pass after the iteration that converged changes
// nothing.
//
// The boundary fills between the passes are folded into the reads.  A wall's
// ghost holds the value its column's neighbour had before this pass, which
// is the value being relaxed itself; a periodic ghost is the point across
// the box (the other colour if the axis has an even number of points; with
// an odd one the ghost is read, and filled by a launch after each pass); the
// lower z ghost is phi(1) plus the flux patch and the upper one zero.
//
// Bound by the latency of a launch and of the column's chain of loads, not
// by bandwidth (a 48^3 box is 18 waves): the loads of the next SOR_U planes
// are issued while this batch is relaxed, which the compiler cannot do
// across the stores, and the largest residual goes to the iteration's slot
// by an atomic maximum (exact, so order does not matter).  An iteration is 2
// launches; with the fills, the reductions and the check as launches of
// their own it was 13.  Per iteration, before and now: 16^3 50.6 and 12.4
// us, 48 x 48 x 40 68.6 and 18.8, 128 x 128 x 100 139 and 46.8.  Batches of
// 4, 12 and 16 planes take 19.1, 20.2 and 20.4 us at 48 x 48 x 40; dividing
// through a reciprocal (a third of the chain's operations) made no difference.
#define SOR_U 8

// State of a batch of iterations: err[q] is the largest |residual| of
// iteration q of the batch (the bits of a non-negative double, which order
// as integers), stop[q] whether the iterations had ended before it.
#define SOR_BATCH 32
struct SorBatch {
  unsigned long long err[SOR_BATCH];
  int stop[SOR_BATCH];
};

__global__ void k_sor_reset(SorBatch *__restrict__ s) {
  const int t = (int)threadIdx.x;
  if (t < SOR_BATCH) {
    s->err[t] = 0;
    s->stop[t] = 0;
  }
}

struct SorArgs {
  double w, dx1, dy1, dz1, tol;
  int q;           // iteration of the batch
  int mapx, mapy;  // 1: wall, 2: wrap to the point across, 0: read the ghost
  int first;       // the first pass of all: phi is zero, ghosts included
};

// One colour pass: z1 = 1 relaxes (ix + iy) even, z1 = 2 (ix + iy) odd.
__global__ __launch_bounds__(64) void k_sor_pass(Geo g, double *__restrict__ phi, const double *__restrict__ flux0,
                                                 int z1, SorArgs a, SorBatch *__restrict__ s) {
  const int ncol = (g.nx + 1) / 2;  // most points of one colour in a row
  const int t = (int)blockIdx.x * 64 + (int)threadIdx.x;
  const int iy = t / ncol + 1, u = t - (iy - 1) * ncol;
  const int x1 = ((iy - 1) & 1) ? 3 - z1 : z1;  // first ix of row iy
  const int ix = x1 + 2 * u;
  const bool in = iy <= g.ny && ix <= g.nx;
  const int Z = g.sz;
  const int c1 = in ? g.idx(ix, iy, 1) : g.idx(1, 1, 1);
  // offsets of the four neighbours from the point (0: the point itself)
  int oxm = -1, oxp = 1, oym = -g.sy, oyp = g.sy;
  if (in) {
    if (a.mapx && ix == 1) oxm = a.mapx == 1 ? 0 : g.nx - 1;
    if (a.mapx && ix == g.nx) oxp = a.mapx == 1 ? 0 : 1 - g.nx;
    if (a.mapy && iy == 1) oym = a.mapy == 1 ? 0 : (g.ny - 1) * g.sy;
    if (a.mapy && iy == g.ny) oyp = a.mapy == 1 ? 0 : (1 - g.ny) * g.sy;
  }
  double v[SOR_U], xm[SOR_U], xp[SOR_U], ym[SOR_U], yp[SOR_U];
  double nv[SOR_U], nxm[SOR_U], nxp[SOR_U], nym[SOR_U], nyp[SOR_U];
  // planes k .. k+SOR_U-1 (planes above nz read plane nz, unused)
  auto fetch = [&](int k) {
#pragma unroll
    for (int q = 0; q < SOR_U; ++q) {
      const int c = c1 + ((k + q < g.nz ? k + q : g.nz) - 1) * Z;
      nv[q] = phi[c];
      nxm[q] = phi[c + oxm];
      nxp[q] = phi[c + oxp];
      nym[q] = phi[c + oym];
      nyp[q] = phi[c + oyp];
    }
  };
  fetch(1);
  const double flux = in && !a.first ? flux0[(ix - 1) + g.nx * (iy - 1)] : 0.0;
  // stopped before this iteration: as the one before it was, or by its
  // residual (pass 1 works it out and keeps it)
  bool stop;
  if (z1 == 1) {
    stop = a.q > 0 && (s->stop[a.q - 1] || __longlong_as_double((long long)s->err[a.q - 1]) < a.tol);
    if (t == 0) s->stop[a.q] = stop;
  } else {
    stop = s->stop[a.q] != 0;
  }
  if (stop) return;  // the same for every thread
  double em = 0.0;
  if (in) {
    const double den = a.dx1 + a.dy1 + a.dz1;
    double below = 0.0;
    for (int k = 1; k <= g.nz; k += SOR_U) {
#pragma unroll
      for (int q = 0; q < SOR_U; ++q) {
        v[q] = nv[q];
        xm[q] = nxm[q];
        xp[q] = nxp[q];
        ym[q] = nym[q];
        yp[q] = nyp[q];
      }
      if (k + SOR_U <= g.nz) fetch(k + SOR_U);
      if (k == 1) below = a.first ? 0.0 : v[0] + flux;
#pragma unroll
      for (int q = 0; q < SOR_U; ++q) {
        if (k + q > g.nz) break;
        const double above = k + q == g.nz ? 0.0 : (q + 1 < SOR_U ? v[q + 1] : nv[0]);
        const double cur = v[q];
        const double r = (((xp[q] - 2.0 * cur) + xm[q]) * a.dx1 + ((yp[q] - 2.0 * cur) + ym[q]) * a.dy1 +
                          ((above - 2.0 * cur) + below) * a.dz1) /
                         2.0 / den;
        below = cur + a.w * r;
        phi[c1 + (k + q - 1) * Z] = below;
        em = dmax(em, fabs(r));
      }
    }
  }
  for (int off = 32; off > 0; off >>= 1) em = dmax(em, __shfl_down(em, off, 64));
  if (threadIdx.x == 0) atomicMax(&s->err[a.q], (unsigned long long)__double_as_longlong(em));
}

// The lower and upper z boundaries of phi_mpi (:268-275): the flux patch
// phi(ix, iy, 0) = phi(ix, iy, 1) + flux0(ix, iy), phi(ix, iy, -1) =
// phi(ix, iy, 0) on 1..nx x 1..ny, and phi = 0 on planes nz+1, nz+2 over
// the whole x-y extent.
__global__ __launch_bounds__(BX * BY) void k_phi_zbc(Geo g, Box b, double *__restrict__ phi,
                                                     const double *__restrict__ flux0) {
  PLANE_POS(b, i, j)
  if (j > b.y1) return;
  if (i >= 1 && i <= g.nx && j >= 1 && j <= g.ny) {
    const int c0 = g.idx(i, j, 0);
    const double p0 = phi[c0 + g.sz] + flux0[(i - 1) + g.nx * (j - 1)];
    phi[c0] = p0;
    phi[c0 - g.sz] = p0;
  }
  phi[g.idx(i, j, g.nz + 1)] = 0.0;
  phi[g.idx(i, j, g.nz + 2)] = 0.0;
}

__global__ __launch_bounds__(BX * BY) void k_fill64(Geo g, Box b, double *__restrict__ a, double v) {
  BOX_INDEX(b, i, j, k);
  a[g.idx(i, j, k)] = v;
}

// B = -grad phi on the faces the reference sets (:198-218): bx on
// 0..nx x 1..ny x 1..nz, by on 1..nx x 0..ny x 1..nz, bz on
// 1..nx x 1..ny x 0..nz; every other face keeps its value.
__global__ __launch_bounds__(BX * BY) void k_phi_to_b(Geo g, Box b, const double *__restrict__ phi,
                                                      double *__restrict__ bx, double *__restrict__ by,
                                                      double *__restrict__ bz) {
  BOX_INDEX(b, i, j, k);
  const int c = g.idx(i, j, k);
  const bool in_x = i >= 1 && i <= g.nx, in_y = j >= 1 && j <= g.ny, in_z = k >= 1 && k <= g.nz;
  if (i >= 0 && i <= g.nx && in_y && in_z) bx[c] = -(phi[c + 1] - phi[c]) / g.dxc[i];
  if (in_x && j >= 0 && j <= g.ny && in_z) by[c] = -(phi[c + g.sy] - phi[c]) / g.dyc[j];
  if (in_x && in_y && k >= 0 && k <= g.nz) bz[c] = -(phi[c + g.sz] - phi[c]) / g.dzc[k];
}

// -bz on the lower boundary plane bz(1:nx, 1:nz, 0) (the y range is 1:nz
// in the reference, :221): per-block partial of the minimum.
__global__ __launch_bounds__(BX * BY) void k_bz_lower(Geo g, Box b, const double *__restrict__ bz,
                                                      double *__restrict__ partial) {
  PLANE_POS(b, i, j)
  double v[1] = {LARGEST};
  if (j <= b.y1) v[0] = -bz[g.idx(i, j, 0)];
  const int ops[1] = {0};
  block_reduce_store<1>(v, ops, partial);
}

// B / bz_max over whole arrays (:224-226); s[15] holds -bz_max.
__global__ __launch_bounds__(BX * BY) void k_scale_b(Geo g, Box b, double *__restrict__ bx, double *__restrict__ by,
                                                     double *__restrict__ bz, const double *__restrict__ s) {
  BOX_INDEX(b, i, j, k);
  const int c = g.idx(i, j, k);
  const double bm = -s[15];
  bx[c] = bx[c] / bm;
  by[c] = by[c] / bm;
  bz[c] = bz[c] / bm;
}
