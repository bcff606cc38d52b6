// runtime.hpp -- device state, launch sequencing and the entry points of one
// precision mode.  lare_dev.hip includes this file twice: in namespace fp64
// with LARE_REAL = double and in namespace fp32 with LARE_REAL = float.
// `real` is the storage type of the bulk fields (density, energy, velocity,
// their Lagrangian and remap work arrays, conduction stages); the face
// magnetic field, its constrained-transport fluxes and resistive EMFs, the
// metrics and every reduction stay FP64, and kernels do their arithmetic in
// FP64 registers.  No include guard: one inclusion per namespace.
typedef LARE_REAL real;
// Arithmetic type of the bulk kernels that have been given one: double in
// the FP64 mode (the reference's arithmetic), float in the FP32 mode.  The
// face field's CT updates, the limiter comparisons and every reduction
// stay FP64 in both.
typedef LARE_ACC acc;

#include "common.hpp"
#include "bc.hpp"
#include "conduct.hpp"
#include "lagran.hpp"
#include "remap.hpp"
#include "surrogate.hpp"
#include "initial.hpp"
#include "neutral.hpp"
#include "openbc.hpp"

// ----------------------------------------------------------------------------
// kernel timing with HIP events on the library stream
// ----------------------------------------------------------------------------
struct ProfRec {
  const char *name;
  hipEvent_t a, b;
};
struct ProfAcc {
  std::string name;
  int count;
  double ms;
};

struct Dev {
  bool ready = false, loaded = false;
  int n[3];
  int sy, sz;
  size_t ntot;
  int bc[6];
  int per[3], user[3];
  bool any_open = false;  // some side is BC_OPEN
  bool clamp = false;     // predictor and corrector of this step clamp the energy they read
  lare_params p;
  double tfac, visc2_norm;
  hipStream_t stream = nullptr;
  double *metric = nullptr;  // 7 arrays of length nmax+5, index i+2
  Geo g;
  // state (bulk fields in the storage precision, face B in FP64)
  real *rho, *rho_alt, *energy, *vx, *vy, *vz, *vx1, *vy1, *vz1;
  double *bx, *by, *bz;
  real *eta, *visc3, *visc_dep, *ohmic_dep;
  // lagrangian scratch
  real *rho_v, *cs_v, *al1, *al2, *al3, *visc_heat, *p0, *pp;
  double *bpx, *bpy, *bpz;       // predictor B
  double *fxr, *fyr, *fzr;       // spare face arrays: a CT sweep's or resistive substep's new B
  real *qx, *qy, *qz;
  // remap scratch: volumes and width (with some Lagrangian arrays: remap_db1,
  // remap_vol), the mass flux, and where the new energy and velocities go
  real *cv1, *cv2, *db1, *Fe, *dm, *Fx, *Fy, *Fz;
  double *F, *F2;  // the potential field's potential and flux patch
  // conduction scratch
  real *larsen, *Lc, *Yb[3];
  // options: gamma_boris (boris), cool_term_v / cool_term_b and the stored
  // curlb of the ohmic cooling (cooling_term); NULL when off
  real *gamma_boris = nullptr, *cool_v = nullptr, *cool_b = nullptr, *curlb = nullptr;
  // rke: delta_ke (cells) and one sweep's edge terms per velocity component
  real *delta_ke = nullptr;
  RkeOut rk = {};
  // FOURTHORDER: one stage's EMFs and curlb, and their weighted sum
  RkK rk4k = {}, rk4s = {};
  // partially ionised EOS: xi_n (cells), eta_perp (nodes, with Cowling), the
  // bracket fault flag of neutral_fraction; ip = ionise_pot (EOS_ION only)
  real *xi = nullptr, *eta_perp = nullptr;
  int *nf_flag = nullptr;
  // BC_OPEN: the pre-corrector energy and density of each open face's first
  // interior layer (6 faces x 2 fields x (nmax+2)^2)
  double *obc_save = nullptr;
  size_t obc_face = 0;
  bool pi_eos = false;
  double ip = 0.0;
  // reductions
  double *partial = nullptr;
  size_t partial_cap = 0;
  double *dscal = nullptr;   // device scalars: [0..3] last reduce, [8] tvh acc, [9] toh acc
  double *hscal = nullptr;   // pinned host mirror of dscal, and the ticket of the last fold written
  unsigned long long ticket = 0;  // tickets handed out
  std::vector<void *> allocs;
  // host scalars
  double dt = 0.0, dt2 = 0.0, dtr = 0.0, time = 0.0;
  int n_s_stages = 0, peak_substeps = 0, last_substeps = 0, first_set_dt = 1, step = 0;
  // profiling
  bool prof = false;
  std::vector<ProfRec> pending;
  std::vector<hipEvent_t> pool;
  std::vector<ProfAcc> acc;
};

Dev S;

hipEvent_t ev_get() {
  if (!S.pool.empty()) {
    hipEvent_t e = S.pool.back();
    S.pool.pop_back();
    return e;
  }
  hipEvent_t e;
  (void)hipEventCreate(&e);
  return e;
}

void prof_flush() {
  if (S.pending.empty()) return;
  (void)hipStreamSynchronize(S.stream);
  for (auto &r : S.pending) {
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, r.a, r.b);
    bool found = false;
    for (auto &a : S.acc)
      if (a.name == r.name) {
        a.count++;
        a.ms += ms;
        found = true;
        break;
      }
    if (!found) S.acc.push_back({r.name, 1, (double)ms});
    S.pool.push_back(r.a);
    S.pool.push_back(r.b);
  }
  S.pending.clear();
}

struct ProfScope {
  const char *name;
  hipEvent_t a = nullptr;
  explicit ProfScope(const char *n) : name(n) {
    if (S.prof) {
      a = ev_get();
      (void)hipEventRecord(a, S.stream);
    }
  }
  ~ProfScope() {
    if (S.prof) {
      hipEvent_t b = ev_get();
      (void)hipEventRecord(b, S.stream);
      S.pending.push_back({name, a, b});
      if (S.pending.size() > 4096) prof_flush();
    }
  }
};

#define LAUNCH(name, kern, grid, block, ...)                                   \
  do {                                                                         \
    ProfScope ps_(name);                                                       \
    hipLaunchKernelGGL(kern, grid, block, 0, S.stream, __VA_ARGS__);           \
    hipError_t e_ = hipGetLastError();                                         \
    if (e_ != hipSuccess) return fail(-(int)e_, "launch %s: %s", name, hipGetErrorString(e_)); \
  } while (0)

#define LAUNCH_BOX(name, kern, box, ...) LAUNCH(name, kern, box_grid(box), box_block(), S.g, box, __VA_ARGS__)

int nx() { return S.n[0]; }
int ny() { return S.n[1]; }
int nz() { return S.n[2]; }
Box full_box() { return mkbox(-2, nx() + 2, -2, ny() + 2, -2, nz() + 2); }
Box cell_box() { return mkbox(-1, nx() + 2, -1, ny() + 2, -1, nz() + 2); }
Box interior() { return mkbox(1, nx(), 1, ny(), 1, nz()); }
Box nodes0n() { return mkbox(0, nx(), 0, ny(), 0, nz()); }

// grid of k_resist over the padded box b: tiles of RS_OUT_X x RS_OUT_Y
// written nodes, b.zc (set here) planes per block
dim3 resist_grid(Box &b, int *tiles_x) {
  *tiles_x = (b.x1 - b.x0 + RS_OUT_X) / RS_OUT_X;
  const int tiles = *tiles_x * ((b.y1 - b.y0 + RS_OUT_Y) / RS_OUT_Y);
  b.zc = march_chunk((unsigned)tiles, b.z1 - b.z0 + 1);
  return dim3((unsigned)tiles, 1, (unsigned)((b.z1 - b.z0 + b.zc) / b.zc));
}

// the box whose zchunk grid a launch marching along axis M (1, 2) uses:
// y and z ranges swapped for M = 1 (MCOLUMN)
Box march_box(const Box &b, int M) {
  return M == 2 ? b : Box{b.x0, b.x1, b.z0, b.z1, b.y0, b.y1, b.zc};
}

// b with the chunk of a launch of plane_blocks columns marching along axis M
Box marched(Box b, int M = 2) {
  const Box m = march_box(b, M);
  b.zc = march_chunk(plane_blocks(m), m.z1 - m.z0 + 1);
  return b;
}

// grid of a z-marching launch: BX*BY columns, b.zc planes per block
dim3 zchunk_grid(const Box &b) { return dim3(plane_blocks(b), 1, (unsigned)((b.z1 - b.z0 + b.zc) / b.zc)); }

// reduction over partials of a grid launched from index 0 on every axis
dim3 grid_from0(int x1, int y1, int z1) { return box_grid(mkbox(0, x1, 0, y1, 0, z1)); }

// Reduction of the per-block partials (rows of nv values; bit q of minmask
// selects min, else sum).  Up to RED_DIRECT rows one block folds them all (at
// most four per thread); beyond, RED_ROWS blocks each fold one contiguous
// chunk of rows and one block folds the RED_ROWS results.  The last block
// stores (or adds) the nv scalars, in device memory and in the pinned host
// mirror, so that reading them takes a synchronisation and no copy: a
// reduction read by the host was three launches (the copy is one), 12 to 14
// us at any size, and is one or two.
#define RED_ROWS 512
#define RED_DIRECT 1024

__global__ __launch_bounds__(256) void k_reduce_rows(const double *__restrict__ partial, int nrows, int nv, int minmask,
                                                     int chunk, double *__restrict__ level1) {
  const int r0 = (int)blockIdx.x * chunk;
  const int r1 = r0 + chunk < nrows ? r0 + chunk : nrows;
  fold_rows(partial, r0, r1, nv, minmask, level1 + (size_t)blockIdx.x * nv, 0);
}

__global__ __launch_bounds__(256) void k_final_reduce(const double *__restrict__ level1, int nrows, int nv, int minmask,
                                                      int accumulate, double *__restrict__ out, HostOut host) {
  fold_rows(level1, 0, nrows, nv, minmask, out, accumulate, host);
}

// Rows per level-1 block of a fold of nb rows and the number of level-1
// results; 0 (and nb rows) when one block folds the rows directly.
int fold_chunk(int nb, int *rows) {
  *rows = nb;
  if (nb <= RED_DIRECT) return 0;
  const int chunk = (nb + RED_ROWS - 1) / RED_ROWS;
  *rows = (nb + chunk - 1) / chunk;  // every level-1 block has >= 1 row
  return chunk;
}

// the pinned mirror of scalar `slot`, and the ticket of a fold that writes it
HostOut host_out(int slot) {
  return HostOut{S.hscal + slot, (unsigned long long *)(S.hscal + 16), ++S.ticket};
}

int final_reduce(dim3 grid, int nv, int minmask, int slot, int accumulate) {
  const int nb = (int)(grid.x * grid.y * grid.z);
  if (nv > RED_MAXV || (size_t)nb * nv > S.partial_cap)
    return fail(LARE_E_ARG, "reduction of %d x %d values exceeds the partial buffer", nb, nv);
  const double *rows = S.partial;
  int nrows = nb;
  if (const int chunk = fold_chunk(nb, &nrows)) {
    double *level1 = S.partial + S.partial_cap;
    LAUNCH("reduce_rows", k_reduce_rows, dim3(nrows), dim3(256), S.partial, nb, nv, minmask, chunk, level1);
    rows = level1;
  }
  LAUNCH("final_reduce", k_final_reduce, dim3(1), dim3(256), rows, nrows, nv, minmask, accumulate, S.dscal + slot,
         host_out(slot));
  return 0;
}

// the fold of one accumulated sum as a job for the launch that follows: the
// level-1 rows are formed here if there are many
int fold_job(dim3 grid, int slot, FoldJob *job) {
  const int nb = (int)(grid.x * grid.y * grid.z);
  if ((size_t)nb > S.partial_cap) return fail(LARE_E_ARG, "reduction of %d values exceeds the partial buffer", nb);
  job->rows = S.partial;
  if (const int chunk = fold_chunk(nb, &job->nrows)) {
    double *level1 = S.partial + S.partial_cap;
    LAUNCH("reduce_rows", k_reduce_rows, dim3(job->nrows), dim3(256), S.partial, nb, 1, 0, chunk, level1);
    job->rows = level1;
  }
  job->out = S.dscal + slot;
  job->host = host_out(slot);
  return 0;
}

// The scalars once the last fold queued has written them: it sets its ticket in
// the pinned mirror, which is seen some microseconds before a stream
// synchronisation returns (a 16^3 step: 157 -> 149 us, 64^3: 322 -> 317).  After SPIN_POLLS looks, some
// hundred microseconds, the wait is left to the runtime.
#define SPIN_POLLS 20000
int read_scalars(int slot, int count, double *out) {
  volatile unsigned long long *t = (volatile unsigned long long *)(S.hscal + 16);
  int q = 0;
  while (q < SPIN_POLLS && *t < S.ticket) {
    __builtin_ia32_pause();
    ++q;
  }
  if (*t < S.ticket) HIPCHK(hipStreamSynchronize(S.stream));
  for (int k = 0; k < count; ++k) out[k] = ((volatile double *)S.hscal)[slot + k];
  return 0;
}

// ----------------------------------------------------------------------------
// boundary groups
// ----------------------------------------------------------------------------
enum FieldKind { FK_CELL, FK_NODE, FK_BX, FK_BY, FK_BZ };

// the fields of h that NB, NC and NN say, every axis at once
template <int NB, int NC, int NN>
int fill_halo(const HaloSet &h, const char *name, const FoldJob &job = FoldJob{}) {
  LAUNCH(name, (k_halo<NB, NC, NN>), dim3(halo_blocks(S.g) + (job.rows ? 1 : 0)), dim3(256), S.g, h, job);
  return 0;
}

// the state's fields, with v1 after v
HaloSet state_halo() {
  return {{S.bx, S.by, S.bz}, {S.energy, S.rho}, {S.vx, S.vy, S.vz, S.vx1, S.vy1, S.vz1}};
}
int bfield_bcs(double *bx, double *by, double *bz) {
  HaloSet h = state_halo();
  h.b[0] = bx;
  h.b[1] = by;
  h.b[2] = bz;
  return fill_halo<1, 0, 0>(h, "bc_bfield");
}
int energy_bcs() { return fill_halo<0, 1, 0>(state_halo(), "bc_energy"); }
int node_bcs(real *ux, real *uy, real *uz, const char *name) {
  HaloSet h = state_halo();
  h.node[0] = ux;
  h.node[1] = uy;
  h.node[2] = uz;
  return fill_halo<0, 0, 3>(h, name);
}
int boundary_conditions() { return fill_halo<1, 2, 3>(state_halo(), "bc_all"); }

// ----------------------------------------------------------------------------
// conduction
// ----------------------------------------------------------------------------
CondArgs cond_args() {
  CondArgs ca;
  ca.kappa_0 = S.p.kappa_0;
  ca.tfac = S.tfac;
  ca.dt = S.dt;
  ca.xi = S.pi_eos ? S.xi : nullptr;
  ca.gm1 = S.p.gamma - 1.0;
  ca.ip = S.ip;
  return ca;
}

int calc_s_stages() {
  const Box b = marched(nodes0n());
  const dim3 gr = zchunk_grid(b);
  if (S.pi_eos)
    LAUNCH("larsen", k_larsen<true>, gr, box_block(), S.g, b, S.energy, S.rho, S.larsen, S.partial, S.p.flux_limiter,
           S.p.kappa_0, cond_args(), S.p.heat_flux_limiter);
  else
    LAUNCH("larsen", k_larsen<false>, gr, box_block(), S.g, b, S.energy, S.rho, S.larsen, S.partial, S.p.flux_limiter,
           S.p.kappa_0, cond_args(), S.p.heat_flux_limiter);
  int rc = final_reduce(gr, 1, 1, 0, 0);
  if (rc) return rc;
  double dtp;
  rc = read_scalars(0, 1, &dtp);
  if (rc) return rc;
  // the reference starts its minimum at 1e10 (conduct.f90:110)
  double dt_parab = dtp < 1.0e10 ? dtp : 1.0e10;
  dt_parab = 0.9 * dt_parab / sqrt(3.0);
  const double stages = 0.5 * (sqrt(9.0 + 16.0 * (S.dt / dt_parab)) - 1.0);
  int ns = (int)ceil(stages);
  if (ns % 2 == 0) ns = ns + 1;
  S.n_s_stages = ns;
  return 0;
}

// blocks per plane of a launch of waves that own `out` points each of a plane
// of npts points
unsigned wave_blocks(long npts, int out) { return (unsigned)(((npts + out - 1) / out + BY - 1) / BY); }

// grid of the z-marching stage kernels over the interior box (in.zc set
// here): waves of RKL_OUT cells over rows of x0-1..x1
dim3 rkl2_grid(Box &in) {
  const unsigned pb = wave_blocks((long)(in.x1 - in.x0 + 2) * (in.y1 - in.y0 + 1), RKL_OUT);
  in.zc = march_chunk(pb, in.z1 - in.z0 + 1);
  return dim3(pb, 1, (unsigned)((in.z1 - in.z0 + in.zc) / in.zc));
}
// stage 1 from E0 (ghosts as stored): Lc and Y1 = E0 + mu_t1 dt Lc
int rkl2_stage1(const real *E0, real *Yout, CondArgs ca, double mu_t1) {
  Box in = interior();
  const dim3 gr = rkl2_grid(in);
  // the stage-1 read is direct: no ghost mapping, BC_OPEN or not
  if (ca.xi)
    LAUNCH("rkl2_stage1", (k_rkl2_z<TMODE_DIRECT, 1, true, false>), gr, box_block(), S.g, in, E0, E0, E0,
           S.rho, S.bx, S.by, S.bz, S.larsen, S.Lc, Yout, ca, 0.0, 0.0, 0.0, mu_t1, 0.0);
  else
    LAUNCH("rkl2_stage1", (k_rkl2_z<TMODE_DIRECT, 1, false, false>), gr, box_block(), S.g, in, E0, E0, E0,
           S.rho, S.bx, S.by, S.bz, S.larsen, S.Lc, Yout, ca, 0.0, 0.0, 0.0, mu_t1, 0.0);
  return 0;
}
// stage j >= 2 from Y2 (and Y1, E0, Lc) under a ghost-read mode
int rkl2_stage(int mode, const real *Y2, const real *Y1, const real *E0, real *Yout, CondArgs ca, double mu, double nu,
               double one_m_mu_nu, double mu_t, double gam_t) {
  Box in = interior();
  const dim3 gr = rkl2_grid(in);
#define RKL2_STAGE(M, P, O)                                                                                       \
  LAUNCH("rkl2_stage", (k_rkl2_z<M, 0, P, O>), gr, box_block(), S.g, in, Y2, Y1, E0, S.rho, S.bx, S.by, \
         S.bz, S.larsen, S.Lc, Yout, ca, mu, nu, one_m_mu_nu, mu_t, gam_t)
  if (S.any_open) {
    if (mode == TMODE_STALE) {
      if (ca.xi) RKL2_STAGE(TMODE_STALE, true, true);
      else RKL2_STAGE(TMODE_STALE, false, true);
    } else {
      if (ca.xi) RKL2_STAGE(TMODE_WRAP, true, true);
      else RKL2_STAGE(TMODE_WRAP, false, true);
    }
  } else if (mode == TMODE_STALE) {
    if (ca.xi) RKL2_STAGE(TMODE_STALE, true, false);
    else RKL2_STAGE(TMODE_STALE, false, false);
  } else {
    if (ca.xi) RKL2_STAGE(TMODE_WRAP, true, false);
    else RKL2_STAGE(TMODE_WRAP, false, false);
  }
#undef RKL2_STAGE
  return 0;
}

int neutral_fraction(const real *Y, int mode);
EosArgs eos_args();

// RKL2 super-step; delta_mode = 1 inside lagrangian_step
int heat_conduct_sts2(int delta_mode) {
  const int s = S.n_s_stages;
  if (s <= 1) {  // the reference's Y(3) is never written: energy unchanged
    if (delta_mode) LAUNCH_BOX("energy_max", k_energy_max, cell_box(), S.energy);
    return 0;
  }
  std::vector<double> b(s + 1), a(s + 1), mu_t(s + 1), mu(s + 1), nu(s + 1), gt(s + 1);
  const double ds = (double)s;
  const double omega_1 = 4.0 / (ds * ds + ds - 2.0);
  for (int j = 0; j <= 2; ++j) b[j] = 1.0 / 3.0;
  for (int j = 3; j <= s; ++j) {
    const double dj = (double)j;
    b[j] = (dj * dj + dj - 2.0) / (2.0 * dj * (dj + 1.0));
  }
  for (int j = 0; j <= s; ++j) a[j] = 1.0 - b[j];
  mu_t[1] = omega_1 / 3.0;
  for (int j = 2; j <= s; ++j) {
    const double dj = (double)j;
    mu_t[j] = ((2.0 * dj - 1.0) / dj) * omega_1 * (b[j] / b[j - 1]);
    mu[j] = ((2.0 * dj - 1.0) / dj) * (b[j] / b[j - 1]);
    nu[j] = -1.0 * ((dj - 1.0) / dj) * (b[j] / b[j - 2]);
    gt[j] = -1.0 * a[j - 1] * mu_t[j];
  }
  CondArgs ca = cond_args();
  real *E0 = S.energy;
  real *outp = S.Yb[0];
  int rc = rkl2_stage1(E0, S.Yb[0], ca, mu_t[1]);
  if (rc) return rc;
  real *y1 = E0, *y2 = outp;
  int next = 1;
  for (int j = 2; j <= s; ++j) {
    real *yo = S.Yb[next];
    next = (next + 1) % 3;
    rc = rkl2_stage(j == 2 ? TMODE_STALE : TMODE_WRAP, y2, y1, E0, yo, ca, mu[j], nu[j], (1.0 - mu[j]) - nu[j],
                    mu_t[j], gt[j]);
    if (rc) return rc;
    // the neutral fraction of the stage value with its boundary fill
    // (conduct.f90:400-405), read by the next stage's temperatures
    if (S.pi_eos && j < s) {
      rc = neutral_fraction(yo, TMODE_WRAP);
      if (rc) return rc;
    }
    y1 = y2;
    y2 = yo;
  }
  LAUNCH_BOX("rkl2_final", k_rkl2_final, cell_box(), y2, S.energy, delta_mode);
  return 0;
}

// ----------------------------------------------------------------------------
// remap
// ----------------------------------------------------------------------------
int strides(int ax) { return ax == 0 ? 1 : (ax == 1 ? S.sy : S.sz); }

// CT fluxes and updates of one sweep in one pass, from the face arrays in
// to the face arrays out (never the same: the stencil reads neighbours that
// other blocks write).  sc = 0: both hold face fluxes.  sc = +1 (first sweep
// of a remap): in holds B, converted on the fly (the scaling pass of
// remap.f90:44-67 folded in).  sc = -1 (last predictor sweep): out gets B
// back (remap.f90:102-125 folded in).
template <int AX>
CtArgs ct_args(const double *const in[3], double *const out[3], const real *vel, const real *db1, double dt,
               dim3 *grid) {
  const int N[3] = {nx(), ny(), nz()};
  const Box ub = mkbox(0, N[0] + 1, 0, N[1] + 1, 0, N[2] + 1);
  // (transverse field t, velocity-average axis, geometry-average axis, box_t, box_a) x 2
  int t1, va1, ga1, t2, va2, ga2;
  Box bt1 = ub, ba1 = ub, bt2 = ub, ba2 = ub;
  if (AX == 0) {
    t1 = 1; va1 = 2; ga1 = 1;  // vx_by_flux
    t2 = 2; va2 = 1; ga2 = 2;  // vx_bz_flux
    bt2 = mkbox(1, N[0], 1, N[1], 0, N[2]);
    ba2 = mkbox(0, N[0], 0, N[1] + 1, 0, N[2] + 1);
  } else if (AX == 1) {
    t1 = 0; va1 = 2; ga1 = 0;  // vy_bx_flux
    t2 = 2; va2 = 0; ga2 = 2;  // vy_bz_flux
    ba2 = mkbox(1, N[0], 0, N[1], 1, N[2]);
  } else {
    t1 = 0; va1 = 1; ga1 = 0;  // vz_bx_flux
    t2 = 1; va2 = 0; ga2 = 1;  // vz_by_flux
  }
  // x sweep: va1 = z and ga2 = z (see the flux table above); tiles of CTX_W
  // points in x by CTX_ROWS - 1 rows in y, marching in z.  y and z sweeps march
  // along the sweep axis; tiles of CTM_XW - 1 points in x by CTM_ROWS - 1 rows
  // along the other transverse axis.
  const int P = AX == 0 ? 1 : 3 - AX, march = AX == 0 ? 2 : AX;
  const int w = AX == 0 ? CTX_W : CTM_XW - 1, rows = (AX == 0 ? CTX_ROWS : CTM_ROWS) - 1;
  const int ntx = (N[0] + 5 + w - 1) / w, nty = (N[P] + 5 + rows - 1) / rows;
  const int mc = cts_chunk((unsigned)(ntx * nty), N[march] + 5);
  *grid = dim3((unsigned)(ntx * nty), 1, (unsigned)((N[march] + 4 + mc) / mc));
  return CtArgs{in[t1],       in[t2],       in[AX],       out[t1],      out[t2], out[AX], vel, db1, strides(va1),
                strides(ga1), strides(va2), strides(ga2), dt,           ntx,     mc,      bt1, ba1, bt2,
                ba2};
}
// sc: 1 the first sweep of a remap, -1 the last, 0 between
template <int AX>
int ct_launch(const CtArgs &a, dim3 grid, int sc) {
  const dim3 blk(CT_THREADS(AX), 1, 1);
  if (sc > 0) LAUNCH("ct_sweep", (k_ct_sweep<AX, 1>), grid, blk, S.g, a);
  else if (sc < 0) LAUNCH("ct_sweep", (k_ct_sweep<AX, -1>), grid, blk, S.g, a);
  else LAUNCH("ct_sweep", (k_ct_sweep<AX, 0>), grid, blk, S.g, a);
  return 0;
}
template <int AX>
int ct_sweep(const double *const in[3], double *const out[3], const real *vel, const real *db1, double dt, int sc) {
  dim3 grid;
  const CtArgs a = ct_args<AX>(in, out, vel, db1, dt, &grid);
  return ct_launch<AX>(a, grid, sc);
}

// the face arrays a and the spare EMF arrays swap roles (the CT output went
// to the spares)
void swap_spare(double *&ax, double *&ay, double *&az) {
  double *t;
  t = ax; ax = S.fxr; S.fxr = t;
  t = ay; ay = S.fyr; S.fyr = t;
  t = az; az = S.fzr; S.fzr = t;
}

// the widths d?b1 of the predictor sweeps live in db1 and, since a predictor
// remap stores no volumes, in cv1 and cv2
real *pred_db1(int ax) { return ax == 0 ? S.db1 : (ax == 1 ? S.cv1 : S.cv2); }

// the geometry of a predictor remap whose last sweep is along `last`, and the
// predictor pressure
int geom_predictor(int last, double dt) {
  const PredP pr = {S.energy, S.rho, S.visc_heat, S.p0, S.pp, S.p.gamma, S.dt2, eos_args(), S.clamp};
  const Box cb = marched(cell_box());
#define GEOM_PRED(L)                                                                                                 \
  LAUNCH("geom", k_geom_pred<L>, zchunk_grid(cb), box_block(), S.g, cb, S.vx, S.vy, S.vz, pred_db1(0), pred_db1(1), \
         pred_db1(2), dt, pr)
  if (last == 0) GEOM_PRED(0);
  else if (last == 1) GEOM_PRED(1);
  else GEOM_PRED(2);
#undef GEOM_PRED
  return 0;
}

// one predictor-mode sweep (B only, no flag reset, no halo refresh) of the
// copy bp of B; the first sweep reads B itself, the last converts back
template <int AX>
int sweep_predictor(double dt, bool first, bool last) {
  const real *vel = AX == 0 ? S.vx : (AX == 1 ? S.vy : S.vz);
  if (first) {
    // B itself stays untouched: the first sweep writes the copy
    const double *const Bin[3] = {S.bx, S.by, S.bz};
    double *const Bp[3] = {S.bpx, S.bpy, S.bpz};
    return ct_sweep<AX>(Bin, Bp, vel, pred_db1(AX), dt, 1);
  }
  const double *const Bp[3] = {S.bpx, S.bpy, S.bpz};
  double *const spare[3] = {S.fxr, S.fyr, S.fzr};
  int rc = ct_sweep<AX>(Bp, spare, vel, pred_db1(AX), dt, last ? -1 : 0);
  if (rc) return rc;
  swap_spare(S.bpx, S.bpy, S.bpz);
  return 0;
}

// The geometry of a full remap lives in Lagrangian work arrays, which nothing
// reads between the corrector and the next step: the widths d?b1 of the three
// axes, and the volumes before the first, second and last sweep (k_geom).
real *remap_db1(int ax) { return ax == 0 ? S.al1 : (ax == 1 ? S.al2 : S.al3); }
real *remap_vol(int q) { return q == 0 ? S.cv1 : (q == 1 ? S.cv2 : S.visc_heat); }
int geom_full(int a0, int a1, double dt) {
  const Box cb = marched(cell_box());
#define GEOM(P, Q)                                                                                                  \
  if (a0 == P && a1 == Q) {                                                                                         \
    LAUNCH("geom", (k_geom<P, Q>), zchunk_grid(cb), box_block(), S.g, cb, S.vx1, S.vy1, S.vz1, remap_vol(0),        \
           remap_vol(1), remap_vol(2), remap_db1(0), remap_db1(1), remap_db1(2), dt);                               \
    return 0;                                                                                                       \
  }
  GEOM(0, 1)
  GEOM(0, 2)
  GEOM(1, 0)
  GEOM(1, 2)
  GEOM(2, 0)
  GEOM(2, 1)
#undef GEOM
  return fail(LARE_E_ARG, "remap axes %d, %d", a0, a1);
}

// the full sweep along AX, number q of the remap
template <int AX>
int sweep_full(double dt, int q) {
  const int N[3] = {nx(), ny(), nz()};
  const real *vel = AX == 0 ? S.vx1 : (AX == 1 ? S.vy1 : S.vz1);
  const bool first = q == 0, last = q == 2;
  const real *db1 = remap_db1(AX), *cv1 = remap_vol(q), *cv2 = last ? nullptr : remap_vol(q + 1);
  int rc;
  const int sc = first ? 1 : (last ? -1 : 0);
  const double *const B[3] = {S.bx, S.by, S.bz};
  double *const spare[3] = {S.fxr, S.fyr, S.fzr};
  dim3 cg;
  const CtArgs ct = ct_args<AX>(B, spare, vel, db1, dt, &cg);
  // the momentum remap's box and grid; it goes together with the CT sweep, whose
  // turn may come anywhere between the geometry and the boundary fill.  Apart,
  // the CT sweep comes first, so that the mass kernel finds the velocity and
  // the width in the cache (100 steps at 256^3 995 -> 992 ms, hardly more than
  // such runs differ by).
  Box xb = full_box();
  dim3 mg;
  if constexpr (AX == 0) {
    const unsigned pb = wave_blocks((long)(xb.x1 - xb.x0 + 1) * (xb.y1 - xb.y0 + 1),
                                    S.delta_ke ? MOMX_OUT_RKE : MOMX_OUT);
    xb.zc = march_chunk(pb, xb.z1 - xb.z0 + 1);
    mg = dim3(pb, 1, (unsigned)((xb.z1 - xb.z0 + xb.zc) / xb.zc));
  } else {
    xb = marched(xb, AX);
    mg = zchunk_grid(march_box(xb, AX));
  }
  const unsigned per = CT_THREADS(AX) / (BX * BY), nm = (mg.x * mg.z + per - 1) / per, nc = cg.x * cg.z;
  const bool together = !S.delta_ke && mom_ct_together(nm + nc);
  if (!together) {
    rc = ct_launch<AX>(ct, cg, sc);
    if (rc) return rc;
  }
  int hi[3] = {N[0] + 1, N[1] + 1, N[2] + 1};
  hi[AX] = N[AX];
  Box mb = mkbox(0, hi[0], 0, hi[1], 0, hi[2]);
  if (AX != 0) mb = marched(mb, AX);
  // mass flux, energy flux and the density and energy updates in one pass
  // over the mass flux's box (updates on cells 1..n); the new energy lands
  // in the energy flux array, which then swaps roles with the energy array
  // (the new density goes to rho_alt as before)
  if constexpr (AX == 0) {
    const dim3 gx(wave_blocks((long)(mb.x1 - mb.x0 + 1) * (mb.y1 - mb.y0 + 1), REX_OUT), 1,
                  (unsigned)(mb.z1 - mb.z0 + 1));
#define RHO_ENERGY(L)                                                                                               \
  LAUNCH("rho_energy", k_mass_rho_energy_x<L>, gx, box_block(), S.g, mb, S.energy, S.rho, vel, db1, S.dm, cv1, \
         cv2, S.rho_alt, S.Fe, dt, S.per[AX] ? 1 : 0)
    if (last) RHO_ENERGY(true);
    else RHO_ENERGY(false);
#undef RHO_ENERGY
  } else {
#define RHO_ENERGY(L)                                                                                               \
  LAUNCH("rho_energy", (k_mass_rho_energy_m<AX, L>), zchunk_grid(march_box(mb, AX)), box_block(), S.g, mb, S.energy, \
         S.rho, vel, db1, S.dm, cv1, cv2, S.rho_alt, S.Fe, dt, S.per[AX] ? 1 : 0)
    if (last) RHO_ENERGY(true);
    else RHO_ENERGY(false);
#undef RHO_ENERGY
  }
  if (S.any_open) {
    // the new energy and density cover cells 1..n; the ghosts of a BC_OPEN
    // side keep their values (no fill there)
    LAUNCH_BOX("copy_open", k_copy_open, full_box(), S.energy, S.Fe, 0);
    LAUNCH_BOX("copy_open", k_copy_open, full_box(), S.rho, S.rho_alt, 0);
  }
  {
    real *te = S.energy;
    S.energy = S.Fe;
    S.Fe = te;
  }
  {
    // vertex quantities, momentum fluxes and update in one pass over the
    // padded box (rho1 = rho before this sweep's update, which went to
    // rho_alt); the new velocities land in the flux arrays, which then swap
    // roles with the velocity arrays
    const MomArgs mo = {xb,   S.vx, S.vy, S.vz, vel, db1,  S.rho, cv1, cv2,
                        S.dm, S.Fx, S.Fy, S.Fz, dt,  S.rk};
    if (together) {
#define MOM_CT(SC) LAUNCH("mom_ct", (k_mom_ct<AX, SC>), dim3(nm + nc), dim3(CT_THREADS(AX)), S.g, mo, mg, ct, cg)
      if (sc > 0) MOM_CT(1);
      else if (sc < 0) MOM_CT(-1);
      else MOM_CT(0);
#undef MOM_CT
    } else {
#define MOM_REMAP(R, L) LAUNCH("mom_remap", (k_mom_remap<AX, R, L>), mg, box_block(), S.g, mo)
      if (S.delta_ke && last) MOM_REMAP(true, true);
      else if (S.delta_ke) MOM_REMAP(true, false);
      else if (last) MOM_REMAP(false, true);
      else MOM_REMAP(false, false);
#undef MOM_REMAP
    }
    swap_spare(S.bx, S.by, S.bz);
    // rke: this sweep's edge terms into delta_ke
    if (S.delta_ke) LAUNCH_BOX("rke_gather", k_rke_gather<AX>, interior(), S.rk, S.delta_ke);
    real *tv;
    tv = S.vx; S.vx = S.Fx; S.Fx = tv;
    tv = S.vy; S.vy = S.Fy; S.Fy = tv;
    tv = S.vz; S.vz = S.Fz; S.Fz = tv;
  }
  real *t = S.rho;
  S.rho = S.rho_alt;
  S.rho_alt = t;
  return boundary_conditions();
}

const int kStrang[6][3] = {{0, 1, 2}, {1, 2, 0}, {2, 0, 1}, {0, 2, 1}, {2, 1, 0}, {1, 0, 2}};

int eulerian_remap(int step, bool predictor) {
  const double dt = S.dt;
  const int c = ((step % 6) + 6) % 6;
  // The B -> face flux scaling (remap.f90:44-67) happens inside the first
  // sweep's CT kernels and the scaling back (remap.f90:102-125) inside the
  // last sweep's update.  In the full remap the last sweep's halo refresh
  // then runs on B instead of on face fluxes, which leaves the halos that the
  // bfield_bcs after the scaling back in the reference writes from the same
  // interior.
  if (predictor) {
    int rc = geom_predictor(kStrang[c][2], dt);
    if (rc) return rc;
    for (int q = 0; q < 3; ++q) {
      const int ax = kStrang[c][q];
      const bool first = q == 0, last = q == 2;
      rc = ax == 0 ? sweep_predictor<0>(dt, first, last)
                       : (ax == 1 ? sweep_predictor<1>(dt, first, last) : sweep_predictor<2>(dt, first, last));
      if (rc) return rc;
    }
    return bfield_bcs(S.bpx, S.bpy, S.bpz);
  }
  // rke: delta_ke = 0 (remap.f90:38); only the interior is ever read
  if (S.delta_ke) LAUNCH_BOX("fill", k_fill, interior(), S.delta_ke, 0.0);
  int rc = geom_full(kStrang[c][0], kStrang[c][1], dt);
  if (rc) return rc;
  for (int q = 0; q < 3; ++q) {
    const int ax = kStrang[c][q];
    rc = ax == 0 ? sweep_full<0>(dt, q) : (ax == 1 ? sweep_full<1>(dt, q) : sweep_full<2>(dt, q));
    if (rc) return rc;
  }
  return 0;
}

// ----------------------------------------------------------------------------
// lagrangian step
// ----------------------------------------------------------------------------
int eta_calc() {
  if (S.p.resistive_mhd) {
    const Box eb = marched(mkbox(-1, nx() + 1, -1, ny() + 1, -1, nz() + 1));
    LAUNCH("eta", k_eta, zchunk_grid(eb), box_block(), S.g, eb, S.bx, S.by, S.bz, S.eta,
               S.p.eta_background, S.p.eta0, S.p.j_max);
  } else {
    LAUNCH_BOX("fill", k_fill, cell_box(), S.eta, 0.0);
  }
  return 0;
}

LagArgs lag_args() {
  LagArgs a;
  a.gamma = S.p.gamma;
  a.visc1 = S.p.visc1;
  a.visc2_norm = S.visc2_norm;
  a.dt = S.dt;
  a.dt2 = S.dt2;
  a.eta_bg = S.p.eta_background;
  a.eta0 = S.p.eta0;
  a.j_max = S.p.j_max;
  a.va_max2 = S.p.va_max * S.p.va_max;
  a.alpha_av = S.p.alpha_av;
  a.resistive = S.p.resistive_mhd;
  a.boris = S.p.boris;
  a.write_gb = !(S.first_set_dt && S.p.restart);
  a.limiter = S.p.shock_limiter;
  a.compression = S.p.shock_compression;
  a.cowling = S.p.cowling_resistivity;
  a.eta_perp = S.eta_perp;
  return a;
}

// ----------------------------------------------------------------------------
// partially ionised plasma (neutral.f90)
// ----------------------------------------------------------------------------
EosArgs eos_args() { return EosArgs{S.pi_eos ? S.xi : nullptr, S.ip}; }

NeutralArgs neutral_args() {
  NeutralArgs a;
  a.gm1 = S.p.gamma - 1.0;
  a.ip = S.ip;
  a.f_bar = S.p.f_bar;
  a.t_bar = S.p.t_bar;
  a.r_bar = S.p.r_bar;
  a.eta_bar = S.p.eta_bar;
  a.t_rad = S.p.t_rad;
  return a;
}

// neutral_fraction over the cell box from Y (energy, or an RKL2 stage value
// read through the boundary map when mode is TMODE_WRAP)
int neutral_fraction(const real *Y, int mode) {
  if (mode == TMODE_WRAP)
    LAUNCH_BOX("neutral", k_neutral<TMODE_WRAP>, cell_box(), Y, S.energy, S.rho, S.xi, S.nf_flag, neutral_args());
  else
    LAUNCH_BOX("neutral", k_neutral<TMODE_DIRECT>, cell_box(), Y, S.energy, S.rho, S.xi, S.nf_flag, neutral_args());
  return 0;
}

int perpendicular_resistivity() {
  LAUNCH_BOX("eta_perp", k_eta_perp, nodes0n(), S.rho, S.energy, S.xi, S.bx, S.by, S.bz, S.eta_perp,
             neutral_args());
  return 0;
}

// ----------------------------------------------------------------------------
// open boundaries (openboundary.f90)
// ----------------------------------------------------------------------------
OpenFace open_face(int a, int hi) {
  OpenFace f;
  const int n = S.n[a];
  f.a = a;
  f.hi = hi;
  f.u = a == 0 ? 1 : 0;
  f.w = a == 2 ? 1 : 2;
  f.ty = a == 1 ? 0 : 1;
  f.tz = a == 2 ? 0 : 2;
  f.lb = hi ? n : 0;
  f.lc = hi ? n : 1;
  f.lfc = hi ? n + 2 : -1;
  f.lfn = hi ? n + 2 : -2;
  f.lset_n = hi ? n + 1 : -1;
  f.lset_c = hi ? n + 1 : 0;
  f.sg = hi ? 1.0 : -1.0;
  return f;
}

unsigned face_points(const OpenFace &f) { return (unsigned)((S.n[f.u] + 2) * (S.n[f.w] + 2)); }

// the pre-corrector energy and density of each open face's first interior layer
int open_save() {
  for (int a = 0; a < 3; ++a)
    for (int hi = 0; hi <= 1; ++hi) {
      if (S.bc[2 * a + hi] != LARE_BC_OPEN) continue;
      const OpenFace f = open_face(a, hi);
      LAUNCH("open_save", k_open_save, dim3((face_points(f) + 255) / 256), dim3(256), S.g, f, S.energy, S.rho,
             S.obc_save + (size_t)(2 * a + hi) * S.obc_face);
    }
  return 0;
}

// open_bcs: the faces one launch each, in the reference's order
int open_bcs() {
  for (int a = 0; a < 3; ++a)
    for (int hi = 0; hi <= 1; ++hi) {
      if (S.bc[2 * a + hi] != LARE_BC_OPEN) continue;
      const OpenFace f = open_face(a, hi);
      LAUNCH("open_bcs", k_open_bcs, dim3((face_points(f) + 255) / 256), dim3(256), S.g, f, S.vx, S.vy, S.vz, S.bx,
             S.by, S.bz, S.rho, S.energy, S.obc_save + (size_t)(2 * a + hi) * S.obc_face, S.p.gamma);
    }
  return 0;
}

// the reference STOPs on an inverted temperature bracket (neutral.f90:172-175):
// report it once the work queued so far has run, and clear the flag
// (the flag is a word of the pinned mirror).  folded: a fold was queued after
// the last neutral_fraction, and its ticket says that it has run; a 45 x 37 x 41
// step waited some 15 us for the end of the remap instead.
int check_neutral_fault(const char *where, bool folded) {
  if (!S.nf_flag) return 0;
  if (folded) {
    const int rc = read_scalars(0, 0, nullptr);
    if (rc) return rc;
  } else {
    HIPCHK(hipStreamSynchronize(S.stream));
  }
  volatile int *flag = S.nf_flag;
  if (!*flag) return 0;
  *flag = 0;
  return fail(LARE_F_TBOUNDS, "%s: neutral_fraction temperature bracket inverted (energy <= 0 in some cell)", where);
}

int set_dt_and_stages(double dt_local, double dtr_local) {
  if (S.first_set_dt) {
    S.first_set_dt = 0;
    if (S.p.restart) {
      S.dt = S.p.dt_from_restart;
      return 0;
    }
  }
  S.dt = 0.9 * dt_local;
  S.dtr = 0.9 * dtr_local;
  if (S.p.conduction) {
    int rc = calc_s_stages();
    if (rc) return rc;
    const int ss_limit = 60;
    if (S.n_s_stages >= ss_limit) {
      const double f = (double)(2 * ss_limit * ss_limit - 9) / (double)(2 * S.n_s_stages * S.n_s_stages - 9);
      S.dt = S.dt * f;
      S.dtr = S.dtr * f;
    }
  }
  S.time = S.time + S.dt;
  return 0;
}

// learned conduction surrogate (surrogate_rt.hpp)
int sur_enabled();
int sur_conduct_step(int delta_mode, double *res_out, int *acc_out);

// One FOURTHORDER resistive substep (lagran.F90:146-149 with :1329-1415):
// eta_calc; B1 = B (in the spare fxr..fzr arrays); rkstep and bstep four
// times; the final bstep with the weighted EMFs; the heating; energy_bcs.
int resist_rk4_substep() {
  int rc = eta_calc();
  if (rc) return rc;
  const size_t nb = sizeof(double) * S.ntot;
  HIPCHK(hipMemcpyAsync(S.fxr, S.bx, nb, hipMemcpyDeviceToDevice, S.stream));
  HIPCHK(hipMemcpyAsync(S.fyr, S.by, nb, hipMemcpyDeviceToDevice, S.stream));
  HIPCHK(hipMemcpyAsync(S.fzr, S.bz, nb, hipMemcpyDeviceToDevice, S.stream));
  const Box n0 = nodes0n();
  const double dt = S.dt, half_dt = dt * 0.5, dt6 = dt * (1.0 / 6.0);
  const double h[3] = {half_dt, half_dt, dt};
  const int w[4] = {0, 2, 2, 1};
  for (int q = 0; q < 4; ++q) {
    if (q > 0) {
      LAUNCH_BOX("rk4_bstep", k_rk4_bstep, n0, S.fxr, S.fyr, S.fzr, S.rk4k, S.bx, S.by, S.bz, h[q - 1]);
      rc = bfield_bcs(S.bx, S.by, S.bz);
      if (rc) return rc;
    }
    if (S.eta_perp)
      LAUNCH_BOX("rk4_emf", k_rk4_emf<true>, n0, S.bx, S.by, S.bz, S.eta, S.rk4k, S.rk4s, w[q], S.eta_perp);
    else
      LAUNCH_BOX("rk4_emf", k_rk4_emf<false>, n0, S.bx, S.by, S.bz, S.eta, S.rk4k, S.rk4s, w[q], S.eta_perp);
  }
  LAUNCH_BOX("rk4_bstep", k_rk4_bstep, n0, S.fxr, S.fyr, S.fzr, S.rk4s, S.bx, S.by, S.bz, dt6);
  rc = bfield_bcs(S.bx, S.by, S.bz);
  if (rc) return rc;
  LAUNCH_BOX("rk4_heat", k_rk4_heat, interior(), S.rk4s.k[3], S.rho, S.energy, dt6);
  rc = energy_bcs();
  if (rc) return rc;
  const dim3 gr = box_grid(n0);
  LAUNCH("ohmic_total", k_ohmic_total, gr, box_block(), S.g, n0, S.rk4s.k[3], S.partial, dt6);
  return final_reduce(gr, 1, 0, 9, 1);
}

// xi_known: xi_n is that of the density and energy on entry, which the first
// resistive substep finds unchanged
int lagrangian_step(bool xi_known) {
  const int N0 = nx(), N1 = ny(), N2 = nz();
  LagArgs a = lag_args();  // dt = previous step's dt (Q1)
  {
    const Box vb = marched(mkbox(-1, N0 + 1, -1, N1 + 1, -1, N2 + 1));
    const EosArgs eq = eos_args();
#define VERTEX_PREP(GB, PI)                                                                                        \
  LAUNCH("vertex_prep", (k_vertex_prep<GB, PI>), zchunk_grid(vb), box_block(), S.g, vb, S.rho, S.energy, S.bx, S.by, \
         S.bz, S.gamma_boris, S.rho_v, S.cs_v, S.p.gamma, eq)
    if (S.gamma_boris) {
      if (S.pi_eos) VERTEX_PREP(true, true);
      else VERTEX_PREP(true, false);
    } else {
      if (S.pi_eos) VERTEX_PREP(false, true);
      else VERTEX_PREP(false, false);
    }
#undef VERTEX_PREP
  }
  if (S.p.use_viscous_damping) {
    LAUNCH_BOX("damp_q", k_damp_q, nodes0n(), S.vx, S.vy, S.vz, S.visc3, S.qx, S.qy, S.qz);
    LAUNCH_BOX("damp_apply", k_damp_apply, nodes0n(), S.vx, S.vy, S.vz, S.qx, S.qy, S.qz, S.dt);
  }
  {
    const Box ab = marched(mkbox(-1, N0 + 1, -1, N1 + 2, 0, N2 + 2));
    LAUNCH("alpha", k_alpha, zchunk_grid(ab), box_block(), S.g, ab, S.vx, S.vy, S.vz, S.rho_v, S.cs_v, S.al1, S.al2,
           S.al3, a);
  }
  const Box vdb = marched(mkbox(0, N0 + 1, 0, N1 + 1, 0, N2 + 1));
  dim3 gr = zchunk_grid(vdb);
  if (S.pi_eos)
    LAUNCH("visc_dt", k_visc_dt<true>, gr, box_block(), S.g, vdb, S.vx, S.vy, S.vz, S.rho, S.energy, S.bx, S.by, S.bz,
           S.eta, S.al1, S.al2, S.al3, S.visc_heat, S.p0, S.gamma_boris, S.partial, a, eos_args());
  else
    LAUNCH("visc_dt", k_visc_dt<false>, gr, box_block(), S.g, vdb, S.vx, S.vy, S.vz, S.rho, S.energy, S.bx, S.by, S.bz,
           S.eta, S.al1, S.al2, S.al3, S.visc_heat, S.p0, S.gamma_boris, S.partial, a, eos_args());
  int rc = final_reduce(gr, 3, 7, 0, 0);
  if (rc) return rc;
  double mins[3];
  rc = read_scalars(0, 3, mins);
  if (rc) return rc;
  if (mins[2] < 0.0) {
    // the state entering the step holds a non-finite value or rho <= 0
    static const char *names[8] = {"rho", "energy", "vx", "vy", "vz", "bx", "by", "bz"};
    const double code = -mins[2];
    const int fid = (int)(code / 4294967296.0) - 1;
    const long cell = (long)(code - (double)(fid + 1) * 4294967296.0);
    const int ci = (int)(cell % N0) + 1, cj = (int)((cell / N0) % N1) + 1, ck = (int)(cell / ((long)N0 * N1)) + 1;
    return fail(LARE_F_NONFINITE, "step %d: %s is not finite%s at (%d, %d, %d) entering lagrangian_step", S.step,
                fid >= 0 && fid < 8 ? names[fid] : "?", fid == 0 ? " or not positive" : "", ci, cj, ck);
  }
  rc = set_dt_and_stages(mins[0], mins[1]);
  if (rc) return rc;
  S.dt2 = 0.5 * S.dt;
  S.last_substeps = 0;

  if (S.p.resistive_mhd) {
    const double dt_sub = S.dtr;
    const int substeps = (int)(S.dt / dt_sub) + 1;
    if (substeps > S.peak_substeps) S.peak_substeps = substeps;
    S.last_substeps = substeps;
    const double actual_dt = S.dt;
    S.dt = S.dt / (double)substeps;
    // eta_calc, rkstep, bstep and the ohmic heating of each substep run in
    // k_resist, which writes the new B to the fxr..fzr arrays; they then
    // swap roles with bx..bz.  The B and energy halos of a substep are
    // refreshed together.
    Box fb = full_box();
    int tiles_x;
    const dim3 g2 = resist_grid(fb, &tiles_x);
    if ((size_t)g2.x * g2.y * g2.z > S.partial_cap)
      return fail(LARE_E_ARG, "resistive grid of %u blocks exceeds the partial buffer", g2.x * g2.z);
    for (int sc = 1; sc <= substeps; ++sc) {
      // eta_calc runs inside the substep kernels; neutral_fraction and
      // perpendicular_resistivity read nothing it writes (lagran.F90:146-149)
      if (S.pi_eos && !(sc == 1 && xi_known)) {
        rc = neutral_fraction(S.energy, TMODE_DIRECT);
        if (rc) return rc;
      }
      if (S.eta_perp) {
        rc = perpendicular_resistivity();
        if (rc) return rc;
      }
      if (S.p.fourth_order) {
        rc = resist_rk4_substep();
        if (rc) return rc;
        continue;
      }
      // the eta of a substep is read within it; the last one's is kept
      real *const eta_out = sc == substeps ? S.eta : nullptr;
      if (S.eta_perp)
        LAUNCH("resist", k_resist<true>, g2, dim3(64, RS_ROWS, 1), S.g, fb, tiles_x, S.bx, S.by, S.bz, S.fxr, S.fyr,
               S.fzr, eta_out, S.energy, S.ohmic_dep, S.rho, S.curlb, S.partial, S.dt, S.p.eta_background, S.p.eta0,
               S.p.j_max, S.eta_perp);
      else
        LAUNCH("resist", k_resist<false>, g2, dim3(64, RS_ROWS, 1), S.g, fb, tiles_x, S.bx, S.by, S.bz, S.fxr, S.fyr,
               S.fzr, eta_out, S.energy, S.ohmic_dep, S.rho, S.curlb, S.partial, S.dt, S.p.eta_background, S.p.eta0,
               S.p.j_max, S.eta_perp);
      FoldJob job = {};
      rc = fold_job(g2, 9, &job);
      if (rc) return rc;
      if (S.curlb)
        LAUNCH_BOX("cool_b", k_cool_b, interior(), S.curlb, S.rho, S.cool_b, S.energy, S.p.alpha_av, S.dt);
      double *tb;
      tb = S.bx; S.bx = S.fxr; S.fxr = tb;
      tb = S.by; S.by = S.fyr; S.fyr = tb;
      tb = S.bz; S.bz = S.fzr; S.fzr = tb;
      rc = fill_halo<1, 1, 0>(state_halo(), "bc_resistive", job);
      if (rc) return rc;
    }
    S.dt = actual_dt;
  }

  if (S.p.conduction) {
    if (sur_enabled()) {
      rc = sur_conduct_step(1, nullptr, nullptr);
      if (rc) return rc;
    } else {
      rc = calc_s_stages();
      if (rc) return rc;
      rc = heat_conduct_sts2(1);
      if (rc) return rc;
    }
  }
  // Without conduction, energy = MAX(energy0 + 0, 0) (lagran.F90:180-181).
  // After a first-order resistive step it changes nothing: the last substep's
  // ohmic heating already clamped the whole cell box (:1305) and energy_bcs
  // only copies clamped values.  Otherwise its two readers, the predictor and
  // the corrector, clamp what they read, and the fill after the corrector
  // writes the ghosts anew; a BC_OPEN side's ghosts are not written again, so
  // then the array itself is clamped.
  const bool clamp = !S.p.conduction && (!S.p.resistive_mhd || S.p.fourth_order);
  if (clamp && S.any_open) LAUNCH_BOX("energy_max", k_energy_max, cell_box(), S.energy);
  S.clamp = clamp && !S.any_open;

  // predictor-corrector (lagran.F90:208-478)
  const Box nb = marched(nodes0n());
  // k_force gives the nodes 0..n of v1 what remap_v_bcs gives them, the only
  // ones that the corrector reads; the ghosts follow in its fill.  With a
  // BC_OPEN side remap_v_bcs comes at once, before v's ghosts are copied.
  const int wall = S.any_open ? 0 : 1;
  if (S.p.cauchy) {
    // the Cauchy solution for the cell-centred B1 (B1 cv1 in the spare
    // predictor-B arrays), cv1 and the predictor pressure; no predictor remap
    real *b1[3] = {(real *)S.bpx, (real *)S.bpy, (real *)S.bpz};
    LAUNCH_BOX("cauchy_b", k_cauchy_b, cell_box(), S.vx, S.vy, S.vz, S.bx, S.by, S.bz, S.cv1, b1[0], b1[1], b1[2],
               S.energy, S.rho, S.visc_heat, S.p0, S.pp, S.p.gamma, S.dt2, eos_args(), S.clamp);
    LAUNCH("force", k_force<true>, zchunk_grid(nb), box_block(), S.g, nb, S.vx, S.vy, S.vz, S.pp,
           S.bx, S.by, S.bz, S.rho_v, S.al1, S.al2, S.al3, S.gamma_boris, S.vx1, S.vy1, S.vz1, S.dt2, S.cv1, b1[0],
           b1[1], b1[2], wall);
  } else {
    const double dt_full = S.dt;
    S.dt = 0.5 * dt_full;
    rc = eulerian_remap(S.step, true);
    S.dt = dt_full;
    if (rc) return rc;
    // the predictor energy and pressure were formed in the predictor
    // remap's geometry pass
    LAUNCH("force", k_force<false>, zchunk_grid(nb), box_block(), S.g, nb, S.vx, S.vy, S.vz, S.pp,
           S.bpx, S.bpy, S.bpz, S.rho_v, S.al1, S.al2, S.al3, S.gamma_boris, S.vx1, S.vy1, S.vz1, S.dt2, S.cv1,
           nullptr, nullptr, nullptr, wall);
  }
  if (S.any_open) {
    rc = node_bcs(S.vx1, S.vy1, S.vz1, "bc_v1");
    if (rc) return rc;
    // v1 = v over the whole array before the predictor remap
    // (lagran.F90:1051-1053); the forces then set nodes 0..n and
    // remap_v_bcs the filled sides, so a BC_OPEN side keeps v's ghosts
    LAUNCH_BOX("copy_open", k_copy_open, full_box(), S.vx, S.vx1, 1);
    LAUNCH_BOX("copy_open", k_copy_open, full_box(), S.vy, S.vy1, 1);
    LAUNCH_BOX("copy_open", k_copy_open, full_box(), S.vz, S.vz1, 1);
  }
  if (S.any_open) {
    rc = open_save();
    if (rc) return rc;
  }
  dim3 g3 = zchunk_grid(nb);
  if (S.cool_v)
    LAUNCH("shock_corr", k_shock_corr<true>, g3, box_block(), S.g, nb, S.vx, S.vy, S.vz, S.vx1, S.vy1, S.vz1,
           S.al1, S.al2, S.al3, S.pp, S.energy, S.rho, S.visc_dep, S.Fx, S.Fy, S.Fz, S.cool_v, S.p.alpha_av,
           S.partial, S.dt, S.clamp);
  else
    LAUNCH("shock_corr", k_shock_corr<false>, g3, box_block(), S.g, nb, S.vx, S.vy, S.vz, S.vx1, S.vy1, S.vz1,
           S.al1, S.al2, S.al3, S.pp, S.energy, S.rho, S.visc_dep, S.Fx, S.Fy, S.Fz, S.cool_v, S.p.alpha_av,
           S.partial, S.dt, S.clamp);
  FoldJob job = {};
  rc = fold_job(g3, 8, &job);
  if (rc) return rc;
  // the new velocities went to the momentum-flux arrays, which swap roles
  // with the velocity arrays; the boundary fill below sets their ghosts
  if (S.any_open) {
    LAUNCH_BOX("copy_open", k_copy_open, full_box(), S.vx, S.Fx, 1);
    LAUNCH_BOX("copy_open", k_copy_open, full_box(), S.vy, S.Fy, 1);
    LAUNCH_BOX("copy_open", k_copy_open, full_box(), S.vz, S.Fz, 1);
  }
  {
    real *tv;
    tv = S.vx; S.vx = S.Fx; S.Fx = tv;
    tv = S.vy; S.vy = S.Fy; S.Fy = tv;
    tv = S.vz; S.vz = S.Fz; S.Fz = tv;
  }
  if (S.any_open) {
    // velocity_bcs, open_bcs, then (with the end of lagrangian_step)
    // energy_bcs and density_bcs (lagran.F90:408-412, :196-198)
    rc = node_bcs(S.vx, S.vy, S.vz, "bc_lagrangian");
    if (rc) return rc;
    rc = open_bcs();
    if (rc) return rc;
    return fill_halo<0, 2, 0>(state_halo(), "bc_lagrangian", job);
  }
  return fill_halo<0, 2, 6>(state_halo(), "bc_lagrangian", job);
}

// ----------------------------------------------------------------------------
// memory
// ----------------------------------------------------------------------------
#include "transfer.hpp"
void sur_free();
void slab_drop();
void free_all() {
  sur_free();
  if (S.stream) (void)hipStreamSynchronize(S.stream);
  xfer_free();
  for (void *p : S.allocs) (void)hipFree(p);
  S.allocs.clear();
  slab_drop();
  if (S.metric) (void)hipFree(S.metric);
  S.metric = nullptr;
  if (S.partial) (void)hipFree(S.partial);
  S.partial = nullptr;
  if (S.dscal) (void)hipFree(S.dscal);
  S.dscal = nullptr;
  if (S.hscal) (void)hipHostFree(S.hscal);
  S.hscal = nullptr;
  for (auto &r : S.pending) {
    (void)hipEventDestroy(r.a);
    (void)hipEventDestroy(r.b);
  }
  S.pending.clear();
  for (auto e : S.pool) (void)hipEventDestroy(e);
  S.pool.clear();
  S.acc.clear();
  S.ready = S.loaded = false;
}

// The arrays of the padded box come out of one allocation, made and cleared at
// once: some 45 of their own took 1.5 ms to open and 3.4 ms to close at 32^3.
// Where it is not to be had, or is used up, an array gets its own.
#define SLAB_ALIGN 256
struct Slab {
  char *p = nullptr;
  size_t cap = 0, used = 0;
};
Slab g_slab;
void slab_drop() { g_slab = Slab(); }

size_t slab_bytes(size_t n) { return (n + SLAB_ALIGN - 1) / SLAB_ALIGN * SLAB_ALIGN; }
int slab_reserve(int reals, int doubles) {
  g_slab = Slab();
  const size_t n = reals * slab_bytes(sizeof(real) * S.ntot) + doubles * slab_bytes(sizeof(double) * S.ntot);
  void *p = nullptr;
  if (hipMalloc(&p, n) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  S.allocs.push_back(p);
  g_slab.p = (char *)p;
  g_slab.cap = n;
  const hipError_t e = hipMemsetAsync(p, 0, n, S.stream);
  return e == hipSuccess ? 0 : fail(-(int)e, "hipMemset failed");
}

template <class T>
int dalloc(T **p) {
  const size_t n = slab_bytes(sizeof(T) * S.ntot);
  if (g_slab.cap - g_slab.used >= n) {
    *p = (T *)(g_slab.p + g_slab.used);
    g_slab.used += n;
    return 0;
  }
  hipError_t e = hipMalloc((void **)p, sizeof(T) * S.ntot);
  if (e != hipSuccess) return fail(LARE_E_NOMEM, "hipMalloc of %zu elements failed: %s", S.ntot, hipGetErrorString(e));
  S.allocs.push_back((void *)*p);
  e = hipMemsetAsync(*p, 0, sizeof(T) * S.ntot, S.stream);
  if (e != hipSuccess) return fail(-(int)e, "hipMemset failed");
  return 0;
}

// Fortran array bounds (lower) per field kind
void lower_of(FieldKind k, int lo[3]) {
  lo[0] = lo[1] = lo[2] = (k == FK_NODE) ? -2 : -1;
  if (k == FK_BX) lo[0] = -2;
  if (k == FK_BY) lo[1] = -2;
  if (k == FK_BZ) lo[2] = -2;
}

// adds the transfer of one device box to or from a host Fortran array (FP64,
// reference bounds); a NULL array is left out
template <class T>
void xfer_add(XferSet &s, T *dev, double *host, FieldKind k) {
  if (!host) return;
  XferField &f = s.f[s.nf++];
  f.dev = dev;
  f.host = host;
  f.wide = sizeof(T) == sizeof(double);
  lower_of(k, f.lo);
  f.first = s.total;
  s.total += (unsigned long)(nx() + 3 - f.lo[0]) * (ny() + 3 - f.lo[1]) * (nz() + 3 - f.lo[2]);
}
XferSet state_xfer(const lare_fields *f) {
  XferSet s = {};
  xfer_add(s, S.rho, f->rho, FK_CELL);
  xfer_add(s, S.energy, f->energy, FK_CELL);
  xfer_add(s, S.vx, f->vx, FK_NODE);
  xfer_add(s, S.vy, f->vy, FK_NODE);
  xfer_add(s, S.vz, f->vz, FK_NODE);
  xfer_add(s, S.bx, f->bx, FK_BX);
  xfer_add(s, S.by, f->by, FK_BY);
  xfer_add(s, S.bz, f->bz, FK_BZ);
  xfer_add(s, S.eta, f->eta, FK_CELL);
  xfer_add(s, S.visc_dep, f->visc_dep, FK_CELL);
  xfer_add(s, S.ohmic_dep, f->ohmic_dep, FK_CELL);
  return s;
}

// ============================================================================
// entry points of this precision (wrapped by the C-ABI in lare_dev.hip)
// ============================================================================


int api_init(const lare_grid *grid, const lare_params *params) {
  if (!grid || !params) return fail(LARE_E_ARG, "lare_dev_init: NULL argument");
  free_all();
  const int n[3] = {grid->nx, grid->ny, grid->nz};
  const int bc[6] = {grid->xbc_min, grid->xbc_max, grid->ybc_min, grid->ybc_max, grid->zbc_min, grid->zbc_max};
  for (int a = 0; a < 3; ++a) {
    if (n[a] < 4) return fail(LARE_E_ARG, "grid size %d on axis %d is below 4", n[a], a);
    const int lo = bc[2 * a], hi = bc[2 * a + 1];
    const bool ok = (lo == LARE_BC_PERIODIC && hi == LARE_BC_PERIODIC) ||
                    ((lo == LARE_BC_USER || lo == LARE_BC_OPEN) && (hi == LARE_BC_USER || hi == LARE_BC_OPEN));
    if (!ok)
      return fail(LARE_E_ARG,
                  "axis %d: boundary codes (%d, %d) unsupported (both periodic, or each side BC_USER or BC_OPEN)", a,
                  lo, hi);
  }
  if (!grid->dxb || !grid->dxc || !grid->dyb || !grid->dyc || !grid->dzb || !grid->dzc)
    return fail(LARE_E_ARG, "lare_dev_init: metric arrays missing");
  memcpy(S.n, n, sizeof(n));
  memcpy(S.bc, bc, sizeof(bc));
  S.any_open = false;
  for (int a = 0; a < 3; ++a) {
    S.per[a] = bc[2 * a] == LARE_BC_PERIODIC;
    S.user[a] = !S.per[a];
    S.any_open = S.any_open || bc[2 * a] == LARE_BC_OPEN || bc[2 * a + 1] == LARE_BC_OPEN;
  }
  const int eos = params->eos_number == 0 ? LARE_EOS_IDEAL : params->eos_number;
  if (eos != LARE_EOS_IDEAL && eos != LARE_EOS_ION && eos != LARE_EOS_PI)
    return fail(LARE_E_ARG, "eos_number %d unknown", params->eos_number);
  const bool pi = eos != LARE_EOS_IDEAL;
  if (params->cowling_resistivity && !pi)
    return fail(LARE_E_ARG, "cowling_resistivity needs a partially ionised eos_number (control.f90:158-161)");
  if (pi && sizeof(real) != sizeof(double))
    return fail(LARE_E_ARG, "the partially ionised equation of state runs in the FP64 mode only");
  for (int q = 0; q < 6; ++q) {
    if (bc[q] == LARE_BC_OPEN && sizeof(real) != sizeof(double))
      return fail(LARE_E_ARG, "BC_OPEN boundaries run in the FP64 mode only");
    // with CAUCHY nothing sets v1 on a BC_OPEN side's ghost nodes before the
    // remap reads them (lagran.F90:1050-1059 copy v to v1 only without it)
    if (bc[q] == LARE_BC_OPEN && params->cauchy)
      return fail(LARE_E_ARG, "BC_OPEN boundaries with the CAUCHY predictor: v1 on the open ghosts is undefined");
  }
  if (pi && !(params->f_bar > 0.0 && params->t_rad > 0.0 && params->r_bar > 0.0 && params->t_bar >= 0.0))
    return fail(LARE_E_ARG, "partially ionised: f_bar, t_rad and r_bar must be > 0, t_bar >= 0");
  if (pi && params->cowling_resistivity && !(params->eta_bar >= 0.0))
    return fail(LARE_E_ARG, "cowling_resistivity: eta_bar must be >= 0");
  S.p = *params;
  S.p.eos_number = eos;
  S.pi_eos = pi;
  S.ip = eos == LARE_EOS_ION ? params->ionise_pot : 0.0;
  S.tfac = (params->gamma - 1.0) / (2.0 - params->xi_n);
  S.visc2_norm = 0.25 * (params->gamma + 1.0) * params->visc2;
  S.sy = ((n[0] + 19 + 15) / 16) * 16;
  S.sz = S.sy * (n[1] + 5);
  S.ntot = (size_t)S.sz * (size_t)(n[2] + 5);
  if (S.ntot > (size_t)2147483647) return fail(LARE_E_ARG, "grid too large for 32-bit indexing");
  if (!S.stream) HIPCHK(hipStreamCreate(&S.stream));  // default priority
  // metrics: 7 arrays, each with index offset 2, length nmax + 6
  const int nmax = n[0] > n[1] ? (n[0] > n[2] ? n[0] : n[2]) : (n[1] > n[2] ? n[1] : n[2]);
  const int L = nmax + 6;
  std::vector<double> hm(7 * (size_t)L, 0.0);
  const double *src[7] = {grid->dxb, grid->dxc, grid->dyb, grid->dyc, grid->dzb, grid->dzc, grid->grav};
  for (int q = 0; q < 7; ++q) {
    const int ax = q < 6 ? q / 2 : 2;
    const int hi = (q < 6 && (q % 2) == 1) ? n[ax] + 1 : n[ax] + 2;
    for (int i = -1; i <= hi; ++i) hm[(size_t)q * L + (i + 2)] = src[q] ? src[q][i + 1] : 0.0;
  }
  HIPCHK(hipMalloc((void **)&S.metric, sizeof(double) * hm.size()));
  HIPCHK(hipMemcpy(S.metric, hm.data(), sizeof(double) * hm.size(), hipMemcpyHostToDevice));
  S.g.nx = n[0];
  S.g.ny = n[1];
  S.g.nz = n[2];
  S.g.sy = S.sy;
  S.g.sz = S.sz;
  const double *m[7];
  for (int q = 0; q < 7; ++q) m[q] = S.metric + (size_t)q * L + 2;
  S.g.dxb = m[0]; S.g.dxc = m[1]; S.g.dyb = m[2]; S.g.dyc = m[3]; S.g.dzb = m[4]; S.g.dzc = m[5]; S.g.grav = m[6];
  for (int a = 0; a < 3; ++a) {
    S.g.per[a] = S.per[a];
    S.g.user[a] = S.user[a];
    S.g.open_lo[a] = bc[2 * a] == LARE_BC_OPEN;
    S.g.open_hi[a] = bc[2 * a + 1] == LARE_BC_OPEN;
  }
  real **bulk[] = {&S.rho, &S.rho_alt, &S.energy, &S.vx, &S.vy, &S.vz, &S.vx1, &S.vy1, &S.vz1, &S.eta,
                    &S.visc3, &S.visc_dep, &S.ohmic_dep, &S.rho_v, &S.cs_v, &S.al1, &S.al2, &S.al3,
                    &S.visc_heat, &S.p0, &S.pp, &S.cv1, &S.cv2, &S.db1, &S.Fe, &S.dm, &S.Fx, &S.Fy,
                    &S.Fz, &S.larsen, &S.Lc, &S.Yb[0], &S.Yb[1], &S.Yb[2]};
  double **wide[] = {&S.bx, &S.by, &S.bz, &S.bpx, &S.bpy, &S.bpz, &S.fxr, &S.fyr, &S.fzr, &S.F, &S.F2};
  {
    // with the arrays of the options taken below
    int reals = (int)(sizeof(bulk) / sizeof(bulk[0]));
    if (params->fourth_order && params->resistive_mhd) reals += 8;
    if (params->rke) reals += 4;
    if (pi) reals += params->cowling_resistivity ? 2 : 1;
    if (params->boris) reals += 1;
    if (params->cooling_term) reals += params->resistive_mhd ? 3 : 2;
    if (params->use_viscous_damping) reals += 3;
    const int rc = slab_reserve(reals, (int)(sizeof(wide) / sizeof(wide[0])));
    if (rc) return rc;
  }
  for (real **pp : bulk) {
    int rc = dalloc(pp);
    if (rc) return rc;
  }
  for (double **pp : wide) {
    int rc = dalloc(pp);
    if (rc) return rc;
  }
  S.gamma_boris = S.cool_v = S.cool_b = S.curlb = nullptr;
  S.delta_ke = nullptr;
  S.rk = RkeOut{};
  S.rk4k = RkK{};
  S.rk4s = RkK{};
  if (params->fourth_order && params->resistive_mhd) {
    int rc = 0;
    for (int q = 0; q < 4 && !rc; ++q) rc = dalloc(&S.rk4k.k[q]);
    for (int q = 0; q < 4 && !rc; ++q) rc = dalloc(&S.rk4s.k[q]);
    if (rc) return rc;
  }
  if (params->rke) {
    int rc = dalloc(&S.delta_ke);
    for (int q = 0; q < 3 && !rc; ++q) rc = dalloc(&S.rk.dk[q]);
    if (rc) return rc;
  }
  S.xi = S.eta_perp = nullptr;
  S.nf_flag = nullptr;
  S.obc_save = nullptr;
  S.obc_face = 0;
  if (S.any_open) {
    const size_t e = (size_t)(nmax + 2) * (size_t)(nmax + 2);
    S.obc_face = 2 * e;
    HIPCHK(hipMalloc((void **)&S.obc_save, sizeof(double) * 6 * S.obc_face));
    S.allocs.push_back(S.obc_save);
  }
  if (pi) {
    // xi_n = 0 until the first neutral_fraction (neutral.f90:38)
    int rc = dalloc(&S.xi);
    if (!rc && params->cowling_resistivity) rc = dalloc(&S.eta_perp);
    if (rc) return rc;
  }
  if (params->boris) {
    int rc = dalloc(&S.gamma_boris);
    if (rc) return rc;
    // 1 until the first set_dt (gamma_boris(:,:,:) = 1, lagran.F90:1092)
    LAUNCH_BOX("fill", k_fill, full_box(), S.gamma_boris, 1.0);
  }
  if (params->cooling_term) {
    int rc = dalloc(&S.cool_v);
    if (!rc) rc = dalloc(&S.cool_b);
    if (!rc && params->resistive_mhd) rc = dalloc(&S.curlb);
    if (rc) return rc;
  }
  if (params->use_viscous_damping) {
    int rc = dalloc(&S.qx);
    if (!rc) rc = dalloc(&S.qy);
    if (!rc) rc = dalloc(&S.qz);
    if (rc) return rc;
  } else {
    S.qx = S.qy = S.qz = nullptr;
  }
  // partial sums: largest reduction grid (0..n+1 per axis) x 4 values
  dim3 gr = grid_from0(n[0] + 2, n[1] + 2, n[2] + 2);
  S.partial_cap = (size_t)gr.x * gr.y * gr.z * 4;
  int tiles_x;
  Box rb = full_box();
  const dim3 grs = resist_grid(rb, &tiles_x);
  if ((size_t)grs.x * grs.y * grs.z > S.partial_cap) S.partial_cap = (size_t)grs.x * grs.y * grs.z;
  // + RED_ROWS x RED_MAXV level-1 results after the per-block partials
  HIPCHK(hipMalloc((void **)&S.partial, sizeof(double) * (S.partial_cap + RED_ROWS * RED_MAXV)));
  HIPCHK(hipMalloc((void **)&S.dscal, sizeof(double) * 16));
  HIPCHK(hipMemset(S.dscal, 0, sizeof(double) * 16));
  HIPCHK(hipHostMalloc((void **)&S.hscal, sizeof(double) * 18));
  memset(S.hscal, 0, sizeof(double) * 18);
  if (pi) S.nf_flag = (int *)(S.hscal + 17);
  S.ticket = 0;
  HIPCHK(hipStreamSynchronize(S.stream));
  S.dt = S.dt2 = S.dtr = S.time = 0.0;
  S.n_s_stages = S.peak_substeps = S.last_substeps = 0;
  S.first_set_dt = 1;
  S.step = 0;
  S.ready = true;
  return 0;
}

int api_upload(const lare_fields *f) {
  if (!S.ready) return fail(LARE_E_STATE, "lare_dev_upload before lare_dev_init");
  if (!f || !f->rho || !f->energy || !f->vx || !f->vy || !f->vz || !f->bx || !f->by || !f->bz)
    return fail(LARE_E_ARG, "lare_dev_upload: missing field");
  if (S.p.use_viscous_damping && !f->visc3) return fail(LARE_E_ARG, "visc3 required with viscous damping");
  HIPCHK(hipStreamSynchronize(S.stream));
  XferSet x = state_xfer(f);
  xfer_add(x, S.visc3, f->visc3, FK_NODE);
  int rc = transfer(x, true);
  if (rc) return rc;
  S.loaded = true;
  return 0;
}

int api_download(lare_fields *f) {
  if (!S.loaded) return fail(LARE_E_STATE, "lare_dev_download before lare_dev_upload");
  if (!f) return fail(LARE_E_ARG, "lare_dev_download: NULL");
  HIPCHK(hipStreamSynchronize(S.stream));
  return transfer(state_xfer(f), false);
}

int api_get_scalars(lare_scalars *o) {
  if (!S.ready) return fail(LARE_E_STATE, "not initialised");
  double acc[2];
  int rc = read_scalars(8, 2, acc);
  if (rc) return rc;
  o->dt = S.dt;
  o->dtr = S.dtr;
  o->time = S.time;
  o->total_visc_heating = acc[0];
  o->total_ohmic_heating = acc[1];
  o->n_s_stages = S.n_s_stages;
  o->peak_substeps = S.peak_substeps;
  o->last_substeps = S.last_substeps;
  o->first_set_dt = S.first_set_dt;
  o->step = S.step;
  return 0;
}

int api_set_scalars(const lare_scalars *in) {
  if (!S.ready) return fail(LARE_E_STATE, "not initialised");
  S.dt = in->dt;
  S.dtr = in->dtr;
  S.time = in->time;
  S.n_s_stages = in->n_s_stages;
  S.peak_substeps = in->peak_substeps;
  S.last_substeps = in->last_substeps;
  S.first_set_dt = in->first_set_dt;
  S.step = in->step;
  double acc[2] = {in->total_visc_heating, in->total_ohmic_heating};
  // a step returns before its last folds have run, and they write the mirror too
  HIPCHK(hipStreamSynchronize(S.stream));
  HIPCHK(hipMemcpy(S.dscal + 8, acc, sizeof(acc), hipMemcpyHostToDevice));
  S.hscal[8] = acc[0];
  S.hscal[9] = acc[1];
  return 0;
}

#define REQUIRE_LOADED() \
  if (!S.loaded) return fail(LARE_E_STATE, "%s before lare_dev_upload", __func__)

int api_lagrangian_step(void) {
  REQUIRE_LOADED();
  int rc = lagrangian_step(false);
  if (rc) return rc;
  return check_neutral_fault("lagrangian_step", false);
}

int api_eulerian_remap(int32_t step) {
  REQUIRE_LOADED();
  return eulerian_remap(step, false);
}

int api_eta_calc(void) {
  REQUIRE_LOADED();
  return eta_calc();
}

int api_conduct_heat(void) {
  REQUIRE_LOADED();
  if (S.p.kappa_0 <= 0.0) return fail(LARE_E_ARG, "conduct_heat needs kappa_0 > 0");
  int rc = calc_s_stages();
  if (rc) return rc;
  rc = heat_conduct_sts2(0);
  if (rc) return rc;
  return check_neutral_fault("conduct_heat", false);
}

int api_boundary_conditions(void) {
  REQUIRE_LOADED();
  return boundary_conditions();
}

int api_neutral_fraction(void) {
  REQUIRE_LOADED();
  if (!S.pi_eos) return fail(LARE_E_STATE, "neutral_fraction needs eos_number EOS_ION or EOS_PI");
  int rc = neutral_fraction(S.energy, TMODE_DIRECT);
  if (rc) return rc;
  return check_neutral_fault("neutral_fraction", false);
}

int api_perpendicular_resistivity(void) {
  REQUIRE_LOADED();
  if (!S.eta_perp) return fail(LARE_E_STATE, "perpendicular_resistivity needs cowling_resistivity");
  return perpendicular_resistivity();
}

// xi_n and eta_perp (0..n, zero elsewhere) in the cell layout
int api_get_neutral(double *xi_h, double *ep_h) {
  REQUIRE_LOADED();
  if ((xi_h && !S.xi) || (ep_h && !S.eta_perp))
    return fail(LARE_E_STATE, "get_neutral: the partially ionised arrays are off");
  HIPCHK(hipStreamSynchronize(S.stream));
  XferSet x = {};
  xfer_add(x, S.xi, xi_h, FK_CELL);
  xfer_add(x, S.eta_perp, ep_h, FK_CELL);
  int rc = transfer(x, false);
  if (rc) return rc;
  if (ep_h) {
    // the array exists at nodes 0..n only (neutral.f90:73-131)
    const long ex = nx() + 4, ey = ny() + 4, ez = nz() + 4;
    for (long k = 0; k < ez; ++k)
      for (long j = 0; j < ey; ++j)
        for (long i = 0; i < ex; ++i)
          if (i < 1 || i > nx() + 1 || j < 1 || j > ny() + 1 || k < 1 || k > nz() + 1) ep_h[(k * ey + j) * ex + i] = 0.0;
  }
  return rc;
}

// the four sums of k_energy to scalars 0..3
int energy_sums() {
  const Box b = marched(nodes0n());
  const dim3 gr = zchunk_grid(b);
  LAUNCH("energy", (k_energy<PadLayout, real>), gr, box_block(), S.g, b, PadLayout{S.g}, S.rho, S.energy, S.vx, S.vy,
         S.vz, S.bx, S.by, S.bz, S.partial);
  return final_reduce(gr, 4, 8, 0, 0);
}

int api_energy_account(double en[3], double *divb) {
  REQUIRE_LOADED();
  if (!en) return fail(LARE_E_ARG, "energy_account: NULL output");
  int rc = energy_sums();
  if (rc) return rc;
  double v[4];
  rc = read_scalars(0, 4, v);
  if (rc) return rc;
  en[0] = v[0];
  en[1] = v[1];
  en[2] = v[2];
  if (divb) *divb = -v[3];
  return 0;
}

// diagnostics.F90:613-629 energy_correction, then energy_bcs
int energy_correction() {
  LAUNCH_BOX("energy_correction", k_energy_correction, interior(), S.delta_ke, S.rho, S.energy);
  return energy_bcs();
}

int api_energy_correction() {
  REQUIRE_LOADED();
  if (!S.delta_ke) return fail(LARE_E_STATE, "energy_correction needs rke on");
  return energy_correction();
}

// lare3d.f90:82-87 loop body (lagrangian_step, eulerian_remap,
// energy_correction when rke, eta_calc)
int api_step(int32_t step, double *dt, double *time) {
  REQUIRE_LOADED();
  S.step = step;
  int rc = 0;
  if (S.pi_eos) {
    rc = neutral_fraction(S.energy, TMODE_DIRECT);
    if (rc) return rc;
  }
  rc = lagrangian_step(true);
  if (rc) return rc;
  rc = eulerian_remap(step, false);
  if (rc) return rc;
  if (S.delta_ke) {
    rc = energy_correction();
    if (rc) return rc;
  }
  rc = eta_calc();
  if (rc) return rc;
  // the fold of the corrector's heating total comes after the step's last
  // neutral_fraction
  rc = check_neutral_fault("step", true);
  if (rc) return rc;
  if (!isfinite(S.dt) || (S.dt <= 0.0 && !S.p.restart))
    return fail(LARE_F_NONFINITE, "step %d: invalid dt %g", step, S.dt);
  if (dt) *dt = S.dt;
  if (time) *time = S.time;
  return 0;
}

int api_profile(int32_t enable) {
  if (!S.ready) return fail(LARE_E_STATE, "not initialised");
  prof_flush();
  if (enable && !S.prof) S.acc.clear();
  S.prof = enable != 0;
  return 0;
}

int api_kernel_stats(char *names, int32_t name_len, int32_t *counts, double *total_ms, int32_t cap) {
  if (!S.ready) return fail(LARE_E_STATE, "not initialised");
  prof_flush();
  int q = 0;
  for (auto &a : S.acc) {
    if (q >= cap) break;
    if (names && name_len > 0) {
      strncpy(names + (size_t)q * name_len, a.name.c_str(), (size_t)name_len - 1);
      names[(size_t)q * name_len + name_len - 1] = 0;
    }
    if (counts) counts[q] = a.count;
    if (total_ms) total_ms[q] = a.ms;
    ++q;
  }
  return q;
}

int api_synchronize(void) {
  if (!S.stream) return 0;
  HIPCHK(hipStreamSynchronize(S.stream));
  return 0;
}

int api_finalize(void) {
  free_all();
  if (S.stream) {
    (void)hipStreamDestroy(S.stream);
    S.stream = nullptr;
  }
  return 0;
}


// ============================================================================
// learned conduction surrogate
// ============================================================================
// Runtime of the learned conduction surrogate (kernels in surrogate.hpp).
//
// Data flow:
//   collect: features of the current state -> random interior cells -> rows
//            of 27 x 12 raw channels; one plain RKL2 super-step on the same
//            state gives the target dT of each row; the state is restored.
//   fit_norm: channel mean / std and the target scale from the rows; the
//            stored rows are standardised in place.
//   train:   Adam on mini-batches drawn from the rows; forward and backward
//            GEMMs in BF16 MFMA with FP32 accumulation.
//   conduct: features -> MFMA inference over the interior -> E1; residual
//            r = |E1 - E0 - dt/2 (L(E0) + L(E1))| / |E0| (L2 norms over the
//            interior, L = heat-flux divergence / rho of conduct.f90:152-291);
//            r <= tol accepts E1, otherwise the super-step is redone by RKL2.



struct Sur {
  char *param_mem = nullptr, *field_mem = nullptr, *batch_mem = nullptr;  // the allocations of the groups below
  float *w = nullptr, *gr = nullptr, *m = nullptr, *v = nullptr;  // SUR_NPARAM each
  unsigned short *w1t = nullptr, *w2t = nullptr;                   // packed BF16 for inference
  bool have_params = false, have_norm = false;
  SurNorm nm;
  int adam_t = 0;
  float *feat = nullptr;      // ntot * SUR_CH
  real *E1 = nullptr, *trap = nullptr, *E0save = nullptr;
  // dataset
  float *X = nullptr, *y = nullptr;
  int *cells = nullptr;
  int rows = 0, cap = 0;
  bool standardised = false;
  // mini-batch work arrays (capacity bcap columns)
  int bcap = 0;
  float *Xb = nullptr, *yb = nullptr, *H1 = nullptr, *H2 = nullptr, *yo = nullptr, *dy = nullptr, *dZ2 = nullptr,
        *dZ1 = nullptr, *lossacc = nullptr, *losshist = nullptr;
  int *row = nullptr;
  int losscap = 0;
  // use inside lagrangian_step
  int enabled = 0;
  double tol = 1.0e-4;
  int accepted = 0, rejected = 0;
  double last_res = 0.0;
};
Sur SU;

template <class T>
void sfree(T *&p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

void sur_free_batch() {
  sfree(SU.batch_mem);
  SU.Xb = SU.yb = SU.H1 = SU.H2 = SU.yo = SU.dy = SU.dZ2 = SU.dZ1 = nullptr;
  SU.lossacc = nullptr;
  SU.row = nullptr;
  SU.bcap = 0;
}

void sur_free() {
  sfree(SU.param_mem);
  sfree(SU.field_mem);
  sfree(SU.X); sfree(SU.y); sfree(SU.cells); sfree(SU.losshist);
  sur_free_batch();
  const int en = SU.enabled;
  const double tol = SU.tol;
  SU = Sur();
  SU.enabled = en;  // the mode survives re-initialisation; parameters do not
  SU.tol = tol;
}

template <class T>
int salloc(T **p, size_t count) {
  hipError_t e = hipMalloc((void **)p, sizeof(T) * count);
  if (e != hipSuccess) return fail(LARE_E_NOMEM, "hipMalloc of %zu bytes failed: %s", sizeof(T) * count,
                                   hipGetErrorString(e));
  return 0;
}

// the arrays of one group in one allocation
struct SurPart {
  void **p;
  size_t bytes;
  template <class T>
  SurPart(T **q, size_t count) : p((void **)q), bytes(slab_bytes(sizeof(T) * count)) {}
};
int salloc_group(char **mem, std::initializer_list<SurPart> parts) {
  size_t total = 0;
  for (const SurPart &q : parts) total += q.bytes;
  int rc = salloc(mem, total);
  if (rc) return rc;
  char *at = *mem;
  for (const SurPart &q : parts) {
    *q.p = at;
    at += q.bytes;
  }
  return 0;
}

int sur_alloc_params() {
  if (SU.w) return 0;
  int rc = salloc_group(&SU.param_mem, {{&SU.w, SUR_NPARAM}, {&SU.gr, SUR_NPARAM}, {&SU.m, SUR_NPARAM},
                                        {&SU.v, SUR_NPARAM}, {&SU.w1t, SUR_H * SUR_KP}, {&SU.w2t, SUR_H * SUR_HP}});
  if (rc) return rc;
  HIPCHK(hipMemsetAsync(SU.m, 0, sizeof(float) * SUR_NPARAM, S.stream));
  HIPCHK(hipMemsetAsync(SU.v, 0, sizeof(float) * SUR_NPARAM, S.stream));
  return 0;
}

int sur_alloc_fields() {
  if (SU.feat) return 0;
  int rc = salloc_group(&SU.field_mem,
                        {{&SU.feat, S.ntot * SUR_CH}, {&SU.E1, S.ntot}, {&SU.trap, S.ntot}, {&SU.E0save, S.ntot}});
  if (rc) return rc;
  // cells never written by the feature kernel are never read by it either;
  // zero them once so no stale bits reach a gather
  HIPCHK(hipMemsetAsync(SU.feat, 0, sizeof(float) * S.ntot * SUR_CH, S.stream));
  return 0;
}

int sur_ensure_batch(int cols) {
  if (cols <= SU.bcap) return 0;
  sur_free_batch();
  const size_t c = (size_t)cols;
  int rc = salloc_group(&SU.batch_mem, {{&SU.Xb, c * SUR_K}, {&SU.yb, c}, {&SU.row, c}, {&SU.H1, c * SUR_H},
                                        {&SU.H2, c * SUR_H}, {&SU.yo, c}, {&SU.dy, c}, {&SU.dZ2, c * SUR_H},
                                        {&SU.dZ1, c * SUR_H}, {&SU.lossacc, (c + 255) / 256}});
  if (rc) return rc;
  SU.bcap = cols;
  return 0;
}

unsigned blocks_for(size_t n, unsigned bs = 256) { return (unsigned)((n + bs - 1) / bs); }

// Forward pass (and, with targets y, backward) over nb columns, a multiple of
// 16, of which the first nreal are rows of X: rows drawn by hash of seed from
// the first `draw`, or (draw = 0) rows 0 .. nreal-1.
SurBatch sur_batch(const float *X, const float *y, int nb, int nreal) {
  return SurBatch{X, y, SU.row, SU.H1, SU.H2, SU.dZ1, SU.dZ2, SU.yo, SU.dy, nb, nreal};
}
int sur_fb(const SurBatch &b, int draw, unsigned long long seed) {
  LAUNCH("sur_fb", k_sur_fb, dim3((unsigned)(b.nb / 16)), dim3(256), b, SU.w, draw, seed);
  return 0;
}

int sur_enabled() { return SU.enabled; }

int sur_pack() {
  LAUNCH("sur_pack", k_sur_pack, dim3(blocks_for((size_t)SUR_H * SUR_KP)), dim3(256), SU.w, SU.w1t, SU.w2t);
  return 0;
}

int sur_features(int normalise) {
  int rc = sur_alloc_fields();
  if (rc) return rc;
  const double logdt = log(S.dt > 0.0 ? S.dt : 1.0e-300);
  LAUNCH_BOX("sur_features", k_sur_features, mkbox(0, nx() + 1, 0, ny() + 1, 0, nz() + 1), S.energy, S.rho, S.bx,
             S.by, S.bz, SU.feat, SU.nm, S.tfac, logdt, normalise);
  return 0;
}

// Trapezoidal residual |E1 - E0 - dt/2 (L(E0) + L(E1))| / |E0| (L2 over the
// interior) of a candidate super-step E1 from E0 = S.energy, using the
// Larsen factor of the last calc_s_stages.  The stage kernels with all
// history weights zero evaluate the trapezoid into SU.trap.
int sur_residual(const real *E1, double *res) {
  CondArgs ca = {S.p.kappa_0, S.tfac, S.dt};
  int rc0 = rkl2_stage1(S.energy, S.Yb[0], ca, 0.0);
  if (rc0) return rc0;
  rc0 = rkl2_stage(TMODE_WRAP, E1, E1, S.energy, SU.trap, ca, 0.0, 0.0, 0.0, 0.5, 0.5);
  if (rc0) return rc0;
  dim3 gr = box_grid(interior());
  LAUNCH("sur_residual", k_sur_residual, gr, box_block(), S.g, S.energy, E1, SU.trap, S.partial);
  int rc = final_reduce(gr, 2, 0, 0, 0);
  if (rc) return rc;
  double v[2];
  rc = read_scalars(0, 2, v);
  if (rc) return rc;
  *res = v[1] > 0.0 ? sqrt(v[0] / v[1]) : 0.0;
  return 0;
}

// One surrogate super-step of length S.dt on S.energy (stages and Larsen
// factor from calc_s_stages), checked and, if rejected, redone by RKL2.
int sur_conduct_step(int delta_mode, double *res_out, int *acc_out) {
  if (!SU.have_params || !SU.have_norm) return fail(LARE_E_STATE, "surrogate: no trained parameters loaded");
  int rc = calc_s_stages();
  if (rc) return rc;
  rc = sur_features(1);
  if (rc) return rc;
  const dim3 gi((unsigned)((nx() + SIT_WX - 1) / SIT_WX), (unsigned)((ny() + SIT_NW - 1) / SIT_NW),
                (unsigned)((nz() + SIT_ZC - 1) / SIT_ZC));
  LAUNCH("sur_infer", k_sur_infer_t, gi, dim3(64 * SIT_NW), S.g, SU.feat, SU.w1t, SU.w2t, SU.w, S.energy, SU.E1,
         S.tfac, SU.nm.y_scale);
  double r;
  rc = sur_residual(SU.E1, &r);
  if (rc) return rc;
  SU.last_res = r;
  const int ok = (r == r) && r <= SU.tol;
  if (res_out) *res_out = r;
  if (acc_out) *acc_out = ok;
  if (ok) {
    ++SU.accepted;
    LAUNCH_BOX("rkl2_final", k_rkl2_final, cell_box(), SU.E1, S.energy, delta_mode);
    return 0;
  }
  ++SU.rejected;
  return heat_conduct_sts2(delta_mode);
}

// rows of standardised inputs (SUR_K floats each) from the host into SU.Xb,
// zero-padded to a multiple of 16 columns
int sur_stage_rows(const float *X, const float *t, int rows, int *nb_out) {
  const int nb = (rows + 15) / 16 * 16;
  int rc = sur_ensure_batch(nb);
  if (rc) return rc;
  HIPCHK(hipMemsetAsync(SU.Xb, 0, sizeof(float) * (size_t)nb * SUR_K, S.stream));
  HIPCHK(hipMemcpyAsync(SU.Xb, X, sizeof(float) * (size_t)rows * SUR_K, hipMemcpyHostToDevice, S.stream));
  if (t) {
    HIPCHK(hipMemsetAsync(SU.yb, 0, sizeof(float) * nb, S.stream));
    HIPCHK(hipMemcpyAsync(SU.yb, t, sizeof(float) * rows, hipMemcpyHostToDevice, S.stream));
  }
  *nb_out = nb;
  return 0;
}


int api_sur_set_params(const float *params, int32_t n) {
  if (!S.ready) return fail(LARE_E_STATE, "not initialised");
  if (!params || n != SUR_NPARAM) return fail(LARE_E_ARG, "surrogate parameters: need %d floats, got %d", SUR_NPARAM, n);
  int rc = sur_alloc_params();
  if (rc) return rc;
  HIPCHK(hipMemcpy(SU.w, params, sizeof(float) * SUR_NPARAM, hipMemcpyHostToDevice));
  HIPCHK(hipMemsetAsync(SU.m, 0, sizeof(float) * SUR_NPARAM, S.stream));
  HIPCHK(hipMemsetAsync(SU.v, 0, sizeof(float) * SUR_NPARAM, S.stream));
  SU.adam_t = 0;
  SU.have_params = true;
  return sur_pack();
}

int api_sur_get_params(float *params, int32_t n) {
  if (!SU.have_params) return fail(LARE_E_STATE, "surrogate: no parameters");
  if (!params || n != SUR_NPARAM) return fail(LARE_E_ARG, "surrogate parameters: need %d floats, got %d", SUR_NPARAM, n);
  HIPCHK(hipStreamSynchronize(S.stream));
  HIPCHK(hipMemcpy(params, SU.w, sizeof(float) * SUR_NPARAM, hipMemcpyDeviceToHost));
  return 0;
}

int api_sur_set_norm(const float *mu, const float *sd, float y_scale) {
  if (!mu || !sd || !(y_scale > 0.0f)) return fail(LARE_E_ARG, "surrogate norm: bad arguments");
  for (int q = 0; q < SUR_CH; ++q) {
    SU.nm.mu[q] = q < SUR_NCH ? mu[q] : 0.0f;
    SU.nm.sd[q] = q < SUR_NCH ? sd[q] : 1.0f;
    if (!(SU.nm.sd[q] > 0.0f)) return fail(LARE_E_ARG, "surrogate norm: std of channel %d is not positive", q);
  }
  SU.nm.y_scale = y_scale;
  SU.have_norm = true;
  return 0;
}

int api_sur_get_norm(float *mu, float *sd, float *y_scale) {
  if (!SU.have_norm) return fail(LARE_E_STATE, "surrogate: no normalisation");
  for (int q = 0; q < SUR_NCH; ++q) {
    if (mu) mu[q] = SU.nm.mu[q];
    if (sd) sd[q] = SU.nm.sd[q];
  }
  if (y_scale) *y_scale = SU.nm.y_scale;
  return 0;
}

int api_sur_collect(int32_t count, uint64_t seed, int32_t *total) {
  REQUIRE_LOADED();
  if (count <= 0) return fail(LARE_E_ARG, "surrogate collect: count %d", count);
  if (SU.standardised) return fail(LARE_E_STATE, "surrogate collect: rows already standardised");
  if (S.p.kappa_0 <= 0.0 || !(S.dt > 0.0)) return fail(LARE_E_ARG, "surrogate collect needs kappa_0 > 0 and dt > 0");
  if (SU.rows + count > SU.cap) {  // grow the row store
    const int ncap = (SU.rows + count) * 2;
    float *X = nullptr, *y = nullptr;
    int *cells = nullptr;
    int rc = salloc(&X, (size_t)ncap * SUR_K);
    if (!rc) rc = salloc(&y, (size_t)ncap);
    if (!rc) rc = salloc(&cells, (size_t)ncap);
    if (rc) return rc;
    if (SU.rows) {
      HIPCHK(hipMemcpyAsync(X, SU.X, sizeof(float) * SU.rows * SUR_K, hipMemcpyDeviceToDevice, S.stream));
      HIPCHK(hipMemcpyAsync(y, SU.y, sizeof(float) * SU.rows, hipMemcpyDeviceToDevice, S.stream));
    }
    HIPCHK(hipStreamSynchronize(S.stream));
    sfree(SU.X); sfree(SU.y); sfree(SU.cells);
    SU.X = X; SU.y = y; SU.cells = cells;
    SU.cap = ncap;
  }
  int rc = calc_s_stages();
  if (rc) return rc;
  rc = sur_features(0);
  if (rc) return rc;
  int *cells = SU.cells + SU.rows;
  LAUNCH("sur_sample", k_sur_sample_cells, dim3(blocks_for(count)), dim3(256), S.g, SU.feat, (unsigned long long)seed,
         count, cells);
  LAUNCH("sur_gather", k_sur_gather, dim3(blocks_for((size_t)count * SUR_K)), dim3(256), S.g, SU.feat, cells, count,
         SU.X + (size_t)SU.rows * SUR_K);
  HIPCHK(hipMemcpyAsync(SU.E0save, S.energy, sizeof(real) * S.ntot, hipMemcpyDeviceToDevice, S.stream));
  rc = heat_conduct_sts2(0);
  if (rc) return rc;
  LAUNCH("sur_target", k_sur_target, dim3(blocks_for(count)), dim3(256), SU.E0save, S.energy, cells, count, S.tfac,
         SU.y + SU.rows);
  HIPCHK(hipMemcpyAsync(S.energy, SU.E0save, sizeof(real) * S.ntot, hipMemcpyDeviceToDevice, S.stream));
  HIPCHK(hipStreamSynchronize(S.stream));
  SU.rows += count;
  if (total) *total = SU.rows;
  return 0;
}

int api_sur_rows(float *X, float *y, int32_t rows) {
  if (rows < 0 || rows > SU.rows) return fail(LARE_E_ARG, "surrogate rows: %d requested, %d held", rows, SU.rows);
  HIPCHK(hipStreamSynchronize(S.stream));
  if (X && rows) HIPCHK(hipMemcpy(X, SU.X, sizeof(float) * (size_t)rows * SUR_K, hipMemcpyDeviceToHost));
  if (y && rows) HIPCHK(hipMemcpy(y, SU.y, sizeof(float) * (size_t)rows, hipMemcpyDeviceToHost));
  return 0;
}

int api_sur_fit_norm(void) {
  if (SU.rows < 2) return fail(LARE_E_STATE, "surrogate fit_norm: %d rows collected", SU.rows);
  if (SU.standardised) return fail(LARE_E_STATE, "surrogate fit_norm: rows already standardised");
  std::vector<float> X((size_t)SU.rows * SUR_K), y(SU.rows);
  HIPCHK(hipStreamSynchronize(S.stream));
  HIPCHK(hipMemcpy(X.data(), SU.X, sizeof(float) * X.size(), hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(y.data(), SU.y, sizeof(float) * y.size(), hipMemcpyDeviceToHost));
  // channel statistics of the centre cell (neighbour 13) of every row
  for (int ch = 0; ch < SUR_CH; ++ch) {
    double s = 0.0, s2 = 0.0;
    for (int r = 0; r < SU.rows; ++r) {
      const double x = X[(size_t)r * SUR_K + 13 * SUR_CH + ch];
      s += x;
      s2 += x * x;
    }
    const double mu = s / SU.rows;
    double var = s2 / SU.rows - mu * mu;
    double sd = var > 1.0e-12 * (1.0 + mu * mu) ? sqrt(var) : 1.0;
    // log dt (channel 5) is nearly constant within one training run; a floor
    // of 1 keeps a step with a somewhat different dt inside the input range
    if (ch == 5 && sd < 1.0) sd = 1.0;
    SU.nm.mu[ch] = ch < SUR_NCH ? (float)mu : 0.0f;
    SU.nm.sd[ch] = ch < SUR_NCH ? (float)sd : 1.0f;
  }
  double sy2 = 0.0;
  for (int r = 0; r < SU.rows; ++r) sy2 += (double)y[r] * y[r];
  const double ys = sqrt(sy2 / SU.rows);
  SU.nm.y_scale = ys > 0.0 ? (float)ys : 1.0f;
  SU.have_norm = true;
  LAUNCH("sur_standardise", k_sur_standardise, dim3(blocks_for((size_t)SU.rows * SUR_K)), dim3(256), SU.X, SU.y,
         SU.rows, SU.nm);
  SU.standardised = true;
  return 0;
}

int api_sur_train(int32_t steps, int32_t batch, float lr, uint64_t seed, float *loss_out) {
  if (!S.ready) return fail(LARE_E_STATE, "not initialised");
  if (!SU.have_params) return fail(LARE_E_STATE, "surrogate train: no initial parameters");
  if (!SU.standardised) return fail(LARE_E_STATE, "surrogate train: call fit_norm after collecting rows");
  if (steps <= 0 || batch < 16 || batch % 16 != 0) return fail(LARE_E_ARG, "surrogate train: steps %d batch %d", steps, batch);
  int rc = sur_ensure_batch(batch);
  if (rc) return rc;
  if (steps > SU.losscap) {
    sfree(SU.losshist);
    rc = salloc(&SU.losshist, (size_t)steps);
    if (rc) return rc;
    SU.losscap = steps;
  }
  const float b1 = 0.9f, b2 = 0.999f;
  for (int s = 0; s < steps; ++s) {
    const unsigned long long bseed = mix64(seed * 0x9E3779B97F4A7C15ull + (unsigned long long)s);
    const SurBatch bt = sur_batch(SU.X, SU.y, batch, batch);
    rc = sur_fb(bt, SU.rows, bseed);
    if (rc) return rc;
    SU.adam_t += 1;
    const float c1 = 1.0f - powf(b1, (float)SU.adam_t), c2 = 1.0f - powf(b2, (float)SU.adam_t);
    const AdamArgs aa = {SU.w, SU.m, SU.v, lr, b1, b2, 1.0e-8f, c1, c2};
    LAUNCH("sur_grads", k_sur_grads<true>, dim3(SUR_GB_ALL), dim3(256), bt, aa, SU.gr, SU.lossacc,
           1.0f / (float)batch, SU.losshist + s, 1);
  }
  rc = sur_pack();
  if (rc) return rc;
  HIPCHK(hipStreamSynchronize(S.stream));
  if (loss_out) HIPCHK(hipMemcpy(loss_out, SU.losshist, sizeof(float) * steps, hipMemcpyDeviceToHost));
  return 0;
}

int api_sur_forward(const float *X, int32_t rows, float *y) {
  if (!S.ready) return fail(LARE_E_STATE, "not initialised");
  if (!SU.have_params) return fail(LARE_E_STATE, "surrogate forward: no parameters");
  if (!X || !y || rows <= 0) return fail(LARE_E_ARG, "surrogate forward: bad arguments");
  int nb;
  int rc = sur_stage_rows(X, nullptr, rows, &nb);
  if (rc) return rc;
  rc = sur_fb(sur_batch(SU.Xb, nullptr, nb, rows), 0, 0);
  if (rc) return rc;
  HIPCHK(hipStreamSynchronize(S.stream));
  HIPCHK(hipMemcpy(y, SU.yo, sizeof(float) * rows, hipMemcpyDeviceToHost));
  return 0;
}

int api_sur_grad(const float *X, const float *t, int32_t rows, float *grad, float *loss) {
  if (!S.ready) return fail(LARE_E_STATE, "not initialised");
  if (!SU.have_params) return fail(LARE_E_STATE, "surrogate grad: no parameters");
  if (!X || !t || !grad || rows <= 0) return fail(LARE_E_ARG, "surrogate grad: bad arguments");
  int nb;
  int rc = sur_stage_rows(X, t, rows, &nb);
  if (rc) return rc;
  const SurBatch bt = sur_batch(SU.Xb, SU.yb, nb, rows);
  rc = sur_fb(bt, 0, 0);
  if (rc) return rc;
  LAUNCH("sur_grads", k_sur_grads<false>, dim3(SUR_GB_ALL), dim3(256), bt, AdamArgs{}, SU.gr, SU.lossacc, 1.0f,
         (float *)nullptr, 0);
  HIPCHK(hipStreamSynchronize(S.stream));
  HIPCHK(hipMemcpy(grad, SU.gr, sizeof(float) * SUR_NPARAM, hipMemcpyDeviceToHost));
  if (loss) {
    const int nblk = (int)blocks_for(nb);
    std::vector<float> part(nblk);
    HIPCHK(hipMemcpy(part.data(), SU.lossacc, sizeof(float) * nblk, hipMemcpyDeviceToHost));
    double s = 0.0;
    for (float p : part) s += p;
    *loss = (float)(s / rows);
  }
  return 0;
}

int api_sur_enable(int32_t on, double tol) {
  if (!(tol > 0.0)) return fail(LARE_E_ARG, "surrogate tolerance must be positive");
  if (on && S.pi_eos) return fail(LARE_E_ARG, "the conduction surrogate is trained for EOS_IDEAL only");
  if (on && S.any_open) return fail(LARE_E_ARG, "the conduction surrogate does not handle BC_OPEN sides");
  if (on && (!SU.have_params || !SU.have_norm)) return fail(LARE_E_STATE, "surrogate enable: no trained parameters");
  SU.enabled = on != 0;
  SU.tol = tol;
  return 0;
}

int api_sur_conduct(double *residual, int32_t *accepted) {
  REQUIRE_LOADED();
  if (S.p.kappa_0 <= 0.0) return fail(LARE_E_ARG, "surrogate conduct needs kappa_0 > 0");
  int acc = 0;
  int rc = sur_conduct_step(0, residual, &acc);
  if (accepted) *accepted = acc;
  return rc;
}

int api_sur_plain_residual(double *residual) {
  REQUIRE_LOADED();
  if (S.p.kappa_0 <= 0.0) return fail(LARE_E_ARG, "plain residual needs kappa_0 > 0");
  if (!residual) return fail(LARE_E_ARG, "plain residual: NULL output");
  int rc = sur_alloc_fields();
  if (!rc) rc = calc_s_stages();
  if (rc) return rc;
  HIPCHK(hipMemcpyAsync(SU.E0save, S.energy, sizeof(real) * S.ntot, hipMemcpyDeviceToDevice, S.stream));
  rc = heat_conduct_sts2(0);
  if (rc) return rc;
  HIPCHK(hipMemcpyAsync(SU.E1, S.energy, sizeof(real) * S.ntot, hipMemcpyDeviceToDevice, S.stream));
  HIPCHK(hipMemcpyAsync(S.energy, SU.E0save, sizeof(real) * S.ntot, hipMemcpyDeviceToDevice, S.stream));
  return sur_residual(SU.E1, residual);
}

int api_sur_stats(int32_t *accepted, int32_t *rejected, double *last_residual) {
  if (accepted) *accepted = SU.accepted;
  if (rejected) *rejected = SU.rejected;
  if (last_residual) *last_residual = SU.last_res;
  return 0;
}

// lare_dev_step followed by the scalars a driver reads after it, and
// optionally energy_account of the new state, read back in one copy.
int api_step_info(int32_t step, int32_t with_energy, lare_step_info *o) {
  REQUIRE_LOADED();
  if (!o) return fail(LARE_E_ARG, "step_info: NULL output");
  double dt = 0.0, t = 0.0;
  int rc = api_step(step, &dt, &t);
  if (rc) return rc;
  if (with_energy) {
    rc = energy_sums();
    if (rc) return rc;
  }
  double v[10];
  rc = read_scalars(0, 10, v);
  if (rc) return rc;
  o->dt = S.dt;
  o->dtr = S.dtr;
  o->time = S.time;
  o->total_visc_heating = v[8];
  o->total_ohmic_heating = v[9];
  o->en_b = with_energy ? v[0] : 0.0;
  o->en_ke = with_energy ? v[1] : 0.0;
  o->en_int = with_energy ? v[2] : 0.0;
  o->max_divb = with_energy ? -v[3] : 0.0;
  o->n_s_stages = S.n_s_stages;
  o->substeps = S.last_substeps;
  o->peak_substeps = S.peak_substeps;
  o->sur_accepted = SU.accepted;
  o->sur_rejected = SU.rejected;
  o->with_energy = with_energy ? 1 : 0;
  return 0;
}

// initial_conditions.f90:114-296 potential_field.  phi lives in the FP64
// scratch array F, the flux patch in F2.
int api_potential_field(const lare_potential *pf, int32_t *iterations, double *residual, double *bz_max) {
  REQUIRE_LOADED();
  if (!pf || !pf->flux0) return fail(LARE_E_ARG, "potential_field: NULL argument");
  const int N0 = nx(), N1 = ny(), N2 = nz();
  if (S.per[2]) return fail(LARE_E_ARG, "potential_field: the z axis must be BC_USER (flux patch below)");
  if (S.any_open) return fail(LARE_E_ARG, "potential_field: BC_OPEN sides are not supported");
  if (N2 > N1 + 2)
    return fail(LARE_E_ARG, "potential_field: nz = %d > ny + 2 = %d (the reference reads bz(1:nx, 1:nz, 0))", N2,
                N1 + 2);
  if (pf->max_iterations < 1) return fail(LARE_E_ARG, "potential_field: max_iterations < 1");
  double *phi = S.F, *flux0 = S.F2;
  HIPCHK(hipStreamSynchronize(S.stream));
  HIPCHK(hipMemcpy(flux0, pf->flux0, sizeof(double) * (size_t)N0 * N1, hipMemcpyHostToDevice));
  LAUNCH_BOX("fill", k_fill64, full_box(), phi, 0.0);
  const int ncol = (N0 + 1) / 2;
  const dim3 gs((unsigned)(((long)ncol * N1 + 63) / 64));
  const Box zb = mkbox(-1, N0 + 2, -1, N1 + 2, 0, 0);
  auto line = [&](int ax, int op) -> int {
    const int u = ax == 0 ? 1 : 0, wa = ax == 2 ? 1 : 2;
    LAUNCH("bc_phi", k_bc_axis, dim3((unsigned)((S.n[u] + 5 + 63) / 64), (unsigned)(S.n[wa] + 5)), dim3(64), S.g, phi,
           op, ax);
    return 0;
  };
  auto phi_bcs = [&]() -> int {
    // phi_mpi: exchanges on periodic axes, the z boundaries, then the
    // zero-gradient x and y walls
    for (int ax = 0; ax < 3; ++ax) {
      int rc = S.per[ax] ? line(ax, BC_PER_CELL) : 0;
      if (rc) return rc;
    }
    LAUNCH("phi_zbc", k_phi_zbc, box_grid(zb), box_block(), S.g, zb, phi, flux0);
    for (int ax = 0; ax < 2; ++ax) {
      int rc = S.per[ax] ? 0 : line(ax, BC_PHI_NEU);
      if (rc) return rc;
    }
    return 0;
  };
  // the batch state lives in the level-1 rows of the reductions
  static_assert(sizeof(SorBatch) <= sizeof(double) * RED_ROWS * RED_MAXV, "batch state");
  SorBatch *const sb = (SorBatch *)(S.partial + S.partial_cap);
  SorBatch hb;
  SorArgs sa = {pf->omega, pf->dx1, pf->dy1, pf->dz1, pf->fractional_error, 0, 0, 0, 1};
  int *const maps[2] = {&sa.mapx, &sa.mapy};
  bool ghost[2] = {false, false};  // periodic with an odd number of points
  for (int ax = 0; ax < 2; ++ax) {
    ghost[ax] = S.per[ax] && (S.n[ax] & 1);
    *maps[ax] = !S.per[ax] ? 1 : (ghost[ax] ? 0 : 2);
  }
  int its = 0;
  double res = 0.0;
  for (bool done = false; !done;) {
    LAUNCH("sor_reset", k_sor_reset, dim3(1), dim3(64), sb);
    const int batch = pf->max_iterations - its < SOR_BATCH ? pf->max_iterations - its : SOR_BATCH;
    for (sa.q = 0; sa.q < batch; ++sa.q)
      for (int z1 = 1; z1 <= 2; ++z1) {
        LAUNCH("sor", k_sor_pass, gs, dim3(64), S.g, phi, flux0, z1, sa, sb);
        sa.first = 0;
        for (int ax = 0; ax < 2; ++ax) {
          int rc = ghost[ax] ? line(ax, BC_PER_CELL) : 0;
          if (rc) return rc;
        }
      }
    HIPCHK(hipMemcpyAsync(&hb, sb, sizeof(hb), hipMemcpyDeviceToHost, S.stream));
    HIPCHK(hipStreamSynchronize(S.stream));
    for (int q = 0; q < batch && !done; ++q) {
      memcpy(&res, &hb.err[q], sizeof(res));
      ++its;
      done = res < pf->fractional_error || its >= pf->max_iterations;
    }
  }
  int rc = phi_bcs();
  if (rc) return rc;
  // B = -grad phi, bfield_bcs, scale by the largest bz below, bfield_bcs
  LAUNCH_BOX("phi_to_b", k_phi_to_b, full_box(), phi, S.bx, S.by, S.bz);
  rc = bfield_bcs(S.bx, S.by, S.bz);
  if (rc) return rc;
  const Box lb = mkbox(1, N0, 1, N2, 0, 0);
  const dim3 gb = box_grid(lb);
  LAUNCH("bz_lower", k_bz_lower, gb, box_block(), S.g, lb, S.bz, S.partial);
  rc = final_reduce(gb, 1, 1, 15, 0);
  if (rc) return rc;
  LAUNCH_BOX("scale_b", k_scale_b, full_box(), S.bx, S.by, S.bz, S.dscal);
  rc = bfield_bcs(S.bx, S.by, S.bz);
  if (rc) return rc;
  double bm;
  rc = read_scalars(15, 1, &bm);
  if (rc) return rc;
  if (iterations) *iterations = its;
  if (residual) *residual = res;
  if (bz_max) *bz_max = -bm;
  return 0;
}
