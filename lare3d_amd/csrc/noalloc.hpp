// noalloc.hpp -- lare_dev_energy_account_noalloc: energy_account on the
// caller's own device arrays, with no device allocation by the library.
//
// For callers that cannot call hipMalloc (code under HIP graph capture,
// tight serving loops, harnesses that forbid it).  The kernels are those of
// lare_dev_energy_account (k_energy with the Fortran layout, then the same
// fold of the per-block partials, in one level or two), so the results are the same
// bits for the same field values.  Instead of the partial buffer that
// lare_dev_init allocates, they use `scratch`, a fixed array in device
// memory that each GPU holds from the library's load to the end of the
// process:
//   [0, NA_MET)            dxb, dyb, dzb of the host grid
//   [NA_MET, +NA_PART)     per-block partial sums, 4 doubles per block
//   [.., +NA_LEVEL1)       level-1 results of the fold
//   [.., +NA_OUT)          the four final sums
// Every call on one GPU uses that GPU's one copy of the array and leaves
// its last contents there: calls that overlap on one GPU (several host
// threads, or streams the caller runs concurrently) race.  Nothing in it
// needs to start at zero -- every value read is written earlier in the
// same call.
//
// Included once by lare_dev.hip, after the fp64 runtime.

#define NA_NMAX 4096                              // cells per axis
#define NA_LEN (NA_NMAX + 8)                       // one metric array, index i + 2
#define NA_MET (3 * NA_LEN)
#define NA_MAX_BLOCKS 262144                       // energy grid blocks (n+1)^3 / 256
#define NA_PART (NA_MAX_BLOCKS * 4)
#define NA_LEVEL1 (RED_ROWS * RED_MAXV)
#define NA_OUT 8
#define NA_TOTAL (NA_MET + NA_PART + NA_LEVEL1 + NA_OUT)

static __device__ __align__(256) double scratch[NA_TOTAL];

// The metrics travel as kernel arguments, NA_ARGS values at a time: a launch is
// queued in about 3 us, where a blocking copy of a few hundred bytes takes
// about 10.  Up to NA_ARG_LAUNCHES of them (about 300 cells per axis); above,
// a copy per axis.  At 64^3 the whole call went from 66 to 32 us.
#define NA_ARGS 480
#define NA_ARG_LAUNCHES 2
struct NaMetrics {
  double v[NA_ARGS];
  int first, count, len[3];  // of the run dxb, dyb, dzb end to end
};
static __global__ __launch_bounds__(NA_ARGS) void k_na_metrics(NaMetrics m, double *__restrict__ met) {
  const int t = (int)threadIdx.x;
  if (t >= m.count) return;
  int e = m.first + t, a = 0;
  while (a < 2 && e >= m.len[a]) e -= m.len[a++];
  met[a * NA_LEN + 1 + e] = m.v[t];
}

namespace {

// Device address of `scratch` on each GPU (the host symbol is only a
// stand-in): looked up once per device with that device current.
#define NA_MAXDEV 64
double *g_na_ptr[NA_MAXDEV] = {};

int na_scratch(double **out) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= NA_MAXDEV) return fail(LARE_E_ARG, "energy_account_noalloc: device %d above %d", dev, NA_MAXDEV);
  if (!g_na_ptr[dev]) {
    void *p = nullptr;
    HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_na_ptr[dev] = (double *)p;
  }
  *out = g_na_ptr[dev];
  return 0;
}

int api_energy_account_noalloc(const lare_grid *grid, const lare_fields *f, double en[3], double *divb) {
  // every argument and size is checked before the first HIP call
  if (!grid || !f || !en) return fail(LARE_E_ARG, "energy_account_noalloc: NULL argument");
  if (!f->rho || !f->energy || !f->vx || !f->vy || !f->vz || !f->bx || !f->by || !f->bz)
    return fail(LARE_E_ARG, "energy_account_noalloc: missing field pointer");
  if (!grid->dxb || !grid->dyb || !grid->dzb) return fail(LARE_E_ARG, "energy_account_noalloc: metric arrays missing");
  const int n[3] = {grid->nx, grid->ny, grid->nz};
  for (int a = 0; a < 3; ++a)
    if (n[a] < 4 || n[a] > NA_NMAX)
      return fail(LARE_E_ARG, "energy_account_noalloc: grid size %d on axis %d outside 4..%d", n[a], a, NA_NMAX);
  const long nodes = (long)(n[0] + 5) * (n[1] + 5) * (n[2] + 5);
  if (nodes > 2147483647L) return fail(LARE_E_ARG, "energy_account_noalloc: grid too large for 32-bit indexing");
  fp64::Box b = fp64::mkbox(0, n[0], 0, n[1], 0, n[2]);
  const unsigned tiles = fp64::plane_blocks(b);
  const long nb = (long)tiles * (n[2] + 1);
  if (nb > NA_MAX_BLOCKS)
    return fail(LARE_E_ARG,
                "energy_account_noalloc: %ld reduction blocks exceed the scratch maximum of %d "
                "(about (n+1)^3 <= 6.7e7 nodes)", nb, NA_MAX_BLOCKS);

  double *sp = nullptr;
  int rc = na_scratch(&sp);
  if (rc) return rc;
  double *met = sp, *partial = sp + NA_MET, *level1 = partial + NA_PART, *out = level1 + NA_LEVEL1;
  // dxb(-1:n+2) of each axis to met[a * NA_LEN + (i + 2)]
  const double *src[3] = {grid->dxb, grid->dyb, grid->dzb};
  const int total = n[0] + n[1] + n[2] + 12;
  if (total <= NA_ARGS * NA_ARG_LAUNCHES) {
    NaMetrics m;
    m.first = m.count = 0;
    for (int a = 0; a < 3; ++a) m.len[a] = n[a] + 4;
    for (int e = 0, a = 0, i = 0; e < total; ++e) {
      m.v[m.count++] = src[a][i++];
      if (i == m.len[a]) {
        ++a;
        i = 0;
      }
      if (m.count == NA_ARGS || e + 1 == total) {
        hipLaunchKernelGGL(k_na_metrics, dim3(1), dim3(NA_ARGS), 0, 0, m, met);
        HIPCHK(hipGetLastError());
        m.first = e + 1;
        m.count = 0;
      }
    }
  } else {
    for (int a = 0; a < 3; ++a)
      HIPCHK(hipMemcpy(met + (size_t)a * NA_LEN + 1, src[a], sizeof(double) * (n[a] + 4), hipMemcpyHostToDevice));
  }
  fp64::Geo g = {};
  g.nx = n[0];
  g.ny = n[1];
  g.nz = n[2];
  g.dxb = met + 2;
  g.dyb = met + NA_LEN + 2;
  g.dzb = met + 2 * NA_LEN + 2;
  const fp64::FtnLayout lay = {n[0], n[1], n[2]};
  b.zc = fp64::march_chunk(tiles, n[2] + 1);
  const dim3 gr(tiles, 1, (unsigned)((n[2] + b.zc) / b.zc));
  hipLaunchKernelGGL((fp64::k_energy<fp64::FtnLayout, double>), gr, fp64::box_block(), 0, 0, g, b, lay, f->rho, f->energy,
                     f->vx, f->vy, f->vz, f->bx, f->by, f->bz, partial);
  HIPCHK(hipGetLastError());
  // the fold of fp64::final_reduce, on the scratch array
  const int nbi = (int)(gr.x * gr.z), nv = 4, minmask = 8;
  int rows;
  const int chunk = fp64::fold_chunk(nbi, &rows);
  if (chunk) {
    hipLaunchKernelGGL(fp64::k_reduce_rows, dim3(rows), dim3(256), 0, 0, partial, nbi, nv, minmask, chunk, level1);
    HIPCHK(hipGetLastError());
  }
  hipLaunchKernelGGL(fp64::k_final_reduce, dim3(1), dim3(256), 0, 0, chunk ? level1 : partial, rows, nv, minmask, 0, out,
                     fp64::HostOut{});
  HIPCHK(hipGetLastError());
  double v[4];
  HIPCHK(hipMemcpy(v, out, sizeof(v), hipMemcpyDeviceToHost));
  en[0] = v[0];
  en[1] = v[1];
  en[2] = v[2];
  if (divb) *divb = -v[3];
  return 0;
}

}  // namespace
