// bc.hpp -- boundary / halo fill on one GPU.
//
// Single-rank semantics of boundary.f90 + mpiboundary.f90: on a periodic
// axis every MPI_SENDRECV is a self-exchange of 2- or 3-layer slabs that
// span the full extent of the other two axes (so corners wrap); on a
// BC_USER axis the MPI exchange is a no-op and the user mirrors / zero
// walls of boundary.f90 apply.  The reference runs all exchanges (x, y, z)
// before all user fills (x, y, z).  A BC_OPEN side (openboundary.f90) gets
// no fill at all: the MPI exchange is a no-op there and the user fills of
// boundary.f90 apply to BC_USER sides only, so the ghosts keep the far-field
// values until open_bcs sets the first layer.
//
// All axes of all fields of a call are filled in one launch (k_halo).  Each
// of the reference's passes copies whole layers, over the full extent of
// the other two axes, so the value left at a point after the sequence is the
// old value at (mx(i), my(j), mz(k)), where m of an axis maps a filled layer
// to its source layer and every other index to itself -- whatever the order
// of the passes; and it is zero if any wall that zeroes its layers covers
// the point.  A source layer is never filled itself, so a point that is read
// is never written and the launch needs no order among its threads.
//
// Why one launch: it is bound by launch and load latency on small grids and
// by the 8-byte stores at both ends of every row on large ones.  A pass per
// axis (and per sweep one for dm) took 24 launches of about 6.5 us, 164 us
// of a 16^3 step's 540; the 6 here take 26 us.  At 256^3 the fills of a step
// went from 0.72 to 0.51 ms.

// Layers that a fill may write on one axis: -2, -1, 0, n, n+1, n+2.
#define HALO_LAYERS 6
__device__ __forceinline__ int halo_layer(int q, int n) { return q < 3 ? q - 2 : n + q - 3; }

// Source of index c on an axis of n cells for the three staggerings along
// that axis: cell centres, faces (the normal axis of a face field), nodes.
// nodez: the wall zeroes the node layer instead (boundary.f90:260-292).
struct HaloMap {
  int cell, face, node;
  bool nodez;
};
__device__ __forceinline__ HaloMap halo_map(int c, int n, int periodic, int open_lo, int open_hi) {
  HaloMap m = {c, c, c, false};
  if (c > 0 && c < n) return m;
  if (periodic) {
    // cells: (n+1:n+2) <- (1:2), (-1:0) <- (n-1:n)   cell_xface
    // faces: the same and -2 <- n-2                  bx_xface / bx_xface1
    // nodes: (n:n+2) <- (0:2), (-2:-1) <- (n-2:n-1)  node_xface1 / node_xface
    if (c <= 0) {
      if (c >= -1) m.cell = c + n;
      m.face = c + n;
      if (c < 0) m.node = c + n;
    } else {
      if (c > n) m.cell = m.face = c - n;
      m.node = c - n;
    }
    return m;
  }
  if (c <= 0 ? open_lo : open_hi) return m;
  // walls: cells 0 <- 1, -1 <- 2, n+1 <- n, n+2 <- n-1 (boundary.f90:134-160);
  // faces -1 <- 1, -2 <- 2, n+1 <- n-1, n+2 <- n-2 (:68-69, :77-78)
  m.nodez = true;
  if (c <= 0) {
    if (c >= -1) m.cell = 1 - c;
    if (c < 0) m.face = -c;
  } else if (c > n) {
    m.cell = 2 * n + 1 - c;
    m.face = 2 * n - c;
  }
  return m;
}

// Fields of one fill: the face field (NB = 1: b[0..2]), NC cell fields and
// NN node fields (0, 3 or 6).
struct HaloSet {
  double *b[3];
  real *cell[2];
  real *node[6];
};

// One thread per point of the shell: the z layers over the whole (x, y)
// extent, the y layers over k = 1..n-1, the x layers over j, k = 1..n-1.  All
// loads of a point are issued before its stores.  One block more folds the
// heating total of the kernel before the fill, if there is one to fold.
template <int NB, int NC, int NN>
__global__ __launch_bounds__(256) void k_halo(Geo g, HaloSet s, FoldJob job) {
  if (job.rows && blockIdx.x + 1 == gridDim.x) {
    fold_rows(job.rows, 0, job.nrows, 1, 0, job.out, 1, job.host);
    return;
  }
  const unsigned t = blockIdx.x * 256u + threadIdx.x;
  const unsigned wx = (unsigned)g.nx + 5u, wy = (unsigned)g.ny + 5u;
  const unsigned my = (unsigned)g.ny - 1u, mz = (unsigned)g.nz - 1u;
  const unsigned nzl = HALO_LAYERS * wx * wy, nyl = HALO_LAYERS * wx * mz, nxl = HALO_LAYERS * my * mz;
  int i, j, k;
  if (t < nzl) {
    const unsigned r = t / wx, l = r / wy;
    i = (int)(t - r * wx) - 2;
    j = (int)(r - l * wy) - 2;
    k = halo_layer((int)l, g.nz);
  } else if (t < nzl + nyl) {
    const unsigned u = t - nzl, r = u / wx, l = r / mz;
    i = (int)(u - r * wx) - 2;
    j = halo_layer((int)l, g.ny);
    k = (int)(r - l * mz) + 1;
  } else if (t < nzl + nyl + nxl) {
    const unsigned u = t - nzl - nyl, r = u / HALO_LAYERS, q = r / my;
    i = halo_layer((int)(u - r * HALO_LAYERS), g.nx);
    j = (int)(r - q * my) + 1;
    k = (int)q + 1;
  } else {
    return;
  }
  const HaloMap mx = halo_map(i, g.nx, g.per[0], g.open_lo[0], g.open_hi[0]);
  const HaloMap my_ = halo_map(j, g.ny, g.per[1], g.open_lo[1], g.open_hi[1]);
  const HaloMap mz_ = halo_map(k, g.nz, g.per[2], g.open_lo[2], g.open_hi[2]);
  const int c = g.idx(i, j, k);
  const bool z = mx.nodez || my_.nodez || mz_.nodez;
  const int sx = g.idx(mx.face, my_.cell, mz_.cell), sy = g.idx(mx.cell, my_.face, mz_.cell),
            sz = g.idx(mx.cell, my_.cell, mz_.face), sc = g.idx(mx.cell, my_.cell, mz_.cell),
            sn = g.idx(mx.node, my_.node, mz_.node);
  double vb[3] = {0.0, 0.0, 0.0};
  real vc[2] = {0, 0}, vn[6] = {0, 0, 0, 0, 0, 0};
  if constexpr (NB) {
    vb[0] = s.b[0][sx];
    vb[1] = s.b[1][sy];
    vb[2] = s.b[2][sz];
  }
#pragma unroll
  for (int q = 0; q < NC; ++q) vc[q] = s.cell[q][sc];
#pragma unroll
  for (int q = 0; q < NN; ++q) vn[q] = s.node[q][sn];
  if constexpr (NB) {
    if (sx != c) s.b[0][c] = vb[0];
    if (sy != c) s.b[1][c] = vb[1];
    if (sz != c) s.b[2][c] = vb[2];
  }
  if (NC > 0 && sc != c)
#pragma unroll
    for (int q = 0; q < NC; ++q) s.cell[q][c] = vc[q];
  if (NN > 0 && (z || sn != c))
#pragma unroll
    for (int q = 0; q < NN; ++q) s.node[q][c] = z ? (real)0 : vn[q];
}
static inline unsigned halo_blocks(const Geo &g) {
  const long wx = g.nx + 5, wy = g.ny + 5, my = g.ny - 1, mz = g.nz - 1;
  return (unsigned)((HALO_LAYERS * (wx * wy + wx * mz + my * mz) + 255) / 256);
}

// Line fills of the potential phi (phi_mpi, initial_conditions.f90:268-291),
// whose walls copy the first interior layer into both ghost layers.
enum BcOp {
  BC_PER_CELL,   // (n+1:n+2) <- (1:2), (-1:0) <- (n-1:n)
  BC_PHI_NEU     // 0 <- 1, -1 <- 1, n+1 <- n, n+2 <- n
};
__global__ __launch_bounds__(64) void k_bc_axis(Geo g, double *__restrict__ a, int op, int axis) {
  // plane coordinates: u runs along the contiguous axis where possible
  const int u = axis == 0 ? 1 : 0;
  const int w = axis == 2 ? 1 : 2;
  const int iu = -2 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int iw = -2 + (int)blockIdx.y;
  if (iu > g.n(u) + 2) return;
  const int n = g.n(axis);
  const int st = g.stride(axis);
  int c[3];
  c[axis] = 0;
  c[u] = iu;
  c[w] = iw;
  const int base = g.idx(c[0], c[1], c[2]);  // index of layer 0 on this line
  const bool per = op == BC_PER_CELL;
  const double l1 = a[base + (per ? n : 1) * st], l2 = a[base + (per ? n - 1 : 1) * st];
  const double h1 = a[base + (per ? 1 : n) * st], h2 = a[base + (per ? 2 : n) * st];
  a[base] = l1;
  a[base - st] = l2;
  a[base + (n + 1) * st] = h1;
  a[base + (n + 2) * st] = h2;
}
