// common.hpp -- device layout and launch helpers shared by all kernels.
//
// Every 3-D field lives in one padded box covering Fortran indices
// -2..n+2 on each axis (the union of the cell, node and face bounds of
// mpi_routines.F90:295-334), x fastest.  Index (i, j, k) maps to
//     (k + 2) * sz + (j + 2) * sy + (i + OX)
// with OX = 16 so that i = 0 sits on a 128-byte boundary for FP64 rows and
// the row pitch sy is a multiple of 16 elements.  All fields share the
// same index arithmetic, which lets one kernel address cell, node and face
// arrays with one offset.


#define OX 16

struct Geo {
  int nx, ny, nz;
  int sy, sz;
  // 1-D metrics, indexable by Fortran index (pointer already offset)
  const double *dxb, *dxc, *dyb, *dyc, *dzb, *dzc, *grav;
  int per[3];     // axis periodic (both sides)
  int user[3];    // axis not periodic (each side BC_USER or BC_OPEN)
  int open_lo[3], open_hi[3];  // that side BC_OPEN: no fill, ghosts as stored
  __host__ __device__ __forceinline__ int idx(int i, int j, int k) const {
    return (k + 2) * sz + (j + 2) * sy + (i + OX);
  }
  __host__ __device__ __forceinline__ int n(int a) const { return a == 0 ? nx : (a == 1 ? ny : nz); }
  __host__ __device__ __forceinline__ int stride(int a) const { return a == 0 ? 1 : (a == 1 ? sy : sz); }
  __device__ __forceinline__ double db(int a, int i) const { return a == 0 ? dxb[i] : (a == 1 ? dyb[i] : dzb[i]); }
  __device__ __forceinline__ double dc(int a, int i) const { return a == 0 ? dxc[i] : (a == 1 ? dyc[i] : dzc[i]); }
  // cell volume of setup.F90:242-246, recomputed from the metrics
  __device__ __forceinline__ double cv(int i, int j, int k) const { return dxb[i] * dyb[j] * dzb[k]; }
};

// Index box [lo, hi] inclusive per axis; zc: points per block along the march
// axis of a marching launch (1 .. ZCHUNK, march_chunk).
struct Box {
  int x0, x1, y0, y1, z0, z1;
  int zc;
};

#define BX 64
#define BY 4

// The block and thread coordinates as parameters of a kernel's body that two
// kernels share: they take the place of the built-in variables, so that the
// index macros below read them.
#define BLOCK_COORDS const dim3 blockIdx, const dim3 gridDim, const dim3 threadIdx

// In-plane position (i, j) of a thread of a box launch.  The (x, y) extent
// of the box is walked as one flattened index, BX*BY consecutive points per
// block, so a box a few points wider than a multiple of 64 (n+1 .. n+4 for
// n = 256) does not launch a column of blocks whose waves are almost empty.
// i always lies inside [x0, x1]; j may pass y1 in the last block.
//
// Blocks are dispatched to the eight XCDs round-robin by linear block id,
// and each XCD has its own L2.  Tile t of a plane goes to block
// xcd_tile(t): the tiles that share an XCD (block ids congruent mod 8) get
// consecutive plane positions, so the rows a tile's stencil reads from its
// neighbour tiles are mostly in the same L2.
__device__ __forceinline__ unsigned xcd_tile(unsigned bx, unsigned gx) {
  const unsigned q = gx >> 3, r = gx & 7u, t = bx & 7u;
  return t * q + (t < r ? t : r) + (bx >> 3);
}
#define PLANE_POS(b, i, j)                                                                  \
  const unsigned pw_ = (unsigned)((b).x1 - (b).x0 + 1);                                     \
  const unsigned pp_ = xcd_tile(blockIdx.x, gridDim.x) * (unsigned)(BX * BY) + threadIdx.y * (unsigned)BX + threadIdx.x; \
  const unsigned pj_ = pp_ / pw_;                                                           \
  const int i = (b).x0 + (int)(pp_ - pj_ * pw_);                                            \
  const int j = (b).y0 + (int)pj_;

// Thread (i, j, k) of a box launch; returns false outside the box.
#define BOX_INDEX(b, i, j, k)                  \
  PLANE_POS(b, i, j)                           \
  const int k = (b).z0 + (int)blockIdx.z;      \
  if (j > (b).y1 || k > (b).z1) return;

static inline unsigned plane_blocks(const Box &b) {
  const long w = b.x1 - b.x0 + 1, h = b.y1 - b.y0 + 1;
  return (unsigned)((w * h + BX * BY - 1) / (BX * BY));
}
static inline dim3 box_grid(const Box &b) { return dim3(plane_blocks(b), 1, (unsigned)(b.z1 - b.z0 + 1)); }
static inline dim3 box_block() { return dim3(BX, BY, 1); }
#define ZCHUNK 8  // most points a block marches over
static inline Box mkbox(int x0, int x1, int y0, int y1, int z0, int z1) {
  Box b = {x0, x1, y0, y1, z0, z1, ZCHUNK};
  return b;
}

// Points a block marches over, for a launch of per_plane blocks on each of
// `points` march positions.  A block of c points costs about c + 1 (the plane
// before them), and a launch takes as many turns as the fullest of the 256 CUs
// has blocks; below three blocks per CU a turn is bound by the serial chain of
// loads of the march and a fuller CU takes no longer.  So: the c with the
// least max(3, blocks per CU, rounded up) * (c + 1), the longer of two alike.
// With chunks of 8 a marching kernel took 14 to 25 us at 16^3 and at 64^3
// alike, and takes 4 to 6 and 7 to 10.  Against the longest of 8, 4, 2, 1 that
// launches 512 blocks, which left 544 blocks of 4 planes to 64 x 64 x 128
// (three on some CUs, two on most): 20 conduction super-steps there 9.9 -> 9.5
// ms, 50 steps with conduction in FP32 28.5 -> 27.6, 50 steps at 97 x 61 x 130
// 38.4 -> 37.7; 16^3, 64^3 and 192^3 and above unchanged.
#define MARCH_CUS 256
#define MARCH_TURNS 3
static inline int march_chunk(unsigned per_plane, int points) {
  int best = 1;
  long least = 0;
  for (int c = 1; c <= ZCHUNK; ++c) {
    long turns = ((long)per_plane * ((points + c - 1) / c) + MARCH_CUS - 1) / MARCH_CUS;
    if (turns < MARCH_TURNS) turns = MARCH_TURNS;
    const long cost = turns * (c + 1);
    if (c == 1 || cost <= least) {
      least = cost;
      best = c;
    }
  }
  return best;
}

__device__ __forceinline__ double dmin(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ double dmax(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ float dmin(float a, float b) { return a < b ? a : b; }
__device__ __forceinline__ float dmax(float a, float b) { return a > b ? a : b; }

// Fortran MAX(x, 0.0_num) as used on energy and visc_heat.
__device__ __forceinline__ double max0(double x) { return x > 0.0 ? x : 0.0; }
__device__ __forceinline__ float max0(float x) { return x > 0.0f ? x : 0.0f; }

// Division by a divisor that serves several numerators, or whose reciprocal is
// known before the numerator: the reciprocal is refined once (Newton steps
// with fused remainders) and each quotient is corrected by its exact
// remainder (Markstein 1990).  The steps are those of the compiler's
// correctly rounded division for gfx950 less its scaling of operands near
// the ends of the exponent range and its fix-up of zeros, infinities and NaN,
// so the bits are those of a / b while |a|, |b| and |a / b| lie within about
// 1e+-290 (FP64) or 1e+-29 (FP32); outside, the last bit may differ, a
// divisor beyond the range of its reciprocal (below 1e-308 or above 1e308;
// 1e-38 and 1e38) gives no quotient, a zero loses its sign, and what would be
// infinite is NaN.  So it divides only where an infinity and a NaN end alike, in
// a value that the state check of the next step finds: where a minimum, a
// MAX(., 0) or a comparison would drop a NaN, the division is the plain one or
// goes through over() or over_all().  A quotient is 3 (FP32: 5) operations on its
// critical path instead of 11, and 4 or 5 by these.  over_all() everywhere took
// 100 steps at 192^3 in FP32 337 -> 350 ms, 256^3 in FP64 996 -> 1009, 20
// conduction super-steps at 64 x 64 x 128 9.5 -> 10.0.
template <class A>
struct Recip {
  A d, y;
};
__device__ __forceinline__ Recip<double> recip(double d) {
  double y = __builtin_amdgcn_rcp(d);
  y = fma(y, fma(-d, y, 1.0), y);
  y = fma(y, fma(-d, y, 1.0), y);
  return Recip<double>{d, y};
}
__device__ __forceinline__ Recip<float> recip(float d) {
  float y = __builtin_amdgcn_rcpf(d);
  y = fmaf(fmaf(-d, y, 1.0f), y, y);
  return Recip<float>{d, y};
}
__device__ __forceinline__ double operator/(double a, const Recip<double> &b) {
  const double q = a * b.y;
  return fma(fma(-b.d, q, a), b.y, q);
}
__device__ __forceinline__ float operator/(float a, const Recip<float> &b) {
  float q = a * b.y;
  q = fmaf(fmaf(-b.d, q, a), b.y, q);
  return fmaf(fmaf(-b.d, q, a), b.y, q);
}
// The same quotient with the zero, infinite and NaN operands of a / b as well, by
// the hardware's fix-up, which also sets the sign.
__device__ __forceinline__ double over(double a, const Recip<double> &b) {
  return __builtin_amdgcn_div_fixup(a / b, b.d, a);
}
__device__ __forceinline__ float over(float a, const Recip<float> &b) {
  return __builtin_amdgcn_div_fixupf(a / b, b.d, a);
}
// And with the infinity of a quotient beyond the range: the maximum takes the
// NaN for one, whose sign the fix-up sets.
__device__ __forceinline__ double over_all(double a, const Recip<double> &b) {
  return __builtin_amdgcn_div_fixup(__builtin_fmax(a / b, -__builtin_inf()), b.d, a);
}
__device__ __forceinline__ float over_all(float a, const Recip<float> &b) {
  return __builtin_amdgcn_div_fixupf(__builtin_fmaxf(a / b, -__builtin_inff()), b.d, a);
}
// Square root of a positive normal number: the steps of the compiler's
// correctly rounded root (Goldschmidt's iteration with fused remainders) less
// its scaling and its cases for zero and infinity.
__device__ __forceinline__ double sqrt_pos(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  h = fma(h, r, h);
  g = fma(g, r, g);
  g = fma(fma(-g, g, x), h, g);
  return fma(fma(-g, g, x), h, g);
}
// sqrt(x): the short form in its range, the library's elsewhere (zero too)
__device__ __forceinline__ double root(double x) {
  return __builtin_expect(x > 1.0e-280 && x < 1.0e280, 1) ? sqrt_pos(x) : sqrt(x);
}
__device__ __forceinline__ float root(float x) { return sqrtf(x); }
// the same divisor for FP64 numerators
__device__ __forceinline__ const Recip<double> &wide(const Recip<double> &r) { return r; }
__device__ __forceinline__ Recip<double> wide(const Recip<float> &r) { return recip((double)r.d); }
// the value of the lane above (lane + 1)
template <class A>
__device__ __forceinline__ Recip<A> lane_next(const Recip<A> &r) {
  return Recip<A>{__shfl_down(r.d, 1, 64), __shfl_down(r.y, 1, 64)};
}
template <class A>
__device__ __forceinline__ Recip<A> select(bool c, const Recip<A> &a, const Recip<A> &b) {
  return Recip<A>{c ? a.d : b.d, c ? a.y : b.y};
}

// Wavefront (64-lane) reductions.
__device__ __forceinline__ double wave_min(double v) {
  for (int off = 32; off > 0; off >>= 1) v = dmin(v, __shfl_down(v, off, 64));
  return v;
}
__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// Block-level reduction of NV values into partial[blockid * NV + q].
// op 0 = min, 1 = sum.  Block size BX*BY = 256 (4 waves).
template <int NV>
__device__ __forceinline__ void block_reduce_store(double (&v)[NV], const int *ops, double *partial) {
  __shared__ double red[4][NV];
  const int lane = threadIdx.x & 63;
  const int wave = (threadIdx.y * BX + threadIdx.x) >> 6;
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = ops[q] == 0 ? wave_min(v[q]) : wave_sum(v[q]);
  if (lane == 0)
#pragma unroll
    for (int q = 0; q < NV; ++q) red[wave][q] = v[q];
  __syncthreads();
  if (threadIdx.x == 0 && threadIdx.y == 0) {
    const int bid = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      double r = red[0][q];
      for (int w = 1; w < 4; ++w) r = ops[q] == 0 ? dmin(r, red[w][q]) : r + red[w][q];
      partial[(size_t)bid * NV + q] = r;
    }
  }
}

// One block of 256 threads folds rows r0 .. r1-1 of nv values (bit q of
// minmask selects min, else sum) and stores (or adds) the nv results, in out
// and, if given, in the pinned host mirror, whose ticket word it then sets.
#define RED_MAXV 4
struct HostOut {
  double *v;
  unsigned long long *ticket, number;
};
__device__ __forceinline__ void fold_rows(const double *__restrict__ rows, int r0, int r1, int nv, int minmask,
                                          double *__restrict__ out, int accumulate, const HostOut &host = HostOut{}) {
  __shared__ double red[4][RED_MAXV];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int q = 0; q < nv; ++q) {
    const bool isMin = (minmask >> q) & 1;
    double v = isMin ? 1.7976931348623157e+308 : 0.0;
    for (int r = r0 + (int)threadIdx.x; r < r1; r += 256) {
      const double x = rows[(size_t)r * nv + q];
      v = isMin ? dmin(v, x) : v + x;
    }
    v = isMin ? wave_min(v) : wave_sum(v);
    if (lane == 0) red[wave][q] = v;
  }
  __syncthreads();
  if ((int)threadIdx.x < nv) {
    const int q = threadIdx.x;
    const bool isMin = (minmask >> q) & 1;
    double r = red[0][q];
    for (int w = 1; w < 4; ++w) r = isMin ? dmin(r, red[w][q]) : r + red[w][q];
    if (accumulate) r = out[q] + r;
    out[q] = r;
    if (host.v) {
      ((volatile double *)host.v)[q] = r;
      __threadfence_system();
    }
  }
  if (host.v) {
    // the values (one wave's stores) reach the host before the ticket
    __syncthreads();
    if (threadIdx.x == 0) *(volatile unsigned long long *)host.ticket = host.number;
  }
}

// A sum of one value per row that a launch folds beside its own work, in a
// block of its own (rows NULL: none).
struct FoldJob {
  const double *rows;
  int nrows;
  double *out;
  HostOut host;
};

// Columns of a z-marching launch: thread (i, j) of the flattened plane tile
// blockIdx.x walks planes k0 .. k1 of its chunk (b.zc planes per block).
#define ZRANGE(b, k0, k1)                                             \
  const int k0 = (b).z0 + (int)blockIdx.z * (b).zc;                    \
  const int k1 = k0 + (b).zc - 1 < (b).z1 ? k0 + (b).zc - 1 : (b).z1;
#define ZCOLUMN(b, i, j, k0, k1) \
  PLANE_POS(b, i, j)             \
  ZRANGE(b, k0, k1)              \
  if (j > (b).y1) return;

// Columns of a launch that marches along axis M (1 = y, 2 = z) for b.zc
// points: the flattened tile covers x and the other transverse axis, whose
// index is p; MJ/MK give j and k at march coordinate m.  The grid is the
// zchunk grid of the box with its y and z ranges swapped when M = 1.
#define MCOLUMN(M, b, i, p, m0, m1)                                                         \
  const Box pb_ = (M) == 2 ? (b) : Box{(b).x0, (b).x1, (b).z0, (b).z1, (b).y0, (b).y1, (b).zc};   \
  PLANE_POS(pb_, i, p)                                                                     \
  ZRANGE(pb_, m0, m1)                                                                      \
  if (p > pb_.y1) return;
#define MJ(M, m, p) ((M) == 1 ? (m) : (p))
#define MK(M, m, p) ((M) == 2 ? (m) : (p))

// A field at the four in-plane points (i, j), (i-1, j), (i, j-1), (i-1, j-1).
struct Quad {
  real p0, px, py, pxy;
};
__device__ __forceinline__ Quad quad_back(const real *__restrict__ u, int c, int Y) {
  Quad q = {u[c], u[c - 1], u[c - Y], u[c - 1 - Y]};
  return q;
}

// A field at the four in-plane points (i, j), (i+1, j), (i, j+1), (i+1, j+1).
__device__ __forceinline__ Quad quad_fwd(const real *__restrict__ u, int c, int Y) {
  Quad q = {u[c], u[c + 1], u[c + Y], u[c + 1 + Y]};
  return q;
}
