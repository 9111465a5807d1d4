// fdfd_nd.h -- nested-dissection (multifrontal) direct solver of the whole
// periodic operator, included by fdfd_hip.hip after its tile helpers.
//
// The block sweep of fdfd_hip.hip is serial in the long axis: m n/32 dependent
// pivot steps to factor, m dependent blocks per sweep, 8 m n^3 flops. Here the
// cells are ordered by nested dissection on a regular tree: about 5n/32
// dependent pivot steps on an n x n grid, one launch per direction of a sweep
// for the lower levels and one per level above, and O(n^3) flops. 512^2
// complex64: factor 65.7 -> 1.87 ms, a sweep 2.1 -> 0.33 ms; 768^2 FP64: 222 ->
// 6.0 ms. The block path keeps what asks for it by kind (pivoted, stepwise and
// batched factors), the grids with a side under ND_MIN_SIDE cells, complex64
// under ND_MIN_SIDE_C64, and very long ones (nd_long).
//
// Tree. Cell column 0 and cell row 0 (the cross) are the root separator, so
// what is left, cells 1..nx-1 x 1..ny-1, is not periodic. A box is split by
// its middle column or row (across its longer side) until it has at most
// ND_LEAF cells. All boxes of one depth come from halving both axes the same
// number of times, so their sides differ by at most one and every index
// below is computed, not stored. The separator of a box and the ring of cells
// around it (its border) form its front; the five-point stencil needs no
// corners. At the top the two ends of an axis that has not been cut are the
// same cells (the cross), and the border holds them once.
//
// Elimination. With E = diag(sqrt(sxf_i syf_j)) the matrix M = a E A E^-1 is
// complex symmetric (a: a power of two that brings its entries near one).
// For a box with front [[F_ss, F_sb], [F_sb^T, F_bb]] summed from its two
// children's updates and its separator's own entries:
//   X = F_ss^-1,  W = X F_sb,  C = F_bb - F_sb^T X F_sb  (to the parent).
// X comes from tiled Gauss-Jordan steps on the upper tiles of [F_ss | F_sb]
// (k_nd_step); C from the panels that these leave, one MFMA product per level.
//
// Solve. Upwards f_s = r_s + (children), z = X f_s, u = (children) - W^T f_s;
// downwards x_s = z - W x_b. Everything is gathered by the reader in a fixed
// order: no atomics, the same bits on every run.

constexpr int ND_LEAF = 32;        // most cells of a leaf box: one pivot tile
constexpr int ND_MIN_SIDE = 16;    // shorter grid side of a tree (measured: nd_fits)
constexpr int ND_MAX_LEVELS = 40;
constexpr size_t ND_HEADER = 256;  // the tag, at the start of the factor
__host__ __device__ inline unsigned long long nd_tag(int i) {
  return 0x6664666400000000ull + 0x9e3779b97f4a7c15ull * (unsigned long long)(i + 1);
}

// Segment idx of the interior 1..N-1 of an axis of N cells halved d times:
// [a, a + len); the middle cell of a segment separates its halves.
__host__ __device__ inline void nd_seg(int N, int d, int idx, int &a, int &len) {
  a = 1;
  len = N - 1;
  for (int t = d - 1; t >= 0; --t) {
    const int l = (len - 1) >> 1;
    if ((idx >> t) & 1) { a += l + 1; len -= l + 1; }
    else len = l;
  }
}
inline int nd_longest(int N, int d) {
  int len = N - 1;
  for (int t = 0; t < d; ++t) len -= 1 + ((len - 1) >> 1);
  return len;
}

// One merge level: boxes of depth (dx, dy), split along axis ax (0: by a
// column, into halves of depth dx + 1). s, b: the largest separator and
// border; sp, bp: padded to tiles; cbp: the children's bp.
struct NdLevel {
  int nx, ny, dx, dy, ax, root;
  int s, b, sp, bp, nbox;
  int cb, cbp;         // the children's b and bp
  size_t xoff, woff;   // X [nbox][2][sp][sp] and W [nbox][2][sp][bp] in the factor's data (elements)
};
struct NdPlan {
  int nx, ny, nlev, Dx, Dy, nleaf, leaf_b, leaf_bp;
  NdLevel lev[ND_MAX_LEVELS];   // from the leaves' parents to the top box, then the root (lev[nlev])
  size_t leaf_off, leafc_off, elems;
};

// false: the grid is outside the path's range
bool nd_plan(const fdfd_grid *g, NdPlan *P) {
  memset(P, 0, sizeof *P);
  const int nx = g->nx, ny = g->ny;
  if (std::min(nx, ny) < ND_MIN_SIDE || (long)nx * ny > (1l << 30)) return false;
  P->nx = nx;
  P->ny = ny;
  NdLevel down[ND_MAX_LEVELS];
  int dx = 0, dy = 0, n = 0;
  for (;;) {
    const int w = nd_longest(nx, dx), h = nd_longest(ny, dy);
    if (w * (long)h <= ND_LEAF) break;
    if (n >= ND_MAX_LEVELS - 1) return false;
    NdLevel &L = down[n++];
    memset(&L, 0, sizeof L);
    L.nx = nx; L.ny = ny; L.dx = dx; L.dy = dy;
    L.ax = w >= h ? 0 : 1;
    L.s = L.ax == 0 ? h : w;
    L.b = (dx ? 2 : 1) * h + (dy ? 2 : 1) * w;
    L.sp = pad_n(L.s);
    L.bp = pad_n(L.b);
    L.nbox = 1 << (dx + dy);
    if (L.ax == 0) ++dx;
    else ++dy;
  }
  if (!dx || !dy || dx + dy > 26) return false;
  P->Dx = dx;
  P->Dy = dy;
  P->nleaf = 1 << (dx + dy);
  P->leaf_b = 2 * (nd_longest(nx, dx) + nd_longest(ny, dy));
  P->leaf_bp = TB;
  if (P->leaf_b > TB) return false;
  P->nlev = n;
  // leaves: X [nleaf][2][TB][TB], then the border couplings [nleaf][TB] complex
  size_t off = 0;
  P->leaf_off = off;  off += (size_t)P->nleaf * 2 * TB * TB;
  P->leafc_off = off; off += (size_t)P->nleaf * TB * 2;
  for (int i = 0; i < n; ++i) {
    NdLevel &L = P->lev[i] = down[n - 1 - i];
    L.cb = i == 0 ? P->leaf_b : P->lev[i - 1].b;
    L.cbp = i == 0 ? P->leaf_bp : P->lev[i - 1].bp;
    L.xoff = off; off += (size_t)L.nbox * 2 * L.sp * L.sp;
    L.woff = off; off += (size_t)L.nbox * 2 * L.sp * L.bp;
  }
  NdLevel &R = P->lev[n];
  R.nx = nx; R.ny = ny; R.root = 1; R.nbox = 1;
  R.s = nx + ny - 1;
  R.sp = pad_n(R.s);
  R.cb = P->lev[n - 1].b;
  R.cbp = P->lev[n - 1].bp;
  R.xoff = R.woff = off;
  off += 2 * (size_t)R.sp * R.sp;
  P->elems = off;
  return true;
}

// Factor buffer: the tag, the tables E_x, 1/E_x [nx], E_y, 1/E_y [ny]
// (complex FP64), then the data of the plan.
inline size_t nd_data_off(const NdPlan &P) { return ND_HEADER + align_up(32 * (size_t)(P.nx + P.ny), 256); }
// Never the size of a block factor of the grid: a buffer's size names its kind.
inline size_t nd_factor_bytes(const fdfd_grid *g, const NdPlan &P, int precision) {
  const size_t n = nd_data_off(P) + align_up(P.elems * elem_size(precision), 256);
  return n == factor_total_bytes(g, base_prec(precision)) ? n + 256 : n;
}
// Which levels k_nd_merge takes: one tile of separator, a border of at most
// nd_merge_tiles tiles (wider ones are few boxes with more tiles than one
// workgroup should form: with 4 and 6 tiles, 256 and 128 boxes, 75 and 72 us
// there, 46 and 45 as a launch each for front, step and update; FP64 with 3
// tiles and 85 KB of LDS 311 against 293). es: bytes of a real.
constexpr int nd_merge_tiles(size_t es) { return es == 8 ? 2 : 3; }
inline bool nd_merges(const NdLevel &L, size_t es) {
  return !L.root && L.sp == TB && L.bp <= nd_merge_tiles(es) * TB;
}
// Factor workspace (after the status header): the scaled bands, the pivot
// inverses of two steps, the ping-pong pairs of [F_ss] and [F_sb], the panels
// U and R of the elimination (k_nd_step), the updates C of two levels. All but
// the bands and C belong to the levels that k_nd_merge does not take: 512^2
// complex64 195 MB instead of 283, 768^2 FP64 1027 instead of 1261.
struct NdWork {
  size_t bands, pinv[2], S[2], B[2], U, R, C[2], total;
};
NdWork nd_work_layout(const NdPlan &P, int precision) {
  const size_t es = elem_size(precision), M = (size_t)P.nx * P.ny;
  size_t boxes = 0, ss = 0, sb = 0, sb1 = 0, cc = (size_t)P.nleaf * P.leaf_bp * P.leaf_bp;
  for (int i = 0; i <= P.nlev; ++i) {
    const NdLevel &L = P.lev[i];
    cc = std::max(cc, (size_t)L.nbox * L.bp * L.bp);
    if (nd_merges(L, es)) continue;
    boxes = std::max(boxes, (size_t)L.nbox);
    if (L.sp > TB) ss = std::max(ss, (size_t)L.nbox * L.sp * L.sp);
    sb = std::max(sb, (size_t)L.nbox * L.sp * L.bp);
    if (L.sp > TB) sb1 = std::max(sb1, (size_t)L.nbox * L.sp * L.bp);
  }
  NdWork w;
  size_t off = WORK_HEADER;
  auto take = [&](size_t bytes) { const size_t at = off; off += align_up(bytes, 256); return at; };
  w.bands = take(3 * 2 * M * es);
  for (int i = 0; i < 2; ++i) w.pinv[i] = take(boxes * 2 * TB * TB * es);
  for (int i = 0; i < 2; ++i) w.S[i] = take(2 * ss * es);
  for (int i = 0; i < 2; ++i) w.B[i] = take(2 * sb1 * es);
  w.U = take(2 * sb * es);
  w.R = take(2 * sb1 * es);
  for (int i = 0; i < 2; ++i) w.C[i] = take(2 * cc * es);
  w.total = off;
  return w;
}
// Scale of M: 2^-e with the stencil's size 4 / (mu0' h^2) (Ez) or 4 /
// (eps0' h^2) (Hz) brought to [0.5, 1)
inline double nd_alpha(const fdfd_grid *g) {
  const double h = g->dl, c = 4.0 / ((g->pol == FDFD_POL_EZ ? MU_0 : EPSILON_0) * g->L0 * h * h);
  int e = 0;
  (void)frexp(c, &e);
  return ldexp(1.0, -e);
}

// -------------------------------------------------------- box geometry
struct NdBox {
  int x0, w, y0, h;   // interior
  int k0, k1;         // the children's numbers
  int c0, c1;         // the children's lengths along the split axis
  int s, b;           // separator and border
  int oB, oT;         // where the border's row sections start (L at 0, R at h)
};
__host__ __device__ inline NdBox nd_box(const NdLevel &L, int k) {
  NdBox B;
  if (L.root) {
    B.x0 = 1; B.w = L.nx - 1; B.y0 = 1; B.h = L.ny - 1;
    B.k0 = 0; B.k1 = 0; B.c0 = B.c1 = 0;
    B.s = L.s; B.b = 0; B.oB = B.oT = 0;
    return B;
  }
  const int ix = k >> L.dy, iy = k & ((1 << L.dy) - 1);
  nd_seg(L.nx, L.dx, ix, B.x0, B.w);
  nd_seg(L.ny, L.dy, iy, B.y0, B.h);
  const int len = L.ax == 0 ? B.w : B.h;
  B.c0 = (len - 1) >> 1;
  B.c1 = len - 1 - B.c0;
  if (L.ax == 0) {
    B.k0 = ((2 * ix) << L.dy) + iy;
    B.k1 = B.k0 + (1 << L.dy);
    B.s = B.h;
  } else {
    B.k0 = (ix << (L.dy + 1)) + 2 * iy;
    B.k1 = B.k0 + 1;
    B.s = B.w;
  }
  B.oB = (L.dx ? 2 : 1) * B.h;
  B.oT = B.oB + B.w;
  B.b = B.oB + (L.dy ? 2 : 1) * B.w;
  return B;
}
// cell of separator entry j
__host__ __device__ inline size_t nd_sep_cell(const NdLevel &L, const NdBox &B, int j) {
  if (L.root) {
    const int h = L.ny - 1, w = L.nx - 1;
    return j < h ? (size_t)(j + 1) : (j < h + w ? (size_t)(j - h + 1) * L.ny : (size_t)0);
  }
  return L.ax == 0 ? (size_t)(B.x0 + B.c0) * L.ny + B.y0 + j : (size_t)(B.x0 + j) * L.ny + B.y0 + B.c0;
}
// cell of border entry j of a box of depth (dx, dy)
__host__ __device__ inline size_t nd_border_cell(int nx, int ny, int dx, int dy, const NdBox &B, int j) {
  if (j < B.h) return (size_t)(B.x0 - 1) * ny + B.y0 + j;
  j -= B.h;
  if (dx) {
    if (j < B.h) return (size_t)(B.x0 + B.w == nx ? 0 : B.x0 + B.w) * ny + B.y0 + j;
    j -= B.h;
  }
  if (j < B.w) return (size_t)(B.x0 + j) * ny + B.y0 - 1;
  return (size_t)(B.x0 + j - B.w) * ny + (B.y0 + B.h == ny ? 0 : B.y0 + B.h);
}
// entry of each child's border (-1: none) for separator entry j
__host__ __device__ inline void nd_sep_map(const NdLevel &L, const NdBox &B, int j, int &m0, int &m1) {
  if (L.root) {   // the top box's border is the cross in the root's order, without the corner
    m0 = j < L.s - 1 ? j : -1;
    m1 = -1;
  } else if (L.ax == 0) {
    m0 = B.h + j;
    m1 = j;
  } else {
    const int sides = L.dx ? 2 : 1;
    m0 = sides * B.c0 + B.w + j;
    m1 = sides * B.c1 + j;
  }
}
// ... for border entry j
__host__ __device__ inline void nd_border_map(const NdLevel &L, const NdBox &B, int j, int &m0, int &m1) {
  const int h = B.h, w = B.w;
  if (L.ax == 0) {
    if (j < h) { m0 = j; m1 = L.dx ? -1 : h + j; return; }
    if (L.dx && j < 2 * h) { m0 = -1; m1 = j; return; }
    const int t = j >= B.oT ? 1 : 0, i = j - (t ? B.oT : B.oB);
    m0 = i < B.c0 ? 2 * h + (t ? B.c0 : 0) + i : -1;
    m1 = i > B.c0 ? 2 * h + (t ? B.c1 : 0) + i - B.c0 - 1 : -1;
  } else {
    if (j < B.oB) {
      const int r = j >= h ? 1 : 0, i = j - (r ? h : 0);
      m0 = i < B.c0 ? (r ? B.c0 : 0) + i : -1;
      m1 = i > B.c0 ? (r ? B.c1 : 0) + i - B.c0 - 1 : -1;
      return;
    }
    const int sides = L.dx ? 2 : 1, o0 = sides * B.c0, o1 = sides * B.c1;
    if (j < B.oT) { m0 = o0 + j - B.oB; m1 = L.dy ? -1 : o1 + w + j - B.oB; return; }
    m0 = -1;
    m1 = o1 + w + j - B.oT;
  }
}

// ------------------------------------------------------------- factor
// Scaled bands: planes [3][nx ny] of complex T, the diagonal and the
// couplings to (i+1, j) and (i, j+1).
template <typename T> struct NdBands {
  const T *c, *x, *y;
};
template <typename T>
__device__ inline void nd_ld(const T *p, size_t at, T &re, T &im) {
  typedef T t2 __attribute__((ext_vector_type(2)));
  const t2 v = *reinterpret_cast<const t2 *>(p + 2 * at);
  re = v.x;
  im = v.y;
}
template <typename T>
__device__ inline void nd_st(T *p, size_t at, T re, T im) {
  typedef T t2 __attribute__((ext_vector_type(2)));
  *reinterpret_cast<t2 *>(p + 2 * at) = t2{re, im};
}

// Square root of s = 1 - i sigma
__device__ inline cd nd_sqrt(cd s) {
  const double re = sqrt(0.5 * (sqrt(s.r * s.r + s.i * s.i) + s.r));
  return {re, s.i / (2 * re)};
}
// The factor's tag and tables; clears the status word and the bytes [gap0,
// data) and [gap1, end) between and after the factor's parts. (The padding
// rows of leaves and merged boxes hold what the buffer held: nothing reads
// them into a result.)
__global__ void __launch_bounds__(NT) k_nd_tables(fdfd_grid g, unsigned long long *head, double *tab, int *status,
                                                  size_t gap0, size_t data, size_t gap1, size_t end) {
  const int t = blockIdx.x * NT + threadIdx.x, nx = g.nx, ny = g.ny;
  if (t < (int)(ND_HEADER / 8)) head[t] = nd_tag(t);
  if (t == 0) *status = 0;
  unsigned char *bytes = reinterpret_cast<unsigned char *>(head);
  if (t < 512) {
    if (gap0 + t < data) bytes[gap0 + t] = 0;
    if (gap1 + t < end) bytes[gap1 + t] = 0;
  }
  if (t >= nx + ny) return;
  const bool xa = t < nx;
  const int i = xa ? t : t - nx, n = xa ? nx : ny;
  const double h = ((double)n * g.dl) / n;
  const cd e = nd_sqrt(sfactor(0, i, n, xa ? g.npml_x : g.npml_y, h, g.omega, g.L0));
  double *ex = tab, *iex = tab + 2 * (size_t)nx, *ey = tab + 4 * (size_t)nx, *iey = ey + 2 * (size_t)ny;
  st_c(xa ? ex : ey, i, e);
  st_c(xa ? iex : iey, i, cinv(e));
}
struct NdTab {
  const double *ex, *iex, *ey, *iey;
};
__host__ __device__ inline NdTab nd_tables(const double *tab, int nx, int ny) {
  return NdTab{tab, tab + 2 * (size_t)nx, tab + 4 * (size_t)nx, tab + 4 * (size_t)nx + 2 * (size_t)ny};
}

template <typename T>
__global__ void __launch_bounds__(NT) k_nd_bands(int nx, int ny, double alpha, const double *__restrict__ op, NdTab tb,
                                                 T *__restrict__ bands) {
  const int j = blockIdx.x * NT + threadIdx.x, i = blockIdx.y;
  if (j >= ny) return;
  const size_t M = (size_t)nx * ny, p = (size_t)i * ny + j;
  const int ip = i + 1 == nx ? 0 : i + 1, jp = j + 1 == ny ? 0 : j + 1;
  const cd c = cscale(ld_c(op, FDFD_OP_C * M + p), alpha);
  const cd x = cscale(cmul(ld_c(op, FDFD_OP_XP * M + p), cmul(ld_c(tb.ex, i), ld_c(tb.iex, ip))), alpha);
  const cd y = cscale(cmul(ld_c(op, FDFD_OP_YP * M + p), cmul(ld_c(tb.ey, j), ld_c(tb.iey, jp))), alpha);
  nd_st<T>(bands, p, (T)c.r, (T)c.i);
  nd_st<T>(bands + 2 * M, p, (T)x.r, (T)x.i);
  nd_st<T>(bands + 4 * M, p, (T)y.r, (T)y.i);
}

// Inverse of a symmetric TB x TB tile with 2 x 2 diagonal pivots taken in the
// order of their size: each step picks, of the adjacent pairs not yet taken,
// the block P with the largest |det P| / max |P_ij| (about 1 / ||P^-1||). The
// fronts of interior boxes are real and indefinite, and a fixed order meets
// small leading minors: on the request stream's 512 x 512 grid the complex64
// factor of seed 7 then does not refine at all, against a contraction of 2e-4
// per sweep with the picked order (2e-4 too for row pivoting inside the tile).
// Diagonal pivots move no rows. Only the upper triangle is read: the fronts
// stay symmetric to the last bit, without which the rounding of a nearly
// resonant box (|X| ~ 10^3) grows by another two digits on the way up.
//
// The steps are sweeps, which keep the tile symmetric: with f = the pivot rows
// and Q = P^-1 the tile becomes M - f^T Q f off the pivots, Q f on the pivot
// rows and columns, -Q on the block, and -M^-1 in the end. The tile lies in
// accumulators of 16x16x4 products, whose four inner indices are the two
// pivots' real and imaginary parts: a step is one product per quadrant and
// part, on the rows f that the lanes holding them publish in LDS (both
// operands, by symmetry). Pivot rows and columns are cleared and f is minus a
// unit vector at the pivots, so the same product leaves Q f and -Q there
// without cancellation. The diagonal blocks are kept aside and updated from f
// too: the next choice does not wait for the products.
__device__ inline float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ inline double lane_value(double v, int l) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const unsigned hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | lo);
}
// maximum over the quads of a wave (uniform)
__device__ inline int wave16_max(unsigned v) {
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false));   // row_ror:4
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false));
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));   // row_bcast:15
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));   // row_bcast:31
  return __builtin_amdgcn_readlane((int)v, 63);
}
template <typename T> struct WaveQ {   // Q = P^-1, uniform
  T q00r, q00i, q01r, q01i, q11r, q11i;
};
// p -= a b (complex)
template <typename T> __device__ inline void wave_sub(T &pr, T &pi, T ar, T ai, T br, T bi) {
  pr = fma(ai, bi, fma(-ar, br, pr));
  pi = fma(-ai, br, fma(-ar, bi, pi));
}
__device__ inline int frexp_of(float x) { return __builtin_amdgcn_frexp_expf(x); }
__device__ inline int frexp_of(double x) { return __builtin_amdgcn_frexp_exp(x); }
// LDS of an inverse: the pivot rows by column, real and imaginary parts
template <typename T> struct alignas(16) PivotRows {
  T v[2][TB][2];
};
// The diagonal blocks: lane 4 m + e of every wave keeps P00, P01, P11, P01 of
// pair m (e = 0 .. 3); quads exchange them by DPP
template <int E0, int E1, int E2, int E3> __device__ inline int quad(int v) {
  return __builtin_amdgcn_update_dpp(0, v, E0 | E1 << 2 | E2 << 4 | E3 << 6, 0xf, 0xf, true);
}
template <int E0, int E1, int E2, int E3> __device__ inline float quad(float v) {
  return __int_as_float(quad<E0, E1, E2, E3>(__float_as_int(v)));
}
template <int E0, int E1, int E2, int E3> __device__ inline double quad(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = quad<E0, E1, E2, E3>((int)(b & 0xffffffffll)), hi = quad<E0, E1, E2, E3>((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | lo);
}
template <typename T> struct PivotBlocks {
  T pr, pi, ar, ai, dr, di, da;
  int e;
  bool taken, bad;
  __device__ inline PivotBlocks(const T (*Ar)[TBP], const T (*Ai)[TBP], int pairs) {
    const int m = (threadIdx.x & 63) >> 2, q = threadIdx.x & 3, x = 2 * m + (q == 2), y = 2 * m + (q != 0);
    pr = Ar[x][y];
    pi = Ai[x][y];
    taken = m >= pairs;
    bad = false;
  }
  // the pair to eliminate next
  __device__ inline int pick() {
    const int m = (threadIdx.x & 63) >> 2;
    // scaled by an exact power of two near 1 / max |P_ij|
    T mx = fabs(pr) + fabs(pi);
    mx = fmax(mx, quad<1, 0, 3, 2>(mx));
    mx = fmax(mx, quad<2, 3, 0, 1>(mx));
    e = frexp_of(mx);
    ar = ldexp(pr, -e);
    ai = ldexp(pi, -e);
    const T a00r = quad<0, 0, 0, 0>(ar), a00i = quad<0, 0, 0, 0>(ai), a01r = quad<1, 1, 1, 1>(ar);
    const T a01i = quad<1, 1, 1, 1>(ai), a11r = quad<2, 2, 2, 2>(ar), a11i = quad<2, 2, 2, 2>(ai);
    dr = fma(a01i, a01i, fma(-a01r, a01r, fma(-a00i, a11i, a00r * a11r)));
    di = fma(T(-2) * a01r, a01i, fma(a00i, a11r, a00r * a11i));
    da = fabs(dr) + fabs(di);
    const unsigned size = __float_as_uint(fabsf((float)ldexp(da, e))) & ~15u;
    const int at = wave16_max(taken ? 0u : size + 16u + (unsigned)m) & 15;
    const bool now = m == at;
    bad |= now & !((da > T(0)) & (da < T(INFINITY)));
    taken |= now;
    return at;
  }
  // its inverse: 1 / det = (dr - i di) / |det|^2, det brought near 1 by an exact scale
  __device__ inline void inverse(int at, WaveQ<T> &Q) const {
    const int g = frexp_of(da);
    const T br = ldexp(dr, -g), bi = ldexp(di, -g);
    T rm = ldexp(rcp_nr(fma(bi, bi, br * br)), -e - g);
    rm = threadIdx.x & 1 ? -rm : rm;
    const T er = br * rm, ei = -bi * rm, nr = quad<2, 1, 0, 1>(ar), ni = quad<2, 1, 0, 1>(ai);
    const T qr = fma(-ni, ei, nr * er), qi = fma(ni, er, nr * ei);
    Q.q00r = lane_value(qr, 4 * at);
    Q.q00i = lane_value(qi, 4 * at);
    Q.q01r = lane_value(qr, 4 * at + 1);
    Q.q01i = lane_value(qi, 4 * at + 1);
    Q.q11r = lane_value(qr, 4 * at + 2);
    Q.q11i = lane_value(qi, 4 * at + 2);
  }
  // P_ab -= f(a)^T Q f(b)
  T xr[2], xi[2], yr[2], yi[2];
  __device__ inline void read(const PivotRows<T> &f) {
    const int m = (threadIdx.x & 63) >> 2, q = threadIdx.x & 3, x = 2 * m + (q == 2), y = 2 * m + (q != 0);
    lds_ld2(f.v[0][x], xr[0], xr[1]);
    lds_ld2(f.v[1][x], xi[0], xi[1]);
    lds_ld2(f.v[0][y], yr[0], yr[1]);
    lds_ld2(f.v[1][y], yi[0], yi[1]);
  }
  __device__ inline void update(const WaveQ<T> &Q) {
    T v0r = 0, v0i = 0, v1r = 0, v1i = 0;   // -Q f
    wave_sub(v0r, v0i, Q.q00r, Q.q00i, xr[0], xi[0]);
    wave_sub(v0r, v0i, Q.q01r, Q.q01i, xr[1], xi[1]);
    wave_sub(v1r, v1i, Q.q01r, Q.q01i, xr[0], xi[0]);
    wave_sub(v1r, v1i, Q.q11r, Q.q11i, xr[1], xi[1]);
    wave_sub(pr, pi, -v0r, -v0i, yr[0], yi[0]);
    wave_sub(pr, pi, -v1r, -v1i, yr[1], yi[1]);
  }
};
// The inner index kk = lane / 16 of a sweep's products (k = kk & 1, imaginary
// part for kk >= 2): w of -(Q f)_k as a combination of f's four values
template <typename T> struct SweepCoef {
  T w0, w1, w2, w3;
  bool part;
  __device__ inline SweepCoef(const WaveQ<T> &Q) {
    const int kk = (threadIdx.x >> 4) & 3, k = kk & 1;
    part = kk >> 1;
    const T s0r = k ? Q.q01r : Q.q00r, s0i = k ? Q.q01i : Q.q00i, s1r = k ? Q.q11r : Q.q01r, s1i = k ? Q.q11i : Q.q01i;
    w0 = part ? s0i : -s0r;
    w1 = part ? s0r : s0i;
    w2 = part ? s1i : -s1r;
    w3 = part ? s1r : s1i;
  }
  // left operands of the real and the imaginary products, for row values f[2]
  __device__ inline void left(T v0, T v1, T v2, T v3, T &re, T &im) const {
    re = fma(v3, w3, fma(v2, w2, fma(v1, w1, v0 * w0)));
    im = part ? -re : re;
  }
};
// Pivot rows jr, jr + 1 of a 16-row quadrant: in accumulators tt, tt + 1 of one
// lane group (f32), in accumulator tt of two groups (f64). Writes this lane's
// column of them, minus a unit vector at the pivots if the quadrant is
// diagonal; whether this lane holds them.
template <typename T> __device__ inline int pivot_acc(int jr) { return sizeof(T) == 8 ? jr >> 2 : jr & 2; }
template <typename T> __device__ inline constexpr int pivot_tt(int t) { return sizeof(T) == 8 ? t : t & 2; }
__device__ inline bool pivot_rows(PivotRows<float> &f, const Mfma<float>::v4 &mr, const Mfma<float>::v4 &mi, int col,
                                  int group, int jr, bool diagonal) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const bool own = group == jr >> 2;
  if (own) {
    const int c = col & 15;
    f2 r = f2{mr[0], mr[1]}, i = f2{mi[0], mi[1]};
    if (jr & 2) { r = f2{mr[2], mr[3]}; i = f2{mi[2], mi[3]}; }
    if (diagonal && (c & ~1) == jr) { r = f2{c == jr ? -1.0f : 0.0f, c == jr ? 0.0f : -1.0f}; i = f2{0, 0}; }
    *reinterpret_cast<f2 *>(f.v[0][col]) = r;
    *reinterpret_cast<f2 *>(f.v[1][col]) = i;
  }
  return own;
}
__device__ inline bool pivot_rows(PivotRows<double> &f, const Mfma<double>::v4 &mr, const Mfma<double>::v4 &mi, int col,
                                  int group, int jr, bool diagonal) {
  const int k = group - (jr & 3);
  const bool own = (k & ~1) == 0;
  if (own) {
    const int c = col & 15;
    double r, i;
    if (jr < 8) {
      if (jr < 4) { r = mr[0]; i = mi[0]; } else { r = mr[1]; i = mi[1]; }
    } else {
      if (jr < 12) { r = mr[2]; i = mi[2]; } else { r = mr[3]; i = mi[3]; }
    }
    if (diagonal && (c & ~1) == jr) { r = c == jr + k ? -1.0 : 0.0; i = 0; }
    f.v[0][col][k] = r;
    f.v[1][col][k] = i;
  }
  return own;
}
// The inverse of the tile in (Ar, Ai), in place, by four waves, a quadrant
// each; every wave keeps all diagonal blocks and makes the same choice, so a
// step has one barrier, between the rows' way into LDS (one of two buffers in
// turn) and out of it. rows: the tile's rows that are not identity padding; the
// pairs beyond are left alone (the step count is (rows + 1) / 2).
// Bound by one step's chain: choice, rows, barrier, blocks; about 150
// instructions, 0.34 us a pair. With the tile in registers row by row, the
// blocks read back from LDS and the update on vector units, 0.53 us: the factor
// of 512^2 complex64 2.04 -> 1.87 ms, of 120^2 FP64 0.61 -> 0.56 ms, of 768^2
// FP64 6.30 -> 6.03 ms. Tried with that layout: a fifth wave that picks and
// inverts the next pair while the others update (a step of 512^2 17 -> 20 us),
// and eight waves (18.6 us).
template <typename T, typename LT>
__device__ void tile_inverse_pairs(LT &L, int rows, int *status) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, qi = wv >> 1, qj = wv & 1, c = lane & 15;
  const int kk = lane >> 4, k = kk & 1, part = kk >> 1, pairs = min(TB, rows + 1) >> 1;
  typename Mfma<T>::v4 mr, mi;
#pragma unroll
  for (int t = 0; t < 4; ++t) {   // the upper triangle
    const int r = 16 * qi + Mfma<T>::crow(lane, t), x = min(r, 16 * qj + c), y = max(r, 16 * qj + c);
    mr[t] = L.Ar[x][y];
    mi[t] = L.Ai[x][y];
  }
  PivotBlocks<T> B(L.Ar, L.Ai, pairs);
#pragma unroll 2
  for (int st = 0; st < pairs; ++st) {
    PivotRows<T> &f = L.f[st & 1];
    const int at = B.pick(), j = 2 * at, jr = j & 15;
    const bool inr = j >> 4 == qi, inc = j >> 4 == qj, pc = inc && (c & ~1) == jr;
    bool own = inr;
    if (inr) own = pivot_rows(f, mr, mi, 16 * qj + c, kk, jr, inc);
    const int tt = pivot_acc<T>(jr);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool zero = pc || (own && pivot_tt<T>(t) == tt);
      mr[t] = zero ? T(0) : mr[t];
      mi[t] = zero ? T(0) : mi[t];
    }
    WaveQ<T> Q;
    B.inverse(at, Q);
    const SweepCoef<T> W(Q);
    __syncthreads();
    T v0, v1, v2, v3, are, aim;
    lds_ld2(f.v[0][16 * qi + c], v0, v2);
    lds_ld2(f.v[1][16 * qi + c], v1, v3);
    const T bre = f.v[part][16 * qj + c][k], bim = f.v[1 - part][16 * qj + c][k];
    B.read(f);
    __builtin_amdgcn_sched_barrier(0);   // all reads first: they wait for LDS once
    W.left(v0, v1, v2, v3, are, aim);
    mr = Mfma<T>::mac(are, bre, mr);
    mi = Mfma<T>::mac(aim, bim, mi);
    B.update(Q);
  }
  // the padding stays
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int r = 16 * qi + Mfma<T>::crow(lane, t);
    L.Ar[r][16 * qj + c] = r < 2 * pairs ? -mr[t] : mr[t];
    L.Ai[r][16 * qj + c] = r < 2 * pairs ? -mi[t] : mi[t];
  }
  if (B.bad) *status = 1;
  __syncthreads();
}

// The same inverse by one wave, for the leaves, of which there are thousands:
// the choice's instructions are issued once a leaf and not by four waves. Bound
// by them: the 8192 leaves of 512^2 complex64 110 -> 51 us, the 16384 of 768^2
// FP64 469 -> 200 us. As the chain of one tile it is slower than four waves
// and takes over 200 registers in FP64.
// within a wave: LDS stores before this are seen by loads after it
__device__ inline void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }
template <typename T> struct WaveTile {
  typename Mfma<T>::v4 r[2][2], i[2][2];
};
// LDS of one wave's inverse: the pivot rows by column, and a second set for
// the lanes that have none to write (a branch on lanes inside the choice of
// the accumulators makes the compiler copy the tile at every join)
template <typename T> struct WaveRows {
  PivotRows<T> rows, none;
};
// The pivot rows j, j + 1 (j = 16 QR + jr, in accumulator TT: of one lane
// group for f32, one each of two for f64) go to f; the pivot rows and columns
// are cleared in the tile.
template <int QR, int TT>
__device__ inline void wave_rows(WaveTile<float> &M, WaveRows<float> &f, int lane, int jr) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const int c = lane & 15;
  const bool own = (lane >> 4) == (jr >> 2), pc = (c & ~1) == jr;
  PivotRows<float> &to = own ? f.rows : f.none;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    *reinterpret_cast<f2 *>(to.v[0][16 * q + c]) = f2{M.r[QR][q][TT], M.r[QR][q][TT + 1]};
    *reinterpret_cast<f2 *>(to.v[1][16 * q + c]) = f2{M.i[QR][q][TT], M.i[QR][q][TT + 1]};
  }
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool row = t == TT || t == TT + 1, both = q == QR && row;
      if (row) {
        M.r[QR][q][t] = own || (both && pc) ? 0.0f : M.r[QR][q][t];
        M.i[QR][q][t] = own || (both && pc) ? 0.0f : M.i[QR][q][t];
      }
      if (!both) {
        M.r[q][QR][t] = pc ? 0.0f : M.r[q][QR][t];
        M.i[q][QR][t] = pc ? 0.0f : M.i[q][QR][t];
      }
    }
}
template <int QR, int TT>
__device__ inline void wave_rows(WaveTile<double> &M, WaveRows<double> &f, int lane, int jr) {
  const int c = lane & 15, k = (lane >> 4) - (jr & 3);
  const bool own = k == 0 || k == 1, pc = (c & ~1) == jr;
  PivotRows<double> &to = own ? f.rows : f.none;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    to.v[0][16 * q + c][k & 1] = M.r[QR][q][TT];
    to.v[1][16 * q + c][k & 1] = M.i[QR][q][TT];
  }
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool row = t == TT, both = q == QR && row;
      if (row) {
        M.r[QR][q][t] = own || (both && pc) ? 0.0 : M.r[QR][q][t];
        M.i[QR][q][t] = own || (both && pc) ? 0.0 : M.i[QR][q][t];
      }
      if (!both) {
        M.r[q][QR][t] = pc ? 0.0 : M.r[q][QR][t];
        M.i[q][QR][t] = pc ? 0.0 : M.i[q][QR][t];
      }
    }
}
// One sweep's products on the rows in accumulator TT of quadrant row QR
template <int QR, int TT, typename T>
__device__ inline void wave_sweep(WaveTile<T> &M, WaveRows<T> &f, int lane, int j, const WaveQ<T> &Q) {
  const int c = lane & 15, kk = lane >> 4, k = kk & 1, part = kk >> 1;
  wave_rows<QR, TT>(M, f, lane, j & 15);
  wave_lds_fence();
  PivotRows<T> &unit = lane < 2 ? f.rows : f.none;   // minus a unit vector at the pivots
  const int l = lane & 1;
  unit.v[0][j + l][0] = l ? T(0) : T(-1);
  unit.v[0][j + l][1] = l ? T(-1) : T(0);
  unit.v[1][j + l][0] = unit.v[1][j + l][1] = 0;
  wave_lds_fence();
  const SweepCoef<T> W(Q);
  T are[2], aim[2], bre[2], bim[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    bre[q] = f.rows.v[part][16 * q + c][k];
    bim[q] = f.rows.v[1 - part][16 * q + c][k];
    T v0, v1, v2, v3;
    lds_ld2(f.rows.v[0][16 * q + c], v0, v2);
    lds_ld2(f.rows.v[1][16 * q + c], v1, v3);
    W.left(v0, v1, v2, v3, are[q], aim[q]);
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      M.r[a][b] = Mfma<T>::mac(are[a], bre[b], M.r[a][b]);
      M.i[a][b] = Mfma<T>::mac(aim[a], bim[b], M.i[a][b]);
    }
}
__device__ inline void wave_sweep_at(WaveTile<float> &M, WaveRows<float> &f, int lane, int j, const WaveQ<float> &Q) {
  if (j < 16) {
    if (j & 2) wave_sweep<0, 2>(M, f, lane, j, Q); else wave_sweep<0, 0>(M, f, lane, j, Q);
  } else {
    if (j & 2) wave_sweep<1, 2>(M, f, lane, j, Q); else wave_sweep<1, 0>(M, f, lane, j, Q);
  }
}
__device__ inline void wave_sweep_at(WaveTile<double> &M, WaveRows<double> &f, int lane, int j,
                                     const WaveQ<double> &Q) {
  if (j < 16) {
    if (j < 8) { if (j < 4) wave_sweep<0, 0>(M, f, lane, j, Q); else wave_sweep<0, 1>(M, f, lane, j, Q); }
    else { if (j < 12) wave_sweep<0, 2>(M, f, lane, j, Q); else wave_sweep<0, 3>(M, f, lane, j, Q); }
  } else {
    if (j < 24) { if (j < 20) wave_sweep<1, 0>(M, f, lane, j, Q); else wave_sweep<1, 1>(M, f, lane, j, Q); }
    else { if (j < 28) wave_sweep<1, 2>(M, f, lane, j, Q); else wave_sweep<1, 3>(M, f, lane, j, Q); }
  }
}
// (Ar, Ai) in LDS -> its inverse in M, entry (16 a + crow(lane, t), 16 b + lane % 16)
// in element t of quadrant (a, b); f: LDS that no other wave uses.
// rows: the tile's rows that are not identity padding; the pairs beyond are
// left alone (the step count is (rows + 1) / 2). False: singular.
template <typename T>
__device__ inline bool wave_inverse(WaveTile<T> &M, const T (*Ar)[TBP], const T (*Ai)[TBP], WaveRows<T> &f, int rows) {
  const int lane = threadIdx.x & 63, mine = lane & 15;
  const int pairs = min(TB, rows + 1) >> 1;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 16 * a + Mfma<T>::crow(lane, t), c = 16 * b + mine;
        const int x = min(r, c), y = max(r, c);
        M.r[a][b][t] = Ar[x][y];
        M.i[a][b][t] = Ai[x][y];
      }
  PivotBlocks<T> B(Ar, Ai, pairs);
#pragma unroll 1
  for (int st = 0; st < pairs; ++st) {
    const int pick = B.pick();
    WaveQ<T> Q;
    B.inverse(pick, Q);
    wave_lds_fence();
    wave_sweep_at(M, f, lane, 2 * pick, Q);
    B.read(f.rows);
    B.update(Q);
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool neg = 16 * a + Mfma<T>::crow(lane, t) < 2 * pairs;   // the padding stays
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        M.r[a][b][t] = neg ? -M.r[a][b][t] : M.r[a][b][t];
        M.i[a][b][t] = neg ? -M.i[a][b][t] : M.i[a][b][t];
      }
    }
  return !B.bad;
}
// M into a tile of pitch `pitch`
template <typename T>
__device__ inline void wave_store(const WaveTile<T> &M, T *re, T *im, int pitch) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int e = (16 * a + Mfma<T>::crow(lane, t)) * pitch + 16 * b + (lane & 15);
        re[e] = M.r[a][b][t];
        im[e] = M.i[a][b][t];
      }
}

// LDS of the kernels that invert a tile: A (the tile, then its inverse), B
// (with A: the exchange buffers of the inverse) and, where used, a third tile.
template <typename T> struct NdLds2 {
  T Ar[TB][TBP], Ai[TB][TBP];
  union {
    struct { T Br[TB][TBP], Bi[TB][TBP]; };
    PivotRows<T> f[2];
  };
};
template <typename T> struct NdLds3 {
  T Ar[TB][TBP], Ai[TB][TBP];
  union {
    struct { T Br[TB][TBP], Bi[TB][TBP]; };
    PivotRows<T> f[2];
  };
  T Pr[TB][TBP], Pi[TB][TBP];
};

// A leaf box per wave: its five-point matrix (cells in (x, y) order,
// identity beyond) inverted as one pivot tile; X, the border couplings c and
// the update C[a][b] = -c_a X[p_a][p_b] c_b, p_a the cell inside border cell a.
template <typename T>
__global__ void __launch_bounds__(64, 2) k_nd_leaf(int nx, int ny, int Dx, int Dy, NdBands<T> bd, T *__restrict__ X,
                                                T *__restrict__ cpl, T *__restrict__ C, int *status) {
  __shared__ T Ar[TB][TBP], Ai[TB][TBP], cr[TB], ci[TB];
  __shared__ WaveRows<T> f;
  __shared__ int cp[TB];
  const int lane = threadIdx.x, k = blockIdx.x;
  const int ix = k >> Dy, iy = k & ((1 << Dy) - 1);
  int x0, w, y0, h;
  nd_seg(nx, Dx, ix, x0, w);
  nd_seg(ny, Dy, iy, y0, h);
  const int s = w * h, b = 2 * (w + h);
  const int b0 = (lane & 7) * 4, a0 = lane >> 3;
#pragma unroll
  for (int e = lane; e < TB * TBP; e += 64) {
    (&Ar[0][0])[e] = 0;
    (&Ai[0][0])[e] = 0;
  }
  wave_lds_fence();
  if (lane < TB) {   // the upper triangle: itself, the next cell in y and in x
    T re = 1, im = 0;
    if (lane < s) {
      const int i = lane / h, j = lane - i * h;
      const size_t p = (size_t)(x0 + i) * ny + y0 + j;
      nd_ld(bd.c, p, re, im);
      T yr = 0, yi = 0, xr = 0, xi = 0;
      if (j + 1 < h) nd_ld(bd.y, p, yr, yi);
      if (i + 1 < w) nd_ld(bd.x, p, xr, xi);
      if (j + 1 < h) { Ar[lane][lane + 1] = yr; Ai[lane][lane + 1] = yi; }
      if (i + 1 < w) { Ar[lane][lane + h] = xr; Ai[lane][lane + h] = xi; }
    }
    Ar[lane][lane] = re;
    Ai[lane][lane] = im;
    re = im = 0;
    int p = 0;
    if (lane < h) {
      p = lane;
      nd_ld(bd.x, (size_t)(x0 - 1) * ny + y0 + lane, re, im);
    } else if (lane < 2 * h) {
      p = (w - 1) * h + lane - h;
      nd_ld(bd.x, (size_t)(x0 + w - 1) * ny + y0 + lane - h, re, im);
    } else if (lane < 2 * h + w) {
      p = (lane - 2 * h) * h;
      nd_ld(bd.y, (size_t)(x0 + lane - 2 * h) * ny + y0 - 1, re, im);
    } else if (lane < b) {
      p = (lane - 2 * h - w) * h + h - 1;
      nd_ld(bd.y, (size_t)(x0 + lane - 2 * h - w) * ny + y0 + h - 1, re, im);
    }
    cr[lane] = re;
    ci[lane] = im;
    cp[lane] = p;
    nd_st<T>(cpl, (size_t)k * TB + lane, re, im);
  }
  wave_lds_fence();
  WaveTile<T> M;
  if (!wave_inverse<T>(M, Ar, Ai, f, s)) *status = 1;
  wave_lds_fence();
  wave_store<T>(M, &Ar[0][0], &Ai[0][0], TBP);
  wave_lds_fence();
  T *Xk = X + (size_t)k * 2 * TB * TB, *Ck = C + (size_t)k * 2 * TB * TB;
  for (int a = a0; a < s; a += 8) {
    store4(Xk + a * TB + b0, &Ar[a][b0]);
    store4(Xk + TB * TB + a * TB + b0, &Ai[a][b0]);
  }
  for (int a = a0; a < b; a += 8) {
    T vr[4], vi[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int x = min(a, b0 + u), y = max(a, b0 + u);   // symmetric to the last bit
      const T xr = Ar[cp[x]][cp[y]], xi = Ai[cp[x]][cp[y]];
      const T tr = cr[x] * xr - ci[x] * xi, ti = cr[x] * xi + ci[x] * xr;
      vr[u] = -(tr * cr[y] - ti * ci[y]);
      vi[u] = -(tr * ci[y] + ti * cr[y]);
    }
    store4(Ck + a * TB + b0, vr);
    store4(Ck + TB * TB + a * TB + b0, vi);
  }
}

// Four consecutive entries (row i of the front, columns given by their
// children's entries) summed from the children's updates.
template <typename T>
__device__ inline void nd_children(const NdLevel &L, const NdBox &B, const T *__restrict__ C, int r0, int r1,
                                   const int (&c0)[4], const int (&c1)[4], T (&re)[4], T (&im)[4]) {
  const size_t pl = (size_t)L.cbp * L.cbp;
  const T *A0 = C + (size_t)B.k0 * 2 * pl + (size_t)(r0 < 0 ? 0 : r0) * L.cbp;
  const T *A1 = C + (size_t)B.k1 * 2 * pl + (size_t)(r1 < 0 ? 0 : r1) * L.cbp;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    re[u] = 0;
    im[u] = 0;
    if (r0 >= 0 && c0[u] >= 0) { re[u] = A0[c0[u]]; im[u] = A0[pl + c0[u]]; }
    if (r1 >= 0 && c1[u] >= 0) { re[u] += A1[c1[u]]; im[u] += A1[pl + c1[u]]; }
  }
}
// The entries of M itself between separator entries i and j
template <typename T>
__device__ inline void nd_own_ss(const NdLevel &L, const NdBox &B, const NdBands<T> &bd, int i, int j, T &re, T &im) {
  re = 0;
  im = 0;
  if (i == j) { nd_ld(bd.c, nd_sep_cell(L, B, i), re, im); return; }
  const int lo = min(i, j), hi = max(i, j);
  if (!L.root) {
    if (hi == lo + 1) nd_ld(L.ax == 0 ? bd.y : bd.x, nd_sep_cell(L, B, lo), re, im);
    return;
  }
  // the cross: rows 1.. of column 0, columns 1.. of row 0, cell (0, 0)
  const int h = L.ny - 1, n = L.s;
  if (hi == n - 1) {
    if (lo == 0) nd_ld(bd.y, 0, re, im);
    else if (lo == h - 1) nd_ld(bd.y, (size_t)(L.ny - 1), re, im);
    else if (lo == h) nd_ld(bd.x, 0, re, im);
    else if (lo == n - 2) nd_ld(bd.x, (size_t)(L.nx - 1) * L.ny, re, im);
  } else if (hi == lo + 1 && hi != h) {
    nd_ld(lo < h ? bd.y : bd.x, nd_sep_cell(L, B, lo), re, im);
  }
}
// ... between separator entry i and border entry j (the separator's ends)
template <typename T>
__device__ inline void nd_own_sb(const NdLevel &L, const NdBox &B, const NdBands<T> &bd, int i, int j, T &re, T &im) {
  const int o = L.ax == 0 ? B.oB : 0, far = L.ax == 0 ? (L.dy ? B.w : 0) : (L.dx ? B.h : 0);
  const T *p = L.ax == 0 ? bd.y : bd.x;
  const size_t step = L.ax == 0 ? 1 : (size_t)L.ny;
  if (i == 0 && j == o + B.c0) {
    T r, m;
    nd_ld(p, nd_sep_cell(L, B, 0) - step, r, m);
    re += r;
    im += m;
  }
  if (i == B.s - 1 && j == o + far + B.c0) {
    T r, m;
    nd_ld(p, nd_sep_cell(L, B, B.s - 1), r, m);
    re += r;
    im += m;
  }
}

// Workgroup g of total items cut into XCDS equal ranges, one per XCD (the
// dispatcher places workgroup b on XCD b % XCDS): neighbouring items, which
// read the same rows and panels, share an L2. -1: past the end.
__device__ inline int nd_item(int g, int total) {
  const int x = g % XCDS, i = (int)((long)total * x / XCDS) + g / XCDS;
  return i < (int)((long)total * (x + 1) / XCDS) ? i : -1;
}
inline int nd_grid(int total) { return XCDS * ((total + XCDS - 1) / XCDS); }

template <typename T> struct NdStep {
  NdLevel L;
  NdBands<T> bd;
  const T *C;              // the children's updates
  const T *Ss, *Sb;        // [F_ss], [F_sb] before the step
  T *Ds, *Db;              // after it
  T *P0, *P1;              // pivot inverses of this step and the next
  T *U, *R;                // rows of the border part as they are eliminated, before and after P
  int *status;
  int p;
};

// The front's [F_ss | F_sb] (tiles I <= J and the border's) from the
// children, and the inverse of the first pivot tile.
template <typename T>
__global__ void __launch_bounds__(NT, 2) k_nd_front(NdStep<T> A) {
  __shared__ NdLds2<T> S;
  const NdLevel &L = A.L;
  const int ns = L.sp / TB, nb = L.bp / TB, tri = ns * (ns + 1) / 2, per = tri + ns * nb;
  int box, t;
  if ((int)blockIdx.x < L.nbox) {       // the tiles inverted here go first
    box = blockIdx.x;
    t = 0;
  } else {
    const int first = (L.nbox + XCDS - 1) / XCDS * XCDS;
    if ((int)blockIdx.x < first) return;
    const int it = nd_item(blockIdx.x - first, L.nbox * (per - 1));
    if (it < 0) return;
    box = it / (per - 1);
    t = 1 + it % (per - 1);
  }
  const NdBox B = nd_box(L, box);
  int I, J;
  if (t < tri) { const int e = upper_tile(ns, t); I = e / ns; J = e % ns; }
  else { I = (t - tri) / nb; J = ns + (t - tri) % nb; }
  const int tid = threadIdx.x, a = tid >> 3, b0 = (tid & 7) * 4;
  const int i = I * TB + a;
  T re[4], im[4];
  int c0[4], c1[4], r0 = -1, r1 = -1;
  if (i < B.s) nd_sep_map(L, B, i, r0, r1);
  if (J < ns) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = J * TB + b0 + u;
      c0[u] = c1[u] = -1;
      if (j < B.s) nd_sep_map(L, B, j, c0[u], c1[u]);
    }
    nd_children(L, B, A.C, r0, r1, c0, c1, re, im);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = J * TB + b0 + u;
      T mr = i == j ? T(1) : T(0), mi = 0;
      if (i < B.s && j < B.s) nd_own_ss(L, B, A.bd, i, j, mr, mi);
      re[u] += mr;
      im[u] += mi;
    }
    if (t == 0) {
#pragma unroll
      for (int u = 0; u < 4; ++u) { S.Ar[a][b0 + u] = re[u]; S.Ai[a][b0 + u] = im[u]; }
      __syncthreads();
      tile_inverse_pairs<T>(S, B.s, A.status);
      store_pinv(S, A.P0 + (size_t)box * 2 * TB * TB);
      return;
    }
    T *D = A.Ds + (size_t)box * 2 * L.sp * L.sp + (size_t)i * L.sp + J * TB + b0;
    store4(D, re);
    store4(D + (size_t)L.sp * L.sp, im);
  } else {
    const int j0 = (J - ns) * TB + b0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      c0[u] = c1[u] = -1;
      if (j0 + u < B.b) nd_border_map(L, B, j0 + u, c0[u], c1[u]);
    }
    nd_children(L, B, A.C, r0, r1, c0, c1, re, im);
    if (i == 0 || i == B.s - 1)
#pragma unroll
      for (int u = 0; u < 4; ++u) nd_own_sb(L, B, A.bd, i, j0 + u, re[u], im[u]);
    T *D = A.U + (size_t)box * 2 * L.sp * L.bp + (size_t)i * L.bp + j0;
    store4(D, re);
    store4(D + (size_t)L.sp * L.bp, im);
  }
}

// Gauss-Jordan step p on the tiles (I, J), I <= J < ns, and (I, J) of the
// border (J >= ns), of every box, as in k_gj_step with D = 1:
//   I == p == J: P;  I == p: P X[p,J];  J == p: -X[I,p] P;
//   else X[I,J] - X[I,p] (P X[p,J]),
// X[p,J] = -X[J,p]^T for J < p and X[I,p] = X[p,I]^T for I > p. The workgroup
// of tile (p+1, p+1) inverts it for the next step; these start first. The
// last step writes X and W into the factor, X with both triangles. The border
// tiles of row p leave X[p,J] (U) and P X[p,J] (R) behind: the update is
// C = F_bb - sum_p U_p^T R_p, as elimination forms it. (F_sb^T W with the
// finished W loses the digits that a nearly resonant box costs twice: the
// complex64 factor of a 512 x 512 stream grid with |X| = 550 in one box then
// contracts by 0.03-0.2 per sweep instead of 2e-4.)
// A workgroup takes two tiles of a column, rows I = 2 i and 2 i + 1, which
// share P X[p,J]: three products for two tiles instead of four, P and X[p,J]
// read once. Bound by the inverse's chain where the tiles are few and by the
// matrix cores and the pass over the front where they are many: a step of 1200
// tiles, complex64 20.2 -> 18.9 us, of 2600 tiles, FP64 37 -> 33 us.
__host__ __device__ inline int nd_step_items(int ns, int nb) {
  const int np = (ns + 1) / 2;
  return np * (np + 1) + np * nb;
}
template <typename T>
__global__ void __launch_bounds__(NT, 2) k_nd_step(NdStep<T> A) {
  __shared__ NdLds3<T> S;
  const NdLevel &L = A.L;
  const int ns = L.sp / TB, nb = L.bp / TB, np = (ns + 1) / 2, per = nd_step_items(ns, nb), p = A.p;
  const bool last = p == ns - 1;
  const int ncrit = last ? 0 : L.nbox, first = (ncrit + XCDS - 1) / XCDS * XCDS;
  int box, I0, J;
  bool crit = false;
  if ((int)blockIdx.x < ncrit) {
    box = blockIdx.x;
    I0 = J = p + 1;
    crit = true;
    __builtin_amdgcn_s_setprio(3);
  } else {
    if ((int)blockIdx.x < first) return;
    const int it = nd_item(blockIdx.x - first, L.nbox * per);
    if (it < 0) return;
    box = it / per;
    const int t = it % per, tri = np * (np + 1);
    if (t < tri) { const int e = upper_tile(np, t >> 1); I0 = e / np * 2; J = e % np * 2 + (t & 1); }
    else { I0 = (t - tri) / nb * 2; J = ns + (t - tri) % nb; }
    if (J < I0 || (J >= ns && t < tri)) return;   // ns is odd
  }
  // which of the two there are
  const auto skips = [&](int I) { return I >= ns || I > J || (!crit && !last && I == p + 1 && J == p + 1); };
  const bool has[2] = {!skips(I0), !crit && !skips(I0 + 1)};
  if (!has[0] && !has[1]) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, qi = wv >> 1, qj = wv & 1;
  const int a = tid >> 3, b0 = (tid & 7) * 4;
  const size_t sp = L.sp, bp = L.bp, ps = sp * sp, pb = sp * bp;
  const T *Ss = A.Ss + (size_t)box * 2 * ps, *Sb = A.Sb + (size_t)box * 2 * pb;
  const T *P = A.P0 + (size_t)box * 2 * TB * TB;
  const bool col = J == p, mirA = J < p;
  // every global read first: P, X[p,J], X[I,p] and the tiles themselves
  T pr[4], pi[4], ar[4], ai[4], br[2][4], bi[2][4];
  typename Mfma<T>::v4 cr[2], ci[2];
  ld_row4(P + a * TB + b0, pr);
  ld_row4(P + TB * TB + a * TB + b0, pi);
  if (!col) {
    const T *q = J >= ns ? Sb + (p * TB + a) * bp + (size_t)(J - ns) * TB + b0
                         : (mirA ? Ss + ((size_t)J * TB + a) * sp + p * TB + b0
                                 : Ss + ((size_t)p * TB + a) * sp + J * TB + b0);
    const size_t pl = J >= ns ? pb : ps;
    ld_row4(q, ar);
    ld_row4(q + pl, ai);
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int I = I0 + h;
    cr[h] = ci[h] = typename Mfma<T>::v4{0, 0, 0, 0};
    if (!has[h] || I == p) continue;
    const T *q = I > p ? Ss + ((size_t)p * TB + a) * sp + I * TB + b0 : Ss + ((size_t)I * TB + a) * sp + p * TB + b0;
    ld_row4(q, br[h]);
    ld_row4(q + ps, bi[h]);
    if (col) continue;
    q = J >= ns ? Sb + (size_t)(J - ns) * TB : Ss + (size_t)J * TB;
    const size_t pitch = J >= ns ? bp : sp, pl = J >= ns ? pb : ps;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const size_t e = (size_t)(I * TB + qi * 16 + Mfma<T>::crow(lane, t)) * pitch + qj * 16 + (lane & 15);
      cr[h][t] = q[e];
      ci[h][t] = q[pl + e];
    }
  }
  // X[I,p] of the first row to B, of the second to A (J == p) or, once P X[p,J] is formed, to P
  const auto put = [&](int h, T (*dr)[TBP], T (*di)[TBP]) {
    if (!has[h] || I0 + h == p) return;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = b0 + u;
      if (I0 + h > p) { dr[c][a] = br[h][u]; di[c][a] = bi[h][u]; }
      else { dr[a][c] = br[h][u]; di[a][c] = bi[h][u]; }
    }
  };
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int c = b0 + u;
    S.Pr[a][c] = pr[u];
    S.Pi[a][c] = pi[u];
    if (!col) {
      if (mirA) { S.Ar[c][a] = -ar[u]; S.Ai[c][a] = -ai[u]; }
      else { S.Ar[a][c] = ar[u]; S.Ai[a][c] = ai[u]; }
    }
  }
  put(0, S.Br, S.Bi);
  if (col) put(1, S.Ar, S.Ai);
  __syncthreads();
  if (col) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!has[h]) continue;
      if (I0 + h == p) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int x = qi * 16 + Mfma<T>::crow(lane, t), y = qj * 16 + (lane & 15);
          cr[h][t] = S.Pr[x][y];
          ci[h][t] = S.Pi[x][y];
        }
      } else {
        cgemm_quad<T>(cr[h], ci[h], h ? S.Ar : S.Br, h ? S.Ai : S.Bi, S.Pr, S.Pi, qi, qj, lane, T(-1));
      }
    }
  } else {
    typename Mfma<T>::v4 rr = {0, 0, 0, 0}, ri = {0, 0, 0, 0};
    cgemm_quad<T>(rr, ri, S.Pr, S.Pi, S.Ar, S.Ai, qi, qj, lane, T(1));
    __syncthreads();   // every wave has read P and X[p,J]
    acc_to_lds<T>(rr, ri, S.Ar, S.Ai, qi, qj, lane);
    put(1, S.Pr, S.Pi);
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!has[h]) continue;
      if (I0 + h == p) { cr[h] = rr; ci[h] = ri; }
      else cgemm_quad<T>(cr[h], ci[h], h ? S.Pr : S.Br, h ? S.Pi : S.Bi, S.Ar, S.Ai, qi, qj, lane, T(-1));
    }
  }
  // out through LDS as whole rows
  __syncthreads();
  if (crit) {   // replaced by its inverse at the next step and read by nobody before
    acc_to_lds<T>(cr[0], ci[0], S.Ar, S.Ai, qi, qj, lane);
    __syncthreads();
    tile_inverse_pairs<T>(S, nd_box(L, box).s - (p + 1) * TB, A.status);
    store_pinv(S, A.P1 + (size_t)box * 2 * TB * TB);
    return;
  }
  if (has[0]) acc_to_lds<T>(cr[0], ci[0], S.Br, S.Bi, qi, qj, lane);
  if (has[1]) acc_to_lds<T>(cr[1], ci[1], S.Pr, S.Pi, qi, qj, lane);
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (!has[h]) continue;
    const int I = I0 + h;
    const T (*Or)[TBP] = h ? S.Pr : S.Br, (*Oi)[TBP] = h ? S.Pi : S.Bi;
    if (J >= ns) {
      const size_t o = (size_t)box * 2 * pb + ((size_t)I * TB + a) * bp + (size_t)(J - ns) * TB + b0;
      store4(A.Db + o, &Or[a][b0]);
      store4(A.Db + o + pb, &Oi[a][b0]);
      if (I == p && ns > 1) {
        store4(A.R + o, &Or[a][b0]);
        store4(A.R + o + pb, &Oi[a][b0]);
        if (p > 0) {   // at p = 0 U holds F_sb itself
          store4(A.U + o, ar);
          store4(A.U + o + pb, ai);
        }
      }
      continue;
    }
    T *D = A.Ds + (size_t)box * 2 * ps;
    store4(D + ((size_t)I * TB + a) * sp + J * TB + b0, &Or[a][b0]);
    store4(D + ps + ((size_t)I * TB + a) * sp + J * TB + b0, &Oi[a][b0]);
    if (last && I != J) {
      T mr[4], mi[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) { mr[u] = Or[b0 + u][a]; mi[u] = Oi[b0 + u][a]; }
      store4(D + ((size_t)J * TB + a) * sp + I * TB + b0, mr);
      store4(D + ps + ((size_t)J * TB + a) * sp + I * TB + b0, mi);
    }
  }
}

// c += sign * A^T[quadrant rows, :] * B[:, quadrant cols], both tiles stored
// with the inner index as rows.
template <typename T>
__device__ inline void cgemm_quad_tn(typename Mfma<T>::v4 &cr, typename Mfma<T>::v4 &ci, const T (*Ar)[TBP],
                                     const T (*Ai)[TBP], const T (*Br)[TBP], const T (*Bi)[TBP], int qi, int qj,
                                     int lane, T sign) {
  const int r = lane & 15, kq = lane >> 4;
  const int k0 = (kq >> 1) + 16 * (kq & 1);
#pragma unroll
  for (int s = 0; s < TB / 4; ++s) {
    const int k = 2 * s + k0;
    const T ar = sign * Ar[k][qi * 16 + r], ai = sign * Ai[k][qi * 16 + r];
    const T br = Br[k][qj * 16 + r], bi = Bi[k][qj * 16 + r];
    cr = Mfma<T>::mac(ar, br, cr);
    cr = Mfma<T>::mac(-ai, bi, cr);
    ci = Mfma<T>::mac(ar, bi, ci);
    ci = Mfma<T>::mac(ai, br, ci);
  }
}

// C = F_bb - U^T R: one tile I <= J of one box per workgroup, stored with
// its mirror image; F_bb is summed from the children as the tile is stored.
template <typename T>
__global__ void __launch_bounds__(NT) k_nd_update(NdLevel L, const T *__restrict__ Cin, const T *__restrict__ U,
                                                  const T *__restrict__ R, T *__restrict__ Cout) {
  __shared__ T Ar[TB][TBP], Ai[TB][TBP], Br[TB][TBP], Bi[TB][TBP];
  const int ns = L.sp / TB, nb = L.bp / TB, per = nb * (nb + 1) / 2;
  const int it = nd_item(blockIdx.x, L.nbox * per);
  if (it < 0) return;
  const int box = it / per, e = upper_tile(nb, it % per), I = e / nb, J = e % nb;
  const NdBox B = nd_box(L, box);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, qi = wv >> 1, qj = wv & 1;
  const int a = tid >> 3, b0 = (tid & 7) * 4;
  const size_t bp = L.bp, pb = (size_t)L.sp * bp;
  const T *F = U + (size_t)box * 2 * pb + (size_t)a * bp + I * TB + b0;
  const T *V = R + (size_t)box * 2 * pb + (size_t)a * bp + J * TB + b0;
  T ar[4], ai[4], br[4], bi[4];
  typename Mfma<T>::v4 cr = {0, 0, 0, 0}, ci = {0, 0, 0, 0};
  ld_row4(F, ar);
  ld_row4(F + pb, ai);
  ld_row4(V, br);
  ld_row4(V + pb, bi);
  for (int k = 0; k < ns; ++k) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      Ar[a][b0 + u] = ar[u];
      Ai[a][b0 + u] = ai[u];
      Br[a][b0 + u] = br[u];
      Bi[a][b0 + u] = bi[u];
    }
    __syncthreads();
    if (k + 1 < ns) {
      const size_t o = (size_t)(k + 1) * TB * bp;
      ld_row4(F + o, ar);
      ld_row4(F + o + pb, ai);
      ld_row4(V + o, br);
      ld_row4(V + o + pb, bi);
    }
    cgemm_quad_tn<T>(cr, ci, Ar, Ai, Br, Bi, qi, qj, lane, T(-1));
    __syncthreads();
  }
  acc_to_lds<T>(cr, ci, Ar, Ai, qi, qj, lane);
  int c0[4], c1[4], r0 = -1, r1 = -1;
  if (I * TB + a < B.b) nd_border_map(L, B, I * TB + a, r0, r1);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    c0[u] = c1[u] = -1;
    if (J * TB + b0 + u < B.b) nd_border_map(L, B, J * TB + b0 + u, c0[u], c1[u]);
  }
  T re[4], im[4];
  nd_children(L, B, Cin, r0, r1, c0, c1, re, im);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    re[u] += Ar[a][b0 + u];
    im[u] += Ai[a][b0 + u];
  }
  T *D = Cout + (size_t)box * 2 * bp * bp;
#pragma unroll
  for (int u = 0; u < 4; ++u) { Ar[a][b0 + u] = re[u]; Ai[a][b0 + u] = im[u]; }
  __syncthreads();
  if (I == J) {   // a diagonal tile's lower triangle mirrors its upper one
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (b0 + u < a) { re[u] = Ar[b0 + u][a]; im[u] = Ai[b0 + u][a]; }
  }
  store4(D + ((size_t)I * TB + a) * bp + J * TB + b0, re);
  store4(D + bp * bp + ((size_t)I * TB + a) * bp + J * TB + b0, im);
  if (I == J) return;
#pragma unroll
  for (int u = 0; u < 4; ++u) { re[u] = Ar[b0 + u][a]; im[u] = Ai[b0 + u][a]; }
  store4(D + ((size_t)J * TB + a) * bp + I * TB + b0, re);
  store4(D + bp * bp + ((size_t)J * TB + a) * bp + I * TB + b0, im);
}

// A whole merge of boxes whose separator fits one tile, in one launch: X, W
// and the update C, a workgroup per box. The border rows U = F_sb of all column
// tiles wait in LDS (dynamic, nb tiles after the fixed part), so the children
// are read once; C's own children entries are fetched while the matrix cores
// form U^T W. Rows beyond the separator and the border are not written.
// Bound by the instructions around its short products (indices, the inverse):
// 512^2 complex64, boxes of 7 x 7, 15 x 7, 15 x 15 and 31 x 15: 148, 109, 67 and
// 53 us as a launch each for the front, the step and the update, 67, 65, 45 and
// 42 us here; 768^2 FP64, 11 x 5 and 11 x 11: 239 and 270 us.
// A: F_ss, then P, then C_IJ on its way out; B: W_J.
template <typename T>
__global__ void __launch_bounds__(NT, 2) k_nd_merge(NdLevel L, NdBands<T> bd, const T *__restrict__ Cin, T *__restrict__ X,
                                                 T *__restrict__ W, T *__restrict__ Cout, int *status) {
  extern __shared__ __align__(16) unsigned char nd_smem[];
  NdLds2<T> &M = *reinterpret_cast<NdLds2<T> *>(nd_smem);
  typedef T Tile[2][TB][TBP];
  Tile *U = reinterpret_cast<Tile *>(nd_smem + sizeof(NdLds2<T>));
  const int box = nd_item(blockIdx.x, L.nbox);
  if (box < 0) return;
  const int nb = L.bp / TB;
  const NdBox B = nd_box(L, box);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, qi = wv >> 1, qj = wv & 1;
  const int a = tid >> 3, b0 = (tid & 7) * 4;
  int r0 = -1, r1 = -1, c0[4], c1[4];
  T re[4], im[4];
  if (a < B.s) nd_sep_map(L, B, a, r0, r1);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    c0[u] = c1[u] = -1;
    if (b0 + u < B.s) nd_sep_map(L, B, b0 + u, c0[u], c1[u]);
  }
  nd_children(L, B, Cin, r0, r1, c0, c1, re, im);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    T mr = a == b0 + u ? T(1) : T(0), mi = 0;
    if (a < B.s && b0 + u < B.s) nd_own_ss(L, B, bd, a, b0 + u, mr, mi);
    M.Ar[a][b0 + u] = re[u] + mr;
    M.Ai[a][b0 + u] = im[u] + mi;
  }
  for (int J = 0; J < nb; ++J) {
    const int j0 = J * TB + b0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      c0[u] = c1[u] = -1;
      if (j0 + u < B.b) nd_border_map(L, B, j0 + u, c0[u], c1[u]);
    }
    nd_children(L, B, Cin, r0, r1, c0, c1, re, im);
    if (a == 0 || a == B.s - 1)
#pragma unroll
      for (int u = 0; u < 4; ++u) nd_own_sb(L, B, bd, a, j0 + u, re[u], im[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) { U[J][0][a][b0 + u] = re[u]; U[J][1][a][b0 + u] = im[u]; }
  }
  __syncthreads();
  tile_inverse_pairs<T>(M, B.s, status);
  if (a < B.s) {
    T *D = X + (size_t)box * 2 * TB * TB + a * TB + b0;
    store4(D, &M.Ar[a][b0]);
    store4(D + TB * TB, &M.Ai[a][b0]);
  }
  // P as the left operand of W_J = P U_J, kept in registers: its tile becomes
  // the staging tile of C (cgemm_quad's order of the inner index)
  const int lr = lane & 15, k0 = (lane >> 5) + 16 * ((lane >> 4) & 1);
  T pr[8], pi[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) { pr[t] = M.Ar[qi * 16 + lr][2 * t + k0]; pi[t] = M.Ai[qi * 16 + lr][2 * t + k0]; }
  const size_t bp = L.bp, pb = TB * bp;
  T *C = Cout + (size_t)box * 2 * bp * bp;
  for (int J = 0; J < nb; ++J) {
    typename Mfma<T>::v4 wr = {0, 0, 0, 0}, wi = {0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const T br = U[J][0][2 * t + k0][qj * 16 + lr], bi = U[J][1][2 * t + k0][qj * 16 + lr];
      wr = Mfma<T>::mac(pr[t], br, wr);
      wr = Mfma<T>::mac(-pi[t], bi, wr);
      wi = Mfma<T>::mac(pr[t], bi, wi);
      wi = Mfma<T>::mac(pi[t], br, wi);
    }
    acc_to_lds<T>(wr, wi, M.Br, M.Bi, qi, qj, lane);
    int d0[4], d1[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      d0[u] = d1[u] = -1;
      if (J * TB + b0 + u < B.b) nd_border_map(L, B, J * TB + b0 + u, d0[u], d1[u]);
    }
    __syncthreads();   // W_J is in place (and, at J = 0, every wave has its P)
    if (a < B.s) {
      T *D = W + (size_t)box * 2 * pb + (size_t)a * bp + J * TB + b0;
      store4(D, &M.Br[a][b0]);
      store4(D + pb, &M.Bi[a][b0]);
    }
    for (int I = 0; I <= J; ++I) {
      int e0 = -1, e1 = -1;
      if (I * TB + a < B.b) nd_border_map(L, B, I * TB + a, e0, e1);
      nd_children(L, B, Cin, e0, e1, d0, d1, re, im);
      typename Mfma<T>::v4 cr = {0, 0, 0, 0}, ci = {0, 0, 0, 0};
      cgemm_quad_tn<T>(cr, ci, U[I][0], U[I][1], M.Br, M.Bi, qi, qj, lane, T(-1));
      acc_to_lds<T>(cr, ci, M.Ar, M.Ai, qi, qj, lane);
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        M.Ar[a][b0 + u] = re[u] += M.Ar[a][b0 + u];
        M.Ai[a][b0 + u] = im[u] += M.Ai[a][b0 + u];
      }
      __syncthreads();
      if (I == J) {   // a diagonal tile's lower triangle mirrors its upper one
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (b0 + u < a) { re[u] = M.Ar[b0 + u][a]; im[u] = M.Ai[b0 + u][a]; }
      }
      if (I * TB + a < B.b) {
        T *E = C + ((size_t)I * TB + a) * bp + J * TB + b0;
        store4(E, re);
        store4(E + bp * bp, im);
      }
      if (I != J && J * TB + a < B.b) {
#pragma unroll
        for (int u = 0; u < 4; ++u) { re[u] = M.Ar[b0 + u][a]; im[u] = M.Ai[b0 + u][a]; }
        T *E = C + ((size_t)J * TB + a) * bp + I * TB + b0;
        store4(E, re);
        store4(E + bp * bp, im);
      }
      __syncthreads();   // the tile is read before the next one replaces it
    }
  }
}
template <typename T>
inline size_t nd_merge_lds(const NdLevel &L) {
  return sizeof(NdLds2<T>) + (size_t)(L.bp / TB) * 2 * TB * TBP * sizeof(T);
}

template <typename T>
int nd_factor(const fdfd_grid *g, const double *op, void *factor, void *work, hipStream_t s) {
  const int prec = sizeof(T) == 8 ? FDFD_PREC_FP64 : FDFD_PREC_C64;
  NdPlan P;
  if (!nd_plan(g, &P)) return fail(FDFD_ERR_ARG, "the grid is outside the nested-dissection factor's range");
  const NdWork w = nd_work_layout(P, prec);
  char *base = (char *)work;
  double *tab = (double *)((char *)factor + ND_HEADER);
  T *data = (T *)((char *)factor + nd_data_off(P));
  int *status = (int *)base;
  const size_t M = (size_t)P.nx * P.ny;
  T *bands = (T *)(base + w.bands);
  NdStep<T> A;
  memset(&A, 0, sizeof A);
  A.bd = NdBands<T>{bands, bands + 2 * M, bands + 4 * M};
  A.U = (T *)(base + w.U);
  A.R = (T *)(base + w.R);
  A.status = status;
  T *C[2] = {(T *)(base + w.C[0]), (T *)(base + w.C[1])};
  T *S[2] = {(T *)(base + w.S[0]), (T *)(base + w.S[1])}, *Bf[2] = {(T *)(base + w.B[0]), (T *)(base + w.B[1])};
  T *pv[2] = {(T *)(base + w.pinv[0]), (T *)(base + w.pinv[1])};
  constexpr size_t lds = sizeof(NdLds2<T>) + nd_merge_tiles(sizeof(T)) * 2 * TB * TBP * sizeof(T);
  if constexpr (lds > LDS_DEFAULT) {   // FP64: 67.6 KB
    static std::atomic<uint64_t> done{0};
    if (int rc = grant_lds(done, {(const void *)k_nd_merge<T>}, lds, s)) return rc;
  }
  hipLaunchKernelGGL(k_nd_tables, dim3((std::max(P.nx + P.ny, 512) + NT - 1) / NT), dim3(NT), 0, s, *g,
                     (unsigned long long *)factor, tab, status, ND_HEADER + 32 * (size_t)(P.nx + P.ny),
                     nd_data_off(P), nd_data_off(P) + P.elems * sizeof(T), nd_factor_bytes(g, P, prec));
  hipLaunchKernelGGL(k_nd_bands<T>, dim3((P.ny + NT - 1) / NT, P.nx), dim3(NT), 0, s, P.nx, P.ny, nd_alpha(g), op,
                     nd_tables(tab, P.nx, P.ny), bands);
  hipLaunchKernelGGL(k_nd_leaf<T>, dim3(P.nleaf), dim3(64), 0, s, P.nx, P.ny, P.Dx, P.Dy, A.bd, data + P.leaf_off,
                     data + P.leafc_off, C[0], status);
  int cin = 0;
  for (int l = 0; l <= P.nlev; ++l) {
    const NdLevel &L = P.lev[l];
    const int ns = L.sp / TB, nb = L.bp / TB, per = ns * (ns + 1) / 2 + ns * nb;
    const int first = (L.nbox + XCDS - 1) / XCDS * XCDS;
    if (nd_merges(L, sizeof(T))) {
      hipLaunchKernelGGL(k_nd_merge<T>, dim3(nd_grid(L.nbox)), dim3(NT), nd_merge_lds<T>(L), s, L, A.bd,
                         (const T *)C[cin], data + L.xoff, data + L.woff, C[cin ^ 1], status);
      cin ^= 1;
      continue;
    }
    A.L = L;
    A.C = C[cin];
    A.Ds = S[1];
    A.P0 = pv[0];
    hipLaunchKernelGGL(k_nd_front<T>, dim3(first + nd_grid(L.nbox * (per - 1))), dim3(NT), 0, s, A);
    for (int p = 0; p < ns; ++p) {
      const bool last = p == ns - 1;
      A.p = p;
      A.Ss = S[(p + 1) & 1];
      A.Sb = p == 0 ? A.U : Bf[(p + 1) & 1];
      A.Ds = last ? data + L.xoff : S[p & 1];
      A.Db = last ? data + L.woff : Bf[p & 1];
      A.P0 = pv[p & 1];
      A.P1 = pv[(p + 1) & 1];
      hipLaunchKernelGGL(k_nd_step<T>, dim3((last ? 0 : first) + nd_grid(L.nbox * nd_step_items(ns, nb))),
                         dim3(NT), 0, s, A);
    }
    if (L.root) break;
    hipLaunchKernelGGL(k_nd_update<T>, dim3(nd_grid(L.nbox * (nb * (nb + 1) / 2))), dim3(NT), 0, s, L,
                       (const T *)C[cin], (const T *)A.U, (const T *)(ns > 1 ? A.R : data + L.woff), C[cin ^ 1]);
    cin ^= 1;
  }
  HIP_TRY(hipGetLastError());
  return FDFD_OK;
}

// -------------------------------------------------------------- solve
// Vectors of one pass of nq right-hand sides, complex T, right-hand sides
// innermost: f (the scaled right-hand side a E r) and v (z, then x, on the
// separators) by cell, u (a level's updates) by border entry. x is complex
// FP64 in the caller's planes.
//
// The levels whose separators fit one tile run as subtrees: one workgroup
// takes a box of level `top` with everything below it, a wave per box, with a
// barrier between levels instead of a launch. Its u live in two regions of
// its own, alternating by level (subtrees run at their own pace); level top
// writes u by box for the launches above.
constexpr int ND_TREE_MAX = 12;      // levels of a subtree
constexpr int ND_TREE_BOXES = 512;   // least subtrees, where the grid has them (see nd_tree)
constexpr int ND_TREE_WAVES = 8;
struct NdTree {
  int nx, ny, Dx, Dy, leaf_b, top, nq, add;
  unsigned reg0, reg1;               // entries of a subtree's two u regions
  NdLevel lev[ND_TREE_MAX];          // 0 .. top
};
template <typename T> struct NdVec {
  const double *iex, *iey;
  const T *data;                     // the factor's data
  const T *f;
  T *v;
  double *x;
  T *u0, *u1, *u2;
};

template <typename T>
__device__ inline void nd_out(const double *iex, const double *iey, double *x, size_t M, int i, int j, int ny, int q,
                              int add, T re, T im) {
  const cd o = cmul(cmul(ld_c(iex, i), ld_c(iey, j)), cd{(double)re, (double)im});
  double *xq = x + 2 * M * q;
  const size_t p = (size_t)i * ny + j;
  st_c(xq, p, add ? cadd(ld_c(xq, p), o) : o);
}
// cells as (i, j)
__device__ inline void nd_sep_ij(const NdLevel &L, const NdBox &B, int j, int &ci, int &cj) {
  if (L.root) {
    const int h = L.ny - 1, w = L.nx - 1;
    ci = j < h || j >= h + w ? 0 : j - h + 1;
    cj = j < h ? j + 1 : 0;
  } else if (L.ax == 0) {
    ci = B.x0 + B.c0;
    cj = B.y0 + j;
  } else {
    ci = B.x0 + j;
    cj = B.y0 + B.c0;
  }
}

// f_s of separator entry j, right-hand side q: f plus the children's updates
// (uin with the children's numbers n0, n1 in it)
template <typename T>
__device__ inline void nd_fs(const NdLevel &L, const NdBox &B, const T *f, const T *uin, int n0, int n1, int nq, int j,
                             int q, T &re, T &im) {
  int ci, cj, m0, m1;
  nd_sep_ij(L, B, j, ci, cj);
  nd_sep_map(L, B, j, m0, m1);
  T a = 0, b = 0, c = 0, d = 0;
  nd_ld(f, ((size_t)ci * L.ny + cj) * nq + q, re, im);
  if (m0 >= 0) nd_ld(uin, ((size_t)n0 * L.cb + m0) * nq + q, a, b);
  if (m1 >= 0) nd_ld(uin, ((size_t)n1 * L.cb + m1) * nq + q, c, d);
  re += a + c;
  im += b + d;
}
// the children's sum at border entry j
template <typename T>
__device__ inline void nd_fb(const NdLevel &L, const NdBox &B, const T *uin, int n0, int n1, int nq, int j, int q,
                             T &re, T &im) {
  int m0, m1;
  nd_border_map(L, B, j, m0, m1);
  T a = 0, b = 0, c = 0, d = 0;
  if (m0 >= 0) nd_ld(uin, ((size_t)n0 * L.cb + m0) * nq + q, a, b);
  if (m1 >= 0) nd_ld(uin, ((size_t)n1 * L.cb + m1) * nq + q, c, d);
  re = a + c;
  im = b + d;
}

// Upwards, one wave: columns 64 chunk .. + 64 of [X | W] of a box whose
// separator fits a tile. F: the wave's staging area.
template <typename T, int R>
__device__ inline void nd_up_wave(const NdTree &t, const NdVec<T> &A, const NdLevel &L, int box, int n0, int n1,
                                  const T *uin, T *uout, int chunk, T (*F)[R][2], int lane) {
  const NdBox B = nd_box(L, box);
  const int nq = t.nq;
  for (int e = lane; e < TB * R; e += 64) {
    const int j = e / R, q = e % R;
    T re = 0, im = 0;
    if (j < B.s && q < nq) nd_fs(L, B, A.f, uin, n0, n1, nq, j, q, re, im);
    F[j][q][0] = re;
    F[j][q][1] = im;
  }
  wave_lds_fence();
  const int c = chunk * 64 + lane;
  const bool inX = c < TB, inW = !inX && c < TB + L.bp;
  if (inX || inW) {
    const int pitch = inX ? TB : L.bp;
    const size_t plane = (size_t)TB * pitch;
    const T *m = A.data + (inX ? L.xoff + (size_t)box * 2 * plane + c : L.woff + (size_t)box * 2 * plane + c - TB);
    T ar[R], ai[R];
#pragma unroll
    for (int q = 0; q < R; ++q) { ar[q] = 0; ai[q] = 0; }
#pragma unroll 4
    for (int j = 0; j < B.s; ++j) {
      const T gr = m[(size_t)j * pitch], gi = m[plane + (size_t)j * pitch];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const T fr = F[j][q][0], fi = F[j][q][1];
        ar[q] += gr * fr - gi * fi;
        ai[q] += gr * fi + gi * fr;
      }
    }
    if (c < B.s) {
      int ci, cj;
      nd_sep_ij(L, B, c, ci, cj);
      const size_t at = ((size_t)ci * L.ny + cj) * nq;
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (q < nq) nd_st<T>(A.v, at + q, ar[q], ai[q]);
    } else if (inW && c - TB < B.b) {
      const int j = c - TB;
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (q < nq) {
          T ur, ui;
          nd_fb(L, B, uin, n0, n1, nq, j, q, ur, ui);
          nd_st<T>(uout, (size_t)j * nq + q, ur - ar[q], ui - ai[q]);
        }
    }
  }
  wave_lds_fence();
}

// Downwards, one wave: x_s = z - W x_b of a box whose separator fits a tile.
// The lanes are RP rows x 64 / RP groups of columns; a lane reads its row of W
// in 16-byte pieces.
template <typename T, int R, int RP>
__device__ inline void nd_down_wave(const NdTree &t, const NdVec<T> &A, const NdLevel &L, int box, T (*XB)[R][2],
                                    int lane) {
  constexpr int G = 64 / RP;
  const NdBox B = nd_box(L, box);
  const int nq = t.nq, row = lane & (RP - 1), g = lane / RP;
  const size_t plane = (size_t)TB * L.bp;
  const T *W = A.data + L.woff + (size_t)box * 2 * plane + (size_t)row * L.bp;
  T ar[R], ai[R];
#pragma unroll
  for (int q = 0; q < R; ++q) { ar[q] = 0; ai[q] = 0; }
  for (int b0 = 0; b0 < L.b; b0 += 64) {
    wave_lds_fence();
    for (int e = lane; e < 64 * R; e += 64) {
      const int c = e / R, q = e % R;
      T xr = 0, xi = 0;
      if (b0 + c < B.b && q < nq)
        nd_ld(A.v, nd_border_cell(L.nx, L.ny, L.dx, L.dy, B, b0 + c) * nq + q, xr, xi);
      XB[c][q][0] = xr;
      XB[c][q][1] = xi;
    }
    wave_lds_fence();
#pragma unroll 2
    for (int c = 4 * g; c < 64; c += 4 * G) {
      if (b0 + c >= L.bp) break;
      T gr[4], gi[4];
      ld_row4(W + b0 + c, gr);
      ld_row4(W + plane + b0 + c, gi);
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const T xr = XB[c + k][q][0], xi = XB[c + k][q][1];
          ar[q] += gr[k] * xr - gi[k] * xi;
          ai[q] += gr[k] * xi + gi[k] * xr;
        }
    }
  }
#pragma unroll
  for (int off = RP; off < 64; off <<= 1)
#pragma unroll
    for (int q = 0; q < R; ++q) {
      ar[q] += __shfl_xor(ar[q], off);
      ai[q] += __shfl_xor(ai[q], off);
    }
  if (row < B.s) {
    int ci, cj;
    nd_sep_ij(L, B, row, ci, cj);
    const size_t at = ((size_t)ci * L.ny + cj) * nq;
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (q % G == g % R && q < nq) {   // the groups share the right-hand sides
        if (G > R && g >= R) continue;
        T zr, zi;
        nd_ld(A.v, at + q, zr, zi);
        zr -= ar[q];
        zi -= ai[q];
        nd_st<T>(A.v, at + q, zr, zi);
        nd_out(A.iex, A.iey, A.x, (size_t)L.nx * L.ny, ci, cj, L.ny, q, t.add, zr, zi);
      }
  }
}

// A leaf, one wave: X is symmetric, so lane c of each half wave sums its
// column over half of the rows. Upwards z = X f and the updates -c_a z[p_a];
// downwards x = X (f - F_sb x_b).
template <typename T, int R, bool DOWN>
__device__ inline void nd_leaf_wave(const NdTree &t, const NdVec<T> &A, const T *X, const T *cpl, int k, T *uout,
                                    T (*F)[R][2], int lane) {
  const int nq = t.nq, nx = t.nx, ny = t.ny, c = lane & 31, half = lane >> 5;
  const int ix = k >> t.Dy, iy = k & ((1 << t.Dy) - 1);
  int x0, w, y0, h;
  nd_seg(nx, t.Dx, ix, x0, w);
  nd_seg(ny, t.Dy, iy, y0, h);
  const int s = w * h, b = 2 * (w + h);
  const T *cp = cpl + (size_t)k * TB * 2;
  const T *Xk = X + (size_t)k * 2 * TB * TB + c;
  const int sh = (s + 1) >> 1, ja = half * sh, jb = half ? s : sh;
  wave_lds_fence();
  for (int e = lane; e < TB * R; e += 64) {
    const int j = e / R, q = e % R;
    T fr = 0, fi = 0;
    if (j < s && q < nq) {
      const int ci = j / h, cj = j - ci * h;
      const size_t cell = (size_t)(x0 + ci) * ny + y0 + cj;
      nd_ld(A.f, cell * nq + q, fr, fi);
      if (DOWN) {
        // the border neighbours of an edge cell (entry order L, R, B, T)
        auto take = [&](int en, size_t nb) {
          T cr, cim, xr, xi;
          nd_ld(cp, en, cr, cim);
          nd_ld((const T *)A.v, nb * nq + q, xr, xi);
          fr -= cr * xr - cim * xi;
          fi -= cr * xi + cim * xr;
        };
        if (ci == 0) take(cj, cell - ny);
        if (ci == w - 1) take(h + cj, x0 + w == nx ? (size_t)(y0 + cj) : cell + ny);
        if (cj == 0) take(2 * h + ci, cell - 1);
        if (cj == h - 1) take(2 * h + w + ci, y0 + h == ny ? (size_t)(x0 + ci) * ny : cell + 1);
      }
    }
    F[j][q][0] = fr;
    F[j][q][1] = fi;
  }
  wave_lds_fence();
  T ar[R], ai[R];
#pragma unroll
  for (int q = 0; q < R; ++q) { ar[q] = 0; ai[q] = 0; }
#pragma unroll 4
  for (int j = ja; j < jb; ++j) {
    const T gr = Xk[j * TB], gi = Xk[TB * TB + j * TB];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const T fr = F[j][q][0], fi = F[j][q][1];
      ar[q] += gr * fr - gi * fi;
      ai[q] += gr * fi + gi * fr;
    }
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    ar[q] += __shfl_xor(ar[q], 32);
    ai[q] += __shfl_xor(ai[q], 32);
  }
  if (DOWN) {
    if (c < s) {
      const int ci = c / h, cj = c - ci * h;
#pragma unroll
      for (int q = 0; q < R; ++q)
        if ((R == 1 ? half == 0 : half == (q & 1)) && q < nq)
          nd_out(A.iex, A.iey, A.x, (size_t)nx * ny, x0 + ci, y0 + cj, ny, q, t.add, ar[q], ai[q]);
    }
    return;
  }
  wave_lds_fence();
  if (half == 0)
#pragma unroll
    for (int q = 0; q < R; ++q) { F[c][q][0] = ar[q]; F[c][q][1] = ai[q]; }
  wave_lds_fence();
  for (int e = lane; e < b * R; e += 64) {
    const int a = e / R, q = e % R;
    if (q >= nq) continue;
    const int p = a < h ? a : a < 2 * h ? (w - 1) * h + a - h : a < 2 * h + w ? (a - 2 * h) * h
                                                                 : (a - 2 * h - w) * h + h - 1;
    T cr, cim;
    nd_ld(cp, a, cr, cim);
    const T zr = F[p][q][0], zi = F[p][q][1];
    nd_st<T>(uout, (size_t)a * nq + q, -(cr * zr - cim * zi), -(cr * zi + cim * zr));
  }
}

// Box n of level L inside the subtree rooted at box (ix, iy) of level Lt
__device__ inline int nd_sub_box(const NdLevel &Lt, int ix, int iy, int dx, int dy, int n) {
  const int ex = dx - Lt.dx, ey = dy - Lt.dy;
  return (((ix << ex) + (n >> ey)) << dy) + (iy << ey) + (n & ((1 << ey) - 1));
}

template <typename T, int R>
__global__ void __launch_bounds__(64 * ND_TREE_WAVES) k_nd_up_tree(NdTree t, NdVec<T> A, const T *__restrict__ X,
                                                                   const T *__restrict__ cpl) {
  __shared__ __align__(16) T F[ND_TREE_WAVES][TB][R][2];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const NdLevel &Lt = t.lev[t.top];
  const int root = blockIdx.x, ix = root >> Lt.dy, iy = root & ((1 << Lt.dy) - 1);
  T *reg[2] = {A.u0 + (size_t)2 * t.reg0 * t.nq * root, A.u1 + (size_t)2 * t.reg1 * t.nq * root};
  const int nleaf = 1 << (t.Dx - Lt.dx + t.Dy - Lt.dy);
  for (int n = wv; n < nleaf; n += ND_TREE_WAVES)
    nd_leaf_wave<T, R, false>(t, A, X, cpl, nd_sub_box(Lt, ix, iy, t.Dx, t.Dy, n),
                              reg[0] + (size_t)2 * n * t.leaf_b * t.nq, F[wv], lane);
  for (int l = 0; l <= t.top; ++l) {
    __syncthreads();
    const NdLevel &L = t.lev[l];
    const int ey = L.dy - Lt.dy, count = 1 << (L.dx - Lt.dx + ey), chunks = (TB + L.bp + 63) / 64;
    for (int it = wv; it < count * chunks; it += ND_TREE_WAVES) {
      const int n = it / chunks, a = n >> ey, b = n & ((1 << ey) - 1);
      const int n0 = L.ax == 0 ? ((2 * a) << ey) + b : (a << (ey + 1)) + 2 * b;
      const int n1 = L.ax == 0 ? n0 + (1 << ey) : n0 + 1;
      T *uout = l == t.top ? A.u2 + (size_t)2 * root * L.b * t.nq : reg[(l + 1) & 1] + (size_t)2 * n * L.b * t.nq;
      nd_up_wave<T, R>(t, A, L, nd_sub_box(Lt, ix, iy, L.dx, L.dy, n), n0, n1, reg[l & 1], uout, it % chunks, F[wv],
                       lane);
    }
  }
}
template <typename T, int R>
__global__ void __launch_bounds__(64 * ND_TREE_WAVES) k_nd_down_tree(NdTree t, NdVec<T> A, const T *__restrict__ X,
                                                                     const T *__restrict__ cpl) {
  __shared__ __align__(16) T F[ND_TREE_WAVES][64][R][2];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const NdLevel &Lt = t.lev[t.top];
  const int root = blockIdx.x, ix = root >> Lt.dy, iy = root & ((1 << Lt.dy) - 1);
  for (int l = t.top; l >= 0; --l) {
    const NdLevel &L = t.lev[l];
    const int count = 1 << (L.dx - Lt.dx + L.dy - Lt.dy);
    for (int n = wv; n < count; n += ND_TREE_WAVES) {
      const int box = nd_sub_box(Lt, ix, iy, L.dx, L.dy, n);
      if (L.s <= 8) nd_down_wave<T, R, 8>(t, A, L, box, F[wv], lane);
      else if (L.s <= 16) nd_down_wave<T, R, 16>(t, A, L, box, F[wv], lane);
      else nd_down_wave<T, R, 32>(t, A, L, box, F[wv], lane);
    }
    __syncthreads();
  }
  const int nleaf = 1 << (t.Dx - Lt.dx + t.Dy - Lt.dy);
  for (int n = wv; n < nleaf; n += ND_TREE_WAVES)
    nd_leaf_wave<T, R, true>(t, A, X, cpl, nd_sub_box(Lt, ix, iy, t.Dx, t.Dy, n), nullptr, F[wv], lane);
}

// Upwards, one level above the subtrees (and the root, whose z is x): 32
// columns of [X | W] of one box per workgroup, the separator's rows spread
// over its half waves, UN at a time. These matrix rows do not depend on f:
// their loads go out before f is gathered, so a batch of 2 NW UN rows costs one
// trip to memory. Bound by the latencies of one launch: 512^2 complex64 with 4
// right-hand sides, the root's 1023 rows 20.6 -> 15 us, the levels below it
// 12.5 .. 7 -> 10 .. 6 us against rows loaded four at a time after f; a solve of
// three sweeps 1.05 -> 0.99 ms, of one (512^2 FP64, one right-hand side) 0.42 ->
// 0.35 ms. The caller's NW and UN make one batch of a separator up to 512
// rows; larger batches than the separator needs would load rows for nothing.
template <typename T, int R, int NW, int UN>
__global__ void __launch_bounds__(64 * NW) k_nd_up(NdLevel L, NdVec<T> A, const T *__restrict__ uin,
                                                   T *__restrict__ uout, int nq, int add) {
  constexpr int RG = 2 * NW, JC = RG * UN;
  __shared__ __align__(16) union {
    T f[JC][R][2];
    T red[NW][2 * R][32];
  } S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c32 = tid & 31, rg = tid >> 5;
  const int chunks = (L.sp + L.bp) / 32, box = blockIdx.x / chunks, c = (blockIdx.x % chunks) * 32 + c32;
  const NdBox B = nd_box(L, box);
  const bool inX = c < L.sp;
  const int pitch = inX ? L.sp : L.bp;
  const size_t plane = (size_t)L.sp * pitch;
  const T *m = A.data + (inX ? L.xoff + (size_t)box * 2 * plane + c : L.woff + (size_t)box * 2 * plane + c - L.sp);
  T ar[R], ai[R];
#pragma unroll
  for (int q = 0; q < R; ++q) { ar[q] = 0; ai[q] = 0; }
  for (int j0 = 0; j0 < B.s; j0 += JC) {
    T gr[UN], gi[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) {   // past the separator: its last row, against f = 0
      const T *row = m + (size_t)min(j0 + rg + u * RG, B.s - 1) * pitch;
      gr[u] = row[0];
      gi[u] = row[plane];
    }
    if (j0) __syncthreads();
    for (int e = tid; e < JC * R; e += 64 * NW) {
      const int j = e / R, q = e % R;
      T re = 0, im = 0;
      if (j0 + j < B.s && q < nq) nd_fs(L, B, A.f, uin, B.k0, B.k1, nq, j0 + j, q, re, im);
      S.f[j][q][0] = re;
      S.f[j][q][1] = im;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const T fr = S.f[rg + u * RG][q][0], fi = S.f[rg + u * RG][q][1];
        ar[q] += gr[u] * fr - gi[u] * fi;
        ai[q] += gr[u] * fi + gi[u] * fr;
      }
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    ar[q] += __shfl_xor(ar[q], 32);
    ai[q] += __shfl_xor(ai[q], 32);
  }
  __syncthreads();
  if (lane < 32)
#pragma unroll
    for (int q = 0; q < R; ++q) {
      S.red[wv][2 * q][c32] = ar[q];
      S.red[wv][2 * q + 1][c32] = ai[q];
    }
  __syncthreads();
  for (int e = tid; e < 32 * R; e += 64 * NW) {
    const int cc = e & 31, q = e >> 5, col = (blockIdx.x % chunks) * 32 + cc;
    if (q >= nq) continue;
    T sr = 0, si = 0;
#pragma unroll
    for (int g = 0; g < NW; ++g) { sr += S.red[g][2 * q][cc]; si += S.red[g][2 * q + 1][cc]; }
    if (col < B.s) {
      int ci, cj;
      nd_sep_ij(L, B, col, ci, cj);
      nd_st<T>(A.v, ((size_t)ci * L.ny + cj) * nq + q, sr, si);
      if (L.root) nd_out(A.iex, A.iey, A.x, (size_t)L.nx * L.ny, ci, cj, L.ny, q, add, sr, si);
    } else if (col >= L.sp && col - L.sp < B.b) {
      T ur, ui;
      nd_fb(L, B, uin, B.k0, B.k1, nq, col - L.sp, q, ur, ui);
      nd_st<T>(uout, ((size_t)box * L.b + col - L.sp) * nq + q, ur - sr, ui - si);
    }
  }
}

// Downwards, one level above the subtrees: 16 rows of W of one box per
// workgroup; a lane reads its row in 16-byte pieces, the columns spread over
// the quarter waves, UN pieces at a time and before x is gathered, as in k_nd_up.
constexpr int ND_DOWN_WAVES = 8;
template <typename T, int R, int UN>
__global__ void __launch_bounds__(64 * ND_DOWN_WAVES) k_nd_down(NdLevel L, NdVec<T> A, int nq, int add) {
  constexpr int GROUPS = 4 * ND_DOWN_WAVES, CC = 4 * GROUPS * UN;
  __shared__ __align__(16) union {
    T x[CC][R][2];
    T red[ND_DOWN_WAVES][2 * R][16];
  } S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r16 = lane & 15, grp = wv * 4 + (lane >> 4);
  const int groups = (L.s + 15) / 16, box = blockIdx.x / groups, row = (blockIdx.x % groups) * 16 + r16;
  const NdBox B = nd_box(L, box);
  const size_t plane = (size_t)L.sp * L.bp;
  const T *W = A.data + L.woff + (size_t)box * 2 * plane + (size_t)row * L.bp;
  T ar[R], ai[R];
#pragma unroll
  for (int q = 0; q < R; ++q) { ar[q] = 0; ai[q] = 0; }
  for (int b0 = 0; b0 < B.b; b0 += CC) {
    T gr[UN][4], gi[UN][4];
#pragma unroll
    for (int u = 0; u < UN; ++u) {   // past the border: its last piece, against x = 0
      const int c = min(b0 + 4 * (grp + u * GROUPS), L.bp - 4);
      ld_row4(W + c, gr[u]);
      ld_row4(W + plane + c, gi[u]);
    }
    if (b0) __syncthreads();
    constexpr int TS = 64 * ND_DOWN_WAVES, G = (CC * R + TS - 1) / TS;
    T xr[G], xi[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int e = tid + u * TS, q = min(e % R, nq - 1);
      nd_ld((const T *)A.v, nd_border_cell(L.nx, L.ny, L.dx, L.dy, B, min(b0 + e / R, B.b - 1)) * nq + q, xr[u], xi[u]);
    }
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int e = tid + u * TS, c = e / R, q = e % R;
      if (CC * R < TS && e >= CC * R) break;
      const bool has = b0 + c < B.b && q < nq;
      S.x[c][q][0] = has ? xr[u] : T(0);
      S.x[c][q][1] = has ? xi[u] : T(0);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const int c = 4 * (grp + u * GROUPS) + k;
          const T xr = S.x[c][q][0], xi = S.x[c][q][1];
          ar[q] += gr[u][k] * xr - gi[u][k] * xi;
          ai[q] += gr[u][k] * xi + gi[u][k] * xr;
        }
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    ar[q] += __shfl_xor(ar[q], 16);
    ai[q] += __shfl_xor(ai[q], 16);
    ar[q] += __shfl_xor(ar[q], 32);
    ai[q] += __shfl_xor(ai[q], 32);
  }
  __syncthreads();
  if (lane < 16)
#pragma unroll
    for (int q = 0; q < R; ++q) {
      S.red[wv][2 * q][r16] = ar[q];
      S.red[wv][2 * q + 1][r16] = ai[q];
    }
  __syncthreads();
  for (int e = tid; e < 16 * R; e += 64 * ND_DOWN_WAVES) {
    const int r = e & 15, q = e >> 4, j = (blockIdx.x % groups) * 16 + r;
    if (q >= nq || j >= B.s) continue;
    T sr = 0, si = 0;
#pragma unroll
    for (int w = 0; w < ND_DOWN_WAVES; ++w) { sr += S.red[w][2 * q][r]; si += S.red[w][2 * q + 1][r]; }
    int ci, cj;
    nd_sep_ij(L, B, j, ci, cj);
    const size_t at = ((size_t)ci * L.ny + cj) * nq + q;
    T zr, zi;
    nd_ld((const T *)A.v, at, zr, zi);
    zr -= sr;
    zi -= si;
    nd_st<T>(A.v, at, zr, zi);
    nd_out(A.iex, A.iey, A.x, (size_t)L.nx * L.ny, ci, cj, L.ny, q, add, zr, zi);
  }
}

// right-hand sides of one pass over the factor
template <typename T> constexpr int nd_rhs_per_pass() { return sizeof(T) == 8 ? 4 : 8; }

// The residual v = b' - A x with b' = b, or D^-1 b in the transposed solve,
// scaled into f (a E v, by pass), and per right-hand side the partial sums of
// |v|^2 (weighted by |D|^2 in the transposed solve). A null x: v = b' and the
// partial sums of |b|^2. Blocks take every gridDim.x-th piece of a row.
constexpr int ND_RES_RHS = 4;     // right-hand sides per thread (grid.y passes)
template <typename T>
__global__ void __launch_bounds__(NT) k_nd_residual(fdfd_grid g, double alpha, NdTab tb, const double *__restrict__ op,
                                                    const double *__restrict__ b, const double *__restrict__ x,
                                                    T *__restrict__ f, int nrhs, int transpose,
                                                    double *__restrict__ part) {
  __shared__ double red[ND_RES_RHS][NT];
  constexpr int most = nd_rhs_per_pass<T>();
  const int nx = g.nx, ny = g.ny, tid = threadIdx.x, q0 = blockIdx.y * ND_RES_RHS;
  const int nq = min(ND_RES_RHS, nrhs - q0), cpr = (ny + NT - 1) / NT;
  const int pass = q0 / most, per = min(most, nrhs - pass * most), at = q0 - pass * most;
  const size_t M = (size_t)nx * ny;
  T *fp = f + 2 * M * (size_t)pass * most;
  double acc[ND_RES_RHS] = {0, 0, 0, 0};
  for (int piece = blockIdx.x; piece < nx * cpr; piece += gridDim.x) {
    const int i = piece / cpr, j = (piece - i * cpr) * NT + tid;
    if (j >= ny) continue;
    const size_t p = (size_t)i * ny + j;
    cd dinv = {1, 0};
    double w2 = 1;
    if (transpose) {
      const double hx = ((double)nx * g.dl) / nx, hy = ((double)ny * g.dl) / ny;
      const cd d = cmul(sfactor(0, i, nx, g.npml_x, hx, g.omega, g.L0), sfactor(0, j, ny, g.npml_y, hy, g.omega, g.L0));
      dinv = cinv(d);
      w2 = d.r * d.r + d.i * d.i;
    }
    const cd e = cscale(cmul(ld_c(tb.ex, i), ld_c(tb.ey, j)), alpha);
    if (!x) {
#pragma unroll
      for (int q = 0; q < ND_RES_RHS; ++q)
        if (q < nq) {
          cd v = ld_c(b + 2 * M * (q0 + q), p);
          acc[q] += v.r * v.r + v.i * v.i;
          if (transpose) v = cmul(v, dinv);
          v = cmul(e, v);
          nd_st<T>(fp, p * per + at + q, (T)v.r, (T)v.i);
        }
      continue;
    }
    const size_t pxm = (i == 0 ? p + M - ny : p - ny), pxp = (i + 1 == nx ? p + ny - M : p + ny);
    const size_t pym = (j == 0 ? p + ny - 1 : p - 1), pyp = (j + 1 == ny ? p + 1 - ny : p + 1);
    const cd c0 = ld_c(op, FDFD_OP_C * M + p), cxm = ld_c(op, FDFD_OP_XM * M + p), cxp = ld_c(op, FDFD_OP_XP * M + p);
    const cd cym = ld_c(op, FDFD_OP_YM * M + p), cyp = ld_c(op, FDFD_OP_YP * M + p);
#pragma unroll
    for (int q = 0; q < ND_RES_RHS; ++q)
      if (q < nq) {
        const double *xq = x + 2 * M * (q0 + q);
        cd a = cmul(c0, ld_c(xq, p));
        a = cadd(a, cmul(cxm, ld_c(xq, pxm)));
        a = cadd(a, cmul(cxp, ld_c(xq, pxp)));
        a = cadd(a, cmul(cym, ld_c(xq, pym)));
        a = cadd(a, cmul(cyp, ld_c(xq, pyp)));
        cd v = ld_c(b + 2 * M * (q0 + q), p);
        if (transpose) v = cmul(v, dinv);
        v = csub(v, a);
        acc[q] += w2 * (v.r * v.r + v.i * v.i);
        v = cmul(e, v);
        nd_st<T>(fp, p * per + at + q, (T)v.r, (T)v.i);
      }
  }
#pragma unroll
  for (int q = 0; q < ND_RES_RHS; ++q) red[q][tid] = acc[q];
  __syncthreads();
  for (int st = NT / 2; st > 0; st >>= 1) {
    if (tid < st)
#pragma unroll
      for (int q = 0; q < ND_RES_RHS; ++q) red[q][tid] += red[q][tid + st];
    __syncthreads();
  }
  if (tid < nq) part[(size_t)(q0 + tid) * gridDim.x + blockIdx.x] = red[tid][0];
}

// The subtrees of a plan: the levels whose separators fit a tile, as far up as
// leaves ND_TREE_BOXES of them (two workgroups of eight waves per CU), a number
// measured on one grid and taken for all: smaller ones, with fewer boxes a
// level, have more of their levels above the subtrees. 512^2
// complex64, a solve of 4 / 8 right-hand sides in three sweeps: 1469 / 2259 us
// with 128 subtrees (half of the CUs idle), 1164 / 1735 with 256, 1042 / 1552
// with 512, 1146 / 1683 with 1024 and 1311 / 1945 with 2048 (more launches
// above); a launch per level for all of them took 1850 / 3610.
inline NdTree nd_tree(const NdPlan &P) {
  NdTree t;
  memset(&t, 0, sizeof t);
  t.nx = P.nx; t.ny = P.ny; t.Dx = P.Dx; t.Dy = P.Dy; t.leaf_b = P.leaf_b;
  while (t.top + 1 < P.nlev && t.top + 1 < ND_TREE_MAX && P.lev[t.top + 1].sp <= TB &&
         P.lev[t.top + 1].nbox >= ND_TREE_BOXES)
    ++t.top;
  const NdLevel &Lt = P.lev[t.top];
  t.reg0 = (unsigned)((P.nleaf / Lt.nbox) * P.leaf_b);
  for (int l = 0; l <= t.top; ++l) {
    t.lev[l] = P.lev[l];
    const unsigned n = (unsigned)(P.lev[l].nbox / Lt.nbox * P.lev[l].b);
    if (l < t.top) {
      if (l & 1) t.reg0 = std::max(t.reg0, n);
      else t.reg1 = std::max(t.reg1, n);
    }
  }
  // the levels above alternate between the same buffers, whole
  for (int l = t.top + 1; l < P.nlev; ++l) {
    const unsigned n = (unsigned)((P.lev[l].nbox * (size_t)P.lev[l].b + Lt.nbox - 1) / Lt.nbox);
    if ((l - t.top) & 1) t.reg0 = std::max(t.reg0, n);
    else t.reg1 = std::max(t.reg1, n);
  }
  return t;
}
// Solve workspace: f of every right-hand side, v and the u buffers of one
// pass, norm partials, norms (`base` bytes), and an iterate within the
// tolerance (nd_solve).
struct NdSolveWork {
  size_t f, v, u[3], part, norms, base, kept, total;
};
inline NdSolveWork nd_solve_layout(const NdPlan &P, int precision, int nrhs) {
  const size_t M = (size_t)P.nx * P.ny, es = elem_size(precision);
  const size_t R = std::min(nrhs, es == 8 ? nd_rhs_per_pass<double>() : nd_rhs_per_pass<float>());
  const NdTree t = nd_tree(P);
  const NdLevel &Lt = P.lev[t.top];
  NdSolveWork w;
  size_t off = 0;
  auto take = [&](size_t bytes) { const size_t at = off; off += align_up(bytes, 256); return at; };
  w.f = take(2 * es * M * nrhs);
  w.v = take(2 * es * M * R);
  w.u[0] = take(2 * es * R * t.reg0 * Lt.nbox);
  w.u[1] = take(2 * es * R * t.reg1 * Lt.nbox);
  w.u[2] = take(2 * es * R * Lt.b * Lt.nbox);
  w.part = take(8 * (size_t)2 * NORM_PARTS * nrhs);
  w.norms = take(8 * 3 * (size_t)nrhs);
  w.base = off;
  w.kept = take(16 * M * nrhs);
  w.total = off;
  return w;
}

// x (+)= E^-1 M^-1 f for one pass
template <typename T, int R>
int nd_pass(const NdPlan &P, NdTree &t, const NdVec<T> &A, int nq, int add, hipStream_t s) {
  t.nq = nq;
  t.add = add;
  const T *X = A.data + P.leaf_off, *cpl = A.data + P.leafc_off;
  const int sub = P.lev[t.top].nbox;
  hipLaunchKernelGGL((k_nd_up_tree<T, R>), dim3(sub), dim3(64 * ND_TREE_WAVES), 0, s, t, A, X, cpl);
  T *uin = A.u2, *uout = A.u0;
  for (int l = t.top + 1; l <= P.nlev; ++l) {
    const NdLevel &L = P.lev[l];
    const int grid = L.nbox * ((L.sp + L.bp) / 32);
    const auto up = L.s <= 64 ? k_nd_up<T, R, 4, 8> : L.s <= 128 ? k_nd_up<T, R, 4, 16>
                  : L.s <= 256 ? k_nd_up<T, R, 8, 16> : k_nd_up<T, R, 16, 16>;
    hipLaunchKernelGGL(up, dim3(grid), dim3(L.s <= 128 ? 256 : L.s <= 256 ? 512 : 1024), 0, s, L, A, uin, uout, nq, add);
    uin = uout;
    uout = uin == A.u0 ? A.u1 : A.u0;
  }
  for (int l = P.nlev - 1; l > t.top; --l) {
    const NdLevel &L = P.lev[l];
    const auto down = L.b <= 256 ? k_nd_down<T, R, 2> : L.b <= 512 || sizeof(T) == 8 ? k_nd_down<T, R, 4>
                                                      : k_nd_down<T, R, 8>;
    hipLaunchKernelGGL(down, dim3(L.nbox * ((L.s + 15) / 16)), dim3(64 * ND_DOWN_WAVES), 0, s, L, A, nq, add);
  }
  hipLaunchKernelGGL((k_nd_down_tree<T, R>), dim3(sub), dim3(64 * ND_TREE_WAVES), 0, s, t, A, X, cpl);
  HIP_TRY(hipGetLastError());
  return FDFD_OK;
}
// x (+)= E^-1 M^-1 f, f as k_nd_residual leaves it
template <typename T>
int nd_sweep(const NdPlan &P, const void *factor, double *x, int nrhs, int add, char *work, const NdSolveWork &w,
             hipStream_t s) {
  const NdTab tb = nd_tables((const double *)((const char *)factor + ND_HEADER), P.nx, P.ny);
  const size_t M = (size_t)P.nx * P.ny;
  NdTree t = nd_tree(P);
  constexpr int most = nd_rhs_per_pass<T>();
  for (int q0 = 0; q0 < nrhs; q0 += most) {
    const int nq = std::min(most, nrhs - q0);
    const NdVec<T> A{tb.iex, tb.iey, (const T *)((const char *)factor + nd_data_off(P)),
                     (const T *)(work + w.f) + 2 * M * q0, (T *)(work + w.v), x + 2 * M * q0,
                     (T *)(work + w.u[0]), (T *)(work + w.u[1]), (T *)(work + w.u[2])};
    int rc = FDFD_OK;
    if (nq == 1) rc = nd_pass<T, 1>(P, t, A, nq, add, s);
    else if (nq == 2) rc = nd_pass<T, 2>(P, t, A, nq, add, s);
    else if (nq <= 4) rc = nd_pass<T, 4>(P, t, A, nq, add, s);
    else if constexpr (most >= 8) rc = nd_pass<T, 8>(P, t, A, nq, add, s);
    if (rc) return rc;
  }
  return FDFD_OK;
}

// The path's range: a plan exists and its solve fits the block path's
// workspace, which fdfd_solve_static is limited by (except the kept iterate,
// which that call does without where it has no room). FP64,
// new permittivity and solve / resident solve through Simulation, block path
// against tree: 16 x 16 1.13 / 0.60 against 0.52 / 0.29 ms, 32 x 32 1.26 /
// 0.60 against 0.64 / 0.32, 48 x 40 2.27 / 0.70 against 0.71 / 0.32, 63 x 63
// 3.21 / 1.13 against 0.80 / 0.35; below 16 cells a tree has hardly a level.
// Complex64 factors of grids with a side below 64 cells stay block factors:
// how far their refinement gets in a given number of steps, and that a
// singular leading pivot sends them to FP64, is what the fallback order is
// tested on. No measurement draws that line: a new permittivity and solve of
// 48 x 40 cells takes 2.15 ms there, 0.94 as a tree.
constexpr int ND_MIN_SIDE_C64 = 64;
inline bool nd_fits(const fdfd_grid *g, int precision, NdPlan *P) {
  const int prec = base_prec(precision);
  if (prec == FDFD_PREC_C64 && std::min(g->nx, g->ny) < ND_MIN_SIDE_C64) return false;
  if (!nd_plan(g, P)) return false;
  for (int k = 1; k <= 8; ++k)
    if (nd_solve_layout(*P, prec, k).base > solve_work_bytes(g, prec, k)) return false;
  return true;
}

// Grids too long for the tree to be the factor of choice. Its root front is the
// cross, of order nx + ny - 1 and eliminated whole: the factor's time grows
// with the cube of the long side and its memory with the square, the block
// chain's with the side itself. FP64 factor, tree against block path: 6144 x 16
// 36 against 58 ms, 8192 x 16 81 / 78 (5.7 GB against 0.13), 12288 x 16 266 /
// 117, 11584 x 64 230 / 326, 16384 x 64 632 / 462, 16384 x 128 645 / 776;
// complex64 11584 x 64 116 / 254, 16384 x 64 317 / 359. A chain's step costs
// about its block's tiles: the lines cross near a^2 = 2^21 b for a long side a
// and a short side padded to b.
inline bool nd_long(const fdfd_grid *g) {
  const size_t a = std::max(g->nx, g->ny), b = pad_n(std::min(g->nx, g->ny));
  return a * a > b << 21;
}

// The launch of k_nd_residual of a solve
template <typename T>
void nd_residual(const fdfd_grid *g, const NdPlan &P, const double *op, const void *factor, const double *b,
                 const double *x, int nrhs, int transpose, char *work, const NdSolveWork &w, int parts, hipStream_t s) {
  hipLaunchKernelGGL(k_nd_residual<T>, dim3(parts, (nrhs + ND_RES_RHS - 1) / ND_RES_RHS), dim3(NT), 0, s, *g,
                     nd_alpha(g), nd_tables((const double *)((const char *)factor + ND_HEADER), P.nx, P.ny), op, b, x,
                     (T *)(work + w.f), nrhs, transpose, (double *)(work + w.part));
}
inline int nd_parts(const NdPlan &P) { return std::min(2 * NORM_PARTS, P.nx * ((P.ny + NT - 1) / NT)); }

// The refinement of fdfd_solve with a nested-dissection factor: x = A^-1 b,
// then x += A^-1 (b - A x) until every right-hand side meets the tolerance.
// With a periodic axis a step is two sweeps, as on the block path. The first
// sweep starts before ||b|| is known on the host; a zero b gives x = 0. room:
// the workspace's bytes.
template <typename T>
int nd_solve(const fdfd_grid *g, const double *op, const void *factor, const double *b, double *x, int nrhs,
             int transpose, double tol, int max_iter, void *work, fdfd_solve_stats *stats, double *rel_res,
             hipStream_t s, double *host, size_t room) {
  const int prec = sizeof(T) == 8 ? FDFD_PREC_FP64 : FDFD_PREC_C64;
  NdPlan P;
  if (!nd_fits(g, prec, &P)) return fail(FDFD_ERR_ARG, "the grid is outside the nested-dissection factor's range");
  const NdSolveWork w = nd_solve_layout(P, prec, nrhs);
  char *base = (char *)work;
  double *part = (double *)(base + w.part), *norms = (double *)(base + w.norms);
  const int parts = nd_parts(P);
  auto residual = [&](const double *xi) { nd_residual<T>(g, P, op, factor, b, xi, nrhs, transpose, base, w, parts, s); };
  fdfd_solve_stats st;
  memset(&st, 0, sizeof st);
  double *nr = host, *nb = host + nrhs, *rel = host + 2 * nrhs, *prev = host + 3 * nrhs;
  for (int q = 0; q < nrhs; ++q) { rel[q] = 0.0; prev[q] = INFINITY; }
  residual(nullptr);
  hipLaunchKernelGGL(k_norm_final, dim3(nrhs), dim3(NT), 0, s, (const double *)part, parts, norms + nrhs);
  const int sweeps = wrap_exact(g) ? 2 : 1;
  // Which iterate within tol is the last. The first one can be a hundred times
  // as far from the solution as the block factor's, whose steps leave the wrap
  // coupling to a second one: what a sweep leaves lies in the directions that
  // A^-1 amplifies most. Errors of 246 drawn operators (40 to 640 cells a side)
  // against the block factor's at the same tol, as the mean of the ratio, its
  // maximum and how many are larger:
  //   FP64, tol 1e-12: one sweep 0.47, 184, 65; two 0.09, 1.4 (rounding), 9.
  //   complex64, tol 1e-12: first iterate below tol 0.19, 311, 57 of 205; one
  //   more from above tol/4 0.10, 46, 38; from above tol/100 0.02, 1.9, 4.
  //   complex64, tol 1e-10: 0.03, 1363, 43; 0.01, 85, 26; 0.004, 85, 12 (the
  //   85: a residual of tol/2 after eight sweeps).
  // So FP64 takes two sweeps at least, the first two without a look between
  // them, and complex64 one more from above tol/100 (0.1 to 0.6 sweeps a solve).
  // The iterate within tol is kept meanwhile: near the floor of the FP64
  // residual the next one may lie above tol, and is then taken back.
  const bool keeps = w.total <= room, pair = sizeof(T) == 8 && sweeps == 1 && max_iter > 1 && keeps;
  const auto enough = [&](double worst) { return sizeof(T) == 8 ? st.sweeps >= 2 : worst <= 0.01 * tol; };
  const auto relative = [](double r2, double b2) {
    const double v = b2 > 0 ? sqrt(r2 / b2) : 0.0;
    return std::isfinite(v) ? v : INFINITY;
  };
  const size_t xbytes = 16 * (size_t)P.nx * P.ny * nrhs;
  bool held = false, looked = false;
  int stall_count = 0;
  for (int it = 1; it <= max_iter; ++it) {
    for (int k = 0; k < sweeps; ++k) {
      const bool first = it == 1 && k == 0;
      if (int rc = nd_sweep<T>(P, factor, x, nrhs, first ? 0 : 1, base, w, s)) return rc;
      residual(x);
    }
    const bool unseen = pair && it == 1;   // its norms are read with the next ones
    hipLaunchKernelGGL(k_norm_final, dim3(nrhs), dim3(NT), 0, s, (const double *)part, parts,
                       norms + (unseen ? 2 * nrhs : 0));
    HIP_TRY(hipGetLastError());
    st.iterations = it;
    st.sweeps += sweeps;
    if (unseen) {
      HIP_TRY(hipMemcpyAsync(base + w.kept, x, xbytes, hipMemcpyDeviceToDevice, s));
      continue;
    }
    // nr, and at the first look nb and (in rel's place) the unseen iterate's
    HIP_TRY(hipMemcpyAsync(nr, norms, sizeof(double) * (looked ? 1 : pair ? 3 : 2) * nrhs, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    if (!looked) {
      looked = true;
      bool all_zero = true;
      for (int q = 0; q < nrhs; ++q) all_zero = all_zero && nb[q] == 0.0;
      if (all_zero) {   // linalg.py:128-129
        HIP_TRY(hipMemsetAsync(x, 0, xbytes, s));
        HIP_TRY(hipStreamSynchronize(s));
        memset(&st, 0, sizeof st);
        st.zero_rhs = 1;
        st.converged = 1;
        if (stats) *stats = st;
        if (rel_res) for (int q = 0; q < nrhs; ++q) rel_res[q] = 0;
        return FDFD_OK;
      }
      if (pair) {
        held = true;
        for (int q = 0; q < nrhs; ++q) {
          prev[q] = relative(rel[q], nb[q]);
          held = held && prev[q] <= tol;
        }
      }
    }
    double worst = 0;
    bool contracting = false;
    for (int q = 0; q < nrhs; ++q) {
      rel[q] = relative(nr[q], nb[q]);
      worst = std::max(worst, rel[q]);
      if (rel[q] > tol && rel[q] < 0.7 * prev[q]) contracting = true;
    }
    st.max_rel_residual = worst;
    if (worst <= tol) {
      st.converged = 1;
      if (enough(worst) || held || it == max_iter || !keeps) break;
      HIP_TRY(hipMemcpyAsync(base + w.kept, x, xbytes, hipMemcpyDeviceToDevice, s));
      held = true;
    } else if (held) {   // back to the iterate before
      st.converged = 1;
      HIP_TRY(hipMemcpyAsync(x, base + w.kept, xbytes, hipMemcpyDeviceToDevice, s));
      HIP_TRY(hipStreamSynchronize(s));
      st.max_rel_residual = 0;
      for (int q = 0; q < nrhs; ++q) st.max_rel_residual = std::max(st.max_rel_residual, rel[q] = prev[q]);
      break;
    } else {
      if (!std::isfinite(worst)) { st.stalled = 1; break; }
      stall_count = contracting ? 0 : stall_count + 1;
      if (stall_count >= 2) { st.stalled = 1; break; }
    }
    for (int q = 0; q < nrhs; ++q) prev[q] = rel[q];
  }
  if (transpose) {   // x = D x'
    hipLaunchKernelGGL(k_stretch_scale, dim3((P.ny + NT - 1) / NT, P.nx, nrhs), dim3(NT), 0, s, *g, x, 0);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
  }
  if (stats) *stats = st;
  if (rel_res) for (int q = 0; q < nrhs; ++q) rel_res[q] = rel[q];
  if (!st.converged)
    return fail(FDFD_ERR_NOT_CONVERGED, "refinement reached %.3e after %d sweeps (tol %.1e)%s",
                st.max_rel_residual, st.iterations, tol, st.stalled ? ", stalled" : "");
  return FDFD_OK;
}

// Whether a factor buffer of unknown kind (on a grid of the path's range)
// holds a nested-dissection factor: its tag; waits for the stream.
int nd_is_factor(const void *factor, hipStream_t s, bool *nd) {
  unsigned long long head[4];
  HIP_TRY(hipMemcpyAsync(head, factor, sizeof head, hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  *nd = true;
  for (int i = 0; i < 4; ++i) *nd = *nd && head[i] == nd_tag(i);
  return FDFD_OK;
}
