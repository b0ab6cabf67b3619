// adjoint.hip -- the differentiable run: reverse-mode gradients of the
// magnetic field energy after N steps of the hot path, with respect to the
// initial particle momenta and positions and the initial fields.
//
// The step is vpic_simulation::advance (src/vpic/advance.cc:25-185) on a
// periodic box with one pushed species: clear_accumulator_array, advance_p
// (advance_p_pipeline.cc:96-238 with move_p.cc:233-375), unload_accumulator
// (unload_accumulator_pipeline.cc:65-67), synchronize_jf (remote.cc:418-507),
// advance_b(0.5) (advance_b_pipeline.h:57-59), the tangential-B ghost copy
// and vacuum_advance_e (vacuum_advance_e_pipeline.h:56-69, damp 0),
// advance_b(0.5), load_interpolator_array (interpolator_array_pipeline.cc:
// 67-121).  The observable is the magnetic part of energy_f
// (vacuum_energy_f_pipeline.h:44-75).
//
// Everything is written once over the scalar type R: R = float is the
// product run (its forward is the reference's arithmetic operation for
// operation, so positions, momenta and cell indices equal the main push's);
// R = double is the same run in FP64, the reference for finite-difference
// checks.
//
// The field operations are linear, so their adjoints are their exact
// transposes over the array elements (ghost planes and the duplicated
// periodic face planes included), each written as a gather (no atomics).
// The particle push is differentiated with its branch held fixed: the cell
// sequence of a crossing particle, the face of each segment and the in-cell
// test are taken from the recomputed forward.  A crossing sets the crossed
// coordinate to exactly +-1, so that coordinate carries no derivative; the
// other quantities of a segment are smooth.  The reverse kernel recomputes
// each particle's forward from its state at the start of the step and the
// step's interpolators, then runs the derivatives backwards; a crossing
// particle's segments are replayed from the start for each segment it
// reverses (the segment count is small), so no per-segment storage is
// needed.
//
// Both pushes run tile by tile over particles sorted by cell every SORT_EVERY
// steps: a workgroup takes the particles of a tile of cells, sums the lanes of
// one cell in registers (a segmented wavefront scan) and adds the sums to a
// window of the tile and its neighbouring cells in LDS; k_merge adds the
// windows.  Deposits outside the window are global atomics, and so are all of
// them where there are no tiles (few particles, axes too long to sort by).
//
// Checkpointing: the forward stores the state (particles and fields) every
// `ckpt` steps; the reverse takes the segments last first, recomputes the
// segment's steps from its checkpoint storing each step's starting state,
// and reverses them.  The forward keeps the permutation and the partition of
// every sort: the recomputed steps are put in the forward's order with them
// (a recomputed state may differ from the forward's in its last bits, and a
// sort of its own could then order the particles differently), and the
// particle adjoints are put back in the order before a sort when the reverse
// passes it.
#include "common.h"

#include <exception>
#include <utility>
#include <vector>

namespace {

template <class R>
struct alignas(16) Part {
  R dx, dy, dz;
  int32_t i;
  R ux, uy, uz, w;
};
static_assert(sizeof(Part<float>) == 32, "particle_t layout");
static_assert(sizeof(Part<double>) == 64, "FP64 particle layout");

// The six field components the step carries between steps plus the current
// the step forms (tca is not carried: with no damping advance_e overwrites
// it before it is read).
template <class R>
struct Fld {
  R ex, ey, ez, cbx, cby, cbz, jfx, jfy, jfz;
};

constexpr int NI = 18;  // interpolator coefficients ex .. dcbzdz

struct Box {
  int nx, ny, nz, sy, sz, nv;
};

template <class R>
struct Coef {
  R qdt_2mc, cdt[3], qsp;
  R bp[3];   // advance_b(0.5): frac c dt / d per axis (0 for one cell)
  R ep[3];   // vacuum_advance_e: c dt / d per axis (0 for one cell)
  R cj;      // dt / eps0
  R uc[3];   // unload: 0.25 rd_y rd_z / dt, cyclic
};

__device__ inline float rsqrt_div(float a, float b) { return a / sqrtf(b); }
__device__ inline double rsqrt_div(double a, double b) { return a / sqrt(b); }
// move_p.cc:277: q*sx*sy*sz promoted to double by (1.0/3.0)
__device__ inline float streak_third(float x) {
  return (float)((double)x * (1.0 / 3.0));
}
__device__ inline double streak_third(double x) { return x * (1.0 / 3.0); }
__device__ inline void atomic_add_r(float *a, float v) { atomic_add_f32(a, v); }
__device__ inline void atomic_add_r(double *a, double v) {
  atomic_add_f64(a, v);
}

__device__ inline void coords(const Box &B, int v, int &x, int &y, int &z) {
  x = v % (B.nx + 2);
  const int t = v / (B.nx + 2);
  y = t % (B.ny + 2);
  z = t / (B.ny + 2);
}

// Tiles of cells.  8x4x4 cells hold 4096 particles at 32 per cell (16 per
// lane), and their windows (one cell more on every side, periodic) of 12 or
// 18 doubles a cell leave room for 4 or 3 workgroups on a CU.  The window is
// in double for both precisions: gfx950 adds doubles in LDS at 7 lanes a
// clock, floats at 0.3.
constexpr int AT_X = 8, AT_Y = 4, AT_Z = 4;
constexpr int AT_BS = 256, AT_WAVES = AT_BS / 64;
constexpr int AT_CELLS = (AT_X + 2) * (AT_Y + 2) * (AT_Z + 2);
constexpr int AT_ROWS = AT_Y * AT_Z;
// Most particles per workgroup without tiles; fewer, whole rounds of its lanes,
// as long as that leaves AT_CHUNKS workgroups or fewer (2100x1x1 cells, 60000
// particles, 16 steps with gradient: 8.3 ms with 4096 in each, 4.3 with 256).
constexpr int AT_CHUNK = 4096, AT_CHUNKS = 2048;
// No tiles for fewer particles than a third of the cells: the windows, their
// merge and the sorts cost by the cell (64^3 cells, 16 steps with gradient, 0.05,
// 0.2, 0.5 particles per cell: 7.8, 8.1, 8.3 ms with tiles, 5.6, 6.9, 9.6
// without; 128x128x64: 27.3, 28.8, 29.4 and 19.1, 24.7, 35.3).
constexpr int AT_SPARSE = 3;
// A thermal particle drifts by one cell in about ten steps; sorting more
// often costs more than the deposits that leave the windows until then.
constexpr int SORT_EVERY = 8;

// Tiles per axis; 0: no tiles (an axis too long for the sort's digits, or few
// particles), the workgroups take `chunk` particles each and have no window.
struct Tiles {
  int nt[3];
  int chunk;
};

struct TileAxis {
  int x0, n, h, w, len;  // first cell, cells, halo, window cells, box cells
  // window coordinate of box coordinate x (1..len), past w when outside
  __device__ __forceinline__ int local(int x) const {
    int l = x - x0 + h;
    if (l < 0) l += len;
    if (l >= len) l -= len;
    return l;
  }
};

__device__ __forceinline__ TileAxis tile_axis(int t, int size, int len) {
  TileAxis a;
  a.x0 = 1 + t * size;
  a.n = min(size, len + 1 - a.x0);
  a.h = len == 1 ? 0 : 1;
  a.w = min(a.n + 2 * a.h, len);
  a.len = len;
  return a;
}

struct TileWin {
  TileAxis x, y, z;
  bool on;
  __device__ __forceinline__ void at(const Tiles &T, const Box &B, int tile) {
    on = T.nt[0] > 0;
    if (!on) return;
    x = tile_axis(tile % T.nt[0], AT_X, B.nx);
    y = tile_axis((tile / T.nt[0]) % T.nt[1], AT_Y, B.ny);
    z = tile_axis(tile / (T.nt[0] * T.nt[1]), AT_Z, B.nz);
  }
  __device__ __forceinline__ int cells() const {
    return on ? x.w * y.w * z.w : 0;
  }
  // window cell of voxel v, -1 outside
  __device__ __forceinline__ int slot(const Box &B, int v) const {
    if (!on) return -1;
    int cx, cy, cz;
    coords(B, v, cx, cy, cz);
    const int lx = x.local(cx), ly = y.local(cy), lz = z.local(cz);
    return lx < x.w && ly < y.w && lz < z.w ? lx + x.w * (ly + y.w * lz) : -1;
  }
};

// The particles of a tile (the partition's rows of its cells, back to back)
// or, without tiles, a chunk of the array.
struct TileRows {
  int start[AT_ROWS], pref[AT_ROWS + 1], nrow;
  __device__ __forceinline__ void load(const TileWin &W, const Box &B,
                                       const Tiles &T, const int *part, int np,
                                       int tile) {
    const int t = threadIdx.x;
    if (!W.on) {
      if (t == 0) {
        nrow = 1;
        start[0] = tile * T.chunk;
        pref[0] = 0;
        pref[1] = min(T.chunk, np - tile * T.chunk);
      }
    } else {
      if (t < W.y.n * W.z.n) {
        const int cy = W.y.x0 + t % W.y.n, cz = W.z.x0 + t / W.y.n;
        int a = part[vox(W.x.x0, cy, cz, B.nx, B.ny)];
        int e = part[vox(W.x.x0 + W.x.n, cy, cz, B.nx, B.ny)];
        a = min(max(a, 0), np);
        e = min(max(e, a), np);
        start[t] = a;
        pref[t + 1] = e - a;
      }
      __syncthreads();
      if (t == 0) {
        nrow = W.y.n * W.z.n;
        pref[0] = 0;
        for (int r = 0; r < nrow; r++) pref[r + 1] += pref[r];
      }
    }
    __syncthreads();
  }
};

// Adds a run's sums to the window (cell-major) or, outside it, to the array.
template <class R, int N>
__device__ __forceinline__ void tile_add(double *win, const TileWin &W,
                                         const Box &B, R *out, int v,
                                         const R (&a)[N]) {
  const int s = W.slot(B, v);
  if (s >= 0) {
#pragma unroll
    for (int k = 0; k < N; k++)
      __hip_atomic_fetch_add(win + N * s + k, (double)a[k], __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
  } else {
#pragma unroll
    for (int k = 0; k < N; k++)
      if (a[k] != R(0)) atomic_add_r(out + (size_t)v * N + k, a[k]);
  }
}

template <class R, int N>
__device__ __forceinline__ void tile_store(const double *win, int ncell,
                                           R *wbuf, int tile) {
  R *w = wbuf + (size_t)tile * (N * AT_CELLS);
  for (int k = threadIdx.x; k < N * ncell; k += AT_BS) w[k] = (R)win[k];
}

// The windows that hold coordinate c of one axis: the tile of c and the ones
// beside it (once each) whose window reaches c.
struct Cover {
  int n, tile[3], l[3], w[3];
  __device__ __forceinline__ void of(int c, int size, int nt, int len) {
    n = 0;
    const int t = (c - 1) / size;
    for (int d = -1; d <= 1; d++) {
      if (d != 0 && (nt == 1 || (nt == 2 && d > 0))) continue;
      int q = t + d;
      q = q < 0 ? q + nt : q >= nt ? q - nt : q;
      const TileAxis a = tile_axis(q, size, len);
      const int l = a.local(c);
      if (l < a.w) {
        tile[n] = q;
        l_set(n, l, a.w);
        n++;
      }
    }
  }
  __device__ __forceinline__ void l_set(int k, int lv, int wv) {
    l[k] = lv;
    w[k] = wv;
  }
};

// out[v] += the windows' sums at v (out holds the deposits outside the
// windows); one thread per voxel.
template <class R, int N>
__global__ void __launch_bounds__(256)
    k_merge(R *__restrict__ out, const R *__restrict__ wbuf, Box B, Tiles T) {
  const int cell = blockIdx.x * blockDim.x + threadIdx.x;
  if (cell >= B.nx * B.ny * B.nz) return;
  const int cx = 1 + cell % B.nx, cy = 1 + (cell / B.nx) % B.ny,
            cz = 1 + cell / (B.nx * B.ny);
  Cover X, Y, Z;
  X.of(cx, AT_X, T.nt[0], B.nx);
  Y.of(cy, AT_Y, T.nt[1], B.ny);
  Z.of(cz, AT_Z, T.nt[2], B.nz);
  R *o = out + (size_t)N * vox(cx, cy, cz, B.nx, B.ny);
  R s[N];
#pragma unroll
  for (int k = 0; k < N; k++) s[k] = o[k];
  for (int iz = 0; iz < Z.n; iz++)
    for (int iy = 0; iy < Y.n; iy++)
      for (int ix = 0; ix < X.n; ix++) {
        const int tile = X.tile[ix] + T.nt[0] * (Y.tile[iy] +
                                                 T.nt[1] * Z.tile[iz]);
        const int l = X.l[ix] + X.w[ix] * (Y.l[iy] + Y.w[iy] * Z.l[iz]);
        const R *w = wbuf + (size_t)tile * (N * AT_CELLS) + N * l;
#pragma unroll
        for (int k = 0; k < N; k++) s[k] += w[k];
      }
#pragma unroll
  for (int k = 0; k < N; k++) o[k] = s[k];
}

// The sort by cell: keys of the particles, the partition from the sorted
// keys, and the moves of particles and adjoints into and out of its order.
template <class R>
__global__ void k_keys(const Part<R> *__restrict__ P, int np,
                       int *__restrict__ keys) {
  for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < np;
       n += gridDim.x * blockDim.x)
    keys[n] = P[n].i;
}

// Counts the particles in no cell of the box (outside the array, or in a ghost
// voxel, whose interpolators nobody writes).
template <class R>
__global__ void k_check_cells(const Part<R> *__restrict__ P, int np, Box B,
                              int *__restrict__ bad) {
  for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < np;
       n += gridDim.x * blockDim.x) {
    const int v = P[n].i;
    bool ok = (unsigned)v < (unsigned)B.nv;
    if (ok) {
      int x, y, z;
      coords(B, v, x, y, z);
      ok = x >= 1 && x <= B.nx && y >= 1 && y <= B.ny && z >= 1 && z <= B.nz;
    }
    if (!ok) atomicAdd(bad, 1);
  }
}

// part[v] = the first slot whose key is not below v: a search per voxel (a
// thread per slot that fills the voxels up to its key takes 130 us on a 64^3
// box, for the ghost plane below the first key).
__global__ void k_partition(const int *__restrict__ keys, int np, int nv,
                            int *__restrict__ part) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v > nv) return;
  int lo = 0, hi = np;
  while (lo < hi) {
    const int mid = lo + ((hi - lo) >> 1);
    if (keys[mid] < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  part[v] = lo;
}

typedef float adj_f4 __attribute__((ext_vector_type(4)));

// out[j] = in[perm[j]], 16 bytes per thread
template <class R>
__global__ void __launch_bounds__(256)
    k_permute(const Part<R> *__restrict__ in, const int *__restrict__ perm,
              int np, Part<R> *__restrict__ out) {
  constexpr int L = sizeof(Part<R>) / 16;
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t j = k / L;
  if (j >= np) return;
  reinterpret_cast<adj_f4 *>(out)[k] =
      reinterpret_cast<const adj_f4 *>(in)[(int64_t)perm[j] * L + k % L];
}

// out[perm[j]] = in[j], 6 values a particle
template <class R>
__global__ void __launch_bounds__(256)
    k_unpermute(const R *__restrict__ in, const int *__restrict__ perm, int np,
                R *__restrict__ out) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= np) return;
  const R *a = in + 6 * (size_t)j;
  R *b = out + 6 * (size_t)perm[j];
#pragma unroll
  for (int k = 0; k < 6; k++) b[k] = a[k];
}

// A wavefront's queue in LDS: crossers wait there until 64 of them fill a
// wavefront (a crosser's walk costs several times the rest of the push, and
// one lane in seven has one).
constexpr int AQ = 128;

__device__ __forceinline__ void wave_sync() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// The twelve updates of one streak in ACCUMULATE_J's order
// (advance_p_pipeline.cc:186-208, move_p.cc:281-303) into out[12].
template <class R>
__device__ inline void streak(R (&out)[12], R qx, R qy, R qz, R mx, R my,
                              R mz, R v5) {
  const R qd[3] = {qx, qy, qz}, m[3] = {mx, my, mz};
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const R mY = m[(c + 1) % 3], mZ = m[(c + 2) % 3];
    R v4 = qd[c], v1 = v4 * mY, v0 = v4 - v1;
    v1 += v4;
    v4 = 1 + mZ;
    R v2 = v0 * v4, v3 = v1 * v4;
    v4 = 1 - mZ;
    v0 *= v4;
    v1 *= v4;
    v0 += v5;
    v1 -= v5;
    v2 -= v5;
    v3 += v5;
    out[4 * c + 0] = v0;
    out[4 * c + 1] = v1;
    out[4 * c + 2] = v2;
    out[4 * c + 3] = v3;
  }
}

// One move_p segment (move_p.cc:240-275): the fraction v3 of the remaining
// displacement that reaches the first face (or all of it), that face's axis
// (3 for none) and direction.
template <class R>
struct Seg {
  R f, dir;
  int axis;
};

// a[axis] = v without an indexed register access
template <class R>
__device__ __forceinline__ void set3(R (&a)[3], int axis, R v) {
#pragma unroll
  for (int k = 0; k < 3; k++)
    if (k == axis) a[k] = v;
}
template <class R>
__device__ __forceinline__ R get3(const R (&a)[3], int axis) {
  return axis == 0 ? a[0] : axis == 1 ? a[1] : a[2];
}

template <class R>
__device__ inline Seg<R> seg_geom(const R (&d)[3], const R (&disp)[3]) {
  R sdir[3], t[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    sdir[k] = (disp[k] > R(0)) ? R(1) : R(-1);
    t[k] = (disp[k] == R(0)) ? R(3.4e38f) : (sdir[k] - d[k]) / disp[k];
  }
  Seg<R> s;
  R v3 = 2;
  s.axis = 3;
  if (t[0] < v3) v3 = t[0], s.axis = 0;
  if (t[1] < v3) v3 = t[1], s.axis = 1;
  if (t[2] < v3) v3 = t[2], s.axis = 2;
  s.f = v3 * R(0.5);
  s.dir = s.axis < 3 ? sdir[s.axis] : R(0);
  return s;
}

// ---------------------------------------------------------------------------
// forward push: advance_p_pipeline.cc:96-238 with the scalar move_p for a
// periodic box
// ---------------------------------------------------------------------------

// What a crosser's walk needs besides the particle.
template <class R>
struct FwdCross {
  int n;
  R disp[3];
};

// Pin and Pout may be the same array.  Bound by arithmetic and the windows'
// LDS adds: 8.4e6 particles of a 64^3 box take 274 us in FP32 (5234 us
// with shuffled run sums and global atomics).
template <class R>
__global__ void __launch_bounds__(AT_BS)
    k_push_fwd(const Part<R> *Pin, Part<R> *Pout, int np,
               const int *__restrict__ part, const R *__restrict__ fi,
               R *__restrict__ acc, R *__restrict__ wbuf, Coef<R> C, GridDev G,
               Box B, Tiles T, int *err) {
  __shared__ double win[12 * AT_CELLS];
  __shared__ FwdCross<R> queue[AT_WAVES][AQ];
  __shared__ TileRows rows;
  const R one = 1, one_third = R(1.0 / 3.0), two_fifteenths = R(2.0 / 15.0);
  const int tile = blockIdx.x, lane = lane_id();
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  TileWin W;
  W.at(T, B, tile);
  const int ncell = W.cells();
  for (int k = threadIdx.x; k < 12 * ncell; k += AT_BS) win[k] = 0;
  rows.load(W, B, T, part, np, tile);
  const int total = rows.pref[rows.nrow];
  FwdCross<R> *q = queue[wv];
  int qn = 0;

  // move_p (move_p.cc:233-375) of the last c crossers in the queue
  auto drain = [&](int c) {
    wave_sync();
    FwdCross<R> m;
    if (lane < c) m = q[qn - c + lane];
    wave_sync();
    qn -= c;
    if (lane >= c) return;
    const Part<R> p = Pin[m.n];
    R d[3] = {p.dx, p.dy, p.dz}, disp[3] = {m.disp[0], m.disp[1], m.disp[2]};
    const R q = p.w * C.qsp;
    int cell = p.i;
    for (int guard = 0; guard < 64; guard++) {
      const Seg<R> s = seg_geom(d, disp);
      R sd[3], mid[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        sd[k] = disp[k] * s.f;
        mid[k] = d[k] + sd[k];
      }
      const R w5 = streak_third(q * sd[0] * sd[1] * sd[2]);
      R st[12];
      streak(st, q * sd[0], q * sd[1], q * sd[2], mid[0], mid[1], mid[2], w5);
      tile_add<R, 12>(win, W, B, acc, cell, st);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        disp[k] -= sd[k];
        d[k] += sd[k] + sd[k];
      }
      if (s.axis == 3) break;
      set3(d, s.axis, s.dir);
      const int face = s.axis + (s.dir > R(0) ? 3 : 0);
      const int64_t nb = grid_neighbor(G, cell, face);
      if (nb < G.rangel || nb > G.rangeh) {
        atomicAdd(err, 1);  // only periodic boxes are differentiated
        break;
      }
      cell = (int)(nb - G.rangel);
      set3(d, s.axis, -s.dir);
    }
    Part<R> &o = Pout[m.n];
    o.dx = d[0];
    o.dy = d[1];
    o.dz = d[2];
    o.i = cell;
  };

  int r = 0;
  for (int base = wv * 64; base < total; base += AT_BS) {
    const int k = base + lane;
    const bool live = k < total;
    R dep[12];
#pragma unroll
    for (int c = 0; c < 12; c++) dep[c] = 0;
    int key = -1, n = 0;
    bool cross = false;
    R ux = 0, uy = 0, uz = 0;
    if (live) {
      while (r + 1 < rows.nrow && k >= rows.pref[r + 1]) r++;
      n = rows.start[r] + (k - rows.pref[r]);
      Part<R> p = Pin[n];
      const int ii = p.i;
      const R *f = fi + (size_t)NI * ii;
      const R dx = p.dx, dy = p.dy, dz = p.dz;
      const R qc = C.qdt_2mc;
      const R hax = qc * ((f[0] + dy * f[1]) + dz * (f[2] + dy * f[3]));
      const R hay = qc * ((f[4] + dz * f[5]) + dx * (f[6] + dz * f[7]));
      const R haz = qc * ((f[8] + dx * f[9]) + dy * (f[10] + dx * f[11]));
      const R cbx = f[12] + dx * f[13];
      const R cby = f[14] + dy * f[15];
      const R cbz = f[16] + dz * f[17];
      ux = p.ux + hax;
      uy = p.uy + hay;
      uz = p.uz + haz;
      R v0 = rsqrt_div(qc, one + (ux * ux + (uy * uy + uz * uz)));
      R v1 = cbx * cbx + (cby * cby + cbz * cbz);
      R v2 = (v0 * v0) * v1;
      R v3 = v0 * (one + v2 * (one_third + v2 * two_fifteenths));
      R v4 = v3 / (one + v1 * (v3 * v3));
      v4 += v4;
      v0 = ux + v3 * (uy * cbz - uz * cby);
      v1 = uy + v3 * (uz * cbx - ux * cbz);
      v2 = uz + v3 * (ux * cby - uy * cbx);
      ux += v4 * (v1 * cbz - v2 * cby);
      uy += v4 * (v2 * cbx - v0 * cbz);
      uz += v4 * (v0 * cby - v1 * cbx);
      ux += hax;
      uy += hay;
      uz += haz;
      p.ux = ux;
      p.uy = uy;
      p.uz = uz;
      v0 = rsqrt_div(one, one + (ux * ux + (uy * uy + uz * uz)));
      ux *= C.cdt[0];
      uy *= C.cdt[1];
      uz *= C.cdt[2];
      ux *= v0;
      uy *= v0;
      uz *= v0;
      v0 = dx + ux;
      v1 = dy + uy;
      v2 = dz + uz;
      v3 = v0 + ux;
      v4 = v1 + uy;
      R v5 = v2 + uz;
      const R qw = p.w * C.qsp;
      cross = !(v3 <= one && v4 <= one && v5 <= one && -v3 <= one &&
                -v4 <= one && -v5 <= one);
      if (!cross) {
        p.dx = v3;
        p.dy = v4;
        p.dz = v5;
        v5 = qw * ux * uy * uz * one_third;
        streak(dep, qw * ux, qw * uy, qw * uz, v0, v1, v2, v5);
        key = ii;
      }
      // (a crosser's position, still the old one here, is written by drain)
      Pout[n] = p;
    }
    const uint64_t cm = __ballot(cross);
    if (cm) {
      if (cross) {
        FwdCross<R> &m = q[qn + lanes_below(cm)];
        m.n = n;
        m.disp[0] = ux;
        m.disp[1] = uy;
        m.disp[2] = uz;
      }
      qn += __popcll(cm);
      if (qn >= 64) drain(64);
    }
    if (run_sums<R, 12>(key, dep) && key >= 0)
      tile_add<R, 12>(win, W, B, acc, key, dep);
  }
  if (qn) drain(qn);
  __syncthreads();
  tile_store<R, 12>(win, ncell, wbuf, tile);
}

// ---------------------------------------------------------------------------
// reverse push
// ---------------------------------------------------------------------------

// Adjoint of one streak's twelve updates: adds d/d(sd) and d/d(mid) of
// sum_k ab[k] * update_k to sdb and mb.
template <class R>
__device__ inline void streak_rev(const R *ab, R qw, const R (&sd)[3],
                                  const R (&m)[3], R (&sdb)[3], R (&mb)[3]) {
  R v5b = 0;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const int Y = (c + 1) % 3, Z = (c + 2) % 3;
    const R a0 = ab[4 * c], a1 = ab[4 * c + 1], a2 = ab[4 * c + 2],
            a3 = ab[4 * c + 3];
    const R mY = m[Y], mZ = m[Z];
    const R qd = qw * sd[c];
    const R qdb = a0 * (1 - mY) * (1 - mZ) + a1 * (1 + mY) * (1 - mZ) +
                  a2 * (1 - mY) * (1 + mZ) + a3 * (1 + mY) * (1 + mZ);
    mb[Y] += qd * ((1 - mZ) * (a1 - a0) + (1 + mZ) * (a3 - a2));
    mb[Z] += qd * ((1 - mY) * (a2 - a0) + (1 + mY) * (a3 - a1));
    v5b += (a0 - a1) - (a2 - a3);
    sdb[c] += qw * qdb;
  }
  const R t = v5b * qw * R(1.0 / 3.0);
  sdb[0] += t * sd[1] * sd[2];
  sdb[1] += t * sd[0] * sd[2];
  sdb[2] += t * sd[0] * sd[1];
}

// pb: per particle (d-bar[3], u-bar[3]) of the state after the step on
// entry, of the state before the step on return.  accb: the accumulator
// adjoint; fib: the interpolator adjoint (atomics).
// CROSS: the particle is known to leave its cell; without it a particle that
// does is left alone and reported (true).
template <class R, bool CROSS>
__device__ __forceinline__ bool rev_particle(
    int n, const Part<R> *__restrict__ P, const R *__restrict__ fi,
    const R *__restrict__ accb, R *__restrict__ pb, const Coef<R> &C,
    const GridDev &G, int &key, R (&gI)[NI]) {
  const R one = 1, c3 = R(1.0 / 3.0), c15 = R(2.0 / 15.0);
  {
    {
      const Part<R> p = P[n];
      const int ii = p.i;
      const R *f = fi + (size_t)NI * ii;
      const R d[3] = {p.dx, p.dy, p.dz};
      const R qc = C.qdt_2mc, qw = p.w * C.qsp;
      // forward, in exact-arithmetic form (the branch from the forward's
      // own rounding below)
      const R ha[3] = {qc * ((f[0] + d[1] * f[1]) + d[2] * (f[2] + d[1] * f[3])),
                       qc * ((f[4] + d[2] * f[5]) + d[0] * (f[6] + d[2] * f[7])),
                       qc * ((f[8] + d[0] * f[9]) + d[1] * (f[10] + d[0] * f[11]))};
      const R b[3] = {f[12] + d[0] * f[13], f[14] + d[1] * f[15],
                      f[16] + d[2] * f[17]};
      const R a[3] = {p.ux + ha[0], p.uy + ha[1], p.uz + ha[2]};
      const R g2 = one + (a[0] * a[0] + (a[1] * a[1] + a[2] * a[2]));
      const R v0 = rsqrt_div(qc, g2);
      const R v1 = b[0] * b[0] + (b[1] * b[1] + b[2] * b[2]);
      const R v2 = (v0 * v0) * v1;
      const R v3 = v0 * (one + v2 * (c3 + v2 * c15));
      const R den = one + v1 * (v3 * v3);
      R v4 = v3 / den;
      v4 += v4;
      const R w[3] = {a[0] + v3 * (a[1] * b[2] - a[2] * b[1]),
                      a[1] + v3 * (a[2] * b[0] - a[0] * b[2]),
                      a[2] + v3 * (a[0] * b[1] - a[1] * b[0])};
      const R wxb[3] = {w[1] * b[2] - w[2] * b[1], w[2] * b[0] - w[0] * b[2],
                        w[0] * b[1] - w[1] * b[0]};
      const R un[3] = {a[0] + v4 * wxb[0] + ha[0], a[1] + v4 * wxb[1] + ha[1],
                       a[2] + v4 * wxb[2] + ha[2]};
      const R r2 = rsqrt_div(one, one + (un[0] * un[0] +
                                         (un[1] * un[1] + un[2] * un[2])));
      const R s[3] = {(un[0] * C.cdt[0]) * r2, (un[1] * C.cdt[1]) * r2,
                      (un[2] * C.cdt[2]) * r2};
      const R e3[3] = {(d[0] + s[0]) + s[0], (d[1] + s[1]) + s[1],
                       (d[2] + s[2]) + s[2]};
      if (!CROSS && !(e3[0] <= one && e3[1] <= one && e3[2] <= one &&
                      -e3[0] <= one && -e3[1] <= one && -e3[2] <= one))
        return true;
      key = ii;
      R db[3] = {pb[6 * (size_t)n], pb[6 * (size_t)n + 1],
                 pb[6 * (size_t)n + 2]};
      R ub[3] = {pb[6 * (size_t)n + 3], pb[6 * (size_t)n + 4],
                 pb[6 * (size_t)n + 5]};
      R sb[3], d0b[3];
      if (!CROSS) {
        // in-cell: new d = d + 2s, streak (s, d + s) in cell ii
        const R mid[3] = {d[0] + s[0], d[1] + s[1], d[2] + s[2]};
        R sdb[3] = {0, 0, 0}, mb[3] = {0, 0, 0};
        streak_rev(accb + (size_t)12 * ii, qw, s, mid, sdb, mb);
#pragma unroll
        for (int k = 0; k < 3; k++) {
          d0b[k] = db[k] + mb[k];
          sb[k] = 2 * db[k] + mb[k] + sdb[k];
        }
      } else {
        // count the segments (the forward's move_p walk)
        int nseg = 0;
        {
          R dd[3] = {d[0], d[1], d[2]}, ds[3] = {s[0], s[1], s[2]};
          int cell = ii;
          for (; nseg < 64;) {
            const Seg<R> g = seg_geom(dd, ds);
            nseg++;
#pragma unroll
            for (int k = 0; k < 3; k++) {
              const R sd = ds[k] * g.f;
              ds[k] -= sd;
              dd[k] += sd + sd;
            }
            if (g.axis == 3) break;
            const int face = g.axis + (g.dir > R(0) ? 3 : 0);
            cell = (int)(grid_neighbor(G, cell, face) - G.rangel);
            set3(dd, g.axis, -g.dir);
          }
        }
        // reverse the segments, each replayed from the start
        R Db[3] = {db[0], db[1], db[2]}, Pb[3] = {0, 0, 0};
        for (int j = nseg - 1; j >= 0; j--) {
          R dd[3] = {d[0], d[1], d[2]}, ds[3] = {s[0], s[1], s[2]};
          int cell = ii;
          Seg<R> g = seg_geom(dd, ds);
          for (int t = 0; t < j; t++) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
              const R sd = ds[k] * g.f;
              ds[k] -= sd;
              dd[k] += sd + sd;
            }
            const int face = g.axis + (g.dir > R(0) ? 3 : 0);
            cell = (int)(grid_neighbor(G, cell, face) - G.rangel);
            set3(dd, g.axis, -g.dir);
            g = seg_geom(dd, ds);
          }
          // segment j: sd = ds f, mid = dd + sd, d' = dd + 2 sd (the crossed
          // coordinate then set to a constant), disp' = ds - sd
          R sd[3], mid[3];
#pragma unroll
          for (int k = 0; k < 3; k++) {
            sd[k] = ds[k] * g.f;
            mid[k] = dd[k] + sd[k];
          }
          if (g.axis < 3) set3(Db, g.axis, R(0));
          R sdb[3], mb[3] = {0, 0, 0};
#pragma unroll
          for (int k = 0; k < 3; k++) sdb[k] = 2 * Db[k] - Pb[k];
          streak_rev(accb + (size_t)12 * cell, qw, sd, mid, sdb, mb);
          R fb = 0;
#pragma unroll
          for (int k = 0; k < 3; k++) {
            sdb[k] += mb[k];
            Db[k] += mb[k];
            Pb[k] += sdb[k] * g.f;
            fb += sdb[k] * ds[k];
          }
          if (g.axis < 3) {
            const R dsa = get3(ds, g.axis);
            set3(Db, g.axis, get3(Db, g.axis) + -R(0.5) * fb / dsa);
            set3(Pb, g.axis, get3(Pb, g.axis) + -fb * g.f / dsa);
          }
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
          d0b[k] = Db[k];
          sb[k] = Pb[k];
        }
      }
      // s = un cdt r2, r2 = (1 + |un|^2)^-1/2
      R rb = 0;
#pragma unroll
      for (int k = 0; k < 3; k++) rb += sb[k] * un[k] * C.cdt[k];
      R unb[3];
#pragma unroll
      for (int k = 0; k < 3; k++)
        unb[k] = ub[k] + sb[k] * C.cdt[k] * r2 - rb * r2 * r2 * r2 * un[k];
      // un = a + v4 (w x b) + ha
      R hab[3] = {unb[0], unb[1], unb[2]};
      R ab[3] = {unb[0], unb[1], unb[2]};
      const R v4b = unb[0] * wxb[0] + unb[1] * wxb[1] + unb[2] * wxb[2];
      R wb[3] = {v4 * (b[1] * unb[2] - b[2] * unb[1]),
                 v4 * (b[2] * unb[0] - b[0] * unb[2]),
                 v4 * (b[0] * unb[1] - b[1] * unb[0])};
      R bb[3] = {v4 * (unb[1] * w[2] - unb[2] * w[1]),
                 v4 * (unb[2] * w[0] - unb[0] * w[2]),
                 v4 * (unb[0] * w[1] - unb[1] * w[0])};
      // w = a + v3 (a x b)
      const R axb[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2],
                        a[0] * b[1] - a[1] * b[0]};
      R v3b = wb[0] * axb[0] + wb[1] * axb[1] + wb[2] * axb[2];
      ab[0] += wb[0] + v3 * (b[1] * wb[2] - b[2] * wb[1]);
      ab[1] += wb[1] + v3 * (b[2] * wb[0] - b[0] * wb[2]);
      ab[2] += wb[2] + v3 * (b[0] * wb[1] - b[1] * wb[0]);
      bb[0] += v3 * (wb[1] * a[2] - wb[2] * a[1]);
      bb[1] += v3 * (wb[2] * a[0] - wb[0] * a[2]);
      bb[2] += v3 * (wb[0] * a[1] - wb[1] * a[0]);
      // v4 = 2 v3 / (1 + v1 v3^2)
      v3b += v4b * (2 / den) * (one - 2 * v1 * v3 * v3 / den);
      R v1b = -v4b * 2 * v3 * v3 * v3 / (den * den);
      // v3 = v0 (1 + v2 (1/3 + v2 2/15))
      R v0b = v3b * (one + v2 * (c3 + v2 * c15));
      const R v2b = v3b * v0 * (c3 + 2 * c15 * v2);
      // v2 = v0^2 v1
      v0b += v2b * 2 * v0 * v1;
      v1b += v2b * v0 * v0;
      // v1 = |b|^2
#pragma unroll
      for (int k = 0; k < 3; k++) bb[k] += 2 * v1b * b[k];
      // v0 = qc / sqrt(1 + |a|^2)
      const R t0 = -v0b * v0 / g2;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        ab[k] += t0 * a[k];
        hab[k] += ab[k];  // a = u + ha
      }
      // interpolation
      R g = qc * hab[0];
      gI[0] = g;
      gI[1] = g * d[1];
      gI[2] = g * d[2];
      gI[3] = g * d[1] * d[2];
      d0b[1] += g * (f[1] + d[2] * f[3]);
      d0b[2] += g * (f[2] + d[1] * f[3]);
      g = qc * hab[1];
      gI[4] = g;
      gI[5] = g * d[2];
      gI[6] = g * d[0];
      gI[7] = g * d[2] * d[0];
      d0b[2] += g * (f[5] + d[0] * f[7]);
      d0b[0] += g * (f[6] + d[2] * f[7]);
      g = qc * hab[2];
      gI[8] = g;
      gI[9] = g * d[0];
      gI[10] = g * d[1];
      gI[11] = g * d[0] * d[1];
      d0b[0] += g * (f[9] + d[1] * f[11]);
      d0b[1] += g * (f[10] + d[0] * f[11]);
      gI[12] = bb[0];
      gI[13] = bb[0] * d[0];
      d0b[0] += bb[0] * f[13];
      gI[14] = bb[1];
      gI[15] = bb[1] * d[1];
      d0b[1] += bb[1] * f[15];
      gI[16] = bb[2];
      gI[17] = bb[2] * d[2];
      d0b[2] += bb[2] * f[17];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        pb[6 * (size_t)n + k] = d0b[k];
        pb[6 * (size_t)n + 3 + k] = ab[k];
      }
    }
  }
  return false;
}

// The particles that stay in their cell first, the crossers 64 at a time.
// Bound by arithmetic: 8.4e6 particles of a 64^3 box take 461 us in FP32
// (6919 us with shuffled run sums and global atomics).
template <class R>
__global__ void __launch_bounds__(AT_BS)
    k_push_rev(const Part<R> *__restrict__ P, int np,
               const int *__restrict__ part, const R *__restrict__ fi,
               const R *__restrict__ accb, R *__restrict__ pb,
               R *__restrict__ fib, R *__restrict__ wbuf, Coef<R> C, GridDev G,
               Box B, Tiles T) {
  __shared__ double win[NI * AT_CELLS];
  __shared__ int queue[AT_WAVES][AQ];
  __shared__ TileRows rows;
  const int tile = blockIdx.x, lane = lane_id();
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  TileWin W;
  W.at(T, B, tile);
  const int ncell = W.cells();
  for (int k = threadIdx.x; k < NI * ncell; k += AT_BS) win[k] = 0;
  rows.load(W, B, T, part, np, tile);
  const int total = rows.pref[rows.nrow];
  int *q = queue[wv];
  int qn = 0;

  auto drain = [&](int c) {
    wave_sync();
    const int n = lane < c ? q[qn - c + lane] : 0;
    wave_sync();
    qn -= c;
    R gI[NI];
#pragma unroll
    for (int k = 0; k < NI; k++) gI[k] = 0;
    int key = -1;
    if (lane < c) rev_particle<R, true>(n, P, fi, accb, pb, C, G, key, gI);
    if (run_sums<R, NI>(key, gI) && key >= 0)
      tile_add<R, NI>(win, W, B, fib, key, gI);
  };

  int r = 0;
  for (int base = wv * 64; base < total; base += AT_BS) {
    const int k = base + lane;
    R gI[NI];
#pragma unroll
    for (int c = 0; c < NI; c++) gI[c] = 0;
    int key = -1, n = 0;
    bool cross = false;
    if (k < total) {
      while (r + 1 < rows.nrow && k >= rows.pref[r + 1]) r++;
      n = rows.start[r] + (k - rows.pref[r]);
      cross = rev_particle<R, false>(n, P, fi, accb, pb, C, G, key, gI);
    }
    if (run_sums<R, NI>(key, gI) && key >= 0)
      tile_add<R, NI>(win, W, B, fib, key, gI);
    const uint64_t cm = __ballot(cross);
    if (cm) {
      if (cross) q[qn + lanes_below(cm)] = n;
      qn += __popcll(cm);
      if (qn >= 64) drain(64);
    }
  }
  if (qn) drain(qn);
  __syncthreads();
  tile_store<R, NI>(win, ncell, wbuf, tile);
}

// ---------------------------------------------------------------------------
// field operations and their transposes (periodic box)
// ---------------------------------------------------------------------------

__device__ inline bool in_box(const Box &B, int x, int y, int z, int x0,
                              int x1, int y0, int y1, int z0, int z1) {
  return x >= x0 && x <= x1 && y >= y0 && y <= y1 && z >= z0 && z <= z1;
}

template <class R>
__global__ void k_fill(R *a, size_t n, R v) {
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < n;
       k += (size_t)gridDim.x * blockDim.x)
    a[k] = v;
}

// load_interpolator_pipeline_scalar (interpolator_array_pipeline.cc:67-121)
template <class R>
__global__ void k_load(R *fi, const Fld<R> *F, Box B) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= B.nv) return;
  int x, y, z;
  coords(B, v, x, y, z);
  if (!in_box(B, x, y, z, 1, B.nx, 1, B.ny, 1, B.nz)) return;
  const R fourth = R(0.25), half = R(0.5);
  const int sx = 1, sy = B.sy, sz = B.sz;
  R *o = fi + (size_t)NI * v;
  R w0, w1, w2, w3;
  w0 = F[v].ex; w1 = F[v + sy].ex; w2 = F[v + sz].ex; w3 = F[v + sy + sz].ex;
  o[0] = fourth * ((w3 + w0) + (w1 + w2));
  o[1] = fourth * ((w3 - w0) + (w1 - w2));
  o[2] = fourth * ((w3 - w0) - (w1 - w2));
  o[3] = fourth * ((w3 + w0) - (w1 + w2));
  w0 = F[v].ey; w1 = F[v + sz].ey; w2 = F[v + sx].ey; w3 = F[v + sz + sx].ey;
  o[4] = fourth * ((w3 + w0) + (w1 + w2));
  o[5] = fourth * ((w3 - w0) + (w1 - w2));
  o[6] = fourth * ((w3 - w0) - (w1 - w2));
  o[7] = fourth * ((w3 + w0) - (w1 + w2));
  w0 = F[v].ez; w1 = F[v + sx].ez; w2 = F[v + sy].ez; w3 = F[v + sx + sy].ez;
  o[8] = fourth * ((w3 + w0) + (w1 + w2));
  o[9] = fourth * ((w3 - w0) + (w1 - w2));
  o[10] = fourth * ((w3 - w0) - (w1 - w2));
  o[11] = fourth * ((w3 + w0) - (w1 + w2));
  w0 = F[v].cbx; w1 = F[v + sx].cbx;
  o[12] = half * (w1 + w0);
  o[13] = half * (w1 - w0);
  w0 = F[v].cby; w1 = F[v + sy].cby;
  o[14] = half * (w1 + w0);
  o[15] = half * (w1 - w0);
  w0 = F[v].cbz; w1 = F[v + sz].cbz;
  o[16] = half * (w1 + w0);
  o[17] = half * (w1 - w0);
}

// Transpose of k_load: Fb += load^T(fib).  Voxel u receives, for each of
// ex/ey/ez, the four corner weights of the interpolators at u, u - Y, u - Z,
// u - Y - Z ((Y, Z) the component's cyclic pair), and for cb the two face
// weights of u and u - X.
template <class R>
__device__ inline R corner_T(const R *fib, const Box &B, int u, int c0,
                             int oy, int oz) {
  // weights of (w0, w1, w2, w3) on (value, d/dY, d/dZ, d2/dYdZ)
  const R q = R(0.25);
  R s = 0;
  const int cand[4] = {u, u - oy, u - oz, u - oy - oz};
  const R sgn[4][4] = {{1, -1, -1, 1}, {1, 1, -1, -1}, {1, -1, 1, -1},
                       {1, 1, 1, 1}};
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int v = cand[k];
    if (v < 0) continue;
    int x, y, z;
    coords(B, v, x, y, z);
    if (!in_box(B, x, y, z, 1, B.nx, 1, B.ny, 1, B.nz)) continue;
    const R *g = fib + (size_t)NI * v + c0;
    s += q * (sgn[k][0] * g[0] + sgn[k][1] * g[1] + sgn[k][2] * g[2] +
              sgn[k][3] * g[3]);
  }
  return s;
}

template <class R>
__device__ inline R face_T(const R *fib, const Box &B, int u, int c0, int ox) {
  const R h = R(0.5);
  R s = 0;
  int x, y, z;
  coords(B, u, x, y, z);
  if (in_box(B, x, y, z, 1, B.nx, 1, B.ny, 1, B.nz)) {
    const R *g = fib + (size_t)NI * u + c0;
    s += h * (g[0] - g[1]);
  }
  const int v = u - ox;
  if (v >= 0) {
    coords(B, v, x, y, z);
    if (in_box(B, x, y, z, 1, B.nx, 1, B.ny, 1, B.nz)) {
      const R *g = fib + (size_t)NI * v + c0;
      s += h * (g[0] + g[1]);
    }
  }
  return s;
}

template <class R>
__global__ void k_load_T(Fld<R> *Fb, const R *fib, Box B) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= B.nv) return;
  const int sx = 1, sy = B.sy, sz = B.sz;
  Fld<R> o = Fb[u];
  o.ex += corner_T(fib, B, u, 0, sy, sz);
  o.ey += corner_T(fib, B, u, 4, sz, sx);
  o.ez += corner_T(fib, B, u, 8, sx, sy);
  o.cbx += face_T(fib, B, u, 12, sx);
  o.cby += face_T(fib, B, u, 14, sy);
  o.cbz += face_T(fib, B, u, 16, sz);
  Fb[u] = o;
}

// clear_jf + unload_accumulator over voxels 1..n+1
// (unload_accumulator_pipeline.cc:65-67)
template <class R>
__device__ void unload_at(Fld<R> *F, const R *acc, const Coef<R> &C,
                          const Box &B, int v) {
  int x, y, z;
  coords(B, v, x, y, z);
  Fld<R> &f = F[v];
  f.jfx = f.jfy = f.jfz = 0;
  if (!in_box(B, x, y, z, 1, B.nx + 1, 1, B.ny + 1, 1, B.nz + 1)) return;
  const int sx = 1, sy = B.sy, sz = B.sz;
  const R *a0 = acc + (size_t)12 * v;
  const R *ax = acc + (size_t)12 * (v - sx), *ay = acc + (size_t)12 * (v - sy),
          *az = acc + (size_t)12 * (v - sz);
  const R *ayz = acc + (size_t)12 * (v - sy - sz),
          *azx = acc + (size_t)12 * (v - sz - sx),
          *axy = acc + (size_t)12 * (v - sx - sy);
  f.jfx += C.uc[0] * (a0[0] + ay[1] + az[2] + ayz[3]);
  f.jfy += C.uc[1] * (a0[4] + az[5] + ax[6] + azx[7]);
  f.jfz += C.uc[2] * (a0[8] + ax[9] + ay[10] + axy[11]);
}

// Transpose of unload_at: accumulator adjoint of voxel u from jf-bar.
template <class R>
__global__ void k_unload_T(R *accb, const Fld<R> *Fb, Coef<R> C, Box B) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= B.nv) return;
  const int sx = 1, sy = B.sy, sz = B.sz;
  auto jb = [&](int v, int comp) -> R {
    if (v >= B.nv) return R(0);
    int x, y, z;
    coords(B, v, x, y, z);
    if (!in_box(B, x, y, z, 1, B.nx + 1, 1, B.ny + 1, 1, B.nz + 1))
      return R(0);
    return comp == 0 ? Fb[v].jfx : comp == 1 ? Fb[v].jfy : Fb[v].jfz;
  };
  R *o = accb + (size_t)12 * u;
  o[0] = C.uc[0] * jb(u, 0);
  o[1] = C.uc[0] * jb(u + sy, 0);
  o[2] = C.uc[0] * jb(u + sz, 0);
  o[3] = C.uc[0] * jb(u + sy + sz, 0);
  o[4] = C.uc[1] * jb(u, 1);
  o[5] = C.uc[1] * jb(u + sz, 1);
  o[6] = C.uc[1] * jb(u + sx, 1);
  o[7] = C.uc[1] * jb(u + sz + sx, 1);
  o[8] = C.uc[2] * jb(u, 2);
  o[9] = C.uc[2] * jb(u + sx, 2);
  o[10] = C.uc[2] * jb(u + sy, 2);
  o[11] = C.uc[2] * jb(u + sx + sy, 2);
}

// synchronize_jf on a periodic box (remote.cc:474-502): along each axis the
// tangential jf of the two face planes 1 and n+1 both become their sum, axis
// after axis.  The map of one axis is symmetric, so the transpose is the axes
// in the other order (`back`).  All axes at once: component c = l / (places)
// is folded along the two others, P < Q; a thread has all copies of an
// element (two on a face, four on an edge).  A launch an axis was 4 us each.
__host__ __device__ inline int fold_places(const Box &B, int C) {
  return C == 0   ? B.nx * (B.nz + B.ny - 1)
         : C == 1 ? B.ny * (B.nz + B.nx - 1)
                  : B.nz * (B.ny + B.nx - 1);
}
__host__ __device__ inline int64_t fold_places(const Box &B) {
  return (int64_t)fold_places(B, 0) + fold_places(B, 1) + fold_places(B, 2);
}
template <class R>
__device__ void fold_jf_at(Fld<R> *F, const Box &B, int64_t l, bool back) {
  int C = 0;
  while (C < 2 && l >= fold_places(B, C)) l -= fold_places(B, C++);
  const int n[3] = {B.nx, B.ny, B.nz};
  const int st[3] = {1, B.sy, B.sz};
  const int P = C == 0 ? 1 : 0, Q = C == 2 ? 1 : 2;
  const int nC = n[C], m = (int)l / nC, c = 1 + (int)l % nC;
  // the P faces (places q = 1..nQ of both planes), then the Q faces off them
  const bool on_p = m < n[Q];
  const int hp = n[P] * st[P], hq = n[Q] * st[Q];
  R *j = &F[c * st[C] + (on_p ? 1 : 2 + m - n[Q]) * st[P] +
            (on_p ? 1 + m : 1) * st[Q]]
              .jfx +
         C;
  auto at = [&](int h) -> R & {
    return *reinterpret_cast<R *>(reinterpret_cast<char *>(j) +
                                  (int64_t)h * sizeof(Fld<R>));
  };
  if (on_p && m == 0) {
    const R a = at(0), b = at(hp), d = at(hq), e = at(hp + hq);
    const R t = back ? (a + d) + (b + e) : (a + b) + (d + e);
    at(0) = t;
    at(hp) = t;
    at(hq) = t;
    at(hp + hq) = t;
  } else {
    const int h = on_p ? hp : hq;
    const R t = at(0) + at(h);
    at(0) = t;
    at(h) = t;
  }
}
template <class R>
__global__ void k_fold_jf_T(Fld<R> *Fb, Box B) {
  const int64_t l = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (l < fold_places(B)) fold_jf_at(Fb, B, l, true);
}

// advance_b (advance_b_pipeline.h:57-59 over voxels 1..n+1)
template <class R>
__device__ void advance_b_at(Fld<R> *F, const Coef<R> &C, const Box &B, int v) {
  int x, y, z;
  coords(B, v, x, y, z);
  if (!in_box(B, x, y, z, 1, B.nx + 1, 1, B.ny + 1, 1, B.nz + 1)) return;
  const R px = C.bp[0], py = C.bp[1], pz = C.bp[2];
  Fld<R> *f = F + v;
  // the +1 neighbours are read only where they lie inside the array
  if (y <= B.ny && z <= B.nz) {
    const Fld<R> *fy = F + v + B.sy, *fz = F + v + B.sz;
    f->cbx -= (py * (fy->ez - f->ez) - pz * (fz->ey - f->ey));
  }
  if (x <= B.nx && z <= B.nz) {
    const Fld<R> *fx = F + v + 1, *fz = F + v + B.sz;
    f->cby -= (pz * (fz->ex - f->ex) - px * (fx->ez - f->ez));
  }
  if (x <= B.nx && y <= B.ny) {
    const Fld<R> *fx = F + v + 1, *fy = F + v + B.sy;
    f->cbz -= (px * (fx->ey - f->ey) - py * (fy->ex - f->ex));
  }
}
template <class R>
__global__ void k_advance_b(Fld<R> *F, Coef<R> C, Box B) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < B.nv) advance_b_at(F, C, B, v);
}
// (jf and B of a voxel, from the accumulator and E: one pass for both)
template <class R>
__global__ void k_unload_advance_b(Fld<R> *F, const R *acc, Coef<R> C, Box B) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= B.nv) return;
  unload_at(F, acc, C, B, v);
  advance_b_at(F, C, B, v);
}

__device__ inline bool in_bx(const Box &B, int v) {
  if (v < 0 || v >= B.nv) return false;
  int x, y, z;
  coords(B, v, x, y, z);
  return in_box(B, x, y, z, 1, B.nx + 1, 1, B.ny, 1, B.nz);
}
__device__ inline bool in_by(const Box &B, int v) {
  if (v < 0 || v >= B.nv) return false;
  int x, y, z;
  coords(B, v, x, y, z);
  return in_box(B, x, y, z, 1, B.nx, 1, B.ny + 1, 1, B.nz);
}
__device__ inline bool in_bz(const Box &B, int v) {
  if (v < 0 || v >= B.nv) return false;
  int x, y, z;
  coords(B, v, x, y, z);
  return in_box(B, x, y, z, 1, B.nx, 1, B.ny, 1, B.nz + 1);
}
__device__ inline bool in_ex(const Box &B, int v) {
  if (v < 0 || v >= B.nv) return false;
  int x, y, z;
  coords(B, v, x, y, z);
  return in_box(B, x, y, z, 1, B.nx, 1, B.ny + 1, 1, B.nz + 1);
}
__device__ inline bool in_ey(const Box &B, int v) {
  if (v < 0 || v >= B.nv) return false;
  int x, y, z;
  coords(B, v, x, y, z);
  return in_box(B, x, y, z, 1, B.nx + 1, 1, B.ny, 1, B.nz + 1);
}
__device__ inline bool in_ez(const Box &B, int v) {
  if (v < 0 || v >= B.nv) return false;
  int x, y, z;
  coords(B, v, x, y, z);
  return in_box(B, x, y, z, 1, B.nx + 1, 1, B.ny + 1, 1, B.nz);
}

// Transpose of k_advance_b: E-bar += T_b^T cb-bar (cb-bar passes through).
template <class R>
__global__ void k_advance_b_T(Fld<R> *Fb, Coef<R> C, Box B) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= B.nv) return;
  const R px = C.bp[0], py = C.bp[1], pz = C.bp[2];
  const int sx = 1, sy = B.sy, sz = B.sz;
  auto bx = [&](int v) { return in_bx(B, v) ? Fb[v].cbx : R(0); };
  auto by = [&](int v) { return in_by(B, v) ? Fb[v].cby : R(0); };
  auto bz = [&](int v) { return in_bz(B, v) ? Fb[v].cbz : R(0); };
  // cbx[v] += -py ez[v+sy] + py ez[v] + pz ey[v+sz] - pz ey[v]
  // cby[v] += -pz ex[v+sz] + pz ex[v] + px ez[v+sx] - px ez[v]
  // cbz[v] += -px ey[v+sx] + px ey[v] + py ex[v+sy] - py ex[v]
  const R exb = pz * (by(u) - by(u - sz)) + py * (bz(u - sy) - bz(u));
  const R eyb = pz * (bx(u - sz) - bx(u)) + px * (bz(u) - bz(u - sx));
  const R ezb = py * (bx(u) - bx(u - sy)) + px * (by(u - sx) - by(u));
  Fb[u].ex += exb;
  Fb[u].ey += eyb;
  Fb[u].ez += ezb;
}

// Tangential cb ghosts of a periodic box (remote.cc:61-134 with the
// self-loop port): the ghost plane X = n+1 takes face plane 1, X = 0 takes
// face plane n, for the two tangential components.
template <class R>
__device__ void ghost_b_at(Fld<R> *F, const Box &B, int v) {
  int c[3];
  coords(B, v, c[0], c[1], c[2]);
  const int n[3] = {B.nx, B.ny, B.nz};
  for (int X = 0; X < 3; X++) {
    const int src = c[X] == 0 ? n[X] : c[X] == n[X] + 1 ? 1 : -1;
    if (src < 0) continue;
    const int Y = (X + 1) % 3, Z = (X + 2) % 3;
    int s[3] = {c[0], c[1], c[2]};
    s[X] = src;
    const int u = vox(s[0], s[1], s[2], B.nx, B.ny);
    R *dst = &F[v].cbx;
    const R *from = &F[u].cbx;
    // cb_Y on (Y in 1..nY+1, Z in 1..nZ); cb_Z on (Y in 1..nY, Z in 1..nZ+1)
    if (c[Y] >= 1 && c[Y] <= n[Y] + 1 && c[Z] >= 1 && c[Z] <= n[Z])
      dst[Y] = from[Y];
    if (c[Y] >= 1 && c[Y] <= n[Y] && c[Z] >= 1 && c[Z] <= n[Z] + 1)
      dst[Z] = from[Z];
  }
}

// The jf fold and the B ghosts, which share no component.
template <class R>
__global__ void k_fold_jf_ghost_b(Fld<R> *F, Box B, int fold_blocks) {
  const int b = blockIdx.x;
  if (b < fold_blocks) {
    const int64_t l = b * (int64_t)blockDim.x + threadIdx.x;
    if (l < fold_places(B)) fold_jf_at(F, B, l, false);
    return;
  }
  const int v = (b - fold_blocks) * blockDim.x + threadIdx.x;
  if (v < B.nv) ghost_b_at(F, B, v);
}

// Transpose of ghost_b_at: each face-plane element adds the ghosts it fed and
// clears them (a ghost is fed by one element, and is no face-plane element of
// another axis, so no other thread touches either).
template <class R>
__global__ void k_ghost_b_T(Fld<R> *Fb, Box B) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= B.nv) return;
  int c[3];
  coords(B, v, c[0], c[1], c[2]);
  const int n[3] = {B.nx, B.ny, B.nz};
  R add[3] = {0, 0, 0};
  bool any[3] = {false, false, false};
  for (int X = 0; X < 3; X++) {
    const int Y = (X + 1) % 3, Z = (X + 2) % 3;
    const bool inY = c[Y] >= 1 && c[Y] <= n[Y] + 1 && c[Z] >= 1 && c[Z] <= n[Z];
    const bool inZ = c[Y] >= 1 && c[Y] <= n[Y] && c[Z] >= 1 && c[Z] <= n[Z] + 1;
    for (int side = 0; side < 2; side++) {
      // face plane 1 feeds ghost n+1; face plane n feeds ghost 0
      const int face = side == 0 ? 1 : n[X];
      if (c[X] != face) continue;
      int g[3] = {c[0], c[1], c[2]};
      g[X] = side == 0 ? n[X] + 1 : 0;
      R *gb = &Fb[vox(g[0], g[1], g[2], B.nx, B.ny)].cbx;
      if (inY) {
        add[Y] += gb[Y];
        gb[Y] = 0;
        any[Y] = true;
      }
      if (inZ) {
        add[Z] += gb[Z];
        gb[Z] = 0;
        any[Z] = true;
      }
    }
  }
  R *b = &Fb[v].cbx;
  for (int k = 0; k < 3; k++)
    if (any[k]) b[k] += add[k];
}

// vacuum_advance_e with no damping (vacuum_advance_e_pipeline.h:56-69;
// decay = drive = rmu = 1), voxels 1..n+1.
template <class R>
__global__ void k_advance_e(Fld<R> *F, Coef<R> C, Box B) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= B.nv) return;
  int x, y, z;
  coords(B, v, x, y, z);
  if (!in_box(B, x, y, z, 1, B.nx + 1, 1, B.ny + 1, 1, B.nz + 1)) return;
  const R px = C.ep[0], py = C.ep[1], pz = C.ep[2], cj = C.cj, one = 1;
  Fld<R> &f = F[v];
  const Fld<R> &fx = F[v - 1], &fy = F[v - B.sy], &fz = F[v - B.sz];
  if (x <= B.nx) {
    const R t = py * (f.cbz - fy.cbz) - pz * (f.cby - fz.cby);
    f.ex = one * f.ex + one * (t - cj * f.jfx);
  }
  if (y <= B.ny) {
    const R t = pz * (f.cbx - fz.cbx) - px * (f.cbz - fx.cbz);
    f.ey = one * f.ey + one * (t - cj * f.jfy);
  }
  if (z <= B.nz) {
    const R t = px * (f.cby - fx.cby) - py * (f.cbx - fy.cbx);
    f.ez = one * f.ez + one * (t - cj * f.jfz);
  }
}

// Transpose of k_advance_e: cb-bar += T_e^T E-bar, jf-bar = -cj E-bar
// (E-bar passes through).
template <class R>
__global__ void k_advance_e_T(Fld<R> *Fb, Coef<R> C, Box B) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= B.nv) return;
  const R px = C.ep[0], py = C.ep[1], pz = C.ep[2], cj = C.cj;
  const int sx = 1, sy = B.sy, sz = B.sz;
  auto ex = [&](int v) { return in_ex(B, v) ? Fb[v].ex : R(0); };
  auto ey = [&](int v) { return in_ey(B, v) ? Fb[v].ey : R(0); };
  auto ez = [&](int v) { return in_ez(B, v) ? Fb[v].ez : R(0); };
  // ex[v] += py (cbz[v] - cbz[v-sy]) - pz (cby[v] - cby[v-sz])
  // ey[v] += pz (cbx[v] - cbx[v-sz]) - px (cbz[v] - cbz[v-sx])
  // ez[v] += px (cby[v] - cby[v-sx]) - py (cbx[v] - cbx[v-sy])
  const R cbxb = pz * (ey(u) - ey(u + sz)) - py * (ez(u) - ez(u + sy));
  const R cbyb = px * (ez(u) - ez(u + sx)) - pz * (ex(u) - ex(u + sz));
  const R cbzb = py * (ex(u) - ex(u + sy)) - px * (ey(u) - ey(u + sx));
  Fld<R> &o = Fb[u];
  o.cbx += cbxb;
  o.cby += cbyb;
  o.cbz += cbzb;
  o.jfx = -cj * ex(u);
  o.jfy = -cj * ey(u);
  o.jfz = -cj * ez(u);
}

// The magnetic part of energy_f (vacuum_energy_f_pipeline.h:44-75): per
// voxel R terms, FP64 block sums.
template <class R>
__global__ void k_benergy(const Fld<R> *F, Box B, double *part) {
  __shared__ double red[256];
  double acc = 0;
  const int ncell = B.nx * B.ny * B.nz;
  for (int l = blockIdx.x * blockDim.x + threadIdx.x; l < ncell;
       l += gridDim.x * blockDim.x) {
    const int x = 1 + l % B.nx, y = 1 + (l / B.nx) % B.ny,
              z = 1 + l / (B.nx * B.ny);
    const int v = vox(x, y, z, B.nx, B.ny);
    const R h = R(0.5);
    const Fld<R> &f = F[v], &fx = F[v + 1], &fy = F[v + B.sy],
                 &fz = F[v + B.sz];
    acc += (double)(h * (f.cbx * f.cbx + fx.cbx * fx.cbx));
    acc += (double)(h * (f.cby * f.cby + fy.cby * fy.cby));
    acc += (double)(h * (f.cbz * f.cbz + fz.cbz * fz.cbz));
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// d(energy)/d(field): the energy counts cbx[u] once as a voxel's own face
// and once as its +x neighbour's (likewise y, z).
template <class R>
__global__ void k_benergy_grad(Fld<R> *Fb, const Fld<R> *F, Box B, R scale) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= B.nv) return;
  int x, y, z;
  coords(B, u, x, y, z);
  Fld<R> o;
  o.ex = o.ey = o.ez = o.jfx = o.jfy = o.jfz = 0;
  const bool iy = y >= 1 && y <= B.ny, iz = z >= 1 && z <= B.nz,
             ix = x >= 1 && x <= B.nx;
  const R nxc = R((x >= 1 && x <= B.nx) + (x >= 2 && x <= B.nx + 1));
  const R nyc = R((y >= 1 && y <= B.ny) + (y >= 2 && y <= B.ny + 1));
  const R nzc = R((z >= 1 && z <= B.nz) + (z >= 2 && z <= B.nz + 1));
  o.cbx = (iy && iz) ? scale * F[u].cbx * nxc : R(0);
  o.cby = (ix && iz) ? scale * F[u].cby * nyc : R(0);
  o.cbz = (ix && iy) ? scale * F[u].cbz * nzc : R(0);
  Fb[u] = o;
}

// The caller's field array (vpic_field_t, or its FP64 twin with the same
// members as doubles) to the run's fields, and the particles' momentum
// adjoints out.
template <class R>
__global__ void k_fields_in(Fld<R> *F, const R *src, int stride_r, int nv) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  const R *s = src + (size_t)stride_r * v;
  Fld<R> o;
  o.ex = s[0];
  o.ey = s[1];
  o.ez = s[2];
  o.cbx = s[4];
  o.cby = s[5];
  o.cbz = s[6];
  o.jfx = o.jfy = o.jfz = 0;
  F[v] = o;
}

template <class R>
__global__ void k_split_pb(const R *pb, R *ub, R *db, int np) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= np) return;
  for (int k = 0; k < 3; k++) {
    ub[3 * (size_t)n + k] = pb[6 * (size_t)n + 3 + k];
    if (db) db[3 * (size_t)n + k] = pb[6 * (size_t)n + k];
  }
}

template <class R>
__global__ void k_fields_out(R *dst, const Fld<R> *Fb, int nv) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  const Fld<R> &f = Fb[v];
  R *o = dst + 6 * (size_t)v;
  o[0] = f.ex;
  o[1] = f.ey;
  o[2] = f.ez;
  o[3] = f.cbx;
  o[4] = f.cby;
  o[5] = f.cbz;
}

// ---------------------------------------------------------------------------
// host driver
// ---------------------------------------------------------------------------

// The device memory of a call, cut into the run's arrays: the caller's
// workspace, or one allocation (each of the dozens of arrays allocated and
// released on its own took longer than its steps; one allocation of 4.3 GB
// still takes 1 to 95 ms against 31 ms of kernels, hence the workspace).
struct Arena {
  char *p = nullptr;
  bool own = false;
  size_t used = 0;
  ~Arena() {
    if (own && p) (void)hipFree(p);
  }
  int reserve(size_t bytes, void *ws, int64_t ws_bytes) {
    if (ws) {
      if (((uintptr_t)ws & 255u) != 0 || (int64_t)bytes > ws_bytes)
        return vpic_set_error(VPIC_EINVAL, "adjoint run: the workspace of %lld "
                              "bytes must be 256-byte aligned and hold %zu",
                              (long long)ws_bytes, bytes);
      p = (char *)ws;
      return VPIC_OK;
    }
    const hipError_t e = hipMalloc((void **)&p, bytes < 256 ? 256 : bytes);
    if (e != hipSuccess) {
      p = nullptr;
      return vpic_set_error(VPIC_ENOMEM, "adjoint: hipMalloc(%zu): %s", bytes,
                            hipGetErrorString(e));
    }
    own = true;
    return VPIC_OK;
  }
  static size_t room(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
  // (first without memory to count, then with it to cut)
  template <class X>
  X *cut(size_t bytes) {
    X *x = (X *)(p ? p + used : nullptr);
    used += room(bytes);
    return x;
  }
};

inline dim3 cover(int64_t n, int bs = 256) {
  int64_t b = (n + bs - 1) / bs;
  return dim3((unsigned)(b < 1 ? 1 : b));
}

template <class R>
struct Run {
  Box B;
  GridDev G;
  Coef<R> C;
  int np = 0;
  hipStream_t s = nullptr;
  Tiles T;
  int nblk = 0;  // workgroups of a push
  Part<R> *p = nullptr, *p2 = nullptr;
  Fld<R> *F = nullptr;
  R *fi = nullptr, *acc = nullptr, *wbuf = nullptr;
  int *err = nullptr, *keys = nullptr;
  double *part = nullptr;
  int eblocks = 256;
  double escale = 0;  // 0.5 eps0 dV

  int setup(const vpic_grid_t *g, int np_, float q, float m, hipStream_t st) {
    B = {g->nx, g->ny, g->nz, g->sy, g->sz, g->nv};
    G = make_grid_dev(g);
    G.neighbor = nullptr;
    np = np_;
    s = st;
    // tiles where the particles can be sorted by cell
    const bool tiled = sort_keys_fit(g) &&
                       (int64_t)np * AT_SPARSE >=
                           (int64_t)B.nx * B.ny * B.nz;
    T.nt[0] = tiled ? (B.nx + AT_X - 1) / AT_X : 0;
    T.nt[1] = tiled ? (B.ny + AT_Y - 1) / AT_Y : 0;
    T.nt[2] = tiled ? (B.nz + AT_Z - 1) / AT_Z : 0;
    const int share = (int)(((int64_t)np / AT_CHUNKS + AT_BS - 1) / AT_BS) *
                      AT_BS;
    T.chunk = share < AT_BS ? AT_BS : share > AT_CHUNK ? AT_CHUNK : share;
    nblk = tiled ? T.nt[0] * T.nt[1] * T.nt[2]
                 : (int)(((int64_t)np + T.chunk - 1) / T.chunk);
    // advance_p_pipeline.cc:279-283 (in float for the FP32 run)
    const R rq = q, rm = m, dt = g->dt, c = g->cvac;
    C.qdt_2mc = (rq * dt) / (2 * rm * c);
    C.cdt[0] = c * dt * R(g->rdx);
    C.cdt[1] = c * dt * R(g->rdy);
    C.cdt[2] = c * dt * R(g->rdz);
    C.qsp = rq;
    const R frac = R(0.5);
    C.bp[0] = g->nx > 1 ? frac * c * dt * R(g->rdx) : R(0);
    C.bp[1] = g->ny > 1 ? frac * c * dt * R(g->rdy) : R(0);
    C.bp[2] = g->nz > 1 ? frac * c * dt * R(g->rdz) : R(0);
    const R one = 1;
    C.ep[0] = (g->nx > 1 ? (one + R(0)) * c * dt * R(g->rdx) : R(0)) * one;
    C.ep[1] = (g->ny > 1 ? (one + R(0)) * c * dt * R(g->rdy) : R(0)) * one;
    C.ep[2] = (g->nz > 1 ? (one + R(0)) * c * dt * R(g->rdz) : R(0)) * one;
    C.cj = dt / R(g->eps0);
    // unload_accumulator_pipeline.cc:137-139: in double, stored in R
    C.uc[0] = (R)(0.25 * g->rdy * g->rdz / g->dt);
    C.uc[1] = (R)(0.25 * g->rdz * g->rdx / g->dt);
    C.uc[2] = (R)(0.25 * g->rdx * g->rdy / g->dt);
    escale = 0.5 * (double)g->eps0 * (double)g->dV;
    return VPIC_OK;
  }

#define ADJ_LAUNCH(kern, grid, ...)                                   \
  do {                                                                \
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, __VA_ARGS__);     \
    VPIC_LAUNCHED(#kern);                                             \
  } while (0)

  int load() {
    ADJ_LAUNCH(k_load<R>, cover(B.nv), fi, (const Fld<R> *)F, B);
    return VPIC_OK;
  }

  bool tiled() const { return T.nt[0] > 0; }

  // Sort the particles of step n by cell (p and p2 swap roles), with the
  // permutation and the partition kept in perm and rows.
  int sort(const vpic_grid_t *g, int *perm, int *rows) {
    ADJ_LAUNCH(k_keys<R>, dim3(nkeyblk()), (const Part<R> *)p, np, keys);
    int rc, *order, *sorted;
    SortScratchUse use;
    if ((rc = use.begin(s)) ||
        (rc = device_sort_keys(keys, np, g, &order, &sorted, use, s)))
      return rc;
    VPIC_HIP(hipMemcpyAsync(perm, order, sizeof(int) * (size_t)np,
                            hipMemcpyDeviceToDevice, s));
    ADJ_LAUNCH(k_partition, cover((int64_t)B.nv + 1), (const int *)sorted, np,
               B.nv, rows);
    if ((rc = permute(p, perm, p2))) return rc;
    std::swap(p, p2);
    return VPIC_OK;
  }

  int nkeyblk() const {
    const int64_t b = ((int64_t)np + 255) / 256;
    return (int)(b < 4096 ? b : 4096);
  }

  int permute(const Part<R> *in, const int *perm, Part<R> *out) {
    ADJ_LAUNCH(k_permute<R>, cover((int64_t)np * (sizeof(Part<R>) / 16)), in,
               perm, np, out);
    return VPIC_OK;
  }

  // One step (advance.cc:25-185 on a periodic box, one species) of the
  // particles `from` into `to` (may be the same), whose rows the partition
  // `rows` gives; fi holds the interpolators of the step's fields on entry
  // and of the new fields on return.
  int step(const Part<R> *from, Part<R> *to, const int *rows) {
    ADJ_LAUNCH(k_fill<R>, cover(12 * (int64_t)B.nv), acc, (size_t)12 * B.nv,
               R(0));
    if (np > 0) {
      ADJ_LAUNCH(k_push_fwd<R>, dim3(nblk), from, to, np, rows, (const R *)fi,
                 acc, wbuf, C, G, B, T, err);
      if (tiled()) {
        auto merge = k_merge<R, 12>;
        ADJ_LAUNCH(merge, cover((int64_t)B.nx * B.ny * B.nz), acc,
                   (const R *)wbuf, B, T);
      }
    }
    ADJ_LAUNCH(k_unload_advance_b<R>, cover(B.nv), F, (const R *)acc, C, B);
    const int fold_blocks = cover(fold_places(B)).x;
    ADJ_LAUNCH(k_fold_jf_ghost_b<R>, dim3(fold_blocks + cover(B.nv).x), F, B,
               fold_blocks);
    ADJ_LAUNCH(k_advance_e<R>, cover(B.nv), F, C, B);
    ADJ_LAUNCH(k_advance_b<R>, cover(B.nv), F, C, B);
    return load();
  }

  int energy(double *out) {
    ADJ_LAUNCH(k_benergy<R>, dim3(eblocks), (const Fld<R> *)F, B, part);
    std::vector<double> h(eblocks);
    VPIC_HIP(hipMemcpyAsync(h.data(), part, sizeof(double) * eblocks,
                            hipMemcpyDeviceToHost, s));
    VPIC_HIP(hipStreamSynchronize(s));
    double e = 0;
    for (double v : h) e += v;
    *out = e * escale;
    return VPIC_OK;
  }

  // A particle in no cell belongs to no tile: refused before the first step.
  int check_cells() {
    if (np == 0) return VPIC_OK;
    int h = 0;
    ADJ_LAUNCH(k_check_cells<R>, dim3(nkeyblk()), (const Part<R> *)p, np, B,
               err + 1);
    VPIC_HIP(hipMemcpyAsync(&h, err + 1, sizeof(int), hipMemcpyDeviceToHost,
                            s));
    VPIC_HIP(hipStreamSynchronize(s));
    if (h)
      return vpic_set_error(VPIC_EINVAL,
                            "adjoint run: %d particles are in no cell of the "
                            "grid (a voxel outside it or a ghost voxel)", h);
    return VPIC_OK;
  }

  int check_err() {
    int h = 0;
    VPIC_HIP(hipMemcpyAsync(&h, err, sizeof(int), hipMemcpyDeviceToHost, s));
    VPIC_HIP(hipStreamSynchronize(s));
    if (h)
      return vpic_set_error(VPIC_EINVAL,
                            "adjoint run: %d particles left the periodic box "
                            "(the differentiated run has no particle "
                            "boundaries)", h);
    return VPIC_OK;
  }

  // Reverse of one step from its starting state (p_n in the order of `rows`,
  // F_n), with pb and Fb the adjoint of the state after the step on entry,
  // before it on return.
  int step_T(const Part<R> *pn, const int *rows, const Fld<R> *Fn, R *pb,
             Fld<R> *Fb, R *fib, R *accb) {
    ADJ_LAUNCH(k_advance_b_T<R>, cover(B.nv), Fb, C, B);
    ADJ_LAUNCH(k_advance_e_T<R>, cover(B.nv), Fb, C, B);
    ADJ_LAUNCH(k_ghost_b_T<R>, cover(B.nv), Fb, B);
    ADJ_LAUNCH(k_advance_b_T<R>, cover(B.nv), Fb, C, B);
    ADJ_LAUNCH(k_fold_jf_T<R>, cover(fold_places(B)), Fb, B);
    ADJ_LAUNCH(k_unload_T<R>, cover(B.nv), accb, (const Fld<R> *)Fb, C, B);
    ADJ_LAUNCH(k_load<R>, cover(B.nv), fi, Fn, B);
    ADJ_LAUNCH(k_fill<R>, cover((int64_t)NI * B.nv), fib, (size_t)NI * B.nv,
               R(0));
    if (np > 0) {
      ADJ_LAUNCH(k_push_rev<R>, dim3(nblk), pn, np, rows, (const R *)fi,
                 (const R *)accb, pb, fib, wbuf, C, G, B, T);
      if (tiled()) {
        auto merge = k_merge<R, NI>;
        ADJ_LAUNCH(merge, cover((int64_t)B.nx * B.ny * B.nz), fib,
                   (const R *)wbuf, B, T);
      }
    }
    ADJ_LAUNCH(k_load_T<R>, cover(B.nv), Fb, (const R *)fib, B);
    return VPIC_OK;
  }
#undef ADJ_LAUNCH
};

int check_periodic(const vpic_grid_t *g) {
  if (!g || g->nx < 1 || g->ny < 1 || g->nz < 1)
    return vpic_set_error(VPIC_EINVAL, "adjoint run: bad grid");
  if (g->sy != g->nx + 2 || g->sz != (g->ny + 2) * g->sy ||
      g->nv != (g->nz + 2) * g->sz)
    return vpic_set_error(VPIC_EINVAL, "adjoint run: inconsistent strides");
  for (int k = 0; k < 6; k++)
    if (g->pbc[k] != VPIC_BC_PERIODIC || g->fbc[k] != VPIC_BC_PERIODIC)
      return vpic_set_error(VPIC_EUNSUPPORTED,
                            "adjoint run: only periodic boxes are "
                            "differentiated (face %d)", k);
  return VPIC_OK;
}

// The forward with checkpoints, then (when grads are wanted) the reverse; or
// only the bytes that takes, when `want` is given.
template <class R>
int adjoint_run(const void *p0, int np, float q, float m, const void *f0,
                const vpic_grid_t *g, int n_step, int ckpt, bool grads,
                double *host_L, void *u_bar, void *d_bar, void *f_bar,
                void *ws, int64_t ws_bytes, int64_t *want, hipStream_t s) {
  int rc;
  if ((rc = check_periodic(g))) return rc;
  if (np < 0 || n_step < 0 ||
      (!want && ((np > 0 && !p0) || !f0 || !host_L)))
    return vpic_set_error(VPIC_EINVAL, "adjoint run: bad arguments");
  if (ckpt < 1 || ckpt > n_step) ckpt = n_step > 0 ? n_step : 1;
  Run<R> run;
  run.setup(g, np, q, m, s);
  const int nv = g->nv;
  const size_t pbytes = sizeof(Part<R>) * (size_t)np;
  const size_t fbytes = sizeof(Fld<R>) * (size_t)nv;
  const size_t kbytes = sizeof(int) * (size_t)np;
  const size_t rbytes = sizeof(int) * ((size_t)nv + 1);
  const bool sorts = run.tiled() && np > 0;
  // checkpoints, and the states of one segment (all of it when shorter)
  const int nseg = grads ? n_step / ckpt + (n_step % ckpt ? 1 : 0) : 0;
  const int nst = grads && n_step > 0 ? ckpt : 0;
  // sorts kept: all for the reverse, the last one otherwise
  const int nsort = !sorts || n_step < 1 ? 0
                    : grads ? 1 + (n_step - 1) / SORT_EVERY : 1;
  std::vector<Part<R> *> cp(nseg), sp(nst);
  std::vector<Fld<R> *> cF(nseg), sF(nst);
  std::vector<int *> perm(nsort), rows(nsort);
  R *pb = nullptr, *pb2 = nullptr, *fib = nullptr, *accb = nullptr;
  Fld<R> *Fb = nullptr;
  Arena A;
  for (int pass = 0; pass < 2; pass++) {
    A.used = 0;
    run.p = A.cut<Part<R>>(pbytes);
    run.p2 = A.cut<Part<R>>(sorts ? pbytes : 0);
    run.keys = A.cut<int>(sorts ? kbytes : 0);
    run.F = A.cut<Fld<R>>(fbytes);
    run.fi = A.cut<R>(sizeof(R) * NI * (size_t)nv);
    run.acc = A.cut<R>(sizeof(R) * 12 * (size_t)nv);
    run.wbuf = A.cut<R>(run.tiled() ? sizeof(R) * (grads ? NI : 12) * AT_CELLS *
                                          (size_t)run.nblk
                                    : 0);
    run.err = A.cut<int>(64);
    run.part = A.cut<double>(sizeof(double) * run.eblocks);
    for (int k = 0; k < nsort; k++) {
      perm[k] = A.cut<int>(kbytes);
      rows[k] = A.cut<int>(rbytes);
    }
    for (int k = 0; k < nseg; k++) {
      cp[k] = A.cut<Part<R>>(pbytes);
      cF[k] = A.cut<Fld<R>>(fbytes);
    }
    for (int k = 0; k < nst; k++) {
      sp[k] = A.cut<Part<R>>(pbytes);
      sF[k] = A.cut<Fld<R>>(fbytes);
    }
    if (grads) {
      pb = A.cut<R>(sizeof(R) * 6 * (size_t)np);
      pb2 = A.cut<R>(sorts ? sizeof(R) * 6 * (size_t)np : 0);
      Fb = A.cut<Fld<R>>(fbytes);
      fib = A.cut<R>(sizeof(R) * NI * (size_t)nv);
      accb = A.cut<R>(sizeof(R) * 12 * (size_t)nv);
    }
    if (want) {
      *want = (int64_t)A.used;
      return VPIC_OK;
    }
    if (pass == 0 && (rc = A.reserve(A.used, ws, ws_bytes))) return rc;
  }
  VPIC_HIP(hipMemsetAsync(run.err, 0, 64, s));
  if (np) VPIC_HIP(hipMemcpyAsync(run.p, p0, pbytes, hipMemcpyDeviceToDevice, s));
  // the caller's fields: 20 (float) or 18 (double) R per record
  const int rstride = sizeof(R) == 4 ? 20 : 18;
  hipLaunchKernelGGL(k_fields_in<R>, cover(nv), dim3(256), 0, s, run.F,
                     (const R *)f0, rstride, nv);
  VPIC_LAUNCHED("k_fields_in");
  if ((rc = run.load())) return rc;
  if (n_step > 0 && (rc = run.check_cells())) return rc;
  // the sort in force at step n (none: null)
  auto rows_at = [&](int n) -> const int * {
    return nsort ? rows[grads ? n / SORT_EVERY : 0] : nullptr;
  };
  for (int n = 0; n < n_step; n++) {
    if (grads && n % ckpt == 0) {
      const int k = n / ckpt;
      if (np)
        VPIC_HIP(hipMemcpyAsync(cp[k], run.p, pbytes, hipMemcpyDeviceToDevice,
                                s));
      VPIC_HIP(hipMemcpyAsync(cF[k], run.F, fbytes, hipMemcpyDeviceToDevice,
                              s));
    }
    if (sorts && n % SORT_EVERY == 0) {
      const int k = grads ? n / SORT_EVERY : 0;
      if ((rc = run.sort(g, perm[k], rows[k]))) return rc;
    }
    if ((rc = run.step(run.p, run.p, rows_at(n)))) return rc;
  }
  if ((rc = run.check_err())) return rc;
  if ((rc = run.energy(host_L))) return rc;
  if (!grads) return VPIC_OK;

  // reverse
  hipLaunchKernelGGL(k_fill<R>, cover(6 * (int64_t)np), dim3(256), 0, s, pb,
                     (size_t)6 * np, R(0));
  VPIC_LAUNCHED("k_fill");
  hipLaunchKernelGGL(k_benergy_grad<R>, cover(nv), dim3(256), 0, s, Fb,
                     (const Fld<R> *)run.F, run.B, (R)run.escale);
  VPIC_LAUNCHED("k_benergy_grad");
  for (int k = nseg - 1; k >= 0; k--) {
    const int n0 = k * ckpt, n1 = n_step - n0 > ckpt ? n0 + ckpt : n_step;
    VPIC_HIP(hipMemcpyAsync(run.F, cF[k], fbytes, hipMemcpyDeviceToDevice, s));
    if ((rc = run.load())) return rc;
    // the segment's states: st[j] before step n0 + j, in the order of the
    // sort in force there
    std::vector<Part<R> *> st(n1 - n0);
    Part<R> *cur = cp[k];
    for (int n = n0; n < n1; n++) {
      const int j = n - n0;
      if (sorts && n % SORT_EVERY == 0) {
        // (a step into p2 here would be put in order into sp[j])
        if ((rc = run.permute(cur, perm[n / SORT_EVERY], sp[j]))) return rc;
        cur = sp[j];
      }
      st[j] = cur;
      VPIC_HIP(hipMemcpyAsync(sF[j], run.F, fbytes, hipMemcpyDeviceToDevice,
                              s));
      if (n + 1 < n1) {
        const bool next = sorts && (n + 1) % SORT_EVERY == 0;
        Part<R> *to = next ? run.p2 : sp[j + 1];
        if ((rc = run.step(cur, to, rows_at(n)))) return rc;
        cur = to;
      }
    }
    for (int n = n1 - 1; n >= n0; n--) {
      const int j = n - n0;
      if ((rc = run.step_T(st[j], rows_at(n), sF[j], pb, Fb, fib, accb)))
        return rc;
      if (sorts && n % SORT_EVERY == 0) {
        hipLaunchKernelGGL(k_unpermute<R>, cover(np), dim3(256), 0, s,
                           (const R *)pb, (const int *)perm[n / SORT_EVERY],
                           np, pb2);
        VPIC_LAUNCHED("k_unpermute");
        std::swap(pb, pb2);
      }
    }
  }
  if (np > 0) {
    hipLaunchKernelGGL(k_split_pb<R>, cover(np), dim3(256), 0, s,
                       (const R *)pb, (R *)u_bar, (R *)d_bar, np);
    VPIC_LAUNCHED("k_split_pb");
  }
  if (f_bar) {
    hipLaunchKernelGGL(k_fields_out<R>, cover(nv), dim3(256), 0, s,
                       (R *)f_bar, (const Fld<R> *)Fb, nv);
    VPIC_LAUNCHED("k_fields_out");
  }
  VPIC_HIP(hipStreamSynchronize(s));
  return VPIC_OK;
}

// (the lists of a run of very many steps may not fit the host's memory)
template <class F>
int no_throw(F run) {
  try {
    return run();
  } catch (const std::exception &e) {
    return vpic_set_error(VPIC_ENOMEM, "adjoint run: %s", e.what());
  }
}

}  // namespace

extern "C" int vpic_hip_adjoint_workspace(int32_t np, const vpic_grid_t *g,
                                          int32_t n_step,
                                          int32_t ckpt_interval,
                                          int32_t precision, int32_t grads,
                                          int64_t *bytes) {
  if (!bytes)
    return vpic_set_error(VPIC_EINVAL, "adjoint workspace: bytes is NULL");
  auto ask = [&](auto zero) {
    return no_throw([&] {
      return adjoint_run<decltype(zero)>(nullptr, np, 1.0f, 1.0f, nullptr, g,
                                         n_step, ckpt_interval, grads != 0,
                                         nullptr, nullptr, nullptr, nullptr,
                                         nullptr, 0, bytes, nullptr);
    });
  };
  if (precision == 4) return ask(0.0f);
  if (precision == 8) return ask(0.0);
  return vpic_set_error(VPIC_EINVAL, "adjoint run: precision %d (4 or 8)",
                        precision);
}

extern "C" int vpic_hip_adjoint_bfield_energy_ws(
    const void *p0, int32_t np, float q, float m, const void *f0,
    const vpic_grid_t *g, int32_t n_step, int32_t ckpt_interval,
    int32_t precision, double *host_energy, void *u_bar, void *d_bar,
    void *f_bar, void *workspace, int64_t workspace_bytes, void *stream) {
  const hipStream_t s = (hipStream_t)stream;
  const bool grads = u_bar != nullptr;
  if (precision == 4)
    return no_throw([&] {
      return adjoint_run<float>(p0, np, q, m, f0, g, n_step, ckpt_interval,
                                grads, host_energy, u_bar, d_bar, f_bar,
                                workspace, workspace_bytes, nullptr, s);
    });
  if (precision == 8)
    return no_throw([&] {
      return adjoint_run<double>(p0, np, q, m, f0, g, n_step, ckpt_interval,
                                 grads, host_energy, u_bar, d_bar, f_bar,
                                 workspace, workspace_bytes, nullptr, s);
    });
  return vpic_set_error(VPIC_EINVAL, "adjoint run: precision %d (4 or 8)",
                        precision);
}

extern "C" int vpic_hip_adjoint_bfield_energy(
    const void *p0, int32_t np, float q, float m, const void *f0,
    const vpic_grid_t *g, int32_t n_step, int32_t ckpt_interval,
    int32_t precision, double *host_energy, void *u_bar, void *d_bar,
    void *f_bar, void *stream) {
  return vpic_hip_adjoint_bfield_energy_ws(
      p0, np, q, m, f0, g, n_step, ckpt_interval, precision, host_energy,
      u_bar, d_bar, f_bar, nullptr, 0, stream);
}
