// hydro.hip -- hydro moments on gfx950: accumulate_hydro_p,
// clear / synchronize of the hydro array.
//
// Reference: src/species_advance/standard/pipeline/hydro_p_pipeline.cc
// (:17-210 per particle, :214-242 driver) and
// src/sf_interface/hydro_array.cc:131-311 (synchronize_hydro_array).
//
// Each particle's half E kick, half Boris rotation, velocity and trilinear
// node weights are the reference's expressions in the same order; the 14
// node sums differ only in summation order.
//
// A particle adds 112 numbers (8 nodes x 14 moments), so what costs is
// adding them up: a sort of the particle indices by their voxels as they are
// now (not as a partition of the last sort_p has them) lets 16 lanes sum the
// particles of one voxel in registers and add the lanes up with DPP; the
// voxels' 112 sums go to a buffer, slab by slab, and every node gathers the
// eight it takes.  No atomics.  1.5e7 particles on 72x64x50 cells that drifted
// by half a cell since the sort: 0.77 ms, of which the sort is 0.33 (6.5
// ms with LDS windows per tile, whose float atomics a drifted particle needs
// one by one).  Grids with an axis too long for that sort, sparse species and calls
// for which its memory is not there go particle by particle with global
// atomics.
#include "common.h"

namespace {

struct HydroCoef {
  float qsp, qdt_2mc, qdt_4mc2, mspc, c, r8V;
};

constexpr int HY_LANES = 16;  // lanes per voxel (one DPP row)
constexpr int HY_SUMS = 8 * 14;
// Fewer particles than one in HY_SPARSE cells go one by one: the starts, sums and
// nodes cost by the voxel, 0.4 to 0.6 ns, the atomics 6 ns a particle (256^3
// cells, 0.05, 0.1, 0.2 particles per cell: 8.2, 9.4, 10.5 ms sorted, 4.8, 9.6,
// 19.3 one by one; 64^3: 196, 217, 233 us and 119, 190, 337).
constexpr int HY_SPARSE = 12;
// Voxels whose sums (448 B each, 128 MiB in all) stay in the 256-MB cache
// between the kernel that writes them and the one that reads them.
constexpr int64_t HY_VOXELS = ((int64_t)128 << 20) / (4 * HY_SUMS);

// The per-particle part of accumulate_hydro_p_pipeline_scalar
// (hydro_p_pipeline.cc:65-172): node weights wn[8] and the 14 moments per
// node, m[k][c], added to acc.
__device__ __forceinline__ void hydro_particle(const float4 A, const float4 B,
                                               const vpic_interpolator_t *fi,
                                               const HydroCoef &C,
                                               float acc[8][14]) {
  const float one = 1.0, one_third = 1.0 / 3.0;
  float dx = A.x, dy = A.y, dz = A.z;
  float ux = B.x, uy = B.y, uz = B.z;
  const float w = B.w;
  const float4 e0 = reinterpret_cast<const float4 *>(fi)[0];
  const float4 e1 = reinterpret_cast<const float4 *>(fi)[1];
  const float4 e2 = reinterpret_cast<const float4 *>(fi)[2];
  const float4 b0 = reinterpret_cast<const float4 *>(fi)[3];
  const float2 b1 = reinterpret_cast<const float2 *>(fi)[8];
  float vx, vy, vz, ke_mc, t, w0, w1, w2, w3, w4, w5, w6, w7;
  ux += C.qdt_2mc * ((e0.x + dy * e0.y) + dz * (e0.z + dy * e0.w));
  uy += C.qdt_2mc * ((e1.x + dz * e1.y) + dx * (e1.z + dz * e1.w));
  uz += C.qdt_2mc * ((e2.x + dx * e2.y) + dy * (e2.z + dx * e2.w));
  w5 = b0.x + dx * b0.y;
  w6 = b0.z + dy * b0.w;
  w7 = b1.x + dz * b1.y;
  ke_mc = ux * ux + uy * uy + uz * uz;
  vz = sqrtf(one + ke_mc);
  ke_mc *= C.c / (vz + one);
  vz = C.c / vz;
  w0 = C.qdt_4mc2 * vz;
  w1 = w5 * w5 + w6 * w6 + w7 * w7;
  w2 = w0 * w0 * w1;
  w3 = w0 * (one + (one_third)*w2 * (one + 0.4f * w2));
  w4 = w3 / (one + w1 * w3 * w3);
  w4 += w4;
  w0 = ux + w3 * (uy * w7 - uz * w6);
  w1 = uy + w3 * (uz * w5 - ux * w7);
  w2 = uz + w3 * (ux * w6 - uy * w5);
  ux += w4 * (w1 * w7 - w2 * w6);
  uy += w4 * (w2 * w5 - w0 * w7);
  uz += w4 * (w0 * w6 - w1 * w5);
  vx = ux * vz;
  vy = uy * vz;
  vz = uz * vz;
  w0 = C.r8V * w;
  dx *= w0;
  w1 = w0 + dx;
  w0 -= dx;
  w3 = one + dy;
  w2 = w0 * w3;
  w3 *= w1;
  dy = one - dy;
  w0 *= dy;
  w1 *= dy;
  w7 = one + dz;
  w4 = w0 * w7;
  w5 = w1 * w7;
  w6 = w2 * w7;
  w7 *= w3;
  dz = one - dz;
  w0 *= dz;
  w1 *= dz;
  w2 *= dz;
  w3 *= dz;
  const float wn[8] = {w0, w1, w2, w3, w4, w5, w6, w7};
#pragma unroll
  for (int k = 0; k < 8; k++) {
    t = C.qsp * wn[k];
    acc[k][0] += t * vx;
    acc[k][1] += t * vy;
    acc[k][2] += t * vz;
    acc[k][3] += t;
    t = C.mspc * wn[k];
    const float px = t * ux, py = t * uy, pz = t * uz;
    acc[k][4] += px;
    acc[k][5] += py;
    acc[k][6] += pz;
    acc[k][7] += t * ke_mc;
    acc[k][8] += px * vx;
    acc[k][9] += py * vy;
    acc[k][10] += pz * vz;
    acc[k][11] += py * vz;
    acc[k][12] += pz * vx;
    acc[k][13] += px * vy;
  }
}

// Node offsets of the 8 trilinear weights (hydro_p_pipeline.cc:194-201):
// i, i+1, i+sy, i+sy+1, i+sz, i+sz+1, i+sz+sy, i+sz+sy+1.
__device__ __forceinline__ int node_off(int k, int sy, int sz) {
  return (k & 1) + ((k >> 1) & 1) * sy + (k >> 2) * sz;
}

// Flat: one lane per particle, global float atomics (no sort).
__global__ __launch_bounds__(256) void k_hydro_flat(
    const vpic_particle_t *__restrict__ p, int np,
    const vpic_interpolator_t *__restrict__ f0, float *__restrict__ hy,
    HydroCoef C, int nv, int sy, int sz, int *__restrict__ nbad) {
  for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n < np;
       n += (int64_t)gridDim.x * blockDim.x) {
    const float4 *pp = reinterpret_cast<const float4 *>(p + n);
    const float4 A = pp[0], B = pp[1];
    const int ii = __float_as_int(A.w);
    if ((unsigned)ii >= (unsigned)nv || ii + sz + sy + 1 >= nv) {
      atomicAdd(nbad, 1);
      continue;
    }
    float acc[8][14];
#pragma unroll
    for (int k = 0; k < 8; k++)
#pragma unroll
      for (int c = 0; c < 14; c++) acc[k][c] = 0.0f;
    hydro_particle(A, B, f0 + ii, C, acc);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      float *h = hy + 16 * (int64_t)(ii + node_off(k, sy, sz));
#pragma unroll
      for (int c = 0; c < 14; c++) atomic_add_f32(h + c, acc[k][c]);
    }
  }
}

// The particles' voxels as sort keys; one whose nodes are not all on the grid
// is counted and takes the last voxel, which no valid particle has.
__global__ __launch_bounds__(256) void k_hydro_keys(
    const vpic_particle_t *__restrict__ p, int np, int vmax, int nv,
    int *__restrict__ keys, int *__restrict__ nbad) {
  for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n < np;
       n += (int64_t)gridDim.x * blockDim.x) {
    int v = p[n].i;
    if ((unsigned)v >= (unsigned)vmax) {
      atomicAdd(nbad, 1);
      v = nv - 1;
    }
    keys[n] = v;
  }
}

// start[v] = the first place whose key is not below v (v = 0..nv).
__global__ __launch_bounds__(256) void k_hydro_starts(
    const int *__restrict__ keys, int np, int nv, int *__restrict__ start) {
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
  start[v] = lo;
}

// Level of the reduce-scatter of N values over a 16-lane row: the upper lanes
// of each pair keep the upper half of the values, the lower the lower, plus
// the partner's.
template <int CTRL, int N>
__device__ __forceinline__ void row_halve(bool upper, const float (&v)[2 * N],
                                          float (&o)[N]) {
#pragma unroll
  for (int k = 0; k < N; k++)
    o[k] = (upper ? v[k + N] : v[k]) +
           dpp_get<CTRL, 0xf>(upper ? v[k] : v[k + N]);
}

// Sums of the particles of voxels [v0, v1), 16 lanes each, to
// sums[(v - v0) * 112 + 14 node + moment]; nothing is written for a voxel
// without particles.
__global__ __launch_bounds__(256) void k_hydro_cells(
    const vpic_particle_t *__restrict__ p, const int *__restrict__ order,
    const int *__restrict__ start, const vpic_interpolator_t *__restrict__ f0,
    float *__restrict__ sums, HydroCoef C, int v0, int v1) {
  const int j = threadIdx.x & (HY_LANES - 1);
  const int v = v0 + (int)((blockIdx.x * (int64_t)blockDim.x + threadIdx.x) /
                           HY_LANES);
  int s = 0, e = 0;
  if (v < v1) {
    s = start[v];
    e = start[v + 1];
  }
  float acc[8][14];
#pragma unroll
  for (int k = 0; k < 8; k++)
#pragma unroll
    for (int c = 0; c < 14; c++) acc[k][c] = 0.0f;
  for (int k = s + j; k < e; k += HY_LANES) {
    const float4 *pp = reinterpret_cast<const float4 *>(p + order[k]);
    const float4 A = pp[0], B = pp[1];
    hydro_particle(A, B, f0 + v, C, acc);
  }
  // (whole rows run from here: the lanes of a row share a voxel)
  float a112[HY_SUMS], a56[56], a28[28], a14[14], a7[7];
#pragma unroll
  for (int k = 0; k < HY_SUMS; k++) a112[k] = acc[k / 14][k % 14];
  row_halve<0x140, 56>(j & 8, a112, a56);  // row_mirror
  row_halve<0x141, 28>(j & 4, a56, a28);   // row_half_mirror
  row_halve<0x1b, 14>(j & 2, a28, a14);    // quad_perm 3,2,1,0
  row_halve<0xb1, 7>(j & 1, a14, a7);      // quad_perm 1,0,3,2
  if (s < e) {
    float *o = sums + (int64_t)(v - v0) * HY_SUMS + 7 * j;
#pragma unroll
    for (int k = 0; k < 7; k++) o[k] = a7[k];
  }
}

// Nodes [n0, n1): 16 lanes each, one per moment, gather the eight voxels a node
// belongs to: voxel v of the node's own plane is at sums[112 (v - vu)], of the
// plane below at sums[112 (v - vl)].
__global__ __launch_bounds__(256) void k_hydro_nodes(
    const float *__restrict__ sums, const int *__restrict__ start,
    float *__restrict__ hy, int vl, int vu, int vmax, int n0, int n1, int sy,
    int sz) {
  const int c = threadIdx.x & 15;
  const int n = n0 + (int)((blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >>
                           4);
  if (n >= n1 || c >= 14) return;
  float s = 0.0f;
  bool any = false;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int v = n - node_off(k, sy, sz);
    if (v < 0 || v >= vmax || start[v] == start[v + 1]) continue;
    any = true;
    s += sums[((int64_t)v - (k < 4 ? vu : vl)) * HY_SUMS + 14 * k + c];
  }
  if (any) hy[16 * (int64_t)n + c] += s;
}

// synchronize_hydro_array (hydro_array.cc:131-311) for one domain: local
// faces doubled, then the periodic node planes of axis X take
// lw*h + rw*remote (lw = rw = 1 for equal cells).
__global__ void k_hydro_adjust(float *hy, int4 n, int4 s, int k) {
  const int X = k % 3, Y = (X + 1) % 3, Z = (X + 2) % 3;
  const int nn[3] = {n.x, n.y, n.z}, ss[3] = {s.x, s.y, s.z};
  const int plane = k >= 3 ? nn[X] + 1 : 1;
  const int wy = nn[Y] + 1, wz = nn[Z] + 1;
  for (int l = blockIdx.x * blockDim.x + threadIdx.x; l < wy * wz;
       l += gridDim.x * blockDim.x) {
    const int yy = 1 + l % wy, zz = 1 + l / wy;
    float *h = hy + 16 * (int64_t)(plane * ss[X] + yy * ss[Y] + zz * ss[Z]);
#pragma unroll
    for (int q = 0; q < 14; q++) h[q] *= 2;
  }
}

__global__ void k_hydro_fold(float *hy, int4 n, int4 s, int X, float lw,
                             float rw) {
  const int Y = (X + 1) % 3, Z = (X + 2) % 3;
  const int nn[3] = {n.x, n.y, n.z}, ss[3] = {s.x, s.y, s.z};
  const int wy = nn[Y] + 1, wz = nn[Z] + 1;
  for (int l = blockIdx.x * blockDim.x + threadIdx.x; l < wy * wz;
       l += gridDim.x * blockDim.x) {
    const int yy = 1 + l % wy, zz = 1 + l / wy;
    const int64_t off = yy * ss[Y] + zz * ss[Z];
    float *a = hy + 16 * (int64_t)(1 * ss[X] + off);
    float *b = hy + 16 * (int64_t)((nn[X] + 1) * ss[X] + off);
#pragma unroll
    for (int q = 0; q < 14; q++) {
      const float va = a[q], vb = b[q];
      b[q] = lw * vb + rw * va;
      a[q] = lw * va + rw * vb;
    }
  }
}

__global__ void k_hydro_clear_count(int *c) {
  if (threadIdx.x == 0) c[0] = 0;
}

__global__ __launch_bounds__(256) void k_hydro_zero(float4 *h, int64_t n4) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n4;
       i += (int64_t)gridDim.x * blockDim.x)
    h[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

struct HydroScratch {
  DeviceScratch nbad, keys, start, sums;
};
HydroScratch &hydro_scratch() {
  static thread_local HydroScratch s[16];
  int dev = 0;
  (void)hipGetDevice(&dev);
  return s[dev & 15];
}

inline int blocks_for(int64_t n, int bs) { return (int)((n + bs - 1) / bs); }

// The sums of all particles by sorted voxels; VPIC_ENOMEM, with nothing added
// to the moments, when its memory is not there.  (vmax: voxels whose eight
// nodes lie on the grid.)
int hydro_sorted(HydroScratch &S, SortScratchUse &use, vpic_hydro_t *h,
                 const vpic_particle_t *p, int np,
                 const vpic_interpolator_t *f, const vpic_grid_t *g,
                 const HydroCoef &C, int vmax, int *nbad, hipStream_t s) {
  int rc;
  // Nodes per slab.  Their voxels reach back by a plane, a row and a cell:
  // one range of voxels, as long as what it reaches back by is at most half
  // of it, or on larger planes (of more than 150,000 voxels) two, a row and a
  // cell longer than the slab each.  A voxel of two slabs is summed for both
  // (1500x1500x2 cells, 4 a cell: 6.5 ms, with particle-by-particle atomics
  // 13.9).
  const int row = g->sy + 1, back = g->sz + row;
  const bool two = 2 * (int64_t)back > HY_VOXELS;
  int64_t slab = two ? HY_VOXELS / 2 - row : HY_VOXELS - back;
  if (slab > g->nv) slab = g->nv;
  if ((rc = scratch_reserve(S.keys, sizeof(int) * (size_t)np)) ||
      (rc = scratch_reserve(S.start, sizeof(int) * ((size_t)g->nv + 1))) ||
      (rc = scratch_reserve(S.sums, sizeof(float) * HY_SUMS *
                                        (size_t)(two ? 2 * (slab + row)
                                                     : slab + back))))
    return rc;
  int *keys = (int *)S.keys.ptr, *start = (int *)S.start.ptr;
  float *sums = (float *)S.sums.ptr;
  int nb = blocks_for(np, 256);
  if (nb > 8192) nb = 8192;
  hipLaunchKernelGGL(k_hydro_keys, dim3(nb), dim3(256), 0, s, p, np, vmax,
                     g->nv, keys, nbad);
  VPIC_LAUNCHED("k_hydro_keys");
  int *order, *sorted;
  if ((rc = use.begin(s)) ||
      (rc = device_sort_keys(keys, np, g, &order, &sorted, use, s)))
    return rc;
  hipLaunchKernelGGL(k_hydro_starts, dim3(blocks_for((int64_t)g->nv + 1, 256)),
                     dim3(256), 0, s, (const int *)sorted, np, g->nv, start);
  VPIC_LAUNCHED("k_hydro_starts");
  for (int64_t n0 = 0; n0 < g->nv; n0 += slab) {
    const int64_t n1 = n0 + slab < g->nv ? n0 + slab : g->nv;
    // voxels [v0, v1) to sums from voxel `at` on; none when there are none
    auto cells = [&](int64_t v0, int64_t v1, int64_t at) {
      if (v0 < 0) v0 = 0;
      if (v1 > vmax) v1 = vmax;
      if (v1 <= v0) return;
      hipLaunchKernelGGL(k_hydro_cells,
                         dim3(blocks_for((v1 - v0) * HY_LANES, 256)),
                         dim3(256), 0, s, p, (const int *)order,
                         (const int *)start, f, sums + (v0 - at) * HY_SUMS,
                         C, (int)v0, (int)v1);
    };
    // the voxel at the start of sums for the plane below and the node's own
    int64_t vl = n0 - back, vu = vl;
    if (two) {
      cells(n0 - back, n1 - g->sz, vl);
      VPIC_LAUNCHED("k_hydro_cells");
      vu = n0 - row - (slab + row);
      cells(n0 - row, n1, vu);
    } else {
      cells(n0 - back, n1, vl);
    }
    VPIC_LAUNCHED("k_hydro_cells");
    hipLaunchKernelGGL(k_hydro_nodes, dim3(blocks_for((n1 - n0) * 16, 256)),
                       dim3(256), 0, s, (const float *)sums,
                       (const int *)start, (float *)h, (int)vl, (int)vu,
                       vmax, (int)n0, (int)n1, g->sy, g->sz);
    VPIC_LAUNCHED("k_hydro_nodes");
  }
  return VPIC_OK;
}

}  // namespace

int launch_clear_hydro(vpic_hydro_t *h, const vpic_grid_t *g, hipStream_t s) {
  const int64_t n4 = (int64_t)g->nv * 4;
  int nb = blocks_for(n4, 256);
  if (nb > 65536) nb = 65536;
  hipLaunchKernelGGL(k_hydro_zero, dim3(nb), dim3(256), 0, s, (float4 *)h, n4);
  VPIC_LAUNCHED("k_hydro_zero");
  return VPIC_OK;
}

int launch_accumulate_hydro_p(vpic_hydro_t *h, const vpic_particle_t *p,
                              int np, float q, float m,
                              const vpic_interpolator_t *f,
                              const vpic_grid_t *g, const int *partition,
                              hipStream_t s) {
  HydroScratch &S = hydro_scratch();
  int rc;
  if ((rc = scratch_reserve(S.nbad, 64))) return rc;
  int *nbad = (int *)S.nbad.ptr;
  hipLaunchKernelGGL(k_hydro_clear_count, dim3(1), dim3(64), 0, s, nbad);
  VPIC_LAUNCHED("k_hydro_clear_count");
  // hydro_p_pipeline.cc:31-36, 232-234
  HydroCoef C;
  C.qsp = q;
  C.qdt_2mc = (q * g->dt) / (2 * m * g->cvac);
  C.qdt_4mc2 = C.qdt_2mc / (2 * g->cvac);
  C.mspc = g->cvac * m;
  C.c = g->cvac;
  C.r8V = g->r8V;
  // (the voxels are the particles' own: the partition of their last sort is
  // not needed)
  (void)partition;
  SortScratchUse use;
  // voxels whose eight nodes lie on the grid
  const int vmax = g->nv - g->sz - g->sy - 1;
  rc = VPIC_ENOMEM;
  const int64_t cells = (int64_t)g->nx * g->ny * g->nz;
  if (np > 0 && sort_keys_fit(g) && (int64_t)np * HY_SPARSE >= cells) {
    rc = hydro_sorted(S, use, h, p, np, f, g, C, vmax, nbad, s);
    if (rc && rc != VPIC_ENOMEM) return rc;
    if (rc) {
      hipLaunchKernelGGL(k_hydro_clear_count, dim3(1), dim3(64), 0, s, nbad);
      VPIC_LAUNCHED("k_hydro_clear_count");
    }
  }
  if (np > 0 && rc) {
    int nb = blocks_for(np, 256);
    if (nb > 16384) nb = 16384;
    hipLaunchKernelGGL(k_hydro_flat, dim3(nb), dim3(256), 0, s, p, np, f,
                       (float *)h, C, g->nv, g->sy, g->sz, nbad);
    VPIC_LAUNCHED("k_hydro_flat");
  }
  int h_bad = 0;
  VPIC_HIP(hipMemcpyAsync(&h_bad, nbad, sizeof(int), hipMemcpyDeviceToHost, s));
  VPIC_HIP(hipStreamSynchronize(s));
  use.synchronised();
  if (h_bad)
    return vpic_set_error(VPIC_EINVAL,
                          "accumulate_hydro_p: %d particles with a voxel "
                          "index outside the interior were skipped", h_bad);
  return VPIC_OK;
}

int launch_synchronize_hydro(vpic_hydro_t *h, const vpic_grid_t *g,
                             hipStream_t s) {
  const int4 n = make_int4(g->nx, g->ny, g->nz, 0);
  const int4 st = make_int4(1, g->sy, g->sz, 0);
  int mm = g->nx > g->ny ? g->nx : g->ny;
  mm = mm > g->nz ? mm : g->nz;
  int fb = blocks_for((int64_t)(mm + 1) * (mm + 1), 256);
  if (fb > 1024) fb = 1024;
  for (int k = 0; k < 6; k++) {
    if (g->fbc[k] == VPIC_BC_PERIODIC) continue;
    hipLaunchKernelGGL(k_hydro_adjust, dim3(fb), dim3(256), 0, s, (float *)h,
                       n, st, k);
    VPIC_LAUNCHED("k_hydro_adjust");
  }
  for (int X = 0; X < 3; X++) {
    if (g->fbc[X] != VPIC_BC_PERIODIC || g->fbc[X + 3] != VPIC_BC_PERIODIC)
      continue;
    // hydro_array.cc END_RECV: the weights in float as there
    const float d = X == 0 ? g->dx : X == 1 ? g->dy : g->dz;
    float rw = d, lw = rw + d;
    rw /= lw;
    lw = d / lw;
    lw += lw;
    rw += rw;
    hipLaunchKernelGGL(k_hydro_fold, dim3(fb), dim3(256), 0, s, (float *)h, n,
                       st, X, lw, rw);
    VPIC_LAUNCHED("k_hydro_fold");
  }
  return VPIC_OK;
}
