// collision.hip -- the Takizuka-Abe binary collision operator
// (src/collision/pipeline/takizuka_abe_pipeline.cc:81-215) over the sort
// partition.
//
// The reference runs the voxels in order on a pipeline's sequential SFMT
// generator.  Here every voxel draws from its own counter-based stream
// (Philox4x32-10, Salmon et al., SC'11: key = the seed, counter = {draw/4,
// voxel, call}), so the voxels are independent and the result does not
// depend on the launch shape.  Within a voxel the operations are the
// reference's, in its order: the Fisher-Yates shuffle of species i with
// rejection sampling, the three-particle start of an odd intra-species
// voxel, the pairing of the larger set round the smaller, and
// takizuka_abe_collision's float arithmetic (the scattering phase's sin and
// cos as correctly rounded floats).  Compiled without FMA contraction, like
// the rest.
//
// Only the shuffle and the density sums of a voxel are sequential: each
// collision takes exactly four words of the voxel's stream, and every
// particle meets its partners in one chain (round the smaller set), so the
// chains of a voxel are independent.  A workgroup takes a batch of voxels:
// the momenta (of both species) go to LDS, all lanes draw the shuffle's
// words, one lane per voxel swaps indices, then a lane runs each chain with
// its own words of the stream, and the particles are stored in their shuffled
// places.  The same draws and the same arithmetic as voxel by voxel on one
// lane, bit for bit.
// 48^3 cells, 64 electrons and ions in each: 269 us a call within a species
// (88e6 wavefront instructions, half of the time on the vector units), 462 us
// between two (537 with the other species' particles left in memory), against
// 1118 us for either with one lane per voxel, a chain of dependent memory
// accesses on 7 wavefronts a CU.
#include "common.h"

#include <cfloat>

namespace {

struct TaRng {
  uint32_t key0, key1, ctr[4], buf[4];
  uint32_t n;

  __device__ void philox() {
    uint32_t c0 = ctr[0], c1 = ctr[1], c2 = ctr[2], c3 = ctr[3];
    uint32_t k0 = key0, k1 = key1;
#pragma unroll
    for (int r = 0; r < 10; r++) {
      const uint32_t hi0 = __umulhi(0xD2511F53u, c0), lo0 = 0xD2511F53u * c0;
      const uint32_t hi1 = __umulhi(0xCD9E8D57u, c2), lo1 = 0xCD9E8D57u * c2;
      c0 = hi1 ^ c1 ^ k0;
      c1 = lo1;
      c2 = hi0 ^ c3 ^ k1;
      c3 = lo0;
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    buf[0] = c0; buf[1] = c1; buf[2] = c2; buf[3] = c3;
  }
  __device__ uint32_t u32() {
    if ((n & 3) == 0) {
      ctr[0] = n >> 2;
      philox();
    }
    return buf[n++ & 3];
  }
};

// The four words of a voxel's stream from word n on.
__device__ __forceinline__ void ta_words(TaRng &rng, uint32_t n,
                                         uint32_t (&w)[4]) {
  rng.ctr[0] = n >> 2;
  rng.philox();
  uint32_t a[4], b[4];
#pragma unroll
  for (int k = 0; k < 4; k++) a[k] = rng.buf[k];
  const uint32_t r = n & 3;
  if (r) {
    rng.ctr[0] = (n >> 2) + 1;
    rng.philox();
  }
#pragma unroll
  for (int k = 0; k < 4; k++) b[k] = rng.buf[k];
#pragma unroll
  for (int k = 0; k < 4; k++)
    w[k] = r == 0   ? a[k]
           : r == 1 ? (k < 3 ? a[k + 1 & 3] : b[0])
           : r == 2 ? (k < 2 ? a[k + 2 & 3] : b[k - 2 & 3])
                    : (k < 1 ? a[3] : b[k - 1 & 3]);
}

__device__ __forceinline__ float ta_unit(uint32_t w) {
  return (float)(w >> 8) * (1.0f / 16777216.0f);
}
__device__ __forceinline__ float ta_normal(uint32_t w0, uint32_t w1) {
  // Box-Muller in double
  const double u1 = ((double)(w0 >> 8) + 1.0) * (1.0 / 16777216.0);
  const double u2 = (double)(w1 >> 8) * (1.0 / 16777216.0);
  return (float)(sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2));
}

// takizuka_abe_collision (takizuka_abe_pipeline.cc:14-79) of momenta a and b
// (x, y, z, weight) with the collision's four words.
__device__ void ta_collide(float4 &a, float4 &b, float mu_i, float mu_j,
                           float std, const uint32_t (&w)[4]) {
  float dd, ur, urx, ury, urz, tx, ty, tz, t0, t1, t2;
  urx = a.x - b.x;
  ury = a.y - b.y;
  urz = a.z - b.z;
  const float wi = a.w, wj = b.w;
  // the axis of the smallest component (d0), its cyclic successors d1, d2
  int d0 = 0;
  t0 = urx * urx; t1 = t0; ur = t0;
  t0 = ury * ury;
  if (t0 < t1) { d0 = 1; t1 = t0; }
  ur += t0;
  t0 = urz * urz;
  if (t0 < t1) d0 = 2;
  ur += t0;
  ur = sqrtf(ur);
  t1 = d0 == 0 ? ury : d0 == 1 ? urz : urx;  // component d1
  t2 = d0 == 0 ? urz : d0 == 1 ? urx : ury;  // component d2
  t0 = 1 / sqrtf(t1 * t1 + t2 * t2 + FLT_MIN);
  const float s1_ = t0 * t2, s2_ = -t0 * t1;  // components d1, d2 of t
  tx = d0 == 0 ? 0.0f : d0 == 1 ? s2_ : s1_;
  ty = d0 == 0 ? s1_ : d0 == 1 ? 0.0f : s2_;
  tz = d0 == 0 ? s2_ : d0 == 1 ? s1_ : 0.0f;
  t0 = 1;
  t2 = 1 / ur;
  t1 = std * sqrtf(t2) * t2;
  if (t0 < t1) t1 = t0;
  dd = t1 * ta_normal(w[0], w[1]);
  t0 = 2 * dd / (1 + dd * dd);
  t1 = (float)(2 * M_PI * ta_unit(w[2]));
  // The reference's sin(t1)/cos(t1) of a float take the float overloads
  // (C++ <cmath>); they are formed here as the double functions rounded to
  // float (the correctly rounded float value, identical on host and
  // device), then multiplied in float as there.
  {
    double sn, cs;
    sincos((double)t1, &sn, &cs);
    t2 = t0 * (float)sn;
    t1 = t0 * ur * (float)cs;
  }
  t0 *= -dd;
  const float s0 = (t0 * urx + t1 * tx) + t2 * (ury * tz - urz * ty);
  const float s1 = (t0 * ury + t1 * ty) + t2 * (urz * tx - urx * tz);
  const float s2 = (t0 * urz + t1 * tz) + t2 * (urx * ty - ury * tx);
  t0 = ta_unit(w[3]);
  t1 = mu_i;
  t2 = mu_j;
  if (wj < wi && wi * t0 > wj) t1 = 0;
  if (wi < wj && wj * t0 > wi) t2 = 0;
  a.x += t1 * s0;
  a.y += t1 * s1;
  a.z += t1 * s2;
  b.x -= t2 * s0;
  b.y -= t2 * s1;
  b.z -= t2 * s2;
}

__global__ void k_ta_clear(int *a) {
  if (threadIdx.x < 2) a[threadIdx.x] = 0;
}

DeviceScratch &collision_scratch() {
  static thread_local DeviceScratch s[16];
  int dev = 0;
  (void)hipGetDevice(&dev);
  return s[dev & 15];
}

struct TaArgs {
  vpic_particle_t *pi, *pj;
  const int *part_i, *part_j;
  int np_i, np_j, same, v1;
  float mu_i, mu_j, dtinterval_dV;
  double cvar;
  uint32_t key0, key1, call0, call1;
};

// What a voxel's chains need: species i's particles after the shuffle (places
// k0.. of nk), species j's (l0.. of nl), the stream's position, the spreads.
struct TaVoxel {
  int k0, nk, l0, nl;
  uint32_t n;
  float std, std3;
  int ii, rn;   // collisions of a chain: ii, one more of the first rn
  bool triple;  // and before them the odd three
};

// Species j's particles of voxel v; false (and none) where its partition does
// not index them.
__device__ __forceinline__ bool ta_other(const TaArgs &a, int v, int &l0,
                                         int &nl) {
  l0 = a.part_j[v];
  nl = a.part_j[v + 1] - l0;
  if (!nl || (l0 >= 0 && nl > 0 && l0 + nl <= a.np_j)) return true;
  nl = 0;
  return false;
}

// The reference's steps between the shuffle and the collisions: pairs of one
// species (the odd three first), or the sets of two (V.l0, V.nl given); false
// when nothing collides.  `density` is species i's, `wj(k)` the weight of species j's k-th.
template <class Weight>
__device__ __forceinline__ bool ta_pairing(const TaArgs &a, int v,
                                           float density, TaVoxel &V,
                                           Weight wj) {
  V.triple = false;
  V.std3 = 0.0f;
  if (a.same) {
    if (V.nk % 2 && V.nk >= 3) {
      V.std3 = sqrtf((float)(0.5 * density * a.cvar * a.dtinterval_dV));
      V.triple = true;
      V.nk -= 3;
      V.k0 += 3;
    }
    V.nl = V.nk = V.nk / 2;
    V.l0 = V.k0 + V.nk;
    V.ii = 1;
    V.rn = 0;
    if (!V.nk) return V.triple;
    V.std = sqrtf((float)(a.cvar * density * a.dtinterval_dV));
    return true;
  }
  if (!V.nl) return false;
  float density_l = 0;
#pragma unroll 8
  for (int i = 0; i < V.nl; ++i) density_l += wj(V.l0 + i);
  V.std = sqrtf((float)(a.cvar * (density_l > density ? density : density_l) *
                        a.dtinterval_dV));
  const int big = V.nk > V.nl ? V.nk : V.nl, small = V.nk > V.nl ? V.nl : V.nk;
  V.ii = big / small;
  V.rn = big - V.ii * small;
  return true;
}

// Chain c of a voxel: the c-th particle of the smaller set (species i's when
// they are equal) meets `len` of the larger from the `many`-th on, which is
// also the number of the voxel's collisions before it.
__device__ __forceinline__ void ta_chain(const TaVoxel &V, int c, int &many,
                                         int &len) {
  len = c < V.rn ? V.ii + 1 : V.ii;
  many = c * V.ii + (c < V.rn ? c : V.rn);
}

__device__ __forceinline__ void ta_stream(const TaArgs &a, int v,
                                          TaRng &rng) {
  rng.key0 = a.key0;
  rng.key1 = a.key1;
  rng.ctr[1] = (uint32_t)v;
  rng.ctr[2] = a.call0;
  rng.ctr[3] = a.call1;
  rng.n = 0;
}

// Sum over the lanes up to this one.
template <class T>
__device__ __forceinline__ T wave_incl(T x) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T o = __shfl_up(x, d);
    if (lane_id() >= d) x += o;
  }
  return x;
}

__device__ __forceinline__ float4 *ta_mom(vpic_particle_t *p, int k) {
  return reinterpret_cast<float4 *>(p + k) + 1;
}

// Particles of a batch, both species': with 28 KiB of momenta four workgroups
// share a CU's LDS.  Voxels in a batch: one lane each shuffles them.
constexpr int TA_BS = 256, TA_CAP = 1792, TA_VOX = 64;
// Where many voxels hold few particles a batch is 64 of them with a handful of
// chains, and a lane per voxel is faster: below TA_SPARSE particles of one
// species, TA_SPARSE2 of two together, in at least TA_SPARSE_CELLS cells (128^3
// cells, 1, 2, 4, 6 of each species: 441, 477, 552, 648 us a call within one in
// batches, 195, 252, 422, 857 with a lane per voxel, between two 555, 757, 1032,
// 1298 and 327, 607, 1169, 1789; 64^3: 87, 93, 103, 112 and 69, 81, 103, 130,
// between two 104, 134, 172, 207 and 104, 153, 242, 320; 24^3: batches always).
constexpr double TA_SPARSE = 4, TA_SPARSE2 = 3;
constexpr int64_t TA_SPARSE_CELLS = 1 << 17;

// One lane, one voxel, in memory: the voxels of more particles than a batch
// holds, or (ALL) every voxel of a sparse plasma.
template <bool ALL>
__global__ __launch_bounds__(256) void k_ta_lane(TaArgs a, int *nbad) {
  const int v = blockIdx.x * 256 + threadIdx.x;
  if (v >= a.v1) return;
  TaVoxel V;
  V.k0 = a.part_i[v];
  V.nk = a.part_i[v + 1] - V.k0;
  if (!V.nk) return;
  if (V.k0 < 0 || V.nk < 0 || V.k0 + V.nk > a.np_i) {
    if (ALL) atomicAdd(nbad, 1);
    return;
  }
  V.l0 = V.nl = 0;
  const bool other = a.same || ta_other(a, v, V.l0, V.nl);
  if (!ALL && (int64_t)V.nk + V.nl <= TA_CAP) return;
  if (!other) atomicAdd(nbad, 1);
  TaRng rng;
  ta_stream(a, v, rng);
  float density = 0;
  const int k1 = V.k0 + V.nk;
  int i;
  for (i = V.k0; i < k1 - 1; ++i) {
    const uint32_t rn = UINT32_MAX / (uint32_t)(k1 - i);
    int j;
    do { j = i + (int)(rng.u32() / rn); } while (j >= k1);
    const vpic_particle_t t = a.pi[j];
    a.pi[j] = a.pi[i];
    a.pi[i] = t;
    density += a.pi[i].w;
  }
  density += a.pi[i].w;
  if (!ta_pairing(a, v, density, V, [&](int k) { return a.pj[k].w; })) return;
  uint32_t w[4];
  auto meet = [&](int k, int l, float std) {
    float4 x = *ta_mom(a.pi, k), y = *ta_mom(a.pj, l);
#pragma unroll
    for (int c = 0; c < 4; c++) w[c] = rng.u32();
    ta_collide(x, y, a.mu_i, a.mu_j, std, w);
    *ta_mom(a.pi, k) = x;
    *ta_mom(a.pj, l) = y;
  };
  if (V.triple)
    for (int c = 0; c < 3; c++)
      meet(V.k0 - (c < 2 ? 3 : 2), V.k0 - (c == 0 ? 2 : 1), V.std3);
  if (!V.nk) return;
  const int small = V.nk > V.nl ? V.nl : V.nk;
  for (int c = 0; c < small; c++) {
    int many, len;
    ta_chain(V, c, many, len);
    for (int j = 0; j < len; j++)
      if (V.nk > V.nl)
        meet(V.k0 + many + j, V.l0 + c, V.std);
      else
        meet(V.k0 + c, V.l0 + many + j, V.std);
  }
}

__global__ __launch_bounds__(TA_BS, 4) void k_takizuka_abe(TaArgs a, int nvox,
                                                        int *nbad) {
  __shared__ float4 U[TA_CAP];           // momentum and weight
  __shared__ unsigned short perm[TA_CAP];  // place -> entry of U
  __shared__ unsigned short swap_[TA_CAP];  // place it is swapped with
  __shared__ unsigned char again[TA_VOX];   // a draw of the voxel is rejected
  __shared__ TaVoxel VX[TA_VOX];
  __shared__ int off[TA_VOX + 1];    // first place of each voxel
  __shared__ int first[TA_VOX];      // its first particle
  __shared__ int off_j[TA_VOX + 1], first_j[TA_VOX];  // of species j
  __shared__ int chain0[2 * TA_VOX + 1];
  __shared__ unsigned char odd[TA_VOX];  // voxels with an odd three
  __shared__ int s_m, s_odd;
  const int t = threadIdx.x, lane = lane_id();
  const int vend = min((int)((blockIdx.x + 1) * nvox), a.v1);
  for (int v = blockIdx.x * nvox; v < vend;) {
    // the batch: as many voxels as fit
    if (t < 64) {
      int k0 = 0, nk = 0;
      if (v + t < vend) {
        k0 = a.part_i[v + t];
        nk = a.part_i[v + t + 1] - k0;
        // a partition that does not index this species' particles: skip the
        // voxel and count it (reported as an error by the host)
        if (nk && (k0 < 0 || nk < 0 || k0 + nk > a.np_i)) nk = -1;
      }
      bool bad = nk < 0;
      if (bad) nk = 0;
      int l0 = 0, nl = 0;
      if (nk > 0 && !a.same) bad = !ta_other(a, v + t, l0, nl);
      const long long incl = wave_incl((long long)nk),
                      incl_j = wave_incl((long long)nl);
      const uint64_t fits =
          __ballot(v + t < vend && incl + incl_j <= TA_CAP);
      const int m = __popcll(fits);  // (incl grows, so the first m lanes)
      if (t < m) {
        if (bad) atomicAdd(nbad, 1);
        off[t + 1] = (int)incl;
        first[t] = k0;
        off_j[t + 1] = (int)incl_j;
        first_j[t] = l0;
        VX[t].nk = nk;
        again[t] = 0;
      }
      if (t == 0) {
        off[0] = 0;
        off_j[0] = 0;
        s_m = m;
      }
    }
    __syncthreads();
    const int m = s_m;
    if (m == 0) {
      if (t == 0) atomicAdd(nbad + 1, 1);  // left for k_ta_lane
      v++;
      __syncthreads();
      continue;
    }
    const int total = off[m], total_j = off_j[m];
    // the last voxel that starts at s or before
    auto find_by = [&](auto at, int s, int hi) {
      int lo = 0;
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (at(mid) <= s) lo = mid; else hi = mid;
      }
      return lo;
    };
    auto find = [&](const int *at, int s) {
      return find_by([&](int q) { return at[q]; }, s, m);
    };
    for (int s = t; s < total; s += TA_BS) {
      const int q = find(off, s);
      U[s] = *ta_mom(a.pi, first[q] + (s - off[q]));
      perm[s] = (unsigned short)s;
    }
    for (int s = t; s < total_j; s += TA_BS) {
      const int q = find(off_j, s);
      U[total + s] = *ta_mom(a.pj, first_j[q] + (s - off_j[q]));
    }
    // The shuffle's draws, four places a lane: place i takes word i unless a
    // draw is rejected (one in 2^32 / places), which shifts those behind it.
    const int nslot = (total >> 2) + m;
    for (int r = t; r < nslot; r += TA_BS) {
      auto slot = [&](int q) { return (off[q] >> 2) + q; };
      const int q = find_by(slot, r, m), nk = off[q + 1] - off[q];
      const int i0 = 4 * (r - slot(q));
      if (i0 >= nk - 1) continue;
      TaRng rng;
      ta_stream(a, v + q, rng);
      rng.ctr[0] = (uint32_t)i0 >> 2;
      rng.philox();
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int i = i0 + k;
        if (i >= nk - 1) break;
        const uint32_t j =
            (uint32_t)i + rng.buf[k] / (UINT32_MAX / (uint32_t)(nk - i));
        if (j >= (uint32_t)nk)
          again[q] = 1;
        else
          swap_[off[q] + i] = (unsigned short)(off[q] + j);
      }
    }
    __syncthreads();
    if (t < 64) {
      int n_long = 0, n_short = 0;
      bool triple = false;
      if (t < m && VX[t].nk > 0) {
        TaVoxel V;
        V.nk = VX[t].nk;
        V.k0 = off[t];
        const int k1 = V.k0 + V.nk;
        V.n = (uint32_t)(V.nk - 1);
        if (again[t]) {
          TaRng rng;
          ta_stream(a, v + t, rng);
          for (int i = V.k0; i < k1 - 1; ++i) {
            const uint32_t rn = UINT32_MAX / (uint32_t)(k1 - i);
            uint32_t j;
            do { j = (uint32_t)i + rng.u32() / rn; } while (j >= (uint32_t)k1);
            swap_[i] = (unsigned short)j;
          }
          V.n = rng.n;
        }
#pragma unroll 4
        for (int i = V.k0; i < k1 - 1; ++i) {
          const int j = swap_[i];
          const unsigned short x = perm[j], y = perm[i];
          perm[j] = y;
          perm[i] = x;
        }
        float density = 0;
#pragma unroll 8
        for (int i = V.k0; i < k1; ++i) density += U[perm[i]].w;
        V.l0 = total + off_j[t];
        V.nl = off_j[t + 1] - off_j[t];
        if (ta_pairing(a, v + t, density, V, [&](int k) { return U[k].w; })) {
          n_long = V.rn;
          n_short = (V.nk < V.nl ? V.nk : V.nl) - V.rn;
          triple = V.triple;
        }
        VX[t] = V;
      }
      // the voxels' longer chains first, then the shorter ones: a wavefront
      // runs as long as its longest
      const int incl_long = wave_incl(n_long), incl_short = wave_incl(n_short);
      const int all_long = __shfl(incl_long, 63);
      if (t < m) {
        chain0[t + 1] = incl_long;
        chain0[m + t + 1] = all_long + incl_short;
      }
      const uint64_t odds = __ballot(triple);
      if (triple) odd[__popcll(odds & ((1ull << t) - 1))] = (unsigned char)t;
      if (t == 0) {
        chain0[0] = 0;
        s_odd = __popcll(odds);
      }
    }
    __syncthreads();
    // the odd threes on the last wavefront, so that the others have pairs only
    if (t >= TA_BS - 64 && lane < s_odd) {
      const int q = odd[lane];
      const TaVoxel V = VX[q];
      TaRng rng;
      ta_stream(a, v + q, rng);
      for (int r = 0; r < 3; r++) {
        float4 &x = U[perm[V.k0 - (r < 2 ? 3 : 2)]];
        float4 &y = U[perm[V.k0 - (r == 0 ? 2 : 1)]];
        float4 xv = x, yv = y;
        uint32_t w[4];
        ta_words(rng, V.n + 4u * (uint32_t)r, w);
        ta_collide(xv, yv, a.mu_i, a.mu_j, V.std3, w);
        x = xv;
        y = yv;
      }
    }
    const int nchain = chain0[2 * m];
    for (int s = t; s < nchain; s += TA_BS) {
      const int e = find_by([&](int q) { return chain0[q]; }, s, 2 * m);
      const int q = e < m ? e : e - m;
      const TaVoxel V = VX[q];
      const int c = s - chain0[e] + (e < m ? 0 : V.rn);
      TaRng rng;
      ta_stream(a, v + q, rng);
      uint32_t w[4];
      int many, len;
      ta_chain(V, c, many, len);
      const uint32_t n0 = V.n + (V.triple ? 12u : 0u);
      const bool round_l = V.nk > V.nl;  // the one particle is species j's
      auto at_l = [&](int l) { return a.same ? &U[perm[l]] : &U[l]; };
      float4 *one = round_l ? at_l(V.l0 + c) : &U[perm[V.k0 + c]];
      float4 ov = *one;
      for (int j = 0; j < len; j++) {
        ta_words(rng, n0 + 4u * (uint32_t)(many + j), w);
        float4 *o = round_l ? &U[perm[V.k0 + many + j]] : at_l(V.l0 + many + j);
        float4 xv = *o;
        if (round_l) {
          const float4 x = xv;
          xv = ov;
          ov = x;
        }
        // ov is species i's, xv species j's
        ta_collide(ov, xv, a.mu_i, a.mu_j, V.std, w);
        if (round_l) {
          const float4 x = xv;
          xv = ov;
          ov = x;
        }
        *o = xv;
      }
      *one = ov;
    }
    __syncthreads();
    // the particles to their places: positions read before any is written
    constexpr int PER = TA_CAP / TA_BS;
    float4 A[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
      const int s = t + r * TA_BS;
      if (s < total) {
        const int q = find(off, s);
        A[r] = *reinterpret_cast<const float4 *>(a.pi + first[q] +
                                                 (perm[s] - off[q]));
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PER; r++) {
      const int s = t + r * TA_BS;
      if (s < total) {
        const int q = find(off, s);
        float4 *o = reinterpret_cast<float4 *>(a.pi + first[q] + (s - off[q]));
        o[0] = A[r];
        o[1] = U[perm[s]];
      }
    }
    for (int s = t; s < total_j; s += TA_BS) {
      const int q = find(off_j, s);
      *ta_mom(a.pj, first_j[q] + (s - off_j[q])) = U[total + s];
    }
    __syncthreads();
    v += m;
  }
}

}  // namespace

int launch_takizuka_abe(vpic_particle_t *pi, const int *part_i, int np_i,
                        float qi, float mi, vpic_particle_t *pj,
                        const int *part_j, int np_j, float qj, float mj,
                        double cvar0, int interval, uint64_t seed,
                        uint64_t call, const vpic_grid_t *g, hipStream_t s) {
  TaArgs a;
  a.pi = pi;
  a.pj = pj;
  a.part_i = part_i;
  a.part_j = part_j;
  a.np_i = np_i;
  a.np_j = np_j;
  a.same = pi == pj;
  a.v1 = g->nx + g->sy * g->ny + g->sz * g->nz + 1;  // VOXEL(nx,ny,nz)+1
  // the coupling constants as takizuka_abe_pipeline.cc:95-99 forms them
  a.dtinterval_dV = (g->dt * (float)interval) / g->dV;
  const float mu = (mi * mj) / (mi + mj);
  a.mu_i = mj / (mi + mj);
  a.mu_j = mi / (mi + mj);
  a.cvar = cvar0 * (qi * qi * qj * qj) / (mu * mu);
  a.key0 = (uint32_t)seed;
  a.key1 = (uint32_t)(seed >> 32);
  a.call0 = (uint32_t)call;
  a.call1 = (uint32_t)(call >> 32);
  DeviceScratch &S = collision_scratch();
  if (int rc = scratch_reserve(S, 64)) return rc;
  int *nbad = (int *)S.ptr;
  hipLaunchKernelGGL(k_ta_clear, dim3(1), dim3(64), 0, s, nbad);
  VPIC_LAUNCHED("k_ta_clear");
  // voxels of a workgroup: three quarters of a batch at the mean number of
  // particles, since a batch that does not hold them all leaves a short second
  // one (64-particle voxels with their spread of 8: 21 of at most 28)
  const int64_t cells = (int64_t)g->nx * g->ny * g->nz;
  const double mean =
      ((double)np_i + (a.same ? 0.0 : (double)np_j)) / (double)cells;
  int nvox = mean > 0 ? (int)(0.75 * TA_CAP / mean) : TA_VOX;
  nvox = nvox < 1 ? 1 : nvox > TA_VOX ? TA_VOX : nvox;
  if (cells >= TA_SPARSE_CELLS &&
      mean < (a.same ? TA_SPARSE : TA_SPARSE2)) {
    hipLaunchKernelGGL(k_ta_lane<true>, dim3((a.v1 + 255) / 256), dim3(256), 0,
                       s, a, nbad);
    VPIC_LAUNCHED("k_ta_lane");
  } else {
    hipLaunchKernelGGL(k_takizuka_abe, dim3((a.v1 + nvox - 1) / nvox),
                       dim3(TA_BS), 0, s, a, nvox, nbad);
    VPIC_LAUNCHED("k_takizuka_abe");
  }
  int h[2] = {0, 0};
  VPIC_HIP(
      hipMemcpyAsync(h, nbad, sizeof(h), hipMemcpyDeviceToHost, s));
  VPIC_HIP(hipStreamSynchronize(s));
  if (h[1]) {
    hipLaunchKernelGGL(k_ta_lane<false>, dim3((a.v1 + 255) / 256), dim3(256),
                       0, s, a, nbad);
    VPIC_LAUNCHED("k_ta_lane");
    VPIC_HIP(
        hipMemcpyAsync(h, nbad, sizeof(int), hipMemcpyDeviceToHost, s));
    VPIC_HIP(hipStreamSynchronize(s));
  }
  if (h[0])
    return vpic_set_error(VPIC_EINVAL,
                          "takizuka_abe: the partition of %d voxels does not "
                          "index the species' particles", h[0]);
  return VPIC_OK;
}
