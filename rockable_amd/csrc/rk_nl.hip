// rk_nl.hip -- neighbour-list rebuild on the GPU.
//
// Restates UpdateNL_bruteForce (Rockable.cpp:1614-1662), UpdateNL_linkCells
// (1667-1809) and AddOrRemoveInteractions_bruteForce (1309-1432) with the
// sub-element predicates of Particle.cpp:88-209, keeping the reference's
// set semantics exactly:
//   * a key that is tested and near is kept (with its history) or created,
//   * a key that is tested and not near is erased,
//   * a key that is not tested (pair not a candidate, vertex gated out, or a
//     type never tested in that direction) is retained unchanged.
//
// Pipeline (each step a kernel; counts come back to the host between steps):
//   k_obb            Particle::updateObb (+ AABB for the cell grid)
//   k_broad_*        candidate body pairs (i < j) whose enlarged OBBs overlap
//   groups           directed (owner, other) groups = candidates x 2 directions
//                    merged with the groups of the current list (placed by counts)
//   k_narrow         one wavefront per candidate pair: global vertices and
//                    vertex gates in LDS, every predicate of both directions
//                    evaluated 64 at a time, near bits kept as ballot masks,
//                    then written as keys in (type, isub, jsub) order with a
//                    wavefront prefix scan (no atomics per key)
//   k_merge          per directed group, merge of the sorted old entries and
//                    the sorted near keys (count pass, scan, write pass of the
//                    keys and of each entry's source); the output is again
//                    sorted by (i, j, type, isub, jsub)
//   k_merge_fill     one thread per new entry: its state record, copied from
//                    the old entry it keeps or started from zero
//   CSR              istart by owner; jlist = entries by j, in any order within
//                    a body's
#include <hip/hip_runtime.h>

#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstring>
#include <functional>
#include <initializer_list>
#include <utility>
#include <vector>

#include "rk_device.hpp"
#include "rk_model.hpp"
#include "rk_nl.hpp"

namespace rk {

namespace {

constexpr int kBlock = 256;

#define RK_CHECK(x)                                                                 \
  do {                                                                              \
    hipError_t e_ = (x);                                                            \
    if (e_ != hipSuccess) {                                                         \
      snprintf(w.err, sizeof(w.err), "%s failed: %s", #x, hipGetErrorString(e_)); \
      return -1;                                                                    \
    }                                                                               \
  } while (0)

__device__ __forceinline__ v3 kpos(const BodyKin& b) { return V(b.px, b.py, b.pz); }
__device__ __forceinline__ qt kq(const BodyKin& b) {
  qt q;
  q.w = b.qw;
  q.x = b.qx;
  q.y = b.qy;
  q.z = b.qz;
  return q;
}
__device__ __forceinline__ obb_t load_obb(const double* o) {
  obb_t r;
  r.c = V(o[0], o[1], o[2]);
  r.e[0] = V(o[3], o[4], o[5]);
  r.e[1] = V(o[6], o[7], o[8]);
  r.e[2] = V(o[9], o[10], o[11]);
  r.ext = V(o[12], o[13], o[14]);
  return r;
}
__device__ __forceinline__ void store_obb(double* o, const obb_t& r) {
  o[0] = r.c.x;
  o[1] = r.c.y;
  o[2] = r.c.z;
  o[3] = r.e[0].x;
  o[4] = r.e[0].y;
  o[5] = r.e[0].z;
  o[6] = r.e[1].x;
  o[7] = r.e[1].y;
  o[8] = r.e[1].z;
  o[9] = r.e[2].x;
  o[10] = r.e[2].y;
  o[11] = r.e[2].z;
  o[12] = r.ext.x;
  o[13] = r.ext.y;
  o[14] = r.ext.z;
}

// Particle::updateObb (Particle.cpp:78-86) and the body AABB of
// Rockable::computeAABB (Rockable.cpp:3934-3941).
__global__ void k_obb(Dev d, double* bobb, double* baabb) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= d.nb) return;
  const BodyKin P = d.kin[b];
  obb_t o = load_obb(d.sh.obb + 15 * P.shape);
  const qt Q = kq(P);
  o.e[0] = qrot(Q, o.e[0]);
  o.e[1] = qrot(Q, o.e[1]);
  o.e[2] = qrot(Q, o.e[2]);
  o.c = qrot(Q, o.c);
  o.ext = vsc(P.h, o.ext);
  o.c = vsc(P.h, o.c);
  o.c = vadd(o.c, kpos(P));
  store_obb(bobb + 15 * (size_t)b, o);
  if (baabb) {
    const double* gb = d.gv + 3 * (size_t)d.bvoff[b];
    v3 mn = V(gb[0], gb[1], gb[2]), mx = mn;
    const int nv = d.sh.nv[P.shape];
    for (int v = 1; v < nv; v++) {
      v3 g = V(gb[3 * v], gb[3 * v + 1], gb[3 * v + 2]);
      mn.x = g.x < mn.x ? g.x : mn.x;
      mn.y = g.y < mn.y ? g.y : mn.y;
      mn.z = g.z < mn.z ? g.z : mn.z;
      mx.x = g.x > mx.x ? g.x : mx.x;
      mx.y = g.y > mx.y ? g.y : mx.y;
      mx.z = g.z > mx.z ? g.z : mx.z;
    }
    const double r = P.R;
    double* a = baabb + 6 * (size_t)b;
    a[0] = mn.x - r;
    a[1] = mn.y - r;
    a[2] = mn.z - r;
    a[3] = mx.x + r;
    a[4] = mx.y + r;
    a[5] = mx.z + r;
  }
}

// Interfaces[i].find((i, j)) on the sorted live-interface keys.
// Whether (i, j) has a live interface: the first key not below (i, j) among
// i's interfaces (their keys are sorted by j), as a binary search over all
// keys would find it, without its chain of dependent loads.
// IfcRange holds i's range, loaded once for all of i's pairs.
struct IfcRange {
  int lo, hi;
};
__device__ __forceinline__ IfcRange ifc_range(const DevInterfaces& f, int i) {
  IfcRange r;
  r.lo = f.n ? f.istart[i] : 0;
  r.hi = f.n ? f.istart[i + 1] : 0;
  return r;
}
__device__ __forceinline__ bool has_live_interface(const DevInterfaces& f, IfcRange r, int j) {
  const uint32_t uj = (uint32_t)j;
  for (int k = r.lo; k < r.hi; k++) {
    const uint32_t kj = (uint32_t)(f.key[k] & 0xffffffffull);
    if (kj >= uj) return kj == uj && f.alive[k];
  }
  return false;
}

// Output counters are striped: stripe s owns counter cnt[s * kStripeStride]
// (its own 128-byte line) and the region [s * rcap, (s + 1) * rcap) of the
// output; a workgroup appends to stripe (its index mod kStripes), one atomic
// per wavefront and emission point.  A single shared counter serialises at
// one L2 channel (~10 ns per atomic, milliseconds per rebuild).
constexpr int kStripes = 256;
constexpr int kStripeStride = 32;

__device__ __forceinline__ int stripe_of_block() {
  return (int)((blockIdx.x + blockIdx.y * gridDim.x) & (kStripes - 1));
}

// every active lane of the wavefront calls this; lanes with emit append i, j
__device__ __forceinline__ void emit_pair(bool emit, uint64_t* cand, int* cnt, int rcap, int i, int j) {
  const unsigned long long m = __ballot(emit);
  if (m == 0ull) return;
  const int lane = threadIdx.x & 63;
  const int leader = __ffsll((long long)m) - 1;
  const int s = stripe_of_block();
  int base = 0;
  if (lane == leader) base = atomicAdd(cnt + s * kStripeStride, __popcll(m));
  base = __shfl(base, leader, 64);
  if (emit) {
    const int k = base + __popcll(m & ((1ull << lane) - 1ull));
    if (k < rcap) cand[(size_t)s * rcap + k] = ((uint64_t)(uint32_t)i << 32) | (uint32_t)j;
  }
}

// one workgroup of kStripes threads: exclusive offsets of the stripes, their
// total and their maximum
__global__ void k_stripe_scan(const int* cnt, int* off, int* total_max) {
  __shared__ int sc[kStripes], mx[kStripes];
  const int t = threadIdx.x;
  const int v = cnt[t * kStripeStride];
  sc[t] = v;
  mx[t] = v;
  __syncthreads();
  for (int o = 1; o < kStripes; o <<= 1) {
    const int x = t >= o ? sc[t - o] : 0;
    __syncthreads();
    sc[t] += x;
    __syncthreads();
  }
  for (int h = kStripes / 2; h > 0; h >>= 1) {
    if (t < h) mx[t] = max(mx[t], mx[t + h]);
    __syncthreads();
  }
  off[t] = sc[t] - v;
  if (t == kStripes - 1) total_max[0] = sc[t];
  if (t == 0) total_max[1] = mx[0];
}

// the stripes, concatenated
__global__ void k_stripe_gather(const uint64_t* src, int rcap, const int* cnt, const int* off, uint64_t* dst) {
  const int s = blockIdx.y;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = min(cnt[s * kStripeStride], rcap);
  if (k < n) dst[off[s] + k] = src[(size_t)s * rcap + k];
}

__device__ __forceinline__ bool pair_overlap(const double* bobb, int i, int j, double half) {
  obb_t oi = load_obb(bobb + 15 * (size_t)i);
  obb_enlarge(&oi, half);
  obb_t oj = load_obb(bobb + 15 * (size_t)j);
  obb_enlarge(&oj, half);
  return obb_intersect(oi, oj);
}

// UpdateNL_bruteForce pair loop (Rockable.cpp:1622-1658): i < j, j >= nDriven
constexpr int kBruteChunk = 128;
__global__ void k_broad_brute(Dev d, const double* bobb, double half, uint64_t* cand, int* cnt, int rcap) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.nb) return;
  int j0 = i + 1;
  if (j0 < d.nDriven) j0 = d.nDriven;
  const int jb = j0 + (int)blockIdx.y * kBruteChunk;
  const int je = min(jb + kBruteChunk, d.nb);
  const IfcRange ir = ifc_range(d.ifc, i);
  for (int j = jb; j < je; j++) {
    const bool emit = pair_overlap(bobb, i, j, half) && !has_live_interface(d.ifc, ir, j);
    emit_pair(emit, cand, cnt, rcap, i, j);
  }
}
// (the OBB test before the interface search in every broad-phase kernel: both
// are pure, and the search costs a chain of dependent loads per pair)

// --- linkCells broad phase ---------------------------------------------
__global__ void k_box_partial(int first, int nb, const double* baabb, double* part) {
  __shared__ double red[6][kBlock];
  const int t = threadIdx.x;
  double v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  for (int b = first + blockIdx.x * blockDim.x + t; b < nb; b += gridDim.x * blockDim.x) {
    const double* a = baabb + 6 * (size_t)b;
    for (int k = 0; k < 3; k++) {
      v[k] = a[k] < v[k] ? a[k] : v[k];
      v[3 + k] = a[3 + k] > v[3 + k] ? a[3 + k] : v[3 + k];
    }
  }
  for (int k = 0; k < 6; k++) red[k][t] = v[k];
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (t < s)
      for (int k = 0; k < 3; k++) {
        red[k][t] = red[k][t + s] < red[k][t] ? red[k][t + s] : red[k][t];
        red[3 + k][t] = red[3 + k][t + s] > red[3 + k][t] ? red[3 + k][t + s] : red[3 + k][t];
      }
    __syncthreads();
  }
  if (t == 0)
    for (int k = 0; k < 6; k++) part[6 * blockIdx.x + k] = red[k][0];
}

struct Grid {
  int N[3];
  double mn[3], sz[3];
};

// Largest distance, per dimension, from a body's position to a point of its
// OBB enlarged by `half` (a celled body sits in the cell of its position).
__device__ __forceinline__ void obb_reach(const double* o, const double p[3], double half, double r[3]) {
  for (int k = 0; k < 3; k++)
    r[k] = fabs(o[k] - p[k]) + fabs(o[3 + k]) * (o[12] + half) + fabs(o[6 + k]) * (o[13] + half) +
           fabs(o[9 + k]) * (o[14] + half);
}

// Cell of each body (oversized bodies to their own list) and, in `reach`
// (bit patterns of non-negative doubles, which order as integers), the
// largest obb_reach over the celled bodies.
__global__ void k_cell_assign(Dev d, const double* bobb, const double* baabb, double half, Grid g, int* cell_of,
                              int* ccount, int* over, int* nover, unsigned long long* reach) {
  __shared__ double red[3][kBlock];
  const int t = threadIdx.x;
  const int b = blockIdx.x * blockDim.x + t;
  double rr[3] = {0.0, 0.0, 0.0};
  if (b < d.nb) {
    const double* a = baabb + 6 * (size_t)b;
    const bool oversized = (a[3] - a[0] > g.sz[0]) || (a[4] - a[1] > g.sz[1]) || (a[5] - a[2] > g.sz[2]);
    if (oversized) {
      cell_of[b] = -1;
      over[atomicAdd(nover, 1)] = b;
    } else {
      const BodyKin& P = d.kin[b];
      const double p[3] = {P.px, P.py, P.pz};
      int c3[3];
      for (int k = 0; k < 3; k++) {
        int q = (int)floor((p[k] - g.mn[k]) / g.sz[k]);
        q = q < 0 ? 0 : q;
        q = q >= g.N[k] ? g.N[k] - 1 : q;
        c3[k] = q;
      }
      const int c = (c3[0] * g.N[1] + c3[1]) * g.N[2] + c3[2];
      cell_of[b] = c;
      atomicAdd(ccount + c, 1);
      obb_reach(bobb + 15 * (size_t)b, p, half, rr);
    }
  }
  for (int k = 0; k < 3; k++) red[k][t] = rr[k];
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (t < s)
      for (int k = 0; k < 3; k++) red[k][t] = red[k][t + s] > red[k][t] ? red[k][t + s] : red[k][t];
    __syncthreads();
  }
  if (t < 3) atomicMax(reach + t, (unsigned long long)__double_as_longlong(red[t][0]));
}

__global__ void k_cell_fill(int nb, const int* cell_of, const int* cstart, int* cfill, int* cbody) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int c = cell_of[b];
  if (c < 0) return;
  cbody[cstart[c] + atomicAdd(cfill + c, 1)] = b;
}

// main loop of UpdateNL_linkCells (Rockable.cpp:1697-1751): 32 lanes per
// body.  Body i's 27 neighbour cells are 9 runs of consecutive cells (the
// cells of a column along z are consecutive in the cell order), so its
// candidates are the bodies of 9 ranges of cbody; lane q < 9 finds range q,
// and the 32 lanes then take the ranges' bodies in turn, so that a lane is
// idle only past the last one (a lane per cell, looping over that cell's
// bodies, leaves the lanes of emptier cells idle while the fullest is
// walked).  The candidates are sorted afterwards, so the order in which
// they are found does not matter.
constexpr int kCellLanes = 32;
__global__ void k_broad_cells(Dev d, const double* bobb, double half, Grid g, const int* cell_of, const int* cstart,
                              const int* cbody, uint64_t* cand, int* cnt, int rcap) {
  constexpr int L = kCellLanes;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int i = (int)(t / L), q = (int)(t % L);
  const int c = i < d.nb ? cell_of[i] : -1;
  int r0 = 0, len = 0;
  if (c >= 0 && q < 9) {
    const int cz = c % g.N[2], cy = (c / g.N[2]) % g.N[1], cx = c / (g.N[2] * g.N[1]);
    const int nx = cx + q / 3 - 1, ny = cy + q % 3 - 1;
    if (nx >= 0 && ny >= 0 && nx < g.N[0] && ny < g.N[1]) {
      const int base = (nx * g.N[1] + ny) * g.N[2];
      const int z0 = cz > 0 ? cz - 1 : 0, z1 = cz + 1 < g.N[2] ? cz + 1 : g.N[2] - 1;
      r0 = cstart[base + z0];
      len = cstart[base + z1 + 1] - r0;
    }
  }
  // inclusive prefix of the range lengths over lanes 0-8 of the body
  int pre = len;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    const int x = __shfl_up(pre, o, L);
    if (q >= o) pre += x;
  }
  // every lane: range k's end in the concatenation and its shift into cbody
  int pend[9], poff[9];
#pragma unroll
  for (int k = 0; k < 9; k++) {
    pend[k] = __shfl(pre, k, L);
    poff[k] = __shfl(r0 - (pre - len), k, L);
  }
  const int total = pend[8];
  const bool own = c >= 0;
  const IfcRange ir = own ? ifc_range(d.ifc, i) : IfcRange{0, 0};
  for (int base = 0; __any(own && base < total); base += L) {
    const int x = base + q;
    bool emit = false;
    int j = 0;
    if (own && x < total) {
      int off = poff[8];
#pragma unroll
      for (int k = 7; k >= 0; k--)
        if (x < pend[k]) off = poff[k];
      j = cbody[x + off];
      emit = !(j < d.nDriven && i < d.nDriven) && j > i && pair_overlap(bobb, i, j, half) &&
             !has_live_interface(d.ifc, ir, j);
    }
    emit_pair(emit, cand, cnt, rcap, i, j);
  }
}

// Oversized bodies against the bodies of the cells (Rockable.cpp:1755-1805):
// workgroup (q, y) takes oversized body over[q] and every gridDim.y-th
// (x, y) column of cells.  The reference visits every cell; a celled body
// whose enlarged OBB meets the oversized body's lies within `reach` of that
// OBB's box, so only the cells covering the box plus reach (one more on each
// side against rounding) can hold one, and the others are skipped.
__global__ void k_broad_over(Dev d, const double* bobb, double half, Grid g, const int* over, int nover,
                             const int* cstart, const int* cbody, const unsigned long long* reach, uint64_t* cand,
                             int* cnt, int rcap) {
  const int q = blockIdx.x;
  if (q >= nover) return;
  const int i = over[q];
  const double* o = bobb + 15 * (size_t)i;
  int lo[3], hi[3];
  for (int k = 0; k < 3; k++) {
    const double ext =
        fabs(o[3 + k]) * (o[12] + half) + fabs(o[6 + k]) * (o[13] + half) + fabs(o[9 + k]) * (o[14] + half);
    const double rch = __longlong_as_double((long long)reach[k]);
    const double top = (double)(g.N[k] - 1);
    const double a = floor((o[k] - ext - rch - g.mn[k]) / g.sz[k]) - 1.0;
    const double b = floor((o[k] + ext + rch - g.mn[k]) / g.sz[k]) + 1.0;
    lo[k] = (int)fmin(fmax(a, 0.0), top);
    hi[k] = (int)fmin(fmax(b, 0.0), top);
  }
  const int ny = hi[1] - lo[1] + 1;
  const int ncol = (hi[0] - lo[0] + 1) * ny;
  const IfcRange ir = ifc_range(d.ifc, i);
  for (int col = blockIdx.y; col < ncol; col += gridDim.y) {
    const int cx = lo[0] + col / ny, cy = lo[1] + col % ny;
    const int cbase = (cx * g.N[1] + cy) * g.N[2];
    const int r0 = cstart[cbase + lo[2]], r1 = cstart[cbase + hi[2] + 1];
    for (int rb = r0; rb < r1; rb += blockDim.x) {
      const int r = rb + (int)threadIdx.x;
      bool emit = false;
      int j = 0;
      if (r < r1) {
        j = cbody[r];
        emit = !(j < d.nDriven && i < d.nDriven) && j > i && pair_overlap(bobb, i, j, half) &&
               !has_live_interface(d.ifc, ir, j);
      }
      emit_pair(emit, cand, cnt, rcap, i, j);
    }
  }
}

// --- directed groups -------------------------------------------------------
// head of each (i, j) run of the current (sorted) entry list
__global__ void k_old_heads(int n, const int32_t* ei, const int32_t* ej, int32_t* flag) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  flag[e] = (e == 0 || ei[e] != ei[e - 1] || ej[e] != ej[e - 1]) ? 1 : 0;
}
__global__ void k_old_compact(int n, const int32_t* ei, const int32_t* ej, const int32_t* flag, const int32_t* pos,
                              uint64_t* okey, int32_t* ostart) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e == n - 1) ostart[pos[e] + flag[e]] = n;
  if (e >= n || !flag[e]) return;
  okey[pos[e]] = ((uint64_t)(uint32_t)ei[e] << 32) | (uint32_t)ej[e];
  ostart[pos[e]] = e;
}

// Placing by counts.  The directed groups ordered by (owner, other) and every
// body's entries as second body ordered by index are both segments of small
// integers that are all different, some tens of them for most bodies, and
// thousands for a wall.  A device-wide radix or merge sort runs its full
// sequence of passes for them and is launch bound below a million keys
// (15 007 spheres: 205 us of a rebuild in the two sorts).  Here a count per
// body, one scan and a fill in any order give the segments, and a member's
// place is the number of smaller members: a loop over the segment, contiguous
// and shared by the neighbouring lanes, up to kSegMax members; above that the
// loop's square would tell, and workgroups mark the members of a window of
// values in an LDS bitmap and count bits.
constexpr int kSegMax = 512;
constexpr int kWinBits = 18;  // values per bitmap window: 32 KB of bits, 16 KB of prefixes
constexpr int kWinWords = 1 << (kWinBits - 6);
constexpr int kWinThreads = 512;
constexpr int kBigGrid = 64;  // workgroups across the list of long segments

// One atomic per run of equal keys in neighbouring lanes (all lanes of the
// wavefront call it): a wall's members come in runs and would queue on its
// counter one by one.  `weight` counts a member in the low 32 bits,
// and may count it in the high ones too (`kind` tells
// the weights apart: a run has one); returns the member's position
// among its key's, runs in lane order.  The counting pass keeps the positions,
// so that the fill needs no atomics (337 000 entries: 27 us with its own,
// under 13 without).  What bounds the count is the queue on the walls'
// counters, one atomic per body that touches the wall (38 us).
template <class T>
__device__ __forceinline__ int run_add(T* count, int key, bool valid, T weight, int kind = 0) {
  const int lane = (int)(threadIdx.x & 63);
  const int k = valid ? key : -1;
  const int prev = __shfl_up(k, 1, 64), pkind = __shfl_up(kind, 1, 64);
  const unsigned long long heads = __ballot(lane == 0 || prev != k || pkind != kind);
  const unsigned long long upto = heads & (~0ull >> (63 - lane));
  const int head = 63 - __clzll((long long)upto);
  const unsigned long long above = lane == 63 ? 0ull : heads >> (lane + 1) << (lane + 1);
  int base = 0;
  if (lane == head && valid) base = (int)atomicAdd(count + key, weight * (T)((above ? __ffsll(above) - 1 : 64) - lane));
  return __shfl(base, head, 64) + lane - head;
}

// The members of [s0, s1) whose values lie in window `win`, as bits with
// exclusive prefixes; returns the number of members below the window.  All
// threads of the workgroup call it; it starts and ends with a barrier.
struct WinLds {
  unsigned long long bits[kWinWords];
  int32_t pre[kWinWords];
  int32_t wsum[kWinThreads / 64];
  int32_t below;
};
__device__ int win_mark(WinLds& L, const int32_t* val, int s0, int s1, int win) {
  const int t = (int)threadIdx.x, lane = t & 63;
  __syncthreads();
  for (int q = t; q < kWinWords; q += kWinThreads) L.bits[q] = 0ull;
  if (t == 0) L.below = 0;
  __syncthreads();
  int under = 0;
  // (four members a round, so that their loads share a latency)
  for (int q0 = s0 + t; q0 < s1; q0 += 4 * kWinThreads) {
    int v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = q0 + k * kWinThreads < s1 ? val[q0 + k * kWinThreads] : INT_MAX;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (q0 + k * kWinThreads >= s1) continue;
      const int vw = v[k] >> kWinBits;
      if (vw < win)
        under++;
      else if (vw == win)
        atomicOr(&L.bits[(v[k] & ((1 << kWinBits) - 1)) >> 6], 1ull << (v[k] & 63));
    }
  }
  if (under) atomicAdd(&L.below, under);
  __syncthreads();
  constexpr int per = kWinWords / kWinThreads;
  int sum = 0;
  for (int q = 0; q < per; q++) sum += __popcll(L.bits[t * per + q]);
  int inc = sum;
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(inc, o, 64);
    if (lane >= o) inc += x;
  }
  if (lane == 63) L.wsum[t >> 6] = inc;
  __syncthreads();
  int run = inc - sum;
  for (int q = 0; q < (t >> 6); q++) run += L.wsum[q];
  for (int q = 0; q < per; q++) {
    L.pre[t * per + q] = run;
    run += __popcll(L.bits[t * per + q]);
  }
  __syncthreads();
  return L.below;
}
// members of the window below value v of the window
__device__ __forceinline__ int win_rank(const WinLds& L, int v) {
  const int x = v & ((1 << kWinBits) - 1);
  return L.pre[x >> 6] + __popcll(L.bits[x >> 6] & ((1ull << (x & 63)) - 1ull));
}

// The directed groups: both directions of every candidate and the groups of
// the current list.  Owner b's part of the group arrays has a slot per member,
// the slot of a group being the number of candidates plus the number of old
// groups below it: a pair that is both takes one slot, the same from either
// side, and leaves the next one empty (no candidate, no old group).
__global__ void k_group_count(int nc, const uint64_t* cand, int32_t* cnt, int2* at) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = t < nc;
  const uint64_t k = valid ? cand[t] : 0;
  const int qi = run_add(cnt, (int)(k >> 32), valid, 1);
  const int qj = run_add(cnt, (int)(k & 0xffffffffu), valid, 1);
  if (valid) at[t] = make_int2(qi, qj);
}
__global__ void k_group_fill(int nc, const uint64_t* cand, const int2* at, const int32_t* gstart, int32_t* gowner,
                             int32_t* gother, int32_t* gref) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nc) return;
  const uint64_t k = cand[t];
  const int i = (int)(k >> 32), j = (int)(k & 0xffffffffu);
  const int2 q = at[t];
  const int a = gstart[i] + q.x, b = gstart[j] + q.y;
  gowner[a] = i;
  gother[a] = j;
  gref[a] = t << 1;
  gowner[b] = j;
  gother[b] = i;
  gref[b] = (t << 1) | 1;
}
struct GroupIn {
  int nc2, ng_old, nold;  // directed candidates, old groups, old entries
  const int32_t* gstart;      // per body: its first directed candidate
  const int32_t* gowner;
  const int32_t* gother;
  const int32_t* gref;
  const int32_t* istart;  // old entries by owner (null without any)
  const int32_t* opos;    // old entries: the groups headed before it
  const uint64_t* okey;
  uint64_t* ukey;
  int32_t* ucand;
  int32_t* uold;
  int32_t* nbig;  // long segments' owners
  int32_t* big;
};
// the first old group of owner b (b up to nb)
__device__ __forceinline__ int old_first(const GroupIn& G, int b) {
  if (!G.ng_old) return 0;
  const int e = G.istart[b];
  return e < G.nold ? G.opos[e] : G.ng_old;
}
// old groups of [o0, o1) whose other body is below v
__device__ __forceinline__ int old_below(const GroupIn& G, int o0, int o1, int v) {
  int lo = o0, hi = o1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if ((int)(G.okey[mid] & 0xffffffffu) < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo - o0;
}
__device__ __forceinline__ void put_cand(const GroupIn& G, int slot, int owner, int other, int ref) {
  G.ukey[slot] = ((uint64_t)(uint32_t)owner << 32) | (uint32_t)other;
  G.ucand[slot] = ref;
}
__device__ __forceinline__ void put_old(const GroupIn& G, int slot, uint64_t key, int g) {
  G.ukey[slot] = key;
  G.uold[slot] = g;
}
__device__ __forceinline__ int seg_below(const int32_t* val, int s0, int s1, int v) {
  int n = 0;
#pragma unroll 8
  for (int q = s0; q < s1; q++) n += val[q] < v ? 1 : 0;
  return n;
}
__global__ void k_group_place(GroupIn G) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < G.nc2) {
    const int b = G.gowner[t];
    const int s0 = G.gstart[b], s1 = G.gstart[b + 1];
    if (s1 - s0 > kSegMax) {
      if (t == s0) G.big[atomicAdd(G.nbig, 1)] = b;
      return;
    }
    const int v = G.gother[t];
    const int o0 = old_first(G, b), o1 = old_first(G, b + 1);
    put_cand(G, s0 + o0 + seg_below(G.gother, s0, s1, v) + old_below(G, o0, o1, v), b, v, G.gref[t]);
  } else if (t < G.nc2 + G.ng_old) {
    const int g = t - G.nc2;
    const uint64_t key = G.okey[g];
    const int b = (int)(key >> 32), v = (int)(key & 0xffffffffu);
    const int s0 = G.gstart[b], s1 = G.gstart[b + 1];
    if (s1 - s0 > kSegMax) return;
    put_old(G, s0 + g + seg_below(G.gother, s0, s1, v), key, g);
  }
}
__global__ void __launch_bounds__(kWinThreads) k_group_place_big(GroupIn G) {
  __shared__ WinLds L;
  const int nbig = *G.nbig, win = (int)blockIdx.y;
  for (int q = (int)blockIdx.x; q < nbig; q += (int)gridDim.x) {
    const int b = G.big[q];
    const int s0 = G.gstart[b], s1 = G.gstart[b + 1];
    const int o0 = old_first(G, b), o1 = old_first(G, b + 1);
    const int below = win_mark(L, G.gother, s0, s1, win);
    for (int t0 = s0 + (int)threadIdx.x; t0 < s1; t0 += 4 * kWinThreads) {
      int v[4], ref[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int t = min(t0 + k * kWinThreads, s1 - 1);
        v[k] = G.gother[t];
        ref[k] = G.gref[t];
      }
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (t0 + k * kWinThreads < s1 && (v[k] >> kWinBits) == win)
          put_cand(G, s0 + o0 + below + win_rank(L, v[k]) + old_below(G, o0, o1, v[k]), b, v[k], ref[k]);
    }
    for (int g = o0 + (int)threadIdx.x; g < o1; g += kWinThreads) {
      const uint64_t key = G.okey[g];
      const int v = (int)(key & 0xffffffffu);
      if ((v >> kWinBits) == win) put_old(G, s0 + g + below + win_rank(L, v), key, g);
    }
  }
}

// --- narrow phase ------------------------------------------------------
struct NarrowCfg {
  int maxv;       // max vertices per shape
  int maxe;       // max edges per shape
  int maxf;       // max faces per shape
  int maxwords;   // max 64-bit bitmask words per pair
  double dmax;    // dVerlet
  // the culls' boxes of every body's edges and faces (k_gate_boxes)
  const float* gedge;  // kGate floats per edge / face
  const float* gface;
};

__device__ __forceinline__ v3 lds_v(const double* a, int k) { return V(a[3 * k], a[3 * k + 1], a[3 * k + 2]); }

// Particle::VertexIsNearVertex/Edge/Face, EdgeIsNearEdge (Particle.cpp:88-209)
// with the global vertices of both bodies read from LDS.
__device__ bool near_vv(const double* gvi, const double* gvj, double Ri, double Rj, int isub, int jsub, double dmax) {
  v3 pi = lds_v(gvi, isub), pj = lds_v(gvj, jsub);
  double sum = Ri + Rj + dmax;
  return vnorm2(vsub(pj, pi)) <= sum * sum;
}
__device__ bool near_ve(const DevShapes& sh, int shj, const double* gvi, const double* gvj, double Ri, double Rj,
                        int isub, int jsub, double dmax) {
  const int* ed = sh.edge + 2 * (sh.eoff[shj] + jsub);
  v3 pi = lds_v(gvi, isub), p0 = lds_v(gvj, ed[0]), p1 = lds_v(gvj, ed[1]);
  v3 E = vsub(p1, p0);
  v3 v = vsub(pi, p0);
  double r = vdot(v, E) / vdot(E, E);
  if (r < -dmax) return false;
  if (r > 1.0 + dmax) return false;
  double sum = Ri + Rj + dmax;
  return vnorm2(vsub(pi, vadd(p0, vsc(r, E)))) <= sum * sum;
}
__device__ bool near_vf(const DevShapes& sh, int shj, const double* gvi, const double* gvj, double Ri, double Rj,
                        int isub, int jsub, double dmax) {
  const int gface = sh.foff[shj] + jsub;
  const int fs = sh.fstart[gface];
  const int nbv = sh.fstart[gface + 1] - fs;
  const int* fv = sh.fidx + fs;
  v3 A = lds_v(gvj, fv[0]), B = lds_v(gvj, fv[1]), C = lds_v(gvj, fv[nbv - 1]);
  v3 pi = lds_v(gvi, isub);
  v3 v = vsub(pi, A);
  v3 v1 = vsub(B, A);
  vnormalize(&v1);
  v3 v2 = vsub(C, A);
  v3 n = vcross(v1, v2);
  vnormalize(&n);
  double dist = vdot(v, n);
  if (dist < 0.0) {
    n = vneg(n);
    dist = -dist;
  }
  v3 P = vsub(pi, vsc(dist, n));
  v2 = vcross(n, v1);
  int odd = 0;
  double ori1 = vdot(P, v1), ori2 = vdot(P, v2);
  for (int iva = 0; iva < nbv; iva++) {
    int ivb = iva + 1;
    if (ivb == nbv) ivb = 0;
    v3 a = lds_v(gvj, fv[iva]), b = lds_v(gvj, fv[ivb]);
    double pa1 = vdot(a, v1), pb1 = vdot(b, v1);
    double pa2 = vdot(a, v2), pb2 = vdot(b, v2);
    if ((pa2 < ori2 && pb2 >= ori2) || (pb2 < ori2 && pa2 >= ori2)) {
      if (pa1 + (ori2 - pa2) / (pb2 - pa2) * (pb1 - pa1) < ori1) odd = 1 - odd;
    }
  }
  if (odd == 1) {
    dist -= (Ri + Rj);
    if (dist <= dmax) return true;
  }
  return false;
}
__device__ bool near_ee(const DevShapes& sh, int shi, int shj, const double* gvi, const double* gvj, double Ri,
                        double Rj, int isub, int jsub, double dmax) {
  const int* edj = sh.edge + 2 * (sh.eoff[shj] + jsub);
  const int* edi = sh.edge + 2 * (sh.eoff[shi] + isub);
  v3 p0j = lds_v(gvj, edj[0]), p1j = lds_v(gvj, edj[1]);
  v3 p0i = lds_v(gvi, edi[0]), p1i = lds_v(gvi, edi[1]);
  v3 Ei = vsub(p1i, p0i);
  v3 Ej = vsub(p1j, p0j);
  v3 v = vsub(p0i, p0j);
  double c = vdot(Ei, Ei), d = vdot(Ej, Ej), e = vdot(Ei, Ej);
  double f = (c * d) - (e * e);
  if (fabs(f) > 1.0e-12) {
    f = 1.0 / f;
    double a = vdot(Ei, v), b = vdot(Ej, v);
    double s = (e * b - a * d) * f;
    double t = (c * b - e * a) * f;
    if (s >= 0.0 && s <= 1.0 && t >= 0.0 && t <= 1.0) {
      v3 n = vsub(vadd(p0i, vsc(s, Ei)), vadd(p0j, vsc(t, Ej)));
      double sum = Ri + Rj + dmax;
      return vnorm2(n) <= sum * sum;
    }
  }
  return false;
}

// vertex gate of AddOrRemoveInteractions_bruteForce (Rockable.cpp:1385-1393):
// obb_other enlarged by dmax against an axis-aligned box around the vertex
__device__ __forceinline__ bool vertex_gate(v3 gv, double Rowner, const obb_t& other, double dmax) {
  obb_t sub;
  sub.c = gv;
  sub.e[0] = V(1, 0, 0);
  sub.e[1] = V(0, 1, 0);
  sub.e[2] = V(0, 0, 1);
  sub.ext = V(0, 0, 0);
  obb_enlarge(&sub, Rowner + dmax);
  obb_t o = other;
  obb_enlarge(&o, dmax);
  return obb_intersect(o, sub);
}

// Sub-element culls.  They only skip tests whose predicate is false, so the
// add / erase / retain outcome is the reference's:
//  * EdgeIsNearEdge is true only if points of the two segments lie within
//    sum = Ri + Rj + dmax of each other, so each edge's AABB grown by sum
//    meets the vertex AABB of the other body;
//  * VertexIsNearEdge accepts r in [-dmax, 1 + dmax] (r is the fraction
//    along the edge), so the point on the line is within dmax |E|_1 of the
//    edge's AABB;
//  * VertexIsNearFace needs the vertex within sum of its projection P on the
//    face plane with P inside the projected polygon, so P lies within the
//    face's thickness along its normal of the face's AABB.
// Every grown box also gets a margin of 1e-9 (1 + |x|max) for rounding.
__device__ __forceinline__ bool box_meets(const double lo[3], const double hi[3], double grow, const double* blo,
                                          const double* bhi) {
  return lo[0] - grow <= bhi[0] && hi[0] + grow >= blo[0] && lo[1] - grow <= bhi[1] && hi[1] + grow >= blo[1] &&
         lo[2] - grow <= bhi[2] && hi[2] + grow >= blo[2];
}
// The parts of the edge and face culls that depend on the body alone, once
// per body and rebuild instead of once per candidate pair: an edge's box and
// the L1 length of its box; a face's box and its thickness along its normal
// (the face normal from its first two edges, as the predicates take it).
// Stored as 8 floats each (lo[3], hi[3], length or thickness, unused),
// rounded outwards: lo down, hi and the growth terms up, so that the culls
// stay conservative at half the bytes (the narrow phase reads them once per
// candidate pair).  Body b's edges from beoff[b], its faces from bfoff[b].
constexpr int kGate = 8;
__device__ __forceinline__ void store_gate(float* o, const double lo[3], const double hi[3], double x) {
  float4 a, b;
  a.x = __double2float_rd(lo[0]);
  a.y = __double2float_rd(lo[1]);
  a.z = __double2float_rd(lo[2]);
  a.w = __double2float_ru(hi[0]);
  b.x = __double2float_ru(hi[1]);
  b.y = __double2float_ru(hi[2]);
  b.z = __double2float_ru(x);
  b.w = 0.0f;
  reinterpret_cast<float4*>(o)[0] = a;
  reinterpret_cast<float4*>(o)[1] = b;
}
// 2^lg lanes per body (lg from 3 to 6: the shapes' largest edge plus face
// count rounded up), each lane taking every 2^lg-th of its body's elements.
__global__ void k_gate_boxes(Dev d, float* gedge, float* gface, int lg) {
  const unsigned t = blockIdx.x * (unsigned)blockDim.x + threadIdx.x;
  const int b = (int)(t >> lg);
  const int lane = (int)(t & ((1u << lg) - 1u));
  if (b >= d.nb) return;
  const int shp = d.kin[b].shape;
  const int ne = d.sh.ne[shp], nf = d.sh.nf[shp];
  const double* gv = d.gv + 3 * (size_t)d.bvoff[b];
  for (int k = lane; k < ne + nf; k += 1 << lg) {
    double lo[3], hi[3], x;
    if (k < ne) {
      const int* ed = d.sh.edge + 2 * (d.sh.eoff[shp] + k);
      const v3 a = lds_v(gv, ed[0]), c = lds_v(gv, ed[1]);
      lo[0] = fmin(a.x, c.x);
      lo[1] = fmin(a.y, c.y);
      lo[2] = fmin(a.z, c.z);
      hi[0] = fmax(a.x, c.x);
      hi[1] = fmax(a.y, c.y);
      hi[2] = fmax(a.z, c.z);
      x = (hi[0] - lo[0]) + (hi[1] - lo[1]) + (hi[2] - lo[2]);
    } else {
      const int gfc = d.sh.foff[shp] + (k - ne);
      const int fs = d.sh.fstart[gfc];
      const int nbv = d.sh.fstart[gfc + 1] - fs;
      const int* fv = d.sh.fidx + fs;
      const v3 A = lds_v(gv, fv[0]), B = lds_v(gv, fv[1]), C = lds_v(gv, fv[nbv - 1]);
      v3 v1 = vsub(B, A);
      vnormalize(&v1);
      v3 n = vcross(v1, vsub(C, A));
      vnormalize(&n);
      lo[0] = hi[0] = A.x;
      lo[1] = hi[1] = A.y;
      lo[2] = hi[2] = A.z;
      x = 0.0;
      for (int q = 1; q < nbv; q++) {
        const v3 p = lds_v(gv, fv[q]);
        lo[0] = fmin(lo[0], p.x);
        lo[1] = fmin(lo[1], p.y);
        lo[2] = fmin(lo[2], p.z);
        hi[0] = fmax(hi[0], p.x);
        hi[1] = fmax(hi[1], p.y);
        hi[2] = fmax(hi[2], p.z);
        x = fmax(x, fabs(vdot(vsub(p, A), n)));
      }
    }
    store_gate(k < ne ? gedge + kGate * ((size_t)d.beoff[b] + k) : gface + kGate * ((size_t)d.bfoff[b] + (k - ne)),
               lo, hi, x);
  }
}

// The culls (they skip only tests whose predicate is provably false):
// EdgeIsNearEdge needs points of both segments within Ri + Rj + dmax, so an
// edge whose box grown by that (and dmax times its L1 length, for
// VertexIsNearEdge's r in [-dmax, 1 + dmax]) misses the other body's box has
// no test to pass; VertexIsNearFace needs the projection inside the face's
// prism (box grown by twice the face's thickness).
__device__ __forceinline__ bool edge_gate_pre(const float* g, double sum, double dmax, double margin,
                                              const double* blo, const double* bhi) {
  const float4 a = reinterpret_cast<const float4*>(g)[0], b = reinterpret_cast<const float4*>(g)[1];
  const double lo[3] = {a.x, a.y, a.z}, hi[3] = {a.w, b.x, b.y};
  return box_meets(lo, hi, sum + dmax * (double)b.z + margin, blo, bhi);
}
__device__ __forceinline__ bool face_gate_pre(const float* g, double sum, double margin, const double* blo,
                                              const double* bhi) {
  const float4 a = reinterpret_cast<const float4*>(g)[0], b = reinterpret_cast<const float4*>(g)[1];
  const double thick = b.z;
  if (!(thick == thick)) return true;  // degenerate face: no cull
  const double lo[3] = {a.x, a.y, a.z}, hi[3] = {a.w, b.x, b.y};
  return box_meets(lo, hi, sum + 2.0 * thick + margin, blo, bhi);
}



// The largest (hi) or smallest projection on axis a of a point of an edge's
// or face's box (the gate data: lo[3], hi[3] as floats).
__device__ __forceinline__ double gate_box_reach(const float* g, v3 a, bool hi) {
  const float4 p = reinterpret_cast<const float4*>(g)[0], q = reinterpret_cast<const float4*>(g)[1];
  const double lo[3] = {p.x, p.y, p.z}, up[3] = {p.w, q.x, q.y}, ak[3] = {a.x, a.y, a.z};
  double s = 0.0;
  for (int k = 0; k < 3; k++) {
    const double x = ak[k] * lo[k], y = ak[k] * up[k];
    s += hi ? fmax(x, y) : fmin(x, y);
  }
  return s;
}

// floor(k / n) for 0 <= k < 2^20 and n >= 1, with inv = 1 / n in FP32:
// (k + 0.5) / n lies at least 0.5 / n from an integer, and the FP32 product
// is within 3e-7 of it relative, less than that for k < 2^20.  Larger k
// (shapes of thousands of sub-elements) take the integer division.
__device__ __forceinline__ int quot_small(int k, int n, float inv) {
  return k < (1 << 20) ? (int)(((float)k + 0.5f) * inv) : k / n;
}

// Compaction of the indices v < n with pred(v) into list (in ascending
// order) by the SW lanes of one pair (sl: lane within them, g: the pair's
// group of lanes in the wavefront); returns the count.
template <int SW, class F>
__device__ __forceinline__ int group_compact(int n, int sl, int g, int* list, F pred) {
  int base = 0;
  for (int v0 = 0; v0 < n; v0 += SW) {
    const int v = v0 + sl;
    const bool f = v < n && pred(v);
    unsigned long long m = __ballot(f);
    if constexpr (SW < 64) m = (m >> (g * SW)) & ((1ull << SW) - 1ull);
    if (f) list[base + __popcll(m & ((1ull << sl) - 1ull))] = v;
    base += __popcll(m);
  }
  return base;
}

template <int SW>
__device__ __forceinline__ int group_sum(int x) {
  for (int off = SW / 2; off > 0; off >>= 1) x += __shfl_xor(x, off, SW);
  return x;
}
template <int SW>
__device__ __forceinline__ double group_max(double x) {
  for (int off = SW / 2; off > 0; off >>= 1) x = fmax(x, __shfl_xor(x, off, SW));
  return x;
}
template <int SW>
__device__ __forceinline__ double group_min(double x) {
  for (int off = SW / 2; off > 0; off >>= 1) x = fmin(x, __shfl_xor(x, off, SW));
  return x;
}

// Every near test of a pair is false when a plane separates the two
// bodies' vertices by more than the tests reach: a vertex-vertex or edge-edge
// test compares the distance of two points of the vertices' convex hulls with
// sum; a vertex-edge test takes a foot on the edge's line up to dVerlet edge
// lengths past its ends; a vertex-face test takes a foot in the face's outline
// projected on a plane the face's vertices lie within reach[1] of.  The planes
// tried are those normal to the line of centres, whose projection is
// 1-Lipschitz, so a gap along it above sum + those allowances + margin
// (rounding) leaves no test true.  A NaN coordinate turns the test off.
__device__ __forceinline__ double apart_slack(const Dev& d, const BodyKin& Ki, const BodyKin& Kj, int shi, int shj,
                                              double sum, double margin, double dmax) {
  const double* ri = d.sh.reach + 2 * shi;
  const double* rj = d.sh.reach + 2 * shj;
  const double reach = dmax * fmax(Ki.h * ri[0], Kj.h * rj[0]) + fmax(Ki.h * ri[1], Kj.h * rj[1]);
  return sum + reach + margin;
}

// The candidate pairs that need no wavefront of their own, one pair per lane.
//  * Two point shapes (one vertex, no edge or face: the spheres).  Their only
//    test is vertex-vertex, so their result is k_narrow's computed directly:
//    the key (VV, 0, 0) when i's vertex passes the reference's gate against
//    j's OBB, j's vertex lies within sum of i's box and VertexIsNearVertex
//    holds.  A wavefront's near keys go to one stripe (one atomic).
//  * Bodies apart (above): zero counts.  They are more than half of a settled
//    packing's pairs; a wavefront each, which found it out after staging both
//    bodies in LDS, cost a launch slot and idle lanes: k_narrow took 928 us
//    for the 50 005-body pour's 434 000 pairs and 174 us for 13 001 bonded
//    cubes, with this pass 59 + 845 us and 14 + 144 us.
// The others go to list for k_narrow, their count in nrest (one atomic per
// workgroup; their order changes no result).
__global__ void __launch_bounds__(kBlock) k_narrow_lanes(Dev d, const double* bobb, const double* baabb, NarrowCfg cfg,
                                                         int nc, const uint64_t* cand, uint32_t* nearbuf, int* near_cnt,
                                                         int near_rcap, int32_t* cbase, int32_t* cnf, int32_t* cnb,
                                                         int32_t* list, int* nrest) {
  __shared__ int wcnt[kBlock / 64], at;
  const int c = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  bool point = false, near = false, rest = false;
  if (c < nc) {
    const uint64_t key = cand[c];
    const int i = (int)(key >> 32), j = (int)(key & 0xffffffffu);
    const BodyKin &Ki = d.kin[i], &Kj = d.kin[j];
    const int shi = Ki.shape, shj = Kj.shape;
    const double Ri = Ki.R, Rj = Kj.R;
    const int nvi = d.sh.nv[shi], nvj = d.sh.nv[shj];
    const double* gvi = d.gv + 3 * (size_t)d.bvoff[i];
    const double* gvj = d.gv + 3 * (size_t)d.bvoff[j];
    const double *bxi = baabb + 6 * (size_t)i, *bxj = baabb + 6 * (size_t)j;
    double xmax = 0.0;
    for (int k = 0; k < 6; k++) xmax = fmax(fmax(xmax, fabs(bxi[k])), fabs(bxj[k]));
    const double dmax = cfg.dmax;
    const double sum = Ri + Rj + dmax;
    const double margin = 1e-9 * (1.0 + xmax + sum);
    point = nvi == 1 && d.sh.ne[shi] == 0 && d.sh.nf[shi] == 0 && nvj == 1 && d.sh.ne[shj] == 0 && d.sh.nf[shj] == 0;
    if (point) {
      const double gvv = sum + margin;
      const v3 pj = lds_v(gvj, 0);
      const bool jnear = pj.x >= bxi[0] - gvv && pj.x <= bxi[3] + gvv && pj.y >= bxi[1] - gvv &&
                         pj.y <= bxi[4] + gvv && pj.z >= bxi[2] - gvv && pj.z <= bxi[5] + gvv;
      near = jnear && vertex_gate(lds_v(gvi, 0), Ri, load_obb(bobb + 15 * (size_t)j), dmax) &&
             near_vv(gvi, gvj, Ri, Rj, 0, 0, dmax);
    } else {
      v3 ax = V(Kj.px - Ki.px, Kj.py - Ki.py, Kj.pz - Ki.pz);
      const double a2 = vdot(ax, ax);
      bool apart = false;
      if (a2 > 0.0) {
        ax = vsc(1.0 / sqrt(a2), ax);
        // (four vertices of each a round, so that their loads share a latency)
        double hi_i = -INFINITY, lo_j = INFINITY;
        const int nv = nvi > 0 && nvj > 0 ? max(nvi, nvj) : 0;
        for (int v = 0; v < nv; v += 4) {
          double qi[4], qj[4];
#pragma unroll
          for (int k = 0; k < 4; k++) {
            qi[k] = vdot(ax, lds_v(gvi, min(v + k, nvi - 1)));
            qj[k] = vdot(ax, lds_v(gvj, min(v + k, nvj - 1)));
          }
#pragma unroll
          for (int k = 0; k < 4; k++) {
            hi_i = qi[k] == qi[k] ? fmax(hi_i, qi[k]) : INFINITY;
            lo_j = qj[k] == qj[k] ? fmin(lo_j, qj[k]) : -INFINITY;
          }
        }
        apart = lo_j - hi_i > apart_slack(d, Ki, Kj, shi, shj, sum, margin, dmax);
      }
      rest = !apart;
      // (k_narrow rewrites the others'; the merge's count may run before it)
      cbase[c] = 0;
      cnf[c] = 0;
      cnb[c] = 0;
    }
  }
  const unsigned long long m = __ballot(near), mr = __ballot(rest);
  if (lane == 0) wcnt[wv] = __popcll(mr);
  const int stripe = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6) & (kStripes - 1);
  int base = 0;
  if (lane == 0 && m) base = atomicAdd(near_cnt + stripe * kStripeStride, __popcll(m));
  base = __shfl(base, 0, 64);
  const unsigned long long below = (1ull << lane) - 1ull;
  if (point) {
    const int local = base + __popcll(m & below);
    // over capacity: no key, and the host re-runs with a larger buffer
    const bool room = local < near_rcap;
    cbase[c] = room ? stripe * near_rcap + local : 0;
    cnf[c] = near && room ? 1 : 0;
    cnb[c] = 0;
    if (near && room) nearbuf[stripe * near_rcap + local] = pack_sub(VV, 0, 0);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int n = wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
    at = n ? atomicAdd(nrest, n) : 0;
  }
  __syncthreads();
  if (rest) {
    int k = at + __popcll(mr & below);
    for (int w = 0; w < wv; w++) k += wcnt[w];
    list[k] = c;
  }
}

// P candidate pairs per wavefront (64 / P lanes each, LDS stride `stride`
// bytes per pair): the work of a pair is mostly a fixed sequence of
// wavefront instructions (gates, compactions, one pass per predicate, the
// key output), which the pairs of a wavefront then share.  Occupancy asked
// of the compiler: 6 wavefronts per SIMD with one pair (80 VGPRs, no
// spill), 3 with two.
template <int P>
__global__ void __launch_bounds__(64, P == 1 ? 6 : 3) k_narrow(Dev d, const double* bobb, const double* baabb, NarrowCfg cfg,
                                               const uint64_t* cand, uint32_t* nearbuf, int* near_cnt,
                                               int near_rcap, int32_t* cbase, int32_t* cnf, int32_t* cnb,
                                               int stride, const int32_t* clist, const int* nrest, int first) {
  constexpr int SW = 64 / P;
  extern __shared__ double lds_all[];
  const int lane = threadIdx.x;
  // (with one pair per wavefront the pair's values stay wavefront-uniform,
  // in scalar registers)
  const int g = P == 1 ? 0 : lane / SW, sl = P == 1 ? lane : lane % SW;
  // the idx-th pair to test: candidate clist[idx], of *nrest (the grid is
  // sized from the last rebuild's count, before this one's is known)
  const int idx = first + xcd_block((int)blockIdx.x, (int)gridDim.x) * P + g;
  const bool valid = idx < *nrest;
  if (P == 1 ? !valid : !__any(valid)) return;
  const int c = valid ? clist[idx] : 0;
  double* lds = lds_all + (size_t)g * (stride / 8);
  uint64_t key = 0;
  if (valid) key = cand[c];
  const int i = (int)(key >> 32), j = (int)(key & 0xffffffffu);
  const int shi = d.kin[i].shape, shj = d.kin[j].shape;
  const double Ri = d.kin[i].R, Rj = d.kin[j].R;
  // an invalid group (past the last pair) takes body 0 twice with no
  // sub-element, so that it runs every pass with nothing to do
  const int nvi = valid ? d.sh.nv[shi] : 0, nvj = valid ? d.sh.nv[shj] : 0;
  const int nei = valid ? d.sh.ne[shi] : 0, nej = valid ? d.sh.ne[shj] : 0;
  const int nfi = valid ? d.sh.nf[shi] : 0, nfj = valid ? d.sh.nf[shj] : 0;
  double* pbox = lds;                // 48 doubles: both OBBs and both body boxes (several pairs per wavefront)
  double* gvi = lds + 48;
  double* gvj = gvi + 3 * cfg.maxv;
  unsigned long long* bits = (unsigned long long*)(gvj + 3 * cfg.maxv);
  int* lst = (int*)(bits + cfg.maxwords);
  int* vg_l = lst;                  // gated vertices: i's as v, j's as maxv + v
  int* vjn_l = vg_l + 2 * cfg.maxv; // vertices of j near i's box (vertex-vertex)
  int* ef_l = vjn_l + cfg.maxv;     // gated edges and faces, tagged (see below)
  int* wpre = ef_l + 2 * cfg.maxe + 2 * cfg.maxf + 8;  // prefix of the bit counts per word

  // test order of the reference (AddOrRemoveInteractions_bruteForce): the
  // bit of test (segment s, own, oth) is segstart[s] + own * n_oth[s] + oth
  const int s1 = nvi * nvj, s2 = s1 + nvi * nej, s3 = s2 + nvi * nfj, s4 = s3 + nei * nej, s5 = s4 + nvj * nei;
  const int T = s5 + nvj * nfi, Tf = s4;
  // (nwords <= maxwords: the shapes are checked at load)
  const int nwords = min((T + 63) / 64, cfg.maxwords);
  for (int w = sl; w < nwords; w += SW) bits[w] = 0ull;
  {
    const double* src_i = d.gv + 3 * (size_t)d.bvoff[i];
    const double* src_j = d.gv + 3 * (size_t)d.bvoff[j];
    for (int q = sl; q < 3 * nvi; q += SW) gvi[q] = src_i[q];
    for (int q = sl; q < 3 * nvj; q += SW) gvj[q] = src_j[q];
  }
  // the OBBs and the body boxes (vertices +- Minkowski radius, from k_obb)
  // of both bodies: read where they lie when the pair's values are uniform
  // over the wavefront (scalar loads), else from copies in the pair's LDS
  // (vector registers would hold them for every lane)
  const double *obi = bobb + 15 * (size_t)i, *obj = bobb + 15 * (size_t)j;
  const double *bxi = baabb + 6 * (size_t)i, *bxj = baabb + 6 * (size_t)j;
  if (P > 1) {
    for (int q = sl; q < 42; q += SW)
      pbox[q] = q < 15 ? obi[q] : q < 30 ? obj[q - 15] : q < 36 ? bxi[q - 30] : bxj[q - 36];
    obi = pbox;
    obj = pbox + 15;
    bxi = pbox + 30;
    bxj = pbox + 36;
  }
  __syncthreads();
  double xmax = 0.0;
  for (int k = 0; k < 6; k++) xmax = fmax(fmax(xmax, fabs(bxi[k])), fabs(bxj[k]));
  const double dmax = cfg.dmax;
  const double sum = Ri + Rj + dmax;
  const double margin = 1e-9 * (1.0 + xmax + sum);

  // Slab culls: the bound that sends pairs apart away (k_narrow_lanes) culls
  // single elements of the others: a test of an element of i needs its hull's
  // projection on the line of centres to reach lo_j - slack (lim_i), one of
  // j's to reach down to hi_i + slack (lim_j); the culls apply it to the
  // vertices and to the edges' and faces' boxes, which hold them.
  v3 ax = V(0.0, 0.0, 0.0);
  double lim_i = -INFINITY, lim_j = INFINITY;
  // bit v: vertex v within the limit (all set where not computed, shapes of
  // more than SW vertices)
  unsigned long long keep_i = ~0ull, keep_j = ~0ull;
  if (valid) {
    const BodyKin& Ki = d.kin[i];
    const BodyKin& Kj = d.kin[j];
    ax = V(Kj.px - Ki.px, Kj.py - Ki.py, Kj.pz - Ki.pz);
    const double a2 = vdot(ax, ax);
    if (a2 > 0.0) {
      ax = vsc(1.0 / sqrt(a2), ax);
      double hi_i = -INFINITY, lo_j = INFINITY, qi = 0.0, qj = 0.0;
      for (int v = sl; v < nvi; v += SW) {
        qi = vdot(ax, lds_v(gvi, v));
        hi_i = qi == qi ? fmax(hi_i, qi) : INFINITY;
      }
      for (int v = sl; v < nvj; v += SW) {
        qj = vdot(ax, lds_v(gvj, v));
        lo_j = qj == qj ? fmin(lo_j, qj) : -INFINITY;
      }
      hi_i = group_max<SW>(hi_i);
      lo_j = group_min<SW>(lo_j);
      const double slack = apart_slack(d, Ki, Kj, shi, shj, sum, margin, dmax);
      const double li = lo_j - slack, lj = hi_i + slack;
      if (li == li) lim_i = li;
      if (lj == lj) lim_j = lj;
      if (nvi <= SW && nvj <= SW) {
        // (qi, qj: the lane's own vertex; a NaN one is dropped, as its tests are false)
        unsigned long long bi = __ballot(sl < nvi && qi >= lim_i), bj = __ballot(sl < nvj && qj <= lim_j);
        if constexpr (SW < 64) {
          bi = (bi >> (g * SW)) & ((1ull << SW) - 1ull);
          bj = (bj >> (g * SW)) & ((1ull << SW) - 1ull);
        }
        keep_i = bi;
        keep_j = bj;
      }
    } else {
      ax = V(0.0, 0.0, 0.0);
    }
  }
  // edges and faces of both bodies in one pass, index q over i's edges, j's
  // edges, i's faces, j's faces (before the vertices, so that ax and the
  // limits are dead in the vertex gates' registers)
  const int ne2 = nei + nej, nef = ne2 + nfi + nfj;
  const float* gei = cfg.gedge + kGate * (size_t)d.beoff[i];
  const float* gej = cfg.gedge + kGate * (size_t)d.beoff[j];
  const float* gfi = cfg.gface + kGate * (size_t)d.bfoff[i];
  const float* gfj = cfg.gface + kGate * (size_t)d.bfoff[j];
  const int nefg = group_compact<SW>(nef, sl, g, ef_l, [&](int q) {
    if (q < nei) {
      const float* gb = gei + kGate * q;
      return gate_box_reach(gb, ax, true) >= lim_i && edge_gate_pre(gb, sum, dmax, margin, bxj, bxj + 3);
    }
    if (q < ne2) {
      const float* gb = gej + kGate * (q - nei);
      return gate_box_reach(gb, ax, false) <= lim_j && edge_gate_pre(gb, sum, dmax, margin, bxi, bxi + 3);
    }
    if (q < ne2 + nfi) {
      const float* gb = gfi + kGate * (q - ne2);
      return gate_box_reach(gb, ax, true) >= lim_i && face_gate_pre(gb, sum, margin, bxj, bxj + 3);
    }
    const float* gb = gfj + kGate * (q - ne2 - nfi);
    return gate_box_reach(gb, ax, false) <= lim_j && face_gate_pre(gb, sum, margin, bxi, bxi + 3);
  });
  // reference vertex gates of both bodies in one pass: i's vertices against
  // j's OBB, j's against i's
  const int nvg = group_compact<SW>(nvi + nvj, sl, g, vg_l, [&](int v) {
    if (v < nvi) return (v >= 64 || ((keep_i >> v) & 1ull)) && vertex_gate(lds_v(gvi, v), Ri, load_obb(obj), dmax);
    const int u = v - nvi;
    return (u >= 64 || ((keep_j >> u) & 1ull)) && vertex_gate(lds_v(gvj, u), Rj, load_obb(obi), dmax);
  });
  // vertex-vertex partners: vertices of j within sum of i's box
  const double gvv = sum + margin;
  const int nvj_n = group_compact<SW>(nvj, sl, g, vjn_l, [&](int v) {
    const v3 p = lds_v(gvj, v);
    return p.x >= bxi[0] - gvv && p.x <= bxi[3] + gvv && p.y >= bxi[1] - gvv && p.y <= bxi[4] + gvv &&
           p.z >= bxi[2] - gvv && p.z <= bxi[5] + gvv && (v >= 64 || ((keep_j >> v) & 1ull));
  });
  // split the compacted lists by kind (they are in ascending q, so each kind
  // is a contiguous run)
  int nvi_g = 0, nei_g = 0, nej_g = 0, nfi_g = 0;
  for (int k = sl; k < nvg; k += SW) nvi_g += vg_l[k] < nvi ? 1 : 0;
  for (int k = sl; k < nefg; k += SW) {
    const int q = ef_l[k];
    nei_g += q < nei ? 1 : 0;
    nej_g += (q >= nei && q < ne2) ? 1 : 0;
    nfi_g += (q >= ne2 && q < ne2 + nfi) ? 1 : 0;
  }
  nvi_g = group_sum<SW>(nvi_g);
  nei_g = group_sum<SW>(nei_g);
  nej_g = group_sum<SW>(nej_g);
  nfi_g = group_sum<SW>(nfi_g);
  const int nvj_g = nvg - nvi_g, nfj_g = nefg - nei_g - nej_g - nfi_g;
  const int* vi_l = vg_l;            // values v
  const int* vj_l = vg_l + nvi_g;    // values nvi + v
  const int* ei_l = ef_l;            // values e
  const int* ej_l = ef_l + nei_g;    // values nei + e
  const int* fi_l = ej_l + nej_g;    // values ne2 + f
  const int* fj_l = fi_l + nfi_g;    // values ne2 + nfi + f
  __syncthreads();

  // one loop per segment, so that a wavefront runs one predicate at a time
  int n = nvi_g * nvj_n;
  float inv = 1.0f / (float)max(nvj_n, 1);
  for (int k = sl; k < n; k += SW) {
    const int q = quot_small(k, nvj_n, inv);
    const int a = vi_l[q], b = vjn_l[k - q * nvj_n];
    if (near_vv(gvi, gvj, Ri, Rj, a, b, dmax)) {
      const int bit = a * nvj + b;
      atomicOr(bits + (bit >> 6), 1ull << (bit & 63));
    }
  }
  // vertex-edge both ways in one pass (i's vertices against j's edges, then
  // j's against i's, the same predicate with the roles swapped per lane),
  // and vertex-face likewise: a wavefront runs each predicate once where
  // the two directions' tests fit its lanes together
  {
    const int n1 = nvi_g * nej_g, n2 = nvj_g * nei_g;
    const float inv1 = 1.0f / (float)max(nej_g, 1), inv2 = 1.0f / (float)max(nei_g, 1);
    for (int k = sl; k < n1 + n2; k += SW) {
      const bool fw = k < n1;
      const int kk = fw ? k : k - n1, no = fw ? nej_g : nei_g;
      const int q = quot_small(kk, no, fw ? inv1 : inv2);
      const int a = fw ? vi_l[q] : vj_l[q] - nvi;
      const int b = fw ? ej_l[kk - q * no] - nei : ei_l[kk - q * no];
      if (near_ve(d.sh, fw ? shj : shi, fw ? gvi : gvj, fw ? gvj : gvi, fw ? Ri : Rj, fw ? Rj : Ri, a, b, dmax)) {
        const int bit = fw ? s1 + a * nej + b : s4 + a * nei + b;
        atomicOr(bits + (bit >> 6), 1ull << (bit & 63));
      }
    }
  }
  {
    const int n1 = nvi_g * nfj_g, n2 = nvj_g * nfi_g;
    const float inv1 = 1.0f / (float)max(nfj_g, 1), inv2 = 1.0f / (float)max(nfi_g, 1);
    for (int k = sl; k < n1 + n2; k += SW) {
      const bool fw = k < n1;
      const int kk = fw ? k : k - n1, no = fw ? nfj_g : nfi_g;
      const int q = quot_small(kk, no, fw ? inv1 : inv2);
      const int a = fw ? vi_l[q] : vj_l[q] - nvi;
      const int b = fw ? fj_l[kk - q * no] - ne2 - nfi : fi_l[kk - q * no] - ne2;
      if (near_vf(d.sh, fw ? shj : shi, fw ? gvi : gvj, fw ? gvj : gvi, fw ? Ri : Rj, fw ? Rj : Ri, a, b, dmax)) {
        const int bit = fw ? s2 + a * nfj + b : s5 + a * nfi + b;
        atomicOr(bits + (bit >> 6), 1ull << (bit & 63));
      }
    }
  }
  n = nei_g * nej_g;
  inv = 1.0f / (float)max(nej_g, 1);
  for (int k = sl; k < n; k += SW) {
    const int q = quot_small(k, nej_g, inv);
    const int a = ei_l[q], b = ej_l[k - q * nej_g] - nei;
    if (near_ee(d.sh, shi, shj, gvi, gvj, Ri, Rj, a, b, dmax)) {
      const int bit = s3 + a * nej + b;
      atomicOr(bits + (bit >> 6), 1ull << (bit & 63));
    }
  }
  __syncthreads();
  // counts per direction
  int cf = 0, cb = 0;
  for (int w = sl; w < nwords; w += SW) {
    const unsigned long long m = bits[w];
    const int lo = w * 64;
    if (lo + 64 <= Tf)
      cf += __popcll(m);
    else if (lo >= Tf)
      cb += __popcll(m);
    else {
      const int k = Tf - lo;
      const unsigned long long fm = (k >= 64) ? ~0ull : ((1ull << k) - 1ull);
      cf += __popcll(m & fm);
      cb += __popcll(m & ~fm);
    }
  }
  cf = group_sum<SW>(cf);
  cb = group_sum<SW>(cb);
  const int stripe = c & (kStripes - 1);
  int local = 0;
  if (valid && sl == 0) local = atomicAdd(near_cnt + stripe * kStripeStride, cf + cb);
  local = __shfl(local, 0, SW);
  const int base_out = stripe * near_rcap + local;
  // over capacity: no keys, and the host re-runs with a larger buffer
  const bool room = valid && local + cf + cb <= near_rcap;
  if (valid && sl == 0) {
    cbase[c] = room ? base_out : 0;
    cnf[c] = room ? cf : 0;
    cnb[c] = room ? cb : 0;
  }
  // write the keys in test order (output slot = rank of the set bit), one
  // key per lane: the exclusive prefix of the words' bit counts in LDS, then
  // key q's word by a binary search over it and its bit as the
  // (q - prefix)-th set bit of the word (a binary search over popcounts)
  {
    int running = 0;
    for (int w0 = 0; w0 < nwords; w0 += SW) {
      const int w = w0 + sl;
      const int pc = w < nwords ? __popcll(bits[w]) : 0;
      int incl = pc;
      for (int off = 1; off < SW; off <<= 1) {
        const int y = __shfl_up(incl, off, SW);
        if (sl >= off) incl += y;
      }
      if (w < nwords) wpre[w] = running + incl - pc;
      running += __shfl(incl, SW - 1, SW);
    }
  }
  __syncthreads();
  const int ntot = room ? cf + cb : 0;
  for (int q = sl; q < ntot; q += SW) {
    int lo = 0, hi = nwords - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (wpre[mid] <= q)
        lo = mid;
      else
        hi = mid - 1;
    }
    unsigned long long m = bits[lo];
    int r = q - wpre[lo], bit = 0;
    for (int width = 32; width > 0; width >>= 1) {
      const int cnt = __popcll(m & ((1ull << width) - 1ull));
      if (r >= cnt) {
        r -= cnt;
        m >>= width;
        bit += width;
      }
    }
    const int t = lo * 64 + bit;
    // the segment of test t: its type, first bit and count of "other" elements
    int type, first, noth;
    if (t < s1) {
      type = VV, first = 0, noth = nvj;
    } else if (t < s2) {
      type = VE, first = s1, noth = nej;
    } else if (t < s3) {
      type = VF, first = s2, noth = nfj;
    } else if (t < s4) {
      type = EE, first = s3, noth = nej;
    } else if (t < s5) {
      type = VE, first = s4, noth = nei;
    } else {
      type = VF, first = s5, noth = nfi;
    }
    const int rt = t - first;
    const int own = quot_small(rt, noth, 1.0f / (float)noth);
    nearbuf[base_out + q] = pack_sub(type, own, rt - own * noth);
  }
}

// --- merge ---------------------------------------------------------------
struct MergeIn {
  int ng;  // group slots
  const uint64_t* ukey;
  const int32_t* ucand;
  const int32_t* uold;
  const int32_t* ostart;  // old group start, size ng_old + 1 (trailing = n_old)
  const int32_t* cbase;
  const int32_t* cnf;
  const int32_t* cnb;
  const uint32_t* nearbuf;
  const double* bobb;
  double dmax;
  // old entries
  const int32_t* oi;
  const int32_t* oj;
  const uint32_t* osub;
  const EState* oest;
  const double* oedn;
  const EGeom* ogeo;
  const double* odamp;
  const int32_t* ostick;
  const uint8_t* oeact;
  const double* oekey;
};
struct MergeOut {
  int32_t* count;   // per group (count pass)
  const int32_t* offset;  // per group (write pass)
  int32_t* src;     // per new entry (write pass): the old entry kept, -1 for a fresh one
  int32_t* ei;
  int32_t* ej;
  uint32_t* esub;
  EState* est;
  double* edn;
  EGeom* egeo;
  double* edamp;
  int32_t* estick;
  uint8_t* eact;
  double* ekey;
};

// Damp of the body pair (Rockable.cpp:1356-1376), pair (i < j)
__device__ double pair_damp(const Dev& d, int i, int j) {
  const int gi = d.kin[i].group, gj = d.kin[j].group;
  if (gi < 0 || gj < 0 || gi >= d.par.G || gj >= d.par.G) return 0.0;
  const int gp = gi * d.par.G + gj;
  const int kind = d.par.damp_kind[gp];
  if (kind == 2) return 0.0;
  const double kn = d.par.tab[(P_KN * d.par.G + gi) * d.par.G + gj];
  double meff;
  if (i < d.nDriven)
    meff = d.mass[j];
  else if (j < d.nDriven)
    meff = d.mass[i];
  else
    meff = (d.mass[i] * d.mass[j]) / (d.mass[i] + d.mass[j]);
  if (kind == 0) return d.par.damp_rate[gp] * 2.0 * sqrt(kn * meff);
  return 2.0 * sqrt(kn * meff);
}

template <bool WRITE>
__global__ void k_merge(Dev d, MergeIn in, MergeOut out) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g > in.ng) return;
  const int cref = g < in.ng ? in.ucand[g] : -1, oref = g < in.ng ? in.uold[g] : -1;
  if (cref < 0 && oref < 0) {  // an empty slot, or the scan's trailing zero
    if (!WRITE) out.count[g] = 0;
    return;
  }
  const uint64_t key = in.ukey[g];
  const int owner = (int)(key >> 32), other = (int)(key & 0xffffffffu);
  int os = 0, on = 0;
  if (oref >= 0) {
    os = in.ostart[oref];
    on = in.ostart[oref + 1] - os;
  }
  int ns = 0, nn = 0;
  bool fwd = true;
  if (cref >= 0) {
    const int c = cref >> 1;
    fwd = (cref & 1) == 0;
    ns = in.cbase[c] + (fwd ? 0 : in.cnf[c]);
    nn = fwd ? in.cnf[c] : in.cnb[c];
  }
  const bool candidate = cref >= 0;
  const BodyKin Po = d.kin[owner];
  obb_t oth;
  if (candidate) oth = load_obb(in.bobb + 15 * (size_t)other);
  int cnt = WRITE ? out.offset[g] : 0;
  int a = 0, b = 0;
  while (a < on || b < nn) {
    const uint32_t sa = (a < on) ? in.osub[os + a] : 0xffffffffu;
    const uint32_t sb = (b < nn) ? in.nearbuf[ns + b] : 0xffffffffu;
    int take;  // 0 old kept, 1 fresh near, 2 old matched by near, -1 old erased
    if (b < nn && (a >= on || sb < sa)) {
      take = 1;
    } else if (a < on && (b >= nn || sa < sb)) {
      bool tested = false;
      if (candidate) {
        const int type = (int)(sa >> 30), isub = (int)((sa >> 15) & 0x7fffu);
        if (fwd && type == EE)
          tested = true;
        else if (type == VV || type == VE || type == VF) {
          if (fwd || type != VV) {
            const double* g = d.gv + 3 * ((size_t)d.bvoff[owner] + isub);
            tested = vertex_gate(V(g[0], g[1], g[2]), Po.R, oth, in.dmax);
          }
        }
      }
      take = tested ? -1 : 0;
    } else {
      take = 2;
    }
    if (take != -1) {
      if (WRITE) {
        // Records are filled by k_merge_fill, one thread per entry: written
        // here, a group's records would be strided stores across the wavefront.
        const int e = cnt;
        out.ei[e] = owner;
        out.ej[e] = other;
        out.esub[e] = take == 1 ? sb : in.osub[os + a];
        out.src[e] = take == 1 ? -1 : os + a;
      }
      cnt++;
    }
    if (take == 1)
      b++;
    else if (take == 2) {
      a++;
      b++;
    } else
      a++;
  }
  if (!WRITE) out.count[g] = cnt;
}

// Records of the merged entries: a fresh entry starts from zero state with the
// damp of its body pair; a kept one carries its old state, active as it was at
// the last accelerations() (Rockable.cpp:1356-1376 for the damp).
__global__ void k_merge_fill(Dev d, int n, MergeIn in, MergeOut out) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int o = out.src[e];
  if (o < 0) {
    const int i = out.ei[e], j = out.ej[e];
    EState s;
    s.fn = 0.0;
    s.ftx = s.fty = s.ftz = 0.0;
    s.momx = s.momy = s.momz = 0.0;
    out.est[e] = s;
    out.edn[e] = 0.0;
    EGeom q;
    q.nx = q.ny = q.nz = q.px = q.py = q.pz = q.vx = q.vy = q.vz = 0.0;
    out.egeo[e] = q;
    out.edamp[e] = pair_damp(d, i < j ? i : j, i < j ? j : i);
    out.estick[e] = -1;
    out.eact[e] = 0;
  } else {
    const double dn = in.oedn[o];
    const int stick = in.ostick[o];
    const EState st = in.oest[o];
    out.est[e] = st;
    out.edn[e] = dn;
    out.egeo[e] = in.ogeo[o];
    out.edamp[e] = in.odamp[o];
    out.estick[e] = stick;
    // bit 1: the history is not all zero (a NaN counts as non-zero); bit 0
    // is kept: the entries active at the last force phase stay the active
    // set until the next one (activeInteractions holds its pointers through
    // UpdateNL, Rockable.cpp:3005-3029), a bond broken in that phase included
    const bool hist = !(st.fn == 0.0 && st.ftx == 0.0 && st.fty == 0.0 && st.ftz == 0.0 && st.momx == 0.0 &&
                        st.momy == 0.0 && st.momz == 0.0);
    out.eact[e] = (in.oeact[o] & 1) | (hist ? 2 : 0);
  }
  // the far-entry key: a kept entry keeps its own (the key bounds the
  // entry's gap through the bodies' accumulated motion, which a rebuild does
  // not reset); a new entry is evaluated at its first step
  out.ekey[e] = o >= 0 ? in.oekey[o] : -INFINITY;
}

// --- CSR -----------------------------------------------------------------
// --- resultant slots -------------------------------------------------------
// compute_resultants (Rockable.cpp:3267-3272) walks the bodies in index order
// and each body's interactions in key order, adding to Particles[i] and
// subtracting from Particles[j]; so body b receives, in this order, the
// entries (a, b) with a < b, then its own entries (b, c), then the entries
// (a, b) with a > b.  Body b's slots are [soff[b], soff[b+1]) with
// soff[b] = istart[b] + jstart[b]; nlow[b] counts b's j-side entries whose
// index is below b's own range: it is the count of b's j-side entries with a < b, and entry
// (i, j) takes slot jstart[i] + nlow[i] + e on its owner's side, and on the
// other the number of j's j-side entries before it, after j's own entries if
// it comes after them.
//
// The j-side counts (whole in the low 32 bits, below the own range in the
// high ones), every entry's position among its j's, and the first entry of
// every owner (ei ascends).
__global__ void k_csr_count(int nb, int n, const int32_t* ei, const int32_t* ej, int32_t* istart, unsigned long long* jcnt,
                            int32_t* at) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = t < n;
  const int i = valid ? ei[t] : 0, j = valid ? ej[t] : 0;
  const int q = run_add(jcnt, j, valid, (unsigned long long)(i < j ? 0x100000001ull : 1ull), i < j);
  if (valid) at[t] = q;
  if (t > nb) return;
  // 8 independent loads a round instead of a binary search's one
  int lo = 0, hi = n;  // the first entry whose owner is t or above lies in [lo, hi]
  while (hi > lo) {
    const int st = (hi - lo + 7) / 8;
    int nlo = lo, nhi = hi;
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int x = lo + st * q;
      if (x < hi) {
        if (ei[x] < t)
          nlo = x + 1 > nlo ? x + 1 : nlo;
        else
          nhi = x < nhi ? x : nhi;
      }
    }
    lo = nlo;
    hi = nhi;
  }
  istart[t] = lo;
}
// the j-side entries by body, in any order, and the bodies' slots; jsum is the
// scan of the counts, whose low 32 bits stay below 2^32
__global__ void k_csr_fill(int nb, int n, const int32_t* ej, const int32_t* istart, const unsigned long long* jcnt,
                           const unsigned long long* jsum, const int32_t* at, int32_t* jstart, int32_t* nlow,
                           int32_t* jlist, int32_t* soff) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) jlist[(int32_t)jsum[ej[t]] + at[t]] = t;
  if (t <= nb) {
    const int32_t js = (int32_t)jsum[t];
    jstart[t] = js;
    soff[t] = istart[t] + js;
    nlow[t] = (int32_t)(jcnt[t] >> 32);
  }
}
struct SlotIn {
  int n;
  const int32_t* ei;
  const int32_t* ej;
  const int32_t* istart;
  const int32_t* jstart;
  const int32_t* jlist;
  const int32_t* nlow;
  const uint8_t* eact;
  int32_t* spos;
  uint8_t* sact;
  int32_t* nbig;
  int32_t* big;
};
// the slot of j-side entry e, `before` of b's j-side entries being below it
// (slot activity of a fresh list: the force phase rewrites it only on change)
__device__ __forceinline__ void put_slot_j(const SlotIn& S, int b, int e, int before) {
  const int i0 = S.istart[b];
  const int at = i0 + S.jstart[b] + before + (e >= i0 ? S.istart[b + 1] - i0 : 0);
  S.spos[2 * e + 1] = at;
  S.sact[at] = S.eact[e] & 1;
}
__global__ void k_csr_slots(SlotIn S) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= S.n) return;
  const int i = S.ei[t];
  const int at = S.jstart[i] + S.nlow[i] + t;
  S.spos[2 * t] = at;
  S.sact[at] = S.eact[t] & 1;
  const int e = S.jlist[t], b = S.ej[e];
  const int s0 = S.jstart[b], s1 = S.jstart[b + 1];
  if (s1 - s0 > kSegMax) {
    if (t == s0) S.big[atomicAdd(S.nbig, 1)] = b;
    return;
  }
  put_slot_j(S, b, e, seg_below(S.jlist, s0, s1, e));
}
__global__ void __launch_bounds__(kWinThreads) k_csr_slots_big(SlotIn S) {
  __shared__ WinLds L;
  const int nbig = *S.nbig, win = (int)blockIdx.y;
  for (int q = (int)blockIdx.x; q < nbig; q += (int)gridDim.x) {
    const int b = S.big[q];
    const int s0 = S.jstart[b], s1 = S.jstart[b + 1];
    const int below = win_mark(L, S.jlist, s0, s1, win);
    for (int t = s0 + (int)threadIdx.x; t < s1; t += kWinThreads) {
      const int e = S.jlist[t];
      if ((e >> kWinBits) == win) put_slot_j(S, b, e, below + win_rank(L, e));
    }
  }
}
// The heavy bodies (more than heavy_min slots) in any order: no sum depends on
// it.  Body and chunk offsets come from one 64-bit counter, so that they
// ascend together: heavy body h has the chunks [hch_off[h], hch_off[h + 1]),
// each a chunk of 64 of its slots.  out: the chunk count in the low and the
// heavy count in the high 32 bits; np the heavy bodies that are not passive.
// (One kernel instead of a flag, a scan, a compaction and a serial pass over
// the list, 38 us in the last alone for 50 005 bodies: 22 us in all.)
__global__ void k_heavy_list(int nb, const int32_t* soff, int heavy_min, const uint8_t* passive, int32_t* heavy,
                             int32_t* hch_off, int2* hch, int cap, unsigned long long* out, int32_t* np) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int k0 = soff[b], k1 = soff[b + 1];
  if (k1 - k0 <= heavy_min) return;
  const int nch = (k1 - k0 + 63) / 64;
  const unsigned long long at = atomicAdd(out, (1ull << 32) + (unsigned long long)nch);
  const int h = (int)(at >> 32), c0 = (int)(uint32_t)at;
  if (!passive[b]) atomicAdd(np, 1);
  heavy[h] = b;
  hch_off[h] = c0;
  hch_off[h + 1] = c0 + nch;  // the next heavy body writes the same
  for (int c = 0; c < nch && c0 + c < cap; c++) hch[c0 + c] = make_int2(k0 + 64 * c, min(k0 + 64 * c + 64, k1));
}

inline int nblk(long n) { return (int)((n + kBlock - 1) / kBlock); }

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <class T>
static int ensure(NLWork& w, T*& p, size_t& cap, size_t n) {
  if (n <= cap && p) return 0;
  if (p) (void)hipFree(p);
  size_t c = n + n / 2 + 256;
  if (hipMalloc(&p, c * sizeof(T)) != hipSuccess) {
    snprintf(w.err, sizeof(w.err), "hipMalloc of %zu bytes failed", c * sizeof(T));
    p = nullptr;
    cap = 0;
    return -1;
  }
  cap = c;
  return 0;
}

template <class T>
static int scan_exclusive(NLWork& w, const T* in, T* out, int n, hipStream_t s) {
  size_t bytes = 0;
  RK_CHECK(rocprim::exclusive_scan(nullptr, bytes, in, out, (T)0, (size_t)n, rocprim::plus<T>(), s));
  if (ensure(w, w.tmp, w.tmp_cap, bytes) != 0) return -1;
  RK_CHECK(rocprim::exclusive_scan((void*)w.tmp, bytes, in, out, (T)0, (size_t)n, rocprim::plus<T>(), s));
  return 0;
}

// windows of values below n for the long segments
static int windows(long n) { return (int)std::max(1L, (n + (1L << kWinBits) - 1) >> kWinBits); }

int nl_build_csr(NLWork& w, int nb, EntryArrays& E, const uint8_t* passive, hipStream_t s) {
  const int n = E.n;
  if (ensure(w, E.istart, E.istart_cap, (size_t)nb + 1) || ensure(w, E.jstart, E.jstart_cap, (size_t)nb + 1) ||
      ensure(w, E.jlist, E.jlist_cap, (size_t)(n > 0 ? n : 1)) || ensure(w, w.i32a, w.i32a_cap, (size_t)nb + 1) ||
      ensure(w, w.i32b, w.i32b_cap, (size_t)(n > 0 ? n : 1)) || ensure(w, w.jsum, w.jsum_cap, 2 * (size_t)nb + 3) ||
      ensure(w, E.edesc, E.edesc_cap, 2 * (size_t)(n > 0 ? n : 1)) ||
      ensure(w, E.soff, E.soff_cap, (size_t)nb + 1) || ensure(w, w.big, w.big_cap, (size_t)nb))
    return -1;
  // zeroed: the j-side counts and, behind them, the count of long segments
  unsigned long long *jcnt = w.jsum, *jsum = jcnt + nb + 2;
  int32_t *nlow = w.i32a, *nbig = reinterpret_cast<int32_t*>(jcnt + nb + 1);
  const int grid = nblk(std::max((long)n, (long)nb + 1));
  RK_CHECK(hipMemsetAsync(jcnt, 0, sizeof(unsigned long long) * ((size_t)nb + 2), s));
  hipLaunchKernelGGL(k_csr_count, dim3(grid), dim3(kBlock), 0, s, nb, n, E.ei, E.ej, E.istart, jcnt, w.i32b);
  if (scan_exclusive(w, jcnt, jsum, nb + 1, s)) return -1;
  hipLaunchKernelGGL(k_csr_fill, dim3(grid), dim3(kBlock), 0, s, nb, n, E.ej, E.istart, jcnt, jsum, w.i32b, E.jstart,
                     nlow, E.jlist, E.soff);
  if (n > 0) {
    SlotIn S{n, E.ei, E.ej, E.istart, E.jstart, E.jlist, nlow, E.eact, E.spos, E.sact, nbig, w.big};
    hipLaunchKernelGGL(k_csr_slots, dim3(nblk(n)), dim3(kBlock), 0, s, S);
    if (n > kSegMax) hipLaunchKernelGGL(k_csr_slots_big, dim3(kBigGrid, windows(n)), dim3(kWinThreads), 0, s, S);
  }
  RK_CHECK(hipGetLastError());
  return nl_build_heavy(w, nb, E, passive, s);
}

// Reads of small device values through the pinned staging buffer: copy_in
// queues the copies (byte offsets into the buffer), wait synchronises the
// stream and copy_out takes the values.
constexpr size_t kPinBytes = 8192;
static char* pin_buf(NLWork& w) {
  if (!w.pin && hipHostMalloc((void**)&w.pin, kPinBytes, hipHostMallocDefault) != hipSuccess) w.pin = nullptr;
  return w.pin;
}
static int read_small(NLWork& w, hipStream_t s, std::initializer_list<std::pair<void*, std::pair<const void*, size_t>>> xs) {
  char* P = pin_buf(w);
  size_t off = 0;
  for (const auto& x : xs) {
    if (P && off + x.second.second <= kPinBytes)
      RK_CHECK(hipMemcpyAsync(P + off, x.second.first, x.second.second, hipMemcpyDeviceToHost, s));
    else
      RK_CHECK(hipMemcpyAsync(x.first, x.second.first, x.second.second, hipMemcpyDeviceToHost, s));
    off += (x.second.second + 7) & ~(size_t)7;
  }
  RK_CHECK(hipStreamSynchronize(s));
  off = 0;
  for (const auto& x : xs) {
    if (P && off + x.second.second <= kPinBytes) memcpy(x.first, P + off, x.second.second);
    off += (x.second.second + 7) & ~(size_t)7;
  }
  return 0;
}

int nl_build_heavy(NLWork& w, int nb, EntryArrays& E, const uint8_t* passive, hipStream_t s) {
  E.nheavy = 0;
  E.nhch = 0;
  E.nheavy_np = 0;
  if (nb <= 0 || !E.soff) return 0;
  if (ensure(w, E.heavy, E.heavy_cap, (size_t)nb) || ensure(w, w.hcount, w.hcount_cap, 2)) return -1;
  // chunk table sized as if every body were heavy: at most (slots of all
  // bodies) / 64 + one per body, so that the heavy count is read once, with
  // the chunks'
  const size_t cap = (size_t)E.cap * 2 / 64 + (size_t)nb + 1;
  if (ensure(w, E.hch, E.hch_cap, cap) || ensure(w, E.hch_off, E.hch_off_cap, (size_t)nb + 1)) return -1;
  if (E.hpart_cap < cap) {
    if (E.hpart) (void)hipFree(E.hpart);
    E.hpart = nullptr;
    E.hpart_cap = 0;
    if (hipMalloc(&E.hpart, cap * 6 * sizeof(double)) != hipSuccess) {
      snprintf(w.err, sizeof(w.err), "out of device memory (heavy-body partial sums)");
      return -1;
    }
    E.hpart_cap = cap;
  }
  RK_CHECK(hipMemsetAsync(w.hcount, 0, 2 * sizeof(unsigned long long), s));
  hipLaunchKernelGGL(k_heavy_list, dim3(nblk(nb)), dim3(kBlock), 0, s, nb, E.soff, w.heavy_min, passive, E.heavy,
                     E.hch_off, E.hch, (int)cap, w.hcount, reinterpret_cast<int32_t*>(w.hcount + 1));
  int32_t cnt[3] = {0, 0, 0};  // chunks, heavy, not passive
  if (read_small(w, s, {{cnt, {w.hcount, 3 * sizeof(int32_t)}}})) return -1;
  if ((size_t)cnt[0] > cap) {
    snprintf(w.err, sizeof(w.err), "heavy-body chunk table overflow");
    return -1;
  }
  E.nhch = cnt[0];
  E.nheavy = cnt[1];
  E.nheavy_np = cnt[2];
  return 0;
}

int nl_rebuild(NLWork& w, Dev& d, const NLParams& p, EntryArrays& cur, EntryArrays& nxt, hipStream_t s) {
  const int nb = d.nb;
  if (nb == 0) return 0;
  const bool cells = p.linkcells != 0;
  if (ensure(w, w.bobb, w.bobb_cap, (size_t)15 * nb)) return -1;
  if (ensure(w, w.baabb, w.baabb_cap, (size_t)6 * nb)) return -1;
  hipLaunchKernelGGL(k_obb, dim3(nblk(nb)), dim3(kBlock), 0, s, d, w.bobb, w.baabb);
  const double half = 0.5 * p.DVerlet;

  // ---- groups of the current list (their count is read with the candidates')
  const int nold = cur.n;
  int ng_old = 0, oend[2] = {0, 0};
  if (ensure(w, w.i32b, w.i32b_cap, (size_t)std::max(nold, 1) + 1) ||
      ensure(w, w.i32c, w.i32c_cap, (size_t)std::max(nold, 1) + 1) ||
      ensure(w, w.okey, w.okey_cap, (size_t)std::max(nold, 1)) ||
      ensure(w, w.ostart, w.ostart_cap, (size_t)std::max(nold, 1) + 1))
    return -1;
  if (nold > 0) {
    hipLaunchKernelGGL(k_old_heads, dim3(nblk(nold)), dim3(kBlock), 0, s, nold, cur.ei, cur.ej, w.i32b);
    if (scan_exclusive(w, w.i32b, w.i32c, nold, s)) return -1;
    hipLaunchKernelGGL(k_old_compact, dim3(nblk(nold)), dim3(kBlock), 0, s, nold, cur.ei, cur.ej, w.i32b, w.i32c,
                       w.okey, w.ostart);
  }
  const int32_t* olast = w.i32c + std::max(nold, 1) - 1;

  // ---- broad phase: candidate pairs
  if (ensure(w, w.counter, w.counter_cap, 4) || ensure(w, w.scnt, w.scnt_cap, (size_t)kStripes * kStripeStride) ||
      ensure(w, w.soff, w.soff_cap, (size_t)kStripes))
    return -1;
  int nc = 0;
  for (int attempt = 0; attempt < 3; attempt++) {
    // striped output: kStripes regions of rcap pairs
    const int rcap = std::max(64, (w.cand_hint + kStripes - 1) / kStripes);
    if (ensure(w, w.cstripe, w.cstripe_cap, (size_t)kStripes * rcap)) return -1;
    RK_CHECK(hipMemsetAsync(w.counter, 0, sizeof(int) * 4, s));
    RK_CHECK(hipMemsetAsync(w.scnt, 0, sizeof(int) * kStripes * kStripeStride, s));
    if (!cells) {
      const int jmax = nb - std::min(nb, std::max(1, d.nDriven));
      const int chunks = std::max(1, (nb + kBruteChunk - 1) / kBruteChunk);
      (void)jmax;
      hipLaunchKernelGGL(k_broad_brute, dim3(nblk(nb), chunks), dim3(kBlock), 0, s, d, w.bobb, half, w.cstripe,
                         w.scnt, rcap);
    } else {
      // bounding box of the bodies [first, nb) (Rockable.cpp:1683-1688, 3943-3947)
      int first = (p.boxForLinkCellsOpt == 1) ? d.nDriven : 0;
      if (first >= nb) first = 0;
      const int pb = 64;
      if (ensure(w, w.f64a, w.f64a_cap, (size_t)6 * pb)) return -1;
      hipLaunchKernelGGL(k_box_partial, dim3(pb), dim3(kBlock), 0, s, first, nb, w.baabb, w.f64a);
      std::vector<double> part(6 * pb);
      if (read_small(w, s, {{part.data(), {w.f64a, sizeof(double) * 6 * pb}}})) return -1;
      double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
      for (int q = 0; q < pb; q++)
        for (int k = 0; k < 3; k++) {
          mn[k] = std::min(mn[k], part[6 * q + k]);
          mx[k] = std::max(mx[k], part[6 * q + 3 + k]);
        }
      Grid g;
      const double ms[3] = {p.cellMinSizes[0], p.cellMinSizes[1], p.cellMinSizes[2]};
      long ncell = 1;
      for (int k = 0; k < 3; k++) {
        const double len = mx[k] - mn[k];
        int n = (ms[k] > 0.0) ? (int)floor(len / ms[k]) : 1;
        g.N[k] = n < 1 ? 1 : n;
        g.mn[k] = mn[k];
        g.sz[k] = len / g.N[k];
        ncell *= g.N[k];
      }
      if (ncell > (1L << 28)) {
        snprintf(w.err, sizeof(w.err), "linkCells: %ld cells (cellMinSizes too small for the domain)", ncell);
        return -1;
      }
      if (ensure(w, w.cell_of, w.cell_of_cap, (size_t)nb) || ensure(w, w.ccount, w.ccount_cap, (size_t)ncell + 1) ||
          ensure(w, w.cstart, w.cstart_cap, (size_t)ncell + 1) || ensure(w, w.cfill, w.cfill_cap, (size_t)ncell) ||
          ensure(w, w.cbody, w.cbody_cap, (size_t)nb) || ensure(w, w.over, w.over_cap, (size_t)nb))
        return -1;
      RK_CHECK(hipMemsetAsync(w.ccount, 0, sizeof(int32_t) * (ncell + 1), s));
      RK_CHECK(hipMemsetAsync(w.cfill, 0, sizeof(int32_t) * ncell, s));
      unsigned long long* reach = reinterpret_cast<unsigned long long*>(w.f64a);
      RK_CHECK(hipMemsetAsync(reach, 0, sizeof(unsigned long long) * 3, s));
      hipLaunchKernelGGL(k_cell_assign, dim3(nblk(nb)), dim3(kBlock), 0, s, d, w.bobb, w.baabb, half, g, w.cell_of,
                         w.ccount, w.over, w.counter + 1, reach);
      if (scan_exclusive(w, w.ccount, w.cstart, (int)ncell + 1, s)) return -1;
      hipLaunchKernelGGL(k_cell_fill, dim3(nblk(nb)), dim3(kBlock), 0, s, nb, w.cell_of, w.cstart, w.cfill, w.cbody);
      int hv[2];
      if (read_small(w, s, {{hv, {w.counter + 1, sizeof(int)}}})) return -1;
      const int nover = hv[0];
      const int ncb = nb - nover;
      hipLaunchKernelGGL(k_broad_cells, dim3(nblk((long)kCellLanes * nb)), dim3(kBlock), 0, s, d, w.bobb, half, g, w.cell_of, w.cstart,
                         w.cbody, w.cstripe, w.scnt, rcap);
      if (nover > 0 && ncb > 0) {
        // enough workgroups to fill the chip when one body (a wall or a plane
        // over the whole domain) meets every cell: each takes every split-th
        // column of cells its box covers
        const int split = std::max(1, std::min(4096, (8192 + nover - 1) / nover));
        hipLaunchKernelGGL(k_broad_over, dim3(nover, split), dim3(kBlock), 0, s, d, w.bobb, half, g, w.over, nover,
                           w.cstart, w.cbody, reach, w.cstripe, w.scnt, rcap);
      }
    }
    hipLaunchKernelGGL(k_stripe_scan, dim3(1), dim3(kStripes), 0, s, w.scnt, w.soff, w.counter + 2);
    int tm[2] = {0, 0};
    if (nold > 0) {
      if (read_small(w, s, {{tm, {w.counter + 2, sizeof(int) * 2}}, {&oend[0], {olast, sizeof(int)}},
                            {&oend[1], {w.i32b + nold - 1, sizeof(int)}}}))
        return -1;
    } else if (read_small(w, s, {{tm, {w.counter + 2, sizeof(int) * 2}}})) {
      return -1;
    }
    nc = tm[0];
    ng_old = oend[0] + oend[1];
    if (tm[1] <= rcap) {
      if (ensure(w, w.cand, w.cand_cap, (size_t)std::max(nc, 1))) return -1;
      hipLaunchKernelGGL(k_stripe_gather, dim3((rcap + kBlock - 1) / kBlock, kStripes), dim3(kBlock), 0, s, w.cstripe,
                         rcap, w.scnt, w.soff, w.cand);
      break;
    }
    w.cand_hint = kStripes * (tm[1] + tm[1] / 4 + 64);
    if (attempt == 2) {
      snprintf(w.err, sizeof(w.err), "broad phase overflow");
      return -1;
    }
  }
  w.last_candidates = nc;

  // ---- narrow phase
  if (ensure(w, w.cbase, w.cbase_cap, (size_t)std::max(nc, 1)) || ensure(w, w.cnf, w.cnf_cap, (size_t)std::max(nc, 1)) ||
      ensure(w, w.cnb, w.cnb_cap, (size_t)std::max(nc, 1)))
    return -1;
  std::function<int(int)> launch_narrow;
  std::function<void(int, int, int)> launch_rest;
  int narrow_rcap = 0, narrow_done = 0;  // pairs the narrow phase's grid has covered
  if (nc > 0) {
    NarrowCfg cfg;
    cfg.maxv = p.maxv;
    cfg.maxe = p.maxe;
    cfg.maxf = p.maxf;
    cfg.maxwords = p.maxwords;
    cfg.dmax = p.dVerlet;
    // the bodies' edge and face boxes for the culls
    if (ensure(w, w.gedge, w.gedge_cap, (size_t)kGate * std::max(d.netot, 1)) ||
        ensure(w, w.gface, w.gface_cap, (size_t)kGate * std::max(d.nftot, 1)))
      return -1;
    int glg = 3;
    while (glg < 6 && (1 << glg) < p.maxe + p.maxf) glg++;
    hipLaunchKernelGGL(k_gate_boxes, dim3((int)((((long)d.nb << glg) + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, d,
                       w.gedge, w.gface, glg);
    cfg.gedge = w.gedge;
    cfg.gface = w.gface;
    // candidate pairs per wavefront: by default 2 for shapes of up to 8
    // vertices, else 1 (measured: 2 pairs are faster for sphero-cubes, 1 for
    // hulls of 8-14 vertices, whose passes fill a wavefront; more pairs cost
    // occupancy, their values being per lane), then as many as the LDS holds
    const size_t stride = (narrow_lds_bytes(p) + 7) & ~(size_t)7;
    int P = w.narrow_pairs;
    if (P <= 0) P = 2 * p.maxv <= 16 ? 2 : 1;
    while (P > 1 && (size_t)P * stride > 65536) P >>= 1;
    const size_t lds = (size_t)P * stride;
    // one run of the narrow phase into stripes of rcap keys; the stripe
    // totals (all, largest) land in counter[2..3]
    // (the stripes' counters use the first word of every 32; the pairs left go to word 1)
    launch_rest = [&, cfg, P, stride, lds](int rcap, int first, int count) {
      const dim3 grid((count + P - 1) / P);
      if (P == 2)
        hipLaunchKernelGGL(k_narrow<2>, grid, dim3(64), lds, s, d, w.bobb, w.baabb, cfg, w.cand, w.nearbuf, w.scnt, rcap,
                           w.cbase, w.cnf, w.cnb, (int)stride, w.plist, w.scnt + 1, first);
      else
        hipLaunchKernelGGL(k_narrow<1>, grid, dim3(64), lds, s, d, w.bobb, w.baabb, cfg, w.cand, w.nearbuf, w.scnt, rcap,
                           w.cbase, w.cnf, w.cnb, (int)stride, w.plist, w.scnt + 1, first);
    };
    launch_narrow = [&, cfg](int rcap) -> int {
      if (ensure(w, w.nearbuf, w.nearbuf_cap, (size_t)kStripes * rcap)) return -1;
      RK_CHECK(hipMemsetAsync(w.scnt, 0, sizeof(int) * kStripes * kStripeStride, s));
      // the pairs of point shapes and those apart one per lane, the others one
      // or two per wavefront; their count is not known yet, so the grid takes
      // the last rebuild's and the rest follows if it was short (below);
      if (ensure(w, w.plist, w.plist_cap, (size_t)nc)) return -1;
      hipLaunchKernelGGL(k_narrow_lanes, dim3(nblk(nc)), dim3(kBlock), 0, s, d, w.bobb, w.baabb, cfg, nc, w.cand,
                         w.nearbuf, w.scnt, rcap, w.cbase, w.cnf, w.cnb, w.plist, w.scnt + 1);
      narrow_done = w.rest_hint >= 0 ? std::min(nc, w.rest_hint + w.rest_hint / 8 + 256) : nc;
      // a first rebuild reads the count where a workgroup for every candidate
      // would cost more (3.3 ns each: 0.85 ms of the 440 000 of 50 005 hulls)
      // than the read (15 us)
      if (w.rest_hint < 0 && nc > 8192) {
        RK_CHECK(hipGetLastError());
        if (read_small(w, s, {{&narrow_done, {w.scnt + 1, sizeof(int)}}})) return -1;
      }
      if (narrow_done > 0) launch_rest(rcap, 0, narrow_done);
      RK_CHECK(hipGetLastError());
      hipLaunchKernelGGL(k_stripe_scan, dim3(1), dim3(kStripes), 0, s, w.scnt, w.soff, w.counter + 2);
      return 0;
    };
    // the stripes' overflow is checked with the merge's totals (one read);
    // on overflow the phase runs again with room, before the merge counts
    narrow_rcap = std::max(64, (w.near_hint + kStripes - 1) / kStripes);
    if (launch_narrow(narrow_rcap)) return -1;
  }

  // ---- directed groups, ordered by (owner, other)
  const int ngk = 2 * nc + ng_old;
  const size_t nz = (size_t)nb + 2;  // zeroed: counts, the count of long segments
  if (ensure(w, w.gstart, w.gstart_cap, (size_t)nb + 1) || ensure(w, w.i32a, w.i32a_cap, nz) ||
      ensure(w, w.big, w.big_cap, (size_t)nb) || ensure(w, w.gseg, w.gseg_cap, 8 * (size_t)std::max(nc, 1)) ||
      ensure(w, w.ukey, w.ukey_cap, (size_t)std::max(ngk, 1)) ||
      ensure(w, w.uref, w.uref_cap, 2 * (size_t)std::max(ngk, 1)) ||
      ensure(w, w.gcount, w.gcount_cap, (size_t)std::max(ngk, 1) + 1) ||
      ensure(w, w.goff, w.goff_cap, (size_t)std::max(ngk, 1) + 1))
    return -1;
  if (ngk > 0) {
    int2* at = reinterpret_cast<int2*>(w.gseg + 6 * (size_t)nc);
    GroupIn G;
    G.nc2 = 2 * nc;
    G.ng_old = ng_old;
    G.nold = nold;
    G.gstart = w.gstart;
    G.gowner = w.gseg;
    G.gother = w.gseg + 2 * (size_t)nc;
    G.gref = w.gseg + 4 * (size_t)nc;
    G.istart = cur.istart;
    G.opos = w.i32c;
    G.okey = w.okey;
    G.ukey = w.ukey;
    G.ucand = w.uref;
    G.uold = w.uref + ngk;
    G.nbig = w.i32a + nb + 1;
    G.big = w.big;
    RK_CHECK(hipMemsetAsync(w.i32a, 0, sizeof(int32_t) * nz, s));
    RK_CHECK(hipMemsetAsync(w.uref, 0xff, sizeof(int32_t) * 2 * (size_t)ngk, s));
    if (nc > 0) hipLaunchKernelGGL(k_group_count, dim3(nblk(nc)), dim3(kBlock), 0, s, nc, w.cand, w.i32a, at);
    if (scan_exclusive(w, w.i32a, w.gstart, nb + 1, s)) return -1;
    if (nc > 0)
      hipLaunchKernelGGL(k_group_fill, dim3(nblk(nc)), dim3(kBlock), 0, s, nc, w.cand, at, w.gstart, w.gseg,
                         w.gseg + 2 * (size_t)nc, w.gseg + 4 * (size_t)nc);
    hipLaunchKernelGGL(k_group_place, dim3(nblk(ngk)), dim3(kBlock), 0, s, G);
    if (2 * nc > kSegMax)
      hipLaunchKernelGGL(k_group_place_big, dim3(kBigGrid, windows(nb)), dim3(kWinThreads), 0, s, G);
    RK_CHECK(hipGetLastError());
  }

  // ---- merge: count, scan, allocate, write
  MergeIn in;
  in.ng = ngk;
  in.ukey = w.ukey;
  in.ucand = w.uref;
  in.uold = w.uref + ngk;
  in.ostart = w.ostart;
  in.cbase = w.cbase;
  in.cnf = w.cnf;
  in.cnb = w.cnb;
  in.nearbuf = w.nearbuf;
  in.bobb = w.bobb;
  in.dmax = p.dVerlet;
  in.oi = cur.ei;
  in.oj = cur.ej;
  in.osub = cur.esub;
  in.oest = cur.est;
  in.oedn = cur.edn;
  in.ogeo = cur.egeo;
  in.odamp = cur.edamp;
  in.ostick = cur.estick;
  in.oeact = cur.eact;
  in.oekey = cur.ekey;
  MergeOut out;
  out.count = w.gcount;
  out.offset = w.goff;
  int nnew = 0;
  if (ngk > 0) {
    // count pass over the groups' slots, its scan, then one read: the merged
    // length and the narrow phase's stripe totals
    auto count_pass = [&]() -> int {
      hipLaunchKernelGGL(k_merge<false>, dim3(nblk((long)ngk + 1)), dim3(kBlock), 0, s, d, in, out);
      if (scan_exclusive(w, w.gcount, w.goff, ngk + 1, s)) return -1;
      return 0;
    };
    if (count_pass()) return -1;
    int rd[2] = {0, 0}, nrest = 0;
    if (launch_narrow) {
      if (read_small(w, s, {{&nnew, {w.goff + ngk, sizeof(int)}},
                            {rd, {w.counter + 2, 2 * sizeof(int)}},
                            {&nrest, {w.scnt + 1, sizeof(int)}}}))
        return -1;
    } else if (read_small(w, s, {{&nnew, {w.goff + ngk, sizeof(int)}}})) {
      return -1;
    }
    bool again = false;
    if (launch_narrow && nrest > narrow_done) {  // more pairs than the grid covered
      launch_rest(narrow_rcap, narrow_done, nrest - narrow_done);
      hipLaunchKernelGGL(k_stripe_scan, dim3(1), dim3(kStripes), 0, s, w.scnt, w.soff, w.counter + 2);
      if (read_small(w, s, {{rd, {w.counter + 2, 2 * sizeof(int)}}})) return -1;
      again = true;
    }
    if (launch_narrow) w.rest_hint = nrest;
    if (launch_narrow && rd[1] > narrow_rcap) {
      for (int attempt = 0;; attempt++) {
        if (attempt == 2) {
          snprintf(w.err, sizeof(w.err), "narrow phase overflow");
          return -1;
        }
        w.near_hint = kStripes * (rd[1] + rd[1] / 4 + 64);
        narrow_rcap = std::max(64, (w.near_hint + kStripes - 1) / kStripes);
        if (launch_narrow(narrow_rcap)) return -1;
        if (read_small(w, s, {{rd, {w.counter + 2, 2 * sizeof(int)}}})) return -1;
        if (rd[1] <= narrow_rcap) break;
      }
      in.nearbuf = w.nearbuf;
      again = true;
    }
    if (again) {
      if (count_pass()) return -1;
      if (read_small(w, s, {{&nnew, {w.goff + ngk, sizeof(int)}}})) return -1;
    }
  }
  if (entries_reserve(w, nxt, nnew) != 0) return -1;
  nxt.n = nnew;
  if (nnew > 0) {
    out.ei = nxt.ei;
    out.ej = nxt.ej;
    out.esub = nxt.esub;
    out.est = nxt.est;
    out.edn = nxt.edn;
    out.egeo = nxt.egeo;
    out.edamp = nxt.edamp;
    out.estick = nxt.estick;
    out.eact = nxt.eact;
    out.ekey = nxt.ekey;
    if (ensure(w, w.msrc, w.msrc_cap, (size_t)nnew)) return -1;
    out.src = w.msrc;
    hipLaunchKernelGGL(k_merge<true>, dim3(nblk(ngk)), dim3(kBlock), 0, s, d, in, out);
    hipLaunchKernelGGL(k_merge_fill, dim3(nblk(nnew)), dim3(kBlock), 0, s, d, nnew, in, out);
  }
  RK_CHECK(hipGetLastError());
  return nl_build_csr(w, nb, nxt, d.passive, s);  // (ends with a read)
}

int entries_reserve(NLWork& w, EntryArrays& E, int n) {
  size_t need = (size_t)(n > 0 ? n : 1);
  if (need <= E.cap && E.ei) return 0;
  entries_free(E);
  size_t c = need + need / 2 + 1024;
  bool ok = hipMalloc(&E.ei, c * sizeof(int32_t)) == hipSuccess && hipMalloc(&E.ej, c * sizeof(int32_t)) == hipSuccess &&
            hipMalloc(&E.esub, c * sizeof(uint32_t)) == hipSuccess && hipMalloc(&E.est, c * sizeof(EState)) == hipSuccess &&
            hipMalloc(&E.edn, c * sizeof(double)) == hipSuccess &&
            hipMalloc(&E.egeo, c * sizeof(EGeom)) == hipSuccess && hipMalloc(&E.edamp, c * sizeof(double)) == hipSuccess &&
            hipMalloc(&E.estick, c * sizeof(int32_t)) == hipSuccess && hipMalloc(&E.eact, c * sizeof(uint8_t)) == hipSuccess &&
            hipMalloc(&E.ekey, c * sizeof(double)) == hipSuccess &&
            hipMalloc(&E.spos, c * 2 * sizeof(int32_t)) == hipSuccess &&
            hipMalloc(&E.sact, c * 2 * sizeof(uint8_t) + 64) == hipSuccess  /* read 16 bytes at a time */ &&
            hipMalloc(&E.sval, c * 12 * sizeof(double)) == hipSuccess &&
            hipMalloc(&E.akin, (c + 512) * sizeof(ActiveKin)) == hipSuccess &&
            hipMalloc(&E.acount, (c / 64 + 2) * sizeof(int32_t)) == hipSuccess;
  if (!ok) {
    snprintf(w.err, sizeof(w.err), "hipMalloc of %zu interaction entries failed", c);
    entries_free(E);
    return -1;
  }
  E.cap = c;
  return 0;
}

void entries_free(EntryArrays& E) {
  void* ps[] = {E.ei, E.ej, E.esub, E.est, E.edn, E.egeo, E.edamp, E.estick, E.eact, E.ekey, E.spos, E.sact, E.sval,
                E.akin, E.acount};
  for (void* q : ps)
    if (q) (void)hipFree(q);
  E.ekey = nullptr;
  E.ei = E.ej = nullptr;
  E.esub = nullptr;
  E.est = nullptr;
  E.edn = nullptr;
  E.egeo = nullptr;
  E.edamp = nullptr;
  E.estick = nullptr;
  E.eact = nullptr;
  E.spos = nullptr;
  E.sact = nullptr;
  E.sval = nullptr;
  E.akin = nullptr;
  E.acount = nullptr;
  E.cap = 0;
}

void nl_work_free(NLWork& w) {
  void* ps[] = {w.plist,
                w.cstripe, w.scnt, w.soff, w.bobb,  w.baabb, w.counter, w.cand,  w.cbase, w.cnf,   w.cnb,   w.nearbuf, w.okey,  w.ostart,
                w.gstart, w.gseg, w.big, w.jsum, w.hcount, w.ukey,  w.uref,  w.gcount,
                w.goff,  w.tmp,   w.i32a,    w.i32b,  w.i32c,  w.f64a,  w.cell_of, w.ccount, w.cstart, w.cfill,
                w.cbody, w.over, w.gedge, w.gface, w.msrc};
  for (void* q : ps)
    if (q) (void)hipFree(q);
  if (w.pin) (void)hipHostFree(w.pin);
  NLWork z;
  w = z;
}

}  // namespace rk
