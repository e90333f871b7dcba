// d2_kernels.hip -- gfx950 kernels of the contact-detection path and the C ABI
// that drives them (include/d2hip.h).
//
// Work is processed breadth-first over all body pairs at once, one tree level
// per step, so every launch sees a flat, load-balanced list regardless of how
// uneven the pairs are:
//
//   CCD level (compareTreesFullContinuous, full_tree_comparison.h:69-219)
//     ccd_cull     soup list: swept-AABB tests of the node pairs' triangle
//                  pairs, the overlapping ones to the item list; connected
//                  (leaf-leaf) list, other blocks: the leaf sub-tests the FP32
//                  culls leave
//     soup_keep    (FP32 form) one thread per item: the sub-tests the FP32
//                  culls leave
//     ccd_sub      one thread per FP64 sub-test, soup and leaf, point-triangle
//                  and edge-edge; a leaf sub-test that hits is a contact
//     soup_reduce  one thread per item: the reference's ordered selection of
//                  the 15 sub-results, hit test, leaf-pair contact emission;
//                  the children of hit node pairs to the next lists
//   Discrete level (compareTreesFull, full_tree_comparison.h:13-67)
//     tri_mask     groups of 64 triangles per wavefront, lane = triangle pair:
//                  FP32 cull, kept pairs to the item list, children of node pairs that hit or may hit to the
//                  next list (dropped there if the parent did not hit)
//     tri_dist     one thread per item: FP64 _comparisonDist, hit -> contact
//                  (leaf-leaf) or the node pair's hit flag
//     disc_expand  (FP64 mode) one thread per node pair: children of hits
//   Post-processing: per-pair ordering of contacts by their breadth-first key,
//   the contact filter (contact.h:44-69, libstdc++ std::sort permutation) and
//   the TOI -> step rule (separate_clusters.cpp:496-564).
//
// Contacts are emitted with a 64-bit key (level, list, child-index path,
// sub-test) whose order is the reference's emission order, so allocation can
// use atomics and the order is restored per pair afterwards.
#include <hip/hip_runtime.h>

#include <hip/hip_ext.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <random>
#include <cstdio>
#include <cstring>
#include <exception>
#include <functional>
#include <initializer_list>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/d2hip.h"
#define D2_HD __host__ __device__ __forceinline__
#include "d2_geom.hpp"
#include "d2_cull.hpp"
#include "d2_sort.hpp"
#include "d2_solver.hpp"

namespace d2 {

// ------------------------------------------------------------------ records
constexpr int NB_STRIDE = 12;  // per-node pruning bounds (d2_trees_upload)
// The FP32 form's copy of the buckets: per triangle (node * 8 + k) 12 floats,
// its corners rounded to float (a.x a.y a.z b.x ... c.z), one unused, and its
// eps's double bits in the last two (low word first); three 16-byte loads.
constexpr int FB_STRIDE = 12;
// and its planes for the CCD point-triangle culls (soup_tri: normal, offset,
// edge normals and offsets, acceptance bound) in 20 floats, five 16-byte loads.
constexpr int ST_STRIDE = 20;
struct NodeRec {
  int32_t id, bucket, inner, depth, parent, child_first, nchild, ntris;
};
struct NP {  // node pair work entry
  uint32_t pair, na, nb, pad;
  unsigned long long key;  // base-8 path of child indices from the root pair
};
struct Item {
  uint32_t np, sub;
};
struct DItem {  // discrete triangle-pair item: node pair, pair, global buckets, sub | inner << 8
  uint32_t np, pair, ga, gb, sub;
};
struct ContactRec {
  unsigned long long key;
  int32_t pair, na, nb, kind, ia, ib, level, pad;
  double r[11];
};
static_assert(sizeof(ContactRec) == 128, "contact record size");

// Pair record (doubles): poses at start/end, the point->triangle frame
// changes, future-state kinematics for the step rule.
enum : int {
  PR_TA0 = 0, PR_TA1 = 16, PR_TB0 = 32, PR_TB1 = 48,
  PR_MAB0 = 64, PR_MAB1 = 80, PR_MBA0 = 96, PR_MBA1 = 112,
  PR_VA = 128, PR_WA = 131, PR_XA = 134, PR_VB = 137, PR_WB = 140, PR_XB = 143,
  PR_GEOA = 146, PR_GEOB = 147, PR_MAXT = 148, PR_SEARCH = 149,
  PR_STRIDE = 152
};
constexpr int PF_STRIDE = 32;  // PF_FLOATS in a cache line of their own
// The CCD culls' pair record: eight 3x4 float matrices -- a's and b's poses at
// both ends with b's start position as origin, and the frame changes -- and the
// search distance.
enum : int {
  CF_A0 = 0, CF_A1 = 12, CF_B0 = 24, CF_B1 = 36, CF_MAB0 = 48, CF_MAB1 = 60, CF_MBA0 = 72, CF_MBA1 = 84,
  CF_SEARCH = 96, CF_STRIDE = 100
};
constexpr int BUCKET = 88;
constexpr int RES_SLOTS = 15;  // sub-results per soup triangle pair
// Global counters (atomics) and per-level sizes.  Level L reads its list sizes
// from lvl[L*LV_STRIDE + ...] and the level's write kernel stores the sizes of
// level L+1; no size ever travels through the host.
enum Counter : int {
  C_CONTACTS = 0, C_OVERFLOW = 1, C_LVL_ITEMS = 2, C_OUT = 3,
  C_GATED_CCD = 4, C_CERT_CCD = 5, C_GATED_DISC = 6, C_CERT_DISC = 7,  // learned gate: proposed / certified pairs
  C_COUNT = 8
};
// LV_PACK (discrete levels): the level's item count (low 32 bits) and its
// children count (high 32 bits), taken together by k_tri_mask's allocation
// atomic and unpacked into LV_ITEMS and the next level's LV_SOUP by k_tri_dist.
// LV_SPT / LV_SEE (CCD levels, FP32 form): the soup sub-tests that survive
// the FP32 culls, point and edge (slot 5 is LV_PACK on discrete levels).
// LV_DEF (discrete levels, FP32 form): the deferred items of inner node pairs
// (k_tri_def), allocated by k_tri_mask (slot 6 is LV_SEE on CCD levels).
enum LevelSlot : int {
  LV_SOUP = 0, LV_CONN = 1, LV_ITEMS = 2, LV_PT = 3, LV_EE = 4, LV_PACK = 5, LV_SPT = 5, LV_SEE = 6, LV_DEF = 6,
  LV_STRIDE = 8
};
constexpr int MAX_LEVELS = 16;  // contact keys hold 16 base-8 path digits
// Key layout: level(5) | list(1) | path(48) | sub(10)
__device__ __forceinline__ unsigned long long make_key(int level, int list, unsigned long long path, int sub) {
  return ((unsigned long long)level << 59) | ((unsigned long long)list << 58) | (path << 10) | (unsigned long long)sub;
}

// std::min / std::max semantics (first argument on ties and NaN).
__device__ __forceinline__ double smin(double a, double b) { return (b < a) ? b : a; }
__device__ __forceinline__ double smax(double a, double b) { return (a < b) ? b : a; }

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }
// Value of lane l (wave-uniform) without going through LDS.
__device__ __forceinline__ double readlane_d(double v, int l) {
  const long long bits = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(bits & 0xffffffffll), l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(bits >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ unsigned long long readlane_u64(unsigned long long v, int l) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(v & 0xffffffffull), l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), l);
  return ((unsigned long long)hi << 32) | lo;
}
// Orders one wavefront's LDS writes before its later LDS reads (the other
// wavefronts of the block are not waited for).
__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ unsigned long long lanes_below() { return (1ull << lane_id()) - 1ull; }
// Inclusive prefix sum over the wavefront.
__device__ __forceinline__ int wave_incl_scan(int v) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d);
    if (lane_id() >= d) v += o;
  }
  return v;
}

// One atomic per wavefront; returns this lane's slot (or -1 when !pred).
__device__ __forceinline__ long long wave_alloc(bool pred, unsigned long long* counter) {
  unsigned long long m = __ballot(pred);
  long long base = 0;
  int leader = m ? __ffsll((long long)m) - 1 : 0;
  if (m && lane_id() == leader) base = (long long)atomicAdd(counter, (unsigned long long)__popcll(m));
  base = __shfl(base, leader);
  return pred ? base + __popcll(m & lanes_below()) : -1;
}

__device__ __forceinline__ void atomic_min_pos(unsigned long long* addr, double v) {
  // Non-negative doubles order like their bit patterns.
  atomicMin(addr, (unsigned long long)__double_as_longlong(v));
}

__device__ __forceinline__ int rl(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// Marks on the lanes of a wavefront divide it into runs: the lane that starts
// lane t's run (marked: lane t starts one; lane 0 always does).
__device__ __forceinline__ int run_start(bool marked) {
  const unsigned long long m = __ballot(marked) | 1ull;
  return 63 - __clzll((long long)(m & (~0ull >> (63 - lane_id()))));
}
// Lanes own runs of consecutive outputs (len of them from position first, in
// lane order, together covering the 64 positions from 0 or their start): the
// lane that owns position lane_id().  own: 64 bytes of LDS of this wavefront.
// All lanes call it.
__device__ __forceinline__ int run_owner(unsigned char* own, int first, int len) {
  own[lane_id()] = 0;
  wave_sync_lds();
  if (len > 0 && first < 64 && first + len > 0) own[first > 0 ? first : 0] = (unsigned char)(lane_id() + 1);
  wave_sync_lds();
  const int owner = (int)own[run_start(own[lane_id()] != 0)] - 1;
  wave_sync_lds();  // read before the next call writes
  return owner;
}
// Position of the r-th set bit of m (r < popcount).
__device__ __forceinline__ int nth_bit(unsigned long long m, int r) {
  unsigned x = (unsigned)m;
  int pos = 0, c = __popc(x);
  if (r >= c) r -= c, x = (unsigned)(m >> 32), pos = 32;
#pragma unroll
  for (int w = 16; w; w >>= 1) {
    c = __popc(x & ((1u << w) - 1u));
    if (r >= c) r -= c, x >>= w, pos += w;
  }
  return pos;
}

// Walks a batch of up to 64 entries, one per lane, each wanting `slots` lanes
// (at most 64; 0: none) and holding `jobs` jobs, in groups of consecutive
// entries of at most 64 slots.  After next(): whether this lane's entry is in
// the group, its first slot and job there, and the group's totals.  All lanes
// call it.
struct Groups {
  int slots, jobs, slot_incl, job_incl, t0 = 0, j0 = 0;
  bool in = false;
  int ts = 0, js = 0, n_slots = 0, n_jobs = 0;
  __device__ __forceinline__ Groups(int slots_, int jobs_) : slots(slots_), jobs(jobs_) {
    slot_incl = wave_incl_scan(slots), job_incl = wave_incl_scan(jobs);
  }
  // fill: a few jobs over a multiple of 64 wait for the next group (an entry
  // has at most 64 jobs)
  __device__ __forceinline__ bool next(bool fill) {
    if (t0 >= rl(slot_incl, 63)) return false;
    ts = slot_incl - slots - t0, js = job_incl - jobs - j0;
    in = slots > 0 && ts >= 0 && ts + slots <= 64;
    int last = 63 - __clzll((long long)__ballot(in));
    if (fill) {
      const int over = rl(job_incl, last) - j0;
      if (over > 64 && (over & 63) < 40) {
        in = in && js + jobs <= (over & ~63);
        last = 63 - __clzll((long long)__ballot(in));
      }
    }
    n_slots = rl(slot_incl, last) - t0, n_jobs = rl(job_incl, last) - j0;
    t0 += n_slots, j0 += n_jobs;
    return true;
  }
  // This lane's entry's share (from bit 0) of 64 answers, the group's jobs
  // from q0 on.
  __device__ __forceinline__ unsigned long long share(unsigned long long answers, int q0) const {
    const int d = js - q0;
    if (!in || d >= 64 || d + jobs <= 0) return 0ull;
    return (d >= 0 ? answers >> d : answers << -d) & (jobs < 64 ? (1ull << jobs) - 1ull : ~0ull);
  }
};
// Tiles of a list of n entries over nblk blocks of nw wavefronts: up to 64
// consecutive entries per wavefront, a block's wavefronts taking consecutive
// ones, a block every nblk-th tile.
struct Tiles {
  long long n, step, b0;
  int part;
  __device__ __forceinline__ Tiles(long long n_, int blk, int nblk, int nw) : n(n_) {
    const long long waves = (long long)nblk * nw;
    part = n < 64 * waves ? (int)((n + waves - 1) / waves) : 64;
    step = waves * part, b0 = (long long)blk * nw * part;
  }
  __device__ __forceinline__ long long first(int wid) const { return b0 + (long long)part * wid; }
};

// arr[key] = min(arr[key], v) for every lane (key -1: none).  Most lanes of a
// wavefront often share one key (a pile is one cluster), and atomics on one
// address take turns (6 ns each here): the lanes of the first keys met are
// reduced to one atomic per key, the others go by themselves, and a value
// that would not lower the entry goes nowhere.  All lanes call it.
template <class V> __device__ __forceinline__ void wave_key_min(int key, V v, V* arr) {
  unsigned long long todo = __ballot(key >= 0);
  for (int round = 0; round < 4 && todo; ++round) {
    const int l = __ffsll((long long)todo) - 1;
    const int k0 = rl(key, l);
    const unsigned long long same = __ballot(key == k0);
    V x = v;
    if (__popcll(same) > 1) {
      if (key != k0) x = (V)(~0ull >> (64 - 8 * sizeof(V) + (V(-1) < V(0) ? 1 : 0)));  // the type's largest value
      for (int off = 32; off > 0; off >>= 1) {
        const V o = __shfl_xor(x, off);
        x = o < x ? o : x;
      }
    }
    if (lane_id() == l && x < __hip_atomic_load(&arr[k0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&arr[k0], x);
    todo &= ~same;
    if (key == k0) key = -1;
  }
  if (key >= 0 && v < __hip_atomic_load(&arr[key], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&arr[key], v);
}

template <class R> __device__ __forceinline__ tri<R> load_tri(const double* bucket, int k) {
  return tri<R>{{(R)bucket[0 * 8 + k], (R)bucket[1 * 8 + k], (R)bucket[2 * 8 + k]},
                {(R)bucket[3 * 8 + k], (R)bucket[4 * 8 + k], (R)bucket[5 * 8 + k]},
                {(R)bucket[6 * 8 + k], (R)bucket[7 * 8 + k], (R)bucket[8 * 8 + k]}};
}
// Corner v (0-2) of triangle k, read from the bucket: with a runtime v this
// is an indexed global load, where selecting from a loaded triangle puts the
// triangle in scratch memory.
__device__ __forceinline__ v3<double> load_corner(const double* bucket, int k, int v) {
  return v3<double>{bucket[(3 * v) * 8 + k], bucket[(3 * v + 1) * 8 + k], bucket[(3 * v + 2) * 8 + k]};
}

struct Dev {
  // trees
  const NodeRec* nodes;
  const double* buckets;
  // pairs
  const int32_t* pair_info;  // a, b, node offset a, node offset b
  const double* pair_rec;
  float* pair_f;               // FP32 form, per pair: the PF_ record (discrete, pair_pose_f32's), the CF_ record (CCD)
  // work lists
  NP* soup;
  NP* conn;
  NP* soup_next;
  NP* conn_next;
  Item* items;
  DItem* ditems;
  DItem* ditems_def;           // FP32 form: deferred items of inner node pairs (k_tri_def)
  Item* pt_items;              // CCD soup sub-tests that survive the FP32 culls, point and edge
  Item* ee_items;
  Item* lpt_items;             // CCD leaf sub-tests, point and edge
  Item* lee_items;
  double* res;  // [items][15][8]
  unsigned* res_mask;  // FP32 form: per soup item, the slots its FP32 culls keep
  int* np_hit;
  int* pair_cnt;               // contacts per pair, counted as they are written
  int* exp_desc;               // per discrete node pair: expansion_desc (FP64 mode)
  const int* np_hit_prev;      // the previous level's hit flags (discrete: parity buffers)
  ContactRec* contacts;
  unsigned long long* cnt;
  unsigned long long* lvl;
  // per pair, min toc of the soup / connected pass (bits) and "a leaf pair
  // had hits in this pass"
  unsigned long long *pass_min_s, *pass_min_c;
  int *pass_flag_s, *pass_flag_c;
  double* min_time;
  const float* tree_eps_out;   // float-barycentric acceptance bound per tree
  const float* fbuckets;       // FP32 form: per triangle its corners rounded to float and its eps (FB_STRIDE)
  const float* stris;          // FP32 form: per triangle its soup_tri planes (ST_STRIDE)
  const float* nbound;         // per node: leaf box, slack, sphere (nodes_apart, spheres_apart)
  const uint8_t* kid_inner;    // per node: bit c set when child c is an inner node
  int prune;                   // skip node pairs nodes_apart proves contact-free
  int defer;                   // FP32 form: inner node pairs send one item to k_tri_dist, the rest to k_tri_def
  int box_test;                // FP32 form: k_tri_mask tests arriving node pairs with boxes_apart_faces_rel
  int conn_blocks;             // CCD: the last blocks of k_ccd_cull, which take the connected list
  const int32_t* body_tree;
  int fp32;                    // FP32 culls of the CCD leaf sub-tests
  int n_pairs;
  long long cap_np, cap_items, cap_res, cap_contacts;  // cap_res: CCD soup items (result slots)
  int level;
  int discrete;
  __device__ long long lv(int level_, int slot) const { return (long long)lvl[level_ * LV_STRIDE + slot]; }
  __device__ long long n_soup() const { long long n = lv(level, LV_SOUP); return n < cap_np ? n : cap_np; }
  __device__ long long n_conn() const { long long n = lv(level, LV_CONN); return n < cap_np ? n : cap_np; }
  __device__ long long n_lv(int slot) const { long long n = lv(level, slot); return n < cap_items ? n : cap_items; }
  __device__ long long n_res() const { long long n = lv(level, LV_ITEMS); return n < cap_res ? n : cap_res; }
};

// ------------------------------------------------- block-level primitives
// Chunked kernels split a list of n entries into gridDim.x contiguous ranges,
// one per block; a producer stores each block's total in part[block], and its
// consumer (launched with the same grid) takes its offset as the sum of the
// partials before it.  This replaces a separate scan and keeps the lists in
// order.
__device__ __forceinline__ void chunk_of(long long n, long long& b, long long& e) {
  const long long ch = (n + gridDim.x - 1) / gridDim.x;
  b = (long long)blockIdx.x * ch;
  e = b + ch;
  if (b > n) b = n;
  if (e > n) e = n;
}
__device__ long long block_sum(long long v) {
  __shared__ long long red[16];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  long long s = 0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += red[i];
  return s;
}
// Exclusive scan over the block; total = sum over the block.
__device__ int block_scan(int v, int& total) {
  __shared__ int ws[16];
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  int x = v;
  for (int o = 1; o < 64; o <<= 1) {
    int y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  __syncthreads();
  if (lane == 63) ws[wid] = x;
  __syncthreads();
  int before = 0, tot = 0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) {
    if (i < wid) before += ws[i];
    tot += ws[i];
  }
  total = tot;
  return before + x - v;
}
__device__ void partial_prefix(const int* part, long long& before, long long& total) {
  long long b = 0, t = 0;
  for (int i = threadIdx.x; i < (int)gridDim.x; i += blockDim.x) {
    long long v = part[i];
    t += v;
    if (i < (int)blockIdx.x) b += v;
  }
  before = block_sum(b);
  total = block_sum(t);
}

// ----------------------------------------------------------------- set-up
// Cluster-step accumulators (separate_clusters.cpp:541-598): per cluster the
// smallest step (as bits) and its first pair / first pair with a non-static
// body; with body_step, every body's step starts as its clamped last step (a
// body in no pair is a cluster of its own without interactions,
// separate_clusters.cpp:594-596, time_step_selection_dynamic_continuous.cpp:19).
struct ClusterAcc {
  int n_clusters, n_bodies;
  float dt;
  unsigned long long* step_bits;  // null: nothing to do
  int *first_any, *first_ns;
  int* read_later;  // per body: its step is read or changed after its cluster's first pair
  const double* bodies;
  double* body_step;
  const int32_t *pairs, *cluster_of_pair;
};
__device__ __forceinline__ void cluster_init_range(const ClusterAcc& A, long long t0, long long stride) {
  const int n = A.n_bodies > A.n_clusters ? A.n_bodies : A.n_clusters;
  for (long long k = t0; k < n; k += stride) {
    if (k < A.n_clusters) A.step_bits[k] = ~0ull, A.first_any[k] = 0x7fffffff, A.first_ns[k] = 0x7fffffff;
    if (k < A.n_bodies) A.read_later[k] = 0;
    if (A.body_step && k < A.n_bodies) {
      double s = A.bodies[40 * (size_t)k + 39];
      const double hi = (double)A.dt;
      s = (hi < s) ? hi : s;
      A.body_step[k] = (s < 1e-3) ? 1e-3 : s;
    }
  }
}
__device__ __forceinline__ void cluster_first_range(const ClusterAcc& A, int n_pairs, long long t0, long long stride) {
  for (long long p0 = t0 - lane_id(); p0 < n_pairs; p0 += stride) {  // wavefront-uniform
    const long long p = p0 + lane_id();
    int k = -1;
    bool ns = false;
    if (p < n_pairs) {
      k = A.cluster_of_pair[p];
      ns = !(A.bodies[40 * (size_t)A.pairs[2 * p] + 38] != 0.0 && A.bodies[40 * (size_t)A.pairs[2 * p + 1] + 38] != 0.0);
    }
    wave_key_min(k, (int)p, A.first_any);
    wave_key_min(ns ? k : -1, (int)p, A.first_ns);
  }
}

// Per pair: poses, frame changes, kinematics (CCD: future = extrapolate(max_time)).
// Four lanes per pair split the record: lane q computes the poses and the
// frame change it writes (q = 0: TA0, inv(TB0) TA0; 1: TA1, inv(TB1) TA1 and
// a's kinematics; 2: TB0, inv(TA0) TB0; 3: TB1, inv(TA1) TB1 and b's
// kinematics), so the longest chain holds two extrapolations, one inverse
// and one product instead of all of them.
// The same kernel starts the phase: per pair the root node pair, the pass
// accumulators, min_time and scale (a step's discrete phase keeps its CCD
// phase's), the post-processing counters; block 0 clears the counters (a
// step's discrete phase keeps the CCD phase's overflow flag and gate counts)
// and sets the level table to one level of n_pairs roots (none when the
// learned gate's certificate appends the phase's roots).
__global__ void __launch_bounds__(256) k_setup(Dev D, const int32_t* pairs, const double* max_time, const double* bodies,
                        const int32_t* body_tree, const int32_t* tree_off, int32_t* pair_info, double* pair_rec,
                        int ccd, int mt_from_bodies, int keep_ccd, double* scale, int* pair_fill, int* kept_cnt,
                        int* n_big, ClusterAcc CA, int gated) {
  const int n_pairs = D.n_pairs;
  if (CA.step_bits)  // a step: its cluster accumulators
    cluster_init_range(CA, (long long)blockIdx.x * blockDim.x + threadIdx.x, (long long)gridDim.x * blockDim.x);
  if (blockIdx.x == 0) {
    for (int i = threadIdx.x; i < C_COUNT; i += blockDim.x)
      if (!(keep_ccd && (i == C_OVERFLOW || i == C_GATED_CCD || i == C_CERT_CCD))) D.cnt[i] = 0;
    for (int i = threadIdx.x; i < (MAX_LEVELS + 1) * LV_STRIDE; i += blockDim.x)  // gated: roots come from k_certify
      D.lvl[i] = i == LV_SOUP && !gated ? (unsigned long long)n_pairs : 0ull;
    if (threadIdx.x == 0) D.pair_cnt[n_pairs] = 0, kept_cnt[n_pairs] = 0, n_big[0] = 0, n_big[1] = 0;
  }
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < 4ll * n_pairs;
       t += (long long)gridDim.x * blockDim.x) {
    const int p = (int)(t >> 2), q = (int)(t & 3);
    int a = pairs[2 * p], b = pairs[2 * p + 1];
    const double* ra = bodies + 40 * (size_t)a;
    const double* rb = bodies + 40 * (size_t)b;
    // max_time: given per pair, or min(last steps of a, b) (separate_clusters.cpp:490)
    const double mt = !ccd ? 0.0 : mt_from_bodies ? ((rb[39] < ra[39]) ? rb[39] : ra[39]) : max_time[p];
    const bool end = q & 1;  // lanes 1, 3 work on the end poses
    const bool of_a = q < 2;  // lanes 0, 1 own a's pose, lanes 2, 3 b's
    // the own body's record and the other's (selecting pointers, not private
    // arrays, keeps the poses in registers)
    const double* ro = of_a ? ra : rb;
    const double* rx = of_a ? rb : ra;
    body_state so, sx;
    if (!end) {
      so = load_state(ro), sx = load_state(rx);
    } else if (ccd) {
      so = extrapolate(load_state(ro), mt, ro + 28);
      sx = extrapolate(load_state(rx), mt, rx + 28);
    } else {
      so = load_state(ro + 14), sx = load_state(rx + 14);
    }
    double* pr = pair_rec + (size_t)PR_STRIDE * p;
    double To[16];
    pose(so.q, so.t, To);
    double* dst = pr + (of_a ? (end ? PR_TA1 : PR_TA0) : (end ? PR_TB1 : PR_TB0));
#pragma unroll
    for (int k = 0; k < 16; ++k) dst[k] = To[k];
    if (ccd) {
      double Tx[16], inv[16];
      pose(sx.q, sx.t, Tx);
      inv44(Tx, inv);
      mul44(inv, To, pr + (of_a ? (end ? PR_MAB1 : PR_MAB0) : (end ? PR_MBA1 : PR_MBA0)));
      if (end) {
        double Iw[9];
        world_inv_inertia(so.q, ro + 28, Iw);
        const v3<double> w = mul33v(Iw, so.L);
        double* k = pr + (of_a ? PR_VA : PR_VB);
        k[0] = so.v.x, k[1] = so.v.y, k[2] = so.v.z;
        k[3] = w.x, k[4] = w.y, k[5] = w.z;  // PR_WA / PR_WB
        k[6] = so.t.x, k[7] = so.t.y, k[8] = so.t.z;  // PR_XA / PR_XB
      }
    }
    if (D.pair_f && ccd) {  // the culls' record, each lane the two matrices it computed
      float* f = D.pair_f + (size_t)CF_STRIDE * p;
      const double org[3] = {rb[4], rb[5], rb[6]};  // b's start position
      const double* M = pr + (of_a ? (end ? PR_MAB1 : PR_MAB0) : (end ? PR_MBA1 : PR_MBA0));
      float* fw = f + (of_a ? (end ? CF_A1 : CF_A0) : (end ? CF_B1 : CF_B0));
      float* fm = f + (of_a ? (end ? CF_MAB1 : CF_MAB0) : (end ? CF_MBA1 : CF_MBA0));
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          fw[4 * r + k] = (float)(k < 3 ? To[4 * r + k] : To[4 * r + 3] - org[r]), fm[4 * r + k] = (float)M[4 * r + k];
      if (q == 0) f[CF_SEARCH] = (float)(ra[37] + rb[37]);
    } else if (D.pair_f && end) {  // pair_pose_f32, each lane the half it has the pose of
      float* f = D.pair_f + (size_t)PF_STRIDE * p;
      const double t[3] = {so.t.x - sx.t.x, so.t.y - sx.t.y, so.t.z - sx.t.z};
#pragma unroll
      for (int r = 0; r < 3; ++r) {
#pragma unroll
        for (int k = 0; k < 3; ++k) f[(of_a ? PF_RA : PF_RB) + 3 * r + k] = (float)To[4 * r + k];
        if (of_a) f[PF_TR + r] = (float)t[r];
      }
      if (!of_a) f[PF_SEARCH] = (float)(ra[37] + rb[37]);
    }
    if (q == 0) {
      pr[PR_GEOA] = ra[37];
      pr[PR_GEOB] = rb[37];
      pr[PR_MAXT] = mt;
      pr[PR_SEARCH] = (double)(float)(ra[37] + rb[37]);  // a float in the reference
      pair_info[4 * p + 0] = a;
      pair_info[4 * p + 1] = b;
      pair_info[4 * p + 2] = tree_off[body_tree[a]];
      pair_info[4 * p + 3] = tree_off[body_tree[b]];
      D.soup[p] = NP{(uint32_t)p, 0u, 0u, 0u, 0ull};
      D.pass_min_s[p] = ~0ull, D.pass_min_c[p] = ~0ull;
      D.pass_flag_s[p] = 0, D.pass_flag_c[p] = 0;
      if (!keep_ccd) D.min_time[p] = mt, scale[p] = 1.0;
      D.pair_cnt[p] = 0, kept_cnt[p] = 0, pair_fill[p] = 0;
    }
  }
}


// Folds one pass: "min toc of every hit of this pass" enters min_time when a
// leaf-leaf node pair of the pair had hits (full_tree_comparison.h:106-108,167-169).
__device__ __forceinline__ void fold_pass(const Dev& D, const double* pair_rec, unsigned long long* pass_min,
                                          int* pass_flag) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < D.n_pairs; p += gridDim.x * blockDim.x) {
    if (pass_flag[p] && pass_min[p] != ~0ull) {
      double t = __longlong_as_double((long long)pass_min[p]) * pair_rec[(size_t)PR_STRIDE * p + PR_MAXT];
      if (t < D.min_time[p]) D.min_time[p] = t;
    }
    pass_min[p] = ~0ull;
    pass_flag[p] = 0;
  }
}
// Keeps the CCD phase's sizes (and its contact count in the reserved field of
// level 0) next to the discrete phase's, for sizing the capacities.
__device__ __forceinline__ void save_ccd_sizes(Dev& D) {
  const int n = (MAX_LEVELS + 1) * LV_STRIDE;
  for (int i = threadIdx.x; i < n; i += blockDim.x)
    D.lvl[n + i] = i == LV_STRIDE - 1 ? D.cnt[C_CONTACTS] : D.lvl[i];
}
// Closing fold of the CCD phase; block 0 also keeps the phase's level sizes
// and contact count in the second half of the level table.
// In a step it also records each cluster's first pairs (accumulators
// initialised by k_setup).
__global__ void k_fold_final(Dev D, ClusterAcc CA) {
  fold_pass(D, D.pair_rec, D.pass_min_s, D.pass_flag_s);
  fold_pass(D, D.pair_rec, D.pass_min_c, D.pass_flag_c);
  if (blockIdx.x == 0) save_ccd_sizes(D);
  if (CA.step_bits)
    cluster_first_range(CA, D.n_pairs, (long long)blockIdx.x * blockDim.x + threadIdx.x,
                        (long long)gridDim.x * blockDim.x);
}

// --------------------------------------------------------- CCD soup level
// Swept box of a triangle: bbox at the start pose expanded by bbox at the end
// pose, then by geo_eps (continuous_comparison.h:804-812); lo xyz, hi xyz.
__device__ __forceinline__ void swept_box(const tri<double>& t, const double* m0, const double* m1, double g,
                                          double* o) {
  const tri<double> u = xform(m0, t), v = xform(m1, t);
  const double ux[3] = {u.a.x, u.b.x, u.c.x}, uy[3] = {u.a.y, u.b.y, u.c.y}, uz[3] = {u.a.z, u.b.z, u.c.z};
  const double vx[3] = {v.a.x, v.b.x, v.c.x}, vy[3] = {v.a.y, v.b.y, v.c.y}, vz[3] = {v.a.z, v.b.z, v.c.z};
  const double* U[3] = {ux, uy, uz};
  const double* V[3] = {vx, vy, vz};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double lo = smin(smin(U[k][0], U[k][1]), U[k][2]), hi = smax(smax(U[k][0], U[k][1]), U[k][2]);
    const double lo2 = smin(smin(V[k][0], V[k][1]), V[k][2]), hi2 = smax(smax(V[k][0], V[k][1]), V[k][2]);
    o[k] = smin(lo, lo2) - g, o[3 + k] = smax(hi, hi2) + g;
  }
}
__device__ __forceinline__ void store_res(double* r, double d, v3<double> P, v3<double> Q, double toc) {
  r[0] = d, r[1] = toc, r[2] = P.x, r[3] = P.y, r[4] = P.z, r[5] = Q.x, r[6] = Q.y, r[7] = Q.z;
}

// The FP32 form's float copy of the buckets (FB_STRIDE floats per triangle)
// and every triangle's soup_tri planes (ST_STRIDE).
__global__ void __launch_bounds__(256) k_bucket_f32(const double* buckets, long long n_nodes, float* fb, float* st) {
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < 8 * n_nodes;
       t += (long long)gridDim.x * blockDim.x) {
    const long long node = t >> 3;
    const int k = (int)(t & 7);
    const double* bk = buckets + (size_t)BUCKET * node;
    const tri<double> T = load_tri<double>(bk, k);
    const double eps = bk[72 + k];
    float4* o = reinterpret_cast<float4*>(fb + (size_t)FB_STRIDE * t);
    o[0] = make_float4((float)T.a.x, (float)T.a.y, (float)T.a.z, (float)T.b.x);
    o[1] = make_float4((float)T.b.y, (float)T.b.z, (float)T.c.x, (float)T.c.y);
    o[2] = make_float4((float)T.c.z, 0.f, __int_as_float(__double2loint(eps)), __int_as_float(__double2hiint(eps)));
    const SoupTri S = soup_tri(T);
    float4* q = reinterpret_cast<float4*>(st + (size_t)ST_STRIDE * t);
    q[0] = make_float4(S.n[0], S.n[1], S.n[2], S.d);
    q[1] = make_float4(S.m[0], S.m[1], S.m[2], S.m[3]);
    q[2] = make_float4(S.m[4], S.m[5], S.m[6], S.m[7]);
    q[3] = make_float4(S.m[8], S.o[0], S.o[1], S.o[2]);
    q[4] = make_float4(S.eo, 0.f, 0.f, 0.f);
  }
}
// A triangle's float corners and its soup_tri planes from the FP32 copies
// (global triangle index = node * 8 + k).
__device__ __forceinline__ void load_corners_f(const float* fb, size_t t, float* c9) {
  const float4* f = reinterpret_cast<const float4*>(fb + (size_t)FB_STRIDE * t);
  const float4 q0 = f[0], q1 = f[1], q2 = f[2];
  c9[0] = q0.x, c9[1] = q0.y, c9[2] = q0.z, c9[3] = q0.w, c9[4] = q1.x, c9[5] = q1.y, c9[6] = q1.z, c9[7] = q1.w;
  c9[8] = q2.x;
}
__device__ __forceinline__ SoupTri load_soup_tri(const float* st, size_t t) {
  const float4* f = reinterpret_cast<const float4*>(st + (size_t)ST_STRIDE * t);
  const float4 q0 = f[0], q1 = f[1], q2 = f[2], q3 = f[3], q4 = f[4];
  SoupTri S;
  S.n[0] = q0.x, S.n[1] = q0.y, S.n[2] = q0.z, S.d = q0.w;
  S.m[0] = q1.x, S.m[1] = q1.y, S.m[2] = q1.z, S.m[3] = q1.w, S.m[4] = q2.x, S.m[5] = q2.y, S.m[6] = q2.z;
  S.m[7] = q2.w, S.m[8] = q3.x, S.o[0] = q3.y, S.o[1] = q3.z, S.o[2] = q3.w, S.eo = q4.x;
  return S;
}
// What a wavefront of k_ccd_cull keeps in LDS: the soup list's part, the
// group's swept boxes and triangle pairs (slot of a's, slot of b's << 6); the
// connected list's, the group's vertices at both ends (world, then the other
// body's frame), its triangles' planes, per node pair the largest magnitude
// (bits), and the surviving sub-tests on their way out.
constexpr int LEAF_PT_BUF = 128, LEAF_EE_BUF = 256;
union CullShare {
  struct {
    double box[64][6];
    unsigned short job[256];
  } s;
  struct {
    float v[64][12];
    float t[21][20];
    unsigned mag[64];
    Item pt[LEAF_PT_BUF], ee[LEAF_EE_BUF];
  } c;
};
// Soup list: per node pair the triangle pairs whose swept AABBs overlap, in
// groups of at most 64 triangles: a lane builds one swept box, then the
// triangle pairs compare boxes one per lane.  The overlapping ones go to the
// level's item list, one slot range per block and round; the list's order is
// free (contacts carry their emission keys).
__device__ __forceinline__ void soup_cull_part(Dev& D, int nblk, CullShare& S, unsigned char* own) {
  __shared__ int s_tot[2][4];
  __shared__ unsigned long long s_base[2];
  const int lane = lane_id(), wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const long long n = D.n_soup();
  int it = 0;
  for (Tiles T(n, blockIdx.x, nblk, 4); T.b0 < n; T.b0 += T.step, ++it) {
    const long long w0 = T.first(wid), wl = w0 + lane;
    const bool in_range = lane < T.part && wl < n;
    int l_pair = 0, l_ga = 0, l_gb = 0, l_nta = 0, l_ntb = 0;
    if (in_range) {
      const NP np = D.soup[wl];
      const int32_t* pi = D.pair_info + 4 * np.pair;
      const NodeRec na = D.nodes[pi[2] + np.na];
      const NodeRec nb = D.nodes[pi[3] + np.nb];
      l_pair = (int)np.pair, l_ga = pi[2] + na.bucket, l_gb = pi[3] + nb.bucket, l_nta = na.ntris, l_ntb = nb.ntris;
      D.np_hit[wl] = 0;
    }
    unsigned long long my_keep = 0;  // bit i * l_ntb + j
    const int my_jobs = l_nta * l_ntb;
    for (Groups g(my_jobs > 0 ? l_nta + l_ntb : 0, my_jobs); g.next(true);) {
      const int src = run_owner(own, g.ts, g.in ? g.slots : 0);
      const int start = __shfl(g.ts, src), jstart = __shfl(g.js, src);
      const int pair = __shfl(l_pair, src), nta = __shfl(l_nta, src), ntb = __shfl(l_ntb, src);
      const int ga = __shfl(l_ga, src), gb = __shfl(l_gb, src);
      if (lane < g.n_slots) {
        const int x = lane - start;
        const bool side = x >= nta;
        const int k = side ? x - nta : x;
        const double* pr = D.pair_rec + (size_t)PR_STRIDE * pair;
        const double* bk = D.buckets + (size_t)BUCKET * (side ? gb : ga);
        swept_box(load_tri<double>(bk, k), side ? pr + PR_TB0 : pr + PR_TA0, side ? pr + PR_TB1 : pr + PR_TA1,
                  side ? pr[PR_GEOB] : pr[PR_GEOA], S.s.box[lane]);
        if (!side)
          for (int j = 0; j < ntb; ++j)
            S.s.job[jstart + k * ntb + j] = (unsigned short)(lane | ((start + nta + j) << 6));
      }
      wave_sync_lds();
      for (int q0 = 0; q0 < g.n_jobs; q0 += 64) {
        bool hit = false;
        if (q0 + lane < g.n_jobs) {
          const int job = S.s.job[q0 + lane];
          const double* A = S.s.box[job & 63];
          const double* B = S.s.box[job >> 6];
          hit = true;
          for (int k = 0; k < 3; ++k) {  // bbox.h:8-23, a is "this"
            const bool o = (B[k] < A[k]) ? (B[3 + k] > A[k]) : (B[k] < A[3 + k]);
            hit = hit && o;
          }
        }
        my_keep |= g.share(__ballot(hit), q0);
      }
      wave_sync_lds();  // read before the next group overwrites
    }
    const int kept = __popcll(my_keep), incl = wave_incl_scan(kept), all = rl(incl, 63), par = it & 1;
    if (lane == 0) s_tot[par][wid] = all;
    __syncthreads();
    if (threadIdx.x == 0) {
      const int tot = s_tot[par][0] + s_tot[par][1] + s_tot[par][2] + s_tot[par][3];
      unsigned long long base = 0;
      if (tot) {
        base = atomicAdd(&D.lvl[D.level * LV_STRIDE + LV_ITEMS], (unsigned long long)tot);
        atomicAdd(&D.cnt[C_LVL_ITEMS], (unsigned long long)tot);
        if ((long long)(base + tot) > D.cap_res) atomicOr(&D.cnt[C_OVERFLOW], 1ull);
      }
      s_base[par] = base;
    }
    __syncthreads();
    long long base = (long long)s_base[par];
    for (int v = 0; v < wid; ++v) base += s_tot[par][v];
    for (int q0 = 0; q0 < all; q0 += 64) {
      const int src = run_owner(own, incl - kept - q0, kept);
      const int r = q0 + lane - __shfl(incl - kept, src), ntb = __shfl(l_ntb, src);
      const unsigned long long m = ((unsigned long long)(unsigned)__shfl((int)(my_keep >> 32), src) << 32) |
                                   (unsigned)__shfl((int)(unsigned)my_keep, src);
      if (q0 + lane < all && base + q0 + lane < D.cap_res) {
        const int b = nth_bit(m, r), i = b / ntb;
        D.items[base + q0 + lane] = Item{(uint32_t)(w0 + src), (uint32_t)(i << 3 | (b - i * ntb))};
      }
    }
  }
}

// ------------------------------------------- FP32 culls of CCD leaf sub-tests
// The bounds of d2_cull.hpp (soup_point_keep: plane side and edge
// half-planes with each triangle's FP64-derived normals and its
// float-barycentric acceptance bound; cull_edge_edge: separating axes).
//
// Connected list: the leaf sub-tests of every node pair (6nm point, 9nm edge;
// the FP64 form keeps all) that the culls leave, to the level's two lists, in
// groups of node pairs with at most 64 vertices: a lane transforms one vertex
// (both ends, in world coordinates relative to b's start position and in the
// other body's frame), another reads a triangle's planes, then the sub-tests
// go one per lane, 64 at a time.  A leaf pair has about 13 vertices, 27 point
// and 40 edge sub-tests: with a pass per node pair, most of its time was the
// latency of the loads and 27 to 60 shuffles per sub-test (a pile's 2.7 M soup
// and 2.6 M connected node pairs: 3.1 + 5.7 + 2.1 ms for the soup list, these
// culls and their lists, 3.7 ms for all in this launch).
// Survivors wait in LDS and leave together (an atomic on one address takes 6
// ns of its turn).
__device__ __forceinline__ M34f load_m34f(const float* p) {
  const float4* q = reinterpret_cast<const float4*>(p);
  const float4 a = q[0], b = q[1], c = q[2];
  return M34f{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w}};
}
// Up to 64 sub-tests more to a wavefront's buffer of cap, which goes to the
// list when another 64 might not fit.  All lanes call it.
__device__ __forceinline__ void leaf_push(const Dev& D, bool keep, Item item, Item* buf, int cap, int& held, int slot_id,
                                          Item* list) {
  const unsigned long long m = __ballot(keep);
  if (keep) buf[held + __popcll(m & lanes_below())] = item;
  held += __popcll(m);
  if (held <= cap - 64) return;
  wave_sync_lds();
  unsigned long long base = 0;
  if (lane_id() == 0) {
    base = atomicAdd(&D.lvl[D.level * LV_STRIDE + slot_id], (unsigned long long)held);
    if ((long long)(base + held) > D.cap_items) atomicOr(&D.cnt[C_OVERFLOW], 1ull);
  }
  base = readlane_u64(base, 0);
  for (int i = lane_id(); i < held; i += 64)
    if ((long long)base + i < D.cap_items) list[base + i] = buf[i];
  held = 0;
  wave_sync_lds();
}
__device__ __forceinline__ void leaf_cull_part(Dev& D, CullShare& S, unsigned char* own) {
  __shared__ int s_held[2][4];
  __shared__ unsigned long long s_out[2];
  const int lane = lane_id(), wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const long long n = D.n_conn();
  int held_pt = 0, held_ee = 0;
  for (Tiles T(n, (int)blockIdx.x - ((int)gridDim.x - D.conn_blocks), D.conn_blocks, 4); T.b0 < n; T.b0 += T.step) {
    const long long w0 = T.first(wid), wl = w0 + lane;
    int l_pair = 0, l_ta = 0, l_tb = 0, l_n = 0, l_m = 0;  // l_ta, l_tb: global triangle 0 of the two leaves
    float l_thr = 0.f;
    if (lane < T.part && wl < n) {
      const NP np = D.conn[wl];
      const int32_t* pi = D.pair_info + 4 * np.pair;
      const NodeRec na = D.nodes[pi[2] + np.na];
      const NodeRec nb = D.nodes[pi[3] + np.nb];
      l_pair = (int)np.pair, l_ta = 8 * (pi[2] + na.bucket), l_tb = 8 * (pi[3] + nb.bucket), l_n = na.ntris, l_m = nb.ntris;
      if (D.fp32) l_thr = D.pair_f[(size_t)CF_STRIDE * np.pair + CF_SEARCH];
    }
    const int nm = l_n * l_m;
    // s / n and s / m of sub-test numbers below 576 by multiplication: exact,
    // the error s (65536 / d rounded up - 65536 / d) stays below 576 * 8 / 65536
    const int inv_n = nm ? (65536 + l_n - 1) / l_n : 0, inv_m = nm ? (65536 + l_m - 1) / l_m : 0;
    if (!D.fp32) {  // every sub-test: the batch's places are known at once, one atomic per list
      const int incl = wave_incl_scan(nm), first = incl - nm, all = rl(incl, 63);
      unsigned long long base = 0;
      if (all && lane < 2) {
        base = atomicAdd(&D.lvl[D.level * LV_STRIDE + (lane ? LV_EE : LV_PT)], (unsigned long long)((lane ? 9 : 6) * all));
        if ((long long)(base + (lane ? 9 : 6) * all) > D.cap_items) atomicOr(&D.cnt[C_OVERFLOW], 1ull);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int k = e ? 9 : 6;
        const long long b = (long long)readlane_u64(base, e);
        for (int q0 = 0; q0 < k * all; q0 += 64) {
          const int src = run_owner(own, k * first - q0, k * nm);
          const int sub = q0 + lane - k * __shfl(first, src);
          if (q0 + lane < k * all && b + q0 + lane < D.cap_items)
            (e ? D.lee_items : D.lpt_items)[b + q0 + lane] = Item{(uint32_t)(w0 + src), (uint32_t)sub};
        }
      }
      continue;
    }
    for (Groups g(nm > 0 ? 3 * (l_n + l_m) : 0, nm); g.next(false);) {
      {
        const int src = run_owner(own, g.ts, g.in ? g.slots : 0);
        const int x = lane - __shfl(g.ts, src);
        const int na = __shfl(l_n, src), ta = __shfl(l_ta, src), tb = __shfl(l_tb, src), pair = __shfl(l_pair, src);
        S.c.mag[lane] = 0u;
        wave_sync_lds();
        const bool of_b = x >= 3 * na;
        const int v = of_b ? x - 3 * na : x, tri = v / 3;
        const size_t tk = (size_t)(of_b ? tb : ta) + tri;
        if (lane < g.n_slots) {
          const float* pf = D.fbuckets + (size_t)FB_STRIDE * tk + 3 * (v - 3 * tri);
          const float p[3] = {pf[0], pf[1], pf[2]};  // the corner rounded to float
          const float* cf = D.pair_f + (size_t)CF_STRIDE * pair;
          const M34f W0 = load_m34f(cf + (of_b ? CF_B0 : CF_A0)), W1 = load_m34f(cf + (of_b ? CF_B1 : CF_A1));
          const M34f F0 = load_m34f(cf + (of_b ? CF_MBA0 : CF_MAB0)), F1 = load_m34f(cf + (of_b ? CF_MBA1 : CF_MAB1));
          float o[12];
          xf_f(W0, p, o), xf_f(W1, p, o + 3), xf_f(F0, p, o + 6), xf_f(F1, p, o + 9);
          float mag = fmaxf(fmaxf(amax3(o), amax3(o + 3)), fmaxf(amax3(o + 6), amax3(o + 9)));
          mag = fmaxf(mag, fmaxf(fmaxf(fmaxf(m34_mag(W0), m34_mag(W1)), fmaxf(m34_mag(F0), m34_mag(F1))), amax3(p)));
#pragma unroll
          for (int q = 0; q < 12; ++q) S.c.v[lane][q] = o[q];
          atomicMax(&S.c.mag[src], __float_as_uint(mag));
        }
        // the triangle of vertex slots 3 t .. 3 t + 2, by lane t
        const int tt = __shfl((int)tk, lane < 21 ? 3 * lane : 63);
        if (3 * lane < g.n_slots) {
          const SoupTri t = load_soup_tri(D.stris, (size_t)tt);
          float* o = S.c.t[lane];
#pragma unroll
          for (int q = 0; q < 3; ++q) o[q] = t.n[q], o[13 + q] = t.o[q];
          o[3] = t.d, o[16] = t.eo;
#pragma unroll
          for (int q = 0; q < 9; ++q) o[4 + q] = t.m[q];
        }
        wave_sync_lds();
      }
      for (int q0 = 0; q0 < 6 * g.n_jobs; q0 += 64) {  // point sub-tests
        const int src = run_owner(own, 6 * g.js - q0, g.in ? 6 * g.jobs : 0);
        const int sub = q0 + lane - 6 * __shfl(g.js, src);
        bool keep = q0 + lane < 6 * g.n_jobs;
        {
          const int na = __shfl(l_n, src), nb = __shfl(l_m, src), vs = __shfl(g.ts, src);
          const int in_ = __shfl(inv_n, src), im = __shfl(inv_m, src);
          const float thr = __shfl(l_thr, src);
          if (keep) {
            const float margin = 1e-6f + 64.f * 5.9604645e-08f * __uint_as_float(S.c.mag[src]);
            const bool of_b = sub >= 3 * na * nb;  // vertex of b against triangle of a
            const int s2 = of_b ? sub - 3 * na * nb : sub;
            const int v = (s2 * (of_b ? in_ : im)) >> 16, k = s2 - v * (of_b ? na : nb);
            const float* f = S.c.v[vs + (of_b ? 3 * na : 0) + v] + 6;
            const float* o = S.c.t[vs / 3 + (of_b ? 0 : na) + k];
            SoupTri t;
#pragma unroll
            for (int q = 0; q < 3; ++q) t.n[q] = o[q], t.o[q] = o[13 + q];
            t.d = o[3], t.eo = o[16];
#pragma unroll
            for (int q = 0; q < 9; ++q) t.m[q] = o[4 + q];
            keep = soup_point_keep(f, f + 3, t, thr, margin);
          }
        }
        leaf_push(D, keep, Item{(uint32_t)(w0 + src), (uint32_t)sub}, S.c.pt, LEAF_PT_BUF, held_pt, LV_PT, D.lpt_items);
      }
      for (int q0 = 0; q0 < 9 * g.n_jobs; q0 += 64) {  // edge sub-tests
        const int src = run_owner(own, 9 * g.js - q0, g.in ? 9 * g.jobs : 0);
        const int sub = q0 + lane - 9 * __shfl(g.js, src);
        bool keep = q0 + lane < 9 * g.n_jobs;
        {
          const int na = __shfl(l_n, src), nb = __shfl(l_m, src), vs = __shfl(g.ts, src), im = __shfl(inv_m, src);
          const float thr = __shfl(l_thr, src);
          if (keep) {
            const float mag = __uint_as_float(S.c.mag[src]);
            const int ea = ((sub * im) >> 16) / 3, eb = sub - 3 * nb * ea;
            const int a1 = ea % 3 == 2 ? ea - 2 : ea + 1, b1 = eb % 3 == 2 ? eb - 2 : eb + 1;
            const float* pa0 = S.c.v[vs + ea];
            const float* pa1 = S.c.v[vs + a1];
            const float* pb0 = S.c.v[vs + 3 * na + eb];
            const float* pb1 = S.c.v[vs + 3 * na + b1];
            keep = !cull_edge_edge(pa0, pa1, pa0 + 3, pa1 + 3, pb0, pb1, pb0 + 3, pb1 + 3, thr, mag);
          }
        }
        leaf_push(D, keep, Item{(uint32_t)(w0 + src), (uint32_t)sub}, S.c.ee, LEAF_EE_BUF, held_ee, LV_EE, D.lee_items);
      }
      wave_sync_lds();  // read before the next group overwrites
    }
  }
  // what is still held, one slot range per block and list
  if (lane == 0) s_held[0][wid] = held_pt, s_held[1][wid] = held_ee;
  __syncthreads();
  if (threadIdx.x < 2) {
    const int* h = s_held[threadIdx.x];
    const int tot = h[0] + h[1] + h[2] + h[3];
    unsigned long long base = 0;
    if (tot) {
      base = atomicAdd(&D.lvl[D.level * LV_STRIDE + (threadIdx.x ? LV_EE : LV_PT)], (unsigned long long)tot);
      if ((long long)(base + tot) > D.cap_items) atomicOr(&D.cnt[C_OVERFLOW], 1ull);
    }
    s_out[threadIdx.x] = base;
  }
  __syncthreads();
  long long bp = (long long)s_out[0], be = (long long)s_out[1];
  for (int v = 0; v < wid; ++v) bp += s_held[0][v], be += s_held[1][v];
  for (int i = lane; i < held_pt; i += 64)
    if (bp + i < D.cap_items) D.lpt_items[bp + i] = S.c.pt[i];
  for (int i = lane; i < held_ee; i += 64)
    if (be + i < D.cap_items) D.lee_items[be + i] = S.c.ee[i];
}
// The level's two lists in one launch: the last conn_blocks blocks take the
// connected list, the others the soup list; all fold the previous level's
// passes, which are complete.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8))) k_ccd_cull(Dev D) {
  __shared__ CullShare s_share[4];
  __shared__ unsigned char s_own[4][64];
  fold_pass(D, D.pair_rec, D.pass_min_s, D.pass_flag_s);
  fold_pass(D, D.pair_rec, D.pass_min_c, D.pass_flag_c);
  const int wid = threadIdx.x >> 6, nblk = (int)gridDim.x - D.conn_blocks;
  if ((int)blockIdx.x < nblk) soup_cull_part(D, nblk, s_share[wid], s_own[wid]);
  else leaf_cull_part(D, s_share[wid], s_own[wid]);
}

// ------------------------------------------- FP32 culls of CCD soup sub-tests
// FP32 form: one thread per soup item (triangle pair) runs the FP32 bounds of
// its 15 sub-tests (k_soup_keep), keeps a 15-bit mask of the survivors per
// item and appends them to two compact lists (point and edge sub-tests); the FP64 sub-tests then run over those lists only, in full
// wavefronts, and k_soup_reduce selects over the surviving slots.  A culled
// sub-test provably reports no distance below the search distance, so it
// cannot be the winner of a hit (its slot would hold +inf, toc 1, which the
// selection never takes).  The bounds (d2_cull.hpp) are those of the leaf
// level: point-triangle by the plane side and the edge half-planes of the
// triangle in its frame (soup_point_keep), edge-edge by cull_edge_edge on
// the lerped world-space edges.  Soup triangles are surrogates, so their
// plane and edge normals are computed per item in FP64 (soup_tri, rounded
// once to float) and the lateral margin adds the FP64 barycentric acceptance
// bound of that triangle.
constexpr unsigned SOUP_PT_BITS = 0xC63u;   // slots 5k and 5k+1 (point-triangle, k = 0..2)
constexpr unsigned SOUP_EE_BITS = 0x739Cu;  // slots 5k+2+l (edge k of a, edge l of b)
// FP32 form: the survivor masks of the level's soup items (soup_cull_mask's
// parts: point slots per item; edge slots by the triangle-level test per item
// and, for the items it leaves, the per-edge culls packed over the
// wavefront, nine per item, with the items' world corners staged in LDS),
// then the two compact sub-test lists (wavefront prefix sums, one atomic per
// block and list; the lists' order is free, results go to fixed slots).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8))) k_soup_keep(Dev D) {
  __shared__ float s_w[4][64][36];        // per wavefront: world corners of the items left for the per-edge culls
  __shared__ float s_thr[4][64];          // their search distances
  __shared__ float s_ex[4][64];           // and their transforms' input magnitudes
  __shared__ unsigned char s_fl[4][64];   // their lanes
  __shared__ unsigned s_em[4][64];        // per lane: surviving edge slots
  __shared__ int s_pt[2][4], s_ee[2][4];  // survivors per wavefront and list
  __shared__ unsigned long long s_at[2][2];
  int par = 0;
  const long long n = D.n_res();
  const int lane = lane_id(), wv = threadIdx.x >> 6;
  unsigned long long* cpt = D.lvl + D.level * LV_STRIDE + LV_SPT;
  unsigned long long* cee = D.lvl + D.level * LV_STRIDE + LV_SEE;
  for (long long b0 = (long long)blockIdx.x * blockDim.x; b0 < n; b0 += (long long)gridDim.x * blockDim.x) {
    const long long it = b0 + threadIdx.x;
    bool need = false;
    const float* cf = nullptr;
    size_t ga = 0, gb = 0;  // global triangle indices (node * 8 + k) of the item's two triangles
    if (it < n) {
      const Item item = D.items[it];
      const NP np = D.soup[item.np];
      const int32_t* pi = D.pair_info + 4 * np.pair;
      cf = D.pair_f + (size_t)CF_STRIDE * np.pair;
      ga = 8 * (size_t)(pi[2] + D.nodes[pi[2] + np.na].bucket) + (item.sub >> 3);
      gb = 8 * (size_t)(pi[3] + D.nodes[pi[3] + np.nb].bucket) + (item.sub & 7);
    }
    {  // the triangle-level edge test; the corners of the items it leaves to LDS
      float w[12][3];
      float thr = 0.f, extra = 0.f;
      if (it < n) {
        float ca[9], cb[9];
        load_corners_f(D.fbuckets, ga, ca), load_corners_f(D.fbuckets, gb, cb);
        thr = cf[CF_SEARCH];
        extra = soup_world(load_m34f(cf + CF_A0), load_m34f(cf + CF_A1), load_m34f(cf + CF_B0), load_m34f(cf + CF_B1),
                           ca, cb, w);
        need = !cull_tri_edges(w, w + 3, w + 6, w + 9, thr, extra);
      }
      const unsigned long long tm = __ballot(need);
      if (need) {
        const int r = __popcll(tm & lanes_below());
#pragma unroll
        for (int q = 0; q < 12; ++q)
#pragma unroll
          for (int c = 0; c < 3; ++c) s_w[wv][r][3 * q + c] = w[q][c];
        s_thr[wv][r] = thr;
        s_ex[wv][r] = extra;
        s_fl[wv][r] = (unsigned char)lane;
      }
    }
    s_em[wv][lane] = 0u;
    unsigned mask = 0u;  // the point slots (the corners are read again: fewer live registers)
    if (it < n) {
      float ca[9], cb[9];
      load_corners_f(D.fbuckets, ga, ca), load_corners_f(D.fbuckets, gb, cb);
      mask = soup_point_mask(load_m34f(cf + CF_MAB0), load_m34f(cf + CF_MAB1), load_m34f(cf + CF_MBA0),
                             load_m34f(cf + CF_MBA1), ca, cb, load_soup_tri(D.stris, ga), load_soup_tri(D.stris, gb),
                             cf[CF_SEARCH]);
    }
    wave_sync_lds();
    const int jobs = 9 * __popcll(__ballot(need));
    for (int q0 = 0; q0 < jobs; q0 += 64) {
      const int q = q0 + lane;
      if (q < jobs) {
        const int r = q / 9, e = q % 9, k = e / 3, l = e % 3;
        if (soup_edge_keep(reinterpret_cast<const float(*)[3]>(s_w[wv][r]), k, l, s_thr[wv][r], s_ex[wv][r]))
          atomicOr(&s_em[wv][s_fl[wv][r]], 1u << (5 * k + 2 + l));
      }
    }
    wave_sync_lds();
    mask |= s_em[wv][lane];
    if (it < n) D.res_mask[it] = mask;
    const int mp = __popc(mask & SOUP_PT_BITS), me = __popc(mask & SOUP_EE_BITS);
    const int ip = wave_incl_scan(mp), ie = wave_incl_scan(me);
    if (lane == 63) s_pt[par][wv] = ip, s_ee[par][wv] = ie;
    __syncthreads();
    if (threadIdx.x < 2) {  // one atomic per block and list
      const int* h = threadIdx.x ? s_ee[par] : s_pt[par];
      const int tot = h[0] + h[1] + h[2] + h[3];
      unsigned long long base = 0;
      if (tot) {
        base = atomicAdd(threadIdx.x ? cee : cpt, (unsigned long long)tot);
        if ((long long)(base + tot) > D.cap_items) atomicOr(&D.cnt[C_OVERFLOW], 1ull);
      }
      s_at[par][threadIdx.x] = base;
    }
    __syncthreads();
    long long sp = (long long)s_at[par][0] + (ip - mp), se = (long long)s_at[par][1] + (ie - me);
    for (int v = 0; v < wv; ++v) sp += s_pt[par][v], se += s_ee[par][v];
    for (unsigned m = mask; m; m &= m - 1u) {
      const int s = __ffs(m) - 1;
      const bool pt = (SOUP_PT_BITS >> s) & 1u;
      const long long slot = pt ? sp++ : se++;
      if (slot < D.cap_items) (pt ? D.pt_items : D.ee_items)[slot] = Item{(uint32_t)it, (uint32_t)s};
    }
    par ^= 1;
    wave_sync_lds();  // LDS read before the next round overwrites it
  }
}

// Point-triangle sub-test of soup item it, slot 5k+dir (k: vertex index,
// dir 0: vertex of a vs triangle of b, dir 1: vertex of b vs triangle of a).
__device__ __forceinline__ void soup_point_one(Dev& D, long long it, int k, int dir) {
  Item item = D.items[it];
  NP np = D.soup[item.np];
  const int32_t* pi = D.pair_info + 4 * np.pair;
  const double* pr = D.pair_rec + (size_t)PR_STRIDE * np.pair;
  const NodeRec na = D.nodes[pi[2] + np.na];
  const NodeRec nb = D.nodes[pi[3] + np.nb];
  int i = item.sub >> 3, j = item.sub & 7;
  const double* ba = D.buckets + (size_t)BUCKET * (pi[2] + na.bucket);
  const double* bb = D.buckets + (size_t)BUCKET * (pi[3] + nb.bucket);
  v3<double> P, Q;
  double toc = 1.0, d;
  if (dir == 0)
    d = point_tri(load_corner(ba, i, k), pr + PR_MAB0, pr + PR_MAB1, load_tri<double>(bb, j), pr + PR_TB0, pr + PR_TB1,
                  P, Q, toc);
  else
    d = point_tri(load_corner(bb, j, k), pr + PR_MBA0, pr + PR_MBA1, load_tri<double>(ba, i), pr + PR_TA0, pr + PR_TA1,
                  P, Q, toc);
  store_res(D.res + ((size_t)it * RES_SLOTS + 5 * k + dir) * 8, d, P, Q, toc);
}

// Edge-edge sub-test of soup item it, slot 5k+2+l (edge k of a, edge l of b).
__device__ __forceinline__ void soup_edge_one(Dev& D, long long it, int k, int l) {
  Item item = D.items[it];
  NP np = D.soup[item.np];
  const int32_t* pi = D.pair_info + 4 * np.pair;
  const double* pr = D.pair_rec + (size_t)PR_STRIDE * np.pair;
  const NodeRec na = D.nodes[pi[2] + np.na];
  const NodeRec nb = D.nodes[pi[3] + np.nb];
  int i = item.sub >> 3, j = item.sub & 7;
  const double* ba = D.buckets + (size_t)BUCKET * (pi[2] + na.bucket);
  const double* bb = D.buckets + (size_t)BUCKET * (pi[3] + nb.bucket);
  v3<double> a0 = load_corner(ba, i, k), a1 = load_corner(ba, i, (k + 1) % 3);
  v3<double> b0 = load_corner(bb, j, l), b1 = load_corner(bb, j, (l + 1) % 3);
  v3<double> P, Q;
  double toc = 1.0;
  double d = edge_edge(xform(pr + PR_TA0, a0), xform(pr + PR_TA0, a1), xform(pr + PR_TA1, a0), xform(pr + PR_TA1, a1),
                       xform(pr + PR_TB0, b0), xform(pr + PR_TB0, b1), xform(pr + PR_TB1, b0), xform(pr + PR_TB1, b1),
                       P, Q, toc);
  store_res(D.res + ((size_t)it * RES_SLOTS + 5 * k + 2 + l) * 8, d, P, Q, toc);
}

// ---------------------------------------------------- CCD leaf-leaf level
// Sub-test numbering of a leaf pair with n (a) and m (b) triangles, in the
// reference's order (continuous_comparison.h:855-907):
//   [0, 3nm)        vertex v = s/m of a   vs triangle s%m of b
//   [3nm, 6nm)      vertex v = s'/n of b  vs triangle s'%n of a
//   edge list       edge s/(3m) of a      vs edge s%(3m) of b   (offset 6nm)
__device__ __forceinline__ void emit_leaf(Dev& D, const NP& np, const double* pr, int kind, int ia, int ib, int sub,
                                          v3<double> A, v3<double> B, double toc) {
  unsigned long long slot = atomicAdd(&D.cnt[C_CONTACTS], 1ull);
  if ((long long)slot >= D.cap_contacts) {
    atomicOr(&D.cnt[C_OVERFLOW], D.discrete ? 2ull : 1ull);
    return;
  }
  atomicAdd(&D.pair_cnt[np.pair], 1);
  ContactRec c;
  c.key = make_key(2 * D.level + 1, 0, np.key, sub);
  c.pair = (int32_t)np.pair, c.na = (int32_t)np.na, c.nb = (int32_t)np.nb, c.kind = kind;
  c.ia = ia, c.ib = ib, c.level = 2 * D.level + 1, c.pad = 0;
  c.r[0] = A.x, c.r[1] = A.y, c.r[2] = A.z, c.r[3] = B.x, c.r[4] = B.y, c.r[5] = B.z;
  c.r[6] = pr[PR_GEOA], c.r[7] = pr[PR_GEOB], c.r[8] = 0.0, c.r[9] = 0.0, c.r[10] = toc;
  D.contacts[slot] = c;
}

__device__ __forceinline__ void leaf_point_one(Dev& D, Item item) {
  NP np = D.conn[item.np];
  const int32_t* pi = D.pair_info + 4 * np.pair;
  const double* pr = D.pair_rec + (size_t)PR_STRIDE * np.pair;
  const NodeRec na = D.nodes[pi[2] + np.na];
  const NodeRec nb = D.nodes[pi[3] + np.nb];
  const double* ba = D.buckets + (size_t)BUCKET * (pi[2] + na.bucket);
  const double* bb = D.buckets + (size_t)BUCKET * (pi[3] + nb.bucket);
  int s = (int)item.sub, n = na.ntris, m = nb.ntris;
  v3<double> P, Q;
  double toc = 1.0, d;
  int kind, ia, ib;
  if (s < 3 * n * m) {
    int v = s / m, j = s % m;
    d = point_tri(load_corner(ba, v / 3, v % 3), pr + PR_MAB0, pr + PR_MAB1, load_tri<double>(bb, j), pr + PR_TB0,
                  pr + PR_TB1, P, Q, toc);
    kind = 1, ia = v, ib = j;
  } else {
    int s2 = s - 3 * n * m, v = s2 / n, i = s2 % n;
    d = point_tri(load_corner(bb, v / 3, v % 3), pr + PR_MBA0, pr + PR_MBA1, load_tri<double>(ba, i), pr + PR_TA0,
                  pr + PR_TA1, P, Q, toc);
    kind = 2, ia = i, ib = v;
  }
  if (d < pr[PR_SEARCH]) {
    D.pass_flag_c[np.pair] = 1;
    atomic_min_pos(&D.pass_min_c[np.pair], toc);
    if (kind == 1) emit_leaf(D, np, pr, kind, ia, ib, s, P, Q, toc);
    else emit_leaf(D, np, pr, kind, ia, ib, s, Q, P, toc);  // continuous_comparison.h:876
  }
}

__device__ __forceinline__ void leaf_edge_one(Dev& D, Item item) {
  NP np = D.conn[item.np];
  const int32_t* pi = D.pair_info + 4 * np.pair;
  const double* pr = D.pair_rec + (size_t)PR_STRIDE * np.pair;
  const NodeRec na = D.nodes[pi[2] + np.na];
  const NodeRec nb = D.nodes[pi[3] + np.nb];
  int s = (int)item.sub, n = na.ntris, m = nb.ntris;
  int ea = s / (3 * m), eb = s % (3 * m);
  const double* ba = D.buckets + (size_t)BUCKET * (pi[2] + na.bucket);
  const double* bb = D.buckets + (size_t)BUCKET * (pi[3] + nb.bucket);
  v3<double> a0 = load_corner(ba, ea / 3, ea % 3), a1 = load_corner(ba, ea / 3, (ea % 3 + 1) % 3);
  v3<double> b0 = load_corner(bb, eb / 3, eb % 3), b1 = load_corner(bb, eb / 3, (eb % 3 + 1) % 3);
  v3<double> P, Q;
  double toc = 1.0;
  double d = edge_edge(xform(pr + PR_TA0, a0), xform(pr + PR_TA0, a1), xform(pr + PR_TA1, a0), xform(pr + PR_TA1, a1),
                       xform(pr + PR_TB0, b0), xform(pr + PR_TB0, b1), xform(pr + PR_TB1, b0), xform(pr + PR_TB1, b1),
                       P, Q, toc);
  if (d < pr[PR_SEARCH]) {
    D.pass_flag_c[np.pair] = 1;
    atomic_min_pos(&D.pass_min_c[np.pair], toc);
    emit_leaf(D, np, pr, 3, ea, eb, 6 * n * m + s, Q, P, toc);  // continuous_comparison.h:903
  }
}
// The level's FP64 sub-tests in one launch: the soup items' (the FP32 form's
// surviving lists, or every item's six and nine) and the connected list's, point
// and edge.  The four lists are dealt out 64 entries at a time, so no wavefront
// mixes code paths and none waits for another list's end.
__global__ void __launch_bounds__(256) k_ccd_sub(Dev D) {
  const int lane = lane_id();
  const long long se = D.fp32 ? D.n_lv(LV_SEE) : 9 * D.n_res(), sp = D.fp32 ? D.n_lv(LV_SPT) : 6 * D.n_res();
  const long long le = D.n_lv(LV_EE), lp = D.n_lv(LV_PT);
  const long long q1 = (se + 63) / 64, q2 = q1 + (le + 63) / 64, q3 = q2 + (sp + 63) / 64, q4 = q3 + (lp + 63) / 64;
  const int nw = (int)(blockDim.x >> 6);
  const long long first = (long long)blockIdx.x * nw + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (long long q = first; q < q4; q += (long long)gridDim.x * nw) {
    if (q < q1) {
      const long long t = 64 * q + lane;
      if (t < se) {
        const Item e = D.fp32 ? D.ee_items[t] : Item{(uint32_t)(t / 9), (uint32_t)(5 * (t % 9 / 3) + 2 + t % 3)};
        soup_edge_one(D, e.np, (int)e.sub / 5, (int)e.sub % 5 - 2);
      }
    } else if (q < q2) {
      const long long t = 64 * (q - q1) + lane;
      if (t < le) leaf_edge_one(D, D.lee_items[t]);
    } else if (q < q3) {
      const long long t = 64 * (q - q2) + lane;
      if (t < sp) {
        const Item e = D.fp32 ? D.pt_items[t] : Item{(uint32_t)(t / 6), (uint32_t)(5 * (t % 6 / 2) + t % 2)};
        soup_point_one(D, e.np, (int)e.sub / 5, (int)e.sub % 5);
      }
    } else {
      const long long t = 64 * (q - q3) + lane;
      if (t < lp) leaf_point_one(D, D.lpt_items[t]);
    }
  }
}

// -------------------------------------------------------------- expansion
__device__ __forceinline__ bool expand_side(const NodeRec& na, const NodeRec& nb) {
  return na.inner && (!nb.inner || na.depth < nb.depth);  // true: advance a
}
// Expansion of a node pair of the discrete list, packed: bit 0 advance a,
// bits 1-4 child count, bits 5-31 first child (0: two leaves, no children).
__device__ __forceinline__ int expansion_desc(const NodeRec& na, const NodeRec& nb) {
  if (!(na.inner || nb.inner)) return 0;
  const bool adv_a = expand_side(na, nb);
  const NodeRec& par = adv_a ? na : nb;
  return (adv_a ? 1 : 0) | (par.nchild << 1) | (par.child_first << 5);
}
// triTriCCDLinear's selection over its 15 sub-results in the reference order
// (continuous_comparison.h:680-779), hit test (continuous_comparison.h:817),
// contact emission for leaf-leaf node pairs.  Returns whether this is the first
// hit found of a node pair with children to visit.
__device__ __forceinline__ bool soup_reduce_one(Dev& D, long long t) {
  Item item = D.items[t];
  const double* r = D.res + (size_t)t * RES_SLOTS * 8;
  double best = 1.0 / 0.0, toc = 1.0;
  int win = -1;
  const unsigned live = D.fp32 ? D.res_mask[t] : (1u << RES_SLOTS) - 1u;  // FP32 form: culled slots hold nothing
  for (int s = 0; s < RES_SLOTS; ++s) {
    if (!((live >> s) & 1u)) continue;
    double d = r[8 * s], tc = r[8 * s + 1];
    if (d < best || (d == best && tc < toc)) best = d, toc = tc, win = s;
  }
  NP np = D.soup[item.np];
  const double* pr = D.pair_rec + (size_t)PR_STRIDE * np.pair;
  bool hit = best < pr[PR_SEARCH];
  if (!hit) return false;
  atomic_min_pos(&D.pass_min_s[np.pair], toc);
  const int32_t* pi = D.pair_info + 4 * np.pair;
  const NodeRec na = D.nodes[pi[2] + np.na];
  const NodeRec nb = D.nodes[pi[3] + np.nb];
  if (na.inner || nb.inner) return atomicOr(&D.np_hit[item.np], 1) == 0;
  D.pass_flag_s[np.pair] = 1;
  unsigned long long slot = atomicAdd(&D.cnt[C_CONTACTS], 1ull);
  if ((long long)slot >= D.cap_contacts) {
    atomicOr(&D.cnt[C_OVERFLOW], D.discrete ? 2ull : 1ull);
    return false;
  }
  atomicAdd(&D.pair_cnt[np.pair], 1);
  ContactRec c;
  c.key = make_key(2 * D.level, 0, np.key, (int)item.sub);
  c.pair = (int32_t)np.pair, c.na = (int32_t)np.na, c.nb = (int32_t)np.nb, c.kind = 0;
  c.ia = (int32_t)(item.sub >> 3), c.ib = (int32_t)(item.sub & 7), c.level = 2 * D.level, c.pad = 0;
  const double* w = r + 8 * win;
  c.r[0] = w[2], c.r[1] = w[3], c.r[2] = w[4], c.r[3] = w[5], c.r[4] = w[6], c.r[5] = w[7];
  c.r[6] = pr[PR_GEOA], c.r[7] = pr[PR_GEOB], c.r[8] = 0.0, c.r[9] = 0.0, c.r[10] = toc;
  D.contacts[slot] = c;
  return false;
}
// The children of the node pairs a block claimed (full_tree_comparison.h:26-62,
// 99-150), one node pair per thread, to the next level's two lists: a child
// pair goes to the soup list when either node is inner -- all of them when the
// node that stays is inner, else the inner children of the one that advances.
// One slot range per list and round; the lists' order is free.
__device__ __forceinline__ void write_ccd_children(Dev& D, const unsigned* claim, int n_claim) {
  __shared__ unsigned long long s_base[2];
  for (int t0 = 0; t0 < n_claim; t0 += blockDim.x) {
    const int t = t0 + threadIdx.x;
    NP np{};
    int ns = 0, nc = 0, first = 0;
    bool adv_a = false, stay_inner = false;
    unsigned kid = 0;
    if (t < n_claim) {
      np = D.soup[claim[t]];
      const int32_t* pi = D.pair_info + 4 * np.pair;
      const NodeRec na = D.nodes[pi[2] + np.na];
      const NodeRec nb = D.nodes[pi[3] + np.nb];
      adv_a = expand_side(na, nb);
      stay_inner = adv_a ? nb.inner : na.inner;
      const int nch = adv_a ? na.nchild : nb.nchild;
      first = adv_a ? na.child_first : nb.child_first;
      kid = stay_inner ? (1u << nch) - 1u : (unsigned)D.kid_inner[(adv_a ? pi[2] : pi[3]) + (adv_a ? np.na : np.nb)];
      ns = __popc(kid), nc = nch - ns;
    }
    int tot;
    const int ex = block_scan(ns | nc << 16, tot);  // (a block's sums stay below 2^16: 8 children x 256)
    if (threadIdx.x < 2) {
      const int k = threadIdx.x, sum = k ? tot >> 16 : tot & 0xffff;
      unsigned long long base = 0;
      if (sum) {
        base = atomicAdd(&D.lvl[(D.level + 1) * LV_STRIDE + (k ? LV_CONN : LV_SOUP)], (unsigned long long)sum);
        if ((long long)(base + sum) > D.cap_np) atomicOr(&D.cnt[C_OVERFLOW], 1ull);
      }
      s_base[k] = base;
    }
    __syncthreads();
    long long ps = (long long)s_base[0] + (ex & 0xffff), pc = (long long)s_base[1] + (ex >> 16);
    for (int c = 0; c < ns + nc; ++c) {
      const uint32_t id = (uint32_t)(first + c);
      const bool to_soup = (kid >> c) & 1u;
      const long long slot = to_soup ? ps++ : pc++;
      if (slot < D.cap_np)
        (to_soup ? D.soup_next : D.conn_next)[slot] =
            NP{np.pair, adv_a ? id : np.na, adv_a ? np.nb : id, 0u, np.key * 8ull + (unsigned long long)c};
    }
    __syncthreads();  // s_base is read before the next round's is written
  }
}
// The first hit of a node pair claims it; the claimed ones collect in LDS and
// are expanded by whole blocks (a level is then complete without the two
// launches that counted and wrote children in list order: on levels of up to
// 26,000 node pairs writing alone took 18 us, claiming here adds 4).
constexpr int CLAIM_CAP = 1024;
__global__ void __launch_bounds__(256) k_soup_reduce(Dev D) {
  __shared__ unsigned s_claim[CLAIM_CAP];
  __shared__ int s_n;
  const long long count = D.n_res();
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  for (long long b0 = (long long)blockIdx.x * blockDim.x; b0 < count; b0 += (long long)gridDim.x * blockDim.x) {
    const long long t = b0 + threadIdx.x;
    if (t < count && soup_reduce_one(D, t)) s_claim[atomicAdd(&s_n, 1)] = D.items[t].np;
    __syncthreads();
    const int n = s_n;
    const bool last = b0 + (long long)gridDim.x * blockDim.x >= count;
    if (n > CLAIM_CAP - (int)blockDim.x || (last && n)) {
      write_ccd_children(D, s_claim, n);
      if (threadIdx.x == 0) s_n = 0;
    }
    __syncthreads();
  }
}

// The child c of a node pair of the discrete list.  Discrete lists: the
// children of a node pair that hits or may hit take slots of the next list,
// each naming its parent: parent 0 for a certain hit, list index + 1 when the
// parent's FP64 tests (k_tri_dist, its hit flag) decide; the next level drops
// the children of parents that did not hit.  The discrete phase's contacts
// carry their emission keys (child index paths) and are ordered by them
// afterwards, so its lists need no breadth-first order and children take slots
// by atomics; the keys keep every child's own index.
__device__ __forceinline__ NP child_of(const NP& np, int desc, int c, uint32_t parent) {
  const bool adv_a = desc & 1;
  const uint32_t id = (uint32_t)((desc >> 5) + c);
  return NP{np.pair, adv_a ? id : np.na, adv_a ? np.nb : id, parent, np.key * 8ull + (unsigned long long)c};
}
__device__ __forceinline__ void load_pose_f(const Dev& D, uint32_t pair, float* f) {
  const float4* p = reinterpret_cast<const float4*>(D.pair_f + (size_t)PF_STRIDE * pair);
#pragma unroll
  for (int q = 0; q < PF_FLOATS / 4; ++q) {
    const float4 v = p[q];
    f[4 * q] = v.x, f[4 * q + 1] = v.y, f[4 * q + 2] = v.z, f[4 * q + 3] = v.w;
  }
}
// ------------------------------------------------ FP32 conservative cull
// Which triangle pairs of the discrete phase need the FP64 test (FP32 form;
// the classification is in d2_cull.hpp: cull_prep, cull_apart, cull_sure):
// certain misses are dropped, and for node pairs with an inner node (they emit
// no contacts, only "any hit" matters) a certain hit settles the node pair
// without FP64 work.
static_assert(sizeof(CullTri) == 112, "prepared triangle: 28 dwords, a conflict-free LDS stride");
// A wavefront takes the node pairs of a batch in groups of at most 64
// triangles, both buckets' together: a lane prepares one triangle, then the
// group's triangle pairs go one per lane, 64 at a time; those that are no
// certain miss, of inner node pairs, move together for the certain-hit bound
// (a third of the arithmetic, needed by a tenth of them), and the candidate
// children and the kept items are spread over the lanes in the same way.
// Buckets at the leaves hold two or three triangles and most node pairs are
// there: with a pass per node pair 5 of 64 lanes worked.  Vector arithmetic
// bounds it now (68% of the chip's issue rate over a 65,536-body pile's step,
// 59-80% on its large levels); the poses come as 96-byte float records, which halved the load addresses per node pair.
// A pile's 37 M node pairs: 16.0 -> 8.4 ms; 5.5 M of 48 small scenes: 2.55 ->
// 1.5 ms; a 4,096-body scene's 0.7 M in nine levels: 516 -> 405 us.
//
// Four wavefronts per SIMD (103 VGPRs); at five it spills, and measures the same.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8))) k_tri_mask(Dev D) {
  __shared__ int s_tot[2][4], s_ch[2][4], s_df[2][4];
  __shared__ union {
    CullTri tri[64];           // per wavefront: the group's prepared triangles,
    unsigned short kid[512];   // then the children to write: child | owning lane << 4
  } s_u[4];
  __shared__ unsigned short s_job[4][256];      // and its triangle pairs: slot of a's, slot of b's << 6, inner << 12
  __shared__ unsigned char s_own[4][64];        // run starts: the owning lane + 1
  __shared__ unsigned long long s_sure[4];      // a's triangles with a certain hit
  __shared__ unsigned long long s_base[2], s_chb[2], s_dfb[2];
  const int lane = lane_id(), nw = blockDim.x >> 6, wid = threadIdx.x >> 6;
  const long long n = D.n_soup();
  // Tiles of up to 64 node pairs per wavefront, a block taking every
  // gridDim-th (how many node pairs are live, and inner, varies along the list:
  // with one long range per block the last blocks ran alone).  The wavefronts
  // of a block take consecutive parts (siblings lie next to each other: their records,
  // pose and nodes come in few cache lines); lane l fetches the record, node
  // offsets and node records of the wave's l-th node pair in one go, so the
  // per-node-pair dependent loads reduce to its pose and buckets.
  int it = 0;
  for (Tiles T(n, blockIdx.x, gridDim.x, nw); T.b0 < n; T.b0 += T.step, ++it) {
    const long long w0 = T.first(wid);
    const long long wl = w0 + lane;
    const bool in_range = lane < T.part && wl < n;
    int l_pair = 0, l_ga = 0, l_gb = 0, l_nta = 0, l_ntb = 0, l_inner = 0, l_desc = 0;  // l_ga, l_gb: global buckets
    int l_offa = 0, l_offb = 0;
    if (in_range) {
      const NP np = D.soup[wl];
      const int hit = np.pad != 0u ? D.np_hit_prev[np.pad - 1u] : 1;
      const int32_t* pi = D.pair_info + 4 * np.pair;
      l_pair = (int)np.pair, l_offa = pi[2], l_offb = pi[3];
      // a child of a parent that did not hit, or a node pair whose leaves are
      // provably apart: no work, no children.  Spheres are tested when a
      // child is written (roots here); the boxes' face-axis test runs here,
      // one node pair per lane, before the node records are loaded (few
      // registers are live).
      bool live = hit != 0;
      if (live && D.prune && (D.level == 0 || D.box_test)) {
        float f[PF_FLOATS];
        load_pose_f(D, np.pair, f);
        const float* bA = D.nbound + NB_STRIDE * ((size_t)l_offa + np.na);
        const float* bB = D.nbound + NB_STRIDE * ((size_t)l_offb + np.nb);
        live = !((D.level == 0 && spheres_apart_rel(f, bA, bB)) || (D.box_test && boxes_apart_faces_rel(f, bA, bB)));
      }
      if (live) {
        const NodeRec na = D.nodes[l_offa + np.na];
        const NodeRec nb = D.nodes[l_offb + np.nb];
        l_ga = l_offa + na.bucket, l_gb = l_offb + nb.bucket, l_nta = na.ntris, l_ntb = nb.ntris;
        l_inner = (na.inner || nb.inner) ? 1 : 0;
        l_desc = expansion_desc(na, nb);
      }
    }
    unsigned long long my_keep = 0;  // bit i * l_ntb + j: triangle i of a against j of b
    int my_settled = 0;
    const int my_jobs = l_nta * l_ntb;
    for (Groups g(my_jobs > 0 ? l_nta + l_ntb : 0, my_jobs); g.next(true);) {
      const int ts = g.ts, js = g.js, jobs = g.n_jobs;
      const bool in = g.in;
      s_own[wid][lane] = 0;
      wave_sync_lds();
      if (in) s_own[wid][ts] = (unsigned char)(lane + 1);
      wave_sync_lds();
      {
        // lane t prepares the group's triangle t.  Every lane takes part in
        // every shuffle (inside divergent code one may read an inactive
        // source lane).
        const int start = run_start(s_own[wid][lane] != 0);
        const int src = (int)s_own[wid][start] - 1, x = lane - start;
        const int pair = __shfl(l_pair, src), nta = __shfl(l_nta, src), ntb = __shfl(l_ntb, src);
        const int ga = __shfl(l_ga, src), gb = __shfl(l_gb, src);
        const int jstart = __shfl(js, src), inner = __shfl(l_inner, src);
        const bool side = x >= nta;
        const int kk = side ? x - nta : x;
        if (lane < g.n_slots) {
          CullTri mine{};
          // (b's rotation, no translation: b's position is the origin)
          const float4* pf = reinterpret_cast<const float4*>(D.pair_f + (size_t)PF_STRIDE * pair + (side ? PF_RB : PF_RA));
          const float search = D.pair_f[(size_t)PF_STRIDE * pair + PF_SEARCH];
          const float4 p0 = pf[0], p1 = pf[1], p2 = pf[2];
          const float rot[9] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w, p2.x};
          const float tr[3] = {side ? 0.f : p2.y, side ? 0.f : p2.z, side ? 0.f : p2.w};
          const float4* fb =
              reinterpret_cast<const float4*>(D.fbuckets + (size_t)FB_STRIDE * (8 * (size_t)(side ? gb : ga) + kk));
          const float4 q0 = fb[0], q1 = fb[1], q2 = fb[2];
          const float c9[9] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w, q2.x};
          cull_prep_f(rot, tr, c9, mine);
          const double eps = __hiloint2double(__float_as_int(q2.w), __float_as_int(q2.z));
          mine.eps = side ? eps : (double)search + eps;  // the reference's sum starts so: (search + eps_a) + eps_b
          s_u[wid].tri[lane] = mine;
          if (!side)
            for (int j = 0; j < ntb; ++j)
              s_job[wid][jstart + kk * ntb + j] =
                  (unsigned short)(lane | ((start + nta + j) << 6) | (inner << 12));
        }
        wave_sync_lds();
      }
      // which are certain misses; the others of inner node pairs move to the
      // front of the list
      int left = 0;
      for (int q0 = 0; q0 < jobs; q0 += 64) {
        int job = 0;
        bool keep = false;
        if (q0 + lane < jobs) {  // operands read from LDS where they are used (fewer live registers)
          job = s_job[wid][q0 + lane];
          const CullTri& A = s_u[wid].tri[job & 63];
          const CullTri& B = s_u[wid].tri[(job >> 6) & 63];
          keep = !cull_apart(A, B, (float)(A.eps + B.eps));
        }
        const unsigned long long kept = __ballot(keep);
        my_keep |= g.share(kept, q0);
        const bool more = keep && job >> 12;
        const unsigned long long m = __ballot(more);
        if (more) s_job[wid][left + __popcll(m & lanes_below())] = (unsigned short)job;
        left += __popcll(m);
      }
      // and which of those are certain hits
      if (left) {
        if (lane == 0) s_sure[wid] = 0ull;
        wave_sync_lds();
        for (int q = lane; q < left; q += 64) {
          const int job = s_job[wid][q];
          const CullTri& A = s_u[wid].tri[job & 63];
          const CullTri& B = s_u[wid].tri[(job >> 6) & 63];
          if (cull_sure(A, B, (float)(A.eps + B.eps))) atomicOr(&s_sure[wid], 1ull << (job & 63));
        }
        wave_sync_lds();
        if (in && (s_sure[wid] >> ts & ((1ull << l_nta) - 1ull)) != 0ull) my_settled = 1;
      }
      wave_sync_lds();  // read before the next group overwrites
    }
    if (my_settled) my_keep = 0ull;
    if (in_range) D.np_hit[wl] = my_settled;
    // The kept triangle pairs go straight to the level's item list, and the
    // children of node pairs that hit (settled) or may hit (kept pairs) to
    // the next list: one slot range each per block and round, one atomic
    // each (order does not matter: contacts carry their emission keys).  An
    // inner node pair's items only decide whether it expands (any FP64 hit):
    // its first kept item goes to the item list, the others (deferred) to
    // k_tri_def, which tests them only while the node pair has no hit.
    const int kept = __popcll(my_keep);
    const int defer = D.defer && l_inner != 0 ? 1 : 0;
    const int mine = defer && kept > 1 ? 1 : kept, mdef = kept - mine;
    // The children: one per lane, 64 at a time; those spheres_apart_rel does
    // not prove contact-free are listed.
    const int cand = my_settled || kept ? (l_desc >> 1) & 15 : 0;
    const int cand_incl = wave_incl_scan(cand), cands = rl(cand_incl, 63);
    int nch = 0;
    for (int q0 = 0; q0 < cands; q0 += 64) {
      const int src = run_owner(s_own[wid], cand_incl - cand - q0, cand);
      const int c = q0 + lane - __shfl(cand_incl - cand, src), desc = __shfl(l_desc, src);
      const int pair = __shfl(l_pair, src), offa = __shfl(l_offa, src), offb = __shfl(l_offb, src);
      bool keep = q0 + lane < cands;
      if (keep && D.prune) {
        const NP child = child_of(D.soup[w0 + src], desc, c, 0u);
        float f[PF_FLOATS];
        load_pose_f(D, pair, f);
        keep = !spheres_apart_rel(f, D.nbound + NB_STRIDE * ((size_t)offa + child.na),
                                  D.nbound + NB_STRIDE * ((size_t)offb + child.nb));
      }
      const unsigned long long m = __ballot(keep);
      if (keep) s_u[wid].kid[nch + __popcll(m & lanes_below())] = (unsigned short)(c | src << 4);
      nch += __popcll(m);
    }
    const int incl = wave_incl_scan(mine), idf = wave_incl_scan(mdef);
    const int par = it & 1;
    if (lane == 63) s_tot[par][wid] = incl, s_ch[par][wid] = nch, s_df[par][wid] = idf;
    __syncthreads();
    if (threadIdx.x == 0) {  // one atomic for both ranges (same-address atomics from every block are costly)
      int sum = 0, sch = 0, sdf = 0;
      for (int v = 0; v < nw; ++v) sum += s_tot[par][v], sch += s_ch[par][v], sdf += s_df[par][v];
      unsigned long long base = 0, chb = 0, dfb = 0;
      if (sum || sch) {
        const unsigned long long old =
            atomicAdd(&D.lvl[D.level * LV_STRIDE + LV_PACK], ((unsigned long long)sch << 32) | (unsigned)sum);
        base = old & 0xffffffffull, chb = old >> 32;
        if ((long long)(base + sum) > D.cap_items || (long long)(chb + sch) > D.cap_np)
          atomicOr(&D.cnt[C_OVERFLOW], 2ull);
      }
      if (sdf) {  // deferred items: their own range (another address)
        dfb = atomicAdd(&D.lvl[D.level * LV_STRIDE + LV_DEF], (unsigned long long)sdf);
        if ((long long)(dfb + sdf) > D.cap_items) atomicOr(&D.cnt[C_OVERFLOW], 2ull);
      }
      s_base[par] = base, s_chb[par] = chb, s_dfb[par] = dfb;
    }
    __syncthreads();
    long long cbase = (long long)s_chb[par];
    for (int v = 0; v < wid; ++v) cbase += s_ch[par][v];
    for (int q0 = 0; q0 < nch; q0 += 64) {
      const int e = q0 + lane < nch ? s_u[wid].kid[q0 + lane] : 0, src = e >> 4;
      const int desc = __shfl(l_desc, src), sure = __shfl(my_settled, src);
      const long long slot = cbase + q0 + lane, w = w0 + src;
      if (q0 + lane < nch && slot < D.cap_np)
        D.soup_next[slot] = child_of(D.soup[w], desc, e & 15, sure ? 0u : (uint32_t)(w + 1));
    }
    long long base = (long long)s_base[par], dbase = (long long)s_dfb[par];
    for (int v = 0; v < wid; ++v) base += s_tot[par][v], dbase += s_df[par][v];
    // the kept triangle pairs, one per lane, 64 at a time; a deferring node
    // pair's first goes to the item list, its others to the deferred list
    const int all_incl = incl + idf, all = rl(all_incl, 63), all_excl = all_incl - kept;
    const int excl = incl - mine, dexcl = idf - mdef;
    for (int q0 = 0; q0 < all; q0 += 64) {
      const int src = run_owner(s_own[wid], all_excl - q0, kept);
      const int r = q0 + lane - __shfl(all_excl, src);
      const unsigned long long m = ((unsigned long long)(unsigned)__shfl((int)(my_keep >> 32), src) << 32) |
                                   (unsigned)__shfl((int)(unsigned)my_keep, src);
      const int ntb = __shfl(l_ntb, src), dfr = __shfl(defer, src);
      const int at = __shfl(excl, src), dat = __shfl(dexcl, src);
      const DItem item{(uint32_t)(w0 + src), (uint32_t)__shfl(l_pair, src),
                       (uint32_t)__shfl(l_ga, src), (uint32_t)__shfl(l_gb, src),
                       __shfl(l_inner, src) ? 256u : 0u};
      if (q0 + lane < all) {
        const int b = nth_bit(m, r), i = b / ntb, j = b - i * ntb;
        const bool to_def = dfr && r > 0;
        const long long slot = to_def ? dbase + dat + r - 1 : base + at + r;
        if (slot < D.cap_items)
          (to_def ? D.ditems_def : D.ditems)[slot] =
              DItem{item.np, item.pair, item.ga, item.gb, item.sub | (uint32_t)(i << 3 | j)};
      }
    }
  }
}


// tri_tri_dist by the four lanes of a quad (each with the whole operands; the
// fourth does the first's share again): lane q takes corner q of either
// triangle against the other's plane, a's edge q against b's three edges, and
// edge q of either triangle through the other, a third of the serial chain.
// The quad then picks what the sequential walk keeps: of the candidate
// distances the smallest, the earliest of equal ones; of the piercings the last.
__device__ __forceinline__ double quad_bcast(double v, int from) {
  return __shfl(v, (lane_id() & ~3) | from);
}
// aq, ae, bq, be: corners q and q + 1 of a and b (read and transformed again by
// the caller: choosing them from a and b puts the triangles in scratch memory).
__device__ __forceinline__ int quad_share() {
  const int k = lane_id() & 3;
  return k == 3 ? 0 : k;
}
__device__ __forceinline__ double tri_tri_dist_quad(const tri<double>& a, const tri<double>& b, v3<double> aq,
                                                    v3<double> ae, v3<double> bq, v3<double> be, v3<double>& P,
                                                    v3<double>& Q) {
  const int q = quad_share();
  double best = 1.0 / 0.0;
  int at = 99;  // place in the sequential order
  bool in;
  {
    const v3<double> p = project_plane(a, bq, in);
    const double d = vlen(sub(p, bq));
    if (in && d < best) P = p, Q = bq, best = d, at = q;
  }
  {
    const v3<double> p = project_plane(b, aq, in);
    const double d = vlen(sub(aq, p));
    if (in && d < best) P = aq, Q = p, best = d, at = 3 + q;
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    v3<double> x, y;
    const double d = seg_closest(aq, ae, corner(b, j), corner(b, (j + 1) % 3), x, y);
    if (d < best) P = x, Q = y, best = d, at = 6 + 3 * q + j;
  }
  int pierce = 0;  // 1 + place in the sequential order
  v3<double> X{0, 0, 0};
  bool tinf, hit;
  double t = segment_hit(a, bq, be, tinf, hit);
  if (hit) X = lerp(bq, be, t), pierce = 1 + q;
  t = segment_hit(b, aq, ae, tinf, hit);
  if (hit) X = lerp(aq, ae, t), pierce = 4 + q;
  int win = 0, wp = 0;
  double wd = quad_bcast(best, 0);
  int wa = __shfl(at, lane_id() & ~3), wv = __shfl(pierce, lane_id() & ~3);
#pragma unroll
  for (int l = 1; l < 3; ++l) {
    const double od = quad_bcast(best, l);
    const int oa = __shfl(at, (lane_id() & ~3) | l), ov = __shfl(pierce, (lane_id() & ~3) | l);
    if (od < wd || (od == wd && oa < wa)) wd = od, wa = oa, win = l;
    if (ov > wv) wv = ov, wp = l;
  }
  P = v3<double>{quad_bcast(P.x, win), quad_bcast(P.y, win), quad_bcast(P.z, win)};
  Q = v3<double>{quad_bcast(Q.x, win), quad_bcast(Q.y, win), quad_bcast(Q.z, win)};
  X = v3<double>{quad_bcast(X.x, wp), quad_bcast(X.y, wp), quad_bcast(X.z, wp)};
  if (wv > 0) P = Q = X;
  return vlen(sub(P, Q));
}
// Items up to which the FP64 triangle tests take a quad each instead of a lane:
// half of what leaves every SIMD its two wavefronts (what the test's registers
// allow).  A launch of 1,000 to 16,000 items takes 15.8 us with a lane per item,
// 12.5 with a quad; at 22,000 to 31,000 both take the same, above a quad loses
// (three lanes repeat the loads and the planes).  A 100-body step: 808 -> 785 us.
constexpr long long QUAD_ITEMS = 1 << 14;
// The FP64 test of one item (comparison_dist.h:205-240's leaf test): the
// reference's triangle distance at the phase's poses against search + eps_a
// + eps_b.
struct ItemTest {
  v3<double> P, Q;
  double ea, eb;
  int i, j;
  bool hit;
};
template <bool QUAD> __device__ __forceinline__ ItemTest item_test(const Dev& D, const DItem& item) {
  ItemTest r;
  const double* pr = D.pair_rec + (size_t)PR_STRIDE * item.pair;
  const double* ba = D.buckets + (size_t)BUCKET * item.ga;
  const double* bb = D.buckets + (size_t)BUCKET * item.gb;
  const int sub = (int)(item.sub & 63u);
  r.i = sub >> 3, r.j = sub & 7;
  const tri<double> A = xform(pr + PR_TA1, load_tri<double>(ba, r.i));
  const tri<double> B = xform(pr + PR_TB1, load_tri<double>(bb, r.j));
  double d;
  if (QUAD) {
    const int q = quad_share(), e = q == 2 ? 0 : q + 1;
    d = tri_tri_dist_quad(A, B, xform(pr + PR_TA1, load_corner(ba, r.i, q)), xform(pr + PR_TA1, load_corner(ba, r.i, e)),
                          xform(pr + PR_TB1, load_corner(bb, r.j, q)), xform(pr + PR_TB1, load_corner(bb, r.j, e)), r.P,
                          r.Q);
  } else {
    d = tri_tri_dist(A, B, r.P, r.Q);
  }
  r.ea = ba[72 + r.i], r.eb = bb[72 + r.j];
  r.hit = d < (pr[PR_SEARCH] + r.ea) + r.eb;
  return r;
}
// FP64 triangle-pair distances of the level's items (grid-stride).
template <bool QUAD> __global__ void __launch_bounds__(256) k_tri_dist(Dev D) {
  const unsigned long long pack = D.lv(D.level, LV_PACK);
  const long long n_items = (long long)(pack & 0xffffffffull);
  const long long count = n_items < D.cap_items ? n_items : D.cap_items;
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // the plain sizes, for the next level and the host
    D.lvl[D.level * LV_STRIDE + LV_ITEMS] = (unsigned long long)n_items;
    D.lvl[(D.level + 1) * LV_STRIDE + LV_SOUP] = pack >> 32;
    atomicAdd(&D.cnt[C_LVL_ITEMS], (unsigned long long)n_items);
  }
  const long long stride = (long long)gridDim.x * blockDim.x / (QUAD ? 4 : 1);
  for (long long t = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / (QUAD ? 4 : 1); t < count; t += stride) {
    const DItem item = D.ditems[t];
    const ItemTest r = item_test<QUAD>(D, item);
    if (!r.hit || (QUAD && (threadIdx.x & 3))) continue;
    D.np_hit[item.np] = 1;
    if (item.sub & 256u) continue;  // an inner node: the hit only expands the node pair
    unsigned long long slot = atomicAdd(&D.cnt[C_CONTACTS], 1ull);
    if ((long long)slot >= D.cap_contacts) {
      atomicOr(&D.cnt[C_OVERFLOW], D.discrete ? 2ull : 1ull);
      continue;
    }
    atomicAdd(&D.pair_cnt[item.pair], 1);
    const NP np = D.soup[item.np];
    ContactRec c;
    const double* pr = D.pair_rec + (size_t)PR_STRIDE * item.pair;
    c.key = make_key(D.level, 0, np.key, (int)(item.sub & 63u));
    c.pair = (int32_t)np.pair, c.na = (int32_t)np.na, c.nb = (int32_t)np.nb, c.kind = 0;
    c.ia = r.i, c.ib = r.j, c.level = D.level, c.pad = 0;
    c.r[0] = r.P.x, c.r[1] = r.P.y, c.r[2] = r.P.z, c.r[3] = r.Q.x, c.r[4] = r.Q.y, c.r[5] = r.Q.z;
    c.r[6] = pr[PR_GEOA] + r.ea, c.r[7] = pr[PR_GEOB] + r.eb;
    c.r[8] = D.buckets[(size_t)BUCKET * item.ga + 80 + r.i], c.r[9] = D.buckets[(size_t)BUCKET * item.gb + 80 + r.j];
    c.r[10] = 0.0;
    D.contacts[slot] = c;
  }
}

// The deferred items of inner node pairs (FP32 form, after k_tri_dist): an
// inner node pair's FP64 tests only decide whether it expands, so a deferred
// item is tested only while its node pair has no hit.  The items still
// needed are queued per wavefront in LDS and tested 64 at a time, so the
// FP64 test runs on full wavefronts; a hit sets the node pair's flag (inner
// node pairs emit no contacts).  Every wavefront walks its 64-item chunks to
// the end of the list, then drains its queue.
__global__ void __launch_bounds__(256) k_tri_def(Dev D) {
  __shared__ uint32_t s_q[4][128];
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  const long long n_def = D.lv(D.level, LV_DEF);
  const long long n = n_def < D.cap_items ? n_def : D.cap_items;
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&D.cnt[C_LVL_ITEMS], (unsigned long long)n_def);
  const long long waves = (long long)gridDim.x * (blockDim.x >> 6);
  int qn = 0;  // queue length (wavefront-uniform), below 64 between chunks
  for (long long c0 = ((long long)blockIdx.x * (blockDim.x >> 6) + wid) * 64;; c0 += waves * 64) {
    const bool more = c0 < n;
    if (more) {
      const long long t = c0 + lane;
      const bool need = t < n && D.np_hit[D.ditems_def[t].np] == 0;
      const unsigned long long b = __ballot(need);
      if (need) s_q[wid][qn + __popcll(b & lanes_below())] = (uint32_t)t;
      qn += __popcll(b);
      wave_sync_lds();
    }
    while (qn >= 64 || (!more && qn > 0)) {
      const int take = qn < 64 ? qn : 64;
      if (lane < take) {
        const DItem item = D.ditems_def[s_q[wid][lane]];
        if (D.np_hit[item.np] == 0 && item_test<false>(D, item).hit) D.np_hit[item.np] = 1;
      }
      const int rest = qn - take;  // below 64: move it to the queue's front
      const uint32_t v = lane < rest ? s_q[wid][take + lane] : 0u;
      wave_sync_lds();
      if (lane < rest) s_q[wid][lane] = v;
      wave_sync_lds();
      qn = rest;
    }
    if (!more) break;
  }
}

// FP64 discrete levels in one pass, with no item list (the reference's own
// form: the triangle pairs of a node pair tested in place,
// full_tree_comparison.h:26-62 with bucketCompare, discrete_comparison.h).
// A wavefront takes G node pairs at a time and packs their valid triangle
// pairs (n_a * n_b each) densely over its lanes: a prefix sum over the counts,
// then each lane finds the node pair of its triangle pair by binary search
// over the sums.  The FP64 test, the contact record and its emission key are
// k_tri_dist's, so the contacts are the same bit for bit; hits set the node
// pair's flag and expansion descriptor for k_disc_expand.
//
// G = 1 to 64 is the level's node pairs over the launch's wavefronts: with 64
// always, a level of 20 000 node pairs ran on 320 of the chip's 2048 resident
// wavefronts, each a chain of up to 64 tests.
//
// CULL (pruning on): FP64 bounds (cull_pair64) first classify every triangle
// pair; certain misses are not tested, an inner node pair with a certain hit
// is settled, and of the others an inner node pair's first kept pair is
// tested before the rest, which run only while it has no hit (an inner node
// pair only asks whether any pair hits).  The kept pairs of the G node pairs
// are queued in LDS and tested 64 at a time.  311 bodies (1.6 M triangle pairs
// in 7 levels): 2734 us of k_tri_full with G = 64 and every pair tested, 363
// us now; what is left is the latency of a level's one or two tests in a row
// (4300 instructions each) behind the loads.
constexpr long long FULL_WAVES = 2048;  // wavefronts resident at its 253 VGPRs: two per SIMD
struct FullSlot {
  int pair, ga, gb, ntb, excl, inner;
  long long w;
};
// The FP64 test of triangle pair (i, j) of slot o: its contact for leaf pairs.
// Every lane of the wavefront calls it (active: has a pair).
__device__ __forceinline__ bool full_test(Dev& D, const FullSlot& o, int i, int j, bool active) {
  bool hit = false, emit = false;
  v3<double> P{}, Q{};
  double ea = 0.0, eb = 0.0;
  if (active) {
    const double* pr = D.pair_rec + (size_t)PR_STRIDE * o.pair;
    const double* ba = D.buckets + (size_t)BUCKET * o.ga;
    const double* bb = D.buckets + (size_t)BUCKET * o.gb;
    const tri<double> A = xform(pr + PR_TA1, load_tri<double>(ba, i));
    const tri<double> B = xform(pr + PR_TB1, load_tri<double>(bb, j));
    const double d = tri_tri_dist(A, B, P, Q);
    ea = ba[72 + i], eb = bb[72 + j];
    hit = d < (pr[PR_SEARCH] + ea) + eb;
    emit = hit && !o.inner;  // an inner node: the hit only expands the node pair
  }
  const long long slot = wave_alloc(emit, &D.cnt[C_CONTACTS]);
  if (!emit) return hit;
  if (slot >= D.cap_contacts) {
    atomicOr(&D.cnt[C_OVERFLOW], 2ull);
    return hit;
  }
  atomicAdd(&D.pair_cnt[o.pair], 1);
  const NP np = D.soup[o.w];
  const double* pr = D.pair_rec + (size_t)PR_STRIDE * o.pair;
  const double* ba = D.buckets + (size_t)BUCKET * o.ga;
  const double* bb = D.buckets + (size_t)BUCKET * o.gb;
  ContactRec c;
  c.key = make_key(D.level, 0, np.key, 8 * i + j);
  c.pair = (int32_t)np.pair, c.na = (int32_t)np.na, c.nb = (int32_t)np.nb, c.kind = 0;
  c.ia = i, c.ib = j, c.level = D.level, c.pad = 0;
  c.r[0] = P.x, c.r[1] = P.y, c.r[2] = P.z, c.r[3] = Q.x, c.r[4] = Q.y, c.r[5] = Q.z;
  c.r[6] = pr[PR_GEOA] + ea, c.r[7] = pr[PR_GEOB] + eb, c.r[8] = ba[80 + i], c.r[9] = bb[80 + j], c.r[10] = 0.0;
  D.contacts[slot] = c;
  return hit;
}
template <bool CULL>
__global__ void __launch_bounds__(256) k_tri_full(Dev D) {
  __shared__ FullSlot s_np[4][64];
  __shared__ int s_hit[4][64];
  __shared__ unsigned long long s_keep[CULL ? 4 : 1][64];  // kept triangle pairs of each node pair (bit 8 i + j)
  __shared__ uint16_t s_q[CULL ? 4 : 1][4096];             // queued tests: slot << 6 | 8 i + j
  __shared__ unsigned long long s_tested;
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  const long long n = D.n_soup();
  const long long nwaves = (long long)gridDim.x * (blockDim.x >> 6);
  const long long spread = nwaves < FULL_WAVES ? nwaves : FULL_WAVES;
  const long long per = (n + spread - 1) / spread;
  const int G = (int)(per < 1 ? 1 : per > 64 ? 64 : per);
  const long long n_groups = (n + G - 1) / G;
  if (threadIdx.x == 0) s_tested = 0ull;
  __syncthreads();
  unsigned long long tested = 0ull;  // kept by lane 0
  for (long long g = (long long)blockIdx.x * (blockDim.x >> 6) + wid; g < n_groups; g += nwaves) {
    const long long w = g * G + lane;
    const bool mine = lane < G && w < n;
    int cnt = 0, desc = 0;
    FullSlot f{0, 0, 0, 1, 0, 0, w};
    if (mine) {
      const NP np = D.soup[w];
      // a child of a parent that did not hit: no work, no children
      const int32_t* pi = D.pair_info + 4 * np.pair;
      const double* pr = D.pair_rec + (size_t)PR_STRIDE * np.pair;
      if ((np.pad == 0u || D.np_hit_prev[np.pad - 1u] != 0) &&
          !(D.prune && D.level == 0 &&
            nodes_apart(pr + PR_TA1, pr + PR_TB1, D.nbound + NB_STRIDE * ((size_t)pi[2] + np.na),
                        D.nbound + NB_STRIDE * ((size_t)pi[3] + np.nb), pr[PR_SEARCH]))) {
        const NodeRec na = D.nodes[pi[2] + np.na];
        const NodeRec nb = D.nodes[pi[3] + np.nb];
        f.pair = (int)np.pair, f.ga = pi[2] + na.bucket, f.gb = pi[3] + nb.bucket;
        f.ntb = nb.ntris > 0 ? nb.ntris : 1;
        f.inner = (na.inner || nb.inner) ? 1 : 0;
        cnt = na.ntris * nb.ntris;
        desc = expansion_desc(na, nb);
      }
    }
    const int incl = wave_incl_scan(cnt);
    f.excl = incl - cnt;
    s_np[wid][lane] = f;
    s_hit[wid][lane] = 0;
    if (CULL) s_keep[wid][lane] = 0ull;
    const int total = rl(incl, 63);
    wave_sync_lds();
    for (int t0 = 0; t0 < total; t0 += 64) {
      const int t = t0 + lane;
      // the owning node pair: how many inclusive sums are <= t (every lane
      // takes part in the shuffles)
      int k = 0;
#pragma unroll
      for (int step = 32; step > 0; step >>= 1)
        if (__shfl(incl, k + step - 1) <= t) k += step;
      k = k < 63 ? k : 63;
      const FullSlot& o = s_np[wid][k];
      const int s = t - o.excl, i = s / o.ntb, j = s - i * o.ntb;
      if (!CULL) {
        if (full_test(D, o, i, j, t < total)) s_hit[wid][k] = 1;
      } else if (t < total) {
        const double* pr = D.pair_rec + (size_t)PR_STRIDE * o.pair;
        const double* ba = D.buckets + (size_t)BUCKET * o.ga;
        const double* bb = D.buckets + (size_t)BUCKET * o.gb;
        const tri<double> A = xform(pr + PR_TA1, load_tri<double>(ba, i));
        const tri<double> B = xform(pr + PR_TB1, load_tri<double>(bb, j));
        const int cls = cull_pair64(A, B, (pr[PR_SEARCH] + ba[72 + i]) + bb[72 + j], o.inner != 0);
        if (cls == 2) s_hit[wid][k] = 1;
        else if (cls == 1) atomicOr(&s_keep[wid][k], 1ull << (8 * i + j));
      }
    }
    if (!CULL) tested += (unsigned long long)total;
    wave_sync_lds();
    if (CULL) {
      // two rounds: leaf pairs' tests and one of each unsettled inner node
      // pair, then the other tests of the inner node pairs without a hit
      for (int round = 0; round < 2; ++round) {
        unsigned long long m = s_hit[wid][lane] ? 0ull : s_keep[wid][lane];
        if (f.inner) m = round == 0 ? (m & (~m + 1ull)) : (m & (m - 1ull));
        else if (round == 1) m = 0ull;
        const int c = __popcll(m), qi = wave_incl_scan(c), nq = rl(qi, 63);
        for (int at = qi - c; m; m &= m - 1ull) s_q[wid][at++] = (uint16_t)(lane << 6 | (__ffsll((long long)m) - 1));
        wave_sync_lds();
        for (int q0 = 0; q0 < nq; q0 += 64) {
          const bool act = q0 + lane < nq;
          const int e = s_q[wid][act ? q0 + lane : 0], k = e >> 6;
          const bool need = act && !(round == 1 && s_hit[wid][k]);
          if (full_test(D, s_np[wid][k], (e >> 3) & 7, e & 7, need)) s_hit[wid][k] = 1;
          tested += (unsigned long long)__popcll(__ballot(need));
          wave_sync_lds();
        }
        wave_sync_lds();
      }
    }
    if (mine) {
      const int h = s_hit[wid][lane];
      D.np_hit[w] = h;
      if (h) D.exp_desc[w] = desc;
    }
    wave_sync_lds();  // s_np and s_hit are rewritten by the next group
  }
  if (lane == 0 && tested) atomicAdd(&s_tested, tested);
  __syncthreads();
  if (threadIdx.x == 0 && s_tested) {
    atomicAdd(&D.lvl[D.level * LV_STRIDE + LV_ITEMS], s_tested);
    atomicAdd(&D.cnt[C_LVL_ITEMS], s_tested);
  }
}

// FP64-mode discrete levels: the children of every hit node pair (from its
// expansion descriptor) to the next list, one atomic per block and round.
// Eight lanes per node pair, one per child: each tests its own child's bounds
// and writes it (18.1 us a launch when one lane walked a node pair's children,
// 8.7 us now, on levels of up to 20 000 node pairs).
// Large levels take up to 8 rounds of 32 node pairs per atomic and barrier (a
// step of 48 scenes without pruning: 2.85 -> 0.63 ms).
__global__ void __launch_bounds__(256) k_disc_expand(Dev D) {
  __shared__ int s_tot[4];
  __shared__ unsigned long long s_base;
  const long long n = D.n_soup();
  const int lane = lane_id(), wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int c = lane & 7;
  constexpr int K = 8;
  const long long turn = (long long)gridDim.x * 32;  // node pairs of one round of all blocks
  const int rounds = n >= K * turn ? K : (int)((n + turn - 1) / turn);
  for (long long b0 = (long long)blockIdx.x * 32 * rounds; b0 < n; b0 += turn * rounds) {  // block-uniform
    unsigned long long m[K];
    int cnt = 0;
#pragma unroll
    for (int r = 0; r < K; ++r) {
      m[r] = 0ull;
      if (r >= rounds) continue;
      const long long w = b0 + 32 * r + (threadIdx.x >> 3);
      bool keep = false;
      if (w < n && D.np_hit[w]) {
        const int desc = D.exp_desc[w];
        keep = c < ((desc >> 1) & 15);
        if (keep && D.prune) {
          const NP child = child_of(D.soup[w], desc, c, 0u);
          const int32_t* pi = D.pair_info + 4 * child.pair;
          const double* pr = D.pair_rec + (size_t)PR_STRIDE * child.pair;
          const float* ba = D.nbound + NB_STRIDE * ((size_t)pi[2] + child.na);
          const float* bb = D.nbound + NB_STRIDE * ((size_t)pi[3] + child.nb);
          keep = !(spheres_apart(pr + PR_TA1, pr + PR_TB1, ba, bb, pr[PR_SEARCH]) ||
                   nodes_apart(pr + PR_TA1, pr + PR_TB1, ba, bb, pr[PR_SEARCH]));
        }
      }
      m[r] = __ballot(keep);
      cnt += __popcll(m[r]);
    }
    if (lane == 0) s_tot[wid] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
      int tot = 0;
      for (int v = 0; v < nw; ++v) tot += s_tot[v];
      unsigned long long base = 0;
      if (tot) {
        base = atomicAdd(&D.lvl[(D.level + 1) * LV_STRIDE + LV_SOUP], (unsigned long long)tot);
        if ((long long)(base + tot) > D.cap_np) atomicOr(&D.cnt[C_OVERFLOW], 2ull);
      }
      s_base = base;
    }
    __syncthreads();
    long long slot = (long long)s_base;
    for (int v = 0; v < wid; ++v) slot += s_tot[v];
#pragma unroll
    for (int r = 0; r < K; ++r) {
      const long long at = slot + __popcll(m[r] & lanes_below());
      if ((m[r] >> lane) & 1ull && at < D.cap_np) {
        const long long w = b0 + 32 * r + (threadIdx.x >> 3);
        D.soup_next[at] = child_of(D.soup[w], D.exp_desc[w], c, 0u);
      }
      slot += __popcll(m[r]);
    }
    __syncthreads();  // s_tot and s_base are rewritten by the next tile
  }
}

// ------------------------------------------- algorithmic-byte accounting
// Instrumentation only (d2_set_touch_stats): which (body, node) records a
// level's traversal tests.  Bit node_base[body] + node of a bitmap stands for
// node `node` of body `body`; one bitmap per level and one per run (the union
// over the run's levels and phases), and one bit per body for each.
struct TouchArgs {
  const NP* soup;
  const NP* conn;
  const unsigned long long* lvl;
  const int* np_hit_prev;
  const int32_t* pair_info;
  const long long* node_base;
  unsigned *lv_nodes, *run_nodes, *lv_bodies, *run_bodies;
  long long cap_np;
  int level, discrete;
};
__device__ __forceinline__ void touch_bit(unsigned* bits, long long idx) {
  atomicOr(bits + (idx >> 5), 1u << (unsigned)(idx & 31));
}
// Marks the nodes of every node pair the level tests: a discrete node pair
// whose parent missed is dropped unread by k_tri_mask (same test here); every
// CCD soup and connected node pair is tested.
__global__ void __launch_bounds__(256) k_touch(TouchArgs T) {
  const unsigned long long* lv = T.lvl + (size_t)T.level * LV_STRIDE;
  const long long ns = (long long)lv[LV_SOUP] < T.cap_np ? (long long)lv[LV_SOUP] : T.cap_np;
  const long long nc = T.discrete ? 0 : ((long long)lv[LV_CONN] < T.cap_np ? (long long)lv[LV_CONN] : T.cap_np);
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < ns + nc; t += (long long)gridDim.x * blockDim.x) {
    const NP np = t < ns ? T.soup[t] : T.conn[t - ns];
    if (T.discrete && np.pad != 0u && T.np_hit_prev[np.pad - 1u] == 0) continue;
    const int a = T.pair_info[4 * np.pair], b = T.pair_info[4 * np.pair + 1];
    const long long ia = T.node_base[a] + np.na, ib = T.node_base[b] + np.nb;
    touch_bit(T.lv_nodes, ia), touch_bit(T.lv_nodes, ib);
    touch_bit(T.run_nodes, ia), touch_bit(T.run_nodes, ib);
    touch_bit(T.lv_bodies, a), touch_bit(T.lv_bodies, b);
    touch_bit(T.run_bodies, a), touch_bit(T.run_bodies, b);
  }
}
// out[0..3] += inner nodes, leaf nodes, triangles of those leaves, bodies
// marked in the bitmaps.
__global__ void __launch_bounds__(256) k_touch_count(const unsigned* nodes_bits, long long n_words, const unsigned* body_bits,
                                                     long long n_body_words, const long long* node_base, int n_bodies,
                                                     const int32_t* body_tree, const int32_t* tree_off,
                                                     const NodeRec* nodes, unsigned long long* out) {
  unsigned long long inner = 0, leaf = 0, tris = 0, bodies = 0;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long w = (long long)blockIdx.x * blockDim.x + threadIdx.x; w < n_words; w += stride) {
    unsigned m = nodes_bits[w];
    while (m) {
      const int k = __ffs(m) - 1;
      m &= m - 1u;
      const long long idx = 32 * w + k;
      int lo = 0, hi = n_bodies - 1;  // the body: the last node_base <= idx
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (node_base[mid] <= idx) lo = mid;
        else hi = mid - 1;
      }
      const NodeRec r = nodes[tree_off[body_tree[lo]] + (idx - node_base[lo])];
      if (r.inner) ++inner;
      else ++leaf, tris += (unsigned long long)r.ntris;
    }
  }
  for (long long w = (long long)blockIdx.x * blockDim.x + threadIdx.x; w < n_body_words; w += stride)
    bodies += (unsigned long long)__popc(body_bits[w]);
  for (int o = 32; o > 0; o >>= 1) {
    inner += __shfl_down(inner, o), leaf += __shfl_down(leaf, o);
    tris += __shfl_down(tris, o), bodies += __shfl_down(bodies, o);
  }
  if (lane_id() == 0) {
    if (inner) atomicAdd(out + 0, inner);
    if (leaf) atomicAdd(out + 1, leaf);
    if (tris) atomicAdd(out + 2, tris);
    if (bodies) atomicAdd(out + 3, bodies);
  }
}

// ---------------------------------------------------- bucket-level entry
// The plugin point's unit of work (strategy::ContactDetectionStrategy::
// findContactsBucketComparison, contact_detection_strategy.h:11, and its
// implementation comparison_dist.h:205-240): a list of node pairs of two
// bodies compared at the bodies' future states.  A wavefront takes consecutive
// node pairs in groups of at most 64 triangle pairs, one per lane, each tested
// in FP64 (tri_tri_dist): the latency of that test's serial chain bounds short
// lists, and a wavefront per node pair left 59 of 64 lanes idle at the leaves
// (6,007 node pairs: 83 -> 29 us).  A node pair's hits are
// consecutive slots of its wavefront's range (one atomic), and k_bucket_scan /
// k_bucket_place put them in the reference's order: node-pair order, then i,
// then j -- the lane order.
struct BucketArgs {
  const int32_t* np_list;  // [n][2] node indices within the two trees
  int n;
  const NodeRec* nodes;
  const double* buckets;
  int off_a, off_b;        // first node / bucket record of each tree
  const double* body_a;    // body records (future state at [14..27])
  const double* body_b;
  ContactRec* hits;        // hit records at provisional slots
  long long cap;
  unsigned long long* counter;  // slots taken
  long long* base;         // per node pair, its first slot
  int* count;              // per node pair, its hits
};
__global__ void __launch_bounds__(256) k_bucket_pairs(BucketArgs A) {
  __shared__ double sT[32];  // future poses of a and b (basic_utils.h:79-86)
  if (threadIdx.x == 0) {
    const double* sa = A.body_a + 14;
    const double* sb = A.body_b + 14;
    pose(quat{sa[0], sa[1], sa[2], sa[3]}, v3<double>{sa[4], sa[5], sa[6]}, sT);
    pose(quat{sb[0], sb[1], sb[2], sb[3]}, v3<double>{sb[4], sb[5], sb[6]}, sT + 16);
  }
  __syncthreads();
  __shared__ unsigned char s_own[4][64];
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  const double geo_a = A.body_a[37], geo_b = A.body_b[37];
  const double search = (double)(float)(geo_a + geo_b);  // float search distance (comparison_dist.h:207)
  for (Tiles T(A.n, blockIdx.x, gridDim.x, 4); T.b0 < A.n; T.b0 += T.step) {
    const long long w0 = T.first(wid), wl = w0 + lane;
    const bool in_range = lane < T.part && wl < A.n;
    int l_a = 0, l_b = 0, l_ga = 0, l_gb = 0, l_m = 0, jobs = 0;
    if (in_range) {
      l_a = A.np_list[2 * wl], l_b = A.np_list[2 * wl + 1];
      const NodeRec na = A.nodes[A.off_a + l_a];
      const NodeRec nb = A.nodes[A.off_b + l_b];
      l_ga = A.off_a + na.bucket, l_gb = A.off_b + nb.bucket, l_m = nb.ntris;
      jobs = na.ntris * nb.ntris;
      if (jobs == 0) A.base[wl] = 0, A.count[wl] = 0;
    }
    for (Groups g(jobs, jobs); g.next(false);) {  // a triangle pair per lane
      const int src = run_owner(s_own[wid], g.js, g.in ? g.jobs : 0);
      const int r = lane - __shfl(g.js, src), m = __shfl(l_m, src);
      const int la = __shfl(l_a, src), lb = __shfl(l_b, src), ga = __shfl(l_ga, src), gb = __shfl(l_gb, src);
      const double* ba = A.buckets + (size_t)BUCKET * ga;
      const double* bb = A.buckets + (size_t)BUCKET * gb;
      bool hit = false;
      int i = 0, j = 0;
      v3<double> P{0, 0, 0}, Q{0, 0, 0};
      if (lane < g.n_jobs) {
        i = r / m, j = r - i * m;
        const tri<double> TA = xform(sT, load_tri<double>(ba, i));
        const tri<double> TB = xform(sT + 16, load_tri<double>(bb, j));
        const double d = tri_tri_dist(TA, TB, P, Q);
        hit = d < (search + ba[72 + i]) + bb[72 + j];
      }
      const unsigned long long mask = __ballot(hit);
      unsigned long long b0 = 0;
      if (lane == 0 && mask) b0 = atomicAdd(A.counter, (unsigned long long)__popcll(mask));
      b0 = readlane_u64(b0, 0);
      if (g.in) {
        A.base[wl] = (long long)b0 + __popcll(mask & ((1ull << g.js) - 1ull));
        A.count[wl] = __popcll(g.share(mask, 0));
      }
      if (hit) {
        const long long slot = (long long)b0 + __popcll(mask & lanes_below());
        if (slot < A.cap) {
          ContactRec c;
          c.key = 0ull;
          c.pair = 0, c.na = la, c.nb = lb, c.kind = 0, c.ia = i, c.ib = j, c.level = 0, c.pad = 0;
          c.r[0] = P.x, c.r[1] = P.y, c.r[2] = P.z, c.r[3] = Q.x, c.r[4] = Q.y, c.r[5] = Q.z;
          c.r[6] = geo_a + ba[72 + i], c.r[7] = geo_b + bb[72 + j];  // Contact(P, Q, geo + eps, ..., inner eps)
          c.r[8] = ba[80 + i], c.r[9] = bb[80 + j], c.r[10] = 0.0;
          A.hits[slot] = c;
        }
      }
    }
  }
}

// Scratch of the allocation-free bucket entry (d2_find_contacts_bucket_noalloc):
// at most NOALLOC_NP node pairs and NOALLOC_HITS hits per call, laid out as
// node pairs | base | count | off | used | hits | out ints | out reals |
// counter.  Each device holds its own copy until the process ends; its
// address comes from hipGetSymbolAddress (the name is a host-side stand-in).
constexpr long long NOALLOC_NP = 1ll << 15;
constexpr long long NOALLOC_HITS = 1ll << 17;
constexpr size_t NOALLOC_BYTES = (size_t)NOALLOC_NP * (8 + 8 + 4 + 8 + 4) +
                                 (size_t)NOALLOC_HITS * (sizeof(ContactRec) + 8 * 4 + 11 * 8) + 256;
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

// The standalone filter's input as one pair: contact i keeps input position i
// as its emission key, so the per-pair finishing kernels see the caller's
// order (the unstable sort's result depends on it).
__global__ void __launch_bounds__(256) k_filter_load(int n, const double* reals, ContactRec* c, int* perm, int* pair_off,
                                                     int* n_big) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    ContactRec r;
    r.key = (unsigned long long)i;
    r.pair = 0, r.na = 0, r.nb = 0, r.kind = 0, r.ia = i, r.ib = 0, r.level = 0, r.pad = 0;
    for (int q = 0; q < 11; ++q) r.r[q] = reals[11 * (size_t)i + q];
    c[i] = r;
    perm[i] = i;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) pair_off[0] = 0, pair_off[1] = n, n_big[0] = 0, n_big[1] = 0;
}

// Exclusive offsets of the node pairs' hits (node-pair order) and the
// reference's cumulative counts (pair_used_out[k] = hits up to and including
// node pair k, comparison_dist.h:238); one block.
__global__ void __launch_bounds__(1024) k_bucket_scan(int n, const int* count, long long* off, int32_t* used) {
  constexpr int K = 8;  // node pairs per thread and round, read at once
  long long carry = 0;
  for (int b0 = 0; b0 < n; b0 += K * 1024) {
    const int per = n - b0 < K * 1024 ? (n - b0 + 1023) / 1024 : K;
    const int b = b0 + (int)threadIdx.x * per;
    int v[K], sum = 0, total;
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = k < per && b + k < n ? count[b + k] : 0;
#pragma unroll
    for (int k = 0; k < K; ++k) sum += v[k];
    long long run = carry + block_scan(sum, total);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k >= per || b + k >= n) break;
      off[b + k] = run;
      run += v[k];
      used[b + k] = (int32_t)run;
    }
    carry += total;
  }
}
// Each node pair's hits from their provisional slots to their final rows, in
// the flat contact layout (8 int32 + 11 doubles per hit).
__global__ void __launch_bounds__(256) k_bucket_place(int n, const long long* base, const int* count,
                                                      const long long* off, const ContactRec* hits, int32_t* out_i,
                                                      double* out_r) {
  const int lane = lane_id();
  const long long wave = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const long long n_waves = ((long long)gridDim.x * blockDim.x) >> 6;
  for (long long k = wave; k < n; k += n_waves) {
    if (lane >= count[k]) continue;
    const ContactRec& c = hits[base[k] + lane];
    const long long row = off[k] + lane;
    int32_t* oi = out_i + 8 * row;
    oi[0] = c.pair, oi[1] = c.na, oi[2] = c.nb, oi[3] = c.kind, oi[4] = c.ia, oi[5] = c.ib, oi[6] = c.level, oi[7] = 0;
    for (int q = 0; q < 11; ++q) out_r[11 * row + q] = c.r[q];
  }
}

// -------------------------------------------------------- post-processing
__device__ __forceinline__ long long n_contacts(const unsigned long long* cnt, long long cap) {
  long long n = (long long)cnt[C_CONTACTS];
  return n < cap ? n : cap;
}
// Pair lists up to this size are scanned inside k_scatter.
constexpr int SCAN_FUSE = 4096;
// Contacts to their pair's segment of perm.  With pair_cnt (n_pairs <=
// SCAN_FUSE) every block first scans the per-pair counts into LDS itself and
// block 0 stores the offsets and their total, so no scan launch precedes it;
// without, pair_off comes from a scan launch.
__global__ void __launch_bounds__(256) k_scatter(const unsigned long long* cnt, long long cap, const ContactRec* c,
                                                 int* pair_off, int* pair_fill, int* perm, const int* pair_cnt,
                                                 int n_pairs, unsigned long long* total_dst) {
  __shared__ int s_off[SCAN_FUSE + 1];
  const int* off = pair_off;
  if (pair_cnt) {
    const int per = (n_pairs + (int)blockDim.x - 1) / (int)blockDim.x;
    const int b = (int)threadIdx.x * per, e = b + per < n_pairs ? b + per : n_pairs;
    int acc = 0;
    for (int i = b; i < e; ++i) acc += pair_cnt[i];
    int total;
    int run = block_scan(acc, total);
    for (int i = b; i < e; ++i) {
      const int v = pair_cnt[i];
      s_off[i] = run;
      if (blockIdx.x == 0) pair_off[i] = run;
      run += v;
    }
    if (threadIdx.x == 0) {
      s_off[n_pairs] = total;
      if (blockIdx.x == 0) {
        pair_off[n_pairs] = total;
        if (total_dst) *total_dst = (unsigned long long)total;
      }
    }
    __syncthreads();
    off = s_off;
  }
  const long long n = n_contacts(cnt, cap);
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long long)gridDim.x * blockDim.x) {
    int p = c[t].pair;
    int k = atomicAdd(&pair_fill[p], 1);
    perm[off[p] + k] = (int)t;
  }
}

// The step rule's scale for one contact (separate_clusters.cpp:496-564):
// false when the contact sets none.  k: the pair's future-state kinematics.
struct StepKin {
  double mt;
  v3<double> va, wa, xa, vb, wb, xb;
};
__device__ __forceinline__ StepKin step_kin(const double* pr) {
  StepKin k;
  k.mt = pr[PR_MAXT];
  k.va = {pr[PR_VA], pr[PR_VA + 1], pr[PR_VA + 2]}, k.wa = {pr[PR_WA], pr[PR_WA + 1], pr[PR_WA + 2]};
  k.xa = {pr[PR_XA], pr[PR_XA + 1], pr[PR_XA + 2]};
  k.vb = {pr[PR_VB], pr[PR_VB + 1], pr[PR_VB + 2]}, k.wb = {pr[PR_WB], pr[PR_WB + 1], pr[PR_WB + 2]};
  k.xb = {pr[PR_XB], pr[PR_XB + 1], pr[PR_XB + 2]};
  return k;
}
__device__ __forceinline__ bool step_rule_scale(const ContactRec& ct, const StepKin& k, double& s) {
  const double mt = k.mt;
  v3<double> A{ct.r[0], ct.r[1], ct.r[2]}, B{ct.r[3], ct.r[4], ct.r[5]};
  v3<double> nrm = sub(A, B);
  double inter = ct.r[6] + ct.r[7], toc = ct.r[10];
  v3<double> rel = sub(add(k.va, cross(k.wa, sub(A, k.xa))), add(k.vb, cross(k.wb, sub(B, k.xb))));
  double len = vlen(nrm);
  if (!(dot(unit(nrm), unit(rel)) <= 0.0 || len < 1e-4)) return false;
  if (len < 1e-4) {
    if (toc == 0.0) return false;
    double st = toc - (vlen(rel) * mt) / inter;
    st = st > 0.0 ? st : 0.0;  // std::max(0.0, x): x when x > 0 (NaN keeps 0)
    s = lerp(st, toc, 0.75);
    return true;
  }
  if (!(toc < 1.0)) return false;
  double pv = -(dot(unit(nrm), rel));
  double depth = inter - len;
  double pd = (pv * toc) * mt;
  if (!(pd > 1e-6)) return false;
  if (depth < pd) {
    s = lerp(toc * (1.0 - depth / pd), toc, 0.5);
  } else {
    double fp = toc + ((1.0 - toc) * inter) / (pv * mt);
    s = lerp(toc, (1.0 < fp) ? 1.0 : fp, 0.8);  // std::min(fp, 1.0)
  }
  return true;
}

// The step rule of a step's CCD phase (separate_clusters.cpp:496-564): a
// pair's scale is the minimum of 1 and its contacts' scales, which no order
// of the contacts changes, and a step never reads its CCD contacts, so they
// stay where the emitting kernels put them (no scatter, no emission order):
// one thread per contact, an atomic minimum on the scale's bits (k_setup sets
// 1.0).  Scales are non-negative (toc >= 0, st >= 0, and the last two forms
// need pv > 0 and depth < pd), so their bit patterns order as their values;
// a NaN never passes s < 1, as std::min(min_scaling, NaN) keeps min_scaling.
__global__ void __launch_bounds__(256) k_step_rule(const unsigned long long* cnt, long long cap, const ContactRec* c,
                                                   const double* pair_rec, double* scale) {
  const long long n = n_contacts(cnt, cap);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const ContactRec& ct = c[i];
    double s;
    if (!step_rule_scale(ct, step_kin(pair_rec + (size_t)PR_STRIDE * ct.pair), s) || !(s < 1.0)) continue;
    atomicMin(reinterpret_cast<unsigned long long*>(scale + ct.pair), (unsigned long long)__double_as_longlong(s));
  }
}

// Contacts a pair may have for the LDS passes of the post-processing: the
// second pass (one 1024-thread block per CU, 143 KB of LDS) takes pairs up to
// POST_CAP_LARGE; above it a pair takes one block with global scratch.
constexpr int POST_CAP_LARGE = 2048;
struct LdsKey {
  double eps, dist;
};
__device__ __forceinline__ bool lds_less(const LdsKey& x, const LdsKey& y) {
  if (x.eps == y.eps) return x.dist < y.dist;
  return x.eps < y.eps;
}
// r + (y < x) by one borrow chain (the rank loops: a pair of 64-bit compares
// with their mask arithmetic takes three times as long).
__device__ __forceinline__ int add_less(int r, unsigned long long y, unsigned long long x) {
  unsigned t;
  asm("v_sub_co_u32 %1, vcc, %2, %3\n\t"
      "v_subb_co_u32 %1, vcc, %4, %5, vcc\n\t"
      "v_addc_co_u32 %0, vcc, 0, %0, vcc"
      : "+v"(r), "=&v"(t)
      : "v"((unsigned)y), "v"((unsigned)x), "v"((unsigned)(y >> 32)), "v"((unsigned)(x >> 32))
      : "vcc");
  return r;
}
__device__ __forceinline__ int add_less(int r, unsigned long long yh, unsigned long long yl, unsigned long long xh,
                                        unsigned long long xl) {
  unsigned t;
  asm("v_sub_co_u32 %1, vcc, %2, %3\n\t"
      "v_subb_co_u32 %1, vcc, %4, %5, vcc\n\t"
      "v_subb_co_u32 %1, vcc, %6, %7, vcc\n\t"
      "v_subb_co_u32 %1, vcc, %8, %9, vcc\n\t"
      "v_addc_co_u32 %0, vcc, 0, %0, vcc"
      : "+v"(r), "=&v"(t)
      : "v"((unsigned)yl), "v"((unsigned)xl), "v"((unsigned)(yl >> 32)), "v"((unsigned)(xl >> 32)), "v"((unsigned)yh),
        "v"((unsigned)xh), "v"((unsigned)(yh >> 32)), "v"((unsigned)(xh >> 32))
      : "vcc");
  return r;
}
// rk[i] = how many of n keys (W 64-bit words each, high word first, at kb in
// LDS) are less than key i.  Wavefront w of NW counts over its share of the
// keys for every i, 128 of them at a time, and the shares meet in rk by LDS
// atomics; the loads of eight keys are in flight together (one key per thread
// against all the others in turn waited out the LDS latency every four keys:
// 17 us for the (eps, dist) ranks of 318 contacts, 9.6 us now).  All threads
// call it; ends with a barrier.
template <int W, int NW>
__device__ __forceinline__ void block_ranks(int n, const unsigned long long* kb, int* rk, int w) {
  const int lane = lane_id();
  for (int i = threadIdx.x; i < n; i += 64 * NW) rk[i] = 0;
  __syncthreads();
  const int j0 = n * w / NW, j1 = n * (w + 1) / NW;
  for (int b = 0; b < n; b += 128) {
    const int i0 = b + lane, i1 = i0 + 64;
    unsigned long long x0[W], x1[W];
#pragma unroll
    for (int q = 0; q < W; ++q) x0[q] = kb[W * (i0 < n ? i0 : 0) + q], x1[q] = kb[W * (i1 < n ? i1 : 0) + q];
    int r0 = 0, r1 = 0, j = j0;
    for (; j + 8 <= j1; j += 8) {
      unsigned long long y[8 * W];
#pragma unroll
      for (int q = 0; q < 8 * W; ++q) y[q] = kb[W * j + q];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (W == 1) r0 = add_less(r0, y[q], x0[0]), r1 = add_less(r1, y[q], x1[0]);
        else r0 = add_less(r0, y[W * q], y[W * q + W - 1], x0[0], x0[W - 1]),
             r1 = add_less(r1, y[W * q], y[W * q + W - 1], x1[0], x1[W - 1]);
      }
    }
    for (; j < j1; ++j) {
      if (W == 1) r0 = add_less(r0, kb[j], x0[0]), r1 = add_less(r1, kb[j], x1[0]);
      else r0 = add_less(r0, kb[W * j], kb[W * j + W - 1], x0[0], x0[W - 1]),
           r1 = add_less(r1, kb[W * j], kb[W * j + W - 1], x1[0], x1[W - 1]);
    }
    if (i0 < n && r0) atomicAdd(&rk[i0], r0);
    if (i1 < n && r1) atomicAdd(&rk[i1], r1);
  }
  __syncthreads();
}
// The same permutation computed by the whole wavefront.  Each Hoare partition
// of [lo, hi) around the pivot at lo-1 is derived from ranks: with A_k the k-th
// position from the left holding an element not less than the pivot and B_k
// the k-th from the right holding one not greater (the pivot's own slot ends
// that list), the scalar loop swaps (A_k, B_k) for every k < K,
// K = #{k : A_k < B_k}, and returns min(A_K, B_{K-1}).  The closing insertion
// sort never moves an element across a leaf segment's border, so it equals a
// stable sort of every leaf segment; heapsort (depth exhausted) stays on lane 0.
// One pass finds both lists (Bpos is filled from the left: B_k is its k-th
// entry from the end), four chunks' keys in flight at a time.
__device__ __forceinline__ int wave_partition(int lo, int hi, int* ord, const int* rk, int* Apos, int* Bpos) {
  const int lane = lane_id();
  const int P = rk[ord[lo - 1]];
  int nA = 0, nB = 0;
  for (int base = lo - 1; base < hi; base += 256) {
    int key[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = base + 64 * q + lane;
      key[q] = ord[i < hi ? i : lo - 1];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) key[q] = rk[key[q]];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = base + 64 * q + lane;
      const bool ge = i >= lo && i < hi && !(key[q] < P), le = i < hi && !(P < key[q]);
      const unsigned long long ma = __ballot(ge), mb = __ballot(le);
      if (ge) Apos[nA + __popcll(ma & lanes_below())] = i;
      if (le) Bpos[nB + __popcll(mb & lanes_below())] = i;
      nA += __popcll(ma), nB += __popcll(mb);
    }
  }
  wave_sync_lds();
  const int lim = nA < nB ? nA : nB;
  int K = 0;
  for (int base = 0; base < lim; base += 64) {  // A_k < B_k holds for a prefix of k
    const int q = base + lane;
    const unsigned long long m = __ballot(q < lim && Apos[q] < Bpos[nB - 1 - q]);
    K += __popcll(m);
    if (m != ~0ull) break;
  }
  const int ak = K < nA ? Apos[K] : hi;
  const int bk1 = K > 0 ? Bpos[nB - K] : hi;
  for (int q = lane; q < K; q += 64) {  // the swapped positions are pairwise distinct
    const int pa = Apos[q], pb = Bpos[nB - 1 - q];
    const int x = ord[pa], y = ord[pb];
    ord[pa] = y;
    ord[pb] = x;
  }
  wave_sync_lds();
  return ak < bk1 ? ak : bk1;
}



// ---- one block (4 wavefronts) per pair: pairs with at most CAP contacts
// (BLK_CAP for every pair, then POST_CAP_LARGE for the larger ones)
constexpr int BLK_CAP = 512;
// queued segments per round (> 16 elements each: at most CAP / 17), 3 ints each
constexpr int blk_segs(int cap) { return 3 * (cap / 17 + 1); }

// The greedy filter's decisions for one group of up to 64 candidates in
// order: a candidate is kept unless it is near a contact kept before the
// group (near_m, one word per wavefront) or a kept candidate before it.
// strike: per candidate, the later ones near it; each kept candidate takes
// them out, so the loop runs once per kept candidate.  One wavefront.
template <int NW>
__device__ __forceinline__ unsigned long long greedy_keep(int m, const unsigned long long* strike,
                                                          const unsigned long long* near_m) {
  const unsigned long long mine = strike[lane_id()];
  unsigned long long blocked = 0ull;
#pragma unroll
  for (int k = 0; k < NW; ++k) blocked |= near_m[k];
  const unsigned long long b0 = readlane_u64(blocked, 0);
  unsigned long long open = (m < 64 ? (1ull << m) - 1ull : ~0ull) & ~b0, kept = 0ull;
  while (open) {
    const int u = __ffsll((long long)open) - 1;
    kept |= 1ull << u;
    open &= ~(readlane_u64(mine, u) | (1ull << u));
  }
  return kept;
}

// near_mid for a group of candidates (one per lane, the same in every
// wavefront) against points held by the lanes, FP32 first: coordinates are
// taken relative to an origin among the contacts, each is off by at most 4 u
// cmax (u = 2^-24, cmax the largest of them), so a distance more than err =
// 16 u cmax + 1e-6 search away from the search distance is decided, and only
// the others run the FP64 test (25 FP64 instructions per test were most of
// the greedy pass).  Distances that FP32 cannot hold, and negative or infinite
// search distances, always run it, and so do search distances of at most
// 1e-15 m (0 aside, which nothing is nearer than): their squares go under
// FP32's normal numbers from 1e-19 m on.
struct NearTest {
  double mx, my, mz, search;
  float fx, fy, fz, lo2, hi2;
  bool exact;
};
__device__ __forceinline__ NearTest near_test(double mx, double my, double mz, double search, const double* org,
                                              float cmax) {
  NearTest t{mx, my, mz, search, (float)(mx - org[0]), (float)(my - org[1]), (float)(mz - org[2]), -1.f, 0.f, false};
  const float s = (float)search, err = 16.f * 5.9604645e-08f * cmax + 1e-6f * s;
  const float lo = s - err, hi = s + err;
  t.lo2 = lo > 0.f ? lo * lo * (1.f - 1e-6f) : -1.f, t.hi2 = hi * hi * (1.f + 1e-6f);
  t.exact = __ballot(!((search == 0.0 || search > 1e-15) && search < 1e15 && cmax < 1e15f)) != 0ull;
  return t;
}
__device__ __forceinline__ float rlf(float v, int l) { return __int_as_float(rl(__float_as_int(v), l)); }
// Candidate against the points lanes u, u + step, ... (four of them, below
// lim) hold (h doubles, g floats): bit q set when near the q-th.  want: the
// lanes that need an answer.  One branch for the four.  All lanes call it.
__device__ __forceinline__ unsigned near_at4(const NearTest& t, int u, int step, int lim, double hx, double hy, double hz,
                                             float gx, float gy, float gz, bool want) {
  unsigned near = 0u, open = 0u;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int v = u + q * step, l = v < lim ? v : u;
    const float dx = t.fx - rlf(gx, l), dy = t.fy - rlf(gy, l), dz = t.fz - rlf(gz, l);
    const float s2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
    const bool in = v < lim;
    near |= (in && s2 < t.lo2) ? 1u << q : 0u;
    open |= (in && !(s2 >= t.hi2)) ? 1u << q : 0u;
  }
  if (t.exact || __ballot(want && (open & ~near)) != 0ull) {
#pragma unroll 1
    for (int q = 0; q < 4; ++q) {
      const int l = u + q * step;
      if (l >= lim) break;
      const bool r =
          near_mid(v3<double>{t.mx - readlane_d(hx, l), t.my - readlane_d(hy, l), t.mz - readlane_d(hz, l)}, t.search);
      near = (near & ~(1u << q)) | (r ? 1u << q : 0u);
    }
  }
  return near;
}

// ord[0, n) := the order std::sort gives, with the
// partitions of one round's segments spread over the block's wavefronts:
// partitions of disjoint segments commute, and every segment keeps its own
// depth budget, so the order equals the sequential introsort's.  Apos/Bpos
// are indexed by position (a segment's lists stay inside its range).
__device__ __forceinline__ void block_std_sort(int n, int* ord, const int* rk, int* Apos, int* Bpos, int* mark, int* segs,
                               int* s_cnt, int seg_stride) {
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = lane_id();
  for (int i = tid; i < n; i += blockDim.x) mark[i] = 0;
  if (tid == 0) {  // thread 0 also zeroed mark[0] above
    s_cnt[0] = 0, s_cnt[1] = 0;
    if (n > 16) segs[0] = 0, segs[1] = n, segs[2] = 2 * (63 - __clzll((long long)n)), s_cnt[0] = 1;
    else if (n > 0) mark[0] = 1;
  }
  __syncthreads();
  if (n <= 1) return;
  int cur = 0;
  for (;;) {
    const int m = s_cnt[cur];
    if (m == 0) break;
    const int* L = segs + cur * seg_stride;
    int* N = segs + (cur ^ 1) * seg_stride;
    for (int q = w; q < m; q += (int)(blockDim.x >> 6)) {
      const int f = L[3 * q], l = L[3 * q + 1];
      int d = L[3 * q + 2];
      if (d == 0) {  // depth exhausted: heapsort (libstdc++ __partial_sort) on one lane
        if (lane == 0) {
          StdSort<RankLess> srt{ord, RankLess{rk}};
          srt.heap_sort(f, l);
          mark[f] = 2;
        }
        wave_sync_lds();
        continue;
      }
      --d;
      {  // median of three to the front
        const int x = f + 1, y = f + (l - f) / 2, z = l - 1;
        const int kx = rk[ord[x]], ky = rk[ord[y]], kz = rk[ord[z]];
        int sel;
        if (kx < ky) sel = ky < kz ? y : (kx < kz ? z : x);
        else sel = kx < kz ? x : (ky < kz ? z : y);
        wave_sync_lds();
        if (lane == 0) {
          const int t = ord[f];
          ord[f] = ord[sel];
          ord[sel] = t;
        }
        wave_sync_lds();
      }
      const int cut = wave_partition(f + 1, l, ord, rk, Apos + f, Bpos + f);
      if (lane == 0) {
        // left part [f, cut) and right part [cut, l), both with depth d
        const int cf[2] = {f, cut}, cl[2] = {cut, l};
        for (int k = 0; k < 2; ++k) {
          if (cl[k] - cf[k] > 16) {
            const int slot = atomicAdd(&s_cnt[cur ^ 1], 1);
            N[3 * slot] = cf[k], N[3 * slot + 1] = cl[k], N[3 * slot + 2] = d;
          } else if (cl[k] > cf[k]) {
            mark[cf[k]] = 1;
          }
        }
      }
      wave_sync_lds();
    }
    __syncthreads();
    if (tid == 0) s_cnt[cur] = 0;
    cur ^= 1;
    __syncthreads();
  }
  // leaf segments tile [0, n): stable-sort each (<= 16 elements).  A
  // position's segment comes from the marks within 16 places, all read at
  // once, and the segment's keys likewise (walking them one by one cost a LDS
  // round trip each).
  for (int j = tid; j < n; j += blockDim.x) Apos[j] = rk[ord[j]];
  __syncthreads();
  for (int j = tid; j < n; j += blockDim.x) {
    unsigned back = 0u, ahead = 0u;  // bit q: a segment starts at j - q, at j + 1 + q
    int kind = 0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int mb = j >= q ? mark[j - q] : 0, ma = j + 1 + q < n ? mark[j + 1 + q] : 1;
      if (mb && back == 0u) kind = mb;
      back |= mb ? 1u << q : 0u, ahead |= ma ? 1u << q : 0u;
    }
    int dst = j;
    if (kind == 1) {  // (0: inside a long heap-sorted segment, 2: at its start)
      const int f = j - (__ffs((int)back) - 1), l = j + (ahead ? __ffs((int)ahead) : 17);
      const int kj = Apos[j];
      int r = 0;
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int i = f + q, ki = Apos[i < n ? i : n - 1];
        r += i < l && (ki < kj || (i < j && !(kj < ki))) ? 1 : 0;
      }
      dst = f + r;
    }
    Bpos[dst] = ord[j];
  }
  __syncthreads();
  for (int j = tid; j < n; j += blockDim.x) ord[j] = Bpos[j];
  __syncthreads();
}

// Post-processing of one pair per block: orders by rank counting instead of sorting
// networks (emission keys are unique; (eps, dist) ranks equal exactly for tied
// keys), the tie replay over the block's wavefronts, and the greedy pass of
// filterContacts 64 candidates at a time with the distance tests spread over
// the wavefronts and the decisions taken in order by the first one.  A serial
// chain bounds it (the replay of the ties, then the greedy groups in order),
// so a block's size is what its LDS leaves room for: 256 threads up to 512
// contacts (four blocks a CU), 1024 up to 2048 (143 KB, one block a CU; with
// 256 the other three SIMD slots stood empty).  One pair of 701 contacts: 350
// us with 256 threads, FP64 near tests and the sort's ranks a key per thread,
// 108 us now; a scene of 4,096 bodies (pairs of up to 318): 149 -> 84 us; a
// pile in a funnel: 2595 + 1629 -> 1488 + 436 us.
// A pair above every LDS capacity without the filter (mode 0 or 2), one block:
// the emission order by rank counting (the keys are unique; each thread ranks
// up to 8 per thread at a time against key tiles of CAP staged in LDS),
// written to perm from a copy of the pair's contact indices in keep (unused
// by these modes); in mode 2 the step rule's minimum over the block.
template <int CAP>
__device__ void pair_finish_huge(int p, const ContactRec* c, const int* pair_off, int* perm, int mode, int* keep,
                                 const double* pair_rec, double* scale, unsigned long long* skey, double* s_min) {
  const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
  const int b = pair_off[p], n = pair_off[p + 1] - b;
  for (int i = tid; i < n; i += blockDim.x) keep[b + i] = perm[b + i];
  __syncthreads();
  constexpr int K = 8;
  for (int q0 = 0; q0 < n; q0 += K * (int)blockDim.x) {
    unsigned long long mk[K];
    int rk[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = q0 + k * (int)blockDim.x + tid;
      mk[k] = i < n ? c[keep[b + i]].key : ~0ull;
      rk[k] = 0;
    }
    for (int t0 = 0; t0 < n; t0 += CAP) {
      const int m = n - t0 < CAP ? n - t0 : CAP;
      for (int j = tid; j < m; j += blockDim.x) skey[j] = c[keep[b + t0 + j]].key;
      __syncthreads();
      for (int j = 0; j < m; ++j) {
        const unsigned long long kj = skey[j];
#pragma unroll
        for (int k = 0; k < K; ++k) rk[k] += kj < mk[k] ? 1 : 0;
      }
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = q0 + k * (int)blockDim.x + tid;
      if (i < n) perm[b + rk[k]] = keep[b + i];
    }
  }
  if (mode == 2) {  // step rule, separate_clusters.cpp:496-564: the minimum over the pair's contacts
    const StepKin kin = step_kin(pair_rec + (size_t)PR_STRIDE * p);
    double ms = 1.0;
    for (int i = tid; i < n; i += blockDim.x) {
      double sc;
      if (step_rule_scale(c[keep[b + i]], kin, sc) && sc < ms) ms = sc;  // NaN never wins
    }
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_xor(ms, off);
      if (o < ms) ms = o;
    }
    if (lane == 0) s_min[w] = ms;
    __syncthreads();
    if (tid == 0) {
      double m = s_min[0];
      for (int k = 1; k < (int)(blockDim.x >> 6); ++k) m = (s_min[k] < m) ? s_min[k] : m;
      scale[p] = m;
    }
  }
}

// Global scratch of the filter above every LDS capacity: six int arrays of
// the run's contact capacity, a pair using positions [b, b + n) of each
// (its contacts' range; the sort's segment queue, at most 6 (n / 17 + 1)
// ints, fits there for n > 16).
struct HugeScratch {
  int *rk, *ord, *apos, *bpos, *mark, *segs;
};

// filterContacts(.., margin) of one pair above every LDS capacity, one block:
// the emission order by rank counting (pair_finish_huge), the (eps, dist)
// ranks by rank counting over LDS key tiles, the std::sort replay
// (block_std_sort) on global scratch when keys tie, then the greedy pass 64
// candidates at a time as in the LDS path, with the kept list in scratch.
// Returns the kept count (every thread).
template <int CAP, int NT>
__device__ int pair_filter_huge(int p, const ContactRec* c, const int* pair_off, int* perm, int* keep, int* kept_cnt,
                                double margin, const HugeScratch& H, unsigned long long* skey, LdsKey* sk,
                                int* s_misc, unsigned long long* strike, unsigned long long* near_m) {
  const int tid = threadIdx.x, lane = lane_id(), w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = pair_off[p], n = pair_off[p + 1] - b;
  pair_finish_huge<CAP>(p, c, pair_off, perm, 0, keep, nullptr, nullptr, skey, nullptr);  // perm: emission order
  if (tid == 0) s_misc[0] = 0;
  __syncthreads();
  int* rk = H.rk + b;
  int* ord = H.ord + b;
  int* eo = H.apos + b;  // the emission order, kept while perm is rewritten
  int* kl = H.mark + b;  // the kept list (emission positions), after the sort
  constexpr int K = 8;
  bool tie = false;
  for (int q0 = 0; q0 < n; q0 += K * (int)blockDim.x) {  // ranks of the (eps, dist) keys; equal keys share one
    LdsKey mk[K];
    int r[K], eq[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = q0 + k * (int)blockDim.x + tid;
      const ContactRec& ct = c[perm[b + (i < n ? i : 0)]];
      mk[k].eps = ct.r[6] + ct.r[7];
      mk[k].dist = vlen(sub(v3<double>{ct.r[0], ct.r[1], ct.r[2]}, v3<double>{ct.r[3], ct.r[4], ct.r[5]}));
      r[k] = 0, eq[k] = 0;
    }
    for (int t0 = 0; t0 < n; t0 += CAP) {
      const int m = n - t0 < CAP ? n - t0 : CAP;
      for (int j = tid; j < m; j += blockDim.x) {
        const ContactRec& ct = c[perm[b + t0 + j]];
        sk[j].eps = ct.r[6] + ct.r[7];
        sk[j].dist = vlen(sub(v3<double>{ct.r[0], ct.r[1], ct.r[2]}, v3<double>{ct.r[3], ct.r[4], ct.r[5]}));
      }
      __syncthreads();
      for (int j = 0; j < m; ++j) {
        const LdsKey y = sk[j];
#pragma unroll
        for (int k = 0; k < K; ++k) {
          if (lds_less(y, mk[k])) ++r[k];
          else if (!lds_less(mk[k], y)) ++eq[k];
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = q0 + k * (int)blockDim.x + tid;
      if (i < n) rk[i] = r[k], tie = tie || eq[k] > 1;
    }
  }
  if (tie) s_misc[0] = 1;
  __syncthreads();
  if (s_misc[0] == 0) {
    for (int i = tid; i < n; i += blockDim.x) ord[rk[i]] = i;
  } else {
    for (int i = tid; i < n; i += blockDim.x) ord[i] = i;
    __syncthreads();
    block_std_sort(n, ord, rk, H.apos + b, H.bpos + b, H.mark + b, H.segs + b, s_misc + 2, blk_segs(n));
  }
  __syncthreads();
  for (int i = tid; i < n; i += blockDim.x) eo[i] = perm[b + i];
  __syncthreads();
  // greedy pass in sorted order
  int nk = 0;
  for (int t0 = 0; t0 < n; t0 += 64) {
    const int m = n - t0 < 64 ? n - t0 : 64;
    const int t = t0 + lane;
    const bool valid = t < n;
    const ContactRec& ct = c[eo[ord[valid ? t : t0]]];
    const v3<double> mid = dvs(add(v3<double>{ct.r[0], ct.r[1], ct.r[2]}, v3<double>{ct.r[3], ct.r[4], ct.r[5]}), 2.0);
    const double mx = mid.x, my = mid.y, mz = mid.z;
    const double search = (ct.r[6] + ct.r[7]) + margin;
    bool near = false;
    for (int q0 = 0; q0 < nk; q0 += 64) {  // contacts kept before this group
      const ContactRec& hc = c[eo[kl[q0 + lane < nk ? q0 + lane : q0]]];
      const v3<double> hm =
          dvs(add(v3<double>{hc.r[0], hc.r[1], hc.r[2]}, v3<double>{hc.r[3], hc.r[4], hc.r[5]}), 2.0);
      const int mm = nk - q0 < 64 ? nk - q0 : 64;
      for (int u = w; u < mm; u += NT / 64) {
        const v3<double> dd{mx - readlane_d(hm.x, u), my - readlane_d(hm.y, u), mz - readlane_d(hm.z, u)};
        near = near || near_mid(dd, search);
      }
    }
    for (int u = w; u < m; u += NT / 64) {  // the later candidates of the group near candidate u
      const v3<double> dd{mx - readlane_d(mx, u), my - readlane_d(my, u), mz - readlane_d(mz, u)};
      const unsigned long long later = __ballot(lane > u && near_mid(dd, search));
      if (lane == 0) strike[u] = later;
    }
    const unsigned long long nm = __ballot(near);
    if (lane == 0) near_m[w] = nm;
    __syncthreads();
    if (w == 0) {
      const unsigned long long kept = greedy_keep<NT / 64>(m, strike, near_m);
      const bool fresh = (kept >> lane) & 1ull;
      if (valid) keep[b + t] = fresh ? 1 : 0;
      if (fresh) kl[nk + __popcll(kept & lanes_below())] = ord[t];
      if (lane == 0) s_misc[1] = nk + __popcll(kept);
    }
    __syncthreads();
    nk = s_misc[1];
  }
  for (int t = tid; t < n; t += blockDim.x) perm[b + t] = eo[ord[t]];
  if (tid == 0) kept_cnt[p] = nk;
  __syncthreads();
  return nk;
}

// CAP = BLK_CAP: every pair (list null); pairs above CAP go to `over` (up to
// POST_CAP_LARGE contacts) or `huge`.  CAP = POST_CAP_LARGE: the pairs of
// `list`, then the pairs of `tail` one block each (above every LDS capacity).
template <int CAP, int NT>
__global__ void __launch_bounds__(NT) k_pair_finish_block(int n_pairs, const int* list, const int* n_list,
                                                           const ContactRec* c, const int* pair_off, int* perm,
                                                           int mode, int* keep, int* kept_cnt,
                                                           const double* pair_rec, double* scale, int* over,
                                                           int* n_over, int* huge, int* n_huge, const int* tail,
                                                           const int* n_tail, unsigned long long* out_total,
                                                           double margin, HugeScratch H) {
  constexpr int SEGS = blk_segs(CAP);
  __shared__ unsigned long long skey[CAP];  // emission keys, then the partition lists of the tie replay
  __shared__ int sidx[CAP];
  __shared__ int eo[CAP];  // contact at each emission position
  __shared__ LdsKey sk[CAP];
  __shared__ double smid[3 * CAP];
  __shared__ int rk[CAP];
  __shared__ int ord[CAP];
  __shared__ int mark[CAP];  // leaf marks of the tie replay, then the kept list
  __shared__ int segs[2 * SEGS];
  __shared__ unsigned long long strike[64];
  __shared__ unsigned long long near_m[NT / 64];
  __shared__ double s_min[NT / 64];
  __shared__ float s_cmax[NT / 64];
  __shared__ int s_misc[4];
  const int tid = threadIdx.x, lane = lane_id();
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // visibly uniform: scalar loops and lane indexes
  const int n_items = list ? *n_list : n_pairs;
  unsigned long long kept_sum = 0;  // (thread 0) the filter's kept contacts of this block's pairs
  for (int it = blockIdx.x; it < n_items; it += gridDim.x) {
    const int p = list ? list[it] : it;
    const int b = pair_off[p], e = pair_off[p + 1], n = e - b;
    if (n > CAP) {  // to the second launch: its LDS pass, or (above its capacity) a block per pair
      if (tid == 0) {
        if (n > POST_CAP_LARGE) huge[atomicAdd(n_huge, 1)] = p;
        else over[atomicAdd(n_over, 1)] = p;
      }
      continue;
    }
    if (n == 0) {  // what the general path writes for a pair without contacts, without its barriers
      if (tid == 0) {
        if (mode == 2) scale[p] = 1.0;
        if (mode == 1) kept_cnt[p] = 0;
      }
      continue;
    }
    for (int i = tid; i < n; i += NT) {
      const int idx = perm[b + i];
      sidx[i] = idx;
      skey[i] = c[idx].key;
    }
    __syncthreads();
    bool asc = true;  // contacts that come in emission order need no ranks
    for (int i = tid; i + 1 < n; i += NT) asc = asc && skey[i] < skey[i + 1];
    asc = __syncthreads_and(asc ? 1 : 0);
    if (asc) {
      for (int i = tid; i < n; i += NT) eo[i] = sidx[i];
    } else {  // emission position = rank of the (unique) key
      block_ranks<1, NT / 64>(n, skey, rk, w);
      for (int i = tid; i < n; i += NT) eo[rk[i]] = sidx[i];
    }
    __syncthreads();
    if (mode == 2) {  // step rule, separate_clusters.cpp:496-564
      const double* pr = pair_rec + (size_t)PR_STRIDE * p;
      double mt = pr[PR_MAXT], ms = 1.0;
      v3<double> va{pr[PR_VA], pr[PR_VA + 1], pr[PR_VA + 2]}, wa{pr[PR_WA], pr[PR_WA + 1], pr[PR_WA + 2]};
      v3<double> xa{pr[PR_XA], pr[PR_XA + 1], pr[PR_XA + 2]};
      v3<double> vb{pr[PR_VB], pr[PR_VB + 1], pr[PR_VB + 2]}, wb{pr[PR_WB], pr[PR_WB + 1], pr[PR_WB + 2]};
      v3<double> xb{pr[PR_XB], pr[PR_XB + 1], pr[PR_XB + 2]};
      for (int i = tid; i < n; i += NT) {
        const ContactRec& ct = c[eo[i]];
        v3<double> A{ct.r[0], ct.r[1], ct.r[2]}, B{ct.r[3], ct.r[4], ct.r[5]};
        v3<double> nrm = sub(A, B);
        double inter = ct.r[6] + ct.r[7], toc = ct.r[10];
        v3<double> rel = sub(add(va, cross(wa, sub(A, xa))), add(vb, cross(wb, sub(B, xb))));
        double len = vlen(nrm);
        if (!(dot(unit(nrm), unit(rel)) <= 0.0 || len < 1e-4)) continue;
        double sc;
        if (len < 1e-4) {
          if (toc == 0.0) continue;
          double st = toc - (vlen(rel) * mt) / inter;
          st = st > 0.0 ? st : 0.0;
          sc = lerp(st, toc, 0.75);
        } else {
          if (!(toc < 1.0)) continue;
          double pv = -(dot(unit(nrm), rel));
          double depth = inter - len;
          double pd = (pv * toc) * mt;
          if (!(pd > 1e-6)) continue;
          if (depth < pd) {
            sc = lerp(toc * (1.0 - depth / pd), toc, 0.5);
          } else {
            double fp = toc + ((1.0 - toc) * inter) / (pv * mt);
            sc = lerp(toc, (1.0 < fp) ? 1.0 : fp, 0.8);
          }
        }
        if (sc < ms) ms = sc;
      }
      for (int off = 32; off > 0; off >>= 1) {
        double o = __shfl_xor(ms, off);
        if (o < ms) ms = o;
      }
      if (lane == 0) s_min[w] = ms;
      __syncthreads();
      if (tid == 0) {
        double m = s_min[0];
        for (int k = 1; k < NT / 64; ++k) m = (s_min[k] < m) ? s_min[k] : m;
        scale[p] = m;
      }
      for (int i = tid; i < n; i += NT) perm[b + i] = eo[i];
    } else if (mode == 1) {  // filterContacts(.., margin)
      for (int i = tid; i < n; i += NT) {
        const ContactRec& ct = c[eo[i]];
        const v3<double> A{ct.r[0], ct.r[1], ct.r[2]}, B{ct.r[3], ct.r[4], ct.r[5]};
        sk[i].eps = (ct.r[6] + ct.r[7]) + 0.0;
        sk[i].dist = vlen(sub(A, B)) + 0.0;
        const v3<double> m = dvs(add(A, B), 2.0);
        smid[3 * i] = m.x, smid[3 * i + 1] = m.y, smid[3 * i + 2] = m.z;
      }
      __syncthreads();
      float cmax = 0.f;  // the largest coordinate relative to contact 0
      for (int i = tid; i < n; i += NT)
        for (int q = 0; q < 3; ++q) {
          const float v = fabsf((float)(smid[3 * i + q] - smid[q]));
          cmax = fmaxf(cmax, v < 1e15f ? v : 1e30f);  // (NaN too)
        }
      for (int off = 32; off > 0; off >>= 1) cmax = fmaxf(cmax, __shfl_xor(cmax, off));
      if (lane == 0) s_cmax[w] = cmax;
      __syncthreads();
      for (int q = 0; q < NT / 64; ++q) cmax = fmaxf(cmax, s_cmax[q]);
      // rank of the (eps, dist) key: how many are less; equal keys share it.
      // Non-negative doubles order like their bits (any other key among the
      // pair's, NaN included, and the comparisons are the doubles' own)
      bool plain = true;
      for (int i = tid; i < n; i += NT) ord[i] = -1, plain = plain && sk[i].eps >= 0.0 && sk[i].dist >= 0.0;
      plain = __syncthreads_and(plain ? 1 : 0);
      if (plain) {
        block_ranks<2, NT / 64>(n, reinterpret_cast<const unsigned long long*>(sk), rk, w);
      } else {
        for (int i = tid; i < n; i += NT) {
          int r = 0;
          for (int j = 0; j < n; ++j) r += lds_less(sk[j], sk[i]) ? 1 : 0;
          rk[i] = r;
        }
        __syncthreads();
      }
      bool tie = false;
      for (int i = tid; i < n; i += NT) tie = tie || atomicExch(&ord[rk[i]], i) != -1;  // two with one rank: a tie
      tie = __syncthreads_or(tie ? 1 : 0);
      if (tie) {
        for (int i = tid; i < n; i += NT) ord[i] = i;
        __syncthreads();
        int* lists = reinterpret_cast<int*>(skey);
        block_std_sort(n, ord, rk, lists, lists + CAP, mark, segs, s_misc + 2, SEGS);
      }
      // greedy pass in sorted order
      int nk = 0;
      for (int t0 = 0; t0 < n; t0 += 64) {
        const int m = n - t0 < 64 ? n - t0 : 64;
        const int t = t0 + lane;
        const bool valid = t < n;
        const int pi = valid ? ord[t] : 0;
        const NearTest nt = near_test(smid[3 * pi], smid[3 * pi + 1], smid[3 * pi + 2], sk[pi].eps + margin, smid, cmax);
        bool near = false;
        for (int q0 = 0; q0 < nk; q0 += 64) {  // contacts kept before the block
          const int h = q0 + lane < nk ? mark[q0 + lane] : 0;
          const double hx = smid[3 * h], hy = smid[3 * h + 1], hz = smid[3 * h + 2];
          const float gx = (float)(hx - smid[0]), gy = (float)(hy - smid[1]), gz = (float)(hz - smid[2]);
          const int mm = nk - q0 < 64 ? nk - q0 : 64;
          for (int u = w; u < mm; u += 4 * (NT / 64)) {
            const unsigned r = near_at4(nt, u, NT / 64, mm, hx, hy, hz, gx, gy, gz, valid && !near);
            near = near || r != 0u;
          }
        }
        for (int u = w; u < m; u += 4 * (NT / 64)) {  // the later candidates of the group near candidates u, ...
          const unsigned r =
              near_at4(nt, u, NT / 64, m, nt.mx, nt.my, nt.mz, nt.fx, nt.fy, nt.fz, u < lane && valid && !near);
          unsigned long long later = 0ull;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const unsigned long long b = __ballot(((r >> q) & 1u) && lane > u + q * (NT / 64));
            if (lane == q) later = b;
          }
          if (lane < 4 && u + lane * (NT / 64) < m) strike[u + lane * (NT / 64)] = later;
        }
        const unsigned long long nm = __ballot(near);
        if (lane == 0) near_m[w] = nm;
        __syncthreads();
        if (w == 0) {
          const unsigned long long kept = greedy_keep<NT / 64>(m, strike, near_m);
          const bool fresh = (kept >> lane) & 1ull;
          if (valid) keep[b + t] = fresh ? 1 : 0;
          if (fresh) mark[nk + __popcll(kept & lanes_below())] = pi;
          if (lane == 0) s_misc[1] = nk + __popcll(kept);
        }
        __syncthreads();
        nk = s_misc[1];
      }
      for (int t = tid; t < n; t += NT) perm[b + t] = eo[ord[t]];
      if (tid == 0) kept_cnt[p] = nk, kept_sum += (unsigned long long)nk;
    } else {
      for (int i = tid; i < n; i += NT) perm[b + i] = eo[i];
    }
    __syncthreads();
  }
  if constexpr (CAP == POST_CAP_LARGE) {  // (kept out of the first launch's code: registers, scratch)
    if (tail) {  // pairs above every LDS capacity (listed by the first launch), one block each
      if (mode == 1) {
        for (int t = blockIdx.x; t < *n_tail; t += gridDim.x) {
          const int nk = pair_filter_huge<CAP, NT>(tail[t], c, pair_off, perm, keep, kept_cnt, margin, H, skey, sk,
                                               s_misc, strike, near_m);
          if (tid == 0) kept_sum += (unsigned long long)nk;
        }
      } else {
        for (int t = blockIdx.x; t < *n_tail; t += gridDim.x) {
          pair_finish_huge<CAP>(tail[t], c, pair_off, perm, mode, keep, pair_rec, scale, skey, s_min);
          __syncthreads();
        }
      }
    }
  }
  if (tid == 0 && out_total && kept_sum) atomicAdd(out_total, kept_sum);  // one atomic per block
}

// Gathers one pair per wavefront into the output arrays (CSR order).
__global__ void __launch_bounds__(64) k_gather_wave(int n_pairs, const ContactRec* c, const int* pair_off, const int* perm,
                                                    const int* keep, const int* out_off, int filtered, int32_t* out_i,
                                                    double* out_r) {
  const int lane = threadIdx.x;
  for (int p = blockIdx.x; p < n_pairs; p += gridDim.x) {
    int b = pair_off[p], e = pair_off[p + 1];
    int o = out_off[p];
    for (int base = b; base < e; base += 64) {
      int i = base + lane;
      bool take = i < e && (!filtered || keep[i]);
      unsigned long long m = __ballot(take);
      if (take) {
        int dst = o + __popcll(m & lanes_below());
        const ContactRec& ct = c[perm[i]];
        int32_t* oi = out_i + 8 * (size_t)dst;
        oi[0] = ct.pair, oi[1] = ct.na, oi[2] = ct.nb, oi[3] = ct.kind, oi[4] = ct.ia, oi[5] = ct.ib, oi[6] = ct.level,
        oi[7] = 0;
        double* orr = out_r + 11 * (size_t)dst;
        for (int k = 0; k < 11; ++k) orr[k] = ct.r[k];
      }
      o += __popcll(m);
    }
  }
}

// Exclusive scan of in[0, n) into out[0, n], out[n] = total (also stored to
// *total_dst when given), in two chunked kernels of the same grid.
__global__ void __launch_bounds__(256) k_scan_part(const int* in, long long n, int* part) {
  long long rb, re;
  chunk_of(n, rb, re);
  long long acc = 0;
  for (long long i = rb + threadIdx.x; i < re; i += blockDim.x) acc += in[i];
  const long long t = block_sum(acc);
  if (threadIdx.x == 0) part[blockIdx.x] = (int)t;
}
__global__ void __launch_bounds__(256) k_scan_apply(const int* in, int* out, long long n, const int* part,
                                                    unsigned long long* total_dst) {
  long long rb, re, before, total;
  chunk_of(n, rb, re);
  partial_prefix(part, before, total);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    out[n] = (int)total;
    if (total_dst) *total_dst = (unsigned long long)total;
  }
  for (long long t0 = rb; t0 < re; t0 += blockDim.x) {
    const long long i = t0 + threadIdx.x;
    int tt;
    const int ex = block_scan(i < re ? in[i] : 0, tt);
    if (i < re) out[i] = (int)(before + ex);
    before += tt;
  }
}

// The same scan for a short array (n <= SCAN_SMALL) in one block of 1024
// threads: thread t sums its run of ceil(n / 1024) elements, the block scans
// the sums, and each thread writes its run.
constexpr long long SCAN_SMALL = 16384;
__global__ void __launch_bounds__(1024) k_scan_small(const int* in, int* out, long long n,
                                                     unsigned long long* total_dst) {
  const long long per = (n + blockDim.x - 1) / blockDim.x;
  const long long b = (long long)threadIdx.x * per;
  const long long e = b + per < n ? b + per : n;
  int acc = 0;
  for (long long i = b; i < e; ++i) acc += in[i];
  int total;
  int run = block_scan(acc, total);
  for (long long i = b; i < e; ++i) {
    const int v = in[i];
    out[i] = run;
    run += v;
  }
  if (threadIdx.x == 0) {
    out[n] = total;
    if (total_dst) *total_dst = (unsigned long long)total;
  }
}

// ------------------------------------------------------ cluster step sizes
// The cluster step (separate_clusters.cpp:555-598,
// time_step_selection_dynamic_continuous.cpp:17-21).  The reference runs two
// loops over the cluster's pairs in order: the first lowers both dynamic
// bodies' steps to use = min(max_time * scale, step[a], step[b]) for a pair
// with CCD contacts; the second starts from step[a] of the first pair that is
// not static-static (:589-590) and takes min(., step[id]) over the others (id
// = a unless a is static).  Since max_time * scale <= max_time <= both last
// steps, every pair's use reaches the step its own pair reads in the second
// loop, so the result is the minimum over pairs of max_time * scale (with
// contacts) and last[id] -- order does not matter -- except for the first
// pair when its body a is static: the second loop reads a's unchanged last
// step there, and that pair's use only counts when its body b is read or
// lowered again later (a later pair whose id is b, or a later pair with
// contacts touching b: every other pair comes later).  read_later marks
// those bodies.  Steps are non-negative, so they order like their bit
// patterns.
__global__ void k_cluster_init(ClusterAcc CA) {
  cluster_init_range(CA, (long long)blockIdx.x * blockDim.x + threadIdx.x, (long long)gridDim.x * blockDim.x);
}
__global__ void k_cluster_first(int n_pairs, ClusterAcc CA) {
  cluster_first_range(CA, n_pairs, (long long)blockIdx.x * blockDim.x + threadIdx.x, (long long)gridDim.x * blockDim.x);
}
__global__ void k_cluster_min(int n_pairs, const int32_t* pairs, const int32_t* cluster_of_pair, const double* bodies,
                              const int* pair_cnt, const double* scale, const int* first_ns, int* read_later,
                              unsigned long long* step_bits) {
  for (int p0 = blockIdx.x * blockDim.x; p0 < n_pairs; p0 += gridDim.x * blockDim.x) {  // block-uniform
    const int p = p0 + threadIdx.x;
    int key = -1;
    double v = 1e300;
    if (p < n_pairs) {
      const int k = cluster_of_pair[p], a = pairs[2 * p], b = pairs[2 * p + 1];
      const double* ra = bodies + 40 * (size_t)a;
      const double* rb = bodies + 40 * (size_t)b;
      const bool sa = ra[38] != 0.0, sb = rb[38] != 0.0;
      if (!(sa && sb)) {
        const bool first = p == first_ns[k];
        const int id = !sa ? a : b;
        if (!first) {  // the second loop reads step[id]; a pair with contacts lowers a's and b's steps
          read_later[id] = 1;
          if (pair_cnt[p] > 0) read_later[a] = 1, read_later[b] = 1;
        }
        const double mt = (rb[39] < ra[39]) ? rb[39] : ra[39];
        if (pair_cnt[p] > 0 && !(first && sa)) {  // a static first pair's own use: see cluster_step_of
          const double s = mt * scale[p];
          v = (s < v) ? s : v;
        }
        const double last = first ? ra[39] : bodies[40 * (size_t)id + 39];
        v = (last < v) ? last : v;
        key = k;
      }
    }
    wave_key_min(key, (unsigned long long)__double_as_longlong(v), step_bits);
  }
}
struct ClusterFinal {
  const int32_t* pairs;
  const double* bodies;
  const unsigned long long* step_bits;
  const int *first_any, *first_ns, *first_member, *pair_cnt, *read_later;
  const double* scale;
};
// A cluster without pairs keeps its first particle's last step (:594-596);
// first_member (clusters built on the device) names it, otherwise dt.  A first
// pair with a static body a adds its use only when its body b is read later.
__device__ __forceinline__ double cluster_step_of(int k, float dt, const ClusterFinal& F) {
  double s;
  if (F.step_bits[k] != ~0ull) s = __longlong_as_double((long long)F.step_bits[k]);
  else if (F.first_any[k] != 0x7fffffff) s = F.bodies[40 * (size_t)F.pairs[2 * F.first_any[k]] + 39];
  else if (F.first_member) s = F.bodies[40 * (size_t)F.first_member[k] + 39];
  else s = (double)dt;
  const int p0 = F.first_ns[k];
  if (p0 != 0x7fffffff && F.pair_cnt[p0] > 0) {
    const double* ra = F.bodies + 40 * (size_t)F.pairs[2 * p0];
    const double* rb = F.bodies + 40 * (size_t)F.pairs[2 * p0 + 1];
    if (ra[38] != 0.0 && F.read_later[F.pairs[2 * p0 + 1]]) {
      const double mt = (rb[39] < ra[39]) ? rb[39] : ra[39];
      const double u = mt * F.scale[p0];
      s = (u < s) ? u : s;
    }
  }
  const double hi = (double)dt;
  s = (hi < s) ? hi : s;         // std::min(s, dt)
  return (s < 1e-3) ? 1e-3 : s;  // std::max(1e-3, .)
}
// Cluster steps, and with body_step the per-body steps of bodies in pairs
// (their cluster's step, computed per pair from the same accumulators).
__global__ void k_cluster_final(int n_clusters, float dt, ClusterFinal F, double* out, int n_pairs,
                                const int32_t* cluster_of_pair, double* body_step) {
  const int n = body_step && n_pairs > n_clusters ? n_pairs : n_clusters;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    if (k < n_clusters) out[k] = cluster_step_of(k, dt, F);
    if (body_step && k < n_pairs) {
      const double s = cluster_step_of(cluster_of_pair[k], dt, F);
      body_step[F.pairs[2 * k]] = s;
      body_step[F.pairs[2 * k + 1]] = s;
    }
  }
}

#include "d2_learned.hpp"
#include "d2_broad.hpp"

// Body future states: future = current.extrapolate(step).
// skip_static: static bodies keep their future state (PDE_explicit.cpp:49-56).
__global__ void k_project(int n, double* bodies, const double* step, int skip_static) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double* r = bodies + 40 * (size_t)i;
    if (skip_static && r[38] != 0.0) continue;
    body_state f = extrapolate(load_state(r), step[i], r + 28);
    store_state(f, r + 14);
  }
}

// ------------------------------------------- sequential impulses (the solver)
// After a filtered step: the clusters' pair lists, particles and hit counts,
// then a block per cluster, or a lane per cluster where many are small, runs
// SequentialImpulses::solve (d2_solver.hpp).
struct SolveArgs {
  int n_pairs, n_clusters, n_bodies;
  const int32_t* pairs;
  const int32_t* cluster_of_pair;
  const int* kept_cnt;    // per pair: filtered contacts
  const int* pair_off;    // per pair: first contact position
  const int* out_off;     // per pair: first output row (filtered CSR)
  const int* perm;        // contact at each position
  const int* keep;        // kept flag at each position
  const ContactRec* contacts;
  const double* cluster_step;
  const double* body_step;
  double* bodies;
  const double* mass;
  const double* fric;
  double gx, gy, gz;
  int* ccount;  // [n_clusters + 1] pairs per cluster, then their offsets (poff)
  int* chits;   // [n_clusters + 1] hits per cluster, then offsets (hoff)
  int* cfill;   // [n_clusters]
  int* cpart;   // [n_clusters] dynamic particles
  int* cpairs;  // [n_pairs] as placed
  int* cps;     // [n_pairs] in index order
  int* inpair;  // [n_bodies] 1 + the cluster of the body's pairs, 0: in no pair
  int* loc;     // [n_bodies] local particle index of a dynamic body
  int* flag;    // set when a dynamic body's pairs lie in two clusters
  int* status;  // [n_clusters]
  int* ploc;    // [2 n_pairs] local particles of each pair (index order)
  int* phit;    // [n_pairs] first hit of each pair (index order)
  int* hl;      // [hits][2]
  int* ord;     // [hits]
  int* hrow;    // [hits] output row
  int* hpc;     // [hits] contacts of the hit's pair
  int* pbody;   // [2 n_pairs]
  int* hint;    // [hits][6] scratch: the sort, then the schedule
  int* lvlo;    // [hits + n_clusters] schedule: level offsets
  int* cntl;    // [hits] schedule: contacts per level
  int* pint;    // [3][2 n_pairs] + n_clusters: per particle scratch of the schedule
  double* hA;   // [hits][3]
  double* hB;   // [hits][3]
  double* heps; // [hits]
  double* hkey; // [hits] |A - B| / (eps_a + eps_b)
  double* hs;     // [hits][SH]: per cluster its CH records (unless in LDS), then its CC records
  double* ps;     // [2 n_pairs][SP] (unless in LDS)
  int* hist;      // [SV_BINS] clusters by size class
  int small;      // clusters up to this size are k_sv_solve_small's (-1: none)
  double* out;  // [hits][11], cluster-gathered order
  WarmTable warm;
};
// ---- results to the host
// Parts of device memory, end to end (each from a multiple of COPY_PIECE on),
// to mapped host memory: a block per COPY_PIECE bytes of the window [off, end)
// of that sequence.  The block that completes a COPY_SLOT of it stores gen in
// the slot's flag, which the host waits for.
constexpr int COPY_PARTS = 6;
constexpr unsigned long long COPY_PIECE = 32ull << 10, COPY_SLOT = 512ull << 10;
struct CopyJob {
  const unsigned char* src[COPY_PARTS];  // 4-byte aligned
  unsigned long long begin[COPY_PARTS], bytes[COPY_PARTS];
  int n;
  unsigned long long off, end;
  unsigned char* dst;
  int* count;
  unsigned long long* flag;
  unsigned long long gen;
};
__global__ void __launch_bounds__(256) k_copy_out(CopyJob J) {
  const unsigned long long v = J.off + blockIdx.x * COPY_PIECE;
  int i = 0;
#pragma unroll
  for (int k = 1; k < COPY_PARTS; ++k)
    if (k < J.n && J.begin[k] <= v) i = k;
  const unsigned long long at = v - J.begin[i], left = at < J.bytes[i] ? J.bytes[i] - at : 0;
  const int len = (int)(left < COPY_PIECE ? left : COPY_PIECE);
  const unsigned char* src = J.src[i] + at;
  unsigned char* dst = J.dst + (v - J.off);
  const int n16 = ((unsigned long long)src & 15ull) ? 0 : len >> 4;
  const uint4* s16 = reinterpret_cast<const uint4*>(src);
  uint4* d16 = reinterpret_cast<uint4*>(dst);
#pragma unroll 4
  for (int k = threadIdx.x; k < n16; k += 256) d16[k] = s16[k];
  for (int k = (n16 << 4) + 4 * (int)threadIdx.x; k < len; k += 1024)
    *reinterpret_cast<unsigned*>(dst + k) = *reinterpret_cast<const unsigned*>(src + k);
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) {
    const int slot = (int)((v - J.off) / COPY_SLOT);
    const unsigned long long first = J.off + slot * COPY_SLOT, rest = J.end - first;
    const int pieces = (int)(((rest < COPY_SLOT ? rest : COPY_SLOT) + COPY_PIECE - 1) / COPY_PIECE);
    if (atomicAdd(&J.count[slot], 1) == pieces - 1) {
      J.count[slot] = 0;
      __threadfence_system();
      __hip_atomic_store(&J.flag[slot], J.gen, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

__global__ void k_fill_i32(int* p, long long n, int v) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}
__global__ void k_sv_count(SolveArgs A) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < A.n_pairs; p += gridDim.x * blockDim.x) {
    const int k = A.cluster_of_pair[p];
    atomicAdd(&A.ccount[k], 1);
    atomicAdd(&A.chits[k], A.kept_cnt[p]);
    for (int e = 0; e < 2; ++e) {  // a dynamic body belongs to the one cluster of its pairs
      const int b = A.pairs[2 * p + e];
      const int old = atomicCAS(&A.inpair[b], 0, k + 1);
      if (old != 0 && old != k + 1 && A.bodies[40 * (size_t)b + 38] == 0.0) atomicOr(A.flag, 1);
    }
  }
}
// A cluster's size for the choice of its solver: its hits and its pairs.
constexpr int SV_BINS = 6;  // sizes up to 2, 4, 8, 16, 32, above
__device__ __forceinline__ int sv_size(const SolveArgs& A, int k) {
  return (A.ccount[k + 1] - A.ccount[k]) + (A.chits[k + 1] - A.chits[k]);
}
// ccount / chits hold the exclusive offsets here (poff / hoff).  The pairs to
// their clusters, the dynamic bodies to their clusters' particles (which
// particle is which changes no result).
__global__ void k_sv_place(SolveArgs A) {
  int n = A.n_pairs > A.n_bodies ? A.n_pairs : A.n_bodies;
  n = A.n_clusters > n ? A.n_clusters : n;
  for (int p0 = blockIdx.x * blockDim.x; p0 < n; p0 += gridDim.x * blockDim.x) {  // block-uniform
    const int p = p0 + threadIdx.x;
    if (p < A.n_pairs) {
      const int k = A.cluster_of_pair[p];
      A.cpairs[A.ccount[k] + atomicAdd(&A.cfill[k], 1)] = p;
    }
    if (p < A.n_bodies && A.inpair[p] && A.bodies[40 * (size_t)p + 38] == 0.0) {
      const int k = A.inpair[p] - 1, q = atomicAdd(&A.cpart[k], 1);
      A.loc[p] = q;
      A.pbody[2 * (size_t)A.ccount[k] + q] = p;
    }
    if (p0 >= A.n_clusters) continue;
    int bin = -1;
    if (p < A.n_clusters) {
      const int size = sv_size(A, p);
      for (bin = 0; bin < SV_BINS - 1 && size > 2 << bin;) ++bin;
    }
    for (int b = 0; b < SV_BINS; ++b) {
      const unsigned long long m = __ballot(bin == b);
      if (m && lane_id() == 0) atomicAdd(&A.hist[b], __popcll(m));
    }
  }
}
// Hit H (contact position t of the pair with local particles la, lb), as the
// cluster's solve takes it.
__device__ __forceinline__ void sv_take_hit(const SolveArgs& A, size_t H, int t, int la, int lb, int row, int cnt) {
  const ContactRec& c = A.contacts[A.perm[t]];
  for (int j = 0; j < 3; ++j) A.hA[3 * H + j] = c.r[j], A.hB[3 * H + j] = c.r[3 + j];
  A.heps[H] = c.r[6] + c.r[7];
  A.hkey[H] = vlen(sub(v3<double>{c.r[0], c.r[1], c.r[2]}, v3<double>{c.r[3], c.r[4], c.r[5]})) / A.heps[H];
  A.hl[2 * H] = la, A.hl[2 * H + 1] = lb;
  A.hrow[H] = row;
  A.hpc[H] = cnt;
}
// Cluster k's solve, once its nh hits from h0 on and np particles are gathered.
__device__ __forceinline__ ClusterSolve sv_cluster(const SolveArgs& A, int k, int h0, int nh, int p0, int np) {
  ClusterSolve S;
  S.nh = nh, S.np = np;
  S.hA = A.hA + 3 * (size_t)h0, S.hB = A.hB + 3 * (size_t)h0, S.heps = A.heps + h0, S.hl = A.hl + 2 * (size_t)h0;
  S.hpc = A.hpc + h0;
  S.ord = A.ord + h0, S.pbody = A.pbody + 2 * (size_t)p0, S.bodies = A.bodies, S.mass = A.mass, S.fric = A.fric;
  S.t = A.cluster_step[k], S.g = v3<double>{A.gx, A.gy, A.gz}, S.warm = A.warm;
  S.hs = A.hs + (size_t)SH * h0, S.ps = A.ps + (size_t)SP * 2 * p0;
  S.out_h = A.out + 11 * (size_t)h0;
  return S;
}
struct KeyLess {
  const double* k;
  D2_HD bool operator()(int x, int y) const { return k[x] < k[y]; }
};
// Value of the neighbouring lane (lane ^ 1), by DPP (no LDS round trip).
__device__ __forceinline__ double lane_xor1(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0xB1, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0xB1, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
// One cluster's solve after gathering and scheduling.  Contacts sit in slots
// ordered by level (a contact's level is one above the highest level of an
// earlier contact that shares a dynamic particle), so the contacts of a level
// touch different dynamic particles and any order of them gives the
// sequential walk's values.  hit: hit of each slot; cab: its two particles;
// csr: per particle, its contacts' slots (2 slot + side) in sorted order.
struct SvRun {
  double *C, *cold, *P;
  const int *hit, *cab, *lvl_off, *csr, *csr_off;
  int n_lvl, n_dyn;
};
template <int NT> __device__ __forceinline__ bool sv_sync_any(bool v) {
  if (NT == 64) {
    wave_sync_lds();
    return __ballot(v) != 0ull;
  }
  return __syncthreads_or(v ? 1 : 0) != 0;
}
// Both sweeps with NT threads.  A contact takes two lanes, one per side: each
// evaluates its particle's point, velocity and prediction, and the two
// exchange their gaps and speeds by DPP.  Static particles' states never
// change, so they order nothing; their accumulated impulse (the convergence
// test reads it) is summed in sorted order after the sweep.
template <int NT> __device__ __forceinline__ void sv_sweeps(const ClusterSolve& S, const SvRun& R, int tid) {
  const int nh = S.nh, np = S.np;
  const double t = S.t;
  const int side = tid & 1;
  for (int k = tid; k < np; k += NT) st3(R.P + (size_t)SP * k + SP_LAST, ld3(R.P + (size_t)SP * k + SP_IMP));
  sv_sync_any<NT>(false);
  for (int it = 0; it < 1000; ++it) {  // normal pass
    for (int l = 0; l < R.n_lvl; ++l) {
      const int end = R.lvl_off[l + 1];
      for (int i = R.lvl_off[l] + (tid >> 1); i < end; i += NT / 2) {
        double* c = R.C + (size_t)CH * i;
        const int li = R.cab[2 * i + side];
        double* p = R.P + (size_t)SP * li;
        const v3<double> n = ld3(c + CH_N);
        const SvSide s = sv_side(p, ld3(c + CH_WA + 3 * side), n);
        const double odn = lane_xor1(s.dn), ovn = lane_xor1(s.vn);
        double du, doff;
        sv_contact_step(c, side ? s.dn - odn : odn - s.dn, side ? ovn - s.vn : s.vn - ovn, t, du, doff);
        const v3<double> u = scl(sv_neg(n), du), uo = scl(sv_neg(n), doff);
        if (li < R.n_dyn) {
          sv_apply(p, side ? sv_neg(u) : u, side ? sv_neg(uo) : uo, s.arm);
          sv_integrate(p, t);
        } else {
          st3(c + CH_U, u);
        }
      }
      sv_sync_any<NT>(false);
    }
    bool moved = false;
    for (int k = tid; k < np; k += NT) {
      double* p = R.P + (size_t)SP * k;
      if (k >= R.n_dyn) {
        v3<double> imp = ld3(p + SP_IMP);
        for (int e = R.csr_off[k]; e < R.csr_off[k + 1]; ++e) {
          const v3<double> u = ld3(R.C + (size_t)CH * (R.csr[e] >> 1) + CH_U);
          imp = (R.csr[e] & 1) ? sub(imp, u) : add(imp, u);
        }
        st3(p + SP_IMP, imp);
      }
      moved = moved || sv_moved(p);
      st3(p + SP_LAST, ld3(p + SP_IMP));
    }
    if (!sv_sync_any<NT>(moved)) break;
  }
  for (int it = 0; it < 100; ++it) {  // friction pass
    bool moved = false;
    for (int i = tid; i < nh; i += NT)
      if (sv_friction(S, R.hit[i], R.C + (size_t)CH * i, R.cold + (size_t)CC * i, R.P + (size_t)SP * R.cab[2 * i],
                      R.P + (size_t)SP * R.cab[2 * i + 1], it & 1))
        moved = true;
    moved = sv_sync_any<NT>(moved);
    for (int k = tid; k < R.n_dyn; k += NT) {
      double* p = R.P + (size_t)SP * k;
      SvAcc a = sv_acc(p);
      for (int e = R.csr_off[k]; e < R.csr_off[k + 1]; ++e)
        sv_friction_apply(a, R.C + (size_t)CH * (R.csr[e] >> 1), R.csr[e] & 1, it & 1);
      sv_acc_store(a, p);
      sv_integrate(p, t);
    }
    sv_sync_any<NT>(false);
    if (!moved) break;
  }
}
// Clusters up to these sizes run from LDS (74 KB, two blocks per CU), larger
// ones from global scratch.
constexpr int SV_CAPH = 192, SV_CAPP = 64;
struct SvLds {
  double C[SV_CAPH * CH];
  double P[SV_CAPP * SP];
  int cab[2 * SV_CAPH], lvl[SV_CAPH], slot[SV_CAPH], csr[2 * SV_CAPH], lvl_off[SV_CAPH + 1], csr_off[SV_CAPP + 1];
};
// Setup, sweeps and results of a gathered, sorted cluster whose schedule
// arrays are at the given pointers (LDS or global).  Returns the status.
__device__ __forceinline__ bool sv_solve_block(const ClusterSolve& S, double* C, double* cold, double* P, int* cab,
                                               int* lvl, int* slot, int* csr, int* lvl_off, int* csr_off, int* last,
                                               int* cur, int* cntl, int n_dyn, int* s_misc, bool lds) {
  const int tid = threadIdx.x, lane = lane_id(), nh = S.nh, np = S.np;
  // contacts per particle -> csr offsets
  for (int k = tid; k <= np; k += blockDim.x) csr_off[k] = 0;
  for (int k = tid; k < nh; k += blockDim.x) cntl[k] = 0;
  __syncthreads();
  for (int c = tid; c < nh; c += blockDim.x) {
    const int h = S.ord[c];
    atomicAdd(&csr_off[S.hl[2 * h]], 1), atomicAdd(&csr_off[S.hl[2 * h + 1]], 1);
  }
  __syncthreads();
  int base = 0;
  for (int k0 = 0; k0 < np; k0 += blockDim.x) {
    const int k = k0 + tid;
    int tot;
    const int ex = block_scan(k < np ? csr_off[k] : 0, tot);
    if (k < np) csr_off[k] = base + ex, cur[k] = base + ex, last[k] = 0;
    base += tot;
  }
  if (tid == 0) csr_off[np] = base;
  __syncthreads();
  // levels and csr entries, contact by contact (one lane; the particles'
  // last levels and cursors are in LDS up to 5000 particles)
  if (tid < 64) {
    int n_lvl = 0;
    for (int c0 = 0; c0 < nh; c0 += 64) {
      const int cc = c0 + lane < nh ? c0 + lane : c0;
      const int h = S.ord[cc], va = S.hl[2 * h], vb = S.hl[2 * h + 1];
      const int m = nh - c0 < 64 ? nh - c0 : 64;
      for (int i = 0; i < m; ++i) {
        const int a = rl(va, i), b = rl(vb, i), c = c0 + i;
        if (lane == 0) {
          const int la = a < n_dyn ? last[a] : 0, lb = b < n_dyn ? last[b] : 0;
          const int lv = la > lb ? la : lb;
          if (a < n_dyn) last[a] = lv + 1;
          if (b < n_dyn) last[b] = lv + 1;
          const int ea = cur[a];
          cur[a] = ea + 1;
          const int eb = cur[b];
          cur[b] = eb + 1;
          csr[ea] = 2 * c, csr[eb] = 2 * c + 1;
          const int at = cntl[lv];
          cntl[lv] = at + 1;
          lvl[c] = lv, slot[c] = at;
          n_lvl = lv + 1 > n_lvl ? lv + 1 : n_lvl;
        }
      }
    }
    if (lane == 0) s_misc[0] = n_lvl;
  }
  __syncthreads();
  const int n_lvl = s_misc[0];
  int lbase = 0, wide = 0;
  for (int k0 = 0; k0 < n_lvl; k0 += blockDim.x) {
    const int k = k0 + tid;
    int tot;
    const int v = k < n_lvl ? cntl[k] : 0;
    const int ex = block_scan(v, tot);
    if (k < n_lvl) lvl_off[k] = lbase + ex;
    wide = v > wide ? v : wide;
    lbase += tot;
  }
  if (tid == 0) lvl_off[n_lvl] = lbase;
  wide = __syncthreads_or(wide > 32 ? 1 : 0);
  for (int c = tid; c < nh; c += blockDim.x) slot[c] += lvl_off[lvl[c]];
  __syncthreads();
  int* hit = lvl;  // the levels are not read again
  for (int e = tid; e < 2 * nh; e += blockDim.x) csr[e] = 2 * slot[csr[e] >> 1] + (csr[e] & 1);
  for (int c = tid; c < nh; c += blockDim.x) {
    const int h = S.ord[c], i = slot[c];
    hit[i] = h, cab[2 * i] = S.hl[2 * h], cab[2 * i + 1] = S.hl[2 * h + 1];
  }
  __syncthreads();  // (also: last, cur and cntl may share C's and P's memory)
  bool bad = false;
  for (int i = tid; i < nh; i += blockDim.x)
    bad = !sv_contact_setup(S, hit[i], C + (size_t)CH * i, cold + (size_t)CC * i) || bad;
  if (__syncthreads_or(bad ? 1 : 0)) return false;
  for (int k = tid; k < np; k += blockDim.x) {
    double* p = P + (size_t)SP * k;
    sv_particle_setup(S, S.pbody[k], p);
    SvAcc a = sv_acc(p);
    for (int e = csr_off[k]; e < csr_off[k + 1]; ++e) sv_warm_apply(a, C + (size_t)CH * (csr[e] >> 1), csr[e] & 1);
    sv_acc_store(a, p);
    if (k < n_dyn) sv_predict(p, S.t);
  }
  __syncthreads();
  for (int i = tid; i < nh; i += blockDim.x)
    sv_contact_turn(C + (size_t)CH * i, cold + (size_t)CC * i, P + (size_t)SP * cab[2 * i],
                    P + (size_t)SP * cab[2 * i + 1]);
  __syncthreads();
  if (nh > 0) {
    const SvRun R{C, cold, P, hit, cab, lvl_off, csr, csr_off, n_lvl, n_dyn};
    // levels of at most 32 contacts fit one wavefront, which needs no
    // barriers; the block's other wavefronts wait for the end
    if (lds && !wide) {
      if (tid < 64) sv_sweeps<64>(S, R, tid);
    } else {
      sv_sweeps<256>(S, R, tid);
    }
  }
  __syncthreads();
  for (int k = tid; k < n_dyn; k += blockDim.x)
    sv_store_future(P + (size_t)SP * k, S.bodies + 40 * (size_t)S.pbody[k]);
  for (int i = tid; i < nh; i += blockDim.x) {
    sv_store_out(C + (size_t)CH * i, cold + (size_t)CC * i, S.out_h + 11 * (size_t)hit[i]);
    // warm store: each body pair keeps its last contact's impulse (the last
    // of a's contacts, in sorted order, with b at the other end)
    const int a = cab[2 * i], b = cab[2 * i + 1];
    const int k = a < n_dyn ? a : b, o = a < n_dyn ? b : a;
    for (int e = csr_off[k + 1] - 1; e >= csr_off[k]; --e) {
      const int j = csr[e] >> 1;
      if (cab[2 * j + ((csr[e] & 1) ^ 1)] != o) continue;
      if (j == i) warm_put(S.warm, warm_key(S.pbody[a], S.pbody[b]), C[(size_t)CH * i + CH_IMP]);
      break;
    }
  }
  return true;
}
// One block per cluster.  The cluster's pairs in index order (the order its
// interactions were gathered in, separate_clusters.cpp:405-434), its hits per
// pair in the filtered order (PDE_explicit.cpp:77-95), the std::sort order of
// the hits by Contact::operator< (contact.h:14-18), then the solve.
//
// Bound by the latency of the normal pass's chain: a sweep is as many
// dependent steps as there are levels (about 12 for 80 contacts among 32
// bodies), each one contact update of FP64 arithmetic and LDS round trips.
// One thread per cluster walking global memory took 125.2 ms for 24 clusters
// of 32 bodies; with levels, two lanes per contact, the state in LDS and the
// rotations hoisted the whole step with that solve takes 6.8 ms (128.7 before),
// bit for bit the same.
__global__ void __launch_bounds__(256) k_sv_solve(SolveArgs A) {
  __shared__ SvLds L;
  __shared__ int s_misc[8];
  __shared__ int s_np;
  const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
  for (int k = blockIdx.x; k < A.n_clusters; k += gridDim.x) {
    if (sv_size(A, k) <= A.small) continue;
    const int p0 = A.ccount[k], np_k = A.ccount[k + 1] - p0;
    const int h0 = A.chits[k], nh = A.chits[k + 1] - h0;
    const int* cu = A.cpairs + p0;
    int* cp = A.cps + p0;
    // pairs in index order: by rank, or (long lists) from one pass over all pairs
    if (np_k <= 1024) {
      for (int i = tid; i < np_k; i += blockDim.x) {
        const int x = cu[i];
        int r = 0;
        for (int j = 0; j < np_k; ++j) r += cu[j] < x ? 1 : 0;
        cp[r] = x;
      }
    } else {
      int at = 0;
      for (int q0 = 0; q0 < A.n_pairs; q0 += blockDim.x) {
        const int q = q0 + tid;
        const bool mine = q < A.n_pairs && A.cluster_of_pair[q] == k;
        int tot;
        const int ex = block_scan(mine ? 1 : 0, tot);
        if (mine) cp[at + ex] = q;
        at += tot;
      }
    }
    const int n_dyn = A.cpart[k];
    int* pb = A.pbody + 2 * (size_t)p0;
    if (tid == 0) s_np = n_dyn;
    __syncthreads();
    // the pairs' first hits and local particles; a static body is one
    // particle per cluster it touches, listed after the dynamic ones
    int at = 0;
    for (int i0 = 0; i0 < np_k; i0 += blockDim.x) {
      const int i = i0 + tid;
      const int p = i < np_k ? cp[i] : -1;
      int tot;
      const int ex = block_scan(p >= 0 ? A.kept_cnt[p] : 0, tot);
      if (p >= 0) A.phit[p0 + i] = at + ex;
      at += tot;
      for (int e = 0; e < 2; ++e) {
        const int b = p >= 0 ? A.pairs[2 * p + e] : 0;
        bool open = false;
        if (p >= 0) {
          if (A.bodies[40 * (size_t)b + 38] == 0.0) A.ploc[2 * (size_t)(p0 + i) + e] = A.loc[b];
          else open = true;
        }
        for (;;) {  // one static body joins the list per round
          const int n_now = s_np;
          for (int q = n_dyn; open && q < n_now; ++q)
            if (pb[q] == b) A.ploc[2 * (size_t)(p0 + i) + e] = q, open = false;
          if (tid == 0) s_misc[1] = 0x7fffffff;
          __syncthreads();
          if (open) atomicMin(&s_misc[1], b);
          __syncthreads();
          const int add = s_misc[1];
          if (add == 0x7fffffff) break;
          if (tid == 0) pb[n_now] = add, s_np = n_now + 1;
          __syncthreads();
        }
        __syncthreads();
      }
    }
    const int np = s_np;
    __syncthreads();
    // the hits, one pair per wavefront at a time
    for (int i = w; i < np_k; i += (int)(blockDim.x >> 6)) {
      const int p = cp[i], la = A.ploc[2 * (size_t)(p0 + i)], lb = A.ploc[2 * (size_t)(p0 + i) + 1];
      const int b = A.pair_off[p], e = A.pair_off[p + 1], row = A.out_off[p], cnt = A.kept_cnt[p];
      int n = 0;
      for (int t0 = b; t0 < e; t0 += 64) {
        const int t = t0 + lane;
        const bool take = t < e && A.keep[t] != 0;
        const unsigned long long m = __ballot(take);
        if (take) {
          const int q = n + __popcll(m & lanes_below());
          sv_take_hit(A, (size_t)h0 + A.phit[p0 + i] + q, t, la, lb, row + q, cnt);
        }
        n += __popcll(m);
      }
    }
    if (tid == 0) s_misc[0] = 0;
    __syncthreads();
    // std::sort's order: ranks of the keys by counting over tiles in LDS, and
    // the introsort replay where keys tie
    const double* key = A.hkey + h0;
    int* ord = A.ord + h0;
    int* wi = A.hint + 6 * (size_t)h0;
    const bool lds = nh <= SV_CAPH && np <= SV_CAPP;
    constexpr int TILE = 2048;  // keys per tile, in L.C
    bool tie = false, nan = false;
    for (int q0 = 0; q0 < nh; q0 += blockDim.x) {
      const int i = q0 + tid;
      const double x = key[i < nh ? i : 0];
      int r = 0, eq = 0;
      for (int t0 = 0; t0 < nh; t0 += TILE) {
        const int m = nh - t0 < TILE ? nh - t0 : TILE;
        __syncthreads();
        for (int j = tid; j < m; j += blockDim.x) L.C[j] = key[t0 + j];
        __syncthreads();
        for (int j = 0; j < m; ++j) {
          const double y = L.C[j];
          r += y < x ? 1 : 0, eq += y == x ? 1 : 0;
        }
      }
      if (i < nh) wi[i] = r, tie = tie || eq > 1, nan = nan || !(x == x);
    }
    tie = __syncthreads_or(tie ? 1 : 0);
    nan = __syncthreads_or(nan ? 1 : 0);
    if (!tie && !nan) {
      for (int i = tid; i < nh; i += blockDim.x) ord[wi[i]] = i;
    } else {
      for (int i = tid; i < nh; i += blockDim.x) ord[i] = i;
      __syncthreads();
      if (nan) {  // keys without an order: the sequential sort itself
        if (tid == 0) StdSort<KeyLess>{ord, KeyLess{key}}.sort(0, nh);
      } else if (lds) {  // (rk, apos, bpos, mark, segs in LDS)
        for (int i = tid; i < nh; i += blockDim.x) L.lvl[i] = wi[i], L.slot[i] = i;
        __syncthreads();
        block_std_sort(nh, L.slot, L.lvl, L.csr, L.csr + SV_CAPH, L.lvl_off, L.cab, s_misc + 2, blk_segs(nh));
        for (int i = tid; i < nh; i += blockDim.x) ord[i] = L.slot[i];
      } else {
        block_std_sort(nh, ord, wi, wi + nh, wi + 2 * (size_t)nh, wi + 3 * (size_t)nh, wi + 4 * (size_t)nh, s_misc + 2,
                       blk_segs(nh));
      }
    }
    __syncthreads();
    const ClusterSolve S = sv_cluster(A, k, h0, nh, p0, np);
    double* cold = S.hs + (size_t)CH * nh;
    // during the schedule the particles' ints share C's memory, the level
    // counts P's (both are filled only after it)
    int* ci = reinterpret_cast<int*>(L.C);
    bool ok;
    if (lds) {
      ok = sv_solve_block(S, L.C, cold, L.P, L.cab, L.lvl, L.slot, L.csr, L.lvl_off, L.csr_off, ci, ci + SV_CAPP,
                          reinterpret_cast<int*>(L.P), n_dyn, s_misc, true);
    } else {
      constexpr int CI = 5000, PI = 5000;  // ints that fit: 2 x 5000 in C, 5000 in P
      static_assert(sizeof(L.C) >= 2 * CI * sizeof(int) && sizeof(L.P) >= PI * sizeof(int) &&
                        SV_CAPH * CH >= TILE, "schedule scratch in LDS");
      int* pi = A.pint + 3 * 2 * (size_t)p0 + k;  // [np + 1] csr offsets, [np] levels, [np] cursors
      ok = sv_solve_block(S, S.hs, cold, S.ps, wi + 4 * (size_t)nh, wi,
                          wi + nh, wi + 2 * (size_t)nh, A.lvlo + h0 + k, pi, np <= CI ? ci : pi + np + 1,
                          np <= CI ? ci + CI : pi + 2 * (size_t)np + 1,
                          nh <= PI ? reinterpret_cast<int*>(L.P) : A.cntl + h0, n_dyn, s_misc, false);
    }
    if (tid == 0) A.status[k] = ok ? 1 : 0;
    __syncthreads();  // LDS is reused by the next cluster
  }
}
// The clusters of size A.small at most, one lane each: gathered, sorted and
// walked contact by contact.
__global__ void __launch_bounds__(64) k_sv_solve_small(SolveArgs A) {
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < A.n_clusters; k += gridDim.x * blockDim.x) {
    if (sv_size(A, k) > A.small) continue;
    const int p0 = A.ccount[k], np_k = A.ccount[k + 1] - p0;
    const int h0 = A.chits[k], nh = A.chits[k + 1] - h0;
    int* cp = A.cps + p0;
    int* pb = A.pbody + 2 * (size_t)p0;
    const int n_dyn = A.cpart[k];
    int np = n_dyn, n = 0;
    for (int i = 0; i < np_k; ++i) {  // the pairs in index order
      const int x = A.cpairs[p0 + i];
      int at = i;
      for (; at > 0 && cp[at - 1] > x; --at) cp[at] = cp[at - 1];
      cp[at] = x;
    }
    for (int i = 0; i < np_k; ++i) {
      const int p = cp[i];
      int l[2];
      for (int e = 0; e < 2; ++e) {  // a static body: one particle per cluster it touches
        const int b = A.pairs[2 * p + e];
        if (A.bodies[40 * (size_t)b + 38] == 0.0) {
          l[e] = A.loc[b];
        } else {
          int q = n_dyn;
          while (q < np && pb[q] != b) ++q;
          if (q == np) pb[np++] = b;
          l[e] = q;
        }
      }
      int row = A.out_off[p];
      for (int t = A.pair_off[p]; t < A.pair_off[p + 1]; ++t) {
        if (!A.keep[t]) continue;
        sv_take_hit(A, (size_t)h0 + n, t, l[0], l[1], row++, A.kept_cnt[p]);
        A.ord[h0 + n] = n;
        ++n;
      }
    }
    StdSort<KeyLess>{A.ord + h0, KeyLess{A.hkey + h0}}.sort(0, nh);
    A.status[k] = solve_cluster(sv_cluster(A, k, h0, nh, p0, np)) ? 1 : 0;
  }
}
// Bodies in no pair: a cluster of their own without contacts (gravity only).
__global__ void k_sv_free(SolveArgs A) {
  for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < A.n_bodies; b += gridDim.x * blockDim.x) {
    double* r = A.bodies + 40 * (size_t)b;
    if (A.inpair[b] || r[38] != 0.0) continue;
    const double t = A.body_step[b];
    const v3<double> g{A.gx, A.gy, A.gz}, z{0.0, 0.0, 0.0};
    const SolverState u = sv_update(sv_load(r + 14), t, scl(sclL(A.mass[b], g), t), z, z, z, A.mass[b], r + 28);
    r[14] = u.q.w, r[15] = u.q.x, r[16] = u.q.y, r[17] = u.q.z;
    r[18] = u.x.x, r[19] = u.x.y, r[20] = u.x.z, r[21] = u.v.x, r[22] = u.v.y, r[23] = u.v.z;
    r[24] = u.L.x, r[25] = u.L.y, r[26] = u.L.z;
  }
}
// Per-hit results to the filtered CSR rows.
__global__ void k_sv_scatter(long long n, const int* hrow, const double* in, double* out) {
  for (long long h = (long long)blockIdx.x * blockDim.x + threadIdx.x; h < n; h += (long long)gridDim.x * blockDim.x)
    for (int j = 0; j < 11; ++j) out[11 * (size_t)hrow[h] + j] = in[11 * (size_t)h + j];
}
// PDEExplicit::step's tail (PDE_explicit.cpp:117-131) for the dynamic bodies:
// current <- future, last step <- the body's step, future <- extrapolate.
__global__ void k_commit(int n, double* bodies, const double* step) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double* r = bodies + 40 * (size_t)i;
    if (r[38] != 0.0) continue;
    for (int j = 0; j < 14; ++j) r[j] = r[14 + j];
    r[39] = step[i];
    store_state(extrapolate(load_state(r), step[i], r + 28), r + 14);
  }
}
// Re-inserts the keys of an old warm table into a new one.
__global__ void k_warm_rehash(const unsigned long long* keys, const double* vals, long long n, WarmTable W) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    if (keys[i] != WARM_EMPTY) warm_put(W, keys[i], vals[i]);
}

}  // namespace d2

// =========================================================================
// Host side: context and the C ABI.
// =========================================================================
using namespace d2;

namespace {

const char* kKernelNames[] = {"setup", "soup_cull", "soup_point", "soup_edge", "soup_reduce", "expand",
                              "leaf_point", "leaf_edge", "tri_mask", "tri_enum", "tri_dist", "post", "post_pairs",
                              "cluster", "gate", "tri_full", "soup_keep", "tri_def"};
// Some launch nothing and only count: K_TRI_ENUM the discrete node pairs
// received (part of k_tri_mask), K_SOUP_POINT, K_LEAF_POINT and K_LEAF_EDGE
// their sub-tests (part of k_ccd_sub, which K_SOUP_EDGE times over all four
// kinds).  K_SOUP_CULL is k_ccd_cull, over both lists.  FP64 contexts run
// K_TRI_FULL (k_tri_full) and K_EXPAND (k_disc_expand) in place of K_TRI_MASK +
// K_TRI_DIST; the other forms expand in the kernels that find the hits.
enum KId { K_SETUP, K_SOUP_CULL, K_SOUP_POINT, K_SOUP_EDGE, K_SOUP_REDUCE, K_EXPAND, K_LEAF_POINT, K_LEAF_EDGE,
           K_TRI_MASK, K_TRI_ENUM, K_TRI_DIST, K_POST, K_POST_PAIRS, K_CLUSTER, K_GATE, K_TRI_FULL, K_SOUP_KEEP, K_TRI_DEF,
           K_NUM };

template <class T> struct DBuf {
  T* p = nullptr;
  size_t n = 0;
};

enum RunKind { RUN_NARROW = 0, RUN_CCD = 1, RUN_STEP = 2, RUN_KINDS = 3 };
constexpr int MAX_SEGMENTS = 3;

// Everything a captured run bakes in besides buffer addresses (a
// reallocation drops every graph).
struct Sig {
  int n_pairs = -1, n_bodies = -1, n_clusters = -1, max_depth = -1, precision = -1, filter = -1;
  float dt = -1.f;
  d2_tune tune{0, 0, 0, 0};
  int levels[2] = {-1, -1};  // graph levels of each phase
  int learned = -1;
  float gate_t = 0.f, gate_s = 0.f;
  int cl_dev = -1;  // clusters built on the device (first members known)
  int big_hulls = -1;  // the gate's certificate has its second launch (k_certify_block)
  unsigned long long grids = 0;  // hash of the per-level launch grids
  bool operator==(const Sig& o) const {
    return grids == o.grids && cl_dev == o.cl_dev && big_hulls == o.big_hulls && levels[0] == o.levels[0] && levels[1] == o.levels[1] && learned == o.learned && gate_t == o.gate_t &&
           gate_s == o.gate_s && n_pairs == o.n_pairs && n_bodies == o.n_bodies && n_clusters == o.n_clusters && max_depth == o.max_depth &&
           precision == o.precision && filter == o.filter && dt == o.dt &&
           tune.chunk_blocks == o.tune.chunk_blocks && tune.stream_blocks == o.tune.stream_blocks &&
           tune.post_blocks == o.tune.post_blocks;
  }
};
struct Captured {  // one instantiated graph per run kind
  hipGraphExec_t exec = nullptr;
  bool valid = false;
  Sig sig;
};

}  // namespace

struct d2_ctx {
  int device = 0;
  int precision = D2_FP64;
  hipStream_t stream = nullptr;
  std::string err;
  // capacities: node pairs per list, triangle-pair / sub-test items per
  // level, contacts per run, CCD soup items with result slots (15 x 64 B)
  long long cap = 1ll << 22;
  long long cap_items = 1ll << 24;
  long long cap_contacts = 1ll << 22;
  long long cap_res = 1ll << 20;
  bool auto_grow = true;  // grow the capacities and re-run on overflow
  int cus = 256;
  d2_tune tune{1024, 2048, 4096, 3};  // 4, 8, 16 per CU of a 256-CU device; reset at creation
  // trees / bodies
  DBuf<NodeRec> nodes;
  DBuf<double> buckets;
  DBuf<float> fbuckets;  // FP32 form: float corners + eps per triangle (FB_STRIDE), built on first use
  DBuf<float> stris;     // FP32 form: soup_tri planes per triangle (ST_STRIDE), built with fbuckets
  bool fb_ready = false;
  long long n_nodes_total = 0;  // nodes of the uploaded trees
  long long graph_captures = 0, graph_launches = 0;  // graph segments captured / launched (d2_graph_stats)
  DBuf<int32_t> tree_off, body_tree;
  DBuf<double> bodies;
  int n_trees = 0, n_bodies = 0;
  int pair_depth = 0;                       // max over pairs of depth(tree a) + depth(tree b)
  std::vector<int> tree_depth, host_body_tree;
  // pairs and clusters
  DBuf<int32_t> pairs, pair_info, cluster_of_pair;
  unsigned char* stage = nullptr;  // copy_out's pinned window, its slots' flags and counters
  unsigned long long* stage_flag = nullptr;
  unsigned long long stage_gen = 0;
  int* stage_cnt = nullptr;
  DBuf<double> max_time, pair_rec;
  DBuf<float> pair_f;
  int n_pairs = 0, n_clusters = 0;
  // a pair list describes the uploaded bodies: a tree upload or a body upload
  // of another count invalidates it (and its clusters) until pairs come again
  bool pairs_valid = false;
  // work
  DBuf<NP> soup_list[2], conn_list[2];  // level l reads [l & 1] and writes [(l + 1) & 1]
  DBuf<Item> items, pt_items, ee_items, lpt_items, lee_items;
  DBuf<DItem> ditems;
  DBuf<DItem> ditems_def;  // FP32 form: deferred items of inner node pairs
  DBuf<double> res;
  DBuf<unsigned> res_mask;  // FP32 form: per soup item, the slots its FP32 culls keep
  DBuf<int> np_hit, np_hit2, exp_desc;
  DBuf<ContactRec> contacts;
  DBuf<unsigned long long> cnt, lvl;
  DBuf<unsigned long long> pass_min_s, pass_min_c;
  DBuf<int> pass_flag_s, pass_flag_c;
  DBuf<double> min_time, scale;
  // post
  DBuf<int> pair_cnt, pair_off, pair_fill, perm, keep, kept_cnt, out_off, big, huge, n_big, scan_part;
  DBuf<int> hscratch;  // 6 x contact capacity: the filter of pairs above every LDS capacity
  DBuf<float> nbound;  // per node: leaf box lo, hi (body frame), largest leaf eps + slack, sphere r, centre, 0
  DBuf<uint8_t> kid_inner;  // per node: which children are inner nodes (bit c: child c)
  bool prune_on = true;  // skip node pairs whose leaf triangles are provably apart
  bool defer_on = true;  // FP32 form: an inner node pair's items after its first go to k_tri_def
  // the solver (d2_solve): per-body mass and friction, per-cluster and per-hit scratch, the warm store
  DBuf<double> sv_mass, sv_fric;
  DBuf<int> sv_ccount, sv_chits, sv_poff, sv_hoff, sv_cfill, sv_cpairs, sv_inpair, sv_loc, sv_status, sv_flag;
  DBuf<int> sv_hl, sv_ord, sv_hrow, sv_hpc, sv_pbody, sv_cpart, sv_cps, sv_ploc, sv_phit, sv_hint, sv_lvlo, sv_cntl, sv_pint;
  DBuf<double> sv_hA, sv_hB, sv_heps, sv_hkey, sv_hs, sv_ps, sv_out, sv_out_csr;
  DBuf<unsigned long long> warm_keys, warm_used;
  DBuf<double> warm_vals;
  int last_kind = -1;         // kind of the last finished run
  long long run_serial = 0;   // finished runs
  long long solved_serial = -1;  // run_serial the last d2_solve worked on
  long long solved_hits = 0;
  DBuf<int32_t> out_i;
  DBuf<double> out_r;
  // clusters
  DBuf<unsigned long long> step_bits;
  DBuf<int> first_any, first_ns, read_later;
  DBuf<double> cluster_step, body_step;
  DBuf<int32_t> tmp_cluster;
  // broad phase (per tree: float AABB of the mesh and bounding radius)
  DBuf<float> tb_box;
  DBuf<double> tb_rad, last_state, bp_R;
  DBuf<int32_t> tree_depth_d, group;
  bool has_groups = false;
  std::vector<int> host_static;
  int n_items = 0, bp_seg = BP_SEG_MIN;
  DBuf<int> bp_statics, bp_item_body, bp_item_seg, bp_item_cnt, bp_item_sorted, bp_item_off, bp_meta, bp_slot,
      bp_rank, bp_counts, bp_start, bp_red;
  DBuf<long long> bp_item_pos;
  DBuf<unsigned long long> bp_keys, bp_fill;
  DBuf<Box8> bp_box, bp_members;
  DBuf<int2> bp_chunk;
  long long bp_cap = 0;
  int* host_red = nullptr;  // pinned: BR_N reductions + pair total
  // clusters built on the device
  DBuf<int> cc_parent, cc_label, cc_root, cc_root_off, cc_of_body, cc_first;
  DBuf<long long> cc_tmin;
  DBuf<unsigned long long> cc_smin;
  bool clusters_on_device = false;
  // learned gate
  DBuf<float> tree_radius, tree_eps_out, hv, feat, pred;
  DBuf<int32_t> hv_off;
  bool big_hulls = false;  // some tree's hull has more vertices than k_certify takes
  DBuf<int> cert;  // per pair: 1 = traverse (not certified)
  int gate_phases = 3;       // bit 0: CCD phase, bit 1: discrete phase
  DBuf<float> mlp_w, mlp_m, mlp_v, mlp_wf, mlp_grad;
  DBuf<short> mlp_wb;
  DBuf<float> tr_x, tr_t, tr_part, tr_loss;
  DBuf<int> tr_idx;
  bool mlp_ready = false, learned_on = false, has_max_time = false;
  float gate_t = 1.1f, gate_s = 0.99f;
  long long mlp_step = 0;
  // host mirrors (pinned)
  unsigned long long* host_cnt = nullptr;
  unsigned long long* host_lvl = nullptr;
  long long n_out = 0;
  int last_mode = -1;  // 0 narrow, 1 ccd (per-pair CCD values valid in both after a step)
  bool ccd_valid = false;
  int last_filter = 1;
  bool out_filtered = false;
  // graphs
  bool graph_on = false;
  bool capturing = false;
  Captured graphs[RUN_KINDS][MAX_SEGMENTS];
  int phase_levels[4] = {-1, -1, -1, -1};  // deepest level count seen per phase (narrow, ccd, step ccd, step narrow)
  int graph_levels[2] = {0, 0};             // level counts of the last graph run's phases
  // level sizes of the last run of each phase (0 discrete, 1 CCD): launch
  // grids of the next runs' levels are sized from them
  long long prev_lv[2][MAX_LEVELS + 1][LV_STRIDE] = {};
  bool prev_ok[2] = {false, false};
  long long prev_contacts[2] = {-1, -1};  // contacts of the last run's discrete / CCD phase (-1: none yet)
  // algorithmic-byte accounting (d2_set_touch_stats): bitmaps over (body, node)
  // and bodies, per level and per run; counts per phase and level, then per run
  bool touch_on = false;
  std::vector<int32_t> host_tree_off;
  DBuf<long long> touch_base;
  DBuf<unsigned> touch_lv, touch_run, touch_lvb, touch_runb;
  DBuf<unsigned long long> touch_acc;
  long long touch_words = 0, touch_body_words = 0;
  std::vector<unsigned long long> touch_host;
  // bucket-level entry and standalone filter
  unsigned char* noalloc = nullptr;  // this device's copy of `scratch` (resolved at creation)
  DBuf<int32_t> bk_np, bk_used, bk_out_i;
  DBuf<long long> bk_base, bk_off;
  DBuf<int> bk_count;
  DBuf<ContactRec> bk_hits;
  DBuf<double> bk_out_r;
  DBuf<unsigned long long> bk_counter;
  // profiling
  bool profiling = false;
  long long k_launch[K_NUM] = {};
  double k_ms[K_NUM] = {};
  double k_items[K_NUM] = {};
  std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> pending;
  std::vector<double> pending_items;
};

namespace {

int fail(d2_ctx* c, int code, const std::string& msg) {
  if (c) c->err = msg;
  return code;
}
#define HIPCHK(ctx, expr)                                                                       \
  do {                                                                                          \
    hipError_t e_ = (expr);                                                                     \
    if (e_ != hipSuccess) return fail(ctx, D2_ERR_HIP, std::string(#expr ": ") + hipGetErrorString(e_)); \
  } while (0)
#define RC(expr)            \
  do {                      \
    int rc_ = (expr);       \
    if (rc_) return rc_;    \
  } while (0)

void drop_graphs(d2_ctx* c) {
  for (auto& row : c->graphs)
    for (auto& g : row) {
      if (g.exec) (void)hipGraphExecDestroy(g.exec);
      g = Captured{};
    }
}

// The pair list, its clusters and every result refer to the uploaded bodies:
// forget them when the bodies they index change (runs then fail with
// D2_ERR_STATE until a new pair list is uploaded or built).
void invalidate_pairs(d2_ctx* c) {
  c->pairs_valid = false;
  c->n_pairs = 0;
  c->n_clusters = 0;
  c->clusters_on_device = false;
  c->last_mode = -1;
  c->ccd_valid = false;
}

// (Re)allocation invalidates captured graphs: they hold buffer addresses.
template <class T> int ensure(d2_ctx* c, DBuf<T>& b, size_t n) {
  if (b.n >= n && b.p) return D2_OK;
  if (c->capturing) return fail(c, D2_ERR_STATE, "internal: allocation during graph capture");
  drop_graphs(c);
  if (b.p) HIPCHK(c, hipFree(b.p));
  b.p = nullptr;
  b.n = 0;
  size_t bytes = std::max<size_t>(n, 1) * sizeof(T);
  HIPCHK(c, hipMalloc((void**)&b.p, bytes));
  b.n = std::max<size_t>(n, 1);
  return D2_OK;
}
template <class T> void release(DBuf<T>& b) {
  if (b.p) (void)hipFree(b.p);
  b.p = nullptr;
  b.n = 0;
}

// The segment length of the static bodies' sweeps.  Few statics need short
// segments to fill the chip (3 among 65,536 bodies: 290 us a broad phase with
// 512 bodies a segment, 298 with 4096, 509 with 32768); with many the items
// themselves cost, on the host at each upload and in the kernels' per-item
// arrays (30,000 among 65,536: 4.1 ms of upload and 7.8 ms of broad phase
// with 512, 2.1 and 5.9 ms with 4096).
int bp_segment(const std::vector<int>& statics, int n_bodies) {
  int seg = BP_SEG_MIN;
  for (; seg < BP_SEG_MAX; seg *= 2) {
    long long items = 0;
    for (int a : statics) items += (n_bodies - 1 - a + seg - 1) / seg;
    if (items <= BP_SEG_ITEMS) break;
  }
  return seg;
}

int grid_for(d2_ctx* c, long long threads, int block = 256) {
  long long g = (threads + block - 1) / block;
  long long maxg = (long long)c->cus * 16;
  if (g > maxg) g = maxg;
  if (g < 1) g = 1;
  return (int)g;
}
int chunk_grid(const d2_ctx* c) { return c->tune.chunk_blocks; }
int stream_grid(const d2_ctx* c) { return c->tune.stream_blocks; }

struct Timer {
  d2_ctx* c;
  int id;
  double items;
  hipEvent_t a = nullptr, b = nullptr;
  bool on;
  Timer(d2_ctx* ctx, int k, double n) : c(ctx), id(k), items(n), on(ctx->profiling && !ctx->capturing) {
    if (on) {
      (void)hipEventCreate(&a);
      (void)hipEventCreate(&b);
      (void)hipEventRecord(a, c->stream);
    }
  }
  ~Timer() {
    if (on) {
      (void)hipEventRecord(b, c->stream);
      c->pending.push_back({id, {a, b}});
      c->pending_items.push_back(items);
    }
  }
};

void collect_timers(d2_ctx* c) {
  for (size_t i = 0; i < c->pending.size(); ++i) {
    auto& pe = c->pending[i];
    float ms = 0.f;
    (void)hipEventSynchronize(pe.second.second);
    (void)hipEventElapsedTime(&ms, pe.second.first, pe.second.second);
    c->k_launch[pe.first] += 1;
    c->k_ms[pe.first] += ms;
    c->k_items[pe.first] += c->pending_items[i];
    (void)hipEventDestroy(pe.second.first);
    (void)hipEventDestroy(pe.second.second);
  }
  c->pending.clear();
  c->pending_items.clear();
}

// Launch of one kernel that, when profiling, is timed by events the GPU
// stamps at the kernel's own start and end (no host submission gaps).
template <typename F, typename... Args>
void timed_launch(d2_ctx* c, int kid, F kernel, dim3 grid, dim3 block, Args... args) {
  if (c->profiling && !c->capturing) {
    hipEvent_t a = nullptr, b = nullptr;
    (void)hipEventCreate(&a);
    (void)hipEventCreate(&b);
    hipExtLaunchKernelGGL(kernel, grid, block, 0, c->stream, a, b, 0, args...);
    c->pending.push_back({kid, {a, b}});
    c->pending_items.push_back(0.0);
  } else {
    hipLaunchKernelGGL(kernel, grid, block, 0, c->stream, args...);
  }
}

Dev make_dev(d2_ctx* c, int level, int discrete) {
  Dev D;
  D.nodes = c->nodes.p;
  D.buckets = c->buckets.p;
  D.pair_info = c->pair_info.p;
  D.pair_rec = c->pair_rec.p;
  D.pair_f = c->precision == D2_FP32 ? c->pair_f.p : nullptr;
  D.soup = c->soup_list[level & 1].p;
  D.conn = c->conn_list[level & 1].p;
  D.soup_next = c->soup_list[(level + 1) & 1].p;
  D.conn_next = c->conn_list[(level + 1) & 1].p;
  D.items = c->items.p;
  D.ditems = c->ditems.p;
  D.ditems_def = c->ditems_def.p;
  D.pt_items = c->pt_items.p;
  D.ee_items = c->ee_items.p;
  D.lpt_items = c->lpt_items.p;
  D.lee_items = c->lee_items.p;
  D.res = c->res.p;
  D.res_mask = c->res_mask.p;
  D.np_hit = (level & 1) ? c->np_hit2.p : c->np_hit.p;
  D.np_hit_prev = (level & 1) ? c->np_hit.p : c->np_hit2.p;
  D.exp_desc = c->exp_desc.p;
  D.pair_cnt = c->pair_cnt.p;
  D.contacts = c->contacts.p;
  D.cnt = c->cnt.p;
  D.lvl = c->lvl.p;
  D.pass_min_s = c->pass_min_s.p, D.pass_min_c = c->pass_min_c.p;
  D.pass_flag_s = c->pass_flag_s.p, D.pass_flag_c = c->pass_flag_c.p;
  D.min_time = c->min_time.p;
  D.tree_eps_out = c->tree_eps_out.p;
  D.fbuckets = c->fbuckets.p;
  D.stris = c->stris.p;
  D.nbound = c->nbound.p;
  D.kid_inner = c->kid_inner.p;
  D.prune = c->prune_on && !c->touch_on && c->nbound.p ? 1 : 0;  // accounting runs walk the reference's node pairs
  D.defer = c->defer_on && c->precision == D2_FP32 && c->ditems_def.p ? 1 : 0;  // per level: enqueue_level
  D.box_test = 1;
  D.conn_blocks = 0;
  D.body_tree = c->body_tree.p;
  D.fp32 = c->precision == D2_FP32 ? 1 : 0;
  D.n_pairs = c->n_pairs;
  D.cap_np = c->cap;
  D.cap_items = c->cap_items;
  D.cap_res = c->cap_res;
  D.cap_contacts = c->cap_contacts;
  D.level = level;
  D.discrete = discrete;
  return D;
}

// A node pair's level is the sum of its nodes' depths, so a pair list needs
// (deepest depth sum) + 1 levels.
int level_budget(const d2_ctx* c) { return std::min(MAX_LEVELS, c->pair_depth + 1); }

// Every buffer a run touches, sized before any launch (and before capture).
int prepare(d2_ctx* c) {
  const size_t np = (size_t)std::max(c->n_pairs, 1);
  const size_t g = (size_t)chunk_grid(c);
  if (c->precision == D2_FP32) RC(ensure(c, c->pair_f, np * std::max((int)PF_STRIDE, (int)CF_STRIDE)));
  for (int k = 0; k < 2; ++k) {
    RC(ensure(c, c->soup_list[k], c->cap));
    RC(ensure(c, c->conn_list[k], c->cap));
  }
  RC(ensure(c, c->items, c->cap_res)); RC(ensure(c, c->lpt_items, c->cap_items));
  RC(ensure(c, c->lee_items, c->cap_items));
  if (c->precision == D2_FP32) {  // FP64: k_tri_full keeps no item list, and every soup sub-test runs
    RC(ensure(c, c->pt_items, c->cap_items));
    RC(ensure(c, c->ee_items, c->cap_items));
    RC(ensure(c, c->ditems, c->cap_items));
    RC(ensure(c, c->ditems_def, c->cap_items));
  }
  RC(ensure(c, c->np_hit, c->cap)); RC(ensure(c, c->np_hit2, c->cap)); RC(ensure(c, c->exp_desc, c->cap));
  RC(ensure(c, c->contacts, c->cap_contacts)); RC(ensure(c, c->cnt, C_COUNT));
  RC(ensure(c, c->hscratch, 6 * (size_t)c->cap_contacts));
  RC(ensure(c, c->lvl, (size_t)2 * (MAX_LEVELS + 1) * LV_STRIDE));
  RC(ensure(c, c->res, (size_t)c->cap_res * RES_SLOTS * 8));
  if (c->precision == D2_FP32) RC(ensure(c, c->res_mask, (size_t)c->cap_res));
  if (c->precision == D2_FP32 && !c->fb_ready) {  // the float copy of the buckets, once per tree upload
    const size_t nodes = (size_t)c->n_nodes_total;
    RC(ensure(c, c->fbuckets, nodes * 8 * FB_STRIDE));
    RC(ensure(c, c->stris, nodes * 8 * ST_STRIDE));
    hipLaunchKernelGGL(k_bucket_f32, dim3(grid_for(c, (long long)nodes * 8)), dim3(256), 0, c->stream, c->buckets.p,
                       (long long)nodes, c->fbuckets.p, c->stris.p);
    HIPCHK(c, hipGetLastError());
    c->fb_ready = true;
  }
  RC(ensure(c, c->pass_min_s, np)); RC(ensure(c, c->pass_min_c, np)); RC(ensure(c, c->pass_flag_s, np));
  RC(ensure(c, c->pass_flag_c, np)); RC(ensure(c, c->min_time, np)); RC(ensure(c, c->scale, np));
  RC(ensure(c, c->pair_cnt, np + 1)); RC(ensure(c, c->pair_off, np + 1)); RC(ensure(c, c->pair_fill, np));
  RC(ensure(c, c->kept_cnt, np + 1)); RC(ensure(c, c->out_off, np + 1)); RC(ensure(c, c->big, np));
  RC(ensure(c, c->n_big, 2)); RC(ensure(c, c->huge, np)); RC(ensure(c, c->perm, c->cap_contacts)); RC(ensure(c, c->keep, c->cap_contacts));
  RC(ensure(c, c->scan_part, g));
  if (c->learned_on) {
    RC(ensure(c, c->feat, np * MLP_IN)); RC(ensure(c, c->pred, np * MLP_OUT)); RC(ensure(c, c->cert, np));
  }
  return D2_OK;
}

// Exclusive scan of n (host-known) ints on the context stream.
void scan_host_n(d2_ctx* c, const int* in, int* out, long long n, unsigned long long* total_dst) {
  if (n <= SCAN_SMALL) {
    hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, c->stream, in, out, n, total_dst);
    return;
  }
  const int g = chunk_grid(c);
  hipLaunchKernelGGL(k_scan_part, dim3(g), dim3(256), 0, c->stream, in, n, c->scan_part.p);
  hipLaunchKernelGGL(k_scan_apply, dim3(g), dim3(256), 0, c->stream, in, out, n, c->scan_part.p, total_dst);
}

// One breadth-first level of a phase.
// Launch grids of one level: the tuned block counts are the caps; a level
// that was small in the last run of its phase gets fewer blocks (at least 16,
// in powers of two, with 25% headroom): the culling kernels keep about one
// node pair per wavefront (they are latency-bound on small levels, so as many
// wavefronts as there is work), the others one unit per thread.
// Any grid gives the same results; only the time changes.
// def: k_tri_def's grid, 0 where the level defers nothing; box: whether
// k_tri_mask runs the face-axis box test.  Both pay on large levels only (on
// small ones the extra launch and the extra dependent load cost more than
// they save), judged by the last run's sizes of the level: at least 64 K
// items, at least 256 K node pairs.
struct LevelGrids {
  int cull, conn, stream, sub, def, box, quad;
};
LevelGrids level_grids(const d2_ctx* c, int discrete, int level) {
  LevelGrids g{chunk_grid(c), chunk_grid(c), stream_grid(c), 2 * stream_grid(c), stream_grid(c), 1, 0};
  const int ph = discrete ? 0 : 1;
  if (!c->prev_ok[ph] || level > MAX_LEVELS) return g;
  const long long* v = c->prev_lv[ph][level];
  const long long ns = v[LV_SOUP];
  auto fit = [](long long n, long long per, int hi) {
    long long b = 16;
    while (b < hi && b * per < n + n / 4) b <<= 1;
    return (int)std::min<long long>(b, hi);
  };
  g.cull = fit(ns, 4, g.cull);
  g.conn = fit(v[LV_CONN], 4, g.conn);
  if (discrete && v[LV_ITEMS] <= QUAD_ITEMS) g.quad = 1;
  g.stream = fit(v[LV_ITEMS], g.quad ? 64 : 256, g.stream);
  if (discrete) {
    g.def = v[LV_ITEMS] + v[LV_DEF] >= (1ll << 16) ? fit(v[LV_DEF], 256, g.def) : 0;
    g.box = ns >= (1ll << 18) ? 1 : 0;
  } else {
    const long long soup = c->precision == D2_FP32 ? v[LV_SPT] + v[LV_SEE] : 15 * v[LV_ITEMS];
    g.sub = fit(soup + v[LV_PT] + v[LV_EE], 256, g.sub);
  }
  return g;
}
unsigned long long grids_hash(const d2_ctx* c, int discrete, int levels) {
  unsigned long long h = 1469598103934665603ull;
  for (int l = 0; l < levels; ++l) {
    const LevelGrids g = level_grids(c, discrete, l);
    for (int f : {g.cull, g.conn, g.stream, g.sub, g.def, 2 * g.quad + g.box})
      h = (h ^ (unsigned long long)f) * 1099511628211ull;
  }
  return h;
}
// Accounting runs (eager only): counts the (body, node) records this level
// tests into touch_acc[phase][level], and marks them in the run's bitmaps.
constexpr int TOUCH_FIELDS = 4;  // inner nodes, leaf nodes, leaf triangles, bodies
constexpr int TOUCH_RUN = 2 * (MAX_LEVELS + 1) * TOUCH_FIELDS;  // offset of the run's union
void touch_level(d2_ctx* c, int level, int discrete) {
  (void)hipMemsetAsync(c->touch_lv.p, 0, sizeof(unsigned) * c->touch_words, c->stream);
  (void)hipMemsetAsync(c->touch_lvb.p, 0, sizeof(unsigned) * c->touch_body_words, c->stream);
  TouchArgs T;
  T.soup = c->soup_list[level & 1].p, T.conn = c->conn_list[level & 1].p, T.lvl = c->lvl.p;
  T.np_hit_prev = (level & 1) ? c->np_hit.p : c->np_hit2.p;
  T.pair_info = c->pair_info.p, T.node_base = c->touch_base.p;
  T.lv_nodes = c->touch_lv.p, T.run_nodes = c->touch_run.p, T.lv_bodies = c->touch_lvb.p, T.run_bodies = c->touch_runb.p;
  T.cap_np = c->cap, T.level = level, T.discrete = discrete;
  hipLaunchKernelGGL(k_touch, dim3(grid_for(c, c->cap)), dim3(256), 0, c->stream, T);
  unsigned long long* out = c->touch_acc.p + ((discrete ? 0 : 1) * (MAX_LEVELS + 1) + level) * TOUCH_FIELDS;
  hipLaunchKernelGGL(k_touch_count, dim3(grid_for(c, c->touch_words)), dim3(256), 0, c->stream, c->touch_lv.p,
                     c->touch_words, c->touch_lvb.p, c->touch_body_words, c->touch_base.p, c->n_bodies,
                     c->body_tree.p, c->tree_off.p, c->nodes.p, out);
}

// Start of an accounting run: the (body, node) numbering of the current
// bodies, cleared bitmaps and counts.
int touch_begin(d2_ctx* c) {
  std::vector<long long> base(c->n_bodies + 1, 0);
  for (int b = 0; b < c->n_bodies; ++b) {
    const int t = c->host_body_tree[b];
    base[b + 1] = base[b] + (c->host_tree_off[t + 1] - c->host_tree_off[t]);
  }
  c->touch_words = std::max<long long>((base[c->n_bodies] + 31) / 32, 1);
  c->touch_body_words = std::max<long long>((c->n_bodies + 31) / 32, 1);
  RC(ensure(c, c->touch_base, base.size()));
  RC(ensure(c, c->touch_lv, c->touch_words)); RC(ensure(c, c->touch_run, c->touch_words));
  RC(ensure(c, c->touch_lvb, c->touch_body_words)); RC(ensure(c, c->touch_runb, c->touch_body_words));
  RC(ensure(c, c->touch_acc, TOUCH_RUN + TOUCH_FIELDS));
  HIPCHK(c, hipMemcpyAsync(c->touch_base.p, base.data(), sizeof(long long) * base.size(), hipMemcpyHostToDevice,
                           c->stream));
  HIPCHK(c, hipMemsetAsync(c->touch_run.p, 0, sizeof(unsigned) * c->touch_words, c->stream));
  HIPCHK(c, hipMemsetAsync(c->touch_runb.p, 0, sizeof(unsigned) * c->touch_body_words, c->stream));
  HIPCHK(c, hipMemsetAsync(c->touch_acc.p, 0, sizeof(unsigned long long) * (TOUCH_RUN + TOUCH_FIELDS), c->stream));
  return D2_OK;
}

// End of an accounting run: the union's counts, and every count to the host.
int touch_end(d2_ctx* c) {
  hipLaunchKernelGGL(k_touch_count, dim3(grid_for(c, c->touch_words)), dim3(256), 0, c->stream, c->touch_run.p,
                     c->touch_words, c->touch_runb.p, c->touch_body_words, c->touch_base.p, c->n_bodies,
                     c->body_tree.p, c->tree_off.p, c->nodes.p, c->touch_acc.p + TOUCH_RUN);
  HIPCHK(c, hipGetLastError());
  c->touch_host.assign(TOUCH_RUN + TOUCH_FIELDS, 0ull);
  HIPCHK(c, hipMemcpyAsync(c->touch_host.data(), c->touch_acc.p, sizeof(unsigned long long) * c->touch_host.size(),
                           hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

void enqueue_level(d2_ctx* c, int level, int discrete) {
  if (c->touch_on && !c->capturing) touch_level(c, level, discrete);
  Dev D = make_dev(c, level, discrete);
  const LevelGrids G = level_grids(c, discrete, level);
  const int cg = G.cull, sg = G.stream;
  D.defer = D.defer && G.def > 0 ? 1 : 0;
  D.box_test = G.box;
  if (discrete && c->precision == D2_FP32) {
    timed_launch(c, K_TRI_MASK, k_tri_mask, dim3(cg), dim3(256), D);
    timed_launch(c, K_TRI_DIST, G.quad ? k_tri_dist<true> : k_tri_dist<false>, dim3(sg), dim3(256), D);
    if (D.defer) timed_launch(c, K_TRI_DEF, k_tri_def, dim3(G.def), dim3(256), D);
  } else if (discrete) {  // as many wavefronts as there are node pairs, up to the tuned blocks
    if (D.prune) timed_launch(c, K_TRI_FULL, k_tri_full<true>, dim3(cg), dim3(256), D);
    else timed_launch(c, K_TRI_FULL, k_tri_full<false>, dim3(cg), dim3(256), D);
  } else {
    // the connected list of level 0 is empty (roots go to the soup list)
    D.conn_blocks = level > 0 ? G.conn : 0;
    timed_launch(c, K_SOUP_CULL, k_ccd_cull, dim3(cg + D.conn_blocks), dim3(256), D);
    if (D.fp32) timed_launch(c, K_SOUP_KEEP, k_soup_keep, dim3(sg), dim3(256), D);  // FP32 culls + survivor lists
    timed_launch(c, K_SOUP_EDGE, k_ccd_sub, dim3(G.sub), dim3(256), D);
    timed_launch(c, K_SOUP_REDUCE, k_soup_reduce, dim3(sg), dim3(256), D);
  }
  if (discrete && c->precision != D2_FP32) {  // FP32 discrete levels are expanded by k_tri_mask
    Timer tm(c, K_EXPAND, 0.0);
    hipLaunchKernelGGL(k_disc_expand, dim3(cg), dim3(256), 0, c->stream, D);
  }
}

// Grid of the per-contact kernels of the post-processing: one contact per
// thread at the last run's count of the phase (mode 2: CCD) with 25%
// headroom, at least 16 blocks, at most the tuned stream grid.
int post_grid(const d2_ctx* c, int mode) {
  const int hi = stream_grid(c);
  const long long n = c->prev_contacts[mode >= 2 ? 1 : 0];
  if (n < 0) return hi;
  long long b = 16;
  while (b < hi && b * 256 < n + n / 4) b <<= 1;
  return (int)std::min<long long>(b, hi);
}

// The per-pair finishing launches over contacts, pair_off and perm: pairs up to
// 512 contacts in the first (wblocks blocks), those up to 2048 in the second
// launch's LDS pass, larger ones by the second launch's per-pair forms, a
// 1024-thread block per pair (n_big[0..1] count the two lists, zeroed before).
// mode 1 applies filterContacts(.., margin).
HugeScratch huge_scratch(d2_ctx* c) {
  const size_t m = c->hscratch.n / 6;
  int* h = c->hscratch.p;
  return HugeScratch{h, h + m, h + 2 * m, h + 3 * m, h + 4 * m, h + 5 * m};
}
void launch_finish(d2_ctx* c, int np, int wblocks, int mode, unsigned long long* kept_total, double margin) {
  hipLaunchKernelGGL((k_pair_finish_block<BLK_CAP, 256>), dim3(wblocks), dim3(256), 0, c->stream, np, (const int*)nullptr,
                     (const int*)nullptr, c->contacts.p, c->pair_off.p, c->perm.p, mode, c->keep.p, c->kept_cnt.p,
                     c->pair_rec.p, c->scale.p, c->big.p, c->n_big.p, c->huge.p, c->n_big.p + 1,
                     (const int*)nullptr, (const int*)nullptr, kept_total, margin, huge_scratch(c));
  hipLaunchKernelGGL((k_pair_finish_block<POST_CAP_LARGE, 1024>), dim3(std::max(1, std::min(np, c->cus))), dim3(1024), 0,
                     c->stream, np, (const int*)c->big.p, (const int*)c->n_big.p, c->contacts.p, c->pair_off.p,
                     c->perm.p, mode, c->keep.p, c->kept_cnt.p, c->pair_rec.p, c->scale.p, c->huge.p,
                     c->n_big.p + 1, c->huge.p, c->n_big.p + 1, (const int*)c->huge.p,
                     (const int*)(c->n_big.p + 1), kept_total, margin, huge_scratch(c));
}

// Post-processing of the contacts of the last phase: per-pair order, then the
// contact filter (mode 1), the step rule (mode 2) or nothing (mode 0); mode 3
// (a step's CCD phase) runs the step rule alone, on the unordered contacts.
int enqueue_post(d2_ctx* c, int mode) {
  const int np = c->n_pairs;
  if (mode == 3) {
    Timer tm(c, K_POST_PAIRS, (double)np);
    hipLaunchKernelGGL(k_step_rule, dim3(post_grid(c, mode)), dim3(256), 0, c->stream, c->cnt.p, c->cap_contacts,
                       c->contacts.p, c->pair_rec.p, c->scale.p);
    HIPCHK(c, hipGetLastError());
    return D2_OK;
  }
  const int sg = post_grid(c, mode);
  const bool filtered = mode == 1;
  {
    Timer tm(c, K_POST, 0.0);  // per-pair counts come from the emitting kernels, zeroed by k_setup
    unsigned long long* total = filtered ? nullptr : c->cnt.p + C_OUT;
    const bool fuse = np <= SCAN_FUSE;  // the scan inside k_scatter
    if (!fuse) scan_host_n(c, c->pair_cnt.p, c->pair_off.p, np, total);
    hipLaunchKernelGGL(k_scatter, dim3(sg), dim3(256), 0, c->stream, c->cnt.p, c->cap_contacts, c->contacts.p,
                       c->pair_off.p, c->pair_fill.p, c->perm.p, fuse ? (const int*)c->pair_cnt.p : nullptr, np,
                       fuse ? total : nullptr);
  }
  {
    Timer tm(c, K_POST_PAIRS, (double)np);
    const int wblocks = std::max(1, std::min(np, c->tune.post_blocks));
    // pairs above the first launch's capacity (512 contacts): the second
    // launch's 2048-contact LDS pass (list big); above that, its per-pair
    // forms on global scratch (list huge, filled by the first launch only)
    // the filter's kept total accumulates into C_OUT (zeroed by k_setup); the
    // output offsets are scanned when the contacts are read (d2_result_contacts)
    unsigned long long* kept_total = filtered ? c->cnt.p + C_OUT : nullptr;
    launch_finish(c, np, wblocks, mode, kept_total, 0.0);  // filterContacts(contacts, 0.0), PDE_explicit.cpp:88
  }
  HIPCHK(c, hipGetLastError());
  return D2_OK;
}

ClusterAcc cluster_acc(d2_ctx* c, const int32_t* cluster_of_pair, int n_clusters, float dt, bool project) {
  ClusterAcc A{};
  A.n_clusters = n_clusters, A.n_bodies = c->n_bodies, A.dt = dt;
  A.step_bits = c->step_bits.p, A.first_any = c->first_any.p, A.first_ns = c->first_ns.p;
  A.read_later = c->read_later.p;
  A.bodies = c->bodies.p, A.body_step = project ? c->body_step.p : nullptr;
  A.pairs = c->pairs.p, A.cluster_of_pair = cluster_of_pair;
  return A;
}
// started: the accumulators were initialised and the first pairs recorded
// by the phase's k_setup / k_fold_final.
int enqueue_clusters(d2_ctx* c, const int32_t* cluster_of_pair, int n_clusters, float dt, bool project,
                     bool first_member, bool started) {
  const int np = c->n_pairs;
  Timer tm(c, K_CLUSTER, np);
  double* body_step = project ? c->body_step.p : nullptr;
  const ClusterAcc A = cluster_acc(c, cluster_of_pair, n_clusters, dt, project);
  if (!started)
    hipLaunchKernelGGL(k_cluster_init, dim3(grid_for(c, std::max(n_clusters, c->n_bodies))), dim3(256), 0, c->stream, A);
  if (np > 0) {
    if (!started) hipLaunchKernelGGL(k_cluster_first, dim3(grid_for(c, np)), dim3(256), 0, c->stream, np, A);
    hipLaunchKernelGGL(k_cluster_min, dim3(grid_for(c, np)), dim3(256), 0, c->stream, np, c->pairs.p, cluster_of_pair,
                       c->bodies.p, c->pair_cnt.p, c->scale.p, c->first_ns.p, c->read_later.p, c->step_bits.p);
  }
  ClusterFinal F;
  F.pairs = c->pairs.p, F.bodies = c->bodies.p, F.step_bits = c->step_bits.p, F.first_any = c->first_any.p;
  F.first_ns = c->first_ns.p, F.first_member = first_member ? c->cc_first.p : (const int*)nullptr;
  F.pair_cnt = c->pair_cnt.p, F.read_later = c->read_later.p, F.scale = c->scale.p;
  hipLaunchKernelGGL(k_cluster_final, dim3(grid_for(c, project ? std::max(n_clusters, np) : n_clusters)), dim3(256), 0,
                     c->stream, n_clusters, dt, F, c->cluster_step.p, np, cluster_of_pair, body_step);
  if (project)
    hipLaunchKernelGGL(k_project, dim3(grid_for(c, c->n_bodies)), dim3(256), 0, c->stream, c->n_bodies, c->bodies.p,
                       c->body_step.p, 1);
  HIPCHK(c, hipGetLastError());
  return D2_OK;
}

// ---------------------------------------------------------------- phases
// A run is a list of traversal phases, each: set-up + roots, breadth-first
// levels, closing fold + post-processing (a step adds the cluster steps and
// projections between its CCD and discrete phases).
struct PhaseSpec {
  int discrete, keep_ccd, mt_from_bodies, post_mode, slot;
};
int phases_of(int kind, int filter, PhaseSpec* out) {
  const int fmode = filter ? 1 : 0;
  if (kind == RUN_NARROW) {
    out[0] = {1, 0, 0, fmode, 0};
    return 1;
  }
  if (kind == RUN_CCD) {
    out[0] = {0, 0, 0, 2, 1};
    return 1;
  }
  out[0] = {0, 0, 1, 3, 2};  // the step never reads its CCD contacts: step rule only
  out[1] = {1, 1, 0, fmode, 3};
  return 2;
}

// Whether the learned gate runs in this phase.
bool gate_on(const d2_ctx* c, const PhaseSpec& ph) {
  return c->learned_on && c->mlp_ready && c->n_pairs > 0 && (c->gate_phases & (ph.discrete ? 2 : 1));
}

// The cluster-step accumulators of a step run, set up by its CCD phase's
// k_setup (initialisation) and k_fold_final (first pairs); none otherwise.
ClusterAcc step_acc(d2_ctx* c, int kind, const PhaseSpec& ph, float dt) {
  if (kind != RUN_STEP || ph.discrete) return ClusterAcc{};
  return cluster_acc(c, c->cluster_of_pair.p, c->n_clusters, dt, true);
}

void enqueue_begin(d2_ctx* c, int kind, const PhaseSpec& ph, float dt) {
  const int np = c->n_pairs;
  Timer tm(c, K_SETUP, np);
  Dev D = make_dev(c, 0, ph.discrete);
  hipLaunchKernelGGL(k_setup, dim3(grid_for(c, 4ll * std::max(np, 1))), dim3(256), 0, c->stream, D, c->pairs.p,
                     c->max_time.p, c->bodies.p, c->body_tree.p, c->tree_off.p, c->pair_info.p, c->pair_rec.p,
                     ph.discrete ? 0 : 1, ph.mt_from_bodies, ph.keep_ccd, c->scale.p, c->pair_fill.p, c->kept_cnt.p,
                     c->n_big.p, step_acc(c, kind, ph, dt), gate_on(c, ph) ? 1 : 0);
}

// The learned gate of a phase: proposals (once per run), certificates, and
// the phase's root list without the certified pairs.
void enqueue_gate(d2_ctx* c, const PhaseSpec& ph) {
  const int np = c->n_pairs;
  if (!gate_on(c, ph)) return;
  {
    Timer tg(c, K_GATE, np);
    Dev D = make_dev(c, 0, ph.discrete);
    if (!ph.keep_ccd || !(c->gate_phases & 1)) {  // a step's discrete phase reuses its CCD phase's proposals
      const double* mt = (ph.mt_from_bodies || !c->has_max_time) ? nullptr : c->max_time.p;
      const int tiles = (np + 15) / 16;  // features computed inside the inference kernel
      hipLaunchKernelGGL(k_mlp_infer<true>, dim3(std::max(1, std::min((tiles + 3) / 4, c->cus * 4))), dim3(256), 0,
                         c->stream, np, (const float*)nullptr, c->mlp_wb.p, c->pred.p,
                         FeatIn{c->pairs.p, c->bodies.p, c->body_tree.p, c->tree_radius.p, mt});
    }
    // at most CERT_LIST pairs per block; the kept pairs are the phase's roots
    const CertIn C{np, c->pair_info.p, c->body_tree.p, c->pair_rec.p, c->pred.p, c->gate_t, c->gate_s,
                   c->hv_off.p, c->hv.p, c->tree_eps_out.p, ph.discrete ? 1 : 0};
    unsigned long long* counts = c->cnt.p + (ph.discrete ? C_GATED_DISC : C_GATED_CCD);
    const int fill = (np + CERT_LIST - 1) / CERT_LIST;
    const int waves = std::max(std::max(1, std::min((np + 3) / 4, c->cus * 8)), fill);
    hipLaunchKernelGGL(k_certify, dim3(waves), dim3(256), 0, c->stream, C, c->cert.p, counts, D.soup, c->lvl.p + LV_SOUP);
    if (c->big_hulls)
      hipLaunchKernelGGL(k_certify_block, dim3(std::max(std::max(1, std::min(np, c->cus * 8)), fill)), dim3(256), 0,
                         c->stream, C, c->cert.p, counts, D.soup, c->lvl.p + LV_SOUP);
  }
}

// Items of level l per kernel, from its sizes (profiling).
void add_level_items(d2_ctx* c, int level, int discrete) {
  const unsigned long long* s = c->host_lvl + level * LV_STRIDE;
  if (discrete && c->precision != D2_FP32) {
    c->k_items[K_TRI_FULL] += (double)s[LV_ITEMS];
    c->k_items[K_EXPAND] += (double)s[LV_SOUP];
  } else if (discrete) {
    c->k_items[K_TRI_MASK] += (double)s[LV_SOUP];
    c->k_items[K_TRI_ENUM] += (double)s[LV_SOUP];
    c->k_items[K_TRI_DIST] += (double)s[LV_ITEMS];
    c->k_items[K_TRI_DEF] += (double)s[LV_DEF];
  } else {
    const bool fp32 = c->precision == D2_FP32;  // FP32 form: the sub-tests its culls keep
    const double point = fp32 ? (double)s[LV_SPT] : 6.0 * (double)s[LV_ITEMS];
    const double edge = fp32 ? (double)s[LV_SEE] : 9.0 * (double)s[LV_ITEMS];
    c->k_items[K_SOUP_CULL] += (double)s[LV_SOUP] + (double)s[LV_CONN];
    if (fp32) c->k_items[K_SOUP_KEEP] += (double)s[LV_ITEMS];
    c->k_items[K_SOUP_POINT] += point;
    c->k_items[K_SOUP_EDGE] += (point + edge) + ((double)s[LV_PT] + (double)s[LV_EE]);
    c->k_items[K_SOUP_REDUCE] += (double)s[LV_ITEMS];
    c->k_items[K_LEAF_POINT] += (double)s[LV_PT];
    c->k_items[K_LEAF_EDGE] += (double)s[LV_EE];
  }
}

struct CopyOut {  // bytes (a multiple of 4) of device memory for the host; none when dst is null
  void* dst;
  const void* src;
  size_t bytes;
};
int read_out(d2_ctx* c, std::initializer_list<CopyOut> parts, int max_threads = 1 << 30);

int read_slots(d2_ctx* c, int first, int count) {
  RC(read_out(c, {{c->host_lvl + first * LV_STRIDE, c->lvl.p + first * LV_STRIDE,
                          sizeof(unsigned long long) * LV_STRIDE * count}}));
  return D2_OK;
}

// Eager levels from `level` on while the lists are not empty (sizes read back
// after every level).  *used receives the index one past the last level run.
int eager_levels(d2_ctx* c, const PhaseSpec& ph, int level, long long n_soup, long long n_conn, int* used) {
  const int budget = level_budget(c);
  for (; level < budget && n_soup + n_conn > 0; ++level) {
    enqueue_level(c, level, ph.discrete);
    HIPCHK(c, hipGetLastError());
    RC(read_slots(c, level, 2));
    if (c->profiling) add_level_items(c, level, ph.discrete);
    n_soup = (long long)c->host_lvl[(level + 1) * LV_STRIDE + LV_SOUP];
    n_conn = (long long)c->host_lvl[(level + 1) * LV_STRIDE + LV_CONN];
  }
  if (n_soup + n_conn > 0) return fail(c, D2_ERR_RUNTIME, "traversal deeper than the level budget of the uploaded trees");
  *used = level;
  return D2_OK;
}

void enqueue_levels(d2_ctx* c, const PhaseSpec& ph, int from, int to) {
  for (int level = from; level < to; ++level) enqueue_level(c, level, ph.discrete);
}

// Closing fold (CCD) and post-processing, then (a step's CCD phase) the
// cluster steps and future states.
int enqueue_end(d2_ctx* c, int kind, const PhaseSpec& ph, int levels, float dt) {
  if (!ph.discrete) {
    Dev D = make_dev(c, levels, 0);
    hipLaunchKernelGGL(k_fold_final, dim3(grid_for(c, std::max(c->n_pairs, 1))), dim3(256), 0, c->stream, D,
                       step_acc(c, kind, ph, dt));
  }
  RC(enqueue_post(c, ph.post_mode));
  if (kind == RUN_STEP && !ph.discrete)
    RC(enqueue_clusters(c, c->cluster_of_pair.p, c->n_clusters, dt, true, c->clusters_on_device, true));
  HIPCHK(c, hipGetLastError());
  return D2_OK;
}

int run_eager(d2_ctx* c, int kind, int filter, float dt) {
  PhaseSpec ph[2];
  const int n = phases_of(kind, filter, ph);
  for (int i = 0; i < n; ++i) {
    enqueue_begin(c, kind, ph[i], dt);
    enqueue_gate(c, ph[i]);
    HIPCHK(c, hipGetLastError());
    int used = 0;
    RC(eager_levels(c, ph[i], 0, c->n_pairs, 0, &used));
    c->phase_levels[ph[i].slot] = std::max(c->phase_levels[ph[i].slot], used);
    RC(enqueue_end(c, kind, ph[i], used, dt));
  }
  return D2_OK;
}

// Graph runs: each phase runs its observed level count inside the graph; when
// that is below the level budget, the graph ends there, the host reads the
// next level's sizes and continues eagerly if a deeper level is needed (and
// the phase's level count grows for the next capture).
int launch_segment(d2_ctx* c, int kind, int seg, const Sig& sig, const std::vector<std::function<int()>>& ops) {
  if (seg >= MAX_SEGMENTS) return fail(c, D2_ERR_RUNTIME, "internal: too many graph segments");
  Captured& g = c->graphs[kind][seg];
  if (!g.valid || !(g.sig == sig)) {
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
    g = Captured{};
    hipGraph_t graph = nullptr;
    HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    c->capturing = true;
    int rc = D2_OK;
    for (auto& op : ops)
      if ((rc = op())) break;
    c->capturing = false;
    hipError_t e = hipStreamEndCapture(c->stream, &graph);
    if (rc) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc;
    }
    if (e != hipSuccess) return fail(c, D2_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    e = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) return fail(c, D2_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
    g.valid = true, g.sig = sig;
    ++c->graph_captures;
  }
  HIPCHK(c, hipGraphLaunch(g.exec, c->stream));
  ++c->graph_launches;
  return D2_OK;
}

// Graph runs need every phase's level count observed by an eager run first.
bool graph_ready(const d2_ctx* c, int kind, int filter) {
  PhaseSpec ph[2];
  const int n = phases_of(kind, filter, ph);
  for (int i = 0; i < n; ++i)
    if (c->phase_levels[ph[i].slot] < 0) return false;
  return true;
}

int run_graph(d2_ctx* c, int kind, int filter, float dt) {
  PhaseSpec ph[2];
  const int n = phases_of(kind, filter, ph);
  const int budget = level_budget(c);
  Sig sig;
  sig.n_pairs = c->n_pairs, sig.n_bodies = c->n_bodies, sig.n_clusters = kind == RUN_STEP ? c->n_clusters : 0;
  sig.max_depth = c->pair_depth, sig.precision = c->precision, sig.filter = filter, sig.dt = dt;
  sig.tune = c->tune;
  sig.learned = (c->learned_on && c->mlp_ready) ? c->gate_phases : 0, sig.gate_t = c->gate_t, sig.gate_s = c->gate_s;
  sig.cl_dev = kind == RUN_STEP && c->clusters_on_device ? 1 : 0;
  sig.big_hulls = sig.learned && c->big_hulls ? 1 : 0;
  for (int i = 0; i < n; ++i) sig.levels[i] = std::min(c->phase_levels[ph[i].slot], budget);
  for (int i = 0; i < n; ++i)
    sig.grids = (sig.grids * 31 + grids_hash(c, ph[i].discrete, sig.levels[i])) * 31 + post_grid(c, ph[i].post_mode);
  std::vector<std::function<int()>> ops;
  int seg = 0;
  for (int i = 0; i < n; ++i) {
    const PhaseSpec p = ph[i];
    const int L = sig.levels[i];
    ops.push_back([c, kind, p, dt] {
      enqueue_begin(c, kind, p, dt);
      enqueue_gate(c, p);
      return D2_OK;
    });
    ops.push_back([c, p, L] { enqueue_levels(c, p, 0, L); return D2_OK; });
    ops.push_back([c, kind, p, L, dt] { return enqueue_end(c, kind, p, L, dt); });
    c->graph_levels[i] = L;
  }
  RC(launch_segment(c, kind, seg, sig, ops));
  return D2_OK;
}

// After a graph run: whether a phase's traversal went on past the levels in
// the graph (its next level is not empty).  The graph runs every phase to the
// deepest level count seen so far without stopping for the host; when a run
// needs more, it is repeated eagerly (the inputs are unchanged by a run) and
// the next capture holds more levels.
bool graph_cut_short(const d2_ctx* c, int kind, int filter) {
  PhaseSpec ph[2];
  const int n = phases_of(kind, filter, ph);
  const int half = (MAX_LEVELS + 1) * LV_STRIDE;
  for (int i = 0; i < n; ++i) {
    const int L = c->graph_levels[i];
    if (L >= level_budget(c)) continue;  // the budget check covers it
    // a step's CCD phase: its sizes as saved by k_fold_final
    const unsigned long long* t = c->host_lvl + (kind == RUN_STEP && !ph[i].discrete ? half : 0) + L * LV_STRIDE;
    if (t[LV_SOUP] || t[LV_CONN]) return true;
  }
  return false;
}

int ensure_clusters(d2_ctx* c, int n_clusters) {
  RC(ensure(c, c->step_bits, n_clusters)); RC(ensure(c, c->first_any, n_clusters)); RC(ensure(c, c->first_ns, n_clusters));
  RC(ensure(c, c->cluster_step, n_clusters)); RC(ensure(c, c->body_step, std::max(c->n_bodies, 1)));
  RC(ensure(c, c->read_later, std::max(c->n_bodies, 1)));
  return D2_OK;
}

// Waits for the run, reads the counters, checks capacity.
int finish_run(d2_ctx* c, int kind, int filter) {
  RC(read_out(c, {{c->host_cnt, c->cnt.p, sizeof(unsigned long long) * C_COUNT},
                         {c->host_lvl, c->lvl.p, sizeof(unsigned long long) * 2 * (MAX_LEVELS + 1) * LV_STRIDE}}));
  HIPCHK(c, hipGetLastError());
  if (c->profiling) collect_timers(c);
  const int budget = level_budget(c);
  const unsigned long long* last = c->host_lvl + budget * LV_STRIDE;
  if (c->host_cnt[C_OVERFLOW] || (long long)c->host_cnt[C_CONTACTS] > c->cap_contacts)
    return fail(c, D2_ERR_CAPACITY, "work list capacity exceeded; raise it with d2_set_capacity");
  if (last[LV_SOUP] || last[LV_CONN])
    return fail(c, D2_ERR_RUNTIME, "traversal deeper than the level budget of the uploaded trees");
  {
    const int half = (MAX_LEVELS + 1) * LV_STRIDE;
    auto keep = [&](int ph, const unsigned long long* src) {
      for (int l = 0; l <= MAX_LEVELS; ++l)
        for (int k = 0; k < LV_STRIDE; ++k) c->prev_lv[ph][l][k] = (long long)src[l * LV_STRIDE + k];
      c->prev_ok[ph] = true;
    };
    if (kind == RUN_CCD) keep(1, c->host_lvl);
    if (kind == RUN_NARROW) keep(0, c->host_lvl);
    if (kind == RUN_STEP) keep(0, c->host_lvl), keep(1, c->host_lvl + half);
    if (kind == RUN_CCD) c->prev_contacts[1] = (long long)c->host_cnt[C_CONTACTS];
    else c->prev_contacts[0] = (long long)c->host_cnt[C_CONTACTS];
    if (kind == RUN_STEP) c->prev_contacts[1] = (long long)c->host_lvl[half + LV_STRIDE - 1];
  }
  c->n_out = (long long)c->host_cnt[C_OUT];
  c->last_kind = kind;
  ++c->run_serial;
  c->last_mode = kind == RUN_CCD ? 1 : 0;
  c->ccd_valid = kind != RUN_NARROW;
  c->out_filtered = kind != RUN_CCD && filter != 0;
  c->last_filter = filter ? 1 : 0;
  return D2_OK;
}

// Capacities large enough for the sizes the failed run recorded (exact for
// the levels it reached; a deeper level may need another round).  The
// discrete phase's sizes are in the first half of the level table, the CCD
// phase's in the second; the overflow counter says which phase overflowed.
void grow_capacities(d2_ctx* c, int kind) {
  const int half = (MAX_LEVELS + 1) * LV_STRIDE;
  long long np = c->n_pairs, items = 0, res = 0, contacts = 0;
  auto scan = [&](const unsigned long long* t, bool ccd) {
    for (int l = 0; l <= MAX_LEVELS; ++l) {
      const unsigned long long* v = t + l * LV_STRIDE;
      np = std::max<long long>(np, (long long)std::max(v[LV_SOUP], v[LV_CONN]));
      if (ccd) {
        res = std::max<long long>(res, (long long)v[LV_ITEMS]);
        items = std::max<long long>(items, (long long)std::max(v[LV_PT], v[LV_EE]));
        items = std::max<long long>(items, (long long)std::max(v[LV_SPT], v[LV_SEE]));  // FP32 form's soup survivors
      } else if (c->precision == D2_FP32) {  // FP64 discrete levels keep no item list (k_tri_full)
        items = std::max<long long>(items, (long long)std::max(v[LV_ITEMS], v[LV_DEF]));
      }
    }
  };
  if (kind != RUN_CCD) scan(c->host_lvl, false), contacts = (long long)c->host_cnt[C_CONTACTS];
  if (kind != RUN_NARROW) scan(c->host_lvl + half, true),
      contacts = std::max<long long>(contacts, (long long)c->host_lvl[half + LV_STRIDE - 1]);
  auto grown = [](long long cur, long long need) { return need > cur ? std::max(2 * cur, need + need / 4) : cur; };
  bool any = false;
  long long v;
  if ((v = grown(c->cap, np)) != c->cap) c->cap = v, any = true;
  if ((v = grown(c->cap_items, items)) != c->cap_items) c->cap_items = v, any = true;
  if ((v = grown(c->cap_res, res)) != c->cap_res) c->cap_res = v, any = true;
  if ((v = grown(c->cap_contacts, contacts)) != c->cap_contacts) c->cap_contacts = v, any = true;
  if (!any) {  // sizes beyond the recorded ones (an overflow cut a level short): double the phase's lists
    const unsigned long long ov = c->host_cnt[C_OVERFLOW];
    c->cap *= 2, c->cap_contacts *= 2;
    if ((ov & 2ull) && c->precision == D2_FP32) c->cap_items *= 2;
    if (ov & 1ull) c->cap_res *= 2, c->cap_items *= 2;
  }
}

int run_once(d2_ctx* c, int kind, int filter, float dt, int64_t* n_contacts_out);

// This device's copy of `scratch`, resolved once per device with the device
// current (the first context created on it) and kept until the process ends;
// nullptr when the runtime cannot resolve it.
unsigned char* noalloc_scratch(int device) {
  static std::mutex mu;
  static unsigned char* addr[256] = {};
  static bool tried[256] = {};
  if (device < 0 || device >= 256) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  if (!tried[device]) {
    tried[device] = true;
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) == hipSuccess) addr[device] = static_cast<unsigned char*>(p);
  }
  return addr[device];
}

// ---- results to the caller's memory
// The caller's buffers are pageable.  The runtime's own copy into such memory
// moves 6 to 17 GB/s (one host thread copying out of its staging buffer), and
// each of a result's arrays is a copy of its own; asynchronous copies to pinned
// memory cost 125 us apiece when an event follows each.  Here one kernel writes
// all arrays into this context's pinned window, and the host copies a slot on
// as soon as its flag says that it is there, from several threads when the
// result is large.  170 MB of contacts: 10.3 -> 4.9 ms (then host memory
// bandwidth); 39 MB: 6.1 -> 1.1 ms; a 100-body step's contacts and per-pair
// values, six small copies before: 0.33 -> 0.09 ms.
constexpr int STAGE_THREADS = 6;
constexpr size_t STAGE_HALF = (size_t)8 << 20, HALF_SLOTS = STAGE_HALF / COPY_SLOT;  // two halves: one fills, one empties
void release_stage(d2_ctx* c) {
  if (c->stage) (void)hipHostFree(c->stage);
  if (c->stage_flag) (void)hipHostFree(c->stage_flag);
  if (c->stage_cnt) (void)hipFree(c->stage_cnt);
  c->stage = nullptr, c->stage_flag = nullptr, c->stage_cnt = nullptr;
}
// The window (at context creation); without one the runtime's copies serve.
void make_stage(d2_ctx* c) {
  const unsigned f = hipHostMallocMapped | hipHostMallocCoherent;
  bool ok = hipHostMalloc((void**)&c->stage, 2 * STAGE_HALF, f) == hipSuccess;
  if (!ok) c->stage = nullptr;
  if (ok && hipHostMalloc((void**)&c->stage_flag, sizeof(unsigned long long) * 2 * HALF_SLOTS, f) != hipSuccess)
    ok = false, c->stage_flag = nullptr;
  if (ok && hipMalloc((void**)&c->stage_cnt, sizeof(int) * 2 * HALF_SLOTS) != hipSuccess) ok = false, c->stage_cnt = nullptr;
  if (ok) {
    std::memset(c->stage_flag, 0, sizeof(unsigned long long) * 2 * HALF_SLOTS);
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(256), 0, c->stream, c->stage_cnt, (long long)(2 * HALF_SLOTS), 0);
    ok = hipGetLastError() == hipSuccess;
  }
  if (ok) return;
  release_stage(c);
  (void)hipGetLastError();
}
// The parts, in stream order after what the stream holds; complete on return.
// At most max_threads host threads, the caller's included.
hipError_t copy_out(d2_ctx* c, std::initializer_list<CopyOut> parts, int max_threads) {
  (void)hipSetDevice(c->device);
  CopyJob J{};
  unsigned char* dst[COPY_PARTS] = {};
  unsigned long long total = 0;
  for (const CopyOut& p : parts) {  // (at most COPY_PARTS)
    if (!p.bytes || !p.dst) continue;
    dst[J.n] = (unsigned char*)p.dst;
    J.src[J.n] = (const unsigned char*)p.src, J.begin[J.n] = total, J.bytes[J.n] = p.bytes;
    total += (p.bytes + COPY_PIECE - 1) / COPY_PIECE * COPY_PIECE;
    ++J.n;
  }
  if (total && !c->stage) {
    for (int i = 0; i < J.n; ++i) {
      const hipError_t e = hipMemcpyAsync(dst[i], J.src[i], J.bytes[i], hipMemcpyDeviceToHost, c->stream);
      if (e != hipSuccess) return e;
    }
    return hipStreamSynchronize(c->stream);
  }
  if (!total) return hipStreamSynchronize(c->stream);
  const size_t window = STAGE_HALF, windows = (total + window - 1) / window, per = HALF_SLOTS;
  const size_t chunks = (total + COPY_SLOT - 1) / COPY_SLOT;
  const unsigned long long gen = c->stage_gen + 1;  // of window 0
  c->stage_gen += windows;
  std::atomic<size_t> next{0}, done[2] = {{0}, {0}};
  std::atomic<size_t> launched[2] = {{0}, {0}};  // per half, windows launched into it so far: w + 1 of the last
  std::atomic<int> err{(int)hipSuccess};
  auto launch = [&](size_t w) {  // window w, into half w & 1 (window w - 2 has been copied on)
    if (w > 1) (void)hipSetDevice(c->device);  // (maybe one of the threads below)
    CopyJob K = J;
    K.off = w * window, K.end = std::min<unsigned long long>(total, K.off + window);
    K.dst = c->stage + (w & 1) * window, K.count = c->stage_cnt + (w & 1) * per, K.flag = c->stage_flag + (w & 1) * per;
    K.gen = gen + w;
    const unsigned blocks = (unsigned)((K.end - K.off + COPY_PIECE - 1) / COPY_PIECE);
    hipLaunchKernelGGL(k_copy_out, dim3(blocks), dim3(256), 0, c->stream, K);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) err.store((int)e);
    launched[w & 1].store(w + 1);
  };
  auto arrived = [&](size_t w, size_t slot) {
    const unsigned long long* f = c->stage_flag + (w & 1) * per + slot;
    for (unsigned spin = 1;; ++spin) {
      if (__atomic_load_n(f, __ATOMIC_ACQUIRE) == gen + w) return true;
      if (err.load(std::memory_order_relaxed) != (int)hipSuccess) return false;
      if (spin % 256 == 0) std::this_thread::yield();
      if (spin % 16384 == 0 && launched[w & 1].load() == w + 1) {  // a failed stream ends the wait
        const hipError_t e = hipStreamQuery(c->stream);
        if (e == hipErrorNotReady) continue;
        if (e == hipSuccess && __atomic_load_n(f, __ATOMIC_ACQUIRE) == gen + w) return true;
        err.store((int)(e == hipSuccess ? hipErrorUnknown : e));
        return false;
      }
    }
  };
  auto work = [&] {
    for (size_t k; (k = next.fetch_add(1)) < chunks;) {
      const size_t w = k / per;
      if (!arrived(w, k % per)) return;
      const unsigned long long a = k * COPY_SLOT, b = a + COPY_SLOT;
      const unsigned char* from = c->stage + (w & 1) * window + (k % per) * COPY_SLOT;
      for (int i = 0; i < J.n; ++i) {
        const unsigned long long lo = std::max(a, J.begin[i]), hi = std::min(b, J.begin[i] + J.bytes[i]);
        if (lo < hi) std::memcpy(dst[i] + (lo - J.begin[i]), from + (lo - a), hi - lo);
      }
      const size_t in_window = std::min(per, chunks - w * per);
      if (done[w & 1].fetch_add(1) + 1 == in_window && w + 2 < windows) {
        done[w & 1].store(0);
        launch(w + 2);
      }
    }
  };
  launch(0);
  if (windows > 1) launch(1);
  // a thread (about 20 us to start) per 2 MB, which takes one 200 us to copy
  const unsigned cores = std::thread::hardware_concurrency();
  const int threads = (int)std::min<size_t>(
      {(size_t)STAGE_THREADS, (size_t)max_threads, std::max<size_t>(cores / 2, 1), (chunks + 3) / 4});
  std::array<std::thread, STAGE_THREADS> pool;
  for (int t = 1; t < threads; ++t) {
    try {
      pool[t] = std::thread(work);
    } catch (const std::exception&) {  // (nothing may unwind past the joinable threads)
      break;  // the threads there are do the work
    }
  }
  work();
  for (std::thread& t : pool)
    if (t.joinable()) t.join();
  if (err.load() != (int)hipSuccess) (void)hipStreamSynchronize(c->stream);  // nothing writes the window any more
  return (hipError_t)err.load();
}

int read_out(d2_ctx* c, std::initializer_list<CopyOut> parts, int max_threads) {
  const hipError_t e = copy_out(c, parts, max_threads);
  return e == hipSuccess ? D2_OK : fail(c, D2_ERR_HIP, std::string("reading results: ") + hipGetErrorString(e));
}

// Which clusters a lane each solves, by size (SV_BINS classes), the others a
// block each.  A lane takes 1.5 to 6 times as long for a cluster as a block
// does (below, us for clusters of each class: measured with spheres in single
// layers and stacks on a floor), but hardly longer for thousands of clusters
// than for one, while two blocks fit a CU: 10,000 single spheres on a floor
// take 5.0 ms with a block each and 0.5 ms with a lane each, 8,192 stacks of
// two 8.5 and 1.8 ms, 512 of them 0.7 and 1.6 ms.
int sv_small_size(const d2_ctx* c, const int* hist) {
  constexpr double LANE[SV_BINS - 1] = {350, 1600, 3000, 5000, 17000};
  constexpr double BLOCK[SV_BINS] = {240, 720, 1100, 1300, 2900, 6000};
  int best = -1;
  double best_us = 0.0, lane = 0.0, n_lane = 0.0;
  for (int b = -1; b < SV_BINS - 1; ++b) {  // classes up to b by lanes
    if (b >= 0 && hist[b]) lane = LANE[b], n_lane += hist[b];
    double one = 0.0, all = 0.0;  // the others' longest, and their share of the chip
    for (int k = b + 1; k < SV_BINS; ++k)
      if (hist[k]) one = BLOCK[k], all += 0.7 * hist[k] * BLOCK[k] / (2.0 * c->cus);
    const double us = lane * (1.0 + n_lane / 20000.0) + std::max(one, all);
    if (b < 0 || us < best_us) best = b < 0 ? -1 : 2 << b, best_us = us;
  }
  return best;
}

// ---- bucket-level entry: scratch and one call
struct BucketScratch {
  int32_t* np;       // [cap_np][2] staged node pairs
  long long* base;   // [cap_np] first provisional slot of each node pair
  int* count;        // [cap_np] hits of each node pair
  long long* off;    // [cap_np] first output row of each node pair
  int32_t* used;     // [cap_np] cumulative hit counts
  ContactRec* hits;  // [cap_hits] provisional hit records
  int32_t* out_i;    // [cap_hits][8]
  double* out_r;     // [cap_hits][11]
  unsigned long long* counter;
  long long cap_np, cap_hits;
};

// Validates a bucket call against the resident trees and bodies.
int bucket_check(d2_ctx* c, int a, int b, int n, const int32_t* node_pairs, const char* who) {
  if (c->n_bodies <= 0) return fail(c, D2_ERR_STATE, std::string(who) + ": upload trees and bodies first");
  if (a < 0 || a >= c->n_bodies || b < 0 || b >= c->n_bodies || n < 0 || (n > 0 && !node_pairs))
    return fail(c, D2_ERR_ARG, std::string(who) + ": bad arguments");
  const int ta = c->host_body_tree[a], tb = c->host_body_tree[b];
  const int na = c->host_tree_off[ta + 1] - c->host_tree_off[ta], nb = c->host_tree_off[tb + 1] - c->host_tree_off[tb];
  for (int k = 0; k < n; ++k)
    if (node_pairs[2 * k] < 0 || node_pairs[2 * k] >= na || node_pairs[2 * k + 1] < 0 || node_pairs[2 * k + 1] >= nb)
      return fail(c, D2_ERR_ARG, std::string(who) + ": node index out of range");
  return D2_OK;
}

// One bucket call on the given scratch.  *total receives the hit count; the
// cumulative counts are always written, the hits when they fit both the
// scratch and max_hits.
int bucket_run(d2_ctx* c, const BucketScratch& S, int a, int b, int n, const int32_t* node_pairs,
               int32_t* pair_used_out, int64_t max_hits, int32_t* ints_out, double* reals_out, long long* total,
               int max_threads) {
  *total = 0;
  if (n == 0) return D2_OK;
  HIPCHK(c, hipMemcpyAsync(S.np, node_pairs, sizeof(int32_t) * 2 * (size_t)n, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, c->stream, S.counter, 1ll, 0ull);
  BucketArgs A;
  A.np_list = S.np, A.n = n, A.nodes = c->nodes.p, A.buckets = c->buckets.p;
  A.off_a = c->host_tree_off[c->host_body_tree[a]], A.off_b = c->host_tree_off[c->host_body_tree[b]];
  A.body_a = c->bodies.p + 40 * (size_t)a, A.body_b = c->bodies.p + 40 * (size_t)b;
  A.hits = S.hits, A.cap = S.cap_hits, A.counter = S.counter, A.base = S.base, A.count = S.count;
  const int blocks = (int)std::min<long long>((n + 3) / 4, (long long)c->cus * 8);  // a node pair per wavefront
  // two wavefronts per SIMD (what fits), then several node pairs per wavefront
  hipLaunchKernelGGL(k_bucket_pairs, dim3(std::min(blocks, c->cus * 2)), dim3(256), 0, c->stream, A);
  hipLaunchKernelGGL(k_bucket_scan, dim3(1), dim3(1024), 0, c->stream, n, (const int*)S.count, S.off, S.used);
  HIPCHK(c, hipGetLastError());
  unsigned long long hits = 0;
  RC(read_out(c, {{&hits, S.counter, sizeof(hits)}, {pair_used_out, S.used, sizeof(int32_t) * (size_t)n}}, max_threads));
  *total = (long long)hits;
  if ((long long)hits > S.cap_hits || (long long)hits > max_hits || hits == 0) return D2_OK;
  hipLaunchKernelGGL(k_bucket_place, dim3(blocks), dim3(256), 0, c->stream, n, (const long long*)S.base,
                     (const int*)S.count, (const long long*)S.off, (const ContactRec*)S.hits, S.out_i, S.out_r);
  HIPCHK(c, hipGetLastError());
  RC(read_out(c, {{ints_out, S.out_i, sizeof(int32_t) * 8 * hits}, {reals_out, S.out_r, sizeof(double) * 11 * hits}},
                     max_threads));
  return D2_OK;
}

int run(d2_ctx* c, int kind, int filter, float dt, int64_t* n_contacts_out) {
  int rc = run_once(c, kind, filter, dt, n_contacts_out);
  for (int attempt = 0; rc == D2_ERR_CAPACITY && c->auto_grow && attempt < 8; ++attempt) {
    grow_capacities(c, kind);
    rc = run_once(c, kind, filter, dt, n_contacts_out);
  }
  return rc;
}

int run_once(d2_ctx* c, int kind, int filter, float dt, int64_t* n_contacts_out) {
  if (!c->pairs_valid || c->n_bodies <= 0 || c->n_trees <= 0)
    return fail(c, D2_ERR_STATE, "upload trees, bodies and pairs first");
  if (c->pair_depth + 1 > MAX_LEVELS)
    return fail(c, D2_ERR_ARG, "a pair's trees are too deep: depth(a) + depth(b) must stay below 16");
  if (kind == RUN_STEP && c->n_clusters <= 0) return fail(c, D2_ERR_STATE, "upload the pairs' clusters first");
  (void)hipSetDevice(c->device);
  if (c->n_pairs > c->cap) return fail(c, D2_ERR_CAPACITY, "more pairs than the work-list capacity");
  RC(prepare(c));
  if (kind == RUN_STEP) RC(ensure_clusters(c, c->n_clusters));
  c->ccd_valid = false;
  c->last_mode = -1;
  // accounting runs are eager: their extra kernels sit between the levels
  const bool graph = c->graph_on && !c->touch_on && graph_ready(c, kind, filter);
  if (c->touch_on) RC(touch_begin(c));
  if (graph) RC(run_graph(c, kind, filter, dt));
  else RC(run_eager(c, kind, filter, dt));
  RC(finish_run(c, kind, filter));
  if (c->touch_on) RC(touch_end(c));
  if (graph && graph_cut_short(c, kind, filter)) {
    RC(run_eager(c, kind, filter, dt));
    RC(finish_run(c, kind, filter));
  }
  if (n_contacts_out) *n_contacts_out = c->n_out;
  return D2_OK;
}

// ---- the solver's warm store
constexpr size_t WARM_MIN = 1u << 20;
WarmTable warm_table(d2_ctx* c) {
  return WarmTable{c->warm_keys.p, c->warm_vals.p, (unsigned long long)c->warm_keys.n - 1, c->warm_used.p};
}
// Room for `extra` more keys at a load factor of at most one half: the table
// doubles (re-inserting its keys) until it fits.  Synchronises the stream.
int warm_reserve(d2_ctx* c, long long extra) {
  if (!c->warm_keys.p) {
    RC(ensure(c, c->warm_keys, WARM_MIN)); RC(ensure(c, c->warm_vals, WARM_MIN)); RC(ensure(c, c->warm_used, 1));
    hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(c, WARM_MIN)), dim3(256), 0, c->stream, c->warm_keys.p,
                       (long long)WARM_MIN, WARM_EMPTY);
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, c->stream, c->warm_used.p, 1ll, 0ull);
  }
  unsigned long long used = 0;
  HIPCHK(c, hipMemcpyAsync(&used, c->warm_used.p, sizeof(used), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  size_t cap = c->warm_keys.n;
  while ((long long)used + extra > (long long)(cap / 2)) cap *= 2;
  if (cap == c->warm_keys.n) return D2_OK;
  DBuf<unsigned long long> old_k = c->warm_keys;
  DBuf<double> old_v = c->warm_vals;
  c->warm_keys = DBuf<unsigned long long>{}, c->warm_vals = DBuf<double>{};
  RC(ensure(c, c->warm_keys, cap)); RC(ensure(c, c->warm_vals, cap));
  hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(c, (long long)cap)), dim3(256), 0, c->stream, c->warm_keys.p,
                     (long long)cap, WARM_EMPTY);
  hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, c->stream, c->warm_used.p, 1ll, 0ull);
  hipLaunchKernelGGL(k_warm_rehash, dim3(grid_for(c, (long long)old_k.n)), dim3(256), 0, c->stream,
                     (const unsigned long long*)old_k.p, (const double*)old_v.p, (long long)old_k.n, warm_table(c));
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->stream));
  release(old_k), release(old_v);
  return D2_OK;
}

}  // namespace

// ------------------------------------------------------------------ C ABI
extern "C" {

int d2_ctx_create(int device, int precision, d2_ctx** out) {
  if (!out) return D2_ERR_ARG;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return D2_ERR_HIP;
  if (device < 0 || device >= ndev) return D2_ERR_ARG;
  if (precision != D2_FP64 && precision != D2_FP32) return D2_ERR_ARG;
  d2_ctx* c = new d2_ctx();
  c->device = device;
  c->precision = precision;
  if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&c->stream) != hipSuccess) {
    delete c;
    return D2_ERR_HIP;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) c->cus = prop.multiProcessorCount;
  c->tune = d2_tune{4 * c->cus, 8 * c->cus, 16 * c->cus, 3};
  if (hipHostMalloc((void**)&c->host_cnt, sizeof(unsigned long long) * C_COUNT, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&c->host_lvl, sizeof(unsigned long long) * 2 * (MAX_LEVELS + 1) * LV_STRIDE,
                    hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&c->host_red, sizeof(int) * (BR_N + 2), hipHostMallocDefault) != hipSuccess) {
    if (c->host_cnt) (void)hipHostFree(c->host_cnt);
    if (c->host_lvl) (void)hipHostFree(c->host_lvl);
    (void)hipStreamDestroy(c->stream);
    delete c;
    return D2_ERR_HIP;
  }
  std::memset(c->host_lvl, 0, sizeof(unsigned long long) * 2 * (MAX_LEVELS + 1) * LV_STRIDE);
  make_stage(c);
  c->noalloc = noalloc_scratch(device);
  *out = c;
  return D2_OK;
}

int d2_ctx_destroy(d2_ctx* c) {
  if (!c) return D2_ERR_ARG;
  (void)hipSetDevice(c->device);
  (void)hipStreamSynchronize(c->stream);
  collect_timers(c);
  drop_graphs(c);
  release(c->nodes), release(c->buckets), release(c->fbuckets), release(c->stris), release(c->tree_off), release(c->body_tree), release(c->bodies);
  release(c->pairs), release(c->pair_info), release(c->cluster_of_pair), release(c->max_time), release(c->pair_rec), release(c->pair_f);
  for (int k = 0; k < 2; ++k) release(c->soup_list[k]), release(c->conn_list[k]);
  release(c->items), release(c->ditems), release(c->ditems_def), release(c->pt_items), release(c->ee_items), release(c->lpt_items), release(c->lee_items), release(c->res), release(c->res_mask), release(c->np_hit), release(c->np_hit2), release(c->exp_desc);
  release(c->contacts), release(c->cnt), release(c->lvl);
  release(c->pass_min_s), release(c->pass_min_c), release(c->pass_flag_s), release(c->pass_flag_c);
  release(c->min_time), release(c->scale);
  release(c->pair_cnt), release(c->pair_off), release(c->pair_fill), release(c->perm), release(c->keep),
      release(c->kept_cnt), release(c->out_off), release(c->out_i), release(c->out_r), release(c->scan_part);
  release(c->big), release(c->huge), release(c->n_big), release(c->hscratch);
  release(c->nbound), release(c->kid_inner);
  release(c->sv_mass), release(c->sv_fric), release(c->sv_ccount), release(c->sv_chits), release(c->sv_poff),
      release(c->sv_hoff), release(c->sv_cfill), release(c->sv_cpairs), release(c->sv_inpair), release(c->sv_loc),
      release(c->sv_status), release(c->sv_flag), release(c->sv_hl), release(c->sv_ord), release(c->sv_hrow),
      release(c->sv_hpc), release(c->sv_pbody), release(c->sv_hA), release(c->sv_hB), release(c->sv_heps),
      release(c->sv_hkey), release(c->sv_hs), release(c->sv_ps), release(c->sv_out),
      release(c->sv_out_csr), release(c->sv_cpart), release(c->sv_cps), release(c->sv_ploc), release(c->sv_phit),
      release(c->sv_hint), release(c->sv_lvlo), release(c->sv_cntl), release(c->sv_pint),
      release(c->warm_keys), release(c->warm_used), release(c->warm_vals);
  release(c->step_bits), release(c->first_any), release(c->first_ns), release(c->cluster_step), release(c->body_step),
      release(c->tmp_cluster), release(c->read_later);
  release(c->touch_base), release(c->touch_lv), release(c->touch_run), release(c->touch_lvb), release(c->touch_runb),
      release(c->touch_acc);
  release(c->bk_np), release(c->bk_used), release(c->bk_out_i), release(c->bk_base), release(c->bk_off),
      release(c->bk_count), release(c->bk_hits), release(c->bk_out_r), release(c->bk_counter);
  release(c->tree_radius), release(c->tree_eps_out), release(c->hv), release(c->feat), release(c->pred), release(c->hv_off);
  release(c->cert), release(c->mlp_w), release(c->mlp_m), release(c->mlp_v), release(c->mlp_wf), release(c->mlp_grad);
  release(c->mlp_wb), release(c->tr_x), release(c->tr_t), release(c->tr_part), release(c->tr_loss);
  release(c->tr_idx);
  release(c->tb_box), release(c->tb_rad), release(c->last_state), release(c->bp_R), release(c->tree_depth_d),
      release(c->group);
  release(c->bp_statics), release(c->bp_item_body), release(c->bp_item_seg), release(c->bp_item_cnt),
      release(c->bp_item_sorted), release(c->bp_item_off), release(c->bp_meta), release(c->bp_slot), release(c->bp_rank),
      release(c->bp_counts), release(c->bp_start), release(c->bp_members), release(c->bp_red);
  release(c->bp_item_pos), release(c->bp_keys), release(c->bp_fill), release(c->bp_box), release(c->bp_chunk);
  release(c->cc_parent), release(c->cc_label), release(c->cc_root), release(c->cc_root_off), release(c->cc_of_body),
      release(c->cc_first), release(c->cc_tmin), release(c->cc_smin);
  if (c->host_red) (void)hipHostFree(c->host_red);
  release_stage(c);
  if (c->host_cnt) (void)hipHostFree(c->host_cnt);
  if (c->host_lvl) (void)hipHostFree(c->host_lvl);
  (void)hipStreamDestroy(c->stream);
  delete c;
  return D2_OK;
}

const char* d2_last_error(const d2_ctx* c) { return c ? c->err.c_str() : "null context"; }

int d2_set_precision(d2_ctx* c, int precision) {
  if (!c) return D2_ERR_ARG;
  if (precision != D2_FP64 && precision != D2_FP32) return fail(c, D2_ERR_ARG, "precision must be D2_FP64 or D2_FP32");
  c->precision = precision;
  return D2_OK;
}

int d2_set_capacity(d2_ctx* c, int64_t entries) {
  if (!c) return D2_ERR_ARG;
  if (entries < 1024) return fail(c, D2_ERR_ARG, "capacity must be >= 1024");
  drop_graphs(c);
  c->cap = entries;
  c->cap_items = entries;
  c->cap_contacts = entries;
  c->cap_res = std::min<long long>(entries, 1ll << 20);
  c->auto_grow = false;
  return D2_OK;
}

int d2_set_auto_grow(d2_ctx* c, int on) {
  if (!c) return D2_ERR_ARG;
  c->auto_grow = on != 0;
  return D2_OK;
}

int d2_set_tune(d2_ctx* c, const d2_tune* t) {
  if (!c || !t) return D2_ERR_ARG;
  if (t->chunk_blocks < 1 || t->chunk_blocks > 4096 || t->stream_blocks < 1 || t->stream_blocks > 16384 ||
      t->post_blocks < 1 || t->post_blocks > 16384 || t->gate_phases < 0 || t->gate_phases > 3)
    return fail(c, D2_ERR_ARG, "d2_set_tune: value out of range");
  c->tune = *t;
  if (c->learned_on) c->gate_phases = t->gate_phases;
  return D2_OK;
}
int d2_get_tune(const d2_ctx* c, d2_tune* t) {
  if (!c || !t) return D2_ERR_ARG;
  *t = c->tune;
  t->gate_phases = c->gate_phases;
  return D2_OK;
}

// Coordinate descent over the launch shapes, timing whole runs of the given
// kind (graph or eager, as the context is set) on the resident inputs.
int d2_autotune(d2_ctx* c, int kind, float dt, int filter, int reps, d2_tune* best_out, double* best_ms_out) {
  if (!c || kind < 0 || kind >= RUN_KINDS || reps < 1) return D2_ERR_ARG;
  d2_tune start = c->tune;
  start.gate_phases = c->gate_phases;
  auto time_it = [&](const d2_tune& t, double* ms) -> int {
    c->tune = t;
    if (c->learned_on) c->gate_phases = t.gate_phases;
    RC(run(c, kind, filter, dt, nullptr));  // warm-up (and capture)
    std::vector<double> v;
    for (int r = 0; r < reps; ++r) {
      auto t0 = std::chrono::steady_clock::now();
      RC(run(c, kind, filter, dt, nullptr));
      v.push_back(std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count());
    }
    std::sort(v.begin(), v.end());
    *ms = v[v.size() / 2];
    return D2_OK;
  };
  const int u = c->cus;
  const std::vector<int> chunk = {u, 2 * u, 4 * u, 8 * u, 16 * u};
  const std::vector<int> stream = {2 * u, 4 * u, 8 * u, 16 * u, 32 * u};
  const std::vector<int> post = {4 * u, 16 * u, 64 * u};
  d2_tune best = start;
  double best_ms = 0.0;
  int rc = time_it(best, &best_ms);
  const std::vector<int> gate = {0, 1, 2, 3};  // 0: the gate gated in no phase (it may not pay for itself)
  const int dims = c->learned_on ? 4 : 3;
  for (int sweep = 0; sweep < 2 && !rc; ++sweep)
    for (int dim = 0; dim < dims && !rc; ++dim) {
      const std::vector<int>& vals = dim == 0 ? chunk : dim == 1 ? stream : dim == 2 ? post : gate;
      for (int v : vals) {
        d2_tune t = best;
        int* f = dim == 0 ? &t.chunk_blocks : dim == 1 ? &t.stream_blocks : dim == 2 ? &t.post_blocks : &t.gate_phases;
        if (*f == v || v > (dim == 0 ? 4096 : 16384)) continue;
        *f = v;
        double ms = 0.0;
        if ((rc = time_it(t, &ms))) break;
        if (ms < best_ms) best_ms = ms, best = t;
      }
    }
  c->tune = rc ? start : best;
  if (c->learned_on) c->gate_phases = c->tune.gate_phases;
  if (rc) return rc;
  if (best_out) *best_out = best;
  if (best_ms_out) *best_ms_out = best_ms;
  return D2_OK;
}

int d2_set_graph(d2_ctx* c, int on) {
  if (!c) return D2_ERR_ARG;
  if (!on) drop_graphs(c);
  c->graph_on = on != 0;
  return D2_OK;
}

int d2_trees_upload(d2_ctx* c, int n_trees, const int32_t* tree_node_offset, const int32_t* nodes, const double* buckets) {
  if (!c) return D2_ERR_ARG;
  if (n_trees <= 0 || !tree_node_offset || !nodes || !buckets) return fail(c, D2_ERR_ARG, "d2_trees_upload: bad arguments");
  int total = tree_node_offset[n_trees];
  if (total <= 0 || tree_node_offset[0] != 0) return fail(c, D2_ERR_ARG, "d2_trees_upload: bad offsets");
  std::vector<int> depth(n_trees, 0);
  for (int t = 0; t < n_trees; ++t) {
    int b = tree_node_offset[t], e = tree_node_offset[t + 1];
    if (e <= b) return fail(c, D2_ERR_ARG, "d2_trees_upload: empty tree");
    for (int i = b; i < e; ++i) {
      const int32_t* r = nodes + 8 * (size_t)i;
      int cnt = e - b;
      if (r[1] < 0 || r[1] >= cnt || r[7] < 0 || r[7] > 8 || r[3] < 0 ||
          (r[2] && (r[5] < 0 || r[5] + r[6] > cnt || r[6] < 1 || r[6] > 8)))
        return fail(c, D2_ERR_ARG, "d2_trees_upload: inconsistent node record");
      depth[t] = std::max(depth[t], (int)r[3]);
    }
  }
  (void)hipSetDevice(c->device);
  c->n_trees = 0;  // no trees until every per-node table of this upload is in place
  RC(ensure(c, c->nodes, total)); RC(ensure(c, c->buckets, (size_t)total * BUCKET)); RC(ensure(c, c->tree_off, n_trees + 1));
  c->n_nodes_total = total, c->fb_ready = false;  // the float copy follows on the next FP32 run
  HIPCHK(c, hipMemcpyAsync(c->nodes.p, nodes, sizeof(NodeRec) * total, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->buckets.p, buckets, sizeof(double) * BUCKET * (size_t)total, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->tree_off.p, tree_node_offset, sizeof(int32_t) * (n_trees + 1), hipMemcpyHostToDevice, c->stream));
  // Per tree, for the learned gate's certificate: the distinct vertices of the
  // leaf triangles (body coordinates), the bounding radius, and how far beyond
  // the search distance a leaf contact can be accepted: the largest distance a
  // float-barycentric "inside" test can accept a point outside a triangle,
  // 64 eps_f kappa L (kappa = d00 d11 / (d00 d11 - d01^2), L the longest edge;
  // 4x the 16 eps_f kappa L rounding bound), plus the largest eps of the leaf
  // buckets (the discrete hit test adds them, comparison_dist.h:233).
  std::vector<float> hv, radius(n_trees), eps_out(n_trees);
  std::vector<int32_t> hv_off(n_trees + 1, 0);
  for (int t = 0; t < n_trees; ++t) {
    std::vector<std::array<double, 3>> vs;
    double rmax = 0.0, eo = 0.0, leaf_eps = 0.0;
    for (int i = tree_node_offset[t]; i < tree_node_offset[t + 1]; ++i) {
      const int32_t* r = nodes + 8 * (size_t)i;
      if (r[2]) continue;
      const double* bk = buckets + (size_t)BUCKET * (tree_node_offset[t] + r[1]);
      for (int k = 0; k < r[7]; ++k) {
        leaf_eps = std::max(leaf_eps, bk[72 + k]);
        std::array<double, 3> v[3];
        for (int q = 0; q < 3; ++q) v[q] = {bk[(3 * q) * 8 + k], bk[(3 * q + 1) * 8 + k], bk[(3 * q + 2) * 8 + k]};
        double e0[3], e1[3], e2[3];
        for (int d = 0; d < 3; ++d) e0[d] = v[1][d] - v[0][d], e1[d] = v[2][d] - v[0][d], e2[d] = v[2][d] - v[1][d];
        const double d00 = e0[0] * e0[0] + e0[1] * e0[1] + e0[2] * e0[2];
        const double d11 = e1[0] * e1[0] + e1[1] * e1[1] + e1[2] * e1[2];
        const double d01 = e0[0] * e1[0] + e0[1] * e1[1] + e0[2] * e1[2];
        const double d22 = e2[0] * e2[0] + e2[1] * e2[1] + e2[2] * e2[2];
        const double den = d00 * d11 - d01 * d01;
        const double kappa = den > 0.0 ? d00 * d11 / den : 1e30;
        eo = std::max(eo, 64.0 * 5.9604645e-08 * kappa * std::sqrt(std::max(d00, std::max(d11, d22))));
        for (int q = 0; q < 3; ++q) {
          vs.push_back(v[q]);
          rmax = std::max(rmax, std::sqrt(v[q][0] * v[q][0] + v[q][1] * v[q][1] + v[q][2] * v[q][2]));
        }
      }
    }
    std::sort(vs.begin(), vs.end());
    vs.erase(std::unique(vs.begin(), vs.end()), vs.end());
    for (auto& v : vs) hv.push_back((float)v[0]), hv.push_back((float)v[1]), hv.push_back((float)v[2]);
    hv_off[t + 1] = hv_off[t] + (int32_t)vs.size();
    radius[t] = (float)rmax * (1.0f + 1e-6f);
    // rounded up so the float margin is never below the double one
    eps_out[t] = (float)std::min((eo + leaf_eps) * (1.0 + 1e-6), 1e30);
  }
  // Per node, for pruning (NB_STRIDE floats): the body-frame box of every
  // leaf-triangle vertex under the node, the largest (leaf eps +
  // float-barycentric acceptance bound 64 eps_f kappa L) of those triangles,
  // and a sphere around the same vertices (their centroid, the largest
  // distance from it), all rounded outward; children follow their parent, so
  // one pass from the back merges the boxes and slacks, and a second pass
  // per node over its leaves' vertices gives the spheres.
  std::vector<float> nb((size_t)total * NB_STRIDE);
  for (int t = 0; t < n_trees; ++t) {
    const int b0 = tree_node_offset[t];
    for (int i = tree_node_offset[t + 1] - 1; i >= b0; --i) {
      const int32_t* r = nodes + 8 * (size_t)i;
      double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY}, E = 0.0;
      if (!r[2]) {
        const double* bk = buckets + (size_t)BUCKET * (b0 + r[1]);
        for (int k = 0; k < r[7]; ++k) {
          double v[3][3];
          for (int q = 0; q < 3; ++q)
            for (int d = 0; d < 3; ++d) v[q][d] = bk[(3 * q + d) * 8 + k];
          E = std::max(E, leaf_slack(v[0], v[1], v[2], bk[72 + k]));
          for (int q = 0; q < 3; ++q)
            for (int d = 0; d < 3; ++d) lo[d] = std::min(lo[d], v[q][d]), hi[d] = std::max(hi[d], v[q][d]);
        }
      } else {
        for (int ch = 0; ch < r[6]; ++ch) {
          const float* cb = nb.data() + NB_STRIDE * ((size_t)b0 + r[5] + ch);
          for (int d = 0; d < 3; ++d) lo[d] = std::min(lo[d], (double)cb[d]), hi[d] = std::max(hi[d], (double)cb[3 + d]);
          E = std::max(E, (double)cb[6]);
        }
      }
      float* o = nb.data() + NB_STRIDE * (size_t)i;
      const bool empty = !(lo[0] <= hi[0]);
      for (int d = 0; d < 3; ++d) {  // an empty node never prunes
        float fl = empty ? -FLT_MAX : (float)lo[d], fh = empty ? FLT_MAX : (float)hi[d];
        if ((double)fl > lo[d]) fl = std::nextafter(fl, -INFINITY);
        if ((double)fh < hi[d]) fh = std::nextafter(fh, INFINITY);
        o[d] = fl, o[3 + d] = fh;
      }
      float fe = (float)std::min(E, 1e30);
      if ((double)fe < E) fe = std::nextafter(fe, INFINITY);
      o[6] = fe, o[7] = FLT_MAX, o[8] = o[9] = o[10] = o[11] = 0.0f;
    }
    // spheres: the leaves under a node are a contiguous run of the tree's
    // leaves in depth-first order, so each node's vertex set is walked once
    // per level of the tree (leaf vertices gathered bottom-up by child lists)
    std::vector<std::vector<int>> leaves_of(tree_node_offset[t + 1] - b0);
    for (int i = tree_node_offset[t + 1] - 1; i >= b0; --i) {
      const int32_t* r = nodes + 8 * (size_t)i;
      std::vector<int>& L = leaves_of[i - b0];
      if (!r[2]) L.push_back(i);
      else
        for (int ch = 0; ch < r[6]; ++ch) {
          std::vector<int>& C = leaves_of[r[5] + ch];
          L.insert(L.end(), C.begin(), C.end());
        }
      double cen[3] = {0.0, 0.0, 0.0};
      long long nv = 0;
      for (int leaf : L) {
        const int32_t* lr = nodes + 8 * (size_t)leaf;
        const double* bk = buckets + (size_t)BUCKET * (b0 + lr[1]);
        for (int k = 0; k < lr[7]; ++k)
          for (int q = 0; q < 3; ++q, ++nv)
            for (int d = 0; d < 3; ++d) cen[d] += bk[(3 * q + d) * 8 + k];
      }
      if (nv == 0) continue;  // no vertices: the sphere never prunes
      float fc[3];
      for (int d = 0; d < 3; ++d) fc[d] = (float)(cen[d] / (double)nv);
      double rad = 0.0;
      for (int leaf : L) {
        const int32_t* lr = nodes + 8 * (size_t)leaf;
        const double* bk = buckets + (size_t)BUCKET * (b0 + lr[1]);
        for (int k = 0; k < lr[7]; ++k)
          for (int q = 0; q < 3; ++q) {
            double s2 = 0.0;
            for (int d = 0; d < 3; ++d) {
              const double x = bk[(3 * q + d) * 8 + k] - (double)fc[d];
              s2 += x * x;
            }
            rad = std::max(rad, std::sqrt(s2));
          }
      }
      float* o = nb.data() + NB_STRIDE * (size_t)i;
      float fr = (float)(rad * (1.0 + 1e-12));
      if ((double)fr < rad) fr = std::nextafter(fr, INFINITY);
      o[7] = fr, o[8] = fc[0], o[9] = fc[1], o[10] = fc[2];
      if (!r[2]) continue;
      for (int ch = 0; ch < r[6]; ++ch) std::vector<int>().swap(leaves_of[r[5] + ch]);  // children are done
    }
  }
  RC(ensure(c, c->nbound, nb.size()));
  HIPCHK(c, hipMemcpyAsync(c->nbound.p, nb.data(), sizeof(float) * nb.size(), hipMemcpyHostToDevice, c->stream));
  // Per node, which of its (at most 8) children are inner nodes: the CCD
  // expansion routes a node pair's children to the soup or the connected
  // list by it instead of reading every child's record.
  std::vector<uint8_t> kid((size_t)total, 0);
  for (int t = 0; t < n_trees; ++t) {
    const int b0 = tree_node_offset[t];
    for (int i = b0; i < tree_node_offset[t + 1]; ++i) {
      const int32_t* r = nodes + 8 * (size_t)i;
      if (!r[2]) continue;
      unsigned m = 0;
      for (int ch = 0; ch < r[6]; ++ch)
        if (nodes[8 * ((size_t)b0 + r[5] + ch) + 2]) m |= 1u << ch;
      kid[i] = (uint8_t)m;
    }
  }
  RC(ensure(c, c->kid_inner, kid.size()));
  HIPCHK(c, hipMemcpyAsync(c->kid_inner.p, kid.data(), kid.size(), hipMemcpyHostToDevice, c->stream));
  // Per tree for the broad phase, as MeshData::initBoudingData (model/mesh.cpp:44-51)
  // computes it over the mesh vertices (here: the leaf triangles' vertices,
  // which are every vertex of a mesh whose vertices all belong to a face):
  // the float AABB and the largest vertex norm.
  std::vector<float> tbox(6 * (size_t)n_trees);
  std::vector<double> trad(n_trees, 0.0);
  for (int t = 0; t < n_trees; ++t) {
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = tree_node_offset[t]; i < tree_node_offset[t + 1]; ++i) {
      const int32_t* r = nodes + 8 * (size_t)i;
      if (r[2]) continue;
      const double* bk = buckets + (size_t)BUCKET * (tree_node_offset[t] + r[1]);
      for (int k = 0; k < r[7]; ++k)
        for (int q = 0; q < 3; ++q) {
          const double x = bk[(3 * q) * 8 + k], y = bk[(3 * q + 1) * 8 + k], z = bk[(3 * q + 2) * 8 + k];
          const float f[3] = {(float)x, (float)y, (float)z};
          for (int d = 0; d < 3; ++d) lo[d] = std::min(lo[d], f[d]), hi[d] = std::max(hi[d], f[d]);
          trad[t] = std::max(trad[t], std::sqrt((x * x + y * y) + z * z));
        }
    }
    for (int d = 0; d < 3; ++d) tbox[6 * t + d] = lo[d], tbox[6 * t + 3 + d] = hi[d];
  }
  RC(ensure(c, c->tb_box, 6 * (size_t)n_trees)); RC(ensure(c, c->tb_rad, n_trees)); RC(ensure(c, c->tree_depth_d, n_trees));
  HIPCHK(c, hipMemcpyAsync(c->tb_box.p, tbox.data(), sizeof(float) * tbox.size(), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->tb_rad.p, trad.data(), sizeof(double) * n_trees, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->tree_depth_d.p, depth.data(), sizeof(int32_t) * n_trees, hipMemcpyHostToDevice, c->stream));
  c->big_hulls = false;
  for (int t = 0; t < n_trees; ++t) c->big_hulls = c->big_hulls || hv_off[t + 1] - hv_off[t] > CERT_WAVEV;
  RC(ensure(c, c->hv, std::max<size_t>(hv.size(), 3))); RC(ensure(c, c->hv_off, n_trees + 1));
  RC(ensure(c, c->tree_radius, n_trees)); RC(ensure(c, c->tree_eps_out, n_trees));
  HIPCHK(c, hipMemcpyAsync(c->hv.p, hv.data(), sizeof(float) * hv.size(), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->hv_off.p, hv_off.data(), sizeof(int32_t) * (n_trees + 1), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->tree_radius.p, radius.data(), sizeof(float) * n_trees, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->tree_eps_out.p, eps_out.data(), sizeof(float) * n_trees, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->n_trees = n_trees;
  c->tree_depth = depth;
  c->host_tree_off.assign(tree_node_offset, tree_node_offset + n_trees + 1);
  c->pair_depth = std::min(MAX_LEVELS - 1, 2 * *std::max_element(depth.begin(), depth.end()));  // until pairs come
  // body records name trees by index: bodies, pairs and clusters must come again
  c->host_body_tree.clear();
  c->n_bodies = 0;
  c->has_groups = false;
  invalidate_pairs(c);
  return D2_OK;
}

int d2_bodies_upload(d2_ctx* c, int n_bodies, const int32_t* tree_of_body, const double* records) {
  if (!c) return D2_ERR_ARG;
  if (n_bodies <= 0 || !tree_of_body || !records) return fail(c, D2_ERR_ARG, "d2_bodies_upload: bad arguments");
  if (c->n_trees <= 0) return fail(c, D2_ERR_STATE, "d2_bodies_upload: upload trees first");
  for (int i = 0; i < n_bodies; ++i)
    if (tree_of_body[i] < 0 || tree_of_body[i] >= c->n_trees) return fail(c, D2_ERR_ARG, "d2_bodies_upload: bad tree index");
  (void)hipSetDevice(c->device);
  RC(ensure(c, c->bodies, (size_t)n_bodies * 40)); RC(ensure(c, c->body_tree, n_bodies));
  HIPCHK(c, hipMemcpyAsync(c->bodies.p, records, sizeof(double) * 40 * (size_t)n_bodies, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->body_tree.p, tree_of_body, sizeof(int32_t) * n_bodies, hipMemcpyHostToDevice, c->stream));
  // last states start equal to the current ones (d2_bodies_last_upload sets them)
  std::vector<double> last(14 * (size_t)n_bodies);
  for (int i = 0; i < n_bodies; ++i) std::memcpy(&last[14 * (size_t)i], records + 40 * (size_t)i, 14 * sizeof(double));
  RC(ensure(c, c->last_state, 14 * (size_t)n_bodies));
  HIPCHK(c, hipMemcpyAsync(c->last_state.p, last.data(), sizeof(double) * last.size(), hipMemcpyHostToDevice, c->stream));
  // broad-phase work items: one per non-static body, one per bp_seg later
  // bodies for a static one (it sweeps all of them)
  c->host_static.clear();
  for (int i = 0; i < n_bodies; ++i)
    if (records[40 * (size_t)i + 38] != 0.0) c->host_static.push_back(i);
  const int seg = c->bp_seg = bp_segment(c->host_static, n_bodies);
  std::vector<int> ib, is;
  for (int i = 0; i < n_bodies; ++i) {
    if (records[40 * (size_t)i + 38] != 0.0) {
      const int segs = std::max(1, (n_bodies - 1 - i + seg - 1) / seg);
      for (int q = 0; q < segs; ++q) ib.push_back(i), is.push_back(q);
    } else {
      ib.push_back(i), is.push_back(0);
    }
  }
  c->n_items = (int)ib.size();
  RC(ensure(c, c->bp_item_body, ib.size())); RC(ensure(c, c->bp_item_seg, is.size()));
  RC(ensure(c, c->bp_statics, std::max<size_t>(c->host_static.size(), 1)));
  HIPCHK(c, hipMemcpyAsync(c->bp_item_body.p, ib.data(), sizeof(int) * ib.size(), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->bp_item_seg.p, is.data(), sizeof(int) * is.size(), hipMemcpyHostToDevice, c->stream));
  if (!c->host_static.empty())
    HIPCHK(c, hipMemcpyAsync(c->bp_statics.p, c->host_static.data(), sizeof(int) * c->host_static.size(),
                             hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (n_bodies != c->n_bodies) {
    // pairs, clusters and scene groups index bodies: a new count voids them
    invalidate_pairs(c);
    c->has_groups = false;
  } else if (c->pairs_valid && !std::equal(tree_of_body, tree_of_body + n_bodies, c->host_body_tree.begin())) {
    // same bodies, other trees: the kept pairs' level budget becomes the
    // deepest any pair of these trees can need
    c->pair_depth = std::min(MAX_LEVELS - 1, 2 * *std::max_element(c->tree_depth.begin(), c->tree_depth.end()));
  }
  c->n_bodies = n_bodies;
  c->host_body_tree.assign(tree_of_body, tree_of_body + n_bodies);
  return D2_OK;
}

int d2_bodies_download(d2_ctx* c, double* records) {
  if (!c || !records) return D2_ERR_ARG;
  if (c->n_bodies <= 0) return fail(c, D2_ERR_STATE, "no bodies uploaded");
  RC(read_out(c, {{records, c->bodies.p, sizeof(double) * 40 * (size_t)c->n_bodies}}));
  return D2_OK;
}

int d2_solver_bodies(d2_ctx* c, int n_bodies, const double* mass, const double* friction) {
  if (!c) return D2_ERR_ARG;
  if (c->n_bodies <= 0 || n_bodies != c->n_bodies) return fail(c, D2_ERR_ARG, "d2_solver_bodies: one value per uploaded body");
  if (!mass || !friction) return fail(c, D2_ERR_ARG, "d2_solver_bodies: bad arguments");
  for (int i = 0; i < n_bodies; ++i)
    if (!(mass[i] > 0.0) || !(friction[i] >= 0.0))
      return fail(c, D2_ERR_ARG, "d2_solver_bodies: masses must be > 0 and friction coefficients >= 0");
  (void)hipSetDevice(c->device);
  RC(ensure(c, c->sv_mass, n_bodies)); RC(ensure(c, c->sv_fric, n_bodies));
  HIPCHK(c, hipMemcpyAsync(c->sv_mass.p, mass, sizeof(double) * n_bodies, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->sv_fric.p, friction, sizeof(double) * n_bodies, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

int d2_solve(d2_ctx* c, const double* gravity, int32_t* cluster_status, int* n_failed) {
  if (!c) return D2_ERR_ARG;
  if (!gravity) return fail(c, D2_ERR_ARG, "d2_solve: gravity is NULL");
  if (c->last_mode != 0 || c->last_kind != RUN_STEP || !c->out_filtered)
    return fail(c, D2_ERR_STATE, "d2_solve needs a preceding d2_step_run with the contact filter");
  if (c->sv_mass.n < (size_t)c->n_bodies || !c->sv_mass.p)
    return fail(c, D2_ERR_STATE, "d2_solve: set the bodies' masses and friction first (d2_solver_bodies)");
  (void)hipSetDevice(c->device);
  const int np = c->n_pairs, nk = c->n_clusters, nb = c->n_bodies;
  const long long nh = c->n_out;
  RC(warm_reserve(c, nh));
  RC(ensure(c, c->sv_ccount, nk + 1)); RC(ensure(c, c->sv_chits, nk + 1)); RC(ensure(c, c->sv_poff, nk + 1));
  RC(ensure(c, c->sv_hoff, nk + 1)); RC(ensure(c, c->sv_cfill, nk)); RC(ensure(c, c->sv_status, nk));
  RC(ensure(c, c->sv_cpairs, std::max(np, 1))); RC(ensure(c, c->sv_pbody, 2 * (size_t)std::max(np, 1)));
  RC(ensure(c, c->sv_inpair, nb)); RC(ensure(c, c->sv_loc, nb)); RC(ensure(c, c->sv_flag, 1 + SV_BINS));
  RC(ensure(c, c->out_off, (size_t)np + 1));
  const size_t H = (size_t)std::max<long long>(nh, 1);
  RC(ensure(c, c->sv_hl, 2 * H)); RC(ensure(c, c->sv_ord, H)); RC(ensure(c, c->sv_hrow, H)); RC(ensure(c, c->sv_hpc, H));
  RC(ensure(c, c->sv_hA, 3 * H)); RC(ensure(c, c->sv_hB, 3 * H)); RC(ensure(c, c->sv_heps, H)); RC(ensure(c, c->sv_hkey, H));
  const size_t P = (size_t)std::max(np, 1), K = (size_t)std::max(nk, 1);
  RC(ensure(c, c->sv_hs, (size_t)SH * H)); RC(ensure(c, c->sv_out, 11 * H));
  RC(ensure(c, c->sv_ps, (size_t)SP * 2 * P)); RC(ensure(c, c->sv_cpart, K)); RC(ensure(c, c->sv_cps, P));
  RC(ensure(c, c->sv_ploc, 2 * P)); RC(ensure(c, c->sv_phit, P)); RC(ensure(c, c->sv_hint, 6 * H));
  RC(ensure(c, c->sv_lvlo, H + K)); RC(ensure(c, c->sv_cntl, H)); RC(ensure(c, c->sv_pint, 6 * P + K));
  SolveArgs A;
  A.n_pairs = np, A.n_clusters = nk, A.n_bodies = nb;
  A.pairs = c->pairs.p, A.cluster_of_pair = c->cluster_of_pair.p, A.kept_cnt = c->kept_cnt.p;
  A.pair_off = c->pair_off.p, A.out_off = c->out_off.p, A.perm = c->perm.p, A.keep = c->keep.p;
  A.contacts = c->contacts.p, A.cluster_step = c->cluster_step.p, A.body_step = c->body_step.p;
  A.bodies = c->bodies.p, A.mass = c->sv_mass.p, A.fric = c->sv_fric.p;
  A.gx = gravity[0], A.gy = gravity[1], A.gz = gravity[2];
  A.ccount = c->sv_ccount.p, A.chits = c->sv_chits.p, A.cfill = c->sv_cfill.p, A.cpairs = c->sv_cpairs.p;
  A.inpair = c->sv_inpair.p, A.loc = c->sv_loc.p, A.status = c->sv_status.p;
  A.hl = c->sv_hl.p, A.ord = c->sv_ord.p, A.hrow = c->sv_hrow.p, A.hpc = c->sv_hpc.p, A.pbody = c->sv_pbody.p;
  A.hA = c->sv_hA.p, A.hB = c->sv_hB.p, A.heps = c->sv_heps.p, A.hkey = c->sv_hkey.p;
  A.hs = c->sv_hs.p, A.cpart = c->sv_cpart.p, A.cps = c->sv_cps.p;
  A.ploc = c->sv_ploc.p, A.phit = c->sv_phit.p, A.hint = c->sv_hint.p, A.lvlo = c->sv_lvlo.p;
  A.cntl = c->sv_cntl.p, A.pint = c->sv_pint.p;
  A.ps = c->sv_ps.p, A.out = c->sv_out.p, A.warm = warm_table(c), A.flag = c->sv_flag.p;
  A.hist = c->sv_flag.p + 1, A.small = -1;
  auto fill = [&](int* p, long long n, int v) {
    hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(c, n)), dim3(256), 0, c->stream, p, n, v);
  };
  fill(A.ccount, nk + 1, 0), fill(A.chits, nk + 1, 0), fill(A.cfill, nk, 0);
  fill(A.inpair, nb, 0), fill(A.cpart, nk, 0), fill(c->sv_flag.p, 1 + SV_BINS, 0);
  hipLaunchKernelGGL(k_sv_count, dim3(grid_for(c, np)), dim3(256), 0, c->stream, A);
  scan_host_n(c, c->sv_ccount.p, c->sv_poff.p, nk, nullptr);
  scan_host_n(c, c->sv_chits.p, c->sv_hoff.p, nk, nullptr);
  scan_host_n(c, c->kept_cnt.p, c->out_off.p, np, nullptr);
  SolveArgs B = A;
  B.ccount = c->sv_poff.p, B.chits = c->sv_hoff.p;  // the offsets from here on
  hipLaunchKernelGGL(k_sv_place, dim3(grid_for(c, std::max(std::max(np, nb), nk))), dim3(256), 0, c->stream, B);
  int head[1 + SV_BINS] = {};  // the flag, the clusters by size class
  RC(read_out(c, {{head, c->sv_flag.p, sizeof(head)}}));
  if (head[0]) return fail(c, D2_ERR_ARG, "d2_solve: a dynamic body's pairs lie in more than one cluster");
  B.small = sv_small_size(c, head + 1);
  int n_small = 0;
  for (int b = 0; b < SV_BINS - 1 && 2 << b <= B.small; ++b) n_small += head[1 + b];
  if (n_small > 0)
    hipLaunchKernelGGL(k_sv_solve_small, dim3(grid_for(c, nk, 64)), dim3(64), 0, c->stream, B);
  if (n_small < nk)
    hipLaunchKernelGGL(k_sv_solve, dim3(std::max(1, std::min(nk, 16 * c->cus))), dim3(256), 0, c->stream, B);
  hipLaunchKernelGGL(k_sv_free, dim3(grid_for(c, nb)), dim3(256), 0, c->stream, B);
  HIPCHK(c, hipGetLastError());
  std::vector<int32_t> st(std::max(nk, 1));
  RC(read_out(c, {{st.data(), c->sv_status.p, sizeof(int32_t) * nk}}));
  int failed = 0;
  for (int k = 0; k < nk; ++k) failed += st[k] == 0;
  if (cluster_status && nk > 0) std::memcpy(cluster_status, st.data(), sizeof(int32_t) * nk);
  if (n_failed) *n_failed = failed;
  c->solved_serial = c->run_serial;
  c->solved_hits = nh;
  return D2_OK;
}

int d2_solve_results(d2_ctx* c, double* per_contact) {
  if (!c || !per_contact) return D2_ERR_ARG;
  if (c->last_mode != 0 || c->solved_serial != c->run_serial)
    return fail(c, D2_ERR_STATE, "d2_solve_results: no solve of the last step run");
  const long long nh = c->solved_hits;
  if (nh == 0) return D2_OK;
  (void)hipSetDevice(c->device);
  RC(ensure(c, c->sv_out_csr, 11 * (size_t)nh));
  hipLaunchKernelGGL(k_sv_scatter, dim3(grid_for(c, nh)), dim3(256), 0, c->stream, nh, (const int*)c->sv_hrow.p,
                     (const double*)c->sv_out.p, c->sv_out_csr.p);
  HIPCHK(c, hipGetLastError());
  RC(read_out(c, {{per_contact, c->sv_out_csr.p, sizeof(double) * 11 * (size_t)nh}}));
  return D2_OK;
}

int d2_commit_step(d2_ctx* c) {
  if (!c) return D2_ERR_ARG;
  if (c->last_kind != RUN_STEP || c->last_mode != 0 || c->body_step.n < (size_t)c->n_bodies)
    return fail(c, D2_ERR_STATE, "d2_commit_step needs a preceding d2_step_run");
  (void)hipSetDevice(c->device);
  hipLaunchKernelGGL(k_commit, dim3(grid_for(c, c->n_bodies)), dim3(256), 0, c->stream, c->n_bodies, c->bodies.p,
                     (const double*)c->body_step.p);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->last_mode = -1;  // the step's results no longer describe the bodies
  c->ccd_valid = false;
  return D2_OK;
}

int d2_solver_reset(d2_ctx* c) {
  if (!c) return D2_ERR_ARG;
  if (!c->warm_keys.p) return D2_OK;
  (void)hipSetDevice(c->device);
  hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(c, (long long)c->warm_keys.n)), dim3(256), 0, c->stream,
                     c->warm_keys.p, (long long)c->warm_keys.n, WARM_EMPTY);
  hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, c->stream, c->warm_used.p, 1ll, 0ull);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

int d2_project_future(d2_ctx* c, const double* step_per_body) {
  if (!c || !step_per_body) return D2_ERR_ARG;
  if (c->n_bodies <= 0) return fail(c, D2_ERR_STATE, "no bodies uploaded");
  RC(ensure(c, c->body_step, c->n_bodies));
  HIPCHK(c, hipMemcpyAsync(c->body_step.p, step_per_body, sizeof(double) * c->n_bodies, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_project, dim3(grid_for(c, c->n_bodies)), dim3(256), 0, c->stream, c->n_bodies, c->bodies.p,
                     c->body_step.p, 0);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

int d2_pairs_upload(d2_ctx* c, int n_pairs, const int32_t* pairs, const double* max_time) {
  if (!c) return D2_ERR_ARG;
  if (n_pairs < 0 || (n_pairs > 0 && !pairs)) return fail(c, D2_ERR_ARG, "d2_pairs_upload: bad arguments");
  if (c->n_bodies <= 0) return fail(c, D2_ERR_STATE, "d2_pairs_upload: upload bodies first");
  for (int p = 0; p < n_pairs; ++p) {
    if (pairs[2 * p] < 0 || pairs[2 * p] >= c->n_bodies || pairs[2 * p + 1] < 0 || pairs[2 * p + 1] >= c->n_bodies)
      return fail(c, D2_ERR_ARG, "d2_pairs_upload: body index out of range");
    if (max_time && !(max_time[p] >= 0.0)) return fail(c, D2_ERR_ARG, "d2_pairs_upload: max_time must be >= 0");
  }
  (void)hipSetDevice(c->device);
  size_t np = std::max(n_pairs, 1);
  RC(ensure(c, c->pairs, 2 * np)); RC(ensure(c, c->max_time, np)); RC(ensure(c, c->pair_rec, np * PR_STRIDE));
  RC(ensure(c, c->pair_info, 4 * np));
  if (n_pairs > 0) {
    HIPCHK(c, hipMemcpyAsync(c->pairs.p, pairs, sizeof(int32_t) * 2 * n_pairs, hipMemcpyHostToDevice, c->stream));
    if (max_time)
      HIPCHK(c, hipMemcpyAsync(c->max_time.p, max_time, sizeof(double) * n_pairs, hipMemcpyHostToDevice, c->stream));
    else
      HIPCHK(c, hipMemsetAsync(c->max_time.p, 0, sizeof(double) * n_pairs, c->stream));
  }
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->n_pairs = n_pairs;
  int deepest = 0;
  for (int p = 0; p < n_pairs; ++p)
    deepest = std::max(deepest, c->tree_depth[c->host_body_tree[pairs[2 * p]]] +
                                    c->tree_depth[c->host_body_tree[pairs[2 * p + 1]]]);
  c->pair_depth = deepest;
  c->n_clusters = 0;  // clusters describe a pair list
  c->clusters_on_device = false;
  c->has_max_time = max_time != nullptr;
  c->last_mode = -1;
  c->ccd_valid = false;
  c->pairs_valid = true;
  return D2_OK;
}

int d2_clusters_upload(d2_ctx* c, const int32_t* cluster_of_pair, int n_clusters) {
  if (!c) return D2_ERR_ARG;
  if (!c->pairs_valid) return fail(c, D2_ERR_STATE, "d2_clusters_upload: upload or build the pair list first");
  if (n_clusters <= 0 || (c->n_pairs > 0 && !cluster_of_pair)) return fail(c, D2_ERR_ARG, "d2_clusters_upload: bad arguments");
  for (int p = 0; p < c->n_pairs; ++p)
    if (cluster_of_pair[p] < 0 || cluster_of_pair[p] >= n_clusters)
      return fail(c, D2_ERR_ARG, "d2_clusters_upload: cluster index out of range");
  (void)hipSetDevice(c->device);
  RC(ensure(c, c->cluster_of_pair, std::max(c->n_pairs, 1)));
  if (c->n_pairs > 0)
    HIPCHK(c, hipMemcpyAsync(c->cluster_of_pair.p, cluster_of_pair, sizeof(int32_t) * c->n_pairs, hipMemcpyHostToDevice,
                             c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->n_clusters = n_clusters;
  c->clusters_on_device = false;
  return D2_OK;
}

int d2_narrow_run(d2_ctx* c, int filter, int64_t* n_contacts_out) {
  if (!c) return D2_ERR_ARG;
  return run(c, RUN_NARROW, filter ? 1 : 0, 0.f, n_contacts_out);
}

int d2_ccd_run(d2_ctx* c, int64_t* n_contacts_out) {
  if (!c) return D2_ERR_ARG;
  return run(c, RUN_CCD, 0, 0.f, n_contacts_out);
}

int d2_step_run(d2_ctx* c, float dt, int filter, double* cluster_step_out, int64_t* n_contacts_out) {
  if (!c) return D2_ERR_ARG;
  if (!(dt > 0.f)) return fail(c, D2_ERR_ARG, "d2_step_run: dt must be > 0");
  RC(run(c, RUN_STEP, filter ? 1 : 0, dt, n_contacts_out));
  if (cluster_step_out) {
    RC(read_out(c, {{cluster_step_out, c->cluster_step.p, sizeof(double) * c->n_clusters}}));
  }
  return D2_OK;
}

int d2_find_contacts_bucket(d2_ctx* c, int body_a, int body_b, int n_node_pairs, const int32_t* node_pairs,
                            int32_t* pair_used_out, int64_t max_hits, int32_t* ints_out, double* reals_out,
                            int64_t* n_hits_out) {
  if (!c) return D2_ERR_ARG;
  RC(bucket_check(c, body_a, body_b, n_node_pairs, node_pairs, "d2_find_contacts_bucket"));
  if (n_node_pairs > 0 && !pair_used_out) return fail(c, D2_ERR_ARG, "d2_find_contacts_bucket: pair_used_out is NULL");
  (void)hipSetDevice(c->device);
  const size_t n = std::max(n_node_pairs, 1);
  RC(ensure(c, c->bk_np, 2 * n)); RC(ensure(c, c->bk_base, n)); RC(ensure(c, c->bk_count, n));
  RC(ensure(c, c->bk_off, n)); RC(ensure(c, c->bk_used, n)); RC(ensure(c, c->bk_counter, 1));
  long long cap = std::max<long long>((long long)c->bk_hits.n, 8ll * (long long)n);
  long long total = 0;
  for (int attempt = 0; attempt < 2; ++attempt) {
    RC(ensure(c, c->bk_hits, cap)); RC(ensure(c, c->bk_out_i, 8 * cap)); RC(ensure(c, c->bk_out_r, 11 * cap));
    const BucketScratch S{c->bk_np.p, c->bk_base.p, c->bk_count.p, c->bk_off.p, c->bk_used.p, c->bk_hits.p,
                          c->bk_out_i.p, c->bk_out_r.p, c->bk_counter.p, (long long)n, cap};
    RC(bucket_run(c, S, body_a, body_b, n_node_pairs, node_pairs, pair_used_out, max_hits, ints_out, reals_out, &total, STAGE_THREADS));
    if (total <= cap) break;
    cap = total;  // the scratch grows to the recorded count and the call repeats
  }
  if (n_hits_out) *n_hits_out = total;
  if (total > max_hits) return fail(c, D2_ERR_CAPACITY, "d2_find_contacts_bucket: more hits than max_hits");
  return D2_OK;
}

int d2_find_contacts_bucket_noalloc(d2_ctx* c, int body_a, int body_b, int n_node_pairs, const int32_t* node_pairs,
                                    int32_t* pair_used_out, int64_t max_hits, int32_t* ints_out, double* reals_out,
                                    int64_t* n_hits_out) {
  if (!c) return D2_ERR_ARG;
  RC(bucket_check(c, body_a, body_b, n_node_pairs, node_pairs, "d2_find_contacts_bucket_noalloc"));
  if (n_node_pairs > 0 && !pair_used_out)
    return fail(c, D2_ERR_ARG, "d2_find_contacts_bucket_noalloc: pair_used_out is NULL");
  if (n_node_pairs > NOALLOC_NP)
    return fail(c, D2_ERR_CAPACITY, "d2_find_contacts_bucket_noalloc: at most 32768 node pairs per call");
  if (!c->noalloc) return fail(c, D2_ERR_HIP, "d2_find_contacts_bucket_noalloc: the scratch array has no address");
  (void)hipSetDevice(c->device);
  // the scratch array carved into the bucket call's buffers (8-byte fields first)
  unsigned char* p = c->noalloc;
  BucketScratch S;
  S.base = reinterpret_cast<long long*>(p), p += 8 * NOALLOC_NP;
  S.off = reinterpret_cast<long long*>(p), p += 8 * NOALLOC_NP;
  S.np = reinterpret_cast<int32_t*>(p), p += 8 * NOALLOC_NP;
  S.count = reinterpret_cast<int*>(p), p += 4 * NOALLOC_NP;
  S.used = reinterpret_cast<int32_t*>(p), p += 4 * NOALLOC_NP;
  S.hits = reinterpret_cast<ContactRec*>(p), p += sizeof(ContactRec) * NOALLOC_HITS;
  S.out_r = reinterpret_cast<double*>(p), p += 11 * 8 * NOALLOC_HITS;
  S.out_i = reinterpret_cast<int32_t*>(p), p += 8 * 4 * NOALLOC_HITS;
  S.counter = reinterpret_cast<unsigned long long*>(p);
  S.cap_np = NOALLOC_NP, S.cap_hits = NOALLOC_HITS;
  long long total = 0;
  RC(bucket_run(c, S, body_a, body_b, n_node_pairs, node_pairs, pair_used_out, max_hits, ints_out, reals_out, &total, 1));
  if (n_hits_out) *n_hits_out = total;
  if (total > NOALLOC_HITS)
    return fail(c, D2_ERR_CAPACITY, "d2_find_contacts_bucket_noalloc: at most 131072 hits per call");
  if (total > max_hits) return fail(c, D2_ERR_CAPACITY, "d2_find_contacts_bucket_noalloc: more hits than max_hits");
  return D2_OK;
}

int d2_filter_contacts(d2_ctx* c, int n, const double* reals, double margin, int32_t* sorted_out, int32_t* kept_out,
                       int* n_kept_out) {
  if (!c) return D2_ERR_ARG;
  if (n < 0 || (n > 0 && (!reals || !sorted_out || !kept_out)) || !(margin >= 0.0 || margin < 0.0))
    return fail(c, D2_ERR_ARG, "d2_filter_contacts: bad arguments");
  if (n_kept_out) *n_kept_out = 0;
  if (n == 0) return D2_OK;
  (void)hipSetDevice(c->device);
  const size_t m = (size_t)n;
  RC(ensure(c, c->contacts, m)); RC(ensure(c, c->perm, m)); RC(ensure(c, c->keep, m));
  RC(ensure(c, c->kept_cnt, 2)); RC(ensure(c, c->pair_off, 2)); RC(ensure(c, c->n_big, 2));
  RC(ensure(c, c->big, 1)); RC(ensure(c, c->huge, 1)); RC(ensure(c, c->pair_rec, PR_STRIDE)); RC(ensure(c, c->scale, 1));
  RC(ensure(c, c->bk_out_r, 11 * m)); RC(ensure(c, c->hscratch, 6 * m));
  // the run buffers now hold this call's contacts: no earlier result stays readable
  c->last_mode = -1;
  c->ccd_valid = false;
  HIPCHK(c, hipMemcpyAsync(c->bk_out_r.p, reals, sizeof(double) * 11 * m, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_filter_load, dim3(grid_for(c, n)), dim3(256), 0, c->stream, n, (const double*)c->bk_out_r.p,
                     c->contacts.p, c->perm.p, c->pair_off.p, c->n_big.p);
  launch_finish(c, 1, 1, 1, nullptr, margin);
  HIPCHK(c, hipGetLastError());
  RC(read_out(c, {{sorted_out, c->perm.p, sizeof(int32_t) * m}, {kept_out, c->keep.p, sizeof(int32_t) * m}}));
  int k = 0;  // keep flags per sorted position -> the kept inputs in sorted order
  for (int t = 0; t < n; ++t)
    if (kept_out[t]) kept_out[k++] = sorted_out[t];
  if (n_kept_out) *n_kept_out = k;
  return D2_OK;
}

int d2_narrow(d2_ctx* c, int n_pairs, const int32_t* pairs, int filter, int64_t* n_contacts_out) {
  int rc = d2_pairs_upload(c, n_pairs, pairs, nullptr);
  return rc ? rc : d2_narrow_run(c, filter, n_contacts_out);
}

int d2_ccd(d2_ctx* c, int n_pairs, const int32_t* pairs, const double* max_time, int64_t* n_contacts_out) {
  if (!max_time) return fail(c, D2_ERR_ARG, "d2_ccd: max_time is required");
  int rc = d2_pairs_upload(c, n_pairs, pairs, max_time);
  return rc ? rc : d2_ccd_run(c, n_contacts_out);
}

int d2_result_contacts(d2_ctx* c, int32_t* offsets, int32_t* ints, double* reals) {
  if (!c) return D2_ERR_ARG;
  if (c->last_mode < 0) return fail(c, D2_ERR_STATE, "no result: run the path first");
  const int np = c->n_pairs;
  if (c->out_filtered) {  // the filtered output's offsets (the run only counted its total)
    scan_host_n(c, c->kept_cnt.p, c->out_off.p, np, nullptr);
    HIPCHK(c, hipGetLastError());
  }
  const int* outoff = c->out_filtered ? c->out_off.p : c->pair_off.p;
  if ((ints || reals) && c->n_out > 0) {  // the CSR total and the record count must agree
    int total = 0;
    RC(read_out(c, {{&total, outoff + np, sizeof(int)}}));
    if ((long long)total != c->n_out) return fail(c, D2_ERR_STATE, "result offsets and contact count disagree");
    RC(ensure(c, c->out_i, (size_t)c->n_out * 8)); RC(ensure(c, c->out_r, (size_t)c->n_out * 11));
    const int wblocks = std::max(1, std::min(np, c->cus * 16));
    hipLaunchKernelGGL(k_gather_wave, dim3(wblocks), dim3(64), 0, c->stream, np, c->contacts.p, c->pair_off.p,
                       c->perm.p, c->keep.p, outoff, c->out_filtered ? 1 : 0, c->out_i.p, c->out_r.p);
    HIPCHK(c, hipGetLastError());
  }
  RC(read_out(c, {{offsets, outoff, sizeof(int) * (np + 1)},
                         {ints, c->out_i.p, sizeof(int32_t) * 8 * (size_t)c->n_out},
                         {reals, c->out_r.p, sizeof(double) * 11 * (size_t)c->n_out}}));
  return D2_OK;
}

int d2_result_pairs(d2_ctx* c, double* per_pair) {
  if (!c || !per_pair) return D2_ERR_ARG;
  if (!c->ccd_valid) return fail(c, D2_ERR_STATE, "per-pair results exist after d2_ccd_run or d2_step_run");
  std::vector<double> sc(c->n_pairs), mt(c->n_pairs);
  RC(read_out(c, {{sc.data(), c->scale.p, sizeof(double) * sc.size()},
                         {mt.data(), c->min_time.p, sizeof(double) * mt.size()}}));
  for (int p = 0; p < c->n_pairs; ++p) per_pair[2 * p] = sc[p], per_pair[2 * p + 1] = mt[p];
  return D2_OK;
}

int d2_cluster_steps(d2_ctx* c, const int32_t* cluster_of_pair, int n_clusters, float dt, double* out) {
  if (!c || !cluster_of_pair || !out || n_clusters <= 0) return D2_ERR_ARG;
  if (c->last_mode != 1) return fail(c, D2_ERR_STATE, "d2_cluster_steps needs a preceding d2_ccd_run");
  const int np = c->n_pairs;
  for (int p = 0; p < np; ++p)
    if (cluster_of_pair[p] < 0 || cluster_of_pair[p] >= n_clusters)
      return fail(c, D2_ERR_ARG, "d2_cluster_steps: cluster index out of range");
  RC(ensure_clusters(c, n_clusters)); RC(ensure(c, c->tmp_cluster, std::max(np, 1)));
  if (np) HIPCHK(c, hipMemcpyAsync(c->tmp_cluster.p, cluster_of_pair, sizeof(int32_t) * np, hipMemcpyHostToDevice, c->stream));
  RC(enqueue_clusters(c, c->tmp_cluster.p, n_clusters, dt, false, false, false));
  HIPCHK(c, hipMemcpyAsync(out, c->cluster_step.p, sizeof(double) * n_clusters, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

// ------------------------------------------------ broad phase, clusters
int d2_tree_bounds_upload(d2_ctx* c, const float* aabb6, const double* radius) {
  if (!c || !aabb6 || !radius) return D2_ERR_ARG;
  if (c->n_trees <= 0) return fail(c, D2_ERR_STATE, "d2_tree_bounds_upload: upload trees first");
  for (int t = 0; t < c->n_trees; ++t)
    if (!(radius[t] >= 0.0)) return fail(c, D2_ERR_ARG, "d2_tree_bounds_upload: radius must be >= 0");
  HIPCHK(c, hipMemcpyAsync(c->tb_box.p, aabb6, sizeof(float) * 6 * c->n_trees, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->tb_rad.p, radius, sizeof(double) * c->n_trees, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

int d2_tree_bounds_download(d2_ctx* c, float* aabb6, double* radius) {
  if (!c || !aabb6 || !radius) return D2_ERR_ARG;
  if (c->n_trees <= 0) return fail(c, D2_ERR_STATE, "no trees uploaded");
  HIPCHK(c, hipMemcpyAsync(aabb6, c->tb_box.p, sizeof(float) * 6 * c->n_trees, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(radius, c->tb_rad.p, sizeof(double) * c->n_trees, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

int d2_bodies_last_upload(d2_ctx* c, const double* last14) {
  if (!c || !last14) return D2_ERR_ARG;
  if (c->n_bodies <= 0) return fail(c, D2_ERR_STATE, "d2_bodies_last_upload: upload bodies first");
  HIPCHK(c, hipMemcpyAsync(c->last_state.p, last14, sizeof(double) * 14 * (size_t)c->n_bodies, hipMemcpyHostToDevice,
                           c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

int d2_bodies_groups_upload(d2_ctx* c, const int32_t* group_of_body) {
  if (!c) return D2_ERR_ARG;
  if (c->n_bodies <= 0) return fail(c, D2_ERR_STATE, "d2_bodies_groups_upload: upload bodies first");
  if (!group_of_body) {
    c->has_groups = false;
    return D2_OK;
  }
  for (int i = 0; i < c->n_bodies; ++i)
    if (group_of_body[i] < 0 || group_of_body[i] > (1 << 29))
      return fail(c, D2_ERR_ARG, "d2_bodies_groups_upload: group out of range");
  RC(ensure(c, c->group, c->n_bodies));
  HIPCHK(c, hipMemcpyAsync(c->group.p, group_of_body, sizeof(int32_t) * c->n_bodies, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->has_groups = true;
  return D2_OK;
}

int d2_broad_phase(d2_ctx* c, int mode, double t, int64_t* n_pairs_out) {
  if (!c) return D2_ERR_ARG;
  if (mode != 0 && mode != 1) return fail(c, D2_ERR_ARG, "d2_broad_phase: mode must be 0 or 1");
  if (mode == 0 && !(t >= 0.0 && t < 1e300)) return fail(c, D2_ERR_ARG, "d2_broad_phase: t must be finite and >= 0");
  if (c->n_bodies <= 0) return fail(c, D2_ERR_STATE, "d2_broad_phase: upload bodies first");
  (void)hipSetDevice(c->device);
  // the resident pair list is replaced (and invalid until this call succeeds)
  invalidate_pairs(c);
  const int n = c->n_bodies;
  long long T = 64;
  while (T < 2ll * n) T <<= 1;
  RC(ensure(c, c->bp_box, n)); RC(ensure(c, c->bp_R, n)); RC(ensure(c, c->bp_meta, n));
  RC(ensure(c, c->bp_slot, n)); RC(ensure(c, c->bp_rank, n)); RC(ensure(c, c->bp_members, n));
  RC(ensure(c, c->bp_keys, T)); RC(ensure(c, c->bp_counts, T)); RC(ensure(c, c->bp_start, T + 1));
  RC(ensure(c, c->bp_red, BR_N + 2)); RC(ensure(c, c->bp_fill, 2));
  RC(ensure(c, c->bp_item_cnt, c->n_items)); RC(ensure(c, c->bp_item_pos, c->n_items));
  RC(ensure(c, c->bp_item_sorted, c->n_items)); RC(ensure(c, c->bp_item_off, c->n_items + 1));
  RC(ensure(c, c->scan_part, chunk_grid(c)));
  if (c->bp_cap <= 0) c->bp_cap = std::max<long long>(1 << 16, 8ll * n);
  const int* grp = c->has_groups ? c->group.p : nullptr;
  const int g = grid_for(c, n);
  for (int attempt = 0; attempt < 4; ++attempt) {
    RC(ensure(c, c->bp_chunk, c->bp_cap)); RC(ensure(c, c->pairs, 2 * c->bp_cap)); RC(ensure(c, c->max_time, c->bp_cap));
    hipLaunchKernelGGL(k_bp_clear, dim3(grid_for(c, T)), dim3(256), 0, c->stream, T, c->bp_keys.p, c->bp_counts.p,
                       c->bp_red.p);
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, c->stream, c->bp_fill.p, 2ll, 0ull);
    hipLaunchKernelGGL(k_bp_bounds, dim3(g), dim3(256), 0, c->stream, n, c->bodies.p, c->last_state.p, c->body_tree.p,
                       c->tb_box.p, c->tb_rad.p, grp, mode, t, c->bp_box.p, c->bp_R.p, c->bp_meta.p, c->bp_red.p);
    hipLaunchKernelGGL(k_bp_insert, dim3(g), dim3(256), 0, c->stream, n, c->bp_box.p, c->bp_meta.p, c->bp_red.p, T,
                       c->bp_keys.p, c->bp_counts.p, c->bp_slot.p, c->bp_rank.p);
    scan_host_n(c, c->bp_counts.p, c->bp_start.p, T, nullptr);
    hipLaunchKernelGGL(k_bp_scatter, dim3(g), dim3(256), 0, c->stream, n, c->bp_box.p, c->bp_meta.p, c->bp_slot.p,
                       c->bp_rank.p, c->bp_start.p, c->bp_members.p);
    BpIn in;
    in.n = n, in.mode = mode, in.seg = c->bp_seg, in.t = t, in.bodies = c->bodies.p, in.last = c->last_state.p, in.box = c->bp_box.p;
    in.R = c->bp_R.p, in.meta = c->bp_meta.p, in.statics = c->bp_statics.p, in.n_static = (int)c->host_static.size();
    in.red = c->bp_red.p, in.T = T, in.keys = c->bp_keys.p, in.counts = c->bp_counts.p, in.start = c->bp_start.p;
    in.members = c->bp_members.p;
    const int gi = (int)std::min<long long>((c->n_items + 3) / 4, (long long)c->cus * 16);
    const int gp = (int)std::min<long long>((c->n_items + 4 * BP_BATCH - 1) / (4 * BP_BATCH), (long long)c->cus * 16);
    hipLaunchKernelGGL(k_bp_pairs, dim3(std::max(gp, 1)), dim3(256), 0, c->stream, in, c->n_items, c->bp_item_body.p,
                       c->bp_item_seg.p, c->bp_cap, c->bp_chunk.p, c->bp_fill.p, c->bp_item_cnt.p, c->bp_item_pos.p,
                       c->bp_item_sorted.p, c->bp_red.p);
    scan_host_n(c, c->bp_item_cnt.p, c->bp_item_off.p, c->n_items, c->bp_fill.p + 1);
    hipLaunchKernelGGL(k_bp_gather, dim3(std::max(gi, 1)), dim3(256), 0, c->stream, c->n_items, c->bp_item_cnt.p,
                       c->bp_item_pos.p, c->bp_item_sorted.p, c->bp_item_off.p, c->bp_chunk.p, c->bodies.p,
                       c->body_tree.p, c->tree_depth_d.p, c->pairs.p, c->max_time.p, c->bp_red.p);
    HIPCHK(c, hipGetLastError());
    RC(read_out(c, {{c->host_red, c->bp_red.p, sizeof(int) * BR_N},
                           {c->host_red + BR_N, c->bp_item_off.p + c->n_items, sizeof(int)}}));
    if (c->host_red[BR_ERR] & 1)
      return fail(c, D2_ERR_RUNTIME, "d2_broad_phase: Invalid args for interpolation (state.cpp:56-58)");
    const long long total = c->host_red[BR_N];
    if (c->host_red[BR_OVF]) {
      c->bp_cap = std::max(c->bp_cap * 2, total + total / 4 + 1024);
      continue;
    }
    const int np = (int)total;
    RC(ensure(c, c->pair_rec, (size_t)std::max(np, 1) * PR_STRIDE)); RC(ensure(c, c->pair_info, 4 * (size_t)std::max(np, 1)));
    c->n_pairs = np;
    c->pair_depth = c->host_red[BR_DEPTH];
    c->has_max_time = true;
    c->pairs_valid = true;
    if (n_pairs_out) *n_pairs_out = np;
    return D2_OK;
  }
  return fail(c, D2_ERR_CAPACITY, "d2_broad_phase: pair list kept overflowing");
}

int d2_pairs_download(d2_ctx* c, int32_t* pairs, double* max_time) {
  if (!c) return D2_ERR_ARG;
  const size_t np = (size_t)std::max(c->n_pairs, 0);
  RC(read_out(c, {{pairs, c->pairs.p, sizeof(int32_t) * 2 * np}, {max_time, c->max_time.p, sizeof(double) * np}}));
  return D2_OK;
}

int d2_clusters_build(d2_ctx* c, int* n_clusters_out) {
  if (!c) return D2_ERR_ARG;
  if (c->n_bodies <= 0) return fail(c, D2_ERR_STATE, "d2_clusters_build: upload bodies first");
  if (!c->pairs_valid) return fail(c, D2_ERR_STATE, "d2_clusters_build: upload or build the pair list first");
  (void)hipSetDevice(c->device);
  const int n = c->n_bodies, np = c->n_pairs;
  c->n_clusters = 0;  // invalid until this call succeeds
  c->clusters_on_device = false;
  RC(ensure(c, c->cc_parent, n)); RC(ensure(c, c->cc_label, n)); RC(ensure(c, c->cc_root, n));
  RC(ensure(c, c->cc_root_off, n + 1)); RC(ensure(c, c->cc_of_body, n)); RC(ensure(c, c->cc_first, n));
  RC(ensure(c, c->cc_tmin, n)); RC(ensure(c, c->cc_smin, n)); RC(ensure(c, c->bp_red, BR_N + 2));
  RC(ensure(c, c->cluster_of_pair, std::max(np, 1))); RC(ensure(c, c->scan_part, chunk_grid(c)));
  RC(ensure(c, c->bp_fill, 2));
  const int g = grid_for(c, n), gp = grid_for(c, std::max(np, 1));
  hipLaunchKernelGGL(k_bp_clear, dim3(1), dim3(64), 0, c->stream, 0ll, c->bp_keys.p, c->bp_counts.p, c->bp_red.p);
  hipLaunchKernelGGL(k_cc_init, dim3(g), dim3(256), 0, c->stream, n, c->cc_parent.p);
  if (np > 0)
    hipLaunchKernelGGL(k_cc_union, dim3(gp), dim3(256), 0, c->stream, np, c->pairs.p, c->bodies.p, c->cc_parent.p,
                       c->bp_red.p);
  hipLaunchKernelGGL(k_cc_roots, dim3(g), dim3(256), 0, c->stream, n, c->bodies.p, c->cc_parent.p, c->cc_label.p,
                     c->cc_root.p);
  scan_host_n(c, c->cc_root.p, c->cc_root_off.p, n, nullptr);
  hipLaunchKernelGGL(k_cc_init_cl, dim3(g), dim3(256), 0, c->stream, n, c->cc_tmin.p, c->cc_smin.p);
  hipLaunchKernelGGL(k_cc_assign, dim3(g), dim3(256), 0, c->stream, n, c->bodies.p, c->cc_label.p, c->cc_root_off.p,
                     c->cc_of_body.p, c->cc_first.p, c->cc_tmin.p, c->cc_smin.p);
  if (np > 0)
    hipLaunchKernelGGL(k_cc_pairs, dim3(gp), dim3(256), 0, c->stream, np, c->pairs.p, c->bodies.p, c->cc_of_body.p,
                       c->cluster_of_pair.p);
  hipLaunchKernelGGL(k_cc_rollback, dim3(g), dim3(256), 0, c->stream, n, c->bodies.p, c->last_state.p, c->cc_of_body.p,
                     c->cc_tmin.p, c->bp_red.p);
  HIPCHK(c, hipGetLastError());
  RC(read_out(c, {{c->host_red, c->bp_red.p, sizeof(int) * BR_N}, {c->host_red + BR_N, c->cc_root_off.p + n, sizeof(int)}}));
  if (c->host_red[BR_ERR] & 2)
    return fail(c, D2_ERR_ARG, "d2_clusters_build: a pair of two static bodies belongs to no cluster");
  if (c->host_red[BR_ERR] & 1)
    return fail(c, D2_ERR_RUNTIME, "d2_clusters_build: Invalid args for interpolation (state.cpp:56-58)");
  const int k = c->host_red[BR_N];
  RC(ensure_clusters(c, std::max(k, 1)));
  c->n_clusters = k;
  c->clusters_on_device = true;
  c->ccd_valid = false;
  if (n_clusters_out) *n_clusters_out = k;
  return D2_OK;
}

int d2_clusters_download(d2_ctx* c, int32_t* cluster_of_pair, int32_t* cluster_of_body, int32_t* first,
                         double* min_time, double* step) {
  if (!c) return D2_ERR_ARG;
  if (!c->clusters_on_device) return fail(c, D2_ERR_STATE, "d2_clusters_download needs d2_clusters_build");
  const int n = c->n_bodies, k = c->n_clusters;
  std::vector<long long> tm(min_time ? k : 0);
  std::vector<unsigned long long> sm(step ? k : 0);
  RC(read_out(c, {{cluster_of_pair, c->cluster_of_pair.p, sizeof(int32_t) * (size_t)std::max(c->n_pairs, 0)},
                         {cluster_of_body, c->cc_of_body.p, sizeof(int32_t) * (size_t)n},
                         {first, c->cc_first.p, sizeof(int32_t) * (size_t)k},
                         {tm.data(), c->cc_tmin.p, sizeof(long long) * tm.size()},
                         {sm.data(), c->cc_smin.p, sizeof(long long) * sm.size()}}));
  for (int i = 0; i < (min_time ? k : 0); ++i) {
    long long o = tm[i];
    o = o >= 0 ? o : o ^ 0x7fffffffffffffffll;
    std::memcpy(&min_time[i], &o, sizeof(double));
  }
  for (int i = 0; i < (step ? k : 0); ++i) std::memcpy(&step[i], &sm[i], sizeof(double));
  return D2_OK;
}

// ----------------------------------------------------------- learned gate
namespace {
int mlp_alloc(d2_ctx* c) {
  RC(ensure(c, c->mlp_w, MLP_PARAMS)); RC(ensure(c, c->mlp_m, MLP_PARAMS)); RC(ensure(c, c->mlp_v, MLP_PARAMS));
  RC(ensure(c, c->mlp_wf, MLP_PARAMS)); RC(ensure(c, c->mlp_grad, MLP_PARAMS)); RC(ensure(c, c->mlp_wb, MLP_PARAMS));
  return D2_OK;
}
// Minibatch forward/backward + parameter gradient (grad in c->mlp_grad,
// per-sample losses in c->tr_loss).
void mlp_batch_grad(d2_ctx* c, const int* idx, int nb, float lw0, float lw1, float delta) {
  const int blocks = std::min((nb + MLP_TILE - 1) / MLP_TILE, MLP_MAX_PART);
  hipLaunchKernelGGL(k_mlp_fwd_bwd, dim3(blocks), dim3(256), 0, c->stream, nb, idx, c->tr_x.p, c->tr_t.p,
                     c->mlp_wf.p, lw0, lw1, delta, c->tr_part.p, c->tr_loss.p);
  hipLaunchKernelGGL(k_mlp_grad_sum, dim3((MLP_PARAMS + 63) / 64), dim3(512), 0, c->stream, blocks, c->tr_part.p,
                     c->mlp_grad.p);
}
int mlp_upload_data(d2_ctx* c, const float* X, const float* T, int n, int batch) {
  RC(ensure(c, c->tr_x, (size_t)n * MLP_IN)); RC(ensure(c, c->tr_t, (size_t)n * MLP_OUT));
  RC(ensure(c, c->tr_part, (size_t)MLP_MAX_PART * MLP_PARAMS));
  RC(ensure(c, c->tr_loss, batch)); RC(ensure(c, c->tr_idx, n));
  HIPCHK(c, hipMemcpyAsync(c->tr_x.p, X, sizeof(float) * MLP_IN * (size_t)n, hipMemcpyHostToDevice, c->stream));
  if (T) HIPCHK(c, hipMemcpyAsync(c->tr_t.p, T, sizeof(float) * MLP_OUT * (size_t)n, hipMemcpyHostToDevice, c->stream));
  return D2_OK;
}
}  // namespace

int d2_mlp_num_params(void) { return MLP_PARAMS; }

int d2_mlp_set_params(d2_ctx* c, const float* params) {
  if (!c || !params) return D2_ERR_ARG;
  (void)hipSetDevice(c->device);
  RC(mlp_alloc(c));
  HIPCHK(c, hipMemcpyAsync(c->mlp_w.p, params, sizeof(float) * MLP_PARAMS, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemsetAsync(c->mlp_m.p, 0, sizeof(float) * MLP_PARAMS, c->stream));
  HIPCHK(c, hipMemsetAsync(c->mlp_v.p, 0, sizeof(float) * MLP_PARAMS, c->stream));
  hipLaunchKernelGGL(k_mlp_round, dim3((MLP_PARAMS + 255) / 256), dim3(256), 0, c->stream, c->mlp_w.p, c->mlp_wb.p,
                     c->mlp_wf.p);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->mlp_ready = true;
  c->mlp_step = 0;
  return D2_OK;
}

int d2_mlp_get_params(d2_ctx* c, float* params) {
  if (!c || !params) return D2_ERR_ARG;
  if (!c->mlp_ready) return fail(c, D2_ERR_STATE, "no network parameters set");
  HIPCHK(c, hipMemcpyAsync(params, c->mlp_w.p, sizeof(float) * MLP_PARAMS, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

int d2_mlp_infer(d2_ctx* c, const float* X, int n, float* Y) {
  if (!c || n < 0 || (n > 0 && (!X || !Y))) return D2_ERR_ARG;
  if (!c->mlp_ready) return fail(c, D2_ERR_STATE, "no network parameters set");
  if (n == 0) return D2_OK;
  RC(ensure(c, c->tr_x, (size_t)n * MLP_IN)); RC(ensure(c, c->tr_t, (size_t)n * MLP_OUT));
  HIPCHK(c, hipMemcpyAsync(c->tr_x.p, X, sizeof(float) * MLP_IN * (size_t)n, hipMemcpyHostToDevice, c->stream));
  const int tiles = (n + 15) / 16;
  hipLaunchKernelGGL(k_mlp_infer<false>, dim3(std::max(1, std::min((tiles + 3) / 4, c->cus * 4))), dim3(256), 0,
                     c->stream, n, (const float*)c->tr_x.p, c->mlp_wb.p, c->tr_t.p, FeatIn{});
  HIPCHK(c, hipGetLastError());
  RC(read_out(c, {{Y, c->tr_t.p, sizeof(float) * MLP_OUT * (size_t)n}}));
  return D2_OK;
}

int d2_mlp_loss_grad(d2_ctx* c, const float* X, const float* T, int n, float lw0, float lw1, float delta, float* loss,
                     float* grad) {
  if (!c || !X || !T || n <= 0 || n > (1 << 20)) return D2_ERR_ARG;
  if (!c->mlp_ready) return fail(c, D2_ERR_STATE, "no network parameters set");
  RC(mlp_upload_data(c, X, T, n, n));
  mlp_batch_grad(c, nullptr, n, lw0, lw1, delta);
  HIPCHK(c, hipGetLastError());
  std::vector<float> l(n);
  RC(read_out(c, {{l.data(), c->tr_loss.p, sizeof(float) * n}, {grad, c->mlp_grad.p, sizeof(float) * MLP_PARAMS}}));
  double sum = 0.0;
  for (float v : l) sum += v;
  if (loss) *loss = (float)(sum / n);
  return D2_OK;
}

int d2_mlp_train(d2_ctx* c, const float* X, const float* T, int n, int epochs, int batch, float lr, float lw0,
                 float lw1, float delta, uint64_t seed, float* epoch_loss) {
  if (!c || !X || !T || n <= 0 || epochs <= 0 || batch <= 0 || !(lr > 0.f)) return D2_ERR_ARG;
  if (!c->mlp_ready) return fail(c, D2_ERR_STATE, "set initial network parameters first");
  batch = std::min(batch, n);
  RC(mlp_upload_data(c, X, T, n, batch));
  std::vector<int> idx(n);
  for (int i = 0; i < n; ++i) idx[i] = i;
  std::mt19937_64 rng(seed);
  std::vector<float> l(batch);
  for (int e = 0; e < epochs; ++e) {
    std::shuffle(idx.begin(), idx.end(), rng);
    HIPCHK(c, hipMemcpyAsync(c->tr_idx.p, idx.data(), sizeof(int) * n, hipMemcpyHostToDevice, c->stream));
    double sum = 0.0;
    for (int b0 = 0; b0 < n; b0 += batch) {
      const int nb = std::min(batch, n - b0);
      mlp_batch_grad(c, c->tr_idx.p + b0, nb, lw0, lw1, delta);
      ++c->mlp_step;
      const float b1 = 0.9f, b2 = 0.999f;
      const float c1 = 1.f - std::pow(b1, (float)c->mlp_step), c2 = 1.f - std::pow(b2, (float)c->mlp_step);
      hipLaunchKernelGGL(k_mlp_adam, dim3((MLP_PARAMS + 255) / 256), dim3(256), 0, c->stream, c->mlp_w.p, c->mlp_m.p,
                         c->mlp_v.p, c->mlp_grad.p, lr, b1, b2, 1e-8f, c1, c2, c->mlp_wb.p, c->mlp_wf.p);
      HIPCHK(c, hipGetLastError());
      HIPCHK(c, hipMemcpyAsync(l.data(), c->tr_loss.p, sizeof(float) * nb, hipMemcpyDeviceToHost, c->stream));
      HIPCHK(c, hipStreamSynchronize(c->stream));
      for (int i = 0; i < nb; ++i) sum += l[i];
    }
    if (epoch_loss) epoch_loss[e] = (float)(sum / n);
  }
  drop_graphs(c);  // captured inferences read the weights in place; shapes are unchanged, but be explicit
  return D2_OK;
}

int d2_pair_features(d2_ctx* c, float* X) {
  if (!c || !X) return D2_ERR_ARG;
  if (c->n_pairs <= 0) return D2_OK;
  RC(ensure(c, c->feat, (size_t)c->n_pairs * MLP_IN));
  hipLaunchKernelGGL(k_pair_features, dim3(grid_for(c, c->n_pairs)), dim3(256), 0, c->stream, c->n_pairs, c->pairs.p,
                     c->bodies.p, c->body_tree.p, c->tree_radius.p, c->has_max_time ? c->max_time.p : nullptr,
                     c->feat.p);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipMemcpyAsync(X, c->feat.p, sizeof(float) * MLP_IN * (size_t)c->n_pairs, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

int d2_set_learned(d2_ctx* c, int on, float t_gate, float s_gate) {
  if (!c || on < 0 || on > 3) return D2_ERR_ARG;
  if (on && !c->mlp_ready) return fail(c, D2_ERR_STATE, "set network parameters before turning the gate on");
  c->learned_on = on != 0;
  c->gate_phases = on;
  c->gate_t = t_gate;
  c->gate_s = s_gate;
  return D2_OK;
}

int d2_set_pruning(d2_ctx* c, int on) {
  if (!c) return D2_ERR_ARG;
  if (c->prune_on != (on != 0)) drop_graphs(c);  // captured launches carry the flag
  c->prune_on = on != 0;
  return D2_OK;
}

int d2_set_touch_stats(d2_ctx* c, int on) {
  if (!c) return D2_ERR_ARG;
  // turning it on forgets the last counts; turning it off keeps them readable
  if (on && !c->touch_on) c->touch_host.clear();
  c->touch_on = on != 0;
  return D2_OK;
}

int d2_touch_stats(const d2_ctx* c, int64_t* out, int n) {
  if (!c) return D2_ERR_ARG;
  const int total = TOUCH_RUN + TOUCH_FIELDS;
  if (out)
    for (int i = 0; i < std::min(n, total); ++i) out[i] = i < (int)c->touch_host.size() ? (int64_t)c->touch_host[i] : 0;
  return total;
}

int d2_set_profiling(d2_ctx* c, int on) {
  if (!c) return D2_ERR_ARG;
  c->profiling = on != 0;
  return D2_OK;
}
int d2_num_kernels(void) { return K_NUM; }
const char* d2_kernel_name(int i) { return (i >= 0 && i < K_NUM) ? kKernelNames[i] : ""; }
int d2_kernel_stats(d2_ctx* c, int i, int64_t* launches, double* total_ms, double* items) {
  if (!c || i < 0 || i >= K_NUM) return D2_ERR_ARG;
  collect_timers(c);
  if (launches) *launches = c->k_launch[i];
  if (total_ms) *total_ms = c->k_ms[i];
  if (items) *items = c->k_items[i];
  return D2_OK;
}
int d2_reset_stats(d2_ctx* c) {
  if (!c) return D2_ERR_ARG;
  collect_timers(c);
  for (int i = 0; i < K_NUM; ++i) c->k_launch[i] = 0, c->k_ms[i] = 0.0, c->k_items[i] = 0.0;
  return D2_OK;
}
int d2_run_info(const d2_ctx* c, int64_t* info, int n) {
  if (!c || !info || n < 0) return D2_ERR_ARG;
  const int total = C_COUNT + 2 * (MAX_LEVELS + 1) * LV_STRIDE;
  for (int i = 0; i < n && i < total; ++i)
    info[i] = (int64_t)(i < C_COUNT ? c->host_cnt[i] : c->host_lvl[i - C_COUNT]);
  return total;
}
int d2_graph_stats(const d2_ctx* c, int64_t* captures, int64_t* launches) {
  if (!c || !captures || !launches) return D2_ERR_ARG;
  *captures = c->graph_captures;
  *launches = c->graph_launches;
  return D2_OK;
}
int d2_sync(d2_ctx* c) {
  if (!c) return D2_ERR_ARG;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return D2_OK;
}

}  // extern "C"
