// fl_kernels.hip -- gfx950 kernels of the uplift-erosion iteration.
//
// One outer iteration of fastlem's generate() loop (src/lem/generator.rs:
// 140-210) runs as:
//
//   k_receivers         stream_tree.rs:109-137  steepest-descent receiver,
//                                               first-match edge length
//   lake join (only when a non-outlet site has no receiver):
//     k_sub_*           stream_tree.rs:139-173  chain ends by pointer jumping
//     k_lake_keys       stream_tree.rs:175-243  per lake: 64-bit atomicMin on
//                                               (visit rank << 32 | slot)
//     k_lake_flip                               reverse the lake's flow path
//   tree decomposition (heavy paths, rebuilt every iteration):
//     k_children        children of each site in row (slot) order
//     k_chain_jump      chain head, position in chain, light depth, root
//     k_bucket_*        chains bucketed by light depth, laid out contiguously
//     k_chain_perm      sites scattered to chain-major positions, with
//                                             each site's light children
//   sweeps, every round (light depth) in one launch, deepest first for
//   drainage area
//     k_da_fold         generator.rs:154-159  drainage area along the chains,
//                       generator.rs:172      exact fold order; then each
//                                             site's 1/(K*A^0.5) * distance
//     k_tau_fold        generator.rs:162-203  response time (+ clamped
//                                             elevation), head to tail
//     k_da_tail, k_tau_tail                   rounds behind barriers in one
//                                             workgroup
//     k_tau_scatter     generator.rs:177-202  elevation, changed flag
//
// Per-site kernels take their site ranges XCD by XCD (xcd_block): each of
// the 8 XCDs works on one contiguous eighth of the sites.
//
// Exactness.  Every floating-point expression is evaluated in the order the
// reference writes it; the library is built with -ffp-contract=off so no
// multiply-add is fused.  No floating-point atomics are used: the drainage
// area of site u is folded as
//     A_u = ((a_u + A_{c_m}) + A_{c_{m-1}}) + ... + A_{c_1}
// (children c_1..c_m in row order), which is the association the reference's
// reverse-BFS accumulation produces; response time is a sequential
// root-to-leaf prefix per chain.  Results are therefore bit-identical to the
// reference for the same inputs.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fl_kernels.h"

#define FL_NONE 0xffffffffu
#define FL_LIST_OVERFLOW 0x10000u   // pcnt flag: more light children than listed
#define FL_ROW 8                    // graph row entries loaded together
static_assert(FL_ROW <= FL_LIST, "a row loaded at once fits its position's list");
#define FL_SENT 0x7ff45eed0badf00dull  // a hand-over word without its value (see the sweeps)
#define FL_TAIL 0x20000u            // pcnt flag: the position is its chain's tail
#define FL_HEAD 0x40000u            // ... its chain's head
#define FL_DEST_OVER 0xfffffffeu    // pdest: the receiver reads the chain's word in cover, not a slot

#if defined(__has_builtin)
#if __has_builtin(__hip_atomic_load) && __has_builtin(__hip_atomic_store)
#define FL_DEVICE_ATOMICS 1
#endif
#if __has_builtin(__builtin_amdgcn_update_dpp)
#define FL_WAVE_SHIFT 1
#endif
#endif

namespace {

// Workgroups are dealt to the GPU's 8 XCDs in turn (workgroup b to XCD
// b % 8), each XCD with an L2 of its own.  The per-site kernels hand each XCD
// one contiguous eighth of the index range instead, so that sites close in
// the breadth-first labels, whose neighbour gathers touch the same lines,
// share an L2.  A bijection of [0, gridDim.x) for any grid size.
__device__ __forceinline__ uint32_t xcd_block() {
  const uint32_t nb = gridDim.x, b = blockIdx.x;
  const uint32_t q = nb >> 3, r = nb & 7u, x = b & 7u;
  return x * q + (x < r ? x : r) + (b >> 3);
}

// bs: the workgroup size the kernel was launched with, passed as an argument
// (blockDim.x is read from the dispatch's implicit arguments by a vector load
// that every wavefront would wait for before its first site load)
__device__ __forceinline__ uint32_t gid(uint32_t bs) { return xcd_block() * bs + threadIdx.x; }

// (pointer, count) pairs of the pointer jumping: pointer in the low word,
// count in the high word below FL_FIN, the mark of a pair whose pointer is
// known to be a fixed point (a chain head, a root).  Counts stay below 2^31
// (they count sites).
#define FL_FIN 0x80000000u
#define FL_HOPS 7  // of a jumping round
__device__ __forceinline__ unsigned long long pair(uint32_t ptr, uint32_t cnt) {
  return ((unsigned long long)cnt << 32) | ptr;
}
__device__ __forceinline__ uint32_t pair_ptr(unsigned long long p) { return (uint32_t)p; }
__device__ __forceinline__ uint32_t pair_cnt(unsigned long long p) { return (uint32_t)(p >> 32) & ~FL_FIN; }
__device__ __forceinline__ bool pair_fin(unsigned long long p) { return (p >> 63) != 0; }

// Kinds of an active site (act).  A leaf has no children: its drainage area is
// its own area, and its response time and elevation follow from its receiver's
// alone, so it is on no chain (two of three sites are leaves): chains, sweeps
// and pointer jumping have the other sites only.  A chain ends at a site whose
// heavy child is a leaf, which is then one more of its listed children (the others,
// chosen light by the previous areas, may head chains of their own).
#define FL_ACTIVE 1u
#define FL_LEAF 2u
#define FL_CHAIN_END 4u

// Is slot s of row k (starting at b) a child of k?
__device__ __forceinline__ bool is_child(unsigned long long m, uint32_t deg, uint32_t s, uint32_t b,
                                         const uint32_t* __restrict__ col, const uint32_t* __restrict__ next,
                                         uint32_t k) {
  return deg <= 64 ? ((m >> s) & 1ull) != 0 : next[col[b + s]] == k;
}

// f64::powf(x, 0.5) as lowered in optimised Rust builds.
__device__ __forceinline__ double rust_pow_half(double x) {
  return (x == -__builtin_inf()) ? __builtin_inf() : __builtin_fabs(__builtin_sqrt(x));
}

// f64::max: the non-NaN operand wins.
__device__ __forceinline__ double rust_max(double a, double b) { return __builtin_fmax(a, b); }

// terrain-graph has_edge(a, b): first entry of row a equal to b; 1.0 when
// absent (generator.rs:164-171).
__device__ __forceinline__ double first_len(const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
                                            const double* __restrict__ len, uint32_t a, uint32_t b) {
  uint32_t e1 = rp[a + 1];
  for (uint32_t k = rp[a]; k < e1; ++k)
    if (col[k] == b) return len[k];
  return 1.0;
}

__device__ __forceinline__ double bits_double(unsigned long long u) {
  return __hiloint2double((int)(uint32_t)(u >> 32), (int)(uint32_t)u);
}

// v, quieted if it is the word that stands for no value.
__device__ __forceinline__ double no_word(double v) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  return u == FL_SENT ? bits_double(u | (1ull << 51)) : v;
}

// Synchronisation of one wavefront's lanes around its own LDS tile: a
// wavefront-scope fence (orders the LDS accesses; the wavefront's LDS
// operations execute in order) and a wave barrier.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// v of the next lane (up) or of the previous one (down); the lane at the
// wavefront's edge gets its `edge`.
#ifndef FL_WAVE_SHIFT
__device__ __forceinline__ double shift_lanes(double edge, double v, int from) {
  __shared__ double fl_shift_tile[16][64];
  const int lane = (int)(threadIdx.x & 63u);
  double* t = fl_shift_tile[threadIdx.x >> 6];
  t[lane] = v;
  wave_sync();
  const int src = lane + from;
  const double r = src >= 0 && src < 64 ? t[src] : edge;
  wave_sync();
  return r;
}
__device__ __forceinline__ double from_next(double edge, double v) { return shift_lanes(edge, v, 1); }
__device__ __forceinline__ double from_prev(double edge, double v) { return shift_lanes(edge, v, -1); }
#else
__device__ __forceinline__ double from_next(double edge, double v) {  // DPP wave_shl:1
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), 0x130, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), 0x130, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_prev(double edge, double v) {  // DPP wave_shr:1
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), 0x138, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), 0x138, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
#endif
__device__ __forceinline__ double of_lane(double v, uint32_t lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), (int)lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), (int)lane);
  return __hiloint2double(hi, lo);
}

// Sums over lanes 0..lane.
#ifndef FL_WAVE_SHIFT
__device__ __forceinline__ double prefix_lanes(double v) {
  for (int off = 1; off < 64; off <<= 1) v = v + shift_lanes(0.0, v, -off);
  return v;
}
#else
template <int ctrl, int rows>
__device__ __forceinline__ double plus_dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), ctrl, rows, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), ctrl, rows, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double prefix_lanes(double v) {
  v = plus_dpp<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8 within rows of 16 lanes
  v = plus_dpp<0x112, 0xf>(v);
  v = plus_dpp<0x114, 0xf>(v);
  v = plus_dpp<0x118, 0xf>(v);
  v = plus_dpp<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = plus_dpp<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}
#endif
__device__ __forceinline__ bool same_bits(double a, double b) {
  return __double_as_longlong(a) == __double_as_longlong(b);
}

}  // namespace

// ------------------------------------------------------------ receivers ---

// next[i]: the neighbour with the strictly largest positive slope
// (h_i - h_j)/len, earliest slot on ties; i itself for outlets and pits.
// flags[FL_FLAG_LAKE] is raised when a non-outlet site has no receiver.
// A receiver depends on the site's and its neighbours' elevations only: with
// chg_prev (per-site flags, raised where the previous iteration, whose tree
// had no lake joins, changed the elevation of the site or of a neighbour), a
// site whose neighbourhood did not change keeps its previous receiver and
// distance.  chg_out (this iteration's flags) is zeroed here for
// k_tau_scatter to mark.
//
// With `dirty` (cleared by the previous iteration's k_tau_scatter), a site
// whose receiver or receiver distance differs from the previous tree's
// marks the previous basins of itself, its new and its old receiver as
// recomputed (the marks of k_dirty, made here without a launch of their
// own).
__global__ void k_receivers(uint32_t bs, uint32_t n, const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
                            const double* __restrict__ len, const double* __restrict__ h,
                            const uint8_t* __restrict__ is_outlet, uint32_t* __restrict__ next,
                            double* __restrict__ dnext, int* __restrict__ flags,
                            const uint8_t* __restrict__ chg_prev, const uint32_t* __restrict__ next_prev,
                            const double* __restrict__ dnext_prev, const uint32_t* __restrict__ root_prev,
                            uint8_t* __restrict__ dirty, uint8_t* __restrict__ chg_out) {
  uint32_t i = gid(bs);
  if (i >= n) return;
  chg_out[i] = 0;  // this iteration's k_tau_scatter marks the changed neighbourhoods
  // the site's own words are loaded together, before the outlet test
  const bool prev = chg_prev || dirty;
  const uint8_t outlet = is_outlet[i];
  const uint32_t b = rp[i], e = rp[i + 1];
  const uint32_t pj = prev ? next_prev[i] : 0u;
  const double pd = prev ? dnext_prev[i] : 0.0;
  if (outlet) {
    next[i] = i;
    dnext[i] = 1.0;
    return;
  }
  if (chg_prev && chg_prev[i] == 0) {
    if (pj == i) flags[FL_FLAG_LAKE] = 1;
    next[i] = pj;
    dnext[i] = pd;
    return;
  }
  // a row is read FL_ROW entries at a time, every load of a group issued
  // before the first is used (indices past the row's end repeat its last
  // entry and are not evaluated)
  uint32_t c[FL_ROW];
  const double hi = h[i];
  double best = 0.0, d = 1.0;
  uint32_t bj = i;
  for (uint32_t k = b; k < e; k += FL_ROW) {
#pragma unroll
    for (int j = 0; j < FL_ROW; ++j) c[j] = col[min(k + j, e - 1)];
    double hj[FL_ROW], lk[FL_ROW];
#pragma unroll
    for (int j = 0; j < FL_ROW; ++j) {
      hj[j] = h[c[j]];
      lk[j] = len[min(k + j, e - 1)];
    }
    // slots in row order: the earliest of equal slopes is kept
#pragma unroll
    for (int j = 0; j < FL_ROW; ++j) {
      if (k + j < e && hi > hj[j]) {
        double s = (hi - hj[j]) / lk[j];
        if (s > best) {
          best = s;
          bj = c[j];
          d = lk[j];  // rows hold no duplicate edges: this slot is has_edge(i, bj)'s
        }
      }
    }
  }
  if (bj == i) flags[FL_FLAG_LAKE] = 1;
  next[i] = bj;
  dnext[i] = d;
  if (dirty) {
    if (bj != pj || __double_as_longlong(d) != __double_as_longlong(pd)) {
      dirty[root_prev[i]] = 1;
      dirty[root_prev[bj]] = 1;
      dirty[root_prev[pj]] = 1;
    }
  }
}

// ------------------------------------------------------------ lake join ---

__global__ void k_fill_u64(uint32_t bs, uint32_t n, uint64_t* __restrict__ dst, uint64_t v) {
  uint32_t i = gid(bs);
  if (i < n) dst[i] = v;
}

__global__ void k_fill_u32(uint32_t bs, uint32_t n, uint32_t* __restrict__ dst, uint32_t v) {
  uint32_t i = gid(bs);
  if (i < n) dst[i] = v;
}

// Chain ends of the receiver forest by pointer jumping: four receivers ahead,
// then rounds in place of three hops (the reach quadruples; a pointer read while
// its owner rewrites it is an older or a newer one of the same path), then the
// rest of the way, which is short after enough rounds for the usual path.
// Nothing is read back in between, so lakes cost no synchronisation (ten of them
// when every round was checked).  The last kernel empties the lakes' keys.
__global__ void k_sub_start(uint32_t bs, uint32_t n, const uint32_t* __restrict__ next, uint32_t* __restrict__ sub) {
  uint32_t i = gid(bs);
  if (i < n) sub[i] = next[next[next[next[i]]]];
}

__global__ void k_sub_jump(uint32_t bs, uint32_t n, uint32_t* sub) {
  uint32_t i = gid(bs);
  if (i >= n) return;
  const uint32_t a = __atomic_load_n(sub + i, __ATOMIC_RELAXED);
  const uint32_t b = __atomic_load_n(sub + a, __ATOMIC_RELAXED);
  if (b == a) return;
  const uint32_t c = __atomic_load_n(sub + b, __ATOMIC_RELAXED);
  __atomic_store_n(sub + i, __atomic_load_n(sub + c, __ATOMIC_RELAXED), __ATOMIC_RELAXED);
}

__global__ void k_sub_settle(uint32_t bs, uint32_t n, uint32_t* sub, unsigned long long* __restrict__ key) {
  uint32_t i = gid(bs);
  if (i >= n) return;
  key[i] = ~0ull;
  const uint32_t a = __atomic_load_n(sub + i, __ATOMIC_RELAXED);
  uint32_t s = a;
  for (;;) {
    const uint32_t t = __atomic_load_n(sub + s, __ATOMIC_RELAXED);
    if (t == s) break;
    s = t;
  }
  if (s != a) __atomic_store_n(sub + i, s, __ATOMIC_RELAXED);
}

// For every reached site i and every neighbour j lying in a different
// chain whose end is a non-outlet pit (a lake), offer the key
// (visit rank of i) << 32 | slot to that lake.  The minimum key names the
// site i* and the slot of j* through which the reference's traversal first
// touches the lake (stream_tree.rs:204-230).
__global__ void k_lake_keys(uint32_t bs, uint32_t n, const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
                            const uint32_t* __restrict__ rank, const uint32_t* __restrict__ sub,
                            const uint8_t* __restrict__ is_outlet, unsigned long long* __restrict__ key) {
  uint32_t i = gid(bs);
  if (i >= n) return;
  uint32_t r = rank[i];
  if (r == FL_NONE) return;
  uint32_t si = sub[i];
  uint32_t b = rp[i], e = rp[i + 1];
  for (uint32_t k = b; k < e; ++k) {
    uint32_t s = sub[col[k]];
    if (s != si && !is_outlet[s]) {
      unsigned long long kv = ((unsigned long long)r << 32) | (unsigned long long)(k - b);
      atomicMin(key + s, kv);
    }
  }
}

// The same keys offered from the lakes' side: each site j of a lake looks its
// neighbours' slots for it up in their rows (rows are symmetric and without
// duplicates).  For the later iterations, whose lakes are a few sites
// (3.4 us at a million sites, where k_lake_keys takes 51 to 81).
__global__ void k_lake_offers(uint32_t bs, uint32_t n, const uint32_t* __restrict__ rp,
                              const uint32_t* __restrict__ col, const uint32_t* __restrict__ rank,
                              const uint32_t* __restrict__ sub, const uint8_t* __restrict__ is_outlet,
                              unsigned long long* __restrict__ key) {
  uint32_t j = gid(bs);
  if (j >= n) return;
  const uint32_t s = sub[j];
  if (is_outlet[s]) return;
  for (uint32_t k = rp[j]; k < rp[j + 1]; ++k) {
    const uint32_t i = col[k], r = rank[i];
    if (r == FL_NONE || sub[i] == s) continue;
    const uint32_t b = rp[i], e = rp[i + 1];
    uint32_t x = b;
    while (x < e && col[x] != j) ++x;
    if (x < e) atomicMin(key + s, ((unsigned long long)r << 32) | (unsigned long long)(x - b));
  }
}

// One thread per lake (indexed by its pit s): reverse the flow path from j*
// to the pit so that j* drains into i* (stream_tree.rs:214-229) and refresh
// the receiver distances of the reversed sites.  Lakes are disjoint, so all
// flips run concurrently without conflicts.
__global__ void k_lake_flip(uint32_t bs, uint32_t n, const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
                            const double* __restrict__ len, const uint32_t* __restrict__ order,
                            const unsigned long long* __restrict__ key, const uint8_t* __restrict__ is_outlet,
                            uint32_t* __restrict__ next, double* __restrict__ dnext) {
  uint32_t s = gid(bs);
  if (s >= n) return;
  if (is_outlet[s] || next[s] != s) return;
  unsigned long long kv = key[s];
  if (kv == ~0ull) return;  // never reached: stays a pit, as in the reference
  uint32_t istar = order[(uint32_t)(kv >> 32)];
  uint32_t jstar = col[rp[istar] + (uint32_t)(kv & 0xffffffffu)];
  uint32_t k = jstar, nk = istar;
  for (uint32_t guard = 0; guard <= n; ++guard) {
    uint32_t nx = next[k];
    if (nx == k) break;
    next[k] = nk;
    dnext[k] = first_len(rp, col, len, k, nk);
    nk = k;
    k = nx;
  }
  next[k] = nk;
  dnext[k] = first_len(rp, col, len, k, nk);
}

// ------------------------------------------------------- decomposition ----

// Children of u are the neighbours v with next[v] == u, in row order (the
// order DrainageBasin::construct appends them, drainage_basin.rs:23-27).
// cmask[u] bit s marks slot s as a child (rows of up to 64 entries; longer
// rows are rescanned by the consumers).  The heavy child (first with the
// largest previous drainage area) continues u's chain; the choice only
// shapes the work, never the results.
// Basins of the previous iteration's tree that are recomputed: those holding
// a site whose receiver or receiver distance changed, or that site's old or
// new receiver (k_receivers marks those of raw receivers; this kernel runs
// after a lake join changed receivers).  Any other basin keeps every parent pointer and distance of
// its tree, and no site of another basin attaches to it, so its drainage
// areas, response times and elevations come out bit for bit as before.
__global__ void k_dirty(uint32_t bs, uint32_t n, const uint32_t* __restrict__ next, const double* __restrict__ dnext,
                        const uint32_t* __restrict__ next_prev, const double* __restrict__ dnext_prev,
                        const uint32_t* __restrict__ root_prev, uint8_t* __restrict__ dirty) {
  uint32_t v = gid(bs);
  if (v >= n) return;
  const uint32_t a = next[v], b = next_prev[v];
  if (a != b || __double_as_longlong(dnext[v]) != __double_as_longlong(dnext_prev[v])) {
    dirty[root_prev[v]] = 1;
    dirty[root_prev[a]] = 1;
    dirty[root_prev[b]] = 1;
  }
}

// Child slots and heavy child of every active site; act[u] (read by the
// iteration's later kernels): u belongs to a dirty basin (every site when
// `dirty` is null) of a terrain still iterating (tid, t_active: per-site
// terrain and per-terrain mask of a union, or null).  Also the chain and
// root pointers for pointer jumping, written by each site for its children
// (every child of an active site is active, and every active site is a root
// or a child of one):
//   cp: (chain parent, 1), (v, 0) at a chain head
//   rt: (receiver, 1 at a head that is not a root: a light edge), (v, 0) at a root
// An inactive site keeps its basin: its root is carried to this iteration's.
__global__ void k_children(uint32_t bs, uint32_t n, const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
                           const uint32_t* __restrict__ next, const double* __restrict__ prev_area,
                           unsigned long long* __restrict__ cmask, uint32_t* __restrict__ hc,
                           uint8_t* __restrict__ act, const uint8_t* __restrict__ dirty,
                           const uint32_t* __restrict__ root_prev, const uint32_t* __restrict__ tid,
                           const uint8_t* __restrict__ t_active, unsigned long long* __restrict__ cp,
                           unsigned long long* __restrict__ rt, uint32_t* __restrict__ root_out) {
  uint32_t u = gid(bs);
  if (u >= n) return;
  // the site's own words together (an inactive site reads its receiver and
  // row for nothing: one load latency less for the active ones)
  const uint32_t ru = root_prev[u], nu = next[u], b = rp[u], e = rp[u + 1];
  const uint32_t tu = tid ? tid[u] : 0u;
  bool a = !dirty || dirty[ru];
  if (tid) a = a && t_active[tu];
  act[u] = a ? 1 : 0;
  if (!a) {
    root_out[u] = ru;
    return;
  }
  if (nu == u) {
    cp[u] = pair(u, FL_FIN);
    rt[u] = pair(u, FL_FIN);
  }
  uint32_t heavy = FL_NONE;
  unsigned long long m = 0;
  double best = 0.0;
  for (uint32_t k = b; k < e; k += FL_ROW) {
    // FL_ROW neighbours at a time, every load issued before the first is
    // used (indices past the row's end repeat its last entry, not evaluated)
    uint32_t c[FL_ROW], nx[FL_ROW];
    double av[FL_ROW];
#pragma unroll
    for (int j = 0; j < FL_ROW; ++j) c[j] = col[min(k + j, e - 1)];
#pragma unroll
    for (int j = 0; j < FL_ROW; ++j) {
      nx[j] = next[c[j]];
      av[j] = prev_area[c[j]];
    }
#pragma unroll
    for (int j = 0; j < FL_ROW; ++j) {
      if (k + j < e && nx[j] == u) {
        const uint32_t v = c[j];
        if (heavy == FL_NONE || av[j] > best) {
          best = av[j];
          heavy = v;
        }
        if (k + j - b < 64) m |= 1ull << (k + j - b);
        // a light child heads its chain (the heavy one is set below)
        cp[v] = pair(v, FL_FIN);
        rt[v] = pair(u, 1u);
      }
    }
  }
  cmask[u] = m;
  hc[u] = heavy;
  if (heavy != FL_NONE) {
    cp[heavy] = pair(u, 1u);
    rt[heavy] = pair(u, 0u);
  }
}

// One jumping round on both pointer systems, in place:
// (a, d) <- (a', d + d') with (a', d') the pair of a, FL_HOPS times (the reach
// grows by a factor of FL_HOPS + 1).  A pair read while its owner rewrites it is
// either its old or its new value (aligned 64-bit accesses are single-copy
// atomic), and both are (ancestor, count) pairs of the same path, so rounds may
// mix them.  After convergence
// cp[v] = (chain head, position in chain), rt[v] = (root of v's tree, light
// edges between v and the root = light depth of v's chain).
//
// Seven hops: a launch is 2 us and its gap before the first load, a hop less
// than 0.7 us for those not at the end, fewer each time.  A solve takes with 3, 5,
// 7, 11, 15 hops: 1M sites 28.4, 28.2, 27.7, 28.0, 28.2 ms; 10k 2.52, 2.45, 2.41,
// 2.43, 2.40; strip 39.5, 38.7, 38.5, 39.1, 38.8.
//
// Fixed points (a head's cp, a root's rt: pairs (x, 0) of x itself) carry
// FL_FIN, and so does a pair that reaches one.  A marked pair never changes and
// its site loads nothing more.  A round flags, in its own control word (zeroed at
// the start of the iteration), whether some pair is still unmarked after it: a
// round without the flag proves convergence in the round that completes it, and
// the rounds launched after it return at once.
//
// The first round also tells the kinds of the sites (hc: heavy children, all
// made by k_children); leaves take part in none.
__global__ void k_chain_jump(uint32_t bs, uint32_t n, unsigned long long* cp, unsigned long long* rt,
                             uint32_t* __restrict__ flag_set, const uint32_t* __restrict__ prev_flag,
                             uint8_t* __restrict__ act, const uint32_t* __restrict__ hc,
                             uint32_t* __restrict__ head_base) {
  uint32_t v = gid(bs);
  // the site's own pairs are read together with the previous round's flag
  // (an inactive site's pairs are stale and unused: no active site points
  // at one, as a dirty basin holds its sites' whole paths)
  bool on = v < n && (act[v] & (FL_ACTIVE | FL_LEAF)) == FL_ACTIVE;
  if (!prev_flag && on) {
    const uint32_t hk = hc[v];
    if (hk == FL_NONE) {
      act[v] = FL_ACTIVE | FL_LEAF;
      head_base[v] = FL_NONE;  // no chain's head
      on = false;
    } else if (hc[hk] == FL_NONE) {
      act[v] = FL_ACTIVE | FL_CHAIN_END;
    }
  }
  unsigned long long c = 0, r = 0;
  if (on) {
    c = __atomic_load_n(cp + v, __ATOMIC_RELAXED);
    r = __atomic_load_n(rt + v, __ATOMIC_RELAXED);
  }
  // a round after a round that left every pair marked has nothing to do
  if (prev_flag && *prev_flag == 0) return;
  bool open = false;
  if (on) {
    // FL_HOPS hops on both; a pair at a fixed point's is (x, 0) of x itself and
    // marks the pair that reaches it
    const bool oc = !pair_fin(c), orr = !pair_fin(r);
    uint32_t dc = pair_cnt(c), dr = pair_cnt(r);
#pragma unroll
    for (int hop = 0; hop < FL_HOPS; ++hop) {
      const bool mc = !pair_fin(c), mr = !pair_fin(r);
      const unsigned long long nc = mc ? __atomic_load_n(cp + pair_ptr(c), __ATOMIC_RELAXED) : c;
      const unsigned long long nr = mr ? __atomic_load_n(rt + pair_ptr(r), __ATOMIC_RELAXED) : r;
      if (mc) dc += pair_cnt(nc);
      if (mr) dr += pair_cnt(nr);
      c = nc;
      r = nr;
    }
    if (oc) {
      __atomic_store_n(cp + v, pair(pair_ptr(c), dc | (pair_fin(c) ? FL_FIN : 0u)), __ATOMIC_RELAXED);
      open = open || !pair_fin(c);
    }
    if (orr) {
      __atomic_store_n(rt + v, pair(pair_ptr(r), dr | (pair_fin(r) ? FL_FIN : 0u)), __ATOMIC_RELAXED);
      open = open || !pair_fin(r);
    }
  }
  if (__any(open) && (threadIdx.x & 63u) == 0) *flag_set = 1;
}

// v's pair p at its fixed point.  Most are after as many rounds as the
// previous iteration's tree took; the others of a tree that needs more hop on
// here, so that no round is launched only to prove that all are.  Bounded by the
// path, which holds for a whole tree only: never called before the guard is seen
// to be down (the pairs of an iteration behind a too deep decomposition are those
// of two trees, and may lead in a circle).
__device__ __forceinline__ unsigned long long settle(unsigned long long p, const unsigned long long* pairs) {
  while (!pair_fin(p)) {
    const unsigned long long q = __atomic_load_n(pairs + pair_ptr(p), __ATOMIC_RELAXED);
    if (pair_ptr(q) == pair_ptr(p)) break;
    p = pair(pair_ptr(q), (pair_cnt(p) + pair_cnt(q)) | (pair_fin(q) ? FL_FIN : 0u));
  }
  return p;
}

// Buckets: 2 * light depth + (chain length >= long_min), so every round
// has a range of short chains followed by long ones; long_min is a launch
// parameter (tuned; any value >= 1 gives the same results).  A short bucket
// counts its chains, a long one the tiles of its chains: FL_TILE positions
// each, counted from the chain's head (its tail's tile may hold fewer).
#define FL_TILE 128
#define FL_CHAIN_PART 0x80000000u  // cmeta.y: not the tile of the chain's head (the tile's end, else the length)
#define FL_CHAIN_TAIL 0x80000000u  // cmeta.x: the tile of the chain's tail
__device__ __forceinline__ uint32_t bucket_weight(uint32_t len, uint32_t long_min) {
  return len >= long_min ? (len + FL_TILE - 1) / FL_TILE : 1u;
}
#define FL_LDS_BUCKETS 128
#define FL_BUCKET_BLOCK 1024
#define FL_BUCKET_PER_THREAD 2

// The chain tails among a thread's FL_BUCKET_PER_THREAD sites of the
// workgroup's range starting at `base`, with their pairs as they are: the kind of
// every site loaded first (clamped in range, all together), the pairs of the tails
// second.  Nothing is followed here: these loads are in flight while the guard is
// read, and settle_tails comes after it.
struct fl_tail {
  unsigned long long r, c;
  bool t, leaf;
};
__device__ __forceinline__ void load_tails(uint32_t base, uint32_t n, const unsigned long long* __restrict__ cp,
                                           const unsigned long long* __restrict__ rt,
                                           const uint8_t* __restrict__ act, fl_tail (&q)[FL_BUCKET_PER_THREAD]) {
  uint8_t a[FL_BUCKET_PER_THREAD];
#pragma unroll
  for (uint32_t j = 0; j < FL_BUCKET_PER_THREAD; ++j) {
    const uint32_t v = base + j * FL_BUCKET_BLOCK + threadIdx.x;
    a[j] = act[v < n ? v : n - 1];
  }
#pragma unroll
  for (uint32_t j = 0; j < FL_BUCKET_PER_THREAD; ++j) {
    const uint32_t v = base + j * FL_BUCKET_BLOCK + threadIdx.x;
    q[j].t = v < n && (a[j] & FL_CHAIN_END);
    q[j].r = q[j].t ? rt[v] : 0ull;
    q[j].c = q[j].t ? cp[v] : 0ull;
    q[j].leaf = v < n && (a[j] & FL_LEAF);
  }
}
// The tails' pairs at their fixed points, and the outlet flag of their roots
// (without lakes every root is an outlet: is_outlet is null and this load, 0.7 us
// in each kernel of the decomposition, is left out).
__device__ __forceinline__ void settle_tails(const unsigned long long* __restrict__ cp,
                                             const unsigned long long* __restrict__ rt,
                                             const uint8_t* __restrict__ is_outlet,
                                             fl_tail (&q)[FL_BUCKET_PER_THREAD]) {
#pragma unroll
  for (uint32_t j = 0; j < FL_BUCKET_PER_THREAD; ++j)
    if (q[j].t) {
      q[j].r = settle(q[j].r, rt);
      q[j].c = settle(q[j].c, cp);
      if (is_outlet) q[j].t = is_outlet[pair_ptr(q[j].r)] != 0;
    }
}

// Light-depth histogram of the chains (buckets' counts and total length), aggregated
// per workgroup in LDS before one global atomic per (workgroup, bucket).
// Each chain is counted by its tail, which knows the chain's length (its
// position + 1) and light depth; leaves_of: each workgroup's leaves (for the
// statistics; summed with the offsets, as one more atomic a workgroup on one word
// took 4 us at a million sites).
__global__ void __launch_bounds__(FL_BUCKET_BLOCK)
k_bucket_count(const uint32_t* __restrict__ guard, uint32_t n, const unsigned long long* __restrict__ cp,
               const unsigned long long* __restrict__ rt, const uint8_t* __restrict__ is_outlet,
               uint32_t* __restrict__ bcnt, uint32_t* __restrict__ bnodes, uint32_t* __restrict__ counters,
               uint32_t* __restrict__ leaves_of,
               uint32_t long_min, const uint8_t* __restrict__ act) {
  const uint32_t base = xcd_block() * (FL_BUCKET_BLOCK * FL_BUCKET_PER_THREAD);
  fl_tail q[FL_BUCKET_PER_THREAD];
  load_tails(base, n, cp, rt, act, q);  // in flight while the guard is read
  if (*guard) return;  // the iteration is redone
  settle_tails(cp, rt, is_outlet, q);
  __shared__ uint32_t s_c[FL_LDS_BUCKETS], s_n[FL_LDS_BUCKETS];
  __shared__ uint32_t s_max, s_leaves;
  for (uint32_t t = threadIdx.x; t < FL_LDS_BUCKETS; t += FL_BUCKET_BLOCK) {
    s_c[t] = 0;
    s_n[t] = 0;
  }
  if (threadIdx.x == 0) {
    s_max = 0;
    s_leaves = 0;
  }
  __syncthreads();
  for (uint32_t j = 0; j < FL_BUCKET_PER_THREAD; ++j) {
    const unsigned long long leaves = __ballot(q[j].leaf);
    if ((threadIdx.x & 63u) == 0 && leaves) atomicAdd(&s_leaves, (uint32_t)__builtin_popcountll(leaves));
    if (q[j].t) {
      uint32_t lw = pair_cnt(q[j].r), len = pair_cnt(q[j].c) + 1, l = 2u * lw + (len >= long_min ? 1u : 0u);
      const uint32_t wt = bucket_weight(len, long_min);
      if (l < FL_LDS_BUCKETS) {
        atomicAdd(s_c + l, wt);
        atomicAdd(s_n + l, len);
      } else {
        atomicAdd(bcnt + l, wt);
        atomicAdd(bnodes + l, len);
      }
      atomicMax(&s_max, lw);
    }
  }
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < FL_LDS_BUCKETS; t += FL_BUCKET_BLOCK) {
    if (s_c[t]) {
      atomicAdd(bcnt + t, s_c[t]);
      atomicAdd(bnodes + t, s_n[t]);
    }
  }
  if (threadIdx.x == 0) {
    atomicMax(counters + FL_CNT_MAXLD, s_max);
    leaves_of[blockIdx.x] = s_leaves;
  }
}

// Exclusive scans of the bucket histograms over the light depths actually
// present (2 * (counters[FL_CNT_MAXLD] + 1) buckets), one workgroup.  The first
// FL_CTRL_HEAD + 1 offsets are mirrored into the control block.  ucum[l]: the
// sweep units (see the sweeps) of the rounds before round l.
#define FL_SCAN_BLOCK 1024  // k_bucket_scan: one workgroup of this size
__global__ void __launch_bounds__(FL_SCAN_BLOCK)
k_bucket_scan(uint32_t n, uint32_t long_min, uint32_t* __restrict__ ctrl,
                              const uint32_t* __restrict__ bcnt, const uint32_t* __restrict__ bnodes,
                              uint32_t* __restrict__ boff, uint32_t* __restrict__ bnoff,
                              uint32_t* __restrict__ ucum, uint32_t groups, const uint32_t* __restrict__ leaves_of) {
  __shared__ uint32_t s_leaves;
  __shared__ uint32_t s_a[FL_SCAN_BLOCK], s_b[FL_SCAN_BLOCK];
  __shared__ uint32_t s_u[FL_SCAN_BLOCK];
  __shared__ uint32_t carry_a, carry_b, carry_u;
  const uint32_t stride = 65u - long_min;
  uint32_t* counters = ctrl + FL_NUM_FLAGS;
  uint32_t nb = 2 * (counters[FL_CNT_MAXLD] + 1);
  if (nb > n + 2) nb = n + 2;
  uint32_t* head_c = counters + FL_NUM_COUNTERS;
  uint32_t* head_n = head_c + FL_CTRL_HEAD + 1;
  if (threadIdx.x == 0) {
    carry_a = 0;
    carry_b = 0;
    carry_u = 0;
    s_leaves = 0;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < groups; i += FL_SCAN_BLOCK) atomicAdd(&s_leaves, leaves_of[i]);
  __syncthreads();
  for (uint32_t base = 0; base < nb; base += FL_SCAN_BLOCK) {
    uint32_t i = base + threadIdx.x;
    uint32_t a = i < nb ? bcnt[i] : 0, b = i < nb ? bnodes[i] : 0;
    // a round's units in its second bucket's place: its long chains' tiles
    // and the tiles of its short chains' positions
    uint32_t q = (i & 1u) && i < nb ? a + (bnodes[i - 1] + stride - 1) / stride : 0u;
    s_a[threadIdx.x] = a;
    s_b[threadIdx.x] = b;
    s_u[threadIdx.x] = q;
    __syncthreads();
    for (uint32_t off = 1; off < FL_SCAN_BLOCK; off <<= 1) {
      uint32_t ta = threadIdx.x >= off ? s_a[threadIdx.x - off] : 0;
      uint32_t tb = threadIdx.x >= off ? s_b[threadIdx.x - off] : 0;
      uint32_t tu = threadIdx.x >= off ? s_u[threadIdx.x - off] : 0;
      __syncthreads();
      s_a[threadIdx.x] += ta;
      s_b[threadIdx.x] += tb;
      s_u[threadIdx.x] += tu;
      __syncthreads();
    }
    if (i < nb) {
      uint32_t oa = carry_a + s_a[threadIdx.x] - a, ob = carry_b + s_b[threadIdx.x] - b;
      boff[i] = oa;
      bnoff[i] = ob;
      if ((i & 1u) == 0) ucum[i >> 1] = carry_u + s_u[threadIdx.x];  // (its own round's sit at i + 1)
      if (i <= FL_CTRL_HEAD) {
        head_c[i] = oa;
        head_n[i] = ob;
      }
    }
    __syncthreads();
    if (threadIdx.x == FL_SCAN_BLOCK - 1) {
      carry_a += s_a[threadIdx.x];
      carry_b += s_b[threadIdx.x];
      carry_u += s_u[threadIdx.x];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    boff[nb] = carry_a;
    bnoff[nb] = carry_b;
    ucum[nb >> 1] = carry_u;
    if (nb <= FL_CTRL_HEAD) {
      head_c[nb] = carry_a;
      head_n[nb] = carry_b;
    }
    counters[FL_CNT_LEAVES] = s_leaves;
    counters[FL_CNT_CHAINS] = carry_a;
    counters[FL_CNT_POSITIONS] = carry_b;
  }
}

// Give every chain (through its tail) a slot in its light-depth bucket and a
// contiguous range of positions: LDS atomics rank the chains of a workgroup,
// one global atomic per (workgroup, bucket) reserves the ranges.  Order
// inside a bucket is immaterial to the results.  A long chain has a record
// per tile, the tail's first, (base, end of the tile), the head's (base, len);
// a chain's head knows its base, and the base's receiver slot starts empty.
__device__ __forceinline__ void place_chain(uint32_t q, uint32_t pos, uint32_t len, uint32_t hd, uint32_t long_min,
                                            uint2* __restrict__ cmeta, uint32_t* __restrict__ head_base,
                                            uint32_t* __restrict__ pdest) {
  if (len >= long_min) {
    uint32_t end = len;
    for (; end > FL_TILE; end = (end - 1) & ~(FL_TILE - 1u))
      cmeta[q++] = make_uint2(pos | (end == len ? FL_CHAIN_TAIL : 0u), end | FL_CHAIN_PART);
    cmeta[q] = make_uint2(pos | (end == len ? FL_CHAIN_TAIL : 0u), len);
  }
  head_base[hd] = pos;
  pdest[pos] = FL_NONE;
}

// `scan`: the bucket offsets are not there yet (no k_bucket_scan before it).
// Every workgroup makes them for itself, one wavefront over the at most 64
// rounds, and the first stores them: a launch of 4.5 us and its gap less.  A
// decomposition with more rounds raises the guard (the iteration is redone).
struct fl_bucket_out {
  uint32_t *boff, *bnoff, *ucum, *ctrl;
  const uint32_t* leaves_of;
};
template <bool scan>
__global__ void __launch_bounds__(FL_BUCKET_BLOCK)
k_bucket_place(uint32_t* __restrict__ guard, uint32_t n, const unsigned long long* __restrict__ cp,
               const unsigned long long* __restrict__ rt, const uint8_t* __restrict__ is_outlet,
               const uint32_t* __restrict__ bcnt, const uint32_t* __restrict__ bnodes,
               fl_bucket_out o, uint32_t* __restrict__ bcur, uint32_t* __restrict__ bncur,
               uint2* __restrict__ cmeta, uint32_t* __restrict__ pdest,
               uint32_t* __restrict__ head_base, uint32_t long_min, const uint8_t* __restrict__ act) {
  const uint32_t base = xcd_block() * (FL_BUCKET_BLOCK * FL_BUCKET_PER_THREAD);
  fl_tail tl[FL_BUCKET_PER_THREAD];
  __shared__ uint32_t s_c[FL_LDS_BUCKETS], s_n[FL_LDS_BUCKETS], s_bc[FL_LDS_BUCKETS], s_bn[FL_LDS_BUCKETS];
  __shared__ uint32_t s_boff[FL_LDS_BUCKETS], s_bnoff[FL_LDS_BUCKETS];
  __shared__ uint32_t s_leaves;
  static_assert(FL_LDS_BUCKETS == 128 && FL_LDS_BUCKETS >= 2 * FL_SCAN_ROUNDS, "one wavefront scans the rounds");
  const uint32_t maxld = o.ctrl[FL_NUM_FLAGS + FL_CNT_MAXLD];
  load_tails(base, n, cp, rt, act, tl);  // in flight while the guard is read
  if (*guard) return;  // the iteration is redone
  settle_tails(cp, rt, is_outlet, tl);
  if (scan && maxld >= FL_SCAN_ROUNDS) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *guard = 1;
    return;
  }
  if (scan && blockIdx.x == 0) {
    // the leaves, by the other wavefronts
    if (threadIdx.x == 0) s_leaves = 0;
    __syncthreads();
    uint32_t sum = 0;
    for (uint32_t i = threadIdx.x - 64u; threadIdx.x >= 64 && i < gridDim.x; i += FL_BUCKET_BLOCK - 64)
      sum += o.leaves_of[i];
    if (sum) atomicAdd(&s_leaves, sum);
  }
  if (scan && threadIdx.x < 64) {
    const uint32_t l = threadIdx.x;  // its round
    const bool in = l <= maxld;
    const uint32_t c0 = in ? bcnt[2 * l] : 0u, c1 = in ? bcnt[2 * l + 1] : 0u;
    const uint32_t n0 = in ? bnodes[2 * l] : 0u, n1 = in ? bnodes[2 * l + 1] : 0u;
    const uint32_t stride = 65u - long_min, u = c1 + (n0 + stride - 1) / stride;
    // (sums below 2^53: exact)
    const uint32_t c = (uint32_t)prefix_lanes((double)(c0 + c1)), m = (uint32_t)prefix_lanes((double)(n0 + n1));
    const uint32_t us = (uint32_t)prefix_lanes((double)u);
    s_boff[2 * l] = c - c1 - c0;
    s_boff[2 * l + 1] = c - c1;
    s_bnoff[2 * l] = m - n1 - n0;
    s_bnoff[2 * l + 1] = m - n1;
    if (blockIdx.x == 0 && in) {
      uint32_t* counters = o.ctrl + FL_NUM_FLAGS;
      uint32_t* head_c = counters + FL_NUM_COUNTERS;
      uint32_t* head_n = head_c + FL_CTRL_HEAD + 1;
      o.ucum[l] = us - u;
      o.boff[2 * l] = head_c[2 * l] = c - c1 - c0;
      o.boff[2 * l + 1] = head_c[2 * l + 1] = c - c1;
      o.bnoff[2 * l] = head_n[2 * l] = m - n1 - n0;
      o.bnoff[2 * l + 1] = head_n[2 * l + 1] = m - n1;
      if (l == maxld) {
        o.ucum[l + 1] = us;
        o.boff[2 * l + 2] = head_c[2 * l + 2] = counters[FL_CNT_CHAINS] = c;
        o.bnoff[2 * l + 2] = head_n[2 * l + 2] = counters[FL_CNT_POSITIONS] = m;
      }
    }
  }
  if (scan && blockIdx.x == 0) {
    __syncthreads();
    if (threadIdx.x == 0) o.ctrl[FL_NUM_FLAGS + FL_CNT_LEAVES] = s_leaves;
  }
  auto c_off = [&](uint32_t l) { return scan ? s_boff[l] : o.boff[l]; };
  auto n_off = [&](uint32_t l) { return scan ? s_bnoff[l] : o.bnoff[l]; };
  for (uint32_t t = threadIdx.x; t < FL_LDS_BUCKETS; t += FL_BUCKET_BLOCK) {
    s_c[t] = 0;
    s_n[t] = 0;
  }
  __syncthreads();
  uint32_t lc[FL_BUCKET_PER_THREAD], ln[FL_BUCKET_PER_THREAD];
  for (uint32_t j = 0; j < FL_BUCKET_PER_THREAD; ++j) {
    lc[j] = FL_NONE;
    ln[j] = 0;
    if (tl[j].t) {
      const unsigned long long c = tl[j].c;
      uint32_t len = pair_cnt(c) + 1, l = 2u * pair_cnt(tl[j].r) + (len >= long_min ? 1u : 0u);
      if (l < FL_LDS_BUCKETS) {
        lc[j] = atomicAdd(s_c + l, bucket_weight(len, long_min));
        ln[j] = atomicAdd(s_n + l, len);
      } else {
        uint32_t q = o.boff[l] + atomicAdd(bcur + l, bucket_weight(len, long_min));
        uint32_t pos = o.bnoff[l] + atomicAdd(bncur + l, len);
        place_chain(q, pos, len, pair_ptr(c), long_min, cmeta, head_base, pdest);
      }
    }
  }
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < FL_LDS_BUCKETS; t += FL_BUCKET_BLOCK) {
    if (s_c[t]) {
      s_bc[t] = atomicAdd(bcur + t, s_c[t]);
      s_bn[t] = atomicAdd(bncur + t, s_n[t]);
    }
  }
  __syncthreads();
  for (uint32_t j = 0; j < FL_BUCKET_PER_THREAD; ++j) {
    if (lc[j] == FL_NONE) continue;
    const unsigned long long c = tl[j].c;
    uint32_t len = pair_cnt(c) + 1;
    uint32_t l = 2u * pair_cnt(tl[j].r) + (len >= long_min ? 1u : 0u);
    uint32_t q = c_off(l) + s_bc[l] + lc[j];
    uint32_t pos = n_off(l) + s_bn[l] + ln[j];
    place_chain(q, pos, len, pair_ptr(c), long_min, cmeta, head_base, pdest);
  }
}

// Scatter the chains' sites to their chain-major positions with the inputs the
// sweeps read there: the drainage-area fold's list counts, area, erodibility and
// receiver distance (with max slopes also uplift, tan(max slope), old elevation
// and the basin outlet's position), for each listed light child that is a leaf
// its drainage area, which is its own area, and for each other one the slot its
// chain's head fills with it (pdest at the child chain's base).  A chain's base
// gets the position of the head's receiver (FL_NONE for an outlet).  spos: a
// chain site's position, a leaf's receiver's.  Sites outside every basin keep
// their elevation, drainage area = own area and response time 0
// (generator.rs:144-145), as the reference leaves them.
struct fl_perm_out {
  uint32_t* perm;
  uint32_t* pcnt;
  uint32_t* pdest;
  double* parea;
  double* pK;
  double* pdn;
  double* up;
  double* tanp;
  double* hop;
  uint32_t* ppos;
  uint32_t* pro;
  double* cval;
  uint32_t* spos;
};

__global__ void k_chain_perm(uint32_t bs, const uint32_t* __restrict__ guard, uint32_t n, unsigned long long* cp,
                             unsigned long long* rt, const uint32_t* __restrict__ next,
                             const uint8_t* __restrict__ is_outlet, const uint32_t* __restrict__ head_base,
                             fl_perm_out o,
                             const double* __restrict__ area, const double* __restrict__ K,
                             const double* __restrict__ dnext, const double* __restrict__ U,
                             const double* __restrict__ tan_ms, int clamp, double* __restrict__ A,
                             double* __restrict__ tau, const double* __restrict__ h, double* __restrict__ h2,
                             const uint32_t* __restrict__ maxld, uint32_t* __restrict__ bcnt,
                             uint32_t* __restrict__ bnodes, uint32_t* __restrict__ bcur,
                             uint32_t* __restrict__ bncur, const uint32_t* __restrict__ rp,
                             const uint32_t* __restrict__ col, const unsigned long long* __restrict__ cmask,
                             const uint32_t* __restrict__ hc, const uint8_t* __restrict__ act,
                             uint32_t* __restrict__ root) {
  uint32_t v = gid(bs);
  // the site's own words are read together with the guard (one load
  // latency; a site of a lake basin reads some it does not use)
  const uint32_t mld = *maxld, redo = *guard;
  const uint32_t kind = v < n ? act[v] : 0u;
  const bool chain = kind != 0 && !(kind & FL_LEAF);
  unsigned long long rv = 0ull, cv = 0ull, m = 0ull;
  uint32_t b = 0u, e = 0u, hk = FL_NONE, p = 0u;
  double Kv = 0.0, dv = 0.0, av = 0.0;
  if (kind) {
    p = next[v];
    av = area[v];
  }
  if (chain) {
    rv = rt[v];
    cv = cp[v];
    b = rp[v];
    e = rp[v + 1];
    m = cmask[v];
    hk = hc[v];
    Kv = K[v];
    dv = dnext[v];
  }
  if (kind & FL_CHAIN_END) hk = FL_NONE;  // a leaf: one more of the list
  // the bucket histograms are used up (count, scan, place): clear the
  // entries this decomposition touched for the next one
  const uint32_t nb = 2u * (mld + 1u);
  for (uint32_t i = v; i <= nb && i < n + FL_BUCKET_PAD; i += gridDim.x * bs) {
    bcnt[i] = 0;
    bnodes[i] = 0;
    bcur[i] = 0;
    bncur[i] = 0;
  }
  if (redo || !kind) return;
  if (!chain) {
    // a leaf: the rest of its words come from its receiver's thread, which has
    // them at hand (20.7 us at a million sites; 16.7 with all sites on chains,
    // which cost the sweeps and the placement 10 us more)
    A[v] = av;
    if (p == v) {
      root[v] = v;
      o.spos[v] = FL_NONE;
      if (is_outlet && !is_outlet[v]) {
        tau[v] = 0.0;
        h2[v] = h[v];
      }
    }
    return;
  }
  if (!pair_fin(rv) || !pair_fin(cv)) {
    rv = settle(rv, rt);
    cv = settle(cv, cp);
    // (others read v's pair from here on only as one to hop over, which
    // either value serves)
    __atomic_store_n(rt + v, rv | (1ull << 63), __ATOMIC_RELAXED);
    __atomic_store_n(cp + v, cv | (1ull << 63), __ATOMIC_RELAXED);
  }
  const uint32_t r = pair_ptr(rv), hd = pair_ptr(cv), deg = e - b;
  root[v] = r;
  // the second level of loads, issued together: the root's outlet flag, the
  // chain's base, the row (up to FL_ROW entries), at a chain head the
  // receiver's pair and with max slopes the outlet's base
  const uint8_t outlet = is_outlet ? is_outlet[r] : 1;
  const uint32_t base = head_base[hd];
  const bool head = hd == v;
  unsigned long long cpp = head ? cp[p] : 0ull;
  const uint32_t hbr = clamp ? head_base[r] : 0u;
  uint32_t cc[FL_ROW];
  const bool short_row = deg <= FL_ROW;
  if (short_row && deg > 0) {
#pragma unroll
    for (int j = 0; j < FL_ROW; ++j) cc[j] = col[min(b + j, e - 1)];
  }
  if (!outlet) {
    A[v] = av;
    tau[v] = 0.0;
    h2[v] = h[v];
    for (uint32_t s = 0; s < deg; ++s) {
      const uint32_t ch = col[b + s];
      if (!is_child(m, deg, s, b, col, next, v) || hc[ch] != FL_NONE) continue;
      root[ch] = r;
      tau[ch] = 0.0;
      h2[ch] = h[ch];
    }
    return;
  }
  const uint32_t P = base + pair_cnt(cv);
  o.spos[v] = P;
  o.perm[P] = v;
  o.pK[P] = Kv;
  o.pdn[P] = dv;
  if (clamp) {
    o.up[P] = U[v];
    o.tanp[P] = tan_ms[v];
    o.hop[P] = h[v];
    o.pro[P] = hbr;
  }
  // the light children in fold order (descending slot): those before the
  // heavy child get their receiver's slots 0, 1, ..., those after it the slots
  // FL_LIST - 1, FL_LIST - 2, ...; with more than FL_LIST the overflow bit is
  // set (the fold walks the row) and all of their heads hand over at their own
  // bases
  {
    uint32_t npre = 0, npost = 0;
    bool after = false;
    if (short_row) {
      // the children's bases loaded together (a row of at most FL_ROW
      // entries, no more than a list holds: the child mask covers it)
      uint32_t hb[FL_ROW];
      double aj[FL_ROW];
#pragma unroll
      for (int j = 0; j < FL_ROW; ++j) {
        hb[j] = 0u;
        aj[j] = 0.0;
        if (j < (int)deg && ((m >> j) & 1ull) && cc[j] != hk) {
          hb[j] = head_base[cc[j]];  // FL_NONE: a leaf
          aj[j] = area[cc[j]];
        }
      }
#pragma unroll
      for (int j = FL_ROW - 1; j >= 0; --j) {
        if (j >= (int)deg || !((m >> j) & 1ull)) continue;
        if (cc[j] == hk) {
          after = true;
          continue;
        }
        const uint32_t slot = after ? FL_LIST - 1 - npost++ : npre++;
        if (hb[j] == FL_NONE) {
          o.cval[(uint64_t)FL_LIST * P + slot] = no_word(aj[j]);
          o.spos[cc[j]] = P;
          root[cc[j]] = r;
        } else {
          o.pdest[hb[j]] = slot;
        }
      }
      o.pcnt[P] = npre | (npost << 8) | (hk == FL_NONE ? FL_TAIL : 0u) | (head ? FL_HEAD : 0u);
    } else {
      // in fold order, FL_ROW entries loaded together: a hub's row is one thread's
      // (20 000 entries 14.6 ms one by one, 5.3 so), and a row of nine or more, which
      // one site in sixty has, is the last of its wavefront to end (solve of 10k
      // random sites 2.36 -> 2.22 ms)
      uint32_t light = (uint32_t)__builtin_popcountll(m);
      if (deg > 64) {
        light = 0;
        for (uint32_t s = 0; s < deg; s += FL_ROW) {
          uint32_t nx[FL_ROW];
#pragma unroll
          for (int j = 0; j < FL_ROW; ++j) nx[j] = next[col[b + min(s + j, deg - 1)]];
#pragma unroll
          for (int j = 0; j < FL_ROW; ++j) light += s + j < deg && nx[j] == v ? 1u : 0u;
        }
      }
      if (hk != FL_NONE) --light;
      const bool over = light > FL_LIST;
      for (uint32_t top = deg; top > 0; top -= min(top, (uint32_t)FL_ROW)) {
        uint32_t ch[FL_ROW], nx[FL_ROW], hb[FL_ROW];
        double aj[FL_ROW];
#pragma unroll
        for (int j = 0; j < FL_ROW; ++j) ch[j] = col[b + (top > (uint32_t)j ? top - 1 - j : 0u)];
#pragma unroll
        for (int j = 0; j < FL_ROW; ++j) {
          nx[j] = next[ch[j]];
          hb[j] = head_base[ch[j]];
          aj[j] = area[ch[j]];
        }
#pragma unroll
        for (int j = 0; j < FL_ROW; ++j) {
          if ((uint32_t)j >= top || nx[j] != v) continue;
          if (ch[j] == hk) {
            after = true;
            continue;
          }
          const uint32_t slot = over ? FL_DEST_OVER : (after ? FL_LIST - 1 - npost : npre);
          if (hb[j] != FL_NONE) {
            o.pdest[hb[j]] = slot;
          } else {
            if (!over) o.cval[(uint64_t)FL_LIST * P + slot] = no_word(aj[j]);
            o.spos[ch[j]] = P;
            root[ch[j]] = r;
          }
          if (after) ++npost;
          else ++npre;
        }
      }
      o.pcnt[P] = (over ? FL_LIST_OVERFLOW : (npre | (npost << 8))) | (hk == FL_NONE ? FL_TAIL : 0u) |
                  (head ? FL_HEAD : 0u);
    }
    o.parea[P] = av;
  }
  if (head) {
    cpp = settle(cpp, cp);
    o.ppos[P] = (p == v) ? FL_NONE : head_base[pair_ptr(cpp)] + pair_cnt(cpp);
  }
}

// --------------------------------------------------------------- sweeps ---
//
// Both sweeps run every round (light depth) in one launch.  A round's work
// is cut into units of one wavefront each: a tile of a long chain (response
// time: the whole chain, at its head's tile), or a tile of 64 consecutive chain
// positions of its short chains.  Wavefronts take the units
// in round order (drainage area deepest round first, response time shallowest
// first) and a unit waits for just the values it reads, not for the round
// before it: a chain's head hands its drainage area to its receiver's list
// slot, a tile of a long chain its last one to the tile after it, a position its
// response time (and, with max slopes, its elevation) to the heads below it,
// and the word itself says whether it is there yet.
//
// What bounds it: the longest path of the forest, one dependent chain of
// FP64 adds, plus a hand-over per light edge on it.  One launch per round made
// every round as long as its longest chain and paid 4.5 us a launch; a
// hand-over between two wavefronts of different XCDs takes 0.57 us.
//
// A hand-over word holds FL_SENT, a signalling NaN that no arithmetic
// produces, until its value is stored (publish() quiets a value that equals
// it).  Words are stored and read with relaxed device-scope atomics: the value
// is the flag, no fence is needed.  Drainage-area words are set back to
// FL_SENT by the one unit that reads them, response times and elevations by
// the drainage-area sweep before.
//
// A workgroup takes FL_FOLD_WAVES units at a time from one counter, once it
// runs; with a wavefront for every unit, which the launch usually has, the
// workgroups that are enough take once and the others none.  That is 17 ns a
// workgroup one after the other on one word.  Units by the workgroups' own
// numbers would save them (solve of 1M sites 28.1 -> 27.4 ms, 400k 14.1 -> 13.9,
// strip 38.5 -> 38.3), but a wavefront would then wait for workgroups that do not
// run yet: with two streams sweeping, each can fill the XCD that the other's next
// workgroup is to start on.  Two or four units a wavefront of one taking: 1M sites
// 32 and 41 ms (the second waits for the first).
//
// Waits end.  Units are in the order of the counter, so every unit a wavefront
// waits for was taken before its own, by a wavefront that runs, in whatever order
// and beside whatever else the workgroups start: the lowest unit not finished
// waits for nothing.  Should a wait still last FL_SPIN_MAX polls (a second: the
// whole queue taken off the GPU), the wavefront raises FL_FLAG_STALL and goes on,
// every other wait sees the flag and ends, and the host redoes the iteration in
// one workgroup with barriers between the rounds (k_da_tail, k_tau_tail).
#define FL_SPIN_MAX (1u << 20)
#ifndef FL_SPIN_FOLD
#define FL_SPIN_FOLD FL_SPIN_MAX  // of the sweeps in one launch (k_da_fold, k_tau_fold)
#endif
#define FL_NEG0 (-0.0)

// The rounds of a decomposition and the counters its units are taken from.
struct fl_flow {
  const uint32_t* maxld;  // the deepest round
  const uint32_t* ucum;   // units before each round
  const uint32_t* boff;   // counts before each bucket (short: chains, long: tiles of each round)
  const uint32_t* bnoff;  // positions before each bucket
  uint32_t* ticket_da;
  uint32_t* ticket_tau;
  uint32_t long_min;
};

namespace {

// A hand-over word, read and written at device scope.
__device__ __forceinline__ unsigned long long peek(const double* p) {
  const unsigned long long* w = reinterpret_cast<const unsigned long long*>(p);
#ifdef FL_DEVICE_ATOMICS
  return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#else
  return __atomic_load_n(w, __ATOMIC_RELAXED);
#endif
}
__device__ __forceinline__ void poke(double* p, unsigned long long u) {
  unsigned long long* w = reinterpret_cast<unsigned long long*>(p);
#ifdef FL_DEVICE_ATOMICS
  __hip_atomic_store(w, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#else
  __atomic_store_n(w, u, __ATOMIC_RELAXED);
#endif
}
__device__ __forceinline__ void publish(double* p, double v) {
  unsigned long long u = (unsigned long long)__double_as_longlong(v);
  if (u == FL_SENT) u |= 1ull << 51;
  poke(p, u);
}

// The flag of ended waits, and the polls after which a wait raises it.
struct fl_patience {
  int* stall;
  uint32_t polls;
};
// One more poll of a wait: false when the wait is to end without its value.
__device__ __forceinline__ bool wait_more(uint32_t& spins, const fl_patience& w) {
  ++spins;
#ifdef FL_WAVE_SHIFT
  __builtin_amdgcn_s_sleep(1);
#endif
  if ((spins & 255u) != 0 && spins < w.polls) return true;
  if (spins >= w.polls) __atomic_store_n(w.stall, 1, __ATOMIC_RELAXED);
  return __atomic_load_n(w.stall, __ATOMIC_RELAXED) == 0;
}

// The word at p where `need`, waited for by the whole wavefront.
__device__ __forceinline__ double await(const double* p, bool need, double otherwise, const fl_patience& w) {
  unsigned long long u = need ? peek(p) : 0ull;
  uint32_t spins = 0;
  while (__any(need && u == FL_SENT)) {
    if (!wait_more(spins, w)) break;
    if (need && u == FL_SENT) u = peek(p);
  }
  return need ? bits_double(u) : otherwise;
}

// A hand-over word in LDS, between wavefronts of a workgroup (read by every
// lane, stored by one).
__device__ __forceinline__ void publish_lds(double* p, double v) {
  unsigned long long u = (unsigned long long)__double_as_longlong(v);
  if (u == FL_SENT) u |= 1ull << 51;
  *reinterpret_cast<volatile unsigned long long*>(p) = u;
}
__device__ __forceinline__ double await_lds(const double* p, const fl_patience& patience) {
  const volatile unsigned long long* w = reinterpret_cast<const volatile unsigned long long*>(p);
  unsigned long long u = *w;
  uint32_t spins = 0;
  while (__any(u == FL_SENT)) {
    if (!wait_more(spins, patience)) break;
    u = *w;
  }
  return bits_double(u);
}

// A value that every lane of the wavefront holds, for scalar registers.
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, 0); }

// Length of the longest run of set bits, plus one: the positions of the
// longest chain of a tile whose non-first positions are marked.
__device__ __forceinline__ uint32_t run_steps(unsigned long long m) {
  uint32_t steps = 1;
  for (; m; m &= m << 1) ++steps;
  return steps;
}

// A long chain's tile: every lane's running value from the lane before it,
// out = step(in), lane 0 from `carry` -- bit for bit what one lane after the
// other gives, without waiting for 64 of them.
//
// A sum of positive terms stays in one binade (a power of two c to 2 c) for
// most of a long chain.  There the running values are multiples of one unit u,
// and a term adds the same multiple of u to all of them unless it lies halfway
// between two: then it rounds to the even one, and what a lane adds depends on
// whether its value is an even or an odd multiple (its lowest bit) -- but after
// it the value is even either way.  So each lane's steps from c (even) and from
// c + u (odd) tell what it adds to either; its value's lowest bit follows from
// the last lane before it with a halfway term and the odd sums since, which
// three ballots hold; and the prefix sum of what the lanes add, exact, is every
// lane's value at once.  All of that is a guess, and it is checked: each lane
// takes its real steps from its guess, and the guess of the lane after it has
// to be the result.  Up to the first lane where it is not, everything is the
// serial fold's value, and from there on it is guessed again (a new binade).
//
// 64 serial steps take 1.3 to 2.5 us, a guess and its check 0.3 us.  A tile
// that begins at a chain's tail, where the binade changes with every few
// positions, one of fewer than FL_GUESS_LANES lanes and one still wrong after
// FL_GUESSES guesses take the serial steps.  `last`: the last lane whose value
// counts.
#define FL_GUESSES 4
#define FL_GUESS_LANES 24
template <class Step>
__device__ __forceinline__ void tile_fold(double carry, uint32_t lane, uint32_t last, Step step) {
  auto bits = [](double v) { return (unsigned long long)__double_as_longlong(v); };
  auto grows = [](double v) { return v > 0.0 && v < __builtin_inf(); };
  const unsigned long long below = (1ull << lane) - 1ull;
  uint32_t at = 0;  // the lanes before it are final, and its `in`
  double in = carry, real = carry, out;
  bool guessed = last >= FL_GUESS_LANES && grows(carry);
#pragma unroll 1
  for (uint32_t k = 0; guessed && k < FL_GUESSES; ++k) {
    const double c0 = bits_double(bits(real) & 0x7ff0000000000000ull), c1 = bits_double(bits(c0) + 1ull);
    const double w0 = step(c0), w1 = step(c1);
    const bool half = bits(w1) != bits(w0) + 1ull, odd = (bits(w0) & 1ull) != 0, here = lane >= at;
    const unsigned long long halves = __ballot(here && half), odds = __ballot(here && odd);
    const unsigned long long hb = halves & below;
    const uint32_t t = 63u - (uint32_t)__builtin_clzll(hb | 1ull);
    // the bit after lane t, then the odd sums of the lanes after it
    const unsigned long long from = hb ? ~0ull << t : ~0ull;
    const uint32_t bit = (hb ? 0u : (uint32_t)(bits(real) & 1ull)) +
                         (uint32_t)__builtin_popcountll(odds & below & from);
    const double add = !here ? 0.0 : ((bit & 1u) ? w1 - c1 : w0 - c0);
    const double before = prefix_lanes(add) - add;
    if (lane >= at) in = real + before;
    if (lane == at) in = real;
    out = step(in);
    const double s = from_prev(carry, out);
    const unsigned long long bad = __ballot(lane <= last && !same_bits(s, in));
    if (bad == 0) return;
    at = (uint32_t)__builtin_ctzll(bad);
    real = of_lane(s, at);
    guessed = grows(real);
  }
  if (lane == at) in = real;
  out = step(in);
#pragma unroll 2
  for (uint32_t i = at; i < last; ++i) {
    in = from_prev(carry, out);
    out = step(in);
  }
}

// The rounds of a decomposition, lane i holding round `first` + i.
struct fl_rounds {
  uint32_t first, u0, u1, c1, c2, n0, n1;
};
__device__ __forceinline__ fl_rounds load_rounds(const fl_flow& f, uint32_t first, uint32_t rounds, uint32_t lane) {
  fl_rounds r{first, 0u, 0u, 0u, 0u, 0u, 0u};
  const uint32_t l = first + lane;
  if (l < rounds) {
    r.u0 = f.ucum[l];
    r.u1 = f.ucum[l + 1];
    r.c1 = f.boff[2ull * l + 1];
    r.c2 = f.boff[2ull * l + 2];
    r.n0 = f.bnoff[2ull * l];
    r.n1 = f.bnoff[2ull * l + 1];
  } else {
    r.u0 = r.u1 = 0xffffffffu;
  }
  return r;
}

// A unit of round l: long tile `chain` (FL_NONE: none), or the short-chain
// positions [n0, n1) from tile start T on.
struct fl_unit {
  uint32_t l, chain, T, n1;
};
__device__ __forceinline__ fl_unit unit_of(uint32_t l, uint32_t off, uint32_t c1, uint32_t c2, uint32_t n0,
                                           uint32_t n1, uint32_t stride) {
  fl_unit u{l, FL_NONE, 0u, n1};
  if (off < c2 - c1) u.chain = c1 + off;
  else u.T = n0 + (off - (c2 - c1)) * stride;
  return u;
}
// Unit v of the units of rounds 0, 1, ... (`back`: its place in the round
// counted from the round's end, so that long chains still come first).
__device__ __forceinline__ fl_unit find_unit(const fl_flow& f, fl_rounds& R, uint32_t rounds, uint32_t v, bool back,
                                             uint32_t lane) {
  uint32_t j;
  for (;;) {
    // (wavefront-uniform: every lane asks for the same unit)
    const uint32_t below = (uint32_t)__builtin_popcountll(__ballot(R.u1 <= v));
    const bool before = R.first > 0 && v < (uint32_t)__builtin_amdgcn_readlane((int)R.u0, 0);
    if (!before && below < 64) {
      j = below;
      break;
    }
    R = load_rounds(f, before ? 0 : R.first + 64, rounds, lane);
  }
  const uint32_t u0 = (uint32_t)__builtin_amdgcn_readlane((int)R.u0, (int)j);
  const uint32_t u1 = (uint32_t)__builtin_amdgcn_readlane((int)R.u1, (int)j);
  const uint32_t c1 = (uint32_t)__builtin_amdgcn_readlane((int)R.c1, (int)j);
  const uint32_t c2 = (uint32_t)__builtin_amdgcn_readlane((int)R.c2, (int)j);
  const uint32_t n0 = (uint32_t)__builtin_amdgcn_readlane((int)R.n0, (int)j);
  const uint32_t n1 = (uint32_t)__builtin_amdgcn_readlane((int)R.n1, (int)j);
  return unit_of(R.first + j, back ? u1 - 1 - v : v - u0, c1, c2, n0, n1, 65u - f.long_min);
}

// A short-chain tile: lane i holds position T + i.  The tile owns the chains
// whose heads lie in its first `stride` positions: with at most
// long_min - 1 = 64 - stride positions they end within the tile, so every
// chain lies whole in the tile that owns it (the tiles overlap).
struct fl_short_tile {
  uint32_t P;  // this lane's position, clamped into the round's
  bool own;
};
__device__ __forceinline__ fl_short_tile short_tile(const uint32_t* __restrict__ pcnt, uint32_t T, uint32_t n1,
                                                    uint32_t stride, uint32_t lane, uint32_t& cn) {
  const bool in = T + lane < n1;
  fl_short_tile t{in ? T + lane : n1 - 1, false};
  cn = pcnt[t.P];
  const unsigned long long heads = __ballot(in && (cn & FL_HEAD) && lane < stride);
  // the last head at or before this lane, of any chain: owned when it is one
  // of `heads`
  const unsigned long long all = __ballot(in && (cn & FL_HEAD));
  const unsigned long long upto = all & (~0ull >> (63u - lane));
  t.own = in && upto != 0 && ((heads >> (63 - __builtin_clzll(upto | 1ull))) & 1ull) != 0;
  return t;
}

}  // namespace

// Drainage area of the site at chain position P, folded in the reference's
// order (generator.rs:154-159 accumulates children in reverse BFS order, so
// A_k = ((a_k + A_{c_m}) + A_{c_{m-1}}) + ... + A_{c_1} over the children in
// row order).  The heavy child's value comes from the position after it: the
// fold is split into `pre` (the part before it) and the light children after
// it, posts p0, p1, ... in fold order.
//
// Absent posts are -0.0, and the chain fold starts from r = -0.0 at the
// tail: x + (-0.0) == x exactly for every x (signed zeros included), so
//     A = ((pre + r) + p0) + p1 ...
// is the reference's value at every position without a branch.
//
// The partial folds of a listed position from the values of its light
// children: those before the heavy child in fold order from its first slot on,
// those after it from its last slot backwards, -0.0 in the others.
struct fl_da_words {
  unsigned long long u[FL_LIST];
};
__device__ __forceinline__ uint32_t da_posts(uint32_t cn, bool mine) { return mine ? (cn >> 8) & 0xffu : 0u; }
// The part before the heavy child; the words it takes become -0.0 (x + (-0.0)
// == x), so that the last ones are the posts p0, p1, ...
__device__ __forceinline__ double da_pre(uint32_t cn, double area_k, fl_da_words& w, bool mine) {
  const uint32_t npre = mine ? cn & 0xffu : 0u;
  double pre = mine ? area_k : FL_NEG0;
#pragma unroll
  for (uint32_t i = 0; i < FL_LIST; ++i) {
    if (!__any(i < npre)) break;
    const bool take = i < npre;
    pre = pre + (take ? bits_double(w.u[i]) : FL_NEG0);
    if (take) w.u[i] = 1ull << 63;
  }
  return pre;
}
// As many posts are added as the tile's largest position has (`posts`: 1, 2, 4
// or all of the list); the others are -0.0.
template <int posts>
__device__ __forceinline__ double da_step(double pre, const fl_da_words& w, double r) {
  r = pre + r;
#pragma unroll
  for (int j = 0; j < posts; ++j) r = r + bits_double(w.u[FL_LIST - 1 - j]);
  return r;
}

// What the drainage-area fold reads at chain position P besides its counts and
// listed children, in chain-major order (written by k_chain_perm): the site,
// its area, erodibility and receiver distance.
struct fl_da_pos {
  uint32_t k;
  double area, K, d;
};

// The arrays of the drainage-area sweep.
struct fl_da_args {
  const uint32_t* perm;
  const uint32_t* pcnt;
  double* cval;   // [FL_LIST n] light children's A by (position, slot): hand-over words
  // [n] at a chain's base: its head's A for a receiver with more light
  // children than listed; at the last position of a long chain's tile: the A
  // that enters it
  double* cover;
  const double* parea;
  const double* pK;
  const double* pdn;
  // at a chain's base position: its head's slot with its receiver, FL_DEST_OVER
  // or FL_NONE, and the receiver's position
  const uint32_t* pdest;
  const uint32_t* ppos;
  const uint2* cmeta;     // long chains' tiles: (base, length or end)
  double* xp;
  double* taup;  // set to FL_SENT
  double* hnp;   // with max slopes, too (else null)
  // the graph, for positions with more light children than listed
  const uint32_t* rp;
  const uint32_t* col;
  const uint32_t* next;
  const unsigned long long* cmask;
  const uint32_t* hc;
  const uint32_t* head_base;
  const double* area;
  double* A;
  fl_patience wait;
};

__device__ __forceinline__ fl_da_pos da_load(const fl_da_args& g, uint32_t P) {
  return fl_da_pos{g.perm[P], g.parea[P], g.pK[P], g.pdn[P]};
}

// The words of position P's listed children (-0.0 in the other slots).
__device__ __forceinline__ bool da_slot(uint32_t cn, uint32_t i) {
  return i < (cn & 0xffu) || i + ((cn >> 8) & 0xffu) >= FL_LIST;
}
__device__ __forceinline__ fl_da_words da_words(const fl_da_args& g, uint32_t P, uint32_t cn, bool mine) {
  const double* w = g.cval + (uint64_t)FL_LIST * P;
  fl_da_words q;
#pragma unroll
  for (uint32_t i = 0; i < FL_LIST; ++i) q.u[i] = mine && da_slot(cn, i) ? peek(w + i) : 1ull << 63;
  return q;
}
__device__ __forceinline__ bool da_missing(const fl_da_words& q) {
  bool m = false;
#pragma unroll
  for (uint32_t i = 0; i < FL_LIST; ++i) m = m || q.u[i] == FL_SENT;
  return m;
}
__device__ __forceinline__ void da_again(const fl_da_args& g, uint32_t P, fl_da_words& q) {
  const double* w = g.cval + (uint64_t)FL_LIST * P;
#pragma unroll
  for (uint32_t i = 0; i < FL_LIST; ++i)
    if (q.u[i] == FL_SENT) q.u[i] = peek(w + i);
}
// Words that were read are given back.
__device__ __forceinline__ void da_give_back(const fl_da_args& g, uint32_t P, uint32_t cn, bool mine) {
  unsigned long long* w = reinterpret_cast<unsigned long long*>(g.cval) + (uint64_t)FL_LIST * P;
#pragma unroll
  for (uint32_t i = 0; i < FL_LIST; ++i)
    if (mine && da_slot(cn, i)) w[i] = FL_SENT;
}

// A position with more light children than listed (rare): the wavefront walks its
// row together, 64 entries at a time in fold order, one a lane.  Their chains' words
// are in cover (a leaf's drainage area is its own), r is the heavy child's value.
// k, its area a, its row and r are the same in every lane.  Bound by the latency of
// three dependent loads per 64 entries; one lane on its own had them per entry: the
// sweep of a hub with 20 000 leaves 15.3 -> 1.2 ms, solve of 30 000 sites in a chain
// with nine leaves each 110 -> 39 ms.
__device__ __forceinline__ double da_over_fold(const fl_da_args& g, uint32_t k, double a, uint32_t b, uint32_t deg,
                                               uint32_t hk, double r, uint32_t lane) {
  double acc = a;
  for (uint32_t top = deg; top > 0; top -= min(top, 64u)) {
    const bool in = lane < top;
    const uint32_t c = g.col[b + (in ? top - 1 - lane : 0u)];
    const bool kid = in && g.next[c] == k, leaf = g.hc[c] == FL_NONE, light = kid && !leaf && c != hk;
    const double area = g.area[c];
    double* w = g.cover + (light ? g.head_base[c] : 0u);
    const double x = await(w, light, area, g.wait);
    if (light) *reinterpret_cast<unsigned long long*>(w) = FL_SENT;
    unsigned long long kids = __ballot(kid);
    const unsigned long long heavy = __ballot(kid && !leaf && c == hk);
    for (; kids; kids &= kids - 1) {
      const uint32_t i = (uint32_t)__builtin_ctzll(kids);
      acc = acc + (((heavy >> i) & 1ull) ? r : of_lane(x, i));
    }
  }
  return acc;
}

// The drainage areas of a short-chain tile, one position a lane, each from the
// position after it:
//   r_i = ((pre_i + r_{i+1}) + p0_i) + p1_i ...
// Every lane takes every step: once lane i + 1 holds its final value, lane i
// gets its own in the next step and keeps it, so `steps` steps settle chains
// of that many positions without a lane ever being singled out (two DPP moves
// and the adds a step, 14 ns).  At a chain's tail the fold starts from -0.0.
template <int posts>
__device__ __forceinline__ double da_short_steps(double pre, const fl_da_words& w, bool tail, uint32_t steps) {
  double s = FL_NEG0, r = FL_NEG0;
#pragma unroll 2
  for (uint32_t i = 0; i < steps; ++i) {
    s = from_next(s, r);
    r = da_step<posts>(pre, w, tail ? FL_NEG0 : s);
  }
  return r;
}
__device__ __forceinline__ double da_short_fold(uint32_t np, double pre, const fl_da_words& w, bool tail,
                                                uint32_t steps) {
  if (!__any(np >= 2)) return da_short_steps<1>(pre, w, tail, steps);
  if (!__any(np >= 3)) return da_short_steps<2>(pre, w, tail, steps);
  if (!__any(np >= 5)) return da_short_steps<4>(pre, w, tail, steps);
  return da_short_steps<FL_LIST>(pre, w, tail, steps);
}

// The drainage areas of a long chain's tile, two positions a lane, the chain's
// tail side first (r[0], then r[1], then the next lane's).  Positions past the
// tile pass the value on (pre and posts -0.0).
template <int posts>
__device__ __forceinline__ void da_long_steps(const double (&pre)[2], const fl_da_words (&w)[2], double carry,
                                              uint32_t lane, uint32_t last, double (&r)[2]) {
  tile_fold(carry, lane, last, [&](double v) {
    r[0] = da_step<posts>(pre[0], w[0], v);
    return r[1] = da_step<posts>(pre[1], w[1], r[0]);
  });
}
__device__ __forceinline__ void da_long_fold(uint32_t np, const double (&pre)[2], const fl_da_words (&w)[2],
                                             double carry, uint32_t lane, uint32_t last, double (&r)[2]) {
  if (!__any(np >= 2)) da_long_steps<1>(pre, w, carry, lane, last, r);
  else if (!__any(np >= 3)) da_long_steps<2>(pre, w, carry, lane, last, r);
  else if (!__any(np >= 5)) da_long_steps<4>(pre, w, carry, lane, last, r);
  else da_long_steps<FL_LIST>(pre, w, carry, lane, last, r);
}

// The same for a tile with positions of more light children than listed: one
// lane after the other, from lane 0 on (`up`) or from lane 63 down.
template <int B, bool up>
__device__ __forceinline__ void da_tile_walk(const fl_da_args& g, const fl_da_pos (&t)[B], const uint32_t (&cn)[B],
                                             const bool (&mine)[B], const double (&pre)[B],
                                             const fl_da_words (&w)[B], bool tail, double carry, uint32_t lane, double (&r)[B]) {
  unsigned long long over[B];
  uint32_t row[B], deg[B], hk[B];
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const bool o = mine[b] && (cn[b] & FL_LIST_OVERFLOW);
    over[b] = __ballot(o);
    row[b] = o ? g.rp[t[b].k] : 0u;
    deg[b] = o ? g.rp[t[b].k + 1] - row[b] : 0u;
    hk[b] = o ? g.hc[t[b].k] : 0u;
  }
  const unsigned long long tails = __ballot(tail);
  auto at = [](uint32_t v, uint32_t e) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)e); };
  double v = carry;
  for (uint32_t i = 0; i < 64; ++i) {
    const uint32_t e = up ? i : 63 - i;
    if ((tails >> e) & 1ull) v = FL_NEG0;
#pragma unroll
    for (int b = 0; b < B; ++b) {
      if ((over[b] >> e) & 1ull)
        v = da_over_fold(g, at(t[b].k, e), of_lane(t[b].area, e), at(row[b], e), at(deg[b], e), at(hk[b], e), v, lane);
      else
        v = of_lane(da_step<FL_LIST>(pre[b], w[b], v), e);
      if (lane == e) r[b] = v;
    }
  }
}

// A position's drainage area is final: store it and the response-time input
// x = 1.0 / (K * a^0.5) * d (generator.rs:172-173, the reference's
// association); the response-time words are to be waited for from here on.
__device__ __forceinline__ void da_store(const fl_da_args& g, uint32_t P, const fl_da_pos& q, double a) {
  g.A[q.k] = a;
  const double celerity = q.K * rust_pow_half(a);
  g.xp[P] = 1.0 / celerity * q.d;
  reinterpret_cast<unsigned long long*>(g.taup)[P] = FL_SENT;
  if (g.hnp) reinterpret_cast<unsigned long long*>(g.hnp)[P] = FL_SENT;
}
// (pd, pp: the words at its base)
__device__ __forceinline__ void da_hand_over(const fl_da_args& g, uint32_t base, uint32_t pd, uint32_t pp, double a) {
  if (pd == FL_NONE) return;
  publish(pd == FL_DEST_OVER ? g.cover + base : g.cval + (uint64_t)FL_LIST * pp + pd, a);
}

// One unit of the drainage-area sweep, tail to head along its chains.
//
// A long chain's tile is 128 positions, two a lane, lane 0 nearest the tail.
// The tiles of a chain are units of their own: all their loads, list waits,
// divisions and stores overlap, and one after the other is only the value that
// a tile hands to the next, through LDS where the next wavefront of the workgroup
// has it (s_carry), else through cover.  A chain of 8192 positions takes 57 us
// (224 with the tiles one after the other on one wavefront, 64 serial steps each).
__device__ __forceinline__ void da_unit(const fl_da_args& g, const fl_unit& un, uint32_t stride, uint32_t lane,
                                        double* s_carry, uint32_t wave) {
  if (un.chain == FL_NONE) {
    uint32_t cn[1];
    const fl_short_tile t = short_tile(g.pcnt, un.T, un.n1, stride, lane, cn[0]);
    const fl_da_pos at[1] = {da_load(g, t.P)};
    const bool head = t.own && (cn[0] & FL_HEAD) != 0, tail = (cn[0] & FL_TAIL) != 0;
    const uint32_t pd = head ? g.pdest[t.P] : FL_NONE, pp = head ? g.ppos[t.P] : FL_NONE;
    fl_da_words w = da_words(g, t.P, cn[0], t.own);
    uint32_t spins = 0;
    while (__any(da_missing(w))) {
      if (!wait_more(spins, g.wait)) break;
      da_again(g, t.P, w);
    }
    const double pre[1] = {da_pre(cn[0], at[0].area, w, t.own)};
    double r[1];
    if (__any(t.own && (cn[0] & FL_LIST_OVERFLOW))) {
      const bool mine[1] = {t.own};
      const fl_da_words ws[1] = {w};
      da_tile_walk<1, false>(g, at, cn, mine, pre, ws, tail, FL_NEG0, lane, r);
    } else {
      r[0] = da_short_fold(da_posts(cn[0], t.own), pre[0], w, tail, run_steps(__ballot(t.own && !tail)));
    }
    if (head) da_hand_over(g, t.P, pd, pp, r[0]);
    da_give_back(g, t.P, cn[0], t.own);
    if (t.own) da_store(g, t.P, at[0], r[0]);
    return;
  }
  const uint2 m = g.cmeta[un.chain];
  const uint32_t base = uniform(m.x) & ~FL_CHAIN_TAIL, my = uniform(m.y);
  const bool first = (uniform(m.x) & FL_CHAIN_TAIL) != 0, head = !(my & FL_CHAIN_PART);
  const uint32_t end = head ? min(my, (uint32_t)FL_TILE) : my & ~FL_CHAIN_PART;
  const uint32_t start = (end - 1) & ~(FL_TILE - 1u), cnt = end - start, last = (cnt - 1) / 2;
  const uint32_t pd = head ? g.pdest[base] : FL_NONE, pp = head ? g.ppos[base] : FL_NONE;
  uint32_t P[2], cn[2];
  bool mine[2];
  fl_da_pos at[2];
  fl_da_words w[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const uint32_t i = 2 * lane + b;
    mine[b] = i < cnt;
    P[b] = base + (mine[b] ? end - 1 - i : start);
    cn[b] = g.pcnt[P[b]];
    at[b] = da_load(g, P[b]);
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) w[b] = da_words(g, P[b], cn[b], mine[b]);
  uint32_t spins = 0;
  while (__any(da_missing(w[0]) || da_missing(w[1]))) {
    if (!wait_more(spins, g.wait)) break;
    da_again(g, P[0], w[0]);
    da_again(g, P[1], w[1]);
  }
  const double pre[2] = {da_pre(cn[0], at[0].area, w[0], mine[0]), da_pre(cn[1], at[1].area, w[1], mine[1])};
  // the value before the tile
  double carry = FL_NEG0;
  if (!first) {
    if (s_carry && wave > 0) {
      carry = await_lds(s_carry + wave - 1, g.wait);
    } else {
      double* word = g.cover + base + end - 1;
      carry = await(word, true, 0.0, g.wait);
      if (lane == 0) *reinterpret_cast<unsigned long long*>(word) = FL_SENT;
    }
  }
  double r[2];
  if (__any((mine[0] && (cn[0] & FL_LIST_OVERFLOW)) || (mine[1] && (cn[1] & FL_LIST_OVERFLOW))))
    da_tile_walk<2, true>(g, at, cn, mine, pre, w, false, carry, lane, r);
  else
    da_long_fold(max(da_posts(cn[0], mine[0]), da_posts(cn[1], mine[1])), pre, w, carry, lane, last, r);
  const double out = of_lane(r[1], last);  // (a position past the tile passed it on)
  if (lane == 0) {
    if (head) da_hand_over(g, base, pd, pp, out);
    else if (s_carry && wave + 1 < FL_FOLD_WAVES) publish_lds(s_carry + wave, out);
    else publish(g.cover + base + start - 1, out);
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    da_give_back(g, P[b], cn[b], mine[b]);
    if (mine[b]) da_store(g, P[b], at[b], r[b]);
  }
}

// Rounds 0..min(deepest, cap - 1) of the drainage-area sweep, deepest first.
__global__ void __launch_bounds__(64 * FL_FOLD_WAVES)
k_da_fold(const uint32_t* __restrict__ guard, uint32_t cap, fl_flow f, fl_da_args g) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t deepest = *f.maxld;
  if (*guard != 0) return;  // the iteration is redone
  const uint32_t rounds = deepest < cap ? deepest + 1 : cap;
  const uint32_t total = f.ucum[rounds];
  fl_rounds R = load_rounds(f, 0, rounds, lane);
  const bool once = (uint64_t)gridDim.x * FL_FOLD_WAVES >= total;
  if (once && (uint64_t)blockIdx.x * FL_FOLD_WAVES >= total) return;  // the others are enough
  __shared__ uint32_t s_ticket;
  __shared__ double s_carry[FL_FOLD_WAVES];  // from each wavefront's tile to the next one's
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_ticket = atomicAdd(f.ticket_da, (uint32_t)FL_FOLD_WAVES);
    if (threadIdx.x < FL_FOLD_WAVES) s_carry[threadIdx.x] = bits_double(FL_SENT);
    __syncthreads();
    const uint32_t t = s_ticket;
    if (t >= total) return;
    if (t + wave < total) {
      const fl_unit un = find_unit(f, R, rounds, total - 1 - (t + wave), true, lane);
      da_unit(g, un, 65u - f.long_min, lane, s_carry, wave);
    }
    if (once) return;
  }
}

// Rounds lsplit..deepest, deepest first, in one workgroup with a barrier
// between rounds: the small deep rounds of an iteration whose sizes the host
// knows, and every round of one whose waits ended without their values.  (A
// chain's tiles still wait for each other: each wavefront takes its units in
// order, so the first one not finished waits for nothing.)
__global__ void __launch_bounds__(64 * FL_TAIL_WAVES)
k_da_tail(const uint32_t* __restrict__ guard, uint32_t lsplit, fl_flow f, fl_da_args g) {
  const uint32_t top = *f.maxld;
  if (*guard != 0 || top > 0xfffffffeu) return;  // the iteration is redone
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  for (uint32_t l = top + 1; l-- > lsplit;) {
    const uint32_t n = f.ucum[l + 1] - f.ucum[l];
    for (uint32_t i = wave; i < n; i += FL_TAIL_WAVES)
      da_unit(g, unit_of(l, i, f.boff[2ull * l + 1], f.boff[2ull * l + 2], f.bnoff[2ull * l], f.bnoff[2ull * l + 1],
                         65u - f.long_min),
              65u - f.long_min, lane, nullptr, wave);
    __syncthreads();
  }
}

// The arrays of the response-time sweep.
struct fl_tau_args {
  const uint32_t* pcnt;
  const uint32_t* ppos;  // at a chain's base: the position of its head's receiver, FL_NONE at a basin outlet
  const uint2* cmeta;     // long chains' tiles: (base, length) at the head's
  const double* xp;
  double* taup;
  // with max slopes: by position the basin outlet's position, uplift,
  // tan(max slope), receiver distance and old elevation; new elevations
  const uint32_t* pro;
  const double* up;
  const double* tanp;
  const double* dp;
  const double* hop;
  double* hnp;
  fl_patience wait;
};

// Response times of a tile, each from the position before it (a chain's head
// from its receiver's value `tp`).
//
// The reference's step rt = 0.0 + (rt_next + x) adds 0.0, which changes
// nothing unless y = rt_next + x is -0.0 (0.0 + -0.0 = +0.0; a NaN y is
// already quiet and passes unchanged).  A sum is -0.0 only when both terms
// are, and no running value is: a basin's outlet starts at 0.0 + (...),
// never -0.0, and every other chain starts from its receiver's value.  So
// the chains take the single add, bit for bit the same.
//
// A short-chain tile, one position a lane, by `steps` serial steps:
__device__ __forceinline__ double tau_short_fold(double x, bool head, double tp, uint32_t steps) {
  double s = tp, r = tp;
#pragma unroll 4
  for (uint32_t i = 0; i < steps; ++i) {
    s = from_prev(s, r);
    r = (head ? tp : s) + x;
  }
  return r;
}
// A long chain's tile, B positions a lane, from the value before it (positions
// past the tile hold -0.0).
template <int B>
__device__ __forceinline__ void tau_long_fold(const double (&x)[B], double tp, uint32_t lane, uint32_t last,
                                              double (&r)[B]) {
  tile_fold(
      tp, lane, last,
      [&](double v) {
#pragma unroll
        for (int b = 0; b < B; ++b) r[b] = v = v + x[b];
        return v;
      });
}

// Elevations of a tile with max slopes (generator.rs:177-202): z the value
// without the limit, hp the receiver's new elevation at a chain's head
// (`first`) and before the tile, t and d tan(max slope) and the receiver's
// distance.  A site is limited when RN((z - hp) / d) > t; then its elevation
// is hp + t * d.  `fixed` lanes keep z.
//
// The division stays off the serial chain: with d > 0 and t finite,
//   z - hp > t * d * (1 + 2^-50)  implies  (z - hp) / d >= the double after t,
//   z - hp < t * d * (1 - 2^-50)  implies  (z - hp) / d < t,
// and rounding is monotonic, so either comparison decides it; only a
// difference between the two bounds divides.  A site that is not limited
// ends what its receiver's elevation changes, so the lanes settle after as many
// steps as the tile's longest run of limited sites takes.
struct fl_clamp_pos {
  double z, t, d;
  bool fixed;
};
template <int B, bool heads>
__device__ __forceinline__ void clamp_tile_fold(const fl_clamp_pos (&q)[B], bool first, double hp, uint32_t steps,
                                                double (&h)[B]) {
  double lo[B], hi[B];
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const double td = q[b].t * q[b].d, mag = __builtin_fabs(td), at = __builtin_fabs(q[b].t);
    if (q[b].fixed || q[b].t != q[b].t) {
      lo[b] = hi[b] = __builtin_inf();  // below both: not limited
    } else if (q[b].d > 0.0 && mag >= 0x1p-900 && mag <= 0x1p900 && at >= 0x1p-900 && at <= 0x1p900) {
      lo[b] = td - mag * 0x1p-50;
      hi[b] = td + mag * 0x1p-50;
    } else {
      lo[b] = -__builtin_inf();  // between both: divides
      hi[b] = __builtin_inf();
    }
    h[b] = q[b].z;
  }
  double s = hp;
  for (uint32_t i = 0; i < steps; ++i) {
    const double was = s;
    s = from_prev(s, h[B - 1]);
    // every lane's value is what its last step started from: settled
    if (i > 0 && !__any(!same_bits(s, was))) break;
    double v = heads && first ? hp : s;
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const double diff = q[b].z - v;
      bool c = diff > hi[b];
      const bool near = !c && !(diff < lo[b]) && !q[b].fixed;
      if (__any(near)) c = near ? diff / q[b].d > q[b].t : c;
      c = c && !q[b].fixed;
      h[b] = v = c ? v + q[b].t * q[b].d : q[b].z;
    }
  }
}

// One unit of the response-time sweep, head to tail along its chains:
// rt_i = rt_next + x_i, the basin outlet first (its receiver is itself).  With
// clamp, also the elevation recurrence, whose max-slope limit depends on the
// receiver's new elevation.
template <bool clamp>
__device__ __forceinline__ void tau_unit(const fl_tau_args& g, const fl_unit& un, uint32_t stride, uint32_t lane) {
  if (un.chain == FL_NONE) {
    uint32_t cn;
    const fl_short_tile t = short_tile(g.pcnt, un.T, un.n1, stride, lane, cn);
    const uint32_t P = t.P;
    const double x = g.xp[P];
    const bool head = t.own && (cn & FL_HEAD) != 0;
    const uint32_t pp = head ? g.ppos[P] : FL_NONE;
    const bool outlet = head && pp == FL_NONE;
    double u = 0.0, tm = 0.0, d = 1.0, ho = 0.0;
    uint32_t ro = 0;
    if (clamp) {
      u = g.up[P];
      tm = g.tanp[P];
      d = g.dp[P];
      ho = g.hop[P];
      ro = g.pro[P];
    }
    const double tp = await(g.taup + pp, head && !outlet, 0.0, g.wait);
    const uint32_t steps = run_steps(__ballot(t.own && !head));
    const double tau[1] = {tau_short_fold(x, head, tp, steps)};
    if (t.own) publish(g.taup + P, tau[0]);
    if (clamp) {
      const bool deep = un.l > 0;
      double to = await(g.taup + ro, deep && t.own, 0.0, g.wait);
      double h0 = await(g.hnp + ro, deep && t.own, 0.0, g.wait);
      if (!deep) {
        // the chains of the outlets: an outlet's elevation is
        // h_o + U_o * max(0, 0), limited against its own old elevation
        to = tau[0];
        h0 = ho + u * rust_max(tau[0] - tau[0], 0.0);
        if ((h0 - ho) / d > tm) h0 = ho + tm * d;
        double st = to, sh = h0;
        for (uint32_t i = 1; i < steps; ++i) {
          st = from_prev(st, to);
          sh = from_prev(sh, h0);
          if (!head) {
            to = st;
            h0 = sh;
          }
        }
      }
      const double z = outlet ? h0 : h0 + u * rust_max(tau[0] - to, 0.0);
      const double hp = await(g.hnp + pp, head && !outlet, 0.0, g.wait);
      const fl_clamp_pos q[1] = {{z, tm, d, outlet || !t.own}};
      double h[1];
      clamp_tile_fold<1, true>(q, head, hp, steps, h);
      if (t.own) publish(g.hnp + P, h[0]);
    }
    return;
  }
  // a long chain: tiles of B positions a lane, loaded two tiles ahead
  constexpr int B = clamp ? 2 : 4;
  constexpr uint32_t tile = 64 * B;
  const uint2 m = g.cmeta[un.chain];
  const uint32_t base = uniform(m.x) & ~FL_CHAIN_TAIL, len = uniform(m.y);
  if (len & FL_CHAIN_PART) return;  // its chain is taken at the head's tile
  const uint32_t pp = uniform(g.ppos[base]);
  const bool outlet = pp == FL_NONE;  // the chain of a basin outlet
  struct In {
    double x[B], u[B], t[B], d[B];
  };
  auto load = [&](uint32_t t0, In& q) {
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const uint32_t i = t0 + B * lane + b, P = base + (i < len ? i : len - 1);
      q.x[b] = g.xp[P];
      if (clamp) {
        q.u[b] = g.up[P];
        q.t[b] = g.tanp[P];
        q.d[b] = g.dp[P];
      }
    }
  };
  double tau_c = 0.0, h_c = 0.0, to = 0.0, h0 = 0.0;
  auto fold = [&](uint32_t t0, const In& q) {
    const uint32_t cnt = len - t0 < tile ? len - t0 : tile;
    const uint32_t P = base + t0 + B * lane;
    const uint32_t last = (cnt - 1) / B;  // the lane of the tile's last position
    double x[B], tau[B];
#pragma unroll
    for (int b = 0; b < B; ++b) x[b] = B * lane + b < cnt ? q.x[b] : FL_NEG0;
    tau_long_fold<B>(x, tau_c, lane, last, tau);
#pragma unroll
    for (int b = 0; b < B; ++b)
      if (B * lane + b < cnt) publish(g.taup + P + b, tau[b]);
    tau_c = of_lane(tau[B - 1], last);  // (positions past the tile pass it on)
    if (clamp) {
      const bool first = t0 == 0 && outlet;
      if (first) {
        // (see the short chains) lane 0's first position is the outlet
        const double ho = g.hop[base];
        double nh = ho + q.u[0] * rust_max(tau[0] - tau[0], 0.0);
        if ((nh - ho) / q.d[0] > q.t[0]) nh = ho + q.t[0] * q.d[0];
        to = of_lane(tau[0], 0);
        h0 = of_lane(nh, 0);
      }
      fl_clamp_pos c[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const bool fixed = first && lane == 0 && b == 0;
        c[b] = fl_clamp_pos{fixed ? h0 : h0 + q.u[b] * rust_max(tau[b] - to, 0.0), q.t[b], q.d[b],
                            fixed || B * lane + b >= cnt};
      }
      double h[B];
      clamp_tile_fold<B, false>(c, false, h_c, last + 1, h);
#pragma unroll
      for (int b = 0; b < B; ++b)
        if (B * lane + b < cnt) publish(g.hnp + P + b, h[b]);
      h_c = of_lane(h[B - 1], last);
    }
  };
  In q0, q1;
  load(0, q0);
  load(tile, q1);
  uint32_t ro = 0;
  if (clamp) ro = g.pro[base];
  tau_c = await(g.taup + pp, !outlet, 0.0, g.wait);
  if (clamp) {
    to = await(g.taup + ro, !outlet, 0.0, g.wait);
    h0 = await(g.hnp + ro, !outlet, 0.0, g.wait);
    h_c = await(g.hnp + pp, !outlet, 0.0, g.wait);
  }
  for (uint32_t t0 = 0;;) {
    fold(t0, q0);
    if ((t0 += tile) >= len) break;
    load(t0 + tile, q0);
    fold(t0, q1);
    if ((t0 += tile) >= len) break;
    load(t0 + tile, q1);
  }
}

// Rounds 0..min(deepest, cap - 1) of the response-time sweep, shallowest
// first.
template <bool clamp>
__global__ void __launch_bounds__(64 * FL_FOLD_WAVES)
k_tau_fold(const uint32_t* __restrict__ guard, uint32_t cap, fl_flow f, fl_tau_args g) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t deepest = *f.maxld;
  if (*guard != 0) return;  // the iteration is redone
  const uint32_t rounds = deepest < cap ? deepest + 1 : cap;
  const uint32_t total = f.ucum[rounds];
  fl_rounds R = load_rounds(f, 0, rounds, lane);
  const bool once = (uint64_t)gridDim.x * FL_FOLD_WAVES >= total;
  if (once && (uint64_t)blockIdx.x * FL_FOLD_WAVES >= total) return;  // the others are enough
  __shared__ uint32_t s_ticket;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_ticket = atomicAdd(f.ticket_tau, (uint32_t)FL_FOLD_WAVES);
    __syncthreads();
    const uint32_t t = s_ticket;
    if (t >= total) return;
    if (t + wave < total) {
      const fl_unit un = find_unit(f, R, rounds, t + wave, false, lane);
      tau_unit<clamp>(g, un, 65u - f.long_min, lane);
    }
    if (once) return;
  }
}

// Rounds lsplit..deepest, shallowest first, in one workgroup (see k_da_tail).
template <bool clamp>
__global__ void __launch_bounds__(64 * FL_TAIL_WAVES)
k_tau_tail(const uint32_t* __restrict__ guard, uint32_t lsplit, fl_flow f, fl_tau_args g) {
  const uint32_t top = *f.maxld;
  if (*guard != 0 || top > 0xfffffffeu) return;  // the iteration is redone
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  for (uint32_t l = lsplit; l <= top; ++l) {
    const uint32_t n = f.ucum[l + 1] - f.ucum[l];
    for (uint32_t i = wave; i < n; i += FL_TAIL_WAVES)
      tau_unit<clamp>(g, unit_of(l, i, f.boff[2ull * l + 1], f.boff[2ull * l + 2], f.bnoff[2ull * l],
                                 f.bnoff[2ull * l + 1], 65u - f.long_min),
                      65u - f.long_min, lane);
    __syncthreads();
  }
}

// Back to site order: response time, new elevation (computed here when no
// site has a max slope: h_i' = h_o' + U_i * max(rt_i - rt_o, 0) with
// h_o' = h_o + U_o * max(0, 0), generator.rs:178-180) and the changed flag
// (generator.rs:201).  One thread per site: the site-ordered accesses are
// coalesced, the position-ordered ones (spos, root: k_chain_perm) are gathers.
// A leaf takes its one step from its receiver's values here: rt_i = rt_next + x_i,
// x_i = 1.0 / (K_i * a_i^0.5) * d_i (generator.rs:162-173), and the max-slope
// limit against the receiver's new elevation.  Sites outside every basin were
// settled by k_chain_perm.  In a batch (tid != null) a terrain that stopped
// iterating keeps its elevations and each terrain has its own flag.
struct fl_leaf_in {
  const double* area;
  const double* K;
  const double* dnext;
  const double* tan_ms;
};
__global__ void k_tau_scatter(uint32_t bs, const uint32_t* __restrict__ guard, uint32_t n, const uint32_t* __restrict__ spos,
                              const uint32_t* __restrict__ root, const uint8_t* __restrict__ is_outlet,
                              const double* __restrict__ taup,
                              const double* __restrict__ hnp, const double* __restrict__ U, fl_leaf_in lf,
                              const double* __restrict__ h, double* __restrict__ h2, double* __restrict__ tau,
                              int* __restrict__ flags, int clamp, const uint32_t* __restrict__ tid,
                              const uint8_t* __restrict__ act, uint32_t* __restrict__ tchanged,
                              uint8_t* __restrict__ chg, uint8_t* __restrict__ dirty,
                              const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col) {
  const uint32_t v = gid(bs);
  // the basin marks were read by this iteration's k_children: clear them for
  // the next iteration's receivers (also when the iteration is redone: a
  // redo marks again from its own receivers)
  if (v < n) dirty[v] = 0;
  // the site's own words are read together with the guard (one load
  // latency), then the second level (outlet flag, positions, the outlet's
  // elevation and uplift) together
  const bool in = v < n;
  const uint32_t kind = in ? act[v] : 0u;
  const double hv = in ? h[v] : 0.0;
  uint32_t o = 0u, P = FL_NONE, rb = 0u, re = 0u, g = 0u;  // (the row, for the change marks)
  double uv = 0.0, K = 0.0, a = 0.0, d = 1.0, tm = 0.0;
  if (kind) {
    o = root[v];
    P = spos[v];
    rb = rp[v];
    re = rp[v + 1];
    uv = U[v];
    g = tid ? tid[v] : 0u;
  }
  const bool leaf = (kind & FL_LEAF) != 0;
  if (leaf) {
    K = lf.K[v];
    a = lf.area[v];
    d = lf.dnext[v];
    if (clamp) tm = lf.tan_ms[v];
  }
  if (*guard != 0) return;  // the iteration is redone
  bool changed = false;
  if (in && !kind) {
    // a site of a basin that keeps its tree (or of a terrain that stopped)
    // keeps its elevation
    h2[v] = hv;
  } else if (kind) {
    const uint8_t outlet = is_outlet ? is_outlet[o] : 1;
    // (a site of a lake basin reads these for nothing; its values were
    // written by k_chain_perm)
    const bool alone = leaf && o == v;  // an outlet that nothing drains to
    const uint32_t Po = alone || (clamp && !leaf) || !outlet ? 0u : spos[o];
    const double h_o = clamp ? 0.0 : h[o], u_o = clamp ? 0.0 : U[o];
    if (outlet) {
      double tk = alone ? 0.0 : taup[P], nh;
      const double hp = clamp && !alone ? hnp[P] : 0.0;
      if (leaf) tk = tk + 1.0 / (K * rust_pow_half(a)) * d;
      if (clamp && !leaf) {
        nh = hp;
      } else {
        const double to = alone ? tk : taup[Po];
        const double ho = clamp ? (alone ? hv + uv * rust_max(to - to, 0.0) : hnp[Po])
                                : h_o + u_o * rust_max(to - to, 0.0);
        nh = (v == o) ? ho : ho + uv * rust_max(tk - to, 0.0);
        if (clamp) {
          const double below = alone ? hv : hp;  // (an outlet: its own old elevation)
          if ((nh - below) / d > tm) nh = below + tm * d;
        }
      }
      tau[v] = tk;
      h2[v] = nh;
      changed = nh != hv;
      if (changed && tchanged) tchanged[g] = 1;
    }
  }
  // neighbourhood change flags for the next iteration's receivers (zeroed by
  // this iteration's k_receivers; sites outside every basin kept their
  // elevation in k_chain_perm): a changed site marks itself and its
  // neighbours (rows are symmetric)
  if (changed) {
    chg[v] = 1;
    for (uint32_t k = rb; k < re; k += FL_ROW) {
      uint32_t c[FL_ROW];  // loaded together (past the row's end: its last entry again)
#pragma unroll
      for (int j = 0; j < FL_ROW; ++j) c[j] = col[min(k + j, re - 1)];
#pragma unroll
      for (int j = 0; j < FL_ROW; ++j) chg[c[j]] = 1;
    }
  }
  if (__any(changed) && (threadIdx.x & 63u) == 0) flags[FL_FLAG_CHANGED] = 1;
}

// ----------------------------------------------------------- compaction ---

namespace {
// Terrain of new site v: the last q with new_off[q] <= v.
__device__ __forceinline__ uint32_t terrain_of(const fl_compact_map& m, uint32_t v) {
  uint32_t lo = 0, hi = m.count;  // new_off[lo] <= v < new_off[hi]
  while (hi - lo > 1) {
    uint32_t mid = (lo + hi) >> 1;
    if (m.new_off[mid] <= v) lo = mid;
    else hi = mid;
  }
  return lo;
}
__device__ __forceinline__ uint32_t shift_site(uint32_t x, const fl_compact_map& m, uint32_t q) {
  return x == FL_NONE ? FL_NONE : x - m.old_off[q] + m.new_off[q];
}
}  // namespace

// New sites [v0, v1) of a union of n_new sites and nnz_new entries, taken
// from the terrains of one source union (m, terrain q of the map becomes
// terrain tid0 + q of the new union).
__global__ void k_compact_sites(uint32_t bs, uint32_t v0, uint32_t v1, uint32_t n_new, uint32_t nnz_new, uint32_t tid0,
                                fl_compact_map m, fl_dev_terrain ot, fl_dev_work ow, fl_dev_terrain nt,
                                fl_dev_work nw, uint32_t* __restrict__ new_tid) {
  uint32_t v = v0 + gid(bs);
  if (v >= v1) return;
  uint32_t q = terrain_of(m, v);
  uint32_t src = v - m.new_off[q] + m.old_off[q];
  nt.row_ptr[v] = ot.row_ptr[src] - m.old_eoff[q] + m.new_eoff[q];
  if (v == n_new - 1) nt.row_ptr[n_new] = nnz_new;
  nt.area[v] = ot.area[src];
  nt.erod[v] = ot.erod[src];
  nt.uplift[v] = ot.uplift[src];
  nt.tan_ms[v] = ot.tan_ms[src];
  nt.init_h[v] = ot.init_h[src];
  nt.is_outlet[v] = ot.is_outlet[src];
  nt.rank[v] = shift_site(ot.rank[src], m, q);
  nt.order[v] = shift_site(ot.order[src], m, q);  // rank positions share the terrain's site range
  nw.h[v] = ow.h[src];
  nw.A[v] = ow.A[src];
  new_tid[v] = tid0 + q;
}

__global__ void k_compact_entries(uint32_t bs, uint32_t v0, uint32_t v1, fl_compact_map m, fl_dev_terrain ot,
                                  fl_dev_terrain nt) {
  uint32_t v = v0 + gid(bs);
  if (v >= v1) return;
  uint32_t q = terrain_of(m, v);
  uint32_t src = v - m.new_off[q] + m.old_off[q];
  uint32_t b = ot.row_ptr[src], e = ot.row_ptr[src + 1];
  uint32_t d = m.new_eoff[q] - m.old_eoff[q];
  for (uint32_t k = b; k < e; ++k) {
    nt.col[k + d] = ot.col[k] - m.old_off[q] + m.new_off[q];
    nt.len[k + d] = ot.len[k];
  }
}

// Verification: the reference's traversal of one basin
// (DrainageBasin::construct, drainage_basin.rs:13-36): start at the outlet,
// then for each site in order append its children in row order.  One
// workgroup; children counts are prefix-summed per chunk of 1024 sites so
// the appended order equals the sequential one.
__global__ void __launch_bounds__(1024)
k_basin_order(uint32_t outlet, uint32_t cap, const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
              const uint32_t* __restrict__ next, const unsigned long long* __restrict__ cmask,
              uint32_t* __restrict__ order, uint32_t* __restrict__ len_out) {
  __shared__ uint32_t s_scan[1024];
  __shared__ uint32_t s_tail;
  uint32_t tid = threadIdx.x;
  if (tid == 0) {
    order[0] = outlet;
    s_tail = 1;
  }
  __syncthreads();
  uint32_t head = 0;
  while (head < s_tail) {
    uint32_t end = s_tail;
    for (uint32_t chunk = head; chunk < end; chunk += 1024) {
      uint32_t i = chunk + tid;
      uint32_t u = FL_NONE, cnt = 0, b = 0, deg = 0;
      unsigned long long m = 0;
      if (i < end) {
        u = order[i];
        b = rp[u];
        deg = rp[u + 1] - b;
        m = cmask[u];
        for (uint32_t s = 0; s < deg; ++s) cnt += is_child(m, deg, s, b, col, next, u) ? 1u : 0u;
      }
      s_scan[tid] = cnt;
      __syncthreads();
      for (uint32_t off = 1; off < 1024; off <<= 1) {
        uint32_t t = tid >= off ? s_scan[tid - off] : 0;
        __syncthreads();
        s_scan[tid] += t;
        __syncthreads();
      }
      uint32_t base = s_tail + s_scan[tid] - cnt;
      if (i < end && cnt) {
        for (uint32_t s = 0; s < deg; ++s)
          if (is_child(m, deg, s, b, col, next, u) && base < cap) order[base++] = col[b + s];
      }
      __syncthreads();
      if (tid == 1023) s_tail = min(cap, s_tail + s_scan[1023]);
      __syncthreads();
    }
    head = end;
  }
  if (tid == 0) *len_out = s_tail;
}

// The arrays of new terrains that are read before they are written: hand-over
// words without values, bucket entries and basin roots zero.  One launch for 16.
struct fl_new_arrays {
  uint32_t* zero[7];  // three of n, four of n + FL_BUCKET_PAD
  unsigned long long *cval, *cover;
};
__global__ void k_init_arrays(uint32_t bs, uint32_t n, fl_new_arrays w) {
  const uint32_t i = gid(bs);
#pragma unroll
  for (int k = 0; k < 7; ++k)
    if (i < (k < 3 ? n : n + FL_BUCKET_PAD)) w.zero[k][i] = 0;
  if (i >= n) return;
  w.cover[i] = FL_SENT;
  for (uint32_t k = 0; k < FL_LIST; ++k) w.cval[(uint64_t)k * n + i] = FL_SENT;
}

// Zero the control block and the first `nb` bucket entries.
__global__ void k_clear_iter(uint32_t bs, uint32_t nb, uint32_t* __restrict__ ctrl, uint32_t* __restrict__ bcnt,
                             uint32_t* __restrict__ bnodes, uint32_t* __restrict__ bcur,
                             uint32_t* __restrict__ bncur) {
  uint32_t i = gid(bs);
  if (i < FL_CTRL_WORDS) ctrl[i] = 0;
  if (i < nb) {
    bcnt[i] = 0;
    bnodes[i] = 0;
    bcur[i] = 0;
    bncur[i] = 0;
  }
}

// A pipelined iteration's end: its control block and the terrains' changed
// flags to their pinned host slots, and both cleared for the next iteration's
// (one launch for two copies and two fills).  The guard of a too deep
// decomposition stays up: it left its tree half made, and an iteration already
// enqueued behind it must not follow that (the redo's k_clear_iter takes it down).
__global__ void k_report(uint32_t bs, uint32_t count, uint32_t* __restrict__ ctrl, uint32_t* __restrict__ host_ctrl,
                         uint32_t G, uint32_t* __restrict__ tchanged, uint32_t* __restrict__ host_tchanged) {
  const uint32_t i = gid(bs);
  if (i >= count) return;
  if (i < FL_CTRL_WORDS) {
    host_ctrl[i] = ctrl[i];
    if (i != FL_FLAG_DEEP) ctrl[i] = 0;
  }
  if (tchanged && i < G) {
    host_tchanged[i] = tchanged[i];
    tchanged[i] = 0;
  }
}

// --------------------------------------------------------- launchers -----

namespace {
inline dim3 grid_for(uint64_t n, uint32_t block) { return dim3((uint32_t)((n + block - 1) / block)); }
}  // namespace

thread_local fl_profiler* fl_current_profiler = nullptr;

hipEvent_t fl_profiler::get() {
  if (!pool.empty()) {
    hipEvent_t e = pool.back();
    pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  (void)hipEventCreate(&e);
  return e;
}

void fl_profiler::record(hipStream_t s, const char* name, hipEvent_t a, hipEvent_t b, uint64_t units) {
  pending.push_back({name, a, b, units});  // flushed on query: the host may fill in units later
  (void)s;
}

void fl_profiler::flush() {
  for (const Rec& r : pending) {
    float ms = 0.f;
    (void)hipEventSynchronize(r.b);
    (void)hipEventElapsedTime(&ms, r.a, r.b);
    auto& t = totals[r.name];
    t.launches += 1;
    t.ms += ms;
    t.units += r.units;
    pool.push_back(r.a);
    pool.push_back(r.b);
  }
  pending.clear();
}

void fl_profiler::reset() {
  flush();
  totals.clear();
}

fl_profiler::~fl_profiler() {
  flush();
  for (hipEvent_t e : pool) (void)hipEventDestroy(e);
}

// `units`: the launch's work items for the profile (sites or positions).  A
// profiled launch passes its two events to the dispatch itself
// (hipExtLaunchKernelGGL), which stamps them with the kernel's own start and
// end: the kernel's execution time, without the queue's dispatch gap.
#define FL_LAUNCH_GRID(kernel, grid, block, units, stream, ...)                    \
  do {                                                                            \
    fl_profiler* prof_ = fl_current_profiler;                                     \
    if (prof_) {                                                                  \
      hipEvent_t a_ = prof_->get(), b_ = prof_->get();                            \
      hipExtLaunchKernelGGL(kernel, (grid), (block), 0, (stream), a_, b_, 0,      \
                            __VA_ARGS__);                                         \
      prof_->record((stream), #kernel, a_, b_, (units));                          \
    } else {                                                                      \
      hipLaunchKernelGGL(kernel, (grid), (block), 0, (stream), __VA_ARGS__);     \
    }                                                                             \
  } while (0)

// Per-site kernels: one thread per item in workgroups of fl_site_block
// threads (the tuned workgroup size of the call in progress).
thread_local uint32_t fl_site_block = 256;
// The workgroup size is also the kernel's first argument, taken into a local
// first: a launch recorded for later replay holds the value of its time.
#define FL_LAUNCH_U(kernel, count, units, stream, ...)                                                    \
  do {                                                                                                      \
    const uint32_t bs_ = fl_site_block;                                                                     \
    if ((count) > 0)                                                                                        \
      FL_LAUNCH_GRID(kernel, grid_for((count), bs_), dim3(bs_), (units), (stream), bs_, __VA_ARGS__);      \
  } while (0)
#define FL_LAUNCH(kernel, count, stream, ...) FL_LAUNCH_U(kernel, count, count, stream, __VA_ARGS__)

void fl_launch_receivers(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool keep_unchanged,
                         bool mark) {
  FL_LAUNCH(k_receivers, t.n, s, t.n, t.row_ptr, t.col, t.len, w.h, t.is_outlet, w.next, w.dnext, w.flags,
            keep_unchanged ? w.chg_prev : (const uint8_t*)nullptr, w.next_prev, w.dnext_prev, w.root_prev,
            mark ? w.dirty : (uint8_t*)nullptr, w.chg);
}

void fl_launch_sub_labels(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w) {
  // rounds until a path of four times sqrt(n) sites is walked
  uint32_t rounds = 0;
  for (uint64_t reach = 4; reach * reach < 16ull * t.n; reach *= 4) rounds++;
  FL_LAUNCH(k_sub_start, t.n, s, t.n, w.next, w.sub);
  for (uint32_t r = 0; r < rounds; r++) FL_LAUNCH(k_sub_jump, t.n, s, t.n, w.sub);
  FL_LAUNCH(k_sub_settle, t.n, s, t.n, w.sub, (unsigned long long*)w.lake_key);
}

void fl_launch_lake_join(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool few) {
  if (few)
    FL_LAUNCH(k_lake_offers, t.n, s, t.n, t.row_ptr, t.col, t.rank, w.sub, t.is_outlet,
              (unsigned long long*)w.lake_key);
  else
    FL_LAUNCH(k_lake_keys, t.n, s, t.n, t.row_ptr, t.col, t.rank, w.sub, t.is_outlet,
              (unsigned long long*)w.lake_key);
  FL_LAUNCH(k_lake_flip, t.n, s, t.n, t.row_ptr, t.col, t.len, t.order, (const unsigned long long*)w.lake_key,
            t.is_outlet, w.next, w.dnext);
}

void fl_launch_dirty(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w) {
  FL_LAUNCH(k_dirty, t.n, s, t.n, w.next, w.dnext, w.next_prev, w.dnext_prev, w.root_prev, w.dirty);
}

void fl_launch_children(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool full, const uint32_t* tid,
                        const uint8_t* t_active) {
  FL_LAUNCH(k_children, t.n, s, t.n, t.row_ptr, t.col, w.next, w.A, (unsigned long long*)w.cmask, w.hc, w.act,
            full ? (const uint8_t*)nullptr : (const uint8_t*)w.dirty, w.root_prev, tid, t_active,
            (unsigned long long*)w.cp, (unsigned long long*)w.rt, w.root);
}

void fl_launch_chain_jump(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t round) {
  uint32_t r = round < FL_MAX_JUMP_ROUNDS ? round : FL_MAX_JUMP_ROUNDS - 1;
  uint32_t* fset = w.ctrl + FL_CTRL_JUMPS + r;
  const uint32_t* prev = r > 0 ? w.ctrl + FL_CTRL_JUMPS + r - 1 : nullptr;
  FL_LAUNCH(k_chain_jump, t.n, s, t.n, (unsigned long long*)w.cp, (unsigned long long*)w.rt, fset, prev, w.act, w.hc,
            w.head_base);
}

void fl_launch_chain_count(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool lakes) {
  uint32_t per = FL_BUCKET_BLOCK * FL_BUCKET_PER_THREAD;
  FL_LAUNCH_GRID(k_bucket_count, dim3((t.n + per - 1) / per), dim3(FL_BUCKET_BLOCK), t.n, s, w.guard, t.n,
                 (const unsigned long long*)w.cp, (const unsigned long long*)w.rt,
                 lakes ? t.is_outlet : (const uint8_t*)nullptr, w.bcnt, w.bnodes, w.counters, w.sub, w.long_min, w.act);
}

void fl_launch_chain_layout(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool lakes, bool scan) {
  const uint8_t* outlets = lakes ? t.is_outlet : (const uint8_t*)nullptr;
  uint32_t per = FL_BUCKET_BLOCK * FL_BUCKET_PER_THREAD;
  const dim3 grid((t.n + per - 1) / per), block(FL_BUCKET_BLOCK);
  const fl_bucket_out bo{w.boff, w.bnoff, w.ucum, w.ctrl, w.sub};
  if (scan) {
    FL_LAUNCH_GRID(k_bucket_place<true>, grid, block, t.n, s, w.guard, t.n, (const unsigned long long*)w.cp,
                   (const unsigned long long*)w.rt, outlets, w.bcnt, w.bnodes, bo, w.bcur, w.bncur, w.cmeta, w.pdest,
                   w.head_base, w.long_min, w.act);
  } else {
    FL_LAUNCH_GRID(k_bucket_scan, dim3(1), dim3(FL_SCAN_BLOCK), 0, s, t.n, w.long_min, w.ctrl, w.bcnt, w.bnodes,
                   w.boff, w.bnoff, w.ucum, grid.x, w.sub);
    FL_LAUNCH_GRID(k_bucket_place<false>, grid, block, t.n, s, w.guard, t.n, (const unsigned long long*)w.cp,
                   (const unsigned long long*)w.rt, outlets, w.bcnt, w.bnodes, bo, w.bcur, w.bncur, w.cmeta, w.pdest,
                   w.head_base, w.long_min, w.act);
  }
  fl_perm_out o{w.perm, w.pcnt, w.pdest, w.parea, w.pK, w.pdn, w.up, w.tanp, w.hop, w.ppos, w.pro, w.cval, w.spos};
  FL_LAUNCH(k_chain_perm, t.n, s, w.guard, t.n, (unsigned long long*)w.cp, (unsigned long long*)w.rt,
            w.next, outlets, w.head_base, o, t.area, t.erod, w.dnext, t.uplift, t.tan_ms,
            t.any_max_slope ? 1 : 0, w.A, w.tau, w.h, w.h2, w.counters + FL_CNT_MAXLD, w.bcnt, w.bnodes, w.bcur,
            w.bncur, t.row_ptr, t.col, (const unsigned long long*)w.cmask, w.hc, w.act, w.root);
}

namespace {
fl_flow flow(const fl_dev_work& w) {
  return fl_flow{w.counters + FL_CNT_MAXLD,       w.ucum, w.boff, w.bnoff, w.counters + FL_CNT_TICKET_DA,
                 w.counters + FL_CNT_TICKET_TAU, w.long_min};
}
fl_da_args da_args(const fl_dev_terrain& t, const fl_dev_work& w, bool clamp, uint32_t polls) {
  return fl_da_args{w.perm, w.pcnt,  w.cval, w.cover, w.parea, w.pK, w.pdn, w.pdest, w.ppos, w.cmeta, w.xp, w.taup,
                    clamp ? w.hnp : nullptr, t.row_ptr, t.col, w.next, (const unsigned long long*)w.cmask, w.hc,
                    w.head_base, t.area, w.A, {w.flags + FL_FLAG_STALL, polls}};
}
fl_tau_args tau_args(const fl_dev_work& w, uint32_t polls) {
  return fl_tau_args{w.pcnt, w.ppos, w.cmeta, w.xp, w.taup, w.pro, w.up, w.tanp, w.pdn, w.hop, w.hnp,
                     {w.flags + FL_FLAG_STALL, polls}};
}
dim3 fold_grid(uint32_t waves) { return dim3((std::max<uint32_t>(waves, 1) + FL_FOLD_WAVES - 1) / FL_FOLD_WAVES); }
}  // namespace

void fl_launch_da_fold(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t cap, uint32_t waves,
                       uint64_t positions, bool clamp) {
  const fl_da_args a = da_args(t, w, clamp, FL_SPIN_FOLD);
  FL_LAUNCH_GRID(k_da_fold, fold_grid(waves), dim3(64 * FL_FOLD_WAVES), positions, s, w.guard, cap, flow(w), a);
}

void fl_launch_da_tail(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t lsplit,
                       uint64_t positions, bool clamp) {
  const fl_da_args a = da_args(t, w, clamp, FL_SPIN_MAX);
  FL_LAUNCH_GRID(k_da_tail, dim3(1), dim3(64 * FL_TAIL_WAVES), positions, s, w.guard, lsplit, flow(w), a);
}

void fl_launch_tau_fold(hipStream_t s, const fl_dev_work& w, uint32_t cap, uint32_t waves, uint64_t positions,
                        bool clamp) {
  const fl_tau_args a = tau_args(w, FL_SPIN_FOLD);
  if (clamp)
    FL_LAUNCH_GRID(k_tau_fold<true>, fold_grid(waves), dim3(64 * FL_FOLD_WAVES), positions, s, w.guard, cap, flow(w),
                   a);
  else
    FL_LAUNCH_GRID(k_tau_fold<false>, fold_grid(waves), dim3(64 * FL_FOLD_WAVES), positions, s, w.guard, cap, flow(w),
                   a);
}

void fl_launch_tau_tail(hipStream_t s, const fl_dev_work& w, uint32_t lsplit, uint64_t positions, bool clamp) {
  const fl_tau_args a = tau_args(w, FL_SPIN_MAX);
  if (clamp)
    FL_LAUNCH_GRID(k_tau_tail<true>, dim3(1), dim3(64 * FL_TAIL_WAVES), positions, s, w.guard, lsplit, flow(w), a);
  else
    FL_LAUNCH_GRID(k_tau_tail<false>, dim3(1), dim3(64 * FL_TAIL_WAVES), positions, s, w.guard, lsplit, flow(w), a);
}

void fl_launch_tau_scatter(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool clamp, bool lakes,
                           const uint32_t* tid, const uint8_t* active, uint32_t* tchanged) {
  const fl_leaf_in lf{t.area, t.erod, w.dnext, t.tan_ms};
  FL_LAUNCH(k_tau_scatter, t.n, s, w.guard, t.n, w.spos, w.root, lakes ? t.is_outlet : (const uint8_t*)nullptr, w.taup,
            w.hnp, t.uplift, lf, w.h, w.h2, w.tau, w.flags, clamp ? 1 : 0, tid, w.act, tchanged, w.chg, w.dirty,
            t.row_ptr, t.col);
}

void fl_launch_clear_iter(hipStream_t s, const fl_dev_work& w, uint32_t nb) {
  uint32_t cnt = nb > FL_CTRL_WORDS ? nb : FL_CTRL_WORDS;
  FL_LAUNCH(k_clear_iter, cnt, s, nb, w.ctrl, w.bcnt, w.bnodes, w.bcur, w.bncur);
}

void fl_launch_report(hipStream_t s, const fl_dev_work& w, uint32_t* host_ctrl, uint32_t G, uint32_t* tchanged,
                      uint32_t* host_tchanged) {
  const uint32_t cnt = tchanged && G > FL_CTRL_WORDS ? G : FL_CTRL_WORDS;
  FL_LAUNCH(k_report, cnt, s, cnt, w.ctrl, host_ctrl, G, tchanged, host_tchanged);
}

void fl_launch_init_arrays(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t* const roots[3]) {
  const fl_new_arrays a{{roots[0], roots[1], roots[2], w.bcnt, w.bnodes, w.bcur, w.bncur},
                        (unsigned long long*)w.cval,
                        (unsigned long long*)w.cover};
  FL_LAUNCH(k_init_arrays, t.n + FL_BUCKET_PAD, s, t.n, a);
}

// (launched in parts: the kernel counts items in 32 bits)
void fl_launch_reset_words(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w) {
  for (uint32_t i = 0; i < FL_LIST; i++)
    FL_LAUNCH(k_fill_u64, t.n, s, t.n, (uint64_t*)w.cval + (uint64_t)i * t.n, FL_SENT);
  FL_LAUNCH(k_fill_u64, t.n, s, t.n, (uint64_t*)w.cover, FL_SENT);
}

void fl_launch_fill_u32(hipStream_t s, uint32_t* p, uint64_t count, uint32_t v) {
  FL_LAUNCH(k_fill_u32, count, s, (uint32_t)count, p, v);
}

void fl_launch_basin_order(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t outlet,
                           uint32_t* order, uint32_t* len_out) {
  FL_LAUNCH_GRID(k_basin_order, dim3(1), dim3(1024), t.n, s, outlet, t.n, t.row_ptr, t.col, w.next,
                 (const unsigned long long*)w.cmask, order, len_out);
}

void fl_launch_compact(hipStream_t s, const fl_compact_map& m, const fl_dev_terrain& ot, const fl_dev_work& ow,
                       const fl_dev_terrain& nt, const fl_dev_work& nw, uint32_t* new_tid, uint32_t v0, uint32_t v1,
                       uint32_t tid0) {
  FL_LAUNCH(k_compact_sites, v1 - v0, s, v0, v1, nt.n, nt.nnz, tid0, m, ot, ow, nt, nw, new_tid);
  FL_LAUNCH(k_compact_entries, v1 - v0, s, v0, v1, m, ot, nt);
}
