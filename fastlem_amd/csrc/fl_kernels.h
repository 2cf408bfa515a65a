// fl_kernels.h -- device buffers of one terrain and the kernel launchers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <map>
#include <string>
#include <vector>

// Per-kernel timing with HIP events recorded on the launch stream.
struct fl_profiler {
  struct Rec {
    const char* name;
    hipEvent_t a, b;
    uint64_t units;  // work items of the launch (sites or chain positions)
  };
  struct Total {
    uint64_t launches = 0;
    double ms = 0.0;
    uint64_t units = 0;
  };
  std::vector<Rec> pending;
  std::vector<hipEvent_t> pool;
  std::map<std::string, Total> totals;
  hipEvent_t get();
  void record(hipStream_t s, const char* name, hipEvent_t a, hipEvent_t b, uint64_t units);
  void flush();
  void reset();
  ~fl_profiler();
};

// Set by the C ABI for the duration of a call on a profiled context.
extern thread_local fl_profiler* fl_current_profiler;

// Control block read back once per phase: [flags | counters | boff head | bnoff head].
// FL_FLAG_DEEP: a pipelined iteration's decomposition is deeper than its
// placement takes (fl_dev_work::guard)
// FL_FLAG_STALL: a sweep's wait ended without its value
enum { FL_FLAG_LAKE = 0, FL_FLAG_DEEP = 1, FL_FLAG_STALL = 2, FL_FLAG_CHANGED = 3, FL_NUM_FLAGS = 4 };
enum {
  FL_CNT_MAXLD = 0,
  FL_CNT_CHAINS = 1,
  FL_CNT_POSITIONS = 2,
  FL_CNT_TICKET_DA = 3,  // units taken from the sweeps
  FL_CNT_TICKET_TAU = 4,
  FL_CNT_LEAVES = 5,  // active sites on no chain
  FL_NUM_COUNTERS = 6
};
// Entries of a bucket array past its n: a light edge has a heavy sibling, so
// a path with d of them needs 2d + 1 sites, the rounds of n sites are at most
// (n + 1) / 2 and their buckets (two a round) at most n + 1.
enum { FL_BUCKET_PAD = 8 };
// Light children listed per chain position.  A position with more walks its
// row: 15 us on a wavefront that every path below it waits for, where a light
// edge takes 2.  A random triangulation has one with seven or more in ten thousand
// sites, one with nine or more in millions.
enum { FL_LIST = 8 };
// Chains are short below at most this length (a sweep's short-chain tile of
// 64 positions advances by 65 - long_min).
enum { FL_LONG_MAX = 33 };
enum { FL_CTRL_HEAD = 512 };  // bucket offsets mirrored into the control block
enum { FL_MAX_JUMP_ROUNDS = 96 };  // one "pointers moved" word per doubling round
enum { FL_CTRL_JUMPS = FL_NUM_FLAGS + FL_NUM_COUNTERS + 2 * (FL_CTRL_HEAD + 1) };
enum { FL_CTRL_WORDS = FL_CTRL_JUMPS + FL_MAX_JUMP_ROUNDS };

// Most sites of a terrain or a union of terrains: the pointer jumping keeps
// its counts (chain positions, light depths) below 2^31, the top bit of the
// count word marking a pair at its fixed point.
#define FL_MAX_SITES 0x7fffffffull

// Read-only inputs of one terrain, resident in HBM.
struct fl_dev_terrain {
  uint32_t n = 0;
  uint32_t nnz = 0;
  uint32_t* row_ptr = nullptr;   // [n+1]
  uint32_t* col = nullptr;       // [nnz]
  double* len = nullptr;         // [nnz]
  double* area = nullptr;        // [n]
  double* erod = nullptr;        // [n]
  double* uplift = nullptr;      // [n]
  double* tan_ms = nullptr;      // [n] tan(max_slope), NaN when None
  double* init_h = nullptr;      // [n]
  bool any_max_slope = false;
  uint8_t* is_outlet = nullptr;  // [n]
  uint32_t* rank = nullptr;      // [n] lake-traversal visit rank (UINT32_MAX: never)
  uint32_t* order = nullptr;     // [n] visited sites by rank
};

// Per-iteration state and scratch of one terrain.
struct fl_dev_work {
  double* h = nullptr;      // [n] elevations (current)
  double* h2 = nullptr;     // [n] elevations being computed
  double* xp = nullptr;     // [n] 1/celerity*distance, chain-major
  double* taup = nullptr;   // [n] response time, chain-major
  double* hnp = nullptr;    // [n] new elevation, chain-major (max-slope form)
  double* up = nullptr;     // [n] uplift, chain-major (max-slope form)
  double* tanp = nullptr;   // [n] tan(max slope), chain-major (max-slope form)
  uint32_t* pro = nullptr;  // [n] the basin outlet's position, chain-major (max-slope form)
  double* hop = nullptr;    // [n] old elevation, chain-major (max-slope form)
  double* A = nullptr;      // [n] drainage area (kept: heavy-child hint)
  double* tau = nullptr;    // [n] response time
  double* dnext = nullptr;  // [n] distance to the receiver
  uint32_t* next = nullptr; // [n]
  // lakes
  uint32_t* sub = nullptr;    // chain ends; from the decomposition on its workgroups' leaf counts
  uint64_t* lake_key = nullptr;
  // decomposition
  uint64_t* cmask = nullptr;  // [n] child slots of each site
  uint32_t* hc = nullptr;     // [n] heavy child
  // drainage-area inputs in chain-major order (written by k_chain_perm):
  // list counts, own area, erodibility, receiver distance; the listed light
  // children's drainage areas (FL_LIST slots per position, filled by the
  // children's rounds: pdest at a chain's base position names the slot of its
  // head, ppos there the position of its receiver)
  uint32_t* pcnt = nullptr;   // [n] npre | npost << 8, or the overflow flag; tail and head flags
  double* parea = nullptr;    // [n]
  double* pK = nullptr;       // [n]
  double* pdn = nullptr;      // [n]
  double* cval = nullptr;     // [FL_LIST n] hand-over words
  double* cover = nullptr;    // [n] hand-over words past the lists, at the children's bases, and between a chain's tiles
  uint32_t* pdest = nullptr;  // [n]
  uint32_t* ppos = nullptr;   // [n]
  uint32_t* spos = nullptr;   // [n] by site: its position, a leaf's receiver's

  // pointer jumping, two (pointer, count) pairs per site, pointer in the low
  // word: cp = (chain ancestor, distance to it), rt = (tree ancestor, light
  // edges to it); converged: (chain head, position), (root, light depth)
  uint64_t* cp = nullptr;
  uint64_t* rt = nullptr;
  uint32_t *bcnt = nullptr, *bnodes = nullptr, *boff = nullptr, *bnoff = nullptr, *bcur = nullptr,
           *bncur = nullptr;                                  // [n + FL_BUCKET_PAD] light-depth buckets
  uint32_t* ucum = nullptr;                                  // [n + FL_BUCKET_PAD] sweep units before each round
  uint2* cmeta = nullptr;                                    // [n] long chains' tiles: (base position, length or end)
  uint32_t* head_base = nullptr;                             // [n] at a chain head: its base position, at a leaf: none
  uint32_t* perm = nullptr;                                  // [n] chain-major site order
  uint32_t* ctrl = nullptr;                                  // [FL_CTRL_WORDS]
  // the kernels after the decomposition do nothing unless it is zero
  uint32_t* guard = nullptr;
  int* flags = nullptr;                                      // = ctrl
  uint32_t* counters = nullptr;                              // = ctrl + FL_NUM_FLAGS
  // chains of at least long_min sites (at most FL_LONG_MAX) take wavefronts of
  // their own, shorter ones share one (a tuning: results do not depend on it)
  uint32_t long_min = 16;
  // Basins recomputed in an iteration.  A new elevation is a function of the
  // drainage tree alone (and the static parameters), so a basin of the
  // previous iteration's tree in which no site's receiver changed -- nor any
  // receiver changed to or from one of its sites -- keeps its tree and its
  // elevations bit for bit; only the other basins' sites are active.
  const uint32_t* next_prev = nullptr;  // [n] the previous iteration's tree
  const double* dnext_prev = nullptr;   // [n]
  const uint32_t* root_prev = nullptr;  // [n] its basin (root) of every site
  uint32_t* root = nullptr;             // [n] this iteration's, for the next one
  uint8_t* dirty = nullptr;             // [n] by root: basin to recompute
  uint8_t* act = nullptr;               // [n] kind of a site recomputed in this iteration, 0: not
  // [n] the previous iteration changed the elevation of the site or of a
  // neighbour (zeroed by k_receivers, marked by k_tau_scatter)
  const uint8_t* chg_prev = nullptr;
  uint8_t* chg = nullptr;               // [n] ... this one
};

// Workgroup size of the per-site kernels launched by the calling thread (a
// tuning: results do not depend on it; 64..1024, a multiple of 64).
extern thread_local uint32_t fl_site_block;

// keep_unchanged: sites whose neighbourhood's elevations the previous
// iteration did not change keep its receivers (valid when that iteration's
// tree had no lake joins).
// mark: flag the previous basins that the changed receivers touch (w.dirty,
// cleared by the previous iteration's k_tau_scatter).
void fl_launch_receivers(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool keep_unchanged,
                         bool mark);
// Chain ends of the receivers into w.sub, the lakes' keys emptied.
void fl_launch_sub_labels(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w);
// Joins the lakes (after fl_launch_sub_labels); few: few sites lie in one.
void fl_launch_lake_join(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool few);
// Marks the dirty basins from the final receivers after a lake join (the
// receivers marked those of their own changes; k_tau_scatter clears the
// marks for the next iteration).
void fl_launch_dirty(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w);
// Children, heavy children and chain pointers of the iteration's active
// sites: every site of the terrains still iterating (`full`, or no previous
// tree), else those of the dirty basins (tid, t_active: per-site terrain and
// per-terrain mask of a union, or null).
void fl_launch_children(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool full, const uint32_t* tid,
                        const uint8_t* t_active);
void fl_launch_chain_jump(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t round);
// lakes: some root may be no outlet (a lake that no outlet reaches): its
// basin's sites are left out.
void fl_launch_chain_count(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool lakes);
// Bucket offsets (scan), chain placement and the chain-major permutation.
// scan: the placement makes the offsets itself; a decomposition of more than
// FL_SCAN_ROUNDS rounds raises the guard instead.
#ifndef FL_SCAN_ROUNDS
#define FL_SCAN_ROUNDS 64
#endif
void fl_launch_chain_layout(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool lakes, bool scan);
// The sweeps.  Rounds 0..min(deepest, cap - 1) in one launch of about `waves`
// wavefronts (any number is correct; the sweep units of the rounds are best);
// the drainage-area sweep also writes the response-time inputs.  positions:
// profiler units (0 when not known at launch).
enum { FL_FOLD_WAVES = 8 };
void fl_launch_da_fold(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t cap, uint32_t waves,
                       uint64_t positions, bool clamp);
void fl_launch_tau_fold(hipStream_t s, const fl_dev_work& w, uint32_t cap, uint32_t waves, uint64_t positions,
                        bool clamp);
// Rounds lsplit..deepest (deepest first, then shallowest first) in one
// workgroup of FL_TAIL_WAVES wavefronts, a barrier between rounds.
enum { FL_TAIL_WAVES = 16 };
void fl_launch_da_tail(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t lsplit,
                       uint64_t positions, bool clamp);
void fl_launch_tau_tail(hipStream_t s, const fl_dev_work& w, uint32_t lsplit, uint64_t positions, bool clamp);
// The drainage-area sweep's hand-over words before a first sweep, or after
// one whose waits ended without their values.
void fl_launch_reset_words(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w);
void fl_launch_clear_iter(hipStream_t s, const fl_dev_work& w, uint32_t nb);
// The work arrays of new terrains (basin roots, bucket entries, hand-over words).
void fl_launch_init_arrays(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t* const roots[3]);
// The control block to host_ctrl and, with tchanged, its G words to
// host_tchanged (pinned host memory); both zeroed on the device, FL_FLAG_DEEP
// apart.
void fl_launch_report(hipStream_t s, const fl_dev_work& w, uint32_t* host_ctrl, uint32_t G, uint32_t* tchanged,
                      uint32_t* host_tchanged);
// Back to site order, one thread per site.
void fl_launch_tau_scatter(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, bool clamp, bool lakes,
                           const uint32_t* tid, const uint8_t* active, uint32_t* tchanged);
void fl_launch_fill_u32(hipStream_t s, uint32_t* p, uint64_t count, uint32_t v);

// Gather of whole terrains of a union into a smaller union (in the same
// order, each keeping its internal layout): new terrain q takes the sites
// [new_off[q], new_off[q+1]) from old sites starting at old_off[q], and its
// entries from old entry old_eoff[q] to new entry new_eoff[q].
struct fl_compact_map {
  uint32_t count;
  const uint32_t* new_off;   // [count + 1]
  const uint32_t* old_off;   // [count]
  const uint32_t* new_eoff;  // [count]
  const uint32_t* old_eoff;  // [count]
};
// Copies the graph, parameters, visit ranks and order, current elevations
// and drainage areas (shifting site and entry indices) and writes new_tid,
// for the new sites [v0, v1): the terrains of the map, all from one source
// union, which become terrains tid0, tid0 + 1, ... of the new union.
void fl_launch_compact(hipStream_t s, const fl_compact_map& m, const fl_dev_terrain& ot, const fl_dev_work& ow,
                       const fl_dev_terrain& nt, const fl_dev_work& nw, uint32_t* new_tid, uint32_t v0, uint32_t v1,
                       uint32_t tid0);
// Verification: the reference's BFS traversal of the basin of `outlet`.
void fl_launch_basin_order(hipStream_t s, const fl_dev_terrain& t, const fl_dev_work& w, uint32_t outlet,
                           uint32_t* order, uint32_t* len_out);
