// ngpu_kernels.h -- kernels of one FCIQMC iteration on the GPU.
//
// Iteration chain (all on the engine stream, no host round trip):
//   k_prepass    per slot: initiator flag, proj-E sums, number of spawn
//                attempts, death (fused: spawning only needs the pre-death
//                sign bit and initiator bit, saved in pinfo); marks the slots
//                it frees; clears the walker hash when a rebuild is due
//   k_scan_apply exclusive scan of attempt counts -> attempt offsets; the
//                freed slots into the free queue; the hash refill of a rebuild
//   k_spawn      per attempt: parent from the scan's tile marks, excitation, H_ij,
//                stochastic rounding, spawn records staged in LDS and written
//                into the bins of their determinants' hashes; heat-bath
//                singles are queued for k_spawn_singles
//   k_merge_annihilate per bin: CompressSpawnedList / FindResidualParticle in
//                LDS, then hash lookup, add/abort/remove
//   k_insert     new dets: slot from the free queue, bucketed open-addressing insert
//   k_stats      per slot: occupied-threshold rounding, TotParts, norm, HF pop
//                (only with real coefficients or a core; whole-number runs sum
//                them in the prepass and the merge)
//   (k_end_iter in the engine: slot and hash bookkeeping, statistics sums)
#pragma once
#include "ngpu_device.h"
#include "../../include/neci_gpu.h"
#include <cstddef>

namespace ngpu {

constexpr int kBlock = 256;
constexpr int kWave = 64;

// statistics fields of ngpu_iter_out_t viewed as a double array
enum {
  F_NBORN = 0, F_NDIED, F_NANNIHIL, F_NABORTED, F_NREMOVED, F_TOTPARTS, F_NORMSQ, F_ENUM,
  F_HFCYC, F_NOATDOUBS, F_SPAWNSING, F_INSTHF, F_NOINITDETS, F_NOINITWALK, F_NONINITDETS,
  F_NONINITWALK, F_NFIELDS
};
constexpr int S_NVALID = F_NFIELDS * kMaxRep;
constexpr int S_NINVALID = S_NVALID + 1;
constexpr int S_MAXSPAWN = S_NVALID + 2;
constexpr int S_BLOOMC = S_NVALID + 3;
constexpr int S_BLOOMS = S_NVALID + 6;
constexpr int S_NDOUBLE = S_NVALID + 9;
__host__ __device__ constexpr int soff(int f, int r) { return f * kMaxRep + r; }
static_assert(sizeof(double) * S_NDOUBLE == offsetof(ngpu_iter_out_t, tot_walkers),
              "statistics block of ngpu_iter_out_t must be S_NDOUBLE doubles");
// block statistics beyond the output block: occupied determinants
constexpr int X_NOCC = S_NDOUBLE;
// Blocks flush their statistics into one of kStatCopies partial rows (chosen
// by block index), so that no address takes more than 1/kStatCopies of the
// device-scope atomics; the end-of-iteration kernel sums the rows.
constexpr int kStatStride = 288;  // doubles per row (2304 B, 9 lines of 256 B)
constexpr int kStatCopies = 32;
static_assert(X_NOCC < kStatStride, "statistics row too short");
__host__ __device__ constexpr bool stat_is_max(int i) {
  return i == S_MAXSPAWN || (i >= S_BLOOMS && i < S_BLOOMS + 3);
}

// Device counters.  Appends reserve ranges of the global lists once per LDS
// flush, never per lane or per wave: device-scope atomics on one address are
// serialised, so their count, not their payload, bounds the kernels that issue
// them.  The fields bumped in one kernel sit in separate 256-byte lines.
struct alignas(256) Counters {
  unsigned long long nslots;
  unsigned long long free_head;
  unsigned long long free_tail0;  // free_tail at the start of the iteration
  unsigned long long n_live, n_tomb, n_occ;
  unsigned long long n_attempts;
  unsigned long long n_fail;      // inserts refused (capacity errors)
  unsigned int ins_refused;       // k_insert placed no new determinant (MaxWalkers would be passed)
  unsigned long long free_tail_ins;  // free_tail as k_insert saw it
  unsigned long long rm_pre;         // slots the iteration's prepass freed
  unsigned int err;
  // the walker hash is rebuilt at the start of the next iteration (set by the
  // end-of-iteration accounting; the prepass clears the table, the attempt
  // scan refills it)
  unsigned int rebuild;
  unsigned int rebuilt;  // set by the attempt scan that refilled the table
  // sticky error: the error mask of the first iteration that reported one,
  // and that iteration's number.  While halt is set every kernel of the
  // iteration chain returns at once, so the walker list stays as the failing
  // iteration left it (the reference stops there, stop_all)
  unsigned int halt;
  unsigned int err_iter;
  unsigned long long n_rebuilds;  // walker-hash rebuilds since creation
  // the iteration's spawn bins (set by the attempt scan): their number, the
  // records each holds, and the log2 distance of their counters in words
  unsigned int nbins;
  unsigned int bin_cap;
  unsigned int bin_shift;
  // spawned records and attempts of the previous iteration (no attempts after
  // an upload or an explicit list): the expected number of records sizes the
  // bins (speed only, results do not depend on it); and its unique ones
  unsigned long long prev_spawned, prev_attempts, prev_unique;
  alignas(256) unsigned long long free_tail;
  alignas(256) unsigned long long n_spawned;
  alignas(256) unsigned long long n_singles;  // queued single-excitation attempts
  alignas(256) unsigned long long n_unique;
  alignas(256) unsigned long long n_new;
  alignas(256) unsigned long long n_ovf;      // spawned records past their bin's end
  // per-block counts of tombstone entries taken by inserts, spread over
  // kSpread lines (one add per block)
  struct alignas(256) Spread { unsigned long long v; };
  static constexpr int kSpread = 32;
  Spread reuse_part[kSpread];
  Spread uniq_part[kSpread];  // unique spawned determinants, per block
};

// probe limit of the walker hash: the load guard (k_hash_check) keeps probe
// sequences short, the cap turns a saturated table into an error, not a stall
constexpr int64_t kMaxProbe = 4096;

// Walker table.  The per-slot state that the random-access kernels update
// together -- the S signs, the flag word and the hash entry -- is one row of
// S+1 doubles (signs, then flags in the low and the hash entry in the high
// 32 bits of the last word), so that a lookup-and-update touches one line.
struct Walk {
  uint64_t* keys;     // cap * W
  double* st;         // cap * srow: S signs | flags, hash entry (bucket*4 + e)
  int64_t srow;       // S + 1
  double* diagH;      // H_ii - Hii
  double* offdiagH;   // H(det, ref)
  int64_t cap;
  uint64_t* htab;     // L buckets of 8W words
  int64_t L;
  int64_t* freeq;     // free-slot queue (ring, cap entries)
  __device__ double& sgn(int64_t slot, int r) const { return st[slot * srow + r]; }
  __device__ uint32_t& flags(int64_t slot) const { return *(uint32_t*)(st + slot * srow + srow - 1); }
  __device__ int32_t& hpos(int64_t slot) const { return *((int32_t*)(st + slot * srow + srow - 1) + 1); }
};

struct Shift { double v[kMaxRep]; };
// per-iteration inputs (time step, shifts, iteration number), read by the
// kernels from device memory so that a captured iteration replays unchanged
struct IterParams {
  double tau;
  Shift sft;
  uint32_t iter;
  uint32_t pad;
};

// The blocks a kernel body runs on: this block's index and the number of
// blocks of its launch share.  A plain launch gives the hardware grid; a
// batch launch (one launch covering several engines) gives each engine's
// share of the blocks, so a body sees the same index space either way.
struct Grid {
  int64_t b, nb;
};
__device__ inline Grid hw_grid() { return Grid{(int64_t)blockIdx.x, (int64_t)gridDim.x}; }

// ----------------------------------------------------------- wave utils
__device__ inline int lane_id() { return __lane_id(); }

__device__ inline uint64_t lanemask_lt() {
  int l = lane_id();
  return l == 0 ? 0ull : (~0ull >> (64 - l));
}

// A lane's value moved by DPP (row_shr within rows of 16, then the rows'
// last lanes to the rows after them); lanes without a source get 0.  A wave
// reduction by these is VALU code of a few dozen cycles; by ds_bpermute
// shuffles it is six LDS round trips (0.3 us), which the 7 to 13 statistics
// of a kernel made 2 to 4 us of each launch.
template <int CTRL, int ROWS>
__device__ inline uint32_t dpp_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, CTRL < 0x140);
}
template <int CTRL, int ROWS>
__device__ inline uint64_t dpp_u64(uint64_t v) {
  return ((uint64_t)dpp_u32<CTRL, ROWS>((uint32_t)(v >> 32)) << 32) | dpp_u32<CTRL, ROWS>((uint32_t)v);
}
template <int CTRL, int ROWS>
__device__ inline double dpp_f64(double v) {
  return __longlong_as_double((long long)dpp_u64<CTRL, ROWS>((uint64_t)__double_as_longlong(v)));
}
constexpr int kRowShr = 0x110, kRowMirror = 0x140, kRowHalfMirror = 0x141, kRowBcast15 = 0x142, kRowBcast31 = 0x143,
              kRowNewbcast = 0x150;
// a value of one lane (wave-uniform index), to every lane
__device__ inline uint32_t lane_value(uint32_t v, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, l); }
__device__ inline uint64_t lane_value(uint64_t v, int l) {
  return ((uint64_t)lane_value((uint32_t)(v >> 32), l) << 32) | lane_value((uint32_t)v, l);
}
// inclusive sums over the lanes (every lane of the wave active)
__device__ inline int64_t wave_scan(int64_t x) {
  uint64_t v = (uint64_t)x;
  v += dpp_u64<kRowShr + 1, 0xF>(v);
  v += dpp_u64<kRowShr + 2, 0xF>(v);
  v += dpp_u64<kRowShr + 4, 0xF>(v);
  v += dpp_u64<kRowShr + 8, 0xF>(v);
  v += dpp_u64<kRowBcast15, 0xA>(v);
  v += dpp_u64<kRowBcast31, 0xC>(v);
  return (int64_t)v;
}
// sum over the wave, to every lane
__device__ inline double wave_sum(double v) {
  v += dpp_f64<kRowShr + 1, 0xF>(v);
  v += dpp_f64<kRowShr + 2, 0xF>(v);
  v += dpp_f64<kRowShr + 4, 0xF>(v);
  v += dpp_f64<kRowShr + 8, 0xF>(v);
  v += dpp_f64<kRowBcast15, 0xA>(v);
  v += dpp_f64<kRowBcast31, 0xC>(v);
  return __longlong_as_double((long long)lane_value((uint64_t)__double_as_longlong(v), kWave - 1));
}
// maximum over the wave of values >= 0, to every lane
__device__ inline double wave_max(double v) {
  auto up = [&](double w) { v = w > v ? w : v; };
  up(dpp_f64<kRowShr + 1, 0xF>(v));
  up(dpp_f64<kRowShr + 2, 0xF>(v));
  up(dpp_f64<kRowShr + 4, 0xF>(v));
  up(dpp_f64<kRowShr + 8, 0xF>(v));
  up(dpp_f64<kRowBcast15, 0xA>(v));
  up(dpp_f64<kRowBcast31, 0xC>(v));
  return __longlong_as_double((long long)lane_value((uint64_t)__double_as_longlong(v), kWave - 1));
}
__device__ inline unsigned long long wave_count(bool p) { return (unsigned long long)popc64(__ballot(p)); }

__device__ inline unsigned long long wave_reserve(unsigned long long* ctr, int n) {
  unsigned long long b = 0;
  if (lane_id() == 0) b = atomicAdd(ctr, (unsigned long long)n);
  return lane_value((uint64_t)b, 0);
}
// orders one wave's LDS accesses of different lanes: a wave's LDS operations
// run in order, so only the compiler has to keep them so.  (A workgroup fence
// would wait for every global access in flight, prefetches and stores too.)
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Block-local statistics in LDS.  Every add/max is a wave-wide call (all 64
// lanes, inactive lanes passing 0): the wave reduces with shuffles and one lane
// updates LDS, so no LDS address is contended by more than one lane per wave.
struct BlockStats {
  double* acc;  // LDS, kStatStride entries
  __device__ void zero() {
    for (int i = threadIdx.x; i < kStatStride; i += blockDim.x) acc[i] = 0.0;
    __syncthreads();
  }
  __device__ void add(int i, double v) {
    double t = wave_sum(v);
    if (lane_id() == 0 && t != 0.0) atomicAdd(&acc[i], t);
  }
  __device__ void max(int i, double v) {  // v >= 0
    double t = wave_max(v);
    if (lane_id() == 0 && t > 0.0)
      atomicMax((unsigned long long*)&acc[i], (unsigned long long)__double_as_longlong(t));
  }
  // into partial row blockIdx % kStatCopies (InstNoAtHF has a single writer, or
  // one writer and the changes after it, so summing the rows reproduces it)
  __device__ void flush(double* part, int64_t blk) {
    __syncthreads();
    double* g = part + (size_t)(blk % kStatCopies) * kStatStride;
    for (int i = threadIdx.x; i < kStatStride; i += blockDim.x) {
      double v = acc[i];
      if (v == 0.0) continue;
      if (stat_is_max(i))
        atomicMax((unsigned long long*)&g[i], (unsigned long long)__double_as_longlong(v));
      else
        atomicAdd(&g[i], v);
    }
  }
};

// ------------------------------------------------------ LDS-staged appends
// A block stages the records it appends to a global list in LDS and reserves
// space in the list once per flush (one device-scope atomic for up to CAP
// records).  push() is wave-wide; flush_begin()/flush_end() are block-wide and
// must be reached by every thread of the block in every trip.
struct Stage {
  uint32_t n;                 // staged records
  unsigned long long base;    // reserved position of the flush in progress
};

// index in the LDS stage for lanes with pred (-1 otherwise)
__device__ inline int stage_push(bool pred, Stage* st) {
  uint64_t m = __ballot(pred);
  if (m == 0) return -1;
  int leader = __ffsll((unsigned long long)m) - 1;
  uint32_t b = 0;
  if (lane_id() == leader) b = atomicAdd(&st->n, (uint32_t)popc64(m));
  b = lane_value(b, leader);
  return pred ? (int)(b + (uint32_t)popc64(m & lanemask_lt())) : -1;
}

// true when the block must flush now (force, or fewer than blockDim free
// entries left); then cnt = staged records and base = their reserved position
__device__ inline bool stage_flush_begin(Stage* st, unsigned long long* gctr, int cap, bool force,
                                         uint32_t& cnt, unsigned long long& base) {
  __syncthreads();
  cnt = st->n;
  __syncthreads();  // every thread has read n before the next trip pushes again
  if (cnt == 0 || (!force && cnt + blockDim.x <= (uint32_t)cap)) return false;
  if (threadIdx.x == 0) st->base = atomicAdd(gctr, (unsigned long long)cnt);
  __syncthreads();
  base = st->base;
  return true;
}
__device__ inline void stage_flush_end(Stage* st) {
  __syncthreads();
  if (threadIdx.x == 0) st->n = 0;
  __syncthreads();
}
__device__ inline void stage_init(Stage* st) {
  if (threadIdx.x == 0) st->n = 0;
  __syncthreads();
}

// pinfo bit of a slot the prepass freed (first replica's byte)
constexpr uint8_t kPinfoFreed = 8;

// Freed slots staged for the free queue (a ring of cap entries).
constexpr int kFreeStage = 512;
struct FreeStage {
  Stage st;
  int64_t slot[kFreeStage];
};

// RemoveHashDet (load_balancer.fpp:631-644) for the lanes with rm set: the
// hash entry becomes a tombstone, the slot is staged for the free queue.
// Wave-wide call; the live and tombstone counts follow from the free-queue
// tail.  (Releasing the entry as empty where the
// bucket already holds an empty entry would also be valid -- such a bucket
// ends every probe -- but it makes each removal read its bucket and, measured,
// cost more in the removing kernels than the rebuilds it saves.)  The prepass
// removes without this helper: it marks the slot, the attempt scan queues it.
template <int W>
__device__ inline void remove_dets(const Walk& wk, FreeStage* fs, bool rm, int64_t slot) {
  int q = stage_push(rm, &fs->st);
  if (rm) {
    int64_t hp = wk.hpos(slot);
    int32_t* sl = (int32_t*)(wk.htab + (size_t)(hp >> 2) * 8 * W + 4 * W);
    sl[hp & 3] = kSlotTomb;
    wk.flags(slot) |= kFlagRemoved;
    fs->slot[q] = slot;
  }
}
// block-wide: drain the staged slots into the free queue when due
__device__ inline void free_flush(const Walk& wk, Counters* cnt, FreeStage* fs, bool force) {
  uint32_t n;
  unsigned long long base;
  if (!stage_flush_begin(&fs->st, &cnt->free_tail, kFreeStage, force, n, base)) return;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x)
    wk.freeq[(base + i) % (unsigned long long)wk.cap] = fs->slot[i];
  stage_flush_end(&fs->st);
}


// hash lookup: returns slot or -1.  Entries of a bucket fill in order and
// become empty only when the table is rebuilt, so the first empty entry ends
// the probe sequence.  A bucket's slots and keys are loaded together (16-byte
// loads of one line) and compared in registers: one round trip per bucket.
template <int W>
__device__ inline int64_t hash_lookup(const Walk& wk, const uint64_t* key, int64_t home, Counters* cnt) {
  int64_t b = home;
  int64_t maxp = wk.L < kMaxProbe ? wk.L : kMaxProbe;
  for (int64_t probe = 0; probe < maxp; ++probe) {
    const uint64_t* bk = wk.htab + (size_t)b * 8 * W;
    const int4 sl = *(const int4*)(bk + 4 * W);
    ulonglong2 k[2 * W];
#pragma unroll
    for (int q = 0; q < 2 * W; ++q) k[q] = ((const ulonglong2*)bk)[q];
    const int32_t slot[kBucketEntries] = {sl.x, sl.y, sl.z, sl.w};
#pragma unroll
    for (int e = 0; e < kBucketEntries; ++e) {
      const int32_t s = slot[e];
      if (s == kSlotEmpty) return -1;
      bool eq;
      if constexpr (W == 1) eq = ((e & 1) ? k[e / 2].y : k[e / 2].x) == key[0];
      else eq = k[e].x == key[0] && k[e].y == key[1];
      if (s >= 0 && eq) return s;
    }
    b = (b + 1 == wk.L) ? 0 : b + 1;
  }
  if (maxp < wk.L) atomicOr(&cnt->err, 1u << NGPU_ERR_HASH_FULL);
  return -1;
}

// bucketed open-addressing insert of an absent key; returns hash position or
// -1; reused is set when the entry claimed was a tombstone
template <int W>
__device__ inline int64_t hash_insert(const Walk& wk, const uint64_t* key, int64_t home, int32_t slot,
                                      bool& reused) {
  int64_t b = home;
  int64_t maxp = wk.L < kMaxProbe ? wk.L : kMaxProbe;
  for (int64_t probe = 0; probe < maxp; ++probe) {
    uint64_t* bk = wk.htab + (size_t)b * 8 * W;
    int32_t* sl = (int32_t*)(bk + 4 * W);
#pragma unroll
    for (int e = 0; e < kBucketEntries; ++e) {
      int32_t cur = sl[e];
      while (cur == kSlotEmpty || cur == kSlotTomb) {
        int32_t prev = atomicCAS(&sl[e], cur, slot);
        if (prev == cur) {
          reused = cur == kSlotTomb;
#pragma unroll
          for (int w = 0; w < W; ++w) bk[e * W + w] = key[w];
          return b * 4 + e;
        }
        cur = prev;
      }
    }
    b = (b + 1 == wk.L) ? 0 : b + 1;
  }
  return -1;
}

// rebuild of the walker hash in two grid-wide phases (a kernel boundary
// between them): every entry emptied, then every live slot reinserted
template <int W>
__device__ inline void hash_clear_part(const Grid& g, const Walk& wk) {
  for (int64_t b = g.b * blockDim.x + threadIdx.x; b < wk.L; b += g.nb * blockDim.x) {
    int32_t* sl = (int32_t*)(wk.htab + (size_t)b * 8 * W + 4 * W);
#pragma unroll
    for (int e = 0; e < kBucketEntries; ++e) sl[e] = kSlotEmpty;
  }
}
template <int W>
__device__ inline void hash_refill_part(const Grid& g, const DevSys& s, const Walk& wk, Counters* cnt,
                                        int64_t nslots) {
  for (int64_t slot = g.b * blockDim.x + threadIdx.x; slot < nslots; slot += g.nb * blockDim.x) {
    if (wk.flags(slot) & kFlagRemoved) continue;
    uint64_t key[W];
#pragma unroll
    for (int w = 0; w < W; ++w) key[w] = wk.keys[slot * W + w];
    int64_t home = find_walker_hash<W>(key, s.rh, s.L) - 1;
    bool reused = false;
    int64_t hp = hash_insert<W>(wk, key, home, (int32_t)slot, reused);
    if (hp < 0) atomicOr(&cnt->err, 1u << NGPU_ERR_HASH_FULL);
    else wk.hpos(slot) = hp;
  }
}

// ----------------------------------------------------------- spawn bins
// The spawning kernels write each record straight into one of nbins bins,
// chosen by a hash of its determinant, so equal determinants meet in one bin
// and one wave merges a bin in LDS: no sort and no gather stands between
// spawning and annihilation.  A record takes its place with one atomic on its
// bin's counter; the counters are spread over as many cache lines as their
// array has (an address, and so a line, takes one atomic in about 12 ns, and
// scattered ones run at 25 G/s).  A bin that is full (one determinant spawned
// very often, or a spawned list near its capacity) sends its further records
// to the overflow list, which holds the spawn capacity; they hang in
// kBinChains chains of the bin, by their place in it, and the bin's wave
// follows one chain a lane.  So a bin's records cost time in proportion to
// their number wherever they are.  (Areas that the waves of all bins
// that spilled searched for their own records took a time quadratic in the
// list: 5.0e6 spawns on 6.2e4 determinants filling the list merged in 101 ms,
// where the sort had taken 12.)  Order within a bin is the
// order of arrival (of an explicit list, the list's): the merge's sums do not
// depend on it beyond FP64 rounding.
constexpr uint32_t kBinChains = 64;
struct Bins {
  uint64_t* rec;     // cap records, bin_cap to each bin
  uint64_t* ovf;     // overflow list (the spawn capacity)
  uint32_t* next;    // of an overflow record, the one behind it in its chain
  uint32_t* head;    // kBinChains per bin; never emptied, as chains are followed by length
  uint32_t* count;   // records of bin b at [b << bin_shift], emptied by the merge
  int64_t cap;
  int64_t ovf_cap;   // the spawn capacity
  uint32_t maxb;     // most bins
  uint32_t words;    // length of count
};
// records per bin aimed at: a wave merges up to 64 in one pass over its lanes
constexpr int kBinFill = 44;
// The least number of spawns expected is attempts / kMinRate.  A bin's merge
// takes (its determinants / 128) rounds over its records, so without a bound
// on a bin's records one iteration's time grows with the square of the list;
// with this one a bin holds kBinFill * kMinRate records at most when every
// attempt spawns, 22 rounds.  Empty bins cost a 64th of a load each.
constexpr int kMinRate = 64;

// the number of bins for a list of the expected length and number of
// determinants, the records each holds and the log2 distance of their counters
struct BinPlan {
  uint32_t nbins, cap, shift;
};
// What a bin's load differs from the mean by is whole determinants with all
// their records: a share 1 / sqrt(l) of it for l determinants a bin.  A list of
// many records per determinant close to the capacity takes fewer bins, up to
// kBinFill determinants in each, so that five such shares fit what is left of
// the room (taken as 1.5 times the capacity: a bin has 1.25 times its share and
// overflows a little for nothing).  Otherwise most of its records would take
// the chains: 5.1e6 spawns on 6.0e4 uneven determinants, the list full, merge
// in 0.40 ms with bins by records alone and in 0.30 ms with these.
__host__ __device__ inline BinPlan bin_plan(const Bins& b, double expect, double dets) {
  double nb = expect * (1.0 / kBinFill) + 1.0;
  const double spare = 1.5 * (double)b.ovf_cap - expect;  // (room / list - 1) list
  const double l = spare > 0.0 && 25.0 * expect * expect < kBinFill * spare * spare
                       ? 25.0 * expect * expect / (spare * spare) : (double)kBinFill;
  if (nb * l > dets + l) nb = dets / l + 1.0;
  const uint32_t n = nb < (double)b.maxb ? (uint32_t)nb : b.maxb;
  uint32_t sh = 0;
  while (sh < 5 && ((uint64_t)n << (sh + 1)) <= b.words) ++sh;
  const int64_t c = b.cap / n;
  return BinPlan{n, (uint32_t)(c < 0x7FFFFFFF ? c : 0x7FFFFFFF), sh};
}
__host__ __device__ inline void set_bins(Counters* cnt, const Bins& b, double expect, double dets) {
  const BinPlan p = bin_plan(b, expect, dets);
  cnt->nbins = p.nbins;
  cnt->bin_cap = p.cap;
  cnt->bin_shift = p.shift;
}

// hash of a determinant: the high word picks the bin, its fraction inside the
// bin the first slot of the merge's table
template <int W>
__host__ __device__ inline uint32_t bin_hash(const uint64_t* d) {
  uint64_t h = d[0] * 0x9E3779B97F4A7C15ull;
  if constexpr (W == 2) {
    h += (d[1] ^ (d[1] >> 29)) * 0xBF58476D1CE4E5B9ull;
    h = (h ^ (h >> 31)) * 0x94D049BB133111EBull;
  }
  return (uint32_t)(h >> 32);
}
__host__ __device__ inline uint32_t bin_of(uint32_t h, uint32_t nb) { return (uint32_t)(((uint64_t)h * nb) >> 32); }

// overflow record o, the k-th past the end of bin b, into its chain; its place
// (null: the overflow list is full, which takes more records than the spawn
// capacity; the merge takes nothing from such a list and the iteration's end
// reports it)
__device__ inline uint64_t* bin_overflow(const Bins& bins, uint32_t b, uint32_t k, unsigned long long o,
                                         int rec_words) {
  if (o >= (unsigned long long)bins.ovf_cap) return nullptr;
  bins.next[o] = atomicExch(&bins.head[(size_t)b * kBinChains + k % kBinChains], (uint32_t)o);
  return bins.ovf + (size_t)o * rec_words;
}

// this block's slots: whole waves, so that a small table does not
// spread over more blocks than it fills (each pays its set-up and its
// statistics' atomics) and every block starts on a line
__device__ inline void chunk_of(const Grid& g, int64_t n, int64_t& begin, int64_t& end) {
  int64_t chunk = ((n + g.nb - 1) / g.nb + kWave - 1) / kWave * kWave;
  begin = g.b * chunk;
  end = begin + chunk;
  if (end > n) end = n;
  if (begin > n) begin = n;
}

// Per-lane statistic accumulator of one field: registers when the kernel is
// built for one or two replicas (the replica of a call is then known at
// compile time), the block's LDS row otherwise.  add() and done() are
// wave-wide calls.
template <int R>
struct LaneSum {
  double v[R <= 2 ? R : 1] = {0.0};
  __device__ void add(BlockStats& bs, int i, double x) {
    if constexpr (R == 1) v[0] += x;
    else if constexpr (R == 2) v[i & (kMaxRep - 1)] += x;
    else bs.add(i, x);
  }
  __device__ void done(BlockStats& bs, int i) {
    if constexpr (R <= 2)
#pragma unroll
      for (int r = 0; r < R; ++r) bs.add(i + r, v[r]);
  }
};
struct LaneMax {
  double v = 0.0;
  __device__ void add(double x) { v = x > v ? x : v; }
  __device__ void done(BlockStats& bs, int i) { bs.max(i, v); }
};

// block exclusive scan of one int64 per thread (blockDim = kBlock)
__device__ inline int64_t block_exclusive_scan(int64_t v, int64_t* lds, int64_t& total) {
  const int lane = lane_id(), wv = threadIdx.x / kWave;
  const int64_t x = wave_scan(v);
  if (lane == kWave - 1) lds[wv] = x;
  __syncthreads();
  int64_t pre = 0, tot = 0;
#pragma unroll
  for (int q = 0; q < kBlock / kWave; ++q) {
    const int64_t n = lds[q];
    if (q < wv) pre += n;
    tot += n;
  }
  __syncthreads();
  total = tot;
  return pre + x - v;
}

// trips of a grid-stride loop that every lane of the grid runs (keeps wave-wide
// calls convergent); the element of this lane in trip t is t*stride + gid
__device__ inline int64_t grid_trips(const Grid& g, int64_t n) {
  int64_t stride = g.nb * blockDim.x;
  return (n + stride - 1) / stride;
}
__device__ inline int64_t grid_elem(const Grid& g, int64_t t) {
  return t * g.nb * blockDim.x + g.b * blockDim.x + threadIdx.x;
}

// ------------------------------------------------- incremental statistics
// CalcHashTableStats's sums (TotParts, norm, occupied determinants, InstNoAtHF)
// need a pass over the walker table only when that pass also rounds (real
// coefficients) or when core amplitudes change outside the merge.  With
// integer walkers the prepass sums what it leaves behind and the merge adds
// what it changes, exactly (sums of integers), so k_stats is not launched:
// 6 us of an iteration over 3e3 determinants, 25 us over 2.9e6.
__host__ __device__ inline bool stats_by_parts(const DevSys& s) { return !s.t_real && s.ncore == 0; }
// The merge counts a new determinant before k_insert has placed it: what the
// insertion refused (the iteration ends in an error) is taken out again by the
// iteration's end, so that the statistics are those of the kept walker list.
// The new list as the end of an iteration sees it, in device memory: only an
// iteration that refused something reads it, and a longer argument block cost
// every one 0.5 us.
struct NewList {
  const uint64_t* key;
  const double* sgn;
  const uint32_t* flag;
  uint64_t ref0, ref1;
  int W;
};
__device__ inline void uncount_refused(const NewList& nl, const Counters* cnt, double* part, int S) {
  const int64_t nn = (int64_t)cnt->n_new;
  const bool all = cnt->ins_refused != 0;
  for (int64_t i = threadIdx.x; i < nn; i += blockDim.x) {
    if (!all && !(nl.flag[i] & kFlagRemoved)) continue;
    const bool isref = nl.key[i * nl.W] == nl.ref0 && (nl.W == 1 || nl.key[i * nl.W + 1] == nl.ref1);
    atomicAdd(&part[X_NOCC], -1.0);
    for (int r = 0; r < S; ++r) {
      const double v = nl.sgn[i * S + r];
      atomicAdd(&part[soff(F_TOTPARTS, r)], -fabs(v));
      atomicAdd(&part[soff(F_NORMSQ, r)], -(v * v));
      if (isref) atomicAdd(&part[soff(F_INSTHF, r)], -v);
    }
  }
  __syncthreads();
}

// ------------------------------------------------------------- prepass
// CalcParentFlag_det + SumEContrib + decide_num_to_spawn + walker_death for
// every occupied slot (FciMCPar.F90:1294-1758, fcimc_helper.F90:518-802,
// 1036-1321, 2160-2407).  Blocks own contiguous slot ranges so that the block
// sums of attempt counts feed the scan directly.
template <int W, int R>
__device__ __forceinline__ void k_prepass_body(const Grid& g_, const DevSys& s, const Walk& wk, Counters* cnt, double* part, int32_t* att_cnt, uint8_t* pinfo, int64_t* blk_part, int64_t* blk_rm, IterParams* prm, const IterParams& v, int use_v) {
  if (cnt->halt) return;
  // the iteration's inputs: from the launch when launches are issued one by
  // one (block 0 publishes them for the later kernels), from device memory
  // in a replayed graph
  const double tau = use_v ? v.tau : prm->tau;
  const uint32_t iter = use_v ? v.iter : prm->iter;
  if (use_v && g_.b == 0 && threadIdx.x == 0) *prm = v;
  __shared__ double acc_lds[kStatStride];
  __shared__ int64_t red[2 * kBlock / kWave];
  const int S = R <= 2 ? R : s.S;
  int64_t nslots = (int64_t)cnt->nslots;
  const bool rebuild = cnt->rebuild != 0;
  if (rebuild) hash_clear_part<W>(g_, wk);  // the attempt scan refills the table
  int64_t begin, end;
  chunk_of(g_, nslots, begin, end);
  if (begin >= end) {  // no slots for this block
    if (threadIdx.x == 0) blk_part[g_.b] = blk_rm[g_.b] = 0;
    return;
  }
  BlockStats bs{acc_lds};
  bs.zero();
  int64_t my_att = 0, my_rm = 0;
  bool death_err = false;
  LaneSum<R> a_idets, a_iwalk, a_ndets, a_nwalk, a_hf, a_doubs, a_enum, a_died, a_born, a_abort, a_tot, a_norm;
  LaneSum<1> a_occ;
  const bool by_parts = stats_by_parts(s);
  for (int64_t base = begin; base < end; base += blockDim.x) {
    int64_t slot = base + threadIdx.x;
    bool valid = slot < end;
    // every field of the slot is loaded at once (lanes past the chunk load
    // the step's first slot) and selected afterwards, so that the loads are
    // one round trip to memory rather than three dependent ones
    const int64_t ls = valid ? slot : base;
    const uint32_t f_ld = wk.flags(ls);
    uint64_t k_ld[W];
    double s_ld[R];
#pragma unroll
    for (int w = 0; w < W; ++w) k_ld[w] = wk.keys[ls * W + w];
    for (int r = 0; r < S; ++r) s_ld[r] = wk.sgn(ls, r);
    const double hoff_ld = wk.offdiagH[ls], kii_ld = wk.diagH[ls];
    uint32_t f = valid ? f_ld : kFlagRemoved;
    bool live = !(f & kFlagRemoved);
    uint64_t key[W];
    double sg[R];
    bool occ = false;
#pragma unroll
    for (int w = 0; w < W; ++w) key[w] = live ? k_ld[w] : 0ull;
    for (int r = 0; r < S; ++r) {
      sg[r] = live ? s_ld[r] : 0.0;
      occ = occ || !(fabs(sg[r]) < 1.e-12);
    }
    bool core = (f & kFlagCore) != 0;
    uint8_t pi0 = 0;
    int exlevel = occ ? excit_level<W>(s.ref, key) : -1;
    double hoff = occ ? hoff_ld : 0.0;
    double kii = occ ? kii_ld : 0.0;
    bool isref = occ && det_eq<W>(key, s.ref);
    bool any_left = false;
    double cp[R];
    for (int r = 0; r < S; ++r) {
      // initiator flag (CalcParentFlag_det / TestInitiator_explicit)
      bool now = false;
      if (occ && s.t_init) {
        bool was = (f >> r) & 1u;
        bool pop = fabs(sg[r]) > s.init_walk_no;
        now = was ? (pop || isref || core) : pop;
        f = now ? (f | (1u << r)) : (f & ~(1u << r));
      }
      if (s.t_init) {
        bool ini = occ && now, non = occ && !now;
        a_idets.add(bs, soff(F_NOINITDETS, r), ini ? 1.0 : 0.0);
        a_iwalk.add(bs, soff(F_NOINITWALK, r), ini ? fabs(sg[r]) : 0.0);
        a_ndets.add(bs, soff(F_NONINITDETS, r), non ? 1.0 : 0.0);
        a_nwalk.add(bs, soff(F_NONINITWALK, r), non ? fabs(sg[r]) : 0.0);
      }
      // SumEContrib
      a_hf.add(bs, soff(F_HFCYC, r), exlevel == 0 ? sg[r] : 0.0);
      a_doubs.add(bs, soff(F_NOATDOUBS, r), exlevel == 2 ? fabs(sg[r]) : 0.0);
      a_enum.add(bs, soff(F_ENUM, r), occ ? hoff * sg[r] : 0.0);
      // decide_num_to_spawn and attempt_die share one Philox block
      double died = 0.0, born = 0.0;
      cp[r] = sg[r];
      if (occ) {
        double ua, ub;
        draw2<W>(s.seed, key, iter, r, 0, 0, ua, ub);
        double pa = sg[r] * s.avmc;
        int64_t nsp = (int64_t)pa;
        if (nsp < 0) nsp = -nsp;
        if (fabs(fabs(pa) - (double)nsp) > 1.e-12) {
          double extra = fabs(pa) - (double)nsp;
          if (extra > ua) nsp++;
        }
        att_cnt[slot * S + r] = (int32_t)nsp;
        my_att += nsp;
        uint8_t pi = (uint8_t)((sg[r] < 0.0 ? 1 : 0) | (((f >> r) & 1u) ? 2 : 0) | (core ? 4 : 0));
        if (r == 0) pi0 = pi;  // written with the removal bit below
        else pinfo[slot * S + r] = pi;
        double fac = tau * (kii - (use_v ? v.sft.v[r] : prm->sft.v[r]));
        if (fac > 2.0) death_err = true;
        double idie = core ? 0.0 : attempt_die(s.t_real != 0, fac, fabs(sg[r]), ub);
        double a = fabs(sg[r]);
        died = idie < a ? idie : a;
        double bb = idie - a;
        born = bb > 0.0 ? bb : 0.0;
        cp[r] = sg[r] - idie * (sg[r] >= 0.0 ? 1.0 : -1.0);
        any_left = any_left || (fabs(cp[r]) > 1.0e-12);
      } else if (valid) {
        att_cnt[slot * S + r] = 0;
      }
      a_died.add(bs, soff(F_NDIED, r), died);
      a_born.add(bs, soff(F_NBORN, r), born);
    }
    bool abort_anti = occ && s.t_init && any_left;
    if (abort_anti) any_left = false;
    for (int r = 0; r < S; ++r) {
      double ab = 0.0;
      if (abort_anti) {
        if ((cp[r] > 0.0) != (sg[r] > 0.0)) {
          ab = fabs(cp[r]);
          cp[r] = 0.0;
        }
        any_left = any_left || (fabs(cp[r]) > 1.0e-12);
      }
      a_abort.add(bs, soff(F_NABORTED, r), ab);
    }
    bool rm = occ && !(any_left || core);
    if (by_parts) {  // what is left of the slot
      bool left = live && core;
      for (int r = 0; r < S; ++r) left = left || (!rm && !(fabs(cp[r]) < 1.e-12));
      for (int r = 0; r < S; ++r) {
        const double v = left ? cp[r] : 0.0;
        a_tot.add(bs, soff(F_TOTPARTS, r), fabs(v));
        a_norm.add(bs, soff(F_NORMSQ, r), v * v);
        if (isref && left) bs.acc[soff(F_INSTHF, r)] = v;
      }
      a_occ.add(bs, X_NOCC, left ? 1.0 : 0.0);
    }
    if (occ) {
      for (int r = 0; r < S; ++r) wk.sgn(slot, r) = rm ? 0.0 : cp[r];
      wk.flags(slot) = rm ? (f | kFlagRemoved) : f;
      if (rm && !rebuild) {  // RemoveHashDet: the entry becomes a tombstone
        int64_t hp = wk.hpos(slot);
        int32_t* sl = (int32_t*)(wk.htab + (size_t)(hp >> 2) * 8 * W + 4 * W);
        sl[hp & 3] = kSlotTomb;
      }
    }
    // bit 3 of the first replica's byte: freed here; the attempt scan queues
    // these slots in the free list (in slot order, no atomics here)
    if (valid) pinfo[slot * S] = (uint8_t)(pi0 | (rm ? kPinfoFreed : 0));
    my_rm += rm ? 1 : 0;
  }
  if (death_err) atomicOr(&cnt->err, 1u << NGPU_ERR_DEATH_PROB);
  a_idets.done(bs, soff(F_NOINITDETS, 0));
  a_iwalk.done(bs, soff(F_NOINITWALK, 0));
  a_ndets.done(bs, soff(F_NONINITDETS, 0));
  a_nwalk.done(bs, soff(F_NONINITWALK, 0));
  a_hf.done(bs, soff(F_HFCYC, 0));
  a_doubs.done(bs, soff(F_NOATDOUBS, 0));
  a_enum.done(bs, soff(F_ENUM, 0));
  a_died.done(bs, soff(F_NDIED, 0));
  a_born.done(bs, soff(F_NBORN, 0));
  a_abort.done(bs, soff(F_NABORTED, 0));
  if (by_parts) {
    a_tot.done(bs, soff(F_TOTPARTS, 0));
    a_norm.done(bs, soff(F_NORMSQ, 0));
    a_occ.done(bs, X_NOCC);
  }
  my_att = wave_scan(my_att);
  my_rm = wave_scan(my_rm);
  if (lane_id() == kWave - 1) {
    red[2 * (threadIdx.x / kWave)] = my_att;
    red[2 * (threadIdx.x / kWave) + 1] = my_rm;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t a = 0, f = 0;
    for (int q = 0; q < kBlock / kWave; ++q) {
      a += red[2 * q];
      f += red[2 * q + 1];
    }
    blk_part[g_.b] = a;
    blk_rm[g_.b] = f;
  }
  bs.flush(part, g_.b);
}
template <int W, int R>
__global__ void __launch_bounds__(kBlock) k_prepass(DevSys s, Walk wk, Counters* cnt, double* part, int32_t* att_cnt, uint8_t* pinfo, int64_t* blk_part, int64_t* blk_rm, IterParams* prm, IterParams v, int use_v) {
  k_prepass_body<W, R>(hw_grid(), s, wk, cnt, part, att_cnt, pinfo, blk_part, blk_rm, prm, v, use_v);
}


// the tiles that begin among the v attempts from o on, of pair i
__device__ inline void tile_mark(int64_t* tile_p, int64_t tcap, int64_t o, int64_t v, int64_t i) {
  for (int64_t t = (o + kWave - 1) / kWave; t * kWave < o + v && t < tcap; ++t) tile_p[t] = i;
}
// pairs of many attempts (a reference of 2e5 walkers holds 3e3 tiles) are
// marked by the whole wave; wave-wide call
constexpr int64_t kTileRun = 16 * kWave;
__device__ inline void tile_mark_runs(int64_t* tile_p, int64_t tcap, int64_t o, int64_t v, int64_t i) {
  for (uint64_t m = __ballot(v > kTileRun); m; m &= m - 1) {
    const int l = ctz64(m);
    const int64_t lo = (int64_t)lane_value((uint64_t)o, l), lv = (int64_t)lane_value((uint64_t)v, l);
    const int64_t li = (int64_t)lane_value((uint64_t)i, l);
    for (int64_t t = (lo + kWave - 1) / kWave + lane_id(); t * kWave < lo + lv && t < tcap; t += kWave) tile_p[t] = li;
  }
}

// attempt offsets per (slot, replica) pair, same chunking as k_prepass; also
// the parent pair of the first attempt of every kWave-attempt tile (the
// spawn kernel's tiles), written by the pair whose attempts contain it.  When
// a rebuild is due, also the refill of the walker hash that the prepass
// cleared, before any lookup of the iteration.
template <int W>
__device__ __forceinline__ void k_scan_apply_body(const Grid& g_, const DevSys& s, const Walk& wk, const int32_t* att_cnt, int64_t* att_off, const int64_t* part, const int64_t* part_rm, const uint8_t* pinfo, Counters* cnt, int S, int64_t* tile_p, int64_t tcap, const Bins& bins) {
  if (cnt->halt) return;
  __shared__ int64_t red[kBlock / kWave];
  int64_t nslots = (int64_t)cnt->nslots;
  if (cnt->rebuild) {
    hash_refill_part<W>(g_, s, wk, cnt, nslots);
    // the prepass's removals left no tombstones: the table now holds the live
    // slots only (the end-of-iteration accounting counts the later removals)
    if (g_.b == 0 && threadIdx.x == 0) {
      cnt->n_tomb = 0;
      cnt->rebuilt = 1;
      cnt->n_rebuilds += 1;
    }
  }
  int64_t begin, end;
  chunk_of(g_, nslots, begin, end);
  // the block of the last slots closes the scan; an empty table is block 0's
  const bool last = end == nslots && (begin < end || (nslots == 0 && g_.b == 0));
  if (begin >= end && !last) return;
  // this block's first attempt offset and first free-queue position: the
  // counts of the blocks before it.  The slots the prepass freed go, in slot
  // order, after the free queue's tail (the prepass appends nothing itself,
  // so the tail is still free_tail0, the value at the last accounting).
  // With one replica both scans run as one over packed counts (attempts in
  // the low 40 bits, freed slots above).
  const unsigned long long tail0 = cnt->free_tail0;
  constexpr int kPackShift = 40;
  int64_t loc = 0, loc_rm = 0;
  for (int q = threadIdx.x; q < (int)g_.b; q += blockDim.x) {
    loc += part[q];
    loc_rm += part_rm[q];
  }
  int64_t run, run_rm;
  (void)block_exclusive_scan(loc, red, run);
  (void)block_exclusive_scan(loc_rm, red, run_rm);
  if (S == 1) {
    for (int64_t b0 = begin; b0 < end; b0 += blockDim.x) {
      int64_t i = b0 + threadIdx.x;
      int64_t v = 0, f = 0;
      if (i < end) {
        v = att_cnt[i];
        f = (pinfo[i] & kPinfoFreed) ? 1 : 0;
      }
      int64_t tot;
      int64_t pre = block_exclusive_scan(v | (f << kPackShift), red, tot);
      const int64_t o = run + (pre & ((1ll << kPackShift) - 1));
      tile_mark_runs(tile_p, tcap, o, v, i);
      if (i < end) {
        att_off[i] = o;
        if (v <= kTileRun) tile_mark(tile_p, tcap, o, v, i);
        if (f) wk.freeq[(tail0 + (unsigned long long)(run_rm + (pre >> kPackShift))) % (unsigned long long)wk.cap] = i;
      }
      run += tot & ((1ll << kPackShift) - 1);
      run_rm += tot >> kPackShift;
    }
  } else {
    for (int64_t b0 = begin; b0 < end; b0 += blockDim.x) {
      int64_t slot = b0 + threadIdx.x;
      int64_t f = (slot < end && (pinfo[slot * S] & kPinfoFreed)) ? 1 : 0;
      int64_t tot;
      int64_t pre = block_exclusive_scan(f, red, tot);
      if (f) wk.freeq[(tail0 + (unsigned long long)(run_rm + pre)) % (unsigned long long)wk.cap] = slot;
      run_rm += tot;
    }
    int64_t pb = begin * S, pe = end * S;
    for (int64_t base = pb; base < pe; base += blockDim.x) {
      int64_t i = base + threadIdx.x;
      int64_t v = i < pe ? att_cnt[i] : 0;
      int64_t tot;
      int64_t pre = block_exclusive_scan(v, red, tot);
      const int64_t o = run + pre;
      tile_mark_runs(tile_p, tcap, o, v, i);
      if (i < pe) {
        att_off[i] = o;
        if (v <= kTileRun) tile_mark(tile_p, tcap, o, v, i);
      }
      run += tot;
    }
  }
  if (last && threadIdx.x == 0) {
    att_off[nslots * S] = run;
    cnt->n_attempts = (unsigned long long)run;
    cnt->free_tail = tail0 + (unsigned long long)run_rm;
    cnt->rm_pre = (unsigned long long)run_rm;
    // spawns expected at the previous iteration's rate per attempt, and no
    // fewer than one in kMinRate attempts: a larger time step, another shift or
    // an iteration that happened to spawn nothing says little about this one
    const double per = cnt->prev_attempts ? (double)cnt->prev_spawned / (double)cnt->prev_attempts : 0.5;
    const double expect = (double)run * (per > 1.0 / kMinRate ? per : 1.0 / kMinRate);
    // of that, determinants: the previous iteration's share, by the same bound
    const double share = cnt->prev_spawned ? (double)cnt->prev_unique / (double)cnt->prev_spawned : 1.0;
    set_bins(cnt, bins, expect, expect * (share > 1.0 / kMinRate ? share : 1.0 / kMinRate));
  }
}
template <int W>
__global__ void __launch_bounds__(kBlock) k_scan_apply(DevSys s, Walk wk, const int32_t* att_cnt, int64_t* att_off, const int64_t* part, const int64_t* part_rm, const uint8_t* pinfo, Counters* cnt, int S, int64_t* tile_p, int64_t tcap, Bins bins) {
  k_scan_apply_body<W>(hw_grid(), s, wk, att_cnt, att_off, part, part_rm, pinfo, cnt, S, tile_p, tcap, bins);
}

// ------------------------------------------------------------- spawning
// parent (slot, replica) of attempt a: last pair p in [lo, hi] with
// att_off[p] <= a (the caller's bounds bracket the answer)
__device__ inline int64_t parent_pair(const int64_t* att_off, int64_t lo, int64_t hi, int64_t a) {
  while (lo < hi) {
    int64_t mid = (lo + hi + 1) >> 1;
    if (att_off[mid] <= a) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// One wave's LDS stages of its spawned records and of the single-excitation
// attempts it queues.  Waves stage and flush on their own: the spawning
// kernels have no block barrier between their set-up and their statistics, so
// a wave that waits for its gathers holds up no other.
constexpr int kParentWindow = 4096;  // pairs of a tile's window, holes included; longer ones are bisected
constexpr int kSpawnStage = 128;     // flushed past 64
template <int W>
struct SpawnStage {
  uint64_t key[kSpawnStage * W];
  double val[kSpawnStage];
  uint32_t info[kSpawnStage];
};
constexpr int kQueueStage = 256;  // flushed past 192: one device atomic on the queue's counter each
struct QueueStage {  // queued attempts as (parent pair, attempt number)
  int64_t p[kQueueStage];
  uint32_t k[kQueueStage];
};

// A spawned-list record with FP64 amplitudes is kRecWords 64-bit words (32
// bytes, so a record never straddles a cache line): the determinant's words,
// the child amplitude (FP64 bits) in word 2 and the info word (bits 0-7
// replica, bit 8 parent initiator) in word 3.  With FP32 amplitudes it is
// W + 1 words: the determinant's words, then info << 32 | the amplitude's FP32
// bits (16 bytes for one-word determinants).  The merge reads one record per
// spawn and sums the amplitudes in FP64.
constexpr int kRecWords = 4;  // the larger of the two record sizes
template <int W>
__device__ inline double rec_val(const DevSys& s, const uint64_t* r) {
  return s.spawn_fp32 ? (double)__uint_as_float((uint32_t)r[W]) : __longlong_as_double((long long)r[2]);
}
template <int W>
__device__ inline uint32_t rec_info(const DevSys& s, const uint64_t* r) {
  return s.spawn_fp32 ? (uint32_t)(r[W] >> 32) : (uint32_t)r[3];
}

template <int W>
__device__ inline void rec_store(const DevSys& s, uint64_t* r, const uint64_t* key, double val, uint32_t info) {
  if (s.spawn_fp32) {  // the value is already FP32-representable (attempt_create)
    const uint64_t last = ((uint64_t)info << 32) | __float_as_uint((float)val);
    if constexpr (W == 1) {
      *(ulonglong2*)r = ulonglong2{key[0], last};
    } else {
      r[0] = key[0];
      r[1] = key[1];
      r[2] = last;
    }
  } else {
    *(ulonglong2*)r = ulonglong2{key[0], W == 2 ? key[W - 1] : 0ull};
    *(ulonglong2*)(r + 2) = ulonglong2{(uint64_t)__double_as_longlong(val), (uint64_t)info};
  }
}
// the mark of a record that found the merge's table full (the info word's top bit)
constexpr uint32_t kInfoLeft = 1u << 31;
template <int W>
__device__ inline void rec_mark(const DevSys& s, uint64_t* r, bool on) {
  const int w = s.spawn_fp32 ? W : 3;
  const uint64_t bit = s.spawn_fp32 ? 1ull << 63 : (uint64_t)kInfoLeft;
  r[w] = on ? r[w] | bit : r[w] & ~bit;
}

// the wave's n staged spawns into their bins, at most two a lane; the counter
// atomics are issued before the first record is written
template <int W>
__device__ inline void spawn_flush(const SpawnStage<W>* ss, int n, Counters* cnt, const Bins& bins, const DevSys& s) {
  wave_sync();
  const uint32_t nb = cnt->nbins, cap = cnt->bin_cap, sh = cnt->bin_shift;
  const int lane = lane_id();
  uint32_t bin[2], pos[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = lane + j * kWave;
    bin[j] = pos[j] = 0;
    if (i < n) {
      bin[j] = bin_of(bin_hash<W>(ss->key + i * W), nb);
      pos[j] = atomicAdd(&bins.count[(size_t)bin[j] << sh], 1u);
    }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = lane + j * kWave;
    const bool over = i < n && pos[j] >= cap;
    uint64_t* r = i < n && !over ? bins.rec + ((size_t)bin[j] * cap + pos[j]) * s.rec_words : nullptr;
    if (const uint64_t om = __ballot(over)) {
      const unsigned long long base = wave_reserve(&cnt->n_ovf, popc64(om));
      if (over)
        r = bin_overflow(bins, bin[j], pos[j] - cap, base + (unsigned long long)popc64(om & lanemask_lt()), s.rec_words);
    }
    if (r) rec_store<W>(s, r, ss->key + i * W, ss->val[i], ss->info[i]);
  }
  wave_sync();
}

// An explicit spawned list (n dense records) into the bins, each record at the
// place the host chose for it: places in list order, so that a wave reads a
// determinant's records, and sums them, in the order of the list.  Places count
// through the bins' records and the overflow list; an overflow record's link is
// the one before it in its chain, or, past kChainHead, the chain it begins.
constexpr int64_t kChainHead = 1ll << 40;
template <int W>
__global__ void __launch_bounds__(kBlock) k_bin_list(DevSys s, Counters* cnt, const uint64_t* list, const int64_t* place, const int64_t* link, int64_t n, Bins bins) {
  const uint32_t nb = cnt->nbins, sh = cnt->bin_shift;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const uint64_t* q = list + i * s.rec_words;
    const int64_t p = place[i];
    const uint32_t bin = bin_of(bin_hash<W>(q), nb);
    atomicAdd(&bins.count[(size_t)bin << sh], 1u);
    uint64_t* r = bins.rec + p * s.rec_words;
    if (p >= bins.cap) {
      const int64_t o = p - bins.cap, l = link[i];
      if (l >= kChainHead) bins.head[l - kChainHead] = (uint32_t)o;
      else bins.next[l] = (uint32_t)o;
      r = bins.ovf + o * s.rec_words;
    }
    for (int w = 0; w < s.rec_words; ++w) r[w] = q[w];
  }
}
__global__ void k_set_bins(Counters* cnt, Bins bins, int64_t n) { set_bins(cnt, bins, (double)n, (double)n); }

// the wave's n staged attempts to the queue from base on
__device__ inline void queue_write(const QueueStage* qs, int n, unsigned long long base, int64_t* sq, int64_t scap,
                                   bool& overflow) {
  for (int i = lane_id(); i < n; i += kWave) {
    const unsigned long long d = base + (unsigned long long)i;
    if (d < (unsigned long long)scap) *(longlong2*)(sq + 2 * d) = longlong2{qs->p[i], (int64_t)qs->k[i]};
    else overflow = true;
  }
}

// is_core_state (semi_stoch_procs.F90:590-605) of the child of an excitation:
// core dets are always resident, so the walker hash and its core flag answer it
template <int W>
__device__ inline bool core_child(const DevSys& s, const Walk& wk, Counters* cnt, const uint64_t* key,
                                  const Excit& ex) {
  uint64_t child[W];
  apply_excit<W>(key, ex, child);
  int64_t home = find_walker_hash<W>(child, s.rh, s.L) - 1;
  int64_t pos = hash_lookup<W>(wk, child, home, cnt);
  return pos >= 0 && (wk.flags(pos) & kFlagCore);
}

// statistics of the spawning kernels, per lane until the end of the kernel
template <int R>
struct SpawnAcc {
  LaneSum<1> valid, invalid, bloomc1, bloomc2;
  LaneMax maxspawn, blooms1, blooms2;
  LaneSum<R> born, sing;
  __device__ void done(BlockStats& bs, int mode) {
    valid.done(bs, S_NVALID);
    invalid.done(bs, S_NINVALID);
    maxspawn.done(bs, S_MAXSPAWN);
    born.done(bs, soff(F_NBORN, 0));
    if (mode != 1) {
      sing.done(bs, soff(F_SPAWNSING, 0));
      bloomc1.done(bs, S_BLOOMC + 1);
      blooms1.done(bs, S_BLOOMS + 1);
    }
    if (mode != 2) {
      bloomc2.done(bs, S_BLOOMC + 2);
      blooms2.done(bs, S_BLOOMS + 2);
    }
  }
};

// generator bound at compile time, one k_spawn instantiation each, so that the
// code of one generator (the uniform one's private arrays in particular) costs
// the others nothing
// generator instances of the spawn kernel: the lattice generator, PCHB with
// FAST-FAST holes and UNIF-UNIF / UNIF-FAST particles (a fixed number of
// uniforms), the uniform molecular generator, and PCHB with weighted
// particles or holes (constrained samplers that may redraw)
constexpr int kGenHubbard = 0, kGenPchb = 1, kGenUniform = 2, kGenPchbW = 3;

// one spawning attempt (attempt_create_normal + create_particle); mode 0: any
// excitation, 1: doubles only (singles are queued), 2: singles only.  Wave-wide.
template <int W, int R, int G>
__device__ inline void spawn_attempt(const DevSys& s, const Walk& wk, Counters* cnt, BlockStats& bs,
                                     SpawnAcc<R>& acc, const uint8_t* pinfo, bool active, int64_t p, uint32_t k,
                                     int mode, SpawnStage<W>* ss, int& n_ss, QueueStage* qs, int& n_qs, double tau,
                                     uint32_t iter) {
  const int S = R <= 2 ? R : s.S;
  bool emit = false, queue = false;
  uint64_t child[W];
  double nspawn = 0.0, an = 0.0, raw = 0.0;
  uint32_t info = 0;
  int r = 0, ic = 0;
  double valid = 0.0, invalid = 0.0;
  if (active) {
    int64_t slot = p / S;
    r = (int)(p - slot * S);
    uint64_t key[W];
#pragma unroll
    for (int w = 0; w < W; ++w) key[w] = wk.keys[slot * W + w];
    double dr[6];
    draw2<W>(s.seed, key, iter, r, k, 1, dr[0], dr[1]);
    constexpr bool kPchb = G == kGenPchb || G == kGenPchbW;
    bool single = kPchb && dr[0] < s.psingles;
    if (mode == 1 && single) {
      queue = true;
    } else {
      // purpose 2: the PCHB hole pair (d3) and the spawn rounding (d5); purpose
      // 3 (d2, d4) only for the generators that read them
      draw2<W>(s.seed, key, iter, r, k, 2, dr[3], dr[5]);
      dr[2] = dr[4] = 0.0;
      if (G == kGenUniform || G == kGenPchbW || (G == kGenPchb && (s.particles == 1 || single)))
        draw2<W>(s.seed, key, iter, r, k, 3, dr[2], dr[4]);
      Excit ex;
      if constexpr (G == kGenHubbard) {
        ex = gen_hubbard<W>(s, key, dr);
      } else if constexpr (G == kGenUniform) {
        bool fail = false;
        ex = gen_excit<W>(s, key, dr, iter, r, k, &fail);
        if (fail) atomicOr(&cnt->err, 1u << NGPU_ERR_EXCITGEN);
      } else if (single) {
        ex = gen_single_heatbath<W>(s, key, dr[1], dr[2]);
        ex.pgen = ex.pgen * s.psingles;
      } else if constexpr (G == kGenPchbW) {
        DrawSeq<W> u(dr, s.seed, key, iter, r, k);
        ex = gen_double_pchb_weighted<W>(s, key, u);
        ex.pgen = ex.pgen * s.pdoubles;
      } else {
        ex = gen_double_pchb<W>(s, key, dr);
        ex.pgen = ex.pgen * s.pdoubles;
      }
      if (ex.ic == 0) {
        invalid = 1.0;
      } else if (s.ncore && (pinfo[p] & 4) && core_child<W>(s, wk, cnt, key, ex)) {
        valid = 1.0;  // spawning from and to the core space is cancelled
      } else {
        valid = 1.0;
        ic = ex.ic;
        double hel = ex.hel_ok ? (ex.parity ? -ex.hel : ex.hel)
                               : helement_ex<W>(s, key, ex.ic, ex.e0, ex.e1, ex.e2, ex.e3, ex.parity);
        uint8_t pi = pinfo[p];
        double wsign = (pi & 1) ? -1.0 : 1.0;
        nspawn = attempt_create(s, tau, hel, ex.pgen, wsign, dr[5], raw);
        raw = fabs(raw);
        if (fabs(nspawn) > kEps) {
          emit = true;
          an = fabs(nspawn);
          apply_excit<W>(key, ex, child);
          info = (uint32_t)r | ((s.t_init && (pi & 2)) ? kInfoInit : 0u);
        }
      }
    }
  }
  if (mode == 1) {
    const uint64_t m = __ballot(queue);
    if (queue) {
      const int qi = n_qs + popc64(m & lanemask_lt());
      qs->p[qi] = p;
      qs->k[qi] = k;
    }
    n_qs += popc64(m);
  }
  acc.invalid.add(bs, S_NINVALID, invalid);
  acc.valid.add(bs, S_NVALID, valid);
  acc.maxspawn.add(raw);
  for (int rr = 0; rr < S; ++rr) {
    acc.born.add(bs, soff(F_NBORN, rr), rr == r ? an : 0.0);
    if (mode != 1) acc.sing.add(bs, soff(F_SPAWNSING, rr), (rr == r && ic == 1) ? an : 0.0);
  }
  bool bloom = emit && an > s.init_walk_no;
  if (mode != 2) {
    acc.bloomc2.add(bs, S_BLOOMC + 2, (bloom && ic == 2) ? 1.0 : 0.0);
    acc.blooms2.add((bloom && ic == 2) ? an : 0.0);
  }
  if (mode != 1) {
    acc.bloomc1.add(bs, S_BLOOMC + 1, (bloom && ic == 1) ? 1.0 : 0.0);
    acc.blooms1.add((bloom && ic == 1) ? an : 0.0);
  }
  const uint64_t em = __ballot(emit);
  if (emit) {
    const int idx = n_ss + popc64(em & lanemask_lt());
#pragma unroll
    for (int w = 0; w < W; ++w) ss->key[idx * W + w] = child[w];
    ss->val[idx] = nspawn;
    ss->info[idx] = info;
  }
  n_ss += popc64(em);
}

// generators whose attempts loop over draws: at 2e4 attempts of the weighted
// one (8e/16o) a wave of 16 attempts and the draws by four take 41 us of 52;
// eight attempts a wave take 45 with eight values of a sum in flight
template <int G>
constexpr bool kSplitTiles = G == kGenUniform || G == kGenPchbW;

// all attempts: Hubbard spawns directly; molecular doubles spawn here while
// singles (the heat-bath list is ~20x longer per attempt) go to a queue so that
// waves do not idle on a few long lanes
template <int W, int R, int G>
__device__ __forceinline__ void k_spawn_body(const Grid& g_, const DevSys& s, const Walk& wk, Counters* cnt, double* part, const int64_t* att_off, const int64_t* tile_p, int64_t tcap, const uint8_t* pinfo, const Bins& bins, int64_t scap, int64_t* sq, const IterParams* prm) {
  if (cnt->halt) return;
  const int64_t total = (int64_t)cnt->n_attempts;
  constexpr int kWaves = kBlock / kWave;
  // waves per tile of 64 attempts: with few attempts a wave takes a part of a
  // tile, as long loops run to the longest of its lanes
  const int64_t twaves = g_.nb * kWaves, tiles = (total + kWave - 1) / kWave;
  const int sub = !kSplitTiles<G> ? 1 : 4 * tiles <= twaves ? 4 : 2 * tiles <= twaves ? 2 : 1;
  if (g_.b * kWaves >= tiles * sub) return;  // no attempts for this block
  const double tau = prm->tau;
  const uint32_t iter = prm->iter;
  constexpr int mode = (G == kGenPchb || G == kGenPchbW) ? 1 : 0;
  __shared__ double acc_lds[kStatStride];
  __shared__ SpawnStage<W> sstages[kWaves];
  __shared__ QueueStage qstages[mode == 1 ? kWaves : 1];
  __shared__ uint32_t parents[kBlock];
  __shared__ uint32_t tail_n[kWaves];
  __shared__ unsigned long long tail_base;
  __shared__ unsigned int blk_spawned;
  BlockStats bs{acc_lds};
  if (threadIdx.x == 0) blk_spawned = 0;
  bs.zero();
  const int wv = threadIdx.x / kWave, lane = lane_id();
  SpawnStage<W>* ss = &sstages[wv];
  QueueStage* qs = &qstages[mode == 1 ? wv : 0];
  uint32_t* par = parents + wv * kWave;
  int n_ss = 0, n_qs = 0;     // staged (wave-uniform)
  unsigned int spawned = 0;
  const int64_t npairs = (int64_t)cnt->nslots * s.S;
  bool overflow = false;
  SpawnAcc<R> acc;
  // tiles of 64 consecutive attempts, one (or a part of one) per wave and trip
  for (int64_t t0 = g_.b * kWaves + wv; t0 < tiles * sub; t0 += twaves) {
    const int64_t tile = sub == 1 ? t0 : t0 / sub, a0 = tile * kWave, a = a0 + lane;
    // the tile's parents lie between its first attempt's and the next tile's
    const bool more = a0 + kWave < total;
    const bool act = a < total && (sub == 1 || (lane * sub) / kWave == (int)(t0 - tile * sub));
    int64_t lo, hi;
    if (tile + 1 < tcap) {
      lo = tile_p[tile];
      hi = more ? tile_p[tile + 1] : npairs - 1;
    } else {  // beyond the tile table: full searches
      lo = parent_pair(att_off, 0, npairs - 1, a0);
      hi = parent_pair(att_off, lo, npairs - 1, (more ? a0 + kWave : total) - 1);
    }
    int64_t p = 0;
    uint32_t k = 0;
    if (hi - lo < kParentWindow) {
      // each pair of the window marks its first attempt in the tile (of pairs
      // at the same place the last one, which has the attempts), and a maximum
      // over the lanes below spreads the marks
      par[lane] = 0;
      wave_sync();
      for (int64_t i = lane; i <= hi - lo; i += kWave) {
        const int64_t o = att_off[lo + i] - a0;
        if (o < kWave) atomicMax(&par[o > 0 ? o : 0], (uint32_t)i);
      }
      wave_sync();
      uint32_t v = par[lane];
      auto up = [&](uint32_t w) { v = w > v ? w : v; };
      up(dpp_u32<kRowShr + 1, 0xF>(v));
      up(dpp_u32<kRowShr + 2, 0xF>(v));
      up(dpp_u32<kRowShr + 4, 0xF>(v));
      up(dpp_u32<kRowShr + 8, 0xF>(v));
      up(dpp_u32<kRowBcast15, 0xA>(v));
      up(dpp_u32<kRowBcast31, 0xC>(v));
      if (act) p = lo + v;
    } else if (act) {
      p = parent_pair(att_off, lo, hi, a);
    }
    if (act) k = (uint32_t)(a - att_off[p]);
    const int before = n_ss;
    spawn_attempt<W, R, G>(s, wk, cnt, bs, acc, pinfo, act, p, k, mode, ss, n_ss, qs, n_qs, tau, iter);
    spawned += (unsigned int)(n_ss - before);
    if (n_ss > kSpawnStage - kWave) {
      spawn_flush<W>(ss, n_ss, cnt, bins, s);
      n_ss = 0;
    }
    if (mode == 1 && n_qs > kQueueStage - kWave) {
      wave_sync();
      queue_write(qs, n_qs, wave_reserve(&cnt->n_singles, n_qs), sq, scap, overflow);
      wave_sync();
      n_qs = 0;
    }
  }
  if (n_ss) spawn_flush<W>(ss, n_ss, cnt, bins, s);
  // what is still queued: one reservation per block
  if (lane == 0) {
    if (spawned) atomicAdd(&blk_spawned, spawned);
    tail_n[wv] = (uint32_t)n_qs;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (blk_spawned) atomicAdd(&cnt->n_spawned, (unsigned long long)blk_spawned);
    unsigned int n = 0;
    for (int q = 0; q < kWaves; ++q) n += tail_n[q];
    if (mode == 1 && n) tail_base = atomicAdd(&cnt->n_singles, (unsigned long long)n);
  }
  if (mode == 1) {
    __syncthreads();
    unsigned int before = 0;
    for (int q = 0; q < wv; ++q) before += tail_n[q];
    queue_write(qs, n_qs, tail_base + before, sq, scap, overflow);
  }
  if (overflow) atomicOr(&cnt->err, 1u << NGPU_ERR_SPAWN_FULL);
  acc.done(bs, mode);
  bs.flush(part, g_.b);
}
template <int W, int R, int G>
__global__ void __launch_bounds__(kBlock) k_spawn(DevSys s, Walk wk, Counters* cnt, double* part, const int64_t* att_off, const int64_t* tile_p, int64_t tcap, const uint8_t* pinfo, Bins bins, int64_t scap, int64_t* sq, const IterParams* prm) {
  k_spawn_body<W, R, G>(hw_grid(), s, wk, cnt, part, att_off, tile_p, tcap, pinfo, bins, scap, sq, prm);
}

// Queued single excitations (molecular, heat-bath singles).  A wave takes up to
// 64 attempts a trip.  What an attempt needs once (queue entry, draws, source,
// element, spawn, statistics) runs with one lane per attempt; the weights
// |hb_weight(src -> b)| of every same-spin orbital b, ~20 times as long, with G
// lanes per attempt (G = 4, 8 or 16, a launch-shape choice), 64/G attempts a
// round: lane g takes every G-th pair of neighbouring orbitals b, the
// reference-relative element fref[src][b], then the Coulomb and (of the same
// spin) exchange rows of the orbitals j in which the parent and the reference
// differ, 16 bytes a lane and a group's loads one contiguous run, added in
// hb_weight's order.  The loads' lanes bound the kernel, so rows that are not
// needed (exchange of the other spin, the second of an odd list) are masked.
//  gen_single_heatbath's two sequential sweeps run over
// the group's registers by DPP broadcasts, in ascending b, so the selected
// orbital, pgen and the spawn's element (the selected weight, signed) are
// bit-identical to the one-lane generator.  The differing orbitals wait in LDS
// as a byte list per attempt, so a round's loop is as long as its longest list
// of both signs.
// Measured (a whole attempt on its G lanes, sums through LDS, interleaved
// (Coulomb, exchange) pairs before; us): 14e/30o at 5e6 walkers 139 -> 115,
// 26e/40o 131 -> 81, 10e/20o 32 -> 30, 2e3 attempts 13.3 -> 12.  Of the 24 at
// 14e/30o the masks of rows not needed are 38, without them the dense lanes
// alone had cost 14: the loads keep the address units busy for two thirds of
// the time.
// Eight lanes per attempt take 124 and 101, sixteen 150 and 132.

// a group's lanes exchange by DPP: lane I's value, and the sum over the lanes
// of values of which at most one is not 0 (or of small counts)
template <int G, int I>
__device__ inline uint32_t group_lane(uint32_t v) {
  if constexpr (G == 4) return dpp_u32<I * 0x55, 0xF>(v);
  else if constexpr (G == 16) return dpp_u32<kRowNewbcast + I, 0xF>(v);
  else {
    const uint32_t lo = dpp_u32<kRowNewbcast + I, 0xF>(v), hi = dpp_u32<kRowNewbcast + 8 + I, 0xF>(v);
    return (threadIdx.x & 8) ? hi : lo;
  }
}
template <int G>
__device__ inline uint32_t group_sum(uint32_t v) {
  v += dpp_u32<0xB1, 0xF>(v);  // quads: lanes 1 0 3 2, then 2 3 0 1
  v += dpp_u32<0x4E, 0xF>(v);
  if constexpr (G >= 8) v += dpp_u32<kRowHalfMirror, 0xF>(v);
  if constexpr (G >= 16) v += dpp_u32<kRowMirror, 0xF>(v);
  return v;
}
template <int G, int I>
__device__ inline double group_lane(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint64_t w = ((uint64_t)group_lane<G, I>((uint32_t)(u >> 32)) << 32) | group_lane<G, I>((uint32_t)u);
  return __longlong_as_double((long long)w);
}
// cum += |v[0]|, |v[1]| of the lanes I = 0..G-1 of the group in order; mine:
// the sums after this lane's own
template <int G, int I>
__device__ inline void group_cum(const double* v, int g, double& cum, double* mine) {
  if constexpr (I < G) {
    const double c0 = cum + fabs(group_lane<G, I>(v[0]));
    cum = c0 + fabs(group_lane<G, I>(v[1]));
    if (g == I) {
      mine[0] = c0;
      mine[1] = cum;
    }
    group_cum<G, I + 1>(v, g, cum, mine);
  }
}

// bytes of an attempt's list: orbital-1, and 0x80 for one that the parent lacks
__host__ __device__ inline int singles_list(int nel, int nbasis) {
  const int m = 2 * (nel < nbasis - nel ? nel : nbasis - nel);
  return m < 8 ? 8 : (m + 7) & ~7;
}

// a wave's attempts between the two divisions of its lanes
template <int W>
struct SingleStage {
  uint64_t key[W * kWave];
  double a[kWave];       // selection uniform, then the normalisation
  double v[kWave];       // the selected signed weight
  double round[kWave];   // the spawn's rounding uniform
  uint32_t meta[kWave];  // source | replica << 8 | parent bits << 16
  uint32_t n[kWave];     // differing orbitals, then the selected b - 1
};

// PP: pairs of spatial orbitals per lane (nsp <= 2*G*PP); dynamic LDS holds the lists
template <int W, int R, int PP, int G>
__device__ __forceinline__ void k_spawn_singles_body(const Grid& g_, const DevSys& s, const Walk& wk, Counters* cnt, double* part, const uint8_t* pinfo, const Bins& bins, int64_t scap, const int64_t* sq, const IterParams* prm) {
  if (cnt->halt) return;
  constexpr int kWaves = kBlock / kWave;
  constexpr int kPer = kWave / G;  // attempts of a round
  int64_t nq = (int64_t)cnt->n_singles;
  if (nq > scap) nq = scap;
  // rounds of a trip: as few as give every wave the same number of trips
  const int64_t nwaves = g_.nb * kWaves;
  const int64_t trips = (nq + nwaves * kWave - 1) / (nwaves * kWave);
  const int rounds = nq > 0 ? (int)((nq + nwaves * trips * kPer - 1) / (nwaves * trips * kPer)) : 1;
  const int per = rounds * kPer;
  if (g_.b * kWaves * per >= nq) return;  // no queued attempts for this block
  const double tau = prm->tau;
  const uint32_t iter = prm->iter;
  __shared__ double acc_lds[kStatStride];
  __shared__ SpawnStage<W> sstages[kWaves];
  __shared__ SingleStage<W> qstages[kWaves];
  __shared__ unsigned int blk_spawned;
  extern __shared__ uint64_t lists_dyn[];
  if (threadIdx.x == 0) blk_spawned = 0;
  const int wv = threadIdx.x / kWave, lane = lane_id();
  SpawnStage<W>* ss = &sstages[wv];
  SingleStage<W>* st = &qstages[wv];
  int n_ss = 0;  // staged (wave-uniform)
  unsigned int spawned = 0;
  BlockStats bs{acc_lds};
  bs.zero();
  const int S = R <= 2 ? R : s.S;
  SpawnAcc<R> acc;
  const int nsp = s.nbasis / 2;
  const int rs = (nsp + 1) & ~1;  // stride of the Coulomb and exchange rows
  const int g = lane % G;
  const int lw = singles_list(s.nel, s.nbasis) / 8;
  uint64_t* lists = lists_dyn + (size_t)wv * kWave * lw;
  for (int64_t q0 = (g_.b * kWaves + wv) * per; q0 < nq; q0 += nwaves * per) {
    const int64_t left = nq - q0;
    const bool act = lane < per && lane < left;
    {
      // idle lanes: any valid determinant, no differing orbitals
      uint64_t key[W];
      int64_t p = 0;
      uint32_t k = 0;
      if (act) {
        p = sq[2 * (q0 + lane)];
        k = (uint32_t)sq[2 * (q0 + lane) + 1];
      }
      const int64_t slot = p / S;
      const int r = (int)(p - slot * S);
#pragma unroll
      for (int w = 0; w < W; ++w) key[w] = act ? wk.keys[slot * W + w] : s.ref[w];
      const uint32_t pi = act ? pinfo[p] : 0u;
      double d0, d1, d2, d3, d4, d5;
      draw2<W>(s.seed, key, iter, r, k, 1, d0, d1);
      draw2<W>(s.seed, key, iter, r, k, 2, d3, d5);
      draw2<W>(s.seed, key, iter, r, k, 3, d2, d4);
      const int src = select_orb<W>(key, ~0ull, 1 + (int)floor(d1 * (double)s.nel));
#pragma unroll
      for (int w = 0; w < W; ++w) st->key[w * kWave + lane] = key[w];
      st->a[lane] = d2;
      st->round[lane] = d5;
      st->meta[lane] = (uint32_t)src | ((uint32_t)r << 8) | (pi << 16);
      // the orbitals the parent occupies beyond the reference, then the
      // reference's orbitals the parent lacks (hb_weight's order)
      uint8_t* list = (uint8_t*)(lists + (size_t)lane * lw);
      uint32_t n = 0;
#pragma unroll
      for (int w = 0; w < 2 * W; ++w) {
        const int ww = w % W;
        uint64_t x = w < W ? key[ww] & ~s.ref[ww] : s.ref[ww] & ~key[ww];
        if ((src - 1) >> 6 == ww) x &= ~(1ull << ((src - 1) & 63));
        while (x) {
          list[n++] = (uint8_t)((64 * ww + ctz64(x)) | (w < W ? 0 : 0x80));
          x &= x - 1;
        }
      }
      st->n[lane] = n;
    }
    wave_sync();
    const int live = left < per ? (int)left : per;
    for (int t0 = 0; t0 < live; t0 += kPer) {
      const int j = t0 + lane / G;
      const int src = (int)(st->meta[j] & 0xFF), n = (int)st->n[j];
      const uint32_t spin = (uint32_t)(src - 1) & 1u;
      const double* frow = s.fref + (size_t)(src - 1) * nsp;
      const double* row = s.jkrow + (size_t)2 * rs * nsp * ((src - 1) >> 1) + 2 * g;
      double v[2 * PP];
#pragma unroll
      for (int m = 0; m < 2 * PP; ++m) {
        const int b = 2 * (g + m / 2 * G) + m % 2;
        v[m] = b < nsp ? frow[b] : 0.0;
      }
      // two orbitals per step so that both rows' loads are in flight before
      // the ordered additions.  (Loads past a row's end stay in the table,
      // which is padded, and their values are dropped below.)
      const uint64_t* list = lists + (size_t)j * lw;
      uint64_t chunk = 0;
      for (int i = 0; i < n; i += 2) {
        if ((i & 7) == 0) chunk = list[i >> 3];
        const uint32_t e1 = (uint32_t)chunk & 0xFF, e2 = (uint32_t)(chunk >> 8) & 0xFF;
        chunk >>= 16;
        const bool two = i + 1 < n;
        const bool x1 = (e1 & 1u) == spin, x2 = two && (e2 & 1u) == spin;
        const double* r1 = row + (size_t)(2 * rs) * ((e1 & 0x7F) >> 1);
        const double* r2 = row + (size_t)(2 * rs) * ((e2 & 0x7F) >> 1);
        double2 j1[PP], k1[PP], j2[PP], k2[PP];
#pragma unroll
        for (int m = 0; m < PP; ++m) j1[m] = *(const double2*)(r1 + 2 * G * m);
        if (x1) {
#pragma unroll
          for (int m = 0; m < PP; ++m) k1[m] = *(const double2*)(r1 + rs + 2 * G * m);
        }
        if (two) {
#pragma unroll
          for (int m = 0; m < PP; ++m) j2[m] = *(const double2*)(r2 + 2 * G * m);
        }
        if (x2) {
#pragma unroll
          for (int m = 0; m < PP; ++m) k2[m] = *(const double2*)(r2 + rs + 2 * G * m);
        }
        // +-1: the products are exact, so these are the plain sums
        const double s1 = (e1 & 0x80) ? -1.0 : 1.0, s2 = (e2 & 0x80) ? -1.0 : 1.0;
        auto add = [&](double f, const double2* a) {
#pragma unroll
          for (int m = 0; m < PP; ++m) {
            v[2 * m] = fma(f, a[m].x, v[2 * m]);
            v[2 * m + 1] = fma(f, a[m].y, v[2 * m + 1]);
          }
        };
        add(s1, j1);
        if (x1) add(-s1, k1);
        if (two) add(s2, j2);
        if (x2) add(-s2, k2);
      }
      // occupied targets and the lanes' orbitals past the last have no weight
      {
        uint64_t key[W];
#pragma unroll
        for (int w = 0; w < W; ++w) key[w] = st->key[w * kWave + j];
#pragma unroll
        for (int m = 0; m < 2 * PP; ++m) {
          // orbital-1 = 4G (m/2) + the rest, which is below 4G, and that divides 64
          const int o = 4 * G * (m / 2), rest = 4 * g + 2 * (m % 2) + (int)spin;
          const bool occ = o / 64 < W && (key[o / 64 < W ? o / 64 : 0] >> (o % 64 + rest)) & 1;
          if (2 * (g + m / 2 * G) + m % 2 >= nsp || occ) v[m] = 0.0;
        }
      }
      // the normalisation in ascending b, then the first b whose running sum
      // reaches r (the last b when none does): the running sums of a second
      // sweep in the same order are the same values, and they do not fall, so
      // that b is the number of sums below r
      double cum = 0.0, own[2 * PP];
#pragma unroll
      for (int m = 0; m < 2 * PP; m += 2) {
        own[m] = own[m + 1] = 0.0;
        group_cum<G, 0>(v + m, g, cum, own + m);
      }
      const double rr = st->a[j] * cum;
      uint32_t below = 0;
#pragma unroll
      for (int m = 0; m < 2 * PP; ++m)
        below += (2 * (g + m / 2 * G) + m % 2 < nsp && own[m] < rr) ? 1u : 0u;
      below = group_sum<G>(below);
      if (below > (uint32_t)(nsp - 1)) below = (uint32_t)(nsp - 1);
      uint64_t sel = 0;
#pragma unroll
      for (int m = 0; m < 2 * PP; ++m)
        sel = (uint32_t)(2 * (g + m / 2 * G) + m % 2) == below ? (uint64_t)__double_as_longlong(v[m]) : sel;
      sel = ((uint64_t)group_sum<G>((uint32_t)(sel >> 32)) << 32) | group_sum<G>((uint32_t)sel);
      if (g == 0) {
        st->a[j] = cum;
        st->v[j] = __longlong_as_double((long long)sel);
        st->n[j] = below;
      }
    }
    wave_sync();
    bool emit = false;
    uint64_t key[W], child[W];
    double nspawn = 0.0, an = 0.0, raw = 0.0, valid = 0.0, invalid = 0.0;
    uint32_t info = 0;
    int r = 0;
    if (act) {
#pragma unroll
      for (int w = 0; w < W; ++w) key[w] = st->key[w * kWave + lane];
      const uint32_t meta = st->meta[lane], pi = meta >> 16;
      const int src = (int)(meta & 0xFF);
      const int tgt = 2 * (int)st->n[lane] + 2 - (is_beta(src) ? 1 : 0);
      const double cum_sum = st->a[lane], vsel = st->v[lane], cpt = fabs(vsel);
      r = (int)((meta >> 8) & 0xFF);
      const bool none = fabs(cum_sum) <= kEps || cpt == 0.0;
      bool cancel = false;
      if (!none && s.ncore && (pi & 4)) {
        Excit ex{};
        ex.ic = 1;
        ex.e0 = src;
        ex.e1 = tgt;
        cancel = core_child<W>(s, wk, cnt, key, ex);  // from and to the core space
      }
      if (none) {
        invalid = 1.0;
      } else if (cancel) {
        valid = 1.0;
      } else {
        valid = 1.0;
        double pg = cpt / cum_sum;
        pg = pg / (double)s.nel;
        pg = pg * s.psingles;
        double hel = single_parity<W>(key, src, tgt) ? -vsel : vsel;  // the weight's own sum
        double wsign = (pi & 1) ? -1.0 : 1.0;
        nspawn = attempt_create(s, tau, hel, pg, wsign, st->round[lane], raw);
        raw = fabs(raw);
        if (fabs(nspawn) > kEps) {
          emit = true;
          an = fabs(nspawn);
#pragma unroll
          for (int w = 0; w < W; ++w) child[w] = key[w];
          flip_orb<W>(child, src);
          flip_orb<W>(child, tgt);
          info = (uint32_t)r | ((s.t_init && (pi & 2)) ? kInfoInit : 0u);
        }
      }
    }
    acc.invalid.add(bs, S_NINVALID, invalid);
    acc.valid.add(bs, S_NVALID, valid);
    acc.maxspawn.add(raw);
    for (int rr2 = 0; rr2 < S; ++rr2) {
      acc.born.add(bs, soff(F_NBORN, rr2), rr2 == r ? an : 0.0);
      acc.sing.add(bs, soff(F_SPAWNSING, rr2), rr2 == r ? an : 0.0);
    }
    bool bloom = emit && an > s.init_walk_no;
    acc.bloomc1.add(bs, S_BLOOMC + 1, bloom ? 1.0 : 0.0);
    acc.blooms1.add(bloom ? an : 0.0);
    const uint64_t em = __ballot(emit);
    if (emit) {
      const int idx = n_ss + popc64(em & lanemask_lt());
#pragma unroll
      for (int w = 0; w < W; ++w) ss->key[idx * W + w] = child[w];
      ss->val[idx] = nspawn;
      ss->info[idx] = info;
    }
    n_ss += popc64(em);
    spawned += (unsigned int)popc64(em);
    if (n_ss > kSpawnStage - kWave) {
      spawn_flush<W>(ss, n_ss, cnt, bins, s);
      n_ss = 0;
    }
    wave_sync();  // the next attempts reuse the LDS
  }
  if (n_ss) spawn_flush<W>(ss, n_ss, cnt, bins, s);
  if (spawned && lane == 0) atomicAdd(&blk_spawned, spawned);
  __syncthreads();
  if (threadIdx.x == 0 && blk_spawned) atomicAdd(&cnt->n_spawned, (unsigned long long)blk_spawned);
  acc.done(bs, 2);
  bs.flush(part, g_.b);
}
template <int W, int R, int PP, int G>
__global__ void __launch_bounds__(kBlock, PP <= 3 ? 4 : PP <= 5 ? 3 : 2) k_spawn_singles(DevSys s, Walk wk, Counters* cnt, double* part, const uint8_t* pinfo, Bins bins, int64_t scap, const int64_t* sq, const IterParams* prm) {
  k_spawn_singles_body<W, R, PP, G>(hw_grid(), s, wk, cnt, part, pinfo, bins, scap, sq, prm);
}

// ---------------------------------------------------------- radix sort
// Stable LSD radix sort, 8-bit digits, reduce-then-scan: per-block digit
// histograms, a per-digit scan over blocks, stable block-local scatter.  The
// set-up paths sort with it (the core space's selection and its connections).
constexpr int kRadixBins = 256;  // digit values
// radix tiles: IT elements per thread, IT*kBlock per tile

// element range of this block in the histogram and scatter passes: whole
// tiles, and no more blocks than there are tiles (blocks past the last tile
// get an empty range), so that a small list is not spread over more
// blocks than it fills
template <int IT>
__device__ inline void radix_chunk(const Grid& g, int64_t n, int64_t& begin, int64_t& end) {
  constexpr int kRadixTile = IT * kBlock;
  int64_t tiles = (n + kRadixTile - 1) / kRadixTile;
  int64_t nb = tiles < g.nb ? tiles : g.nb;
  if (nb < 1) nb = 1;
  int64_t per = (tiles + nb - 1) / nb * kRadixTile;
  begin = g.b * per;
  end = begin + per;
  if (end > n) end = n;
  if (begin > n) begin = n;
}

// sort key: NW words of type K per element; FLIP compares word 0 as signed
// DB-bit digit (kRadixBins is the largest digit range)
template <typename K, int NW, bool FLIP, int DB = 8>
__device__ inline uint32_t radix_digit(const K* k, int word, int shift) {
  K x = k[word];
  if (FLIP && word == 0) x ^= (K)1 << (sizeof(K) * 8 - 1);
  return (uint32_t)(x >> shift) & ((1u << DB) - 1u);
}

template <typename K, int NW, bool FLIP, int IT, int DB>
__global__ void __launch_bounds__(kBlock) k_radix_hist(const K* keys, int kstride, const unsigned long long* n_ptr, int64_t ncap, int word, int shift, uint32_t* hist) {
  const Grid g_ = hw_grid();
  constexpr int RB = 1 << DB;
  __shared__ uint32_t h[RB];
  for (int i = threadIdx.x; i < RB; i += blockDim.x) h[i] = 0;
  __syncthreads();
  int64_t n = (int64_t)*n_ptr;
  if (n > ncap) n = ncap;
  int64_t begin, end;
  radix_chunk<IT>(g_, n, begin, end);
  for (int64_t i = begin + threadIdx.x; i < end; i += blockDim.x)
    atomicAdd(&h[radix_digit<K, NW, FLIP, DB>(keys + i * kstride, word, shift)], 1u);
  __syncthreads();
  for (int d = threadIdx.x; d < RB; d += blockDim.x) hist[(size_t)d * g_.nb + g_.b] = h[d];
}

// one block per digit: exclusive scan of that digit's per-block counts
__global__ void __launch_bounds__(kBlock) k_radix_scan(uint32_t* hist, int nb, uint32_t* digit_tot) {
  const Grid g_ = hw_grid();
  __shared__ int64_t red[kBlock / kWave];
  uint32_t* row = hist + (size_t)g_.b * nb;
  int per = (nb + kBlock - 1) / kBlock;
  int b0 = threadIdx.x * per;
  int64_t loc = 0;
  for (int i = 0; i < per; ++i)
    if (b0 + i < nb) loc += row[b0 + i];
  int64_t tot;
  int64_t pre = block_exclusive_scan(loc, red, tot);
  for (int i = 0; i < per; ++i)
    if (b0 + i < nb) {
      uint32_t v = row[b0 + i];
      row[b0 + i] = (uint32_t)pre;
      pre += v;
    }
  if (threadIdx.x == 0) digit_tot[g_.b] = (uint32_t)tot;
}

// Stable scatter of one digit, in tiles of IT*kBlock elements: the
// tile is ranked by digit (ballot peers within a wave, LDS counts across waves
// and rounds, in element order), reordered by digit in LDS, then written out
// so that consecutive threads write consecutive positions of each digit's run.
template <typename K, int NW, bool FLIP, int IT, int DB>
__global__ void __launch_bounds__(kBlock) k_radix_scatter(const K* kin, int kstride, const uint32_t* iin, K* kout, uint32_t* iout, const unsigned long long* n_ptr, int64_t ncap, int word, int shift, const uint32_t* hist, const uint32_t* digit_tot) {
  const Grid g_ = hw_grid();
  constexpr int RB = 1 << DB;          // digit values
  constexpr int DPT = RB / kBlock;     // digits owned by each thread (consecutive)
  constexpr int TILE = IT * kBlock;
  __shared__ uint32_t run[RB];     // next global position of each digit (this block)
  __shared__ uint32_t cnt[RB];     // digit counts of the tile so far
  __shared__ uint32_t tstart[RB];  // start of each digit inside the reordered tile
  __shared__ uint32_t wcnt[kBlock / kWave][RB];
  __shared__ K lk[TILE * NW];
  __shared__ uint32_t lv[TILE];
  __shared__ int64_t red[kBlock / kWave];
  const int wv = threadIdx.x / kWave;
  const int d0 = threadIdx.x * DPT;
  {
    // digit bases: exclusive scan of the digit totals in digit order
    int64_t loc = 0;
#pragma unroll
    for (int q = 0; q < DPT; ++q) loc += digit_tot[d0 + q];
    int64_t tot;
    int64_t base = block_exclusive_scan(loc, red, tot);
#pragma unroll
    for (int q = 0; q < DPT; ++q) {
      const int d = d0 + q;
      run[d] = (uint32_t)base + hist[(size_t)d * g_.nb + g_.b];
      base += digit_tot[d];
      cnt[d] = 0;
      for (int w = 0; w < kBlock / kWave; ++w) wcnt[w][d] = 0;
    }
  }
  __syncthreads();
  int64_t n = (int64_t)*n_ptr;
  if (n > ncap) n = ncap;
  int64_t begin, end;
  radix_chunk<IT>(g_, n, begin, end);
  const uint64_t ltmask = lanemask_lt();
  for (int64_t tb = begin; tb < end; tb += TILE) {
    K k[IT][NW];
    uint32_t v[IT], d[IT], off[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      int64_t e = tb + (int64_t)j * kBlock + threadIdx.x;
      bool valid = e < end;
      d[j] = 0;
      v[j] = 0;
      if (valid) {
#pragma unroll
        for (int w = 0; w < NW; ++w) k[j][w] = kin[e * kstride + w];
        v[j] = iin ? iin[e] : (uint32_t)e;
        d[j] = radix_digit<K, NW, FLIP, DB>(k[j], word, shift);
      }
      // lanes of this wave with the same digit, by one ballot per digit bit
      uint64_t peers = __ballot(valid);
#pragma unroll
      for (int bit = 0; bit < DB; ++bit) {
        uint64_t m = __ballot(valid && ((d[j] >> bit) & 1u));
        peers &= ((d[j] >> bit) & 1u) ? m : ~m;
      }
      int rank = popc64(peers & ltmask);
      if (valid && rank == 0) wcnt[wv][d[j]] = (uint32_t)popc64(peers);
      __syncthreads();
      if (valid) {
        uint32_t o = cnt[d[j]] + (uint32_t)rank;
        for (int q = 0; q < wv; ++q) o += wcnt[q][d[j]];
        off[j] = o;
      } else {
        off[j] = 0xFFFFFFFFu;
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < DPT; ++q) {
        const int dd = d0 + q;
        uint32_t sum = 0;
        for (int w = 0; w < kBlock / kWave; ++w) { sum += wcnt[w][dd]; wcnt[w][dd] = 0; }
        cnt[dd] += sum;
      }
      __syncthreads();
    }
    // digit starts inside the tile
    {
      int64_t loc = 0;
#pragma unroll
      for (int q = 0; q < DPT; ++q) loc += cnt[d0 + q];
      int64_t tot;
      int64_t st = block_exclusive_scan(loc, red, tot);
#pragma unroll
      for (int q = 0; q < DPT; ++q) {
        tstart[d0 + q] = (uint32_t)st;
        st += cnt[d0 + q];
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      if (off[j] != 0xFFFFFFFFu) {
        uint32_t lp = tstart[d[j]] + off[j];
#pragma unroll
        for (int w = 0; w < NW; ++w) lk[lp * NW + w] = k[j][w];
        lv[lp] = v[j];
      }
    }
    __syncthreads();
    const int tn = (int)((end - tb) < TILE ? (end - tb) : TILE);
    for (int i = threadIdx.x; i < tn; i += blockDim.x) {
      K kk[NW];
#pragma unroll
      for (int w = 0; w < NW; ++w) kk[w] = lk[i * NW + w];
      uint32_t dd = radix_digit<K, NW, FLIP, DB>(kk, word, shift);
      uint32_t gp = run[dd] + (uint32_t)i - tstart[dd];
#pragma unroll
      for (int w = 0; w < NW; ++w) kout[(size_t)gp * NW + w] = kk[w];
      iout[gp] = lv[i];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < DPT; ++q) {
      run[d0 + q] += cnt[d0 + q];
      cnt[d0 + q] = 0;
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------- merging
// CompressSpawnedList (Annihilation.F90:249-515) + FindResidualParticle
// (:551-634), then AnnihilateSpawnedParts (:965-1352): one wave per spawn bin
// merges the bin's records by determinant in an LDS table, then looks each
// determinant up in the walker hash.
//
// The time goes into random accesses of the walker table (a bucket line and a
// state row per determinant), so the point is to have many in flight and
// nothing else in their way: waves share no barrier, a bin's records are read
// as one contiguous run, and equal determinants meet in LDS instead of in a
// serial run-length loop over gathered records.  Measured against the sort of
// (key, index) pairs and the merge of its runs that it replaced (us per
// iteration, sort + merge before, now): 14e/30o, 1.34e6 spawns 124 + 115, 85;
// 10e/20o, 5.0e5 spawns 48 + 45, 38; 18-site chain, 5.1e5 spawns 109 + 101,
// 39; two-word 26e/40o, 3.0e5 spawns 213 + 41, 39; 1400 spawns 36 + 14, 10.
// Writing the bins costs the spawning kernels 5 to 20 us of that.

// One wave's table of the determinants of a bin.  It is left empty by the
// lanes that take the merged determinants out.
template <int W, int R>
struct MergeTab {
  static constexpr int kSize = R <= 2 ? 128 : 64;
  uint64_t key[kSize * W];
  double sum[kSize * R];
  uint32_t tag[kSize];   // bits 0-15 initiator flags, kTag* bits
  uint8_t list[kSize];   // the slots in use, in order of arrival
};
// an empty slot's key: one-word determinants have at most 63 orbitals
constexpr unsigned long long kTabEmpty = ~0ull;
constexpr uint32_t kTagMulti = 1u << 16;  // more than one record
constexpr uint32_t kTagTaken = 1u << 17;  // two-word keys: claimed,
constexpr uint32_t kTagKey = 1u << 18;    // then key written

// a determinant list (key, S signs, flag) and a list of freed slots, staged
// per wave; each list's place in memory is reserved once per flush.  Rows of
// many signs are not staged: they would take the LDS of the wave's table.
template <int W, int R>
struct WaveStage {
  static constexpr int kCap = R <= 2 ? 128 : 0;
  uint64_t key[kCap ? kCap * W : 1];
  double sgn[kCap ? kCap * R : 1];
  uint32_t flag[kCap ? kCap : 1];
  int32_t freed[128];
};

// the staged determinants (n of them, wave-uniform) to the list at base
template <int W, int R>
__device__ inline void wave_list_write(const WaveStage<W, R>* ws, int n, unsigned long long base, uint64_t* okey,
                                       double* osgn, uint32_t* oflag, int S) {
  for (int i = lane_id(); i < n; i += kWave) {
    const unsigned long long d = base + (unsigned long long)i;
#pragma unroll
    for (int w = 0; w < W; ++w) okey[d * W + w] = ws->key[i * W + w];
    for (int r = 0; r < S; ++r) osgn[d * S + r] = ws->sgn[i * R + r];
    oflag[d] = ws->flag[i];
  }
}
template <int W, int R>
__device__ inline void wave_free_write(const Walk& wk, const WaveStage<W, R>* ws, int n, unsigned long long base) {
  for (int i = lane_id(); i < n; i += kWave)
    wk.freeq[(base + (unsigned long long)i) % (unsigned long long)wk.cap] = ws->freed[i];
}
// the table slot of each todo lane's key (one record per lane): inserted if
// absent.  won: this lane inserted it; -1: the table is full of other keys.
// Every lane probes slot by slot, so either all records of a determinant find
// its slot in a round or none does.
template <int W, int R>
__device__ inline int merge_slot(MergeTab<W, R>* tb, bool todo, const uint64_t* key, uint32_t first, bool& won) {
  constexpr int T = MergeTab<W, R>::kSize;
  int slot = (int)first, found = -1, probes = 0;
  won = false;
  while (__ballot(todo)) {
    if (todo) {
      bool next = false;
      if constexpr (W == 1) {
        const uint64_t old = atomicCAS((unsigned long long*)&tb->key[slot], kTabEmpty, (unsigned long long)key[0]);
        if (old == kTabEmpty || old == key[0]) {
          found = slot;
          won = old == kTabEmpty;
          todo = false;
        } else {
          next = true;
        }
      } else {
        const uint32_t t = __hip_atomic_load(&tb->tag[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (t & kTagKey) {
          if (det_eq<W>(&tb->key[slot * W], key)) {
            found = slot;
            todo = false;
          } else {
            next = true;
          }
        } else if (!(t & kTagTaken) && atomicCAS(&tb->tag[slot], 0u, kTagTaken) == 0u) {
#pragma unroll
          for (int w = 0; w < W; ++w) tb->key[slot * W + w] = key[w];
          wave_sync();
          atomicOr(&tb->tag[slot], kTagKey);
          found = slot;
          won = true;
          todo = false;
        }  // else claimed by a lane of this step, whose key is there at the next
      }
      if (next) {
        slot = (slot + 1) & (T - 1);
        if (++probes == T) todo = false;
      }
    }
  }
  return found;
}

// LIST: only the merged list is written (the explicit-list entry point), the
// bins stay as they are and nothing is counted
template <int W, int R, bool LIST>
__device__ __forceinline__ void k_merge_body(const Grid& g_, const DevSys& s, const Walk& wk, Counters* cnt, double* part, const Bins& bins, uint64_t* n_key, double* n_sgn, uint32_t* n_flag, unsigned long long* n_ctr, const IterParams* prm, bool by_parts) {
  constexpr int kWaves = kBlock / kWave;
  const uint32_t nb = cnt->nbins, cap = cnt->bin_cap, sh = cnt->bin_shift;
  const unsigned long long spawned = LIST ? 0ull : cnt->n_spawned;  // in the same round trip
  if (cnt->halt || g_.b * kWaves >= (int64_t)nb) return;
  // checkValidSpawnedList (fcimc_helper.F90:483-510) stops between spawning
  // and annihilation when the list is past its capacity: no record is merged,
  // the iteration's end reports it.  The bins and the overflow list together
  // hold 2.25 times the capacity, the new list max(capacity,
  // MaxWalkers) rows; past this line the new determinants are no more than
  // the capacity, so that no append needs a bound of its own.
  if (spawned > (unsigned long long)bins.ovf_cap) {
    for (int64_t b = g_.b * blockDim.x + threadIdx.x; b < (int64_t)nb; b += g_.nb * blockDim.x)
      bins.count[(size_t)b << sh] = 0;
    return;
  }
  constexpr int T = MergeTab<W, R>::kSize;
  constexpr int kCap = WaveStage<W, R>::kCap;
  __shared__ MergeTab<W, R> tabs[kWaves];
  __shared__ WaveStage<W, R> stages[kWaves];
  __shared__ double acc_lds[LIST ? 1 : kStatStride];
  __shared__ uint32_t tail_n[kWaves][2];
  __shared__ unsigned long long tail_base[2];
  __shared__ unsigned int blk_unique;
  const uint32_t iter = LIST ? 0u : prm->iter;
  const int wv = threadIdx.x / kWave, lane = lane_id();
  MergeTab<W, R>* tb = &tabs[wv];
  WaveStage<W, R>* ws = &stages[wv];
  BlockStats bs{acc_lds};
  if constexpr (!LIST) bs.zero();
  if (threadIdx.x == 0) blk_unique = 0;
  for (int i = lane; i < T; i += kWave) {
    for (int w = 0; w < W; ++w) tb->key[i * W + w] = kTabEmpty;
    for (int r = 0; r < R; ++r) tb->sum[i * R + r] = 0.0;
    tb->tag[i] = 0;
  }
  __syncthreads();
  const int S = R <= 2 ? R : s.S;
  int n_list = 0, n_free = 0;  // staged (wave-uniform)
  unsigned int uniq = 0;
  double ann[R], st_ab[R], st_an[R], st_rm[R], st_bn[R], d_tot[R], d_norm[R];
  for (int r = 0; r < S; ++r) ann[r] = st_ab[r] = st_an[r] = st_rm[r] = st_bn[r] = d_tot[r] = d_norm[r] = 0.0;
  int d_occ = 0;  // by_parts: changes of the statistics
  // The wave's bins, 64 counters per load; the records of the next bin are on
  // their way while a bin's determinants are looked up.
  const int64_t nwaves = g_.nb * kWaves;
  const int64_t first_seg = g_.b * kWaves + wv;
  uint32_t my_c = 0;  // lane l: records of bin seg0 + l * nwaves
  int64_t seg0 = first_seg - kWave * nwaves;
  uint64_t have = 0;  // bins of this group of 64 not yet taken that hold records
  auto next_bin = [&](int64_t& seg, uint32_t& c_all) -> bool {
    while (have == 0) {
      seg0 += kWave * nwaves;
      if (seg0 >= (int64_t)nb) return false;
      const int64_t mine = seg0 + lane * nwaves;
      my_c = mine < (int64_t)nb ? bins.count[(size_t)mine << sh] : 0u;
      if (!LIST && my_c) bins.count[(size_t)mine << sh] = 0;
      have = __ballot(my_c != 0);
    }
    const int l = ctz64(have);
    have &= have - 1;
    seg = seg0 + l * nwaves;
    c_all = lane_value(my_c, l);
    return true;
  };
  struct Rec {  // a lane's record
    uint64_t key[W];
    double v;
    uint32_t inf;
  };
  auto load_rec = [&](const uint64_t* r, bool on) {
    Rec q;
#pragma unroll
    for (int w = 0; w < W; ++w) q.key[w] = on ? r[w] : 0ull;
    q.v = on ? rec_val<W>(s, r) : 0.0;
    q.inf = on ? rec_info<W>(s, r) : 0u;
    return q;
  };
  int64_t seg = 0, seg_n = 0;
  uint32_t c_all = 0, c_n = 0;
  Rec rec_n;
  bool more = next_bin(seg_n, c_n);
  if (more) rec_n = load_rec(bins.rec + ((size_t)seg_n * cap + lane) * s.rec_words, (uint32_t)lane < (c_n < cap ? c_n : cap));
  while (more) {
    seg = seg_n;
    c_all = c_n;
    const Rec rec_0 = rec_n;
    more = next_bin(seg_n, c_n);
    if (more) rec_n = load_rec(bins.rec + ((size_t)seg_n * cap + lane) * s.rec_words, (uint32_t)lane < (c_n < cap ? c_n : cap));
    const int64_t c = c_all < cap ? c_all : cap;
    const uint32_t over = c_all - (uint32_t)c;  // records in the bin's chains, and in this lane's
    const uint32_t chain_n = (over + kBinChains - 1 - lane) / kBinChains;
    static_assert(kBinChains == kWave, "a chain a lane");
    const int64_t steps = (c + kWave - 1) / kWave, all_steps = steps + (over + kBinChains - 1) / kBinChains;
    uint64_t* seg_rec = bins.rec + (size_t)seg * cap * s.rec_words;
    bool again = false;  // records are left for another round
    do {
      const bool first_round = !again;
      again = false;
      int nu = 0;
      uint32_t link = 0;
      for (int64_t st = 0; st < all_steps; ++st) {
        const int64_t i = st * kWave + lane;
        bool act = i < c;
        uint64_t* rec = seg_rec + i * s.rec_words;
        if (st >= steps) {  // the next record of the lane's chain
          const uint32_t k = (uint32_t)(st - steps);
          act = k < chain_n;
          if (act) link = k == 0 ? bins.head[(size_t)seg * kBinChains + lane] : bins.next[link];
          rec = bins.ovf + (size_t)link * s.rec_words;
        }
        const Rec q = st == 0 && first_round && act && i < c ? rec_0 : load_rec(rec, act);
        const uint64_t* key = q.key;
        const double v = q.v;
        const uint32_t inf = q.inf;
        uint32_t frac = 0;
        if (act) {
          const uint32_t h = bin_hash<W>(key);
          frac = h * nb;  // the position inside the bin
          if (!first_round) act = act && (inf & kInfoLeft);
        }
        bool won;
        const int slot = merge_slot<W, R>(tb, act, key, frac >> (T == 128 ? 25 : 26), won);
        const bool left = act && slot < 0;
        if (left && first_round) rec_mark<W>(s, rec, true);
        if (act && !left && !first_round) rec_mark<W>(s, rec, false);
        again = again || __ballot(left) != 0;
        if (act && !left) {
          // the record joins its determinant, in order of arrival
          const int r = (int)(inf & 0xFFu);
          const double cv = atomicAdd(&tb->sum[slot * R + r], v);
          uint32_t t = won ? 0u : kTagMulti;
          if ((inf & kInfoInit) || (s.t_init && fabs(cv) > 1.e-12 && fabs(v) > 1.e-12)) t |= 1u << r;
          if (t) atomicOr(&tb->tag[slot], t);
          if (cv * v < 0.0) {
            const double x = fabs(cv), y = fabs(v);
            ann[r] += 2.0 * (x < y ? x : y);
          }
        }
        const uint64_t wm = __ballot(won);
        if (won) tb->list[nu + popc64(wm & lanemask_lt())] = (uint8_t)slot;
        nu += popc64(wm);
      }
      wave_sync();
      // the merged determinants, one per lane
      for (int u0 = 0; u0 < nu; u0 += kWave) {
        const bool act = u0 + lane < nu;
        uint64_t key[W];
        double ss[R];
        uint32_t tag = 0;
        if (act) {
          const int slot = tb->list[u0 + lane];
#pragma unroll
          for (int w = 0; w < W; ++w) {
            key[w] = tb->key[slot * W + w];
            tb->key[slot * W + w] = kTabEmpty;
          }
          for (int r = 0; r < S; ++r) {
            ss[r] = tb->sum[slot * R + r];
            tb->sum[slot * R + r] = 0.0;
          }
          tag = tb->tag[slot];
          tb->tag[slot] = 0;
        }
        const bool multi = (tag & kTagMulti) != 0;
        // a single record carries its flag as it is, several only under the
        // initiator approximation
        const uint32_t sflag = multi && !s.t_init ? 0u : tag & 0xFFFFu;
        bool keep = false;
        if (act) {
          double tot = 0.0;
          for (int r = 0; r < S; ++r) tot += fabs(ss[r]);
          keep = multi ? tot > 1.e-12 : !(tot < 1.e-12);
        }
        uniq += (unsigned int)wave_count(keep);
        bool isnew = false, rm = false;
        int64_t pos = -1;
        if (LIST) {
          isnew = keep;
        } else if (keep) {
          int64_t home = find_walker_hash<W>(key, s.rh, s.L) - 1;
          pos = hash_lookup<W>(wk, key, home, cnt);
          if (pos >= 0) {
            double cs[R];  // the walkers there
            double tot = 0.0;
            for (int r = 0; r < S; ++r) { cs[r] = wk.sgn(pos, r); tot += fabs(cs[r]); }
            bool determ = (wk.flags(pos) & kFlagCore) != 0;
            if (tot >= 1.e-12 || determ) {
              for (int r = 0; r < S; ++r) {
                double prod = cs[r] * ss[r];
                if (fabs(cs[r]) < 1.0e-12 && s.t_init && !((sflag >> r) & 1u) && !determ) {
                  st_ab[r] += fabs(ss[r]);
                  ss[r] = 0.0;
                }
                if (prod < 0.0) {
                  double x = fabs(cs[r]), y = fabs(ss[r]);
                  st_an[r] += 2.0 * (x < y ? x : y);
                }
              }
              bool occ = false;
              for (int r = 0; r < S; ++r) {
                if (by_parts) {
                  d_tot[r] -= fabs(cs[r]);
                  d_norm[r] -= cs[r] * cs[r];
                  if (det_eq<W>(key, s.ref)) atomicAdd(&bs.acc[soff(F_INSTHF, r)], ss[r]);
                }
                cs[r] = ss[r] + cs[r];
                wk.sgn(pos, r) = cs[r];
                occ = occ || !(fabs(cs[r]) < 1.e-12);
              }
              rm = !determ && !occ;
              if (by_parts) {
                if (rm) d_occ -= 1;
                for (int r = 0; r < S; ++r)
                  if (!rm) {
                    d_tot[r] += fabs(cs[r]);
                    d_norm[r] += cs[r] * cs[r];
                  }
              }
            }
          } else {
            if (s.t_init)
              for (int r = 0; r < S; ++r)
                if (!((sflag >> r) & 1u)) {
                  st_ab[r] += fabs(ss[r]);
                  ss[r] = 0.0;
                }
            bool occ = false;
            for (int r = 0; r < S; ++r) occ = occ || !(fabs(ss[r]) < 1.e-12);
            if (occ) {
              // stochRoundSpawn (Annihilation.F90:1354-1418)
              double thr = s.occ_thresh;
              for (int r = 0; r < S; ++r) {
                if (fabs(ss[r]) > 1.e-12 && fabs(ss[r]) < thr) {
                  double pRemove = 1.0 - fabs(ss[r]) / thr;
                  double u, dummy;
                  draw2<W>(s.seed, key, iter, r, 0, 4, u, dummy);
                  if (pRemove > u) {
                    st_rm[r] += fabs(ss[r]);
                    ss[r] = 0.0;
                  } else {
                    st_bn[r] += thr - fabs(ss[r]);
                    ss[r] = ss[r] >= 0.0 ? thr : -thr;
                  }
                }
              }
              occ = false;
              for (int r = 0; r < S; ++r) occ = occ || !(fabs(ss[r]) < 1.e-12);
              isnew = occ;
              if (by_parts && isnew) {
                d_occ += 1;
                for (int r = 0; r < S; ++r) {
                  d_tot[r] += fabs(ss[r]);
                  d_norm[r] += ss[r] * ss[r];
                  if (det_eq<W>(key, s.ref)) atomicAdd(&bs.acc[soff(F_INSTHF, r)], ss[r]);
                }
              }
            }
          }
          if (rm) {  // RemoveHashDet (load_balancer.fpp:631-644): the entry becomes a tombstone
            const int64_t hp = wk.hpos(pos);
            int32_t* sl = (int32_t*)(wk.htab + (size_t)(hp >> 2) * 8 * W + 4 * W);
            sl[hp & 3] = kSlotTomb;
            wk.flags(pos) |= kFlagRemoved;
          }
        }
        const uint64_t nm = __ballot(isnew), fm = __ballot(rm);
        if (nm && kCap == 0) {
          const unsigned long long q = wave_reserve(n_ctr, popc64(nm)) + (unsigned long long)popc64(nm & lanemask_lt());
          if (isnew) {
#pragma unroll
            for (int w = 0; w < W; ++w) n_key[q * W + w] = key[w];
            for (int r = 0; r < S; ++r) n_sgn[q * S + r] = ss[r];
            n_flag[q] = sflag;
          }
        } else if (nm) {
          if (n_list + popc64(nm) > kCap) {
            wave_sync();
            wave_list_write<W, R>(ws, n_list, wave_reserve(n_ctr, n_list), n_key, n_sgn, n_flag, S);
            wave_sync();
            n_list = 0;
          }
          if (isnew) {
            const int q = n_list + popc64(nm & lanemask_lt());
#pragma unroll
            for (int w = 0; w < W; ++w) ws->key[q * W + w] = key[w];
            for (int r = 0; r < S; ++r) ws->sgn[q * R + r] = ss[r];
            ws->flag[q] = sflag;
          }
          n_list += popc64(nm);
        }
        if (fm) {
          if (n_free + popc64(fm) > 128) {
            wave_sync();
            wave_free_write<W, R>(wk, ws, n_free, wave_reserve(&cnt->free_tail, n_free));
            wave_sync();
            n_free = 0;
          }
          if (rm) ws->freed[n_free + popc64(fm & lanemask_lt())] = (int32_t)pos;
          n_free += popc64(fm);
        }
      }
      wave_sync();
    } while (again);
  }
  // what is still staged: one reservation per block
  if (lane == 0) {
    tail_n[wv][0] = (uint32_t)n_list;
    tail_n[wv][1] = (uint32_t)n_free;
    if (uniq) atomicAdd(&blk_unique, uniq);
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    unsigned int n = 0;
    for (int q = 0; q < kWaves; ++q) n += tail_n[q][threadIdx.x];
    if (n) tail_base[threadIdx.x] = atomicAdd(threadIdx.x ? &cnt->free_tail : n_ctr, (unsigned long long)n);
  }
  __syncthreads();
  unsigned int before[2] = {0, 0};
  for (int q = 0; q < wv; ++q) {
    before[0] += tail_n[q][0];
    before[1] += tail_n[q][1];
  }
  wave_list_write<W, R>(ws, n_list, tail_base[0] + before[0], n_key, n_sgn, n_flag, S);
  if constexpr (!LIST) {
    wave_free_write<W, R>(wk, ws, n_free, tail_base[1] + before[1]);
    for (int r = 0; r < S; ++r) {
      bs.add(soff(F_NABORTED, r), st_ab[r]);
      bs.add(soff(F_NANNIHIL, r), st_an[r] + ann[r]);
      bs.add(soff(F_NREMOVED, r), st_rm[r]);
      bs.add(soff(F_NBORN, r), st_bn[r]);
      if (by_parts) {
        bs.add(soff(F_TOTPARTS, r), d_tot[r]);
        bs.add(soff(F_NORMSQ, r), d_norm[r]);
      }
    }
    if (by_parts) bs.add(X_NOCC, (double)d_occ);
    if (threadIdx.x == 0 && blk_unique)
      atomicAdd(&cnt->uniq_part[g_.b % Counters::kSpread].v, (unsigned long long)blk_unique);
    bs.flush(part, g_.b);
  }
}
template <int W, int R>
__global__ void __launch_bounds__(kBlock, R <= 2 && W == 1 ? 5 : 1) k_merge_annihilate(DevSys s, Walk wk, Counters* cnt, double* part, Bins bins, uint64_t* n_key, double* n_sgn, uint32_t* n_flag, const IterParams* prm, int by_parts) {
  k_merge_body<W, R, false>(hw_grid(), s, wk, cnt, part, bins, n_key, n_sgn, n_flag, &cnt->n_new, prm, by_parts != 0);
}
template <int W, int R>
__global__ void __launch_bounds__(kBlock) k_merge_list(DevSys s, Walk wk, Counters* cnt, Bins bins, uint64_t* u_key, double* u_sgn, uint32_t* u_flag, unsigned long long* u_count) {
  k_merge_body<W, R, true>(hw_grid(), s, wk, cnt, nullptr, bins, u_key, u_sgn, u_flag, u_count, nullptr, false);
}

// ------------------------------------------------------ semistochastic core
// Core amplitudes before the projection (no death acts on core dets, so the
// signs after the prepass are the iteration's starting amplitudes):
// x[i * xs + r] = the amplitude of core det i, replica r (xs = S for an
// engine's own vector; a wider stride for a vector shared by a batch group)
template <int R>
__device__ __forceinline__ void k_core_gather_body(const Grid& g_, const int64_t* core_slot, const Walk& wk, int S, int64_t ncore, double* x, int xs) {
  for (int64_t i = (int64_t)g_.b * blockDim.x + threadIdx.x; i < ncore; i += (int64_t)g_.nb * blockDim.x)
    for (int r = 0; r < S; ++r) x[i * xs + r] = wk.sgn(core_slot[i], r);
}
template <int R>
__global__ void __launch_bounds__(kBlock) k_core_gather(const int64_t* core_slot, Walk wk, int S, int64_t ncore, double* x) {
  k_core_gather_body<R>(hw_grid(), core_slot, wk, S, ncore, x, S);
}

// determ_projection (semi_stoch_procs.F90:105-241), one wave per core row:
// lane l sums the row's nonzeros q = l, l+64, ... as acc = acc - H*x, the
// butterfly acc = acc + shfl_xor(acc, o) for o = 32..1 combines the lanes, and
// y = (acc + S*x_i) * tau.  The CPU restatement sums in exactly this order.
template <int R, typename VT>
__device__ __forceinline__ void k_core_spmv_body(const Grid& g_, const int64_t* rowptr, const int32_t* cols, const VT* vals, const double* x, double* y, int64_t ncore, int S, const IterParams* prm) {
  const double tau = prm->tau;
  const double* sftv = prm->sft.v;
  const int lane = lane_id();
  const int64_t nwaves = (int64_t)g_.nb * blockDim.x / kWave;
  for (int64_t i = ((int64_t)g_.b * blockDim.x + threadIdx.x) / kWave; i < ncore; i += nwaves) {
    double acc[R];
    for (int r = 0; r < S; ++r) acc[r] = 0.0;
    const int64_t e = rowptr[i + 1];
    for (int64_t q = rowptr[i] + lane; q < e; q += kWave) {
      double v = (double)vals[q];
      const double* xc = x + (size_t)cols[q] * S;
      for (int r = 0; r < S; ++r) acc[r] = acc[r] - v * xc[r];
    }
    for (int r = 0; r < S; ++r) {
#pragma unroll
      for (int o = kWave / 2; o > 0; o >>= 1) acc[r] = acc[r] + __shfl_xor(acc[r], o);
    }
    if (lane == 0)
      for (int r = 0; r < S; ++r) y[i * S + r] = (acc[r] + sftv[r] * x[i * S + r]) * tau;
  }
}
template <int R, typename VT>
__global__ void __launch_bounds__(kBlock) k_core_spmv(const int64_t* rowptr, const int32_t* cols, const VT* vals, const double* x, double* y, int64_t ncore, int S, const IterParams* prm) {
  k_core_spmv_body<R, VT>(hw_grid(), rowptr, cols, vals, x, y, ncore, S, prm);
}

// deterministic_annihilation (Annihilation.F90:930-963): the projected
// amplitudes join the core dets' signs (births and annihilations counted)
template <int R>
__device__ __forceinline__ void k_core_apply_body(const Grid& g_, const DevSys& s, const Walk& wk, const Counters* cnt, const int64_t* core_slot, const double* y, int64_t ncore, double* part, int ys) {
  if (cnt->halt) return;
  __shared__ double acc_lds[kStatStride];
  BlockStats bs{acc_lds};
  bs.zero();
  const int S = R <= 2 ? R : s.S;
  LaneSum<R> born, ann;
  int64_t trips = grid_trips(g_, ncore);
  for (int64_t t = 0; t < trips; ++t) {
    int64_t i = grid_elem(g_, t);
    bool act = i < ncore;
    int64_t slot = act ? core_slot[i] : 0;
    for (int r = 0; r < S; ++r) {
      double b = 0.0, a = 0.0;
      if (act) {
        double yy = y[i * ys + r], c = wk.sgn(slot, r);
        wk.sgn(slot, r) = yy + c;
        b = fabs(yy);
        if (c * yy < 0.0) {
          double x1 = fabs(c), x2 = fabs(yy);
          a = 2.0 * (x1 < x2 ? x1 : x2);
        }
      }
      born.add(bs, soff(F_NBORN, r), b);
      ann.add(bs, soff(F_NANNIHIL, r), a);
    }
  }
  born.done(bs, soff(F_NBORN, 0));
  ann.done(bs, soff(F_NANNIHIL, 0));
  bs.flush(part, g_.b);
}
template <int R>
__global__ void __launch_bounds__(kBlock) k_core_apply(DevSys s, Walk wk, const Counters* cnt, const int64_t* core_slot, const double* y, int64_t ncore, double* part) {
  k_core_apply_body<R>(hw_grid(), s, wk, cnt, core_slot, y, ncore, part, R <= 2 ? R : s.S);
}

// core Hamiltonian rows (calc_determ_hamil, fast_determ_hamil.F90:892-1548):
// one wave per row i scans every core det j in ascending order; H_ij for
// connected pairs (diagonal H_ii - Hii), off-diagonal zeros dropped.  Pass 0
// counts, pass 1 writes columns and values at rowptr[i].
template <int W, typename VT>
__device__ __forceinline__ void k_core_rows_body(const Grid& g_, const DevSys& s, const uint64_t* keys, int64_t ncore, int pass, int64_t* count, const int64_t* rowptr, int32_t* cols, VT* vals) {
  const int lane = lane_id();
  const int64_t nwaves = (int64_t)g_.nb * blockDim.x / kWave;
  for (int64_t i = ((int64_t)g_.b * blockDim.x + threadIdx.x) / kWave; i < ncore; i += nwaves) {
    const uint64_t* di = keys + i * W;
    int64_t base = pass ? rowptr[i] : 0;
    for (int64_t j0 = 0; j0 < ncore; j0 += kWave) {
      int64_t j = j0 + lane;
      bool keep = false;
      double h = 0.0;
      if (j < ncore) {
        const uint64_t* dj = keys + j * W;
        if (excit_level<W>(di, dj) <= 2) {
          h = (i == j) ? diag_helement<W>(s, di) - s.hii : helement_pair<W>(s, di, dj);
          keep = (i == j) || h != 0.0;
        }
      }
      uint64_t m = __ballot(keep);
      if (pass && keep) {
        int64_t q = base + popc64(m & lanemask_lt());
        cols[q] = (int32_t)j;
        vals[q] = (VT)h;
      }
      base += popc64(m);
    }
    if (!pass && lane == 0) count[i] = base;
  }
}
template <int W, typename VT>
__global__ void __launch_bounds__(kBlock) k_core_rows(DevSys s, const uint64_t* keys, int64_t ncore, int pass, int64_t* count, const int64_t* rowptr, int32_t* cols, VT* vals) {
  k_core_rows_body<W, VT>(hw_grid(), s, keys, ncore, pass, count, rowptr, cols, vals);
}

// place the core dets: resident ones get the core (and initiator) flags and
// their slot; absent ones are appended to the new list with zero signs
template <int W>
__device__ __forceinline__ void k_core_place_body(const Grid& g_, const DevSys& s, const Walk& wk, Counters* cnt, const uint64_t* keys, int64_t ncore, uint32_t cflags, int64_t* core_slot, uint64_t* n_key, double* n_sgn, uint32_t* n_flag) {
  const int S = s.S;
  for (int64_t i = (int64_t)g_.b * blockDim.x + threadIdx.x; i < ncore; i += (int64_t)g_.nb * blockDim.x) {
    const uint64_t* d = keys + i * W;
    int64_t home = find_walker_hash<W>(d, s.rh, s.L) - 1;
    int64_t pos = hash_lookup<W>(wk, d, home, cnt);
    if (pos >= 0) {
      wk.flags(pos) |= cflags;
      core_slot[i] = pos;
    } else {
      unsigned long long q = atomicAdd(&cnt->n_new, 1ull);
#pragma unroll
      for (int w = 0; w < W; ++w) n_key[q * W + w] = d[w];
      for (int r = 0; r < S; ++r) n_sgn[q * S + r] = 0.0;
      n_flag[q] = cflags;
      core_slot[i] = -1;
    }
  }
}
template <int W>
__global__ void __launch_bounds__(kBlock) k_core_place(DevSys s, Walk wk, Counters* cnt, const uint64_t* keys, int64_t ncore, uint32_t cflags, int64_t* core_slot, uint64_t* n_key, double* n_sgn, uint32_t* n_flag) {
  k_core_place_body<W>(hw_grid(), s, wk, cnt, keys, ncore, cflags, core_slot, n_key, n_sgn, n_flag);
}

// Diagonal elements of new molecular determinants by a group of G lanes.
// sltcnd_0's sums run over nel (nel - 1) / 2 pairs; on one lane their loads
// were about 50 dependent round trips at 14 electrons and 150 at 26, and a
// list of new determinants is too short to hide them.  Here the rows of pairs
// are spread over the group: lane g sums the Coulomb terms of the electrons
// g, g + G, ... with the electrons above them (each row's sum is its own in
// sltcnd_0 too) and leaves the exchange terms, whose order the sum fixes, in
// LDS; then three lanes add the one-electron terms, the rows and the exchange
// terms, each list in sltcnd_0's order, so the value is sltcnd_0's to the last
// bit.
// LDS per determinant: nel one-electron terms, nel rows, the same-spin pairs.
__host__ __device__ inline int diag_pairs(int na, int nb) { return na * (na - 1) / 2 + nb * (nb - 1) / 2; }
__host__ __device__ inline int diag_lds(const DevSys& s) {  // doubles
  return 2 * s.nel + diag_pairs(s.nalpha_ref, s.nbeta_ref);
}
template <int W, int G>
__device__ inline double diag_group(const DevSys& s, const uint64_t* d, int g, double* lds) {
  const uint64_t kA = 0xAAAAAAAAAAAAAAAAull;
  int na = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) na += popc64(d[w] & kA);
  const int nel = s.nel, nb = nel - na, np = diag_pairs(na, nb);
  const bool fits = np <= diag_pairs(s.nalpha_ref, s.nbeta_ref);  // else other spin counts than the run's
  double *sing = lds, *rows = lds + nel, *ex = lds + 2 * nel;
  wave_sync();
  if (fits) {
    for (int e = g; e < nel; e += G) {
      const int o = select_orb<W>(d, ~0ull, e + 1), wi = (o - 1) >> 6, bit = (o - 1) & 63;
      const bool beta = is_beta(o);
      sing[e] = s.tmat[(size_t)(o - 1) * (s.nbasis + 1)];
      // same-spin pairs of the electrons below this one
      int a = 0;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const uint64_t below = w < wi ? ~0ull : w == wi ? (1ull << bit) - 1ull : 0ull;
        a += popc64(d[w] & below & kA);
      }
      const int b = e - a;
      double* k = ex + a * (na - 1) - a * (a - 1) / 2 + b * (nb - 1) - b * (b - 1) / 2;
      const double2* row = (const double2*)(s.jk0 + 2 * (size_t)(spat(o) - 1) * s.nsp);
      double t = 0.0;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        uint64_t x = w < wi ? 0ull : w > wi ? d[w] : bit == 63 ? 0ull : d[w] & (~0ull << (bit + 1));
        while (x) {  // eight pairs' (J, K) per round trip
          constexpr int N = 8;
          int oj[N], n = 0;
          double2 v[N];
#pragma unroll
          for (int q = 0; q < N; ++q)
            if (x) {
              oj[q] = 64 * w + ctz64(x) + 1;
              x &= x - 1;
              n = q + 1;
            }
#pragma unroll
          for (int q = 0; q < N; ++q) v[q] = q < n ? row[spat(oj[q]) - 1] : double2{0.0, 0.0};
#pragma unroll
          for (int q = 0; q < N; ++q)
            if (q < n) {
              t += v[q].x;
              if (is_beta(oj[q]) == beta) *k++ = -v[q].y;
            }
        }
      }
      rows[e] = t;
    }
  }
  wave_sync();
  if (!fits) return diag_helement<W>(s, d);  // (group-uniform)
  static_assert(G >= 3, "three lanes add the three lists");
  const double* list = g == 0 ? sing : g == 1 ? rows : ex;
  const int n = g == 0 ? nel : g == 1 ? nel - 1 : g == 2 ? np : 0;
  double sum = 0.0;
  for (int p = 0; p < n; p += 8) {
    double v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = p + q < n ? list[p + q] : 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (p + q < n) sum += v[q];
  }
  const int lead = lane_id() - g;
  const double hel_sing = __shfl(sum, lead), hel_doub = __shfl(sum, lead + 1), hel_tmp = __shfl(sum, lead + 2);
  return hel_doub + hel_tmp + hel_sing + s.ecore;
}

// AddNewHashDet (load_balancer.fpp:514-629) for the new list.  A wave takes D
// determinants, one lane each for the hash entry and the walker row.  On a
// short list (up to kShortList) the diagonal elements follow, by
// groups of G lanes: its time is the length of one wave's instruction stream,
// which the groups shorten (us per iteration, one lane before: 10e/20o, 700
// new determinants 24 -> 13; two-word 26e/40o, 2.8e4 92 -> 49).  A long list
// fills the lanes and is bound by issue and L1 gathers, which groups make
// worse (14e/30o, 1.3e5: 55 with one lane, 56 with four, 102 with 16), so
// there the lane sums its own.  The line between them: at 32000 determinants
// the groups take 21 us against 22 at 10 electrons, 25 against 32 at 14 and 55
// against 115 at 26 (one lane takes 23, 31 and 120 for 33000), so it is right
// for 10 electrons and early for 26.  G is 16, or 64 when a block's LDS does
// not hold 16 determinants' terms; 1 for the lattice.
// A determinant that is refused, in an iteration that ends in an error, has
// its list entry marked (kFlagRemoved).
constexpr int64_t kShortList = 32768;
template <int W, int R, int G>
__device__ __forceinline__ void k_insert_body(const Grid& g_, const DevSys& s, const Walk& wk, Counters* cnt, const uint64_t* n_key, const double* n_sgn, uint32_t* n_flag, const unsigned long long* n_ptr, double* lds) {
  if (cnt->halt) return;
  const int S = R <= 2 ? R : s.S;
  int64_t nn = (int64_t)*n_ptr;
  // new det i takes the i-th queued free slot, past the queue a fresh slot
  // at the end of the table: positions follow from i, no atomics
  const unsigned long long head = cnt->free_head;
  const unsigned long long tail = cnt->free_tail;
  const int64_t avail = (int64_t)(tail - head);
  const int64_t ns0 = (int64_t)cnt->nslots;
  if (g_.b == 0 && threadIdx.x == 0) cnt->free_tail_ins = tail;  // for the slot bookkeeping
  // MaxWalkers would be passed (AddNewHashDet's stop, load_balancer.fpp:540-544):
  // no new determinant is placed, so the walker list the halted engine keeps
  // does not depend on the order of the new list
  if (ns0 + (nn > avail ? nn - avail : 0) > wk.cap) {
    if (g_.b == 0 && threadIdx.x == 0) {
      atomicOr(&cnt->err, 1u << NGPU_ERR_WALKERS_FULL);
      cnt->n_fail = (unsigned long long)nn;
      cnt->ins_refused = 1u;
    }
    return;
  }
  unsigned long long my_reused = 0;
  constexpr int kWaves = kBlock / kWave;
  const int lane = lane_id(), wv = threadIdx.x / kWave;
  const int64_t nwaves = g_.nb * kWaves;
  // short: at most kShortList determinants on the chip, the engine's share of
  // them by its share of a batch launch
  const bool group = G > 1 && nn * (int64_t)gridDim.x <= kShortList * g_.nb;
  constexpr int kPer = kWave / G;  // determinants of a wave's group step
  int64_t D = kWave;
  if (group) {
    D = ((nn + nwaves - 1) / nwaves + kPer - 1) / kPer * kPer;
    if (D > kWave) D = kWave;
  }
  if (g_.b * kWaves * D >= nn) return;  // no determinant for this block
  for (int64_t base = (g_.b * kWaves + wv) * D; base < nn; base += nwaves * D) {
    const int64_t i = base + lane;
    const bool act = lane < D && i < nn;
    int64_t slot = -1;  // the determinant's row; -1: none
    uint64_t key[W];
#pragma unroll
    for (int w = 0; w < W; ++w) key[w] = act ? n_key[i * W + w] : s.ref[w];
    if (act) {
      slot = i < avail ? wk.freeq[(head + (unsigned long long)i) % (unsigned long long)wk.cap] : ns0 + (i - avail);
      int64_t hp = -1;
      if (slot >= wk.cap) {
        atomicOr(&cnt->err, 1u << NGPU_ERR_WALKERS_FULL);
        atomicAdd(&cnt->n_fail, 1ull);
        n_flag[i] = kFlagRemoved;
        slot = -1;
      } else {
        int64_t home = find_walker_hash<W>(key, s.rh, s.L) - 1;
        bool reused = false;
        hp = hash_insert<W>(wk, key, home, (int32_t)slot, reused);
        my_reused += reused ? 1 : 0;
        if (hp < 0) {
          atomicOr(&cnt->err, 1u << NGPU_ERR_HASH_FULL);
          atomicAdd(&cnt->n_fail, 1ull);
          wk.flags(slot) = kFlagRemoved;
          n_flag[i] = kFlagRemoved;
          slot = -1;
        }
      }
      if (slot >= 0) {
#pragma unroll
        for (int w = 0; w < W; ++w) wk.keys[slot * W + w] = key[w];
        for (int r = 0; r < S; ++r) wk.sgn(slot, r) = n_sgn[i * S + r];
        wk.flags(slot) = n_flag[i] & ~kFlagRemoved;
        wk.hpos(slot) = hp;
        wk.offdiagH[slot] = offdiag_helement<W>(s, key);
        if (!group) wk.diagH[slot] = diag_helement<W>(s, key) - s.hii;
      }
    }
    if constexpr (G > 1) {
      const int n_here = group ? (int)(nn - base < D ? nn - base : D) : 0;
      for (int r = 0; r < n_here; r += kPer) {  // wave-uniform
        const int src = r + lane / G;           // the lane that holds this group's determinant
        uint64_t k[W];
#pragma unroll
        for (int w = 0; w < W; ++w) k[w] = __shfl((unsigned long long)key[w], src);
        const int64_t row = __shfl((long long)slot, src);
        const double d = diag_group<W, G>(s, k, lane % G, lds + (size_t)(threadIdx.x / G) * diag_lds(s));
        if (lane % G == 0 && row >= 0) wk.diagH[row] = d - s.hii;
      }
    }
  }
  // one no-return atomic per wave that reused entries
  // one add per block, spread over kSpread lines
  __shared__ unsigned int blk_reused;
  if (threadIdx.x == 0) blk_reused = 0;
  __syncthreads();
  unsigned int c = (unsigned int)wave_sum((double)my_reused);
  if (c && lane_id() == 0) atomicAdd(&blk_reused, c);
  __syncthreads();
  if (threadIdx.x == 0 && blk_reused)
    atomicAdd(&cnt->reuse_part[g_.b % Counters::kSpread].v, (unsigned long long)blk_reused);
}
template <int W, int R, int G>
__global__ void __launch_bounds__(kBlock) k_insert(DevSys s, Walk wk, Counters* cnt, const uint64_t* n_key, const double* n_sgn, uint32_t* n_flag, const unsigned long long* n_ptr) {
  extern __shared__ double insert_dyn[];
  k_insert_body<W, R, G>(hw_grid(), s, wk, cnt, n_key, n_sgn, n_flag, n_ptr, insert_dyn);
}

// bookkeeping of k_insert: queued slots used, fresh slots appended (beyond
// the capacity refused), live entries added
// slots after k_insert placed nn new determinants: the first ones took the
// queued free slots, the rest fresh slots at the end of the table.  A pure
// function of counters that nothing changes between k_insert and the
// bookkeeping, so k_stats evaluates it for its loop bound while the
// bookkeeping (k_end_iter, or k_post_insert on the set-up paths) applies it.
__device__ inline void slots_after_insert(const Counters* cnt, unsigned long long nn, int64_t cap,
                                          unsigned long long& used, unsigned long long& ns) {
  if (cnt->ins_refused) {  // nothing was placed
    used = 0;
    ns = cnt->nslots;
    return;
  }
  unsigned long long avail = cnt->free_tail_ins - cnt->free_head;
  used = nn < avail ? nn : avail;
  ns = cnt->nslots + (nn - used);
  if (ns > (unsigned long long)cap) ns = (unsigned long long)cap;
}
// reused: tombstone entries the inserts took (the sum of reuse_part, which
// the caller has emptied)
__device__ inline void post_insert(Counters* cnt, unsigned long long nn, int64_t cap, unsigned long long reused) {
  unsigned long long used, ns;
  slots_after_insert(cnt, nn, cap, used, ns);
  cnt->free_head += used;
  cnt->nslots = ns;
  cnt->n_live += nn - cnt->n_fail;
  cnt->n_tomb -= reused;
}
__global__ void k_post_insert(Counters* cnt, const unsigned long long* n_ptr, int64_t cap) {
  unsigned long long reused = 0;
  for (int q = 0; q < Counters::kSpread; ++q) {
    reused += cnt->reuse_part[q].v;
    cnt->reuse_part[q].v = 0;
  }
  post_insert(cnt, *n_ptr, cap, reused);
}

// CalcHashTableStats (load_balancer.fpp:646-805)
template <int W, int R>
__device__ __forceinline__ void k_stats_body(const Grid& g_, const DevSys& s, const Walk& wk, Counters* cnt, double* part, const IterParams* prm) {
  if (cnt->halt) return;
  unsigned long long used, ns;
  slots_after_insert(cnt, cnt->n_new, wk.cap, used, ns);  // the bookkeeping applies it later
  const int64_t nslots = (int64_t)ns;
  if (g_.b * blockDim.x >= nslots) return;  // no slots for this block
  const uint32_t iter = prm->iter;
  __shared__ double acc_lds[kStatStride];
  __shared__ FreeStage fs;
  BlockStats bs{acc_lds};
  bs.zero();
  stage_init(&fs.st);
  const int S = R <= 2 ? R : s.S;
  unsigned long long my_occ = 0;
  double tp[R], nq[R], rmv[R], bn[R];
  for (int r = 0; r < S; ++r) tp[r] = nq[r] = rmv[r] = bn[r] = 0.0;
  int64_t trips = grid_trips(g_, nslots);
  for (int64_t t = 0; t < trips; ++t) {
    int64_t slot = grid_elem(g_, t);
    bool rm = false;
    // the slot's flags, signs and determinant in one round trip to memory
    // (lanes past the table load slot 0, which exists when any lane runs)
    const int64_t ls = slot < nslots ? slot : 0;
    const uint32_t f_ld = wk.flags(ls);
    double s_ld[R];
    uint64_t k_ld[W];
    for (int r = 0; r < S; ++r) s_ld[r] = wk.sgn(ls, r);
#pragma unroll
    for (int w = 0; w < W; ++w) k_ld[w] = wk.keys[ls * W + w];
    if (slot < nslots) {
      uint32_t f = f_ld;
      if (!(f & kFlagRemoved)) {
        bool determ = (f & kFlagCore) != 0;
        double sg[R];
        bool occ = false;
        for (int r = 0; r < S; ++r) { sg[r] = s_ld[r]; occ = occ || !(fabs(sg[r]) < 1.e-12); }
        if (occ || determ) {
          uint64_t key[W];
#pragma unroll
          for (int w = 0; w < W; ++w) key[w] = k_ld[w];
          if (s.t_real) {
            double thr = s.occ_thresh;
            bool changed = false;
            for (int r = 0; r < S; ++r) {
              if (!determ && fabs(sg[r]) > 1.e-12 && fabs(sg[r]) < thr) {
                double pRemove = (thr - fabs(sg[r])) / thr;
                double u, dummy;
                draw2<W>(s.seed, key, iter, r, 0, 5, u, dummy);
                if (pRemove > u) {
                  rmv[r] += fabs(sg[r]);
                  sg[r] = 0.0;
                } else {
                  bn[r] += thr - fabs(sg[r]);
                  sg[r] = sg[r] >= 0.0 ? thr : -thr;
                }
                changed = true;
              }
            }
            if (changed) {
              occ = false;
              for (int r = 0; r < S; ++r) { wk.sgn(slot, r) = sg[r]; occ = occ || !(fabs(sg[r]) < 1.e-12); }
              rm = !occ && !determ;
            }
          }
          if (!rm) {
            my_occ++;
            for (int r = 0; r < S; ++r) {
              tp[r] += fabs(sg[r]);
              nq[r] += sg[r] * sg[r];
            }
            if (det_eq<W>(key, s.ref))
              for (int r = 0; r < S; ++r) bs.acc[soff(F_INSTHF, r)] = sg[r];
          }
        }
      }
    }
    remove_dets<W>(wk, &fs, rm, slot);
    free_flush(wk, cnt, &fs, false);
  }
  free_flush(wk, cnt, &fs, true);
  for (int r = 0; r < S; ++r) {
    bs.add(soff(F_TOTPARTS, r), tp[r]);
    bs.add(soff(F_NORMSQ, r), nq[r]);
    bs.add(soff(F_NREMOVED, r), rmv[r]);
    bs.add(soff(F_NBORN, r), bn[r]);
  }
  bs.add(X_NOCC, (double)my_occ);
  bs.flush(part, g_.b);
}
template <int W, int R>
__global__ void __launch_bounds__(kBlock) k_stats(DevSys s, Walk wk, Counters* cnt, double* part, const IterParams* prm) {
  k_stats_body<W, R>(hw_grid(), s, wk, cnt, part, prm);
}

// ---------------------------------------------------------- hash upkeep
// Tombstones left by removals are reclaimed by rebuilding the index in place
// once live + tombstone entries pass 60% of the entries and tombstones alone
// pass 10%; more than 80% live
// entries is a capacity error (MEMORYFACHASH too small), reported instead of
// letting probe sequences grow without bound.
// the table is rebuilt once live + tombstone entries pass this share (and
// tombstones pass 10 %): later rebuilds against longer probe sequences
constexpr unsigned long long kRebuildUsedPct = 60;

// the rebuild decision, a pure function of the counters after the removals
// since the last accounting (nothing changes them between the removing
// kernels and the accounting), so the in-place clear, refill and bookkeeping
// kernels each evaluate it; an iteration's accounting publishes it for the
// next iteration instead
__device__ inline bool hash_rebuild_due(const Counters* cnt, int64_t entries) {
  unsigned long long removed = cnt->free_tail - cnt->free_tail0;  // each left a tombstone
  unsigned long long live = cnt->n_live - removed, tomb = cnt->n_tomb + removed;
  return (live + tomb) * 100ull > (unsigned long long)entries * kRebuildUsedPct &&
         tomb * 10ull > (unsigned long long)entries;
}

// bookkeeping of the removals since the last call and of an in-place rebuild
// by k_hash_clear/k_hash_refill (one thread; set-up paths)
__device__ inline void hash_done(Counters* cnt, int64_t entries) {
  bool rebuilt = hash_rebuild_due(cnt, entries);
  if (rebuilt) cnt->n_rebuilds += 1;
  unsigned long long removed = cnt->free_tail - cnt->free_tail0;
  cnt->n_live -= removed;
  cnt->n_tomb = rebuilt ? 0ull : cnt->n_tomb + removed;
  cnt->free_tail0 = cnt->free_tail;
  cnt->rebuild = 0;
  if (cnt->n_live * 10ull > (unsigned long long)entries * 8ull) cnt->err |= 1u << NGPU_ERR_HASH_FULL;
}

// end of an iteration (one thread): the removals' tombstones are counted, and
// a rebuild that has become due is left to the next iteration's prepass and
// attempt scan, which run before any other access to the table
__device__ inline void hash_account(Counters* cnt, int64_t entries) {
  unsigned long long removed = cnt->free_tail - cnt->free_tail0;
  cnt->n_live -= removed;
  // after a rebuild in this iteration only the removals after the attempt
  // scan's refill left tombstones; the refill zeroed n_tomb
  cnt->n_tomb += cnt->rebuilt ? removed - cnt->rm_pre : removed;
  cnt->rebuilt = 0;
  cnt->free_tail0 = cnt->free_tail;
  cnt->rebuild = hash_rebuild_due(cnt, entries) ? 1u : 0u;
  if (cnt->n_live * 10ull > (unsigned long long)entries * 8ull) cnt->err |= 1u << NGPU_ERR_HASH_FULL;
}

// in-place rebuild for the set-up paths (upload, core placement, explicit
// lists); iterations rebuild inside k_prepass and k_scan_apply instead
template <int W>
__device__ __forceinline__ void k_hash_clear_body(const Grid& g_, const Walk& wk, const Counters* cnt) {
  if (hash_rebuild_due(cnt, wk.L * (int64_t)kBucketEntries)) hash_clear_part<W>(g_, wk);
}
template <int W>
__global__ void __launch_bounds__(kBlock) k_hash_clear(Walk wk, const Counters* cnt) {
  k_hash_clear_body<W>(hw_grid(), wk, cnt);
}

template <int W>
__device__ __forceinline__ void k_hash_refill_body(const Grid& g_, const DevSys& s, const Walk& wk, Counters* cnt) {
  if (hash_rebuild_due(cnt, wk.L * (int64_t)kBucketEntries)) hash_refill_part<W>(g_, s, wk, cnt, (int64_t)cnt->nslots);
}
template <int W>
__global__ void __launch_bounds__(kBlock) k_hash_refill(DevSys s, Walk wk, Counters* cnt) {
  k_hash_refill_body<W>(hw_grid(), s, wk, cnt);
}

__global__ void k_hash_done(Counters* cnt, int64_t entries) { hash_done(cnt, entries); }

}  // namespace ngpu
