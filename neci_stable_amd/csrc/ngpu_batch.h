// ngpu_batch.h -- batch launches: one launch of a kernel of the iteration
// chain covers every engine of a batch group.
//
// A group is a set of engines whose chains use the same kernel instances
// (words per determinant, replica layout, generator, spawn-record precision,
// core precision, launch knobs).  Each engine
// keeps its own walker table, hash, spawn buffers, counters and statistics;
// an EngDev in device memory describes them, and each launch kind gives every
// engine a contiguous share of the launch's blocks.  A block finds its engine
// from a block map (or from its index, for the kinds with a fixed count per
// engine) and runs the same kernel body as a plain launch, on its share of
// the blocks, so every engine's results are those of iterating it alone.
#pragma once
#include "ngpu_kernels.h"

namespace ngpu {

// launch kinds of a batch chain and how each engine's share is sized
enum {
  kLkChunk = 0,  // chunked kernels: prepass, attempt scan
  kLkGrid,       // grid-stride kernels: spawns, insert, statistics
  kLkMerge,      // merge and annihilation
  kLkCore,       // core gather and apply (one element per thread)
  kLkCoreRow,    // core H.v (one row per wave)
  kLkKinds
};
// One engine of a batch group as its kernels see it.
struct EngDev {
  DevSys s;
  Walk wk;
  Counters* cnt;
  double* part;
  int32_t* att_cnt;
  int64_t* att_off;
  uint8_t* pinfo;
  int64_t* blk_part;
  int64_t* blk_rm;
  int64_t* tile_p;
  int64_t tcap;
  Bins bins;
  int64_t scap;
  int64_t* sq;
  uint64_t* n_key;
  double* n_sgn;
  uint32_t* n_flag;
  IterParams* prm;
  ngpu_iter_out_t* dout;
  ngpu_iter_out_t* dcyc;
  int64_t ncore;
  int64_t* core_slot;
  int64_t* core_rowptr;
  int32_t* core_cols;
  const void* core_vals;
  double* core_x;
  double* core_y;
  int32_t core_col0;     // shared core space: this engine's first column of the group's vectors
  int32_t b0[kLkKinds];  // first block of this engine's share, per launch kind
  int32_t nb[kLkKinds];  // blocks of the share
};

// A pointer of a descriptor, read as one to global memory: what the compiler
// loads from memory is a generic pointer to it, and it would reach through
// those with flat accesses, which wait for LDS and global memory alike.
// (16 replicas of 14e/30o and 16 Hubbard chains, ms per iteration: spawning
// 3.18 -> 2.87, merge 1.54 -> 1.45, the whole 9.65 -> 9.13.)
template <typename T>
__device__ inline void read_global(T*& p, T* const& field) {
  typedef T __attribute__((address_space(1))) GT;
  p = (T*)*(GT* const*)&field;
}
// this block's engine (a copy, of which only what a kernel uses is read) and
// its share of a kind with a block map
__device__ __forceinline__ EngDev eng_of(const EngDev* __restrict__ ed, const uint16_t* __restrict__ map, int kind,
                                         Grid& g) {
  const EngDev& d = ed[map[blockIdx.x]];
  g.b = (int64_t)blockIdx.x - d.b0[kind];
  g.nb = d.nb[kind];
  EngDev a = d;
#define NGPU_GLOBAL(f) read_global(a.f, d.f)
  NGPU_GLOBAL(s.rh); NGPU_GLOBAL(s.nbr); NGPU_GLOBAL(s.tmat); NGPU_GLOBAL(s.umat); NGPU_GLOBAL(s.ab_tab);
  NGPU_GLOBAL(s.ab_prob); NGPU_GLOBAL(s.ab_ok); NGPU_GLOBAL(s.j_tab); NGPU_GLOBAL(s.j_prob); NGPU_GLOBAL(s.j_ok);
  NGPU_GLOBAL(s.ab_tgt); NGPU_GLOBAL(s.i_tab); NGPU_GLOBAL(s.i_prob); NGPU_GLOBAL(s.a_tab); NGPU_GLOBAL(s.a_prob);
  NGPU_GLOBAL(s.a_ok); NGPU_GLOBAL(s.b_tab); NGPU_GLOBAL(s.b_prob); NGPU_GLOBAL(s.b_ok); NGPU_GLOBAL(s.jk);
  NGPU_GLOBAL(s.jkrow); NGPU_GLOBAL(s.jk0); NGPU_GLOBAL(s.fref);
  NGPU_GLOBAL(wk.keys); NGPU_GLOBAL(wk.st); NGPU_GLOBAL(wk.diagH); NGPU_GLOBAL(wk.offdiagH); NGPU_GLOBAL(wk.htab);
  NGPU_GLOBAL(wk.freeq);
  NGPU_GLOBAL(cnt); NGPU_GLOBAL(part); NGPU_GLOBAL(att_cnt); NGPU_GLOBAL(att_off); NGPU_GLOBAL(pinfo);
  NGPU_GLOBAL(blk_part); NGPU_GLOBAL(blk_rm); NGPU_GLOBAL(tile_p);
  NGPU_GLOBAL(bins.rec); NGPU_GLOBAL(bins.ovf); NGPU_GLOBAL(bins.next); NGPU_GLOBAL(bins.head);
  NGPU_GLOBAL(bins.count);
  NGPU_GLOBAL(sq); NGPU_GLOBAL(n_key); NGPU_GLOBAL(n_sgn); NGPU_GLOBAL(n_flag); NGPU_GLOBAL(prm);
  NGPU_GLOBAL(core_slot); NGPU_GLOBAL(core_rowptr); NGPU_GLOBAL(core_cols); NGPU_GLOBAL(core_x); NGPU_GLOBAL(core_y);
#undef NGPU_GLOBAL
  return a;
}

template <int W, int R>
__global__ void __launch_bounds__(kBlock) km_prepass(const EngDev* __restrict__ ed, const uint16_t* __restrict__ map) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkChunk, g);
  const IterParams none{};
  k_prepass_body<W, R>(g, a.s, a.wk, a.cnt, a.part, a.att_cnt, a.pinfo, a.blk_part, a.blk_rm, a.prm, none, 0);
}

template <int W>
__global__ void __launch_bounds__(kBlock) km_scan_apply(const EngDev* __restrict__ ed, const uint16_t* __restrict__ map) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkChunk, g);
  k_scan_apply_body<W>(g, a.s, a.wk, a.att_cnt, a.att_off, a.blk_part, a.blk_rm, a.pinfo, a.cnt, a.s.S, a.tile_p,
                       a.tcap, a.bins);
}

template <int W, int R, int G>
__global__ void __launch_bounds__(kBlock) km_spawn(const EngDev* __restrict__ ed, const uint16_t* __restrict__ map) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkGrid, g);
  k_spawn_body<W, R, G>(g, a.s, a.wk, a.cnt, a.part, a.att_off, a.tile_p, a.tcap, a.pinfo, a.bins,
                        a.scap, a.sq, a.prm);
}

template <int W, int R, int PP, int G>
__global__ void __launch_bounds__(kBlock, PP <= 3 ? 4 : PP <= 5 ? 3 : 2) km_spawn_singles(const EngDev* __restrict__ ed,
                                                           const uint16_t* __restrict__ map) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkGrid, g);
  k_spawn_singles_body<W, R, PP, G>(g, a.s, a.wk, a.cnt, a.part, a.pinfo, a.bins, a.scap, a.sq, a.prm);
}

template <int W, int R>
__global__ void __launch_bounds__(kBlock, R <= 2 && W == 1 ? 5 : 1) km_merge_annihilate(const EngDev* __restrict__ ed,
                                                              const uint16_t* __restrict__ map) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkMerge, g);
  k_merge_body<W, R, false>(g, a.s, a.wk, a.cnt, a.part, a.bins, a.n_key, a.n_sgn, a.n_flag, &a.cnt->n_new, a.prm,
                            stats_by_parts(a.s));
}

template <int R>
__global__ void __launch_bounds__(kBlock) km_core_gather(const EngDev* __restrict__ ed,
                                                         const uint16_t* __restrict__ map) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkCore, g);
  k_core_gather_body<R>(g, a.core_slot, a.wk, a.s.S, a.ncore, a.core_x, a.s.S);
}

// Core space shared by every engine of the group (the same determinants, so
// the same Hamiltonian, as replicas of one system have under a global core
// space): the engines' amplitudes are the C columns of one interleaved vector
// X[i * C + column], the Hamiltonian is read once for all of them, and
// Y[i * C + column] = (H.X + shift * X) * tau per column.
template <int R>
__global__ void __launch_bounds__(kBlock) km_core_gather_shared(const EngDev* __restrict__ ed,
                                                                const uint16_t* __restrict__ map, double* X, int C) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkCore, g);
  k_core_gather_body<R>(g, a.core_slot, a.wk, a.s.S, a.ncore, X + a.core_col0, C);
}

constexpr int kCoreCols = 16;  // columns per pass of the shared projection

// One wave per row; lane l works on column c0 + (l & 15) and the row's
// nonzeros q = q0 + (l >> 4), +4, ..., so each load instruction of the wave
// reads four whole 128-byte rows of X (16 columns) instead of 64 scattered
// elements; the four partial sums of a column meet in two butterfly steps.
// The order of the additions differs from an engine's own projection
// (k_core_spmv_body), so the results agree with it to rounding.
// colmap[c] = engine << 8 | replica of column c.
template <typename VT>
__global__ void __launch_bounds__(kBlock) km_core_spmv_shared(const EngDev* __restrict__ ed, const int32_t* colmap,
                                                              const double* X, double* Y, int C) {
  const EngDev& a = ed[0];
  const int64_t* rowptr = a.core_rowptr;
  const int32_t* cols = a.core_cols;
  const VT* vals = (const VT*)a.core_vals;
  const int64_t ncore = a.ncore;
  const int lane = lane_id(), k = lane & (kCoreCols - 1), sub = lane / kCoreCols;
  constexpr int kSubs = kWave / kCoreCols;
  const int64_t nwaves = (int64_t)gridDim.x * blockDim.x / kWave;
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave; i < ncore; i += nwaves) {
    const int64_t q0 = rowptr[i], q1 = rowptr[i + 1];
    for (int c0 = 0; c0 < C; c0 += kCoreCols) {
      const bool on = c0 + k < C;
      double acc = 0.0;
      for (int64_t q = q0 + sub; q < q1; q += kSubs) {
        const double v = (double)vals[q];
        if (on) acc = acc - v * X[(size_t)cols[q] * C + c0 + k];
      }
#pragma unroll
      for (int o = kCoreCols; o < kWave; o <<= 1) acc = acc + __shfl_xor(acc, o);
      if (sub == 0 && on) {
        const int c = c0 + k, m = colmap[c];
        const IterParams* prm = ed[m >> 8].prm;
        Y[i * C + c] = (acc + prm->sft.v[m & 255] * X[i * C + c]) * prm->tau;
      }
    }
  }
}

template <int R>
__global__ void __launch_bounds__(kBlock) km_core_apply_shared(const EngDev* __restrict__ ed,
                                                               const uint16_t* __restrict__ map, const double* Y,
                                                               int C) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkCore, g);
  k_core_apply_body<R>(g, a.s, a.wk, a.cnt, a.core_slot, Y + a.core_col0, a.ncore, a.part, C);
}
template <int R, typename VT>
__global__ void __launch_bounds__(kBlock) km_core_spmv(const EngDev* __restrict__ ed, const uint16_t* __restrict__ map) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkCoreRow, g);
  k_core_spmv_body<R, VT>(g, a.core_rowptr, a.core_cols, (const VT*)a.core_vals, a.core_x, a.core_y, a.ncore, a.s.S,
                          a.prm);
}
template <int R>
__global__ void __launch_bounds__(kBlock) km_core_apply(const EngDev* __restrict__ ed,
                                                        const uint16_t* __restrict__ map) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkCore, g);
  k_core_apply_body<R>(g, a.s, a.wk, a.cnt, a.core_slot, a.core_y, a.ncore, a.part, a.s.S);
}

template <int W, int R, int GL>
__global__ void __launch_bounds__(kBlock) km_insert(const EngDev* __restrict__ ed, const uint16_t* __restrict__ map) {
  extern __shared__ double insert_dyn[];
  Grid g;
  const EngDev a = eng_of(ed, map, kLkGrid, g);
  k_insert_body<W, R, GL>(g, a.s, a.wk, a.cnt, a.n_key, a.n_sgn, a.n_flag, &a.cnt->n_new, insert_dyn);
}

template <int W, int R>
__global__ void __launch_bounds__(kBlock) km_stats(const EngDev* __restrict__ ed, const uint16_t* __restrict__ map) {
  Grid g;
  const EngDev a = eng_of(ed, map, kLkGrid, g);
  if (stats_by_parts(a.s)) return;
  k_stats_body<W, R>(g, a.s, a.wk, a.cnt, a.part, a.prm);
}

}  // namespace ngpu
