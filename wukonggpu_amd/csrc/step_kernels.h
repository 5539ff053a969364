// Pattern-step kernels: probe, tile scan, finalize (compaction of the rows
// that produce output), merge-path partition, load-balanced expand,
// single-key probe and list copy.
//
// One known_to_unknown step (RCache::known_to_unknown, core/rcache.hpp:
// 232-414) runs as
//   k_probe -> k_follow (up to kScanChunk probe tiles and an output that fits), or
//   k_probe -> tile scan -> [totals read back] -> k_hit_splits -> k_expand_hits, or
//   k_probe -> tile scan -> k_finalize -> [totals] -> k_partition -> k_expand (large fan-outs)
// replacing the reference's keygen, probe, edge-list fetch, Thrust scan and
// one-thread-per-row update (core/gpu_hash.cu:145-316, 527-610, 685-694).
// known_to_known / known_to_const (core/gpu_hash.cu:320-466, 613-682) run as
//   k_probe -> k_follow, or
//   k_probe -> tile scan -> k_finalize (stable compaction of kept rows)
// index_to_unknown / const_to_unknown are k_probe_copy (+ k_copy_list for a
// list above kListCap entries).
//
// The probe writes, per tile, the list of rows that have edges (or that a
// filter keeps) and the tile's sums; the tile scan turns the sums into
// prefixes; the finalize pass moves each tile's list to its global place.
// Everything after the probe touches only rows that produce output. (This is
// reduce-then-scan: a single-pass decoupled look-back serialises on
// device-scope loads that cross the XCDs' separate L2s.)
//
// The per-tile bodies are shared with the batched kernels, which run many
// independent steps in one launch.
#pragma once

#include "../../include/wukong_gpu.h"
#include "device.h"

namespace wkg {
namespace {

enum StepMode : int { kModeK2U = 0, kModeK2K = 1, kModeK2C = 2 };


// One step's view for the probe / scan / finalize passes.
struct StepParams {
  const int32_t *T;    // input table (null for a single-key step)
  uint64_t R;          // input rows (1 for a single-key step); < 2^32
  uint32_t c;          // input columns
  uint32_t sc, ec;     // start column; K2K end column
  uint32_t pid, dir;
  uint32_t target;     // K2C constant
  uint32_t target_ok;  // K2C constant fits u32 (otherwise nothing matches)
  int mode;            // kMode*
  uint64_t key;        // != 0: single-key step (index / const start), R == 1
  uint4 *hits;         // per tile, one entry per tile row: (row, offset, degree, K2U: the tile's output rows
                       // before this one (mod 2^32)) of rows with output
  uint2 *cinfo;        // K2U, compacted rows: (row, offset)
  uint64_t *cexcl;     // K2U, compacted rows: exclusive output-row offset
  int32_t *O;          // filters: compacted output, capacity R x c
  uint64_t *tile_sum;  // per tile: output rows; after the tile scan, the tile's prefix
  uint64_t *tile_nz;   // per tile: rows with output; after the tile scan, the prefix
  uint64_t *tile_ex;   // per tile: edges examined (filters) / keys probed (K2U)
  uint64_t *totals;    // [0] output rows, [1] edges examined (filters) or keys probed (K2U),
                       // [2] rows with output
  uint64_t ntiles;     // tiles of this step
  // two-level tile scan (null when one block scans all tiles): per chunk of
  // kScanChunk tiles, the chunk's prefix of output rows / rows with output
  uint64_t *chunk_sum, *chunk_nz, *chunk_ex;
  // per-step path: the totals are also published to the host by the kernel
  // that computes them (null: not published)
  Signal sg = {nullptr, 0};
  uint64_t tile0 = 0;  // k_probe / k_finalize: the launch's first tile (the per-step path's launches are split)
  // filters: each row's edges examined count `T[row * c + wc]` times (a
  // row standing for that many rows of another table)
  uint32_t weighted = 0, wc = 0;
};

constexpr int kScanChunk = 8 * kBlock;  // tiles per block in the two-level tile scan

// Membership of `target` in an 8-lane group's edge list (known_to_known/const
// test, core/engine.hpp:179-184,211-216), for lists that need not be sorted:
// 8 entries at a time with early exit, like the reference's linear scan. The
// work count is the reference's: index of the first match + 1, or the
// degree when absent.
template <bool FRAMED>
__device__ __forceinline__ void group_scan(const GraphView &g, uint64_t estart, uint64_t efb, uint32_t off,
                                           uint32_t deg, uint32_t target, bool valid, bool &found,
                                           uint32_t &examined) {
  const uint32_t lane = lane_id(), l8 = lane & 7, gbase = lane & ~7u;
  const bool act = valid && deg > 0;
  found = false;
  uint32_t idx = 0, j = 0;
  while (true) {
    const bool go = act && !found && j < deg;
    if (!wave_ballot(go)) break;
    bool eq = false;
    if (go && j + l8 < deg) eq = edge_at<FRAMED>(g, estart, efb, (uint64_t)off + j + l8) == target;
    const uint32_t gb = (uint32_t)(wave_ballot(eq) >> gbase) & 0xffu;
    if (go) {
      if (gb) {
        found = true;
        idx = j + (uint32_t)__builtin_ctz(gb);
      } else {
        j += 8;
      }
    }
  }
  examined = found ? idx + 1 : deg;
}

// Membership of every lane's own target in its own edge list (one row per
// lane; the whole wave calls it): found and the reference's work count.
// Sorted lists: each lane searches by itself, three pivots loaded together
// per round, so a round quarters the range and the last <= 4 entries are
// compared at once. What bounds it is the chain of dependent loads, and a
// wave has 64 of them in flight; an 8-lane 9-ary search,
// which this replaced, ran a group's 8 rows one after another (8
// chains in flight, 8 times as long): a known_to_known step over
// 3M rows, half of them walked edges, 401 -> 210 us; known_to_const over 12M
// rows of one-entry lists 443 -> 370 us (before tag words: 404 with them).
// Unsorted lists: the 8 lanes of a group scan the group's 8 lists in turn.
template <bool SORTED, bool FRAMED>
__device__ __forceinline__ void rows_member(const GraphView &g, uint64_t estart, uint64_t efb, uint32_t off,
                                            uint32_t deg, uint32_t target, bool valid, bool &found,
                                            uint32_t &examined) {
  found = false;
  examined = deg;
  if constexpr (SORTED) {
    if (valid && deg) {
      uint32_t lo = 0, hi = deg - 1;  // the first match, if any, is in [lo, hi]
      while (hi - lo > 3) {
        const uint32_t q = (hi - lo) >> 2, p1 = lo + q, p2 = p1 + q, p3 = p2 + q;
        const uint32_t v1 = edge_at<FRAMED>(g, estart, efb, (uint64_t)off + p1);
        const uint32_t v2 = edge_at<FRAMED>(g, estart, efb, (uint64_t)off + p2);
        const uint32_t v3 = edge_at<FRAMED>(g, estart, efb, (uint64_t)off + p3);
        lo = v3 < target ? p3 + 1 : v2 < target ? p2 + 1 : v1 < target ? p1 + 1 : lo;
        hi = v3 < target ? hi : v2 < target ? p3 : v1 < target ? p2 : p1;
      }
      uint32_t v[4];
#pragma unroll
      for (int k = 0; k < 4; k++) v[k] = lo + k <= hi ? edge_at<FRAMED>(g, estart, efb, (uint64_t)off + lo + k) : ~target;
#pragma unroll
      for (int k = 3; k >= 0; k--)
        if (v[k] == target) {
          found = true;
          examined = lo + k + 1;
        }
    }
  } else {
    const uint32_t lane = lane_id(), gbase = lane & ~7u, l8 = lane & 7;
#pragma unroll 1
    for (uint32_t u = 0; u < 8; u++) {
      const uint32_t src = gbase + u;
      bool f;
      uint32_t x;
      group_scan<FRAMED>(g, estart, efb, shfl32(off, src), shfl32(deg, src), shfl32(target, src),
                         shfl32(valid ? 1u : 0u, src) != 0, f, x);
      if (l8 == u) {
        found = f;
        examined = x;
      }
    }
  }
}

// Probe pass over one tile (TR rows; `lt` is the tile's index within its
// step). Wave w owns the tile's rows [w * TR/4, (w+1) * TR/4) and probes
// them 64 consecutive rows per round, carrying the last key across rounds.
// Writes the tile's list of rows with output and its sums.
template <int TR, bool SORTED, bool FRAMED, bool TAGS = !FRAMED>
__device__ __forceinline__ void probe_tile(const GraphView &g, const StepParams &p, uint64_t lt) {
  constexpr int kRounds = TR / kBlock;  // one row per lane per round
  constexpr int kRowsPerThread = TR / kBlock;
  static_assert(TR % kBlock == 0, "tile rows must be a multiple of the block");
  __shared__ uint32_t s_cnt[TR];  // degree, or kept flag
  __shared__ uint32_t s_aux[TR];  // segment offset, or edges examined
  __shared__ uint64_t s_tmp[kBlock / kWave];
  __shared__ uint32_t s_probed[kBlock / kWave];
  __shared__ WaveProbeLds s_wp[kBlock / kWave];
  const uint32_t tid = threadIdx.x, lane = lane_id();
  const uint32_t wave = tid / kWave;
  const uint64_t base = lt * TR;
  const DevMeta m = g.meta[p.pid < g.num_metas ? p.pid : 0];

  // all rounds' table reads are issued up front
  constexpr uint32_t kWaveRows = TR / (kBlock / kWave);
  const auto T = gmem(p.T);
  int32_t cells[kRounds], ends[kRounds];
#pragma unroll
  for (int rd = 0; rd < kRounds; rd++) {
    const uint64_t row = base + wave * kWaveRows + rd * kWave + lane;
    const bool in = row < p.R && !p.key;
    cells[rd] = in ? T[row * p.c + p.sc] : -1;
    ends[rd] = in && p.mode == kModeK2K ? T[row * p.c + p.ec] : 0;
  }
  auto plan = [&](int rd, uint64_t before63) {
    const uint64_t row = base + wave * kWaveRows + rd * kWave + lane;
    uint64_t key = 0;
    if (row < p.R) {
      if (p.key) key = p.key;
      else if (cells[rd] >= 0) key = make_key((uint32_t)cells[rd], p.pid, p.dir);
    }
    return probe_plan<FRAMED, TAGS>(g, m, key, before63);
  };
  uint32_t probed = 0;
  // The wave's rows' degrees and list offsets into s_cnt and s_aux. Round rd
  // is finished while round rd + 1's slots and round rd + 2's tag words are on
  // their way.
  ProbePlan pl[3];
  pl[0] = plan(0, 0);
  if (kRounds > 1) pl[1] = plan(1, lane63_64(pl[0].key));
  probe_pick<TAGS>(g, pl[0]);
  if constexpr (TAGS) {
    // The rows that must walk (few) wait for all rounds: their walks, chains
    // of dependent reads, then run once per tile, not once per round.
    uint4 *kb = s_wp[wave].kb;
    uint32_t pending = 0;                   // (wave-uniform)
    uint64_t lead[kRounds], have[kRounds];  // leaders and rows with a key (wave-uniform)
    const uint64_t below = lanes_below();
    auto put = [&](uint32_t row, uint32_t d, uint32_t o) {
      s_cnt[row] = d;
      s_aux[row] = o;
    };
#pragma unroll
    for (int rd = 0; rd < kRounds; rd++) {
      const uint32_t local = wave * kWaveRows + rd * kWave + lane;
      if (rd + 2 < kRounds) pl[(rd + 2) % 3] = plan(rd + 2, lane63_64(pl[(rd + 1) % 3].key));
      if (rd + 1 < kRounds && pl[(rd + 1) % 3].leaders) probe_pick<TAGS>(g, pl[(rd + 1) % 3]);
      const ProbePlan &cur = pl[rd % 3];
      lead[rd] = cur.leaders;
      have[rd] = wave_ballot(cur.key != 0);
      if (!cur.leaders) {  // (wave-uniform: a long run goes on, or no keys)
        put(local, 0, 0);
        continue;
      }
      probed += (uint32_t)__builtin_popcountll(cur.leaders);
      uint32_t deg, off;
      const bool walk = !probe_slot<true>(g, m, cur, deg, off);
      put(local, deg, off);
      const uint64_t walkers = wave_ballot(walk);
      const uint32_t nw = (uint32_t)__builtin_popcountll(walkers);
      if (pending + nw > (uint32_t)kWave) {  // (wave-uniform)
        wave_lds_sync();
        walk_pending<false, 2>(g, m, kb, pending, put);
        pending = 0;
      }
      if (walk)
        kb[pending + (uint32_t)__builtin_popcountll(walkers & below)] =
            make_uint4((uint32_t)cur.key, (uint32_t)(cur.key >> 32), cur.bucket, local);
      pending += nw;
    }
    if (pending) {
      wave_lds_sync();
      walk_pending<false, 2>(g, m, kb, pending, put);
    }
    // rows that follow a leader take its result (a run may have begun in an earlier round)
    uint32_t last = 0;  // the last leader's row so far
#pragma unroll
    for (int rd = 0; rd < kRounds; rd++) {
      const uint32_t first = wave * kWaveRows + rd * kWave;
      if (have[rd] != lead[rd]) {  // (wave-uniform)
        wave_lds_sync();
        const uint64_t mine = lead[rd] & (below | (1ull << lane));
        const uint32_t src = mine ? first + 63u - (uint32_t)__builtin_clzll(mine) : last;
        const uint32_t d = s_cnt[src], o = s_aux[src];
        if ((have[rd] & ~lead[rd]) >> lane & 1) put(first + lane, d, o);
      }
      if (lead[rd]) last = first + 63u - (uint32_t)__builtin_clzll(lead[rd]);
    }
  } else {
    ProbeCarry carry;
#pragma unroll
    for (int rd = 0; rd < kRounds; rd++) {
      const uint32_t local = wave * kWaveRows + rd * kWave + lane;
      if (rd + 2 < kRounds) pl[(rd + 2) % 3] = plan(rd + 2, lane63_64(pl[(rd + 1) % 3].key));
      if (rd + 1 < kRounds) probe_pick<TAGS>(g, pl[(rd + 1) % 3]);
      probed += probe_finish<FRAMED, TAGS>(g, m, pl[rd % 3], s_wp[wave], s_cnt[local], s_aux[local], carry);
    }
  }
  if (p.mode != kModeK2U) {  // filters: kept flags and edges examined in their place
    wave_lds_sync();
    const bool k2k = p.mode == kModeK2K;
#pragma unroll
    for (int rd = 0; rd < kRounds; rd++) {
      const uint32_t local = wave * kWaveRows + rd * kWave + lane;
      const uint32_t deg = s_cnt[local], off = s_aux[local];
      bool found;
      uint32_t examined;
      rows_member<SORTED, FRAMED>(g, m.edge_start, m.eframe_base, off, deg, k2k ? (uint32_t)ends[rd] : p.target,
                                  k2k ? ends[rd] >= 0 : p.target_ok != 0, found, examined);
      s_cnt[local] = found ? 1u : 0u;
      s_aux[local] = examined;
    }
  }
  if (lane == 0) s_probed[wave] = probed;
  __syncthreads();
  // thread t owns the tile's rows [t * kRowsPerThread, (t + 1) * kRowsPerThread)
  uint64_t sum = 0, ex = 0;
  uint32_t nz = 0;
#pragma unroll
  for (int k = 0; k < kRowsPerThread; k++) {
    const uint32_t c = s_cnt[tid * kRowsPerThread + k];
    sum += c;
    nz += c ? 1u : 0u;
    uint64_t w = 1;
    if (p.weighted) {
      const uint64_t row = base + tid * kRowsPerThread + k;
      w = row < p.R ? (uint32_t)T[row * p.c + p.wc] : 0u;
    }
    ex += (uint64_t)s_aux[tid * kRowsPerThread + k] * w;
  }
  uint64_t nz_total, sum_total, ex_total = 0;
  uint32_t pos = (uint32_t)block_excl_scan(nz, s_tmp, nz_total);
  uint32_t before = (uint32_t)block_excl_scan(sum, s_tmp, sum_total);
  if (p.mode != kModeK2U) (void)block_excl_scan(ex, s_tmp, ex_total);
  uint4 *hits = p.hits + lt * TR;
#pragma unroll
  for (int k = 0; k < kRowsPerThread; k++) {
    const uint32_t local = tid * kRowsPerThread + k;
    const uint32_t c = s_cnt[local];
    if (c) gstore(hits + pos++, make_uint4((uint32_t)(base + local), p.mode == kModeK2U ? s_aux[local] : 0u, c, before));
    before += c;
  }
  if (tid == 0) {
    gmem(p.tile_sum)[lt] = sum_total;
    gmem(p.tile_nz)[lt] = nz_total;
    uint32_t keys = 0;
#pragma unroll
    for (int w = 0; w < kBlock / kWave; w++) keys += s_probed[w];
    gmem(p.tile_ex)[lt] = p.mode == kModeK2U ? (uint64_t)keys : ex_total;
  }
}

// At most 128 VGPRs, so four waves per SIMD hide the probe's load chains.
template <int TR, bool SORTED, bool FRAMED>
__global__ __launch_bounds__(kBlock, 4) void k_probe(GraphView g, StepParams p) {
  probe_tile<TR, SORTED, FRAMED>(g, p, p.tile0 + blockIdx.x);
}

// In-place exclusive scan of a[0, n) by one block; returns the total.
__device__ __forceinline__ uint64_t block_scan_array(uint64_t *a_, uint64_t n, uint64_t *s_tmp) {
  const auto a = gmem(a_);
  const uint64_t per = (n + kBlock - 1) / kBlock;
  const uint64_t lo = threadIdx.x * per < n ? threadIdx.x * per : n;
  const uint64_t hi = lo + per < n ? lo + per : n;
  uint64_t s = 0;
  uint64_t i = lo;
  for (; i + 8 <= hi; i += 8) {  // 8 independent loads in flight
    uint64_t v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = a[i + k];
#pragma unroll
    for (int k = 0; k < 8; k++) s += v[k];
  }
  for (; i < hi; i++) s += a[i];
  uint64_t total;
  uint64_t run = block_excl_scan(s, s_tmp, total);
  for (i = lo; i < hi; i++) {
    const uint64_t v = a[i];
    a[i] = run;
    run += v;
  }
  return total;
}

// Tile scan of one step (one block): tile_sum and tile_nz become prefixes;
// writes the step's totals.
__device__ __forceinline__ void scan_step_tiles(const StepParams &p) {
  __shared__ uint64_t s_tmp[kBlock / kWave];
  const uint64_t rows = block_scan_array(p.tile_sum, p.ntiles, s_tmp);
  const uint64_t nz = block_scan_array(p.tile_nz, p.ntiles, s_tmp);
  uint64_t ex = 0, e = 0;
  for (uint64_t i = threadIdx.x; i < p.ntiles; i += kBlock) e += p.tile_ex[i];
  (void)block_excl_scan(e, s_tmp, ex);
  if (threadIdx.x == 0) {
    p.totals[0] = rows;
    p.totals[1] = ex;
    p.totals[2] = nz;
    if (p.sg.h) {
      const uint64_t v[3] = {rows, ex, nz};
      publish(p.sg, v, 3);
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_scan_tiles(StepParams p) { scan_step_tiles(p); }

// Two-level tile scan, level 1: chunk k (kScanChunk tiles) is scanned in
// place (chunk-local prefixes) and its sums stored. With a single chunk the
// step's totals and zero chunk prefixes are written directly.
__device__ __forceinline__ void scan_chunk(const StepParams &p, uint64_t chunk, uint64_t nchunks) {
  __shared__ uint64_t s_tmp[kBlock / kWave];
  constexpr int PT = kScanChunk / kBlock;
  const uint64_t lo = chunk * (uint64_t)kScanChunk + threadIdx.x * PT;
  const auto tile_sum = gmem(p.tile_sum), tile_nz = gmem(p.tile_nz);
  uint64_t vs[PT], vn[PT], s = 0, nzs = 0, e = 0;
#pragma unroll
  for (int k = 0; k < PT; k++) {
    const bool in = lo + k < p.ntiles;
    vs[k] = in ? tile_sum[lo + k] : 0;
    vn[k] = in ? tile_nz[lo + k] : 0;
    if (in) e += gmem(p.tile_ex)[lo + k];
    s += vs[k];
    nzs += vn[k];
  }
  uint64_t ts, tn, te;
  uint64_t rs = block_excl_scan(s, s_tmp, ts);
  uint64_t rn = block_excl_scan(nzs, s_tmp, tn);
  (void)block_excl_scan(e, s_tmp, te);
#pragma unroll
  for (int k = 0; k < PT; k++)
    if (lo + k < p.ntiles) {
      tile_sum[lo + k] = rs;
      tile_nz[lo + k] = rn;
      rs += vs[k];
      rn += vn[k];
    }
  if (threadIdx.x == 0) {
    if (nchunks == 1) {
      gmem(p.totals)[0] = ts;
      gmem(p.totals)[1] = te;
      gmem(p.totals)[2] = tn;
      gmem(p.chunk_sum)[0] = 0;
      gmem(p.chunk_nz)[0] = 0;
      if (p.sg.h) {
        const uint64_t v[3] = {ts, te, tn};
        publish(p.sg, v, 3);
      }
    } else {
      gmem(p.chunk_sum)[chunk] = ts;
      gmem(p.chunk_nz)[chunk] = tn;
      gmem(p.chunk_ex)[chunk] = te;
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_scan_chunks(StepParams p) { scan_chunk(p, blockIdx.x, gridDim.x); }

// Level 2 (one block): chunk sums become chunk prefixes; writes the totals.
__device__ __forceinline__ void scan_top(const StepParams &p, uint64_t nchunks) {
  __shared__ uint64_t s_tmp[kBlock / kWave];
  const uint64_t rows = block_scan_array(p.chunk_sum, nchunks, s_tmp);
  const uint64_t nz = block_scan_array(p.chunk_nz, nchunks, s_tmp);
  uint64_t e = 0, ex = 0;
  for (uint64_t i = threadIdx.x; i < nchunks; i += kBlock) e += gmem(p.chunk_ex)[i];
  (void)block_excl_scan(e, s_tmp, ex);
  if (threadIdx.x == 0) {
    gmem(p.totals)[0] = rows;
    gmem(p.totals)[1] = ex;
    gmem(p.totals)[2] = nz;
    if (p.sg.h) {
      const uint64_t v[3] = {rows, ex, nz};
      publish(p.sg, v, 3);
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_scan_top(StepParams p, uint64_t nchunks) { scan_top(p, nchunks); }

// Finalize pass over one tile of TR rows, by one wave: K2U moves the tile's
// rows with edges to the compacted row list with their exclusive output
// offsets; the filters copy the kept rows, in order, to the compacted output.
// Waves work on their tiles independently (no block barrier), so tiles with
// few rows cost one short chain of loads each.
template <int TR>
__device__ __forceinline__ void finalize_tile(const StepParams &p, uint64_t lt) {
  const uint32_t lane = lane_id();
  auto nz_prefix = [&](uint64_t t) -> uint64_t {
    if (t >= p.ntiles) return gmem(p.totals)[2];
    return gmem(p.tile_nz)[t] + (p.chunk_nz ? gmem(p.chunk_nz)[t / kScanChunk] : 0);
  };
  const uint64_t nz0 = nz_prefix(lt);
  const uint32_t nnz = (uint32_t)(nz_prefix(lt + 1) - nz0);
  if (nnz == 0) return;
  const uint64_t out0 = gmem(p.tile_sum)[lt] + (p.chunk_sum ? gmem(p.chunk_sum)[lt / kScanChunk] : 0);
  const uint4 *hits = p.hits + lt * TR;
  const auto T = gmem(p.T);
  const auto O = gmem(p.O);
  if (p.mode == kModeK2U) {
    uint64_t carry = 0;
    for (uint32_t k0 = 0; k0 < nnz; k0 += kWave) {
      const uint32_t j = k0 + lane;
      const uint4 h = j < nnz ? gload(hits + j) : make_uint4(0, 0, 0, 0);
      const uint64_t inc = wave_incl_scan(h.z);
      if (j < nnz) {
        gstore(p.cinfo + nz0 + j, make_uint2(h.x, h.y));
        gmem(p.cexcl)[nz0 + j] = out0 + carry + inc - h.z;
      }
      carry += shfl64(inc, kWave - 1);
    }
  } else {
    // kept rows k0.. of this tile go to output rows out0 + k0 ..
    const uint32_t c = p.c;
    for (uint32_t k0 = 0; k0 < nnz; k0 += kWave) {
      const uint32_t nsel = nnz - k0 < (uint32_t)kWave ? nnz - k0 : (uint32_t)kWave;
      const uint32_t myrow = lane < nsel ? gload(hits + k0 + lane).x : 0u;
      if (c <= (uint32_t)kWave) {  // 64 / c rows per pass, one column per lane
        const uint32_t rpp = kWave / c, col = lane % c, r0 = lane / c;
        for (uint32_t it = 0; it * rpp < nsel; it++) {
          const uint32_t r = it * rpp + r0;
          const uint32_t src = shfl32(myrow, r < (uint32_t)kWave ? r : 0u);
          if (r0 < rpp && r < nsel) O[(out0 + k0 + r) * c + col] = T[(uint64_t)src * c + col];
        }
      } else {
        for (uint32_t r = 0; r < nsel; r++) {
          const uint32_t src = shfl32(myrow, r);
          for (uint32_t col = lane; col < c; col += kWave) O[(out0 + k0 + r) * c + col] = T[(uint64_t)src * c + col];
        }
      }
    }
  }
}

// One wave per tile: tile blockIdx.x * 4 + wave.
template <int TR>
__global__ __launch_bounds__(kBlock) void k_finalize(StepParams p) {
  const uint64_t t = p.tile0 + blockIdx.x * (uint64_t)(kBlock / kWave) + threadIdx.x / kWave;
  if (t < p.ntiles) finalize_tile<TR>(p, t);
}

// Merge-path partition of the (row starts, output rows) sequence over the
// compacted rows: part[k] = number of rows whose start item lies before
// diagonal k * NV. Row i's start item sits at i + cexcl[i].
template <int NV>
__device__ __forceinline__ uint64_t merge_split(const uint64_t *cexcl, uint64_t R, uint64_t E, uint64_t k) {
  const uint64_t diag = k * (uint64_t)NV < R + E ? k * (uint64_t)NV : R + E;
  uint64_t lo = 0, hi = R;  // first i with i + cexcl[i] >= diag (R if none)
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (mid + cexcl[mid] < diag) lo = mid + 1; else hi = mid;
  }
  return lo;
}

__global__ void k_partition(const uint64_t *cexcl, uint64_t R, uint64_t E, uint64_t ntiles, uint64_t *part) {
  const uint64_t k = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  if (k <= ntiles) part[k] = merge_split<kExpandNV>(cexcl, R, E, k);
}

struct ExpandParams {
  uint32_t pid;
  const int32_t *T;      // input table
  uint32_t c;            // input columns
  uint64_t R;            // compacted rows (rows with at least one edge)
  const uint2 *cinfo;    // compacted rows: (input row, segment offset)
  const uint64_t *cexcl; // compacted rows: exclusive output-row offset
  const uint64_t *part;  // ntiles + 1 split points
  uint64_t E;
  int32_t *O;  // E x (c+1)
  uint64_t tile0;  // k_expand: the launch's first tile
};

// Load-balanced expand (known_to_unknown result update): a tile owns
// NV = kBlock * VT items of the merged sequence of row starts and output rows, so a
// hub row's outputs spread over many workgroups. Output row o of compacted
// row i is (input row, edge k) with k = o - cexcl[i]; rows come out in input
// order and edges in list order (core/engine.hpp:142-150).
// Phase 1 stages the tile's rows in LDS; phase 2 walks the merge path and
// issues each thread's (up to VT) edge loads together, parking the
// edges in LDS; phase 3 writes the tile's contiguous output region with
// aligned 16-byte stores. `tile` is the tile index within the step.
template <int VT, bool FRAMED>
__device__ __forceinline__ void expand_tile(const GraphView &g, const ExpandParams &a, uint64_t tile) {
  constexpr int NV = kBlock * VT;
  static_assert(NV < 65536, "local output rows are kept in 16 bits");
  __shared__ int32_t s_ex[NV + 1];
  __shared__ uint32_t s_off[NV + 1];
  __shared__ uint32_t s_row[NV + 1];
  __shared__ uint16_t s_orow[NV];
  __shared__ uint32_t s_edge[NV];
  const uint32_t tid = threadIdx.x;
  const uint64_t d0 = tile * (uint64_t)NV;
  const uint64_t dend = a.R + a.E;
  const uint64_t d1 = d0 + NV < dend ? d0 + NV : dend;
  const uint64_t i0 = gmem(a.part)[tile], i1 = gmem(a.part)[tile + 1];
  const uint64_t j0 = d0 - i0, j1 = d1 - i1;
  const uint32_t nr = (uint32_t)(i1 - i0 + 1);  // local row r <-> compacted row i0 - 1 + r
  for (uint32_t r = tid; r < nr; r += kBlock) {
    if (r == 0 && i0 == 0) {
      s_ex[0] = 0;
      s_off[0] = 0;
      s_row[0] = 0;
    } else {
      const uint64_t i = i0 + r - 1;
      const uint2 ci = gload(a.cinfo + i);
      s_ex[r] = (int32_t)((int64_t)gmem(a.cexcl)[i] - (int64_t)j0);
      s_row[r] = ci.x;
      s_off[r] = ci.y;
    }
  }
  __syncthreads();
  // local merged position of local row r's start item: (r - 1) + s_ex[r]
  const int32_t span = (int32_t)(d1 - d0);
  const int32_t x0 = (int32_t)(tid * VT);
  const DevMeta m = g.meta[a.pid];
  if (x0 < span) {
    uint32_t lo = 1, hi = nr;  // rows r >= 1 whose start lies before x0
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if ((int32_t)(mid - 1) + s_ex[mid] < x0) lo = mid + 1; else hi = mid;
    }
    uint32_t cur = lo - 1;
    int32_t oidx[VT];
    uint32_t epos[VT];
#pragma unroll
    for (int v = 0; v < VT; v++) {
      const int32_t x = x0 + v;
      oidx[v] = -1;
      epos[v] = 0;
      if (x < span) {
        if (cur + 1 < nr && (int32_t)cur + s_ex[cur + 1] == x) {
          cur++;
        } else {
          const int32_t o = x - (int32_t)cur;
          oidx[v] = o;
          epos[v] = s_off[cur] + (uint32_t)(o - s_ex[cur]);
          s_orow[o] = (uint16_t)cur;
        }
      }
    }
    uint32_t ev[VT];
#pragma unroll
    for (int v = 0; v < VT; v++)
      ev[v] = oidx[v] >= 0 ? edge_at<FRAMED>(g, m.edge_start, m.eframe_base, epos[v]) : 0u;
#pragma unroll
    for (int v = 0; v < VT; v++)
      if (oidx[v] >= 0) s_edge[oidx[v]] = ev[v];
  }
  __syncthreads();
  // the tile's output is the contiguous int range [j0 * nc, j1 * nc)
  const uint32_t nout = (uint32_t)(j1 - j0);
  const uint32_t c = a.c, nc = c + 1;
  const uint32_t nint = nout * nc;
  const uint64_t g0 = j0 * nc;
  auto cell = [&](uint32_t r, uint32_t col) -> int32_t {
    return col < c ? gmem(a.T)[(uint64_t)s_row[s_orow[r]] * c + col] : (int32_t)s_edge[r];
  };
  // streaming (nontemporal) stores: the table is far larger than the caches
  typedef int32_t v4i __attribute__((ext_vector_type(4)));
  const uint32_t head = (uint32_t)((4 - (g0 & 3)) & 3) < nint ? (uint32_t)((4 - (g0 & 3)) & 3) : nint;
  const auto O = gmem(a.O);
  if (tid < head) __builtin_nontemporal_store(cell(tid / nc, tid % nc), &O[g0 + tid]);
  const uint32_t nquad = (nint - head) / 4;
  WKG_GLOBAL v4i *oq = (WKG_GLOBAL v4i *)(O + g0 + head);
  for (uint32_t q = tid; q < nquad; q += kBlock) {
    const uint32_t e = head + 4 * q;
    uint32_t r = e / nc, col = e - r * nc;
    v4i v;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      v[k] = cell(r, col);
      if (++col == nc) {
        col = 0;
        r++;
      }
    }
    __builtin_nontemporal_store(v, &oq[q]);
  }
  const uint32_t tail0 = head + 4 * nquad;
  if (tid < nint - tail0) {
    const uint32_t e = tail0 + tid;
    __builtin_nontemporal_store(cell(e / nc, e % nc), &O[g0 + e]);
  }
  __syncthreads();  // LDS is reused by the caller's next tile
}

template <bool FRAMED>
__global__ __launch_bounds__(kBlock) void k_expand(GraphView g, ExpandParams a) {
  expand_tile<kExpandVT, FRAMED>(g, a, a.tile0 + blockIdx.x);
}

// ---- expand and compaction straight from the probe's lists ----
// A workgroup takes NV consecutive output rows and finds their hits (the
// probe's per-tile lists) itself: the tile and the hit of its first and last
// row by 64-ary searches over the tiles' prefixes and the tile's running
// counts, so neither a compaction of the hits nor split points are needed
// (two launches and 32 B moved per hit less than k_finalize, k_partition and
// k_expand). Every hit has output, so NV rows need at most that many
// hits. What bounds it: the output rows' stores and one random edge read per
// row; the searches are a chain of dependent reads, hidden by the other
// workgroups of the CU on large outputs.
constexpr int kHitNV = kBlock * 4;     // output rows per block, large outputs
constexpr int kFollowNV = kBlock * 2;  // and in k_follow: its outputs are small, their blocks few
// (18M rows of 4 cells with 2048 / 1024 / 512 rows a block: 115 / 94 / 120 us;
// 16 interactive queries, 2048 / 1024 / 512 in k_follow: 577 / 584 / 560 us.)
struct HitExpand {
  uint32_t pid;
  const int32_t *T;  // input table
  uint32_t c, tr;    // input columns; probe tile rows
  const uint4 *hits;
  uint64_t ntiles;
  int32_t *O;        // known_to_unknown: rows x (c + 1); filters: rows x c
  // known_to_unknown: where the compacted rows go (null: nowhere)
  uint2 *cinfo;
  uint64_t *cexcl;
};

// Largest i in [0, n) with f(i) <= x, by the whole wave (f ascends, f(0) <= x).
template <class F>
__device__ __forceinline__ uint64_t wave_last_le(uint64_t n, uint64_t x, F f) {
  uint64_t lo = 0, hi = n;
  while (hi - lo > 1) {
    const uint64_t step = (hi - lo + kWave - 1) / kWave, i = lo + lane_id() * step;
    const uint32_t k = (uint32_t)__builtin_popcountll(wave_ballot(i < hi && f(i) <= x));
    lo += (k - 1) * step;
    hi = lo + step < hi ? lo + step : hi;
  }
  return lo;
}

typedef int32_t v4i32 __attribute__((ext_vector_type(4)));
// The block's nrows x nc output cells, cell(row, column), to out (16-byte
// aligned) as whole quads.
template <class F>
__device__ __forceinline__ void store_rows(int32_t *out, uint32_t nrows, uint32_t nc, F cell) {
  const uint32_t tid = threadIdx.x, nint = nrows * nc;
  for (uint32_t q = tid; q < nint / 4; q += kBlock) {
    uint32_t r = 4 * q / nc, col = 4 * q - r * nc;
    v4i32 v;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      v[k] = cell(r, col);
      if (++col == nc) {
        col = 0;
        r++;
      }
    }
    __builtin_nontemporal_store(v, (v4i32 *)out + q);
  }
  if (tid < (nint & 3)) {
    const uint32_t e = (nint & ~3u) + tid;
    out[e] = cell(e / nc, e % nc);
  }
}

// The tile (from t0, of nt tiles) of hit n0 + r: the last whose first hit is
// at most it (an empty tile shares its with the next). s_first: the tiles'
// first hits from n0, or null: then nzp is read.
template <class F>
__device__ __forceinline__ uint64_t hit_tile(uint64_t t0, uint32_t nt, uint64_t n0, uint32_t r, const uint32_t *s_first,
                                             F nzp) {
  uint32_t lo = 0, hi = nt - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (s_first ? s_first[mid] <= r : nzp(t0 + mid) <= n0 + r) lo = mid;
    else hi = mid - 1;
  }
  return t0 + lo;
}

// The tile and the hit (counted over all tiles) of output row o, by the whole wave.
template <class FP, class FN>
__device__ __forceinline__ void find_hit(const HitExpand &a, uint64_t o, FP pre, FN nzp, uint64_t &tile, uint64_t &hit) {
  tile = wave_last_le(a.ntiles, o, pre);
  const uint64_t n = nzp(tile), cnt = nzp(tile + 1) - n, local = o - pre(tile);
  hit = n + wave_last_le(cnt, local, [&](uint64_t k) -> uint64_t { return a.hits[tile * a.tr + k].w; });
}

// A block's LDS, shared by the two forms below.
template <int NV>
struct RowsLds {
  int32_t start[NV + 1];             // per hit: its first output row, from the block's first
  uint32_t off[NV + 1], row[NV + 1]; // per hit: list offset, input row
  uint32_t edge[NV];                 // per tile of the block (first), per output row (then)
  alignas(4) uint16_t map[NV];       // the hit that starts at an output row; then every row's hit
  uint64_t t[2], n[2];               // tile and hit of the block's first row and of its end
  uint32_t wmax[kBlock / kWave];
};

// Output rows [o0, o0 + nout), nout <= NV, of a known_to_unknown step. pre(t)
// and nzp(t): output rows and hits before tile t (nzp(ntiles): all hits). split:
// (tile, hit) of the block's first row and of the next block's (the last
// block's: of the last row), or null: then they are searched here. With
// compact, the hits that start in the block also go to cinfo / cexcl.
template <int NV, bool FRAMED, class FP, class FN>
__device__ __forceinline__ void expand_hits_block(RowsLds<NV> &lds, const GraphView &g, const HitExpand &a,
                                                  uint64_t o0, uint32_t nout, bool compact, const uint2 *split, FP pre, FN nzp) {
  constexpr int PER = NV / kBlock;
  auto &s_start = lds.start;
  auto &s_off = lds.off;
  auto &s_row = lds.row;
  auto &s_edge = lds.edge;
  auto &s_map = lds.map;
  auto &s_t = lds.t;
  auto &s_n = lds.n;
  auto &s_wmax = lds.wmax;
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  for (uint32_t i = tid; i < NV / 2; i += kBlock) ((uint32_t *)s_map)[i] = 0;
  if (split) {
    if (tid < 2) {
      const uint2 v = gload(split + tid);
      s_t[tid] = v.x;
      s_n[tid] = v.y;
    }
  } else if (wave < 2) {
    uint64_t t, n;
    find_hit(a, wave ? o0 + nout - 1 : o0, pre, nzp, t, n);
    if (lane == 0) {
      s_t[wave] = t;
      s_n[wave] = n;
    }
  }
  __syncthreads();
  const uint64_t t0 = s_t[0], n0 = s_n[0];
  const uint32_t nt = (uint32_t)(s_t[1] - t0 + 1), nr = (uint32_t)(s_n[1] - n0 + 1);
  const uint32_t c = a.c, nc = c + 1;
  const DevMeta mt = g.meta[a.pid];
  if (nt == 1 && c <= (uint32_t)NV && (nr == 1 || (nr == 2 && split))) {
    // The block may lie inside one hit (a hub's list; with splits nr also
    // counts the next block's hit): its row's cells and its run of the list
    // through LDS, no map. (A heavy query of 200M rows in the executor: 2499 us
    // through the map, 2210 so; 2M rows to 18M 145 -> 140 us.)
    const uint64_t i = t0 * a.tr + (n0 - nzp(t0));
    const uint4 h = gload(a.hits + i);
    const int64_t start = (int64_t)(pre(t0) + h.w) - (int64_t)o0;
    if (start + (int64_t)h.z >= (int64_t)nout) {  // (uniform)
      if (compact && start >= 0 && tid == 0) {
        gstore(a.cinfo + n0, make_uint2(h.x, h.y));
        gmem(a.cexcl)[n0] = o0 + (uint64_t)start;
      }
      for (uint32_t col = tid; col < c; col += kBlock) s_row[col] = (uint32_t)gmem(a.T)[(uint64_t)h.x * c + col];
      uint32_t ev[PER];
#pragma unroll
      for (int k = 0; k < PER; k++) {
        const uint32_t o = tid + k * kBlock;
        ev[k] = o < nout ? edge_at<FRAMED>(g, mt.edge_start, mt.eframe_base, h.y + (uint32_t)((int64_t)o - start)) : 0u;
      }
#pragma unroll
      for (int k = 0; k < PER; k++) s_edge[tid + k * kBlock] = ev[k];
      __syncthreads();
      store_rows(a.O + o0 * nc, nout, nc, [&](uint32_t r, uint32_t col) -> int32_t {
        return (int32_t)(col < c ? s_row[col] : s_edge[r]);
      });
      return;
    }
  }
  const bool staged = nt <= (uint32_t)NV;  // the tiles' first hits, from n0, fit s_edge
  if (staged && nt > 1) {
    for (uint32_t i = tid; i < nt; i += kBlock) {
      const uint64_t n = nzp(t0 + i);
      s_edge[i] = n > n0 ? (uint32_t)(n - n0) : 0u;
    }
    __syncthreads();
  }
  for (uint32_t r = tid; r < nr; r += kBlock) {
    const uint64_t t = hit_tile(t0, nt, n0, r, staged ? s_edge : nullptr, nzp);
    const uint4 h = gload(a.hits + t * a.tr + (n0 + r - nzp(t)));
    const int64_t start = (int64_t)(pre(t) + h.w) - (int64_t)o0;
    s_start[r] = (int32_t)start;
    s_row[r] = h.x;
    s_off[r] = h.y;
    // (hit 0 starts at or before the block's first row; the next block's hit may start at its first)
    const bool inside = start < (int64_t)nout;
    if (r && inside) s_map[start] = (uint16_t)r;
    if (compact && start >= 0 && inside) {
      gstore(a.cinfo + n0 + r, make_uint2(h.x, h.y));
      gmem(a.cexcl)[n0 + r] = o0 + (uint64_t)start;
    }
  }
  __syncthreads();
  // every output row's hit: the last that starts at or before it
  uint32_t hit[PER], m = 0;
#pragma unroll
  for (int k = 0; k < PER; k++) {
    const uint32_t v = s_map[tid * PER + k];
    m = v > m ? v : m;
    hit[k] = m;
  }
  uint32_t run = m;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t y = shfl32(run, (lane - d) & 63);
    if (lane >= (uint32_t)d && y > run) run = y;
  }
  if (lane == kWave - 1) s_wmax[wave] = run;
  uint32_t base = shfl32(run, (lane - 1) & 63);  // (by every lane: a masked lane's value cannot be read)
  if (lane == 0) base = 0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kBlock / kWave - 1; w++)
    if (w < (int)wave && s_wmax[w] > base) base = s_wmax[w];
  uint32_t ev[PER];
#pragma unroll
  for (int k = 0; k < PER; k++) {
    hit[k] = hit[k] > base ? hit[k] : base;
    const uint32_t o = tid * PER + k;
    ev[k] = o < nout ? edge_at<FRAMED>(g, mt.edge_start, mt.eframe_base,
                                       s_off[hit[k]] + (uint32_t)((int32_t)o - s_start[hit[k]]))
                     : 0u;
  }
#pragma unroll
  for (int k = 0; k < PER; k++) {
    s_map[tid * PER + k] = (uint16_t)hit[k];
    s_edge[tid * PER + k] = ev[k];
  }
  __syncthreads();
  // the block's output is contiguous and (NV being a multiple of 4) 16-byte aligned
  store_rows(a.O + o0 * nc, nout, nc, [&](uint32_t r, uint32_t col) -> int32_t {
    return col < c ? gmem(a.T)[(uint64_t)s_row[s_map[r]] * c + col] : (int32_t)s_edge[r];
  });
}

// Kept rows [o0, o0 + nout) of a filter step (a hit each).
template <int NV, class FN>
__device__ __forceinline__ void compact_hits_block(RowsLds<NV> &lds, const HitExpand &a, uint64_t o0, uint32_t nout,
                                                   FN nzp) {
  auto &s_row = lds.row;
  auto &s_t = lds.t;  // tile of the block's first and last row
  const uint32_t tid = threadIdx.x, wave = tid / kWave;
  if (wave < 2) {
    const uint64_t t = wave_last_le(a.ntiles, wave ? o0 + nout - 1 : o0, nzp);
    if (lane_id() == 0) s_t[wave] = t;
  }
  __syncthreads();
  const uint64_t t0 = s_t[0];
  const uint32_t nt = (uint32_t)(s_t[1] - t0 + 1);
  for (uint32_t r = tid; r < nout; r += kBlock) {
    const uint64_t t = hit_tile(t0, nt, o0, r, nullptr, nzp);
    s_row[r] = gload(a.hits + t * a.tr + (o0 + r - nzp(t))).x;
  }
  __syncthreads();
  const uint32_t c = a.c;
  store_rows(a.O + o0 * c, nout, c, [&](uint32_t r, uint32_t col) -> int32_t {
    return gmem(a.T)[(uint64_t)s_row[r] * c + col];
  });
}

// Large known_to_unknown outputs, after the tile scan (E < 2^32): the
// blocks' first hits by one wave each, then the blocks. (Searched in the
// blocks themselves the five dependent reads were half of a block's chain:
// 2M rows to 18M of 4 cells 152 us a step, 146 with the splits.)
struct ScannedTiles {
  const uint64_t *tile_sum, *tile_nz, *chunk_sum, *chunk_nz;
  uint64_t nz, E;
  uint64_t block0;  // the launch's first block of kHitNV rows
  uint2 *split;     // per block (+1): (tile, hit) of its first row
  __device__ __forceinline__ uint64_t pre(uint64_t i) const { return tile_sum[i] + chunk_sum[i / kScanChunk]; }
  __device__ __forceinline__ uint64_t nzp(uint64_t i, uint64_t ntiles) const {
    return i >= ntiles ? nz : tile_nz[i] + chunk_nz[i / kScanChunk];
  }
};
__global__ __launch_bounds__(kBlock) void k_hit_splits(HitExpand a, ScannedTiles t, uint64_t nblocks) {
  const uint64_t b = blockIdx.x * (uint64_t)(kBlock / kWave) + threadIdx.x / kWave;
  if (b > nblocks) return;
  uint64_t tile, hit;
  find_hit(a, b < nblocks ? b * kHitNV : t.E - 1, [&](uint64_t i) -> uint64_t { return t.pre(i); },
           [&](uint64_t i) -> uint64_t { return t.nzp(i, a.ntiles); }, tile, hit);
  if (lane_id() == 0) t.split[b] = make_uint2((uint32_t)tile, (uint32_t)hit);
}
template <bool FRAMED>
__global__ __launch_bounds__(kBlock) void k_expand_hits(GraphView g, HitExpand a, ScannedTiles t) {
  const uint64_t b = t.block0 + blockIdx.x, o0 = b * (uint64_t)kHitNV;
  const uint32_t nout = (uint32_t)(t.E - o0 < (uint64_t)kHitNV ? t.E - o0 : (uint64_t)kHitNV);
  __shared__ RowsLds<kHitNV> s_rows;
  expand_hits_block<kHitNV, FRAMED>(
      s_rows, g, a, o0, nout, a.cinfo != nullptr, t.split + b, [&](uint64_t i) -> uint64_t { return t.pre(i); },
      [&](uint64_t i) -> uint64_t { return t.nzp(i, a.ntiles); });
}

// ---- the second launch of a step of at most kScanChunk tiles ----
// Every workgroup scans the tile sums itself (a read of 16 B per tile and one
// block scan), so no scan kernel runs between the probe and this one, and
// the first workgroup publishes the step's counts. It is queued right behind
// the probe, before the host knows the counts, into a table of `cap` rows:
//  - filters (cap: the input's rows) copy their kept rows;
//  - a known_to_unknown whose E rows fit cap expands them, and keeps the
//    compacted rows when it fans out (E >= 4 hits);
//  - one whose output does not fit compacts its hits (cinfo / cexcl, with
//    64-bit offsets) for the expand that the host launches into a table of
//    E rows.
struct FollowStep {
  int mode;
  uint64_t cap;
  const uint64_t *tile_sum, *tile_nz, *tile_ex;  // the probe's, not scanned
  uint64_t *totals;
  Signal sg;
};
template <bool FRAMED>
__global__ __launch_bounds__(kBlock) void k_follow(GraphView g, HitExpand a, FollowStep f) {
  constexpr int PT = kScanChunk / kBlock;
  __shared__ RowsLds<kFollowNV> s_rows;
  __shared__ uint64_t s_pre[kScanChunk];
  __shared__ uint32_t s_nzp[kScanChunk + 1];
  __shared__ uint64_t s_tmp[2 * (kBlock / kWave)];
  const uint32_t tid = threadIdx.x, lane = lane_id(), n = (uint32_t)a.ntiles;
  const uint32_t lo = tid * PT;
  uint64_t vs[PT], vn[PT], v[2] = {0, 0}, tot[2];
#pragma unroll
  for (int k = 0; k < PT; k++) {
    vs[k] = lo + k < n ? f.tile_sum[lo + k] : 0;
    vn[k] = lo + k < n ? f.tile_nz[lo + k] : 0;
  }
#pragma unroll
  for (int k = 0; k < PT; k++) {
    v[0] += vs[k];
    v[1] += vn[k];
  }
  block_excl_scan_n<2>(v, s_tmp, tot);
  const uint64_t E = tot[0], nz = tot[1];
  if (blockIdx.x == 0) {
    uint64_t e = 0, ex;
    for (uint32_t i = tid; i < n; i += kBlock) e += f.tile_ex[i];
    (void)block_excl_scan(e, s_tmp, ex);
    if (tid == 0) {
      const uint64_t w[3] = {E, ex, nz};
      f.totals[0] = E;
      f.totals[1] = ex;
      f.totals[2] = nz;
      publish(f.sg, w, 3);
    }
  }
#pragma unroll
  for (int k = 0; k < PT; k++) {
    if (lo + k < n) {
      s_pre[lo + k] = v[0];
      s_nzp[lo + k] = (uint32_t)v[1];
    }
    v[0] += vs[k];
    v[1] += vn[k];
  }
  if (tid == 0) s_nzp[n] = (uint32_t)nz;
  __syncthreads();
  auto pre = [&](uint64_t t) -> uint64_t { return s_pre[t]; };
  auto nzp = [&](uint64_t t) -> uint64_t { return s_nzp[t]; };
  if (E > f.cap) {  // (known_to_unknown) one wave per tile
    for (uint32_t t = blockIdx.x * (kBlock / kWave) + tid / kWave; t < n; t += gridDim.x * (kBlock / kWave)) {
      const uint64_t n0 = s_nzp[t], out0 = s_pre[t];
      const uint32_t cnt = (uint32_t)(s_nzp[t + 1] - n0);
      uint64_t carry = 0;
      for (uint32_t k0 = 0; k0 < cnt; k0 += kWave) {
        const uint32_t j = k0 + lane;
        const uint4 h = j < cnt ? gload(a.hits + (uint64_t)t * a.tr + j) : make_uint4(0, 0, 0, 0);
        const uint64_t inc = wave_incl_scan(h.z);
        if (j < cnt) {
          gstore(a.cinfo + n0 + j, make_uint2(h.x, h.y));
          gmem(a.cexcl)[n0 + j] = out0 + carry + inc - h.z;
        }
        carry += shfl64(inc, kWave - 1);
      }
    }
    return;
  }
  constexpr uint64_t NV = kFollowNV;
  for (uint64_t o0 = blockIdx.x * NV; o0 < E; o0 += gridDim.x * NV) {
    const uint32_t nout = (uint32_t)(E - o0 < NV ? E - o0 : NV);
    if (f.mode == kModeK2U)
      expand_hits_block<kFollowNV, FRAMED>(s_rows, g, a, o0, nout, a.cinfo && E >= 4 * nz, nullptr, pre, nzp);
    else
      compact_hits_block<kFollowNV>(s_rows, a, o0, nout, nzp);
    __syncthreads();  // the block's LDS is reused
  }
}

// ---- a whole small query in one workgroup ----
// Every step of a query whose tables stay small runs in one 1024-thread
// workgroup with every table in LDS (two ping-pong tables of kSQCells
// cells), so the only global accesses are the graph's buckets and lists and
// the final copy of the result to the host:
//  - an index / constant start: wave 0 probes the key, the workgroup copies
//    its list into the table;
//  - a known-start step: wave w probes rows [64 w r, 64 (w + 1) r) of the
//    input (r = rounds of 64 rows, at most 4), filters test membership with
//    the probe pass's search, then a workgroup scan of the degrees (kept
//    flags) gives every row its first output row; known_to_unknown writes
//    output row k = (the last row whose first output row is <= k, its list
//    entry k - that first row), filters copy the kept rows in order. Output
//    order is the reference's (core/engine.hpp:126-194).
// A table past the caps ends the query early with status 1 (the caller then
// runs it step by step), so the result is always the per-step path's.
// Two kernels run this body: k_small_query, one launch per query, and
// k_sq_server, a persistent server that takes queries from a ring in pinned
// host memory as they arrive.
constexpr int kSQThreads = 1024;
constexpr int kSQWaves = kSQThreads / kWave;
constexpr uint32_t kSQSteps = 8;        // patterns
constexpr uint32_t kSQRows = 4096;      // input rows of a known-start step
constexpr uint32_t kSQCells = 8192;     // cells of a table (32 KB)
constexpr int kSQHalf = 4;  // list entries / output rows a thread gathers at once
static_assert(kSQCells * 4 <= kStageBytes, "a small query's result fits the staging area");
struct SmallQuery {
  wkg_plan_step steps[kSQSteps];
  DevMeta meta[kSQSteps];  // each step's predicate metadata (passed in, not loaded)
  uint32_t nsteps;
  uint32_t pad[15];
};
static_assert(sizeof(SmallQuery) % 64 == 0, "whole cache lines");

struct SQShared {
  WaveProbeLds wp[kSQWaves];
  uint32_t deg[kSQRows];  // degree (known_to_unknown) or kept flag (filters)
  uint32_t off[kSQRows];  // list offset (known_to_unknown)
  uint32_t pos[kSQRows];  // first output row
  alignas(16) int32_t tab[2][kSQCells];
  uint64_t tmp[2][kSQWaves];
  SmallQuery q;           // the query (copied in)
};

// Exclusive u64 scan over the kSQThreads threads; `total` gets the sum.
__device__ __forceinline__ uint64_t sq_block_scan(uint64_t v, uint64_t *tmp, uint64_t &total) {
  const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
  const uint64_t inc = wave_incl_scan(v);
  if (lane == kWave - 1) tmp[wave] = inc;
  __syncthreads();
  uint64_t pre = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < kSQWaves; w++) {
    const uint64_t t = tmp[w];
    if ((uint32_t)w < wave) pre += t;
    tot += t;
  }
  __syncthreads();
  total = tot;
  return pre + inc - v;
}

__device__ __forceinline__ uint32_t sq_uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ uint64_t sq_uniform(uint64_t v) {
  return ((uint64_t)sq_uniform((uint32_t)(v >> 32)) << 32) | sq_uniform((uint32_t)v);
}

// Runs sh.q; wave 0 writes the result table to dst (rows x cols cells, 16-
// byte aligned) unless the status is 1. res = {status, rows, cols,
// expanded, the step that declined}. Every thread of the workgroup calls
// it; wave 0 then releases its stores to the host.
template <bool SORTED, bool FRAMED>
__device__ __forceinline__ void sq_run(const GraphView &g, SQShared &sh, int32_t *dst, uint64_t (&res)[5]) {
  const SmallQuery &q = sh.q;
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  uint64_t expanded = 0, status = 0;
  uint32_t rows = 0, cols = 0, cur = 0, l = 0;
  const uint32_t nsteps = sq_uniform((uint32_t)q.nsteps);
  for (; l < nsteps; l++) {
    // the step and its metadata are the same in every lane: into scalar registers
    wkg_plan_step d;
    d.kind = (int32_t)sq_uniform((uint32_t)q.steps[l].kind);
    d.pid = (int32_t)sq_uniform((uint32_t)q.steps[l].pid);
    d.dir = (int32_t)sq_uniform((uint32_t)q.steps[l].dir);
    d.start_col = (int32_t)sq_uniform((uint32_t)q.steps[l].start_col);
    d.end_col = (int32_t)sq_uniform((uint32_t)q.steps[l].end_col);
    d.vid = (int64_t)sq_uniform((uint64_t)q.steps[l].vid);
    DevMeta m;
    m.main_start = sq_uniform(q.meta[l].main_start);
    m.psz = sq_uniform(q.meta[l].psz);
    m.magic = sq_uniform(q.meta[l].magic);
    m.indrct_start = sq_uniform(q.meta[l].indrct_start);
    m.edge_start = sq_uniform(q.meta[l].edge_start);
    m.edge_len = 0;
    m.vframe_base = sq_uniform(q.meta[l].vframe_base);
    m.eframe_base = sq_uniform(q.meta[l].eframe_base);
    const int32_t *in = sh.tab[cur];
    int32_t *out = sh.tab[cur ^ 1];
    if (d.kind == WKG_STEP_I2U || d.kind == WKG_STEP_C2U) {  // one key: its list is the table
      const uint64_t key = d.kind == WKG_STEP_I2U ? make_key(0, (uint64_t)d.pid, (uint64_t)d.dir)
                                                  : make_key((uint64_t)d.vid, (uint64_t)d.pid, (uint64_t)d.dir);
      if (wave == 0) {
        uint32_t deg, off;
        ProbeCarry carry;
        wave_probe<FRAMED>(g, m, lane == 0 ? key : 0, sh.wp[0], deg, off, carry);
        if (lane == 0) {
          sh.deg[0] = deg;
          sh.off[0] = off;
        }
      }
      __syncthreads();
      const uint32_t deg = sh.deg[0], off = sh.off[0];
      expanded += deg;
      if (deg > kSQCells) {
        status = 1;
        break;
      }
#pragma unroll 1
      for (uint32_t j0 = 0; j0 < deg; j0 += kSQHalf * kSQThreads) {
        uint32_t v[kSQHalf];  // a thread's list loads in flight together
#pragma unroll
        for (int k = 0; k < kSQHalf; k++) {
          const uint32_t j = j0 + tid + k * kSQThreads;
          if (j < deg) v[k] = edge_at<FRAMED>(g, m.edge_start, m.eframe_base, (uint64_t)off + j);
        }
#pragma unroll
        for (int k = 0; k < kSQHalf; k++) {
          const uint32_t j = j0 + tid + k * kSQThreads;
          if (j < deg) out[j] = (int32_t)v[k];
        }
      }
      rows = deg;
      cols = 1;
    } else {
      if (rows > kSQRows) {
        status = 1;
        break;
      }
      const int mode = d.kind == WKG_STEP_K2U ? kModeK2U : d.kind == WKG_STEP_K2K ? kModeK2K : kModeK2C;
      const uint32_t sc = (uint32_t)d.start_col, ec = mode == kModeK2K ? (uint32_t)d.end_col : 0u;
      const bool target_ok = mode == kModeK2C && d.vid >= 0 && d.vid <= 0xffffffffLL;
      const uint32_t rounds = (rows + kSQThreads - 1) / kSQThreads;  // 64-row rounds of a wave
      ProbeCarry carry;
      uint64_t ex = 0;  // filters: edges examined by this lane's rows
      for (uint32_t rd = 0; rd < rounds; rd++) {
        const uint32_t row = (wave * rounds + rd) * kWave + lane;
        uint64_t key = 0;
        int32_t end_cell = -1;
        if (row < rows) {
          const int32_t cell = in[row * cols + sc];
          if (cell >= 0) key = make_key((uint32_t)cell, (uint64_t)d.pid, (uint64_t)d.dir);
          if (mode == kModeK2K) end_cell = in[row * cols + ec];
        }
        uint32_t deg, off;
        wave_probe<FRAMED>(g, m, key, sh.wp[wave], deg, off, carry);
        if (mode == kModeK2U) {
          if (row < rows) {
            sh.deg[row] = deg;
            sh.off[row] = off;
          }
        } else {
          bool my_found;
          uint32_t my_ex;
          rows_member<SORTED, FRAMED>(g, m.edge_start, m.eframe_base, off, deg,
                                      mode == kModeK2K ? (uint32_t)end_cell : (uint32_t)d.vid,
                                      mode == kModeK2K ? end_cell >= 0 : target_ok, my_found, my_ex);
          if (row < rows) sh.deg[row] = my_found ? 1u : 0u;
          ex += my_ex;
        }
      }
      __syncthreads();
      // thread t owns rows [t r, t r + r) of the scan
      uint64_t cnt = 0;
      for (uint32_t k = 0; k < rounds; k++) {
        const uint32_t row = tid * rounds + k;
        if (row < rows) cnt += sh.deg[row];
      }
      uint64_t total, ex_total = 0;
      uint64_t pre = sq_block_scan(cnt, sh.tmp[0], total);
      if (mode != kModeK2U) (void)sq_block_scan(ex, sh.tmp[1], ex_total);
      for (uint32_t k = 0; k < rounds; k++) {
        const uint32_t row = tid * rounds + k;
        if (row < rows) {
          sh.pos[row] = (uint32_t)pre;  // (a total past the caps declines below before any use)
          pre += sh.deg[row];
        }
      }
      __syncthreads();
      if (mode == kModeK2U) {
        expanded += total;
        const uint32_t nc = cols + 1;
        if (total * nc > kSQCells) {
          status = 1;
          break;
        }
        const uint32_t E = (uint32_t)total;  // <= kSQCells
#pragma unroll 1
        for (uint32_t r0 = 0; r0 < E; r0 += kSQHalf * kSQThreads) {  // kSQHalf output rows a thread at once
          uint32_t par[kSQHalf], v[kSQHalf];
#pragma unroll
          for (int k = 0; k < kSQHalf; k++) {  // the last row whose first output row is <= r
            const uint32_t r = r0 + tid + k * kSQThreads;
            uint32_t lo = 0;
#pragma unroll
            for (uint32_t step = kSQRows / 2; step; step >>= 1)
              if (lo + step < rows && sh.pos[lo + step] <= r) lo += step;
            par[k] = lo;
          }
#pragma unroll
          for (int k = 0; k < kSQHalf; k++) {  // the gathered edges in flight together
            const uint32_t r = r0 + tid + k * kSQThreads;
            if (r < E) v[k] = edge_at<FRAMED>(g, m.edge_start, m.eframe_base, (uint64_t)sh.off[par[k]] + (r - sh.pos[par[k]]));
          }
#pragma unroll
          for (int k = 0; k < kSQHalf; k++) {
            const uint32_t r = r0 + tid + k * kSQThreads;
            if (r < E) {
              int32_t *o = out + r * nc;
              for (uint32_t j = 0; j < cols; j++) o[j] = in[par[k] * cols + j];
              o[cols] = (int32_t)v[k];
            }
          }
        }
        rows = E;
        cols = nc;
      } else {
        expanded += ex_total;
        for (uint32_t row = tid; row < rows; row += kSQThreads)
          if (sh.deg[row])
            for (uint32_t j = 0; j < cols; j++) out[sh.pos[row] * cols + j] = in[row * cols + j];
        rows = (uint32_t)total;
      }
    }
    __syncthreads();  // the output is complete before it is the next step's input
    cur ^= 1;
  }
  // the result to the host: wave 0 alone (one wave's system-scope release
  // then covers every store), 16 bytes a lane
  if (status == 0 && wave == 0) {
    const uint32_t cells = rows * cols, nq = cells / 4;
    const uint4 *src = (const uint4 *)sh.tab[cur];
    for (uint32_t i = lane; i < nq; i += kWave) ((uint4 *)dst)[i] = src[i];
    if (lane < cells - 4 * nq) dst[4 * nq + lane] = sh.tab[cur][4 * nq + lane];
  }
  res[0] = status;
  res[1] = rows;
  res[2] = cols;
  res[3] = expanded;
  res[4] = l;
}

// One query, one launch: the result into the pinned staging area, then
// {status, rows, cols, expanded} and the flag.
template <bool SORTED, bool FRAMED>
__global__ __launch_bounds__(kSQThreads) void k_small_query(GraphView g, SmallQuery q, int32_t *stage, Signal sg) {
  __shared__ SQShared sh;
  if (threadIdx.x == 0) sh.q = q;
  __syncthreads();
  uint64_t res[5];
  sq_run<SORTED, FRAMED>(g, sh, stage, res);
  if (threadIdx.x < kWave) {
    __threadfence_system();
    if (threadIdx.x == 0) publish(sg, res, 5);
  }
}

// ---- the persistent small-query server ----
// A ring of slots in pinned host memory: the host writes a query into slot
// t mod nslots, then publishes t + 1 as the ring's tail. Each workgroup of
// k_sq_server claims the next unclaimed ticket (a compare-and-swap on a
// device-memory head counter, so every ticket is taken once, in order),
// copies the query into LDS, runs it, writes the result table and
// {status, rows, cols, expanded, device ticks} into the slot, then t + 1 as
// the slot's done word (system-scope release). A workgroup exits when no
// ticket arrived for idle_ticks, when it has run for life_ticks, or when
// the host sets stop; every wait is bounded by those clocks (the device's
// constant wall clock), so the grid always drains. Queries arriving while
// others run are admitted as soon as a workgroup is free.
struct SQResp {
  uint64_t status, rows, cols, expanded, ticks;
  uint64_t step;  // status 1: the step that outgrew the limits
  uint64_t pad;
  uint64_t done;  // ticket + 1, written last
};
struct SQSlot {
  SmallQuery q;
  SQResp resp;
  int32_t cells[kSQCells];
};
struct SQBox {
  const uint64_t *tail;  // pinned: tickets issued (host-written)
  const uint64_t *stop;  // pinned: nonzero asks the workgroups to exit
  uint64_t *head;        // device memory: tickets claimed
  SQSlot *slots;         // pinned ring (device address)
  uint64_t nslots;       // a power of two
  uint64_t idle_ticks, life_ticks;
};
constexpr uint64_t kSQNoClaim = ~uint64_t(0);

template <bool SORTED>
__global__ __launch_bounds__(kSQThreads) void k_sq_server(GraphView g, SQBox box) {
  __shared__ SQShared sh;
  __shared__ uint64_t s_claim;
  const uint64_t t_start = wall_clock64();
  uint64_t t_idle = t_start;  // (thread 0) since when the ring is idle
  // (thread 0) the head as last seen: a stale value only fails one
  // compare-and-swap, which returns the current one
  uint64_t h = threadIdx.x == 0 ? __hip_atomic_load(box.head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
  for (;;) {
    if (threadIdx.x == 0) {
      uint64_t claim = kSQNoClaim;
      for (;;) {
        const uint64_t now = wall_clock64();
        if (now - t_start > box.life_ticks || now - t_idle > box.idle_ticks) break;
        // (both words on their way at once: a poll is one round trip over
        // the bus, not two: a 2-hop query of 1000 rows 22.9 -> 22.3 us)
        const uint64_t stop = __hip_atomic_load(box.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        const uint64_t tail = __hip_atomic_load(box.tail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (stop) break;
        if (h < tail) {
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");
          if (__hip_atomic_compare_exchange_strong(box.head, &h, h + 1, __ATOMIC_ACQUIRE, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT)) {
            claim = h++;
            break;
          }
          continue;  // another workgroup took it (h is now the current head)
        }
        __builtin_amdgcn_s_sleep(4);
      }
      s_claim = claim;
    }
    __syncthreads();
    const uint64_t claim = s_claim;
    if (claim == kSQNoClaim) break;
    const uint64_t t0 = wall_clock64();
    SQSlot *slot = box.slots + (claim & (box.nslots - 1));
    // the query into LDS, word by word past every cache
    const uint32_t *src = (const uint32_t *)&slot->q;
    uint32_t *qw = (uint32_t *)&sh.q;
    for (uint32_t i = threadIdx.x; i < sizeof(SmallQuery) / 4; i += kSQThreads)
      qw[i] = __hip_atomic_load(src + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __syncthreads();
    uint64_t res[5];
    sq_run<SORTED, false>(g, sh, slot->cells, res);
    // (wave 0 wrote the cells: the release of the done word by its lane 0
    // waits for the wave's stores, so they need no round trip of their own)
    if (threadIdx.x < kWave) wave_lds_sync();
    if (threadIdx.x == 0) {
      slot->resp.status = res[0];
      slot->resp.rows = res[1];
      slot->resp.cols = res[2];
      slot->resp.expanded = res[3];
      slot->resp.step = res[4];
      slot->resp.ticks = wall_clock64() - t0;
      __hip_atomic_store(&slot->resp.done, claim + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
      t_idle = wall_clock64();
    }
    __syncthreads();  // s_claim and sh are reused
  }
}

// A small table to the host: copies n cells into the pinned staging area,
// then publishes (every wave's stores complete at system scope first).
__global__ __launch_bounds__(kBlock) void k_stage(const int32_t *src, uint64_t n, int32_t *dst, Signal sg) {
  for (uint64_t i = threadIdx.x; i < n; i += kBlock) dst[i] = src[i];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) publish(sg, nullptr, 0);
}

// Index / const start in one launch: wave 0 probes the key; when the list
// has at most `cap` entries the workgroup copies it to out; then the degree
// and offset are published.
constexpr uint64_t kListCap = 8192;
template <bool FRAMED>
__global__ __launch_bounds__(kBlock) void k_probe_copy(GraphView g, uint64_t key, uint32_t pid, uint64_t cap,
                                                       int32_t *out, Signal sg) {
  __shared__ WaveProbeLds s_wp;
  __shared__ uint32_t s_deg, s_off;
  const DevMeta m = g.meta[pid];
  if (threadIdx.x < kWave) {
    uint32_t deg, off;
    ProbeCarry carry;
    wave_probe<FRAMED>(g, m, threadIdx.x == 0 ? key : 0, s_wp, deg, off, carry);
    if (threadIdx.x == 0) {
      s_deg = deg;
      s_off = off;
    }
  }
  __syncthreads();
  const uint64_t deg = s_deg, off = s_off;
  if (deg <= cap)
    for (uint64_t j = threadIdx.x; j < deg; j += kBlock) out[j] = (int32_t)edge_at<FRAMED>(g, m.edge_start, m.eframe_base, off + j);
  if (threadIdx.x == 0) {
    const uint64_t v[2] = {deg, off};
    publish(sg, v, 2);
  }
}

// out[j] = list[j] for j < n, the list starting at segment offset `off` of pid.
template <bool FRAMED>
__global__ __launch_bounds__(kBlock) void k_copy_list(GraphView g, uint32_t pid, uint64_t off, uint64_t n,
                                                      int32_t *out) {
  const DevMeta m = g.meta[pid];
  for (uint64_t j = blockIdx.x * (uint64_t)kBlock + threadIdx.x; j < n; j += (uint64_t)gridDim.x * kBlock)
    out[j] = (int32_t)edge_at<FRAMED>(g, m.edge_start, m.eframe_base, off + j);
}

// ---- known_to_unknown on an inherited column (probe once per parent row) ----
// A known_to_unknown output repeats compacted input row i (parent row
// info_p[i].x) in its rows [excl_p[i], excl_p[i+1]). A later step whose key
// column is one of the parent's gathers that key once per compacted parent
// row (k_gather_col), probes those keys as a one-column table, and spreads
// each kept parent row (m, with d list entries) back to its f child rows:
// child k of it gets output rows [out_pre[m] + k d, out_pre[m] + (k+1) d).

// K[i] = T[info[i].x * c + sc]
__global__ __launch_bounds__(kBlock) void k_gather_col(const int32_t *T, uint32_t c, uint32_t sc, const uint2 *info,
                                                       uint64_t n, int32_t *K) {
  for (uint64_t i = blockIdx.x * (uint64_t)kBlock + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kBlock)
    K[i] = T[(uint64_t)info[i].x * c + sc];
}

// The kept parent rows: m < nk is key-table row info2[m].x (a compacted
// parent row i) with list length d = excl2[m+1] - excl2[m] (the last: dtot -
// excl2[m]); its child rows number f = excl_p[i+1] - excl_p[i] (the last
// compacted row's: rows - excl_p[i]).
struct KeptRows {
  const uint2 *info2;
  const uint64_t *excl2;
  uint64_t nk, dtot;
  const uint64_t *excl_p;
  uint64_t np, rows;
  __device__ __forceinline__ uint64_t deg(uint64_t m) const { return (m + 1 < nk ? excl2[m + 1] : dtot) - excl2[m]; }
  __device__ __forceinline__ uint64_t fan(uint32_t i) const {
    return (i + 1 < np ? excl_p[i + 1] : rows) - excl_p[i];
  }
};

// cnt[m] = f, out[m] = f d
__global__ __launch_bounds__(kBlock) void k_lift(KeptRows k, uint64_t *cnt, uint64_t *out) {
  for (uint64_t m = blockIdx.x * (uint64_t)kBlock + threadIdx.x; m < k.nk; m += (uint64_t)gridDim.x * kBlock) {
    const uint64_t f = k.fan(k.info2[m].x);
    cnt[m] = f;
    out[m] = f * k.deg(m);
  }
}

// Kept child row j (of kc): its parent m is the last with cnt_pre(m) <= j
// (cnt_pre strictly ascends: every compacted parent row has a child). The
// prefixes are the two-level tile scan's: chunk-local value + chunk prefix.
__global__ __launch_bounds__(kBlock) void k_spread(KeptRows k, const uint64_t *cnt_loc, const uint64_t *cnt_chunk,
                                                   const uint64_t *out_loc, const uint64_t *out_chunk, uint64_t kc,
                                                   uint2 *cinfo, uint64_t *cexcl) {
  auto cnt_pre = [&](uint64_t m) { return cnt_loc[m] + cnt_chunk[m / kScanChunk]; };
  for (uint64_t j = blockIdx.x * (uint64_t)kBlock + threadIdx.x; j < kc; j += (uint64_t)gridDim.x * kBlock) {
    uint64_t lo = 0, hi = k.nk;  // cnt_pre(lo) <= j < cnt_pre(hi)
    while (hi - lo > 1) {
      const uint64_t mid = (lo + hi) >> 1;
      if (cnt_pre(mid) <= j) lo = mid;
      else hi = mid;
    }
    const uint64_t kk = j - cnt_pre(lo);
    const uint2 pi = k.info2[lo];
    cinfo[j] = make_uint2((uint32_t)(k.excl_p[pi.x] + kk), pi.y);
    cexcl[j] = out_loc[lo] + out_chunk[lo / kScanChunk] + kk * k.deg(lo);
  }
}

// ---- filters on a star arm's output (decide once per parent group) ----
// An output A of the inherited-column known_to_unknown above consists of
// groups: group m < ng is kept key row m, i.e. grandparent row ginfo[m].x
// whose list (segment offset ginfo[m].y, d_m = gs[m+1] - gs[m] entries)
// was joined to each of its f_m child rows. Its rows are
// [go[m], go[m] + f_m d_m), child by child, so row r of group m holds list
// entry (r - go[m]) mod d_m in its last column and the grandparent row's
// cells in its first columns. A known_to_known / known_to_const step from
// that last column (with a grandparent column as the end) gives the same
// answer for all f_m rows that hold one entry: it is decided once per
// (group, entry) -- the d_m rows of a table S -- and each decision is
// counted f_m times.

// Group m's first child row of the output, its grandparent row and list.
__global__ __launch_bounds__(kBlock) void k_keep_groups(KeptRows k, const uint2 *pinfo, const uint64_t *out_loc,
                                                        const uint64_t *out_chunk, uint2 *ginfo, uint64_t *gs,
                                                        uint64_t *go) {
  for (uint64_t m = blockIdx.x * (uint64_t)kBlock + threadIdx.x; m < k.nk; m += (uint64_t)gridDim.x * kBlock) {
    const uint2 i2 = k.info2[m];
    ginfo[m] = make_uint2(pinfo[i2.x].x, i2.y);
    gs[m] = k.excl2[m];
    go[m] = out_loc[m] + out_chunk[m / kScanChunk];
  }
}

// The groups of an arm that was probed row by row: the arm's compacted rows
// (cinfo, cexcl: nz rows, E output rows) hold all child rows of a kept parent
// row i or none, so its first child row is searched among them.
struct ArmRows {
  const uint2 *cinfo;
  const uint64_t *cexcl;
  uint64_t nz, E;
  const uint2 *pinfo;      // the input's lineage: parent row of compacted row i,
  const uint64_t *excl_p;  // and its first child row
  uint64_t np;
  __device__ __forceinline__ bool find(uint64_t i, uint64_t &at) const {
    const uint64_t r = excl_p[i];
    uint64_t lo = 0, hi = nz;
    while (lo < hi) {
      const uint64_t mid = (lo + hi) >> 1;
      if (cinfo[mid].x < r) lo = mid + 1;
      else hi = mid;
    }
    at = lo;
    return lo < nz && cinfo[lo].x == r;
  }
};

// Parent row i: its list's length (0: not kept) and whether it is kept.
__global__ __launch_bounds__(kBlock) void k_arm_lift(ArmRows a, uint64_t *deg, uint64_t *kept) {
  for (uint64_t i = blockIdx.x * (uint64_t)kBlock + threadIdx.x; i < a.np; i += (uint64_t)gridDim.x * kBlock) {
    uint64_t at;
    const bool k = a.find(i, at);
    deg[i] = k ? (at + 1 < a.nz ? a.cexcl[at + 1] : a.E) - a.cexcl[at] : 0;
    kept[i] = k;
  }
}

// The kept parent rows' groups, as k_keep_groups'; the prefixes are the
// two-level scan's of what k_arm_lift wrote.
__global__ __launch_bounds__(kBlock) void k_arm_groups(ArmRows a, StepParams q, uint2 *ginfo, uint64_t *gs,
                                                       uint64_t *go) {
  for (uint64_t i = blockIdx.x * (uint64_t)kBlock + threadIdx.x; i < a.np; i += (uint64_t)gridDim.x * kBlock) {
    uint64_t at;
    if (!a.find(i, at)) continue;
    const uint64_t m = q.tile_nz[i] + q.chunk_nz[i / kScanChunk];
    ginfo[m] = make_uint2(a.pinfo[i].x, a.cinfo[at].y);
    gs[m] = q.tile_sum[i] + q.chunk_sum[i / kScanChunk];
    go[m] = a.cexcl[at];
  }
}

// The group table: G[m] = (end cell of the grandparent row (0 without an
// end column), f_m), the list of G row m at segment offset ginfo[m].y.
__global__ __launch_bounds__(kBlock) void k_group_table(const int32_t *P, uint32_t pc, int32_t ec, const uint2 *ginfo,
                                                        const uint64_t *gs, const uint64_t *go, uint64_t ng,
                                                        uint64_t dtot, uint64_t rows, int32_t *G, uint2 *gci) {
  for (uint64_t m = blockIdx.x * (uint64_t)kBlock + threadIdx.x; m < ng; m += (uint64_t)gridDim.x * kBlock) {
    const uint2 gi = ginfo[m];
    const uint64_t d = (m + 1 < ng ? gs[m + 1] : dtot) - gs[m];
    const uint64_t f = ((m + 1 < ng ? go[m + 1] : rows) - go[m]) / d;
    G[2 * m] = ec >= 0 ? P[(uint64_t)gi.x * pc + (uint32_t)ec] : 0;
    G[2 * m + 1] = (int32_t)(uint32_t)f;
    gci[m] = make_uint2((uint32_t)m, gi.y);
  }
}

// D[row] = 1 for every row of a filter's probe pass that was kept: tile lt's
// kept rows are hits[lt * tr + i], i below its count (tile prefixes of the
// two-level scan).
__global__ __launch_bounds__(kBlock) void k_hits_flags(const uint4 *hits, const uint64_t *tile_nz,
                                                       const uint64_t *chunk_nz, uint64_t ntiles, uint64_t nz_total,
                                                       uint32_t tr, uint8_t *D) {
  auto pre = [&](uint64_t t) -> uint64_t {
    return t >= ntiles ? nz_total : tile_nz[t] + chunk_nz[t / kScanChunk];
  };
  for (uint64_t lt = blockIdx.x; lt < ntiles; lt += gridDim.x) {
    const uint64_t a = pre(lt), n = pre(lt + 1) - a;
    for (uint64_t i = threadIdx.x; i < n; i += kBlock) D[hits[lt * tr + i].x] = 1;
  }
}

__global__ __launch_bounds__(kBlock) void k_zero_bytes(uint8_t *D, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)kBlock + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kBlock) D[i] = 0;
}

// Largest i in [lo, hi] with a[i] <= x (a ascending, a[lo] <= x).
__device__ __forceinline__ uint64_t last_le(const uint64_t *a, uint64_t lo, uint64_t hi, uint64_t x) {
  while (lo < hi) {
    const uint64_t mid = (lo + hi + 1) >> 1;
    if (a[mid] <= x) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Filter pass over one TR-row tile of a group-structured table: row r of
// group m is kept iff D[gs[m] + (r - go[m]) mod d_m]. Writes the tile's
// kept rows and sums exactly as the probe pass of a filter does (no edges
// examined: they were counted on S), so the tile scan and the compaction
// that follow are the filter's own.
template <int TR>
__global__ __launch_bounds__(kBlock) void k_flag_groups(StepParams p, const uint64_t *go, const uint64_t *gs,
                                                        uint64_t ng, uint64_t dtot, const uint8_t *D) {
  constexpr int kRowsPerThread = TR / kBlock;
  static_assert(TR % kBlock == 0, "tile rows must be a multiple of the block");
  __shared__ uint64_t s_tmp[kBlock / kWave];
  __shared__ uint64_t s_m[2];
  const uint64_t lt = p.tile0 + blockIdx.x;
  const uint32_t tid = threadIdx.x;
  const uint64_t base = lt * TR;
  if (tid == 0) {  // the groups this tile's rows lie in: [m0, m1]
    const uint64_t last = (base + TR < p.R ? base + TR : p.R) - 1;
    const uint64_t m0 = last_le(go, 0, ng - 1, base);
    s_m[0] = m0;
    s_m[1] = last_le(go, m0, ng - 1, last);
  }
  __syncthreads();
  const uint64_t m0 = s_m[0], m1 = s_m[1];
  const uint64_t r0 = base + (uint64_t)tid * kRowsPerThread;
  uint32_t keep = 0, nz = 0;  // bit k: row r0 + k kept
  if (r0 < p.R) {
    uint64_t m = last_le(go, m0, m1, r0);
#pragma unroll
    for (int k = 0; k < kRowsPerThread; k++) {
      const uint64_t r = r0 + k;
      if (r < p.R) {
        while (m < m1 && go[m + 1] <= r) m++;  // every group has rows: at most one step
        const uint64_t d = (m + 1 < ng ? gs[m + 1] : dtot) - gs[m];
        const uint32_t e = (uint32_t)(r - go[m]) % (uint32_t)d;
        if (D[gs[m] + e]) {
          keep |= 1u << k;
          nz++;
        }
      }
    }
  }
  uint64_t nz_total;
  uint32_t pos = (uint32_t)block_excl_scan(nz, s_tmp, nz_total);
  uint4 *hits = p.hits + lt * TR;
#pragma unroll
  for (int k = 0; k < kRowsPerThread; k++)
    if (keep >> k & 1u) hits[pos++] = make_uint4((uint32_t)(r0 + k), 0u, 1u, 0u);
  if (tid == 0) {
    p.tile_sum[lt] = nz_total;
    p.tile_nz[lt] = nz_total;
    p.tile_ex[lt] = 0;
  }
}


// ---- filters from a fan-out's new column (the parent's list decided per entry once) ----
// A known_to_unknown output T with lineage repeats compacted parent row i
// (parent table row info[i].x, list at segment offset info[i].y) in its rows
// [excl[i], excl[i+1]); row excl[i] + j holds the list's entry j in its last
// column. A known_to_known / known_to_const step from that column (the end
// column, if any, one of the parent's) keeps row excl[i] + j iff the filter
// target of parent i is in the list of (entry j, pid, dir). Parents that
// share a list share its entries' keys, so each distinct list's entries are
// probed once (D: (segment offset, degree) per entry under the filter's
// predicate); each row then only tests its target against that list, and
// the input table's cells are read for kept rows alone.
struct FanoutFilter {
  const uint64_t *excl;   // first child row per compacted parent (ascending)
  const uint2 *info;      // (parent row, list offset) per compacted parent
  uint64_t np;            // compacted parents
  const uint64_t *pbase;  // per compacted parent: its list's first entry in D
  const uint2 *D;         // per distinct-list entry: (segment offset, or the entry if degree 1; degree) of its key
  const int32_t *P;       // parent table
  uint32_t pc;            // parent columns
  int32_t ec;             // known_to_known end column (a parent column); -1: known_to_const
  uint32_t *bits;         // per tile: TR / 32 words, bit k of word w: row 32 w + k kept
};

// Keys of the distinct lists: K[k] = entry k - lbase[L] of list L (segment
// offset ly[L] of pid), L the list holding k.
template <bool FRAMED>
__global__ __launch_bounds__(kBlock) void k_gather_lists(GraphView g, uint32_t pid, const uint64_t *lbase,
                                                         const uint32_t *ly, uint64_t nl, uint64_t total, int32_t *K) {
  const DevMeta m = g.meta[pid];
  for (uint64_t k = blockIdx.x * (uint64_t)kBlock + threadIdx.x; k < total; k += (uint64_t)gridDim.x * kBlock) {
    uint64_t lo = 0, hi = nl - 1;  // last L with lbase[L] <= k
    while (lo < hi) {
      const uint64_t mid = (lo + hi + 1) >> 1;
      if (lbase[mid] <= k) lo = mid;
      else hi = mid - 1;
    }
    K[k] = (int32_t)edge_at<FRAMED>(g, m.edge_start, m.eframe_base, (uint64_t)ly[lo] + (k - lbase[lo]));
  }
}

// D[k] = (0, 0) for every key, then (x, degree) for the keys with edges
// (the compacted rows of a known_to_unknown probe pass over K): x is the
// list's only entry when the degree is 1 (a row then needs no list read),
// else the list's segment offset.
__global__ __launch_bounds__(kBlock) void k_zero_u64(uint64_t *a, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)kBlock + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kBlock) a[i] = 0;
}
__global__ __launch_bounds__(kBlock) void k_key_degrees(GraphView g, uint32_t pid, const uint2 *cinfo,
                                                        const uint64_t *cexcl, uint64_t nz, uint64_t E, uint2 *D) {
  const DevMeta m = g.meta[pid];
  for (uint64_t k = blockIdx.x * (uint64_t)kBlock + threadIdx.x; k < nz; k += (uint64_t)gridDim.x * kBlock) {
    const uint64_t deg = (k + 1 < nz ? cexcl[k + 1] : E) - cexcl[k];
    const uint32_t x = deg == 1 ? edge_at<false>(g, m.edge_start, m.eframe_base, cinfo[k].y) : cinfo[k].y;
    D[cinfo[k].x] = make_uint2(x, (uint32_t)deg);
  }
}

// Filter pass over one TR-row tile of T. Each thread takes RPT consecutive
// rows: its parent (a binary search for the first row, then walking), list
// entry, D entry and target; a list of at most kLaneList entries is scanned
// by the row's own lane (the reference's early-exit scan, so its work count
// is the scan's: first match + 1, or the degree). Longer lists go through
// the probe pass's membership test in a second phase, which a block
// skips when it has none. Kept flags become the tile's bit words; the tile's
// sums are kept rows and edges examined.
template <int TR, bool SORTED>
__global__ __launch_bounds__(kBlock) void k_fanout_filter(GraphView g, StepParams p, FanoutFilter f) {
  constexpr int RPT = TR / kBlock;
  constexpr uint32_t kLaneList = 8;
  static_assert(TR % kBlock == 0 && (TR / 32) <= kBlock, "tile rows");
  __shared__ uint32_t s_off[TR], s_deg[TR], s_tgt[TR];
  __shared__ uint8_t s_keep[TR], s_big[TR];
  __shared__ uint64_t s_m[2];
  __shared__ uint32_t s_any;
  const uint64_t lt = p.tile0 + blockIdx.x;
  const uint32_t tid = threadIdx.x, lane = lane_id();
  const uint64_t base = lt * TR;
  const DevMeta m = g.meta[p.pid < g.num_metas ? p.pid : 0];
  if (tid == 0) {  // the parents this tile's rows lie in: [i0, i1]
    const uint64_t last = (base + TR < p.R ? base + TR : p.R) - 1;
    const uint64_t i0 = last_le(f.excl, 0, f.np - 1, base);
    s_m[0] = i0;
    s_m[1] = last_le(f.excl, i0, f.np - 1, last);
    s_any = 0;
  }
  __syncthreads();
  uint64_t ex = 0;
  {
    const uint64_t i0 = s_m[0], i1 = s_m[1];
    const uint64_t r0 = base + (uint64_t)tid * RPT;
    uint64_t i = r0 < p.R ? last_le(f.excl, i0, i1, r0) : i0;
    uint32_t off[RPT], deg[RPT], tgt[RPT];
    bool valid[RPT];
#pragma unroll
    for (int k = 0; k < RPT; k++) {  // the D entries and targets, loads issued together
      const uint64_t r = r0 + k;
      off[k] = 0;
      deg[k] = 0;
      tgt[k] = 0;
      valid[k] = false;
      if (r < p.R) {
        while (i < i1 && f.excl[i + 1] <= r) i++;  // every parent has rows: one step at most per row
        const uint2 e = f.D[f.pbase[i] + (r - f.excl[i])];
        off[k] = e.x;
        deg[k] = e.y;
        if (f.ec >= 0) {
          const int32_t cell = f.P[(uint64_t)f.info[i].x * f.pc + (uint32_t)f.ec];
          tgt[k] = (uint32_t)cell;
          valid[k] = cell >= 0;
        } else {
          tgt[k] = p.target;
          valid[k] = p.target_ok != 0;
        }
      }
    }
    bool big_any = false;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const uint32_t local = tid * RPT + k;
      uint8_t keep = 0, big = 0;
      if (valid[k] && deg[k] > kLaneList) {
        big = 1;
        s_off[local] = off[k];
        s_deg[local] = deg[k];
        s_tgt[local] = tgt[k];
      } else if (deg[k] == 1) {  // D holds the list's only entry
        keep = valid[k] && off[k] == tgt[k] ? 1 : 0;
        ex += 1;
      } else {
        uint32_t x = deg[k];
        if (valid[k])
          for (uint32_t j = 0; j < deg[k]; j++)
            if (edge_at<false>(g, m.edge_start, m.eframe_base, (uint64_t)off[k] + j) == tgt[k]) {
              keep = 1;
              x = j + 1;
              break;
            }
        ex += x;
      }
      s_keep[local] = keep;
      s_big[local] = big;
      big_any |= big != 0;
    }
    if (big_any) s_any = 1;
  }
  __syncthreads();
  if (s_any) {  // long lists: the membership test of the probe pass, 64 rows per wave per round
    constexpr uint32_t kWaveRows = TR / (kBlock / kWave);
    const uint32_t wave = tid / kWave;
    for (int rd = 0; rd < TR / kBlock; rd++) {
      const uint32_t local = wave * kWaveRows + rd * kWave + lane;
      const bool big = s_big[local] != 0;
      const uint32_t off = big ? s_off[local] : 0u, deg = big ? s_deg[local] : 0u, tgt = big ? s_tgt[local] : 0u;
      if (!wave_ballot(big)) continue;
      bool found;
      uint32_t examined;
      rows_member<SORTED, false>(g, m.edge_start, m.eframe_base, off, deg, tgt, big, found, examined);
      if (big) {
        s_keep[local] = found ? 1 : 0;
        ex += examined;
      }
    }
  }
  __syncthreads();
  uint32_t word = 0, nz = 0;
  if (tid < TR / 32) {
#pragma unroll
    for (int b = 0; b < 32; b++) word |= (uint32_t)s_keep[tid * 32 + b] << b;
    nz = __builtin_popcount(word);
    f.bits[lt * (TR / 32) + tid] = word;
  }
  uint64_t v[2] = {nz, ex}, tot[2];
  __shared__ uint64_t s_tmp2[2 * (kBlock / kWave)];
  block_excl_scan_n<2>(v, s_tmp2, tot);
  if (tid == 0) {
    p.tile_sum[lt] = tot[0];
    p.tile_nz[lt] = tot[0];
    p.tile_ex[lt] = tot[1];
  }
}

// The same decisions over parent-aligned units: unit (i, jb) is rows
// [excl[i] + jb TR, ...) of parent i, at most TR of them, all with one
// target. Units are ranked in row order (rank = ubase[i] + jb: the order of
// the scan and the compaction) but executed list by list, j-block by
// j-block, the parents sharing a list innermost (block e of list L: j-block
// (e - xbase[L]) / |parents of L|), so the blocks that read one slice of a
// shared list's D entries run together and find it in their L2.
struct FanoutUnits {
  const uint64_t *xbase;  // per distinct list (+1): first execution index
  const uint64_t *poff;   // per distinct list (+1): its parents' first slot in par
  const uint32_t *par;    // compacted parents, grouped by list, row order within a list
  const uint64_t *ubase;  // per compacted parent: rank of its first unit
  uint64_t nl;            // distinct lists
  uint64_t *row0;         // per unit rank: its first row
};

template <int TR, bool SORTED>
__global__ __launch_bounds__(kBlock) void k_fanout_units(GraphView g, StepParams p, FanoutFilter f, FanoutUnits u) {
  constexpr int RPT = TR / kBlock;
  constexpr uint32_t kLaneList = 8;
  static_assert(RPT == 8 && (TR / 32) <= kBlock, "a thread's rows are one byte of kept bits");
  __shared__ uint32_t s_off[TR], s_deg[TR];
  __shared__ uint8_t s_keep[TR];             // long lists' decisions (phase 2)
  __shared__ uint8_t s_bigb[kBlock];         // per thread: which of its rows have long lists
  __shared__ __align__(4) uint8_t s_kb[kBlock];  // per thread: its rows' kept bits
  __shared__ uint32_t s_any;
  const uint32_t tid = threadIdx.x, lane = lane_id();
  const uint64_t e = p.tile0 + blockIdx.x;
  // the unit: list L, j-block, parent
  uint64_t L = 0, hi = u.nl - 1;
  while (L < hi) {
    const uint64_t mid = (L + hi + 1) >> 1;
    if (u.xbase[mid] <= e) L = mid;
    else hi = mid - 1;
  }
  const uint64_t npl = u.poff[L + 1] - u.poff[L], e2 = e - u.xbase[L];
  const uint64_t jb = e2 / npl;
  const uint32_t i = u.par[u.poff[L] + e2 % npl];
  const uint64_t first = f.excl[i];
  const uint64_t n = (i + 1 < f.np ? f.excl[i + 1] : p.R) - first;
  const uint64_t j0 = jb * TR;
  const uint32_t nrows = (uint32_t)(n - j0 < (uint64_t)TR ? n - j0 : (uint64_t)TR);
  const uint64_t rank = u.ubase[i] + jb;
  uint32_t tgt;
  bool valid;
  if (f.ec >= 0) {
    const int32_t cell = f.P[(uint64_t)f.info[i].x * f.pc + (uint32_t)f.ec];
    tgt = (uint32_t)cell;
    valid = cell >= 0;
  } else {
    tgt = p.target;
    valid = p.target_ok != 0;
  }
  const DevMeta m = g.meta[p.pid < g.num_metas ? p.pid : 0];
  if (tid == 0) s_any = 0;
  const uint2 *Dp = f.D + f.pbase[i] + j0;
  uint2 d[RPT];
#pragma unroll
  for (int k = 0; k < RPT; k++) {  // the unit's D entries, loads issued together
    const uint32_t local = tid * RPT + k;
    d[k] = local < nrows ? Dp[local] : make_uint2(0u, 0u);
  }
  __syncthreads();
  uint64_t ex = 0;
  uint32_t kb = 0, bigb = 0;  // this thread's rows: kept bits, long-list bits
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const uint32_t local = tid * RPT + k;
    const uint32_t off = d[k].x, deg = d[k].y;
    if (valid && deg > kLaneList) {
      bigb |= 1u << k;
      s_off[local] = off;
      s_deg[local] = deg;
    } else if (deg == 1) {  // D holds the list's only entry
      kb |= (valid && off == tgt ? 1u : 0u) << k;
      ex += 1;
    } else {
      uint32_t x = deg;
      if (valid)
        for (uint32_t j = 0; j < deg; j++)
          if (edge_at<false>(g, m.edge_start, m.eframe_base, (uint64_t)off + j) == tgt) {
            kb |= 1u << k;
            x = j + 1;
            break;
          }
      ex += x;
    }
  }
  s_bigb[tid] = (uint8_t)bigb;
  if (bigb) s_any = 1;
  __syncthreads();
  if (s_any) {  // long lists: the membership test of the probe pass, 64 rows per wave per round
    constexpr uint32_t kWaveRows = TR / (kBlock / kWave);
    const uint32_t wave = tid / kWave;
    for (int rd = 0; rd < TR / kBlock; rd++) {
      const uint32_t local = wave * kWaveRows + rd * kWave + lane;
      const bool big = (s_bigb[local / RPT] >> (local % RPT)) & 1u;
      const uint32_t off = big ? s_off[local] : 0u, deg = big ? s_deg[local] : 0u;
      if (!wave_ballot(big)) continue;
      bool found;
      uint32_t examined;
      rows_member<SORTED, false>(g, m.edge_start, m.eframe_base, off, deg, tgt, big, found, examined);
      if (big) {
        s_keep[local] = found ? 1 : 0;
        ex += examined;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RPT; k++)
      if (bigb >> k & 1u) kb |= (uint32_t)s_keep[tid * RPT + k] << k;
  }
  s_kb[tid] = (uint8_t)kb;
  __syncthreads();
  uint32_t word = 0, nz = 0;
  if (tid < TR / 32) {  // rows 32 tid .. 32 tid + 31: four threads' bytes
    word = ((const uint32_t *)s_kb)[tid];
    nz = __builtin_popcount(word);
    f.bits[rank * (TR / 32) + tid] = word;
  }
  uint64_t v[2] = {nz, ex}, tot[2];
  __shared__ uint64_t s_tmp2[2 * (kBlock / kWave)];
  block_excl_scan_n<2>(v, s_tmp2, tot);
  if (tid == 0) {
    p.tile_sum[rank] = tot[0];
    p.tile_nz[rank] = tot[0];
    p.tile_ex[rank] = tot[1];
    u.row0[rank] = first + j0;
  }
}

// The fan-out filter for long shared lists of unsorted images or of many
// parents, a block of list entries at a time: a workgroup takes kFBRows entries of one distinct list and up to
// kFBGroup (= 64) of the parents sharing that list, and tests every parent
// against every entry's list, holding the block in registers:
//  - thread t takes entries t, t + 256, ...: their D entries are read once;
//    an entry whose list has one element keeps it in a register (D holds
//    it), so a (parent, entry) test is one compare;
//  - the few entries with longer lists are tested before the parent loop,
//    each by one wave with lane pi testing parent pi (the list's entries
//    broadcast lane by lane, or a binary search per lane for a long sorted
//    list), leaving a 64-bit parent mask per entry;
//  - per parent, each wave's compares are ballots: 64 rows' kept flags at
//    once (kept rows are rare: pass 1 only notes the parents with one in a
//    mask, and pass 2 redoes those parents' ballots);
//  - a workgroup's time is its chain of dependent loads (list, parent slot,
//    parent row, end cell), so the block's D entries are loaded first, from
//    the list's base, and arrive while the parents' targets are fetched.
// The output is per unit (parent x block of kFBRows rows, ranked
// ubase[parent] + block) its kept rows and edges examined, for the tile
// scan, and a list of the kept rows with their unit and index in it, for
// k_compact_kept. Work counts follow the reference's scan: first match + 1,
// or the degree.
constexpr int kFBRows = 2048;
constexpr int kFBPer = kFBRows / kBlock;
constexpr int kFBGroup = 64;
struct FanoutBlocks {
  const uint64_t *xb;     // per distinct list (+1): first work index (blocks x parent groups)
  const uint64_t *poff;   // per distinct list (+1): its parents' first slot in par
  const uint32_t *par;    // compacted parents, grouped by list, row order within a list
  const uint64_t *ubase;  // per compacted parent: rank of its first unit of kFBRows rows
  const uint64_t *ln;     // per distinct list: its entries
  const uint64_t *lbase;  // per distinct list: its first entry in D
  uint64_t nl;
  uint64_t *row0;         // per unit rank: its first row
  // kept rows, unordered: (row, unit rank, index within the unit, 0); a row
  // past the capacity is counted but not stored (the caller then reruns)
  uint4 *kept;
  uint64_t *nkept;
  uint64_t cap;
};

template <bool SORTED>
__global__ __launch_bounds__(kBlock) void k_fanout_blocks(GraphView g, StepParams p, FanoutFilter f, FanoutBlocks u) {
  constexpr int W = kBlock / kWave;
  constexpr uint32_t kNone = 0xffffffffu, kNoTarget = 0xfffffffeu;  // (ids and valid targets are below 2^31)
  static_assert(kFBGroup == kWave, "lane pi tests parent pi");
  __shared__ uint32_t s_boff[kFBRows], s_bdeg[kFBRows];
  __shared__ uint64_t s_bmask[kFBRows];            // per longer list: the parents in it
  __shared__ uint16_t s_pc[kFBGroup][kFBPer][W];   // per parent: kept rows per (k, wave) ballot
  __shared__ uint32_t s_kcnt[kFBGroup];            // per parent: kept rows in the block
  __shared__ uint32_t s_tgt[kFBGroup], s_par[kFBGroup];
  __shared__ uint64_t s_rank[kFBGroup];
  __shared__ uint64_t s_bex[W][kWave], s_tmp[W];
  __shared__ uint32_t s_nb;
  __shared__ unsigned long long s_hit;            // parents with a kept row in the block
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  const uint64_t e = p.tile0 + blockIdx.x;
  uint64_t L = 0, hi = u.nl - 1;  // the list: the last with xb <= e
  while (L < hi) {
    const uint64_t mid = (L + hi + 1) >> 1;
    if (u.xb[mid] <= e) L = mid;
    else hi = mid - 1;
  }
  const uint64_t cnt = u.poff[L + 1] - u.poff[L], ngr = (cnt + kFBGroup - 1) / kFBGroup;
  const uint64_t e2 = e - u.xb[L], jb = e2 / ngr, grp = e2 % ngr;
  const uint64_t n = u.ln[L], j0 = jb * kFBRows;
  const uint32_t nrows = (uint32_t)(n - j0 < (uint64_t)kFBRows ? n - j0 : (uint64_t)kFBRows);
  const uint32_t npg = (uint32_t)(cnt - grp * kFBGroup < (uint64_t)kFBGroup ? cnt - grp * kFBGroup : kFBGroup);
  // the block's D entries, loaded now and used once the parents' targets
  // (a chain of dependent loads) are in
  const uint2 *Dp = f.D + u.lbase[L] + j0;
  uint2 dv[kFBPer];
#pragma unroll
  for (int k = 0; k < kFBPer; k++) {
    const uint32_t row = tid + k * kBlock;
    dv[k] = row < nrows ? Dp[row] : make_uint2(0u, 0u);
  }
  const DevMeta m = g.meta[p.pid < g.num_metas ? p.pid : 0];
  if (tid == 0) {
    s_nb = 0;
    s_hit = 0;
  }
  for (uint32_t z = tid; z < kFBGroup * kFBPer * W / 2; z += kBlock) ((uint32_t *)&s_pc[0][0][0])[z] = 0;
  if (tid < kFBGroup) {
    uint32_t tg = kNoTarget, i = 0;
    if (tid < npg) {
      i = u.par[u.poff[L] + grp * kFBGroup + tid];
      if (f.ec >= 0) {
        const int32_t cell = f.P[(uint64_t)f.info[i].x * f.pc + (uint32_t)f.ec];
        if (cell >= 0) tg = (uint32_t)cell;
      } else if (p.target_ok) {
        tg = p.target;
      }
      s_rank[tid] = u.ubase[i] + jb;
    }
    s_par[tid] = i;
    s_tgt[tid] = tg;
    s_kcnt[tid] = 0;
  }
  __syncthreads();
  uint32_t c0[kFBPer], bi[kFBPer];  // single entry (or kNone); a longer list's index (or kNone)
  uint64_t ex1 = 0;  // single-entry rows: one edge examined each, for every parent
#pragma unroll
  for (int k = 0; k < kFBPer; k++) {
    const uint2 d = dv[k];
    c0[k] = d.y == 1 ? d.x : kNone;
    ex1 += d.y == 1 ? 1u : 0u;
    bi[k] = kNone;
    if (d.y >= 2) {
      const uint32_t b = atomicAdd(&s_nb, 1u);
      bi[k] = b;
      s_boff[b] = d.x;
      s_bdeg[b] = d.y;
    }
  }
  __syncthreads();
  const uint32_t nb = s_nb;
  {
    // each longer list by one wave, lane pi testing parent pi
    const uint32_t tgt = s_tgt[lane];
    uint64_t exl = 0;
    for (uint32_t b = wave; b < nb; b += W) {
      const uint32_t off = s_boff[b], deg = s_bdeg[b];
      bool fnd = false;
      uint32_t x = deg;
      if (SORTED && deg > kWave) {
        if (tgt != kNoTarget) {
          uint32_t lo = 0, hi2 = deg;
          while (lo < hi2) {
            const uint32_t mid = (lo + hi2) >> 1;
            if (edge_at<false>(g, m.edge_start, m.eframe_base, (uint64_t)off + mid) < tgt) lo = mid + 1;
            else hi2 = mid;
          }
          if (lo < deg && edge_at<false>(g, m.edge_start, m.eframe_base, (uint64_t)off + lo) == tgt) {
            fnd = true;
            x = lo + 1;
          }
        }
      } else {  // wave-uniform: 64 entries at a time, broadcast lane by lane
        for (uint32_t q0 = 0; q0 < deg; q0 += kWave) {
          const uint32_t ev = q0 + lane < deg ? edge_at<false>(g, m.edge_start, m.eframe_base, (uint64_t)off + q0 + lane) : kNone;
          const uint32_t qn = deg - q0 < (uint32_t)kWave ? deg - q0 : (uint32_t)kWave;
          for (uint32_t q = 0; q < qn; q++) {
            const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)ev, (int)q);
            if (!fnd && tgt != kNoTarget && v == tgt) {
              fnd = true;
              x = q0 + q + 1;
            }
          }
        }
      }
      const uint64_t mask = wave_ballot(fnd);
      if (lane == 0) s_bmask[b] = mask;
      exl += x;
    }
    s_bex[wave][lane] = exl;
  }
  uint64_t ex1_total;
  (void)block_excl_scan(ex1, s_tmp, ex1_total);  // (its barriers also order the masks above)
  uint64_t mk[kFBPer];
  uint32_t kmulti = 0;  // wave-uniform: bit k set when a row k of the wave has a longer list
#pragma unroll
  for (int k = 0; k < kFBPer; k++) {
    mk[k] = bi[k] != kNone ? s_bmask[bi[k]] : 0ull;
    kmulti |= wave_ballot(bi[k] != kNone) ? 1u << k : 0u;
  }
  const uint32_t tgt_l = s_tgt[lane];  // lane pi: parent pi's target
  auto ballot_k = [&](uint32_t pi, uint32_t tgt, int k) -> uint64_t {
    const uint64_t m1 = __builtin_amdgcn_uicmp(c0[k], tgt, 32);  // (32: equal) 64 rows' compares at once
    if (kmulti >> k & 1u) return m1 | wave_ballot(((mk[k] >> pi) & 1u) != 0);
    return m1;
  };
  // pass 1: every parent against every single-entry row: one compare per
  // 64 rows, only noting parents with a match (rare) in a wave-uniform mask
  uint64_t hit = 0;
  for (uint32_t pi = 0; pi < npg; pi++) {
    const uint32_t tgt = (uint32_t)__builtin_amdgcn_readlane((int)tgt_l, (int)pi);
    uint64_t any = 0;
#pragma unroll
    for (int k = 0; k < kFBPer; k++) any |= __builtin_amdgcn_uicmp(c0[k], tgt, 32);
    hit |= (any ? 1ull : 0ull) << pi;
  }
  if (hit && lane == 0) atomicOr(&s_hit, (unsigned long long)hit);
  // ... and the parents a longer list keeps
  for (uint32_t b = tid; b < nb; b += kBlock)
    if (s_bmask[b]) atomicOr(&s_hit, (unsigned long long)s_bmask[b]);
  __syncthreads();
  // pass 2, parents with kept rows only: the ballots again, counted per
  // (k, wave), then each kept row listed with its index among its parent's
  // kept rows (row order: k, then wave, then lane)
  for (uint64_t hm = s_hit; hm; hm &= hm - 1) {  // block-uniform
    const uint32_t pi = (uint32_t)__builtin_ctzll(hm);
    const uint32_t tgt = (uint32_t)__builtin_amdgcn_readlane((int)tgt_l, (int)pi);
    uint64_t bw[kFBPer];
#pragma unroll
    for (int k = 0; k < kFBPer; k++) {
      bw[k] = ballot_k(pi, tgt, k);
      if (lane == 0) s_pc[pi][k][wave] = (uint16_t)__builtin_popcountll(bw[k]);
    }
    __syncthreads();
    const uint64_t rank = s_rank[pi], first = f.excl[s_par[pi]] + j0;
    uint32_t before = 0;  // kept rows of parent pi at smaller (k, wave)
#pragma unroll
    for (int k = 0; k < kFBPer; k++) {
      for (int w = 0; w < W; w++)
        if (w < (int)wave) before += s_pc[pi][k][w];
      if (bw[k]) {
        uint64_t base = 0;
        if (lane == 0) base = atomicAdd((unsigned long long *)u.nkept, (unsigned long long)__builtin_popcountll(bw[k]));
        base = shfl64(base, 0);
        if ((bw[k] >> lane) & 1u) {
          const uint32_t lr = (uint32_t)__builtin_popcountll(bw[k] & lanes_below());
          const uint64_t slot = base + lr;
          if (slot < u.cap)
            u.kept[slot] = make_uint4((uint32_t)(first + (uint32_t)k * kBlock + wave * kWave + lane), (uint32_t)rank,
                                      before + lr, 0u);
        }
      }
      for (int w = (int)wave; w < W; w++) before += s_pc[pi][k][w];
    }
    if (tid == 0) s_kcnt[pi] = before;  // (wave 0 counted every wave's rows)
  }
  __syncthreads();
  if (tid < npg) {
    uint64_t xt = ex1_total;
#pragma unroll
    for (int w = 0; w < W; w++) xt += s_bex[w][tid];
    const uint64_t rank = s_rank[tid];
    p.tile_sum[rank] = s_kcnt[tid];
    p.tile_nz[rank] = s_kcnt[tid];
    p.tile_ex[rank] = xt;
  }
}

// ---- the fan-out filter through its lists (sorted images) ----
// The pairs (parent, list entry) of a fan-out need not be tested one by one:
// row (i, j) is kept iff parent i's target is in the filter list of entry j
// of i's list, so the targets of the parents sharing a list are hashed once
// (k_list_parents), and every element of every entry's filter list is looked
// up among them (k_list_filter; elements of long filter lists in
// k_list_long). The work is one probe per distinct list entry and one lookup
// per element of the lists it finds, whatever the number of parents; the work
// count is, per list, its parents times its entries' degrees, less what the
// reference's early exit spares each kept row. Kept rows are listed
// unordered and ranked by their row (k_list_rows); where they are more than
// the list holds, the pass is made again with a bit per row.
// What bounds it: the probe of the distinct entries (cache misses); nearly
// all lookups end at a bit of a filter in L1. The cycle's closing filter over
// 1.9G pairs of 1.6M distinct entries: its query 618 -> 205 us (pair by pair in
// k_fanout_blocks 256 us, on top of the probe's 46 us, its passes' 40 us, and
// 150 us of lists gathered on the host).
struct ListFilter {
  // the fan-out's parents
  const uint2 *info;     // (parent row, list offset)
  const uint64_t *excl;  // first child row
  uint64_t np, R;
  const int32_t *P;
  uint32_t pc;
  int32_t ec;            // known_to_known end column (a parent column); -1: known_to_const
  uint32_t target, target_ok;
  uint32_t lpid, pid, dir;  // the fan-out's predicate; the filter's pattern
  // distinct lists, in first-come order: offset, entries before, length, parents
  uint32_t *l_off, *l_base, *l_len, *l_np;
  uint32_t *seen, *seen_list, mask1;  // offset -> list (open addressing)
  uint32_t *p_list, *p_tgt, *p_slot;  // per parent: list, target, its slot below
  uint32_t *head, *count, log2;       // (list, target) -> a parent (+1), parents (open addressing, 2^log2)
  uint32_t *start, *order;            // the slot's parents: order[start .. start + count)
  uint32_t *bits, blog2;              // two bits of a word per (list, target), 2^blog2 words
  unsigned long long *ctr;            // kList*
  uint4 *kept;                        // (row, parent, entry, 0)
  uint64_t cap;
  uint32_t *rbits;                    // or a bit per row (BITS)
  uint64_t *ex;                       // per wave of k_list_filter: its share of the work count (mod 2^64)
  // long filter lists in kListQueues queues of long_cap items (a workgroup
  // appends to one of them: thousands of workgroups adding to one word take
  // 17 ns each): (entry, offset, degree, first element)
  uint4 *longs;
  unsigned long long *long_n;         // per queue, kListPad words apart
  uint64_t long_cap;
};
// (kListBits: three words, the totals of the tile scan over the bits)
enum { kListSums = 0, kListUnits, kListKept, kListEx, kListSpared, kListLost, kListBits, kListCtrs = kListBits + 3 };
constexpr uint32_t kListQueues = 64, kListPad = 16;
constexpr uint32_t kNoList = 0xffffffffu;  // (segments hold fewer than 2^32 edges)
constexpr uint32_t kListInline = 16;       // longer filter lists go to k_list_long,
constexpr uint32_t kListChunk = 1024;      // this many elements an item
constexpr int kListTile = 512;             // list entries per workgroup
constexpr uint64_t kListKeptCap = 32768;   // ranking compares all kept rows with each other; more: bits
constexpr int kListBitRows = 1024;         // rows per tile of the bits

__device__ __forceinline__ uint32_t pair_hash(uint32_t l, uint32_t t) {
  uint32_t h = (l * 0x9E3779B1u + t) * 0x85EBCA6Bu;
  h ^= h >> 15;
  return h * 0xC2B2AE35u;
}
__device__ __forceinline__ uint32_t pair_slot(const ListFilter &f, uint32_t h) { return (h * 0x27D4EB2Fu) >> (32 - f.log2); }
__device__ __forceinline__ uint32_t pair_bits(uint32_t h) { return (1u << (h & 31)) | (1u << ((h >> 5) & 31)); }

// The distinct lists and the parents' targets, by one workgroup (its phases
// are separated by barriers; words changed by atomics are read as atomics).
// Up to kListLds parents the hash tables are built in LDS and copied out: the
// parents of a popular list all meet at its words, which serialises in memory
// (800 parents: 54 us, in LDS 31 us). The parents of one list and target end
// up side by side, so that whoever keeps a row for each of them can do so with
// a wave's lanes at once.
constexpr uint32_t kListLds = 2048;
__global__ __launch_bounds__(1024) void k_list_parents(ListFilter fg, Signal sg) {
  __shared__ uint32_t s_tab[(4 * 2 + 2) * kListLds];  // seen, seen_list, head, count: two slots a parent; l_np, bits
  __shared__ unsigned long long s_ctr[kListCtrs];
  __shared__ uint32_t s_used;  // parents placed in order
  const uint32_t tid = threadIdx.x, np = (uint32_t)fg.np;
  ListFilter f = fg;
  const bool lds = np <= kListLds;
  if (lds) {
    f.seen = s_tab;
    f.seen_list = s_tab + 2 * kListLds;
    f.head = s_tab + 4 * kListLds;
    f.count = s_tab + 6 * kListLds;
    f.l_np = s_tab + 8 * kListLds;
    f.bits = s_tab + 9 * kListLds;
    f.ctr = s_ctr;
    f.start = f.seen_list;  // (which is done with by then)
  }
  for (uint32_t i = tid; i <= f.mask1; i += 1024) f.seen[i] = kNoList;
  for (uint32_t i = tid; i < 1u << f.log2; i += 1024) f.head[i] = f.count[i] = 0;
  for (uint32_t i = tid; i < 1u << f.blog2; i += 1024) f.bits[i] = 0;
  for (uint32_t i = tid; i < np; i += 1024) f.l_np[i] = 0;
  if (tid == 0) s_used = 0;
  if (tid < kListCtrs) f.ctr[tid] = 0;
  if (tid < kListQueues) f.long_n[tid * kListPad] = 0;
  __threadfence();
  __syncthreads();
  uint64_t units = 0;
  for (uint32_t i = tid; i < np; i += 1024) {
    const uint32_t off = f.info[i].y;
    const uint64_t n = (i + 1 < np ? f.excl[i + 1] : f.R) - f.excl[i];
    units += (n + kFBRows - 1) / kFBRows;
    uint32_t s = (off * 0x9E3779B1u) & f.mask1;
    for (;; s = (s + 1) & f.mask1) {
      uint32_t old = __hip_atomic_load(&f.seen[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (old == kNoList) old = atomicCAS(&f.seen[s], kNoList, off);
      if (old == kNoList) {  // the first parent of this list
        const unsigned long long v = atomicAdd(&f.ctr[kListSums], (1ull << 40) | n);
        const uint32_t l = (uint32_t)(v >> 40);
        f.l_off[l] = off;
        f.l_base[l] = (uint32_t)v;
        f.l_len[l] = (uint32_t)n;
        f.seen_list[s] = l;
        break;
      }
      if (old == off) break;
    }
    f.p_slot[i] = s;  // (the list's slot, for now)
  }
  if (units) atomicAdd(&f.ctr[kListUnits], (unsigned long long)units);
  __threadfence();
  __syncthreads();
  for (uint32_t i = tid; i < np; i += 1024) {
    const uint32_t l = f.seen_list[f.p_slot[i]];
    f.p_list[i] = l;
    f.p_tgt[i] = f.ec >= 0 ? (uint32_t)f.P[(uint64_t)f.info[i].x * f.pc + (uint32_t)f.ec] : f.target;
    atomicAdd(&f.l_np[l], 1u);
  }
  __threadfence();
  __syncthreads();
  // each parent's slot and its place among the slot's parents (in seen, which is done with)
  uint32_t *rank = f.seen;
  for (uint32_t i = tid; i < np; i += 1024) {
    const uint32_t l = f.p_list[i], t = f.p_tgt[i];
    uint32_t slot = kNoList;
    if (f.ec >= 0 ? (int32_t)t >= 0 : f.target_ok) {
      const uint32_t h = pair_hash(l, t);
      atomicOr(&f.bits[h >> (32 - f.blog2)], pair_bits(h));
      for (slot = pair_slot(f, h);; slot = (slot + 1) & ((1u << f.log2) - 1)) {
        const uint32_t old = atomicCAS(&f.head[slot], 0u, i + 1);
        if (old == 0 || (f.p_list[old - 1] == l && f.p_tgt[old - 1] == t)) break;
      }
      rank[i] = atomicAdd(&f.count[slot], 1u);
    }
    f.p_slot[i] = slot;
  }
  __threadfence();
  __syncthreads();
  for (uint32_t i0 = 0; i0 < np; i0 += 1024) {  // a slot's first parent makes its room (one add a wave)
    const uint32_t i = i0 + tid, slot = i < np ? f.p_slot[i] : kNoList;
    const bool lead = slot != kNoList && rank[i] == 0;
    const uint32_t n = lead ? __hip_atomic_load(&f.count[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
    const uint32_t inc = wave_incl_scan32(n);
    uint32_t base = 0;
    if (lane_id() == kWave - 1) base = atomicAdd(&s_used, inc);
    base = lane63(base);
    if (lead) f.start[slot] = fg.start[slot] = base + inc - n;
  }
  __syncthreads();
  for (uint32_t i = tid; i < np; i += 1024)
    if (f.p_slot[i] != kNoList) f.order[f.start[f.p_slot[i]] + rank[i]] = i;
  if (lds) {
    for (uint32_t i = tid; i < 1u << f.log2; i += 1024) {
      fg.head[i] = f.head[i];
      fg.count[i] = f.count[i];
    }
    for (uint32_t i = tid; i < 1u << f.blog2; i += 1024) fg.bits[i] = f.bits[i];
    for (uint32_t i = tid; i < np; i += 1024) fg.l_np[i] = f.l_np[i];
    if (tid < kListCtrs) fg.ctr[tid] = f.ctr[tid];
  }
  if (tid == 0) {
    const uint64_t sums = __hip_atomic_load(&f.ctr[kListSums], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t v[3] = {sums & ((1ull << 40) - 1), sums >> 40,
                           __hip_atomic_load(&f.ctr[kListUnits], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
    publish(sg, v, 3);
  }
}

// Element idx (x) of a filter list that list l's entry found: the parents of
// l with target x, order[first .. first + the result), keep a row each.
__device__ __forceinline__ uint32_t list_match(const GraphView &g, uint64_t estart, const ListFilter &f, uint32_t l,
                                               uint32_t off, uint32_t idx, uint32_t x, uint32_t &first) {
  const uint32_t h = pair_hash(l, x), b = pair_bits(h);
  if ((f.bits[h >> (32 - f.blog2)] & b) != b) return 0;
  for (uint32_t s = pair_slot(f, h);; s = (s + 1) & ((1u << f.log2) - 1)) {
    const uint32_t hd = f.head[s];
    if (!hd) return 0;
    if (f.p_list[hd - 1] != l || f.p_tgt[hd - 1] != x) continue;
    if (idx && g.edges[estart + off + idx - 1] == x) return 0;  // (only the first match counts)
    first = f.start[s];
    return f.count[s];
  }
}

// The whole wave: each lane's n parents from order[first] on keep their row
// of entry j (e); spare: the edges that each of them need not examine, summed
// per lane in spared. The wave's rows are one sequence, a lane each, and take
// one add of the counter. (A lane that wrote its own n rows one after another,
// along a chain of parents, took 250 ns a row: 4096 parents of one list, one
// target for all, 1196 us a call, now 328.) With BITS every kept row becomes a
// bit of rbits; else it is listed, and false says that the list has
// overflown: the rest of the pass is not needed.
template <bool BITS>
__device__ __forceinline__ bool list_keep(const ListFilter &f, uint32_t n, uint32_t first, uint32_t j, uint32_t e,
                                          uint32_t spare, uint64_t &spared) {
  if (!wave_ballot(n != 0)) return true;
  const uint32_t lane = lane_id();
  const uint32_t inc = wave_incl_scan32(n), all = lane63(inc), before = inc - n;
  spared += (uint64_t)n * spare;
  uint64_t base = 0;
  if constexpr (!BITS) {
    if (lane == 0) base = atomicAdd(&f.ctr[kListKept], (unsigned long long)all);
    base = shfl64(base, 0);
    if (base + all > f.cap) return false;
  }
  for (uint32_t t0 = 0; t0 < all; t0 += kWave) {  // (wave-uniform)
    const uint32_t t = t0 + lane;
    uint32_t src = 0;  // the last lane whose rows start at or before t (lanes without any share their next's)
#pragma unroll
    for (uint32_t step = kWave / 2; step; step >>= 1)
      if (shfl32(before, src + step) <= t) src += step;
    const uint32_t q = shfl32(first, src) + (t - shfl32(before, src)), kj = shfl32(j, src), ke = shfl32(e, src);
    if (t < all) {
      const uint32_t p = f.order[q];
      const uint64_t row = f.excl[p] + kj;
      if constexpr (BITS) {
        if (row < f.R) atomicOr(&f.rbits[row >> 5], 1u << (row & 31));  // (always: lists at one offset are alike)
      } else {
        f.kept[base + t] = make_uint4((uint32_t)row, p, ke, 0u);
      }
    }
  }
  return true;
}

template <bool BITS>
__global__ __launch_bounds__(kBlock) void k_list_filter(GraphView g, ListFilter f, uint32_t total, uint32_t nl,
                                                        uint32_t block0) {
  const uint32_t block = block0 + blockIdx.x;
  constexpr int RD = kListTile / kBlock;
  __shared__ WaveProbeLds s_wp[kBlock / kWave];
  const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
  const DevMeta ml = g.meta[f.lpid], m = g.meta[f.pid];
  uint32_t l[RD], j[RD], e[RD], deg[RD], off[RD];
  bool in[RD];
  {
    const uint32_t w0 = block * (uint32_t)kListTile + wave * RD * kWave;
    if (w0 >= total) {  // (waves are independent: no barrier below)
      if (lane == 0) f.ex[block * (kBlock / kWave) + wave] = 0;
      return;
    }
    // the wave's first list, and whether all its rows are in it
    const uint32_t l0 = (uint32_t)wave_last_le(nl, w0, [&](uint64_t i) -> uint64_t { return f.l_base[i]; });
    const uint32_t b0 = f.l_base[l0], o0 = f.l_off[l0];
    const bool one = l0 + 1 >= nl || f.l_base[l0 + 1] >= w0 + RD * kWave;
    const uint32_t most = nl - 1 < l0 + RD * kWave ? nl - 1 : l0 + RD * kWave;  // (every list has an entry)
#pragma unroll
    for (int r = 0; r < RD; r++) {
      const uint32_t k = w0 + r * kWave + lane;
      in[r] = k < total;
      uint32_t lo = l0, base = b0, o = o0;
      if (!one) {
        uint32_t hi = most;
        while (lo < hi) {
          const uint32_t mid = (lo + hi + 1) >> 1;
          if (f.l_base[mid] <= k) lo = mid;
          else hi = mid - 1;
        }
        base = f.l_base[lo];
        o = f.l_off[lo];
      }
      l[r] = lo;
      j[r] = k - base;
      e[r] = in[r] ? g.edges[ml.edge_start + o + j[r]] : 0u;
    }
  }
  auto plan = [&](int r, uint64_t before63) {
    return probe_plan<false, true>(g, m, in[r] && (int32_t)e[r] >= 0 ? make_key(e[r], f.pid, f.dir) : 0, before63);
  };
  ProbeCarry carry;
  ProbePlan pl[3];
  pl[0] = plan(0, 0);
  if (RD > 1) pl[1] = plan(1, lane63_64(pl[0].key));
  probe_pick<true>(g, pl[0]);
#pragma unroll
  for (int r = 0; r < RD; r++) {
    if (r + 2 < RD) pl[(r + 2) % 3] = plan(r + 2, lane63_64(pl[(r + 1) % 3].key));
    if (r + 1 < RD) probe_pick<true>(g, pl[(r + 1) % 3]);
    (void)probe_finish<false, true>(g, m, pl[r % 3], s_wp[wave], deg[r], off[r], carry);
  }
  uint64_t ex = 0, spared = 0;  // work counts: all lists whole, and what kept rows need not examine
  uint32_t x[RD];
#pragma unroll
  for (int r = 0; r < RD; r++) {
    ex += deg[r] ? (uint64_t)deg[r] * f.l_np[l[r]] : 0;
    x[r] = deg[r] && deg[r] <= kListInline ? g.edges[m.edge_start + off[r]] : 0u;
  }
#pragma unroll
  for (int r = 0; r < RD; r++) {
    uint32_t n = 0, first = 0;
    if (deg[r] && deg[r] <= kListInline) n = list_match(g, m.edge_start, f, l[r], off[r], 0, x[r], first);
    if (!list_keep<BITS>(f, n, first, j[r], e[r], deg[r] - 1, spared)) return;
    // the further elements of all lanes' lists as one sequence, a lane each
    const uint32_t more = deg[r] > 1 && deg[r] <= kListInline ? deg[r] - 1 : 0u;
    if (wave_ballot(more != 0)) {
      const uint32_t inc = wave_incl_scan32(more), all = lane63(inc), before = inc - more;
      for (uint32_t t0 = 0; t0 < all; t0 += kWave) {  // (wave-uniform)
        const uint32_t t = t0 + lane;
        uint32_t src = 0;  // the last lane whose elements start at or before t (lanes without any share their next's)
#pragma unroll
        for (uint32_t step = kWave / 2; step; step >>= 1)
          if (shfl32(before, src + step) <= t) src += step;
        const uint32_t q = t - shfl32(before, src) + 1, ol = shfl32(l[r], src), oo = shfl32(off[r], src);
        const uint32_t od = shfl32(deg[r], src), oj = shfl32(j[r], src), oe = shfl32(e[r], src);
        n = t < all ? list_match(g, m.edge_start, f, ol, oo, q, g.edges[m.edge_start + oo + q], first) : 0u;
        if (!list_keep<BITS>(f, n, first, oj, oe, od - (q + 1), spared)) return;
      }
    }
    if (deg[r] > kListInline) {
      const uint32_t n = (deg[r] + kListChunk - 1) / kListChunk;
      const uint32_t q = block % kListQueues;
      const uint64_t b = atomicAdd(&f.long_n[q * kListPad], (unsigned long long)n);
      for (uint32_t c = 0; c < n && b + c < f.long_cap; c++)
        f.longs[q * f.long_cap + b + c] = make_uint4(f.l_base[l[r]] + j[r], off[r], deg[r], c * kListChunk);
    }
  }
  ex = lane63_64(wave_incl_scan(ex - spared));
  if (lane == 0) f.ex[block * (kBlock / kWave) + wave] = ex;
}

// The long filter lists, a chunk per workgroup at a time; the first workgroup
// also adds up the work count.
template <bool BITS>
__global__ __launch_bounds__(kBlock) void k_list_long(GraphView g, ListFilter f, uint32_t nl, uint32_t nex) {
  const uint32_t queue = blockIdx.x % kListQueues;
  const uint64_t all = f.long_n[queue * kListPad], n = all < f.long_cap ? all : f.long_cap;
  if (all > n && threadIdx.x == 0) f.ctr[kListLost] = 1;
  if (blockIdx.x == 0) {
    __shared__ uint64_t s_tmp[kBlock / kWave];
    uint64_t v = 0, sum;
#pragma unroll 8
    for (uint32_t i = threadIdx.x; i < nex; i += kBlock) v += f.ex[i];
    (void)block_excl_scan(v, s_tmp, sum);
    if (threadIdx.x == 0) f.ctr[kListEx] = sum;
  }
  uint64_t spared = 0;
  const DevMeta ml = g.meta[f.lpid], m = g.meta[f.pid];
  for (uint64_t i = blockIdx.x / kListQueues; i < n; i += gridDim.x / kListQueues) {
    const uint4 it = f.longs[queue * f.long_cap + i];
    const uint32_t l = (uint32_t)wave_last_le(nl, it.x, [&](uint64_t q) -> uint64_t { return f.l_base[q]; });
    const uint32_t j = it.x - f.l_base[l], e = g.edges[ml.edge_start + f.l_off[l] + j];
    uint32_t v[kListChunk / kBlock];
#pragma unroll
    for (int u = 0; u < (int)(kListChunk / kBlock); u++) {
      const uint32_t q = it.w + threadIdx.x + u * kBlock;
      v[u] = q < it.z ? g.edges[m.edge_start + it.y + q] : 0u;
    }
#pragma unroll
    for (int u = 0; u < (int)(kListChunk / kBlock); u++) {
      const uint32_t q = it.w + threadIdx.x + u * kBlock;
      uint32_t first = 0;
      const uint32_t n = q < it.z ? list_match(g, m.edge_start, f, l, it.y, q, v[u], first) : 0u;
      if (!list_keep<BITS>(f, n, first, j, e, it.z - (q + 1), spared)) return;  // (a wave as a whole; no barrier below)
    }
  }
  spared = lane63_64(wave_incl_scan(spared));
  if (spared && lane_id() == 0) atomicAdd(&f.ctr[kListSpared], (unsigned long long)spared);
}

// Kept rows of each tile of 1024 rows, for the tile scan; the work count is
// the list pass's.
__global__ __launch_bounds__(kBlock) void k_bit_tiles(StepParams p, const uint32_t *bits) {
  const uint64_t lt = blockIdx.x * (uint64_t)kBlock + threadIdx.x;
  if (lt >= p.ntiles) return;
  const uint4 *w = (const uint4 *)(bits + lt * (kListBitRows / 32));
  uint32_t n = 0;
#pragma unroll
  for (int k = 0; k < kListBitRows / 128; k++) {
    const uint4 v = gload(w + k);
    n += __builtin_popcount(v.x) + __builtin_popcount(v.y) + __builtin_popcount(v.z) + __builtin_popcount(v.w);
  }
  p.tile_sum[lt] = p.tile_nz[lt] = n;
  p.tile_ex[lt] = 0;
}

// The n kept rows in row order: the 16 lanes of a group count the rows before
// their own, then write it (the parent's cells and the list entry).
constexpr uint32_t kRankLanes = 16;
__global__ __launch_bounds__(kBlock) void k_list_rows(ListFilter f, uint32_t n, int32_t *O) {
  constexpr uint32_t kTile = kBlock * 4;
  __shared__ __align__(16) uint32_t s_row[kTile];
  const uint32_t k = blockIdx.x * (kBlock / kRankLanes) + threadIdx.x / kRankLanes, g16 = threadIdx.x % kRankLanes;
  const uint4 mine = k < n ? f.kept[k] : make_uint4(0, 0, 0, 0);
  uint32_t rank = 0;
  for (uint32_t b = 0; b < n; b += kTile) {
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kTile; i += kBlock) s_row[i] = b + i < n ? f.kept[b + i].x : 0xffffffffu;
    __syncthreads();
    for (uint32_t i = g16 * 4; i < kTile; i += kRankLanes * 4) {
      const uint4 q = *(const uint4 *)&s_row[i];
      rank += (q.x < mine.x) + (q.y < mine.x) + (q.z < mine.x) + (q.w < mine.x);
    }
  }
#pragma unroll
  for (uint32_t d = kRankLanes / 2; d; d >>= 1) rank += shfl32(rank, lane_id() ^ d);
  if (k >= n) return;
  const int32_t *prow = f.P + (uint64_t)f.info[mine.y].x * f.pc;
  int32_t *o = O + (uint64_t)rank * (f.pc + 1);
  for (uint32_t c = g16; c < f.pc; c += kRankLanes) o[c] = prow[c];
  if (g16 == 0) o[f.pc] = (int32_t)mine.z;
}

// Compaction of the kept rows k_fanout_blocks listed: one thread per kept
// row, its place = its unit's prefix from the two-level scan + its index in
// the unit; the row is built from its lineage as in k_compact_lineage.
__global__ __launch_bounds__(kBlock) void k_compact_kept(GraphView g, StepParams p, const uint4 *kept, uint64_t n,
                                                         FanoutFilter f, uint64_t edge_start) {
  const uint64_t k = blockIdx.x * (uint64_t)kBlock + threadIdx.x;
  if (k >= n) return;
  const uint4 e = kept[k];
  const uint64_t r = e.x, rank = e.y;
  const uint64_t o = p.tile_nz[rank] + (p.chunk_nz ? p.chunk_nz[rank / kScanChunk] : 0) + e.z;
  uint64_t lo = 0, hi = f.np - 1;
  while (lo < hi) {
    const uint64_t mid = (lo + hi + 1) >> 1;
    if (f.excl[mid] <= r) lo = mid;
    else hi = mid - 1;
  }
  const uint32_t c = p.c, pc = f.pc;
  const uint2 inf = f.info[lo];
  const int32_t *prow = f.P + (uint64_t)inf.x * pc;
  for (uint32_t col = 0; col < pc; col++) p.O[o * c + col] = prow[col];
  p.O[o * c + pc] = (int32_t)g.edges[edge_start + inf.y + (r - f.excl[lo])];
}

// Compaction of a fan-out filter's kept rows: one wave per tile reads the
// tile's TR / 32 bit words and copies each kept row of T to its place in O
// (the tile's prefix from the two-level scan, then bit order).
template <int TR>
__global__ __launch_bounds__(kBlock) void k_compact_bits(StepParams p, const uint32_t *bits, const uint64_t *row0) {
  static_assert(TR / 32 <= kWave, "one word per lane");
  const uint64_t lt = p.tile0 + blockIdx.x * (uint64_t)(kBlock / kWave) + threadIdx.x / kWave;
  if (lt >= p.ntiles) return;
  const uint64_t r_base = row0 ? row0[lt] : lt * TR;  // unit-ranked tiles carry their first row
  const uint32_t lane = lane_id();
  const uint32_t w = lane < TR / 32 ? bits[lt * (TR / 32) + lane] : 0u;
  if (!wave_ballot(w != 0)) return;
  const uint64_t pre = p.tile_nz[lt] + (p.chunk_nz ? p.chunk_nz[lt / kScanChunk] : 0);
  const uint64_t inc = wave_incl_scan((uint64_t)__builtin_popcount(w));
  uint64_t o = pre + inc - (uint64_t)__builtin_popcount(w);
  const uint32_t c = p.c;
  for (uint32_t x = w; x; x &= x - 1) {
    const uint64_t r = r_base + (uint64_t)lane * 32 + (uint32_t)__builtin_ctz(x);
    for (uint32_t col = 0; col < c; col++) p.O[o * c + col] = p.T[r * c + col];
    o++;
  }
}

// The same compaction for a fan-out that was never written: kept row r is
// built from its lineage -- the parent row (the last compacted parent whose
// first child row is <= r, a binary search) and that parent's list entry
// r - its first child row, of the step's predicate (resident graph).
template <int TR>
__global__ __launch_bounds__(kBlock) void k_compact_lineage(GraphView g, StepParams p, const uint32_t *bits,
                                                            const uint64_t *row0, FanoutFilter f,
                                                            uint64_t edge_start) {
  static_assert(TR / 32 <= kWave, "one word per lane");
  const uint64_t lt = p.tile0 + blockIdx.x * (uint64_t)(kBlock / kWave) + threadIdx.x / kWave;
  if (lt >= p.ntiles) return;
  const uint64_t r_base = row0 ? row0[lt] : lt * TR;
  const uint32_t lane = lane_id();
  const uint32_t w = lane < TR / 32 ? bits[lt * (TR / 32) + lane] : 0u;
  if (!wave_ballot(w != 0)) return;
  const uint64_t pre = p.tile_nz[lt] + (p.chunk_nz ? p.chunk_nz[lt / kScanChunk] : 0);
  const uint64_t inc = wave_incl_scan((uint64_t)__builtin_popcount(w));
  uint64_t o = pre + inc - (uint64_t)__builtin_popcount(w);
  const uint32_t c = p.c, pc = f.pc;
  for (uint32_t x = w; x; x &= x - 1) {
    const uint64_t r = r_base + (uint64_t)lane * 32 + (uint32_t)__builtin_ctz(x);
    uint64_t lo = 0, hi = f.np - 1;
    while (lo < hi) {
      const uint64_t mid = (lo + hi + 1) >> 1;
      if (f.excl[mid] <= r) lo = mid;
      else hi = mid - 1;
    }
    const uint2 inf = f.info[lo];
    const int32_t *prow = f.P + (uint64_t)inf.x * pc;
    for (uint32_t col = 0; col < pc; col++) p.O[o * c + col] = prow[col];
    p.O[o * c + pc] = (int32_t)g.edges[edge_start + inf.y + (r - f.excl[lo])];
    o++;
  }
}

}  // namespace
}  // namespace wkg
