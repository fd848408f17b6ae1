// Stable counting sort of one species' particles by cell key.
//
// Semantics: the stable counting sort of LPFx's host sort
// (include/lpfx/algorithm/particle/host/sort.hpp:210-305): counts[bin] is the
// key histogram over the (nx+4)(ny+4)(nz+4) halo-2 bins, offsets its exclusive
// scan with offsets[bins] = N, and the particles of a bin keep their input
// order. The reference's device sort
// (include/lpfx/algorithm/particle/device/cuda_hip/sort.hpp:27-260) gives the
// same counts and offsets but an atomic, run-dependent order inside a bin;
// this sort is deterministic and equals the stable order.
//
// MI355X design: after a mover the keys are nearly sorted, so the input is a
// short sequence of runs of equal keys. The sort counts and orders RUNS, not
// particles: (1) run heads per 4096-particle tile, (2) tile scan, (3) run
// table, (4) run histogram with run lengths, (5) bin scans, (6) runs scattered
// to their bins, (7) inside a bin, runs ordered by run id (= input order) give
// each run its destination, (8) one destination-ordered pass (a wave per bin)
// copies the nine SoA attributes, so every output line is written whole and
// only the particles that changed cell are scattered loads. Particle traffic
// is two key passes for the runs and the attribute copy (about 144 B per FP64
// particle). In the cycle, a species sorted before a block move is planned
// from the particles that move changed instead (launch_sort_plan_incremental).
#include "internal.hpp"

namespace tpic_mi {
namespace {

constexpr unsigned kThreads = 256;
constexpr unsigned kItems = 16;
constexpr unsigned kTile = kThreads * kItems;

// Exclusive prefix of a per-thread flag over a 256-thread block, in thread
// order; also returns the block total.
__device__ inline uint32_t scan_flags(bool flag, uint32_t* lds, uint32_t& total) {
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const unsigned long long mask = __ballot(flag);
  const unsigned long long below = lane == 0 ? 0ull : (mask & ((1ull << lane) - 1ull));
  const uint32_t within = uint32_t(__popcll(below));
  if (lane == 0) lds[wave] = uint32_t(__popcll(mask));
  __syncthreads();
  uint32_t before = 0, sum = 0;
#pragma unroll
  for (unsigned w = 0; w < kThreads / 64; ++w) {
    const uint32_t v = lds[w];
    before += w < wave ? v : 0u;
    sum += v;
  }
  __syncthreads();
  total = sum;
  return before + within;
}

__device__ inline uint32_t block_sum(uint32_t v, uint32_t* lds) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  if (lane == 0) lds[wave] = v;
  __syncthreads();
  uint32_t sum = 0;
  for (unsigned w = 0; w < blockDim.x / 64; ++w) sum += lds[w];
  __syncthreads();
  return sum;
}

__global__ __launch_bounds__(kThreads) void k_tile_heads(const int32_t* __restrict__ keys, uint32_t n,
                                                         uint32_t bins, uint32_t* __restrict__ tile_runs,
                                                         uint32_t* __restrict__ failure) {
  __shared__ uint32_t lds[kThreads / 64];
  const uint32_t base = blockIdx.x * kTile;
  uint32_t heads = 0;
  bool bad = false;
#pragma unroll 4
  for (unsigned r = 0; r < kItems; ++r) {
    const uint32_t i = base + r * kThreads + threadIdx.x;
    if (i < n) {
      const int32_t key = keys[i];
      bad |= key < 0 || uint32_t(key) >= bins;
      heads += (i == 0 || keys[i - 1] != key) ? 1u : 0u;
    }
  }
  if (bad) atomicOr(failure, 1u);
  const uint32_t total = block_sum(heads, lds);
  if (threadIdx.x == 0) tile_runs[blockIdx.x] = total;
}

// Each wave of a tile takes a contiguous span of kWaveSpan keys, 64 at a
// time, and keeps the head flags of its span as ballot words.
constexpr unsigned kWaveSpan = kTile / (kThreads / 64);
constexpr unsigned kWaveItems = kWaveSpan / 64;

__device__ inline uint64_t lanes_below(unsigned lane) { return lane == 0 ? 0ull : ((1ull << lane) - 1ull); }

// Set bits of the words (lo, hi) below this lane (v_mbcnt_lo/hi).
__device__ __forceinline__ uint32_t bits_below(uint32_t lo, uint32_t hi) {
  return __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
}

// Waits for every vector memory load of the wave (s_waitcnt vmcnt(0)): the
// stores that follow, each under its own lane mask, then need no further waits
// on the loaded values.
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }


// Run table and histogram in one pass over the keys, after the scan of the
// tile head counts: run_start[r] and run_key[r] for every head in input
// order; counts[key] gains each run's length and rcounts[key] one per run,
// as integer atomics per run segment (a run continued from an earlier wave
// span adds its leading segment there), so the sums do not depend on their
// order. wave_base[] keeps the number of heads before each wave span for
// k_tile_sources; the tile holding the last key closes the run table.
__global__ __launch_bounds__(kThreads) void k_tile_runs(const int32_t* __restrict__ keys, uint32_t n,
                                                        uint32_t tiles, const uint32_t* __restrict__ tile_base,
                                                        uint32_t* __restrict__ run_start,
                                                        int32_t* __restrict__ run_key,
                                                        uint32_t* __restrict__ counts,
                                                        uint32_t* __restrict__ rcounts,
                                                        uint32_t* __restrict__ wave_base,
                                                        const uint32_t* __restrict__ failure) {
  if (*failure) return;
  __shared__ uint32_t lds[kThreads / 64];
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t sub = blockIdx.x * kTile + wave * kWaveSpan;
  uint64_t heads[kWaveItems];
  int32_t key[kWaveItems];
  uint32_t count = 0;
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint32_t i = sub + r * 64 + lane;
    bool head = false;
    key[r] = 0;
    if (i < n) {
      key[r] = keys[i];
      head = i == 0 || keys[i - 1] != key[r];
    }
    heads[r] = __ballot(head);
    count += uint32_t(__popcll(heads[r]));
  }
  if (lane == 0) lds[wave] = count;
  __syncthreads();
  uint32_t before = tile_base[blockIdx.x];
  uint32_t tile_total = before;
#pragma unroll
  for (unsigned w = 0; w < kThreads / 64; ++w) {
    before += w < wave ? lds[w] : 0u;
    tile_total += lds[w];
  }
  if (lane == 0) wave_base[blockIdx.x * (kThreads / 64) + wave] = before;
  if (blockIdx.x == tiles - 1 && threadIdx.x == 0) run_start[tile_total] = n;
  const uint32_t end = sub + kWaveSpan < n ? sub + kWaveSpan : n;
  uint32_t rank = before;
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint64_t m = heads[r];
    if ((m >> lane) & 1ull) {
      const uint32_t i = sub + r * 64 + lane;
      const uint32_t id = rank + uint32_t(__popcll(m & lanes_below(lane)));
      run_start[id] = i;
      run_key[id] = key[r];
      // The run's segment in this span ends at the span's next head.
      uint32_t next = end;
      const uint64_t above = lane == 63 ? 0ull : (m >> (lane + 1));
      if (above) {
        next = i + 1u + uint32_t(__builtin_ctzll(above));
      } else {
#pragma unroll
        for (unsigned r2 = r + 1; r2 < kWaveItems; ++r2)
          if (next == end && heads[r2]) next = sub + r2 * 64 + uint32_t(__builtin_ctzll(heads[r2]));
      }
      atomicAdd(counts + key[r], next - i);
      atomicAdd(rcounts + key[r], 1u);
    }
    rank += uint32_t(__popcll(m));
  }
  // The span's keys before its first head continue a run of an earlier span.
  if (lane == 0 && sub < n && !(heads[0] & 1ull)) {
    uint32_t first = end;
#pragma unroll
    for (unsigned r2 = 0; r2 < kWaveItems; ++r2)
      if (first == end && heads[r2]) first = sub + r2 * 64 + uint32_t(__builtin_ctzll(heads[r2]));
    atomicAdd(counts + key[0], first - sub);
  }
}

// The plan alone, in source order: particle i of run r lands at
// run_dest[r] + (i - run_start[r]), so source[that] = i (and, when recorded,
// permutation[i] = that). A particle's run is the last head at or before it:
// its rank among the heads, counted from the wave span's base.
__global__ __launch_bounds__(kThreads) void k_tile_sources(const int32_t* __restrict__ keys, uint32_t n,
                                                           const uint32_t* __restrict__ wave_base,
                                                           const uint32_t* __restrict__ run_start,
                                                           const uint32_t* __restrict__ run_dest,
                                                           uint32_t* __restrict__ source,
                                                           uint32_t* __restrict__ permutation,
                                                           const uint32_t* __restrict__ failure) {
  if (*failure) return;
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t sub = blockIdx.x * kTile + wave * kWaveSpan;
  if (sub >= n) return;
  // All keys of the span first (the key before each one comes from the lane
  // below, or the item before), then every run's table entries, then the
  // stores: the loads of a phase are in flight together.
  int32_t key[kWaveItems];
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint32_t i = sub + r * 64 + lane;
    key[r] = i < n ? keys[i] : -1;
  }
  const int32_t before_span = (lane == 0 && sub > 0) ? keys[sub - 1] : -1;
  uint32_t before = wave_base[blockIdx.x * (kThreads / 64) + wave];
  const uint64_t upto = lanes_below(lane) | (1ull << lane);
  uint32_t run[kWaveItems];
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint32_t i = sub + r * 64 + lane;
    const int32_t below = __shfl_up(key[r], 1u, 64);
    const int32_t carried = __shfl(r == 0 ? before_span : key[r > 0 ? r - 1 : 0], 63, 64);
    const int32_t prev = lane == 0 ? (r == 0 ? before_span : carried) : below;
    const bool head = i < n && (i == 0 || prev != key[r]);
    const uint64_t m = __ballot(head);
    run[r] = before + uint32_t(__popcll(m & upto)) - 1u;
    before += uint32_t(__popcll(m));
  }
  uint32_t dest[kWaveItems], start[kWaveItems];
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint32_t i = sub + r * 64 + lane;
    dest[r] = i < n ? run_dest[run[r]] : 0u;
    start[r] = i < n ? run_start[run[r]] : 0u;
  }
  wait_loads();
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint32_t i = sub + r * 64 + lane;
    if (i < n) {
      const uint32_t d = dest[r] + (i - start[r]);
      source[d] = i;
      if (permutation) permutation[i] = d;
    }
  }
}

__global__ __launch_bounds__(kThreads) void k_run_scatter(const uint32_t* __restrict__ tile_base, uint32_t tiles,
                                                          const int32_t* __restrict__ run_key,
                                                          const uint32_t* __restrict__ roffsets,
                                                          uint32_t* __restrict__ cursor,
                                                          uint32_t* __restrict__ bin_runs,
                                                          const uint32_t* __restrict__ failure) {
  if (*failure) return;
  const uint32_t runs = tile_base[tiles];
  for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < runs; r += gridDim.x * blockDim.x) {
    const int32_t key = run_key[r];
    bin_runs[roffsets[key] + atomicAdd(cursor + key, 1u)] = r;
  }
}

// Destination of every run: the bin offset plus the lengths of the bin's runs
// with a smaller run id (earlier in the input). Bins with at most kSmall runs
// are done by one thread; others are listed for k_bin_large.
constexpr uint32_t kSmall = 24;

__global__ __launch_bounds__(kThreads) void k_bin_small(Grid g, const uint32_t* __restrict__ rcounts,
                                                        const uint32_t* __restrict__ roffsets,
                                                        const uint32_t* __restrict__ offsets,
                                                        const uint32_t* __restrict__ bin_runs,
                                                        const uint32_t* __restrict__ run_start,
                                                        uint32_t* __restrict__ run_dest,
                                                        uint32_t* __restrict__ large,
                                                        unsigned* __restrict__ validation,
                                                        const uint32_t* __restrict__ failure) {
  if (*failure) return;
  const uint32_t bins = g.bins();
  for (uint32_t b = blockIdx.x * blockDim.x + threadIdx.x; b < bins; b += gridDim.x * blockDim.x) {
    const uint32_t nr = rcounts[b];
    if (nr == 0) continue;
    int i, j, k;
    g.decode(int32_t(b), i, j, k);
    if (!g.interior(i, j, k)) atomicOr(validation, kInvalidHalo);
    const uint32_t first = roffsets[b];
    if (nr > kSmall) {
      large[1 + atomicAdd(large, 1u)] = b;
      continue;
    }
    uint32_t id[kSmall], len[kSmall];
    for (uint32_t t = 0; t < nr; ++t) {
      id[t] = bin_runs[first + t];
      len[t] = run_start[id[t] + 1] - run_start[id[t]];
    }
    const uint32_t base = offsets[b];
    for (uint32_t t = 0; t < nr; ++t) {
      uint32_t d = base;
      for (uint32_t f = 0; f < nr; ++f) d += id[f] < id[t] ? len[f] : 0u;
      run_dest[id[t]] = d;
    }
  }
}

__global__ __launch_bounds__(kThreads) void k_bin_large(const uint32_t* __restrict__ large,
                                                        const uint32_t* __restrict__ rcounts,
                                                        const uint32_t* __restrict__ roffsets,
                                                        const uint32_t* __restrict__ offsets,
                                                        const uint32_t* __restrict__ bin_runs,
                                                        const uint32_t* __restrict__ run_start,
                                                        uint32_t* __restrict__ run_dest,
                                                        const uint32_t* __restrict__ failure) {
  if (*failure) return;
  __shared__ uint32_t s_id[kThreads], s_len[kThreads];
  const uint32_t listed = large[0];
  for (uint32_t l = blockIdx.x; l < listed; l += gridDim.x) {
    const uint32_t b = large[1 + l];
    const uint32_t nr = rcounts[b], first = roffsets[b], base = offsets[b];
    for (uint32_t e0 = 0; e0 < nr; e0 += kThreads) {
      const uint32_t e = e0 + threadIdx.x;
      const uint32_t mine = e < nr ? bin_runs[first + e] : 0u;
      uint32_t d = base;
      for (uint32_t f0 = 0; f0 < nr; f0 += kThreads) {
        __syncthreads();
        const uint32_t f = f0 + threadIdx.x;
        if (f < nr) {
          const uint32_t r = bin_runs[first + f];
          s_id[threadIdx.x] = r;
          s_len[threadIdx.x] = run_start[r + 1] - run_start[r];
        }
        __syncthreads();
        const uint32_t m = nr - f0 < kThreads ? nr - f0 : kThreads;
        for (uint32_t t = 0; t < m; ++t) d += s_id[t] < mine ? s_len[t] : 0u;
      }
      if (e < nr) run_dest[mine] = d;
    }
    __syncthreads();
  }
}

// The nine attributes of one particle (68 B).
struct Record {
  double rx, ry, rz, u, v, w, q;
  int32_t cell;
  uint64_t id;
};

__device__ __forceinline__ void load_record(const ParticleView& p, uint32_t i, Record& r) {
  r.rx = p.rx[i];
  r.ry = p.ry[i];
  r.rz = p.rz[i];
  r.u = p.u[i];
  r.v = p.v[i];
  r.w = p.w[i];
  r.q = p.q[i];
  r.cell = p.cell[i];
  r.id = p.id[i];
}

__device__ __forceinline__ void store_record(const ParticleView& p, uint32_t i, const Record& r) {
  p.rx[i] = r.rx;
  p.ry[i] = r.ry;
  p.rz[i] = r.rz;
  p.u[i] = r.u;
  p.v[i] = r.v;
  p.w[i] = r.w;
  p.q[i] = r.q;
  p.cell[i] = r.cell;
  p.id[i] = r.id;
}

// Destination-ordered copy: one wave per bin writes the bin's destination
// range [offsets[b], offsets[b] + count) in order, each lane taking the next
// particle from the run that covers its destination (run r covers
// [run_dest[r], run_dest[r] + length) and starts at source run_start[r]).
// Stores are contiguous per bin, so every line of the output is written whole
// by one or two waves close in time; the particles that changed cell are the
// only scattered accesses, and they are loads. Bins with more than 64 runs
// take the general loop.
__global__ __launch_bounds__(kThreads) void k_gather_bins(Grid g, ParticleView src, ParticleView dst, RunPlan plan,
                                                          uint32_t* __restrict__ permutation) {
  if (*plan.failure) return;
  const uint32_t bins = g.bins();
  const unsigned lane = threadIdx.x & 63u;
  const uint32_t waves = gridDim.x * (kThreads / 64);
  // XCD-aware: an XCD's waves take neighbouring bins, so the output lines two
  // adjacent bins share are completed in one L2.
  const uint32_t first_bin = xcd_logical_block(blockIdx.x, gridDim.x) * (kThreads / 64) + (threadIdx.x >> 6);
  for (uint32_t b = __builtin_amdgcn_readfirstlane(first_bin); b < bins; b += waves) {
    if (plan.rcounts[b] == 0) continue;
    BinRuns br;
    load_bin_runs(plan, b, lane, br);
    const uint32_t count = plan.counts[b], base = plan.offsets[b];
    for (uint32_t i = lane; i < count; i += 64) {
      const uint32_t d = base + i;
      const uint32_t from = run_source(plan, br, d);
      Record rec;
      load_record(src, from, rec);
      store_record(dst, d, rec);
      if (permutation) permutation[from] = d;
    }
  }
}

// The records of the halo bins of a plan (particles left outside the
// interior, flagged by k_bin_small): the fused gather and deposition visits
// interior cells only, so these are copied here, one thread per bin.
__global__ __launch_bounds__(kThreads) void k_copy_halo_bins(Grid g, ParticleView src, ParticleView dst,
                                                             const uint32_t* __restrict__ counts,
                                                             const uint32_t* __restrict__ offsets,
                                                             const uint32_t* __restrict__ source,
                                                             const uint32_t* __restrict__ failure) {
  if (*failure) return;
  const uint32_t bins = g.bins();
  for (uint32_t b = blockIdx.x * blockDim.x + threadIdx.x; b < bins; b += gridDim.x * blockDim.x) {
    const uint32_t count = counts[b];
    if (count == 0) continue;
    int i, j, k;
    g.decode(int32_t(b), i, j, k);
    if (g.interior(i, j, k)) continue;
    for (uint32_t d = offsets[b]; d < offsets[b] + count; ++d) {
      Record rec;
      load_record(src, source[d], rec);
      store_record(dst, d, rec);
    }
  }
}

// Identity copy after a failed plan (invalid keys): particles keep their
// order (and, when given, every destination is its own source).
__global__ __launch_bounds__(kThreads) void k_copy_on_failure(ParticleView src, ParticleView dst, uint32_t n,
                                                              uint32_t* __restrict__ permutation,
                                                              const uint32_t* __restrict__ failure,
                                                              uint32_t* __restrict__ source) {
  if (*failure == 0) return;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    Record rec;
    load_record(src, i, rec);
    store_record(dst, i, rec);
    if (permutation) permutation[i] = i;
    if (source) source[i] = i;
  }
}

__global__ void k_sort_failed(const uint32_t* failure, unsigned* validation) {
  if (*failure) atomicOr(validation, kInvalidSort);
}

// ---- device-wide exclusive scan of uint32 (out has n + 1 entries) --------
constexpr unsigned kScanItems = 8;
constexpr unsigned kScanBlock = kThreads * kScanItems;

__global__ __launch_bounds__(kThreads) void k_scan_reduce(const uint32_t* __restrict__ in, uint32_t n,
                                                          uint32_t* __restrict__ sums) {
  __shared__ uint32_t lds[kThreads / 64];
  const uint32_t base = blockIdx.x * kScanBlock;
  uint32_t s = 0;
#pragma unroll
  for (unsigned r = 0; r < kScanItems; ++r) {
    const uint32_t i = base + r * kThreads + threadIdx.x;
    s += i < n ? in[i] : 0u;
  }
  const uint32_t total = block_sum(s, lds);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// Exclusive scan of one block of kScanBlock items with an added offset;
// writes out[n] (the total) from the block holding the last item.
__global__ __launch_bounds__(kThreads) void k_scan_apply(const uint32_t* __restrict__ in, uint32_t n,
                                                         const uint32_t* __restrict__ block_offset,
                                                         uint32_t* __restrict__ out) {
  __shared__ uint32_t lds[kThreads / 64];
  const uint32_t base = blockIdx.x * kScanBlock;
  // Blocked arrangement: thread t owns items t*8 .. t*8+7 of the block.
  uint32_t v[kScanItems];
  uint32_t s = 0;
#pragma unroll
  for (unsigned r = 0; r < kScanItems; ++r) {
    const uint32_t i = base + threadIdx.x * kScanItems + r;
    v[r] = i < n ? in[i] : 0u;
    s += v[r];
  }
  // Exclusive scan of per-thread sums across the block.
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t inc = s;
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t t = __shfl_up(inc, off, 64);
    if (int(lane) >= off) inc += t;
  }
  if (lane == 63) lds[wave] = inc;
  __syncthreads();
  uint32_t before = 0, total = 0;
  for (unsigned w = 0; w < kThreads / 64; ++w) {
    before += w < wave ? lds[w] : 0u;
    total += lds[w];
  }
  uint32_t running = (block_offset ? block_offset[blockIdx.x] : 0u) + before + inc - s;
#pragma unroll
  for (unsigned r = 0; r < kScanItems; ++r) {
    const uint32_t i = base + threadIdx.x * kScanItems + r;
    if (i < n) out[i] = running;
    running += v[r];
  }
  const uint32_t last_block = n == 0 ? 0 : (n - 1) / kScanBlock;
  if (blockIdx.x == last_block && threadIdx.x == 0)
    out[n] = (block_offset ? block_offset[blockIdx.x] : 0u) + total;
}

// ---- The incremental plan: a sorted species after the block mover ----
//
// The block mover records, per aligned 64-particle block, the lanes whose key
// it changed (crossers). Every other particle (a stayer) still lies in its
// key's bin range of the previous plan, in input order. The stable order of a
// bin is therefore: its arrivals (crossers with the bin as new key) from
// earlier positions (lower bins), in position order; its stayers, in position
// order; its arrivals from later positions. Every stayer's destination is its
// bin's base plus its position less the crossers before it; each bin orders
// its arrivals by position. A bin with more than kArrivalsMax arrivals, or an
// old state in which the stayers and crossers do not add up to the particles
// (a previous plan that failed), sets the species' plan status: the run-based
// plan is then run instead.
//
// Seven launches for one or two species (blockIdx.y), each with what it needs
// cleared, counted or scanned folded in: a scan over tiles is two passes, the
// second of which adds the tiles before its own by itself. As clears, counts
// and three-launch scans of their own they were nineteen a species, 130 us of
// launches a cycle at 16^3.
constexpr uint32_t kArrivalsMax = 1024;
constexpr uint32_t kArrivalsInRegisters = 12;

struct CrossPlan {
  const int32_t* keys;
  const uint64_t* cross;
  uint32_t n, blocks;       // particles, 64-particle blocks
  uint32_t* block_base;     // [blocks + 1] crossers before each block
  uint32_t* arrivals;       // [bins]
  uint32_t* arrival_offset; // [bins + 1]
  uint32_t* lower;          // [bins] arrivals from lower bins
  uint32_t* slot;           // per crosser: its index among its bin's arrivals
  uint32_t* shift;          // [bins] crossers before the old range less its start
  uint32_t* bin_base;       // [bins] stayer destination base
  uint32_t* bin_arrivals;   // positions of the arrivals, by bin
  uint32_t* tile_a;         // tile sums: crossers, then counts
  uint32_t* tile_b;         // tile sums: arrivals
  uint32_t* counts;
  uint32_t* offsets;
  uint32_t* source;
  uint32_t* status;
  ParticleView src, dst;
};

struct CrossPlans {
  CrossPlan species[2];
};

// Bins and 64-particle blocks per tile of the plan's scans: two a thread, so a
// small grid's few thousand still spread over the chip (eight a thread: 15 us
// instead of 5 for the new counts at 16^3).
constexpr unsigned kPlanItems = 2;
constexpr unsigned kPlanTile = kThreads * kPlanItems;

// Sum of tiles[0 .. last), in every thread.
__device__ inline uint32_t tiles_before(const uint32_t* __restrict__ tiles, uint32_t last, uint32_t* lds) {
  uint32_t v = 0;
  for (uint32_t t = threadIdx.x; t < last; t += kThreads) v += tiles[t];
  return block_sum(v, lds);
}

// Exclusive prefix of a value per thread over the block.
__device__ inline uint32_t block_exclusive(uint32_t v, uint32_t* lds) {
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t inc = v;
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t t = __shfl_up(inc, off, 64);
    if (int(lane) >= off) inc += t;
  }
  if (lane == 63) lds[wave] = inc;
  __syncthreads();
  uint32_t before = 0;
  for (unsigned w = 0; w < kThreads / 64; ++w) before += w < wave ? lds[w] : 0u;
  __syncthreads();
  return before + inc - v;
}

__device__ __forceinline__ uint32_t crossers_before(const uint64_t* __restrict__ cross,
                                                    const uint32_t* __restrict__ block_base, uint32_t blocks,
                                                    uint32_t p) {
  const uint32_t blk = p >> 6, bit = p & 63u;
  if (blk >= blocks) return block_base[blocks];
  const uint32_t below = bit ? uint32_t(__popcll(cross[blk] & ((1ull << bit) - 1ull))) : 0u;
  return block_base[blk] + below;
}

// Crossers per tile of kPlanTile blocks, the bins' arrival counts cleared.
__global__ __launch_bounds__(kThreads) void k_cross_begin(CrossPlans plans, uint32_t bins) {
  const CrossPlan& s = plans.species[blockIdx.y];
  __shared__ uint32_t lds[kThreads / 64];
  const uint32_t base = blockIdx.x * kPlanTile + threadIdx.x;
  if (base == 0) *s.status = 0;
  uint32_t sum = 0;
#pragma unroll
  for (unsigned r = 0; r < kPlanItems; ++r) {
    const uint32_t i = base + r * kThreads;
    if (i < s.blocks) sum += uint32_t(__popcll(s.cross[i]));
    if (i < bins) {
      s.arrivals[i] = 0;
      s.lower[i] = 0;
    }
  }
  const uint32_t total = block_sum(sum, lds);
  if (threadIdx.x == 0 && blockIdx.x * kPlanTile < s.blocks) s.tile_a[blockIdx.x] = total;
}

// Crossers before each block.
__global__ __launch_bounds__(kThreads) void k_cross_bases(CrossPlans plans) {
  const CrossPlan& s = plans.species[blockIdx.y];
  if (blockIdx.x * kPlanTile >= s.blocks) return;
  __shared__ uint32_t lds[kThreads / 64];
  const uint32_t first = blockIdx.x * kPlanTile + threadIdx.x * kPlanItems;
  uint32_t v[kPlanItems], sum = 0;
#pragma unroll
  for (unsigned r = 0; r < kPlanItems; ++r) {
    v[r] = first + r < s.blocks ? uint32_t(__popcll(s.cross[first + r])) : 0u;
    sum += v[r];
  }
  uint32_t running = tiles_before(s.tile_a, blockIdx.x, lds);
  running += block_exclusive(sum, lds);
#pragma unroll
  for (unsigned r = 0; r < kPlanItems; ++r) {
    if (first + r < s.blocks) s.block_base[first + r] = running;
    running += v[r];
    if (first + r + 1 == s.blocks) s.block_base[s.blocks] = running;
  }
}

// The present lanes of a wave that hold the lane's key: the first, how many,
// and how many before it. A turn per distinct key.
struct KeyGroup {
  uint32_t first, size, rank;
};
__device__ __forceinline__ KeyGroup key_group(bool present, int32_t key, unsigned lane) {
  KeyGroup g{lane, 1u, 0u};
  uint64_t left = __ballot(present);
  while (left) {
    const unsigned first = unsigned(__builtin_ctzll(left));
    const bool same = present && key == __builtin_amdgcn_readlane(key, first);
    const uint64_t lanes = __ballot(same);
    if (same) g = KeyGroup{first, uint32_t(__popcll(lanes)), bits_below(uint32_t(lanes), uint32_t(lanes >> 32))};
    left &= ~lanes;
  }
  return g;
}

// Per crosser one arrival in its new bin (integer atomics: crosser t of the
// position-ordered crosser list keeps the arrival's index j within the bin in
// slot[t]; the bins order their arrivals by position afterwards), counted as
// from a lower bin when its position precedes the bin's old range. Tiles of
// kTile particles: the crosser words of a wave span and every crosser's key
// are loaded first, then the atomics and range starts, then the stores.
// Grouped: the crossers of a wave's item that enter the same bin arrive with
// one atomic of their number. Atomics at one address follow one another, and in
// full cells the neighbours cross into the same few bins: a line of 1000 a cell
// 423 us a cycle one by one, 389 grouped; 512 x 512 of 100 a cell 5992 and 5894.
// In cells of few particles nearly every key is its own turn of the grouping,
// so below 80 a cell each arrives alone.
template <bool Grouped>
__global__ __launch_bounds__(kThreads) void k_cross_arrivals(CrossPlans plans, uint32_t bins) {
  const CrossPlan& s = plans.species[blockIdx.y];
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t sub = blockIdx.x * kTile + wave * kWaveSpan;
  if (sub >= s.n) return;
  const uint32_t blk0 = sub >> 6;  // sub is a multiple of 64
  const bool item_lane = lane < kWaveItems && sub + lane * 64u < s.n;
  const uint64_t words = item_lane ? s.cross[blk0 + lane] : 0ull;
  const uint32_t bases = item_lane ? s.block_base[blk0 + lane] : 0u;
  uint32_t crossers = 0;  // bit r: the lane's particle of item r is a crosser
  uint32_t list[kWaveItems];  // its index in the crosser list
  int32_t key[kWaveItems];
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(words)), int(r)));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(words >> 32)), int(r)));
    const bool crosser = ((lane < 32u ? lo : hi) >> (lane & 31u)) & 1u;
    crossers |= uint32_t(crosser) << r;
    list[r] = uint32_t(__builtin_amdgcn_readlane(int(bases), int(r))) + bits_below(lo, hi);
    key[r] = crosser ? s.keys[sub + r * 64 + lane] : -1;
  }
  if (crossers == 0) return;
  wait_loads();
  uint32_t j[kWaveItems], start[kWaveItems];
  KeyGroup group[kWaveItems];
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const int32_t k = key[r];
    const bool ok = ((crossers >> r) & 1u) && k >= 0 && uint32_t(k) < bins;
    if constexpr (Grouped) {
      group[r] = key_group(ok, k, lane);
      j[r] = ok && group[r].first == lane ? atomicAdd(s.arrivals + k, group[r].size) : 0u;
    } else {
      j[r] = ok ? atomicAdd(s.arrivals + k, 1u) : 0u;
    }
    start[r] = ok ? s.offsets[k] : 0u;
  }
  wait_loads();
  if constexpr (Grouped) {
#pragma unroll
    for (unsigned r = 0; r < kWaveItems; ++r) {
      const bool ok = ((crossers >> r) & 1u) && key[r] >= 0 && uint32_t(key[r]) < bins;
      j[r] = uint32_t(__shfl(int(j[r]), int(group[r].first))) + group[r].rank;
      const bool below = ok && sub + r * 64 + lane < start[r];
      const KeyGroup lower = key_group(below, key[r], lane);
      if (below && lower.first == lane) atomicAdd(s.lower + key[r], lower.size);
    }
  }
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    if (!((crossers >> r) & 1u)) continue;
    const int32_t k = key[r];
    if (k < 0 || uint32_t(k) >= bins) {
      atomicOr(s.status, 4u);
      continue;
    }
    s.slot[list[r]] = j[r];
    if constexpr (!Grouped)
      if (sub + r * 64 + lane < start[r]) atomicAdd(s.lower + k, 1u);
  }
}

// Per bin: new count (old count less the bin's crossers plus its arrivals)
// and `shift`, the crossers before the old range less the range's start (the
// stayer base less the new offset and the arrivals from lower bins), and the
// tiles' sums of counts and arrivals. Reads the previous plan's offsets,
// before the scan of the new counts replaces them.
__global__ __launch_bounds__(kThreads) void k_cross_counts_new(CrossPlans plans, uint32_t bins) {
  const CrossPlan& s = plans.species[blockIdx.y];
  __shared__ uint32_t lds[kThreads / 64];
  uint32_t count_sum = 0, arrival_sum = 0;
  bool many = false;
#pragma unroll
  for (unsigned r = 0; r < kPlanItems; ++r) {
    const uint32_t b = blockIdx.x * kPlanTile + r * kThreads + threadIdx.x;
    if (b >= bins) continue;
    const uint32_t o = s.offsets[b], e = s.offsets[b + 1];
    const uint32_t lo = crossers_before(s.cross, s.block_base, s.blocks, o);
    const uint32_t hi = crossers_before(s.cross, s.block_base, s.blocks, e);
    const uint32_t arrive = s.arrivals[b], count = (e - o) - (hi - lo) + arrive;
    many |= arrive > kArrivalsMax;
    s.counts[b] = count;
    s.shift[b] = lo - o;
    count_sum += count;
    arrival_sum += arrive;
  }
  if (many) atomicOr(s.status, 1u);
  count_sum = block_sum(count_sum, lds);
  arrival_sum = block_sum(arrival_sum, lds);
  if (threadIdx.x == 0) {
    s.tile_a[blockIdx.x] = count_sum;
    s.tile_b[blockIdx.x] = arrival_sum;
  }
}

// The scans of counts and arrivals, and per bin the stayer base (stayer p of
// the bin lands at base + p - crossers_before(p)). With a consistent old state
// (the new counts add up to the particles) a non-empty halo bin is flagged as
// by the run-based plan.
__global__ __launch_bounds__(kThreads) void k_cross_offsets(CrossPlans plans, Grid g,
                                                            unsigned* __restrict__ validation) {
  const CrossPlan& s = plans.species[blockIdx.y];
  __shared__ uint32_t lds[kThreads / 64];
  const uint32_t bins = g.bins(), tiles = (bins + kPlanTile - 1) / kPlanTile;
  const uint32_t first = blockIdx.x * kPlanTile + threadIdx.x * kPlanItems;
  uint32_t count[kPlanItems], arrive[kPlanItems], base[kPlanItems], count_sum = 0, arrival_sum = 0;
#pragma unroll
  for (unsigned r = 0; r < kPlanItems; ++r) {
    const bool in = first + r < bins;
    count[r] = in ? s.counts[first + r] : 0u;
    arrive[r] = in ? s.arrivals[first + r] : 0u;
    base[r] = in ? s.lower[first + r] + s.shift[first + r] : 0u;
    count_sum += count[r];
    arrival_sum += arrive[r];
  }
  const uint32_t total = tiles_before(s.tile_a, tiles, lds);
  uint32_t at = tiles_before(s.tile_a, blockIdx.x, lds);
  uint32_t arrival_at = tiles_before(s.tile_b, blockIdx.x, lds);
  at += block_exclusive(count_sum, lds);
  arrival_at += block_exclusive(arrival_sum, lds);
  const bool consistent = total == s.n;
  if (blockIdx.x == 0 && threadIdx.x == 0 && !consistent) atomicOr(s.status, 2u);
#pragma unroll
  for (unsigned r = 0; r < kPlanItems; ++r) {
    const uint32_t b = first + r;
    if (b < bins) {
      s.offsets[b] = at;
      s.arrival_offset[b] = arrival_at;
      s.bin_base[b] = at + base[r];
      if (consistent && count[r] != 0) {
        int i, j, k;
        g.decode(int32_t(b), i, j, k);
        if (!g.interior(i, j, k)) atomicOr(validation, kInvalidHalo);
      }
    }
    at += count[r];
    arrival_at += arrive[r];
    if (b + 1 == bins) {
      s.offsets[bins] = at;
      s.arrival_offset[bins] = arrival_at;
    }
  }
}

// Source-ordered pass over tiles of kTile particles: a stayer writes its own
// source entry; a crosser is listed among its new bin's arrivals (at its
// index j within the bin).
__global__ __launch_bounds__(kThreads) void k_cross_sources(CrossPlans plans, uint32_t bins) {
  const CrossPlan& s = plans.species[blockIdx.y];
  const uint32_t n = s.n;
  if (*s.status) return;
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t sub = blockIdx.x * kTile + wave * kWaveSpan;
  if (sub >= n) return;
  // Lane r < kWaveItems holds the crosser word and crossers-before of item r.
  const uint32_t blk0 = sub >> 6;  // sub is a multiple of 64
  const bool item_lane = lane < kWaveItems && sub + lane * 64u < n;
  const uint64_t words = item_lane ? s.cross[blk0 + lane] : 0ull;
  const uint32_t bases = item_lane ? s.block_base[blk0 + lane] : 0u;
  int32_t key[kWaveItems];
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint32_t i = sub + r * 64 + lane;
    key[r] = i < n ? s.keys[i] : -1;
  }
  // Every item's crosser bit and crossers-before first (lane reads only), so
  // the gathers below are issued back to back.
  uint32_t crossers = 0;  // bit r: the lane's particle of item r is a crosser
  uint32_t before[kWaveItems];
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(words)), int(r)));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(words >> 32)), int(r)));
    crossers |= (((lane < 32u ? lo : hi) >> (lane & 31u)) & 1u) << r;
    before[r] = uint32_t(__builtin_amdgcn_readlane(int(bases), int(r))) + bits_below(lo, hi);
  }
  // A crosser's arrival slot (its bin's arrival offset plus its index j), or
  // a stayer's bin base less the crossers before it.
  uint32_t target[kWaveItems];
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const bool valid = key[r] >= 0 && uint32_t(key[r]) < bins;
    const bool crosser = (crossers >> r) & 1u;
    const uint32_t* table = crosser ? s.arrival_offset : s.bin_base;
    const uint32_t base_or_offset = valid ? table[key[r]] : 0u;
    const uint32_t j = (valid && crosser) ? s.slot[before[r]] : 0u;
    target[r] = crosser ? base_or_offset + j : base_or_offset - before[r];
  }
  wait_loads();
#pragma unroll
  for (unsigned r = 0; r < kWaveItems; ++r) {
    const uint32_t i = sub + r * 64 + lane;
    if (key[r] < 0 || uint32_t(key[r]) >= bins) continue;
    if ((crossers >> r) & 1u) {
      s.bin_arrivals[target[r]] = i;
    } else {
      const uint32_t dest = target[r] + i;
      if (dest < n) s.source[dest] = i;
    }
  }
}

// One bin's arrivals: where they lie in bin_arrivals, the bin's first
// destination, those from lower bins and the stayers.
struct Arrivals {
  uint32_t k, at, first, below, stay;
  // Destination of the arrival of rank r in position order: before the stayers
  // those from lower bins, after them the others.
  __device__ __forceinline__ uint32_t destination(uint32_t r) const { return first + r + (r >= below ? stay : 0u); }
};

__device__ __forceinline__ Arrivals bin_arrivals_of(const CrossPlan& s, uint32_t b) {
  Arrivals a;
  a.k = s.arrivals[b];
  a.at = s.arrival_offset[b];
  a.first = s.offsets[b];
  a.below = s.lower[b];
  a.stay = s.counts[b] - a.k;
  return a;
}

// Per bin: the arrivals in position order (rank = arrivals at smaller
// positions; positions are distinct) at their destinations. A thread takes a
// bin of up to kArrivalsInRegisters arrivals; the block's waves share the
// others, a lane per arrival (100 particles a cell with a sixth of them
// crossing: a thread per such bin read them k^2 times, 186 us per species of a
// 512 x 512 plane). The halo bins' records are then copied, as after the
// run-based plan (the fused gather and deposition visits interior cells only).
// A block takes `per_block` bins (at most its threads): fewer where most bins
// have more arrivals than a thread orders.
__global__ __launch_bounds__(kThreads) void k_cross_bins(CrossPlans plans, Grid g, uint32_t per_block) {
  const CrossPlan& s = plans.species[blockIdx.y];
  if (*s.status) return;
  __shared__ uint32_t s_listed, s_list[kThreads];
  const uint32_t n = s.n, end = (blockIdx.x + 1) * per_block;
  const uint32_t bins = end < g.bins() ? end : g.bins();  // of this block and those before it
  const uint32_t b = threadIdx.x < per_block ? blockIdx.x * per_block + threadIdx.x : bins;
  if (threadIdx.x == 0) s_listed = 0;
  __syncthreads();
  if (b < bins) {
    const Arrivals a = bin_arrivals_of(s, b);
    if (a.k > kArrivalsInRegisters) {
      s_list[atomicAdd(&s_listed, 1u)] = b;
    } else if (a.k != 0) {
      uint32_t pos[kArrivalsInRegisters];
#pragma unroll
      for (uint32_t r = 0; r < kArrivalsInRegisters; ++r) pos[r] = r < a.k ? s.bin_arrivals[a.at + r] : 0xffffffffu;
#pragma unroll
      for (uint32_t r = 0; r < kArrivalsInRegisters; ++r) {
        if (r >= a.k) break;
        uint32_t rank = 0;
#pragma unroll
        for (uint32_t q = 0; q < kArrivalsInRegisters; ++q) rank += pos[q] < pos[r] ? 1u : 0u;
        const uint32_t dest = a.destination(rank);
        if (dest < n) s.source[dest] = pos[r];
      }
    }
  }
  __syncthreads();
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t listed = s_listed;
  for (uint32_t l = wave; l < listed; l += kThreads / 64) {
    const Arrivals a = bin_arrivals_of(s, uint32_t(__builtin_amdgcn_readfirstlane(int(s_list[l]))));
    for (uint32_t r0 = 0; r0 < a.k; r0 += 64) {
      const uint32_t pos = r0 + lane < a.k ? s.bin_arrivals[a.at + r0 + lane] : 0xffffffffu;
      uint32_t rank = 0;
      for (uint32_t q0 = 0; q0 < a.k; q0 += 64) {
        const uint32_t other = q0 == r0 ? pos : (q0 + lane < a.k ? s.bin_arrivals[a.at + q0 + lane] : 0xffffffffu);
        const uint32_t m = a.k - q0 < 64u ? a.k - q0 : 64u;
        for (uint32_t t = 0; t < m; ++t)
          rank += uint32_t(__builtin_amdgcn_readlane(int(other), int(t))) < pos ? 1u : 0u;
      }
      const uint32_t dest = a.destination(rank);
      if (r0 + lane < a.k && dest < n) s.source[dest] = pos;
    }
  }
  // The halo bins of this block: their sources are complete now (a listed
  // bin's were written by another wave of the block).
  __threadfence_block();
  __syncthreads();
  if (b >= bins) return;
  const uint32_t count = s.counts[b];
  if (count == 0) return;
  int i, j, k;
  g.decode(int32_t(b), i, j, k);
  if (g.interior(i, j, k)) return;
  for (uint32_t d = s.offsets[b]; d < s.offsets[b] + count; ++d) {
    Record rec;
    load_record(s.src, s.source[d], rec);
    store_record(s.dst, d, rec);
  }
}

}  // namespace

// Device-wide exclusive scan on stream st with the scratch of workspace ws.
static int exclusive_scan(Context& ctx, SortWorkspace& ws, hipStream_t st, const uint32_t* in, uint32_t* out,
                          uint32_t n) {
  if (n == 0) {
    return check_hip(ctx, hipMemsetAsync(out, 0, sizeof(uint32_t), st), "scan");
  }
  const uint32_t blocks = (n + kScanBlock - 1) / kScanBlock;
  if (blocks == 1) {
    k_scan_apply<<<1, kThreads, 0, st>>>(in, n, nullptr, out);
    return check_hip(ctx, hipGetLastError(), "scan");
  }
  // Level scratch: block sums [blocks], their exclusive scan [blocks + 1].
  uint32_t* sums = ws.scan_scratch;
  uint32_t* scanned = sums + blocks;
  if (size_t(2 * blocks + 1) > ws.scan_scratch_words)
    return fail(ctx, -3, "scan scratch too small");
  k_scan_reduce<<<blocks, kThreads, 0, st>>>(in, n, sums);
  // Recurse on the block sums with the remaining scratch.
  {
    uint32_t* saved = ws.scan_scratch;
    const size_t saved_words = ws.scan_scratch_words;
    ws.scan_scratch = scanned + blocks + 1;
    ws.scan_scratch_words = saved_words - (2 * size_t(blocks) + 1);
    const int rc = exclusive_scan(ctx, ws, st, sums, scanned, blocks);
    ws.scan_scratch = saved;
    ws.scan_scratch_words = saved_words;
    if (rc) return rc;
  }
  k_scan_apply<<<blocks, kThreads, 0, st>>>(in, n, scanned, out);
  return check_hip(ctx, hipGetLastError(), "scan");
}

int launch_exclusive_scan(Context& ctx, const uint32_t* in, uint32_t* out, uint32_t n) {
  return exclusive_scan(ctx, ctx.sort, ctx.stream, in, out, n);
}

// Runs, histogram and run destinations of `keys` (stage 1-7 of the sort):
// counts/offsets receive the bin histogram and its scan; returns the tile
// base of the run scan in *tile_base_out.
static int build_runs(Context& ctx, SortWorkspace& ws, hipStream_t st, const int32_t* keys, uint32_t n,
                      uint32_t* counts, uint32_t* offsets, uint32_t** tile_base_out) {
  const Grid& g = ctx.grid;
  const uint32_t bins = g.bins();
  int rc = 0;
#define TPIC_TRY(expr, what)                         \
  do {                                              \
    rc = check_hip(ctx, (expr), what);              \
    if (rc) return rc;                              \
  } while (0)
  TPIC_TRY(hipMemsetAsync(counts, 0, bins * sizeof(uint32_t), st), "sort clear");
  const uint32_t tiles = (n + kTile - 1) / kTile;
  const unsigned grid_stride_blocks = unsigned(ctx.cus > 0 ? ctx.cus * 8 : 2048);
  TPIC_TRY(hipMemsetAsync(ws.failure, 0, sizeof(uint32_t), st), "sort clear");
  TPIC_TRY(hipMemsetAsync(ws.rcounts, 0, bins * sizeof(uint32_t), st), "sort clear");
  TPIC_TRY(hipMemsetAsync(ws.cursor, 0, bins * sizeof(uint32_t), st), "sort clear");
  TPIC_TRY(hipMemsetAsync(ws.large, 0, sizeof(uint32_t), st), "sort clear");
  k_tile_heads<<<tiles, kThreads, 0, st>>>(keys, n, bins, ws.tile_runs, ws.failure);
  TPIC_TRY(hipGetLastError(), "sort heads");
  // tile_runs holds the counts; scan into tile_runs + (tiles + 1).
  uint32_t* tile_base = ws.tile_runs + (ws.tiles + 1);
  if ((rc = exclusive_scan(ctx, ws, st, ws.tile_runs, tile_base, tiles))) return rc;
  k_tile_runs<<<tiles, kThreads, 0, st>>>(keys, n, tiles, tile_base, ws.run_start, ws.run_key, counts, ws.rcounts,
                                          ws.wave_base, ws.failure);
  TPIC_TRY(hipGetLastError(), "sort runs");
  if ((rc = exclusive_scan(ctx, ws, st, counts, offsets, bins))) return rc;
  if ((rc = exclusive_scan(ctx, ws, st, ws.rcounts, ws.roffsets, bins))) return rc;
  k_run_scatter<<<grid_stride_blocks, kThreads, 0, st>>>(tile_base, tiles, ws.run_key, ws.roffsets, ws.cursor,
                                                         ws.bin_runs, ws.failure);
  TPIC_TRY(hipGetLastError(), "sort run scatter");
  k_bin_small<<<(bins + kThreads - 1) / kThreads, kThreads, 0, st>>>(
      g, ws.rcounts, ws.roffsets, offsets, ws.bin_runs, ws.run_start, ws.run_dest, ws.large, ctx.validation,
      ws.failure);
  TPIC_TRY(hipGetLastError(), "sort bins");
  k_bin_large<<<grid_stride_blocks, kThreads, 0, st>>>(ws.large, ws.rcounts, ws.roffsets, offsets, ws.bin_runs,
                                                       ws.run_start, ws.run_dest, ws.failure);
  TPIC_TRY(hipGetLastError(), "sort large bins");
#undef TPIC_TRY
  *tile_base_out = tile_base;
  return 0;
}

static RunPlan sort_run_plan(const SortWorkspace& ws, const uint32_t* counts, const uint32_t* offsets) {
  return RunPlan{counts, offsets, ws.rcounts, ws.roffsets, ws.bin_runs, ws.run_start, ws.run_dest, ws.failure};
}

int launch_sort(Context& ctx, int s) {
  SpeciesState& sp = ctx.species[size_t(s)];
  SortWorkspace& ws = ctx.sort;
  const uint32_t n = sp.count;
  const uint32_t bins = ctx.grid.bins();
  hipStream_t st = ctx.stream;
  phase_begin(ctx, Phase::sort);
  int rc = 0;
  if (n == 0) {
    rc = check_hip(ctx, hipMemsetAsync(sp.counts, 0, bins * sizeof(uint32_t), st), "sort clear");
    if (!rc) rc = check_hip(ctx, hipMemsetAsync(sp.offsets, 0, (bins + 1) * sizeof(uint32_t), st), "sort clear");
    if (rc) return rc;
    sp.sorted = true;
    phase_end(ctx, Phase::sort);
    return 0;
  }
  const ParticleView src = sp.view(), dst = sp.scratch();
  uint32_t* tile_base = nullptr;
  if ((rc = build_runs(ctx, ws, st, src.cell, n, sp.counts, sp.offsets, &tile_base))) return rc;
  (void)tile_base;
  const Grid& g = ctx.grid;
  k_gather_bins<<<(bins + kThreads / 64 - 1) / (kThreads / 64), kThreads, 0, st>>>(g, src, dst, sort_run_plan(ws, sp.counts, sp.offsets),
                                                                                  ws.permutation);
  if ((rc = check_hip(ctx, hipGetLastError(), "sort gather"))) return rc;
  k_copy_on_failure<<<unsigned(ctx.cus > 0 ? ctx.cus * 8 : 2048), kThreads, 0, st>>>(src, dst, n, ws.permutation,
                                                                                     ws.failure, nullptr);
  if ((rc = check_hip(ctx, hipGetLastError(), "sort fallback copy"))) return rc;
  k_sort_failed<<<1, 1, 0, st>>>(ws.failure, ctx.validation);
  if ((rc = check_hip(ctx, hipGetLastError(), "sort status"))) return rc;
  sp.current ^= 1;
  sp.sorted = true;
  phase_end(ctx, Phase::sort);
  return 0;
}

int launch_sort_plan(Context& ctx, int s, SortWorkspace& ws, hipStream_t st) {
  SpeciesState& sp = ctx.species[size_t(s)];
  const uint32_t n = sp.count;
  const uint32_t bins = ctx.grid.bins();
  // Phase times are events on the context stream: a plan on another stream
  // is not timed.
  const bool timed = st == ctx.stream;
  if (timed) phase_begin(ctx, Phase::sort);
  int rc = 0;
  if (n == 0) {
    rc = check_hip(ctx, hipMemsetAsync(sp.counts, 0, bins * sizeof(uint32_t), st), "sort clear");
    if (!rc) rc = check_hip(ctx, hipMemsetAsync(sp.offsets, 0, (bins + 1) * sizeof(uint32_t), st), "sort clear");
    if (rc) return rc;
    if (timed) phase_end(ctx, Phase::sort);
    return 0;
  }
  const ParticleView src = sp.view(), dst = sp.scratch();
  uint32_t* tile_base = nullptr;
  if ((rc = build_runs(ctx, ws, st, src.cell, n, sp.counts, sp.offsets, &tile_base))) return rc;
  const Grid& g = ctx.grid;
  const uint32_t tiles = (n + kTile - 1) / kTile;
  k_tile_sources<<<tiles, kThreads, 0, st>>>(src.cell, n, ws.wave_base, ws.run_start, ws.run_dest, sp.source,
                                             ws.permutation, ws.failure);
  if ((rc = check_hip(ctx, hipGetLastError(), "sort plan"))) return rc;
  k_copy_halo_bins<<<(bins + kThreads - 1) / kThreads, kThreads, 0, st>>>(g, src, dst, sp.counts, sp.offsets,
                                                                          sp.source, ws.failure);
  if ((rc = check_hip(ctx, hipGetLastError(), "sort halo copy"))) return rc;
  k_copy_on_failure<<<unsigned(ctx.cus > 0 ? ctx.cus * 8 : 2048), kThreads, 0, st>>>(src, dst, n, ws.permutation,
                                                                                     ws.failure, sp.source);
  if ((rc = check_hip(ctx, hipGetLastError(), "sort fallback copy"))) return rc;
  k_sort_failed<<<1, 1, 0, st>>>(ws.failure, ctx.validation);
  if ((rc = check_hip(ctx, hipGetLastError(), "sort status"))) return rc;
  if (timed) phase_end(ctx, Phase::sort);
  return 0;
}

int launch_sort_plan_incremental(Context& ctx, int first, int species, SortWorkspace* const* ws, hipStream_t st) {
  const Grid& g = ctx.grid;
  const uint32_t bins = g.bins();
  const bool timed = st == ctx.stream;
  if (timed) phase_begin(ctx, Phase::sort);
  CrossPlans plans{};
  uint32_t blocks = 0, tiles = 0;
  for (int t = 0; t < species; ++t) {
    SpeciesState& sp = ctx.species[size_t(first + t)];
    SortWorkspace& w = *ws[t];
    if (sp.count > w.capacity || !sp.cross || sp.count == 0) return fail(ctx, -3, "plan workspace too small");
    CrossPlan& p = plans.species[t];
    p.src = sp.view();
    p.dst = sp.scratch();
    p.keys = p.src.cell;
    p.cross = sp.cross;
    p.n = sp.count;
    p.blocks = (p.n + 63u) / 64u;
    p.block_base = w.block_base;
    // Arrays of the run-based plan's table.
    p.arrivals = w.rcounts;
    p.arrival_offset = w.roffsets;
    p.slot = w.run_start;
    p.shift = w.large;
    p.bin_arrivals = w.bin_runs;
    p.lower = w.bin_lower;
    p.bin_base = w.bin_base;
    const uint32_t sums = (std::max(p.blocks, bins) + kPlanTile - 1) / kPlanTile;
    if (2 * size_t(sums) > w.scan_scratch_words) return fail(ctx, -3, "scan scratch too small");
    p.tile_a = w.scan_scratch;
    p.tile_b = w.scan_scratch + sums;
    p.counts = sp.counts;
    p.offsets = sp.offsets;
    p.source = sp.source;
    p.status = ctx.plan_status + first + t;
    blocks = std::max(blocks, p.blocks);
    tiles = std::max(tiles, (p.n + kTile - 1) / kTile);
  }
  const unsigned y = unsigned(species);
  const unsigned block_tiles = (blocks + kPlanTile - 1) / kPlanTile, bin_tiles = (bins + kPlanTile - 1) / kPlanTile;
  uint64_t particles = 0;
  for (int t = 0; t < species; ++t) particles = std::max<uint64_t>(particles, plans.species[t].n);
  const bool grouped = particles >= 80ull * g.cells();
  k_cross_begin<<<dim3(std::max(block_tiles, bin_tiles), y), kThreads, 0, st>>>(plans, bins);
  k_cross_bases<<<dim3(block_tiles, y), kThreads, 0, st>>>(plans);
  if (grouped)
    k_cross_arrivals<true><<<dim3(tiles, y), kThreads, 0, st>>>(plans, bins);
  else
    k_cross_arrivals<false><<<dim3(tiles, y), kThreads, 0, st>>>(plans, bins);
  k_cross_counts_new<<<dim3(bin_tiles, y), kThreads, 0, st>>>(plans, bins);
  k_cross_offsets<<<dim3(bin_tiles, y), kThreads, 0, st>>>(plans, g, ctx.validation);
  k_cross_sources<<<dim3(tiles, y), kThreads, 0, st>>>(plans, bins);
  // A species' arrivals a bin grow with its particles a cell (a few percent to
  // a sixth of them): at 1000 a cell nearly every bin is listed, and 256 bins
  // a block leave four waves 64 lists each (479 us for a 1024-cell line).
  const uint32_t per_block = particles >= 256ull * g.cells() ? 4u : (particles >= 80ull * g.cells() ? 64u : kThreads);
  k_cross_bins<<<dim3((bins + per_block - 1) / per_block, y), kThreads, 0, st>>>(plans, g, per_block);
  const int rc = check_hip(ctx, hipGetLastError(), "sort plan from crossers");
  if (timed) phase_end(ctx, Phase::sort);
  return rc;
}

// Words of scan scratch that the plan from the crossers needs (two tile sums).
size_t cross_plan_words(size_t blocks, size_t bins) { return 2 * ((std::max(blocks, bins) + kPlanTile - 1) / kPlanTile); }

int launch_sort_plan(Context& ctx, int s) { return launch_sort_plan(ctx, s, ctx.sort, ctx.stream); }

}  // namespace tpic_mi
