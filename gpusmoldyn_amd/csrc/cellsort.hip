// The step's key sort and cell table as one counting kernel.
//
// A segment is a run of particles whose keys fall in one range of cells: a
// replica (its particles are contiguous), or, for one large system, a bin of
// the keys' high bits after one stable digit pass.  A workgroup owns a slice
// of a segment's cells.  It reads all keys of the segment once, counts those
// of its slice per cell in LDS and collects them, in index order, in an LDS
// list of (cell, index in the segment); the scanned counts are the slice's
// part of the cell table; the list is sorted by cell with two stable digit
// passes inside LDS; then the records are gathered and written in sorted
// order.  The order is that of the stable digit sort by key: every segment's
// particles are read in index order and every pass keeps it.
//
// What bounds it: the record gather and the sorted writes (16 + 16 + 4 bytes
// per particle), the cell table, and latency: each workgroup's phases (keys,
// scan, list, gather) follow one another, so four workgroups of 512 threads
// share a CU (40 KB of LDS, 64 VGPRs).  The ordered path below is kept small
// in registers for that.  The digit sort moved keys and values through memory
// once per digit, counted them in kernels of their own and needed a further
// pass over the keys for the table.  Sort and cell table, us, digit passes
// before / this kernel: one system of 16k particles (2^18 cells) 41 / 8,
// 256 replicas of 2k 39 / 8, 512 replicas of 2k to 64k 225 / 125, 48 of 4k to
// 131k 64 / 27; with the digit pass over the high bits in front, 100k 45 / 20,
// 1M 58 / 37, 4M clustered 138 / 131.  A slice with more particles than its
// list holds, or a cell of more than a few, takes the ordered path, 5 to 10 us
// for each of its windows; what that came to is reported to the host
// (CellSortArgs::work), which turns to the digit passes where they are faster.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "smd_device.h"
#include "smd_kernels.h"

namespace smd {

namespace {

constexpr uint32_t T = kCellThreads;
constexpr uint32_t W = T / 64;                        // waves
constexpr uint32_t kVecs = 2;                         // vectors of four keys per thread per counting round
constexpr uint32_t kVecRound = T * kVecs;
// With at most a workgroup per CU, registers are free and the key reads are a
// chain of latencies: step of one system, us, in rounds / kept: 8k particles
// 26.4 / 25.6, 16k 27.2 / 26.0, 32k 33.9 / 32.4, 48k 40.0 / 38.2.  With more
// workgroups four of them share a CU, which 148 VGPRs would not allow.
constexpr uint32_t kKeepGroups = 256;
constexpr int kKeepVecs = 24;
constexpr uint32_t kRounds = 64;                      // counting rounds that a wave remembers
constexpr int kKeys = 4;                              // keys per thread per round of the ordered path
constexpr uint32_t kRound = T * kKeys;
constexpr int kIndexBits = 32 - kCellSliceBits;       // list entry: cell << kIndexBits | index
constexpr uint32_t kIndexMask = (1u << kIndexBits) - 1u;
constexpr int kLow = 7, kHigh = kCellSliceBits - kLow;  // digits of the ordered path's passes over the list
// About what a slice on the ordered path takes: this for each of its windows
// (with the values to look up in bins), and 1 for each round over the keys.
constexpr uint32_t kWindowHalfUs = 12, kWindowHalfUsBins = 15;
// Cells of at most this many particles are put in order by comparing
// neighbours in the list; a fuller one sends the slice to the ordered path.
constexpr uint32_t kFew = 32;

struct CsLds {
  uint32_t hist[kCellSlice];               // counts per cell, then where each cell's next particle goes
  uint32_t padded[kCellList + 2 * kFew];   // the list, with room for limits before and behind it
  uint16_t cnt[W << kLow];                 // digit counts per wave
  uint32_t wsum[2][W];
  uint32_t red[2][W];
};
static_assert(sizeof(CsLds) <= 40 * 1024, "four workgroups per CU");
static_assert(kRound <= kCellList && kRound < 65536u, "a round fits the list, its ranks fit 16 bits");
static_assert(4u * kRounds * kVecRound <= kIndexMask + 1u, "the remembered rounds' indices fit an entry");
static_assert(kCellKeys + 4u == 4u * kRounds * kVecRound, "one vector more when the first is cut");

// Exclusive prefix of one value per thread over the workgroup; total gets the
// sum.  The caller's next use of wsum must be behind another barrier.
__device__ __forceinline__ uint32_t cs_exscan(uint32_t v, uint32_t* wsum, uint32_t& total) {
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, 64);
    if (lane >= (uint32_t)o) x += y;
  }
  if (lane == 63u) wsum[w] = x;
  __syncthreads();
  uint32_t pre = 0, all = 0;
#pragma unroll
  for (uint32_t q = 0; q < W; ++q) {
    const uint32_t s = wsum[q];
    pre += q < w ? s : 0u;
    all += s;
  }
  total = all;
  return pre + x - v;
}

__device__ __forceinline__ uint32_t cs_sum(uint32_t v, uint32_t* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63u) == 0u) red[threadIdx.x >> 6] = v;
  __syncthreads();
  uint32_t all = 0;
#pragma unroll
  for (int q = 0; q < (int)W; ++q) all += red[q];
  __syncthreads();
  return all;
}

// One stable digit pass over list[0, n): wave w ranks entries
// [w * 64 * items, (w + 1) * 64 * items) in order.
template <int BITS>
__device__ __forceinline__ void cs_digit_pass(CsLds& s, uint32_t n, int shift) {
  constexpr uint32_t RADIX = 1u << BITS;
  constexpr int ITEMS = kKeys;
  constexpr uint32_t PER = (W * RADIX + T - 1) / T;  // counters per thread
  static_assert(W % PER == 0, "a thread's counters belong to one digit");
  uint32_t* const list = s.padded + kFew;
  const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
  const int items = (int)((n + T - 1u) / T);
  for (uint32_t k = t; k < W * RADIX; k += T) s.cnt[k] = 0;
  __syncthreads();
  uint32_t rk[(ITEMS + 1) / 2];  // two 16-bit ranks per word
  const uint32_t base = w * 64u * (uint32_t)items + lane;
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    if (it < items) {
      const uint32_t p = base + 64u * it;
      const bool valid = p < n;
      const uint32_t d = ((valid ? list[p] : 0u) >> shift) & (RADIX - 1u);
      const uint64_t mm = wave_digit_peers<BITS>(d, valid);
      // every lane of the digit writes the same new count
      const uint32_t prev = s.cnt[w * RADIX + d];
      const uint32_t r = prev + lanes_below(mm);
      rk[it / 2] = (it & 1) ? (rk[it / 2] | (r << 16)) : r;
      s.cnt[w * RADIX + d] = (uint16_t)(prev + (uint32_t)__popcll(mm));
    }
  }
  __syncthreads();
  // starts: digit by digit, and wave by wave inside a digit
  {
    const uint32_t k0 = t * PER;
    uint32_t v[PER], sum = 0;
    const uint32_t d = k0 / W, w0 = k0 % W;
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
      v[q] = d < RADIX ? s.cnt[(w0 + q) * RADIX + d] : 0u;
      sum += v[q];
    }
    uint32_t tot;
    uint32_t run = cs_exscan(sum, s.wsum[0], tot);
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
      if (d < RADIX) s.cnt[(w0 + q) * RADIX + d] = (uint16_t)run;
      run += v[q];
    }
  }
  uint32_t e[ITEMS];
#pragma unroll
  for (int it = 0; it < ITEMS; ++it)
    if (it < items && base + 64u * it < n) e[it] = list[base + 64u * it];
  __syncthreads();
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    if (it < items && base + 64u * it < n) {
      const uint32_t d = (e[it] >> shift) & (RADIX - 1u);
      list[s.cnt[w * RADIX + d] + ((it & 1) ? rk[it / 2] >> 16 : rk[it / 2] & 0xFFFFu)] = e[it];
    }
  }
  __syncthreads();
}

}  // namespace

// PART: segments are the bins of a digit pass (a.vals holds the particles'
// indices, a.binTotals the bin sizes); otherwise the replicas.
// KEEP > 0: the keys of a segment of at most KEEP * T vectors stay in registers
// between counting and the list, requested at once; a larger segment reads them
// again, in rounds.
template <bool PART, int KEEP>
__global__ __launch_bounds__(T, KEEP ? 2 : 8) void k_cell_sort(CellSortArgs a, const ReplicaTables* __restrict__ tables,
                                                    const uint32_t* __restrict__ keys,
                                                    const float4* __restrict__ src) {
  __shared__ CsLds s;
  uint32_t* const list = s.padded + kFew;
  const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
  // this workgroup's segment (seg: replica or bin) and slice
  uint32_t seg, n, cellBase, cells, slice, room;
  if (PART) {
    // workgroups are dealt round robin over the 8 XCDs: each gets a run of
    // neighbouring bins, whose keys and records its L2 then shares
    const uint32_t b = blockIdx.x, q8 = gridDim.x >> 3, r8 = gridDim.x & 7u;
    const uint32_t wg = (b & 7u) * q8 + min(b & 7u, r8) + (b >> 3);
    seg = wg / a.slicesPerBin;
    slice = wg % a.slicesPerBin;
    room = a.slicesPerBin;
    n = a.binTotals[seg];
    cellBase = seg << a.binBits;
    cells = min(1u << a.binBits, a.deadKey - cellBase);
  } else {
    const uint32_t g = a.groups[blockIdx.x];
    if (g == kCellNoGroup) return;
    seg = g >> kCellGroupShift;
    slice = g & ((1u << kCellGroupShift) - 1u);
    room = a.groupSlices[seg];
    n = a.segCount[seg];
    cellBase = a.bucketOff[seg];
    cells = tables[seg].numBuckets;
  }
  // As many slices as the list needs with a tenth to spare, at least
  // minSlices (small systems spread over the CUs).
  uint32_t slices = max((cells + kCellSlice - 1u) / kCellSlice, (n + kCellFill - 1u) / kCellFill);
  slices = min(max(slices, min(a.minSlices, (cells + 63u) / 64u)), room);
  const uint32_t width = (cells + slices - 1u) / slices;
  const uint32_t c0 = slice * width;
  const bool works = slice < slices && c0 < cells;
  if (!works && blockIdx.x != 0u) return;
  const uint32_t nAll = min(*a.dN, a.maxN);
  uint32_t off, before = 0;  // the segment's first key; live particles of earlier segments
  if (PART) {
    uint32_t lower = 0;
    for (uint32_t q = t; q < seg; q += T) lower += a.binTotals[q];
    before = off = cs_sum(lower, s.red[0]);
  } else {
    off = a.segOff[seg];
    if (a.R > 1) {
      uint32_t lower = 0;
      for (uint32_t q = t; q < seg; q += T) lower += a.segCount[q] - a.segDead[q];
      before = cs_sum(lower, s.red[0]);
    }
  }
  off = min(off, nAll);
  n = min(n, nAll - off);
  if (blockIdx.x == 0) {
    // the live count and the two table entries past the last cell
    uint32_t dead = 0;
    for (uint32_t q = t; q < (uint32_t)a.R; q += T) dead += a.segDead[q];
    dead = cs_sum(dead, s.red[1]);
    if (t == 0) {
      *a.dLive = nAll - dead;
      a.first[a.deadKey] = nAll - dead;
      a.first[a.deadKey + 1u] = nAll;
    }
    if (!works) return;
  }
  const uint32_t nc = min(width, cells - c0);
  const uint32_t key0 = cellBase + c0;

  for (uint32_t c = t * 4u; c < nc; c += 4u * T) *(uint4*)&s.hist[c] = make_uint4(0u, 0u, 0u, 0u);
  __syncthreads();

  // Keys of the segment in rounds: thread order is index order (wave w, then
  // its kKeys chunks of 64).
  auto load = [&](uint32_t t0, uint32_t (&kk)[kKeys]) __attribute__((always_inline)) {
    const uint32_t e0 = t0 + w * (64u * kKeys) + lane;
#pragma unroll
    for (int q = 0; q < kKeys; ++q) kk[q] = e0 + 64u * q < n ? keys[off + e0 + 64u * q] : 0xFFFFFFFFu;
  };
  // Counting reads the keys as aligned vectors of four, in any order, with no
  // barrier between rounds; vectors without a key of the slice (most of them
  // when the particles are stored near cell order) cost a few compares.
  const uint4* __restrict__ const keys4 = (const uint4*)keys;
  const uint32_t v0 = off >> 2, v1 = (off + n + 3u) >> 2;
  const uint32_t rounds = n ? (v1 - v0 + kVecRound - 1u) / kVecRound : 0u;
  auto loadv = [&](uint32_t r, uint32_t (&kk)[4 * kVecs]) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t q = 0; q < kVecs; ++q) {
      const uint32_t v = v0 + r * kVecRound + q * T + t;
      const uint4 x = v < v1 ? keys4[v] : make_uint4(~0u, ~0u, ~0u, ~0u);
      kk[4 * q] = x.x, kk[4 * q + 1] = x.y, kk[4 * q + 2] = x.z, kk[4 * q + 3] = x.w;
    }
    if (r == 0u || r + 1u == rounds) {  // keys of the neighbouring segments in the end vectors
#pragma unroll
      for (uint32_t q = 0; q < 4 * kVecs; ++q) {
        const uint32_t e = 4u * (v0 + r * kVecRound + q / 4 * T + t) + q % 4;
        if (e - off >= n) kk[q] = ~0u;
      }
    }
  };
  uint32_t below = 0, kk[4 * kVecs];
  uint64_t mine = 0;  // rounds in which this wave met keys of the slice
  uint4 kept[KEEP ? KEEP : 1];
  auto count = [&](uint32_t key) __attribute__((always_inline)) {
    const uint32_t c = key - key0;
    below += key < key0 ? 1u : 0u;
    if (c < nc) atomicAdd(&s.hist[c], 1u);
  };
  // the segment's keys fit the registers of the workgroup
  const bool keeps = KEEP > 0 && v1 - v0 <= (uint32_t)KEEP * T;
  if (keeps) {
#pragma unroll
    for (uint32_t q = 0; q < KEEP; ++q) {
      const uint32_t v = v0 + q * T + t;
      kept[q] = v < v1 ? keys4[v] : make_uint4(~0u, ~0u, ~0u, ~0u);
    }
#pragma unroll
    for (uint32_t q = 0; q < KEEP; ++q) {
      if (v0 + q * T >= v1) break;
      const uint32_t v = v0 + q * T + t, e = 4u * v - off;
      if (v == v0 || v + 1u == v1) {  // keys of the neighbouring segments in the end vectors
        if (e >= n) kept[q].x = ~0u;
        if (e + 1u >= n) kept[q].y = ~0u;
        if (e + 2u >= n) kept[q].z = ~0u;
        if (e + 3u >= n) kept[q].w = ~0u;
      }
      count(kept[q].x);
      count(kept[q].y);
      count(kept[q].z);
      count(kept[q].w);
    }
  } else {
    loadv(0u, kk);
    for (uint32_t r = 0; r < rounds; ++r) {
      // the next round's keys are requested before this round's are counted
      uint32_t kn[4 * kVecs];
      if (r + 1u < rounds) loadv(r + 1u, kn);
      uint64_t any = 0;
#pragma unroll
      for (uint32_t q = 0; q < 4 * kVecs; ++q) {
        any |= __ballot(kk[q] - key0 < nc);
        count(kk[q]);
      }
      if (any != 0 && r < kRounds) mine |= 1ull << r;
      if (r + 1u == rounds) break;  // kk keeps the last round's keys
#pragma unroll
      for (uint32_t q = 0; q < 4 * kVecs; ++q) kk[q] = kn[q];
    }
  }
  below = wave_sum(below);
  if (lane == 0u) s.red[0][w] = below;
  __syncthreads();
  // sorted position of the slice's first particle
  uint32_t start = before;
  if (slice) {
#pragma unroll
    for (uint32_t q = 0; q < W; ++q) start += s.red[0][q];
  }
  // where each cell starts
  uint32_t have, most = 0;
  {
    constexpr uint32_t PER = kCellSlice / T;
    static_assert(PER % 4 == 0, "vector accesses");
    const uint32_t c = t * PER;
    uint32_t v[PER], sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < PER; q += 4) {
      const uint4 x = c + q < nc ? *(const uint4*)&s.hist[c + q] : make_uint4(0u, 0u, 0u, 0u);
      v[q] = x.x, v[q + 1] = x.y, v[q + 2] = x.z, v[q + 3] = x.w;
    }
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
      sum += v[q];
      most = max(most, v[q]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, 64));
    if (lane == 0u) s.red[1][w] = most;
    uint32_t run = cs_exscan(sum, s.wsum[0], have);
#pragma unroll
    for (uint32_t q = 0; q < W; ++q) most = max(most, s.red[1][q]);
#pragma unroll
    for (uint32_t q = 0; q < PER; q += 4) {
      uint4 x;
      x.x = run, run += v[q];
      x.y = run, run += v[q + 1];
      x.z = run, run += v[q + 2];
      x.w = run, run += v[q + 3];
      if (c + q < nc) *(uint4*)&s.hist[c + q] = x;
    }
  }
  most = __builtin_amdgcn_readfirstlane(most);
  have = __builtin_amdgcn_readfirstlane(have);
  __syncthreads();
  // the slice's part of the cell table
  for (uint32_t q = t; q < nc; q += T) a.first[key0 + q] = start + s.hist[q];

  // Writes the record of list entry `ent` to its place in sorted order.
  bool bad = false;
  auto store = [&](uint32_t ent, uint32_t idx, float4 rec, uint32_t dst) __attribute__((always_inline)) {
    if (dst >= nAll) {
      bad = true;
      return;
    }
    a.keysOut[dst] = key0 + (ent >> kIndexBits);
    if (a.packIndex) {
      rec.w = __int_as_float(pack_index_type(idx, __float_as_int(rec.w) & kTypeMask));
    } else {
      a.valsOut[dst] = idx;
    }
    a.dst[dst] = rec;
  };

  if (have <= kCellList && rounds <= kRounds && most <= kFew) {
    // Into the list by cell through the cells' cursors, in any order within
    // a cell; each entry then counts the neighbours on its wrong side.
    // Entries compare as (cell, index), so neighbours of other cells never
    // count, and an entry is at most most - 1 places off.
    __syncthreads();  // the table was read from the cursors
    if (t < kFew) {
      s.padded[t] = 0u;
      list[have + t] = 0xFFFFFFFFu;
    }
    if (keeps) {
      auto place = [&](uint32_t key, uint32_t idx) __attribute__((always_inline)) {
        const uint32_t c = key - key0;
        if (c < nc) list[atomicAdd(&s.hist[c], 1u)] = (c << kIndexBits) | idx;
      };
#pragma unroll
      for (uint32_t q = 0; q < KEEP; ++q) {
        if (v0 + q * T >= v1) break;
        const uint32_t e = 4u * (v0 + q * T + t) - off;
        place(kept[q].x, e);
        place(kept[q].y, e + 1u);
        place(kept[q].z, e + 2u);
        place(kept[q].w, e + 3u);
      }
    } else {
      bool ready = false;  // kk holds the round's keys (the last round's are still there)
      while (mine) {
        const uint32_t r = 63u - (uint32_t)__clzll((long long)mine);
        mine &= ~(1ull << r);
        uint32_t kn[4 * kVecs];
        if (r + 1u != rounds && !ready) loadv(r, kk);
        if (mine) loadv(63u - (uint32_t)__clzll((long long)mine), kn);
#pragma unroll
        for (uint32_t q = 0; q < 4 * kVecs; ++q) {
          const uint32_t c = kk[q] - key0;
          if (c < nc)
            list[atomicAdd(&s.hist[c], 1u)] =
                (c << kIndexBits) |
                (4u * (v0 + r * kVecRound + q / 4 * T + t) + q % 4 - off);
        }
#pragma unroll
        for (uint32_t q = 0; q < 4 * kVecs; ++q) kk[q] = kn[q];
        ready = true;
      }
    }
    __syncthreads();
    for (uint32_t p0 = t; p0 < have; p0 += 4u * T) {
      uint32_t ent[4], dst[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t p = min(p0 + (uint32_t)q * T, have - 1u);
        ent[q] = list[p];
        dst[q] = start + p;
      }
      for (uint32_t d = 1; d < most; ++d) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t* at = list + min(p0 + (uint32_t)q * T, have - 1u);
          dst[q] += at[d] < ent[q] ? 1u : 0u;
          dst[q] -= *(at - d) > ent[q] ? 1u : 0u;
        }
      }
      uint32_t idx[4];
      float4 rec[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        idx[q] = off + (ent[q] & kIndexMask);
        if (PART) idx[q] = a.vals[idx[q]];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) rec[q] = src[idx[q]];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (p0 + (uint32_t)q * T < have) store(ent[q], idx[q], rec[q], dst[q]);
    }
  } else {
    // Windows of the segment whose keys fit the list, collected in index
    // order and put in cell order by stable digit passes.
    uint32_t t0 = 0, windows = 0;
    for (;;) {
      ++windows;
      const uint32_t winBase = t0;
      uint32_t par = 0;
      have = 0;
      __syncthreads();
      while (t0 < n && t0 + kRound - winBase <= kIndexMask + 1u) {
        uint32_t kk[kKeys];
        load(t0, kk);
        uint32_t in = 0;
#pragma unroll
        for (int q = 0; q < kKeys; ++q) in += (uint32_t)__popcll(__ballot(kk[q] - key0 < nc));
        if (lane == 0u) s.wsum[par][w] = in;
        __syncthreads();
        uint32_t at = have, all = 0;
#pragma unroll
        for (uint32_t q = 0; q < W; ++q) {
          const uint32_t x = s.wsum[par][q];
          at += q < w ? x : 0u;
          all += x;
        }
        par ^= 1u;
        if (have + all > kRound) break;
#pragma unroll
        for (int q = 0; q < kKeys; ++q) {
          const uint32_t c = kk[q] - key0;
          const uint64_t m = __ballot(c < nc);
          if (c < nc)
            list[at + lanes_below(m)] =
                (c << kIndexBits) | (t0 - winBase + w * (64u * kKeys) + 64u * q + lane);
          at += (uint32_t)__popcll(m);
        }
        have += all;
        t0 += kRound;
      }
      __syncthreads();
      cs_digit_pass<kLow>(s, have, kIndexBits);
      if (nc > (1u << kLow)) cs_digit_pass<kHigh>(s, have, kIndexBits + kLow);
      // a cell's particles of this window are the list entries [b, e): its
      // cursor becomes (next place) - b for the write, then moves on by e - b
      for (uint32_t p = t; p < have; p += T) {
        const uint32_t c = list[p] >> kIndexBits;
        if (p == 0u || (list[p - 1u] >> kIndexBits) != c) s.hist[c] -= p;
      }
      __syncthreads();
      for (uint32_t p = t; p < have; p += T) {
        const uint32_t c = list[p] >> kIndexBits;
        uint32_t idx = off + winBase + (list[p] & kIndexMask);
        if (PART) idx = a.vals[idx];
        store(list[p], idx, src[idx], start + p + s.hist[c]);
      }
      if (t0 >= n) break;
      __syncthreads();
      for (uint32_t p = t; p < have; p += T) {
        const uint32_t c = list[p] >> kIndexBits;
        if (p + 1u == have || (list[p + 1u] >> kIndexBits) != c) s.hist[c] += p + 1u;
      }
    }
    if (t == 0u) {
      const uint32_t r = (n + kRound - 1u) / kRound;
      atomicMax(&a.work[0], windows * (PART ? kWindowHalfUsBins : kWindowHalfUs) + r);
      atomicAdd(&a.work[1], r);
    }
  }
  if (bad) atomicOr(a.status, kStatusSortLayout);
}

// The removed particles' keys and indices behind the live ones, in index
// order (read by the stage hooks only).  One workgroup.
__global__ __launch_bounds__(T) void k_cell_sort_removed(const uint32_t* __restrict__ keys,
                                                                  const uint32_t* __restrict__ vals,
                                                                  const uint32_t* __restrict__ dN, uint32_t maxN,
                                                                  uint32_t deadKey, const uint32_t* __restrict__ dLive,
                                                                  uint32_t* __restrict__ keysOut,
                                                                  uint32_t* __restrict__ valsOut) {
  __shared__ uint32_t wsum[W];
  const uint32_t n = min(*dN, maxN);
  uint32_t at = *dLive;
  for (uint32_t t0 = 0; t0 < n; t0 += T) {
    const uint32_t e = t0 + threadIdx.x;
    const bool dead = e < n && keys[e] == deadKey;
    uint32_t tot;
    const uint32_t dst = at + cs_exscan(dead ? 1u : 0u, wsum, tot);
    if (dead && dst < n) {
      keysOut[dst] = deadKey;
      valsOut[dst] = vals ? vals[e] : e;
    }
    at += tot;
    __syncthreads();
  }
}

hipError_t launch_cell_sort(const CellSortArgs& a, bool part, uint32_t workgroups, hipStream_t stream) {
  if (workgroups == 0) return hipSuccess;
  const dim3 grid(workgroups), blk(T);
  if (part) hipLaunchKernelGGL((k_cell_sort<true, 0>), grid, blk, 0, stream, a, a.tables, a.keys, a.src);
  else if (workgroups <= kKeepGroups)
    hipLaunchKernelGGL((k_cell_sort<false, kKeepVecs>), grid, blk, 0, stream, a, a.tables, a.keys, a.src);
  else hipLaunchKernelGGL((k_cell_sort<false, 0>), grid, blk, 0, stream, a, a.tables, a.keys, a.src);
  return hipGetLastError();
}

hipError_t launch_cell_sort_removed(const uint32_t* keys, const uint32_t* vals, const uint32_t* dN, uint32_t maxN,
                                    uint32_t deadKey, const uint32_t* dLive, uint32_t* keysOut, uint32_t* valsOut,
                                    hipStream_t stream) {
  hipLaunchKernelGGL(k_cell_sort_removed, dim3(1), dim3(T), 0, stream, keys, vals, dN, maxN, deadKey, dLive,
                     keysOut, valsOut);
  return hipGetLastError();
}

}  // namespace smd
