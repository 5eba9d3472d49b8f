// Kernel argument blocks and launch wrappers (host-visible).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "smd_types.h"

namespace smd {

// Tile table of the segmented sort (k_seg_tiles): tiles of tileSize keys
// inside each replica's segment, laid out from the per-replica counts.
struct SegTilesArgs {
  const uint32_t* segOff;
  const uint32_t* segCount;
  int R;
  uint32_t tileSize;
  uint32_t maxTiles;
  uint2* tpos;
  uint32_t* tseg;
  uint32_t* nTiles;
  uint32_t* segFirst;
  uint32_t* nLong;
  uint32_t* repDead;
  const uint32_t* dN;
  uint32_t* status;
};

// Where the particles that enter a step are.  The step that wrote them left
// removed ones in place: replica r's survivors are the slots from srcOff[r]
// on, in order, except the holes [holeOff[r], holeOff[r] + holeN[r]) of the
// sorted hole list; behind its alive[r] survivors come the particles it
// gained, at extraBase + extraOff[r] of the same array.
struct CanonMap {
  const uint32_t* srcOff;
  const uint32_t* alive;
  const uint32_t* holeOff;
  const uint32_t* holeN;
  const uint32_t* holes;
  const uint32_t* extraOff;
  uint32_t extraBase;
};

// Particles removed in a step: a bit per slot and a count per tile.
struct DeathMarks {
  uint32_t* bits;
  uint32_t* tileDead;
};

struct ProducerArgs {
  const ReplicaTables* tables;
  const int* streamReplica;   // per global stream: replica id (padding lanes of a replica included), -1 none
  const uint32_t* repOff;     // per replica: first particle
  const uint32_t* repCount;   // per replica: particle count
  uint32_t* mtState;          // [20][Stot]
  const uint32_t* mtPar;      // [3][Stot]
  uint32_t Stot;
  const float* gauss;         // entries 1 to 2048 of the 4096-entry table (gauss_entry)
  const float4* ptIn;         // canonical records entering the step, through map
  CanonMap map;
  float4* pt;                 // canonical records of the step, dense; also the pair-search source
  const float* wIn;           // fourth position components, as ptIn and pt (nullptr: in the records)
  float* w;
  float4* addedPos;
  int* birthType;
  uint32_t* key;
  uint32_t deadKey;
  uint32_t* repDeaths;
  uint32_t* repBirths;
  DeathMarks deaths;
  uint32_t* tileBirth;
  const uint32_t* retire;     // per replica: remove every particle this step (nullptr: none)
  // 1: one extra workgroup of the launch lays out the segmented sort's tiles
  // (it reads only the per-replica counts the step starts with)
  int segTilesOn = 0;
  SegTilesArgs segTiles;
};

struct SortBuffers {
  uint32_t* keys;
  uint32_t* vals;
  uint32_t* keysAlt;
  uint32_t* valsAlt;
  uint32_t* counts;  // sort_counts_words(maxN, radixBits)
  uint32_t* status;  // sticky status word (kStatusSortSpin), or nullptr
  int algo;          // 0: single sweep with look-back, 1: count / scan / scatter per digit
  // optional gather into sorted order: gatherDst[j] = gatherSrc[vals[j]] for
  // keys[j] < gatherDeadKey (fused into the last digit pass when possible)
  const float4* gatherSrc;
  float4* gatherDst;
  uint32_t gatherDeadKey;
  uint32_t sizeHint;  // expected key count (tile size choice only), 0: maxN
  // with the gather fused into the last pass (algo 1): 1 puts each particle's
  // index into its sorted record (w = index << kIndexShift | type, indices
  // below kMaxPackedIndex) instead of writing the sorted values
  int packIndex;
};

// Segments of an ensemble's replica-major keys for the segmented sort:
// segment r is [segOff[r], segOff[r] + segCount[r]), its keys are
// bucketOff[r] + (a local cell below 2^(2 bits - 1)) or deadKey.
struct SegSortArgs {
  int R;
  const uint32_t* segOff;
  const uint32_t* segCount;
  const uint32_t* bucketOff;
  uint32_t deadKey;
  int lowBits;         // first-pass digit width (7 to 10 bits)
  int highBits;        // second-pass digit width (7 to 10 bits)
  uint32_t* scratch;   // seg_sort_words(maxN, R, max(lowBits, highBits)) words
  int tilesLaid = 0;   // 1: the tile table is already laid out (seg_tiles_args, by the producer launch)
};

// Digit widths of the segmented sort for replica grids of at most 2^maxGridBits
// buckets: {low, high} with low + high > maxGridBits, or {0, 0} when two
// passes of at most 9 bits cannot cover them (the engine then sorts global
// keys).
void seg_sort_digits(uint32_t maxGridBits, int& lowBits, int& highBits);

// The counting cell sort (k_cell_sort): slices of at most kCellSlice cells,
// aiming at kCellFill particles, whose list holds kCellList.
constexpr int kCellThreads = 512;
constexpr int kCellSliceBits = 12;
constexpr uint32_t kCellSlice = 1u << kCellSliceBits;
constexpr uint32_t kCellList = 5376;
constexpr uint32_t kCellFill = 4838;
// Keys of a segment, at any alignment, whose rounds a slice remembers; a larger
// one takes the ordered path.
constexpr uint32_t kCellKeys = (1u << 18) - 4u;
constexpr int kCellGroupShift = 12;  // workgroup table: replica << kCellGroupShift | slice
constexpr uint32_t kCellNoGroup = 0xFFFFFFFFu;  // an entry without work

struct CellSortArgs {
  const ReplicaTables* tables;
  const uint32_t* keys;        // in canonical order, or binned (then vals holds the indices)
  const uint32_t* vals;
  const float4* src;           // canonical records
  const uint32_t* dN;
  uint32_t maxN;
  int R;
  const uint32_t* segOff;      // per replica: first particle, particles, removed particles
  const uint32_t* segCount;
  const uint32_t* segDead;
  const uint32_t* bucketOff;
  // by replica: the slice of each workgroup, and the slices each replica has
  // workgroups for (at least ceil(cells / kCellSlice))
  const uint32_t* groups;
  const uint32_t* groupSlices;
  uint32_t minSlices;          // slices per segment for small systems
  // by bins of the keys' high bits: 2^binBits cells each
  uint32_t binBits, slicesPerBin;
  const uint32_t* binTotals;   // keys per bin
  uint32_t deadKey;
  uint32_t* dLive;
  uint32_t* first;             // first_words(deadKey + 1) words
  uint32_t* keysOut;
  uint32_t* valsOut;           // written unless packIndex
  float4* dst;                 // records in sorted order
  int packIndex;
  uint32_t* status;
  // what the slices cost that did not fit their lists (SortWork): the most
  // expensive one, in half microseconds, and the rounds of all
  uint32_t* work;
};

// Pair candidates of a step: cand[j] = (partner, step tag) for the sorted
// particles that have one; entries whose tag is not *stepCount + 1 are of
// earlier steps.  The list holds, in any order, the possible pairs by their
// lower index: (j, its candidate c > j, stream that j draws from, replica).
struct CandList {
  uint2* cand;
  uint4* list;
  // entries of the list; the finalize kernel sets it to 0 for the next step,
  // or past pair_list_size() where the step had too many pairs for a list:
  // then none is kept
  uint32_t* count;
  uint32_t* acting;  // reacting pairs found without a list; reset likewise
  const uint32_t* stepCount;
};

struct CandArgs {
  const ReplicaTables* tables;
  const uint32_t* bucketStart;  // per replica bucketOff, [R] = deadKey
  const int* bucketRep;         // replica of bucket chunk key >> repShift (nullptr: search bucketStart)
  uint32_t repShift;
  int R;
  const uint32_t* keys;         // sorted
  const float4* sortedPT;
  const uint32_t* first;
  const uint32_t* dLive;
  CandList cand;
};

struct ResolveArgs {
  const ReplicaTables* tables;
  const int* streamReplica;
  uint32_t* mtState;
  const uint32_t* mtPar;
  uint32_t Stot;
  const uint32_t* first;
  CandList cand;
  const float4* sortedPT;
  const uint32_t* vals;
  int packed;  // sortedPT carries the particles' indices (vals unused)
  float4* pt;
  float* w;  // nullptr: in the records
  uint32_t* repDeaths;
  DeathMarks deaths;
};

struct FinalizeArgs {
  int R;
  const uint32_t* repCount;
  uint32_t* repDeaths;
  uint32_t* repBirths;
  uint32_t* newOff;     // [R+1]
  uint32_t* newCount;
  // the map of the next step (CanonMap) and where the gained particles go
  uint32_t* alive;
  uint32_t* holeOff;
  uint32_t* holeN;
  uint32_t* holes;
  uint32_t* extraOff;
  uint32_t* birthBase;  // births of earlier replicas
  uint32_t* dNnext;
  const uint32_t* dN;
  DeathMarks deaths;    // the bits are cleared here
  uint32_t* tileDeadNext;  // the other step parity's counts: cleared here
  uint32_t* tileBirth;     // nullptr: no particle can be born
  uint32_t* tileBirthPre;
  // CandList::count and acting, then CellSortArgs::work (nullptr: no pairs)
  uint4* pairCounts;
  unsigned long long* hostSort;  // host-visible: step << 32 | most << 16 | rounds / 64 of the last step with such slices
  unsigned long long* particleSteps;  // += particles entering the step
  uint32_t* stepCount;                // steps completed (incremented here)
  unsigned long long* countRing;      // host-visible: slot (steps & ringMask) = steps << 32 | particles
  uint32_t ringMask;
  const uint32_t* status;  // sticky error bits, and their host-visible copy
  uint32_t* hostStatus;
  const uint32_t* zCount;  // per replica: particles created this step (nullptr: none)
  uint32_t* zeroBase;      // per replica: where its created particles go (from extraBase)
  uint32_t* injCount;      // per replica: particles admitted this step (nullptr: none); reset
  uint32_t* injBase;       // per replica: where its admitted particles go (from extraBase)
  uint32_t* retire;        // per replica retire flags (nullptr: none); reset
  uint32_t* blockSum;      // births of each workgroup's tiles
  uint32_t blockTiles;     // tiles per workgroup (finalize_block_tiles)
  uint32_t tilesCap;       // tiles of the allocated capacity
};

struct ZeroArgs {
  const ReplicaTables* tables;
  int R;
  uint32_t* zMt;         // [20][R] one creation stream per replica
  const uint32_t* zPar;  // [3][R]
  float4* zPos;          // creation buffer (replica r at tables[r].zeroOff)
  int* zType;
  uint32_t* zCount;      // per replica: particles created this step
  uint32_t* status;      // sticky error bits (kStatusZeroOverflow)
};

struct InjectArgs {
  const float4* injPos;
  const int* injType;
  const int* injRep;          // replica of each admitted particle
  const uint32_t* injSrcOff;  // first admitted particle of each replica
  uint32_t nInj;
  const uint32_t* injBase;
  float4* extra;   // gained particles' records and fourth components (nullptr: in the records)
  float* extraW;
};

// Births of a step, in parent order behind their replica's survivors.
struct BirthArgs {
  int R;
  const uint32_t* dN;
  const uint32_t* repOff;
  const uint32_t* birthBase;
  const uint32_t* extraOff;
  const uint32_t* tileBirthPre;
  const float4* addedPos;
  int* birthType;          // nonzero only at births; cleared as they are taken
  uint32_t* tileBirth;     // births per tile (producer); cleared here
  const uint32_t* blockSum;
  uint32_t blockTiles;
  float4* extra;
  float* extraW;           // nullptr: in the records
};

// Reads replica rep's canonical particles (all replicas, as one array, when
// rep < 0) through the map into pos4 / types (either may be nullptr, both may
// be host memory); header gets the particle count.
struct ExportArgs {
  const float4* pt;
  const float* w;  // nullptr: in the records
  CanonMap map;
  const uint32_t* repOff;    // [R+1]
  const uint32_t* repCount;
  int R, rep;
  uint32_t cap;              // the first cap particles
  float4* pos4;
  int* types;
  uint32_t* header;          // nullptr: none
};

hipError_t launch_mt_init(uint32_t* st, const uint32_t* seeds, uint32_t S, hipStream_t stream);
hipError_t launch_mt_fill(uint32_t* st, const uint32_t* par, uint32_t S, uint32_t nStreams, int count, int batch3,
                          uint32_t* out, hipStream_t stream);
// blockSize: 128, 256 or 512 threads (identical results)
hipError_t launch_producer(const ProducerArgs& a, int blockSize, hipStream_t stream);
int sort_passes(uint32_t keyBits, int radixBits);
size_t sort_counts_words(uint32_t maxN, int radixBits);
hipError_t launch_sort(SortBuffers& b, const uint32_t* dN, uint32_t maxN, uint32_t keyBits, int radixBits,
                       bool identityVals, hipStream_t stream);
// One stable 8-bit digit pass (count / scan / scatter) on the key bits from
// `shift` (keys past the last digit go into the last bin), values = indices; totals gets the address of the 256 digit counts.
// Swaps the buffers.
hipError_t launch_sort_bins(SortBuffers& b, const uint32_t* dN, uint32_t maxN, int shift, const uint32_t** totals,
                            hipStream_t stream);
// Sorted keys (live ones), records and cell table in one kernel; part: by
// bins of launch_sort_bins.
hipError_t launch_cell_sort(const CellSortArgs& a, bool part, uint32_t workgroups, hipStream_t stream);
// The removed keys and values behind the live ones, in index order (vals
// nullptr: keys are in canonical order).
hipError_t launch_cell_sort_removed(const uint32_t* keys, const uint32_t* vals, const uint32_t* dN, uint32_t maxN,
                                    uint32_t deadKey, const uint32_t* dLive, uint32_t* keysOut, uint32_t* valsOut,
                                    hipStream_t stream);
// Segmented two-pass sort of an ensemble's keys (same output as launch_sort
// with identityVals over all keys: live keys in order, removed ones after
// them in index order).
size_t seg_sort_words(uint32_t maxN, int R, int maxBits);
hipError_t launch_sort_seg(SortBuffers& b, const SegSortArgs& g, const uint32_t* dN, uint32_t maxN,
                           bool identityVals, hipStream_t stream);
// The tile-table arguments of a segmented sort of at most maxN keys (the
// addresses inside g.scratch that launch_sort_seg uses).
SegTilesArgs seg_tiles_args(const SegSortArgs& g, const uint32_t* dN, uint32_t maxN, uint32_t* status);
// Counter words the count / scan / scatter sort (SortBuffers::algo = 1)
// uses for maxN keys: per-tile digit counts and the digit totals.
size_t sort3k_counts_words(uint32_t maxN, uint32_t sizeHint, int radixBits);
// first: first_words(nb) words (first[0..nb]).  slotBits > 0 (slot engines,
// slots of 2^slotBits buckets): entries of slot s past offset
// tables[s].numBuckets are not written.
size_t first_words(uint32_t nb);
hipError_t launch_first(const uint32_t* keys, const uint32_t* dN, uint32_t maxN, uint32_t nb, uint32_t* first,
                        uint32_t* dLive, const ReplicaTables* tables, uint32_t slotBits, uint32_t nSlots,
                        hipStream_t stream);
hipError_t launch_gather(const uint32_t* keys, const uint32_t* vals, const float4* src, const uint32_t* dN,
                         uint32_t maxN, uint32_t deadKey, float4* sortedPT, hipStream_t stream);
// blockSize: 64, 128 or 256 threads (identical results)
hipError_t launch_candidates(const CandArgs& a, uint32_t maxN, int blockSize, hipStream_t stream);
// Entries of CandList::list.
size_t pair_list_size();
hipError_t launch_resolve(const ResolveArgs& a, hipStream_t stream);
// Tiles per finalize workgroup when there are `tiles` of them.
uint32_t finalize_block_tiles(uint32_t tiles);
hipError_t launch_finalize(const FinalizeArgs& a, hipStream_t stream);
hipError_t launch_births(const BirthArgs& a, uint32_t maxN, hipStream_t stream);
hipError_t launch_export(const ExportArgs& a, uint32_t maxN, hipStream_t stream);
// Dense copy of the canonical records (and fourth components) through the
// map, and the map of dense records.
hipError_t launch_compact(const ExportArgs& a, uint32_t maxN, float4* out, float* wOut, hipStream_t stream);
hipError_t launch_identity_map(int R, const uint32_t* repOff, const uint32_t* repCount, uint32_t* srcOff,
                               uint32_t* alive, uint32_t* holeN, hipStream_t stream);
// Moves the fourth components out of n records into w.
hipError_t launch_split_w(float4* pt, float* w, uint32_t n, hipStream_t stream);
hipError_t launch_inject(const InjectArgs& a, hipStream_t stream);
hipError_t launch_zero(const ZeroArgs& a, hipStream_t stream);
// Replica r's created particles, behind its survivors and births.
hipError_t launch_zero_place(int R, const ReplicaTables* tables, const float4* zPos, const int* zType,
                             const uint32_t* zCount, const uint32_t* zeroBase, float4* extra, float* extraW,
                             hipStream_t stream);
hipError_t launch_mt_init_range(uint32_t* st, const uint32_t* seeds, uint32_t Stot, uint32_t off, uint32_t count,
                                hipStream_t stream);

}  // namespace smd
