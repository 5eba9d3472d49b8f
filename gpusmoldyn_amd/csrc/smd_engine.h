// The ensemble engine behind the smd_engine C handle.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "smd_kernels.h"
#include "smd_setup.h"

namespace smd {

struct StageTimer {
  hipEvent_t ev[8];
};

class Engine {
 public:
  Engine(int device, int radixBits);
  ~Engine();
  int add_replica(const smd_sim_spec& spec, const float* pos4, const int* types, uint32_t n);
  smd_status finalize(uint32_t capacity);
  smd_status step(int nsteps);
  smd_status sync();
  smd_status counts(uint32_t* out);
  smd_status get(int r, float* pos4, int* types, uint32_t capN, uint32_t* nOut);
  smd_status get_streams(int r, uint32_t* words, uint32_t capStreams, bool set);
  smd_status debug_stage(int stage, float* pos4, int* types, uint32_t* keysSorted, uint32_t* valsSorted, int* cand,
                         uint32_t* nTotal, uint32_t* nLive);
  smd_status profile(int nsteps, double* us, int maxStages, char* names, int namesCap, int* nStages);
  smd_status particle_steps(unsigned long long* out);
  // Replace the particles of a single-replica engine (setArray / reset).
  smd_status set_particles(const float* pos4, const int* types, uint32_t n);
  // Device arrays of the current particles in the caller layout (pos4 =
  // (x, y, z, w), int types), unpacked from the canonical state into view
  // buffers that stay valid until the next step or view call.
  smd_status view(float4** pos4, int** types, uint32_t* n);

  int device;
  int radixBits;
  bool finalized = false;
  bool broken = false;
  hipStream_t stream = nullptr;
  std::vector<smd_sim_spec> specs;
  std::vector<ReplicaTables> tabs;
  std::vector<std::vector<smd_rxn_derived>> derived;
  std::vector<std::vector<float>> pos0;
  std::vector<std::vector<int>> type0;
  uint32_t R = 0, Stot = 0, deadKey = 0, keyBits = 0, nb = 0, cap = 0, nTilesCap = 0;
  bool anySplit = false, anyBim = false, anyZero = false;
  uint32_t zeroTotal = 0;  // order-0 creations per step, all replicas, at most
  uint64_t Nub = 0, knownN = 0, stepsDone = 0;
  int cur = 0;

  // device state
  ReplicaTables* dTables = nullptr;
  int* dStreamReplica = nullptr;
  uint32_t* dBucketStart = nullptr;
  int* dBucketRep = nullptr;  // replica of each 2^repShift-bucket chunk (nullptr: search bucketStart)
  uint32_t repShift = 0;
  uint32_t *dRepOff = nullptr, *dRepCount = nullptr, *dNewOff = nullptr, *dNewCount = nullptr;
  // where the particles entering the next step are (CanonMap; dNewOff holds
  // the slots' replica offsets)
  uint32_t *dAlive = nullptr, *dHoleOff = nullptr, *dHoleN = nullptr, *dExtraOff = nullptr, *dHoles = nullptr;
  uint32_t* dBirthBase = nullptr;
  uint32_t *dRepDeaths = nullptr, *dRepBirths = nullptr;
  uint32_t* dCounters = nullptr;
  unsigned long long* dParticleSteps = nullptr;  // running sum of particles entering each step
  uint32_t *dN = nullptr, *dNnext = nullptr, *dLive = nullptr;
  uint32_t *dMtState = nullptr, *dMtPar = nullptr;
  float* dGauss = nullptr;
  uint32_t* dFirst = nullptr;
  // canonical particle state: the producer reads one buffer through the map
  // and writes the other densely.  Records (x, y, z, type and fourth
  // component); the fourth components apart (dW) only when they do not pack.
  // Each buffer holds cap slots, then extraCap for the particles a step gains.
  float4* dPT[2] = {nullptr, nullptr};
  float* dW[2] = {nullptr, nullptr};
  bool wApart = false;
  uint32_t extraCap = 0;
  uint32_t stepCap = 0;  // particles that a step can start with
  float4* dAddedPos = nullptr;
  int* dBirthType = nullptr;
  float4* dSortedPT = nullptr;
  uint2* dCand = nullptr;           // pair candidates (CandList)
  uint4* dCandList = nullptr;
  float4* dViewPos = nullptr;  // view() buffers
  int* dViewType = nullptr;
  uint32_t viewCap = 0;
  SortBuffers sb = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 1, nullptr, nullptr, 0, 0};
  uint32_t* dDeadBits = nullptr;                // a bit per slot removed in this step
  uint32_t* dTileDead[2] = {nullptr, nullptr};  // removed per tile, one per step parity (cur)
  uint32_t *dTileBirth = nullptr, *dTileBirthPre = nullptr;
  uint32_t* dBlockSum = nullptr;  // births per finalize workgroup
  uint32_t finBlockTiles = 0;     // its tiles
  uint32_t* dStatus = nullptr;    // sticky kernel error bits
  // host memory that kernels write: the error bits' copy (finalize kernel),
  // and particles read back a few at a time (get)
  static constexpr uint32_t kStage = 1u << 15;  // particles
  uint32_t* hostStatus = nullptr;
  float4* stagePos = nullptr;
  int* stageType = nullptr;
  uint32_t* stageHead = nullptr;
  uint32_t stageCap = 0;
  char* stage = nullptr;            // the allocation behind them
  std::vector<uint32_t> lastN;      // per replica: a recent count (which way get() takes)
  std::mutex readMutex;             // several threads may read: one at a time uses this memory
  uint32_t* dHostStatus = nullptr;  // its device address
  unsigned long long *hostSort = nullptr, *dHostSort = nullptr;
  // order-0 creation: one stream per replica, a per-step creation buffer
  uint32_t *dZMt = nullptr, *dZPar = nullptr, *dZCount = nullptr, *dZeroBase = nullptr;
  float4* dZPos = nullptr;
  int* dZType = nullptr;

  // particle count after each step, written by the finalize kernel into
  // host-visible memory: slot (step & (kRing - 1)) = step << 32 | count
  static constexpr uint32_t kRing = 64;
  unsigned long long* countRing = nullptr;   // host pointer
  unsigned long long* dCountRing = nullptr;  // its device address
  uint32_t* dStepCount = nullptr;
  uint64_t lastSeen = 0;  // latest step whose count has been read

  // Serving: fixed replica slots filled and emptied between steps.
  smd_status finalize_slots(uint32_t nSlots, uint32_t slotBucketBits, uint32_t slotStreams, uint32_t capacity,
                            uint32_t injectCap);
  smd_status admit(int slot, const smd_sim_spec& spec, const float* pos4, const int* types, uint32_t n);
  smd_status retire(int slot);
  bool slotsMode = false;
  uint32_t slotBits = 0, slotStreams = 0;
  uint32_t *dRetire = nullptr, *dInjCount = nullptr, *dInjBase = nullptr, *dInjSrcOff = nullptr;
  float4* dInjPos = nullptr;
  int* dInjType = nullptr;
  int* dInjRep = nullptr;
  uint32_t injCap = 0, injN = 0;
  std::vector<uint8_t> slotBusy;     // admitted and not yet retired
  std::vector<uint8_t> slotPending;  // admitted, particles not yet entered

  // launch shapes and the sort's form (identical results for every setting;
  // see set_knob)
  int producerBlock = 256, pairBlock = 64, segSort = 1;
  int segLow = 0, segHigh = 0;       // digit widths of the segmented sort, 0: not applicable
  uint32_t* dSegScratch = nullptr;   // its tile table and counters
  smd_status set_knob(int knob, int value);
  // the counting cell sort's workgroups when segments are the replicas:
  // replica << kCellGroupShift | slice, largest replicas first
  uint32_t* dCellGroups = nullptr;
  uint32_t* dCellSlices = nullptr;  // per replica: its slices
  uint32_t cellGroups = 0;          // 0: not applicable
  uint32_t cellMinSlices = 1;
  uint64_t cellGroupsN = 0;         // particles (all replicas) up to which they serve
  uint32_t cellBinBits = 0;         // cells per bin (log2) when segments are bins of the high key bits

  // hipGraph replay of two-step pairs and of single steps, one executable
  // graph per ping-pong parity (a single step flips the parity)
  bool useGraphs = true;
  // and per form of the sort
  static constexpr int kForms = 3;
  hipGraphExec_t gexec[kForms][2] = {};
  uint32_t gMaxN[kForms][2] = {};
  hipGraphExec_t oneExec[kForms][2] = {};
  uint32_t oneMaxN[kForms][2] = {};
  bool oneSeen[2] = {false, false};  // a single step of this parity has been launched
  // Waits for the stream, then destroys the executable graph of parity
  // `which` (-1: both), of every form.
  void drop_graph(int which = -1);

  // one replica's count is the total that the finalize kernel published
  // (after sync)
  bool count_known() const { return R == 1 && !slotsMode && lastSeen >= stepsDone; }
  bool seg_sorted() const;  // this engine's digit form sorts replica by replica
  smd_sort_form form_now() const;

 private:
  smd_status enqueue_kernels(uint32_t maxN, StageTimer* timer);
  SegSortArgs seg_args() const;
  // How the step sorts its keys: digit passes (global or segmented) and the
  // cell table kernel, or the counting cell sort by replica or by bins of
  // the high key bits, which writes the cell table itself.
  enum class SortForm { kDigits, kCellsByReplica, kCellsByBin };
  SortForm sort_form(uint32_t maxN) const;
  smd_status plan_cell_sort();
  // Counting keys per cell depends on how the particles lie: a slice that
  // holds too many for its list works through them window by window.  Steps
  // report such slices to the host (hostSort), which takes the digit passes
  // for digitsHold steps where they are the faster form, then looks again.
  void watch_sort();
  bool digits_faster(uint32_t most, uint32_t rounds) const;
  int graph_form(uint64_t n) const {
    return anyBim ? (int)sort_form((uint32_t)std::min<uint64_t>(n, 0xFFFFFFFFu)) : 0;
  }
  void restart_sort_watch();
  static constexpr uint64_t kDigitsHold = 1024;
  uint64_t digitsUntil = 0;           // steps done until which the digit passes run (0: they need not)
  uint64_t digitsHold = kDigitsHold;  // doubled each time
  uint64_t sortFrom = 0;              // reports of steps up to here are settled
  bool sortSeen = false;              // a report could have been read since
  // sorted keys, records and cell table of the step (debug: also the values
  // and the removed particles)
  hipError_t sort_keys(uint32_t maxN, bool tilesLaid, StageTimer* timer, bool debug);
  smd_status step_graph(int pairs);
  smd_status alloc_particle_buffers(uint32_t c);
  smd_status alloc_apart();
  smd_status take_apart(const float* pos4, size_t n);
  CanonMap canon_map() const;
  CandArgs cand_args() const;
  ResolveArgs resolve_args() const;
  ProducerArgs producer_args() const;
  ExportArgs export_args(int r) const;
  smd_status set_dense();
  smd_status alloc_stage();
  float4* dStagePos = nullptr;
  int* dStageType = nullptr;
  uint32_t* dStageHead = nullptr;
  void free_particle_buffers();
  void refresh_bound(bool block);
  smd_status grow(uint64_t need);
  smd_status ensure_capacity();
  // Upper bound of the particle count after one step that starts with x.
  uint64_t step_bound(uint64_t x) const { return (anySplit ? 2 * x : x) + zeroTotal; }
  smd_status check_status();
  smd_status enqueue_step(StageTimer* timer);
  // Host-side buffer selection that enqueue_kernels advances by one step.
  struct HostSnapshot {
    int cur;
    uint32_t *repOff, *newOff, *repCount, *newCount, *n, *nnext;
    SortBuffers sb;
  };
  HostSnapshot snapshot() const;
  void restore(const HostSnapshot& s);
  HostSnapshot oneAfter[kForms][2] = {};  // the selection after a single-step graph
  smd_status capture(int steps, uint32_t maxN, hipGraphExec_t* exec, HostSnapshot* after);
  smd_status step_one();
};

}  // namespace smd

// The opaque C handle of include/gpusmoldyn.h.
struct smd_engine {
  smd::Engine* impl;
};
