// Host orchestration of the timestep over an ensemble of replicas (a plain
// simulation is an ensemble of one).  Replaces ParticleSystem::_initialize
// (particleSystem.cpp:573-751) and ParticleSystem::update (:829-1001): the
// particle state stays in HBM, particle counts live on the device, and the
// host only reads a count back (asynchronously) to bound grid sizes and to
// grow the buffers before they could overflow.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "smd_engine.h"

namespace smd {

#define HIPCHK(x)                                                                          \
  do {                                                                                     \
    hipError_t e_ = (x);                                                                   \
    if (e_ != hipSuccess) {                                                                \
      set_error(std::string("HIP error '") + hipGetErrorString(e_) + "' in " #x);          \
      return SMD_ERR_HIP;                                                                  \
    }                                                                                      \
  } while (0)

template <typename T>
static hipError_t dalloc(T** p, size_t count) {
  *p = nullptr;
  if (count == 0) count = 1;
  return hipMalloc((void**)p, count * sizeof(T));
}

template <typename T>
static void dfree(T*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

static inline uint32_t round64(uint32_t x) { return (x + 63u) & ~63u; }

// Whether every fourth component's bits leave room for a type.
static bool components_pack(const float* pos4, size_t n) {
  for (size_t i = 0; i < n; ++i) {
    uint32_t b;
    std::memcpy(&b, &pos4[4 * i + 3], sizeof(b));
    if (b & (uint32_t)kTypeMask) return false;
  }
  return true;
}

// Caller layout (pos4 = x, y, z, w; int types) to the canonical device layout
// (w in the records, or in dw when that is given).
static hipError_t upload_particles(const float* pos4, const int* types, size_t n, float4* dpt, float* dw) {
  std::vector<float4> pt(n);
  std::vector<float> w(dw ? n : 0);
  for (size_t i = 0; i < n; ++i) {
    uint32_t b = 0;
    if (dw) w[i] = pos4[4 * i + 3];
    else std::memcpy(&b, &pos4[4 * i + 3], sizeof(b));
    b |= (uint32_t)types[i];
    float wb;
    std::memcpy(&wb, &b, sizeof(wb));
    pt[i] = make_float4(pos4[4 * i], pos4[4 * i + 1], pos4[4 * i + 2], wb);
  }
  hipError_t e = hipMemcpy(dpt, pt.data(), n * sizeof(float4), hipMemcpyHostToDevice);
  if (e == hipSuccess && dw) e = hipMemcpy(dw, w.data(), n * sizeof(float), hipMemcpyHostToDevice);
  return e;
}

Engine::Engine(int dev, int rbits) : device(dev), radixBits(rbits == 4 || rbits == 8 || rbits == 11 ? rbits : 0) {}

Engine::~Engine() {
  drop_graph();
  if (stream) {
    (void)hipSetDevice(device);
    (void)hipStreamSynchronize(stream);
  }
  free_particle_buffers();
  dfree(dTables);
  dfree(dStreamReplica);
  dfree(dBucketStart);
  dfree(dBucketRep);
  dfree(dRepOff);
  dfree(dRepCount);
  dfree(dNewOff);
  dfree(dNewCount);
  dfree(dAlive);
  dfree(dHoleOff);
  dfree(dHoleN);
  dfree(dExtraOff);
  dfree(dBirthBase);
  dfree(dRepDeaths);
  dfree(dRepBirths);
  dfree(dCounters);
  dfree(dParticleSteps);
  dfree(dMtState);
  dfree(dMtPar);
  dfree(dGauss);
  dfree(dFirst);
  dfree(dCellGroups);
  dfree(dCellSlices);
  dfree(dRetire);
  dfree(dInjCount);
  dfree(dInjBase);
  dfree(dStatus);
  dfree(dZMt);
  dfree(dZPar);
  dfree(dZCount);
  dfree(dZeroBase);
  dfree(dZPos);
  dfree(dZType);
  dfree(dInjSrcOff);
  dfree(dInjPos);
  dfree(dInjType);
  dfree(dInjRep);
  if (countRing) (void)hipHostFree(countRing);
  if (stage) (void)hipHostFree(stage);
  dfree(dStepCount);
  if (stream) (void)hipStreamDestroy(stream);
}

void Engine::free_particle_buffers() {
  for (int k = 0; k < 2; ++k) {
    dfree(dPT[k]);
    dfree(dW[k]);
  }
  dfree(dAddedPos);
  dfree(dBirthType);
  dfree(dSortedPT);
  dfree(dCand);
  dfree(dCandList);
  dfree(dViewPos);
  dfree(dViewType);
  viewCap = 0;
  dfree(sb.keys);
  dfree(sb.vals);
  dfree(sb.keysAlt);
  dfree(sb.valsAlt);
  dfree(sb.counts);
  dfree(dDeadBits);
  dfree(dTileDead[0]);
  dfree(dTileDead[1]);
  dfree(dHoles);
  dfree(dTileBirth);
  dfree(dTileBirthPre);
  dfree(dBlockSum);
  dfree(dSegScratch);
}

int Engine::add_replica(const smd_sim_spec& spec, const float* pos4, const int* types, uint32_t n) {
  if (finalized) {
    set_error("add_replica after finalize");
    return -SMD_ERR_INVALID;
  }
  ReplicaTables T;
  std::string err;
  std::vector<smd_rxn_derived> der(spec.num_reactions > 0 ? spec.num_reactions : 1);
  if (!derive_tables(spec, T, der.data(), err)) {
    set_error(err);
    return -SMD_ERR_RXN_SETUP;
  }
  for (uint32_t i = 0; i < n; ++i)
    if (types[i] < 1 || types[i] >= spec.num_types) {
      set_error("initial particle type out of range");
      return -SMD_ERR_INVALID;
    }
  specs.push_back(spec);
  tabs.push_back(T);
  derived.push_back(der);
  pos0.emplace_back(pos4, pos4 + 4 * (size_t)n);
  type0.emplace_back(types, types + n);
  return (int)tabs.size() - 1;
}

smd_status Engine::alloc_particle_buffers(uint32_t c) {
  cap = c;
  // A step only starts where its outcome fits the capacity if every particle
  // splits and all that can be created or admitted is (step_bound): half the
  // capacity enters at most, and as much is gained.
  const bool gains = anySplit || slotsMode;
  stepCap = gains ? cap / 2 + 1 : cap;
  extraCap = (gains ? cap / 2 + 1 : 0) + zeroTotal;
  for (int k = 0; k < 2; ++k) HIPCHK(dalloc(&dPT[k], (size_t)cap + extraCap));
  if (wApart) {
    smd_status st = alloc_apart();
    if (st != SMD_OK) return st;
  }
  if (gains) {
    HIPCHK(dalloc(&dAddedPos, stepCap));
    HIPCHK(dalloc(&dBirthType, stepCap));
    HIPCHK(hipMemsetAsync(dBirthType, 0, (size_t)stepCap * sizeof(int), stream));
  }
  HIPCHK(dalloc(&dSortedPT, stepCap));
  HIPCHK(dalloc(&dCand, stepCap));
  HIPCHK(hipMemsetAsync(dCand, 0, (size_t)stepCap * sizeof(uint2), stream));  // tag 0: no step's
  HIPCHK(dalloc(&dCandList, pair_list_size()));
  // the cell sort reads keys as whole vectors of four
  HIPCHK(dalloc(&sb.keys, (size_t)stepCap + 4));
  HIPCHK(dalloc(&sb.vals, stepCap));
  HIPCHK(dalloc(&sb.keysAlt, (size_t)stepCap + 4));
  HIPCHK(dalloc(&sb.valsAlt, stepCap));
  HIPCHK(dalloc(&sb.counts, sort_counts_words(stepCap, radixBits)));
  nTilesCap = stepCap / kCompactTile + 2;
  const size_t words = (size_t)nTilesCap * (kCompactTile / 32);
  HIPCHK(dalloc(&dDeadBits, words));
  HIPCHK(dalloc(&dHoles, stepCap));
  HIPCHK(dalloc(&dTileBirth, nTilesCap));
  HIPCHK(dalloc(&dTileBirthPre, nTilesCap));
  finBlockTiles = finalize_block_tiles(nTilesCap);
  HIPCHK(dalloc(&dBlockSum, (size_t)nTilesCap / finBlockTiles + 1));
  if (segHigh) HIPCHK(dalloc(&dSegScratch, seg_sort_words(stepCap, (int)R, std::max(segLow, segHigh))));
  HIPCHK(hipMemsetAsync(dDeadBits, 0, words * sizeof(uint32_t), stream));
  for (int k = 0; k < 2; ++k) {
    HIPCHK(dalloc(&dTileDead[k], nTilesCap));
    HIPCHK(hipMemsetAsync(dTileDead[k], 0, nTilesCap * sizeof(uint32_t), stream));
  }
  HIPCHK(hipMemsetAsync(dTileBirth, 0, nTilesCap * sizeof(uint32_t), stream));
  return SMD_OK;
}

// Both arrays or none: the kernels tell by the pointers whether components
// live apart.
smd_status Engine::alloc_apart() {
  float* w[2] = {nullptr, nullptr};
  hipError_t e = hipSuccess;
  for (int k = 0; k < 2 && e == hipSuccess; ++k) e = dalloc(&w[k], (size_t)cap + extraCap);
  if (e != hipSuccess)
    for (float*& x : w) dfree(x);
  HIPCHK(e);
  for (int k = 0; k < 2; ++k) dW[k] = w[k];
  return SMD_OK;
}

// New particles whose fourth components do not pack: from here on all
// components live apart.
smd_status Engine::take_apart(const float* pos4, size_t n) {
  if (wApart || components_pack(pos4, n)) return SMD_OK;
  drop_graph();
  HIPCHK(hipStreamSynchronize(stream));
  smd_status st = alloc_apart();
  if (st != SMD_OK) return st;
  wApart = true;
  HIPCHK(launch_split_w(dPT[cur], dW[cur], cap + extraCap, stream));
  HIPCHK(hipStreamSynchronize(stream));
  return SMD_OK;
}

CanonMap Engine::canon_map() const {
  CanonMap m;
  m.srcOff = dNewOff;  // the layout of the last step: swapped with the next one's
  m.alive = dAlive;
  m.holeOff = dHoleOff;
  m.holeN = dHoleN;
  m.holes = dHoles;
  m.extraOff = dExtraOff;
  m.extraBase = cap;
  return m;
}

// The map of particles that lie densely by dRepOff / dRepCount in dPT[cur].
smd_status Engine::set_dense() {
  HIPCHK(launch_identity_map((int)R, dRepOff, dRepCount, dNewOff, dAlive, dHoleN, stream));
  return SMD_OK;
}

smd_status Engine::finalize(uint32_t capacity) {
  if (finalized) return SMD_OK;
  if (tabs.empty()) {
    set_error("no replicas");
    return SMD_ERR_INVALID;
  }
  HIPCHK(hipSetDevice(device));
  HIPCHK(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
  R = (uint32_t)tabs.size();
  // Bucket and stream layout.
  uint64_t buckets = 0, streams = 0, total = 0;
  anySplit = false;
  anyBim = false;
  anyZero = false;
  uint64_t zeros = 0;
  for (uint32_t r = 0; r < R; ++r) {
    ReplicaTables& T = tabs[r];
    T.bucketOff = (uint32_t)buckets;
    buckets += T.numBuckets;
    T.streamOff = (uint32_t)streams;
    streams += round64(T.numStreams);
    total += type0[r].size();
    for (int x = 0; x < T.numRxn; ++x)
      if (specs[r].rxn[x].order == 1 && T.prodY[x] > 0) anySplit = true;
    if (T.hasBim) anyBim = true;
    T.zeroOff = (uint32_t)zeros;
    zeros += T.zeroMax;
    if (T.numZero) anyZero = true;
  }
  if (buckets >= (1ull << 31) || streams >= (1ull << 31) || zeros >= (1ull << 30)) {
    set_error("too many buckets, streams or order-0 creations");
    return SMD_ERR_INVALID;
  }
  zeroTotal = (uint32_t)zeros;
  deadKey = (uint32_t)buckets;
  keyBits = 0;
  while ((1ull << keyBits) <= deadKey) ++keyBits;
  // automatic digit width: 8 bits (11-bit digits save a pass for 17-22-bit
  // keys but each pass costs more than the pass saved: 80 KB of LDS per
  // workgroup and 2048 scan rows)
  if (radixBits == 0) radixBits = 8;
  nb = deadKey + 1;
  // Ensembles sort each replica's segment on its local cells: two digit
  // passes cover the largest replica grid plus the removed mark.
  {
    uint32_t maxGb = 0;
    for (uint32_t r = 0; r < R; ++r) {
      uint32_t b = 0;
      while ((1u << b) < tabs[r].numBuckets) ++b;
      maxGb = std::max(maxGb, b);
    }
    seg_sort_digits(maxGb, segLow, segHigh);
    if (R <= 1) segLow = segHigh = 0;
  }
  Stot = (uint32_t)streams;
  uint64_t c = capacity ? capacity : std::max<uint64_t>(anySplit ? 8 * total : total, 1024);
  if (c < step_bound(total)) c = step_bound(total);
  if (c >= (1ull << 31)) {
    set_error("capacity too large");
    return SMD_ERR_CAPACITY;
  }

  // Per-replica arrays.
  HIPCHK(dalloc(&dTables, R));
  HIPCHK(hipMemcpy(dTables, tabs.data(), R * sizeof(ReplicaTables), hipMemcpyHostToDevice));
  std::vector<int> streamRep(Stot, -1);
  for (uint32_t r = 0; r < R; ++r)
    for (uint32_t k = 0; k < round64(tabs[r].numStreams); ++k) streamRep[tabs[r].streamOff + k] = (int)r;
  HIPCHK(dalloc(&dStreamReplica, Stot));
  HIPCHK(hipMemcpy(dStreamReplica, streamRep.data(), Stot * sizeof(int), hipMemcpyHostToDevice));
  std::vector<uint32_t> bstart(R + 1);
  for (uint32_t r = 0; r < R; ++r) bstart[r] = tabs[r].bucketOff;
  bstart[R] = deadKey;
  HIPCHK(dalloc(&dBucketStart, R + 1));
  HIPCHK(hipMemcpy(dBucketStart, bstart.data(), (R + 1) * sizeof(uint32_t), hipMemcpyHostToDevice));
  // Replica of a bucket by one lookup: every replica owns a power-of-two run
  // of buckets at an offset that is a multiple of the smallest such run, so
  // chunks of that size never straddle two replicas.
  {
    uint32_t minBits = 31;
    for (uint32_t r = 0; r < R; ++r) {
      uint32_t b = 0;
      while ((1u << b) < tabs[r].numBuckets) ++b;
      minBits = std::min(minBits, b);
    }
    const uint64_t chunks = ((uint64_t)deadKey + (1ull << minBits) - 1) >> minBits;
    if (R > 1 && chunks <= (1ull << 22)) {
      std::vector<int> rep((size_t)std::max<uint64_t>(chunks, 1), -1);
      for (uint32_t r = 0; r < R; ++r)
        for (uint64_t c = tabs[r].bucketOff >> minBits; c < ((uint64_t)tabs[r].bucketOff + tabs[r].numBuckets) >> minBits;
             ++c)
          rep[c] = (int)r;
      HIPCHK(dalloc(&dBucketRep, rep.size()));
      HIPCHK(hipMemcpy(dBucketRep, rep.data(), rep.size() * sizeof(int), hipMemcpyHostToDevice));
      repShift = minBits;
    }
  }
  std::vector<uint32_t> off(R + 1), cnt(R);
  uint64_t o = 0;
  for (uint32_t r = 0; r < R; ++r) {
    off[r] = (uint32_t)o;
    cnt[r] = (uint32_t)type0[r].size();
    o += cnt[r];
  }
  off[R] = (uint32_t)o;
  for (uint32_t** p : {&dRepOff, &dNewOff}) HIPCHK(dalloc(p, R + 1));
  for (uint32_t** p : {&dRepCount, &dNewCount, &dAlive, &dHoleOff, &dHoleN, &dExtraOff, &dBirthBase, &dRepDeaths,
                       &dRepBirths})
    HIPCHK(dalloc(p, R));
  HIPCHK(hipMemset(dHoleOff, 0, R * sizeof(uint32_t)));
  HIPCHK(hipMemset(dExtraOff, 0, R * sizeof(uint32_t)));
  HIPCHK(hipMemcpy(dRepOff, off.data(), (R + 1) * sizeof(uint32_t), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dRepCount, cnt.data(), R * sizeof(uint32_t), hipMemcpyHostToDevice));
  HIPCHK(hipMemset(dRepDeaths, 0, R * sizeof(uint32_t)));
  HIPCHK(hipMemset(dRepBirths, 0, R * sizeof(uint32_t)));
  HIPCHK(dalloc(&dCounters, 8));
  HIPCHK(hipMemset(dCounters, 0, 8 * sizeof(uint32_t)));
  HIPCHK(dalloc(&dParticleSteps, 1));
  HIPCHK(hipMemset(dParticleSteps, 0, sizeof(unsigned long long)));
  dN = dCounters;
  dNnext = dCounters + 1;
  dLive = dCounters + 2;
  const uint32_t tot32 = (uint32_t)total;
  HIPCHK(hipMemcpy(dN, &tot32, sizeof(uint32_t), hipMemcpyHostToDevice));
  HIPCHK(dalloc(&dFirst, first_words(nb)));
  {
    smd_status st = plan_cell_sort();
    if (st != SMD_OK) return st;
  }

  // Gaussian table: the producer keeps its half t[1 .. kGaussDim / 2], from
  // which the antisymmetry rebuilds every entry (gauss_entry).
  std::vector<float> g(kGaussDim);
  gauss_table(g.data(), kGaussDim);
  for (int u = 0; u < kGaussDim; ++u) {
    const int k = u - 1;
    const float want = (u >= 1 && u <= kGaussDim / 2) ? g[k + 1] : -g[((kGaussDim - u) & (kGaussDim / 2 - 1)) + 1];
    if (std::memcmp(&want, &g[u], sizeof(float)) != 0) {
      set_error("Gaussian table is not antisymmetric");
      return SMD_ERR_INVALID;
    }
  }
  HIPCHK(dalloc(&dGauss, kGaussDim / 2));
  HIPCHK(hipMemcpy(dGauss, g.data() + 1, kGaussDim / 2 * sizeof(float), hipMemcpyHostToDevice));

  // Random streams: stream k of a replica uses MersenneTwister.dat record
  // k % 32768 and seed k of that replica's seed sequence.
  std::string err;
  const uint32_t* dat = mt_dat(err);
  if (!dat) {
    set_error(err);
    return SMD_ERR_IO;
  }
  std::vector<uint32_t> seeds(Stot, 0u), par(3 * (size_t)Stot, 0u);
  for (uint32_t r = 0; r < R; ++r) {
    const ReplicaTables& T = tabs[r];
    if (!stream_seeds(specs[r].seed, T.numStreams, &seeds[T.streamOff], err)) {
      set_error(err);
      return SMD_ERR_IO;
    }
    for (uint32_t k = 0; k < T.numStreams; ++k) {
      const uint32_t rec = k % kMtParamSets;
      par[T.streamOff + k] = dat[4 * rec];
      par[(size_t)Stot + T.streamOff + k] = dat[4 * rec + 1];
      par[2 * (size_t)Stot + T.streamOff + k] = dat[4 * rec + 2];
    }
  }
  HIPCHK(dalloc(&dMtState, (size_t)kMtWords * Stot));
  HIPCHK(dalloc(&dMtPar, 3 * (size_t)Stot));
  HIPCHK(hipMemcpy(dMtPar, par.data(), par.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
  uint32_t* dSeeds = nullptr;
  HIPCHK(dalloc(&dSeeds, Stot));
  HIPCHK(hipMemcpy(dSeeds, seeds.data(), Stot * sizeof(uint32_t), hipMemcpyHostToDevice));
  HIPCHK(launch_mt_init(dMtState, dSeeds, Stot, stream));
  HIPCHK(hipStreamSynchronize(stream));
  dfree(dSeeds);
  HIPCHK(dalloc(&dStatus, 1));
  HIPCHK(hipMemset(dStatus, 0, sizeof(uint32_t)));
  sb.status = dStatus;
  if (anyZero) {
    // Replica r's creation stream: the next stream after its S particle
    // streams (seed S of its seed sequence, MersenneTwister.dat record S).
    std::vector<uint32_t> zs(R), zp(3 * (size_t)R);
    for (uint32_t r = 0; r < R; ++r) {
      const uint32_t S = tabs[r].numStreams;
      std::vector<uint32_t> sq(S + 1);
      if (!stream_seeds(specs[r].seed, S + 1, sq.data(), err)) {
        set_error(err);
        return SMD_ERR_IO;
      }
      zs[r] = sq[S];
      const uint32_t rec = S % kMtParamSets;
      for (int w = 0; w < 3; ++w) zp[(size_t)w * R + r] = dat[4 * rec + w];
    }
    HIPCHK(dalloc(&dZMt, (size_t)kMtWords * R));
    HIPCHK(dalloc(&dZPar, 3 * (size_t)R));
    HIPCHK(dalloc(&dZCount, R));
    HIPCHK(dalloc(&dZeroBase, R));
    HIPCHK(dalloc(&dZPos, zeroTotal));
    HIPCHK(dalloc(&dZType, zeroTotal));
    HIPCHK(hipMemcpy(dZPar, zp.data(), zp.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    uint32_t* dzs = nullptr;
    HIPCHK(dalloc(&dzs, R));
    HIPCHK(hipMemcpy(dzs, zs.data(), R * sizeof(uint32_t), hipMemcpyHostToDevice));
    HIPCHK(launch_mt_init(dZMt, dzs, R, stream));
    HIPCHK(hipStreamSynchronize(stream));
    dfree(dzs);
  }

  // Particles.
  for (uint32_t r = 0; r < R && !wApart; ++r) wApart = !components_pack(pos0[r].data(), cnt[r]);
  smd_status st = alloc_particle_buffers((uint32_t)c);
  if (st != SMD_OK) return st;
  for (uint32_t r = 0; r < R; ++r) {
    if (cnt[r] == 0) continue;
    HIPCHK(upload_particles(pos0[r].data(), type0[r].data(), cnt[r], dPT[0] + off[r],
                            wApart ? dW[0] + off[r] : nullptr));
  }
  cur = 0;
  st = set_dense();
  if (st != SMD_OK) return st;
  Nub = total;
  knownN = total;
  stepsDone = 0;
  HIPCHK(hipHostMalloc((void**)&countRing, kRing * sizeof(unsigned long long),
                       hipHostMallocMapped | hipHostMallocCoherent));
  std::memset(countRing, 0, kRing * sizeof(unsigned long long));
  HIPCHK(hipHostGetDevicePointer((void**)&dCountRing, countRing, 0));
  st = alloc_stage();
  if (st != SMD_OK) return st;
  lastN = cnt;
  HIPCHK(dalloc(&dStepCount, 1));
  HIPCHK(hipMemset(dStepCount, 0, sizeof(uint32_t)));
  lastSeen = 0;
  HIPCHK(hipStreamSynchronize(stream));
  finalized = true;
  return SMD_OK;
}

smd_status Engine::alloc_stage() {
  stageCap = std::min(kStage, cap);
  const size_t head = 256, pos = (size_t)stageCap * sizeof(float4);
  HIPCHK(hipHostMalloc((void**)&stage, head + pos + (size_t)stageCap * sizeof(int),
                       hipHostMallocMapped | hipHostMallocCoherent));
  char* dev = nullptr;
  HIPCHK(hipHostGetDevicePointer((void**)&dev, stage, 0));
  std::memset(stage, 0, head);
  hostStatus = (uint32_t*)stage;
  dHostStatus = (uint32_t*)dev;
  hostSort = (unsigned long long*)(stage + 128);
  dHostSort = (unsigned long long*)(dev + 128);
  stageHead = (uint32_t*)(stage + 64);
  dStageHead = (uint32_t*)(dev + 64);
  stagePos = (float4*)(stage + head);
  dStagePos = (float4*)(dev + head);
  stageType = (int*)(stage + head + pos);
  dStageType = (int*)(dev + head + pos);
  return SMD_OK;
}

// Bound on the particle count after all enqueued steps, refreshed from the
// latest count the finalize kernel has published (blocking: after the stream
// has drained, the count after the last step).
void Engine::refresh_bound(bool block) {
  if (lastSeen >= stepsDone) return;
  if (block) (void)hipStreamSynchronize(stream);
  const uint64_t oldest = stepsDone >= kRing ? stepsDone - kRing + 1 : 1;
  for (uint64_t s = stepsDone; s > lastSeen && s >= oldest; --s) {
    const unsigned long long v = __atomic_load_n(&countRing[s & (kRing - 1)], __ATOMIC_ACQUIRE);
    if ((uint32_t)(v >> 32) != (uint32_t)s) continue;
    knownN = (uint32_t)v;
    uint64_t b = knownN;
    for (uint64_t k = 0; k < stepsDone - s && b < (1ull << 40); ++k) b = step_bound(b);
    Nub = std::min<uint64_t>(Nub, b);
    lastSeen = s;
    break;
  }
}

smd_status Engine::grow(uint64_t need) {
  drop_graph();
  HIPCHK(hipStreamSynchronize(stream));
  uint64_t nc = std::max<uint64_t>(need, 2ull * cap);
  if (nc >= (1ull << 31)) {
    set_error("particle count exceeds the 2^31 capacity limit");
    return SMD_ERR_CAPACITY;
  }
  const uint32_t n = (uint32_t)knownN;
  float4* keepPT = nullptr;
  float* keepW = nullptr;
  HIPCHK(dalloc(&keepPT, n));
  if (wApart) HIPCHK(dalloc(&keepW, n));
  HIPCHK(launch_compact(export_args(-1), n, keepPT, keepW, stream));
  HIPCHK(hipStreamSynchronize(stream));
  free_particle_buffers();
  smd_status st = alloc_particle_buffers((uint32_t)nc);
  if (st != SMD_OK) return st;
  cur = 0;
  if (n) {
    HIPCHK(hipMemcpyAsync(dPT[0], keepPT, n * sizeof(float4), hipMemcpyDeviceToDevice, stream));
    if (wApart) HIPCHK(hipMemcpyAsync(dW[0], keepW, n * sizeof(float), hipMemcpyDeviceToDevice, stream));
  }
  st = set_dense();
  HIPCHK(hipStreamSynchronize(stream));
  dfree(keepPT);
  dfree(keepW);
  return st;
}

smd_status Engine::ensure_capacity() {
  refresh_bound(false);
  watch_sort();
  const uint64_t needAfter = step_bound(Nub);
  if (needAfter <= cap) return SMD_OK;
  refresh_bound(true);
  const uint64_t need2 = step_bound(Nub);
  if (need2 <= cap) return SMD_OK;
  return grow(2 * need2);
}

smd_status Engine::enqueue_step(StageTimer* timer) {
  const uint32_t maxN = (uint32_t)std::min<uint64_t>(Nub, stepCap);
  smd_status st = enqueue_kernels(maxN, timer);
  if (st != SMD_OK) return st;
  ++stepsDone;
  Nub = std::min<uint64_t>(step_bound(Nub), (uint64_t)cap);
  return SMD_OK;
}

void Engine::drop_graph(int which) {
  const int lo = which < 0 ? 0 : which, hi = which < 0 ? 1 : which;
  bool any = false;
  for (int f = 0; f < kForms; ++f)
    for (int p = lo; p <= hi; ++p) any = any || gexec[f][p] || oneExec[f][p];
  if (!any) return;
  // A launch of the graph may still be queued or running: the executable
  // graph (and the kernel arguments it owns) must outlive it.
  if (stream) {
    (void)hipSetDevice(device);
    (void)hipStreamSynchronize(stream);
  }
  for (int f = 0; f < kForms; ++f)
    for (int p = lo; p <= hi; ++p) {
      if (gexec[f][p]) (void)hipGraphExecDestroy(gexec[f][p]);
      if (oneExec[f][p]) (void)hipGraphExecDestroy(oneExec[f][p]);
      gexec[f][p] = oneExec[f][p] = nullptr;
      gMaxN[f][p] = oneMaxN[f][p] = 0;
    }
}

Engine::HostSnapshot Engine::snapshot() const {
  return HostSnapshot{cur, dRepOff, dNewOff, dRepCount, dNewCount, dN, dNnext, sb};
}

void Engine::restore(const HostSnapshot& s) {
  cur = s.cur;
  dRepOff = s.repOff;
  dNewOff = s.newOff;
  dRepCount = s.repCount;
  dNewCount = s.newCount;
  dN = s.n;
  dNnext = s.nnext;
  sb = s.sb;
}

// Captures `steps` steps of at most maxN particles; the host-side buffer
// selection stays as it is (after: what the steps would make of it).
smd_status Engine::capture(int steps, uint32_t maxN, hipGraphExec_t* exec, HostSnapshot* after) {
  const HostSnapshot before = snapshot();
  hipGraph_t g = nullptr;
  HIPCHK(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
  smd_status st = SMD_OK;
  for (int k = 0; k < steps && st == SMD_OK; ++k) st = enqueue_kernels(maxN, nullptr);
  hipError_t e = hipStreamEndCapture(stream, &g);
  // nothing ran: the host-side buffer selection goes back to where it was
  if (after) *after = snapshot();
  restore(before);
  if (st != SMD_OK) {
    if (g) (void)hipGraphDestroy(g);
    return st;
  }
  HIPCHK(e);
  hipGraphExec_t x = nullptr;
  e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e != hipSuccess) {
    if (x) (void)hipGraphExecDestroy(x);
    HIPCHK(e);
  }
  *exec = x;
  return SMD_OK;
}

// One step: launch by launch the first time (a capture costs more than it
// saves then), from a graph after that (the loop of a program that looks at
// the particles after every step: 5 launches as one).
smd_status Engine::step_one() {
  smd_status st = ensure_capacity();
  if (st != SMD_OK) return st;
  const int p = cur;
  if (!useGraphs || !oneSeen[p]) {
    oneSeen[p] = true;
    return enqueue_step(nullptr);
  }
  const int f = graph_form(Nub);
  if (oneExec[f][p] && Nub > oneMaxN[f][p]) refresh_bound(true);
  if (oneExec[f][p] && Nub > oneMaxN[f][p]) drop_graph(p);
  if (!oneExec[f][p]) {
    // headroom where the bound only follows stale counts
    const uint32_t maxN = (uint32_t)std::min<uint64_t>(Nub + Nub / 2, stepCap);
    st = capture(1, maxN, &oneExec[f][p], &oneAfter[f][p]);
    if (st != SMD_OK) return st;
    oneMaxN[f][p] = maxN;
  }
  HIPCHK(hipGraphLaunch(oneExec[f][p], stream));
  restore(oneAfter[f][p]);
  std::fill(slotPending.begin(), slotPending.end(), (uint8_t)0);
  ++stepsDone;
  Nub = std::min<uint64_t>(step_bound(Nub), (uint64_t)cap);
  return SMD_OK;
}

// Two consecutive steps captured as one hipGraph: after two steps every
// ping-pong buffer is back in place, so the graph can be replayed as long as
// the particle bound stays within the grid sizes it was captured with.  An
// eager step (an admission in a slot engine) flips the ping-pong parity, so
// one graph is kept per parity.
smd_status Engine::step_graph(int pairs) {
  for (int k = 0; k < pairs; ++k) {
    // before a long run of steps is queued, one look at how the first ones
    // sorted (a wait of some 20 us; short runs are looked at by the next call)
    const bool look = k > 0 && !sortSeen && pairs - k >= 16 && graph_form(Nub) != (int)SortForm::kDigits;
    sortSeen = sortSeen || look;
    refresh_bound(look);
    watch_sort();
    uint64_t need = step_bound(step_bound(Nub));  // output of the second step
    if (need > cap) {
      refresh_bound(true);
      need = step_bound(step_bound(Nub));
      if (need > cap) {
        smd_status st = grow(2 * need);  // waits for the stream and drops the graphs
        if (st != SMD_OK) return st;
      }
    }
    uint64_t bound = step_bound(Nub);  // input bound of the second step
    const int p = cur;
    const int f = graph_form(bound);
    if (gexec[f][p] && bound > gMaxN[f][p]) {
      // a stale count alone must not force a new capture: read the exact one
      refresh_bound(true);
      bound = step_bound(Nub);
    }
    uint64_t want = bound;
    if (gexec[f][p] && bound > gMaxN[f][p]) {
      // outgrown: grids with headroom, so that a growing system re-captures rarely
      want = std::max<uint64_t>(bound, (uint64_t)gMaxN[f][p] + gMaxN[f][p] / 2);
      drop_graph(p);
    }
    if (!gexec[f][p]) {
      const uint32_t maxN = (uint32_t)std::min<uint64_t>(want, stepCap);
      smd_status st = capture(2, maxN, &gexec[f][p], nullptr);
      if (st != SMD_OK) return st;
      gMaxN[f][p] = maxN;
    }
    HIPCHK(hipGraphLaunch(gexec[f][p], stream));
    // two steps: every ping-pong selection is back where it was
    std::fill(slotPending.begin(), slotPending.end(), (uint8_t)0);
    stepsDone += 2;
    Nub = std::min<uint64_t>(step_bound(step_bound(Nub)), (uint64_t)cap);
  }
  return SMD_OK;
}

// The step's key sort: segmented by replica when the engine holds several
// replicas and the knob allows it (the same sorted keys, values and records
// either way), else over all keys at once.
bool Engine::seg_sorted() const { return segHigh && segSort && sb.algo == 1; }

SegSortArgs Engine::seg_args() const {
  SegSortArgs g;
  g.R = (int)R;
  g.segOff = dRepOff;
  g.segCount = dRepCount;
  g.bucketOff = dBucketStart;
  g.deadKey = deadKey;
  g.lowBits = segLow;
  g.highBits = segHigh;
  g.scratch = dSegScratch;
  return g;
}

// Form and workgroups of the counting cell sort.  By replica, every slice of
// a replica's cells reads all of the replica's keys; by bins, a digit pass
// over the keys' high bits comes first and every slice of a bin reads the
// bin's.  Measured, us per sort, by replica / by bins / by digits (replica by
// replica where that applies): 512 replicas of 2k to 64k 115 / 255 / 211, with
// one of 140k beside them 119 / 250 / 225, 16 of 140k 50 / 66 / 81, 16 of 262k
// 108 / 115 / 145, but 9 of 262k 97 / 67 / 145, 2 of 140k 39 / 31 / 64, one
// system of 16k 8 / 17, one of 100k 35 / 20.  So bins take single systems from
// 48k particles, replicas above 262k (whose slices would read too many keys)
// and those above 131k unless they are a sixteenth of the whole.  Ensembles
// whose cells outnumber their particles so that most slices are empty keep the
// digits (an empty workgroup costs its start, 4 to 6 us per 1000): 512 replicas
// of 2k on 2^17 cells 154 by replica, 107 by digits; 300, 98 / 83; 256, 84 / 75;
// of 20k 267 / 305.  So do slot engines (16 jobs of 1k to 262k: 121 / 71 / 65).
smd_status Engine::plan_cell_sort() {
  uint64_t most = 1, total = 0;
  for (uint32_t r = 0; r < R; ++r) {
    most = std::max<uint64_t>(most, type0[r].size());
    total += type0[r].size();
  }
  uint32_t bits = 0;
  while ((1ull << bits) < deadKey) ++bits;
  // bins of up to 16 slices: more would read their keys over too often
  cellBinBits = std::max<uint32_t>(11, bits > 8 ? bits - 8 : 0);
  if (cellBinBits > kCellSliceBits + 4 || slotsMode) cellBinBits = 0;
  if (slotsMode || most > kCellKeys || (most > 131072 && total < 16 * most) || (R == 1 && most > 49152)) return SMD_OK;
  std::vector<uint32_t> slices(R), order(R);
  // a few systems get more slices than their lists need, to spread over the
  // CUs, up to 2M keys read
  cellMinSlices = R < 256 ? (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(256 / R, (2u << 20) / most)) : 1u;
  for (uint32_t r = 0; r < R; ++r) {
    order[r] = r;
    const uint64_t n = type0[r].size(), c = tabs[r].numBuckets;
    uint64_t k = std::max<uint64_t>((c + kCellSlice - 1) / kCellSlice, (n + kCellFill - 1) / kCellFill);
    k = std::max<uint64_t>(k, std::min<uint64_t>(cellMinSlices, (c + 63) / 64));
    if (k > 1024 || R >= (1u << (32 - kCellGroupShift))) return SMD_OK;
    slices[r] = (uint32_t)k;
  }
  // Workgroups are dealt round robin over the 8 XCDs: a replica's slices go
  // to one XCD, whose L2 then holds its keys and records (the largest
  // replicas first); a few replicas are spread.
  std::sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) {
    return type0[a].size() != type0[b].size() ? type0[a].size() > type0[b].size() : a < b;
  });
  std::vector<uint32_t> lists[8];
  for (uint32_t r : order) {
    int x = 0;
    for (int q = 1; q < 8; ++q)
      if (lists[q].size() < lists[x].size()) x = q;
    for (uint32_t k = 0; k < slices[r]; ++k) lists[R < 8 ? (x + k) % 8 : x].push_back(r << kCellGroupShift | k);
  }
  size_t longest = 0, all = 0;
  for (uint32_t r = 0; r < R; ++r) all += slices[r];
  if (all > 8192 + total / 1024) return SMD_OK;
  for (const auto& l : lists) longest = std::max(longest, l.size());
  std::vector<uint32_t> tab(8 * longest, kCellNoGroup);
  for (int x = 0; x < 8; ++x)
    for (size_t k = 0; k < lists[x].size(); ++k) tab[8 * k + x] = lists[x][k];
  HIPCHK(dalloc(&dCellGroups, tab.size()));
  HIPCHK(dalloc(&dCellSlices, R));
  HIPCHK(hipMemcpy(dCellGroups, tab.data(), tab.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dCellSlices, slices.data(), R * sizeof(uint32_t), hipMemcpyHostToDevice));
  cellGroups = (uint32_t)tab.size();
  cellGroupsN = R == 1 ? 49152 : 2 * std::max<uint64_t>(total, 4096ull * R);
  return SMD_OK;
}

// Estimates, us, fitted to single systems of 20k to 48M particles (grids of 2^6
// to 2^24 cells, uniform, in slabs and in blocks) and ensembles of 8 to 512:
// the counting form with its overfull slices against the digit passes and the
// cell table kernel, which reads 4096 cells' keys per workgroup.  Step, us,
// counted / by digits (knob 0): 100k on 2^12 cells 185 / 118, 1M on 2^14 482 /
// 274, 1M in 1/32 of the height 450 / 190, 48k so 129 / 75, 4M in a block of
// 1/64 606 / 394, 8 systems of 100k in slabs 381 / 139; where no slice is
// overfull, 100k 44 / 69, 1M 74 / 98.  The tenth keeps ties as they are.
bool Engine::digits_faster(uint32_t most, uint32_t rounds) const {
  const double m = (double)knownN / (1 << 20), spans = std::max(1.0, deadKey / 4096.0);
  const bool bins = sort_form(1) == SortForm::kCellsByBin;
  const double counted = (bins ? 20.0 + 22.0 * m : 15.0 + 11.0 * m) + 0.5 * most + rounds * (1.2 / 1024.0);
  const double passes = seg_sorted() ? 2.0 : sort_passes(keyBits, radixBits);
  const double digits = passes * (14.0 + 8.0 * m) + 8.0 + (double)knownN / spans / 2000.0;
  return counted > 1.1 * digits;
}

void Engine::restart_sort_watch() {
  digitsUntil = 0;
  digitsHold = kDigitsHold;
  sortFrom = stepsDone;
  sortSeen = false;
}

void Engine::watch_sort() {
  if (digitsUntil && stepsDone >= digitsUntil) {  // look again
    digitsUntil = 0;
    sortFrom = stepsDone;
    sortSeen = false;
  }
  if (digitsUntil || !hostSort) return;
  const unsigned long long v = __atomic_load_n(hostSort, __ATOMIC_ACQUIRE);
  if (!v || (int32_t)((uint32_t)(v >> 32) - (uint32_t)sortFrom) <= 0) return;
  if (!digits_faster((uint32_t)(v >> 16) & 0xFFFFu, ((uint32_t)v & 0xFFFFu) << 6)) return;
  if (stepsDone - sortFrom > 4 * kDigitsHold) digitsHold = kDigitsHold;  // it went well for a while
  digitsUntil = stepsDone + digitsHold;
  digitsHold = std::min<uint64_t>(2 * digitsHold, 1024 * kDigitsHold);
}

Engine::SortForm Engine::sort_form(uint32_t maxN) const {
  if (digitsUntil || !segSort || sb.algo != 1 || radixBits != 8 || maxN == 0) return SortForm::kDigits;
  // a system that has grown well past what the slices were laid out for
  // takes the bins
  // (an ensemble whose bins would hold more than 8 slices stays by replica: 512
  // grown to 14.8M particles 676 us a step, by bins 884; 256 grown to 7.7M 390 /
  // 491)
  const bool bins = cellBinBits && !(R > 1 && cellBinBits > 15);
  if (cellGroups && (knownN <= cellGroupsN || !bins)) return SortForm::kCellsByReplica;
  return cellBinBits ? SortForm::kCellsByBin : SortForm::kDigits;
}

smd_sort_form Engine::form_now() const {
  switch (sort_form((uint32_t)std::max<uint64_t>(knownN, 1))) {
    case SortForm::kCellsByReplica: return SMD_SORT_REPLICAS;
    case SortForm::kCellsByBin: return SMD_SORT_BINS;
    default: return seg_sorted() ? SMD_SORT_SEGMENTS : SMD_SORT_DIGITS;
  }
}

hipError_t Engine::sort_keys(uint32_t maxN, bool tilesLaid, StageTimer* timer, bool debug) {
  const SortForm form = sort_form(maxN);
  hipError_t e;
  if (form == SortForm::kDigits) {
    if (seg_sorted()) {
      SegSortArgs g = seg_args();
      g.tilesLaid = tilesLaid ? 1 : 0;
      e = launch_sort_seg(sb, g, dN, maxN, true, stream);
    } else {
      e = launch_sort(sb, dN, maxN, keyBits, radixBits, true, stream);
    }
    if (timer) (void)hipEventRecord(timer->ev[2], stream);
    if (e != hipSuccess) return e;
    return launch_first(sb.keys, dN, maxN, nb, dFirst, dLive, dTables, slotsMode ? slotBits : 0u, R, stream);
  }
  CellSortArgs a;
  a.tables = dTables;
  a.src = sb.gatherSrc;
  a.dN = dN;
  a.maxN = maxN;
  a.R = (int)R;
  a.segOff = dRepOff;
  a.segCount = dRepCount;
  a.segDead = dRepDeaths;
  a.bucketOff = dBucketStart;
  a.groups = dCellGroups;
  a.groupSlices = dCellSlices;
  a.minSlices = cellMinSlices;
  a.binBits = cellBinBits;
  a.slicesPerBin = 0;
  a.binTotals = nullptr;
  a.deadKey = deadKey;
  a.dLive = dLive;
  a.first = dFirst;
  a.dst = sb.gatherDst;
  a.packIndex = sb.packIndex;
  a.status = sb.status;
  a.work = dCounters + 6;
  uint32_t wg = cellGroups;
  const bool part = form == SortForm::kCellsByBin;
  if (part) {
    e = launch_sort_bins(sb, dN, maxN, (int)cellBinBits, &a.binTotals, stream);
    if (e != hipSuccess) return e;
    // twice the slices that the cells need: bins of clustered systems hold
    // more particles than the average
    a.slicesPerBin = std::max(2u, 2u * ((1u << cellBinBits) / kCellSlice));
    wg = ((deadKey + (1u << cellBinBits) - 1u) >> cellBinBits) * a.slicesPerBin;
  }
  a.keys = sb.keys;
  a.vals = sb.vals;
  a.keysOut = sb.keysAlt;
  a.valsOut = sb.valsAlt;
  e = launch_cell_sort(a, part, wg, stream);
  if (e == hipSuccess && debug)
    e = launch_cell_sort_removed(sb.keys, part ? sb.vals : nullptr, dN, maxN, deadKey, dLive, sb.keysAlt, sb.valsAlt,
                                 stream);
  std::swap(sb.keys, sb.keysAlt);
  std::swap(sb.vals, sb.valsAlt);
  if (timer) (void)hipEventRecord(timer->ev[2], stream);
  return e;
}

ProducerArgs Engine::producer_args() const {
  ProducerArgs pa;
  pa.tables = dTables;
  pa.streamReplica = dStreamReplica;
  pa.repOff = dRepOff;
  pa.repCount = dRepCount;
  pa.mtState = dMtState;
  pa.mtPar = dMtPar;
  pa.Stot = Stot;
  pa.gauss = dGauss;
  pa.ptIn = dPT[cur];
  pa.map = canon_map();
  pa.pt = dPT[cur ^ 1];
  pa.wIn = dW[cur];
  pa.w = dW[cur ^ 1];
  pa.addedPos = dAddedPos;
  pa.birthType = dBirthType;
  pa.key = sb.keys;
  pa.deadKey = deadKey;
  pa.repDeaths = dRepDeaths;
  pa.repBirths = dRepBirths;
  pa.deaths = DeathMarks{dDeadBits, dTileDead[cur]};
  pa.tileBirth = dTileBirth;
  pa.retire = dRetire;
  return pa;
}

CandArgs Engine::cand_args() const {
  CandArgs a;
  a.tables = dTables;
  a.bucketStart = dBucketStart;
  a.bucketRep = dBucketRep;
  a.repShift = repShift;
  a.R = (int)R;
  a.keys = sb.keys;
  a.sortedPT = dSortedPT;
  a.first = dFirst;
  a.dLive = dLive;
  a.cand = CandList{dCand, dCandList, dCounters + 4, dCounters + 5, dStepCount};
  return a;
}

ResolveArgs Engine::resolve_args() const {
  ResolveArgs a;
  a.tables = dTables;
  a.streamReplica = dStreamReplica;
  a.mtState = dMtState;
  a.mtPar = dMtPar;
  a.Stot = Stot;
  a.first = dFirst;
  a.cand = CandList{dCand, dCandList, dCounters + 4, dCounters + 5, dStepCount};
  a.sortedPT = dSortedPT;
  a.vals = sb.vals;
  a.packed = sb.packIndex;
  a.pt = dPT[cur ^ 1];
  a.w = dW[cur ^ 1];
  a.repDeaths = dRepDeaths;
  a.deaths = DeathMarks{dDeadBits, dTileDead[cur]};
  return a;
}

smd_status Engine::enqueue_kernels(uint32_t maxN, StageTimer* timer) {
  auto mark = [&](int stage) {
    if (timer) (void)hipEventRecord(timer->ev[stage], stream);
  };
  mark(0);
  ProducerArgs pa = producer_args();
  // the segmented sort's tile table by one more workgroup of the producer's
  // launch (it reads only the per-replica counts the step starts with)
  const bool tilesLaid = anyBim && seg_sorted() && sort_form(maxN) == SortForm::kDigits;
  if (tilesLaid) {
    pa.segTilesOn = 1;
    pa.segTiles = seg_tiles_args(seg_args(), dN, maxN, sb.status);
  }
  HIPCHK(launch_producer(pa, producerBlock, stream));
  if (anyZero) {
    ZeroArgs za;
    za.tables = dTables;
    za.R = (int)R;
    za.zMt = dZMt;
    za.zPar = dZPar;
    za.zPos = dZPos;
    za.zType = dZType;
    za.zCount = dZCount;
    za.status = dStatus;
    HIPCHK(launch_zero(za, stream));
  }
  mark(1);
  if (anyBim) {
    sb.gatherSrc = dPT[cur ^ 1];
    sb.gatherDst = dSortedPT;
    sb.gatherDeadKey = deadKey;
    sb.sizeHint = (uint32_t)std::min<uint64_t>(knownN, 0xFFFFFFFFu);
    // the sort's last pass puts each particle's index into its sorted record
    // when the gather is fused into it and every index fits
    sb.packIndex = (sb.algo == 1 && cap <= kMaxPackedIndex) ? 1 : 0;
    HIPCHK(sort_keys(maxN, tilesLaid, timer, false));
    mark(3);
    HIPCHK(launch_candidates(cand_args(), maxN, pairBlock, stream));
    mark(4);
    HIPCHK(launch_resolve(resolve_args(), stream));
    mark(5);
  } else {
    for (int s = 2; s <= 5; ++s) mark(s);
  }
  FinalizeArgs fa;
  fa.R = (int)R;
  fa.repCount = dRepCount;
  fa.repDeaths = dRepDeaths;
  fa.repBirths = dRepBirths;
  fa.newOff = dNewOff;
  fa.newCount = dNewCount;
  fa.alive = dAlive;
  fa.holeOff = dHoleOff;
  fa.holeN = dHoleN;
  fa.holes = dHoles;
  fa.extraOff = dExtraOff;
  fa.birthBase = dBirthBase;
  fa.dNnext = dNnext;
  fa.dN = dN;
  fa.deaths = pa.deaths;
  fa.tileDeadNext = dTileDead[cur ^ 1];
  fa.tileBirth = anySplit ? dTileBirth : nullptr;
  fa.tileBirthPre = dTileBirthPre;
  fa.pairCounts = anyBim ? (uint4*)(dCounters + 4) : nullptr;  // 16-byte aligned
  fa.hostSort = dHostSort;
  fa.particleSteps = dParticleSteps;
  fa.stepCount = dStepCount;
  fa.countRing = dCountRing;
  fa.ringMask = kRing - 1;
  fa.status = dStatus;
  fa.hostStatus = dHostStatus;
  fa.injCount = dInjCount;
  fa.zCount = anyZero ? dZCount : nullptr;
  fa.zeroBase = dZeroBase;
  fa.injBase = dInjBase;
  fa.retire = dRetire;
  fa.blockSum = dBlockSum;
  fa.blockTiles = finBlockTiles;
  fa.tilesCap = nTilesCap;
  HIPCHK(launch_finalize(fa, stream));
  mark(6);
  float4* const extra = dPT[cur ^ 1] + cap;
  float* const extraW = wApart ? dW[cur ^ 1] + cap : nullptr;
  if (anySplit) {
    BirthArgs ba;
    ba.R = (int)R;
    ba.dN = dN;
    ba.repOff = dRepOff;
    ba.birthBase = dBirthBase;
    ba.extraOff = dExtraOff;
    ba.tileBirthPre = dTileBirthPre;
    ba.addedPos = dAddedPos;
    ba.birthType = dBirthType;
    ba.tileBirth = dTileBirth;
    ba.blockSum = dBlockSum;
    ba.blockTiles = finBlockTiles;
    ba.extra = extra;
    ba.extraW = extraW;
    HIPCHK(launch_births(ba, maxN, stream));
  }
  if (anyZero)
    HIPCHK(launch_zero_place((int)R, dTables, dZPos, dZType, dZCount, dZeroBase, extra, extraW, stream));
  if (injN) {
    InjectArgs ia;
    ia.injPos = dInjPos;
    ia.injType = dInjType;
    ia.injRep = dInjRep;
    ia.injSrcOff = dInjSrcOff;
    ia.nInj = injN;
    ia.injBase = dInjBase;
    ia.extra = extra;
    ia.extraW = extraW;
    HIPCHK(launch_inject(ia, stream));
    injN = 0;
  }
  // every admission (empty ones too) has entered with this step
  std::fill(slotPending.begin(), slotPending.end(), (uint8_t)0);
  mark(7);
  cur ^= 1;
  std::swap(dRepOff, dNewOff);
  std::swap(dRepCount, dNewCount);
  std::swap(dN, dNnext);
  return SMD_OK;
}

smd_status Engine::step(int nsteps) {
  if (!finalized) {
    set_error("engine not finalized");
    return SMD_ERR_INVALID;
  }
  if (broken) {
    set_error("engine state was consumed by a debug stage call");
    return SMD_ERR_INVALID;
  }
  HIPCHK(hipSetDevice(device));
  if (injN && nsteps > 0) {
    // admitted particles enter through an eager step (graphs hold no injection)
    smd_status st = ensure_capacity();
    if (st != SMD_OK) return st;
    st = enqueue_step(nullptr);
    if (st != SMD_OK) return st;
    --nsteps;
  }
  if (useGraphs && nsteps >= 2) {
    smd_status st = step_graph(nsteps / 2);
    if (st != SMD_OK) return st;
    nsteps -= 2 * (nsteps / 2);
  }
  for (int s = 0; s < nsteps; ++s) {
    smd_status st = step_one();
    if (st != SMD_OK) return st;
  }
  return SMD_OK;
}

smd_status Engine::sync() {
  HIPCHK(hipSetDevice(device));
  HIPCHK(hipStreamSynchronize(stream));
  refresh_bound(false);  // the stream has drained: the last step's count is there
  return check_status();
}

// Error bits the kernels set since finalize (they stay set: the state after
// such a step is not trustworthy).
smd_status Engine::check_status() {
  if (!hostStatus) return SMD_OK;
  const uint32_t v = __atomic_load_n(hostStatus, __ATOMIC_ACQUIRE);
  if (v & kStatusZeroOverflow) {
    set_error("order-0 reactions created more particles in one step than the per-step limit");
    return SMD_ERR_CAPACITY;
  }
  if (v & kStatusSortSpin) {
    set_error("sort look-back wait exceeded its bound");
    return SMD_ERR_HIP;
  }
  if (v & kStatusSortLayout) {
    set_error("segmented sort: a destination fell outside the particle array");
    return SMD_ERR_HIP;
  }
  return SMD_OK;
}

smd_status Engine::set_knob(int knob, int value) {
  int* slot = nullptr;
  bool ok = false;
  if (knob == SMD_KNOB_PRODUCER_BLOCK) {
    slot = &producerBlock;
    ok = value == 128 || value == 256 || value == 512;
  } else if (knob == SMD_KNOB_PAIR_BLOCK) {
    slot = &pairBlock;
    ok = value == 64 || value == 128 || value == 256;
  } else if (knob == SMD_KNOB_SEGMENTED_SORT) {
    slot = &segSort;
    ok = value == 0 || value == 1;
  }
  if (!slot || !ok) {
    set_error("unknown knob or value out of range");
    return SMD_ERR_INVALID;
  }
  if (*slot != value) {
    drop_graph();  // captured launches keep the old shape
    *slot = value;
  }
  return SMD_OK;
}

// Serving layout: nSlots replicas with fixed bucket ranges (2^slotBucketBits
// each) and stream ranges (slotStreams each), all empty at first.
smd_status Engine::finalize_slots(uint32_t nSlots, uint32_t slotBucketBits, uint32_t slotStreamsMax,
                                  uint32_t capacity, uint32_t injectCap) {
  if (finalized || !tabs.empty()) {
    set_error("finalize_slots needs a fresh engine");
    return SMD_ERR_INVALID;
  }
  if (nSlots == 0 || slotBucketBits < 6 || slotBucketBits > 24 || slotStreamsMax == 0 ||
      ((uint64_t)nSlots << slotBucketBits) >= (1ull << 31)) {
    set_error("bad slot layout");
    return SMD_ERR_INVALID;
  }
  // Placeholder replicas: no particles, no streams, no reactions.
  smd_sim_spec s;
  std::memset(&s, 0, sizeof(s));
  s.num_types = 2;
  s.dt = 1.0f;
  for (int d = 0; d < 3; ++d) {
    s.box_hi[d] = 1.0f;
    s.grid_bits[d] = 2;
  }
  for (int f = 0; f < 6; ++f) s.face[f] = kReflect;
  s.num_streams = slotStreamsMax;
  for (uint32_t r = 0; r < nSlots; ++r) {
    const int id = add_replica(s, nullptr, nullptr, 0);
    if (id < 0) return (smd_status)(-id);
    tabs[r].numBuckets = 1u << slotBucketBits;  // reserve the whole range
  }
  slotsMode = true;
  slotBits = slotBucketBits;
  slotStreams = slotStreamsMax;
  injCap = injectCap;
  smd_status st = finalize(capacity);
  if (st != SMD_OK) return st;
  anySplit = true;  // jobs may create particles
  anyBim = true;
  // placeholders own no streams
  std::vector<int> none(Stot, -1);
  HIPCHK(hipMemcpy(dStreamReplica, none.data(), Stot * sizeof(int), hipMemcpyHostToDevice));
  // placeholders own no streams and no buckets (their ranges stay reserved)
  for (uint32_t r = 0; r < R; ++r) {
    tabs[r].numStreams = 0;
    tabs[r].numBuckets = 0;
  }
  HIPCHK(hipMemcpy(dTables, tabs.data(), R * sizeof(ReplicaTables), hipMemcpyHostToDevice));
  for (uint32_t** p : {&dRetire, &dInjCount, &dInjBase, &dInjSrcOff}) {
    HIPCHK(dalloc(p, R));
    HIPCHK(hipMemset(*p, 0, R * sizeof(uint32_t)));
  }
  HIPCHK(dalloc(&dInjPos, injCap));
  HIPCHK(dalloc(&dInjType, injCap));
  HIPCHK(dalloc(&dInjRep, injCap));
  slotBusy.assign(R, 0);
  slotPending.assign(R, 0);
  return SMD_OK;
}

smd_status Engine::admit(int slot, const smd_sim_spec& spec, const float* pos4, const int* types, uint32_t n) {
  if (!slotsMode || slot < 0 || (uint32_t)slot >= R) {
    set_error("admit needs a slot engine and a valid slot");
    return SMD_ERR_INVALID;
  }
  if (slotBusy[slot] || slotPending[slot]) {
    set_error("slot is occupied (retire its job first, and step once after an admission)");
    return SMD_ERR_INVALID;
  }
  if (injN + n > injCap) {
    set_error("admission exceeds the injection buffer of this step");
    return SMD_ERR_CAPACITY;
  }
  ReplicaTables T;
  std::string err;
  std::vector<smd_rxn_derived> der(spec.num_reactions > 0 ? spec.num_reactions : 1);
  if (!derive_tables(spec, T, der.data(), err)) {
    set_error(err);
    return SMD_ERR_RXN_SETUP;
  }
  if (T.numZero) {
    set_error("order-0 reactions are not supported in slot engines");
    return SMD_ERR_INVALID;
  }
  if (T.gbits[0] + T.gbits[1] + T.gbits[2] > slotBits || T.numStreams > slotStreams) {
    set_error("job grid or stream count exceeds the slot");
    return SMD_ERR_INVALID;
  }
  for (uint32_t i = 0; i < n; ++i)
    if (types[i] < 1 || types[i] >= spec.num_types) {
      set_error("particle type out of range");
      return SMD_ERR_INVALID;
    }
  smd_status st = sync();
  if (st == SMD_OK) st = take_apart(pos4, n);
  if (st != SMD_OK) return st;
  const uint32_t S = T.numStreams;
  T.bucketOff = tabs[slot].bucketOff;
  T.streamOff = tabs[slot].streamOff;
  tabs[slot] = T;
  specs[slot] = spec;
  derived[slot] = der;
  HIPCHK(hipMemcpy(dTables + slot, &T, sizeof(ReplicaTables), hipMemcpyHostToDevice));
  std::vector<int> rep(round64(slotStreams), -1);
  for (uint32_t k = 0; k < round64(S); ++k) rep[k] = slot;
  HIPCHK(hipMemcpy(dStreamReplica + T.streamOff, rep.data(), rep.size() * sizeof(int), hipMemcpyHostToDevice));
  const uint32_t* dat = mt_dat(err);
  if (!dat) {
    set_error(err);
    return SMD_ERR_IO;
  }
  std::vector<uint32_t> seeds(S), par(S);
  if (!stream_seeds(spec.seed, S, seeds.data(), err)) {
    set_error(err);
    return SMD_ERR_IO;
  }
  for (int w = 0; w < 3; ++w) {
    for (uint32_t k = 0; k < S; ++k) par[k] = dat[4 * (k % kMtParamSets) + w];
    HIPCHK(hipMemcpy(dMtPar + (size_t)w * Stot + T.streamOff, par.data(), S * sizeof(uint32_t),
                     hipMemcpyHostToDevice));
  }
  uint32_t* dSeeds = nullptr;
  HIPCHK(dalloc(&dSeeds, S));
  HIPCHK(hipMemcpy(dSeeds, seeds.data(), S * sizeof(uint32_t), hipMemcpyHostToDevice));
  HIPCHK(launch_mt_init_range(dMtState, dSeeds, Stot, T.streamOff, S, stream));
  HIPCHK(hipStreamSynchronize(stream));
  dfree(dSeeds);
  // particles enter during the next step's compaction
  if (n) {
    HIPCHK(hipMemcpy(dInjPos + injN, pos4, n * sizeof(float4), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(dInjType + injN, types, n * sizeof(int), hipMemcpyHostToDevice));
    std::vector<int> r(n, slot);
    HIPCHK(hipMemcpy(dInjRep + injN, r.data(), n * sizeof(int), hipMemcpyHostToDevice));
  }
  HIPCHK(hipMemcpy(dInjSrcOff + slot, &injN, sizeof(uint32_t), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dInjCount + slot, &n, sizeof(uint32_t), hipMemcpyHostToDevice));
  injN += n;
  Nub += n;
  slotBusy[slot] = 1;
  slotPending[slot] = 1;
  return SMD_OK;
}

smd_status Engine::retire(int slot) {
  if (!slotsMode || slot < 0 || (uint32_t)slot >= R) {
    set_error("retire needs a slot engine and a valid slot");
    return SMD_ERR_INVALID;
  }
  if (slotPending[slot]) {
    set_error("the slot's job has not entered yet (step once after an admission)");
    return SMD_ERR_INVALID;
  }
  smd_status st = sync();
  if (st != SMD_OK) return st;
  const uint32_t one = 1u;
  HIPCHK(hipMemcpy(dRetire + slot, &one, sizeof(uint32_t), hipMemcpyHostToDevice));
  slotBusy[slot] = 0;
  return SMD_OK;
}

smd_status Engine::set_particles(const float* pos4, const int* types, uint32_t n) {
  if (!finalized || R != 1) {
    set_error("set_particles needs a finalized single-replica engine");
    return SMD_ERR_INVALID;
  }
  for (uint32_t i = 0; i < n; ++i)
    if (types[i] < 1 || types[i] >= specs[0].num_types) {
      set_error("particle type out of range");
      return SMD_ERR_INVALID;
    }
  smd_status st = sync();
  if (st == SMD_OK) st = take_apart(pos4, n);
  if (st != SMD_OK) return st;
  if (step_bound(n) > cap) {
    knownN = 0;
    st = grow(4ull * n);
    if (st != SMD_OK) return st;
  }
  if (n) HIPCHK(upload_particles(pos4, types, n, dPT[cur], wApart ? dW[cur] : nullptr));
  const uint32_t off[2] = {0u, n};
  HIPCHK(hipMemcpy(dRepOff, off, 2 * sizeof(uint32_t), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dRepCount, &n, sizeof(uint32_t), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dN, &n, sizeof(uint32_t), hipMemcpyHostToDevice));
  st = set_dense();
  if (st != SMD_OK) return st;
  HIPCHK(hipStreamSynchronize(stream));
  Nub = n;
  knownN = n;
  lastSeen = stepsDone;  // counts published before this call are stale
  restart_sort_watch();
  return SMD_OK;
}

smd_status Engine::particle_steps(unsigned long long* out) {
  smd_status st = sync();
  if (st != SMD_OK) return st;
  HIPCHK(hipMemcpy(out, dParticleSteps, sizeof(unsigned long long), hipMemcpyDeviceToHost));
  return SMD_OK;
}

smd_status Engine::counts(uint32_t* out) {
  if (R && !finalized) {  // finalize failed: no count has been published
    set_error("engine not finalized");
    return SMD_ERR_INVALID;
  }
  smd_status st = sync();
  if (st != SMD_OK) return st;
  if (count_known()) {
    out[0] = (uint32_t)knownN;
    return SMD_OK;
  }
  HIPCHK(hipMemcpy(out, dRepCount, R * sizeof(uint32_t), hipMemcpyDeviceToHost));
  return SMD_OK;
}

ExportArgs Engine::export_args(int r) const {
  ExportArgs a;
  a.pt = dPT[cur];
  a.w = wApart ? dW[cur] : nullptr;
  a.map = canon_map();
  a.repOff = dRepOff;
  a.repCount = dRepCount;
  a.R = (int)R;
  a.rep = r;
  a.cap = 0xFFFFFFFFu;
  a.pos4 = nullptr;
  a.types = nullptr;
  a.header = nullptr;
  return a;
}

smd_status Engine::get(int r, float* pos4, int* types, uint32_t capN, uint32_t* nOut) {
  if (r < 0 || (uint32_t)r >= R) {
    set_error("replica id out of range");
    return SMD_ERR_INVALID;
  }
  if (!finalized) {  // finalize failed after it had set R
    set_error("engine not finalized");
    return SMD_ERR_INVALID;
  }
  std::lock_guard<std::mutex> lock(readMutex);
  const bool wants = capN && (pos4 || types);
  uint32_t n = 0;
  if (wants && lastN[r] <= stageCap) {
    // a few particles: the export kernel writes them and their number into
    // host memory, one launch and one wait
    HIPCHK(hipSetDevice(device));
    ExportArgs a = export_args(r);
    a.cap = std::min(capN, stageCap);
    a.pos4 = pos4 ? dStagePos : nullptr;
    a.types = types ? dStageType : nullptr;
    a.header = dStageHead;
    HIPCHK(launch_export(a, a.cap, stream));
    smd_status st = sync();
    if (st != SMD_OK) return st;
    n = lastN[r] = __atomic_load_n(stageHead, __ATOMIC_ACQUIRE);
    if (nOut) *nOut = n;
    const uint32_t m = std::min(n, capN);
    if (m <= stageCap) {
      if (pos4) std::memcpy(pos4, stagePos, m * sizeof(float4));
      if (types) std::memcpy(types, stageType, m * sizeof(int));
      return SMD_OK;
    }
  }
  smd_status st = sync();
  if (st != SMD_OK) return st;
  if (count_known()) n = (uint32_t)knownN;
  else HIPCHK(hipMemcpy(&n, dRepCount + r, sizeof(uint32_t), hipMemcpyDeviceToHost));
  lastN[r] = n;
  if (nOut) *nOut = n;
  const uint32_t m = std::min(n, capN);
  if (!m || !wants) return SMD_OK;
  // into memory that only steps use: the other canonical buffer and, for the
  // types, the sorted records (not the view, which its caller may still hold)
  float4* const outPos = dPT[cur ^ 1];
  int* const outType = (int*)dSortedPT;
  ExportArgs a = export_args(r);
  a.cap = m;
  a.pos4 = pos4 ? outPos : nullptr;
  a.types = types ? outType : nullptr;
  HIPCHK(launch_export(a, m, stream));
  HIPCHK(hipStreamSynchronize(stream));
  if (pos4) HIPCHK(hipMemcpy(pos4, outPos, m * sizeof(float4), hipMemcpyDeviceToHost));
  if (types) HIPCHK(hipMemcpy(types, outType, m * sizeof(int), hipMemcpyDeviceToHost));
  return SMD_OK;
}

smd_status Engine::view(float4** pos4, int** types, uint32_t* nOut) {
  if (!finalized) {
    set_error("engine not finalized");
    return SMD_ERR_INVALID;
  }
  smd_status st = sync();
  if (st != SMD_OK) return st;
  uint32_t n = 0;
  HIPCHK(hipMemcpy(&n, dN, sizeof(uint32_t), hipMemcpyDeviceToHost));
  if (n > viewCap || !dViewPos) {
    dfree(dViewPos);
    dfree(dViewType);
    viewCap = std::max<uint32_t>(n, 1u);
    HIPCHK(dalloc(&dViewPos, viewCap));
    HIPCHK(dalloc(&dViewType, viewCap));
  }
  ExportArgs a = export_args(-1);
  a.pos4 = dViewPos;
  a.types = dViewType;
  HIPCHK(launch_export(a, n, stream));
  HIPCHK(hipStreamSynchronize(stream));
  *pos4 = dViewPos;
  *types = dViewType;
  *nOut = n;
  return SMD_OK;
}

smd_status Engine::get_streams(int r, uint32_t* words, uint32_t capStreams, bool set) {
  if (r < 0 || (uint32_t)r >= R) {
    set_error("replica id out of range");
    return SMD_ERR_INVALID;
  }
  smd_status st = sync();
  if (st != SMD_OK) return st;
  const ReplicaTables& T = tabs[r];
  const uint32_t m = std::min(T.numStreams, capStreams);
  std::vector<uint32_t> buf((size_t)m);
  for (int w = 0; w < kMtWords; ++w) {
    uint32_t* dsrc = dMtState + (size_t)w * Stot + T.streamOff;
    if (set) {
      for (uint32_t k = 0; k < m; ++k) buf[k] = words[(size_t)k * kMtWords + w];
      HIPCHK(hipMemcpy(dsrc, buf.data(), m * sizeof(uint32_t), hipMemcpyHostToDevice));
    } else {
      HIPCHK(hipMemcpy(buf.data(), dsrc, m * sizeof(uint32_t), hipMemcpyDeviceToHost));
      for (uint32_t k = 0; k < m; ++k) words[(size_t)k * kMtWords + w] = buf[k];
    }
  }
  return SMD_OK;
}

smd_status Engine::debug_stage(int stage, float* pos4, int* types, uint32_t* keysSorted, uint32_t* valsSorted,
                               int* cand, uint32_t* nTotal, uint32_t* nLive) {
  if (!finalized || broken) {
    set_error("engine not usable");
    return SMD_ERR_INVALID;
  }
  HIPCHK(hipSetDevice(device));
  smd_status st = sync();
  if (st == SMD_OK) st = ensure_capacity();
  if (st != SMD_OK) return st;
  uint32_t n = 0;
  HIPCHK(hipMemcpy(&n, dN, sizeof(uint32_t), hipMemcpyDeviceToHost));
  const uint32_t maxN = n;
  broken = true;
  ProducerArgs pa = producer_args();
  pa.retire = nullptr;
  HIPCHK(launch_producer(pa, producerBlock, stream));
  uint32_t live = 0;
  if (stage >= 2) {
    sb.gatherSrc = dPT[cur ^ 1];
    sb.gatherDst = dSortedPT;
    sb.gatherDeadKey = deadKey;
    sb.sizeHint = (uint32_t)std::min<uint64_t>(knownN, 0xFFFFFFFFu);
    sb.packIndex = 0;  // the sorted values are returned
    HIPCHK(sort_keys(maxN, false, nullptr, true));
  }
  if (stage >= 3) {
    HIPCHK(launch_candidates(cand_args(), maxN, pairBlock, stream));
  }
  if (stage >= 4) HIPCHK(launch_resolve(resolve_args(), stream));
  HIPCHK(hipStreamSynchronize(stream));
  // no finalize kernel ran to copy the error bits
  uint32_t bits = 0;
  HIPCHK(hipMemcpy(&bits, dStatus, sizeof(uint32_t), hipMemcpyDeviceToHost));
  __atomic_store_n(hostStatus, bits, __ATOMIC_RELEASE);
  if (stage >= 2) HIPCHK(hipMemcpy(&live, dLive, sizeof(uint32_t), hipMemcpyDeviceToHost));
  if (nTotal) *nTotal = n;
  if (nLive) *nLive = live;
  if (n) {
    if (pos4 || types) {
      // the stage's records are dense in the other buffer
      std::vector<float4> pt(n);
      std::vector<float> w(wApart ? n : 0);
      HIPCHK(hipMemcpy(pt.data(), dPT[cur ^ 1], n * sizeof(float4), hipMemcpyDeviceToHost));
      if (wApart) HIPCHK(hipMemcpy(w.data(), dW[cur ^ 1], n * sizeof(float), hipMemcpyDeviceToHost));
      for (uint32_t i = 0; i < n; ++i) {
        uint32_t b;
        std::memcpy(&b, &pt[i].w, sizeof(b));
        // an absent product's type is -1
        const int ty = (int)(b & (uint32_t)kTypeMask);
        if (types) types[i] = ty == kTypeMask ? -1 : ty;
        b &= ~(uint32_t)kTypeMask;
        if (pos4) {
          pos4[4 * i] = pt[i].x;
          pos4[4 * i + 1] = pt[i].y;
          pos4[4 * i + 2] = pt[i].z;
          if (wApart) pos4[4 * i + 3] = w[i];
          else std::memcpy(&pos4[4 * i + 3], &b, sizeof(b));
        }
      }
    }
    if (stage == 1 && keysSorted) HIPCHK(hipMemcpy(keysSorted, sb.keys, n * sizeof(uint32_t), hipMemcpyDeviceToHost));
    if (stage >= 2 && keysSorted)
      HIPCHK(hipMemcpy(keysSorted, sb.keys, n * sizeof(uint32_t), hipMemcpyDeviceToHost));
    if (stage >= 2 && valsSorted)
      HIPCHK(hipMemcpy(valsSorted, sb.vals, n * sizeof(uint32_t), hipMemcpyDeviceToHost));
    if (stage >= 3 && cand && live) {
      std::vector<uint2> cd(live);
      uint32_t steps = 0;
      HIPCHK(hipMemcpy(cd.data(), dCand, live * sizeof(uint2), hipMemcpyDeviceToHost));
      HIPCHK(hipMemcpy(&steps, dStepCount, sizeof(uint32_t), hipMemcpyDeviceToHost));
      for (uint32_t j = 0; j < live; ++j) cand[j] = cd[j].y == steps + 1u ? (int)cd[j].x : -1;
    }
  }
  return SMD_OK;
}

smd_status Engine::profile(int nsteps, double* us, int maxStages, char* names, int namesCap, int* nStages) {
  static const char* kNames[7] = {"producer", "sort", "first", "candidates", "resolve", "finalize", "scatter"};
  if (!finalized || broken) {
    set_error("engine not usable");
    return SMD_ERR_INVALID;
  }
  HIPCHK(hipSetDevice(device));
  StageTimer tm;
  for (int k = 0; k < 8; ++k) HIPCHK(hipEventCreate(&tm.ev[k]));
  std::vector<double> acc(7, 0.0);
  for (int s = 0; s < nsteps; ++s) {
    smd_status st = ensure_capacity();
    if (st != SMD_OK) return st;
    st = enqueue_step(&tm);
    if (st != SMD_OK) return st;
    HIPCHK(hipEventSynchronize(tm.ev[7]));
    for (int k = 0; k < 7; ++k) {
      float ms = 0;
      HIPCHK(hipEventElapsedTime(&ms, tm.ev[k], tm.ev[k + 1]));
      acc[k] += ms * 1000.0;
    }
  }
  for (int k = 0; k < 8; ++k) (void)hipEventDestroy(tm.ev[k]);
  const int m = std::min(7, maxStages);
  for (int k = 0; k < m; ++k) us[k] = nsteps > 0 ? acc[k] / nsteps : 0.0;
  if (nStages) *nStages = m;
  if (names && namesCap > 0) {
    std::string s;
    for (int k = 0; k < m; ++k) {
      s += kNames[k];
      if (k + 1 < m) s += "\n";
    }
    std::strncpy(names, s.c_str(), (size_t)namesCap - 1);
    names[namesCap - 1] = 0;
  }
  return SMD_OK;
}

}  // namespace smd
