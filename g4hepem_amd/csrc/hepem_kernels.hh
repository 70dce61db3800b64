// hepem_kernels.hh -- kernels of the stepping library (one translation unit,
// included by hepem_capi.hip).
//
// The step without the process sort is two launches (the sorted forms are
// described where they stand, below):
//   k_classify  compaction of track slots by particle type into one queue:
//               e-/e+ slots fill it from the front, gamma slots from the back
//               (wave ballots and an LDS scan per tile of kClassifyTile slots,
//               one atomic per tile and kind);
//   k_step      one thread per queue entry; the e-/e+ and gamma paths are
//               therefore taken by whole waves (only the one wave that straddles
//               the boundary diverges), and the long e-/e+ blocks are dealt out
//               before the short gamma blocks.
// Every track writes only its own slot, so results do not depend on the queue
// order and are bit-identical to an unsorted pass.
#pragma once

#include <type_traits>

#include "device/dev_final.hh"
#include "device/dev_physics.hh"
#include "device/dev_soa.hh"
#include "device/dev_tracking.hh"
#include "g4hepem_amd.h"

namespace hepem {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;

// counters[0]: e-/e+ tracks, counters[1]: gammas, counters[2]: rejected tracks,
// counters[3]: 1 when the queue holds the tile-local partition (counters[4..63]
// reserved)
constexpr int kCounterWords = 64;
constexpr int kCounterLayout = 3;
__global__ void k_fill_u32(uint32_t* p, int n, uint32_t v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Each block compacts a tile of kClassifyTile consecutive slots in two
// passes over the tile: count per wave (ballot + popcount), one atomic per
// block and kind for the tile's base, then scatter. The tile keeps atomic
// traffic on the two queue counters to a few hundred operations per launch.
constexpr int kClassifyBlock = 1024;  // threads of the classification kernels
constexpr int kClassifyWaves = kClassifyBlock / 64;
constexpr int kClassifyItems = 4;
constexpr int kClassifyTile = kClassifyBlock * kClassifyItems;

// Compacts tile `tile` of a batch of n slots into its queue (e-/e+ from the
// front, gammas from the back); counters[0..1] count e-/e+ and gammas.
__device__ void ClassifyTile(int n, const int8_t* __restrict__ ptype, uint32_t* __restrict__ queue,
                             uint32_t* __restrict__ counters, int tile) {
  __shared__ uint32_t sE[kClassifyWaves], sG[kClassifyWaves], sBase[2];
  const int lane = __lane_id();
  const int wave = threadIdx.x >> 6;
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int tile0 = tile * kClassifyTile;
  uint32_t cE = 0, cG = 0;
  for (int it = 0; it < kClassifyItems; ++it) {
    const int i = tile0 + it * kClassifyBlock + threadIdx.x;
    const bool valid = i < n;
    const int8_t pt = valid ? ptype[i] : (int8_t)-1;
    const bool isE = valid && (pt == 0 || pt == 1);
    cE += (uint32_t)__popcll(__ballot(isE));
    cG += (uint32_t)__popcll(__ballot(valid && !isE));
  }
  if (lane == 0) {
    sE[wave] = cE;
    sG[wave] = cG;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tE = 0, tG = 0;
    for (int w = 0; w < kClassifyWaves; ++w) {
      const uint32_t e = sE[w], g = sG[w];
      sE[w] = tE;
      sG[w] = tG;
      tE += e;
      tG += g;
    }
    sBase[0] = tE ? atomicAdd(&counters[0], tE) : 0u;
    sBase[1] = tG ? atomicAdd(&counters[1], tG) : 0u;
  }
  __syncthreads();
  uint32_t pE = sBase[0] + sE[wave], pG = sBase[1] + sG[wave];
  for (int it = 0; it < kClassifyItems; ++it) {
    const int i = tile0 + it * kClassifyBlock + threadIdx.x;
    const bool valid = i < n;
    const int8_t pt = valid ? ptype[i] : (int8_t)-1;
    const bool isE = valid && (pt == 0 || pt == 1);
    const bool isG = valid && !isE;
    const uint64_t mE = __ballot(isE), mG = __ballot(isG);
    if (isE) queue[pE + __popcll(mE & below)] = (uint32_t)i;
    if (isG) queue[(uint32_t)n - 1u - (pG + __popcll(mG & below))] = (uint32_t)i;
    pE += (uint32_t)__popcll(mE);
    pG += (uint32_t)__popcll(mG);
  }
}

__global__ void __launch_bounds__(kClassifyBlock) k_classify(int n, const int8_t* __restrict__ ptype, uint32_t* __restrict__ queue,
                                                     uint32_t* __restrict__ counters) {
  ClassifyTile(n, ptype, queue, counters, blockIdx.x);
}

// kinds of slots a kernel steps: a queue-ordered mixed batch, or a batch of
// one kind (other slots rejected)
enum SlotKind : int { kMixed = 0, kOnlyElectrons = 1, kOnlyGammas = 2 };

// Resolves thread j of a stepping kernel to (slot, is-e-/e+); false if the
// thread has no slot or the slot does not hold a track of the batch's kind.
template <int KIND>
HD bool ResolveSlot(const hepem_tracks& t, int j, const uint32_t* queue, const uint32_t* counters, int& i, bool& isE) {
  if (KIND == kMixed) {
    i = (int)queue[j];
    isE = (uint32_t)j < counters[0];
    return true;
  }
  i = j;
  const int8_t pt = t.ptype[i];
  isE = pt == 0 || pt == 1;
  return KIND == kOnlyElectrons ? isE : pt == 2;
}

// ---- TrackElectron's sub-step loop driven by the caller (device/dev_tracking.hh) ----------------
// counters[4]: tracks that take another sub-step after the last begin/along call

// Adds the number of lanes of the wave with `pred` to *c (one atomic per wave);
// every lane of the wave must call it.
__device__ inline void CountWave(uint32_t* c, bool pred) {
  const uint64_t m = __ballot(pred);
  if (m && __lane_id() == __ffsll((unsigned long long)m) - 1) atomicAdd(c, (uint32_t)__popcll(m));
}

struct LoopIn {
  double stepLeft, truePath, meanLoss, preEkin;
  int iDProc, nsub;
  uint8_t more, stopped, left;
};
HD LoopIn LoadLoopIn(const hepem_substep_state& ss, int i) {
  LoopIn r;
  r.iDProc = ss.discrete_winner[i];
  r.stepLeft = ss.step_left[i];
  r.truePath = ss.true_path[i];
  r.meanLoss = ss.mean_eloss[i];
  r.preEkin = ss.pre_ekin[i];
  r.more = ss.more[i];
  r.stopped = ss.stopped[i];
  r.left = ss.left_world[i];
  r.nsub = ss.nsub[i];
  return r;
}
HD void KeepLoaded(LoopIn& r) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(r.stepLeft), "+v"(r.truePath), "+v"(r.meanLoss), "+v"(r.preEkin), "+v"(r.iDProc), "+v"(r.nsub));
#endif
}
template <typename R> HD void SetLoop(const LoopIn& r, StepLoop<R>& L) {
  L.iDProc = r.iDProc;
  L.stepLeft = (R)r.stepLeft;
  L.truePath = (R)r.truePath;
  L.meanLoss = r.meanLoss;
  L.preEkin = r.preEkin;
  L.preLEkin = L.preEkin > 0. ? vlog((R)L.preEkin) : (R)-30;
  L.cont = r.more != 0;
  L.stopped = r.stopped != 0;
  L.left = r.left != 0;
  L.nsub = r.nsub;
}
// The whole state of an e-/e+ slot between the calls, loaded at once (left to
// itself the compiler moves loads down to the branches that use them, and the
// wave waits for memory at each). With the active slots closed up (ActiveSlot)
// and the end's final states sorted by process, 100k e-/e+ through 27 sub-steps
// take 1.88 ms instead of 2.15: the along-step kernel 20 us instead of 32 (the
// median of its sub-steps), the MSC HowFar 10 instead of 13, the end 41 instead
// of 52.
template <typename R>
HD void LoadSubstep(const hepem_tracks& t, const hepem_howfar_state& hs, const hepem_substep_state& ss, int n, int i, uint64_t seed,
                    ElState<R>& el, StepLoop<R>& L, Rng& rng) {
  TrackIn r = LoadTrackIn(t, n, i);
  const MscIn q = LoadMscIn(t, i);
  HowFarIn h = LoadHowFarIn(hs, n, i);
  LoopIn l = LoadLoopIn(ss, i);
  KeepLoaded(r);
  KeepLoaded(h);
  KeepLoaded(l);
  InitElectron(r, q, seed, el, rng);
  SetHowFar(h, el);
  SetLoop(l, L);
}
// The block's active slots, closed up: returns the slot of this thread (of the
// block's active ones in slot order), or -1 past their number. After the first
// sub-steps few slots of a wave still are within their step, and each wave with
// one left runs its whole chain; closed up, a block's fit fewer waves.
__device__ __forceinline__ int ActiveSlot(const uint8_t* __restrict__ active, int n) {
  __shared__ uint32_t sCount[kWaves];
  __shared__ uint8_t sSlot[kBlock];
  static_assert(kBlock <= 256, "slots of a block are 8 bits");
  const int lane = __lane_id(), wave = threadIdx.x >> 6;
  const int i0 = blockIdx.x * kBlock, i = i0 + (int)threadIdx.x;
  const bool act = i < n && active[i] != 0;
  const uint64_t m = __ballot(act);
  if (lane == 0) sCount[wave] = (uint32_t)__popcll(m);
  __syncthreads();
  uint32_t before = 0u, total = 0u;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint32_t c = sCount[w];
    before += w < wave ? c : 0u;
    total += c;
  }
  if (act) sSlot[before + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint8_t)threadIdx.x;
  __syncthreads();
  return threadIdx.x < total ? i0 + (int)sSlot[threadIdx.x] : -1;
}
template <typename R> HD void StoreLoop(const hepem_substep_state& ss, int i, const StepLoop<R>& L) {
  ss.discrete_winner[i] = L.iDProc;
  ss.step_left[i] = (double)L.stepLeft;
  ss.true_path[i] = (double)L.truePath;
  ss.mean_eloss[i] = L.meanLoss;
  ss.pre_ekin[i] = L.preEkin;
  ss.more[i] = L.cont ? 1 : 0;
  ss.stopped[i] = L.stopped ? 1 : 0;
  ss.nsub[i] = L.nsub;
}

template <typename R>
__global__ void __launch_bounds__(kBlock) k_el_begin(DevTables<R> T, uint64_t seed, hepem_tracks t, hepem_howfar_state hs,
                                                     hepem_substep_state ss, uint32_t* __restrict__ counters) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = t.n;
  bool active = false;
  if (i < n) {
    const int8_t pt = t.ptype[i];
    if ((pt != 0 && pt != 1) || !TrackValid(T, t, i)) {
      atomicAdd(&counters[2], 1u);
      hs.winner[i] = -99;
      hs.geom_step[i] = 0.0;
      ss.active[i] = 0;
      ss.more[i] = 0;
    } else {
      ElState<R> el;
      Rng rng;
      InitElectron(t, n, i, seed, el, rng);
      StepLoop<R> L;
      LoopBegin(T, el, L, rng);
      StoreElectronState(t, n, i, el, rng);
      StoreElectronHowFar(hs, n, i, el);
      StoreLoop(ss, i, L);
      ss.geom_path[i] = 0.0;
#pragma unroll
      for (int c = 0; c < 3; ++c) ss.displacement[c * n + i] = 0.0;
      ss.active[i] = 1;
      ss.left_world[i] = 0;
      active = true;
    }
  }
  CountWave(&counters[4], active);
}

template <typename R>
__global__ void __launch_bounds__(kBlock) k_el_substep_howfar(DevTables<R> T, uint64_t seed, hepem_tracks t,
                                                              hepem_howfar_state hs, hepem_substep_state ss) {
  const int n = t.n;
  const int i = ActiveSlot(ss.active, n);
  if (i < 0) return;
  ElState<R> el;
  Rng rng;
  StepLoop<R> L;
  LoadSubstep(t, hs, ss, n, i, seed, el, L, rng);
  el.pstep = L.stepLeft;
  LoopMsc(T, el, L, rng);
  StoreElectronState(t, n, i, el, rng);
  StoreElectronHowFar(hs, n, i, el);
  ss.more[i] = L.cont ? 1 : 0;
  ss.nsub[i] = L.nsub;
}

template <typename R>
__global__ void __launch_bounds__(kBlock) k_el_substep_along(DevTables<R> T, uint64_t seed, hepem_tracks t,
                                                             hepem_howfar_state hs, hepem_substep_state ss,
                                                             uint32_t* __restrict__ counters) {
  const int n = t.n;
  const int i = ActiveSlot(ss.active, n);
  bool again = false;
  if (i >= 0) {
    const double path = ss.geom_path[i];
    ElState<R> el;
    Rng rng;
    StepLoop<R> L;
    LoadSubstep(t, hs, ss, n, i, seed, el, L, rng);
    ss.geom_path[i] = path + hs.geom_step[i];
    if (L.left) {
      ss.active[i] = 0;
      ss.more[i] = 0;
    } else {
      el.preEkin = el.t.ekin;
      el.preLEkin = el.t.logE();
      const bool sampled = LoopAlong(T, el, L, rng);
      StoreElectronState(t, n, i, el, rng);
      t.ekin[i] = el.t.ekin;
#pragma unroll
      for (int c = 0; c < 3; ++c) t.dir[c * n + i] = (double)el.t.dir[c];
      StoreElectronHowFar(hs, n, i, el);
      StoreLoop(ss, i, L);
#pragma unroll
      for (int c = 0; c < 3; ++c) ss.displacement[c * n + i] = sampled ? (double)el.msc.displ[c] : 0.0;
      again = L.cont;
      ss.active[i] = again ? 1 : 0;
    }
  }
  CountWave(&counters[4], again);
}

// Stage 2 of an e-/e+ slot: the final state of the chosen interaction
// (PerformDiscrete, G4HepEmElectronManager.icc:443-458).
template <typename R>
HD void ElectronInteract(const DevTables<R>& T, uint64_t seed, hepem_tracks& out, const hepem_step_out& res, int n, int i,
                         const Staged& r, uint8_t code) {
  Trk<R> t;
  Rng rng;
  Unstage(r, code, seed, t, rng);
  SecList<R> sl;
  sl.ns = 0;
  ElectronFinal(T, t, code & kCodeProc, sl, rng);
  out.ekin[i] = t.ekin;
#pragma unroll
  for (int c = 0; c < 3; ++c) out.dir[c * n + i] = (double)t.dir[c];
  StoreRng(out, i, rng);
  res.stopped[i] = t.ekin <= 0.0 ? 1 : 0;
  WriteSecondaries(res, n, i, sl);
}

// The end of a slot's step up to its final state: the code of a pending one
// (its record at st[j]), or 0.
template <typename R>
HD uint8_t EndStep(const DevTables<R>& T, uint64_t seed, hepem_tracks& t, const hepem_howfar_state& hs, hepem_substep_state& ss,
                   const hepem_step_out& res, int n, int i, Staged* st, int j) {
  ElState<R> el;
  Rng rng;
  StepLoop<R> L;
  LoadSubstep(t, hs, ss, n, i, seed, el, L, rng);
  const double path = ss.geom_path[i];
  SecList<R> sl;
  sl.ns = 0;
  const uint8_t proc = ElectronProc(T, el.t, LoopFinishSelect(T, el, L, sl, rng));
  StoreElectronState(t, n, i, el, rng);
  ss.stopped[i] = L.stopped ? 1 : 0;
  res.true_step[i] = (double)L.truePath;
  res.geom_step[i] = path;
  res.edep[i] = el.t.edep;
#pragma unroll
  for (int c = 0; c < 3; ++c) res.displacement[c * n + i] = 0.0;
  res.winner[i] = el.t.winner;
  if (proc != kPNone) {
    const double d[3] = {(double)el.t.dir[0], (double)el.t.dir[1], (double)el.t.dir[2]};
    return StageTrack(st, j, proc, el.t.isEl, el.t.imc, t.id[i], StreamHi(t, i), el.t.ekin, d, rng, 0.0);
  }
  t.ekin[i] = el.t.ekin;
#pragma unroll
  for (int c = 0; c < 3; ++c) t.dir[c * n + i] = (double)el.t.dir[c];
  res.stopped[i] = el.t.ekin <= 0.0 ? 1 : 0;
  WriteSecondaries(res, n, i, sl);
  return kPNone;
}

template <typename R>
__global__ void __launch_bounds__(kBlock) k_el_end(DevTables<R> T, uint64_t seed, hepem_tracks t, hepem_howfar_state hs,
                                                   hepem_substep_state ss, hepem_step_out res) {
  __shared__ BlockFinals<kBlock> fin;
  const int i0 = blockIdx.x * kBlock, i = i0 + (int)threadIdx.x;
  const int n = t.n;
  uint8_t code = kPNone;
  if (i < n) {
    const int8_t pt = t.ptype[i];
    if ((pt != 0 && pt != 1) || hs.winner[i] == -99) WriteRejected<R>(t, t, res, n, i);
    else code = EndStep(T, seed, t, hs, ss, res, n, i, fin.st, (int)threadIdx.x);
  }
  SampleBlock<kBlock, kPIoniEl, kPAnnih>(fin, code, [&](int j, const Staged& r, uint8_t c, int) {
    ElectronInteract<R>(T, seed, t, res, n, i0 + j, r, c);
  });
}

// ---- two-stage step: particle sort, then process sort ----------------------------------------
// (the FP32-table form and the smaller FP64 batches take the step in one launch
// instead: k_step_block)
// k_step_select_local does HowFar, the continuous step and the choice of the
// discrete interaction (one thread per particle-queue entry), records the chosen process
// per slot and, for a pending interaction, the 64-byte record of what the
// final-state sampling needs (at the slot: one line per track instead of ten
// scattered fields); k_classify_tiles orders each tile's pending slots by
// process; k_interact_tiles samples the final states, so each wave runs one
// sampler. (The batched step does the same over the tiles of all its batches,
// k_classify_tiles_batched and k_interact_tiles_batched.)

// Stage 1 of an e-/e+ slot after its HowFar: the continuous step and
// PerformDiscrete's choice (G4HepEmElectronManager.icc:425-441,461-483).
// Returns the slot code; a complete step (kPNone) also gets its post-step
// kinematics, secondaries and stopped flag here, a pending one its staged
// record at st[j].
//
// Every field is stored as soon as it is final, not at the end: the MSC state,
// the interaction lengths and the mean free paths would otherwise hold about 30
// VGPRs through the MSC and fluctuation sampling. Of the interaction lengths
// the winner's alone waits (a discrete interaction resets it). Measured: the
// split Perform's first stage 164 -> 122 VGPRs (4 waves per SIMD instead of 3;
// 118 by now), the step's 140 -> 135, and held to 128 it runs 4 waves too (by
// now 125 and nothing spills: ArgsView): 3M ordered tracks 765 us instead of
// 800, 300k split calls 162 instead of 169, 1M mixed tracks 314 instead of 318.
template <typename R>
HD uint8_t ElectronSelectAfterHowFar(const DevTables<R>& T, ElState<R>& el, Rng& rng, const hepem_tracks& in,
                                     hepem_tracks& out, const hepem_step_out& res, int n, int i, Staged* st, int j) {
  Trk<R>& t = el.t;
  const int winner = t.winner;
  {
    const Msc<R>& m = el.msc;
    out.msc_init_range[i] = (double)m.initRange;
    out.msc_dyn_range_factor[i] = (double)m.dynRangeFactor;
    out.msc_tlimit_min[i] = (double)m.tlimitMin;
    out.msc_first_step[i] = m.firstStep ? 1 : 0;
    res.geom_step[i] = (double)t.gstep;
    res.winner[i] = winner;
  }
  const ContStep go = ElectronBeginContinuous(el);
  res.true_step[i] = (double)el.pstep;
  const R winnerLeft = PickMFP(t.nial, winner), winnerMfp = PickMFP(t.mfp, winner);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k != winner) out.num_ia_left[k * n + i] = (double)t.nial[k];
  // the direction is not needed before the scattering turns it: loaded here, it
  // holds no registers through HowFar
#pragma unroll
  for (int c = 0; c < 3; ++c) t.dir[c] = (R)in.dir[c * n + i];
  bool stopped = false;
  if (go == kMoved) {
    stopped = ApplyMeanEnergyLoss(T, el);
    if (!stopped) SampleMSC(T, el, rng);
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) res.displacement[c * n + i] = (double)el.msc.displ[c];
  if (go == kMoved && !stopped) stopped = SampleLossFluctuations(T, el, rng);
  res.edep[i] = t.edep;
  const bool discrete = winner >= 0 && go != kNoMove && !stopped && !t.onBoundary;
  if (winner >= 0) out.num_ia_left[winner * n + i] = discrete ? -1.0 : (double)winnerLeft;
  SecList<R> sl;
  sl.ns = 0;
  uint8_t proc = kPNone;
  if (stopped) {
    if (!t.isEl) AnnihilateAtRest(sl, rng);
  } else if (discrete && !CheckDelta(T, t, winnerMfp, (R)rng.flat())) {
    proc = ElectronProc(T, t, winner);
  }
  if (proc != kPNone) {
    const double d[3] = {(double)t.dir[0], (double)t.dir[1], (double)t.dir[2]};
    return StageTrack(st, j, proc, t.isEl, t.imc, in.id[i], StreamHi(in, i), t.ekin, d, rng, 0.0);
  }
  out.ekin[i] = t.ekin;
#pragma unroll
  for (int c = 0; c < 3; ++c) out.dir[c * n + i] = (double)t.dir[c];
  StoreRng(out, i, rng);
  res.stopped[i] = t.ekin <= 0.0 ? 1 : 0;
  WriteSecondaries(res, n, i, sl);
  return kPNone;
}

// Stage 1 of an e-/e+ slot of the split Perform: the HowFar state comes from
// the hand-over (with the caller's geometrical step).
template <typename R>
HD uint8_t PerformElectronSelect(const DevTables<R>& T, uint64_t seed, hepem_tracks& t, const hepem_howfar_state& hs,
                                 const hepem_step_out& res, Staged* st, int n, int i) {
  ElState<R> el;
  Rng rng;
  InitElectron(t, n, i, seed, el, rng);
  LoadElectronHowFar(hs, n, i, el);
  return ElectronSelectAfterHowFar(T, el, rng, t, t, res, n, i, st, i);
}

// Stage 1 of a gamma slot after its HowFar: SelectInteraction and the
// interaction-length update of Perform, or only that update on a boundary
// (G4HepEmGammaManager.icc:54-62,173-219; G4HepEmTrackingManager.cc:1092-1108).
template <typename R>
HD uint8_t GammaSelectAfterHowFar(const DevTables<R>& T, Trk<R>& t, R pe, Rng& rng, const hepem_tracks& in,
                                  hepem_tracks& out, const hepem_step_out& res, int n, int i, Staged* st, int j) {
  const uint8_t proc = GammaProc(T, t, pe, rng);
#pragma unroll
  for (int k = 0; k < 4; ++k) out.num_ia_left[k * n + i] = (double)t.nial[k];
  res.true_step[i] = (double)t.gstep;
  res.geom_step[i] = (double)t.gstep;
#pragma unroll
  for (int c = 0; c < 3; ++c) res.displacement[c * n + i] = 0.0;
  res.winner[i] = t.winner;
  if (proc != kPNone) {
    const double d[3] = {(double)t.dir[0], (double)t.dir[1], (double)t.dir[2]};
    return StageTrack(st, j, proc, false, t.imc, in.id[i], StreamHi(in, i), t.ekin, d, rng, (double)pe);
  }
  out.ekin[i] = t.ekin;
#pragma unroll
  for (int c = 0; c < 3; ++c) out.dir[c * n + i] = (double)t.dir[c];
  StoreRng(out, i, rng);
  res.edep[i] = t.edep;
  res.stopped[i] = t.ekin <= 0.0 ? 1 : 0;
  SecList<R> sl;
  sl.ns = 0;
  WriteSecondaries(res, n, i, sl);
  return kPNone;
}

// What stage 1 of the step works on.
template <typename R> struct StepView {
  const DevTables<R>& T;
  uint64_t seed;
  const hepem_tracks& in;
  hepem_tracks& out;
  const hepem_step_out& res;
  uint32_t* counters;
};

// Stage 1 of slot i of the step: its whole state loaded at once, the test of
// its couple and energy, the identity copy, HowFar and the selection. Returns
// the slot's code; a pending slot's record goes to st[j]. view() gives the
// StepView; it is asked for again after HowFar.
template <typename R, typename V> HD uint8_t StepSelect(V view, int n, int i, bool isE, Staged* st, int j) {
  const StepView<R> v = view();
  TrackIn r = LoadTrackIn(v.in, n, i);
  MscIn q{};
  if (isE) q = LoadMscIn(v.in, i);
  KeepLoaded(r);
  if (!TrackValid(v.T, r.imc, r.ekin)) {
    atomicAdd(&v.counters[2], 1u);
    WriteRejected<R>(v.in, v.out, v.res, n, i);
    return kPNone;
  }
  StoreIdentity(v.in, v.out, i, r);
  Rng rng;
  if (isE) {
    ElState<R> el;
    InitElectron(r, q, v.seed, el, rng);
    ElectronHowFar(v.T, el, rng);
    const StepView<R> w = view();
    return ElectronSelectAfterHowFar(w.T, el, rng, w.in, w.out, w.res, n, i, st, j);
  }
  Trk<R> t;
  t.isEl = false;
  InitTrack(r, t);
  InitRng(r, v.seed, rng);
  const R pe = GammaHowFar(v.T, t, rng);
  const StepView<R> w = view();
  return GammaSelectAfterHowFar(w.T, t, pe, rng, w.in, w.out, w.res, n, i, st, j);
}

// Stage 1 of a gamma slot of the split Perform: step, mean free path and PE
// cross section from the hand-over.
template <typename R>
HD uint8_t PerformGammaSelect(const DevTables<R>& T, uint64_t seed, hepem_tracks& t, const hepem_howfar_state& hs,
                              const hepem_step_out& res, Staged* st, int n, int i) {
  Trk<R> g;
  g.isEl = false;
  LoadTrack(t, n, i, g);
  g.gstep = (R)hs.geom_step[i];
  g.mfp[0] = (R)hs.mfp[i];
  Rng rng;
  rng.init(seed, (uint32_t)t.id[i], StreamHi(t, i), t.rng_ctr[i], t.rng_has_gauss[i] != 0, t.rng_gauss[i]);
  return GammaSelectAfterHowFar(T, g, (R)hs.pe_xsec[i], rng, t, t, res, n, i, st, i);
}

// Stage 2 of a gamma slot: the interaction and the gamma tracking cut of
// G4HepEmGammaManager::Perform (G4HepEmGammaManager.icc:63-93).
template <typename R>
HD void GammaInteract(const DevTables<R>& T, uint64_t seed, hepem_tracks& out, const hepem_step_out& res, int n, int i,
                      const Staged& r, uint8_t code) {
  Trk<R> t;
  Rng rng;
  Unstage(r, code, seed, t, rng);
  SecList<R> sl;
  sl.ns = 0;
  GammaFinal(T, t, code & kCodeProc, (R)r.pe, sl, rng);
  out.ekin[i] = t.ekin;
#pragma unroll
  for (int c = 0; c < 3; ++c) out.dir[c * n + i] = (double)t.dir[c];
  StoreRng(out, i, rng);
  res.edep[i] = t.edep;
  res.stopped[i] = t.ekin <= 0.0 ? 1 : 0;
  WriteSecondaries(res, n, i, sl);
}

// Process sort and final states, tile by tile (the single-batch two-stage
// step and Perform).
//
// k_classify_tiles lays the pending slots of each tile of kClassifyTile
// slots out process by process, within the tile's own range of `tlist` (tile
// offsets, 16 bits), and writes the tile's process offsets and chunk counts
// to `tinfo` (packed scans over a wave and over the waves' totals; no atomics, so
// the layout is deterministic).
//
// k_interact_tiles gives each wave one chunk of up to 64 entries of one
// process. A tile's chunks are spread over kInteractParts blocks that go to
// the same XCD one after another (blocks are dealt to the XCDs round-robin),
// so all final-state writes to the tile's cache lines come from one XCD
// within a short time and its L2 merges them into whole lines before they go
// to HBM. With a global process-sorted queue each wave's writes land a few
// slots per line and reach HBM as partial lines.
constexpr int kXcds = 8;
constexpr int kTileInfo = 2 * (kNumProc + 1);   // per tile: process offsets, first chunks
constexpr int kInteractWaves = kBlock / 64;
// blocks of a tile of `items` * kClassifyBlock slots: at most one chunk per 64
// slots plus one partial chunk per process, kInteractWaves chunks per block
constexpr int InteractParts(int items) { return (items * kClassifyBlock / 64 + kNumProc + kInteractWaves - 1) / kInteractWaves; }
constexpr int kInteractParts = InteractParts(kClassifyItems);

inline int InteractGridTiles(int tiles, int parts = kInteractParts) { return (tiles + kXcds - 1) / kXcds * kXcds * parts; }
inline int InteractGrid(int n) { return InteractGridTiles((n + kClassifyTile - 1) / kClassifyTile); }

// Tile-local particle partition of tile `tile` of a batch of n slots: the
// tile's e-/e+ slots first, then its gammas, each in slot order, at the
// tile's own range of the batch's queue; *ecount = the tile's e-/e+ count.
// One kClassifyBlock-thread block per tile, kClassifyItems consecutive slots
// per thread, read once. Bound by the latency of its few dependent stages, not
// by its bytes: one scan over the wave's e-/e+ counts and one over the waves'
// (each wave sums the waves before it by itself) take the place of ballots
// per item, a second read of the types and a serial scan by one thread.
__device__ void ClassifyLocalTile(int n, const int8_t* __restrict__ ptype, uint32_t* __restrict__ queue, int tile,
                                  uint32_t* __restrict__ ecount) {
  __shared__ uint32_t sE[kClassifyWaves];
  const int lane = __lane_id();
  const int wave = threadIdx.x >> 6;
  const int tile0 = tile * kClassifyTile;
  const int first = tile0 + (int)threadIdx.x * kClassifyItems;
  uint32_t mask = 0u, cE = 0u;  // the thread's e-/e+ slots and their number
#pragma unroll
  for (int k = 0; k < kClassifyItems; ++k) {
    const int8_t pt = first + k < n ? ptype[first + k] : (int8_t)-1;
    const bool isE = pt == 0 || pt == 1;
    mask |= isE ? 1u << k : 0u;
    cE += isE ? 1u : 0u;
  }
  uint32_t x = cE;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(x, o, 64);
    if (lane >= o) x += u;
  }
  if (lane == 63) sE[wave] = x;
  __syncthreads();
  uint32_t before = 0u, total = 0u;
#pragma unroll
  for (int w = 0; w < kClassifyWaves; ++w) {
    const uint32_t e = sE[w];
    before += w < wave ? e : 0u;
    total += e;
  }
  if (threadIdx.x == 0) *ecount = total;
  uint32_t pE = before + x - cE;                                     // e-/e+ of the tile before the thread's slots
  uint32_t pG = total + threadIdx.x * (uint32_t)kClassifyItems - pE;  // first entry of its gammas
#pragma unroll
  for (int k = 0; k < kClassifyItems; ++k) {
    if (first + k < n) {
      const bool isE = ((mask >> k) & 1u) != 0u;
      queue[tile0 + (isE ? pE : pG)] = (uint32_t)(first + k);
      pE += isE ? 1u : 0u;
      pG += isE ? 0u : 1u;
    }
  }
}

// The tile-local particle partition of one batch, one block per tile, with
// tinfo[tile * kTileInfo] = the tile's e-/e+ count. The first block also
// clears the step's counters and marks the layout in counters[kCounterLayout]
// (no counter is read before the next kernel).
__global__ void __launch_bounds__(kClassifyBlock) k_classify_local(int n, const int8_t* __restrict__ ptype,
                                                                   uint32_t* __restrict__ queue, uint32_t* __restrict__ tinfo,
                                                                   uint32_t* __restrict__ counters) {
  if (blockIdx.x == 0 && threadIdx.x < kCounterWords) counters[threadIdx.x] = threadIdx.x == kCounterLayout ? 1u : 0u;
  ClassifyLocalTile(n, ptype, queue, (int)blockIdx.x, tinfo + (size_t)blockIdx.x * kTileInfo);
}

constexpr int kTileChunks = kClassifyTile / kBlock;
// tiles at the end of each XCD's share whose second halves (mostly gammas,
// short) run after all their first halves (mostly e-/e+, long)
constexpr int kTailTiles = 8;
static_assert(kTileChunks % 2 == 0, "a tile splits into two halves of whole blocks");
inline int LocalSelectGridTiles(int ntiles) { return (ntiles + kXcds - 1) / kXcds * kXcds * kTileChunks; }
inline int LocalSelectGrid(int n) { return LocalSelectGridTiles((n + kClassifyTile - 1) / kClassifyTile); }

// Block -> (tile, chunk of kBlock slots) of stage 1 over the tile-local
// particle partition of ntiles tiles: XCD x takes tiles x, x + kXcds, ...,
// each as kTileChunks consecutive blocks of its share, so a tile's e-/e+ and
// gamma blocks run on one XCD close together and its lines are read and
// written through one L2. In the last kTailTiles tiles of a share the blocks
// of the first halves come first, then those of the second halves, so the
// launch ends on short gamma blocks rather than on long e-/e+ ones. False for
// the blocks of a grid of LocalSelectGridTiles(ntiles) that have no chunk.
__device__ inline bool LocalSelectChunk(int ntiles, int& tile, int& chunk) {
  const int x = blockIdx.x % kXcds, q = blockIdx.x / kXcds;
  const int share = ntiles > x ? (ntiles - x + kXcds - 1) / kXcds : 0;
  const int tail = min(kTailTiles, share), body = (share - tail) * kTileChunks;
  int k;
  if (q < body) {
    k = q / kTileChunks;
    chunk = q % kTileChunks;
  } else {
    const int r = q - body, h = kTileChunks / 2;
    if (r >= tail * kTileChunks) return false;
    const bool first = r < tail * h;
    const int r2 = first ? r : r - tail * h;
    k = share - tail + r2 / h;
    chunk = (first ? 0 : h) + r2 % h;
  }
  tile = k * kXcds + x;
  return true;
}

// The arguments of the step's kernels.
template <typename R> struct StepArgs {
  DevTables<R> T;
  uint64_t seed;
  hepem_tracks in, out;
  hepem_step_out res;
  const uint32_t* queue;
  uint32_t* counters;
  const uint32_t* tinfo;
  uint8_t* code;   // of the two-stage step
  Staged* st;
};
// The StepView of a kernel that takes one StepArgs. Read anew after HowFar, the
// arguments leave k_step_select_local 125 VGPRs and no spills (128 and 10 with
// them held: 1M tracks 288 us instead of 294, 3M ordered 681 instead of 699) and
// the FP32-table form of k_step_block 97 instead of 119.
template <typename R> HD StepView<R> ArgsView() {
  const StepArgs<R>& a = KernelArgs<StepArgs<R>>();
  return {a.T, a.seed, a.in, const_cast<hepem_tracks&>(a.out), a.res, a.counters};
}
// The slot of this thread in a grid of LocalSelectGrid(n) blocks and whether it
// holds an e-/e+, in the layout hepem_step_prepare chose (tile-local, or e-/e+
// first over the batch); -1 without a slot. `none`: so is the whole block.
template <typename R> __device__ __forceinline__ int StepSlot(bool& isE, bool& none) {
  const StepArgs<R>& a = KernelArgs<StepArgs<R>>();
  const int n = a.in.n;
  int tile, chunk;
  none = true;
  if (!LocalSelectChunk((n + kClassifyTile - 1) / kClassifyTile, tile, chunk)) return -1;
  const int tile0 = tile * kClassifyTile;
  const int m = min(kClassifyTile, n - tile0);
  none = chunk * kBlock >= m;
  const int jl = chunk * kBlock + (int)threadIdx.x;
  if (jl >= m) return -1;
  isE = a.counters[kCounterLayout] ? jl < (int)a.tinfo[(size_t)tile * kTileInfo] : (uint32_t)(tile0 + jl) < a.counters[0];
  return (int)a.queue[tile0 + jl];
}

// Stage 1 of the step over one batch's particle queue, its blocks placed tile by
// tile as LocalSelectChunk places them (the tile-local partition that
// hepem_step_prepare lays out with the process sort; a queue laid out over the
// whole batch is read correctly too).
template <typename R> __global__ void __launch_bounds__(kBlock, 4) k_step_select_local(StepArgs<R>) {
  bool isE = false, none;
  const int i = StepSlot<R>(isE, none);
  if (i < 0) return;
  const uint8_t c = StepSelect<R>([]() HEPEM_INLINE { return ArgsView<R>(); }, KernelArgs<StepArgs<R>>().in.n, i, isE,
                                  KernelArgs<StepArgs<R>>().st, i);
  KernelArgs<StepArgs<R>>().code[i] = c;
}
static_assert(std::is_same_v<decltype(k_step_select_local<double>), void(StepArgs<double>)>);

// The whole step in one launch: stage 1 as k_step_select_local, then the final
// states of the block's pending slots, sorted by process within the block.
//
// Bound by the latency of one wave's chain in a small batch, by VALU issue in a
// large one. Against the three launches of the two-stage step it keeps the
// pending state in LDS instead of 130 bytes a slot through memory and runs the
// chain of a track in one go; the two-stage step fills the waves of the final
// states better and, in FP64, has 4 waves per SIMD (this kernel 3: held to 4 it
// spills and 1M tracks take 320 us). The FP32-table form runs 5 waves per SIMD
// (4 VGPRs spilled; left alone it takes 97 VGPRs, 4 waves, and 1M tracks 243 us)
// and is faster at every size: 16k ordered tracks 44.5 us instead of 50, 1M
// mixed 225 instead of 260, 3M 588 instead of 756. FP64 up to one resident
// round: 131k 66 instead of 78; 1M 309 against 294 (StepsInOneLaunch has both
// sides of the line).
template <typename R> constexpr int kStepBlockWaves = sizeof(R) == sizeof(double) ? 3 : 5;
template <typename R>
__global__ void __launch_bounds__(kBlock, kStepBlockWaves<R>) k_step_block(StepArgs<R>) {
  __shared__ BlockFinals<kBlock> fin;
  __shared__ int32_t slot[kBlock];
  uint8_t code = kPNone;
  bool isE = false, none;
  const int i = StepSlot<R>(isE, none);
  if (none) return;  // the whole block
  slot[threadIdx.x] = i;
  if (i >= 0)
    code = StepSelect<R>([]() HEPEM_INLINE { return ArgsView<R>(); }, KernelArgs<StepArgs<R>>().in.n, i, isE, fin.st, (int)threadIdx.x);
  SampleBlock<kBlock, kPIoniEl, kPPE>(fin, code, [&](int j, const Staged& r, uint8_t c, int proc) HEPEM_INLINE {
    const StepArgs<R>& a = KernelArgs<StepArgs<R>>();
    hepem_tracks& out = const_cast<hepem_tracks&>(a.out);
    if (proc < kPConv) ElectronInteract<R>(a.T, a.seed, out, a.res, a.in.n, slot[j], r, c);
    else GammaInteract<R>(a.T, a.seed, out, a.res, a.in.n, slot[j], r, c);
  });
}
static_assert(std::is_same_v<decltype(k_step_block<double>), void(StepArgs<double>)>);

// Thread -> (slot, is-e-/e+) of the split HowFar and Perform kernels. A
// mixed batch's queue is read in the layout its hepem_howfar prepare chose
// (counters[kCounterLayout]): tile-local, with the blocks placed as
// k_step_select_local places them (grid LocalSelectGrid(n)), or e-/e+ first
// over the batch (one thread per entry). False if the thread has no slot;
// kindOk false if the slot holds a track of the other kind.
template <int KIND>
__device__ inline bool ThreadSlot(const hepem_tracks& t, const uint32_t* __restrict__ queue,
                                  const uint32_t* __restrict__ counters, const uint32_t* __restrict__ tinfo, int& i,
                                  bool& isE, bool& kindOk) {
  const int n = t.n;
  if (KIND == kMixed && counters[kCounterLayout]) {
    int tile, chunk;
    if (!LocalSelectChunk((n + kClassifyTile - 1) / kClassifyTile, tile, chunk)) return false;
    const int tile0 = tile * kClassifyTile, jl = chunk * kBlock + (int)threadIdx.x;
    if (tile0 + jl >= n) return false;
    i = (int)queue[tile0 + jl];
    isE = jl < (int)tinfo[(size_t)tile * kTileInfo];
    kindOk = true;
    return true;
  }
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return false;
  kindOk = ResolveSlot<KIND>(t, j, queue, counters, i, isE);
  return true;
}

template <typename R, int KIND>
__global__ void __launch_bounds__(kBlock, 4) k_howfar(DevTables<R> T, uint64_t seed, hepem_tracks t, hepem_howfar_state hs,
                                                   const uint32_t* __restrict__ queue, uint32_t* __restrict__ counters,
                                                   const uint32_t* __restrict__ tinfo) {
  const int n = t.n;
  int i;
  bool isE, kindOk;
  if (!ThreadSlot<KIND>(t, queue, counters, tinfo, i, isE, kindOk)) return;
  if (!kindOk || !TrackValid(T, t, i)) {
    atomicAdd(&counters[2], 1u);
    hs.winner[i] = -99;
    hs.geom_step[i] = 0.0;
    return;
  }
  if (isE) {
    ElState<R> el;
    Rng rng;
    InitElectron(t, n, i, seed, el, rng);
    ElectronHowFar(T, el, rng);
    StoreElectronState(t, n, i, el, rng);
    StoreElectronHowFar(hs, n, i, el);
  } else {
    Trk<R> g;
    g.isEl = false;
    LoadTrack(t, n, i, g);
    Rng rng;
    rng.init(seed, (uint32_t)t.id[i], StreamHi(t, i), t.rng_ctr[i], t.rng_has_gauss[i] != 0, t.rng_gauss[i]);
    const R pe = GammaHowFar(T, g, rng);
#pragma unroll
    for (int k = 0; k < 4; ++k) t.num_ia_left[k * n + i] = (double)g.nial[k];
    StoreRng(t, i, rng);
    hs.geom_step[i] = (double)g.gstep;
    hs.mfp[i] = (double)g.mfp[0];
    hs.winner[i] = g.winner;
    hs.pe_xsec[i] = (double)pe;
  }
}

template <typename R, int KIND>
__global__ void __launch_bounds__(kBlock, 3) k_perform(DevTables<R> T, uint64_t seed, hepem_tracks t, hepem_howfar_state hs,
                                                    hepem_step_out res, const uint32_t* __restrict__ queue,
                                                    uint32_t* __restrict__ counters, const uint32_t* __restrict__ tinfo) {
  const int n = t.n;
  int i;
  bool isE, kindOk;
  if (!ThreadSlot<KIND>(t, queue, counters, tinfo, i, isE, kindOk)) return;
  if (!kindOk || hs.winner[i] == -99) {
    WriteRejected<R>(t, t, res, n, i);
    return;
  }
  SecList<R> sl;
  sl.ns = 0;
  if (isE) {
    ElState<R> el;
    Rng rng;
    InitElectron(t, n, i, seed, el, rng);
    LoadElectronHowFar(hs, n, i, el);
    ElectronPerform(T, el, sl, rng);
    StoreElectronState(t, n, i, el, rng);
    StoreElectronResult(t, res, n, i, el, sl);
  } else {
    Trk<R> g;
    g.isEl = false;
    LoadTrack(t, n, i, g);
    g.gstep = (R)hs.geom_step[i];
    g.mfp[0] = (R)hs.mfp[i];
    Rng rng;
    rng.init(seed, (uint32_t)t.id[i], StreamHi(t, i), t.rng_ctr[i], t.rng_has_gauss[i] != 0, t.rng_gauss[i]);
    GammaPerform(T, g, (R)hs.pe_xsec[i], sl, rng);
    StoreGamma(t, res, n, i, g, sl, rng);
  }
}

// Stage 1 of the split Perform (as k_perform up to the choice of the
// interaction).
template <typename R, int KIND>
__global__ void __launch_bounds__(kBlock) k_perform_select(DevTables<R> T, uint64_t seed, hepem_tracks t,
                                                           hepem_howfar_state hs, hepem_step_out res,
                                                           const uint32_t* __restrict__ queue, uint32_t* __restrict__ counters,
                                                           const uint32_t* __restrict__ tinfo, uint8_t* __restrict__ code,
                                                           Staged* __restrict__ st) {
  const int n = t.n;
  int i;
  bool isE, kindOk;
  if (!ThreadSlot<KIND>(t, queue, counters, tinfo, i, isE, kindOk)) return;
  if (!kindOk || hs.winner[i] == -99) {
    WriteRejected<R>(t, t, res, n, i);
    code[i] = kPNone;
    return;
  }
  code[i] = isE ? PerformElectronSelect<R>(T, seed, t, hs, res, st, n, i) : PerformGammaSelect<R>(T, seed, t, hs, res, st, n, i);
}

// The fused step over either particle layout of the queue (the one
// hepem_step_prepare chose, as counters[kCounterLayout] records): e-/e+ are
// the first counters[0] entries, or the first tinfo[tile * kTileInfo] entries
// of each tile.
template <typename R>
__global__ void __launch_bounds__(kBlock) k_step(DevTables<R> T, uint64_t seed, hepem_tracks in, hepem_tracks out,
                                                 hepem_step_out res, const uint32_t* __restrict__ queue,
                                                 uint32_t* __restrict__ counters, const uint32_t* __restrict__ tinfo) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = in.n;
  if (j >= n) return;
  const bool isE = counters[kCounterLayout] ? j % kClassifyTile < (int)tinfo[(size_t)(j / kClassifyTile) * kTileInfo]
                                            : (uint32_t)j < counters[0];
  const int i = (int)queue[j];
  if (RejectTrack(T, in, out, res, n, i, counters)) return;
  CopyIdentity(in, out, i);
  if (isE) StepElectron(T, seed, in, out, res, n, i);
  else StepGamma(T, seed, in, out, res, n, i);
}

// the process layout of tile `tile` of a batch of n slots (codes, tile list
// and the tile's info words of that batch); a tile is ITEMS * kClassifyBlock
// slots, ITEMS consecutive ones per thread; entries are in slot order within
// their process.
//
// Bound by latency (one block per tile, a few dependent stages): a thread
// counts its slots in eight 16-bit fields, one packed scan over the wave and
// one over the waves' totals, in (process, wave) order by the lanes of one
// wave, give every entry its place. One thread scanning 128 totals in turn
// after two rounds of 32 ballots took 15.4 us for a batch of one tile and
// 8.7 us for 1M slots.
template <int ITEMS = kClassifyItems>
__device__ void ClassifyTileLayout(int n, const uint8_t* __restrict__ code, uint16_t* __restrict__ tlist,
                                   uint32_t* __restrict__ info, int tile) {
  static_assert(ITEMS * kClassifyBlock <= 65536, "tile-local offsets are 16 bits");
  static_assert(kNumProc == 8 && kClassifyWaves == 16 && 64 * ITEMS < 65536, "eight 16-bit fields; 64 lanes hold 2 waves each per process");
  __shared__ uint64_t sTot[kClassifyWaves][2];
  __shared__ uint32_t sOff[kNumProc][kClassifyWaves];
  const int lane = __lane_id();
  const int wave = threadIdx.x >> 6;
  const int tile0 = tile * ITEMS * kClassifyBlock;
  const int first = (int)threadIdx.x * ITEMS;
  int c[ITEMS];
  uint64_t lo = 0, hi = 0;  // counts of processes 1..4 and 5..8
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int i = tile0 + first + k;
    c[k] = i < n ? (int)(code[i] & kCodeProc) : 0;
    const uint64_t one = 1ull << (16 * ((c[k] - 1) & 3));
    lo += c[k] >= 1 && c[k] <= 4 ? one : 0ull;
    hi += c[k] > 4 ? one : 0ull;
  }
  uint64_t xl = lo, xh = hi;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t ul = __shfl_up(xl, o, 64), uh = __shfl_up(xh, o, 64);
    xl += lane >= o ? ul : 0ull;
    xh += lane >= o ? uh : 0ull;
  }
  if (lane == 63) {
    sTot[wave][0] = xl;
    sTot[wave][1] = xh;
  }
  __syncthreads();
  if (wave == 0) {
    // lane 8q + j: the totals of process q in waves 2j and 2j + 1
    const int q = lane >> 3, w = 2 * (lane & 7), sh = 16 * (q & 3);
    const uint32_t t0 = (uint32_t)(sTot[w][q >> 2] >> sh) & 0xFFFFu, t1 = (uint32_t)(sTot[w + 1][q >> 2] >> sh) & 0xFFFFu;
    uint32_t x = t0 + t1;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t u = __shfl_up(x, o, 64);
      x += lane >= o ? u : 0u;
    }
    const uint32_t ex = x - t0 - t1;
    sOff[q][w] = ex;
    sOff[q][w + 1] = ex + t0;
    // lane p < 8: process p's first entry, end and chunks
    const uint32_t off = __shfl(ex, 8 * (lane & 7), 64), end = __shfl(x, 8 * (lane & 7) + 7, 64);
    const uint32_t nc = (end - off + 63u) / 64u;
    uint32_t y = nc;
#pragma unroll
    for (int o = 1; o < kNumProc; o <<= 1) {
      const uint32_t u = __shfl_up(y, o, 64);
      y += lane >= o ? u : 0u;
    }
    if (lane < kNumProc) {
      info[lane] = off;
      info[kNumProc + 1 + lane] = y - nc;
      if (lane == kNumProc - 1) {
        info[kNumProc] = end;
        info[2 * kNumProc + 1] = y;
      }
    }
  }
  __syncthreads();
  xl -= lo;
  xh -= hi;
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    if (c[k] != 0) {
      const int q = c[k] - 1, sh = 16 * (q & 3);
      const uint32_t rank = (uint32_t)((q < 4 ? xl : xh) >> sh) & 0xFFFFu;
      tlist[tile0 + sOff[q][wave] + rank] = (uint16_t)(first + k);
      const uint64_t one = 1ull << sh;
      xl += q < 4 ? one : 0ull;
      xh += q < 4 ? 0ull : one;
    }
  }
}

__global__ void __launch_bounds__(kClassifyBlock) k_classify_tiles(int n, const uint8_t* __restrict__ code,
                                                                   uint16_t* __restrict__ tlist, uint32_t* __restrict__ tinfo) {
  ClassifyTileLayout(n, code, tlist, tinfo + (size_t)blockIdx.x * kTileInfo, (int)blockIdx.x);
}

// block -> (tile, chunk of this wave): XCD x takes tiles x, x + kXcds, ...,
// each as kInteractParts consecutive blocks of its share; false past the last
// tile
template <int PARTS = kInteractParts> __device__ inline bool TileChunk(uint32_t ntiles, uint32_t& tile, uint32_t& chunk) {
  const uint32_t x = blockIdx.x % kXcds;
  const uint32_t inXcd = blockIdx.x / kXcds;
  tile = (inXcd / PARTS) * kXcds + x;
  chunk = (inXcd % PARTS) * kInteractWaves + (threadIdx.x >> 6);
  return tile < ntiles;
}

// final state of this lane's entry of chunk `chunk` of a tile whose first
// slot is tile0 (codes, staged records and tile list of its batch)
template <typename R>
__device__ void InteractTileChunk(const DevTables<R>& T, uint64_t seed, hepem_tracks& out, const hepem_step_out& res, int n,
                                  const uint8_t* __restrict__ code, const Staged* __restrict__ st,
                                  const uint16_t* __restrict__ tlist, const uint32_t* __restrict__ info, int tile0,
                                  uint32_t chunk) {
  // the chunk is the same for the whole wave: its process is found in scalar
  // registers from one load of the tile's words (a search through them in
  // memory was a chain of up to eight dependent loads)
  chunk = (uint32_t)__builtin_amdgcn_readfirstlane((int)chunk);
  uint32_t w[kTileInfo];
#pragma unroll
  for (int k = 0; k < kTileInfo; ++k) w[k] = info[k];
  if (chunk >= w[2 * kNumProc + 1]) return;
  int q = 0;
  uint32_t first = w[0], end = w[1], chunk0 = w[kNumProc + 1];
#pragma unroll
  for (int p = 1; p < kNumProc; ++p) {
    const bool here = chunk >= w[kNumProc + 1 + p];
    q = here ? p : q;
    first = here ? w[p] : first;
    end = here ? w[p + 1] : end;
    chunk0 = here ? w[kNumProc + 1 + p] : chunk0;
  }
  const uint32_t k = (chunk - chunk0) * 64u + (uint32_t)__lane_id();
  if (k >= end - first) return;
  const int i = tile0 + (int)tlist[tile0 + first + k];
  const uint8_t c = code[i];
  const Staged r = st[i];
  if (q + 1 < kPConv) ElectronInteract<R>(T, seed, out, res, n, i, r, c);
  else GammaInteract<R>(T, seed, out, res, n, i, r, c);
}

// Held to 4 waves per SIMD: left alone the FP64 form takes 139 VGPRs (3 waves);
// at 127 nothing spills.
template <typename R>
__global__ void __launch_bounds__(kBlock, 4) k_interact_tiles(DevTables<R> T, uint64_t seed, hepem_tracks out, hepem_step_out res,
                                                           const uint8_t* __restrict__ code, const Staged* __restrict__ st,
                                                           const uint16_t* __restrict__ tlist,
                                                           const uint32_t* __restrict__ tinfo) {
  const int n = out.n;
  uint32_t tile, chunk;
  if (!TileChunk((uint32_t)((n + kClassifyTile - 1) / kClassifyTile), tile, chunk)) return;
  InteractTileChunk<R>(T, seed, out, res, n, code, st, tlist, tinfo + (size_t)tile * kTileInfo, (int)tile * kClassifyTile,
                       chunk);
}

// ---- batched stepping ---------------------------------------------------------------------------
// Block sizes of the batched step kernel, selected at run time.
constexpr int kNumShapes = 3;
constexpr int ShapeBlock(int s) { return 64 << s; }
// Process-sort tile sizes of the batched step, selected at run time:
// TileSlots(t) = 1024 << t slots (1024 ... 8192), TileItems(t) per thread of
// the classification block.
constexpr int kNumTiles = 4;
constexpr int TileItems(int t) { return 1 << t; }
constexpr int TileSlots(int t) { return kClassifyBlock << t; }
// the tile size of the particle classification among them
constexpr int kParticleTiles = 2;
static_assert(TileSlots(kParticleTiles) == kClassifyTile, "particle tiles are one of the sort tile sizes");
// Words of a plan's work counters after its per-batch counters: the next
// chunk of the persistent step kernel, then the next work item of each XCD's
// share of the persistent tile kernel.
constexpr int kQueueWords = 1 + kXcds;

// Device descriptor of one batch of a plan. A plan holds nbatch + 1 of them;
// the last carries only the totals of the prefix fields.
struct BatchDev {
  hepem_tracks in, out;
  hepem_step_out res;
  uint32_t qoff;                 // first entry of the batch's queue
  uint32_t tile0;                // first particle-classify tile of the batch (kClassifyTile slots)
  uint32_t ptile0[kNumTiles];    // first process-sort tile of the batch for tile size TileSlots(t)
  uint32_t chunk0[kNumShapes];   // first step chunk for block size ShapeBlock(s)
};


// bcounters[4b + 0..2]: e-/e+, gammas, rejected tracks of batch b
__global__ void __launch_bounds__(kClassifyBlock) k_classify_batched(const BatchDev* __restrict__ d,
                                                             const uint32_t* __restrict__ tbatch,
                                                             uint32_t* __restrict__ queue, uint32_t* __restrict__ bcounters) {
  const uint32_t t = blockIdx.x;
  const int b = __builtin_amdgcn_readfirstlane((int)tbatch[t]);
  ClassifyTile(d[b].in.n, d[b].in.ptype, queue + d[b].qoff, bcounters + 4 * b, (int)(t - d[b].tile0));
}

// One thread per queue entry of every batch: block c takes chunk c of the
// chunk sequence (all batches' chunks of BS entries, in batch order). The
// batch index is uniform over the block: it (and the descriptor loads) stay
// scalar.
template <typename R, int S>
__device__ void StepChunk(const DevTables<R>& T, uint64_t seed, const BatchDev* __restrict__ d,
                          const uint32_t* __restrict__ cbatch, uint32_t c,
                          const uint32_t* __restrict__ queue, uint32_t* __restrict__ bcounters) {
  constexpr int BS = ShapeBlock(S);
  const int b = __builtin_amdgcn_readfirstlane((int)cbatch[c]);
  const hepem_tracks in = d[b].in;
  hepem_tracks out = d[b].out;
  const hepem_step_out res = d[b].res;
  const int n = in.n;
  const int j = (int)(c - d[b].chunk0[S]) * BS + (int)threadIdx.x;
  if (j >= n) return;
  uint32_t* cnt = bcounters + 4 * b;
  const int i = (int)queue[d[b].qoff + j];
  if (RejectTrack(T, in, out, res, n, i, cnt)) return;
  CopyIdentity(in, out, i);
  if ((uint32_t)j < cnt[0]) StepElectron(T, seed, in, out, res, n, i);
  else StepGamma(T, seed, in, out, res, n, i);
}

// Stage 1 of the two-stage form over every batch: records the process code
// and staged record of slot i of batch b at global index qoff_b + i;
// k_classify_tiles_batched and k_interact_tiles_batched then sort and sample
// them tile by tile, as the single-batch step does (tiles numbered across
// the batches).
template <typename R, int S>
__device__ void StepSelectChunk(const DevTables<R>& T, uint64_t seed, const BatchDev* __restrict__ d,
                                const uint32_t* __restrict__ cbatch, uint32_t c,
                                const uint32_t* __restrict__ queue, uint32_t* __restrict__ bcounters,
                                uint8_t* __restrict__ code, Staged* __restrict__ st) {
  constexpr int BS = ShapeBlock(S);
  const int b = __builtin_amdgcn_readfirstlane((int)cbatch[c]);
  const hepem_tracks in = d[b].in;
  hepem_tracks out = d[b].out;
  const hepem_step_out res = d[b].res;
  const int n = in.n;
  const int j = (int)(c - d[b].chunk0[S]) * BS + (int)threadIdx.x;
  if (j >= n) return;
  uint32_t* cnt = bcounters + 4 * b;
  const uint32_t qoff = d[b].qoff;
  const int i = (int)queue[qoff + j];
  code[qoff + i] = StepSelect<R>([&] { return StepView<R>{T, seed, in, out, res, cnt}; }, n, i, (uint32_t)j < cnt[0], st + qoff, i);
}

// The tile-local particle partition over every batch: block t lays out
// particle-classify tile t of the plan (tiles numbered across the batches, as
// BatchDev::tile0), within its batch's queue; ecount[t] = its e-/e+ count.
__global__ void __launch_bounds__(kClassifyBlock) k_classify_local_batched(const BatchDev* __restrict__ d,
                                                                           const uint32_t* __restrict__ tbatch,
                                                                           uint32_t* __restrict__ queue,
                                                                           uint32_t* __restrict__ ecount) {
  const uint32_t t = blockIdx.x;
  const int b = __builtin_amdgcn_readfirstlane((int)tbatch[t]);
  ClassifyLocalTile(d[b].in.n, d[b].in.ptype, queue + d[b].qoff, (int)(t - d[b].tile0), ecount + t);
}

// Stage 1 of the two-stage form over the tile-local partition of every
// batch (kBlock threads, a grid of LocalSelectGridTiles(ntiles)): the blocks
// of the plan's tiles are placed as k_step_select_local places a single
// batch's, and each records what StepSelectChunk records.
template <typename R> struct BatchArgs {
  DevTables<R> T;
  uint64_t seed;
  const BatchDev* d;
  const uint32_t* tbatch;
  int ntiles;
  const uint32_t* queue;
  uint32_t* bcounters;
  const uint32_t* ecount;
  uint8_t* code;
  Staged* st;
};
// Descriptor of batch b: constant memory while a kernel runs, so its words are
// scalar loads wherever they are read.
template <typename R> HD const BatchDev& Descriptor(int b) {
  return *(const BatchDev*)((const __attribute__((address_space(4))) BatchDev*)KernelArgs<BatchArgs<R>>().d + b);
}
template <typename R> __global__ void __launch_bounds__(kBlock, 4) k_step_select_local_batched(BatchArgs<R>) {
  int tile, chunk, b, n, i;
  uint32_t qoff;
  bool isE;
  {
    const BatchArgs<R>& a = KernelArgs<BatchArgs<R>>();
    if (!LocalSelectChunk(a.ntiles, tile, chunk)) return;
    b = __builtin_amdgcn_readfirstlane((int)a.tbatch[tile]);
    const BatchDev& d = Descriptor<R>(b);
    n = d.in.n;
    const int tile0 = (tile - (int)d.tile0) * kClassifyTile;
    const int m = min(kClassifyTile, n - tile0);
    const int jl = chunk * kBlock + (int)threadIdx.x;
    if (jl >= m) return;
    qoff = d.qoff;
    i = (int)a.queue[qoff + tile0 + jl];
    isE = jl < (int)a.ecount[tile];
  }
  const auto view = [b]() HEPEM_INLINE {
    const BatchArgs<R>& a = KernelArgs<BatchArgs<R>>();
    const BatchDev& d = Descriptor<R>(b);
    return StepView<R>{a.T, a.seed, d.in, const_cast<hepem_tracks&>(d.out), d.res, a.bcounters + 4 * b};
  };
  const uint8_t c = StepSelect<R>(view, n, i, isE, KernelArgs<BatchArgs<R>>().st + qoff, i);
  KernelArgs<BatchArgs<R>>().code[qoff + i] = c;
}
static_assert(std::is_same_v<decltype(k_step_select_local_batched<double>), void(BatchArgs<double>)>);

// Next work item of a persistent kernel: thread 0 takes it from *next and the
// block reads it from LDS (the second barrier keeps thread 0 from overwriting
// it before every thread has read it).
__device__ inline uint32_t NextItem(uint32_t* next) {
  __shared__ uint32_t sItem;
  if (threadIdx.x == 0) sItem = atomicAdd(next, 1u);
  __syncthreads();
  const uint32_t c = sItem;
  __syncthreads();
  return c;
}

// Dispatched form: block c takes chunk c.
template <typename R, int S>
__global__ void __launch_bounds__(ShapeBlock(S)) k_step_batched(DevTables<R> T, uint64_t seed, const BatchDev* __restrict__ d,
                                                                const uint32_t* __restrict__ cbatch, uint32_t nchunks,
                                                                const uint32_t* __restrict__ queue,
                                                                uint32_t* __restrict__ bcounters) {
  if (blockIdx.x < nchunks) StepChunk<R, S>(T, seed, d, cbatch, blockIdx.x, queue, bcounters);
}

// Persistent form: one resident round of blocks, each taking chunks from the
// counter *next (zero at launch) until they run out. Nothing but the chunk
// index is carried from one chunk to the next.
template <typename R, int S>
__global__ void __launch_bounds__(ShapeBlock(S)) k_step_batched_q(DevTables<R> T, uint64_t seed, const BatchDev* __restrict__ d,
                                                                  const uint32_t* __restrict__ cbatch, uint32_t nchunks,
                                                                  const uint32_t* __restrict__ queue,
                                                                  uint32_t* __restrict__ bcounters, uint32_t* __restrict__ next) {
  for (uint32_t c = NextItem(next); c < nchunks; c = NextItem(next)) StepChunk<R, S>(T, seed, d, cbatch, c, queue, bcounters);
}

template <typename R, int S>
__global__ void __launch_bounds__(ShapeBlock(S)) k_step_select_batched(DevTables<R> T, uint64_t seed,
                                                                       const BatchDev* __restrict__ d, const uint32_t* __restrict__ cbatch,
                                                                       uint32_t nchunks, const uint32_t* __restrict__ queue,
                                                                       uint32_t* __restrict__ bcounters,
                                                                       uint8_t* __restrict__ code, Staged* __restrict__ st) {
  if (blockIdx.x < nchunks) StepSelectChunk<R, S>(T, seed, d, cbatch, blockIdx.x, queue, bcounters, code, st);
}

template <typename R, int S>
__global__ void __launch_bounds__(ShapeBlock(S)) k_step_select_batched_q(DevTables<R> T, uint64_t seed,
                                                                         const BatchDev* __restrict__ d, const uint32_t* __restrict__ cbatch,
                                                                         uint32_t nchunks, const uint32_t* __restrict__ queue,
                                                                         uint32_t* __restrict__ bcounters,
                                                                         uint8_t* __restrict__ code, Staged* __restrict__ st,
                                                                         uint32_t* __restrict__ next) {
  for (uint32_t c = NextItem(next); c < nchunks; c = NextItem(next))
    StepSelectChunk<R, S>(T, seed, d, cbatch, c, queue, bcounters, code, st);
}

// The tile-local process sort over all batches of a plan, in tiles of
// TileSlots(TI) slots: tiles are numbered across the batches
// (BatchDev::ptile0[TI]), each batch's tile list and codes sit at its queue
// offset.
template <int TI>
__global__ void __launch_bounds__(kClassifyBlock) k_classify_tiles_batched(const BatchDev* __restrict__ d,
                                                                           const uint32_t* __restrict__ tbatch,
                                                                           const uint8_t* __restrict__ code,
                                                                           uint16_t* __restrict__ tlist,
                                                                           uint32_t* __restrict__ tinfo) {
  const uint32_t t = blockIdx.x;
  const int b = __builtin_amdgcn_readfirstlane((int)tbatch[t]);
  const uint32_t qoff = d[b].qoff;
  ClassifyTileLayout<TileItems(TI)>(d[b].in.n, code + qoff, tlist + qoff, tinfo + (size_t)t * kTileInfo,
                                    (int)(t - d[b].ptile0[TI]));
}

template <typename R, int TI>
__device__ void InteractBatchedTile(const DevTables<R>& T, uint64_t seed, const BatchDev* __restrict__ d,
                                    const uint32_t* __restrict__ tbatch, uint32_t tile, uint32_t chunk,
                                    const uint8_t* __restrict__ code, const Staged* __restrict__ st,
                                    const uint16_t* __restrict__ tlist, const uint32_t* __restrict__ tinfo) {
  const int b = __builtin_amdgcn_readfirstlane((int)tbatch[tile]);
  hepem_tracks& out = const_cast<hepem_tracks&>(d[b].out);
  const uint32_t qoff = d[b].qoff;
  InteractTileChunk<R>(T, seed, out, d[b].res, out.n, code + qoff, st + qoff, tlist + qoff, tinfo + (size_t)tile * kTileInfo,
                       (int)(tile - d[b].ptile0[TI]) * TileSlots(TI), chunk);
}

template <typename R, int TI>
__global__ void __launch_bounds__(kBlock, 4) k_interact_tiles_batched(DevTables<R> T, uint64_t seed, const BatchDev* __restrict__ d,
                                                                   const uint32_t* __restrict__ tbatch, uint32_t ntiles,
                                                                   const uint8_t* __restrict__ code,
                                                                   const Staged* __restrict__ st,
                                                                   const uint16_t* __restrict__ tlist,
                                                                   const uint32_t* __restrict__ tinfo) {
  uint32_t tile, chunk;
  if (!TileChunk<InteractParts(TileItems(TI))>(ntiles, tile, chunk)) return;
  InteractBatchedTile<R, TI>(T, seed, d, tbatch, tile, chunk, code, st, tlist, tinfo);
}

// Persistent form of k_interact_tiles_batched: one resident round of blocks.
// Block b works for XCD b % kXcds (blocks are dealt to the XCDs round-robin)
// and takes that XCD's work items, tiles x, x + kXcds, ... in
// InteractParts blocks' worth each, from its counter next[x] (zero at launch).
template <typename R, int TI>
__global__ void __launch_bounds__(kBlock) k_interact_tiles_batched_q(DevTables<R> T, uint64_t seed,
                                                                     const BatchDev* __restrict__ d,
                                                                     const uint32_t* __restrict__ tbatch, uint32_t ntiles,
                                                                     const uint8_t* __restrict__ code,
                                                                     const Staged* __restrict__ st,
                                                                     const uint16_t* __restrict__ tlist,
                                                                     const uint32_t* __restrict__ tinfo,
                                                                     uint32_t* __restrict__ next) {
  constexpr uint32_t P = InteractParts(TileItems(TI));
  const uint32_t x = blockIdx.x % kXcds;
  for (uint32_t k = NextItem(next + x);; k = NextItem(next + x)) {
    const uint32_t tile = (k / P) * kXcds + x;
    if (tile >= ntiles) return;
    const uint32_t chunk = (k % P) * kInteractWaves + (threadIdx.x >> 6);
    InteractBatchedTile<R, TI>(T, seed, d, tbatch, tile, chunk, code, st, tlist, tinfo);
  }
}

// the five config-1 quantities of query i at (mc, E, lnE): restricted dE/dx,
// range, inverse range of that range, ioni and brem cross sections; NaN for
// an invalid couple. Those are computed at couple 0 and then replaced, so
// every lane stores at the same places in the code (no branch around the
// memory operations: the wait for the next query's inputs then covers no
// store that a branch left unaccounted). The results are streamed out
// (non-temporal stores): nothing in the kernel reads them back.
template <typename R>
HD void LookupStore(const DevEl<R>& e, int nmc, int n, int i, int mc, double E, double lnE, double* __restrict__ out) {
  const size_t sn = (size_t)n;  // 5 n entries may exceed the int range
  const bool ok = mc >= 0 && mc < nmc;
  const double nan = __longlong_as_double(0x7FF8000000000000LL);
  mc = ok ? mc : 0;
  const R lE = (R)lnE;
  // the range's loss-grid bin is where its inverse is searched first (the
  // spline's grid energies are the inverse's ordinates there)
  const int bin = LogBin(lE, e.lossLogMin, e.lossILD, e.N);
  const R r = GetRestRange(e, mc, E, lE);
  __builtin_nontemporal_store(ok ? (double)GetRestDEDX(e, mc, E, lE) : nan, out + i);
  __builtin_nontemporal_store(ok ? (double)r : nan, out + sn + i);
  __builtin_nontemporal_store(ok ? GetInvRangeInBin(e, mc, (double)r, bin, e.lossGrid64[bin], e.lossGrid64[bin + 1]) : nan, out + 2 * sn + i);
  __builtin_nontemporal_store(ok ? (double)GetRestMacXSec(e, mc, E, lE, true) : nan, out + 3 * sn + i);
  __builtin_nontemporal_store(ok ? (double)GetRestMacXSec(e, mc, E, lE, false) : nan, out + 4 * sn + i);
}

template <typename R>
__global__ void __launch_bounds__(kBlock) k_lookup(DevTables<R> T, int ptype, int n, const int32_t* __restrict__ imc,
                                                   const double* __restrict__ ekin, const double* __restrict__ lekin,
                                                   double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  LookupStore(T.el[ptype], T.nmc, n, i, imc[i], ekin[i], lekin[i], out);
}

// Gamma macroscopic cross sections and the interaction they select, one query
// per thread, as the reference's TestMacXSecDataKernel drives
// G4HepEmGammaManager::GetTotalMacXSec and SampleInteraction
// (testing/GammaXSections/src/GammaMacXSecs.cu:20-31): the total cross section,
// the photoelectric one the track holds after SampleInteraction, and the
// process chosen for the uniform draw u. An invalid couple gives NaN and -99.
template <typename R>
__global__ void __launch_bounds__(kBlock) k_gamma_lookup(DevTables<R> T, int n, const int32_t* __restrict__ imc,
                                                         const double* __restrict__ ekin, const double* __restrict__ lekin,
                                                         const double* __restrict__ urnd, double* __restrict__ out_xs,
                                                         double* __restrict__ out_pe, int32_t* __restrict__ out_pid) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int mc = imc[i];
  if (mc < 0 || mc >= T.nmc) {
    out_xs[i] = out_pe[i] = __longlong_as_double(0x7FF8000000000000LL);
    out_pid[i] = -99;
    return;
  }
  Trk<R> t;
  t.ekin = ekin[i];
  t.lekin = (R)lekin[i];
  t.imc = mc;
  t.winner = -1;
  for (int k = 0; k < 4; ++k) t.mfp[k] = t.nial[k] = (R)0.0;
  R pe = (R)0.0;
  const R tot = GetTotalMacXSec(T, t, pe);
  t.mfp[0] = (tot > (R)0.) ? (R)1. / tot : (R)kALargeValue;
  SampleInteraction(T, t, pe, (R)urnd[i]);
  out_xs[i] = (double)tot;
  out_pe[i] = (double)pe;
  out_pid[i] = t.winner;
}

// LDS staging of the config-1 lookups. The loss grid and data and the
// cross-section blocks of every couple (the doubles, and in the FP32 form
// the floats too) are a few kB per couple; each block copies them to LDS
// once and then serves a contiguous chunk of the queries from there, so the
// table gathers leave the texture path to the query stream.
constexpr size_t kLookupLdsMax = 64 * 1024;  // larger images use k_lookup
constexpr int kLookupBlocks = 2048;          // resident blocks if the occupancy query gives nothing
constexpr int kLookupPerThread = 16;         // queries per thread of a chunk, at most

__host__ __device__ inline size_t Al16(size_t b) { return (b + 15) & ~size_t(15); }

// LDS bytes of the image (the arrays in the order k_lookup_lds stages them)
template <typename R> __host__ __device__ size_t LookupLdsBytes(const DevEl<R>& e, int nmc) {
  const size_t N = (size_t)e.N, L = 5 * N * (size_t)nmc, X = (size_t)e.xsN;
  size_t b = Al16(N * sizeof(double)) + Al16(L * sizeof(double)) + Al16(X * sizeof(double)) +
             Al16(2 * (size_t)nmc * sizeof(XsBlock<R>));
  if (sizeof(R) != sizeof(double)) b += Al16(N * sizeof(R)) + Al16(L * sizeof(R)) + Al16(X * sizeof(R));
  return b;
}

// copies `bytes` (a multiple of 4) from src to lds + off with the whole block;
// returns the LDS copy and advances off
__device__ inline const void* StageArray(unsigned char* lds, size_t& off, const void* src, size_t bytes) {
  unsigned char* dst = lds + off;
  if ((bytes & 15) == 0) {
    const uint4* s4 = reinterpret_cast<const uint4*>(src);
    uint4* d4 = reinterpret_cast<uint4*>(dst);
    for (size_t k = threadIdx.x; k < bytes / 16; k += blockDim.x) d4[k] = s4[k];
  } else {
    const uint32_t* s1 = reinterpret_cast<const uint32_t*>(src);
    uint32_t* d1 = reinterpret_cast<uint32_t*>(dst);
    for (size_t k = threadIdx.x; k < bytes / 4; k += blockDim.x) d1[k] = s1[k];
  }
  off += Al16(bytes);
  return dst;
}

template <typename R>
__global__ void __launch_bounds__(kBlock) k_lookup_lds(DevTables<R> T, int ptype, int n, const int32_t* __restrict__ imc,
                                                       const double* __restrict__ ekin, const double* __restrict__ lekin,
                                                       double* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char lds[];
  DevEl<R> e = T.el[ptype];
  const int nmc = T.nmc;
  const size_t N = (size_t)e.N, L = 5 * N * (size_t)nmc, X = (size_t)e.xsN;
  size_t off = 0;
  e.lossGrid64 = static_cast<const double*>(StageArray(lds, off, e.lossGrid64, N * sizeof(double)));
  e.lossData64 = static_cast<const double*>(StageArray(lds, off, e.lossData64, L * sizeof(double)));
  e.xsData64 = static_cast<const double*>(StageArray(lds, off, e.xsData64, X * sizeof(double)));
  e.xsBlock = static_cast<const XsBlock<R>*>(StageArray(lds, off, e.xsBlock, 2 * (size_t)nmc * sizeof(XsBlock<R>)));
  if constexpr (sizeof(R) == sizeof(double)) {
    // the FP64 form's value arrays are the double arrays
    e.lossGrid = reinterpret_cast<const R*>(e.lossGrid64);
    e.lossData = reinterpret_cast<const R*>(e.lossData64);
    e.xsData = reinterpret_cast<const R*>(e.xsData64);
  } else {
    e.lossGrid = static_cast<const R*>(StageArray(lds, off, e.lossGrid, N * sizeof(R)));
    e.lossData = static_cast<const R*>(StageArray(lds, off, e.lossData, L * sizeof(R)));
    e.xsData = static_cast<const R*>(StageArray(lds, off, e.xsData, X * sizeof(R)));
  }
  __syncthreads();
  // each block serves one contiguous chunk of `per` queries per thread; the
  // next query's inputs are loaded before this one is computed, so their HBM
  // latency overlaps the table work (the chunk's last round reloads its own
  // query instead, so the loads are unconditional)
  const int64_t threads = (int64_t)gridDim.x * blockDim.x;
  const int64_t per = ((int64_t)n + threads - 1) / threads;
  const int64_t base = (int64_t)blockIdx.x * blockDim.x * per;
  const int64_t end = min((int64_t)n, base + per * (int64_t)blockDim.x);
  const int64_t stride = blockDim.x;
  int64_t i = base + threadIdx.x;
  if (i >= end) return;
  int mc = imc[i];
  double E = ekin[i], lnE = lekin[i];
  while (true) {
    const int64_t next = i + stride;
    const int64_t ld = next < end ? next : i;
    const int mcN = imc[ld];
    const double EN = ekin[ld], lnEN = lekin[ld];
    LookupStore(e, nmc, n, (int)i, mc, E, lnE, out);
    if (next >= end) break;
    i = next;
    mc = mcN;
    E = EN;
    lnE = lnEN;
  }
}

__global__ void k_reset_state(hepem_tracks t) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = t.n;
  if (i >= n) return;
#pragma unroll
  for (int k = 0; k < 4; ++k) t.num_ia_left[k * n + i] = -1.0;
  t.msc_init_range[i] = 1.0e+21;
  t.msc_dyn_range_factor[i] = 0.04;
  t.msc_tlimit_min[i] = 1.0E-7;
  t.msc_first_step[i] = 1;
  t.rng_ctr[i] = 0u;
  t.rng_gauss[i] = 0.0;
  t.rng_has_gauss[i] = 0;
}

}  // namespace hepem
