// dev_final.hh -- the final states of discrete interactions, sampled apart from
// their choice: the process code and the staged state that the choice leaves
// behind, the samplers by code, and the block-wide process sort that hands each
// wave the pending interactions of one process.
#pragma once

#include "dev_physics.hh"

namespace hepem {

// processes of the second stage (0: none pending), in the low 4 bits of the
// per-slot code; bit 4: the track is an e-, bit 5: a Gaussian deviate is cached
enum ProcCode : uint8_t {
  kPNone = 0,
  kPIoniEl,    // Moller
  kPIoniPos,   // Bhabha
  kPBremSB,    // Seltzer-Berger brem (E < model limit)
  kPBremRB,    // relativistic brem
  kPAnnih,     // e+ annihilation in flight
  kPConv,      // gamma conversion
  kPCompton,   // Klein-Nishina
  kPPE,        // photoelectric
};
constexpr int kNumProc = 8;          // codes 1..8
constexpr uint8_t kCodeProc = 0x0F, kCodeElectron = 0x10, kCodeGauss = 0x20;

// state handed from the selection to the final-state sampling of one slot
struct alignas(16) Staged {
  double ekin, dir[3], gauss, pe;
  int32_t imc, id;
  uint32_t stream, ctr;
};
static_assert(sizeof(Staged) == 64, "one 64-byte record per pending slot");

HD uint8_t StageTrack(Staged* st, int i, uint8_t proc, bool isEl, int imc, int32_t id, uint32_t stream, double ekin,
                      const double* dir, const Rng& rng, double pe) {
  Staged r;
  r.ekin = ekin;
  r.dir[0] = dir[0];
  r.dir[1] = dir[1];
  r.dir[2] = dir[2];
  r.gauss = rng.gauss;
  r.pe = pe;
  r.imc = imc;
  r.id = id;
  r.stream = stream;
  r.ctr = rng.ctr;
  st[i] = r;
  return (uint8_t)(proc | (isEl ? kCodeElectron : 0) | (rng.has_gauss ? kCodeGauss : 0));
}

// Track state of a pending slot from its staged record.
template <typename R> HD void Unstage(const Staged& r, uint8_t code, uint64_t seed, Trk<R>& t, Rng& rng) {
  t.isEl = (code & kCodeElectron) != 0;
  t.setE(r.ekin);
#pragma unroll
  for (int c = 0; c < 3; ++c) t.dir[c] = (R)r.dir[c];
  t.imc = r.imc;
  t.edep = 0.0;
  rng.init(seed, (uint32_t)r.id, r.stream, r.ctr, (code & kCodeGauss) != 0, r.gauss);
}

// The code of the interaction PerformDiscrete chose for an e-/e+ (0 ionisation,
// 1 brem, 2 annihilation in flight, else none: an e-/e+ nuclear interaction has
// no final state).
template <typename R> HD uint8_t ElectronProc(const DevTables<R>& T, const Trk<R>& t, int chosen) {
  return chosen == 0   ? (t.isEl ? kPIoniEl : kPIoniPos)
         : chosen == 1 ? (t.ekin < T.bremModelLim ? kPBremSB : kPBremRB)
         : chosen == 2 ? kPAnnih
                       : kPNone;
}

// What follows the gamma's move up to the final state: on a boundary only the
// interaction-length update, otherwise SelectInteraction and Perform's reset
// (G4HepEmTrackingManager.cc:1092-1108; G4HepEmGammaManager.icc:54-62,173-219).
// pe becomes the PE cross section that SelectInteraction leaves in the track.
template <typename R> HD uint8_t GammaProc(const DevTables<R>& T, Trk<R>& t, R& pe, Rng& rng) {
  if (t.onBoundary) {
    t.nial[0] -= t.gstep / t.mfp[0];
    return kPNone;
  }
  SampleInteraction(T, t, pe, (R)rng.flat());
  if (t.winner == 3) return kPNone;
  t.nial[0] -= t.gstep / t.mfp[0];
  ResetNumIALeft(t.nial, t.winner);
  return t.winner == 0 ? kPConv : t.winner == 1 ? kPCompton : kPPE;
}

// The final state of the chosen e-/e+ interaction (PerformDiscrete,
// G4HepEmElectronManager.icc:443-458).
template <typename R> HD void ElectronFinal(const DevTables<R>& T, Trk<R>& t, int proc, SecList<R>& sl, Rng& rng) {
  switch (proc) {
    case kPIoniEl:
    case kPIoniPos: IoniPerform(T, t, sl, rng); break;
    case kPBremSB: BremPerform(T, t, sl, rng, true); break;
    case kPBremRB: BremPerform(T, t, sl, rng, false); break;
    default: AnnihilateInFlight(t, sl, rng); break;
  }
}

// The final state of the chosen gamma interaction and the gamma tracking cut of
// G4HepEmGammaManager::Perform (G4HepEmGammaManager.icc:63-93).
template <typename R> HD void GammaFinal(const DevTables<R>& T, Trk<R>& t, int proc, R pe, SecList<R>& sl, Rng& rng) {
  switch (proc) {
    case kPConv: ConvPerform(T, t, sl, rng); break;
    case kPCompton: ComptonPerform(t, sl, rng); break;
    default: PEPerform(T, t, pe, sl, rng); break;
  }
  const double finalEkin = t.ekin;
  if (finalEkin > 0.0 && finalEkin <= T.gamTrackCut) {
    t.setE(0.0);
    t.edep += finalEkin;
  }
}

// The pending interactions of one block of NT threads, sorted by process within
// the block.
template <int NT> struct BlockFinals {
  Staged st[NT];                        // by thread
  uint8_t code[NT];                     // by thread
  uint8_t list[NT];                     // threads, process by process
  uint32_t count[kNumProc][NT / 64];    // per process and wave
};

// Hands the block's pending interactions (code: this thread's, or 0; its record
// in b.st[threadIdx.x]) to the waves, up to 64 of one process at a time, and
// calls sample(thread, record, code, process) for each. Every thread of the
// block calls it; codes are of the processes P0..P1. Memory written before the
// call is visible to sample. It ends without a barrier: what sample writes is
// there for the rest of the block, and b free for another use, only after the
// caller's next __syncthreads().
template <int NT, int P0, int P1, typename F>
__device__ __forceinline__ void SampleBlock(BlockFinals<NT>& b, uint8_t code, F sample) {
  static_assert(NT <= 256, "list entries are 8 bits");
  constexpr int NW = NT / 64, NP = P1 - P0 + 1;
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const uint64_t below = (1ull << lane) - 1ull;
  const int mine = (int)(code & kCodeProc) - P0;  // negative: none pending
  uint32_t rank = 0u;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const uint64_t m = __ballot(mine == p);
    if (mine == p) rank = (uint32_t)__popcll(m & below);
    if (lane == p) b.count[p][wave] = (uint32_t)__popcll(m);
  }
  b.code[threadIdx.x] = code;
  __syncthreads();
  uint32_t first[NP + 1], before = 0u;
  first[0] = 0u;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    uint32_t sum = 0u;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const uint32_t c = b.count[p][w];
      if (mine == p && w < wave) before += c;
      sum += c;
    }
    first[p + 1] = (uint32_t)__builtin_amdgcn_readfirstlane((int)(first[p] + sum));
    if (mine == p) before += first[p];
  }
  if (mine >= 0) b.list[before + rank] = (uint8_t)threadIdx.x;
  __syncthreads();
  // chunk c of the block's sequence goes to wave c mod NW
  uint32_t chunk = 0u;
#pragma unroll 1
  for (int p = 0; p < NP; ++p) {
    uint32_t lo = first[0], hi = first[1];
#pragma unroll
    for (int q = 1; q < NP; ++q) {
      lo = p == q ? first[q] : lo;
      hi = p == q ? first[q + 1] : hi;
    }
    for (uint32_t k0 = lo; k0 < hi; k0 += 64u, ++chunk) {
      if (chunk % (uint32_t)NW != (uint32_t)wave) continue;
      const uint32_t k = k0 + (uint32_t)lane;
      if (k < hi) {
        const int j = b.list[k];
        sample(j, b.st[j], b.code[j], p + P0);
      }
    }
  }
}

}  // namespace hepem
