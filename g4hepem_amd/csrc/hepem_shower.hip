// hepem_shower.hip -- showers in a 1D stack of slabs (include/g4hepem_amd_shower.h).
//
// The track stack is a pair of structure-of-arrays buffers of `capacity`
// slots. One stepping round over the n tracks in flight:
//   k_sh_move      the e-/e+ (the first part of the stack): one sub-step of
//                  G4HepEmTrackingManager::TrackElectron's step each, after
//                  the step's pre-step part where a track is not within a step
//                  (device/dev_tracking.hh), with the slab as the geometry and
//                  the MSC displacement applied; a track within its step
//                  carries the loop state to the next round, one whose step
//                  ended finishes it: the loss fluctuation, at-rest
//                  annihilation or the discrete interaction;
//                  the gammas: HowFar, the cut at the next plane along x (or,
//                  with Woodcock tracking on and above its energy limit, a
//                  step through the stack to its next interaction point or out
//                  of it), then the boundary update or SelectInteraction +
//                  Perform;
//                  then, for both, slab crossing, leakage, scoring, the stack
//                  slots each track needs next round and their exclusive scan
//                  within the block
//   k_scan_sums    exclusive scans of the block totals (one block)
//   k_sh_scatter   survivors and their secondaries into the other buffer:
//                  e-/e+ first, then gammas, each in slot order of the parents
//                  (deterministic), planar with the new count
//   k_sh_inject    when the stack runs low, the primaries of the next events
//                  after them.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstring>
#include <limits>
#include <new>
#include <type_traits>
#include <vector>

#include "device/dev_final.hh"
#include "device/dev_physics.hh"
#include "device/dev_scan.hh"
#include "device/dev_soa.hh"
#include "device/dev_tracking.hh"
#include "g4hepem_amd_shower.h"
#include "hepem_internal.hh"

namespace {

constexpr int kB = 256;
constexpr double kFix = 1.0e9;           // fixed-point units per MeV
constexpr double kGeomMinLength = 5.0e-8;
constexpr double kElectronMass = 0.51099895000;
constexpr int kMaxRounds = 1 << 20;       // stepping rounds without new primaries

#define SH_OK(call)                                   \
  do {                                                \
    if ((call) != hipSuccess) return HEPEM_ERR_HIP;   \
  } while (0)

// splitmix64 finaliser: the stream selector of a primary and of every secondary
__host__ __device__ inline uint64_t Mix64(uint64_t x) {
  uint64_t z = x + 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__host__ __device__ inline uint64_t PrimaryStream(int event) { return Mix64(0x5EED000000000000ull ^ (uint64_t)event); }
__host__ __device__ inline uint64_t ChildStream(uint64_t parent, int nstep, int slot) {
  return Mix64(parent ^ Mix64(((uint64_t)(uint32_t)nstep << 2) | (uint64_t)(slot + 1)));
}

// slab geometry, passed by value
struct Slabs {
  int nbins;          // nlayers * nabs
  int nabs;
  int imc[HEPEM_SLAB_MAX_ABS];
  const double* plane;  // nbins + 1 plane positions [mm], plane[0] = 0
  // per absorber: production thresholds (e-, e+, gamma) of its couple and
  // whether its region applies them to secondaries
  double cutE[HEPEM_SLAB_MAX_ABS], cutP[HEPEM_SLAB_MAX_ABS], cutG[HEPEM_SLAB_MAX_ABS];
  int applyCuts[HEPEM_SLAB_MAX_ABS];
  // Woodcock tracking: gammas above wdtMin (0: off) through the whole stack,
  // whose exit planes are 0 and xmax, with the couple wdtImc of its densest
  // material wdtMat; mat[a] = material of absorber a
  double wdtMin, xmax;
  int wdtImc, wdtMat;
  int mat[HEPEM_SLAB_MAX_ABS];
  unsigned wdtMask;  // bit a: absorber a is of material wdtMat
};

static_assert(HEPEM_SLAB_MAX_ABS == 4, "AbsorberCouple selects over four absorbers");
// g.imc[a] as selects (a per-lane index into the kernel argument would be a
// memory load in the innermost loop)
__device__ inline int AbsorberCouple(const Slabs& g, int a) {
  return a == 0 ? g.imc[0] : (a == 1 ? g.imc[1] : (a == 2 ? g.imc[2] : g.imc[3]));
}

// one stack buffer
// What an e-/e+ carries between the sub-steps of one TrackElectron step
// (G4HepEmTrackingManager.cc:427-606), which run one per stepping round: the
// step's pre-step part sets it and each sub-step updates it. Gamma slots do not
// carry it.
constexpr uint8_t kInStep = 1;   // between sub-steps of a step (else the next round begins a step)
constexpr uint8_t kCont = 2;     // continueStepping: MSC may limit the next sub-step too
struct ElLoop {
  double* range;       // restricted range, reduced over the sub-steps
  double* stepLeft;    // what is left of the discrete step
  double* mfp;         // [4][n] macroscopic mean free paths of the step's pre-step point
  double* preEkin;     // the step's pre-step energy
  double* meanLoss;    // summed mean energy losses
  int32_t* nsub;       // sub-steps taken in the step
  int8_t* iDProc;      // the discrete process HowFarToDiscreteInteraction chose
  uint8_t* flags;      // kInStep | kCont, or 0
};

struct Stack {
  hepem_tracks t;     // t.n = tracks in it (stride of the planar fields)
  double* x;
  int32_t* layer;     // slab index
  int32_t* event;     // deposit row of the event (events resident at once)
  int32_t* nstep;     // steps taken by the track
  ElLoop lp;          // e-/e+ slots: the state between sub-steps
};

__global__ void k_sh_fill64(int64_t* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Primaries of events e0 + j, j in [0, k): at x = 0, moving along +x,
// entering slab 0; deposit row ev0 + j. They go to slots base[0] + j of a
// buffer of total[0] tracks (base = total = NULL: slots j of a buffer of k).
// Writes nothing if the buffer would exceed `cap`.
__global__ void k_sh_inject(Stack s, Slabs g, int ptype, double ekin, int e0, int ev0, int k,
                            const uint32_t* __restrict__ base, const uint32_t* __restrict__ total, int cap) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= k) return;
  const int m = total ? (int)*total : k;
  if (m > cap) return;
  const int i = (base ? (int)*base : 0) + j;
  const hepem_tracks& t = s.t;
  const uint64_t sid = PrimaryStream(e0 + j);
  t.ptype[i] = (int8_t)ptype;
  t.id[i] = (int32_t)(uint32_t)sid;
  t.rng_stream[i] = (uint32_t)(sid >> 32);
  t.imc[i] = g.imc[0];
  t.ekin[i] = ekin;
  t.dir[i] = 1.0;
  t.dir[m + i] = 0.0;
  t.dir[2 * m + i] = 0.0;
  t.safety[i] = 0.0;
  t.on_boundary[i] = 1;
  for (int c = 0; c < 4; ++c) t.num_ia_left[c * m + i] = -1.0;
  t.msc_init_range[i] = 1.0e+21;
  t.msc_dyn_range_factor[i] = 0.04;
  t.msc_tlimit_min[i] = 1.0E-7;
  t.msc_first_step[i] = 1;
  t.rng_ctr[i] = 0u;
  t.rng_gauss[i] = 0.0;
  t.rng_has_gauss[i] = 0;
  s.x[i] = 0.0;
  s.layer[i] = 0;
  s.event[i] = ev0 + j;
  s.nstep[i] = 0;
  s.lp.flags[i] = 0;
}

// isotropic safety of a point in slab l: distance to the nearer plane
__device__ inline double Safety(const Slabs& g, int l, double x) {
  return fmax(0.0, fmin(x - g.plane[l], g.plane[l + 1] - x));
}

// Cuts the proposed geometrical step at the next plane along the pre-step
// direction; xend = end point of the straight move, side = +1/-1 when the
// step ends on the upper/lower plane of the slab, 0 inside.
// Moves (l, a, lo = plane[l], hi = plane[l + 1]) to the slab holding x:
// plane[l] <= x < plane[l + 1], clamped to [0, nbins); a = l % nabs. The
// planes increase, so the walk ends at the one slab a bisection would find;
// a gamma's delta step crosses few slabs, so it reads few planes.
__device__ inline void WalkToSlab(const Slabs& g, double x, int& l, int& a, double& lo, double& hi) {
  while (true) {
    if (l < g.nbins - 1 && x >= hi) {
      ++l;
      a = a + 1 == g.nabs ? 0 : a + 1;
      lo = hi;
      hi = g.plane[l + 1];
    } else if (l > 0 && x < lo) {
      --l;
      a = a == 0 ? g.nabs - 1 : a - 1;
      hi = lo;
      lo = g.plane[l];
    } else {
      break;
    }
  }
}

constexpr int kWdtMaxIter = 1 << 20;  // delta steps of one Woodcock step (then: taken to the exit)

// Woodcock tracking of a gamma through the stack
// (G4HepEmWoodcockHelper::KeepTracking, G4HepEm/G4HepEm/src/G4HepEmWoodcockHelper.cc:145-300,
// and its driver, G4HepEmTrackingManager.cc:955-1062), after its HowFar. The
// distance to the stack's exit less 1e-3 mm is eaten up in steps sampled with
// the densest material's total cross section Sigma_w; a point in another
// material is an interaction with probability Sigma/Sigma_w, one in the densest
// material always. On an interaction the gamma moves there (layer l, position
// xe) with the couple, total mean free path and PE cross section of the point;
// on reaching the exit it ends on the stack's boundary (side sd). Either way
// the number of interaction lengths left is reset and the step adds nothing to
// it. Returns false (nothing changed) if the gamma is within 1e-3 + 1e-6 mm of
// the exit (FindWDTVolume, :141-142).
template <typename R>
__device__ bool WoodcockStep(const hepem::DevTables<R>& T, const Slabs& g, hepem::Trk<R>& gt, hepem::Rng& rng, R& pe, int& l,
                             double x, double ux, double& xe, int& sd) {
  using namespace hepem;
  const double distOut = ux > 0.0 ? (g.xmax - x) / ux : (ux < 0.0 ? (0.0 - x) / ux : 1.0e300);
  double dist = distOut - 1.0E-3 > 0.0 ? distOut - 1.0E-3 : 0.0;
  if (!(dist >= 1.0E-6)) return false;
  constexpr R kBig = std::numeric_limits<R>::max();
  Trk<R> xt;  // cross-section evaluations at the gamma's energy
  xt.isEl = false;
  xt.setE(gt.ekin);
  xt.imc = g.wdtImc;
  R wpe = (R)0.0;
  const R wmx = GetTotalMacXSec(T, xt, wpe);
  const R wmfp = wmx > (R)0.0 ? (R)1.0 / wmx : kBig;
  // total and PE cross sections of the other absorbers' couples at this energy
  // (the energy stays the same through the step), ahead of the loop so that
  // its lanes do not diverge over them
  R mxa[HEPEM_SLAB_MAX_ABS], pea[HEPEM_SLAB_MAX_ABS];
#pragma unroll
  for (int k = 0; k < HEPEM_SLAB_MAX_ABS; ++k) {
    mxa[k] = pea[k] = (R)0.0;
    if (k < g.nabs && !((g.wdtMask >> k) & 1u)) {
      xt.imc = g.imc[k];
      mxa[k] = GetTotalMacXSec(T, xt, pea[k]);
    }
  }
  R mfp = wmfp, pint = wpe;
  int lp = l, ap = l % g.nabs, imcp = g.wdtImc;
  double plo = g.plane[l], phi = g.plane[l + 1];
  bool boundary = false;
  double L = 0.0;
  for (int it = 0;; ++it) {
    if (it >= kWdtMaxIter) {
      L += dist;
      boundary = true;
      break;
    }
    const R pstep = wmfp < kBig ? -vlog((R)rng.flat()) * wmfp : kBig;
    if (dist < (double)pstep) {
      L += dist;
      boundary = true;
      break;
    }
    L += (double)pstep;
    dist -= (double)pstep;
    WalkToSlab(g, x + L * ux, lp, ap, plo, phi);
    if (!((g.wdtMask >> ap) & 1u)) {
      const R mx = ap == 0 ? mxa[0] : (ap == 1 ? mxa[1] : (ap == 2 ? mxa[2] : mxa[3]));
      if ((double)(mx * wmfp) > rng.flat()) {
        imcp = AbsorberCouple(g, ap);
        mfp = mx > (R)0.0 ? (R)1.0 / mx : kBig;
        pint = ap == 0 ? pea[0] : (ap == 1 ? pea[1] : (ap == 2 ? pea[2] : pea[3]));
        break;
      }
    } else {
      imcp = g.wdtImc;
      mfp = wmfp;
      pint = wpe;
      break;
    }
  }
  gt.nial[0] = (R)-1.0;
  gt.gstep = (R)0.0;
  if (boundary) {
    sd = ux < 0.0 ? -1 : 1;
    l = sd > 0 ? g.nbins - 1 : 0;
    gt.onBoundary = true;
    xe = sd > 0 ? g.xmax : 0.0;
  } else {
    l = lp;
    gt.imc = imcp;
    gt.mfp[0] = mfp;
    pe = pint;
    gt.onBoundary = false;
    sd = 0;
    xe = x + L * ux;
  }
  return true;
}

// What a slot's step leaves after its final state: kinematics, random stream and
// secondaries for the scatter, and in place of the slot's staged record what the
// end of the round needs of it (its energy, the deposit, the secondaries' number,
// kinds and energies).
template <typename R>
__device__ __forceinline__ void StoreFinal(const hepem_tracks& t, const hepem_step_out& res, int n, int i, const hepem::Trk<R>& k,
                                           const hepem::Rng& rng, const hepem::SecList<R>& sl, double edep, hepem::Staged& r) {
  t.ekin[i] = k.ekin;
#pragma unroll
  for (int c = 0; c < 3; ++c) t.dir[c * n + i] = (double)k.dir[c];
  hepem::StoreRng(t, i, rng);
  r.ekin = k.ekin;
  r.dir[0] = edep;
  r.imc = sl.ns;
  if (sl.ns > 0) {
    hepem::WriteSlot<R>(res, n, i, 0, sl.s0);
    r.dir[1] = sl.s0.ekin;
    r.id = sl.s0.ptype;
  }
  if (sl.ns > 1) {
    hepem::WriteSlot<R>(res, n, i, 1, sl.s1);
    r.dir[2] = sl.s1.ekin;
    r.stream = (uint32_t)sl.s1.ptype;
  }
}
// The arguments of the stepping kernel.
template <typename R> struct MoveArgs {
  Stack s;
  Slabs g;
  hepem_step_out res;
  hepem::DevTables<R> T;
  uint64_t seed;
  int ne, ge;
  unsigned long long *dep, *leak;
  uint8_t* next;
  uint32_t *offE, *offG, *bsumE, *bsumG, *bsec;
};

// Where a slot's move ended, held by its thread to the end of the round.
struct Moved {
  double x;      // position
  int layer;     // the slab the deposit is scored in
  int side;      // +1/-1: on the upper/lower plane of the slab, 0: inside
  bool ended;    // the step ended (an e-/e+ within its sub-steps has not)
};

// Slot i of the e-/e+ part of G4HepEmTrackingManager::TrackElectron's step with
// the slab as the caller's geometry (device/dev_tracking.hh), one sub-step
// per stepping round, after beginning a step if the slot is not within one: the
// pre-step safety (kept in t.safety for the step), the interaction lengths and
// HowFarToDiscreteInteraction; then SlabSubstep (HowFarToMSC, the move, the
// along-step part, the MSC displacement). A slot within a step stays in the stack with its loop state, deposits nothing and
// creates nothing until its step ends; then the end of the step follows here:
// the loss fluctuation on the summed mean loss, at-rest annihilation, or the
// choice of the discrete interaction. Every round thus does one uniform unit of
// work per e-/e+, whatever the length of its sub-step chain. Returns the code of
// an interaction whose final state is pending, with its record at st[j] (and the
// step's deposit in its pe), or 0.
template <typename R>
__device__ __forceinline__ uint8_t ElectronSubstep(int n, int i, Moved& mv, hepem::Staged* st, int j) {
  using namespace hepem;
  ElState<R> el;
  Rng rng;
  StepLoop<R> L;
  SlabPos p;
  int l;
  TrackIn in;
  {
    const MoveArgs<R>& a = KernelArgs<MoveArgs<R>>();
    const Stack& s = a.s;
    const Slabs& g = a.g;
    const hepem_tracks& t = s.t;
    l = s.layer[i];
    in = LoadTrackIn(t, n, i);
    const MscIn q = LoadMscIn(t, i);
    KeepLoaded(in);
    InitElectron(in, q, a.seed, el, rng);
    p = SlabPos{s.x[i], g.plane[l], g.plane[l + 1], l == 0, l == g.nbins - 1, 0};
    const uint8_t f0 = s.lp.flags[i];
    if (!(f0 & kInStep)) {
      SlabBegin(a.T, el, L, rng, p);
      t.safety[i] = (double)el.t.safety;
      s.lp.preEkin[i] = L.preEkin;
      s.lp.iDProc[i] = (int8_t)L.iDProc;
#pragma unroll
      for (int k = 0; k < 4; ++k) s.lp.mfp[k * n + i] = (double)el.t.mfp[k];
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) el.t.mfp[k] = (R)s.lp.mfp[k * n + i];
      el.range = (R)s.lp.range[i];
      el.pstep = (R)s.lp.stepLeft[i];
      el.t.gstep = el.pstep;  // HowFarToMSC keeps it where MSC is off
      el.preEkin = el.t.ekin;
      el.preLEkin = el.t.logE();
      L.iDProc = s.lp.iDProc[i];
      el.t.winner = L.iDProc;
      L.stepLeft = el.pstep;
      L.truePath = (R)0.;
      L.meanLoss = s.lp.meanLoss[i];
      L.preEkin = s.lp.preEkin[i];
      L.preLEkin = (R)0.;
      L.cont = (f0 & kCont) != 0;
      L.stopped = false;
      L.left = false;
      L.nsub = s.lp.nsub[i];
    }
  }
  const bool done = SlabSubstep(KernelArgs<MoveArgs<R>>().T, el, L, rng, p);
  const MoveArgs<R>& a = KernelArgs<MoveArgs<R>>();
  const Stack& s = a.s;
  const hepem_tracks& t = s.t;
  const R rangeLeft = el.range;
  t.on_boundary[i] = p.side != 0 ? 1 : 0;
  mv.x = p.x;
  mv.layer = l;
  mv.side = p.side;
  mv.ended = done;
  {
    const Msc<R>& m = el.msc;
    t.msc_init_range[i] = (double)m.initRange;
    t.msc_dyn_range_factor[i] = (double)m.dynRangeFactor;
    t.msc_tlimit_min[i] = (double)m.tlimitMin;
    t.msc_first_step[i] = m.firstStep ? 1 : 0;
  }
  SecList<R> sl;
  sl.ns = 0;
  double edep = 0.0;
  uint8_t proc = kPNone;
  if (done) {
    L.preLEkin = L.preEkin > 0. ? vlog((R)L.preEkin) : (R)-30;
    s.lp.flags[i] = 0;
    proc = ElectronProc(a.T, el.t, LoopFinishSelect(a.T, el, L, sl, rng));
    edep = el.t.edep;
  } else {
    s.lp.range[i] = (double)rangeLeft;
    s.lp.stepLeft[i] = (double)L.stepLeft;
    s.lp.meanLoss[i] = L.meanLoss;
    s.lp.nsub[i] = L.nsub;
    s.lp.flags[i] = (uint8_t)(kInStep | kCont);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) t.num_ia_left[k * n + i] = (double)el.t.nial[k];
  if (proc != kPNone) {
    const double d[3] = {(double)el.t.dir[0], (double)el.t.dir[1], (double)el.t.dir[2]};
    return StageTrack(st, j, proc, el.t.isEl, el.t.imc, in.id, in.stream, el.t.ekin, d, rng, edep);
  }
  StoreFinal(t, a.res, n, i, el.t, rng, sl, edep, st[j]);
  return kPNone;
}

// One step of gamma slot i, as G4HepEmTrackingManager::TrackGamma
// takes it (G4HepEmTrackingManager.cc:893-1145): HowFar, the cut at the next
// plane along x (or, with Woodcock tracking on and above its energy limit, a
// Woodcock step through the stack), then the boundary update or
// SelectInteraction. The pending interaction as ElectronSubstep's (pe = the PE
// cross section); the slab of the deposit is changed only by a Woodcock step.
template <typename R, bool kWoodcock>
__device__ __forceinline__ uint8_t GammaStep(int n, int i, Moved& mv, hepem::Staged* st, int j) {
  using namespace hepem;
  const MoveArgs<R>& a = KernelArgs<MoveArgs<R>>();
  const Stack& s = a.s;
  const Slabs& g = a.g;
  const hepem_tracks& t = s.t;
  int l = s.layer[i];
  const double x = s.x[i];
  Trk<R> gt;
  gt.isEl = false;
  TrackIn in = LoadTrackIn(t, n, i);
  KeepLoaded(in);
  InitTrack(in, gt);
  Rng rng;
  InitRng(in, a.seed, rng);
  R pe = GammaHowFar(a.T, gt, rng);
  const double ux = (double)gt.dir[0];
  double xe;
  int sd = 0;
  if (!(kWoodcock && gt.ekin > g.wdtMin && WoodcockStep(a.T, g, gt, rng, pe, l, x, ux, xe, sd))) {
    const double gs = (double)gt.gstep;
    double dist = 1.0e300;
    if (ux > 0.0) {
      dist = (g.plane[l + 1] - x) / ux;
      sd = 1;
    } else if (ux < 0.0) {
      dist = (g.plane[l] - x) / ux;
      sd = -1;
    }
    if (dist < gs) {
      gt.gstep = (R)dist;
      gt.onBoundary = true;
      xe = sd > 0 ? g.plane[l + 1] : g.plane[l];
    } else {
      gt.onBoundary = false;
      sd = 0;
      xe = fmin(fmax(x + gs * ux, g.plane[l]), g.plane[l + 1]);
    }
  } else {
    s.layer[i] = l;
    t.imc[i] = gt.imc;
  }
  const uint8_t proc = GammaProc(a.T, gt, pe, rng);
  t.num_ia_left[i] = (double)gt.nial[0];
  t.on_boundary[i] = gt.onBoundary ? 1 : 0;
  mv.x = xe;
  mv.layer = l;
  mv.side = sd;
  mv.ended = true;
  if (proc != kPNone) {
    const double d[3] = {(double)gt.dir[0], (double)gt.dir[1], (double)gt.dir[2]};
    return StageTrack(st, j, proc, false, gt.imc, in.id, in.stream, gt.ekin, d, rng, (double)pe);
  }
  SecList<R> sl;
  sl.ns = 0;
  StoreFinal(t, a.res, n, i, gt, rng, sl, 0.0, st[j]);
  return kPNone;
}

// Block -> slots of a round's stack: the e-/e+ slots [0, ne) in the first `ge`
// blocks, the gammas after them in the others. i = the block's first slot; the
// slots of its kind end before the returned one.
__device__ __forceinline__ int BlockSlots(int n, int ne, int ge, int& i0) {
  const bool isE = (int)blockIdx.x < ge;
  i0 = isE ? (int)blockIdx.x * kB : ne + ((int)blockIdx.x - ge) * kB;
  return isE ? ne : n;
}

// One sub-step of the e-/e+ slots and one step of the gammas (blocks as
// BlockSlots), the final states of the interactions they end in, and the end of
// the round for the block's slots.
//
// Bound by the latency of one wave's chain as long as a round leaves most SIMDs
// with a wave or two, by VALU issue in the largest rounds. In one launch the
// gamma waves run beside the e-/e+ waves instead of after them, and an e-/e+
// whose step ends goes on with its state in registers. The final states are
// sampled by process within the block: a wave with lanes in several processes
// would run their samplers one after the other. The end of the round (a kernel
// of its own read back ten arrays that this one had just written) takes the
// position from registers and the rest from LDS. 1000 showers: 38.1 ms with the
// sorted final states instead of 38.7, 35.1 instead of 36.5 without the kernel
// that ended the round. The arguments are read anew at each stage (MoveArgs): held
// to the end they spilled from scalar registers into VGPR lanes; 33.0 ms became
// 32.1, in the FP32-table form 28.0 became 26.7 (168 -> 153 VGPRs, 128 -> 99).
// Held to 3 waves per SIMD in FP64, 4 in the FP32-table form.
//
// End of the round. The next stack holds the e-/e+ first and the gammas after
// them, each part in slot order of the parents. next[i]: bit s = secondary slot
// s is stacked, kSurvives = the track itself goes on; offE/offG[i] = exclusive
// scans within the block of the e-/e+ and gamma slots track i needs;
// bsumE/bsumG/bsec[block] = the block's totals of those and of its secondaries
// (with the steps that ended in bits 16 and up). Deposits are summed per block
// and (event, slab) before the global atomic; the fixed-point sum does not
// depend on the grouping.
constexpr uint8_t kSurvives = 4;
constexpr int kHash = 2 * kB;
template <typename R, bool kWoodcock>
__global__ void __launch_bounds__(kB, sizeof(R) == sizeof(double) ? 3 : 4)
    k_sh_move(MoveArgs<R>) {
  using namespace hepem;
  __shared__ union {
    BlockFinals<kB> fin;
    struct {
      unsigned long long key[kHash], val[kHash];
    } hash;
  } sh;
  int i0, last;
  bool isE;
  uint8_t code = kPNone;
  Moved mv;
  {
    const MoveArgs<R>& a = KernelArgs<MoveArgs<R>>();
    last = BlockSlots(a.s.t.n, a.ne, a.ge, i0);
    isE = (int)blockIdx.x < a.ge;
  }
  const int i = i0 + (int)threadIdx.x;
  const bool valid = i < last;
  if (isE) {
    if (valid) code = ElectronSubstep<R>(KernelArgs<MoveArgs<R>>().s.t.n, i, mv, sh.fin.st, (int)threadIdx.x);
    SampleBlock<kB, kPIoniEl, kPAnnih>(sh.fin, code, [&](int j, Staged& r, uint8_t c, int proc) HEPEM_INLINE {
      const MoveArgs<R>& a = KernelArgs<MoveArgs<R>>();
      Trk<R> k;
      Rng rng;
      SecList<R> sl;
      sl.ns = 0;
      const double edep = r.pe;
      Unstage(r, c, a.seed, k, rng);
      ElectronFinal(a.T, k, proc, sl, rng);
      const MoveArgs<R>& w = KernelArgs<MoveArgs<R>>();
      StoreFinal(w.s.t, w.res, w.s.t.n, i0 + j, k, rng, sl, edep, r);
    });
  } else {
    if (valid) code = GammaStep<R, kWoodcock>(KernelArgs<MoveArgs<R>>().s.t.n, i, mv, sh.fin.st, (int)threadIdx.x);
    SampleBlock<kB, kPConv, kPPE>(sh.fin, code, [&](int j, Staged& r, uint8_t c, int proc) HEPEM_INLINE {
      const MoveArgs<R>& a = KernelArgs<MoveArgs<R>>();
      Trk<R> k;
      Rng rng;
      SecList<R> sl;
      sl.ns = 0;
      const R pe = (R)r.pe;
      Unstage(r, c, a.seed, k, rng);
      GammaFinal(a.T, k, proc, pe, sl, rng);
      const MoveArgs<R>& w = KernelArgs<MoveArgs<R>>();
      StoreFinal(w.s.t, w.res, w.s.t.n, i0 + j, k, rng, sl, k.edep, r);
    });
  }
  const MoveArgs<R>& a = KernelArgs<MoveArgs<R>>();
  const Stack& s = a.s;
  const Slabs& g = a.g;
  const hepem_tracks& t = s.t;
  __syncthreads();
  const Staged r = sh.fin.st[threadIdx.x];
  __syncthreads();  // the hash table takes the records' place
  const uint32_t ended = valid && mv.ended ? 1u : 0u;
  constexpr unsigned long long kNone = ~0ull;
  unsigned long long key = kNone, val = 0ull;
  uint32_t cE = 0u, cG = 0u, ns = 0u;
  if (valid) {
    const int ev = s.event[i];
    const int l0 = mv.layer;  // the pre-step slab: scoring and the couple's cuts
    int l = l0;
    const double ekin = r.ekin;
    double edep = r.dir[0];
    const int sd = mv.side;
    bool alive = ekin > 0.0;
    int nsec = r.imc;
    if (sd != 0 && (l + sd < 0 || l + sd >= g.nbins)) {
      // leaves the stack: its kinetic energy, the annihilation energy of an e+
      // in flight and anything its last step created are lost
      double e = ekin + (t.ptype[i] == 1 && ekin > 0.0 ? 2.0 * kElectronMass : 0.0);
      if (nsec > 0) e += r.dir[1];
      if (nsec > 1) e += r.dir[2];
      atomicAdd(&a.leak[ev], (unsigned long long)llrint(e * kFix));
      alive = false;
      nsec = 0;
    } else if (alive && sd != 0) {
      l += sd;
    }
    s.x[i] = mv.x;
    s.layer[i] = l;
    // StackSecondaries (G4HepEmTrackingManager.cc:1274-1313): where the
    // couple's region applies cuts, a secondary below its production
    // threshold is deposited at the step instead of stacked (an e+ with its
    // annihilation energy, when the gamma threshold exceeds the electron mass)
    const int ab = l0 % g.nabs;
    uint32_t mask = 0u;
#pragma unroll
    for (int sl = 0; sl < 2; ++sl) {
      if (sl >= nsec) continue;
      const int pt = sl ? (int)r.stream : r.id;
      const double se = sl ? r.dir[2] : r.dir[1];
      bool cut = false;
      if (g.applyCuts[ab]) {
        if (pt == 0) cut = se < g.cutE[ab];
        else if (pt == 1) cut = kElectronMass < g.cutG[ab] && se < g.cutP[ab];
        else cut = se < g.cutG[ab];
      }
      if (cut) {
        edep += pt == 1 ? se + 2.0 * kElectronMass : se;
      } else {
        mask |= 1u << sl;
        ++ns;
        if (pt == 2) ++cG;
        else ++cE;
      }
    }
    a.next[i] = (uint8_t)(mask | (alive ? kSurvives : 0));
    if (alive) {
      if (isE) ++cE;
      else ++cG;
    }
    if (edep > 0.0) {
      key = (unsigned long long)ev * (unsigned long long)g.nbins + (unsigned long long)l0;
      val = (unsigned long long)llrint(edep * kFix);
    }
  }
  // per-block aggregation of the deposits in an LDS hash table (open
  // addressing, at most kB keys in 2 kB entries, so every probe sequence ends):
  // one global atomic per distinct (event, slab) of the block
  for (int e = threadIdx.x; e < kHash; e += kB) {
    sh.hash.key[e] = kNone;
    sh.hash.val[e] = 0ull;
  }
  __syncthreads();
  if (key != kNone) {
    uint32_t h = (uint32_t)((key * 0x9E3779B97F4A7C15ull) >> 55) & (kHash - 1);
    while (true) {
      const unsigned long long prev = atomicCAS(&sh.hash.key[h], kNone, key);
      if (prev == kNone || prev == key) {
        atomicAdd(&sh.hash.val[h], val);
        break;
      }
      h = (h + 1) & (kHash - 1);
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kHash; e += kB) {
    const unsigned long long k = sh.hash.key[e];
    if (k != kNone) atomicAdd(&a.dep[k], sh.hash.val[e]);
  }
  uint32_t xE, xG, tE, tG, tns;
  hepem::BlockScan2<kB>(cE, cG, ns | (ended << 16), xE, xG, tE, tG, tns);
  if (valid) {
    a.offE[i] = xE;
    a.offG[i] = xG;
  }
  if (threadIdx.x == 0) {
    a.bsumE[blockIdx.x] = tE;
    a.bsumG[blockIdx.x] = tG;
    a.bsec[blockIdx.x] = tns;
  }
}
static_assert(std::is_same_v<decltype(k_sh_move<double, false>), void(MoveArgs<double>)>);

// In-place exclusive scans of the nb block sums of e-/e+ and gamma slots by
// one block; the round's secondaries are added to *nsecTotal. The `inject`
// primaries (e-/e+ if injectE) go to the end of their part of the next stack:
// total[0] = tracks of the next stack, total[1] = first slot of the injected
// primaries, total[2] = slots of the e-/e+ part. The track count is also
// written to host memory, followed by `tag` once it is visible there.
constexpr int kScanB = 1024;  // threads of the one-block scan
__global__ void __launch_bounds__(kScanB) k_scan_sums(uint32_t* bsumE, uint32_t* bsumG, const uint32_t* __restrict__ bsec, int nb,
                                                  int inject, int injectE, uint32_t* total, unsigned long long* nsecTotal,
                                                  unsigned long long* nstepsTotal, volatile uint32_t* hostCount, uint32_t tag) {
  __shared__ uint32_t carryE, carryG;
  __shared__ unsigned long long secs, steps;
  if (threadIdx.x == 0) {
    carryE = 0u;
    carryG = 0u;
    secs = 0ull;
    steps = 0ull;
  }
  __syncthreads();
  unsigned long long myEnded = 0ull;
  for (int base = 0; base < nb; base += kScanB) {
    const int i = base + threadIdx.x;
    const uint32_t a = i < nb ? bsumE[i] : 0u;
    const uint32_t b = i < nb ? bsumG[i] : 0u;
    const uint32_t packed = i < nb ? bsec[i] : 0u;  // secondaries | steps ended << 16
    const uint32_t w = packed & 0xFFFFu;
    myEnded += packed >> 16;
    uint32_t xa, xb, ta, tb, tw;
    hepem::BlockScan2<kScanB>(a, b, w, xa, xb, ta, tb, tw);
    if (i < nb) {
      bsumE[i] = carryE + xa;
      bsumG[i] = carryG + xb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      carryE += ta;
      carryG += tb;
      secs += tw;
    }
    __syncthreads();
  }
  for (int o = 32; o > 0; o >>= 1) myEnded += __shfl_xor(myEnded, o, 64);
  if (__lane_id() == 0) atomicAdd(&steps, myEnded);
  __syncthreads();
  if (threadIdx.x == 0) {
    *nstepsTotal += steps;
    const uint32_t k = (uint32_t)inject;
    const uint32_t elen = carryE + (injectE ? k : 0u);
    total[0] = carryE + carryG + k;
    total[1] = injectE ? carryE : elen + carryG;
    total[2] = elen;
    *nsecTotal += secs;
    // the host reads the next round's track count while the scatter runs
    hostCount[0] = carryE + carryG + k;
    hostCount[2] = elen;  // its e-/e+ part
    __threadfence_system();
    hostCount[1] = tag;
  }
}

// Survivor i and its stacked secondaries go to the next e-/e+ slots from
// bsumE[block] + offE[i] and the next gamma slots from total[2] +
// bsumG[block] + offG[i], in the order survivor, secondary 0, secondary 1;
// each starts with the isotropic safety of its position. Writes nothing beyond
// `cap` (the host then reports the overflow).
//
// Bound by latency in small rounds, by its bytes in large ones. Everything is
// loaded before the first store: the arrays may overlap as far as the compiler
// knows, so copied field by field each load waited for the one before it to be
// stored (1000 showers 35.1 ms, now 33.3).
struct ElSlot {  // what an e-/e+ slot carries beyond a gamma's
  double nial[3], initRange, dynRangeFactor, tlimitMin, safety, range, stepLeft, mfp[4], preEkin, meanLoss;
  int32_t nsub;
  int8_t iDProc;
  uint8_t firstStep, flags;
};
__global__ void __launch_bounds__(kB) k_sh_scatter(Stack a, Stack b, Slabs g, hepem_step_out res, int ne, int ge,
                             const uint8_t* __restrict__ next, const uint32_t* __restrict__ offE,
                             const uint32_t* __restrict__ offG, const uint32_t* __restrict__ bsumE,
                             const uint32_t* __restrict__ bsumG, const uint32_t* __restrict__ total, int cap) {
  const int n = a.t.n;
  int i0;
  const int last = BlockSlots(n, ne, ge, i0), i = i0 + (int)threadIdx.x;
  if (i >= last) return;
  const hepem_tracks& s = a.t;
  const hepem_tracks& d = b.t;
  const bool isE = (int)blockIdx.x < ge;
  // A gamma reads only the first interaction-length slot (its total) and
  // neither the safety nor the MSC state: those fields of a gamma slot are not
  // carried.
  const uint32_t mask = next[i];
  const int m = (int)total[0];
  int jE = (int)(bsumE[blockIdx.x] + offE[i]);
  int jG = (int)(total[2] + bsumG[blockIdx.x] + offG[i]);
  const double x = a.x[i], ekin = s.ekin[i], gauss = s.rng_gauss[i], nial0 = s.num_ia_left[i];
  const double dir0 = s.dir[i], dir1 = s.dir[n + i], dir2 = s.dir[2 * n + i];
  const int l = a.layer[i], ev = a.event[i], nstep = a.nstep[i];
  const int32_t id = s.id[i];
  const uint32_t stream = s.rng_stream[i], ctr = s.rng_ctr[i];
  const int8_t pt = s.ptype[i];
  const uint8_t onb = s.on_boundary[i], hasGauss = s.rng_has_gauss[i];
  ElSlot e;
  if (isE) {
    for (int k = 0; k < 3; ++k) e.nial[k] = s.num_ia_left[(k + 1) * n + i];
    e.initRange = s.msc_init_range[i];
    e.dynRangeFactor = s.msc_dyn_range_factor[i];
    e.tlimitMin = s.msc_tlimit_min[i];
    e.firstStep = s.msc_first_step[i];
    e.flags = a.lp.flags[i];
    // within a step: its pre-step safety and the loop state go along
    if ((mask & kSurvives) && (e.flags & kInStep)) {
      e.safety = s.safety[i];
      e.range = a.lp.range[i];
      e.stepLeft = a.lp.stepLeft[i];
      for (int k = 0; k < 4; ++k) e.mfp[k] = a.lp.mfp[k * n + i];
      e.preEkin = a.lp.preEkin[i];
      e.meanLoss = a.lp.meanLoss[i];
      e.nsub = a.lp.nsub[i];
      e.iDProc = a.lp.iDProc[i];
    }
  }
  int8_t secType[2];
  double secE[2], secDir[2][3];
#pragma unroll
  for (int sl = 0; sl < 2; ++sl) {
    if (!((mask >> sl) & 1u)) continue;
    secType[sl] = res.sec_ptype[sl * n + i];
    secE[sl] = res.sec_ekin[sl * n + i];
    for (int c = 0; c < 3; ++c) secDir[sl][c] = res.sec_dir[(c * 2 + sl) * n + i];
  }
  if (m > cap) return;
  const double safety = Safety(g, l, x);
  const int imc = AbsorberCouple(g, l % g.nabs);
  const uint64_t sid = ((uint64_t)stream << 32) | (uint32_t)id;
  const int ns1 = nstep + 1;
  if (mask & kSurvives) {
    const int j = isE ? jE++ : jG++;
    d.ptype[j] = pt;
    d.id[j] = id;
    d.rng_stream[j] = stream;
    d.imc[j] = imc;
    d.ekin[j] = ekin;
    d.dir[j] = dir0;
    d.dir[m + j] = dir1;
    d.dir[2 * m + j] = dir2;
    d.on_boundary[j] = onb;
    d.num_ia_left[j] = nial0;
    bool inStep = false;
    if (isE) {
      for (int k = 0; k < 3; ++k) d.num_ia_left[(k + 1) * m + j] = e.nial[k];
      d.msc_init_range[j] = e.initRange;
      d.msc_dyn_range_factor[j] = e.dynRangeFactor;
      d.msc_tlimit_min[j] = e.tlimitMin;
      d.msc_first_step[j] = e.firstStep;
      inStep = (e.flags & kInStep) != 0;
      b.lp.flags[j] = inStep ? e.flags : (uint8_t)0;
      if (inStep) {
        d.safety[j] = e.safety;
        b.lp.range[j] = e.range;
        b.lp.stepLeft[j] = e.stepLeft;
        for (int k = 0; k < 4; ++k) b.lp.mfp[k * m + j] = e.mfp[k];
        b.lp.preEkin[j] = e.preEkin;
        b.lp.meanLoss[j] = e.meanLoss;
        b.lp.nsub[j] = e.nsub;
        b.lp.iDProc[j] = e.iDProc;
      } else {
        d.safety[j] = safety;
      }
    }
    d.rng_ctr[j] = ctr;
    d.rng_gauss[j] = gauss;
    d.rng_has_gauss[j] = hasGauss;
    b.x[j] = x;
    b.layer[j] = l;
    b.event[j] = ev;
    b.nstep[j] = inStep ? nstep : ns1;  // a step counts once it ends
  }
#pragma unroll
  for (int sl = 0; sl < 2; ++sl) {
    if (!((mask >> sl) & 1u)) continue;
    const uint64_t cid = ChildStream(sid, ns1, sl);
    const bool secIsE = secType[sl] != 2;
    const int j = secIsE ? jE++ : jG++;
    d.ptype[j] = secType[sl];
    d.id[j] = (int32_t)(uint32_t)cid;
    d.rng_stream[j] = (uint32_t)(cid >> 32);
    d.imc[j] = imc;
    d.ekin[j] = secE[sl];
    for (int c = 0; c < 3; ++c) d.dir[c * m + j] = secDir[sl][c];
    d.on_boundary[j] = 0;
    d.num_ia_left[j] = -1.0;
    if (secIsE) {
      d.safety[j] = safety;
      b.lp.flags[j] = 0;
      for (int k = 1; k < 4; ++k) d.num_ia_left[k * m + j] = -1.0;
      d.msc_init_range[j] = 1.0e+21;
      d.msc_dyn_range_factor[j] = 0.04;
      d.msc_tlimit_min[j] = 1.0E-7;
      d.msc_first_step[j] = 1;
    }
    d.rng_ctr[j] = 0u;
    d.rng_gauss[j] = 0.0;
    d.rng_has_gauss[j] = 0;
    b.x[j] = x;
    b.layer[j] = l;
    b.event[j] = ev;
    b.nstep[j] = 0;
  }
}

// Device memory of one run, freed on every exit path: the arrays are asked for
// with get(), then allocated together by commit(). One allocation of 2.3 GB takes
// 0.7 ms with its release; 70 separate ones took 20 ms (18 of them in hipFree),
// a third of a run of 1000 showers.
struct Arena {
  struct Part {
    void** p;
    size_t off;
  };
  std::vector<Part> parts;
  size_t bytes = 0;
  void* base = nullptr;
  Arena() = default;
  Arena(const Arena&) = delete;
  Arena& operator=(const Arena&) = delete;
  ~Arena() {
    if (base) (void)hipFree(base);
  }
  template <typename T> void get(T*& p, size_t n) {
    parts.push_back({reinterpret_cast<void**>(&p), bytes});
    bytes += ((n ? n : 1) * sizeof(T) + 255) & ~size_t(255);
  }
  // false if the memory is not to be had; the arrays are then not set
  bool commit() {
    if (hipMalloc(&base, bytes) != hipSuccess) {
      base = nullptr;
      return false;
    }
    for (const Part& x : parts) *x.p = static_cast<uint8_t*>(base) + x.off;
    return true;
  }
};

// Three words of pinned, device-mapped, coherent host memory: the next round's
// track count, the tag of the round that wrote it and the count's e-/e+ part. Freed on every exit
// path (after the stream has drained).
struct HostCount {
  uint32_t* p = nullptr;  // host address
  uint32_t* d = nullptr;  // device address of the same words
  bool alloc() {
    if (hipHostMalloc(reinterpret_cast<void**>(&p), 64, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) return false;
    p[0] = 0u;
    p[1] = 0u;
    p[2] = 0u;
    return hipHostGetDevicePointer(reinterpret_cast<void**>(&d), p, 0) == hipSuccess;
  }
  ~HostCount() {
    if (p) (void)hipHostFree(p);
  }
  // Waits until a kernel has published `tag`; false on a stream error, or if
  // the stream drained without it.
  bool wait(uint32_t tag, hipStream_t st) const {
    for (uint64_t spin = 1;; ++spin) {
      if (__atomic_load_n(&p[1], __ATOMIC_ACQUIRE) == tag) return true;
      if ((spin & 1023u) == 0u) {
        const hipError_t e = hipStreamQuery(st);
        if (e == hipSuccess) return __atomic_load_n(&p[1], __ATOMIC_ACQUIRE) == tag;
        if (e != hipErrorNotReady) return false;
      }
    }
  }
  uint32_t count() const { return __atomic_load_n(&p[0], __ATOMIC_ACQUIRE); }
  uint32_t electrons() const { return __atomic_load_n(&p[2], __ATOMIC_ACQUIRE); }
};

// Synchronises the stream when the run ends, on every path, before the
// buffers its kernels use are freed.
struct StreamDrain {
  hipStream_t s;
  ~StreamDrain() { (void)hipStreamSynchronize(s); }
};

void AskStack(Arena& A, Stack& s, size_t cap) {
  hepem_tracks& t = s.t;
  t.n = 0;
  A.get(t.ptype, cap);
  A.get(t.id, cap);
  A.get(t.imc, cap);
  A.get(t.ekin, cap);
  A.get(t.dir, 3 * cap);
  A.get(t.safety, cap);
  A.get(t.on_boundary, cap);
  A.get(t.num_ia_left, 4 * cap);
  A.get(t.msc_init_range, cap);
  A.get(t.msc_dyn_range_factor, cap);
  A.get(t.msc_tlimit_min, cap);
  A.get(t.msc_first_step, cap);
  A.get(t.rng_ctr, cap);
  A.get(t.rng_gauss, cap);
  A.get(t.rng_has_gauss, cap);
  A.get(t.rng_stream, cap);
  A.get(s.x, cap);
  A.get(s.layer, cap);
  A.get(s.event, cap);
  A.get(s.nstep, cap);
  A.get(s.lp.range, cap);
  A.get(s.lp.stepLeft, cap);
  A.get(s.lp.mfp, 4 * cap);
  A.get(s.lp.preEkin, cap);
  A.get(s.lp.meanLoss, cap);
  A.get(s.lp.nsub, cap);
  A.get(s.lp.iDProc, cap);
  A.get(s.lp.flags, cap);
}

// Kahan-compensated accumulator
struct Kahan {
  double s = 0.0, c = 0.0;
  void add(double v) {
    const double y = v - c;
    const double t = s + y;
    c = (t - s) - y;
    s = t;
  }
};

}  // namespace

extern "C" int hepem_slab_run(const hepem_ctx* ctx, const hepem_slab_setup* su, int32_t nevents, uint64_t seed,
                              hepem_slab_result* r, void* stream) {
  if (!ctx || !su || !r || !r->edep_sum || !r->edep_sum2 || nevents < 0) return HEPEM_ERR_INVALID;
  if (su->nlayers < 1 || su->nabs < 1 || su->nabs > HEPEM_SLAB_MAX_ABS || su->capacity < 1 || su->events_per_chunk < 1 ||
      !(su->ekin0 > 0.0) || su->primary < 0 || su->primary > 2 || su->refill_below < 0 || !(su->woodcock_min_ekin >= 0.0))
    return HEPEM_ERR_INVALID;
  for (int a = 0; a < su->nabs; ++a)
    if (!(su->thickness[a] > 0.0) || su->imc[a] < 0) return HEPEM_ERR_INVALID;
  const int nbins = su->nlayers * su->nabs;
  const int cap = su->capacity;
  const int chunk = su->events_per_chunk < cap ? su->events_per_chunk : cap;
  const hipStream_t st = static_cast<hipStream_t>(stream);

  std::vector<double> planes((size_t)nbins + 1);
  planes[0] = 0.0;
  for (int k = 0; k < nbins; ++k) planes[k + 1] = planes[k] + su->thickness[k % su->nabs];

  // per-event deposit rows resident at once (events beyond are run afterwards)
  constexpr int64_t kDepBytes = int64_t(1) << 30;
  const int64_t rowBytes = (int64_t)nbins * (int64_t)sizeof(unsigned long long);
  int64_t span = kDepBytes / rowBytes;
  if (span < chunk) span = chunk;
  if (span > nevents) span = nevents;
  if (span < 1) span = 1;
  const int refill = su->refill_below;
  int growRounds = -1;  // rounds from stacking the first events to their largest stack (-1: not yet seen)

  Arena A;
  Stack s[2];
  hepem_step_out res;  // the secondaries, from the stepping kernel to the scatter
  res.true_step = nullptr;
  res.geom_step = nullptr;
  res.winner = nullptr;
  res.displacement = nullptr;
  res.stopped = nullptr;
  res.edep = nullptr;
  res.nsec = nullptr;
  double* dPlanes;
  uint8_t* goesOn;
  uint32_t *offs, *bsum, *bsec, *total;  // offs: e-/e+ then gamma block offsets (2 x cap); bsum: 2 x nblk
  unsigned long long *dep, *leak, *nsec;
  const int nblk = (cap + kB - 1) / kB + 1;  // the e-/e+ and the gamma part of a round each end with a block
  AskStack(A, s[0], (size_t)cap);
  AskStack(A, s[1], (size_t)cap);
  A.get(res.sec_ptype, 2 * (size_t)cap);
  A.get(res.sec_ekin, 2 * (size_t)cap);
  A.get(res.sec_dir, 6 * (size_t)cap);
  A.get(dPlanes, planes.size());
  A.get(goesOn, (size_t)cap);
  A.get(offs, 2 * (size_t)cap);
  A.get(bsum, 2 * (size_t)nblk);
  A.get(bsec, (size_t)nblk);
  A.get(total, 3);
  A.get(dep, (size_t)span * nbins);
  A.get(leak, (size_t)span);
  A.get(nsec, 2);
  if (!A.commit()) return HEPEM_ERR_ALLOC;
  HostCount hc;  // next round's track count, published by k_scan_sums
  if (!hc.alloc()) return HEPEM_ERR_ALLOC;
  StreamDrain drain{st};  // declared last: drains the stream before hc and A are freed
  uint32_t tag = 0;
  SH_OK(hipMemcpy(dPlanes, planes.data(), planes.size() * sizeof(double), hipMemcpyHostToDevice));

  Slabs g;
  g.nbins = nbins;
  g.nabs = su->nabs;
  for (int a = 0; a < HEPEM_SLAB_MAX_ABS; ++a) {
    g.imc[a] = a < su->nabs ? su->imc[a] : 0;
    g.cutE[a] = g.cutP[a] = g.cutG[a] = 0.0;
    g.applyCuts[a] = 0;
    if (a < su->nabs) {
      double cuts[3];
      if (HepemCoupleCuts(ctx, su->imc[a], cuts, &g.applyCuts[a]) != HEPEM_OK) return HEPEM_ERR_INVALID;
      g.cutE[a] = cuts[0];
      g.cutP[a] = cuts[1];
      g.cutG[a] = cuts[2];
    }
  }
  g.plane = dPlanes;
  // Woodcock tracking: the stack is one envelope whose densest material (the
  // first absorber of the largest density, G4HepEmWoodcockHelper::FindWDTMaterial,
  // G4HepEmWoodcockHelper.cc:318-338) sets the majorant cross section
  g.wdtMin = su->woodcock_min_ekin;
  g.xmax = planes[(size_t)nbins];
  g.wdtImc = su->imc[0];
  g.wdtMat = -1;
  {
    double maxDensity = -1.0;
    for (int a = 0; a < HEPEM_SLAB_MAX_ABS; ++a) {
      g.mat[a] = -1;
      if (a >= su->nabs) continue;
      double density;
      if (HepemCoupleMaterial(ctx, su->imc[a], &g.mat[a], &density) != HEPEM_OK) return HEPEM_ERR_INVALID;
      if (density > maxDensity) {
        maxDensity = density;
        g.wdtMat = g.mat[a];
        g.wdtImc = su->imc[a];
      }
    }
    g.wdtMask = 0u;
    for (int a = 0; a < su->nabs; ++a)
      if (g.mat[a] == g.wdtMat) g.wdtMask |= 1u << a;
  }
  const bool woodcock = g.wdtMin > 0.0;
  const bool fp64 = HepemPrecision(ctx) == HEPEM_FP64;

  std::vector<Kahan> ks(nbins), ks2(nbins);
  Kahan kleak, ktot;
  std::vector<unsigned long long> hdep((size_t)span * nbins), hleak((size_t)span);
  r->steps = 0;
  r->tracks = 0;
  r->substeps = 0;
  r->iterations = 0;
  r->max_in_flight = 0;
  unsigned long long hnsec[2] = {0ull, 0ull};  // secondaries stacked, steps ended
  hipLaunchKernelGGL(k_sh_fill64, dim3(1), dim3(kB), 0, st, reinterpret_cast<int64_t*>(nsec), 2);

  for (int64_t s0 = 0; s0 < nevents; s0 += span) {
    const int ns = (int)((nevents - s0) < span ? (nevents - s0) : span);
    hipLaunchKernelGGL(k_sh_fill64, dim3((unsigned)(((int64_t)ns * nbins + kB - 1) / kB)), dim3(kB), 0, st,
                       reinterpret_cast<int64_t*>(dep), ns * nbins);
    hipLaunchKernelGGL(k_sh_fill64, dim3((ns + kB - 1) / kB), dim3(kB), 0, st, reinterpret_cast<int64_t*>(leak), ns);
    int next = 0;  // next event of this span to stack
    int n = 0;     // tracks in flight
    int ne = 0;    // the e-/e+ among them (the first ne slots)
    int cur = 0;
    int rounds = 0;
    int sinceInject = 0;  // rounds stepped since primaries were last stacked
    while (true) {
      if (n == 0) {
        if (next >= ns) break;
        const int k = (ns - next) < chunk ? (ns - next) : chunk;
        s[cur].t.n = k;
        hipLaunchKernelGGL(k_sh_inject, dim3((k + kB - 1) / kB), dim3(kB), 0, st, s[cur], g, su->primary, su->ekin0,
                           (int)(s0 + next), next, k, nullptr, nullptr, cap);
        SH_OK(hipGetLastError());
        r->tracks += k;
        next += k;
        n = k;
        ne = su->primary != 2 ? k : 0;
        rounds = 0;
        sinceInject = 0;
      }
      // every step of an e-/e+ loses energy and every gamma step ends on a plane
      // or in an interaction, so the tracks in flight run out; the bound only
      // turns a broken invariant into an error instead of an endless loop
      if (++rounds > kMaxRounds) return HEPEM_ERR_CAPACITY;
      if (n > r->max_in_flight) r->max_in_flight = n;
      Stack& a = s[cur];
      Stack& b = s[cur ^ 1];
      a.t.n = n;
      // the e-/e+ part of the stack comes first
      const int ge = (ne + kB - 1) / kB, gg = (n - ne + kB - 1) / kB;
      const auto move = [&](auto kernel, const auto& T) {
        hipLaunchKernelGGL(kernel, dim3(ge + gg), dim3(kB), 0, st,
                           {a, g, res, T, seed, ne, ge, dep, leak, goesOn, offs, offs + cap, bsum, bsum + nblk, bsec});
      };
      if (fp64) move(woodcock ? k_sh_move<double, true> : k_sh_move<double, false>, HepemTables64(ctx));
      else move(woodcock ? k_sh_move<float, true> : k_sh_move<float, false>, HepemTables32(ctx));
      r->substeps += ne;
      // primaries of the next events join once the stack runs low, and no
      // sooner after the last ones than the first events took to reach their
      // largest stack: the stack then stays below about refill plus one chunk's
      // largest stack
      const bool refillNow = refill > 0 && n < refill && next < ns && growRounds >= 0 && sinceInject >= growRounds;
      const int k = refillNow ? ((ns - next) < chunk ? (ns - next) : chunk) : 0;
      ++tag;
      hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScanB), 0, st, bsum, bsum + nblk, bsec, ge + gg, k, su->primary != 2 ? 1 : 0,
                         total, nsec, nsec + 1, hc.d, tag);
      hipLaunchKernelGGL(k_sh_scatter, dim3(ge + gg), dim3(kB), 0, st, a, b, g, res, ne, ge, goesOn, offs, offs + cap, bsum,
                         bsum + nblk, total, cap);
      if (k > 0) {
        hipLaunchKernelGGL(k_sh_inject, dim3((k + kB - 1) / kB), dim3(kB), 0, st, b, g, su->primary, su->ekin0,
                           (int)(s0 + next), next, k, total + 1, total, cap);
        r->tracks += k;
        next += k;
        rounds = 0;
      }
      SH_OK(hipGetLastError());
      // the next round is enqueued as soon as its size is known; stream order
      // keeps it behind this round's scatter
      if (!hc.wait(tag, st)) return HEPEM_ERR_HIP;
      const uint32_t m = hc.count();
      r->iterations += 1;
      if (m > (uint32_t)cap) return HEPEM_ERR_CAPACITY;
      if (growRounds < 0 && (int)m < n) growRounds = sinceInject + 1;  // the stack shrank for the first time
      sinceInject = k > 0 ? 0 : sinceInject + 1;
      n = (int)m;
      ne = (int)hc.electrons();
      cur ^= 1;
    }
    SH_OK(hipMemcpyAsync(hdep.data(), dep, (size_t)ns * nbins * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
    SH_OK(hipMemcpyAsync(hleak.data(), leak, (size_t)ns * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
    SH_OK(hipStreamSynchronize(st));
    if (r->edep_event)
      for (size_t k = 0; k < (size_t)ns * nbins; ++k) r->edep_event[(size_t)s0 * nbins + k] = (int64_t)hdep[k];
    if (r->leak_event)
      for (int e = 0; e < ns; ++e) r->leak_event[s0 + e] = (int64_t)hleak[e];
    for (int e = 0; e < ns; ++e) {
      for (int k = 0; k < nbins; ++k) {
        const double v = (double)hdep[(size_t)e * nbins + k] / kFix;
        ks[k].add(v);
        ks2[k].add(v * v);
        ktot.add(v);
      }
      kleak.add((double)hleak[e] / kFix);
    }
  }
  SH_OK(hipMemcpyAsync(hnsec, nsec, 2 * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
  SH_OK(hipStreamSynchronize(st));
  r->tracks += (int64_t)hnsec[0];
  r->steps = (int64_t)hnsec[1];
  for (int k = 0; k < nbins; ++k) {
    r->edep_sum[k] = ks[k].s;
    r->edep_sum2[k] = ks2[k].s;
  }
  r->leak_sum = kleak.s;
  r->edep_total = ktot.s;
  return HEPEM_OK;
}
