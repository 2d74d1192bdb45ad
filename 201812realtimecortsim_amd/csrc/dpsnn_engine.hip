// dpsnn_engine.hip -- MI355X engine for DPSNN's per-millisecond LIFCA step.
//
// One network = one process's whole local network on one GPU.  Step t (one
// reference completeTimeStep_ms, DPSNN_localNet_sim.c:22-307) is:
//
//   k_bath         the step's external events (DPSNN_neuron_sim.c:604-640).
//   phase 1        per target neuron, the items of its in-list (delivery
//                  insertion order) whose source fired in step t-delay,
//                  ordered with the bath by arrival time (wave-wide bucket
//                  sort in LDS on exact 64-bit keys; internal first on ties):
//                  k_gather, or for large networks k_collect + k_sort.
//                  Replaces delivery + addInputSpike (:837-999,
//                  DPSNN_neuron_sim.c:289-300).
//   phase 2        LIFCADynamic per event in FP64, one lane per neuron:
//                  k_integrate_records, k_integrate_pipe or (bath merged
//                  here) k_integrate.  Replaces regularDynamicTimeStep +
//                  LIFCADynamic (:522-824).  Its tail is the fired scan of
//                  step t+1: each wave ballots its 64 neurons' spikes into
//                  one word of the spike bitmap of slot t+1, stores their
//                  emission times in the slot's Te history, the last-spike ms
//                  and the per-(column, subPop) counts.  That replaces the
//                  fired scan + compaction + world-size-1 axonal exchange +
//                  ring insert (:103-148, :620-806, DPSNN_spike.c:209-239).
//   k_ltp, k_stdp  STDP of a step, or of a block of steps at once
//                  (DPSNN_neuron_sim.c:94-277).
//   k_step         phases 1 and 2 in one launch (an option).
//   k_compact      (only when a raster is wanted) ascending spike list of
//                  slot t+1 appended to the device raster buffer.
//   k_commit       (STDP, ms % 1000 == 999) the per-second weight commit.
//
// The device holds no per-step event queue: a target pulls its live events
// from its static in-list and the spike history (bitmap + Te per slot), so
// the only per-step traffic is the in-list stream, the history lookups and
// the neuron state.  Built with -ffp-contract=off: the reference's FP64
// update is second order and unfused, and must round where it rounds.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "dpsnn_exp.h"
#include "dpsnn_hip.h"
#include "dpsnn_host.h"

namespace dpsnn {

constexpr int kBlock = 256;      // integrate / scan block (4 waves)
constexpr uint32_t kPad = 0xFFFFFFFFu;
constexpr int kExtRing = 8;      // replayed external steps in flight
constexpr uint32_t kMaxInList = 3900;  // per-neuron in-list (12-bit key field, LDS)

static thread_local std::string g_err;
static int fail(int code, const char *fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}
#define HIP_TRY(expr)                                                              \
  do {                                                                             \
    hipError_t e_ = (expr);                                                        \
    if (e_ != hipSuccess)                                                          \
      return fail(DPSNN_ERR_DEVICE, "%s failed: %s", #expr, hipGetErrorString(e_)); \
  } while (0)

constexpr int kWave = 64;
constexpr double kNotFired = -1.0;  // Te history entry of a neuron that did not fire (spike times are >= 0)

// XCD-aware persistent walk over work items [0, total).  The dispatcher deals
// workgroups to the 8 XCDs round-robin (workgroup b on XCD b % 8), and each
// XCD has its own L2: the blocks of one XCD walk one contiguous eighth of
// the items, so neighbouring neurons, which share most of their sources,
// read the spike history through the same L2.  gridDim.x is a multiple of 8.
constexpr uint32_t kXcds = 8;
struct XcdWalk {
  uint32_t first, end, stride;
};
__device__ inline XcdWalk xcd_walk(uint32_t total) {
  const uint32_t x = blockIdx.x % kXcds, lb = blockIdx.x / kXcds, per = gridDim.x / kXcds;
  const uint32_t begin = (uint32_t)((uint64_t)total * x / kXcds);
  const uint32_t end = (uint32_t)((uint64_t)total * (x + 1) / kXcds);
  return XcdWalk{begin + lb, end, per};
}

// XCD-ordered work queue over items [0, total): XCD x (= blockIdx.x % 8, as
// the dispatcher deals workgroups) owns the x-th contiguous eighth, and its
// waves take the items in order from the XCD's counter, so the items in
// flight on one XCD stay a narrow window (neighbouring neurons, shared
// sources, one L2).  An XCD whose eighth is exhausted helps the next ones.
// A wave takes a run of consecutive items per counter update (guided: a
// share of what is left of the range for each of the XCD's waves, between
// kGrabMin and kGrabMax, so that counter updates are few while much is left
// and the tail stays balanced); next_item returns the first item and the
// run's end (*last), or `total` when none is left.  Whole wave; ctr holds
// kXcds counters that are zero at the launch.  Each counter sits on its own
// 128-byte line (ctr[x * kCtrStride]); an exhausted counter is recognised by
// a plain read before any atomic.  The counters live in device-coherent
// memory, where each update costs a round trip: with runs of 4, the 24x24-column network's
// phase 1 was 9% slower than with the guided runs, with runs of 1 twice as
// slow.
constexpr uint32_t kGrabMin = 4, kGrabMax = 16;
// Up to this many targets per wave, k_gather deals them out in a fixed strided
// order instead: with the queue's runs of four, 5,000 targets keep half of
// the resident waves busy with four each (ms per step, queue and fixed order:
// 1,250 neurons 0.27 and 0.23, 5,000 neurons 0.187 and 0.163; 31,250 neurons,
// 12 targets a wave: 0.51 and 0.55).
constexpr uint32_t kStaticTargets = 4;
constexpr uint32_t kCtrStride = 32;
__device__ inline uint32_t next_item(uint32_t *ctr, uint32_t total, uint32_t &x, uint32_t home, uint32_t *last) {
  const uint32_t wavesPerXcd = max(1u, gridDim.x * (blockDim.x / 64u) / kXcds);
  for (;;) {
    const uint32_t begin = (uint32_t)((uint64_t)total * x / kXcds);
    const uint32_t end = (uint32_t)((uint64_t)total * (x + 1) / kXcds);
    uint32_t *c = ctr + x * kCtrStride;
    uint32_t k = end - begin, g = kGrabMin;
    if ((threadIdx.x & 63) == 0) {
      k = __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (begin + k < end) {
        g = min(kGrabMax, max(kGrabMin, (end - begin - k) / (2u * wavesPerXcd)));
        k = atomicAdd(c, g);
      }
    }
    k = __builtin_amdgcn_readfirstlane(k);  // lane 0's values, known uniform (scalar registers)
    g = __builtin_amdgcn_readfirstlane(g);
    if (begin + k < end) {
      *last = min(end, begin + k + g);
      return begin + k;
    }
    x = (x + 1) % kXcds;
    if (x == home) return total;
  }
}

// LDS written by some lanes of a wave and read by others: order the wave's
// accesses around this point.  The one-wave workgroups of phase 1 use it in
// place of __syncthreads(), whose workgroup-scope fence would also wait for
// every global load in flight (the records loaded ahead for the next target).
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
constexpr int kWaveLTP = 256;    // STDP kernels: 4 waves per block

// Per-sub-population LIFCA parameters, in this order.
enum { kTheta, kH, kTarp, kAlphaC, kGC, kInvTau, kInvTauLo, kInvTauC, kInvTauCLo, kParams };

struct DevNet {
  uint32_t N, NW, RS, nsub, npc, ncols, cap, drive;
  uint32_t denseMax;       // phase 1 takes its fast path for up to this many live items (<= kDense * 64)
  float w2f;
  uint64_t philoxSeed;
  const uint8_t *subPop;
  const double *sp;        // [nsub][kParams]
  const double *lut;       // [nsub][256]
  const double *invNuExt;
  const uint32_t *maxExt;
  // The bath of a step with packed records drawn ahead of phase 1 (k_bath),
  // which sorts it in among the internal events; null: phase 2 draws and
  // merges it
  double *bathT;           // [bath cap][N] event times
  uint32_t *bathN;         // [N] their count
  const float *bathV;      // [nsub] their value (one per sub-population)
  double *v, *c, *Tr, *Te, *assigned;
  uint64_t *philoxCtr;
  uint64_t *bits;          // [RS][NW], RS a power of two
  double *teHist;          // [RS][N] emission time, or kNotFired
  const uint64_t *inOff;   // [N+1] start of each neuron's in-list
  const uint32_t *inPD;    // pre | delay << 24, in delivery insertion order (padded by one wave)
  const int16_t *inW;      // (padded by one wave)
  uint64_t *keys;          // sorted event ticks, per tile of 64 neurons [cap/kRun][64][kRun];
                           // from step kPackT on tick << 16 | weight
  int16_t *keyW;           // their weights before step kPackT, same layout
  uint16_t *keyPos;        // STDP, general path: their in-list positions, same layout
  uint32_t *keyCount;      // [grid][64] or [N/64][64]
  uint32_t *workCtr;       // [kXcds][kCtrStride] phase-1 work counters (zero between steps)
  unsigned long long *counters;  // [kCounterSlots][kCounterStride]: [0] events, [1] external, [2] spikes
  // STDP (null when plasticity never runs).  Synapse state is kept in
  // target-major order: synapse k of neuron j's incoming list lives at
  // incOff[j] + k; in-list items name it by k (inSyn).
  int32_t *lastSpike;      // [N] last emission step (ms) of each neuron
  uint32_t *spikeMask;     // [N] bit b: the neuron fired in slot t1 - b (t1: the last scan)
  int32_t *lastSpike0;     // [N] lastSpike where the block of deferred steps began (k_stdp)
  const uint64_t *incOff;  // [N+1]
  int16_t *wT;
  float *tdT, *tdPre;      // timeDerivative; tdPre: before the decay (probes)
  int32_t *lastT;          // lastActivationTime
  const uint8_t *kindT;    // presynaptic sub-population
  const uint16_t *inSyn;   // per in-list item
  const float *causal, *anti;        // [128] each
  const float *maxSyn, *revMax;      // [nsub][nsub]
  float f2w, drift, decayMul;
  int decayReset;
  // Stencil-window form of phase 1 (k_collect + k_sort; null when the
  // network has no window layout): the in-lists regrouped per unit of
  // targets of one column, per pass (run delay, descending) and per wave,
  // in padded chunks of kWindowChunk items (window index << 16 | weight).
  const uint32_t *winItem;
  const uint16_t *winDesc;   // per chunk: its target's index in the unit
  const uint64_t *winChunk;  // [units][passes][kWindowWaves] + 1: first chunk
  const int32_t *winCols;    // [columns][slots]: source column of each stencil slot, or -1
  uint32_t winSlots, winPasses, winUnit, winUnitsPerCol, winUnits;
  uint32_t *winCtr;          // [kXcds][kCtrStride] unit counters (zero between steps)
  uint32_t *bigList;         // [N] targets k_sort leaves to k_sort_big
  uint32_t *bigCount;        // their count (zero between steps)
  uint32_t sortCap;          // k_sort keeps targets of up to this many records (<= kSortCap)
  uint32_t fuseSort;         // 1: k_collect sorts each unit's targets itself (no k_sort)
  // Steps replayed from a captured graph count from the t that stands here
  // (the kernel argument is then the step's place in the graph); null: t is
  // the argument.
  const uint32_t *tDev;
};

// The step's counters are spread over kCounterSlots cache lines (a block
// adds to the line of blockIdx % kCounterSlots; the host sums them), so
// that the per-wave updates of one step do not all queue on one line.
constexpr uint32_t kCounterSlots = 16, kCounterStride = 16;
__device__ inline unsigned long long *counter_slot(unsigned long long *counters) {
  return counters + (blockIdx.x % kCounterSlots) * kCounterStride;
}

// --------------------------------------------------------------------------
// Philox4x32-10 (Salmon et al., SC'11): counter-based stream for the
// on-device external drive.  Key = (seed, neuron), counter = call index.
// --------------------------------------------------------------------------
__device__ inline void philox4x32(uint32_t c[4], uint32_t k0, uint32_t k1) {
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c[0], p1 = (uint64_t)0xCD9E8D57u * c[2];
    const uint32_t h0 = (uint32_t)(p0 >> 32), l0 = (uint32_t)p0;
    const uint32_t h1 = (uint32_t)(p1 >> 32), l1 = (uint32_t)p1;
    c[0] = h1 ^ c[1] ^ k0;
    c[1] = l1;
    c[2] = h0 ^ c[3] ^ k1;
    c[3] = l0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

struct PhiloxStream {
  uint32_t k0, k1;
  uint64_t ctr;
  double spare;  // second uniform of the last block
  int have;
  // one block: two uniforms in [0, 1)
  __device__ inline void block(double &first, double &second) {
    uint32_t c[4] = {(uint32_t)ctr, (uint32_t)(ctr >> 32), 0u, 0x44505300u};
    philox4x32(c, k0, k1);
    ++ctr;
    const uint64_t a = ((uint64_t)c[0] << 21) ^ (uint64_t)c[1];
    const uint64_t b = ((uint64_t)c[2] << 21) ^ (uint64_t)c[3];
    first = (double)(a & ((1ull << 53) - 1)) * 0x1p-53;
    second = (double)(b & ((1ull << 53) - 1)) * 0x1p-53;
  }
  __device__ double next() {
    if (have) {
      have = 0;
      return spare;
    }
    double first;
    block(first, spare);
    have = 1;
    return first;
  }
};

// a / b, correctly rounded (as IEEE division), for a normal b with
// y = RN(1/b) and a / b within the normal range: q0 = RN(a y) is within two
// ulps of a / b; one correction q1 = RN(q0 + (a - b q0) y) makes it faithful;
// the second, q2 = RN(q1 + r1 y) with the exact residual r1 = a - b q1, is
// RN(a / b) (Markstein's theorem: q faithful, y = RN(1/b)).  Five FMA-unit
// operations instead of the general division's scaled Newton sequence.
__device__ inline double div_rn(double a, double b, double y) {
  const double q0 = a * y;
  const double q1 = fma(fma(-q0, b, a), y, q0);
  return fma(fma(-q1, b, a), y, q1);
}

// a / b, correctly rounded, for a divisor whose significand has an odd part B
// below 2^50 (every float, so every time constant DPSNN reads), with
// yh = RN(1/b) and yl = RN(1/b - yh).  a yh + RN(a yl) is within 2^-105 of
// a / b relative, 2^-52 of an ulp of the quotient, and one fma rounds it.
// A midpoint m between two doubles is further away: with a = A 2^i, A < 2^53,
// b = B 2^j, |a / b - m| B is a non-zero multiple of half an ulp (i - j is at
// least the exponent of that half ulp, or A would need 54 bits; a tie would
// need A >= 2^53 too), so |a / b - m| >= ulp / (2 B).  Two FMA-unit operations
// in place of div_rn's five.
__device__ inline double div_short(double a, double yh, double yl) { return fma(a, yh, a * yl); }
// The divisor's odd significand part is below 2^50 (see div_short).
static inline bool short_divisor(double b) {
  int e;
  const double m = std::frexp(std::fabs(b), &e);  // m 2^53 is an integer
  return std::ldexp(m, 50) == std::floor(std::ldexp(m, 50));
}

// --------------------------------------------------------------------------
// LIFCADynamic, DPSNN_neuron_sim.c:664-824 (second-order, non-Perseo path).
// The divisions by Tau and TauC use their reciprocals (div_short); the
// results are the IEEE quotients.  expTab: dpsnn_exp's table, in LDS.
// --------------------------------------------------------------------------
typedef __attribute__((address_space(3))) double lds_f64;
typedef __attribute__((address_space(3))) uint64_t lds_u64;
typedef __attribute__((address_space(3))) int16_t lds_i16;
struct Lifca {
  double v, c, Tr, Te;
  double Theta, H, Tarp, AlphaC, gC, invTau, invTauLo, invTauC, invTauCLo;
  const lds_u64 *expTab;
  uint32_t fired;
  __device__ inline void load(const DevNet &P, uint32_t j) {
    const double *prm = P.sp + (size_t)P.subPop[j] * kParams;
    v = P.v[j]; c = P.c[j]; Tr = P.Tr[j]; Te = P.Te[j];
    Theta = prm[kTheta]; H = prm[kH]; Tarp = prm[kTarp]; AlphaC = prm[kAlphaC]; gC = prm[kGC];
    invTau = prm[kInvTau]; invTauLo = prm[kInvTauLo];
    invTauC = prm[kInvTauC]; invTauCLo = prm[kInvTauCLo];
  }
  // What an event takes from the time since the one before it alone: half
  // of it, that over Tau, and the factor c decays by.
  __device__ inline void decay(double deltaT, double &dtHalf, double &rmHalf, double &cDecay) const {
    dtHalf = deltaT / 2;
    rmHalf = div_short(dtHalf, invTau, invTauLo);
    const double rc = div_short(deltaT, invTauC, invTauCLo);
    cDecay = 1 - rc + rc * rc / 2;
  }
  // Both of the reference's branches (out of / in the refractory period)
  // decay c by the same expression; the out-of-refractory one also moves v.
  // The lanes of a wave take different branches, so v's update is computed
  // for every lane and kept where the neuron is out of its refractory
  // period: the same operations in the same order, without divergent
  // control flow.  Only the refractory exit (exp) stays a branch; it is rare.
  // A lane without an event (on = false) passes t = Tr: no time elapses, so
  // c is multiplied by one, and v and Te are kept; nothing changes.  AHEAD:
  // dtHalf, rmHalf and cDecay are decay(t - Tr)'s, already computed.
  template <bool AHEAD = false>
  __device__ __attribute__((always_inline)) inline void event(bool on, double t, double I, double dtHalf = 0,
                                                              double rmHalf = 0, double cDecay = 0) {
    double deltaT = t - Tr;
    const double TFLES = t - Te;
    const bool active = on && TFLES > Tarp;
    if (active && Tr - Te < Tarp) {
      c *= dpsnn_exp_with(div_short(-(deltaT - TFLES + Tarp), invTauC, invTauCLo), expTab);
      deltaT = TFLES - Tarp;
      if (AHEAD) decay(deltaT, dtHalf, rmHalf, cDecay);
    }
    if (!AHEAD) decay(deltaT, dtHalf, rmHalf, cDecay);
    double w = v - v * rmHalf - gC * c * dtHalf;
    w = w - w * rmHalf - gC * c * dtHalf;
    w += I;
    // (kept here: the compiler would move v's update under a branch on
    // `active`, apart from c's, and lose what overlaps the two)
    asm volatile("" : "+v"(w));
    c = c * cDecay;
    const bool fire = active && w >= Theta;
    v = fire ? H : (active ? w : v);
    c = fire ? c + AlphaC : c;
    Te = fire ? t : Te;
    fired = fire ? 1u : fired;
    Tr = t;
  }
};

// --------------------------------------------------------------------------
// Fired scan of step t1 = t + 1, run by the wave that integrated 64
// consecutive neurons j0..j0+63 (j0 % 64 == 0) in step t: one bitmap word,
// the emission times of the neurons that fired, their last-spike ms
// (setLastEmittedSpikeTime_ms, DPSNN_neuron_init.c:200-202) and the
// per-(column, subPop) counts.  Every word of the slot and every neuron's
// entry in the slot's Te history (its emission time, or kNotFired) is
// written by exactly one wave, so the slot needs no clearing.  Whole wave,
// uniform.
// --------------------------------------------------------------------------
__device__ __attribute__((always_inline)) inline uint64_t publish_spikes(const DevNet &P, uint32_t t1, uint32_t j, bool f, double te,
                                          uint32_t *popCnt, int count) {
  const uint64_t mask = __ballot(f);
  const uint32_t slot = t1 & (P.RS - 1);
  if ((threadIdx.x & 63) == 0 && (j >> 6) < P.NW) {
    P.bits[(size_t)slot * P.NW + (j >> 6)] = mask;
    if (mask && count) atomicAdd(counter_slot(P.counters) + 2, (unsigned long long)__popcll(mask));
  }
  if (j < P.N) P.teHist[(size_t)slot * P.N + j] = f ? te : kNotFired;
  if (P.spikeMask && j < P.N) {
    P.spikeMask[j] = P.spikeMask[j] << 1 | (f ? 1u : 0u);
    if (f) P.lastSpike[j] = (int32_t)t1;
  }
  if (popCnt && mask) {
    // one counter update per distinct (column, sub-population) among the
    // wave's fired lanes (64 consecutive neurons span at most a few)
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t key = f ? (j / P.npc) * P.nsub + P.subPop[j] : 0u;
    uint64_t pending = mask;
    while (pending) {
      const uint32_t lead = (uint32_t)__ffsll((long long)pending) - 1;
      const uint32_t k = (uint32_t)__shfl((int)key, (int)lead);
      const uint64_t same = __ballot(f && key == k) & pending;
      if (lane == lead) atomicAdd(&popCnt[k], (uint32_t)__popcll(same));
      pending &= ~same;
    }
  }
  return mask;
}

// --------------------------------------------------------------------------
// STDP.  LTP (causalSTDP_ms_ofBackwardSynapses, DPSNN_neuron_sim.c:94-177):
// when the scan of step t finds that neuron j fired (in step t-1's
// dynamics), each incoming synapse with lastActivationTime != 0 gets
// timeDerivative += causal[t - 1 - last] (0 past the 128 ms table).  One
// wave per firing neuron, its incoming synapses contiguous.
// --------------------------------------------------------------------------
__device__ __attribute__((always_inline)) inline void ltp_neuron(const DevNet &P, uint32_t t, uint32_t j) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t end = P.incOff[j + 1];
  constexpr int U = 4;  // independent synapses per lane per round: loads first, then stores
  for (uint64_t s0 = P.incOff[j] + lane; s0 < end; s0 += U * kWave) {
    int32_t last[U];
    float td[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t s = s0 + (uint64_t)u * kWave;
      last[u] = s < end ? P.lastT[s] : 0;
      td[u] = s < end ? P.tdT[s] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t s = s0 + (uint64_t)u * kWave;
      if (s < end) {
        float f = 0.0f;
        if (last[u] != 0) {
          const int dt = (int)t - 1 - last[u];
          if (dt < kStdpSpan) f = P.causal[dt];
        }
        P.tdT[s] = td[u] + f;
      }
    }
  }
}

// LTP of the scan at step t for the neurons of one bitmap word (whole wave).
__device__ inline void ltp_word(const DevNet &P, uint32_t t, uint64_t mask, uint32_t j0) {
  while (mask) {
    const uint32_t b = (uint32_t)__ffsll((long long)mask) - 1;
    mask &= mask - 1;
    ltp_neuron(P, t, j0 + b);
  }
}

// Stand-alone LTP of the scan at step t: one wave per neuron that fired
// (so the sweeps of different neurons overlap), the bitmap of slot t telling
// which.  Runs after the step's phase 2 (and after a commit at ms % 1000 ==
// 999, which must come first).
__global__ __launch_bounds__(kWaveLTP) void k_ltp(DevNet P, uint32_t t) {
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t waves = (gridDim.x * blockDim.x) >> 6;
  const uint64_t *bits = P.bits + (size_t)(t & (P.RS - 1)) * P.NW;
  for (uint32_t j = wave; j < P.N; j += waves)
    if ((bits[j >> 6] >> (j & 63)) & 1ull) ltp_neuron(P, t, j);
}

// The LTD and LTP of a block of K steps t0 .. t0 + K - 1 at once, after the
// last one's phase 2 (slot t0 + K is the last scan; the steps ran without
// LTD and LTP).  A synapse's updates depend on spike times only: it is
// delivered in step t when its source fired in slot t - delay, and its target
// fired in slot t + 1 or did not; spikeMask holds both for the last 32 slots.
// Each synapse's additions are made in the order the single steps make them
// (LTD of t, then LTP of the scan t + 1), in float, so td and last come out
// the same bit for bit.  Plasticity is on in all K steps and at slot t0 + K,
// and no commit falls in the block; a synapse has one in-list item (no
// spill-over runs), so its item names all its deliveries.
//
// One wave per target.  It moves each synapse's td and last once a block
// instead of once a step (LTD) and once a spike (LTP): 22 B per synapse and
// block against about 9 B per synapse and step.  202 M synapses (180,000
// neurons, blocks of 10 and 16 steps): 1.56 ms per block; updating step by
// step, LTD made phase 1 take 1.78 ms a step (0.91 without it, in the window
// form) and LTP 0.26.
constexpr uint32_t kMaskSlots = 32;
constexpr uint32_t kStdpBlock = 16;    // steps per block
// A single step updates its synapses itself: a block moves every synapse's td
// and last, one step's LTD and LTP only those of the delivered ones and of the
// targets that spike (180,000 neurons, ms per step in calls of 3: 1.75 in
// blocks, 2.46 step by step; 31,250 neurons: 0.52 and 0.61; calls of one: 2.5
// and 2.46 by the kernels' times).
constexpr uint32_t kStdpBlockMin = 2;
constexpr int kStdpU = 4;              // independent synapses per lane
__global__ __launch_bounds__(kWaveLTP) void k_stdp(DevNet P, uint32_t t0, uint32_t K) {
  __shared__ float causal[kStdpSpan], anti[kStdpSpan];
  for (uint32_t i = threadIdx.x; i < kStdpSpan; i += blockDim.x) {
    causal[i] = P.causal[i];
    anti[i] = P.anti[i];
  }
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
  const uint32_t waves = (gridDim.x * blockDim.x) >> 6;
  for (uint32_t j = wave; j < P.N; j += waves) {
    const uint32_t mj = P.spikeMask[j];
    // lane k: the LTD increment of step t0 + k, from the last spike at or
    // before slot t0 + k (bits K - 1 .. K - k of mj are the slots t0 + 1 ..)
    float av = 0.0f;
    if (lane < K) {
      const uint32_t y = (mj >> (K - lane)) & ((1u << lane) - 1u);
      const int lastS = y ? (int)(t0 + lane) - __builtin_ctz(y) : P.lastSpike0[j];
      const int dt = (int)(t0 + lane) - lastS;
      av = dt < (int)kStdpSpan ? anti[dt] : 0.0f;
    }
    const uint64_t beg = P.inOff[j], sbase = P.incOff[j];
    const uint32_t len = (uint32_t)(P.inOff[j + 1] - beg);
    for (uint32_t base = 0; base < len; base += kStdpU * kWave) {
      uint32_t pd[kStdpU], sy[kStdpU], z[kStdpU];
      int32_t last[kStdpU];
      float td[kStdpU];
#pragma unroll
      for (int u = 0; u < kStdpU; ++u) {
        const uint32_t i = min(base + (uint32_t)u * kWave + lane, len - 1);
        pd[u] = P.inPD[beg + i];
        sy[u] = P.inSyn[beg + i];
      }
#pragma unroll
      for (int u = 0; u < kStdpU; ++u) {
        // the delivery of step t0 + k in bit 31 - k
        z[u] = (P.spikeMask[pd[u] & 0xFFFFFFu] >> (pd[u] >> 24)) << (kMaskSlots - 1 - K);
        last[u] = P.lastT[sbase + sy[u]];
        td[u] = P.tdT[sbase + sy[u]];
      }
      for (uint32_t k = 0; k < K; ++k) {
        const int t = (int)(t0 + k);
        const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(av), (int)k));
#pragma unroll
        for (int u = 0; u < kStdpU; ++u) {
          const bool delivered = (int32_t)z[u] < 0;
          z[u] <<= 1;
          td[u] = delivered ? td[u] + a : td[u];
          last[u] = delivered ? t : last[u];
        }
        if ((mj >> (K - 1 - k)) & 1u) {  // uniform: the target fired in slot t + 1
#pragma unroll
          for (int u = 0; u < kStdpU; ++u) {
            const int dt = t - last[u];
            const float f = causal[min((uint32_t)dt, kStdpSpan - 1)];
            td[u] += last[u] != 0 && dt < (int)kStdpSpan ? f : 0.0f;
          }
        }
      }
#pragma unroll
      for (int u = 0; u < kStdpU; ++u)
        if (base + (uint32_t)u * kWave + lane < len) {
          P.lastT[sbase + sy[u]] = last[u];
          P.tdT[sbase + sy[u]] = td[u];
        }
    }
  }
}

// lastSpike0 = lastSpike.
__global__ __launch_bounds__(kWaveLTP) void k_stdp_begin(DevNet P) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < P.N) P.lastSpike0[j] = P.lastSpike[j];
}

// spikeMask from the spike bitmaps (a restored network): slots t, t - 1, ...
__global__ __launch_bounds__(kWaveLTP) void k_mask_from_bits(DevNet P, uint32_t t) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= P.N) return;
  uint32_t m = 0;
  for (uint32_t b = 0; b < min(min(P.RS, kMaskSlots), t + 1); ++b) {
    const uint64_t w = P.bits[(size_t)((t - b) & (P.RS - 1)) * P.NW + (j >> 6)];
    m |= (uint32_t)((w >> (j & 63)) & 1ull) << b;
  }
  P.spikeMask[j] = m;
}

// longTermPlasticity (DPSNN_localNet_sim.c:312-414), once per simulated
// second at ms % 1000 == 999: exc->exc synapses take w + td (+drift),
// clipped to [0, 2J] in float and re-quantized to int16; td then decays
// (or resets when tauDerivativeDecay_s == 1).
__global__ __launch_bounds__(kWaveLTP) void k_commit(DevNet P) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t waves = (gridDim.x * blockDim.x) >> 6;
  for (uint32_t j = wave; j < P.N; j += waves) {
    const uint32_t tgt = P.subPop[j];
    for (uint64_t s = P.incOff[j] + lane; s < P.incOff[j + 1]; s += 64) {
      const uint32_t src = P.kindT[s];
      const float maxSyn = P.maxSyn[src * P.nsub + tgt];
      const float rev = P.revMax[src * P.nsub + tgt];
      float clamp = 0.0f;
      if (maxSyn > 0.0 && rev > 0.0) {
        float w = (float)(P.wT[s] * P.w2f);
        float td = P.tdT[s];
        td += P.drift;
        w = w + td;
        if (w > maxSyn) {
          clamp = (w - maxSyn);
          td = td - clamp;
          w = maxSyn;
        }
        if (w < 0.0) {
          clamp = w;
          td = td - clamp;
          w = 0.0;
        }
        P.wT[s] = (int16_t)(w * P.f2w);
        P.tdT[s] = td;
      }
      if (P.tdPre) P.tdPre[s] = P.tdT[s];
      if (P.decayReset)
        P.tdT[s] = 0.0;
      else
        P.tdT[s] = (P.tdT[s] - P.drift + clamp) * P.decayMul;
    }
  }
}

// After a commit the in-list items pick up their synapse's new weight.
__global__ __launch_bounds__(kWaveLTP) void k_refresh_weights(DevNet P) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t waves = (gridDim.x * blockDim.x) >> 6;
  for (uint32_t j = wave; j < P.N; j += waves) {
    const uint64_t base = P.incOff[j];
    for (uint64_t it = P.inOff[j] + lane; it < P.inOff[j + 1]; it += 64)
      const_cast<int16_t *>(P.inW)[it] = P.wT[base + P.inSyn[it]];
  }
}

// ... and so do the window layout's: one wave per (unit, pass, wave) stream,
// a lane per chunk.  A chunk's items are its target's items of the pass's run
// delay from 8 times its place in the target's run of chunks on; the in-list
// is run delay descending, so the pass's first item is found by bisection.
__global__ __launch_bounds__(kWaveLTP) void k_refresh_window(DevNet P) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t waves = (gridDim.x * blockDim.x) >> 6;
  const uint32_t streams = P.winUnits * P.winPasses * kWindowWaves;
  for (uint32_t st = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; st < streams; st += waves) {
    const uint32_t u = st / (P.winPasses * kWindowWaves), pass = st / kWindowWaves % P.winPasses;
    const uint32_t d = P.winPasses - 1 - pass;
    const uint32_t col = u / P.winUnitsPerCol, j0 = col * P.npc + (u - col * P.winUnitsPerCol) * P.winUnit;
    const uint64_t cb = P.winChunk[st], ce = P.winChunk[st + 1];
    uint32_t carry = 0;  // chunks of the run that the next 64 chunks go on with
    for (uint64_t c0 = cb; c0 < ce; c0 += 64) {
      const uint64_t c = c0 + lane;
      const uint32_t q = c < ce ? P.winDesc[c] : kWindowFirst;
      const uint64_t first = __ballot(q >= kWindowFirst) & (~0ull >> (63 - lane));
      const uint32_t place = first ? lane - (63 - (uint32_t)__clzll((long long)first)) : carry + lane;
      carry = (uint32_t)__shfl((int)place, 63) + 1;
      if (c >= ce) continue;
      const uint32_t j = j0 + (q & kWindowTarget);
      const uint64_t end = P.inOff[j + 1];
      uint64_t lo = P.inOff[j], hi = end;  // first item of run delay <= d
      while (lo < hi) {
        const uint64_t mid = (lo + hi) / 2;
        if ((P.inPD[mid] >> 24) > d) lo = mid + 1; else hi = mid;
      }
      uint32_t *item = const_cast<uint32_t *>(P.winItem) + c * kWindowChunk;
      const uint64_t from = lo + (uint64_t)place * kWindowChunk;
      for (uint32_t i = 0; i < kWindowChunk && from + i < end && (P.inPD[from + i] >> 24) == d; ++i)
        item[i] = (item[i] & 0xFFFF0000u) | (uint16_t)P.inW[from + i];
    }
  }
}

// --------------------------------------------------------------------------
// k_compact: single workgroup; ascending ids of slot t's bitmap with their
// emission times, appended at *rasterCount.
// --------------------------------------------------------------------------
constexpr int kCompactThreads = 1024;
__global__ __launch_bounds__(kCompactThreads) void k_compact(DevNet P, uint32_t t, uint32_t *ids,
                                                             double *te, uint32_t *rasterCount,
                                                             uint32_t *stepCount) {
  __shared__ uint32_t part[kCompactThreads];
  const uint32_t slot = t & (P.RS - 1);
  const uint64_t *w = P.bits + (size_t)slot * P.NW;
  const uint32_t per = (P.NW + kCompactThreads - 1) / kCompactThreads;
  const uint32_t w0 = threadIdx.x * per, w1 = min(P.NW, w0 + per);
  uint32_t n = 0;
  for (uint32_t k = w0; k < w1; ++k) n += __popcll(w[k]);
  part[threadIdx.x] = n;
  __syncthreads();
  for (int off = 1; off < kCompactThreads; off <<= 1) {  // inclusive scan
    const uint32_t add = threadIdx.x >= (uint32_t)off ? part[threadIdx.x - off] : 0;
    __syncthreads();
    part[threadIdx.x] += add;
    __syncthreads();
  }
  const uint32_t base = *rasterCount;
  uint32_t pos = base + part[threadIdx.x] - n;
  for (uint32_t k = w0; k < w1; ++k) {
    uint64_t m = w[k];
    while (m) {
      const int b = __ffsll((long long)m) - 1;
      m &= m - 1;
      const uint32_t id = k * 64 + (uint32_t)b;
      ids[pos] = id;
      te[pos] = P.teHist[(size_t)slot * P.N + id];
      ++pos;
    }
  }
  __syncthreads();
  if (threadIdx.x == kCompactThreads - 1) {
    *rasterCount = base + part[kCompactThreads - 1];
    *stepCount = part[kCompactThreads - 1];
  }
}

// --------------------------------------------------------------------------
// k_step: the delivery + ordering + dynamics of one step.
//
// Event key.  An event of step t arrives at k = t + frac(Te_pre) (the
// reference's double, DPSNN_neuron_sim.c:297, :579) and the reference's
// stable merge sort orders equal k by insertion order, which is the order
// of the neuron's in-list.  For t >= 1 every k lies in [t, 2t], so
// tick = bits(k) - bits(t) is exact and order-preserving (< 2^52), and
//     key = tick << 12 | position-in-in-list
// is unique and sorts exactly as (k, insertion order).  The key also
// recovers k (bits(t) + tick) and the synapse (position).
//
// Phase 1, one neuron per wave, all 64 lanes: stream the in-list
// (coalesced), keep the live items (source fired in step t - delay: one bit
// of the spike history), compact them into LDS in in-list order, load their
// emission times and form the keys, bucket the keys by the top bits of the
// tick (LDS counters), rank each key within its bucket, and store the
// sorted ticks with their weights to the scratch.
// Phase 2, one lane per neuron of the tile: merge the sorted internal
// events with the external bath (internal first on equal time) and run
// LIFCADynamic for each, in FP64.
// --------------------------------------------------------------------------
struct ExtView {  // replayed external events of this step
  const uint32_t *off;
  const double *time, *value;
};


__device__ inline uint64_t lane_mask_lt() {
  const uint32_t lane = threadIdx.x & 63;
  return lane ? (~0ull >> (64 - lane)) : 0ull;
}

// External bath of one neuron in step t, one event at a time in time order:
// at() is the next event's time (kNoEvent when none is pending); take() returns its
// value and moves on.
constexpr double kNoEvent = __builtin_huge_val();
struct ExtReplayCursor {
  const double *time, *value;
  uint32_t x, xe;
  __device__ inline double at() const { return x < xe ? time[x] : kNoEvent; }
  __device__ inline double take() { return value[x++]; }
  __device__ inline void skip() { ++x; }
  __device__ inline void finish() {}
};

// The reference's Poisson bath (DPSNN_neuron_sim.c:604-640, :844-851) from
// the Philox stream: the first due event is always drawn (do-while), the
// following ones while fewer than the per-ms cap; past the cap only the
// lapses are drawn.  An event takes one Philox block (its value from the
// first uniform, the lapse to the next event from the second).
struct ExtPhiloxCursor {
  double a, inv, nextF;
  const double *lut;
  uint32_t cap, nExt;
  bool onE;
  PhiloxStream R;
  __device__ inline double at() const {
    return onE && a < nextF && (nExt == 0 || nExt < cap) ? a : kNoEvent;
  }
  __device__ inline double take() {
    double pick, lapse;
    R.block(pick, lapse);
    const double val = lut[(uint32_t)(pick * kLutDepth)];
    ++nExt;
    const double u = 1.0 - lapse;
    a += -logf((float)u) * inv;
    return val;
  }
  __device__ inline void skip() {  // take() without the value
    double pick, lapse;
    R.block(pick, lapse);
    ++nExt;
    const double u = 1.0 - lapse;
    a += -logf((float)u) * inv;
  }
  __device__ inline void finish() {
    if (onE && nExt >= cap && a < nextF) {
      do {
        const double u = 1.0 - R.next();
        a += -logf((float)u) * inv;
      } while (a < nextF);
    }
  }
};

// The bath with its events drawn ahead of the merge, by all lanes of the
// wave together, into LDS: up to kQueue (time, value) pairs per lane, then a
// time of kNoEvent (qt/qv: the lane's columns of [kQueue + 1][64] and
// [kQueue][64]).  A lane that has taken its last drawn event while another
// one is due draws the next ones there and then, through LDS as well: the
// merge loop itself never waits on a global load.  The stream is consumed in
// the same order either way, so the events are the same.  Whether another
// event is due after the drawn ones (its time is not kept: the cursor has it).
constexpr int kQueue = 4;
template <class Cursor>
__device__ __attribute__((always_inline)) inline bool draw_bath(Cursor &x, bool on, lds_f64 *qt, lds_f64 *qv) {
  uint32_t n = 0;
  double a = on ? x.at() : kNoEvent;
  for (;;) {
    const bool d = n < (uint32_t)kQueue && a < kNoEvent;
    if (!__ballot(d)) break;
    if (d) {
      qt[n * kWave] = a;
      qv[n * kWave] = x.take();
      a = x.at();
      ++n;
    }
  }
  qt[n * kWave] = kNoEvent;
  return a < kNoEvent;
}

template <bool REPLAY>
using BathCursor = std::conditional_t<REPLAY, ExtReplayCursor, ExtPhiloxCursor>;

// Neuron j's bath in step t (`on`: the lane has a neuron).
template <bool REPLAY>
__device__ inline BathCursor<REPLAY> bath_cursor(const DevNet &P, uint32_t t, const ExtView &X, uint32_t j, bool on) {
  BathCursor<REPLAY> x{};
  if (on) {
    if constexpr (REPLAY) {
      x = ExtReplayCursor{X.time, X.value, X.off[j], X.off[j + 1]};
    } else {
      x.a = P.assigned[j];
      x.inv = P.invNuExt[j];
      x.nextF = (double)t + 1.0;
      x.lut = P.lut + (size_t)P.subPop[j] * kLutDepth;
      x.cap = P.maxExt[j];
      x.nExt = 0;
      x.onE = x.inv > 0;
      x.R = PhiloxStream{(uint32_t)P.philoxSeed, (uint32_t)(P.philoxSeed >> 32) ^ j, P.philoxCtr[j], 0.0, 0};
    }
  }
  return x;
}
// Leaves neuron j's bath where the step ends; returns its event count.
template <class Cursor>
__device__ inline uint32_t finish_bath(const DevNet &P, const ExtView &X, uint32_t j, Cursor &x) {
  if constexpr (std::is_same_v<Cursor, ExtReplayCursor>) {
    return x.xe - X.off[j];
  } else {
    x.finish();
    P.assigned[j] = x.a;
    P.philoxCtr[j] = x.R.ctr;
    return x.nExt;
  }
}

constexpr int kChunk = 8;  // internal events per lane per LDS-staged chunk
// From step kPackT on, a scratch entry carries its weight in the low 16 bits
// (tick << 16 | weight): for t >= 32 every tick is at most 2^47 (t + frac
// stays within [t, t + 1] and 2^(52 - floor(log2 t)) <= 2^47).  Earlier
// steps keep the weight in its own array.
constexpr uint32_t kPackT = 32;
constexpr int kRun = 16;   // events per neuron run in the blocked scratch
// Weight of a bath event's record: no synapse has it (weights are quantised
// to at most 32767 in magnitude).
constexpr int16_t kBathWeight = -32768;
constexpr uint32_t kBathMax = 128;  // most bath events of a neuron and ms that k_bath takes
// The bath of step t, one lane per neuron, into bathT and bathN; its state
// (and its counter) are where the step ends.  REPLAY: the host's events.
// One value per sub-population, so an event is its time.
template <bool REPLAY>
__device__ inline void bath_step(const DevNet &P, uint32_t t, const ExtView &X, uint32_t j) {
  const bool on = j < P.N;
  BathCursor<REPLAY> x = bath_cursor<REPLAY>(P, t, X, j, on);
  uint32_t n = 0;
  if (on) {
    for (double a; (a = x.at()) < kNoEvent; ++n) {
      P.bathT[(size_t)n * P.N + j] = a;
      x.skip();
    }
    P.bathN[j] = n;
  }
  unsigned long long ex = on ? finish_bath(P, X, j, x) : 0u;
  for (int o = 32; o > 0; o >>= 1) ex += __shfl_down(ex, o);
  if ((threadIdx.x & 63) == 0 && ex) atomicAdd(counter_slot(P.counters) + 1, ex);
}
__global__ __launch_bounds__(kWave) void k_bath(DevNet P, uint32_t t, ExtView X) {
  if (P.tDev) t += *P.tDev;
  const uint32_t j = blockIdx.x * kWave + threadIdx.x;
  if (P.drive == DPSNN_DRIVE_REPLAY)
    bath_step<true>(P, t, X, j);
  else
    bath_step<false>(P, t, X, j);
}

// The bath events of neuron j that phase 1 of step t sorts in (uniform j).
__device__ inline uint32_t bath_count(const DevNet &P, uint32_t t, uint32_t j) {
  return P.bathT && t >= kPackT ? P.bathN[j] : 0u;
}
// The tick of its event i.
__device__ inline uint64_t bath_tick(const DevNet &P, uint64_t tBits, uint32_t j, uint32_t i) {
  return dpsnn_asu64(P.bathT[(size_t)i * P.N + j]) - tBits;
}

// LDS of one wave in phase 2: a ring of two chunks of 64 lanes' ticks, a row
// of kStageRow per event, then the bath queue (values, then times and their
// end mark: [kQueue][64] and [kQueue + 1][64] doubles) and, for steps before kPackT, the
// ring's weights.  The lanes
// move through the ring each at its own pace (a lane that takes bath events
// falls behind the others): a chunk is stored over the one before the last
// when every lane is past that.  A row is 64 ticks plus padding: the
// transposing stores write 8 rows x 8 neurons per instruction, which 64-wide
// rows would put on one bank per neuron.
constexpr uint32_t kRing = 2 * kChunk;
constexpr uint32_t kStageRow = kWave + 1;
constexpr size_t kStageKBytes = kRing * kStageRow * sizeof(uint64_t);
constexpr size_t kStagePackedBytes = kStageKBytes + (2 * kQueue + 1) * kWave * sizeof(double);
constexpr size_t kStageBytes = kStagePackedBytes + kRing * kWave * sizeof(int16_t);
constexpr uint32_t kExpTab = 256;  // words of dpsnn_exp's table
constexpr size_t kExpTabBytes = kExpTab * sizeof(uint64_t);

// A buffer view of `bytes` (< 2^31) bytes at base (raw: stride 0, byte
// offsets; the gfx9 descriptor word).  An access at kDropOffset is out of
// range: a load returns zero and a store is dropped, without touching
// memory and without a branch.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kDropOffset = 0x80000000u;
__device__ inline __amdgpu_buffer_rsrc_t buffer_view(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
// A pointer that is the same in every lane of the wave, as a scalar value
// (a buffer view needs its base in scalar registers).
template <class T>
__device__ inline T *wave_uniform(T *p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return (T *)(((uint64_t)hi << 32) | lo);
}

// Chunk c (events 8c..8c+7 of every lane) from the tile's blocked scratch
// [i / kRun][q][i % kRun]: each neuron's 8 ticks are one 64-byte piece of
// its run, loaded by the wave in 8 coalesced instructions (instruction r:
// neurons 8r..8r+7) and transposed through LDS; each lane's 8 weights are
// one 16-byte load.  Only the pieces of neurons with events in the chunk
// (bit q of act) are fetched; the others read as zero from an
// out-of-range offset.  Entries past a neuron's count are never consumed.
static_assert(kChunk == 8 && kRun % kChunk == 0, "chunks are whole pieces of a run");
__device__ inline void load_chunk(const __amdgpu_buffer_rsrc_t &tileK, const int16_t *tileW, uint32_t c,
                                  uint64_t act, uint64_t (&rk)[kChunk], uint4 &rw, bool packed) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t blk = (c * kChunk / kRun) * (kWave * kRun) + (c * kChunk) % kRun;
  const uint64_t mine = act >> (lane >> 3);  // bit 8r: neuron 8r + lane / 8 has events in chunk c
#pragma unroll
  for (int r = 0; r < kChunk; ++r) {
    const uint32_t off = (blk + (uint32_t)(r * 8 + (lane >> 3)) * kRun + (lane & 7)) * 8u;
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(tileK, ((mine >> (8 * r)) & 1u) ? off : kDropOffset, 0, 0);
    rk[r] = (uint64_t)v.x | ((uint64_t)v.y << 32);
  }
  if (!packed) rw = *(const uint4 *)(tileW + blk + (size_t)lane * kRun);
}
// Chunk c into its half of the ring.
__device__ inline void store_chunk(lds_u64 *ring, lds_i16 *ringW, uint32_t c, const uint64_t (&rk)[kChunk],
                                   const uint4 &rw, bool packed) {
  const uint32_t lane = threadIdx.x & 63, e = lane & 7, half = (c & 1) * kChunk;
#pragma unroll
  for (int r = 0; r < kChunk; ++r) ring[(half + e) * kStageRow + (uint32_t)r * 8 + (lane >> 3)] = rk[r];
  if (!packed) {
    const uint32_t w[4] = {rw.x, rw.y, rw.z, rw.w};
#pragma unroll
    for (int i = 0; i < kChunk; ++i) ringW[(half + i) * kWave + lane] = (int16_t)(w[i / 2] >> (16 * (i & 1)));
  }
}

// dpsnn_exp's table into LDS, by the block's threads (a barrier must follow).
__device__ inline void load_exp_table(lds_u64 *tab) {
  for (uint32_t i = threadIdx.x; i < kExpTab; i += blockDim.x) tab[i] = dpsnn_exp_tab_d[i];
}

// Phase 2, one lane per neuron: lane q integrates neuron j0 + q (q < m) over
// its n sorted internal events (the tile's blocked scratch tileK/tileW:
// ticks relative to bits(t) and int16 weights) merged with its external
// bath, LIFCADynamic per event in FP64.  Returns the lane's external event
// count and whether (and when) its neuron fired.  Whole wave, uniform.
// PK 1: every entry carries its weight (t >= kPackT), PK 2: t decides at
// run time.
//
// A neuron's events are one serial chain, so a wave's time is its longest
// neuron's events times the latency of one turn of the merge loop, and what
// bounds the kernel is that latency while there are fewer waves than SIMDs
// (grids up to 8x8 columns) and FP64 issue beyond.  Hence the loop:
//  * takes nothing from global memory: the events are staged through LDS two
//    chunks deep with the third in flight, the bath is queued in LDS and
//    exp's table is there (stage, kStageBytes; expTab).  A load anywhere in
//    the loop makes the compiler wait for all of them on every turn, the
//    chunk in flight included;
//  * lets every lane go on at its own pace through the ring, so that a
//    wave's turns are the most events of one lane, not the sum over chunks
//    of the most events in the chunk;
//  * is one straight block: a lane without an event runs one that changes
//    nothing; drawing more of the bath and the refractory exit are the only
//    branches, and rare.
// Measured, us per launch, against a loop with those loads and chunk by chunk:
// 5,000 neurons 145 (208), 80,000 neurons 226 (308), 720,000 neurons 964
// (1155).
template <bool REPLAY, int PK = 2>
__device__ __attribute__((always_inline)) inline uint32_t integrate_wave(const DevNet &P, uint32_t t, const ExtView &X, uint32_t j0, uint32_t m,
                                          const uint64_t *tileK, const int16_t *tileW, uint32_t n, lds_u64 *stage,
                                          const lds_u64 *expTab, bool &fired, double &te) {
  const uint32_t lane = threadIdx.x & 63;
  const bool on = lane < m;
  const uint32_t j = j0 + lane;
  if (!on) n = 0;
  uint32_t nmax = n;
  for (int o = 32; o > 0; o >>= 1) nmax = max(nmax, (uint32_t)__shfl_xor((int)nmax, o));
  nmax = (uint32_t)__builtin_amdgcn_readfirstlane((int)nmax);
  const double tF = (double)t, nextF = (double)(tF + 1.0);
  const uint64_t tBits = dpsnn_asu64(tF);
  const bool packed = PK == 2 ? t >= kPackT : PK == 1;
  const __amdgpu_buffer_rsrc_t tileR = buffer_view(wave_uniform(tileK), P.cap * kWave * (uint32_t)sizeof(uint64_t));
  const uint32_t chunks = (nmax + kChunk - 1) / kChunk;
  lds_u64 *ring = stage;
  lds_i16 *ringW = (lds_i16 *)((__attribute__((address_space(3))) uint8_t *)stage + kStagePackedBytes);
  uint64_t rk[kChunk];
  uint4 rw = make_uint4(0, 0, 0, 0);
  if (chunks) load_chunk(tileR, tileW, 0, __ballot(n > 0), rk, rw, packed);
  Lifca L{};
  L.expTab = expTab;
  if (on) L.load(P, j);
  BathCursor<REPLAY> bath = bath_cursor<REPLAY>(P, t, X, j, on);
  lds_f64 *qv = (lds_f64 *)stage + kRing * kStageRow + lane, *qt = qv + kQueue * kWave;
  bool due = draw_bath(bath, on, qt, qv);  // a bath event is due after the drawn ones
  uint32_t qi = 0;                         // the next bath event
  double head = qt[0], headV = qv[0];
  if (chunks) store_chunk(ring, ringW, 0, rk, rw, packed);
  if (chunks > 1) {
    load_chunk(tileR, tileW, 1, __ballot(n > kChunk), rk, rw, packed);
    store_chunk(ring, ringW, 1, rk, rw, packed);
  }
  // the loads above are waited for here: one that is still in flight at the
  // loop's entry would be waited for, with the chunk in flight, on every turn
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  uint32_t staged = min(chunks, 2u);   // chunks stored so far
  uint32_t e = 0;                     // the lane's next internal event
  for (;;) {
    const bool more = staged < chunks;
    if (more) load_chunk(tileR, tileW, staged, __ballot(n > staged * kChunk), rk, rw, packed);
    wave_sync();
    // events of the lane that are staged, those it must be past before the
    // next chunk is stored, and what a lane without a staged event may take:
    // any bath event once its internal ones are used up, else none
    const uint32_t have = min(n, staged * kChunk), need = more ? min(n, (staged - 1) * kChunk) : 0u;
    const uint64_t final = more ? 0ull : ~0ull;  // the last chunks: on while a lane has an event
    const double without = n <= staged * kChunk ? kNoEvent : -kNoEvent;
    // the entry of the next internal event is read as soon as the one before
    // it is taken, so that the LDS read overlaps the event's dynamics
    uint64_t kv = ring[(e % kRing) * kStageRow + lane];
    int16_t kw = packed ? 0 : ringW[(e % kRing) * kWave + lane];
    // merge: the bath event goes first when strictly earlier
    bool inner = e < have;
    double kI = dpsnn_asf64(tBits + (packed ? kv >> 16 : kv));
    bool outer = head < (inner ? kI : without);
    const auto go_on = [&] {
      return (__ballot(e < need) | ((__ballot(inner) | __ballot(outer)) & final)) != 0ull;
    };
    if (go_on()) do {
      const double at = outer ? head : (inner ? kI : L.Tr);
      const int16_t w16 = packed ? (int16_t)(uint16_t)kv : kw;
      const double val = outer ? headV : (double)(((float)w16) * P.w2f);
      const bool some = inner || outer;
      e += inner && !outer ? 1u : 0u;
      qi += outer ? 1u : 0u;
      kv = ring[(e % kRing) * kStageRow + lane];
      if (!packed) kw = ringW[(e % kRing) * kWave + lane];
      if (due && qi == (uint32_t)kQueue) {
        due = draw_bath(bath, true, qt, qv);
        qi = 0;
      }
      head = qt[qi * kWave];
      headV = qv[qi * kWave];
      L.event(some, at, val);
      inner = e < have;
      kI = dpsnn_asf64(tBits + (packed ? kv >> 16 : kv));
      outer = head < (inner ? kI : without);
    } while (go_on());
    if (!more) break;
    wave_sync();
    store_chunk(ring, ringW, staged, rk, rw, packed);
    ++staged;
  }
  uint32_t nExt = 0;
  if (on) {
    nExt = finish_bath(P, X, j, bath);
    P.v[j] = L.v; P.c[j] = L.c; P.Tr[j] = L.Tr; P.Te[j] = L.Te;
  }
  fired = on && L.fired != 0;
  te = L.Te;
  wave_sync();  // the stage is free again
  return nExt;
}

// The time and value of a record of phase 1 with the bath sorted in
// (t >= kPackT).
__device__ inline double record_time(uint64_t tBits, uint64_t kv) { return dpsnn_asf64(tBits + (kv >> 16)); }
__device__ inline float record_value(uint64_t kv, float w2f, float bathV) {
  const int16_t w = (int16_t)(uint16_t)kv;
  return w == kBathWeight ? bathV : ((float)w) * w2f;
}

// Phase 2 over records that hold the bath too: integrate_wave without the
// merge.  Every lane is at the same event, so a chunk is stored over the one
// before when the wave is done with that.  Whole wave, uniform.  Bound by
// instruction issue (about 57 an event against 75 with the merge).  us per
// launch, with the merge and without: 5,000 neurons 145 and 89, 80,000
// neurons 226 and 148, 720,000 neurons 964 and 689 (k_bath 6, 8 and 22).
__device__ __attribute__((always_inline)) inline void integrate_records(const DevNet &P, uint32_t t, uint32_t j0, uint32_t m,
                                                                        const uint64_t *tileK, uint32_t n, lds_u64 *stage,
                                                                        const lds_u64 *expTab, bool &fired, double &te) {
  const uint32_t lane = threadIdx.x & 63;
  const bool on = lane < m;
  const uint32_t j = j0 + lane;
  if (!on) n = 0;
  uint32_t nmax = n;
  for (int o = 32; o > 0; o >>= 1) nmax = max(nmax, (uint32_t)__shfl_xor((int)nmax, o));
  nmax = (uint32_t)__builtin_amdgcn_readfirstlane((int)nmax);
  const uint64_t tBits = dpsnn_asu64((double)t);
  const __amdgpu_buffer_rsrc_t tileR = buffer_view(wave_uniform(tileK), P.cap * kWave * (uint32_t)sizeof(uint64_t));
  const uint32_t chunks = (nmax + kChunk - 1) / kChunk;
  uint64_t rk[kChunk];
  uint4 rw = make_uint4(0, 0, 0, 0);
  if (chunks) load_chunk(tileR, nullptr, 0, __ballot(n > 0), rk, rw, true);
  Lifca L{};
  L.expTab = expTab;
  float bathV = 0.0f;
  if (on) {
    L.load(P, j);
    bathV = P.bathV[P.subPop[j]];
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), as in integrate_wave
  if (chunks) store_chunk(stage, nullptr, 0, rk, rw, true);
  for (uint32_t c = 0; c < chunks; ++c) {
    if (c + 1 < chunks) load_chunk(tileR, nullptr, c + 1, __ballot(n > (c + 1) * kChunk), rk, rw, true);
    wave_sync();
    const uint32_t from = c * kChunk, turns = min((uint32_t)kChunk, nmax - from);
    uint64_t kv = stage[lane];
    for (uint32_t e = 0; e < turns; ++e) {
      const bool some = from + e < n;
      const double at = some ? record_time(tBits, kv) : L.Tr;
      const double val = (double)record_value(kv, P.w2f, bathV);
      kv = stage[min(e + 1, (uint32_t)kChunk - 1) * kStageRow + lane];
      L.event(some, at, val);
    }
    wave_sync();
    if (c + 1 < chunks) store_chunk(stage, nullptr, 0, rk, rw, true);
  }
  if (on) {
    P.v[j] = L.v; P.c[j] = L.c; P.Tr[j] = L.Tr; P.Te[j] = L.Te;
  }
  fired = on && L.fired != 0;
  te = L.Te;
  wave_sync();  // the stage is free again
}

// The same by three waves per tile: two compute, each for half of the tile's
// neurons, what an event takes from its time alone (Lifca::decay), the third
// runs the recurrence on v and c for all of them.  In round c the first two
// put chunk c into LDS and the third works on chunk c - 1, one barrier a
// round.  A lane of the first two holds, in register r, event lane % 8 of
// neuron 8 r + lane / 8, as the loads deliver them; the time before an event
// is the lane's below (the first event's: the last of the chunk before).
//
// While there are fewer tiles than SIMDs a step's phase 2 is one wave's
// instructions, whatever they depend on (measured: a lone wave issues an
// FP64, a 64-bit integer or a compare instruction at the same rate in a chain
// or not, and a branch that a mask decides costs it more than ten), so the
// chain is left with the instructions that need v or c.  us per launch here
// and in integrate_records: 1,250 and 5,000 neurons 79 and 89, 31,250 neurons
// (489 tiles) 129 and 129, 80,000 neurons 261 and 148 (the work is more, with
// its LDS traffic, and four workgroups fit a CU); ms per 20 steps: 313 tiles
// 5.54 and 5.83, 388 tiles 2.58 and 2.63, 489 tiles equal.  Hence kPipeTiles.
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) f64x2 lds_f64x2;
typedef __attribute__((address_space(3))) float lds_f32;
struct RecordsLds {
  uint64_t expTab[kExpTab];
  uint64_t stage[kBlock / kWave][kChunk * kStageRow];
};
struct PipeLds {
  f64x2 decay[2][kChunk][kWave];  // dtHalf, rmHalf
  double cDecay[2][kChunk][kWave];
  double time[2][kChunk][kWave];
  float value[2][kChunk][kWave];
  uint64_t expTab[kExpTab];
};
constexpr int kPipeThreads = 3 * kWave;
constexpr uint32_t kPipeTiles = 448;

// Barrier of a pipelined tile: LDS is ordered around it, global loads in
// flight stay in flight.
__device__ inline void pipe_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __attribute__((always_inline)) inline void integrate_pipe(const DevNet &P, uint32_t t, uint32_t j0, uint32_t m,
                                                                     const uint64_t *tileK, uint32_t n, PipeLds &S,
                                                                     bool &fired, double &te) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t role = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (lane >= m) n = 0;
  uint32_t nmax = n;
  for (int o = 32; o > 0; o >>= 1) nmax = max(nmax, (uint32_t)__shfl_xor((int)nmax, o));
  const uint32_t chunks = (uint32_t)__builtin_amdgcn_readfirstlane((int)((nmax + kChunk - 1) / kChunk));
  load_exp_table((lds_u64 *)S.expTab);
  fired = false;
  te = 0.0;
  if (role < 2) {
    constexpr int R = kChunk / 2;
    const uint64_t tBits = dpsnn_asu64((double)t);
    const __amdgpu_buffer_rsrc_t tileR = buffer_view(wave_uniform(tileK), P.cap * kWave * (uint32_t)sizeof(uint64_t));
    const uint32_t e = lane & 7, q0 = role * R * 8 + (lane >> 3);  // neuron of register r: q0 + 8 r
    // per register: the neuron's reciprocals, bath value, record count, and
    // the time its chunk before ended at
    Lifca L[R];
    double tr[R];
    float bathV[R];
    uint32_t nq[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t q = q0 + 8 * r;
      nq[r] = (uint32_t)__shfl((int)n, (int)q);
      const uint32_t jq = j0 + min(q, m - 1), sp = P.subPop[jq];
      const double *prm = P.sp + (size_t)sp * kParams;
      L[r].invTau = prm[kInvTau]; L[r].invTauLo = prm[kInvTauLo];
      L[r].invTauC = prm[kInvTauC]; L[r].invTauCLo = prm[kInvTauCLo];
      bathV[r] = P.bathV[sp];
      tr[r] = P.Tr[jq];
    }
    uint64_t rk[R];
    const auto load = [&](uint32_t c) {  // records past a neuron's last are not fetched
      const uint32_t blk = (c * kChunk / kRun) * (kWave * kRun) + (c * kChunk) % kRun;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t off = (blk + (q0 + 8 * r) * kRun + e) * 8u;
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(tileR, c * kChunk < nq[r] ? off : kDropOffset, 0, 0);
        rk[r] = (uint64_t)v.x | ((uint64_t)v.y << 32);
      }
    };
    if (chunks) load(0);
    pipe_barrier();
    for (uint32_t c = 0; c <= chunks; ++c) {
      if (c < chunks) {
        const uint32_t half = c & 1;
        lds_f64x2 *decay = (lds_f64x2 *)&S.decay[half][e][q0];
        lds_f64 *cDecay = (lds_f64 *)&S.cDecay[half][e][q0], *time = (lds_f64 *)&S.time[half][e][q0];
        lds_f32 *value = (lds_f32 *)&S.value[half][e][q0];
        double at[R];
        float val[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (c) tr[r] = ((const lds_f64 *)&S.time[half ^ 1][kChunk - 1][q0])[8 * r];
          at[r] = record_time(tBits, rk[r]);
          val[r] = record_value(rk[r], P.w2f, bathV[r]);
        }
        if (__ballot(n < (c + 1) * kChunk)) {
          // past its last event a neuron stays where it is: the time of that
          // event (or of the chunk before), a value that changes nothing
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const uint32_t left = nq[r] - min(nq[r], c * kChunk);
            const double stay = __shfl(at[r], (int)((lane & 56) + (left && left < 8 ? left - 1 : 0)));
            at[r] = e < left ? at[r] : (left ? stay : tr[r]);
            val[r] = e < left ? val[r] : -0.0f;
          }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const uint64_t ab = dpsnn_asu64(at[r]);
          // the lane below's time (row_shr:1)
          const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)ab, 0x111, 0xf, 0xf, false);
          const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(ab >> 32), 0x111, 0xf, 0xf, false);
          const double below = dpsnn_asf64((uint64_t)hi << 32 | lo);
          double dtHalf, rmHalf, cd;
          L[r].decay(at[r] - (e ? below : tr[r]), dtHalf, rmHalf, cd);
          decay[8 * r] = f64x2{dtHalf, rmHalf};
          cDecay[8 * r] = cd;
          time[8 * r] = at[r];
          value[8 * r] = val[r];
        }
        if (c + 1 < chunks) load(c + 1);
      }
      pipe_barrier();
    }
    return;
  }
  Lifca L{};
  L.expTab = (lds_u64 *)S.expTab;
  const bool on = lane < m;
  const uint32_t j = j0 + lane;
  if (on) L.load(P, j);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), as in integrate_wave
  pipe_barrier();
  for (uint32_t round = 0; round <= chunks; ++round) {
    if (round) {
      const uint32_t c = round - 1, half = c & 1, left = n - min(n, c * (uint32_t)kChunk);
      const lds_f64x2 *decay = (const lds_f64x2 *)&S.decay[half][0][lane];
      const lds_f64 *cDecay = (const lds_f64 *)&S.cDecay[half][0][lane], *time = (const lds_f64 *)&S.time[half][0][lane];
      const lds_f32 *value = (const lds_f32 *)&S.value[half][0][lane];
#pragma unroll
      for (uint32_t i = 0; i < (uint32_t)kChunk; ++i) {
        const f64x2 d = decay[i * kWave];
        L.event<true>(i < left, time[i * kWave], (double)value[i * kWave], d.x, d.y, cDecay[i * kWave]);
      }
    }
    pipe_barrier();
  }
  if (on) {
    P.v[j] = L.v; P.c[j] = L.c; P.Tr[j] = L.Tr; P.Te[j] = L.Te;
  }
  fired = on && L.fired != 0;
  te = L.Te;
}

constexpr uint64_t kNoKey = ~0ull;

// Bucket of a key: the top log2(B) bits of its tick (tick < 2^(52 - e),
// e = floor(log2 t)), clamped.
template <int B>
__device__ inline uint32_t key_bucket(uint64_t tick, int shift) {
  const uint64_t b = tick >> shift;
  return b < (uint64_t)B ? (uint32_t)b : (uint32_t)(B - 1);
}

// *(base + byteOff): a 32-bit byte offset from a uniform base, so that a
// load needs one address register (the spike history is under 4 GiB:
// checked at build).
template <class T>
__device__ inline T load_at(const T *base, uint32_t byteOff) {
  return *(const T *)((const char *)base + byteOff);
}

// Byte offsets of source `pre`'s entries of slot s: its emission time in the
// Te history ([RS][N] doubles) and the 32-bit word of the fired bitmap
// ([RS][NW] u64, read as [RS][2NW] u32) that holds its bit (bit pre & 31).
// N < 2^24 (checked at build), so the products are 24-bit multiplies.
__device__ inline uint32_t te_offset(const DevNet &P, uint32_t s, uint32_t pre) {
  return (__umul24(s, P.N) + pre) * 8u;
}
__device__ inline uint32_t bit_offset(const DevNet &P, uint32_t s, uint32_t pre) {
  return (__umul24(s, 2u * P.NW) + (pre >> 5)) * 4u;
}

// LTD, synapseSetLastActiveTime_antiCausalSTDP (DPSNN_neuron_sim.c:
// 207-277): every synapse delivered to neuron j in step t gets last = t and
// td += anti[t - lastSpike_j], one increment per target, taken before step
// t's dynamics move lastSpike.
__device__ inline float ltd_increment(const DevNet &P, uint32_t t, uint32_t j) {
  const int dt = (int)t - P.lastSpike[j];
  return dt < kStdpSpan ? P.anti[dt] : 0.0f;
}

// Applies it to the n synapses whose in-list positions phase 1 left in the
// blocked scratch (pos = neuron j's [0][q][0]).  A synapse is delivered at
// most once per step (refractory >= 1 ms), so the updates are independent:
// rounds of 4 per lane issue the position loads, the synapse-index loads,
// the value loads, then the stores.  Whole wave.
__device__ __attribute__((always_inline)) inline void ltd_neuron(const DevNet &P, uint32_t t, uint32_t j, float a, uint32_t n, const uint16_t *pos) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t beg = P.inOff[j], sbase = P.incOff[j];
  const uint32_t len = (uint32_t)(P.inOff[j + 1] - beg);  // positions from len on are bath events
  constexpr int U = 4;
  for (uint32_t i0 = lane; i0 < n; i0 += U * kWave) {
    uint32_t p[U], sy[U];
    float td[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = i0 + (uint32_t)u * kWave;
      p[u] = i < n ? pos[(size_t)(i / kRun) * (kWave * kRun) + (i % kRun)] : len;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) sy[u] = p[u] < len ? P.inSyn[beg + p[u]] : 0u;
#pragma unroll
    for (int u = 0; u < U; ++u) td[u] = p[u] < len ? P.tdT[sbase + sy[u]] : 0.0f;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (p[u] < len) {
        P.lastT[sbase + sy[u]] = (int32_t)t;
        P.tdT[sbase + sy[u]] = td[u] + a;
      }
  }
}

constexpr int kDense = 16;  // fast path: up to kDense * 64 live keys per neuron, kDense per lane in registers
constexpr int kSlowK = 8;   // register batches (of 64 items) of the general path

// Fast path, rounds one and two: the live items of neuron j's in-list
// (beg, len), compacted into rec[0, n) in in-list order as
// item | position << 32 | synapse << 44 (with plastic, the item's synapse
// in j's incoming list, for LTD); returns n (uniform).  K batches of 64
// in-list words are loaded at once, then the bitmap words of their sources
// (a target's sources are a few neighbouring columns, so these mostly hit
// the CU's L1).  The in-list arrays are padded by one wave, so the words
// past len that the last batch loads exist; they are never live.
template <int K>
__device__ __attribute__((always_inline)) inline uint32_t compact_live(const DevNet &P, uint32_t t, uint64_t beg, uint32_t len, uint64_t *rec,
                                        int plastic) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t *bw = (const uint32_t *)P.bits;
  uint32_t n = 0;
  for (uint32_t base = 0; base < len; base += (uint32_t)K * kWave) {
    uint32_t it[K], wb[K], sy[K];
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (base + k * kWave < len) {
        it[k] = P.inPD[beg + base + k * kWave + lane];
        sy[k] = plastic ? P.inSyn[beg + base + k * kWave + lane] : 0u;
      }
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (base + k * kWave < len)
        wb[k] = load_at(bw, bit_offset(P, (t - (it[k] >> 24)) & (P.RS - 1), it[k] & 0xFFFFFFu));
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (base + k * kWave < len) {
        const uint32_t idx = base + k * kWave + lane;
        const bool live = idx < len && (it[k] >> 24) <= t && ((wb[k] >> (it[k] & 31u)) & 1u);
        const uint64_t m = __ballot(live);
        if (live) {
          const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
          rec[n + below] = (uint64_t)it[k] | ((uint64_t)idx << 32) | ((uint64_t)sy[k] << 44);
        }
        n += (uint32_t)__popcll(m);
      }
  }
  return n;
}

// Keys of in-list items base + k*64 + lane (k < K) of neuron j; kNoKey for
// items that are absent or not live (the source did not fire in step
// t - delay: its bit in that slot's fired bitmap is clear).  With `first`,
// also counts the live keys per bucket (LDS) and keeps their weights in LDS
// by position (ldsW).  Three rounds of K independent loads: the in-list
// words; the bitmap words of their sources (a target's sources are a few
// neighbouring columns, so these mostly hit the CU's L1); then, for live
// items only, the emission times and weights.  A source's bitmap bit is set
// exactly when its Te history entry is an emission time (publish_spikes
// writes both), so the emission-time loads go to L2 only for delivered
// events.
template <int K, int B>
__device__ __attribute__((always_inline)) inline uint32_t gather_keys(const DevNet &P, uint32_t t, uint32_t j, uint64_t beg, uint32_t len,
                                       uint32_t base, uint64_t (&key)[K], uint32_t *bcnt, int16_t *ldsW,
                                       int shift, uint64_t tBits, bool first, int plastic) {
  static_assert(K <= 32, "live items are kept in one 32-bit mask");
  const uint32_t lane = threadIdx.x & 63;
  const double tF = (double)t;
  const uint32_t *bw = (const uint32_t *)P.bits;
  uint32_t it[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t idx = base + k * kWave + lane;
    it[k] = idx < len ? P.inPD[beg + idx] : kPad;
  }
  uint32_t wb[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t d = it[k] >> 24, pre = it[k] & 0xFFFFFFu;
    wb[k] = 0u;
    if (it[k] != kPad && d <= t) wb[k] = load_at(bw, bit_offset(P, (t - d) & (P.RS - 1), pre));
  }
  uint32_t live = 0u;
#pragma unroll
  for (int k = 0; k < K; ++k) live |= ((wb[k] >> (it[k] & 31u)) & 1u) << k;
  double te[K];
  int16_t w[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t d = it[k] >> 24, pre = it[k] & 0xFFFFFFu;
    te[k] = kNotFired;
    if ((live >> k) & 1u) {
      te[k] = load_at(P.teHist, te_offset(P, (t - d) & (P.RS - 1), pre));
      if (first) w[k] = P.inW[beg + base + k * kWave + lane];
    }
  }
  uint32_t n = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const bool on = te[k] >= 0.0;
    key[k] = kNoKey;
    if (on) {
      const uint32_t idx = base + k * kWave + lane;
      const double kk = tF + (te[k] - trunc(te[k]));  // modf, exact
      const uint64_t tick = dpsnn_asu64(kk) - tBits;
      key[k] = (tick << 12) | idx;
      if (first) {
        atomicAdd(&bcnt[key_bucket<B>(tick, shift)], 1u);
        ldsW[idx] = w[k];
      }
    }
    n += (uint32_t)__popcll(__ballot(on));
  }
  return n;
}

template <int K, int B>
__device__ __attribute__((always_inline)) inline void scatter_keys(const uint64_t (&key)[K], uint32_t *bcnt, uint64_t *sorted, int shift) {
#pragma unroll
  for (int k = 0; k < K; ++k)
    if (key[k] != kNoKey) sorted[atomicAdd(&bcnt[key_bucket<B>(key[k] >> 12, shift)], 1u)] = key[k];
}

// Keys that rank_in_buckets reads at a time, and the padding after the sort
// buffer that lets it read past the last bucket's end.
constexpr uint32_t kRankReads = 6;

// LDS of one phase-1 wave: sort buffer (u64) and weights by position (i16)
// for the longest in-list, then the bucket counters after a zero.
__host__ __device__ inline size_t phase1_lds(uint32_t cap, int B) {
  return (size_t)(cap + kRankReads) * sizeof(uint64_t) + (size_t)cap * sizeof(int16_t) + (size_t)(B + 2) * sizeof(uint32_t);
}

// Offset of event p of a neuron in the tile's blocked scratch, from the
// neuron's [0][q][0].
__device__ inline size_t run_offset(uint32_t p) { return (size_t)(p / kRun) * (kWave * kRun) + (p % kRun); }

// Exclusive scan of the B bucket counters in place (R = B / 64 per lane);
// bcnt[B] receives the total.  Whole wave.
template <int B>
__device__ __attribute__((always_inline)) inline void bucket_scan(uint32_t *bcnt) {
  constexpr int R = B / kWave;
  const uint32_t lane = threadIdx.x & 63;
  uint32_t c[R], sum = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) { c[r] = bcnt[lane * R + r]; sum += c[r]; }
  uint32_t incl = sum;
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t v = __shfl_up(incl, o);
    if (lane >= (uint32_t)o) incl += v;
  }
  uint32_t run = incl - sum;
  wave_sync();
#pragma unroll
  for (int r = 0; r < R; ++r) { bcnt[lane * R + r] = run; run += c[r]; }
  if (lane == kWave - 1) bcnt[B] = run;
}

// The n keys in sorted[] are scattered into their buckets (bcnt[b] = end of
// bucket b).  Within a bucket each key's place is its rank (keys are
// unique): the count of the bucket's smaller keys.  Calls put(key, place)
// once per key.  Lanes take the keys in bucket order, so lanes of one bucket
// read the same words together.  The kRankReads independent reads of a round
// may pass the bucket's end: the keys there are larger (a later bucket, or
// the padding).  The sorts are bound by their instructions and LDS reads, and
// most are here (a bucket holds 4-14 keys, most of them one spike time):
// rounds of 4 with the remainder one key at a time took 189 us at 80,000
// neurons (k_sort, now 180), 1,206 for a batch of 150,000 (k_batch_gather,
// now 1,157).  Reads of 4 and 8: 180 and 182, 1,163 and 1,152.  bcnt[-1] is a
// word of its own.  Whole wave.
template <int B, class Put>
__device__ __attribute__((always_inline)) inline void rank_in_buckets(uint64_t *sorted, uint32_t *bcnt,
                                                                      uint32_t n, int shift, Put &&put) {
  const uint32_t lane = threadIdx.x & 63;
  if (lane < kRankReads) sorted[n + lane] = kNoKey;
  if (lane == 0) bcnt[-1] = 0;
  wave_sync();
  for (uint32_t i = lane; i < n; i += kWave) {
    const uint64_t x = sorted[i];
    const uint32_t b = key_bucket<B>(x, shift + 12);
    const uint32_t lo = (bcnt - 1)[b], hi = bcnt[b];
    uint32_t r = lo;
    for (uint32_t y = lo; y < hi; y += kRankReads) {
      uint64_t a[kRankReads];
#pragma unroll
      for (uint32_t k = 0; k < kRankReads; ++k) a[k] = sorted[y + k];
#pragma unroll
      for (uint32_t k = 0; k < kRankReads; ++k) r += a[k] < x ? 1u : 0u;
    }
    put(x, r);
  }
}

// A target's bath events among the keys to be sorted: lane's events lane and
// lane + 64, position `from` + event (after every internal one, so that equal
// times keep internal events first), weight kBathWeight in ldsW.
static_assert(kBathMax <= 2 * kWave, "two bath keys per lane");
template <int B>
__device__ __attribute__((always_inline)) inline void bath_keys(const DevNet &P, uint64_t tBits, uint32_t j, uint32_t nb,
                                                                uint32_t from, int shift, uint32_t *bcnt, int16_t *ldsW,
                                                                uint64_t (&key)[2]) {
  const uint32_t lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const uint32_t i = lane + (uint32_t)r * kWave;
    key[r] = kNoKey;
    if ((uint32_t)r * kWave < nb && i < nb) {
      const uint64_t tick = bath_tick(P, tBits, j, i);
      key[r] = tick << 12 | (from + i);
      ldsW[from + i] = kBathWeight;
      atomicAdd(&bcnt[key_bucket<B>(tick, shift)], 1u);
    }
  }
}

// Phase 1 for neuron j, whole wave: live keys of its in-list, bucket-sorted
// in LDS (lds: sorted[cap], ldsW[cap], bcnt[B + 1]), stored in arrival order
// as ticks relative to bits(t) (outK) with their weights (outW) and, with
// plastic, their in-list positions (outP, for LTD); returns their count n and
// stores the count of records, with the bath's (bath_count), in *total.
// The scratch of a tile of 64 neurons is blocked by runs of kRun events:
// event i of neuron q at [i / kRun][q][i % kRun] (a neuron's keys fill whole
// 128-byte lines), and outK/outW point at neuron q's [0][q][0].
// Fast path (n <= denseMax): the live items are compacted into sorted[]
// (compact_live), then each lane takes live items p = lane, lane + 64, ...:
// emission time and weight loads for delivered events only, keys in
// registers, bucket counts, scatter.  Otherwise the general path gathers
// the in-list in register batches of kSlowK * 64 items, twice.
// With plastic, the step's LTD of neuron j's delivered synapses is applied
// here too: inline on the fast path, from the stored positions (ltd_neuron)
// on the general path.
template <int K, int B>
__device__ __attribute__((always_inline)) inline uint32_t gather_sort_neuron(const DevNet &P, uint32_t t, uint32_t j, int plastic, uint8_t *lds,
                                              uint32_t cap, uint64_t *outK, int16_t *outW, uint16_t *outP,
                                              uint32_t *total) {
  static_assert(B % kWave == 0, "bucket count must be a multiple of 64");
  constexpr int LOG2B = B == 64 ? 6 : B == 128 ? 7 : B == 256 ? 8 : B == 512 ? 9 : 10;
  uint64_t *sorted = (uint64_t *)lds;
  int16_t *ldsW = (int16_t *)(sorted + cap + kRankReads);
  uint32_t *bcnt = (uint32_t *)(ldsW + cap) + 1;
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t tBits = dpsnn_asu64((double)t);
  const double tF = (double)t;
  const int e = t ? (31 - __clz((int)t)) : 0;
  const int shift = 52 - LOG2B - e;
  constexpr uint32_t kSuper = (uint32_t)kSlowK * kWave;
  const uint64_t beg = P.inOff[j];
  const uint32_t len = (uint32_t)(P.inOff[j + 1] - beg);
  for (uint32_t b = lane; b <= (uint32_t)B; b += kWave) bcnt[b] = 0;
  uint32_t n = 0;
  if (t > 0) n = compact_live<K>(P, t, beg, len, sorted, plastic);
  wave_sync();
  const bool fast = n <= P.denseMax;
  uint64_t key[kDense];
  if (fast) {
    uint64_t rc[kDense];
#pragma unroll
    for (int r = 0; r < kDense; ++r)
      if ((uint32_t)r * kWave < n) {
        const uint32_t p = r * kWave + lane;
        rc[r] = sorted[p < n ? p : 0u];
      }
    double te[kDense];
    int16_t w[kDense];
    float td[kDense];
#pragma unroll
    for (int r = 0; r < kDense; ++r)
      if ((uint32_t)r * kWave < n) {
        const uint32_t it = (uint32_t)rc[r], idx = (uint32_t)(rc[r] >> 32) & 0xFFFu;
        te[r] = load_at(P.teHist, te_offset(P, (t - (it >> 24)) & (P.RS - 1), it & 0xFFFFFFu));
        w[r] = P.inW[beg + idx];
      }
    if (plastic) {
      // LTD (synapseSetLastActiveTime_antiCausalSTDP): each delivered
      // synapse gets last = t and td += a; a synapse is delivered at most
      // once per step (refractory >= 1 ms), so the updates are independent
      const uint64_t sbase = P.incOff[j];
      const float a = ltd_increment(P, t, j);
#pragma unroll
      for (int r = 0; r < kDense; ++r)
        if ((uint32_t)r * kWave < n) td[r] = P.tdT[sbase + (uint32_t)(rc[r] >> 44)];
#pragma unroll
      for (int r = 0; r < kDense; ++r)
        if ((uint32_t)r * kWave < n && r * kWave + lane < n) {
          const uint64_t s = sbase + (uint32_t)(rc[r] >> 44);
          P.lastT[s] = (int32_t)t;
          P.tdT[s] = td[r] + a;
        }
    }
#pragma unroll
    for (int r = 0; r < kDense; ++r)
      if ((uint32_t)r * kWave < n) {
        const uint32_t idx = (uint32_t)(rc[r] >> 32) & 0xFFFu;
        const double kk = tF + (te[r] - trunc(te[r]));  // modf, exact
        const uint64_t tick = dpsnn_asu64(kk) - tBits;
        key[r] = (tick << 12) | idx;
        if (r * kWave + lane < n) {
          atomicAdd(&bcnt[key_bucket<B>(tick, shift)], 1u);
          ldsW[idx] = w[r];
        }
      }
  } else {
    n = 0;
    uint64_t k8[kSlowK];
    for (uint32_t base = 0; base < len; base += kSuper)
      n += gather_keys<kSlowK, B>(P, t, j, beg, len, base, k8, bcnt, ldsW, shift, tBits, true, plastic);
  }
  const uint32_t nb = bath_count(P, t, j), all = n + nb;
  uint64_t bk[2];
  bath_keys<B>(P, tBits, j, nb, len, shift, bcnt, ldsW, bk);
  wave_sync();
  bucket_scan<B>(bcnt);
  wave_sync();
  // scatter into buckets (order inside a bucket is fixed below); the general
  // path gathers its batches again (L2 hits)
  if (fast) {
#pragma unroll
    for (int r = 0; r < kDense; ++r)
      if ((uint32_t)r * kWave < n && r * kWave + lane < n)
        sorted[atomicAdd(&bcnt[key_bucket<B>(key[r] >> 12, shift)], 1u)] = key[r];
  } else {
    uint64_t k8[kSlowK];
    for (uint32_t base = 0; base < len; base += kSuper) {
      gather_keys<kSlowK, B>(P, t, j, beg, len, base, k8, bcnt, ldsW, shift, tBits, false, 0);
      scatter_keys<kSlowK, B>(k8, bcnt, sorted, shift);
    }
  }
  if (nb) scatter_keys<2, B>(bk, bcnt, sorted, shift);
  wave_sync();
  rank_in_buckets<B>(sorted, bcnt, all, shift, [&](uint64_t x, uint32_t p) {
    const size_t at = run_offset(p);
    const int16_t wv = ldsW[x & 0xFFFu];
    if (t >= kPackT) {
      outK[at] = ((x >> 12) << 16) | (uint16_t)wv;
    } else {
      outK[at] = x >> 12;
      outW[at] = wv;
    }
    if (plastic && !fast) outP[at] = (uint16_t)(x & 0xFFFu);
  });
  wave_sync();
  if (plastic && !fast) ltd_neuron(P, t, j, ltd_increment(P, t, j), all, outP);
  if (lane == 0) *total = all;
  return n;
}

// What the tail of step t does for the scan of step t+1: where its counts
// go (null: not collected) and whether LTP runs there.
struct NextScan {
  uint32_t *popCnt;
  int ltp;
  int count;  // step t+1 is simulated: its scan counts the spikes
};

// LDS of one wave of the fused step: phase 1's sort, then phase 2's stage.
__host__ __device__ inline size_t step_lds(uint32_t cap, int B) {
  const size_t p1 = phase1_lds(cap, B), p2 = kStageBytes + kExpTabBytes;
  return p1 > p2 ? p1 : p2;
}

// One tile (neurons 64*tile .. 64*tile+63) of step t, one wave: phase 1 for
// each neuron into the wave's blocked scratch wkeys/wW[cap/8][64][8] and
// wcnt[64],
// phase 2 one lane per neuron, then the fired scan of step t+1.  Returns the
// tile's delivered events (uniform) and adds external events to *exSum (per
// lane).
template <int K, int B>
__device__ __attribute__((always_inline)) inline unsigned long long step_tile(const DevNet &P, uint32_t t, const ExtView &X, int ltd,
                                               const NextScan &S, uint32_t tile, uint32_t cap, uint8_t *lds,
                                               uint64_t *wkeys, int16_t *wW, uint16_t *wP, uint32_t *wcnt,
                                               unsigned long long &exSum) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t j0 = tile * kWave;
  const uint32_t m = min((uint32_t)kWave, P.N - j0);
  unsigned long long evSum = 0;
  for (uint32_t q = 0; q < m; ++q) {
    evSum += gather_sort_neuron<K, B>(P, t, j0 + q, ltd, lds, cap, wkeys + q * kRun, wW + q * kRun, wP + q * kRun,
                                      wcnt + q);
  }
  __threadfence_block();
  __syncthreads();
  // ---------------- phase 2 ----------------
  const uint32_t n = lane < m ? wcnt[lane] : 0u;
  lds_u64 *stage = (lds_u64 *)lds, *expTab = stage + kStageBytes / sizeof(uint64_t);
  load_exp_table(expTab);
  __syncthreads();
  bool f = false;
  double te = 0.0;
  if (P.drive == DPSNN_DRIVE_REPLAY)
    exSum += integrate_wave<true>(P, t, X, j0, m, wkeys, wW, n, stage, expTab, f, te);
  else
    exSum += integrate_wave<false>(P, t, X, j0, m, wkeys, wW, n, stage, expTab, f, te);
  // ---------------- fired scan of step t+1 ----------------
  const uint64_t mask = publish_spikes(P, t + 1, j0 + lane, f, te, S.popCnt, S.count);
  if (S.ltp) ltp_word(P, t + 1, mask, j0);
  __syncthreads();
  return evSum;
}

// Fused step of one network: each wave owns tiles blockIdx.x, +gridDim.x, ...
template <int K, int B>
__global__ __launch_bounds__(kWave) void k_step(DevNet P, uint32_t t, ExtView X, int ltd, NextScan S) {
  extern __shared__ uint64_t lds[];
  uint64_t *wkeys = P.keys + (size_t)blockIdx.x * kWave * P.cap;
  int16_t *wW = P.keyW + (size_t)blockIdx.x * kWave * P.cap;
  uint16_t *wP = P.keyPos ? P.keyPos + (size_t)blockIdx.x * kWave * P.cap : nullptr;
  uint32_t *wcnt = P.keyCount + (size_t)blockIdx.x * kWave;
  unsigned long long evSum = 0, exSum = 0;
  const XcdWalk w = xcd_walk(P.NW);
  for (uint32_t tile = w.first; tile < w.end; tile += w.stride)
    evSum += step_tile<K, B>(P, t, X, ltd, S, tile, P.cap, (uint8_t *)lds, wkeys, wW, wP, wcnt, exSum);
  for (int o = 32; o > 0; o >>= 1) exSum += __shfl_down(exSum, o);
  if (threadIdx.x == 0) {
    atomicAdd(counter_slot(P.counters) + 0, evSum);
    atomicAdd(counter_slot(P.counters) + 1, exSum);
  }
}

// Per-network, per-step arguments of a batched launch.
struct BatchItem {
  uint32_t t;
  int ltd;
  NextScan S;
  ExtView X;
  uint32_t tileBegin;  // first global tile of this network
  uint32_t net;        // index into the batch's DevNet array
};

// Batched step: many independent networks (each at its own ms) in one
// persistent launch.  Global tile g belongs to the network whose
// [tileBegin, tileBegin + NW) holds it; each wave walks g = blockIdx.x,
// +gridDim.x, ... with scratch sized for the batch's longest in-list.
template <int K, int B>
__global__ __launch_bounds__(kWave) void k_batch_step(const DevNet *nets, const BatchItem *items, uint32_t count,
                                                      uint32_t totalTiles, uint32_t cap, uint64_t *keys,
                                                      int16_t *keyW, uint16_t *keyPos, uint32_t *keyCount) {
  extern __shared__ uint64_t lds[];
  uint64_t *wkeys = keys + (size_t)blockIdx.x * kWave * cap;
  int16_t *wW = keyW + (size_t)blockIdx.x * kWave * cap;
  uint16_t *wP = keyPos + (size_t)blockIdx.x * kWave * cap;
  uint32_t *wcnt = keyCount + (size_t)blockIdx.x * kWave;
  const XcdWalk w = xcd_walk(totalTiles);
  for (uint32_t g = w.first; g < w.end; g += w.stride) {
    uint32_t lo = 0, hi = count;  // last item with tileBegin <= g
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) / 2;
      if (items[mid].tileBegin <= g) lo = mid; else hi = mid;
    }
    const BatchItem &it = items[lo];
    const DevNet &P = nets[it.net];
    unsigned long long exSum = 0;
    const unsigned long long ev = step_tile<K, B>(P, it.t, it.X, it.ltd, it.S, g - it.tileBegin, cap,
                                                  (uint8_t *)lds, wkeys, wW, wP, wcnt, exSum);
    for (int o = 32; o > 0; o >>= 1) exSum += __shfl_down(exSum, o);
    if (threadIdx.x == 0) {
      atomicAdd(counter_slot(P.counters) + 0, ev);
      if (exSum) atomicAdd(counter_slot(P.counters) + 1, exSum);
    }
  }
}

// Split form: k_gather sorts every neuron's live events into its own rows
// of network-wide buffers (one wave per neuron), then k_integrate runs
// phase 2 one lane per neuron and the fired scan of step t+1.  Each kernel
// gets its own register budget.
template <int K, int B>
__global__ __launch_bounds__(kWave) void k_gather(DevNet P, uint32_t t, int ltd) {
  extern __shared__ uint64_t lds[];
  if (P.tDev) t += *P.tDev;
  unsigned long long evSum = 0;
  const uint32_t home = blockIdx.x % kXcds;
  uint32_t x = home;
  const bool queue = P.N > kStaticTargets * gridDim.x;
  for (uint32_t j0 = blockIdx.x, j1 = P.N;;) {
    if (queue && (j0 = next_item(P.workCtr, P.N, x, home, &j1)) >= P.N) break;
    for (uint32_t j = j0; j < j1; j += queue ? 1u : gridDim.x) {
      const size_t at = (size_t)(j >> 6) * P.cap * kWave + (j & 63) * kRun;  // the tile's blocked scratch
      evSum += gather_sort_neuron<K, B>(P, t, j, ltd, (uint8_t *)lds, P.cap, P.keys + at, P.keyW + at,
                                        ltd ? P.keyPos + at : nullptr, P.keyCount + j);
    }
    if (!queue) break;
  }
  if (threadIdx.x == 0) atomicAdd(counter_slot(P.counters) + 0, evSum);
}

// ---------------------------------------------------------------------------
// Stencil-window form of phase 1 (steps t >= kPackT without LTD).
//
// k_collect: one workgroup of kWindowWaves waves per unit (a range of the
// targets of one column), handed out by an XCD-ordered queue.  For each
// run delay d, in the in-lists' order (descending), the workgroup stages
// the emission times of slot t - d of the column's stencil columns into
// LDS, already turned into packed ticks (bits(t + frac(Te)) - bits(t)) << 16,
// or kNoKey where the source did not fire.  Its waves then stream the
// unit's items of delay d (window index << 16 | weight, coalesced chunks):
// an item is live when its window entry holds a tick, and its record
// (tick << 16 | weight) is appended to its target's run in the blocked
// scratch.  Each target's records come out in the order of its live
// in-list items, so a record's place in the run breaks equal ticks exactly
// as the in-list position does.  No per-event global load: the only
// per-event memory access besides the item stream is the LDS lookup.
//
// k_sort: one wave per target orders its records by (tick, place) in LDS
// (bucket counts, scatter, rank within bucket) and writes them back in
// place, as phase 2 reads them.
// ---------------------------------------------------------------------------
constexpr int kCollectThreads = kWindowWaves * kWave;
// The window form by default from this size.  k_gather is bound by the L1
// misses of its emission-time loads, one line per event (68% of its cycles;
// more waves a CU don't help), which the window's LDS saves; below, k_gather
// deals its targets out in the fixed order and the window's passes cost more
// than its events (ms per step, gather and window: 5,000 neurons 0.070 and
// 0.080, 10,000 neurons 0.091 and 0.103, 12,000 0.144 and 0.151, 12,500 0.106
// and 0.091, 18,252 0.127 and 0.110, 31,250 0.49 and 0.38, 45,000 0.53 and
// 0.39).
constexpr uint32_t kWindowMinNeurons = 12288;
// In a batch a window-form member steps on launches of its own: from this
// size on they fill the device.
constexpr uint32_t kBatchWindowMin = 1u << 16;
// Units per column: k_collect runs one workgroup per CU, so a step takes as
// many rounds of units as there are CUs' worth of them, each as long as a
// unit's targets and its window loads (worth some 50 targets).  The fewest
// target times win.  ms per 20 steps with the units per column chosen here
// and with units of at most 320 targets: 81 columns of 1,250 neurons 13.4 (3)
// and 14.9 (4), 100 columns 16.1 (5) and 17.1, 144 columns 23.4 (5) and 24.6,
// 169 columns of 507 6.0 (3) and 6.5 (2); 36 columns of 1,250: 7 (252 units)
// 7.9, 6 8.2, 8 (288) 9.1.
constexpr uint32_t kWindowRound = 256, kWindowLoad = 50, kWindowUnitTargets = 640;
static uint32_t window_units_per_col(uint32_t npc, uint32_t ncols) {
  uint32_t best = 1;
  uint64_t least = ~0ull;
  for (uint32_t u = std::max(1u, (npc + kWindowUnitTargets - 1) / kWindowUnitTargets); u <= std::min(npc, kWindowRound); ++u) {
    const uint64_t rounds = ((uint64_t)ncols * u + kWindowRound - 1) / kWindowRound;
    const uint64_t cost = rounds * ((npc + u - 1) / u + kWindowLoad);
    if (cost < least) {
      least = cost;
      best = u;
    }
  }
  return best;
}
constexpr uint32_t kWindowMaxEntries = 12 * 1024;  // window entries: kWinPerThread per thread of k_collect

// Block-wide work queue: the next unit for the whole workgroup (one unit
// per counter update), XCD-ordered as next_item.  sh: two LDS words.
__device__ inline uint32_t next_unit(uint32_t *ctr, uint32_t total, uint32_t &x, uint32_t home, uint32_t *sh) {
  __syncthreads();  // every wave has read the previous hand-out
  if (threadIdx.x == 0) {
    uint32_t got = total;
    for (;;) {
      const uint32_t begin = (uint32_t)((uint64_t)total * x / kXcds);
      const uint32_t end = (uint32_t)((uint64_t)total * (x + 1) / kXcds);
      uint32_t *c = ctr + x * kCtrStride;
      if (begin + __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < end) {
        const uint32_t k = atomicAdd(c, 1u);
        if (begin + k < end) {
          got = begin + k;
          break;
        }
      }
      x = (x + 1) % kXcds;
      if (x == home) break;
    }
    sh[0] = got;
    sh[1] = x;
  }
  __syncthreads();
  x = sh[1];
  return sh[0];
}

// LDS of k_collect: the window (entries + 1 u64), the per-target record
// counts and run offsets of a unit plus one slot for padding chunks, two
// queue words.
__host__ __device__ inline size_t collect_lds(uint32_t entries, uint32_t unit) {
  return ((size_t)entries + 1) * sizeof(uint64_t) + ((size_t)unit + 1) * sizeof(uint2) + 2 * sizeof(uint32_t);
}

// Window entries per thread of k_collect (W <= kWinPerThread * 1024): each
// thread keeps its entries' history offsets in registers and loads all of
// a pass's emission times at once.
constexpr int kWinPerThread = 12;
constexpr int kCollectBatches = 4;  // 64-item batches per round of loads (the next round is in flight too)

template <int B, int CH>
__device__ __attribute__((always_inline)) inline void sort_records(const DevNet &P, uint32_t t, uint32_t j, uint32_t n,
                                                                   uint32_t nb, uint8_t *lds, uint32_t cap);
__device__ inline uint64_t *record_runs(const DevNet &P, uint32_t j);
constexpr uint32_t kSortCap = 768;
constexpr int kSortChunks = (int)(kSortCap / kWave);
constexpr int kFusedSortB = 256;  // buckets of the sort inside k_collect
constexpr int kFusedSortChunks = 8;  // records per lane it holds in registers (more: read twice)
constexpr bool kFusedSortDefault = false;
// one wave's sort area inside k_collect, 16-byte aligned (it holds u64s)
__host__ __device__ inline size_t fused_sort_stride() { return (phase1_lds(kSortCap, kFusedSortB) + 15) / 16 * 16; }

__global__ __launch_bounds__(kCollectThreads) void k_collect(DevNet P, uint32_t t) {
  extern __shared__ uint64_t lds[];
  if (P.tDev) t += *P.tDev;
  const uint32_t W = P.winSlots * P.npc;  // entry W: the padding items' (never live)
  uint64_t *win = lds;
  // per target of the unit (+ padding's slot): records so far (.x) and the
  // element offset of its run in the unit's scratch (.y)
  uint2 *ct = (uint2 *)(win + W + 1);
  uint32_t *sh = (uint32_t *)(ct + P.winUnit + 1);
  const uint32_t pad = P.winUnit;  // the target index of padding chunks past a stream's end
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const uint32_t field = (lane >> 3) * 4;  // this lane's chunk's field in a batch's run-start table
  const bool chunkEnd = (lane & 7) == 7;
  const double tF = (double)t;
  const uint64_t tBits = dpsnn_asu64(tF);
  unsigned long long evSum = 0;
  const uint32_t home = blockIdx.x % kXcds;
  uint32_t x = home;
  for (;;) {
    const uint32_t u = (uint32_t)__builtin_amdgcn_readfirstlane((int)next_unit(P.winCtr, P.winUnits, x, home, sh));
    if (u >= P.winUnits) break;
    const uint32_t col = u / P.winUnitsPerCol, part = u - col * P.winUnitsPerCol;
    const uint32_t j0 = col * P.npc + part * P.winUnit;
    const uint32_t m = min(P.winUnit, (col + 1) * P.npc - j0);
    // the unit's records: tile (j >> 6) of the blocked scratch relative to
    // the unit's first tile, so that a record's offset fits 32 bits
    uint64_t *unitKeys = P.keys + (size_t)(j0 >> 6) * P.cap * kWave;
    const uint32_t j0lo = j0 & 63, tileElems = P.cap * kWave;
    const __amdgpu_buffer_rsrc_t keyRsrc = buffer_view(unitKeys, ((j0lo + m + 63) >> 6) * tileElems * 8u);
    for (uint32_t i = threadIdx.x; i < m; i += blockDim.x) {
      const uint32_t jj = j0lo + i;
      ct[i] = make_uint2(0u, (jj >> 6) * tileElems + (jj & 63) * kRun);
    }
    if (threadIdx.x == 0) {
      win[W] = kNoKey;  // the fused sort's LDS may have overlaid it
      ct[pad] = make_uint2(0u, 0u);
    }
    // this thread's window entries e = tid + r * blockDim: the history
    // offset of their source (or ~0u: no source column in that slot)
    uint32_t off[kWinPerThread];
#pragma unroll
    for (int r = 0; r < kWinPerThread; ++r) {
      const uint32_t e = threadIdx.x + (uint32_t)r * blockDim.x;
      off[r] = ~0u;
      if (e < W) {
        const uint32_t k = e / P.npc;
        const int32_t sc = P.winCols[(size_t)col * P.winSlots + k];
        if (sc >= 0) off[r] = (uint32_t)sc * P.npc + (e - k * P.npc);
      }
    }
    for (uint32_t pass = 0; pass < P.winPasses; ++pass) {
      // emission times of the pass's slot (run delay d: slot t - d)
      const double *slot = P.teHist + (size_t)((t - (P.winPasses - 1 - pass)) & (P.RS - 1)) * P.N;
      double wv[kWinPerThread];
#pragma unroll
      for (int r = 0; r < kWinPerThread; ++r) wv[r] = off[r] != ~0u ? slot[off[r]] : kNotFired;
      __syncthreads();  // the previous pass's lookups are done
#pragma unroll
      for (int r = 0; r < kWinPerThread; ++r) {
        const uint32_t e = threadIdx.x + (uint32_t)r * blockDim.x;
        const double v = wv[r];
        if (e < W) win[e] = v >= 0.0 ? (dpsnn_asu64(tF + (v - trunc(v))) - tBits) << 16 : kNoKey;  // modf, exact
      }
      __syncthreads();
      const uint64_t *co = P.winChunk + ((size_t)u * P.winPasses + pass) * kWindowWaves + wave;
      const uint32_t cb = (uint32_t)co[0], ce = (uint32_t)co[1];
      // The wave's targets come in order, each one's chunks contiguous, the
      // first flagged.  A live item's place is the count of its target at
      // the start of the pass (read where the target's first chunk is) or,
      // for the target carried over from the previous batch, the carried
      // count, plus the live items before it in its run of chunks: the
      // live lanes below it (mbcnt) less those below its run's first lane,
      // taken from that lane in one permute.
      uint32_t carry = 0;
      uint32_t it[kCollectBatches], q[kCollectBatches], itN[kCollectBatches], qN[kCollectBatches];
      // the stream's items and descriptors, addressed by 32-bit offsets.
      // Every load is issued (lanes past the stream's end read its last
      // chunk and take padding instead), and records are stored through a
      // buffer view of the unit's scratch with an out-of-range offset where
      // an item is not live (the store is dropped): a round issues a fixed
      // number of memory operations, so the next round's loads stay in
      // flight while this one is processed.
      const uint32_t *sItem = P.winItem + (size_t)cb * kWindowChunk;
      const uint16_t *sDesc = P.winDesc + cb;
      const uint32_t last = ce - cb - 1;  // used only when the stream is not empty
      auto load = [&](uint32_t c0, uint32_t (&I)[kCollectBatches], uint32_t (&Q)[kCollectBatches]) {
#pragma unroll
        for (int v = 0; v < kCollectBatches; ++v) {
          const uint32_t rel = c0 - cb + (uint32_t)v * kWindowChunk + (lane >> 3);
          const uint32_t at = min(rel, last);
          const uint32_t i = __builtin_nontemporal_load(
              (const uint32_t *)((const char *)sItem + (at * kWindowChunk + (lane & 7)) * 4u));
          const uint32_t d = (uint32_t)load_at(sDesc, at * 2u);
          I[v] = rel <= last ? i : W << 16;
          Q[v] = rel <= last ? d : (pad | kWindowFirst);
        }
      };
      if (cb < ce) load(cb, it, q);
      for (uint32_t c0 = cb; c0 < ce; c0 += kWindowChunk * kCollectBatches) {
        const uint32_t cn = c0 + kWindowChunk * kCollectBatches;
        load(cn, itN, qN);  // past the end on the last round: the last chunk again, unused
        uint64_t r[kCollectBatches];
        uint2 base[kCollectBatches];
#pragma unroll
        for (int v = 0; v < kCollectBatches; ++v) {
          r[v] = win[it[v] >> 16];
          base[v] = ct[q[v] & kWindowTarget];
        }
#pragma unroll
        for (int v = 0; v < kCollectBatches; ++v) {
          if (c0 + (uint32_t)v * kWindowChunk >= ce) break;  // uniform
          const uint32_t qd = q[v];
          const bool live = r[v] != kNoKey;  // never on padding
          const bool first = qd >= kWindowFirst;
          const uint64_t liveM = __ballot(live);
          const uint64_t startM = __ballot(first) & 0x0101010101010101ull;  // chunks' first lanes
          // the run-start chunk of every chunk of the batch (4-bit fields):
          // the last chunk at or before it that is a target's first; 0 before
          // the first such chunk (the carried target's run)
          uint32_t T = 0;
          for (uint64_t sm = startM; sm; sm &= sm - 1) {
            const uint32_t k = (uint32_t)__builtin_ctzll(sm) >> 3;
            const uint32_t fill = ~0u << (4 * k);
            T = (T & ~fill) | ((k * 0x11111111u) & fill);
          }
          const uint32_t pre =
              __builtin_amdgcn_mbcnt_hi((uint32_t)(liveM >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)liveM, 0u));
          const uint32_t val = (first ? base[v].x : carry) - pre;
          const uint32_t p = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(((T >> field) & 15u) << 5), (int)val) + pre;
          const uint32_t at = base[v].y + (p / kRun) * (kWave * kRun) + p % kRun;
          const uint64_t rec = r[v] | (it[v] & 0xFFFFu);
          __builtin_amdgcn_raw_buffer_store_b64(u32x2{(uint32_t)rec, (uint32_t)(rec >> 32)}, keyRsrc,
                                                live ? at * 8u : kDropOffset, 0, 0);
          const uint32_t after = p + (live ? 1u : 0u);
          // a run's count grows along it: the largest of its chunks' last
          // lanes is the count after this batch
          if (chunkEnd) atomicMax(&ct[qd & kWindowTarget].x, after);
          carry = (uint32_t)__builtin_amdgcn_readlane((int)after, 63);
        }
#pragma unroll
        for (int v = 0; v < kCollectBatches; ++v) {
          it[v] = itN[v];
          q[v] = qN[v];
        }
      }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < m; i += blockDim.x) {
      P.keyCount[j0 + i] = ct[i].x;
      evSum += ct[i].x;
    }
    if (P.fuseSort) {
      // Sort the unit's targets while their records are recent: wave w
      // takes targets w + 16 k (k < 64, as m <= 1024), its count held in
      // lane k, since the waves' sort areas overlay the window and counts.
      const uint32_t mi = wave + kWindowWaves * lane;
      const uint32_t held = mi < m ? ct[mi].x : 0u;
      __syncthreads();
      uint8_t *area = (uint8_t *)lds + (size_t)wave * fused_sort_stride();
      for (uint32_t k = 0; wave + k * kWindowWaves < m; ++k) {
        const uint32_t j = j0 + wave + k * kWindowWaves;
        const uint32_t nrec = (uint32_t)__builtin_amdgcn_readlane((int)held, (int)k);
        if (nrec > P.sortCap) {
          if (lane == 0) P.bigList[atomicAdd(P.bigCount, 1u)] = j;
          continue;
        }
        sort_records<kFusedSortB, kFusedSortChunks>(P, t, j, nrec, 0u, area, kSortCap);
      }
    }
  }
  for (int o = 32; o > 0; o >>= 1) evSum += __shfl_down(evSum, o);
  if (lane == 0 && evSum) atomicAdd(counter_slot(P.counters) + 0, evSum);
}

// Orders neuron j's n records (tick << 16 | weight, in live in-list order)
// in place, its nb bath events among them (at its [0][q][0] of the blocked
// scratch).  Sort key tick << 12 | place: unique, ordered as (arrival time,
// in-list position; bath events last).  LDS: phase1_lds(cap, B), cap >= n +
// nb.  Up to CH * 64 records are held in registers; more are read again from
// the scratch.  Whole wave.
template <int B, int CH>
__device__ __attribute__((always_inline)) inline void sort_records(const DevNet &P, uint32_t t, uint32_t j, uint32_t n,
                                                                   uint32_t nb, uint8_t *lds, uint32_t cap) {
  uint64_t *out = record_runs(P, j);
  constexpr int LOG2B = B == 64 ? 6 : B == 128 ? 7 : B == 256 ? 8 : B == 512 ? 9 : 10;
  uint64_t *sorted = (uint64_t *)lds;
  int16_t *ldsW = (int16_t *)(sorted + cap + kRankReads);
  uint32_t *bcnt = (uint32_t *)(ldsW + cap) + 1;
  const uint32_t lane = threadIdx.x & 63;
  const int shift = 52 - LOG2B - (31 - __clz((int)t));
  for (uint32_t b = lane; b <= (uint32_t)B; b += kWave) bcnt[b] = 0;
  wave_sync();
  const bool fast = n <= (uint32_t)CH * kWave;
  uint64_t key[CH];
  if (fast) {
    uint64_t rec[CH];
#pragma unroll
    for (int r = 0; r < CH; ++r)
      if ((uint32_t)r * kWave < n) {
        const uint32_t p = r * kWave + lane;
        rec[r] = out[run_offset(p < n ? p : 0u)];
      }
#pragma unroll
    for (int r = 0; r < CH; ++r)
      if ((uint32_t)r * kWave < n) {
        const uint32_t p = r * kWave + lane;
        key[r] = ((rec[r] >> 16) << 12) | p;
        if (p < n) {
          ldsW[p] = (int16_t)(uint16_t)rec[r];
          atomicAdd(&bcnt[key_bucket<B>(rec[r] >> 16, shift)], 1u);
        }
      }
  } else {
    for (uint32_t p = lane; p < n; p += kWave) {
      const uint64_t rc = out[run_offset(p)];
      ldsW[p] = (int16_t)(uint16_t)rc;
      atomicAdd(&bcnt[key_bucket<B>(rc >> 16, shift)], 1u);
    }
  }
  uint64_t bk[2];
  bath_keys<B>(P, dpsnn_asu64((double)t), j, nb, n, shift, bcnt, ldsW, bk);
  wave_sync();
  bucket_scan<B>(bcnt);
  wave_sync();
  if (fast) {
#pragma unroll
    for (int r = 0; r < CH; ++r)
      if ((uint32_t)r * kWave < n && r * kWave + lane < n)
        sorted[atomicAdd(&bcnt[key_bucket<B>(key[r] >> 12, shift)], 1u)] = key[r];
  } else {
    for (uint32_t p = lane; p < n; p += kWave) {
      const uint64_t k = ((out[run_offset(p)] >> 16) << 12) | p;
      sorted[atomicAdd(&bcnt[key_bucket<B>(k >> 12, shift)], 1u)] = k;
    }
  }
  if (nb) scatter_keys<2, B>(bk, bcnt, sorted, shift);
  wave_sync();  // every record has been read: the runs are rewritten in place
  rank_in_buckets<B>(sorted, bcnt, n + nb, shift, [&](uint64_t x, uint32_t p) {
    out[run_offset(p)] = ((x >> 12) << 16) | (uint16_t)ldsW[x & 0xFFFu];
  });
  wave_sync();
}

// k_sort sizes each wave's LDS for kSortCap records, far above a step's
// live events per target (a few hundred at the saturated rate) but below
// the longest in-list, so that more waves fit a CU; a target with more
// records is listed for k_sort_big, whose LDS holds the longest in-list.

__device__ inline uint64_t *record_runs(const DevNet &P, uint32_t j) {
  return P.keys + (size_t)(j >> 6) * P.cap * kWave + (j & 63) * kRun;
}

// One wave per block, targets j = blockIdx.x + k * gridDim.x: each target's
// records are its own lines, so there is no locality for a work queue to
// keep (its counter round trips measured slower than this static order).
template <int B>
__global__ __launch_bounds__(kWave) void k_sort(DevNet P, uint32_t t) {
  extern __shared__ uint64_t lds[];
  if (P.tDev) t += *P.tDev;
  for (uint32_t j = blockIdx.x; j < P.N; j += gridDim.x) {
    const uint32_t n = P.keyCount[j], nb = bath_count(P, t, j);
    if (n + nb > P.sortCap) {
      if ((threadIdx.x & 63) == 0) P.bigList[atomicAdd(P.bigCount, 1u)] = j;
      continue;
    }
    sort_records<B, kSortChunks>(P, t, j, n, nb, (uint8_t *)lds, kSortCap);
    if (nb && (threadIdx.x & 63) == 0) P.keyCount[j] = n + nb;
  }
}

// The targets k_sort left (more than kSortCap records), one wave each;
// bigCount is cleared by the next k_integrate.  Runs after every k_collect.
template <int B>
__global__ __launch_bounds__(kWave) void k_sort_big(DevNet P, uint32_t t) {
  extern __shared__ uint64_t lds[];
  if (P.tDev) t += *P.tDev;
  if (blockIdx.x == 0 && threadIdx.x < kXcds) P.winCtr[threadIdx.x * kCtrStride] = 0;  // for the next k_collect
  const uint32_t count = *P.bigCount;
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    const uint32_t j = P.bigList[i], n = P.keyCount[j], nb = bath_count(P, t, j);
    sort_records<B, kDense>(P, t, j, n, nb, (uint8_t *)lds, P.cap);
    if (nb && (threadIdx.x & 63) == 0) P.keyCount[j] = n + nb;
  }
}

// LDS of an integration block: exp's table and each wave's stage.
template <int PK>
struct IntegrateLds {
  uint64_t expTab[kExpTab];
  uint64_t stage[kBlock / kWave][(PK == 1 ? kStagePackedBytes : kStageBytes) / sizeof(uint64_t)];
};

// Blocks of kBlock threads: each wave holds 64 consecutive neurons starting
// at a multiple of 64, as publish_spikes requires.
template <int PK>
__global__ __launch_bounds__(kBlock) void k_integrate(DevNet P, uint32_t t, ExtView X, NextScan S) {
  __shared__ IntegrateLds<PK> S2;
  if (P.tDev) t += *P.tDev;
  load_exp_table((lds_u64 *)S2.expTab);
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (blockIdx.x == 0 && threadIdx.x < kXcds) P.workCtr[threadIdx.x * kCtrStride] = 0;  // for the next k_gather
  if (blockIdx.x == 0 && threadIdx.x == 0 && P.bigCount) *P.bigCount = 0;                 // for the next k_sort
  const uint32_t j0 = blockIdx.x * kBlock + wave * kWave;
  const uint32_t m = j0 < P.N ? min((uint32_t)kWave, P.N - j0) : 0u;
  const uint32_t n = lane < m ? P.keyCount[j0 + lane] : 0u;
  const size_t at = (size_t)(min(j0, P.N) >> 6) * P.cap * kWave;  // the wave's tile
  bool f = false;
  double te = 0.0;
  unsigned long long ex;
  if (P.drive == DPSNN_DRIVE_REPLAY)
    ex = integrate_wave<true, PK>(P, t, X, j0, m, P.keys + at, P.keyW + at, n, (lds_u64 *)S2.stage[wave],
                                  (lds_u64 *)S2.expTab, f, te);
  else
    ex = integrate_wave<false, PK>(P, t, X, j0, m, P.keys + at, P.keyW + at, n, (lds_u64 *)S2.stage[wave],
                                   (lds_u64 *)S2.expTab, f, te);
  publish_spikes(P, t + 1, j0 + lane, f, te, S.popCnt, S.count);  // LTP follows in k_ltp
  for (int o = 32; o > 0; o >>= 1) ex += __shfl_down(ex, o);
  if (lane == 0 && ex) atomicAdd(counter_slot(P.counters) + 1, ex);
}

// Phase 2 of a step with the bath in its records: one lane per neuron ...
__global__ __launch_bounds__(kBlock) void k_integrate_records(DevNet P, uint32_t t, NextScan S) {
  __shared__ RecordsLds S2;
  if (P.tDev) t += *P.tDev;
  load_exp_table((lds_u64 *)S2.expTab);
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (blockIdx.x == 0 && threadIdx.x < kXcds) P.workCtr[threadIdx.x * kCtrStride] = 0;  // for the next k_gather
  if (blockIdx.x == 0 && threadIdx.x == 0 && P.bigCount) *P.bigCount = 0;                 // for the next k_sort
  const uint32_t j0 = blockIdx.x * kBlock + wave * kWave;
  const uint32_t m = j0 < P.N ? min((uint32_t)kWave, P.N - j0) : 0u;
  const uint32_t n = lane < m ? P.keyCount[j0 + lane] : 0u;
  const size_t at = (size_t)(min(j0, P.N) >> 6) * P.cap * kWave;  // the wave's tile
  bool f = false;
  double te = 0.0;
  integrate_records(P, t, j0, m, P.keys + at, n, (lds_u64 *)S2.stage[wave], (lds_u64 *)S2.expTab, f, te);
  publish_spikes(P, t + 1, j0 + lane, f, te, S.popCnt, S.count);  // LTP follows in k_ltp
}

// ... or three waves per tile of 64 neurons.
__global__ __launch_bounds__(kPipeThreads) void k_integrate_pipe(DevNet P, uint32_t t, NextScan S) {
  __shared__ PipeLds L;
  if (P.tDev) t += *P.tDev;
  const uint32_t lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && threadIdx.x < kXcds) P.workCtr[threadIdx.x * kCtrStride] = 0;  // for the next k_gather
  if (blockIdx.x == 0 && threadIdx.x == 0 && P.bigCount) *P.bigCount = 0;                 // for the next k_sort
  const uint32_t j0 = blockIdx.x * kWave;
  const uint32_t m = min((uint32_t)kWave, P.N - j0);
  const uint32_t n = lane < m ? P.keyCount[j0 + lane] : 0u;
  bool f = false;
  double te = 0.0;
  integrate_pipe(P, t, j0, m, P.keys + (size_t)blockIdx.x * P.cap * kWave, n, L, f, te);
  if (threadIdx.x >= 2 * kWave)
    publish_spikes(P, t + 1, j0 + lane, f, te, S.popCnt, S.count);  // LTP follows in k_ltp
}

// The item of global tile g: the last one with tileBegin <= g.
__device__ inline uint32_t batch_item_of(const BatchItem *items, uint32_t count, uint32_t g) {
  uint32_t lo = 0, hi = count;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) / 2;
    if (items[mid].tileBegin <= g) lo = mid; else hi = mid;
  }
  return lo;
}

// Split form of a batched step over the global tiles [g0, g1) (one chunk of
// the members' concatenated tiles): k_batch_gather runs phase 1 one wave per
// neuron into the chunk's blocked scratch (tile g at (g - g0)), then
// k_batch_integrate runs phase 2, one wave per tile, and the fired scan of
// each member's next step.
template <int K, int B>
__global__ __launch_bounds__(kWave) void k_batch_gather(const DevNet *nets, const BatchItem *items, uint32_t count,
                                                        uint32_t g0, uint32_t g1, uint32_t cap, uint64_t *keys,
                                                        int16_t *keyW, uint16_t *keyPos, uint32_t *keyCount,
                                                        uint32_t *workCtr) {
  extern __shared__ uint64_t lds[];
  const uint32_t total = (g1 - g0) * kWave, home = blockIdx.x % kXcds;
  uint32_t x = home;
  // delivered events are summed per member and added to its counter when
  // the wave moves to another member (one update per run, not per neuron)
  unsigned long long *evCtr = nullptr;
  unsigned long long evSum = 0;
  for (uint32_t u0, u1; (u0 = next_item(workCtr, total, x, home, &u1)) < total;)
  for (uint32_t u = u0; u < u1; ++u) {
    const uint32_t g = g0 + u / kWave, q = u % kWave;
    const BatchItem &it = items[batch_item_of(items, count, g)];
    const DevNet &P = nets[it.net];
    const uint32_t j = (g - it.tileBegin) * kWave + q;
    if (j >= P.N) continue;
    const size_t at = (size_t)(u / kWave) * cap * kWave + q * kRun;
    const uint32_t n = gather_sort_neuron<K, B>(P, it.t, j, it.ltd, (uint8_t *)lds, cap, keys + at, keyW + at,
                                                it.ltd ? keyPos + at : nullptr, keyCount + u);
    if (P.counters != evCtr) {
      if (threadIdx.x == 0 && evSum) atomicAdd(counter_slot(evCtr), evSum);
      evCtr = P.counters;
      evSum = 0;
    }
    evSum += n;
  }
  if (threadIdx.x == 0 && evSum) atomicAdd(counter_slot(evCtr), evSum);
}

// k_bath for the members of global tiles [g0, g1), one wave per tile.
__global__ __launch_bounds__(kWave) void k_batch_bath(const DevNet *nets, const BatchItem *items, uint32_t count,
                                                      uint32_t g0) {
  const uint32_t g = g0 + blockIdx.x;
  const BatchItem &it = items[batch_item_of(items, count, g)];
  const DevNet &P = nets[it.net];
  if (!P.bathT || it.t < kPackT) return;
  const uint32_t j = (g - it.tileBegin) * kWave + threadIdx.x;
  if (P.drive == DPSNN_DRIVE_REPLAY)
    bath_step<true>(P, it.t, it.X, j);
  else
    bath_step<false>(P, it.t, it.X, j);
}

template <int PK>
__global__ __launch_bounds__(kBlock) void k_batch_integrate(const DevNet *nets, const BatchItem *items,
                                                            uint32_t count, uint32_t g0, uint32_t g1, uint32_t cap,
                                                            const uint64_t *keys, const int16_t *keyW,
                                                            const uint32_t *keyCount, uint32_t *workCtr) {
  __shared__ IntegrateLds<PK> S2;
  load_exp_table((lds_u64 *)S2.expTab);
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (blockIdx.x == 0 && threadIdx.x < kXcds) workCtr[threadIdx.x * kCtrStride] = 0;  // for the next chunk's gather
  const uint32_t g = g0 + blockIdx.x * (kBlock / kWave) + wave;
  if (g >= g1) return;  // whole wave
  const BatchItem &it = items[batch_item_of(items, count, g)];
  const DevNet &P = nets[it.net];
  const uint32_t j0 = (g - it.tileBegin) * kWave;
  const uint32_t m = min((uint32_t)kWave, P.N - j0);
  const uint32_t u = (g - g0) * kWave;
  const uint32_t n = lane < m ? keyCount[u + lane] : 0u;
  const size_t at = (size_t)(g - g0) * cap * kWave;
  bool f = false;
  double te = 0.0;
  unsigned long long ex;
  if (P.bathT && it.t >= kPackT) {
    DevNet Q = P;  // the batch's scratch has its own longest list
    Q.cap = cap;
    integrate_records(Q, it.t, j0, m, keys + at, n, (lds_u64 *)S2.stage[wave], (lds_u64 *)S2.expTab, f, te);
    ex = 0;
  } else if (P.drive == DPSNN_DRIVE_REPLAY)
    ex = integrate_wave<true, PK>(P, it.t, it.X, j0, m, keys + at, keyW + at, n, (lds_u64 *)S2.stage[wave],
                                  (lds_u64 *)S2.expTab, f, te);
  else
    ex = integrate_wave<false, PK>(P, it.t, it.X, j0, m, keys + at, keyW + at, n, (lds_u64 *)S2.stage[wave],
                                   (lds_u64 *)S2.expTab, f, te);
  publish_spikes(P, it.t + 1, j0 + lane, f, te, it.S.popCnt, it.S.count);  // LTP follows in k_batch_ltp
  for (int o = 32; o > 0; o >>= 1) ex += __shfl_down(ex, o);
  if (lane == 0 && ex) atomicAdd(counter_slot(P.counters) + 1, ex);
}

// LTP of the members' next scans over global tiles [g0, g1), one wave per
// neuron that fired (item S.ltp: the member's next scan runs LTP).
__global__ __launch_bounds__(kWaveLTP) void k_batch_ltp(const DevNet *nets, const BatchItem *items, uint32_t count,
                                                        uint32_t g0, uint32_t g1) {
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t waves = (gridDim.x * blockDim.x) >> 6;
  for (uint32_t u = wave; u < (g1 - g0) * kWave; u += waves) {
    const uint32_t g = g0 + u / kWave;
    const BatchItem &it = items[batch_item_of(items, count, g)];
    if (!it.S.ltp) continue;
    const DevNet &P = nets[it.net];
    const uint32_t j = (g - it.tileBegin) * kWave + u % kWave;
    if (j >= P.N) continue;
    const uint64_t *bits = P.bits + (size_t)((it.t + 1) & (P.RS - 1)) * P.NW;
    if ((bits[j >> 6] >> (j & 63)) & 1ull) ltp_neuron(P, it.t + 1, j);
  }
}

// The first step of a graph replay, set before it.
__global__ void k_set_t(uint32_t *t, uint32_t v) { *t = v; }

// The state after step t - 1 (slot t holds its spikes) into pinned host memory:
// v, c, Tr, Te [N] each, then a byte per neuron that fired.
__global__ __launch_bounds__(kBlock) void k_read_state(DevNet P, uint32_t t, double *out) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= P.N) return;
  out[i] = P.v[i];
  out[(size_t)P.N + i] = P.c[i];
  out[2 * (size_t)P.N + i] = P.Tr[i];
  out[3 * (size_t)P.N + i] = P.Te[i];
  const uint64_t w = P.bits[(size_t)(t & (P.RS - 1)) * P.NW + (i >> 6)];
  ((uint8_t *)(out + 4 * (size_t)P.N))[i] = (uint8_t)((w >> (i & 63)) & 1ull);
}

// The window layout's items and chunk descriptors from the in-lists (the
// host's build_window with fill; there they cost the host 50 ms and their
// upload for 45,000 neurons of 1,250 items, here a launch of 0.3 ms).  One
// workgroup per unit, wave w its targets q = w, w + kWindowWaves, ...: the
// first item of each run of one delay leaves its place in start[], every item
// finds its own from it, and base[] moves on by the run's chunks.
constexpr uint32_t kMaxPasses = 256;  // run delays are bytes
__global__ __launch_bounds__(kCollectThreads) void k_window_fill(DevNet P, uint32_t *item, uint16_t *desc) {
  __shared__ uint32_t startOf[kWindowWaves][kMaxPasses], baseOf[kWindowWaves][kMaxPasses];
  constexpr uint32_t C = kWindowChunk;
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63, u = blockIdx.x;
  uint32_t *start = startOf[wave], *base = baseOf[wave];
  const uint32_t col = u / P.winUnitsPerCol, part = u - col * P.winUnitsPerCol;
  const uint32_t j0 = col * P.npc + part * P.winUnit;
  const uint32_t m = min(P.winUnit, (col + 1) * P.npc - j0);
  const int32_t *cols = P.winCols + (size_t)col * P.winSlots;
  for (uint32_t d = lane; d < P.winPasses; d += kWave)
    base[d] = (uint32_t)P.winChunk[((size_t)u * P.winPasses + (P.winPasses - 1 - d)) * kWindowWaves + wave];
  for (uint32_t q = wave; q < m; q += kWindowWaves) {
    const uint64_t beg = P.inOff[j0 + q];
    const uint32_t len = (uint32_t)(P.inOff[j0 + q + 1] - beg);
    const uint32_t *in = P.inPD + beg;
    for (uint32_t i = lane; i < len; i += kWave) {
      const uint32_t d = in[i] >> 24;
      if (i == 0 || in[i - 1] >> 24 != d) start[d] = i;
    }
    wave_sync();
    for (uint32_t i = lane; i < len; i += kWave) {
      const uint32_t d = in[i] >> 24, src = in[i] & 0xFFFFFFu, sc = src / P.npc, off = i - start[d];
      uint32_t lo = 0, hi = P.winSlots;  // the slot of column sc: cols ascends, then -1
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if ((uint32_t)cols[mid] <= sc) lo = mid;  // -1: the largest
        else hi = mid;
      }
      const size_t ch = (size_t)base[d] + off / C;
      item[ch * C + off % C] = (lo * P.npc + (src - sc * P.npc)) << 16 | (uint16_t)P.inW[beg + i];
      if (off % C == 0) desc[ch] = (uint16_t)(q | (off == 0 ? kWindowFirst : 0u));
    }
    wave_sync();
    for (uint32_t i = lane; i < len; i += kWave) {
      const uint32_t d = in[i] >> 24;
      if (i + 1 < len && in[i + 1] >> 24 == d) continue;
      const uint32_t off = i - start[d], ch = base[d] + off / C;  // the run's last item
      for (uint32_t x = off % C + 1; x < C; ++x) item[(size_t)ch * C + x] = P.winSlots * P.npc << 16;
      base[d] = ch + 1;
    }
    wave_sync();
  }
}

// The sums of the first kReadCounters counters into pinned host memory.
constexpr uint32_t kReadCounters = 4;
__global__ void k_read_counters(const unsigned long long *counters, unsigned long long *out) {
  unsigned long long sum = 0;
  for (uint32_t k = 0; k < kCounterSlots; ++k) sum += counters[k * kCounterStride + threadIdx.x];
  out[threadIdx.x] = sum;
}

// Fills n doubles with v.
__global__ void k_fill_f64(double *p, double v, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// Launch shapes: K = in-list chunks of 64 items held in registers per
// pass, B = arrival-time buckets of the LDS sort.  Every shape computes the
// same result bit for bit; they differ only in speed.
using StepFn = void (*)(DevNet, uint32_t, ExtView, int, NextScan);
using GatherFn = void (*)(DevNet, uint32_t, int);
using BatchFn = void (*)(const DevNet *, const BatchItem *, uint32_t, uint32_t, uint32_t, uint64_t *, int16_t *,
                         uint16_t *, uint32_t *);
using BatchGatherFn = void (*)(const DevNet *, const BatchItem *, uint32_t, uint32_t, uint32_t, uint32_t, uint64_t *,
                               int16_t *, uint16_t *, uint32_t *, uint32_t *);
using SortFn = void (*)(DevNet, uint32_t);
struct KernelShape {
  int K, B;
  StepFn step;
  GatherFn gather;
  BatchFn batch;
  BatchGatherFn batchGather;
  SortFn sort, sortBig;
};
#define DPSNN_SHAPE(k, b) \
  {k, b, k_step<k, b>, k_gather<k, b>, k_batch_step<k, b>, k_batch_gather<k, b>, k_sort<b>, k_sort_big<b>}
static const KernelShape kShapes[] = {
    DPSNN_SHAPE(8, 64),  DPSNN_SHAPE(8, 256),  DPSNN_SHAPE(8, 1024),
    DPSNN_SHAPE(16, 64), DPSNN_SHAPE(16, 256), DPSNN_SHAPE(16, 1024),
    DPSNN_SHAPE(24, 64), DPSNN_SHAPE(24, 256), DPSNN_SHAPE(24, 1024),
};
#undef DPSNN_SHAPE
constexpr int kNumShapes = (int)(sizeof(kShapes) / sizeof(kShapes[0]));

static uint32_t round_up(uint32_t x, uint32_t m) { return (x + m - 1) / m * m; }

// Phase-1 waves (one-wave workgroups) resident per CU for a kernel and its
// LDS, from the runtime's occupancy calculator.
static uint32_t resident_waves(const void *kernel, size_t lds) {
  int blocks = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, kWave, lds) != hipSuccess || blocks < 1)
    blocks = 1;
  return (uint32_t)blocks;
}

static int find_shape(int K, int B) {
  for (int i = 0; i < kNumShapes; ++i)
    if (kShapes[i].K == K && kShapes[i].B == B) return i;
  return -1;
}

static size_t lds_bytes(uint32_t cap, int B) { return step_lds(cap, B); }

}  // namespace dpsnn

// ============================================================================
// Host engine
// ============================================================================
using namespace dpsnn;

struct ExtSlot {
  uint32_t *h_off = nullptr;
  double *h_time = nullptr, *h_value = nullptr;
  size_t capEv = 0;
  uint32_t *d_off = nullptr;
  double *d_time = nullptr, *d_value = nullptr;
  hipEvent_t done = nullptr;
  bool pending = false;
};

struct dpsnn_net {
  Params par;
  Connectome con;
  Ran3 rng;
  ExternalReplay replay;
  ExternalStep extStep;
  StatWriter writer;
  bool writing = false;
  StdpEventWriter stdpWriter;  // the STDPevent file (host restatement from the spikes)
  bool stdpEvents = false;
  dpsnn_options opt{};
  hipStream_t stream = nullptr;
  DevNet dev{};
  std::vector<void *> allocs;
  uint64_t devBytes = 0;
  // history
  uint32_t t = 0;
  // external ring
  ExtSlot ext[kExtRing];
  uint32_t extNext = 0;
  // raster drain
  uint32_t *d_rasterIds = nullptr;
  double *d_rasterTe = nullptr;
  uint32_t *d_rasterCount = nullptr;  // [1]
  uint32_t *d_stepCount = nullptr;    // [drain]
  uint32_t *d_popCnt = nullptr;       // [drain][ncols*nsub]
  uint32_t rasterCap = 0, drainEvery = 100, pendingSteps = 0, pendingFrom = 0;
  bool wantRaster = false;
  std::vector<uint32_t> h_ids, h_steps, h_pop;
  std::vector<double> h_te;
  // last spikes
  std::vector<uint32_t> lastIds, aheadIds;
  std::vector<double> lastTe, aheadTe;
  uint32_t aheadMs = UINT32_MAX;
  double initSeconds = 0;
  uint64_t items = 0;
  uint32_t grid = 0;
  size_t ldsBytes = 0;
  bool stdp = false;         // plasticity runs at some step of [0, total)
  uint32_t stdpBlock = 0;    // most steps whose LTD and LTP one k_stdp may make (0: step by step)
  bool deferring = false;    // inside such a block: its first step, and the steps left of it
  uint32_t blockFrom = 0, blockLeft = 0;
  bool uploaded = false;     // build_device done (dpsnn_upload)
  std::string outDir;        // owned copy of opt.output_dir
  uint32_t stdpBlocks = 0;
  int shape = 0;             // kShapes index
  struct dpsnn_batch *batch = nullptr;  // stepped by this batch (its stream)
  hipStream_t ownStream = nullptr;
  bool split = false;        // k_gather + k_integrate instead of the fused k_step
  bool pipe = false;         // k_integrate_pipe instead of k_integrate (t >= kPackT)
  uint32_t gatherGrid = 0;
  std::vector<uint16_t> inSynLocal;
  // stencil-window phase 1 (k_collect + k_sort)
  WindowLayout window;       // host staging until upload
  bool winOn = false;        // the device holds the layout
  uint32_t winGrid = 0, sortGrid = 0, sortBigGrid = 0;
  size_t winLds = 0;
  // profiling
  bool profile = false;
  struct ProfEv {
    hipEvent_t a, b;
    uint32_t steps;  // steps between a and b
  };
  std::vector<ProfEv> profEv;
  size_t profUsed = 0;
  // graph-replayed steps (kGraphSteps consecutive plain steps per replay)
  hipGraphExec_t stepGraph = nullptr;
  const uint64_t *graphKeys = nullptr;  // the key scratch the graph was captured with
  uint32_t *d_t = nullptr;
  bool graphs = true;        // DPSNN_GRAPH=0: plain launches only
  uint64_t graphSteps = 0;   // steps replayed from the graph so far
  bool collect = false;  // raster / rates are being produced
  // pinned host memory of read-backs, allocated at the first one; readMu: two
  // threads may read one network's state or counters at a time
  std::mutex readMu;
  double *h_state = nullptr;                 // k_read_state's
  unsigned long long *h_counters = nullptr;  // k_read_counters'
  uint8_t *h_drain = nullptr;                // kDrainBytes
};

template <class T>
static int dev_alloc(dpsnn_net *n, T **p, size_t count) {
  const size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
  hipError_t e = hipMalloc((void **)p, bytes);
  if (e != hipSuccess)
    return fail(DPSNN_ERR_MEMORY, "hipMalloc of %zu bytes failed: %s", bytes, hipGetErrorString(e));
  n->allocs.push_back(*p);
  n->devBytes += bytes;
  return 0;
}
template <class T>
static int upload(dpsnn_net *n, T *d, const T *h, size_t count) {
  HIP_TRY(hipMemcpyAsync(d, h, count * sizeof(T), hipMemcpyHostToDevice, n->stream));
  return 0;
}

static void free_all(dpsnn_net *n) {
  if (n->stream) hipStreamSynchronize(n->stream);
  for (void *p : n->allocs) hipFree(p);
  n->allocs.clear();
  for (auto &s : n->ext) {
    if (s.h_off) hipHostFree(s.h_off);
    if (s.h_time) hipHostFree(s.h_time);
    if (s.h_value) hipHostFree(s.h_value);
    if (s.d_off) hipFree(s.d_off);
    if (s.d_time) hipFree(s.d_time);
    if (s.d_value) hipFree(s.d_value);
    if (s.done) hipEventDestroy(s.done);
    s = ExtSlot{};
  }
  for (void *p : {(void *)n->h_state, (void *)n->h_counters, (void *)n->h_drain})
    if (p) (void)hipHostFree(p);
  n->h_state = nullptr;
  n->h_counters = nullptr;
  n->h_drain = nullptr;
  for (auto &e : n->profEv) {
    hipEventDestroy(e.a);
    hipEventDestroy(e.b);
  }
  if (n->stepGraph) hipGraphExecDestroy(n->stepGraph);
  n->stepGraph = nullptr;
  n->profEv.clear();
  if (n->stream) hipStreamDestroy(n->stream);
  n->stream = nullptr;
}

// Uploads the stencil-window layout and sizes k_collect (one workgroup of
// kCollectThreads per CU: its LDS holds a whole window) and k_sort.
static int upload_window(dpsnn_net *n, int cus) {
  const WindowLayout &L = n->window;
  DevNet &P = n->dev;
  size_t lds = collect_lds(L.slots * L.npc, L.unit);
  int maxLds = 0;
  HIP_TRY(hipDeviceGetAttribute(&maxLds, hipDeviceAttributeMaxSharedMemoryPerBlock, n->opt.device));
  if (lds > (size_t)maxLds) return 0;  // the gather form stays
  // the sort fused into k_collect: its waves' sort areas overlay the window
  const KernelShape &K = kShapes[n->shape];
  const size_t fusedLds = std::max(lds, (size_t)kWindowWaves * fused_sort_stride());
  // (DPSNN_FUSED_SORT=0/1 overrides the default, for tests and timing)
  const char *fe = getenv("DPSNN_FUSED_SORT");
  const bool fuse = fe ? atoi(fe) != 0 : kFusedSortDefault;
  P.fuseSort = fuse && K.B == kFusedSortB && L.unit <= (uint32_t)kCollectThreads && fusedLds <= (size_t)maxLds;
  if (P.fuseSort) lds = fusedLds;
  // the device's limit, not this network's size: networks of other sizes
  // launch the same kernel
  if (lds > (size_t)64 * 1024)
    HIP_TRY(hipFuncSetAttribute((const void *)k_collect, hipFuncAttributeMaxDynamicSharedMemorySize, maxLds));
  uint32_t *d_item;
  uint16_t *d_desc;
  uint64_t *d_chunk;
  int32_t *d_cols;
  int rc;
  if (L.passes > kMaxPasses) return fail(DPSNN_ERR_CONFIG, "%u run delays", L.passes);
  if ((rc = dev_alloc(n, &d_item, L.items())) || (rc = dev_alloc(n, &d_desc, L.chunks())) ||
      (rc = dev_alloc(n, &d_chunk, L.chunk.size())) || (rc = upload(n, d_chunk, L.chunk.data(), L.chunk.size())) ||
      (rc = dev_alloc(n, &d_cols, L.cols.size())) || (rc = upload(n, d_cols, L.cols.data(), L.cols.size())) ||
      (rc = dev_alloc(n, &P.winCtr, kXcds * kCtrStride)) || (rc = dev_alloc(n, &P.bigList, P.N)) ||
      (rc = dev_alloc(n, &P.bigCount, 1)))
    return rc;
  HIP_TRY(hipMemsetAsync(P.winCtr, 0, sizeof(uint32_t) * kXcds * kCtrStride, n->stream));
  HIP_TRY(hipMemsetAsync(P.bigCount, 0, sizeof(uint32_t), n->stream));
  P.winItem = d_item; P.winDesc = d_desc; P.winChunk = d_chunk; P.winCols = d_cols;
  P.winSlots = L.slots; P.winPasses = L.passes; P.winUnit = L.unit; P.winUnitsPerCol = L.unitsPerCol;
  P.winUnits = L.units;
  hipLaunchKernelGGL(k_window_fill, dim3(L.units), dim3(kCollectThreads), 0, n->stream, P, d_item, d_desc);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(n->stream));  // the host staging is dropped after upload
  // DPSNN_SORT_CAP lowers k_sort's limit, so that tests send targets through
  // k_sort_big
  P.sortCap = kSortCap;
  if (const char *e = getenv("DPSNN_SORT_CAP")) P.sortCap = std::min<uint32_t>(kSortCap, (uint32_t)atoi(e));
  n->winLds = lds;
  n->winGrid = round_up(std::min<uint32_t>(L.units, (uint32_t)cus), kXcds);
  n->sortGrid = round_up(
      std::min<uint32_t>(P.N, (uint32_t)cus * resident_waves((const void *)K.sort, phase1_lds(kSortCap, K.B))), kXcds);
  n->sortBigGrid = std::min<uint32_t>(P.N, (uint32_t)cus * 4);
  n->winOn = true;
  return 0;
}

static uint32_t round_scratch(uint32_t records) {  // to a whole number of scratch runs
  return (std::max<uint32_t>(records, 1) + (kRun - 1)) / kRun * kRun;
}

// The most bath events of a neuron and ms, where a step's bath can be drawn
// ahead of phase 1 and sorted in there: every sub-population's bath events
// have one value (a float; DJExt = 0), and the records of a target stay
// within the 12 bits of the sort key's position.  0: phase 2 draws and merges
// the bath.  DPSNN_BATH=0 asks for that (tests; the results are the same).
static uint32_t bath_cap(const dpsnn_net *n) {
  const Connectome &c = n->con;
  if (const char *e = std::getenv("DPSNN_BATH"))
    if (std::atoi(e) == 0) return 0;
  const char *split = std::getenv("DPSNN_SPLIT"), *fused = std::getenv("DPSNN_FUSED_SORT");
  if ((split && std::atoi(split) == 0) || (fused && std::atoi(fused) != 0)) return 0;
  for (uint32_t s = 0; s < n->par.pub.subPopNumber; ++s) {
    const double *lut = &c.bathLut[size_t(s) * kLutDepth];
    for (uint32_t i = 0; i < kLutDepth; ++i)
      if (lut[i] != lut[0] || lut[0] != (double)(float)lut[0]) return 0;
  }
  uint32_t cap = 1;
  for (uint32_t i = 0; i < c.N; ++i) cap = std::max(cap, c.maxExt[i]);
  return cap <= kBathMax && c.max_in + cap < (1u << 12) - 1 ? cap : 0;
}

// Bath lists and values on the device, and the scratch's record cap with them.
static int plan_bath(dpsnn_net *n) {
  DevNet &P = n->dev;
  const uint32_t cap = bath_cap(n);
  if (!cap) return 0;
  std::vector<float> value(P.nsub);
  for (uint32_t s = 0; s < P.nsub; ++s) value[s] = (float)n->con.bathLut[size_t(s) * kLutDepth];
  float *d_value;
  int rc;
  if ((rc = dev_alloc(n, &d_value, P.nsub)) || (rc = upload(n, d_value, value.data(), P.nsub)) ||
      (rc = dev_alloc(n, &P.bathT, (size_t)cap * P.N)) || (rc = dev_alloc(n, &P.bathN, P.N)))
    return rc;
  HIP_TRY(hipStreamSynchronize(n->stream));  // `value` ends here
  P.bathV = d_value;
  P.cap = round_scratch(n->con.max_in + cap);
  return 0;
}

static int build_device(dpsnn_net *n) {
  Connectome &c = n->con;
  const dpsnn_parameters &q = n->par.pub;
  DevNet &P = n->dev;
  P.N = c.N;
  P.NW = (c.N + 63) / 64;
  // live slots t-maxDelay..t plus the one step t+1 writes, rounded to a
  // power of two (slot = ms & (RS - 1))
  P.RS = 1;
  while (P.RS < c.max_delay + 2) P.RS <<= 1;
  // phase 1 addresses the spike history with 32-bit byte offsets and 24-bit
  // neuron indices
  if (c.N >= (1u << 24)) return fail(DPSNN_ERR_CONFIG, "%u neurons; the engine handles fewer than 2^24", c.N);
  if (uint64_t(P.RS) * c.N * sizeof(double) > (1ull << 32))
    return fail(DPSNN_ERR_CONFIG, "spike history (%u slots x %u neurons) larger than 4 GiB", P.RS, c.N);
  P.nsub = q.subPopNumber;
  P.npc = q.neuronsPerCM;
  P.ncols = q.globCFT;
  P.cap = round_scratch(c.max_in);  // records of a target (plan_bath adds the bath's)
  // DPSNN_PHASE1_DENSE_MAX lowers the fast path's limit (0: every neuron on
  // the general path), so that tests can compare the two paths
  P.denseMax = kDense * kWave;
  if (const char *e = getenv("DPSNN_PHASE1_DENSE_MAX")) P.denseMax = std::min<uint32_t>(P.denseMax, (uint32_t)atoi(e));
  P.drive = (uint32_t)n->opt.drive;
  P.w2f = q.factorWeightType_2_Float;
  P.philoxSeed = n->opt.philox_seed;
  int rc;
  const uint32_t N = c.N;
  // per-subPop parameters and LUT
  std::vector<double> sp(size_t(P.nsub) * kParams, 0.0);
  for (uint32_t s = 0; s < P.nsub; ++s) {
    const SubPop &x = n->par.sp[s];
    double *o = &sp[size_t(s) * kParams];
    o[kTheta] = x.Theta; o[kH] = x.H; o[kTarp] = x.Tarp;
    o[kAlphaC] = x.AlphaC; o[kGC] = x.gC;
    // div_short's divisors: floats (as the ini files are read), not zero
    for (double d : {x.Tau, x.TauC})
      if (!(std::fabs(d) > 0 && std::isfinite(d) && short_divisor(d)))
        return fail(DPSNN_ERR_CONFIG, "sub-population %u: time constant %g outside the supported range", s, d);
    o[kInvTau] = 1.0 / x.Tau;
    o[kInvTauLo] = std::fma(-x.Tau, o[kInvTau], 1.0) / x.Tau;
    o[kInvTauC] = 1.0 / x.TauC;
    o[kInvTauCLo] = std::fma(-x.TauC, o[kInvTauC], 1.0) / x.TauC;
  }
  double *d_sp, *d_lut, *d_inv;
  uint8_t *d_sub;
  uint32_t *d_maxExt;
  if ((rc = dev_alloc(n, &d_sp, sp.size())) || (rc = upload(n, d_sp, sp.data(), sp.size()))) return rc;
  if ((rc = dev_alloc(n, &d_lut, c.bathLut.size())) || (rc = upload(n, d_lut, c.bathLut.data(), c.bathLut.size()))) return rc;
  if ((rc = dev_alloc(n, &d_inv, N)) || (rc = upload(n, d_inv, c.invNuExt.data(), N))) return rc;
  if ((rc = dev_alloc(n, &d_sub, N)) || (rc = upload(n, d_sub, c.subPop.data(), N))) return rc;
  if ((rc = dev_alloc(n, &d_maxExt, N)) || (rc = upload(n, d_maxExt, c.maxExt.data(), N))) return rc;
  P.sp = d_sp; P.lut = d_lut; P.invNuExt = d_inv; P.subPop = d_sub; P.maxExt = d_maxExt;
  // neuron state, initNeuralKind DPSNN_neuron_init.c:99-115
  std::vector<double> v(N), zeros(N, 0.0), te(N, -1000.0);
  for (uint32_t i = 0; i < N; ++i) v[i] = n->par.sp[c.subPop[i]].H;
  if ((rc = dev_alloc(n, &P.v, N)) || (rc = upload(n, P.v, v.data(), N))) return rc;
  if ((rc = dev_alloc(n, &P.c, N)) || (rc = upload(n, P.c, zeros.data(), N))) return rc;
  if ((rc = dev_alloc(n, &P.Tr, N)) || (rc = upload(n, P.Tr, zeros.data(), N))) return rc;
  if ((rc = dev_alloc(n, &P.Te, N)) || (rc = upload(n, P.Te, te.data(), N))) return rc;
  if ((rc = dev_alloc(n, &P.assigned, N)) || (rc = upload(n, P.assigned, zeros.data(), N))) return rc;
  if ((rc = dev_alloc(n, &P.philoxCtr, N))) return rc;
  HIP_TRY(hipMemsetAsync(P.philoxCtr, 0, sizeof(uint64_t) * N, n->stream));
  // history
  if ((rc = dev_alloc(n, &P.bits, size_t(P.RS) * P.NW))) return rc;
  HIP_TRY(hipMemsetAsync(P.bits, 0, sizeof(uint64_t) * size_t(P.RS) * P.NW, n->stream));
  if ((rc = dev_alloc(n, &P.teHist, size_t(P.RS) * N))) return rc;
  hipLaunchKernelGGL(k_fill_f64, dim3(1024), dim3(256), 0, n->stream, P.teHist, kNotFired, uint64_t(P.RS) * N);
  HIP_TRY(hipGetLastError());
  // in-lists (CSR in delivery insertion order)
  if (c.max_in >= kMaxInList)
    return fail(DPSNN_ERR_CONFIG, "a neuron has %u in-list items; the engine handles up to %u", c.max_in,
                kMaxInList - 1);
  n->items = c.in_off[N];
  if ((rc = plan_bath(n))) return rc;
  {
    uint64_t *d_off;
    uint32_t *d_pd;
    int16_t *d_w;
    const uint64_t items = c.in_off[N];
    if ((rc = dev_alloc(n, &d_off, N + 1)) || (rc = upload(n, d_off, c.in_off.data(), N + 1))) return rc;
    // one wave of padding: phase 1 loads whole waves of in-list words
    if ((rc = dev_alloc(n, &d_pd, items + kWave)) || (rc = upload(n, d_pd, c.in_pre_d.data(), items))) return rc;
    HIP_TRY(hipMemsetAsync(d_pd + items, 0, sizeof(uint32_t) * kWave, n->stream));
    if ((rc = dev_alloc(n, &d_w, items)) || (rc = upload(n, d_w, c.in_w.data(), items))) return rc;
    P.inOff = d_off; P.inPD = d_pd; P.inW = d_w;
    HIP_TRY(hipStreamSynchronize(n->stream));  // host staging is dropped after create
  }
  // STDP state, target-major (see DevNet)
  if (n->stdp) {
    const uint64_t S = c.S;
    std::vector<int16_t> wT(S);
    std::vector<uint8_t> kindT(S);
    for (uint64_t k = 0; k < S; ++k) {
      wT[k] = c.weight[c.inc_syn[k]];
      kindT[k] = c.kind[c.inc_syn[k]];
    }
    uint64_t *d_incOff;
    uint8_t *d_kind;
    uint16_t *d_inSyn;
    float *d_causal, *d_anti, *d_max, *d_rev;
    if ((rc = dev_alloc(n, &d_incOff, N + 1)) || (rc = upload(n, d_incOff, c.inc_off.data(), N + 1))) return rc;
    if ((rc = dev_alloc(n, &P.wT, S)) || (rc = upload(n, P.wT, wT.data(), S))) return rc;
    if ((rc = dev_alloc(n, &d_kind, S)) || (rc = upload(n, d_kind, kindT.data(), S))) return rc;
    if ((rc = dev_alloc(n, &d_inSyn, c.in_off[N] + kWave)) ||  // padded like the in-list words
        (rc = upload(n, d_inSyn, n->inSynLocal.data(), c.in_off[N])))
      return rc;
    HIP_TRY(hipMemsetAsync(d_inSyn + c.in_off[N], 0, sizeof(uint16_t) * kWave, n->stream));
    if ((rc = dev_alloc(n, &P.tdT, S)) || (rc = dev_alloc(n, &P.lastT, S))) return rc;
    HIP_TRY(hipMemsetAsync(P.tdT, 0, 4 * S, n->stream));
    HIP_TRY(hipMemsetAsync(P.lastT, 0, 4 * S, n->stream));
    if (!q.statSynPeriodicProbe_writeDisable) {
      if ((rc = dev_alloc(n, &P.tdPre, S))) return rc;
    }
    std::vector<int32_t> lastSpike(N, -100000);  // DPSNN_localNet_init.c:217
    if ((rc = dev_alloc(n, &P.lastSpike, N)) || (rc = upload(n, P.lastSpike, lastSpike.data(), N))) return rc;
    if ((rc = dev_alloc(n, &P.lastSpike0, N)) || (rc = dev_alloc(n, &P.spikeMask, N))) return rc;
    HIP_TRY(hipMemsetAsync(P.spikeMask, 0, 4 * (size_t)N, n->stream));
    // tables, initLongTermPlasticity DPSNN_neuron_sim.c:45-92
    std::vector<float> causal, anti;
    stdp_tables(q, causal, anti);
    std::vector<float> maxSyn(size_t(P.nsub) * P.nsub), rev(size_t(P.nsub) * P.nsub);
    for (uint32_t a = 0; a < P.nsub; ++a)
      for (uint32_t b = 0; b < P.nsub; ++b) {
        maxSyn[a * P.nsub + b] = 2.0 * n->par.sp[a].J[b];  // source a -> target b
        rev[a * P.nsub + b] = 2.0 * n->par.sp[b].J[a];
      }
    if ((rc = dev_alloc(n, &d_causal, kStdpSpan)) || (rc = upload(n, d_causal, causal.data(), kStdpSpan))) return rc;
    if ((rc = dev_alloc(n, &d_anti, kStdpSpan)) || (rc = upload(n, d_anti, anti.data(), kStdpSpan))) return rc;
    if ((rc = dev_alloc(n, &d_max, maxSyn.size())) || (rc = upload(n, d_max, maxSyn.data(), maxSyn.size()))) return rc;
    if ((rc = dev_alloc(n, &d_rev, rev.size())) || (rc = upload(n, d_rev, rev.data(), rev.size()))) return rc;
    P.incOff = d_incOff; P.kindT = d_kind; P.inSyn = d_inSyn;
    P.causal = d_causal; P.anti = d_anti; P.maxSyn = d_max; P.revMax = d_rev;
    P.f2w = q.factorFloat_2_weightType;
    P.drift = q.derivativeDrift;
    P.decayReset = q.tauDerivativeDecay_s == 1.0 ? 1 : 0;
    P.decayMul = (1 - 1 / q.tauDerivativeDecay_s);
    HIP_TRY(hipStreamSynchronize(n->stream));
  }
  // launch shapes.  The split form (k_gather, one wave per neuron, then
  // k_integrate) is the default; the fused k_step (each wave whole tiles of
  // 64 neurons) is kept as an option (DPSNN_SPLIT=0).
  int cus = 0;
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, n->opt.device));
  cus = std::max(cus, 1);
  const uint32_t tiles = P.NW;
  int K = c.max_in <= 8 * 64 ? 8 : (c.max_in <= 16 * 64 ? 16 : 24), B = 256;
  if (const char *e = std::getenv("DPSNN_CHUNKS")) K = std::atoi(e);
  if (const char *e = std::getenv("DPSNN_BUCKETS")) B = std::atoi(e);
  n->shape = find_shape(K, B);
  if (n->shape < 0) return fail(DPSNN_ERR_ARG, "no kernel shape with %d register chunks and %d buckets", K, B);
  n->ldsBytes = lds_bytes(P.cap, B);
  const uint32_t wavesPerCu = std::max<uint32_t>(1, std::min<uint32_t>(16, (uint32_t)((160u << 10) / n->ldsBytes)));
  n->grid = round_up(std::min<uint32_t>(tiles, (uint32_t)cus * wavesPerCu), kXcds);
  n->stdpBlocks = std::min<uint32_t>((N + 3) / 4, (uint32_t)cus * 16);
  n->split = true;
  if (const char *e = std::getenv("DPSNN_SPLIT")) n->split = std::atoi(e) != 0;
  // k_stdp's blocks: the mask holds slots t0 - delay .. t0 + K, and every
  // synapse has one item.  DPSNN_STDP_BLOCK lowers their steps (0: step by
  // step), for tests and timing; the results are the same
  if (n->stdp && n->split && c.in_off[N] == c.S && c.max_delay + 1 + kStdpBlockMin < kMaskSlots) {
    n->stdpBlock = std::min<uint32_t>(kStdpBlock, kMaskSlots - 1 - c.max_delay);
    if (const char *e = std::getenv("DPSNN_STDP_BLOCK"))
      n->stdpBlock = std::min<uint32_t>(n->stdpBlock, (uint32_t)std::max(0, std::atoi(e)));
  }
  // DPSNN_PIPE=0/1: phase 2 in one wave or three waves per tile (tests; the
  // results are the same)
  n->pipe = P.NW <= kPipeTiles;
  if (const char *e = std::getenv("DPSNN_PIPE")) n->pipe = std::atoi(e) != 0;
  if (const char *e = std::getenv("DPSNN_GRAPH")) n->graphs = std::atoi(e) != 0;
  n->gatherGrid = round_up(
      std::min<uint32_t>(N, (uint32_t)cus * resident_waves((const void *)kShapes[n->shape].gather,
                                                               phase1_lds(P.cap, kShapes[n->shape].B))),
      kXcds);
  if (n->window.ok && (rc = upload_window(n, cus))) return rc;
  // the key scratch of stand-alone steps is allocated at the first
  // dpsnn_step (a network stepped only by a batch uses the batch's)
  if ((rc = dev_alloc(n, &P.workCtr, kXcds * kCtrStride))) return rc;
  HIP_TRY(hipMemsetAsync(P.workCtr, 0, sizeof(uint32_t) * kXcds * kCtrStride, n->stream));
  if ((rc = dev_alloc(n, &P.counters, kCounterSlots * kCounterStride))) return rc;
  HIP_TRY(hipMemsetAsync(P.counters, 0, sizeof(unsigned long long) * kCounterSlots * kCounterStride, n->stream));
  // raster / rates drain buffers
  n->drainEvery = n->opt.drain_every_ms ? n->opt.drain_every_ms : 100;
  const size_t popPer = size_t(P.ncols) * P.nsub;
  if ((rc = dev_alloc(n, &n->d_popCnt, popPer * n->drainEvery))) return rc;
  HIP_TRY(hipMemsetAsync(n->d_popCnt, 0, sizeof(uint32_t) * popPer * n->drainEvery, n->stream));
  n->wantRaster = (n->writing && !q.spikes_writeDisable) || n->opt.keep_spikes || n->stdpEvents;
  n->collect = n->writing || n->opt.keep_spikes;
  if (n->wantRaster) {
    n->rasterCap = N * std::min<uint32_t>(n->drainEvery, 1000) + 1;
    if ((rc = dev_alloc(n, &n->d_rasterIds, n->rasterCap)) || (rc = dev_alloc(n, &n->d_rasterTe, n->rasterCap)) ||
        (rc = dev_alloc(n, &n->d_rasterCount, 1)) || (rc = dev_alloc(n, &n->d_stepCount, n->drainEvery)))
      return rc;
    HIP_TRY(hipMemsetAsync(n->d_rasterCount, 0, sizeof(uint32_t), n->stream));
  }
  // external replay slots
  if (P.drive == DPSNN_DRIVE_REPLAY) {
    for (auto &s : n->ext) {
      HIP_TRY(hipHostMalloc((void **)&s.h_off, sizeof(uint32_t) * (N + 1), 0));
      HIP_TRY(hipMalloc((void **)&s.d_off, sizeof(uint32_t) * (N + 1)));
      HIP_TRY(hipEventCreateWithFlags(&s.done, hipEventDisableTiming));
    }
  }
  HIP_TRY(hipStreamSynchronize(n->stream));
  return 0;
}

static int ensure_ext_cap(ExtSlot &s, size_t need) {
  if (need <= s.capEv) return 0;
  const size_t cap = need + need / 2 + 1024;
  if (s.h_time) hipHostFree(s.h_time);
  if (s.h_value) hipHostFree(s.h_value);
  if (s.d_time) hipFree(s.d_time);
  if (s.d_value) hipFree(s.d_value);
  HIP_TRY(hipHostMalloc((void **)&s.h_time, sizeof(double) * cap, 0));
  HIP_TRY(hipHostMalloc((void **)&s.h_value, sizeof(double) * cap, 0));
  HIP_TRY(hipMalloc((void **)&s.d_time, sizeof(double) * cap));
  HIP_TRY(hipMalloc((void **)&s.d_value, sizeof(double) * cap));
  s.capEv = cap;
  return 0;
}

// Device-to-host copies gathered in pinned memory: a copy into pageable memory
// costs the caller 30 us and a wait each.  add() queues one (a piece that does
// not fit goes straight to its place); fetch() waits for the stream and moves
// the pieces to theirs.
constexpr size_t kDrainBytes = size_t(1) << 18;
struct PinnedCopies {
  dpsnn_net *n;
  size_t used = 0;
  struct Piece {
    void *to;
    size_t at, bytes;
  };
  std::vector<Piece> pieces;
  int add(void *to, const void *from, size_t bytes) {
    if (!n->h_drain) HIP_TRY(hipHostMalloc((void **)&n->h_drain, kDrainBytes, 0));
    if (used + bytes > kDrainBytes) {
      HIP_TRY(hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToHost, n->stream));
      return 0;
    }
    HIP_TRY(hipMemcpyAsync(n->h_drain + used, from, bytes, hipMemcpyDeviceToHost, n->stream));
    pieces.push_back({to, used, bytes});
    used += (bytes + 63) / 64 * 64;
    return 0;
  }
  int fetch() {
    HIP_TRY(hipStreamSynchronize(n->stream));
    for (const Piece &p : pieces) std::memcpy(p.to, n->h_drain + p.at, p.bytes);
    pieces.clear();
    used = 0;
    return 0;
  }
};

// Copies the pending raster / rates out of device memory and writes files.
static int drain(dpsnn_net *n) {
  if (n->opt.keep_spikes && n->aheadMs != UINT32_MAX && n->aheadMs + 1 == n->t) {
    n->lastIds.swap(n->aheadIds);
    n->lastTe.swap(n->aheadTe);
    n->aheadMs = UINT32_MAX;
  }
  if (n->pendingSteps == 0) return 0;
  const DevNet &P = n->dev;
  const size_t popPer = size_t(P.ncols) * P.nsub;
  const uint32_t steps = n->pendingSteps;
  PinnedCopies copies{n};
  int rc;
  n->h_pop.resize(popPer * steps);
  if ((rc = copies.add(n->h_pop.data(), n->d_popCnt, sizeof(uint32_t) * popPer * steps))) return rc;
  uint32_t total = 0;
  if (n->wantRaster) {
    n->h_steps.resize(steps);
    if ((rc = copies.add(n->h_steps.data(), n->d_stepCount, sizeof(uint32_t) * steps)) ||
        (rc = copies.add(&total, n->d_rasterCount, sizeof(uint32_t))) || (rc = copies.fetch()))
      return rc;
    n->h_ids.resize(total);
    n->h_te.resize(total);
    if (total && ((rc = copies.add(n->h_ids.data(), n->d_rasterIds, sizeof(uint32_t) * total)) ||
                  (rc = copies.add(n->h_te.data(), n->d_rasterTe, sizeof(double) * total))))
      return rc;
    HIP_TRY(hipMemsetAsync(n->d_rasterCount, 0, sizeof(uint32_t), n->stream));
  }
  HIP_TRY(hipMemsetAsync(n->d_popCnt, 0, sizeof(uint32_t) * popPer * steps, n->stream));
  if ((rc = copies.fetch())) return rc;
  uint32_t pos = 0;
  for (uint32_t k = 0; k < steps; ++k) {
    const uint32_t cnt = n->wantRaster ? n->h_steps[k] : 0;
    if (n->writing &&
        !n->writer.step(n->pendingFrom + k, n->h_ids.data() + pos, n->h_te.data() + pos, cnt,
                        n->h_pop.data() + popPer * k))
      return fail(DPSNN_ERR_IO, "writing output files in %s failed", n->opt.output_dir);
    if (n->stdpEvents && !n->stdpWriter.step(n->pendingFrom + k, n->h_ids.data() + pos, cnt))
      return fail(DPSNN_ERR_IO, "writing the STDPevent file in %s failed", n->opt.output_dir);
    // last_spikes reports the scan of the last completed step (ms t - 1);
    // the record of ms t, already produced, waits for the next step
    const uint32_t m = n->pendingFrom + k;
    if (n->opt.keep_spikes && (m + 1 == n->t || m == n->t)) {
      std::vector<uint32_t> &ids = m + 1 == n->t ? n->lastIds : n->aheadIds;
      std::vector<double> &te = m + 1 == n->t ? n->lastTe : n->aheadTe;
      ids.assign(n->h_ids.begin() + pos, n->h_ids.begin() + pos + cnt);
      te.assign(n->h_te.begin() + pos, n->h_te.begin() + pos + cnt);
      if (m == n->t) n->aheadMs = m;
    }
    pos += cnt;
  }
  n->pendingSteps = 0;
  // the files hold every drained step once a drain returns (dpsnn_sync and
  // the end of the run read them complete)
  if (n->writing) n->writer.flush();
  return 0;
}

// Downloads the target-major STDP state into backward-list order.
static int synapse_state(dpsnn_net *n, int16_t *w, float *td, int32_t *last, const float *tdSrc = nullptr) {
  const Connectome &c = n->con;
  const uint64_t S = c.S;
  std::vector<int16_t> wT(S);
  std::vector<float> tdT(S);
  std::vector<int32_t> lastT(S);
  HIP_TRY(hipStreamSynchronize(n->stream));
  HIP_TRY(hipMemcpy(wT.data(), n->dev.wT, 2 * S, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(tdT.data(), tdSrc ? tdSrc : n->dev.tdT, 4 * S, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(lastT.data(), n->dev.lastT, 4 * S, hipMemcpyDeviceToHost));
  for (uint64_t k = 0; k < S; ++k) {
    const uint32_t b = c.inc_syn[k];
    if (w) w[b] = wT[k];
    if (td) td[b] = tdT[k];
    if (last) last[b] = lastT[k];
  }
  return 0;
}

// synPeriodicProbe_A/B (DPSNN_localNet_sim.c:361-364, :394-397 with the
// record format of DPSNN_synapse.h:63-91): every synapse before and after
// the commit, backward-list order.
static int write_probe(dpsnn_net *n, const char *prefix, uint32_t sec, const float *tdSrc) {
  const Connectome &c = n->con;
  const dpsnn_parameters &q = n->par.pub;
  std::vector<int16_t> w(c.S);
  std::vector<float> td(c.S);
  int rc = synapse_state(n, w.data(), td.data(), nullptr, tdSrc);
  if (rc) return rc;
  char name[512];
  if (q.howManyOutputFiles == 1)
    std::snprintf(name, sizeof name, "%s/%s-sec%u-C%u-H%u-h%03u.dat", n->opt.output_dir, prefix, sec, q.globCFT,
                  q.globH, 0u);
  else if (sec == 0)
    std::snprintf(name, sizeof name, "%s/%s-start-C%u-H%u-h%u.dat", n->opt.output_dir, prefix, q.globCFT, q.globH, 0u);
  else
    std::snprintf(name, sizeof name, "%s/%s-%s-C%u-H%u-h%u.dat", n->opt.output_dir, prefix,
                  sec % 2 == 0 ? "lasteven" : "lastodd", q.globCFT, q.globH, 0u);
  FILE *f = std::fopen(name, "w");
  if (!f) return fail(DPSNN_ERR_IO, "cannot open %s", name);
  std::vector<char> line(256);
  for (uint64_t s = 0; s < c.S; ++s) {
    const float wf = (float)(w[s] * q.factorWeightType_2_Float);
    const int len = std::snprintf(line.data(), line.size(), "%d %d %d %d %d %f %f\n", (int)c.pre[s], (int)c.post[s],
                                  (int)(c.post[s] / c.N), (int)c.delay[s], (int)c.kind[s], wf, td[s]);
    std::fwrite(line.data(), 1, (size_t)len, f);
  }
  std::fclose(f);
  return 0;
}

// The in-list items' weights (both layouts) from the synapses'.
static void refresh_weights(dpsnn_net *n) {
  hipLaunchKernelGGL(k_refresh_weights, dim3(n->stdpBlocks), dim3(kWaveLTP), 0, n->stream, n->dev);
  if (n->winOn) hipLaunchKernelGGL(k_refresh_window, dim3(n->stdpBlocks), dim3(kWaveLTP), 0, n->stream, n->dev);
}

static int commit(dpsnn_net *n, uint32_t t) {
  const dpsnn_parameters &q = n->par.pub;
  const uint32_t sec = t / 1000;
  const bool probes = n->writing && !q.statSynPeriodicProbe_writeDisable && sec >= q.startStatFiles_s &&
                      sec <= q.stopStatFiles_s && sec % q.moduloSec == 0 && sec >= q.startSynPeriodicProbe_s &&
                      sec <= q.stopSynPeriodicProbe_s;
  int rc;
  if (probes && (rc = write_probe(n, "synPeriodicProbe_A", sec, nullptr))) return rc;
  hipLaunchKernelGGL(k_commit, dim3(n->stdpBlocks), dim3(kWaveLTP), 0, n->stream, n->dev);
  refresh_weights(n);
  HIP_TRY(hipGetLastError());
  if (probes && (rc = write_probe(n, "synPeriodicProbe_B", sec, n->dev.tdPre))) return rc;
  return 0;
}

static int prof_begin(dpsnn_net *n) {
  if (!n->profile) return 0;
  if (n->profUsed == n->profEv.size()) {
    hipEvent_t a, b;
    HIP_TRY(hipEventCreate(&a));
    HIP_TRY(hipEventCreate(&b));
    n->profEv.push_back({a, b, 0});
  }
  HIP_TRY(hipEventRecord(n->profEv[n->profUsed].a, n->stream));
  return 0;
}
static int prof_end(dpsnn_net *n, uint32_t steps = 1) {
  if (!n->profile) return 0;
  HIP_TRY(hipEventRecord(n->profEv[n->profUsed].b, n->stream));
  n->profEv[n->profUsed].steps = steps;
  n->profUsed++;
  return 0;
}

// Opens the raster/rates record of ms m (records are contiguous) and returns
// its index in the drain buffers; drains first when they are full.
static int open_record(dpsnn_net *n, uint32_t m, uint32_t *idx) {
  int rc;
  if (n->pendingSteps == n->drainEvery && (rc = drain(n))) return rc;
  if (n->pendingSteps == 0) n->pendingFrom = m;
  *idx = n->pendingSteps++;
  return 0;
}

static int compact(dpsnn_net *n, uint32_t m, uint32_t rec) {
  if (n->wantRaster)
    hipLaunchKernelGGL(k_compact, dim3(1), dim3(kCompactThreads), 0, n->stream, n->dev, m, n->d_rasterIds,
                       n->d_rasterTe, n->d_rasterCount, n->d_stepCount + rec);
  return 0;
}

static bool plastic_at(const dpsnn_net *n, uint32_t t) {
  const dpsnn_parameters &q = n->par.pub;
  return n->stdp && t >= q.startPlasticity_ms && t <= q.stopPlasticity_ms;
}

// Phase 2 of a step with packed records (t >= kPackT): where they hold the
// bath, by three waves per tile while the tiles are few.
static void launch_integrate(const dpsnn_net *n, const DevNet &P, uint32_t t, const ExtView &X, const NextScan &S,
                             hipStream_t stream) {
  const uint32_t blocks = (P.N + kBlock - 1) / kBlock;
  if (!P.bathT)
    hipLaunchKernelGGL(k_integrate<1>, dim3(blocks), dim3(kBlock), 0, stream, P, t, X, S);
  else if (n->pipe)
    hipLaunchKernelGGL(k_integrate_pipe, dim3(P.NW), dim3(kPipeThreads), 0, stream, P, t, S);
  else
    hipLaunchKernelGGL(k_integrate_records, dim3(blocks), dim3(kBlock), 0, stream, P, t, S);
}
// Its bath, ahead of phase 1.
static void launch_bath(const DevNet &P, uint32_t t, const ExtView &X, hipStream_t stream) {
  if (P.bathT) hipLaunchKernelGGL(k_bath, dim3(P.NW), dim3(kWave), 0, stream, P, t, X);
}

// Key scratch of stand-alone steps, blocked by 8 events per neuron:
// [grid][cap/8][64][8] (fused) or [N/64][cap/8][64][8] (split).
static int ensure_scratch(dpsnn_net *n) {
  DevNet &P = n->dev;
  if (P.keys) return 0;
  const size_t slots = n->split ? size_t(P.NW) * kWave : size_t(n->grid) * kWave;
  int rc;
  if ((rc = dev_alloc(n, &P.keys, slots * P.cap)) || (rc = dev_alloc(n, &P.keyW, slots * P.cap)) ||
      (rc = dev_alloc(n, &P.keyCount, slots)))
    return rc;
  if (n->stdp && (rc = dev_alloc(n, &P.keyPos, slots * P.cap))) return rc;
  return 0;
}

// Key scratch of the allocation-free step (dpsnn_step_noalloc): one static
// array per device, held from the library's load on that device until the
// process ends.  Every allocation-free step on a device uses the same
// array, so such steps of two networks that overlap in time on one device
// race on it.  Nothing in it needs to start at zero: each step's phase 1
// writes every count and key its phase 2 reads.
constexpr size_t kStaticScratchBytes = size_t(128) << 20;
static __device__ __align__(256) uint8_t scratch[kStaticScratchBytes];
constexpr int kMaxDevices = 64;
static std::mutex g_scratchMu;
static void *g_scratchPtr[kMaxDevices];

// The device address of `scratch` on the current device (set up once per
// device: the name is a host-side stand-in, not a device address).
static int static_scratch_ptr(int device, uint8_t **out) {
  if (device < 0 || device >= kMaxDevices) return fail(DPSNN_ERR_ARG, "device %d out of range", device);
  std::lock_guard<std::mutex> lock(g_scratchMu);
  if (!g_scratchPtr[device]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(DPSNN_ERR_DEVICE, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
    g_scratchPtr[device] = p;
  }
  *out = (uint8_t *)g_scratchPtr[device];
  return 0;
}

// n's device view with its key scratch carved from the static array, in
// the layout ensure_scratch allocates; refuses networks whose scratch is
// larger than the array.
static int static_scratch_view(dpsnn_net *n, DevNet &P) {
  P = n->dev;
  // the bath stays in phase 2, as the array was sized: a record per in-list item
  P.bathT = nullptr;
  P.cap = round_scratch(n->con.max_in);
  const size_t slots = n->split ? size_t(P.NW) * kWave : size_t(n->grid) * kWave;
  auto al = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t kb = al(slots * P.cap * sizeof(uint64_t)), wb = al(slots * P.cap * sizeof(int16_t)),
               cb = al(slots * sizeof(uint32_t)), pb = n->stdp ? al(slots * P.cap * sizeof(uint16_t)) : 0;
  const size_t need = kb + wb + cb + pb;
  if (need > kStaticScratchBytes)
    return fail(DPSNN_ERR_ARG, "the network's step needs %zu bytes of key scratch; the allocation-free step holds %zu",
                need, kStaticScratchBytes);
  uint8_t *base;
  int rc = static_scratch_ptr(n->opt.device, &base);
  if (rc) return rc;
  P.keys = (uint64_t *)base;
  P.keyW = (int16_t *)(base + kb);
  P.keyCount = (uint32_t *)(base + kb + wb);
  P.keyPos = n->stdp ? (uint16_t *)(base + kb + wb + cb) : nullptr;
  return 0;
}

// What one step of a network needs around its kernel launch.
struct StepPlan {
  uint32_t t = 0;
  int ltd = 0;
  bool commitNow = false, ltpNext = false, recordNext = false;
  uint32_t rec = 0;
  NextScan S{nullptr, 0, 0};
  ExtView X{nullptr, nullptr, nullptr};
  ExtSlot *slot = nullptr;
};

// Host work before step t's kernel: raster/rates records, the replayed
// bath of step t, and the flags of the step.
static int pre_step(dpsnn_net *n, StepPlan &sp) {
  DevNet &P = n->dev;
  const uint32_t t = n->t, next = t + 1;
  const uint32_t T = n->par.pub.totalSimTime_ms;
  const size_t popPer = size_t(P.ncols) * P.nsub;
  int rc;
  sp = StepPlan{};
  sp.t = t;
  if (n->collect && t == 0) {
    uint32_t rec0;
    if ((rc = open_record(n, 0, &rec0)) || (rc = compact(n, 0, rec0))) return rc;
  }
  sp.ltd = plastic_at(n, t) && !n->deferring;
  sp.commitNow = sp.ltd && t % 1000 == 999;
  sp.ltpNext = next < T && plastic_at(n, next) && !n->deferring;
  sp.recordNext = n->collect && next < T;
  sp.S = NextScan{nullptr, sp.ltpNext && !sp.commitNow, next < T};
  if (sp.recordNext) {
    if ((rc = open_record(n, next, &sp.rec))) return rc;
    sp.S.popCnt = n->d_popCnt + popPer * sp.rec;
  }
  if (P.drive == DPSNN_DRIVE_REPLAY) {
    ExtSlot &s = n->ext[n->extNext];
    sp.slot = &s;
    n->extNext = (n->extNext + 1) % kExtRing;
    if (s.pending) HIP_TRY(hipEventSynchronize(s.done));
    n->replay.generate(t, n->extStep);
    const size_t ne = n->extStep.time.size();
    if ((rc = ensure_ext_cap(s, ne))) return rc;
    std::memcpy(s.h_off, n->extStep.off.data(), sizeof(uint32_t) * (P.N + 1));
    if (ne) {
      std::memcpy(s.h_time, n->extStep.time.data(), sizeof(double) * ne);
      std::memcpy(s.h_value, n->extStep.value.data(), sizeof(double) * ne);
    }
    HIP_TRY(hipMemcpyAsync(s.d_off, s.h_off, sizeof(uint32_t) * (P.N + 1), hipMemcpyHostToDevice, n->stream));
    if (ne) {
      HIP_TRY(hipMemcpyAsync(s.d_time, s.h_time, sizeof(double) * ne, hipMemcpyHostToDevice, n->stream));
      HIP_TRY(hipMemcpyAsync(s.d_value, s.h_value, sizeof(double) * ne, hipMemcpyHostToDevice, n->stream));
    }
    sp.X = ExtView{s.d_off, s.d_time, s.d_value};
  }
  return 0;
}

// Host work after step t's kernel: the per-second STDP commit (and the LTP
// of the scan of t+1, which follows it), the raster of t+1.
static int post_step(dpsnn_net *n, StepPlan &sp) {
  int rc;
  const uint32_t next = sp.t + 1;
  if (sp.commitNow) {
    if ((rc = commit(n, sp.t))) return rc;
    if (sp.ltpNext) hipLaunchKernelGGL(k_ltp, dim3(n->stdpBlocks), dim3(kWaveLTP), 0, n->stream, n->dev, next);
  }
  if (sp.recordNext && (rc = compact(n, next, sp.rec))) return rc;
  if (sp.slot) {
    HIP_TRY(hipEventRecord(sp.slot->done, n->stream));
    sp.slot->pending = true;
  }
  HIP_TRY(hipGetLastError());
  n->t = next;
  if (n->opt.keep_spikes) return drain(n);
  return 0;
}

// Step t of one network: delivery + dynamics of t, and the fired scan of
// t+1 (which the reference runs at the head of step t+1; nothing reads the
// scan's outputs in between).  The scan of step 0 finds no spikes.  P is
// the network's device view with the key scratch the kernels use (the
// network's own, or the allocation-free step's static one).
// Whether step sp of n runs phase 1 in the window form: split form, a
// window layout on the device, packed records (t >= kPackT), no LTD.
static bool window_step(const dpsnn_net *n, const StepPlan &sp) {
  return n->split && n->winOn && sp.t >= kPackT && !sp.ltd;
}

// The launches of a window-form step of n on `stream`, with the device view
// P (the network's own, or one whose key scratch is a batch's).
static void launch_window_step(const dpsnn_net *n, const DevNet &P, const StepPlan &sp, hipStream_t stream) {
  const KernelShape &K = kShapes[n->shape];
  launch_bath(P, sp.t, sp.X, stream);
  hipLaunchKernelGGL(k_collect, dim3(n->winGrid), dim3(kCollectThreads), n->winLds, stream, P, sp.t);
  if (!P.fuseSort)
    hipLaunchKernelGGL(K.sort, dim3(n->sortGrid), dim3(kWave), phase1_lds(kSortCap, K.B), stream, P, sp.t);
  hipLaunchKernelGGL(K.sortBig, dim3(n->sortBigGrid), dim3(kWave), phase1_lds(P.cap, K.B), stream, P, sp.t);
  launch_integrate(n, P, sp.t, sp.X, sp.S, stream);
  if (sp.S.ltp) hipLaunchKernelGGL(k_ltp, dim3(n->stdpBlocks), dim3(kWaveLTP), 0, stream, P, sp.t + 1);
}

static int one_step(dpsnn_net *n, const DevNet &P) {
  StepPlan sp;
  int rc;
  if ((rc = pre_step(n, sp)) || (rc = prof_begin(n))) return rc;
  const KernelShape &K = kShapes[n->shape];
  if (window_step(n, sp)) {
    launch_window_step(n, P, sp, n->stream);
  } else if (n->split) {
    if (sp.t >= kPackT) launch_bath(P, sp.t, sp.X, n->stream);
    hipLaunchKernelGGL(K.gather, dim3(n->gatherGrid), dim3(kWave), n->ldsBytes, n->stream, P, sp.t, sp.ltd);
    const uint32_t blocks = (P.N + kBlock - 1) / kBlock;
    if (sp.t >= kPackT)
      launch_integrate(n, P, sp.t, sp.X, sp.S, n->stream);
    else
      hipLaunchKernelGGL(k_integrate<2>, dim3(blocks), dim3(kBlock), 0, n->stream, P, sp.t, sp.X, sp.S);
    if (sp.S.ltp) hipLaunchKernelGGL(k_ltp, dim3(n->stdpBlocks), dim3(kWaveLTP), 0, n->stream, P, sp.t + 1);
  } else {
    hipLaunchKernelGGL(K.step, dim3(n->grid), dim3(kWave), n->ldsBytes, n->stream, P, sp.t, sp.X, sp.ltd, sp.S);
  }
  if ((rc = prof_end(n))) return rc;
  return post_step(n, sp);
}

// ----------------------------------------------------------------------------
// Graph-replayed steps.  kGraphSteps consecutive plain steps are captured
// once into a HIP graph whose kernels take the step's t from the device
// word d_t (set before each replay) and their step's place in the graph, so
// that the same graph replays any run of such steps.  Steps
// qualify when nothing the host does around a step is needed: split form,
// Philox drive, no raster or rates collected, no plasticity, t >= kPackT
// (the packed scratch), and the next step still inside the run.
// ----------------------------------------------------------------------------
constexpr uint32_t kGraphSteps = 10;

static bool graph_run_ok(const dpsnn_net *n, uint32_t steps) {
  const uint32_t t = n->t, T = n->par.pub.totalSimTime_ms;
  if (!n->graphs || !n->split || n->dev.drive != DPSNN_DRIVE_PHILOX || n->collect) return false;
  if (t < kPackT || (uint64_t)t + steps >= T) return false;
  for (uint32_t k = 0; k <= steps; ++k)
    if (plastic_at(n, t + k) && !n->deferring) return false;
  return true;
}

// Steps from n->t on, at most `left`, that may run as one block of k_stdp:
// plastic throughout and at the scan after them, no commit among them, the
// run not over.
static uint32_t stdp_block(const dpsnn_net *n, uint32_t left) {
  const uint32_t t = n->t, T = n->par.pub.totalSimTime_ms;
  if (!n->stdpBlock || t >= T || !plastic_at(n, t)) return 0;
  const uint64_t stop = std::min<uint64_t>(T - 1, n->par.pub.stopPlasticity_ms);  // the last scan
  const uint64_t K = std::min<uint64_t>({left, n->stdpBlock, 999 - t % 1000, stop - std::min<uint64_t>(stop, t)});
  return K >= kStdpBlockMin ? (uint32_t)K : 0;
}

// Opens a block where the next steps (at most `left`) may run as one.
static void stdp_open(dpsnn_net *n, uint32_t left) {
  if (n->deferring || !(n->blockLeft = stdp_block(n, left))) return;
  n->deferring = true;
  n->blockFrom = n->t;
  hipLaunchKernelGGL(k_stdp_begin, dim3((n->dev.N + kWaveLTP - 1) / kWaveLTP), dim3(kWaveLTP), 0, n->stream, n->dev);
}
// After `steps` steps (or a failed one): the open block's updates once it is
// complete, or cut short by the failure.
static int stdp_close(dpsnn_net *n, uint32_t steps, bool failed) {
  if (!n->deferring || ((n->blockLeft -= steps) != 0 && !failed)) return 0;
  n->deferring = false;
  if (n->t > n->blockFrom)
    hipLaunchKernelGGL(k_stdp, dim3(n->stdpBlocks), dim3(kWaveLTP), 0, n->stream, n->dev, n->blockFrom,
                       n->t - n->blockFrom);
  HIP_TRY(hipGetLastError());
  return 0;
}

// Launches of the graph's step k (t from G.tDev).
static void launch_graph_step(dpsnn_net *n, const DevNet &G, uint32_t k) {
  const KernelShape &K = kShapes[n->shape];
  launch_bath(G, k, ExtView{nullptr, nullptr, nullptr}, n->stream);
  if (n->winOn) {
    hipLaunchKernelGGL(k_collect, dim3(n->winGrid), dim3(kCollectThreads), n->winLds, n->stream, G, k);
    if (!G.fuseSort)
      hipLaunchKernelGGL(K.sort, dim3(n->sortGrid), dim3(kWave), phase1_lds(kSortCap, K.B), n->stream, G, k);
    hipLaunchKernelGGL(K.sortBig, dim3(n->sortBigGrid), dim3(kWave), phase1_lds(G.cap, K.B), n->stream, G, k);
  } else {
    hipLaunchKernelGGL(K.gather, dim3(n->gatherGrid), dim3(kWave), n->ldsBytes, n->stream, G, k, 0);
  }
  launch_integrate(n, G, k, ExtView{nullptr, nullptr, nullptr}, NextScan{nullptr, 0, 1}, n->stream);
}

static int capture_step_graph(dpsnn_net *n, const DevNet &P) {
  if (n->stepGraph) {
    HIP_TRY(hipGraphExecDestroy(n->stepGraph));
    n->stepGraph = nullptr;
  }
  if (!n->d_t) {
    int rc = dev_alloc(n, &n->d_t, 1);
    if (rc) return rc;
  }
  DevNet G = P;
  G.tDev = n->d_t;
  hipGraph_t g = nullptr;
  HIP_TRY(hipStreamBeginCapture(n->stream, hipStreamCaptureModeThreadLocal));
  for (uint32_t k = 0; k < kGraphSteps; ++k) launch_graph_step(n, G, k);
  const hipError_t e = hipStreamEndCapture(n->stream, &g);
  if (e != hipSuccess) return fail(DPSNN_ERR_DEVICE, "graph capture of the step failed: %s", hipGetErrorString(e));
  const hipError_t ei = hipGraphInstantiate(&n->stepGraph, g, nullptr, nullptr, 0);
  hipGraphDestroy(g);
  if (ei != hipSuccess) {
    n->stepGraph = nullptr;
    return fail(DPSNN_ERR_DEVICE, "graph instantiation failed: %s", hipGetErrorString(ei));
  }
  n->graphKeys = P.keys;
  return 0;
}

// kGraphSteps steps from n->t by one graph replay.
static int graph_steps(dpsnn_net *n, const DevNet &P) {
  int rc;
  if ((!n->stepGraph || n->graphKeys != P.keys) && (rc = capture_step_graph(n, P))) return rc;
  hipLaunchKernelGGL(k_set_t, dim3(1), dim3(1), 0, n->stream, n->d_t, n->t);
  if ((rc = prof_begin(n))) return rc;
  HIP_TRY(hipGraphLaunch(n->stepGraph, n->stream));
  if ((rc = prof_end(n, kGraphSteps))) return rc;
  HIP_TRY(hipGetLastError());
  n->t += kGraphSteps;
  n->graphSteps += kGraphSteps;
  return 0;
}

// Up to nsteps steps with the device view P (graph replays where the steps
// qualify and `graphs` allows them).
static int run_steps(dpsnn_net *n, const DevNet &P, uint32_t nsteps, bool graphs) {
  int rc;
  for (uint32_t k = 0; k < nsteps;) {
    if (n->t >= n->par.pub.totalSimTime_ms) {
      rc = drain(n);
      return rc ? rc : DPSNN_DONE;
    }
    stdp_open(n, nsteps - k);
    const uint32_t left = n->deferring ? n->blockLeft : nsteps - k;
    const uint32_t steps = graphs && left >= kGraphSteps && graph_run_ok(n, kGraphSteps) ? kGraphSteps : 1;
    rc = steps > 1 ? graph_steps(n, P) : one_step(n, P);
    k += steps;
    const int rc2 = stdp_close(n, rc ? 0 : steps, rc != 0);
    if (rc || rc2) return rc ? rc : rc2;
  }
  return 0;
}

// ============================================================================
// C ABI
// ============================================================================
// --------------------------------------------------------------------------
// Device connectome generator (dpsnn_options.generator = device): the
// distributions of the reference's generator (generate_column;
// DPSNN_LIFCAcorticalModuleGen.cpp:62-220, DPSNN_LIFCAconnectome.cpp:
// 1079-1133) drawn from Philox4x32-10, one thread per source neuron, instead
// of the sequential ran3 stream: for each target sub-population and stencil
// cell with connection probability q, targets at geometric gaps over the
// cell's column (smallest n >= 1 with 1 - (1 - q)^n >= r, at most span + 1,
// as the reference's linear search), then per target a uniform delay
// (uniform_delay's level arithmetic) and a truncated Gaussian weight (the
// reference's rejection bounds), int16-quantised.  Pass 0 counts each
// source's synapses, pass 1 writes them at their offsets in generation
// order; the host then sorts them into the backward list as for the
// reference's.  Statistically equivalent, not bit-exact.
// --------------------------------------------------------------------------
struct GenView {
  uint32_t N, npc, CFX, CFY, nsub, sx, sy, mdx, mdy, overall, D;
  float f2w, minW, delayLo, delayHi;
  uint64_t seed;
  const float *prob;                 // [nsub][nsub][sx][sy]
  const float *J, *DJ, *DMin, *DMax;  // [nsub][nsub], source-major
  const uint32_t *subOff, *subCnt;   // [nsub], within a column
  uint32_t *count;
  const uint64_t *off;
  uint32_t *post;
  uint8_t *delay;
  int16_t *w;
  uint32_t *error;                   // bit 0: q in (0, 1e-5]; 1: 7500 or more
                                     // synapses; 2: weight bound; 3: delay >= env_D;
                                     // 4: no weight within the draw bounds
};

__device__ inline uint32_t gen_round_half_up(double r) {
  const double f = floor(r);
  return (f + 0.5 > r) ? (uint32_t)f : (uint32_t)(f + 1.0);
}

template <int PASS>
__global__ __launch_bounds__(256) void k_generate(GenView G) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= G.N) return;
  const uint32_t col = i / G.npc, inCM = i - col * G.npc, cfx = col % G.CFX, cfy = col / G.CFX;
  uint32_t src = 0;
  for (uint32_t s = 0; s < G.nsub; ++s)
    if (inCM >= G.subOff[s] && inCM < G.subOff[s] + G.subCnt[s]) src = s;
  PhiloxStream A{(uint32_t)G.seed, (uint32_t)(G.seed >> 32) ^ i, 0ull, 0.0, 0};
  PhiloxStream Bw{(uint32_t)G.seed ^ 0x5bd1e995u, (uint32_t)(G.seed >> 32) ^ i, 0ull, 0.0, 0};
  const uint64_t at0 = PASS ? G.off[i] : 0ull;
  uint32_t n = 0, err = 0;
  for (uint32_t ts = 0; ts < G.nsub; ++ts)
    for (uint32_t x = 0; x < G.sx; ++x)
      for (uint32_t y = 0; y < G.sy; ++y) {
        int32_t tx, ty;
        if (G.overall == 0) {
          tx = (int32_t)cfx + (int32_t)x - (int32_t)G.mdx;
          ty = (int32_t)cfy + (int32_t)y - (int32_t)G.mdy;
        } else {
          tx = (int32_t)x;
          ty = (int32_t)y;
        }
        if (tx < 0 || tx >= (int32_t)G.CFX || ty < 0 || ty >= (int32_t)G.CFY) continue;
        const float q = G.prob[((src * G.nsub + ts) * G.sx + x) * G.sy + y];
        if (!(q > 0.0f)) continue;
        if (!(q > 0.00001f)) {
          err |= 1u;
          continue;
        }
        const uint32_t first = G.subOff[ts], end = first + G.subCnt[ts];
        const uint32_t colBase = (uint32_t)tx * G.npc + (uint32_t)ty * G.npc * G.CFX;
        uint32_t cur = first - 1;  // wraps as the reference's uint32 arithmetic
        const uint32_t span = end - cur;
        const double lq = log1p(-(double)q);
        const float mean = G.J[src * G.nsub + ts], sigma = G.DJ[src * G.nsub + ts] * mean;
        for (;;) {
          const double r = A.next();
          double g = q >= 1.0f ? 1.0 : ceil(log1p(-r) / lq);
          g = fmin(fmax(g, 1.0), (double)span + 1.0);
          cur += (uint32_t)g;
          if (cur >= end) break;
          if (n + 1 >= kMaxOutDegree) {
            err |= 2u;
            break;
          }
          if (PASS) {
            // delay: uniform_delay's levels
            float DMin = G.DMin[src * G.nsub + ts], DMax = G.DMax[src * G.nsub + ts];
            float lo = G.delayLo, hi = G.delayHi;
            const float step = (hi - lo) / (float)kDelaySlots;
            hi -= step / 2;
            lo += step / 2;
            DMax = gen_round_half_up((DMax - lo) / step) * step + lo;
            DMin = gen_round_half_up((DMin - lo) / step) * step + lo;
            const float level = (float)((Bw.next() * (DMax - DMin) + DMin - lo) / step);
            const uint32_t d = gen_round_half_up(level * step);
            // weight: Gaussian (Box-Muller) within the reference's bounds
            // (at most 64 draws: a bound the draws cannot meet, such as a
            // zero mean, is reported instead of looping)
            float wv = mean;
            bool inBounds = false;
            for (int tries = 0; tries < 64 && !inBounds; ++tries) {
              const double u1 = 1.0 - Bw.next(), u2 = Bw.next();
              const double z = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
              wv = (float)(mean + z * sigma);
              inBounds = mean > 0.0f ? !(wv < 0.0f || wv >= 2.0f * mean) : !(wv <= 2.0f * mean || wv > 0.0f);
            }
            if (!inBounds) err |= 16u;
            if (wv < G.minW || wv > -G.minW) err |= 4u;
            if (d >= kDelaySlots || d >= G.D) err |= 8u;
            G.post[at0 + n] = colBase + cur;
            G.delay[at0 + n] = (uint8_t)min(d, kDelaySlots - 1);
            G.w[at0 + n] = (int16_t)(wv * G.f2w);
          }
          ++n;
        }
      }
  if (!PASS) G.count[i] = n;
  if (err) atomicOr(G.error, err);
}

// The connectome of n drawn on its device (k_generate), then sorted into the
// backward list on the host.
static int generate_on_device(dpsnn_net *n, std::string &err) {
  const Params &p = n->par;
  const dpsnn_parameters &q = p.pub;
  Connectome &c = n->con;
  connectome_neurons(p, c);
  const uint32_t N = c.N, npc = q.neuronsPerCM, nsub = q.subPopNumber;
  for (uint32_t i = 0; i < N; ++i) {
    const uint32_t inCM = i % npc;
    uint32_t src = 0;
    for (uint32_t s = 0; s < nsub; ++s)
      if (inCM >= p.sp[s].offset && inCM < p.sp[s].offset + p.sp[s].count) src = s;
    c.subPop[i] = (uint8_t)src;
    neuron_bath(p, i, src, c);
  }
  std::vector<float> prob(size_t(nsub) * nsub * p.stencilX * p.stencilY), J(nsub * nsub), DJ(nsub * nsub),
      DMin(nsub * nsub), DMax(nsub * nsub);
  std::vector<uint32_t> off(nsub), cnt(nsub);
  for (uint32_t s = 0; s < nsub; ++s) {
    off[s] = p.sp[s].offset;
    cnt[s] = p.sp[s].count;
    for (uint32_t t = 0; t < nsub; ++t) {
      J[s * nsub + t] = (float)p.sp[s].J[t];
      DJ[s * nsub + t] = (float)p.sp[s].DJ[t];
      DMin[s * nsub + t] = (float)p.sp[s].DMin[t];
      DMax[s * nsub + t] = (float)p.sp[s].DMax[t];
      for (uint32_t x = 0; x < p.stencilX; ++x)
        for (uint32_t y = 0; y < p.stencilY; ++y)
          prob[((s * nsub + t) * p.stencilX + x) * p.stencilY + y] = p.prob_at(s, t, x, y);
    }
  }
  HIP_TRY(hipSetDevice(n->opt.device));
  hipStream_t st;
  HIP_TRY(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  std::vector<void *> bufs;
  auto fin = [&](int rc) {
    (void)hipStreamSynchronize(st);
    for (void *b : bufs) (void)hipFree(b);
    (void)hipStreamDestroy(st);
    return rc;
  };
  auto alloc = [&](void **ptr, size_t bytes) -> bool {
    if (hipMalloc(ptr, bytes ? bytes : 1) != hipSuccess) return false;
    bufs.push_back(*ptr);
    return true;
  };
  auto put = [&](void **ptr, const void *src, size_t bytes) -> bool {
    return alloc(ptr, bytes) && hipMemcpyAsync(*ptr, src, bytes, hipMemcpyHostToDevice, st) == hipSuccess;
  };
  GenView G{};
  G.N = N; G.npc = npc; G.CFX = q.globCFX; G.CFY = q.globCFY; G.nsub = nsub;
  G.sx = p.stencilX; G.sy = p.stencilY; G.mdx = p.maxModDeltaX; G.mdy = p.maxModDeltaY;
  G.overall = q.overallConnectivity; G.D = q.D;
  G.f2w = q.factorFloat_2_weightType; G.minW = q.minSynWeight_f;
  G.delayLo = (float)q.delayMin; G.delayHi = (float)q.delayMax;
  G.seed = n->opt.generator_seed;
  void *dProb, *dJ, *dDJ, *dDMin, *dDMax, *dOff, *dCnt, *dCount, *dErr;
  if (!put(&dProb, prob.data(), 4 * prob.size()) || !put(&dJ, J.data(), 4 * J.size()) ||
      !put(&dDJ, DJ.data(), 4 * DJ.size()) || !put(&dDMin, DMin.data(), 4 * DMin.size()) ||
      !put(&dDMax, DMax.data(), 4 * DMax.size()) || !put(&dOff, off.data(), 4 * nsub) ||
      !put(&dCnt, cnt.data(), 4 * nsub) || !alloc(&dCount, 4 * (size_t)N) || !alloc(&dErr, 4))
    return fin(fail(DPSNN_ERR_MEMORY, "device generator: out of device memory"));
  G.prob = (const float *)dProb; G.J = (const float *)dJ; G.DJ = (const float *)dDJ;
  G.DMin = (const float *)dDMin; G.DMax = (const float *)dDMax;
  G.subOff = (const uint32_t *)dOff; G.subCnt = (const uint32_t *)dCnt;
  G.count = (uint32_t *)dCount; G.error = (uint32_t *)dErr;
  if (hipMemsetAsync(G.error, 0, 4, st) != hipSuccess) return fin(fail(DPSNN_ERR_DEVICE, "device generator: memset failed"));
  const dim3 grid((N + 255) / 256);
  hipLaunchKernelGGL(k_generate<0>, grid, dim3(256), 0, st, G);
  if (hipGetLastError() != hipSuccess) return fin(fail(DPSNN_ERR_DEVICE, "device generator: launch failed"));
  std::vector<uint32_t> counts(N);
  uint32_t errBits = 0;
  if (hipMemcpyAsync(counts.data(), dCount, 4 * (size_t)N, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipMemcpyAsync(&errBits, dErr, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return fin(fail(DPSNN_ERR_DEVICE, "device generator: count pass failed"));
  std::vector<uint64_t> gen_off(N + 1, 0);
  for (uint32_t i = 0; i < N; ++i) gen_off[i + 1] = gen_off[i] + counts[i];
  const uint64_t S = gen_off[N];
  void *dGenOff, *dPost, *dDelay, *dW;
  if (!put(&dGenOff, gen_off.data(), 8 * (size_t)N) || !alloc(&dPost, 4 * S) || !alloc(&dDelay, S) ||
      !alloc(&dW, 2 * S))
    return fin(fail(DPSNN_ERR_MEMORY, "device generator: out of device memory for %llu synapses",
                    (unsigned long long)S));
  G.off = (const uint64_t *)dGenOff; G.post = (uint32_t *)dPost; G.delay = (uint8_t *)dDelay; G.w = (int16_t *)dW;
  hipLaunchKernelGGL(k_generate<1>, grid, dim3(256), 0, st, G);
  if (hipGetLastError() != hipSuccess) return fin(fail(DPSNN_ERR_DEVICE, "device generator: launch failed"));
  std::vector<uint32_t> g_post(S);
  std::vector<uint8_t> g_delay(S);
  std::vector<int16_t> g_w(S);
  if (hipMemcpyAsync(g_post.data(), dPost, 4 * S, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipMemcpyAsync(g_delay.data(), dDelay, S, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipMemcpyAsync(g_w.data(), dW, 2 * S, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipMemcpyAsync(&errBits, dErr, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return fin(fail(DPSNN_ERR_DEVICE, "device generator: fill pass failed"));
  fin(0);
  if (errBits & 1u) { err = "connection probabilities in (0, 1e-5] are not supported"; return DPSNN_ERR_CONFIG; }
  if (errBits & 2u) { err = "a neuron would get 7500 or more synapses (DSD__maxM)"; return DPSNN_ERR_CONFIG; }
  if (errBits & 4u) { err = "synaptic weight outside [env_minSynWeight_f, -env_minSynWeight_f]"; return DPSNN_ERR_CONFIG; }
  if (errBits & 8u) { err = "a stored delay is not below env_D"; return DPSNN_ERR_CONFIG; }
  if (errBits & 16u) { err = "synaptic weights cannot be drawn within their bounds (zero mean?)"; return DPSNN_ERR_CONFIG; }
  inflate_backward(c, gen_off, g_post, g_delay, g_w, n->opt.host_threads);
  return 0;
}

extern "C" {

const char *dpsnn_last_error(void) { return g_err.c_str(); }

int dpsnn_get_parameters(const char *inidir, dpsnn_parameters *out) {
  if (!inidir || !out) return fail(DPSNN_ERR_ARG, "null argument");
  Params p;
  std::string err;
  if (!read_params(inidir, p, err)) return fail(DPSNN_ERR_CONFIG, "%s", err.c_str());
  *out = p.pub;
  return 0;
}

int dpsnn_write_ini_files(const char *inidir, const char *outdir, const char *env) {
  if (!inidir || !outdir) return fail(DPSNN_ERR_ARG, "null argument");
  Params p;
  std::string err;
  EnvMap over;
  if (env && !parse_env_overrides(env, over, err)) return fail(DPSNN_ERR_ARG, "%s", err.c_str());
  if (!read_params(inidir, p, err, env ? &over : nullptr)) return fail(DPSNN_ERR_CONFIG, "%s", err.c_str());
  if (!write_ini_files(p, outdir, err)) return fail(DPSNN_ERR_IO, "%s", err.c_str());
  return 0;
}

int dpsnn_prepare(const char *inidir, const dpsnn_options *opt, dpsnn_net **out) {
  if (!inidir || !out) return fail(DPSNN_ERR_ARG, "null argument");
  *out = nullptr;
  auto t0 = std::chrono::steady_clock::now();
  std::unique_ptr<dpsnn_net> n(new dpsnn_net());
  if (opt) n->opt = *opt;
  if (n->opt.drive != DPSNN_DRIVE_REPLAY && n->opt.drive != DPSNN_DRIVE_PHILOX)
    return fail(DPSNN_ERR_ARG, "unknown drive mode %d", n->opt.drive);
  std::string err;
  EnvMap over;
  if (!parse_env_overrides(n->opt.env, over, err) || !read_params(inidir, n->par, err, &over))
    return fail(DPSNN_ERR_CONFIG, "%s", err.c_str());
  n->opt.env = nullptr;  // not kept past the call
  if (n->opt.output_dir) {
    n->outDir = n->opt.output_dir;
    n->opt.output_dir = n->outDir.c_str();
  }
  const dpsnn_parameters &q = n->par.pub;
  n->stdp = q.startPlasticity_ms <= q.stopPlasticity_ms && q.startPlasticity_ms < q.totalSimTime_ms;
  if (n->stdp)
    for (uint32_t s = 0; s < q.subPopNumber; ++s)
      if (!(n->par.sp[s].Tarp >= 1.0))
        // a source could then fire in consecutive steps and one synapse be
        // delivered twice in a step (own bucket + spill-over run)
        return fail(DPSNN_ERR_CONFIG, "STDP on device needs refractory periods >= 1 ms");
  // localNet init: seed with env_globalSeed (DPSNN_localNet_init.c:119),
  // generate, then continue the stream from SetRandomSeed(loc_h=0) (:283)
  n->rng.seed((int32_t)q.globalSeed);
  if (n->opt.generator == DPSNN_GENERATOR_DEVICE) {
    const int grc = generate_on_device(n.get(), err);
    if (grc) return grc == DPSNN_ERR_CONFIG ? fail(DPSNN_ERR_CONFIG, "%s", err.c_str()) : grc;
  } else if (n->opt.generator != DPSNN_GENERATOR_HOST) {
    return fail(DPSNN_ERR_ARG, "unknown generator %u", n->opt.generator);
  } else if (!generate_connectome(n->par, n->rng, n->con, err, n->opt.host_threads)) {
    return fail(DPSNN_ERR_CONFIG, "%s", err.c_str());
  }
  build_delivery(n->par, n->con, /*with_incoming=*/n->stdp, n->opt.host_threads);
  n->rng.seed(0);
  // DPSNN_REPLAY_STREAM=k > 0: the replayed bath continues from
  // SetRandomSeed(k) instead, the stream process loc_h = k would draw --
  // the reference's own drive with another stream, to measure its
  // run-to-run spread; unset or 0 is the reference's stream
  if (const char *e = std::getenv("DPSNN_REPLAY_STREAM"))
    if (const int k = std::atoi(e)) n->rng.seed(k);
  if (n->stdp) {
    // each in-list item names its synapse by its rank in the target's
    // incoming list (backward-list order)
    const Connectome &c = n->con;
    std::vector<uint32_t> rank(c.S);
    for (uint32_t j = 0; j < c.N; ++j) {
      if (c.inc_off[j + 1] - c.inc_off[j] > 65535)
        return fail(DPSNN_ERR_CONFIG, "neuron %u has more than 65535 incoming synapses", j);
      for (uint64_t k = c.inc_off[j]; k < c.inc_off[j + 1]; ++k) rank[c.inc_syn[k]] = (uint32_t)(k - c.inc_off[j]);
    }
    n->inSynLocal.resize(c.in_off[c.N]);
    for (uint64_t it = 0; it < c.in_off[c.N]; ++it) n->inSynLocal[it] = (uint16_t)rank[c.in_syn[it]];
  }
  if (n->con.max_in >= kMaxInList)
    return fail(DPSNN_ERR_CONFIG, "a neuron has %u in-list items; the engine handles up to %u", n->con.max_in,
                kMaxInList - 1);
  // stencil-window phase 1: on for large networks; DPSNN_WINDOW=1 forces
  // it on (tests of small networks), 0 off.  A connectome whose stencil
  // window does not fit the LDS keeps the gather form.
  {
    bool want = n->con.N >= kWindowMinNeurons;
    if (const char *e = std::getenv("DPSNN_WINDOW")) want = std::atoi(e) != 0;
    if (want) {
      // DPSNN_WINDOW_UNITS: units wanted per step instead (tuning; results do
      // not change)
      const char *ue = getenv("DPSNN_WINDOW_UNITS");
      const uint32_t unitsPerCol = ue && atoi(ue) > 0
                                       ? std::max<uint32_t>(1, ((uint32_t)atoi(ue) + q.globCFT - 1) / q.globCFT)
                                       : window_units_per_col(q.neuronsPerCM, std::max(q.globCFT, 1u));
      build_window(n->par, n->con, unitsPerCol, kWindowMaxEntries, n->window, n->opt.host_threads,
                   /*fill=*/false);
    }
  }
  if (n->opt.drive == DPSNN_DRIVE_REPLAY) n->replay.init(n->con, &n->rng);
  n->writing = n->opt.output_dir && n->opt.output_dir[0];
  if (n->opt.drop_host_synapses && n->stdp && n->writing && !q.statSynPeriodicProbe_writeDisable)
    return fail(DPSNN_ERR_CONFIG, "synPeriodicProbe files need the host synapse list (drop_host_synapses is set)");
  if (n->writing && !n->writer.init(n->par, n->opt.output_dir))
    return fail(DPSNN_ERR_IO, "cannot write output files in %s", n->opt.output_dir);
  n->stdpEvents = n->writing && n->stdp && !n->par.stdpEventDisable;
  if (n->stdpEvents) {
    if (n->opt.drop_host_synapses)
      return fail(DPSNN_ERR_CONFIG, "the STDPevent file needs the host synapse list (drop_host_synapses is set)");
    if (!n->stdpWriter.init(n->par, n->con, n->opt.output_dir))
      return fail(DPSNN_ERR_CONFIG, "cannot set up the STDPevent writer");
  }
  n->initSeconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  *out = n.release();
  return 0;
}

uint64_t dpsnn_device_bytes_needed(const dpsnn_net *n) {
  if (!n) return 0;
  if (n->uploaded) return n->devBytes;
  const Connectome &c = n->con;
  const dpsnn_parameters &q = n->par.pub;
  const uint64_t N = c.N, NW = (N + 63) / 64, items = c.in_off.empty() ? 0 : c.in_off[N];
  uint64_t RS = 1;
  while (RS < c.max_delay + 2) RS <<= 1;
  auto r = [](uint64_t b) { return (std::max<uint64_t>(b, 1) + 255) / 256 * 256; };
  uint64_t b = r(8 * q.subPopNumber * kParams) + r(8 * c.bathLut.size()) + r(8 * N) + r(N) + r(4 * N);
  b += 5 * r(8 * N) + r(8 * N);                                // state, Philox counters
  b += r(8 * RS * NW) + r(8 * RS * N);                         // spike history
  b += r(8 * (N + 1)) + r(4 * (items + kWave)) + r(2 * items);  // in-lists
  if (const uint64_t cap = bath_cap(n)) b += r(4 * q.subPopNumber) + r(8 * cap * N) + r(4 * N);
  if (n->stdp) {
    const uint64_t S = c.S;
    b += r(8 * (N + 1)) + r(2 * S) + r(S) + r(2 * items) + 2 * r(4 * S) + 3 * r(4 * N);
    if (!q.statSynPeriodicProbe_writeDisable) b += r(4 * S);
    b += 2 * r(4 * kStdpSpan) + 2 * r(4 * q.subPopNumber * q.subPopNumber);
  }
  const uint64_t drainEvery = n->opt.drain_every_ms ? n->opt.drain_every_ms : 100;
  b += r(8 * kCounterSlots * kCounterStride) + r(4 * kXcds * kCtrStride) + r(4 * (uint64_t)q.globCFT * q.subPopNumber * drainEvery);
  const bool raster = (n->writing && !q.spikes_writeDisable) || n->opt.keep_spikes;
  if (raster) {
    const uint64_t cap = N * std::min<uint64_t>(drainEvery, 1000) + 1;
    b += r(4 * cap) + r(8 * cap) + r(4) + r(4 * drainEvery);
  }
  if (n->opt.drive == DPSNN_DRIVE_REPLAY) b += kExtRing * r(4 * (N + 1));
  const WindowLayout &L = n->window;
  if (L.ok)
    b += r(4 * L.items()) + r(2 * L.chunks()) + r(8 * L.chunk.size()) + r(4 * L.cols.size()) +
         r(4 * kXcds * kCtrStride) + r(4 * N) + r(4);
  return b;
}

uint64_t dpsnn_host_bytes(const dpsnn_net *n) {
  if (!n) return 0;
  auto v = [](const auto &x) { return uint64_t(x.capacity()) * sizeof(x[0]); };
  const Connectome &c = n->con;
  const WindowLayout &L = n->window;
  return v(c.pre) + v(c.post) + v(c.delay) + v(c.kind) + v(c.weight) + v(c.in_off) + v(c.in_pre_d) + v(c.in_w) +
         v(c.in_syn) + v(c.inc_off) + v(c.inc_syn) + v(n->inSynLocal) + v(L.cols) + v(L.item) + v(L.desc) +
         v(L.chunk);
}

int dpsnn_upload(dpsnn_net *n) {
  if (!n) return fail(DPSNN_ERR_ARG, "null network");
  if (n->uploaded) return 0;
  auto t0 = std::chrono::steady_clock::now();
  HIP_TRY(hipSetDevice(n->opt.device));
  HIP_TRY(hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking));
  n->ownStream = n->stream;
  int rc = build_device(n);
  if (rc) {
    free_all(n);
    return rc;
  }
  n->uploaded = true;
  // the device holds the in-lists; the host keeps the backward list for
  // dumps (unless asked not to) and drops the delivery staging
  std::vector<uint32_t>().swap(n->con.in_pre_d);
  std::vector<int16_t>().swap(n->con.in_w);
  std::vector<uint32_t>().swap(n->con.in_syn);
  std::vector<uint16_t>().swap(n->inSynLocal);
  n->window = WindowLayout{};
  if (n->opt.drop_host_synapses) {
    std::vector<uint32_t>().swap(n->con.pre);
    std::vector<uint32_t>().swap(n->con.post);
    std::vector<uint8_t>().swap(n->con.delay);
    std::vector<uint8_t>().swap(n->con.kind);
    std::vector<int16_t>().swap(n->con.weight);
    std::vector<uint64_t>().swap(n->con.inc_off);
    std::vector<uint32_t>().swap(n->con.inc_syn);
  }
  n->initSeconds += std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return 0;
}

int dpsnn_create(const char *inidir, const dpsnn_options *opt, dpsnn_net **out) {
  if (!out) return fail(DPSNN_ERR_ARG, "null argument");
  dpsnn_net *n = nullptr;
  int rc = dpsnn_prepare(inidir, opt, &n);
  if (rc) return rc;
  if ((rc = dpsnn_upload(n))) {
    std::string keep = g_err;
    dpsnn_destroy(n);
    g_err = keep;
    return rc;
  }
  *out = n;
  return 0;
}

int dpsnn_step(dpsnn_net *n, uint32_t nsteps) {
  if (!n) return fail(DPSNN_ERR_ARG, "null network");
  if (n->batch) return fail(DPSNN_ERR_ARG, "network is a member of a batch: step it through dpsnn_batch_step");
  if (!n->uploaded) return fail(DPSNN_ERR_ARG, "network not uploaded (dpsnn_upload)");
  HIP_TRY(hipSetDevice(n->opt.device));
  int rc0 = ensure_scratch(n);
  if (rc0) return rc0;
  return run_steps(n, n->dev, nsteps, true);
}

int dpsnn_step_noalloc(dpsnn_net *n, uint32_t nsteps) {
  if (!n) return fail(DPSNN_ERR_ARG, "null network");
  if (n->batch) return fail(DPSNN_ERR_ARG, "network is a member of a batch: step it through dpsnn_batch_step");
  if (!n->uploaded) return fail(DPSNN_ERR_ARG, "network not uploaded (dpsnn_upload)");
  if (n->dev.drive == DPSNN_DRIVE_REPLAY)
    // the replayed bath's staging buffers grow with the step's event count
    return fail(DPSNN_ERR_ARG, "the allocation-free step runs the Philox drive only");
  HIP_TRY(hipSetDevice(n->opt.device));
  DevNet P;
  int rc = static_scratch_view(n, P);
  if (rc) return rc;
  // graph instantiation allocates: plain launches only
  return run_steps(n, P, nsteps, false);
}

int dpsnn_sync(dpsnn_net *n) {
  if (!n) return fail(DPSNN_ERR_ARG, "null network");
  HIP_TRY(hipStreamSynchronize(n->stream));
  return drain(n);
}

uint32_t dpsnn_now_ms(const dpsnn_net *n) { return n ? n->t : 0; }
uint32_t dpsnn_total_ms(const dpsnn_net *n) { return n ? n->par.pub.totalSimTime_ms : 0; }

// Up to this many neurons one kernel writes the state to pinned memory: five
// copies into pageable memory took 30 us each whatever their size.  A step and
// its read-backs: one column 206 -> 143 us, 2x2 with its spikes 351 -> 259.
// Above, a ms takes 400 us and more; the line bounds the pinned memory of a
// network (4.3 MB).
static constexpr size_t kStateDirect = size_t(1) << 17;

int dpsnn_get_state(dpsnn_net *n, double *v, double *c, double *Tr, double *Te, uint8_t *fired) {
  if (!n) return fail(DPSNN_ERR_ARG, "null network");
  const size_t N = n->dev.N;
  if (n->uploaded && N <= kStateDirect) {
    std::lock_guard<std::mutex> lk(n->readMu);
    HIP_TRY(hipSetDevice(n->opt.device));
    if (!n->h_state) HIP_TRY(hipHostMalloc((void **)&n->h_state, N * 33 + 8, 0));
    hipLaunchKernelGGL(k_read_state, dim3((uint32_t)((N + kBlock - 1) / kBlock)), dim3(kBlock), 0, n->stream, n->dev,
                       n->t, n->h_state);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(n->stream));
    double *to[4] = {v, c, Tr, Te};
    for (int i = 0; i < 4; ++i)
      if (to[i]) std::memcpy(to[i], n->h_state + N * (size_t)i, N * 8);
    if (fired) std::memcpy(fired, n->h_state + 4 * N, N);
    return 0;
  }
  HIP_TRY(hipStreamSynchronize(n->stream));
  if (v) HIP_TRY(hipMemcpy(v, n->dev.v, N * 8, hipMemcpyDeviceToHost));
  if (c) HIP_TRY(hipMemcpy(c, n->dev.c, N * 8, hipMemcpyDeviceToHost));
  if (Tr) HIP_TRY(hipMemcpy(Tr, n->dev.Tr, N * 8, hipMemcpyDeviceToHost));
  if (Te) HIP_TRY(hipMemcpy(Te, n->dev.Te, N * 8, hipMemcpyDeviceToHost));
  if (fired) {
    // neurons that fired in the last completed step: bitmap of slot t
    std::vector<uint64_t> w(n->dev.NW);
    const size_t slot = n->t & (n->dev.RS - 1);
    HIP_TRY(hipMemcpy(w.data(), n->dev.bits + slot * n->dev.NW, 8 * w.size(), hipMemcpyDeviceToHost));
    for (size_t i = 0; i < N; ++i) fired[i] = (uint8_t)((w[i >> 6] >> (i & 63)) & 1u);
  }
  return 0;
}

int dpsnn_last_spikes(dpsnn_net *n, uint32_t *ids, double *te, uint32_t *count) {
  if (!n) return fail(DPSNN_ERR_ARG, "null network");
  if (!n->opt.keep_spikes) return fail(DPSNN_ERR_ARG, "network created without keep_spikes");
  int rc = dpsnn_sync(n);
  if (rc) return rc;
  const uint32_t cnt = (uint32_t)n->lastIds.size();
  if (count) *count = cnt;
  if (ids) std::memcpy(ids, n->lastIds.data(), sizeof(uint32_t) * cnt);
  if (te) std::memcpy(te, n->lastTe.data(), sizeof(double) * cnt);
  return 0;
}

uint64_t dpsnn_num_synapses(const dpsnn_net *n) { return n ? n->con.S : 0; }

int dpsnn_get_synapses(dpsnn_net *n, uint32_t *pre, uint32_t *post, uint8_t *delay, int16_t *weight,
                       float *tderiv, int32_t *last_act) {
  if (!n) return fail(DPSNN_ERR_ARG, "null network");
  if (n->opt.drop_host_synapses) return fail(DPSNN_ERR_ARG, "the host synapse list was dropped (drop_host_synapses)");
  const Connectome &c = n->con;
  if (pre) std::memcpy(pre, c.pre.data(), 4 * c.S);
  if (post) std::memcpy(post, c.post.data(), 4 * c.S);
  if (delay) std::memcpy(delay, c.delay.data(), c.S);
  if (n->stdp) return synapse_state(n, weight, tderiv, last_act);
  if (weight) std::memcpy(weight, c.weight.data(), 2 * c.S);
  if (tderiv) std::memset(tderiv, 0, 4 * c.S);
  if (last_act) std::memset(last_act, 0, 4 * c.S);
  return 0;
}

int dpsnn_write_synapse_dump(dpsnn_net *n, const char *path);
int dpsnn_get_stats(dpsnn_net *n, dpsnn_stats *out) {
  if (!n || !out) return fail(DPSNN_ERR_ARG, "null argument");
  if (!n->uploaded) return fail(DPSNN_ERR_ARG, "network not uploaded (dpsnn_upload)");
  std::lock_guard<std::mutex> lk(n->readMu);
  HIP_TRY(hipSetDevice(n->opt.device));
  if (!n->h_counters) HIP_TRY(hipHostMalloc((void **)&n->h_counters, kReadCounters * sizeof(unsigned long long), 0));
  hipLaunchKernelGGL(k_read_counters, dim3(1), dim3(kReadCounters), 0, n->stream, n->dev.counters, n->h_counters);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(n->stream));
  const unsigned long long *cnt = n->h_counters;
  out->steps = n->t;
  out->synaptic_events = cnt[0];
  out->external_events = cnt[1];
  out->spikes = cnt[2];
  out->synapses = n->con.S;
  out->delivery_items = n->items;
  out->neurons = n->con.N;
  out->max_in_items = n->con.max_in;
  out->init_seconds = n->initSeconds;
  out->device_bytes = n->devBytes;
  out->window_form = n->winOn ? 1u : 0u;
  out->reserved = 0;
  out->graph_steps = n->graphSteps;
  return 0;
}

void *dpsnn_stream(dpsnn_net *n) { return n ? (void *)n->stream : nullptr; }

int dpsnn_profile(dpsnn_net *n, int enable) {
  if (!n) return fail(DPSNN_ERR_ARG, "null network");
  HIP_TRY(hipStreamSynchronize(n->stream));
  n->profile = enable != 0;
  n->profUsed = 0;
  return 0;
}

int dpsnn_kernel_time(dpsnn_net *n, int kernel, double *avg_ms, uint64_t *launches) {
  if (!n) return fail(DPSNN_ERR_ARG, "null network");
  if (kernel != 0) return fail(DPSNN_ERR_ARG, "kernel 0 (k_step) is the only timed kernel");
  HIP_TRY(hipStreamSynchronize(n->stream));
  double total = 0;
  uint64_t steps = 0;
  for (size_t k = 0; k < n->profUsed; ++k) {
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, n->profEv[k].a, n->profEv[k].b));
    total += ms;
    steps += n->profEv[k].steps;
  }
  if (avg_ms) *avg_ms = steps ? total / (double)steps : 0.0;
  if (launches) *launches = steps;
  n->profUsed = 0;
  return 0;
}

void dpsnn_destroy(dpsnn_net *n) {
  if (!n) return;
  if (n->batch) dpsnn_batch_remove(n->batch, n);
  drain(n);
  n->writer.close();
  n->stdpWriter.close();
  free_all(n);
  delete n;
}

}  // extern "C"

// ============================================================================
// Checkpoint / restore of a network between steps: the device-resident
// state (neurons, bath cursors, Philox counters, spike history, counters,
// STDP synapse state) and the host stream state (ran3 with its NormDev
// cache, the replayed bath's next times, the open output files and the
// counts of the open rates window).  The connectome is not stored: restore
// rebuilds it from the same ini files (the generator is deterministic) and
// checks the sizes recorded in the file.
// ============================================================================
namespace {
constexpr char kCkptMagic[8] = {'D', 'P', 'S', 'N', 'N', 'C', 'K', '1'};
struct CkptHeader {
  char magic[8];
  uint32_t N, RS, NW, drive, stdp, t, nsub, ncols, writer, spikesOpen, ratesOpen, pad;
  uint64_t S, items;
};

struct CkptFile {
  FILE *f = nullptr;
  ~CkptFile() {
    if (f) std::fclose(f);
  }
};

template <class T>
int ck_write(FILE *f, const T *h, size_t n) {
  if (n && std::fwrite(h, sizeof(T), n, f) != n) return fail(DPSNN_ERR_IO, "checkpoint write failed");
  return 0;
}
template <class T>
int ck_read(FILE *f, T *h, size_t n) {
  if (n && std::fread(h, sizeof(T), n, f) != n) return fail(DPSNN_ERR_IO, "checkpoint file truncated");
  return 0;
}
template <class T>
int ck_dev_write(FILE *f, const T *d, size_t n) {
  std::vector<T> h(n);
  HIP_TRY(hipMemcpy(h.data(), d, n * sizeof(T), hipMemcpyDeviceToHost));
  return ck_write(f, h.data(), n);
}
template <class T>
int ck_dev_read(FILE *f, T *d, size_t n) {
  std::vector<T> h(n);
  int rc = ck_read(f, h.data(), n);
  if (rc) return rc;
  HIP_TRY(hipMemcpy(d, h.data(), n * sizeof(T), hipMemcpyHostToDevice));
  return 0;
}

// The device arrays of the state, in file order (the STDP ones last).
template <class Fn>
int ck_device_arrays(dpsnn_net *n, Fn &&fn) {
  DevNet &P = n->dev;
  const size_t N = P.N, S = n->con.S;
  int rc;
  if ((rc = fn(P.v, N)) || (rc = fn(P.c, N)) || (rc = fn(P.Tr, N)) || (rc = fn(P.Te, N)) ||
      (rc = fn(P.assigned, N)) || (rc = fn(P.philoxCtr, N)) || (rc = fn(P.bits, size_t(P.RS) * P.NW)) ||
      (rc = fn(P.teHist, size_t(P.RS) * N)) || (rc = fn(P.counters, size_t(kCounterSlots) * kCounterStride)))
    return rc;
  if (n->stdp && ((rc = fn(P.lastSpike, N)) || (rc = fn(P.wT, S)) || (rc = fn(P.tdT, S)) || (rc = fn(P.lastT, S))))
    return rc;
  return 0;
}
}  // namespace

extern "C" {

int dpsnn_checkpoint(dpsnn_net *n, const char *path) {
  if (!n || !path) return fail(DPSNN_ERR_ARG, "null argument");
  if (!n->uploaded) return fail(DPSNN_ERR_ARG, "network not uploaded (dpsnn_upload)");
  if (n->batch) return fail(DPSNN_ERR_ARG, "network is a member of a batch: remove it first");
  if (n->stdpEvents) return fail(DPSNN_ERR_ARG, "a network writing the STDPevent file cannot be checkpointed");
  HIP_TRY(hipSetDevice(n->opt.device));
  int rc = dpsnn_sync(n);  // every step's files are written up to now
  if (rc) return rc;
  n->writer.flush();
  CkptFile cf;
  if (!(cf.f = std::fopen(path, "wb"))) return fail(DPSNN_ERR_IO, "cannot open %s", path);
  const StatWriter::State ws = n->writer.state();
  CkptHeader h{};
  std::memcpy(h.magic, kCkptMagic, sizeof h.magic);
  h.N = n->dev.N; h.RS = n->dev.RS; h.NW = n->dev.NW; h.drive = n->dev.drive; h.stdp = n->stdp;
  h.t = n->t; h.nsub = n->dev.nsub; h.ncols = n->dev.ncols; h.writer = n->writing;
  h.spikesOpen = ws.spikesOpen; h.ratesOpen = ws.ratesOpen;
  h.S = n->con.S; h.items = n->items;
  if ((rc = ck_write(cf.f, &h, 1))) return rc;
  if ((rc = ck_device_arrays(n, [&](auto *d, size_t cnt) { return ck_dev_write(cf.f, d, cnt); }))) return rc;
  const Ran3::State rs = n->rng.state();
  if ((rc = ck_write(cf.f, &rs, 1))) return rc;
  if (n->dev.drive == DPSNN_DRIVE_REPLAY && (rc = ck_write(cf.f, n->replay.next_times().data(), h.N))) return rc;
  if (n->writing && (rc = ck_write(cf.f, ws.perPop.data(), ws.perPop.size()))) return rc;
  if (std::fflush(cf.f) != 0) return fail(DPSNN_ERR_IO, "checkpoint write failed");
  return 0;
}

int dpsnn_restore(const char *inidir, const dpsnn_options *opt, const char *path, dpsnn_net **out) {
  if (!inidir || !path || !out) return fail(DPSNN_ERR_ARG, "null argument");
  *out = nullptr;
  CkptFile cf;
  if (!(cf.f = std::fopen(path, "rb"))) return fail(DPSNN_ERR_IO, "cannot open %s", path);
  CkptHeader h{};
  int rc = ck_read(cf.f, &h, 1);
  if (rc) return rc;
  if (std::memcmp(h.magic, kCkptMagic, sizeof h.magic) != 0)
    return fail(DPSNN_ERR_IO, "%s is not a network checkpoint", path);
  dpsnn_net *n = nullptr;
  if ((rc = dpsnn_create(inidir, opt, &n))) return rc;
  std::unique_ptr<dpsnn_net, void (*)(dpsnn_net *)> guard(n, dpsnn_destroy);
  if (h.N != n->dev.N || h.S != n->con.S || h.items != n->items || h.RS != n->dev.RS || h.NW != n->dev.NW ||
      h.nsub != n->dev.nsub || h.ncols != n->dev.ncols || h.stdp != (uint32_t)n->stdp)
    return fail(DPSNN_ERR_CONFIG, "the checkpoint was taken on another network (sizes differ)");
  if (h.drive != n->dev.drive) return fail(DPSNN_ERR_CONFIG, "the checkpoint was taken with another drive");
  if (h.t > n->par.pub.totalSimTime_ms)
    return fail(DPSNN_ERR_CONFIG, "the checkpoint is at %u ms, past env_totalSimTime_ms", h.t);
  HIP_TRY(hipSetDevice(n->opt.device));
  HIP_TRY(hipStreamSynchronize(n->stream));
  if ((rc = ck_device_arrays(n, [&](auto *d, size_t cnt) { return ck_dev_read(cf.f, d, cnt); }))) return rc;
  if (n->stdp) {
    // what the restored arrays determine: the spike masks and, after a
    // commit, the in-list items' weights
    hipLaunchKernelGGL(k_mask_from_bits, dim3((n->dev.N + kWaveLTP - 1) / kWaveLTP), dim3(kWaveLTP), 0, n->stream,
                       n->dev, h.t);
    refresh_weights(n);
    HIP_TRY(hipGetLastError());
  }
  Ran3::State rs{};
  if ((rc = ck_read(cf.f, &rs, 1))) return rc;
  n->rng.set_state(rs);
  if (h.drive == DPSNN_DRIVE_REPLAY && (rc = ck_read(cf.f, n->replay.next_times().data(), h.N))) return rc;
  if (h.writer) {
    StatWriter::State ws;
    ws.perPop.resize(size_t(h.ncols) * h.nsub);
    ws.spikesOpen = h.spikesOpen;
    ws.ratesOpen = h.ratesOpen;
    if ((rc = ck_read(cf.f, ws.perPop.data(), ws.perPop.size()))) return rc;
    if (n->writing && !n->writer.resume(ws, h.t / 1000))
      return fail(DPSNN_ERR_IO, "cannot reopen the output files in %s", n->opt.output_dir);
  }
  n->t = h.t;
  *out = guard.release();
  return 0;
}

}  // extern "C"

// ============================================================================
// Batching: many independent networks advance in one persistent launch per
// step (k_batch_step).  Members keep their own state, history, in-lists,
// counters and output files; the batch owns the stream, the per-step item
// ring and the key scratch.
// ============================================================================
struct dpsnn_batch {
  int device = 0;
  int cus = 1;
  hipStream_t stream = nullptr;
  std::vector<dpsnn_net *> nets;
  bool dirty = true;
  DevNet *d_nets = nullptr;
  size_t netsCap = 0;
  static constexpr int kRing = 4;
  BatchItem *h_items[kRing] = {};
  BatchItem *d_items[kRing] = {};
  hipEvent_t done[kRing] = {};
  bool pending[kRing] = {};
  size_t itemsCap = 0;
  int ringNext = 0;
  uint64_t *keys = nullptr;
  int16_t *keyW = nullptr;
  uint16_t *keyPos = nullptr;
  uint32_t *keyCount = nullptr;
  uint32_t *workCtr = nullptr;  // [kXcds], zero between launches
  size_t scratchSlots = 0;
  uint32_t scratchCap = 0;
  uint32_t totalTiles = 0;   // of all members
  uint32_t chunkTiles = 0;   // split form: tiles per chunk (scratch bound)
  int shape = -1;
  uint32_t wavesPerCu = 0;
  bool split = true;         // k_batch_gather + k_batch_integrate per chunk; else k_batch_step
  bool useGraph = true;      // replay each step's launches from a captured HIP graph
  struct Graph {
    hipGraphExec_t exec = nullptr;
    uint32_t count = 0, tiles = 0, chunkTiles = 0, wpc = 0;
    int shape = -1;
    bool split = false, packed = false, ltp = false;
  } graphs[kRing];
  bool profile = false;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> ev;
  size_t evUsed = 0;
  std::vector<StepPlan> plans;
  std::vector<dpsnn_net *> active;
  std::vector<uint32_t> windowed;  // this step's members (indices into active) in the window form
};

// Scratch the split form may use for one chunk of tiles.
constexpr size_t kBatchScratchBytes = size_t(11) << 29;  // also holds a 16 x 16-column member in the window form

namespace {

uint32_t batch_cap(const dpsnn_batch *b) {
  uint32_t cap = 1;
  for (auto *n : b->nets) cap = std::max(cap, n->dev.cap);
  return cap;
}

uint32_t lds_waves(size_t lds) {
  return std::max<uint32_t>(1, std::min<uint32_t>(16, (uint32_t)((160u << 10) / lds)));
}

void batch_free_items(dpsnn_batch *b) {
  for (int r = 0; r < dpsnn_batch::kRing; ++r) {
    if (b->h_items[r]) hipHostFree(b->h_items[r]);
    if (b->d_items[r]) hipFree(b->d_items[r]);
    b->h_items[r] = nullptr;
    b->d_items[r] = nullptr;
  }
  b->itemsCap = 0;
}

// Device copy of the members' DevNet structs, scratch for the longest
// in-list at the largest grid any shape uses, item ring for every member.
int batch_prepare(dpsnn_batch *b) {
  if (!b->dirty) return 0;
  HIP_TRY(hipStreamSynchronize(b->stream));
  // captured graphs name the buffers below, which may move
  for (auto &g : b->graphs) {
    if (g.exec) HIP_TRY(hipGraphExecDestroy(g.exec));
    g = dpsnn_batch::Graph{};
  }
  const size_t count = b->nets.size();
  if (count > b->netsCap) {
    if (b->d_nets) HIP_TRY(hipFree(b->d_nets));
    b->d_nets = nullptr;
    HIP_TRY(hipMalloc((void **)&b->d_nets, sizeof(DevNet) * count));
    b->netsCap = count;
  }
  std::vector<DevNet> h(count);
  for (size_t i = 0; i < count; ++i) {
    h[i] = b->nets[i]->dev;
    if (!b->split) h[i].bathT = nullptr;  // the fused launch merges the bath in phase 2
  }
  if (count) HIP_TRY(hipMemcpy(b->d_nets, h.data(), sizeof(DevNet) * count, hipMemcpyHostToDevice));
  if (count > b->itemsCap) {
    batch_free_items(b);
    const size_t cap = count + 8;
    for (int r = 0; r < dpsnn_batch::kRing; ++r) {
      HIP_TRY(hipHostMalloc((void **)&b->h_items[r], sizeof(BatchItem) * cap, 0));
      HIP_TRY(hipMalloc((void **)&b->d_items[r], sizeof(BatchItem) * cap));
      b->pending[r] = false;
    }
    b->itemsCap = cap;
  }
  const uint32_t cap = batch_cap(b);
  b->totalTiles = 0;
  for (auto *n : b->nets) b->totalTiles += n->dev.NW;
  const size_t perTile = (size_t)cap * kWave * (sizeof(uint64_t) + 2 * sizeof(int16_t));
  b->chunkTiles = (uint32_t)std::max<size_t>(1, std::min<size_t>(b->totalTiles, kBatchScratchBytes / perTile));
  const size_t fusedSlots = (size_t)round_up((uint32_t)b->cus * lds_waves(lds_bytes(cap, 64)), kXcds) * kWave;
  const size_t slots = std::max(fusedSlots, (size_t)b->chunkTiles * kWave);
  if (cap > b->scratchCap || slots > b->scratchSlots) {
    if (b->keys) HIP_TRY(hipFree(b->keys));
    if (b->keyW) HIP_TRY(hipFree(b->keyW));
    if (b->keyPos) HIP_TRY(hipFree(b->keyPos));
    if (b->keyCount) HIP_TRY(hipFree(b->keyCount));
    b->keys = nullptr;
    b->keyW = nullptr;
    b->keyPos = nullptr;
    b->keyCount = nullptr;
    hipError_t e = hipMalloc((void **)&b->keys, sizeof(uint64_t) * slots * cap);
    if (e != hipSuccess) return fail(DPSNN_ERR_MEMORY, "batch key scratch: %s", hipGetErrorString(e));
    e = hipMalloc((void **)&b->keyW, sizeof(int16_t) * slots * cap);
    if (e != hipSuccess) return fail(DPSNN_ERR_MEMORY, "batch weight scratch: %s", hipGetErrorString(e));
    e = hipMalloc((void **)&b->keyPos, sizeof(uint16_t) * slots * cap);
    if (e != hipSuccess) return fail(DPSNN_ERR_MEMORY, "batch position scratch: %s", hipGetErrorString(e));
    HIP_TRY(hipMalloc((void **)&b->keyCount, sizeof(uint32_t) * slots));
    b->scratchCap = cap;
    b->scratchSlots = slots;
  }
  if (b->shape < 0) {
    const int K = cap <= 8 * 64 ? 8 : (cap <= 16 * 64 ? 16 : 24);
    b->shape = find_shape(K, 256);
  }
  b->dirty = false;
  return 0;
}

// The device copies of the members depend on the form (batch_prepare).
void batch_set_split(dpsnn_batch *b, bool split) {
  b->dirty = b->dirty || split != b->split;
  b->split = split;
}

uint32_t batch_waves(const dpsnn_batch *b, size_t lds) {
  uint32_t wpc = lds_waves(lds);
  if (b->wavesPerCu) wpc = std::min(wpc, b->wavesPerCu);
  return wpc;
}

// The device work of one batched step: the items of ring slot r, then either
// the persistent fused kernel or, chunk by chunk, phase 1 and phase 2
// (packed: every member is at t >= kPackT, so phase 2 runs its packed-only
// instance; ltp: some member's next scan runs LTP).
int batch_launch(dpsnn_batch *b, int r, uint32_t count, uint32_t tiles, bool packed, bool ltp) {
  HIP_TRY(hipMemcpyAsync(b->d_items[r], b->h_items[r], sizeof(BatchItem) * count, hipMemcpyHostToDevice, b->stream));
  const KernelShape &K = kShapes[b->shape];
  const uint32_t cap = b->scratchCap;
  if (!b->split) {
    const size_t lds = lds_bytes(cap, K.B);
    const uint32_t grid = round_up(std::min<uint32_t>(tiles, (uint32_t)b->cus * batch_waves(b, lds)), kXcds);
    hipLaunchKernelGGL(K.batch, dim3(grid), dim3(kWave), lds, b->stream, b->d_nets, b->d_items[r], count, tiles, cap,
                       b->keys, b->keyW, b->keyPos, b->keyCount);
  } else {
    const size_t lds = phase1_lds(cap, K.B);
    for (uint32_t g0 = 0; g0 < tiles; g0 += b->chunkTiles) {
      const uint32_t g1 = std::min(tiles, g0 + b->chunkTiles);
      const uint32_t grid = round_up(
          std::min<uint32_t>((g1 - g0) * kWave,
                             (uint32_t)b->cus * std::min(batch_waves(b, lds), resident_waves((const void *)K.batchGather, lds))),
          kXcds);
      hipLaunchKernelGGL(k_batch_bath, dim3(g1 - g0), dim3(kWave), 0, b->stream, b->d_nets, b->d_items[r], count, g0);
      hipLaunchKernelGGL(K.batchGather, dim3(grid), dim3(kWave), lds, b->stream, b->d_nets, b->d_items[r], count, g0,
                         g1, cap, b->keys, b->keyW, b->keyPos, b->keyCount, b->workCtr);
      const uint32_t blocks = (g1 - g0 + kBlock / kWave - 1) / (kBlock / kWave);
      if (packed)
        hipLaunchKernelGGL(k_batch_integrate<1>, dim3(blocks), dim3(kBlock), 0, b->stream, b->d_nets, b->d_items[r],
                           count, g0, g1, cap, b->keys, b->keyW, b->keyCount, b->workCtr);
      else
        hipLaunchKernelGGL(k_batch_integrate<2>, dim3(blocks), dim3(kBlock), 0, b->stream, b->d_nets, b->d_items[r],
                           count, g0, g1, cap, b->keys, b->keyW, b->keyCount, b->workCtr);
      if (ltp)
        hipLaunchKernelGGL(k_batch_ltp, dim3(std::min<uint32_t>((g1 - g0) * (kWave * kWave / kWaveLTP), b->cus * 16u)),
                           dim3(kWaveLTP), 0, b->stream, b->d_nets, b->d_items[r], count, g0, g1);
    }
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

void batch_drop_graphs(dpsnn_batch *b) {
  for (auto &g : b->graphs) {
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
    g = dpsnn_batch::Graph{};
  }
}

// The same work replayed from a graph captured once per ring slot and launch
// configuration (the per-step arguments live in the slot's items).
int batch_graph_launch(dpsnn_batch *b, int r, uint32_t count, uint32_t tiles, bool packed, bool ltp) {
  dpsnn_batch::Graph &g = b->graphs[r];
  const uint32_t wpc = b->wavesPerCu;
  if (!g.exec || g.count != count || g.tiles != tiles || g.chunkTiles != b->chunkTiles || g.wpc != wpc ||
      g.shape != b->shape || g.split != b->split || g.packed != packed || g.ltp != ltp) {
    if (g.exec) HIP_TRY(hipGraphExecDestroy(g.exec));
    g = dpsnn_batch::Graph{};
    hipGraph_t graph = nullptr;
    HIP_TRY(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    const int rc = batch_launch(b, r, count, tiles, packed, ltp);
    const hipError_t e = hipStreamEndCapture(b->stream, &graph);
    if (rc) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc;
    }
    if (e != hipSuccess) return fail(DPSNN_ERR_DEVICE, "graph capture failed: %s", hipGetErrorString(e));
    const hipError_t ei = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (ei != hipSuccess) {
      g.exec = nullptr;
      return fail(DPSNN_ERR_DEVICE, "graph instantiation failed: %s", hipGetErrorString(ei));
    }
    g.count = count;
    g.tiles = tiles;
    g.chunkTiles = b->chunkTiles;
    g.wpc = wpc;
    g.shape = b->shape;
    g.split = b->split;
    g.packed = packed;
    g.ltp = ltp;
  }
  HIP_TRY(hipGraphLaunch(g.exec, b->stream));
  return 0;
}

// One batched step of every member that has steps left; *any = false when
// none has.
int batch_one_step(dpsnn_batch *b, bool *any) {
  b->active.clear();
  for (auto *n : b->nets)
    if (n->t < n->par.pub.totalSimTime_ms) b->active.push_back(n);
  *any = !b->active.empty();
  if (!*any) return 0;
  int rc;
  if ((rc = batch_prepare(b))) return rc;
  const int r = b->ringNext;
  b->ringNext = (r + 1) % dpsnn_batch::kRing;
  if (b->pending[r]) HIP_TRY(hipEventSynchronize(b->done[r]));
  b->plans.resize(b->active.size());
  b->windowed.clear();
  uint32_t tiles = 0, count = 0;
  bool packed = true, ltp = false;
  for (size_t i = 0; i < b->active.size(); ++i) {
    dpsnn_net *n = b->active[i];
    StepPlan &sp = b->plans[i];
    if ((rc = pre_step(n, sp))) return rc;
    // a member whose step runs in the window form, and whose tiles fit the
    // batch's key scratch, steps on its own launches (below)
    if (n->dev.N >= kBatchWindowMin && window_step(n, sp) && (size_t)n->dev.NW * kWave <= b->scratchSlots) {
      b->windowed.push_back((uint32_t)i);
      continue;
    }
    packed = packed && sp.t >= kPackT;
    ltp = ltp || sp.S.ltp;
    const uint32_t idx = (uint32_t)(std::find(b->nets.begin(), b->nets.end(), n) - b->nets.begin());
    b->h_items[r][count++] = BatchItem{sp.t, sp.ltd, sp.S, sp.X, tiles, idx};
    tiles += n->dev.NW;
  }
  if (b->profile) {
    if (b->evUsed == b->ev.size()) {
      hipEvent_t x, y;
      HIP_TRY(hipEventCreate(&x));
      HIP_TRY(hipEventCreate(&y));
      b->ev.emplace_back(x, y);
    }
    HIP_TRY(hipEventRecord(b->ev[b->evUsed].first, b->stream));
  }
  if (count && b->useGraph) {
    if ((rc = batch_graph_launch(b, r, count, tiles, packed, ltp))) return rc;
  } else if (count) {
    if ((rc = batch_launch(b, r, count, tiles, packed, ltp))) return rc;
  }
  // window-form members, one after another on the batch's stream and key
  // scratch (its cap is the largest member's, so their tiles fit it)
  for (uint32_t i : b->windowed) {
    const dpsnn_net *n = b->active[i];
    DevNet P = n->dev;
    P.keys = b->keys;
    P.keyW = b->keyW;
    P.keyCount = b->keyCount;
    P.cap = b->scratchCap;
    P.tDev = nullptr;
    launch_window_step(n, P, b->plans[i], b->stream);
  }
  HIP_TRY(hipGetLastError());
  if (b->profile) HIP_TRY(hipEventRecord(b->ev[b->evUsed++].second, b->stream));
  HIP_TRY(hipEventRecord(b->done[r], b->stream));
  b->pending[r] = true;
  for (size_t i = 0; i < b->active.size(); ++i)
    if ((rc = post_step(b->active[i], b->plans[i]))) return rc;
  return 0;
}

int batch_kernel_ms(dpsnn_batch *b, double *avg, uint64_t *launches) {
  HIP_TRY(hipStreamSynchronize(b->stream));
  double total = 0;
  for (size_t k = 0; k < b->evUsed; ++k) {
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, b->ev[k].first, b->ev[k].second));
    total += ms;
  }
  if (avg) *avg = b->evUsed ? total / (double)b->evUsed : 0.0;
  if (launches) *launches = b->evUsed;
  b->evUsed = 0;
  return 0;
}

}  // namespace

extern "C" {

int dpsnn_batch_create(int device, dpsnn_batch **out) {
  if (!out) return fail(DPSNN_ERR_ARG, "null argument");
  *out = nullptr;
  std::unique_ptr<dpsnn_batch> b(new dpsnn_batch());
  b->device = device;
  HIP_TRY(hipSetDevice(device));
  HIP_TRY(hipDeviceGetAttribute(&b->cus, hipDeviceAttributeMultiprocessorCount, device));
  b->cus = std::max(b->cus, 1);
  HIP_TRY(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
  for (int r = 0; r < dpsnn_batch::kRing; ++r) HIP_TRY(hipEventCreateWithFlags(&b->done[r], hipEventDisableTiming));
  HIP_TRY(hipMalloc((void **)&b->workCtr, sizeof(uint32_t) * kXcds * kCtrStride));
  HIP_TRY(hipMemset(b->workCtr, 0, sizeof(uint32_t) * kXcds * kCtrStride));
  if (const char *e = std::getenv("DPSNN_GRAPH")) b->useGraph = std::atoi(e) != 0;
  if (const char *e = std::getenv("DPSNN_SPLIT")) b->split = std::atoi(e) != 0;
  *out = b.release();
  return 0;
}

int dpsnn_batch_add(dpsnn_batch *b, dpsnn_net *n) {
  if (!b || !n) return fail(DPSNN_ERR_ARG, "null argument");
  if (n->batch) return fail(DPSNN_ERR_ARG, "network is already a member of a batch");
  if (n->opt.device != b->device) return fail(DPSNN_ERR_ARG, "network and batch are on different devices");
  if (!n->uploaded) return fail(DPSNN_ERR_ARG, "network not uploaded (dpsnn_upload)");
  HIP_TRY(hipSetDevice(b->device));
  HIP_TRY(hipStreamSynchronize(n->stream));
  n->ownStream = n->stream;
  n->stream = b->stream;
  n->batch = b;
  b->nets.push_back(n);
  b->dirty = true;
  return 0;
}

int dpsnn_batch_remove(dpsnn_batch *b, dpsnn_net *n) {
  if (!b || !n) return fail(DPSNN_ERR_ARG, "null argument");
  auto it = std::find(b->nets.begin(), b->nets.end(), n);
  if (it == b->nets.end() || n->batch != b) return fail(DPSNN_ERR_ARG, "network is not a member of this batch");
  HIP_TRY(hipSetDevice(b->device));
  HIP_TRY(hipStreamSynchronize(b->stream));
  b->nets.erase(it);
  n->stream = n->ownStream;
  n->ownStream = nullptr;
  n->batch = nullptr;
  b->dirty = true;
  return 0;
}

uint32_t dpsnn_batch_size(const dpsnn_batch *b) { return b ? (uint32_t)b->nets.size() : 0; }

int dpsnn_batch_step(dpsnn_batch *b, uint32_t nsteps) {
  if (!b) return fail(DPSNN_ERR_ARG, "null batch");
  HIP_TRY(hipSetDevice(b->device));
  for (uint32_t k = 0; k < nsteps; ++k) {
    bool any = false;
    // a member's blocks are its own: each ends within this call
    if (b->split)
      for (auto *n : b->nets) stdp_open(n, nsteps - k);
    int rc = batch_one_step(b, &any);
    for (auto *n : b->nets) {
      const int rc2 = stdp_close(n, rc || !any ? 0 : 1, rc || !any);
      rc = rc ? rc : rc2;
    }
    if (rc) return rc;
    if (!any) {
      for (auto *n : b->nets)
        if ((rc = drain(n))) return rc;
      return DPSNN_DONE;
    }
  }
  return 0;
}

int dpsnn_batch_sync(dpsnn_batch *b) {
  if (!b) return fail(DPSNN_ERR_ARG, "null batch");
  HIP_TRY(hipSetDevice(b->device));
  HIP_TRY(hipStreamSynchronize(b->stream));
  int rc;
  for (auto *n : b->nets)
    if ((rc = drain(n))) return rc;
  return 0;
}

int dpsnn_batch_get_shape(const dpsnn_batch *b, dpsnn_batch_shape *s) {
  if (!b || !s) return fail(DPSNN_ERR_ARG, "null argument");
  const int i = b->shape < 0 ? find_shape(24, 256) : b->shape;
  s->chunks = kShapes[i].K;
  s->buckets = kShapes[i].B;
  s->waves_per_cu = (int)b->wavesPerCu;
  s->ms_per_step = 0;
  s->split = b->split ? 1 : 0;
  return 0;
}

int dpsnn_batch_set_shape(dpsnn_batch *b, const dpsnn_batch_shape *s) {
  if (!b || !s) return fail(DPSNN_ERR_ARG, "null argument");
  const int i = find_shape(s->chunks, s->buckets);
  if (i < 0) return fail(DPSNN_ERR_ARG, "no kernel shape with %d register chunks and %d buckets", s->chunks, s->buckets);
  if (s->waves_per_cu < 0 || s->waves_per_cu > 16) return fail(DPSNN_ERR_ARG, "waves_per_cu must be in 0..16");
  b->shape = i;
  b->wavesPerCu = (uint32_t)s->waves_per_cu;
  batch_set_split(b, s->split != 0);
  return 0;
}

int dpsnn_batch_profile(dpsnn_batch *b, int enable) {
  if (!b) return fail(DPSNN_ERR_ARG, "null batch");
  HIP_TRY(hipStreamSynchronize(b->stream));
  b->profile = enable != 0;
  b->evUsed = 0;
  return 0;
}

int dpsnn_batch_kernel_time(dpsnn_batch *b, double *avg_ms, uint64_t *launches) {
  if (!b) return fail(DPSNN_ERR_ARG, "null batch");
  return batch_kernel_ms(b, avg_ms, launches);
}

int dpsnn_batch_tune(dpsnn_batch *b, uint32_t trial_steps, dpsnn_batch_shape *chosen) {
  if (!b) return fail(DPSNN_ERR_ARG, "null batch");
  if (trial_steps == 0) trial_steps = 1;
  HIP_TRY(hipSetDevice(b->device));
  const bool wasProfiling = b->profile;
  int rc;
  if ((rc = batch_prepare(b))) return rc;
  const uint32_t cap = batch_cap(b);
  double best = 1e300;
  int bestShape = b->shape;
  uint32_t bestWaves = b->wavesPerCu;
  bool bestSplit = b->split, any = true;
  // every candidate computes the same result; the trial steps are real steps
  for (int split = 1; split >= 0 && any; --split)
    for (int i = 0; i < kNumShapes && any; ++i) {
      const uint32_t top = lds_waves(split ? phase1_lds(cap, kShapes[i].B) : lds_bytes(cap, kShapes[i].B));
      for (uint32_t w : {0u, std::max<uint32_t>(1, top / 2)}) {
        b->shape = i;
        b->wavesPerCu = w;
        batch_set_split(b, split != 0);
        HIP_TRY(hipStreamSynchronize(b->stream));
        b->profile = true;
        b->evUsed = 0;
        for (uint32_t k = 0; k < trial_steps && any; ++k)
          if ((rc = batch_one_step(b, &any))) return rc;
        double ms = 0;
        uint64_t launches = 0;
        if ((rc = batch_kernel_ms(b, &ms, &launches))) return rc;
        if (launches && ms < best) {
          best = ms;
          bestShape = i;
          bestWaves = w;
          bestSplit = b->split;
        }
        if (!any) break;
      }
    }
  b->shape = bestShape;
  b->wavesPerCu = bestWaves;
  batch_set_split(b, bestSplit);
  b->profile = wasProfiling;
  if (chosen) {
    chosen->chunks = kShapes[bestShape].K;
    chosen->buckets = kShapes[bestShape].B;
    chosen->waves_per_cu = (int)bestWaves;
    chosen->ms_per_step = best < 1e300 ? best : 0.0;
    chosen->split = bestSplit ? 1 : 0;
  }
  return 0;
}

void dpsnn_batch_destroy(dpsnn_batch *b) {
  if (!b) return;
  hipSetDevice(b->device);
  while (!b->nets.empty()) dpsnn_batch_remove(b, b->nets.back());
  (void)hipStreamSynchronize(b->stream);
  batch_drop_graphs(b);
  batch_free_items(b);
  if (b->d_nets) (void)hipFree(b->d_nets);
  if (b->keys) hipFree(b->keys);
  if (b->keyW) hipFree(b->keyW);
  if (b->keyCount) (void)hipFree(b->keyCount);
  if (b->keyPos) (void)hipFree(b->keyPos);
  if (b->workCtr) (void)hipFree(b->workCtr);
  for (int r = 0; r < dpsnn_batch::kRing; ++r)
    if (b->done[r]) hipEventDestroy(b->done[r]);
  for (auto &e : b->ev) {
    hipEventDestroy(e.first);
    hipEventDestroy(e.second);
  }
  hipStreamDestroy(b->stream);
  delete b;
}

}  // extern "C"

// ============================================================================
// Host-only access and diagnostics
// ============================================================================
struct dpsnn_host_net {
  Params par;
  Connectome con;
  Ran3 rng;
  ExternalReplay replay;
  ExternalStep step;
  uint32_t t = 0;
  WindowLayout window;
  uint32_t windowUnitsPerCol = 0;
};

namespace {
int write_dump(const Connectome &c, float w2f, const char *path) {
  FILE *f = std::fopen(path, "w");
  if (!f) return fail(DPSNN_ERR_IO, "cannot open %s", path);
  std::vector<char> line(256);
  for (uint64_t s = 0; s < c.S; ++s) {
    const float w = (float)(c.weight[s] * w2f);
    const int len = std::snprintf(line.data(), line.size(), "%d %d %d %d %d %f %f\n", (int)c.pre[s],
                                  (int)c.post[s], (int)(c.post[s] / c.N), (int)c.delay[s], (int)c.kind[s],
                                  w, 0.0f);
    std::fwrite(line.data(), 1, (size_t)len, f);
  }
  std::fclose(f);
  return 0;
}
__global__ void k_exp(const double *x, double *y, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = dpsnn_exp(x[i]);
}
// yl[i] != 0: b[i] is a short divisor (yl = 0 goes with an exact reciprocal,
// where both forms are one rounded product).
__global__ void k_div(const double *a, const double *b, const double *y, const double *yl, double *q, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) q[i] = yl[i] != 0.0 ? div_short(a[i], y[i], yl[i]) : div_rn(a[i], b[i], y[i]);
}
}  // namespace

extern "C" {

int dpsnn_host_build(const char *inidir, dpsnn_host_net **out) {
  if (!inidir || !out) return fail(DPSNN_ERR_ARG, "null argument");
  *out = nullptr;
  std::unique_ptr<dpsnn_host_net> h(new dpsnn_host_net());
  std::string err;
  if (!read_params(inidir, h->par, err)) return fail(DPSNN_ERR_CONFIG, "%s", err.c_str());
  h->rng.seed((int32_t)h->par.pub.globalSeed);
  const bool verbose = std::getenv("DPSNN_VERBOSE") != nullptr;
  auto t0 = std::chrono::steady_clock::now();
  if (!generate_connectome(h->par, h->rng, h->con, err)) return fail(DPSNN_ERR_CONFIG, "%s", err.c_str());
  auto t1 = std::chrono::steady_clock::now();
  build_delivery(h->par, h->con);
  auto t2 = std::chrono::steady_clock::now();
  if (verbose)
    std::fprintf(stderr, "[dpsnn] generate %.2f s, delivery layout %.2f s\n",
                 std::chrono::duration<double>(t1 - t0).count(), std::chrono::duration<double>(t2 - t1).count());
  h->rng.seed(0);
  h->replay.init(h->con, &h->rng);
  *out = h.release();
  return 0;
}
uint32_t dpsnn_host_num_neurons(const dpsnn_host_net *h) { return h ? h->con.N : 0; }
uint64_t dpsnn_host_num_synapses(const dpsnn_host_net *h) { return h ? h->con.S : 0; }
uint64_t dpsnn_host_num_items(const dpsnn_host_net *h) { return h ? h->con.in_off[h->con.N] : 0; }
int dpsnn_host_get_synapses(const dpsnn_host_net *h, uint32_t *pre, uint32_t *post, uint8_t *delay,
                            int16_t *weight) {
  if (!h) return fail(DPSNN_ERR_ARG, "null argument");
  const Connectome &c = h->con;
  if (pre) std::memcpy(pre, c.pre.data(), 4 * c.S);
  if (post) std::memcpy(post, c.post.data(), 4 * c.S);
  if (delay) std::memcpy(delay, c.delay.data(), c.S);
  if (weight) std::memcpy(weight, c.weight.data(), 2 * c.S);
  return 0;
}
int dpsnn_host_get_inlists(const dpsnn_host_net *h, uint64_t *off, uint32_t *pre_delay, int16_t *weight,
                           uint32_t *syn) {
  if (!h) return fail(DPSNN_ERR_ARG, "null argument");
  const Connectome &c = h->con;
  const uint64_t items = c.in_off[c.N];
  if (off) std::memcpy(off, c.in_off.data(), 8 * (c.N + 1));
  if (pre_delay) std::memcpy(pre_delay, c.in_pre_d.data(), 4 * items);
  if (weight) std::memcpy(weight, c.in_w.data(), 2 * items);
  if (syn) std::memcpy(syn, c.in_syn.data(), 4 * items);
  return 0;
}
int dpsnn_host_window(dpsnn_host_net *h, uint32_t units_per_col, uint32_t dims[6], uint64_t sizes[4],
                      uint32_t *item, uint16_t *desc, uint64_t *chunk, int32_t *cols) {
  if (!h || !dims || !sizes) return fail(DPSNN_ERR_ARG, "null argument");
  WindowLayout &L = h->window;
  if (!L.ok || h->windowUnitsPerCol != units_per_col) {
    build_window(h->par, h->con, units_per_col, kWindowMaxEntries, L);
    h->windowUnitsPerCol = units_per_col;
    if (!L.ok) return fail(DPSNN_ERR_CONFIG, "no stencil-window layout: %s", L.why.c_str());
  }
  const uint32_t d[6] = {L.slots, L.npc, L.passes, L.unit, L.unitsPerCol, L.units};
  std::memcpy(dims, d, sizeof d);
  sizes[0] = L.item.size(); sizes[1] = L.desc.size(); sizes[2] = L.chunk.size(); sizes[3] = L.cols.size();
  if (item) std::memcpy(item, L.item.data(), 4 * L.item.size());
  if (desc) std::memcpy(desc, L.desc.data(), 2 * L.desc.size());
  if (chunk) std::memcpy(chunk, L.chunk.data(), 8 * L.chunk.size());
  if (cols) std::memcpy(cols, L.cols.data(), 4 * L.cols.size());
  return 0;
}
int dpsnn_host_get_external(const dpsnn_host_net *h, double *invNuExt, uint32_t *maxCount) {
  if (!h) return fail(DPSNN_ERR_ARG, "null argument");
  if (invNuExt) std::memcpy(invNuExt, h->con.invNuExt.data(), 8 * h->con.N);
  if (maxCount) std::memcpy(maxCount, h->con.maxExt.data(), 4 * h->con.N);
  return 0;
}
int dpsnn_host_write_synapse_dump(const dpsnn_host_net *h, const char *path) {
  if (!h || !path) return fail(DPSNN_ERR_ARG, "null argument");
  return write_dump(h->con, h->par.pub.factorWeightType_2_Float, path);
}
int dpsnn_host_external_step(dpsnn_host_net *h, uint32_t *off, double *time, double *value, uint64_t cap,
                             uint64_t *count) {
  if (!h) return fail(DPSNN_ERR_ARG, "null argument");
  h->replay.generate(h->t++, h->step);
  const uint64_t ne = h->step.time.size();
  if (count) *count = ne;
  if (off) std::memcpy(off, h->step.off.data(), 4 * (size_t(h->con.N) + 1));
  if (ne > cap) return fail(DPSNN_ERR_ARG, "external buffer holds %llu events, %llu needed",
                            (unsigned long long)cap, (unsigned long long)ne);
  if (time) std::memcpy(time, h->step.time.data(), 8 * ne);
  if (value) std::memcpy(value, h->step.value.data(), 8 * ne);
  return 0;
}
void dpsnn_host_destroy(dpsnn_host_net *h) { delete h; }

int dpsnn_write_synapse_dump(dpsnn_net *n, const char *path) {
  if (!n || !path) return fail(DPSNN_ERR_ARG, "null argument");
  if (n->opt.drop_host_synapses) return fail(DPSNN_ERR_ARG, "the host synapse list was dropped (drop_host_synapses)");
  if (!n->stdp) return write_dump(n->con, n->par.pub.factorWeightType_2_Float, path);
  // plastic network: the device's current weights and derivatives
  const Connectome &c = n->con;
  std::vector<int16_t> w(c.S);
  std::vector<float> td(c.S);
  int rc = synapse_state(n, w.data(), td.data(), nullptr);
  if (rc) return rc;
  FILE *f = std::fopen(path, "w");
  if (!f) return fail(DPSNN_ERR_IO, "cannot open %s", path);
  std::vector<char> line(256);
  const float w2f = n->par.pub.factorWeightType_2_Float;
  for (uint64_t s = 0; s < c.S; ++s) {
    const int len = std::snprintf(line.data(), line.size(), "%d %d %d %d %d %f %f\n", (int)c.pre[s], (int)c.post[s],
                                  (int)(c.post[s] / c.N), (int)c.delay[s], (int)c.kind[s], (float)(w[s] * w2f), td[s]);
    std::fwrite(line.data(), 1, (size_t)len, f);
  }
  std::fclose(f);
  return 0;
}

int dpsnn_device_memory(int device, uint64_t *free_bytes, uint64_t *total_bytes) {
  HIP_TRY(hipSetDevice(device));
  size_t f = 0, t = 0;
  HIP_TRY(hipMemGetInfo(&f, &t));
  if (free_bytes) *free_bytes = f;
  if (total_bytes) *total_bytes = t;
  return 0;
}

int dpsnn_device_exp(int device, const double *x, double *y, uint64_t n) {
  if (!x || !y) return fail(DPSNN_ERR_ARG, "null argument");
  HIP_TRY(hipSetDevice(device));
  double *dx = nullptr, *dy = nullptr;
  HIP_TRY(hipMalloc((void **)&dx, 8 * std::max<uint64_t>(n, 1)));
  HIP_TRY(hipMalloc((void **)&dy, 8 * std::max<uint64_t>(n, 1)));
  HIP_TRY(hipMemcpy(dx, x, 8 * n, hipMemcpyHostToDevice));
  const uint64_t blocks = (n + 255) / 256;
  if (n) hipLaunchKernelGGL(k_exp, dim3((uint32_t)blocks), dim3(256), 0, 0, dx, dy, n);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpy(y, dy, 8 * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipFree(dx));
  HIP_TRY(hipFree(dy));
  return 0;
}

int dpsnn_device_div(int device, const double *a, const double *b, double *q, uint64_t n) {
  if (!a || !b || !q) return fail(DPSNN_ERR_ARG, "null argument");
  HIP_TRY(hipSetDevice(device));
  std::vector<double> y(n), yl(n);
  for (uint64_t i = 0; i < n; ++i) {  // as the engine's set-up computes them
    y[i] = 1.0 / b[i];
    yl[i] = short_divisor(b[i]) ? std::fma(-b[i], y[i], 1.0) / b[i] : 0.0;
  }
  double *d = nullptr;
  const size_t bytes = 8 * std::max<uint64_t>(n, 1);
  HIP_TRY(hipMalloc((void **)&d, 5 * bytes));
  HIP_TRY(hipMemcpy(d, a, 8 * n, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d + n, b, 8 * n, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d + 2 * n, y.data(), 8 * n, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d + 3 * n, yl.data(), 8 * n, hipMemcpyHostToDevice));
  const uint64_t blocks = (n + 255) / 256;
  if (n)
    hipLaunchKernelGGL(k_div, dim3((uint32_t)blocks), dim3(256), 0, 0, d, d + n, d + 2 * n, d + 3 * n, d + 4 * n, n);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpy(q, d + 4 * n, 8 * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipFree(d));
  return 0;
}

}  // extern "C"
