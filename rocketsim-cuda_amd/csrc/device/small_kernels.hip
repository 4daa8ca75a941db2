// The decision kernel for small batches: one to three arenas per wave, each ArenaState in LDS.
//
// A wave's time grows with its arenas (it pays for the union of their paths), and a batch of few arenas leaves most SIMDs
// idle, so a small batch is spread over many waves. With so few arenas a wave's states fit the LDS: the tick's dependent
// reads of the state then wait on LDS instead of on private memory (which a wave holds lane-interleaved, one 256-byte row
// per word however few lanes use it, so that spread-out waves would also crowd each other out of the caches). The lanes
// past the wave's arenas help with the copies in and out, where each instruction moves 64 words of one arena.
//
// An arena's two cars and its ball are lanes of their own in the phases that treat them alike (P0, P1, P2, P6, P8 and the
// swept boxes of P3a: SPLIT): with the state in LDS another lane reaches it as well, and a phase that did three bodies or two
// cars in turn takes the time of one. The mesh walks, the batched separating-axis tests and the passes over all boost pads,
// whose work items any lane can take, are spread over every lane of the wave's arenas: all 64 where a wave has three, 22
// where it has one (lane = arena + 3 * role either way, and the lanes of arenas it does not have stay idle). Ms per decision, one lane an arena -> bodies and cars
// split -> walks and tests over all lanes -> boxes and pads too: kickoffs 1,024 arenas 1.01 -> 0.72 -> 0.66 -> 0.61 (P1 109K ->
// 64K cycles per wave and tick); contact mix 64 arenas 1.36 -> 1.29 -> 1.11 -> 1.07, 1,000 arenas 2.05 -> 1.76 -> 1.52 ->
// 1.47.
//
// What bounds it: the tick's own instruction chain and its remaining waits, one wave a SIMD. When it was introduced, still
// one lane an arena, ms per decision over four decisions against one arena per lane in private memory: contact mix 64
// arenas 2.71 -> 1.53, 1,000 arenas 3.55 -> 2.23, 3,072 arenas 3.89 -> 2.96; kickoffs 1,024 arenas 1.26 -> 1.14.
#include "device/launch.h"
#include "device/aosoa.h"

namespace rs {
namespace dev {

// The wave's LDS: the stepper's lane slices and the pooled walks' area (which share the words from 0), then the states.
constexpr uint32_t SMALL_SLICE_WORDS = InLds::ARENAS * InLds::ROLES * (uint32_t)LANE_LDS_WORDS;
#if defined(__HIP_DEVICE_COMPILE__)
static_assert(PoolArea<InLds::WALKERS>::WORDS <= POOL_WORDS, "the pooled walk fits below the states");
#endif
constexpr uint32_t SMALL_STATE_W = POOL_WORDS;
static_assert(SMALL_SLICE_WORDS <= SMALL_STATE_W && SMALL_STATE_W % 4 == 0, "the slices fit below the states");
static uint32_t small_lds_bytes(uint32_t per_wave) { return (SMALL_STATE_W + per_wave * (uint32_t)ARENA_WORDS) * 4u; }

#if defined(__HIP_DEVICE_COMPILE__)
typedef RS_LDS_AS uint32_t LdsWord;
// One wave per work-group: its LDS accesses execute in order, the fences only hold the compiler.
__device__ inline LdsWord* small_state(uint32_t j) { return (LdsWord*)((SMALL_STATE_W + j * (uint32_t)ARENA_WORDS) * 4u); }
// The tick-boundary words of arena a from its AoSoA lane into the wave's state j, the mid-tick tail zeroed: by all 64 lanes,
// every load in flight before the first store.
__device__ inline void small_load(uint32_t j, const uint32_t* __restrict__ buf, uint32_t a) {
  constexpr uint32_t ROUNDS = (uint32_t)(TICK_WORDS + 63) / 64u;
  const uint32_t lane = threadIdx.x;
  const uint32_t* src = buf + block_base(a);
  LdsWord* d = small_state(j);
  uint32_t v[ROUNDS];
#pragma unroll
  for (uint32_t i = 0; i < ROUNDS; ++i) {
    const uint32_t w = i * 64u + lane;
    v[i] = w < (uint32_t)TICK_WORDS ? src[(size_t)w * AOSOA_LANES] : 0u;
  }
#pragma unroll
  for (uint32_t i = 0; i < ROUNDS; ++i) d[i * 64u + lane] = v[i];
  for (uint32_t w = ROUNDS * 64u + lane; w < (uint32_t)ARENA_WORDS; w += 64u) d[w] = 0u;
}
__device__ inline void small_store(uint32_t* __restrict__ buf, uint32_t a, uint32_t j) {
  uint32_t* dst = buf + block_base(a);
  const LdsWord* s = small_state(j);
#pragma unroll 8
  for (uint32_t w = threadIdx.x; w < (uint32_t)TICK_WORDS; w += 64u) dst[(size_t)w * AOSOA_LANES] = s[w];
}
#endif

// `decisions` decisions of arenas per_wave * blockIdx.x onwards: the results of k_sim8 (one decision, with TRACE the state
// after each tick) and k_run. UW: every lane of the wave steps in the same world (no variant array, or one arena per wave).
template <bool UW, bool TRACE>
__global__ void __launch_bounds__(64) k_small(Sim8Args p, uint32_t per_wave, uint32_t decisions) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t a0 = blockIdx.x * per_wave, lane = threadIdx.x;
  const uint32_t cnt = p.n - a0 < per_wave ? p.n - a0 : per_wave;
  const bool part = split_arena() < cnt, mine = lane < cnt;  // role 0 of an arena is its own lane
  const uint32_t slot = part ? split_arena() : 0u, a = a0 + slot;
  const uint32_t v = p.variant ? p.variant[a] : 0u;
  const bool bad = v >= p.nworlds;
  const StaticData& w = p.worlds[bad ? 0u : v];
  for (uint32_t j = 0; j < cnt; ++j) small_load(j, p.buf, a0 + j);
  wave_lds_sync();
  ArenaState& s = *(ArenaState*)(RS_LDS_AS ArenaState*)small_state(slot);
  for (uint32_t d = 0; d < decisions; ++d) {
    if (d > 0) {  // the mid-tick tail is clear at a decision's start, as the copy clears it
      for (uint32_t j = 0; j < cnt; ++j)
        for (uint32_t k = (uint32_t)TICK_WORDS + lane; k < (uint32_t)ARENA_WORDS; k += 64u) small_state(j)[k] = 0u;
      wave_lds_sync();
    }
    uint32_t word = 0u;
    bool live = part && !bad;
    for (uint32_t t = 1; t <= TICKS_PER_DECISION; ++t) {  // run_decision, with the wave's copies out between the ticks
      if (live) {
        const Controls* c = p.ctl + ((size_t)d * p.n + a) * NUM_CARS;
        if (mine)
          for (int i = 0; i < NUM_CARS; ++i) s.cars[i].controls = c[i];
        if (step_tick<UW, InLds>(s, w) != PHASE_OK) word |= SIM8_UNIMPLEMENTED;
      }
      const uint64_t stepped = __ballot(live);
      if (stepped == 0) break;
      if (TRACE) {
        wave_lds_sync();
        for (uint32_t j = 0; j < cnt; ++j)
          if ((stepped >> j) & 1u) small_store(p.trace + (size_t)(t - 1) * aosoa_words(p.n), a0 + j, j);
        wave_lds_sync();
      }
      if (live && ball_scored(s, w)) {
        word |= t;
        live = false;
      }
    }
    if (mine) p.result[(size_t)d * p.n + a] = bad ? SIM8_BAD_VARIANT : word | (any_overflow(s) ? SIM8_OVERFLOW : 0u);
  }
  wave_lds_sync();
  const uint64_t skip = __ballot(mine && bad);
  for (uint32_t j = 0; j < cnt; ++j)
    if (!((skip >> j) & 1u)) small_store(p.buf, a0 + j, j);
#endif
}

// Arenas per wave: one while the waves fill at most two of a CU's four SIMDs, three (what a fourth of a CU's LDS holds)
// above. Waves on one CU share its caches and instruction fetch, which from there on costs more than further arenas in the
// wave (ms per decision with 1 / 2 / 3 per wave, contact mix: 256 arenas 1.23 / 1.29 / 1.38, 512 arenas 1.35 / 1.41 / 1.44,
// 768 arenas 1.45 / 1.43 / 1.43, 1,536 arenas 1.97 / 1.61 / 1.59; kickoffs: 256 arenas 0.57 / 0.59 / 0.59, 768 arenas
// 0.68 / 0.64 / 0.61). Past three on every SIMD a second round of waves follows: at 4,096 arenas contact mix takes 2.36 ms
// here and 2.96 with the states in private memory, but kickoffs 1.42 and 1.07, and at 8,192 both are slower here.
static uint32_t small_per_wave(uint32_t n) { return n <= 512 ? 1u : InLds::ARENAS; }
hipError_t launch_small(hipStream_t st, const Sim8Args& p, uint32_t decisions) {
  const uint32_t per_wave = small_per_wave(p.n), lds = small_lds_bytes(per_wave);
  const dim3 g((p.n + per_wave - 1) / per_wave);
  const bool uw = !p.variant || per_wave == 1;
  if (p.trace && uw) k_small<true, true><<<g, 64, lds, st>>>(p, per_wave, decisions);
  else if (p.trace) k_small<false, true><<<g, 64, lds, st>>>(p, per_wave, decisions);
  else if (uw) k_small<true, false><<<g, 64, lds, st>>>(p, per_wave, decisions);
  else k_small<false, false><<<g, 64, lds, st>>>(p, per_wave, decisions);
  return hipGetLastError();
}
hipError_t small_static_lds(size_t* bytes) {
  const void* kernels[] = {(const void*)k_small<true, true>, (const void*)k_small<false, true>, (const void*)k_small<true, false>,
                           (const void*)k_small<false, false>};
  size_t most = 0;
  for (const void* k : kernels) {
    hipFuncAttributes a;
    hipError_t e = hipFuncGetAttributes(&a, k);
    if (e != hipSuccess) return e;
    most = a.sharedSizeBytes > most ? a.sharedSizeBytes : most;
  }
  *bytes = most;
  return hipSuccess;
}

}  // namespace dev
}  // namespace rs
