// gfx950 kernels of the propagate-to-z + Kalman-update path.
//
// Mapping: one track per lane (wave64), track g = blockIdx.x*blockDim.x +
// threadIdx.x lives in AoSoA block b = g / W at lane l = g % W.  Every load and
// store of a wave touches 64/W contiguous runs of 4W bytes (element-major
// AoSoA, reference OMP:159-161), so track and hit traffic is fully coalesced
// without any transpose.  The track state stays in VGPRs for all layers; the
// hits of layer L+1 are loaded before layer L is computed.
#include "p2z_internal.hpp"
#include "p2z_lane.hpp"

#include <algorithm>
#include <array>
#include <map>
#include <mutex>

namespace p2z {
namespace {

// kStream: non-temporal loads, for the ragged and serving passes, whose track
// input (706 MB for 2000 events) is larger than the 256 MB last-level cache
// and is not read again by the next pass (about 0.8% faster there).  The fused
// pass loads its tracks through the caches: run again on the same buffers it
// takes part of them from the last-level cache (0.115 against 0.121 ms).
template <int W, bool kStream = false>
__device__ inline void load_track(Track& t, const float* __restrict__ tb) {
  auto ld = [&](const float* p) { return kStream ? __builtin_nontemporal_load(p) : *p; };
#pragma unroll
  for (int e = 0; e < 6; ++e) t.p[e] = ld(tb + e * W);
#pragma unroll
  for (int e = 0; e < 21; ++e) t.P[e] = ld(tb + (6 + e) * W);
  const int32_t* q = reinterpret_cast<const int32_t*>(tb) + 27 * W;
  t.q = kStream ? __builtin_nontemporal_load(q) : *q;
}

// The output is written once and not read by the pass: non-temporal stores
// keep it from displacing what the caches hold.  Measured on the 100-event
// pass cycling through three buffer sets (nothing reused across passes from
// the 256 MB last-level cache): 0.131 -> 0.123 ms; on the same buffers every
// pass, where the track input is partly served from that cache, unchanged;
// the 2000-event ragged pass 1-1.5% faster.  Non-temporal track loads as well
// gave the same cold-cache time but lost that reuse (0.121 ms on the same
// buffers).
template <int W>
__device__ inline void store_track(const Track& t, float* __restrict__ ob) {
#pragma unroll
  for (int e = 0; e < 6; ++e) __builtin_nontemporal_store(t.p[e], ob + e * W);
#pragma unroll
  for (int e = 0; e < 21; ++e) __builtin_nontemporal_store(t.P[e], ob + (6 + e) * W);
  __builtin_nontemporal_store(t.q, reinterpret_cast<int32_t*>(ob) + 27 * W);
}

// Hits are read exactly once: non-temporal loads keep them out of the way of
// the track state in the caches.
template <int W>
__device__ inline Hit load_hit(const float* __restrict__ hb) {
  Hit h;
  h.x = __builtin_nontemporal_load(hb + 0 * W);
  h.y = __builtin_nontemporal_load(hb + 1 * W);
  h.z = __builtin_nontemporal_load(hb + 2 * W);
  h.xx = __builtin_nontemporal_load(hb + 3 * W);
  h.xy = __builtin_nontemporal_load(hb + 4 * W);
  h.yy = __builtin_nontemporal_load(hb + 5 * W);
  return h;
}

// Whether a wave's layers have to be computed again in the reference typing's
// full form (redo_ref); no other arithmetic marks tracks.  The whole wave: the
// marked lanes alone took 99 us for 20 layers (two of 64 lanes), all of them 28.
template <int kMath>
__device__ inline bool marked(const Track& t, const Carry<kMath>& g) {
  if constexpr (kMath == kRef)
    return any_lane(g.redo || !ref_finite(t));
  else
    return false;
}

// Whether a wave leaves the reference typing's short layers after the first:
// with one lane marked all are, since computing all of them again takes no
// longer.
template <int kMath>
__device__ inline bool leaves(Carry<kMath>& g) {
  if constexpr (kMath == kRef) {
    if (any_lane(g.redo)) {
      g.redo = true;
      return true;
    }
  }
  return false;
}

// The n layers of a track again, from its input state and in the full
// form: the exception (an operand that overflows or is not finite).  128 waves,
// 20 layers, W = 32: 20.9 us; 30 with an unused lane in every block (139 where
// the short layers all came first and NaN took the calls of ref_rcp_any and
// sincosf_large).
template <int W>
__device__ inline void redo_ref(Track& t, const float* __restrict__ tb, const float* __restrict__ hb, int n) {
  // the address hidden from common-subexpression elimination: otherwise the
  // track's input would be kept in registers through all layers for this load
  asm volatile("" : "+v"(tb));
  load_track<W>(t, tb);
  const RefCarry c = ref_carry(t);
  Hit next{};
  if (0 < n) next = load_hit<W>(hb);
  for (int lay = 0; lay < n; ++lay) {
    const Hit h = next;
    if (lay + 1 < n) next = load_hit<W>(hb + (int64_t)(lay + 1) * (kHitWords * W));
    step_ref_full(t, h, c);
  }
}

// Layers [0, n) of one track whose hits start at hb (consecutive layers 9W
// words apart), with the hits of the next kDepth layers (1 or 2) in flight
// while a layer is computed; n is the same for every lane.  The loop is
// unrolled by kDepth + 1 over rotating hit buffers, so a prefetched hit is
// never copied between registers.
// No load is conditional: loads return in order and a wait counts the loads
// behind the wanted one, so after a load that may not have been issued the
// compiler waits for everything, the hits requested a moment ago included (one
// layer in two had none in flight).  Near the end the last record is read
// again instead (at most kDepth times per track), and the last layers follow
// the loop.  20 layers, W = 32: 1500 waves 19.75 -> 17.65 us FAST; 15000 waves
// 121.2 -> 118.0 FAST, 204.4 -> 200.9 REF, 198.4 -> 196.1 FP64 gain.
// At depth 1 the end has one code path for one layer left and one for two, so
// nothing is read again (of the FAST figure 119.6 -> 118.0); with the FP64 gain
// steps the second path would take 130 VGPRs, 3 waves per SIMD instead of 4
// (192.3 -> 193.2 us), and the last record is read again.
template <int W, int kMath, int kDepth>
__device__ __forceinline__ bool run_layers(Track& t, const float* __restrict__ hb, int n) {
  static_assert(kDepth == 1 || kDepth == 2, "prefetch depth 1 or 2");
  if (n <= 0) return false;
  auto at = [&](int lay) { return load_hit<W>(hb + (int64_t)(lay < n ? lay : n - 1) * (kHitWords * W)); };
  Carry<kMath> g;
  Hit a = at(0), b = at(1);
  int lay = 1;
  if constexpr (kDepth == 1) {
    layer_step<kMath, true>(t, a, g);
    if (leaves<kMath>(g)) n = 0;
    for (; lay + 2 < n; lay += 2) {  // b holds layer lay
      a = at(lay + 1);
      layer_step<kMath, false>(t, b, g);
      b = at(lay + 2);
      layer_step<kMath, false>(t, a, g);
    }
    if constexpr (kMath == kFp64Gain) {
      if (lay < n) {
        a = at(lay + 1);
        layer_step<kMath, false>(t, b, g);
        if (lay + 1 < n) layer_step<kMath, false>(t, a, g);
      }
    } else if (lay + 1 < n) {
      a = at(lay + 1);
      layer_step<kMath, false>(t, b, g);
      layer_step<kMath, false>(t, a, g);
    } else if (lay < n) {
      layer_step<kMath, false>(t, b, g);
    }
  } else {
    Hit c = at(2);
    layer_step<kMath, true>(t, a, g);
    if (leaves<kMath>(g)) n = 0;
    for (; lay + 4 < n; lay += 3) {  // b holds layer lay, c layer lay + 1
      a = at(lay + 2);
      layer_step<kMath, false>(t, b, g);
      b = at(lay + 3);
      layer_step<kMath, false>(t, c, g);
      c = at(lay + 4);
      layer_step<kMath, false>(t, a, g);
    }
    if (lay < n) {  // at most 4 layers
      a = at(lay + 2);
      layer_step<kMath, false>(t, b, g);
      b = at(lay + 3);
      if (lay + 1 < n) layer_step<kMath, false>(t, c, g);
      if (lay + 2 < n) layer_step<kMath, false>(t, a, g);
      if (lay + 3 < n) layer_step<kMath, false>(t, b, g);
    }
  }
  return marked<kMath>(t, g);
}

// Maximum of v over each group of kLanes lanes, in every lane of the group
// (every lane of the wave must be active).
template <int kLanes>
__device__ inline int group_max(int v) {
#pragma unroll
  for (int o = kLanes / 2; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o));
  return v;
}

__device__ inline int64_t lane_i64(int64_t v, int lane) {
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)((uint64_t)v >> 32), lane);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Ragged form of run_layers: every lane has its own layer count n, the loop
// runs to the wave's largest with each lane's steps masked by its own n (all
// lanes of the wave must be active).  The loads are never masked, so that
// their number is the same on every path and a wait is for the layer it needs
// only: past its block's largest count a lane reads its last record again, and
// the lanes of a block with no layers read a live block's.  A rolled loop whose
// loads were masked and moved from buffer to buffer took, 16 events (54062
// tracks) with the FP64 gain steps, 21.7 us (now 20.7), 20 events FAST 18.8
// (17.9), 4 events REF 28.8 (27.9), 300 events REF 172.7 (170.0), 500 events
// FAST 185.6 (185.5).  Two layers ahead: 187.4, 20.6.
// Two layers ahead with two layers left reading on would cost 2000 events FAST
// 0.825 ms on the queue (now 0.820; the rolled loop 0.814).
// On the queue and in the resident loop it takes registers that the rolled loop
// did not (FAST one layer ahead 99 against 93 VGPRs): with more than 16 waves
// per CU, FAST loses 1-5% (500 events 205.5 against 201 us, 200 events 86
// against 82).  Every other shape is level or gains (64 threads, 8 waves per CU
// 231 against 239), and the loop's median at 20000 events/s is 1.5-2 us less.
template <int W, int kMath, int kDepth>
__device__ __forceinline__ bool run_layers_lanes(Track& t, const float* __restrict__ hit, int64_t at, int n) {
  static_assert(kDepth == 1 || kDepth == 2, "prefetch depth 1 or 2");
  int m = group_max<(W < 64 ? W : 64)>(n);  // the block's, at most 64 lanes of it
  int most = m;
  if constexpr (W < 64) {
#pragma unroll
    for (int o = 32; o >= W; o >>= 1) most = max(most, __shfl_xor(most, o));
  }
  int nmax = __builtin_amdgcn_readfirstlane(most);
  if (nmax <= 0) return false;
  if constexpr (W < 64) {
    const int from = __builtin_ctzll(__ballot(m > 0));
    const int64_t other = lane_i64(at, from);
    const int other_m = __builtin_amdgcn_readlane(m, from);
    at = m > 0 ? at : other;
    m = m > 0 ? m : other_m;
  }
  const float* hb = hit + at;
  int loaded = 0;
  auto next = [&]() {
    const Hit h = load_hit<W>(hb);
    hb += ++loaded < m ? kHitWords * W : 0;
    return h;
  };
  Carry<kMath> g;
  Hit a = next(), b = next();
  int lay = 1;
  if constexpr (kDepth == 1) {
    if (0 < n) layer_step<kMath, true>(t, a, g);
    if (leaves<kMath>(g)) n = nmax = 0;
    for (; lay + 2 < nmax; lay += 2) {  // b holds layer lay
      a = next();
      if (lay < n) layer_step<kMath, false>(t, b, g);
      b = next();
      if (lay + 1 < n) layer_step<kMath, false>(t, a, g);
    }
    if constexpr (kMath == kFp64Gain) {  // ends as in run_layers
      if (lay < nmax) {
        a = next();
        if (lay < n) layer_step<kMath, false>(t, b, g);
        if (lay + 1 < n) layer_step<kMath, false>(t, a, g);
      }
    } else if (lay + 1 < nmax) {
      a = next();
      if (lay < n) layer_step<kMath, false>(t, b, g);
      if (lay + 1 < n) layer_step<kMath, false>(t, a, g);
    } else if (lay < n) {
      layer_step<kMath, false>(t, b, g);
    }
  } else {
    Hit c = next();
    if (0 < n) layer_step<kMath, true>(t, a, g);
    if (leaves<kMath>(g)) n = nmax = 0;
    for (; lay + 4 < nmax; lay += 3) {  // b holds layer lay, c layer lay + 1
      a = next();
      if (lay < n) layer_step<kMath, false>(t, b, g);
      b = next();
      if (lay + 1 < n) layer_step<kMath, false>(t, c, g);
      c = next();
      if (lay + 2 < n) layer_step<kMath, false>(t, a, g);
    }
    if (lay + (kMath == kFp64Gain ? 0 : 2) < nmax) {  // at most 4 layers
      a = next();
      if (lay < n) layer_step<kMath, false>(t, b, g);
      b = next();
      if (lay + 1 < n) layer_step<kMath, false>(t, c, g);
      if (lay + 2 < n) layer_step<kMath, false>(t, a, g);
      if (lay + 3 < n) layer_step<kMath, false>(t, b, g);
    } else if constexpr (kMath != kFp64Gain) {
      if (lay < n) layer_step<kMath, false>(t, b, g);
      if (lay + 1 < n) layer_step<kMath, false>(t, c, g);
    }
  }
  return marked<kMath>(t, g);
}

// ---------------------------------------------------------------------------
// fused driver pass (reference OMP:733-747 for every block at once)
// ---------------------------------------------------------------------------
template <int W, int kMath, int kDepth>
__global__ __launch_bounds__(256) void k_fused(const float* __restrict__ trk,
                                               const float* __restrict__ hit,
                                               float* __restrict__ out, int64_t ntracks,
                                               int nlayer) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ntracks) return;
  const int64_t b = g / W;
  const int l = (int)(g % W);
  Track t;
  const float* tb = trk + b * (kTrkWords * W) + l;
  const float* hb = hit + b * (int64_t)nlayer * (kHitWords * W) + l;
  load_track<W>(t, tb);
  const bool redo = run_layers<W, kMath, kDepth>(t, hb, nlayer);
  if constexpr (kMath == kRef)
    if (redo) redo_ref<W>(t, tb, hb, nlayer);
  store_track<W>(t, out + b * (kTrkWords * W) + l);
}

// ---------------------------------------------------------------------------
// ragged events: per-block descriptors, per-lane layer counts
// ---------------------------------------------------------------------------

// Work item = 64 consecutive track slots of the descriptor table (one wave):
// slot s is lane s % W of descriptor s / W.  Each lane runs its own layer
// count; the wave's loop runs to the largest.  All 64 lanes of the wave must
// be active (slots past the table take part with no layers).
template <int W, int kMath, int kPrefetch>
__device__ __forceinline__ void ragged_item(const float* __restrict__ trk, const float* __restrict__ hit,
                                   float* __restrict__ out, const int32_t* __restrict__ lane_nlay,
                                   const BlockDesc* __restrict__ blocks, int64_t nblocks, int64_t item, int lane) {
  const int64_t slot = item * 64 + lane;
  const int64_t di = slot / W;
  const int l = (int)(slot % W);
  const bool valid = di < nblocks;
  Track t{};
  int n = 0;
  int64_t ho = 0;
  const float* tb = trk;
  BlockDesc d{};
  if (valid) {
    d = blocks[di];
    tb = trk + d.trk_block * (kTrkWords * W) + l;
    load_track<W, true>(t, tb);
    n = lane_nlay[d.trk_block * W + l];
    n = n < d.nlayer ? n : d.nlayer;
    n = n > 0 ? n : 0;
    ho = d.hit_block * (kHitWords * W) + l;
  }
  const bool redo = run_layers_lanes<W, kMath, kPrefetch>(t, hit, ho, n);
  if constexpr (kMath == kRef)
    if (valid && redo) redo_ref<W>(t, tb, hit + ho, n);
  if (valid) store_track<W>(t, out + d.out_block * (kTrkWords * W) + l);
}

// Persistent form: the items are cut into chunks of `claim` consecutive items.
// Wave w of the grid (nwaves in all) computes chunk w first, with no atomic:
// a counter that every wave hit at start would serialise thousands of atomics
// before the first item is computed.  The chunks after those are striped over
// ns = min(kQueueStripes, workgroups) counters: a wave of workgroup g (stripe
// s = g % ns) takes chunk nwaves + s + ns * atomicAdd(counter[s], 1) until it
// is handed a chunk past the end (every wave reaches that exit).  A single
// counter serialises its atomics where they meet (a few times 1e7 per
// second); striping spreads them, so that one or two items per claim keep the
// load even at the end without the counter becoming the limit.  The atomic is
// issued when the last item of the current chunk starts, so its round trip
// overlaps that item; a wave never holds a whole chunk in reserve while others
// run dry at the end.  Each stripe hands out its chunk indexes in order, once
// each, and every workgroup runs (none waits on another), so every item is
// computed exactly once.  The counters start at 0 (k_reset_counter runs first
// on the same stream).
// FP64 gain: at most 128 VGPRs (4 waves per SIMD instead of 3).
template <int W, int kMath, int kPrefetch>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kMath == kFp64Gain ? 4 : 1))) void
k_ragged_persistent(const float* __restrict__ trk, const float* __restrict__ hit, float* __restrict__ out,
                    const int32_t* __restrict__ lane_nlay, const BlockDesc* __restrict__ blocks, int64_t nblocks,
                    unsigned* __restrict__ counter, int claim) {
  const int64_t nitems = (nblocks * W + 63) / 64;
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x / 64);
  const int ns = gridDim.x < (unsigned)kQueueStripes ? (int)gridDim.x : kQueueStripes;
  const int stripe = (int)(blockIdx.x % (unsigned)ns);
  unsigned* ctr = counter + stripe * kQueueStride;
  int64_t chunk = (int64_t)blockIdx.x * (blockDim.x / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  while (chunk * claim < nitems) {
    const int64_t first = chunk * claim;
    const int64_t last = first + claim < nitems ? first + claim : nitems;
    unsigned next = 0;
    for (int64_t item = first; item < last; ++item) {
      if (item == last - 1 && lane == 0) next = atomicAdd(ctr, 1u);
      int lane_i = lane;
      // the lane index hidden from loop-invariant code motion, so that
      // lane-dependent values are not hoisted out of the item loop into
      // registers held across all of it (10 VGPRs in every mode)
      asm volatile("" : "+v"(lane_i));
      ragged_item<W, kMath, kPrefetch>(trk, hit, out, lane_nlay, blocks, nblocks, item, lane_i);
    }
    // lane 0's claim read into a scalar: the chunk index, and with it the
    // loop's control, stay wave-uniform scalars
    chunk = nwaves + stripe + (int64_t)ns * (int64_t)__builtin_amdgcn_readlane(next, 0);
  }
}

// One-shot form: one wave per item (the hardware dispatcher hands out the
// items, in descriptor order).
template <int W, int kMath, int kPrefetch>
__global__ __launch_bounds__(256) void k_ragged_oneshot(const float* __restrict__ trk,
                                                        const float* __restrict__ hit,
                                                        float* __restrict__ out,
                                                        const int32_t* __restrict__ lane_nlay,
                                                        const BlockDesc* __restrict__ blocks,
                                                        int64_t nblocks) {
  const int64_t nitems = (nblocks * W + 63) / 64;
  const int64_t item = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
  if (item >= nitems) return;
  ragged_item<W, kMath, kPrefetch>(trk, hit, out, lane_nlay, blocks, nblocks, item, threadIdx.x & 63);
}

// ---------------------------------------------------------------------------
// device-resident serving loop
// ---------------------------------------------------------------------------
// One persistent launch serves requests as the host publishes them: the host
// writes work items (ServeItem, 64 track slots of one request) into a ring in
// coherent pinned host memory and advances ServeCtl::tail; wave 0 of
// workgroup 0 (the dispatcher) polls that word over PCIe and copies it into
// device memory (ServeDev::dev_tail), where the worker waves wait for it.  A
// worker claims item indexes in order (ServeDev::head), computes the item as
// the ragged pass does, and counts it against its request; the worker that
// completes a request writes a completion record into host memory.
// Termination: the dispatcher stops when the host sets ServeCtl::stop or when
// the host's heartbeat has not moved for idle_ticks (100 MHz s_memrealtime
// ticks); it then sets dev_stop, and every worker ends once the item it holds
// is past the last published one.  Every wait loop therefore ends.
// Memory: the loop takes no acquire or release at agent or system scope: on
// this GPU those write back or invalidate the L2 of the wave's XCD, and
// thousands of waiting waves would keep every L2 flushing.  Instead
//  - counters and flags are atomics (coherent at the scope they name, so
//    every poll reads the current value);
//  - item fields are read with system-scope loads straight from host memory
//    (the host writes an item before its tail; a worker reads the item only
//    after it has seen the tail);
//  - results are written with system-scope (write-through) stores, and a wave
//    waits for its stores to complete before it counts its item, so a
//    request's results are in memory before its completion is counted, and
//    the completion record's fields before its seq word.

__device__ inline uint32_t lane0_u32(uint32_t v) { return __builtin_amdgcn_readlane(v, 0); }
__device__ inline uint64_t lane0_u64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, 0);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), 0);
  return ((uint64_t)hi << 32) | lo;
}

template <class T>
__device__ inline T sys_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
template <class T>
__device__ inline T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ inline void sys_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// Waits until this wave's vector memory operations have completed
// (s_waitcnt vmcnt(0); gfx9 encoding: vmcnt 0, expcnt 7, lgkmcnt 15): a store
// is then acknowledged at the scope it was issued with.  No cache operation.
__device__ inline void wait_stores() { __builtin_amdgcn_s_waitcnt(0x0F70); }

template <int W>
__device__ inline void store_track_through(const Track& t, float* __restrict__ ob) {
  uint32_t* o = reinterpret_cast<uint32_t*>(ob);
#pragma unroll
  for (int e = 0; e < 6; ++e) sys_store(o + e * W, __builtin_bit_cast(uint32_t, t.p[e]));
#pragma unroll
  for (int e = 0; e < 21; ++e) sys_store(o + (6 + e) * W, __builtin_bit_cast(uint32_t, t.P[e]));
  sys_store(o + 27 * W, (uint32_t)t.q);
}

__device__ void serve_dispatch(const ServeLaunch& a) {
  uint64_t seen = ~0ull;
  uint64_t hb = lane0_u64(sys_load(&a.ctl->heartbeat));
  uint64_t t_hb = __builtin_amdgcn_s_memrealtime();
  bool run = true;
  while (run) {
    const uint64_t t = lane0_u64(sys_load(&a.ctl->tail));
    if (t != seen) {
      __hip_atomic_store(&a.dev->dev_tail, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      seen = t;
    }
    const uint32_t stop = lane0_u32(sys_load(&a.ctl->stop));
    const uint64_t h = lane0_u64(sys_load(&a.ctl->heartbeat));
    const uint64_t now = __builtin_amdgcn_s_memrealtime();
    if (h != hb) {
      hb = h;
      t_hb = now;
    }
    run = stop == 0u && now - t_hb <= a.idle_ticks;
    if (run) __builtin_amdgcn_s_sleep(2);
  }
  // the final tail is stored before the stop flag, and the host learns that
  // this launch's dispatcher has left
  wait_stores();
  __hip_atomic_store(&a.dev->dev_stop, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  sys_store(&a.ctl->exited, lane0_u32(sys_load(&a.ctl->epoch)));
}

template <int W, int kMath, int kPrefetch>
__device__ __forceinline__ void serve_item(const ServeLaunch& a, uint64_t k, int lane) {
  const ServeItem* it = a.items + (int64_t)(k % (uint64_t)a.item_cap);
  const int di = W <= 64 ? lane / W : 0;
  // The whole 144-byte record in one load instruction, one round trip over
  // PCIe: lane j < 18 reads the record's 8-byte word j (18 lanes of
  // consecutive words: a few PCIe requests, where a load per field costs one
  // request each).  Each lane then takes its descriptor's fields from the
  // lanes that hold them: desc[d] is words 4d .. 4d + 3 (trk_block,
  // hit_block, out_block, nlayer | event), the header words 16 (ndesc | half)
  // and 17 (req_slot | req_items).  A padding descriptor is read too: it lies
  // inside the record.
  static_assert(sizeof(ServeItem) == 18 * sizeof(uint64_t), "serve item: 18 words");
  static_assert(offsetof(ServeItem, ndesc) == 16 * 8 && offsetof(ServeItem, req_slot) == 17 * 8, "header words");
  uint64_t word = 0;
  if (lane < 18) word = sys_load(reinterpret_cast<const uint64_t*>(it) + lane);
  const int wlo = (int)(uint32_t)word, whi = (int)(uint32_t)(word >> 32);
  auto pick = [&](int j) -> int64_t {
    return (int64_t)(((uint64_t)(uint32_t)__shfl(whi, j) << 32) | (uint32_t)__shfl(wlo, j));
  };
  const int64_t tb = pick(4 * di);
  const int64_t hblk = pick(4 * di + 1);
  const int64_t ob = pick(4 * di + 2);
  const int nl = __shfl(wlo, 4 * di + 3);
  const int ndesc = (int)__builtin_amdgcn_readlane((uint32_t)wlo, 16);
  const int half = (int)__builtin_amdgcn_readlane((uint32_t)whi, 16);
  const int req_slot = (int)__builtin_amdgcn_readlane((uint32_t)wlo, 17);
  const uint32_t req_items = __builtin_amdgcn_readlane((uint32_t)whi, 17);
  const int l = W <= 64 ? lane % W : half * 64 + lane;
  const bool valid = di < ndesc;
  Track t{};
  int n = 0;
  int64_t ho = 0;
  const float* tin = a.trk;
  if (valid) {
    tin = a.trk + tb * (kTrkWords * W) + l;
    load_track<W, true>(t, tin);
    n = a.lanes[tb * W + l];
    n = n < nl ? n : nl;
    n = n > 0 ? n : 0;
    ho = hblk * (kHitWords * W) + l;
  }
  const bool redo = run_layers_lanes<W, kMath, kPrefetch>(t, a.hit, ho, n);
  if constexpr (kMath == kRef)
    if (valid && redo) redo_ref<W>(t, tin, a.hit + ho, n);
  if (valid) store_track_through<W>(t, a.out + ob * (kTrkWords * W) + l);
  wait_stores();
  if (lane == 0) {
    const uint32_t old =
        __hip_atomic_fetch_add(&a.done[req_slot], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old + 1u == req_items) {
      // the request's last item: reset its counter for the slot's next
      // request and report it
      __hip_atomic_store(&a.done[req_slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint64_t c =
          __hip_atomic_fetch_add(&a.dev->comp_tail, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      ServeCompletion* r = a.comps + (int64_t)(c % (uint64_t)a.comp_cap);
      sys_store(&r->req_slot, req_slot);
      wait_stores();
      sys_store(&r->seq, c + 1);
    }
  }
}

// Claims the item indexes of its workgroup's stripe in order and computes
// them; ends once it holds an index past the last published item after the
// dispatcher has stopped.  Every stripe has workers (the grid has at least two
// workgroups per stripe, dispatched in order), so every published item is
// claimed.  The
// next index is claimed (by lane 0) while the current item starts, as in the
// persistent ragged kernel: the claim's round trip overlaps the item, and the
// lane-0 branch sits inside the loop body, never on the edge back to the
// loop's head (where the compiler may split a loop whose back edges differ by
// lane, letting the other lanes run on without lane 0 and its claim).  Every
// loop condition is a wave-uniform value (lane 0's, read into a scalar).
template <int W, int kMath, int kPrefetch>
__device__ void serve_work(const ServeLaunch& a, int lane) {
  const uint64_t stripe = blockIdx.x % kServeStripes;
  uint64_t* head = &a.dev->head[stripe][0];
  uint64_t claimed = 0;
  if (lane == 0) claimed = __hip_atomic_fetch_add(head, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  uint64_t k = lane0_u64(claimed) * kServeStripes + stripe;
  bool have = true;
  while (have) {
    bool wait = true;
    while (wait) {
      if (k < lane0_u64(agent_load(&a.dev->dev_tail))) {
        wait = false;
      } else if (lane0_u32(agent_load(&a.dev->dev_stop))) {
        // stop comes after the final tail: an item past it is never published
        have = k < lane0_u64(agent_load(&a.dev->dev_tail));
        wait = false;
      } else {
        __builtin_amdgcn_s_sleep(32);
      }
    }
    if (have) {
      uint64_t next = 0;
      if (lane == 0) next = __hip_atomic_fetch_add(head, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      int lane_i = lane;
      asm volatile("" : "+v"(lane_i));  // as in the persistent ragged pass
      serve_item<W, kMath, kPrefetch>(a, k, lane_i);
      k = lane0_u64(next) * kServeStripes + stripe;
    }
  }
}

__global__ void k_serve_reset(ServeDev* dev) {
  const uint64_t t = dev->dev_tail;
  const int j = threadIdx.x;
  if (j < kServeStripes) dev->head[j][0] = t > (uint64_t)j ? (t - j + kServeStripes - 1) / kServeStripes : 0;
  if (j == 0) dev->dev_stop = 0u;
}

template <int W, int kMath, int kPrefetch>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kMath == kFp64Gain ? 4 : 1))) void
k_serve_resident(ServeLaunch a) {
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    serve_dispatch(a);
    return;
  }
  serve_work<W, kMath, kPrefetch>(a, threadIdx.x & 63);
}

__global__ void k_reset_counter(unsigned* counter) {
  if (blockIdx.x == 0 && threadIdx.x < kQueueStripes) counter[threadIdx.x * kQueueStride] = 0u;
}

// ---------------------------------------------------------------------------
// per-function kernels (reference propagateToZ / KalmanUpdate_v2 on blocks)
// ---------------------------------------------------------------------------
template <int W, int kMath>
__global__ __launch_bounds__(256) void k_propagate(const float* inErr, const float* inPar,
                                                   const int32_t* inChg, const float* msP,
                                                   float* outErr, float* outPar,
                                                   int64_t ntracks, int64_t ts, int64_t hs) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ntracks) return;
  const int64_t b = g / W;
  const int l = (int)(g % W);
  Track t;
  const int64_t o = b * ts + l;
#pragma unroll
  for (int e = 0; e < 21; ++e) t.P[e] = inErr[o + e * W];
#pragma unroll
  for (int e = 0; e < 6; ++e) t.p[e] = inPar[o + e * W];
  t.q = inChg[o];
  const float hz = msP[b * hs + 2 * W + l];
  if constexpr (kMath == kRef) {
    bool unused = false;
    propagate_ref<false>(t, hz, ref_carry(t), unused);
  } else
    propagate_fast<false, kMath == kFp64Gain>(t, hz);
#pragma unroll
  for (int e = 0; e < 21; ++e) outErr[o + e * W] = t.P[e];
#pragma unroll
  for (int e = 0; e < 6; ++e) outPar[o + e * W] = t.p[e];
}

template <int W, int kMath>
__global__ __launch_bounds__(256) void k_update(float* trkErr, float* inPar, const float* hitErr,
                                                const float* msP, int64_t ntracks, int64_t ts,
                                                int64_t hs) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ntracks) return;
  const int64_t b = g / W;
  const int l = (int)(g % W);
  Track t;
  const int64_t o = b * ts + l;
#pragma unroll
  for (int e = 0; e < 21; ++e) t.P[e] = trkErr[o + e * W];
#pragma unroll
  for (int e = 0; e < 6; ++e) t.p[e] = inPar[o + e * W];
  t.q = 0;
  const int64_t ho = b * hs + l;
  Hit h;
  h.x = msP[ho];
  h.y = msP[ho + W];
  h.z = msP[ho + 2 * W];
  h.xx = hitErr[ho];
  h.xy = hitErr[ho + W];
  h.yy = hitErr[ho + 2 * W];
  if constexpr (kMath == kRef) {
    bool unused = false;
    update_ref<false>(t, h, unused);
  } else if constexpr (kMath == kFast)
    update_fast<false>(t, h);
  else
    update_fp64gain<false>(t, h);
#pragma unroll
  for (int e = 0; e < 21; ++e) trkErr[o + e * W] = t.P[e];
#pragma unroll
  for (int e = 0; e < 6; ++e) inPar[o + e * W] = t.p[e];
}

// KalmanUpdate v1 (OMP:375-501) on blocks, in place; kFixed selects the
// textbook form.  hitErr: the 6 hit covariance words of each lane.
template <int W, bool kFixed>
__global__ __launch_bounds__(256) void k_update_v1(float* trkErr, float* inPar, const float* hitErr,
                                                   const float* msP, int64_t ntracks, int64_t ts,
                                                   int64_t hs) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ntracks) return;
  const int64_t b = g / W;
  const int l = (int)(g % W);
  Track t;
  const int64_t o = b * ts + l;
#pragma unroll
  for (int e = 0; e < 21; ++e) t.P[e] = trkErr[o + e * W];
#pragma unroll
  for (int e = 0; e < 6; ++e) t.p[e] = inPar[o + e * W];
  t.q = 0;
  const int64_t ho = b * hs + l;
  float hc[6];
#pragma unroll
  for (int e = 0; e < 6; ++e) hc[e] = hitErr[ho + e * W];
  if constexpr (kFixed)
    update_v1_fixed(t, hc, msP[ho], msP[ho + W], msP[ho + 2 * W]);
  else
    update_v1_ref(t, hc, msP[ho], msP[ho + W]);
#pragma unroll
  for (int e = 0; e < 21; ++e) trkErr[o + e * W] = t.P[e];
#pragma unroll
  for (int e = 0; e < 6; ++e) inPar[o + e * W] = t.p[e];
}

// ---------------------------------------------------------------------------
// report statistics (OMP:758-851), deterministic fixed-order reduction
// ---------------------------------------------------------------------------
// One launch over the tracks.  A workgroup takes kSumTracks tracks per thread,
// sums them, forms the means of its own tracks and, from the values still in
// registers, the sums of squares about those means; its partial results go to
// memory.  The workgroup that finishes last combines the partials in their
// fixed order: means from the sums, then
//   sum (x - mean)^2 = sum over workgroups of M2 + n (mean of the workgroup - mean)^2,
// whose terms are all positive, so it is as accurate as the reference's second
// pass over the tracks without one.  It writes the result into host memory
// with a sequence number behind it, which the host waits for.
// Bound: latency.  960000 tracks (23 MB read): 75 us per call as two passes
// over the tracks, two final launches and a copy back; 28 us now (20 us of it
// the kernel: loads, the divisions in double, four sums over a workgroup, the
// last of which nothing overlaps; 4 or 2 tracks per thread: 29 and 33 us).
constexpr int kSumThreads = 256;
constexpr int kSumTracks = 8;
constexpr int kSumMeans = 9;  // x y z dx dy dz pt phi theta
constexpr int kSumRms = 6;    // x y z dx dy dz
constexpr int kSumVals = kSumMeans + kSumRms + 3;  // sums, squares about the workgroup's means, counts

// Sum over each row of 16 lanes, the same in all of them (all active).
template <int kCtrl>
__device__ inline double add_dpp(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kCtrl, 0xf, 0xf, true);
  return v + __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ inline double row_sum(double v) {
  v = add_dpp<0xB1>(v);     // lanes 1 0 3 2 of each four
  v = add_dpp<0x4E>(v);     // lanes 2 3 0 1
  v = add_dpp<0x141>(v);    // mirrored within 8
  return add_dpp<0x140>(v); // mirrored within 16
}

// Adds v over the workgroup; every thread gets the totals.  The values go
// through LDS once, 16 threads then add up each: 60 instructions per thread
// for 12 values, where a butterfly of shuffles takes 140 LDS operations and
// one of data-parallel primitives 280 instructions.
constexpr int kSumRow = kSumThreads + 16;  // padded: rows of 16 threads read different banks
struct SumLds {
  double v[(kSumMeans + 3) * kSumRow];
  double total[kSumMeans + 3];
};
template <int kN>
__device__ inline void block_sum(double (&v)[kN], SumLds& lds) {
  const int t = threadIdx.x;
#pragma unroll
  for (int k = 0; k < kN; ++k) lds.v[k * kSumRow + t] = v[k];
  __syncthreads();
  const int k0 = t / 16;
  if (k0 < kN) {  // whole rows of 16 lanes
    double s = 0.;
#pragma unroll
    for (int i = 0; i < 16; ++i) s += lds.v[k0 * kSumRow + i * 16 + t % 16];
    s = row_sum(s);
    if (t % 16 == 0) lds.total[k0] = s;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kN; ++k) v[k] = lds.total[k];
  __syncthreads();
}

// Counts the caller in; true for the last of n, which sets the counter back.
__device__ inline bool last_of(unsigned* counter, unsigned n) {
  if (__hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u != n) return false;
  __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

template <int W>
__global__ __launch_bounds__(kSumThreads) void k_summary(const float* __restrict__ out, int64_t nb, int64_t ntrks,
                                                         int64_t total, double hx, double hy, double hz,
                                                         double* part, unsigned* done, SummaryResult* res,
                                                         uint64_t seq) {
  __shared__ SumLds lds;
  __shared__ double own[kSumVals];
  __shared__ unsigned last;
  // a thread's tracks are kSumThreads apart, all their words loaded at once
  const int64_t idx0 = (int64_t)blockIdx.x * (kSumThreads * kSumTracks) + threadIdx.x;
  int64_t ie, it;
  if (total < (int64_t)1 << 31) {  // a 64-bit division takes a hundred instructions
    ie = (uint32_t)idx0 / (uint32_t)ntrks;
    it = (uint32_t)idx0 % (uint32_t)ntrks;
  } else {
    ie = idx0 / ntrks;
    it = idx0 % ntrks;
  }
  float w[kSumTracks][6];
#pragma unroll
  for (int k = 0; k < kSumTracks; ++k) {
    if (idx0 + k * kSumThreads < total) {
      const float* blk = out + ((it / W) + nb * ie) * (int64_t)(kTrkWords * W) + it % W;
#pragma unroll
      for (int e = 0; e < 6; ++e) w[k][e] = blk[e * W];
    }
    it += kSumThreads;
    if (it >= ntrks) {
      if (it < 2 * ntrks) {
        it -= ntrks;
        ++ie;
      } else {
        ie += it / ntrks;
        it %= ntrks;
      }
    }
  }
  double x[kSumTracks][kSumRms];
  bool good[kSumTracks];
  double v[kSumMeans + 3];  // sums of the means' values, then nnans, nfail, ngood
#pragma unroll
  for (int k = 0; k < kSumMeans + 3; ++k) v[k] = 0.;
#pragma unroll
  for (int k = 0; k < kSumTracks; ++k) {
    good[k] = false;
    if (idx0 + k * kSumThreads < total) {
      const double X = w[k][0], Y = w[k][1], Z = w[k][2], ipt = w[k][3], phi = w[k][4], theta = w[k][5];
      const double pt = 1. / ipt;
      if (!isfinite(X) || !isfinite(Y) || !isfinite(Z) || !isfinite(pt) || !isfinite(phi) || !isfinite(theta)) {
        v[kSumMeans] += 1.;
      } else if (fabs(X - hx) > fabs(hx) || fabs(Y - hy) > fabs(hy) || fabs(Z - hz) > fabs(hz) ||
                 fabs(pt - 12.) > 12. || fabs(phi - 1.3) > 1.3 || fabs(theta - 2.8) > 2.8) {
        // the window |(x - hx) / hx| > 1 without its division: a quotient of
        // doubles rounds above 1 exactly when the numerator is the larger
        v[kSumMeans + 1] += 1.;
      } else {
        good[k] = true;
        x[k][0] = X;
        x[k][1] = Y;
        x[k][2] = Z;
        x[k][3] = (X - hx) / X;
        x[k][4] = (Y - hy) / Y;
        x[k][5] = (Z - hz) / Z;
#pragma unroll
        for (int e = 0; e < kSumRms; ++e) v[e] += x[k][e];
        v[6] += pt;
        v[7] += phi;
        v[8] += theta;
        v[kSumMeans + 2] += 1.;
      }
    }
  }
  block_sum(v, lds);
  double m2[kSumRms];
  const double n = v[kSumMeans + 2];
#pragma unroll
  for (int e = 0; e < kSumRms; ++e) {
    const double mean = n > 0. ? v[e] / n : 0.;
    m2[e] = 0.;
#pragma unroll
    for (int k = 0; k < kSumTracks; ++k)
      if (good[k]) m2[e] += (x[k][e] - mean) * (x[k][e] - mean);
  }
  block_sum(m2, lds);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < kSumMeans + 3; ++k) own[k] = v[k];
#pragma unroll
    for (int e = 0; e < kSumRms; ++e) own[kSumMeans + 3 + e] = m2[e];
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    // one store instruction for the partials, written through to where every
    // XCD sees them, and complete before the workgroup is counted
    if (threadIdx.x < kSumVals)
      __hip_atomic_store(reinterpret_cast<uint64_t*>(part + (int64_t)blockIdx.x * kSumVals) + threadIdx.x,
                         __builtin_bit_cast(uint64_t, own[threadIdx.x]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    wait_stores();
  }
  if (threadIdx.x == 0) {
    // counted in two steps: one counter for all workgroups would take them one
    // after another (about 15 ns each)
    const unsigned ns = gridDim.x < (unsigned)kSumStripes ? gridDim.x : kSumStripes;
    const unsigned stripe = blockIdx.x % ns;
    last = last_of(done + (1 + stripe) * kSumStride, (gridDim.x - stripe + ns - 1) / ns) && last_of(done, ns);
  }
  __syncthreads();
  if (!last) return;

  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // no partial is read from a cache filled before
  const int64_t groups = gridDim.x;
#pragma unroll
  for (int k = 0; k < kSumMeans + 3; ++k) v[k] = 0.;
  for (int64_t g = threadIdx.x; g < groups; g += kSumThreads) {
#pragma unroll
    for (int k = 0; k < kSumMeans + 3; ++k) v[k] += part[g * kSumVals + k];
  }
  block_sum(v, lds);
  const double ngood = v[kSumMeans + 2];
#pragma unroll
  for (int e = 0; e < kSumRms; ++e) m2[e] = 0.;
  for (int64_t g = threadIdx.x; g < groups; g += kSumThreads) {
    const double* p = part + g * kSumVals;
    const double ng = p[kSumMeans + 2];
    if (ng > 0.) {
#pragma unroll
      for (int e = 0; e < kSumRms; ++e) {
        const double d = p[e] / ng - v[e] / ngood;
        m2[e] += p[kSumMeans + 3 + e] + ng * (d * d);
      }
    }
  }
  block_sum(m2, lds);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < kSumMeans; ++k) own[k] = v[k] / ngood;
#pragma unroll
    for (int k = 0; k < 3; ++k) own[kSumMeans + k] = v[kSumMeans + k];
#pragma unroll
    for (int e = 0; e < kSumRms; ++e) own[kSumMeans + 3 + e] = (double)sqrtf((float)(m2[e] / ngood));
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    if (threadIdx.x < kSumVals) sys_store(&res->bits[threadIdx.x], __builtin_bit_cast(uint64_t, own[threadIdx.x]));
    wait_stores();
    if (threadIdx.x == 0) sys_store(&res->seq, seq);
  }
}

// sin and cos of the reference-typing mode (sincosf_glibc) for the float bit
// patterns first, first+1, ... (n of them, n <= 2^32 - first).
__global__ __launch_bounds__(256) void k_sincosf_range(uint32_t first, int64_t n, float* __restrict__ s,
                                                       float* __restrict__ c) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float y = __builtin_bit_cast(float, (uint32_t)(first + (uint64_t)i));
  float sv, cv;
  sincosf_glibc(y, &sv, &cv);
  s[i] = sv;
  c[i] = cv;
}

template <typename F>
hipError_t dispatch_width(int width, F&& f) {
  switch (width) {
    case 16: return f(std::integral_constant<int, 16>{});
    case 32: return f(std::integral_constant<int, 32>{});
    case 64: return f(std::integral_constant<int, 64>{});
    case 128: return f(std::integral_constant<int, 128>{});
  }
  return hipErrorInvalidValue;
}

template <typename F>
hipError_t dispatch_math(int math, F&& f) {
  switch (math) {
    case kFast: return f(std::integral_constant<int, kFast>{});
    case kRef: return f(std::integral_constant<int, kRef>{});
    case kFp64Gain: return f(std::integral_constant<int, kFp64Gain>{});
  }
  return hipErrorInvalidValue;
}

inline int64_t grid_for(int64_t n, int tpw) { return (n + tpw - 1) / tpw; }

}  // namespace

hipError_t launch_fused(const float* trk, const float* hit, float* out, int64_t nblocks, int nlayer,
                        int width, int math, const LaunchCfg& cfg, hipStream_t s) {
  const int64_t ntracks = nblocks * width;
  if (ntracks == 0) return hipSuccess;
  const int tpw = cfg.tracks_per_wg;
  return dispatch_width(width, [&](auto wc) {
    return dispatch_math(math, [&](auto mc) {
      constexpr int W = decltype(wc)::value, M = decltype(mc)::value;
      const int depth = cfg.hit_stage ? cfg.hit_stage : default_hit_stage(math, ntracks, cfg.cus);
      if (depth == 1)
        hipLaunchKernelGGL((k_fused<W, M, 1>), dim3((unsigned)grid_for(ntracks, tpw)), dim3(tpw), 0, s,
                           trk, hit, out, ntracks, nlayer);
      else
        hipLaunchKernelGGL((k_fused<W, M, 2>), dim3((unsigned)grid_for(ntracks, tpw)), dim3(tpw), 0, s,
                           trk, hit, out, ntracks, nlayer);
      return hipGetLastError();
    });
  });
}

hipError_t launch_propagate(const float* inErr, const float* inPar, const int32_t* inChg,
                            const float* msP, float* outErr, float* outPar, int64_t nblocks,
                            int64_t ts, int64_t hs, int width, int math, const LaunchCfg& cfg,
                            hipStream_t s) {
  const int64_t ntracks = nblocks * width;
  if (ntracks == 0) return hipSuccess;
  const int tpw = cfg.tracks_per_wg;
  return dispatch_width(width, [&](auto wc) {
    return dispatch_math(math, [&](auto mc) {
      constexpr int W = decltype(wc)::value, M = decltype(mc)::value;
      hipLaunchKernelGGL((k_propagate<W, M>), dim3((unsigned)grid_for(ntracks, tpw)), dim3(tpw), 0,
                         s, inErr, inPar, inChg, msP, outErr, outPar, ntracks, ts, hs);
      return hipGetLastError();
    });
  });
}

hipError_t launch_update(float* trkErr, float* inPar, const float* hitErr, const float* msP,
                         int64_t nblocks, int64_t ts, int64_t hs, int width, int math,
                         const LaunchCfg& cfg, hipStream_t s) {
  const int64_t ntracks = nblocks * width;
  if (ntracks == 0) return hipSuccess;
  const int tpw = cfg.tracks_per_wg;
  return dispatch_width(width, [&](auto wc) {
    return dispatch_math(math, [&](auto mc) {
      constexpr int W = decltype(wc)::value, M = decltype(mc)::value;
      hipLaunchKernelGGL((k_update<W, M>), dim3((unsigned)grid_for(ntracks, tpw)), dim3(tpw), 0, s,
                         trkErr, inPar, hitErr, msP, ntracks, ts, hs);
      return hipGetLastError();
    });
  });
}

hipError_t launch_update_v1(float* trkErr, float* inPar, const float* hitErr, const float* msP, int64_t nblocks,
                            int64_t ts, int64_t hs, int width, bool fixed, const LaunchCfg& cfg, hipStream_t s) {
  const int64_t ntracks = nblocks * width;
  if (ntracks == 0) return hipSuccess;
  const int tpw = cfg.tracks_per_wg;
  return dispatch_width(width, [&](auto wc) {
    constexpr int W = decltype(wc)::value;
    if (fixed)
      hipLaunchKernelGGL((k_update_v1<W, true>), dim3((unsigned)grid_for(ntracks, tpw)), dim3(tpw), 0, s, trkErr,
                         inPar, hitErr, msP, ntracks, ts, hs);
    else
      hipLaunchKernelGGL((k_update_v1<W, false>), dim3((unsigned)grid_for(ntracks, tpw)), dim3(tpw), 0, s, trkErr,
                         inPar, hitErr, msP, ntracks, ts, hs);
    return hipGetLastError();
  });
}

int ragged_persistent_groups_per_cu(int width, int math, int prefetch, int tpw) {
  static std::mutex mu;
  static std::map<std::array<int, 4>, int> cache;
  const std::array<int, 4> key{width, math, prefetch >= 2 ? 2 : 1, tpw};
  std::lock_guard<std::mutex> lock(mu);
  const auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  int n = 0;
  const hipError_t e = dispatch_width(width, [&](auto wc) {
    return dispatch_math(math, [&](auto mc) {
      constexpr int W = decltype(wc)::value, M = decltype(mc)::value;
      const void* k = prefetch >= 2 ? reinterpret_cast<const void*>(&k_ragged_persistent<W, M, 2>)
                                    : reinterpret_cast<const void*>(&k_ragged_persistent<W, M, 1>);
      return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, tpw, 0);
    });
  });
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  cache.emplace(key, n);
  return n;
}

hipError_t launch_ragged(const float* trk, const float* hit, float* out, const int32_t* lane_nlay,
                         const BlockDesc* blocks, int64_t nblocks, int width, int math, bool persistent,
                         int prefetch, int tpw, int64_t grid, int claim, unsigned* counter, hipStream_t s) {
  const int64_t nitems = (nblocks * width + 63) / 64;
  if (nitems == 0) return hipSuccess;
  return dispatch_width(width, [&](auto wc) {
    return dispatch_math(math, [&](auto mc) {
      constexpr int W = decltype(wc)::value, M = decltype(mc)::value;
      if (!persistent) {
        const dim3 grid1((unsigned)grid_for(nitems * 64, tpw));
        if (prefetch >= 2)
          hipLaunchKernelGGL((k_ragged_oneshot<W, M, 2>), grid1, dim3(tpw), 0, s, trk, hit, out, lane_nlay, blocks,
                             nblocks);
        else
          hipLaunchKernelGGL((k_ragged_oneshot<W, M, 1>), grid1, dim3(tpw), 0, s, trk, hit, out, lane_nlay, blocks,
                             nblocks);
        return hipGetLastError();
      }
      hipLaunchKernelGGL(k_reset_counter, dim3(1), dim3(64), 0, s, counter);
      const int64_t items_per_wg = (int64_t)(tpw / 64) * claim;
      int64_t g = grid > 0 ? grid : 1;
      g = std::min<int64_t>(g, (nitems + items_per_wg - 1) / items_per_wg);
      if (prefetch >= 2)
        hipLaunchKernelGGL((k_ragged_persistent<W, M, 2>), dim3((unsigned)g), dim3(tpw), 0, s, trk, hit, out,
                           lane_nlay, blocks, nblocks, counter, claim);
      else
        hipLaunchKernelGGL((k_ragged_persistent<W, M, 1>), dim3((unsigned)g), dim3(tpw), 0, s, trk, hit, out,
                           lane_nlay, blocks, nblocks, counter, claim);
      return hipGetLastError();
    });
  });
}

hipError_t launch_serve_reset(ServeDev* dev, hipStream_t s) {
  hipLaunchKernelGGL(k_serve_reset, dim3(1), dim3(64), 0, s, dev);
  return hipGetLastError();
}

hipError_t launch_serve_resident(const ServeLaunch& a, int width, int math, int prefetch, int tpw, int64_t grid,
                                 hipStream_t s) {
  if (grid < 2 * kServeStripes) return hipErrorInvalidValue;  // every stripe needs workers
  return dispatch_width(width, [&](auto wc) {
    return dispatch_math(math, [&](auto mc) {
      constexpr int W = decltype(wc)::value, M = decltype(mc)::value;
      if (prefetch >= 2)
        hipLaunchKernelGGL((k_serve_resident<W, M, 2>), dim3((unsigned)grid), dim3(tpw), 0, s, a);
      else
        hipLaunchKernelGGL((k_serve_resident<W, M, 1>), dim3((unsigned)grid), dim3(tpw), 0, s, a);
      return hipGetLastError();
    });
  });
}

hipError_t launch_sincosf_range(uint32_t first, int64_t n, float* s, float* c, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sincosf_range, dim3((unsigned)grid_for(n, 256)), dim3(256), 0, st, first, n, s, c);
  return hipGetLastError();
}

size_t summary_scratch_doubles(int64_t nevts, int64_t ntrks) {
  return (size_t)grid_for(nevts * ntrks, kSumThreads * kSumTracks) * kSumVals;
}

hipError_t launch_summary(const float* out, int64_t nevts, int64_t nb, int width, int64_t ntrks,
                          double hx, double hy, double hz, double* part, unsigned* done, SummaryResult* res,
                          uint64_t seq, hipStream_t s) {
  const int64_t total = nevts * ntrks;
  const int64_t groups = grid_for(total, kSumThreads * kSumTracks);
  if (groups == 0) return hipErrorInvalidValue;
  return dispatch_width(width, [&](auto wc) {
    constexpr int W = decltype(wc)::value;
    hipLaunchKernelGGL((k_summary<W>), dim3((unsigned)groups), dim3(kSumThreads), 0, s, out, nb, ntrks, total, hx, hy,
                       hz, part, done, res, seq);
    return hipGetLastError();
  });
}

}  // namespace p2z
