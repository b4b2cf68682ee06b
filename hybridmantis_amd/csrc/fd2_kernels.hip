// fd2_kernels.hip -- HIP kernels of the MI355X fastDETECT2 transport.
//
//   k_queue_*     device work queue: exclusive scan of the events' photon
//                 counts (replaces the reference's host load
//                 balancer, main/hybridMANTIS_tallyEnergyDepositionEvents.f:
//                 195-250, and its one-thread-per-event launch,
//                 main/hybridMANTIS_cuda_ver1_0.cu:277)
//   k_transport   persistent kernel: each wave takes spans of consecutive
//                 photons from the queue with one atomic per span and hands
//                 photons to its idle lanes, so events of very uneven size
//                 keep every lane busy
//   k_trace_ranecu one lane per event, photons in sequence, the reference's
//                 per-event RANECU stream (trajectory test)
//   k_debug_steps per-step FP32 trace of a few photons (FP64 re-trace check)
//   k_debug_math  the device arithmetic on given arguments
#include "fd2_internal.h"

namespace fd2 {

// ------------------------------------------------------------ helpers

template <typename T>
__device__ __forceinline__ T wave_incl_scan(T x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    T y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  return x;
}

// photon and work-item (chunk) counts of event e; an event with a bad count
// or geometry has none and flags the launch
__device__ __forceinline__ void event_counts(const QueueArgs& q, int64_t e,
                                             uint32_t& chunks, uint32_t& photons) {
  chunks = 0;
  photons = 0;
  if (e >= q.n_events) return;
  const int32_t n = q.events[e].N;
  const uint32_t geom = q.events[e].geom;
  if (n < 0 || n > FD2_MAX_PHOTONS_PER_EVENT || geom >= (uint32_t)q.n_geoms) {
    if (n != 0) atomicOr(q.error_flag, 1u);
    return;
  }
  photons = (uint32_t)n;
  chunks = (photons + (1u << q.chunk_log2) - 1u) >> q.chunk_log2;
}

// A block's kScanTile events, a wave's 256 consecutive ones as kScanItems
// rows of 64 (each row one coalesced load): photon counts per row in ph, the
// number of photons before this wave's events in `before`, block totals in
// tp (photons) and tc (work items).  A block's totals fit 32 bits (4096
// events of at most 900,000 photons).
__device__ __forceinline__ void block_counts(const QueueArgs& q, int64_t base,
                                             uint32_t (&ph)[kScanItems], uint32_t& before,
                                             uint32_t& tp, uint32_t& tc) {
  constexpr int kWaves = kScanThreads / 64;
  __shared__ uint32_t s_p[kWaves], s_c[kWaves];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  uint32_t p = 0, c = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    uint32_t cc;
    event_counts(q, base + wid * (64 * kScanItems) + i * 64 + lane, cc, ph[i]);
    p += ph[i];
    c += cc;
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    p += __shfl_xor(p, o, 64);
    c += __shfl_xor(c, o, 64);
  }
  __syncthreads();
  if (lane == 0) {
    s_p[wid] = p;
    s_c[wid] = c;
  }
  __syncthreads();
  before = tp = tc = 0;
  for (int w = 0; w < kWaves; ++w) {
    if (w < wid) before += s_p[w];
    tp += s_p[w];
    tc += s_c[w];
  }
}

// photon_off of the block's events, `start` photons before the block
__device__ __forceinline__ void write_offsets(const QueueArgs& q, int64_t base,
                                              const uint32_t (&ph)[kScanItems],
                                              unsigned long long start) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    const uint32_t inc = wave_incl_scan(ph[i]);
    const int64_t e = base + wid * (64 * kScanItems) + i * 64 + lane;
    if (e < q.n_events) q.photon_off[e] = start + inc - ph[i];
    start += (uint32_t)__shfl((int)inc, 63, 64);
  }
}

// Totals, and how the launch is cut up (one thread).  A launch of more work
// items than q.max_chunks sets error bit 4 and gets a total of 0, so the
// transport takes nothing.
//
// A large launch uses all its waves and takes spans of half a wave's share, at
// most the tuning's chunk.  A small one ends with a long tail: it lasts as long
// as its longest photon's chain of passes (some hundreds), and a pass takes the
// longer the more waves share a SIMD (a wave alone waits for its own
// instructions; six issue 3 times as many as fit meanwhile).  So photons go to
// one wave per SIMD first, lane_cap to a wave, and the number of waves per SIMD,
// k, grows with the square root of the photons: the tail grows with
// k, the rest falls with the issue slots that k waves fill.  Every SIMD gets
// the same number of waves, as the launch waits for the fullest one.  lane_cap is
// the power of two with which the planned waves can take all photons, so a wave
// has up to twice the even share and some have none (33 photons per planned
// wave: half the waves take 64), and above 32 per planned wave a launch uses all
// lanes.  On MI355X with k = 1 to 6, 25 keV in 150 um (the only layer measured),
// kernel ms (chosen k marked):
//   2.7e5 photons   2.49 2.35* 2.40  2.62  2.65  2.63
//   6.5e5           3.70 3.07* 3.13  3.54  3.93  4.17
//   1.6e6           6.82 4.81  4.40* 4.57  4.79  5.15
//   5.5e6          18.83 11.2  9.28  8.74  8.73* 8.99
//   1.1e7          36.44 20.6  16.5  14.9  14.3  14.2*
// One wave more per 256 photons, as before: 2.42, 3.16, 5.13, 9.00, 14.2 ms.
// A single event of 1,375 photons takes 0.46 ms with lane_cap 2 and 0.8 ms in
// spans of 128 on all waves.
__device__ __forceinline__ void plan_queue(const QueueArgs& q, unsigned long long photons,
                                           uint64_t chunks) {
  constexpr uint32_t kWaves = kTransportThreads / 64;
  const bool over = chunks > q.max_chunks;
  if (over) atomicOr(q.error_flag, 4u);
  q.photon_off[q.n_events] = over ? 0ull : photons;
  const uint32_t alone = min(q.n_simds, q.n_waves);
  unsigned long long per_simd = photons < 128ull * alone ? 1u : 2u;
  while (per_simd >= 2u && per_simd * alone < q.n_waves &&
         photons >= (2u * per_simd + 1u) * (2u * per_simd + 1u) * 64ull * alone)
    ++per_simd;
  unsigned long long waves = per_simd * alone;
  if (waves > q.n_waves) waves = q.n_waves;
  uint32_t span_log2 = 0, lane_cap = 64;
  if (photons >= 64u * waves) {
    const unsigned long long share = photons / waves;
    while (span_log2 < (uint32_t)q.chunk_log2 && (4ull << span_log2) <= share) ++span_log2;
  } else {
    while ((waves << span_log2) < photons) ++span_log2;
    lane_cap = 1u << span_log2;
    if ((uint32_t)q.chunk_log2 < span_log2) span_log2 = (uint32_t)q.chunk_log2;
  }
  q.plan->cursor = 0u;
  q.plan->span_log2 = span_log2;
  q.plan->lane_cap = lane_cap;
  q.plan->blocks = (uint32_t)((waves + kWaves - 1u) / kWaves);
}

// the whole build for at most kScanTile events (one block)
__global__ void __launch_bounds__(kScanThreads) k_queue_small(QueueArgs q) {
  uint32_t ph[kScanItems], before, tp, tc;
  block_counts(q, 0, ph, before, tp, tc);
  write_offsets(q, 0, ph, before);
  if (threadIdx.x == 0) plan_queue(q, tp, tc);
}

// pass 1: per-block totals
__global__ void __launch_bounds__(kScanThreads) k_queue_totals(QueueArgs q) {
  uint32_t ph[kScanItems], before, tp, tc;
  block_counts(q, (int64_t)blockIdx.x * kScanTile, ph, before, tp, tc);
  if (threadIdx.x == 0) {
    q.block_chunks[blockIdx.x] = tc;
    q.block_photons[blockIdx.x] = tp;
  }
}

// pass 2: scan of the block totals and grand totals (one wave)
__global__ void __launch_bounds__(64) k_queue_blocks(QueueArgs q) {
  uint64_t chunks = 0;
  unsigned long long photons = 0;
  for (int b0 = 0; b0 < q.n_blocks; b0 += 64) {
    const int b = b0 + (int)threadIdx.x;
    const uint64_t c = b < q.n_blocks ? q.block_chunks[b] : 0u;
    const unsigned long long p = b < q.n_blocks ? q.block_photons[b] : 0ull;
    const uint64_t ic = wave_incl_scan(c);
    const unsigned long long ip = wave_incl_scan(p);
    if (b < q.n_blocks) q.block_photons[b] = photons + ip - p;
    chunks += __shfl(ic, 63, 64);
    photons += __shfl(ip, 63, 64);
  }
  if (threadIdx.x == 0) plan_queue(q, photons, chunks);
}

// pass 3: per-event exclusive offsets
__global__ void __launch_bounds__(kScanThreads) k_queue_offsets(QueueArgs q) {
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  uint32_t ph[kScanItems], before, tp, tc;
  block_counts(q, base, ph, before, tp, tc);
  write_offsets(q, base, ph, q.block_photons[blockIdx.x] + before);
}

hipError_t launch_queue_build(const QueueArgs& q, hipStream_t s) {
  if (q.n_blocks <= 0 || q.n_waves == 0u) return hipErrorInvalidValue;
  if (q.n_blocks == 1) {
    hipLaunchKernelGGL(k_queue_small, dim3(1), dim3(kScanThreads), 0, s, q);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_queue_totals, dim3(q.n_blocks), dim3(kScanThreads), 0, s, q);
  hipLaunchKernelGGL(k_queue_blocks, dim3(1), dim3(64), 0, s, q);
  hipLaunchKernelGGL(k_queue_offsets, dim3(q.n_blocks), dim3(kScanThreads), 0, s, q);
  return hipGetLastError();
}

// ------------------------------------------------------------ tallies

// Counter-mode initial direction of photon k: photon 0 takes the driver's
// first direction (|2u-1| > 0.01 by rejection,
// main/hybridMANTIS_c_ver1_0.c:257-277), the others the direction algo()
// draws at the previous photon's end (main/kernel_cuda_c_ver1_0.cu:578-602)
// followed by the RoughSurface draws of the (never read) initial normal.
__device__ __forceinline__ void counter_initial_dir(CounterRng& rng, Photon& p,
                                                    uint32_t k, const ColumnGeom& g) {
  float r = rng.u() * 2.0f - 1.0f;
  if (k == 0)
    while (fabsf(r) <= 0.01f) r = rng.u() * 2.0f - 1.0f;
  p.uz = r;
  azimuth<MathDevice>(fd2_sqrt_01(1.0f - r * r), rng, p.ux, p.uy);
  renorm(p.ux, p.uy, p.uz, g);
  if (k != 0 && g.beta > 0.0f) {
    (void)rng.u();
    (void)rng.u();
  }
}

// ------------------------------------------------------- transport

// Register budget of the transport kernel: 6 waves per SIMD (80 VGPRs, 7
// values of rare paths in scratch; without a limit the wall branch takes 92).
// mono25x50 on MI355X at 20 and 24 waves per CU: 94.5 ms with 5 waves per
// SIMD, 89.9 ms with 6; the LDS (26.5 KB per workgroup) holds no more.
// FD2_WAVES_PER_EU=0 lets the compiler choose.
#ifndef FD2_WAVES_PER_EU
#define FD2_WAVES_PER_EU 6
#endif
// With several geometries per launch (the geometry table in LDS, read per
// lane, and a geometry index per photon) and with records the LDS holds 5 (4
// from some 25 geometries on).
#if FD2_WAVES_PER_EU > 0
#define FD2_TRANSPORT_ATTR \
  __attribute__((amdgpu_waves_per_eu(MULTI || REC ? FD2_WAVES_PER_EU - 1 : FD2_WAVES_PER_EU, \
                                     MULTI || REC ? FD2_WAVES_PER_EU - 1 : FD2_WAVES_PER_EU)))
#else
#define FD2_TRANSPORT_ATTR
#endif

// log-radial bin of a detection offset (FD2_RADIAL_BINS layout)
__device__ __forceinline__ int radial_bin(float dx, float dy) {
  const float r = sqrtf(dx * dx + dy * dy);
  if (!(r >= 0.5f)) return 0;
  if (r >= 800.0f) return FD2_RADIAL_BINS - 1;
  // 1 + floor(62 * ln(r/0.5) / ln(1600))
  int b = 1 + (int)(fd2_log(r * 2.0f) * 8.40363595f);
  return b < 1 ? 1 : (b > FD2_RADIAL_BINS - 2 ? FD2_RADIAL_BINS - 2 : b);
}

// first pixel row/column of a geometry's LDS tile
__device__ __forceinline__ int tile_origin(int dim, int side) {
  return dim > side ? (dim - side) >> 1 : 0;
}

// Adds a lane's run of detections of one event to the event's history
// count (the event's history and geometry are read here, once per run, not
// once per detection).  `gt` is the launch's geometry unless MULTI.
template <bool MULTI>
__device__ __forceinline__ void flush_run(const GeomDev& gt, const GeomDev* geoms,
                                          const fd2_event* __restrict__ events, uint32_t run_ev,
                                          uint32_t run_cnt) {
  const fd2_event& ev = events[run_ev];
  const int32_t hist = ev.hist;
  const GeomDev& g = MULTI ? geoms[ev.geom] : gt;
  if (hist >= 1 && hist <= g.num_hist) tally_add(&g.hist[hist - 1], run_cnt);
}

// Tallies of an ended photon: fate counter, PRF pixel (LDS tile or HBM),
// per-lane run of the event's detections, radial bin, record.
template <bool MULTI, bool REC, bool RADIAL>
__device__ __forceinline__ void finish_photon(const TransportArgs& a, const GeomDev& gt,
                                              const GeomDev* geoms,
                                              const fd2_event* __restrict__ events, Photon& p,
                                              uint32_t gi, uint32_t lane_ev, uint32_t lane_k,
                                              uint32_t* s_cnt, uint32_t* s_tile, uint32_t* run) {
  atomicAdd(&s_cnt[gi * kCounters + fate_counter(p.fate)], 1u);
  const bool det = p.fate == kDetectOut;
  Pixel x{0, 0};
  if (det) {
    x = detected_pixel(p, gt);
    if (p.fate == kDetect) {
      bool in_tile = false;
      if ((int)gi < a.n_tiles) {
        const int side = a.tile_side;
        const uint32_t ti = (uint32_t)(x.i - tile_origin(gt.xdim, side));
        const uint32_t tj = (uint32_t)(x.j - tile_origin(gt.ydim, side));
        if (ti < (uint32_t)side && tj < (uint32_t)side) {
          atomicAdd(&s_tile[(gi * side + ti) * side + tj], 1u);
          in_tile = true;
        }
      }
      if (!in_tile) tally_add(&gt.prf[pix_index(x, gt)], 1ull);
    }
    if (lane_ev == run[0]) {
      ++run[1];
    } else {
      if (run[1]) flush_run<MULTI>(gt, geoms, events, run[0], run[1]);
      run[0] = lane_ev;
      run[1] = 1;
    }
    if (RADIAL) {
      const fd2_event& ev = events[lane_ev];
      tally_add(
          &a.radial[(size_t)lane_ev * FD2_RADIAL_BINS + radial_bin(p.px - ev.x, p.py - ev.y)], 1u);
    }
  }
  if (REC) {
    fd2_photon rec;
    rec.fate = p.fate;
    rec.pix = p.fate == kDetect ? pix_index(x, gt) : -1;
    rec.x = det ? p.px : 0.0f;
    rec.y = det ? p.py : 0.0f;
    a.records[a.photon_off[lane_ev] + lane_k] = rec;
  }
}

// A photon's words in the LDS queue and the HBM queues: everything a photon
// in flight carries (not the surface normal: every path writes it before
// reading it); gap-queue entries also the wall branch's loop state
// (PrptState).  An entry's words lie `S` words apart from its first: kQBlock
// in the HBM queues, kWallSlots in a wave's LDS queue (word-major, one row of
// slots per word).  The geometry index is stored only for several geometries
// per launch (MULTI; else 0) and the photon index only for per-photon records
// (REC).
template <bool MULTI, bool REC, int S>
__device__ __forceinline__ void q_put(uint32_t* w, const Photon& p, const CounterRng& r,
                                      uint32_t ev, uint32_t gi, uint32_t k) {
  w[0 * S] = __float_as_uint(p.px);
  w[1 * S] = __float_as_uint(p.py);
  w[2 * S] = __float_as_uint(p.pz);
  w[3 * S] = __float_as_uint(p.ux);
  w[4 * S] = __float_as_uint(p.uy);
  w[5 * S] = __float_as_uint(p.uz);
  w[6 * S] = __float_as_uint(p.xc);
  w[7 * S] = __float_as_uint(p.yc);
  w[8 * S] = p.st;
  w[9 * S] = r.s0;
  w[10 * S] = r.s1;
  w[11 * S] = r.s2;
  w[12 * S] = r.s3;
  w[13 * S] = ev;
  if (MULTI) w[14 * S] = gi;
  if (REC) w[(14 + MULTI) * S] = k;
}

template <bool MULTI, bool REC, int S>
__device__ __forceinline__ void q_get(const uint32_t* w, Photon& p, CounterRng& r, uint32_t& ev,
                                      uint32_t& gi, uint32_t& k) {
  p.px = __uint_as_float(w[0 * S]);
  p.py = __uint_as_float(w[1 * S]);
  p.pz = __uint_as_float(w[2 * S]);
  p.ux = __uint_as_float(w[3 * S]);
  p.uy = __uint_as_float(w[4 * S]);
  p.uz = __uint_as_float(w[5 * S]);
  p.nx = p.ny = p.nz = 0.0f;  // written before it is read
  p.xc = __uint_as_float(w[6 * S]);
  p.yc = __uint_as_float(w[7 * S]);
  p.st = w[8 * S];
  r.s0 = w[9 * S];
  r.s1 = w[10 * S];
  r.s2 = w[11 * S];
  r.s3 = w[12 * S];
  ev = w[13 * S];
  gi = MULTI ? w[14 * S] : 0u;
  k = REC ? w[(14 + MULTI) * S] : 0u;
}

// Per-wave gap queue and backlog in HBM (kQSlots entries of kQWords words).
// Slots come in blocks of kQBlock = 32; word j of slot s is at
// [(s / 32) * 32 * kQWords + 32 j + s % 32], so the lanes of a wave write
// whole 128-byte lines and all words of a slot lie within 3 KB of its first
// (one address per lane, the rest immediate offsets).
__device__ __forceinline__ size_t q_base(uint32_t slot) {
  return (size_t)(slot / kQBlock) * (kQBlock * kQWords) + slot % kQBlock;
}

__device__ __forceinline__ void q_put_state(uint32_t* w, const PrptState& st) {
  w[16 * kQBlock] = st.tries;
  w[17 * kQBlock] = __float_as_uint(st.pr);
  w[18 * kQBlock] = __float_as_uint(st.s2);
  w[19 * kQBlock] = __float_as_uint(st.c2);
}

__device__ __forceinline__ void q_get_state(const uint32_t* w, PrptState& st) {
  st.tries = w[16 * kQBlock];
  st.pr = __uint_as_float(w[17 * kQBlock]);
  st.s2 = __uint_as_float(w[18 * kQBlock]);
  st.c2 = __uint_as_float(w[19 * kQBlock]);
}

// number of set bits of a wave-wide mask below this lane (v_mbcnt)
__device__ __forceinline__ uint32_t rank_below(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
__device__ __forceinline__ uint32_t count(unsigned long long mask) {
  return (uint32_t)__popcll(mask);
}
// whether this lane is in a wave-wide mask (the mask becomes the lane predicate)
__device__ __forceinline__ bool in(unsigned long long mask) {
  return __builtin_amdgcn_inverse_ballot_w64(mask);
}

// the lowest `t` lanes of a mask, given their ranks in it
__device__ __forceinline__ unsigned long long lowest(unsigned long long mask, uint32_t rank,
                                                     uint32_t t) {
  return mask & __ballot(rank < t);
}

// A table entry at a wave-uniform address by scalar loads of the members that
// are used.  The pointer is opaque: the loads stay where they are asked for,
// instead of the values being kept in scalar registers over the whole loop
// (spilled, and refilled 16 at a time around every use).
template <class T>
__device__ __forceinline__ T load_uniform(const void* p) {
  auto one = (const __attribute__((address_space(4))) T*)p;
  asm volatile("" : "+s"(one));
  T c;
  __builtin_memcpy(&c, one, sizeof c);  // typed: the alignment makes them scalar loads
  return c;
}

__device__ __forceinline__ ColumnGeom load_column(const void* p) {
  typedef uint32_t Words __attribute__((ext_vector_type(16)));
  auto one = (const __attribute__((address_space(4))) Words*)p;
  asm volatile("" : "+s"(one));
  Words w = *one;
  asm volatile("" : "+s"(w));
  ColumnGeom g;
  __builtin_memcpy(&g, &w, sizeof g);
  return g;
}

// Event of photon g of the launch: the largest e with photon_off[e] <= g
// (skips events without photons).  Each round the 64 lanes (all active) probe
// 64 points of [lo, hi) with one vector load, and the wave keeps the step
// after the last probe at or below g -- 3 rounds for 2e5 events where a
// binary search makes 18 dependent loads.
__device__ __forceinline__ uint32_t event_of(const unsigned long long* __restrict__ photon_off,
                                             int64_t n_events, uint64_t g, int lane) {
  int64_t lo = 0, hi = n_events;
  while (hi - lo > 1) {
    const int64_t step = (hi - lo + 63) >> 6;
    const int64_t pos = lo + (int64_t)lane * step;
    const bool le = pos < hi && photon_off[pos] <= g;
    const unsigned long long m = __ballot(le);
    lo += (int64_t)(63 - __clzll(m)) * step;
    hi = min(hi, lo + step);
  }
  return (uint32_t)lo;
}

// Events of photons g .. g + n - 1 (n <= 64, lane j's of photon g + j), the
// first of event e0, where they span several (reference event buffers hold
// about two photons per event).  A round reads the starts of the 64 events
// after the current one and every unresolved lane counts those at or before
// its photon (a binary search over the lanes' values); a window without a
// photon's event (a long run of empty events) is left by a search.
__device__ __forceinline__ uint32_t events_of(const unsigned long long* __restrict__ photon_off,
                                              int64_t n_events, uint32_t e0, uint64_t g,
                                              uint32_t n, int lane) {
  uint32_t e = e0, done = 0;
  while (done < n) {
    const uint64_t first = g + done;
    const int64_t i = (int64_t)e0 + 1 + lane;
    uint32_t v = 0xffffffffu;  // start of event i, in photons after `first`
    if (i <= n_events) {
      const uint64_t o = photon_off[i];
      v = o <= first ? 0u : (uint32_t)min(o - first, (uint64_t)0xffffffffu);
    }
    const bool open = (uint32_t)lane >= done && (uint32_t)lane < n;
    const uint32_t rel = (uint32_t)lane - done;
    uint32_t at = 0;
#pragma unroll
    for (uint32_t s = 32; s != 0u; s >>= 1) {
      const uint32_t t = (uint32_t)__shfl((int)v, (int)(at + s - 1u), 64);
      if (t <= rel) at += s;
    }
    const uint32_t last = (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
    const bool found = open && last > rel;
    if (found) e = e0 + at;
    const uint32_t m = (uint32_t)__popcll(__ballot(found));
    if (m != 0u) {
      done += m;
      e0 = (uint32_t)__builtin_amdgcn_readlane((int)e, (int)(done - 1u));
    } else {
      e0 = event_of(photon_off, n_events, first, lane);
    }
  }
  return e;
}

// Persistent transport.  A wave keeps the state of its lanes in wave-uniform
// masks: step_m (a photon that takes in-column passes) and wall_m (a photon
// that waits for the wall's Fresnel branch); the other lanes are free.  Its
// loop:
//
//   serve   once refill_lanes lanes do not step: count 64 ended photons if as
//           many wait, put the photons waiting for the wall into the wave's LDS
//           queue and fill the free lanes (LDS queue, HBM backlog, then new
//           photons of the work queue, which all lanes start together into the
//           LDS queue)
//   pass    one in-column pass of the stepping lanes
//   wall    once 64 photons wait (in lanes and in the LDS queue): the branch
//           runs with all 64 lanes, up to a refraction out of the column;
//           photons that were stepping change places with queue entries, so
//           they stay in LDS
//   gap     the flights through the gap between columns, again 64 at a time
//           (HBM gap queue), one flight per photon and round; photons that
//           were stepping go to the HBM backlog meanwhile
//
// The LDS queue holds waiting photons from its bottom up (n_wall) and photons
// ready to step from its top down (n_ready).  n_wall + n_ready <= kLdsCap
// outside of serve: a waiting photon enters from a lane that then takes a
// ready one, and the wall phase swaps at most as many in as it takes out.  The
// slots above kLdsCap let a lane write before it reads.  Moving the stepping photons to
// HBM and back around every wall phase, as the gap phase still does, took
// 1.2e11 of 1.5e11 bytes of a mono25x50 launch and a wait for HBM at each
// refill.
//
// Draining (no span, ready photon or backlog left), and throughout when
// the queues are not used (tuning) or a launch has at most 32 photons per
// planned wave (lane_cap < 64), waiting photons stay in their lanes: the branch
// and the flights run where they are, with the other lanes masked off, once at least as many
// wait as step (without queues: park_lanes).
//
// The loop's scalar work counts as much as its vector work: six waves share a
// SIMD's issue slots.  So only a serve decides the mode and when the next serve
// is due, a round without a phase does nothing else, and a lane mask is made
// before the branch that uses it (made inside, it becomes a lane flag and a
// mask again).  mono25x50 on MI355X: 103.7 -> 89.7 ms, 793 -> 711 vector and 365
// -> 276 scalar instructions per photon, most of it spilled scalar registers.
//
// Every photon keeps its own state and random stream, so the results are the
// same in either mode and in any order.
//
// `geoms_in`, `events` and `photon_off` are a.geoms, a.events and
// a.photon_off again, as parameters of their own: the kernel never writes
// these tables (only the tallies the geometries point to), and saying so
// (__restrict__) lets the compiler read them with scalar loads where they
// are uniform instead of reloading them with vector loads around every
// store.
template <bool MULTI, bool REC, bool RADIAL>
__global__ void __launch_bounds__(kTransportThreads) FD2_TRANSPORT_ATTR
k_transport(TransportArgs a, const GeomDev* __restrict__ geoms_in,
            const fd2_event* __restrict__ events,
            const unsigned long long* __restrict__ photon_off) {
  // With several geometries a lane's geometry is its own, so their constants
  // cannot be scalar loads: the table goes to LDS instead.
  static_assert(sizeof(GeomDev) % 8 == 0, "GeomDev copied as words");
  if (blockIdx.x >= a.plan->blocks) return;  // a small launch (plan_queue)
  extern __shared__ __align__(16) uint32_t s_dyn[];  // geometry table (MULTI), then PRF tiles
  const int geom_words = MULTI ? a.n_geoms * (int)(sizeof(GeomDev) / 4) : 0;
  if (MULTI) {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(geoms_in);
    for (int i = threadIdx.x; i < geom_words; i += blockDim.x) s_dyn[i] = src[i];
  }
  const GeomDev* __restrict__ geoms = MULTI ? reinterpret_cast<const GeomDev*>(s_dyn) : geoms_in;
  uint32_t* s_tile = s_dyn + geom_words;  // n_tiles x tile_side^2
  __shared__ uint32_t s_cnt[FD2_MAX_GEOMS * kCounters];
  // the waves' LDS queues, word-major
  __shared__ uint32_t s_queue[kTransportThreads / 64][14 + MULTI + REC][kWallSlots];
  for (int i = threadIdx.x; i < a.n_geoms * kCounters; i += blockDim.x) s_cnt[i] = 0;
  for (int i = threadIdx.x; i < a.n_tiles * a.tile_side * a.tile_side; i += blockDim.x)
    s_tile[i] = 0;
  __syncthreads();

  // per-lane run of detections of one event (event, count), added to the
  // event's history count when the lane's detections move on to another
  // event (consecutive photons share their event); in LDS, as it is touched
  // only when a photon ends
  __shared__ uint32_t s_run[kTransportThreads][2];
  uint32_t* run = s_run[threadIdx.x];
  run[0] = 0u;
  run[1] = 0u;

  const int lane = threadIdx.x & 63;
  // the wave's index in the block, uniform across the wave: the compiler
  // then keeps the wave's queue and LDS bases in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // wave-uniform work pool: pool_left of the launch's photons from
  // pool_next on, the first of event pool_ev
  uint64_t pool_next = 0;
  uint32_t pool_left = 0, pool_ev = 0;
  bool pool_done = false;

  Photon p;
  p.fate = kAlive;
  CounterRng rng;
  unsigned long long step_m = 0, wall_m = 0;
  uint32_t gi = 0;
  uint32_t lane_ev = 0;  // the lane's event (index into events)
  uint32_t lane_k = 0;   // photon index within the event
  StepSink nosink{nullptr, nullptr, 0, 0, false};

  uint32_t* lq = &s_queue[wave][0][0];
  // the wave's queues in HBM: gap queue [0, n_gap), backlog [0, n_back), ended
  // photons [0, n_end)
  uint32_t* wq = a.wave_queue + (size_t)(blockIdx.x * (kTransportThreads / 64) + wave) * kWaveWords;
  uint32_t n_wall = 0, n_ready = 0, n_gap = 0, n_back = 0, n_end = 0, idle = 0;
  const uint32_t lane_cap = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.plan->lane_cap);
  const bool queued = a.queues != 0 && lane_cap == 64u;
  const uint32_t park = a.queues != 0 ? 0u : (uint32_t)a.park_lanes;
  const uint32_t serve_at = min((uint32_t)a.refill_lanes, lane_cap);
  const unsigned long long use_m = lane_cap == 64u ? ~0ull : (1ull << lane_cap) - 1ull;

  // the launch's arguments, read again where they are needed: held over the
  // loop they would take the scalar registers of its lane masks
  const void* kernarg = (const void*)__builtin_amdgcn_kernarg_segment_ptr();
  auto args = [&]() { return load_uniform<TransportArgs>(kernarg); };
  // f(the lane's geometry)
  auto with_geom = [&](auto f) {
    if constexpr (MULTI)
      f(geoms[gi]);
    else
      f(load_uniform<GeomDev>(kernarg));
  };
  // Ended photons wait in HBM until 64 of them are counted at once: about one
  // lane of a wave ends in two passes, and its tallies are as long as a third
  // of a pass (mono25x50: 104.5 ms counted in each serve, 103.7 here).
  auto end_put = [&](unsigned long long m) {
    if (m == 0ull) return;
    if (in(m)) {
      uint32_t* w = wq + kQWords * kQSlots + n_end + rank_below(m);
      w[0] = (uint32_t)p.fate | (MULTI ? gi << 8 : 0u);
      w[kEndCap] = __float_as_uint(p.px);
      w[2 * kEndCap] = __float_as_uint(p.py);
      w[3 * kEndCap] = lane_ev;
      if (REC) w[4 * kEndCap] = lane_k;
    }
    n_end += count(m);
  };
  auto end_count = [&]() {
    const uint32_t t = min(n_end, 64u);
    n_end -= t;
    __threadfence_block();  // the wave's queue stores are complete before its loads
    if ((uint32_t)lane < t) {
      const uint32_t* w = wq + kQWords * kQSlots + n_end + lane;
      Photon q;
      q.fate = (int)(w[0] & 0xffu);
      const uint32_t g2 = MULTI ? w[0] >> 8 : 0u;
      q.px = __uint_as_float(w[kEndCap]);
      q.py = __uint_as_float(w[2 * kEndCap]);
      const uint32_t ev = w[3 * kEndCap], k = REC ? w[4 * kEndCap] : 0u;
      const auto count_one = [&](const GeomDev& g) {
        finish_photon<MULTI, REC, RADIAL>(args(), g, geoms, events, q, g2, ev, k, s_cnt, s_tile,
                                          run);
      };
      if constexpr (MULTI)
        count_one(geoms[g2]);
      else
        count_one(load_uniform<GeomDev>(kernarg));
    }
  };
  auto lds_put = [&](uint32_t slot) {
    q_put<MULTI, REC, kWallSlots>(lq + slot, p, rng, lane_ev, gi, lane_k);
  };
  auto lds_get = [&](uint32_t slot) {
    q_get<MULTI, REC, kWallSlots>(lq + slot, p, rng, lane_ev, gi, lane_k);
  };
  // fills up to n_ready of the lanes in `want` from the ready photons
  auto take_ready = [&](unsigned long long want) {
    const uint32_t t = min(count(want), n_ready);
    if (t == 0u) return;
    const uint32_t rank = rank_below(want);
    const unsigned long long got = lowest(want, rank, t);
    lds_order();
    if (in(got)) lds_get((uint32_t)kWallSlots - n_ready + rank);
    lds_order();
    n_ready -= t;
    step_m |= got;
  };

  // How waiting photons are served, decided in each serve: 0 through the
  // queues, 1 in their lanes (no queues, or a small launch), 2 in their lanes
  // while the wave drains.  A serve is due once at most busy_max lanes step
  // (or, in place, wait).
  int mode = queued ? 0 : 1;
  int busy_max = (int)(lane_cap - serve_at);
  bool last = false;  // no photon is left; the ended ones are still to be counted
  for (;;) {
    unsigned long long gap_m = 0;  // lanes whose photon's gap flight is next
    // ---- serve
    if (step_m == 0ull || (int)count(mode == 0 ? step_m : step_m | wall_m) <= busy_max) {
      while (n_end >= 64u || (last && n_end != 0u)) end_count();
      if (last) break;
      {
        if (mode == 0 && n_wall + count(wall_m) < 64u) {
          while (wall_m != 0ull) {
            const uint32_t k =
                min(count(wall_m), (uint32_t)kWallSlots - n_wall - n_ready);
            const uint32_t rank = rank_below(wall_m);
            const unsigned long long put = lowest(wall_m, rank, k);
            if (in(put)) lds_put(n_wall + rank);
            n_wall += k;
            wall_m &= ~put;
            take_ready(~(step_m | wall_m));
          }
        }
        take_ready(use_m & ~(step_m | wall_m));
        unsigned long long need = use_m & ~(step_m | wall_m);
        if (need != 0ull && n_back != 0u) {
          __threadfence_block();  // the wave's queue stores are complete before its loads
          const uint32_t t = min(count(need), n_back);
          const uint32_t rank = rank_below(need);
          const unsigned long long got = lowest(need, rank, t);
          if (in(got))
            q_get<MULTI, REC, kQBlock>(wq + q_base(kBackBase + n_back - 1u - rank), p, rng,
                                       lane_ev, gi, lane_k);
          n_back -= t;
          step_m |= got;
          need = use_m & ~(step_m | wall_m);
        }
        while (need != 0ull && !pool_done) {
          const TransportArgs b = args();
          if (pool_left == 0u) {
            uint32_t c = 0;
            if (lane == 0) c = atomicAdd(&b.plan->cursor, 1u);
            c = (uint32_t)__builtin_amdgcn_readfirstlane((int)c);
            const uint64_t total = photon_off[b.n_events];
            const uint32_t span_log2 = b.plan->span_log2;
            pool_next = (uint64_t)c << span_log2;
            if (pool_next >= total) {
              pool_done = true;
              break;
            }
            pool_left = (uint32_t)min(total - pool_next, (uint64_t)1 << span_log2);
            pool_ev = event_of(photon_off, b.n_events, pool_next, lane);
          }
          // Seeding a stream (Philox) and drawing the first direction are
          // long: every lane starts one of the next photons here, as many as
          // the LDS queue has room for.
          const uint32_t n = min(min((uint32_t)kLdsCap - n_wall, 64u), pool_left);
          uint32_t e = pool_ev;
          if (photon_off[pool_ev + 1u] - pool_next < n)
            e = events_of(photon_off, b.n_events, pool_ev, pool_next, n, lane);
          if ((uint32_t)lane < n) {
            const fd2_event ev = events[e];
            const uint32_t k = (uint32_t)(pool_next + (uint32_t)lane - photon_off[e]);
            CounterRng r;
            Photon q;
            start_photon(q, ev);
            const uint64_t event_base = b.event_base_dev ? *b.event_base_dev : b.event_base;
            r.seed(b.seed, event_base + (uint64_t)e, k);
            if constexpr (MULTI) {
              counter_initial_dir(r, q, k, geoms[ev.geom]);
              atomicAdd(&s_cnt[ev.geom * kCounters + FD2_C_GENERATED], 1u);
            } else {
              counter_initial_dir(r, q, k, load_uniform<ColumnGeom>(kernarg));
              if (lane == 0) atomicAdd(&s_cnt[FD2_C_GENERATED], n);
            }
            q_put<MULTI, REC, kWallSlots>(lq + (uint32_t)kWallSlots - n + lane, q, r, e,
                                          MULTI ? ev.geom : 0u, k);
          }
          n_ready = n;
          pool_next += n;
          pool_left -= n;
          pool_ev = (uint32_t)__builtin_amdgcn_readlane((int)e, (int)(n - 1u));
          take_ready(need);
          need = use_m & ~(step_m | wall_m);
        }
        const bool drain = pool_done && n_ready == 0u && n_back == 0u;
        if (drain && queued && need != 0ull && (n_wall | n_gap) != 0u) {
          // the queues' last photons back into free lanes
          uint32_t t = min(count(need), n_wall);
          const uint32_t rank = rank_below(need);
          const unsigned long long got = lowest(need, rank, t);
          lds_order();
          if (in(got)) lds_get(n_wall - t + rank);
          n_wall -= t;
          wall_m |= got;
          need &= ~got;
          t = min(count(need), n_gap);
          if (t != 0u) gap_m = lowest(need, rank_below(need), t);  // loaded in the gap section
        }
        mode = drain ? 2 : queued ? 0 : 1;
        busy_max = drain && (n_wall | n_gap) == 0u ? -1 : (int)(lane_cap - serve_at);
        // nothing in a lane: the queues and the work queue are empty
        last = (step_m | wall_m | gap_m) == 0ull;
        if (last) continue;
      }
    }
    const bool stepped = step_m != 0ull;
    // ---- pass
    {
      if (in(step_m)) {
        auto pass = [&](const ColumnGeom& g) {
          hot_step<CounterRng, false>(rng, p, g, &nosink);
          if (__builtin_expect(p.fate == kTrapped, 0)) {
            atomicAdd(&s_cnt[gi * kCounters + FD2_C_REGEN], 1u);
            restart_trapped(rng, p, g, events[lane_ev]);
          }
        };
        if constexpr (MULTI)
          pass(geoms[gi]);
        else
          pass(load_column(kernarg));
      }
      const unsigned long long e = step_m & __ballot(ended(p.fate));
      const unsigned long long w = step_m & __ballot(p.fate == kWall);
      end_put(e);
      wall_m |= w;
      step_m &= ~(e | w);
    }
    // ---- wall
    const uint32_t n_lane = count(wall_m), n_step = count(step_m);
    const bool in_place = mode != 0;
    bool wall = n_wall + n_lane >= 64u;
    if (in_place) wall = n_lane != 0u && (n_step == 0u || n_lane >= (park != 0u ? park : n_step));
    // every round steps a photon or runs a phase; a wave that does neither
    // for many rounds has a broken queue state: it stops and flags the launch
    // rather than spin
    if (stepped || wall || gap_m != 0ull) {
      idle = 0;
    } else if (++idle > kMaxIdlePasses) {
      if (lane == 0) atomicOr(args().error_flag, 2u);
      break;
    }
    if (!wall && gap_m == 0ull) continue;
    PrptState st = prpt_initial();
    const unsigned long long fetch_m = gap_m;
    gap_m = 0ull;
    if (wall) {
      if (!in_place) {
        // every lane without a waiting photon takes one; a photon that was
        // stepping takes a ready slot (all reads come before the writes)
        const unsigned long long need = ~wall_m;
        const uint32_t t = 64u - n_lane, rank = rank_below(need);
        Photon q;
        CounterRng r;
        uint32_t ev = 0, g2 = 0, k2 = 0;
        lds_order();
        if (in(need)) {
          q_get<MULTI, REC, kWallSlots>(lq + n_wall - t + rank, q, r, ev, g2, k2);
          lds_order();
          if (in(step_m))
            lds_put((uint32_t)kWallSlots - n_ready - n_step + rank_below(step_m));
          p = q;
          rng = r;
          lane_ev = ev;
          gi = g2;
          lane_k = k2;
        }
        n_wall -= t;
        n_ready += n_step;
        step_m = 0ull;
        wall_m = ~0ull;
      }
      int r = kPrAlive;
      if (in(wall_m))
        with_geom([&](const GeomDev& g) { r = prpt_loop(rng, p, g, st, true, true); });
      const unsigned long long e = __ballot(r == kPrEnded);
      gap_m = __ballot(r == kPrGap);
      end_put(e);
      step_m |= wall_m & ~(e | gap_m);
      wall_m = 0ull;
    }
    if (fetch_m != 0ull) {
      // a draining wave's free lanes take photons of the gap queue
      n_gap -= count(fetch_m);
      __threadfence_block();
      if (in(fetch_m)) {
        const uint32_t* w = wq + q_base(kGapBase + n_gap + rank_below(fetch_m));
        q_get<MULTI, REC, kQBlock>(w, p, rng, lane_ev, gi, lane_k);
        q_get_state(w, st);
      }
      gap_m |= fetch_m;
    }
    // ---- gap: one flight per photon and round (to the next column and its
    // Fresnel decision); a photon reflected off the outside of that column
    // waits for its next flight.  The gap queue holds at most 63 + 64 entries
    // here, and 63 between rounds.
    bool failed = false;
    for (;;) {
      if (!in_place) {
        if (gap_m != 0ull) {
          if (in(gap_m)) {
            uint32_t* w = wq + q_base(kGapBase + n_gap + rank_below(gap_m));
            q_put<MULTI, REC, kQBlock>(w, p, rng, lane_ev, gi, lane_k);
            q_put_state(w, st);
          }
          n_gap += count(gap_m);
          gap_m = 0ull;
        }
        if (n_gap < 64u) break;
        const uint32_t s = count(step_m);
        if (n_back + s > (uint32_t)kBackCap) {  // ruled out by the photons in flight
          failed = true;
          break;
        }
        if (in(step_m))
          q_put<MULTI, REC, kQBlock>(wq + q_base(kBackBase + n_back + rank_below(step_m)), p, rng,
                                     lane_ev, gi, lane_k);
        n_back += s;
        step_m = 0ull;
        __threadfence_block();
        const uint32_t* w = wq + q_base(kGapBase + n_gap - 64u + (uint32_t)lane);
        q_get<MULTI, REC, kQBlock>(w, p, rng, lane_ev, gi, lane_k);
        q_get_state(w, st);
        n_gap -= 64u;
        gap_m = ~0ull;
      } else if (gap_m == 0ull) {
        break;
      }
      int r = kPrAlive;
      if (in(gap_m))
        with_geom([&](const GeomDev& g) { r = prpt_loop(rng, p, g, st, false, true); });
      const unsigned long long e = __ballot(r == kPrEnded);
      const unsigned long long again = __ballot(r == kPrGap);
      end_put(e);
      step_m |= gap_m & ~(e | again);
      gap_m = again;
    }
    if (failed) {
      if (lane == 0) atomicOr(args().error_flag, 2u);
      break;
    }
  }

  if (run[1]) flush_run<MULTI>(geoms_in[0], geoms, events, run[0], run[1]);
  __syncthreads();
  const TransportArgs b = args();
  const int side = b.tile_side;
  const int tile_area = side * side;
  for (int i = threadIdx.x; i < b.n_geoms * kCounters; i += blockDim.x)
    if (s_cnt[i]) tally_add(&b.counters[i], (unsigned long long)s_cnt[i]);
  for (int t = 0; t < b.n_tiles; ++t) {
    const GeomDev& gt = geoms[t];
    const int i0 = tile_origin(gt.xdim, side), j0 = tile_origin(gt.ydim, side);
    for (int e = threadIdx.x; e < tile_area; e += blockDim.x) {
      const uint32_t v = s_tile[t * tile_area + e];
      if (v) {
        const int ti = e / side;
        tally_add(&gt.prf[(size_t)(i0 + ti) * gt.ydim + (j0 + e - ti * side)],
                  (unsigned long long)v);
      }
    }
  }
}

template <bool MULTI, bool REC, bool RADIAL>
static void launch_one(const TransportArgs& a, dim3 grid, hipStream_t s) {
  const size_t smem =
      transport_dynamic_lds(MULTI, a.n_geoms, (size_t)a.n_tiles * a.tile_side * a.tile_side);
  hipLaunchKernelGGL((k_transport<MULTI, REC, RADIAL>), grid, dim3(kTransportThreads), smem, s, a,
                     a.geoms, a.events, a.photon_off);
}

hipError_t launch_transport(const TransportArgs& a, bool multi, bool record,
                            bool radial, int n_blocks, hipStream_t s) {
  const dim3 grid(n_blocks);
  if (radial) {
    if (multi) launch_one<true, false, true>(a, grid, s);
    else launch_one<false, false, true>(a, grid, s);
  } else if (multi) {
    if (record) launch_one<true, true, false>(a, grid, s);
    else launch_one<true, false, false>(a, grid, s);
  } else {
    if (record) launch_one<false, true, false>(a, grid, s);
    else launch_one<false, false, false>(a, grid, s);
  }
  return hipGetLastError();
}

template <bool MULTI, bool REC, bool RADIAL>
static int occupancy_of(size_t smem) {
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_transport<MULTI, REC, RADIAL>,
                                                   kTransportThreads, smem) != hipSuccess)
    return 1;
  return nb > 0 ? nb : 1;
}

template <bool MULTI, bool REC, bool RADIAL>
static size_t static_lds_of() {
  hipFuncAttributes at{};
  if (hipFuncGetAttributes(&at, reinterpret_cast<const void*>(&k_transport<MULTI, REC, RADIAL>)) !=
      hipSuccess)
    return 0;
  return at.sharedSizeBytes;
}

size_t transport_static_lds() {
  const size_t a = static_lds_of<true, false, false>();
  const size_t b = static_lds_of<true, true, false>();
  const size_t c = static_lds_of<true, false, true>();
  const size_t m = a > b ? a : b;
  return m > c ? m : c;
}

int transport_max_blocks_per_cu(bool multi, bool record, bool radial, size_t smem) {
  if (radial)
    return multi ? occupancy_of<true, false, true>(smem) : occupancy_of<false, false, true>(smem);
  if (multi)
    return record ? occupancy_of<true, true, false>(smem) : occupancy_of<true, false, false>(smem);
  return record ? occupancy_of<false, true, false>(smem) : occupancy_of<false, false, false>(smem);
}

// ------------------------------------------------ RANECU trajectory mode

template <class M>
__global__ void __launch_bounds__(64) k_trace_ranecu(
    const fd2_event* events, int64_t n, int64_t event_base, int32_t seed_input,
    const GeomDev* geoms, unsigned long long* counters,
    const unsigned long long* photon_off, fd2_photon* records) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const fd2_event ev = events[i];
  const GeomDev& g = geoms[ev.geom];
  uint32_t cnt[kCounters] = {0, 0, 0, 0, 0, 0, 0, 0};
  RanecuRng rng;
  ranecu_init(rng, (int)(event_base + i), seed_input);
  StepSink nosink{nullptr, nullptr, 0, 0, false};
  Photon p;
  start_photon(p, ev);
  if (ev.N > 0) emit_first_dir<RanecuRng, M>(rng, p, g);  // driver, normal stays 0
  for (int32_t k = 0; k < ev.N; ++k) {
    // direction and normal carry over from the previous photon's end
    const float ux = p.ux, uy = p.uy, uz = p.uz, nx = p.nx, ny = p.ny, nz = p.nz;
    start_photon(p, ev);
    p.ux = ux; p.uy = uy; p.uz = uz;
    p.nx = nx; p.ny = ny; p.nz = nz;
    cnt[FD2_C_GENERATED]++;
    for (;;) {
      photon_step<RanecuRng, false, M>(rng, p, g, &nosink);
      if (ended(p.fate)) break;
      if (p.fate == kTrapped) {
        cnt[FD2_C_REGEN]++;
        restart_trapped<RanecuRng, M>(rng, p, g, ev);
      }
    }
    cnt[fate_counter(p.fate)]++;
    const bool det = p.fate == kDetectOut;
    const Pixel x = det ? detected_pixel(p, g) : Pixel{0, 0};
    if (p.fate == kDetect) atomicAdd(&g.prf[pix_index(x, g)], 1ull);
    if (det && ev.hist >= 1 && ev.hist <= g.num_hist) atomicAdd(&g.hist[ev.hist - 1], 1u);
    if (records) {
      fd2_photon rec;
      rec.fate = p.fate;
      rec.pix = p.fate == kDetect ? pix_index(x, g) : -1;
      rec.x = det ? p.px : 0.0f;
      rec.y = det ? p.py : 0.0f;
      records[photon_off[i] + k] = rec;
    }
    // next photon's direction and normal draws (main/kernel_cuda_c_ver1_0.cu:578-602)
    emit_dir<RanecuRng, M>(rng, p, g);
    if (g.beta > 0.0f) {
      (void)rng.u();
      (void)rng.u();
    }
  }
  unsigned long long* c = counters + (size_t)ev.geom * kCounters;
  for (int j = 0; j < kCounters; ++j)
    if (cnt[j]) atomicAdd(&c[j], (unsigned long long)cnt[j]);
}

hipError_t launch_trace_ranecu(const fd2_event* events, int64_t n,
                               int64_t event_base, int32_t seed_input,
                               const GeomDev* geoms, int32_t n_geoms,
                               unsigned long long* counters,
                               const unsigned long long* photon_off,
                               fd2_photon* records, bool faithful, hipStream_t s) {
  (void)n_geoms;
  if (n <= 0) return hipSuccess;
  const int64_t nb = (n + 63) / 64;
  if (faithful)
    hipLaunchKernelGGL(k_trace_ranecu<MathFaithful>, dim3((unsigned)nb), dim3(64), 0, s, events,
                       n, event_base, seed_input, geoms, counters, photon_off, records);
  else
    hipLaunchKernelGGL(k_trace_ranecu<MathDevice>, dim3((unsigned)nb), dim3(64), 0, s, events,
                       n, event_base, seed_input, geoms, counters, photon_off, records);
  return hipGetLastError();
}

// ----------------------------------------------------- step trace (debug)

__global__ void __launch_bounds__(64) k_debug_steps(
    const fd2_event* events, uint64_t event_base, uint32_t seed,
    const GeomDev* geoms, int32_t n_photons, float* steps, int32_t* n_steps,
    int32_t max_steps) {
  const int32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  const fd2_event ev = events[0];
  if (k >= n_photons || k >= ev.N) return;
  const GeomDev& g = geoms[ev.geom];
  StepSink sink{steps, n_steps, max_steps, k, true};
  Photon p;
  CounterRng rng;
  start_photon(p, ev);
  rng.seed(seed, event_base, (uint32_t)k);
  counter_initial_dir(rng, p, (uint32_t)k, g);
  for (;;) {
    photon_step<CounterRng, true>(rng, p, g, &sink);
    if (ended(p.fate)) break;
    if (p.fate == kTrapped) restart_trapped(rng, p, g, ev);
  }
}

hipError_t launch_debug_steps(const fd2_event* events, uint64_t event_base,
                              uint32_t seed, const GeomDev* geoms,
                              int32_t n_photons, float* steps,
                              int32_t* n_steps, int32_t max_steps,
                              hipStream_t s) {
  if (n_photons <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_debug_steps, dim3((n_photons + 63) / 64), dim3(64), 0, s,
                     events, event_base, seed, geoms, n_photons, steps, n_steps,
                     max_steps);
  return hipGetLastError();
}

// Device arithmetic on its own: y[i] = f(x[i]) for the functions the
// transport uses, numbered as FD2_MATH_* (the oracle evaluates the same
// functions on the CPU, so the two can be compared bit for bit).
__global__ void k_debug_math(int fn, const float* x, float* y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float v = x[i];
  float r;
  float sn, cs;
  switch (fn) {
    case FD2_MATH_SIN: r = fd2_sin(v); break;
    case FD2_MATH_COS: r = fd2_cos(v); break;
    case FD2_MATH_LOG: r = fd2_log(v); break;
    case FD2_MATH_ASIN: r = fd2_asin(v); break;
    case FD2_MATH_ACOS: r = fd2_acos(v); break;
    case FD2_MATH_SIN_TURNS: fd2_sincos_turns(v, &sn, &cs); r = sn; break;
    case FD2_MATH_COS_TURNS: fd2_sincos_turns(v, &sn, &cs); r = cs; break;
    case FD2_MATH_RSQRT: r = fd2_rsqrt(v); break;
    case FD2_MATH_SQRT_UNIT: r = fd2_sqrt_unit(v); break;
    case FD2_MATH_ANGLE_OVER_157: r = angle_over_157(v) ? 1.0f : 0.0f; break;
    case FD2_MATH_ACOSF_LIBC: r = fd2x_acosf(v); break;
    case FD2_MATH_ASINF_LIBC: r = fd2x_asinf(v); break;
    case FD2_MATH_FF_SIN: r = fd2x_sin(v).hi; break;
    case FD2_MATH_FF_COS: r = fd2x_cos(v).hi; break;
    case FD2_MATH_FF_LOG: r = fd2x_log(v).hi; break;
    case FD2_MATH_SQRT_01: r = fd2_sqrt_01(v); break;
    case FD2_MATH_SQRT_POS: r = fd2_sqrt_pos(v); break;
    case FD2_MATH_RECIP: r = fd2_recip(v); break;
    case FD2_MATH_DIV: r = fd2_div(0.7310586f, v); break;
    case FD2_MATH_SIN_QUARTERS: fd2_sincos_quarters(4.0f * v, &sn, &cs); r = sn; break;
    case FD2_MATH_COS_QUARTERS: fd2_sincos_quarters(4.0f * v, &sn, &cs); r = cs; break;
    default: r = 0.0f; break;
  }
  y[i] = r;
}

hipError_t launch_debug_math(int fn, const float* x, float* y, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_debug_math, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, fn, x, y,
                     n);
  return hipGetLastError();
}

// ------------------------------------------------------------- fills

__global__ void k_fill_u64(unsigned long long* p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0ull;
}
__global__ void k_fill_u32(uint32_t* p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

hipError_t launch_fill_u64(unsigned long long* p, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const size_t nb = (n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096;
  hipLaunchKernelGGL(k_fill_u64, dim3((unsigned)nb), dim3(256), 0, s, p, n);
  return hipGetLastError();
}
hipError_t launch_fill_u32(uint32_t* p, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const size_t nb = (n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)nb), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

__global__ void k_set_u32(uint32_t* p, uint32_t v) {
  if (threadIdx.x == 0) p[0] = v;
}

hipError_t launch_set_u32(uint32_t* p, uint32_t v, hipStream_t s) {
  hipLaunchKernelGGL(k_set_u32, dim3(1), dim3(64), 0, s, p, v);
  return hipGetLastError();
}

__global__ void k_set_u64(unsigned long long* p, unsigned long long v) {
  if (threadIdx.x == 0) p[0] = v;
}

hipError_t launch_set_u64(unsigned long long* p, unsigned long long v, hipStream_t s) {
  hipLaunchKernelGGL(k_set_u64, dim3(1), dim3(64), 0, s, p, v);
  return hipGetLastError();
}

}  // namespace fd2
