// fd2_internal.h -- declarations shared by the host library and the kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/fd2.h"
#include "fd2_device.h"
#include "fd2_hostcopy.h"

namespace fd2 {

enum { kCounters = FD2_NCOUNT };

// How a launch's photons are handed out, made by the queue build.
struct QueuePlan {
  uint32_t cursor;      // spans taken so far
  uint32_t span_log2;   // photons per span
  uint32_t lane_cap;    // lanes of a wave that take photons
  uint32_t blocks;      // workgroups of the transport that take part
};

struct TransportArgs {
  // geometry 0, first in the kernel's arguments: with one geometry its
  // constants are one scalar load away, not two
  GeomDev geom0;
  const fd2_event* events;             // device
  const unsigned long long* photon_off;  // n_events + 1 (exclusive scan)
  const GeomDev* geoms;                // n_geoms
  unsigned long long* counters;        // n_geoms * FD2_NCOUNT
  QueuePlan* plan;
  fd2_photon* records;                 // per-photon records (recording only)
  uint32_t* radial;                    // n_events x FD2_RADIAL_BINS (radial mode)
  const unsigned long long* event_base_dev;  // if set, read the number of events[0] here
  uint32_t* wave_queue;                // per-wave photon queues
  int32_t queues;                      // use them (0: park in place)
  uint32_t* error_flag;                // bit 1: a wave's loop limit was reached
  int64_t n_events;
  uint32_t seed;
  uint64_t event_base;                 // global number of events[0]
  int32_t n_geoms;
  int32_t park_lanes;                  // lanes waiting before a Fresnel phase
  int32_t refill_lanes;                // free lanes before new photons start
  int32_t tile_side;                   // LDS PRF tile side (pixels), 0 = none
  int32_t n_tiles;                     // geometries [0, n_tiles) have a tile
};

// LDS PRF tiles of the persistent kernel: geometry g < n_tiles counts the
// detections in a tile_side^2 pixel square centred on its PRF image in LDS
// (u32) and adds the block's counts to the PRF at the end.
constexpr int kTileDefault = 0;  // no tile: the LDS holds the wall queues
constexpr int kTileBudget = 64 * 64;   // u32 entries per block (16 KiB)
// per-wave photon queues of the persistent kernel: photons waiting for the
// wall branch (at most 63) and photons ready to step in LDS, together at most
// kLdsCap (so that new photons start at least 33 at a time, the last of a span
// excepted), and 8 slots to write before reading; the gap queue and the backlog in HBM (slots
// in that order).  At most 64 + kLdsCap + kGapCap photons are in flight per
// wave.
constexpr int kLdsCap = 96;
constexpr int kWallSlots = kLdsCap + 8;
constexpr int kGapCap = 128;
constexpr int kBackCap = 64 + kLdsCap + kGapCap;
constexpr int kGapBase = 0;
constexpr int kBackBase = kGapCap;
constexpr int kQSlots = kGapCap + kBackCap;
constexpr int kQWords = 20;  // 16 photon words + 4 of wall-branch state
constexpr int kQBlock = 32;  // queue slots per block (word stride 128 bytes)
// ended photons that wait to be counted: 63 between rounds, and at most every
// photon in flight ends in one; 5 words each, kEndCap apart
constexpr int kEndCap = 64 + 64 + kLdsCap + kGapCap;
constexpr int kWaveWords = kQWords * kQSlots + 5 * kEndCap;
static_assert(kQSlots % kQBlock == 0 && kGapBase % kQBlock == 0 && kBackBase % kQBlock == 0,
              "queue regions are whole blocks");
constexpr uint32_t kMaxIdlePasses = 256;  // passes without a step or a wall branch
// largest LDS tile side: 49 KiB of tile, plus the kernel's static LDS (26 to 29
// KiB, transport_lds_bytes) and the table of several geometries; fd2_set_tuning checks
// the sum against the device's LDS per workgroup (160 KiB on gfx950)
constexpr int kTileMax = 112;

struct QueueArgs {
  const fd2_event* events;
  unsigned long long* photon_off;
  uint32_t* block_chunks;      // per scan block
  unsigned long long* block_photons;
  QueuePlan* plan;
  uint32_t* error_flag;        // set when an event is invalid
  int64_t n_events;
  int32_t n_geoms;
  int32_t chunk_log2;
  int32_t n_blocks;
  uint32_t n_waves;            // waves of the transport launch
  uint32_t n_simds;            // SIMDs of the device
  uint64_t max_chunks;         // more work items than this: error bit 4, nothing runs
};

constexpr int kScanThreads = 1024;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;
constexpr int kTransportThreads = 256;

// static LDS of the transport: the waves' photon queues, the lanes' history runs
// and the counters; per CU it leaves room for 6 workgroups (one geometry) and 5
// (a short table of several, or records)
constexpr size_t transport_lds_bytes(bool multi, bool record) {
  return sizeof(uint32_t) * ((size_t)(kTransportThreads / 64) * (14 + multi + record) * kWallSlots +
                             2 * kTransportThreads + FD2_MAX_GEOMS * kCounters);
}
constexpr size_t kLdsPerCu = 160 * 1024;
static_assert(transport_lds_bytes(false, false) == 26496 && 6 * transport_lds_bytes(false, false) <= kLdsPerCu);
static_assert(transport_lds_bytes(true, false) == 28160 && transport_lds_bytes(true, true) == 29824 &&
              5 * (transport_lds_bytes(true, true) + 16 * sizeof(GeomDev)) <= kLdsPerCu);
static_assert(sizeof(GeomDev) == 168);

// dynamic LDS of the transport: the geometry table (several geometries) and
// `tile_words` words of PRF tiles
inline size_t transport_dynamic_lds(bool multi, int n_geoms, size_t tile_words) {
  return (multi ? (size_t)n_geoms * sizeof(GeomDev) : 0) + tile_words * sizeof(uint32_t);
}

// launch wrappers (fd2_kernels.hip)
hipError_t launch_queue_build(const QueueArgs& q, hipStream_t s);
hipError_t launch_transport(const TransportArgs& a, bool multi, bool record,
                            bool radial, int n_blocks, hipStream_t s);
hipError_t launch_trace_ranecu(const fd2_event* events, int64_t n,
                               int64_t event_base, int32_t seed_input,
                               const GeomDev* geoms, int32_t n_geoms,
                               unsigned long long* counters,
                               const unsigned long long* photon_off,
                               fd2_photon* records, bool faithful, hipStream_t s);
hipError_t launch_debug_steps(const fd2_event* events, uint64_t event_base,
                              uint32_t seed, const GeomDev* geoms,
                              int32_t n_photons, float* steps,
                              int32_t* n_steps, int32_t max_steps,
                              hipStream_t s);
hipError_t launch_debug_math(int fn, const float* x, float* y, int64_t n, hipStream_t s);
hipError_t launch_fill_u64(unsigned long long* p, size_t n, hipStream_t s);
hipError_t launch_fill_u32(uint32_t* p, size_t n, hipStream_t s);
hipError_t launch_set_u32(uint32_t* p, uint32_t v, hipStream_t s);
hipError_t launch_set_u64(unsigned long long* p, unsigned long long v, hipStream_t s);
int transport_max_blocks_per_cu(bool multi, bool record, bool radial, size_t smem);
size_t transport_static_lds();  // largest static LDS of the transport kernels

}  // namespace fd2

// The transport context (host side).
struct fd2_ctx {
  int device = 0;
  int n_cu = 0;
  size_t lds_per_block = 0;   // the device's LDS per workgroup
  size_t lds_static = 0;      // the transport kernels' static LDS (largest)
  hipStream_t stream = nullptr;
  hipEvent_t ev_start = nullptr, ev_stop = nullptr;
  bool timed = false;

  int n_geoms = 0;
  fd2_params params[FD2_MAX_GEOMS];
  fd2::GeomDev hgeom[FD2_MAX_GEOMS];
  fd2::GeomDev* d_geoms = nullptr;
  unsigned long long* d_prf[FD2_MAX_GEOMS] = {};
  uint32_t* d_hist[FD2_MAX_GEOMS] = {};
  unsigned long long* d_counters = nullptr;

  // staging and queue buffers, grown on demand
  fd2::HostCopy copy;             // to and from the caller's memory
  fd2_event* d_events = nullptr;
  size_t cap_events = 0;
  unsigned long long* d_photon_off = nullptr;
  size_t cap_off = 0;
  uint32_t* d_block_chunks = nullptr;
  unsigned long long* d_block_photons = nullptr;
  size_t cap_blocks = 0;
  fd2::QueuePlan* d_plan = nullptr;
  uint32_t* d_error = nullptr;
  uint32_t* d_wave_queue = nullptr;    // kWaveWords words per resident wave
  int max_waves = 0;

  uint32_t seed = 271828182u;
  int64_t next_event = 0;
  fd2_tuning tune{};
};

namespace fd2 {

// Stage n events through the context's pinned buffer and enqueue their
// transport, with per-event radial tallies into d_radial (n x
// FD2_RADIAL_BINS u32, cleared here), on the context's stream without
// waiting for it: the events take the next n event numbers, as in
// fd2_submit_radial, and fd2_sync waits for them and checks the error flag.
int submit_radial_async(fd2_ctx* c, const fd2_event* events, int64_t n, uint32_t* d_radial);

}  // namespace fd2
