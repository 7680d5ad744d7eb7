// vh_kernels.hip - gfx950 kernels of libvh.
//
// Per batch of k consecutive frames: k_alloc (one lane per
// pixel of each frame: truncation-band DDA, hash insert, per-frame marks, compaction of the
// batch's block list) -> k_integrate (one wave per listed block, grid-stride: the block's
// voxels are read once, updated by each frame that touched it, written once; the last
// workgroup to finish closes the batch). Bound sequences run k_integrate_alloc: batch b is
// integrated while batch b+1 is allocated.
// Extraction: k_mc (one workgroup per pool block; 9^3 halo in LDS; wave prefix sums).
// Queries: k_query / k_backward / k_gn_accum + k_gn_solve (FP64 reductions).
//
// Kernel code follows the op order of vh_math.h exactly and is compiled with
// -ffp-contract=off, so FP32 results match a CPU twin of the same algorithm bit-for-bit.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "vh.h"
#include "vh_internal.h"
#include "vh_math.h"
#include "vh_mc_table.h"

namespace vh {

namespace {

__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
__device__ __forceinline__ uint32_t read_lane_u32(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ int first_lane(uint64_t m) { return __ffsll((unsigned long long)m) - 1; }
// A value every lane holds identically, moved to a scalar register.
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ unsigned long long uniform64(unsigned long long v) {
  return (unsigned long long)uniform((uint32_t)v) | (unsigned long long)uniform((uint32_t)(v >> 32)) << 32;
}

__device__ __forceinline__ void raise_flag(FrameCtl* ctl, uint32_t f) { atomicOr(&ctl->flags, f); }


// Lock-free find-or-insert. A key is written once into the first empty slot of its probe
// sequence by a compare-and-swap; a stale cached read can only show EMPTY where a key now
// lives, and the CAS then returns the real occupant, so no lane ever spins on another.
// Returns the slot id (or -1 when the probe limit is exhausted); `inserted` is set for the
// lane whose CAS created the key.
__device__ __forceinline__ int64_t find_or_insert(const HashView& h, uint64_t key, bool& inserted) {
  uint64_t b = bucket_of(key, h.log2_buckets);
  for (int p = 0; p < kMaxProbe; ++p) {
    unsigned long long* bk = h.keys + b * kSlotsPerBucket;
    const ulonglong2* bp = reinterpret_cast<const ulonglong2*>(bk);
    const ulonglong2 k01 = bp[0], k23 = bp[1];
    const uint64_t ks[4] = {k01.x, k01.y, k23.x, k23.y};
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (ks[s] == key) return (int64_t)(b * kSlotsPerBucket + s);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (ks[s] != kEmptyKey) continue;
      const unsigned long long old = atomicCAS(bk + s, (unsigned long long)kEmptyKey, (unsigned long long)key);
      if (old == kEmptyKey) {
        inserted = true;
        return (int64_t)(b * kSlotsPerBucket + s);
      }
      if (old == key) return (int64_t)(b * kSlotsPerBucket + s);
    }
    b = (b + 1) & h.bucket_mask;
  }
  return -1;
}

template <bool kU16>
__device__ __forceinline__ float depth_at(const void* base, float scale, int pix) {
  if (kU16) return (float)reinterpret_cast<const uint16_t*>(base)[(uint32_t)pix] * scale;
  return reinterpret_cast<const float*>(base)[(uint32_t)pix];
}

// ============================================================================ host images
// A small image from page-locked host memory, read over the bus by the lanes themselves. Through the
// copy engine on a second stream a queued frame cost the host 64 us, most of it for the copy's and the
// kernels' waits for each other; in the kernels' own stream it costs its time on the bus (640 x
// 480 uint16: 15 us) and a launch. System-scope loads: the host writes this memory between frames.
// Units of 8 bytes from the source's first multiple of 8, the bytes before and after apart (a load is a
// request of its own on the bus: queued frames of 511 x 383 uint16 took 43 us in units of 2 bytes, 37 so, of
// 511 x 383 float 51 us in units of 4, 46 so); the destination, a slot that starts where the one before
// ends, is written unaligned.
__global__ __launch_bounds__(256) void k_copy_in(char* dst, const char* src, size_t bytes) {
  const size_t before = min(bytes, (size_t)(-reinterpret_cast<uintptr_t>(src) & 7u)), n = (bytes - before) / 8;
  const uint64_t* units = reinterpret_cast<const uint64_t*>(src + before);
  for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += gridDim.x * (size_t)256) {
    const uint64_t x = __hip_atomic_load(units + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_memcpy(dst + before + 8 * i, &x, 8);
  }
  if (blockIdx.x == 0 && threadIdx.x < bytes - 8 * n) {  // the first `before` bytes, then the last
    const size_t at = threadIdx.x < before ? threadIdx.x : 8 * n + threadIdx.x;
    dst[at] = __hip_atomic_load(src + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Device words into page-locked host memory, where the copy engine and its hand-over take longer.
__global__ __launch_bounds__(256) void k_words_out(uint32_t* dst, const uint32_t* a, int na, const uint32_t* b, int nb) {
  for (int k = threadIdx.x; k < na + nb; k += 256)
    __hip_atomic_store(dst + k, k < na ? a[k] : b[k - na], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ============================================================================ allocation
// Workgroup = a tile of 64 x 16 pixels (16 x 16 in a single frame's launch), 256 lanes, each lane
// one pixel in each of the tile's 16 x 16 bands, so a workgroup reads and writes whole cache lines
// of the image rows. Phase 1: the blocks that the pixels' truncation bands cross go into an LDS hash
// set, so each distinct block of the tile is kept once. Phase 2: the distinct keys go to the global
// hash (find or insert), take a pool index if new, and mark the block for this frame of the batch
// (an atomic OR of the frame's bit into the slot's mark); the lanes that found the mark empty append
// the slot to the workgroup's stripe of the batch's block list, and the lanes that found their
// frame's bit clear count the block for that frame.
// What bounds it: vector issue (about 270 instructions per wave and band) with the latency of the
// set and of phase 2's four dependent round trips between. 8 frames of 640 x 480 launched alone:
// 5 mm 42.6 -> 32.3 us, 1 cm 37.9 -> 28.1 us against a walk per lane with a compare-and-swap per key
// (a launch without the bands takes 7.7 us, without the set 22.6).
constexpr int kSetSlots = 1024;  // LDS key set (8 KB)
// 16 x 16 bands per tile of a batched launch. One workgroup per four bands pays the LDS clear,
// the barriers and the chain of dependent global atomics of phase 2 once for all four, and
// merges the bands' keys: 500 frames at 5 mm take 6.41 ms with 2 bands, 6.00 with 4, 6.01 with 5. A
// single frame's launch keeps one band per workgroup, which fills the GPU with 4x as many
// workgroups.
constexpr int kAllocBands = 4;
__host__ __device__ constexpr uint32_t alloc_tiles(int W, int H, int bands) {
  return (uint32_t)(((W + 16 * bands - 1) / (16 * bands)) * ((H + 15) >> 4));
}

// Home slot of a packed key in a tile's set. pack_key is linear in the block coordinates, so a step
// along an axis adds a constant (key_step).
static_assert(kSetSlots == 1 << 10, "set_hash gives 10 bits");
__device__ __forceinline__ uint32_t set_hash(uint64_t key) {
  return (((uint32_t)key ^ (uint32_t)(key >> 32)) * 0x9e3779b1u) >> 22;
}
__device__ __forceinline__ uint64_t key_step(int dx, int dy, int dz) {
  return ((uint64_t)(int64_t)dx << (2 * kKeyBits)) + ((uint64_t)(int64_t)dy << kKeyBits) + (uint64_t)(int64_t)dz;
}

// The block list, its stripe lengths and the slot marks are double-buffered by batch
// parity, so the allocation of batch b+1 can run while batch b is integrated. Line s of a
// parity's counters: word 0 = listed blocks of stripe s, word 1 + j = blocks that frame j of
// the batch touched first in that stripe.
__device__ __forceinline__ uint32_t* list_count_of(FrameCtl* ctl, uint32_t parity) {
  return ctl->tcount + parity * (kStripes * kLine);
}
__device__ __forceinline__ uint32_t* list_of(const FrameArgs& a, uint32_t parity) {
  return a.touched + (size_t)parity * kStripes * a.stripe_cap;
}
__device__ __forceinline__ uint32_t* marks_of(const FrameArgs& a, uint32_t parity) {
  return a.marks + (size_t)parity * a.n_slots;
}
// Input slot of frame j of a batch whose first frame is input `cur` (consecutive, wrapping).
__device__ __forceinline__ uint32_t input_slot(uint32_t cur, uint32_t j, uint32_t n_seq) {
  uint32_t fs = cur % n_seq + j;
  while (fs >= n_seq) fs -= n_seq;
  return fs;
}

// Global part for the active lanes' keys: find-or-insert, pool index for new keys (one
// atomic per wave), the frame's mark, the list append and the frame's count (one atomic per
// wave each). `frame` is the frame's id (stored as the birth frame of new blocks), jb its
// index in the batch.
__device__ void claim_keys(const FrameArgs& a, uint64_t key, bool act, uint32_t frame, uint32_t jb,
                           uint32_t parity, int lane, uint32_t stripe) {
  FrameCtl* ctl = a.ctl;
  bool inserted = false;
  int64_t slot = -1;
  if (act) {
    slot = find_or_insert(a.hash, key, inserted);
    if (slot < 0) raise_flag(ctl, kFlagHashFull);
  }
  // The pool reservation and the mark depend only on the slot: both are in flight together,
  // and the slot-value stores go out just before the stripe atomics, so the chain is bucket
  // load -> (CAS) -> pool + mark -> stripe.
  const uint64_t im = __ballot(inserted);
  const int leader = im ? first_lane(im) : 0;
  uint32_t pbase = 0;
  if (im && lane == leader) pbase = atomicAdd(&ctl->pool_count, (uint32_t)__popcll(im));
  const uint32_t bit = 1u << jb;
  uint32_t old_mark = bit;
  if (slot >= 0) old_mark = atomicOr(&marks_of(a, parity)[slot], bit);
  if (im) {
    pbase = read_lane_u32(pbase, leader);
    if (inserted) {
      const uint32_t idx = pbase + lanes_below(im);
      uint32_t stored = kNoBlock;
      if (idx < a.pool_cap) {
        a.block_keys[idx] = key;
        a.block_info[idx] = (unsigned long long)slot | ((unsigned long long)frame << 32);
        stored = idx;
      } else {
        raise_flag(ctl, kFlagPoolFull);
      }
      a.hash.vals[slot] = (unsigned long long)stored | ((unsigned long long)frame << 32);
    }
  }
  uint32_t* line = list_count_of(ctl, parity) + stripe * kLine;
  const uint64_t cm = __ballot((old_mark & bit) == 0u);  // first touch of the block by this frame
  if (cm && lane == first_lane(cm)) atomicAdd(&line[1 + jb], (uint32_t)__popcll(cm));
  const bool first = old_mark == 0u;  // first touch by the batch: list the block
  const uint64_t fm = __ballot(first);
  if (fm) {
    const int fl = first_lane(fm);
    uint32_t tbase = 0;
    if (lane == fl) tbase = atomicAdd(&line[0], (uint32_t)__popcll(fm));
    tbase = read_lane_u32(tbase, fl);
    if (first) {
      const uint32_t pos = tbase + lanes_below(fm);
      if (pos < a.stripe_cap) {
        list_of(a, parity)[(size_t)stripe * a.stripe_cap + pos] = (uint32_t)slot;
      } else {
        // the block cannot be listed: its mark goes back to zero, so that a later lane of this
        // batch that marks it tries to list it again, and no mark outlives the batch unlisted
        atomicExch(&marks_of(a, parity)[slot], 0u);
        raise_flag(ctl, kFlagTouchedFull);
      }
    }
  }
}

// The allocation's LDS: the key set, the tile's distinct keys and, for carving volumes, the
// bands' largest depths.
template <int kBands>
struct AllocLds {
  unsigned long long set[kSetSlots];
  unsigned long long uniq[kSetSlots];
  uint32_t nuniq;
  float tmax[4][kBands];
};

// Puts the active lanes' keys into the tile's set; a key new to the set joins the list of distinct
// keys (at most one entry per slot). True for lanes whose key found no room within 32 probes. A
// probe reads before it swaps: a key that is there is found by a read, which serves equal keys of
// the wave at once.
template <int kBands>
__device__ __forceinline__ bool set_insert(AllocLds<kBands>& L, unsigned long long key, bool act) {
  bool spill = act;
  if (act) {
    uint32_t h = set_hash(key);
#pragma unroll 1
    for (int p = 0; p < 32; ++p) {
      unsigned long long old = __hip_atomic_load(&L.set[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (old == kEmptyKey) {
        old = atomicCAS(&L.set[h], (unsigned long long)kEmptyKey, key);
        if (old == kEmptyKey) L.uniq[atomicAdd(&L.nuniq, 1u)] = key;
      }
      if (old == key || old == kEmptyKey) { spill = false; break; }
      h = (h + 1) & (kSetSlots - 1);
    }
  }
  return spill;
}

// x of another lane of the row of 16 (DPP control kCtrl).
template <int kCtrl>
__device__ __forceinline__ int32_t dpp(int32_t x) { return __builtin_amdgcn_mov_dpp(x, kCtrl, 0xf, 0xf, false); }
// Windows of a wave's pixels in a single frame's launch; the lanes left then walk. Near surfaces are done
// with one or two windows, far and noisy ones would need many of few lanes each, where a walk is
// the faster. Launch times in us with at most 0 / 1 / 2 / 3 / any number of windows: a small room at 1 cm 9.5 / 8.2 / 8.3 /
// 8.3 / 8.3, a room at 5 mm 9.4 / 10.0 / 9.9 / 9.7 / 9.6, at 4 mm 9.3 / 10.3 / 10.5 / 10.3 / 9.9, a floor at 4 mm 9.8 / 11.4 /
// 12.6 / 13.5 / 15.3, tracked 14.4 / 14.8 / 15.1 / 15.7 / 17.2; and a frame of the small room with its
// integration, one by one, 19.1 with 0, 19.4 with 1, 18.6 with 2 or 3. A batch's launch, with four bands per workgroup, is 1 to 3 %
// slower with a limit.
constexpr int kMaxWindows = 2;

// OR of x over the wave's lanes (in every lane's result; DPP within rows of 16, then the rows').
__device__ __forceinline__ uint32_t wave_or(uint32_t x) {
  x |= (uint32_t)dpp<0xB1>((int32_t)x);
  x |= (uint32_t)dpp<0x4E>((int32_t)x);
  x |= (uint32_t)dpp<0x141>((int32_t)x);
  x |= (uint32_t)dpp<0x140>((int32_t)x);
  return read_lane_u32(x, 0) | read_lane_u32(x, 16) | read_lane_u32(x, 32) | read_lane_u32(x, 48);
}

// The distinct blocks of a tile's bands, claimed. A wave's 8 x 8 pixels cross a handful of
// blocks near one another, so they are gathered as bits: the window is the 4 x 4 x 4 blocks
// around one lane's band, every lane whose band lies in it sets the bits of its blocks in a
// 64-bit word, the words are ORed over the wave, and lane i then holds block i of the window
// where its bit is set: at most one key per lane, all distinct, go to the tile's set in one round
// (each lane's keys in turn took a round trip and its mask arithmetic per key: 12 of 36 us of a
// batch of 8 frames launched alone). Lanes outside take the next window.
// The blocks of a band that moves at most one block per axis are known without a walk: the
// first; the first after one step along the axis crossed first; the last before the step along
// the axis crossed last; the last (band_next's order: smallest crossing parameter first, ties to
// the lower axis). Bands of two blocks along an axis walk within the window, longer ones
// (truncations of more than four voxels) insert block by block.
template <int kBands>
__device__ __forceinline__ void tile_bands(const FrameArgs& a, const float* T, const float* dr, int u0, int v,
                                           uint32_t frame, uint32_t jb, uint32_t parity, uint32_t stripe,
                                           AllocLds<kBands>& L) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // lane i's block of a window: (i >> 4, (i >> 2) & 3, i & 3) from its corner
  const uint64_t lane_off = key_step(lane >> 4, (lane >> 2) & 3, lane & 3);
#pragma unroll 1
  for (int r = 0; r < kBands; ++r) {
    const int u = u0 + 16 * r;
    bool active = u < a.W && v < a.H && depth_valid(dr[r], a.max_depth);
    if (!__ballot(active)) continue;
    float A[3], B[3];
    const bool in_range = band_segment(T, a.K, a.band, a.mu, a.min_depth, u, v, dr[r], A, B);
    if (active && !in_range) raise_flag(a.ctl, kFlagRange);
    active = active && in_range;
    BandDDA s;
    band_start(A, B, s, [](float x) { return recip_rn(x); });
    const int sx = s.ex - s.ix, sy = s.ey - s.iy, sz = s.ez - s.iz;
    const int reach = max(max(abs(sx), abs(sy)), abs(sz)), moves = abs(sx) + abs(sy) + abs(sz);
    // one-block moves: the faces' crossing parameters (band_t), infinite along an axis that stays
    const float tx = sx ? ((float)max(s.ix, s.ex) - s.ax) * s.rx : INFINITY;
    const float ty = sy ? ((float)max(s.iy, s.ey) - s.ay) * s.ry : INFINITY;
    const float tz = sz ? ((float)max(s.iz, s.ez) - s.az) * s.rz : INFINITY;
    const int bx = 16 * sx, by = 4 * sy, bz = sz;  // steps in window bits
    const int b_first = tx <= ty && tx <= tz ? bx : (ty <= tz ? by : bz);
    const int b_last = tz >= tx && tz >= ty ? bz : (ty >= tx ? by : bx);  // used where all three move
    uint64_t left = __ballot(active && reach <= 2);
    bool walking = active && reach > 2;
    for (int windows = 0;; ++windows) {
      uint64_t key;
      bool want;
      if (left && (kBands > 1 || windows < kMaxWindows)) {
        const int lead = (left >> 27) & 1u ? 27 : first_lane(left);  // a lane in the middle if it can be
        const int wx = __builtin_amdgcn_readlane(min(s.ix, s.ex), lead) - 1,
                  wy = __builtin_amdgcn_readlane(min(s.iy, s.ey), lead) - 1,
                  wz = __builtin_amdgcn_readlane(min(s.iz, s.ez), lead) - 1;
        const int x0 = s.ix - wx, y0 = s.iy - wy, z0 = s.iz - wz;
        const bool in = __builtin_amdgcn_inverse_ballot_w64(left) &&
                        (uint32_t)((x0 | y0 | z0) | ((x0 + sx) | (y0 + sy) | (z0 + sz))) < 4u;
        const int i0 = 16 * x0 + 4 * y0 + z0, i3 = i0 + ((bx + by) + bz);
        uint64_t bits = 0u;
        if (in) {
          bits = (1ull << (i0 & 63)) | (1ull << (i3 & 63));
          if (moves > 1) bits |= 1ull << ((i0 + b_first) & 63);
          if (moves > 2) bits |= 1ull << ((i3 - b_last) & 63);
        }
        const bool two = in && reach > 1;
        if (__ballot(two)) {
          BandDDA w = s;
          bool more = two;
          if (two) bits = 0u;
          while (__ballot(more)) {
            if (more) {
              bits |= 1ull << ((16 * (w.ix - wx) + 4 * (w.iy - wy) + (w.iz - wz)) & 63);
              more = band_next(w);
            }
          }
        }
        want = __builtin_amdgcn_inverse_ballot_w64((uint64_t)wave_or((uint32_t)bits) |
                                                   (uint64_t)wave_or((uint32_t)(bits >> 32)) << 32);
        key = pack_key(wx, wy, wz) + lane_off;
        left &= ~__ballot(in);
      } else {
        walking = walking || __builtin_amdgcn_inverse_ballot_w64(left);
        left = 0u;
        if (!__ballot(walking)) break;
        key = pack_key(s.ix, s.iy, s.iz);
        want = walking;
        if (walking) walking = band_next(s);
      }
      const uint64_t home = __hip_atomic_load(&L.set[set_hash(key)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      const bool need = want && home != key;
      if (__ballot(need)) {
        const bool spill = set_insert(L, key, need);
        if (__ballot(spill)) claim_keys(a, key, spill, frame, jb, parity, lane, stripe);
      }
    }
  }
  __syncthreads();
  // the tile's distinct keys
  const uint32_t n = L.nuniq;
  for (uint32_t b0 = 0; b0 < n; b0 += 256) {
    const uint32_t i = b0 + tid;
    const bool act = i < n;
    const uint32_t wave_first = b0 + (uint32_t)(wave << 6);
    if (wave_first >= n) break;  // whole wave idle (uniform per wave)
    claim_keys(a, act ? L.uniq[i] : kEmptyKey, act, frame, jb, parity, lane, stripe);
  }
}

// Allocation of one tile of frame `frame` (index jb of its batch, input slot fs): 16 pixel
// rows by 16 * kBands columns, 256 lanes, each lane one pixel of every 16 x 16 band (a wave 8 x 8
// of them).
// kColor: the volume keeps colour (a.rgba is set), known at compile time so that no branch
// separates the tile's loads.
template <bool kU16, int kBands, bool kColor>
__device__ void alloc_tile(const FrameArgs& a, uint32_t tile, uint32_t frame, uint32_t jb, uint32_t parity,
                           uint32_t fs, AllocLds<kBands>& L) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int tiles_x = (a.W + 16 * kBands - 1) / (16 * kBands);
  const int tx = (int)(tile % tiles_x), ty = (int)(tile / tiles_x);
  const int u0 = tx * (16 * kBands) + ((wave & 1) << 3) + (lane & 7);
  const int v = ty * 16 + ((wave >> 1) << 3) + (lane >> 3);
  const uint32_t stripe = tile & (kStripes - 1);
  float T[12];
  if (kBands > 1 || a.poses) {  // a host frame is a launch of its own
#pragma unroll
    for (int k = 0; k < 12; ++k) T[k] = a.poses[16 * (size_t)fs + k];
  } else {
#pragma unroll
    for (int k = 0; k < 12; ++k) T[k] = a.pose[k];
  }
  const size_t elem = kU16 ? 2 : 4;
  const void* base = reinterpret_cast<const char*>(a.depth) + (size_t)fs * a.W * a.H * elem;

  // the lane's depths (and colours) of all bands: every load is issued before the first use
  // (a pixel outside the image loads a pixel inside it, whose value is not used), so the loads
  // are in flight together
  float dr[kBands];
  uint32_t px3[kBands][3];
  const int vc = min(v, a.H - 1);
#pragma unroll
  for (int r = 0; r < kBands; ++r) {
    const int uc = min(u0 + 16 * r, a.W - 1);
    dr[r] = depth_at<kU16>(base, a.depth_scale, vc * a.W + uc);
    if constexpr (kColor) {
      const uint8_t* px = a.rgb + ((size_t)fs * a.W * a.H + (size_t)vc * a.W + uc) * 3;
#pragma unroll
      for (int c = 0; c < 3; ++c) px3[r][c] = px[c];
    }
  }
#pragma unroll
  for (int r = 0; r < kBands; ++r) {
    const int u = u0 + 16 * r;
    if (u < a.W && v < a.H) {
      const size_t staged = (((size_t)parity * kMaxBatch + jb) * a.H + v) * a.pitch + u;
      // the pixel's colour, packed for the integration's one-word gathers
      if constexpr (kColor) a.rgba[staged] = px3[r][0] | px3[r][1] << 8 | px3[r][2] << 16;
      // the pre-scaled depth the integration of this frame gathers
      a.dm[staged] = scaled_depth(dr[r], a.max_depth, a.inv_mu);
    } else {
      dr[r] = 0.0f;
    }
  }

  // carving volumes: the largest valid depth of each 16 x 16 band (a max-depth tile)
  float (*s_tmax)[kBands] = L.tmax;
  if (a.tilemax) {
#pragma unroll
    for (int r = 0; r < kBands; ++r) {
      float m = depth_valid(dr[r], a.max_depth) ? dr[r] : 0.0f;
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
      if (lane == 0) s_tmax[wave][r] = m;
    }
  }
  for (int i = tid; i < kSetSlots; i += 256) L.set[i] = kEmptyKey;
  if (tid == 0) L.nuniq = 0;
  __syncthreads();
  if (a.tilemax && tid < kBands) {
    const int mx = tx * kBands + tid;
    if (mx < a.tiles_x)
      a.tilemax[(((size_t)parity * kMaxBatch + jb) * a.tiles_y + ty) * a.tiles_x + mx] =
          fmaxf(fmaxf(s_tmax[0][tid], s_tmax[1][tid]), fmaxf(s_tmax[2][tid], s_tmax[3][tid]));
  }
  tile_bands(a, T, dr, u0, v, frame, jb, parity, stripe, L);
}

// Allocation of the batch about to be integrated: `tiles` workgroups per frame.
template <bool kU16, int kBands, bool kColor>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_alloc(FrameArgs a, uint32_t tiles) {
  __shared__ AllocLds<kBands> L;
  const uint32_t jb = blockIdx.x / tiles;
  const FrameCtl* ctl = a.ctl;
  alloc_tile<kU16, kBands, kColor>(a, blockIdx.x - jb * tiles, ctl->frame_id + jb, jb, ctl->batch_id & 1u,
                          input_slot(ctl->cursor[a.cursor_id], jb, a.n_seq), L);
}

// ============================================================================ integration
// tsdf_update (vh_math.h) with RN(1/(w + 1)) by recip_rn (the correctly rounded reciprocal).
// cap_or_inf: the weight cap, +inf when uncapped (min is then the identity). kTab: RN(1/w)
// from the workgroup's table (rcp_table) instead of the reciprocal instructions; the launch
// takes it when every weight it can meet is below kRcpTab - 1 (the values are equal).
constexpr uint32_t kRcpTab = 1024;
template <bool kTab>
__device__ __forceinline__ void mean_update(float& s, float& w, float dist, float cap_or_inf, const float* rcp_tab) {
  const float w_new = w + 1.0f;
  const float r = kTab ? rcp_tab[(uint32_t)w_new] : recip_rn(w_new);
  s = __builtin_fmaf(dist - s, r, s);
  w = fminf(w_new, cap_or_inf);
}

// Colour update of the reference (src/tsdf.cu:743-745): per channel (c * w_old + rgb) / w_new
// in FP32 (the product and sum are exact integers below 2^24; the quotient correctly rounded
// as in div_rn), truncated to 8 bits. w_old is the stored weight before this update, w_new
// = w_old + 1 and y = RN(1/w_new); c and px are packed {r | g << 8 | b << 16}.
__device__ __forceinline__ uint32_t color_update(uint32_t c, float w_old, float w_new, float y, uint32_t px) {
  uint32_t out = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float num = __builtin_fmaf((float)((c >> (8 * k)) & 255u), w_old, (float)((px >> (8 * k)) & 255u));
    const float q0 = num * y;
    out |= (uint32_t)(uint8_t)__builtin_fmaf(__builtin_fmaf(-w_new, q0, num), y, q0) << (8 * k);
  }
  return out;
}

// One wave per listed block: lane l owns voxels l + 64k (x = k, y = l >> 3, z = l & 7), so
// each of its 8 loads is one coalesced 512-byte wave access and all 8 are in flight at once.
// A launch integrates a batch of k frames (ids f0 .. f0+k-1, inputs cur .. cur+k-1): the list
// holds every block that any of them touched, once, with the mask of those frames. The
// block's voxels are read once, updated by each marked frame in frame order (each update
// unpacks and packs the storage word, exactly as that frame's own load and store would), and
// written once; a voxel gets the same sequence of updates as frame-by-frame integration.
// Worker w of `workers` (one wave each) takes an equal share of the list, its 64 stripes
// seen as one index space; workers synchronise only within their own wave.
// kColor: the colour pool is updated from each frame's packed RGB at the same pixels.
// Where a block's voxels fall in a frame, which selects frame_update's variant:
constexpr int kPlaceEdge = 0;    // some voxel may project outside the image: per-voxel checks
constexpr int kPlaceInside = 1;  // every voxel inside: no checks, depth gathered from the image
constexpr int kPlaceWindow = 2;  // every voxel inside, its pixels in a window staged in LDS
// LDS window per wave (pixels): the pre-scaled depth of the pixel rectangle that a block's
// voxels project into, rows of a power-of-two pitch of 4 to 64. A 5 mm block at 2 m covers about
// 12 x 12 pixels; at 0.5 m about 50 x 50, which does not fit and is gathered from the image.
constexpr uint32_t kWin = 512;

// A block's window in a frame: the image rectangle of columns ulo .. ulo + cols - 1 (ulo a
// multiple of 4) and rows vlo .. vlo + rows - 1, in LDS at pitch 2^shift.
struct DepthWindow {
  uint32_t first;  // byte offset 4 (vlo pitch + ulo) of the rectangle's first pixel in the image
  uint32_t shift;  // log2 of the LDS row pitch in pixels, 2 .. 6
  uint32_t rows, cols;
  uint32_t bias;   // LDS byte offset of pixel (u, v) = (bits(M + v) << (shift + 2)) + (bits(M + u) << 2) - bias
};

// Smallest and largest of x over the 8 lanes of an aligned group (DPP: the quad's pairs, the
// quad's halves, the half-row mirror).
__device__ __forceinline__ int32_t oct_min(int32_t x) {
  x = min(x, dpp<0xB1>(x));
  x = min(x, dpp<0x4E>(x));
  return min(x, dpp<0x141>(x));
}
__device__ __forceinline__ int32_t oct_max(int32_t x) {
  x = max(x, dpp<0xB1>(x));
  x = max(x, dpp<0x4E>(x));
  return max(x, dpp<0x141>(x));
}

// Placement of a block in up to 8 frames at once: lanes 8 j .. 8 j + 7 hold the block's 8
// corners in frame j (hb: the frame's homogeneous block origin, off: the corner's homogeneous
// offset), so one pass over the lanes places the block in every frame of the batch (a pass per
// frame spent about 75 vector instructions on wave-uniform values in each). The block's lattice
// box is the convex hull of its corners. For depths > 0 the perspective image of a convex
// combination is a convex combination of the images, and where every corner's z is at least
// near_depth, a voxel's own projection and the corners' each differ from the exact ones by less
// than 1/8 pixel. So if every corner also has z in [2^-60, 2^60], every voxel's z lies in
// [2^-64, 2^64], and with umin, umax the least and largest u = X/z of the corners a voxel's
// pixel round(u) lies in [round(umin - 1/2), round(umax + 1/2)] (for errors below 1/2 these
// roundings cannot cross the voxel's); likewise v. A corner nearer than that (640 x 480, a block 1 m
// from the camera: 1 cm) leaves the block to the checks per voxel. That rectangle, its left edge moved down to a multiple of 4 pixels, is the block's window.
// kPlaceEdge unless the rectangle lies inside the image; then kPlaceWindow when it fits kWin at
// a pitch of at most 64 pixels, else kPlaceInside. The bounds are the bits of (u -+ 1/2) + M as
// signed integers: for positive sums below 2^24 they are M's plus the rounded bound, larger
// sums (and NaN) exceed every image bound and negative ones lie below them.
struct Placement {
  uint32_t first, bias;  // DepthWindow's
  uint32_t desc;         // placement | shift << 2 | cols << 5 | rows << 12
};
__device__ __forceinline__ Placement block_place(const FrameArgs& a, const float hb[3], const float off[3], float steps) {
  const float z = hb[2] + off[2];
  const float iz = __builtin_amdgcn_rcpf(z);  // within 1 ulp: the bounds leave 1/2 pixel
  const float u = (hb[0] + off[0]) * iz, v = (hb[1] + off[1]) * iz;
  const uint64_t zin = __builtin_amdgcn_ballot_w64((z >= near_depth(steps, hb, a.near)) & (z >= 0x1p-60f) & (z <= 0x1p60f));
  const int32_t lu = oct_min((int32_t)__float_as_uint((u - 0.5f) + kPixMagic));
  const int32_t hu = oct_max((int32_t)__float_as_uint((u + 0.5f) + kPixMagic));
  const int32_t lv = oct_min((int32_t)__float_as_uint((v - 0.5f) + kPixMagic));
  const int32_t hv = oct_max((int32_t)__float_as_uint((v + 0.5f) + kPixMagic));
  const int32_t mb = (int32_t)kPixMagicBits;
  const uint32_t lane = threadIdx.x & 63u;
  const bool inside = ((zin >> (lane & 56u)) & 255u) == 255u && lu >= mb && hu <= mb + a.W - 1 && lv >= mb &&
                      hv <= mb + a.H - 1;
  const int32_t la = lu & ~3;  // M's bits are a multiple of 4
  const uint32_t cols = (uint32_t)(hu - la) + 1u, rows = (uint32_t)(hv - lv) + 1u;
  // pitch: the power of two >= cols, at least 4 and at most 64
  const uint32_t shift = 32u - (uint32_t)__builtin_clz(min(cols - 1u, 63u) | 3u);
  const bool fits = cols <= 64u && rows <= (kWin >> shift);
  Placement p;
  p.first = 4u * (((uint32_t)lv - kPixMagicBits) * (uint32_t)a.pitch + ((uint32_t)la - kPixMagicBits));
  p.bias = ((uint32_t)lv << (shift + 2u)) + ((uint32_t)la << 2);
  p.desc = inside ? (fits ? (uint32_t)kPlaceWindow | shift << 2 | cols << 5 | rows << 12 : (uint32_t)kPlaceInside)
                  : (uint32_t)kPlaceEdge;
  return p;
}

// Smallest and largest of x over lanes 0, 7, 56 and 63: the half-row mirror pairs lane 0 with 7 and 56
// with 63, then two reads.
__device__ __forceinline__ int32_t ends_min(int32_t x) {
  x = min(x, dpp<0x141>(x));
  return min(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 56));
}
__device__ __forceinline__ int32_t ends_max(int32_t x) {
  x = max(x, dpp<0x141>(x));
  return max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 56));
}

// block_place for the launch of a single frame: the lane's column of voxels runs from cl to cl + 7 ax,
// and the columns of lanes 0, 7, 56 and 63 end at the block's 8 corners. hb: the homogeneous block origin.
// By lane groups, as in block_place, a single frame's block is placed eight times over and read back with
// readlane. Per frame, by lane groups / in this form: 640 x 480 into a far floor at 4 mm, binary16 43.1 / 42.0 us,
// FP32 32.4 / 31.9; into a room at 5 mm, binary16 23.7 / 22.7; at 4 mm, F16R 37.1 / 34.7.
__device__ __forceinline__ int block_place_one(const FrameArgs& a, const float ax[3], const float cl[3], const float hb[3],
                                               float steps, DepthWindow& w) {
  const float near = near_depth(steps, hb, a.near);
  bool zin = true;
  float u[2], v[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float z = e ? __builtin_fmaf(7.0f, ax[2], cl[2]) : cl[2];
    const float iz = recip_rn(z);
    u[e] = (e ? __builtin_fmaf(7.0f, ax[0], cl[0]) : cl[0]) * iz;
    v[e] = (e ? __builtin_fmaf(7.0f, ax[1], cl[1]) : cl[1]) * iz;
    zin = zin & (z >= near) & (z >= 0x1p-60f) & (z <= 0x1p60f);
  }
  const int32_t lu = ends_min((int32_t)__float_as_uint((fminf(u[0], u[1]) - 0.5f) + kPixMagic));
  const int32_t hu = ends_max((int32_t)__float_as_uint((fmaxf(u[0], u[1]) + 0.5f) + kPixMagic));
  const int32_t lv = ends_min((int32_t)__float_as_uint((fminf(v[0], v[1]) - 0.5f) + kPixMagic));
  const int32_t hv = ends_max((int32_t)__float_as_uint((fmaxf(v[0], v[1]) + 0.5f) + kPixMagic));
  const int32_t mb = (int32_t)kPixMagicBits, la = lu & ~3;
  const uint32_t cols = (uint32_t)(hu - la) + 1u, rows = (uint32_t)(hv - lv) + 1u;
  const uint32_t shift = 32u - (uint32_t)__builtin_clz(min(cols - 1u, 63u) | 3u);
  w.first = 4u * (((uint32_t)lv - kPixMagicBits) * (uint32_t)a.pitch + ((uint32_t)la - kPixMagicBits));
  w.shift = shift;
  w.rows = rows;
  w.cols = cols;
  w.bias = ((uint32_t)lv << (shift + 2u)) + ((uint32_t)la << 2);
  const bool inside = __builtin_amdgcn_ballot_w64(!zin) == 0 && lu >= mb && hu <= mb + a.W - 1 && lv >= mb &&
                      hv <= mb + a.H - 1;
  const bool fits = cols <= 64u && rows <= (kWin >> shift);
  return inside ? (fits ? kPlaceWindow : kPlaceInside) : kPlaceEdge;
}

// LDS addresses as integers: the byte address of an LDS location, and a read from one.
typedef __attribute__((address_space(3))) float LdsFloat;
__device__ __forceinline__ uint32_t lds_address(const float* p) { return (uint32_t)(size_t)(const LdsFloat*)p; }
__device__ __forceinline__ float lds_read(uint32_t byte_address) { return *(const LdsFloat*)(size_t)byte_address; }

// The window's pixels of pre-scaled depth image dmf into the wave's LDS window at byte address
// win (row r at win + 4 (r << shift)), by 16-byte loads that write LDS directly: load t covers
// rows t * 256 >> shift onwards, lane l the four pixels from column 4 (l mod 2^(shift - 2)) of row
// l >> (shift - 2), and writes words 256 t + 4 l onwards. Image rows and the window's left edge
// are multiples of 4 pixels, so every access is 16-byte aligned; the last load of a row may read
// up to 3 pixels past the rectangle (the images are followed by 64 bytes). A typical window of
// 12 x 12 pixels is one load (three with 4-byte loads). The loads use no registers, so the caller
// computes its pixels while they are in flight and waits for them (window_ready) before its first
// read.
__device__ __forceinline__ void stage_window(const FrameArgs& a, const float* dmf, const DepthWindow& w, uint32_t win) {
  const uint32_t lane = threadIdx.x & 63u, w4 = 4u * (uint32_t)a.pitch, per = w.shift - 2u;
  const uint32_t row = lane >> per, col = 4u * (lane & ((1u << per) - 1u)), step = 64u >> per;
  const char* src = reinterpret_cast<const char*>(dmf) + w.first;
  const uint32_t off = __umul24(row, w4) + 4u * col;  // both below 2^24
  const int left = col < w.cols ? (int)(w.rows - row) : 0;  // rows from the lane's own to the window's end
  const uint32_t n_it = (w.rows + step - 1u) >> (6u - per);
  for (uint32_t t = 0; t < n_it; ++t) {
    const char* rows_t = src + t * step * w4;  // uniform
    if ((int)(t * step) < left)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(rows_t + off),
                                       (__attribute__((address_space(3))) void*)(size_t)(win + 1024u * t), 16, 0, 0);
  }
}
// Wait for the window's loads (vmcnt 0; the compiler does not order a read through an integer
// LDS address after them by itself).
__device__ __forceinline__ void window_ready() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// The 8 voxels of a lane between a block's load and its store. kReg (launches of several frames
// with the reciprocal table, storage FP32 or FP16): the value s as the storage rounds it and the
// weight as the byte offset t = 4 w of RN(1/w) in the table, so a frame's update reads the
// table at t + 4 with no conversion, and an unobserved voxel reads the table's entry 0, which is
// 0: its value is then s + 0 * (-1 - s) = s bit for bit, with no selects (|s| <= 1). The two
// conversions each way per voxel are paid once per block. Otherwise the storage word itself
// (F16R's word is not a function of its value: the residual of a tie has two forms).
template <int kStorage, bool kReg>
struct LaneVoxels {
  using IO = VoxelIO<kStorage>;
  using Word = typename IO::Word;
  Word w[8];
  __device__ __forceinline__ void load(int q, Word x) { w[q] = x; }
  __device__ __forceinline__ Word word(int q) const { return w[q]; }
};
template <>
struct LaneVoxels<VH_STORAGE_F32, true> {
  using Word = float2;
  float s[8];
  uint32_t t[8];
  __device__ __forceinline__ void load(int q, Word x) { s[q] = x.x; t[q] = (uint32_t)(x.y * 4.0f); }
  __device__ __forceinline__ Word word(int q) const { return make_float2(s[q], (float)t[q] * 0.25f); }
  __device__ __forceinline__ void set(int q, float v) { s[q] = v; }
};
template <>
struct LaneVoxels<VH_STORAGE_F16, true> {
  using Word = uint32_t;
  float s[8];
  uint32_t t[8];
  __device__ __forceinline__ void load(int q, Word x) {
    s[q] = (float)__builtin_bit_cast(_Float16, (uint16_t)(x & 0xffffu));
    t[q] = (x >> 16) << 2;
  }
  __device__ __forceinline__ Word word(int q) const {
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)s[q]) | t[q] << 14;  // s[q] is a binary16 value
  }
  __device__ __forceinline__ void set(int q, float v) {
    s[q] = (float)__builtin_bit_cast(_Float16, f32_to_f16_rn(v));
  }
};

// One frame's update of the lane's 8 voxels of a block (homogeneous column cl, step ax): per
// half, all projections, then all pre-scaled depth (and colour) fetches, then the updates, so
// the fetches are in flight together. Branch-free per lane: every lane computes, the observation
// flag selects. dmf: the frame's pre-scaled depth image (scaled_depth of each pixel).
// place (block_place's result, wave-uniform) chooses how a half's depths are fetched; the
// projection and the update around it are common, so the voxels stay in their registers (a
// variant of the whole update per placement cost 16 register copies per frame where the
// variants join). kPlaceInside and kPlaceWindow leave out the range checks, which are known to
// pass; kPlaceWindow reads the depth from the window that stage_window is loading (pitch
// 2^wshift; wbase: the LDS byte address of pixel (u, v) is (bits(M + v) << (wshift + 2)) +
// (bits(M + u) << 2) + wbase modulo 2^32, the window's address minus DepthWindow::bias). A voxel
// outside the image gets depth -inf, which no update follows. (Issuing the next frame's gathers
// before this frame's updates, with two register sets, was slower: 92 against 86 us per FP32
// batch launch.)
template <int kStorage, bool kColor, bool kTab, bool kReg>
__device__ __forceinline__ void frame_update(const FrameArgs& a, uint32_t place, const float ax[3], const float cl[3],
                                             const float* dmf, const uint32_t* rgba, uint32_t wshift,
                                             uint32_t wbase, uint32_t t_cap, LaneVoxels<kStorage, kReg>& vx,
                                             uint32_t cold[8], uint32_t& upd, const float* rcp_tab) {
  using IO = VoxelIO<kStorage>;
  using Word = typename IO::Word;
  const uint32_t w4 = (4u * (uint32_t)a.pitch) & 0xffffffu, bias = pix_bias(a.pitch);
  // two halves of 4 voxels: fewer values live at once (occupancy) for 4 fetches in flight
#pragma unroll
  for (int h = 0; h < 8; h += 4) {
    float zc[4], uf[4], vf[4];  // camera depth; M + column, M + row of the pixel
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float fq = (float)(h + r);  // voxel 0 is the column itself (fma(0, a, c) = c but for -0)
      const float X = h + r ? __builtin_fmaf(fq, ax[0], cl[0]) : cl[0];
      const float Y = h + r ? __builtin_fmaf(fq, ax[1], cl[1]) : cl[1];
      zc[r] = h + r ? __builtin_fmaf(fq, ax[2], cl[2]) : cl[2];
      const float iz = recip_rn(zc[r]);
      uf[r] = __builtin_fmaf(X, iz, kPixMagic);
      vf[r] = __builtin_fmaf(Y, iz, kPixMagic);
    }
    float dv[4];
    uint32_t px[4];
    if (place == (uint32_t)kPlaceWindow) {
      uint32_t loff[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t ub = __float_as_uint(uf[r]), vb = __float_as_uint(vf[r]);
        loff[r] = (((vb << wshift) + ub) << 2) + wbase;
        if constexpr (kColor)
          px[r] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(rgba) +
                                                     ((vb & 0xffffffu) * w4 + ((ub << 2) - bias)));
      }
      if (h == 0) window_ready();  // the pixels are computed: now wait for the window
#pragma unroll
      for (int r = 0; r < 4; ++r) dv[r] = lds_read(loff[r]);
    } else if (place == (uint32_t)kPlaceInside) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t ub = __float_as_uint(uf[r]), vb = __float_as_uint(vf[r]);
        const uint32_t off = (vb & 0xffffffu) * w4 + ((ub << 2) - bias);
        dv[r] = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(dmf) + off);
        if constexpr (kColor) px[r] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(rgba) + off);
      }
    } else {
      int pix[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pix[r] = pixel_of(uf[r], vf[r], zc[r], a.W, a.H, a.pitch);
        dv[r] = dmf[max(pix[r], 0)];
        if constexpr (kColor) px[r] = rgba[max(pix[r], 0)];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) dv[r] = pix[r] >= 0 ? dv[r] : -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int q = h + r;
      const float t = __builtin_fmaf(-zc[r], a.inv_mu, dv[r]);
      const bool ok = t > -1.0f;
      if constexpr (kReg) {
        const float dist = __builtin_amdgcn_fmed3f(t, -1.0f, 1.0f);  // min(1, t) where observed, -1 elsewhere
        const uint32_t tn = ok ? vx.t[q] + 4u : 0u;
        const float y = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(rcp_tab) + tn);
        if constexpr (kColor) {
          const float w_old = (float)vx.t[q] * 0.25f;
          const uint32_t c = color_update(cold[q], w_old, w_old + 1.0f, y, px[r]);
          cold[q] = ok ? c : cold[q];
          upd |= (uint32_t)ok << q;
        }
        vx.set(q, __builtin_fmaf(dist - vx.s[q], y, vx.s[q]));
        vx.t[q] = min(max(vx.t[q], tn), t_cap);
      } else {
        const float dist = fminf(1.0f, t);
        float sv, wv;
        IO::unpack(vx.w[q], sv, wv);
        if constexpr (kColor) {
          const uint32_t c = color_update(cold[q], wv, wv + 1.0f, recip_rn(wv + 1.0f), px[r]);
          cold[q] = ok ? c : cold[q];
          upd |= (uint32_t)ok << q;
        }
        mean_update<kTab>(sv, wv, dist, a.cap, rcp_tab);
        const Word nw = IO::pack(sv, wv);
        vx.w[q] = ok ? nw : vx.w[q];
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // keep the halves apart: the scheduler would merge them
  }
}

// Per frame of a batch, staged in LDS by stage_frames: the pose (row-major 3x4) and the
// frame's homogeneous voxel steps (block_frame_h), each padded to 16 bytes; ax[3] holds their
// near_steps.
struct __align__(16) FrameLds {
  float T[12];
  float ax[4], ay[4], az[4];
};
// Per frame and lane: the column's homogeneous offset from the block origin, the
// same for every block.
struct __align__(16) ColumnLds {
  float off[64][4];
};

// my_off, n: lane s holds the exclusive offset of the list's stripe s; the list's length. s_frm,
// s_col: the batch's k frames; rcp_tab: RN(1/w) for w < kRcpTab with 0 at w = 0 (read when
// kTab); s_win: the LDS byte address of the wave's depth window (kWin pixels). kBatch: a launch of
// several frames (k > 1), whose blocks are placed in all of them at once (block_place); a single
// frame's are placed by block_place_one, with no s_col.
template <int kStorage, bool kColor, bool kTab, bool kBatch>
__device__ void integrate_worker(const FrameArgs& a, uint32_t worker, uint32_t workers, uint32_t my_off, uint32_t n,
                                 uint32_t f0, uint32_t k, uint32_t parity, unsigned long long* s_val,
                                 unsigned long long* s_key, uint32_t* s_mark, const FrameLds* s_frm,
                                 const ColumnLds* s_col, const float* rcp_tab, uint32_t s_win) {
  using IO = VoxelIO<kStorage>;
  using Word = typename IO::Word;
  constexpr bool kReg = kTab && kBatch && kStorage != VH_STORAGE_F16R;
  FrameCtl* ctl = a.ctl;
  const int lane = threadIdx.x & 63;
  const uint32_t* list = list_of(a, parity);
  uint32_t* marks = marks_of(a, parity);
  const size_t frame_px = (size_t)a.pitch * a.H;
  const uint32_t t_cap = a.cap < (float)kRcpTab ? 4u * (uint32_t)a.cap : ~0u;

  // lanes 8 j .. 8 j + 7: the 8 corners of a block in frame j of the batch, as homogeneous
  // offsets from its origin
  const uint32_t jl = kBatch ? min((uint32_t)lane >> 3, k - 1u) : 0u;
  float corner[3];
  if constexpr (kBatch) {
    const float c0 = (lane & 1) ? 7.0f : 0.0f, c1 = (lane & 2) ? 7.0f : 0.0f, c2 = (lane & 4) ? 7.0f : 0.0f;
#pragma unroll
    for (int r = 0; r < 3; ++r)
      corner[r] = __builtin_fmaf(c0, s_frm[jl].ax[r], __builtin_fmaf(c1, s_frm[jl].ay[r], c2 * s_frm[jl].az[r]));
  }

  // Lane j fetches the list entry, slot value, key and mark of this worker's j-th block
  // (clearing the mark for the next batch of this parity) and parks them in LDS, so the
  // per-block chain is a single round trip (voxels + depth). The block loop reads them back
  // from LDS: a use of the loaded registers inside the loop would make the compiler wait for
  // every outstanding vector memory operation, the previous block's stores included (vmcnt
  // counts stores on this architecture).
  for (uint32_t t0 = worker; t0 < n; t0 += 64u * workers) {
    const uint32_t tj = t0 + (uint32_t)lane * workers;
    const uint32_t tq = min(tj, n - 1u);
    int lo = 0, hi = 63;  // stripe of entry tq: the last stripe whose offset is <= tq
#pragma unroll
    for (int it = 0; it < 6; ++it) {  // all lanes active: the shuffles read defined values
      const int mid = (lo + hi + 1) >> 1;
      const uint32_t om = (uint32_t)__shfl((int)my_off, mid);
      if (om <= tq) lo = mid;
      else hi = mid - 1;
    }
    const uint32_t stripe_off = (uint32_t)__shfl((int)my_off, lo);
    unsigned long long jval = ~0ull, jkey = 0ull;
    uint32_t jmark = 0u;
    if (tj < n) {
      const uint32_t sl = list[(size_t)lo * a.stripe_cap + (tj - stripe_off)];
      jval = a.hash.vals[sl];
      jkey = a.hash.keys[sl];
      jmark = marks[sl];
      marks[sl] = 0u;
    }
    s_val[lane] = jval;
    s_key[lane] = jkey;
    s_mark[lane] = jmark;
    __builtin_amdgcn_wave_barrier();  // one wave owns this slice: it only needs its own writes
    const uint32_t nj = min(64u, (n - t0 + workers - 1) / workers);
    for (uint32_t j = 0; j < nj; ++j) {
      const unsigned long long val = uniform64(s_val[j]);
      const unsigned long long keyj = uniform64(s_key[j]);
      const uint32_t mark = uniform(s_mark[j]) & ((1u << k) - 1u);
      const uint32_t idx = (uint32_t)val;
      if (idx >= a.pool_cap) {
        if (lane == 0) raise_flag(ctl, kFlagPoolFull);
        continue;
      }
      const bool fresh = (uint32_t)(val >> 32) - f0 < k;  // born in this batch: starts at zero
      int bx, by, bz;
      unpack_key(keyj, bx, by, bz);
      Word* vp = reinterpret_cast<Word*>(a.voxels) + (size_t)idx * kB3;
      uint32_t* cp = kColor ? a.colors + (size_t)idx * kB3 : nullptr;
      LaneVoxels<kStorage, kReg> vx;
      uint32_t cold[8];
      {
        Word old[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) old[q] = fresh ? IO::zero() : vp[lane + 64 * q];
        if constexpr (kColor) {
#pragma unroll
          for (int q = 0; q < 8; ++q) cold[q] = fresh ? 0u : cp[lane + 64 * q];
        }
        // the block's origin (kBatch: its placement too, lane group j holding frame j's for the frame loop to
        // take with readlane), while its voxels are on their way
        float hb[3];
        {
          float T[12], cb[3];
#pragma unroll
          for (int q = 0; q < 12; ++q) T[q] = s_frm[jl].T[q];
          block_origin_cam(T, a.vox, bx, by, bz, cb);
          to_pixel_h(a.K, cb, hb);
        }
        Placement pl{};
        if constexpr (kBatch) pl = block_place(a, hb, corner, s_frm[jl].ax[3]);
#pragma unroll
        for (int q = 0; q < 8; ++q) vx.load(q, old[q]);
        uint32_t upd = 0u;  // colour volumes: bit q set when voxel q was observed in the batch
        if constexpr (!kBatch) {
          if (mark) {
            const FrameLds& F = s_frm[0];
            float ax[3], cl[3];
#pragma unroll
            for (int r = 0; r < 3; ++r) {
              ax[r] = F.ax[r];
              cl[r] = hb[r] + __builtin_fmaf((float)(lane >> 3), F.ay[r], (float)(lane & 7) * F.az[r]);
            }
            const size_t fo = (size_t)parity * kMaxBatch * frame_px;
            const uint32_t* rgba = kColor ? a.rgba + fo : nullptr;
            const float* dmf = a.dm + fo;
            DepthWindow win;
            const int place = block_place_one(a, ax, cl, hb, F.ax[3], win);
            // the update once per placement: its variants' registers don't join before another frame's
            if (place == kPlaceWindow) {
              stage_window(a, dmf, win, s_win);
              frame_update<kStorage, kColor, kTab, kReg>(a, kPlaceWindow, ax, cl, dmf, rgba, win.shift, s_win - win.bias, t_cap, vx,
                                                         cold, upd, rcp_tab);
            } else if (place == kPlaceInside) {
              frame_update<kStorage, kColor, kTab, kReg>(a, kPlaceInside, ax, cl, dmf, rgba, 0u, 0u, t_cap, vx, cold, upd, rcp_tab);
            } else {
              frame_update<kStorage, kColor, kTab, kReg>(a, kPlaceEdge, ax, cl, dmf, rgba, 0u, 0u, t_cap, vx, cold, upd, rcp_tab);
            }
          }
        }
        for (uint32_t m = kBatch ? mark : 0u; m != 0u; m &= m - 1u) {
          const uint32_t jf = (uint32_t)__builtin_ctz(m);
          const int src = 8 * (int)jf;
          float ax[3], cl[3];
#pragma unroll
          for (int r = 0; r < 3; ++r) {
            ax[r] = s_frm[jf].ax[r];
            // the block origin plus the column's offset
            cl[r] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hb[r]), src)) + s_col[jf].off[lane][r];
          }
          const size_t fo = ((size_t)parity * kMaxBatch + jf) * frame_px;
          const uint32_t* rgba = kColor ? a.rgba + fo : nullptr;
          const float* dmf = a.dm + fo;
          const uint32_t desc = read_lane_u32(pl.desc, src);
          const uint32_t place = desc & 3u;
          uint32_t wshift = 0u, wbase = 0u;
          if (place == (uint32_t)kPlaceWindow) {
            DepthWindow win;
            win.first = read_lane_u32(pl.first, src);
            win.bias = read_lane_u32(pl.bias, src);
            win.shift = (desc >> 2) & 7u;
            win.cols = (desc >> 5) & 127u;
            win.rows = desc >> 12;
            stage_window(a, dmf, win, s_win);
            wshift = win.shift;
            wbase = s_win - win.bias;
          }
          frame_update<kStorage, kColor, kTab, kReg>(a, place, ax, cl, dmf, rgba, wshift, wbase, t_cap, vx, cold, upd,
                                                     rcp_tab);
        }
        // Depth-only volumes write the block whole (unobserved voxels keep the words read,
        // fresh blocks zero there; the wave owns the block in this launch), which saves the
        // per-voxel mask; colour volumes (12 B per voxel) write fresh blocks whole and other
        // blocks where observed.
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          if constexpr (kColor) {
            if (fresh || ((upd >> q) & 1u)) {
              vp[lane + 64 * q] = vx.word(q);
              cp[lane + 64 * q] = cold[q];
            }
          } else {
            vp[lane + 64 * q] = vx.word(q);
          }
        }
      }
    }
    __builtin_amdgcn_wave_barrier();  // the next batch of entries overwrites s_val / s_key / s_mark
  }
}

// End of a workgroup of a batch launch (all 256 lanes call it): the last of `groups`
// workgroups to finish (two-level striped counter) closes the batch (first frame f0, k
// frames, list parity): its per-frame counts are summed into the statistics and cleared with
// the list lengths; the frame id, input cursor and batch id advance. No fence before the
// counters: the closing workgroup reads no voxel data, and the voxel writes are published by
// the kernel boundary (a device-scope fence per workgroup would write back the L2 thousands
// of times per batch).
__device__ void batch_done(const FrameArgs& a, uint32_t groups, uint32_t f0, uint32_t k, uint32_t parity) {
  __shared__ uint32_t s_closes;
  FrameCtl* ctl = a.ctl;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t g = blockIdx.x & (kStripes - 1);
    const uint32_t in_group = groups / kStripes + (g < groups % kStripes ? 1u : 0u);
    const uint32_t live = min(groups, (uint32_t)kStripes);  // stripes holding a workgroup
    uint32_t closes = 0;
    if (atomicAdd(&ctl->done[g * kLine], 1u) == in_group - 1) closes = atomicAdd(&ctl->done_top, 1u) == live - 1;
    s_closes = closes;
  }
  __syncthreads();
  if (threadIdx.x >= 64 || !s_closes) return;
  // The counts were final before this launch started (the batch's allocation ran earlier):
  // each lane reads and clears one stripe's line, one round trip in all.
  const int lane = threadIdx.x;
  uint32_t* line = list_count_of(ctl, parity) + lane * kLine;
  uint32_t listed = min(line[0], a.stripe_cap);
  uint32_t carved = line[kLineCarve];
  uint32_t per[kMaxBatch];
#pragma unroll
  for (int j = 0; j < kMaxBatch; ++j) per[j] = (uint32_t)j < k ? line[1 + j] : 0u;
#pragma unroll
  for (int j = 0; j <= kMaxBatch; ++j)
    if ((uint32_t)j <= k) line[j] = 0u;
  line[kLineCarve] = 0u;
  ctl->done[lane * kLine] = 0u;
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    listed += (uint32_t)__shfl_xor((int)listed, m);
    carved += (uint32_t)__shfl_xor((int)carved, m);
#pragma unroll
    for (int j = 0; j < kMaxBatch; ++j) per[j] += (uint32_t)__shfl_xor((int)per[j], m);
  }
  if (lane == 0) {
    unsigned long long sum = 0;
#pragma unroll
    for (int j = 0; j < kMaxBatch; ++j) sum += per[j];
    uint32_t last = 0;
#pragma unroll
    for (int j = 0; j < kMaxBatch; ++j)
      if ((uint32_t)j + 1u == k) last = per[j];
    ctl->touched_last = last;
    ctl->touched_total += sum;
    ctl->integrated_total += listed;
    ctl->carved_total += carved;
    ctl->frames += k;
    ctl->cursor[a.cursor_id] += k;
    ctl->frame_id = f0 + k;
    ctl->batch_id += 1u;
    ctl->done_top = 0u;
  }
}

constexpr int kIntegrateWaves = 4;  // independent workers per workgroup
// Register budget of the integration kernels: depth only, 6 waves per SIMD (80 VGPRs, at most one
// value spills; 500 frames of a room at 5 mm in batches of 8, FP32: 6.22 ms at 5 waves, 5.94 at 6,
// with the fused launch's 4,096 workers; before the values and weights of a block stayed in
// registers in the form the update takes them, 6 waves spilled into the frame loop); a single frame's
// launch 5, all its workers at once (FP32 needs 84 VGPRs; at 6 waves four values spill: a room at
// 4 mm 33.0 us, at 5 waves 31.9); colour, 4
// waves (128 VGPRs: at 96 about 50 values spill into the frame loop, 13 % slower).
#define VH_INTEGRATE_OCCUPANCY(kBatch) __attribute__((amdgpu_waves_per_eu(kColor ? 4 : kBatch ? 6 : 5)))

// Entry q of the pose of the batch's frame j (kBatch: of a bound sequence).
template <bool kBatch>
__device__ __forceinline__ float pose_entry(const FrameArgs& a, uint32_t cur, uint32_t j, uint32_t q) {
  return kBatch || a.poses ? a.poses[16 * (size_t)input_slot(cur, j, a.n_seq) + q] : a.pose[q];
}

// The k poses of a batch (inputs cur .. cur+k-1) into LDS, read by every block of the
// workgroup's workers (a global load per block and frame would put a memory round trip in
// front of each frame's projections). All 256 lanes call it.
__device__ __forceinline__ void stage_poses(const FrameArgs& a, uint32_t cur, uint32_t k, float (*s_pose)[12]) {
  const uint32_t t = threadIdx.x;
  if (t < 12u * k) {
    const uint32_t j = t / 12u, q = t - 12u * j;
    s_pose[j][q] = pose_entry<false>(a, cur, j, q);
  }
  __syncthreads();
}
// The poses, homogeneous steps and column offsets of a batch's frames into LDS, and the
// reciprocal table. pose: the t-th of the batch's 12 k pose entries in lane t. All 256 lanes call
// it. Each wave forms the steps of the frames whose columns it fills (the same values in every
// lane), so that one barrier separates the poses from everything made of them. A single frame (not
// kBatch) has no columns.
template <bool kBatch>
__device__ __forceinline__ void stage_frames(const FrameArgs& a, float pose, uint32_t k, FrameLds* s_frm,
                                             ColumnLds* s_col, float* rcp_tab, bool tab) {
  const uint32_t t = threadIdx.x;
  if (t < 12u * k) {
    const uint32_t j = t / 12u, q = t - 12u * j;
    s_frm[j].T[q] = pose;
  }
  if (tab)
    for (uint32_t i = t; i < kRcpTab; i += blockDim.x) rcp_tab[i] = i ? recip_rn((float)i) : 0.0f;
  __syncthreads();
  const uint32_t lane = t & 63u;
  for (uint32_t j = t >> 6; j < k; j += kIntegrateWaves) {
    float T[12];
    BlockFrame h;
#pragma unroll
    for (int q = 0; q < 12; ++q) T[q] = s_frm[j].T[q];
    block_frame_h(T, a.vox, a.K, h);
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      if (lane == 0) {
        s_frm[j].ax[r] = h.ax[r];
        s_frm[j].ay[r] = h.ay[r];
        s_frm[j].az[r] = h.az[r];
        if (r == 0) s_frm[j].ax[3] = near_steps(h, a.near);
      }
      if constexpr (kBatch) s_col[j].off[lane][r] = __builtin_fmaf((float)(lane >> 3), h.ay[r], (float)(lane & 7u) * h.az[r]);
    }
  }
  __syncthreads();
}

// True when every weight the batch can meet is below kRcpTab - 1: capped below it, or fewer
// frames integrated (with this batch) than that (a voxel gains at most 1 per frame; a merge
// of streamed blocks adds the weights of disjoint frames).
__device__ __forceinline__ bool rcp_table_covers(const FrameArgs& a, const FrameCtl* ctl, uint32_t k) {
  return a.cap < (float)(kRcpTab - 1) || uniform64(ctl->frames) + k < (unsigned long long)(kRcpTab - 1);
}

// The integration's LDS: per wave the staged list entries, slot values, keys and marks and
// the depth window; per workgroup the batch's frames and the reciprocal table (kBatch: 26,368 bytes, 6
// workgroups per CU, as many as its registers allow; a single frame: 17,504).
template <bool kBatch>
struct IntegrateLds {
  float rcp[kRcpTab];
  FrameLds frm[kBatch ? kMaxBatch : 1];
  ColumnLds col[kBatch ? kMaxBatch : 0];
  float win[kIntegrateWaves][kWin];
  unsigned long long val[kIntegrateWaves][64], key[kIntegrateWaves][64];
  uint32_t mark[kIntegrateWaves][64];
};
static_assert(offsetof(IntegrateLds<false>, win) % 16 == 0 && offsetof(IntegrateLds<true>, win) % 16 == 0,
              "stage_window writes 16 bytes per lane");

// The workgroup's share of the batch of k frames (first frame f0, list parity, first input
// cur). All 256 lanes call it.
template <int kStorage, bool kColor, bool kBatch>
__device__ __forceinline__ void integrate_group(const FrameArgs& a, uint32_t group, uint32_t groups, uint32_t f0,
                                                uint32_t k, uint32_t parity, uint32_t cur, IntegrateLds<kBatch>& L) {
  const uint32_t t = threadIdx.x, lane = t & 63u;
  const int wave = t >> 6;
  // the pose entries and the list's lengths, in flight together
  float pose = 0.0f;
  if (t < 12u * k) {
    const uint32_t j = t / 12u, q = t - 12u * j;
    pose = pose_entry<kBatch>(a, cur, j, q);
  }
  const uint32_t my_len = min(list_count_of(a.ctl, parity)[lane * kLine], a.stripe_cap);
  const bool tab = rcp_table_covers(a, a.ctl, k);
  // lane s holds stripe s's length and exclusive offset
  uint32_t incl = my_len;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)incl, off);
    if ((int)lane >= off) incl += y;
  }
  const uint32_t my_off = incl - my_len, n = read_lane_u32(incl, 63);
  const uint32_t worker = group * kIntegrateWaves + wave, workers = groups * kIntegrateWaves;
  if (group * kIntegrateWaves >= n) return;  // a short list: no block for this workgroup
  stage_frames<kBatch>(a, pose, k, L.frm, L.col, L.rcp, tab);
  const uint32_t win = uniform(lds_address(L.win[wave]));
  if (tab)
    integrate_worker<kStorage, kColor, true, kBatch>(a, worker, workers, my_off, n, f0, k, parity, L.val[wave],
                                                     L.key[wave], L.mark[wave], L.frm, L.col, L.rcp, win);
  else
    integrate_worker<kStorage, kColor, false, kBatch>(a, worker, workers, my_off, n, f0, k, parity, L.val[wave],
                                                      L.key[wave], L.mark[wave], L.frm, L.col, L.rcp, win);
}

// Integration of the batch of k frames that the last allocation launch prepared (kBatch: k > 1).
template <int kStorage, bool kColor, bool kBatch>
__global__ __launch_bounds__(64 * kIntegrateWaves) VH_INTEGRATE_OCCUPANCY(kBatch) void k_integrate(FrameArgs a, uint32_t k) {
  __shared__ IntegrateLds<kBatch> L;
  const FrameCtl* ctl = a.ctl;
  // control values are uniform: keep them (and what derives from them) in scalar registers
  const uint32_t f0 = uniform(ctl->frame_id), parity = uniform(ctl->batch_id) & 1u,
                 cur = uniform(ctl->cursor[a.cursor_id]);
  integrate_group<kStorage, kColor, kBatch>(a, blockIdx.x, gridDim.x, f0, k, parity, cur, L);
  batch_done(a, gridDim.x, f0, k, parity);
}

// Integration of batch b (k_int frames) and allocation of batch b+1 (k_alloc frames) in one
// launch (bound sequences): the integration workgroups come first in the grid, so they take
// every CU slot at the start, and the allocation workgroups (short, latency-bound) fill the
// slots that the integration's tail frees. Every workgroup counts towards the close of batch
// b, so the frame id, cursor and batch id the allocation workgroups read at their start
// cannot advance under them.
template <int kStorage, bool kU16, bool kColor>
__global__ __launch_bounds__(64 * kIntegrateWaves) VH_INTEGRATE_OCCUPANCY(true) void k_integrate_alloc(FrameArgs a, uint32_t int_groups,
                                                                         uint32_t alloc_groups, uint32_t tiles,
                                                                         uint32_t k_int) {
  // a workgroup either allocates or integrates: the two share the LDS
  __shared__ union {
    AllocLds<kAllocBands> alloc;
    IntegrateLds<true> integ;
  } L;
  const uint32_t b = blockIdx.x;
  const bool alloc = b >= int_groups;
  const uint32_t idx = alloc ? b - int_groups : b;
  const FrameCtl* ctl = a.ctl;
  const uint32_t f0 = uniform(ctl->frame_id), batch = uniform(ctl->batch_id), cur = uniform(ctl->cursor[a.cursor_id]);
  if (alloc) {
    const uint32_t jb = idx / tiles;
    alloc_tile<kU16, kAllocBands, kColor>(a, idx - jb * tiles, f0 + k_int + jb, jb, (batch + 1u) & 1u,
                                 input_slot(cur, k_int + jb, a.n_seq), L.alloc);
  } else {  // uniform branch: the whole workgroup integrates
    integrate_group<kStorage, kColor, true>(a, idx, int_groups, f0, k_int, batch & 1u, cur, L.integ);
  }
  batch_done(a, gridDim.x, f0, k_int, batch & 1u);
}

// ============================================================================ carving
// Conservative form of the observation test for a whole block: false only if no voxel of block
// (bx, by, bz) can pass frame T's test (z >= 2^-64, its pixel inside the image, 0 < d <=
// max_depth and d - z > -mu there). The voxels lie in the box spanned by the block's lattice
// points 0..7 along each axis. The box's 8 corners in camera coordinates bound every voxel's z
// (the camera map is affine), and, when the whole box lies in front of the camera, every
// voxel's projection (the perspective image of a convex set in z > 0 is the convex hull of its
// corners' images). Margins cover the rounding of the voxel arithmetic of the integration
// (frame_update) against these bounds: every camera coordinate it forms is within
// 4 * 2^-23 * mag of the exact one (mag bounds the magnitudes summed), so dz bounds the depth
// error and eps the pixel error ((fx + |u - cx|) * error / z for u = fx x / z + cx).
// tmax: the frame's max-depth tiles; a voxel is only updated if its z is below its pixel's
// depth + mu, so a block whose nearest corner lies beyond the largest valid depth of the tiles
// its pixels fall in, plus mu, is not.
__device__ bool block_may_update(const FrameArgs& a, const float* T, int bx, int by, int bz, const float* tmax) {
  BlockFrame bf;
  block_frame(T, a.vox, bf);
  float cb[3];
  block_origin_cam(T, a.vox, bx, by, bz, cb);
  const float mag = fabsf(cb[0]) + fabsf(cb[1]) + fabsf(cb[2]) + 24.0f * a.vox;
  const float dz = 1e-4f + 4e-6f * mag;
  const float zfar = a.max_depth + a.mu + dz;
  // bounding sphere of the box in z first (centre at lattice offset 3.5, radius 3.5 sqrt(3) vox)
  const float zc = cb[2] + 3.5f * ((bf.ax[2] + bf.ay[2]) + bf.az[2]);
  const float rad = 6.07f * a.vox;
  if (zc + rad < -dz || zc - rad > zfar) return false;
  float P[8][3];
  float zmin = INFINITY, zmax = -INFINITY;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float ex = (c & 1) ? 7.0f : 0.0f, ey = (c & 2) ? 7.0f : 0.0f, ez = (c & 4) ? 7.0f : 0.0f;
#pragma unroll
    for (int r = 0; r < 3; ++r) P[c][r] = cb[r] + ((ex * bf.ax[r] + ey * bf.ay[r]) + ez * bf.az[r]);
    zmin = fminf(zmin, P[c][2]);
    zmax = fmaxf(zmax, P[c][2]);
  }
  if (zmax < -dz || zmin > zfar) return false;
  if (!(zmin > dz)) return true;  // the box reaches the camera plane: no projection bound
  float umin = INFINITY, umax = -INFINITY, vmin = INFINITY, vmax = -INFINITY;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float iz = __builtin_amdgcn_rcpf(P[c][2]);
    const float u = a.K.fx * (P[c][0] * iz) + a.K.cx, v = a.K.fy * (P[c][1] * iz) + a.K.cy;
    umin = fminf(umin, u);
    umax = fmaxf(umax, u);
    vmin = fminf(vmin, v);
    vmax = fmaxf(vmax, v);
  }
  const float rel = 2e-6f * mag / zmin;
  const float eu = 1.0f + rel * (a.K.fx + fmaxf(fabsf(umin - a.K.cx), fabsf(umax - a.K.cx)));
  const float ev = 1.0f + rel * (a.K.fy + fmaxf(fabsf(vmin - a.K.cy), fabsf(vmax - a.K.cy)));
  if (umax < -0.5f - eu || umin > (float)a.W - 0.5f + eu || vmax < -0.5f - ev || vmin > (float)a.H - 0.5f + ev)
    return false;
  // pixels the voxels can round to (fmaxf / fminf also map NaN bounds to the whole image)
  const int x0 = (int)fmaxf(0.0f, floorf(umin - eu)), x1 = (int)fminf((float)(a.W - 1), ceilf(umax + eu));
  const int y0 = (int)fmaxf(0.0f, floorf(vmin - ev)), y1 = (int)fminf((float)(a.H - 1), ceilf(vmax + ev));
  if (!tmax) return true;
  const int tx0 = x0 / kTile, tx1 = x1 / kTile, ty0 = y0 / kTile, ty1 = y1 / kTile;
  if ((tx1 - tx0 + 1) * (ty1 - ty0 + 1) > 64) return true;  // a near block: not worth the reads
  float D = 0.0f;
  for (int ty = ty0; ty <= ty1; ++ty)
    for (int tx = tx0; tx <= tx1; ++tx) D = fmaxf(D, tmax[ty * a.tiles_x + tx]);
  return zmin <= D + a.mu + dz;
}

// Carve pass of the allocated batch (k frames, first frame id f0, list parity): one lane per
// resident pool block (the lanes of a fixed grid stride over the pool). Frame j may update a
// block born at or before frame f0 + j (a block born later in the batch did not exist when
// frame j was integrated); for each such frame that may update it (block_may_update) the
// block's mark gets bit j, and a block whose mark was empty (no band of the batch crossed it)
// is appended to the batch's list, in the workgroup's stripe; the carve word of that stripe's
// line counts the mark bits the pass added. Runs after the batch's allocation and before its
// integration.
constexpr uint32_t kCarveGroups = 2048;
__global__ __launch_bounds__(256) void k_carve(FrameArgs a, uint32_t k) {
  __shared__ float s_pose[kMaxBatch][12];
  FrameCtl* ctl = a.ctl;
  const uint32_t f0 = uniform(ctl->frame_id), parity = uniform(ctl->batch_id) & 1u,
                 cur = uniform(ctl->cursor[a.cursor_id]);
  const uint32_t n = min(uniform(ctl->pool_count), a.pool_cap);
  stage_poses(a, cur, k, s_pose);
  const int lane = threadIdx.x & 63;
  const uint32_t stripe = blockIdx.x & (kStripes - 1);
  uint32_t* line = list_count_of(ctl, parity) + stripe * kLine;
  uint32_t* marks = marks_of(a, parity);
  const size_t ntile = (size_t)a.tiles_x * a.tiles_y;
  for (uint32_t b0 = blockIdx.x * 256u; b0 < n; b0 += gridDim.x * 256u) {
    const uint32_t b = b0 + threadIdx.x;
    uint32_t mask = 0u, slot = 0u;
    if (b < n) {
      const unsigned long long info = a.block_info[b];
      slot = (uint32_t)info;
      // birth frame relative to f0; for a block born in this batch the first frame whose bands
      // cross it (the recorded frame is that of the lane that inserted the key, in no fixed order)
      int32_t born = (int32_t)((uint32_t)(info >> 32) - f0);
      if (born >= 0) born = (int32_t)__builtin_ctz(marks[slot] | 1u << (k - 1u));
      int bx, by, bz;
      unpack_key(a.block_keys[b], bx, by, bz);
      for (uint32_t j = 0; j < k; ++j)
        if (born <= (int32_t)j &&
            block_may_update(a, s_pose[j], bx, by, bz, a.tilemax + ((size_t)parity * kMaxBatch + j) * ntile))
          mask |= 1u << j;
    }
    uint32_t old = 0u;
    if (mask) old = atomicOr(&marks[slot], mask);
    // block-frame updates the carve pass adds (frames whose bands did not cross the block)
    uint32_t added = (uint32_t)__popc(mask & ~old);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) added += (uint32_t)__shfl_xor((int)added, o);
    if (lane == 0 && added) atomicAdd(&line[kLineCarve], added);
    const bool first = mask != 0u && old == 0u;  // no band of the batch listed the block
    const uint64_t fm = __ballot(first);
    if (fm) {
      const int fl = first_lane(fm);
      uint32_t tbase = 0;
      if (lane == fl) tbase = atomicAdd(&line[0], (uint32_t)__popcll(fm));
      tbase = read_lane_u32(tbase, fl);
      if (first) {
        const uint32_t pos = tbase + lanes_below(fm);
        if (pos < a.stripe_cap) {
          list_of(a, parity)[(size_t)stripe * a.stripe_cap + pos] = slot;
        } else {
          atomicExch(&marks[slot], 0u);
          raise_flag(ctl, kFlagTouchedFull);
        }
      }
    }
  }
}

// ============================================================================ marching cubes
constexpr int kHalo = 9;
constexpr int kHalo3 = kHalo * kHalo * kHalo;
constexpr int kItemCap = 512;  // (cube, triangle) items listed per round (a block averages ~80)
// Extraction workgroups: kMcWaves independent waves, one block each, each with its own LDS
// (McShared). A wave only exchanges data with itself through LDS, and executes its LDS
// instructions in order, so wave_sync (a barrier to the compiler's reordering) suffices
// between a write and other lanes' reads. One wave per workgroup: four (24 instead of 16
// resident waves per CU) made the room_medium_5mm extraction slower, 0.87 against 0.69 ms.
constexpr int kMcWaves = 1;
__device__ __forceinline__ int mc_lane() { return (int)(threadIdx.x & 63u); }
__device__ __forceinline__ int mc_wave() { return (int)(threadIdx.x >> 6); }
__device__ __forceinline__ void wave_sync() { __builtin_amdgcn_wave_barrier(); }

// Cases in corner-plane order: bit 4 * dx + 2 * dy + dz of a permuted case is the sign bit of
// the cube corner at offset (dx, dy, dz), so that the low nibble holds the x = cx face and the
// high nibble the x = cx + 1 face, each in slot order (dy << 1) | dz. kPermOfCase maps a case
// (bit c: reference corner c) to its permuted form, four cases per word.
struct McPerm {
  uint32_t w[64];
};
constexpr McPerm mc_perm_table() {
  McPerm t{};
  for (int ci = 0; ci < 256; ++ci) {
    uint32_t p = 0;
    for (int c = 0; c < 8; ++c)
      p |= (uint32_t)((ci >> c) & 1) << (4 * corner_dx(c) + 2 * corner_dy(c) + corner_dz(c));
    t.w[ci >> 2] |= p << (8 * (ci & 3));
  }
  return t;
}
constexpr McPerm kPermHost = mc_perm_table();  // the compile-time copy that mc_perm_ok checks
constexpr bool mc_perm_ok() {  // a bijection fixing 0 and 255, and corner 0 of the x = cx face at bit 0
  bool seen[256] = {};
  for (int ci = 0; ci < 256; ++ci) {
    const uint32_t p = (kPermHost.w[ci >> 2] >> (8 * (ci & 3))) & 255u;
    if (seen[p]) return false;
    seen[p] = true;
  }
  return (kPermHost.w[0] & 255u) == 0u && (kPermHost.w[63] >> 24) == 255u && ((kPermHost.w[0] >> 8) & 255u) == 1u;
}
static_assert(mc_perm_ok(), "permuted case table is not a bijection");
// What a wave's LDS holds of the case table, as words: by permuted case the case and its triangles << 8
// (case 255 as 0), two per word, then the triangles of each case, four per word.
struct McCaseWords {
  uint32_t pc[128], cnt[64];
};
constexpr McCaseWords mc_case_words() {
  McCaseWords t{};
  for (int ci = 0; ci < 256; ++ci) {
    const uint32_t p = (kPermHost.w[ci >> 2] >> (8 * (ci & 3))) & 255u, n = (uint32_t)(kTriTable[ci] >> 60);
    t.pc[p >> 1] |= ((ci == 255 ? 0u : (uint32_t)ci) | n << 8) << (16 * (p & 1u));
    t.cnt[ci >> 2] |= n << (8 * (ci & 3));
  }
  return t;
}
__device__ __constant__ const McCaseWords kCaseWords = mc_case_words();

// LDS of one extraction wave (about 4.9 KB).
struct McShared {
  float val[kHalo3];   // 9^3 tile (x*81 + y*9 + z): tsdf, NaN where unobserved
  uint64_t col[81];    // column words (mc_col_bits) of the 9 x 9 (y, z) columns, index y*9 + z
  uint32_t nb[8];      // pool blocks of the neighbourhood, index (dx << 2) | (dy << 1) | dz
  uint16_t pc[256];    // by permuted case: case | triangles << 8 (case 255 stored as 0)
  uint8_t cnt[256];    // triangles of each case (table count)
  uint8_t cases[512];  // case per cube (x*64 + y*8 + z); 0 = no triangles
};
static_assert(offsetof(McShared, cnt) % 4 == 0 && offsetof(McShared, pc) % 8 == 0, "mc_put_counts writes four entries at a time");
// Item lists of the write passes (k_mc_write, k_ix_write).
struct McItems {
  uint32_t lane_off[65];     // exclusive prefix of table triangles per lane
  uint16_t items[kItemCap];  // (cube << 3) | t of the current round
};

// The case words into S.pc and S.cnt in two steps, so that the loads can be
// issued first and the LDS writes made after the block's own loads are out. As a table of their own
// they are 12 bytes a lane; from kTriTable (32 bytes a lane) and the permutation they were
// a third of a block's load cycles (the writing pass of 144,600 blocks, FP32: 289 -> 283 us).
struct McCounts {
  uint2 pc;
  uint32_t cnt;
};
__device__ __forceinline__ McCounts mc_fetch_counts() {
  const int lane = mc_lane();
  return {*reinterpret_cast<const uint2*>(&kCaseWords.pc[2 * lane]), kCaseWords.cnt[lane]};
}
__device__ __forceinline__ void mc_put_counts(McShared& S, const McCounts& c) {
  const int lane = mc_lane();
  *reinterpret_cast<uint2*>(&S.pc[4 * lane]) = c.pc;
  *reinterpret_cast<uint32_t*>(&S.cnt[4 * lane]) = c.cnt;
}

// Column word of one (y, z) column of the tile, built from its 9 values (x = 0..8) by
// mc_col_bits: bit 4x (x < 8) or bit 32 (x = 8) set iff the value is negative, bit 33 + x
// iff it is unobserved (NaN), bit 42 + x iff |value| < tiny. The 4x spacing interleaves the
// four columns of a cube's corners into one nibble per x-plane.
template <bool kTiny>
__device__ __forceinline__ void mc_col_bits(float v, int x, float tiny, uint32_t& q, uint32_t& m) {
  const uint32_t neg = v < 0.0f ? 1u : 0u;
  if (x < 8) q |= neg << (4 * x);
  else m |= neg;
  m |= (__builtin_isnan(v) ? 2u : 0u) << x;
  if (kTiny) m |= (__builtin_fabsf(v) < tiny ? 1024u : 0u) << x;
}
__device__ __forceinline__ uint64_t mc_col_word(uint32_t q, uint32_t m) { return (uint64_t)q | (uint64_t)m << 32; }

// Threshold of mc_count_exact for the block at lattice origin (gx0, gy0, gz0): above the
// snap bound 1e-5 and above ulp(c) for every lattice coordinate c of the block and its
// +1 layer (ulp(c) <= |c| * 2^-23).
__device__ __forceinline__ float mc_tiny(int gx0, int gy0, int gz0) {
  const int m = max(max(max(abs(gx0), abs(gx0 + 8)), max(abs(gy0), abs(gy0 + 8))), max(abs(gz0), abs(gz0 + 8)));
  return 2e-5f + (float)(m + 1) * 0x1p-22f;
}

// The neighbourhood word of lane l of block b (k_mc_neighbours): lanes 0..7 hold the 8 entries.
__device__ __forceinline__ uint32_t mc_nbr(const McArgs& a, uint32_t b) {
  return a.nbrs[(size_t)b * 8 + (mc_lane() & 7)];
}
// A lane's values of the block's 9^3 tile (NaN where unobserved): column (y, z) = (lane >> 3, lane & 7)
// of the block itself, the faces' values (8, y, z), (y, 8, z) and (y, z, 8), and in lanes 0..24 one of the three
// edges' and the corner's (tile index, column and x in edst, ecol, ex).
struct McTile {
  float own[8], fx, fy, fz, e;
  int edst, ecol, ex;
};
// One wave per pool block. The block's 8^3 voxels and the +x/+y/+z faces, edges and corner
// of its 7 neighbours (one hash lookup each) are loaded: eight
// coalesced rows of the block itself, one load per face, one for the three edges and the
// corner, so no lane divides an index. A corner is observed iff its block exists and its
// weight is > 0. kColor: the colour pool words of the same
// voxels go to col (9^3 tile order) with the same accesses.
// nbr: mc_nbr(a, b), which the caller may have loaded early.
template <int kStorage, bool kColor>
__device__ __forceinline__ void mc_load(const McArgs& a, uint32_t b, uint32_t nbr, McShared& S, uint32_t* col, McTile& T,
                                        int& gx0, int& gy0, int& gz0) {
  using IO = VoxelIO<kStorage>;
  using Word = typename IO::Word;
  const int lane = mc_lane();
  int bx, by, bz;
  unpack_key(a.block_keys[b], bx, by, bz);
  // the neighbourhood in lanes 0..7, read by the wave from its registers; loaded before the
  // block's own voxels, so that waiting for it does not wait for them
  const uint32_t nbv = lane < 8 ? nbr : kNoBlock;
  auto nb_of = [&](int o) { return (uint32_t)__builtin_amdgcn_readlane((int)nbv, o); };
  const Word* vox = reinterpret_cast<const Word*>(a.voxels);
  const float nan = __builtin_nanf("");
  auto value = [&](Word w) {
    float sv, wv;
    IO::unpack(w, sv, wv);
    return wv > 0.0f ? sv : nan;
  };
  const int hi = lane >> 3, lo = lane & 7;
  // this block: voxel lane + 64k = (k, hi, lo)
  const Word* own = vox + (size_t)b * kB3 + lane;
  Word w[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) w[k] = own[64 * k];
  if (lane < 8) S.nb[lane] = nbv;
  // faces x = 8 (voxel (0, hi, lo) of +x), y = 8 ((hi, 0, lo) of +y), z = 8 ((hi, lo, 0) of +z);
  // an absent neighbour's loads read this block instead (their values are not used), so that
  // every load is issued at once, with no wait between them
  const uint32_t nfx = nb_of(4), nfy = nb_of(2), nfz = nb_of(1);
  const auto safe = [&](uint32_t n) { return (size_t)(n != kNoBlock ? n : b) * kB3; };
  const Word wfx = vox[safe(nfx) + lane];
  const Word wfy = vox[safe(nfy) + hi * 64 + lo];
  const Word wfz = vox[safe(nfz) + hi * 64 + lo * 8];
  // edges (8, 8, z) of +x+y, (8, y, 8) of +x+z, (x, 8, 8) of +y+z (8 lanes each), corner
  // (8, 8, 8) of +x+y+z (lane 24)
  int edst = 0, ecol = 0, ex = 8;
  uint32_t enb = kNoBlock;
  int esrc = 0;
  const uint32_t ne6 = nb_of(6), ne5 = nb_of(5), ne3 = nb_of(3), ne7 = nb_of(7);
  if (lane < 8) { enb = ne6; esrc = lane; edst = 8 * 81 + 8 * 9 + lane; ecol = 72 + lane; }
  else if (lane < 16) { enb = ne5; esrc = (lane - 8) * 8; edst = 8 * 81 + (lane - 8) * 9 + 8; ecol = (lane - 8) * 9 + 8; }
  else if (lane < 24) { enb = ne3; esrc = (lane - 16) * 64; edst = (lane - 16) * 81 + 8 * 9 + 8; ecol = 80; ex = lane - 16; }
  else if (lane == 24) { enb = ne7; esrc = 0; edst = kHalo3 - 1; ecol = 80; }
  const Word we = vox[safe(enb) + esrc];
  if constexpr (kColor) {
    const uint32_t* cp = a.colors;
    uint32_t c[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) c[k] = cp[(size_t)b * kB3 + lane + 64 * k];
    const uint32_t rfx = cp[safe(nfx) + lane], rfy = cp[safe(nfy) + hi * 64 + lo], rfz = cp[safe(nfz) + hi * 64 + lo * 8],
                   re = cp[safe(enb) + esrc];
    const uint32_t cfx = nfx != kNoBlock ? rfx : 0u, cfy = nfy != kNoBlock ? rfy : 0u, cfz = nfz != kNoBlock ? rfz : 0u,
                   ce = enb != kNoBlock ? re : 0u;
#pragma unroll
    for (int k = 0; k < 8; ++k) col[k * 81 + hi * 9 + lo] = c[k];
    col[8 * 81 + hi * 9 + lo] = cfx;
    col[hi * 81 + 8 * 9 + lo] = cfy;
    col[hi * 81 + lo * 9 + 8] = cfz;
    if (lane < 25) col[edst] = ce;
  }
  gx0 = bx * kB;
  gy0 = by * kB;
  gz0 = bz * kB;
#pragma unroll
  for (int k = 0; k < 8; ++k) T.own[k] = value(w[k]);
  T.fx = nfx != kNoBlock ? value(wfx) : nan;
  T.fy = nfy != kNoBlock ? value(wfy) : nan;
  T.fz = nfz != kNoBlock ? value(wfz) : nan;
  T.e = enb != kNoBlock ? value(we) : nan;  // lanes 25..: NaN
  T.edst = edst;
  T.ecol = ecol;
  T.ex = ex;
}
// True iff some lane's value satisfies f; gathered as ballots, one scalar instruction per value.
template <class F>
__device__ __forceinline__ bool mc_any(const McTile& T, F f) {
  uint64_t m = __builtin_amdgcn_ballot_w64(f(T.fx)) | __builtin_amdgcn_ballot_w64(f(T.fy)) |
               __builtin_amdgcn_ballot_w64(f(T.fz)) | __builtin_amdgcn_ballot_w64(f(T.e));
#pragma unroll
  for (int k = 0; k < 8; ++k) m |= __builtin_amdgcn_ballot_w64(f(T.own[k]));
  return m != 0u;
}
// Whether the observed values include both a negative value and a non-negative one: otherwise
// every cube's case is 0 or 255 (or it is unobserved), and the block has no triangles. Asked before
// anything else is made of the values: some four blocks in ten have none.
__device__ __forceinline__ bool mc_crossed(const McTile& T) {
  return mc_any(T, [](float v) { return v < 0.0f; }) && mc_any(T, [](float v) { return v >= 0.0f; });
}
// The values into S.val.
__device__ __forceinline__ void mc_put_values(McShared& S, const McTile& T) {
  const int lane = mc_lane(), hi = lane >> 3, lo = lane & 7;
#pragma unroll
  for (int k = 0; k < 8; ++k) S.val[k * 81 + hi * 9 + lo] = T.own[k];
  S.val[8 * 81 + hi * 9 + lo] = T.fx;
  S.val[hi * 81 + 8 * 9 + lo] = T.fy;
  S.val[hi * 81 + lo * 9 + 8] = T.fz;
  if (lane < 25) S.val[T.edst] = T.e;
}
// The column words of the 81 columns into S.col, with kTiny the |value| < tiny bits (otherwise none).
template <bool kTiny>
__device__ __forceinline__ void mc_put_columns(McShared& S, const McTile& T, float tiny) {
  const int lane = mc_lane(), hi = lane >> 3, lo = lane & 7;
  // the border columns (y, 8), (8, z) and (8, 8) collect their values from other lanes
  if (lane < 17) S.col[lane < 8 ? lane * 9 + 8 : 64 + lane] = 0u;
  // own column (hi, lo): x = 0..7 from the block, x = 8 from the +x face
  uint32_t cq = 0u, cm = 0u;
#pragma unroll
  for (int k = 0; k < 8; ++k) mc_col_bits<kTiny>(T.own[k], k, tiny, cq, cm);
  mc_col_bits<kTiny>(T.fx, 8, tiny, cq, cm);
  S.col[hi * 9 + lo] = mc_col_word(cq, cm);
  wave_sync();  // the border words are clear
  uint32_t yq = 0u, ym = 0u, zq = 0u, zm = 0u, eq = 0u, em = 0u;
  mc_col_bits<kTiny>(T.fy, hi, tiny, yq, ym);  // (hi, 8, lo): column (8, lo) at x = hi
  mc_col_bits<kTiny>(T.fz, hi, tiny, zq, zm);  // (hi, lo, 8): column (lo, 8) at x = hi
  mc_col_bits<kTiny>(T.e, T.ex, tiny, eq, em);
  atomicOr(reinterpret_cast<unsigned long long*>(&S.col[72 + lo]), (unsigned long long)mc_col_word(yq, ym));
  atomicOr(reinterpret_cast<unsigned long long*>(&S.col[lo * 9 + 8]), (unsigned long long)mc_col_word(zq, zm));
  if (lane < 25) atomicOr(reinterpret_cast<unsigned long long*>(&S.col[T.ecol]), (unsigned long long)mc_col_word(eq, em));
  wave_sync();
}
// The staging of the write passes: values and columns of block b.
template <int kStorage, bool kColor>
__device__ __forceinline__ void mc_stage(const McArgs& a, uint32_t b, uint32_t nbr, McShared& S, uint32_t* col, int& gx0,
                                         int& gy0, int& gz0) {
  McTile T;
  mc_load<kStorage, kColor>(a, b, nbr, S, col, T, gx0, gy0, gz0);
  mc_put_values(S, T);
  mc_put_columns<false>(S, T, 0.0f);
}

// Lane l classifies the 8 cubes of its (y, z) column (x = 0..7) from the column words of
// its 4 corner columns (slot k = (dy << 1) | dz: column (y + dy, z + dz)): interleaved, each
// x-plane is one nibble, and a cube's permuted case is the byte of its two faces. A cube has
// triangles iff its 8 corners are observed and its case is not 0 or 255 (bit c set iff
// corner c < 0, reference corner order); its case goes to S.cases. Returns the lane's table
// triangle count. near: bit x set iff cube x of the column has triangles and a corner with
// |value| < tiny (the kTiny bits of mc_put_columns; see mc_count_exact).
__device__ __forceinline__ uint32_t mc_classify(McShared& S, uint32_t& near) {
  const int lane = mc_lane(), i = (lane >> 3) * 9 + (lane & 7);
  const uint64_t w0 = S.col[i], w1 = S.col[i + 1], w2 = S.col[i + 9], w3 = S.col[i + 10];
  const uint32_t q = (uint32_t)w0 | (uint32_t)w1 << 1 | (uint32_t)w2 << 2 | (uint32_t)w3 << 3;
  const uint32_t m0 = (uint32_t)(w0 >> 32), m1 = (uint32_t)(w1 >> 32), m2 = (uint32_t)(w2 >> 32),
                 m3 = (uint32_t)(w3 >> 32);
  const uint32_t q8 = (m0 & 1u) | (m1 & 1u) << 1 | (m2 & 1u) << 2 | (m3 & 1u) << 3;  // x = 8 nibble
  const uint32_t um = m0 | m1 | m2 | m3;  // unobserved / small bits of any corner column
  uint32_t ntri = 0;
  near = 0u;
#pragma unroll
  for (int cx = 0; cx < 8; ++cx) {
    const uint32_t p = cx < 7 ? (q >> (4 * cx)) & 255u : (q >> 28) | (q8 << 4);
    const uint32_t e = S.pc[p];
    const bool obs = ((um >> (1 + cx)) & 3u) == 0u;
    const uint32_t ci = obs ? e & 255u : 0u, n = obs ? e >> 8 : 0u;
    if (n != 0u && ((um >> (10 + cx)) & 3u) != 0u) near |= 1u << cx;
    S.cases[cx * 64 + lane] = (uint8_t)ci;
    ntri += n;
  }
  return ntri;
}

// Exclusive prefix of the lanes' counts n into I.lane_off, I.lane_off[64] the total, which it
// returns.
__device__ __forceinline__ uint32_t mc_lane_prefix(McItems& I, uint32_t n) {
  const int lane = mc_lane();
  uint32_t x = n;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)x, off);
    if (lane >= off) x += y;
  }
  I.lane_off[lane] = x - n;
  if (lane == 63) I.lane_off[64] = x;
  wave_sync();
  return I.lane_off[64];
}

__device__ __forceinline__ uint32_t mc_wave_sum(uint32_t n) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) n += (uint32_t)__shfl_xor((int)n, m);
  return n;
}

// Per cube edge e, 5 bits at 5e: the offset of its lower end point in the cube (dx | dy << 1
// | dz << 2) and its axis << 3 (0 x, 1 y, 2 z).
constexpr uint64_t edge_lo_table() {
  uint64_t t = 0;
  for (int e = 0; e < 12; ++e) {
    const int a = edge_a(e), b = edge_b(e);
    const int dx = corner_dx(a) < corner_dx(b) ? corner_dx(a) : corner_dx(b);
    const int dy = corner_dy(a) < corner_dy(b) ? corner_dy(a) : corner_dy(b);
    const int dz = corner_dz(a) < corner_dz(b) ? corner_dz(a) : corner_dz(b);
    const int axis = corner_dx(a) != corner_dx(b) ? 0 : (corner_dy(a) != corner_dy(b) ? 1 : 2);
    t |= (uint64_t)(dx | dy << 1 | dz << 2 | axis << 3) << (5 * e);
  }
  return t;
}
constexpr uint64_t kEdgeLo = edge_lo_table();
// kEdgeUp bit e: the reference's first end point of cube edge e (edge_a) is its upper end.
constexpr uint32_t edge_up_table() {
  uint32_t m = 0;
  for (int e = 0; e < 12; ++e) {
    const int a = edge_a(e), b = edge_b(e);
    if (corner_dx(a) + corner_dy(a) + corner_dz(a) > corner_dx(b) + corner_dy(b) + corner_dz(b)) m |= 1u << e;
  }
  return m;
}
constexpr uint32_t kEdgeUp = edge_up_table();

// vertex_interp (the reference's VertexInterp, src/tsdf.cu:1640-1660) from tile corner ia to
// tile corner ib of one lattice edge along axis, with kColor vertex_interp_rgb's colour. The
// end points differ along that axis only, so the other two coordinates are the lower end
// point's (fx, fy, fz) exactly (mu * 0 adds zero), and p2 - p1 along the axis is exactly +-1
// (g: the lower end point's lattice coordinate on the axis; up: ia is the upper end). The
// quotient is formed on every lane and dropped where a snap applies, so that the wave takes no
// branch.
template <bool kColor>
__device__ __forceinline__ void mc_interp(const McShared& S, const uint32_t* col, int ia, int ib, uint32_t axis, int g,
                                          bool up, float fx, float fy, float fz, float& x, float& y, float& z,
                                          uint32_t& c) {
  const float va = S.val[ia], vb = S.val[ib];
  const float pl = (float)g, pu = (float)(g + 1);
  const float pa = up ? pu : pl, pb = up ? pl : pu;
  const bool sa = near_iso(va), sb = !sa && near_iso(vb), sd = !sa && !sb && near_iso(va - vb);
  const float mu = (0.0f - va) / (vb - va);
  const float t = sa || sd ? pa : (sb ? pb : pa + mu * (pb - pa));
  x = axis == 0u ? t : fx;
  y = axis == 1u ? t : fy;
  z = axis == 2u ? t : fz;
  if constexpr (kColor) {
    const uint32_t c1 = col[ia], c2 = col[ib];
    uint32_t cl = 0u;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int a = (int)((c1 >> (8 * k)) & 255u), b = (int)((c2 >> (8 * k)) & 255u);
      const float v = (float)a + mu * (float)(b - a);
      cl |= (uint32_t)(uint8_t)v << (8 * k);
    }
    c = sa || sd ? c1 : (sb ? c2 : cl);
  }
}

// Vertex (voxel units) of cube edge e of cube (cx, cy, cz): mc_interp from corner edge_a(e) to
// edge_b(e), the edge decoded from the packed tables.
template <bool kColor>
__device__ __forceinline__ void mc_vertex(const McShared& S, const uint32_t* col, int e, int cx, int cy, int cz,
                                          int gx0, int gy0, int gz0, float& x, float& y, float& z, uint32_t& c) {
  const uint32_t info = (uint32_t)(kEdgeLo >> (5 * e)) & 31u;
  const int lx = cx + (int)(info & 1u), ly = cy + (int)((info >> 1) & 1u), lz = cz + (int)((info >> 2) & 1u);
  const uint32_t axis = info >> 3;
  const int il = lx * 81 + ly * 9 + lz, iu = il + (axis == 0u ? 81 : (axis == 1u ? 9 : 1));
  const bool up = ((kEdgeUp >> e) & 1u) != 0u;
  const int g = axis == 0u ? gx0 + lx : (axis == 1u ? gy0 + ly : gz0 + lz);
  mc_interp<kColor>(S, col, up ? iu : il, up ? il : iu, axis, g, up, (float)(gx0 + lx), (float)(gy0 + ly),
                    (float)(gz0 + lz), x, y, z, c);
}

// Vertices (voxel units) of table triangle t of cube (cx, cy, cz) with case ci, and with
// kColor their colours; false for a degenerate triangle (two equal vertices; the
// reference's test at src/tsdf.cu:1055-1058, with its typo corrected).
template <bool kColor>
__device__ __forceinline__ bool mc_triangle(const McShared& S, const uint32_t* col, int ci, int t, int cx, int cy,
                                            int cz, int gx0, int gy0, int gz0, float* P, uint32_t* C) {
  const uint64_t pk = kTriTable[ci];
#pragma unroll
  for (int j = 0; j < 3; ++j)
    mc_vertex<kColor>(S, col, (int)((pk >> (4 * (3 * t + j))) & 15u), cx, cy, cz, gx0, gy0, gz0, P[3 * j],
                      P[3 * j + 1], P[3 * j + 2], C[j]);
  const bool d01 = P[0] == P[3] && P[1] == P[4] && P[2] == P[5];
  const bool d12 = P[3] == P[6] && P[4] == P[7] && P[5] == P[8];
  const bool d20 = P[6] == P[0] && P[7] == P[1] && P[8] == P[2];
  return !(d01 || d12 || d20);
}

// Triangles that k_mc_write will emit for the lane's column, without computing vertices
// where none can coincide. Vertices of one triangle lie on three distinct cube edges, in
// the closed edge segments (the other two coordinates are exact lattice values, the
// interpolation parameter lies in [0, 1]); two such points can only be equal at a corner
// the two edges share, and a vertex lands exactly on corner a of its edge only by a snap
// (|v_a| <= 1e-5, or |v_a - v_b| <= 1e-5 with opposite signs) or by rounding a + mu*(b - a)
// to a, which needs |mu| <= ulp(a)/2 and so |v_a| <= ulp(a) (|v_b - v_a| <= 2); likewise for
// b. A cube whose corners all have |value| >= tiny (tiny above both bounds) therefore emits
// exactly its table count; the others ("near" bits) are counted triangle by triangle.

// Edges of case ci whose two corners lie on opposite sides (bit e): corners 0-3 and 4-7 form
// the z = 0 and z = 1 rings (edges 0-3 and 4-7 join ring neighbours i, i + 1 mod 4), edges
// 8-11 join corner i to corner i + 4.
__host__ __device__ constexpr uint32_t crossed_edges(int ci) {
  const uint32_t lo = (uint32_t)ci & 15u, hi = ((uint32_t)ci >> 4) & 15u;
  const uint32_t rlo = ((lo >> 1) | (lo << 3)) & 15u, rhi = ((hi >> 1) | (hi << 3)) & 15u;
  return (lo ^ rlo) | ((hi ^ rhi) << 4) | ((lo ^ hi) << 8);
}
constexpr bool crossed_edges_ok() {
  for (int ci = 0; ci < 256; ++ci)
    for (int e = 0; e < 12; ++e)
      if ((((ci >> edge_a(e)) ^ (ci >> edge_b(e))) & 1) != (int)((crossed_edges(ci) >> e) & 1u)) return false;
  return true;
}
static_assert(crossed_edges_ok(), "crossed_edges disagrees with the edge table");

// Non-degenerate table triangles of a near cube (case ci at (cx, cy, cz)): vertex_end tells
// on which corner, if any, each vertex lands, so no positions are formed; a triangle is
// degenerate when two of its vertices land on the same corner (the only way two vertices
// on distinct edges coincide), which is what mc_triangle's position test finds. Corners are
// named by their tile index; edges are decoded as in mc_vertex.
__device__ __forceinline__ uint32_t mc_count_near(const McShared& S, int ci, int cx, int cy, int cz, int gx0,
                                                  int gy0, int gz0) {
  const uint64_t pk = kTriTable[ci];
  const int nt = S.cnt[ci];
  uint32_t n = 0;
  for (int t = 0; t < nt; ++t) {
    int cid[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int e = (int)((pk >> (4 * (3 * t + j))) & 15u);
      const uint32_t info = (uint32_t)(kEdgeLo >> (5 * e)) & 31u;
      const int lx = cx + (int)(info & 1u), ly = cy + (int)((info >> 1) & 1u), lz = cz + (int)((info >> 2) & 1u);
      const uint32_t axis = info >> 3;
      const int il = lx * 81 + ly * 9 + lz, iu = il + (axis == 0u ? 81 : (axis == 1u ? 9 : 1));
      const bool up = ((kEdgeUp >> e) & 1u) != 0u;
      const int ia = up ? iu : il, ib = up ? il : iu;
      const int g = axis == 0u ? gx0 + lx : (axis == 1u ? gy0 + ly : gz0 + lz);
      const float pl = (float)g, pu = (float)(g + 1);
      const int end = vertex_end(up ? pu : pl, up ? pl : pu, S.val[ia], S.val[ib]);
      cid[j] = end == 0 ? ia : (end == 1 ? ib : -1 - j);
    }
    n += (cid[0] != cid[1] && cid[1] != cid[2] && cid[2] != cid[0]) ? 1u : 0u;
  }
  return n;
}

// The lane's emitted triangles from its table count n: near cubes are counted triangle by
// triangle.
__device__ __forceinline__ uint32_t mc_count_exact(const McShared& S, uint32_t near, uint32_t n, int gx0, int gy0,
                                                   int gz0) {
  const int lane = mc_lane(), cy = lane >> 3, cz = lane & 7;
  for (uint32_t m = near; m; m &= m - 1u) {
    const int cx = __builtin_ctz(m);
    const int ci = S.cases[cx * 64 + lane];
    n += mc_count_near(S, ci, cx, cy, cz, gx0, gy0, gz0) - (uint32_t)S.cnt[ci];
  }
  return n;
}

// The block's (cube, table triangle) items in order lane, x, t, in rounds of kItemCap: each
// lane lists its own items of the round in LDS, then the wave takes them one per lane.
// Emit receives (valid, cube x/y/z, case, t, P[9], C[3]) per item slot of a 64-item step;
// With kPos, valid is false for empty slots and for degenerate triangles (two equal
// vertices; the reference's test at src/tsdf.cu:1055-1058, with its typo corrected), and
// kColor makes C hold the vertex colours interpolated from the colour tile col (otherwise
// zeros). Without kPos, P and C are not computed and every item is valid.
template <bool kColor, bool kPos, class Emit>
__device__ __forceinline__ void mc_items(McShared& S, McItems& I, const uint32_t* col, uint32_t total, int gx0, int gy0,
                                         int gz0, Emit emit) {
  const int lane = mc_lane();
  const uint32_t my0 = I.lane_off[lane], my1 = I.lane_off[lane + 1];
  for (uint32_t r0 = 0; r0 < total; r0 += kItemCap) {
    const uint32_t r1 = min(total, r0 + (uint32_t)kItemCap);
    if (my0 < r1 && my1 > r0) {
      uint32_t idx = my0;
      for (int cx = 0; cx < 8 && idx < r1; ++cx) {
        const int cube = cx * 64 + lane;
        const int n = S.cnt[S.cases[cube]];
        for (int t = 0; t < n; ++t, ++idx)
          if (idx >= r0 && idx < r1) I.items[idx - r0] = (uint16_t)((cube << 3) | t);
      }
    }
    wave_sync();
    for (uint32_t i0 = r0; i0 < r1; i0 += 64) {
      const uint32_t item = i0 + lane;
      bool valid = false;
      int ci = 0, t = 0, cx = 0, cy = 0, cz = 0;
      float P[9];
      uint32_t C[3] = {0u, 0u, 0u};
      if (item < r1) {
        const int it = I.items[item - r0];
        const int cube = it >> 3;
        t = it & 7;
        cx = cube >> 6;
        cy = (cube >> 3) & 7;
        cz = cube & 7;
        ci = S.cases[cube];
        if constexpr (kPos) valid = mc_triangle<kColor>(S, col, ci, t, cx, cy, cz, gx0, gy0, gz0, P, C);
        else valid = true;
      }
      emit(valid, gx0 + cx, gy0 + cy, gz0 + cz, ci, t, P, C);
    }
    wave_sync();  // the next round overwrites the items
  }
}


// The pool indices of each block's 8 neighbourhood blocks (+x/+y/+z and their combinations,
// index (dx << 2) | (dy << 1) | dz; itself at 0; kNoBlock where absent), one lane per entry,
// so that the extraction passes read one word instead of walking the hash per neighbour.
// With ebits (indexed mesh), each lane also clears 6 of its block's 48 used-edge words.
__global__ __launch_bounds__(256) void k_mc_neighbours(McArgs a) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)a.n_blocks * 8) return;
  const uint32_t b = (uint32_t)(i >> 3), d = (uint32_t)(i & 7);
  if (a.ebits) {
#pragma unroll
    for (int k = 0; k < 6; ++k) a.ebits[(size_t)b * kEdgeWords + d * 6 + k] = 0u;
  }
  uint32_t nb = b;
  if (d > 0) {
    int bx, by, bz;
    unpack_key(a.block_keys[b], bx, by, bz);
    const int nx = bx + (int)(d >> 2), ny = by + (int)((d >> 1) & 1), nz = bz + (int)(d & 1);
    nb = key_in_range(nx, ny, nz) ? find_block(a.hash, pack_key(nx, ny, nz)) : kNoBlock;
    if (nb >= a.pool_cap) nb = kNoBlock;
  }
  a.nbrs[i] = nb;
}

// Bound by the lines it fetches: 144,600 blocks (FP32) take 202 us and fetch about 1.4 GB for 592 MB of
// own voxels, since the +z face and the edges touch a line per value. Asking mc_crossed first and
// leaving out the values and the near-zero bits took a third of the instructions out and left the
// time as it was.
template <int kStorage>
__global__ __launch_bounds__(64 * kMcWaves) void k_mc_count(McArgs a) {
  __shared__ McShared SS[kMcWaves];
  McShared& S = SS[mc_wave()];
  const int lane = mc_lane();
  const uint32_t b = blockIdx.x * kMcWaves + (uint32_t)mc_wave();
  if (b >= a.n_blocks) return;
  const McCounts counts = mc_fetch_counts();
  McTile T;
  int gx0, gy0, gz0;
  mc_load<kStorage, false>(a, b, mc_nbr(a, b), S, nullptr, T, gx0, gy0, gz0);
  if (!mc_crossed(T)) {  // no triangles
    if (lane == 0) a.counts[b] = 0u;
    return;
  }
  mc_put_counts(S, counts);
  // only a block with a value near zero can hold degenerate triangles: the values themselves and
  // the bits that mark them are for these (one block in a hundred or so)
  const float tiny = mc_tiny(gx0, gy0, gz0);
  const bool near_zero = mc_any(T, [&](float v) { return __builtin_fabsf(v) < tiny; });
  if (near_zero) {
    mc_put_values(S, T);
    mc_put_columns<true>(S, T, tiny);
  } else {
    mc_put_columns<false>(S, T, 0.0f);
  }
  uint32_t near;
  uint32_t cnt = mc_classify(S, near);
  if (near_zero && __ballot(near != 0u)) cnt = mc_count_exact(S, near, cnt, gx0, gy0, gz0);
  cnt = mc_wave_sum(cnt);
  if (lane == 0) a.counts[b] = cnt;
}

// Exclusive scan of counts within chunks of kScanChunk blocks (one workgroup of 256 each,
// 4 counts per lane); chunk totals go to chunk_sums.
__global__ __launch_bounds__(256) void k_scan_chunks(McArgs a) {
  __shared__ uint32_t s_w[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t c0 = blockIdx.x * kScanChunk;
  uint32_t v[4], sum = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t i = c0 + 4 * tid + k;
    v[k] = i < a.n_blocks ? a.counts[i] : 0u;
    sum += v[k];
  }
  uint32_t x = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)x, off);
    if (lane >= off) x += y;
  }
  if (lane == 63) s_w[wave] = x;
  __syncthreads();
  uint32_t pre = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wave) pre += s_w[w];
    tot += s_w[w];
  }
  uint32_t run = pre + x - sum;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t i = c0 + 4 * tid + k;
    if (i < a.n_blocks) a.counts[i] = run;
    run += v[k];
  }
  if (tid == 0) a.chunk_sums[blockIdx.x] = tot;
}

// Exclusive scan of the chunk totals (one workgroup, sequential over groups of 256).
__global__ __launch_bounds__(256) void k_scan_top(McArgs a, uint32_t n_chunks) {
  __shared__ uint32_t s_w[4];
  __shared__ uint32_t s_carry;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) s_carry = 0;
  __syncthreads();
  for (uint32_t b0 = 0; b0 < n_chunks; b0 += 256) {
    const uint32_t i = b0 + tid;
    const uint32_t v = i < n_chunks ? a.chunk_sums[i] : 0u;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)x, off);
      if (lane >= off) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < wave) pre += s_w[w];
      tot += s_w[w];
    }
    const uint32_t carry = s_carry;
    if (i < n_chunks) a.chunk_sums[i] = carry + pre + x - v;
    __syncthreads();
    if (tid == 0) s_carry = carry + tot;
    __syncthreads();
  }
  if (tid == 0) *a.total = s_carry;
}

// Exclusive offset of block b after k_scan_chunks / k_scan_top (the total for b == n).
__device__ __forceinline__ uint32_t block_offset(const uint32_t* counts, const uint32_t* chunk_sums, uint32_t b) {
  return chunk_sums[b / kScanChunk] + counts[b];
}
__device__ __forceinline__ uint32_t block_offset(const uint32_t* counts, const uint32_t* chunk_sums, uint32_t b,
                                                 uint32_t n, const uint32_t* total) {
  return b < n ? block_offset(counts, chunk_sums, b) : *total;
}

template <int kStorage, bool kColor>
__global__ __launch_bounds__(64 * kMcWaves) void k_mc_write(McArgs a) {
  __shared__ McShared SS[kMcWaves];
  __shared__ McItems IS[kMcWaves];
  __shared__ uint32_t s_cols[kMcWaves][kColor ? kHalo3 : 1];
  McShared& S = SS[mc_wave()];
  McItems& I = IS[mc_wave()];
  uint32_t* s_col = s_cols[mc_wave()];
  const uint32_t b = blockIdx.x * kMcWaves + (uint32_t)mc_wave();
  if (b >= a.n_blocks) return;
  {
    const uint32_t nbr = mc_nbr(a, b);  // with the offsets: the staging then needs one round trip
    const McCounts counts = mc_fetch_counts();
    uint32_t pos = block_offset(a.counts, a.chunk_sums, b);
    if (block_offset(a.counts, a.chunk_sums, b + 1, a.n_blocks, a.total) == pos) return;  // no triangles
    int gx0, gy0, gz0;
    mc_stage<kStorage, kColor>(a, b, nbr, S, s_col, gx0, gy0, gz0);
    mc_put_counts(S, counts);
    wave_sync();
    uint32_t near;
    const uint32_t total = mc_lane_prefix(I, mc_classify(S, near));
    mc_items<kColor, true>(S, I, s_col, total, gx0, gy0, gz0,
                           [&](bool valid, int x, int y, int z, int ci, int t, const float* P, const uint32_t* C) {
      const uint64_t m = __ballot(valid);
      const uint32_t p = pos + lanes_below(m);
      if (valid && p < a.capacity) {
        float* o = a.tris + (size_t)p * 9;
#pragma unroll
        for (int k = 0; k < 9; ++k) o[k] = P[k] * a.vox;
        if (a.cubes) {
          int32_t* q = a.cubes + (size_t)p * 4;
          q[0] = x; q[1] = y; q[2] = z; q[3] = (ci << 8) | t;
        }
        if (kColor && a.rgb) {
          uint8_t* o8 = a.rgb + (size_t)p * 9;
#pragma unroll
          for (int k = 0; k < 9; ++k) o8[k] = (uint8_t)(C[k / 3] >> (8 * (k % 3)));
        }
      }
      pos += (uint32_t)__popcll(m);
    });
  }
}

// ---------------------------------------------------------------- indexed mesh
// One vertex per used lattice edge (an edge some face lies on), owned by the block that holds
// the edge's lower end point; its id is the owner's vertex offset plus the edge's rank among
// the owner's used edges (bit order axis * 512 + in-block index). Faces are every table
// triangle of every cube with 8 observed corners (zero-area ones included: dropping them
// would open the mesh where the surface passes exactly through a lattice point), in the
// order of k_mc_write; the table's triangles of a case use exactly the edges whose corners
// differ in sign, so those are the edges marked. Vertices are interpolated from the lower
// end point to the upper one (VertexInterp, src/tsdf.cu:1640-1660, with that orientation):
// every face that uses an edge gets the same vertex, and the mesh has no cracks where
// neighbouring cubes would interpolate an edge in opposite directions (the reference welds
// float-identical coordinates instead, src/tsdf.cu:1772-1850).


// Owner slot (index into S.nb) of edge e of cube (cx, cy, cz) and the edge's bit in its
// owner's used-edge words: the lower end point (block-local, 0..8 per axis) decides both.
__device__ __forceinline__ void edge_owner(int e, int cx, int cy, int cz, int& o, int& bit) {
  const uint32_t info = (uint32_t)(kEdgeLo >> (5 * e)) & 31u;
  const int lx = cx + (int)(info & 1u), ly = cy + (int)((info >> 1) & 1u), lz = cz + (int)((info >> 2) & 1u);
  o = ((lx >> 3) << 2) | ((ly >> 3) << 1) | (lz >> 3);
  bit = (int)(info >> 3) * kB3 + (((lx & 7) << 6) | ((ly & 7) << 3) | (lz & 7));
}

// Marks the used edges and counts the faces (table counts) of each block. Edges are gathered in LDS,
// the block's own and those of its +x/+y/+z neighbours, and merged with one atomic OR per word: what bounds the
// pass is the atomic requests that leave the XCD (one per line and instruction). With the
// neighbours' edges sent one by one, 36 requests a block, 35,900 blocks (FP16) took 87 us, now 61.
template <int kStorage>
__global__ __launch_bounds__(64 * kMcWaves) void k_ix_mark(McArgs a) {
  __shared__ McShared SS[kMcWaves];
  __shared__ uint32_t s_bitss[kMcWaves][8 * kEdgeWords];  // by owner (S.nb)
  McShared& S = SS[mc_wave()];
  uint32_t* s_bits = s_bitss[mc_wave()];
  const int lane = mc_lane();
  const uint32_t b = blockIdx.x * kMcWaves + (uint32_t)mc_wave();
  if (b >= a.n_blocks) return;
  const McCounts counts = mc_fetch_counts();
  {
    McTile T;
    int gx0, gy0, gz0;
    mc_load<kStorage, false>(a, b, mc_nbr(a, b), S, nullptr, T, gx0, gy0, gz0);
    if (!mc_crossed(T)) {  // no faces, no edges
      if (lane == 0) a.counts[b] = 0u;
      return;
    }
    mc_put_counts(S, counts);
    for (int w = lane; w < 8 * kEdgeWords; w += 64) s_bits[w] = 0u;
    mc_put_columns<false>(S, T, 0.0f);
    uint32_t near;
    const uint32_t total = mc_wave_sum(mc_classify(S, near));
    const int cy = lane >> 3, cz = lane & 7;
    for (int cx = 0; cx < 8; ++cx) {
      const int ci = S.cases[cx * 64 + lane];
      for (uint32_t m = ci ? crossed_edges(ci) : 0u; m; m &= m - 1u) {
        const int e = __builtin_ctz(m);
        int o, bit;
        edge_owner(e, cx, cy, cz, o, bit);
        atomicOr(&s_bits[o * kEdgeWords + (bit >> 5)], 1u << (bit & 31));
      }
    }
    if (lane == 0) a.counts[b] = total;
    wave_sync();
#pragma unroll
    for (int k = 0; k < 8 * kEdgeWords / 64; ++k) {
      const int w = 64 * k + lane, o = w / kEdgeWords;
      const uint32_t bits = s_bits[w];  // an absent neighbour's cubes are unobserved: no bits
      if (bits) atomicOr(&a.ebits[(size_t)S.nb[o] * kEdgeWords + (w - o * kEdgeWords)], bits);
    }
  }
}

// Per block: popcount prefixes of the 48 used-edge words and the block's vertex count (one
// wave per block, lanes 0..47 one word each).
__global__ __launch_bounds__(256) void k_ix_count(McArgs a) {
  const int lane = threadIdx.x & 63;
  for (uint32_t b = blockIdx.x * 4u + (threadIdx.x >> 6); b < a.n_blocks; b += gridDim.x * 4u) {
    const uint32_t w = lane < kEdgeWords ? a.ebits[(size_t)b * kEdgeWords + lane] : 0u;
    const uint32_t c = (uint32_t)__popc(w);
    uint32_t x = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)x, off);
      if (lane >= off) x += y;
    }
    if (lane < kEdgeWords) a.epre[(size_t)b * kEdgeWords + lane] = (uint16_t)(x - c);
    if (lane == kEdgeWords - 1) a.vcounts[b] = x;
  }
}

// Faces (vertex ids of each table triangle's corners) and the vertices each block owns.
template <int kStorage, bool kColor>
__global__ __launch_bounds__(64 * kMcWaves) void k_ix_write(McArgs a) {
  __shared__ McShared SS[kMcWaves];
  __shared__ McItems IS[kMcWaves];
  __shared__ uint32_t s_cols[kMcWaves][kColor ? kHalo3 : 1];
  __shared__ uint32_t s_vbases[kMcWaves][8];
  McShared& S = SS[mc_wave()];
  McItems& I = IS[mc_wave()];
  uint32_t* s_col = s_cols[mc_wave()];
  uint32_t* s_vbase = s_vbases[mc_wave()];
  const int lane = mc_lane();
  const uint32_t b = blockIdx.x * kMcWaves + (uint32_t)mc_wave();
  if (b >= a.n_blocks) return;
  {
    uint32_t pos = block_offset(a.counts, a.chunk_sums, b);
    if (block_offset(a.counts, a.chunk_sums, b + 1, a.n_blocks, a.total) == pos &&
        block_offset(a.vcounts, a.vchunks, b + 1, a.n_blocks, a.vtotal) == block_offset(a.vcounts, a.vchunks, b))
      return;  // no faces and no vertices of its own
    const McCounts counts = mc_fetch_counts();
    int gx0, gy0, gz0;
    mc_stage<kStorage, kColor>(a, b, mc_nbr(a, b), S, s_col, gx0, gy0, gz0);
    mc_put_counts(S, counts);
    wave_sync();
    if (lane < 8) {
      const uint32_t nb = S.nb[lane];
      s_vbase[lane] = nb != kNoBlock ? a.vchunks[nb / kScanChunk] + a.vcounts[nb] : 0u;
    }
    uint32_t near;
    const uint32_t total = mc_lane_prefix(I, mc_classify(S, near));  // ends with a barrier
    mc_items<false, false>(S, I, nullptr, total, gx0, gy0, gz0,
                           [&](bool valid, int x, int y, int z, int ci, int t, const float*, const uint32_t*) {
      const uint64_t m = __ballot(valid);
      const uint32_t p = pos + lanes_below(m);
      if (valid && p < a.capacity) {
        const uint64_t pk = kTriTable[ci];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          int o, bit;
          edge_owner((int)((pk >> (4 * (3 * t + j))) & 15u), x - gx0, y - gy0, z - gz0, o, bit);
          const size_t wi = (size_t)S.nb[o] * kEdgeWords + (bit >> 5);
          const uint32_t below = a.ebits[wi] & ((1u << (bit & 31)) - 1u);
          a.faces[(size_t)p * 3 + j] = (int32_t)(s_vbase[o] + a.epre[wi] + (uint32_t)__popc(below));
        }
      }
      pos += (uint32_t)__popcll(m);
    });
    // the block's own vertices: lane l < 48 walks the set bits of word l
    if (lane < kEdgeWords) {
      uint32_t w = a.ebits[(size_t)b * kEdgeWords + lane];
      uint32_t id = s_vbase[0] + a.epre[(size_t)b * kEdgeWords + lane];
      while (w) {
        const int bit = lane * 32 + __builtin_ctz(w);
        w &= w - 1u;
        const int axis = bit / kB3, vi = bit % kB3;
        const int lx = vi >> 6, ly = (vi >> 3) & 7, lz = vi & 7;
        const int ux = lx + (axis == 0), uy = ly + (axis == 1), uz = lz + (axis == 2);
        const int i0 = lx * 81 + ly * 9 + lz, i1 = ux * 81 + uy * 9 + uz;
        float px, py, pz;
        uint32_t c = 0u;
        const int g = axis == 0 ? gx0 + lx : (axis == 1 ? gy0 + ly : gz0 + lz);
        mc_interp<kColor>(S, s_col, i0, i1, (uint32_t)axis, g, false, (float)(gx0 + lx), (float)(gy0 + ly),
                          (float)(gz0 + lz), px, py, pz, c);
        if (id < a.vertex_cap) {
          float* q = a.vertices + (size_t)id * 3;
          q[0] = px * a.vox;
          q[1] = py * a.vox;
          q[2] = pz * a.vox;
          if (kColor) {
            uint8_t* q8 = a.vrgb + (size_t)id * 3;
            q8[0] = (uint8_t)c;
            q8[1] = (uint8_t)(c >> 8);
            q8[2] = (uint8_t)(c >> 16);
          }
        }
        ++id;
      }
    }
  }
}

// ============================================================================ streaming
// Out-of-core streaming (the reference's streamOutGPU2CPU / streamInCPU2GPU, src/tsdf.cu:
// 277-596, re-designed: whole 8^3 blocks move, not 5^3-block chunks, the pool stays dense,
// and the kernels read and write the pinned host store directly, so each block crosses the
// link once with no staging copy). One wave per block in the copy kernels, 64 lanes
// striding over its words.

__device__ __forceinline__ uint32_t* slab_words(const StreamArgs& a, uint32_t slot) {
  return a.slab_words[slot >> kSlabShift] + (size_t)(slot & (kSlabBlocks - 1u)) * a.wpb;
}
__device__ __forceinline__ uint32_t* slab_cols(const StreamArgs& a, uint32_t slot) {
  return a.slab_cols[slot >> kSlabShift] + (size_t)(slot & (kSlabBlocks - 1u)) * kB3;
}

__global__ __launch_bounds__(256) void k_st_out(StreamArgs a) {
  const int lane = threadIdx.x & 63;
  for (uint32_t i = blockIdx.x * 4u + (threadIdx.x >> 6); i < a.n; i += gridDim.x * 4u) {
    const size_t b = a.src[i];
    uint32_t* w = slab_words(a, a.slots[i]);
    for (uint32_t k = lane; k < a.wpb; k += 64) w[k] = a.pool[b * a.wpb + k];
    if (a.colors) {
      uint32_t* c = slab_cols(a, a.slots[i]);
      for (uint32_t k = lane; k < kB3; k += 64) c[k] = a.colors[b * kB3 + k];
    }
  }
}

__global__ __launch_bounds__(256) void k_st_move(StreamArgs a) {
  const int lane = threadIdx.x & 63;
  for (uint32_t i = blockIdx.x * 4u + (threadIdx.x >> 6); i < a.n; i += gridDim.x * 4u) {
    const size_t s = a.src[i], d = a.dst[i];
    for (uint32_t k = lane; k < a.wpb; k += 64) a.pool[d * a.wpb + k] = a.pool[s * a.wpb + k];
    if (a.colors)
      for (uint32_t k = lane; k < kB3; k += 64) a.colors[d * kB3 + k] = a.colors[s * kB3 + k];
    if (lane == 0) a.block_keys[d] = a.block_keys[s];
  }
}

__global__ __launch_bounds__(256) void k_st_rehash(StreamArgs a) {
  const uint32_t b = blockIdx.x * 256u + threadIdx.x;
  if (b >= a.n) return;
  bool inserted = false;
  const int64_t slot = find_or_insert(a.hash, a.block_keys[b], inserted);
  if (slot < 0) {
    raise_flag(a.ctl, kFlagHashFull);
  } else {
    a.hash.vals[slot] = (unsigned long long)b | ((unsigned long long)a.birth << 32);
    a.block_info[b] = (unsigned long long)slot | ((unsigned long long)a.birth << 32);
  }
}

// One lane per staged block: find or insert its key; new keys take pool blocks (one counter
// atomic per wave), resident keys are marked for merging.
__global__ __launch_bounds__(256) void k_st_insert(StreamArgs a) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool act = i < a.n;
  bool inserted = false;
  int64_t slot = -1;
  if (act) {
    slot = find_or_insert(a.hash, a.keys[i], inserted);
    if (slot < 0) raise_flag(a.ctl, kFlagHashFull);
  }
  const uint64_t im = __ballot(inserted);
  const int leader = im ? first_lane(im) : 0;
  uint32_t pbase = 0;
  if (im && lane == leader) pbase = atomicAdd(&a.ctl->pool_count, (uint32_t)__popcll(im));
  if (im) pbase = read_lane_u32(pbase, leader);
  if (!act) return;
  uint32_t placed = kNoBlock;
  if (inserted) {
    const uint32_t idx = pbase + lanes_below(im);
    uint32_t stored = kNoBlock;
    if (idx < a.pool_cap) {
      a.block_keys[idx] = a.keys[i];
      a.block_info[idx] = (unsigned long long)slot | ((unsigned long long)a.birth << 32);
      stored = placed = idx;
    } else {
      raise_flag(a.ctl, kFlagPoolFull);
    }
    a.hash.vals[slot] = (unsigned long long)stored | ((unsigned long long)a.birth << 32);
  } else if (slot >= 0) {
    const uint32_t v = (uint32_t)a.hash.vals[slot];
    if (v < a.pool_cap) placed = v | kMergeBit;
  }
  a.placed[i] = placed;
}

// Host-store blocks into the pool: copied, or merged voxel by voxel into a resident block
// of the same key (the observation histories combine): weights add (capped), the TSDF value
// is the weighted mean (s_r w_r + s_s w_s) / (w_r + w_s), colours per channel
// (c_r w_r + c_s w_s) / (w_r + w_s) truncated to 8 bits; a side with weight 0 contributes
// nothing (the other side is kept bit for bit).
template <int kStorage>
__global__ __launch_bounds__(256) void k_st_place(StreamArgs a) {
  using IO = VoxelIO<kStorage>;
  using Word = typename IO::Word;
  const int lane = threadIdx.x & 63;
  for (uint32_t i = blockIdx.x * 4u + (threadIdx.x >> 6); i < a.n; i += gridDim.x * 4u) {
    const uint32_t p = a.placed[i];
    if (p == kNoBlock) continue;
    const size_t d = p & ~kMergeBit;
    const uint32_t* hw = slab_words(a, a.slots[i]);
    const uint32_t* hc = a.colors ? slab_cols(a, a.slots[i]) : nullptr;
    if (!(p & kMergeBit)) {
      for (uint32_t k = lane; k < a.wpb; k += 64) a.pool[d * a.wpb + k] = hw[k];
      if (a.colors)
        for (uint32_t k = lane; k < kB3; k += 64) a.colors[d * kB3 + k] = hc[k];
      continue;
    }
    Word* rw = reinterpret_cast<Word*>(a.pool) + d * kB3;
    const Word* sw = reinterpret_cast<const Word*>(hw);
    for (uint32_t k = lane; k < kB3; k += 64) {
      float sr, wr, ss, ws;
      const Word r = rw[k], q = sw[k];
      IO::unpack(r, sr, wr);
      IO::unpack(q, ss, ws);
      if (!(ws > 0.0f)) continue;
      uint32_t* col = a.colors ? a.colors + d * kB3 + k : nullptr;
      const uint32_t cs = a.colors ? hc[k] : 0u;
      if (!(wr > 0.0f)) {
        rw[k] = q;
        if (col) *col = cs;
        continue;
      }
      const float wsum = wr + ws;
      const float pr = sr * wr, ps = ss * ws;
      const float sv = div_rn(pr + ps, wsum);
      const float wv = (a.cap > 0.0f && wsum > a.cap) ? a.cap : wsum;
      rw[k] = IO::pack(sv, wv);
      if (col) {
        const uint32_t cr = *col;
        uint32_t out = 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float xr = (float)((cr >> (8 * c)) & 255u) * wr, xs = (float)((cs >> (8 * c)) & 255u) * ws;
          out |= (uint32_t)(uint8_t)div_rn(xr + xs, wsum) << (8 * c);
        }
        *col = out;
      }
    }
  }
}

// ============================================================================ queries
// a / b from y = RN(1 / b): q0 = RN(a y) is within 1.5 ulp, and RN(q0 + (a - q0 b) y), Markstein's
// correction, takes 3 operations instead of the division's 11. Correctly rounded where b has 24
// significant bits, as the voxel size has: a - q0 b then has 25 and is exact under FMA, the corrected sum is
// off by 1.5 ulp 2^-53 at most, and a / b is no midpoint of two doubles nor within 2^-25 ulp of one. For a divisor of 53 bits (gn_step's
// pivots) a - q0 b may round, and only a quotient within some 2^-50 ulp of a midpoint can come out as its neighbour. No
// subnormal quotients.
__device__ __forceinline__ double quotient(double a, double b, double y) {
  const double q0 = a * y;
  return __builtin_fma(__builtin_fma(-q0, b, a), y, q0);
}

// The four keys of a bucket, as one pair of 16-byte loads.
struct BucketKeys {
  ulonglong2 k01, k23;
};
__device__ __forceinline__ BucketKeys load_bucket(const HashView& h, uint64_t b) {
  const ulonglong2* bp = reinterpret_cast<const ulonglong2*>(h.keys + b * kSlotsPerBucket);
  return {bp[0], bp[1]};
}
constexpr int kAbsent = -1, kElsewhere = -2;
// Slot of the key in its home bucket; kAbsent when an empty slot ends the search there,
// kElsewhere when the bucket is full of other keys (the search goes on in the next).
__device__ __forceinline__ int match_bucket(const BucketKeys& k, uint64_t key) {
  const uint64_t ks[4] = {k.k01.x, k.k01.y, k.k23.x, k.k23.y};
  int slot = kElsewhere;
#pragma unroll
  for (int s = 3; s >= 0; --s) {
    slot = ks[s] == kEmptyKey ? kAbsent : slot;
    slot = ks[s] == key ? s : slot;
  }
  return slot;
}

// Trilinear sample of the normalised TSDF at world point q; false unless all 8 lattice
// corners are allocated and observed. The lattice position q/vox and its cell fraction are
// formed in FP64 (an FP32 q/vox at |q| ~ 3 m is off by ~2e-5 of a voxel), the blend runs in
// FP32. vid/w receive the pool voxel ids and weights; g the gradient w.r.t. q.
//
// What bounds it: dependent memory round trips, and the L1's one cache line a cycle. The cell's
// corners lie in one block, or in 2, 4 or 8 where it crosses block faces (a third of all cells, some
// lane of nearly every wave). The lookups are made together in two stages, the cell's own block and
// its neighbours across one face, then those across edges and the corner, each stage loading every
// bucket before the first is looked at: with the voxels five round trips, where one lookup after
// another took up to 18. The 8 corners come as 4 pairs. Solver evaluation of 300,000 points (FP32): 30.6
// us with 8 voxel loads, 26.6 with pairs.
template <int kStorage>
__device__ __forceinline__ bool sample_sdf(const QueryArgs& q, double px, double py, double pz,
                                           float& sdf, float g[3], uint32_t vid[8], float w[8]) {
  using IO = VoxelIO<kStorage>;
  using Word = typename IO::Word;
  const double vox = (double)q.vox;
  const double gxd = quotient(px, vox, q.inv_vox), gyd = quotient(py, vox, q.inv_vox), gzd = quotient(pz, vox, q.inv_vox);
  if (!(fabs(gxd) < 8.0e6 && fabs(gyd) < 8.0e6 && fabs(gzd) < 8.0e6)) return false;
  const double flx = floor(gxd), fly = floor(gyd), flz = floor(gzd);
  const int ix = (int)flx, iy = (int)fly, iz = (int)flz;
  const float fx = (float)(gxd - flx), fy = (float)(gyd - fly), fz = (float)(gzd - flz);
  const Word* voxw = reinterpret_cast<const Word*>(q.voxels);
  // blocks by the faces crossed to reach them: bit 2 x, bit 1 y, bit 0 z
  const int cross = (((ix & 7) == 7) << 2) | (((iy & 7) == 7) << 1) | ((iz & 7) == 7);
  const uint64_t key0 = pack_key(ix >> 3, iy >> 3, iz >> 3);
  const auto key_of = [&](int c) {
    return key0 + ((uint64_t)((c >> 2) & 1) << (2 * kKeyBits)) + ((uint64_t)((c >> 1) & 1) << kKeyBits) + (uint64_t)(c & 1);
  };
  const auto needs = [&](int c) { return (cross & c) == c; };
  uint32_t blk[8];
  int elsewhere = 0;
  constexpr int kStage[2][4] = {{0, 1, 2, 4}, {3, 5, 6, 7}};
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    BucketKeys bk[4];
    uint64_t home[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = kStage[st][i];
      blk[c] = kNoBlock;
      if (needs(c)) {
        home[i] = bucket_of(key_of(c), q.hash.log2_buckets);
        bk[i] = load_bucket(q.hash, home[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = kStage[st][i];
      if (needs(c)) {
        const int slot = match_bucket(bk[i], key_of(c));
        if (slot >= 0) blk[c] = (uint32_t)q.hash.vals[home[i] * kSlotsPerBucket + slot];
        elsewhere |= slot == kElsewhere ? 1 << c : 0;
      }
    }
  }
  while (elsewhere) {  // a home bucket full of other keys: the whole search
    const int c = __ffs(elsewhere) - 1;
    elsewhere &= elsewhere - 1;
    const uint32_t found = find_block(q.hash, key_of(c));
#pragma unroll
    for (int k = 0; k < 8; ++k) blk[k] = k == c ? found : blk[k];
  }
  // a corner across no further face lies in the block without it
  if (!(cross & 1)) { blk[1] = blk[0]; blk[3] = blk[2]; blk[5] = blk[4]; blk[7] = blk[6]; }
  if (!(cross & 2)) { blk[2] = blk[0]; blk[3] = blk[1]; blk[6] = blk[4]; blk[7] = blk[5]; }
  if (!(cross & 4)) { blk[4] = blk[0]; blk[5] = blk[1]; blk[6] = blk[2]; blk[7] = blk[3]; }
  bool seen = true;
#pragma unroll
  for (int k = 0; k < 8; ++k) seen = seen & (blk[k] < q.pool_cap);
  if (!seen) return false;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int cx = ix + (k >> 2), cy = iy + ((k >> 1) & 1), cz = iz + (k & 1);
    vid[k] = blk[k] * kB3 + (uint32_t)((((cx & 7) * 8) + (cy & 7)) * 8 + (cz & 7));
  }
  // z neighbours in one load (z is the fastest index of a block); where the cell crosses a z
  // face the pair is the last of its row, and the neighbour's first voxel a load of its own
  struct __attribute__((packed, aligned(sizeof(Word)))) Pair {
    Word a, b;
  };
  const bool cross_z = (cross & 1) != 0;
  Pair pair[4];
  Word next[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    pair[k] = *reinterpret_cast<const Pair*>(voxw + (vid[2 * k] - (cross_z ? 1u : 0u)));
    next[k] = IO::zero();
  }
  if (cross_z) {
#pragma unroll
    for (int k = 0; k < 4; ++k) next[k] = voxw[vid[2 * k + 1]];
  }
  float s[8];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float sa, wa, sb, wb, sn, wn;
    IO::unpack(pair[k].a, sa, wa);
    IO::unpack(pair[k].b, sb, wb);
    IO::unpack(next[k], sn, wn);
    s[2 * k] = cross_z ? sb : sa;
    s[2 * k + 1] = cross_z ? sn : sb;
    seen = seen & ((cross_z ? wb : wa) > 0.0f) & ((cross_z ? wn : wb) > 0.0f);
  }
  if (!seen) return false;
  trilinear_weights(fx, fy, fz, w);
  float acc = 0.0f;
#pragma unroll
  for (int k = 0; k < 8; ++k) acc = acc + w[k] * s[k];
  sdf = acc;
  trilinear_dfrac(fx, fy, fz, s, g);
  g[0] = g[0] / q.vox;
  g[1] = g[1] / q.vox;
  g[2] = g[2] / q.vox;
  return true;
}

template <int kStorage>
__global__ __launch_bounds__(256) void k_query(QueryArgs q, const float* pts, int64_t n, float* sdf,
                                               uint8_t* valid) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    float r = 0.0f, g[3], w[8];
    uint32_t vid[8];
    const bool ok = sample_sdf<kStorage>(q, (double)pts[3 * i], (double)pts[3 * i + 1], (double)pts[3 * i + 2], r,
                                         g, vid, w);
    if (sdf) sdf[i] = ok ? r : 0.0f;
    if (valid) valid[i] = ok ? 1 : 0;
  }
}

// q = R p + t in FP64 from a row-major 3x4 pose (float or double entries).
template <class P>
__device__ __forceinline__ void pose_apply_d(const P* T, float x, float y, float z, double& qx, double& qy, double& qz) {
  const double X = x, Y = y, Z = z;
  qx = ((X * (double)T[0] + Y * (double)T[1]) + Z * (double)T[2]) + (double)T[3];
  qy = ((X * (double)T[4] + Y * (double)T[5]) + Z * (double)T[6]) + (double)T[7];
  qz = ((X * (double)T[8] + Y * (double)T[9]) + Z * (double)T[10]) + (double)T[11];
}

__device__ __forceinline__ double shfl_xor_d(double v, int m) {
  const long long b = __double_as_longlong(v);
  const int lo = __shfl_xor((int)(b & 0xffffffffll), m);
  const int hi = __shfl_xor((int)(b >> 32), m);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ double shfl_d(double v, int src) {
  const long long b = __double_as_longlong(v);
  const int lo = __shfl((int)(b & 0xffffffffll), src);
  const int hi = __shfl((int)(b >> 32), src);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Sums acc[0..N) over the workgroup (256 lanes) into out[0..N); fixed tree, deterministic.
template <int N>
__device__ __forceinline__ void wg_reduce_store(double (&acc)[N], double* out) {
  __shared__ double s_part[4][N];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    double v = acc[k];
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += shfl_xor_d(v, m);
    acc[k] = v;
  }
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) s_part[wave][k] = acc[k];
  }
  __syncthreads();
  if (threadIdx.x < N) {
    const int k = threadIdx.x;
    out[k] = ((s_part[0][k] + s_part[1][k]) + s_part[2][k]) + s_part[3][k];
  }
  __syncthreads();
}

// Sums acc[0..N) (N <= 32) over each four waves of the workgroup by recursive halving
// within each wave: at lane distance m = 32, 16, 8, 4, 2 every lane sends the half of its
// values its partner (lane ^ m) keeps and adds the partner's half of its own, so the values
// per lane halve each step (31 double exchanges instead of 6 per value); a last exchange at
// distance 1 completes the wave's sums, which wave_sums stores in s_part; sum_of_four then adds
// four waves' in order. Fixed tree, deterministic.
//
// The first two steps' exchanges are one instruction per word (v_permlane32_swap and
// v_permlane16_swap hand one half of a register for the other half of another), no LDS permute and no
// selects.
template <int kDistance>
__device__ __forceinline__ double exchange_add(double lower, double upper) {  // each lane's half, with its partner's part
  const long long a = __double_as_longlong(lower), b = __double_as_longlong(upper);
  const uint32_t w[2][2] = {{(uint32_t)a, (uint32_t)b}, {(uint32_t)(a >> 32), (uint32_t)(b >> 32)}};
  uint32_t x[2], y[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const auto r = kDistance == 32 ? __builtin_amdgcn_permlane32_swap(w[k][0], w[k][1], false, false)
                                   : __builtin_amdgcn_permlane16_swap(w[k][0], w[k][1], false, false);
    x[k] = r[0];
    y[k] = r[1];
  }
  return __longlong_as_double((long long)((uint64_t)x[1] << 32 | x[0])) + __longlong_as_double((long long)((uint64_t)y[1] << 32 | y[0]));
}
template <int N>
__device__ __forceinline__ void wave_sums(const double (&acc)[N], double (&s_part)[32]) {
  static_assert(N <= 32, "at most 32 values");
  const int lane = threadIdx.x & 63;
  double v[32];
#pragma unroll
  for (int k = 0; k < 32; ++k) v[k] = k < N ? acc[k] : 0.0;
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = exchange_add<32>(v[i], v[i + 16]);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = exchange_add<16>(v[i], v[i + 8]);
#pragma unroll
  for (int h = 4; h >= 1; h >>= 1) {  // h values per lane after this step; distance 2h
    const bool upper = (lane & (2 * h)) != 0;  // this lane keeps the upper half
#pragma unroll
    for (int i = 0; i < h; ++i) {
      const double send = upper ? v[i] : v[i + h];
      const double keep = upper ? v[i + h] : v[i];
      v[i] = keep + shfl_xor_d(send, 2 * h);
    }
  }
  const double total = v[0] + shfl_xor_d(v[0], 1);
  // value index of this lane: the halves it kept, from bit 5 (most significant) to bit 1
  const int idx = ((lane >> 5) & 1) * 16 + ((lane >> 4) & 1) * 8 + ((lane >> 3) & 1) * 4 + ((lane >> 2) & 1) * 2 +
                  ((lane >> 1) & 1);
  if ((lane & 1) == 0) s_part[idx] = total;
}
__device__ __forceinline__ double sum_of_four(const double (*s_part)[32], int k) {
  return ((s_part[0][k] + s_part[1][k]) + s_part[2][k]) + s_part[3][k];
}

// The chunk of a list that a workgroup takes, so that the workgroups of one XCD (dispatched round
// robin over 8) take neighbouring chunks and their blocks are fetched into one L2 instead of eight.
__device__ __forceinline__ uint32_t xcd_chunk(uint32_t wg, uint32_t grid) {
  const uint32_t xcd = wg & 7u, rest = grid & 7u;
  return xcd * (grid >> 3) + (xcd < rest ? xcd : rest) + (wg >> 3);
}

// Residuals r_i = sdf(R p_i + t) and their derivatives with respect to a left se(3)
// perturbation (rho, phi): dr/drho = grad, dr/dphi = q x grad. Workgroup chunk c takes the points
// [c per, (c + 1) per), per a multiple of 256.
//
// What bounds it: the voxel gradients' float atomics, which leave the XCD (a gradient row may be
// written from any of them) as one request per cache line and instruction. A lane's own eight corners,
// one instruction each, made 64 points' lines per instruction; the wave turns its 64 x 8
// additions over in LDS, so that an instruction holds all eight corners of 8 neighbouring points,
// which lie in two lines per point and mostly in their neighbours' too. 300,000 points of a frame
// (FP16): 123 us with a lane's corners and points dealt out grid-wide, 59 so (2.19e6 atomic
// requests, 9.8e5); adding up in an LDS hash set of the workgroup's lines first (7.8e5) took 65.
template <int kStorage>
__global__ __launch_bounds__(256) void k_backward(QueryArgs q, const float* pts, int64_t n, int64_t per, const float* T12,
                                                  const float* grad_r, float* r_out, uint8_t* valid, float* J,
                                                  double* partials, float* voxel_grad) {
  __shared__ float4 s_add[4][128];
  __shared__ uint4 s_vid[4][128];
  constexpr uint32_t kNoVoxel = 0xffffffffu;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t first = per * (int64_t)xcd_chunk(blockIdx.x, gridDim.x);
  const int64_t end = first + per < n ? first + per : n;
  double acc[6] = {0, 0, 0, 0, 0, 0};
  for (int64_t base = first + 64 * wave; base < end; base += 256) {  // base: the wave's first point
    const int64_t i = base + lane;
    uint32_t vid[8];
    float add[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) vid[k] = kNoVoxel, add[k] = 0.0f;
    if (i < end) {
      double qx, qy, qz;
      pose_apply_d(T12, pts[3 * i], pts[3 * i + 1], pts[3 * i + 2], qx, qy, qz);
      float r = 0.0f, g[3] = {0, 0, 0}, w[8];
      const bool ok = sample_sdf<kStorage>(q, qx, qy, qz, r, g, vid, w);
      float j[6] = {0, 0, 0, 0, 0, 0};
      if (ok) {
        const double gx = g[0], gy = g[1], gz = g[2];
        j[0] = g[0]; j[1] = g[1]; j[2] = g[2];
        j[3] = (float)(qy * gz - qz * gy);
        j[4] = (float)(qz * gx - qx * gz);
        j[5] = (float)(qx * gy - qy * gx);
      }
      if (r_out) r_out[i] = ok ? r : 0.0f;
      if (valid) valid[i] = ok ? 1 : 0;
      if (J) {
#pragma unroll
        for (int k = 0; k < 6; ++k) J[6 * i + k] = j[k];
      }
      const float up = grad_r ? grad_r[i] : 0.0f;
      if (ok) {
#pragma unroll
        for (int k = 0; k < 6; ++k) acc[k] += (double)up * (double)j[k];
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (ok) add[k] = up * w[k];
        else vid[k] = kNoVoxel;
      }
    }
    if (voxel_grad) {
      wave_sync();  // the previous round's reads are issued
      s_add[wave][2 * lane] = make_float4(add[0], add[1], add[2], add[3]);
      s_add[wave][2 * lane + 1] = make_float4(add[4], add[5], add[6], add[7]);
      s_vid[wave][2 * lane] = make_uint4(vid[0], vid[1], vid[2], vid[3]);
      s_vid[wave][2 * lane + 1] = make_uint4(vid[4], vid[5], vid[6], vid[7]);
      wave_sync();
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t v = reinterpret_cast<const uint32_t*>(s_vid[wave])[64 * k + lane];
        const float a = reinterpret_cast<const float*>(s_add[wave])[64 * k + lane];
        if (v != kNoVoxel) atomicAdd(voxel_grad + v, a);
      }
    }
  }
  if (partials) wg_reduce_store<6>(acc, partials + 6 * (size_t)blockIdx.x);
}

// Sums the workgroups' partials, one wave per accumulator: each lane every 64th in order, then a
// fixed tree (one lane per accumulator took 66 us over 512 partials).
__global__ __launch_bounds__(384) void k_reduce6(const double* partials, int grid, double* out6) {
  const int lane = threadIdx.x & 63, k = threadIdx.x >> 6;
  double s = 0.0;
#pragma unroll 8
  for (int g = lane; g < grid; g += 64) s += partials[6 * (size_t)g + k];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += shfl_xor_d(s, m);
  if (lane == 0) out6[k] = s;
}

// ============================================================================ tracking
__device__ __forceinline__ uint32_t track_slot(const TrackArgs& t) { return t.ctl->cursor[1] % t.n_seq; }

// A tracked frame's starting pose, into s_pose (lanes 0..11 of every workgroup): with increments,
// out[f-1] * prior[f] in FP64, each entry summed in column order ((a0 b0 + a1 b1) + a2 b2) +
// a3 b3. Workgroup 0 makes it the candidate and clears the solver state (the first evaluation, not a
// memset node, so the captured graph replays it exactly).
__device__ __forceinline__ void track_start(const TrackArgs& t, uint32_t fs, double* s_pose) {
  const int k = threadIdx.x;
  const bool w0 = blockIdx.x == 0;
  const float* P = t.prior + 16 * (size_t)fs;
  if (k < 12) {
    double p;
    if (t.increment && fs > 0) {
      const float* A = t.out + 16 * (size_t)(fs - 1);
      const int r = k >> 2, c = k & 3;
      p = (((double)A[4 * r] * (double)P[c] + (double)A[4 * r + 1] * (double)P[4 + c]) +
           (double)A[4 * r + 2] * (double)P[8 + c]) + (double)A[4 * r + 3] * (double)P[12 + c];
    } else {
      p = (double)P[k];
    }
    s_pose[k] = p;
    if (w0) {
      t.pose[k] = p;
      t.state->cand[k] = p;   // the first evaluation's pose
      t.state->start[k] = p;  // the motion prior's centre
    }
  }
  if (w0 && k == 0) {  // no accepted pose yet (the other fields are set by the first acceptance)
    t.state->has = 0;
    t.state->lambda = 1e-4;
    const double st = t.prior_sigma_t, sr = t.prior_sigma_r;
    t.state->lam_t = st > 0.0 ? 1.0 / (st * st) : 0.0;
    t.state->lam_r = sr > 0.0 ? 1.0 / (sr * sr) : 0.0;
    t.state->n_eff = t.n_eff;
  }
}

// Point i of a tracked frame: one stride-th pixel back-projected to the camera frame ((u - cx) d / fx,
// (v - cy) d / fy, d) in FP32 with this operation order; a pixel without a valid depth gives
// NaN (skipped by the solver). Stored for the frame's further evaluations.
__device__ __forceinline__ void track_point(const TrackArgs& t, uint32_t fs, int i, float& x, float& y, float& z) {
  const int u = (i % t.pw) * t.stride, v = (i / t.pw) * t.stride;
  const size_t first = (size_t)fs * t.W * t.H;
  const float d = t.depth_u16 ? depth_at<true>(reinterpret_cast<const uint16_t*>(t.depth) + first, t.depth_scale, v * t.W + u)
                              : depth_at<false>(reinterpret_cast<const float*>(t.depth) + first, t.depth_scale, v * t.W + u);
  x = y = z = __builtin_nanf("");
  if (depth_valid(d, t.max_depth)) {
    x = (((float)u - t.K.cx) * d) / t.K.fx;
    y = (((float)v - t.K.cy) * d) / t.K.fy;
    z = d;
  }
  t.pts[3 * i] = x;
  t.pts[3 * i + 1] = y;
  t.pts[3 * i + 2] = z;
}

// ============================================================================ Gauss-Newton
// Huber loss of a scaled residual e and its iteratively reweighted least-squares weight
// psi(e)/e (kHuber, vh_internal.h).
__device__ __forceinline__ double huber_rho(double e) {
  const double ae = fabs(e);
  return ae <= kHuber ? 0.5 * e * e : kHuber * (ae - 0.5 * kHuber);
}
__device__ __forceinline__ double huber_weight(double e) {
  const double ae = fabs(e);
  return ae <= kHuber ? 1.0 : kHuber / ae;
}

// Per point (camera frame p, depth z = p.z): s = mu / sigma(z); with a valid sample r at
// q = R p + t and e = s r, the point adds W J J^T and W r J with W = huber_weight(e) s^2 (one
// Gauss-Newton step of the iteratively reweighted problem), r^2, and rho(e) to the cost; a
// point without a valid sample adds rho(s), the cost of a saturated residual r = 1.
struct GnPoint {
  float x, y, z;  // camera frame
  float r, g[3];  // the sample at q
};
__device__ __forceinline__ GnPoint gn_load(const GnArgs& a, uint32_t fs, int64_t i) {
  GnPoint p{};
  if (a.track) {
    track_point(a.t, fs, (int)i, p.x, p.y, p.z);
  } else {
    p.x = a.pts[3 * i];
    p.y = a.pts[3 * i + 1];
    p.z = a.pts[3 * i + 2];
  }
  return p;
}
// A non-finite coordinate (no depth at this pixel) leaves the point out.
__device__ __forceinline__ bool gn_considered(const GnPoint& p) { return isfinite(p.x) && isfinite(p.y) && isfinite(p.z); }
template <int kStorage>
__device__ __forceinline__ bool gn_sample(const GnArgs& a, const double* pose, GnPoint& p) {
  double qx, qy, qz;
  pose_apply_d(pose, p.x, p.y, p.z, qx, qy, qz);
  float w[8];
  uint32_t vid[8];
  return sample_sdf<kStorage>(a.q, qx, qy, qz, p.r, p.g, vid, w);
}
// acc: kGnAcc sums; counts [28] and [29] are whole numbers and exact.
__device__ __forceinline__ void gn_add(const GnArgs& a, const double* pose, const GnPoint& p, bool ok, double (&acc)[kGnAcc]) {
  acc[29] += 1.0;
  const double zt = (double)p.z - 0.4;
  const double sc = (double)a.mu / (0.0012 + 0.0019 * (zt * zt));
  if (!ok) {
    acc[30] += huber_rho(sc);
    return;
  }
  double qx, qy, qz;
  pose_apply_d(pose, p.x, p.y, p.z, qx, qy, qz);
  const double rd = (double)p.r, e = sc * rd;
  const double W = huber_weight(e) * sc * sc;
  const double gx = p.g[0], gy = p.g[1], gz = p.g[2];
  const double j[6] = {gx, gy, gz, qy * gz - qz * gy, qz * gx - qx * gz, qx * gy - qy * gx};
  double wj[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) wj[c] = W * j[c];
  int m = 0;
#pragma unroll
  for (int r = 0; r < 6; ++r)
#pragma unroll
    for (int c = r; c < 6; ++c) acc[m++] += wj[r] * j[c];
#pragma unroll
  for (int c = 0; c < 6; ++c) acc[21 + c] += wj[c] * rd;
  acc[27] += rd * rd;
  acc[28] += 1.0;
  acc[30] += huber_rho(e);
}

// One evaluation. With a previous evaluation (prev_grid > 0) every workgroup first takes its
// Levenberg-Marquardt step itself (gn_solve_wg over the previous partials: the same sums in
// the same order, so every workgroup gets the same candidate; workgroup 0 stores the state,
// the candidate and the stats row), which saves a launch per evaluation and needs no ordering
// between workgroups; otherwise the candidate is a.start.pose.
//
// Partial sum b of the a.grid is over the points b 256 + t (t < 256), and every a.grid 256th
// after them, added in order per t. What bounds an evaluation is latency: of the step's serial FP64
// chain and of the points' lookups. Two launch shapes (launch_gn_accum):
// - k_gn_accum, while each point has a lane of its own: a workgroup of 256 per partial sum, one point
//   to a lane, loaded before the step; a fifth wave takes the motion prior's part of the step.
// - k_gn_accum_wide above: 16 waves, two partial sums a workgroup, a workgroup per CU. All waves
//   sample, 1,536 points at a time, into LDS, and 8 of them add those up in order; a sampling wave
//   doesn't hold the 31 FP64 sums (62 registers), so twice as many lookups are in flight
//   as with both in one loop.
// Workgroups take neighbouring points by XCD (xcd_chunk): 300,000 points made 0.70e6 read requests beyond
// the L2, now 0.29e6.
// Measured, per evaluation: 19,200 points (F16) 12.4 -> 8.9 us, 300,000 (FP32) 35.0 -> 23.3 us;
// 3.5 and 3.3 us of that by the step's shorter chain (gn_step) and the prior's own wave.
struct GnStepOut {
  GnState* st;
  double *cand, *row;
};
__device__ __forceinline__ GnStepOut gn_step_out(const GnArgs& a) {
  const bool w0 = blockIdx.x == 0;
  return {w0 ? a.st_out : nullptr, w0 ? a.cand_out : nullptr, w0 ? a.stats_row : nullptr};
}
template <int kThreads>
__device__ __forceinline__ void gn_solve_wg(const double* partials, int grid, const GnState* st_in, const GnStepOut& out,
                                            double* s_cand, int final_step);
// Start of a refinement: the first evaluation's pose comes with its launch, and workgroup 0 clears the solver
// state to it and the initial damping (all words of the state: 69).
__device__ __forceinline__ void gn_start(const GnArgs& a, double* s_pose) {
  constexpr int kWords = (int)(sizeof(GnState) / sizeof(double)), kCand = (int)(offsetof(GnState, cand) / sizeof(double)),
                kLambda = (int)(offsetof(GnState, lambda) / sizeof(double));
  const int t = threadIdx.x;
  if (t < 12) s_pose[t] = a.start.pose[t];
  if (blockIdx.x == 0 && t < kWords) {
    double v = t == kLambda ? a.start.lambda : 0.0;
    if (t >= kCand && t < kCand + 12) v = a.start.pose[t - kCand];
    reinterpret_cast<double*>(a.st_start)[t] = v;
  }
}
template <int kThreads>
__device__ __forceinline__ void gn_pose(const GnArgs& a, uint32_t fs, double* s_pose) {
  if (a.prev_grid > 0) {
    gn_solve_wg<kThreads>(a.prev_partials, a.prev_grid, a.st_in, gn_step_out(a), s_pose, 0);
    return;
  }
  if (a.track) track_start(a.t, fs, s_pose);
  else gn_start(a, s_pose);
  __syncthreads();
}

constexpr int kGnThreads = 320, kGnWideThreads = 1024;
template <int kStorage>
__global__ __launch_bounds__(kGnThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_gn_accum(GnArgs a) {
  __shared__ double s_pose[12];
  __shared__ double s_part[4][32];
  const int b = (int)xcd_chunk(blockIdx.x, gridDim.x), t = threadIdx.x;
  const uint32_t fs = a.track ? track_slot(a.t) : 0u;
  const int64_t i = b * (int64_t)256 + t;
  const bool mine = t < 256 && i < a.n;
  GnPoint p{};
  if (mine) p = gn_load(a, fs, i);
  gn_pose<kGnThreads>(a, fs, s_pose);
  if (t < 256) {
    double acc[kGnAcc];
#pragma unroll
    for (int k = 0; k < kGnAcc; ++k) acc[k] = 0.0;
    if (mine && gn_considered(p)) {
      const bool ok = gn_sample<kStorage>(a, s_pose, p);
      gn_add(a, s_pose, p, ok, acc);
    }
    wave_sums<kGnAcc>(acc, s_part[t >> 6]);
  }
  __syncthreads();
  if (t < kGnAcc) a.partials[kGnAcc * (size_t)b + t] = sum_of_four(s_part, t);
}

template <int kStorage>
__global__ __launch_bounds__(kGnWideThreads) void k_gn_accum_wide(GnArgs a) {
  constexpr int kRounds = 3;  // points of a lane (of the 512 that add) sampled before they are added
  enum : uint32_t { kSkip, kMiss, kHit };
  __shared__ double s_pose[12];
  __shared__ double s_part[8][32];
  __shared__ float4 s_smp[kRounds * 512];  // r, g
  __shared__ float4 s_pt[kRounds * 512];   // the point, and whether it was sampled
  const int c = (int)xcd_chunk(blockIdx.x, gridDim.x), t = threadIdx.x;
  const uint32_t fs = a.track ? track_slot(a.t) : 0u;
  gn_pose<kGnWideThreads>(a, fs, s_pose);
  // the sums between two turns: in memory by intent, or they'd take registers while sampling
  volatile double held[kGnAcc];
  const int64_t stride = a.grid * (int64_t)256;  // a.grid is even
  for (int64_t first = c * (int64_t)512, turn = 0; turn == 0 || first < a.n; first += kRounds * stride, ++turn) {
    for (int k = t; k < kRounds * 512; k += kGnWideThreads) {
      const int64_t i = first + (k >> 9) * stride + (k & 511);
      if (i >= a.n) break;
      GnPoint p = gn_load(a, fs, i);
      uint32_t hit = kSkip;
      if (gn_considered(p)) hit = gn_sample<kStorage>(a, s_pose, p) ? kHit : kMiss;
      s_smp[k] = make_float4(p.r, p.g[0], p.g[1], p.g[2]);
      s_pt[k] = make_float4(p.x, p.y, p.z, __uint_as_float(hit));
    }
    __syncthreads();
    if (t < 512) {
      double acc[kGnAcc];
#pragma unroll
      for (int k = 0; k < kGnAcc; ++k) acc[k] = 0.0;
      if (turn > 0) {
#pragma unroll
        for (int k = 0; k < kGnAcc; ++k) acc[k] = held[k];
      }
      for (int r = 0; r < kRounds; ++r) {
        const int64_t i = first + r * stride + t;
        if (i >= a.n) break;
        const float4 m = s_pt[512 * r + t], s = s_smp[512 * r + t];
        if (__float_as_uint(m.w) == kSkip) continue;
        gn_add(a, s_pose, GnPoint{m.x, m.y, m.z, s.x, {s.y, s.z, s.w}}, __float_as_uint(m.w) == kHit, acc);
      }
      if (first + kRounds * stride >= a.n) {
        wave_sums<kGnAcc>(acc, s_part[t >> 6]);
      } else {
#pragma unroll
        for (int k = 0; k < kGnAcc; ++k) held[k] = acc[k];
      }
    }
    __syncthreads();  // the next points overwrite the samples
  }
  if (t < 512 && (t & 255) < kGnAcc)
    a.partials[kGnAcc * (size_t)(2 * c + (t >> 8)) + (t & 255)] = sum_of_four(s_part + 4 * (t >> 8), t & 255);
}

// One workgroup, FP64: deterministic sum of the partials at the candidate pose, then a
// Levenberg-Marquardt decision and step.
//   cost(candidate) = the robust cost of k_gn_accum (every point with finite coordinates
//   counts, an invalid one as a saturated residual), so costs at different poses compare;
//   skipped points count neither way. A tracked frame scales that term (and its A, b) by
//   n_eff / (points considered) and adds its motion prior (motion_prior). The candidate is
//   accepted if its cost does not exceed
//   the accepted one (lambda /= 3) and rejected otherwise (lambda *= 4). Unless `final`, the
//   next candidate is exp(delta^) T_acc with (A + lambda diag(A)) delta = -b, A = J^T W J and
//   b = J^T W r at the accepted pose, delta = (rho, phi), T <- exp(delta^) T.
//   stats_row: [n_valid, rms, |delta|, lambda, accepted, accepted pose (12)].
// Entry k (< 12, row-major 3x4) of exp((rho, phi)^) pose, x = (rho, phi): one lane per entry.
__device__ __forceinline__ double se3_left_update(const double* x, const double* pose, int k) {
  const double rho[3] = {x[0], x[1], x[2]}, ph[3] = {x[3], x[4], x[5]};
  const double th2 = ph[0] * ph[0] + ph[1] * ph[1] + ph[2] * ph[2];
  const double th = sqrt(th2);
  double A1, B1, C1;  // sin/th, (1-cos)/th^2, (th - sin)/th^3
  if (th < 1e-5) {
    A1 = 1.0 - th2 / 6.0;
    B1 = 0.5 - th2 / 24.0;
    C1 = 1.0 / 6.0 - th2 / 120.0;
  } else {
    double sn, cs;
    sincos(th, &sn, &cs);
    A1 = sn / th;
    B1 = (1.0 - cs) / th2;
    C1 = (th - sn) / (th2 * th);
  }
  const double K[3][3] = {{0.0, -ph[2], ph[1]}, {ph[2], 0.0, -ph[0]}, {-ph[1], ph[0], 0.0}};
  const int p = k >> 2, c = k & 3;
  double Kp[3];  // row p
#pragma unroll
  for (int q = 0; q < 3; ++q) Kp[q] = p == 0 ? K[0][q] : p == 1 ? K[1][q] : K[2][q];
  double R[3], V[3];  // row p of both
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    double k2 = 0.0;
#pragma unroll
    for (int m = 0; m < 3; ++m) k2 += Kp[m] * K[m][q];
    const double I = p == q ? 1.0 : 0.0;
    R[q] = I + A1 * Kp[q] + B1 * k2;
    V[q] = I + B1 * Kp[q] + C1 * k2;
  }
  const double turned = R[0] * pose[c] + R[1] * pose[4 + c] + R[2] * pose[8 + c];
  return c < 3 ? turned : turned + (V[0] * rho[0] + V[1] * rho[1] + V[2] * rho[2]);
}

// Motion prior of a tracked frame at pose T (row-major 3x4): xi = log(S^-1 T) with S the
// frame's starting pose, translation first; the angle from atan2(|w|/2, (tr - 1)/2) (no loss of
// precision near zero), phi = theta / (2 sin theta) w, rho = V(phi)^-1 D_t with
// V^-1 = I - K/2 + (1/theta^2 - (1 + cos theta) / (2 theta sin theta)) K^2 (series below 1e-5).
// Its Jacobian for T <- exp(delta^) T is taken as M = Ad(T^-1) (the exact one is
// Jr^-1(xi) M; xi is a few noise standard deviations), so with Lam = diag(lam_t I3, lam_r I3) it
// adds M^T Lam M to J^T W J, M^T Lam xi to J^T W r and xi^T Lam xi / 2 to the cost.
__device__ __forceinline__ void motion_prior(const GnState& S, double* Ab, double& cost) {
  const double* P = S.start;
  const double* T = S.cand;
  double D[3][3], dt[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int j = 0; j < 3; ++j) D[i][j] = P[i] * T[j] + P[4 + i] * T[4 + j] + P[8 + i] * T[8 + j];
    dt[i] = P[i] * (T[3] - P[3]) + P[4 + i] * (T[7] - P[7]) + P[8 + i] * (T[11] - P[11]);
  }
  const double wv[3] = {D[2][1] - D[1][2], D[0][2] - D[2][0], D[1][0] - D[0][1]};
  const double sn = 0.5 * sqrt(wv[0] * wv[0] + wv[1] * wv[1] + wv[2] * wv[2]);
  const double cs = 0.5 * (D[0][0] + D[1][1] + D[2][2] - 1.0);
  const double th = atan2(sn, cs);
  double f, c2;
  if (th < 1e-5) {
    f = 0.5 + th * th / 12.0;
    c2 = 1.0 / 12.0 + th * th / 720.0;
  } else {
    f = th / (2.0 * sn);
    c2 = 1.0 / (th * th) - (1.0 + cs) / (2.0 * th * sn);
  }
  const double ph[3] = {f * wv[0], f * wv[1], f * wv[2]};
  const double K[3][3] = {{0.0, -ph[2], ph[1]}, {ph[2], 0.0, -ph[0]}, {-ph[1], ph[0], 0.0}};
  double xi[6];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    double a = dt[i] - 0.5 * (K[i][0] * dt[0] + K[i][1] * dt[1] + K[i][2] * dt[2]);
#pragma unroll
    for (int k = 0; k < 3; ++k) a += c2 * (K[i][0] * K[0][k] + K[i][1] * K[1][k] + K[i][2] * K[2][k]) * dt[k];
    xi[i] = a;
    xi[3 + i] = ph[i];
  }
  // With M = Ad(T^-1) = [[R^T, [p]x R^T], [0, R^T]], p = -R^T t, and R R^T = I:
  // M^T Lam M = [[lt I, -lt [t]x], [lt [t]x, lt (|t|^2 I - t t^T) + lr I]] and
  // M^T Lam xi = (g, t x g + lr R xi_phi) with g = lt R xi_rho.
  const double lt = S.lam_t, lr = S.lam_r;
  const double tv[3] = {T[3], T[7], T[11]};
  const double tt = tv[0] * tv[0] + tv[1] * tv[1] + tv[2] * tv[2];
  const double Kt[3][3] = {{0.0, -tv[2], tv[1]}, {tv[2], 0.0, -tv[0]}, {-tv[1], tv[0], 0.0}};
  cost += 0.5 * (lt * (xi[0] * xi[0] + xi[1] * xi[1] + xi[2] * xi[2]) +
                 lr * (xi[3] * xi[3] + xi[4] * xi[4] + xi[5] * xi[5]));
#pragma unroll
  for (int a = 0, m = 0; a < 6; ++a)
#pragma unroll
    for (int b = a; b < 6; ++b, ++m) {
      double v;
      if (a < 3 && b < 3) v = a == b ? lt : 0.0;
      else if (a < 3) v = -lt * Kt[a][b - 3];
      else v = lt * ((a == b ? tt : 0.0) - tv[a - 3] * tv[b - 3]) + (a == b ? lr : 0.0);
      Ab[m] += v;
    }
  double g[3], gr[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    g[i] = lt * (T[4 * i] * xi[0] + T[4 * i + 1] * xi[1] + T[4 * i + 2] * xi[2]);
    gr[i] = lr * (T[4 * i] * xi[3] + T[4 * i + 1] * xi[4] + T[4 * i + 2] * xi[5]);
  }
  Ab[21] += g[0];
  Ab[22] += g[1];
  Ab[23] += g[2];
  Ab[24] += (tv[1] * g[2] - tv[2] * g[1]) + gr[0];
  Ab[25] += (tv[2] * g[0] - tv[0] * g[2]) + gr[1];
  Ab[26] += (tv[0] * g[1] - tv[1] * g[0]) + gr[2];
}

struct GnPrior {
  double Ab[27], cost;  // what the motion prior adds to A, b and the cost
};

// The Levenberg-Marquardt decision and step of one evaluation by one wave, on the solver state
// staged in LDS (updated in place; the workgroup writes it out afterwards). One lane's serial chain
// set its time (of an evaluation of 19,200 points, 4.3 us of 9.6), at an instruction every few cycles: so what is per entry (the matrix and
// pose kept, the update of the pose, the outputs) goes one lane per entry, the rest is computed by all
// lanes alike, and the triangular solves divide by a pivot through its reciprocal, taken once (quotient).
__device__ __forceinline__ void gn_step(const double* tot, const GnPrior& prior, GnState& S, double* s_cand,
                                        const GnStepOut& out, int final_step) {
  const int lane = threadIdx.x & 63;
  const double cnt = tot[28];
  // tracking: depth term scaled to n_eff points, plus the motion prior
  const double al = S.n_eff > 0.0 && tot[29] > 0.0 ? S.n_eff / tot[29] : 1.0;
  const double cost = al * tot[30] + prior.cost;
  const bool had = S.has != 0;
  const bool accept = !had || cost <= S.cost;
  const double lambda = !accept ? fmin(S.lambda * 4.0, 1e9) : had ? fmax(S.lambda / 3.0, 1e-9) : S.lambda;
  wave_sync();  // every lane has the state it decides on
  if (accept) {
    if (lane < 12) S.pose[lane] = S.cand[lane];  // the pose this evaluation was made at
    if (lane < 27) S.Ab[lane] = al * tot[lane] + prior.Ab[lane];
    if (lane == 0) {
      S.cost = cost;
      S.has = 1;
    }
  }
  if (lane == 0) S.lambda = lambda;
  wave_sync();
  // damped normal equations, Cholesky (in the lower triangle of A, with the forward
  // substitution), back substitution (all loops unrolled: the matrix stays in registers); a
  // matrix that is not positive definite proposes the accepted pose again
  double A[6][6], inv[6], x[6], y[6];
#pragma unroll
  for (int p = 0, m = 0; p < 6; ++p)
#pragma unroll
    for (int q = p; q < 6; ++q, ++m) A[q][p] = S.Ab[m];
#pragma unroll
  for (int p = 0; p < 6; ++p) A[p][p] += lambda * A[p][p] + 1e-12;
  bool pd = true;
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    double d = A[q][q];
#pragma unroll
    for (int k = 0; k < q; ++k) d -= A[q][k] * A[q][k];
    pd = pd && d > 0.0;
    A[q][q] = sqrt(d);
    inv[q] = 1.0 / A[q][q];
#pragma unroll
    for (int p = q + 1; p < 6; ++p) {
      double a = A[p][q];
#pragma unroll
      for (int k = 0; k < q; ++k) a -= A[p][k] * A[q][k];
      A[p][q] = quotient(a, A[q][q], inv[q]);
    }
    double a = -S.Ab[21 + q];
#pragma unroll
    for (int k = 0; k < q; ++k) a -= A[q][k] * y[k];
    y[q] = quotient(a, A[q][q], inv[q]);
  }
#pragma unroll
  for (int p = 5; p >= 0; --p) {
    double a = y[p];
#pragma unroll
    for (int k = p + 1; k < 6; ++k) a -= A[k][p] * x[k];
    x[p] = quotient(a, A[p][p], inv[p]);
  }
  const bool step = !final_step && pd;
  if (lane < 12) {
    const double c = step ? se3_left_update(x, S.pose, lane) : S.pose[lane];
    s_cand[lane] = c;
    if (out.cand) out.cand[lane] = c;
  }
  if (out.row && lane < kGnStats) {
    const double sq = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3] + x[4] * x[4] + x[5] * x[5];
    const double root = sqrt(lane == 1 ? tot[27] / cnt : sq);
    const double head = lane == 0 ? cnt : lane == 1 ? (cnt > 0.0 ? root : 0.0) : lane == 2 ? (step ? root : 0.0)
                        : lane == 3 ? lambda : accept ? 1.0 : 0.0;
    out.row[lane] = lane < 5 ? head : S.pose[lane < 5 ? 0 : lane - 5];
  }
  wave_sync();  // the accepted pose is read
  if (lane < 12) S.cand[lane] = s_cand[lane];
}

// All kThreads lanes call it. Accumulator v's sum over the partials g = j, j + 8, ... in order is a
// term (v, j), v < kGnAcc, j < 8; then one lane per v adds its 8 terms in a fixed tree, so every
// workgroup gets the same sums in the same order. kThreads = 320: a lane per term, 16 loads in
// flight; 1,024: four lanes (16 apart) per term, each with a quarter of its partials in flight
// at once, their sums continued from quarter to quarter. Lanes below the state's size stage the
// solver state in LDS, the last wave computes the motion prior's terms, which need only the
// candidate, and the first wave takes the step (gn_step). The new candidate is in s_cand on return;
// out's pointers (global, each may be null) receive the new state, the candidate and the evaluation's row.
template <int kThreads>
__device__ __forceinline__ void gn_solve_wg(const double* partials, int grid, const GnState* st_in, const GnStepOut& out,
                                            double* s_cand, int final_step) {
  constexpr int kWays = 8, kTerms = kWays * kGnAcc, kStateWords = (int)(sizeof(GnState) / sizeof(double));
  static_assert(kTerms <= 256 && kStateWords <= 256 && sizeof(GnState) % sizeof(double) == 0, "layout");
  static_assert(kThreads == kGnThreads || kThreads == kGnWideThreads, "one lane per term, or four");
  constexpr int kFlight = 16;
  __shared__ double s_sum[kTerms];
  __shared__ double tot[kGnAcc];
  __shared__ double s_st[kStateWords];
  __shared__ GnPrior s_prior;
  const int t = threadIdx.x, lane = t & 63;
  if (t < kStateWords) s_st[t] = reinterpret_cast<const double*>(st_in)[t];
  const auto load = [&](double (&p)[kFlight], int term, int r0) {  // the term's partials r0, r0 + 1, ...
#pragma unroll
    for (int r = 0; r < kFlight; ++r) {
      const int g = (r0 + r) * kWays + term / kGnAcc;
      p[r] = 0.0;
      if (g < grid) p[r] = partials[kGnAcc * (size_t)g + term % kGnAcc];
    }
  };
  const auto add = [&](double s, const double (&p)[kFlight]) {  // 0.0 beyond the grid leaves a sum as it is
#pragma unroll
    for (int r = 0; r < kFlight; ++r) s += p[r];
    return s;
  };
  double p[kFlight];
  if constexpr (kThreads == kGnThreads) {
    if (t < kTerms) {
      double s = 0.0;
      for (int r0 = 0; r0 * kWays < grid; r0 += kFlight) {
        load(p, t, r0);
        s = add(s, p);
      }
      s_sum[t] = s;
    }
  } else {
    const int term = 16 * (t >> 6) + (lane & 15), quarter = lane >> 4;
    if (term < kTerms) {
      load(p, term, kFlight * quarter);
      double s = add(0.0, p);
#pragma unroll
      for (int k = 1; k < 4; ++k) {
        const double before = shfl_d(s, (lane & 15) + 16 * (k - 1));
        const double next = add(before, p);
        s = quarter == k ? next : s;
      }
      if (quarter == 3) s_sum[term] = s;
    }
  }
  if (t == kThreads - 1) {
    GnPrior pr{};
    if (st_in->lam_t > 0.0 || st_in->lam_r > 0.0) motion_prior(*st_in, pr.Ab, pr.cost);
    s_prior = pr;
  }
  __syncthreads();
  if (t < kGnAcc) {
    const double* s = s_sum + t;
    tot[t] = ((s[0] + s[kGnAcc]) + (s[2 * kGnAcc] + s[3 * kGnAcc])) +
             ((s[4 * kGnAcc] + s[5 * kGnAcc]) + (s[6 * kGnAcc] + s[7 * kGnAcc]));
  }
  __syncthreads();
  if (t < 64) gn_step(tot, s_prior, *reinterpret_cast<GnState*>(s_st), s_cand, out, final_step);
  __syncthreads();
  if (out.st && t < kStateWords) reinterpret_cast<double*>(out.st)[t] = s_st[t];
}

// The last evaluation's step alone (one workgroup): the accepted pose is the candidate written to cand.
template <int kThreads>
__global__ __launch_bounds__(kThreads) void k_gn_solve(const double* partials, int grid, const GnState* st_in,
                                                       GnState* st_out, double* cand, double* stats_row) {
  __shared__ double s_cand[12];
  gn_solve_wg<kThreads>(partials, grid, st_in, GnStepOut{st_out, cand, stats_row}, s_cand, 1);
}

// A tracked frame's: the accepted pose, rounded to FP32, is the frame's pose; the solver's rows of
// this frame go to the per-frame stats.
template <int kThreads>
__global__ __launch_bounds__(kThreads) void k_track_solve(const double* partials, int grid, const GnState* st_in,
                                                          GnState* st_out, double* cand, TrackArgs t) {
  __shared__ double s_cand[12];
  const uint32_t fs = track_slot(t);
  const int k = threadIdx.x, before = t.iters * kGnStats;  // the earlier evaluations' rows are there
  double* rows = t.stats ? t.stats + (size_t)fs * (before + kGnStats) : nullptr;
  if (rows)
    for (int j = k; j < before; j += kThreads) rows[j] = t.eval_stats[j];
  gn_solve_wg<kThreads>(partials, grid, st_in, GnStepOut{st_out, cand, rows ? rows + before : nullptr}, s_cand, 1);
  if (k < 16) t.out[16 * (size_t)fs + k] = k < 12 ? (float)s_cand[k] : (k == 15 ? 1.0f : 0.0f);
}

}  // namespace

// ============================================================================ launchers
template <class F>
static void with_input(bool u16, bool color, F f) {
  using T = std::true_type;
  using N = std::false_type;
  if (u16) {
    if (color) f(T(), T());
    else f(T(), N());
  } else {
    if (color) f(N(), T());
    else f(N(), N());
  }
}

hipError_t launch_alloc(const FrameArgs& a, int depth_u16, int k, hipStream_t st) {
  const int bands = k > 1 ? kAllocBands : 1;
  const uint32_t tiles = alloc_tiles(a.W, a.H, bands);
  const dim3 g(tiles * k), b(256);
  with_input(depth_u16 != 0, a.rgba != nullptr, [&](auto U, auto C) {
    constexpr bool u16 = decltype(U)::value, col = decltype(C)::value;
    if (bands > 1) hipLaunchKernelGGL((k_alloc<u16, kAllocBands, col>), g, b, 0, st, a, tiles);
    else hipLaunchKernelGGL((k_alloc<u16, 1, col>), g, b, 0, st, a, tiles);
  });
  return hipGetLastError();
}

// Calls f(std::integral_constant<int, storage>) for the runtime storage format.
template <class F>
static void with_storage(int storage, F f) {
  switch (storage) {
    case VH_STORAGE_F16: f(std::integral_constant<int, VH_STORAGE_F16>()); break;
    case VH_STORAGE_F16R: f(std::integral_constant<int, VH_STORAGE_F16R>()); break;
    default: f(std::integral_constant<int, VH_STORAGE_F32>()); break;
  }
}

hipError_t launch_integrate(const FrameArgs& a, int storage, int grid, int k, hipStream_t st) {
  with_storage(storage, [&](auto S) {
    const dim3 g(grid / kIntegrateWaves), b(64 * kIntegrateWaves);
    constexpr int kS = decltype(S)::value;
    const auto kern = a.colors ? (k > 1 ? k_integrate<kS, true, true> : k_integrate<kS, true, false>)
                               : (k > 1 ? k_integrate<kS, false, true> : k_integrate<kS, false, false>);
    hipLaunchKernelGGL(kern, g, b, 0, st, a, (uint32_t)k);
  });
  return hipGetLastError();
}

hipError_t launch_carve(const FrameArgs& a, int k, hipStream_t st) {
  const uint32_t g = min(kCarveGroups, (a.pool_cap + 255u) / 256u);
  hipLaunchKernelGGL(k_carve, dim3(g), dim3(256), 0, st, a, (uint32_t)k);
  return hipGetLastError();
}

hipError_t launch_integrate_alloc(const FrameArgs& a, int storage, int depth_u16, int grid, int k_int, int k_alloc,
                                  hipStream_t st) {
  const uint32_t ig = (uint32_t)(grid / kIntegrateWaves);
  const uint32_t tiles = alloc_tiles(a.W, a.H, kAllocBands);
  const uint32_t ag = tiles * (uint32_t)k_alloc;
  with_storage(storage, [&](auto S) {
    with_input(depth_u16 != 0, a.colors != nullptr, [&](auto U, auto C) {
      const dim3 g(ig + ag), b(64 * kIntegrateWaves);
      hipLaunchKernelGGL((k_integrate_alloc<decltype(S)::value, decltype(U)::value, decltype(C)::value>), g, b, 0,
                         st, a, ig, ag, tiles, (uint32_t)k_int);
    });
  });
  return hipGetLastError();
}

// Grid of the per-block extraction kernels: one wave per block, kMcWaves per workgroup, so
// the dispatcher balances blocks of unequal work (empty, dense, near-corner). Measured on the
// final room_medium_5mm volume: 0.74 ms per extraction with one-wave workgroups against
// 0.87 ms with 8,192 block-striding workgroups and 0.85 ms with one resident round of them.
template <class Kernel>
static uint32_t block_grid(Kernel, uint32_t n_blocks) {
  return (n_blocks + kMcWaves - 1) / kMcWaves;
}

hipError_t launch_mc(const McArgs& a, int storage, hipStream_t st) {
  if (a.n_blocks == 0) return hipSuccess;
  const uint32_t n_chunks = (a.n_blocks + kScanChunk - 1) / kScanChunk;
  hipLaunchKernelGGL(k_mc_neighbours, dim3((uint32_t)(((size_t)a.n_blocks * 8 + 255) / 256)), dim3(256), 0, st, a);
  with_storage(storage, [&](auto S) {
    auto kc = k_mc_count<decltype(S)::value>;
    hipLaunchKernelGGL(kc, dim3(block_grid(kc, a.n_blocks)), dim3(64 * kMcWaves), 0, st, a);
  });
  hipLaunchKernelGGL(k_scan_chunks, dim3(n_chunks), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(256), 0, st, a, n_chunks);
  with_storage(storage, [&](auto S) {
    auto kw = a.colors ? k_mc_write<decltype(S)::value, true> : k_mc_write<decltype(S)::value, false>;
    hipLaunchKernelGGL(kw, dim3(block_grid(kw, a.n_blocks)), dim3(64 * kMcWaves), 0, st, a);
  });
  return hipGetLastError();
}

hipError_t launch_mesh_index_count(const McArgs& a, int storage, hipStream_t st) {
  if (a.n_blocks == 0) return hipSuccess;
  const uint32_t n_chunks = (a.n_blocks + kScanChunk - 1) / kScanChunk;
  hipLaunchKernelGGL(k_mc_neighbours, dim3((uint32_t)(((size_t)a.n_blocks * 8 + 255) / 256)), dim3(256), 0, st, a);
  with_storage(storage, [&](auto S) {
    auto km = k_ix_mark<decltype(S)::value>;
    hipLaunchKernelGGL(km, dim3(block_grid(km, a.n_blocks)), dim3(64 * kMcWaves), 0, st, a);
  });
  hipLaunchKernelGGL(k_ix_count, dim3(min((a.n_blocks + 3u) / 4u, 16384u)), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_scan_chunks, dim3(n_chunks), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(256), 0, st, a, n_chunks);
  McArgs v = a;  // the same scans over the vertex counts
  v.counts = a.vcounts;
  v.chunk_sums = a.vchunks;
  v.total = a.vtotal;
  hipLaunchKernelGGL(k_scan_chunks, dim3(n_chunks), dim3(256), 0, st, v);
  hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(256), 0, st, v, n_chunks);
  return hipGetLastError();
}

hipError_t launch_mesh_index_write(const McArgs& a, int storage, hipStream_t st) {
  if (a.n_blocks == 0) return hipSuccess;
  with_storage(storage, [&](auto S) {
    auto kw = (a.colors && a.vrgb) ? k_ix_write<decltype(S)::value, true> : k_ix_write<decltype(S)::value, false>;
    hipLaunchKernelGGL(kw, dim3(block_grid(kw, a.n_blocks)), dim3(64 * kMcWaves), 0, st, a);
  });
  return hipGetLastError();
}

static uint32_t stream_grid(uint32_t n) { return min((n + 3u) / 4u, 16384u); }

hipError_t launch_stream_out(const StreamArgs& a, hipStream_t st) {
  if (a.n) hipLaunchKernelGGL(k_st_out, dim3(stream_grid(a.n)), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_stream_move(const StreamArgs& a, hipStream_t st) {
  if (a.n) hipLaunchKernelGGL(k_st_move, dim3(stream_grid(a.n)), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_stream_rehash(const StreamArgs& a, hipStream_t st) {
  if (a.n) hipLaunchKernelGGL(k_st_rehash, dim3((a.n + 255u) / 256u), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_stream_insert(const StreamArgs& a, int storage, hipStream_t st) {
  if (!a.n) return hipSuccess;
  hipLaunchKernelGGL(k_st_insert, dim3((a.n + 255u) / 256u), dim3(256), 0, st, a);
  with_storage(storage, [&](auto S) {
    hipLaunchKernelGGL(k_st_place<decltype(S)::value>, dim3(stream_grid(a.n)), dim3(256), 0, st, a);
  });
  return hipGetLastError();
}

static int query_grid(int64_t n) {
  int64_t g = (n + 255) / 256;
  if (g > 4096) g = 4096;
  if (g < 1) g = 1;
  return (int)g;
}

hipError_t launch_copy_in(void* dst, const void* src, size_t bytes, hipStream_t st) {
  if (bytes == 0) return hipSuccess;
  const size_t g = std::min<size_t>(bytes / 2048 + 1, 1024);
  hipLaunchKernelGGL(k_copy_in, dim3((uint32_t)g), dim3(256), 0, st, static_cast<char*>(dst), static_cast<const char*>(src), bytes);
  return hipGetLastError();
}

hipError_t launch_words_out(uint32_t* dst, const void* a, int na, const void* b, int nb, hipStream_t st) {
  hipLaunchKernelGGL(k_words_out, dim3(1), dim3(256), 0, st, dst, static_cast<const uint32_t*>(a), na,
                     static_cast<const uint32_t*>(b), nb);
  return hipGetLastError();
}

hipError_t launch_query(const QueryArgs& q, int storage, const float* pts, int64_t n, float* sdf, uint8_t* valid,
                        hipStream_t st) {
  const int g = query_grid(n);
  with_storage(storage, [&](auto S) {
    hipLaunchKernelGGL(k_query<decltype(S)::value>, dim3(g), dim3(256), 0, st, q, pts, n, sdf, valid);
  });
  return hipGetLastError();
}

hipError_t launch_backward(const QueryArgs& q, int storage, const float* pts, int64_t n, const float* T12,
                           const float* grad_r, float* r, uint8_t* valid, float* J, double* partials, int grid,
                           float* voxel_grad, hipStream_t st) {
  const int64_t per = ((n + grid - 1) / grid + 255) / 256 * 256;
  with_storage(storage, [&](auto S) {
    hipLaunchKernelGGL(k_backward<decltype(S)::value>, dim3(grid), dim3(256), 0, st, q, pts, n, per, T12, grad_r, r,
                       valid, J, partials, voxel_grad);
  });
  return hipGetLastError();
}

hipError_t launch_reduce6(const double* partials, int grid, double* out6, hipStream_t st) {
  hipLaunchKernelGGL(k_reduce6, dim3(1), dim3(384), 0, st, partials, grid, out6);
  return hipGetLastError();
}

hipError_t launch_gn_accum(const GnArgs& a, int storage, hipStream_t st) {
  with_storage(storage, [&](auto S) {
    constexpr int kS = decltype(S)::value;
    if (a.n <= 256 * (int64_t)a.grid) hipLaunchKernelGGL(k_gn_accum<kS>, dim3(a.grid), dim3(kGnThreads), 0, st, a);
    else hipLaunchKernelGGL(k_gn_accum_wide<kS>, dim3(a.grid / 2), dim3(kGnWideThreads), 0, st, a);
  });
  return hipGetLastError();
}

// 128 partials: one round of loads for a lane per term.
hipError_t launch_gn_solve(const double* partials, int grid, const GnState* st_in, GnState* st_out, double* cand,
                           double* stats_row, hipStream_t st) {
  if (grid <= 128) hipLaunchKernelGGL(k_gn_solve<kGnThreads>, dim3(1), dim3(kGnThreads), 0, st, partials, grid, st_in, st_out, cand, stats_row);
  else hipLaunchKernelGGL(k_gn_solve<kGnWideThreads>, dim3(1), dim3(kGnWideThreads), 0, st, partials, grid, st_in, st_out, cand, stats_row);
  return hipGetLastError();
}

hipError_t launch_track_solve(const double* partials, int grid, const GnState* st_in, GnState* st_out, double* cand,
                              const TrackArgs& t, hipStream_t st) {
  if (grid <= 128) hipLaunchKernelGGL(k_track_solve<kGnThreads>, dim3(1), dim3(kGnThreads), 0, st, partials, grid, st_in, st_out, cand, t);
  else hipLaunchKernelGGL(k_track_solve<kGnWideThreads>, dim3(1), dim3(kGnWideThreads), 0, st, partials, grid, st_in, st_out, cand, t);
  return hipGetLastError();
}

}  // namespace vh
