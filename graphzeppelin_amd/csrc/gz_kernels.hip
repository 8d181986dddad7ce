// gz_kernels.hip -- hand-written gfx950 kernels for GraphZeppelin's streaming-CC hot path.
//
// Data layout in HBM (one "slab" per algorithm instance): row v holds vertex v's sketch as packed
// bucket records {u64 alpha; G gamma} (G = u32 for the 12-byte reference bucket, u64 for the
// 16-byte one).  The low depths of two columns share a 128-B line (with the deterministic bucket in
// the pairing's last slot) and deeper depths follow per column in an overflow region (RowLayout in
// gz_common.hpp).  Kernels address buckets by the reference's index b = c*D + d (deterministic
// bucket last, b = C*D, src/sketch.cpp:69-83), so packing a row reproduces the reference's image.
// Everything is integer work; nothing here is a dense contraction, so no MFMA is used.
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <type_traits>
#include <utility>

#include "gz_kernels.hpp"

namespace gz {

namespace {

constexpr int kWave = 64;

__device__ inline uint32_t lane_id() { return __lane_id(); }

__device__ inline uint32_t rd_lane_u32(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ inline uint64_t rd_lane_u64(uint64_t v, int lane) {
  uint32_t lo = rd_lane_u32((uint32_t)v, lane), hi = rd_lane_u32((uint32_t)(v >> 32), lane);
  return ((uint64_t)hi << 32) | lo;
}
__device__ inline uint64_t shfl_u64(uint64_t v, int src) {
  uint32_t lo = __shfl((unsigned)(uint32_t)v, src), hi = __shfl((unsigned)(uint32_t)(v >> 32), src);
  return ((uint64_t)hi << 32) | lo;
}
__device__ inline uint64_t shfl_xor_u64(uint64_t v, int o) {
  uint32_t lo = __shfl_xor((unsigned)(uint32_t)v, o), hi = __shfl_xor((unsigned)(uint32_t)(v >> 32), o);
  return ((uint64_t)hi << 32) | lo;
}
__device__ inline uint64_t wave_xor_u64(uint64_t v) {
  for (int o = 32; o > 0; o >>= 1) {
    uint32_t lo = __shfl_xor((unsigned)(uint32_t)v, o), hi = __shfl_xor((unsigned)(uint32_t)(v >> 32), o);
    v ^= ((uint64_t)hi << 32) | lo;
  }
  return v;
}
// XOR over the wave of a 32-bit value, returned to every lane: DPP row shifts build each row's XOR
// in its lane 15, two row broadcasts carry it to lane 63 (no LDS round trips).  Every lane must be
// active.
__device__ inline uint32_t wave_xor_dpp_u32(uint32_t v) {
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return (uint32_t)__builtin_amdgcn_readlane((int)v, kWave - 1);
}
__device__ inline uint64_t wave_xor_dpp_u64(uint64_t v) {
  const uint32_t lo = wave_xor_dpp_u32((uint32_t)v), hi = wave_xor_dpp_u32((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}
__device__ inline uint64_t wave_incl_scan_u64(uint64_t x) {
  const uint32_t lane = lane_id();
  for (int o = 1; o < kWave; o <<= 1) {
    uint32_t lo = __shfl_up((unsigned)(uint32_t)x, o), hi = __shfl_up((unsigned)(uint32_t)(x >> 32), o);
    uint64_t y = ((uint64_t)hi << 32) | lo;
    if (lane >= (uint32_t)o) x += y;
  }
  return x;
}

template <class T>
__device__ inline void lds_xor(T* p, T v) {
  __hip_atomic_fetch_xor(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <class T>
__device__ inline void gbl_xor(T* p, T v) {
  __hip_atomic_fetch_xor(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ inline void gbl_or(T* p, T v) {
  __hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ inline T ld_acq(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ inline void st_rlx(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- the slab: packed bucket records -----------------------------------------------------------
// Every bucket is the record {u64 alpha; G gamma} -- the reference's packed Bucket, 12 or 16 bytes.
// Row v of the slab holds sketch v (layout in gz_common.hpp, RowLayout): depths below g.low of two
// columns share a 128-B line, with the deterministic bucket in the pairing's slot C; deeper depths
// of each column follow in the overflow region, each column's run on its own lines.  A 12-byte
// record is only 4-byte aligned, so it is moved as 32-bit words, and a 64-bit XOR atomic on it
// becomes two 32-bit ones (XOR acts bit by bit, so the result is the same).
// rec_col_off: byte of (column c, depth d) within a row; det_col_off: byte of the deterministic
// bucket; rec_off: byte of the reference's bucket index b (c * D + d, the deterministic bucket last)
// of sketch v.
template <class G>
__device__ inline uint32_t rec_col_off(const Geo& g, uint32_t c, uint32_t d) {
  constexpr uint32_t RB = 8 + sizeof(G);
  return d < g.low ? (c >> 1) * 128u + (c & 1u) * 64u + d * RB : g.ovf + c * g.opitch + (d - g.low) * RB;
}
__device__ inline uint32_t det_col_off(const Geo& g) { return (g.C >> 1) * 128u + (g.C & 1u) * 64u; }
// Deep flags (rows of 12-byte records only): the word after a column's at most five low records,
// byte 60 of its half-line, becomes 1 once any record of the column that ends past the first line
// of its overflow run (depth >= low + 10) has been written nonzero: every writer of such a record
// (the update kernel's deep path, k_packed) stores 1 there, and only a reset of the row clears it.
// A Borůvka reduce reads those records only for members whose flag is set; for the others they are
// zero.  An update reaches such a depth once in 2^15 (update, column) pairs, so most vertices never
// set their flags, and the reduce reads one overflow line of the column instead of three.
template <class G>
constexpr bool kDeepFlags = sizeof(G) == 4;
__device__ inline uint32_t deep_flag_off(uint32_t c) { return (c >> 1) * 128u + (c & 1u) * 64u + 60u; }
__device__ inline bool rec_is_deep(const Geo& g, uint32_t d) { return d >= g.low && (d - g.low) * 12u + 11u >= 128u; }
template <class G>
__device__ inline size_t rec_off(const Geo& g, uint32_t v, uint32_t b) {
  if (b == g.nb - 1) return (size_t)v * g.row + det_col_off(g);
  const uint32_t c = b / g.D, d = b - c * g.D;
  return (size_t)v * g.row + rec_col_off<G>(g, c, d);
}
template <class G>
__device__ inline void ld_rec(const unsigned char* p, uint64_t* a, G* gm) {
  if (sizeof(G) == 4) {
    const uint32_t* w = reinterpret_cast<const uint32_t*>(p);
    *a = ((uint64_t)w[1] << 32) | w[0];
    *gm = (G)w[2];
  } else {
    const uint64_t* w = reinterpret_cast<const uint64_t*>(p);
    *a = w[0];
    *gm = (G)w[1];
  }
}
template <class G>
__device__ inline void st_rec(unsigned char* p, uint64_t a, G gm) {
  if (sizeof(G) == 4) {
    uint32_t* w = reinterpret_cast<uint32_t*>(p);
    w[0] = (uint32_t)a;
    w[1] = (uint32_t)(a >> 32);
    w[2] = (uint32_t)gm;
  } else {
    uint64_t* w = reinterpret_cast<uint64_t*>(p);
    w[0] = a;
    w[1] = (uint64_t)gm;
  }
}
template <class G>
__device__ inline void xor_rec_atomic(unsigned char* p, uint64_t a, G gm) {
  if (sizeof(G) == 4) {
    uint32_t* w = reinterpret_cast<uint32_t*>(p);
    if ((uint32_t)a) gbl_xor(w, (uint32_t)a);
    if ((uint32_t)(a >> 32)) gbl_xor(w + 1, (uint32_t)(a >> 32));
    if (gm) gbl_xor(w + 2, (uint32_t)gm);
  } else {
    uint64_t* w = reinterpret_cast<uint64_t*>(p);
    if (a) gbl_xor(w, a);
    if (gm) gbl_xor(w + 1, (uint64_t)gm);
  }
}

// ---- DSU (include/dsu.h:101-174 restated for the device) --------------------------------------
// Priorities are a bijective 32-bit mix of the vertex id, so (priority, id) is a strict total
// order and linking the lower-priority root under the higher one can never form a cycle.
__device__ inline uint32_t dsu_prio(uint32_t v, uint32_t seed) {
  uint32_t h = v ^ seed;
  h ^= h >> 16; h *= 0x85ebca6bu; h ^= h >> 13; h *= 0xc2b2ae35u; h ^= h >> 16;
  return h;
}
// path halving, dsu.h:145-152, from u whose parent p is already loaded
__device__ inline uint32_t dsu_find_from(uint32_t* parent, uint32_t u, uint32_t p) {
  while (p != u) {
    const uint32_t gp = ld_acq(parent + p);
    if (gp == p) return p;
    st_rlx(parent + u, gp);
    u = gp;
    p = ld_acq(parent + u);
  }
  return u;
}
__device__ inline uint32_t dsu_find(uint32_t* parent, uint32_t u) { return dsu_find_from(parent, u, ld_acq(parent + u)); }
// find for kernels in which no thread links roots (only compression writes, which keep every
// pointer on the path to the root): cached loads are enough.
__device__ inline uint32_t dsu_find_stable(uint32_t* parent, uint32_t u) {
  uint32_t p = parent[u];
  while (true) {
    const uint32_t gp = parent[p];
    if (gp == p) return p;
    u = p;
    p = gp;
  }
}

constexpr uint32_t kNoLink = 0xFFFFFFFFu;
// CAS union ordered by rank (dsu.h:155-167): the higher hint first (when hints are given), then the
// higher priority, then the smaller id.  Any total order that stays fixed while links run
// concurrently keeps the forest acyclic (a root is only linked under a root that ranks higher), so
// the order may differ between launches.  Hints that rank high-degree vertices first let the many
// merges into a hub go through the smaller roots' own parent words instead of all contending for
// the hub's.  Returns the root that was linked under the other one, or kNoLink when a and b were
// already connected.
// LATE: the hints are loaded once the roots are known to differ (a batch whose edges are mostly
// connected already); otherwise with the parents (Borůvka's samples, which mostly link).
//
// The first walk takes its parents through the caches: a stale parent is still an ancestor, so equal
// roots are connected, and the CAS finds out whether the lower root is one still; a winner that was
// linked meanwhile ranks higher all the same.  After a lost CAS the walk goes on from the parent the
// CAS returned, with device-coherent loads.
template <class T>
__device__ inline T ld_cached(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
template <bool LATE = false>
__device__ inline uint32_t dsu_link(uint32_t* parent, uint32_t a, uint32_t b, uint32_t pseed,
                                    const unsigned char* hint) {
  // both first parents (and hints) in one round trip; a root (the common case) needs no more
  uint32_t pa = ld_cached(parent + a), pb = ld_cached(parent + b);
  uint32_t ha = 0, hb = 0;
  if (!LATE) {
    ha = hint[a];
    hb = hint[b];
  }
  // one step of both walks per round trip, splitting the paths
  while (pa != a || pb != b) {
    const uint32_t ga = pa != a ? ld_cached(parent + pa) : pa, gb = pb != b ? ld_cached(parent + pb) : pb;
    if (!LATE && pa != a) ha = hint[pa];
    if (!LATE && pb != b) hb = hint[pb];
    if (pa != a && ga != pa) st_rlx(parent + a, ga);
    if (pb != b && gb != pb) st_rlx(parent + b, gb);
    a = pa;
    pa = ga;
    b = pb;
    pb = gb;
  }
  while (true) {
    if (a == b) return kNoLink;
    if (LATE) {
      ha = hint[a];
      hb = hint[b];
    }
    const uint32_t wa = dsu_prio(a, pseed), wb = dsu_prio(b, pseed);
    const bool a_wins = ha != hb ? ha > hb : wa != wb ? wa > wb : a < b;
    if (!a_wins) {
      uint32_t t = a; a = b; b = t;
      t = ha; ha = hb; hb = t;
    }
    uint32_t expected = b;
    if (__hip_atomic_compare_exchange_strong(parent + b, &expected, a, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
      return b;
    const uint32_t a_up = ld_acq(parent + a);
    const uint32_t rb = dsu_find_from(parent, b, expected), ra = dsu_find_from(parent, a, a_up);
    if (!LATE && rb != b) hb = hint[rb];
    if (!LATE && ra != a) ha = hint[ra];
    a = ra;
    b = rb;
  }
}

// ---- spanning-forest edge set (open addressing on 64-bit edge ids) ----------------------------
constexpr uint64_t kEmpty = ~0ull;
__device__ inline uint64_t mix64(uint64_t k) {
  k ^= k >> 33; k *= 0xff51afd7ed558ccdULL; k ^= k >> 33; k *= 0xc4ceb9fe1a85ec53ULL; k ^= k >> 33;
  return k;
}
// Linear probing at a load of at most a half: most keys end in their home slot, but the longest of 2^18
// probe sequences, taken slot by slot, had a launch wait for 20 dependent round trips.  Past the home slot
// a line's worth of slots is read at once: the deletion check of 5000 updates on 2^18 vertices 8.8 -> 4.9 us.
constexpr uint32_t kSfStep = 8;
__device__ inline void sf_insert(const DsuDev& d, uint64_t key) {
  uint64_t h = mix64(key) & d.sf_mask;
  for (uint64_t probe = 0; probe <= d.sf_mask; ++probe) {
    uint64_t expected = kEmpty;
    if (__hip_atomic_compare_exchange_strong(d.sf_hash + h, &expected, key, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT) ||
        expected == key)
      return;
    uint32_t skip = 0;
    while (skip == 0 && probe <= d.sf_mask) {  // to the next slot that is empty or holds the key
      uint64_t cur[kSfStep];
#pragma unroll
      for (uint32_t k = 0; k < kSfStep; ++k) cur[k] = ld_acq(d.sf_hash + ((h + 1 + k) & d.sf_mask));
#pragma unroll
      for (uint32_t k = 0; k < kSfStep; ++k)
        if (skip == 0 && (cur[k] == kEmpty || cur[k] == key)) skip = k + 1;
      h = (h + (skip ? skip : kSfStep)) & d.sf_mask;
      if (!skip) probe += kSfStep;
    }
  }
}
__device__ inline bool sf_contains(const DsuDev& d, uint64_t key) {
  const uint64_t home = mix64(key) & d.sf_mask;
  const uint64_t first = ld_acq(d.sf_hash + home);
  if (first == key) return true;
  if (first == kEmpty) return false;
  for (uint64_t probe = 1; probe <= d.sf_mask; probe += kSfStep) {
    uint64_t cur[kSfStep];
#pragma unroll
    for (uint32_t k = 0; k < kSfStep; ++k) cur[k] = ld_acq(d.sf_hash + ((home + probe + k) & d.sf_mask));
#pragma unroll
    for (uint32_t k = 0; k < kSfStep; ++k) {
      if (cur[k] == key) return true;
      if (cur[k] == kEmpty) return false;
    }
  }
  return false;
}

// Sample records of round 0: a GOOD sample stores its edge index, whose endpoints are both below
// n <= 2^32 - 1 after the range check, so it never equals the two sentinels (high half all ones)
// that stand for ZERO and FAIL.
constexpr uint64_t kSampZero = ~0ull;
constexpr uint64_t kSampEmpty = ~0ull - 1;  // ZERO, and the column's buckets that were read are empty as well
constexpr uint64_t kSampFail = ~0ull - 2;

// An index whose endpoints are out of range (a checksum collision) counts as FAIL and raises the
// bad-sample flag (plain store: every writer stores the same value).
constexpr int kEmptyCode = 3;  // beside SampleCode
__device__ inline uint64_t sample_record(int code, uint64_t idx, uint32_t n, uint32_t* flags) {
  if (code == kZero) return kSampZero;
  if (code == kEmptyCode) return kSampEmpty;
  if (code != kGood) return kSampFail;
  if ((uint32_t)(idx >> 32) >= n || (uint32_t)idx >= n) {
    flags[kFlagBad] = 1;
    return kSampFail;
  }
  return idx;
}

// ---- sample (src/sketch.cpp:94-116) over one wave --------------------------------------------
// Lane l < D holds bucket (column, depth l), lane D the deterministic bucket.  Every lane checks its
// own record with one hash, so the deterministic bucket's check runs alongside the column's.
// Returns the code, kEmptyCode for a ZERO without a nonzero bucket; *idx gets the sampled index on GOOD.
template <class G>
__device__ inline int wave_sample(uint64_t a, G gm, uint32_t D, uint64_t chk_bf, uint64_t* idx) {
  const uint32_t lane = lane_id();
  const uint64_t mask = __ballot(lane <= D && (G)xxh3_mix(xxh3_prep(a), chk_bf) == gm);
  const uint64_t det_a = rd_lane_u64(a, (int)D);
  const G det_g = (G)rd_lane_u64((uint64_t)gm, (int)D);
  if (det_a == 0 && det_g == 0) { *idx = 0; return __ballot((a | (uint64_t)gm) != 0) ? kZero : kEmptyCode; }
  if ((mask >> D) & 1) { *idx = det_a; return kGood; }
  const uint64_t col = mask & ((1ull << D) - 1);
  if (col) {
    *idx = rd_lane_u64(a, __builtin_ctzll(col));
    return kGood;
  }
  *idx = 0;
  return kFail;
}

// ================================================================================================
// fills
// ================================================================================================
__global__ void k_fill_u32(uint32_t* p, uint32_t v, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_fill_u64(uint64_t* p, uint64_t v, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// ================================================================================================
// Sketch update: Sketch::update over a batch (src/sketch.cpp:69-83) fused with the delta merge
// (src/cc_sketch_alg.cpp:106-118, src/sketch.cpp:149-154).
//
// One wave (a 64-thread workgroup) per tile of <= tile-size destinations of one vertex, so a CU
// keeps up to 32 tiles in flight: most tiles of a flush hold a handful of updates, and a tile's
// time is the latency of its few dependent memory round trips, not bandwidth.  Lanes take
// (update, column) pairs; the tile's delta for the lower depths of every column lives in LDS
// (lds_depth), and the rare deeper contributions are XORed straight into the vertex's records
// with device-scope atomics (setting the column's deep flag when the record lies past the first
// line of the column's overflow run).  The deterministic bucket is kept in registers and reduced
// once per tile.
// Long tiles are bound by VALU issue (a pair's hash is two 64-bit products, six quarter-rate
// multiplies of about 50 instructions before), so everything of the hash that is linear is taken out
// of the pairs: an update's index and a column's bitflip are spread once (xxh3_spread) and a pair
// XORs them; the depth is read from the hash's low word, whose second product then needs two 24-bit
// multiplies instead of two of the quarter-rate ones (hash_low28), and a pair's two LDS addresses come
// from one multiply-add; indices are rebuilt from the other end, so the pair still costs one 16-byte LDS
// read.  24M Chung-Lu updates on 2^18 vertices 2153 -> 1290 us in all (hash_low28 and the addresses 1530
// -> 1415), 16M R-MAT on 2^20 2189 -> 1550 us, flushes of a serving trace (about 6 updates per vertex,
// bound by the tiles' memory round trips) 206 -> 193 us.  The write-back is a read-xor-write of the touched records, or device-scope
// atomic XOR when the vertex is split across tiles of the same launch.  Workgroups walk the tiles
// grid-stride (no shared counter), so a persistent grid can cover a tile count that only the
// device knows.
// ================================================================================================
// Entries of the LDS delta that a lane writes back in one pass, and the depths of a column held there.
// With 4-byte checksums as many as one pass takes, 9 (28 columns, a deep pair in 512) to 14 (18 columns),
// and a CU still has LDS for its 32 tiles: 24M Chung-Lu updates on 2^18 vertices (25 columns, 10 depths
// against 9) 1415 -> 1290 us.  With 8-byte checksums the larger delta would take tiles from a CU, which
// costs flushes of a few updates per vertex 3% (dense ones would gain 8%), and where a pass does not hold
// 9 depths there are several.  Deep records that need a flag begin at depth 15.
constexpr uint32_t kPerLane = 4, kLdsDepthMin = 9, kLdsDepthMax = 14;
uint32_t lds_depth(uint32_t C, int gbytes) {
  const uint32_t d = gbytes == 4 ? (kPerLane * kWave - 1) / C : 0;
  return d < kLdsDepthMin ? kLdsDepthMin : d > kLdsDepthMax ? kLdsDepthMax : d;
}
// (a mod 2^24) * (b mod 2^24) + c; from plain C the compiler takes the quarter-rate 32-bit multiply.
__device__ inline uint32_t mad24(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "Is"(b), "v"(c));
  return r;
}
// Low word of the hash of x, a spread index ^ bitflip (xxh3_products and the last step), exact in its low
// 28 bits.  They need the second product only up to bit 55, so its cross terms are taken modulo 2^24:
// full-rate 24-bit multiplies instead of quarter-rate 32-bit ones.
__device__ inline uint32_t hash_low28(uint64_t x) {
  x *= kPrimeMx2;
  const uint32_t hi = (uint32_t)(x >> 32), lo = (uint32_t)x ^ ((hi >> 3) + 8);
  const uint64_t p = (uint64_t)lo * (uint32_t)kPrimeMx2;
  uint32_t ph = mad24(lo, (uint32_t)(kPrimeMx2 >> 32), (uint32_t)(p >> 32));
  ph = mad24(hi, (uint32_t)kPrimeMx2, ph);
  return (uint32_t)p ^ __builtin_amdgcn_alignbit(ph, (uint32_t)p, 28);
}
// Depth of a bucket from x, the spread index ^ bitflip, and low, hash_low28 of it; at least D: no bucket.
__device__ inline uint32_t bucket_depth(uint32_t low, uint64_t x, uint64_t depth_cap) {
  low &= (1u << 28) - 1;
  if (low) return (uint32_t)__builtin_ctz(low);
  const uint64_t h = xxh3_products(x);
  return (uint32_t)__builtin_ctzll((h ^ (h >> 28)) | depth_cap);
}
// Updates of a chunk from which each lane takes its own one: C steps against m * C / 64 longer ones.
// 24M Chung-Lu updates on 2^18 vertices 1667 -> 1567 us, 3M R-MAT on 2^17 with 8-byte checksums 343 ->
// 307 us, a serving trace's flushes 192 -> 189 us.
constexpr uint32_t kOwnMin = 56;
// s_waitcnt immediate for vmcnt(0), with expcnt and lgkmcnt at their maxima (not waited on)
constexpr unsigned kWaitVmcnt0 = 0x0F70;

// WIDE: more than 28 columns, so the write-back takes more than one pass over the LDS delta (a
// separate instance keeps the one-pass form free of the loop, whose merged paths would make the
// compiler wait on this tile's stores at the next tile's first use of the prefetch register).
template <class G, bool WIDE>
__global__ void __launch_bounds__(kWave, 8)  // 8 waves per SIMD: 32 tiles in flight per CU
k_update_tiles(const Tile* __restrict__ tiles, const uint32_t* __restrict__ ntiles_dev, uint32_t ntiles_host,
               const uint32_t* __restrict__ dsts, unsigned char* __restrict__ slab, Geo g,
               const uint64_t* __restrict__ col_bf, uint32_t ldepth, uint32_t ldepth_inv) {
  extern __shared__ __align__(16) unsigned char smem[];
  const uint32_t C = g.C, D = g.D;
  const uint32_t det_slot = C * ldepth;
  const uint32_t lds_n = det_slot + 1;
  // per chunk, read by the lanes that take an update's columns: its spread index, and the other end
  // and the checksum (kTight: one 16-byte slot), or the index with the checksum in an array of its own
  constexpr bool kTight = sizeof(G) == 4;
  ulonglong2* s_pc = reinterpret_cast<ulonglong2*>(smem);
  uint64_t* s_bf = reinterpret_cast<uint64_t*>(smem + kWave * sizeof(ulonglong2));  // spread bitflips
  uint64_t* s_a = s_bf + C;
  G* s_g = reinterpret_cast<G*>(s_a + lds_n);
  G* s_ck = s_g + lds_n;
  uint16_t* s_bo = reinterpret_cast<uint16_t*>(s_ck + (kTight ? 0 : kWave));  // each delta entry's word in the row
  const uint32_t lane = threadIdx.x;

  for (uint32_t i = lane; i < C; i += kWave) s_bf[i] = xxh3_spread(col_bf[i]);
  const uint64_t chk_sbf = xxh3_spread(g.chk_bf);
  // The delta is zeroed once here; afterwards the write-back clears every entry it reads.  Entries
  // at depth >= D are never written: offset 0.
  for (uint32_t i = lane; i < lds_n; i += kWave) {
    s_a[i] = 0;
    s_g[i] = 0;
    const uint32_t cc = (i * ldepth_inv) >> 16, d = i - cc * ldepth;  // i / ldepth
    s_bo[i] =
        (uint16_t)((i == det_slot ? det_col_off(g) : (d < D ? rec_col_off<G>(g, cc, d) : 0u)) / 4);
  }
  const uint32_t ntiles = ntiles_dev ? *ntiles_dev : ntiles_host;
  const uint64_t depth_cap = 1ull << D;
  const uint32_t lds_d = D < ldepth ? D : ldepth, near_cap = 1u << ldepth;
  // pair p = i * C + c: lane starts at pair `lane` and advances 64 pairs (di updates, dc columns)
  const uint32_t i0 = lane / C, c0 = lane % C;
  const uint32_t di = kWave / C, dc = kWave % C;
  __syncthreads();

  // Updates are taken in chunks of 64: lane l loads update u0 + l once and hashes its index and
  // checksum once into a 16-byte LDS slot; the chunk's (update, column) pairs then read their
  // update's slot with one LDS load, so each pair costs one column hash and no memory round trip.
  // The next tile's descriptor and each lane's first destination are loaded
  // before the current tile's write-back, and that chunk is hashed between the write-back's
  // record loads and its stores, where the wave waits for those loads anyway.  No tile then
  // starts with a wait, which would also wait for the previous tile's stores (the vector memory
  // counter covers stores too).
  // per-lane XOR of the tile's indices and checksums: the deterministic bucket's delta
  uint64_t det_a = 0;
  G det_g = 0;
  auto hash_chunk = [&](const Tile& tt, uint32_t u0, uint32_t dst) {
    const uint32_t m = tt.count - u0 < kWave ? tt.count - u0 : kWave;
    if (lane < m) {
      const uint64_t idx = concat_pairing(tt.vertex, dst);
      const uint64_t sp = xxh3_spread(xxh3_prep(idx));
      uint64_t ck = xxh3_products(sp ^ chk_sbf);
      ck ^= ck >> 28;
      det_a ^= idx;
      det_g ^= (G)ck;
      // the wave's LDS ops stay in order
      s_pc[lane] = make_ulonglong2(sp, kTight ? (ck << 32) | dst : idx);
      if (!kTight) s_ck[lane] = (G)ck;
    }
  };
  uint32_t t = blockIdx.x;
  Tile tl{0, 0, 0, 0};
  if (t < ntiles) {
    tl = tiles[t];
    hash_chunk(tl, 0, lane < tl.count ? dsts[tl.begin + lane] : 0);
  }
  while (t < ntiles) {
    unsigned char* row = slab + (size_t)tl.vertex * g.row;

    for (uint32_t u0 = 0; u0 < tl.count; u0 += kWave) {
      const uint32_t m = tl.count - u0 < kWave ? tl.count - u0 : kWave;
      if (u0 != 0) hash_chunk(tl, u0, lane < m ? dsts[tl.begin + u0 + lane] : 0);
      // one column's bucket of one update
      auto add = [&](uint64_t x, uint32_t c, uint64_t idx, G chk) {
        const uint32_t low = hash_low28(x);
        const uint32_t near = (uint32_t)__builtin_ctz(low | near_cap);
        if (near < lds_d) {
          const uint32_t e = mad24(c, ldepth, near);  // one full-rate step, and one for either address
          lds_xor(s_a + e, idx);
          lds_xor(s_g + e, chk);
        } else {
          const uint32_t depth = bucket_depth(low, x, depth_cap);
          if (depth < D) {
            xor_rec_atomic<G>(row + rec_col_off<G>(g, c, depth), idx, chk);
            if (kDeepFlags<G> && rec_is_deep(g, depth))  // the flag only ever goes from 0 to 1
              st_rlx(reinterpret_cast<uint32_t*>(row + deep_flag_off(c)), 1u);
          }
        }
      };
      if (m >= kOwnMin) {
        // a nearly full chunk: every lane takes its own update through all columns, starting at a
        // column of its own (C steps, none of them with a slot to read)
        if (lane < m) {
          const ulonglong2 pc = s_pc[lane];
          const G chk = kTight ? (G)(pc.y >> 32) : s_ck[lane];
          const uint64_t idx = kTight ? concat_pairing(tl.vertex, (uint32_t)pc.y) : pc.y;
          uint32_t c = c0;
          for (uint32_t k = 0; k < C; ++k) {
            add(pc.x ^ s_bf[c], c, idx, chk);
            ++c;
            c = c < c - C ? c : c - C;  // C - C, or c - C below zero
          }
        }
        continue;
      }
      const uint32_t np = m * C;
      const uint32_t iters = (np + kWave - 1) / kWave;  // uniform over the wave
      uint32_t q = i0, c = c0;
      for (uint32_t it = 0; it < iters; ++it) {
        if (it * kWave + lane < np) {  // q < m here
          const ulonglong2 pc = s_pc[q];
          const uint64_t x = pc.x ^ s_bf[c];
          const G chk = kTight ? (G)(pc.y >> 32) : s_ck[q];
          const uint64_t idx = kTight ? concat_pairing(tl.vertex, (uint32_t)pc.y) : pc.y;
          add(x, c, idx, chk);
        }
        q += di;
        c += dc;
        if (c >= C) {
          c -= C;
          ++q;
        }
      }
    }
    {
      const uint64_t da = wave_xor_dpp_u64(det_a);
      const G dg = sizeof(G) == 4 ? (G)wave_xor_dpp_u32((uint32_t)det_g) : (G)wave_xor_dpp_u64((uint64_t)det_g);
      if (lane == 0 && (da | (uint64_t)dg)) {
        s_a[det_slot] ^= da;
        s_g[det_slot] ^= dg;
      }
      det_a = 0;
      det_g = 0;
    }
    __syncthreads();

    const uint32_t tn = t + gridDim.x;
    // The previous tile's stores complete before this tile's loads are issued (measured: letting
    // them overlap is slower).
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    Tile tl_next{0, 0, 0, 0};
    uint32_t dst_next = 0;
    if (tn < ntiles) {
      tl_next = tiles[tn];
      if (lane < tl_next.count) dst_next = dsts[tl_next.begin + lane];
    }

    // write-back: read-xor-write of the touched records, four LDS entries per lane in flight
    auto write_back = [&](uint32_t e0, bool first) {
      uint64_t da[kPerLane], ga[kPerLane];
      G dg[kPerLane], gg[kPerLane];
      uint32_t bo[kPerLane];
#pragma unroll
      for (uint32_t k = 0; k < kPerLane; ++k) {
        const uint32_t e = e0 + k * kWave + lane;
        da[k] = 0;
        dg[k] = 0;
        bo[k] = 0;
        if (e < lds_n) {
          bo[k] = (uint32_t)s_bo[e] * 4u;
          da[k] = s_a[e];
          dg[k] = s_g[e];
          if ((da[k] | (uint64_t)dg[k]) != 0) {
            s_a[e] = 0;
            s_g[e] = 0;
          }
        }
      }
      if (!tl.split) {
#pragma unroll
        for (uint32_t k = 0; k < kPerLane; ++k)
          if ((da[k] | (uint64_t)dg[k]) != 0) ld_rec<G>(row + bo[k], &ga[k], &gg[k]);
      }
      // The next tile's first chunk, hashed while this tile's record loads are in flight.  The
      // empty asm, on every path of the first pass, keeps the compiler from hoisting the hash
      // above the loads (it would wait there for the prefetch) and leaves no prefetch pending
      // into the next tile, where a reuse of its register would wait on all of this tile's
      // stores.  The record loads leave ga/gg unset for entries they skip, so no zero fill of
      // those registers waits on earlier memory operations either.
      if (first) {
        asm volatile("" : "+v"(dst_next)::"memory");
        if (tn < ntiles) hash_chunk(tl_next, 0, dst_next);
      }
      if (tl.split) {
#pragma unroll
        for (uint32_t k = 0; k < kPerLane; ++k)
          if ((da[k] | (uint64_t)dg[k]) != 0) xor_rec_atomic<G>(row + bo[k], da[k], dg[k]);
      } else {
#pragma unroll
        for (uint32_t k = 0; k < kPerLane; ++k)
          if ((da[k] | (uint64_t)dg[k]) != 0) st_rec<G>(row + bo[k], ga[k] ^ da[k], (G)(gg[k] ^ dg[k]));
      }
    };
    write_back(0, true);  // the delta holds at least the deterministic bucket's entry
    for (uint32_t e0 = kPerLane * kWave; WIDE && e0 < lds_n; e0 += kPerLane * kWave) {
      write_back(e0, false);
      __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);  // none of these passes' loads stays pending into the next tile
    }
    __syncthreads();
    t = tn;
    tl = tl_next;
  }
}

// Sketch::update over a batch of indices of one sketch (row 0 of slab).  All waves of a workgroup XOR
// into one LDS delta of `depth` records per column (odd, so columns start in different banks) and the
// workgroups add theirs to the row with device-scope atomics, so a record takes one atomic per
// workgroup where the tiles of 1024 indices, each with its own delta, took one per tile on 2700
// words and one per deep pair.  A lane keeps its index and takes the columns one after the other from
// a column of its own on, which spreads a step's 64 lanes over the columns.  VALU-bound like the long
// tiles of k_update_tiles: 4.19M indices of 25 columns 446 -> 113 us.
// SPLIT (batches that leave lanes of one workgroup idle): 2^sub lanes share an index and take every
// 2^sub-th column, where one lane's walk through all columns was most of the kernel: a call with one index
// of 30, 160 and 300 columns 21, 49 and 68 us -> 16, 17 and 17 (tiles of a wave each: 20, 25 and 32), 48
// indices of 300 columns 22 (82 by tiles).
constexpr uint32_t kOneBlock = 1024, kOneGrid = 512;
constexpr uint32_t kOneDepth = 17, kOneMaxCols = 160;  // deltas of kOneDepth records up to this many columns
template <class G, bool SPLIT>
__global__ void __launch_bounds__(kOneBlock, 8)
k_sketch_update(const uint64_t* __restrict__ idxs, size_t count, unsigned char* __restrict__ slab, Geo g,
                const uint64_t* __restrict__ col_bf, uint32_t depth, uint32_t sub) {
  extern __shared__ __align__(16) unsigned char smem[];
  const uint32_t C = g.C, D = g.D, lds_n = C * depth + 1, lds_d = D < depth ? D : depth;
  uint64_t* s_bf = reinterpret_cast<uint64_t*>(smem);  // spread bitflips
  uint64_t* s_a = s_bf + C;
  G* s_g = reinterpret_cast<G*>(s_a + lds_n);
  for (uint32_t i = threadIdx.x; i < C; i += blockDim.x) s_bf[i] = xxh3_spread(col_bf[i]);
  for (uint32_t i = threadIdx.x; i < lds_n; i += blockDim.x) {
    s_a[i] = 0;
    s_g[i] = 0;
  }
  __syncthreads();
  const uint64_t chk_sbf = xxh3_spread(g.chk_bf), depth_cap = 1ull << D;
  const uint32_t near_cap = 1u << depth;
  uint64_t det_a = 0;
  G det_g = 0;
  auto add = [&](uint64_t sp, uint32_t c, uint64_t idx, G chk) {
    const uint64_t x = sp ^ s_bf[c];
    const uint32_t low = hash_low28(x);
    const uint32_t near = (uint32_t)__builtin_ctz(low | near_cap);
    if (near < lds_d) {
      const uint32_t e = mad24(c, depth, near);
      lds_xor(s_a + e, idx);
      lds_xor(s_g + e, chk);
    } else {
      const uint32_t d = bucket_depth(low, x, depth_cap);
      if (d < D) {
        xor_rec_atomic<G>(slab + rec_col_off<G>(g, c, d), idx, chk);
        if (kDeepFlags<G> && rec_is_deep(g, d)) st_rlx(reinterpret_cast<uint32_t*>(slab + deep_flag_off(c)), 1u);
      }
    }
  };
  const size_t lanes = SPLIT ? count << sub : count;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < lanes; i += (size_t)gridDim.x * blockDim.x) {
    const uint64_t idx = idxs[SPLIT ? i >> sub : i];
    const uint64_t sp = xxh3_spread(xxh3_prep(idx));
    uint64_t ck = xxh3_products(sp ^ chk_sbf);
    ck ^= ck >> 28;
    const G chk = (G)ck;
    const uint32_t part = SPLIT ? (uint32_t)i & ((1u << sub) - 1) : 0u;
    if (part == 0) {
      det_a ^= idx;
      det_g ^= chk;
    }
    if (SPLIT) {
      for (uint32_t c = part; c < C; c += 1u << sub) add(sp, c, idx, chk);
      continue;
    }
    uint32_t c = lane_id() % C;
    for (uint32_t k = 0; k < C; ++k) {
      add(sp, c, idx, chk);
      ++c;
      c = c < c - C ? c : c - C;  // C - C, or c - C below zero
    }
  }
  // lanes past the end hold zeros, and every lane is active again
  const uint64_t da = wave_xor_dpp_u64(det_a);
  const G dg = sizeof(G) == 4 ? (G)wave_xor_dpp_u32((uint32_t)det_g) : (G)wave_xor_dpp_u64((uint64_t)det_g);
  if (lane_id() == 0) {
    lds_xor(s_a + lds_n - 1, da);
    lds_xor(s_g + lds_n - 1, dg);
  }
  __syncthreads();
  for (uint32_t e = threadIdx.x; e < lds_n; e += blockDim.x) {
    const uint64_t a = s_a[e];
    const G gm = s_g[e];
    if ((a | (uint64_t)gm) == 0) continue;  // also the entries at depth >= D
    const uint32_t c = e / depth, d = e - c * depth;
    const bool det = e == lds_n - 1;
    xor_rec_atomic<G>(slab + (det ? det_col_off(g) : rec_col_off<G>(g, c, d)), a, gm);
    if (kDeepFlags<G> && !det && rec_is_deep(g, d)) st_rlx(reinterpret_cast<uint32_t*>(slab + deep_flag_off(c)), 1u);
  }
}

// ================================================================================================
// Grouping a stream of (src,dst) pairs by vertex: the device form of the reference's gutters
// (both directions of every update, include/graph_sketch_driver.h:171-172).
// ================================================================================================
// Pairs naming a vertex >= n are skipped by every kernel and reported through bad_flag.
__global__ void k_count_pairs(const uint2* __restrict__ pairs, size_t count, uint32_t n, uint32_t* __restrict__ cnt,
                              uint32_t* __restrict__ bad_flag) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    const uint2 p = pairs[i];
    if (p.x >= n || p.y >= n) {
      st_rlx(bad_flag, 1u);
      continue;
    }
    atomicAdd(cnt + p.x, 1u);
    atomicAdd(cnt + p.y, 1u);
  }
}
__global__ void k_scatter_pairs(const uint2* __restrict__ pairs, size_t count, uint32_t n,
                                uint32_t* __restrict__ cursor, uint32_t* __restrict__ dst_arr) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    const uint2 p = pairs[i];
    if (p.x >= n || p.y >= n) continue;
    const uint32_t pu = atomicAdd(cursor + p.x, 1u);
    dst_arr[pu] = p.y;
    const uint32_t pv = atomicAdd(cursor + p.y, 1u);
    dst_arr[pv] = p.x;
  }
}

// Exclusive scan of per-vertex counts (and of per-vertex tile counts ceil(cnt/tile) when tile>0),
// packed as (tiles << 32 | cnt) in one u64 so a single pass scans both.
constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;
constexpr uint32_t kScanSpan = kScanBlock * kScanItems;

// Tiles of c destinations; almost every vertex has at most one, which spares the division's ~40
// instructions.
__device__ inline uint32_t tile_count(uint32_t c, uint32_t tile) {
  return c <= tile ? (c != 0 ? 1u : 0u) : (c - 1) / tile + 1;
}
__device__ inline uint64_t pack_ct(uint32_t c, uint32_t tile) { return ((uint64_t)tile_count(c, tile) << 32) | c; }
__device__ inline uint64_t block_excl_scan_u64(uint64_t x, uint64_t* total) {
  __shared__ uint64_t wsum[kScanBlock / kWave];
  const uint32_t lane = lane_id(), wid = threadIdx.x / kWave;
  const uint64_t incl = wave_incl_scan_u64(x);
  if (lane == kWave - 1) wsum[wid] = incl;
  __syncthreads();
  uint64_t pre = 0, tot = 0;
  for (uint32_t w = 0; w < kScanBlock / kWave; ++w) {
    if (w < wid) pre += wsum[w];
    tot += wsum[w];
  }
  __syncthreads();
  *total = tot;
  return pre + incl - x;
}
__global__ void __launch_bounds__(kScanBlock)
k_scan_partials(const uint32_t* __restrict__ cnt, uint32_t n, uint32_t tile, uint64_t* __restrict__ partials) {
  const uint32_t base = blockIdx.x * kScanSpan + threadIdx.x * kScanItems;
  uint64_t s = 0;
  for (int k = 0; k < kScanItems; ++k) {
    const uint32_t i = base + k;
    if (i < n) s += pack_ct(cnt[i], tile);
  }
  uint64_t tot;
  block_excl_scan_u64(s, &tot);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}
__global__ void __launch_bounds__(kScanBlock)
k_scan_block_sums(uint64_t* __restrict__ partials, uint32_t nparts, uint32_t n, uint32_t* __restrict__ off,
                  uint32_t* __restrict__ toff, uint32_t* __restrict__ totals) {
  const uint32_t per = (nparts + kScanBlock - 1) / kScanBlock;
  const uint32_t b0 = threadIdx.x * per;
  uint64_t s = 0;
  for (uint32_t k = 0; k < per; ++k)
    if (b0 + k < nparts) s += partials[b0 + k];
  uint64_t tot;
  uint64_t run = block_excl_scan_u64(s, &tot);
  for (uint32_t k = 0; k < per; ++k)
    if (b0 + k < nparts) {
      const uint64_t v = partials[b0 + k];
      partials[b0 + k] = run;
      run += v;
    }
  if (threadIdx.x == 0) {
    totals[0] = (uint32_t)tot;
    totals[1] = (uint32_t)(tot >> 32);
    off[n] = (uint32_t)tot;
    if (toff) toff[n] = (uint32_t)(tot >> 32);
  }
}
__global__ void __launch_bounds__(kScanBlock)
k_scan_apply(const uint32_t* __restrict__ cnt, uint32_t n, uint32_t tile, const uint64_t* __restrict__ partials,
             uint32_t* __restrict__ off, uint32_t* __restrict__ toff, uint32_t* __restrict__ cursor) {
  const uint32_t base = blockIdx.x * kScanSpan + threadIdx.x * kScanItems;
  uint32_t c[kScanItems];
  uint64_t s = 0;
  for (int k = 0; k < kScanItems; ++k) {
    const uint32_t i = base + k;
    c[k] = i < n ? cnt[i] : 0;
    s += pack_ct(c[k], tile);
  }
  uint64_t tot;
  uint64_t run = block_excl_scan_u64(s, &tot) + partials[blockIdx.x];
  for (int k = 0; k < kScanItems; ++k) {
    const uint32_t i = base + k;
    if (i < n) {
      off[i] = (uint32_t)run;
      if (toff) toff[i] = (uint32_t)(run >> 32);
      if (cursor) cursor[i] = (uint32_t)run;
    }
    run += pack_ct(c[k], tile);
  }
}
// Also accumulates, when acc is given, the flush's algorithmic bytes (sum over vertices of
// 4k + 2*min(S, k*(C+1)*B)) into acc[blockIdx.x]: one slot per block, so no atomics; the grid
// never exceeds kProfSlots blocks and launches on one stream are ordered.
__global__ void __launch_bounds__(256)
k_make_tiles(const uint32_t* __restrict__ cnt, const uint32_t* __restrict__ off, const uint32_t* __restrict__ toff,
             uint32_t n, uint32_t tile, Tile* __restrict__ tiles, uint64_t* __restrict__ acc, uint64_t S,
             uint64_t per_update) {
  uint64_t bytes = 0;
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
    const uint32_t c = cnt[v];
    if (!c) continue;
    const uint64_t touched = (uint64_t)c * per_update;
    bytes += 4ull * c + 2 * (touched < S ? touched : S);
    const uint32_t nt = (c + tile - 1) / tile, o = off[v], t0 = toff[v];
    for (uint32_t j = 0; j < nt; ++j) {
      const uint32_t b = j * tile;
      tiles[t0 + j] = Tile{v, o + b, (c - b) < tile ? (c - b) : tile, nt > 1 ? 1u : 0u};
    }
  }
  if (!acc) return;  // uniform over the grid
  __shared__ uint64_t s_part[256 / kWave];
  for (int o = 32; o > 0; o >>= 1) bytes += shfl_xor_u64(bytes, o);
  if (lane_id() == 0) s_part[threadIdx.x / kWave] = bytes;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t t = 0;
    for (int w = 0; w < 256 / kWave; ++w) t += s_part[w];
    acc[blockIdx.x] += t;
  }
}

// Grouping by vertex without device-scope atomics per update (vertex counts up to 2^24): a bucket
// partition over bins of 2^shift vertices, then one workgroup per bin.
//   1. k_part_hist: each workgroup takes a contiguous chunk of the pairs and counts the directed
//      entries per bin in LDS; one device atomic per (workgroup, bin) gives its place in the bin.
//   2. k_part_scatter: the same chunks again; LDS cursors place the records in bin order.
//   3. k_part_group: one workgroup per bin counts its vertices' entries in LDS, scans them, writes
//      each vertex's destinations contiguously and its tiles (the bin's share of the tile list taken
//      with one device atomic).  The order of one vertex's destinations, and of the tiles, is
//      arbitrary, which XOR does not see.
// Bound by the scattered record writes (k_part_scatter: a workgroup's run in a bin is a few lines) and,
// for small flushes, by the launches' latency.  With the direct writes alone, against contiguous ranges of ids, 8-byte records, a
// count matrix with two scan launches and a per-vertex scan for the tiles (7 launches): 24M Chung-Lu
// updates on 2^18 vertices 1025 -> 777 us, 16M R-MAT on 2^20 2190 -> 504 us (one range held 4% of the
// entries), flushes of about 730k updates of a serving trace 87 -> 35 us.
// A vertex's place p is its id times an odd number modulo 2^nb (a bijection), and its bin the high
// bits of p: streams whose busy vertices sit side by side (R-MAT: the 256 lowest of 2^20 ids take 4% of
// all entries) spread over the bins.  A record holds the place within the bin and the other end in
// one word when both fit (PACK: nb + shift <= 32), else in two.
constexpr uint32_t kPartBins = 1024, kPartBlock = 1024, kPartMaxBlocks = 256, kPartMaxShift = 14;
constexpr uint32_t kPlaceMul = 2654435761u;  // odd, near 2^32 / the golden ratio
constexpr uint32_t inverse_odd(uint32_t m) {  // Newton: each step doubles the correct low bits
  uint32_t x = m;
  for (int k = 0; k < 5; ++k) x *= 2u - m * x;
  return x;
}
constexpr uint32_t kPlaceInv = inverse_odd(kPlaceMul);
static_assert(kPlaceMul * kPlaceInv == 1u, "inverse modulo 2^32");

template <bool PACK>
struct PartRec {
  using T = uint32_t;
  static __device__ inline T make(uint32_t local, uint32_t other, uint32_t nb) { return (local << nb) | other; }
  static __device__ inline uint32_t local(T r, uint32_t nb) { return r >> nb; }
  static __device__ inline uint32_t other(T r, uint32_t nb) { return r & ((1u << nb) - 1); }
};
template <>
struct PartRec<false> {
  using T = uint2;
  static __device__ inline T make(uint32_t local, uint32_t other, uint32_t) { return make_uint2(local, other); }
  static __device__ inline uint32_t local(T r, uint32_t) { return r.x; }
  static __device__ inline uint32_t other(T r, uint32_t) { return r.y; }
};

__device__ inline void part_chunk(size_t count, uint32_t nblk, size_t* lo, size_t* hi) {
  const size_t per = (count + nblk - 1) / nblk;
  *lo = (size_t)blockIdx.x * per < count ? (size_t)blockIdx.x * per : count;
  *hi = *lo + per < count ? *lo + per : count;
}
// Calls f(pair) for the thread's pairs of [lo, hi), four loads in flight.
template <class F>
__device__ inline void part_walk(const uint2* __restrict__ pairs, size_t lo, size_t hi, F&& f) {
  constexpr uint32_t U = 4;
  size_t k = lo + threadIdx.x;
  for (; k + (U - 1) * kPartBlock < hi; k += U * kPartBlock) {
    uint2 p[U];
#pragma unroll
    for (uint32_t j = 0; j < U; ++j) p[j] = pairs[k + j * kPartBlock];
#pragma unroll
    for (uint32_t j = 0; j < U; ++j) f(p[j]);
  }
  for (; k < hi; k += kPartBlock) f(pairs[k]);
}
// Exclusive scan over a workgroup of kPartBlock threads.
__device__ inline uint64_t part_scan(uint64_t x, uint64_t* wsum, uint64_t* total) {
  const uint32_t lane = lane_id(), wid = threadIdx.x / kWave;
  const uint64_t incl = wave_incl_scan_u64(x);
  if (lane == kWave - 1) wsum[wid] = incl;
  __syncthreads();
  uint64_t pre = 0, tot = 0;
  for (uint32_t w = 0; w < kPartBlock / kWave; ++w) {
    const uint64_t v = wsum[w];
    if (w < wid) pre += v;
    tot += v;
  }
  *total = tot;
  return pre + incl - x;
}

// binned: entries per bin, all zero on entry (k_part_group clears them); place: the workgroup's first
// slot within each bin.  Also clears the tile count for k_part_group.
__global__ void __launch_bounds__(kPartBlock)
k_part_hist(const uint2* __restrict__ pairs, size_t count, uint32_t n, uint32_t nb, uint32_t shift, uint32_t bins,
            uint32_t nblk, uint32_t* __restrict__ binned, uint32_t* __restrict__ place,
            uint32_t* __restrict__ totals, uint32_t* __restrict__ bad_flag) {
  __shared__ uint32_t h[kPartBins];
  for (uint32_t b = threadIdx.x; b < bins; b += kPartBlock) h[b] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) totals[1] = 0;
  __syncthreads();
  size_t lo, hi;
  part_chunk(count, nblk, &lo, &hi);
  const uint32_t mask = (1u << nb) - 1;
  part_walk(pairs, lo, hi, [&](uint2 p) {
    if (p.x >= n || p.y >= n) {
      st_rlx(bad_flag, 1u);
      return;
    }
    atomicAdd(h + (((p.x * kPlaceMul) & mask) >> shift), 1u);
    atomicAdd(h + (((p.y * kPlaceMul) & mask) >> shift), 1u);
  });
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < bins; b += kPartBlock) {
    const uint32_t c = h[b];
    place[(size_t)blockIdx.x * bins + b] = c ? atomicAdd(binned + b, c) : 0u;
  }
}

// Large flushes move their records through LDS: a workgroup sorts a tile of up to kTile records by
// bin there and writes each bin's records as one run, where single records written straight to their
// places kept 256 * 1024 partly filled lines open, which were evicted from the L2s before they filled.
// 24M Chung-Lu updates on 2^18 vertices 450 -> 168 us, 16M R-MAT on 2^20 298 -> 115 us.  (2048 bins: 215
// and 154, which the group kernel wins back on the first only, 293 -> 231 and 178 -> 187 us.)
template <class T>
struct StageLds {
  static constexpr uint32_t kTile = sizeof(T) == 4 ? 16384 : 8192, kPer = kTile / kPartBlock;
  uint32_t* cnt;    // kPartBins: records per key in the tile
  uint32_t* first;  // kPartBins: a key's first record in the sorted tile
  T* item;          // kTile
  uint16_t* key;    // kTile
  uint64_t* wsum;
  static constexpr size_t bytes() { return 2 * 4 * kPartBins + kTile * (sizeof(T) + 2); }
  __device__ StageLds(unsigned char* p, uint64_t* w) : wsum(w) {
    cnt = reinterpret_cast<uint32_t*>(p);
    first = cnt + kPartBins;
    item = reinterpret_cast<T*>(first + kPartBins);
    key = reinterpret_cast<uint16_t*>(item + kTile);
  }
  // Writes the workgroup's records r[j] with k[j] < kPartBins (others are left out) to out[cur[key]...]
  // and moves the cursors on.  cur: kPartBins words in LDS.
  __device__ void write(const T* r, const uint32_t* k, uint32_t* cur, T* __restrict__ out) {
    constexpr uint32_t M = kPartBins / kPartBlock;  // keys of a thread
    const uint32_t t = threadIdx.x;
    __syncthreads();  // the previous tile's reads are done, and cur is written
#pragma unroll
    for (uint32_t j = 0; j < M; ++j) cnt[M * t + j] = 0;
    __syncthreads();
    uint32_t rank[kPer];
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) rank[j] = k[j] < kPartBins ? atomicAdd(cnt + k[j], 1u) : 0u;
    __syncthreads();
    uint32_t c[M], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < M; ++j) {
      c[j] = cnt[M * t + j];
      sum += c[j];
    }
    uint64_t total;
    const uint32_t f = (uint32_t)part_scan(sum, wsum, &total);
    for (uint32_t j = 0, at = f; j < M; at += c[j], ++j) first[M * t + j] = at;
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j)
      if (k[j] < kPartBins) {
        const uint32_t at = first[k[j]] + rank[j];
        item[at] = r[j];
        key[at] = (uint16_t)k[j];
      }
    __syncthreads();
    for (uint32_t j = 0, at = f; j < M; at += c[j], ++j) {
      first[M * t + j] = cur[M * t + j] - at;  // a record's place is its place in the tile plus its key's base
      cur[M * t + j] += c[j];
    }
    __syncthreads();
    for (uint32_t i = t; i < (uint32_t)total; i += kPartBlock) out[first[key[i]] + i] = item[i];
  }
};

// binoff: bins + 1 words, the bins' starts in the record list.  STAGED: through LDS (StageLds).
template <bool PACK, bool STAGED>
__global__ void __launch_bounds__(kPartBlock)
k_part_scatter(const uint2* __restrict__ pairs, size_t count, uint32_t n, uint32_t nb, uint32_t shift, uint32_t bins,
               uint32_t nblk, const uint32_t* __restrict__ binned, const uint32_t* __restrict__ place,
               uint32_t* __restrict__ binoff, typename PartRec<PACK>::T* __restrict__ rec) {
  __shared__ uint32_t cur[kPartBins];
  __shared__ uint64_t wsum[kPartBlock / kWave];
  constexpr uint32_t M = kPartBins / kPartBlock;  // bins of a thread
  const uint32_t t = threadIdx.x;
  uint32_t c[M], pl[M], sum = 0;
#pragma unroll
  for (uint32_t j = 0; j < M; ++j) {
    const uint32_t b = M * t + j;
    c[j] = b < bins ? binned[b] : 0u;
    pl[j] = b < bins ? place[(size_t)blockIdx.x * bins + b] : 0u;
    sum += c[j];
  }
  uint64_t tot;
  uint32_t off = (uint32_t)part_scan(sum, wsum, &tot);
#pragma unroll
  for (uint32_t j = 0; j < M; ++j) {
    const uint32_t b = M * t + j;
    cur[b] = off + pl[j];
    if (blockIdx.x == 0 && b < bins) binoff[b] = off;
    off += c[j];
  }
  if (blockIdx.x == 0 && t == 0) binoff[bins] = (uint32_t)tot;
  __syncthreads();
  size_t lo, hi;
  part_chunk(count, nblk, &lo, &hi);
  const uint32_t mask = (1u << nb) - 1, lmask = (1u << shift) - 1;
  if constexpr (STAGED) {
    using R = typename PartRec<PACK>::T;
    extern __shared__ __align__(16) unsigned char smem[];
    StageLds<R> stage(smem, wsum);
    constexpr uint32_t P = StageLds<R>::kPer / 2;
    for (size_t k0 = lo; k0 < hi; k0 += P * kPartBlock) {  // uniform over the workgroup
      uint2 p[P];
#pragma unroll
      for (uint32_t j = 0; j < P; ++j) {
        const size_t k = k0 + j * kPartBlock + t;
        p[j] = k < hi ? pairs[k] : make_uint2(0xFFFFFFFFu, 0);
      }
      R r[2 * P];
      uint32_t key[2 * P];
#pragma unroll
      for (uint32_t j = 0; j < P; ++j) {
        const bool ok = p[j].x < n && p[j].y < n;
        const uint32_t px = (p[j].x * kPlaceMul) & mask, py = (p[j].y * kPlaceMul) & mask;
        r[2 * j] = PartRec<PACK>::make(px & lmask, p[j].y, nb);
        r[2 * j + 1] = PartRec<PACK>::make(py & lmask, p[j].x, nb);
        key[2 * j] = ok ? px >> shift : kPartBins;
        key[2 * j + 1] = ok ? py >> shift : kPartBins;
      }
      stage.write(r, key, cur, rec);
    }
    return;
  }
  part_walk(pairs, lo, hi, [&](uint2 p) {
    if (p.x >= n || p.y >= n) return;
    const uint32_t px = (p.x * kPlaceMul) & mask, py = (p.y * kPlaceMul) & mask;
    const uint32_t a = atomicAdd(cur + (px >> shift), 1u), b = atomicAdd(cur + (py >> shift), 1u);
    rec[a] = PartRec<PACK>::make(px & lmask, p.y, nb);
    rec[b] = PartRec<PACK>::make(py & lmask, p.x, nb);
  });
}

// Writes the tiles of a vertex with c destinations starting at o, from tile t0 on, and returns their
// algorithmic bytes (4c + 2 min(S, c * per_update)).
__device__ inline uint64_t write_tiles(uint32_t v, uint32_t o, uint32_t c, uint32_t tile, Tile* __restrict__ tiles,
                                       uint32_t t0, uint64_t S, uint64_t per_update) {
  const uint32_t nt = tile_count(c, tile);
  for (uint32_t j = 0; j < nt; ++j) {
    const uint32_t b = j * tile;
    tiles[t0 + j] = Tile{v, o + b, (c - b) < tile ? (c - b) : tile, nt > 1 ? 1u : 0u};
  }
  const uint64_t touched = (uint64_t)c * per_update;
  return 4ull * c + 2 * (touched < S ? touched : S);
}
// Adds a workgroup's profiling bytes to its slot of acc (nullptr: no profiling).
__device__ inline void add_bytes(uint64_t* acc, uint64_t bytes) {
  if (!acc) return;
  for (int o = 32; o > 0; o >>= 1) bytes += shfl_xor_u64(bytes, o);
  if (lane_id() == 0)
    atomicAdd(reinterpret_cast<unsigned long long*>(acc + blockIdx.x % kProfSlots), (unsigned long long)bytes);
}

template <bool PACK>
__global__ void __launch_bounds__(kPartBlock)
k_part_group(const typename PartRec<PACK>::T* __restrict__ rec, uint32_t nb, uint32_t shift,
             uint32_t* __restrict__ binned, const uint32_t* __restrict__ binoff, uint32_t* __restrict__ totals,
             uint32_t* __restrict__ dst_arr, uint32_t tile, Tile* __restrict__ tiles, uint64_t* __restrict__ acc,
             uint64_t S, uint64_t per_update) {
  extern __shared__ __align__(16) unsigned char smem[];
  uint32_t* lc = reinterpret_cast<uint32_t*>(smem);  // 2^shift counters, then cursors
  __shared__ uint64_t wsum[kPartBlock / kWave];
  __shared__ uint32_t s_tile0;
  const uint32_t b = blockIdx.x, R = 1u << shift, t = threadIdx.x;
  const uint32_t s = binoff[b], e = binoff[b + 1];
  if (t == 0) binned[b] = 0;
  if (s == e) return;  // uniform over the workgroup
  for (uint32_t k = t; k < R; k += kPartBlock) lc[k] = 0;
  // the first kKeep records of every thread stay in registers between the two passes
  constexpr uint32_t kKeep = 8;
  typename PartRec<PACK>::T keep[kKeep];
#pragma unroll
  for (uint32_t k = 0; k < kKeep; ++k)
    if (s + k * kPartBlock + t < e) keep[k] = rec[s + k * kPartBlock + t];
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < kKeep; ++k)
    if (s + k * kPartBlock + t < e) atomicAdd(lc + PartRec<PACK>::local(keep[k], nb), 1u);
  const uint32_t rest = s + kKeep * kPartBlock + t;
  for (uint32_t j = rest; j < e; j += kPartBlock) atomicAdd(lc + PartRec<PACK>::local(rec[j], nb), 1u);
  __syncthreads();
  // exclusive scan of the entries and tiles per vertex: thread t owns vertices t, t + 1024, ... (their
  // runs' order is free, and consecutive lanes read consecutive banks)
  uint64_t mine = 0;
  for (uint32_t k = t; k < R; k += kPartBlock) mine += pack_ct(lc[k], tile);
  uint64_t tot;
  uint64_t run = part_scan(mine, wsum, &tot);
  if (t == 0) s_tile0 = atomicAdd(totals + 1, (uint32_t)(tot >> 32));
  __syncthreads();
  const uint32_t t0 = s_tile0, pmask = (1u << nb) - 1;
  uint64_t bytes = 0;
  for (uint32_t k = t; k < R; k += kPartBlock) {
    const uint32_t c = lc[k];
    const uint32_t o = s + (uint32_t)run;
    if (c)
      bytes += write_tiles((((b << shift) | k) * kPlaceInv) & pmask, o, c, tile, tiles, t0 + (uint32_t)(run >> 32), S,
                           per_update);
    lc[k] = o;  // becomes the vertex's cursor
    run += pack_ct(c, tile);
  }
  add_bytes(acc, bytes);
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < kKeep; ++k)
    if (s + k * kPartBlock + t < e)
      dst_arr[atomicAdd(lc + PartRec<PACK>::local(keep[k], nb), 1u)] = PartRec<PACK>::other(keep[k], nb);
  for (uint32_t j = rest; j < e; j += kPartBlock) {
    const auto r = rec[j];
    dst_arr[atomicAdd(lc + PartRec<PACK>::local(r, nb), 1u)] = PartRec<PACK>::other(r, nb);
  }
}

// A flush of at most kSmallPairs updates in one workgroup, one launch instead of three: vertices are
// counted in an LDS hash table (2^tbits slots, at least 4/3 of the entries), whose scan gives the
// destinations' places and the tiles.  The limit is what 2^14 slots hold.  5000 updates: 29 us, where
// the seven launches took 50 us and their gaps; 1000 updates: 8 us against 38.
constexpr uint32_t kSmallPairs = 6144, kSmallPer = kSmallPairs / kPartBlock;
__global__ void __launch_bounds__(kPartBlock)
k_group_small(const uint2* __restrict__ pairs, uint32_t count, uint32_t n, uint32_t tbits, uint32_t* __restrict__ totals,
              uint32_t* __restrict__ dst_arr, uint32_t tile, Tile* __restrict__ tiles, uint64_t* __restrict__ acc,
              uint64_t S, uint64_t per_update, uint32_t* __restrict__ bad_flag) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ uint64_t wsum[kPartBlock / kWave];
  const uint32_t T = 1u << tbits, t = threadIdx.x;
  uint32_t* key = reinterpret_cast<uint32_t*>(smem);
  uint32_t* cnt = key + T;
  uint2 p[kSmallPer];
#pragma unroll
  for (uint32_t k = 0; k < kSmallPer; ++k) p[k] = k * kPartBlock + t < count ? pairs[k * kPartBlock + t] : make_uint2(0, 0);
  for (uint32_t k = t; k < T; k += kPartBlock) {
    key[k] = 0xFFFFFFFFu;  // no vertex: ids are below 2^31
    cnt[k] = 0;
  }
  __syncthreads();
  auto slot_of = [&](uint32_t v) -> uint32_t {
    uint32_t h = (v * kPlaceMul) >> (32 - tbits);
    while (true) {
      const uint32_t prev = atomicCAS(key + h, 0xFFFFFFFFu, v);
      if (prev == 0xFFFFFFFFu || prev == v) return h;
      h = (h + 1) & (T - 1);
    }
  };
  uint32_t sx[kSmallPer], sy[kSmallPer], ox[kSmallPer], oy[kSmallPer];
#pragma unroll
  for (uint32_t k = 0; k < kSmallPer; ++k) {
    sx[k] = 0xFFFFFFFFu;
    if (k * kPartBlock + t >= count) continue;
    if (p[k].x >= n || p[k].y >= n) {
      st_rlx(bad_flag, 1u);
      continue;
    }
    sx[k] = slot_of(p[k].x);
    sy[k] = slot_of(p[k].y);
    ox[k] = atomicAdd(cnt + sx[k], 1u);
    oy[k] = atomicAdd(cnt + sy[k], 1u);
  }
  __syncthreads();
  uint64_t mine = 0;
  for (uint32_t k = t; k < T; k += kPartBlock) mine += pack_ct(cnt[k], tile);
  uint64_t tot;
  uint64_t run = part_scan(mine, wsum, &tot);
  uint64_t bytes = 0;
  for (uint32_t k = t; k < T; k += kPartBlock) {
    const uint32_t c = cnt[k];
    if (c) bytes += write_tiles(key[k], (uint32_t)run, c, tile, tiles, (uint32_t)(run >> 32), S, per_update);
    cnt[k] = (uint32_t)run;
    run += pack_ct(c, tile);
  }
  if (t == 0) totals[1] = (uint32_t)(tot >> 32);
  add_bytes(acc, bytes);
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < kSmallPer; ++k) {
    if (sx[k] == 0xFFFFFFFFu) continue;
    dst_arr[cnt[sx[k]] + ox[k]] = p[k].y;
    dst_arr[cnt[sy[k]] + oy[k]] = p[k].x;
  }
}

void scan_counts(const uint32_t* cnt, uint32_t n, uint32_t tile, uint64_t* partials, uint32_t* off, uint32_t* toff,
                 uint32_t* cursor, uint32_t* totals, hipStream_t s) {
  const uint32_t nparts = (n + kScanSpan - 1) / kScanSpan;
  hipLaunchKernelGGL(k_scan_partials, dim3(nparts), dim3(kScanBlock), 0, s, cnt, n, tile, partials);
  hipLaunchKernelGGL(k_scan_block_sums, dim3(1), dim3(kScanBlock), 0, s, partials, nparts, n, off, toff, totals);
  hipLaunchKernelGGL(k_scan_apply, dim3(nparts), dim3(kScanBlock), 0, s, cnt, n, tile, partials, off, toff, cursor);
}

inline uint32_t grid_for(size_t work, uint32_t block, uint32_t cap = 8192) {
  size_t g = (work + block - 1) / block;
  if (g < 1) g = 1;
  return (uint32_t)(g < cap ? g : cap);
}

// ================================================================================================
// Eager DSU over a batch of updates (pre_insert, src/cc_sketch_alg.cpp:79-104), in three phases
// separated by kernel boundaries:
//   1. every update attempts the CAS union of its endpoints; winners are marked merged;
//   2. merged edges are inserted into the spanning-forest set;
//   3. an update that did not merge and whose edge is in the forest invalidates the DSU.
// The outcome equals the reference's for the linearisation the CAS order defines (the
// reference's stream threads are concurrent as well): a deleted forest edge always invalidates,
// and any edge that merged and occurs again in the batch invalidates.
// ================================================================================================
// Rank classes for a batch on an instance that no query has ranked yet (RoundBufs::hint): every
// update draws a level that is l or more with probability 2^-l, and a vertex's class is the highest
// level among its updates, about the logarithm of its degree in the batch.  Plain stores race, which
// can only lose a level: any classes give the same components.
__global__ void k_eager_rank(const uint2* __restrict__ pairs, size_t count, uint32_t n, unsigned char* hint) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    const unsigned char level = (unsigned char)__builtin_ctzll(mix64(i) | (1ull << 40));
    if (level == 0) continue;
    const uint2 p = pairs[i];
    if (p.x >= n || p.y >= n) continue;
    if (hint[p.x] < level) hint[p.x] = level;
    if (hint[p.y] < level) hint[p.y] = level;
  }
}

// A bit per vertex: whether it is in the largest component, as far as 64 sampled vertices name it (any
// component would do).  No links run beside this kernel.
__global__ void __launch_bounds__(256)
k_dsu_map(DsuDev d, uint64_t* __restrict__ map) {
  __shared__ uint32_t s_root;
  if (ld_acq(d.flags + kFlagEagerInvalid)) return;
  if (threadIdx.x < kWave) {
    const uint32_t r = dsu_find_stable(d.parent, (uint32_t)(mix64(threadIdx.x) % d.n));
    uint32_t best = 0, most = 0;
    for (int l = 0; l < kWave; ++l) {
      const uint32_t c = rd_lane_u32(r, l), m = (uint32_t)__popcll(__ballot(r == c));
      if (m > most) {
        most = m;
        best = c;
      }
    }
    if (threadIdx.x == 0) s_root = best;
  }
  __syncthreads();
  const uint32_t v = blockIdx.x * 256 + threadIdx.x;
  const uint64_t in = __ballot(v < d.n && dsu_find_stable(d.parent, v < d.n ? v : 0) == s_root);
  if (lane_id() == 0 && v < d.n) map[v / kWave] = in;
}

// src != pairs: the batch is also copied from src into pairs (the staging buffer) on the way, so
// ingesting device pairs needs no separate copy launch; the copy happens whether or not the DSU
// is still valid.
// build_sf: the first batch after a query also fills the forest membership set from the query's
// forest edges (sf_edge) -- lock-free inserts like this batch's own, so the two need no order.
// MAP: an update with both ends in map's component is known to be connected, whatever this batch links,
// from two LDS reads; a graph's component bits fit LDS where its parents, read at random, take two L2
// requests per update at least.
template <bool MAP>
__global__ void k_eager_union(const uint2* __restrict__ src, uint2* __restrict__ pairs, size_t count,
                              uint8_t* __restrict__ merged, DsuDev d, uint32_t build_sf,
                              const unsigned char* __restrict__ hint, const uint32_t* __restrict__ map) {
  extern __shared__ uint32_t s_map[];
  const bool live = !ld_acq(d.flags + kFlagEagerInvalid);
  if (!live && src == pairs) return;
  if (MAP && live) {  // uniform: nothing sets the flag beside this kernel
    for (uint32_t w = threadIdx.x; w < (d.n + 31) / 32; w += blockDim.x) s_map[w] = map[w];
    __syncthreads();
  }
  if (build_sf && live)
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < d.n; v += gridDim.x * blockDim.x) {
      const uint64_t e = d.sf_edge[v];
      if (e != kEmpty) sf_insert(d, e);
    }
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    const uint2 p = src[i];
    if (src != pairs) pairs[i] = p;
    if (!live) continue;
    if (p.x >= d.n || p.y >= d.n) {
      merged[i] = 0;
      st_rlx(d.flags + kFlagBadInput, 1u);
      continue;
    }
    if (MAP && (s_map[p.x / 32] >> (p.x % 32)) & (s_map[p.y / 32] >> (p.y % 32)) & 1u) {
      merged[i] = 0;
      continue;
    }
    const uint32_t child = dsu_link<true>(d.parent, p.x, p.y, d.prio_seed, hint);
    merged[i] = child != kNoLink ? 1 : 0;
    if (child != kNoLink) {
      const uint64_t key = concat_pairing(p.x, p.y);
      d.sf_edge[child] = key;
      sf_insert(d, key);  // into the forest set; the deletion check runs once the whole batch is merged
    }
  }
}
__global__ void k_eager_sf_check(const uint2* __restrict__ pairs, size_t count, const uint8_t* __restrict__ merged,
                                 DsuDev d) {
  // One deleted forest edge decides the whole batch, so every wave looks at the flag before each of
  // its steps and stops once it is set.  Bound by the probes of the forest set when nothing is
  // deleted; with deletes, every hit used to store the flag over the bus and fence the system, which
  // serialised them: 24M updates, half of them deletes, went from 1950 to 20 us.
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    if (ld_acq(d.flags + kFlagEagerInvalid)) return;
    if (merged[i]) continue;
    const uint2 p = pairs[i];
    if (p.x == p.y || p.x >= d.n || p.y >= d.n) continue;
    if (sf_contains(d, concat_pairing(p.x, p.y)) && !ld_acq(d.flags + kFlagEagerInvalid)) {
      st_rlx(d.flags + kFlagEagerInvalid, 1u);  // same value from every writer
      // lets the host stop launching eager batches without a synchronisation
      if (d.inv_mirror) __hip_atomic_store(d.inv_mirror, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// ================================================================================================
// Borůvka (boruvka_emulation, src/cc_sketch_alg.cpp:464-513)
// ================================================================================================


// Round 0 (run_round_zero, 223-244): every vertex samples column 0 of its own sketch
// (Sketch::sample, src/sketch.cpp:94-116).  A wave takes four vertices in groups of 16 lanes: lane
// 16j + i (i < 15) checks depth i of vertex v0 + j and lane 16j + 15 its deterministic bucket, so
// one hash per lane serves four vertices.  The first good depth of a vertex is almost always below
// 15 (a bucket at depth d holds about deg / 2^(d+1) edges); a vertex with no good bucket there
// (very high degree, or none at all) is finished by the whole wave over depths 15..D-1.
template <class G>
__global__ void __launch_bounds__(256)
k_sample_round0(const unsigned char* __restrict__ slab, Geo g, uint64_t* __restrict__ samp,
                uint32_t* __restrict__ flags, unsigned char* __restrict__ det_cpy, unsigned char* __restrict__ hint,
                DsuDev d) {
  constexpr uint32_t V = 4, GL = kWave / V, GD = GL - 1;  // vertices per wave, lanes per vertex, depths
  constexpr uint32_t RB = 8 + sizeof(G);
  // Round-0 hooking: every vertex is a root when round 0 begins, and only its own thread would link
  // it under a higher-ranked vertex, so a sampled edge (v, u) whose other end u ranks above v
  // (priority, then the smaller id) is merged here with plain stores -- v under u, parents always
  // ranking higher, so the forest stays acyclic.  The other samples wait in samp for
  // k_apply_samples, which links them with the CAS union.
  bool hooked = false;
  auto put = [&](uint32_t v, uint64_t rec) {
    if (rec < kSampFail) {  // a GOOD sample: an edge index with both ends below n
      const uint32_t x = (uint32_t)(rec >> 32), y = (uint32_t)rec;
      const uint32_t u = x == v ? y : x;
      if ((x == v || y == v) && u != v) {
        const uint32_t pv = dsu_prio(v, d.prio_seed), pu = dsu_prio(u, d.prio_seed);
        if (pu > pv || (pu == pv && u < v)) {
          d.parent[v] = u;
          d.sf_edge[v] = rec;  // the forest edge, in the slot of the root it linked
          samp[v] = kSampZero;
          hooked = true;
          return;
        }
      }
    }
    samp[v] = rec;
  };
  if (ld_acq(d.flags + kFlagSkip)) return;  // the query keeps the eager DSU
  const uint32_t lane = lane_id(), i = lane % GL, base = lane - i;
  const uint32_t nd = g.D < GD ? g.D : GD;  // depths checked in the grouped pass
  const uint32_t waves = (gridDim.x * blockDim.x) / kWave;
  for (uint32_t v0 = (blockIdx.x * blockDim.x + threadIdx.x) / kWave * V; v0 < g.n; v0 += waves * V) {
    const uint32_t v = v0 + lane / GL;
    uint64_t a = 0;
    G gm = 0;
    const bool live = v < g.n && (i < nd || i == GD);
    if (live) ld_rec<G>(slab + (size_t)v * g.row + (i == GD ? det_col_off(g) : rec_col_off<G>(g, 0, i)), &a, &gm);
    const uint64_t mask = __ballot(live && (G)xxh3_mix(xxh3_prep(a), g.chk_bf) == gm);
    const uint32_t gmask = (uint32_t)(mask >> base) & ((1u << GL) - 1);
    const uint32_t colm = gmask & ((1u << nd) - 1);
    // degree class: one past the deepest nonzero bucket among the grouped depths (a bucket at depth
    // d is nonzero about when the degree reaches 2^d)
    const uint64_t nzm = __ballot(live && i < nd && (a | (uint64_t)gm) != 0);
    const uint32_t gnz = (uint32_t)(nzm >> base) & ((1u << nd) - 1);
    // every lane takes part in the shuffles; lane i == 0 of a group decides
    const uint64_t det_a = shfl_u64(a, (int)(base + GD));
    const G det_g = (G)shfl_u64((uint64_t)gm, (int)(base + GD));
    const uint64_t col_a = shfl_u64(a, (int)(base + (colm ? __builtin_ctz(colm) : 0)));
    bool undecided = false;
    if (i == 0 && v < g.n) {
      hint[v] = (unsigned char)(gnz ? 32 - __builtin_clz(gnz) : 0);
      if (det_a == 0 && det_g == 0) samp[v] = gnz ? kSampZero : kSampEmpty;
      else if ((gmask >> GD) & 1) put(v, sample_record(kGood, det_a, g.n, flags));
      else if (colm) put(v, sample_record(kGood, col_a, g.n, flags));
      else if (g.D <= GD) samp[v] = kSampFail;
      else undecided = true;
    }
    // the deterministic bucket does not depend on the round: later rounds read this compact copy
    if (i == GD && v < g.n) st_rec<G>(det_cpy + (size_t)v * RB, a, gm);
    for (uint64_t und = __ballot(undecided); und; und &= und - 1) {  // uniform over the wave
      const uint32_t u = v0 + (uint32_t)__builtin_ctzll(und) / GL;
      const uint32_t dep = GD + lane;  // D - GD <= 64 lanes for every supported n
      uint64_t b = 0;
      G bg = 0;
      if (dep < g.D) ld_rec<G>(slab + (size_t)u * g.row + rec_col_off<G>(g, 0, dep), &b, &bg);
      const uint64_t m2 = __ballot(dep < g.D && (G)xxh3_mix(xxh3_prep(b), g.chk_bf) == bg);
      const uint64_t ia = m2 ? rd_lane_u64(b, __builtin_ctzll(m2)) : 0;
      if (lane == 0) put(u, m2 ? sample_record(kGood, ia, g.n, flags) : kSampFail);
    }
  }
  if (__ballot(hooked) && lane_id() == 0) d.mod[0] = 1;  // round 0 merged something
}

// The merge of a supernode's sample (sample_supernode, src/cc_sketch_alg.cpp:137-166): round 0's in
// k_apply_samples, one thread per vertex, the later rounds' where the sample is taken (k_bv_reduce,
// k_bv_finish).  The round is modified by a FAIL or a merge.  Links rank roots by the degree class
// round 0 recorded (hint), so hubs stay roots and absorb their neighbours without contention.
constexpr uint32_t kNoRoot = 0xFFFFFFFFu;  // no supernode (unused partial slot, no giant)

// Round state words (RoundBufs::totals).  A query starts with kStGiantFirst = kNoRoot.
//   kStSeg + 2(r & 1) entries regrouped in round r (the level-1 entry count, and the length of the
//                     active list of round r + 1)
//   kStGiantRound     root of this round's giant supernode, or kNoRoot
//   kStGiantFirst     the root elected giant first in this query (any member identifies the giant,
//                     which only grows), or kNoRoot
//   kStActMode        1 when this round walks the active list instead of every vertex
// Round 1 walks every vertex in id order.  Round r >= 2 walks the member list regrouped in round
// r - 1: every vertex outside the giant (all of them before one is elected), grouped by the
// previous round's roots, so the members of a new supernode mostly sit next to each other and a
// wave meets few distinct roots.  Vertices that joined the giant are dropped as they are met.
//   kStBest (u64)     before any giant: max over this round's roots holding >= n/kCandidateDiv
//                     vertices of (count << 32 | root); the next round excludes that supernode.
//                     The complement sum needs no majority -- any supernode's sum is the XOR of the
//                     vertices outside it -- so a large one can be left out a round early.
//   kStSeg + 2(r & 1) + 1  supernodes outside the giant in round r (entries of RoundBufs::segs[r & 1])
//   kStDropped        vertices of the supernodes taken out of the lists in this query (see k_bv_alloc)
// The two counts of one round parity share a 64-bit word, so a block takes its share of both with
// one atomic: entries at kStSeg + 2 * (r & 1), supernodes at kStSeg + 2 * (r & 1) + 1.
constexpr uint32_t kStGiantRound = 2, kStGiantFirst = 3, kStActMode = 4, kStBest = 6, kStSeg = 8;
constexpr uint32_t kStDropped = 12, kStWords = 13;
constexpr uint32_t kCandidateDiv = 32;
constexpr uint32_t kMaxStatRounds = 64;  // per round: vertices regrouped and the giant's root, then vertices dropped

// cnt / st (a query's start, or nullptr): the root counts are cleared too, and the round state
// words are set to their start values (no giant), so a query begins with one launch.
//
// force (a query's start, or nullptr): when it reads 0 and the eager DSU is still valid, the query
// keeps that DSU -- its answer is the cached one -- so the kernel only clears the round flags (every
// round kernel of the query then returns at once), sets the round state words to their start values
// and sets kFlagSkip.  The eager-invalid flag is only read here (every workgroup sees the same value)
// and is cleared by round 0 of a query that runs.
__global__ void k_dsu_reset(uint32_t* parent, uint32_t n, uint64_t* sf_hash, uint64_t sf_cap, uint64_t* sf_edge,
                            uint32_t* flags, uint32_t* mod, uint32_t nmod, uint32_t* cnt, uint32_t* st,
                            const uint32_t* force) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (force && !*force && !ld_acq(flags + kFlagEagerInvalid)) {
    if (t == 0) flags[kFlagSkip] = 1;
    for (size_t i = t; i < nmod; i += stride) mod[i] = 0;
    // The round kernels read their walk counts and member lists before they look at the round
    // flag, so the state words get their start values (empty walks) here as well.
    if (st && t < kStWords) st[t] = (t == kStGiantRound || t == kStGiantFirst) ? kNoRoot : 0u;
    return;
  }
  for (size_t i = t; i < n; i += stride) {
    parent[i] = (uint32_t)i;
    sf_edge[i] = kEmpty;
    if (cnt) cnt[i] = 0;
  }
  for (size_t i = t; i < sf_cap; i += stride) sf_hash[i] = kEmpty;
  // The bad-input flag is left alone: pairs grouped by the flush just before a query set it, and the
  // query's answer reports it (it is cleared where it is reported).  A query's reset leaves the
  // eager-invalid flag to round 0 (see above).
  if (t < kNumFlags && t != kFlagBadInput && !(force && t == kFlagEagerInvalid)) flags[t] = 0;
  for (size_t i = t; i < nmod; i += stride) mod[i] = 0;
  if (st && t < kStWords) st[t] = (t == kStGiantRound || t == kStGiantFirst) ? kNoRoot : 0u;
}

__device__ inline uint32_t walk_count(const uint32_t* st, uint32_t round, uint32_t n) {
  return round >= 2 ? st[kStSeg + 2 * ((round - 1) & 1)] : n;
}
__device__ inline uint32_t walk_vertex(const uint32_t* act_list, uint32_t round, uint32_t i) {
  return round >= 2 ? act_list[i] : i;
}

__device__ inline bool apply_sample(const DsuDev& d, uint64_t s, const unsigned char* hint) {
  if (s == kSampZero || s == kSampEmpty) return false;
  if (s == kSampFail) return true;
  const uint32_t a = (uint32_t)(s >> 32), b = (uint32_t)s;
  const uint32_t child = dsu_link(d.parent, a, b, d.prio_seed, hint);
  if (child == kNoLink) return false;
  // A merge records its edge in the spanning forest (cc_sketch_alg.cpp:152-162), in the slot of
  // the root it linked (every root is linked at most once between resets, so slots never
  // collide); the membership set the eager DSU uses is filled from these slots by the first eager
  // batch after the query (k_eager_union), off the merge's critical path.
  d.sf_edge[child] = a < b ? ((uint64_t)a << 32) | b : ((uint64_t)b << 32) | a;
  return true;
}

// The merges of round 0 that k_sample_round0 left in samp.  Nothing to do when the query keeps the
// eager DSU; else the DSU restarts valid.
__global__ void __launch_bounds__(256)
k_apply_samples(const uint64_t* __restrict__ samp, DsuDev d, const unsigned char* __restrict__ hint) {
  if (ld_acq(d.flags + kFlagSkip)) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) d.flags[kFlagEagerInvalid] = 0;
  bool modified = false;
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < d.n; v += gridDim.x * blockDim.x)
    if (apply_sample(d, samp[v], hint)) modified = true;
  if (__syncthreads_or(modified) && threadIdx.x == 0) d.mod[0] = 1;  // one plain store per block
}

// ---- rounds >= 1 (perform_boruvka_round 246-380 + create_merge_instructions 382-462) ----------
// Every kernel of round r first reads mod[r-1]: when round r-1 changed nothing the whole round is
// a no-op, which lets the host queue several rounds before it looks at the flags.
//
// Regrouping by root (round 1, every vertex): A) root of every vertex, members per root, and each
// vertex's place in its root's segment (the value its root's counter had when the vertex was
// counted); B) each root gets a contiguous segment [off, off+cnt) from one running cursor
// (contiguous, not in root order, which Borůvka does not need), and the round's segment list;
// C) every vertex to off[root] + its place.  Counts are aggregated per 1024-thread block in an LDS
// table first, so a root shared by the whole block costs one device atomic per block instead of
// one per wave or per vertex.
constexpr int kAggBlock = 1024;
constexpr uint32_t kAggTable = 2048;  // >= 2 * kAggBlock, power of two
constexpr uint32_t kEmptyKey = 0xFFFFFFFFu;

__device__ inline uint32_t lds_table_slot(uint32_t* keys, uint32_t key) {
  uint32_t h = (key * 2654435761u) & (kAggTable - 1);
  while (true) {
    const uint32_t prev = atomicCAS(keys + h, kEmptyKey, key);
    if (prev == kEmptyKey || prev == key) return h;
    h = (h + 1) & (kAggTable - 1);
  }
}

__global__ void __launch_bounds__(kAggBlock)
k_bv_find_count(uint32_t* __restrict__ parent, uint32_t n, uint2* __restrict__ nd, uint32_t* __restrict__ cnt,
                uint32_t* __restrict__ st, uint32_t round, const uint32_t* __restrict__ act_list,
                const uint32_t* __restrict__ prev_mod) {
  // The round flag is loaded together with the first reads (all in bounds whether or not the
  // round runs: counts and lists are those of an earlier round of this query), saving a round trip.
  const uint32_t live = ld_acq(prev_mod);
  uint32_t gfirst = st[kStGiantFirst];
  const uint64_t best = *reinterpret_cast<const uint64_t*>(st + kStBest);
  const uint32_t i = blockIdx.x * kAggBlock + threadIdx.x;
  const uint32_t walk = walk_count(st, round, n);
  const bool in_walk = i < walk;
  const uint32_t v = in_walk ? walk_vertex(act_list, round, i) : 0;
  // the grid covers n; blocks past the walk have nothing to count (block 0 writes the round state)
  if (!live || (blockIdx.x > 0 && blockIdx.x * kAggBlock >= walk)) return;
  __shared__ uint32_t t_key[kAggTable], t_cnt[kAggTable];
  for (uint32_t k = threadIdx.x; k < kAggTable; k += kAggBlock) {
    t_key[k] = kEmptyKey;
    t_cnt[k] = 0;
  }
  if (gfirst == kNoRoot && best) gfirst = (uint32_t)best;  // a candidate recorded by the previous round
  const bool act = gfirst != kNoRoot;
  const uint32_t gcur = act ? dsu_find_stable(parent, gfirst) : kNoRoot;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st[kStSeg + 2 * (round & 1)] = 0;
    st[kStSeg + 2 * (round & 1) + 1] = 0;
    st[kStGiantRound] = gcur;
    st[kStGiantFirst] = gfirst;
    st[kStActMode] = act ? 1u : 0u;
  }
  __syncthreads();
  __shared__ uint32_t t_base[kAggTable];
  uint32_t r = 0;
  if (in_walk) r = dsu_find_stable(parent, v);
  __syncthreads();
  // full path compression: every walked vertex now points at its root (no links in this kernel)
  if (in_walk) parent[v] = r;
  const bool active = in_walk && r != gcur;  // members of the giant are not counted
  // every lane inserts its root at once: LDS atomics absorb lanes that share a root, and no wave
  // walks its distinct roots one by one; the returned counts give each vertex its place in its
  // root's segment
  uint32_t my_slot = 0, my_pos = 0;
  if (active) {
    my_slot = lds_table_slot(t_key, r);
    my_pos = atomicAdd(t_cnt + my_slot, 1u);
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < kAggTable; k += kAggBlock)
    if (t_key[k] != kEmptyKey) t_base[k] = atomicAdd(cnt + t_key[k], t_cnt[k]);
  __syncthreads();
  if (in_walk) nd[v] = make_uint2(r, active ? t_base[my_slot] + my_pos : 0u);
}

// Segments for the roots met in this round's walk (every non-giant root is a member of its own
// supernode, so it is walked).  cnt is cleared here, its last reader.  Without a giant yet, a root
// holding more than half of the vertices is elected: at most one can.
// drop_ok: every update reached both of its ends' sketches, so a supernode without cut edges stays one:
// no other supernode has an edge into it, and its sums are zero.  A root that was one vertex (rounds >= 2:
// one supernode) in the last round and whose sums were all empty (kSampEmpty) gets no segment
// (off = kDropped), so finished components are not walked again.  The giant's election comes first.
// The deterministic bucket alone does not decide: edges whose indices cancel (any four of the form (v, x),
// (v, x'), (v, y), (v, y') with x ^ x' == y ^ y') leave it zero when their checksums do, once in 2^32 such
// sets, and the supernodes that later link with it would be walked without its members, or not at all
// where its root stays one.  In a column such a set is empty only when all of it falls on one depth.
// A query on 2^20 R-MAT vertices, a third of them isolated: the rounds' launches 1560 -> 700 us.
// A root's segment goes into the round's segment list too (block scan of the counts and of the
// roots, packed in one 64-bit scan: counts in the low 40 bits, roots above).
constexpr uint32_t kSegShift = 40;
constexpr uint32_t kDropped = 0xFFFFFFFFu;

__global__ void __launch_bounds__(kAggBlock)
k_bv_alloc(uint32_t* __restrict__ cnt, uint32_t n, uint32_t* __restrict__ off, uint32_t* __restrict__ cursor,
           uint32_t* __restrict__ st, uint32_t round, const uint32_t* __restrict__ act_list, uint32_t giant_ok,
           const uint32_t* __restrict__ prev_mod, RoundSeg* __restrict__ segs, const uint64_t* __restrict__ samp,
           uint32_t drop_ok) {
  const uint32_t live = ld_acq(prev_mod);  // checked after the first reads (see k_bv_find_count)
  __shared__ uint64_t wsum[kAggBlock / kWave];
  __shared__ uint32_t s_base, s_sbase;
  const bool act = st[kStActMode] != 0;
  const uint32_t lane = lane_id(), wid = threadIdx.x / kWave;
  const uint32_t i = blockIdx.x * kAggBlock + threadIdx.x;
  const uint32_t walk = walk_count(st, round, n);
  const bool in_walk = i < walk;
  const uint32_t v = in_walk ? walk_vertex(act_list, round, i) : 0;
  uint32_t c = in_walk ? cnt[v] : 0;
  const uint64_t sv = in_walk && drop_ok ? samp[v] : kSampFail;
  if (!live || blockIdx.x * kAggBlock >= walk) return;  // whole blocks past the walk
  if (c) cnt[v] = 0;
  if (!act && giant_ok && 2ull * c > n) {
    st[kStGiantFirst] = v;
    st[kStGiantRound] = v;
    c = 0;
  } else if (!act && giant_ok && c >= 2 && c >= n / kCandidateDiv) {  // at most kCandidateDiv roots
    atomicMax(reinterpret_cast<unsigned long long*>(st + kStBest), ((unsigned long long)c << 32) | v);
  }
  const bool drop = c == 1 && sv == kSampEmpty;
  if (drop) {
    c = 0;
    off[v] = kDropped;
  }
  if (drop_ok) {  // uniform
    const uint32_t d = (uint32_t)__syncthreads_count(drop);
    if (threadIdx.x == 0 && d) atomicAdd(st + kStDropped, d);
  }
  const uint64_t x = c ? ((uint64_t)1 << kSegShift) | c : 0;
  const uint64_t incl = wave_incl_scan_u64(x);
  if (lane == kWave - 1) wsum[wid] = incl;
  __syncthreads();
  uint64_t pre = 0, tot = 0;
  for (uint32_t w = 0; w < kAggBlock / kWave; ++w) {
    if (w < wid) pre += wsum[w];
    tot += wsum[w];
  }
  constexpr uint64_t kCntMask = ((uint64_t)1 << kSegShift) - 1;
  if (threadIdx.x == 0) {
    // entries and supernodes of the block in one 64-bit atomic (neither sum can reach 2^32)
    const uint64_t add = ((tot >> kSegShift) << 32) | (tot & kCntMask);
    const uint64_t old =
        add ? atomicAdd(reinterpret_cast<unsigned long long*>(st + kStSeg + 2 * (round & 1)), (unsigned long long)add) : 0;
    s_base = (uint32_t)old;
    s_sbase = (uint32_t)(old >> 32);
  }
  __syncthreads();
  if (c) {
    const uint64_t ex = pre + incl - x;
    const uint32_t o = s_base + (uint32_t)(ex & kCntMask);
    const uint32_t k = s_sbase + (uint32_t)(ex >> kSegShift);
    off[v] = o;
    cursor[v] = o + c;  // the segment end
    if (k < n) segs[k] = RoundSeg{v, o, c, 0};
  }
}

__global__ void __launch_bounds__(kAggBlock)
k_bv_scatter(const uint2* __restrict__ nd, uint32_t n, const uint32_t* __restrict__ off,
             uint32_t* __restrict__ members, uint32_t* __restrict__ mroot, const uint32_t* __restrict__ st, uint32_t round,
             const uint32_t* __restrict__ act_list, const uint32_t* __restrict__ prev_mod) {
  const uint32_t live = ld_acq(prev_mod);  // checked after the first reads (see k_bv_find_count)
  const uint32_t gr = st[kStGiantRound];
  const uint32_t e = st[kStSeg + 2 * (round & 1)];
  const uint32_t i = blockIdx.x * kAggBlock + threadIdx.x;
  const uint32_t walk = walk_count(st, round, n);
  const bool in_walk = i < walk;
  const uint32_t v = in_walk ? walk_vertex(act_list, round, i) : 0;
  const uint2 t = in_walk && v < n ? nd[v] : make_uint2(0u, 0u);
  if (!live || !in_walk || v >= n) return;
  if (t.x == gr || t.x >= n) return;  // the giant supernode's members are not regrouped
  const uint32_t o = off[t.x], p = o + t.y;
  if (o == kDropped || p >= e || p >= n) return;
  members[p] = v;  // the root beside the member, so the reduce reads both in list order
  mroot[p] = t.x;
}

// ---- regrouping by segments (rounds >= 2) ------------------------------------------------------
// A supernode of round r is a union of supernodes of round r - 1, and those are contiguous runs
// ("segments") of round r - 1's member list.  So round r regroups whole runs: A) the new root of
// every old segment, and the run's offset inside its new root's segment, taken from the root's
// member counter (atomics aggregated per block in LDS); B) a contiguous segment per new root and
// the round's segment list; C) one pass over the old member list copying each member to its place
// (its root's segment start + its run's offset + its place in the run), with its new root beside
// it and its parent pointer compressed to that root.  A and B walk the old segments (one per old
// supernode), only C walks the members, in list order.  Runs whose new root is the giant are dropped, as the vertex walk drops
// the giant's members.  Every kernel loads its counts and lists before it looks at the round flag
// (all in range: they are those of an earlier round of this query, or the start values) and writes
// nothing when the round is not live; indices computed from device data are bounded by n before
// every store.

// What a round's segments are written to.
struct SegOut {
  uint32_t *off, *cursor;
  RoundSeg* segs;
};
// A segment of c members for root v, whose segment of the last round had old_len (threads without one
// pass c == 0), and the giant's election and candidate as in k_bv_alloc; every thread of the workgroup
// takes part.  SINGLE: this workgroup has all of the round's segments, and one thread writes the round's
// state, the giant elected here or the one known (gfirst, by its root gcur).
template <bool SINGLE>
__device__ inline void seg_allocate(uint32_t c, uint32_t v, uint32_t old_len, uint64_t sv, bool act, uint32_t n,
                                    const SegOut& out, uint32_t* __restrict__ st, uint32_t round, uint32_t giant_ok,
                                    uint32_t drop_ok, uint32_t gfirst, uint32_t gcur) {
  __shared__ uint64_t wsum[kAggBlock / kWave];
  __shared__ uint32_t s_base, s_sbase, s_drop, s_elect;
  const uint32_t lane = lane_id(), wid = threadIdx.x / kWave;
  if (SINGLE || drop_ok) {  // uniform
    if (threadIdx.x == 0) {
      s_drop = 0;
      s_elect = kNoRoot;
    }
    __syncthreads();
  }
  if (!act && giant_ok && 2ull * c > n) {
    if (SINGLE) {
      s_elect = v;
    } else {
      st[kStGiantFirst] = v;
      st[kStGiantRound] = v;
    }
    c = 0;
  } else if (!act && giant_ok && c >= 2 && c >= n / kCandidateDiv) {
    atomicMax(reinterpret_cast<unsigned long long*>(st + kStBest), ((unsigned long long)c << 32) | v);
  } else if (c != 0 && c == old_len && sv == kSampEmpty) {
    atomicAdd(&s_drop, c);
    c = 0;
    out.off[v] = kDropped;
  }
  const uint64_t x = c ? ((uint64_t)1 << kSegShift) | c : 0;
  const uint64_t incl = wave_incl_scan_u64(x);
  if (lane == kWave - 1) wsum[wid] = incl;
  __syncthreads();
  uint64_t pre = 0, tot = 0;
  for (uint32_t w = 0; w < kAggBlock / kWave; ++w) {
    if (w < wid) pre += wsum[w];
    tot += wsum[w];
  }
  constexpr uint64_t kCntMask = ((uint64_t)1 << kSegShift) - 1;
  if (threadIdx.x == 0) {
    if (drop_ok && s_drop) atomicAdd(st + kStDropped, s_drop);
    // entries and supernodes of the block in one 64-bit word (neither sum can reach 2^32)
    auto* both = reinterpret_cast<unsigned long long*>(st + kStSeg + 2 * (round & 1));
    const uint64_t add = ((tot >> kSegShift) << 32) | (tot & kCntMask);
    uint64_t base = 0;
    if (SINGLE) {
      *both = add;
      st[kStGiantRound] = s_elect != kNoRoot ? s_elect : gcur;
      st[kStGiantFirst] = s_elect != kNoRoot ? s_elect : gfirst;
      st[kStActMode] = act ? 1u : 0u;
    } else if (add) base = atomicAdd(both, (unsigned long long)add);
    s_base = (uint32_t)base;
    s_sbase = (uint32_t)(base >> 32);
  }
  __syncthreads();
  if (c) {
    const uint64_t ex = pre + incl - x;
    const uint32_t o = s_base + (uint32_t)(ex & kCntMask);
    const uint32_t k = s_sbase + (uint32_t)(ex >> kSegShift);
    out.off[v] = o;
    out.cursor[v] = o + c;  // the segment end
    if (k < n) out.segs[k] = RoundSeg{v, o, c, 0};
  }
}

__global__ void __launch_bounds__(kAggBlock)
k_seg_find(uint32_t* __restrict__ parent, uint32_t n, uint32_t* __restrict__ cnt, uint2* __restrict__ nd,
           SegOut out, uint32_t* __restrict__ st, uint32_t round, const RoundSeg* __restrict__ segs_old,
           uint32_t giant_ok, const uint32_t* __restrict__ prev_mod, const uint64_t* __restrict__ samp,
           uint32_t drop_ok) {
  const uint32_t live = ld_acq(prev_mod);
  uint32_t gfirst = st[kStGiantFirst];
  const uint64_t best = *reinterpret_cast<const uint64_t*>(st + kStBest);
  const uint32_t nseg = st[kStSeg + 2 * ((round - 1) & 1) + 1];
  const uint32_t i = blockIdx.x * kAggBlock + threadIdx.x;
  const bool in = i < nseg;
  RoundSeg sg{0, 0, 0, 0};
  if (in) sg = segs_old[i];
  const bool single = nseg <= kAggBlock;  // this workgroup meets every member of every new supernode
  // block 0 writes the round state even with no segments to walk
  if (!live || (blockIdx.x > 0 && blockIdx.x * kAggBlock >= nseg)) return;
  __shared__ uint32_t t_key[kAggTable], t_cnt[kAggTable];
  for (uint32_t k = threadIdx.x; k < kAggTable; k += kAggBlock) {
    t_key[k] = kEmptyKey;
    t_cnt[k] = 0;
  }
  if (gfirst == kNoRoot && best) gfirst = (uint32_t)best;  // a candidate recorded by the previous round
  const bool act = gfirst != kNoRoot;
  const uint32_t gcur = act ? dsu_find_stable(parent, gfirst) : kNoRoot;
  if (!single && blockIdx.x == 0 && threadIdx.x == 0) {
    st[kStSeg + 2 * (round & 1)] = 0;
    st[kStSeg + 2 * (round & 1) + 1] = 0;
    st[kStGiantRound] = gcur;
    st[kStGiantFirst] = gfirst;
    st[kStActMode] = act ? 1u : 0u;
  }
  __shared__ uint32_t t_base[kAggTable];
  const bool ok = in && sg.root < n;
  const uint64_t sv = single && ok && drop_ok ? samp[sg.root] : kSampFail;
  uint32_t r = 0;
  if (ok) r = dsu_find_stable(parent, sg.root);
  __syncthreads();
  const bool counted = ok && r != gcur;
  uint32_t my_slot = 0, my_pos = 0;
  if (ok) parent[sg.root] = r;  // path compression of the old root (members are compressed in C)
  if (counted) {
    my_slot = lds_table_slot(t_key, r);
    my_pos = atomicAdd(t_cnt + my_slot, sg.len);
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < kAggTable; k += kAggBlock)
    if (t_key[k] != kEmptyKey) t_base[k] = single ? 0u : atomicAdd(cnt + t_key[k], t_cnt[k]);
  __syncthreads();
  // the run's offset in its new root's segment, minus its old start: a member at old position i
  // goes to off[new root] + i + nd.y
  if (ok) nd[sg.root] = make_uint2(r, counted ? t_base[my_slot] + my_pos - sg.start : 0u);
  // few supernodes: their segments are given out here, without the counters, and k_seg_alloc has nothing
  // to do: a query over 32k vertices in 64 components 500 -> 490 us, a point query on 2^18 519 -> 510
  if (single)
    seg_allocate<true>(counted && r == sg.root ? t_cnt[my_slot] : 0u, sg.root, sg.len, sv, act, n, out, st, round,
                       giant_ok, drop_ok, gfirst, gcur);
}

// B: a segment for every new root (an old root that is still a root) outside the giant; cnt is
// cleared here, its last reader.
__global__ void __launch_bounds__(kAggBlock)
k_seg_alloc(uint32_t* __restrict__ cnt, uint32_t n, const uint2* __restrict__ nd, SegOut out, uint32_t* __restrict__ st,
            uint32_t round, const RoundSeg* __restrict__ segs_old, uint32_t giant_ok,
            const uint32_t* __restrict__ prev_mod, const uint64_t* __restrict__ samp, uint32_t drop_ok) {
  const uint32_t live = ld_acq(prev_mod);
  const bool act = st[kStActMode] != 0;
  const uint32_t nseg = st[kStSeg + 2 * ((round - 1) & 1) + 1];
  if (!live || nseg <= kAggBlock || blockIdx.x * kAggBlock >= nseg) return;  // whole blocks past the segments
  const uint32_t i = blockIdx.x * kAggBlock + threadIdx.x;
  const bool in = i < nseg;
  const uint32_t v = in ? segs_old[i].root : 0, old_len = in ? segs_old[i].len : 0;
  const bool ok = in && v < n;
  const bool is_root = ok && nd[v].x == v;
  const uint32_t c = is_root ? cnt[v] : 0;  // zero for the giant's root: its members are not counted
  const uint64_t sv = ok && drop_ok ? samp[v] : kSampFail;
  if (c) cnt[v] = 0;
  seg_allocate<false>(c, v, old_len, sv, act, n, out, st, round, giant_ok, drop_ok, kNoRoot, kNoRoot);
}

// C: every member of the old list to its place, its new root beside it, its parent compressed to
// that root.
__global__ void __launch_bounds__(256)
k_seg_copy(uint32_t n, const uint2* __restrict__ nd, const uint32_t* __restrict__ off, uint32_t* __restrict__ parent,
           const uint32_t* __restrict__ members_old, const uint32_t* __restrict__ mroot_old,
           uint32_t* __restrict__ members_new, uint32_t* __restrict__ mroot_new, const uint32_t* __restrict__ st,
           uint32_t round, const uint32_t* __restrict__ prev_mod) {
  const uint32_t live = ld_acq(prev_mod);
  const uint32_t gr = st[kStGiantRound];
  const uint32_t e_old = st[kStSeg + 2 * ((round - 1) & 1)];
  const uint32_t e_new = st[kStSeg + 2 * (round & 1)];
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool in = i < e_old && i < n;
  uint32_t v = 0, R = 0;
  if (in) {
    v = members_old[i];
    R = mroot_old[i];
  }
  if (!live || !in || R >= n || v >= n) return;
  const uint2 t = nd[R];
  if (t.x == gr || t.x >= n) return;
  const uint32_t o = off[t.x], p = o + i + t.y;
  if (o == kDropped || p >= e_new || p >= n) return;
  members_new[p] = v;
  mroot_new[p] = t.x;
  parent[v] = t.x;
}

// Segmented XOR-reduce + sample (range_merge of column `round` + the deterministic bucket over
// every member of a supernode, then sample_supernode).  Entries are the member list, grouped by
// root.  A wave takes 64 consecutive entries (reduce_members).  A supernode whose entries all lie
// inside the range is sampled from registers; its sample record goes to samp[root].  A supernode that crosses the range's first (head) or last (tail) boundary leaves
// its partial XOR in the range's head or tail slot under its root; a slot left unused gets root
// kNoRoot and a zero value.
//
// A workgroup of 16 waves covers 1024 entries (512 or 256 in smaller rounds): the waves leave their slots in LDS, then the wave in
// which a crossing supernode starts adds up that supernode's slots, so at most two supernodes of a
// workgroup are unfinished: the one continuing from the previous workgroup and the one continuing
// into the next.
//
// The round's merges are made here too: a wave keeps the samples of its supernodes one to a lane and
// links them all at once at its end (no kernel of the round reads the parents beside this one).  Taken
// in the loop that samples them, one by one, the links cost three times the launch that they spare;
// before the workgroup's barrier, 2 us a round more than after it.  Against a launch of their own
// (5 to 11 us a round), a query over 32k vertices in 64 components went from 579 to 537 us with its
// updates, a point query on 2^18 vertices from 600 to 570 us; full rounds of 2^18 gain nothing.
//
// A full round over 2^18 members reads three lines per member (122 MB) and is bound by them: a
// workgroup's records arrive over 7..20 us of its 28 and the sampling runs behind.  Before the rows of
// 16 lanes a member filled 16 of a load's 64 lanes and a wave took its members in 8 dependent
// batches: the launched rounds of a 24M-update, 2^18-vertex serving trace went from 39.1 to 25.0 us on
// average, those of 32k vertices from 34.3 to 15.0 us, of 2^20 R-MAT vertices from 147 to 79 us, and
// the single-workgroup finish of about 1500 members from 95 to 47 us (30 with its own changes).
//
// Cross-workgroup supernodes.  A supernode whose entries span workgroups f..l (f < l) is combined
// with device-scope XOR atomics into the accumulator slot of f, its first workgroup (only one
// supernode per workgroup can continue past its end, so f identifies it).  Every workgroup of f..l
// adds its part once and then counts itself in slot f's counter; the one that brings the count to
// l - f + 1 samples the sum and clears the slot and the counter for the next round.  The parts are
// added with atomics that return, so they have been performed when the count is made, and the last one
// takes the sum with exchanges that leave zeros: no fence, which would write caches back and invalidate
// them for every part.  That order is a property of this card (a device-scope atomic that has returned was
// performed where every workgroup's next one sees it), not of the language's memory model: until the last
// workgroup has cleared a slot, every access to it and to its counter has to stay a returning
// read-modify-write of device scope.  A reduce of 2^18 vertices took 29.7 us on average with a full fence before the
// count and after the last one, 26.0 with a release and an acquire, 23.2 now; of 32k vertices 13.7, 11.8
// and 10.8.  The segment bounds are those that k_bv_alloc or seg_allocate gave out (off = start, cursor =
// end).  No workgroup waits for another, and the XOR is order-free, so the sum is exactly the member-wise merge.
//
// Giant supernode.  Every edge update XORs the same buckets into both endpoints' sketches, so the
// XOR of all vertex sketches is zero and a supernode's sum equals the XOR of every vertex outside
// it.  When a supernode is summed from its complement (the sketches known to sum to zero) its
// members are not regrouped: each workgroup XORs all of its entries into a total and adds it to
// the giant's accumulator slot (slot gridDim.x), counted like the others, and the last workgroup
// samples the giant from that sum -- the same bytes the member-wise merge would give.
constexpr uint32_t kRedWaves = 16, kRedBlock = kRedWaves * kWave;

// Slot of a range's boundary partial: 128 u64 (alpha of lanes 0..63, then gamma) and a root.
struct Slot {
  uint64_t* vals;
  uint32_t* root;
};

// Cross-workgroup accumulators: nslots slots of 128 u64 and as many arrival counters, all zero
// between rounds.  Slots 0 .. gridDim.x - 1 belong to the workgroups, slot nslots - 1 to the giant;
// the launcher checks gridDim.x + 1 <= nslots.
struct XAcc {
  uint64_t* vals;
  uint32_t* cnt;
  uint32_t nslots;
  const uint32_t* seg_off;  // segment start per root
  const uint32_t* seg_end;  // segment end per root
};

// Value of lane K of every row of 16 lanes, given to all lanes of that row.  Every lane must be active.
template <uint32_t K>
__device__ inline uint32_t row_bcast(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + K, 0xf, 0xf, false);  // row_newbcast:K
}
template <class F, uint32_t... K>
__device__ inline void for_each_index(F&& f, std::integer_sequence<uint32_t, K...>) {
  (f(std::integral_constant<uint32_t, K>{}), ...);
}
// Bits 0 .. k - 1 (k <= 64).
__device__ inline uint64_t low_bits(uint32_t k) { return k >= 64 ? ~0ull : (1ull << k) - 1; }

// Reduce entries [p0, p0 + len) of a grouped member list with one wave (len <= 4q, q <= 16).  members /
// mroot: the list and its roots by position, list_end entries (global or LDS).
//
// Four entries per load: row j of 16 lanes takes entries p0 + jq .. p0 + jq + q - 1 one after the
// other; lane i < 15 of a row reads depth i of column `round`, lane 15 the deterministic bucket from
// the compact copy.  All q records of a lane are loaded at once, so the entries of a wave cost one
// dependent round trip instead of one per 8 entries, and a load fills all 64 lanes where 16 of 64
// did the work.  A run of entries of one supernode that lies inside the wave is sampled from
// registers; runs crossing rows are carried from row to row.  The entries' deeper records (depths
// >= 15) are read by the whole wave, one entry per load, only where the sum needs them: for a run
// without a good bucket below, and for the parts that leave the wave.  With deep flags and deep_on
// only the entries whose flag is set are read (the others hold zeros); otherwise all of them.
//
// A run that started before the range is left in the head slot under its root, one that continues
// past it in the tail slot; one that does both is left in the head slot, with a zero value under the
// same root in the tail slot, so the supernode's entries stay contiguous in the next reduce.  A slot
// left unused gets root kNoRoot and a zero value.  s_tot, if given, gets the XOR of every entry.  With
// s_bnd, the wave holding the workgroup's first entry [blk_b0] loads that entry's segment bounds into
// s_bnd[0..1], the one holding its last entry the end of that entry's segment into s_bnd[2].  pend, if
// given, gets in each lane the sample record of the run that begins at the lane's entry, or ZERO.
constexpr uint32_t kRow = 16, kRowDet = kRow - 1;  // lanes of a row; the lane of the deterministic bucket
typedef uint32_t Words __attribute__((ext_vector_type(16)));  // one word of a row's 16 entries per lane
template <class G>
__device__ inline void reduce_members(uint32_t p0, uint32_t len, uint32_t q, uint32_t list_end,
                                      const uint32_t* members, const uint32_t* mroot,
                                      const unsigned char* __restrict__ slab, const Geo& g, uint32_t round, Slot head,
                                      Slot tail, uint64_t* __restrict__ samp, uint32_t* __restrict__ flags,
                                      const unsigned char* __restrict__ det_cpy, bool deep_on, uint64_t* s_tot,
                                      const XAcc* xa, uint32_t blk_b0, uint32_t blk_b1, uint32_t* s_bnd,
                                      uint64_t* pend, bool ahead = false) {
  constexpr uint32_t RB = 8 + sizeof(G);
  const uint32_t lane = lane_id(), i = lane % kRow, base = lane - i, row = lane / kRow;
  // lane base + k holds entry k of its row
  const bool mine = i < q && row * q + i < len;
  const uint32_t pe = p0 + row * q + i;
  uint32_t m = 0, rt = kNoRoot, before = kNoRoot;
  if (mine) {
    m = members[pe];
    rt = mroot[pe];
    if (pe > 0) before = mroot[pe - 1];
  }
  const uint32_t p1 = p0 + len;
  const uint32_t next_root = p1 < list_end ? mroot[p1] : kNoRoot;
  // bit l: lane l's entry begins a run.  Lanes without an entry continue the run before them with zeros.
  const uint64_t starts = __ballot(mine && rt != before);
  const uint32_t rowst = (uint32_t)(starts >> base) & 0xffffu;
  const uint32_t first_root = rd_lane_u32(rt, 0);
  const uint32_t last_root = rd_lane_u32(rt, (int)((len - 1) / q * kRow + (len - 1) % q));
  const bool tail_open = next_root == last_root;
  const bool holds_first = s_bnd && p0 == blk_b0;
  const bool holds_last = s_bnd && p1 == blk_b1;
  uint32_t bnd = 0;
  if (holds_first && lane == 0) bnd = xa->seg_off[first_root];
  if (holds_first && lane == 1) bnd = xa->seg_end[first_root];
  if (holds_last && lane == 2) bnd = xa->seg_end[last_root];

  const bool live = i == kRowDet || i < g.D;
  const unsigned char* src = i == kRowDet ? det_cpy : slab + (live ? rec_col_off<G>(g, round, i) : 0u);
  const uint32_t stride = i == kRowDet ? RB : g.row;
  const uint32_t row_n = row * q < len ? (len - row * q < q ? len - row * q : q) : 0u;  // the row's entries
  constexpr bool kWide = sizeof(G) == 8;
  Words lo = 0, hi = 0, glo = 0, ghi = 0;
  for_each_index(
      [&](auto kc) {
        constexpr uint32_t k = kc;
        const uint32_t mv = row_bcast<k>(m);
        uint64_t a = 0;
        G gm = 0;
        if (live && k < row_n) ld_rec<G>(src + (size_t)mv * stride, &a, &gm);
        lo[k] = (uint32_t)a;
        hi[k] = (uint32_t)(a >> 32);
        glo[k] = (uint32_t)gm;
        if constexpr (kWide) ghi[k] = (uint32_t)((uint64_t)gm >> 32);
      },
      std::make_integer_sequence<uint32_t, kRow>{});
  // ahead: the entries' lines of the next column, touched here so that the next round finds them in the L2
  uint32_t near_line = 0, far_line = 0, last_line = 0;
  if (ahead && mine) {
    const unsigned char* nrow = slab + (size_t)m * g.row;
    near_line = *reinterpret_cast<const uint32_t*>(nrow + rec_col_off<G>(g, round + 1, 0));
    if (g.D > g.low) far_line = *reinterpret_cast<const uint32_t*>(nrow + rec_col_off<G>(g, round + 1, g.low));
    if (kWide && g.D > g.low + 8)
      last_line = *reinterpret_cast<const uint32_t*>(nrow + rec_col_off<G>(g, round + 1, g.low + 8));
  }
  uint32_t flag = 1;
  if (kDeepFlags<G> && deep_on && mine)
    flag = *reinterpret_cast<const uint32_t*>(slab + (size_t)m * g.row + deep_flag_off(round));

  // What was sampled of the run whose first entry is lane l's, at recs[l] (in the head slot, which is
  // written last): its index or one of these.  The runs leave no more than that here; their records are
  // written by one step for the wave, each by its first lane.
  constexpr uint64_t kRecBad = kSampFail - 1, kRecLeft = kSampFail - 2, kRecNone = kSampFail - 3;
  uint64_t* recs = head.vals;
  recs[lane] = kRecNone;
  // lanes that go before this one where several buckets of a run are good: the deterministic bucket, then
  // the lower depths
  const uint32_t before_me = i == kRowDet ? 0u : (1u << kRowDet) | ((1u << i) - 1);
  // Sample the runs of the rows with `done` set (the same in all lanes of a row); first: the run's first lane.
  auto emit = [&](bool done, uint64_t a, G gm, uint32_t first) {
    const bool held = (a | (uint64_t)gm) != 0, zero = i == kRowDet && !held;
    const bool empty = ((__ballot(held) >> base) & 0xffffu) == 0;
    const bool ok = done && live && (zero || (G)xxh3_mix(xxh3_prep(a), g.chk_bf) == gm);
    const uint32_t good = (uint32_t)(__ballot(ok) >> base) & 0xffffu;
    const bool left = done && i == kRowDet && good == 0;
    if (left || (ok && (good & before_me) == 0)) {
      const uint32_t x = (uint32_t)(a >> 32), y = (uint32_t)a;
      recs[first] = left ? kRecLeft : zero ? (empty ? kSampEmpty : kSampZero) : (x > y ? x : y) < g.n ? a : kRecBad;
    }
  };

  // The XOR of every prefix of the row's entries; a run is the XOR of two of them.  The runs are then
  // taken in a loop over the places where one ends in some row (a uniform register index), not in 16
  // unrolled copies of the sampling code, whose instruction fetches cost more than the sampling.
  for_each_index(
      [&](auto kc) {
        constexpr uint32_t k = kc + 1;
        lo[k] ^= lo[k - 1];
        hi[k] ^= hi[k - 1];
        glo[k] ^= glo[k - 1];
        if constexpr (kWide) ghi[k] ^= ghi[k - 1];
      },
      std::make_integer_sequence<uint32_t, kRow - 1>{});
  auto prefix = [&](uint32_t k, uint64_t* a, G* gm) {
    *a = ((uint64_t)hi[k] << 32) | lo[k];
    *gm = kWide ? (G)(((uint64_t)ghi[k] << 32) | glo[k]) : (G)glo[k];
  };
  // h: the row's first run, when it began before the row and ends inside it; acc: its last run
  uint64_t acc, h_a = 0, tot, done_a = 0;
  G accg, h_g = 0, totg, done_g = 0;
  for (uint32_t at = (uint32_t)(starts | starts >> kRow | starts >> 2 * kRow | starts >> 3 * kRow) & 0xfffeu; at;
       at &= at - 1) {
    const uint32_t k = (uint32_t)__builtin_ctz(at);
    uint64_t pa;
    G pg;
    prefix(k - 1, &pa, &pg);
    const bool ends = (rowst >> k) & 1u;
    const uint32_t earlier = rowst & ((1u << k) - 1);
    if (ends && !earlier) {
      h_a = pa;
      h_g = pg;
    }
    emit(ends && earlier, pa ^ done_a, (G)(pg ^ done_g), base + 31u - (uint32_t)__builtin_clz(earlier | 1u));
    if (ends) {
      done_a = pa;
      done_g = pg;
    }
  }
  prefix(kRow - 1, &tot, &totg);
  acc = tot ^ done_a;
  accg = totg ^ done_g;
  // carry each row's last run into the next row while it continues there
  const bool cont = !(rowst & 1u), single = (rowst >> 1) == 0;
  for (uint32_t r = 1; r < 4; ++r) {
    if ((starts >> (kRow * r)) & 1) continue;  // uniform
    const uint64_t ca = shfl_u64(acc, (int)(lane - kRow));
    const G cg = sizeof(G) == 4 ? (G)__shfl((unsigned)accg, (int)(lane - kRow)) : (G)shfl_u64((uint64_t)accg, (int)(lane - kRow));
    if (row == r) {
      if (single) {
        acc ^= ca;
        accg ^= cg;
      } else {
        h_a ^= ca;
        h_g ^= cg;
      }
    }
  }
  const uint64_t st_h = starts & low_bits(base), st_x = starts & low_bits(base + kRow);
  const bool has_h = cont && !single;
  const bool ends_x = row == 3 ? !tail_open : ((starts >> (base + kRow)) & 1) != 0;
  if (__ballot(has_h && st_h)) {
    const uint32_t f = 63u - (uint32_t)__builtin_clzll(st_h | 1ull);
    emit(has_h && st_h, h_a, h_g, f);
  }
  if (__ballot(ends_x && st_x)) {
    const uint32_t f = 63u - (uint32_t)__builtin_clzll(st_x | 1ull);
    emit(ends_x && st_x, acc, accg, f);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  uint64_t rec = recs[lane];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  uint64_t again = __ballot(rec == kRecLeft);  // first lanes of the runs left to the deep records
  if (rec == kRecBad) {  // an index out of range, as in sample_record
    flags[kFlagBad] = 1;
    rec = kSampFail;
  }
  if (rec != kRecNone && rec != kRecLeft) samp[rt] = rec;
  else rec = kSampZero;

  // deep records: lane d < D of depths >= kRowDet; the XOR over the entries in lanes `of`
  const uint64_t deep = g.D > kRowDet ? __ballot(mine && flag != 0) : 0;
  auto deep_sum = [&](uint64_t of, uint64_t* a_out, G* g_out) {
    const bool in = lane >= kRowDet && lane < g.D;
    const unsigned char* dsrc = slab + (in ? rec_col_off<G>(g, round, lane) : 0u);
    uint64_t a = 0;
    G gm = 0;
    constexpr uint32_t U = 8;  // loads in flight per lane
    for (of &= deep; of;) {
      uint64_t da[U];
      G dg[U];
#pragma unroll
      for (uint32_t k = 0; k < U; ++k) {
        da[k] = 0;
        dg[k] = 0;
        if (of) {
          const uint32_t mv = rd_lane_u32(m, __builtin_ctzll(of));
          of &= of - 1;
          if (in) ld_rec<G>(dsrc + (size_t)mv * g.row, &da[k], &dg[k]);
        }
      }
#pragma unroll
      for (uint32_t k = 0; k < U; ++k) {
        a ^= da[k];
        gm ^= dg[k];
      }
    }
    *a_out = a;
    *g_out = gm;
  };
  for (; again; again &= again - 1) {
    const uint32_t f = (uint32_t)__builtin_ctzll(again);
    const uint64_t later = starts & ~low_bits(f + 1);
    const uint32_t end = later ? (uint32_t)__builtin_ctzll(later) : 64u;
    uint64_t a;
    G gm;
    deep_sum(low_bits(end) & ~low_bits(f), &a, &gm);
    const uint64_t good =
        __ballot(lane >= kRowDet && lane < g.D && (G)xxh3_mix(xxh3_prep(a), g.chk_bf) == gm);
    const uint64_t idx = good ? rd_lane_u64(a, __builtin_ctzll(good)) : 0;
    const uint64_t deep_rec = sample_record(good ? kGood : kFail, idx, g.n, flags);
    if (lane == f) samp[rt] = rec = deep_rec;
  }
  if (pend) *pend = rec;

  // Every lane stores the root (the same value), so every lane of this wave may read it back
  // without a barrier.  Slots are ordered by depth, the deterministic bucket at D.
  const uint32_t pos = i == kRowDet ? g.D : i;
  auto put = [&](Slot sl, uint32_t R, bool holds, uint64_t a, G gm, uint64_t of) {
    uint64_t da;
    G dg;
    deep_sum(of, &da, &dg);
    sl.vals[lane] = da;
    sl.vals[kWave + lane] = (uint64_t)dg;
    if (holds && live) {
      sl.vals[pos] = a;
      sl.vals[kWave + pos] = (uint64_t)gm;
    }
    *sl.root = R;
  };
  if (!(starts & 1)) {  // the first run began before the wave
    const bool from_h = has_h && !st_h;
    const bool from_x = row == 3 && tail_open ? !starts : (ends_x && !st_x);
    put(head, first_root, from_h || from_x, from_h ? h_a : acc, from_h ? h_g : accg,
        starts ? low_bits((uint32_t)__builtin_ctzll(starts)) : ~0ull);
  } else {
    put(head, kNoRoot, false, 0, 0, 0);
  }
  if (!tail_open) put(tail, kNoRoot, false, 0, 0, 0);
  else if (!starts) put(tail, last_root, false, 0, 0, 0);
  else put(tail, last_root, row == 3, acc, accg, ~low_bits(63u - (uint32_t)__builtin_clzll(starts)));
  if (s_tot) {
    uint64_t da;
    G dg;
    deep_sum(~0ull, &da, &dg);
    if (da) lds_xor(s_tot + lane, da);
    if (dg) lds_xor(s_tot + kWave + lane, (uint64_t)dg);
    if (live) {
      lds_xor(s_tot + pos, tot);
      lds_xor(s_tot + kWave + pos, (uint64_t)totg);
    }
  }
  if (ahead) asm volatile("" ::"v"(near_line), "v"(far_line), "v"(last_line));
  if (holds_first && lane < 2) s_bnd[lane] = bnd;
  if (holds_last && lane == 2) s_bnd[2] = bnd;
}

// Per lane: XOR (a, gm) into an accumulator slot with device-scope atomics (zero words skipped), and wait
// for their results, after which they have been performed.
// (See "Cross-workgroup supernodes" above: the wait is what orders the part before the count.)
__device__ inline void xacc_add(uint64_t* slot, uint64_t a, uint64_t gm) {
  const uint32_t lane = lane_id();
  uint64_t was_a = 0, was_g = 0;
  if (a) was_a = __hip_atomic_fetch_xor(slot + lane, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (gm) was_g = __hip_atomic_fetch_xor(slot + kWave + lane, gm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::"v"(was_a), "v"(was_g) : "memory");
}
// An accumulator word, left zero.
__device__ inline uint64_t xacc_take(uint64_t* word) {
  return __hip_atomic_exchange(word, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// LDS of one reduce workgroup: 32 slots of 128 u64 and their roots, the giant total and the segment
// bounds of its first and last entries.
#define GZ_REDUCE_LDS                                             \
  __shared__ uint64_t s_vals[2 * kRedWaves * 2 * kWave];          \
  __shared__ uint32_t s_root[2 * kRedWaves];                      \
  __shared__ uint64_t s_tot[2 * kWave];                           \
  __shared__ uint32_t s_bnd[3];

// The reduce of a whole round: one workgroup per 1024, 512 or 256 entries of the member list (e1 entries,
// written by k_bv_scatter; ReduceShape), gridDim.x >= reduce_blocks(n).
template <class G>
__global__ void __launch_bounds__(kRedBlock)
k_bv_reduce(const uint32_t* __restrict__ st, const uint32_t* __restrict__ members,
            const uint32_t* __restrict__ mroot, const unsigned char* __restrict__ slab, Geo g, uint32_t round,
            XAcc xa, uint64_t* __restrict__ samp, DsuDev d,
            const uint32_t* __restrict__ prev_mod, uint32_t* __restrict__ cur_mod, uint32_t* __restrict__ rstats,
            const unsigned char* __restrict__ det_cpy, const unsigned char* __restrict__ hint, uint32_t upto16,
            uint32_t upto32, uint32_t deep_skip) {
  const uint32_t live = ld_acq(prev_mod);  // checked after the first reads
  GZ_REDUCE_LDS
  const uint32_t giant = st[kStGiantRound];
  const uint32_t e1 = st[kStSeg + 2 * (round & 1)];
  if (!live) return;
  if (rstats && blockIdx.x == 0 && threadIdx.x == 0 && round < kMaxStatRounds) {
    rstats[2 * round] = e1;  // diagnostics: vertices regrouped and the giant's root in this round
    rstats[2 * round + 1] = giant;
    rstats[2 * kMaxStatRounds + round] = st[kStDropped];
  }
  if (giant != kNoRoot && e1 == 0) {  // every vertex is in the giant: its sum is zero
    if (blockIdx.x == 0 && threadIdx.x == 0) samp[giant] = kSampZero;
    return;
  }
  const uint32_t W = e1 <= upto16 ? kWave / 4 : e1 <= upto32 ? kWave / 2 : kWave;  // see ReduceShape
  const uint32_t span = kRedWaves * W;
  const uint32_t blk = blockIdx.x;
  if (blk * span >= e1) return;  // uniform over the workgroup
  const uint32_t lane = lane_id(), wid = threadIdx.x / kWave;
  const uint32_t nblk = (e1 + span - 1) / span;
  const uint32_t b0 = blk * span;
  const uint32_t b1 = b0 + span < e1 ? b0 + span : e1;
  const bool giant_tot = giant != kNoRoot;
  if (giant_tot)
    for (uint32_t k = threadIdx.x; k < 2 * kWave; k += blockDim.x) s_tot[k] = 0;
  __syncthreads();
  // phase 1: every wave reduces its entries, leaving its boundary partials in LDS slots
  const uint32_t p0 = b0 + wid * W;
  Slot hs{s_vals + (size_t)(2 * wid) * 2 * kWave, s_root + 2 * wid};
  Slot ts{s_vals + (size_t)(2 * wid + 1) * 2 * kWave, s_root + 2 * wid + 1};
  uint64_t pend = kSampZero;  // lane l: the sample record of a supernode still to be merged
  if (p0 < b1) {
    const uint32_t len = b1 - p0 < W ? b1 - p0 : W;
    reduce_members<G>(p0, len, W / 4, e1, members, mroot, slab, g, round, hs, ts, samp, d.flags, det_cpy,
                      deep_skip != 0, giant_tot ? s_tot : nullptr, &xa, b0, b1, s_bnd, &pend);
  } else {
    hs.vals[lane] = 0;
    hs.vals[kWave + lane] = 0;
    ts.vals[lane] = 0;
    ts.vals[kWave + lane] = 0;
    if (lane == 0) {
      *hs.root = kNoRoot;
      *ts.root = kNoRoot;
    }
  }
  __syncthreads();
  // phase 2, no barrier follows: the supernodes that cross waves, each summed by one wave.  Lane w
  // holds the head and tail roots of wave w.
  const uint32_t nw = (b1 - b0 + W - 1) / W;  // waves with entries
  const uint32_t hr = lane < nw ? s_root[2 * lane] : kNoRoot, tr = lane < nw ? s_root[2 * lane + 1] : kNoRoot;
  // XOR the head slots of waves x, x + 1, ... that R covers whole, and of the one it ends in; returns
  // whether it goes on past the workgroup
  auto follow = [&](uint32_t R, uint32_t x, uint64_t& a, uint64_t& gm) -> bool {
    const uint32_t whole = (uint32_t)__ballot(hr == R && tr == R) >> x;
    const uint32_t open = x + (uint32_t)__builtin_ctz(~whole);
    const uint32_t end = open < nw ? open + 1 : nw;
#pragma unroll 4
    for (; x < end; ++x) {
      a ^= s_vals[(size_t)(2 * x) * 2 * kWave + lane];
      gm ^= s_vals[(size_t)(2 * x) * 2 * kWave + kWave + lane];
    }
    return open >= nw;
  };
  bool modified = false;
  auto sample_to = [&](uint32_t R, uint64_t a, uint64_t gm) {
    uint64_t idx;
    const int code = wave_sample<G>(a, (G)gm, g.D, g.chk_bf, &idx);
    const uint64_t rec = sample_record(code, idx, g.n, d.flags);
    if (lane == 0) samp[R] = rec;
    const uint64_t idle = __ballot(pend > kSampFail);
    if (!idle) modified |= lane == 0 && apply_sample(d, rec, hint);
    else if (lane == (uint32_t)__builtin_ctzll(idle)) pend = rec;
  };
  // one of the `parts` workgroups that hold R adds its part to accumulator slot `slot`; the last one
  // samples the sum and clears the slot for the next round
  auto cross = [&](uint32_t slot, uint32_t parts, uint32_t R, uint64_t a, uint64_t gm) {
    uint64_t* sv = xa.vals + (size_t)slot * 2 * kWave;
    xacc_add(sv, a, gm);
    uint32_t before = 0;
    if (lane == 0) before = atomicAdd(xa.cnt + slot, 1u);
    if (rd_lane_u32(before, 0) != parts - 1) return;
    const uint64_t sum_a = xacc_take(sv + lane), sum_g = xacc_take(sv + kWave + lane);
    sample_to(R, sum_a, sum_g);
    if (lane == 0) st_rlx(xa.cnt + slot, 0u);
  };
  if (wid < nw) {  // the supernode that starts in this wave and goes on
    const uint32_t R = rd_lane_u32(tr, (int)wid);
    if (R != kNoRoot && R != rd_lane_u32(hr, (int)wid)) {
      const uint64_t* sl = s_vals + (size_t)(2 * wid + 1) * 2 * kWave;
      uint64_t a = sl[lane], gm = sl[kWave + lane];
      if (!follow(R, wid + 1, a, gm)) sample_to(R, a, gm);
      else cross(blk, (s_bnd[2] - 1) / span - blk + 1, R, a, gm);  // it ends where its last entry is
    }
  }
  if (wid == kRedWaves - 1) {  // the supernode that the workgroup's first entry continues
    const uint32_t R = rd_lane_u32(hr, 0);
    if (R != kNoRoot) {
      uint64_t a = 0, gm = 0;
      (void)follow(R, 0, a, gm);  // one covering the whole range is counted here only
      const uint32_t fh = s_bnd[0] / span;
      cross(fh, (s_bnd[1] - 1) / span - fh + 1, R, a, gm);
    }
  }
  if (wid == kRedWaves - 2 && giant_tot) {
    if (nblk == 1) sample_to(giant, s_tot[lane], s_tot[kWave + lane]);  // the giant's whole sum
    else cross(xa.nslots - 1, nblk, giant, s_tot[lane], s_tot[kWave + lane]);
  }
  if (apply_sample(d, pend, hint)) modified = true;
  if (__ballot(modified) && lane == 0) *cur_mod = 1;  // one plain store per wave
}

// ---- the last rounds in one workgroup ----------------------------------------------------------
// Once a giant supernode exists, a round walks only the vertices outside it that are not in a finished
// component, and after a few rounds they are few; a small graph's are few from the start.  k_bv_finish then runs every remaining round inside one workgroup -- the same
// regrouping, reduce, sample and merge as k_bv_find_count .. k_bv_reduce, with barriers between
// the steps instead of kernel boundaries -- so a round costs a few round trips instead of four
// dependent launches.  It takes over at round r0 only when round r0 - 1 changed something and the walk
// holds at most kFinishMax vertices; otherwise it returns without touching any state and the rounds
// continue as launches.  A giant is elected in it as in the launched rounds, so both regroup the same
// vertices.
// It then sets mod[r] for every modified round, as the launched rounds do, and records the last
// round it ran in mod[nmod - 1] (a word no round uses), so one copy of mod tells the host both.
//
// The workgroup reduces its grouped list in chunks of 64 entries (one wave each, reduce_members).  A
// supernode continuing past a chunk is accumulated in LDS under the chunk where it starts (only one
// supernode per chunk can continue past its end) and sampled after a barrier.  Parents that an earlier
// round of this kernel may have changed are read with device-coherent loads.
//
// A round is a chain of about eight steps between barriers, 15 to 45 thousand cycles with everything it
// reads at hand, so the steps are few: roots are looked up from the old roots, the giant's beside them;
// segments are taken from a cursor by each supernode's first member, without a scan of the table; a wave
// links its samples as soon as it has them, without a pass over the table behind a device-wide fence
// (each of the two a fifth of a round); the next round's lines are touched while this round's arrive.
// 1000 vertices (5 rounds) 88 -> 61 us, the last 400 vertices of 2^18 44 -> 30, of a serving trace 23.6
// -> 17.2, 8-byte checksums 38 -> 25.
constexpr uint32_t kFinishMax = 2048;
constexpr uint32_t kFinishTable = 4096;  // LDS hash table of roots, >= 2 * kFinishMax, power of two
constexpr uint32_t kFinishChunks = kFinishMax / kWave;
constexpr uint32_t kFinishPer = kFinishMax / kRedBlock;  // walked vertices per thread

__device__ inline uint32_t dsu_find_coherent(uint32_t* parent, uint32_t u) {
  uint32_t p = ld_acq(parent + u);
  while (true) {
    const uint32_t gp = ld_acq(parent + p);
    if (gp == p) return p;
    u = p;
    p = gp;
  }
}

__device__ inline uint32_t finish_slot(uint32_t* keys, uint32_t key) {
  uint32_t h = (key * 2654435761u) & (kFinishTable - 1);
  while (true) {
    const uint32_t prev = atomicCAS(keys + h, kEmptyKey, key);
    if (prev == kEmptyKey || prev == key) return h;
    h = (h + 1) & (kFinishTable - 1);
  }
}

template <class G>
__global__ void __launch_bounds__(kRedBlock)
k_bv_finish(DsuDev d, uint32_t* __restrict__ st, const uint32_t* __restrict__ act0,
            const uint32_t* __restrict__ mroot0, const unsigned char* __restrict__ slab, Geo g, uint32_t r0, uint32_t last_round,
            uint64_t* __restrict__ samp, uint32_t* __restrict__ rstats, const unsigned char* __restrict__ det_cpy,
            const unsigned char* __restrict__ hint, uint32_t* __restrict__ rep, uint32_t deep_skip) {
  __shared__ uint32_t s_key[kFinishTable], s_cnt[kFinishTable];
  __shared__ uint32_t s_mem[kFinishMax], s_mroot[kFinishMax], s_seg[kFinishMax];
  __shared__ uint64_t s_acc[kFinishChunks * 2 * kWave];
  __shared__ uint32_t s_accroot[kFinishChunks];
  __shared__ uint64_t s_slot[kRedWaves * 2 * 2 * kWave];  // per wave: head and tail of its chunk
  __shared__ uint32_t s_slotroot[kRedWaves * 2];
  __shared__ uint64_t s_tot[2 * kWave];
  __shared__ uint32_t s_take, s_gfirst, s_walk, s_gcur, s_e, s_elect;
  __shared__ unsigned long long s_best;
  const uint32_t tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
  if (tid == 0) {
    const uint32_t live = ld_acq(d.mod + (r0 - 1));
    uint32_t gfirst = st[kStGiantFirst];
    const uint64_t best = *reinterpret_cast<const uint64_t*>(st + kStBest);
    if (gfirst == kNoRoot && best) gfirst = (uint32_t)best;  // as k_bv_find_count takes the candidate
    const uint32_t walk = st[kStSeg + 2 * ((r0 - 1) & 1)];
    s_take = (live && walk <= kFinishMax) ? 1u : 0u;
    s_gfirst = gfirst;
    s_gcur = kNoRoot;
    s_best = 0;
    s_walk = walk;
  }
  // The last kernel of every group of rounds: on exit it copies the round flags and the per-round
  // diagnostics to rep (mapped host memory), where the host reads them after its wait, so no copy
  // launch follows the group.
  auto report = [&]() {
    __syncthreads();
    for (uint32_t t = tid; t < d.nmod; t += kRedBlock) rep[t] = ld_acq(d.mod + t);
    for (uint32_t t = tid; t < 3 * kMaxStatRounds; t += kRedBlock) rep[d.nmod + t] = ld_acq(rstats + t);
    __threadfence_system();
  };
  __syncthreads();
  if (!s_take) {
    if (rep) report();
    return;
  }
  uint32_t walk = s_walk;
  // the walked vertices and their roots of the round before
  uint32_t v[kFinishPer], old[kFinishPer];
#pragma unroll
  for (uint32_t k = 0; k < kFinishPer; ++k) {
    const bool in = tid + k * kRedBlock < walk;
    v[k] = in ? act0[tid + k * kRedBlock] : 0u;
    old[k] = in ? mroot0[tid + k * kRedBlock] : 0u;
  }
  for (uint32_t c = tid; c < kFinishChunks * 2 * kWave; c += kRedBlock) s_acc[c] = 0;
  for (uint32_t c = tid; c < kFinishChunks; c += kRedBlock) s_accroot[c] = kNoRoot;

  for (uint32_t r = r0;; ++r) {
    for (uint32_t k = tid; k < kFinishTable; k += kRedBlock) {
      s_key[k] = kEmptyKey;
      s_cnt[k] = 0;
    }
    if (tid < 2 * kWave) s_tot[tid] = 0;
    // The giant's root (it only grows) by the last thread, beside the roots of the walked vertices, which
    // start at the vertices' old roots: one round trip where the old root is one still.
    if (tid == kRedBlock - 1) {
      if (s_gfirst == kNoRoot && s_best) s_gfirst = (uint32_t)s_best;
      if (s_gcur == kNoRoot) s_gcur = s_gfirst;
      if (s_gcur != kNoRoot) s_gcur = dsu_find_coherent(d.parent, s_gcur);
      s_elect = kNoRoot;
      s_e = 0;
    }
    uint32_t rr[kFinishPer], up[kFinishPer], slot[kFinishPer], pos[kFinishPer];
    bool more = false;
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; ++k) {
      rr[k] = old[k];
      up[k] = tid + k * kRedBlock < walk ? ld_acq(d.parent + old[k]) : old[k];
    }
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; ++k) more |= up[k] != rr[k];
    while (more) {
      more = false;
#pragma unroll
      for (uint32_t k = 0; k < kFinishPer; ++k)
        if (up[k] != rr[k]) {
          rr[k] = up[k];
          up[k] = ld_acq(d.parent + rr[k]);
        }
#pragma unroll
      for (uint32_t k = 0; k < kFinishPer; ++k) more |= up[k] != rr[k];
    }
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; ++k)
      if (tid + k * kRedBlock >= walk) rr[k] = kNoRoot;
    __syncthreads();
    uint32_t gcur = s_gcur;
    // path compression, members per root (k_bv_find_count)
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; ++k) {
      if (rr[k] == kNoRoot) continue;
      if (rr[k] != old[k]) st_rlx(d.parent + v[k], rr[k]);
      if (rr[k] != gcur) {  // members of the giant are not regrouped
        slot[k] = finish_slot(s_key, rr[k]);
        pos[k] = atomicAdd(s_cnt + slot[k], 1u);
      }
    }
    __syncthreads();
    // The first member counted takes its supernode's segment, from a cursor (segments need no order); its
    // slot's count becomes the segment's start.
    if (gcur == kNoRoot) {  // the giant's election and candidates, as in k_bv_alloc
#pragma unroll
      for (uint32_t k = 0; k < kFinishPer; ++k) {
        if (rr[k] == kNoRoot || pos[k] != 0) continue;
        const uint32_t c = s_cnt[slot[k]];
        if (2ull * c > d.n) s_elect = s_gfirst = rr[k];  // at most one
        else if (c >= 2 && c >= d.n / kCandidateDiv) atomicMax(&s_best, ((unsigned long long)c << 32) | rr[k]);
      }
      __syncthreads();
      gcur = s_elect;
    }
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; ++k) {
      if (rr[k] == kNoRoot || rr[k] == gcur || pos[k] != 0) continue;
      s_cnt[slot[k]] = atomicAdd(&s_e, s_cnt[slot[k]]);
    }
    __syncthreads();
    const uint32_t e = s_e;
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; ++k) {
      if (rr[k] == kNoRoot || rr[k] == gcur) continue;
      const uint32_t p = s_cnt[slot[k]] + pos[k];
      s_mem[p] = v[k];
      s_mroot[p] = rr[k];
      s_seg[p] = s_cnt[slot[k]];
    }
    if (tid == 0 && rstats && r < kMaxStatRounds) {
      rstats[2 * r] = e;
      rstats[2 * r + 1] = gcur;
      rstats[2 * kMaxStatRounds + r] = st[kStDropped];
    }
    __syncthreads();
    // reduce + sample (k_bv_reduce): one wave per chunk of cw <= 64 entries, the entries spread
    // over all waves (at least 8 per chunk), so a small round is a short chain of gathers; at most
    // 16 chunks below 64 entries each, at most kFinishChunks of 64
    const uint32_t per_wave = (e + kRedWaves - 1) / kRedWaves;
    const uint32_t cw = per_wave >= kWave ? kWave : (per_wave < 8 ? 8u : (per_wave + 7) & ~7u);
    const uint32_t nchunks = (e + cw - 1) / cw;
    Slot hs{s_slot + (size_t)(2 * wid) * 2 * kWave, s_slotroot + 2 * wid};
    Slot ts{s_slot + (size_t)(2 * wid + 1) * 2 * kWave, s_slotroot + 2 * wid + 1};
    bool modified = false;
    uint64_t pend;
    for (uint32_t c = wid; c < nchunks; c += kRedWaves) {
      const uint32_t p0 = c * cw;
      const uint32_t len = e - p0 < cw ? e - p0 : cw;
      reduce_members<G>(p0, len, cw / 4, e, s_mem, s_mroot, slab, g, r, hs, ts, samp, d.flags, det_cpy, deep_skip != 0,
                        gcur != kNoRoot ? s_tot : nullptr, nullptr, 0, 0, nullptr, &pend, r < last_round);
      const uint32_t hr = *hs.root, tr = *ts.root;
      if (hr != kNoRoot) {  // started in an earlier chunk
        uint64_t* acc = s_acc + (size_t)(s_seg[p0] / cw) * 2 * kWave;
        lds_xor(acc + lane, hs.vals[lane]);
        lds_xor(acc + kWave + lane, hs.vals[kWave + lane]);
      }
      if (tr != kNoRoot && tr != hr) {  // starts here and continues
        uint64_t* acc = s_acc + (size_t)c * 2 * kWave;
        lds_xor(acc + lane, ts.vals[lane]);
        lds_xor(acc + kWave + lane, ts.vals[kWave + lane]);
        if (lane == 0) s_accroot[c] = tr;
      }
      if (apply_sample(d, pend, hint)) modified = true;
    }
    pend = kSampZero;
    uint32_t pended = 0;  // the wave's samples of supernodes past a chunk, one to a lane
    __syncthreads();
    for (uint32_t c = wid; c < nchunks; c += kRedWaves) {
      const uint32_t R = s_accroot[c];
      if (R == kNoRoot) continue;
      uint64_t* acc = s_acc + (size_t)c * 2 * kWave;
      uint64_t idx;
      const int code = wave_sample<G>(acc[lane], (G)acc[kWave + lane], g.D, g.chk_bf, &idx);
      const uint64_t rec = sample_record(code, idx, g.n, d.flags);
      if (lane == pended++) pend = rec;
      acc[lane] = 0;  // zero for the next round
      acc[kWave + lane] = 0;
      if (lane == 0) s_accroot[c] = kNoRoot;
    }
    if (wid == kRedWaves - 1 && gcur != kNoRoot && e != 0) {  // the giant, from the complement
      uint64_t idx;
      const int code = wave_sample<G>(s_tot[lane], (G)s_tot[kWave + lane], g.D, g.chk_bf, &idx);
      const uint64_t rec = sample_record(code, idx, g.n, d.flags);
      if (lane == pended) pend = rec;
    }
    if (apply_sample(d, pend, hint)) modified = true;
    const bool any = __syncthreads_or(modified);
    if (tid == 0 && any) st_rlx(d.mod + r, 1u);
    if (!any || r >= last_round) {
      if (tid == 0) st_rlx(d.mod + (d.nmod - 1), r);
      if (rep) report();
      return;
    }
    // the next round walks this round's members
    walk = e;
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; ++k) {
      const bool in = tid + k * kRedBlock < walk;
      v[k] = in ? s_mem[tid + k * kRedBlock] : 0u;
      old[k] = in ? s_mroot[tid + k * kRedBlock] : 0u;
    }
    __syncthreads();
  }
}

// ConnectedComponents (src/return_types.cpp:5-19): root of every vertex and the root count.  The count
// takes one atomic per workgroup of 1024: one per wave with a root, on one address at 11 ns each, was
// the kernel's time on graphs with many components (2^20 R-MAT vertices, a third isolated: 169 us).
constexpr uint32_t kLabelBlock = 1024;
__global__ void __launch_bounds__(kLabelBlock)
k_labels(uint32_t* __restrict__ parent, uint32_t n, uint32_t* __restrict__ labels, uint32_t* __restrict__ ncc) {
  const uint32_t v = blockIdx.x * kLabelBlock + threadIdx.x;
  bool is_root = false;
  if (v < n) {
    const uint32_t r = dsu_find(parent, v);
    labels[v] = r;
    is_root = r == v;
  }
  const uint32_t roots = (uint32_t)__syncthreads_count(is_root);
  if (threadIdx.x == 0 && roots) atomicAdd(ncc, roots);
}
__global__ void k_point_queries(uint32_t* __restrict__ parent, const uint32_t* __restrict__ qa,
                                const uint32_t* __restrict__ qb, uint32_t nq, uint8_t* __restrict__ out) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nq; i += gridDim.x * blockDim.x)
    out[i] = dsu_find(parent, qa[i]) == dsu_find(parent, qb[i]) ? 1 : 0;
}

// The point queries of a query group and the error flags, read from and written to mapped host
// memory directly (a few words, so no copy launches around the kernel).
__global__ void k_answer_points(uint32_t* __restrict__ parent, const uint32_t* __restrict__ flags,
                                const uint32_t* __restrict__ q, uint32_t nq, uint32_t* __restrict__ out) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < kNumFlags) out[t] = flags[t];
  uint8_t* ans = reinterpret_cast<uint8_t*>(out + kNumFlags);
  for (uint32_t i = t; i < nq; i += gridDim.x * blockDim.x)
    ans[i] = dsu_find(parent, q[i]) == dsu_find(parent, q[nq + i]) ? 1 : 0;
  __threadfence_system();
}

// ================================================================================================
// Standalone sketch ops
// ================================================================================================
// Sketch::sample for any cols_per_sample: deterministic bucket first, then the sample's columns
// in bucket order; one wave walks them 64 buckets at a time.
template <class G>
__global__ void k_sketch_sample(const unsigned char* __restrict__ slab, Geo g, uint32_t sample_idx,
                                uint32_t* __restrict__ out) {
  const uint32_t lane = lane_id();
  uint64_t det_a;
  G det_g;
  ld_rec<G>(slab + rec_off<G>(g, 0, g.nb - 1), &det_a, &det_g);
  int code;
  uint64_t idx = 0;
  if (det_a == 0 && det_g == 0) {
    code = kZero;
  } else if ((G)xxh3_mix(xxh3_prep(det_a), g.chk_bf) == det_g) {
    code = kGood;
    idx = det_a;
  } else {
    code = kFail;
    const uint32_t b0 = sample_idx * g.cps * g.D, b1 = b0 + g.cps * g.D;
    for (uint32_t b = b0; b < b1; b += kWave) {
      const bool valid = b + lane < b1;
      uint64_t a = 0;
      G gm = 0;
      if (valid) ld_rec<G>(slab + rec_off<G>(g, 0, b + lane), &a, &gm);
      const bool good = valid && (G)xxh3_mix(xxh3_prep(a), g.chk_bf) == gm;
      const uint64_t mask = __ballot(good);
      if (mask) {
        idx = rd_lane_u64(a, __builtin_ctzll(mask));
        code = kGood;
        break;
      }
    }
  }
  if (lane == 0) {
    out[0] = (uint32_t)code;
    out[1] = (uint32_t)idx;
    out[2] = (uint32_t)(idx >> 32);
  }
}

template <class G>
__global__ void k_xor_range(unsigned char* __restrict__ dst, const unsigned char* __restrict__ src, Geo g,
                            uint32_t nsk, uint32_t b0, uint32_t cnt, int with_det) {
  const uint32_t per = cnt + (with_det ? 1 : 0);
  const size_t total = (size_t)nsk * per;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    const uint32_t s = (uint32_t)(i / per), k = (uint32_t)(i % per);
    const uint32_t b = k < cnt ? b0 + k : g.nb - 1;
    const size_t o = rec_off<G>(g, s, b);
    uint64_t da, sa;
    G dg, sg;
    ld_rec<G>(dst + o, &da, &dg);
    ld_rec<G>(src + o, &sa, &sg);
    st_rec<G>(dst + o, da ^ sa, (G)(dg ^ sg));
  }
}

// Packed reference image: record i of sketch v at byte (v * nb + i) * (8 + sizeof(G)); the slab row
// holds the same records, padding and the deep flags (set here for every deep record written
// nonzero; a stale set flag only costs the reduce a read).
template <class G, int MODE>  // 0 = xor image into slab, 1 = overwrite slab, 2 = slab to image
__global__ void k_packed(unsigned char* __restrict__ slab, Geo g, uint32_t v0, uint32_t nv,
                         unsigned char* __restrict__ packed) {
  const size_t rec = 8 + sizeof(G);
  const size_t total = (size_t)nv * g.nb;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    const uint32_t v = (uint32_t)(i / g.nb), b = (uint32_t)(i % g.nb);
    unsigned char* r = slab + rec_off<G>(g, v0 + v, b);
    uint64_t a, pa;
    G gm, pg;
    ld_rec<G>(r, &a, &gm);
    if (MODE == 2) {
      st_rec<G>(packed + i * rec, a, gm);
    } else {
      ld_rec<G>(packed + i * rec, &pa, &pg);
      const uint64_t na = MODE == 0 ? a ^ pa : pa;
      const G ng = MODE == 0 ? (G)(gm ^ pg) : pg;
      st_rec<G>(r, na, ng);
      if (kDeepFlags<G> && b != g.nb - 1 && (na | (uint64_t)ng) != 0) {
        const uint32_t c = b / g.D;
        if (rec_is_deep(g, b - c * g.D))
          st_rlx(reinterpret_cast<uint32_t*>(slab + (size_t)(v0 + v) * g.row + deep_flag_off(c)), 1u);
      }
    }
  }
}

// Bucket-wise XOR of every vertex sketch into out_a / out_g (nb entries each, zero on entry): one
// thread per (bucket, chunk of vertices), one device-scope atomic per thread.  The chunks are cut so
// that a small graph still fills the chip: 1024 vertices in one chunk took 290 us.
constexpr uint32_t kSumChunkMax = 1024, kSumChunks = 512;
uint32_t sum_chunk(uint32_t n) {
  const uint32_t c = (n + kSumChunks - 1) / kSumChunks;
  return c < 4 ? 4 : c > kSumChunkMax ? kSumChunkMax : c;
}
template <class G>
__global__ void __launch_bounds__(256)
k_sum_all(const unsigned char* __restrict__ slab, Geo g, uint32_t chunk, uint64_t* __restrict__ out_a,
          G* __restrict__ out_g) {
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= g.nb) return;
  const uint32_t v0 = blockIdx.y * chunk;
  const uint32_t v1 = v0 + chunk < g.n ? v0 + chunk : g.n;
  uint64_t a = 0;
  G gm = 0;
  for (uint32_t v = v0; v < v1; ++v) {
    uint64_t ra;
    G rg;
    ld_rec<G>(slab + rec_off<G>(g, v, b), &ra, &rg);
    a ^= ra;
    gm ^= rg;
  }
  if (a) gbl_xor(out_a + b, a);
  if (gm) gbl_xor(out_g + b, gm);
}

// Order-sensitive digest of every vertex's bucket array:
//   D = sum over vertices v, buckets b of fmix64(x + pos), pos = v*nb + b,
//   x = alpha ^ fmix64(gamma ^ pos * 0x9E3779B97F4A7C15)   (all mod 2^64)
// A sum is independent of reduction order, so the value is deterministic.
//
// A wave takes 64 buckets of every vertex of a chunk: its record offsets are computed once, the positions
// go up by nb, and no record costs a division.  One atomic per workgroup of 16 waves, at most
// kDigestGrid of them: 16384 of them, one per wave, on the one word took 180 us by themselves.
// Now bound by the read: five graphs of 2^12 to 2^17 vertices (2.7 GB) 1261 -> 649 us in all.
constexpr uint32_t kDigestBlock = 1024, kDigestGrid = 1024;
template <class G>
__global__ void __launch_bounds__(kDigestBlock)
k_digest(const unsigned char* __restrict__ slab, Geo g, uint32_t groups, uint32_t chunk,
         unsigned long long* __restrict__ out) {
  constexpr uint64_t kPhi = 0x9E3779B97F4A7C15ULL;
  __shared__ uint64_t s_sum[kDigestBlock / kWave];
  const uint32_t wave = blockIdx.x * (kDigestBlock / kWave) + threadIdx.x / kWave;
  const uint32_t b = wave % groups * kWave + lane_id();
  const uint64_t first = (uint64_t)(wave / groups) * chunk;
  uint64_t acc = 0;
  if (b < g.nb && first < g.n) {
    const uint32_t v0 = (uint32_t)first, v1 = g.n - v0 < chunk ? g.n : v0 + chunk;
    const unsigned char* p = slab + rec_off<G>(g, v0, b);
    uint64_t pos = (uint64_t)v0 * g.nb + b, mul = pos * kPhi;
    const uint64_t step = g.nb * kPhi;
#pragma unroll 4
    for (uint32_t v = v0; v < v1; ++v) {
      uint64_t a;
      G gm;
      ld_rec<G>(p, &a, &gm);
      acc += mix64((a ^ mix64((uint64_t)gm ^ mul)) + pos);
      p += g.row;
      pos += g.nb;
      mul += step;
    }
  }
  for (int o = 32; o > 0; o >>= 1) acc += shfl_u64(acc, (int)(lane_id() ^ (uint32_t)o));
  if (lane_id() == 0) s_sum[threadIdx.x / kWave] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < kDigestBlock / kWave; ++w) acc += s_sum[w];
    atomicAdd(out, (unsigned long long)acc);
  }
}

}  // namespace

// ================================================================================================
// launchers
// ================================================================================================
void launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n, 256)), dim3(256), 0, s, p, v, n);
}
void launch_fill_u64(uint64_t* p, uint64_t v, size_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(n, 256)), dim3(256), 0, s, p, v, n);
}

size_t update_tiles_lds_bytes(const Geo& g, int gbytes) {
  const size_t lds_n = (size_t)g.C * lds_depth(g.C, gbytes) + 1;
  return kWave * 16 + g.C * 8 + lds_n * 8 + (lds_n + kWave) * (size_t)gbytes + lds_n * 2;
}

void launch_update_tiles(int gbytes, const Tile* tiles, const uint32_t* ntiles_dev, uint32_t ntiles_host,
                         uint32_t grid_cap, const uint32_t* dsts, unsigned char* slab, const Geo& g,
                         const uint64_t* col_bf, hipStream_t s) {
  // tile count known on the host: one workgroup per tile (capped, then grid-stride);
  // known only on the device: a persistent grid of grid_cap workgroups
  uint32_t grid = ntiles_dev ? grid_cap : (grid_cap && ntiles_host > grid_cap ? grid_cap : ntiles_host);
  if (grid == 0) return;
  const size_t lds = update_tiles_lds_bytes(g, gbytes);
  const uint32_t ldepth = lds_depth(g.C, gbytes);
  const bool wide = g.C * ldepth + 1 > kPerLane * kWave;
  const uint32_t rb = 8 + gbytes, end = std::min(g.D, ldepth);  // the last column's deepest place in the delta
  if (g.ovf + (end > g.low ? (g.C - 1) * g.opitch + (end - 1 - g.low) * rb : 0u) > 4u * 0xFFFFu)
    throw std::logic_error("a row's records lie past the update kernel's 16-bit places");
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kWave), lds, s, tiles, ntiles_dev, ntiles_host, dsts, slab, g, col_bf,
                       ldepth, 65536 / ldepth + 1);
  };
  if (gbytes == 4) wide ? go(k_update_tiles<uint32_t, true>) : go(k_update_tiles<uint32_t, false>);
  else wide ? go(k_update_tiles<uint64_t, true>) : go(k_update_tiles<uint64_t, false>);
}

void launch_sketch_update(int gbytes, const uint64_t* idx, size_t count, unsigned char* slab, const Geo& g,
                          const uint64_t* col_bf, hipStream_t s) {
  if (!count) return;
  const uint32_t depth = g.C <= kOneMaxCols ? kOneDepth : kLdsDepthMin;
  const uint32_t lds_n = g.C * depth + 1;
  // Lanes of an index: as many as one workgroup has for the batch, at most a wave's or one per column.  Its
  // threads then also cover the delta's entries, which a wave alone would clear and write back in up to 80
  // steps.
  uint32_t sub = 0;
  while (sub < 6 && (1u << sub) < g.C && (count << (sub + 1)) <= kOneBlock) ++sub;
  const size_t work = sub ? std::max<size_t>(count << sub, lds_n) : count;
  const uint32_t block = (uint32_t)std::min<size_t>(kOneBlock, (work + kWave - 1) / kWave * kWave);
  const uint32_t grid = sub ? 1u : (uint32_t)std::min<size_t>(kOneGrid, (count + block - 1) / block);
  const size_t lds = g.C * size_t(8) + (size_t)lds_n * (8 + gbytes);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(block), lds, s, idx, count, slab, g, col_bf, depth, sub);
  };
  if (gbytes == 4) sub ? go(k_sketch_update<uint32_t, true>) : go(k_sketch_update<uint32_t, false>);
  else sub ? go(k_sketch_update<uint64_t, true>) : go(k_sketch_update<uint64_t, false>);
}

size_t group_partials_len(uint32_t n) { return (n + kScanSpan - 1) / kScanSpan + 1; }

// Entries from which records move through LDS: with fewer than 1024 bins of 8192 entries, the open
// lines fit the L2s, and the direct writes (12 us for 730k updates) take no sorting.
constexpr size_t kStagedMin = size_t(1) << 23;
// Bits of a vertex's place, and the log2 of a bin's vertices.
struct PartShape {
  uint32_t nb, shift;
};
uint32_t part_bits(uint32_t n) {
  uint32_t nb = 5;
  while (nb < 24 && (1u << nb) < n) ++nb;
  return nb;
}
// One-word records: with at least 1024 bins, at most nb - 10 bits of place stand beside nb bits of id.
bool part_packed(uint32_t n) { return part_bits(n) <= 21; }
// About 8192 entries a bin (what a workgroup keeps in registers between its passes), at least 64 bins
// and at most kPartBins, of at most 2^kPartMaxShift vertices (the LDS counters) and at least 8.
PartShape part_shape(uint32_t n, size_t count) {
  const uint32_t nb = part_bits(n);
  uint32_t lb = 6;
  while (lb < 10 && (size_t(8192) << lb) < 2 * count) ++lb;
  if (part_packed(n) && 2 * nb > 32 + lb) lb = 2 * nb - 32;
  if (nb > kPartMaxShift + lb) lb = nb - kPartMaxShift;
  if (lb + 3 > nb) lb = nb - 3;
  return PartShape{nb, nb - lb};
}

void launch_group(const uint32_t* pairs, size_t count, uint32_t n, uint32_t tile, const GroupBufs& b, hipStream_t s,
                  const FlushBytes* fb) {
  const uint2* p2 = reinterpret_cast<const uint2*>(pairs);
  uint64_t* acc = fb ? fb->acc : nullptr;
  const uint64_t S = fb ? fb->S : 0, per_update = fb ? fb->per_update : 0;
  if (!count) {
    launch_fill_u32(b.totals, 0, 2, s);
    return;
  }
  if (count <= kSmallPairs) {
    uint32_t tbits = 10;
    while ((2 * count) > (size_t(3) << tbits) / 4) ++tbits;  // at most three quarters full
    const size_t lds = (size_t(8) << tbits);
    hipLaunchKernelGGL(k_group_small, dim3(1), dim3(kPartBlock), lds, s, p2, (uint32_t)count, n, tbits, b.totals,
                       b.dst_arr, tile, b.tiles, acc, S, per_update, b.bad);
    return;
  }
  if (b.rec) {
    const PartShape sh = part_shape(n, count);
    const uint32_t nblk = (uint32_t)std::min<size_t>(kPartMaxBlocks, (count + 4095) / 4096);
    const uint32_t bins = 1u << (sh.nb - sh.shift);
    const size_t lds = size_t(4) << sh.shift;
    hipLaunchKernelGGL(k_part_hist, dim3(nblk), dim3(kPartBlock), 0, s, p2, count, n, sh.nb, sh.shift, bins, nblk,
                       b.binned, b.place, b.totals, b.bad);
    auto go = [&](auto pack, auto staged) {
      constexpr bool PACK = decltype(pack)::value, STAGED = decltype(staged)::value;
      using R = typename PartRec<PACK>::T;
      R* rec = reinterpret_cast<R*>(b.rec);
      hipLaunchKernelGGL((k_part_scatter<PACK, STAGED>), dim3(nblk), dim3(kPartBlock), STAGED ? StageLds<R>::bytes() : 0,
                         s, p2, count, n, sh.nb, sh.shift, bins, nblk, b.binned, b.place, b.binoff, rec);
      hipLaunchKernelGGL(k_part_group<PACK>, dim3(bins), dim3(kPartBlock), lds, s, rec, sh.nb, sh.shift, b.binned,
                         b.binoff, b.totals, b.dst_arr, tile, b.tiles, acc, S, per_update);
    };
    const std::true_type yes{};
    const std::false_type no{};
    const bool large = 2 * count >= kStagedMin;
    if (part_packed(n)) large ? go(yes, yes) : go(yes, no);
    else large ? go(no, yes) : go(no, no);
    return;
  }
  launch_fill_u32(b.cnt, 0, n, s);
  hipLaunchKernelGGL(k_count_pairs, dim3(grid_for(count, 256)), dim3(256), 0, s, p2, count, n, b.cnt, b.bad);
  scan_counts(b.cnt, n, tile, b.partials, b.off, b.toff, b.cursor, b.totals, s);
  hipLaunchKernelGGL(k_scatter_pairs, dim3(grid_for(count, 256)), dim3(256), 0, s, p2, count, n, b.cursor, b.dst_arr);
  hipLaunchKernelGGL(k_make_tiles, dim3(grid_for(n, 256, kProfSlots)), dim3(256), 0, s, b.cnt, b.off, b.toff, n, tile,
                     b.tiles, acc, S, per_update);
}

size_t part_place_len() { return (size_t)kPartBins * kPartMaxBlocks; }
size_t part_bins_len() { return kPartBins + 1; }

// A large batch on an instance that no query has ranked gets classes first and is merged in launches
// of doubling size.  The time of the first merges is failed CAS attempts on hubs' words: every update
// in flight that joins two hubs' components tries the lower hub.  With hubs ranked first and few
// updates in flight until the largest component holds the hubs, the rest mostly find themselves
// connected.  First batch of 936k updates on 2^17 vertices, median of 5, one launch unranked -> this:
// R-MAT 2249 -> 157 us, uniform 963 -> 267; 1M Chung-Lu updates on 2^18 vertices 1932 -> 210.  With
// first launches of 32768 or steps of 8 it takes up to ten times as long.  Below kRankMin one launch
// costs less than these.
constexpr size_t kRankMin = 32768, kRankFirst = 8192;
// Updates in all and per vertex from which a batch looks its updates up in the component's bits first,
// and the vertices whose bits fit a workgroup's LDS.  24M updates on a connected graph of 2^18 vertices
// 298 -> 101 us with the bits' launch, 16M R-MAT on 2^20 277 -> 198 (the rest fills the forest set), 1M
// on 2^17 36 -> 24; 512k on 2^15 vertices in 64 components 22 -> 27.
constexpr size_t kMapMin = 4, kMapMinCount = size_t(1) << 20;
constexpr uint32_t kMapMaxVertices = 1u << 20;
void launch_eager(const uint32_t* src, uint32_t* pairs, size_t count, uint8_t* merged, const DsuDev& d,
                  hipStream_t s, bool build_sf, unsigned char* hint, bool ranked, uint64_t* map) {
  if (!count) return;
  uint2* p2 = reinterpret_cast<uint2*>(pairs);
  const uint2* s2 = reinterpret_cast<const uint2*>(src);
  const uint32_t grid = grid_for(count, 256);
  size_t lo = 0, hi = count;
  if (!ranked && count >= kRankMin) {
    hipLaunchKernelGGL(k_eager_rank, dim3(grid), dim3(256), 0, s, s2, count, d.n, hint);
    hi = std::min(count, kRankFirst);
  }
  while (lo < count) {
    const size_t m = hi - lo;
    if (m >= kMapMinCount && m >= kMapMin * (size_t)d.n && d.n <= kMapMaxVertices) {
      hipLaunchKernelGGL(k_dsu_map, dim3((d.n + 255) / 256), dim3(256), 0, s, d, map);
      hipLaunchKernelGGL(k_eager_union<true>, dim3(grid_for(m, 1024, 512)), dim3(1024), ((size_t)d.n + 31) / 32 * 4, s,
                         s2 + lo, p2 + lo, m, merged + lo, d, build_sf ? 1u : 0u, hint,
                         reinterpret_cast<const uint32_t*>(map));
    } else {
      const uint32_t ugrid = build_sf ? std::max(grid_for(m, 256), grid_for(d.n, 256, 4096)) : grid_for(m, 256);
      hipLaunchKernelGGL(k_eager_union<false>, dim3(ugrid), dim3(256), 0, s, s2 + lo, p2 + lo, m, merged + lo, d,
                         build_sf ? 1u : 0u, hint, nullptr);
    }
    build_sf = false;
    lo = hi;
    hi = std::min(count, 2 * hi);
  }
  hipLaunchKernelGGL(k_eager_sf_check, dim3(grid), dim3(256), 0, s, p2, count, merged, d);
}


void launch_dsu_reset(const DsuDev& d, hipStream_t s, const RoundBufs* rb) {
  const size_t work = std::max<size_t>(d.n, d.sf_mask + 1);
  hipLaunchKernelGGL(k_dsu_reset, dim3(grid_for(work, 256)), dim3(256), 0, s, d.parent, d.n, d.sf_hash,
                     d.sf_mask + 1, d.sf_edge, d.flags, d.mod, d.nmod, rb ? rb->cnt : nullptr,
                     rb ? rb->totals : nullptr, rb ? d.query_force : nullptr);
}

void launch_round_state_init(const RoundBufs& rb, uint32_t n, hipStream_t s) {
  launch_fill_u32(rb.totals, 0, kStWords, s);
  launch_fill_u32(rb.totals + kStGiantRound, kNoRoot, 1, s);
  launch_fill_u32(rb.totals + kStGiantFirst, kNoRoot, 1, s);
  launch_fill_u32(rb.members[0], 0, n, s);
  launch_fill_u32(rb.members[1], 0, n, s);
  launch_fill_u32(rb.mroot[0], 0, n, s);
  launch_fill_u32(rb.mroot[1], 0, n, s);
}

void launch_sample_round0(int gbytes, const unsigned char* slab, const Geo& g, const DsuDev& d, const RoundBufs& rb,
                          hipStream_t s) {
  uint64_t* samp = rb.samp;
  const uint32_t grid = grid_for((size_t)(g.n + 3) / 4 * kWave, 256, 16384);
  if (gbytes == 4)
    hipLaunchKernelGGL(k_sample_round0<uint32_t>, dim3(grid), dim3(256), 0, s, slab, g, samp, d.flags, rb.det_cpy,
                       rb.hint, d);
  else
    hipLaunchKernelGGL(k_sample_round0<uint64_t>, dim3(grid), dim3(256), 0, s, slab, g, samp, d.flags, rb.det_cpy,
                       rb.hint, d);
  hipLaunchKernelGGL(k_apply_samples, dim3(grid_for(g.n, 256, 4096)), dim3(256), 0, s, samp, d, rb.hint);
}

// Entries per wave of the reduce: 64, but 16 in rounds of at most upto16 entries and 32 up to upto32.  Up
// to 256 workgroups of 16 waves, fewer entries per wave cost nothing but bring in more CUs: 64 entries
// per wave would leave a round of 32k entries on 32 of 256 CUs, each waiting for 16 loads per lane and
// sampling for 16 waves.  Past that they cost atomics on the sums of supernodes that cross workgroups,
// which a round much smaller than n, grouped into few supernodes or mostly into the giant, has less of.
// Against bounds of n / 16 and n / 2 alone: reduces of 2^17 vertices with 8-byte checksums 29.3 -> 24.9 us
// on average, of 2^18 31.3 -> 29.7, of 1000 vertices 23.4 -> 15.4.
struct ReduceShape {
  uint32_t upto16, upto32;
  explicit ReduceShape(uint32_t n)
      : upto16(std::max(n / 16, 256u * kRedWaves * 16)), upto32(std::max(n / 2, 256u * kRedWaves * 32)) {}
};
// Workgroups of a reduce, for any round of at most n entries.
uint32_t reduce_blocks(uint32_t n) {
  const ReduceShape s(n);
  auto blocks = [](uint32_t entries, uint32_t per_wave) {
    return (uint32_t)(((uint64_t)entries + kRedWaves * per_wave - 1) / (kRedWaves * per_wave));
  };
  return std::max({1u, blocks(std::min(n, s.upto16), 16), blocks(std::min(n, s.upto32), 32), blocks(n, 64)});
}

void launch_round(int gbytes, uint32_t round, const unsigned char* slab, const Geo& g,
                  const DsuDev& d, const RoundBufs& rb, bool giant_ok, bool drop_ok, hipStream_t s, bool deep_skip) {
  const uint32_t n = g.n;
  const uint32_t* prev = d.mod + (round - 1);
  uint32_t* cur = d.mod + round;
  uint32_t* st = rb.totals;
  const uint32_t par = round & 1, opar = (round - 1) & 1;
  uint32_t* members = rb.members[par];
  const uint32_t grid = (n + kAggBlock - 1) / kAggBlock;  // one vertex, or one old segment, per thread
  if (round == 1) {  // every vertex in id order
    const uint32_t* act_list = rb.members[opar];  // not read in round 1
    hipLaunchKernelGGL(k_bv_find_count, dim3(grid), dim3(kAggBlock), 0, s, d.parent, n, rb.nd, rb.cnt, st, round,
                       act_list, prev);
    hipLaunchKernelGGL(k_bv_alloc, dim3(grid), dim3(kAggBlock), 0, s, rb.cnt, n, rb.off, rb.cursor, st, round,
                       act_list, giant_ok ? 1u : 0u, prev, rb.segs[par], rb.samp, drop_ok ? 1u : 0u);
    hipLaunchKernelGGL(k_bv_scatter, dim3(grid), dim3(kAggBlock), 0, s, rb.nd, n, rb.off, members, rb.mroot[par],
                       st, round, act_list, prev);
  } else {  // whole runs of the previous round's member list
    const SegOut out{rb.off, rb.cursor, rb.segs[par]};
    hipLaunchKernelGGL(k_seg_find, dim3(grid), dim3(kAggBlock), 0, s, d.parent, n, rb.cnt, rb.nd, out, st, round,
                       rb.segs[opar], giant_ok ? 1u : 0u, prev, rb.samp, drop_ok ? 1u : 0u);
    hipLaunchKernelGGL(k_seg_alloc, dim3(grid), dim3(kAggBlock), 0, s, rb.cnt, n, rb.nd, out, st, round,
                       rb.segs[opar], giant_ok ? 1u : 0u, prev, rb.samp, drop_ok ? 1u : 0u);
    hipLaunchKernelGGL(k_seg_copy, dim3(grid_for(n, 256)), dim3(256), 0, s, n, rb.nd, rb.off, d.parent, rb.members[opar],
                       rb.mroot[opar], members, rb.mroot[par], st, round, prev);
  }
  // one accumulator slot per workgroup and one for the giant
  const uint32_t rgrid = reduce_blocks(n);
  const ReduceShape shape(n);
  if (rgrid + 1 > rb.xslots) throw std::logic_error("reduce grid exceeds its cross-workgroup accumulator slots");
  const XAcc xa{rb.xacc, rb.xcnt, rb.xslots, rb.off, rb.cursor};
  if (gbytes == 4)
    hipLaunchKernelGGL(k_bv_reduce<uint32_t>, dim3(rgrid), dim3(kRedBlock), 0, s, st, members, rb.mroot[par],
                       slab, g, round, xa, rb.samp, d, prev, cur, rb.rstats, rb.det_cpy, rb.hint, shape.upto16,
                       shape.upto32, deep_skip ? 1u : 0u);
  else
    hipLaunchKernelGGL(k_bv_reduce<uint64_t>, dim3(rgrid), dim3(kRedBlock), 0, s, st, members, rb.mroot[par],
                       slab, g, round, xa, rb.samp, d, prev, cur, rb.rstats, rb.det_cpy, rb.hint, shape.upto16,
                       shape.upto32, deep_skip ? 1u : 0u);
}

bool launch_finish(int gbytes, uint32_t r0, uint32_t last_round, const unsigned char* slab, const Geo& g,
                   const DsuDev& d, const RoundBufs& rb, hipStream_t s, uint32_t* rep, bool deep_skip) {
  if (r0 < 2 || r0 > last_round) return false;  // round r0 walks round r0 - 1's member list
  const uint32_t* act0 = rb.members[(r0 - 1) & 1];
  const uint32_t* mroot0 = rb.mroot[(r0 - 1) & 1];
  if (gbytes == 4)
    hipLaunchKernelGGL(k_bv_finish<uint32_t>, dim3(1), dim3(kRedBlock), 0, s, d, rb.totals, act0, mroot0, slab, g, r0,
                       last_round, rb.samp, rb.rstats, rb.det_cpy, rb.hint, rep, deep_skip ? 1u : 0u);
  else
    hipLaunchKernelGGL(k_bv_finish<uint64_t>, dim3(1), dim3(kRedBlock), 0, s, d, rb.totals, act0, mroot0, slab, g, r0,
                       last_round, rb.samp, rb.rstats, rb.det_cpy, rb.hint, rep, deep_skip ? 1u : 0u);
  return true;
}
uint32_t finish_max() { return kFinishMax; }


void launch_sum_all(int gbytes, const unsigned char* slab, const Geo& g, uint64_t* out_a, void* out_g, hipStream_t s) {
  launch_fill_u64(out_a, 0, g.nb, s);
  if (gbytes == 4) launch_fill_u32((uint32_t*)out_g, 0, g.nb, s);
  else launch_fill_u64((uint64_t*)out_g, 0, g.nb, s);
  const uint32_t chunk = sum_chunk(g.n);
  const dim3 grid((g.nb + 255) / 256, (g.n + chunk - 1) / chunk);
  if (gbytes == 4)
    hipLaunchKernelGGL(k_sum_all<uint32_t>, grid, dim3(256), 0, s, slab, g, chunk, out_a, (uint32_t*)out_g);
  else
    hipLaunchKernelGGL(k_sum_all<uint64_t>, grid, dim3(256), 0, s, slab, g, chunk, out_a, (uint64_t*)out_g);
}

void launch_digest(int gbytes, const unsigned char* slab, const Geo& g, uint64_t* out, hipStream_t s) {
  launch_fill_u64(out, 0, 1, s);
  constexpr uint32_t waves = kDigestBlock / kWave;
  const uint32_t groups = (g.nb + kWave - 1) / kWave;
  const uint32_t chunks = std::min(std::max(1u, kDigestGrid * waves / groups), std::max(1u, g.n / 8));
  const uint32_t chunk = (g.n + chunks - 1) / chunks;
  const uint32_t total = groups * ((g.n + chunk - 1) / chunk);
  const dim3 grid((total + waves - 1) / waves);
  auto* o = reinterpret_cast<unsigned long long*>(out);
  if (gbytes == 4)
    hipLaunchKernelGGL(k_digest<uint32_t>, grid, dim3(kDigestBlock), 0, s, slab, g, groups, chunk, o);
  else
    hipLaunchKernelGGL(k_digest<uint64_t>, grid, dim3(kDigestBlock), 0, s, slab, g, groups, chunk, o);
}

void launch_labels(const DsuDev& d, uint32_t* labels, uint32_t* ncc, hipStream_t s) {
  launch_fill_u32(ncc, 0, 1, s);
  hipLaunchKernelGGL(k_labels, dim3((d.n + kLabelBlock - 1) / kLabelBlock), dim3(kLabelBlock), 0, s, d.parent, d.n, labels, ncc);
}
void launch_answer_points(const DsuDev& d, const uint32_t* q, uint32_t nq, uint32_t* out, hipStream_t s) {
  hipLaunchKernelGGL(k_answer_points, dim3(grid_for(nq > kNumFlags ? nq : kNumFlags, 256)), dim3(256), 0, s, d.parent,
                     d.flags, q, nq, out);
}
void launch_point_queries(const DsuDev& d, const uint32_t* qa, const uint32_t* qb, uint32_t nq, uint8_t* out,
                          hipStream_t s) {
  if (!nq) return;
  hipLaunchKernelGGL(k_point_queries, dim3(grid_for(nq, 256)), dim3(256), 0, s, d.parent, qa, qb, nq, out);
}

void launch_sketch_sample(int gbytes, const unsigned char* slab, const Geo& g, uint32_t sample_idx, uint32_t* out,
                          hipStream_t s) {
  if (gbytes == 4)
    hipLaunchKernelGGL(k_sketch_sample<uint32_t>, dim3(1), dim3(kWave), 0, s, slab, g, sample_idx, out);
  else
    hipLaunchKernelGGL(k_sketch_sample<uint64_t>, dim3(1), dim3(kWave), 0, s, slab, g, sample_idx, out);
}
void launch_xor_range(int gbytes, unsigned char* dst, const unsigned char* src, const Geo& g, uint32_t nsk, uint32_t b0,
                      uint32_t cnt, bool with_det, hipStream_t s) {
  const size_t total = (size_t)nsk * (cnt + (with_det ? 1 : 0));
  if (!total) return;
  if (gbytes == 4)
    hipLaunchKernelGGL(k_xor_range<uint32_t>, dim3(grid_for(total, 256)), dim3(256), 0, s, dst, src, g, nsk, b0, cnt,
                       with_det ? 1 : 0);
  else
    hipLaunchKernelGGL(k_xor_range<uint64_t>, dim3(grid_for(total, 256)), dim3(256), 0, s, dst, src, g, nsk, b0, cnt,
                       with_det ? 1 : 0);
}

template <int MODE>
static void launch_packed(int gbytes, unsigned char* slab, const Geo& g, uint32_t v0, uint32_t nv, const void* packed,
                          hipStream_t s) {
  const size_t total = (size_t)nv * g.nb;
  if (!total) return;
  unsigned char* p = (unsigned char*)packed;
  if (gbytes == 4)
    hipLaunchKernelGGL((k_packed<uint32_t, MODE>), dim3(grid_for(total, 256)), dim3(256), 0, s, slab, g, v0, nv, p);
  else
    hipLaunchKernelGGL((k_packed<uint64_t, MODE>), dim3(grid_for(total, 256)), dim3(256), 0, s, slab, g, v0, nv, p);
}
void launch_merge_packed(int gbytes, unsigned char* slab, const Geo& g, uint32_t v0, uint32_t nv, const void* packed,
                         hipStream_t s) {
  launch_packed<0>(gbytes, slab, g, v0, nv, packed, s);
}
void launch_unpack(int gbytes, unsigned char* slab, const Geo& g, uint32_t v0, uint32_t nv, const void* packed,
                   hipStream_t s) {
  launch_packed<1>(gbytes, slab, g, v0, nv, packed, s);
}
void launch_pack(int gbytes, const unsigned char* slab, const Geo& g, uint32_t v0, uint32_t nv, void* packed,
                 hipStream_t s) {
  launch_packed<2>(gbytes, const_cast<unsigned char*>(slab), g, v0, nv, packed, s);
}

}  // namespace gz
