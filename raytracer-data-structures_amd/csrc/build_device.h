// Block-level device functions of the LBVH build (Morton -> onesweep radix
// sort -> Karras emission -> two-pass refit). Each function is one unit of
// work for one block of BUILD_BLOCK (256) threads (the triangle passes take
// the block size as a parameter): the standalone kernels in
// build_kernels.hip launch one block per unit, the batch kernels in
// batch_kernels.hip one per unit of every mesh. LDS scratch is
// passed in so that a kernel calling several phases holds one buffer.
//
// Replaces constructLBVHTree (accelerators.h:570-586): its Morton step
// (morton3D :385-394 on (centre + 30)/1000, :577), its sort (the decimal LSD
// radixSort :348-369, which sorts a discarded copy) and its tree step (the
// median split :452-564); results are bit-exact with the CPU restatement in
// oracle/.
#pragma once
#include "rq_internal.h"

namespace rq {

constexpr int BUILD_BLOCK = 256;
constexpr int TRI_TILE = 4096;   // triangles per bounds / Morton unit
constexpr int NODE_TILE = 4096;  // internal nodes per Karras unit
// LDS words needed by the largest phase (the onesweep tile)
__host__ __device__ constexpr int sort_lds_words(int items) {
  return SORT_WAVES * 256 + SORT_BLOCK * items + 256 + 256 + 2 * SORT_WAVES;
}
constexpr int BUILD_LDS_WORDS = sort_lds_words(SORT_ITEMS);

// Everything one mesh build reads and writes.
// Triangles: vx/vy/vz vertices, idx 3 per primitive, vr null. Spheres
// (the reference's primitive, accelerators.h:54-92): vx/vy/vz centres, vr
// radii, idx unused.
struct BuildView {
  const float *vx, *vy, *vz;
  const uint32_t* idx;
  uint32_t n;
  int mode;
  BuildBuffers B;
  const float* vr = nullptr;
  int32_t sphere = 0;  // vr is set (an integer flag: device code tests it, not the pointer)
};

// ---- helpers ------------------------------------------------------------------
// Element i of a per-primitive array (i < MAX_PRIMS < 2^30): the byte offset
// fits 32 bits, so the access takes a scalar base and a 32-bit lane offset
// (one VGPR per address instead of a 64-bit pair).
template <typename T>
__device__ inline T& el32(T* base, uint32_t i) {
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + (uint32_t)(i * (uint32_t)sizeof(T)));
}
template <typename T>
__device__ inline const T& el32(const T* base, uint32_t i) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) +
                                     (uint32_t)(i * (uint32_t)sizeof(T)));
}
__device__ inline uint32_t f2ord(float f) {
  uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float ord2f(uint32_t u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

// Spread the 10 low bits of v to bit positions 3k (shift-or-mask form).
__device__ inline uint32_t spread3(uint32_t v) {
  v &= 0x3FFu;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

// morton3D semantics (accelerators.h:387-393): clamp(a*1024, 0, 1023) with
// the std::max/std::min comparisons, truncate, x is the high bit of a triple.
__device__ inline uint32_t quant10(float a) {
  a = a * 1024.0f;
  a = (a < 0.0f) ? 0.0f : a;
  a = (1023.0f < a) ? 1023.0f : a;
  return (a != a) ? 0u : (uint32_t)a;
}
__device__ inline uint32_t morton30(float x, float y, float z) {
  return (spread3(quant10(x)) << 2) | (spread3(quant10(y)) << 1) | spread3(quant10(z));
}

// Triangle centroid ((v0 + v1) + v2) / 3 per axis; a sphere's centre
// (main.cpp:680-683 places each object at its centre). Zeros canonicalised.
__device__ inline float3 centroid(const BuildView& v, uint32_t t) {
  if (v.sphere) return make_float3(v.vx[t] + 0.0f, v.vy[t] + 0.0f, v.vz[t] + 0.0f);
  const uint32_t a = v.idx[3 * t], b = v.idx[3 * t + 1], c = v.idx[3 * t + 2];
  float3 r;
  r.x = ((v.vx[a] + v.vx[b]) + v.vx[c]) / 3.0f + 0.0f;
  r.y = ((v.vy[a] + v.vy[b]) + v.vy[c]) / 3.0f + 0.0f;
  r.z = ((v.vz[a] + v.vz[b]) + v.vz[c]) / 3.0f + 0.0f;
  return r;
}

__device__ inline uint32_t ld_agent(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_agent(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Inclusive scan across the 64 lanes of a wave.
__device__ inline uint32_t wave_incl_scan(uint32_t v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

__host__ __device__ inline uint32_t tiles_of(uint32_t n, uint32_t tile) {
  return (n + tile - 1) / tile;
}

// ---- phase 0: reset the build's counters, histograms and look-back words --------
// Threads [first, first + stride) of the caller's grid share the work.
__device__ inline void build_init_misc(const BuildView& v, uint32_t first, uint32_t stride) {
  uint32_t* misc = v.B.misc;
  for (uint32_t k = first; k < (uint32_t)MISC_BOUNDS; k += stride) misc[k] = 0u;  // hist, tickets
  if (first == 0) misc[MISC_ERR] = 0u, misc[MISC_HEIGHT] = HEIGHT_UNKNOWN;
  if (first < 3) {
    misc[MISC_BOUNDS + first] = 0xFFFFFFFFu;  // lo (ordered min)
    misc[MISC_BOUNDS + 3 + first] = 0u;        // hi (ordered max)
  }
}
__device__ inline void build_init_status(const BuildView& v, uint32_t first, uint32_t stride) {
  const uint32_t nstatus = SORT_PASSES * tiles_of(v.n, SORT_TILE_LEAN) * 256;  // both tilings
  for (uint32_t k = first; k < nstatus; k += stride) v.B.status[k] = 0u;
}
__device__ inline void build_init_part(const BuildView& v, uint32_t first, uint32_t stride) {
  build_init_status(v, first, stride);
  build_init_misc(v, first, stride);
}

// The centroids of primitives t, t + BLOCK, ... below end (the last one again
// past it): their index and vertex fetches are in flight together.
constexpr int CENTROIDS = 4;
template <int BLOCK>
__device__ inline void centroids(const BuildView& v, uint32_t t, uint32_t end, float3* c) {
#pragma unroll
  for (int j = 0; j < CENTROIDS; ++j) c[j] = centroid(v, min(t + j * BLOCK, end - 1u));
}

// ---- phase 1: centroid bounds of one tile (SCENE_AABB map) ------------------------
template <int BLOCK = BUILD_BLOCK>
__device__ inline void bounds_tile(const BuildView& v, uint32_t tile, uint32_t* lds) {
  constexpr int W = BLOCK / 64;  // waves; lds holds 6 * W words
  uint32_t lo[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, hi[3] = {0u, 0u, 0u};
  const uint32_t end = min((tile + 1) * (uint32_t)TRI_TILE, v.n);
  for (uint32_t t = tile * TRI_TILE + threadIdx.x; t < end; t += CENTROIDS * BLOCK) {
    float3 c[CENTROIDS];
    centroids<BLOCK>(v, t, end, c);  // (a clamped index repeats one: no harm)
#pragma unroll
    for (int j = 0; j < CENTROIDS; ++j) {
      const uint32_t o[3] = {f2ord(c[j].x), f2ord(c[j].y), f2ord(c[j].z)};
#pragma unroll
      for (int k = 0; k < 3; ++k) lo[k] = min(lo[k], o[k]), hi[k] = max(hi[k], o[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      lo[k] = min(lo[k], (uint32_t)__shfl_xor((int)lo[k], off, 64));
      hi[k] = max(hi[k], (uint32_t)__shfl_xor((int)hi[k], off, 64));
    }
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < 3; ++k) lds[k * W + wave] = lo[k], lds[(3 + k) * W + wave] = hi[k];
  }
  __syncthreads();
  if (threadIdx.x < 6) {  // at most one device atomic per bound per tile: they
                          // queue on one line, so one that changes nothing is left out
    const int k = threadIdx.x;
    uint32_t m = lds[k * W];
    for (int w = 1; w < W; ++w) m = k < 3 ? min(m, lds[k * W + w]) : max(m, lds[k * W + w]);
    const uint32_t now = ld_agent(&v.B.misc[MISC_BOUNDS + k]);
    if (k < 3 && m < now)
      atomicMin(&v.B.misc[MISC_BOUNDS + k], m);
    else if (k >= 3 && m > now)
      atomicMax(&v.B.misc[MISC_BOUNDS + k], m);
  }
  __syncthreads();
}

// ---- phase 2: Morton codes of one tile + the four 8-bit digit histograms ------
template <int BLOCK = BUILD_BLOCK>
__device__ inline void morton_tile(const BuildView& v, uint32_t tile, uint32_t* lds) {
  uint32_t* s_hist = lds;  // SORT_PASSES * 256
  for (int i = threadIdx.x; i < SORT_PASSES * 256; i += BLOCK) s_hist[i] = 0u;
  float lo[3] = {0, 0, 0}, ext[3] = {0, 0, 0};
  if (v.mode == RQ_MORTON_SCENE_AABB) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lo[k] = ord2f(v.B.misc[MISC_BOUNDS + k]);
      ext[k] = ord2f(v.B.misc[MISC_BOUNDS + 3 + k]) - lo[k];
    }
  }
  __syncthreads();
  const uint32_t end = min((tile + 1) * (uint32_t)TRI_TILE, v.n);
  for (uint32_t t = tile * TRI_TILE + threadIdx.x; t < end; t += CENTROIDS * BLOCK) {
    float3 c[CENTROIDS];
    centroids<BLOCK>(v, t, end, c);
#pragma unroll
    for (int j = 0; j < CENTROIDS; ++j) {
      if (t + j * BLOCK >= end) break;
      float q[3] = {c[j].x, c[j].y, c[j].z};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        if (v.mode == RQ_MORTON_SCENE_AABB)
          q[k] = ext[k] > 0.0f ? (q[k] - lo[k]) / ext[k] : 0.0f;
        else
          q[k] = (q[k] + 30.0f) / 1000.0f;
      }
      const uint32_t code = morton30(q[0], q[1], q[2]);
      v.B.codes[t + j * BLOCK] = code;
#pragma unroll
      for (int p = 0; p < SORT_PASSES; ++p)
        atomicAdd(&s_hist[p * 256 + ((code >> (8 * p)) & 255u)], 1u);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < SORT_PASSES * 256; i += BLOCK) {
    const uint32_t c = s_hist[i];
    if (c) atomicAdd(&v.B.misc[MISC_HIST + i], c);
  }
  __syncthreads();
}

// ---- phases 3-6: one stable 8-bit LSD pass over one tile ------------------------
// onesweep: wave w of the tile owns keys [w*64*ITEMS, (w+1)*64*ITEMS), lane l
// its keys i*64 + l; ranking wave by wave, item by item (8 ballots give the
// peers with the same digit) keeps input order among equal digits. Tile digit
// counts go to a decoupled look-back (flag in the top 2 bits of one word,
// agent-scope relaxed atomics, bounded wait), keys and then values are staged
// in one LDS tile buffer so the global writes of each digit are contiguous.
// Every earlier tile of the pass must already be running (ticket order).
template <int PASS, int ITEMS = SORT_ITEMS>
__device__ inline void onesweep_tile(const BuildView& v, uint32_t tile, uint32_t* lds) {
  constexpr int pass = PASS;  // static: buffer selection never indexes the view
  constexpr int TILE = SORT_BLOCK * ITEMS;
  static_assert(BUILD_BLOCK == SORT_BLOCK && SORT_BLOCK == 256, "one thread per digit");
  uint32_t* s_cnt = lds;                        // [SORT_WAVES][256]
  uint32_t* s_stage = s_cnt + SORT_WAVES * 256;  // [TILE] keys, then values
  uint32_t* s_excl = s_stage + TILE;         // [256]
  uint32_t* s_base = s_excl + 256;              // [256]
  uint32_t* s_wsum = s_base + 256;              // [2][SORT_WAVES]

  const uint32_t n = v.n;
  const uint32_t* kin = pass == 0 ? v.B.codes : ((pass & 1) ? v.B.keys_b : v.B.keys_a);
  const uint32_t* vin = pass == 0 ? nullptr : ((pass & 1) ? v.B.vals_b : v.B.vals_a);
  uint32_t* kout = (pass & 1) ? v.B.keys_a : v.B.keys_b;
  uint32_t* vout = (pass & 1) ? v.B.vals_a : v.B.vals_b;
  static_assert(PASS >= 0 && PASS < SORT_PASSES, "30-bit codes: four 8-bit passes");
  uint32_t* status = v.B.status + (size_t)pass * tiles_of(n, TILE) * 256;
  uint32_t* misc = v.B.misc;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int shift = 8 * pass;
  for (int i = tid; i < SORT_WAVES * 256; i += SORT_BLOCK) s_cnt[i] = 0u;
  __syncthreads();
  const uint32_t base = tile * TILE;
  const uint32_t wbase = base + wave * (64 * ITEMS);
  const uint64_t lt = (1ull << lane) - 1ull;

  // Full tiles load the values with the keys (their latency hides behind
  // the ranking); lean tiles, whose register budget is tight, read them only
  // when they are staged, after the keys went out.
  constexpr bool PREFETCH = ITEMS >= 16;
  uint32_t key[ITEMS], rank[ITEMS], val[PREFETCH ? ITEMS : 1];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t g = wbase + i * 64 + lane;
    key[i] = g < n ? el32(kin, g) : 0u;
    if (PREFETCH) val[i] = g < n ? (vin ? el32(vin, g) : g) : 0u;
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const bool ok = wbase + i * 64 + lane < n;
    const uint32_t d = (key[i] >> shift) & 255u;
    uint64_t peers = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint64_t bal = __ballot((d >> b) & 1u);
      peers &= ((d >> b) & 1u) ? bal : ~bal;
    }
    const uint32_t before = (uint32_t)__popcll(peers & lt);
    const uint32_t c = ok ? s_cnt[wave * 256 + d] : 0u;
    rank[i] = c + before;
    if (ok && before == 0) s_cnt[wave * 256 + d] = c + (uint32_t)__popcll(peers);
  }
  __syncthreads();
  // Only key[] and rank[] stay live across the scans below: hiding the keys
  // and the lane id from the optimiser makes it recompute digits, indices and
  // LDS addresses after the scans instead of holding them in registers.
  uint32_t lane_r = (uint32_t)lane;
  asm volatile("" : "+v"(lane_r));
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) asm volatile("" : "+v"(key[i]));

  // per digit (thread = digit): wave-exclusive prefix and tile total
  const uint32_t d = (uint32_t)tid;
  uint32_t total = 0;
#pragma unroll
  for (int w = 0; w < SORT_WAVES; ++w) {
    const uint32_t c = s_cnt[w * 256 + d];
    s_cnt[w * 256 + d] = total;
    total += c;
  }
  uint32_t* st = status + (size_t)tile * 256 + d;
  st_agent(st, (tile == 0 ? LB_INC : LB_AGG) | total);

  // block-exclusive scans of the tile totals and of the global histogram
  const uint32_t hcount = misc[MISC_HIST + pass * 256 + d];
  const uint32_t inc_t = wave_incl_scan(total, lane);
  const uint32_t inc_h = wave_incl_scan(hcount, lane);
  if (lane == 63) s_wsum[wave] = inc_t, s_wsum[SORT_WAVES + wave] = inc_h;
  __syncthreads();
  uint32_t pre_t = 0, pre_h = 0;
  for (int w = 0; w < wave; ++w) pre_t += s_wsum[w], pre_h += s_wsum[SORT_WAVES + w];
  const uint32_t blk_excl = pre_t + inc_t - total;
  const uint32_t glb_excl = pre_h + inc_h - hcount;

  // decoupled look-back over earlier tiles for this digit, LB_WINDOW status
  // words per round: the loads of a window are in flight together, and they
  // are consumed in order up to the first inclusive prefix (done) or the first
  // word not yet published (polled again from there). Tile 0 publishes an
  // inclusive prefix, so the walk ends at tile 0 at the latest.
  constexpr int LB_WINDOW = 8;
  uint32_t prefix = 0;
  if (tile > 0) {
    int64_t j = (int64_t)tile - 1;
    uint32_t spins = 0;
    for (;;) {
      uint32_t w[LB_WINDOW];
#pragma unroll
      for (int q = 0; q < LB_WINDOW; ++q)
        w[q] = j - q >= 0 ? ld_agent(status + (size_t)(j - q) * 256 + d) : 0u;
      int used = 0;
      bool done = false;
#pragma unroll
      for (int q = 0; q < LB_WINDOW; ++q) {
        if (done || used < q || j - q < 0) break;
        const uint32_t f = w[q] & ~LB_MASK;
        if (f == 0u) break;
        prefix += w[q] & LB_MASK;
        ++used;
        done = f == LB_INC;
      }
      if (done) break;
      j -= used;
      if (used == 0) {
        if (++spins > LOOKBACK_SPIN_LIMIT) {  // bounded wait: report, never hang
          atomicOr(&misc[MISC_ERR], ERR_LOOKBACK_SPIN);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    st_agent(st, LB_INC | (prefix + total));
  }
  s_excl[d] = blk_excl;
  s_base[d] = glb_excl + prefix - blk_excl;
  __syncthreads();

  // keys: rank[i] becomes the tile position, dst[j] the global position of
  // staged slot tid + j * SORT_BLOCK (reused for the values)
  static_assert(TILE % SORT_BLOCK == 0, "whole rounds");
  constexpr int ROUNDS = TILE / SORT_BLOCK;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t dd = (key[i] >> shift) & 255u;
    rank[i] += s_excl[dd] + s_cnt[wave * 256 + dd];
    if (wbase + i * 64 + lane_r < n) {
      if (rank[i] < (uint32_t)TILE)
        s_stage[rank[i]] = key[i];
      else
        atomicOr(&misc[MISC_ERR], ERR_SCATTER_RANGE);
    }
  }
  __syncthreads();
  const uint32_t cnt = min((uint32_t)TILE, n - base);
  uint32_t dst[ROUNDS];
#pragma unroll
  for (int j = 0; j < ROUNDS; ++j) {
    const uint32_t p = tid + j * SORT_BLOCK;
    dst[j] = n;
    if (p < cnt) {
      const uint32_t k = s_stage[p];
      const uint32_t g = s_base[(k >> shift) & 255u] + p;
      if (g < n) {
        el32(kout, g) = k;
        dst[j] = g;
      } else {
        atomicOr(&misc[MISC_ERR], ERR_SCATTER_RANGE);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t g = wbase + i * 64 + lane_r;
    if (g < n && rank[i] < (uint32_t)TILE)
      s_stage[rank[i]] = PREFETCH ? val[i] : (vin ? el32(vin, g) : g);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ROUNDS; ++j)
    if (dst[j] < n) el32(vout, dst[j]) = s_stage[tid + j * SORT_BLOCK];
  __syncthreads();
}

// Child links of the internal nodes as Karras emits them, (left, right) per
// node: kept in the slot_h words (2(n-1), free until a treelet pass uses them
// as scratch) until the refit writes each node record whole.
__device__ inline int2* links_of(const BuildBuffers& B) { return reinterpret_cast<int2*>(B.slot_h); }

// ---- phase 7: Karras 2012 emission for a tile of internal nodes ----------------
// Internal node i in [0, n-2] from the sorted codes; equal codes fall back to
// the index (augmented key code<<32 | i).
//
// A node's searches read the keys around it, a chain of dependent loads (the
// direction, the doubling bound, the binary searches for the far end and the
// split); most nodes span a few leaves. A unit first stages the keys of its
// nodes and KARRAS_HALO on each side in LDS, and a search reads a key from
// there when it lies in that window, from global memory otherwise.
constexpr int KARRAS_HALO = 256;
typedef __attribute__((address_space(3))) const uint32_t* LdsWords;  // an LDS array
struct KeyWindow {
  const uint32_t* __restrict__ keys;  // all n sorted keys (global)
  LdsWords win;                       // keys[lo, hi), read with LDS loads
  int64_t lo, hi;
  // The LDS word is read at a clamped index whatever j, and replaced by the
  // global one only outside the window: with one read per branch the
  // compiler merges them into a generic (flat) load, which waits on both the
  // LDS and the vector memory counters.
  __device__ uint32_t operator()(int64_t j) const {
    uint32_t k = win[min(max(j - lo, (int64_t)0), hi - lo - 1)];
    if (j < lo || j >= hi) k = keys[j];
    return k;
  }
};
// Stages keys [lo, hi) of the n keys into win (the block's threads); the
// caller synchronises before the searches read it.
__device__ inline KeyWindow stage_keys(const uint32_t* __restrict__ keys, int64_t n, int64_t lo,
                                       int64_t hi, uint32_t* win) {
  lo = max(lo, (int64_t)0), hi = min(hi, n);
  for (int64_t j = lo + threadIdx.x; j < hi; j += blockDim.x) win[j - lo] = keys[j];
  return KeyWindow{keys, (LdsWords)win, lo, hi};
}

template <class K>
__device__ inline int kdelta(const K& k, int64_t n, int64_t i, uint32_t ki, int64_t j) {
  if (j < 0 || j >= n) return -1;
  const uint32_t kj = k(j);
  return ki != kj ? __clz(ki ^ kj) : 32 + __clz((uint32_t)i ^ (uint32_t)j);
}

template <class K>
__device__ inline void karras_node(const BuildView& v, const K& keys, int64_t i) {
  const int64_t N = v.n;
  const uint32_t ki = keys(i);
  const int d = kdelta(keys, N, i, ki, i + 1) > kdelta(keys, N, i, ki, i - 1) ? 1 : -1;
  const int dmin = kdelta(keys, N, i, ki, i - d);
  int64_t lmax = 2;
  while (kdelta(keys, N, i, ki, i + lmax * d) > dmin) lmax <<= 1;
  int64_t l = 0;
  for (int64_t t = lmax >> 1; t >= 1; t >>= 1)
    if (kdelta(keys, N, i, ki, i + (l + t) * d) > dmin) l += t;
  const int64_t j = i + l * d;
  const int dnode = kdelta(keys, N, i, ki, j);
  int64_t s = 0, t = l;
  do {
    t = (t + 1) >> 1;
    if (kdelta(keys, N, i, ki, i + (s + t) * d) > dnode) s += t;
  } while (t > 1);
  const int64_t g = i + s * d + min(d, 0);
  const int32_t left = (min(i, j) == g) ? ~(int32_t)g : (int32_t)g;
  const int32_t right = (max(i, j) == g + 1) ? ~(int32_t)(g + 1) : (int32_t)(g + 1);
  // the child links go to a compact array (consecutive nodes, whole lines);
  // the refit writes them into the node records with the boxes
  links_of(v.B)[i] = make_int2(left, right);
  const int64_t ul = left >= 0 ? left : (N - 1) + ~left;
  const int64_t ur = right >= 0 ? right : (N - 1) + ~right;
  v.B.flags[i] = 0u;
  v.B.range[i] = make_uint2((uint32_t)min(i, j), (uint32_t)max(i, j));
  if (g < 0 || g + 1 > N - 1 || ul >= 2 * N - 1 || ur >= 2 * N - 1) {
    atomicOr(&v.B.misc[MISC_ERR], ERR_TOPOLOGY);
    return;
  }
  v.B.parent[ul] = (int32_t)(i << 1);
  v.B.parent[ur] = (int32_t)((i << 1) | 1);
}

// LDS words of a Karras unit of TILE nodes: its keys and the halo.
template <int TILE>
constexpr int karras_lds_words() {
  return TILE + 2 * KARRAS_HALO;
}

// TILE internal nodes per unit: the kernels take one node per thread (each node
// is an independent chain of dependent key loads, so more units hide more
// latency). lds holds karras_lds_words<TILE>() words.
template <int TILE>
__device__ inline void karras_tile(const BuildView& v, uint32_t tile, uint32_t* lds) {
  if (v.n < 2) return;
  const int64_t begin = (int64_t)tile * TILE;
  const int64_t end = min(begin + TILE, (int64_t)v.n - 1);
  const KeyWindow w = stage_keys(v.B.keys_a, v.n, begin - KARRAS_HALO, end + 1 + KARRAS_HALO, lds);
  __syncthreads();
  for (int64_t i = begin + threadIdx.x; i < end; i += blockDim.x) karras_node(v, w, i);
}

// ---- phases 8-9: bottom-up refit ---------------------------------------------------
// Helpers of the chunk-union refit below: a node's box goes into its parent's
// child slot (put_slot); the root box and height into misc (put_root).
__device__ inline void put_slot(NodeRec* nodes, uint32_t node, uint32_t side, const float* lo,
                                const float* hi) {
  float* slo = side ? &nodes[node].lo1.x : &nodes[node].lo0.x;
  float* shi = side ? &nodes[node].hi1.x : &nodes[node].hi0.x;
  slo[0] = lo[0], slo[1] = lo[1], slo[2] = lo[2];
  shi[0] = hi[0], shi[1] = hi[1], shi[2] = hi[2];
}
__device__ inline void put_root(uint32_t* misc, const float* lo, const float* hi, uint32_t h) {
  float* root = reinterpret_cast<float*>(misc + MISC_ROOT);
  for (int q = 0; q < 3; ++q) root[q] = lo[q], root[3 + q] = hi[q];
  misc[MISC_HEIGHT] = h;
}

// Leaf record of sorted position k and its box (the leaf's slot value).
__device__ inline void leaf_record(const BuildView& v, uint32_t k, TriRec& tr, float* lo,
                                   float* hi) {
  const uint32_t p = v.B.vals_a[k];
  if (v.sphere) {
    // sphere leaf: centre and radius, box centre -/+ radius (main.cpp:687-689);
    // the record keeps r and r*r (the reference's radius2)
    const float cx = v.vx[p], cy = v.vy[p], cz = v.vz[p], r = v.vr[p];
    tr.v0 = make_float4(cx, cy, cz, __int_as_float((int32_t)p));
    tr.e1 = make_float4(r, r * r, 0.0f, 0.0f);
    tr.e2 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    lo[0] = (cx - r) + 0.0f, lo[1] = (cy - r) + 0.0f, lo[2] = (cz - r) + 0.0f;
    hi[0] = (cx + r) + 0.0f, hi[1] = (cy + r) + 0.0f, hi[2] = (cz + r) + 0.0f;
  } else {
    const uint32_t a = v.idx[3 * p], b = v.idx[3 * p + 1], c = v.idx[3 * p + 2];
    const float3 v0 = make_float3(v.vx[a], v.vy[a], v.vz[a]);
    const float3 v1 = make_float3(v.vx[b], v.vy[b], v.vz[b]);
    const float3 v2 = make_float3(v.vx[c], v.vy[c], v.vz[c]);
    tr.v0 = make_float4(v0.x, v0.y, v0.z, __int_as_float((int32_t)p));
    tr.e1 = make_float4(v1.x - v0.x, v1.y - v0.y, v1.z - v0.z, 0.0f);
    tr.e2 = make_float4(v2.x - v0.x, v2.y - v0.y, v2.z - v0.z, 0.0f);
    lo[0] = fminf(fminf(v0.x, v1.x), v2.x) + 0.0f, lo[1] = fminf(fminf(v0.y, v1.y), v2.y) + 0.0f;
    lo[2] = fminf(fminf(v0.z, v1.z), v2.z) + 0.0f;
    hi[0] = fmaxf(fmaxf(v0.x, v1.x), v2.x) + 0.0f, hi[1] = fmaxf(fmaxf(v0.y, v1.y), v2.y) + 0.0f;
    hi[2] = fmaxf(fmaxf(v0.z, v1.z), v2.z) + 0.0f;
  }
}

// ---- 4-wide collapse ------------------------------------------------------------
// The wide node of binary internal node i holds, in binary order, for each
// child c of i: c's box if c is a leaf (one slot, the next one unused), else
// the boxes of c's two children (two slots). Every internal node gets its
// wide node (only the root and even-depth nodes are reached from the root).
struct WideSlots {
  float lo[4][3], hi[4][3];
  int32_t link[4];
};
__device__ inline void wide_empty(WideSlots& w, int k) {
  w.lo[k][0] = w.lo[k][1] = w.lo[k][2] = INFINITY;
  w.hi[k][0] = w.hi[k][1] = w.hi[k][2] = -INFINITY;
  w.link[k] = 0;
}
// One axis of the record's grid: the slots' planes on base + (1024 + q) * step.
// The step is the slots' extent over 252 (two steps to spare on a byte), at
// least 2^-21 of the largest coordinate, so that the rounding of the base
// (2^-24 of a magnitude of at most 2^21 + 1024 steps) stays within an eighth
// of a step, and 2^-60. The base lies one step further down, so no lo plane
// needs a negative q. The quotient (1024 + q) is computed with an error below
// 2^-12 of a step and rounded outward by 2^-9 more, so the plane the walk
// computes contains the exact one by over 2^-10 of a step: the walk's own
// rounding is below that for an origin within the grid, and relative to the
// distance (covered by its slack) for one further away. An extent or a
// coordinate of 2^100 or more (or one that is not finite) makes the step NaN,
// and the walk reads a NaN plane as a box that reaches everywhere; other steps
// are at most 2^92, which the walk relies on (steep in trace_device.h).
__device__ inline void wide_axis(const float* lo, const float* hi, float* base, float* step,
                                 uint32_t* qlo, uint32_t* qhi) {
  const float l = fminf(fminf(lo[0], lo[1]), fminf(lo[2], lo[3]));
  const float h = fmaxf(fmaxf(hi[0], hi[1]), fmaxf(hi[2], hi[3]));
  const float ext = h - l, mag = fmaxf(fabsf(l), fabsf(h));
  const bool sane = ext < 0x1p100f && mag < 0x1p100f;
  const float s =
      sane ? fmaxf(fmaxf(ext * (1.0f / 252.0f), mag * 0x1p-21f), 0x1p-60f) : NAN;
  const float b = sane ? l - (WIDE_Q0 + 1.0f) * s : 0.0f;
  const float rs = 1.0f / s;
  uint32_t ql = 0u, qh = 0u;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float a = floorf((lo[k] - b) * rs - (WIDE_Q0 + 0x1p-9f));
    const float c = ceilf((hi[k] - b) * rs - (WIDE_Q0 - 0x1p-9f));
    ql |= (uint32_t)fminf(fmaxf(a, 0.0f), 255.0f) << (8 * k);
    qh |= (uint32_t)fminf(fmaxf(c, 0.0f), 255.0f) << (8 * k);
  }
  *base = b, *step = s, *qlo = ql, *qhi = qh;
}
__device__ inline void wide_store(WideNode* W, const WideSlots& w) {
  float lo[3][4], hi[3][4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int x = 0; x < 3; ++x) lo[x][k] = w.lo[k][x], hi[x][k] = w.hi[k][x];
  WideNode n;
  wide_axis(lo[0], hi[0], &n.base.x, &n.base.w, &n.lox, &n.hix);
  wide_axis(lo[1], hi[1], &n.base.y, &n.step_y, &n.loy, &n.hiy);
  wide_axis(lo[2], hi[2], &n.base.z, &n.step_z, &n.loz, &n.hiz);
  n.link = make_int4(w.link[0], w.link[1], w.link[2], w.link[3]);
  *W = n;
}
// From the finished binary node records in global memory.
__device__ inline void widen_global(const BuildBuffers& B, uint32_t i) {
  const NodeRec N = B.nodes[i];
  WideSlots w;
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const int32_t c = __float_as_int(side ? N.hi0.w : N.lo0.w);
    const float4 clo = side ? N.lo1 : N.lo0, chi = side ? N.hi1 : N.hi0;
    if (c < 0) {
      w.lo[2 * side][0] = clo.x, w.lo[2 * side][1] = clo.y, w.lo[2 * side][2] = clo.z;
      w.hi[2 * side][0] = chi.x, w.hi[2 * side][1] = chi.y, w.hi[2 * side][2] = chi.z;
      w.link[2 * side] = c;
      wide_empty(w, 2 * side + 1);
    } else {
      const NodeRec C = B.nodes[c];
      w.lo[2 * side][0] = C.lo0.x, w.lo[2 * side][1] = C.lo0.y, w.lo[2 * side][2] = C.lo0.z;
      w.hi[2 * side][0] = C.hi0.x, w.hi[2 * side][1] = C.hi0.y, w.hi[2 * side][2] = C.hi0.z;
      w.lo[2 * side + 1][0] = C.lo1.x, w.lo[2 * side + 1][1] = C.lo1.y;
      w.lo[2 * side + 1][2] = C.lo1.z;
      w.hi[2 * side + 1][0] = C.hi1.x, w.hi[2 * side + 1][1] = C.hi1.y;
      w.hi[2 * side + 1][2] = C.hi1.z;
      w.link[2 * side] = __float_as_int(C.lo0.w), w.link[2 * side + 1] = __float_as_int(C.hi0.w);
    }
  }
  wide_store(B.wide + i, w);
}

// Tree height on demand (the chunk-union refit leaves it open): the depth of
// node i's leaf children, d + 1 for a node at depth d with a leaf child (walk
// up the parent links, at most 64 steps), else 0; the height is the maximum.
__device__ inline uint32_t leaf_depth(const BuildBuffers& B, uint32_t n, uint32_t i) {
  const NodeRec N = B.nodes[i];
  if (__float_as_int(N.lo0.w) >= 0 && __float_as_int(N.hi0.w) >= 0) return 0u;
  uint32_t d = 0, cur = i;
  while (cur != 0u) {
    const int32_t pe = B.parent[cur];
    cur = (uint32_t)pe >> 1;
    if (pe < 0 || cur >= n - 1 || ++d > 64) {
      atomicOr(&B.misc[MISC_ERR], ERR_WIDEN_DEPTH);
      return 0u;
    }
  }
  return d + 1u;
}

// ---- chunk-union refit ------------------------------------------------------------
// Pass 1, one block of CHUNK threads per chunk of CHUNK leaves. Every box a chunk has to give is
// the union of a run of its leaves: of a node whose leaf range lies inside the
// chunk; of the leaves from a on, or up to b, for the nodes [a, b] that span
// chunks; of all. Thread t has one such run at most, that of node chunk start
// + t (a Karras node's index is an end of its own range). The unions of 2^j
// leaves from each leaf on are made in LDS for one j after the other, and a run
// of 2^j + 1 to 2^(j+1) leaves is the union of the two of them at its ends,
// which may overlap: min and max are order-independent and idempotent, so this
// is the box a climb would build.
// (The climb it replaced, each leaf up to the first node whose other child had
// not arrived, ran every wave through the levels of its longest lane: 3400
// instructions a wave in chunks of 1024, where this takes 10 levels of 60:
// 115 -> 88 us for 1.3 M triangles of a sphere, 35 -> 27 for 100 k.)
// Pass 2 gives every spanning node [a, b] its box: suffix(a) | chunks strictly
// between | prefix(b). The height is left to the on-demand depth walk.
__device__ inline void box_union(float* b, const float* o) {
  b[0] = fminf(b[0], o[0]), b[1] = fminf(b[1], o[1]), b[2] = fminf(b[2], o[2]);
  b[3] = fmaxf(b[3], o[3]), b[4] = fmaxf(b[4], o[4]), b[5] = fmaxf(b[5], o[5]);
}
// The union of a wave's boxes, in every lane (all of them active): rows of 16
// by lane exchange within the row, then each row's last lane to the next ones.
template <int CTRL>
__device__ inline void union_dpp(float* b) {
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const int x = __float_as_int(b[q]);
    const float o = __int_as_float(__builtin_amdgcn_update_dpp(x, x, CTRL, 0xF, 0xF, false));
    b[q] = q < 3 ? fminf(b[q], o) : fmaxf(b[q], o);
  }
}
__device__ inline void wave_union(float* b) {
  union_dpp<0xB1>(b);   // lane ^ 1
  union_dpp<0x4E>(b);   // lane ^ 2
  union_dpp<0x141>(b);  // 7 - lane in each half row
  union_dpp<0x140>(b);  // 15 - lane in each row
  union_dpp<0x142>(b);  // lane 15 of the row before
  union_dpp<0x143>(b);  // lane 31, to the upper half
#pragma unroll
  for (int q = 0; q < 6; ++q)
    b[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b[q]), 63));
}
__device__ inline void box_store(float* dst, const float* b) {
  float2* d = reinterpret_cast<float2*>(dst);  // 24-byte records, 8-byte aligned
  d[0] = make_float2(b[0], b[1]), d[1] = make_float2(b[2], b[3]), d[2] = make_float2(b[4], b[5]);
}
__device__ inline void box_load(const float* src, float* b) {
  const float2* q = reinterpret_cast<const float2*>(src);
  const float2 a = q[0], c = q[1], e = q[2];
  b[0] = a.x, b[1] = a.y, b[2] = c.x, b[3] = c.y, b[4] = e.x, b[5] = e.y;
}

// LDS (8-byte aligned): the boxes of the chunk's leaves, the table of the level (later the boxes
// of its nodes), three rows of CHUNK pairs each, and its internal nodes'
// ranges and children.
template <int CHUNK>
constexpr int refit_chunk_lds_words() {
  return CHUNK * 16;
}
typedef float Pair __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) Pair* LdsBoxes;  // box i: [i], [CHUNK + i], [2 CHUNK + i]
template <int CHUNK>
__device__ inline void lds_box_store(LdsBoxes dst, uint32_t i, const float* b) {
  dst[i] = Pair{b[0], b[1]}, dst[CHUNK + i] = Pair{b[2], b[3]};
  dst[2 * CHUNK + i] = Pair{b[4], b[5]};
}
template <int CHUNK>
__device__ inline void lds_box_load(LdsBoxes src, uint32_t i, float* b) {
  const Pair x = src[i], y = src[CHUNK + i], z = src[2 * CHUNK + i];
  b[0] = x.x, b[1] = x.y, b[2] = y.x, b[3] = y.y, b[4] = z.x, b[5] = z.y;
}

// Whether internal node i's leaf range crosses a boundary of CHUNK-leaf chunks.
template <int CHUNK>
__device__ inline bool spans_chunks(const BuildBuffers& B, uint32_t i) {
  const uint2 rg = B.range[i];
  return rg.x / CHUNK != rg.y / CHUNK;
}

template <int CHUNK>
__device__ inline void refit_chunk_tile(const BuildView& v, uint32_t chunk, uint32_t* lds) {
  static_assert(CHUNK % 64 == 0 && CHUNK <= 1024, "one leaf per thread, whole waves");
  static_assert(CHUNK >= REFIT_CHUNK_MIN, "the chunk unions are allocated for REFIT_CHUNK_MIN");
  const LdsBoxes s_leaf = (LdsBoxes)lds, s_tab = (LdsBoxes)(lds + 6 * CHUNK);
  uint2* s_rng = reinterpret_cast<uint2*>(lds + 12 * CHUNK);  // range of node
  int2* s_kid = reinterpret_cast<int2*>(s_rng + CHUNK);       // children of node
  const BuildBuffers& B = v.B;
  const uint32_t n = v.n;
  const uint32_t tid = threadIdx.x;
  const uint32_t chunk_lo = chunk * CHUNK;
  const uint32_t chunk_hi = min(chunk_lo + CHUNK, n) - 1, cnt = chunk_hi - chunk_lo + 1u;
  const uint32_t k = chunk_lo + tid;
  const bool valid = k <= chunk_hi, node = k < n - 1;  // (n >= 1)
  int32_t pleaf = 0, pnode = 0;  // parents of leaf k and node k
  uint2 rg = make_uint2(k, k);
  int2 kid = make_int2(0, 0);
  if (valid && n > 1) pleaf = B.parent[(n - 1) + k];
  if (node) {
    pnode = k == 0u ? -1 : B.parent[k];  // the root has no parent
    rg = B.range[k], kid = links_of(B)[k];
    s_rng[tid] = rg, s_kid[tid] = kid;
  }
  float leaf[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  if (valid) {
    TriRec tr;
    leaf_record(v, k, tr, leaf, leaf + 3);
    B.tris[k] = tr;
  }
  lds_box_store<CHUNK>(s_leaf, tid, leaf);
  // The thread's run [qa, qb]: its node's if that lies in the chunk; else what
  // pass 2 reads of the spanning nodes, suffix(a) and prefix(b). The largest
  // node that starts at leaf a is node a (a right child, or the root), the
  // largest that ends at leaf b is node b (a left child) or the root, so the
  // others need none stored.
  const bool inside = node && rg.x >= chunk_lo && rg.y <= chunk_hi;
  const bool suffix = node && rg.x == k && rg.y > chunk_hi;
  const bool prefix = valid && chunk_lo > 0u && (k == n - 1 || (rg.y == k && rg.x < chunk_lo));
  const uint32_t qa = prefix ? 0u : (inside ? rg.x : k) - chunk_lo;
  const uint32_t qb = (suffix ? chunk_hi : inside ? rg.y : k) - chunk_lo;
  const bool query = inside || suffix || prefix;
  const uint32_t len = qb - qa + 1u, lev = len > 1u ? 31u - __clz(len - 1u) : 0u;
  const uint32_t levels = cnt > 1u ? 32u - __clz(cnt - 1u) : 1u;
  float cur[6], box[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) cur[q] = leaf[q], box[q] = leaf[q];
  __syncthreads();
  for (uint32_t j = 0; j < levels; ++j) {
    const LdsBoxes tab = j == 0u ? s_leaf : s_tab;
    if (query && lev == j) {
      float o[6];
      lds_box_load<CHUNK>(tab, qa, box);
      lds_box_load<CHUNK>(tab, qb + (len > 1u ? 1u - (1u << j) : 0u), o);
      box_union(box, o);
    }
    if (tid + (1u << j) < (uint32_t)CHUNK) {  // past the end: the run is the rest
      float o[6];
      lds_box_load<CHUNK>(tab, tid + (1u << j), o);
      box_union(cur, o);
    }
    if (j + 1u == levels) break;
    if (j > 0u) __syncthreads();  // the table is read before it is overwritten
    lds_box_store<CHUNK>(s_tab, tid, cur);
    __syncthreads();
  }
  if (tid == 0) box_store(B.cbox + 6ull * chunk, cur);  // every leaf from the first on
  if (suffix) box_store(B.suf + 6ull * k, box);
  if (prefix) box_store(B.pre + 6ull * k, box);
  if (n == 1) {
    if (valid) put_root(B.misc, leaf, leaf + 3, 0u);
    return;
  }
  __syncthreads();  // the last table is read
  if (inside) lds_box_store<CHUNK>(s_tab, tid, box);
  // A leaf or node of the chunk whose parent is not: its box goes to the slot
  // in the parent's record (pass 2 finishes it; a parent inside the chunk
  // writes its record whole, below).
  auto give = [&](int32_t pe, const float* b) {
    const uint32_t p = (uint32_t)pe >> 1;
    if (pe < 0 || p >= n - 1) {
      atomicOr(&B.misc[MISC_ERR], ERR_REFIT_DEPTH);
      return;
    }
    if (p < chunk_lo || p > chunk_hi || s_rng[p - chunk_lo].x < chunk_lo ||
        s_rng[p - chunk_lo].y > chunk_hi)
      put_slot(B.nodes, p, (uint32_t)pe & 1u, b, b + 3);
  };
  if (valid) give(pleaf, leaf);
  if (inside) {
    if (k == 0u) {  // the whole tree lies in this chunk
      float* root = reinterpret_cast<float*>(B.misc + MISC_ROOT);
      for (int q = 0; q < 6; ++q) root[q] = box[q];
    } else {
      give(pnode, box);
    }
  }
  // Node records and wide records of the chunk's nodes: thread t writes node
  // chunk start + t, so the 64-byte records go out in consecutive lines. An
  // internal child of such a node lies in the chunk too.
  __syncthreads();
  if (!inside) return;
  auto box_of = [&](int32_t c, float* b) {
    lds_box_load<CHUNK>(c < 0 ? s_leaf : s_tab, (uint32_t)(c < 0 ? ~c : c) - chunk_lo, b);
  };
  WideSlots ws;
  float cb[2][6];
#pragma unroll
  for (int sd = 0; sd < 2; ++sd) {
    const int32_t c = sd ? kid.y : kid.x;
    box_of(c, cb[sd]);
    if (c < 0) {
      ws.lo[2 * sd][0] = cb[sd][0], ws.lo[2 * sd][1] = cb[sd][1], ws.lo[2 * sd][2] = cb[sd][2];
      ws.hi[2 * sd][0] = cb[sd][3], ws.hi[2 * sd][1] = cb[sd][4], ws.hi[2 * sd][2] = cb[sd][5];
      ws.link[2 * sd] = c;
      wide_empty(ws, 2 * sd + 1);
    } else {
      const int2 gk = s_kid[(uint32_t)c - chunk_lo];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        float gb[6];
        box_of(g ? gk.y : gk.x, gb);
        ws.lo[2 * sd + g][0] = gb[0], ws.lo[2 * sd + g][1] = gb[1], ws.lo[2 * sd + g][2] = gb[2];
        ws.hi[2 * sd + g][0] = gb[3], ws.hi[2 * sd + g][1] = gb[4], ws.hi[2 * sd + g][2] = gb[5];
        ws.link[2 * sd + g] = g ? gk.y : gk.x;
      }
    }
  }
  NodeRec nr;
  nr.lo0 = make_float4(cb[0][0], cb[0][1], cb[0][2], __int_as_float(kid.x));
  nr.hi0 = make_float4(cb[0][3], cb[0][4], cb[0][5], __int_as_float(kid.y));
  nr.lo1 = make_float4(cb[1][0], cb[1][1], cb[1][2], 0.0f);
  nr.hi1 = make_float4(cb[1][3], cb[1][4], cb[1][5], 0.0f);
  B.nodes[k] = nr;
  if (B.wide) wide_store(B.wide + k, ws);
}

// Pass 2: the lanes of a wave each take internal node i; the wave then works
// through its spanning nodes one at a time, all 64 lanes striding over the
// chunks strictly inside the span (a node near the root spans them all).
// Every lane must reach this call (the wave shuffles).
template <int CHUNK>
__device__ inline void refit_span_wave(const BuildBuffers& B, uint32_t n, uint32_t i) {
  const uint32_t lane = threadIdx.x & 63u;
  uint2 rg = make_uint2(0u, 0u);
  bool span = false;
  if (i < n - 1) {
    rg = B.range[i];
    span = rg.x / CHUNK != rg.y / CHUNK;
  }
  uint64_t m = __ballot(span);
  while (m) {
    const int src = __ffsll((unsigned long long)m) - 1;
    m &= m - 1ull;
    const uint32_t ca = (uint32_t)__shfl((int)(rg.x / CHUNK), src, 64);
    const uint32_t cb = (uint32_t)__shfl((int)(rg.y / CHUNK), src, 64);
    float box[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY}, o[6];
    for (uint32_t c = ca + 1 + lane; c < cb; c += 64) {
      box_load(B.cbox + 6ull * c, o);
      box_union(box, o);
    }
    wave_union(box);
    if ((int)lane != src) continue;
    // the spanning node's own links (its slots were filled by its children)
    const int2 kid = links_of(B)[i];
    reinterpret_cast<int32_t*>(&B.nodes[i].lo0)[3] = kid.x;
    reinterpret_cast<int32_t*>(&B.nodes[i].hi0)[3] = kid.y;
    box_load(B.suf + 6ull * rg.x, o);
    box_union(box, o);
    box_load(B.pre + 6ull * rg.y, o);
    box_union(box, o);
    if (i == 0u) {
      float* root = reinterpret_cast<float*>(B.misc + MISC_ROOT);
      for (int q = 0; q < 6; ++q) root[q] = box[q];
      continue;
    }
    const int32_t pe = B.parent[i];
    const uint32_t node = (uint32_t)pe >> 1, side = (uint32_t)pe & 1u;
    if (pe < 0 || node >= n - 1) {
      atomicOr(&B.misc[MISC_ERR], ERR_REFIT_DEPTH);
      continue;
    }
    put_slot(B.nodes, node, side, box, box + 3);
  }
}


}  // namespace rq
