// Batch kernels: build the LBVH of many meshes and trace their ray batches.
// One device work queue holds the items (mesh, tile) of every mesh, phase after
// phase (init, bounds, Morton, four sort passes, Karras, refit, spanning nodes,
// widen, trace); a phase of the build is one launch with a block or more per
// item, whatever mesh it belongs to, and the trace phase one launch of
// persistent waves that pull its items.
//
// One persistent kernel used to run all the build phases with grid barriers
// between them. A barrier cost 33 ns a block (each block's write-back and
// invalidation of its L2, one after another on an XCD): 42 us at 1280 blocks,
// ten times a build, and the kernel's registers and LDS were the largest
// phase's. Between launches the device does that once: the build of 48 meshes
// of 64 triangles 490 -> 59 us, of 30 k triangles 1160 -> 390.
#include <algorithm>

#include "batch_internal.h"
#include "build_device.h"
#include "trace_device.h"

namespace rq {
namespace {

// Phase stamps (BATCH_CTL_CLOCK).
__device__ inline unsigned long long* clock_stamp(uint32_t* ctl, uint32_t k) {
  return reinterpret_cast<unsigned long long*>(ctl + BATCH_CTL_CLOCK) + k;
}

// The next item of a queue of n items whose first `owned` are taken without a
// ticket, by the unit (block or wave) of their number: its number, or n or
// more. An atomic on one word takes 12 ns, and each unit used to end every
// queue with a failed one, so the word is read first: an empty queue costs a
// load, one whose items all have an owner nothing.
__device__ inline uint32_t next_item(uint32_t* ticket, uint32_t owned, uint32_t n) {
  if (owned >= n || owned + ld_agent(ticket) >= n) return n;
  return owned + atomicAdd(ticket, 1u);
}

// Loads a block-uniform descriptor into scalar registers: every dword goes
// through readfirstlane, so the struct is provably uniform and is never copied
// to per-lane scratch.
template <typename T>
__device__ inline T load_uniform(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "dword-sized descriptor");
  constexpr int W = sizeof(T) / 4;
  const uint32_t* src = reinterpret_cast<const uint32_t*>(p);
  uint32_t w[W];
#pragma unroll
  for (int i = 0; i < W; ++i) w[i] = __builtin_amdgcn_readfirstlane(src[i]);
  T t;
  __builtin_memcpy(&t, w, sizeof(T));
  return t;
}

// What a walk over the rays of mesh `mesh` from r0 on needs seldom, read from the
// kernel's argument memory and the mesh's descriptor each time (the empty asm hides
// that they never change): as scalars they crowded out the walk's own.
template <typename T>
using Constant = __attribute__((address_space(4))) const T*;
struct ColdArgs : TraceArgs {
  __device__ const ColdArgs* operator->() const { return this; }
};
struct MeshCold {
  uint32_t mesh, r0;
  __device__ Constant<BatchArgs> args() const {
    Constant<BatchArgs> p = (Constant<BatchArgs>)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
  }
  __device__ ColdArgs operator()() const {
    const Constant<BatchArgs> p = args();
    const Constant<BatchMeshDev> m = (Constant<BatchMeshDev>)p->meshes + mesh;
    ColdArgs c{};
    c.rays = rq_rays{m->rays.ox + r0, m->rays.oy + r0, m->rays.oz + r0,   m->rays.dx + r0,
                     m->rays.dy + r0, m->rays.dz + r0, m->rays.tmin + r0, m->rays.tmax + r0};
    c.prim = m->prim + r0;
    c.t = m->t ? m->t + r0 : nullptr;
    c.u = m->u ? m->u + r0 : nullptr;
    c.v = m->v_ ? m->v_ + r0 : nullptr;
    c.occ = m->occ + r0;
    c.gstack = p->gstack;
    c.gdepth = p->gdepth;
    c.gwords = p->gwords;
    c.err = p->ctl + BATCH_CTL_TRACE_ERR;
    return c;
  }
  __device__ LeafBoxes leaf_boxes() const {
    const Constant<BatchMeshDev> m = (Constant<BatchMeshDev>)args()->meshes + mesh;
    return LeafBoxes{m->v.B.parent, m->v.B.nodes};
  }
};
// What it needs all the time.
__device__ inline TraceArgs hot_args(const BatchMeshDev& m, uint32_t nrays, uint32_t refill_idle) {
  TraceArgs t{};
  t.nodes = m.v.B.nodes;
  t.wide = m.v.B.wide;
  t.tris = m.v.B.tris;
  t.nprims = m.v.n;
  t.nrays = nrays;
  t.refill_idle = refill_idle;
  t.sphere = 0;  // batch meshes are triangle scenes
  return t;
}

// One trace item (a tile of one mesh's rays), shared by the block's waves: a
// ray counter in LDS hands out chunks of the tile as lanes go idle; the waves
// meet at a barrier when it is done.
template <int DEPTH, bool TSTACK, bool WIDE>
__device__ inline void trace_item(const BatchArgs& a, const BatchWork& w, uint32_t* lds,
                                  uint32_t* s_ctr, SplitSlots* slots) {
  const BatchMeshDev m = load_uniform(a.meshes + w.mesh);
  const uint32_t r0 = (w.tile & ~BATCH_ANY_BIT) * a.ray_tile;
  const uint32_t nr = min(a.ray_tile, m.nrays - r0);
  const TraceArgs t = hot_args(m, nr, a.refill_idle);
  if (threadIdx.x == 0) *s_ctr = 0u;
  __syncthreads();
  int32_t* s_node = reinterpret_cast<int32_t*>(lds);
  float* s_tn = reinterpret_cast<float*>(lds + DEPTH * BUILD_BLOCK);
  ItemRays src{s_ctr, nr};
  const MeshCold cold{w.mesh, r0};
  if (w.tile & BATCH_ANY_BIT)
    trace_loop<true, false, BUILD_BLOCK, DEPTH, false, false, WIDE, true>(t, cold, src, s_node,
                                                                          s_tn, slots);
  else
    trace_loop<false, false, BUILD_BLOCK, DEPTH, TSTACK, false, WIDE, true>(t, cold, src, s_node,
                                                                            s_tn, slots);
  __syncthreads();
}

// The trace items a unit (a wave, or a block whose waves share an item) takes:
// the item of its own number in its XCD's segment, then by ticket what has no
// owner, its own segment first. Blocks go to the XCDs in turn. One lane's.
constexpr uint32_t NO_ITEM = ~0u;
template <uint32_t PER_BLOCK>
struct SegQueue {
  uint32_t index;   // the unit's number in its segment
  uint32_t k = 0;   // cursor: segment (XCD + k) % BATCH_XCDS
  bool own = true;  // its own item not taken yet
  __device__ explicit SegQueue(uint32_t unit)
      : index(seg_index(blockIdx.x, BATCH_XCDS) * PER_BLOCK + unit) {}
  __device__ uint32_t take(const BatchArgs& a) {
    for (; k < (uint32_t)BATCH_XCDS; ++k) {
      const uint32_t q = (blockIdx.x + k) % BATCH_XCDS;
      const uint32_t b0 = a.trace_seg[q], n = a.trace_seg[q + 1] - b0;
      if (own) {
        own = false;
        if (index < n) return b0 + index;
      }
      const uint32_t it = next_item(a.ctl + BATCH_XTICKET_BASE + q * BATCH_XTICKET_STRIDE,
                                    seg_blocks(q, BATCH_XCDS, gridDim.x) * PER_BLOCK, n);
      if (it < n) return b0 + it;
    }
    return NO_ITEM;
  }
};
typedef SegQueue<BUILD_BLOCK / 64> SegItems;

// Slices of one wave's walk over one mesh and query kind (the batch run): the
// tile of the item the walk starts with, then the tiles of the items the wave
// takes next from the XCD segments while they are of the same mesh and kind.
// A mesh's items sit in a row in its segment (closest-hit tiles, then any-hit
// tiles), so a wave lets its lanes run dry once per run of one mesh's items
// rather than once per tile; the first item of another mesh or kind ends the
// walk and starts the next one.
struct ItemSlices {
  const BatchArgs& args;
  SegItems seg;
  uint32_t mesh, kind, nrays;
  BatchWork held;   // the walk's first item, then the item that ended it
  bool first, have_held;
  // The wave's next item (every lane active).
  __device__ bool take(BatchWork& w) {
    uint32_t it = 0;
    if ((threadIdx.x & 63u) == 0) it = seg.take(args);
    it = __builtin_amdgcn_readfirstlane(it);
    if (it == NO_ITEM) return false;
    w = load_uniform(args.items + it);
    return true;
  }
  __device__ bool next(uint32_t& b, uint32_t& e) {
    BatchWork w;
    if (first) {
      w = held;
      first = false;
    } else {
      if (!take(w)) return false;
      if (w.mesh != mesh || (w.tile & BATCH_ANY_BIT) != kind) {
        held = w, have_held = true;
        return false;
      }
    }
    b = (w.tile & ~BATCH_ANY_BIT) * args.ray_tile;
    e = min(b + args.ray_tile, nrays);
    return true;
  }
};

// One wave's walk over the rays of one mesh and query kind, its slices from
// src (the whole mesh's arrays: a ray's index is its index in the mesh).
template <int DEPTH, bool TSTACK, bool WIDE>
__device__ inline void trace_mesh(const BatchArgs& a, const BatchMeshDev& m, uint32_t* lds,
                                  ItemSlices* src) {
  const TraceArgs t = hot_args(m, m.nrays, a.refill_idle);
  const MeshCold cold{src->mesh, 0u};
  int32_t* s_node = reinterpret_cast<int32_t*>(lds);
  float* s_tn = reinterpret_cast<float*>(lds + DEPTH * BUILD_BLOCK);
  if (src->kind)
    trace_loop<true, false, BUILD_BLOCK, DEPTH, false, false, WIDE, false>(t, cold, *src, s_node,
                                                                           s_tn);
  else
    trace_loop<false, false, BUILD_BLOCK, DEPTH, TSTACK, false, WIDE, false>(t, cold, *src, s_node,
                                                                             s_tn);
}

// ---- the build phases: a launch each ----------------------------------------
// Block of phase ph: part (block mod parts) of item (block / parts).
// Descriptors are loaded into scalar registers.
template <uint32_t PARTS>
struct PhaseUnit {
  BuildView v;
  uint32_t tile;  // the part's number in its mesh
  __device__ PhaseUnit(const BatchArgs& a, int ph) {
    // the phase's start, the end of the one before
    if (blockIdx.x == 0 && threadIdx.x == 0) *clock_stamp(a.ctl, ph) = wall_clock64();
    const BatchWork w = load_uniform(a.items + a.phase_begin[ph] + blockIdx.x / PARTS);
    v = load_uniform(&a.meshes[w.mesh].v);
    tile = w.tile * PARTS + blockIdx.x % PARTS;
  }
};
// The end of what may be the last phase with items (near enough: its last
// block's).
__device__ inline void stamp_end(const BatchArgs& a, int ph) {
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *clock_stamp(a.ctl, ph + 1) = wall_clock64();
}

// Clears the control words before a run; block 0 of the init phase, so that the
// reset lives in the same captured graph as the run.
__device__ inline void reset_ctl(uint32_t* ctl) {
  static_assert(BATCH_CTL_WORDS <= 64, "one wave clears the control words");
  if (threadIdx.x < BATCH_CTL_WORDS) ctl[threadIdx.x] = 0u;
  if (threadIdx.x < BATCH_XCDS) {
    uint32_t* x = ctl + BATCH_XTICKET_BASE + threadIdx.x * BATCH_XTICKET_STRIDE;
    x[0] = x[BATCH_XBLOCKS] = 0u;
  }
}
__global__ void k_batch_reset(uint32_t* ctl) { reset_ctl(ctl); }

// (launched with a block at least, for the reset)
__global__ __launch_bounds__(BUILD_BLOCK) void k_batch_init(BatchArgs a) {
  if (blockIdx.x == 0) {
    reset_ctl(a.ctl);
    __syncthreads();
  }
  if (a.phase_begin[PH_INIT] + blockIdx.x >= a.phase_begin[PH_INIT + 1]) return;
  const PhaseUnit<1> u(a, PH_INIT);
  build_init_misc(u.v, threadIdx.x, BUILD_BLOCK);
}
constexpr int TRI_BLOCK = 1024;
__global__ __launch_bounds__(TRI_BLOCK) void k_batch_bounds(BatchArgs a) {
  __shared__ uint32_t lds[6 * (TRI_BLOCK / 64)];
  const PhaseUnit<1> u(a, PH_BOUNDS);
  bounds_tile<TRI_BLOCK>(u.v, u.tile, lds);
}
// Also clears the sort's look-back words, a part a tile (in the init phase's
// one item a mesh they took 0.1 ms of one block).
__global__ __launch_bounds__(TRI_BLOCK) void k_batch_morton(BatchArgs a) {
  __shared__ uint32_t lds[SORT_PASSES * 256];
  const PhaseUnit<1> u(a, PH_MORTON);
  build_init_status(u.v, u.tile * TRI_BLOCK + threadIdx.x, tiles_of(u.v.n, TRI_TILE) * TRI_BLOCK);
  morton_tile<TRI_BLOCK>(u.v, u.tile, lds);
}
// The tile comes from the mesh's ticket of the pass, so a tile's look-back only
// waits on tiles whose blocks are already running (a mesh has a block for each
// of its tiles).
template <int PASS, int WAVES>
__global__ __launch_bounds__(BUILD_BLOCK) __attribute__((amdgpu_waves_per_eu(WAVES))) void
k_batch_sort(BatchArgs a) {
  __shared__ uint32_t lds[sort_lds_words(SORT_ITEMS_LEAN)];
  __shared__ uint32_t s_tile;
  const PhaseUnit<1> u(a, PH_SORT0 + PASS);
  if (threadIdx.x == 0) s_tile = atomicAdd(&u.v.B.misc[MISC_TILECTR + PASS], 1u);
  __syncthreads();
  onesweep_tile<PASS, SORT_ITEMS_LEAN>(u.v, s_tile, lds);
}
constexpr uint32_t KARRAS_PARTS = NODE_TILE / BUILD_BLOCK;  // a node a thread
__global__ __launch_bounds__(BUILD_BLOCK) void k_batch_karras(BatchArgs a) {
  __shared__ uint32_t lds[karras_lds_words<BUILD_BLOCK>()];
  const PhaseUnit<KARRAS_PARTS> u(a, PH_KARRAS);
  karras_tile<BUILD_BLOCK>(u.v, u.tile, lds);
}
// Chunk-union refit, pass 1 (with the chunks' wide records), a block a chunk.
// (48 meshes: 512 leaves a chunk 1815 us, 256 1825.)
constexpr int BATCH_REFIT_CHUNK = 2 * BUILD_BLOCK;
constexpr uint32_t REFIT_PARTS = BATCH_REFIT_CHUNKS / 2;
static_assert(BATCH_REFIT_CHUNK >= REFIT_CHUNK_MIN, "the chunk unions are allocated for this");
__global__ __launch_bounds__(BATCH_REFIT_CHUNK) void k_batch_refit(BatchArgs a) {
  __shared__ __align__(8) uint32_t lds[refit_chunk_lds_words<BATCH_REFIT_CHUNK>()];
  const PhaseUnit<REFIT_PARTS> u(a, PH_REFIT);
  if (u.tile * BATCH_REFIT_CHUNK < u.v.n) refit_chunk_tile<BATCH_REFIT_CHUNK>(u.v, u.tile, lds);
  stamp_end(a, PH_REFIT);
}
// Pass 2: the nodes spanning chunks, a wave per 64 nodes; then their wide
// records.
__global__ __launch_bounds__(BUILD_BLOCK) void k_batch_span(BatchArgs a) {
  const PhaseUnit<BATCH_SPAN_TILES> u(a, PH_TOP);
  refit_span_wave<BATCH_REFIT_CHUNK>(u.v.B, u.v.n, u.tile * BUILD_BLOCK + threadIdx.x);
}
__global__ __launch_bounds__(BUILD_BLOCK) void k_batch_widen(BatchArgs a) {
  const PhaseUnit<BATCH_SPAN_TILES> u(a, PH_WIDEN);
  const uint32_t i = u.tile * BUILD_BLOCK + threadIdx.x;
  if (i + 1u < u.v.n && spans_chunks<BATCH_REFIT_CHUNK>(u.v.B, i)) widen_global(u.v.B, i);
  stamp_end(a, PH_WIDEN);
}

// The trace phase (ray tiles over built BVHs): after the build in a batch run
// (WIDE: walking the 4-wide nodes of the widen phase), or as the
// continuous-batching step of the serving loop (its binary or wide nodes).
// WAVES waves per SIMD cap the registers: the 4-wide walk fits 8 (64 VGPRs)
// where its LDS stack allows, the binary walk 7-8. WAVE_ITEMS (the batch run):
// waves take items on their own and never wait for the rest of their block;
// otherwise (the serving step, whose tiles are sized for a block) a block
// takes an item and its waves share it.
template <int DEPTH, bool TSTACK, int WAVES, bool WIDE, bool WAVE_ITEMS = WIDE>
__global__ __launch_bounds__(BUILD_BLOCK) __attribute__((amdgpu_waves_per_eu(WAVES))) void
k_batch_trace(BatchArgs a) {
  __shared__ uint32_t lds[DEPTH * BUILD_BLOCK * (TSTACK ? 2 : 1)];
  __shared__ uint32_t s_item, s_ctr;
  if (threadIdx.x == 0)
    atomicAdd(a.ctl + BATCH_XTICKET_BASE + blockIdx.x % BATCH_XCDS * BATCH_XTICKET_STRIDE +
                  BATCH_XBLOCKS, 1u);
  if constexpr (WAVE_ITEMS) {
    ItemSlices src{a, SegItems(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)), 0u, 0u, 0u,
                   BatchWork{}, false, false};
    if (!src.take(src.held)) return;
    for (;;) {
      const BatchMeshDev m = load_uniform(a.meshes + src.held.mesh);
      src.mesh = src.held.mesh, src.kind = src.held.tile & BATCH_ANY_BIT, src.nrays = m.nrays;
      src.first = true, src.have_held = false;
      trace_mesh<DEPTH, TSTACK, WIDE>(a, m, lds, &src);
      if (!src.have_held) return;
    }
  } else {
    __shared__ SplitSlots s_split[WIDE ? BUILD_BLOCK / 64 : 1];
    SplitSlots* const slots =
        s_split + (WIDE ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0u);
    SegQueue<1> queue(0u);
    for (;;) {
      if (threadIdx.x == 0) s_item = queue.take(a);
      __syncthreads();
      const uint32_t it = __builtin_amdgcn_readfirstlane(s_item);
      __syncthreads();
      if (it == NO_ITEM) return;
      const BatchWork w = load_uniform(a.items + it);
      trace_item<DEPTH, TSTACK, WIDE>(a, w, lds, &s_ctr, slots);
    }
  }
}

typedef void (*BatchFn)(BatchArgs);
struct BatchVariant {
  int depth;
  bool tstack;
  BatchFn fn;
};
// The sort passes of a batch build, by waves per SIMD (the register cap trades
// occupancy against spills of their look-back window).
#define RQ_SORTS(W) {k_batch_sort<0, W>, k_batch_sort<1, W>, k_batch_sort<2, W>, k_batch_sort<3, W>}
const BatchFn kSort[][SORT_PASSES] = {RQ_SORTS(8), RQ_SORTS(7), RQ_SORTS(6), RQ_SORTS(5), RQ_SORTS(4)};
#undef RQ_SORTS
constexpr int kBuildWaves[] = {8, 7, 6, 5, 4};
constexpr int kNumBuildVariants = sizeof(kBuildWaves) / sizeof(kBuildWaves[0]);
// Trace kernels of a batch run (4-wide walk): the batch configurations.
const BatchVariant kBatchVariants[] = {
    {24, false, k_batch_trace<24, false, 6, true>},
    {16, false, k_batch_trace<16, false, 8, true>},
    {32, false, k_batch_trace<32, false, 4, true>},
    {12, true, k_batch_trace<12, true, 6, true>},
    {28, false, k_batch_trace<28, false, 5, true>},
    {30, false, k_batch_trace<30, false, 5, true>}};
// Trace kernels of the serving loop: binary walks (0-5), then 4-wide walks
// with block-shared items (6-7; the slots keep wide nodes).
const BatchVariant kServeVariants[] = {
    {16, false, k_batch_trace<16, false, 7, false>}, {20, false, k_batch_trace<20, false, 7, false>},
    {8, true, k_batch_trace<8, true, 7, false>},     {10, true, k_batch_trace<10, true, 7, false>},
    {16, false, k_batch_trace<16, false, 8, false>}, {8, true, k_batch_trace<8, true, 8, false>},
    {16, false, k_batch_trace<16, false, 5, true, false>},
    {16, false, k_batch_trace<16, false, 8, true, false>}};
constexpr int kServeWideFirst = 6;
constexpr int kNumBatchVariants = sizeof(kBatchVariants) / sizeof(kBatchVariants[0]);
constexpr int kNumServeVariants = sizeof(kServeVariants) / sizeof(kServeVariants[0]);

uint32_t grid_blocks(int device, BatchFn fn) {
  int cus = 0, per = 0;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, BUILD_BLOCK, 0);
  if (cus <= 0) cus = 256;
  if (per <= 0) per = 1;
  return (uint32_t)(cus * per);
}

}  // namespace

int batch_num_variants() { return kNumBatchVariants; }
void batch_variant_info(int v, int* depth, int* tstack) {
  *depth = kBatchVariants[v].depth;
  *tstack = kBatchVariants[v].tstack ? 1 : 0;
}
int serve_num_variants() { return kNumServeVariants; }
void serve_variant_info(int v, int* depth, int* tstack, int* wide) {
  *depth = kServeVariants[v].depth;
  *tstack = kServeVariants[v].tstack ? 1 : 0;
  *wide = v >= kServeWideFirst ? 1 : 0;
}
int batch_num_build_variants() { return kNumBuildVariants; }
int batch_build_waves(int b) { return kBuildWaves[b]; }
uint32_t batch_trace_grid_blocks(int device, int v) {
  return grid_blocks(device, kBatchVariants[v].fn);
}
uint32_t serve_grid_blocks(int device, int v) { return grid_blocks(device, kServeVariants[v].fn); }

hipError_t launch_batch(const LaunchCtx& lc, const BatchArgs& a, int build, int variant,
                        uint32_t trace_grid) {
  {
    ProfScope ps(lc, "batch_build");
    auto phase = [&](int ph, BatchFn fn, uint32_t parts, int block) {
      const uint32_t items = a.phase_begin[ph + 1] - a.phase_begin[ph];
      const uint32_t grid = ph == PH_INIT ? std::max(1u, items) : items * parts;
      if (grid) hipLaunchKernelGGL(fn, dim3(grid), dim3(block), 0, lc.stream, a);
    };
    phase(PH_INIT, k_batch_init, 1, BUILD_BLOCK);
    phase(PH_BOUNDS, k_batch_bounds, 1, TRI_BLOCK);
    phase(PH_MORTON, k_batch_morton, 1, TRI_BLOCK);
    for (int p = 0; p < SORT_PASSES; ++p) phase(PH_SORT0 + p, kSort[build][p], 1, BUILD_BLOCK);
    phase(PH_KARRAS, k_batch_karras, KARRAS_PARTS, BUILD_BLOCK);
    phase(PH_REFIT, k_batch_refit, REFIT_PARTS, BATCH_REFIT_CHUNK);
    phase(PH_TOP, k_batch_span, BATCH_SPAN_TILES, BUILD_BLOCK);
    phase(PH_WIDEN, k_batch_widen, BATCH_SPAN_TILES, BUILD_BLOCK);
  }
  {
    ProfScope ps(lc, "batch_trace");
    hipLaunchKernelGGL(kBatchVariants[variant].fn, dim3(trace_grid), dim3(BUILD_BLOCK), 0,
                       lc.stream, a);
  }
  return hipGetLastError();
}

hipError_t launch_serve_trace(const LaunchCtx& lc, const BatchArgs& a, int variant, uint32_t grid) {
  ProfScope ps(lc, "batch_trace");
  hipLaunchKernelGGL(k_batch_reset, dim3(1), dim3(64), 0, lc.stream, a.ctl);
  hipLaunchKernelGGL(kServeVariants[variant].fn, dim3(grid), dim3(BUILD_BLOCK), 0, lc.stream, a);
  return hipGetLastError();
}

}  // namespace rq
