// Internal types of the batch kernels (batch_kernels.hip <-> batch.cpp).
#pragma once
#include "build_device.h"

namespace rq {

enum BatchPhase {
  PH_INIT = 0,
  PH_BOUNDS,
  PH_MORTON,
  PH_SORT0,
  PH_SORT1,
  PH_SORT2,
  PH_SORT3,
  PH_KARRAS,
  PH_REFIT,
  PH_TOP,
  PH_WIDEN,  // 4-wide nodes from the refitted binary records
  PH_TRACE,
  BATCH_PHASES
};

// The trace items are split into one queue segment per XCD (each XCD has its
// own L2): a mesh's rays are traced on one XCD, or two, so that its BVH stays
// in those L2s; a block drains its own XCD's segment first, then takes from
// the others.
constexpr int BATCH_XCDS = 8;
static_assert(BATCH_XCDS == (int)TRACE_SEGS, "blocks go to the segments in turn (seg_blocks)");

// control words of one batch
constexpr int BATCH_CTL_TRACE_ERR = 0;  // stack deeper than provided (this run)
// BATCH_PHASES 64-bit wall-clock stamps (8-byte aligned) of a run: stamp p =
// the start of phase p, or the build's end (0 where the phase has no items)
constexpr int BATCH_CTL_CLOCK = 2;
constexpr int BATCH_CTL_WORDS = BATCH_CTL_CLOCK + 2 * BATCH_PHASES;
// The tickets of the trace segments, after the control words, each on a 4 KB
// page of its own: atomics on one line queue (12 ns each).
constexpr int BATCH_XTICKET_STRIDE = 1024;  // words
constexpr int BATCH_XTICKET_BASE = BATCH_XTICKET_STRIDE;
constexpr int BATCH_CTL_ALLOC_WORDS = BATCH_XTICKET_BASE + BATCH_XCDS * BATCH_XTICKET_STRIDE;
static_assert(BATCH_CTL_WORDS <= BATCH_XTICKET_BASE, "control words before the tickets");
// A segment's page also counts the trace blocks that started on it, on another line.
constexpr int BATCH_XBLOCKS = 64;
constexpr uint32_t BATCH_ANY_BIT = 0x80000000u;            // trace item tile: any-hit query
// Work items of the refit phases (see batch_kernels.hip): BATCH_REFIT_CHUNKS
// times BUILD_BLOCK leaves an item of the first; spanning nodes in tiles of
// BUILD_BLOCK, BATCH_SPAN_TILES per item.
constexpr uint32_t BATCH_REFIT_CHUNKS = 4;
constexpr uint32_t BATCH_SPAN_TILES = 8;

struct BatchMeshDev {
  BuildView v;
  rq_rays rays;
  uint32_t nrays;
  int32_t* prim;
  float *t, *u, *v_;
  uint8_t* occ;
};

struct BatchWork {
  uint32_t mesh;
  uint32_t tile;  // unit of the phase; trace: ray tile, BATCH_ANY_BIT for any-hit
};

struct BatchArgs {
  const BatchMeshDev* meshes;
  const BatchWork* items;               // every phase's items, phase after phase
  uint32_t phase_begin[BATCH_PHASES + 1];
  uint32_t trace_seg[BATCH_XCDS + 1];   // trace items of XCD q: [trace_seg[q], trace_seg[q + 1])
  uint32_t* ctl;                        // BATCH_CTL_WORDS
  int32_t* gstack;                      // traversal stack overflow of the persistent grid
  uint32_t gdepth, gwords;              // its entries per thread, and their words
  uint32_t ray_tile;
  uint32_t refill_idle;
};

// Batch configurations: the trace kernels of a batch run (4-wide walk).
int batch_num_variants();
void batch_variant_info(int v, int* depth, int* tstack);
// The build's sort kernels by waves per SIMD (8, 7, 6, 5, 4).
int batch_num_build_variants();
int batch_build_waves(int build);
uint32_t batch_trace_grid_blocks(int device, int v);
// The serving loop's trace kernels (binary walk over its slots).
int serve_num_variants();
void serve_variant_info(int v, int* depth, int* tstack, int* wide);
uint32_t serve_grid_blocks(int device, int v);
// A batch run: resets the control words, then the build phases, a launch each
// (sort kernels `build`), and the trace kernel of `variant`.
hipError_t launch_batch(const LaunchCtx& lc, const BatchArgs& a, int build, int variant,
                        uint32_t trace_grid);
// The serving step: resets the control words, then the trace phase alone.
hipError_t launch_serve_trace(const LaunchCtx& lc, const BatchArgs& a, int variant, uint32_t grid);

}  // namespace rq
