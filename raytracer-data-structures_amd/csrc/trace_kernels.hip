// Standalone closest-hit / any-hit query kernels on gfx950: persistent waves
// running trace_loop (trace_device.h), a table of kernel variants for the
// autotuner, and the launcher.
//
// Kernel shape: persistent waves take slices of the ray stream from their
// segment's counter; when enough lanes have finished (wave ballot), the wave refills the
// idle lanes from its slice (ray compaction), so long rays do not hold a wave
// of finished lanes. The per-lane stack lives in LDS ([depth][lane],
// conflict-free) and spills to a global [depth][thread] area past the LDS
// depth of the variant.
#include <algorithm>

#include "trace_device.h"

namespace rq {
namespace {

// The kernel's arguments, read from its argument memory anew at each call
// (the empty asm hides that the address never changes).
typedef __attribute__((address_space(4))) const TraceArgs* ArgsPtr;
struct KernelArgs {
  __device__ ArgsPtr operator()() const {
    ArgsPtr p = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
  }
  __device__ LeafBoxes leaf_boxes() const {
    const ArgsPtr p = (*this)();
    return LeafBoxes{p->parent, p->nodes};
  }
};

// WAVES > 0: registers capped so that this many waves fit a SIMD.
template <bool ANY, bool COUNT, int BLOCK, int DEPTH, bool TSTACK, bool WIDE = false, int WAVES = 0>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WAVES > 0 ? WAVES : 1)))
void k_trace(TraceArgs a) {
  __shared__ int32_t s_node[DEPTH * BLOCK];
  __shared__ float s_tn[TSTACK ? DEPTH * BLOCK : 1];
  constexpr uint32_t WPB = BLOCK / 64;
  __shared__ SplitSlots s_split[WIDE ? WPB : 1];
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  QuerySlices<KernelArgs, (int)WPB> src(KernelArgs{}, wave);
  trace_loop_split<ANY, COUNT, BLOCK, DEPTH, TSTACK, WIDE>(a, KernelArgs{}, src, s_node, s_tn,
                                                           s_split + (WIDE ? wave : 0u));
}

// Device scratch of the allocation-free closest-hit entry
// (rq_closest_hit_noalloc): the launch's ray-stream counters in the first
// NOALLOC_COUNTER_BYTES, then the traversal stack overflow area
// ([depth][thread] entries). One copy per device, held from module load until
// the process ends; its address comes from hipGetSymbolAddress
// (noalloc_scratch_address), never from the array's name in host code. Calls
// that overlap on one device share it and race.
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

__global__ __launch_bounds__(64) void k_counter_reset(unsigned long long* ctr) {
  if (threadIdx.x < TRACE_SEGS) ctr[threadIdx.x * COUNTER_STRIDE] = 0ull;
}

typedef void (*TraceFn)(TraceArgs);
struct Variant {
  int block, depth;
  bool tstack, wide;
  int closest_waves, any_waves;  // waves per SIMD that are promised (0: none)
  TraceFn closest, any;
};

// Variant 0 is the canonical binary configuration (the counted kernels run
// it); the wide variants need the BVH's 4-wide nodes. A wide walk waits on
// dependent record fetches, so its kernels are compiled for as many waves per
// SIMD as their LDS stack leaves room for: eight (64 VGPRs) with 16 entries,
// six with 24. Left to itself the compiler takes 70 VGPRs and over 96 SGPRs,
// six waves. 8.3 M camera rays over 1.31 M triangles 0.78 ms at six, 0.73 at
// seven, 0.68 at eight; 8.3 M uniform rays over 5.24 M triangles 0.60, 0.55,
// 0.54 ms closest and 0.53, 0.48, 0.45 ms any hit. The launch grid follows
// each kernel's own occupancy.
constexpr int wide_waves(int depth, bool tstack) {
  int w = 8;
  while (w > 1 && w * 4 * (64 * depth * (tstack ? 8 : 4) + (int)sizeof(SplitSlots)) > 160 * 1024)
    --w;
  return w;
}
// What rq_trace_variant_get promises: six waves or more for the any-hit
// kernels with that much LDS, and for the closest-hit kernels of the last two
// variants.
constexpr int promised(bool wide, int depth) { return wide && depth <= 26 ? 6 : 0; }
#define RQ_WIDE(B, D, T, C)                                                  \
  {                                                                          \
    B, D, T, true, C, promised(true, D),                                     \
        k_trace<false, false, B, D, T, true, wide_waves(D, T)>,              \
        k_trace<true, false, B, D, false, true, wide_waves(D, false)>        \
  }
#define RQ_BINARY(B, D, T)                                                   \
  {                                                                          \
    B, D, T, false, 0, 0, k_trace<false, false, B, D, T>,                    \
        k_trace<true, false, B, D, false>                                    \
  }
const Variant kVariants[] = {
    RQ_BINARY(128, 24, false),   RQ_BINARY(128, 16, false),   RQ_BINARY(64, 24, false),
    RQ_BINARY(256, 16, false),   RQ_BINARY(128, 24, true),    RQ_BINARY(128, 16, true),
    RQ_BINARY(64, 16, true),     RQ_BINARY(64, 32, false),    RQ_BINARY(64, 12, true),
    RQ_WIDE(128, 16, false, 0),  RQ_WIDE(128, 32, false, 0),  RQ_WIDE(64, 32, false, 0),
    RQ_WIDE(128, 24, true, 0),   RQ_WIDE(64, 24, true, 0),    RQ_WIDE(256, 16, false, 0),
    RQ_WIDE(256, 24, false, 0),  RQ_WIDE(256, 28, false, 0),  RQ_WIDE(256, 16, false, 6),
    RQ_WIDE(128, 24, false, 6),
};
#undef RQ_WIDE
#undef RQ_BINARY
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);
static_assert(TRACE_DEFAULT_CLOSEST < kNumVariants && TRACE_DEFAULT_ANY < kNumVariants,
              "default variants in the table");

}  // namespace

int trace_num_variants() { return kNumVariants; }

static_assert(sizeof(kVariants) / sizeof(kVariants[0]) <= TRACE_MAX_VARIANTS, "variant table");

void trace_variant_info(int v, int* block, int* depth, int* tstack, int* wide,
                        int* closest_waves, int* any_waves) {
  const Variant& x = kVariants[v];
  *block = x.block, *depth = x.depth, *tstack = x.tstack ? 1 : 0;
  if (wide) *wide = x.wide ? 1 : 0;
  if (closest_waves) *closest_waves = x.closest_waves;
  if (any_waves) *any_waves = x.any_waves;
}

int trace_max_stack(int v) { return kVariants[v].wide ? TRACE_MAX_STACK_WIDE : TRACE_MAX_STACK; }

int trace_first_variant(int v, bool any) {
  for (int f = 0; f < v; ++f) {
    const Variant &a = kVariants[f], &b = kVariants[v];
    if (a.tstack == b.tstack && (any ? a.any == b.any : a.closest == b.closest)) return f;
  }
  return v;
}

uint32_t trace_grid_blocks(int device, int v, bool any) {
  int cus = 0, per = 0;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &per, any ? kVariants[v].any : kVariants[v].closest, kVariants[v].block, 0);
  if (cus <= 0) cus = 256;
  if (per <= 0) per = 2;
  return (uint32_t)(cus * per);
}

hipError_t noalloc_scratch_address(void** ptr) {
  *ptr = nullptr;
  return hipGetSymbolAddress(ptr, HIP_SYMBOL(scratch));
}

hipError_t launch_counter_reset(const LaunchCtx& lc, unsigned long long* counter) {
  hipLaunchKernelGGL(k_counter_reset, dim3(1), dim3(64), 0, lc.stream, counter);
  return hipGetLastError();
}

hipError_t launch_trace(const LaunchCtx& lc, const TraceArgs& a, bool any, bool counted,
                        int variant) {
  if (a.nrays == 0) return hipSuccess;
  // the instrumented kernels always run the canonical configuration (variant 0);
  // a wide variant needs the wide nodes
  if (!counted && kVariants[variant].wide && !a.wide) return hipErrorInvalidValue;
  const Variant& V = kVariants[counted ? 0 : variant];
  dim3 g(a.grid), blk(V.block);
  hipStream_t s = lc.stream;
  if (any) {
    ProfScope ps(lc, counted ? "trace_any_counted" : "trace_any");
    if (counted)
      hipLaunchKernelGGL((k_trace<true, true, 128, 24, false>), g, blk, 0, s, a);
    else
      hipLaunchKernelGGL(V.any, g, blk, 0, s, a);
  } else {
    ProfScope ps(lc, counted ? "trace_closest_counted" : "trace_closest");
    if (counted)
      hipLaunchKernelGGL((k_trace<false, true, 128, 24, false>), g, blk, 0, s, a);
    else
      hipLaunchKernelGGL(V.closest, g, blk, 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace rq
