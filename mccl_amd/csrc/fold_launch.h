// fold_launch.h -- host/device shared argument blocks of the fold kernels and
// the internal launch entry used by the C ABI (mcclx_api.cpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mcclx.h"

namespace mcclx {

// Segments that travel by value in the kernel arguments (32 x 88 B = 2.8 KB).
// A block that finds its descriptor there starts loading data at once; one that
// must first fetch it from a device table loses 5-10 % on large segments.
constexpr int kFewSegs = 32;

// Device-side view of mcclx_seg (same layout: the table is uploaded verbatim).
struct SegArgs {
    void* out;
    void* wire_out;
    const void* in[MCCLX_MAX_INPUTS];
    uint64_t count;
};
static_assert(sizeof(SegArgs) == sizeof(mcclx_seg), "SegArgs must mirror mcclx_seg");

// Launch-timeline instrumentation (a tuning build only, -DMCCLX_TUNE_TIMELINE=1):
// every block of a by-value fold launch records when it started, when its
// arguments had arrived and when it had issued its last store.
#ifndef MCCLX_TUNE_TIMELINE
#define MCCLX_TUNE_TIMELINE 0
#endif
struct TimelineRecord {
    uint64_t t_start, t_args, t_end;  // 100 MHz wall clock (10 ns ticks)
    uint32_t hw_id, xcc_id;           // where the block ran: HW_ID register, XCC_ID register
};

struct FewArgs {
    SegArgs seg[kFewSegs];
    float scale;        // the constant as the fp32 value the kernel multiplies by
    int32_t has_scale;
    int32_t nseg;
    int32_t fan;        // further destinations of the result, in[k .. k+fan-1] (fan-out kernels only)
    int32_t op;         // the operator, where the kernel takes it from here (to-all kernels of MIN, MAX, PRODUCT)
    // Fan-out and to-all kernels, where not null: the last block to end writes `mark_number` there.
    uint64_t* mark_word;
    uint32_t* mark_count;  // blocks that have ended, 0 between launches
    uint64_t mark_number;
    uint32_t mark_blocks;  // blocks of the launch
#if MCCLX_TUNE_TIMELINE
    TimelineRecord* timeline;  // this launch's records, one per block (x fastest, then y), or null
#endif
};

struct TableArgs {
    const SegArgs* __restrict__ segs;         // device memory, nseg entries
    const uint64_t* __restrict__ first_item;  // device memory, nseg+1 prefix sums (unused when uniform)
    const uint2* __restrict__ item_map;       // device memory, (segment, tile) of every work item, or null
    uint64_t total_items;
    uint64_t uniform_items;      // >0: every segment has this many work items
    uint32_t nseg;
    float scale;
    int32_t has_scale;
    int32_t fan;                 // further destinations of the result, in[k .. k+fan-1] (fan-out kernels only)
    int32_t op;                  // as FewArgs::op
};

// Kernel-side operator codes beyond the public MCCLX_* ones: MIN / MAX with the
// accumulator in the reference's `src` role (plan flag MCCLX_PLAN_ACC_IS_SRC).
enum { MCCLX_MIN_ACC_SRC = 5, MCCLX_MAX_ACC_SRC = 6 };

struct PlanKey {
    int dtype, io, k, topo, op, acc;
};

// A launch that tells the host of its own end (mcclx_queue_wait's word), if it has few enough blocks.
struct LaunchMark {
    uint64_t* word;
    uint32_t* count;
    uint64_t number;
    bool taken = false;
};

struct LaunchParams {
    LaunchMark* mark = nullptr;
    const FewArgs* few = nullptr;      // exactly one of few / table is set
    const TableArgs* table = nullptr;
    uint32_t max_blocks = 0;           // cap on the grid (persistent sizing)
    int fan = 0;                       // > 0: the fan-out form of the kernel (plans in fan_plan_ok only)
    bool to_all = false;               // the to-all form: the result goes back into every operand (all_plan_ok only)
    // Reads-then-writes form of a by-value launch that one generation of blocks covers:
    // taken when the launch reads at least hold_min_read_bytes (0 = never); no lane stores
    // before hold_latency_ticks + read bytes / hold_bytes_per_tick ticks of the 100 MHz
    // wall clock have passed since its block started.
    int cus = 0;
    bool far_out = false;              // a large cast's result lies outside the device's memory
    bool* held = nullptr;              // set when the launch took that form (diagnostic)
    bool* four = nullptr;              // set when a by-value launch took blocks of four wavefronts (diagnostic)
    uint64_t hold_min_read_bytes = 0;
    uint32_t hold_latency_ticks = 40;
    uint32_t hold_bytes_per_tick = 72000;
};
// Plans that have a fan-out form: sums with per-step rounding, 2..7 operands.
bool fan_plan_ok(const PlanKey& key);
// Plans that have a to-all form: per-step rounding, every operand in the form of the result.
bool all_plan_ok(const PlanKey& key);

// One launch that folds segments 0..nfold-1 of `few` (a fan-out plan of up to four operands over
// the wire codec, the owner's operand fp32) and encodes the others (fp32 -> bf16), tile by tile in
// turn.  fold_encode_ok: the plans there are.
bool fold_encode_ok(const PlanKey& key);
hipError_t launch_fold_encode(hipStream_t st, const PlanKey& key, const FewArgs& few, uint32_t nfold);

// One tensor to its wire form or back, as the plans of one operand without a scale give it (per-step rounding):
// dst <- src, up to 2^33 elements.  `far`: dst lies outside the device's memory (a choice of shape).
hipError_t launch_cast(hipStream_t st, bool decode, void* dst, const void* src, uint64_t count, int cus, bool far);

// Can a segment of `count` elements be launched by value?  A grid has at most 2^32 threads, one
// per packet there (more are dropped without an error); the table kernels loop.
bool few_fits(const PlanKey& key, uint64_t count);

// Packets-per-lane unroll and threads per block the kernel template uses for this plan.
int plan_unroll(const PlanKey& key);
int plan_block(const PlanKey& key);
// Work items (tiles) a segment of `count` elements splits into under this plan.
uint32_t items_for(const PlanKey& key, uint64_t count);
// hipErrorInvalidValue = no kernel for this plan.
hipError_t launch_fold(hipStream_t st, const PlanKey& key, const LaunchParams& lp);

// How many one-wavefront blocks share a CU in a large launch of several streams (by value; what
// launch_table takes of it is said there).
//
// A full CU holds 32 of them, and a launch of k operands then has 32 * k KiB of loads per CU
// under way, spread over a range of every stream that is wider than what the memory channels
// keep open: the more streams, the more rows each channel switches between, and the slower
// the launch (measured on 1-4 GB, TB/s at 32 waves: one stream in and one out 6.7, three in
// one out 6.4, four tensors reduced in place 5.9, eight in place 5.5, one to eight 5.3).
// With fewer waves resident the same launches run at 6.1-6.8 TB/s: what a channel sees at
// one time shrinks with the bytes under way, and 70-80 KiB per CU (20 MB on the device) still
// covers the latency.  The optimum, swept over 3..20 waves per CU, lies near one number of
// bytes for every shape, waves x bytes a lane moves: 1160 (8 operands into one: 8 waves;
// 4 into one: 14; 3 into one: 18), a little less where one source is copied to several
// destinations (4 / 6 / 8: 12 / 9 / 7 waves, 33 M elements to four 214 -> 206 us against 14)
// and a little more or less where tensors are reduced in place or to several (Cfg::kInPlaceBudget, kFanBudget).  A reservation of LDS nobody uses
// sets the number: it is granted in units of 1280 bytes of a CU's 160 KiB.
//
// A launch that ends soon needs its waves to get going: the limit pays from 160 MB moved on
// (200 MB, eight operands into one: 36.2 -> 35.4 us; 80 MB: 5.5 TB/s without it, 5.1 with),
// and not where 20 waves or more would be left of a launch with one output.  Copies, whose waves have
// nothing to do between load and store, gain from 90 MB on (eight to eight, 144 MB: 30.5 -> 28.6 us, 86 MB
// level; two to two, 96 MB: 17.9 -> 16.8).
constexpr uint64_t kResidentMinBytes = 160'000'000;
constexpr uint64_t kResidentMinBytesCopy = 90'000'000;
constexpr int kLaneBytes = 1160, kLaneBytesInPlace = 1280, kLaneBytesCopy = 1020;
constexpr int kMostResident = 18;
inline uint32_t resident_lds(uint64_t launch_bytes, int lane_bytes, int outputs, int budget = kLaneBytes,
                             uint64_t min_bytes = kResidentMinBytes) {
    int waves = budget / lane_bytes;
    if (launch_bytes < min_bytes || (outputs == 1 && waves >= 20)) return 0;
    waves = waves > kMostResident ? kMostResident : waves < 3 ? 3 : waves;  // three blocks reserve 53 KiB each: a launch may ask for 64 KiB
    return 163840u / (uint32_t)waves / 1280u * 1280u;
}

// Launches that one generation of waves nearly covers (8192 on 256 CUs) start sooner in
// blocks of four wavefronts: 4 MB copied in 2.5 us against 2.9, an encode of 4 MB 2.3 against
// 2.7; larger ones stream faster in one-wavefront blocks, whose slots turn over one by one
// (27 MB copied: 10.1 -> 9.2 us, a two-operand wire fold of a 25 MiB bucket: 12.5 -> 11.4 us).
constexpr uint64_t kOneWaveBlocksFrom = 12288;

// Many copies in one launch: descriptors and n+1 work-item prefix sums in
// device memory.  A descriptor is one source and everybody who gets it: copies
// that share a source (the allgather leg hands every chunk to every other rank)
// read it once.
constexpr int kCopyDsts = 8;
struct CopyDesc {
    const void* src;
    uint64_t nbytes;
    uint64_t n;  // destinations, 1..kCopyDsts
    void* dst[kCopyDsts];
};
struct CopyTable {
    const CopyDesc* __restrict__ descs;
    const uint64_t* __restrict__ first_item;
    const uint2* __restrict__ item_map;  // (copy, tile) of every work item, or null
    uint32_t total_items;
    uint32_t uniform_items;  // >0: every copy has this many work items
    uint32_t n;
};
// A few copies by value in the kernel arguments (one grid: y = copy, x = tile).
constexpr int kFewCopies = 32;
struct CopyFew {
    CopyDesc d[kFewCopies];
    uint32_t n;
};
// `spread`: one destination after another (copy_spread_pays).  For memory of this device alone: its caches hold no other
// sources, and destinations behind links of their own want to be written side by side.
hipError_t launch_copy_few(hipStream_t st, const CopyFew& copies, bool spread);
// Is `spread` the faster form of these copies, where all of their memory is this device's?
bool copy_spread_pays(const CopyFew& copies);
// Work items (tiles) one copy of nbytes splits into.
uint64_t copy_items(uint64_t nbytes);
// `most`: the largest number of destinations any descriptor of the launch has.
hipError_t launch_copy_many(hipStream_t st, const CopyTable& t, int most, uint32_t max_blocks);

// Plain device copy with the same packet shape (also the calibration kernel for
// the memory counters): dst <- src, nbytes.
hipError_t launch_copy(hipStream_t st, void* dst, const void* src, uint64_t nbytes);

// Behind everything on the stream: *word = number, in pinned host memory (`word` as the device addresses it).
hipError_t launch_word(hipStream_t st, uint64_t* word, uint64_t number);

// Reads (write == false) or writes nbytes of `buf` once, one 16-byte packet per
// lane like the copy kernel: the one-directional ceilings of a launch of that size.
hipError_t launch_stream_probe(hipStream_t st, void* buf, uint64_t nbytes, bool write);

// The allocation-free batched fold keeps its descriptor table in a static
// device array of kStaticTableBytes (one per GPU): room for
// MCCLX_NOALLOC_MAX_SEGS descriptors of 88 bytes plus their work-item prefix
// sums.  `static_table_resolve` returns that array's address on `device`, which
// must be the current device; `launch_table_write` stores up to kUploadWords
// 8-byte words there, carried in the kernel arguments of a one-block launch.
constexpr size_t kStaticTableBytes = 128 * 1024;
constexpr uint32_t kUploadWords = 448;  // 3584 bytes of payload per writer launch
static_assert((size_t)MCCLX_NOALLOC_MAX_SEGS * sizeof(SegArgs) +
                  ((size_t)MCCLX_NOALLOC_MAX_SEGS + 1) * sizeof(uint64_t) <= kStaticTableBytes,
              "the static table must hold the largest allocation-free launch");
hipError_t static_table_resolve(int device, void** out);
hipError_t launch_table_write(hipStream_t st, void* dst_words, const uint64_t* words, uint32_t n);

}  // namespace mcclx
