// Internal interface between the C ABI (dz_api.hip) and the kernels (dz_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dz_common.h"

namespace dz {

enum RmwMode : int {
  kModePerturb = 0,               // theta + b(z)
  kModeUpdate = 1,                // theta - d(z)
  kModeRestoreUpdate = 2,         // theta + b(z) - d(z)
  kModeRestoreUpdatePerturb = 3,  // theta + b(z) - d(z) + b(z'), z' from a second seed
  kModePerturbUnit = 4,           // perturb with scale 1 (rmw_short_kernel only)
};
// Modes whose table entries hold the pair (b, -d).
__host__ __device__ constexpr bool rmw_pair_mode(int mode) {
  return mode == kModeRestoreUpdate || mode == kModeRestoreUpdatePerturb;
}
enum ProjMode : int {
  kProjSumsq = 0,         // per-chunk sums of R_T(theta - theta0)^2
  kProjApply = 1,         // theta <- R(R(R(theta - theta0) * alpha) + theta0), alpha in T
  kProjReverse = 2,       // theta <- R(R(R(theta - theta0) / alpha) + theta0)
  kProjReverseSumsq = 3,  // REVERSE, then the sums of the new theta
  kProjApplyF32 = 4,      // theta <- R_T(fp32(R(theta - theta0)) * alpha + theta0), alpha fp32
  kProjDot = 5,           // per-chunk sums of fp32(other) * fp32(R_T(theta - theta0))
};
// Modes that write theta (and read an alpha), and modes that sum.
__host__ __device__ constexpr bool proj_stores(int mode) { return mode != kProjSumsq && mode != kProjDot; }
__host__ __device__ constexpr bool proj_sums(int mode) {
  return mode == kProjSumsq || mode == kProjReverseSumsq || mode == kProjDot;
}
// Most groups one dot launch takes (their pointers travel as kernel arguments, of
// which a launch has 4 KB); dz_group_dot launches once per batch of groups. With
// 128, 3,000 fp16 groups of 33,001 elements took 742 us, with 448 298; 24 groups
// of 20,480 6.7 and 6.6.
constexpr int kMaxDotGroups = 448;
struct DotGroups {
  uint64_t other[kMaxDotGroups];  // of groups group_base, group_base + 1, ...
  uint32_t group_base;
  uint32_t chunk_base;  // short tables: the launch's first chunk in the table's list
};

// Read-modify-write kernel geometry. A workgroup of 1024 threads takes one
// tile at a time from the table's work counters; each thread owns
// rmw_groups(dtype, mode) groups of 8 elements per tile. Measured on the MI355X at
// OPT-13B size (643 tensors, fp16): 64 KB tiles (four groups per thread) and
// one workgroup per CU stream best for every mode: perturb 6.4 TB/s against
// 6.05 with 16 KB tiles and two workgroups per CU (which a 64 KB table would
// allow); 32 KB and 128 KB tiles were no better, and the three-way pass took
// 7.96 ms with six groups per thread and spilled with eight. fp32 uses 32 KB
// tiles (one group of 8 fp32 per thread): OPT-125m (347 MB of parameters,
// about 40 tiles per CU) runs its perturb / three-way pass in 108 / 109 us that
// way against 112 / 114 us with 64 KB tiles, 2^28 elements in 322 / 324 against
// 336 / 331 us. The bf16 restore + update + next
// perturbation pass (prefetching loop, ALU-bound) takes three groups per
// thread (48 KB tiles): at OPT-30B 18.87-18.94 ms against 19.79-19.86 ms with
// four and 19.57-19.62 with two (same box, alternating builds), where the
// single-value bf16 passes take 19.3 ms with three and 17.6 with four, and
// the fp16 three-way pass 8.07 ms with three against 7.60 with four. A table
// whose three-way tile size differs keeps a second tile list for it.
constexpr int kRmwThreads = 1024;
__host__ __device__ constexpr int rmw_groups(int dtype, int mode) {
  return dtype == DZ_F32 ? 1 : (dtype == DZ_BF16 && mode == kModeRestoreUpdatePerturb) ? 3 : 4;
}
// Elements per tile of an RMW launch (the size of the table's tile list it runs over).
__host__ __device__ constexpr int rmw_chunk_elems(int dtype, int mode) {
  return kRmwThreads * rmw_groups(dtype, mode) * 8;
}

// Short tables: up to short_elems(dtype, mode) elements in all, where a pass runs
// rmw_short_kernel over tiles of kShortTile elements. Where the lines lie: pass
// times in us (perturb / update / restore + update / three-way) of the short
// kernel and of the persistent one, three tables used in turn: fp16 2^24
// elements 12.6 / 13.0 / 14.1 / 18.2 and 17.4 / 18.1 / 19.6 / 21.7, 2^24.5 16.5
// / 17.0 / 18.0 / 23.8 and 19.0 / 19.2 / 20.3 / 22.2, 2^25.5 31.9 / 30.5 / 31.2
// / 38.2 and 34.1 / 31.7 / 32.0 / 33.8, 2^26 43.7 / 42.3 / 43.1 / 51.4 and 46.0
// / 41.7 / 42.4 / 43.9; bf16 2^23.5 10.7 / 11.0 / 13.2 / 17.5 and 18.2 / 19.1 /
// 21.3 / 19.8, 2^24 13.2 / 14.0 / 17.3 / 22.7 and 19.0 / 19.9 / 21.7 / 20.2,
// 2^25 21.7 / 22.5 / 27.3 / 38.0 and 24.8 / 25.1 / 26.4 / 28.1, 2^26 44.1 / 43.1
// / 48.1 / 69.4 and 46.0 / 42.8 / 44.1 / 46.6; fp32 2^24 21.8 / 21.8 / 21.8 /
// 22.7 and 22.4 / 22.6 / 22.5 / 23.6, 2^24.5 32.4 / 30.3 / 30.4 / 31.4 and 30.6
// / 29.9 / 29.8 / 30.5.
constexpr uint32_t kShortTile = kRmwThreads * 8;
constexpr uint64_t short_elems(int dtype, int mode) {
  if (dtype == DZ_F32) return 1u << 24;
  if (mode == kModeRestoreUpdatePerturb) return dtype == DZ_F16 ? 5u << 22 : 3u << 22;
  if (mode == kModeRestoreUpdate) return dtype == DZ_F16 ? 3u << 24 : 3u << 23;
  return 1u << 26;
}

// Tensors of up to kPlainBytes in all, the size of the Infinity Cache, are read
// and written with plain accesses by the persistent kernel; longer tables'
// accesses carry the non-temporal hint. What a plain pass leaves in the cache the
// forward reads there: GPU time in us of perturb + products of 1,536 tokens with
// all the weights + three-way pass + products, with the hint and without, fp16 81
// MB 908 and 859, 121 MB 1340 and 1258, 162 MB 1879 and 1664, 229 MB 2638 and 2429
// (of 256 tokens 1977 and 1598), bf16 229 MB 2609 and 2398, fp32 108 MB 2041 and
// 2017, 216 MB 3856 and 3821. The passes themselves, kernel time in us (perturb /
// three-way), three tables used in turn: fp16 2^26 elements (128 MB) 47.0 / 51.0
// and 47.3 / 45.7, 2^27 87.5 / 91.6 and 82.9 / 84.7, 2^27.25 104 / 110 and 113 /
// 115, 2^28 169 / 173 and 183 / 185; fp32 2^25 44.9 / 45.4 and 43.1 / 40.8, 2^26
// (256 MB) 83.7 / 85.0 and 78.2 / 78.0, 2^26.25 99 / 101 and 111 / 104, 2^28 323 /
// 326 and 358 / 356. (Between 64 and 256 MB a plain pass's write-backs fall into
// what follows: passes back to back over three tables, fp16 2^27 elements 93.4 /
// 94.9 a pass, with the hint 88.0 / 92.4.)
constexpr uint64_t kPlainBytes = 1u << 28;

// LDS bytes of the per-launch delta table of an RMW launch: 16-bit entries
// for perturb/update of 16-bit T, 32-bit entries otherwise (fp32 deltas, or
// the (restore delta, update delta) pair of a fused restore+update).
__host__ __device__ constexpr int rmw_lds_table_bytes(int dtype, int mode) {
  return (dtype == DZ_F32 || rmw_pair_mode(mode)) ? kDzTabEntries * 4 : kDzTabEntries * 2;
}

// Work counters of a table, one set per table, 128 bytes apart: kCounters
// tile (chunk) dispensers, then (slot kDoneSlot) the number of finished
// workgroups. Zeroed when the table is created; the last workgroup of every
// launch puts them back to zero, so consecutive launches on one stream need
// no reset (and no memset in a captured graph). Launches of one table must
// not overlap in time. Four counters stream as fast as eight at OPT-13B
// (every mode within 0.3 %), sixteen 0.6-1.2 % slower; a single counter
// serialises at about 11 ns per atomic.
constexpr int kCounters = 8;
constexpr int kDoneSlot = kCounters;
constexpr int kCounterStride = 32;  // uint32 slots (128 bytes)
constexpr int kCounterWords = (kDoneSlot + 1) * kCounterStride;

// Tile loops of the RMW launches. The restore + update + next perturbation
// passes, whose ALU work per tile is the largest, run the prefetching loop
// (rmw_tiles_prefetch: the next full tile's loads go out once the tile's
// first group is stored). Measured on the MI355X, same box, alternating builds,
// kernel microbench, plain loop against loads half-way: OPT-13B fp16 7.86-7.90
// -> 7.58-7.61 ms, OPT-30B bf16 20.10-20.16 -> 19.83-19.95 ms. The
// single-Philox passes run the same
// on either loop (OPT-13B fp16 perturb 7.66-7.69 ms both, OPT-30B bf16
// 17.76 ms both) and keep the plain loop (rmw_tiles).
__host__ __device__ constexpr bool rmw_prefetch_mode(int dtype, int mode) {
  return mode == kModeRestoreUpdatePerturb;
}
// A table's default for the launches that use the prefetching loop: those of
// at least this many tiles (dz_table_set_prefetch_min_tiles sets it per
// table). 0: every launch of such a mode. With the next tile's loads issued
// inside the tile's work, the prefetching loop is also the faster one for a short pass
// (OPT-2.7B fp16, 77 K tiles, in the ZO step: 1.544-1.545 against
// 1.562-1.563 ms).
constexpr uint32_t kPrefetchMinTilesDefault = 0;

// Projection kernel geometry: persistent 1024-thread workgroups, one per CU,
// taking chunks of proj_chunk_elems(dtype) elements: 32768 for 16-bit T (64 KB
// of theta and 64 KB of theta0, 4 16-byte vectors of each per thread), 8192
// for fp32 (32 KB, 2 vectors). Two workgroups per CU streamed slower (6.49
// against 6.76 TB/s for a bare two-read-one-write kernel), as did smaller
// workgroups on one counter. fp32's only workload, OPT-125m, projects 57 MB
// per stream: 432 chunks of 32768 left two thirds of the CUs with two chunks
// and the rest with one. In its ZO step (same box, two alternating runs
// each), apply / norm / reverse+norm took 46 / 36 / 47 us with 32768-element
// chunks, 34 / 30 / 40 with 16384, 32 / 31 / 40 with 8192 and 31 / 37 / 44
// with 4096.
constexpr int kProjThreads = 1024;
__host__ __device__ constexpr int proj_chunk_elems(int dtype) { return dtype == DZ_F32 ? 8192 : 32768; }
// Groups whose alphas a projection workgroup keeps in LDS (16 KB of fp32);
// beyond that each chunk reads its group's alpha from memory.
constexpr int kProjAlphaLds = 4096;

// Short projection tables: up to kShortProjTotal elements in all, whose launches
// run proj_short_kernel over chunks of short_proj_elems(dtype) elements, a
// workgroup of kShortProjThreads each. Pass times in us (norms / apply / reverse
// + norms / dot; with the group sums), against the persistent kernel, passes back
// to back, three tables used in turn: fp16 128 x 20,480 elements 5.6 / 4.6 / 6.4
// and 14.9 / 11.9 / 22.1 (norms to reverse), 24 x 174,762 6.7 / 5.9 / 9.2 / 8.3
// and 16.8 / 16.2 / 25.9 / 21.0, 24 x 699,050 15.1 / 16.0 / 20.4 / 20.8 and 22.3 /
// 25.3 / 30.7 / 29.0, 2^24 in one group 15.2 / 15.5 / 20.9 / 21.7 and 20.2 / 22.1 /
// 29.4 / 25.8, 2^25 in 24 26.8 / 35.4 / 39.1 / 39.1 and 29.8 / 40.8 / 47.2 / 40.3,
// in one 28.4 / 35.3 / 40.8 / 41.7 and 28.7 / 35.6 / 41.3 / 37.9, 3 x 2^24 in 24
// 36.9 / 55.1 / 59.3 / 55.2 and 39.3 / 50.7 / 56.8 / 54.9; fp32 2^24 in eight 26.6 /
// 35.4 / 39.5 / 38.3 and 31.5 / 35.9 / 43.0 / 39.8, 5,000 x 4,097 37.0 / 46.5 /
// 51.0 / - and 64.0 / 50.1 / 75.0 / -, 3 x 2^24 in 48 69.4 / 110.5 / 113.1 / 102.3
// and 74.1 / 95.1 / 113.2 / 102.0. From 2^26 bytes on the persistent kernel's
// streaming stores make an apply faster when passes follow one another; with
// products over the projected weights between them, as in the gamma search, the
// plain stores are the better ones up to here (they leave the weights in the
// Infinity Cache): apply + reverse and the products in us, short and persistent,
// fp16 36 x 2^20 elements 75 + 708 and 88 + 853, 44 x 2^20 89 + 866 and 102 + 1039,
// fp32 32 x 2^20 133 + 2285 and 146 + 2307, 44 x 2^20 175 + 3059 and 192 + 3068.
// Larger tables whose groups fill the persistent kernel's chunks to at most one
// kShortProjFill-th run it too: fp16 60,000 x 1,100 143 / 84 / 182 and 626 / 394 /
// 793 (norms to reverse), 20,000 x 3,000 57 / 68 / 71 and 189 / 109 / 234, fp32
// 30,000 x 2,003 112 / 130 / 149 and 325 / 209 / 399 (fuller chunks: fp16 4,000 x
// 16,384 50 / 73 / 76 and 67 / 63 / 89).
// Chunks of half the size cost more counting (fp16 24 x 589,824: norms 17.4
// against 12.6), of twice the size run the same.
constexpr int kShortProjThreads = 256;
__host__ __device__ constexpr int short_proj_elems(int dtype) { return dtype == DZ_F32 ? 2048 : 4096; }
constexpr uint64_t kShortProjTotal = 3u << 24;
constexpr uint64_t kShortProjFill = 4;
constexpr uint64_t kShortProjChunks = 1u << 22;  // workgroups of a launch
// Tables whose largest group has more chunks than this, or of more groups (whose
// counts would take over 8 MB), keep no counts: a second launch adds up the chunk
// sums (short_sums_kernel). A group's counts queue up,
// 13 ns each: norms in us with counts and with a second launch, fp16 2^20 elements
// in one group (256 chunks) 7.0 and 8.8, 2^22 in four (256) 8.6 and 8.3, in two
// (512) 13.5 and 8.5, in one (1,024) 17.4 and 8.8, 2^23 in 12 (171) 10.2 and 10.8,
// in eight (256) 10.6 and 10.4, 2^24 in 16 (256) 16.2 and 14.6, in one (4,096) 57.5
// and 15.0; fp32 2^24 in one (8,192) 109.8 and 28.3.
constexpr uint32_t kShortCountChunks = 256;
constexpr int32_t kShortCountGroups = 1 << 16;
// The groups' finished-chunk counts lie 128 bytes apart: side by side, every
// workgroup's atomic met in the same lines (12 ns each: the norms of fp16 24 x
// 589,824, 3,456 counts, took 43 us against 13).
constexpr int kDoneStride = 32;  // uint32 slots

// By-value scalars of one RMW launch.
struct DzScalars {
  uint64_t seed;
  uint64_t seed2;  // seed of the next step's perturbation (kModeRestoreUpdatePerturb)
  float scale;  // scaling_factor s of the perturbation
  float eps;    // zo_eps
  float grad;   // projected_grad g
  float lr;     // learning rate of this update
};

// Optional device-resident overrides (read by the kernel when non-null), so a
// captured graph can replay with a new seed / gradient / learning rate.
struct DzScalarPtrs {
  const uint64_t* seed;   // device uint64
  const uint64_t* seed2;  // device uint64
  const void* grad;      // device scalar of the table dtype T
  const float* lr;       // device fp32
};

// Timing events of one launch: when set, the runtime records `start` as the
// kernel starts and `stop` as it ends (hipExtLaunchKernel), so an event pair
// brackets the kernel itself rather than the host's launch work as well.
struct LaunchEvents {
  hipEvent_t start = nullptr;
  hipEvent_t stop = nullptr;
};

// The chunk list holds its full tiles first; the rest are partial. prefetch: run the prefetching tile loop where the mode
// allows it (rmw_prefetch_mode); the caller sets it for long launches.
hipError_t launch_rmw(int dtype, int mode, const DzChunk* chunks, uint32_t nchunks, uint32_t grid,
                      const void* qtab, const DzScalars& s, const DzScalarPtrs& p, uint32_t* counters,
                      bool prefetch, bool plain, hipStream_t st, const LaunchEvents& ev = {});
// Launches of short tables, over tiles of kShortTile elements.
hipError_t launch_rmw_short(int dtype, int mode, const DzChunk* chunks, uint32_t nchunks, uint32_t cus,
                            const void* qtab, const DzScalars& s, const DzScalarPtrs& p, hipStream_t st,
                            const LaunchEvents& ev = {});
// Persistent: `grid` workgroups share the chunks through `counters` (zero
// before the launch; the launch leaves them at zero).
hipError_t launch_proj(int dtype, int mode, const DzChunk* chunks, uint32_t nchunks, uint32_t ngroups,
                       uint32_t grid, const void* alpha, double* partials, uint32_t* counters, hipStream_t st,
                       const LaunchEvents& ev = {});
// Per-group results of a norm pass; any may be NULL.
struct GroupOutputs {
  double* sumsq;
  float* norm_f32;
  void* norm_T;
};
// A projection launch over a short table: its chunk list (nchunks of them; an
// empty group has one of no elements) and each group's first chunk, the groups'
// finished-chunk counts (zero before the launch, which leaves them at zero;
// NULL: the launch stops at the chunks' partial sums).
struct ProjShort {
  const DzChunk* chunks;
  const uint32_t* group_begin;
  uint32_t* group_done;
  const void* alpha;
  double* partials;
  GroupOutputs out;
};
// The groups of a norm pass without a table: they travel as kernel arguments,
// kStaticPlanGroups to a launch. What short inputs leave in the scratch that all
// calls of a device share does not matter to the next call. Groups of up to
// kStaticSmallChunks chunks are summed by one workgroup each, larger ones by a
// second launch, kStaticSumGroups to a launch. (With a short table's
// finished-chunk counts, two calls that overlapped once left every later one
// wrong.) Call times in us, one launch / two launches / with counts, the host's
// launch work in them: 4 fp16 groups of 4 chunks 4.7-5.8 / 7.0-9.8 / 5.7, of 8
// 7.1 / 7.0-9.8 / 5.7, of 16 10.6 / 7.0-9.8 / 5.8; 4 fp32 groups of 8 5.7 /
// 7.0-9.8 / 5.8; 24 fp16 groups of 8 7.7 / 9.3-11.6 / 7.6. Two launches / with
// counts: 64 fp16 groups of 128 chunks 29 / 30, 24 fp32 groups of 288 (OPT-125m)
// 23.2-23.7 / 25.2-25.6, one fp16 group of 4,096 18 / 58.
constexpr int kStaticPlanGroups = 64;
struct StaticGroups {
  uint64_t ptr[kStaticPlanGroups];
  uint64_t anchor[kStaticPlanGroups];
  int64_t numel[kStaticPlanGroups];
  uint32_t chunk_begin[kStaticPlanGroups + 1];  // within the launch
  uint32_t ngroups;
  uint32_t group_base;
};
constexpr uint32_t kStaticSmallChunks = 8;
constexpr int kStaticSumGroups = 512;
// First chunks of the groups (and of the one behind the last) whose chunk sums a
// launch adds up: as arguments, or a table's list in device memory.
struct StaticSums {
  uint32_t chunk_begin[kStaticSumGroups + 1];
  uint32_t group_base;
};
struct TableSums {
  const uint32_t* chunk_begin;
  uint32_t group_base;
};
hipError_t launch_proj_short(int dtype, int mode, uint32_t nchunks, const ProjShort& a, hipStream_t st,
                             const LaunchEvents& ev = {});
// DOT launches, over the chunks of the groups in dg. The first: persistent, as
// launch_proj.
hipError_t launch_dot(int dtype, const DzChunk* chunks, uint32_t nchunks, uint32_t grid, const DotGroups& dg,
                      double* partials, uint32_t* counters, hipStream_t st, const LaunchEvents& ev = {});
hipError_t launch_dot_short(int dtype, uint32_t nchunks, const ProjShort& a, const DotGroups& dg, hipStream_t st,
                            const LaunchEvents& ev = {});
hipError_t launch_static_small(int dtype, const StaticGroups& sg, const GroupOutputs& out, hipStream_t st);
hipError_t launch_static_sumsq(int dtype, uint32_t nchunks, double* partials, const StaticGroups& sg, hipStream_t st);
hipError_t launch_static_sums(int dtype, uint32_t ngroups, const double* partials, const StaticSums& ss,
                              const GroupOutputs& out, hipStream_t st);
// The group sums of a launch over a short table without counts.
hipError_t launch_short_sums(int dtype, uint32_t ngroups, const double* partials, const TableSums& ts,
                             const GroupOutputs& out, bool take_sqrt, hipStream_t st, const LaunchEvents& ev = {});
// take_sqrt: norms (sqrt of the sums) or plain sums in the fp32 / T outputs.
hipError_t launch_finalize(int dtype, const double* partials, const uint32_t* gbegin, uint32_t ngroups,
                           double* sumsq, float* norm_f32, void* norm_T, bool take_sqrt, hipStream_t st,
                           const LaunchEvents& ev = {});
// Chunk plan of a projection launch without a table (dz_group_sumsq_static):
// kStaticPlanGroups groups per plan launch, their descriptors and the
// group -> chunk index written into caller-provided device memory.
struct StaticPlanBatch {
  uint64_t ptr[kStaticPlanGroups];
  uint64_t anchor[kStaticPlanGroups];
  int64_t numel[kStaticPlanGroups];
  uint32_t chunk_begin[kStaticPlanGroups];  // first chunk of each group of the batch
  uint32_t ngroups;                         // groups in this batch
  uint32_t group_base;                      // index of the batch's first group
  uint32_t total_groups;
  uint32_t total_chunks;
  int32_t elem_size;
  int32_t chunk_elems;  // proj_chunk_elems(dtype)
  uint32_t first;       // the first batch also zeroes the work counters
};
hipError_t launch_static_plan(const StaticPlanBatch& b, DzChunk* chunks, uint32_t* group_begin, uint32_t* counters,
                              hipStream_t st);
// z export: ranges of at least kNormalsLdsGroups Philox blocks of 8 elements
// run the persistent kernel with the quantile table in LDS. Kernel times by
// elements, table in memory against in LDS: fp16 2^16 2.8 / 3.6 us, 2^18 3.0 /
// 3.7, 2^19 3.5 / 3.8, 2^20 4.9 / 3.8, 2^22 12.7 / 5.4; fp32 2^18 3.5 / 4.1,
// 2^19 4.2 / 4.3, 2^20 6.0 / 4.6. The gathers from memory run at about one
// lane per clock and CU, so they cost more from 2^19 elements on.
constexpr int kNormalsThreads = 1024;
constexpr uint64_t kNormalsLdsGroups = 1u << 16;
hipError_t launch_normals(int dtype, const void* tab, uint64_t seed, uint32_t stream, uint64_t offset,
                          uint64_t n, void* out, uint32_t cus, hipStream_t st);
hipError_t launch_philox(uint64_t seed, uint32_t stream, uint64_t q0, uint64_t n, uint32_t* out,
                         hipStream_t st);

}  // namespace dz
