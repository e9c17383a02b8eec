// Fused NW DP launches (one per kernel family), defined in nw_fam_*.hip.
// Block = one wave = one task (bucket kB, wave index in the bucket) of the
// family's list in the device plan; the grid is an upper bound on the tasks,
// so it does not depend on the bucket histogram.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"

namespace crispy {

// Register-kernel families: bucket ranges sharing one occupancy target
// (3 VGPRs per band cell + ~64: 4 waves/SIMD up to kB 10, 3 up to 16, 2 above);
// kB 17..32 is split in two only to keep each translation unit's compile short.
struct RegFamily {
  int lo, hi;
};
constexpr RegFamily kRegFamilies[] = {{0, 10}, {11, 16}, {17, 24}, {25, kKbRegMax}};
constexpr int kNumRegFamilies = 4;
static_assert(kRegFamilies[0].lo == 0 && kRegFamilies[0].hi + 1 == kRegFamilies[1].lo &&
                  kRegFamilies[1].hi + 1 == kRegFamilies[2].lo &&
                  kRegFamilies[2].hi + 1 == kRegFamilies[3].lo && kRegFamilies[3].hi == kKbRegMax,
              "the register families cover kB 0..kKbRegMax without gaps");
// Lane-sliced families: G = ceil(W / C) lanes per pair, C band cells per lane,
// one family per slice width.  Which width a bucket runs at comes from
// slice_width_for().
constexpr int kNumSliceWidths = 2;
constexpr int kSliceWidths[kNumSliceWidths] = {24, 32};
// Packed families (nw_pk.hpp): G = pk_lanes lanes per pair, each two slices of
// pk_cells positions; one family per range of slice widths.  `cap` bounds the
// slice width (at most kPkMaxCells): small jobs take narrower slices, so that
// their few pairs spread over more lanes (pk_plan in nw.hip).
constexpr int kPkMaxCells = 40;   // 80 state registers: 3 waves per SIMD
constexpr int kPkMaxLanes = 16;   // lanes per pair
constexpr int kPkMaxKb = 639;     // 2 kB + 1 positions over kPkMaxLanes x 2 slices of kPkMaxCells
static_assert(2 * kPkMaxKb + 1 <= 2 * kPkMaxLanes * kPkMaxCells, "the widest band fits the lanes of a pair");
// The waves are set above what the widest slices' registers leave: the ACGT
// kernels spill 150, 135, 318 and 241 registers, those with upper code bits 85,
// 51, 185 and 7, mostly around the steps and not in them.  Measured over six
// calls: one wave more in every family 0 to 4 % slower (7e3 long reads and reads
// with N 4 %, 1,000 reads 3 %, 20,000 reads 1 %); one fewer, which spills less,
// 1.0 to 1.4 % faster with 1e3 to 2.5e5 ACGT reads and 8.5 % with long ones,
// 0.7 % slower with N.  So the ACGT column may drop by one; the cost model in
// nw.hip was fitted to the counts here and would have to follow.
struct PkFamily {
  int lo, hi;     // slice widths
  int waves;      // per SIMD, by registers
  int ext_waves;  // with the upper code bits
};
constexpr int kNumPkFamilies = 4;
constexpr PkFamily kPkFamilies[kNumPkFamilies] = {
    {1, 16, 5, 4}, {17, 24, 4, 3}, {25, 32, 4, 3}, {33, kPkMaxCells, 3, 2}};
constexpr int kFirstPkFamily = kNumRegFamilies + kNumSliceWidths;
constexpr int kNumFamilies = kFirstPkFamily + kNumPkFamilies;
constexpr int kPkBlockWaves = 4;  // waves (direction slots) per block, at most
constexpr int kPkTraceSteps = 8;  // steps of directions staged in LDS at a time by the trace

__host__ __device__ constexpr int pk_lanes(int kb, int cap) { return (2 * kb + 1 + 2 * cap - 1) / (2 * cap); }
__host__ __device__ constexpr int pk_cells(int kb, int cap) {
  return (2 * kb + 1 + 2 * pk_lanes(kb, cap) - 1) / (2 * pk_lanes(kb, cap));
}
// 32-bit words of directions per lane and step: 8 cells of both halves each
__host__ __device__ constexpr int pk_dir_words(int cells) { return (cells + 7) / 8; }
// The largest key of bucket kb with at most `rows` rows fits 16 bits (nw_pk.hpp:
// 9 per row from the -4 frame, 7 per position, a margin for the offers).
__host__ __device__ constexpr bool pk_keys_fit(int kb, int rows, int cap, int key_top = 0xFFFF) {
  return kb <= kPkMaxKb && pk_lanes(kb, cap) <= kPkMaxLanes &&
         9 * (rows + 1) + 7 * 2 * pk_lanes(kb, cap) * pk_cells(kb, cap) + 100 <= key_top >> 2;
}
constexpr int kPkF16Top = 0x7BFF;  // the largest finite half-precision pattern

// How a DP phase's buckets map to kernels: `forced` slice width of the sliced
// kernel (0 = cost model), kB up to pk_top run packed with slices of at most
// pk_cap cells (pk_top -1: none).
struct NwMap {
  int forced, pk_top, pk_cap;
};

__host__ __device__ constexpr int slice_lanes(int kb, int C) { return (2 * kb + 1 + C - 1) / C; }

// Cost model of one wave step of the sliced kernel: ~13.5 C VALU ops for the C
// cells of every lane plus ~45 per step (match words, neighbour exchange,
// window slide), shared by the 64 / G pairs of the wave.  Measured on MI355X
// the model holds for wide bands but not for G <= 6 lanes at 24 cells (kB up
// to ~71: 24 cells ran 3 % faster on kB 33..55 where the model favours 32), so
// the wider slice is taken only from 7 lanes up.  `forced` (24 or 32)
// overrides the choice.  Integer form (cost x 2, cross-multiplied), so the
// host and the device plan agree exactly.
__host__ __device__ inline int slice_width_for(int kb, int forced) {
  if (forced == 24 || forced == 32) return forced;
  const int g24 = slice_lanes(kb, 24), p24 = 64 / g24, p32 = 64 / slice_lanes(kb, 32);
  // c32 <= c24  <=>  (13.5*32 + 45) / p32 <= (13.5*24 + 45) / p24
  return g24 >= 7 && (27 * 32 + 90) * p24 <= (27 * 24 + 90) * p32 ? 32 : 24;
}

// Kernel family of bucket kB (kB <= kKbSliceMax).
__host__ __device__ inline int nw_family_of(int kb, const NwMap &m) {
  if (kb <= m.pk_top) {
    int f = 0;
    while (pk_cells(kb, m.pk_cap) > kPkFamilies[f].hi) ++f;
    return kFirstPkFamily + f;
  }
  if (kb > kKbRegMax) return kNumRegFamilies + (slice_width_for(kb, m.forced) == kSliceWidths[0] ? 0 : 1);
  int f = 0;
  while (kb > kRegFamilies[f].hi) ++f;
  return f;
}

// Pairs one wave task of bucket kB covers in family f.
__host__ __device__ inline int nw_pairs_per_wave(int kb, int f, int pk_cap) {
  if (f >= kFirstPkFamily) return 64 / pk_lanes(kb, pk_cap);
  return f >= kNumRegFamilies ? 64 / slice_lanes(kb, kSliceWidths[f - kNumRegFamilies]) : 64;
}

// Device plan of one DP phase, written by nw_plan_kernel from the bucket
// histogram.  btab[b] = (first position in `order`, pairs) of bucket b.  Per
// family f: its non-empty buckets in task order, list[f][k] = (bucket, first
// task), ntasks[f] tasks in all; the tasks of a family run its buckets by
// descending mean cells per pair and a bucket's waves from its longest pairs
// (the end of the R order) down, so the grid drains like a
// longest-processing-time schedule.
struct NwPlan {
  uint2 btab[kNumBuckets];
  uint2 list[kNumFamilies][kNumBuckets];
  uint32_t ntasks[kNumFamilies];
  uint32_t nbuckets[kNumFamilies];
  uint32_t next[kNumFamilies];  // packed families: tasks taken past the first one of each block
};

struct NwFusedArgs {
  const uint32_t *pack;
  const int64_t *poff;
  const int32_t *len;
  const int2 *pairs;
  const uint32_t *order;
  NwPlan *plan;
  float *out;
};
// A packed family's launch: one direction slot per wave, the slice width cap,
// and the read set's upper code bits (null when every read is ACGT only).
struct PkLaunchArgs {
  uint32_t *dirs;
  int64_t words;  // per slot
  int cap;
  unsigned block_waves;
  bool f16;  // every key of the family's buckets is at most kPkF16Top
  const uint32_t *pack_hi;
};

// Each launcher runs `blocks` one-wave blocks of its family, a packed one
// `slots` waves in blocks of k.block_waves.
void launch_nw_reg_family0(hipStream_t s, unsigned blocks, const NwFusedArgs &a);
void launch_nw_reg_family1(hipStream_t s, unsigned blocks, const NwFusedArgs &a);
void launch_nw_reg_family2(hipStream_t s, unsigned blocks, const NwFusedArgs &a);
void launch_nw_reg_family3(hipStream_t s, unsigned blocks, const NwFusedArgs &a);
void launch_nw_sliced_family24(hipStream_t s, unsigned blocks, const NwFusedArgs &a);
void launch_nw_sliced_family32(hipStream_t s, unsigned blocks, const NwFusedArgs &a);
void launch_nw_pk_family0(hipStream_t s, unsigned slots, const NwFusedArgs &a, const PkLaunchArgs &k);
void launch_nw_pk_family1(hipStream_t s, unsigned slots, const NwFusedArgs &a, const PkLaunchArgs &k);
void launch_nw_pk_family2(hipStream_t s, unsigned slots, const NwFusedArgs &a, const PkLaunchArgs &k);
void launch_nw_pk_family3(hipStream_t s, unsigned slots, const NwFusedArgs &a, const PkLaunchArgs &k);

}  // namespace crispy
