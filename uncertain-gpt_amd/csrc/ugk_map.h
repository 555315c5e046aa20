// ugk_map.h - the streaming map shared by the elementwise kernels.
//
// An operator maps kLoads input floats of element i to kStores output floats.
// Each thread owns Op::kUnroll float4 (16-byte) slots strided by the
// workgroup size, so every load and store instruction of a wavefront covers
// one contiguous 1 KiB span, all of a thread's loads are issued before its
// first arithmetic instruction, and every access is non-temporal (each byte
// is touched once). Launch-shape sweeps on MI355X over inputs too large for
// the last-level cache (unroll 1-8, 256-1024 threads, flat or grid-stride,
// with and without nt) put nt loads and stores with unroll 1-2 and 256-512
// threads on top; each operator picks its own (the spread is a few percent).
//
// Any n takes this path, in one launch, and any address beyond kEachTo
// elements. gfx950 accepts a
// 16-byte access at a 4-byte address, so the slots start at the first element
// whose address in the first output is a cache line's (full lines are then
// written there whatever the streams' offsets: 478 against 482 us for a whole
// block of layer kernels whose arrays are 8 bytes off, with the slots started at
// element 0 instead), and the up to 31 elements before them and 3 after them
// are taken one by one by a workgroup of their own, told from the others by a
// scalar compare. Against dwords for misaligned arrays: residual forward over
// 11.1M elements 23.0 against 31.6 us, its backward 37.4 against 45.1; against a
// second launch for a ragged end: 4.4-4.8 us less per call (six such calls over
// 11,061,531 parameters: 281 against 268 us).
//
// Few elements at a misaligned address go one to a thread instead (k_map_each):
// the chip is not filled then, and a thread with four elements takes longer.
// The operators whose element is long notice (98,305 elements 8 bytes off:
// AdamW 3.5 against 5.0 us, materialize 3.1 against 4.4), the others don't
// either way. Where the two meet is the operator's kEachTo, 1,000,000 elements
// at most (AdamW 6.1 against 5.7 us at 600,000, materialize 4.8 against 5.5) but for
// the one-pass update: fifteen misaligned streams of 16-byte accesses from
// element 0 on are slower at any size (40M elements 543 against 524 us).
//
// An operator is a struct with
//   kLoads, kStores          stream counts;
//   kTable                   stage expf's 2^(i/32) table in LDS (tab != null);
//   kUnroll, kThreads        float4 slots per thread, threads per workgroup;
//   kLdsReserve              bytes of LDS each workgroup reserves without
//                            using them (0: none), which caps the workgroups
//                            resident on a CU (160 KiB of LDS each);
//   Params                   per-launch scalars passed by value;
//   kIndexed                 whether apply reads i: the slots then start at
//                            element 0 (their indexes need no 64-bit add per
//                            element, which the ops that draw eps are short of
//                            the cycles for);
//   apply(ld, st, tab, i, p) the per-element body; i is the element index;
//   kEachTo                  up to how many elements misaligned arrays take one
//                            thread per element;
//   kPre, Pre, pre(i, p)     optionally (kPre true), the part of the body that
//                            reads no stream (a Philox draw): the kernel
//                            computes it for all of a thread's elements while
//                            their loads are in flight and hands it to
//                            apply_pre(ld, st, tab, i, p, pre) instead.
#pragma once

#include "ugk_internal.h"
#include "ugk_libm_dev.h"

namespace ugk {
namespace {

struct MapOp {
  struct Params {};
  static constexpr bool kTable = false;
  static constexpr int kUnroll = 2;
  static constexpr int kThreads = kBlock;
  static constexpr unsigned kLdsReserve = 0;
  static constexpr bool kIndexed = false;
  static constexpr size_t kEachTo = (size_t)1 << 19;
  static constexpr bool kPre = false;
  struct Pre {};
};

template <class Op>
struct Streams {
  const float *ld[Op::kLoads];
  float *st[Op::kStores];
  typename Op::Params p;
};

constexpr unsigned kLine = 32;  // floats of a cache line

// Element i of the pointers alone (before them, where i is negative).
template <class Op>
__device__ __forceinline__ void map_one(const Streams<Op> &s, ptrdiff_t i, const uint64_t *tab) {
  float in[Op::kLoads], out[Op::kStores];
#pragma unroll
  for (int l = 0; l < Op::kLoads; l++) in[l] = s.ld[l][i];
  if constexpr (Op::kPre)
    Op::apply_pre(in, out, tab, i, s.p, Op::pre(i, s.p));
  else
    Op::apply(in, out, tab, i, s.p);
#pragma unroll
  for (int o = 0; o < Op::kStores; o++) s.st[o][i] = out[o];
}

// Float4 slots [0, n4) from the pointers on; the `rest` elements around them,
// the first `lead` of those before the pointers, by workgroup `full`.
template <class Op>
__global__ __launch_bounds__(Op::kThreads) void k_map_vec4(Streams<Op> s, size_t n4, unsigned full, unsigned lead, unsigned rest) {
  __shared__ uint64_t tab[Op::kTable ? 32 : 1];
  if (Op::kTable) {
    ugk_exp2_stage(tab);
    __syncthreads();
  }
  constexpr int kU = Op::kUnroll, kT = Op::kThreads;
  if (blockIdx.x == full) {  // the workgroup past the float4 slots: the elements around them
    for (unsigned k = threadIdx.x; k < rest; k += kT)
      map_one<Op>(s, (ptrdiff_t)k - (ptrdiff_t)lead + (ptrdiff_t)(k < lead ? 0 : 4 * n4), tab);
    return;
  }
  const size_t base = (size_t)blockIdx.x * (kT * kU) + threadIdx.x;
  float4 v[kU][Op::kLoads];
#pragma unroll
  for (int u = 0; u < kU; u++) {
    const size_t i = base + (size_t)u * kT;
    if (i < n4) {
#pragma unroll
      for (int l = 0; l < Op::kLoads; l++) v[u][l] = ld_nt4(s.ld[l] + 4 * i);
    }
  }
  typename Op::Pre pre[kU][4];
  if constexpr (Op::kPre) {
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const size_t i = base + (size_t)u * kT;
      if (i < n4) {
#pragma unroll
        for (int e = 0; e < 4; e++) pre[u][e] = Op::pre(4 * i + e, s.p);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < kU; u++) {
    const size_t i = base + (size_t)u * kT;
    if (i < n4) {
      float in[4][Op::kLoads], out[4][Op::kStores];
#pragma unroll
      for (int l = 0; l < Op::kLoads; l++) {
        in[0][l] = v[u][l].x; in[1][l] = v[u][l].y;
        in[2][l] = v[u][l].z; in[3][l] = v[u][l].w;
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if constexpr (Op::kPre)
          Op::apply_pre(in[e], out[e], tab, 4 * i + e, s.p, pre[u][e]);
        else
          Op::apply(in[e], out[e], tab, 4 * i + e, s.p);
      }
#pragma unroll
      for (int o = 0; o < Op::kStores; o++)
        st_nt4(s.st[o] + 4 * i, make_float4(out[0][o], out[1][o], out[2][o], out[3][o]));
    }
  }
}

// One element per thread (and more where that would take over kEachBlocks workgroups).
constexpr unsigned kEachBlocks = 65536;
template <class Op>
__global__ __launch_bounds__(kBlock) void k_map_each(Streams<Op> s, size_t n) {
  __shared__ uint64_t tab[Op::kTable ? 32 : 1];
  if (Op::kTable) {
    ugk_exp2_stage(tab);
    __syncthreads();
  }
  for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
    map_one<Op>(s, (ptrdiff_t)i, tab);
}

template <class Op>
int run_map(Streams<Op> s, size_t n, const char *name) {
  if (n == 0) return 0;
  if (n <= Op::kEachTo) {
    bool aligned = true;
    for (int l = 0; l < Op::kLoads; l++) aligned = aligned && aligned16(s.ld[l]);
    for (int o = 0; o < Op::kStores; o++) aligned = aligned && aligned16(s.st[o]);
    if (!aligned) {
      const size_t blocks = (n - 1) / kBlock + 1;
      launch(k_map_each<Op>, dim3(blocks < kEachBlocks ? (unsigned)blocks : kEachBlocks), dim3(kBlock), 0, s, n);
      return check_launch(name);
    }
  }
  size_t lead = Op::kIndexed ? 0 : (0 - ((uintptr_t)s.st[0] >> 2)) & (kLine - 1);
  if (lead > n) lead = n;
  for (int l = 0; l < Op::kLoads; l++) s.ld[l] += lead;
  for (int o = 0; o < Op::kStores; o++) s.st[o] += lead;
  const size_t n4 = (n - lead) / 4;
  const unsigned full = grid_for(n4, (size_t)Op::kThreads * Op::kUnroll);
  launch(k_map_vec4<Op>, dim3(full + (n != 4 * n4 ? 1 : 0)), dim3(Op::kThreads), Op::kLdsReserve, s, n4, full,
         (unsigned)lead, (unsigned)(n - 4 * n4));
  return check_launch(name);
}

}  // namespace
}  // namespace ugk
