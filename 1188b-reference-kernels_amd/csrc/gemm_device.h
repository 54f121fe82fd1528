// Device building blocks shared by the grouped GEMM kernels (gfx950): LDS
// DMA through buffer resources, wait counters, barriers that the scheduler
// does not move, and instruction-group schedules.
#pragma once

#include "moe_common.h"

namespace moe {
namespace gemm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

constexpr int kBK = 64;  // reduction depth of one pipeline stage

// Loads of data that nothing writes while the kernel runs (group offsets, the
// lists an earlier kernel made): through the constant address space, so that a
// wave-uniform index becomes a scalar load. A vector load would sit in the
// wavefront's in-order vector-memory counter behind its LDS DMAs, and the wait
// for its value would wait for all of them.
typedef __attribute__((address_space(4))) const int32_t const_i32;
typedef __attribute__((address_space(4))) const int16_t const_i16;
__device__ __forceinline__ int32_t ld_inv(const int32_t *p, int64_t i) { return ((const const_i32 *)p)[i]; }
__device__ __forceinline__ int32_t ld_inv(const int16_t *p, int64_t i) { return ((const const_i16 *)p)[i]; }

// s_waitcnt immediates (gfx9 encoding: vmcnt [3:0],[15:14]; expcnt [6:4]; lgkmcnt [11:8]).
constexpr int kWaitVm0 = 0x0f70;    // vmcnt(0)
constexpr int kWaitLgkm0 = 0xc07f;  // lgkmcnt(0)

__device__ __forceinline__ void compiler_fence() { asm volatile("" ::: "memory"); }

// Workgroup barrier that neither the compiler nor the instruction scheduler
// moves any instruction across.
__device__ __forceinline__ void barrier() {
  compiler_fence();
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  compiler_fence();
}

// Waits for this thread's outstanding vector-memory (DMA, stores) or LDS operations.
__device__ __forceinline__ void wait_dma() {
  compiler_fence();
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
  compiler_fence();
}
__device__ __forceinline__ void wait_lds() {
  compiler_fence();
  __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
  compiler_fence();
}
// Waits until at most kN of this thread's vector-memory operations are
// outstanding (they complete in issue order).
template <int kN>
__device__ __forceinline__ void wait_vm_n() {
  static_assert(kN >= 0 && kN <= 63, "vmcnt range");
  compiler_fence();
  __builtin_amdgcn_s_waitcnt((kN & 0xf) | ((kN >> 4) << 14) | (0x7 << 4) | (0xf << 8));
  compiler_fence();
}

// Buffer resource over [base, base + bytes): raw buffer loads past `bytes`
// return zeros and stores past it are dropped, without touching memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
// Offset that lies past every resource this code builds (all stay below 2 GiB).
constexpr uint32_t kNoAccess = 0x80000000u;

// 16-byte buffer -> LDS copy: lane i writes bytes [16 i, 16 i + 16) of the 1 KiB
// block at `lds` (wave-uniform); the global address is rsrc base + voff + soff.
// kAux: cache policy bits (2: nt, a streaming load whose lines are not kept for reuse).
template <int kAux = 0>
__device__ __forceinline__ void dma16b(__amdgpu_buffer_rsrc_t rsrc, lds_void *lds, int voff, int soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds, 16, voff, soff, 0, kAux);
#else
  (void)rsrc; (void)lds; (void)voff; (void)soff;
#endif
}

// Instruction-group order spreading kReads LDS reads and kVmem vector-memory
// reads evenly behind kMfma MFMAs.
template <int kMfma, int kReads, int kVmem, int kR = 0>
__device__ __forceinline__ void sched_mix() {
  if constexpr (kR < kMfma) {
    constexpr int nr = kReads * (kR + 1) / kMfma - kReads * kR / kMfma;
    constexpr int nv = kVmem * (kR + 1) / kMfma - kVmem * kR / kMfma;
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if constexpr (nr > 0) __builtin_amdgcn_sched_group_barrier(0x100, nr, 0);
    if constexpr (nv > 0) __builtin_amdgcn_sched_group_barrier(0x020, nv, 0);
    sched_mix<kMfma, kReads, kVmem, kR + 1>();
  }
}

// Compute units of the current device (cached per device).
inline int num_cus() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cache[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev] = n;
  }
  return cache[dev];
}

// Tail list of the ping-pong kernels (workspace layout, ints): a group whose
// last 256-row tile would have 1 to 128 rows leaves that tile to the 128-row
// form of the kernel. tails_list lists those groups in order; after
// their 256-row tiles the persistent workgroups take (group, column tile)
// units u = 0, 1, ... of the list from the counter, unit u = list[u / ntiles],
// column tile u % ntiles.
constexpr int kTailCtr = 0;     // units handed out
constexpr int kTailCount = 32;  // groups in the list (own 128-byte line)
constexpr int kTailNone = 33;   // 1: another kernel has computed the whole GEMM
constexpr int kTailList = 64;   // the groups, ascending
#ifndef MOE_GEMM_TAILS_MIN_K
#define MOE_GEMM_TAILS_MIN_K 4096
#endif
constexpr int64_t kTailsMinK = MOE_GEMM_TAILS_MIN_K;  // shortest reduction that uses the 128-row tail tiles
inline size_t tails_bytes(int64_t G) { return sizeof(int) * static_cast<size_t>(kTailList + G); }
constexpr int kTailMaxRows = 128;  // longest tail of the list (the 128-row form's height)

__device__ __forceinline__ bool has_tail(int64_t m) {
  const int64_t r = m % 256;
  return r >= 1 && r <= kTailMaxRows;
}
// 256-row tiles of a group of m rows when its tail (if has_tail) is left to the list.
__device__ __forceinline__ int main_row_tiles(int m) { return (m + 255 - kTailMaxRows) / 256; }

// The list, by one wavefront: 64 neighbouring groups at a time, a lane each, ranked by a ballot; sixteen such sets are loaded
// before the first of them is ranked. Group g is rows offsets[g] .. offsets[g + 1] - 1, clamped to [0, M].
// Measured (MI355X, us for the launch of 64, 1024 and 4096 groups): 4.8, 4.8 and 7.4; a run of groups for each lane, walked
// twice: 4.8, 7.2 and 23.3, by 256 threads 4.8, 5.8 and 9.6.
__device__ __forceinline__ void tails_list(const int32_t *offsets, int64_t G, int64_t M, int *tails) {
  constexpr int kSets = 16;
  const int lane = lane_id(), n = static_cast<int>(G), rows = static_cast<int>(M);  // M < 2^31
  int pos = 0;
  for (int g0 = 0; g0 < n; g0 += kSets * kWave) {
    int lo[kSets], hi[kSets];
#pragma unroll
    for (int i = 0; i < kSets; ++i) {
      const int g = min(g0 + i * kWave + lane, n - 1);
      lo[i] = offsets[g];
      hi[i] = offsets[g + 1];
    }
#pragma unroll
    for (int i = 0; i < kSets; ++i) {
      const int g = g0 + i * kWave + lane;
      const int first = min(max(lo[i], 0), rows);
      const int m = g < n ? min(max(hi[i], first), rows) - first : 0;
      const uint64_t tail = __ballot(has_tail(m));
      if (has_tail(m)) tails[kTailList + pos + lanes_below(tail)] = g;
      pos += __popcll(tail);
    }
  }
  if (lane == 0) {
    tails[kTailCount] = pos;
    tails[kTailNone] = 0;
    tails[kTailCtr] = 0;
  }
}

// The list of a GEMM that needs no ping-pong kernel (one thread).
__device__ __forceinline__ void no_tails(int *tails) {
  tails[kTailCount] = 0;
  tails[kTailNone] = 1;
  tails[kTailCtr] = 0;
}

// The list in a launch of its own, before a ping-pong kernel (grouped_gemm.hip).
void launch_tails_init(const int32_t *offsets, int64_t G, int64_t M, int *tails, hipStream_t s);

}  // namespace gemm
}  // namespace moe
