// tf32 operands of the router backward GEMMs as scaled fp16 values.
//
// A tf32 value has 11 significant bits, as many as fp16. Scaled by a power of
// two 2^e that brings the largest magnitude of its row or column near the top of
// fp16's range, every tf32-rounded value of it is an fp16 value, exactly unless
// it lies some 2^25 or more below that largest one (it then rounds to an fp16
// subnormal). The product of two fp16 values is exact in fp32, so one fp16 MFMA
// takes the place of a tf32 product, and the fp32 sums are scaled back by the
// two exponents (exact). The scale comes from the largest finite magnitude
// (Inf and NaN entries stay Inf and NaN when scaled, so every finite value still
// converts exactly).
#pragma once

#include "moe_common.h"

namespace moe {

// kernel_cases/case39_ref_musa_asm_tf32_ssgemm_nn_384x256.py:51-58 (round_tf32_rne): nearest even of the 13 dropped bits.
__device__ __forceinline__ uint32_t tf32_rne_bits(uint32_t b) { return (b + 0xFFFu + ((b >> 13) & 1u)) & 0xFFFFE000u; }
__device__ __forceinline__ float finite_abs(float x) {
  const float a = fabsf(x);
  return a < __builtin_huge_valf() ? a : 0.f;  // Inf and NaN -> 0
}
// Exponent that brings a largest magnitude mx into [2^14, 2^15); 0 if there is no finite nonzero value.
__device__ __forceinline__ int scale_exp(float mx) {
  if (!(mx > 0.f) || !(mx < __builtin_huge_valf())) return 0;
  int e = 0;
  (void)__builtin_frexpf(mx, &e);  // mx = f 2^e, f in [0.5, 1)
  return 15 - e;                   // mx 2^(15 - e) in [2^14, 2^15)
}

// ---- router wgrad (router_wgrad.hip)

// The work: ceil(K / 256) column tiles x row tiles of 16 mi rows x s reduction chunks of c rows (a multiple of 64).
struct RouterWgradPlan {
  int mi;
  bool wide;  // 64-bit addresses
  int64_t row_tiles, s, c;
};
// most_chunks (>= 1): for how many there is room.
RouterWgradPlan router_wgrad_plan(int64_t M, int64_t N, int64_t K, int64_t most_chunks);

// grad_output [M, N] fp32 -> its transpose in fp16, [N, M8] (M8 = M rounded up to 8, zeros past M), each row scaled by
// 2^exp[n]; exp[n] from the column maxima of `slabs` slabs (part [slabs, N]).
void launch_router_wgrad_rows(const float *grad_output, int64_t M, int64_t N, const float *part, int slabs, uint16_t *rows, int32_t *exp,
                              hipStream_t s);
// planes[chunk][N][K], scaled by exp and col_exp[chunk][K], then their sum in chunk order, scaled back (s == 1: the result
// itself, neither is used).
void launch_router_wgrad(const RouterWgradPlan &pl, const uint16_t *rows, const int32_t *exp, const float *inp, int64_t M, int64_t N,
                         int64_t K, float *planes, int32_t *col_exp, float *out, hipStream_t s);

// ---- router dgrad (router_dgrad.hip): reductions of at most 320

bool router_dgrad_applies(int64_t K);
struct RouterDgradLayout {  // workspace, byte offsets
  size_t a = 0, b = 0, a_exp = 0, b_exp = 0, total = 0;
};
RouterDgradLayout router_dgrad_layout(int64_t M, int64_t K, int64_t N);
void launch_router_dgrad(const float *go, int64_t M, int64_t K, const float *w, int64_t N, float *out, void *workspace, hipStream_t s);

}  // namespace moe
