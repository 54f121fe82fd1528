// Per-row router top-k on one wavefront (shared by the stand-alone top-k
// kernel and the router GEMM's fused epilogue).
//
// Math: kernel_cases/case23_ref_aten_topk.py:47-62 -- values/indices are the
// first k entries of a stable descending sort of each row (torch.topk with
// largest=True, sorted=True): larger value first, equal values by smaller
// index, NaN above every number, -0.0 equal to +0.0.  The mask is
// zeros(T,E,bool).scatter_(1, idx, True) (case18...py:86-88) and the merge
// probs are softmax over the k selected values (fp32), scattered to [T, E].
//
// Lane l holds elements l, l+64, ... (kEPL per lane) as 32-bit order keys,
// sorted once (odd-even transposition: only neighbours trade places, so equal
// keys stay in slot order; up to 8 elements). Each of the k rounds takes the wave-wide maximum of
// the lanes' first keys (DPP row operations, no LDS crossbar); a ballot names
// the lane that holds it, whose list moves up by one. Where several lanes hold
// it, the smallest index among their first slots wins (a DPP minimum), so ties
// go to the smaller index. Lane j keeps round j's winner, so lanes < k store
// values/indices coalesced.
// What bounds it is the chain of a round, not the bytes; 16384 rows, k = 8, us, with
// the index always found by a second DPP chain and the winner's list searched
// again every round, and with this form: 320 experts 29.5 and 19.3 (8 slots a lane
// before, 5 now), 160 21.6 and 14.4, 64 10.6 and 9.7. Above 8 slots the sort costs
// more than the searches (1024 experts: 58 against 50), so the list stays unsorted; so it does above 5 for one or two
// selected of many rows (topk_searches).
#pragma once

#include "moe_common.h"

namespace moe {

// Order key: a > b as floats (with NaN largest, -0 == +0) iff key(a) > key(b).
__device__ __forceinline__ uint32_t order_key(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0xffffffffu;  // any NaN
  if ((u & 0x7fffffffu) == 0u) u = 0u;                        // -0 -> +0
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Wave-wide maximum / minimum of a 32-bit value, valid in lane 63: quad
// permutes (xor 1, xor 2), half-row and row mirrors (8, 16 lanes), then row
// broadcasts of lanes 15 and 31 (rows 0+1, 2+3, all four). Lanes a step does
// not write keep their value, so each step combines disjoint lane sets.
template <bool kMax>
__device__ __forceinline__ uint32_t wave_reduce_u32(uint32_t v) {
  auto comb = [](uint32_t a, uint32_t b) { return kMax ? (a > b ? a : b) : (a < b ? a : b); };
  const int iv = static_cast<int>(v);
  v = comb(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(iv, iv, 0xB1, 0xF, 0xF, false)));  // quad_perm 1,0,3,2
  int jv = static_cast<int>(v);
  v = comb(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(jv, jv, 0x4E, 0xF, 0xF, false)));  // quad_perm 2,3,0,1
  jv = static_cast<int>(v);
  v = comb(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(jv, jv, 0x141, 0xF, 0xF, false)));  // row_half_mirror
  jv = static_cast<int>(v);
  v = comb(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(jv, jv, 0x140, 0xF, 0xF, false)));  // row_mirror
  jv = static_cast<int>(v);
  v = comb(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(jv, jv, 0x142, 0xA, 0xF, false)));  // row_bcast:15
  jv = static_cast<int>(v);
  v = comb(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(jv, jv, 0x143, 0xC, 0xF, false)));  // row_bcast:31
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// One DPP step of a sum: v + the source lane's v (lanes the step does not
// write add 0: bound_ctrl with old = 0).
template <int kCtrl, int kRowMask>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, kRowMask, 0xF, true));
}

// Wave-wide fp32 sum by the same DPP steps (a fixed order), valid in every lane.
__device__ __forceinline__ float wave_sum_f32(float x) {
  float v = dpp_add<0xB1, 0xF>(x);
  v = dpp_add<0x4E, 0xF>(v);
  v = dpp_add<0x141, 0xF>(v);
  v = dpp_add<0x140, 0xF>(v);
  v = dpp_add<0x142, 0xA>(v);
  v = dpp_add<0x143, 0xC>(v);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Whether lists of 6 to 8 elements are searched every round instead of sorted once: for one or two rounds where the rows
// fill the chip. us, sorted and searched: 16384 rows of 512, k = 1 12.4 and 9.9, k = 2 13.1 and 10.9; 32768 of 448, k = 1
// 21.4 and 18.0; 2048 of 512, k = 2 4.3 and 4.0; but 93 of 512, k = 2 3.8 and 4.0, k = 4 4.3 and 5.0; 16384 of 320, k = 4
// 8.7 and 8.9.
inline bool topk_searches(int64_t rows, int64_t k) { return k <= 2 && rows >= 1024; }

// Top-k of row t (elements load(e), e < E) by the calling wavefront; writes
// values/indices [T, k] and, when non-null, routing_map [T, E] and probs [T, E].
template <int kEPL, bool kSorted = (kEPL <= 8), typename Load>
__device__ __forceinline__ void topk_row(Load load, int64_t t, int E, int k, float *values, int64_t *indices,
                                         uint8_t *routing_map, float *probs) {
  const int lane = lane_id();
  float val[kEPL];
  uint32_t key[kEPL], slot[kEPL];  // key 0 = nothing left (every float's order key is above 0)
#pragma unroll
  for (int s = 0; s < kEPL; ++s) {
    const int e = s * kWave + lane;
    val[s] = 0.0f;
    key[s] = 0u;
    slot[s] = s;
    if (e < E) {
      val[s] = load(e);
      key[s] = order_key(val[s]);
    }
  }
  if constexpr (kSorted) {
#pragma unroll
    for (int r = 0; r < kEPL; ++r) {
#pragma unroll
      for (int s = r % 2; s + 1 < kEPL; s += 2) {
        const bool up = key[s + 1] > key[s];
        const uint32_t ka = key[s], kb = key[s + 1], sa = slot[s], sb = slot[s + 1];
        key[s] = up ? kb : ka;
        key[s + 1] = up ? ka : kb;
        slot[s] = up ? sb : sa;
        slot[s + 1] = up ? sa : sb;
      }
    }
  }
  // The lane's first: its largest key, the smaller slot on equal keys.
  uint32_t first_key, first_slot;
  auto first = [&]() {
    first_key = key[0];
    first_slot = slot[0];
    if constexpr (!kSorted) {
#pragma unroll
      for (int s = 1; s < kEPL; ++s) {
        const bool up = key[s] > first_key;
        first_key = up ? key[s] : first_key;
        first_slot = up ? s : first_slot;
      }
    }
  };
  first();

  uint32_t chosen = 0;  // bit s: element lane + 64 s selected
  int my_idx = 0;
  for (int j = 0; j < k; ++j) {
    const uint32_t kmax = wave_reduce_u32<true>(first_key);
    const uint64_t holders = __ballot(first_key == kmax);
    int widx, wlane = __builtin_ctzll(holders);
    if (kEPL == 1) {
      widx = wlane;
    } else if ((holders & (holders - 1)) == 0) {
      widx = __builtin_amdgcn_readlane(static_cast<int>(first_slot), wlane) * kWave + wlane;
    } else {
      widx = static_cast<int>(wave_reduce_u32<false>(first_key == kmax ? first_slot * kWave + lane : 0xffffffffu));
      wlane = widx % kWave;
    }
    if (lane == wlane) {
      chosen |= 1u << first_slot;
      if constexpr (kSorted) {
#pragma unroll
        for (int s = 0; s + 1 < kEPL; ++s) {
          key[s] = key[s + 1];
          slot[s] = slot[s + 1];
        }
        key[kEPL - 1] = 0u;
      } else {
#pragma unroll
        for (int s = 0; s < kEPL; ++s) key[s] = s == static_cast<int>(first_slot) ? 0u : key[s];
      }
      first();
    }
    if (lane == j) my_idx = widx;
  }
  const float my_val = lane < k ? load(my_idx) : 0.0f;  // (the key does not hold -0 or a NaN's bits)
  if (lane < k) {
    values[t * k + lane] = my_val;
    indices[t * k + lane] = my_idx;
  }

  if (routing_map != nullptr || probs != nullptr) {
    float inv_sum = 0.0f, vmax = 0.0f;
    if (probs != nullptr) {
      vmax = readlane_f32(my_val, 0);
      const float ex = lane < k ? expf(my_val - vmax) : 0.0f;
      inv_sum = wave_sum_f32(ex);
    }
#pragma unroll
    for (int s = 0; s < kEPL; ++s) {
      const int e = s * kWave + lane;
      if (e < E) {
        const bool c = (chosen >> s) & 1u;
        if (routing_map != nullptr) routing_map[t * E + e] = c ? 1 : 0;
        if (probs != nullptr) probs[t * E + e] = c ? expf(val[s] - vmax) / inv_sum : 0.0f;
      }
    }
  }
}

}  // namespace moe
