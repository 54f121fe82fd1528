// Grouped GEMM forward for short groups: a stream of the weights.
//
// With a few rows per expert (a decode step) a weight element is used for a
// handful of rows and the time is that of reading the active experts' weights
// once: 6.9-7.1 TB/s is what non-temporal LDS DMA of 128-byte row pieces reaches
// here (5.8-6.6 where the rows are 4, 8 or 16 KiB apart). What it takes is bytes in flight,
// i.e. LDS for the weight ring, and no time lost between tiles:
//   * 8 wavefronts, on each SIMD one computing and one loading, as in
//     grouped_gemm_fwd128_kernel: two DMA the tile's rows into one ring of
//     64-deep stages, two the weight rows into another, each with its own
//     lookahead; one barrier per stage; a workgroup's tiles form one stream;
//   * a group's last row tile runs in the lowest of three heights (32, 64, 128)
//     that holds it, so its rows take no more LDS than they need: 8 weight stages
//     of 16 KiB at 32 and 64 rows (6 at 128), where 128-row tiles throughout left
//     4. 16-wide blocks, v_mfma_f32_16x16x32_bf16, K ascending from zero: each
//     output element is the ping-pong kernel's MFMA sequence, bit for bit;
//   * the columns are cut so that the units fill whole rounds of the workgroups
//     (struct Plan), counted on the device from the groups that have rows;
//   * the groups are looked up by the lanes (one group each, a scan, a ballot)
//     and not by a loop over the offsets: that loop, 64 groups of dependent
//     scalar loads per walk, cost 25 us per call.
// Measured (MI355X, 64 experts, fc1: K 7168, 2 x 2048 columns, SwiGLU, gathered; fc2: K 2048, 7168 columns; us per
// call, before: the ping-pong kernel's tail tiles / grouped_gemm_fwd128_kernel), top-8 of 1, 8, 32, 93 and 256 tokens
// with skewed routing: fc1 122 -> 71, 278 -> 203 (5.1 -> 6.9 TB/s), 418 -> 322, 457 -> 399, 475 -> 465; fc2 61 -> 51,
// 149 -> 123 (4.7 -> 5.7 TB/s: rows 4 KiB apart), 201 -> 183, 241 -> 220, 279 -> 262. What is left above the read
// rate grows with the rows: the stores of the output (60 rows per group: 290 us, 240 without them) and the row tiles
// that read a group's weights a second time.
#include <algorithm>
#include <type_traits>

#include "grouped_gemm.h"

namespace moe {
namespace {

using namespace gemm;

constexpr int kBRows = 128;                      // weight rows of a tile (SwiGLU: 64 gate and 64 up rows)
constexpr int kBStage = kBRows * kRowBytes;      // 16 KiB
constexpr int kLds = 160 * 1024;

// Rows of a tile of each class, ring stages of the rows and of the weights.
template <int kTM>
struct Ring {
  static constexpr int kAStage = kTM * kRowBytes;
  static constexpr int kSA = kTM == 32 ? 7 : 4;
  static constexpr int kSB = kTM == 128 ? 6 : 8;
  static_assert(kSA * kAStage + kSB * kBStage <= kLds, "LDS budget");
};

// Row tiles of a group of m rows: whole tiles of 128 rows, then one of the rest, in the lowest class that holds it.
template <int kTM>
__device__ __forceinline__ int class_tiles(int m) {
  const int rest = m % 128;
  if constexpr (kTM == 128) return m / 128 + (rest > 64 ? 1 : 0);
  if constexpr (kTM == 64) return rest > 32 && rest <= 64 ? 1 : 0;
  return rest > 0 && rest <= 32 ? 1 : 0;
}

struct Roles {
  int lane, simd, loader;  // loader: 0 computes, 1 loads
};

// How the work is cut into units of one row tile x some 16-column slabs. The row tiles (class by class, group by
// group) share `units` units evenly: those before row tile i are i * units / row_tiles, so the units fill whole
// rounds of the workgroups and differ by at most one slab where a group's columns do not divide.
struct Plan {
  int row_tiles, units, c16;  // c16: 16-column slabs of the output
  // i * units / row_tiles: the product is exact in a double, and a quotient below 2^31 that is no whole number is
  // further from the next one than the division rounds.
  __device__ __forceinline__ int before(int i) const {
    return static_cast<int>(static_cast<double>(i) * static_cast<double>(units) / static_cast<double>(row_tiles));
  }
};

// Rows of group `g`, as every lane's own group.
struct Rows {
  int lo, m;
};
__device__ __forceinline__ Rows group_rows(const GemmArgs &p, int g) {
  const int m32 = static_cast<int>(p.M);
  const int gc = min(g, static_cast<int>(p.G) - 1);
  const int lo = min(max(p.offsets[gc], 0), m32);
  const int hi = min(max(p.offsets[gc + 1], lo), m32);
  return {lo, g < static_cast<int>(p.G) ? hi - lo : 0};
}

// Row tiles of one class: `first` (group rows of the lane's own group of the first 64) and `tile0`, the row tiles
// of the classes before.
template <int kTM, bool kSwiglu, bool kGather>
__device__ __forceinline__ void run_class(const GemmArgs &p, const Plan &plan, const Roles &role, uint32_t lds, Rows first, int tile0) {
  using R = Ring<kTM>;
  constexpr int kSA = R::kSA, kSB = R::kSB;
  constexpr int kDmaA = R::kAStage / 1024 / 2, kDmaB = kBStage / 1024 / 2;  // per loading wavefront
  static_assert((kSA - 1) * kDmaA <= 63 && (kSB - 1) * kDmaB <= 63, "vmcnt range");
  constexpr int kWR = kTM == 128 ? 2 : 1, kWC = 4 / kWR;  // computing wavefronts: rows x columns
  constexpr int kMI = kTM / kWR / 16, kNI = kBRows / kWC / 16;
  const uint32_t a_lds = lds, b_lds = lds + kSA * R::kAStage;
  const int lane = role.lane;
  const int64_t K = p.K, N = p.N;
  const int ktiles = static_cast<int>(K / kBK);
  const uint32_t row_bytes = static_cast<uint32_t>(K) * 2u;

  struct Tile {
    int g, i0, rows, col0, cols;  // columns [col0, col0 + cols) of the output, in 16s
  };
  // ---- unit walker (every wavefront walks the same units). Each lane holds one group of the current 64: its rows,
  // its row tiles and the units they share; a unit's group is the first lane whose units end past it.
  int gb = 0;
  Rows v = first;
  int v_mt, v_us, v_ue, tiles_end = tile0;
  auto scan = [&]() {
    v_mt = class_tiles<kTM>(v.m);
    int s = v_mt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(s, d);
      s += lane >= d ? o : 0;
    }
    v_us = plan.before(tiles_end + s - v_mt);
    v_ue = plan.before(tiles_end + s);
    tiles_end += __builtin_amdgcn_readlane(s, 63);
  };
  scan();
  const int P = static_cast<int>(gridDim.x), b = static_cast<int>(blockIdx.x);
  const int r0 = (b % 8) * (P / 8) + b / 8;  // an XCD takes neighbouring units: a group's rows come from its L2
  // this workgroup's units: r0 + i P, of this class those from its first one on
  const int u0 = plan.before(tile0);
  int L = (r0 >= u0 ? r0 : r0 + (u0 - r0 + P - 1) / P * P) - P;
  auto find = [&](Tile &t) -> bool {
    L += P;
    uint64_t hit;
    while ((hit = __ballot(L < v_ue)) == 0) {
      gb += 64;
      if (gb >= static_cast<int>(p.G)) return false;
      v = group_rows(p, gb + lane);
      scan();
    }
    const int src = __builtin_ctzll(hit);
    const int lo = __builtin_amdgcn_readlane(v.lo, src), m = __builtin_amdgcn_readlane(v.m, src);
    const int mt_g = __builtin_amdgcn_readlane(v_mt, src), us = __builtin_amdgcn_readlane(v_us, src);
    const int n = __builtin_amdgcn_readlane(v_ue, src) - us, q = L - us;
    // row tile fastest: the row tiles of about the same columns are neighbours, and the second reads the weights from L2
    const int j = q / mt_g, mt = q - j * mt_g;
    const int slabs = (n - mt + mt_g - 1) / mt_g;  // units of this row tile
    t.g = gb + src;
    t.i0 = kTM == 128 ? lo + mt * 128 : lo + m - m % 128;
    t.rows = min(kTM, lo + m - t.i0);
    t.col0 = static_cast<int>(static_cast<uint32_t>(j) * static_cast<uint32_t>(plan.c16) / static_cast<uint32_t>(slabs));
    t.cols = static_cast<int>(static_cast<uint32_t>(j + 1) * static_cast<uint32_t>(plan.c16) / static_cast<uint32_t>(slabs)) - t.col0;
    return true;
  };

  Tile t;
  if (!find(t)) return;

  if (role.loader) {
    const bool is_a = role.simd < 2;
    const int li = role.simd & 1;
    int ln = lane;
    asm volatile("" : "+v"(ln));
    auto run = [&](auto is_a_c) {
      constexpr bool kA = decltype(is_a_c)::value;
      constexpr bool kIdx = kA && kGather;
      constexpr int kS = kA ? kSA : kSB;
      constexpr int kN = kA ? kDmaA : kDmaB;
      constexpr int kSlot = kA ? R::kAStage : kBStage;
      const uint32_t ring = (kA ? a_lds : b_lds) + li * kN * 1024;
      const int r_0 = li * kN * 8 + (ln >> 3);  // row of this wavefront's 1 KiB block j (8 rows): r_0 + 8 j
      int off[kN];
      int32_t idx[kIdx ? kN : 1];
      // Source rows of a tile's rows (gather); rows past the tile's read the last one and are not loaded.
      auto load_idx = [&](const Tile &u) {
        if constexpr (kIdx) {
#pragma unroll
          for (int j = 0; j < kN; ++j) idx[j] = p.a_rows[u.i0 + min(r_0 + j * 8, u.rows - 1)];
        }
      };
      auto set_idx = [&](const Tile &u) {
        if constexpr (kIdx) {
          const int src_rows = static_cast<int>(min(p.a_src_rows, int64_t(0x7fffffff)));
#pragma unroll
          for (int j = 0; j < kN; ++j) {
            const int r = r_0 + j * 8;
            off[j] = r < u.rows && idx[j] >= 0 && idx[j] < src_rows
                         ? static_cast<int>(static_cast<uint32_t>(idx[j]) * row_bytes + static_cast<uint32_t>(((ln & 7) ^ swz(r)) << 4))
                         : static_cast<int>(kNoAccess);
          }
        }
      };
      // Offsets of the tile's rows: A rows in order, weight rows of the tile's columns (others: none).
      auto set_off = [&](const Tile &u) {
#pragma unroll
        for (int j = 0; j < kN; ++j) {
          const int r = r_0 + j * 8;
          uint32_t o = static_cast<uint32_t>(r);
          bool in = true;
          if constexpr (!kA) {
            int c = r;
            if constexpr (kSwiglu) {
              // a computing wavefront's 16 kNI rows: gate rows, then the up rows of the same columns
              const int wc = r / (16 * kNI), q = r % (16 * kNI);
              c = wc * (8 * kNI) + q % (8 * kNI);
              o = static_cast<uint32_t>(c) + (q >= 8 * kNI ? static_cast<uint32_t>(p.ncols) : 0u);
            }
            in = c < u.cols * 16;
          }
          off[j] = static_cast<int>(in ? o * row_bytes + static_cast<uint32_t>(((ln & 7) ^ swz(r)) << 4) : kNoAccess);
        }
      };
      auto rsrc = [&](const Tile &u) {
        if constexpr (kA) {
          // Rows past the tile's lie past the resource (gather: have no offset): zeros.
          return kGather ? make_rsrc(p.a, static_cast<uint32_t>(p.a_src_rows) * row_bytes)
                         : make_rsrc(p.a + static_cast<int64_t>(u.i0) * K, static_cast<uint32_t>(u.rows) * row_bytes);
        } else {
          // From the tile's first column to the end of the expert's weights; a gate column past ncols reads an
          // up row and its up row zeros, and its result is dropped.
          const int64_t n0 = static_cast<int64_t>(u.col0) * 16;
          return make_rsrc(p.w + (static_cast<int64_t>(u.g) * N + n0) * K, static_cast<uint32_t>(N - n0) * row_bytes);
        }
      };
      // The stages of this workgroup's tiles form one stream (tile by tile, K ascending), so the rings run on
      // from one tile into the next; past the last one the last stage is loaded again (the same number of
      // loads in flight in every step), into slots nothing reads any more.
      __amdgpu_buffer_rsrc_t rs = rsrc(t);
      set_off(t);
      load_idx(t);
      set_idx(t);
      Tile nx{};
      bool more = find(nx);
      if (more) load_idx(nx);
      int kt = 0;
      int64_t issued = 0, end = INT64_MAX;
      bool last = false;  // the last tile's last stage has been issued
      auto one = [&](int slot) {
        const int k = last ? ktiles - 1 : kt;
        const uint32_t dst = ring + slot * kSlot;
#pragma unroll
        for (int j = 0; j < kN; ++j) dma16b<kA ? 0 : 2>(rs, (lds_void *)(uintptr_t)(dst + j * 1024), off[j], k * kBK * 2);
        ++issued;
        if (!last && ++kt == ktiles) {
          kt = 0;
          if (more) {
            t = nx;
            rs = rsrc(t);
            if constexpr (!kA) set_off(t);
            set_idx(t);
            more = find(nx);
            if (more) load_idx(nx);
          } else {
            last = true;
            end = issued;
          }
        }
      };
      for (int st = 0; st < kS - 1; ++st) one(st);
      wait_vm_n<(kS - 2) * kN>();  // stage 0 has landed
      barrier();
      int slot = kS - 1;
      // Step s: the computing wavefronts read stage s; its barrier is passed once stage s + 1 has landed.
      // `end` is known by the step that reads the last stage: `issued` runs kS - 1 stages ahead.
      for (int64_t s = 0; s < end; ++s) {
        one(slot);  // into the slot of stage s - 1, read before the last barrier
        slot = slot + 1 == kS ? 0 : slot + 1;
        wait_vm_n<(kS - 2) * kN>();
        barrier();
      }
      wait_dma();
    };
    if (is_a) run(std::true_type{});
    else run(std::false_type{});
    barrier();  // no load of this class is in flight when the next one lays out its rings
    return;
  }

  const int wr = role.simd / kWC, wc = role.simd % kWC;
  const int frow = lane & 15, fq = lane >> 4;
  auto frag_addr = [&](uint32_t slot_base, int r, int ks) { return slot_base + r * kRowBytes + ((((ks << 2) | fq) ^ swz(r)) << 4); };
  bf16x8 fa[2][kMI], fb[2][kNI];
  int sa = 0, sb = 0;  // ring slots of the stage being read
  auto read_half = [&](int ks, int buf) {
    const uint32_t ab = a_lds + sa * R::kAStage, bb = b_lds + sb * kBStage;
#pragma unroll
    for (int i = 0; i < kMI; ++i)
      fa[buf][i] = *reinterpret_cast<const lds_bf16x8 *>((uintptr_t)frag_addr(ab, wr * 16 * kMI + i * 16 + frow, ks));
#pragma unroll
    for (int j = 0; j < kNI; ++j)
      fb[buf][j] = *reinterpret_cast<const lds_bf16x8 *>((uintptr_t)frag_addr(bb, wc * 16 * kNI + j * 16 + frow, ks));
  };
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  f32x4 acc[kMI][kNI];
  auto mfma_half = [&](int buf, bool zero) {
#pragma unroll
    for (int i = 0; i < kMI; ++i)
#pragma unroll
      for (int j = 0; j < kNI; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[buf][j], fa[buf][i], zero ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][j],
                                                           0, 0, 0);
  };
  const uint32_t ld = static_cast<uint32_t>(p.ncols) * 2u;
  barrier();  // stage 0 has landed
  for (;;) {
    read_half(0, 0);
    for (int kt = 0; kt < ktiles; ++kt) {
      read_half(1, 1);
      mfma_half(0, kt == 0);
      __builtin_amdgcn_sched_barrier(0);
      wait_lds();  // this wavefront's reads of stage kt are done before its slot can be refilled
      barrier();   // the next stage has landed
      sa = sa + 1 == kSA ? 0 : sa + 1;
      sb = sb + 1 == kSB ? 0 : sb + 1;
      if (kt + 1 < ktiles) read_half(0, 0);
      mfma_half(1, false);
      __builtin_amdgcn_sched_barrier(0);
    }
    // acc[i][j] register r of lane l: row i 16 + l % 16, column j 16 + 4 (l / 16) + r of the wavefront's block.
    constexpr int kOut = kSwiglu ? kNI / 2 : kNI;
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.out + static_cast<int64_t>(t.i0) * p.ncols, static_cast<uint32_t>(t.rows) * ld);
    auto value = [&](int i, int j, int q) -> float {
      if constexpr (kSwiglu) {
        const float gt = acc[i][j][q];
        return gt * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gt * -1.4426950408889634f)) * acc[i][j + kOut][q];
      } else {
        return acc[i][j][q];
      }
    };
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
      const uint32_t orow = static_cast<uint32_t>((wr * kMI + i) * 16 + frow);
#pragma unroll
      for (int j = 0; j < kOut; ++j) {
        const bf16x2 lo = {(__bf16)value(i, j, 0), (__bf16)value(i, j, 1)};
        const bf16x2 hi = {(__bf16)value(i, j, 2), (__bf16)value(i, j, 3)};
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 v2 = {__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
        const int c = (wc * kOut + j) * 16 + fq * 4;  // column of the tile
        const int64_t col = static_cast<int64_t>(t.col0) * 16 + c;
        const uint32_t off = c < t.cols * 16 && col < p.ncols ? orow * ld + static_cast<uint32_t>(col) * 2u : kNoAccess;
#if defined(__HIP_DEVICE_COMPILE__)
        __builtin_amdgcn_raw_buffer_store_b64(v2, ro, static_cast<int>(off), 0, 0);
#else
        (void)off;
        (void)v2;
        (void)ro;
#endif
      }
    }
    if (!find(t)) break;
  }
  barrier();  // as the loading wavefronts' last one
}

template <bool kSwiglu, bool kGather>
__global__ __launch_bounds__(512) void expert_stream_kernel(GemmArgs p) {
  __shared__ __attribute__((aligned(1024))) char smem[kLds];
  const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char *)smem));
  Roles role;
  role.lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const Rows first = group_rows(p, role.lane);
  int tiles[3] = {0, 0, 0};  // row tiles of the classes 128, 64, 32
  {
    // Roles: the first wavefront of each SIMD computes (index = its SIMD), the second loads (SIMD 0 and 1: the
    // tile's rows, 2 and 3: weight rows), read from HW_ID and exchanged through LDS. Beside them the row tiles
    // of each class, counted by each wavefront in its share of the groups.
    const int simd = __builtin_amdgcn_readfirstlane(__builtin_amdgcn_s_getreg((1 << 11) | (4 << 6) | 4)) & 3;
    volatile int *sid = reinterpret_cast<volatile int *>(smem);
    int n[3] = {0, 0, 0};
#pragma unroll 4
    for (int g = threadIdx.x; g < static_cast<int>(p.G); g += 512) {
      const int m = group_rows(p, g).m;
      n[0] += class_tiles<128>(m);
      n[1] += class_tiles<64>(m);
      n[2] += class_tiles<32>(m);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1)
#pragma unroll
      for (int c = 0; c < 3; ++c) n[c] += __shfl_xor(n[c], d);
    if (role.lane == 0) {
      sid[wave] = simd;
#pragma unroll
      for (int c = 0; c < 3; ++c) sid[8 + 8 * c + wave] = n[c];
    }
    __syncthreads();
    int before = 0, per_simd[4] = {0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      const int sv = sid[w] & 3;
      per_simd[sv] += 1;
      before += (sv == simd) && (w < wave);
#pragma unroll
      for (int c = 0; c < 3; ++c) tiles[c] += sid[8 + 8 * c + w];
    }
    __syncthreads();
    const bool ok = per_simd[0] == 2 && per_simd[1] == 2 && per_simd[2] == 2 && per_simd[3] == 2;
    role.simd = __builtin_amdgcn_readfirstlane(ok ? simd : (wave & 3));
    role.loader = __builtin_amdgcn_readfirstlane(ok ? before : (wave >> 2));
#pragma unroll
    for (int c = 0; c < 3; ++c) tiles[c] = __builtin_amdgcn_readfirstlane(tiles[c]);
  }
  if (p.tails != nullptr) {
    // Only if every group is short; otherwise the ping-pong kernel that follows takes them all, and needs its list.
    if (tiles[0] > 0) {
      if (blockIdx.x == 0 && wave == 0) tails_list(p.offsets, p.G, p.M, p.tails);
      return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) no_tails(p.tails);
  }
  Plan plan;
  plan.row_tiles = tiles[0] + tiles[1] + tiles[2];
  if (plan.row_tiles == 0) return;
  {
    // Whole rounds of the workgroups, as many as units of the full width need; no unit narrower than a slab.
    // (32 bits: at most 64 rows per group on average, 4096 groups and 2^19 columns.)
    constexpr uint32_t kMax = kSwiglu ? kBRows / 32 : kBRows / 16;
    const uint32_t c16 = static_cast<uint32_t>(p.ncols + 15) / 16, P = gridDim.x, n = static_cast<uint32_t>(plan.row_tiles);
    const uint32_t need = n * ((c16 + kMax - 1) / kMax);
    plan.c16 = static_cast<int>(c16);
    plan.units = static_cast<int>(min((need + P - 1) / P * P, n * c16));
  }
  if (tiles[0] > 0) run_class<128, kSwiglu, kGather>(p, plan, role, lds, first, 0);
  if (tiles[1] > 0) run_class<64, kSwiglu, kGather>(p, plan, role, lds, first, tiles[0]);
  if (tiles[2] > 0) run_class<32, kSwiglu, kGather>(p, plan, role, lds, first, tiles[0] + tiles[1]);
}

}  // namespace

void launch_expert_stream(const GemmArgs &p, bool swiglu, bool gather, hipStream_t s) {
  const dim3 grid(static_cast<uint32_t>(std::max<int64_t>(8, gemm::num_cus() / 8 * 8))), block(512);
  if (swiglu) {
    if (gather) expert_stream_kernel<true, true><<<grid, block, 0, s>>>(p);
    else expert_stream_kernel<true, false><<<grid, block, 0, s>>>(p);
  } else {
    if (gather) expert_stream_kernel<false, true><<<grid, block, 0, s>>>(p);
    else expert_stream_kernel<false, false><<<grid, block, 0, s>>>(p);
  }
}

}  // namespace moe
