// tf32 router weight gradient: grad_weight [N, K] = tf32(grad_output [M, N])^T tf32(inp [M, K]), fp32 in and out, on
// the fp16 matrix cores (tf32_device.h).
//
// inp is the large operand (M x K fp32, 537 MB at 16384 x 8192) and is read once, straight from memory into the
// registers of the wavefront that multiplies it:
//   * a wavefront owns 32 columns of inp and all N (<= 320 a row tile) rows of the result. In the B operand of
//     v_mfma_f32_16x16x32_f16 lane l holds 8 consecutive reduction rows 8 (l / 16) .. + 7 of column l % 16, so a lane that
//     loads two neighbouring columns of those 8 rows (8 bytes each, 128 contiguous bytes per row over 16 lanes) holds
//     the fragments of two blocks, the even columns and the odd ones: no LDS, no transpose, no fp16 copy in memory;
//   * the columns' scales are found on the way: a lane compares its magnitudes with the largest its column's scale
//     takes (one ballot per 32 rows); only when one exceeds it (in the first rows, then rarely) the column's maximum is
//     formed across the lanes and scaled into [2^14, 2^15), and the sums so far, whose column is the lane's own, are
//     multiplied by the change, a power of two. The scale holds up to fp16's largest value, so it is never below the
//     one that the column's largest magnitude as a whole would take, and small values keep as many bits;
//   * the small operand (grad_output, transposed and scaled in fp16 by a kernel before) comes through a ring of three
//     LDS stages of 64 reduction rows, shared by the 8 wavefronts (256 columns);
//   * M is cut into chunks so that there is a unit for every CU; the units of one XCD share a chunk, whose part of the
//     small operand then stays in its L2. The planes of the chunks stay scaled, each column with its chunk's exponent;
//     they are brought to the column's smallest exponent, added in order and scaled back once.
// Measured (MI355X, 16384 x 320 x 8192, us, calls in a graph): 370 -> 157-167 for the whole call; the GEMM 122-135
// (4.0-4.4 TB/s of inp; 150 for the call without the multiplications and conversions, so it is the loads), the planes' sum
// 17, grad_output's maxima and copy 21. Before: column maxima of inp 90, its fp16 copy 180, a GEMM on the copies 143, the
// sum 10. 16384 x 64 x 7168: 308 -> 100; 4096 x 128 x 7168: 100 -> 46; 1024 x 320 x 1024: 44 -> 33; 100 x 64 x 7168: 34 -> 19.
#include <algorithm>
#include <type_traits>

#include "gemm_device.h"
#include "tf32_device.h"

namespace moe {
namespace {

using namespace gemm;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) f16x8 lds_f16x8;

constexpr int kColsWave = 32, kColsTile = 256;
constexpr int kRowB = kBK * 2;  // 128 bytes: one row of the small operand in a stage
constexpr int64_t kWideK = int64_t(1) << 22;
constexpr uint32_t kSkip = 0xfffffff0u;  // an offset past rows, which may span a little more than 2 GiB
constexpr float kF16Max = 65504.f;
constexpr int kNoExp = 1 << 20;  // a column without a finite nonzero value yet: its sums are 0, Inf or NaN, whatever the scale

__device__ __forceinline__ int swz128(int row) { return (row >> 1) & 7; }

struct WgradArgs {
  const uint16_t *rows;  // [N, M8] fp16
  const int32_t *exp;    // [N]
  const float *inp;      // [M, K]
  float *out;            // planes [s, N, K], or (one chunk) the result
  int32_t *col_exp;      // the planes' column exponents [s, K]
  int64_t M, M8, N, K;   // M8: M rounded up to 8
  int64_t chunk;         // reduction rows of a chunk
  int col_tiles, row_tiles, units;
};

// kWide: 64-bit addresses for inp (rows so long that 64 of them do not fit 32-bit offsets, or no room for the planes of
// the chunks that 32-bit ones need). kNt: non-temporal loads of it.
// kOne: one chunk, whose sums are scaled back here.
template <int kMI, bool kWide, bool kNt, bool kOne>
__global__ __launch_bounds__(512) void router_wgrad_kernel(WgradArgs p) {
  constexpr int kStage = kMI * 16 * kRowB;
  constexpr int kSlots = 3;
  constexpr int kDma = kMI * 2 / 8;  // 1 KiB blocks per wavefront and stage
  constexpr int kBufs = 3;           // halves (32 reduction rows) of inp in registers
  static_assert(kMI % 4 == 0 && kSlots * kStage <= 160 * 1024, "stage");
  __shared__ __attribute__((aligned(1024))) char smem[kSlots * kStage];
  const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char *)smem));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int c16 = lane & 15, q = lane >> 4;

  // Units chunk by chunk, then column tile by column tile, the row tiles of one fastest (they read the same inp).
  const int b = static_cast<int>(blockIdx.x), P = static_cast<int>(gridDim.x);
  const int u = (b % 8) * (P / 8) + b / 8;
  if (u >= p.units) return;
  const int per_chunk = p.col_tiles * p.row_tiles;
  const int chunk = u / per_chunk, tile = u - chunk * per_chunk;
  const int ct = tile / p.row_tiles, n0 = (tile - ct * p.row_tiles) * kMI * 16;
  const int64_t m0 = chunk * p.chunk, mrows = min(p.chunk, p.M - m0);
  const int steps = static_cast<int>((mrows + kBK - 1) / kBK);
  [[maybe_unused]] const int halves = 2 * steps;

  // ---- the small operand: this wavefront's blocks wave + 8 j of 8 rows
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.rows + static_cast<int64_t>(n0) * p.M8 + m0,
                                              static_cast<uint32_t>(((min<int64_t>(p.N - n0, kMI * 16) - 1) * p.M8 + p.M8 - m0) * 2));
  int a_off[kDma];
#pragma unroll
  for (int j = 0; j < kDma; ++j) {
    const int r = (wave + 8 * j) * 8 + (lane >> 3);
    a_off[j] = n0 + r < p.N ? static_cast<int>(static_cast<uint32_t>(r) * static_cast<uint32_t>(p.M8 * 2) +
                                               static_cast<uint32_t>(((lane & 7) ^ swz128(r)) << 4))
                            : static_cast<int>(kSkip);
  }
  // Stage st into its slot; past the last one the last one again, into a slot that nothing reads any more. A lane's eight
  // values are the same ones of every row (the swizzle depends on wave % 2 alone); past M8 they are the next row's, and
  // none are read.
  const int a_row = ((lane & 7) ^ swz128(wave * 8 + (lane >> 3))) * 8;
  const int rows8 = static_cast<int>(p.M8 - m0 < p.chunk ? p.M8 - m0 : p.chunk);
  auto dma = [&](int st) {
    const uint32_t dst = lds + (st % kSlots) * kStage;
    const int sc = min(st, steps - 1), k = sc * kRowB;
    const bool in = sc * kBK + a_row < rows8;
#pragma unroll
    for (int j = 0; j < kDma; ++j)
      dma16b(ra, (lds_void *)(uintptr_t)(dst + (wave + 8 * j) * 1024), in ? a_off[j] : static_cast<int>(kSkip), k);
  };

  // ---- inp: columns col, col + 1, rows 32 h + 8 q + r of half h; rows past the chunk and columns past K read zeros
  const int col = ct * kColsTile + wave * kColsWave + 2 * c16;
  const uint32_t ldb = static_cast<uint32_t>(p.K) * 4u;
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(p.inp + m0 * p.K, kWide ? 0u : static_cast<uint32_t>(mrows) * ldb);
  const uint32_t b_off = col < p.K ? static_cast<uint32_t>(8 * q) * ldb + static_cast<uint32_t>(col) * 4u : kNoAccess;
  u32x2 buf[kBufs][8];
  auto load = [&](int h, u32x2 *dst) {
    const uint32_t row = static_cast<uint32_t>(min(h, halves - 1)) * 32u;
    if constexpr (kWide) {
#pragma unroll
      for (uint32_t r = 0; r < 8; ++r) {
        const int64_t m = row + 8 * q + r;
        dst[r] = m < mrows && col < p.K ? *reinterpret_cast<const u32x2 *>(p.inp + (m0 + m) * p.K + col) : u32x2{0u, 0u};
      }
      return;
    }
#if defined(__HIP_DEVICE_COMPILE__)
    // The rows' offsets are in the vector offset: the scalar one is not part of the range check.
#pragma unroll
    for (uint32_t r = 0; r < 8; ++r) dst[r] = __builtin_amdgcn_raw_buffer_load_b64(rb, static_cast<int>(b_off + (row + r) * ldb), 0, kNt ? 2 : 0);
#else
    (void)row;
    (void)b_off;
    (void)rb;
    (void)dst;
#endif
  };

  f32x4 acc[kMI][2];
#pragma unroll
  for (int i = 0; i < kMI; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  int e[2] = {kNoExp, kNoExp};   // the columns' scale exponents
  // Magnitudes below it fit the scale; at first the smallest there is, which only zeros are below.
  float most[2] = {__uint_as_float(1u), __uint_as_float(1u)};
  f16x8 fb[2];
  auto convert = [&](const u32x2 *v) {
    float mx[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      mx[0] = fmaxf(mx[0], fabsf(__uint_as_float(v[r].x)));
      mx[1] = fmaxf(mx[1], fabsf(__uint_as_float(v[r].y)));
    }
    if (__ballot(mx[0] >= most[0] || mx[1] >= most[1]) != 0) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float m = 0.f;
#pragma unroll
        for (int r = 0; r < 8; ++r) m = fmaxf(m, finite_abs(__uint_as_float(j ? v[r].y : v[r].x)));
        m = fmaxf(m, __shfl_xor(m, 16));
        m = fmaxf(m, __shfl_xor(m, 32));
        if (m >= most[j]) {
          const int ne = scale_exp(m), d = ne - e[j];
          e[j] = ne;
          most[j] = __builtin_ldexpf(kF16Max, -ne);  // (tf32 rounding takes no value below it past it)
#pragma unroll
          for (int i = 0; i < kMI; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[i][j][t] = __builtin_ldexpf(acc[i][j][t], d);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 8; ++r)
        fb[j][r] = static_cast<_Float16>(__builtin_ldexpf(__uint_as_float(tf32_rne_bits(j ? v[r].y : v[r].x)), e[j]));
  };
  // Half h of stage st (ks: which half of the stage).
  auto multiply = [&](int slot, int ks) {
    const uint32_t base = lds + slot * kStage;
    const uint32_t at = base + c16 * kRowB + ((((ks << 2) | q) ^ swz128(c16)) << 4);  // 16 rows on: the same swizzle
    f16x8 fa[2][2];
    auto read = [&](int i, f16x8 *f) {
      f[0] = *reinterpret_cast<const lds_f16x8 *>((uintptr_t)(at + i * 16 * kRowB));
      f[1] = *reinterpret_cast<const lds_f16x8 *>((uintptr_t)(at + (i + 1) * 16 * kRowB));
    };
    read(0, fa[0]);
#pragma unroll
    for (int i = 0; i < kMI; i += 2) {
      if (i + 2 < kMI) read(i + 2, fa[(i / 2 + 1) & 1]);
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        acc[i + d][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[(i / 2) & 1][d], fb[0], acc[i + d][0], 0, 0, 0);
        acc[i + d][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[(i / 2) & 1][d], fb[1], acc[i + d][1], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  if (steps > 0) {
    dma(0);
    dma(1);
#pragma unroll
    for (int h = 0; h < kBufs; ++h) load(h, buf[h]);
    // One round: three stages, six halves, so that the slots and register sets are fixed. The wait before a stage's
    // barrier leaves in flight what was issued after the loads of its first half, which follow its own DMA: the next
    // stage's DMA and two halves' loads.
    for (int st = 0; st < steps; st += 3) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        if (st + k < steps) {
          // (kWide: a load that no lane of a wavefront takes is not issued, so the operations in flight cannot be counted.)
          if constexpr (kWide) wait_dma();
          else wait_vm_n<kDma + 16>();
          barrier();  // stage st + k has landed, and every wavefront is done with the stage before
          dma(st + k + 2);
          convert(buf[(2 * k) % 3]);
          __builtin_amdgcn_sched_barrier(0);
          load(2 * (st + k) + 3, buf[(2 * k) % 3]);
          __builtin_amdgcn_sched_barrier(0);
          multiply(k, 0);
          convert(buf[(2 * k + 1) % 3]);
          __builtin_amdgcn_sched_barrier(0);
          load(2 * (st + k) + 4, buf[(2 * k + 1) % 3]);
          __builtin_amdgcn_sched_barrier(0);
          multiply(k, 1);
        }
      }
    }
    wait_dma();  // no LDS DMA outlives the workgroup
  }

  // acc[i][j] register t: row n0 + 16 i + 4 q + t, column col + j.
  float *const out = p.out + (static_cast<int64_t>(chunk) * p.N + n0) * p.K;
  if (col < p.K) {
    if (!kOne && n0 == 0 && q == 0) {
      *reinterpret_cast<u32x2 *>(p.col_exp + chunk * p.K + col) = u32x2{static_cast<uint32_t>(e[0]), static_cast<uint32_t>(e[1])};
    }
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = i * 16 + q * 4 + t;
        if (n0 + r < p.N) {
          float v0 = acc[i][0][t], v1 = acc[i][1][t];
          if constexpr (kOne) {
            const int er = p.exp[n0 + r];
            v0 = __builtin_ldexpf(v0, -(er + e[0]));
            v1 = __builtin_ldexpf(v1, -(er + e[1]));
          }
          *reinterpret_cast<u32x2 *>(out + static_cast<int64_t>(r) * p.K + col) = u32x2{__float_as_uint(v0), __float_as_uint(v1)};
        }
      }
    }
  }
}

// Block (x, y): reduction rows 64 x .. + 63 and columns 64 y .. + 63 of grad_output, transposed through LDS. Each block
// forms its columns' exponents from the slab maxima; those of x = 0 write them.
__global__ __launch_bounds__(256) void router_wgrad_rows_kernel(const float *src, int64_t M, int64_t M8, int64_t N, const float *part,
                                                                int slabs, uint16_t *dst, int32_t *exp) {
  __shared__ int ex[64];
  __shared__ float red[4][64];
  __shared__ uint16_t tile[64][66];  // [column][row], padded against bank conflicts
  const int t = threadIdx.x;
  const int64_t m0 = static_cast<int64_t>(blockIdx.x) * 64, n0 = static_cast<int64_t>(blockIdx.y) * 64;
  {
    const int c = t & 63;
    float m = 0.f;
    if (n0 + c < N)
      for (int s = t >> 6; s < slabs; s += 4) m = fmaxf(m, part[static_cast<int64_t>(s) * N + n0 + c]);
    red[t >> 6][c] = m;
  }
  __syncthreads();
  if (t < 64) {
    const int e = scale_exp(fmaxf(fmaxf(red[0][t], red[1][t]), fmaxf(red[2][t], red[3][t])));
    ex[t] = e;
    if (blockIdx.x == 0 && n0 + t < N) exp[n0 + t] = e;
  }
  __syncthreads();
  if (m0 >= M8) return;  // M = 0: the exponents only
  {
    const int c = (t & 15) * 4;  // N % 8 == 0: the four columns are all valid or all past N
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = (t >> 4) + 16 * k;
      const bool in = m0 + r < M && n0 + c < N;
      const u32x4 v = in ? __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src + (m0 + r) * N + n0 + c)) : u32x4{0u, 0u, 0u, 0u};
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        tile[c + i][r] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(__builtin_ldexpf(__uint_as_float(tf32_rne_bits(w[i])), ex[c + i])));
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int c = (t >> 3) + 32 * k, r = (t & 7) * 8;
    if (n0 + c >= N || m0 + r >= M8) continue;
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = *reinterpret_cast<const uint32_t *>(&tile[c][r + 2 * i]);
    *reinterpret_cast<u32x4 *>(dst + (n0 + c) * M8 + m0 + r) = u32x4{w[0], w[1], w[2], w[3]};
  }
}

// out[n][k] = 2^-(exp[n] + E[k]) sum over s of 2^(E[k] - col_exp[s][k]) planes[s][n][k], s ascending, E[k] the smallest
// col_exp[.][k] (the smallest so far on the way): no plane is made larger, and none leaves the scaled range before the
// total does. N K is a multiple of 64 and below 2^30.
__global__ __launch_bounds__(256) void router_wgrad_sum_kernel(const float *planes, int s, int64_t N, int64_t K, const int32_t *exp,
                                                               const int32_t *col_exp, float *out) {
  const uint32_t quads = static_cast<uint32_t>(K / 4), i = blockIdx.x * 256u + threadIdx.x;
  const uint32_t n = i / quads, c = (i - n * quads) * 4;
  if (n >= static_cast<uint32_t>(N)) return;
  f32x4 sum = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(planes) + i);
  i32x4 least = *reinterpret_cast<const i32x4 *>(col_exp + c);
#pragma unroll 4
  for (int k = 1; k < s; ++k) {
    const f32x4 a = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(planes + k * N * K) + i);
    const i32x4 v = *reinterpret_cast<const i32x4 *>(col_exp + k * K + c);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = min(least[j], v[j]);
      sum[j] = __builtin_ldexpf(sum[j], e - least[j]) + __builtin_ldexpf(a[j], e - v[j]);
      least[j] = e;
    }
  }
  const int er = exp[n];
#pragma unroll
  for (int j = 0; j < 4; ++j) sum[j] = __builtin_ldexpf(sum[j], -(er + least[j]));
  reinterpret_cast<f32x4 *>(out)[i] = sum;
}

}  // namespace

RouterWgradPlan router_wgrad_plan(int64_t M, int64_t N, int64_t K, int64_t most_chunks) {
  RouterWgradPlan pl;
  pl.row_tiles = std::max<int64_t>(1, ceil_div(N, 320));
  const int64_t blocks = ceil_div(ceil_div(std::max<int64_t>(N, 1), pl.row_tiles), 16);
  pl.wide = K >= kWideK;
  pl.mi = pl.wide || blocks <= 4 ? 4 : blocks <= 8 ? 8 : blocks <= 16 ? 16 : 20;
  pl.row_tiles = std::max<int64_t>(1, ceil_div(N, 16 * pl.mi));
  const int64_t tiles = pl.row_tiles * std::max<int64_t>(1, ceil_div(K, kColsTile));
  // At most a unit for every CU (a second round for a few more costs a whole one: 16384 x 64 x 7168, 28 tiles, 10 chunks
  // 139 us, 9 101), of at least 128 rows; and a chunk of inp below 2 GiB (32-bit offsets).
  const int64_t least = pl.wide ? 1 : std::max<int64_t>(1, ceil_div(M * K, (int64_t(1) << 29) - 64 * K));
  int64_t s = std::max(least, std::min(256 / tiles, M / 128));
  s = std::min(s, most_chunks);
  if (s < least) {
    s = 1;
    pl.wide = true;
    pl.mi = 4;
    pl.row_tiles = std::max<int64_t>(1, ceil_div(N, 64));
  }
  pl.c = std::max<int64_t>(1, ceil_div(ceil_div(M, s), kBK)) * kBK;
  pl.s = std::max<int64_t>(1, ceil_div(M, pl.c));
  return pl;
}

void launch_router_wgrad_rows(const float *grad_output, int64_t M, int64_t N, const float *part, int slabs, uint16_t *rows, int32_t *exp,
                              hipStream_t s) {
  router_wgrad_rows_kernel<<<dim3(static_cast<uint32_t>(std::max<int64_t>(1, ceil_div(M, 64))), static_cast<uint32_t>(ceil_div(N, 64))),
                             dim3(256), 0, s>>>(grad_output, M, ceil_div(M, 8) * 8, N, part, slabs, rows, exp);
}

void launch_router_wgrad(const RouterWgradPlan &pl, const uint16_t *rows, const int32_t *exp, const float *inp, int64_t M, int64_t N,
                         int64_t K, float *planes, int32_t *col_exp, float *out, hipStream_t s) {
  WgradArgs p;
  p.rows = rows;
  p.exp = exp;
  p.inp = inp;
  p.out = pl.s > 1 ? planes : out;
  p.col_exp = col_exp;
  p.M = M;
  p.M8 = ceil_div(M, 8) * 8;
  p.N = N;
  p.K = K;
  p.chunk = pl.c;
  p.col_tiles = static_cast<int>(ceil_div(K, kColsTile));
  p.row_tiles = static_cast<int>(pl.row_tiles);
  const int64_t units = pl.s * p.col_tiles * pl.row_tiles;
  p.units = static_cast<int>(units);
  const dim3 grid(static_cast<uint32_t>((units + 7) / 8 * 8)), block(512);
  // Around the Infinity Cache's 256 MB plain loads are faster (us, non-temporal and plain: 117 MB 54 and 49, 268 MB 81 and
  // 72), well above it non-temporal ones (470 MB 101 and 108, 537 MB 171 and 177).
  auto go = [&](auto nt, auto one) {
    constexpr bool kNt = decltype(nt)::value, kOne = decltype(one)::value;
    switch (pl.mi) {
      case 4: router_wgrad_kernel<4, false, kNt, kOne><<<grid, block, 0, s>>>(p); break;
      case 8: router_wgrad_kernel<8, false, kNt, kOne><<<grid, block, 0, s>>>(p); break;
      case 16: router_wgrad_kernel<16, false, kNt, kOne><<<grid, block, 0, s>>>(p); break;
      default: router_wgrad_kernel<20, false, kNt, kOne><<<grid, block, 0, s>>>(p); break;
    }
  };
  const bool nt = M * K > 96 << 20;
  if (pl.wide) router_wgrad_kernel<4, true, false, true><<<grid, block, 0, s>>>(p);  // (one chunk)
  else if (pl.s == 1) go(std::false_type{}, std::true_type{});
  else if (nt) go(std::true_type{}, std::false_type{});
  else go(std::false_type{}, std::false_type{});
  if (pl.s > 1) {
    router_wgrad_sum_kernel<<<dim3(static_cast<uint32_t>(ceil_div(N * K / 4, 256))), dim3(256), 0, s>>>(
        planes, static_cast<int>(pl.s), N, K, exp, col_exp, out);
  }
}

}  // namespace moe
