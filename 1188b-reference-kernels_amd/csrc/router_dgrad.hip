// tf32 router input gradient: grad_input [M, N] = tf32(grad_output [M, K]) tf32(weight [K, N]), fp32 in and out, on the
// fp16 matrix cores (tf32_device.h), for reductions of at most 320 (the number of experts).
//
// The work is the output: 4 M N bytes written (537 MB at 16384 x 8192) for a reduction of a few hundred, so the kernel
// is built around the stores:
//   * the weight stays where it is used: a wavefront owns 64 columns and holds all their MFMA fragments (40 of 16 bytes
//     a lane at K = 320) in registers for its whole run; only grad_output's rows stream by, through a ring of three LDS
//     stages of 64 rows that the 8 wavefronts (512 columns; 2 or 4 where there are few rows) share, with one barrier a
//     stage;
//   * block j of a wavefront's four is columns 4 c + j, c = 0 .. 15, so a lane's four accumulators of a row are four
//     neighbouring columns: one 16-byte store, 256 contiguous bytes of a row over 16 lanes;
//   * nothing waits for the stores: they are older than the loads that the next stages wait for only by whole stages.
// grad_output is scaled per row, weight per column (transposed, so that both are read along the reduction), in one launch
// before; the epilogue undoes both.
// Measured (MI355X, us for the call in a graph): 16384 x 320 x 8192 217 -> 125-140 (the GEMM 209 -> 107-122: 4.4-5.0 TB/s
// of output; its operands' preparation 25 in four launches -> 18 in one), 16384 x 64 x 7168 163 -> 95, 1024 x 320 x 1024
// 21.5 -> 18.2, 100 x 64 x 7168 19.0 -> 9.5.
// Before: 128 x 128 tiles of five reduction steps, 32 bytes of a row per store, still what longer reductions run
// (grouped_gemm_dgrad128_kernel in grouped_gemm_bwd.hip).
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
typedef __attribute__((address_space(3))) f16x8 lds_f16x8;
typedef __attribute__((address_space(3))) uint32_t lds_u32;

constexpr int kRowsStage = 64, kColsWave = 64;
// Rows' exponents as bytes: scale_exp is -113 to 163, and a row whose largest magnitude is below 2^-128 (above 142) is as
// exact with 142: its values, multiples of 2^-149, become multiples of 2^-7 below 2^14.
constexpr int kExpBias = 15, kExpMost = 127 + kExpBias;

struct DgradArgs {
  const uint16_t *a;    // [M, K] fp16: scaled rows of grad_output
  const uint16_t *b;    // [N, K] fp16: scaled columns of weight
  const int8_t *a_exp;  // [M rounded up to 4]: exponents, kExpBias less
  const int32_t *b_exp; // [N]
  float *out;
  int64_t M, N;
  int K;                // (a row's 64 kKS2 values past K are zeros)
  int64_t chunk;        // rows of a unit (a multiple of 64)
  int col_tiles, units;
};

// kKS2: 64-deep steps of the reduction. kWaves: wavefronts of a workgroup.
template <int kKS2, int kWaves>
__global__ __launch_bounds__(64 * kWaves) void router_dgrad_kernel(DgradArgs p) {
  constexpr int kColsTile = kWaves * kColsWave;
  constexpr int kKS = 2 * kKS2;                  // MFMAs per block
  constexpr int kRowB = 128 * kKS2;              // bytes of a row in LDS
  constexpr int kStage = kRowsStage * kRowB;     // 8 kKS2 KiB
  constexpr int kExp = kRowsStage * 4;           // the rows' exponents
  constexpr int kSlots = 3;
  constexpr int kDma = 8 * kKS2 / kWaves;        // 1 KiB blocks per wavefront and stage
  constexpr int kStores = kRowsStage / 16 * 4;   // per lane and stage
  constexpr int kLds = kSlots * (kStage + kExp);
  static_assert(kLds <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) char smem[kLds];
  const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char *)smem));
  const uint32_t lds_exp = lds + kSlots * kStage;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int c16 = lane & 15, q = lane >> 4;
  const int b = static_cast<int>(blockIdx.x), P = static_cast<int>(gridDim.x);
  const int u = (b % 8) * (P / 8) + b / 8;  // an XCD takes neighbouring units: the column tiles of one chunk of rows
  if (u >= p.units) return;
  const int ct = u % p.col_tiles;
  const int64_t m0 = static_cast<int64_t>(u / p.col_tiles) * p.chunk, m1 = min(p.M, m0 + p.chunk);
  const int stages = static_cast<int>((m1 - m0 + kRowsStage - 1) / kRowsStage);

  // ---- rows: block wave + kWaves j of a stage; 16-byte chunks of a row are XORed with the row within each 128 bytes, those past
  // K and rows past M read zeros. The offsets are formed anew for each stage (from a lane index the compiler takes for
  // another): the registers are the weight's.
  const int row_bytes = p.K * 2;
  auto dma = [&](int st) {
    const int sc = min(st, stages - 1);  // past the last stage the last one again, into a slot nothing reads any more
    const int64_t m = m0 + static_cast<int64_t>(sc) * kRowsStage;
    const int slot = st % kSlots;
    if (wave == 0) {
#if defined(__HIP_DEVICE_COMPILE__)
      const uint32_t bytes = static_cast<uint32_t>(min<int64_t>(kRowsStage, (p.M - m + 3) & ~int64_t(3)));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(p.a_exp + m, bytes), (lds_void *)(uintptr_t)(lds_exp + slot * kExp), 4, lane * 4, 0, 0, 0);
#endif
    }
    const __amdgpu_buffer_rsrc_t ra =
        make_rsrc(p.a + m * p.K, static_cast<uint32_t>(static_cast<int>(min<int64_t>(kRowsStage, p.M - m)) * row_bytes));
    int ln = lane;
    asm volatile("" : "+v"(ln));
#pragma unroll
    for (int j = 0; j < kDma; ++j) {
      const int at = (wave + kWaves * j) * 64 + ln;  // chunk of the stage, as it lies in LDS
      const int r = at / (8 * kKS2), c = at % (8 * kKS2);
      const int from = ((c & ~7) | ((c ^ r) & 7)) * 16;
      dma16b(ra, (lds_void *)(uintptr_t)(lds + slot * kStage + (wave + kWaves * j) * 1024),
             from < row_bytes ? r * row_bytes + from : static_cast<int>(kNoAccess), 0);
    }
  };
  dma(0);
  dma(1);

  // ---- this wavefront's columns
  const int64_t n0 = static_cast<int64_t>(ct) * kColsTile + wave * kColsWave + 4 * c16;
  const bool in = n0 < p.N;  // N % 8 == 0: a lane's four columns are all valid or all past N
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(p.b, static_cast<uint32_t>(p.N) * static_cast<uint32_t>(row_bytes));  // 3 K N < 2^30
  f16x8 fb[kKS][4];
  int eb[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t n = in ? n0 + j : 0;
    eb[j] = p.b_exp[n] + kExpBias;
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks) {
      const int k = ks * 32 + q * 8;
#if defined(__HIP_DEVICE_COMPILE__)
      fb[ks][j] = __builtin_bit_cast(
          f16x8, __builtin_amdgcn_raw_buffer_load_b128(
                     rb, k < p.K ? static_cast<int>(n) * row_bytes + k * 2 : static_cast<int>(kNoAccess), 0, 0));
#else
      (void)k;
      (void)rb;
      fb[ks][j] = f16x8{};
#endif
    }
  }
  const uint32_t ld = static_cast<uint32_t>(p.N) * 4u;
  const uint32_t o_lane = in ? static_cast<uint32_t>(4 * q) * ld + static_cast<uint32_t>(n0) * 4u : kNoAccess;
  const uint32_t a_lane = static_cast<uint32_t>(c16) * kRowB + (((q ^ c16) & 7) << 4);

  for (int st = 0; st < stages; ++st) {
    // The stage's DMA has landed: after it came the stores of two stages and the next stage's DMA.
    if (st == 0) wait_dma();
    else wait_vm_n<2 * kStores + kDma>();
    barrier();
    dma(st + 2);  // into the slot of stage st - 1, which every wavefront has left
    const int64_t m = m0 + static_cast<int64_t>(st) * kRowsStage;
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.out + m * p.N, static_cast<uint32_t>(min<int64_t>(m1 - m, kRowsStage)) * ld);
    const uint32_t base = lds + (st % kSlots) * kStage + a_lane, ebase = lds_exp + (st % kSlots) * kExp;
#pragma unroll 1
    for (int i = 0; i < kRowsStage / 16; ++i) {
      f32x4 acc[4];
      f16x8 fa[2];
      // chunk 4 ks + q of the row: its 128 bytes, and within them the swizzled place (the odd ks's differs by 64 bytes)
      auto read = [&](int ks) {
        return *reinterpret_cast<const lds_f16x8 *>((uintptr_t)((base ^ ((ks & 1) << 6)) + i * 16 * kRowB + (ks >> 1) * 128));
      };
      fa[0] = read(0);
      const uint32_t ea = *reinterpret_cast<const lds_u32 *>((uintptr_t)(ebase + i * 16 + 4 * q));  // four rows' bytes
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) {
        if (ks + 1 < kKS) fa[(ks + 1) & 1] = read(ks + 1);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[ks & 1], fb[ks][j], ks == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);  // no further reads ahead: the registers are the weight's
      }
      // acc[j] register t: row 16 i + 4 q + t, column n0 + j
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        u32x4 v;
        const int er = static_cast<int8_t>(ea >> (8 * t));
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __float_as_uint(__builtin_ldexpf(acc[j][t], -(er + eb[j])));
#if defined(__HIP_DEVICE_COMPILE__)
        __builtin_amdgcn_raw_buffer_store_b128(v, ro, static_cast<int>(in ? o_lane + static_cast<uint32_t>(i * 16 + t) * ld : kNoAccess), 0, 0);
#else
        (void)ro;
        (void)o_lane;
        (void)v;
#endif
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  wait_dma();  // no LDS DMA outlives the workgroup
}

// Both operands in one launch. Blocks [0, wb): 64 columns of weight [K, N] each, all K <= 64 kV / 4 rows: its columns'
// largest finite magnitudes, their exponents, the scaled columns as rows of b. The other blocks: four rows of grad_output
// each, one per wavefront.
template <int kV>
__global__ __launch_bounds__(256) void router_dgrad_prepare_kernel(const float *w, const float *go, int64_t M, int K, int64_t N, int wb,
                                                                   uint16_t *a, uint16_t *bt, int8_t *a_exp, int32_t *b_exp) {
  constexpr int kRows = 16 * kV;              // rows of weight held by a block
  constexpr int kPitch = kRows + 8;           // LDS row of a column, in values (16-byte rows; a bank offset per column)
  __shared__ __attribute__((aligned(16))) uint16_t tile[64 * kPitch];
  __shared__ float red[16][64];
  const int t = threadIdx.x;
  if (static_cast<int>(blockIdx.x) < wb) {
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * 64;
    const int c = (t & 15) * 4, r0 = t >> 4;
    u32x4 v[kV];
    float mx[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kV; ++i) {
      const int r = r0 + 16 * i;
      v[i] = r < K && n0 + c < N ? *reinterpret_cast<const u32x4 *>(w + static_cast<int64_t>(r) * N + n0 + c) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < kV; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) mx[k] = fmaxf(mx[k], finite_abs(__uint_as_float(v[i][k])));
#pragma unroll
    for (int k = 0; k < 4; ++k) red[r0][c + k] = mx[k];
    __syncthreads();
    int e[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float m = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) m = fmaxf(m, red[i][c + k]);
      e[k] = scale_exp(m);
      if (r0 == 0 && n0 + c + k < N) b_exp[n0 + c + k] = e[k];
    }
#pragma unroll
    for (int i = 0; i < kV; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        tile[(c + k) * kPitch + r0 + 16 * i] =
            __builtin_bit_cast(uint16_t, static_cast<_Float16>(__builtin_ldexpf(__uint_as_float(tf32_rne_bits(v[i][k])), e[k])));
    __syncthreads();
    const int per = K / 8;  // 16-byte pieces of a column
    for (int i = t; i < 64 * per; i += 256) {
      const int n = i / per, k = i - n * per;
      if (n0 + n < N) *reinterpret_cast<u32x4 *>(bt + (n0 + n) * K + k * 8) = *reinterpret_cast<const u32x4 *>(&tile[n * kPitch + k * 8]);
    }
    return;
  }
  const int64_t m = static_cast<int64_t>(blockIdx.x - wb) * 4 + t / kWave;
  const int lane = t % kWave;
  if (m >= M) return;
  constexpr int kU = (kRows + 255) / 256;  // 4 values a lane at a time
  u32x4 v[kU];
  float mx = 0.f;
#pragma unroll
  for (int i = 0; i < kU; ++i) {
    const int k = (lane + i * kWave) * 4;
    v[i] = k < K ? __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(go + m * K + k)) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 4; ++j) mx = fmaxf(mx, finite_abs(__uint_as_float(v[i][j])));
  }
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
  const int e = min(scale_exp(mx), kExpMost);
  if (lane == 0) a_exp[m] = static_cast<int8_t>(e - kExpBias);
#pragma unroll
  for (int i = 0; i < kU; ++i) {
    const int k = (lane + i * kWave) * 4;
    if (k >= K) continue;
    uint32_t h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      h[j] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(__builtin_ldexpf(__uint_as_float(tf32_rne_bits(v[i][j])), e)));
    *reinterpret_cast<u32x2 *>(a + m * K + k) = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
  }
}

int64_t round64(int64_t v) { return ceil_div(v, 64) * 64; }

}  // namespace

bool router_dgrad_applies(int64_t K) { return K > 0 && K <= 320; }

RouterDgradLayout router_dgrad_layout(int64_t M, int64_t K, int64_t N) {
  RouterDgradLayout l;
  auto take = [&](int64_t bytes) {
    const size_t at = l.total;
    l.total += static_cast<size_t>(ceil_div(bytes, 256) * 256);
    return at;
  };
  l.a = take(M * K * 2);
  l.b = take(K * N * 2);
  l.a_exp = take(ceil_div(M, 4) * 4);
  l.b_exp = take(N * 4);
  return l;
}

void launch_router_dgrad(const float *go, int64_t M, int64_t K, const float *w, int64_t N, float *out, void *workspace, hipStream_t s) {
  const RouterDgradLayout l = router_dgrad_layout(M, K, N);
  char *ws = static_cast<char *>(workspace);
  const int64_t wb = ceil_div(N, 64);
  uint16_t *a = reinterpret_cast<uint16_t *>(ws + l.a), *b = reinterpret_cast<uint16_t *>(ws + l.b);
  int8_t *a_exp = reinterpret_cast<int8_t *>(ws + l.a_exp);
  int32_t *b_exp = reinterpret_cast<int32_t *>(ws + l.b_exp);
  DgradArgs p;
  p.a = a;
  p.b = b;
  p.a_exp = a_exp;
  p.b_exp = b_exp;
  p.out = out;
  p.M = M;
  p.N = N;
  p.K = static_cast<int>(K);
  // The fewer columns a workgroup owns, the less weight it waits for at its start: 2 or 4 wavefronts where all units of one
  // stage then have a CU each (us, 2, 4 and 8 wavefronts, reductions of 320: 16 x 2048 16.8, 18.0, 23.1; 1024 x 1024 18.2,
  // 19.3, 23.7; 2048 x 2048, twice the CUs with 2, 25.5, 23.1, 27.6; 8192 x 4096, four times with 4, 78.6, 50.7, 45.1).
  auto fits = [&](int64_t n) { return ceil_div(N, n * kColsWave) * ceil_div(M, kRowsStage) <= num_cus(); };
  const int waves = fits(2) ? 2 : fits(4) ? 4 : 8;
  p.col_tiles = static_cast<int>(ceil_div(N, waves * kColsWave));
  // A unit for every CU, of whole stages.
  p.chunk = round64(std::max<int64_t>(64, ceil_div(M, std::max<int64_t>(1, num_cus() / p.col_tiles))));
  p.units = static_cast<int>(ceil_div(M, p.chunk)) * p.col_tiles;
  const dim3 grid(static_cast<uint32_t>((p.units + 7) / 8 * 8)), pgrid(static_cast<uint32_t>(wb + ceil_div(M, 4)));
  auto go_ = [&](auto steps) {
    constexpr int kSteps = decltype(steps)::value;
    router_dgrad_prepare_kernel<4 * kSteps><<<pgrid, dim3(256), 0, s>>>(w, go, M, static_cast<int>(K), N, static_cast<int>(wb), a, b, a_exp,
                                                                        b_exp);
    if (waves == 2) router_dgrad_kernel<kSteps, 2><<<grid, dim3(128), 0, s>>>(p);
    else if (waves == 4) router_dgrad_kernel<kSteps, 4><<<grid, dim3(256), 0, s>>>(p);
    else router_dgrad_kernel<kSteps, 8><<<grid, dim3(512), 0, s>>>(p);
  };
  switch (ceil_div(K, 64)) {
    case 1: go_(std::integral_constant<int, 1>{}); break;
    case 2: go_(std::integral_constant<int, 2>{}); break;
    case 3: go_(std::integral_constant<int, 3>{}); break;
    case 4: go_(std::integral_constant<int, 4>{}); break;
    default: go_(std::integral_constant<int, 5>{}); break;
  }
}

}  // namespace moe
