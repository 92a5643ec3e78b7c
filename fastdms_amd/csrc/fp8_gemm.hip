// FP8 GEMM for prefill row counts on the gfx950 FP8 matrix cores: the
// reference's _fp8_linear for rows above the small-M kernels
// (fastdms/layers/linear.py:635-662: x quantised per row to e4m3fn, then
// torch._scaled_mm(xq, W8^T, scale_a = x_scale_inv, scale_b = w_scale_inv,
// out_dtype = bf16), bias added in bf16):
//
//   y[m, n] = bf16((sum_k xq[m, k] * w8[n, k]) * x_inv[m] * w_inv[n])
//   y[m, n] = bf16(y[m, n] + bias[n])                       (with a bias)
//
// The products of two e4m3 values are exact in fp32; the matrix cores
// accumulate them in fp32 (v_mfma_scale_f32_32x32x64_f8f6f4 with unit E8M0
// block scales), so the result differs from torch's only in summation order.
//
// Tiles are assigned XCD by XCD (block ids are dispatched round robin over the
// 8 XCDs), each XCD taking a contiguous run of tiles.
#include <type_traits>

#include "fdms_common.h"

using namespace fdms;

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));

constexpr int kGemmXcds = 8;

// Two fp32 -> bf16 (round to nearest even) in one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  const bf16x2_t r = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, r);
}

__device__ __forceinline__ i32x8 as_i32x8(const uint4& a, const uint4& b) {
  return i32x8{(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)b.x, (int)b.y, (int)b.z, (int)b.w};
}

}  // namespace

// Workgroup tiles of (32 TM WM) x rows by (32 TN WN) w rows on
// v_mfma_scale_f32_32x32x64_f8f6f4 (lane l holds bytes 32 (l / 32) .. + 31 of row
// l % 32 of a 64-byte k-step), WM x WN waves of TM x TN tiles.  k runs in stages
// of 64 bytes per row, loaded straight into one of NS LDS buffers
// (global_load_lds_dwordx4: no staging registers), so NS - 1 stages are in
// flight while one multiplies.  Iteration t multiplies the fragments of stage t
// from registers beside the LDS reads of stage t + 1; its one barrier says both
// that stage t + 1 has landed and that stage t's buffer has been read.
// LDS rows are 64 bytes with the 16-byte chunks XOR-swizzled (chunk q of row r
// at slot q ^ ((r / 4) & 3)), so the 16 rows a fragment read touches at a time
// spread over the banks.
//
// What bounds it: the latency of a stage's loads while few workgroups run.  Once
// the chip is full the matrix cores are 43 % busy (counters at 12000 x 16384 x
// 2048, clock 2.0 GHz, no LDS bank conflicts; the fragment reads would take 96 of
// 128 bytes a cycle at full matrix rate), so neither they nor LDS is saturated:
// what is left is the barrier per 64-byte stage and, at K = 2048, a tile's
// prologue and epilogue.  Measured with the row quantisation in front (M x N x K,
// against register-staged 256 x 256 tiles of four waves with one k-block in
// flight): 12000 x 16384 x 2048 1 019 -> 455 us (1.77 PFLOP/s; the GEMM alone 418
// us, 1.93), 8192 x 24576 x 4096 1 563 -> 831 (1.98), 12000 x 2048 x 2048 181 -> 80,
// 1500 x 4096 x 4096 141 -> 45, 64 x 2048 x 8192 105 -> 30.
namespace {
constexpr int kStage = 64;  // bytes of a row per stage
constexpr int kGroupM = 4;  // x tiles that share a run of w tiles (4 x 8 tiles per XCD at a time)

// 16 bytes per lane straight into LDS at lds + 16 * lane (lds wave-uniform), from
// a wave-uniform base + 32-bit lane offset, or from a lane's own address.  The
// compiler does not count them: lds_dma_barrier() waits for them.
__device__ __forceinline__ void lds_dma16(const uint8_t* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base)
               : "memory", "m0");
}
__device__ __forceinline__ void lds_dma16_wide(const uint8_t* p, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "memory", "m0");
}
// At most N of this wave's LDS-DMA loads are still in flight and every LDS read
// of it has returned, then the workgroup's barrier.
template <int N>
__device__ __forceinline__ void lds_dma_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
}  // namespace

template <bool BIAS, bool VEC_OUT, bool WIDE, int WM, int WN, int TM, int TN, int NS>
__global__ __launch_bounds__(WM * WN * 64, 2) void fp8_gemm_tile_kernel(
    const uint8_t* __restrict__ x, int64_t x_s, const float* __restrict__ x_inv, const uint8_t* __restrict__ w,
    int64_t w_s, const float* __restrict__ w_inv, const bf16_t* __restrict__ bias, bf16_t* __restrict__ y,
    int64_t y_s, int M, int N, int K, int tiles_m, int tiles_n, int total, int per_xcd) {
  constexpr int NW = WM * WN;
  constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN;
  constexpr int XB = BM * kStage, WB = BN * kStage;  // bytes of a stage of x / w
  constexpr int NX = XB / (1024 * NW), NWI = WB / (1024 * NW);  // LDS-DMA instructions per wave and stage
  static_assert(NX * 1024 * NW == XB && NWI * 1024 * NW == WB, "whole LDS-DMA instructions per wave");
  constexpr int PER = NX + NWI;
  __shared__ __attribute__((aligned(1024))) uint8_t s_buf[NS * (XB + WB)];

  const int lin = blockIdx.x;
  const int t = (lin % kGemmXcds) * per_xcd + lin / kGemmXcds;
  if (t >= total) return;  // uniform per workgroup
  const int grp = t / (kGroupM * tiles_n), rem = t - grp * kGroupM * tiles_n;
  const int gm = min(kGroupM, tiles_m - grp * kGroupM);  // the last group may hold fewer x tiles
  const int tn = rem / gm, tm = grp * kGroupM + rem - tn * gm;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lc = lane & 31, half = lane >> 5;
  const int mb = tm * BM, nb0 = tn * BN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)s_buf;

  // LDS-DMA: instruction i of this wave moves rows 16 (i NW + wave) .. + 15 of
  // the stage, lane l slot l % 4 of row l / 4; rows past M / N repeat the last
  const int drow = lane >> 2, dchunk = (lane & 3) ^ ((lane >> 4) & 3);
  using Off = typename std::conditional<WIDE, int64_t, uint32_t>::type;
  Off xoff[NX], woff[NWI];
#pragma unroll
  for (int i = 0; i < NX; ++i) xoff[i] = (Off)min(16 * (i * NW + wave) + drow, M - 1 - mb) * (Off)x_s;
#pragma unroll
  for (int i = 0; i < NWI; ++i) woff[i] = (Off)min(16 * (i * NW + wave) + drow, N - 1 - nb0) * (Off)w_s;
  const uint8_t* xb = x + (int64_t)mb * x_s;
  const uint8_t* wb = w + (int64_t)nb0 * w_s;
  const int nst = K / kStage + (K % kStage != 0);  // K may be near 2^31
  auto load_stage = [&](int st) {
    const uint32_t buf = lds0 + (uint32_t)(st % NS) * (XB + WB);
    const int k0 = st * kStage;
    // the last stage's chunks past K read chunk 0 of their row (in bounds)
    const uint32_t ko = k0 + 16 * dchunk < K ? (uint32_t)(k0 + 16 * dchunk) : 0u;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const uint32_t dst = buf + (uint32_t)((i * NW + wave) * 1024);
      if constexpr (WIDE) lds_dma16_wide(xb + xoff[i] + ko, dst); else lds_dma16(xb, xoff[i] + ko, dst);
    }
#pragma unroll
    for (int i = 0; i < NWI; ++i) {
      const uint32_t dst = buf + XB + (uint32_t)((i * NW + wave) * 1024);
      if constexpr (WIDE) lds_dma16_wide(wb + woff[i] + ko, dst); else lds_dma16(wb, woff[i] + ko, dst);
    }
  };

  // fragments: lane (half, lc) holds bytes 32 half .. + 31 of row lc of a 32-row tile
  const int xr0 = (wave / WN) * 32 * TM, wr0 = (wave % WN) * 32 * TN;
  const int f = (lc >> 2) & 3;
  const uint32_t a0 = lc * kStage + (((2 * half) ^ f) << 4), a1 = lc * kStage + (((2 * half + 1) ^ f) << 4);
  struct Frags {
    i32x8 x[TM], w[TN];
  };
  auto read_frags = [&](Frags& fr, int st) {
    const uint8_t* xs = s_buf + (st % NS) * (XB + WB) + xr0 * kStage;
    const uint8_t* ws = s_buf + (st % NS) * (XB + WB) + XB + wr0 * kStage;
#pragma unroll
    for (int i = 0; i < TN; ++i)
      fr.w[i] = as_i32x8(*reinterpret_cast<const uint4*>(ws + i * 32 * kStage + a0),
                         *reinterpret_cast<const uint4*>(ws + i * 32 * kStage + a1));
#pragma unroll
    for (int j = 0; j < TM; ++j)
      fr.x[j] = as_i32x8(*reinterpret_cast<const uint4*>(xs + j * 32 * kStage + a0),
                         *reinterpret_cast<const uint4*>(xs + j * 32 * kStage + a1));
  };
  // a partial last stage: the 16-byte chunks past K become zero in LDS
  auto landed = [&](int st) {
    if (K % kStage == 0 || st != nst - 1) return;  // uniform
    uint8_t* buf = s_buf + (st % NS) * (XB + WB);
    for (int u = tid; u < (BM + BN) * 4; u += NW * 64)
      if (st * kStage + 16 * ((u & 3) ^ ((u >> 4) & 3)) >= K) *reinterpret_cast<uint4*>(buf + 16 * u) = uint4{0u, 0u, 0u, 0u};
    lds_dma_barrier<0>();
  };
  f32x16 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x16{};
  auto mma = [&](const Frags& fr) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fr.w[i], fr.x[j], acc[i][j], 0, 0, 0, 127, 0, 127);
  };

#pragma unroll
  for (int st = 0; st < NS; ++st)
    if (st < nst) load_stage(st);
  // stage 0 has landed (fewer stages in flight than NS - 1: all have)
  if (nst >= NS) lds_dma_barrier<(NS - 1) * PER>(); else lds_dma_barrier<0>();
  Frags fa, fb;
  landed(0);
  read_frags(fa, 0);
  // multiplies stage st (fragments cur) while stage st + 1's fragments are read
  // into nxt: the reads are issued before the products, which hide them
  auto step = [&](int st, Frags& cur, Frags& nxt) {
    if (st + NS - 1 < nst) lds_dma_barrier<(NS - 2) * PER>(); else lds_dma_barrier<0>();
    if (st + NS < nst) load_stage(st + NS);
    landed(st + 1);
    read_frags(nxt, st + 1);  // past the last stage: bytes no one uses
    __builtin_amdgcn_sched_barrier(0);
    mma(cur);
    __builtin_amdgcn_sched_barrier(0);
  };
  int st = 0;
  for (; st + 1 < nst; st += 2) {
    step(st, fa, fb);
    step(st + 1, fb, fa);
  }
  if (st < nst) step(st, fa, fb);

  // lane (lc, half) holds C[n = wr0 + 32 i + 8 (r / 4) + 4 half + r % 4][m = xr0 + 32 j + lc]
  __builtin_amdgcn_sched_barrier(0);  // the scales are not worth registers during the products
  float xsc[TM];
#pragma unroll
  for (int j = 0; j < TM; ++j) xsc[j] = x_inv[min(mb + xr0 + 32 * j + lc, M - 1)];
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int nt = nb0 + wr0 + 32 * i;
    float wsc[16], bs[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int n = min(nt + 8 * (r / 4) + 4 * half + r % 4, N - 1);
      wsc[r] = w_inv[n];
      bs[r] = BIAS ? bf16_to_f32(bias[n].bits) : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int m = mb + xr0 + 32 * j + lc;
      bf16_t* yr = y + (int64_t)min(m, M - 1) * y_s;
      uint32_t o[8];
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          v[e] = acc[i][j][r + e] * xsc[j] * wsc[r + e];
          if (BIAS) v[e] = bf16_to_f32(f32_to_bf16(v[e])) + bs[r + e];
        }
        o[r / 2] = pack_bf16(v[0], v[1]);
      }
      if (VEC_OUT && nt + 32 <= N) {  // uniform: the halves swap quads so that a lane stores 8 columns at once
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const auto s0 = __builtin_amdgcn_permlane32_swap(o[4 * q], o[4 * q + 2], false, false);
          const auto s1 = __builtin_amdgcn_permlane32_swap(o[4 * q + 1], o[4 * q + 3], false, false);
          if (m < M) *reinterpret_cast<u32x4_a8*>(yr + nt + 16 * q + 8 * half) = u32x4_a8{s0[0], s1[0], s0[1], s1[1]};
        }
      } else if (m < M) {
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          const int n = nt + 8 * (r / 4) + 4 * half;
          if (VEC_OUT && n + 3 < N) {
            *reinterpret_cast<uint2*>(yr + n) = uint2{o[r / 2], o[r / 2 + 1]};
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < N) yr[n + e].bits = (uint16_t)(o[(r + e) / 2] >> (16 * (e & 1)));
          }
        }
      }
    }
    if (BIAS) __builtin_amdgcn_sched_barrier(0);
  }
}

// y [M, N] bf16 (row stride y_s elements) = the FP8 product above.  x, w:
// e4m3fn rows [M, K] / [N, K] with byte strides x_s / w_s; K, the strides and
// the pointers 16-byte multiples.  x_inv [M], w_inv [N] fp32; bias [N] bf16 or
// NULL.
FDMS_EXPORT int fdms_fp8_gemm(const void* x, int64_t x_s, const float* x_inv, const void* w, int64_t w_s,
                              const float* w_inv, const void* bias, void* y, int64_t y_s, int M, int N, int K,
                              void* stream) {
  if (M < 0 || N <= 0 || K <= 0 || (K & 15) || (x_s & 15) || (w_s & 15) || x_s < K || w_s < K || y_s < N)
    return (int)hipErrorInvalidValue;
  if (M == 0) return 0;
  if (!x || !x_inv || !w || !w_inv || !y) return (int)hipErrorInvalidValue;
  if (((uintptr_t)x | (uintptr_t)w) & 15) return (int)hipErrorInvalidValue;
  // 8-byte aligned rows: whole 32-column tiles leave as 16-byte stores (a global store needs 4-byte alignment),
  // the last columns as 8-byte ones (12000 x 16384 x 2048 with a row stride of 16388: 494 us, 810 in 2-byte stores)
  const bool vec = (y_s % 4) == 0 && ((uintptr_t)y % 8) == 0;
#define FDMS_GEMM_TILE(B, V, ...)                                                                                  \
  hipLaunchKernelGGL((fp8_gemm_tile_kernel<B, V, __VA_ARGS__>), grid, dim3(threads), 0, (hipStream_t)stream,        \
                     (const uint8_t*)x, x_s, x_inv, (const uint8_t*)w, w_s, w_inv, (const bf16_t*)bias, (bf16_t*)y,  \
                     y_s, M, N, K, (int)tm, (int)tn, (int)total, per_xcd)
#define FDMS_GEMM_TILES(THREADS, BM, BN, ...)                                                                     \
  {                                                                                                                \
    constexpr int threads = THREADS;                                                                               \
    const int64_t tm = tiles(M, BM), tn = tiles(N, BN), total = tm * tn;                                           \
    if (total > (int64_t)0x7FFFFFFF - kGemmXcds) return (int)hipErrorInvalidValue;                                 \
    const int per_xcd = (int)((total + kGemmXcds - 1) / kGemmXcds);                                                \
    const dim3 grid((unsigned)(per_xcd * kGemmXcds));                                                              \
    if (bias) {                                                                                                    \
      if (vec) FDMS_GEMM_TILE(true, true, __VA_ARGS__); else FDMS_GEMM_TILE(true, false, __VA_ARGS__);             \
    } else {                                                                                                       \
      if (vec) FDMS_GEMM_TILE(false, true, __VA_ARGS__); else FDMS_GEMM_TILE(false, false, __VA_ARGS__);           \
    }                                                                                                              \
    FDMS_LAUNCH_CHECK();                                                                                           \
    return 0;                                                                                                      \
  }
  const auto tiles = [](int n, int b) { return ((int64_t)n + b - 1) / b; };
  // row offsets inside a tile are 32-bit below a row stride of 16 MiB
  if (x_s >= (1 << 24) || w_s >= (1 << 24)) FDMS_GEMM_TILES(256, 64, 64, true, 2, 2, 1, 1, 6)
  // 256 x 256 tiles (one workgroup per CU) when they fill their last round of
  // the 256 CUs to four fifths on average: 4096^3 74 us against 92 for 128 x 128
  // tiles (two workgroups per CU), but 5000 x 4096 x 4096 (320 tiles) 125 against
  // 113 and 12000 x 2048 x 2048 (376 tiles) 81 against 79
  const int64_t big = tiles(M, 256) * tiles(N, 256), rounds = (big + 255) / 256;
  if (5 * big >= 4 * 256 * rounds) FDMS_GEMM_TILES(512, 256, 256, false, 4, 2, 2, 4, 5)
  // 64 x 64 tiles (six stages) while 128 x 128 ones leave half the chip idle:
  // 300 x 2048 x 8192 (48 tiles) 31 us against 46, 500 x 6144 x 4096 (192) 32 against 28
  if (tiles(M, 128) * tiles(N, 128) >= 128) FDMS_GEMM_TILES(256, 128, 128, false, 2, 2, 2, 2, 4)
  FDMS_GEMM_TILES(256, 64, 64, false, 2, 2, 1, 1, 6)
#undef FDMS_GEMM_TILES
#undef FDMS_GEMM_TILE
}
