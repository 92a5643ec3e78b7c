// Dense causal prefill attention over a ragged batch (the reference calls
// flash_attn_varlen_func(q, k, v, cu_seqlens_q, cu_seqlens_k, causal=True),
// attention.py:85-92: evictions act only at pack time, so prefill attends to
// the full prompt).  A sequence's query rows are the last of its keys
// (flash-attn's bottom-right causal alignment): a chunk of a long prompt
// attends to the retained earlier chunks plus itself.
//
// bf16 in/out, fp32 softmax, GQA.  A workgroup takes 128 query rows -- P =
// 128 / G positions of the G query heads that share a KV head (G = 1, 2, 4;
// other group sizes run G = 1, one query head at a time) -- four waves of 32
// rows.  Per 64-key block a wave computes, on v_mfma_f32_32x32x16_bf16,
//   S^T (keys x queries) = K . Q^T,   p = exp2(S * scale - m),
//   O^T (d x queries)   += V^T . P^T.
// Operand layout (lane l, half = l / 32, 8 values i each):
//   A[row = l % 32][k = 8 * half + i],  B[k = 8 * half + i][col = l % 32],
//   C[row = 8 * (r / 4) + 4 * half + r % 4][col = l % 32], r = 0 .. 15.
// A lane owns one query: its max, its sum and its rescale factor are scalars
// of that lane (one half swap per block, no broadcasts).  S^T's C layout is
// the B operand of V^T . P^T once the 16 keys of a step are taken in the order
// 8 * (i / 4) + 4 * half + i % 4, which is the order V is read in.
#include <cfloat>
#include <type_traits>

#include "fdms_common.h"
#include "fdms_prefill_blocks.h"

using namespace fdms;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kKeys = kPrefillKeys;  // keys per LDS block
constexpr int kThreads = 256;
constexpr int kWaveRows = kPrefillWaveRows;  // query rows per wave

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) {
  bf16x8 r;
  __builtin_memcpy(&r, &v, 16);
  return r;
}

// Two fp32 -> bf16 (round to nearest even) in one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
  const bf16x2 r = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, r);
}

__device__ __forceinline__ f32x4 mfma16x16x32(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32x32x16(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 16 bytes per lane from base + voff straight into LDS at lds + 16 * lane
// (lds wave-uniform).  The compiler does not count it: lds_dma_barrier() below
// waits for it before the workgroup's barrier.
__device__ __forceinline__ void lds_dma16(const uint8_t* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base)
               : "memory", "m0");
}
// Every LDS-DMA of this wave has landed and every LDS read of it has
// returned, then the workgroup's barrier.
__device__ __forceinline__ void lds_dma_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Max over the two lanes of a query (l and l ^ 32).
__device__ __forceinline__ float halves_max(float v) {
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __builtin_elementwise_maximum(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// K/V rows in LDS are row-major and unpadded with the 16-byte chunks of a row
// XOR-swizzled.  K: chunk c of row r at slot c ^ (r & 15) (head_dim 128; (r / 2)
// & 7 at 64), so the 32 rows of an A operand spread over all banks.  V: chunk c
// at slot c ^ 4 * (r & 3) (4 * ((r / 2) & 1)); its A operand is read with the
// transposing ds_read_b64_tr_b16 (16 lanes: four keys x 16 dims).
template <int D>
__device__ __forceinline__ int k_swizzle(int row) {
  return D == 128 ? row & 15 : (row >> 1) & 7;
}
template <int D>
__device__ __forceinline__ int v_swizzle(int row) {
  return D == 128 ? (row & 3) << 2 : ((row >> 1) & 1) << 2;
}
// Byte offset of a lane's part of the K operand (32 keys x 16 dims from dim 16 j).
template <int D>
__device__ __forceinline__ uint32_t k_operand(int lane, int j) {
  const int row = lane & 31;
  return row * 2 * D + (((2 * j + (lane >> 5)) ^ k_swizzle<D>(row)) << 4);
}
// Byte offset of a lane's first read of the V operand (32 dims from dim 32 c x the
// first 16 keys): l16 its place in its group of 16, g1 the group's half of the
// dims, row = v_row(l16, lane / 32); the second read is eight rows on.
__device__ __forceinline__ int v_row(int l16, int half) { return 4 * half + (l16 >> 2); }
template <int D>
__device__ __forceinline__ uint32_t v_operand(int row, int l16, int g1, int c) {
  return row * 2 * D + (((4 * c + 2 * g1 + ((l16 & 3) >> 1)) ^ v_swizzle<D>(row)) << 4) + 8 * (l16 & 1);
}
// The two transposing reads of a V operand at LDS byte address `at`, rows of `row_bytes`.
__device__ __forceinline__ bf16x8 read_v(uint32_t at, int row_bytes) {
  using lds_s16x4 = __attribute__((address_space(3))) s16x4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)at);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(at + 8 * row_bytes));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

}  // namespace

// K/V blocks go from global memory straight into LDS (the lane picks which
// chunk it loads, see the swizzles above), double-buffered.
//
// What bounds it: the matrix cores are 51 % (head_dim 64) / 59 % (128) and the
// VALU 72 % / 47 % busy, without LDS bank conflicts, at a clock that falls to
// 1.5-1.8 GHz (2.3-2.5 GHz under the memory-bound kernels of the same run; all
// from counters), and variants that only move work around change little, so what
// counts is work per score.  32 rows per wave in 32x32 tiles keep two waves per
// SIMD at head_dim 128 and three at 64 (227 / 159 VGPRs); the direct LDS loads
// and the transposing reads take the V transposition and the staging registers
// away, one lane per query the softmax broadcasts, and v_dot2 the extra P . 1
// tile.  Measured against 16x16 tiles staged through registers (both in turn on
// one card; cards differ by a tenth): eight ragged prompts of 6 144 tokens on
// average, 32 / 8 heads, head_dim 64 1 690 -> 1 390 us (968 TFLOP/s), head_dim 128
// 3 197 -> 2 435 us (1 104); 4 096 queries over a 12 300 token prefix, head_dim 128
// 1 099 -> 843 us (1 142); 24 prompts of 400 tokens 46 -> 37 us.
// P.V delayed by a block (so that one straight-line region holds both products
// and the exponentials) measured +2 % / -0.5 %, and replacing the per-block max by
// a check of the running sum -2.7 % at head_dim 64 but +1 to +5 % at 128.
//
// Software pipeline over the blocks: iteration t holds S of block t, issues
// the loads of K(t + 2) and V(t + 1), multiplies K(t + 1) . Q^T beside the
// exponentials of block t, then V(t) . P beside the max of block t + 1.
// Softmax rescaling is lazy: the running max only moves (and O / the sum are
// rescaled) when a block raises it by more than 8 in the log2 domain, so p
// stays below 256.  The running max starts at a finite floor instead of -inf
// (the lowest fp32 whose product with the scale is still finite): the first
// block with a visible key then takes the same grow test as every later one,
// its rescale factor exp2((floor - m) * scale) is exactly 0, and a row whose
// keys so far all score -inf keeps the floor with p = 0.
// The running max is of raw scores, so the softmax scale has to be positive:
// the host hands over its magnitude, and its sign (0 for a scale of 0, with
// the magnitude 1) multiplies Q, exactly, as the rows are read.
//
// SUM32: the row sum is of the fp32 probabilities (group sizes other than 1, 2
// and 4, which keep the sum they always had) instead of the bf16 ones that the
// numerator multiplies, whose pairs v_dot2 adds in one instruction.  Four
// prompts of 3 000 tokens, 32 / 4 heads: head_dim 64 180 us against 183 with
// the bf16 sum, 128 302 against 305; 24 / 4 heads of 64 142 against 140.
template <int D, int G, bool SUM32>
__global__ __launch_bounds__(kThreads, 2) void prefill_attn_kernel(
    const bf16_t* __restrict__ q, int64_t qs_t, int64_t qs_h, const bf16_t* __restrict__ k, int64_t ks_t,
    int64_t ks_h, const bf16_t* __restrict__ v, int64_t vs_t, int64_t vs_h, bf16_t* __restrict__ out, int64_t os_t,
    int64_t os_h, const int32_t* __restrict__ cu_q, const int32_t* __restrict__ cu_k, int group, int vec_out,
    float scale_log2, float q_sign, float max_floor) {
  constexpr int P = 4 * kWaveRows / G;  // query positions per workgroup
  constexpr int RB = 2 * D;             // bytes of a K / V row
  constexpr int CH = D / 8;             // 16-byte chunks of a row
  constexpr int TILE = kKeys * RB;
  constexpr int RPI = 1024 / RB;        // rows one wave's LDS-DMA instruction moves
  constexpr int NI = kKeys / (4 * RPI);  // such instructions per wave and tile
  constexpr int KS = D / 16;            // MFMA steps of QK^T
  constexpr int DT = D / 32;            // 32-dim tiles of O^T
  __shared__ __attribute__((aligned(1024))) uint8_t s_kv[4 * TILE];  // K0, K1, V0, V1

  // block ids run over (head group, query block) with the head group fastest,
  // so with 8 KV heads every XCD (ids go round-robin over them) keeps one
  // head's K / V in its L2; a head's heaviest (diagonal-last) blocks go first
  const int seq = blockIdx.z;
  const uint32_t lin = blockIdx.x + gridDim.x * blockIdx.y;
  const int hg = (int)(lin % gridDim.y), qb = (int)(lin / gridDim.y);
  // query rows are the last len of the klen keys (bottom-right causal
  // alignment): row i is position off + i and sees keys 0 .. off + i
  const int start = cu_q[seq];
  const int len = cu_q[seq + 1] - start;
  const int kstart = cu_k[seq];
  const int klen = cu_k[seq + 1] - kstart;
  const int off = klen - len;
  if (off < 0) return;  // rejected: more queries than keys
  const int nqb = (len + P - 1) / P;
  if (qb >= nqb) return;
  const int q0 = (nqb - 1 - qb) * P;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int lc = lane & 31, half = lane >> 5;
  const int qh = hg * G + wave % G;
  const int kvh = (hg * G) / group;
  const int wq0 = q0 + (wave / G) * kWaveRows;  // first position of this wave
  // blocks the workgroup loads, this wave sees, and every row of it sees whole
  // (the others need the mask); a wave past the sequence only loads its share
  const PrefillBlocks blocks = prefill_blocks(len, klen, q0, P, wq0);
  const int nkb = blocks.loaded, nw = blocks.seen, nfull = blocks.whole;

  const uint8_t* kbase = reinterpret_cast<const uint8_t*>(k + (int64_t)kstart * ks_t + (int64_t)kvh * ks_h);
  const uint8_t* vbase = reinterpret_cast<const uint8_t*>(v + (int64_t)kstart * vs_t + (int64_t)kvh * vs_h);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)s_kv;
  // this lane's part of an LDS-DMA instruction: row drow (+ 4 * RPI * i), the
  // chunk whose swizzled slot is lane % CH
  const int drow = wave * RPI + lane / CH;
  const int kchunk = (lane % CH) ^ k_swizzle<D>(drow);
  const int vchunk = (lane % CH) ^ v_swizzle<D>(drow);
  const uint32_t ksb = (uint32_t)(ks_t * 2), vsb = (uint32_t)(vs_t * 2);  // row strides in bytes
  auto load_tile = [&](const uint8_t* base, uint32_t stride, int chunk, int blk, uint32_t lds) {
    const int k0 = blk * kKeys;
    const uint8_t* b = base + (int64_t)k0 * stride;
    const int last = klen - 1 - k0;  // rows past the sequence end repeat its last (their scores are masked)
#pragma unroll
    for (int i = 0; i < NI; ++i)
      lds_dma16(b, (uint32_t)min(drow + 4 * RPI * i, last) * stride + 16 * chunk,
                lds + (uint32_t)((i * 4 + wave) * 1024));
  };
  auto load_k = [&](int blk, int buf) { load_tile(kbase, ksb, kchunk, blk, lds0 + buf * TILE); };
  auto load_v = [&](int blk, int buf) { load_tile(vbase, vsb, vchunk, blk, lds0 + (2 + buf) * TILE); };

  load_k(0, 0);
  load_v(0, 0);
  if (nkb > 1) load_k(1, 1);
  bf16x8 qop[KS];
  {
    const int qrow = min(wq0 + lc, len - 1);
    const bf16_t* qp = q + (int64_t)(start + qrow) * qs_t + (int64_t)qh * qs_h + 8 * half;
#pragma unroll
    for (int j = 0; j < KS; ++j) qop[j] = as_bf16x8(*reinterpret_cast<const uint4*>(qp + 16 * j));
    if (q_sign != 1.0f) {  // uniform
#pragma unroll
      for (int j = 0; j < KS; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) qop[j][i] = (__bf16)((float)qop[j][i] * q_sign);
    }
  }
  // LDS byte offsets of this lane's operands (buffer, key tile and key step
  // are added as constants)
  uint32_t kaddr[KS], vaddr[DT];
#pragma unroll
  for (int j = 0; j < KS; ++j) kaddr[j] = k_operand<D>(lane, j);
  {
    const int l16 = lane & 15, g1 = (lane >> 4) & 1;
    const int vr = v_row(l16, half);
#pragma unroll
    for (int c = 0; c < DT; ++c) vaddr[c] = v_operand<D>(vr, l16, g1, c);
  }

  float m_run = max_floor;  // raw-score running max of this lane's query (see the rescale note above)
  float l_run = 0.0f;       // this half's share of its row sum
  f32x16 o[DT];
#pragma unroll
  for (int c = 0; c < DT; ++c) o[c] = f32x16{};
  f32x16 s0[2], s1[2];
  const int lim = off + min(wq0 + lc, len - 1) - 4 * half;  // last visible key - 4 * half

  auto qk = [&](f32x16 (&sx)[2], int buf) {
    const uint8_t* kt = s_kv + buf * TILE;
    sx[0] = sx[1] = f32x16{};
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      const bf16x8 a0 = as_bf16x8(*reinterpret_cast<const uint4*>(kt + kaddr[j]));
      const bf16x8 a1 = as_bf16x8(*reinterpret_cast<const uint4*>(kt + 32 * RB + kaddr[j]));
      sx[0] = mfma32x32x16(a0, qop[j], sx[0]);
      sx[1] = mfma32x32x16(a1, qop[j], sx[1]);
    }
  };
  auto mask = [&](f32x16 (&sx)[2], int blk) {
    const int rel = lim - blk * kKeys;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) sx[t][r] = 32 * t + 8 * (r / 4) + r % 4 > rel ? -INFINITY : sx[t][r];
  };
  // NaN-propagating max (one instruction per two scores): a row with a NaN
  // score is NaN whatever its max is
  auto row_max = [&](const f32x16 (&sx)[2]) {
    float b0 = __builtin_elementwise_maximum(sx[0][0], sx[1][0]);
    float b1 = __builtin_elementwise_maximum(sx[0][1], sx[1][1]);
#pragma unroll
    for (int r = 2; r < 16; r += 2) {
      b0 = __builtin_elementwise_maximum(__builtin_elementwise_maximum(b0, sx[0][r]), sx[1][r]);
      b1 = __builtin_elementwise_maximum(__builtin_elementwise_maximum(b1, sx[0][r + 1]), sx[1][r + 1]);
    }
    return halves_max(__builtin_elementwise_maximum(b0, b1));
  };
  auto rescale = [&](float bmax) {
    // lazy: move the max only when it grows by more than 2^8 in p
    const bool grow = (bmax - m_run) * scale_log2 > 8.0f;  // bmax = -inf (all masked): false
    if (__builtin_amdgcn_ballot_w64(grow)) {               // wave-uniform
      const float m_new = fmaxf(m_run, bmax);
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2);  // 0 from the floor
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int c = 0; c < DT; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[c][r] *= alpha;
    }
  };
  // p of block t as the B operands of its four 16-key steps, and their sum
  auto probs = [&](const f32x16 (&sx)[2], uint4 (&pb)[4]) {
    const float mb = m_run * scale_log2;
    const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 8 * (st & 1) + 2 * i;
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sx[st >> 1][r], scale_log2, -mb));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sx[st >> 1][r + 1], scale_log2, -mb));
        w[i] = cvt_pk_bf16(p0, p1);
        if constexpr (SUM32)
          l_run += p0 + p1;
        else
          l_run = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w[i]), one, l_run, false);
      }
      pb[st] = uint4{w[0], w[1], w[2], w[3]};
    }
  };
  auto pv = [&](const uint4 (&pb)[4], int buf) {
    const uint32_t vt = lds0 + (2 + buf) * TILE;
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int c = 0; c < DT; ++c)
        o[c] = mfma32x32x16(read_v(vt + vaddr[c] + (16 * st) * RB, RB), as_bf16x8(pb[st]), o[c]);
  };

  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), known to the compiler: Q has landed, no use of it waits again
  lds_dma_barrier();
  if (nw > 0) {
    qk(s0, 0);
    if (nfull < 1) mask(s0, 0);
    rescale(row_max(s0));
  }
  lds_dma_barrier();  // K(0) has been read by every wave: its buffer takes K(2)
  // B = t & 1; cur = S(t), nxt receives S(t + 1)
  auto full = [&](int t, auto parity, f32x16 (&cur)[2], f32x16 (&nxt)[2]) {
    constexpr int B = decltype(parity)::value;
    uint4 pb[4];
    qk(nxt, 1 - B);
    probs(cur, pb);
    pv(pb, B);
    rescale(row_max(nxt));
  };
  auto loads = [&](int t, auto parity) {
    constexpr int B = decltype(parity)::value;
    if (t + 2 < nkb) load_k(t + 2, B);
    if (t + 1 < nkb) load_v(t + 1, 1 - B);
  };
  auto iteration = [&](int t, auto parity, f32x16 (&cur)[2], f32x16 (&nxt)[2]) {
    constexpr int B = decltype(parity)::value;
    loads(t, parity);
    if (t < nw) {  // wave-uniform, as the branch below
      uint4 pb[4];
      probs(cur, pb);
      pv(pb, B);
      if (t + 1 < nw) {
        qk(nxt, 1 - B);
        mask(nxt, t + 1);
        rescale(row_max(nxt));
      }
    }
    if (t + 1 < nkb) lds_dma_barrier();
  };
  const std::integral_constant<int, 0> even{};
  const std::integral_constant<int, 1> odd{};
  int t = 0;
  for (; t + 2 < nfull; t += 2) {
    loads(t, even);
    full(t, even, s0, s1);
    lds_dma_barrier();
    loads(t + 1, odd);
    full(t + 1, odd, s1, s0);
    lds_dma_barrier();
  }
  for (; t < nkb; t += 2) {
    iteration(t, even, s0, s1);
    if (t + 1 < nkb) iteration(t + 1, odd, s1, s0);
  }

  const float inv = 1.0f / halves_sum(l_run);
  const int row = wq0 + lc;
  // lane (lc, half) holds dims 32 c + 8 g + 4 half + 0 .. 3 of its query in o[c][4 g ..]
  bf16_t* op = out + (int64_t)(start + min(row, len - 1)) * os_t + (int64_t)qh * os_h;
#pragma unroll
  for (int c = 0; c < DT; ++c) {
    uint32_t w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = cvt_pk_bf16(o[c][2 * i] * inv, o[c][2 * i + 1] * inv);
    if (vec_out) {  // uniform: 16-byte rows; the halves swap quads so that a lane stores 8 dims at once
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const auto x = __builtin_amdgcn_permlane32_swap(w[4 * m], w[4 * m + 2], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(w[4 * m + 1], w[4 * m + 3], false, false);
        if (row < len)
          *reinterpret_cast<uint4*>(op + 32 * c + 16 * m + 8 * half) = uint4{x[0], y[0], x[1], y[1]};
      }
    } else if (row < len) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int d = 32 * c + 8 * (i / 2) + 4 * half + 2 * (i & 1);
        op[d].bits = (uint16_t)w[i];
        op[d + 1].bits = (uint16_t)(w[i] >> 16);
      }
    }
  }
}

FDMS_EXPORT int fdms_prefill_attention_varlen(const void* q, int64_t qs_t, int64_t qs_h, const void* k,
                                              int64_t ks_t, int64_t ks_h, const void* v, int64_t vs_t, int64_t vs_h,
                                              void* out, int64_t os_t, int64_t os_h, const int32_t* cu_seqlens_q,
                                              const int32_t* cu_seqlens_k, int num_seqs, int max_seqlen_q,
                                              int num_q_heads, int num_kv_heads, int head_dim, float scale,
                                              void* stream) {
  if (num_seqs < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads) return (int)hipErrorInvalidValue;
  if (num_seqs == 0 || max_seqlen_q <= 0) return 0;
  if (!q || !k || !v || !out || !cu_seqlens_q || !cu_seqlens_k) return (int)hipErrorInvalidValue;
  if (num_seqs > 65535 || num_q_heads > 65535) return (int)hipErrorInvalidValue;
  // token strides in elements: 64 rows of either stay in 32-bit byte offsets
  if (ks_t < 0 || vs_t < 0 || ks_t >= (1 << 24) || vs_t >= (1 << 24)) return (int)hipErrorInvalidValue;
  if (head_dim != 64 && head_dim != 128) return (int)hipErrorInvalidValue;
  const float signed_sl2 = scale * 1.4426950408889634f;
  const float q_sign = signed_sl2 < 0.0f ? -1.0f : signed_sl2 == 0.0f ? 0.0f : 1.0f;
  const float sl2 = signed_sl2 == 0.0f ? 1.0f : signed_sl2 * q_sign;
  const float max_floor = sl2 > 1.0f ? -0x1p127f / sl2 : -FLT_MAX;
  const int group = num_q_heads / num_kv_heads;
  const int packed = group == 2 || group == 4 ? group : 1;  // query heads per workgroup
  const int pos = 4 * kWaveRows / packed;                   // query positions per workgroup
  const int vec_out = ((uintptr_t)out % 16) == 0 && os_t % 8 == 0 && os_h % 8 == 0;
  const dim3 grid((unsigned)((max_seqlen_q + pos - 1) / pos), (unsigned)(num_q_heads / packed), (unsigned)num_seqs);
#define FDMS_PREFILL(DD, ...)                                                                                      \
  hipLaunchKernelGGL((prefill_attn_kernel<DD, __VA_ARGS__>), grid, dim3(kThreads), 0, (hipStream_t)stream,            \
                     (const bf16_t*)q, qs_t, qs_h, (const bf16_t*)k, ks_t, ks_h, (const bf16_t*)v, vs_t,      \
                     vs_h, (bf16_t*)out, os_t, os_h, cu_seqlens_q, cu_seqlens_k, group, vec_out, sl2, q_sign, max_floor)
#define FDMS_PREFILL_GROUP(DD)                                                                                     \
  do {                                                                                                             \
    if (group == 1) FDMS_PREFILL(DD, 1, false); else if (group == 2) FDMS_PREFILL(DD, 2, false);                   \
    else if (group == 4) FDMS_PREFILL(DD, 4, false); else FDMS_PREFILL(DD, 1, true);                               \
  } while (0)
  if (head_dim == 64) FDMS_PREFILL_GROUP(64); else FDMS_PREFILL_GROUP(128);
#undef FDMS_PREFILL_GROUP
#undef FDMS_PREFILL
  FDMS_LAUNCH_CHECK();
  return 0;
}

FDMS_EXPORT int fdms_prefill_attention(const void* q, int64_t qs_t, int64_t qs_h, const void* k, int64_t ks_t,
                                       int64_t ks_h, const void* v, int64_t vs_t, int64_t vs_h, void* out,
                                       int64_t os_t, int64_t os_h, const int32_t* cu_seqlens, int num_seqs,
                                       int max_seqlen, int num_q_heads, int num_kv_heads, int head_dim, float scale,
                                       void* stream) {
  return fdms_prefill_attention_varlen(q, qs_t, qs_h, k, ks_t, ks_h, v, vs_t, vs_h, out, os_t, os_h, cu_seqlens,
                                       cu_seqlens, num_seqs, max_seqlen, num_q_heads, num_kv_heads, head_dim, scale,
                                       stream);
}

// One v_mfma_f32_16x16x32_bf16 of a 16x32 A and a 32x16 B (row-major bf16)
// loaded with the operand layout the decode linears assume; C row-major fp32.
// Exists so a test can confirm that layout against a host matmul.
__global__ void mfma_probe_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ b, float* __restrict__ c) {
  const int l = threadIdx.x;
  uint16_t av[8], bv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    av[i] = a[(l % 16) * 32 + 8 * (l / 16) + i].bits;
    bv[i] = b[(8 * (l / 16) + i) * 16 + (l % 16)].bits;
  }
  uint4 ua, ub;
  __builtin_memcpy(&ua, av, 16);
  __builtin_memcpy(&ub, bv, 16);
  const f32x4 r = mfma16x16x32(as_bf16x8(ua), as_bf16x8(ub), f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
  for (int i = 0; i < 4; ++i) c[(4 * (l / 16) + i) * 16 + (l % 16)] = r[i];
}

FDMS_EXPORT int fdms_mfma_probe(const void* a, const void* b, float* c, void* stream) {
  if (!a || !b || !c) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, (const bf16_t*)a,
                     (const bf16_t*)b, c);
  FDMS_LAUNCH_CHECK();
  return 0;
}

// The prefill kernel's two products through its own operand addresses: S^T [32
// keys, 32 queries] = K . Q^T of k, q [32, D], and O [32 queries, D] = P . V of p
// [32 queries, 16 keys], v [16 keys, D], V read transposed in the permuted key
// order.  One wave; exists so a test can confirm the layouts against host matmuls.
template <int D>
__global__ void prefill_mfma_probe_kernel(const bf16_t* __restrict__ k, const bf16_t* __restrict__ q,
                                          float* __restrict__ s, const bf16_t* __restrict__ p,
                                          const bf16_t* __restrict__ v, float* __restrict__ o) {
  constexpr int RB = 2 * D, CH = D / 8;
  __shared__ __attribute__((aligned(1024))) uint8_t s_k[32 * RB], s_v[16 * RB];
  const int lane = threadIdx.x, lc = lane & 31, half = lane >> 5;
  for (int u = lane; u < 32 * CH; u += kWave)
    *reinterpret_cast<uint4*>(s_k + (u / CH) * RB + (((u % CH) ^ k_swizzle<D>(u / CH)) << 4)) =
        reinterpret_cast<const uint4*>(k)[u];
  for (int u = lane; u < 16 * CH; u += kWave)
    *reinterpret_cast<uint4*>(s_v + (u / CH) * RB + (((u % CH) ^ v_swizzle<D>(u / CH)) << 4)) =
        reinterpret_cast<const uint4*>(v)[u];
  __syncthreads();
  f32x16 acc{};
  for (int j = 0; j < D / 16; ++j)
    acc = mfma32x32x16(as_bf16x8(*reinterpret_cast<const uint4*>(s_k + k_operand<D>(lane, j))),
                       as_bf16x8(*reinterpret_cast<const uint4*>(q + lc * D + 16 * j + 8 * half)), acc);
#pragma unroll
  for (int r = 0; r < 16; ++r) s[(8 * (r / 4) + 4 * half + r % 4) * 32 + lc] = acc[r];
  uint16_t pv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) pv[i] = p[lc * 16 + 8 * (i / 4) + 4 * half + i % 4].bits;
  uint4 pb;
  __builtin_memcpy(&pb, pv, 16);
  const uint32_t vt = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)s_v;
  const int l16 = lane & 15, g1 = (lane >> 4) & 1;
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    const uint32_t at = vt + v_operand<D>(v_row(l16, half), l16, g1, c);
    acc = mfma32x32x16(read_v(at, RB), as_bf16x8(pb), f32x16{});
#pragma unroll
    for (int r = 0; r < 16; ++r) o[lc * D + 32 * c + 8 * (r / 4) + 4 * half + r % 4] = acc[r];
  }
}

FDMS_EXPORT int fdms_prefill_mfma_probe(int head_dim, const void* k, const void* q, float* s, const void* p,
                                        const void* v, float* o, void* stream) {
  if (!k || !q || !s || !p || !v || !o || (head_dim != 64 && head_dim != 128) || !fdms_aligned16(k, q, v))
    return (int)hipErrorInvalidValue;
  if (head_dim == 64)
    hipLaunchKernelGGL(prefill_mfma_probe_kernel<64>, dim3(1), dim3(kWave), 0, (hipStream_t)stream, (const bf16_t*)k,
                       (const bf16_t*)q, s, (const bf16_t*)p, (const bf16_t*)v, o);
  else
    hipLaunchKernelGGL(prefill_mfma_probe_kernel<128>, dim3(1), dim3(kWave), 0, (hipStream_t)stream, (const bf16_t*)k,
                       (const bf16_t*)q, s, (const bf16_t*)p, (const bf16_t*)v, o);
  FDMS_LAUNCH_CHECK();
  return 0;
}
