// Element-wise model ops around the DMS path, fused so a decode layer issues
// few launches: residual-add + RMSNorm (reference layernorm.py:16-40) and
// SiLU(gate) * up (activation.py:8-11).  bf16 in/out, fp32 math; one block
// per row, 16-byte vector loads.  HBM-bound: 2-3 bf16 reads + 2 writes per
// element.
#include "fdms_vec.h"

using namespace fdms;

namespace {
constexpr int kThreads = 256;
constexpr int kSiluUnits = 4;  // 8-column units per thread of a large silu_mul

__device__ __forceinline__ float block_sum(float v, float* s_red) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_red[w] = v;
  __syncthreads();
  float t = 0.0f;
#pragma unroll
  for (int i = 0; i < kThreads / kWave; ++i) t += s_red[i];
  __syncthreads();
  return t;
}
// Two fp32 -> bf16 (round to nearest even) in one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  const bf16x2_t r = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, float* s_red) {
  v = wave_max_u32(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_red[w] = __uint_as_float(v);
  __syncthreads();
  uint32_t t = 0;
#pragma unroll
  for (int i = 0; i < kThreads / kWave; ++i) t = max(t, __float_as_uint(s_red[i]));
  __syncthreads();
  return t;
}
}  // namespace

// x_out = bf16(bf16(x * rsqrt(mean(x^2) + eps)) * w), where x = in (+ residual
// in fp32, and residual_out = bf16(x)) — layernorm.py:19-40.
// PART: the input is the fp32 split-K partial sums of the preceding linear,
// part[s * split_stride + row * hidden + c], s < k_splits, and x = bf16 of
// their sum taken in split order (the linear kernel's own merge).
// PART: the input is the fp32 split-K partials; KS > 0 is their count known
// at compile time, KS = 0 reads k_splits at run time.  With row_scale /
// col_scale (an FP8 linear's 1/x_s[row] and weight scale_inv[c]) the input is
// x = bf16(sum * row_scale[row] * col_scale[c]), the linear's own finalisation.
// amax_out[row] (optional) = max |out[row, :]| (NaN if the row holds one), the
// statistic the next FP8 linear's activation quantisation needs; q_out
// (optional, with amax_out) receives that quantisation itself, e4m3fn(out *
// s) with s = 448 / amax (q_mode 2: the torch rounding), and out may then be
// null.  PER = 8-column chunks
// per thread (hidden <= PER * 8 * kThreads).  Every load of the row goes out
// before the first use, with addresses clamped in bounds instead of loads
// under a condition (a conditional load makes the compiler wait for it at
// the end of its block, one memory round trip per load).
template <bool PART, int KS, int PER>
__global__ __launch_bounds__(kThreads) void rmsnorm_kernel(const bf16_t* __restrict__ in, const bf16_t* residual,
                                                           const bf16_t* __restrict__ weight, bf16_t* __restrict__ out,
                                                           bf16_t* residual_out, int hidden, int64_t in_stride,
                                                           int64_t in_head_stride, int heads, int64_t out_stride,
                                                           float eps, const float* __restrict__ part, int k_splits,
                                                           int64_t split_stride, const float* __restrict__ row_scale,
                                                           const float* __restrict__ col_scale,
                                                           float* __restrict__ amax_out, uint8_t* __restrict__ q_out,
                                                           int64_t q_stride, int q_mode,
                                                           const int64_t* __restrict__ ids, int64_t vocab) {
  __shared__ float s_red[kThreads / kWave];
  const int64_t row = blockIdx.x;
  // ids (optional, embedding rows): input row r is table row ids[r] (in_stride
  // per row); an id outside [0, vocab) reads row 0 and yields NaN rows
  const int64_t id = ids ? ids[row] : 0;
  const bool id_ok = !ids || (id >= 0 && id < vocab);
  const bf16_t* x = PART ? nullptr
                         : ids ? in + (id_ok ? id : 0) * in_stride
                               : in + (row / heads) * in_stride + (row % heads) * in_head_stride;
  const bool has_res = residual != nullptr;  // uniform
  const bf16_t* rs = has_res ? residual + row * (int64_t)hidden : weight;  // a valid address either way
  constexpr int V = 8;
  constexpr int NS = KS > 0 ? KS : 1;
  Vec<bf16_t, V> wv[PER], xv[PER], rv[PER];
  Vec<float, V> pv[PER][NS], cs[PER];
  const float* csrc = (PART && col_scale) ? col_scale : part;  // a valid address either way (PART)
  const float rscale = (PART && row_scale) ? row_scale[row] : 1.0f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int cc = min(((int)threadIdx.x + j * kThreads) * V, hidden - V);  // int min (an unsigned operand picks the double overload)
    wv[j] = *reinterpret_cast<const Vec<bf16_t, V>*>(weight + cc);
    if constexpr (PART) cs[j] = *reinterpret_cast<const Vec<float, V>*>(csrc + cc);
    if constexpr (PART && KS > 0) {
#pragma unroll
      for (int sp = 0; sp < KS; ++sp)
        pv[j][sp] = *reinterpret_cast<const Vec<float, V>*>(part + sp * split_stride + row * hidden + cc);
    }
    if constexpr (!PART) xv[j] = *reinterpret_cast<const Vec<bf16_t, V>*>(x + cc);
    rv[j] = *reinterpret_cast<const Vec<bf16_t, V>*>(rs + cc);
  }
  float vals[PER][V];
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int c = (threadIdx.x + j * kThreads) * V;
    const bool valid = c < hidden;
    float xf[V];
    if constexpr (PART) {
#pragma unroll
      for (int i = 0; i < V; ++i) xf[i] = 0.0f;
      if constexpr (KS > 0) {
#pragma unroll
        for (int sp = 0; sp < KS; ++sp)
#pragma unroll
          for (int i = 0; i < V; ++i) xf[i] += pv[j][sp].v[i];
      } else if (valid) {
        for (int sp = 0; sp < k_splits; ++sp) {
          const Vec<float, V> p = *reinterpret_cast<const Vec<float, V>*>(part + sp * split_stride + row * hidden + c);
#pragma unroll
          for (int i = 0; i < V; ++i) xf[i] += p.v[i];
        }
      }
      if (row_scale) {
#pragma unroll
        for (int i = 0; i < V; ++i) xf[i] *= rscale;
      }
      if (col_scale) {
#pragma unroll
        for (int i = 0; i < V; ++i) xf[i] *= cs[j].v[i];
      }
#pragma unroll
      for (int i = 0; i < V; ++i) xf[i] = bf16_to_f32(f32_to_bf16(xf[i]));
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) xf[i] = id_ok ? bf16_to_f32(xv[j].v[i].bits) : __builtin_nanf("");
    }
#pragma unroll
    for (int i = 0; i < V; ++i) {
      float f = xf[i];
      if (has_res) f += bf16_to_f32(rv[j].v[i].bits);
      vals[j][i] = f;
      ss += valid ? f * f : 0.0f;
    }
    if (residual_out && valid) {
      Vec<bf16_t, V> ro;
#pragma unroll
      for (int i = 0; i < V; ++i) ro.v[i].bits = (uint16_t)f32_to_bf16(vals[j][i]);
      *reinterpret_cast<Vec<bf16_t, V>*>(residual_out + row * (int64_t)hidden + c) = ro;
    }
  }
  const float total = block_sum(ss, s_red);
  const float inv = rsqrtf(total / (float)hidden + eps);  // torch.rsqrt (layernorm.py:24, 38)
  uint32_t amax = 0;
  float ov[PER][V];  // the bf16 outputs as fp32
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int c = (threadIdx.x + j * kThreads) * V;
    Vec<bf16_t, V> o;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const float xn = bf16_to_f32(f32_to_bf16(vals[j][i] * inv));
      o.v[i].bits = (uint16_t)f32_to_bf16(xn * bf16_to_f32(wv[j].v[i].bits));
      ov[j][i] = bf16_to_f32(o.v[i].bits);
      if (c < hidden) amax = max(amax, abs_bits(ov[j][i]));
    }
    if (out && c < hidden) *reinterpret_cast<Vec<bf16_t, V>*>(out + row * out_stride + c) = o;
  }
  if (amax_out) {  // uniform
    amax = block_max_u32(amax, s_red);
    const float a = __uint_as_float(amax);
    if (threadIdx.x == 0) amax_out[row] = a;
    if (q_out) {
      const float qs = fp8_row_scale(a, q_mode == 2);
      const bool finite = fp8_row_finite(a, qs);
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const int c = (threadIdx.x + j * kThreads) * V;
        if (c < hidden) {
          uint32_t w[V / 4];
#pragma unroll
          for (int i = 0; i < V / 4; ++i) {
            const float* f = &ov[j][4 * i];
            w[i] = finite ? f32x4_to_fp8x4_finite(f[0] * qs, f[1] * qs, f[2] * qs, f[3] * qs)
                          : f32x4_to_fp8x4_sw(f[0] * qs, f[1] * qs, f[2] * qs, f[3] * qs);
          }
          *reinterpret_cast<uint2*>(q_out + row * q_stride + c) = uint2{w[0], w[1]};
        }
      }
    }
  }
}

// Row r of the input is at in + (r / heads) * in_stride + (r % heads) * in_head_stride
// (heads = 1 for plain rows; heads > 1 normalises every head of a strided
// [tokens, heads, head_dim] view, as Qwen3's q_norm / k_norm do).  Output row r
// is at out + r * out_stride; residual / residual_out are contiguous rows.
// Short rows (hidden = 8 T, T = 4 .. 64 lanes, e.g. Qwen3's per-head q / k
// norms at head_dim 128): T lanes per row, 256 / T rows per workgroup, the
// row's sum of squares a segmented wave reduction; the same formula as
// rmsnorm_kernel, without residual or quantised outputs.  (One 256-thread
// workgroup per 128-element head row left 15 of 16 threads idle and launched
// millions of workgroups per prefill layer.)
template <int T>
__global__ __launch_bounds__(kThreads) void rmsnorm_rows_kernel(const bf16_t* __restrict__ in, int64_t in_stride,
                                                                int64_t in_head_stride, int heads,
                                                                const bf16_t* __restrict__ weight,
                                                                bf16_t* __restrict__ out, int64_t out_stride,
                                                                int64_t rows, float eps) {
  constexpr int kRows = kThreads / T;
  const int64_t r = (int64_t)blockIdx.x * kRows + threadIdx.x / T;
  const int c = (threadIdx.x % T) * 8;
  const bool ok = r < rows;
  Vec<bf16_t, 8> xv{};
  if (ok) {
    const int64_t tok = r / heads, hd = r - tok * heads;
    xv = *reinterpret_cast<const Vec<bf16_t, 8>*>(in + tok * in_stride + hd * in_head_stride + c);
  }
  float xf[8];
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    xf[i] = bf16_to_f32(xv.v[i].bits);
    ss += xf[i] * xf[i];
  }
  ss = segment_sum<T>(ss);  // every lane, rows past the end included
  if (!ok) return;
  const float inv = rsqrtf(ss / (float)(8 * T) + eps);  // torch.rsqrt (layernorm.py:24, 38)
  const Vec<bf16_t, 8> wv = *reinterpret_cast<const Vec<bf16_t, 8>*>(weight + c);
  Vec<bf16_t, 8> o;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float xn = bf16_to_f32(f32_to_bf16(xf[i] * inv));
    o.v[i].bits = (uint16_t)f32_to_bf16(xn * bf16_to_f32(wv.v[i].bits));
  }
  *reinterpret_cast<Vec<bf16_t, 8>*>(out + r * out_stride + c) = o;
}

FDMS_EXPORT int fdms_rmsnorm(const void* in, int64_t in_stride, int64_t in_head_stride, int heads,
                             const void* residual, const void* weight, void* out, int64_t out_stride,
                             void* residual_out, int64_t rows, int hidden, float eps, float* amax_out,
                             void* q_out, int64_t q_stride, int q_mode, void* stream) {
  if (rows < 0 || hidden <= 0 || hidden % 8 || hidden > 8 * kThreads * 4 || heads <= 0) return (int)hipErrorInvalidValue;
  if (heads > 1 && (residual || residual_out)) return (int)hipErrorInvalidValue;
  if (q_out && (!amax_out || q_mode < 1 || q_mode > 2 || q_stride < hidden || q_stride % 8 || (uintptr_t)q_out % 8))
    return (int)hipErrorInvalidValue;
  if (rows == 0) return 0;
  if (!in || !weight || (!out && !q_out) || rows > 0x7FFFFFFF) return (int)hipErrorInvalidValue;
  // rows move as 16-byte vectors
  if (!fdms_aligned16(in, weight, out, residual, residual_out) || (in_stride | in_head_stride | out_stride) % 8)
    return (int)hipErrorInvalidValue;
  const int lanes = hidden / 8;
  if (!residual && !residual_out && !amax_out && !q_out && hidden <= 512 && lanes >= 4 && !(lanes & (lanes - 1))) {
    const int64_t blocks = (rows * lanes + kThreads - 1) / kThreads;
#define FDMS_RMSNORM_ROWS(TV)                                                                                   \
  hipLaunchKernelGGL((rmsnorm_rows_kernel<TV>), dim3((unsigned)blocks), dim3(kThreads), 0, (hipStream_t)stream,  \
                     (const bf16_t*)in, in_stride, in_head_stride, heads, (const bf16_t*)weight, (bf16_t*)out,       \
                     out_stride, rows, eps)
    switch (lanes) {
      case 4: FDMS_RMSNORM_ROWS(4); break;
      case 8: FDMS_RMSNORM_ROWS(8); break;
      case 16: FDMS_RMSNORM_ROWS(16); break;
      case 32: FDMS_RMSNORM_ROWS(32); break;
      default: FDMS_RMSNORM_ROWS(64); break;
    }
#undef FDMS_RMSNORM_ROWS
    FDMS_LAUNCH_CHECK();
    return 0;
  }
#define FDMS_RMSNORM(PERV)                                                                                      \
  hipLaunchKernelGGL((rmsnorm_kernel<false, 0, PERV>), dim3((unsigned)rows), dim3(kThreads), 0,                  \
                     (hipStream_t)stream, (const bf16_t*)in, (const bf16_t*)residual, (const bf16_t*)weight,        \
                     (bf16_t*)out, (bf16_t*)residual_out, hidden, in_stride, in_head_stride, heads, out_stride, eps, \
                     nullptr, 0, (int64_t)0, nullptr, nullptr, amax_out, (uint8_t*)q_out, q_stride, q_mode, nullptr,    \
                     (int64_t)0)
  const int per = (hidden + 8 * kThreads - 1) / (8 * kThreads);
  if (per == 1) FDMS_RMSNORM(1);
  else if (per == 2) FDMS_RMSNORM(2);
  else FDMS_RMSNORM(4);
#undef FDMS_RMSNORM
  FDMS_LAUNCH_CHECK();
  return 0;
}

// RMSNorm (+ residual) of x = bf16(sum of the k_splits fp32 partials
// partials[s * split_stride + r * hidden + c]) -- the consumer side of
// fdms_linear_small_m's epilogue 3.  residual / residual_out contiguous rows.
FDMS_EXPORT int fdms_rmsnorm_partials(const float* partials, int k_splits, int64_t split_stride,
                                      const void* residual, const void* weight, void* out, int64_t out_stride,
                                      void* residual_out, int64_t rows, int hidden, float eps,
                                      const float* row_scale, const float* col_scale, float* amax_out,
                                      void* q_out, int64_t q_stride, int q_mode, void* stream) {
  if (rows < 0 || hidden <= 0 || hidden % 8 || hidden > 8 * kThreads * 4 || k_splits < 1) return (int)hipErrorInvalidValue;
  if (q_out && (!amax_out || q_mode < 1 || q_mode > 2 || q_stride < hidden || q_stride % 8 || (uintptr_t)q_out % 8))
    return (int)hipErrorInvalidValue;
  if (rows == 0) return 0;
  if (!partials || !weight || (!out && !q_out) || rows > 0x7FFFFFFF || split_stride < rows * (int64_t)hidden)
    return (int)hipErrorInvalidValue;
  if ((uintptr_t)partials % 32 || split_stride % 8 || (uintptr_t)col_scale % 32) return (int)hipErrorInvalidValue;
  if (!fdms_aligned16(weight, out, residual, residual_out) || out_stride % 8) return (int)hipErrorInvalidValue;
#define FDMS_RMSNORM_PART(KSV, PERV)                                                                              \
  hipLaunchKernelGGL((rmsnorm_kernel<true, KSV, PERV>), dim3((unsigned)rows), dim3(kThreads), 0,                   \
                     (hipStream_t)stream, nullptr, (const bf16_t*)residual, (const bf16_t*)weight, (bf16_t*)out,      \
                     (bf16_t*)residual_out, hidden, (int64_t)0, (int64_t)0, 1, out_stride, eps, partials, k_splits,   \
                     split_stride, row_scale, col_scale, amax_out, (uint8_t*)q_out, q_stride, q_mode, nullptr,        \
                     (int64_t)0)
#define FDMS_RMSNORM_PART_PER(PERV)                   \
  if (k_splits == 1) FDMS_RMSNORM_PART(1, PERV);      \
  else if (k_splits == 2) FDMS_RMSNORM_PART(2, PERV); \
  else if (k_splits == 4) FDMS_RMSNORM_PART(4, PERV); \
  else if (k_splits == 8) FDMS_RMSNORM_PART(8, PERV); \
  else FDMS_RMSNORM_PART(0, PERV)
  const int per = (hidden + 8 * kThreads - 1) / (8 * kThreads);
  if (per == 1) {
    FDMS_RMSNORM_PART_PER(1);
  } else if (per == 2) {
    FDMS_RMSNORM_PART_PER(2);
  } else {
    FDMS_RMSNORM_PART_PER(4);
  }
#undef FDMS_RMSNORM_PART_PER
#undef FDMS_RMSNORM_PART
  FDMS_LAUNCH_CHECK();
  return 0;
}

// Embedding gather + RMSNorm of the gathered rows in one launch (the decode
// step's first layer: F.embedding, embed_head.py:87-104, then the first
// input_layernorm without residual, layernorm.py:16-28): rows_out[i] =
// table[ids[i]] (the first residual), out[i] = RMSNorm(rows_out[i]), the same
// bits as fdms_rmsnorm of the gathered rows.  An id outside [0, vocab) gives
// NaN rows in both (the reference's index_select raises there).
FDMS_EXPORT int fdms_embedding_rmsnorm(const int64_t* ids, int64_t n, const void* table, int64_t table_stride,
                                       int64_t vocab, const void* weight, float eps, void* out, int64_t out_stride,
                                       void* rows_out, int64_t rows_stride, int hidden, void* stream) {
  if (n < 0 || hidden <= 0 || hidden % 8 || hidden > 8 * kThreads * 4 || vocab <= 0) return (int)hipErrorInvalidValue;
  if (n == 0) return 0;
  if (!ids || !table || !weight || !out || !rows_out || n > 0x7FFFFFFF) return (int)hipErrorInvalidValue;
  if (!fdms_aligned16(table, weight, out, rows_out) || (table_stride | out_stride | rows_stride) % 8 ||
      table_stride < hidden || out_stride < hidden || rows_stride != hidden)
    return (int)hipErrorInvalidValue;
#define FDMS_EMB_RMSNORM(PERV)                                                                                    \
  hipLaunchKernelGGL((rmsnorm_kernel<false, 0, PERV>), dim3((unsigned)n), dim3(kThreads), 0, (hipStream_t)stream,   \
                     (const bf16_t*)table, nullptr, (const bf16_t*)weight, (bf16_t*)out, (bf16_t*)rows_out, hidden,  \
                     table_stride, (int64_t)0, 1, out_stride, eps, nullptr, 0, (int64_t)0, nullptr, nullptr, nullptr, \
                     nullptr, (int64_t)0, 0, ids, vocab)
  const int per = (hidden + 8 * kThreads - 1) / (8 * kThreads);
  if (per == 1) FDMS_EMB_RMSNORM(1);
  else if (per == 2) FDMS_EMB_RMSNORM(2);
  else FDMS_EMB_RMSNORM(4);
#undef FDMS_EMB_RMSNORM
  FDMS_LAUNCH_CHECK();
  return 0;
}

// FP8 embedding rows: out[i, :] = bf16(e4m3fn(table[ids[i], :]) * bf16(scale_inv[ids[i]]))
// (embed_head.py:422-432: the FP8 row and its scale_inv, each in bf16, then
// multiplied).  One workgroup per id, 8 columns per thread; an id outside
// [0, vocab) yields a row of NaN (the reference's index_select raises there)
// and reads nothing.
__global__ __launch_bounds__(kThreads) void embedding_fp8_kernel(const int64_t* __restrict__ ids,
                                                                 const uint8_t* __restrict__ table, int64_t t_s,
                                                                 const float* __restrict__ scale_inv, int64_t vocab,
                                                                 bf16_t* __restrict__ out, int64_t o_s, int dim) {
  const int64_t i = blockIdx.x;
  const int64_t id = ids[i];
  const bool ok = id >= 0 && id < vocab;
  const float s = ok ? bf16_to_f32(f32_to_bf16(scale_inv[id])) : __builtin_nanf("");
  const uint8_t* src = table + (ok ? id : 0) * t_s;
  for (int c = threadIdx.x * 8; c < dim; c += kThreads * 8) {
    const uint2 v = ok ? *reinterpret_cast<const uint2*>(src + c) : uint2{0u, 0u};
    const uint32_t w[2] = {v.x, v.y};
    uint32_t o[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[h], false);  // exact
      const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[h], true);
      o[2 * h] = f32_to_bf16(lo[0] * s) | (f32_to_bf16(lo[1] * s) << 16);
      o[2 * h + 1] = f32_to_bf16(hi[0] * s) | (f32_to_bf16(hi[1] * s) << 16);
    }
    *reinterpret_cast<uint4*>(out + i * o_s + c) = uint4{o[0], o[1], o[2], o[3]};
  }
}

FDMS_EXPORT int fdms_embedding_fp8(const int64_t* ids, int64_t n, const void* table, int64_t table_stride,
                                   const float* scale_inv, int64_t vocab, void* out, int64_t out_stride, int dim,
                                   void* stream) {
  if (n < 0 || dim <= 0 || dim % 8 || vocab <= 0 || table_stride < dim || out_stride < dim) return (int)hipErrorInvalidValue;
  if (n == 0) return 0;
  if (!ids || !table || !scale_inv || !out || n > 0x7FFFFFFF) return (int)hipErrorInvalidValue;
  if ((uintptr_t)table % 8 || table_stride % 8 || !fdms_aligned16(out) || out_stride % 8) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(embedding_fp8_kernel, dim3((unsigned)n), dim3(kThreads), 0, (hipStream_t)stream, ids,
                     (const uint8_t*)table, table_stride, scale_inv, vocab, (bf16_t*)out, out_stride, dim);
  FDMS_LAUNCH_CHECK();
  return 0;
}

// Everything a prefill attention layer does to q and k between the qkv linear
// and the pack / attention, in place on views of the qkv rows: (Qwen3) the
// per-head RMSNorm of q and k, the DMS decision of each kv head's first query
// head (channel D - 1, then zeroed), RoPE of q and k -- the bits of
// rmsnorm_rows_kernel, extract_dms_kernel and rope_inplace_kernel one after the
// other, which read and write the rows up to three times in five launches.
// One workgroup per token, T = D / 8 lanes per head, two heads per lane group
// with both loads issued before the first use; a head's two halves meet
// through a lane shuffle of the bf16 pairs.  Bound by HBM: 4 D bytes per head
// and token, and the cos / sin row once per token.
// 12 000 tokens of the 8B shape (32 + 8 heads of 128): the five launches 132 us,
// this one 47 us (5.2 TB/s).
__device__ __forceinline__ float rope_half(float x, float other, float c, float signed_s) {
#pragma clang fp contract(off)
  const float a = x * c, b = other * signed_s;  // rope_f32's products and sum: x1 c + x2 (-s) or x2 c + x1 s
  return a + b;
}
template <int T, bool NORM>
__global__ __launch_bounds__(1024) void prefill_qk_kernel(
    bf16_t* __restrict__ q, int64_t qs_t, int64_t qs_h, int hq, bf16_t* __restrict__ k, int64_t ks_t, int64_t ks_h,
    int hkv, const bf16_t* __restrict__ q_weight, float q_eps, const bf16_t* __restrict__ k_weight, float k_eps,
    uint8_t* __restrict__ evict, int64_t es_t, int64_t es_h, float alpha_scale, float alpha_offset, float threshold,
    int positive_scale, const float* __restrict__ cos_sin, int64_t cs_p, const int64_t* __restrict__ positions) {
  constexpr int V = 8, P = 2, kHalf = T * V / 2;
  const int64_t t = blockIdx.x;
  const int groups = blockDim.x / T, lane = threadIdx.x % T, c = lane * V;
  const int heads = hq + hkv, group = hq / hkv;
  bf16_t* rows[P];
  Vec<bf16_t, V> xv[P], wv[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int h = min((int)(threadIdx.x / T) + p * groups, heads - 1);
    rows[p] = h < hq ? q + t * qs_t + h * qs_h : k + t * ks_t + (h - hq) * ks_h;
    xv[p] = *reinterpret_cast<const Vec<bf16_t, V>*>(rows[p] + c);
    if constexpr (NORM) wv[p] = *reinterpret_cast<const Vec<bf16_t, V>*>((h < hq ? q_weight : k_weight) + c);
  }
  const bool upper = c >= kHalf;
  const float* cs = cos_sin + positions[t] * cs_p + (upper ? c - kHalf : c);
  const Vec<float, 4> cv[2] = {*reinterpret_cast<const Vec<float, 4>*>(cs), *reinterpret_cast<const Vec<float, 4>*>(cs + 4)};
  Vec<float, 4> sv[2] = {*reinterpret_cast<const Vec<float, 4>*>(cs + kHalf),
                         *reinterpret_cast<const Vec<float, 4>*>(cs + kHalf + 4)};
#pragma unroll
  for (int i = 0; i < V; ++i) sv[i / 4].v[i % 4] = upper ? sv[i / 4].v[i % 4] : -sv[i / 4].v[i % 4];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int h = (int)(threadIdx.x / T) + p * groups;
    const bool valid = h < heads;  // the lanes past the last head repeat it without storing
    float x[V];
#pragma unroll
    for (int i = 0; i < V; ++i) x[i] = bf16_to_f32(xv[p].v[i].bits);
    if constexpr (NORM) {
      float ss = 0.0f;
#pragma unroll
      for (int i = 0; i < V; ++i) ss += x[i] * x[i];
      ss = segment_sum<T>(ss);
      const float inv = rsqrtf(ss / (float)(V * T) + (h < hq ? q_eps : k_eps));
#pragma unroll
      for (int i = 0; i < V; i += 2) {
        const uint32_t xn = pack_bf16(x[i] * inv, x[i + 1] * inv);
        const uint32_t o = pack_bf16(__uint_as_float(xn << 16) * bf16_to_f32(wv[p].v[i].bits),
                                     __uint_as_float(xn & 0xFFFF0000u) * bf16_to_f32(wv[p].v[i + 1].bits));
        x[i] = __uint_as_float(o << 16);
        x[i + 1] = __uint_as_float(o & 0xFFFF0000u);
      }
    }
    if (valid && h < hq && h % group == 0 && lane == T - 1) {
      evict[t * es_t + (h / group) * es_h] =
          dms_decide(x[V - 1], alpha_scale, alpha_offset, threshold, positive_scale) ? 1 : 0;
      x[V - 1] = 0.0f;
    }
    uint32_t o[V / 2];
#pragma unroll
    for (int i = 0; i < V / 2; ++i) {
      // exact: the values are bf16
      const uint32_t mine = (__float_as_uint(x[2 * i]) >> 16) | (__float_as_uint(x[2 * i + 1]) & 0xFFFF0000u);
      const uint32_t other = __shfl_xor(mine, T / 2);
      float y[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float xo = __uint_as_float(e ? other & 0xFFFF0000u : other << 16);
        y[e] = rope_half(x[2 * i + e], xo, cv[i / 2].v[(2 * i + e) % 4], sv[i / 2].v[(2 * i + e) % 4]);
      }
      o[i] = pack_bf16(y[0], y[1]);
    }
    if (valid) *reinterpret_cast<uint4*>(rows[p] + c) = uint4{o[0], o[1], o[2], o[3]};
  }
}

// q [tokens, hq, D] and k [tokens, hkv, D] bf16 views (element strides), D 64 or
// 128, (hq + hkv) * D / 8 <= 2048 lanes; q_weight / k_weight both [D] or both
// NULL (no norm); evict [tokens, hkv] bytes; cos_sin fp32 rows cat(cos, sin) of D
// values, cs_p apart.
FDMS_EXPORT int fdms_prefill_qk(void* q, int64_t qs_t, int64_t qs_h, int hq, void* k, int64_t ks_t, int64_t ks_h,
                                int hkv, int64_t num_tokens, int head_dim, const void* q_weight, float q_eps,
                                const void* k_weight, float k_eps, uint8_t* evict, int64_t es_t, int64_t es_h,
                                float alpha_scale, float alpha_offset, float threshold, int positive_scale,
                                const float* cos_sin, int64_t cs_p, const int64_t* positions, void* stream) {
  if (num_tokens < 0 || hkv <= 0 || hq <= 0 || hq % hkv || (head_dim != 64 && head_dim != 128))
    return (int)hipErrorInvalidValue;
  const int lanes = head_dim / 8;
  if ((int64_t)(hq + hkv) * lanes > 2048 || (q_weight == nullptr) != (k_weight == nullptr)) return (int)hipErrorInvalidValue;
  if (num_tokens == 0) return 0;
  if (!q || !k || !evict || !cos_sin || !positions || num_tokens > 0x7FFFFFFF) return (int)hipErrorInvalidValue;
  if (!fdms_aligned16(q, k, q_weight, k_weight, cos_sin) || (qs_t | qs_h | ks_t | ks_h) % 8 || cs_p % 4)
    return (int)hipErrorInvalidValue;
  const int threads = ((hq + hkv + 1) / 2 * lanes + kWave - 1) / kWave * kWave;
#define FDMS_PREFILL_QK(TV, NV)                                                                                    \
  hipLaunchKernelGGL((prefill_qk_kernel<TV, NV>), dim3((unsigned)num_tokens), dim3((unsigned)threads), 0,             \
                     (hipStream_t)stream, (bf16_t*)q, qs_t, qs_h, hq, (bf16_t*)k, ks_t, ks_h, hkv,                     \
                     (const bf16_t*)q_weight, q_eps, (const bf16_t*)k_weight, k_eps, evict, es_t, es_h, alpha_scale,   \
                     alpha_offset, threshold, positive_scale, cos_sin, cs_p, positions)
  if (lanes == 8) {
    if (q_weight) FDMS_PREFILL_QK(8, true); else FDMS_PREFILL_QK(8, false);
  } else {
    if (q_weight) FDMS_PREFILL_QK(16, true); else FDMS_PREFILL_QK(16, false);
  }
#undef FDMS_PREFILL_QK
  FDMS_LAUNCH_CHECK();
  return 0;
}

// out[r, j] = bf16(silu(x[r, j]) * x[r, F + j]) in fp32 (activation.py:8-11).
// A workgroup takes 256 U consecutive 8-column units of the output, a thread U
// of them, 256 apart; all its loads (2 U of 16 bytes) go out before the first
// use.  The row of the workgroup's first unit comes from one 64-bit division,
// the threads' from a 32-bit one.  Bound by HBM (6 bytes per output), with the
// exponential and the division close behind.  16384 rows of 2 x 8192 (805 MB):
// 163 -> 154 us, 5.2 TB/s (a grid-stride loop with a 64-bit division and one
// unit in flight per thread before).
template <int U>
__global__ __launch_bounds__(kThreads) void silu_mul_kernel(const bf16_t* __restrict__ x, bf16_t* __restrict__ out,
                                                            int64_t units, int per_row) {
  constexpr int V = 8;
  const int64_t u0 = (int64_t)blockIdx.x * (kThreads * U);
  const int64_t r0 = u0 / per_row;
  const uint32_t c0 = (uint32_t)(u0 - r0 * per_row);
  const int64_t f = (int64_t)per_row * V;
  Vec<bf16_t, V> g[U], up[U];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    // units past the end repeat the last one
    const uint32_t off = c0 + (uint32_t)min((int64_t)(threadIdx.x + j * kThreads), units - 1 - u0);
    const uint32_t dr = off / (uint32_t)per_row;
    const bf16_t* p = x + (r0 + dr) * 2 * f + (int64_t)(off - dr * per_row) * V;
    g[j] = *reinterpret_cast<const Vec<bf16_t, V>*>(p);
    up[j] = *reinterpret_cast<const Vec<bf16_t, V>*>(p + f);
  }
#pragma unroll
  for (int j = 0; j < U; ++j) {
    float o[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const float a = bf16_to_f32(g[j].v[i].bits);
      o[i] = a / (1.0f + expf(-a)) * bf16_to_f32(up[j].v[i].bits);
    }
    const int64_t u = u0 + threadIdx.x + j * kThreads;
    if (u < units)
      *reinterpret_cast<uint4*>(out + u * V) =
          uint4{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3]), pack_bf16(o[4], o[5]), pack_bf16(o[6], o[7])};
  }
}

FDMS_EXPORT int fdms_silu_mul(const void* x, void* out, int64_t rows, int f, void* stream) {
  if (rows < 0 || f <= 0 || f % 8) return (int)hipErrorInvalidValue;
  if (rows == 0) return 0;
  if (!x || !out) return (int)hipErrorInvalidValue;
  const int per_row = f / 8;
  const int64_t units = rows * per_row;
  const auto blocks = [&](int u) { return (units + kThreads * u - 1) / (kThreads * u); };
  if (blocks(kSiluUnits) > 0x7FFFFFFF) return (int)hipErrorInvalidValue;
  // several units a thread once that still gives every CU eight workgroups (a full
  // set of waves); below, one unit a thread spreads the call over more of the chip
  if (blocks(kSiluUnits) >= 2048)
    hipLaunchKernelGGL(silu_mul_kernel<kSiluUnits>, dim3((unsigned)blocks(kSiluUnits)), dim3(kThreads), 0,
                       (hipStream_t)stream, (const bf16_t*)x, (bf16_t*)out, units, per_row);
  else
    hipLaunchKernelGGL(silu_mul_kernel<1>, dim3((unsigned)blocks(1)), dim3(kThreads), 0, (hipStream_t)stream,
                       (const bf16_t*)x, (bf16_t*)out, units, per_row);
  FDMS_LAUNCH_CHECK();
  return 0;
}

// Row argmax with torch.argmax's semantics (embed_head.py:142, 160): ties go
// to the lowest index and NaN counts as larger than every number (the lowest
// NaN index wins), so a row always yields an index in [0, n).

// One 1024-thread block per row; 16-byte vector loads, four in flight per
// thread, when the row is 16-byte aligned; fp32 or bf16 logits; int64 output.
constexpr int kArgmaxThreads = 1024;

template <typename T>
struct ArgmaxVec;
template <>
struct ArgmaxVec<float> {
  static constexpr int kN = 4;
  static __device__ __forceinline__ void load(const float* p, float* v) {
    const float4 x = *reinterpret_cast<const float4*>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  }
};
template <>
struct ArgmaxVec<bf16_t> {
  static constexpr int kN = 8;
  static __device__ __forceinline__ void load(const bf16_t* p, float* v) {
    const uint4 x = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
  }
};

template <typename T, bool VEC>
__global__ __launch_bounds__(kArgmaxThreads) void argmax_rows_kernel(const T* __restrict__ x, int64_t stride, int n,
                                                                     int64_t* __restrict__ out) {
  constexpr int kW = kArgmaxThreads / kWave;
  __shared__ float s_v[kW];
  __shared__ int s_i[kW];
  const T* row = x + (int64_t)blockIdx.x * stride;
  float best = -INFINITY;
  int bi = 0x7FFFFFFF;  // no element yet: loses every comparison
  auto take = [&](float v, int j) {
    if (bi == 0x7FFFFFFF || argmax_better(v, j, best, bi)) {
      best = v;
      bi = j;
    }
  };
  int tail = 0;
  if (VEC) {
    constexpr int N = ArgmaxVec<T>::kN;
    constexpr int kU = 4;  // vectors in flight per thread
    const int nvec = n / N;
    for (int v0 = threadIdx.x; v0 < nvec; v0 += kArgmaxThreads * kU) {
      float vals[kU][N];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int vi = v0 + u * kArgmaxThreads;
        if (vi < nvec) ArgmaxVec<T>::load(row + (int64_t)vi * N, vals[u]);
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int vi = v0 + u * kArgmaxThreads;
        if (vi < nvec) {
#pragma unroll
          for (int e = 0; e < N; ++e) take(vals[u][e], vi * N + e);
        }
      }
    }
    tail = nvec * N;
  }
  for (int j = tail + threadIdx.x; j < n; j += kArgmaxThreads) take(ld<T>(row + j), j);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o);
    const int oi = __shfl_xor(bi, o);
    if (oi != 0x7FFFFFFF && (bi == 0x7FFFFFFF || argmax_better(ov, oi, best, bi))) {
      best = ov;
      bi = oi;
    }
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    s_v[w] = best;
    s_i[w] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < kW; ++i) {
      if (s_i[i] != 0x7FFFFFFF && (bi == 0x7FFFFFFF || argmax_better(s_v[i], s_i[i], best, bi))) {
        best = s_v[i];
        bi = s_i[i];
      }
    }
    out[blockIdx.x] = bi;
  }
}

FDMS_EXPORT int fdms_argmax_rows(const void* x, int dtype, int64_t stride, int64_t rows, int n, int64_t* out,
                                 void* stream) {
  if (rows < 0 || n <= 0 || rows > 0x7FFFFFFF) return (int)hipErrorInvalidValue;
  if (rows == 0) return 0;
  if (!x || !out) return (int)hipErrorInvalidValue;
  const int esz = dtype == kF32 ? 4 : 2;
  const bool vec = ((uintptr_t)x % 16) == 0 && (stride * esz) % 16 == 0;
  const dim3 grid((unsigned)rows), block(kArgmaxThreads);
  if (dtype == kF32) {
    if (vec) hipLaunchKernelGGL((argmax_rows_kernel<float, true>), grid, block, 0, (hipStream_t)stream, (const float*)x, stride, n, out);
    else hipLaunchKernelGGL((argmax_rows_kernel<float, false>), grid, block, 0, (hipStream_t)stream, (const float*)x, stride, n, out);
  } else if (dtype == kBF16) {
    if (vec) hipLaunchKernelGGL((argmax_rows_kernel<bf16_t, true>), grid, block, 0, (hipStream_t)stream, (const bf16_t*)x, stride, n, out);
    else hipLaunchKernelGGL((argmax_rows_kernel<bf16_t, false>), grid, block, 0, (hipStream_t)stream, (const bf16_t*)x, stride, n, out);
  } else {
    return (int)hipErrorInvalidValue;
  }
  FDMS_LAUNCH_CHECK();
  return 0;
}
