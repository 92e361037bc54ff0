// The minimal engine's per-layer elementwise work around the attention
// path, fused: the residual add with the RMSNorm that follows it, and the
// SiLU gate of the MLP. Same arithmetic as the model's torch ops (and the
// reference's LlamaRMSNorm / LlamaMLP, liteinfer/models/llama.py:34-48,
// :101-116): sums in fp32, the normalised row rounded to the model dtype
// before the weight multiplies it, every torch-visible intermediate rounded
// where torch rounds it.
#include "li_common.h"

namespace {

constexpr int kNormThreads = 256;  // (twice that for few rows: kFewNormRows)

template <typename T>
struct Vec8 {
  typedef __attribute__((__vector_size__(8 * sizeof(T)))) T type;
};

// One work-group of NT threads per row of `hidden` elements (a multiple of 8 and
// at most 8 * kNormThreads * kNormPer), each thread up to kNormPer (or half
// that) chunks of 8.
constexpr int kNormPer = 4;
// Up to this many rows a work-group's loads are the call's latency, and a row
// takes twice the threads (a decode step of 4 layers of 4096 wide rows, nine
// norms of eight runs' sums: 455 -> 445 us at one row, 1420 -> 1412 at 256).
constexpr int kFewNormRows = 256;

// h <- h + delta (when delta is given), rounded to T; out <- weight *
// T(h * rsqrt(mean(h^2) + eps)), the product rounded to T. With `splits` > 0
// delta is a projection's fp32 sums over as many runs of its K
// ([splits][rows][hidden], skinny_gemm.hip), added here and rounded to T: one
// launch less than rounding them on their own.
template <typename T, int NT>
__global__ __launch_bounds__(NT) void add_rms_norm(T* h, const T* delta, const T* weight, T* out,
                                                            int hidden, int64_t h_s, int64_t d_s, int64_t o_s,
                                                            float eps, const float* part, int splits) {
  typedef typename Vec8<T>::type V;
  constexpr int kPer = kNormPer * kNormThreads / NT;
  const int64_t row = blockIdx.x;
  T* hrow = h + row * h_s;
  const T* drow = delta ? delta + row * d_s : nullptr;
  T* orow = out + row * o_s;
  const int chunks = hidden / 8;
  float x[kPer][8];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int c = threadIdx.x + k * NT;
    if (c < chunks) {
      V v = *reinterpret_cast<const V*>(hrow + 8 * c);
      if (drow) {
        const V dv = *reinterpret_cast<const V*>(drow + 8 * c);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = li_from_float<T>((float)v[e] + (float)dv[e]);
        *reinterpret_cast<V*>(hrow + 8 * c) = v;
      } else if (splits > 0) {
        float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int p0 = 0; p0 < splits; p0 += 8) {  // eight runs' loads together
          floatx4_t lo[8], hi[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const float* src = part + ((int64_t)min(p0 + u, splits - 1) * gridDim.x + row) * hidden + 8 * c;
            lo[u] = *reinterpret_cast<const floatx4_t*>(src);
            hi[u] = *reinterpret_cast<const floatx4_t*>(src + 4);
          }
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (p0 + u < splits) {
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                sum[e] += lo[u][e];
                sum[4 + e] += hi[u][e];
              }
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = li_from_float<T>((float)v[e] + (float)li_from_float<T>(sum[e]));
        *reinterpret_cast<V*>(hrow + 8 * c) = v;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[k][e] = (float)v[e];
        ss = fmaf(x[k][e], x[k][e], ss);
      }
    }
  }
  __shared__ float partial[NT / 64];
  ss = li_wave_sum(ss);
  if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = ss;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) total += partial[w];
  const float inv = rsqrtf(total / (float)hidden + eps);
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int c = threadIdx.x + k * NT;
    if (c < chunks) {
      const V wv = *reinterpret_cast<const V*>(weight + 8 * c);
      V o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float normed = (float)li_from_float<T>(x[k][e] * inv);
        o[e] = li_from_float<T>((float)wv[e] * normed);
      }
      *reinterpret_cast<V*>(orow + 8 * c) = o;
    }
  }
}

// out[r, i] = T(T(silu(gate)) * up) with gate = gu[r, i], up = gu[r, F + i]
// (torch's F.silu(gate) * up on the two halves of the fused projection).
// With `splits` > 0 the projection is given as its fp32 sums over as many
// runs of K, [splits][rows][2 F], added and rounded to T first.
template <typename T>
__global__ __launch_bounds__(256) void silu_mul(const T* gu, T* out, int64_t rows, int f, int64_t gu_s, int64_t o_s,
                                                const float* part, int splits) {
  typedef typename Vec8<T>::type V;
  const int chunks = f / 8;
  const int64_t total = rows * chunks;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / chunks;
    const int c = (int)(i - r * chunks);
    V g, u;
    if (splits > 0) {
      float gs[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, us[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int p = 0; p < splits; ++p) {
        const float* src = part + ((int64_t)p * rows + r) * 2 * f + 8 * c;
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
          const floatx4_t gv = *reinterpret_cast<const floatx4_t*>(src + e);
          const floatx4_t uv = *reinterpret_cast<const floatx4_t*>(src + f + e);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            gs[e + q] += gv[q];
            us[e + q] += uv[q];
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        g[e] = li_from_float<T>(gs[e]);
        u[e] = li_from_float<T>(us[e]);
      }
    } else {
      g = *reinterpret_cast<const V*>(gu + r * gu_s + 8 * c);
      u = *reinterpret_cast<const V*>(gu + r * gu_s + f + 8 * c);
    }
    V o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float gf = (float)g[e];
      const float s = (float)li_from_float<T>(gf / (1.f + expf(-gf)));
      o[e] = li_from_float<T>(s * (float)u[e]);
    }
    *reinterpret_cast<V*>(out + r * o_s + 8 * c) = o;
  }
}

// cos / sin of positions[i] * inv_freq[d mod half], d < 2 half, in fp32 then
// rounded to T: the model's rotary tables (liteinfer/models/llama.py:70-78)
// in one launch instead of torch's seven.
template <typename T>
__global__ __launch_bounds__(256) void rotary_tables(const int64_t* positions, const float* inv_freq, T* cos_out,
                                                     T* sin_out, int64_t tokens, int half) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= tokens * half) return;
  const int64_t t = i / half;
  const int d = (int)(i - t * half);
  const float x = (float)positions[t] * inv_freq[d];
  const T c = li_from_float<T>(cosf(x)), s = li_from_float<T>(sinf(x));
  T* crow = cos_out + t * 2 * half;
  T* srow = sin_out + t * 2 * half;
  crow[d] = crow[d + half] = c;
  srow[d] = srow[d + half] = s;
}

// A decode step's inputs into the static buffers its captured graph reads:
// rows 0 .. n - 1 as given, rows n .. width - 1 a one-token context in the
// reserved slot (ten torch copies and fills otherwise).
struct StageArgs {
  const int64_t *ids, *positions, *write_slots, *slots;
  const int32_t* context_lens;
  int64_t *ids_out, *positions_out, *write_out, *table_out;
  int32_t* lens_out;
  int64_t slots_s, table_s;
  int n, cols, width;
  int64_t pad_slot;
};

__global__ __launch_bounds__(256) void stage_decode(StageArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < a.width) {
    const bool real = i < a.n;
    a.ids_out[i] = real ? a.ids[i] : 0;
    a.positions_out[i] = real ? a.positions[i] : 0;
    a.write_out[i] = real ? a.write_slots[i] : a.pad_slot;
    a.lens_out[i] = real ? a.context_lens[i] : 1;
    if (!real) a.table_out[i * a.table_s] = a.pad_slot;
  }
  if (i < (int64_t)a.n * a.cols) {
    const int64_t r = i / a.cols, c = i - r * a.cols;
    a.table_out[r * a.table_s + c] = a.slots[r * a.slots_s + c];
  }
}

bool rows_ok(const void* p, int64_t stride, int esize) {
  return li::aligned16(p) && (stride * esize) % 16 == 0;
}

}  // namespace

namespace {

int add_rms_norm_impl(const char* who, void* h, const void* delta, const float* partials, int splits, const void* weight,
                      void* out, int64_t rows, int hidden, int64_t h_stride, int64_t delta_stride, int64_t out_stride,
                      float eps, int dtype, void* stream) {
  li::clear_error();
  if (dtype != LI_BF16 && dtype != LI_F16) return li::fail(LI_EUNSUPPORTED, "%s: bf16 or f16 rows only", who);
  if (rows < 0 || hidden <= 0 || hidden % 8 != 0 || hidden > 8 * kNormThreads * kNormPer)
    return li::fail(LI_EINVAL, "%s: hidden size %d must be a multiple of 8 up to %d", who, hidden,
                    8 * kNormThreads * kNormPer);
  if (rows == 0) return LI_OK;
  if (rows > 0x7fffffffLL) return li::fail(LI_EINVAL, "%s: too many rows", who);
  if (!h || !weight || !out || !rows_ok(h, h_stride, 2) || !rows_ok(out, out_stride, 2) || !li::aligned16(weight) ||
      (delta && !rows_ok(delta, delta_stride, 2)) || (splits > 0 && (!partials || !li::aligned16(partials))))
    return li::fail(LI_EINVAL, "%s: rows must be 16-byte aligned with the last axis contiguous", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool few = rows <= kFewNormRows && hidden > 8 * kNormThreads;
  const dim3 g((unsigned)rows), b(few ? 2 * kNormThreads : kNormThreads);
#define LI_NORM(T, NT)                                                                                           \
  hipLaunchKernelGGL((add_rms_norm<T, NT>), g, b, 0, s, static_cast<T*>(h), static_cast<const T*>(delta),        \
                     static_cast<const T*>(weight), static_cast<T*>(out), hidden, h_stride, delta_stride,        \
                     out_stride, eps, partials, splits)
  if (dtype == LI_BF16) {
    if (few) LI_NORM(li_bf16, 2 * kNormThreads);
    else LI_NORM(li_bf16, kNormThreads);
  } else {
    if (few) LI_NORM(li_f16, 2 * kNormThreads);
    else LI_NORM(li_f16, kNormThreads);
  }
#undef LI_NORM
  return li::check_launch(who);
}

int silu_mul_impl(const char* who, const void* gate_up, const float* partials, int splits, void* out, int64_t rows,
                  int ffn, int64_t gate_up_stride, int64_t out_stride, int dtype, void* stream) {
  li::clear_error();
  if (dtype != LI_BF16 && dtype != LI_F16) return li::fail(LI_EUNSUPPORTED, "%s: bf16 or f16 rows only", who);
  if (rows < 0 || ffn <= 0 || ffn % 8 != 0) return li::fail(LI_EINVAL, "%s: ffn %d must be a multiple of 8", who, ffn);
  if (rows == 0) return LI_OK;
  if ((splits > 0 ? !partials || !li::aligned16(partials) : !gate_up || !rows_ok(gate_up, gate_up_stride, 2)) || !out ||
      !rows_ok(out, out_stride, 2) || (ffn * 2) % 16)
    return li::fail(LI_EINVAL, "%s: rows must be 16-byte aligned with the last axis contiguous", who);
  const int64_t work = rows * (ffn / 8);
  const int64_t blocks = std::min<int64_t>(li::cdiv64(work, 256), 65536);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == LI_BF16)
    hipLaunchKernelGGL(silu_mul<li_bf16>, dim3((unsigned)blocks), dim3(256), 0, s,
                       static_cast<const li_bf16*>(gate_up), static_cast<li_bf16*>(out), rows, ffn, gate_up_stride,
                       out_stride, partials, splits);
  else
    hipLaunchKernelGGL(silu_mul<li_f16>, dim3((unsigned)blocks), dim3(256), 0, s, static_cast<const li_f16*>(gate_up),
                       static_cast<li_f16*>(out), rows, ffn, gate_up_stride, out_stride, partials, splits);
  return li::check_launch(who);
}

}  // namespace

extern "C" int li_add_rms_norm(void* h, const void* delta, const void* weight, void* out, int64_t rows, int hidden,
                               int64_t h_stride, int64_t delta_stride, int64_t out_stride, float eps, int dtype,
                               void* stream) {
  return add_rms_norm_impl("li_add_rms_norm", h, delta, nullptr, 0, weight, out, rows, hidden, h_stride, delta_stride,
                           out_stride, eps, dtype, stream);
}

extern "C" int li_add_rms_norm_partials(void* h, const float* partials, int splits, const void* weight, void* out,
                                        int64_t rows, int hidden, int64_t h_stride, int64_t out_stride, float eps,
                                        int dtype, void* stream) {
  if (splits < 1) return li::fail(LI_EINVAL, "li_add_rms_norm_partials: %d splits", splits);
  return add_rms_norm_impl("li_add_rms_norm_partials", h, nullptr, partials, splits, weight, out, rows, hidden, h_stride,
                           0, out_stride, eps, dtype, stream);
}

extern "C" int li_silu_mul(const void* gate_up, void* out, int64_t rows, int ffn, int64_t gate_up_stride,
                           int64_t out_stride, int dtype, void* stream) {
  return silu_mul_impl("li_silu_mul", gate_up, nullptr, 0, out, rows, ffn, gate_up_stride, out_stride, dtype, stream);
}

extern "C" int li_silu_mul_partials(const float* partials, int splits, void* out, int64_t rows, int ffn,
                                    int64_t out_stride, int dtype, void* stream) {
  if (splits < 1) return li::fail(LI_EINVAL, "li_silu_mul_partials: %d splits", splits);
  return silu_mul_impl("li_silu_mul_partials", nullptr, partials, splits, out, rows, ffn, 0, out_stride, dtype, stream);
}

extern "C" int li_rotary_tables(const int64_t* positions, const float* inv_freq, void* cos_out, void* sin_out,
                                int64_t tokens, int half, int dtype, void* stream) {
  li::clear_error();
  if (dtype != LI_F32 && dtype != LI_BF16 && dtype != LI_F16)
    return li::fail(LI_EINVAL, "li_rotary_tables: unknown dtype %d", dtype);
  if (tokens < 0 || half <= 0) return li::fail(LI_EINVAL, "li_rotary_tables: bad extents");
  if (tokens == 0) return LI_OK;
  if (!positions || !inv_freq || !cos_out || !sin_out) return li::fail(LI_EINVAL, "li_rotary_tables: null pointer");
  const int64_t blocks = li::cdiv64(tokens * half, 256);
  if (blocks > 0x7fffffffLL) return li::fail(LI_EINVAL, "li_rotary_tables: too many tokens");
  hipStream_t s = static_cast<hipStream_t>(stream);
#define LI_ROTARY(T)                                                                                                 \
  hipLaunchKernelGGL(rotary_tables<T>, dim3((unsigned)blocks), dim3(256), 0, s, positions, inv_freq,                 \
                     static_cast<T*>(cos_out), static_cast<T*>(sin_out), tokens, half)
  if (dtype == LI_F32) LI_ROTARY(float);
  else if (dtype == LI_BF16) LI_ROTARY(li_bf16);
  else LI_ROTARY(li_f16);
#undef LI_ROTARY
  return li::check_launch("li_rotary_tables");
}

extern "C" int li_stage_decode(const int64_t* ids, const int64_t* positions, const int64_t* write_slots,
                               const int64_t* slots, int64_t slots_stride, const int32_t* context_lens,
                               int64_t* ids_out, int64_t* positions_out, int64_t* write_out, int64_t* table_out,
                               int64_t table_stride, int32_t* lens_out, int n, int cols, int width, int64_t pad_slot,
                               void* stream) {
  li::clear_error();
  if (n < 0 || cols < 0 || width < n || cols > table_stride)
    return li::fail(LI_EINVAL, "li_stage_decode: %d rows of %d columns do not fit %d of %lld", n, cols, width,
                    (long long)table_stride);
  if (width == 0) return LI_OK;
  if (!ids_out || !positions_out || !write_out || !table_out || !lens_out ||
      (n > 0 && (!ids || !positions || !write_slots || !context_lens || (cols > 0 && !slots))))
    return li::fail(LI_EINVAL, "li_stage_decode: null pointer");
  const StageArgs a{ids,       positions,    write_slots, slots, context_lens, ids_out, positions_out, write_out,
                    table_out, lens_out,     slots_stride, table_stride, n,    cols,    width,         pad_slot};
  const int64_t work = std::max<int64_t>((int64_t)n * cols, width);
  hipLaunchKernelGGL(stage_decode, dim3((unsigned)li::cdiv64(work, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), a);
  return li::check_launch("li_stage_decode");
}
