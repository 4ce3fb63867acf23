// Memory-bound kernels of the hot-expert path: GGUF dequantisation to bf16 (through the
// grouped GEMMs' decoder), the hot
// cache's route lookup, q8_1 activation quantisation, SiLU*mul and the weighted top-k
// combine.
#include <type_traits>

#include "bpiece.h"
#include "kernels.h"

namespace ktmi {

// ---------------------------------------------------------------- dequant
// The grouped GEMMs' own decoder (bpiece.h) run stand-alone, so the bytes-to-bf16 step the
// GEMMs feed to the matrix cores is the one this entry point exposes (and its tests pin): the
// same load_head / load / decode bodies, half h = lane / 32 of a 64-value step as there.
// P:11471-11498 contract, all four formats.
//
// Bound by HBM: a value is read as half a byte to a byte and written as two. A wave takes 16
// consecutive (row, 256-value column) units, four lanes (step parity p, half h) to a unit, so
// the raw bytes of a wave are one contiguous range and so is its output; each lane's decoded
// chunks (16 bytes, 64 to 192 bytes apart) pass through LDS, where the wave picks them up in
// memory order: every store instruction writes whole 256-byte segments. With a lane to a row
// and the chunks stored straight from the registers, an instruction touched 64 segments and
// eight 7168 x 2048 Q6_K experts took 144 us (2.3 TB/s); so they take 67 us (4.9 TB/s,
// the rate of a large copy on this card). The stores are non-temporal: 43 against 54 us for
// eight such Q4_K experts, and no slower for a reader that follows, down to one expert of 1024 x
// 2048 (with a pass over the output behind it 11.4 us either way).
constexpr int DQ_UNITS = 16;                      // (row, column) units a wave
constexpr int DQ_STG = DQ_UNITS * 256;            // staging bytes a wave: 128 bf16 values a unit

template <int TYPE>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ raw, int64_t raw_stride,
                                                      int64_t rows, int64_t cols, int64_t rb,
                                                      uint16_t* __restrict__ out, int64_t out_stride) {
  using BP = BPiece<TYPE>;
  __shared__ uint32_t grid[TYPE == GGML_IQ3_S ? 512 : 1];
  __shared__ __attribute__((aligned(16))) uint8_t stage[4 * DQ_STG];
  if constexpr (TYPE == GGML_IQ3_S) {
    stage_iq3s_sel(grid);
    __syncthreads();
  }
  const int64_t e = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int p = lane & 1, h = lane >> 5, ul = (lane & 31) >> 1;
  const int64_t nsb = (cols + 255) / 256, total = rows * nsb;
  const int64_t u0 = ((int64_t)blockIdx.x * 4 + wave) * DQ_UNITS;  // the wave's first unit
  if (u0 >= total) return;
  const int64_t r0 = u0 / nsb;
  const uint32_t sb0 = (uint32_t)(u0 - r0 * nsb);
  // row and column of the wave's unit q
  auto place = [&](int q, int64_t& r, int& sb) {
    const uint32_t t = sb0 + (uint32_t)q, dr = t / (uint32_t)nsb;
    r = r0 + dr;
    sb = (int)(t - dr * (uint32_t)nsb);
  };
  // a lane past the last unit reads the last one (its values are not stored): no branch, so that
  // every load is on its way before the first is waited for
  int64_t r;
  int sb;
  place((int)(u0 + ul < total ? ul : total - 1 - u0), r, sb);
  const uint8_t* row = raw + e * raw_stride + r * rb;
  typename BP::Head hd;
  typename BP::Raw rw[2];
  // Q8_0 rows may end inside a column (a piece is one 32-value block): the pieces past the
  // row's end are not loaded
  auto inside = [&](int ks) {
    return TYPE != GGML_Q8_0 || 256 * (int64_t)sb + ks + BP::off0(h) < cols;
  };
  BP::load_head(row, sb, h, hd);
  if (inside(BP::template ksub_hp<0>(p))) BP::template load_hp<0>(row, sb, h, p, grid, rw[0]);
  if (inside(BP::template ksub_hp<1>(p))) BP::template load_hp<1>(row, sb, h, p, grid, rw[1]);
  __builtin_amdgcn_sched_barrier(0);  // the same eight experts back to back: 62 us, 65 without it
  uint8_t* stg = stage + wave * DQ_STG;
  uint16_t* oe = out + e * out_stride;
  auto half = [&](auto s2c) {
    constexpr int S2 = decltype(s2c)::value;
    uint32_t v[16];
    BP::template decode_hp<S2>(hd, rw[S2], grid, p, v);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int q = c < 2 ? BP::off0(h) / 8 + c : BP::off1(h) / 8 + c - 2;
      const int slot = (BP::template ksub_hp<S2>(p) - 128 * S2 + BP::coff(q)) / 8;  // 16-byte slot of the unit
      const u32x4_t w = {v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]};
      *(u32x4_t*)(stg + ul * 256 + 16 * (slot ^ ul)) = w;  // slot ^ unit: no bank conflicts
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int q = 4 * it + (lane >> 4), slot = lane & 15;
      const u32x4_t w = *(const u32x4_t*)(stg + q * 256 + 16 * (slot ^ q));
      int64_t qr;
      int qs;
      place(q, qr, qs);
      const int64_t k = 256 * (int64_t)qs + 128 * S2 + 8 * slot;
      if (u0 + q < total && k < cols) __builtin_nontemporal_store(w, (u32x4_t*)(oe + qr * cols + k));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  half(std::integral_constant<int, 0>{});
  half(std::integral_constant<int, 1>{});
}

int launch_dequant(const uint8_t* raw, int64_t raw_stride, int type, int64_t n, int64_t rows, int64_t cols,
                   uint16_t* out, int64_t out_stride, hipStream_t stream) {
  const int64_t units = rows * ((cols + 255) / 256);
  dim3 grid((unsigned)((units + 4 * DQ_UNITS - 1) / (4 * DQ_UNITS)), (unsigned)n);
  const int64_t rb = row_bytes(cols, type);
  switch (type) {
    case GGML_Q8_0: dequant_kernel<GGML_Q8_0><<<grid, 256, 0, stream>>>(raw, raw_stride, rows, cols, rb, out, out_stride); break;
    case GGML_Q4_K: dequant_kernel<GGML_Q4_K><<<grid, 256, 0, stream>>>(raw, raw_stride, rows, cols, rb, out, out_stride); break;
    case GGML_Q6_K: dequant_kernel<GGML_Q6_K><<<grid, 256, 0, stream>>>(raw, raw_stride, rows, cols, rb, out, out_stride); break;
    case GGML_IQ3_S: dequant_kernel<GGML_IQ3_S><<<grid, 256, 0, stream>>>(raw, raw_stride, rows, cols, rb, out, out_stride); break;
    default: set_error("dequant: ggml type %d has no kernel", type); return KTMI_ETYPE;
  }
  KTMI_HIP_TRY(hipGetLastError());
  return KTMI_OK;
}

// ---------------------------------------------------------------- hot-cache route
// hot/kt_hot_cache.py:62-75: two table lookups and a count per route. fp32 counts of
// +1.0 stay exact below 2^24, so the atomic order does not change them.
//
// What bounds a prefill chunk's call is the counts: device-scope atomics on one address take
// about 12.5 ns each, one after the other, and a popular expert is on nearly every token (one
// atomic a route: 131072 routes of a Zipf-1.1 router over 256 experts 206 us, its 1.6 MB of
// ids about 1 us). So a long call counts in LDS and each block adds its totals once: 131072
// routes 206 -> 4.6 us. Up to ROUTE_LDS_MIN routes (decode
// windows and short prompts) the route's own atomic is cheaper than the histogram's two barriers.
constexpr int64_t ROUTE_LDS_MIN = 1024;
constexpr int ROUTE_BINS = 2048;  // experts counted in LDS; a larger id takes its own atomic
constexpr int ROUTE_PER = 4;      // routes a thread and pass

__global__ __launch_bounds__(256) void route_kernel(const int32_t* __restrict__ ids, int64_t n,
                                                    const int32_t* __restrict__ log2slot,
                                                    const int32_t* __restrict__ log2cpu, float* counts,
                                                    int32_t* __restrict__ slot_ids, int32_t* __restrict__ cpu_ids) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t e = ids[i];
  slot_ids[i] = log2slot[e];
  cpu_ids[i] = log2cpu[e];
  if (counts) atomicAdd(counts + e, 1.0f);
}

__global__ __launch_bounds__(1024) void route_count_kernel(const int32_t* __restrict__ ids, int64_t n,
                                                           const int32_t* __restrict__ log2slot,
                                                           const int32_t* __restrict__ log2cpu, float* counts,
                                                           int32_t* __restrict__ slot_ids,
                                                           int32_t* __restrict__ cpu_ids) {
  __shared__ uint32_t bins[ROUTE_BINS];
  for (int b = threadIdx.x; b < ROUTE_BINS; b += 1024) bins[b] = 0;
  __syncthreads();
  const int64_t span = 1024 * ROUTE_PER;
  for (int64_t base = blockIdx.x * span; base < n; base += gridDim.x * span) {
    int32_t e[ROUTE_PER];
#pragma unroll
    for (int j = 0; j < ROUTE_PER; ++j) {
      const int64_t i = base + 1024 * j + threadIdx.x;
      e[j] = i < n ? ids[i] : 0;
    }
#pragma unroll
    for (int j = 0; j < ROUTE_PER; ++j) {
      const int64_t i = base + 1024 * j + threadIdx.x;
      if (i < n) {
        slot_ids[i] = log2slot[e[j]];
        cpu_ids[i] = log2cpu[e[j]];
        if ((uint32_t)e[j] < (uint32_t)ROUTE_BINS) atomicAdd(&bins[e[j]], 1u);
        else atomicAdd(counts + e[j], 1.0f);
      }
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < ROUTE_BINS; b += 1024) {
    const uint32_t c = bins[b];
    if (c) atomicAdd(counts + b, (float)c);
  }
}

int launch_route(const int32_t* ids, int64_t n, const int32_t* log2slot, const int32_t* log2cpu, float* counts,
                 int32_t* slot_ids, int32_t* cpu_ids, hipStream_t stream) {
  if (n == 0) return KTMI_OK;
  if (counts && n > ROUTE_LDS_MIN) {
    const int64_t want = (n + 1024 * ROUTE_PER - 1) / (1024 * ROUTE_PER);
    route_count_kernel<<<(unsigned)(want < 256 ? want : 256), 1024, 0, stream>>>(ids, n, log2slot, log2cpu, counts,
                                                                                 slot_ids, cpu_ids);
  } else {
    route_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(ids, n, log2slot, log2cpu, counts, slot_ids, cpu_ids);
  }
  KTMI_HIP_TRY(hipGetLastError());
  return KTMI_OK;
}

// ---------------------------------------------------------------- q8_1 quantisation
// kt_gguf_moe_multi.cu:600-650: one thread per value of the padded row; the 32 values
// of a block are 32 consecutive lanes (half a wave64). amax and sum reduce over the
// half-wave in xor-butterfly order; lane 0 of the block writes (half d, half sum).
template <typename T>
__device__ __forceinline__ float to_f32(T v);
template <>
__device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ float to_f32<_Float16>(_Float16 v) { return (float)v; }
template <>
__device__ __forceinline__ float to_f32<__bf16>(__bf16 v) { return (float)v; }

template <typename T>
__global__ __launch_bounds__(256) void quantize_q8_1_kernel(const T* __restrict__ x, uint8_t* __restrict__ y,
                                                            int64_t kx, int64_t kx_padded, int64_t tokens) {
  const int64_t ix = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t iy = blockIdx.y;
  if (ix >= kx_padded || iy >= tokens) return;  // kx_padded is a multiple of 512: whole waves exit
  const float xi = ix < kx ? to_f32<T>(x[iy * kx + ix]) : 0.0f;
  float amax = fabsf(xi);
  float sum = xi;
#pragma unroll
  for (int mask = 16; mask > 0; mask >>= 1) {
    amax = fmaxf(amax, __shfl_xor(amax, mask, 32));
    sum += __shfl_xor(sum, mask, 32);
  }
  const float d = amax / 127.0f;
  const int8_t q = amax == 0.0f ? 0 : (int8_t)roundf(xi / d);
  uint8_t* blk = y + iy * (kx_padded / 32 * QB8_1) + (ix / 32) * QB8_1;
  blk[4 + (ix % 32)] = (uint8_t)q;
  if ((ix % 32) == 0) {
    *(uint32_t*)blk = (uint32_t)float_to_half_bits(d) | ((uint32_t)float_to_half_bits(sum) << 16);
  }
}

int launch_quantize_q8_1(const void* x, int dtype, int64_t cols, int64_t tokens, uint8_t* out, hipStream_t stream) {
  if (tokens == 0) return KTMI_OK;
  const int64_t kp = q8_1_cols_padded(cols);
  // grid.y is limited to 65535: slice the tokens
  for (int64_t t0 = 0; t0 < tokens; t0 += 65535) {
    const int64_t nt = tokens - t0 < 65535 ? tokens - t0 : 65535;
    dim3 grid((unsigned)(kp / 256), (unsigned)nt);
    uint8_t* o = out + t0 * (kp / 32 * QB8_1);
    switch (dtype) {
      case KTMI_F32: quantize_q8_1_kernel<float><<<grid, 256, 0, stream>>>((const float*)x + t0 * cols, o, cols, kp, nt); break;
      case KTMI_F16: quantize_q8_1_kernel<_Float16><<<grid, 256, 0, stream>>>((const _Float16*)x + t0 * cols, o, cols, kp, nt); break;
      case KTMI_BF16: quantize_q8_1_kernel<__bf16><<<grid, 256, 0, stream>>>((const __bf16*)x + t0 * cols, o, cols, kp, nt); break;
      default: set_error("quantize_q8_1: dtype %d", dtype); return KTMI_EINVAL;
    }
  }
  KTMI_HIP_TRY(hipGetLastError());
  return KTMI_OK;
}

// ---------------------------------------------------------------- SiLU * mul
template <typename T>
__device__ __forceinline__ T from_f32(float v) { return (T)v; }

template <typename T>
__global__ __launch_bounds__(256) void silu_and_mul_kernel(const T* __restrict__ h, int64_t R, int64_t N,
                                                           T* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= R * N) return;
  const int64_t r = i / N, n = i % N;
  const float g = to_f32<T>(h[r * 2 * N + n]);
  const float u = to_f32<T>(h[r * 2 * N + N + n]);
  out[i] = from_f32<T>(g / (1.0f + expf(-g)) * u);
}

int launch_silu_and_mul(const void* h, int dtype, int64_t R, int64_t N, void* out, hipStream_t stream) {
  const int64_t n = R * N;
  if (n == 0) return KTMI_OK;
  const unsigned g = (unsigned)((n + 255) / 256);
  switch (dtype) {
    case KTMI_F32: silu_and_mul_kernel<float><<<g, 256, 0, stream>>>((const float*)h, R, N, (float*)out); break;
    case KTMI_F16: silu_and_mul_kernel<_Float16><<<g, 256, 0, stream>>>((const _Float16*)h, R, N, (_Float16*)out); break;
    case KTMI_BF16: silu_and_mul_kernel<__bf16><<<g, 256, 0, stream>>>((const __bf16*)h, R, N, (__bf16*)out); break;
    default: set_error("silu_and_mul: dtype %d", dtype); return KTMI_EINVAL;
  }
  KTMI_HIP_TRY(hipGetLastError());
  return KTMI_OK;
}

// ---------------------------------------------------------------- combine
// hot/kt_gguf_hot.py:43-71: res[t, c] = round(sum_k fp32(round(out[t,k,c] * round(w[t,k])))),
// k ascending, one thread per 4 columns of a token.
template <typename T>
__global__ __launch_bounds__(256) void combine_kernel(const T* __restrict__ out, const float* __restrict__ w,
                                                      int64_t T_, int top_k, int64_t K, T* __restrict__ res) {
  const int64_t t = blockIdx.y;
  const int64_t c = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
  if (c >= K) return;
  float acc = 0.0f;
  for (int k = 0; k < top_k; ++k) {
    const float wk = to_f32<T>(from_f32<T>(w[t * top_k + k]));
    const float o = to_f32<T>(out[(t * top_k + k) * K + c]);
    acc += to_f32<T>(from_f32<T>(o * wk));
  }
  res[t * K + c] = from_f32<T>(acc);
}

int launch_combine(const void* out, int dtype, const float* w, int64_t T_, int64_t top_k, int64_t K, void* res,
                   hipStream_t stream) {
  if (T_ == 0 || K == 0) return KTMI_OK;
  for (int64_t t0 = 0; t0 < T_; t0 += 65535) {
    const int64_t nt = T_ - t0 < 65535 ? T_ - t0 : 65535;
    dim3 grid((unsigned)((K + 255) / 256), (unsigned)nt);
    switch (dtype) {
      case KTMI_F32:
        combine_kernel<float><<<grid, 256, 0, stream>>>((const float*)out + t0 * top_k * K, w + t0 * top_k, nt,
                                                        (int)top_k, K, (float*)res + t0 * K);
        break;
      case KTMI_F16:
        combine_kernel<_Float16><<<grid, 256, 0, stream>>>((const _Float16*)out + t0 * top_k * K, w + t0 * top_k, nt,
                                                           (int)top_k, K, (_Float16*)res + t0 * K);
        break;
      case KTMI_BF16:
        combine_kernel<__bf16><<<grid, 256, 0, stream>>>((const __bf16*)out + t0 * top_k * K, w + t0 * top_k, nt,
                                                         (int)top_k, K, (__bf16*)res + t0 * K);
        break;
      default: set_error("combine: dtype %d", dtype); return KTMI_EINVAL;
    }
  }
  KTMI_HIP_TRY(hipGetLastError());
  return KTMI_OK;
}

}  // namespace ktmi
