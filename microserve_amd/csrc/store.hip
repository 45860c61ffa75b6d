// store_kvcache for the FP8 paged cache: quantize K/V rows to e4m3fn with a
// per-(token, kv head) fp32 scale and scatter them through slot_mapping.
//
// Follows microserve/layers/fp8_kv_cache.py:11-39 (kernel) and :42-61
// (wrapper).  Layout of the work: eight lanes own one (token, kv head) pair
// and each lane holds 16 of its 128 elements of K and of V, so a lane issues
// two 16-byte loads per tensor and one 16-byte streaming store per tensor; the row
// amax is an 8-lane DPP reduction.  The division x / scale gives the bytes
// of the IEEE fp32 division with its reciprocal hoisted per row (see
// RowDivider), and the e4m3fn conversion is the hardware RNE convert on the
// clamped value, which matches torch's CPU cast bit for bit (sign kept on
// zero, subnormals kept).
#include "fp8_row.h"
#include "mskv_device.h"
#include "../../include/mskv.h"

namespace mskv {

constexpr int kStoreLanesPerRow = kHeadDim / 16;  // 8
constexpr int kStoreThreads = 256;
constexpr int kStoreRowsPerBlock = kStoreThreads / kStoreLanesPerRow;

// This lane's 16 elements of the row that starts at element `at`, as fp32
// (streaming loads: each row is read once).  16-bit inputs convert exactly;
// fp32 inputs are used as they are, as the reference's upcast leaves them.
template <typename T>
__device__ __forceinline__ void load16(const void* base, int64_t at, int sub, float* x) {
  if constexpr (sizeof(T) == 4) {
    const u32x4* p = reinterpret_cast<const u32x4*>(
        reinterpret_cast<const float*>(base) + at + sub * 16);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const u32x4 v = __builtin_nontemporal_load(p + c);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[4 * c + i] = __uint_as_float(v[i]);
    }
  } else {
    const u32x4* p = reinterpret_cast<const u32x4*>(
        reinterpret_cast<const uint16_t*>(base) + at + sub * 16);
    const u32x4 a = __builtin_nontemporal_load(p);
    const u32x4 b = __builtin_nontemporal_load(p + 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = Act<T>::to_f32((uint16_t)(a[i] & 0xFFFFu));
      x[2 * i + 1] = Act<T>::to_f32((uint16_t)(a[i] >> 16));
      x[8 + 2 * i] = Act<T>::to_f32((uint16_t)(b[i] & 0xFFFFu));
      x[8 + 2 * i + 1] = Act<T>::to_f32((uint16_t)(b[i] >> 16));
    }
  }
}

// kPacked: both inputs are contiguous, so a row's number is its place
// (the 262,144-token fill: 296 us, 298 with two strides)
template <typename T, typename SlotT, bool kPacked>
__global__ __launch_bounds__(kStoreThreads) void store_fp8_kernel(
    const void* __restrict__ key, const void* __restrict__ value,
    uint8_t* __restrict__ k_cache, uint8_t* __restrict__ v_cache,
    float* __restrict__ k_scale, float* __restrict__ v_scale,
    const SlotT* __restrict__ slots, int64_t rows, int num_kv_heads,
    int64_t num_slots, int64_t key_stride, int64_t value_stride) {
  const int sub = threadIdx.x % kStoreLanesPerRow;
  const int64_t row =
      (int64_t)blockIdx.x * kStoreRowsPerBlock + threadIdx.x / kStoreLanesPerRow;
  if (row >= rows) return;  // whole 8-lane groups leave together
  const int64_t tok = row / num_kv_heads;
  const int head = (int)(row - tok * num_kv_heads);
  const int64_t slot = (int64_t)slots[tok];

  // Tokens may lie apart (the v view of a qkv projection): the copy that
  // would pack them costs a launch, 4 to 5 us on a decode step or a chunk.
  float x[16];
  u32x4 kq, vq;
  load16<T>(key, kPacked ? row * kHeadDim : tok * key_stride + head * kHeadDim, sub, x);
  const float ks = quantize16(x, kq);
  load16<T>(value, kPacked ? row * kHeadDim : tok * value_stride + head * kHeadDim, sub, x);
  const float vs = quantize16(x, vq);

  if (slot < 0 || slot >= num_slots) return;
  // the cache rows are written once here and read by later attention
  // calls: streaming (nt) stores, 4.2% faster on the 262,144-token fill
  // (309 against 322 us, four alternations of A/B builds on one box)
  const int64_t dst = slot * num_kv_heads + head;
  __builtin_nontemporal_store(kq, reinterpret_cast<u32x4*>(k_cache + dst * kHeadDim + sub * 16));
  __builtin_nontemporal_store(vq, reinterpret_cast<u32x4*>(v_cache + dst * kHeadDim + sub * 16));
  if (sub == 0) {
    __builtin_nontemporal_store(ks, k_scale + dst);
    __builtin_nontemporal_store(vs, v_scale + dst);
  }
}

template <typename T>
static hipError_t launch_store(const void* key, const void* value, void* kc,
                               void* vc, float* ks, float* vs,
                               const void* slots, int slot_dtype,
                               int64_t num_tokens, int hk, int64_t num_slots,
                               int64_t key_stride, int64_t value_stride, hipStream_t stream) {
  const int64_t rows = num_tokens * hk;
  const int64_t blocks = (rows + kStoreRowsPerBlock - 1) / kStoreRowsPerBlock;
  auto launch = [&](auto kernel, auto* typed_slots) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kStoreThreads), 0, stream, key, value,
                       (uint8_t*)kc, (uint8_t*)vc, ks, vs, typed_slots, rows, hk, num_slots,
                       key_stride, value_stride);
  };
  const bool packed = key_stride == (int64_t)hk * kHeadDim && value_stride == key_stride;
  if (slot_dtype == MSKV_INT64) {
    const auto* p = (const int64_t*)slots;
    packed ? launch(store_fp8_kernel<T, int64_t, true>, p)
           : launch(store_fp8_kernel<T, int64_t, false>, p);
  } else {
    const auto* p = (const int32_t*)slots;
    packed ? launch(store_fp8_kernel<T, int32_t, true>, p)
           : launch(store_fp8_kernel<T, int32_t, false>, p);
  }
  return hipGetLastError();
}

}  // namespace mskv

extern "C" int mskv_store_fp8_kvcache_strided(
    const void* key, int64_t key_stride, const void* value, int64_t value_stride, void* k_cache,
    void* v_cache, float* k_scale_cache, float* v_scale_cache, const void* slot_mapping,
    int slot_dtype, int64_t num_tokens, int num_kv_heads, int head_dim, int64_t num_slots,
    int act_dtype, void* stream) {
  if (num_tokens < 0 || num_kv_heads <= 0 || num_slots < 0) return MSKV_EINVAL;
  if (slot_dtype != MSKV_INT32 && slot_dtype != MSKV_INT64) return MSKV_EINVAL;
  if (act_dtype != MSKV_FLOAT16 && act_dtype != MSKV_BFLOAT16 && act_dtype != MSKV_FLOAT32)
    return MSKV_EINVAL;
  if (head_dim != mskv::kHeadDim) return MSKV_EUNSUPPORTED;
  // rows start on 16 bytes
  const int64_t row = (int64_t)num_kv_heads * head_dim;
  const int64_t unit = act_dtype == MSKV_FLOAT32 ? 4 : 8;
  if (key_stride < row || value_stride < row || key_stride % unit != 0 ||
      value_stride % unit != 0)
    return MSKV_EINVAL;
  if (num_tokens == 0) return MSKV_OK;
  if (!key || !value || !k_cache || !v_cache || !k_scale_cache ||
      !v_scale_cache || !slot_mapping)
    return MSKV_EINVAL;
  if ((num_tokens * num_kv_heads + mskv::kStoreRowsPerBlock - 1) /
          mskv::kStoreRowsPerBlock > 0x7FFFFFFFLL)
    return MSKV_EUNSUPPORTED;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  hipError_t e;
  if (act_dtype == MSKV_BFLOAT16)
    e = mskv::launch_store<__bf16>(key, value, k_cache, v_cache, k_scale_cache, v_scale_cache,
                                   slot_mapping, slot_dtype, num_tokens, num_kv_heads,
                                   num_slots, key_stride, value_stride, s);
  else if (act_dtype == MSKV_FLOAT16)
    e = mskv::launch_store<_Float16>(key, value, k_cache, v_cache, k_scale_cache,
                                     v_scale_cache, slot_mapping, slot_dtype, num_tokens,
                                     num_kv_heads, num_slots, key_stride, value_stride, s);
  else
    e = mskv::launch_store<float>(key, value, k_cache, v_cache, k_scale_cache, v_scale_cache,
                                  slot_mapping, slot_dtype, num_tokens, num_kv_heads,
                                  num_slots, key_stride, value_stride, s);
  return (int)e;
}

extern "C" int mskv_store_fp8_kvcache(const void* key, const void* value,
                                      void* k_cache, void* v_cache,
                                      float* k_scale_cache,
                                      float* v_scale_cache,
                                      const void* slot_mapping, int slot_dtype,
                                      int64_t num_tokens, int num_kv_heads,
                                      int head_dim, int64_t num_slots,
                                      int act_dtype, void* stream) {
  const int64_t row = (int64_t)num_kv_heads * head_dim;
  return mskv_store_fp8_kvcache_strided(key, row, value, row, k_cache, v_cache, k_scale_cache,
                                        v_scale_cache, slot_mapping, slot_dtype, num_tokens,
                                        num_kv_heads, head_dim, num_slots, act_dtype, stream);
}
