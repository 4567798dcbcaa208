// Chunked-prefill attention: prefill_tile.h, one tile and KV head a workgroup.
#include "prefill_tile.h"

namespace pkv {

template <typename T, int D, int G>
__global__ __launch_bounds__(kPrefillThreads) void prefill_kernel(
    const T* __restrict__ q, T* __restrict__ out, const T* __restrict__ kpool,
    const T* __restrict__ vpool, int64_t num_blocks, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ kv_indptr, const int32_t* __restrict__ kv_indices,
    const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ plan,
    int32_t n_kv_heads, float scale_log2, int32_t* status) {
  __shared__ __align__(16) unsigned char smem[PrefillLds<T, D>::BYTES];
  prefill_tile<T, D, G>(smem, blockIdx.x, q, out, kpool, vpool, num_blocks, cu_q, kv_indptr,
                        kv_indices, kv_lens, plan, n_kv_heads, scale_log2, status);
}

template <typename T, int D, int G>
static void launch_prefill(const void* q, void* out, const void* kp, const void* vp, int64_t nb,
                           const int32_t* cu_q, const int32_t* indptr, const int32_t* indices,
                           const int32_t* kv_lens, const int32_t* plan, int32_t n_tiles,
                           int32_t Hkv, float sl2, int32_t* status, hipStream_t s) {
  hipLaunchKernelGGL((prefill_kernel<T, D, G>), dim3((unsigned)(n_tiles * Hkv)), dim3(kPrefillThreads), 0,
                     s, (const T*)q, (T*)out, (const T*)kp, (const T*)vp, nb, cu_q, indptr,
                     indices, kv_lens, plan, Hkv, sl2, status);
}

typedef void (*PrefillFn)(const void*, void*, const void*, const void*, int64_t, const int32_t*,
                          const int32_t*, const int32_t*, const int32_t*, const int32_t*,
                          int32_t, int32_t, float, int32_t*, hipStream_t);

template <typename T, int D>
static PrefillFn prefill_g(int G) {
  switch (G) {
    case 1: return launch_prefill<T, D, 1>;
    case 2: return launch_prefill<T, D, 2>;
    case 4: return launch_prefill<T, D, 4>;
    case 8: return launch_prefill<T, D, 8>;
    case 16: return launch_prefill<T, D, 16>;
    default: return nullptr;
  }
}

template <typename T>
static PrefillFn prefill_d(int D, int G) {
  switch (D) {
    case 64: return prefill_g<T, 64>(G);
    case 128: return prefill_g<T, 128>(G);
    default: return nullptr;
  }
}

int f32_q_tile(int32_t Hq, int32_t Hkv, int32_t D, int32_t page_size);  // attention_f32.hip

// The MFMA prefill kernel for this geometry, or null (generic kernel).
PrefillFn fast_prefill(int32_t dtype, int32_t Hq, int32_t Hkv, int32_t D, int32_t page_size) {
  if (page_size != 16 || Hkv <= 0 || Hq % Hkv) return nullptr;
  const int G = Hq / Hkv;
  if (dtype == PKV_DTYPE_F16) return prefill_d<_Float16>(D, G);
  if (dtype == PKV_DTYPE_BF16) return prefill_d<__bf16>(D, G);
  return nullptr;
}

}  // namespace pkv

using namespace pkv;

extern "C" int pkv_prefill_q_tile(int32_t n_heads, int32_t n_kv_heads, int32_t head_dim,
                                  int32_t page_size, int32_t dtype) {
  if (fast_prefill(dtype, n_heads, n_kv_heads, head_dim, page_size))
    return kPrefillRows / (n_heads / n_kv_heads);
  return dtype == PKV_DTYPE_F32 ? f32_q_tile(n_heads, n_kv_heads, head_dim, page_size) : 0;
}

namespace pkv {
int run_fast_prefill(const void* q, void* out, const void* kp, const void* vp, int64_t nb,
                     const int32_t* cu_q, const int32_t* indptr, const int32_t* indices,
                     const int32_t* kv_lens, int32_t Hq, int32_t Hkv, int32_t D,
                     int32_t page_size, float scale, int32_t dtype, const int32_t* plan,
                     int32_t n_tiles, int32_t q_tile, int32_t* status, hipStream_t s,
                     bool* ran) {
  *ran = false;
  PrefillFn fn = fast_prefill(dtype, Hq, Hkv, D, page_size);
  if (!fn || !plan || n_tiles <= 0 || q_tile != kPrefillRows / (Hq / Hkv) || !(scale > 0.f))
    return PKV_OK;
  if ((int64_t)n_tiles * Hkv > 0x7fffffffLL) return fail(PKV_ERR_INVALID, "too many tiles");
  if (((uintptr_t)q | (uintptr_t)kp | (uintptr_t)vp) % 16)
    return fail(PKV_ERR_INVALID, "q and pools must be 16-byte aligned");
  fn(q, out, kp, vp, nb, cu_q, indptr, indices, kv_lens, plan, n_tiles, Hkv, scale * kLog2e,
     status, s);
  PKV_LAUNCH_CHECK();
  *ran = true;
  return PKV_OK;
}
}  // namespace pkv
