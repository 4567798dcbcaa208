// A mixed batch's attention in one launch: prefill tiles (prefill_tile.h) and
// the pieces of its one-token sequences (decode_piece.h) side by side, where
// neither fills the chip. One after the other, each leaves most compute
// units idle: 48 decodes (520 piece workgroups, 12 us) beside a 300-token chunk
// behind 720 (80 prefill workgroups, 18 us). Prefill tiles come first in the
// grid: they take longest. Every workgroup runs the code it would run in the
// launch of its own kind, so the bits are the same.
#include "decode_piece.h"
#include "prefill_tile.h"

namespace pkv {

template <typename T, int D, int G>
__global__ __launch_bounds__(256, kPieceWaves<D>) void mixed_kernel(
    const T* __restrict__ q, T* __restrict__ out, T* __restrict__ kpool, T* __restrict__ vpool,
    int64_t num_blocks, int32_t n_kv_heads, float scale_log2, int32_t* status,
    int32_t prefill_blocks, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ kv_indptr, const int32_t* __restrict__ kv_indices,
    const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ prefill_plan,
    const int32_t* __restrict__ plan, int32_t stride, DecodeWorkspace w) {
  constexpr int A = PieceLds<T, D, G>::BYTES, B = PrefillLds<T, D>::BYTES;
  static_assert(kPrefillThreads == 256, "both kinds of workgroup have four waves");
  __shared__ __align__(16) unsigned char smem[A > B ? A : B];
  const int block = blockIdx.x;
  if (block < prefill_blocks) {
    prefill_tile<T, D, G>(smem, block, q, out, kpool, vpool, num_blocks, cu_q, kv_indptr,
                          kv_indices, kv_lens, prefill_plan, n_kv_heads, scale_log2, status);
  } else {
    const int bin = (block - prefill_blocks) / n_kv_heads;
    decode_piece<T, D, G>(smem, block - prefill_blocks - bin * n_kv_heads, bin, q, out, kpool,
                          vpool, num_blocks, plan, stride, n_kv_heads, scale_log2, nullptr,
                          nullptr, nullptr, w.part_o, w.part_ml, w.o_bytes, w.ml_bytes,
                          w.counters, status);
  }
}

struct MixedArgs {
  const void* q; void* out; void* kp; void* vp; int64_t nb;
  const int32_t* cu_q; const int32_t* indptr; const int32_t* indices; const int32_t* kv_lens;
  int32_t Hkv; float sl2; const int32_t* pplan; int32_t n_tiles;
  const int32_t* dplan; int32_t bins, stride; DecodeWorkspace w; int32_t* status;
};

template <typename T, int D, int G>
static void launch_mixed(const MixedArgs& a, hipStream_t s) {
  const int pre = a.n_tiles * a.Hkv;
  hipLaunchKernelGGL((mixed_kernel<T, D, G>), dim3((unsigned)(pre + a.bins * a.Hkv)), dim3(256), 0,
                     s, (const T*)a.q, (T*)a.out, (T*)a.kp, (T*)a.vp, a.nb, a.Hkv, a.sl2, a.status,
                     pre, a.cu_q, a.indptr, a.indices, a.kv_lens, a.pplan, a.dplan, a.stride, a.w);
}

typedef void (*MixedFn)(const MixedArgs&, hipStream_t);

template <typename T, int D>
static MixedFn mixed_g(int G) {
  switch (G) {
    case 1: return launch_mixed<T, D, 1>;
    case 2: return launch_mixed<T, D, 2>;
    case 4: return launch_mixed<T, D, 4>;
    case 8: return launch_mixed<T, D, 8>;
    case 16: return launch_mixed<T, D, 16>;
    default: return nullptr;
  }
}

static MixedFn mixed_fn(int32_t dtype, int32_t D, int32_t G) {
  if (dtype == PKV_DTYPE_F16)
    return D == 64 ? mixed_g<_Float16, 64>(G) : D == 128 ? mixed_g<_Float16, 128>(G) : nullptr;
  if (dtype == PKV_DTYPE_BF16)
    return D == 64 ? mixed_g<__bf16, 64>(G) : D == 128 ? mixed_g<__bf16, 128>(G) : nullptr;
  return nullptr;
}

int split_workspace(void* workspace, int64_t workspace_bytes, int32_t n_seqs, int32_t n_slots,
                    int32_t n_heads, int32_t n_kv_heads, int32_t head_dim, DecodeWorkspace* w);
int check_geometry(int32_t Hq, int32_t Hkv, int32_t D, int32_t ps, int32_t dtype);

}  // namespace pkv

using namespace pkv;

extern "C" int pkv_attend_mixed(const void* q, void* out, void* k_pool, void* v_pool,
                                int64_t num_blocks, const int32_t* cu_query_lens,
                                const int32_t* kv_indptr, const int32_t* kv_indices,
                                const int32_t* kv_lens, const int32_t* batch_indices,
                                int32_t n_seqs, int32_t n_tokens, int32_t n_heads,
                                int32_t n_kv_heads, int32_t head_dim, int32_t page_size,
                                float scale, int32_t dtype, const int32_t* prefill_plan,
                                int32_t n_tiles, int32_t q_tile, const int32_t* decode_plan,
                                int32_t n_decodes, int32_t n_work, int32_t n_slots,
                                int32_t plan_stride, void* workspace, int64_t workspace_bytes,
                                int32_t* status_word, void* stream) {
  int rc = check_geometry(n_heads, n_kv_heads, head_dim, page_size, dtype);
  if (rc) return rc;
  // Without a plan-driven decode kernel the decode call would take the batch's
  // first n_decodes sequences for the decodes.
  if (n_decodes > 0 && !pkv_decode_fast_path(n_heads, n_kv_heads, head_dim, page_size, dtype, 1))
    return fail(PKV_ERR_INVALID, "a mixed batch's decodes need the fast decode path "
                "(see pkv_decode_fast_path)");
  const int32_t G = n_heads / n_kv_heads;
  const int32_t groups = n_kv_heads / heads_per_wg(n_kv_heads);
  const uintptr_t al = (uintptr_t)q | (uintptr_t)out | (uintptr_t)k_pool | (uintptr_t)v_pool;
  MixedFn fn = page_size == 16 ? mixed_fn(dtype, head_dim, G) : nullptr;
  // One launch takes both kinds up to one prefill workgroup a compute unit.
  // Beyond, the tiles fill the chip by themselves, and the joint kernel's
  // registers and LDS (those of the larger body) would cost them occupancy.
  if (fn && scale > 0.f && prefill_plan && n_tiles > 0 && q_tile == kPrefillRows / G &&
      (int64_t)n_tiles * n_kv_heads <= compute_units() && decode_plan && n_decodes > 0 &&
      n_work > 0 && n_work % groups == 0 && n_slots >= 0 &&
      plan_stride >= kHdrInts + kStageMax * kItemInts &&
      few_pieces(n_work, plan_stride, n_kv_heads, head_dim) && al % 16 == 0) {
    MixedArgs a{q, out, k_pool, v_pool, num_blocks, cu_query_lens, kv_indptr, kv_indices, kv_lens,
                n_kv_heads, scale * kLog2e, prefill_plan, n_tiles, decode_plan, n_work / groups,
                plan_stride, {}, status_word};
    rc = split_workspace(workspace, workspace_bytes, n_decodes, n_slots, n_heads, n_kv_heads,
                         head_dim, &a.w);
    if (rc) return rc;
    fn(a, (hipStream_t)stream);
    PKV_LAUNCH_CHECK();
    return PKV_OK;
  }
  rc = pkv_attend_prefill(q, out, k_pool, v_pool, num_blocks, cu_query_lens, kv_indptr,
                          kv_indices, kv_lens, batch_indices, n_seqs, n_tokens, n_heads,
                          n_kv_heads, head_dim, page_size, scale, dtype, prefill_plan, n_tiles,
                          q_tile, status_word, stream);
  if (rc) return rc;
  return pkv_attend_decode(q, out, k_pool, v_pool, num_blocks, kv_indptr, kv_indices, kv_lens,
                           n_decodes, n_heads, n_kv_heads, head_dim, page_size, scale, dtype,
                           decode_plan, n_work, n_slots, plan_stride, nullptr, nullptr, nullptr,
                           workspace, workspace_bytes, status_word, stream);
}

static_assert(sizeof(pkv_batch) == 152, "the layout the Python binding fills");

extern "C" int pkv_append_batch(const void* batch, void* k_pool, void* v_pool, const void* k,
                                const void* v, void* stream) {
  if (!batch) return fail(PKV_ERR_INVALID, "null batch");
  const pkv_batch& b = *static_cast<const pkv_batch*>(batch);
  return pkv_append_kv(k_pool, v_pool, b.num_blocks * b.page_size, k, v, b.slot_mapping,
                       b.n_tokens, b.n_kv_heads, b.head_dim, b.dtype, b.status_word, stream);
}

extern "C" int pkv_attend_batch(const void* batch, const void* q, void* out, void* k_pool,
                                void* v_pool, float scale, const void* k_new, const void* v_new,
                                void* stream) {
  if (!batch) return fail(PKV_ERR_INVALID, "null batch");
  const pkv_batch& b = *static_cast<const pkv_batch*>(batch);
  if (!b.is_prefill)
    return pkv_attend_decode(q, out, k_pool, v_pool, b.num_blocks, b.kv_indptr, b.kv_indices,
                             b.kv_lens, b.n_seqs, b.n_heads, b.n_kv_heads, b.head_dim,
                             b.page_size, scale, b.dtype, b.decode_plan, b.n_work, b.n_slots,
                             b.plan_stride, k_new, v_new, k_new ? b.slot_mapping : nullptr,
                             b.workspace, b.workspace_bytes, b.status_word, stream);
  if (k_new || v_new)
    return fail(PKV_ERR_INVALID, "a fused append needs a batch of decodes only");
  if (b.n_decodes > 0)
    return pkv_attend_mixed(q, out, k_pool, v_pool, b.num_blocks, b.cu_query_lens, b.kv_indptr,
                            b.kv_indices, b.kv_lens, b.batch_indices, b.n_seqs, b.n_tokens,
                            b.n_heads, b.n_kv_heads, b.head_dim, b.page_size, scale, b.dtype,
                            b.prefill_plan, b.n_tiles, b.q_tile, b.decode_plan, b.n_decodes,
                            b.n_work, b.n_slots, b.plan_stride, b.workspace, b.workspace_bytes,
                            b.status_word, stream);
  return pkv_attend_prefill(q, out, k_pool, v_pool, b.num_blocks, b.cu_query_lens, b.kv_indptr,
                            b.kv_indices, b.kv_lens, b.batch_indices, b.n_seqs, b.n_tokens,
                            b.n_heads, b.n_kv_heads, b.head_dim, b.page_size, scale, b.dtype,
                            b.prefill_plan, b.n_tiles, b.q_tile, b.status_word, stream);
}
