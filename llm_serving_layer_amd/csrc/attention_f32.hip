// Paged attention over fp32 pools on gfx950 matrix cores: decode, chunked
// prefill and mixed batches, any number of query heads per KV head,
// head_dim 64 or 128, page size 16. Everything stays in fp32: the products
// run on v_mfma_f32_16x16x4_f32 (fp32 operands and accumulators), scores,
// probabilities and sums are fp32.
//
// One workgroup (8 waves) owns one KV head and 16 * NR query rows of one
// sequence (row r = token r / G, query head h * G + r % G). Its waves split
// the keys: wave w takes pages w, w + 8, ... and keeps its own running
// (max, sum, output), and the eight meet in LDS at the end (halves, quarters,
// pairs). Which wave takes a key and the order of every sum depend only on
// the key's position, so a row's bits depend neither on the batch, nor on
// the tile it falls into, nor on whether it runs as a decode or as part of a
// chunk: recomputing a preempted sequence by prefill gives the bits its
// decode steps gave.
//
// Per wave and page (lane = 16 g + n), with no LDS and no barrier:
//  * S^T = K Q^T: lane (key n, g) loads K[n][16 c + 4 g .. + 3] as one
//    16-byte load; element e of chunk c of K and of Q^T (in registers) are
//    the operands of one MFMA (the contraction runs over dims in that
//    order). Lane (row n, g) gets the scores of keys 4 g .. 4 g + 3.
//  * online softmax per row; probabilities 2^((s - m) * scale * log2 e) from
//    the raw score difference, so the exponent of the large terms is exact
//    to a few roundings whatever the scores' size.
//  * O = P V: the lane's probability of key 4 g + i is the A operand,
//    V[4 g + i][4 n + c] the B operand (one 16-byte load per row and lane:
//    whole rows, dim 4 n + c in output column n of block c).
// K of the next page is loaded beside this page's softmax and PV, V of the
// next page beside its scores (a second page in registers costs a workgroup of
// occupancy and measured slower: 81 against 72 us at 256 sequences). Q sits in
// LDS, since all waves share it: in registers it takes the second workgroup
// off the compute unit.
//
// Bound: a decode reads every K and V row once (HBM), but a 16-row MFMA tile
// holds only the G query heads of one token, so below 16 heads the fp32
// matrix rate (157 TFLOP/s) weighs as much; long chunks are bound by that
// rate alone. Measured per launch and its append (8 KV heads, 32 query heads,
// d 64): 128 sequences of lognormal mean 250, 43 us (3.1 TB/s); a 900-token
// prompt, 50 us (66 TFLOP/s); four of them behind 400 tokens, 264 us (95
// TFLOP/s). A batch of 24 such decodes and two prompts of 77 and 107 tokens
// takes 15 us in this kernel against 600 in the generic one, whose waves (one
// per token and head) read every K row three times, each lane its own row.
#include <algorithm>

#include "mfma.h"

namespace pkv {

constexpr int kF32Waves = 8;
constexpr int kF32Threads = kF32Waves * 64;
constexpr int64_t kF32WideBlocks = 512;   // two workgroups on each of 256 compute units

// One tile: the query rows of `qn` tokens of sequence `seq` from its token
// `qs` on, as pkv_plan_prefill lists them; without a plan, tile i is
// sequence i's only token (decode).
template <int D, int NR>
__global__ __launch_bounds__(kF32Threads) void f32_kernel(
    const float* __restrict__ q, float* __restrict__ out, const float* __restrict__ kpool,
    const float* __restrict__ vpool, int64_t num_blocks, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ kv_indptr, const int32_t* __restrict__ kv_indices,
    const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ plan, int32_t row_tiles,
    int32_t n_kv_heads, int32_t G, float scale, int32_t* status) {
  constexpr int PS = 16;
  constexpr int NC = D / 16;            // 16-byte chunks of a K row per lane
  constexpr int NH = D / 64;            // 64-dim halves of a V row
  constexpr int NB = D / 16;            // output blocks (16 columns each)
  constexpr int NW = kF32Waves;
  __shared__ f32x4 lds_q[NR][NC][64];
  __shared__ f32x4 lds_o[NW][NR][4][NH][64];
  __shared__ f32x2 lds_ml[NW][NR][16];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int n = lane & 15, g = lane >> 4;
  const int item = blockIdx.x / n_kv_heads;
  const int h = blockIdx.x - item * n_kv_heads;
  const int tile = item / row_tiles;
  const int r0 = (item - tile * row_tiles) * (16 * NR);   // first query row of the workgroup
  int seq = tile, qn = 1, qs = 0, q_len = 1, tok0 = tile;
  if (plan) {
    seq = plan[4 * tile];
    qs = plan[4 * tile + 1];
    qn = plan[4 * tile + 2];
    tok0 = cu_q[seq];
    q_len = cu_q[seq + 1] - tok0;
    tok0 += qs;
  }
  const int rows = qn * G;
  if (r0 >= rows) return;
  const int kv_len = kv_lens[seq];
  const int base = kv_len - q_len + qs;                   // position of the tile's first token
  const int last_tok = (min(r0 + 16 * NR, rows) - 1) / G;
  const int kv_end = min(base + last_tok + 1, kv_len);    // keys any row sees
  const int n_pages = kv_end > 0 ? (kv_end + PS - 1) / PS : 0;
  const int all_see = base + r0 / G + 1;                  // keys below this: seen by every row
  const int n_rb = min(NR, (rows - r0 + 15) / 16);        // row blocks with rows
  const int Hq = n_kv_heads * G;
  const int64_t row = (int64_t)n_kv_heads * D;
  const uint32_t rowbytes = (uint32_t)(row * sizeof(float));
  // the running max is a max of raw scores: a negative scale's sign moves
  // into Q
  const float sl2 = fabsf(scale) * kLog2e;

  // This wave's page ids, 64 at a time: lane j holds that of its page j.
  const int32_t* pages = kv_indices + kv_indptr[seq];
  auto load_ids = [&](int j0) {
    const int t = wave + NW * (j0 + lane);
    int id = t < n_pages ? pages[t] : 0;
    if (id < 0 || (int64_t)id >= num_blocks) {
      flag(status, PKV_STATUS_BAD_PAGE);
      id = 0;
    }
    return id;
  };
  int ids = load_ids(0);

  // Q^T, the same for every wave: chunk c of row block rb, lane (row n, g)
  // Q[row][16 c + 4 g .. + 3]
  for (int u = wave; u < NR * NC; u += NW) {
    const int rb = u / NC, c = u - rb * NC;
    const int r = r0 + rb * 16 + n;
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    if (r < rows) {
      const int tok = r / G;
      x = *reinterpret_cast<const f32x4*>(
          q + ((int64_t)(tok0 + tok) * Hq + h * G + (r - tok * G)) * D + 16 * c + 4 * g);
      if (scale < 0.f) x = -x;
    }
    lds_q[rb][c][lane] = x;
  }
  int pos[NR];                  // lane n's row: the last key it sees (-1: no such row)
#pragma unroll
  for (int rb = 0; rb < NR; ++rb) {
    const int r = r0 + rb * 16 + n;
    pos[rb] = r < rows ? min(base + r / G, kv_len - 1) : -1;
  }

  // Page t of the sequence into registers: its rows below kv_end (the others,
  // and every row past the last page, are outside the buffer range and read
  // as zeros).
  struct Page { f32x4 k[NC], v[4][NH]; };
  const uint32_t koff = (uint32_t)n * rowbytes + (uint32_t)(h * D + 4 * g) * 4;
  const uint32_t voff = (uint32_t)(4 * g) * rowbytes + (uint32_t)(h * D + 4 * n) * 4;
  auto rsrc = [&](const float* pool, int t) {
    const int id = __builtin_amdgcn_readlane(ids, (t / NW) & 63);
    const int live = min(PS, kv_end - t * PS);
    return ws_rsrc(const_cast<float*>(pool) + (int64_t)id * PS * row,
                   t < n_pages ? (uint32_t)live * rowbytes : 0u);
  };
  auto load_k = [&](int t, Page& p) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = rsrc(kpool, t);
#pragma unroll
    for (int c = 0; c < NC; ++c)
      p.k[c] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, koff + 64 * c, 0, 0));
  };
  auto load_v = [&](int t, Page& p) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = rsrc(vpool, t);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int b = 0; b < NH; ++b)
        p.v[i][b] = __builtin_bit_cast(
            f32x4,
            __builtin_amdgcn_raw_buffer_load_b128(rs, voff + i * rowbytes + 256 * b, 0, 0));
  };

  float m[NR], l[NR];           // of lane n's row (the same in every g)
  f32x4 o[NR][NB];              // rows 4 g + i, dim 64 (b / 4) + 4 n + b % 4
#pragma unroll
  for (int rb = 0; rb < NR; ++rb) {
    m[rb] = -INFINITY;
    l[rb] = 0.f;
#pragma unroll
    for (int b = 0; b < NB; ++b) o[rb][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // 2^((a - b) * scale log2 e), 0 for a = -inf (no key seen yet)
  auto weight = [&](float a, float b) {
    return a == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((a - b) * sl2);
  };
  auto scores = [&](const Page& p, f32x4* s) __attribute__((always_inline)) {
    asm volatile("" ::: "memory");   // Q stays in LDS: hoisted, it would cost its registers
#pragma unroll
    for (int rb = 0; rb < NR; ++rb) {
      s[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (rb < n_rb) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const f32x4 x = lds_q[rb][c][lane];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            s[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.k[c][e], x[e], s[rb], 0, 0, 0);
        }
      }
    }
  };
  auto softmax_pv = [&](int t, const Page& p, const f32x4* s) __attribute__((always_inline)) {
    // A key that only later rows see meets the earlier rows with probability
    // 0; if its V row holds an infinity or NaN, 0 * V would reach them.
    bool odd_v = false;
    if (t * PS + PS > all_see) {
      float z = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int b = 0; b < NH; ++b)
#pragma unroll
          for (int c = 0; c < 4; ++c) z = __builtin_fmaf(p.v[i][b][c], 0.f, z);
      odd_v = __builtin_amdgcn_ballot_w64(!(z == 0.f)) != 0;
    }
#pragma unroll
    for (int rb = 0; rb < NR; ++rb) {
      if (rb >= n_rb) continue;
      bool see[4];
      float mx = m[rb];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        see[i] = t * PS + 4 * g + i <= pos[rb];
        mx = fmaxf(mx, see[i] ? s[rb][i] : -INFINITY);
      }
      mx = max_x32(max_x16(mx));
      // (a row whose max stays has a factor of exactly 1: skipping it
      // changes no bits)
      if (__builtin_amdgcn_ballot_w64(mx > m[rb])) {
        const float a = weight(m[rb], mx);
        l[rb] *= a;
        m[rb] = mx;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float ai = __shfl(a, 4 * g + i, 64);   // row 4 g + i's factor
#pragma unroll
          for (int b = 0; b < NB; ++b) o[rb][b][i] *= ai;
        }
      }
      const float ref = mx == -INFINITY ? 0.f : mx;
      float pr[4], ls = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pr[i] = see[i] ? __builtin_amdgcn_exp2f((s[rb][i] - ref) * sl2) : 0.f;
        ls += pr[i];
      }
      l[rb] += sum_x32(sum_x16(ls));
      if (!odd_v) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int b = 0; b < NB; ++b)
            o[rb][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(pr[i], p.v[i][b / 4][b % 4],
                                                            o[rb][b], 0, 0, 0);
      } else {   // key by key, each only into the rows that see it
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll 1
          for (int gs = 0; gs < 4; ++gs) {
            const int key = t * PS + 4 * gs + i;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float pj = __shfl(pr[i], 16 * gs + 4 * g + j, 64);
              const bool seen = key <= __shfl(pos[rb], 4 * g + j, 64);
#pragma unroll
              for (int b = 0; b < NB; ++b) {
                const float v = __shfl(p.v[i][b / 4][b % 4], 16 * gs + n, 64);
                o[rb][b][j] = seen ? __builtin_fmaf(pj, v, o[rb][b][j]) : o[rb][b][j];
              }
            }
          }
      }
    }
  };

  f32x4 s[NR];
  Page p;
  load_k(wave, p);
  load_v(wave, p);
  __syncthreads();   // Q
  for (int t = wave; t < n_pages; t += NW) {
    if ((((t + NW) / NW) & 63) == 0) ids = load_ids((t + NW) / NW);
    scores(p, s);
    load_k(t + NW, p);
    softmax_pv(t, p, s);
    load_v(t + NW, p);
  }

  // The waves meet in LDS: every wave leaves its (max, sum, output), then the
  // (row block, row of four, half) units are shared out and each sums the
  // waves' outputs in wave order. Waves that had no page left nothing.
#pragma unroll
  for (int rb = 0; rb < NR; ++rb) {
    if (g == 0) lds_ml[wave][rb][n] = f32x2{m[rb], l[rb]};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int b = 0; b < NH; ++b)
        lds_o[wave][rb][i][b][lane] =
            f32x4{o[rb][4 * b][i], o[rb][4 * b + 1][i], o[rb][4 * b + 2][i], o[rb][4 * b + 3][i]};
  }
  __syncthreads();
  const int nw = min(NW, n_pages);
  for (int u = wave; u < NR * 4 * NH; u += NW) {
    const int b = u % NH, i = u / NH % 4, rb = u / NH / 4;
    const int r = r0 + rb * 16 + 4 * g + i;
    float mx = -INFINITY;
    for (int w = 0; w < nw; ++w) mx = fmaxf(mx, lds_ml[w][rb][4 * g + i][0]);
    float ls = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < nw; ++w) {
      const f32x2 ml = lds_ml[w][rb][4 * g + i];
      const float a = weight(ml[0], mx);
      ls += a * ml[1];
      acc += a * lds_o[w][rb][i][b][lane];
    }
    if (r < rows) {
      const int tok = r / G;
      // (a row that sees no key, kv_len 0, is 0)
      *reinterpret_cast<f32x4*>(
          out + ((int64_t)(tok0 + tok) * Hq + h * G + (r - tok * G)) * D + 64 * b + 4 * n) =
          acc * (min(base + tok, kv_len - 1) >= 0 ? 1.f / ls : 0.f);
    }
  }
}

static bool f32_geometry(int32_t D, int32_t page_size) {
  return page_size == 16 && (D == 64 || D == 128);
}

// Tokens a plan tile should hold: the 32 query rows of one workgroup (a larger
// tile is served too, by several workgroups, those past its end idle).
int f32_q_tile(int32_t Hq, int32_t Hkv, int32_t D, int32_t page_size) {
  if (Hkv <= 0 || Hq <= 0 || Hq % Hkv || !f32_geometry(D, page_size)) return 0;
  return std::max(1, 32 / (Hq / Hkv));
}

// Runs the matrix-core kernel for an fp32 pool where it applies (*ran);
// otherwise the caller takes the generic kernel. `plan` is null for a decode
// batch (n_tiles sequences of one token).
int run_f32(const void* q, void* out, const void* kp, const void* vp, int64_t nb,
            const int32_t* cu_q, const int32_t* indptr, const int32_t* indices,
            const int32_t* kv_lens, int32_t Hq, int32_t Hkv, int32_t D, int32_t page_size,
            float scale, const int32_t* plan, int32_t n_tiles, int32_t q_tile, int32_t* status,
            hipStream_t s, bool* ran) {
  *ran = false;
  if (!f32_geometry(D, page_size) || n_tiles <= 0 || q_tile <= 0) return PKV_OK;
  // 16-byte accesses; a page's rows within a 31-bit buffer range
  if (((uintptr_t)q | (uintptr_t)out | (uintptr_t)kp | (uintptr_t)vp) % 16) return PKV_OK;
  if ((int64_t)Hkv * D * 4 * page_size > 0x7fffffffLL) return PKV_OK;
  const int32_t G = Hq / Hkv;
  // 32 rows a workgroup share each K and V load: 5% faster once they fill the
  // chip twice over (900-token prompt: 50.1 against 52.8 us; 600: 30.4 against
  // 31.3). Below that 16 rows spread the same products over twice the
  // compute units (20 tokens behind 1000: 18.1 against 28.6 us; 128: 21.8
  // against 32.0). The bits are the same either way.
  const int64_t rows = (int64_t)q_tile * G;
  const int64_t wide = (rows + 31) / 32;
  const bool one = rows <= 16 || (int64_t)n_tiles * wide * Hkv < kF32WideBlocks;
  const int64_t row_tiles = one ? (rows + 15) / 16 : wide;
  const int64_t blocks = (int64_t)n_tiles * row_tiles * Hkv;
  if (blocks > 0x7fffffffLL) return PKV_OK;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kF32Threads), 0, s, (const float*)q,
                       (float*)out, (const float*)kp, (const float*)vp, nb, cu_q, indptr,
                       indices, kv_lens, plan, (int32_t)row_tiles, Hkv, G, scale, status);
  };
  if (D == 64 && one) go(f32_kernel<64, 1>);
  else if (D == 64) go(f32_kernel<64, 2>);
  else if (one) go(f32_kernel<128, 1>);
  else go(f32_kernel<128, 2>);
  PKV_LAUNCH_CHECK();
  *ran = true;
  return PKV_OK;
}

}  // namespace pkv
