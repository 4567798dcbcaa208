// What the decode kernels share: the plan's layout, the merge of cut sequences,
// and the body of the small-batch kernel (a workgroup per piece and KV head),
// which mixed.hip runs beside prefill tiles in one launch.
#pragma once

#include "mfma.h"

namespace pkv {

constexpr int kMaxPartPages = 64;   // bound on part_pages (ABI)
constexpr int kMaxWaves = 4;        // KV heads (one per wave) per workgroup
constexpr int kPageIdBits = 27;     // a plan page word: id | (live rows - 1) << 27 | bad << 31
constexpr int kHdrInts = 4;         // bin header {n_items, n_pages, 0, 0}
constexpr int kItemInts = 8;        // {seq, n_pages, first token, kv_len, slot, n_pieces,
                                    //  first slot, flags}
constexpr int kItemLast = 1;        // flags: the piece holds its sequence's last page
constexpr int kRowShift = 1;        // flags: the sequence's row of q, out, k_new, v_new and
                                    // slot_mapping from this bit on (its index, unless the
                                    // batch is part of a larger one)
constexpr int kStageMax = 8;        // items staged in LDS at a time (at most)
constexpr int kPlanTail = 64;       // zero ints after the last bin (words read past its end)
constexpr int kMinTail = 4;         // a remainder of a cut below this (and below half a
                                    // piece) joins the piece before it

// KV heads per workgroup: one wave each, at most kMaxWaves, dividing Hkv.
__host__ __device__ static inline int heads_per_wg(int hkv) { return hkv % 4 == 0 ? 4 : hkv % 2 == 0 ? 2 : 1; }

// Layout of one partition's partial output: per (slot, KV head), NGR groups
// of 4 head rows, each NDB dim blocks of 16 lanes x 4 rows (float4 per
// lane) -- exactly the MFMA accumulator layout, so a wave stores and loads
// it with one 16-byte access per lane and dim block.
template <int D, int G> struct PartLayout {
  static constexpr int NGR = (G + 3) / 4;
  static constexpr int NDB = D / 16;
  static constexpr int FLOATS = NGR * NDB * 64;  // per (slot, KV head)
};

// Split-K merge for one KV head h of a sequence (row orow of out), run by the wave that
// published the last partial, or by the sequence's last piece with its own
// partial still in registers (`own`). Lanes run over partitions for each
// head row's max M and sum L; then, 64 partitions at a time, the weights
// 2^(m_s - M) go to this wave's LDS scratch as [partition][GS rows], and the
// partial outputs are read in the producers' own layout: lane (n, g) takes
// row group rg = g % NGR of the chunk's partitions cn - 1 - j for j = g / NGR,
// g / NGR + SPLIT, ..., and the SPLIT lane groups that share a row group are
// summed by shuffles at the end. The chunk's last partition goes to lane
// group 0, whose lanes (n, rg) hold exactly that row group of an own
// partial in their accumulators, so `own` needs no data movement for o and
// enters the sums in the same place with the same bits a store and load
// would give. The summation order depends only on the partition count, so
// the result does not depend on the batch or on which wave merges.
// NBW dim blocks from b0 on are merged (all of them by default).
template <typename T, int D, int G, int NBW = D / 16>
__device__ __forceinline__ void merge_head(T* __restrict__ out, float* wts, int orow, int h,
                                           int n_kv_heads, int nparts, int slot0,
                                           __amdgpu_buffer_rsrc_t ro, __amdgpu_buffer_rsrc_t rm,
                                           bool own, const f32x4* own_o, float own_m,
                                           float own_l, int b0 = 0) {
  typedef PartLayout<D, G> PL;
  constexpr int NDB = D / 16;
  constexpr int NGR = PL::NGR;
  constexpr int SPLIT = 4 / NGR;
  constexpr int GS = 4 * NGR;              // weight rows per partition (>= G)
  const int lane = threadIdx.x & 63;
  const int n = lane & 15, g = lane >> 4;
  const int rg = g % NGR, so = g / NGR;
  const int Hq = n_kv_heads * G;
  const int own_part = own ? nparts - 1 : -1;
  // (m, l) of every head of partitions c0 + lane; an own partition's come
  // from lanes 0 .. G - 1, which hold head r's running max and sum
  auto load_ml = [&](int c0, float* mr, float* lr) {
    const bool mine = c0 + lane == own_part;
    const bool ok = c0 + lane < nparts && !mine;
    const uint32_t b2 = (uint32_t)(((int64_t)(slot0 + (ok ? c0 + lane : 0)) * Hq + h * G) * 8);
#pragma unroll
    for (int r = 0; r < G; ++r) {
      const f32x2 ml =
          __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rm, b2 + 8 * r, 0, kSc1));
      const float m_own = lane_value(own_m, r), l_own = lane_value(own_l, r);
      mr[r] = ok ? ml[0] : mine ? m_own : -INFINITY;
      lr[r] = ok ? ml[1] : mine ? l_own : 0.f;
    }
  };
  // Partition c0 + cn - 1 - j of this lane's row group (j < cn).
  auto load_part = [&](int c0, int j, f32x4* v) {
    const int cn = min(64, nparts - c0);
    const int pi = c0 + cn - 1 - (j < cn ? j : 0);
    const bool mine = pi == own_part;   // then j == 0: lane group 0
    const uint32_t off = (uint32_t)(((int64_t)(slot0 + pi) * n_kv_heads + h) * PL::FLOATS * 4);
#pragma unroll
    for (int b = 0; b < NBW; ++b)
      v[b] = j >= cn ? f32x4{0.f, 0.f, 0.f, 0.f}
             : mine ? own_o[b]
                    : __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                    ro, off + ((rg * NDB + b0 + b) * 16 + n) * 16, 0,
                                                    kSc1));
  };
  // The first partitions do not depend on the maximum: their loads go out
  // with the (m, l) loads, so a sequence of up to SPLIT partitions merges in
  // one round trip.
  f32x4 v[NBW];
  load_part(0, so, v);
  float mr[G], lr[G], M[G], L[G];
#pragma unroll
  for (int r = 0; r < G; ++r) { M[r] = -INFINITY; L[r] = 0.f; }
  for (int c0 = 0; c0 < nparts; c0 += 64) {
    load_ml(c0, mr, lr);
#pragma unroll
    for (int r = 0; r < G; ++r) M[r] = fmaxf(M[r], wave_max(mr[r]));
  }
  f32x4 acc[NBW];
#pragma unroll
  for (int b = 0; b < NBW; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < nparts; c0 += 64) {
    if (nparts > 64) load_ml(c0, mr, lr);  // else still in registers
#pragma unroll
    for (int r = 0; r < GS; ++r) {
      float wv = 0.f;
      if (r < G) {
        wv = c0 + lane < nparts ? __builtin_amdgcn_exp2f(mr[r] - M[r]) : 0.f;
        L[r] += wave_sum(wv * lr[r]);
      }
      wts[lane * GS + r] = wv;
    }
    wave_lds_sync();
    const int cn = min(64, nparts - c0);
    for (int j = so; j < cn; j += SPLIT) {
      if (c0 > 0 || j > so) load_part(c0, j, v);
      const f32x4 wr = *reinterpret_cast<const f32x4*>(wts + (cn - 1 - j) * GS + 4 * rg);
#pragma unroll
      for (int b = 0; b < NBW; ++b) acc[b] += wr * v[b];
    }
    wave_lds_sync();  // the next chunk rewrites the weights
  }
#pragma unroll
  for (int b = 0; b < NBW; ++b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (SPLIT >= 4) acc[b][i] = sum_x16(acc[b][i]);
      if (SPLIT >= 2) acc[b][i] = sum_x32(acc[b][i]);
    }
  }
  if (so == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 4 * rg + i;
      float lr_ = L[0];
#pragma unroll
      for (int rr = 1; rr < G; ++rr)  // static indices keep L in registers
        if (r == rr) lr_ = L[rr];
      if (r < G) {
        const float inv = 1.f / lr_;   // one division per row, not per element
#pragma unroll
        for (int b = 0; b < NBW; ++b)
          out[((int64_t)orow * Hq + h * G + r) * D + 16 * (b0 + b) + n] = (T)(acc[b][i] * inv);
      }
    }
  }
}

// ---------------------------------------------------- one piece a workgroup ---
// The same pieces with the same arithmetic for batches of few pieces: a
// workgroup of four waves takes one KV head of one piece. With few pieces
// decode_kernel's time is not memory but one wave's walk through a piece,
// page after page, at ~200 instructions a page and no other wave on its SIMD
// (17 pages: 11 us of a 16 us launch). Here all of a piece's loads go out at
// once and the work of a page is spread without changing the order of
// any sum, so a sequence's bits do not depend on which kernel its batch took:
//  * the waves share the pages (page j: wave j % 4) for K (straight into
//    registers as the QK operand), scores and row maxima, which meet in LDS;
//  * every wave replays the running reference over the pages (it moves
//    exactly where it does in decode_kernel), then takes its pages'
//    probabilities, which go to LDS with their sums;
//  * the waves share the output dims for PV: each walks all pages in order
//    for its own dims (V in LDS), and merges those dims of a cut sequence.
// One 1371-token sequence (5 pieces, 8 KV heads, 32 query heads, d 64): 16.4
// us a launch in decode_kernel; 9.4 here; 16 layers of such steps 271 -> 157 us.
template <typename T, int D, int G> struct PieceLds {
  static constexpr int CH = 20;                   // pages staged at a time: any piece of
                                                  // the default cut (17 + a folded tail)
  static constexpr int VPAGE = 16 * D * (int)sizeof(T);
  static constexpr int V = CH * VPAGE;            // V rows, chunks swizzled
  static constexpr int P = CH * 512;              // probabilities, lane order
  static constexpr int MS = 16 * CH * 4;          // per head: page maxima (sums)
  static constexpr int BYTES = V + P + 2 * MS + 16;
  static_assert(4 * 64 * 16 * PartLayout<D, G>::NGR <= V, "the merge's weights fit");
};

template <typename T, int D, int G>
__device__ __forceinline__ void decode_piece(
    unsigned char* smem, int h, int bin,
    const T* __restrict__ q, T* __restrict__ out, T* __restrict__ kpool, T* __restrict__ vpool,
    int64_t num_blocks, const int32_t* __restrict__ plan, int32_t stride, int32_t n_kv_heads,
    float scale_log2, const T* __restrict__ k_new, const T* __restrict__ v_new,
    const int32_t* __restrict__ slot_mapping, float* part_o, float* part_ml, uint32_t o_bytes,
    uint32_t ml_bytes, int32_t* counters, int32_t* status) {
#pragma clang fp contract(off)
  typedef typename Mma<T>::vec8 vec8;
  typedef typename Mma<T>::vec4 vec4;
  typedef PartLayout<D, G> PL;
  typedef PieceLds<T, D, G> L;
  constexpr int PS = 16;
  constexpr int NCH = D / 32;          // QK MFMA k-chunks per head row
  constexpr int NDB = D / 16;          // PV dim blocks
  constexpr int NBW = NDB / 4;         // of a wave
  constexpr int RB = D * (int)sizeof(T);
  constexpr int CPR = RB / 16;         // 16-byte chunks per head row
  constexpr int RPI = 64 / CPR;        // rows per wave load instruction
  constexpr int NLD = PS / RPI;        // V load instructions per page
  constexpr int CH = L::CH, PW = CH / 4;   // pages a chunk, of a wave
  constexpr int NGR = PL::NGR;

  unsigned char* vt = smem;
  unsigned char* pt = smem + L::V;
  float* mxs = reinterpret_cast<float*>(smem + L::V + L::P);   // [head][page]
  float* lss = mxs + 16 * CH;
  int* arrived = reinterpret_cast<int*>(lss + 16 * CH);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int Hq = n_kv_heads * G;
  const uint32_t frow = (uint32_t)(n_kv_heads * RB);
  const int64_t row_elems = (int64_t)n_kv_heads * D;
  const int lrow0 = lane / CPR, lc = lane % CPR;

  const int32_t* bp = plan + (int64_t)bin * stride;
  const int32_t* words = bp + kHdrInts;
  const __amdgpu_buffer_rsrc_t ro = ws_rsrc(part_o, o_bytes);
  const __amdgpu_buffer_rsrc_t rm = ws_rsrc(part_ml, ml_bytes);

  // One item where the launch follows few_pieces; any plan is served. (The
  // count, the item and its words come in one round trip; the slot below a
  // bin's last item still lies inside its plan block.)
  const int n_items = bp[0];
  int p0 = 0;
  for (int item = 0;; ++item) {
    const int32_t* it = bp + stride - (int64_t)(item + 1) * kItemInts;
    const int seq = it[0], np = it[1], tok0 = it[2], kv = it[3], slot = it[4], nparts = it[5],
              slot0 = it[6];
    const int row = it[7] >> kRowShift;
    const bool fuse = k_new != nullptr && (it[7] & kItemLast);
    // the first chunk's page words, word i in lane i (reads past the bin's
    // words stay inside the plan: kPlanTail)
    int wd = words[p0 + lane];
    asm volatile("" ::"s"(seq), "s"(np), "s"(kv), "s"(it[7]), "s"(n_items));
    if (item >= n_items) break;

    // Q^T, the QK B operand (column n = query head h*G + n, zero beyond G)
    vec8 qb[NCH], kx[NCH], vx{};
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      qb[c] = vec8{};
      kx[c] = vec8{};
      if (n < G)
        qb[c] = *reinterpret_cast<const vec8*>(q + ((int64_t)row * Hq + h * G + n) * D + c * 32 +
                                               g * 8);
    }
    // the new row: K as the QK A operand has it, V in 16-byte chunks
    int new_slot = 0;
    if (fuse) {
      const int64_t at = (int64_t)row * row_elems + h * D;
#pragma unroll
      for (int c = 0; c < NCH; ++c)
        kx[c] = *reinterpret_cast<const vec8*>(k_new + at + c * 32 + g * 8);
      vx = *reinterpret_cast<const vec8*>(v_new + at + lc * 8);
      new_slot = slot_mapping[row];
    }

    f32x4 o[NBW];
    float m_run = -INFINITY, l_run = 0.f;  // per head column n (replicated over g)
#pragma unroll
    for (int b = 0; b < NBW; ++b) o[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Lane 4 g + i's value of v, in every lane of group g (1 for padding rows)
    auto from_lane = [&](float v, int i) __attribute__((always_inline)) {
      float x = 1.f;
#pragma unroll
      for (int gg = 0; 4 * gg < G; ++gg) x = g == gg ? lane_value(v, 4 * gg + i) : x;
      return x;
    };

    bool bad = false;
    for (int c0 = 0; c0 < np; c0 += CH) {
      const int cn = min(CH, np - c0);
      if (c0 > 0) wd = words[p0 + c0 + lane];
      bad |= lane < cn && wd < 0;   // an id outside the pool: the plan put page 0
      // This wave's pages c0 + 4 i + wave: K into registers, lane (row n, g)
      // its chunks 4 c + g, V into LDS. Only rows below kv_len are inside a
      // page's buffer range, and nothing past the chunk's last page.
      vec8 kr[PW][NCH];
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int j = 4 * i + wave;
        const bool in = j < cn;
        const uint32_t w = (uint32_t)__builtin_amdgcn_readlane(wd, j);
        const int64_t at = in ? (int64_t)(w & ((1u << kPageIdBits) - 1)) * PS * row_elems : 0;
        const uint32_t range = in ? (((w >> kPageIdBits) & 15u) + 1u) * frow : 0u;
        const __amdgpu_buffer_rsrc_t rk = ws_rsrc(kpool + at, range);
        const __amdgpu_buffer_rsrc_t rv = ws_rsrc(vpool + at, range);
#pragma unroll
        for (int c = 0; c < NCH; ++c)
          kr[i][c] = __builtin_bit_cast(
              vec8, __builtin_amdgcn_raw_buffer_load_b128(
                        rk, (uint32_t)n * frow + (uint32_t)(h * RB + (4 * c + g) * 16), 0, kNt));
        if (in) {
#pragma unroll
          for (int k = 0; k < NLD; ++k) {
            // position lc of a row takes the chunk the swizzle stores there
            const int r = k * RPI + lrow0;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rv, (__attribute__((address_space(3))) void*)(vt + j * L::VPAGE + k * 1024), 16,
                (uint32_t)r * frow + (uint32_t)(h * RB + (((lc ^ xr(r)) & 7) | (lc & ~7)) * 16), 0,
                0, kNt);
          }
        }
      }
      // The sequence's last page: the new row goes to its slot and, when
      // slot_mapping agrees with the page table, into the loaded copy.
      const bool tail = c0 + cn == np;
      const int jt = cn - 1;
      const uint32_t wt = (uint32_t)__builtin_amdgcn_readlane(wd, jt);
      bool patch = false, store = false;
      const int tl = (kv - 1) % PS;
      if (fuse && tail && wave == (jt & 3)) {
        if (new_slot < 0 || (int64_t)new_slot >= num_blocks * PS) {
          if (lane == 0) flag(status, PKV_STATUS_BAD_SLOT);
        } else {
          patch = (int64_t)new_slot == (int64_t)(wt & ((1u << kPageIdBits) - 1)) * PS + tl;
          store = true;
#pragma unroll
          for (int i = 0; i < PW; ++i) {
            if (patch && 4 * i + wave == jt && n == tl) {
#pragma unroll
              for (int c = 0; c < NCH; ++c) kr[i][c] = kx[c];
            }
          }
        }
      }

      // scores and row maxima of this wave's pages
      f32x4 sc[PW];
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        sc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NCH; ++c) sc[i] = Mma<T>::qk(kr[i][c], qb[c], sc[i]);
      }
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int j = 4 * i + wave;
        const int tp = tok0 + (c0 + j) * PS;
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sc[i][e] = tp + 4 * g + e < kv ? sc[i][e] * scale_log2 : -INFINITY;
          mx = fmaxf(mx, sc[i][e]);
        }
        mx = max_x32(max_x16(mx));
        // (a page past the chunk's last moves nothing)
        if (g == 0) mxs[n * CH + j] = j < cn ? mx : -INFINITY;
      }
      // V has landed; the rows past kv_len are cleared (their probabilities
      // are 0, but what LDS holds there need not be finite)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (tail && wave == (jt & 3)) {
        const int live = ((wt >> kPageIdBits) & 15) + 1;
#pragma unroll
        for (int k = 0; k < NLD; ++k) {
          const int r = k * RPI + lrow0;
          unsigned char* at = vt + jt * L::VPAGE + swz<RB>(r, lc * 8);
          if (patch && r == tl) *reinterpret_cast<vec8*>(at) = vx;
          if (r >= live) *reinterpret_cast<vec8*>(at) = vec8{};
        }
      }
      __syncthreads();
      if (store) {   // (here, so that the wait for V is not a wait for it)
        const int64_t dst = (int64_t)new_slot * row_elems + h * D;
        if (n == 0) {
#pragma unroll
          for (int c = 0; c < NCH; ++c)
            *reinterpret_cast<vec8*>(kpool + dst + c * 32 + g * 8) = kx[c];
        }
        if (lane < CPR) *reinterpret_cast<vec8*>(vpool + dst + lc * 8) = vx;
      }

      // The running reference over the chunk's pages: it moves at a page when
      // some head's maximum is more than 8 above it. mv: bit j set where it
      // moves; m_at: its value at this wave's pages.
      float mx[CH];
#pragma unroll
      for (int j = 0; j < CH; j += 4) {
        const f32x4 t = *reinterpret_cast<const f32x4*>(mxs + n * CH + j);
#pragma unroll
        for (int e = 0; e < 4; ++e) mx[j + e] = t[e];
      }
      float m = m_run, m_at[PW];
      uint32_t mv = 0;
      if (__builtin_amdgcn_ballot_w64(mx[0] > m + 8.f)) {
        m = fmaxf(m, mx[0]);
        mv = 1;
      }
      float top = mx[1];
#pragma unroll
      for (int j = 2; j < CH; ++j) top = fmaxf(top, mx[j]);
      if (!__builtin_amdgcn_ballot_w64(top > m + 8.f)) {   // no later page moves it
#pragma unroll
        for (int i = 0; i < PW; ++i) m_at[i] = m;
      } else {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
          if (j > 0 && __builtin_amdgcn_ballot_w64(mx[j] > m + 8.f)) {
            m = fmaxf(m, mx[j]);
            mv |= 1u << j;
          }
          if ((j & 3) == wave) m_at[j / 4] = m;
        }
      }
      // probabilities and their sums
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int j = 4 * i + wave;
        vec4 pr;
        float ls = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = __builtin_amdgcn_exp2f(sc[i][e] - m_at[i]);
          ls += x;
          pr[e] = (T)x;
        }
        ls = sum_x32(sum_x16(ls));
        *reinterpret_cast<vec4*>(pt + j * 512 + lane * 8) = pr;
        if (g == 0) lss[n * CH + j] = ls;
      }
      __syncthreads();

      // PV over the chunk's pages in order, this wave's dims
      float lsum[CH];
#pragma unroll
      for (int j = 0; j < CH; j += 4) {
        const f32x4 t = *reinterpret_cast<const f32x4*>(lss + n * CH + j);
#pragma unroll
        for (int e = 0; e < 4; ++e) lsum[j + e] = t[e];
      }
      auto move = [&](int j) __attribute__((always_inline)) {
        const float m_new = fmaxf(m_run, mx[j]);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= alpha;
        m_run = m_new;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = from_lane(alpha, e);
#pragma unroll
          for (int b = 0; b < NBW; ++b) o[b][e] *= a;
        }
      };
      auto read_page = [&](int j, vec4& pr, vec4* v) __attribute__((always_inline)) {
        pr = *reinterpret_cast<const vec4*>(pt + j * 512 + lane * 8);
#pragma unroll
        for (int b = 0; b < NBW; ++b)
          v[b] = __builtin_bit_cast(
              vec4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(
                        vt + j * L::VPAGE +
                        swz<RB>(4 * g + (n >> 2), 16 * (wave * NBW + b) + 4 * (n & 3)))));
      };
      auto add_page = [&](int j, const vec4& pr, const vec4* v) __attribute__((always_inline)) {
        l_run += lsum[j];
#pragma unroll
        for (int b = 0; b < NBW; ++b) o[b] = Mma<T>::pv(pr, v[b], o[b]);
      };
      if (mv & 1) move(0);
      const bool moves = mv > 1;
#pragma unroll
      for (int j0 = 0; j0 < CH; j0 += 4) {
        if (!moves && j0 + 4 <= cn) {   // four pages' reads at once
          vec4 pr[4], v[4][NBW];
#pragma unroll
          for (int j = 0; j < 4; ++j) read_page(j0 + j, pr[j], v[j]);
#pragma unroll
          for (int j = 0; j < 4; ++j) add_page(j0 + j, pr[j], v[j]);
        } else {
#pragma unroll
          for (int j = j0; j < j0 + 4; ++j) {
            if (j < cn) {
              vec4 pr, v[NBW];
              read_page(j, pr, v);
              if (j > 0 && (mv >> j & 1)) move(j);
              add_page(j, pr, v);
            }
          }
        }
      }
      __syncthreads();   // before the next chunk, or the merge's weights
    }
    if (__builtin_amdgcn_ballot_w64(bad) && wave == 0 && lane == 0)
      flag(status, PKV_STATUS_BAD_PAGE);

    if (slot < 0) {   // a whole sequence
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * g + e;
        const float li = from_lane(l_run, e);
        if (r < G) {
          const float inv = 1.f / li;
#pragma unroll
          for (int b = 0; b < NBW; ++b)
            out[((int64_t)row * Hq + h * G + r) * D + 16 * (wave * NBW + b) + n] =
                (T)(o[b][e] * inv);
        }
      }
    } else {          // publish, count the arrival; the last one merges
      const uint32_t head_off = (uint32_t)(((int64_t)slot * n_kv_heads + h) * PL::FLOATS * 4);
      if (g < NGR) {
#pragma unroll
        for (int b = 0; b < NBW; ++b)
          __builtin_amdgcn_raw_buffer_store_b128(
              __builtin_bit_cast(u32x4, o[b]), ro,
              head_off + ((g * NDB + wave * NBW + b) * 16 + n) * 16, 0, kSc1);
      }
      if (wave == 0 && lane < G)
        __builtin_amdgcn_raw_buffer_store_b64(
            __builtin_bit_cast(u32x2, f32x2{m_run, l_run}), rm,
            (uint32_t)(((int64_t)slot * Hq + h * G + lane) * 8), 0, kSc1);
      // every wave's stores have completed before the count
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      int32_t* cnt = counters + (int64_t)seq * n_kv_heads + h;
      if (threadIdx.x == 0)
        *arrived = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (*arrived == nparts - 1) {
        merge_head<T, D, G, NBW>(out, reinterpret_cast<float*>(vt) + wave * 64 * 4 * NGR, row, h,
                                 n_kv_heads, nparts, slot0, ro, rm, false, o, m_run, l_run,
                                 wave * NBW);
        if (threadIdx.x == 0)
          __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    p0 += np;
    if (item + 1 < n_items) __syncthreads();   // LDS is free again
  }
}

// Waves a SIMD the kernel is compiled for: three workgroups a compute unit at
// d = 64, one at d = 128 (what their LDS allows).
template <int D> constexpr int kPieceWaves = D == 64 ? 3 : 1;

// Whether every bin of a plan holds one piece, which pkv_plan_decode says in
// the stride: a multiple of 8 ints then, 4 more than one otherwise.
static inline bool one_piece_bins(int32_t plan_stride) { return plan_stride % 8 == 0; }

// Compute units of the current device, 0 if it cannot be asked.
int compute_units();

// One piece a workgroup where no bin holds more than one and those workgroups
// are all resident at once (3 a compute unit at d = 64, 1 at d = 128; 768 and
// 256 here), the streaming kernel beyond: at d = 64, us a layer and piece
// against streaming, 40 workgroups 9.8 against 17.0, 480 13.9 against 17.6,
// 1280 16.7 against 15.8; at d = 128, 144 12.6 against 17.6, 456 19.0 against
// 19.3. Bins of several pieces always stream: the piece kernel would take them
// one after another with no page in flight between them (1024 sequences of 16
// to 64 tokens in 32 bins of 8 heads: 113 us against 83). From a streaming
// workgroup a compute unit on, batches stream too, which matters to numbers of
// KV heads that 4 does not divide: 200 pieces of 1 head 6.5 us (pieces), 300
// 11.3 (streaming), where the piece kernel would take 6.9.
static inline bool few_pieces(int32_t n_work, int32_t plan_stride, int32_t Hkv, int32_t D) {
  if (!one_piece_bins(plan_stride)) return false;
  const int64_t cus = compute_units(), bins = n_work / (Hkv / heads_per_wg(Hkv));
  return n_work < cus && bins * Hkv <= cus * (D == 64 ? 3 : 1);
}

// The parts of a decode workspace.
struct DecodeWorkspace {
  int32_t* counters;
  float* part_o;
  float* part_ml;
  uint32_t o_bytes, ml_bytes;
};

}  // namespace pkv
