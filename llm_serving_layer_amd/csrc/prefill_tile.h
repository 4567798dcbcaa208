// Chunked-prefill attention over a paged prefix on gfx950 matrix cores.
//
// One workgroup (4 waves) owns one KV head h and one tile of a sequence's
// query rows: 128 rows = BQ query tokens x G query heads (BQ = 128 / G), so
// every K/V tile it loads serves all G query heads of the KV head. Each wave
// owns 32 rows. Query row r of the tile is token r / G (of the tile) and
// query head h*G + r % G; it sits at absolute position kv_len - q_len +
// token (bottom-right causal alignment, as the reference's
// triu(diagonal = kv_len - q_len + 1) mask) and sees keys 0..position.
//
// The KV axis is walked 32 tokens (two pages) at a time. A tile of K and of
// V (those rows x head_dim of head h) goes straight from memory into one of
// four LDS buffers (a ring; direct-to-LDS buffer loads two tiles ahead, each
// wave one page of one tensor, rows unpadded with their 16-byte chunks
// swizzled) and is read by every wave. All products are 32x32x16 MFMAs, so every LDS byte read feeds 32
// query rows:
//  * S^T = K Q^T: K rows from LDS as the A operand, Q^T held in registers
//    as the B operand. Lane (row n, group g) gets 16 scores of its query row
//    n: keys 8 i + 4 g + 0..3, i = 0..3;
//  * online softmax per query row, lane-local; the two half-waves holding a
//    row meet (v_permlane32_swap) only for a row max and for the final sum;
//  * O^T = V^T P^T: V^T from transposing LDS reads as the A operand, the
//    lane's own 8 probabilities of a 16-key block as the B operand (the
//    contraction index runs over keys 4 g + 0..3, 8 + 4 g + 0..3 of the
//    block). Every O^T accumulator of a lane belongs to its own query row,
//    so rescaling needs no cross-lane traffic.
// The running reference moves lazily: probabilities are taken against it,
// and only when some lane's sum of a tile's probabilities passes 2^12 is
// the row max taken and the accumulators rescaled, so probabilities stay at
// most 2^12 and o / l is unchanged. Tiles wholly below the causal diagonal
// skip the mask. Each wave's share of a tile lies within one page, so page
// ids are scalar reads and pages are buffer ranges: rows past kv_len read
// zeros without a memory access.
// Numerics as serving/backends/paged_torch.py:443-485: scores, softmax and
// accumulation in fp32; probabilities rounded to the pool dtype before PV.
// The scale must be positive (the row max is taken before scaling); other
// scales run the generic kernel.
#pragma once

#include "mfma.h"

namespace pkv {

constexpr int kPrefillRows = 128;   // query rows per workgroup (tokens x heads)
constexpr int kPrefillThreads = 256; // 4 waves x 32 rows

typedef float f32x16 __attribute__((ext_vector_type(16)));
template <typename T> struct Mma32;
template <> struct Mma32<_Float16> {
  __device__ static f32x16 mma(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma32<__bf16> {
  __device__ static f32x16 mma(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

// LDS of one workgroup: a ring of four K/V tile buffers, rows unpadded with
// 16-byte chunks XOR-swizzled by row.
template <typename T, int D> struct PrefillLds {
  static constexpr int TT = 32;                        // KV tokens per tile
  static constexpr int RB = D * (int)sizeof(T);        // bytes of one head's row
  static constexpr int TILE = TT * RB;                 // one K (or V) tile
  static constexpr int BYTES = 4 * 2 * TILE;
  static constexpr int LPT = TILE / 2 / 1024;          // wave loads of a page of one tensor
};

template <typename T, int D, int G>
__device__ __forceinline__ void prefill_tile(
    unsigned char* smem, int block,
    const T* __restrict__ q, T* __restrict__ out, const T* __restrict__ kpool,
    const T* __restrict__ vpool, int64_t num_blocks, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ kv_indptr, const int32_t* __restrict__ kv_indices,
    const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ plan,
    int32_t n_kv_heads, float scale_log2, int32_t* status) {
  typedef typename Mma<T>::vec8 vec8;
  typedef typename Mma<T>::vec4 vec4;
  typedef PrefillLds<T, D> L;
  constexpr int TT = L::TT;
  constexpr int PS = 16;
  constexpr int NH = TT / 32;            // 32-key halves per tile
  constexpr int NC = D / 16;             // QK k-chunks of 16 dims
  constexpr int NDH = D / 32;            // PV blocks of 32 dims
  constexpr int RB = L::RB;
  constexpr int CPR = RB / 16;           // 16-byte chunks per row
  constexpr int LPT = L::LPT;
  static_assert(64 % CPR == 0 && PS % (64 / CPR) == 0, "a wave load stays in one page");
  unsigned char* const buf0 = smem + 0 * 2 * L::TILE;
  unsigned char* const buf1 = smem + 1 * 2 * L::TILE;
  unsigned char* const buf2 = smem + 2 * 2 * L::TILE;
  unsigned char* const buf3 = smem + 3 * 2 * L::TILE;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int n = lane & 31, g = lane >> 5;
  const int item = block / n_kv_heads;
  const int h = block - item * n_kv_heads;
  const int seq = plan[4 * item], qs = plan[4 * item + 1], qn = plan[4 * item + 2];
  const int q0 = cu_q[seq];
  const int q_len = cu_q[seq + 1] - q0;
  const int kv_len = kv_lens[seq];
  const int pbase = kv_indptr[seq];
  const int Hq = n_kv_heads * G;
  const int64_t row = (int64_t)n_kv_heads * D;
  const int base_pos = kv_len - q_len + qs;
  const int kv_end = base_pos + qn;
  const int ntiles = (kv_end + TT - 1) / TT;

  // This lane's query row (column n of every 32x32 tile) and Q^T as the B
  // operand of S^T = K Q^T: lane (n, g) holds Q[row][16c + 8g .. + 7].
  const int r = wave * 32 + n;
  const int tok = r / G;
  const bool valid = tok < qn;
  const int qpos = valid ? base_pos + tok : kv_len - 1;
  vec8 qb[NC];
  {
    const T* qr = q + ((int64_t)(q0 + qs + (valid ? tok : 0)) * Hq + h * G + r % G) * D + g * 8;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const vec8 t = *reinterpret_cast<const vec8*>(qr + c * 16);
      qb[c] = valid ? t : vec8{};
    }
  }

  // A wave loads one page of one tensor of a tile, 16 rows of the KV head: one
  // buffer range to set up instead of one per page and tensor (about 45 scalar
  // instructions a step instead of 130; a 777-token prompt, head_dim 128, 8
  // layers with their appends: 205 -> 195 us, with the ring no longer zeroed
  // at the start; no change where four waves share a SIMD). The page id is
  // read with a scalar load a tile ahead. (Scalar loads, so the vector-memory count holds
  // tile loads only: a plain vector load may complete before a direct-to-LDS
  // load issued earlier, so the count cannot prove a tile landed if the two
  // mix.)
  const int npages = (kv_len + PS - 1) / PS;
  const uint32_t rowbytes = (uint32_t)(row * sizeof(T));
  const uint32_t pagebytes = PS * rowbytes;
  // ids at or past this are out of range (kv_indices entries are int32)
  const uint32_t nb32 = num_blocks > 0x7fffffffLL ? 0x80000000u : (uint32_t)num_blocks;
  static_assert(TT == 2 * PS, "a tile is two pages");
  const int wpage = wave & 1;
  const T* const wpool = wave < 2 ? kpool : vpool;
  const uint32_t wdst = (wave < 2 ? 0 : L::TILE) + wpage * PS * RB;
  constexpr int RPI = 64 / CPR;                  // rows of a wave load
  uint32_t voff[LPT];
#pragma unroll
  for (int k = 0; k < LPT; ++k) {
    const int rr = k * RPI + lane / CPR;
    const int lc = ((lane % CPR) ^ xr(rr)) & 7 | ((lane % CPR) & ~7);
    voff[k] = (uint32_t)rr * rowbytes + (uint32_t)(h * RB + lc * 16);
  }
  auto load_id = [&](int t) {   // this wave's page id for tile t
    return __builtin_amdgcn_readfirstlane(kv_indices[pbase + min(2 * t + wpage, npages - 1)]);
  };
  // Rows past kv_len, pages past the last and out-of-range pages are outside
  // the buffer range: zeros land in LDS without a memory access.
  auto load_tile = [&](int t, int raw, const unsigned char* dst) {
    const int pg = 2 * t + wpage;
    const bool bad = (uint32_t)raw >= nb32;   // (negative ids too)
    if (bad && pg < npages && lane == 0) flag(status, PKV_STATUS_BAD_PAGE);
    const int live_rows = bad ? 0 : min(PS, kv_len - pg * PS);   // <= 0 past the end
    const uint32_t pid = bad ? 0u : (uint32_t)raw;
    load_to_lds<LPT>(
        raw_rsrc(reinterpret_cast<const char*>(wpool) + (uint64_t)pid * pagebytes,
                 live_rows > 0 ? (uint32_t)live_rows * rowbytes : 0u),
        voff, lds_address(dst) + wdst);
  };

  // O^T accumulators: o[dh][rr] = O[row][32 dh + 8 (rr / 4) + 4 g + rr % 4].
  f32x16 o[NDH];
#pragma unroll
  for (int dh = 0; dh < NDH; ++dh) o[dh] = f32x16{};
  float m_run = -INFINITY, l_run = 0.f;
  // the transposing V reads: lane i of each 16-lane block points at key
  // (i / 4) of a 4-key group and dims 4 (i % 4) .. + 3 of its 16-dim block
  const int vrow = lane & 15;
  const int vcol = (lane & 16) + 4 * (vrow & 3);

  // P^T of the previous tile (the B operand of its PV), kept for the next step.
  vec8 pb[NH * 2];
#pragma unroll
  for (int i = 0; i < NH * 2; ++i) pb[i] = vec8{};
  // O^T += V^T P^T for a tile: V^T as the A operand, lane (dim, g) holding
  // V[key][dim] for keys 16 kb + 4 g + 0..3 and 16 kb + 8 + 4 g + 0..3.
  auto read_v = [&](const unsigned char* vl, vec8* va) {
#pragma unroll
    for (int kb = 0; kb < NH * 2; ++kb) {
      const int key = 16 * kb + 4 * g + (vrow >> 2);
#pragma unroll
      for (int dh = 0; dh < NDH; ++dh) {
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_i16x4*)(vl + swz<RB>(key, vcol + 32 * dh)));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_i16x4*)(vl + swz<RB>(key + 8, vcol + 32 * dh)));
        va[kb * NDH + dh] = __builtin_bit_cast(
            vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    }
  };
  auto pv_mma = [&](const vec8* va) {
#pragma unroll
    for (int kb = 0; kb < NH * 2; ++kb) {
#pragma unroll
      for (int dh = 0; dh < NDH; ++dh) o[dh] = Mma32<T>::mma(va[kb * NDH + dh], pb[kb], o[dh]);
    }
  };
  auto pv = [&](const unsigned char* vl) {
    vec8 va[NH * 2 * NDH];
    read_v(vl, va);
    pv_mma(va);
  };

  // Tile t: S^T = K Q^T, then its softmax beside the previous tile's PV
  // (independent of it), which leaves tile t's probabilities in pb.
  auto compute = [&](int t, const unsigned char* kl, const unsigned char* vprev) {
    const int t0 = t * TT;
    const bool full = t0 + TT - 1 <= base_pos;
    // the previous tile's V operands, read while QK runs
    vec8 va[NH * 2 * NDH];
    read_v(vprev, va);
    // S^T = K Q^T: s[hf][rr] = score of key t0 + 32 hf + 8 (rr / 4) + 4 g + rr % 4.
    f32x16 s[NH];
#pragma unroll
    for (int hf = 0; hf < NH; ++hf) {
      s[hf] = f32x16{};
      const int kr = hf * 32 + n;
#pragma unroll
      for (int c = 0; c < NC; ++c)
        s[hf] = Mma32<T>::mma(*reinterpret_cast<const vec8*>(kl + swz<RB>(kr, 16 * c + 8 * g)),
                              qb[c], s[hf]);
    }
    // Keys past the row's position are masked only on tiles that reach them.
    if (!full) {
#pragma unroll
      for (int hf = 0; hf < NH; ++hf) {
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          const int key = t0 + 32 * hf + 8 * (rr >> 2) + 4 * g + (rr & 3);
          if (key > qpos) s[hf][rr] = -INFINITY;
        }
      }
    }
    // The previous tile's PV (zero probabilities before the first tile), its
    // matrix instructions interleaved with the softmax's vector ones below.
    pv_mma(va);
    // Probabilities against the running reference m_run: 16-key block
    // (hf, qq) of P^T uses the lane's scores rr = 8 qq .. 8 qq + 7 in that
    // order.
    float ls = 0.f;
    auto probs = [&]() {
      ls = 0.f;
#pragma unroll
      for (int hf = 0; hf < NH; ++hf) {
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[hf][rr], scale_log2, -m_run));
          ls += e;
          pb[2 * hf + (rr >> 3)][rr & 7] = (T)e;
        }
      }
    };
    probs();
    // (pinned here: otherwise the compiler moves them behind the max test)
#pragma unroll
    for (int i = 0; i < NH * 2; ++i) {
      u32x4 w = __builtin_bit_cast(u32x4, pb[i]);
      asm volatile("" : "+v"(w));
      pb[i] = __builtin_bit_cast(vec8, w);
    }
    asm volatile("" : "+v"(ls));
#pragma unroll
    for (int i = 0; i < NH * 2 * NDH; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 12, 0);  // then vector work
    }
    // Lazy rescale: the reference only moves when some lane's sum of its
    // probabilities passes 2^12, which bounds every one of them by 2^12
    // (within the pool dtype's range; NaN or inf counts as past it, as on the
    // first tile, whose reference is -inf); the result o / l does not depend
    // on which reference is used. Only then is the row max taken: it is at
    // least 8 above the reference (a sum past 2^12 over 16 keys has a term
    // past 2^8), so the reference grows, o (with the previous tile's PV
    // added) and l are rescaled and the probabilities taken again.
    if (__builtin_amdgcn_ballot_w64(!(ls <= 4096.f))) {
      // raw-score row max (scale_log2 > 0, so scaling commutes with max)
      float mx = -INFINITY;
#pragma unroll
      for (int hf = 0; hf < NH; ++hf) {
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) mx = fmaxf(mx, s[hf][rr]);
      }
      mx = max_x32(mx) * scale_log2;
      const float m_new = fmaxf(m_run, mx);   // finite: key 0 is visible to every row
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
      m_run = m_new;
#pragma unroll
      for (int dh = 0; dh < NDH; ++dh) o[dh] *= alpha;
      probs();
    }
    // l_run: this lane's half of its row's keys; the halves meet at the end
    l_run += ls;
  };

  // The ring: tile t in buffer t % 4. Each step waits for its tile's loads
  // (this wave's, then every wave's at the barrier, which also ends every
  // wave's reads of the buffer the step then refills: the one of tile t - 2,
  // whose PV ran in the previous step), loads the pages of tile t + 2,
  // computes tile t beside the PV of tile t - 1, and loads the page ids of
  // tile t + 3.
  // The first step's PV meets zero probabilities in buf3, which no tile has
  // filled yet: zeros there (visible to every wave at the step's barrier).
  for (int i = tid; i < L::TILE / 16; i += kPrefillThreads)
    reinterpret_cast<u32x4*>(buf3 + L::TILE)[i] = u32x4{0u, 0u, 0u, 0u};
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  int id0 = load_id(0), id1 = load_id(1), id2 = load_id(2), id3;   // of tile j in id(j % 4)
  load_tile(0, id0, buf0);
  load_tile(1, id1, buf1);
  // Q arrives here: waited for inside the loop, where the compiler cannot see
  // the tile loads, it would drain them in every step
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    u32x4 w = __builtin_bit_cast(u32x4, qb[c]);
    asm volatile("" : "+v"(w));
    qb[c] = __builtin_bit_cast(vec8, w);
  }
  auto step = [&](int t, unsigned char* cur, unsigned char* prev, unsigned char* nxt2,
                  int& id_t2, int& id_t3) {
    // Every tile load but the latest step's has landed; after the barrier,
    // every wave's have. (A fenced barrier would wait for all of them.)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPT) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load_tile(t + 2, id_t2, nxt2);
    compute(t, cur, prev + L::TILE);
    // (after the tile's LDS reads: a scalar load in flight would make every
    // wait for them a wait for it too)
    id_t3 = load_id(t + 3);
  };
  unsigned char* last = buf0;   // the buffer of the last tile computed
  for (int t = 0;; t += 4) {
    step(t, buf0, buf3, buf2, id2, id3);
    last = buf0;
    if (t + 1 >= ntiles) break;
    step(t + 1, buf1, buf0, buf3, id3, id0);
    last = buf1;
    if (t + 2 >= ntiles) break;
    step(t + 2, buf2, buf1, buf0, id0, id1);
    last = buf2;
    if (t + 3 >= ntiles) break;
    step(t + 3, buf3, buf2, buf1, id1, id2);
    last = buf3;
    if (t + 4 >= ntiles) break;
  }
  pv(last + L::TILE);   // the last tile's PV
  // the loads of the tiles past the end land in LDS before the workgroup ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  l_run = sum_x32(l_run);
  if (valid) {
    const float inv = 1.f / l_run;
    T* orow = out + ((int64_t)(q0 + qs + tok) * Hq + h * G + r % G) * D + 4 * g;
#pragma unroll
    for (int dh = 0; dh < NDH; ++dh) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        vec4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (T)(o[dh][4 * j + e] * inv);
        *reinterpret_cast<vec4*>(orow + 32 * dh + 8 * j) = v;
      }
    }
  }
}

}  // namespace pkv
