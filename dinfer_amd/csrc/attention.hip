// MFMA attention over the paged cache for bf16, gfx950.
//
// Both kernels compute S^T = K . Q^T and O^T = V^T . P with
// v_mfma_f32_16x16x32_bf16, whose operands want, per lane, 8 consecutive
// elements of the contraction dimension:
//   A (16 x 32): lane l holds A[l % 16][8 * (l / 16) .. + 8]
//   B (32 x 16): lane l holds B[8 * (l / 16) .. + 8][l % 16]
//   D (16 x 16): lane l holds D[4 * (l / 16) + r][l % 16], r = 0..3
// K pages [Hkv][D / 8][page][8] give A = 8-element pieces of K rows straight from
// memory (contraction over d; the pieces of consecutive keys are contiguous, so
// a quad of lanes reads 64 contiguous bytes); V pages [Hkv][D][page] (transposed)
// give A = V^T rows straight from memory (contraction over keys). K and V are
// not staged through LDS.
//
// A block of 32 keys is scored by two MFMA chains (a = 0, 1). Row i of chain a
// is key  kb + 8 * (i / 4) + 4 * a + (i % 4),  so lane group g = l / 16 ends up
// with the scores of keys kb + 8 g .. kb + 8 g + 7 in its eight result
// registers: exactly the B operand of the P.V product, with no shuffle.
// A query (a column, l % 16) keeps its running maximum, sum and output column in
// the same lanes through both products.
//
//   flash:  query rows with or without history, causal, optional window; many
//           rows of head size 128 in attention_pair.cuh, all others here: a
//           workgroup owns QT x 16 query rows of one head, its four waves walk a
//           quarter of the keys each in blocks of 32 (online softmax in base 2)
//           and combine their results in LDS.
//   decode: all requests bring one row; the G query heads of a kv head are the
//           16 columns, so K and V are read once per group; the keys are split
//           over workgroups, each writing (m, l, o) partials; a merge kernel
//           combines them.
//
// The flash kernel's options are in another library (attention_ext.hip); the tile and the kernel itself in
// attention_tile.cuh.
//
// Sizes: head_dim a multiple of 16 from the instantiated list, page size a
// multiple of 8, G <= 16 for decode. Anything else is refused (the caller then
// uses the plain kernel).
//
// Reference behaviour: crates/kernels/cuda/gqa.cu:167-369 (flash prefill and
// paged: 64-key tiles, base-2 online softmax, P rounded to bf16 before P.V),
// gqa_decode_v3_core.cuh:72-242 and gqa.cu:1423-1461 (split-K decode, merge of
// (m, l, o) partials).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "attention_pair.cuh"
#include "attention_tile.cuh"

using namespace dinfer;

namespace {

// What the decode kernel does itself in a step of single rows only, so that no kernel runs between the q|k|v product
// and the attention: the per-head norm of q and k, the rotation (pairs (i, i + D/2), whole head, angles of the row's
// position), and the new key and value into their pages. Same arithmetic, in the same order, as qkv_post_vec_kernel.
struct DecodePost {
  const bf16* wq;        // gains of the q and k norms (null: no norm)
  const bf16* wk;
  float eps, w_offset;
  const int32_t* pos;    // [rows] position of each row
  const float* cos_sin;  // [positions][D]: cos of the D/2 angles, then sin (null: no rotation)
  const int64_t* slots;  // [rows] block * page + offset of the new key; negative or null: nothing is written
  const bf16* k_new;     // the rows' new keys and values, [rows, ld_q] like q
  const bf16* v_new;
  bf16* k_cache;         // the same pages the kernel reads
  bf16* v_cache;
};

// One head of D = 16 DT dims (DT % 4 == 0) in MFMA operand order: a lane holds the pieces d = 32 ks + 8 g4 .. + 8,
// ks < KS, of the head its lane group of 16 selects; the partner of a pair lies KS / 2 pieces further in the same lane.
// In three steps, so that the kernel can issue every load whose address it knows before it waits for any: load (the
// head and the gains: addresses known at once), Angles::load (needs the position), finish (arithmetic only).
template <int DT>
struct HeadPost {
  static constexpr int KS = DT / 2, D = DT * 16, HALF = D / 2;
  struct Angles {
    f32x4 c[KS / 2][2], s[KS / 2][2];
    __device__ __forceinline__ void load(const float* cs) {
      const int g4 = (threadIdx.x & 63) >> 4;
#pragma unroll
      for (int ks = 0; ks < KS / 2; ++ks) {
        const int pi = ks * 32 + g4 * 8;
        c[ks][0] = *(const f32x4*)(cs + pi);
        c[ks][1] = *(const f32x4*)(cs + pi + 4);
        s[ks][0] = *(const f32x4*)(cs + HALF + pi);
        s[ks][1] = *(const f32x4*)(cs + HALF + pi + 4);
      }
    }
  };
  bf16x8 x[KS];
  bf16x8 g[KS];  // the gains (bf16)

  __device__ __forceinline__ void load(const bf16* src, bool active) {
    const int g4 = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) x[ks] = active ? *(const bf16x8*)(src + ks * 32 + g4 * 8) : zero8();
  }
  __device__ __forceinline__ void load_gains(const bf16* w) {
    const int g4 = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) g[ks] = *(const bf16x8*)(w + ks * 32 + g4 * 8);
  }

  // normed: gains were loaded; rotate: a holds the angles of the row's position
  __device__ __forceinline__ void finish(const Angles& a, bool normed, float eps, float w_offset, bool rotate,
                                         bf16x8 (&r)[KS]) const {
    float inv = 1.f;
    if (normed) {
      float s[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        s[ks] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) s[ks] = add_square(s[ks], (float)x[ks][e]);
      }
      // the sum of squares over the head's D / 8 pieces as a butterfly over the piece index, highest bit first
#pragma unroll
      for (int o = KS / 2; o > 0; o >>= 1)
#pragma unroll
        for (int ks = 0; ks < o; ++ks) s[ks] = s[ks] + s[ks + o];
      float ss = s[0];
      ss = add_over<16>(add_over<32>(ss));
      inv = 1.f / sqrtf(ss / (float)D + eps);
    }
#pragma unroll
    for (int ks = 0; ks < KS / 2; ++ks) {
      const int k2 = ks + KS / 2;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float y1 = (float)x[ks][e], y2 = (float)x[k2][e];
        if (normed) {
          y1 = y1 * inv * ((float)g[ks][e] + w_offset);
          y2 = y2 * inv * ((float)g[k2][e] + w_offset);
        }
        const float c = rotate ? a.c[ks][e >> 2][e & 3] : 1.f, sn = rotate ? a.s[ks][e >> 2][e & 3] : 0.f;
        r[ks][e] = (bf16)rotated_first(y1, y2, c, sn);
        r[k2][e] = (bf16)rotated_second(y1, y2, c, sn);
      }
    }
  }
};

// The keys a request's row sees, [first, seq), are cut into `splits` equal parts of a multiple of
// 32 keys; short requests leave the last parts empty. Computed alike by the decode and merge kernels.
__device__ __forceinline__ void split_range(int seq, int window, int splits, int sp, int* k_lo, int* k_hi, int* kps) {
  const int first = window > 0 ? (seq - window > 0 ? seq - window : 0) : 0;  // the row's position is seq - 1
  const int base = first & ~31;
  const int per = (((seq - base) + splits - 1) / splits + 31) & ~31;
  const int lo = base + sp * per, hi = lo + per;
  *k_lo = lo > first ? lo : first;
  *k_hi = hi < seq ? hi : seq;
  *kps = per;
}

// One wave per (split, kv head, request). part: [B, H, splits, D + 4] float = (m in base-2 units, l, -, -, o[D]).
// JOIN (up to JOIN_SPLITS parts: many requests): the parts of a (kv head, request) are the waves of one workgroup,
// meet in LDS and are combined there as attn_decode_merge_kernel combines them, so that kernel does not run.
constexpr int JOIN_SPLITS = 4;
constexpr int64_t STREAM_FROM_BYTES = 100 * 1000 * 1000;
constexpr int64_t STREAM_FROM_BYTES_FEW = 170 * 1000 * 1000;  // for one or two requests

// POST: q arrives as the product left it; the kernel norms and rotates it on the way into its registers (every part
// for itself: the head is 2 D bytes), and the wave whose part ends with the row's own position norms and rotates the
// new key and stores it and the new value into their pages before it reads its last block.
// (The pages are written through post.k_cache / v_cache and read through kc / vc: no __restrict__ on those.)
// LATE (POST only): the new key is dealt with inside the walk instead of before it (see there).
// OWN (JOIN, fewer requests than LATE is for): the row's own key and value are a part of their own, the last, of one more wave.
// With POST that wave norms and rotates q and the new key in registers, scores the one with the other and stores key and value, while
// the others walk the keys before it, so that nobody waits for a store to come back (one request of 250 keys, 16 heads on 8
// of 128: 8.5 -> 7.7 us, in a step of 28 layers 1,019 -> 985; 8 requests 9.3 -> 8.5, 28 of 2,048 keys, 40 heads,
// 45.1 -> 43.0; where the parts are workgroups of their own it loses 0.4 us and more from 2,048 keys on). Where its at most
// four parts meet, at 8 kv heads: engines of at most 256 positions, or 26 to 31 requests at any length. Without POST, and for
// a row that is written nowhere, the wave walks that key: the same parts, the same bits.
// stream_from: from this many bytes of keys and values in a step on (the request's own visible keys times the number
// of requests: a wave knows no more) they are read with non-temporal loads.
template <int DT, bool P2, bool LATE, bool JOIN = false, bool POST = false>
// (These launches aim at about one wave a SIMD, and JOIN runs where a CU holds 4 to 8 of its waves: registers are no
// limit; POST holds a head, gains and angles at once in its prologue.)
__global__ void __launch_bounds__(JOIN ? 64 * (JOIN_SPLITS + 1) : 64)
__attribute__((amdgpu_waves_per_eu(2, 8)))
attn_decode_kernel(
    const bf16* __restrict__ q, int64_t ld_q, float* __restrict__ part, const bf16* kc, const bf16* vc,
    const int32_t* __restrict__ block_table, int64_t max_blocks, const int32_t* __restrict__ cu_seqlens,
    const int32_t* __restrict__ seq_lens, int splits, float scale_log2e, int window, int H, int Hkv, int ps,
    int64_t stream_from, bf16* __restrict__ out = nullptr, int64_t ld_out = 0, DecodePost post = DecodePost{}) {
  constexpr int D = DT * 16;
  constexpr int KS = (DT + 1) / 2;
  constexpr bool OWN = JOIN && !LATE;
  static_assert(!POST || DT % 4 == 0, "the fused norm and rotation keep both elements of a pair in one lane");
  const int sp = JOIN ? (int)(threadIdx.x >> 6) : (int)blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
  const int G = H / Hkv;
  int row = b;  // without cu_seqlens every request has exactly one row
  if (cu_seqlens) {
    row = cu_seqlens[b];
    if (cu_seqlens[b + 1] - row != 1) return;  // a longer run of rows belongs to the flash kernel
  }
  const int lane = threadIdx.x & 63, i16 = lane & 15, g4 = lane >> 4;
  const int32_t* bt = block_table + (int64_t)b * max_blocks;
  const bf16* qp = q + (int64_t)row * ld_q + (int64_t)(hk * G + (i16 < G ? i16 : 0)) * D;
  int k_lo, k_hi, kps, seq;   // (not set, and not read, where the wave holds its part without a walk)
  bf16x8 qf[1][KS];
  Tile<DT, 1, P2> tl;
  bool writer = false;
  int w_pos = 0;
  int64_t w_slot = -1;
  const bool own = OWN && (int)blockDim.x > 64 * splits, own_part = own && sp == splits;   // (wave-uniform)
  bool held = false;   // the own part needs no walk
  float own_l = 0.f;
  if constexpr (OWN && POST) {
    if (own_part) {
      const bf16* vn = post.v_new + (int64_t)row * ld_q + (int64_t)hk * D;
      HeadPost<DT> qh, kh;
      bf16x4 v4[DT];
      bf16x8 vv, kr[KS];
      qh.load(qp, i16 < G);
      kh.load(post.k_new + (int64_t)row * ld_q + (int64_t)hk * D, i16 == 0);
      if (post.wq) qh.load_gains(post.wq), kh.load_gains(post.wk);
      const int pos_row = post.cos_sin ? post.pos[row] : 0;
      const int64_t slot = post.slots ? post.slots[row] : -1;
#pragma unroll
      for (int d = 0; d < DT; ++d) v4[d] = *(const bf16x4*)(vn + d * 16 + 4 * g4);
      if (lane < D / 8) vv = *(const bf16x8*)(vn + lane * 8);
      typename HeadPost<DT>::Angles ang;
      if (post.cos_sin) ang.load(post.cos_sin + (int64_t)pos_row * D);
      kh.finish(ang, post.wk != nullptr, post.eps, post.w_offset, post.cos_sin != nullptr, kr);
      qh.finish(ang, post.wq != nullptr, post.eps, post.w_offset, post.cos_sin != nullptr, qf[0]);
      held = slot >= 0;
      if (!held) {   // nothing is written: the pages hold the key
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[0][ks] = i16 < G ? qf[0][ks] : zero8();
        seq = seq_lens[b];
        k_hi = max(seq, 0);
        k_lo = max(seq - 1, 0);
        tl.init(kc, vc, bt, (int)max_blocks, hk, Hkv, ps, k_lo, k_hi, scale_log2e);
      } else {
        const auto [blk, off] = page_slot(slot, ps);
        const int64_t head = (blk * Hkv + hk) * (int64_t)ps * D;
        if (i16 == 0) {
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            *(bf16x8*)(post.k_cache + head + k_page_offset(off, ks * 32 + g4 * 8, ps)) = kr[ks];
        }
        if (lane < D / 8) {  // V pages are transposed: the 8 dims of a piece go to 8 rows of keys
          bf16* vd = post.v_cache + head + (int64_t)(lane * 8) * ps + off;
#pragma unroll
          for (int e = 0; e < 8; ++e) vd[(int64_t)e * ps] = vv[e];
        }
        f32x4 x = {0.f, 0.f, 0.f, 0.f};   // row 0 is the key: lane group 0 gets its scores
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) x = mfma16(i16 == 0 ? kr[ks] : zero8(), i16 < G ? qf[0][ks] : zero8(), x);
        // (as a walk of this one key leaves it: a score of -inf has the weight 0)
        tl.m[0] = __shfl(x[0], i16, 64);
        own_l = exp2_raw(fmaf(tl.m[0], scale_log2e, -((tl.m[0] == -INFINITY ? 0.f : tl.m[0]) * scale_log2e)));
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int e = 0; e < 4; ++e) tl.o[0][d][e] = (float)v4[d][e] * (float)(bf16)own_l;
      }
    }
  }
  if (POST && own_part) {
  } else if constexpr (POST) {
    // in the order of what is known when: the head, its gains, the row's position and slot at once; ...
    HeadPost<DT> qh;
    qh.load(qp, i16 < G);
    if (post.wq) qh.load_gains(post.wq);
    const int pos_row = post.cos_sin ? post.pos[row] : 0;
    const int64_t slot = post.slots ? post.slots[row] : -1;
    seq = seq_lens[b];
    split_range(seq, window, splits, sp, &k_lo, &k_hi, &kps);
    if (!JOIN && k_lo >= k_hi) return;
    if (own) k_hi = min(k_hi, seq - 1);
    // ... with the length the block table, with the position the angles; the part that ends with the row's own
    // position (wave-uniform) also takes the new key and value
    tl.init(kc, vc, bt, (int)max_blocks, hk, Hkv, ps, k_lo, k_hi, scale_log2e);
    typename HeadPost<DT>::Angles ang;
    if (post.cos_sin) ang.load(post.cos_sin + (int64_t)pos_row * D);
    writer = !own && slot >= 0 && k_lo < k_hi && k_hi == seq;
    qh.finish(ang, post.wq != nullptr, post.eps, post.w_offset, post.cos_sin != nullptr, qf[0]);
    if (i16 >= G) {  // columns beyond the group stay zero whatever the norm made of nothing
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[0][ks] = zero8();
    }
    w_pos = pos_row;
    w_slot = slot;
    if (!LATE && writer) {
      // few requests, short parts: the new key and value are dealt with here, at once (the loads are asked for only now,
      // when the registers of q's head are free); see below for the launches of many requests
      const auto [blk, off] = page_slot(slot, ps);
      const int64_t head = (blk * Hkv + hk) * (int64_t)ps * D;
      HeadPost<DT> kh;
      bf16x8 vv;
      kh.load(post.k_new + (int64_t)row * ld_q + (int64_t)hk * D, i16 == 0);
      if (post.wk) kh.load_gains(post.wk);
      if (lane < D / 8) vv = *(const bf16x8*)(post.v_new + (int64_t)row * ld_q + (int64_t)hk * D + lane * 8);
      bf16x8 kr[KS];
      kh.finish(ang, post.wk != nullptr, post.eps, post.w_offset, post.cos_sin != nullptr, kr);
      if (i16 == 0) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          *(bf16x8*)(post.k_cache + head + k_page_offset(off, ks * 32 + g4 * 8, ps)) = kr[ks];
      }
      if (lane < D / 8) {  // V pages are transposed: the 8 dims of a piece go to 8 rows of keys
        bf16* vd = post.v_cache + head + (int64_t)(lane * 8) * ps + off;
#pragma unroll
        for (int e = 0; e < 8; ++e) vd[(int64_t)e * ps] = vv[e];
      }
    }
  } else {
    seq = seq_lens[b];
    split_range(seq, window, splits, sp, &k_lo, &k_hi, &kps);
    // an empty part writes nothing; the merge kernel skips it by the same rule. (JOIN: it walks no block and
    // leaves m = -inf, which weighs nothing; its wave must reach the barrier below.)
    if (!JOIN && k_lo >= k_hi) return;
    if (own_part) {
      k_hi = max(seq, 0);
      k_lo = max(seq - 1, 0);
    } else if (own) {
      k_hi = min(k_hi, seq - 1);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d = ks * 32 + g4 * 8;
      qf[0][ks] = (d < D && i16 < G) ? *(const bf16x8*)(qp + d) : zero8();
    }
    tl.init(kc, vc, bt, (int)max_blocks, hk, Hkv, ps, k_lo, k_hi, scale_log2e);
  }
  // (reading the first block before q is normed, or two blocks ahead, was measured at 1 and 8 requests: no gain)
  const auto partial = [&](int kb) { return kb < k_lo || kb + 32 > k_hi; };
  // Where a step's keys and values exceed the caches they are read past them (every layer has keys of its own, so
  // none is read twice anyway): 8 kv heads of 128, 8 requests of 32k keys 193 -> 175 us, 16 of 2k 33.7 -> 31.7,
  // 8 of 4k 33.6 -> 31.7; below about 100 MB a step the plain loads are faster (one request of 8k keys 19.0 against
  // 21.6 us, 4 of 2k 16.1 against 17.6; one or two requests up to 170 MB: one of 32k 39.7 against 42.1, of 48k 51.5
  // against 48.9). Both walks are in the kernel, the choice is uniform over the wave.
  const auto walk = [&](auto hook) {
    const int col_lo[1] = {k_lo}, col_hi[1] = {k_hi}, seen = window > 0 && window < seq ? window : seq;
    // (LATE is for many requests, whose keys exceed the caches at any length worth a thought)
    if (LATE || (int64_t)gridDim.z * seen * (Hkv * D * 4) >= stream_from)
      tl.template walk<false, true>(qf, col_lo, col_hi, partial, hook);
    else
      tl.template walk<false, false>(qf, col_lo, col_hi, partial, hook);
  };
  if constexpr (OWN) {
    if (!held) walk([](int, bool) {});
  } else if constexpr (POST && !LATE) {
    // the key was stored in the prologue; the fence lets the wave's own loads of its last block see it
    walk([&](int, bool last) {
      if (writer && last) __threadfence_block();
    });
  } else if constexpr (POST) {
    // Many requests (parts of dozens of blocks, every workgroup waiting for the wave that writes):
    // The wave whose part ends with the row's own position brings the new key and value: their loads (the head, the
    // value) go out three blocks before the end, a block later the key is normed (gains and angles asked for there:
    // kept through a block they would cost the walk a hundred registers), rotated and stored with the value, and
    // before the last block a fence lets the wave's own loads of that block see them: the latencies lie under the
    // blocks' work instead of on the path of the wave that ends its workgroup (64 requests of 2,064 keys: 96.9 ->
    // 92.3 us, of 4,080 keys 181 -> 174.5; at 8 requests, where a part is five blocks, the larger kernel loses 1.5 us,
    // hence the two forms). A part of fewer blocks does the steps as early as it can.
    HeadPost<DT> kh;   // only its head is kept from one block to the next: the gains and angles are asked for where
    bf16x8 vv;         // they are used (they come from L2), or the walk would hold a hundred registers for them
    bool fetched = false;
    const auto fetch_key = [&]() {
      kh.load(post.k_new + (int64_t)row * ld_q + (int64_t)hk * D, i16 == 0);
      if (lane < D / 8) vv = *(const bf16x8*)(post.v_new + (int64_t)row * ld_q + (int64_t)hk * D + lane * 8);
      fetched = true;
    };
    const auto store_key = [&]() {
      const auto [blk, off] = page_slot(w_slot, ps);
      const int64_t head = (blk * Hkv + hk) * (int64_t)ps * D;
      typename HeadPost<DT>::Angles kang;
      if (post.wk) kh.load_gains(post.wk);
      if (post.cos_sin) kang.load(post.cos_sin + (int64_t)w_pos * D);
      bf16x8 kr[KS];
      kh.finish(kang, post.wk != nullptr, post.eps, post.w_offset, post.cos_sin != nullptr, kr);
      if (i16 == 0) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          *(bf16x8*)(post.k_cache + head + k_page_offset(off, ks * 32 + g4 * 8, ps)) = kr[ks];
      }
      if (lane < D / 8) {  // V pages are transposed: the 8 dims of a piece go to 8 rows of keys
        bf16* vd = post.v_cache + head + (int64_t)(lane * 8) * ps + off;
#pragma unroll
        for (int e = 0; e < 8; ++e) vd[(int64_t)e * ps] = vv[e];
      }
    };
    bool stored = false;
    walk([&](int kb, bool last) {
      if (!writer) return;
      if (fetched && !stored) store_key(), stored = true;   // (the loads went out a block ago)
      if (!fetched && kb + 96 >= k_hi) fetch_key();
      if (last) {
        if (!stored) store_key(), stored = true;
        __threadfence_block();
      }
    });
  } else {
    walk([](int, bool) {});
  }
  const float lt = held ? own_l : tl.sum_l(0);
  if constexpr (JOIN) {
    const int parts = splits + (own ? 1 : 0);
    __shared__ __attribute__((aligned(16))) float joined[JOIN_SPLITS + 1][16][D + 4];
    if (i16 < G) {
      float* pp = &joined[sp][i16][0];
      if (g4 == 0) {
        // -inf for an empty part; a score of the own key that is no number may not pass for one (the sum then tells it)
        pp[0] = own_part && lt != lt && tl.m[0] != INFINITY ? 0.f : tl.m[0] * scale_log2e;
        pp[1] = lt;
      }
#pragma unroll
      for (int d = 0; d < DT; ++d) *(f32x4*)(pp + 4 + d * 16 + 4 * g4) = tl.o[0][d];
    }
    __syncthreads();
    // out[head, d] = sum_s 2^(m_s - M) o_s / sum_s 2^(m_s - M) l_s, parts in ascending order
    for (int idx = threadIdx.x; idx < G * D; idx += blockDim.x) {
      const int i = idx / D, d = idx - i * D;
      float M = -INFINITY;
      for (int s = 0; s < parts; ++s) M = fmaxf(M, joined[s][i][0]);
      const int keep = own && M != INFINITY ? splits : -1;
      float L = 0.f, acc = 0.f;
      for (int s = 0; s < parts; ++s) {
        const float m = joined[s][i][0];
        const float a = m == -INFINITY ? 0.f : exp2f(m - M);
        // (the own part also at a weight of 0: what is no number in it stays so, as it does in a walk that meets the key
        // beside others; beside an infinite score it goes like the other parts)
        if (a > 0.f || s == keep) {
          L += a * joined[s][i][1];
          acc += a * joined[s][i][4 + d];
        }
      }
      const float inv = L > 0.f ? 1.f / L : 0.f;
      out[(int64_t)row * ld_out + (int64_t)(hk * G + i) * D + d] = (bf16)(acc * inv);
    }
  } else if (i16 < G) {
    float* pp = part + (((int64_t)b * H + hk * G + i16) * splits + sp) * (D + 4);
    if (g4 == 0) {
      pp[0] = tl.m[0] * scale_log2e;  // the tile keeps raw maxima; partials carry base-2 units
      pp[1] = lt;
    }
#pragma unroll
    for (int d = 0; d < DT; ++d) *(f32x4*)(pp + 4 + d * 16 + 4 * g4) = tl.o[0][d];
  }
}

constexpr int MAX_SPLITS = 256;

// out[b, h, :] = sum_s 2^(m_s - M) o_s / sum_s 2^(m_s - M) l_s over the non-empty parts. One wave per (head, request).
// The kernel is a chain of memory round trips and little else, so everything whose address is known at the start
// is asked for at the start: the length, every part's (m, l), and the outputs of the first MERGE_AHEAD parts; which
// parts are empty (they hold anything) is settled afterwards. Head sizes up to 256, up to MAX_SPLITS parts.
constexpr int MERGE_AHEAD = 8;
__global__ void __launch_bounds__(64) attn_decode_merge_kernel(const float* __restrict__ part, bf16* __restrict__ out,
                                                               int64_t ld_out, const int32_t* __restrict__ cu_seqlens,
                                                               const int32_t* __restrict__ seq_lens, int splits,
                                                               int window, int H, int D) {
  __shared__ float wgt[MAX_SPLITS];
  const int h = blockIdx.x, b = blockIdx.y, lane = threadIdx.x;
  int row = b;
  if (cu_seqlens) {
    row = cu_seqlens[b];
    if (cu_seqlens[b + 1] - row != 1) return;
  }
  const float* pp = part + ((int64_t)b * H + h) * splits * (D + 4);
  f32x2 ml[MAX_SPLITS / 64];
#pragma unroll
  for (int j = 0; j < MAX_SPLITS / 64; ++j) {
    const int s = lane + 64 * j < splits ? lane + 64 * j : splits - 1;  // clamped, not skipped: no branch around a load
    ml[j] = *(const f32x2*)(pp + (int64_t)s * (D + 4));
  }
  float ahead[MERGE_AHEAD][4];
#pragma unroll
  for (int s = 0; s < MERGE_AHEAD; ++s)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int sc = s < splits ? s : splits - 1, d = lane + 64 * j < D ? lane + 64 * j : D - 1;
      ahead[s][j] = pp[(int64_t)sc * (D + 4) + 4 + d];
    }
  const int seq = seq_lens[b];
  float mloc = -INFINITY;
#pragma unroll
  for (int j = 0; j < MAX_SPLITS / 64; ++j) {
    const int s = lane + 64 * j;
    int k_lo, k_hi, kps;
    split_range(seq, window, splits, s, &k_lo, &k_hi, &kps);
    const float m = s < splits && k_lo < k_hi ? ml[j][0] : -INFINITY;
    ml[j][0] = m;
    mloc = fmaxf(mloc, m);
  }
  const float M = wave_max(mloc);
  float lloc = 0.f;
#pragma unroll
  for (int j = 0; j < MAX_SPLITS / 64; ++j) {
    const int s = lane + 64 * j;
    const float m = ml[j][0];
    const float a = m == -INFINITY ? 0.f : exp2f(m - M);
    if (s < splits) wgt[s] = a;
    lloc += a > 0.f ? a * ml[j][1] : 0.f;
  }
  const float L = wave_sum(lloc);
  __syncthreads();
  const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int d = lane + 64 * j;
    if (d >= D) break;
    float acc = 0.f;
#pragma unroll
    for (int s = 0; s < MERGE_AHEAD; ++s) {
      const float a = s < splits ? wgt[s] : 0.f;
      acc += a > 0.f ? a * ahead[s][j] : 0.f;
    }
#pragma unroll 8
    for (int s = MERGE_AHEAD; s < splits; ++s) {
      const float a = wgt[s];
      const float v = pp[(int64_t)s * (D + 4) + 4 + d];  // loads do not wait for the weights
      acc += a > 0.f ? a * v : 0.f;
    }
    out[(int64_t)row * ld_out + (int64_t)h * D + d] = (bf16)(acc * inv);
  }
}

inline bool aligned16(const void* p) { return ((uintptr_t)p % 16) == 0; }

// The kernel of paired waves over all tiles of a step (see its header).
template <bool HALVES>
int launch_pair(const bf16* q, int64_t ld_q, bf16* out, int64_t ld_out, const bf16* kc, const bf16* vc, const int32_t* bt,
                int64_t max_blocks, const int32_t* cu, const int32_t* sl, int num_reqs, int64_t tokens, int max_q_len, float scale,
                int H, int Hkv, int ps, int skip_single, hipStream_t stream) {
  constexpr int COLS = pair_columns(HALVES);
  const int64_t G = H / Hkv, tiles = (max_q_len * G + COLS - 1) / COLS;
  // Counted where that takes a tenth fewer workgroups: a whole CU each, they cost more than the count where they find nothing, but
  // otherwise the longest tiles of all requests come first. 2,300 steps of several requests where it does take 0.93 of the time
  // (geometric mean), 6,100 others would 1.03.
  const int64_t all = tiles * num_reqs, some = tokens * G / COLS + num_reqs;
  const bool count = all * 10 >= some * 11;
  const int64_t blocks = (count ? some : all) * Hkv;
  if (blocks > 0x7fffffff) return ERR_UNSUPPORTED;
  auto kernel = attn_pair_kernel<HALVES>;
  if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, pair_lds(HALVES)) != hipSuccess) return ERR_LAUNCH;
  kernel<<<(unsigned)blocks, 512, pair_lds(HALVES), stream>>>(q, ld_q, out, ld_out, kc, vc, bt, max_blocks, cu, sl, num_reqs, (int)tiles,
                                                              count, scale * LOG2E, H, Hkv, ps, skip_single, PairExpanded{});
  return launch_status();
}

// (16 keys of a block lie in one page, and every row sees all keys before it)
inline bool takes_pair(int ps, int window) { return window == 0 && ps >= 16 && (ps & (ps - 1)) == 0; }

// Whether a step's rows are many enough for the kernel of paired waves: 0 no, 1 with 256 columns a workgroup, 2 with 128 and
// two halves of the keys. One workgroup fills a CU, the tiles of rows are two a CU. The histories are not known here.
//
// One request: what counts is how many workgroups there are for the CUs, w1 and w2, and that the tiles are full (w2 by the rows there
// are); the tiles grow with the causal mask and end apart. us with the tile of rows, 1 and 2 (H heads over 8):
//   from nothing     H 32: 1,000 rows (w2 256) 21.5, 30.6, 23.5; 1,300 (328) 31.8, 37.2, 31.7; 2,001 (w1 256) 57, 53, 48; 2,500 (320)
//                    81, 68, 76; 4,000 165, 128, 150. H 16: 2,500 (w2 320) 44, 60, 42. 64 over 64: 531 (w1 192, w2 265 of rows) 25, 33, 31
//   behind 6,000     H 32: 1,300 200, 156, 176; 2,001 274, 213, 216; 4,000 583, 444, 477
// Several: form 1 or none, by the rounds that the tiles of each make over its places, taken half for requests as long as the longest and
// half for any lengths, a last round that is not full by a quarter as a whole one. A round of form 1 costs 2.9 of the tile of rows, and
// where lengths differ its last long tiles run alone, three more at most; 3 where one request has nearly all rows. Fitted over 27,900
// steps of 2 to 48 requests with 4 to 64 heads and 24,700 of 16 to 40 heads over 4 or 8 whose lengths differ by a quarter at most or
// are one portion beside single rows: 0.969 and 0.974 of the time with the tile of rows alone (geometric means), 2.7 % and 0.3 % more
// than 3 % slower; with form 2 as well no better. us with the tile of rows, 1 and 2:
//   equal            16 x 256, H 32 62, 46, 62; 4 x 500 behind 1,500 91, 68, 75; two of 1,000, H 16 24, 34, 26; 8 x 130, H 16 13, 16, 14;
//                    H 32 18.5, 16.5, 23.5; 21 x 20, 64 over 64 18, 37, 46
//   unequal          22 of 19 to 134 behind up to 2,955, H 16 50, 69, 51; 19 of 8 to 77 behind up to 3,598, 32 over 32 74, 85, 62
inline int pair_form(int64_t tokens, int num_reqs, int max_q_len, int H, int Hkv) {
  const int cus = compute_units();
  if (num_reqs == 1) {
    const int64_t w1 = ((int64_t)max_q_len * (H / Hkv) + 255) / 256 * Hkv, full = std::min<int64_t>(tokens, max_q_len) * H;
    return w1 >= cus + cus / 4 ? 1 : full >= (int64_t)128 * (cus + cus / 4) ? 2 : 0;
  }
  const double T = (double)tokens, long_ones = (double)std::max<int64_t>(1, std::min<int64_t>(num_reqs, (tokens + max_q_len / 2) / max_q_len));
  const double apart = std::max(0., 1. - T / ((double)num_reqs * max_q_len));
  auto rounds = [&](int cols, int group, int heads, int places) {   // of tiles of `cols` columns
    const double equal = long_ones * std::ceil(T / long_ones * group / cols), any = T * group / cols + .5 * num_reqs;
    const double x = (equal + any) / 2 * heads / places;
    return x < 1. ? 1. : .75 * x + .25 * std::ceil(x);
  };
  const double r1 = rounds(256, H / Hkv, Hkv, cus);
  return (long_ones == 1. ? 3. * r1 : 2.9 * r1 + 3. * apart) < rounds(32, 1, H, 2 * cus) ? 1 : 0;
}

// How many tiles of 16 rows there are at most; single rows that are left to the split-K kernel count as one each, as elsewhere here.
inline int64_t few_tiles(int64_t tokens, int num_reqs, int max_q_len) {
  return std::min<int64_t>((int64_t)((max_q_len + 15) / 16) * num_reqs, tokens / 16 + num_reqs);
}

template <int DT>
int launch_flash(const bf16* q, int64_t ld_q, bf16* out, int64_t ld_out, const bf16* kc, const bf16* vc,
                 const int32_t* bt, int64_t max_blocks, const int32_t* cu, const int32_t* sl, int num_reqs, int64_t tokens,
                 int max_q_len, float scale, int window, int H, int Hkv, int ps, int skip_single, hipStream_t stream) {
  const float sl2 = scale * LOG2E;
  const bool p2 = (ps & (ps - 1)) == 0;
  // 32 rows per workgroup where the head size leaves room for two row tiles (registers, and the LDS the
  // waves meet in), and the portions are longer than one tile; otherwise 16
  auto lds_of = [](int qt, int waves) { return (size_t)(waves - 1) * qt * 64 * (sizeof(f32x4) * DT + 2 * sizeof(float)); };
  // 48 rows per workgroup at head size 128: every K and V fragment a wave loads serves three row tiles instead of two
  // (the path on which loads return is what this kernel fills first), at 256 registers, still two waves a SIMD.
  // It pays where the rows still make several rounds of workgroups over the chip (measured, 32 heads: 3,072 rows
  // 135 -> 121 us, 8,192 rows 783 -> 642 us = 34 % of the MFMA peak, 32,768 rows 37 %). Head size 64 gains nothing. (Rows of
  // at most two tiles a request never fill the third: many single rows of many heads are no case.)
  const auto run = [&](auto qt, auto waves) {
    constexpr int QT = decltype(qt)::value, W = decltype(waves)::value;
    const int tiles = (max_q_len + 16 * QT - 1) / (16 * QT);
    // A workgroup for every tile that a request might have: beside decoding requests nearly all of them find none (31 of them and
    // a portion of 512 rows: 14,520 workgroups for 440), so there the tiles are counted up instead: that portion behind 1,024
    // keys, 40 heads, 37 -> 29 us, 1,024 rows of 32 heads beside 48 requests 51 -> 29, 200 beside 16 17.7 -> 13.5. Where few are
    // empty the count is a microsecond more for nothing.
    const int64_t all = (int64_t)tiles * num_reqs, some = tokens / (16 * QT) + num_reqs;
    const bool count = all >= 4 * some;
    const int64_t blocks = (count ? some : all) * H;
    if (blocks > 0x7fffffff) return (int)ERR_UNSUPPORTED;
    auto kernel = p2 ? attn_flash_kernel<DT, QT, true, PLAIN, DT, false, false, W> : attn_flash_kernel<DT, QT, false, PLAIN, DT, false, false, W>;
    if (count) kernel = p2 ? attn_flash_kernel<DT, QT, true, PLAIN, DT, false, true, W> : attn_flash_kernel<DT, QT, false, PLAIN, DT, false, true, W>;
    // (more than the 64 KB of LDS a launch may ask for without saying so)
    if (QT == 3 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_of(QT, W)) != hipSuccess)
      return (int)ERR_LAUNCH;
    kernel<<<(unsigned)blocks, 64 * W, lds_of(QT, W), stream>>>(q, ld_q, out, ld_out, kc, vc, bt, max_blocks, cu, sl, count ? num_reqs : tiles,
                                                         sl2, window, H, Hkv, ps, skip_single, FlashExt{});
    return launch_status();
  };
  constexpr std::integral_constant<int, 4> four;
  if constexpr (DT == 8) {
    if (takes_pair(ps, window)) {
      const int form = pair_form(tokens, num_reqs, max_q_len, H, Hkv);
      if (form)
        return (form == 1 ? launch_pair<false> : launch_pair<true>)(q, ld_q, out, ld_out, kc, vc, bt, max_blocks, cu, sl, num_reqs,
                                                                    tokens, max_q_len, scale, H, Hkv, ps, skip_single, stream);
    }
    // One request, us at 32 and at 48 rows a tile (32 heads), from nothing and behind 8,000 keys: 992 workgroups of 48 rows 40 and
    // 42, 285 and 254; 1,120 50 and 53, 340 and 326; 1,312 61 and 61, 380 and 363; 1,472 75 and 70, 449 and 384. Several begin
    // later, taken for as long as the longest: 8 x 256 rows (1,536) 30 and 36, 4 x 500 (1,408) 35 and 40, behind 1,000 76 and
    // 76. Where one is long and the others are not, fewer exist than that, and 48 rows have to save a round of the places,
    // two a CU: behind 8,000 keys beside 12 rows 440 rows (360 workgroups, one round for two) 150 and 113 at 40 heads, 89 and
    // 112 at 32 (288, one each); 1,000 rows of 32 heads (two each) 184 and 206, 1,500 (two for three) 274 and 245.
    const int64_t longest = (int64_t)((max_q_len + 47) / 48) * num_reqs * H, places = 2 * compute_units();
    auto rounds = [&](int64_t rows) { return (tokens / rows * H + places - 1) / places; };
    const bool wide = num_reqs == 1 ? tokens / 48 * H >= 1300 : longest >= 2000 && rounds(48) < rounds(32);
    if (max_q_len > 32 && wide) return run(std::integral_constant<int, 3>{}, four);
  }
  if constexpr (DT <= 8) {
    // Tiles of 16 rows where 32 would leave CUs idle, up to two a CU of them: a tile's walk is as many blocks of keys long, each with half
    // the work. Up to one a CU eight waves share its keys, at portions of at most 128 rows (240 from nothing 1 % slower with eight than
    // before, 2 % faster with four). A step of 28 layers of 16 heads, us, 32 rows, 16, 16 with eight waves: 100 rows behind 3,000 (112 tiles of
    // 16) 2,533, 2,242, 1,992, from nothing 1,528, 1,492, 1,492; 4 x 120 behind 500 (512) 2,197, 2,170, 2,237; 700 behind 2,000 (704) 3,115,
    // 3,187. Eight layers of 32 heads: 120 behind 3,000 (256) 1,649, 1,570, 1,491; 240 behind 2,000 (480) 1,876, 1,824, 1,846; 300 behind 3,000
    // (608) 2,232, 2,268, 2,297. Heads of 32, 64 and 96, 8 to 64 of them, 1 to 4 requests of 20 to 500 rows behind 0, 500 and 3,000 keys, the kernel
    // alone, over 32 rows: eight waves 0.54 to 0.84 (the worst 0.90), four 0.68 to 0.95 (0.99).
    const int64_t small = few_tiles(tokens, num_reqs, max_q_len) * H;
    if (small <= compute_units() && max_q_len <= 128) return run(std::integral_constant<int, 1>{}, std::integral_constant<int, 8>{});
    if (max_q_len > 16 && small > 2 * compute_units()) return run(std::integral_constant<int, 2>{}, four);
  }
  return run(std::integral_constant<int, 1>{}, four);
}

// The form of the decode kernel for a launch. LATE exists where the new key is the kernel's business and its
// registers allow it (head size 256 would spill).
template <int DT, bool P2, bool JOIN, bool POST>
auto decode_kernel_for(bool late) {
  if constexpr (POST && DT <= 8) {
    if (late) return attn_decode_kernel<DT, P2, true, JOIN, POST>;
  }
  return attn_decode_kernel<DT, P2, false, JOIN, POST>;
}

template <int DT, bool POST>
int launch_decode(const bf16* q, int64_t ld_q, bf16* out, int64_t ld_out, float* part, const bf16* kc, const bf16* vc,
                  const int32_t* bt, int64_t max_blocks, const int32_t* cu, const int32_t* sl, int num_reqs,
                  int splits, float scale, int window, int H, int Hkv, int ps, const DecodePost& post,
                  hipStream_t stream) {
  // many requests (parts of dozens of blocks): the new key is dealt with inside the walk
  const bool p2 = (ps & (ps - 1)) == 0, late = num_reqs >= 32;
  // (one or two requests: measured level at 134 MB a step or behind by 6 %, ahead by 5 to 8 % from 200 MB on)
  const int64_t stream_from = num_reqs <= 2 ? STREAM_FROM_BYTES_FEW : STREAM_FROM_BYTES;
  if constexpr (DT <= 8) {  // (the parts of head size 256 do not fit the LDS of a workgroup)
    // Workgroups of `splits` waves are placed whole: where their number leaves the last round over the CUs thin
    // (320 workgroups on 256 CUs: some CUs get two, most one) single waves spread better and the merge kernel is the
    // lesser cost. Measured at 8 kv heads: 32, 56 and 64 requests gain 0.12 to 0.17 ms a step, 40 and 48 lose.
    // (beside single rows at least one request brings more: its workgroups leave at once)
    const double per_cu = (double)Hkv * (cu && num_reqs > 1 ? num_reqs - 1 : num_reqs) / compute_units();
    if (splits <= JOIN_SPLITS && (per_cu <= 1. || ceil(per_cu) <= 1.15 * per_cu)) {
      auto kernel = p2 ? decode_kernel_for<DT, true, true, POST>(late) : decode_kernel_for<DT, false, true, POST>(late);
      kernel<<<dim3(1, (unsigned)Hkv, (unsigned)num_reqs), 64 * (splits + (late ? 0 : 1)), 0, stream>>>(
          q, ld_q, part, kc, vc, bt, max_blocks, cu, sl, splits, scale * LOG2E, window, H, Hkv, ps, stream_from, out, ld_out,
          post);
      return launch_status();
    }
  }
  auto kernel = p2 ? decode_kernel_for<DT, true, false, POST>(late) : decode_kernel_for<DT, false, false, POST>(late);
  kernel<<<dim3((unsigned)splits, (unsigned)Hkv, (unsigned)num_reqs), 64, 0, stream>>>(
      q, ld_q, part, kc, vc, bt, max_blocks, cu, sl, splits, scale * LOG2E, window, H, Hkv, ps, stream_from,
      (bf16*)nullptr, (int64_t)0, post);
  const int D = DT * 16;
  attn_decode_merge_kernel<<<dim3((unsigned)H, (unsigned)num_reqs), 64, 0, stream>>>(part, out, ld_out, cu, sl, splits,
                                                                                     window, H, D);
  return launch_status();
}

#define DINFER_DISPATCH_HEAD_DIM(head_dim, CALL) \
  switch (head_dim) {                            \
    case 32: { constexpr int DT = 2; CALL; }     \
    case 48: { constexpr int DT = 3; CALL; }     \
    case 64: { constexpr int DT = 4; CALL; }     \
    case 96: { constexpr int DT = 6; CALL; }     \
    case 128: { constexpr int DT = 8; CALL; }    \
    case 256: { constexpr int DT = 16; CALL; }   \
    default: return ERR_UNSUPPORTED;             \
  }

}  // namespace

// 1 if the MFMA kernels take this geometry, else 0 (the caller uses the plain kernel).
extern "C" int dinfer_attn_mfma_supports(int head_dim, int page_size, int heads, int kv_heads) {
  switch (head_dim) {
    case 32: case 48: case 64: case 96: case 128: case 256: break;
    default: return 0;
  }
  if (!(page_size > 0 && page_size % 8 == 0 && kv_heads > 0 && heads % kv_heads == 0)) return 0;
  // the kernels keep the elements of one page (all kv heads) in 32-bit arithmetic
  return (int64_t)kv_heads * page_size * head_dim < (int64_t)1 << 30 ? 1 : 0;
}

// Which kernel dinfer_attn_flash takes at head size 128 without a window: 0 the tile of rows, 1 and 2 the paired waves' (see pair_form).
extern "C" int dinfer_attn_flash_form(int64_t tokens, int num_reqs, int max_q_len, int heads, int kv_heads, int page_size) {
  return takes_pair(page_size, 0) ? pair_form(tokens, num_reqs, max_q_len, heads, kv_heads) : 0;
}

// dinfer_attn_flash at head size 128 without a window by the kernel of paired waves in one of its forms, whatever the counts.
extern "C" int dinfer_attn_flash_pair(int form, const void* q, int64_t ld_q, void* out, int64_t ld_out, const void* k_cache,
                                      const void* v_cache, const int32_t* block_table, int64_t max_blocks,
                                      const int32_t* cu_seqlens, const int32_t* seq_lens, int num_reqs, int64_t tokens, int max_q_len,
                                      float scale, int heads, int kv_heads, int page_size, int skip_single, hipStream_t stream) {
  if (num_reqs <= 0 || max_q_len <= 0 || tokens <= 0) return OK;
  if (!dinfer_attn_mfma_supports(128, page_size, heads, kv_heads) || !takes_pair(page_size, 0) || form < 1 || form > 2) return ERR_UNSUPPORTED;
  if (max_blocks <= 0 || ld_q % 8 || ld_out % 4 || !aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || ((uintptr_t)out % 8))
    return ERR_BAD_SHAPE;
  return (form == 1 ? launch_pair<false> : launch_pair<true>)((const bf16*)q, ld_q, (bf16*)out, ld_out, (const bf16*)k_cache,
                                                              (const bf16*)v_cache, block_table, max_blocks, cu_seqlens, seq_lens, num_reqs,
                                                              tokens, max_q_len, scale, heads, kv_heads, page_size, skip_single, stream);
}

// tokens: rows of all requests together. skip_single: requests with one row are left to the split-K kernel.
extern "C" int dinfer_attn_flash(const void* q, int64_t ld_q, void* out, int64_t ld_out, const void* k_cache,
                                 const void* v_cache, const int32_t* block_table, int64_t max_blocks,
                                 const int32_t* cu_seqlens, const int32_t* seq_lens, int num_reqs, int64_t tokens, int max_q_len,
                                 float scale, int window, int heads, int kv_heads, int head_dim, int page_size,
                                 int skip_single, hipStream_t stream) {
  if (num_reqs <= 0 || max_q_len <= 0 || tokens <= 0) return OK;
  if (!dinfer_attn_mfma_supports(head_dim, page_size, heads, kv_heads)) return ERR_UNSUPPORTED;
  if (window < 0 || max_blocks <= 0 || ld_q % 8 || ld_out % 4 || !aligned16(q) || !aligned16(k_cache) ||
      !aligned16(v_cache) || ((uintptr_t)out % 8))
    return ERR_BAD_SHAPE;
  DINFER_DISPATCH_HEAD_DIM(head_dim, return launch_flash<DT>(
      (const bf16*)q, ld_q, (bf16*)out, ld_out, (const bf16*)k_cache, (const bf16*)v_cache, block_table, max_blocks,
      cu_seqlens, seq_lens, num_reqs, tokens, max_q_len, scale, window, heads, kv_heads, page_size, skip_single, stream));
}

// Single-row requests only. cu_seqlens null: every request brings exactly one row (row b belongs to
// request b). cu_seqlens given: requests with one row are served, the others are left alone.
// Each request's visible keys are cut into `splits` (1..256) equal parts, one wave each.
// part: float workspace of num_reqs * heads * splits * (head_dim + 4) elements.
extern "C" int dinfer_attn_decode(const void* q, int64_t ld_q, void* out, int64_t ld_out, float* part,
                                  int64_t part_elems, const void* k_cache, const void* v_cache,
                                  const int32_t* block_table, int64_t max_blocks, const int32_t* cu_seqlens,
                                  const int32_t* seq_lens, int num_reqs, int splits, float scale, int window,
                                  int heads, int kv_heads, int head_dim, int page_size, hipStream_t stream) {
  if (num_reqs <= 0) return OK;
  if (!dinfer_attn_mfma_supports(head_dim, page_size, heads, kv_heads)) return ERR_UNSUPPORTED;
  if (heads / kv_heads > 16) return ERR_UNSUPPORTED;
  if (window < 0 || max_blocks <= 0 || splits <= 0 || splits > MAX_SPLITS || ld_q % 8 || !aligned16(q) ||
      !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(part) || num_reqs > 65535 || kv_heads > 65535)
    return ERR_BAD_SHAPE;
  if ((int64_t)num_reqs * heads * splits * (head_dim + 4) > part_elems) return 5;
  DINFER_DISPATCH_HEAD_DIM(head_dim, return (launch_decode<DT, false>(
      (const bf16*)q, ld_q, (bf16*)out, ld_out, part, (const bf16*)k_cache, (const bf16*)v_cache, block_table,
      max_blocks, cu_seqlens, seq_lens, num_reqs, splits, scale, window, heads, kv_heads, page_size, DecodePost{},
      stream)));
}

// 1 if dinfer_attn_decode_post takes this head size (both elements of a rotated pair must lie in one lane).
extern "C" int dinfer_attn_decode_post_supports(int head_dim) { return head_dim == 64 || head_dim == 128 || head_dim == 256; }

// dinfer_attn_decode for a step in which every request brings exactly one row, with what otherwise runs as a kernel of
// its own before it: q [rows, ld_q], k_new and v_new (rows of the same stride) come as the q|k|v product left them.
// q and k get their per-head RMSNorm (gains q_gain and k_gain of head_dim bf16 elements; null: none) and are
// rotated by the angles of positions[row] (cos_sin [positions, head_dim] float: cos of the head_dim / 2 angles, then
// sin; pairs (i, i + head_dim / 2); null: no rotation); the new key and value go to slot_mapping[row] of the pages
// (null or negative: nowhere; then the pages must already hold them). q, k_new and v_new are left as they were.
extern "C" int dinfer_attn_decode_post(const void* q, const void* k_new, const void* v_new, int64_t ld_q, void* out,
                                       int64_t ld_out, float* part, int64_t part_elems, void* k_cache, void* v_cache,
                                       const int32_t* block_table, int64_t max_blocks, const int32_t* seq_lens,
                                       int num_reqs, int splits, float scale, int window, int heads, int kv_heads,
                                       int head_dim, int page_size, const void* q_gain, const void* k_gain,
                                       float eps, float gain_offset, const int32_t* positions,
                                       const float* cos_sin, const int64_t* slot_mapping, hipStream_t stream) {
  if (num_reqs <= 0) return OK;
  if (!dinfer_attn_mfma_supports(head_dim, page_size, heads, kv_heads) || !dinfer_attn_decode_post_supports(head_dim))
    return ERR_UNSUPPORTED;
  if (heads / kv_heads > 16) return ERR_UNSUPPORTED;
  if (window < 0 || max_blocks <= 0 || splits <= 0 || splits > MAX_SPLITS || ld_q % 8 || !aligned16(q) ||
      !aligned16(k_new) || !aligned16(v_new) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(part) ||
      !aligned16(q_gain) || !aligned16(k_gain) || !aligned16(cos_sin) || num_reqs > 65535 || kv_heads > 65535 ||
      (cos_sin && !positions) || (!q_gain != !k_gain))
    return ERR_BAD_SHAPE;
  if ((int64_t)num_reqs * heads * splits * (head_dim + 4) > part_elems) return 5;
  DecodePost post{(const bf16*)q_gain, (const bf16*)k_gain, eps, gain_offset, positions, cos_sin, slot_mapping,
                  (const bf16*)k_new, (const bf16*)v_new, (bf16*)k_cache, (bf16*)v_cache};
  switch (head_dim) {
    case 64: return launch_decode<4, true>((const bf16*)q, ld_q, (bf16*)out, ld_out, part, (const bf16*)k_cache,
                                           (const bf16*)v_cache, block_table, max_blocks, nullptr, seq_lens, num_reqs,
                                           splits, scale, window, heads, kv_heads, page_size, post, stream);
    case 128: return launch_decode<8, true>((const bf16*)q, ld_q, (bf16*)out, ld_out, part, (const bf16*)k_cache,
                                            (const bf16*)v_cache, block_table, max_blocks, nullptr, seq_lens, num_reqs,
                                            splits, scale, window, heads, kv_heads, page_size, post, stream);
    default: return launch_decode<16, true>((const bf16*)q, ld_q, (bf16*)out, ld_out, part, (const bf16*)k_cache,
                                            (const bf16*)v_cache, block_table, max_blocks, nullptr, seq_lens, num_reqs,
                                            splits, scale, window, heads, kv_heads, page_size, post, stream);
  }
}
