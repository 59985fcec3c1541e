// Latent attention over prompts with keys and values made again (bf16): where a step brings many rows a request, the products with
// Wuk and Wuv cost less on the key side, once a key, than on the query side, where every score is 576 instead of 192 and every value
// 512 instead of 128 wide:
//
//   k_h,j = [ Wuk_h c_j | kr_j ]     v_h,j = Wuv_h c_j          (heads of 128, values of 128, kr of 64)
//   o_h   = sum_j softmax(scale <[qn_h | rot(qr_h)], k_h,j>) v_h,j, times the sigmoid gate where there is one
//
//   latent_expand_kernel   the keys and values of a step's requests from the cache pages [page][R + 64], straight into the layouts
//                          the attention reads: 16 keys of a head [16 pieces][16][8], its values [128][16], the rotated parts
//                          [8 pieces][16][8] once; request after request, each from a chunk of 16 on
//   attn_pair_kernel       (attention_pair.cuh) over them
//
// The same sums in another order as in latent.hip, with keys and values rounded where that form rounds queries and outputs.
//
// 16 heads over latents of 512, us with the products of the queries' side (which this form has not) and here: 16 x 256 rows behind
// 1,000 keys 437 and 164 (93 for 20,096 keys, 910 TFLOP/s, 165 MB written, and 64), 2,048 rows from nothing 200 and 84, 4,000 592 and 138,
// 512 behind 4,000 317 and 150. Its error against 64 bits is no larger: 2.7e-3 for 3.1e-3 at the first of these. Bound by the matrix
// cores: 2.1 million multiply-adds a key, 192 + 128 a head and score.
#include <algorithm>

#include "attention_pair.cuh"

using namespace dinfer;

namespace {

constexpr int ROWS = 256, KEYS = 256, STAGE = 32768, STAGES = 4;   // a tile; bytes of both operands' 32 k; stages in LDS

// What a workgroup knows of the tiles before it, TILES at most at a time: where their keys are (request, first key, the request's
// length and its first chunk of those that are written), which 256 rows of the weights, and a page for 16 keys or for each page's.
constexpr int TILES = 64, PAGES = 7168;
struct Tile {
  int request, key0, len, chunk0, rows;
};
constexpr int EXPAND_LDS = STAGE * STAGES + TILES * (int)sizeof(Tile) + 16 + PAGES * 4;

// C = W c^T in tiles of 256 weight rows x 256 keys, eight waves of 64 x 128 in v_mfma_f32_32x32x16_bf16. Both operands go from memory
// straight into LDS, 32 k a stage, four stages ahead, 16 rows x 64 bytes an instruction; a row's four pieces are exchanged by bits
// 2 and 3 of its number, so that the fragments' reads meet no bank twice. Fragments are read one set of eight MFMAs ahead in program
// order. Key tiles compute [weight rows][keys], value tiles [keys][weight rows]: two lanes end up with eight consecutive entries of
// a key's piece, or eight consecutive keys of a value row, which one of them stores.
//
// A tile is 16 stages of 32 k for latents of 512, not much longer than its beginning (lengths, table, first loads) and its 128 KB of
// stores. So workgroups stay, one a CU, and walk tiles: where the tiles lie is worked out for all of them before the first, the last
// four steps of a tile send the first stages of the next, and its stores leave beside the next one's first two steps (the third waits
// for them too: it counts what was sent since). 20,096 keys, 16
// heads, 5 tiles a workgroup: 111 us with a workgroup a tile, 97 with this one's walk, 93 with a stage sent as soon as the middle of the
// step that read its place is behind all waves (three steps before its use instead of one to two); one tile each 22 and 23. A step
// is 0.85 us, 1.26 PFLOP/s, and what is left is the beginning, the ends of tiles and the caches' writing back at the end. (Two
// workgroups of 128 weight rows x 256 keys a CU, one's beginning and end beside the other's products: a quarter slower than a workgroup a tile; the row tiles
// of a key tile on one XCD, or half of them: level.)
template <bool VALUES, class Next>
__device__ __forceinline__ void expand_tile(const char* (&src)[4], int steps, uint32_t& stage, char* lds, bf16x8 (&fw)[2][2],
                                            bf16x8 (&fk)[2][4], f32x16 (&acc)[2][4], Next next) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  const uint32_t row = (uint32_t)((wave >> 1) * 64 + l32) * 64, key = 16384u + (uint32_t)((wave & 1) * 128 + l32) * 64;
  const uint32_t slot = (uint32_t)((half ^ ((l32 >> 2) & 3)) * 16);   // of the first 16 k; of the second: 32 bytes over or back
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
#pragma nounroll
  for (int s = 0; s < steps; ++s, ++stage) {
    if (s == steps - 4) next();
    char* const from = lds + ((stage & (STAGES - 1)) * STAGE);
    const char* const ahead = lds + (((stage + 1) & (STAGES - 1)) * STAGE);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const char* const p = (u ? ahead : from) + (slot ^ ((u ^ 1) * 32));
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        const int a = x >> 2, b = x & 3;
        acc[a][b] = VALUES ? mfma32(fk[u][b], fw[u][a], acc[a][b]) : mfma32(fw[u][a], fk[u][b], acc[a][b]);
        if (x == 0) fw[u ^ 1][0] = *(const bf16x8*)(p + row), fw[u ^ 1][1] = *(const bf16x8*)(p + row + 2048);
        if (x == 1 || x == 2)
          fk[u ^ 1][2 * x - 2] = *(const bf16x8*)(p + key + (2 * x - 2) * 2048), fk[u ^ 1][2 * x - 1] = *(const bf16x8*)(p + key + (2 * x - 1) * 2048);
        if (u == 1 && x >= 2 && x < 6) {
          load_to_lds((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)from + wave * 2048 + ((x - 2) >> 1) * 16384 + (x & 1) * 1024,
                      src[x - 2]);
          src[x - 2] += 64;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // Stage s + 1 is here (the first three of a tile were waited for at the end of the one before), and every wave has all of
      // stage s in registers: its place is free for stage s + 4.
      if (u == 0) {
        if (s < 2) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) latent_expand_kernel(
    const bf16* __restrict__ wk, const bf16* __restrict__ wv, const bf16* __restrict__ cache, const int32_t* __restrict__ block_table,
    int64_t max_blocks, const int32_t* __restrict__ seq_lens, int num_reqs, int H, int R, int page_shift, bf16* __restrict__ keys,
    bf16* __restrict__ values, bf16* __restrict__ rot) {
  extern __shared__ __attribute__((aligned(1024))) char expand_smem[];
  Tile* const tiles = (Tile*)(expand_smem + STAGE * STAGES);
  int* const count = (int*)(tiles + TILES);   // of them that there are
  int* const pages = count + 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  const int half_tiles = (H + 1) / 2, row_tiles = 2 * half_tiles;   // (neighbours share the keys, an XCD a few row tiles)
  const int row_bytes = (R + 64) * 2, steps = R / 32, piece_shift = min(page_shift, 4), per_tile = KEYS >> piece_shift;
  const int batch = min(TILES, PAGES / per_tile);   // tiles looked up at once
  const int64_t stride = gridDim.x;
  uint32_t stage = 0;
  for (int64_t t0 = blockIdx.x;; t0 += stride * batch) {   // tile i of the batch: t0 + i * stride, row tile by row tile of a key tile
    if (wave == 0) {   // a lane a request, in order: which of the batch's tiles are its
      int before = 0, chunks_before = 0;
      for (int b0 = 0; b0 < num_reqs; b0 += 64) {
        const int n = b0 + lane < num_reqs ? seq_lens[b0 + lane] : 0, own = (n + KEYS - 1) / KEYS, own_chunks = (n + 15) >> 4;
        int upto = own, chunks = own_chunks;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int v = __builtin_amdgcn_ds_bpermute((lane - o) * 4, upto), w = __builtin_amdgcn_ds_bpermute((lane - o) * 4, chunks);
          if (lane >= o) upto += v, chunks += w;
        }
        const int64_t first = before + upto - own, from = first * row_tiles, to = (int64_t)(before + upto) * row_tiles;
        for (int64_t i = from > t0 ? (from - t0 + stride - 1) / stride : 0; i < batch && t0 + i * stride < to; ++i)
          tiles[i] = Tile{b0 + lane, (int)((t0 + i * stride) / row_tiles - first) * KEYS, n, chunks_before + chunks - own_chunks,
                          (int)((t0 + i * stride) % row_tiles)};
        before += __builtin_amdgcn_readlane(upto, 63);
        chunks_before += __builtin_amdgcn_readlane(chunks, 63);
      }
      const int64_t left = (int64_t)before * row_tiles - t0;
      if (lane == 0) *count = left > 0 ? (int)min((left + stride - 1) / stride, (int64_t)batch) : 0;
    }
    __syncthreads();
    const int n = __builtin_amdgcn_readfirstlane(*count);
    if (n == 0) return;   // (the whole workgroup)
    for (int e = threadIdx.x; e < n * per_tile; e += 512) {   // (keys past the request's: the last one again)
      const Tile t = tiles[e / per_tile];
      pages[e] = block_table[t.request * max_blocks + (min(t.key0 + ((e % per_tile) << piece_shift), t.len - 1) >> page_shift)];
    }
    __syncthreads();
    auto key_at = [&](int i, const Tile& t, int r) __attribute__((always_inline)) {   // key r of tile i
      const int k = min(t.key0 + r, t.len - 1);
      return (const char*)cache +
             ((int64_t)pages[i * per_tile + ((k - t.key0) >> piece_shift)] * (1 << page_shift) + (k & ((1 << page_shift) - 1))) * row_bytes;
    };
    const char* src[4];   // of this wave's 32 rows of W, and its 32 keys
    auto sources = [&](int i) __attribute__((always_inline)) {
      const Tile t = tiles[i];
      const int rt = __builtin_amdgcn_readfirstlane(t.rows), row0 = (rt >= half_tiles ? rt - half_tiles : rt) * ROWS;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int r = wave * 32 + x * 16 + (lane >> 2), piece = ((lane & 3) ^ ((r >> 2) & 3)) * 16;
        src[x] = (const char*)(rt >= half_tiles ? wv : wk) + (int64_t)min(row0 + r, H * 128 - 1) * (R * 2) + piece;
        src[2 + x] = key_at(i, t, r) + piece;
      }
    };
    bf16x8 fw[2][2], fk[2][4];
    sources(0);
#pragma unroll
    for (int x = 0; x < 4; ++x) asm volatile("" : "+v"(src[x]));
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        load_to_lds((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)expand_smem + ((stage + s) & (STAGES - 1)) * STAGE +
                        wave * 2048 + (x >> 1) * 16384 + (x & 1) * 1024, src[x]);
        src[x] += 64;
      }
    // the rotated parts of the keys, a row tile's share of the pieces of 16 bytes
    const int share = (KEYS * 8 + row_tiles - 1) / row_tiles;
    for (int e = threadIdx.x; e < n * share; e += 512) {
      const int i = e / share;
      const Tile t = tiles[i];
      const int p = t.rows * share + e % share, k = p >> 3;
      if (p >= KEYS * 8 || ((t.key0 + k) >> 4) >= ((t.len + 15) >> 4)) continue;
      *(bf16x8*)(rot + ((int64_t)(t.chunk0 + ((t.key0 + k) >> 4)) * 8 + (p & 7)) * 128 + (k & 15) * 8) =
          *(const bf16x8*)(key_at(i, t, k) + R * 2 + (p & 7) * 16);
    }
    loads_barrier<4>();
    {
      const uint32_t row = (uint32_t)((wave >> 1) * 64 + l32) * 64, key = 16384u + (uint32_t)((wave & 1) * 128 + l32) * 64;
      const char* const p = expand_smem + (stage & (STAGES - 1)) * STAGE + (half ^ ((l32 >> 2) & 3)) * 16;
#pragma unroll
      for (int x = 0; x < 2; ++x) fw[0][x] = *(const bf16x8*)(p + row + x * 2048);
#pragma unroll
      for (int x = 0; x < 4; ++x) fk[0][x] = *(const bf16x8*)(p + key + x * 2048);
    }
    for (int i = 0; i < n; ++i) {
      const Tile t = tiles[i];
      const int rt = __builtin_amdgcn_readfirstlane(t.rows);
      const bool is_value = rt >= half_tiles;
      const int row0 = (is_value ? rt - half_tiles : rt) * ROWS;
      // (past the last tile: its own first stages again, into LDS that nobody reads)
      auto next = [&]() __attribute__((always_inline)) {
        sources(min(i + 1, n - 1));
      };
      f32x16 acc[2][4];
      if (is_value) expand_tile<true>(src, steps, stage, expand_smem, fw, fk, acc, next);
      else expand_tile<false>(src, steps, stage, expand_smem, fw, fk, acc, next);
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");   // the next tile's first three stages (not the stores below)
      bf16* const out = is_value ? values : keys;
      const int first = __builtin_amdgcn_readfirstlane(t.chunk0 + (t.key0 >> 4));
      const int chunks = __builtin_amdgcn_readfirstlane(((t.len + 15) >> 4) - (t.key0 >> 4));   // from this tile's first on
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int d0 = row0 + (wave >> 1) * 64 + a * 32, head = d0 >> 7;   // 32 rows of a head
        if (head >= H) break;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            // a lane's four of sets i and i + 1, and the other half's: of set i + half all eight
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            bf16x4 r0, r1;
#pragma unroll
            for (int e = 0; e < 4; ++e) r0[e] = (bf16)acc[a][c][4 * i + e], r1[e] = (bf16)acc[a][c][4 * i + 4 + e];
            typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
            const u32x2 w0 = __builtin_bit_cast(u32x2, r0), w1 = __builtin_bit_cast(u32x2, r1);
            const auto lo = __builtin_amdgcn_permlane32_swap(w0[0], w1[0], false, false), hi = __builtin_amdgcn_permlane32_swap(w0[1], w1[1], false, false);
            const u32x4 r = {lo[0], hi[0], lo[1], hi[1]};
            // key tiles: key l32 of the 32, entries 8 (i + half) ..; value tiles: row l32, keys 8 (i + half) ..
            const int k = (wave & 1) * 128 + c * 32 + (is_value ? 8 * i : l32), chunk = k >> 4;
            if (chunk >= chunks) continue;
            bf16* page = out + ((int64_t)(first + chunk) * H + head) * 2048;
            if (is_value) *(u32x4*)(page + ((d0 & 127) + l32) * 16 + 8 * half) = r;
            else *(u32x4*)(page + (((d0 & 127) >> 3) + i + half) * 128 + (k & 15) * 8) = r;
          }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing on its way into LDS
    __syncthreads();   // before the next batch is looked up
  }
}

}  // namespace

// Whether latent_attn_expanded takes these sizes.
extern "C" int dinfer_latent_expanded_supports(int dn, int dr, int dv, int R, int page_size) {
  return dn == 128 && dr == 64 && dv == 128 && R >= 128 && R <= 512 && R % 32 == 0 && page_size > 0 && (page_size & (page_size - 1)) == 0;
}

// bf16. Attention of the requests' rows, causal, over latent pages [blocks][page][R + 64]. q: head h's 128 unrotated entries at
// h * q_stride, qr its 64 rotated ones at h * qr_stride; wk, wv [heads * 128][R]; out [rows][heads * 128]. gate: see PairExpanded.
// keys, values: room for `chunks` pieces of 16 keys of heads * 128 entries, rot the same of 64; total_keys: the requests' lengths summed
// up, longest: the longest (both known on the host, or bounds of them).
extern "C" int dinfer_latent_attn_expanded(const void* q, int64_t ld_q, int q_stride, const void* qr, int64_t ld_qr, int qr_stride,
                                           const void* wk, const void* wv, void* out, int64_t ld_out, const void* gate,
                                           int64_t ld_gate, int gate_entries, const void* cache, const int32_t* block_table,
                                           int64_t max_blocks, const int32_t* cu_seqlens, const int32_t* seq_lens, int num_reqs,
                                           int64_t total_keys, int max_q_len, float scale, int heads, int R, int page_size,
                                           void* keys, void* values, void* rot, int64_t chunks, hipStream_t stream) {
  if (num_reqs <= 0 || max_q_len <= 0) return OK;
  if (!dinfer_latent_expanded_supports(128, 64, 128, R, page_size)) return ERR_UNSUPPORTED;
  auto off = [](const void* p, int n) { return (uintptr_t)p % n != 0; };
  if (heads <= 0 || max_blocks <= 0 || total_keys <= 0 || ld_q % 8 || q_stride % 8 || ld_qr % 8 || qr_stride % 8 || ld_out % 4 ||
      off(q, 16) || off(qr, 16) || off(wk, 16) || off(wv, 16) || off(out, 8) || off(cache, 16) || off(keys, 16) || off(values, 16) ||
      off(rot, 16) || (gate && gate_entries && (ld_gate % 4 || off(gate, 8))))
    return ERR_BAD_SHAPE;
  if (total_keys / 16 + num_reqs > chunks || chunks > 0x7fffffff / 16) return ERR_WORKSPACE;
  const int64_t row_tiles = 2 * ((heads + 1) / 2), blocks = (total_keys / KEYS + num_reqs) * row_tiles;
  const int64_t tiles = (max_q_len + 255) / 256, pairs = tiles * num_reqs * heads;
  if (blocks > 0x7fffffff || pairs > 0x7fffffff || (int64_t)heads * 4096 > 0x7fffffff) return ERR_UNSUPPORTED;
  const unsigned places = (unsigned)std::min<int64_t>(blocks, compute_units());
  auto attention = attn_pair_kernel<false, true>;
  if (hipFuncSetAttribute((const void*)latent_expand_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, EXPAND_LDS) != hipSuccess ||
      hipFuncSetAttribute((const void*)attention, hipFuncAttributeMaxDynamicSharedMemorySize, pair_lds(false, true)) != hipSuccess)
    return ERR_LAUNCH;
  latent_expand_kernel<<<places, 512, EXPAND_LDS, stream>>>((const bf16*)wk, (const bf16*)wv, (const bf16*)cache, block_table,
                                                                         max_blocks, seq_lens, num_reqs, heads, R,
                                                                         __builtin_ctz(page_size), (bf16*)keys, (bf16*)values, (bf16*)rot);
  if (launch_status() != OK) return ERR_LAUNCH;
  const PairExpanded ex{(const bf16*)rot, (const bf16*)qr, ld_qr, q_stride, qr_stride, (const bf16*)gate, ld_gate, gate_entries};
  attention<<<(unsigned)pairs, 512, pair_lds(false, true), stream>>>((const bf16*)q, ld_q, (bf16*)out, ld_out, (const bf16*)keys,
                                                                     (const bf16*)values, nullptr, 0, cu_seqlens, seq_lens, num_reqs,
                                                                     (int)tiles, 0, scale * LOG2E, heads, heads, 16, 0, ex);
  return launch_status();
}
