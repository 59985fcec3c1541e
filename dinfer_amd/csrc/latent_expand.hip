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
// 1,000 keys 438 and 178 (some 125 for 20,096 keys, 670 TFLOP/s, 165 MB written, and 48), 2,048 rows from nothing 200 and 85, 4,000 595 and 136,
// 512 behind 4,000 318 and 151. Its error against 64 bits is no larger: 2.7e-3 for 3.1e-3 at the first of these. Bound by the matrix
// cores: 2.1 million multiply-adds a key, 192 + 128 a head and score.
#include <algorithm>

#include "attention_pair.cuh"

using namespace dinfer;

namespace {

constexpr int ROWS = 256, KEYS = 256, STAGE = 32768, STAGES = 4;   // a tile; bytes of both operands' 32 k; stages in LDS

// C = W c^T in tiles of 256 weight rows x 256 keys, eight waves of 64 x 128 in v_mfma_f32_32x32x16_bf16. Both operands go from memory
// straight into LDS, 32 k a stage, three stages ahead, 16 rows x 64 bytes an instruction; a row's four pieces are exchanged by bits
// 2 and 3 of its number, so that the fragments' reads meet no bank twice. Fragments are read one set of eight MFMAs ahead in program
// order. Key tiles compute [weight rows][keys], value tiles [keys][weight rows]: a lane ends up with four consecutive entries of a
// key's piece, or four consecutive keys of a value row, either way 8 bytes of what lies together. (Two workgroups of 128 weight rows x 256
// keys a CU, one's beginning and end beside the other's products: 20,096 keys 158 us for 125, more bytes of both operands a product.)
template <bool VALUES>
__device__ __forceinline__ void expand_tile(const char* const (&src)[4], int steps, char* lds, f32x16 (&acc)[2][4]) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds + wave * 2048;
  // instructions 0, 1: this wave's 32 rows of W, 2, 3: its 32 keys
  auto send = [&](int s, int x) __attribute__((always_inline)) {
    // (past the last: that one again, into a stage that nobody reads)
    load_to_lds(at + (uint32_t)((s & (STAGES - 1)) * STAGE + (x >> 1) * 16384 + (x & 1) * 1024), src[x] + min(s, steps - 1) * 64);
  };
  const uint32_t row = (uint32_t)((wave >> 1) * 64 + l32) * 64, key = 16384u + (uint32_t)((wave & 1) * 128 + l32) * 64;
  const uint32_t slot = (uint32_t)((half ^ ((l32 >> 2) & 3)) * 16);   // of the first 16 k; of the second: 32 bytes over or back
  bf16x8 fw[2][2], fk[2][4];
  auto frag = [&](int s, int u, int x) __attribute__((always_inline)) {   // fragment x of a set of six
    const char* p = lds + (s & (STAGES - 1)) * STAGE + (slot ^ (u * 32));
    if (x < 2) fw[u][x] = *(const bf16x8*)(p + row + x * 2048);
    else fk[u][x - 2] = *(const bf16x8*)(p + key + (x - 2) * 2048);
  };
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int x = 0; x < 4; ++x) send(s, x);
  loads_barrier<8>();
#pragma unroll
  for (int x = 0; x < 6; ++x) frag(0, 0, x);
#pragma nounroll
  for (int s = 0; s < steps; ++s) {
    loads_barrier<4>();   // stage s + 1 is here, and every wave is done with stage s - 1
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        const int a = x >> 2, b = x & 3;
        acc[a][b] = VALUES ? mfma32(fk[u][b], fw[u][a], acc[a][b]) : mfma32(fw[u][a], fk[u][b], acc[a][b]);
        if (x < 6) frag(u ? s + 1 : s, u ^ 1, x);   // (past the last step: a stage that is not used)
        if (x == 3 || x == 7) send(s + 3, u * 2 + (x >> 2));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  loads_barrier<0>();
}

__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) latent_expand_kernel(
    const bf16* __restrict__ wk, const bf16* __restrict__ wv, const bf16* __restrict__ cache, const int32_t* __restrict__ block_table,
    int64_t max_blocks, const int32_t* __restrict__ seq_lens, int num_reqs, int H, int R, int page_shift, bf16* __restrict__ keys,
    bf16* __restrict__ values, bf16* __restrict__ rot) {
  extern __shared__ __attribute__((aligned(1024))) char expand_smem[];
  const int half_tiles = (H + 1) / 2, rt = blockIdx.x % (2 * half_tiles);   // (neighbours share the keys, an XCD a few row tiles)
  int at = blockIdx.x / (2 * half_tiles), b = -1, len = 0, chunk0 = 0;
  {   // the request of key tile `at`, and its first chunk
    const int ln = threadIdx.x & 63;
    for (int b0 = 0; b0 < num_reqs && b < 0; b0 += 64) {
      const int n = b0 + ln < num_reqs ? seq_lens[b0 + ln] : 0;
      int upto = (n + KEYS - 1) / KEYS, chunks = (n + 15) >> 4;
      const int own = chunks;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __builtin_amdgcn_ds_bpermute((ln - o) * 4, upto), w = __builtin_amdgcn_ds_bpermute((ln - o) * 4, chunks);
        if (ln >= o) upto += v, chunks += w;
      }
      const unsigned long long holds = __ballot(at < upto);
      if (holds) {
        const int l = __ffsll((long long)holds) - 1;
        b = b0 + l;
        len = __builtin_amdgcn_readlane(n, l);
        at -= __builtin_amdgcn_readlane(upto, l) - (len + KEYS - 1) / KEYS;
        chunk0 += __builtin_amdgcn_readlane(chunks, l) - __builtin_amdgcn_readlane(own, l);
      } else {
        at -= __builtin_amdgcn_readlane(upto, 63);
        chunk0 += __builtin_amdgcn_readlane(chunks, 63);
      }
    }
    if (b < 0) return;   // (the whole workgroup)
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  const bool is_value = rt >= half_tiles;
  const int row0 = (is_value ? rt - half_tiles : rt) * ROWS, key0 = at * KEYS, row_bytes = (R + 64) * 2;
  const int32_t* bt = block_table + (int64_t)b * max_blocks;
  auto key_at = [&](int k) __attribute__((always_inline)) {   // (keys past the request's: the last one again)
    k = min(k, len - 1);
    return (const char*)cache + ((int64_t)bt[k >> page_shift] * (1 << page_shift) + (k & ((1 << page_shift) - 1))) * row_bytes;
  };
  const char* src[4];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int r = wave * 32 + x * 16 + (lane >> 2), piece = ((lane & 3) ^ ((r >> 2) & 3)) * 16;
    src[x] = (const char*)(is_value ? wv : wk) + (int64_t)min(row0 + r, H * 128 - 1) * (R * 2) + piece;
    src[2 + x] = key_at(key0 + r) + piece;
  }
  const int chunks = ((len + 15) >> 4) - (key0 >> 4);   // from this tile's first on
  if (rt == 0) {   // the rotated parts: a thread a key's piece
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int i = x * 512 + threadIdx.x, k = i >> 3, piece = i & 7;
      if ((k >> 4) < chunks)
        *(bf16x8*)(rot + ((int64_t)(chunk0 + ((key0 + k) >> 4)) * 8 + piece) * 128 + (k & 15) * 8) =
            *(const bf16x8*)(key_at(key0 + k) + R * 2 + piece * 16);
    }
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) asm volatile("" : "+v"(src[x]));   // (addresses here before the first counted wait)
  f32x16 acc[2][4];
  if (is_value) expand_tile<true>(src, R / 32, expand_smem, acc);
  else expand_tile<false>(src, R / 32, expand_smem, acc);
  bf16* const out = is_value ? values : keys;
  const int first = chunk0 + (key0 >> 4);
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int d0 = row0 + (wave >> 1) * 64 + a * 32, head = d0 >> 7;   // 32 rows of a head
    if (head >= H) break;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bf16x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = (bf16)acc[a][c][4 * i + e];
        // key tiles: key l32 of the 32, entries 8 i + 4 half ..; value tiles: row l32, keys 8 i + 4 half ..
        const int k = (wave & 1) * 128 + c * 32 + (is_value ? 8 * i : l32), chunk = k >> 4;
        if (chunk >= chunks) continue;
        bf16* page = out + ((int64_t)(first + chunk) * H + head) * 2048;
        if (is_value) *(bf16x4*)(page + ((d0 & 127) + l32) * 16 + (k & 15) + 4 * half) = r;
        else *(bf16x4*)(page + (((d0 & 127) >> 3) + i) * 128 + (k & 15) * 8 + 4 * half) = r;
      }
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
  auto attention = attn_pair_kernel<false, true>;
  if (hipFuncSetAttribute((const void*)latent_expand_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, STAGE * STAGES) != hipSuccess ||
      hipFuncSetAttribute((const void*)attention, hipFuncAttributeMaxDynamicSharedMemorySize, pair_lds(false, true)) != hipSuccess)
    return ERR_LAUNCH;
  latent_expand_kernel<<<(unsigned)blocks, 512, STAGE * STAGES, stream>>>((const bf16*)wk, (const bf16*)wv, (const bf16*)cache, block_table,
                                                                         max_blocks, seq_lens, num_reqs, heads, R,
                                                                         __builtin_ctz(page_size), (bf16*)keys, (bf16*)values, (bf16*)rot);
  if (launch_status() != OK) return ERR_LAUNCH;
  const PairExpanded ex{(const bf16*)rot, (const bf16*)qr, ld_qr, q_stride, qr_stride, (const bf16*)gate, ld_gate, gate_entries};
  attention<<<(unsigned)pairs, 512, pair_lds(false, true), stream>>>((const bf16*)q, ld_q, (bf16*)out, ld_out, (const bf16*)keys,
                                                                     (const bf16*)values, nullptr, 0, cu_seqlens, seq_lens, num_reqs,
                                                                     (int)tiles, 0, scale * LOG2E, heads, heads, 16, 0, ex);
  return launch_status();
}
