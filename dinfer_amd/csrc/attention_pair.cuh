// Flash attention over long runs of rows (bf16, head size 128, causal, no options): eight waves a workgroup in two groups of
// four, a wave of each on every SIMD, that take turns: while one group's waves fill the matrix cores with the scores of a block
// of 64 keys and the values of the block before, the other's work on their softmax.
//
// A wave owns 32 columns, a column being a query head of the kv head and a row: column c of a request is row c / G, head c % G
// of the group, so that keys and values are read once for all heads of a group whatever their number. S^T = K . Q^T and
// O^T = V^T . P in v_mfma_f32_32x32x16_bf16, whose operands want, per lane, 8 consecutive elements of the contraction dimension:
//   A (32 x 16): lane l holds A[l % 32][8 * (l / 32) .. + 8]
//   B (16 x 32): lane l holds B[8 * (l / 32) .. + 8][l % 32]
//   D (32 x 32): lane l holds D[8 * (i / 4) + 4 * (l / 32) + i % 4][l % 32], i = 0..15
// Row 8 b + 4 h + r of a score tile stands for key 16 (b / 2) + 8 h + 4 (b % 2) + r, so that a lane ends up with the weights of
// eight consecutive keys twice: the B operand of the second product, with no shuffle.
//
// Keys and values go from their pages straight into LDS (global_load_lds, 1 KB an instruction: 16 keys x 4 pieces, 32 value
// rows x 16 keys, both contiguous in a page of 16), into rings of blocks that run two to three turns ahead; the waits for them
// are counted, and nothing else waits on vmcnt inside the loop.
//
//   HALVES = false  the workgroup's 256 columns, every block for all eight waves
//   HALVES = true   128 columns; the first four waves take the even blocks, the others the odd ones, each with a ring of
//                   their own, and the two results meet in LDS at the end: twice the tiles, half as long each
//
// Bound by the two phases, a group's 1,180 cycles of MFMAs (1,024 at least) beside the other's 1,250 of softmax, and by power:
// behind a long history the MFMAs fill 61 to 63 % of the cycles and the chip lowers its clock to 1.4 to 1.7 GHz (a prompt of 4,096:
// 46 %, 2.0 GHz). LDS is read in 31 % of the cycles, at 256 bytes each.
//
// 2,001 rows behind 28,000, 32 heads over 8: 1,272 us with the tile of rows (747 TFLOP/s; keys and values through registers, a
// wave's softmax and its MFMAs after each other) and 818 here (1,160). Of that: fragments read eight ahead of their MFMA in program
// order 1,111 -> 880; table entries looked up a turn ahead, behind the MFMAs, and keys and values of one page an instruction 862 ->
// 818; blocks further ahead or the loads beside the softmax nothing, or slower (846, 906).
#pragma once
#include <type_traits>

#include "attention_tile.cuh"
#include "lds_loads.cuh"

namespace dinfer {
namespace {

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// At most N of this wave's loads into LDS still on their way, then the workgroup's barrier (reads of LDS need no wait here: what
// a turn reads is used before the barrier behind it, and no ring overwrites a block within a turn of its last use).
template <int N>
__device__ __forceinline__ void loads_barrier() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

constexpr int least(int a, int b) { return a < b ? a : b; }
constexpr int pair_columns(bool halves) { return halves ? 128 : 256; }
constexpr int PAIR_BLOCK = 16384;   // bytes of 64 keys of 128, or of their values
constexpr int pair_ahead(bool halves) { return halves ? 2 : 3; }    // turns from a block of keys' loads to its scores
constexpr int pair_behind(bool halves) { return halves ? 2 : 1; }   // turns from a block of keys' loads to its values'
constexpr int pair_keys(bool halves) { return pair_ahead(halves) + 1; }
constexpr int pair_values(bool halves) { return pair_ahead(halves) - pair_behind(halves) + 2; }
constexpr int PAIR_ROT = 8192;      // bytes of 64 keys' rotated parts of 64 (EXPANDED)
constexpr int pair_lds(bool halves, bool expanded = false) {
  return (pair_keys(halves) * (PAIR_BLOCK + (expanded ? PAIR_ROT : 0)) + pair_values(halves) * PAIR_BLOCK) * (halves ? 2 : 1);
}

// EXPANDED: keys and values of every head made from a latent cache for this step (H of 16 keys' pages each, request after request
// without a table), a key's last 64 entries shared by the heads: `rot`, a page of 16 keys [8 pieces][16][8] each. q holds the first 128
// entries of a head's query, qr the others. gate (may be null): a row's outputs are multiplied by the sigmoid of entry h, or
// (gate_entries) by that of entry 128 h + d.
struct PairExpanded {
  const bf16* rot;
  const bf16* qr;
  int64_t ld_qr;
  int q_stride, qr_stride;   // from head to head
  const bf16* gate;
  int64_t ld_gate;
  int gate_entries;
};

// ps: a power of two, 16 or more. count: `tiles_x` is not a request's tiles; those that exist are counted up over the requests.
template <bool HALVES, bool EXPANDED = false>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) attn_pair_kernel(
    const bf16* __restrict__ q, int64_t ld_q, bf16* __restrict__ out, int64_t ld_out, const bf16* __restrict__ kc,
    const bf16* __restrict__ vc, const int32_t* __restrict__ block_table, int64_t max_blocks,
    const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ seq_lens, int num_reqs, int tiles_x, int count,
    float scale_log2e, int H, int Hkv, int ps, int skip_single, PairExpanded ex = PairExpanded{}) {
  constexpr int D = 128, COLS = pair_columns(HALVES);
  constexpr int AK = pair_ahead(HALVES), LAG = pair_behind(HALVES), AV = AK - LAG, NK = pair_keys(HALVES), NV = pair_values(HALVES);
  constexpr int LOADS = HALVES ? 4 : 2;   // instructions a wave brings of a block's 16 of keys, and of its values
  constexpr int PIECES = EXPANDED ? 12 : 8, KEY_FRAGS = 2 * PIECES, KEY_BLOCK = PAIR_BLOCK + (EXPANDED ? PAIR_ROT : 0);
  static_assert(!(HALVES && EXPANDED), "does not fit LDS");
  // (the reference the weights are taken against follows the maximum once that has risen by this much, in base-2 units: with 6
  // instead of 2 1 % faster, but the largest weights, 1 exactly where the reference is their own score, are rounded more often)
  constexpr float LAZY = 2.f;
  extern __shared__ __attribute__((aligned(1024))) char pair_smem[];
  // An XCD (workgroup id modulo 8) keeps to few kv heads; tiles with the most keys first. Workgroups go to the XCDs, and inside one to
  // its four shader engines, in turn: with an even number of requests one of them would meet the same engines (of few kv heads, the
  // same XCDs) with all its tiles, and a long one beside short ones leave the others idle. So the requests move on by one from tile
  // to tile. 2,001 rows behind 283 beside seven requests of 2 to 588, 16 heads over 4: 201 us without and 57 with; 1,684 behind 7,612
  // beside three of 4 to 1,235, 32 over 8: 679 and 258.
  const int hk = blockIdx.x % Hkv, rest = blockIdx.x / Hkv, G = H / Hkv;
  int tile = tiles_x - 1 - rest / num_reqs, b = (num_reqs & 1 ? rest : rest + rest / num_reqs) % num_reqs;
  if (count) {
    int ln = threadIdx.x & 63;
    asm volatile("" : "+v"(ln));   // (nothing of the count lives on in registers)
    int at = rest;
    b = -1;
    for (int b0 = 0; b0 < num_reqs && b < 0; b0 += 64) {
      const int len = b0 + ln < num_reqs ? cu_seqlens[b0 + ln + 1] - cu_seqlens[b0 + ln] : 0;
      int upto = skip_single && len == 1 ? 0 : (len * G + COLS - 1) / COLS;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __builtin_amdgcn_ds_bpermute((ln - o) * 4, upto);   // (below lane 0: any lane, not taken)
        if (ln >= o) upto += v;
      }
      const unsigned long long holds = __ballot(at < upto);
      if (holds) {
        const int l = __ffsll((long long)holds) - 1;
        b = b0 + l;
        tile = __builtin_amdgcn_readlane(upto, l) - 1 - at;
      } else {
        at -= __builtin_amdgcn_readlane(upto, 63);
      }
    }
    if (b < 0) return;   // (the whole workgroup, here and below)
  }
  const int q_begin = cu_seqlens[b];
  const int q_len = cu_seqlens[b + 1] - q_begin;
  const int hist = seq_lens[b] - q_len;
  const int c_first = tile * COLS;
  if (c_first >= q_len * G || (skip_single && q_len == 1)) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  const int grp = wave >> 2, member = HALVES ? wave & 3 : wave;   // member: of those that share a ring
  const int cw = c_first + member * 32;                           // this wave's first column
  const int last_row = q_len - 1;
  const int col = cw + l32;
  const int row = min(col / G, last_row), head = hk * G + col % G;   // (columns past the last row: computed, not stored)
  const int pos = hist + row;
  const int w_hi = hist + min((cw + 31) / G, last_row) + 1;          // keys that some column of the wave sees
  const int all_hi = hist + min((c_first + COLS - 1) / G, last_row) + 1;
  const int blocks = (all_hi + 63) >> 6, whole = (hist + c_first / G + 1) >> 6;   // whole: blocks that every row sees whole
  // this group's turns (of an odd number the last of the second group sees nothing), and how many need no mask
  const int turns = HALVES ? (blocks + 1) >> 1 : blocks;
  const int plain = min(turns, HALVES ? (whole + 1 - grp) >> 1 : whole);
  auto first_key = [&](int j) __attribute__((always_inline)) { return (HALVES ? 2 * j + grp : j) * 64; };

  // ---- loads: chunk c (16 keys) and quarter t of its pieces, or of its value rows, an instruction --------------------------
  constexpr int VALUES = NK * KEY_BLOCK;   // where the ring of values begins
  char* const ring = pair_smem + (HALVES ? grp * (NK + NV) * PAIR_BLOCK : 0);
  const uint32_t ring_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring;
  const int n0 = member * LOADS;
  const char* const kh = (const char*)kc + (int64_t)hk * ps * D * 2 + (uint32_t)((4 * (n0 & 3) + (lane >> 4)) * ps + (lane & 15)) * 16;
  const char* const vh = (const char*)vc + (int64_t)hk * ps * D * 2 + (uint32_t)((32 * (n0 & 3) + l32) * ps + half * 8) * 2;
  typedef const __attribute__((address_space(4))) int32_t* Entries;   // (scalar loads)
  const Entries bt = (Entries)(block_table + (int64_t)b * max_blocks);
  const uint32_t page_bytes = (uint32_t)Hkv * ps * D * 2;             // (the host checks that this fits)
  const int ps_shift = __builtin_ctz(ps), last_chunk = (all_hi - 1) >> 4;
  int chunk = (HALVES ? grp * 4 : 0) + (n0 >> 2), page;
  uint64_t k_at, v_at[LAG + 1];
  const char *k_src, *v_src, *r_src = nullptr;
  int first_page = 0;                    // EXPANDED: the request's
  if constexpr (EXPANDED) {
    int ln = threadIdx.x & 63, pages = 0;
    asm volatile("" : "+v"(ln));
    for (int b0 = ln; b0 < b; b0 += 64) pages += (seq_lens[b0] + 15) >> 4;
#pragma unroll
    for (int x = 32; x > 0; x >>= 1) pages += __shfl_xor(pages, x, 64);
    first_page = __builtin_amdgcn_readfirstlane(pages);
  }
  const char* const rh = (const char*)ex.rot + (uint32_t)((4 * (member & 1) + (lane >> 4)) * 16 + (lane & 15)) * 16;
  // The entry of the next block's chunk (past the last: that one again, its keys are masked), and a turn later what follows from it.
  auto look = [&]() __attribute__((always_inline)) {
    page = EXPANDED ? first_page + min(chunk, last_chunk) : bt[(min(chunk, last_chunk) << 4) >> ps_shift];
  };
  auto aim = [&]() __attribute__((always_inline)) {
    const uint64_t at = (uint64_t)(uint32_t)page * page_bytes;
    const int off = EXPANDED ? 0 : (min(chunk, last_chunk) << 4) & (ps - 1);
    if constexpr (EXPANDED) r_src = rh + (uint64_t)(uint32_t)page * 2048;
    k_at = at + (uint32_t)(off * 16);
#pragma unroll
    for (int i = 0; i < LAG; ++i) v_at[i] = v_at[i + 1];
    v_at[LAG] = at + (uint32_t)(off * 2);
    chunk += HALVES ? 8 : 4;
  };
  auto send_k = [&](int j, int x) __attribute__((always_inline)) {
    load_to_lds(ring_at + (uint32_t)(j % NK * KEY_BLOCK + (n0 + x) * 1024), k_src + (uint32_t)(x * 64 * ps));
  };
  auto send_v = [&](int j, int x) __attribute__((always_inline)) {
    load_to_lds(ring_at + (uint32_t)(VALUES + j % NV * PAIR_BLOCK + (n0 + x) * 1024), v_src + (uint32_t)(x * 64 * ps));
  };
  auto send_r = [&](int j) __attribute__((always_inline)) {   // (chunk member / 2: the one this wave brings keys of)
    load_to_lds(ring_at + (uint32_t)(j % NK * KEY_BLOCK + PAIR_BLOCK + member * 1024), r_src);
  };

  bf16x8 qf[PIECES];
  {
    const bf16* qp = q + (int64_t)(q_begin + row) * ld_q + (int64_t)head * (EXPANDED ? ex.q_stride : D) + half * 8;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = *(const bf16x8*)(qp + ks * 16);
    if constexpr (EXPANDED) {
      const bf16* rp = ex.qr + (int64_t)(q_begin + row) * ex.ld_qr + (int64_t)head * ex.qr_stride + half * 8;
#pragma unroll
      for (int ks = 8; ks < PIECES; ++ks) qf[ks] = *(const bf16x8*)(rp + (ks - 8) * 16);
    }
#pragma unroll
    for (int ks = 0; ks < PIECES; ++ks) asm volatile("" : "+v"(qf[ks]));   // here before the first counted wait
  }
  f32x16 o[4], s[2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[t][i] = 0.f;
  float m = -INFINITY, l = 0.f;
  bf16x8 pf[4], fr[8];   // weights; fragments of keys and values, eight ahead

  // a turn's fragments: keys (piece x / 2 of the tile x % 2), then values (chunk x / 4, rows 32 (x % 4) ..)
  const uint32_t k_frag = (uint32_t)(half * 256 + (8 * ((l32 >> 2) & 1) + 4 * ((l32 >> 3) & 1) + (l32 & 3)) * 16), k_page = l32 >> 4;
  auto key_frag = [&](int j, int x) __attribute__((always_inline)) {
    const char* at = ring + j % NK * KEY_BLOCK + k_frag;
    return EXPANDED && x >= 16 ? *(const bf16x8*)(at + k_page * 2048 + PAIR_BLOCK + (x & 1) * 4096 + ((x >> 1) - 8) * 512)
                               : *(const bf16x8*)(at + k_page * 4096 + (x & 1) * 8192 + (x >> 1) * 512);
  };
  auto value_frag = [&](int j, int x) __attribute__((always_inline)) {
    return *(const bf16x8*)(ring + VALUES + j % NV * PAIR_BLOCK + lane * 16 + x * 1024);
  };
  auto first_frags = [&](int j) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < 8; ++x) fr[x] = key_frag(j, x);
  };
  // a stale slot may hold anything; its weight is 0, but 0 * inf would poison the sum
  auto clean = [&](bf16x8& v, int key) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = key + e < w_hi ? v[e] : (bf16)0.f;
  };

  // Scores of block j and values of block j - 1, in this order: an MFMA, the fragment eight on, and somewhere between them what
  // the loads of the blocks ahead need (beside the softmax, which has no issue slots to spare, they cost 5 %).
  auto products = [&](int j, auto first, auto masked) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first)::value, MASK = decltype(masked)::value;
    constexpr int LAST = KEY_FRAGS + (FIRST ? 0 : 16);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[a][i] = 0.f;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < LAST; ++x) {
      if (x < KEY_FRAGS) {
        s[x & 1] = mfma32(fr[x & 7], qf[x >> 1], s[x & 1]);
      } else {
        if constexpr (MASK) clean(fr[x & 7], first_key(j - 1) + 16 * ((x - KEY_FRAGS) >> 2) + 8 * half);
        o[x & 3] = mfma32(fr[x & 7], pf[(x - KEY_FRAGS) >> 2], o[x & 3]);
      }
      if (x + 8 < LAST) fr[x & 7] = x + 8 < KEY_FRAGS ? key_frag(j, x + 8) : value_frag(j - 1, x + 8 - KEY_FRAGS);
      if (x == 1) { aim(); k_src = kh + k_at; }
      if (x == 3) v_src = vh + v_at[0];
      if constexpr (HALVES) {
        if (x >= 4 && x < 8) send_v(j + AV, x - 4);
        if (x >= 9 && x < 13) send_k(j + AK, x - 9);
      } else {
        if (x == 4 || x == 6) send_k(j + AK, (x - 4) / 2);
        if (EXPANDED && x == 8) send_r(j + AK);
        if (x == 9 || x == 12) send_v(j + AV, (x - 9) / 3);
      }
      if (x == LAST - 1) look();
      if constexpr (!MASK) __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto softmax = [&](int j, auto masked) __attribute__((always_inline)) {
    if constexpr (decltype(masked)::value) {
      const int kg = first_key(j) + 8 * half;
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[a][i] = kg + 32 * a + 16 * (i >> 3) + (i & 7) <= pos ? s[a][i] : -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[a][i]);
    // (both halves of a column keep the same m: they need to meet only where it moves)
    if (__any((mx - m) * scale_log2e > LAZY)) {
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m, mx);
      const float alpha = m_new == m ? 1.f : exp2_raw((m - m_new) * scale_log2e);   // m = -inf: 0
      l *= alpha;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] *= alpha;
      m = m_new;
    }
    const float mc = (m == -INFINITY ? 0.f : m) * scale_log2e;   // nothing visible yet: everything stays zero
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = exp2_raw(fmaf(s[a][i], scale_log2e, -mc));
        sum[i & 3] += p;
        pf[a * 2 + (i >> 3)][i & 7] = (bf16)p;
      }
    l += (sum[0] + sum[1]) + (sum[2] + sum[3]);
  };

  // ---- the turns ----------------------------------------------------------------------------------------------------------------
  // Barrier 2 j comes before the first group's products of block j and behind the second's of block j - 1, barrier 2 j + 1 the other
  // way round. Behind barrier 2 j values j - 1 and keys j must have landed, behind 2 j + 1 keys j + 1 (the fragments that the first
  // group reads beside its softmax) and values j - 1; HALVES, where a group waits for its own loads only: keys j + 1 behind the
  // products of block j, values j - 1 before them. What may then still be on its way, in instructions of a wave:
  constexpr int TURN = EXPANDED ? 5 : 4;   // keys, then 2 of values
  constexpr int TOP_1 = HALVES ? 4 : least(TURN * AV, TURN * (AK - 1) + 2), END_1 = HALVES ? 8 : least(TURN * (AK - 1) + 2, TURN * (AV + 1));
  constexpr int TOP_2 = HALVES ? 4 : least(TURN * (AK - 2) + 2, TURN * AV), END_2 = HALVES ? 8 : TOP_1;
  static_assert(HALVES ? AK == 2 && AV == 0 : AV == AK - 1, "the counts above");
  auto turn = [&](int j, auto first, auto masked) __attribute__((always_inline)) {
    if (grp) loads_barrier<TOP_2>(); else loads_barrier<TOP_1>();
    __builtin_amdgcn_s_setprio(1);
    products(j, first, masked);
    __builtin_amdgcn_s_setprio(0);
    if (grp) loads_barrier<END_2>(); else loads_barrier<END_1>();
    first_frags(j + 1);
    __builtin_amdgcn_sched_barrier(0);
    softmax(j, masked);
    __builtin_amdgcn_sched_barrier(0);
  };
  using Yes = std::true_type;
  using No = std::false_type;
#pragma unroll
  for (int i = 0; i < AK; ++i) {
    look();
    aim();
    k_src = kh + k_at;
#pragma unroll
    for (int x = 0; x < LOADS; ++x) send_k(i, x);
    if (EXPANDED) send_r(i);
    if (i >= LAG) {
      v_src = vh + v_at[0];
#pragma unroll
      for (int x = 0; x < LOADS; ++x) send_v(i - LAG, x);
    }
  }
  look();
  loads_barrier<HALVES ? 4 : TURN * (AK - 1)>();   // keys 0
  first_frags(0);
  if (grp) loads_barrier<END_2>();
  if (plain > 0) turn(0, Yes{}, No{}); else turn(0, Yes{}, Yes{});
  int j = 1;
#pragma nounroll
  for (; j < plain; ++j) turn(j, No{}, No{});
#pragma nounroll
  for (; j < turns; ++j) turn(j, No{}, Yes{});
  loads_barrier<0>();   // (what was loaded past the last block has landed too: LDS is the waves' own from the last barrier on)
#pragma unroll
  for (int x = 0; x < 16; ++x) {
    bf16x8 v = value_frag(turns - 1, x);
    clean(v, first_key(turns - 1) + 16 * (x >> 2) + 8 * half);
    o[x & 3] = mfma32(v, pf[x >> 2], o[x & 3]);
  }
  if (!grp) loads_barrier<0>();

  if constexpr (HALVES) {   // o = 2^(c (m_1 - M)) o_1 + 2^(c (m_2 - M)) o_2, likewise l; a lane's share lies in the same places in both
    __syncthreads();
    f32x4* const part = (f32x4*)pair_smem;
    float* const part_ml = (float*)(part + 16 * 256);
    const int at = member * 64 + lane;
    if (grp) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[(t * 4 + i) * 256 + at] = f32x4{o[t][4 * i], o[t][4 * i + 1], o[t][4 * i + 2], o[t][4 * i + 3]};
      part_ml[at] = m;
      part_ml[256 + at] = l;
    }
    __syncthreads();
    if (grp) return;
    const float m2 = part_ml[at], l2 = part_ml[256 + at];
    const float M = fmaxf(m, m2), mc = (M == -INFINITY ? 0.f : M) * scale_log2e;
    const float a1 = exp2_raw(fmaf(m, scale_log2e, -mc)), a2 = exp2_raw(fmaf(m2, scale_log2e, -mc));   // nothing seen: 0
    l = l * a1 + l2 * a2;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 x = part[(t * 4 + i) * 256 + at];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[t][4 * i + e] = o[t][4 * i + e] * a1 + x[e] * a2;
      }
  }
  l += __shfl_xor(l, 32, 64);
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (col >= q_len * G) return;
  const bf16* gate = nullptr;
  if constexpr (EXPANDED) {
    if (ex.gate) {
      gate = ex.gate + (int64_t)(q_begin + row) * ex.ld_gate + (ex.gate_entries ? head * D + 4 * half : head);
      if (!ex.gate_entries) inv *= 1.f / (1.f + expf(-(float)*gate));
    }
  }
  bf16* op = out + (int64_t)(q_begin + row) * ld_out + (int64_t)head * D + 4 * half;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      bf16x4 r;
#pragma unroll
      for (int k = 0; k < 4; ++k) r[k] = (bf16)(o[t][4 * i + k] * inv);
      if constexpr (EXPANDED) {
        if (gate && ex.gate_entries) {
          const bf16x4 g = *(const bf16x4*)(gate + 32 * t + 8 * i);
#pragma unroll
          for (int k = 0; k < 4; ++k) r[k] = (bf16)(o[t][4 * i + k] * inv * (1.f / (1.f + expf(-(float)g[k]))));
        }
      }
      *(bf16x4*)(op + 32 * t + 8 * i) = r;
    }
}

}  // namespace
}  // namespace dinfer
