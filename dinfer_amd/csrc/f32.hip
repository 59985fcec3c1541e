// The 32-bit path on the matrix cores: matrix products and paged attention with v_mfma_f32_16x16x4_f32 (operands,
// products and sums in 32 bits; 256 flop a cycle and CU, as much as the vector ALUs' fused multiply-adds but without a
// load of LDS per multiply). gemm_ref.hip and attention_ref.hip take what does not fit here.
//
// What an output's sum is made of depends on its own operands only, never on the number of rows, the tile or the kernel:
//   products   k is cut into segments of SEG; a segment is summed from zero by one chain of MFMAs in ascending k, the
//              segments are added in ascending order. Both kernels below do exactly this, so a row computed alone has
//              the bits it has inside a prompt. (The error against 64 bits is below that of one chain over all of k:
//              2,048 long, 2.9e-7 against 8.1e-7.)
//   attention  keys are visited in blocks of 64 that begin at multiples of 64; block b belongs to wave b % 4, the waves'
//              parts are joined in wave order, and a block that a row does not see leaves its sums as they are.
//
// Operand order: lane l gives row l % 16 and, of 16 consecutive k, the four from 4 * (l / 16) on, one 16-byte load that
// feeds four MFMAs; which k meet in one MFMA does not matter as long as both operands agree.
//
// Reference behaviour: crates/layers/src/nn.rs:16-76 (y = x . W^T), crates/kernels/cuda/gqa.cu:1037-1118 (plain paged
// attention: causal inclusive, query head h reads kv head h / G).
#include <algorithm>

#include "common.cuh"

using namespace dinfer;

namespace {

constexpr int SEG = 256;   // k summed in one chain

__device__ __forceinline__ f32x4 mfma4(const f32x4& a, const f32x4& b, f32x4 c) {
#pragma unroll
  for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
  return c;
}

// ---- products of many rows --------------------------------------------------------------------------------------
// A workgroup of KG groups of WM x WN waves computes BM rows x BN columns, a wave a tile of 32 x 32; the groups deal the
// segments of k among themselves and their sums are added in the segments' order. Steps of 32 k go through two LDS buffers: the
// loads of a step go out three steps before it, it is written to LDS one step before, and of the two halves of a step the second is
// read while the first is multiplied and the next step's first while the second is, so that a wave meets neither LDS nor
// the barrier between its MFMAs. Loads are buffer loads (one addition an address; past the last row's k they give zero): 64-bit
// addresses cost the vector ALUs a tenth of the MFMAs' time. v_mfma_f32_32x32x2_f32 with k in the order of the few-row kernel's
// 16x16x4 rounds to the same bits. Rows of LDS are 36 floats apart: the lanes that a 16-byte read serves at a time lie in
// different banks. Bound by the matrix cores and, where a CU gets one workgroup, by a step's latency (before: steps
// of 64 k through 16x16x4 tiles, fetched two ahead, LDS read behind each barrier, accumulators moved between register files
// every step): 500 rows x 6,144 x 1,024 74 -> 59 us (107 TFLOP/s where a large library product reaches 153), x 4,096 x 1,024
// 49 -> 40, x 1,024 x 2,048 31 -> 26, x 1,024 x 3,072 44 -> 36; 2,000 x 6,144 x 1,024 256 -> 196.
constexpr int KB = 32, LROW = KB + 4;

template <int WM, int WN, int KG>
__global__ void __launch_bounds__(64 * WM * WN * KG) gemm_f32_kernel(const float* __restrict__ A, int64_t lda,
                                                                     const float* __restrict__ W, int64_t ldw,
                                                                     float* __restrict__ C, int64_t ldc, int M, int N, int K) {
  constexpr int BM = 32 * WM, BN = 32 * WN, GT = 64 * WM * WN;             // threads of a group
  constexpr int PASS = GT / (KB / 4);                                      // rows a pass of 16-byte loads
  constexpr int LA = BM / PASS, LW = BN / PASS;                            // passes a step
  constexpr int STEPS = SEG / KB;                                          // of a segment
  __shared__ float As[KG][2][BM * LROW];
  __shared__ float Ws[KG][2][BN * LROW];
  __shared__ f32x4 part[KG][KG > 1 ? 4 * GT : 1];
  const int tid = threadIdx.x % GT, group = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / GT) : 0;
  const int lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = wave / WN * 32, wn = wave % WN * 32;
  const int lr = lane & 31, lh = lane >> 5;
  const int row = tid / (KB / 4), piece = tid % (KB / 4) * 4;

  // rows past the last one are the last one; what lies behind its k reads as zero
  const int a_last = min(BM, M - m0) - 1, w_last = min(BN, N - n0) - 1;
  const auto ab = __builtin_amdgcn_make_buffer_rsrc((void*)(A + (int64_t)m0 * lda), 0, (int)(((int64_t)a_last * lda + K) * 4), 0x00020000);
  const auto wb = __builtin_amdgcn_make_buffer_rsrc((void*)(W + (int64_t)n0 * ldw), 0, (int)(((int64_t)w_last * ldw + K) * 4), 0x00020000);
  uint32_t oa[LA], ow[LW];
#pragma unroll
  for (int e = 0; e < LA; ++e) oa[e] = ((uint32_t)min(row + PASS * e, a_last) * (uint32_t)lda + piece) * 4;
#pragma unroll
  for (int e = 0; e < LW; ++e) ow[e] = ((uint32_t)min(row + PASS * e, w_last) * (uint32_t)ldw + piece) * 4;

  f32x4 ra[2][LA], rw[2][LW];
  auto fetch = [&](int k0, f32x4(&fa)[LA], f32x4(&fw)[LW]) {
#pragma unroll
    for (int e = 0; e < LA; ++e) fa[e] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ab, oa[e] + k0 * 4, 0, 0));
#pragma unroll
    for (int e = 0; e < LW; ++e) fw[e] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, ow[e] + k0 * 4, 0, 0));
  };
  auto put = [&](int b, int k0, f32x4(&fa)[LA], f32x4(&fw)[LW]) {
    if (k0 + KB > K) {
      const bool keep = k0 + piece < K;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int e = 0; e < LA; ++e) fa[e][i] = keep ? fa[e][i] : 0.f;
#pragma unroll
        for (int e = 0; e < LW; ++e) fw[e][i] = keep ? fw[e][i] : 0.f;
      }
    }
#pragma unroll
    for (int e = 0; e < LA; ++e) *(f32x4*)&As[group][b][(row + PASS * e) * LROW + piece] = fa[e];
#pragma unroll
    for (int e = 0; e < LW; ++e) *(f32x4*)&Ws[group][b][(row + PASS * e) * LROW + piece] = fw[e];
  };
  struct Half { f32x4 a[2], w[2]; };   // of a step: 16 k
  auto read = [&](int b, int c, Half& f) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f.a[h] = *(const f32x4*)&As[group][b][(wm + lr) * LROW + 16 * c + 8 * h + 4 * lh];
      f.w[h] = *(const f32x4*)&Ws[group][b][(wn + lr) * LROW + 16 * c + 8 * h + 4 * lh];
    }
  };
  constexpr int OWN = 4 / KG;   // with groups, a thread sums up the four columns of every KG-th of the four row pieces
  f32x16 acc;
  f32x4 tot[OWN];
#pragma unroll
  for (auto& t : tot) t = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Half& f) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(f.w[h][q], f.a[h][q], acc, 0, 0, 0);
  };

  const int segs = (K + SEG - 1) / SEG;
  const int rounds = (segs + KG - 1) / KG;
  Half f0, f1;
  {
    const int k0 = group * SEG;
    fetch(k0, ra[0], rw[0]);
    fetch(k0 + KB, ra[1], rw[1]);
    put(0, k0, ra[0], rw[0]);
    fetch(k0 + 2 * KB, ra[0], rw[0]);
    lds_barrier();
    read(0, 0, f0);
  }
  for (int r0 = 0; r0 < rounds; ++r0) {
    const int k0 = (r0 * KG + group) * SEG, next = k0 + KG * SEG;   // this segment, the group's next
    const int steps = KG > 1 ? STEPS : (min(K - r0 * SEG, SEG) + 2 * KB - 1) / (2 * KB) * 2;
    auto at = [&](int s) { return s < steps ? k0 + s * KB : next + (s - steps) * KB; };
    acc = f32x16{};
#pragma unroll 1
    for (int s0 = 0; s0 < steps; s0 += 2) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        read(b, 1, f1);
        put(b ^ 1, at(s0 + b + 1), ra[b ^ 1], rw[b ^ 1]);
        fetch(at(s0 + b + 3), ra[b ^ 1], rw[b ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f0);
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        read(b ^ 1, 0, f0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const f32x4 x = {acc[4 * r], acc[4 * r + 1], acc[4 * r + 2], acc[4 * r + 3]};
      if (KG > 1) part[group][r * GT + tid] = x;
      else tot[r] += x;
    }
    if (KG > 1) {   // (the parts are written again behind the barriers of the next segment)
      lds_barrier();
      const int have = min(KG, segs - r0 * KG);
#pragma unroll
      for (int o = 0; o < OWN; ++o)
        for (int g = 0; g < have; ++g) tot[o] += part[g][o * KG * GT + threadIdx.x];
    }
  }
  // a lane holds four consecutive columns of one row at a time
  const bool wide = ldc % 4 == 0 && ((uintptr_t)C & 15) == 0;
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
    const int m = m0 + wm + lr, n = n0 + wn + 8 * (o * KG + group) + 4 * lh;
    if (m >= M) continue;
    float* c = C + (int64_t)m * ldc + n;
    if (wide && n + 3 < N) *(f32x4*)c = tot[o];
    else
#pragma unroll
      for (int y = 0; y < 4; ++y)
        if (n + y < N) c[y] = tot[o][y];
  }
}

// ---- products of few rows ---------------------------------------------------------------------------------------
// A workgroup takes 16 rows of the weight and 16 * MT rows of A and streams both straight into registers: its waves deal
// the segments of k among themselves (no barrier inside one), GROUP pieces of 16 k in flight at a time, and after each
// round the parts are added in segment order. Bound by the weight's bytes, and by latency where the weight is small:
// 151,936 x 1,024 in 124 us at one row (5.0 TB/s; the vector-ALU kernel 401), 1,024 x 3,072 in 12 us (365), at 32 rows 21.
template <int NW, int MT>
__global__ void __launch_bounds__(NW * 64) gemm_f32_few_kernel(const float* __restrict__ A, int64_t lda, const float* __restrict__ W,
                                                               int64_t ldw, float* __restrict__ C, int64_t ldc, int M, int N,
                                                               int K) {
  constexpr int GROUP = 16 / MT, GROUPS = SEG / 16 / GROUP;
  __shared__ float part[NW][MT][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT;
  const float* w = W + (int64_t)min(n0 + lr, N - 1) * ldw;
  const float* a[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) a[i] = A + (int64_t)min(m0 + 16 * i + lr, M - 1) * lda;
  const int segs = (K + SEG - 1) / SEG;
  constexpr int OWN = (MT * 256 + NW * 64 - 1) / (NW * 64);   // outputs a thread
  float tot[OWN];
#pragma unroll
  for (int x = 0; x < OWN; ++x) tot[x] = 0.f;
  for (int s0 = 0; s0 < segs; s0 += NW) {
    const int s = s0 + wave;
    if (s < segs) {
      f32x4 acc[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int k0 = s * SEG + 4 * lg;
      if (s * SEG + SEG <= K) {
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) {
          f32x4 fw[GROUP], fa[GROUP][MT];
#pragma unroll
          for (int c = 0; c < GROUP; ++c) {
            fw[c] = *(const f32x4*)(w + k0 + 16 * (g * GROUP + c));
#pragma unroll
            for (int i = 0; i < MT; ++i) fa[c][i] = *(const f32x4*)(a[i] + k0 + 16 * (g * GROUP + c));
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int c = 0; c < GROUP; ++c)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i] = mfma4(fw[c], fa[c][i], acc[i]);
        }
      } else {
        for (int k = k0; k - 4 * lg < K; k += 16) {
          const int kk = min(k, K - 4);
          f32x4 fw = *(const f32x4*)(w + kk);
#pragma unroll
          for (int r = 0; r < 4; ++r) fw[r] = k < K ? fw[r] : 0.f;
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            f32x4 fa = *(const f32x4*)(a[i] + kk);
#pragma unroll
            for (int r = 0; r < 4; ++r) fa[r] = k < K ? fa[r] : 0.f;
            acc[i] = mfma4(fw, fa, acc[i]);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) *(f32x4*)&part[wave][i][lane * 4] = acc[i];
    }
    __syncthreads();
#pragma unroll
    for (int x = 0; x < OWN; ++x) {
      const int e = x * NW * 64 + threadIdx.x;
      if (e < MT * 256)
        for (int i = 0; i < min(NW, segs - s0); ++i) tot[x] += part[i][e >> 8][e & 255];
    }
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < OWN; ++x) {
    const int e = x * NW * 64 + threadIdx.x, l = (e & 255) >> 2;
    const int m = m0 + 16 * (e >> 8) + (l & 15), n = n0 + 4 * (l >> 4) + (e & 3);
    if (e < MT * 256 && m < M && n < N) C[(int64_t)m * ldc + n] = tot[x];
  }
}

template <int MT>
void launch_few(const float* a, int64_t lda, const float* w, int64_t ldw, float* c, int64_t ldc, int M, int N, int K, hipStream_t stream) {
  constexpr int MOST = 65535 * 16 * MT;   // rows that a grid's y holds
  for (int m0 = 0; m0 < M; m0 += std::min(MOST, M - m0)) {
    const int rows = std::min(MOST, M - m0);
    const dim3 grid((unsigned)((N + 15) / 16), (unsigned)((rows + 16 * MT - 1) / (16 * MT)));
    if (K > 4 * SEG)
      gemm_f32_few_kernel<8, MT><<<grid, 512, 0, stream>>>(a + m0 * lda, lda, w, ldw, c + m0 * ldc, ldc, rows, N, K);
    else
      gemm_f32_few_kernel<4, MT><<<grid, 256, 0, stream>>>(a + m0 * lda, lda, w, ldw, c + m0 * ldc, ldc, rows, N, K);
  }
}

// ---- attention --------------------------------------------------------------------------------------------------
// A workgroup takes 16 * CT query rows (token, head of the group) of one kv head; its four waves take the key blocks in
// turn. Scores are K . Q^T, so that a lane holds 4 consecutive keys of one query and its probabilities are the operand
// that V^T . P wants: nothing passes between lanes but the row maxima. The pages' layouts give both operands as 16-byte
// loads (K [D / 8][page][8], V [D][page]). Bound by the matrix cores and the waves' unequal shares: a prompt of 500 tokens of 16 heads on
// 8 of 128 in 35 us (the plain kernel 1,177), 8 rows behind 700 keys each in 27 (514), one behind 4,000 in 101 (2,856).
template <int DT, int CT>
__global__ void __launch_bounds__(256, DT <= 8 ? 2 : 1) attn_f32_kernel(
    const float* __restrict__ q, int64_t ld_q, float* __restrict__ out, int64_t ld_out, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, const int32_t* __restrict__ block_table, int64_t max_blocks,
    const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ seq_lens, float scale, int window, int G, int Hkv,
    int page) {
#pragma clang fp contract(off)   // the instances must round alike
  constexpr int D = 16 * DT, WAVES = 4;
  __shared__ float po[WAVES - 1][CT][DT][256];
  __shared__ float pm[WAVES][CT][16], pl[WAVES][CT][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  // Workgroups in the order of their dispatch: kv heads fastest, then a request's row tiles, the later half from its end down
  // (most keys), then the earlier half from its start up, so that the two or so workgroups that share a CU are a long and a
  // short one (500 rows, 63 tiles x 8 heads: 30.0 us, 32.4 with the tiles of a head in ascending order).
  const int tiles = (int)gridDim.x / Hkv;
  const int hk = (int)blockIdx.x % Hkv, x = (int)blockIdx.x / Hkv, later = (tiles + 1) / 2;
  const int tile = x < later ? tiles - 1 - x : x - later;
  const int b = blockIdx.y;
  const int t0 = cu_seqlens[b], q_len = cu_seqlens[b + 1] - t0;
  const int rows = q_len * G, r0 = tile * 16 * CT;
  if (r0 >= rows) return;   // the whole workgroup
  const int hist = seq_lens[b] - q_len;
  const int32_t* bt = block_table + (int64_t)b * max_blocks;

  int pos[CT];
  f32x4 fq[CT][DT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int r = min(r0 + 16 * c + lr, rows - 1);
    pos[c] = hist + r / G;
    const float* qr = q + (int64_t)(t0 + r / G) * ld_q + (int64_t)(hk * G + r % G) * D + 4 * lg;
#pragma unroll
    for (int d = 0; d < DT; ++d) fq[c][d] = *(const f32x4*)(qr + 16 * d);
  }
  const int p_first = hist + r0 / G, p_last = hist + min(r0 + 16 * CT - 1, rows - 1) / G;
  const int first = window > 0 ? max(p_first - window + 1, 0) : 0;

  f32x4 o[CT][DT];
  float m[CT], l[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    m[c] = -INFINITY;
    l[c] = 0.f;
#pragma unroll
    for (int d = 0; d < DT; ++d) o[c][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  int blk = first / 64;
  blk += (wave - blk % WAVES + WAVES) % WAVES;
  for (; blk * 64 <= p_last; blk += WAVES) {
    const int j0 = blk * 64;
    f32x4 s[CT][4];
    // the pieces of the next tile of 16 keys (behind the last one: of the first values) travel while one is multiplied
    constexpr bool AHEAD = DT <= 8;   // (beyond, registers do not hold two tiles' pieces)
    f32x4 fk[AHEAD ? 2 : 1][DT];
    auto keys = [&](int t, f32x4(&f)[DT]) {
      const int j = max(min(j0 + 16 * t + lr, p_last), first);   // (pages behind the window may be given back)
      const float* kr = k_cache + ((int64_t)bt[j / page] * Hkv + hk) * page * D + (int64_t)((lg >> 1) * page + j % page) * 8 + 4 * (lg & 1);
#pragma unroll
      for (int d = 0; d < DT; ++d) f[d] = *(const f32x4*)(kr + (int64_t)d * 16 * page);
    };
    auto values = [&](int t, f32x4(&f)[DT]) {
      const int j = max(min(j0 + 16 * t + 4 * lg, p_last & ~3), first & ~3);
      const float* vr = v_cache + (((int64_t)bt[j / page] * Hkv + hk) * D + lr) * page + j % page;
#pragma unroll
      for (int d = 0; d < DT; ++d) f[d] = *(const f32x4*)(vr + (int64_t)d * 16 * page);
    };
    if (AHEAD) keys(0, fk[0]);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (!AHEAD) keys(t, fk[0]);
      else if (t < 3) keys(t + 1, fk[(t + 1) & 1]);
      else values(0, fk[0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < CT; ++c) s[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int c = 0; c < CT; ++c) s[c][t] = mfma4(fk[AHEAD ? t & 1 : 0][d], fq[c][d], s[c][t]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      float top = -INFINITY;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = j0 + 16 * t + 4 * lg + i;
          const bool seen = j <= pos[c] && (window == 0 || j > pos[c] - window);
          s[c][t][i] = seen ? s[c][t][i] * scale : -INFINITY;
          top = fmaxf(top, s[c][t][i]);
        }
      top = fmaxf(top, __shfl_xor(top, 16, 64));
      top = fmaxf(top, __shfl_xor(top, 32, 64));
      const float m_new = fmaxf(m[c], top);
      const float base = m_new == -INFINITY ? 0.f : m_new;   // a row that has seen nothing yet
      const float alpha = expf(m[c] - base);                 // 1 where the maximum stands, 0 at a row's first block
      m[c] = m_new;
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[c][t][i] = expf(s[c][t][i] - base);
          sum += s[c][t][i];
        }
      l[c] = __builtin_fmaf(l[c], alpha, sum);
#pragma unroll
      for (int d = 0; d < DT; ++d) o[c][d] *= alpha;
    }
    const bool edge = j0 + 63 > p_first || (window > 0 && j0 <= p_last - window);   // some row does not see some key
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x4(&fv)[DT] = fk[AHEAD ? t & 1 : 0];
      if (!AHEAD) values(t, fv);
      else if (t < 3) values(t + 1, fk[(t + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      if (edge) {
        bool odd = false;   // an infinity or NaN among the values: 0 times it is not 0
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            fv[d][i] = j0 + 16 * t + 4 * lg + i <= p_last ? fv[d][i] : 0.f;   // beyond the tile's last key: unwritten
            odd |= !(fabsf(fv[d][i]) < INFINITY);
          }
        if (__any(odd)) {
          // key by key, kept only where the row sees it (never taken while a model's numbers are finite)
#pragma unroll 1
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int key = j0 + 16 * t + 4 * g + i;
#pragma unroll
              for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                  const bool seen = key <= pos[c] && (window == 0 || key > pos[c] - window);
                  const f32x4 x = __builtin_amdgcn_mfma_f32_16x16x4f32(lg == g ? fv[d][i] : 0.f, lg == g ? s[c][t][i] : 0.f, o[c][d], 0, 0, 0);
#pragma unroll
                  for (int r = 0; r < 4; ++r) o[c][d][r] = seen ? x[r] : o[c][d][r];
                }
            }
          continue;
        }
      }
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int c = 0; c < CT; ++c) o[c][d] = mfma4(fv[d], s[c][t], o[c][d]);
    }
  }

  // the waves' parts, joined in wave order
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    l[c] += __shfl_xor(l[c], 16, 64);
    l[c] += __shfl_xor(l[c], 32, 64);
    if (lg == 0) {
      pm[wave][c][lr] = m[c];
      pl[wave][c][lr] = l[c];
    }
    if (wave > 0)
#pragma unroll
      for (int d = 0; d < DT; ++d) *(f32x4*)&po[wave - 1][c][d][lane * 4] = o[c][d];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    float top = m[c];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = fmaxf(top, pm[w][c][lr]);
    const float base = top == -INFINITY ? 0.f : top;
    float share[WAVES], sum = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      share[w] = expf(pm[w][c][lr] - base);
      sum = __builtin_fmaf(pl[w][c][lr], share[w], sum);
    }
    const float inv = sum > 0.f ? 1.f / sum : 0.f;
    const int r = r0 + 16 * c + lr;
    float* orow = out + (int64_t)(t0 + min(r, rows - 1) / G) * ld_out + (int64_t)(hk * G + min(r, rows - 1) % G) * D + 4 * lg;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      f32x4 x = o[c][d] * share[0];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) {
        const f32x4 y = *(const f32x4*)&po[w - 1][c][d][lane * 4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = __builtin_fmaf(y[i], share[w], x[i]);
      }
      if (r < rows) *(f32x4*)(orow + 16 * d) = x * inv;
    }
  }
}

template <int DT, int CT>
void launch_attn(const float* q, int64_t ld_q, float* out, int64_t ld_out, const float* k, const float* v, const int32_t* bt,
                 int64_t max_blocks, const int32_t* cu, const int32_t* sl, int reqs, int max_q, float scale, int window, int G,
                 int Hkv, int page, hipStream_t stream) {
  const dim3 grid((unsigned)(((int64_t)max_q * G + 16 * CT - 1) / (16 * CT) * Hkv), (unsigned)reqs);
  attn_f32_kernel<DT, CT><<<grid, 256, 0, stream>>>(q, ld_q, out, ld_out, k, v, bt, max_blocks, cu, sl, scale, window, G, Hkv, page);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

// Whether dinfer_gemm_f32 takes operands of these strides (in floats) and addresses: 16-byte pieces along k, which ends so
// early that two steps or a segment behind it are still 32-bit numbers.
extern "C" int dinfer_gemm_f32_supports(const void* A, int64_t lda, const void* W, int64_t ldw, int64_t K) {
  return K >= 4 && K % 4 == 0 && K <= 0x7fffffff - 2 * SEG && lda % 4 == 0 && ldw % 4 == 0 && aligned16(A) && aligned16(W);
}

// C[M, N] = A[M, K] . W[N, K]^T, all float32.
extern "C" int dinfer_gemm_f32(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, int64_t M,
                               int64_t N, int64_t K, hipStream_t stream) {
  if (M <= 0 || N <= 0) return OK;
  if (K <= 0 || lda < K || ldw < K || ldc < N || M > 0x7fffffff - 64 || N > 0x7fffffff - 64) return ERR_BAD_SHAPE;
  if (!dinfer_gemm_f32_supports(A, lda, W, ldw, K) || (M + 63) / 64 > 65535) return ERR_UNSUPPORTED;   // (as many rows as gemm_ref)
  const float *a = (const float*)A, *w = (const float*)W;
  float* c = (float*)C;
  const int m = (int)M, n = (int)N, k = (int)K;
  // Up to 16 rows, and up to 32 of a weight that gives its workgroups of 16 columns no second round of the CUs, the kernel
  // whose waves split k (17 and 32 rows x 1,024 x 2,048: 12 and 15 us, 17 and 18 in tiles; x 6,144 x 1,024 15 and 17 against 13
  // and 14; from 33 rows on it would need two more tiles of 16: 64 rows x 1,024 x 2,048 22 against 18, x 151,936 x 1,024
  // 373 against 207), and where a tile's rows reach past 2^31 bytes. Otherwise the tile whose workgroups take a CU the least
  // time: x workgroups a CU and 1,024 k cost it these us, measured at 64 to 2,000 rows of six weights (workgroups of 32 x 128
  // share a CU three at a time; alone, a group of waves waits for its latencies, which is what groups over k are for).
  auto spans = [&](int64_t rows, int64_t ld) { return ((rows - 1) * ld + K + 8 * SEG) * 4 < 0x7fffffff; };
  if (M <= 16) launch_few<1>(a, lda, w, ldw, c, ldc, m, n, k, stream);
  else if ((M <= 32 && N <= 4096) || !spans(std::min<int64_t>(M, 64), lda) || !spans(std::min<int64_t>(N, 128), ldw)) launch_few<2>(a, lda, w, ldw, c, ldc, m, n, k, stream);
  else {
    auto a_cu = [&](int64_t bm, int64_t bn) { return (double)((((M + bm - 1) / bm) * ((N + bn - 1) / bn) + 255) / 256); };
    const double t64x64 = a_cu(64, 64), t32x64 = a_cu(32, 64);
    const double cost[] = {31 * a_cu(64, 128), 17 * a_cu(32, 128) + 4, 19 * t64x64, t32x64 < 2 ? 12 : 10 * t32x64,
                           t32x64 < 2 ? 10 : 11.5 * t32x64, 7 * a_cu(32, 32)};
    const int best = (int)(std::min_element(cost, cost + 6) - cost);
#define DINFER_GEMM_F32(WM, WN, KG)                                                                                      \
  gemm_f32_kernel<WM, WN, KG><<<dim3((unsigned)((N + 32 * WN - 1) / (32 * WN)), (unsigned)((M + 32 * WM - 1) / (32 * WM))), \
                                64 * WM * WN * KG, 0, stream>>>(a, lda, w, ldw, c, ldc, m, n, k)
    switch ((M + 31) / 32 > 65535 ? 0 : best) {   // (the grid's y)
      case 0: DINFER_GEMM_F32(2, 4, 1); break;
      case 1: DINFER_GEMM_F32(1, 4, 1); break;
      case 2: DINFER_GEMM_F32(2, 2, 2); break;
      case 3: DINFER_GEMM_F32(1, 2, 2); break;
      case 4: DINFER_GEMM_F32(1, 2, 4); break;
      default: DINFER_GEMM_F32(1, 1, 4);
    }
#undef DINFER_GEMM_F32
  }
  return launch_status();
}

// Whether dinfer_attn_f32 takes a geometry: whole tiles of 16 in the head, four keys of a page side by side.
extern "C" int dinfer_attn_f32_supports(int head_dim, int page_size, int heads, int kv_heads) {
  if (head_dim <= 0 || page_size <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || page_size % 4 != 0) return 0;
  switch (head_dim) {
    case 16: case 32: case 48: case 64: case 80: case 96: case 112: case 128: case 192: case 256: return 1;
    default: return 0;
  }
}

// Paged attention in 32 bits; operands as dinfer_attn_paged_ref. max_q: at least the longest portion of the step.
extern "C" int dinfer_attn_f32(const void* q, int64_t ld_q, void* out, int64_t ld_out, const void* k_cache, const void* v_cache,
                               const int32_t* block_table, int64_t max_blocks, const int32_t* cu_seqlens, const int32_t* seq_lens,
                               int num_reqs, int max_q, float scale, int window, int heads, int kv_heads, int head_dim,
                               int page_size, hipStream_t stream) {
  if (num_reqs <= 0 || max_q <= 0) return OK;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || max_blocks <= 0 || window < 0) return ERR_BAD_SHAPE;
  if (!dinfer_attn_f32_supports(head_dim, page_size, heads, kv_heads) || num_reqs > 65535 || kv_heads > 65535 || ld_q % 4 != 0 ||
      ld_out % 4 != 0 || !aligned16(q) || !aligned16(out) || !aligned16(k_cache) || !aligned16(v_cache) ||
      (int64_t)max_q * (heads / kv_heads) > 0x7fffffff - 64 || ((int64_t)max_q * (heads / kv_heads) + 15) / 16 * kv_heads > 0x7fffffff)
    return ERR_UNSUPPORTED;
  const int G = heads / kv_heads;
  const bool two = (int64_t)max_q * G > 16;   // two tiles of rows share the keys and values a wave loads (up to heads of 64: registers)
#define DINFER_ATTN_F32(DT, CT)                                                                                              \
  launch_attn<DT, CT>((const float*)q, ld_q, (float*)out, ld_out, (const float*)k_cache, (const float*)v_cache, block_table, \
                      max_blocks, cu_seqlens, seq_lens, num_reqs, max_q, scale, window, G, kv_heads, page_size, stream)
#define DINFER_ATTN_F32_CASE(DT) \
  case 16 * DT:                  \
    if (two) DINFER_ATTN_F32(DT, (DT <= 4 ? 2 : 1)); else DINFER_ATTN_F32(DT, 1); \
    break
  switch (head_dim) {
    DINFER_ATTN_F32_CASE(1);
    DINFER_ATTN_F32_CASE(2);
    DINFER_ATTN_F32_CASE(3);
    DINFER_ATTN_F32_CASE(4);
    DINFER_ATTN_F32_CASE(5);
    DINFER_ATTN_F32_CASE(6);
    DINFER_ATTN_F32_CASE(7);
    DINFER_ATTN_F32_CASE(8);
    DINFER_ATTN_F32_CASE(12);
    DINFER_ATTN_F32_CASE(16);
    default: return ERR_UNSUPPORTED;
  }
#undef DINFER_ATTN_F32_CASE
#undef DINFER_ATTN_F32
  return launch_status();
}
