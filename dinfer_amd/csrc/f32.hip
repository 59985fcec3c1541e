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
// A workgroup of 2 x 2 waves computes BM rows x BN columns; steps of 64 k go through two LDS buffers, the 16-byte loads
// of the two steps after it in flight while one is multiplied (one step ahead, a workgroup a CU waits for memory most of
// the time: 1,024 columns of K = 3,072 at 500 rows 70 us). Rows of LDS are 68 floats apart: the eight lanes that a
// 16-byte read serves at a time lie in different banks. Bound by the matrix cores and, where the columns give a CU one
// workgroup, by a step's latency: 500 rows x 6,144
// x 1,024 in 73 us (86 TFLOP/s where a large library product reaches 153; the vector-ALU kernel 165), x 1,024 x 3,072 in
// 43 (452).
constexpr int KB = 64, LROW = KB + 4;

template <int BM, int BN>
__global__ void __launch_bounds__(256) gemm_f32_kernel(const float* __restrict__ A, int64_t lda, const float* __restrict__ W,
                                                       int64_t ldw, float* __restrict__ C, int64_t ldc, int M, int N, int K) {
  constexpr int MT = BM / 32, NT = BN / 32;                       // tiles of 16 a wave
  constexpr int LA = BM * KB / 4 / 256, LW = BN * KB / 4 / 256;   // 16-byte loads a thread and step
  __shared__ float As[2][BM * LROW];
  __shared__ float Ws[2][BN * LROW];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int lr = lane & 15, lg = lane >> 4;
  const int row = threadIdx.x >> 4, piece = (threadIdx.x & 15) * 4;   // 16 rows of 16 pieces a pass

  const float* pa[LA];
  const float* pw[LW];
#pragma unroll
  for (int e = 0; e < LA; ++e) pa[e] = A + (int64_t)min(m0 + row + 16 * e, M - 1) * lda;
#pragma unroll
  for (int e = 0; e < LW; ++e) pw[e] = W + (int64_t)min(n0 + row + 16 * e, N - 1) * ldw;

  f32x4 ra[2][LA], rw[2][LW];
  auto fetch = [&](int k0, f32x4(&fa)[LA], f32x4(&fw)[LW]) {   // pieces past K are read at K - 4 (and cleared below)
    const int kk = min(k0 + piece, K - 4);
#pragma unroll
    for (int e = 0; e < LA; ++e) fa[e] = *(const f32x4*)(pa[e] + kk);
#pragma unroll
    for (int e = 0; e < LW; ++e) fw[e] = *(const f32x4*)(pw[e] + kk);
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
    for (int e = 0; e < LA; ++e) *(f32x4*)&As[b][(row + 16 * e) * LROW + piece] = fa[e];
#pragma unroll
    for (int e = 0; e < LW; ++e) *(f32x4*)&Ws[b][(row + 16 * e) * LROW + piece] = fw[e];
  };

  f32x4 acc[MT][NT], tot[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = tot[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int steps = (K + KB - 1) / KB;
  fetch(0, ra[0], rw[0]);
  fetch(KB, ra[1], rw[1]);
  put(0, 0, ra[0], rw[0]);
  __syncthreads();
  for (int s0 = 0; s0 < steps; s0 += 2) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int s = s0 + b;
      if (s >= steps) break;
      fetch((s + 2) * KB, ra[b], rw[b]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < KB / 16; ++c) {
        f32x4 fa[MT], fw[NT];
#pragma unroll
        for (int i = 0; i < MT; ++i) fa[i] = *(const f32x4*)&As[b][(wm + 16 * i + lr) * LROW + 16 * c + 4 * lg];
#pragma unroll
        for (int j = 0; j < NT; ++j) fw[j] = *(const f32x4*)&Ws[b][(wn + 16 * j + lr) * LROW + 16 * c + 4 * lg];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[j][q], fa[i][q], acc[i][j], 0, 0, 0);
      }
      if (s + 1 == steps || (s + 1) % (SEG / KB) == 0) {   // a segment is whole
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            tot[i][j] += acc[i][j];
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (s + 1 < steps) put(b ^ 1, (s + 1) * KB, ra[b ^ 1], rw[b ^ 1]);
      __syncthreads();
    }
  }
  // a lane holds four consecutive columns of one row
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + wm + 16 * i + lr;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = n0 + wn + 16 * j + 4 * lg;
      if (m >= M) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) C[(int64_t)m * ldc + n + r] = tot[i][j][r];
    }
  }
}

// ---- products of few rows ---------------------------------------------------------------------------------------
// A workgroup takes 16 rows of the weight and 16 * MT rows of A and streams both straight into registers: its waves deal
// the segments of k among themselves (no barrier inside one), GROUP pieces of 16 k in flight at a time, and after each
// round the parts are added in segment order. Bound by the weight's bytes, and by latency where the weight is small:
// 151,936 x 1,024 in 124 us at one row (5.0 TB/s; the vector-ALU kernel 401), 1,024 x 3,072 in 12 us (365), at 64 rows 32.
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
  const dim3 grid((unsigned)((N + 15) / 16), (unsigned)((M + 16 * MT - 1) / (16 * MT)));
  if (K > 4 * SEG)
    gemm_f32_few_kernel<8, MT><<<grid, 512, 0, stream>>>(a, lda, w, ldw, c, ldc, M, N, K);
  else
    gemm_f32_few_kernel<4, MT><<<grid, 256, 0, stream>>>(a, lda, w, ldw, c, ldc, M, N, K);
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
  auto groups = [&](int64_t bm, int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  const dim3 blocks[] = {dim3((unsigned)((N + 63) / 64), (unsigned)((M + 63) / 64)), dim3((unsigned)((N + 63) / 64), (unsigned)((M + 31) / 32))};
  // Up to 64 rows, and wherever tiles of 32 x 64 would leave CUs without one, the kernel whose waves split k (100 rows x
  // 1,024 x 3,072: 30 us against 70 through LDS in steps of 32); from there the largest tile that gives every CU two
  // workgroups (500 x 4,096 x 1,024: 51 us), or one of half the rows (500 x 1,024 x 3,072: 43 us, 128 tiles of 64 x 64
  // being half the chip).
  if (M <= 16) launch_few<1>(a, lda, w, ldw, c, ldc, m, n, k, stream);
  else if (M <= 32) launch_few<2>(a, lda, w, ldw, c, ldc, m, n, k, stream);
  else if (M <= 64 || groups(32, 64) < 256) launch_few<4>(a, lda, w, ldw, c, ldc, m, n, k, stream);
  else if (groups(64, 64) >= 512) gemm_f32_kernel<64, 64><<<blocks[0], 256, 0, stream>>>(a, lda, w, ldw, c, ldc, m, n, k);
  else gemm_f32_kernel<32, 64><<<blocks[1], 256, 0, stream>>>(a, lda, w, ldw, c, ldc, m, n, k);
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
