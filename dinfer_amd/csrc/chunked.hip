// Recurrences over prompt portions in chunks of 64 tokens, on the 32-bit matrix instruction.
//
//   decay        S <- a_t S + c_t k_t v_t^T;                                   o_t = S^T q_t
//   delta rule   S <- a_t S;   u_t = c_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
//
// a token at a time (decay.hip, delta.hip) a prompt is a serial chain of some 0.25 us a token with vector sums over the
// rows of S at its middle, whatever the rest of the chip does. Within a chunk that starts from the state S0, with
// G_t = a_0 .. a_t and d(t, s) = a_{s+1} .. a_t, both are
//
//   S_t = G_t S0 + sum_{s <= t} d(t, s) k_s u_s^T,    o_t = G_t S0^T q_t + sum_{s <= t} d(t, s) (q_t . k_s) u_s
//
// with u_t = c_t v_t for the decay, and for the delta rule the solution of the lower triangular system
//
//   u_t + sum_{s < t} c_t d(t, s) (k_t . k_s) u_s = x_t = c_t (v_t - G_t S0^T k_t),     u = T x
//
// whose matrix does not need the state. So what multiplies u is multiplied by T beforehand (T^T on the other side), and
// the same scan serves both, with x in the place of u:
//
//   chunk_prep   one workgroup a chunk and head, all chunks of the step at once: products of decays, P = d (q . k); for the
//                delta rule P T and K^T T (triangular systems in blocks of 16: the diagonal blocks inverted by
//                substitution, the rest by matrix instructions). What the scan multiplies with is written in the order
//                of its lanes.
//   chunk_scan   one workgroup a request, head and 16 columns of S, chunk after chunk: x, o and the next S. Of the eight
//                waves the first four make the chunk's x, the others its o, and each keeps 16 rows of S as an accumulator.
//
// A decay d(t, s) is a product, taken factor by factor, never a quotient: decays of zero are as good as any. An infinity or NaN of
// a token reaches that token and what follows it, as token by token: no row before it multiplies it, not by 0 either. Everything
// stays in 32 bits, long sums are trees of short chains: about the error that the trees of lanes of
// the token-by-token kernels leave (x is made from S0 itself, not as a difference of two solutions, for the same reason).
// An accumulator of the 16 x 16 x 4 instruction holds rows 4 g + i (lane l: g = l / 16, column l % 16) in its register i,
// which is what the next product wants of its second operand if step i of a block of 16 contracts over 4 g + i: S and x
// pass from one product to the next as they are, through LDS only to reach the other waves.
// Chunks are cut from the start of the request's rows in the step: a chunk never holds tokens of two requests.
#include "common.cuh"

#include <algorithm>

using namespace dinfer;

namespace {

constexpr int C = 64;             // tokens of a chunk
constexpr int BLOCKS = 10;        // blocks of 16 x 16 on and below the diagonal of a chunk's square
constexpr int SCALARS = 3 * C;    // G_t, d(63, t), c_t

struct Rows {
  const float* q; int64_t ldq;        // [T, G D]
  const float* k; int64_t ldk;        // [T, G D]
  const float* v; int64_t ldv;        // [T, H V]
  const float* decay; int64_t ldd;    // [T, H], or [H] with ldd = 0
  const float* gain; int64_t ldg;     // [T, H] or null
};

// The pieces of the scratch: what the scan reads of a chunk, each 64-lane piece of 16 bytes a lane in one line of 1 KB.
struct Pieces {
  f32x4* q;      // [chunks][G][4][KT][64]        rows of q, 16 tokens x 16 entries
  f32x4* k;      // decay: [chunks][G][KT][4][64] k transposed, 16 entries x 16 tokens; delta rule: rows of k as of q
  f32x4* w;      // delta rule: [chunks][H][KT][4][64]  (K^T with the decays behind every token) T
  f32x4* p;      // [chunks][H][BLOCKS][64]       P, or P T
  float* s;      // [chunks][H][SCALARS]
};

__device__ __forceinline__ int chunks_of(const int32_t* __restrict__ cu, int num_reqs, int min_rows, int b) {
  if (b >= num_reqs) return 0;
  const int n = cu[b + 1] - cu[b];
  return n >= min_rows ? (n + C - 1) / C : 0;
}

__device__ __forceinline__ int inclusive_sum(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(v, o, 64);
    if (lane >= o) v += x;
  }
  return v;
}

// The request that chunk `chunk` belongs to and the chunk's place in it; false if there are not as many.
__device__ __forceinline__ bool find_chunk(const int32_t* __restrict__ cu, int num_reqs, int min_rows, int chunk, int& req,
                                           int& place) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int b0 = 0; b0 < num_reqs; b0 += 64) {
    const int c = chunks_of(cu, num_reqs, min_rows, b0 + lane);
    const int upto = before + inclusive_sum(c, lane);
    const uint64_t beyond = __ballot(upto > chunk);
    if (beyond) {
      const int l = __ffsll((unsigned long long)beyond) - 1;
      req = __builtin_amdgcn_readfirstlane(b0 + l);
      place = __builtin_amdgcn_readfirstlane(chunk - __shfl(upto - c, l, 64));
      return true;
    }
    before = __shfl(upto, 63, 64);
  }
  return false;
}

__device__ __forceinline__ int first_chunk(const int32_t* __restrict__ cu, int num_reqs, int min_rows, int req) {
  const int lane = threadIdx.x & 63;
  int sum = 0;
  for (int b = lane; b < req; b += 64) sum += chunks_of(cu, num_reqs, min_rows, b);
#pragma unroll
  for (int o = 32; o; o >>= 1) sum += __shfl_xor(sum, o, 64);
  return __builtin_amdgcn_readfirstlane(sum);
}

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// A B over 16 N entries: chains of 8 terms and the tree of their sums, which rounds about as often as lanes that add in pairs do
// (one chain over 128 entries: 1.8 times the error, four: 1.3 times)
template <int N, class A, class B>
__device__ __forceinline__ f32x4 mfma_tree(const A& a, const B& b) {
  if constexpr (N == 1) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f}, x = a(0), y = b(0);
    return mfma(x[1], y[1], mfma(x[0], y[0], zero)) + mfma(x[3], y[3], mfma(x[2], y[2], zero));
  } else {
    return mfma_tree<N / 2>(a, b) + mfma_tree<N - N / 2>([&](int i) { return a(i + N / 2); }, [&](int i) { return b(i + N / 2); });
  }
}

__device__ __forceinline__ constexpr int block_of(int i, int j) { return i * (i + 1) / 2 + j; }

// LDS: k and q of the chunk, 16 bytes of padding a row, and the blocks (78 KB at D = 128: two workgroups a CU). 2,048 tokens of
// 16 heads of 128 x 128: 28 us for the delta rule, of which the matrix instructions 14, 24 us for a decay, most of it the
// latencies of a workgroup's one pass (its rows, the blocks' sums, the decays, what it writes).
template <int KT, bool DELTA>
__global__ void __launch_bounds__(256, 2) chunk_prep_kernel(Rows p, Pieces out, const int32_t* __restrict__ cu, int num_reqs,
                                                         int min_rows, int chunk0, int G, int H, int heads) {
  constexpr int D = 16 * KT, LD = D + 4;
  __shared__ __attribute__((aligned(16))) float ks[C][LD];
  __shared__ __attribute__((aligned(16))) float qs[C][LD];
  __shared__ f32x4 blk[BLOCKS][64];    // d(t, s), then P: lane t % 16 + 16 g, s = 4 g + i
  // the system's blocks, lane s % 16 + 16 g, t = 4 g + i: in the place of q, whose rows have been read by then
  f32x4 (*sys)[64] = (f32x4 (*)[64])&qs[0][0];
  static_assert(sizeof(qs) >= sizeof(blk), "the system's blocks fit where q was");
  __shared__ __attribute__((aligned(16))) float ends[C];
  __shared__ int odd[5];               // delta rule: whether the system, or the inverses (4), hold an infinity or NaN
  const int h0 = blockIdx.x * heads, chunk = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  int req, place;
  if (!find_chunk(cu, num_reqs, min_rows, chunk0 + chunk, req, place)) return;
  const int64_t t0 = cu[req] + place * C;
  const int n = min(C, cu[req + 1] - (int)t0);
  const int per = H / G, g = h0 / per;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

  for (int i = tid; i < C * KT * 4; i += 256) {
    const int t = i / (KT * 4), d = i % (KT * 4) * 4;
    f32x4 kv = zero, qv = zero;
    if (t < n) {
      kv = *(const f32x4*)(p.k + (t0 + t) * p.ldk + g * D + d);
      qv = *(const f32x4*)(p.q + (t0 + t) * p.ldq + g * D + d);
    }
    *(f32x4*)&ks[t][d] = kv;
    *(f32x4*)&qs[t][d] = qv;
  }
  __syncthreads();

  // the blocks on and below the diagonal, number wave + 4 x to a wave: k . q, lane t, registers s; k . k, lane s, registers t
  constexpr int MINE = (BLOCKS + 3) / 4;
  f32x4 kq[MINE], kk[DELTA ? MINE : 1];
#pragma unroll
  for (int x = 0; x < MINE; ++x) {
    const int bl = wave + 4 * x;
    if (bl < BLOCKS) {
      const int i = bl >= 6 ? 3 : bl >= 3 ? 2 : bl >= 1 ? 1 : 0, j = bl - block_of(i, 0);
      auto row = [&](float (*m)[LD], int tile) {
        return [=](int kt) { return *(const f32x4*)&m[16 * tile + lr][16 * kt + 4 * lg]; };
      };
      kq[x] = mfma_tree<KT>(row(ks, j), row(qs, i));
      if (DELTA) kk[x] = mfma_tree<KT>(row(ks, i), row(ks, j));
    }
  }
  if (h0 % per == 0) {   // the first head of a group writes what its heads share
    f32x4* qo = out.q + ((int64_t)chunk * G + g) * 4 * KT * 64 + lane;
    f32x4* ko = out.k + ((int64_t)chunk * G + g) * 4 * KT * 64 + lane;
    for (int i = wave; i < 4 * KT; i += 4) {
      qo[i * 64] = *(const f32x4*)&qs[16 * (i / KT) + lr][16 * (i % KT) + 4 * lg];
      f32x4 x;
      if (DELTA) {
        x = *(const f32x4*)&ks[16 * (i / KT) + lr][16 * (i % KT) + 4 * lg];
      } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) x[m] = ks[16 * (i % 4) + 4 * lg + m][16 * (i / 4) + lr];
      }
      ko[i * 64] = x;
    }
  }
  __syncthreads();   // (q has been read)

  for (int h = h0; h < h0 + heads; ++h) {
    const int64_t ch = (int64_t)chunk * H + h;
    float* so = out.s + ch * SCALARS;
    // d(t, s): lane s runs down its column, wave w keeps rows 16 w .. 16 w + 15; lane t holds the decay of token t. The
    // products run in 64 bits: a rounding in one of them would be shared by all that a token adds to a later one
    const float av = lane < n ? p.decay[p.ldd ? (t0 + lane) * p.ldd + h : h] : 1.f;
    const float cv = lane < n ? (p.gain ? p.gain[(t0 + lane) * p.ldg + h] : 1.f) : 0.f;
    if (wave == 0) so[2 * C + lane] = cv;
    {
      double d = 0.0;
      float rows[16];
#pragma unroll
      for (int t = 0; t < C; ++t) {
        if (t < 16 * wave + 16) {
          const float a = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, av), t));
          d = t > lane ? d * a : t == lane ? 1.0 : 0.0;
          rows[t & 15] = (float)d;
        }
      }
      const float a0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, av), 0));
      float* to = (float*)&blk[block_of(wave, lg)][16 * (lr >> 2)] + (lr & 3);
      if (lane < 16 * wave + 16) {
#pragma unroll
        for (int e = 0; e < 16; ++e) to[4 * e] = rows[e];
        if (DELTA) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const f32x4 x = {rows[4 * e], rows[4 * e + 1], rows[4 * e + 2], rows[4 * e + 3]};
            sys[block_of(wave, lg)][lr + 16 * e] = x;
          }
        }
      }
      if (lane == 0) {
#pragma unroll
        for (int e = 0; e < 16; ++e) so[16 * wave + e] = a0 * rows[e];
      }
      if (wave == 3) {
        so[C + lane] = rows[15];
        ends[lane] = rows[15];
      }
    }
    __syncthreads();
    float off = 0.f;   // 0 times every entry of the system
#pragma unroll
    for (int x = 0; x < MINE; ++x) {
      const int bl = wave + 4 * x;
      if (bl < BLOCKS) {
        const int i = bl >= 6 ? 3 : bl >= 3 ? 2 : bl >= 1 ? 1 : 0;
        const bool diagonal = bl == block_of(i, i);
        f32x4 pv = kq[x] * blk[bl][lane];
#pragma unroll
        for (int m = 0; m < 4; ++m) pv[m] = diagonal && 4 * lg + m > lr ? 0.f : pv[m];   // (not 0 times a later token's infinity)
        if (!DELTA) {
          out.p[(ch * BLOCKS + bl) * 64 + lane] = pv;
        } else {
          const f32x4 d = sys[bl][lane];
          f32x4 a;
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            const float c = __shfl(cv, 16 * i + 4 * lg + m, 64);   // (by all lanes)
            a[m] = diagonal && 4 * lg + m <= lr ? 0.f : -c * d[m] * kk[x][m];
            off = __builtin_fmaf(a[m], 0.f, off);
          }
          blk[bl][lane] = pv;
          sys[bl][lane] = a;
        }
      }
    }
    if (DELTA) odd[wave] = __any(off != 0.f);
    __syncthreads();
    if constexpr (DELTA) {
      // the inverses of the four diagonal blocks, less the ones on their diagonals, in their place: a lane a block and column
      if (wave == 0) {
        f32x4* b = sys[block_of(lg, lg)];
        float x[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) x[t] = t == lr ? 1.f : 0.f;
#pragma unroll
        for (int c = 0; c < 15; ++c) {
#pragma unroll
          for (int e = (c + 1) / 4; e < 4; ++e) {
            const f32x4 a = b[c + 16 * e];
#pragma unroll
            for (int m = 0; m < 4; ++m)
              if (4 * e + m > c) x[4 * e + m] = __builtin_fmaf(a[m], x[c], x[4 * e + m]);
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        float off_x = 0.f;
#pragma unroll
        for (int t = 0; t < 16; ++t) off_x = __builtin_fmaf(x[t], 0.f, off_x);
        odd[4] = __any(off_x != 0.f);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f32x4 o;
#pragma unroll
          for (int m = 0; m < 4; ++m) o[m] = 4 * e + m == lr ? 0.f : x[4 * e + m];
          b[lr + 16 * e] = o;
        }
      }
      __syncthreads();
      // From a row that is not finite on everything is not (what a token adds to the state goes into all that follows), but the rows
      // before it must not meet it: as rows of zeros it stays out of their sums. Never taken while a model's numbers are finite.
      int first_bad = C;
      if (odd[0] | odd[1] | odd[2] | odd[3] | odd[4]) {
#pragma unroll 1
        for (int t = C - 1; t >= 0; --t)
          for (int j = 0; j <= t >> 4; ++j)
            if (!(fabsf(((const float*)sys[block_of(t >> 4, j)])[4 * (lr + (t & 12) * 4) + (t & 3)]) < INFINITY)) first_bad = t;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) first_bad = min(first_bad, __shfl_xor(first_bad, o, 64));
        __syncthreads();   // (every wave has counted)
      }
      if (first_bad < C) {
#pragma unroll 1
        for (int bl = wave; bl < BLOCKS; bl += 4) {
          const int t = 16 * (bl >= 6 ? 3 : bl >= 3 ? 2 : bl >= 1 ? 1 : 0) + 4 * lg;
          f32x4 a = sys[bl][lane];
#pragma unroll
          for (int m = 0; m < 4; ++m) a[m] = t + m >= first_bad ? 0.f : a[m];
          sys[bl][lane] = a;
        }
        __syncthreads();
      }
      // T^T times 16 columns: entries of k with the decays behind each token, or rows of P; upwards from the last block
#pragma unroll 1
      for (int ct = wave; ct < KT + 4; ct += 4) {
        f32x4 x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (ct < KT) {
            const f32x4 e = *(const f32x4*)&ends[16 * i + 4 * lg];
#pragma unroll
            for (int m = 0; m < 4; ++m) x[i][m] = e[m] * ks[16 * i + 4 * lg + m][16 * ct + lr];
          } else {
            x[i] = i <= ct - KT ? blk[block_of(ct - KT, 0) + i][lane] : zero;
          }
        }
#pragma unroll
        for (int i = 3; i >= 0; --i) {
          f32x4 y[3] = {zero, zero, zero};
#pragma unroll
          for (int j = i + 1; j < 4; ++j)
            y[j - i - 1] = mfma_tree<1>([&](int) { return sys[block_of(j, i)][lane]; }, [&](int) { return x[j]; });
          x[i] += y[0] + (y[1] + y[2]);
          x[i] += mfma_tree<1>([&](int) { return sys[block_of(i, i)][lane]; }, [&](int) { return x[i]; });
        }
        if (first_bad < C && (ct < KT || 16 * (ct - KT) + lr >= first_bad)) {   // what is added to the state; the later rows of P T
          const float nan = __builtin_nanf("");
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] = f32x4{nan, nan, nan, nan};
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (ct < KT) out.w[((ch * KT + ct) * 4 + i) * 64 + lane] = x[i];
          else if (i <= ct - KT) out.p[(ch * BLOCKS + block_of(ct - KT, 0) + i) * 64 + lane] = x[i];
        }
      }
      __syncthreads();
    }
  }
}

// A block of x that holds infinities or NaNs, for the product with the rows of its own tokens: those become zeros, and the result is
// NaN from their row on in their column (lane: column lane % 16, rows 4 (lane / 16) + m, of x and of the result).
__device__ __forceinline__ f32x4 cut_at_rows(f32x4& x) {
  const int lane = threadIdx.x & 63;
  f32x4 y;
  float sum = 0.f;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    sum += x[m] * 0.f;
    y[m] = sum;
    x[m] = fabsf(x[m]) < INFINITY ? x[m] : 0.f;
  }
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) {
    const float before = __shfl_up(sum, o, 64);
    if (lane >= o) sum += before;
  }
  const float before = __shfl_up(sum, 16, 64);
#pragma unroll
  for (int m = 0; m < 4; ++m) y[m] += lane >= 16 ? before : 0.f;
  return y;
}

// A chunk is two rounds of matrix instructions with a barrier between: with S of the chunk's start (waves 0 to 3: x,
// waves 4 to 7: q S), then with x (o, and S of the chunk's end). Its operands are fetched while the chunk before is worked
// through (delta rule: 256 registers a lane), or each round's while the other runs (decay: 128, two workgroups a CU).
// A prompt of 2,048 tokens, 16 heads of 128 x 128: 99 us for the delta rule (token by token 545), 3.1 us a chunk, of which
// the matrix instructions of a SIMD 1.4 and the two exchanges through LDS most of the rest; its 128 workgroups leave half the
// chip idle (fewer columns than the instruction's 16 would be work for nothing). 4 prompts of 512: decays 42 us (132), 64
// heads of 128 x 64 77 us (235), 40 percent of the time in matrix instructions. Without its loads the kernel takes 10
// percent less, without its stores 4.
template <int KT, bool DELTA>
__global__ void __launch_bounds__(512, DELTA ? 2 : 4) chunk_scan_kernel(Rows p, Pieces in, float* __restrict__ state,
                                                         const int32_t* __restrict__ slots, const int32_t* __restrict__ cu,
                                                         const int32_t* __restrict__ seq_lens, float* __restrict__ out,
                                                         int64_t ld_out, int num_reqs, int min_rows, int chunk0, int chunks,
                                                         int G, int H, int V) {
  constexpr int D = 16 * KT;
  constexpr bool AHEAD = DELTA;
  __shared__ f32x4 s_state[KT][64];
  __shared__ f32x4 s_x[2][4][64];     // x; x times the decay behind it (decay only)
  __shared__ int s_odd[4];            // whether a block of x holds an infinity or NaN: 0 times it is not 0 for the rows before it
  // the head is the fastest index of the grid: the workgroups of a head's columns, which read the same pieces, share an
  // XCD (consecutive workgroups go to consecutive XCDs) where the heads are a multiple of 8
  const int h = blockIdx.x, cb = blockIdx.y, b = blockIdx.z;
  const int r0 = cu[b], rows = cu[b + 1] - r0;
  if (rows < min_rows) return;
  const int first = first_chunk(cu, num_reqs, min_rows, b);
  const int lo = max(first, chunk0), hi = min(first + (rows + C - 1) / C, chunk0 + chunks);
  if (lo >= hi) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int r = wave & 3;
  const bool is_o = wave >= 4, has_s = wave < KT;
  const int g = h / (H / G);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

  float* sp = state + (((int64_t)slots[b] * H + h) * V + 16 * cb + lr) * D + 16 * (has_s ? wave : 0) + 4 * lg;
  f32x4 S = zero;
  if (has_s && (seq_lens[b] > rows || lo > first)) S = *(const f32x4*)sp;

  struct First { f32x4 a[KT], v, c, end, dec; } fa;   // dec: G_t of the rows of x or of o
  struct Second { f32x4 k[4], p[4]; float all; } fb;
  auto fetch_first = [&](int c, First& f) {
    const int64_t cg = (int64_t)(c - chunk0) * G + g, ch = (int64_t)(c - chunk0) * H + h;
    const float* sc = in.s + ch * SCALARS + 16 * r + 4 * lg;
    if (DELTA || is_o) {
      const f32x4* src = (is_o ? in.q : in.k) + (cg * 4 + r) * KT * 64 + lane;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) f.a[kt] = src[kt * 64];
      f.dec = *(const f32x4*)sc;
    }
    if (!is_o) {
      f.c = *(const f32x4*)(sc + 2 * C);
      if (!DELTA) f.end = *(const f32x4*)(sc + C);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int t = (c - first) * C + 16 * r + 4 * lg + m;
        f.v[m] = t < rows ? p.v[(int64_t)(r0 + t) * p.ldv + (int64_t)h * V + 16 * cb + lr] : 0.f;
      }
    }
  };
  auto fetch_second = [&](int c, Second& f) {
    const int64_t cg = (int64_t)(c - chunk0) * G + g, ch = (int64_t)(c - chunk0) * H + h;
    if (has_s) {
      const f32x4* src = (DELTA ? in.w + (ch * KT + wave) * 4 * 64 : in.k + (cg * KT + wave) * 4 * 64) + lane;
#pragma unroll
      for (int st = 0; st < 4; ++st) f.k[st] = src[st * 64];
      f.all = in.s[ch * SCALARS + C - 1];
    }
    if (is_o) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j <= r) f.p[j] = in.p[(ch * BLOCKS + block_of(r, 0) + j) * 64 + lane];
    }
  };
  fetch_first(lo, fa);
  fetch_second(lo, fb);
  for (int c = lo; c < hi; ++c) {
    First na = fa;
    Second nb = fb;
    if (AHEAD && c + 1 < hi) {
      fetch_first(c + 1, na);
      fetch_second(c + 1, nb);
    }
    if (has_s) s_state[wave][lane] = S;
    lds_barrier();
    f32x4 x = zero;
    if (DELTA || is_o) {
      x = mfma_tree<KT>([&](int kt) { return fa.a[kt]; }, [&](int kt) { return s_state[kt][lane]; }) * fa.dec;
    }
    if (!is_o) {
      x = DELTA ? fa.c * (fa.v - x) : fa.c * fa.v;
      s_x[0][r][lane] = x;
      const bool odd = !(fabsf(x[0]) < INFINITY && fabsf(x[1]) < INFINITY && fabsf(x[2]) < INFINITY && fabsf(x[3]) < INFINITY);
      s_odd[r] = __any(odd);
      if (!DELTA) s_x[1][r][lane] = x * fa.end;
    }
    if (!AHEAD && c + 1 < hi) fetch_first(c + 1, fa);
    lds_barrier();
    if (has_s) {
      S = S * fb.all + mfma_tree<4>([&](int st) { return fb.k[st]; }, [&](int st) { return s_x[DELTA ? 0 : 1][st][lane]; });
    }
    if (is_o) {
      f32x4 y = zero;
      f32x4 own = s_x[0][r][lane];
      if (__builtin_amdgcn_readfirstlane(s_odd[r])) y = cut_at_rows(own);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j <= r) y += mfma_tree<1>([&](int) { return fb.p[j]; }, [&](int) { return j < r ? s_x[0][j][lane] : own; });
      x += y;
      const int t = (c - first) * C + 16 * r + 4 * lg;
      float* o = out + (int64_t)(r0 + t) * ld_out + (int64_t)h * V + 16 * cb + lr;
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (t + m < rows) o[m * ld_out] = x[m];
    }
    if (AHEAD) {
      fa = na;
      fb = nb;
    } else if (c + 1 < hi) {
      fetch_second(c + 1, fb);
    }
  }
  if (has_s) *(f32x4*)sp = S;
}

}  // namespace

// Floats of scratch a chunk (of 64 tokens) for these sizes; 0: sizes that the chunked form does not take.
extern "C" int dinfer_chunk_floats(int delta, int G, int H, int D, int V) {
  if ((D != 64 && D != 128) || V <= 0 || V % 16 || V > 1024 || G <= 0 || H <= 0 || H > 4096 || H % G) return 0;
  return 2 * G * C * D + H * ((delta ? C * D : 0) + BLOCKS * 256 + SCALARS);
}

// The requests of min_rows rows or more of a step of `tokens` rows; the others are left alone. scratch: `chunks` times
// dinfer_chunk_floats; a step of more chunks goes through it in turns, with the state carried by `state`.
extern "C" int dinfer_chunked_recurrence(int delta, const float* q, int64_t ldq, const float* k, int64_t ldk, const float* v,
                                         int64_t ldv, const float* decay, int64_t ld_decay, const float* gain,
                                         int64_t ld_gain, float* state, const int32_t* state_slots,
                                         const int32_t* cu_seqlens, const int32_t* seq_lens, float* out, int64_t ld_out,
                                         float* scratch, int chunks, int tokens, int num_reqs, int min_rows, int G, int H,
                                         int D, int V, hipStream_t stream) {
  if (num_reqs <= 0 || tokens <= 0) return OK;
  if (!dinfer_chunk_floats(delta, G, H, D, V)) return ERR_UNSUPPORTED;
  if (chunks <= 0 || min_rows <= 0 || num_reqs > 65535 || !decay || (delta && !gain)) return ERR_BAD_SHAPE;
  if (ldq % 4 || ldk % 4 || ((uintptr_t)q | (uintptr_t)k | (uintptr_t)state | (uintptr_t)scratch) % 16) return ERR_UNSUPPORTED;
  const Rows p{q, ldq, k, ldk, v, ldv, decay, ld_decay, gain, ld_gain};
  const int KT = D / 16;
  Pieces x;
  f32x4* at = (f32x4*)scratch;
  auto take = [&](int64_t pieces) {
    f32x4* a = at;
    at += pieces * 64 * chunks;
    return a;
  };
  x.q = take((int64_t)G * 4 * KT);
  x.k = take((int64_t)G * 4 * KT);
  x.w = delta ? take((int64_t)H * 4 * KT) : nullptr;
  x.p = take((int64_t)H * BLOCKS);
  x.s = (float*)at;
  // no more requests of min_rows rows than this, and no more chunks than with one row in the last chunk of each
  const int64_t long_reqs = std::min<int64_t>(num_reqs, tokens / min_rows);
  const int64_t total = (tokens + (C - 1) * long_reqs) / C;
  // heads of a group share k . q where that leaves the chip filled (two workgroups a CU) all the same
  int heads = delta ? 1 : H / G;
  while (heads > 1 && (heads % 2 || H / heads * std::min<int64_t>(total, chunks) < 512)) heads = heads % 2 ? 1 : heads / 2;
  for (int64_t c0 = 0; c0 < total; c0 += chunks) {
    const int now = (int)std::min<int64_t>(chunks, total - c0);
    const dim3 prep((unsigned)(H / heads), (unsigned)now), scan((unsigned)H, (unsigned)(V / 16), (unsigned)num_reqs);
#define CHUNKED(KT_, DELTA_)                                                                                              \
  do {                                                                                                                    \
    chunk_prep_kernel<KT_, DELTA_><<<prep, 256, 0, stream>>>(p, x, cu_seqlens, num_reqs, min_rows, (int)c0, G, H, heads); \
    chunk_scan_kernel<KT_, DELTA_><<<scan, 512, 0, stream>>>(p, x, state, state_slots, cu_seqlens, seq_lens, out, ld_out,  \
                                                             num_reqs, min_rows, (int)c0, now, G, H, V);                  \
  } while (0)
    if (delta && KT == 8) CHUNKED(8, true);
    else if (delta) CHUNKED(4, true);
    else if (KT == 8) CHUNKED(8, false);
    else CHUNKED(4, false);
#undef CHUNKED
  }
  return launch_status();
}
