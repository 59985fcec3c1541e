// C = A . W^T for many rows (prompt portions, full batches), bf16 operands, float accumulation, with what follows the product in
// its end:
//
//   plain   C = act(A W^T), act nothing, silu, the square of relu or gelu (error function)
//   add     C += A W^T, the sum of the float accumulators and C rounded once
//   gated   W = [gate; up] stacked [2N, K], C = silu(A gate^T) * (A up^T)
//   floats  C = A W^T in float (logits)
//
// A workgroup of eight waves computes a tile of C with both operands brought from memory straight into LDS, 64 k a step (rows of
// 128 bytes: eight rows an instruction, whole lines), a wave RM x RN blocks of 16 x 16 in v_mfma_f32_16x16x32_bf16, the weight as its
// first operand, so that a lane ends up with consecutive columns of one row. A row's eight pieces of 16 bytes are exchanged by bits
// 1..3 of its number, so that the 16 lanes that LDS serves at once find all its banks (no conflicts). The rows of the weight are
// put down in the order in which two blocks side by side give a lane eight consecutive columns; gated, a gate block beside its up block.
//
// What bounds it: a CU has at most 256 lines of 128 bytes on their way (measured: 32 KB in flight give 53 GB/s a CU from HBM,
// 100 from the memory-side cache, 140 from L2, and more of them give no more), and the CUs of an XCD ask for the same lines at about the same time,
// so all of them wait as long as the first. So the rate is that of a tile's bytes, (rows + columns) * 128 a step at 45 to 75 GB/s a
// CU, beside MFMAs that alone reach 1.6 PFLOP/s in this loop: large tiles where there are enough of them, else tiles that come out as
// one round of workgroups. (Lines brought into L2 ahead of their use, by touches of a ninth wave or by scalar loads: 10 to 50 %
// slower. Loads into registers have the same limit.)
//
// Against the library's measured choice (with an activation: and its kernel), in trains of launches with copies of the weight in turn, us:
//   gated  1,152 x 3,072 x 1,024    26    20      relu^2  4,096 x 8,192 x 2,048   124   116
//          2,048 x 8,192 x 2,048   120   110              2,048 x 8,192 x 2,048    66    61
//          2,048 x 12,288 x 4,096  306   299      and without an activation
//          4,096 x 2,816 x 2,048    98    87        543 x 7,168 x 5,120            56    53
//          544 x 17,408 x 5,120    200   189        1,033 x 4,096 x 1,024          17    16
// Without an end that is a pass of its own the library is level or ahead in most steps (2,048 x 4,096 x 12,288 169 and 171, 2,023 x 7,168 x 2,048
// 49 and 57, 4,096 x 2,048 x 8,192 112 and 121, 1,033 x 1,024 x 3,072 18.5 and 19.8, 543 x 5,120 x 17,408 128 and 132). Logits of 64 rows, floats:
// 151,936 x 4,096 250 and 230, 32,768 x 2,048 35 and 30.
// Which of them runs a shape is measured where the library's own kernels are (blaslt.py).
//
// Reference behaviour: crates/kernels/src/gemm.rs:605-647 (the product; the reference hands it to its vendor library),
// crates/kernels/cuda/activation.cu:8-16 (the gated activation).
#include <algorithm>
#include <type_traits>

#include "lds_loads.cuh"

using namespace dinfer;

namespace {

enum : int { PLAIN = 0, ADD = 1, GATED = 2, FLOATS = 3 };

struct Product {
  const char* A; int64_t lda;
  const char* W; int64_t ldw;
  void* C; int64_t ldc;
  int M, N, K;
  int row_tiles, col_tiles;
  int act;   // PLAIN: 0 nothing, 1 silu, 2 the square of relu, 3 gelu
};

__device__ __forceinline__ float silu(float x) { return x / (1.f + expf(-x)); }
__device__ __forceinline__ float activated(float x, int act) {
  if (act == 1) return silu(x);
  if (act == 2) return x > 0.f ? x * x : 0.f;
  if (act == 3) return 0.5f * x * (1.f + erff(x * 0.7071067811865476f));
  return x;
}

// This wave's loads into LDS but the last N are here, its reads of LDS are done, and every wave's with it.
template <int N>
__device__ __forceinline__ void step_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Where a tile lies. Tiles are numbered down the rows first; an XCD (workgroup id modulo 8) has a run of them, so that it reads few columns'
// weights and few XCDs read the same ones.
struct Walk {
  int at, end, stride;
  __device__ __forceinline__ Walk(const Product& p) {
    const int64_t tiles = (int64_t)p.row_tiles * p.col_tiles;
    const int xcd = blockIdx.x & 7;
    at = (int)(tiles * xcd / 8) + (int)(blockIdx.x >> 3);
    end = (int)(tiles * (xcd + 1) / 8);
    stride = gridDim.x >> 3;
  }
};

// The byte offset in A of what this lane brings of instruction g (rows 8 g .. 8 g + 7 of the tile; past the last row that one again).
__device__ __forceinline__ uint32_t a_offset(const Product& p, int m0, int g, int lane) {
  const int r = g * 8 + (lane >> 3);
  return (uint32_t)(min(m0 + r, p.M - 1) * (p.lda * 2)) + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
}
// The same of W: place r of LDS holds column c0 + column(r).
template <int RN, int MODE>
__device__ __forceinline__ uint32_t w_offset(const Product& p, int c0, int g, int lane) {
  const int r = g * 8 + (lane >> 3), i = r & 15;
  int n;
  if constexpr (MODE == GATED) {
    static_assert(RN % 4 == 0 || RN == 2, "gate blocks beside their up blocks");
    if constexpr (RN % 4 == 0)   // two blocks of the gate, two of the up projection: 32 columns
      n = min(c0 + (r >> 6) * 32 + 8 * (i >> 2) + 4 * ((r >> 4) & 1) + (i & 3), p.N - 1) + ((r >> 5) & 1) * p.N;
    else
      n = min(c0 + (r >> 5) * 16 + i, p.N - 1) + ((r >> 4) & 1) * p.N;
  } else {
    const int w = r % (RN * 16);   // of the wave's columns; blocks two by two, an odd last one as it is
    n = RN % 2 == 1 && (w >> 4) == RN - 1 ? r : (r - w) + (w & ~31) + 8 * (i >> 2) + 4 * ((w >> 4) & 1) + (i & 3);
    n = min(c0 + n, p.N - 1);
  }
  return (uint32_t)(n * (p.ldw * 2)) + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
}

// A wave's blocks: rows m0 + 16 r + lane % 16, columns from c0 on (N % 8 == 0: a piece of eight is inside or outside).
template <int RM, int RN, int MODE>
__device__ __forceinline__ void store_blocks(const Product& p, int m0, int c0, const f32x4 (&acc)[RM][RN]) {
  const int lane = threadIdx.x & 63, i16 = lane & 15, q4 = lane >> 4;
#pragma unroll
  for (int r = 0; r < RM; ++r) {
    const int m = m0 + r * 16 + i16;
    if (m >= p.M) continue;
    bf16* const row = (bf16*)p.C + (int64_t)m * p.ldc;
    if constexpr (MODE == FLOATS) {
      float* const c = (float*)p.C + (int64_t)m * p.ldc;
#pragma unroll
      for (int j = 0; j < RN; ++j) {   // (two blocks side by side: the lane's first and last four of eight)
        const int n = c0 + ((j | 1) < RN ? (j & ~1) * 16 + 8 * q4 + 4 * (j & 1) : j * 16 + 4 * q4);
        if (n < p.N) *(f32x4*)(c + n) = acc[r][j];
      }
    } else if constexpr (MODE == GATED && RN % 4 == 0) {
#pragma unroll
      for (int j = 0; j < RN; j += 4) {
        const int n = c0 + j * 8 + 8 * q4;
        bf16x8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (bf16)(silu(acc[r][j + (e >> 2)][e & 3]) * acc[r][j + 2 + (e >> 2)][e & 3]);
        if (n < p.N) *(bf16x8*)(row + n) = v;
      }
    } else if constexpr (MODE == GATED) {
      const int n = c0 + 4 * q4;
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (bf16)(silu(acc[r][0][e]) * acc[r][1][e]);
      if (n < p.N) *(bf16x4*)(row + n) = v;
    } else {
#pragma unroll
      for (int j = 0; j < RN; j += 2) {
        if (j + 1 < RN) {
          const int n = c0 + j * 16 + 8 * q4;
          if (n >= p.N) continue;
          bf16x8 v;
          if constexpr (MODE == ADD) v = *(const bf16x8*)(row + n);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float x = acc[r][j + (e >> 2)][e & 3];
            v[e] = (bf16)(MODE == ADD ? x + (float)v[e] : activated(x, p.act));
          }
          *(bf16x8*)(row + n) = v;
        } else {
          const int n = c0 + j * 16 + 4 * q4;
          if (n >= p.N) continue;
          bf16x4 v;
          if constexpr (MODE == ADD) v = *(const bf16x4*)(row + n);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = acc[r][j][e];
            v[e] = (bf16)(MODE == ADD ? x + (float)v[e] : activated(x, p.act));
          }
          *(bf16x4*)(row + n) = v;
        }
      }
    }
  }
}

// Tiles of 96 x 64, 64 to 224 x 128, 96 x 192, 64 x 320 and 128 x 256 (two sets of fragments and the sums in 256 registers), waves 2 x 4, NS stages of both operands.
// A step's first half computes on fragments read beside the MFMAs before, while the second half's are read; behind the barrier between
// the halves every wave has all of the step in registers, so its place is sent anew, NS steps ahead, and the next step is here to be read.
// The last NS steps of a tile send the first stages of the workgroup's next one (behind its last tile its own again, for nobody), whose
// fragments are in registers when it begins; a tile's results leave beside the next one's first steps.
template <int RM, int RN, int NS, int MODE>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) gemm_tile_kernel(Product p) {
  constexpr int BM = 32 * RM, BN = 64 * RN, COLS = MODE == GATED ? BN / 2 : BN;
  constexpr int INSTR = (BM + BN) / 8, L = (INSTR + 7) / 8, FULL = INSTR - (L - 1) * 8;   // instructions of a stage, of a wave; waves with L
  constexpr int STAGE = (BM + BN) * 128;
  extern __shared__ __attribute__((aligned(1024))) char tile_smem[];
  Walk walk(p);
  if (walk.at >= walk.end) return;   // (the whole workgroup)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, i16 = lane & 15, q4 = lane >> 4;
  const int wm = wave >> 2, wn = wave & 3, steps = p.K / 64;
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)tile_smem;
  const bool many = wave < FULL;
  const uint32_t piece = (uint32_t)((q4 ^ ((i16 >> 1) & 7)) * 16);   // of the first 32 k; of the others 64 bytes over or back
  const uint32_t fa_at = (uint32_t)((wm * RM * 16 + i16) * 128) + piece, fw_at = (uint32_t)((BM + wn * RN * 16 + i16) * 128) + piece;
  uint32_t off[L];
  const char* base[L];
  int k_at = 0;   // bytes along the rows
  // One tile of rows: the weights stream past it, every tile from a step of its own on. Workgroups that all stood at the same k would ask
  // the same few memory channels where a row is a power of two long (64 x 32,768 x 2,048 33 -> 29 us, 64 x 24,576 x 4,096 46 -> 40).
  auto sources = [&](int t) __attribute__((always_inline)) {
    k_at = p.row_tiles == 1 ? t % steps * 128 : 0;
#pragma unroll
    for (int x = 0; x < L; ++x) {
      const int g = wave + x * 8;
      const bool a = g < BM / 8;
      off[x] = a ? a_offset(p, t % p.row_tiles * BM, g, lane) : w_offset<RN, MODE>(p, t / p.row_tiles * COLS, g - BM / 8, lane);
      base[x] = a ? p.A : p.W;
    }
  };
  auto send = [&](uint32_t stage, int x) __attribute__((always_inline)) {
    if (x < L - 1 || many) load_to_lds(lds + stage + (uint32_t)(wave + x * 8) * 1024u, off[x], base[x] + k_at);
    if (x == L - 1) k_at = k_at + 128 == steps * 128 ? 0 : k_at + 128;
  };
  bf16x8 fa[2][RM], fw[2][RN];
  auto frag = [&](uint32_t stage, int b, int x) __attribute__((always_inline)) {
    if (x < RN) fw[b][x] = *(const bf16x8*)(tile_smem + stage + (fw_at ^ (b * 64)) + x * 2048);
    else fa[b][x - RN] = *(const bf16x8*)(tile_smem + stage + (fa_at ^ (b * 64)) + (x - RN) * 2048);
  };
  sources(walk.at);
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int x = 0; x < L; ++x) send(s * STAGE, x);
  if (many) step_barrier<(NS - 1) * L>(); else step_barrier<(NS - 1) * (L - 1)>();
#pragma unroll
  for (int x = 0; x < RN + RM; ++x) frag(0, 0, x);
  uint32_t to = 0;   // the step's stage
  for (;;) {
    const int t = walk.at;
    const bool last = t + walk.stride >= walk.end;
    f32x4 acc[RM][RN];
#pragma unroll
    for (int r = 0; r < RM; ++r)
#pragma unroll
      for (int j = 0; j < RN; ++j) acc[r][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int MFMAS = RM * RN, FRAGS = RM + RN;
#pragma nounroll
    for (int s = 0; s < steps; ++s) {
      if (s == steps - NS) sources(last ? t : t + walk.stride);
      const uint32_t ahead = to + STAGE == NS * STAGE ? 0 : to + STAGE;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int x = 0; x < MFMAS; ++x) {
          acc[x / RN][x % RN] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[b][x % RN], fa[b][x / RN], acc[x / RN][x % RN], 0, 0, 0);
          // the other set's fragments beside the first three quarters of the MFMAs, the sends over all of them
#pragma unroll
          for (int y = x * FRAGS * 4 / (MFMAS * 3); y < (x + 1) * FRAGS * 4 / (MFMAS * 3) && y < FRAGS; ++y) frag(b ? ahead : to, b ^ 1, y);
          if (b == 1) {
#pragma unroll
            for (int y = x * L / MFMAS; y < (x + 1) * L / MFMAS; ++y) send(to, y);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if (b == 0) {
          if (many) step_barrier<(NS - 2) * L>(); else step_barrier<(NS - 2) * (L - 1)>();
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      to = ahead;
    }
    store_blocks<RM, RN, MODE>(p, t % p.row_tiles * BM + wm * RM * 16, t / p.row_tiles * COLS + wn * (COLS / 4), acc);
    if (last) break;
    walk.at += walk.stride;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing on its way into LDS
}

// Tiles of 256 x 128, 192 x 256, 256 x 192 and 256 x 256: registers hold one set of a wave's row fragments, each read anew as soon as its MFMAs
// are issued, and LDS NA steps of A's rows and one more of the weight's, which come from HBM where A's, just written, are nearer: sent NA and
// NA + 1 steps ahead (the other way round 2,048 x 12,288 x 4,096, gated, 296 us for 286, 543 x 17,408 x 5,120 222 for 182). The barrier of
// a step comes behind the first rows of its second half, whose MFMAs cover the last reads.
template <int RM, int RN, int NA, int MODE>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) gemm_tile_large_kernel(Product p) {
  constexpr int BM = 32 * RM, BN = 64 * RN, COLS = MODE == GATED ? BN / 2 : BN;
  constexpr int LA = BM / 64, LW = BN / 64, L = LA + LW;   // instructions of a wave
  constexpr int NW = NA + 1, SA = BM * 128, SW = BN * 128, FIRST = 2;
  static_assert(BM % 64 == 0 && NA >= 2, "whole instructions of every wave");
  extern __shared__ __attribute__((aligned(1024))) char tile_smem[];
  Walk walk(p);
  if (walk.at >= walk.end) return;   // (the whole workgroup)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, i16 = lane & 15, q4 = lane >> 4;
  const int wm = wave >> 2, wn = wave & 3, steps = p.K / 64;
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)tile_smem;
  const uint32_t piece = (uint32_t)((q4 ^ ((i16 >> 1) & 7)) * 16);
  const uint32_t fa_at = (uint32_t)((wm * RM * 16 + i16) * 128) + piece, fw_at = (uint32_t)(NA * SA + (wn * RN * 16 + i16) * 128) + piece;
  uint32_t off_a[LA], off_w[LW];
  const char *base_a, *base_w;
  auto sources_a = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < LA; ++x) off_a[x] = a_offset(p, t % p.row_tiles * BM, wave + x * 8, lane);
    base_a = p.A;
  };
  auto sources_w = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < LW; ++x) off_w[x] = w_offset<RN, MODE>(p, t / p.row_tiles * COLS, wave + x * 8, lane);
    base_w = p.W;
  };
  uint32_t to_a = 0, to_w = 0, from_a = 0, from_w = 0;   // places sent to and read from next
  auto send_a = [&](int x) __attribute__((always_inline)) {
    load_to_lds(lds + to_a + (uint32_t)(wave + x * 8) * 1024u, off_a[x], base_a);
    if (x == LA - 1) { base_a += 128; to_a = to_a + SA == NA * SA ? 0 : to_a + SA; }
  };
  auto send_w = [&](int x) __attribute__((always_inline)) {
    load_to_lds(lds + NA * SA + to_w + (uint32_t)(wave + x * 8) * 1024u, off_w[x], base_w);
    if (x == LW - 1) { base_w += 128; to_w = to_w + SW == NW * SW ? 0 : to_w + SW; }
  };
  bf16x8 fa[RM], fw[2][RN];
  auto read_a = [&](int b, int x) __attribute__((always_inline)) { fa[x] = *(const bf16x8*)(tile_smem + from_a + (fa_at ^ (b * 64)) + x * 2048); };
  auto read_w = [&](int b, int x) __attribute__((always_inline)) { fw[b][x] = *(const bf16x8*)(tile_smem + from_w + (fw_at ^ (b * 64)) + x * 2048); };
  sources_a(walk.at);
  sources_w(walk.at);
#pragma unroll
  for (int i = -NW; i < 0; ++i) {
#pragma unroll
    for (int x = 0; x < LA; ++x)
      if (i + NA >= 0) send_a(x);
#pragma unroll
    for (int x = 0; x < LW; ++x) send_w(x);
  }
  step_barrier<LW + (NA - 1) * L>();
#pragma unroll
  for (int x = 0; x < RN; ++x) read_w(0, x);
#pragma unroll
  for (int x = 0; x < RM; ++x) read_a(0, x);
  for (;;) {
    const int t = walk.at;
    const bool last = t + walk.stride >= walk.end;
    f32x4 acc[RM][RN];
#pragma unroll
    for (int r = 0; r < RM; ++r)
#pragma unroll
      for (int j = 0; j < RN; ++j) acc[r][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma nounroll
    for (int s = 0; s < steps; ++s) {
      if (s == steps - NA) sources_a(last ? t : t + walk.stride);
      if (s == steps - NW) sources_w(last ? t : t + walk.stride);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < RM; ++r) {
#pragma unroll
        for (int j = 0; j < RN; ++j) {
          acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[0][j], fa[r], acc[r][j], 0, 0, 0);
          if (r == 0) read_w(1, j);
          __builtin_amdgcn_sched_barrier(0);
        }
        read_a(1, r);
        __builtin_amdgcn_sched_barrier(0);
      }
      from_a = from_a + SA == NA * SA ? 0 : from_a + SA;
      from_w = from_w + SW == NW * SW ? 0 : from_w + SW;
      constexpr int MFMAS = (RM - FIRST) * RN;   // behind the barrier
#pragma unroll
      for (int r = 0; r < RM; ++r) {
        if (r == FIRST) {
          step_barrier<LW + (NA - 2) * L>();   // (on their way: the weight's rows behind A's of the next step, and the steps after it)
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int x = 0; x < FIRST; ++x) read_a(0, x);
        }
#pragma unroll
        for (int j = 0; j < RN; ++j) {
          acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[1][j], fa[r], acc[r][j], 0, 0, 0);
          if (r == FIRST) read_w(0, j);
          if (r >= FIRST) {
            const int x = (r - FIRST) * RN + j;
#pragma unroll
            for (int y = x * L / MFMAS; y < (x + 1) * L / MFMAS; ++y) {
              if (y < LA) send_a(y); else send_w(y - LA);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if (r >= FIRST) read_a(0, r);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    store_blocks<RM, RN, MODE>(p, t % p.row_tiles * BM + wm * RM * 16, t / p.row_tiles * COLS + wn * (COLS / 4), acc);
    if (last) break;
    walk.at += walk.stride;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing on its way into LDS
}

// The shapes of tiles: a wave's blocks, the steps of A and of the weight in LDS (not as many of both: the large kernel).
struct Shape {
  int RM, RN, NA, NW;
  constexpr int rows() const { return 32 * RM; }
  constexpr int cols() const { return 64 * RN; }   // (gated: of both halves together)
  constexpr int lds() const { return (NA * rows() + NW * cols()) * 128; }
};
constexpr Shape SHAPES[] = {{2, 2, 6, 6}, {2, 5, 3, 3}, {3, 1, 6, 6}, {3, 2, 5, 5}, {4, 2, 4, 4}, {5, 2, 4, 4}, {7, 2, 3, 3}, {3, 3, 4, 4},
                            {4, 4, 3, 3}, {8, 2, 3, 4}, {6, 4, 2, 3}, {8, 3, 2, 3}, {8, 4, 2, 3}};
constexpr int NUM_SHAPES = sizeof(SHAPES) / sizeof(SHAPES[0]);
constexpr bool takes_gated(const Shape& s) { return s.RN == 2 || s.RN == 4; }

template <int S, int MODE>
int launch(Product p, hipStream_t stream) {
  constexpr Shape s = SHAPES[S];
  static_assert(s.lds() <= 160 * 1024, "LDS");
  constexpr int cols = MODE == GATED ? s.cols() / 2 : s.cols();
  p.row_tiles = (p.M + s.rows() - 1) / s.rows();
  p.col_tiles = (p.N + cols - 1) / cols;
  const int64_t tiles = (int64_t)p.row_tiles * p.col_tiles;
  if (tiles > 0x7fffffff / 8) return ERR_UNSUPPORTED;
  void (*kernel)(Product);
  if constexpr (s.NW > s.NA) kernel = gemm_tile_large_kernel<s.RM, s.RN, s.NA, MODE>;
  else kernel = gemm_tile_kernel<s.RM, s.RN, s.NA, MODE>;
  if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, s.lds()) != hipSuccess) return ERR_LAUNCH;
  const int64_t places = std::min<int64_t>((tiles + 7) / 8, std::max(1, compute_units() / 8));   // of an XCD
  kernel<<<(unsigned)(places * 8), 512, s.lds(), stream>>>(p);
  return launch_status();
}

template <int S>
int launch_mode(const Product& p, int mode, hipStream_t stream) {
  if (mode == PLAIN) return launch<S, PLAIN>(p, stream);
  if (mode == ADD) return launch<S, ADD>(p, stream);
  if (mode == FLOATS) return launch<S, FLOATS>(p, stream);
  if constexpr (takes_gated(SHAPES[S])) return launch<S, GATED>(p, stream);
  return ERR_UNSUPPORTED;
}

template <int S = 0>
int dispatch(int shape, const Product& p, int mode, hipStream_t stream) {
  if constexpr (S < NUM_SHAPES) return shape == S ? launch_mode<S>(p, mode, stream) : dispatch<S + 1>(shape, p, mode, stream);
  return ERR_UNSUPPORTED;
}

}  // namespace

// The number of shapes of tiles.
extern "C" int dinfer_gemm_tile_shapes() { return NUM_SHAPES; }

// Shape `shape`: out[0] rows, out[1] columns (gated: of both halves together), out[2] the least K, out[3] whether it takes gated products.
extern "C" int dinfer_gemm_tile_shape(int shape, int64_t* out) {
  if (shape < 0 || shape >= NUM_SHAPES) return ERR_BAD_SHAPE;
  const Shape s = SHAPES[shape];
  out[0] = s.rows();
  out[1] = s.cols();
  out[2] = s.NW * 64;
  out[3] = takes_gated(s);
  return OK;
}

// C[M,N] = act(A . W^T) (mode 0; act 0 nothing, 1 silu, 2 the square of relu, 3 gelu), C += A . W^T (1), or with W = [gate; up]
// [2N, K] C = silu(A . gate^T) * (A . up^T) (2), or C float = A . W^T (3), in tiles of `shape`. bf16; K a multiple of 64, N of 8, rows on 16 bytes, either operand
// within 4 GB. A and W must not overlap C.
extern "C" int dinfer_gemm_tile(int shape, int mode, int act, const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
                                int64_t M, int64_t N, int64_t K, hipStream_t stream) {
  if (M <= 0 || N <= 0) return OK;
  if (shape < 0 || shape >= NUM_SHAPES || mode < PLAIN || mode > FLOATS || act < 0 || act > 3 || (act && mode != PLAIN)) return ERR_UNSUPPORTED;
  if (K % 64 || K < SHAPES[shape].NW * 64 || N % 8 || M > 0x7fffffff / 2 || N > 0x7fffffff / 4 || K > 0x7fffffff) return ERR_UNSUPPORTED;
  auto off = [](const void* q) { return (uintptr_t)q % 16 != 0; };
  if (lda < K || ldw < K || ldc < N || lda % 8 || ldw % 8 || ldc % 8 || off(A) || off(W) || off(C)) return ERR_BAD_SHAPE;
  const int64_t w_rows = mode == GATED ? 2 * N : N, limit = ((int64_t)1 << 32) / 2;   // offsets in bytes, 32 bits
  if (lda > limit / M || ldw > limit / w_rows) return ERR_UNSUPPORTED;
  const Product p{(const char*)A, lda, (const char*)W, ldw, C, ldc, (int)M, (int)N, (int)K, 0, 0, act};
  return dispatch(shape, p, mode, stream);
}
