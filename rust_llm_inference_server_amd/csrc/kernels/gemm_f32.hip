// The 32-bit product y = x * W^T, all operands float32 (weights (out, in) row-major, as the
// reference's Linear holds them: crates/model/src/layers.rs:17-19, 65-69, 82), on the matrix
// cores' 32-bit form (v_mfma_f32_16x16x4_f32: float32 operands, float32 fused multiply-adds; no
// operand is cut).  K a multiple of 4, rows on 16-byte boundaries; other sizes and dtype mixes
// take gemm_plain.
//
// One arithmetic for any number of rows.  k is cut into at most sixteen runs of equal length
// (a multiple of 16, from K alone: f32_run).  Inside a run the sum grows in steps of 16 k, four
// instructions a step, instruction i multiplying k = 16 j + 4 g + i of the four lane groups g.
// The sums of four runs in a row are added in ascending order to a part, the parts likewise to
// the result.  All kernels below do exactly that, so a row's result does not depend on how many
// rows share the call, nor on the kernel or tile that takes it.
//
//  * gemm_f32_ring: up to 16 rows over K in whole 1024s, bound by reading W once.  W and x come
//    into LDS by direct loads that leave a wave 16 KB ahead of its products, with no registers held
//    for them and whole lines (256 bytes of a row) per load.  At 4 rows, weights cold (MI355X, us,
//    stream kernel -> this): 3072 x 2048 10.8 -> 8.3, 2048 x 2048 10.2 -> 7.4, 16384 x 2048 30.2 ->
//    25.4 (5.3 TB/s), 2048 x 8192 30 -> 18, 128256 x 2048 182 -> 171 (6.2 TB/s), 4096 x 14336 39
//    (6.0 TB/s); at 16 rows 2048 x 8192 37 -> 21.
//  * gemm_f32_stream: other K, 17 to 32 rows, and 5 to 16 over short runs and many tiles (see the
//    dispatch).  A workgroup takes 16 weight rows
//    at a time, one wave per run of k, so a wave's loads of a tile are all in flight at once
//    (8 KB) and the next tile's are asked for before this one's products; runs of up to 128 k
//    keep x in registers over all tiles.  The waves' sums meet in LDS.  At 32 rows of the 1B
//    shape, weights cold: q/k/v 16, output 16, gate/up 38, head 242, down 58 us: there, and
//    wherever the long form runs, x is loaded as often as W, and a load of either takes its
//    compute unit about 24 ns (56 clocks, sixteen row pieces of 64 bytes), which bounds it.
//  * gemm_f32_tiles: more rows, bound by the matrix cores (154 TFLOP/s for a large library
//    product here).  Tiles of 16 to 80 rows of x, by what comes out even over the compute units.  384
//    rows of the 1B shape, us, tiles of 64 x 64 or 64 x 32 with both operands through LDS -> this:
//    q/k/v 68 -> 50 (98 TFLOP/s), output 45 -> 32 (100), gate/up 225 -> 214 (120), down 162 -> 112 (115).
//
// Gated (gate and up rows side by side in a tile, SwiGLU behind the sums): the same bits as the product
// and the SwiGLU kernel, without the intermediate.  16384 x 2048 at 4 / 16 / 32 / 64 / 384 rows, us, product and
// SwiGLU kernel -> gated: 27.7 -> 26.2, 30.9 -> 29.2, 39.1 -> 38.6, 48.1 -> 45.5, 221 -> 215.
// The sums in parts also halve the error and more: 2.1e-7 of the result's norm against 64 bits at
// K = 2048 (gemm_plain 8.1e-7), 4.1e-7 at 8192 (1.6e-6).
#include "common.h"
#include "gemm_stream.h"

#include <algorithm>

namespace {

constexpr int kMaxRuns = 16, kPartRuns = 4;

// Length of the runs that a sum over K is made of; ceil(K / length) runs.
__host__ __device__ inline int f32_run(int K) {
  return ((K + kMaxRuns - 1) / kMaxRuns + 15) / 16 * 16;
}

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The four float32 at p[k .. k + 3]; CUT: zeros from `end` on (end a multiple of 4).  The load
// itself always reads inside the row.  The forms without CUT carry no select: the compiler
// moves selects in front of later loads, which then leave only when the earlier ones are back.
template <bool CUT>
__device__ __forceinline__ f32x4 load4(const float* __restrict__ p, int k, int end) {
  const f32x4 v = *(const f32x4*)(p + min(k, end - 4));
  if (!CUT) return v;
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
  return k < end ? v : z;
}

// silu(gate) * up in float32's own exponential and division, as the SwiGLU kernel has it.
__device__ __forceinline__ float silu_times(float gate, float up) {
  const float s = gate / (1.0f + expf(-gate));
  return s * up;
}

// ------------------------------------------------------------------ up to 32 rows
// What a call computes: Y (T, N) = X W^T, or gated, with W (2 N, K) gate rows then up rows, Y =
// silu(gate) * up.
struct F32Args {
  const float* X;
  const float* W;
  float* Y;
  int T, N, K, run;
  long long ldx, ldw, ldy;
  int vec;                     // rows of Y lie on 16-byte boundaries
};

// The weight row that lane r of a tile's products holds; rows: weight rows of a tile (lanes beyond
// hold a row twice), gated 8 gate rows and the 8 up rows of the same columns.
template <bool GATED>
__device__ __forceinline__ int weight_row(int tile, int r, int rows, int N) {
  if (GATED) return min(tile * 8 + r % 8, N - 1) + (r < 8 ? 0 : N);
  return min(tile * rows + (r < rows ? r : r - rows), N - 1);
}

// Columns n .. n + 3 of a token's row.
__device__ __forceinline__ void store_four(const F32Args& a, f32x4 s, int token, int n) {
  float* y = a.Y + token * a.ldy + n;
  if (a.vec && n + 4 <= a.N) {
    *(f32x4*)y = s;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < a.N) y[i] = s[i];
  }
}

// The gated results of a wave's 16 weight rows, columns n0 .. n0 + 7 of a lane's token.  Lanes below 32
// hold the gates of four columns, lane + 32 the ups of the same: the lower takes the first two columns,
// the upper the last two (half of the exponentials each).
__device__ __forceinline__ void store_gated(const F32Args& a, f32x4 s, int token, int n0) {
  const int lane = threadIdx.x % 64, g = lane / 16;
  float o[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float other = __shfl_xor(lane < 32 ? s[2 + i] : s[i], 32, 64);
    o[i] = silu_times(lane < 32 ? s[i] : other, lane < 32 ? other : s[2 + i]);
  }
  const int n = n0 + (g & 1) * 4 + (g >> 1) * 2;
  if (token >= a.T) return;
  float* y = a.Y + token * a.ldy + n;
  if (n < a.N) y[0] = o[0];
  if (n + 1 < a.N) y[1] = o[1];
}

// The sum of a tile's runs, which lie in LDS as [run][group of rows][lane], for rows t * 16 .. + 15
// of x: stored by one wave.
template <int TG, bool GATED>
__device__ __forceinline__ void store_tile(const F32Args& a, const float* red, int runs, int t,
                                           int tile, int rows) {
  const int lane = threadIdx.x % 64, r = lane % 16, g = lane / 16;
  f32x4 s;
  for (int q0 = 0; q0 < runs; q0 += kPartRuns) {
    f32x4 v[kPartRuns];
#pragma unroll
    for (int q = 0; q < kPartRuns; ++q)
      v[q] = *(const f32x4*)(red + (min(q0 + q, runs - 1) * TG + t) * 256 + lane * 4);
#pragma unroll
    for (int q = 1; q < kPartRuns; ++q)
      if (q0 + q < runs) v[0] += v[q];
    s = q0 == 0 ? v[0] : s + v[0];
  }
  const int token = t * 16 + r;
  if (GATED) store_gated(a, s, token, tile * 8);
  else if (token < a.T && 4 * g < rows) store_four(a, s, token, tile * rows + 4 * g);
}

// Runs of at most 16 J k: a wave per run, x in registers.  TG groups of 16 rows of x.  CUT: not
// every run is 16 J k.  J as small as holds a run: what a load of a place past it costs (56 clocks of its
// compute unit) is most of a small model's product (192 and 640 x 192, 3 rows: 6.5 to 7 us with places for
// 128 k, 3.3 to 4 with 16).
template <int TG, int J, bool CUT, bool GATED>
__global__ __launch_bounds__(kMaxRuns * 64) void gemm_f32_stream_kernel(
    const F32Args a, int tiles) {
  extern __shared__ __attribute__((aligned(16))) float red[];   // [2][runs][TG][64 lanes][4]
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, waves = blockDim.x / 64;
  const int r = lane % 16, g = lane / 16;
  const int run = a.run, k0 = wave * run, k1 = min(a.K, k0 + run);   // this wave's run
  f32x4 x[TG][J], w[2][J];
#pragma unroll
  for (int t = 0; t < TG; ++t) {
    const float* xr = a.X + (long long)min(t * 16 + r, a.T - 1) * a.ldx;
#pragma unroll
    for (int j = 0; j < J; ++j) x[t][j] = load4<CUT>(xr, k0 + 16 * j + 4 * g, k1);
  }
  const auto ask = [&](f32x4(&wn)[J], int tile) {
    // (past the last tile its last row is read again: no load under a condition)
    const float* wr = a.W + (long long)weight_row<GATED>(tile, r, 16, a.N) * a.ldw;
#pragma unroll
    for (int j = 0; j < J; ++j) wn[j] = load4<CUT>(wr, k0 + 16 * j + 4 * g, k1);
  };
  if (TG == 1) ask(w[0], blockIdx.x);
  int buf = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, buf ^= 1) {
    f32x4 acc[TG];
#pragma unroll
    for (int t = 0; t < TG; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // (two groups of x leave no registers for a second tile of weights)
    if (TG == 1) ask(w[1], tile + gridDim.x);
    else ask(w[0], tile);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      if (CUT && 16 * j >= run) break;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int t = 0; t < TG; ++t) acc[t] = mfma_f32(w[0][j][i], x[t][j][i], acc[t]);
      }
    }
    if (TG == 1) {
#pragma unroll
      for (int j = 0; j < J; ++j) w[0][j] = w[1][j];
    }
    float* part = red + (size_t)buf * waves * TG * 256;
#pragma unroll
    for (int t = 0; t < TG; ++t) *(f32x4*)(part + (wave * TG + t) * 256 + lane * 4) = acc[t];
    __syncthreads();
    // (the next tile writes the other buffer; this one is written again behind the barrier that
    // its readers reach only when they are done)
    for (int t = wave; t < TG; t += waves) store_tile<TG, GATED>(a, part, waves, t, tile, 16);
  }
}

// Longer runs: a wave per two runs (at most eight waves, so that a lane has 256 registers), each
// walked in chunks of 64 k; a ring of RING chunks of weights and x keeps RING - 1 of them in
// flight, over the ends of runs and tiles.  CUT: a run is no multiple of 64, or not all are whole.
template <int TG, bool CUT, bool GATED>
__global__ __launch_bounds__(kMaxRuns * 32) void gemm_f32_stream_long_kernel(const F32Args a, int runs,
                                                                             int tiles) {
  extern __shared__ __attribute__((aligned(16))) float red[];   // [2][runs][TG][64 lanes][4]
  constexpr int J = 4, RING = TG == 1 ? 5 : 4;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int r = lane % 16, g = lane / 16;
  const int run = a.run, K = a.K;
  const int chunks = (run + 16 * J - 1) / (16 * J);             // of a run
  const float* xr[TG];
#pragma unroll
  for (int t = 0; t < TG; ++t) xr[t] = a.X + (long long)min(t * 16 + r, a.T - 1) * a.ldx;
  f32x4 w[RING][J], x[RING][TG][J];

  // where the next chunk that is asked for lies
  int a_tile = blockIdx.x, a_run = 0, a_chunk = 0;
  const auto ask = [&](f32x4(&wn)[J], f32x4(&xn)[TG][J]) {
    const float* wr = a.W + (long long)weight_row<GATED>(a_tile, r, 16, a.N) * a.ldw;
    const int k0 = (2 * wave + a_run) * run, k1 = min(K, k0 + run);
    // (a wave's second run may lie past K: the row's last elements are read and, cut, zeroed)
    const int at = k0 + a_chunk * 16 * J + 4 * g;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int k = at + 16 * j, kc = min(k, max(k1, 4) - 4);
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      const f32x4 wv = *(const f32x4*)(wr + min(kc, K - 4));
      wn[j] = CUT && k >= k1 ? z : wv;
#pragma unroll
      for (int t = 0; t < TG; ++t) {
        const f32x4 xv = *(const f32x4*)(xr[t] + min(kc, K - 4));
        xn[t][j] = CUT && k >= k1 ? z : xv;
      }
    }
    __builtin_amdgcn_sched_barrier(0);                 // the loads leave before the products
    if (++a_chunk == chunks) {
      a_chunk = 0;
      if (++a_run == 2) { a_run = 0; a_tile += gridDim.x; }
    }
  };
#pragma unroll
  for (int q = 0; q < RING - 1; ++q) ask(w[q], x[q]);

  f32x4 acc[TG];
#pragma unroll
  for (int t = 0; t < TG; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  int tile = blockIdx.x, m_run = 0, m_chunk = 0, buf = 0;
  while (tile < tiles) {
#pragma unroll
    for (int q = 0; q < RING; ++q) {
      ask(w[(q + RING - 1) % RING], x[(q + RING - 1) % RING]);
#pragma unroll
      for (int j = 0; j < J; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int t = 0; t < TG; ++t) acc[t] = mfma_f32(w[q][j][i], x[q][t][j][i], acc[t]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (++m_chunk == chunks) {                       // the end of a run
        m_chunk = 0;
        float* part = red + (size_t)buf * runs * TG * 256;
        const int mine = 2 * wave + m_run;
        if (mine < runs) {
#pragma unroll
          for (int t = 0; t < TG; ++t)
            *(f32x4*)(part + (mine * TG + t) * 256 + lane * 4) = acc[t];
        }
#pragma unroll
        for (int t = 0; t < TG; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (++m_run == 2) {                            // the end of a tile
          m_run = 0;
          __syncthreads();
          if (wave < TG) store_tile<TG, GATED>(a, part, runs, wave, tile, 16);
          buf ^= 1;
          tile += gridDim.x;
          if (tile >= tiles) break;
        }
      }
    }
  }
}

// Up to 16 rows over K in whole 1024s (whole runs of a multiple of 64 k): W and x go straight from
// memory into LDS, every wave through a ring of its own, so that nothing waits for another wave but
// the tile's end.  What bounds it is the bytes in flight (a compute unit holds 128 KB of them; reading
// W once runs at 5.5 to 6 TB/s from 100 MB up).  Eight waves of two runs each; a chunk is 64 k (256 bytes) of RW * 4 weight rows
// and XW * 4 rows of x, asked for as soon as its place has been read.  Row r's piece i lies at piece
// i ^ (r % 16).  Tiles of 8 or 12 rows fill half or three quarters of a product (lanes beyond read
// a row twice).  The chunks a wave asks for ahead of its last products do not exist; they are asked of a buffer of no
// bytes, so that the counts of loads under way stay what they are and memory is not asked (the last row read again
// instead, up to as many bytes as a short tile's own: four tokens of the 1B shape behind prompts of 96, a pass 14,672 ->
// 14,526 us).  Where the waves' runs start an odd number of 4 KB apart or nearly so (ring_turns), every other workgroup
// takes them the other way round: walked in step by all workgroups they meet on the same few channels.
template <int RW, int XW>
__host__ __device__ constexpr int ring_chunks() {
  return std::min(6, 16384 / ((RW + XW) * 1024));
}
template <int RW, int XW, bool GATED>
__global__ __launch_bounds__(512) void gemm_f32_ring_kernel(const F32Args a, int tiles, int grid, int turns) {
#ifdef __HIP_DEVICE_COMPILE__   // (the host pass knows no buffer resources)
  constexpr int PER = RW + XW, CHUNK = PER * 1024, NB = ring_chunks<RW, XW>();
  typedef __attribute__((address_space(3))) void* lds_ptr;
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring_smem[];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int r = lane % 16, g = lane / 16;
  const uint32_t ldx = (uint32_t)a.ldx, ldw = (uint32_t)a.ldw;
  unsigned char* ring = ring_smem + wave * NB * CHUNK;
  float* red = (float*)(ring_smem + 8 * NB * CHUNK);            // [2][16 runs][64 lanes][4]
  const int chunks = a.run / 64 * 2;                            // of this wave's two runs
  const int flip = blockIdx.x & turns, turned = flip * (chunks / 2);  // (turns: odd workgroups take the later run first)
  // instruction i brings rows 4 i .. + 3 of a chunk, 16 lanes a row
  uint32_t src[PER];
  const auto place = [&](int row) { return (uint32_t)((r ^ (row & 15)) * 16); };
#pragma unroll
  for (int i = 0; i < XW; ++i) src[RW + i] = (uint32_t)min(4 * i + g, a.T - 1) * ldx * 4 + place(4 * i + g);
  const auto weight_rows = [&](int tile) {
#pragma unroll
    for (int i = 0; i < RW; ++i)
      src[i] = (uint32_t)weight_row<GATED>(tile, 4 * i + g, 4 * RW, a.N) * ldw * 4 + place(4 * i + g);
  };
  int a_tile = blockIdx.x, a_chunk = 0;
  constexpr uint32_t kWhole = 0xfffffff0u;   // (x and W end there at most; past the last tile nothing is read)
  uint32_t a_bytes = kWhole;
  const auto ask = [&](int buf) {
    const auto xr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.X + 2 * wave * a.run), 0, a_bytes, 0x00027000);
    const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.W + 2 * wave * a.run), 0, a_bytes, 0x00027000);
    unsigned char* base = ring + buf * CHUNK;
    const int at = (a_chunk + turned < chunks ? a_chunk + turned : a_chunk + turned - chunks) * 256;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (i < RW)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_ptr)(base + i * 1024), 16, src[i], at, 0, 2);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)(base + i * 1024), 16, src[i], at, 0, 0);
    }
    if (++a_chunk == chunks) {
      a_chunk = 0;
      a_tile += grid;
      a_bytes = a_tile < tiles ? kWhole : 0;
      weight_rows(a_tile);
    }
  };
  weight_rows(a_tile);
#pragma unroll
  for (int b = 0; b < NB; ++b) ask(b);
  const int w_row = r < 4 * RW ? r : r - 4 * RW, x_row = min(r, 4 * XW - 1);
  int buf = 0, side = 0, turn = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += grid, side ^= 1) {
    float* part = red + side * 16 * 256;
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < chunks / 2; ++c) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER * (NB - 1)) : "memory");
        const unsigned char* base = ring + buf * CHUNK;
        f32x4 w[4], x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          w[j] = *(const f32x4*)(base + w_row * 256 + ((4 * j + g) ^ w_row) * 16);
          x[j] = *(const f32x4*)(base + RW * 1024 + x_row * 256 + ((4 * j + g) ^ x_row) * 16);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the chunk has been read
        __builtin_amdgcn_sched_barrier(0);
        ask(buf);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
          for (int i = 0; i < 4; ++i) acc = mfma_f32(w[j][i], x[j][i], acc);
        }
        buf = buf + 1 == NB ? 0 : buf + 1;
      }
      *(f32x4*)(part + (2 * wave + (half ^ flip)) * 256 + lane * 4) = acc;
    }
    __syncthreads();
    // (the next tile writes the other side; this one is written again behind the barrier that its
    // reader reaches only when it is done)
    // (the waves take turns: the one that stores is behind the others when the next tile ends)
    if (wave == turn) store_tile<1, GATED>(a, part, 16, 0, tile, 4 * RW);
    turn = (turn + 1) % 8;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                // (loads past the last tile)
#endif
}

// ------------------------------------------------------------------ more rows
// Tile of 16 * MI rows of x and 64 weight rows by G groups of four waves, each group with 1 / G of
// the parts of k, 32 k a step.  A wave takes all rows of x and 16 weight rows, which no other wave
// needs: they go from memory into its registers, two steps ahead.  x goes through LDS (two buffers
// taking turns, two more steps on their way; rows 160 bytes apart, so that the 16-byte reads of a
// fragment are free of bank conflicts).  At the end the first group adds the parts of the others to its
// own, in order.  ENDS: where K ends.  GATED: a wave's weight rows are 8 gate rows and the 8 up rows of the
// same columns.
//
// A K that is no sixteen whole runs: groups that would hold none are not launched and steps past K are not
// multiplied, and where K ends with a step no load is selected (2,048 x 8,192 over 64 / 320 us: sixteen runs walked
// 106 / 179, no others 36 / 108, no selects 35 / 106).
enum { kWholeRuns = 0, kWholeSteps = 1, kAnywhere = 2 };
constexpr int kTileStride = 32 + 8;                  // floats
template <int MI>
constexpr int tile_bytes(int groups) {
  return groups * 2 * 16 * MI * kTileStride * 4;
}
template <int MI, int G, int ENDS, bool GATED>
__global__ __launch_bounds__(256 * G, 4) void gemm_f32_tiles_kernel(const F32Args a, int tiles_m,
                                                                    int tiles, int share) {
  constexpr int BM = 16 * MI, BK = 32, D = 2, COLS = GATED ? 32 : 64;
  constexpr bool CUT = ENDS == kAnywhere, SHORT = ENDS != kWholeRuns;
  constexpr int LOADS = (MI + 1) / 2;                // 16-byte pieces of x a thread stages
  extern __shared__ __attribute__((aligned(16))) float smem[];   // [groups][2][BM][kTileStride]
  // workgroups of one die (blockIdx % 8) take neighbouring tiles, the tiles of x fastest, so
  // that its L2 serves the weight rows that they share
  const int tile = (int)(blockIdx.x % 8) * share + (int)(blockIdx.x / 8);
  if (tile >= tiles) return;
  const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m * COLS;
  const int groups = blockDim.x / 256, group = __builtin_amdgcn_readfirstlane(threadIdx.x / 256);
  const int tid = threadIdx.x % 256, lane = tid % 64, wave = tid / 64;
  const int r = lane % 16, g = lane / 16;
  float* lds = smem + group * 2 * BM * kTileStride;
  const int run = a.run, K = a.K;
  const int span = kMaxRuns / G * run;
  const int k_begin = group * span;
  // (in 64s; every group walks as many steps: they share the barriers)
  const int k_count = SHORT ? min(span, (K + D * BK - 1) / (D * BK) * (D * BK)) : span;

  const float* wr = a.W + (long long)weight_row<GATED>(tile / tiles_m * 4 + wave, r, 16, a.N) * a.ldw;
  const float* src[LOADS];
  const int xk = k_begin + tid % 8 * 4;
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    src[i] = a.X + (long long)min(m0 + tid / 8 + i * 32, a.T - 1) * a.ldx;
  // acc: the run under way; part: its part so far; total: the parts (of the first group their
  // sum, of a later one the first of its two)
  f32x4 total[MI], part[MI], acc[MI];
  int part_runs = 0, parts = 0;
#pragma unroll
  for (int b = 0; b < MI; ++b) total[b] = part[b] = acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const auto end_part = [&]() {
    if (G < 4 && (group == 0 || parts == 0)) {
#pragma unroll
      for (int b = 0; b < MI; ++b) total[b] = parts == 0 ? part[b] : total[b] + part[b];
    }
    part_runs = 0;
    ++parts;
  };
  f32x4 w[D][2], x[D][LOADS];
  const auto ask_x = [&](f32x4(&xn)[LOADS], int k0) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) xn[i] = load4<CUT>(src[i], xk + k0, K);
  };
  const auto keep_x = [&](const f32x4(&xn)[LOADS], int buf) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      if (MI % 2 == 0 || i + 1 < LOADS || tid < 128)
        *(f32x4*)(lds + (buf * BM + tid / 8 + i * 32) * kTileStride + tid % 8 * 4) = xn[i];
    }
  };
  int left = run;                                    // k left of the run
  const auto step = [&](f32x4(&wn)[2], f32x4(&x_ask)[LOADS], const f32x4(&x_keep)[LOADS], int k0, int buf) {
    ask_x(x_ask, k0 + D * BK);
    const float* xs = lds + (buf * BM + r) * kTileStride + 4 * g;
    const bool live = !SHORT || k_begin + k0 < K;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (live) {
        f32x4 xv[MI];
#pragma unroll
        for (int b = 0; b < MI; ++b) xv[b] = *(const f32x4*)(xs + b * 16 * kTileStride + h * 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int b = 0; b < MI; ++b) acc[b] = mfma_f32(wn[h][i], xv[b][i], acc[b]);
        }
      }
      wn[h] = load4<CUT>(wr, k_begin + k0 + D * BK + h * 16 + 4 * g, K);
      left -= 16;
      if (left == 0) {                               // the end of a run
        left = run;
#pragma unroll
        for (int b = 0; b < MI; ++b) {
          part[b] = part_runs == 0 ? acc[b] : part[b] + acc[b];
          acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        if (++part_runs == kPartRuns) end_part();
      }
    }
    keep_x(x_keep, buf ^ 1);
    __syncthreads();
  };
#pragma unroll
  for (int q = 0; q < D; ++q) {
    ask_x(x[q], q * BK);
#pragma unroll
    for (int h = 0; h < 2; ++h) w[q][h] = load4<CUT>(wr, k_begin + q * BK + h * 16 + 4 * g, K);
  }
  keep_x(x[0], 0);
  __syncthreads();
  for (int k0 = 0; k0 < k_count; k0 += D * BK) {
#pragma unroll
    for (int q = 0; q < D; ++q) step(w[q], x[q], x[(q + 1) % D], k0 + q * BK, q % 2);
  }
  if (G == 1 && SHORT && (left < run || part_runs > 0)) {   // K ended inside a part
#pragma unroll
    for (int b = 0; b < MI; ++b) part[b] = part_runs == 0 ? acc[b] : part[b] + acc[b];
    end_part();
  }
  if (G == 4) {
#pragma unroll
    for (int b = 0; b < MI; ++b) total[b] = part[b];
  }
  // [group - 1][the group's part][wave][block][lane]
  constexpr int EACH = 4 / G;
  static_assert((G - 1) * EACH * 4 * MI * 1024 <= tile_bytes<MI>(G), "the parts fit the tiles' LDS");
  f32x4* hand = (f32x4*)smem;
  const auto place = [&](int q, int b) { return hand + ((q * 4 + wave) * MI + b) * 64 + lane; };
  if (group > 0) {
#pragma unroll
    for (int b = 0; b < MI; ++b) {
      *place((group - 1) * EACH, b) = total[b];
      if (EACH > 1) *place((group - 1) * EACH + 1, b) = part[b];
    }
  }
  __syncthreads();
  if (group > 0) return;
#pragma unroll
  for (int q = 0; q < (G - 1) * EACH; ++q) {
    if (SHORT && q >= (groups - 1) * EACH) break;
#pragma unroll
    for (int b = 0; b < MI; ++b) total[b] += *place(q, b);
  }
#pragma unroll
  for (int b = 0; b < MI; ++b) {
    const int token = m0 + b * 16 + r;
    if (GATED) {
      store_gated(a, total[b], token, n0 + wave * 8);
    } else if (token < a.T) {
      store_four(a, total[b], token, n0 + wave * 16 + 4 * g);
    }
  }
}

// Whether odd workgroups of the rings take their waves' runs the other way round (1) or all go in step (0); the same
// bits.  At 4 rows, us, in step -> turned: 1,536 x 8,192 16.7 -> 15.6, 2,048 x 8,192 20.1 -> 16.1, 4,096 x 8,192 36.9 ->
// 24.4, 16,384 x 8,192 113 -> 88, 4,096 x 24,576 71.7 -> 61.5, 4,096 x 9,216 27.6 -> 25.3, 3,072 x 7,168 18.4 -> 18.1;
// 1,024 x 8,192 14.7 -> 15.4, 2,048 x 7,168 14.9 -> 15.9, and 0.97 to 1.06 of the time over every other k in 1,024s up to
// 32,768 (6,144 x 4,096 19.3 -> 19.8, 3,072 x 16,384 35.9 -> 37.1).
int ring_turns(int rows_of_w, int K) {
  return (K % 16384 == 8192 && rows_of_w > 1024) || (K >= 7168 && K <= 9216 && rows_of_w >= 2560);
}

template <int RW, int XW, bool GATED>
int launch_ring(const F32Args& a, int cus, hipStream_t stream) {
  static LdsGrant grant;
  constexpr int bytes = 8 * ring_chunks<RW, XW>() * (RW + XW) * 1024 + 2 * 16 * 1024;
  const auto kernel = gemm_f32_ring_kernel<RW, XW, GATED>;
  const hipError_t e = grant_lds(grant, (const void*)kernel, bytes);
  RLIS_REQUIRE(e == hipSuccess, "gemm_f32: %s", hipGetErrorString(e));
  const int tiles = ceil_div(a.N, GATED ? 8 : 4 * RW);
  const int grid = std::min(tiles, cus);
  kernel<<<grid, 512, bytes, stream>>>(a, tiles, grid, ring_turns(GATED ? 2 * a.N : a.N, a.K));
  return 0;
}

template <int TG, bool GATED>
void launch_stream(const F32Args& a, int cus, hipStream_t stream) {
  const int tiles = ceil_div(a.N, GATED ? 8 : 16), runs = ceil_div(a.K, a.run), lds = 2 * runs * TG * 1024;
  if (a.run <= 128) {
    // as many workgroups as the registers of a compute unit hold (128 a lane at 16 waves)
    const int grid = std::min(tiles, cus * std::max(1, kMaxRuns / runs));
    const auto kernel = a.run == 16   ? gemm_f32_stream_kernel<TG, 1, true, GATED>
                        : a.run == 32 ? gemm_f32_stream_kernel<TG, 2, true, GATED>
                        : a.run <= 64 ? gemm_f32_stream_kernel<TG, 4, true, GATED>
                        : a.K % a.run || a.run != 128 ? gemm_f32_stream_kernel<TG, 8, true, GATED>
                                                      : gemm_f32_stream_kernel<TG, 8, false, GATED>;
    kernel<<<grid, runs * 64, lds, stream>>>(a, tiles);
  } else {
    const auto kernel = a.K % a.run || runs % 2 || a.run % 64 ? gemm_f32_stream_long_kernel<TG, true, GATED>
                                                              : gemm_f32_stream_long_kernel<TG, false, GATED>;
    kernel<<<std::min(tiles, cus), ceil_div(runs, 2) * 64, lds, stream>>>(a, runs, tiles);
  }
}

template <int MI, int G, int ENDS, bool GATED>
int launch_tiles_form(const F32Args& a, hipStream_t stream) {
  static LdsGrant grant;
  const auto kernel = gemm_f32_tiles_kernel<MI, G, ENDS, GATED>;
  const hipError_t e = grant_lds(grant, (const void*)kernel, tile_bytes<MI>(G));
  RLIS_REQUIRE(e == hipSuccess, "gemm_f32: %s", hipGetErrorString(e));
  const int groups = ceil_div(a.K, kMaxRuns / G * a.run);   // (no more than have a part)
  const int tm = ceil_div(a.T, 16 * MI), tiles = tm * ceil_div(a.N, GATED ? 32 : 64);
  const int share = ceil_div(tiles, 8);
  kernel<<<share * 8, 256 * groups, tile_bytes<MI>(groups), stream>>>(a, tm, tiles, share);
  return 0;
}

template <int MI, int G, bool GATED>
int launch_tiles(const F32Args& a, hipStream_t stream) {
  if (a.K == kMaxRuns * a.run) return launch_tiles_form<MI, G, kWholeRuns, GATED>(a, stream);
  return a.K % 32 == 0 ? launch_tiles_form<MI, G, kWholeSteps, GATED>(a, stream)
                       : launch_tiles_form<MI, G, kAnywhere, GATED>(a, stream);
}

template <bool GATED>
int by_rows(const F32Args& a, int cus, hipStream_t stream) {
  const int T = a.T, rows_of_w = GATED ? 2 * a.N : a.N;
  // Rows whose bytes a buffer's 32-bit offset reaches.  More than 4 rows bring half as much x as W
  // into the rings and more: over more than eight tiles a compute unit the stream kernel, which
  // keeps x of short runs in registers, is ahead (128256 x 2048 at 16 rows: 192 us against 242, at 8
  // no slower than the 192; 16384 x 2048, four tiles, 16 rows: 33 against 27).
  const bool ring = a.K % 1024 == 0 && 4 * (a.ldw * (rows_of_w - 1) + a.K) < (1LL << 32) &&
                    4 * (a.ldx * (T - 1) + a.K) < (1LL << 32) &&
                    (T <= 4 || a.run > 128 || ceil_div(rows_of_w, 16) <= 8 * cus);
  if (T <= 16 && ring) {
    if (GATED) {
      if (T <= 4) return launch_ring<4, 1, GATED>(a, cus, stream);
      if (T <= 8) return launch_ring<4, 2, GATED>(a, cus, stream);
      return launch_ring<4, 4, GATED>(a, cus, stream);
    }
    // Tiles of 16 weight rows, or of 12 or 8 where that takes rows off the busiest compute unit
    // (3072 x 2048 at 4 rows: 8.6 us with 12, 2048 x 2048: 7.9 with 8)
    int rows = 16, most = ceil_div(ceil_div(a.N, 16), cus) * 16;
    for (int c = 12; c >= 8; c -= 4) {
      const int m = ceil_div(ceil_div(a.N, c), cus) * c;
      if (m < most) { rows = c; most = m; }
    }
#define BY_X(RW)                                                     \
  (T <= 4 ? launch_ring<RW, 1, false>(a, cus, stream)                \
          : T <= 8 ? launch_ring<RW, 2, false>(a, cus, stream)       \
                   : launch_ring<RW, 4, false>(a, cus, stream))
    return rows == 16 ? BY_X(4) : rows == 12 ? BY_X(3) : BY_X(2);
#undef BY_X
  }
  if (T <= 32) {
    if (T <= 16) launch_stream<1, GATED>(a, cus, stream);
    else launch_stream<2, GATED>(a, cus, stream);
    return 0;
  }
  // Every tile and number of groups gives the same bits; the matrix cores bound them, so what counts is
  // the blocks of 16 rows that the busiest compute unit works through: the height that makes least of
  // rounds of tiles times the time of a round.  A round of 16, 32, ... 80 rows over K = 2048 takes 18, 20,
  // 30, 38 and 48 us (one of 16 rows is bound by its loads of W, 56 clocks each).  384 rows, by height: 3072 x 2048
  // 93 / 62 / 62 / 77 / 50 us, 2048 x 2048 58 / 43 / 33 / 40 / 49; 200 rows of 16384 x 2048 244 / 145 / 152 / 154 / 145.
  // Four groups take a tile's k in quarters where no compute unit has a second tile (2048 x 2048, 384
  // rows: 33 us against 34 with two, 2048 x 8192: 112 against 119); two otherwise, so that a second tile
  // works through its first and last steps beside them (16384 x 2048, 384 rows: 212 against 231), but
  // 80 rows, whose sums leave no room for a second tile (3072 x 2048, 384 rows: 49 us against 53 with two).
  // Over a short k a group is soon done and one does with the fewest steps for nothing (8192 x 192, 768 rows: 37 us
  // with two, 33 with one; x 384 59 and 52; x 768 88 and 86; x 1024 equal), two where all four
  // would have a part to do (640 x 256, 512 rows: 7.3 us with four, 6.6).  16 rows take two always:
  // their loads of W bound them, whoever waits (640 x 512, 64 rows: 8.0 us with four, 7.1).
  const int tn = ceil_div(a.N, GATED ? 32 : 64);
  constexpr int kRound[] = {0, 18, 20, 30, 38, 48};
  int mi = 1;
  long long least = 1LL << 62;
  for (int m = 5; m > 0; --m) {
    const long long us = ceil_div_ll((long long)ceil_div(T, 16 * m) * tn, cus) * kRound[m];
    if (us < least) { least = us; mi = m; }
  }
  const bool pairs = (long long)ceil_div(T, 16 * mi) * tn > cus;
  const bool halves = pairs || (a.K <= 512 && a.K == kMaxRuns * a.run);
#define GO(M)                                                                      \
  case M:                                                                          \
    return pairs && a.K <= 768 ? launch_tiles<M, 1, GATED>(a, stream)              \
                               : halves ? launch_tiles<M, 2, GATED>(a, stream)     \
                                        : launch_tiles<M, 4, GATED>(a, stream)
  switch (mi) {
    case 1: return launch_tiles<1, 2, GATED>(a, stream);
    GO(2); GO(3); GO(4);
    default: return launch_tiles<5, 4, GATED>(a, stream);
  }
#undef GO
}

}  // namespace

// Y (T,N) = X (T,K) * W (N,K)^T, float32, row strides in elements; K and the strides of X and W
// multiples of 4, X and W on 16-byte boundaries.  gated: W (2 N,K) gate rows then up rows, Y =
// silu(gate) * up.
RLIS_API int rlis_gemm_f32(const void* X_, const void* W_, void* Y_, int T, int N, int K,
                           long long ldx, long long ldw, long long ldy, int gated, hipStream_t stream) {
  const float *X = (const float*)X_, *W = (const float*)W_;
  float* Y = (float*)Y_;
  RLIS_REQUIRE(T >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes T=%d N=%d K=%d", T, N, K);
  RLIS_REQUIRE(ldx >= K && ldw >= K && ldy >= N, "gemm_f32: row strides shorter than rows");
  RLIS_REQUIRE(K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && (uintptr_t)X % 16 == 0 &&
                   (uintptr_t)W % 16 == 0,
               "gemm_f32: K and the strides of x and W must be multiples of 4, x and W on 16-byte "
               "boundaries");
  RLIS_REQUIRE(ceil_div(T, 64) <= 65535 && N <= (1 << (gated ? 25 : 26)), "gemm_f32: T=%d N=%d is too large",
               T, N);
  if (T == 0) return 0;
  const int cus = rlis_stream_compute_units();
  RLIS_REQUIRE(cus > 0, "gemm_f32: cannot read the device properties");
  const F32Args a = {X, W, Y, T, N, K, f32_run(K), ldx, ldw, ldy, ldy % 4 == 0 && (uintptr_t)Y % 16 == 0};
  const int rc = gated ? by_rows<true>(a, cus, stream) : by_rows<false>(a, cus, stream);
  if (rc) return rc;
  RLIS_LAUNCH_CHECK("gemm_f32");
  return 0;
}
