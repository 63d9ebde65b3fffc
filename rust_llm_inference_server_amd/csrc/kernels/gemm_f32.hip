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
//    stream kernel -> this): 3072 x 2048 10.8 -> 8.6, 2048 x 2048 10.2 -> 7.9, 16384 x 2048 30.2 ->
//    24.7 (5.4 TB/s), 2048 x 8192 30 -> 21, 128256 x 2048 182 -> 177 (5.9 TB/s), 4096 x 14336 39
//    (6.1 TB/s); at 16 rows 2048 x 8192 37 -> 22.
//  * gemm_f32_stream: other K, and 17 to 32 rows.  A workgroup takes 16 weight rows
//    at a time, one wave per run of k, so a wave's loads of a tile are all in flight at once
//    (8 KB) and the next tile's are asked for before this one's products; runs of up to 128 k
//    keep x in registers over all tiles.  The waves' sums meet in LDS.  At 32 rows of the 1B
//    shape, weights cold: q/k/v 16, output 16, gate/up 40, head 242, down 59 us: there, and
//    wherever the long form runs, x is loaded as often as W, and a load of either takes its
//    compute unit about 24 ns (56 clocks, sixteen row pieces of 64 bytes), which bounds it.
//  * gemm_f32_tiles: more rows, bound by the matrix cores (154 TFLOP/s for a large library
//    product here).  Tiles of x and W go through two LDS buffers taking turns, 32 k at a time,
//    rows 160 bytes apart so that the 16-byte reads of a fragment are free of bank conflicts.
//    384 rows of the 1B shape: q/k/v 310 -> 70 us (69 TFLOP/s; 288 tiles do not come out even
//    over 256 compute units), output 300 -> 46, gate/up 461 -> 237 (109), down 1100 -> 164.
// The sums in parts also halve the error and more: 2.1e-7 of the result's norm against 64 bits at
// K = 2048 (gemm_plain 8.1e-7), 4.1e-7 at 8192 (1.6e-6).
#include "common.h"

#include <algorithm>

typedef float f32x4 __attribute__((ext_vector_type(4)));

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

// ------------------------------------------------------------------ up to 32 rows
// The sum of a tile's runs, which lie in LDS as [run][group of rows][lane], for rows t * 16 .. + 15
// of x: stored by one wave.
template <int TG>
__device__ __forceinline__ void store_tile(const float* red, int runs, int t, int tile, int rows,
                                           float* Y, int T, int N, long long ldy, int vec_out) {
  const int lane = threadIdx.x % 64, r = lane % 16, g = lane / 16;
  f32x4 s;
  for (int q0 = 0; q0 < runs; q0 += kPartRuns) {
    f32x4 p = *(const f32x4*)(red + (q0 * TG + t) * 256 + lane * 4);
    for (int q = q0 + 1; q < min(runs, q0 + kPartRuns); ++q)
      p += *(const f32x4*)(red + (q * TG + t) * 256 + lane * 4);
    s = q0 == 0 ? p : s + p;
  }
  const int token = t * 16 + r, n = tile * rows + 4 * g;
  if (token >= T || 4 * g >= rows) return;
  float* y = Y + token * ldy + n;
  if (vec_out && n + 4 <= N) {
    *(f32x4*)y = s;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < N) y[i] = s[i];
  }
}

// Runs of at most 128 k: a wave per run, x in registers.  TG groups of 16 rows of x.  CUT: not
// every run is 128 k.
template <int TG, bool CUT>
__global__ __launch_bounds__(kMaxRuns * 64) void gemm_f32_stream_kernel(
    const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int T, int N,
    int K, int run, int tiles, long long ldx, long long ldw, long long ldy, int vec_out) {
  extern __shared__ __attribute__((aligned(16))) float red[];   // [2][runs][TG][64 lanes][4]
  constexpr int J = 8;                                          // steps of 16 k
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, waves = blockDim.x / 64;
  const int r = lane % 16, g = lane / 16;
  const int k0 = wave * run, k1 = min(K, k0 + run);             // this wave's run
  f32x4 x[TG][J], w[2][J];
#pragma unroll
  for (int t = 0; t < TG; ++t) {
    const float* xr = X + (long long)min(t * 16 + r, T - 1) * ldx;
#pragma unroll
    for (int j = 0; j < J; ++j) x[t][j] = load4<CUT>(xr, k0 + 16 * j + 4 * g, k1);
  }
  const auto ask = [&](f32x4(&wn)[J], int tile) {
    // (past the last tile its last row is read again: no load under a condition)
    const float* wr = W + (long long)min(tile * 16 + r, N - 1) * ldw;
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
    for (int t = wave; t < TG; t += waves) store_tile<TG>(part, waves, t, tile, 16, Y, T, N, ldy, vec_out);
  }
}

// Longer runs: a wave per two runs (at most eight waves, so that a lane has 256 registers), each
// walked in chunks of 64 k; a ring of RING chunks of weights and x keeps RING - 1 of them in
// flight, over the ends of runs and tiles.  CUT: a run is no multiple of 64, or not all are whole.
template <int TG, bool CUT>
__global__ __launch_bounds__(kMaxRuns * 32) void gemm_f32_stream_long_kernel(
    const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int T, int N,
    int K, int run, int runs, int tiles, long long ldx, long long ldw, long long ldy, int vec_out) {
  extern __shared__ __attribute__((aligned(16))) float red[];   // [2][runs][TG][64 lanes][4]
  constexpr int J = 4, RING = TG == 1 ? 5 : 4;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int r = lane % 16, g = lane / 16;
  const int chunks = (run + 16 * J - 1) / (16 * J);             // of a run
  const float* xr[TG];
#pragma unroll
  for (int t = 0; t < TG; ++t) xr[t] = X + (long long)min(t * 16 + r, T - 1) * ldx;
  f32x4 w[RING][J], x[RING][TG][J];

  // where the next chunk that is asked for lies
  int a_tile = blockIdx.x, a_run = 0, a_chunk = 0;
  const auto ask = [&](f32x4(&wn)[J], f32x4(&xn)[TG][J]) {
    const float* wr = W + (long long)min(a_tile * 16 + r, N - 1) * ldw;
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
          for (int t = 0; t < TG; ++t) *(f32x4*)(part + (mine * TG + t) * 256 + lane * 4) = acc[t];
        }
#pragma unroll
        for (int t = 0; t < TG; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (++m_run == 2) {                            // the end of a tile
          m_run = 0;
          __syncthreads();
          if (wave < TG) store_tile<TG>(part, runs, wave, tile, 16, Y, T, N, ldy, vec_out);
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
// a row twice).
template <int RW, int XW>
__host__ __device__ constexpr int ring_chunks() {
  return std::min(6, 16384 / ((RW + XW) * 1024));
}
template <int RW, int XW>
__global__ __launch_bounds__(512) void gemm_f32_ring_kernel(
    const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int T, int N,
    int run, int tiles, uint32_t ldx, uint32_t ldw, long long ldy, int vec_out) {
#ifdef __HIP_DEVICE_COMPILE__   // (the host pass knows no buffer resources)
  constexpr int PER = RW + XW, CHUNK = PER * 1024, NB = ring_chunks<RW, XW>();
  typedef __attribute__((address_space(3))) void* lds_ptr;
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring_smem[];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int r = lane % 16, g = lane / 16;
  unsigned char* ring = ring_smem + wave * NB * CHUNK;
  float* red = (float*)(ring_smem + 8 * NB * CHUNK);            // [2][16 runs][64 lanes][4]
  const int chunks = run / 64 * 2;                              // of this wave's two runs
  const auto xr = __builtin_amdgcn_make_buffer_rsrc((void*)(X + 2 * wave * run), 0, 0xffffffff, 0x00027000);
  const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)(W + 2 * wave * run), 0, 0xffffffff, 0x00027000);
  // instruction i brings rows 4 i .. + 3 of a chunk, 16 lanes a row
  uint32_t src[PER];
  const auto place = [&](int row) { return (uint32_t)((r ^ (row & 15)) * 16); };
#pragma unroll
  for (int i = 0; i < XW; ++i) src[RW + i] = (uint32_t)min(4 * i + g, T - 1) * ldx * 4 + place(4 * i + g);
  const auto weight_rows = [&](int tile) {
#pragma unroll
    for (int i = 0; i < RW; ++i)
      src[i] = (uint32_t)min(tile * 4 * RW + 4 * i + g, N - 1) * ldw * 4 + place(4 * i + g);
  };
  int a_tile = blockIdx.x, a_chunk = 0;
  const auto ask = [&](int buf) {
    unsigned char* base = ring + buf * CHUNK;
    const int at = a_chunk * 256;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (i < RW)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_ptr)(base + i * 1024), 16, src[i], at, 0, 2);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)(base + i * 1024), 16, src[i], at, 0, 0);
    }
    if (++a_chunk == chunks) {             // (past the last tile its last row is read again)
      a_chunk = 0;
      a_tile += gridDim.x;
      weight_rows(a_tile);
    }
  };
  weight_rows(a_tile);
#pragma unroll
  for (int b = 0; b < NB; ++b) ask(b);
  const int w_row = r < 4 * RW ? r : r - 4 * RW, x_row = min(r, 4 * XW - 1);
  int buf = 0, side = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, side ^= 1) {
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
      *(f32x4*)(part + (2 * wave + half) * 256 + lane * 4) = acc;
    }
    __syncthreads();
    // (the next tile writes the other side; this one is written again behind the barrier that its
    // reader reaches only when it is done)
    if (wave == 0) store_tile<1>(part, 16, 0, tile, 4 * RW, Y, T, N, ldy, vec_out);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                // (loads past the last tile)
#endif
}

// ------------------------------------------------------------------ more rows
// Tile of BM rows of x and BN weight rows by G groups of four waves, each group with its own
// LDS tiles and 1 / G of the parts of k; the waves of a group as 2 x 2, each BM / 2 x BN / 2.  At
// the end the first group adds the parts of the others to its own, in order.  CUT: k does not
// come out even (K no multiple of 32, the last run or the last parts not whole).
template <int BM, int BN, int G, bool CUT>
__global__ __launch_bounds__(256 * G) void gemm_f32_tiles_kernel(
    const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int T, int N,
    int K, int run, int tiles_m, int tiles, int share, long long ldx, long long ldw, long long ldy,
    int vec_out) {
  constexpr int BK = 32, STRIDE = BK + 8;            // floats; 160 bytes a row
  constexpr int MI = BM / 32, NI = BN / 32;          // 16 x 16 blocks of a wave
  constexpr int LOADS = (BM + BN) * (BK / 4) / 256;  // 16-byte pieces a thread stages
  constexpr int TILE = (BM + BN) * STRIDE;
  extern __shared__ __attribute__((aligned(16))) float smem[];   // [G][2][TILE]
  // workgroups of one die (blockIdx % 8) take neighbouring tiles, the tiles of x fastest, so
  // that its L2 serves the weight rows that they share
  const int tile = (int)(blockIdx.x % 8) * share + (int)(blockIdx.x / 8);
  if (tile >= tiles) return;
  const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m * BN;
  const int group = G == 1 ? 0 : threadIdx.x / 256;
  const int tid = threadIdx.x % 256, lane = tid % 64, wave = tid / 64;
  const int r = lane % 16, g = lane / 16;
  const int wm = wave / 2 * (BM / 2), wn = wave % 2 * (BN / 2);
  float* lds = smem + group * 2 * TILE;
  const int span = kMaxRuns / G * run;               // a multiple of 64
  const int k_begin = group * span;
  const int k_count = G > 1 ? span : ((K + run - 1) / run * run + BK - 1) / BK * BK;

  const float* src[LOADS];
  int dst[LOADS], kk[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int p = tid + i * 256, rw = p / (BK / 4);  // rows of x first, then weight rows
    kk[i] = k_begin + p % (BK / 4) * 4;
    dst[i] = rw * STRIDE + p % (BK / 4) * 4;
    src[i] = rw < BM ? X + (long long)min(m0 + rw, T - 1) * ldx
                     : W + (long long)min(n0 + rw - BM, N - 1) * ldw;
  }
  // acc: the run under way; part: its part so far; total: the parts (of the first group their
  // sum, of a later one the first of its two)
  f32x4 total[NI][MI], part[NI][MI], acc[NI][MI], st[LOADS];
  int part_runs = 0, parts = 0;
#pragma unroll
  for (int a = 0; a < NI; ++a) {
#pragma unroll
    for (int b = 0; b < MI; ++b) total[a][b] = part[a][b] = acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const auto end_part = [&]() {
    if (group == 0 || parts == 0) {
#pragma unroll
      for (int a = 0; a < NI; ++a) {
#pragma unroll
        for (int b = 0; b < MI; ++b)
          total[a][b] = parts == 0 ? part[a][b] : total[a][b] + part[a][b];
      }
    }
    part_runs = 0;
    ++parts;
  };
#pragma unroll
  for (int i = 0; i < LOADS; ++i) st[i] = load4<CUT>(src[i], kk[i], K);
#pragma unroll
  for (int i = 0; i < LOADS; ++i) *(f32x4*)(lds + dst[i]) = st[i];
  __syncthreads();
  int buf = 0, left = run;                           // k left of the run
  for (int k0 = 0; k0 < k_count; k0 += BK, buf ^= 1) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) st[i] = load4<CUT>(src[i], k0 + BK + kk[i], K);
    const float* xs = lds + buf * TILE + (wm + r) * STRIDE + 4 * g;
    const float* ws = lds + buf * TILE + (BM + wn + r) * STRIDE + 4 * g;
#pragma unroll
    for (int h = 0; h < BK; h += 16) {
      f32x4 x[MI], w[NI];
#pragma unroll
      for (int b = 0; b < MI; ++b) x[b] = *(const f32x4*)(xs + b * 16 * STRIDE + h);
#pragma unroll
      for (int a = 0; a < NI; ++a) w[a] = *(const f32x4*)(ws + a * 16 * STRIDE + h);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int a = 0; a < NI; ++a) {
#pragma unroll
          for (int b = 0; b < MI; ++b) acc[a][b] = mfma_f32(w[a][i], x[b][i], acc[a][b]);
        }
      }
      left -= 16;
      if (left == 0) {                               // the end of a run
        left = run;
#pragma unroll
        for (int a = 0; a < NI; ++a) {
#pragma unroll
          for (int b = 0; b < MI; ++b) {
            part[a][b] = part_runs == 0 ? acc[a][b] : part[a][b] + acc[a][b];
            acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
        if (++part_runs == kPartRuns) end_part();
      }
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i) *(f32x4*)(lds + (buf ^ 1) * TILE + dst[i]) = st[i];
    __syncthreads();
  }
  if (part_runs > 0) end_part();
  if (G > 1) {
    // [group - 1][the group's part][wave][block][lane]
    constexpr int EACH = 4 / G;
    static_assert((G - 1) * EACH * BM * BN <= G * 2 * TILE, "the parts fit the tiles' LDS");
    f32x4* hand = (f32x4*)smem;
    const auto place = [&](int q, int a, int b) {
      return hand + (((q * 4 + wave) * NI + a) * MI + b) * 64 + lane;
    };
    if (group > 0) {
#pragma unroll
      for (int a = 0; a < NI; ++a) {
#pragma unroll
        for (int b = 0; b < MI; ++b) {
          *place((group - 1) * EACH, a, b) = total[a][b];
          if (EACH > 1) *place((group - 1) * EACH + 1, a, b) = part[a][b];
        }
      }
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int q = 0; q < (G - 1) * EACH; ++q) {
#pragma unroll
      for (int a = 0; a < NI; ++a) {
#pragma unroll
        for (int b = 0; b < MI; ++b) total[a][b] += *place(q, a, b);
      }
    }
  }
#pragma unroll
  for (int a = 0; a < NI; ++a) {
#pragma unroll
    for (int b = 0; b < MI; ++b) {
      const f32x4 s = total[a][b];
      const int token = m0 + wm + b * 16 + r, n = n0 + wn + a * 16 + 4 * g;
      if (token >= T) continue;
      float* y = Y + token * ldy + n;
      if (vec_out && n + 4 <= N) {
        *(f32x4*)y = s;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) y[i] = s[i];
      }
    }
  }
}

int compute_units() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return n;
}

template <int RW, int XW>
int launch_ring(const float* X, const float* W, float* Y, int T, int N, int run, int cus, long long ldx,
                long long ldw, long long ldy, int vec, hipStream_t stream) {
  static LdsGrant grant;
  constexpr int bytes = 8 * ring_chunks<RW, XW>() * (RW + XW) * 1024 + 2 * 16 * 1024;
  const auto kernel = gemm_f32_ring_kernel<RW, XW>;
  const hipError_t e = grant_lds(grant, (const void*)kernel, bytes);
  RLIS_REQUIRE(e == hipSuccess, "gemm_f32: %s", hipGetErrorString(e));
  const int tiles = ceil_div(N, 4 * RW);
  kernel<<<std::min(tiles, cus), 512, bytes, stream>>>(X, W, Y, T, N, run, tiles, (uint32_t)ldx,
                                                       (uint32_t)ldw, ldy, vec);
  return 0;
}

template <int TG>
void launch_stream(const float* X, const float* W, float* Y, int T, int N, int K, int run, int cus,
                   long long ldx, long long ldw, long long ldy, int vec, hipStream_t stream) {
  const int tiles = ceil_div(N, 16), runs = ceil_div(K, run), lds = 2 * runs * TG * 1024;
  if (run <= 128) {
    // as many workgroups as the registers of a compute unit hold (128 a lane at 16 waves)
    const int grid = std::min(tiles, cus * std::max(1, kMaxRuns / runs));
    const auto kernel = K % run || run != 128 ? gemm_f32_stream_kernel<TG, true>
                                              : gemm_f32_stream_kernel<TG, false>;
    kernel<<<grid, runs * 64, lds, stream>>>(X, W, Y, T, N, K, run, tiles, ldx, ldw, ldy, vec);
  } else {
    const auto kernel = K % run || runs % 2 || run % 64 ? gemm_f32_stream_long_kernel<TG, true>
                                                        : gemm_f32_stream_long_kernel<TG, false>;
    kernel<<<std::min(tiles, cus), ceil_div(runs, 2) * 64, lds, stream>>>(
        X, W, Y, T, N, K, run, runs, tiles, ldx, ldw, ldy, vec);
  }
}

template <int BM, int BN, int G, bool CUT>
int launch_tiles_form(const float* X, const float* W, float* Y, int T, int N, int K, int run,
                      long long ldx, long long ldw, long long ldy, int vec, hipStream_t stream) {
  static LdsGrant grant;
  constexpr int bytes = G * 2 * (BM + BN) * 40 * 4;
  const auto kernel = gemm_f32_tiles_kernel<BM, BN, G, CUT>;
  const hipError_t e = grant_lds(grant, (const void*)kernel, bytes);
  RLIS_REQUIRE(e == hipSuccess, "gemm_f32: %s", hipGetErrorString(e));
  const int tm = ceil_div(T, BM), tiles = tm * ceil_div(N, BN), share = ceil_div(tiles, 8);
  kernel<<<share * 8, 256 * G, bytes, stream>>>(X, W, Y, T, N, K, run, tm, tiles, share, ldx, ldw,
                                                ldy, vec);
  return 0;
}

template <int BM, int BN, int G>
int launch_tiles(const float* X, const float* W, float* Y, int T, int N, int K, int run,
                 long long ldx, long long ldw, long long ldy, int vec, hipStream_t stream) {
  const bool cut = K % 32 || K % run || (G > 1 && kMaxRuns * run != K);
  return cut ? launch_tiles_form<BM, BN, G, true>(X, W, Y, T, N, K, run, ldx, ldw, ldy, vec, stream)
             : launch_tiles_form<BM, BN, G, false>(X, W, Y, T, N, K, run, ldx, ldw, ldy, vec, stream);
}

}  // namespace

// Y (T,N) = X (T,K) * W (N,K)^T, float32, row strides in elements; K and the strides of X and W
// multiples of 4, X and W on 16-byte boundaries.
RLIS_API int rlis_gemm_f32(const void* X_, const void* W_, void* Y_, int T, int N, int K,
                           long long ldx, long long ldw, long long ldy, hipStream_t stream) {
  const float *X = (const float*)X_, *W = (const float*)W_;
  float* Y = (float*)Y_;
  RLIS_REQUIRE(T >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes T=%d N=%d K=%d", T, N, K);
  RLIS_REQUIRE(ldx >= K && ldw >= K && ldy >= N, "gemm_f32: row strides shorter than rows");
  RLIS_REQUIRE(K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && (uintptr_t)X % 16 == 0 &&
                   (uintptr_t)W % 16 == 0,
               "gemm_f32: K and the strides of x and W must be multiples of 4, x and W on 16-byte "
               "boundaries");
  RLIS_REQUIRE(T <= (1 << 24) && N <= (1 << 26), "gemm_f32: T=%d N=%d is too large", T, N);
  if (T == 0) return 0;
  const int run = f32_run(K), cus = compute_units();
  RLIS_REQUIRE(cus > 0, "gemm_f32: cannot read the device properties");
  const int vec = ldy % 4 == 0 && (uintptr_t)Y % 16 == 0;
  // Rows whose bytes a buffer's 32-bit offset reaches.  More than 4 rows bring half as much x as W
  // into the rings and more: over more than eight tiles a compute unit the stream kernel, which
  // keeps x of short runs in registers, is ahead (128256 x 2048 at 16 rows: 192 us against 242, at 8
  // no slower than the 192; 16384 x 2048, four tiles, 16 rows: 33 against 27).
  const bool ring = K % 1024 == 0 && 4 * (ldw * (N - 1) + K) < (1LL << 32) &&
                    4 * (ldx * (T - 1) + K) < (1LL << 32) &&
                    (T <= 4 || run > 128 || ceil_div(N, 16) <= 8 * cus);
  if (T <= 16 && ring) {
    // Tiles of 16 weight rows, or of 12 or 8 where that takes rows off the busiest compute unit
    // (3072 x 2048 at 4 rows: 8.6 us with 12, 2048 x 2048: 7.9 with 8)
    int rows = 16, most = ceil_div(ceil_div(N, 16), cus) * 16;
    for (int c = 12; c >= 8; c -= 4) {
      const int m = ceil_div(ceil_div(N, c), cus) * c;
      if (m < most) { rows = c; most = m; }
    }
    int rc;
#define GO(RW, XW) rc = launch_ring<RW, XW>(X, W, Y, T, N, run, cus, ldx, ldw, ldy, vec, stream)
#define BY_X(RW)                        \
  do {                                  \
    if (T <= 4) GO(RW, 1);              \
    else if (T <= 8) GO(RW, 2);         \
    else GO(RW, 4);                     \
  } while (0)
    if (rows == 16) BY_X(4);
    else if (rows == 12) BY_X(3);
    else BY_X(2);
#undef BY_X
#undef GO
    if (rc) return rc;
  } else if (T <= 32) {
    if (T <= 16) launch_stream<1>(X, W, Y, T, N, K, run, cus, ldx, ldw, ldy, vec, stream);
    else launch_stream<2>(X, W, Y, T, N, K, run, cus, ldx, ldw, ldy, vec, stream);
  } else {
    // Every tile and number of groups gives the same bits; the matrix cores bound all of them,
    // so the compute units should have the same work and four waves a SIMD.  Where half tiles
    // number at most one a compute unit, four groups take a tile's k in quarters (1B output
    // projection, 2048 x 2048, 128 rows: 30 us; one group 52); likewise whole tiles (384 rows:
    // 45 us; one group 64).  Beyond that half tiles only where they save part of a round
    // (3072 x 2048, 384 rows: 68 us against 77), and two groups up to two tiles a compute unit
    // (16384 x 2048, 128 rows: 83 us against 89).
    const int t64 = ceil_div(T, 64) * ceil_div(N, 64), t32 = ceil_div(T, 64) * ceil_div(N, 32);
    int rc;
#define GO(BN, G) rc = launch_tiles<64, BN, G>(X, W, Y, T, N, K, run, ldx, ldw, ldy, vec, stream)
    if (t32 <= cus) GO(32, 4);
    else if (t64 <= cus) GO(64, 4);
    else if (ceil_div(t32, cus) < 2 * ceil_div(t64, cus) && t64 <= 2 * cus) GO(32, 1);
    else if (t64 <= 2 * cus) GO(64, 2);
    else GO(64, 1);
#undef GO
    if (rc) return rc;
  }
  RLIS_LAUNCH_CHECK("gemm_f32");
  return 0;
}
