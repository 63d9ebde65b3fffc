// bfloat16 products y = x * W^T for 17 to 64 rows of x: decode steps of many requests.
//
// Bound by reading W once, beside as many bytes of x through the L2 (every workgroup reads all
// rows of x).  A workgroup takes 64, 32 or 16 weight rows at a time; W and x go straight from
// memory into LDS (buffer_load ... lds) in stages of 128 k, three to seven of them under way
// (about 100 KB a compute unit: a stage takes 1.5 us to arrive, so what is in flight bounds the
// rate), over the ends of tiles.  Rows of a stage are 256 bytes; piece i of row r lies at piece
// i ^ (r % 16), which the load does by choosing what each lane reads, so that fragments are read
// without bank conflicts.  Each of the four waves multiplies a quarter of a stage's k for the
// whole tile (32 k: one v_mfma_f32_16x16x32_bf16 per block), which reads every fragment from LDS
// once; with the waves side by side over the tile's rows every wave read all of x and a stage
// took 1.4 times as long.  The waves' sums meet in LDS, wave 0 first.  Tile t starts at stage
// t % steps and wraps round, so that workgroups do not walk one column of W in step; W is loaded
// non-temporally where the model is larger than the memory-side cache (64 rows, gate/up with the
// SwiGLU, 1B: 20.1 -> 19.0 us; 32 rows, 8B: 52 -> 46).
// The order of a sum follows from N and K alone: a row's bits do not depend on the rows beside it.
// What ends a slice: with the join, the last of a tile's slices to store its sum (past the die's cache, then an
// atomic count) adds all of them to the residual; the sums of squares that scale the rows of the product behind
// are asked for in front of its first stages, not behind them (the wait for them is in order: q/k/v of 27 rows of
// the 3B shape 11.6 -> 10.8 us, gate/up 21.8 -> 21.3).
// Weights loaded straight into registers instead (16 rows x 64 bytes an instruction, more bytes
// under way): 10 to 20 % slower.
//
// MI355X, us, weights cold, 64 rows (27 rows), library or split-k kernel, with SwiGLU and norm
// kernels, -> this; q/k/v, gate/up with the SwiGLU, output and down with the norm that adds their
// partial sums:
//   1B  12.2 -> 8.2, 20.9 -> 17.7, 10.2 -> 9.5, 18.0 -> 14.5 (19.5 -> 15.8 gate/up scaled; down 14.5 -> 12.1)
//   3B  17.2 -> 13.5, 26.5 -> 23.7, 16.6 -> 13.5, 23.4 -> 19.5 (24.3 -> 21.1; down 20.0 -> 16.1)
//   8B  18.4 -> 17.1, 55.9 -> 53.3, 18.1 -> 15.0, 42.6 -> 30.0 (16.4 -> 13.2, 56.3 -> 41.8, 14.8 -> 12.9, 34.7 -> 25.4)
#include "common.h"
#include "gemm_stream.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int kWaves = 4;
constexpr int kBK = 128;                   // k of a stage: 256 bytes a row

template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void barrier() { asm volatile("s_barrier" ::: "memory"); }

// What the last of a tile's slices to finish does with their sum (JOINS).
struct RowsJoin {
  float* resid;           // (T,N): the sum is added to it
  const void* weight;     // (N) the next norm's, bfloat16 or float32
  bf16_t* xw;             // (T,N): resid times the weight
  float* ss;              // (T, ss_stride): a tile's sums of resid squared
  unsigned* arrivals;     // one a tile, zero before and after
  int ss_stride, weight_f32, round_sum;
};

struct RowsArgs {
  const bf16_t* X;
  const bf16_t* W;
  void* Y;
  int T, N, steps, tiles; // N: output columns; steps: stages of a tile (of its slice of k)
  int ldx, ldw;           // elements
  int grid;               // workgroups a slice
  long long ldy, slice_stride;
  const float* ss;        // scaled: (T, ss_stride) partial sums of squares, ss_count a row
  int ss_count, ss_stride;
  float eps;
};

struct RowsJoinArgs : RowsArgs {
  RowsJoin join;
};
template <bool JOINS>
using ArgsOf = std::conditional_t<JOINS, RowsJoinArgs, RowsArgs>;

// Sums that workgroups of one launch hand to each other, 16 bytes at a time, past the caches that only one die
// sees (device scope: what an atomic of that scope does, see attention_mfma.hip).
constexpr int kDeviceScope = 16;           // (sc1)

// The sum of a tile's slices joins the residual, and the rows that the next product reads are made of it.
// Slices are added in order and, with round_sum, rounded once to bfloat16: the floats of the norm kernel that
// adds a stack of partial sums (elementwise.hip).
template <int NI>
__device__ __forceinline__ void join_tile(const RowsArgs& p, const RowsJoin& j, int slices, int tile) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int LANES = 4 * NI;            // lanes a row, four columns each
  const auto parts = __builtin_amdgcn_make_buffer_rsrc(p.Y, 0, 0xffffffff, 0x00027000);
  const int c = threadIdx.x % LANES * 4, n = tile * 16 * NI + c;
  const bool inside = n < p.N;
  f32x4 weight{0.f, 0.f, 0.f, 0.f};        // (one by one: the norm's weight lies where its model has it)
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (inside) weight[e] = j.weight_f32 ? ((const float*)j.weight)[n + e] : bf16_to_f32(((const bf16_t*)j.weight)[n + e]);
  constexpr int kRows = kWaves * 64 / LANES;     // rows at a time
  for (int t0 = 0; t0 < p.T; t0 += kRows) {
    const int token = t0 + threadIdx.x / LANES;
    const bool live = inside && token < p.T;
    const long long at = live ? (long long)token * p.ldy + n : 0;
    f32x4 part[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const long long from = at + (q < slices ? q : 0) * p.slice_stride;
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(parts, (int)(from * 4), 0, kDeviceScope);
      part[q] = __builtin_bit_cast(f32x4, v);
    }
    f32x4 r = *(const f32x4*)(j.resid + (live ? (long long)token * p.N + n : 0));
    float squares = 0.f;
    uint32_t o[2];
    float scaled[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float sum = part[0][e];
#pragma unroll
      for (int q = 1; q < 4; ++q) sum = q < slices ? sum + part[q][e] : sum;
      if (j.round_sum) sum = bf16_to_f32(f32_to_bf16(sum));
      r[e] += sum;
      squares += r[e] * r[e];
      scaled[e] = r[e] * weight[e];
    }
    o[0] = f32_to_bf16(scaled[0]) | (uint32_t)f32_to_bf16(scaled[1]) << 16;
    o[1] = f32_to_bf16(scaled[2]) | (uint32_t)f32_to_bf16(scaled[3]) << 16;
    if (!live) squares = 0.f;
#pragma unroll
    for (int d = 1; d < LANES; d *= 2) squares += __shfl_xor(squares, d, 64);
    if (live) {
      *(f32x4*)(j.resid + (long long)token * p.N + n) = r;
      *(uint2*)(j.xw + (long long)token * p.N + n) = make_uint2(o[0], o[1]);
      if (c == 0) j.ss[(long long)token * j.ss_stride + tile] = squares;
    }
  }
#endif
}

// MI groups of 16 rows of x, NI groups of 16 weight rows, BUFS stages in LDS.
template <int MI, int NI, int BUFS, bool SCALED, bool GATED, bool NT, bool JOINS, typename TY, typename Args>
__global__ __launch_bounds__(kWaves * 64) void gemm_rows_kernel(const Args p) {
#ifdef __HIP_DEVICE_COMPILE__   // (the host pass knows no buffer resources)
  constexpr int ROWS = 16 * (MI + NI), STAGE = ROWS * kBK * 2;
  constexpr int PER = MI + NI;             // load instructions of a wave and stage, 4 rows each
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  // sums of a tile's blocks, kRound of them at a time, by wave: [kWaves][kRound][64]
  constexpr int kRound = NI * MI < 8 ? NI * MI : 8;
  f32x4* red = (f32x4*)(smem + BUFS * STAGE);
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int r = lane % 16, g = lane / 16;
  const long long k_slice = (long long)blockIdx.y * p.steps * kBK;

  // instruction i of this wave brings rows (i * 4 + wave) * 4 .. + 3 of a stage, x rows first
  uint32_t src[PER];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int row = (i * kWaves + wave) * 4 + g;
    src[i] = ((uint32_t)min(row, p.T - 1) * p.ldx + (uint32_t)((r ^ (row & 15)) * 8)) * 2;
  }
  const auto weight_rows = [&](int tile) {
#pragma unroll
    for (int i = MI; i < PER; ++i) {
      const int row = ((i - MI) * kWaves + wave) * 4 + g;
      int n;
      if (GATED) {
        // a group of 16: 8 gate rows and the 8 up rows of the same columns
        n = min(tile * 8 * NI + row / 16 * 8 + row % 8, p.N - 1) + (row % 16 < 8 ? 0 : p.N);
      } else {
        n = min(tile * 16 * NI + row, p.N - 1);
      }
      src[i] = ((uint32_t)n * p.ldw + (uint32_t)((r ^ (row & 15)) * 8)) * 2;
    }
  };
  const auto first = [&](int tile) { return (int)((uint32_t)(tile + blockIdx.y) % (uint32_t)p.steps); };
  int a_left = p.steps, a_tile = blockIdx.x, a_buf = 0, a_step = first(a_tile);
  // x and W end 16 bytes below 4 GB at most.  Past the last tile nothing is read: a buffer of no bytes gives zeros
  // without asking memory.  (All ones or none, chosen at each load, went through the vector unit: 64 rows of 512 x 1,024 in
  // two slices 3.9 -> 4.2 us.)
  constexpr uint32_t kWhole = 0xfffffff0u;
  uint32_t a_bytes = kWhole;
  const auto ask = [&]() {
    const auto xr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.X + k_slice), 0, a_bytes, 0x00027000);
    const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.W + k_slice), 0, a_bytes, 0x00027000);
    unsigned char* base = smem + a_buf * STAGE;
    const int at = a_step * kBK * 2;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (i < MI)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)(base + (i * kWaves + wave) * 1024), 16,
                                                 src[i], at, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_ptr)(base + (i * kWaves + wave) * 1024), 16,
                                                 src[i], at, 0, NT ? 2 : 0);
    }
    a_buf = a_buf + 1 == BUFS ? 0 : a_buf + 1;
    a_step = a_step + 1 == p.steps ? 0 : a_step + 1;
    if (--a_left == 0) {
      a_left = p.steps;
      a_tile += p.grid;
      a_bytes = a_tile < p.tiles ? kWhole : 0;
      a_step = first(a_tile);
      weight_rows(a_tile);
    }
  };
  // The rows' sums of squares, a quarter of a row's partial sums per lane: the first 64 are asked for in front of the
  // stages, behind which they would be waited for.
  constexpr int kFirst = 4;
  f32x4 first_sums[SCALED ? kFirst : 1];
  const int ss_token = threadIdx.x / 4, ss_q = threadIdx.x % 4;
  const float* ss_row = SCALED ? p.ss + (long long)min(ss_token, p.T - 1) * p.ss_stride : nullptr;
  if (SCALED) {
#pragma unroll
    for (int k = 0; k < kFirst; ++k) first_sums[k] = *(const f32x4*)(ss_row + min(ss_q * 4 + 16 * k, (p.ss_count - 1) & ~3));
    __builtin_amdgcn_sched_barrier(0);
  }
  weight_rows(a_tile);
#pragma unroll
  for (int s = 0; s < BUFS - 1; ++s) ask();

  if (SCALED) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < kFirst; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) s += ss_q * 4 + 16 * k + e < p.ss_count ? first_sums[k][e] : 0.f;
    for (int i = ss_q * 4 + 16 * kFirst; i < p.ss_count; i += 16) {
      const f32x4 v = *(const f32x4*)(ss_row + i);
#pragma unroll
      for (int e = 0; e < 4; ++e) s += i + e < p.ss_count ? v[e] : 0.f;
    }
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    if (ss_token < 16 * MI && ss_q == 0)
      ((float*)red)[ss_token] = rsqrtf(s / (float)(p.steps * kBK) + p.eps);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();                             // (the stages stay under way)
  }
  // (a wave stores the rows of one group of x: blocks are dealt out in fours, MI is 2 or 4)
  static_assert(MI == 2 || MI == 4, "");
  const int token = wave % MI * 16 + r;
  const bool live = token < p.T;
  const float scale = SCALED ? ((float*)red)[token] : 1.f;

  int buf = 0;
  for (int tile = blockIdx.x; tile < p.tiles; tile += p.grid) {
    f32x4 acc[NI][MI];
#pragma unroll
    for (int a = 0; a < NI; ++a)
#pragma unroll
      for (int m = 0; m < MI; ++m) acc[a][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int step = 0; step < p.steps; ++step) {
      wait_loads<PER*(BUFS - 2)>();
      barrier();                           // the stage is whole; the one before it is free
      // each wave multiplies a quarter of the stage's k
      const unsigned char* base = smem + buf * STAGE + r * 256 + (((wave * 4 + g) ^ r) * 16);
      bf16x8 x[MI], w[NI];
#pragma unroll
      for (int a = 0; a < NI; ++a) w[a] = *(const bf16x8*)(base + (MI + a) * 16 * 256);
#pragma unroll
      for (int m = 0; m < MI; ++m) x[m] = *(const bf16x8*)(base + m * 16 * 256);
      __builtin_amdgcn_sched_barrier(0);
      ask();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < NI; ++a)
#pragma unroll
        for (int m = 0; m < MI; ++m)
          acc[a][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[a], x[m], acc[a][m], 0, 0, 0);
      buf = buf + 1 == BUFS ? 0 : buf + 1;
    }
#pragma unroll
    for (int round = 0; round < NI * MI / kRound; ++round) {
      __syncthreads();                     // whoever still reads the sums before is done
#pragma unroll
      for (int b = 0; b < kRound; ++b)
        red[(wave * kRound + b) * 64 + lane] = acc[(round * kRound + b) / MI][(round * kRound + b) % MI];
      __syncthreads();
#pragma unroll
      for (int b0 = 0; b0 < kRound; b0 += kWaves) {
        if (kRound < kWaves && wave >= kRound) break;
        const int b = b0 + wave;
        const int a = (round * kRound + b) / MI;
        f32x4 v = red[b * 64 + lane];
#pragma unroll
        for (int q = 1; q < kWaves; ++q) v += red[(q * kRound + b) * 64 + lane];
        if (SCALED) v *= scale;
        if (GATED) {
          // lanes below 32 hold gates of four columns, lane + 32 the ups of the same: the lower
          // takes the first two columns, the upper the last two (half of the exponentials each)
          float o[2];
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const float other = __shfl_xor(lane < 32 ? v[2 + i] : v[i], 32, 64);
            o[i] = gated_result(lane < 32 ? v[i] : other, lane < 32 ? other : v[2 + i], 0);
          }
          const int n = tile * 8 * NI + a * 8 + (g & 1) * 4 + (g >> 1) * 2;
          if (live && n < p.N)
            *(uint32_t*)((bf16_t*)p.Y + (long long)token * p.ldy + n) =
                f32_to_bf16(o[0]) | (uint32_t)f32_to_bf16(o[1]) << 16;
          continue;
        }
        const int n = tile * 16 * NI + a * 16 + 4 * g;
        if (!live || n >= p.N) continue;
        if constexpr (JOINS) {
          const auto parts = __builtin_amdgcn_make_buffer_rsrc(p.Y, 0, 0xffffffff, 0x00027000);
          const long long to = blockIdx.y * p.slice_stride + (long long)token * p.ldy + n;
          typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), parts, (int)(to * 4), 0, kDeviceScope);
        } else if (sizeof(TY) == 4) {
          *(f32x4*)((float*)p.Y + blockIdx.y * p.slice_stride + (long long)token * p.ldy + n) = v;
        } else {
          uint2 o;
          o.x = f32_to_bf16(v[0]) | (uint32_t)f32_to_bf16(v[1]) << 16;
          o.y = f32_to_bf16(v[2]) | (uint32_t)f32_to_bf16(v[3]) << 16;
          *(uint2*)((bf16_t*)p.Y + (long long)token * p.ldy + n) = o;
        }
      }
    }
    if constexpr (JOINS) {
      // The last of the tile's slices to get here joins them: everybody's stores have arrived before it is counted in.
      int& last = *(int*)red;              // (behind the barrier nobody reads sums)
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (threadIdx.x == 0) {
        unsigned* slot = p.join.arrivals + tile;
        const bool end = __hip_atomic_fetch_add(slot, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.y - 1;
        last = end;
        if (end) __hip_atomic_store(slot, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      if (last) join_tile<NI>(p, p.join, gridDim.y, tile);
    }
  }
  wait_loads<0>();                         // (loads past the last tile still write LDS)
#endif
}

template <int MI, int NI, int BUFS, bool SCALED, bool GATED, bool NT, bool JOINS, typename TY>
int launch_form(ArgsOf<JOINS> a, int slices, hipStream_t stream) {
  static LdsGrant grant;
  constexpr int bytes = BUFS * 16 * (MI + NI) * kBK * 2 + kWaves * (NI * MI < 8 ? NI * MI : 8) * 1024;
  static_assert(bytes <= 160 * 1024, "");
  const auto kernel = gemm_rows_kernel<MI, NI, BUFS, SCALED, GATED, NT, JOINS, TY, ArgsOf<JOINS>>;
  const hipError_t e = grant_lds(grant, (const void*)kernel, bytes);
  RLIS_REQUIRE(e == hipSuccess, "gemm_rows: %s", hipGetErrorString(e));
  a.tiles = ceil_div(a.N, (GATED ? 8 : 16) * NI);
  const int cus = rlis_stream_compute_units();
  RLIS_REQUIRE(cus > 0, "gemm_rows: cannot read the device properties");
  a.grid = std::min(a.tiles, cus);
  kernel<<<dim3(a.grid, slices), kWaves * 64, bytes, stream>>>(a);
  return 0;
}

template <int MI, int NI, int BUFS, bool SCALED, bool GATED, typename TY, bool JOINS = false>
int launch(const ArgsOf<JOINS>& a, int slices, int nt, hipStream_t stream) {
  return nt ? launch_form<MI, NI, BUFS, SCALED, GATED, true, JOINS, TY>(a, slices, stream)
            : launch_form<MI, NI, BUFS, SCALED, GATED, false, JOINS, TY>(a, slices, stream);
}

// out: 0 bfloat16, 1 float32 (slices of k, slice_stride apart), 2 gated
template <int MI, int NI, int BUFS>
int form(const RowsArgs& a, int out, int slices, int nt, hipStream_t stream) {
  if (a.ss) {
    if (out == 0) return launch<MI, NI, BUFS, true, false, bf16_t>(a, slices, nt, stream);
    if (out == 1) return launch<MI, NI, BUFS, true, false, float>(a, slices, nt, stream);
    return launch<MI, NI, BUFS, true, true, bf16_t>(a, slices, nt, stream);
  }
  if (out == 0) return launch<MI, NI, BUFS, false, false, bf16_t>(a, slices, nt, stream);
  if (out == 1) return launch<MI, NI, BUFS, false, false, float>(a, slices, nt, stream);
  return launch<MI, NI, BUFS, false, true, bf16_t>(a, slices, nt, stream);
}

// Groups of 16 weight rows a tile, and slices of k (all of 1, 2, 4) of a product with partial
// sums.  Small tiles read x more often, so: the smallest that leave no compute unit a second one
// (q/k/v of the 1B shape at 64 rows with 1 / 2 / 4 groups: 8.2 / 9.5 / 12.6 us; of the 3B shape
// 18.8 / 13.5 / 17.8; gate/up 28 / 21 / 18).  Four slices are best at every shape where the
// product is small enough (down at 64 rows, norm included, 2 / 4 / 8 slices at the best tile: 1B
// 17.4 / 14.5 / 14.7, 3B 22.9 / 19.5 / 22.7, 8B 33.6 / 30.0 / 37.2).
constexpr int kUnits = 256;                // compute units of the chip
int row_groups(int rows, int slices) {
  for (int ni = 1; ni < 4; ni *= 2)
    if ((long long)ceil_div(rows, 16 * ni) * slices <= kUnits) return ni;
  return 4;
}
int slices_of(int N, int K) {
  const int steps = K / kBK;
  int s = 4;
  while (s > 1 && (steps % s || steps / s < 4 || ceil_div(N, 64) * s > kUnits)) s /= 2;
  return s;
}

int dispatch(const RowsArgs& a, int out, int slices, int nt, hipStream_t stream) {
  const int ni = row_groups(out == 2 ? 2 * a.N : a.N, slices);
  int rc;
  if (a.T <= 32) {
    rc = ni == 1 ? form<2, 1, 8>(a, out, slices, nt, stream) : ni == 2 ? form<2, 2, 8>(a, out, slices, nt, stream)
                                                                   : form<2, 4, 5>(a, out, slices, nt, stream);
  } else {
    rc = ni == 1 ? form<4, 1, 6>(a, out, slices, nt, stream) : ni == 2 ? form<4, 2, 5>(a, out, slices, nt, stream)
                                                                   : form<4, 4, 4>(a, out, slices, nt, stream);
  }
  if (rc) return rc;
  RLIS_LAUNCH_CHECK("gemm_rows");
  return 0;
}

int dispatch_join(const RowsJoinArgs& a, int slices, int nt, hipStream_t stream) {
  const int ni = row_groups(a.N, slices);
  const int rc = ni == 1   ? launch<2, 1, 8, false, false, float, true>(a, slices, nt, stream)
                 : ni == 2 ? launch<2, 2, 8, false, false, float, true>(a, slices, nt, stream)
                           : launch<2, 4, 5, false, false, float, true>(a, slices, nt, stream);
  if (rc) return rc;
  RLIS_LAUNCH_CHECK("gemm_rows_join");
  return 0;
}

}  // namespace

// Slices of k that a product with partial sums comes in (out 1); K a multiple of 128.
RLIS_API int rlis_gemm_bf16_rows_slices(int N, int K) { return slices_of(N, K); }

// Y (T,N) = X (T,K) * W (N,K)^T for up to 64 rows, K a multiple of 128 times the slices, N of 8.
// out 0: bfloat16; 1: float32, `slices` partial results slice_stride elements apart; 2: gated, W
// (2 N,K) gate rows then up rows, Y = silu(gate) * up in bfloat16.  ss: the products of a row are
// scaled by rsqrt(sum of its ss_count partial sums / K + eps).  nt: W is loaded non-temporally
// (load_weights).
RLIS_API int rlis_gemm_bf16_rows(const void* X, const void* W, void* Y, int out, int T, int N, int K,
                                 int slices, long long ldx, long long ldw, long long ldy,
                                 long long slice_stride, const float* ss, int ss_count, int ss_stride,
                                 float eps, int nt, hipStream_t stream) {
  RLIS_REQUIRE(T > 0 && T <= 64 && N > 0 && N % 8 == 0 && slices > 0 && K > 0 && K % (slices * kBK) == 0,
               "gemm_rows: bad sizes T=%d N=%d K=%d slices=%d", T, N, K, slices);
  RLIS_REQUIRE(out >= 0 && out <= 2 && (slices == 1 || (out == 1 && !ss)), "gemm_rows: no such form");
  RLIS_REQUIRE(ldx >= K && ldw >= K && ldy >= N && ldx % 8 == 0 && ldw % 8 == 0 && ldy % 8 == 0 &&
                   slice_stride % 4 == 0 && (uintptr_t)X % 16 == 0 && (uintptr_t)W % 16 == 0 &&
                   (uintptr_t)Y % 16 == 0,
               "gemm_rows: rows must lie on 16-byte boundaries");
  RLIS_REQUIRE(ldx * 2 * T < (1LL << 32) && ldw * 2 * N * (out == 2 ? 2 : 1) < (1LL << 32),
               "gemm_rows: x or W passes 4 GB");
  RLIS_REQUIRE(!ss || (ss_count > 0 && ss_stride >= ss_count && ss_stride % 4 == 0 && (uintptr_t)ss % 16 == 0),
               "gemm_rows: the sums of squares must be rows on 16-byte boundaries");
  const RowsArgs a = {(const bf16_t*)X, (const bf16_t*)W, Y, T, N, K / slices / kBK, 0, (int)ldx, (int)ldw, 0,
                      ldy, slice_stride, ss, ss_count, ss_stride, eps};
  return dispatch(a, out, slices, nt, stream);
}

// Tiles of weight rows of a product with `slices` partial sums: sums of squares a row, and arrival counters.
RLIS_API int rlis_gemm_bf16_rows_join_tiles(int N, int slices) {
  return N > 0 && slices > 0 ? ceil_div(N, 16 * row_groups(N, slices)) : 0;
}

// resid (T,N) += X (T,K) * W (N,K)^T for up to 32 rows over two or four slices of k, the sum of the slices rounded to
// bfloat16 first with round_sum; xw (T,N) = resid * weight in bfloat16, ss (T, ss_stride) the sums of resid squared over
// each of rlis_gemm_bf16_rows_join_tiles(N, slices) tiles of columns.  parts: (slices,T,N) float32 of scratch.  arrivals:
// a counter a tile, all zero before the launch and again after it; launches that overlap in time must not share
// them.  In place of the partial sums and the norm that adds them: down of the 3B shape at 27 rows in a step 11.6 + 4.8 ->
// 15.6 us, and the q/k/v product behind it, scaled here, 12.6 -> 10.8.  At 64 rows of the 1B shape output and down got 3.5
// us slower for a norm of 5.0 less, the scaled gate/up and q/k/v took 1.2 us more, and the step as a whole 1 %
// more.
RLIS_API int rlis_gemm_bf16_rows_join(const void* X, const void* W, float* parts, int T, int N, int K, int slices,
                                      long long ldx, long long ldw, float* resid, const void* weight, int weight_dtype,
                                      int round_sum, void* xw, float* ss, int ss_stride, unsigned* arrivals, int arrival_slots,
                                      int nt, hipStream_t stream) {
  RLIS_REQUIRE(T > 0 && T <= 32 && N > 0 && N % 8 == 0 && (slices == 2 || slices == 4) && K > 0 && K % (slices * kBK) == 0,
               "gemm_rows_join: bad sizes T=%d N=%d K=%d slices=%d", T, N, K, slices);
  const int tiles = rlis_gemm_bf16_rows_join_tiles(N, slices);
  RLIS_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0 && (uintptr_t)X % 16 == 0 && (uintptr_t)W % 16 == 0 &&
                   (uintptr_t)parts % 16 == 0 && (uintptr_t)resid % 16 == 0 && (uintptr_t)xw % 16 == 0,
               "gemm_rows_join: rows must lie on 16-byte boundaries");
  RLIS_REQUIRE(parts && resid && weight && xw && ss && ss_stride >= tiles && arrivals && arrival_slots >= tiles,
               "gemm_rows_join: an operand is missing or too short for %d tiles", tiles);
  RLIS_REQUIRE(weight_dtype == RLIS_F32 || weight_dtype == RLIS_BF16, "gemm_rows_join: unknown weight dtype %d", weight_dtype);
  RLIS_REQUIRE(ldx * 2 * T < (1LL << 32) && ldw * 2 * N < (1LL << 32) && 4LL * slices * T * N < (1LL << 31),
               "gemm_rows_join: x or W passes 4 GB, or the partial sums 2 GB");
  const RowsJoinArgs a = {{(const bf16_t*)X, (const bf16_t*)W, parts, T, N, K / slices / kBK, 0, (int)ldx, (int)ldw, 0,
                           N, (long long)T * N, nullptr, 0, 0, 0.f},
                          {resid, weight, (bf16_t*)xw, ss, arrivals, ss_stride, weight_dtype == RLIS_F32, round_sum}};
  return dispatch_join(a, slices, nt, stream);
}
