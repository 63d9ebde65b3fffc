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
// non-temporally (64 rows, gate/up with the SwiGLU, 1B: 20.1 -> 19.0 us; 32 rows, 8B: 52 -> 46).
// The order of a sum follows from N and K alone: a row's bits do not depend on the rows beside it.
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

#include <algorithm>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int kWaves = 4;
constexpr int kBK = 128;                   // k of a stage: 256 bytes a row

template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void barrier() { asm volatile("s_barrier" ::: "memory"); }

struct RowsArgs {
  const bf16_t* X;
  const bf16_t* W;
  void* Y;
  int T, N, steps, tiles; // N: output columns; steps: stages of a tile (of its slice of k)
  int ldx, ldw;           // elements
  long long ldy, slice_stride;
  const float* ss;        // scaled: (T, ss_stride) partial sums of squares, ss_count a row
  int ss_count, ss_stride;
  float eps;
};

// MI groups of 16 rows of x, NI groups of 16 weight rows, BUFS stages in LDS.
template <int MI, int NI, int BUFS, bool SCALED, bool GATED, typename TY>
__global__ __launch_bounds__(kWaves * 64) void gemm_rows_kernel(const RowsArgs p) {
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

  const auto xr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.X + k_slice), 0, 0xffffffff, 0x00027000);
  const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.W + k_slice), 0, 0xffffffff, 0x00027000);
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
  const auto ask = [&]() {
    unsigned char* base = smem + a_buf * STAGE;
    const int at = a_step * kBK * 2;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (i < MI)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)(base + (i * kWaves + wave) * 1024), 16,
                                                 src[i], at, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_ptr)(base + (i * kWaves + wave) * 1024), 16,
                                                 src[i], at, 0, 2);
    }
    a_buf = a_buf + 1 == BUFS ? 0 : a_buf + 1;
    a_step = a_step + 1 == p.steps ? 0 : a_step + 1;
    if (--a_left == 0) {
      // (past the last tile its last row is read again)
      a_left = p.steps;
      a_tile += gridDim.x;
      a_step = first(a_tile);
      weight_rows(a_tile);
    }
  };
  weight_rows(a_tile);
#pragma unroll
  for (int s = 0; s < BUFS - 1; ++s) ask();

  if (SCALED) {
    // the rows' sums of squares, a quarter of a row's partial sums per lane
    const int token = threadIdx.x / 4, q = threadIdx.x % 4;
    float s = 0.f;
    if (token < 16 * MI) {
      const float* row = p.ss + (long long)min(token, p.T - 1) * p.ss_stride;
      for (int i = q * 4; i < p.ss_count; i += 16) {
        const f32x4 v = *(const f32x4*)(row + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) s += i + e < p.ss_count ? v[e] : 0.f;
      }
    }
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    if (token < 16 * MI && q == 0)
      ((float*)red)[token] = rsqrtf(s / (float)(p.steps * kBK) + p.eps);
    __syncthreads();
  }
  // (a wave stores the rows of one group of x: blocks are dealt out in fours, MI is 2 or 4)
  static_assert(MI == 2 || MI == 4, "");
  const int token = wave % MI * 16 + r;
  const bool live = token < p.T;
  const float scale = SCALED ? ((float*)red)[token] : 1.f;

  int buf = 0;
  for (int tile = blockIdx.x; tile < p.tiles; tile += gridDim.x) {
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
          // lanes below 32 hold gates of four columns, lane + 32 the ups of the same
          float o[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float other = __shfl_xor(v[i], 32, 64);
            const float gt = lane < 32 ? v[i] : other, up = lane < 32 ? other : v[i];
            const float e = __builtin_amdgcn_exp2f(gt * -1.4426950408889634f);
            o[i] = gt * __builtin_amdgcn_rcpf(1.0f + e) * up;
          }
          const int n = tile * 8 * NI + a * 8 + (g & 1) * 4 + (g >> 1) * 2;
          if (live && n < p.N)
            *(uint32_t*)((bf16_t*)p.Y + (long long)token * p.ldy + n) =
                g >> 1 ? f32_to_bf16(o[2]) | (uint32_t)f32_to_bf16(o[3]) << 16
                       : f32_to_bf16(o[0]) | (uint32_t)f32_to_bf16(o[1]) << 16;
          continue;
        }
        const int n = tile * 16 * NI + a * 16 + 4 * g;
        if (!live || n >= p.N) continue;
        if (sizeof(TY) == 4) {
          *(f32x4*)((float*)p.Y + blockIdx.y * p.slice_stride + (long long)token * p.ldy + n) = v;
        } else {
          uint2 o;
          o.x = f32_to_bf16(v[0]) | (uint32_t)f32_to_bf16(v[1]) << 16;
          o.y = f32_to_bf16(v[2]) | (uint32_t)f32_to_bf16(v[3]) << 16;
          *(uint2*)((bf16_t*)p.Y + (long long)token * p.ldy + n) = o;
        }
      }
    }
  }
  wait_loads<0>();                         // (loads past the last tile still write LDS)
#endif
}

int compute_units() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return n;
}

template <int MI, int NI, int BUFS, bool SCALED, bool GATED, typename TY>
int launch(const RowsArgs& a, int slices, hipStream_t stream) {
  static LdsGrant grant;
  constexpr int bytes = BUFS * 16 * (MI + NI) * kBK * 2 + kWaves * (NI * MI < 8 ? NI * MI : 8) * 1024;
  static_assert(bytes <= 160 * 1024, "");
  const auto kernel = gemm_rows_kernel<MI, NI, BUFS, SCALED, GATED, TY>;
  const hipError_t e = grant_lds(grant, (const void*)kernel, bytes);
  RLIS_REQUIRE(e == hipSuccess, "gemm_rows: %s", hipGetErrorString(e));
  RowsArgs b = a;
  b.tiles = ceil_div(a.N, (GATED ? 8 : 16) * NI);
  const int cus = compute_units();
  RLIS_REQUIRE(cus > 0, "gemm_rows: cannot read the device properties");
  kernel<<<dim3(std::min(b.tiles, cus), slices), kWaves * 64, bytes, stream>>>(b);
  return 0;
}

// out: 0 bfloat16, 1 float32 (slices of k, slice_stride apart), 2 gated
template <int MI, int NI, int BUFS>
int form(const RowsArgs& a, int out, int slices, hipStream_t stream) {
  if (a.ss) {
    if (out == 0) return launch<MI, NI, BUFS, true, false, bf16_t>(a, slices, stream);
    if (out == 1) return launch<MI, NI, BUFS, true, false, float>(a, slices, stream);
    return launch<MI, NI, BUFS, true, true, bf16_t>(a, slices, stream);
  }
  if (out == 0) return launch<MI, NI, BUFS, false, false, bf16_t>(a, slices, stream);
  if (out == 1) return launch<MI, NI, BUFS, false, false, float>(a, slices, stream);
  return launch<MI, NI, BUFS, false, true, bf16_t>(a, slices, stream);
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

}  // namespace

// Slices of k that a product with partial sums comes in (out 1); K a multiple of 128.
RLIS_API int rlis_gemm_bf16_rows_slices(int N, int K) { return slices_of(N, K); }

// Y (T,N) = X (T,K) * W (N,K)^T for up to 64 rows, K a multiple of 128 times the slices, N of 8.
// out 0: bfloat16; 1: float32, `slices` partial results slice_stride elements apart; 2: gated, W
// (2 N,K) gate rows then up rows, Y = silu(gate) * up in bfloat16.  ss: the products of a row are
// scaled by rsqrt(sum of its ss_count partial sums / K + eps).
RLIS_API int rlis_gemm_bf16_rows(const void* X, const void* W, void* Y, int out, int T, int N, int K,
                                 int slices, long long ldx, long long ldw, long long ldy,
                                 long long slice_stride, const float* ss, int ss_count, int ss_stride,
                                 float eps, hipStream_t stream) {
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
  const RowsArgs a = {(const bf16_t*)X, (const bf16_t*)W, Y, T, N, K / slices / kBK, 0, (int)ldx, (int)ldw,
                      ldy, slice_stride, ss, ss_count, ss_stride, eps};
  const int ni = row_groups(out == 2 ? 2 * N : N, slices);
  int rc;
  if (T <= 32) {
    rc = ni == 1 ? form<2, 1, 8>(a, out, slices, stream) : ni == 2 ? form<2, 2, 8>(a, out, slices, stream)
                                                                   : form<2, 4, 5>(a, out, slices, stream);
  } else {
    rc = ni == 1 ? form<4, 1, 6>(a, out, slices, stream) : ni == 2 ? form<4, 2, 5>(a, out, slices, stream)
                                                                   : form<4, 4, 4>(a, out, slices, stream);
  }
  if (rc) return rc;
  RLIS_LAUNCH_CHECK("gemm_rows");
  return 0;
}
