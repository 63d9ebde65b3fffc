// bfloat16 products y = x * W^T of more than 64 rows of x (portions of prompts; of 33 on over many weight
// rows), on the matrix cores.
//
// At these sizes what bounds a product is how fast a compute unit is fed, not the matrix cores: every
// tile brings its rows of x and of W into LDS once per stage of 64 k (buffer_load ... lds, 128 bytes a
// row), and what a die's 32 units ask for while a line is still on its way from memory is served at
// about 60 bytes a nanosecond and unit, against 135 for lines that its L2 holds already (reads alone,
// eight units to a line; the same with 32 or 160 KB under way).  So a tile starts its walk over k a
// stage behind its neighbour along W: each line of x is asked for by one of them and found by the others.
// Tiles along x start at the same stage, so that the order of a row's sum does not depend on where in x
// the row lies; two stages apart as well, lines of W would be found likewise (512 rows of the 1B shape, us:
// output with its norm 16.1 for 16.7, gate/up 37.9 for 36.6; 1,024 x 1,024 x 2,048 10.1 for 12.1), and two equal prompts
// of a step would differ in their last bits.  Ids go round the dies and each die takes a run of tiles,
// eight along x for each along W, so that those that share a line share an L2.
//
// Each wave holds MI x NI blocks of 16 x 16 (v_mfma_f32_16x16x32_bf16).  One barrier a stage, in its
// middle: behind it the stage to come is whole and the one before it free.  Reads of the next half
// stage and loads of a later stage stand one by one between the products: issued in a row, a stage's
// loads alone hold a wave for as long as its products take (512 x 3,072 x 2,048 in 128 x 128: 19 us,
// then 16).  Piece c (16 bytes) of row r of a stage lies at c ^ (r / 2 % 8), which the load does by
// choosing what a lane reads, so that fragments are read without bank conflicts.  Which weight rows
// a group of 16 holds is chosen so that a lane stores 16 bytes of neighbouring columns; gated, gate
// and up rows of the same columns lie in turn and a lane holds both.
//
// The order of a sum follows from the sizes and from where in W the tile lies.
//
// 33 to 64 rows take it too where there is much of W (gate/up, the output head): one row of tiles, each
// line of W read once and non-temporally.  64 rows, us: head 1B 117 (library) -> 88, 3B 164 -> 130; gate/up
// against gemm_rows.hip 1B 16.4 -> 15.0, 3B 22.5 -> 22.1, 8B 50.0 -> 42.6.
//
// q, k and v (kOutHeads): the weight rows of dims j and j + d / 2 of a head lie in turn like gate and up, so a lane
// holds both halves of what a rotation turns; it turns the keys and stores keys and values to the cache's pages, and
// the queries stay as they are for the attention kernels to turn.  In place of the library's product and a pass of
// 6 to 8 us over its rows (elementwise.hip); weights cold, us: 1B 128 / 512 / 1,024 / 2,048 rows 16.3 -> 10.5, 21.8 ->
// 16.8, 27.7 -> 23.9, 36.8 -> 34.7; 3B 24.3 -> 19.5, 32.7 -> 33.1, 46.2 -> 42.0, - ; 8B 29.2 -> 23.9, 42.9 -> 39.1, 59.6
// -> 57.3, - .  Tiles 96 wide make even rounds of 3,072 and 6,144 weight rows.  Values are stored two bytes
// at a time, sixteen tokens side by side: the tiles that hold them end a microsecond later than the others.
//
// 256 x 256 has the most operations to a byte that is fed (the accumulators fill half of a wave's registers).
//
// Tiles of 128 to 256 rows by 128, in steps of 32, so that a round comes out even over the compute units
// (gate/up of the 1B shape at 381 rows in a step: two of 192 31.3 us, three of 128 35.4, the library's with
// the SwiGLU kernel 36.7).  More stages under way than the tiles have here change nothing.
//
// MI355X, us, weights cold, the library's product, tried out (with SwiGLU kernel; with the norm that adds
// output's and down's partial sums) -> this, at 96 / 256 / 512 rows (-: the library's):
//   1B  q/k/v 13.0 -> 12.0, 14.1 -> 12.7, -               output 15.6 -> 10.4, 16.1 -> 13.2, 18.0 -> 16.7
//       gate/up 23.5 -> 20.0, 31.3 -> 27.1, 42.2 -> 36.6  down 16.3 -> 16.0, 24.8 -> 23.2, 33.0 -> 31.6
//   3B  q/k/v -, at 112 rows 19.1 -> 17.4                 output 17.9 -> 14.3, 21.7 -> 22.5, 27.4 -> 27.6
//       gate/up 30.4 -> 29.5, 41.8 -> 40.1, 60.7 -> 51.4  down 22.6 -> 22.0, -, -
//   (gate/up 1,024 / 2,048 / 8,192 rows in 256 x 256: 1B 67.8 -> 61.4, 120.8 -> 115.7, 453 -> 434; 3B 91.8 -> 84.1, 169.3 ->
//   160.7, 635 -> 607; down of 2,048 rows of the 1B shape 76.6 -> 75.2)
//   8B  q/k/v 20.6 -> 21.3, at 112 rows 25.9 -> 22.2      output 20.8 -> 16.6, 26.1 -> 26.9, 36.7 -> 32.9
//       gate/up 62.2 -> 55.4, 77.1 -> 70.2, -             down 36.0 -> 35.2, 47.6 -> 46.7, 71.4 -> 69.3
// In a step, where a row count between those tried out takes another's algorithm, the library is further behind
// (prompts of 72 / 128 / 200 tokens, twelve layers, us: 1B 1,204 -> 1,037, 1,232 -> 1,099, 1,429 -> 1,248; 8B 2,107 ->
// 1,824, 2,334 -> 2,043, 2,666 -> 2,342).
#include "common.h"
#include "gemm_stream.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int kBK = 64;                    // k of a stage: 128 bytes a row

// Waits until at most N loads from memory, and no read from LDS, are under way.  The builtin, so that
// the compiler, which places waits of its own before a fragment is used, knows that it has arrived.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | 7 << 4 | 0 << 8 | (N >> 4) << 14);
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void barrier() { asm volatile("s_barrier" ::: "memory"); }

// The step's q, k and v rows on their way out (kOutHeads): q as it is, k turned by its position and v into
// the cache's pages.
struct HeadsArgs {
  const float* cos;        // (positions, d / 2) float32; null: nothing is turned
  const float* sin;
  const int* positions;    // (T)
  const int* slots;        // (T) page * page size + offset; below 0: not stored
  bf16_t* k_pages;         // (pages, nkv, page size, d)
  bf16_t* v_pages;         // (pages, nkv, d, page size)
  int nh, nkv, half_shift, page_shift;   // d / 2 and the page size are powers of two
};

struct TilesArgs {
  const bf16_t* X;
  const bf16_t* W;
  void* Y;
  int T, N, steps;         // N: output columns; steps: stages of a slice of k
  int mt, nt, slices;      // tiles along x's rows and W's, slices of k
  int group;               // tiles of x's rows that are walked together
  int ldx, ldw;            // elements
  int grid;                // workgroups
  long long ldy, slice_stride;
};

// (apart: handed to every kernel they made 1,024 x 1,024 products of 4.8 us 0.25 us longer)
struct HeadsTilesArgs : TilesArgs {
  HeadsArgs heads;
};

// (kOutGated, kOutHeads: N counts pairs of weight rows whose products meet in a lane)
enum { kOutBf16 = 0, kOutF32 = 1, kOutGated = 2, kOutHeads = 3 };
constexpr bool in_pairs(int out) { return out >= kOutGated; }
template <int OUT>
using ArgsOf = std::conditional_t<OUT == kOutHeads, HeadsTilesArgs, TilesArgs>;

// Four or eight neighbouring dims of a head.
template <int Q>
__device__ __forceinline__ void store_dims(bf16_t* to, const float (&v)[4 * Q]) {
  uint32_t o[2 * Q];
#pragma unroll
  for (int i = 0; i < 2 * Q; ++i) o[i] = bf16_pair(v[2 * i], v[2 * i + 1]);
  if (Q == 2) *(uint4*)to = make_uint4(o[0], o[1], o[2 * Q - 2], o[2 * Q - 1]);
  else *(uint2*)to = make_uint2(o[0], o[1]);
}

// The sums that a lane holds of one token: dims j .. and j + d / 2 .. of whichever heads its columns are.
template <int MI, int NI>
__device__ __forceinline__ void store_heads(const HeadsTilesArgs& p, const f32x4 (&acc)[NI][MI], int m, int token,
                                            int first, int g) {
  constexpr int Q = NI % 4 == 0 ? 2 : 1;   // pairs of blocks whose dims are neighbours
  const HeadsArgs& h = p.heads;
  const int half = 1 << h.half_shift, d = 2 * half;
#pragma unroll
  for (int a = 0; a < NI / 2; a += Q) {
    const int n = first + a * 16 + g * 4 * Q;
    if (n >= p.N) continue;
    const int head = n >> h.half_shift, j = n & (half - 1);
    float lo[4 * Q], hi[4 * Q];
#pragma unroll
    for (int e = 0; e < 4 * Q; ++e) {
      lo[e] = acc[2 * (a + e / 4)][m][e % 4];
      hi[e] = acc[2 * (a + e / 4) + 1][m][e % 4];
    }
    if (head < h.nh) {
      bf16_t* to = (bf16_t*)p.Y + (long long)token * p.ldy + head * d + j;
      store_dims<Q>(to, lo);
      store_dims<Q>(to + half, hi);
      continue;
    }
    const int slot = h.slots[token];
    if (slot < 0) continue;
    const long long page = slot >> h.page_shift;
    const int off = slot & ((1 << h.page_shift) - 1);
    if (head < h.nh + h.nkv) {
      bf16_t* to = h.k_pages + (((page * h.nkv + head - h.nh) << h.page_shift) + off) * d + j;
      if (h.cos) {
        const long long at = (long long)h.positions[token] * half + j;
#pragma unroll
        for (int e = 0; e < 4 * Q; e += 4) {
          const f32x4 c = *(const f32x4*)(h.cos + at + e), s = *(const f32x4*)(h.sin + at + e);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            // (the product is rounded first, as one that goes through memory is)
            const float x = bf16_to_f32(f32_to_bf16(lo[e + i])), y = bf16_to_f32(f32_to_bf16(hi[e + i]));
            lo[e + i] = fmaf(x, c[i], -(y * s[i]));
            hi[e + i] = fmaf(y, c[i], x * s[i]);
          }
        }
      }
      store_dims<Q>(to, lo);
      store_dims<Q>(to + half, hi);
    } else {
      bf16_t* to = h.v_pages + ((((page * h.nkv + head - h.nh - h.nkv) * d + j) << h.page_shift) + off);
#pragma unroll
      for (int e = 0; e < 4 * Q; ++e) {
        to[(long long)e << h.page_shift] = f32_to_bf16(lo[e]);
        to[(long long)(e + half) << h.page_shift] = f32_to_bf16(hi[e]);
      }
    }
  }
}

// WM x WN waves, each MI groups of 16 rows of x by NI groups of 16 weight rows; BUFS stages in LDS.
template <int MI, int NI, int WM, int WN, int BUFS, int OUT, bool NT, typename Args>
__global__ __launch_bounds__(WM * WN * 64) void gemm_tiles_kernel(const Args p) {
#ifdef __HIP_DEVICE_COMPILE__   // (the host pass knows no buffer resources)
  constexpr int WAVES = WM * WN, BM = 16 * MI * WM, BN = 16 * NI * WN;
  constexpr int STAGE = (BM + BN) * kBK * 2;
  constexpr int XI = BM / 8 / WAVES, WI = BN / 8 / WAVES, PER = XI + WI;
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "");
  static_assert(NI % 2 == 0, "");
  // The largest tile has room for two stages and a half: its ring is one of quarter stages (half of x's
  // rows, half of W's), ten of them, and a stage's x is asked for half a stage ahead of its W.
  constexpr bool QUARTERS = BUFS == 2 && WAVES == 8;
  static_assert(!QUARTERS || (BM == BN && WM == 2 && WN % 2 == 0), "");
  constexpr int RING = QUARTERS ? STAGE / 2 * 5 : STAGE * BUFS;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int r = lane % 16, g = lane / 16;
  const int wm = wave % WM, wn = wave / WM;

  // Workgroup id -> tile.  Ids go round the eight dies; each die takes a run of the walk.
  const int per_slice = p.mt * p.nt, total = per_slice * p.slices;
  const auto place = [&](int id, int& m0, int& n0, int& slice) {
    id = min(id, total - 1);
    const int die = id & 7, at = id >> 3;
    int lin = die * (total >> 3) + min(die, total & 7) + at;
    slice = lin / per_slice;
    lin -= slice * per_slice;
    const int band = lin / (p.group * p.nt), rows = min(p.group, p.mt - band * p.group);
    lin -= band * p.group * p.nt;
    m0 = (band * p.group + lin % rows) * BM;
    n0 = lin / rows * (in_pairs(OUT) ? BN / 2 : BN);
  };

  // Instruction i of this wave brings rows (i * WAVES + wave) * 8 .. + 7 of a stage, x rows first;
  // piece c of row q of the stage lies at c ^ (q / 2 % 8).
  uint32_t src[PER];
  int a_k = 0, a_from = 0;                 // bytes into a row: the stage to ask for, the slice's start
  const auto sources = [&](int id) {
    int m0, n0, slice;
    place(id, m0, n0, slice);
    const int q8 = lane / 8, c = lane % 8;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int q = (i * WAVES + wave) * 8 + q8;
      src[i] = ((uint32_t)min(m0 + q, p.T - 1) * p.ldx + (uint32_t)((c ^ (q / 2 % 8)) * 8)) * 2;
    }
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int q = (i * WAVES + wave) * 8 + q8;
      const int b = q / 16, o = q % 16;
      int n;
      if (in_pairs(OUT)) {
        // groups of 16 in turn: gate and up rows of the same columns, or dims j and j + d / 2 of a head
        const int pair = b / 2;
        const int col = NI % 4 == 0 ? pair / 2 * 32 + o / 4 * 8 + pair % 2 * 4 + o % 4 : pair * 16 + o;
        n = min(n0 + col, p.N - 1);
        if constexpr (OUT == kOutHeads)
          n += (n >> p.heads.half_shift << p.heads.half_shift) + (b % 2 << p.heads.half_shift);
        else
          n += b % 2 ? p.N : 0;
      } else if (OUT == kOutBf16) {
        // two groups of 16 share 32 columns so that a lane holds eight neighbours
        n = min(n0 + b / 2 * 32 + o / 4 * 8 + b % 2 * 4 + o % 4, p.N - 1);
      } else {
        n = min(n0 + q, p.N - 1);
      }
      src[XI + i] = ((uint32_t)n * p.ldw + (uint32_t)((c ^ (q / 2 % 8)) * 8)) * 2;
    }
    a_from = slice * p.steps * (kBK * 2);
    const int turn = n0 / (in_pairs(OUT) ? BN / 2 : BN);   // (of the weight rows alone)
    a_k = a_from + turn % p.steps * (kBK * 2);
  };
  int a_id = blockIdx.x, a_left = p.steps, a_buf = 0;
  // x and W end 16 bytes below 4 GB at most.  Past the last tile nothing is read: a buffer of no bytes gives zeros
  // without asking memory.  (All ones or none, chosen at each load, went through the vector unit between the products:
  // 2,048 x 2,048 at 512 rows 12.0 -> 12.4 us.)
  constexpr uint32_t kWhole = 0xfffffff0u;
  uint32_t a_bytes = kWhole;
  const auto ask = [&](int i) {
    int at = a_buf;
    if (QUARTERS && i * 4 / PER * (STAGE / 4) + at >= RING) at -= RING;
    const lds_ptr to = (lds_ptr)(smem + at + (i * WAVES + wave) * 1024);
    const auto xr = __builtin_amdgcn_make_buffer_rsrc((void*)p.X, 0, a_bytes, 0x00027000);
    const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)p.W, 0, a_bytes, 0x00027000);
    if (i < XI) __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, to, 16, src[i], a_k, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, to, 16, src[i], a_k, 0, NT ? 2 : 0);
  };
  const auto asked = [&]() {               // the stage has been asked for, on to the next
    a_buf = a_buf + STAGE >= RING ? a_buf + STAGE - RING : a_buf + STAGE;
    a_k += kBK * 2;
    if (a_k == a_from + p.steps * (kBK * 2)) a_k = a_from;
    if (--a_left == 0) {
      a_left = p.steps;
      a_id += p.grid;
      a_bytes = a_id < total ? kWhole : 0;
      sources(a_id);
    }
  };

  // fragments of a half stage (32 k)
  constexpr int X_PART = QUARTERS ? 16 * MI : BM;  // rows of a part of the ring
  const int x_at = (wm * 16 * MI % X_PART + r) * 128 + ((g ^ (r / 2)) * 16);
  const int w_at = ((QUARTERS ? 0 : BM) + wn * 16 * NI % (QUARTERS ? BN / 2 : BN) + r) * 128 + ((g ^ (r / 2)) * 16);
  const int w_part = QUARTERS ? (2 + wn / (WN / 2)) * (STAGE / 4) : 0, x_part = QUARTERS ? wm * (STAGE / 4) : 0;
  int x_buf = x_part, w_buf = w_part;
  const auto onward = [&]() {              // to the next stage's parts
    x_buf = x_buf + STAGE >= RING ? x_buf + STAGE - RING : x_buf + STAGE;
    if (QUARTERS) w_buf = w_buf + STAGE >= RING ? w_buf + STAGE - RING : w_buf + STAGE;
  };
  struct Half {
    bf16x8 x[MI], w[NI];
  };
  const auto read = [&](Half& h, int ks, int i) {
    if (i < MI) h.x[i] = *(const bf16x8*)(smem + x_buf + (x_at ^ (ks * 64)) + i * 2048);
    else h.w[i - MI] = *(const bf16x8*)(smem + (QUARTERS ? w_buf : x_buf) + (w_at ^ (ks * 64)) + (i - MI) * 2048);
  };
  f32x4 acc[NI][MI];
  const auto clear = [&]() {
#pragma unroll
    for (int a = 0; a < NI; ++a)
#pragma unroll
      for (int m = 0; m < MI; ++m) acc[a][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  // The products of one half stage.  Between them, one at a time, so that neither the LDS nor the
  // memory pipe makes a wave wait before its products: the reads of the half stage to come and loads of
  // later stages.
  constexpr int PRODUCTS = NI * MI, READS = MI + NI, LATE = PER / 2;
  const auto half = [&](const Half& h, Half& next, int ks, auto loads) {
#pragma unroll
    for (int j = 0; j < PRODUCTS; ++j) {
      const int a = j / MI, m = j % MI;
      acc[a][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h.w[a], h.x[m], acc[a][m], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < READS; ++i)
        if (i * 3 * PRODUCTS / (READS * 4) == j) read(next, ks, i);
      loads(j);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // loads from .. from + count - 1 of the stage to ask for, spread over `places` products from `first` on
  const auto some = [&](int j, int from, int count, int first, int places) {
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (i < count && first + i * places / count == j) ask(from + i);
  };
  // Beside a stage's earlier half the later loads of the stage that takes the place of the last one,
  // beside its later half the first ones of the next.  In quarters all of a stage beside its later half: the W
  // that the ring has room for now, then the next stage's x (gate/up of 2,048 rows of the 1B shape 116 us with x beside
  // the earlier half, 110 so).
  const auto early = [&](int j) {
    if (!QUARTERS) some(j, PER - LATE, LATE, 0, PRODUCTS);
  };
  const auto late = [&](int j) {
    if (!QUARTERS) {
      some(j, 0, PER - LATE, 0, PRODUCTS);
    } else {
      some(j, PER / 2, PER / 2, 0, PRODUCTS / 2);
      if (j == PRODUCTS / 2 - 1) asked();
      some(j, 0, PER / 2, PRODUCTS / 2, PRODUCTS / 2);
    }
  };
  // (loads that may still be under way when a stage must be whole)
  constexpr int AHEAD = QUARTERS ? PER / 2 : PER * (BUFS - 2);

  sources(a_id);
#pragma unroll
  for (int s = 0; s < (QUARTERS ? BUFS : BUFS - 1); ++s) {
#pragma unroll
    for (int i = 0; i < PER; ++i) ask(i);
    asked();
  }
#pragma unroll
  for (int i = 0; i < PER - LATE; ++i) ask(i);
  Half h0, h1;
  wait_loads<PER*(QUARTERS ? 1 : BUFS - 2) + PER - LATE>();
  barrier();
#pragma unroll
  for (int i = 0; i < READS; ++i) read(h0, 0, i);
  wait_loads<63>();
  for (int id = blockIdx.x; id < total; id += p.grid) {
    clear();
    for (int step = 0; step < p.steps; ++step) {
      half(h0, h1, 1, early);
      if (!QUARTERS) asked();
      wait_loads<AHEAD>();
      barrier();                           // the next stage is whole, this one has been read
      onward();
      half(h1, h0, 0, late);
      wait_loads<63>();                    // (of h0)
    }
    int m0, n0, slice;
    place(id, m0, n0, slice);
#pragma unroll
    for (int m = 0; m < MI; ++m) {
      const int token = m0 + (wm * MI + m) * 16 + r;
      if (token >= p.T) continue;
      if (OUT == kOutGated) {
        bf16_t* row = (bf16_t*)p.Y + (long long)token * p.ldy;
        constexpr int Q = NI % 4 == 0 ? 2 : 1;   // pairs of blocks whose columns are neighbours
#pragma unroll
        for (int a = 0; a < NI / 2; a += Q) {
          uint32_t o[2 * Q];
#pragma unroll
          for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
              const f32x4 gate = acc[2 * (a + q)][m], up = acc[2 * (a + q) + 1][m];
              o[q * 2 + i / 2] = bf16_pair(gated_result(gate[i], up[i], 0), gated_result(gate[i + 1], up[i + 1], 0));
            }
          const int n = n0 + wn * NI * 8 + a * 16 + g * 4 * Q;
          if (n >= p.N) continue;
          if (Q == 2) *(uint4*)(row + n) = make_uint4(o[0], o[1], o[2 * Q - 2], o[2 * Q - 1]);
          else *(uint2*)(row + n) = make_uint2(o[0], o[1]);
        }
      } else if constexpr (OUT == kOutHeads) {
        store_heads<MI, NI>(p, acc, m, token, n0 + wn * NI * 8, g);
      } else if (OUT == kOutBf16) {
        bf16_t* row = (bf16_t*)p.Y + (long long)token * p.ldy;
#pragma unroll
        for (int a = 0; a < NI; a += 2) {
          const f32x4 u = acc[a][m], v = acc[a + 1][m];
          const int n = n0 + (wn * NI + a) * 16 + g * 8;
          if (n >= p.N) continue;
          *(uint4*)(row + n) = make_uint4(bf16_pair(u[0], u[1]), bf16_pair(u[2], u[3]), bf16_pair(v[0], v[1]),
                                          bf16_pair(v[2], v[3]));
        }
      } else {
        float* row = (float*)p.Y + slice * p.slice_stride + (long long)token * p.ldy;
#pragma unroll
        for (int a = 0; a < NI; ++a) {
          const int n = n0 + (wn * NI + a) * 16 + g * 4;
          if (n < p.N) *(f32x4*)(row + n) = acc[a][m];
        }
      }
    }
  }
  wait_loads<0>();                         // (loads past the last tile still write LDS)
#endif
}

template <int MI, int NI, int WM, int WN, int BUFS, int OUT, bool NT>
int launch_tiles(ArgsOf<OUT> a, hipStream_t stream) {
  static LdsGrant grant;
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN;
  constexpr int bytes = (BUFS * 2 + (BUFS == 2 && WM * WN == 8)) * (BM + BN) * kBK;
  static_assert(bytes <= 160 * 1024, "");
  const auto kernel = gemm_tiles_kernel<MI, NI, WM, WN, BUFS, OUT, NT, ArgsOf<OUT>>;
  const hipError_t e = grant_lds(grant, (const void*)kernel, bytes);
  RLIS_REQUIRE(e == hipSuccess, "gemm_tiles: %s", hipGetErrorString(e));
  a.mt = ceil_div(a.T, BM);
  a.nt = ceil_div(a.N, in_pairs(OUT) ? BN / 2 : BN);
  a.group = std::min(a.mt, 8);
  const int cus = rlis_stream_compute_units();
  RLIS_REQUIRE(cus > 0, "gemm_tiles: cannot read the device properties");
  const int resident = std::max(1, std::min(160 * 1024 / bytes, 8 / (WM * WN)));
  const long long total = (long long)a.mt * a.nt * a.slices;
  RLIS_REQUIRE(total < (1 << 30), "gemm_tiles: too many tiles");
  a.grid = (int)std::min<long long>(total, (long long)cus * resident);
  kernel<<<dim3(a.grid), WM * WN * 64, bytes, stream>>>(a);
  return 0;
}

template <int MI, int NI, int WM, int WN, int BUFS>
int launch_out(const TilesArgs& a, int out, int nt, hipStream_t stream) {
  // (rows of W that a second tile reads too must stay in the caches: the output head of the 1B shape at 96
  // rows in tiles of 64 x 256 132 us, non-temporally 178)
  if (nt && a.T <= 16 * MI * WM) {
    if (out == kOutBf16) return launch_tiles<MI, NI, WM, WN, BUFS, kOutBf16, true>(a, stream);
    if (out == kOutF32) return launch_tiles<MI, NI, WM, WN, BUFS, kOutF32, true>(a, stream);
    return launch_tiles<MI, NI, WM, WN, BUFS, kOutGated, true>(a, stream);
  }
  if (out == kOutBf16) return launch_tiles<MI, NI, WM, WN, BUFS, kOutBf16, false>(a, stream);
  if (out == kOutF32) return launch_tiles<MI, NI, WM, WN, BUFS, kOutF32, false>(a, stream);
  return launch_tiles<MI, NI, WM, WN, BUFS, kOutGated, false>(a, stream);
}

int launch_form(const TilesArgs& a, int out, int tile, int nt, hipStream_t stream) {
  int rc = 0;
  switch (tile) {
    case 0: rc = launch_out<4, 4, 2, 4, 3>(a, out, nt, stream); break;   // 128 x 256
    case 1: rc = launch_out<4, 4, 4, 2, 3>(a, out, nt, stream); break;   // 256 x 128
    case 2: rc = launch_out<7, 4, 2, 2, 3>(a, out, nt, stream); break;   // 224 x 128
    case 3: rc = launch_out<6, 4, 2, 2, 3>(a, out, nt, stream); break;   // 192 x 128
    case 4: rc = launch_out<5, 4, 2, 2, 4>(a, out, nt, stream); break;   // 160 x 128
    case 5: rc = launch_out<4, 2, 2, 4, 5>(a, out, nt, stream); break;   // 128 x 128
    case 6: rc = launch_out<4, 2, 2, 2, 3>(a, out, nt, stream); break;   // 128 x 64, two to a compute unit
    case 7: rc = launch_out<2, 2, 2, 2, 4>(a, out, nt, stream); break;   // 64 x 64, two to a compute unit
    case 8: rc = launch_out<4, 2, 1, 4, 3>(a, out, nt, stream); break;   // 64 x 128, two to a compute unit
    case 9: rc = launch_out<4, 4, 1, 4, 2>(a, out, nt, stream); break;   // 64 x 256, two to a compute unit
    case 10: rc = launch_out<8, 4, 2, 4, 2>(a, out, nt, stream); break;  // 256 x 256
    default: RLIS_REQUIRE(false, "gemm_tiles: no tile %d", tile);
  }
  if (rc) return rc;
  RLIS_LAUNCH_CHECK("gemm_tiles");
  return 0;
}

// Tiles of which a compute unit holds two, unless there are not that many: a unit with one has all of the LDS
// for its ring (q/k/v, cold weights, us: 200 x 5,120 x 3,072 in 128 x 64 26.2 with three stages, 23.8 with six; 65 x
// 6,144 x 4,096 in 64 x 64 22.0 with four, 19.5 with nine; output of 512 rows of the 1B shape no faster).
template <int MI, int NI, int WM, int WN, int BUFS, int ALONE>
int launch_deep(const HeadsTilesArgs& a, hipStream_t stream) {
  const long long tiles = (long long)ceil_div(a.T, 16 * MI * WM) * ceil_div(a.N, 8 * NI * WN);
  if (tiles <= rlis_stream_compute_units()) return launch_tiles<MI, NI, WM, WN, ALONE, kOutHeads, false>(a, stream);
  return launch_tiles<MI, NI, WM, WN, BUFS, kOutHeads, false>(a, stream);
}

// (the numbers of the tiles above, and two of their own)
int launch_heads(const HeadsTilesArgs& a, int tile, hipStream_t stream) {
  int rc = 0;
  switch (tile) {
    case 0: rc = launch_tiles<4, 4, 2, 4, 3, kOutHeads, false>(a, stream); break;
    case 1: rc = launch_tiles<4, 4, 4, 2, 3, kOutHeads, false>(a, stream); break;
    case 3: rc = launch_tiles<6, 4, 2, 2, 3, kOutHeads, false>(a, stream); break;
    case 4: rc = launch_tiles<5, 4, 2, 2, 4, kOutHeads, false>(a, stream); break;
    case 5: rc = launch_tiles<4, 2, 2, 4, 5, kOutHeads, false>(a, stream); break;
    case 6: rc = launch_deep<4, 2, 2, 2, 3, 6>(a, stream); break;
    case 7: rc = launch_deep<2, 2, 2, 2, 4, 9>(a, stream); break;
    case 10: rc = launch_tiles<8, 4, 2, 4, 2, kOutHeads, false>(a, stream); break;
    case 11: rc = launch_tiles<2, 6, 4, 1, 5, kOutHeads, false>(a, stream); break;  // 128 x 96
    case 12: rc = launch_tiles<1, 6, 4, 1, 4, kOutHeads, false>(a, stream); break;  // 64 x 96, two to a compute unit
    default: RLIS_REQUIRE(false, "gemm_tiles_heads: no tile %d", tile);
  }
  if (rc) return rc;
  RLIS_LAUNCH_CHECK("gemm_tiles_heads");
  return 0;
}

// The tiles: rows of x by weight rows, and how long a stage takes (us; where two workgroups share a
// compute unit, half of what it takes both).  Fitted to some 1,200 products of the 1B, 3B and 8B shapes at 72
// to 2,048 rows, which the sums below give to 8 %.
struct TileForm {
  int rows, cols;
  float stage;
};
constexpr TileForm kForms[] = {{128, 256, 0.75f}, {256, 128, 0.72f}, {224, 128, 0.66f}, {192, 128, 0.60f},
                               {160, 128, 0.55f}, {128, 128, 0.48f}, {128, 64, 0.35f}, {64, 64, 0.215f},
                               {64, 128, 0.33f}, {64, 256, 0.46f}, {256, 256, 1.38f}};
constexpr int kFormCount = sizeof(kForms) / sizeof(kForms[0]);
constexpr int kWideForms = 8;              // those that products of more than 64 rows choose from
constexpr int kLargest = 10;               // and gate/up beyond 512 rows, output heads beyond 128
// of tiles of 128 x 256 that store partial sums over a k in 8,192s for weight rows in 2,048s, ahead of 256 x 128 there
// (2,048 x 8,192 at 2,048 rows 62.0 against 64.0 us; else up to 8 % behind: 1,536 rows of 2,560 x 6,912 57.1 against 52.8)
constexpr float kPartialStage = 0.71f;
constexpr float kPartial = 1.75e-6f;       // us to write and add one float32 partial sum

// The same for q, k and v on their way to the cache: a stage's time with two workgroups to a compute unit and
// alone (where there is no more than one tile a unit), and what ends a round (us).
struct HeadsForm {
  int tile, rows, cols;
  float stage, alone, end;
};
constexpr HeadsForm kHeadsForms[] = {
    {0, 128, 256, 0.73f, 0.73f, 2.7f}, {1, 256, 128, 0.67f, 0.67f, 3.6f}, {3, 192, 128, 0.545f, 0.545f, 5.1f},
    {4, 160, 128, 0.48f, 0.48f, 3.9f}, {5, 128, 128, 0.47f, 0.47f, 1.4f}, {6, 128, 64, 0.32f, 0.36f, 0.f},
    {7, 64, 64, 0.204f, 0.215f, 0.f},  {10, 256, 256, 1.17f, 1.17f, 8.6f}, {11, 128, 96, 0.40f, 0.40f, 2.4f},
    {12, 64, 96, 0.27f, 0.30f, 0.f}};
constexpr int kHeadsFormCount = sizeof(kHeadsForms) / sizeof(kHeadsForms[0]);

// The library's: tiles that explain its times, whose rounds cost it as the rounds here do, and a stage's time.
constexpr TileForm kLibraryForms[] = {{256, 256, 0.985f}, {256, 128, 0.563f}, {128, 256, 0.605f}, {128, 128, 0.40f},
                                      {192, 256, 0.818f}, {256, 192, 0.845f}, {64, 128, 0.276f}};

}  // namespace

// How the product of T rows with N weight rows (gated: gate and up rows together) is cut: the tile (an
// index that rlis_gemm_bf16_tiles takes) + 16 times the slices of k, or -1 where the library should
// have it.  partials: the result may come as `slices` partial sums (0: as many of 1, 2 and 4 as suit).
// units: the device's compute units (the figures are those of 256).
//
// The tile (and the number of slices) is what makes least of the rounds over the compute units times
// a round's stages, with what partial sums cost.  Which products are taken is measured against the library's, tried
// out as it is, with weights that no cache holds: 64 to 57,344 weight rows over a k of 64 to 28,672, 65 to
// 2,048 rows.  In one slice a tile walks all of k, which the library cuts where there are few tiles (160 x
// 4096 at 128 rows 13.9 us against its 6.4, 1024 x 8192 35 against 15, 3072 x 4096 22 against 17), so:
//
//   plain    k of 256 to 512, and to 1,024 from 1,024 weight rows on: up to 256 rows, to 1,024 over up to
//            8,192 weight rows (0.27 to 1.06 of the library's time); k up to 2,048 from 1,024 weight rows on while
//            tiles of 64 x 64 make one round with at least 3/16 of the units in it (0.75 to 1.06; two rounds 0.9 to
//            1.15), k up to 4,096 up to 160 rows while that round has 3/4 of the units, from 97 rows on, where the
//            library takes a step, 5/8 (0.81 to 1.03; else 0.94 to 1.3, but 6,144 weight rows at 136 rows 0.75);
//            16,384 weight rows and more (there are tiles enough): up to 128 rows at any k (0.56 to 1.09), to
//            256 over up to 32,768 (0.65 to 1.06), beyond where rounds come out even (else up to 1.5).  There
//            tiles of 256 x 256 pay from some 200 rows on (128,256 x 2,048 at 256 rows, float32, us: library 182,
//            256 x 128 154, these 139; 65,536 x 4,096 156, 136, 127).  Even rounds beyond 32,768 over a k of 2,048 and
//            more: 0.81 to 1.03, but 1.0 to 1.14 over a k of 3,072 where weight rows come in 4,096s; over 1,024 and
//            1,536 0.90 to 1.16.  More rows of x are the library's: at 257 to 512 rows the tiles take 0.8 to 0.95 of its
//            time over 128,256 and 151,936 weight rows, which leave it with broken tiles, and 1.0 to 1.2 of it over
//            126,976, 131,072, 160,000 and most others.
//   partials k below 8,192: up to 512 rows (0.49 to 1.08; over 1,024 < k <= 2,048 and more than 2,048 weight rows
//            beyond 256 rows only where the rounds come out even: else up to 1.1), to 2,048 where one even round
//            fills the chip.  k from 8,192 on, which the library has in slices too: up to 192 rows (0.67 to 1.15
//            alone; down in a step of the 3B shape, where the library's algorithm is another row count's, 4 us ahead
//            at 66 to 152 rows), to 2,048 where one even round fills the chip (0.9 to 1.04; uneven up to 1.26,
//            two rounds of 768 to 2,048 rows 1.06 to 1.26); over more than 4,096 weight rows up to 128 rows of a
//            k of 16,384 and more (0.64 to 1.02; else up to 1.25).
//   gated    k up to 1,024, and to 2,048 from 1,024 weight rows on: up to 256 rows, to 512 where the rounds come out
//            even or there is one (0.36 to 1.03).  Longer k from 5,632 weight rows on: up to 192 rows, beyond where
//            rounds come out nearly even (0.66 to 1.1; fewer weight rows up to 2.0).  From 1,024 rows on (over a k of
//            1,024 beyond 512) where rounds come out even, k of 1,024 to 3,072 from 8,192 weight rows on: k of 1,024 as it is
//            (0.78 to 1.01); longer ones in tiles of 256 x 256 where their last round is nearly full, in 256 x 128 and
//            128 x 256 where it is full (334 products of 16 shapes at 1,024 to 8,192 rows: 220 taken, up to 1.02, 0.92 on
//            average, 0.67 where the library has a broken round more; the smaller tiles up to 1.15; uneven rounds up to 1.12, 640 and 768 rows 1.05 to 1.14).  Where tiles of
//            256 x 256 waste less than a tenth of their rounds, over a k of up to 5,120 and from 513 rows on (the product
//            alone, us: 28,672 x 4,096 at 2,304 / 4,096 / 8,192 rows 402 -> 393, 691 -> 674, 1,368 -> 1,326; 22,016 x
//            4,096 at 8,192 1,211 -> 1,037; 37,888 x 3,584 at 1,280 / 2,048 386 -> 255, 544 -> 417; 27,648 x 5,120 at
//            4,096 1,046 -> 819; 16,384 x 2,048 and 3,072 at 1,000 68 -> 59, 94 -> 85: 110 products 0.63 to 1.0, those of
//            24,576 x 4,096 and 36,864 x 4,608 the closest, 0.96 to 1.0).
RLIS_API int rlis_gemm_bf16_tiles_plan(int T, int N, int K, int gated, int partials, int slices, int units) {
  if (T <= 0 || N <= 0 || K <= 0 || units <= 0) return -1;
  float least = 0.f;
  int best = -1, best_rounds = 0, best_tiles = 0;
  for (int s = slices > 0 ? slices : 1; s <= (slices > 0 ? slices : partials ? 4 : 1); s *= 2) {
    if (K % (s * kBK) || (slices <= 0 && s > 1 && K / s < 512)) continue;
    for (int f = 0; f < kFormCount; ++f) {
      const bool largest = f == kLargest && (gated ? T > 512 : !partials && T > 128 && N >= 64 * units);
      if (T <= 64 ? kForms[f].rows > 64 : f >= kWideForms && !largest) continue;
      const long long tiles = (long long)ceil_div(T, kForms[f].rows) * ceil_div(N, kForms[f].cols) * s;
      const long long rounds = (tiles + units - 1) / units;
      if (rounds > 1 << 20) continue;
      const float stage = f == 0 && partials && K % 8192 == 0 && N % 2048 == 0 ? kPartialStage : kForms[f].stage;
      const float us = (float)rounds * (K / s / kBK) * stage +
                       (s > 1 ? kPartial * s : kPartial / 2) * (float)T * N;
      if (best < 0 || us < least) least = us, best = f + 16 * s, best_rounds = (int)rounds, best_tiles = (int)tiles;
    }
  }
  if (best < 0) return -1;
  // (nine in ten places of the rounds have a tile)
  const bool even = best_tiles * 10LL >= best_rounds * (units * 9LL), one = best_rounds == 1;
  // (nine tenths of what tiles of 256 x 256 work out in their rounds is wanted)
  const long long largest_rounds =
      ((long long)ceil_div(T, kForms[kLargest].rows) * ceil_div(N, kForms[kLargest].cols) + units - 1) / units;
  const bool largest_full = K > 1024 && K <= 5120 && N >= 8192 &&
                            (long long)T * N * 10 >= largest_rounds * units * kForms[kLargest].rows * kForms[kLargest].cols * 9;
  bool here;
  if (T <= 64) {
    here = true;                           // (the caller knows which)
  } else if (partials) {
    if (K < 8192) {
      here = T <= 256 || (T <= 512 && (K <= 1024 || K > 2048 || N <= 2048 || even)) || (T <= 2048 && one && even);
    } else if (N > 4096) {
      here = T <= 128 && K >= 16384;
    } else {
      here = T <= 192 || (T <= 2048 && one && even && (T <= 512 || N >= 1024));
    }
  } else if (gated && T > 512 && largest_full) {
    here = true;
    best = kLargest + 16;
  } else if (gated && T > 512) {
    here = even && K >= 1024 && K <= 3072 && N >= 8192 && (T >= 1024 || K == 1024);
    if (here && K > 1024) {
      const int most = ceil_div(T, kForms[kLargest].rows) * ceil_div(N, kForms[kLargest].cols);
      if (most * 20LL >= ceil_div(most, units) * (units * 17LL))
        best = kLargest + 16;
      else
        here = best % 16 <= 1 && best_tiles * 20LL >= best_rounds * (units * 19LL);
    }
  } else if (gated) {
    if (K > 2048)
      here = N >= 5632 && (T <= 192 || (T <= 256 && best_tiles * 20LL >= best_rounds * (units * 17LL)) || (T <= 512 && even));
    else
      here = (K <= 1024 || N >= 1024) && (T <= 256 || (T <= 512 && (even || one)));
  } else if (N >= 64 * units) {
    here = T <= 128 || (T <= 256 && (N <= 128 * units || (even && K >= 2048)));
  } else if (K <= 1024) {
    here = (K <= 512 ? K >= 256 : N >= 1024) && (T <= 256 || (T <= 1024 && N <= 8192));
  } else {
    const long long tiles = (long long)ceil_div(T, 64) * ceil_div(N, 64);
    here = tiles <= units && (K <= 2048 ? N >= 1024 && tiles >= units * 3 / 16
                                        : K <= 4096 && T <= 160 && tiles >= units * (T <= 96 ? 6 : 5) / 8);
  }
  return here ? best : -1;
}

// The tile that rlis_gemm_bf16_tiles_heads should take for T rows and N weight rows, or -1 where the library's
// product and the kernel that turns and stores (elementwise.hip) are ahead.  Both sides are estimated: a tile's stages,
// what ends a round and what is fixed; the library's as rounds of tiles too, with the rows that pass through memory.
// 529 products of 20 shapes, 1,536 to 12,288 weight rows over a k of 512 to 8,192, at 65 to 8,192 rows, weights cold:
// tiles 0.95 to 1.06 of what they take in half of all cases, 0.88 to 1.14 in nine of ten; the library 0.95 to 1.05 and
// 0.89 to 1.12.  So the tiles have to be ahead by an estimated 2 to 7 %, the more rows the more (above 1,024 rows the
// library runs its heuristics' first algorithm: 2,560 rows of 6,144 x 4,096 97 us, 2,800 160), past 4,096 rows by 14 %
// but for many weight rows over a short k, where the tiles were behind nowhere (0.71 to 0.98).  Of the 529 this takes
// 398, 0.53 to 1.07 of the library's time, 0.81 on average; the tiles are behind at 1,600 rows of 6,144 x 2,048
// (1.07), 512 of 4,608 x 3,584 (1.03), 505 and 512 of 5,120 x 3,072 and 333 of 8,192 x 6,144 (1.02).
// Figures are those of 256 units.
RLIS_API int rlis_gemm_bf16_tiles_heads_plan(int T, int N, int K, int units) {
  if (T <= 0 || N <= 0 || K <= 0 || units <= 0) return -1;
  const auto rounds_of = [&](int rows, int cols) {
    const long long tiles = (long long)ceil_div(T, rows) * ceil_div(N, cols);
    return (float)((tiles + units - 1) / units);
  };
  float least = 0.f;
  int best = -1;
  for (int f = 0; f < kHeadsFormCount; ++f) {
    const HeadsForm& form = kHeadsForms[f];
    const float rounds = rounds_of(form.rows, form.cols);
    const float us = rounds * (K / kBK * (rounds == 1.f ? form.alone : form.stage) + form.end);
    if (best < 0 || us < least) least = us, best = form.tile;
  }
  const float here = least + 4.9f + (0.095e-6f * K + 0.6e-6f * T) * N;
  float stages = rounds_of(kLibraryForms[0].rows, kLibraryForms[0].cols) * kLibraryForms[0].stage;
  for (const TileForm& form : kLibraryForms) stages = std::min(stages, rounds_of(form.rows, form.cols) * form.stage);
  const float library = 7.9f + stages * (K / kBK) + (0.2e-6f * K + 1.65e-6f * T) * N;
  const float margin = T <= 4096 ? 0.99f - 1.9e-5f * T : N >= 5120 && K <= 3072 ? 1.f : 0.86f;
  return here < library * margin ? best : -1;
}

// Y (T,N) = X (T,K) * W (N,K)^T, N a multiple of 8, K of 64 times the slices.  out 0: bfloat16; 1:
// float32, `slices` partial results slice_stride elements apart; 2: gated, W (2 N,K) gate rows then up
// rows, Y = silu(gate) * up in bfloat16.  tile: as rlis_gemm_bf16_tiles_plan gives it.  nt: W is loaded
// non-temporally (load_weights) where one row of tiles holds all of x.
RLIS_API int rlis_gemm_bf16_tiles(const void* X, const void* W, void* Y, int out, int T, int N, int K,
                                  int slices, long long ldx, long long ldw, long long ldy,
                                  long long slice_stride, int tile, int nt, hipStream_t stream) {
  RLIS_REQUIRE(T > 0 && N > 0 && N % 8 == 0 && slices > 0 && K > 0 && K % (slices * kBK) == 0,
               "gemm_tiles: bad sizes T=%d N=%d K=%d slices=%d", T, N, K, slices);
  RLIS_REQUIRE(out >= 0 && out <= 2 && (slices == 1 || out == 1), "gemm_tiles: no such form");
  RLIS_REQUIRE(ldx >= K && ldw >= K && ldy >= N && ldx % 8 == 0 && ldw % 8 == 0 && ldy % 8 == 0 &&
                   slice_stride % 4 == 0 && (uintptr_t)X % 16 == 0 && (uintptr_t)W % 16 == 0 &&
                   (uintptr_t)Y % 16 == 0,
               "gemm_tiles: rows must lie on 16-byte boundaries");
  RLIS_REQUIRE(ldx * 2 * T < (1LL << 32) && ldw * 2 * N * (out == 2 ? 2 : 1) < (1LL << 32),
               "gemm_tiles: x or W passes 4 GB");
  const TilesArgs a = {(const bf16_t*)X, (const bf16_t*)W, Y, T, N, K / slices / kBK, 0, 0, slices, 0,
                       (int)ldx, (int)ldw, 0, ldy, slice_stride};
  return launch_form(a, out, tile, nt, stream);
}

// Q, and the cache's pages, from X (T,K) * W ((nh + 2 nkv) d,K)^T, W's rows the query, key and value heads: Q
// (T, nh d) holds the query heads as they come, keys go to k_pages (pages, nkv, page_size, d) turned by
// positions (rotate-half over the whole head, cos and sin (positions, d / 2); null: as they come), values to
// v_pages (pages, nkv, d, page_size), at slots (below 0: not stored).  d 64, 128 or 256, page_size a power of two.
// Products are rounded to bfloat16 before they are turned.  Where a tile holds whole heads (weight rows in ds) the bits
// are those of rlis_gemm_bf16_tiles in the same tile and rlis_rope_kv_write; elsewhere some dims of a head lie in another
// tile than there and start their walk over k at another stage.
RLIS_API int rlis_gemm_bf16_tiles_heads(const void* X, const void* W, void* Q, int T, int nh, int nkv, int d, int K,
                                        long long ldx, long long ldw, long long ldq, const float* cos,
                                        const float* sin, const int* positions, const int* slots, void* k_pages,
                                        void* v_pages, int page_size, int tile, hipStream_t stream) {
  RLIS_REQUIRE(T > 0 && nh > 0 && nkv > 0 && K > 0 && K % kBK == 0, "gemm_tiles_heads: bad sizes T=%d nh=%d nkv=%d K=%d",
               T, nh, nkv, K);
  RLIS_REQUIRE(d == 64 || d == 128 || d == 256, "gemm_tiles_heads: heads of %d, 64, 128 or 256 only", d);
  RLIS_REQUIRE(page_size > 0 && (page_size & (page_size - 1)) == 0, "gemm_tiles_heads: page size %d must be a power of two",
               page_size);
  const long long rows = (nh + 2LL * nkv) * d;
  RLIS_REQUIRE(ldx >= K && ldw >= K && ldq >= (long long)nh * d && ldx % 8 == 0 && ldw % 8 == 0 && ldq % 8 == 0 &&
                   (uintptr_t)X % 16 == 0 && (uintptr_t)W % 16 == 0 && (uintptr_t)Q % 16 == 0 &&
                   (uintptr_t)k_pages % 16 == 0 && (uintptr_t)v_pages % 16 == 0,
               "gemm_tiles_heads: rows must lie on 16-byte boundaries");
  RLIS_REQUIRE(positions && slots && k_pages && v_pages && !cos == !sin && (uintptr_t)cos % 16 == 0 &&
                   (uintptr_t)sin % 16 == 0,
               "gemm_tiles_heads: pages, slots, positions and both tables of angles are needed");
  RLIS_REQUIRE(ldx * 2 * T < (1LL << 32) && ldw * 2 * rows < (1LL << 32), "gemm_tiles_heads: x or W passes 4 GB");
  HeadsTilesArgs a = {{(const bf16_t*)X, (const bf16_t*)W, Q, T, (int)(rows / 2), K / kBK, 0, 0, 1, 0,
                       (int)ldx, (int)ldw, 0, ldq, 0}, {}};
  a.heads = {cos, sin, positions, slots, (bf16_t*)k_pages, (bf16_t*)v_pages, nh, nkv, 0, 0};
  while (2 << a.heads.half_shift < d) ++a.heads.half_shift;
  while (1 << a.heads.page_shift < page_size) ++a.heads.page_shift;
  return launch_heads(a, tile, stream);
}
