// Prefill attention of whole heads of 64 or 128 dims in tiles of 128 queries (attention_mfma.hip holds the form for
// every other size, for 64 queries, windows, chunks and shaped scores, and the notation).
//
// A workgroup of four waves serves 128 consecutive new tokens of one sequence for one query head, each wave 32 of
// them, on v_mfma_f32_32x32x16_bf16 with both products transposed:
//   S^T = K Q^T   (rows: 32 keys, columns: 32 queries)
//   O^T = V^T P^T (rows: 32 dims, columns: 32 queries)
// A lane holds one query (column l % 32), and of 32 keys the sixteen whose probabilities its half of the second
// product's operand takes: row 8 j + 4 h + r of the first product (h = l / 32) is key 16 (j / 2) + 8 h + 4 (j % 2) + r.
// So a row's maximum takes one exchange and P never leaves the registers.
//
// K and V come into LDS by direct loads, a tile of 64 keys ahead, in two places taking turns: no registers are held for
// them, and as every load lies in one page, addresses are scalar but for an offset that a lane computes once.  Piece c
// (16 bytes) of a row lies where the reads of a fragment, sixteen lanes a cycle, fall on sixteen quarters of the banks.
// The page ids of 64 pages are held one to a lane.
//
// G groups of four waves take a workgroup's tiles of keys in turn, each with LDS of its own, and the first adds up: a
// walk of half the length where few workgroups leave the units to it (ops/attention_plan.py says where).
//
// The denominator is the float32 sum of the float32 probabilities, as in the other form: the sum of the rounded ones, as the
// second product takes them, is one instruction for two and no faster (8,192 tokens of 32 heads of 128 549 us either way,
// 2,048 of 32 heads of 64 30.7), and a row whose probabilities round one way is off by up to 2^-8 with it.  Error against 64
// bits, of the result's norm, other form -> this: 1,024 tokens at head size 64 2.009e-3 -> 1.992e-3, 464 on 2,000 at 128
// 2.230e-3 -> 2.196e-3, scores six times as wide 1.682e-3 -> 1.670e-3; where the other form has blocks of 16 queries and tiles
// of 32 keys as before, 8,192 tokens 2.061e-3 -> 2.068e-3 (84 inputs: 0.977 to 1.004 times as much, the worst row 0.88 to
// 1.06).  (A maximum that follows the true one only by steps of 2^8 spares the rescaling and 3 to 10 % of the time, but puts
// the largest probabilities anywhere between powers of two: 5 % more error.)
//
// What bounds it is the vector unit beside the matrix cores: 210 instructions and 33 exponentials a wave and tile at head size
// 128, against 32 products; the vector unit is busy 48 % of 8,192 tokens' time and the matrix cores 40 % (counters; at head
// size 64, 2,048 tokens, 60 and 23 %), and a loop that issues the next tile's products between this one's exponentials is
// slower (8,192 tokens of 32 heads of 128 595 us for 545).  Tiles of 32 keys 598, three places 709 (one workgroup a unit).
//
// MI355X, us, the other form in the tiles that it took -> this, in turn: 32 heads of 128, 8,192 tokens 699 -> 549 (1.0 PFLOP/s),
// 2,048 on 30,000 1,250 -> 993, 512 on 8,192 116 -> 90, 24 heads, 464 on 2,000 49.0 -> 34.7; 32 heads of 64, 2,048 tokens
// 42.3 -> 30.6, 512 12.2 -> 9.3, 8,192 409 -> 317.
#pragma once

#if RLIS_HEAD_DIM == 64 || RLIS_HEAD_DIM == 128
#define RLIS_PREFILL_WHOLE 1
#define WHOLE_KERNEL_NAME RLIS_CAT(rlis_attn_prefill_whole_kernel_d, RLIS_HEAD_DIM)

typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace {
constexpr int kWholeTile = 64;                     // keys of a tile
constexpr int kWholeHalves = kWholeTile / 16;      // runs of 16 keys, each inside one page
constexpr int kHalfBytes = 16 * D * 2;             // of K, and of V
constexpr int kTileBytes = 2 * kWholeHalves * kHalfBytes;
constexpr int whole_lds(int groups) { return groups * 2 * kTileBytes; }

// In front of the barrier behind which a tile's place is filled anew: this wave's own part of the next tile has come, and
// its reads of the last one have returned (the barrier is an asm statement, which does not hold back the products that
// would otherwise wait for them).
__device__ __forceinline__ void whole_wait_tile() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0 | 7 << 4 | 0 << 8);     // vmcnt(0) lgkmcnt(0)
  asm volatile("" ::: "memory");
}
}  // namespace

template <int G>
__global__ __launch_bounds__(G * 256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : 2, D == 64 ? 4 : 2)))
void WHOLE_KERNEL_NAME(
    const bf16_t* __restrict__ q, long long q_stride, bf16_t* __restrict__ out, long long out_stride,
    const bf16_t* __restrict__ k_pages, const bf16_t* __restrict__ v_pages, const int* __restrict__ block_tables,
    int max_pages, const int* __restrict__ cu_seqlens, const int* __restrict__ start_pos,
    const int* __restrict__ unit_map, int nh, int nkv, int page_shift, float scale, int num_tiles, int tiles_per_round,
    int part_stride, int row0, float* __restrict__ part_ml, float* __restrict__ part_acc,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, const float* __restrict__ sinks) {
#ifdef __HIP_DEVICE_COMPILE__   // (the host pass knows no buffer resources)
  typedef __attribute__((address_space(3))) void* lds_ptr;
  constexpr int KS = D / 16, DB = D / 32, NB = kWholeTile / 32;
  extern __shared__ __attribute__((aligned(1024))) unsigned char whole_smem[];

  const int lane = threadIdx.x % 64, wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wave = wave_all % 4, group = wave_all / 4;
  unsigned char* ring = whole_smem + group * 2 * kTileBytes;
  const int l32 = lane % 32, hf = lane / 32;
  // Heads fastest, as in the other form; the heads of a die (blockIdx % 8) are neighbours, so that those that share
  // keys and values share an L2.
  int h = blockIdx.x % nh, tile = blockIdx.x / nh;
  if (nh % 8 == 0) h = h % 8 * (nh / 8) + h / 8;
  if (tiles_per_round > 0) {
    const int round = tile / tiles_per_round, within = tile % tiles_per_round;
    if ((round & 1) && (round + 1) * tiles_per_round <= num_tiles)
      tile = round * tiles_per_round + (tiles_per_round - 1 - within);
  }
  const int seq = unit_map[4 * tile], qb = unit_map[4 * tile + 1];
  const int split = unit_map[4 * tile + 2], splits = unit_map[4 * tile + 3];
  const int tok_begin = cu_seqlens[seq], n_new = cu_seqlens[seq + 1] - tok_begin, P = start_pos[seq];
  const int kvh = h / (nh / nkv);
  const int* table = block_tables + (long long)seq * max_pages;

  const int wave_q = qb + wave * 32, my_qi = wave_q + l32, my_pos = P + my_qi;
  Frag8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const bf16_t* p = q + (long long)(tok_begin + min(my_qi, n_new - 1)) * q_stride + h * D + ks * 16 + hf * 8;
    qf[ks].u = *(const uint4*)p;
  }

  // ---- the keys of this workgroup: tiles kt0 .. of positions [kt0, khi)
  const int khi_all = P + min(n_new, qb + 128);
  int kt0 = 0, khi = khi_all;
  if (splits > 1) {
    const int per = ((khi_all + 31) / 32 + splits - 1) / splits * 32;
    kt0 = split * per;
    khi = min(khi_all, kt0 + per);
  }
  const int tiles = khi > kt0 ? (khi - kt0 + kWholeTile - 1) / kWholeTile : 0;
  const int last_page = max(khi - 1, 0) >> page_shift, page_mask = (1 << page_shift) - 1;

  // ---- loads.  Instruction i of a wave: head size 128: half i / 2, rows (or dims) of this wave's fourth, K or V;
  // 64: this wave's half, K's two and V's two.
  const long long page_elems = (long long)nkv << page_shift << (D == 64 ? 6 : 7);
  const bf16_t* k_head = k_pages + ((long long)kvh << page_shift) * D;
  const bf16_t* v_head = v_pages + ((long long)kvh << page_shift) * D;
  uint32_t k_off[D == 64 ? 2 : 1], v_off[D == 64 ? 2 : 1];
#pragma unroll
  for (int j = 0; j < (D == 64 ? 2 : 1); ++j) {
    if (D == 64) {
      const int row = j * 8 + lane / 8;
      k_off[j] = row * D * 2 + ((lane % 8) ^ (row / 2)) * 16;
    } else {
      const int row = wave * 4 + lane / 16;
      k_off[j] = row * D * 2 + ((lane % 16) ^ row) * 16;
    }
    const int dim = (D == 64 ? j : wave) * 32 + lane / 2;
    v_off[j] = (dim << (page_shift + 1)) + ((lane % 2) ^ hf) * 16;
  }
  int a_key = kt0 + group * kWholeTile, a_slot = 0;   // the next tile to ask for, and its place
  int page_base = a_key >> page_shift;                // of the ids that the lanes hold, 64 of them
  int ids = table[min(page_base + lane, last_page)], ids_next = table[min(page_base + 64 + lane, last_page)];
  const auto ask = [&]() {
    if ((min(a_key + kWholeTile - 1, khi - 1) >> page_shift) - page_base >= 64) {
      // (by the page that the tile starts in: all 64, or, where a run starts inside pages of 64 and more, 63 of them)
      const int by = (a_key >> page_shift) - page_base;
      if (by >= 64) {
        ids = ids_next;
      } else {
        const int low = __shfl(ids, (lane + by) % 64, 64), high = __shfl(ids_next, (lane + by) % 64, 64);
        ids = lane + by < 64 ? low : high;
      }
      page_base += by;
      ids_next = table[min(page_base + 64 + lane, last_page)];
      asm volatile("" : "+v"(ids), "+v"(ids_next));    // (waited for here: behind the branch it would be at every tile)
    }
#pragma unroll
    for (int i = 0; i < (D == 64 ? 1 : kWholeHalves); ++i) {
      const int half = D == 64 ? wave : i, key = a_key + half * 16;
      const int page = __builtin_amdgcn_readlane(ids, min(key >> page_shift, last_page) - page_base);
      const int at = key & page_mask;
      const auto kr = __builtin_amdgcn_make_buffer_rsrc((void*)(k_head + page * page_elems), 0, 0xfffffff0u, 0x00027000);
      const auto vr = __builtin_amdgcn_make_buffer_rsrc((void*)(v_head + page * page_elems), 0, 0xfffffff0u, 0x00027000);
      unsigned char* to = ring + a_slot + half * kHalfBytes;
#pragma unroll
      for (int j = 0; j < (D == 64 ? 2 : 1); ++j) {
        const int part = (D == 64 ? j : wave) * 1024;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (lds_ptr)(to + part), 16, k_off[j], at * D * 2, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, (lds_ptr)(to + kWholeHalves * kHalfBytes + part), 16, v_off[j],
                                                 at * 2, 0, 0);
      }
    }
    a_key += G * kWholeTile;
    a_slot ^= kTileBytes;
  };
  if (group < tiles) ask();

  // With cos_t the queries arrive unrotated and are turned by their positions (rotate-half over the whole head): dim j
  // of a lane's fragment ks meets dim j + D / 2 in its fragment ks + KS / 2.
  if (cos_t != nullptr) {
    const long long row = (long long)(P + min(my_qi, n_new - 1)) * (D / 2) + hf * 8;
#pragma unroll
    for (int ks = 0; ks < KS / 2; ++ks) {
      float c[8], s[8];
      *(float4*)&c[0] = *(const float4*)(cos_t + row + ks * 16);
      *(float4*)&c[4] = *(const float4*)(cos_t + row + ks * 16 + 4);
      *(float4*)&s[0] = *(const float4*)(sin_t + row + ks * 16);
      *(float4*)&s[4] = *(const float4*)(sin_t + row + ks * 16 + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x1 = (float)qf[ks].v[e], x2 = (float)qf[ks + KS / 2].v[e];
        qf[ks].v[e] = (__bf16)(x1 * c[e] - x2 * s[e]);
        qf[ks + KS / 2].v[e] = (__bf16)(x2 * c[e] + x1 * s[e]);
      }
    }
  }

  // ---- places of a lane's fragments in a tile
  // (row i of the first product's operand is key 16 (i / 16) + 8 (i / 4 % 2) + 4 (i / 8 % 2) + i % 4)
  const int k_row = l32 / 16 * 16 + l32 / 4 % 2 * 8 + l32 / 8 % 2 * 4 + l32 % 4;
  const int k_turn = D == 64 ? k_row / 2 % 8 : k_row % 16;
  // (piece 2 ks + hf of a row of K lies at (2 ks + hf) ^ turn = 2 ks ^ (hf ^ turn))
  const int k_at = k_row * D * 2 + (hf ^ k_turn) * 16;
  const int v_at = kWholeHalves * kHalfBytes + l32 * 32 + (hf ^ (l32 / 16)) * 16;
  const float in_exp = scale * 1.4426950408889634f;   // scores in the base-2 domain
  float m_run = -INFINITY, m_use = 0.f, l_run = 0.f;
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[db][v] = 0.f;
  const int wave_last = P + min(n_new - 1, wave_q + 31), my_last = min(my_pos, khi - 1);
  int slot = 0;
  // What was loaded in front of the loop is there (else the loop would wait for it, and with it for later tiles).
  asm volatile("" : "+v"(ids), "+v"(ids_next));
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks].v));
  for (int t = group; t < tiles + group; t += G) {
    const int k0 = kt0 + t * kWholeTile;
    whole_wait_tile();
    asm volatile("s_barrier" ::: "memory");            // the tile is whole, the one before it has been read
    if (t + G < tiles) ask();
    if (wave_q < n_new && t < tiles && k0 <= wave_last) {
      const unsigned char* base = ring + slot;
      f32x16 s[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int v = 0; v < 16; ++v) s[nb][v] = 0.f;
        bf16x8 kf[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          kf[ks] = *(const bf16x8*)(ring + ((slot + k_at) ^ (ks * 32)) + nb * 2 * kHalfBytes);
        __builtin_amdgcn_sched_barrier(0);             // all of them on their way before the first product
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          s[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks], qf[ks].v, s[nb], 0, 0, 0);
      }
      // (V's fragments of the first half arrive beside the softmax)
      bf16x8 vf[DB];
#pragma unroll
      for (int db = 0; db < DB; ++db) vf[db] = *(const bf16x8*)(base + v_at + db * 1024);
      __builtin_amdgcn_sched_barrier(0);
      if (k0 + kWholeTile - 1 > P + wave_q || k0 + kWholeTile > khi) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int key = k0 + nb * 32 + v / 8 * 16 + hf * 8 + v % 8;
            if (key > my_last) s[nb][v] = -INFINITY;
          }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 16; ++v) mx = fmaxf(mx, s[nb][v]);
      mx = xor32_max(mx) * in_exp;
      if (__any(mx > m_run)) {
        const float m_new = fmaxf(m_run, mx);
        m_use = m_new == -INFINITY ? 0.f : m_new;      // (a query with no key yet)
        const float corr = __builtin_amdgcn_exp2f(m_run - m_use);
        m_run = m_new;
        l_run *= corr;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int v = 0; v < 16; ++v) o[db][v] *= corr;
      }
      bf16x8 p[NB * 2];
      float sum[2] = {0.f, 0.f};
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 16; v += 2) {
          const float a = __builtin_amdgcn_exp2f(fmaf(s[nb][v], in_exp, -m_use));
          const float b = __builtin_amdgcn_exp2f(fmaf(s[nb][v + 1], in_exp, -m_use));
          sum[0] += a;
          sum[1] += b;
          p[nb * 2 + v / 8][v % 8] = (__bf16)a;
          p[nb * 2 + v / 8][v % 8 + 1] = (__bf16)b;
        }
      l_run += sum[0] + sum[1];                                  // (the two lanes of a query are added at the end)
#pragma unroll
      for (int st = 0; st < NB * 2; ++st)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[db], p[st], o[db], 0, 0, 0);
          if (st + 1 < NB * 2) vf[db] = *(const bf16x8*)(base + v_at + (st + 1) * kHalfBytes + db * 1024);
        }
    }
    slot ^= kTileBytes;
  }

  // ---- the later groups hand their sums to the first
  if (G > 1) {
    f32x4* hand = (f32x4*)whole_smem;
    float2* hand_ml = (float2*)(whole_smem + (G - 1) * 4 * DB * 4096);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");            // (every tile has been read)
    if (group > 0) {
      const int at = (group - 1) * 4 + wave;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          hand[((at * DB + db) * 4 + j) * 64 + lane] =
              f32x4{o[db][4 * j], o[db][4 * j + 1], o[db][4 * j + 2], o[db][4 * j + 3]};
      hand_ml[at * 64 + lane] = make_float2(m_run, l_run);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    if (group > 0) return;
#pragma unroll
    for (int other = 0; other < G - 1; ++other) {
      const int at = other * 4 + wave;
      const float2 ml = hand_ml[at * 64 + lane];
      const float m_new = fmaxf(m_run, ml.x), m_all = m_new == -INFINITY ? 0.f : m_new;
      const float mine = __builtin_amdgcn_exp2f(m_run - m_all), theirs = __builtin_amdgcn_exp2f(ml.x - m_all);
      m_run = m_new;
      l_run = l_run * mine + ml.y * theirs;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x4 v = hand[((at * DB + db) * 4 + j) * 64 + lane];
#pragma unroll
          for (int r = 0; r < 4; ++r) o[db][4 * j + r] = o[db][4 * j + r] * mine + v[r] * theirs;
        }
    }
  }

  // ---- normalise and store: this lane holds dims db * 32 + 8 j + 4 hf + [0, 4) of its query
  l_run = xor32_sum(l_run);
  if (splits > 1) {
    if (my_qi >= n_new) return;
    const long long idx = (((long long)tok_begin + my_qi - row0) * nh + h) * part_stride + split;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *(float4*)(part_acc + idx * D + db * 32 + j * 8 + hf * 4) =
            make_float4(o[db][4 * j], o[db][4 * j + 1], o[db][4 * j + 2], o[db][4 * j + 3]);
    if (hf == 0) {
      part_ml[idx * 2] = m_run * 0.6931471805599453f;
      part_ml[idx * 2 + 1] = l_run;
    }
    return;
  }
  float scale_out = 1.f;
  if (sinks) {
    const float sink2 = sinks[h] * 1.4426950408889634f;
    const float m_new = fmaxf(m_run, sink2);
    scale_out = __builtin_amdgcn_exp2f(m_run - m_new);
    l_run = l_run * scale_out + __builtin_amdgcn_exp2f(sink2 - m_new);
  }
  scale_out *= 1.0f / l_run;
  bf16_t* row = out + ((long long)tok_begin + my_qi) * out_stride + h * D + hf * 8;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      // the lower lanes of a pair take the dims of j, the upper those of j + 1
      const f32x16& v = o[db];
      const auto lo = __builtin_amdgcn_permlane32_swap(
          bf16_pair(v[4 * j] * scale_out, v[4 * j + 1] * scale_out),
          bf16_pair(v[4 * j + 4] * scale_out, v[4 * j + 5] * scale_out), false, false);
      const auto hi = __builtin_amdgcn_permlane32_swap(
          bf16_pair(v[4 * j + 2] * scale_out, v[4 * j + 3] * scale_out),
          bf16_pair(v[4 * j + 6] * scale_out, v[4 * j + 7] * scale_out), false, false);
      if (my_qi < n_new) *(uint4*)(row + db * 32 + j * 8) = make_uint4(lo[0], hi[0], lo[1], hi[1]);
    }
#endif
}
#endif  // RLIS_HEAD_DIM
