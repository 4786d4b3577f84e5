// Paged "extend" attention, 8-wave 32x32-MFMA kernel (gfx950), for large q
// tiles: one workgroup = 8 waves = a 256-row Q tile of one (seq, q-head); each
// wave owns 32 q rows. K/V are iterated in 64-key tiles.
//
// What bounds it are the matrix cores (55 % busy, and with them the chip's
// power) and, as much again, the softmax between them. So the waves form two
// groups of four, one wave of each per SIMD, that take turns: while one
// multiplies (scores of the next tile, then this tile's weighted values), the
// other works out its softmax, and a barrier swaps them. Tiles go from memory
// straight into LDS three tiles ahead (no registers, no copies); a multiplying
// wave reads its operands between the matrix operations. 28/4 heads x 128, 1 x
// 8192 rows: 475 us (1013 TFLOP/s); with all waves in step, tiles through
// registers and a drained queue at each tile 628. D 64, 32/8 heads: 369 (430).
//
// QK^T uses swapped operands on v_mfma_f32_32x32x16_bf16 (A = K-tile,
// B = Q) so each lane's C fragment holds 16 scores for ONE q-row
// (col = lane&31); the online softmax is then fully in-register: row max =
// in-lane tree + one swap of halves, P stays in VGPRs and is
// packed into the PV A-fragment with v_cvt_pk_bf16_f32 + permlane32_swap
// (16 cvt_pk + 8 swaps per 64-key tile) — no P round trip through LDS.
// V is read with ds_read_b64_tr_b16. O-accumulator rescale is skipped while
// the running max is within RESCALE_THR of the tile max (defer-max).
//
// Which waits make it safe (slot: the time between two barriers): a tile's
// loads are waited for by the wave that asked for them at the end of a softmax
// slot, both groups' slots ending before the first one reads its keys; the
// tile's stage is loaded again from the multiplying slot after the one that
// read its values, behind both groups' barriers.
//
// Sliding-window attention: `window > 0` restricts visibility to the last
// `window` key positions per query (Mistral-style); the KV loop starts at
// the first tile any of this workgroup's rows can see.
//
// BIASED: a distance bias slopes[h] * (i - j) off the scaled scores (the
// score accumulators start from it) and a sink of a score per head
// (sink_w[h]: the running softmax starts from it).
//
// SKIP: waves without rows only help to stage: 65 rows over 6113 keys in 8
// parts 34 us, with their masked scores worked out more. Launches without
// split tiles go without that branch (whole prompts are mostly full tiles).
//
// This is the prefix-caching / chunked-prefill attention of the runtime
// slot (the reference delegates it to vLLM/SGLang images
// at arksapplication_controller.go:941-1002).
#include "common.h"

#include <cfloat>
#include <type_traits>

namespace arks {

typedef __attribute__((ext_vector_type(8))) __bf16 e2_bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 e2_bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

__device__ __forceinline__ f32x16 e2_mfma32(e2_bf16x8 a, e2_bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

constexpr int E2_WAVES = 8;
constexpr int E2_QTILE = 256;      // q rows per workgroup (32 per wave)
constexpr int E2_KVBLK = 64;       // keys per LDS tile
constexpr int E2_PAGE = 16;        // KV page size (tokens)
constexpr float E2_LOG2E = 1.44269504088896340736f;
constexpr float RESCALE_THR = 8.f; // defer-max threshold (exp2 domain)

// v_cvt_pk_bf16_f32: pack two f32 into one dword of two bf16 (RNE).
__device__ __forceinline__ uint32_t cvt_pk_bf16(float lo, float hi) {
  uint32_t r;
  asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
  return r;
}

constexpr int E2_STAGES = 4;  // K and V tiles in LDS

typedef __attribute__((ext_vector_type(4))) int e2_buffer;

__device__ __forceinline__ e2_buffer e2_buffer_of(const void* p) {
  const uint64_t at = reinterpret_cast<uint64_t>(p);
  return e2_buffer{(int)at, (int)(at >> 32) & 0xffff, -1, 0x00027000};
}
// 1 KB of a buffer into LDS, 16 B a lane (the second: another one behind it).
// In asm, since the compiler would wait for all such loads before every
// transposed read of LDS (they write no registers; waits are the caller's).
// s_nop 4: for scalars that a vector instruction wrote last.
__device__ __forceinline__ void e2_load(const e2_buffer& b, const uint32_t to,
                                        const uint32_t offset) {
  asm volatile(
      "s_nop 4\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(to), "v"(offset), "s"(b)
      : "memory", "m0");
}
__device__ __forceinline__ void e2_load(const e2_buffer& b, const uint32_t to,
                                        const uint32_t offset,
                                        const uint32_t offset_2) {
  asm volatile(
      "s_nop 4\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %2, %4, 0 offen lds\n\t"
      "s_mov_b32 m0, %1\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %3, %4, 0 offen lds" ::"s"(to), "s"(to + 1024),
      "v"(offset), "v"(offset_2), "s"(b)
      : "memory", "m0");
}
// The next N matrix operations go out with R reads of LDS behind each.
template <int N, int R>
__device__ __forceinline__ void e2_interleave() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, R, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ e2_bf16x4 e2_read_tr(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
      (__attribute__((address_space(3))) e2_bf16x4*)p);
}
__device__ __forceinline__ void e2_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
// at most N loads under way (all before: !more), LDS reads and writes done
template <int N>
__device__ __forceinline__ void e2_wait(const bool more) {
  __builtin_amdgcn_sched_barrier(0);
  if (more) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
  else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}
__device__ __forceinline__ float e2_max3(const float a, const float b,
                                         const float c) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}
// over the two halves of a wave
__device__ __forceinline__ float e2_halves_max(const float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x),
                                                  __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float e2_halves_sum(const float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x),
                                                  __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The head and tile of a workgroup. Workgroups go round the XCDs in launch
// order. An XCD keeps to as few key/value heads as it can, so that their tiles
// meet in its L2: heads that 8 is a multiple of take 8 / heads XCDs each,
// multiples of 8 go round.
struct E2Place {
  int h, y;
};
__device__ __forceinline__ E2Place e2_place(const int num_q_heads,
                                            const int num_kv_heads) {
  const int gq = num_q_heads / num_kv_heads, xcd = blockIdx.x % 8;
  int at = blockIdx.x / 8, kvh;
  if (8 % num_kv_heads == 0) {
    const int per = 8 / num_kv_heads;
    kvh = xcd / per;
    at = at * per + xcd % per;
  } else if (num_kv_heads % 8 == 0) {
    const int per = num_kv_heads / 8;
    kvh = xcd * per + at / gq % per;
    at = at / (gq * per) * gq + at % gq;
  } else {
    const int all = blockIdx.x % num_q_heads;
    kvh = all / gq;
    at = blockIdx.x / num_q_heads * gq + all % gq;
  }
  return E2Place{kvh * gq + at % gq, at / gq};
}
// Workgroups for so many tiles of every head: where heads share XCDs, 8 times
// those of the fullest one (the places behind the last tile return).
static inline int e2_grid(const int num_q_heads, const int num_kv_heads,
                          const int tiles) {
  const int per_head = num_q_heads / num_kv_heads * tiles;
  return 8 % num_kv_heads == 0
             ? 8 * ((per_head + 8 / num_kv_heads - 1) / (8 / num_kv_heads))
             : num_q_heads * tiles;
}

template <int HEAD_DIM, bool BIASED, bool SKIP>
__global__ __launch_bounds__(512, 2) void attn_extend2_kernel(
    bf16* __restrict__ out,            // [Tq, Hq, D]
    const bf16* __restrict__ q,        // [Tq, Hq, D] (packed new tokens)
    const bf16* __restrict__ k_cache,  // [nblocks, Hkv, 16, D]
    const bf16* __restrict__ v_cache,  // [nblocks, Hkv, 16, D]
    const int* __restrict__ block_tables,  // [num_seqs, max_blocks]
    const int* __restrict__ kv_lens,       // [num_seqs]
    const int* __restrict__ cu_seqlens_q,  // [num_seqs + 1]
    // [ntiles, 4] = (seq_idx, q0, part_idx, nparts): nparts > 1 splits the
    // KV range flash-decode-style; partials go to `part_ws` and a combine
    // kernel merges them (load balance: causal q-tiles differ 4x in KV
    // depth and small batches leave the chip half idle otherwise)
    const int* __restrict__ tile_info,
    float* __restrict__ part_ws,  // [ntiles, Hq, QTILE, D+2] f32 slabs
    const float scale, const int num_q_heads, const int num_kv_heads,
    const int max_blocks, const int64_t q_stride, const int window,
    const int sink,
    // keys per cache row: a key row holds `maps` keys of D dims side by
    // side that share the row's value (k_cache [nblocks, Hkv / maps, 16,
    // maps * D], v_cache [nblocks, Hkv / maps, 16, D]); key group g reads
    // key g % maps of the rows of head g / maps
    const int maps,
    // BIASED: [Hq] each, or null
    const float* __restrict__ sink_w, const float* __restrict__ slopes,
    const int num_tiles) {
  constexpr int STEPS = HEAD_DIM / 16;   // QK^T K-contraction steps
  constexpr int DTILES = HEAD_DIM / 32;  // 32-dim output tiles
  constexpr int ROWB = HEAD_DIM * 2;     // bytes of a row
  constexpr int PIECES = ROWB / 16;      // 16-byte pieces of it
  constexpr int KBYTES = E2_KVBLK * ROWB, STAGE = 2 * KBYTES;
  constexpr int HALF_LOADS = KBYTES / 8192;  // loads of K of a wave and tile
  constexpr int LOADS = 2 * HALF_LOADS;      // with V's
  // how the pieces of row r are permuted (xor), see below
  auto k_turn = [](const int r) {
    return HEAD_DIM == 128 ? r & 15 : (r >> 1) & 7;
  };
  auto v_turn = [](const int r) {
    return HEAD_DIM == 128 ? (r & 3) << 2 : (r & 2) << 1;
  };

  const E2Place place = e2_place(num_q_heads, num_kv_heads);
  const int h = place.h, y = place.y;
  if (y >= num_tiles) return;
  const int kvh = h / (num_q_heads / num_kv_heads);
  const int seq_idx = tile_info[y * 4];
  const int q0 = tile_info[y * 4 + 1];
  const int part = tile_info[y * 4 + 2];
  const int nparts = tile_info[y * 4 + 3];
  const int q_start = cu_seqlens_q[seq_idx];
  const int q_len = cu_seqlens_q[seq_idx + 1] - q_start;
  const int kv_len = kv_lens[seq_idx];
  const int kv_off = kv_len - q_len;  // cached-prefix length
  const int* __restrict__ bt = block_tables + (int64_t)seq_idx * max_blocks;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int lane = tid % WAVE_SIZE;
  const int col = lane & 31;   // q-row within wave (QK^T) / dim col (PV)
  const int half = lane >> 5;  // lane half

  // E2_STAGES of [64 key rows][64 value rows]. Their 16-byte pieces are
  // permuted so that what LDS serves in a cycle lies on all of its banks: 16
  // lanes of a key read (16 rows, one piece), 32 of a transposed value read (4
  // rows, two neighbouring units of 32 bytes). With permutations that did so
  // for 8 and 16 lanes half of LDS' busy cycles were conflicts (1 x 8192 rows
  // 504 us, now 488).
  extern __shared__ __attribute__((aligned(1024))) char lds[];

  const uint32_t lds_at = (uint32_t)reinterpret_cast<uint64_t>(
      (__attribute__((address_space(3))) char*)lds);

  // --- Q fragments (registers, loaded once): lane's q-row = q0+32w+col,
  // frag s holds dims 16s+8*half .. +7.
  const int my_qrow = q0 + wave * 32 + col;
  const bool qrow_valid = my_qrow < q_len;
  const int my_pos = kv_off + my_qrow;  // global kv position of this q row
  e2_bf16x8 qfrag[STEPS];
  {
    const int64_t qbase =
        (int64_t)(q_start + (qrow_valid ? my_qrow : 0)) * q_stride +
        (int64_t)h * HEAD_DIM + 8 * half;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      ushort8 u = *reinterpret_cast<const ushort8*>(q + qbase + s * 16);
      qfrag[s] = *reinterpret_cast<e2_bf16x8*>(&u);
    }
  }

  // Online-softmax state (per lane for q-row `my_qrow`, replicated across
  // the two halves). The running max is kept in RAW score units (scale is
  // folded into the exp2 argument); masked scores use a sentinel so far
  // below any real score that exp2(fma(sentinel, scale2, -m*scale2))
  // underflows to 0 with no per-element select.
  constexpr float MASKED = -3e38f;
  // sink (a value-less key of score 0 in every softmax): the first KV part
  // of a tile starts from (max 0, sum 1); the flash merge of split tiles
  // then carries it like any other key
  float m_run = (sink && part == 0) ? 0.f : -1e30f;
  float l_run = (sink && part == 0) ? 1.f : 0.f;
  // in raw score units, like the running max
  const float slope = BIASED && slopes ? slopes[h] / scale : 0.f;
  if (BIASED && sink_w && part == 0) {
    m_run = sink_w[h] / scale;
    l_run = 1.f;
  }
  f32x16 oacc[DTILES];
#pragma unroll
  for (int n = 0; n < DTILES; ++n) oacc[n] = {};

  const int kmax = min(kv_len, kv_off + q0 + E2_QTILE);
  const int all_tiles = (kmax + E2_KVBLK - 1) / E2_KVBLK;
  // Sliding window: the first key visible to any row of this tile.
  const int jw =
      (window > 0) ? max(0, (kv_off + q0 - window + 1) / E2_KVBLK) : 0;
  // this part's contiguous slice of the KV tile range
  const int span = all_tiles - jw;
  const int per = (span + nparts - 1) / nparts;
  const int j0 = jw + part * per;
  const int ntiles = min(all_tiles, j0 + per);
  const float scale2 = scale * E2_LOG2E;

  // Staging: a wave loads rows 8 * wave .. + 7 of K and V, which lie in one
  // page.
  const int64_t page_rows = (int64_t)(num_kv_heads / maps) * E2_PAGE;
  const int64_t head_row = (int64_t)(kvh / maps) * E2_PAGE;
  const int64_t kstride = (int64_t)maps * HEAD_DIM;
  const int kcol = (kvh % maps) * HEAD_DIM;
  uint32_t koff[HALF_LOADS], voff[HALF_LOADS];
#pragma unroll
  for (int i = 0; i < HALF_LOADS; ++i) {
    const int r = (i * WAVE_SIZE + lane) / PIECES, p = lane % PIECES;
    const int row = 8 * (wave & 1) + r;
    koff[i] = (row * (int)kstride + kcol) * 2 + (p ^ k_turn(row)) * 16;
    voff[i] = row * ROWB + (p ^ v_turn(row)) * 16;
  }
  auto whole = [&](const int j) { return (j + 1) * E2_KVBLK <= kmax; };
  // window-dropped pages are -1 in the block table; sanitized to 0 (their
  // tokens are masked out)
  auto page_of = [&](const int j) {
    return max(0, bt[j * (E2_KVBLK / E2_PAGE) + wave / 2]);
  };
  auto load_tile = [&](const int j, const int page, const int stage) {
    const int64_t row0 = page * page_rows + head_row;
    const e2_buffer kb = e2_buffer_of(k_cache + row0 * kstride);
    const e2_buffer vb = e2_buffer_of(v_cache + row0 * HEAD_DIM);
    const uint32_t to = lds_at + stage * STAGE + wave * 8 * ROWB;
    if constexpr (HALF_LOADS == 2) {
      e2_load(kb, to, koff[0], koff[1]);
      e2_load(vb, to + KBYTES, voff[0], voff[1]);
    } else {
      e2_load(kb, to, koff[0]);
      e2_load(vb, to + KBYTES, voff[0]);
    }
  };
  // The last tile where keys end inside it: rows behind them count as zero (a
  // page's stale rows may hold anything, and 0 * inf is not 0).
  auto load_tail = [&](const int j, const int stage) {
    char* to = lds + stage * STAGE + wave * 8 * ROWB + lane * 16;
#pragma unroll
    for (int i = 0; i < HALF_LOADS; ++i) {
      const int r = (i * WAVE_SIZE + lane) / PIECES;
      const int kg = j * E2_KVBLK + 8 * wave + r;
      ushort8 kv{}, vv{};
      if (kg < kmax) {
        const int64_t row0 = max(0, bt[kg / E2_PAGE]) * page_rows + head_row;
        kv = *reinterpret_cast<const ushort8*>(
            reinterpret_cast<const char*>(k_cache + row0 * kstride) + koff[i]);
        vv = *reinterpret_cast<const ushort8*>(
            reinterpret_cast<const char*>(v_cache + row0 * HEAD_DIM) + voff[i]);
      }
      *reinterpret_cast<ushort8*>(to + i * 1024) = kv;
      *reinterpret_cast<ushort8*>(to + KBYTES + i * 1024) = vv;
    }
  };

  const bool has_rows = __builtin_amdgcn_readfirstlane(q0 + wave * 32) < q_len;
  const int wrow0 = q0 + wave * 32;  // this wave's first row
  // ---- QK^T (swapped): A = K rows (32 keys), B = Q. C[key][qrow=col].
  // The two subtiles interleave so consecutive MFMAs hit independent
  // accumulators (the 32x32 dependent-accumulator latency exceeds the
  // 32-cycle issue interval).
  ushort8 kf[STEPS][2];
  f32x16 sc[2];
  const int k_lane = col * ROWB + ((half ^ k_turn(col)) << 4);
  auto read_k = [&](const int stage, const int s0, const int s1) {
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int sub = 0; sub < 2 && s >= s0 && s < s1; ++sub)
        kf[s][sub] = *reinterpret_cast<const ushort8*>(
            lds + (stage * STAGE + (k_lane ^ (s << 5)) + sub * 32 * ROWB));
  };
  auto score = [&](const int j, const int s0, const int s1) {
    if (s0 == 0) {
      sc[0] = {};
      sc[1] = {};
      if constexpr (BIASED) {
        const float b0 = -slope * (float)(my_pos - j * E2_KVBLK - 4 * half);
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int r16 = 0; r16 < 16; ++r16)
            sc[sub][r16] = __builtin_fmaf(
                slope, (float)(32 * sub + 8 * (r16 >> 2) + (r16 & 3)), b0);
      }
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      if (s < s0 || s >= s1) continue;
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
        sc[sub] = e2_mfma32(*reinterpret_cast<e2_bf16x8*>(&kf[s][sub]), qfrag[s],
                            sc[sub]);
    }
  };

  // ---- Masked softmax, fully in-register (exp2 domain). Lane's 32
  // scores are all for q-row `my_qrow`; C reg 4g+r of subtile `sub` is
  // key key_base + 32*sub + 8g + 4*half + r. Tiles fully visible to
  // every row of this wave (the bulk of the causal region) skip the 32
  // per-key compares; the reductions are trees, not 31-deep chains.
  const int last_key = qrow_valid ? min(my_pos, kmax - 1) : -1;
  const int first_key = window > 0 ? my_pos - window + 1 : 0;
  uint32_t afrag[4][4];  // [k-step t][4 dwords = 8 bf16]
  auto softmax = [&](const int j) {
    const int key_base = j * E2_KVBLK;
    const bool full_vis =
        (wrow0 + 31 < q_len) && (key_base + E2_KVBLK - 1 <= kv_off + wrow0) &&
        (key_base + E2_KVBLK <= kmax) &&
        (window <= 0 || key_base > kv_off + wrow0 + 31 - window);
    if (!full_vis) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int kb_s = key_base + 32 * sub + 4 * half;
#pragma unroll
        for (int r16 = 0; r16 < 16; ++r16) {
          const int kg = kb_s + 8 * (r16 >> 2) + (r16 & 3);
          sc[sub][r16] =
              (kg >= first_key) & (kg <= last_key) ? sc[sub][r16] : MASKED;
        }
      }
    }
    float p[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) p[i] = sc[i / 16][i % 16];
    // (the maximum that NaN goes through: fmaxf would first quiet each score)
    float mt[11];
#pragma unroll
    for (int i = 0; i < 11; ++i)
      mt[i] = i < 10 ? e2_max3(p[3 * i], p[3 * i + 1], p[3 * i + 2])
                     : __builtin_elementwise_maximum(p[30], p[31]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      mt[i] = i < 3 ? e2_max3(mt[3 * i], mt[3 * i + 1], mt[3 * i + 2])
                    : __builtin_elementwise_maximum(mt[9], mt[10]);
    const float tmax = e2_halves_max(
        __builtin_elementwise_maximum(e2_max3(mt[0], mt[1], mt[2]), mt[3]));

    // Defer-max (T13): only rescale O when the tile max meaningfully
    // exceeds the running max (threshold in raw units; exp2(THR)=256
    // stays comfortably finite).
    const float thr_raw = RESCALE_THR / scale2;
    if (!__all(tmax - m_run <= thr_raw)) {
      const float m_new = fmaxf(m_run, tmax);
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * scale2);
      l_run *= alpha;
      m_run = m_new;
      // O rows live across regs (C layout): fetch each row's alpha from
      // the lane that owns that q-row.
#pragma unroll
      for (int r16 = 0; r16 < 16; ++r16) {
        const int row = 8 * (r16 >> 2) + 4 * half + (r16 & 3);
        const float a_r = __shfl(alpha, 32 * (lane >> 5) + row, WAVE_SIZE);
#pragma unroll
        for (int n = 0; n < DTILES; ++n) oacc[n][r16] *= a_r;
      }
    }

    // p = exp2((s - m) * scale2) as one fma + exp2; MASKED entries
    // underflow to exactly 0 (|MASKED*scale2| >> |m*scale2|).
    const float nms = -m_run * scale2;
#pragma unroll
    for (int i = 0; i < 32; ++i)
      p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[i], scale2, nms));
    float st[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) st[i] = p[i] + p[i + 16];
#pragma unroll
    for (int w = 8; w > 0; w >>= 1)
#pragma unroll
      for (int i = 0; i < w; ++i) st[i] += st[i + w];
    l_run += e2_halves_sum(st[0]);

    // ---- P -> bf16 PV A-fragments: per subtile, 8 cvt_pk words
    // W[g][0] = pk(p[4g], p[4g+1]), W[g][1] = pk(p[4g+2], p[4g+3]); the
    // permlane32_swap pairs (W[2t][*], W[2t+1][*]) then give each half its
    // step-t fragment from both halves' key sets.
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      uint32_t w0[4], w1[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int b = sub * 16 + 4 * g;
        w0[g] = cvt_pk_bf16(p[b + 0], p[b + 1]);
        w1[g] = cvt_pk_bf16(p[b + 2], p[b + 3]);
      }
#pragma unroll
      for (int tau = 0; tau < 2; ++tau) {
        auto r0 = __builtin_amdgcn_permlane32_swap(w0[2 * tau], w0[2 * tau + 1],
                                                   false, false);
        auto r1 = __builtin_amdgcn_permlane32_swap(w1[2 * tau], w1[2 * tau + 1],
                                                   false, false);
        const int t = sub * 2 + tau;
        afrag[t][0] = r0[0];
        afrag[t][1] = r1[0];
        afrag[t][2] = r0[1];
        afrag[t][3] = r1[1];
      }
    }
  };

  // ---- PV: O[qrow][dim] += P[qrow][key] V[key][dim]; B fragments via
  // tr16 reads of V (per step t: keys 16t+8*half+0..7 at column
  // 16*(colhalf)+l&15: 4-key groups 4t+2*half (+1), 16-column units 2n + one
  // per 16 lanes).
  e2_bf16x8 vf[4][DTILES];
  const int v_row = (lane >> 2) & 3;
  const int v_lane = (8 * half + v_row) * ROWB +
                     (((lane >> 3) & 2) * 16 ^ v_turn(v_row) * 16) +
                     (lane & 3) * 8;
  auto read_v = [&](const int stage, const int t) {
#pragma unroll
    for (int n = 0; n < DTILES; ++n) {
      const char* at = lds + (stage * STAGE + KBYTES + t * 16 * ROWB);
      const e2_bf16x4 v1 = e2_read_tr(at + (v_lane ^ (n << 6)));
      const e2_bf16x4 v2 = e2_read_tr(at + 4 * ROWB + (v_lane ^ (n << 6)));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        vf[t][n][e] = v1[e];
        vf[t][n][e + 4] = v2[e];
      }
    }
  };
  // t outer / n inner: consecutive MFMAs accumulate into the DTILES
  // independent oacc registers instead of chaining one.
  auto weigh = [&](const int t) {
#pragma unroll
    for (int n = 0; n < DTILES; ++n)
      oacc[n] = e2_mfma32(*reinterpret_cast<e2_bf16x8*>(&afrag[t][0]), vf[t][n],
                          oacc[n]);
  };

  if (j0 < ntiles) {
    auto load = [&](const int j, const int page, const int stage) {
      if (whole(j)) load_tile(j, page, stage);
      else load_tail(j, stage);
    };
#pragma unroll
    for (int t = 0; t < E2_STAGES - 1; ++t)
      if (j0 + t < ntiles)
        load(j0 + t, whole(j0 + t) ? page_of(j0 + t) : 0, t);
    // the first two tiles are there, the third may be under way
    e2_wait<LOADS>(j0 + 2 < ntiles && whole(j0 + 2));
    e2_barrier();
    // (the scores of a tile behind the last are worked out too, from whatever
    // its stage holds, and not used)
    const bool works = !SKIP || has_rows;
    if (works) {
      read_k(0, 0, STEPS);
      score(j0, 0, STEPS);
    }
    if (wave >= 4) e2_barrier();  // the second group runs one slot behind
    int st = 0;
    auto turn = [&](const int j, auto on) {
      constexpr bool ON = decltype(on)::value;
      auto stage = [&](const int ahead) {
        return st + ahead >= E2_STAGES ? st + ahead - E2_STAGES : st + ahead;
      };
      const int far = j + E2_STAGES - 1;
      const int page = far < ntiles && whole(far) ? page_of(far) : 0;
      // ---- the other group multiplies
      if constexpr (ON) {
        read_k(stage(1), 0, STEPS / 2);
        softmax(j);
      }
      e2_wait<0>(false);  // tile j + 2, asked for two slots ago, is there
      e2_barrier();
      // ---- this group multiplies. Operands are read between the matrix
      // operations, where earlier ones have been used: registers for all of K
      // and V at once would not be there.
      if constexpr (ON) {
        __builtin_amdgcn_s_setprio(1);
        score(j + 1, 0, STEPS / 2);
        read_k(stage(1), STEPS / 2, STEPS);
        e2_interleave<STEPS, 1>();
      }
      if (far < ntiles) load(far, page, stage(E2_STAGES - 1));
      if constexpr (ON) {
        __builtin_amdgcn_sched_barrier(0);
        score(j + 1, STEPS / 2, STEPS);
        read_v(st, 0);
        read_v(st, 1);
        e2_interleave<STEPS, 4 * DTILES / STEPS>();
        weigh(0);
        weigh(1);
        read_v(st, 2);
        read_v(st, 3);
        e2_interleave<2 * DTILES, 2>();
        weigh(2);
        weigh(3);
        __builtin_amdgcn_s_setprio(0);
      }
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      e2_barrier();
      st = stage(1);
    };
    if (works)
      for (int j = j0; j < ntiles; ++j) turn(j, std::true_type{});
    else
      for (int j = j0; j < ntiles; ++j) turn(j, std::false_type{});
    if (wave < 4) e2_barrier();
  }

  // ---- Epilogue. O reg 4g+r of dim-tile n is q-row 8g+4*half+r, dim
  // 32n+col; l_run for row `row` lives in lane row (either half).
  if (nparts > 1) {
    // partial: UNNORMALIZED O + per-row (m, l) into this part's slab
    // [QTILE rows][D+2] f32 (combined by attn_extend2_combine)
    float* slab = part_ws +
        ((int64_t)y * num_q_heads + h) * E2_QTILE * (HEAD_DIM + 2);
#pragma unroll
    for (int r16 = 0; r16 < 16; ++r16) {
      const int row = 8 * (r16 >> 2) + 4 * half + (r16 & 3);
      if (q0 + wave * 32 + row >= q_len) continue;
      float* wr = slab + (int64_t)(wave * 32 + row) * (HEAD_DIM + 2) + col;
#pragma unroll
      for (int n = 0; n < DTILES; ++n) wr[32 * n] = oacc[n][r16];
    }
    if (half == 0) {
      // lane `col` owns q-row `col` of this wave: write its m/l
      float* wr = slab + (int64_t)(wave * 32 + col) * (HEAD_DIM + 2);
      wr[HEAD_DIM] = m_run;
      wr[HEAD_DIM + 1] = l_run;
    }
    return;
  }
#pragma unroll
  for (int r16 = 0; r16 < 16; ++r16) {
    const int row = 8 * (r16 >> 2) + 4 * half + (r16 & 3);
    const int qrow = q0 + wave * 32 + row;
    const float lr = __shfl(l_run, 32 * (lane >> 5) + row, WAVE_SIZE);
    if (qrow >= q_len) continue;
    const float inv = lr > 0.f ? 1.f / lr : 0.f;
    const int64_t obase =
        ((int64_t)(q_start + qrow) * num_q_heads + h) * HEAD_DIM + col;
#pragma unroll
    for (int n = 0; n < DTILES; ++n) {
      out[obase + 32 * n] = float_to_bf16_bits(oacc[n][r16] * inv);
    }
  }
}

// Merge the flash partials of split tiles: a workgroup has a head, a split tile
// and 8 of its rows (LOCAL: heads as in the kernel above); combine_table rows = (first_y, nparts, seq, q0).
// Standard flash merge in f32: m* = max m_p; out = sum_p exp(m_p - m*) O_p / sum_p
// exp(m_p - m*) l_p (m is base-2: exp2). Reading the slabs bounds it, so the
// loads of 2, 4 or 8 parts, as many as there are, are in flight together, two
// dims a thread. Tiles of 3 parts, 28 heads, chunks of up to 2048 rows: 14.2 us
// on the mean (90 MB at the most; with 8 loads for any number of parts 23.2).
// A head's workgroups are on the XCD that wrote its slabs, where one did:
// read on another one, their next writing was slower too (32/8 heads, 256 rows
// behind 5000 keys in 8 parts: 22.4 + 7.3 us with a window of 1024, now 19.8 +
// 7.0; of 128, 19.6 + 7.2, now 15.4 + 7.1).
template <int HEAD_DIM, int PARTS>
__device__ __forceinline__ void e2_combine_rows(
    bf16* __restrict__ to, const float* __restrict__ base,
    const int64_t slab_stride, const int64_t out_stride, const int row0,
    const int rows, const int nparts, const float scale2) {
  constexpr int TPR = HEAD_DIM / 2;  // threads of a row
  const int d = threadIdx.x % TPR * 2;
  for (int i = threadIdx.x / TPR; i < 8; i += 256 / TPR) {
    const int row = row0 + i;
    if (row >= rows) continue;
    const float* r0 = base + (int64_t)row * (HEAD_DIM + 2);
    float m_star = -1e30f, l_tot = 0.f, acc0 = 0.f, acc1 = 0.f;
    for (int p0 = 0; p0 < nparts; p0 += PARTS) {
      float2 ml[PARTS], v[PARTS];
#pragma unroll
      for (int p = 0; p < PARTS; ++p) {
        const float* r = r0 + (int64_t)min(p0 + p, nparts - 1) * slab_stride;
        ml[p] = *reinterpret_cast<const float2*>(r + HEAD_DIM);
        v[p] = *reinterpret_cast<const float2*>(r + d);
      }
      float m_new = m_star;
#pragma unroll
      for (int p = 0; p < PARTS; ++p) m_new = fmaxf(m_new, ml[p].x);
      const float keep = __builtin_amdgcn_exp2f((m_star - m_new) * scale2);
      l_tot *= keep;
      acc0 *= keep;
      acc1 *= keep;
      m_star = m_new;
#pragma unroll
      for (int p = 0; p < PARTS; ++p) {
        const float e = __builtin_amdgcn_exp2f((ml[p].x - m_star) * scale2);
        const float a = p0 + p < nparts ? e : 0.f;
        l_tot += a * ml[p].y;
        acc0 += a * v[p].x;
        acc1 += a * v[p].y;
      }
    }
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    const uint32_t two = (uint32_t)float_to_bf16_bits(acc0 * inv) |
                         ((uint32_t)float_to_bf16_bits(acc1 * inv) << 16);
    *reinterpret_cast<uint32_t*>(to + row * out_stride + d) = two;
  }
}

template <int HEAD_DIM, bool LOCAL>
__global__ __launch_bounds__(256) void attn_extend2_combine_kernel(
    bf16* __restrict__ out, const float* __restrict__ part_ws,
    const int* __restrict__ combine_table,
    const int* __restrict__ cu_seqlens_q, const float scale,
    const int num_q_heads, const int num_kv_heads, const int n_split) {
  int h = blockIdx.x, tile = blockIdx.y, group = blockIdx.z;
  if constexpr (LOCAL) {
    const E2Place place = e2_place(num_q_heads, num_kv_heads);
    h = place.h, tile = place.y % n_split, group = place.y / n_split;
    if (group >= E2_QTILE / 8) return;
  }
  const int* entry = combine_table + tile * 4;
  const int nparts = entry[1], seq_idx = entry[2], q0 = entry[3];
  const int q_start = cu_seqlens_q[seq_idx];
  const int q_len = cu_seqlens_q[seq_idx + 1] - q_start;
  const int64_t slab_stride = (int64_t)num_q_heads * E2_QTILE * (HEAD_DIM + 2);
  const float* base = part_ws + (int64_t)entry[0] * slab_stride +
                      (int64_t)h * E2_QTILE * (HEAD_DIM + 2);
  const int64_t out_stride = (int64_t)num_q_heads * HEAD_DIM;
  bf16* to = out + (q_start + q0) * out_stride + (int64_t)h * HEAD_DIM;
  const int row0 = group * 8, rows = q_len - q0;
  const float scale2 = scale * E2_LOG2E;
#define ARKS_ROWS(P)                                                         \
  e2_combine_rows<HEAD_DIM, P>(to, base, slab_stride, out_stride, row0, rows, \
                               nparts, scale2)
  if (nparts <= 2) ARKS_ROWS(2);
  else if (nparts <= 4) ARKS_ROWS(4);
  else ARKS_ROWS(8);
#undef ARKS_ROWS
}

}  // namespace arks

using namespace arks;

extern "C" void arks_attn_extend_paged2(
    void* out, const void* q, const void* k_cache, const void* v_cache,
    const void* block_tables, const void* kv_lens, const void* cu_seqlens_q,
    const void* tile_info, void* part_ws, int ntiles, float scale,
    int num_q_heads, int num_kv_heads, int head_dim, int max_blocks,
    int64_t q_stride, int window, int sink, int maps, const void* sink_w,
    const void* slopes, hipStream_t stream) {
  const int grid = e2_grid(num_q_heads, num_kv_heads, ntiles);
  const dim3 block(512);
  static bool attr_set[6] = {};
  auto launch = [&](auto kern, int lds_bytes, int idx) {
    if (!attr_set[idx]) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          lds_bytes);
      attr_set[idx] = true;
    }
    hipLaunchKernelGGL(kern, dim3(grid), block, lds_bytes, stream, (bf16*)out,
                       (const bf16*)q, (const bf16*)k_cache,
                       (const bf16*)v_cache, (const int*)block_tables,
                       (const int*)kv_lens, (const int*)cu_seqlens_q,
                       (const int*)tile_info, (float*)part_ws, scale,
                       num_q_heads, num_kv_heads, max_blocks, q_stride,
                       window, sink, maps, (const float*)sink_w,
                       (const float*)slopes, ntiles);
  };
  if (head_dim == 128) {
    constexpr int LDS = E2_STAGES * 2 * 64 * 128 * 2;
    if (sink_w || slopes) launch(attn_extend2_kernel<128, true, true>, LDS, 2);
    else if (part_ws) launch(attn_extend2_kernel<128, false, true>, LDS, 4);
    else launch(attn_extend2_kernel<128, false, false>, LDS, 0);
  } else if (head_dim == 64) {
    constexpr int LDS = E2_STAGES * 2 * 64 * 64 * 2;
    if (sink_w || slopes) launch(attn_extend2_kernel<64, true, true>, LDS, 3);
    else if (part_ws) launch(attn_extend2_kernel<64, false, true>, LDS, 5);
    else launch(attn_extend2_kernel<64, false, false>, LDS, 1);
  }
}

extern "C" void arks_attn_extend2_combine(
    void* out, const void* part_ws, const void* combine_table,
    const void* cu_seqlens_q, int n_split, float scale, int num_q_heads,
    int num_kv_heads, int head_dim, hipStream_t stream) {
  if (n_split == 0) return;
  constexpr int GROUPS = E2_QTILE / 8;
  // heads whose slabs one XCD wrote (where a group of them goes unevenly over
  // XCDs, every other slab of a head is on another one, and launch order without
  // the divisions is as fast: 28/4 heads, 2017 rows in 3 parts 15.3 us and 15.6)
  const bool local =
      num_kv_heads % 8 == 0 ||
      (8 % num_kv_heads == 0 &&
       num_q_heads / num_kv_heads % (8 / num_kv_heads) == 0);
  const dim3 grid = local ? dim3(e2_grid(num_q_heads, num_kv_heads,
                                         n_split * GROUPS))
                          : dim3(num_q_heads, n_split, GROUPS);
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream, (bf16*)out,
                       (const float*)part_ws, (const int*)combine_table,
                       (const int*)cu_seqlens_q, scale, num_q_heads,
                       num_kv_heads, n_split);
  };
  if (head_dim == 128 && local) launch(attn_extend2_combine_kernel<128, true>);
  else if (head_dim == 128) launch(attn_extend2_combine_kernel<128, false>);
  else if (head_dim == 64 && local) launch(attn_extend2_combine_kernel<64, true>);
  else if (head_dim == 64) launch(attn_extend2_combine_kernel<64, false>);
}
