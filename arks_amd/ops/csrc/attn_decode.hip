// Paged decode attention for CDNA4 (gfx950), flash-decode style: every query
// row (one per sequence) over its sequence's paged keys and values.
//
// What bounds it is the KV stream (one read of every page, at HBM rate), and
// the length of the longest chain of dependent loads: a batch holds contexts
// of very different lengths, and a decode graph fixes the grid before they
// are known. So the work is cut by what it is and not by the grid: a unit is
// 32 tokens (2 pages) of one sequence; the units of all sequences are one
// line, cut into runs of equal length (where runs hold many short sequences,
// the start of each counts too), one run per WAVE, 4 or 8 waves per CU. A run that covers a whole sequence writes its rows of the output, any other
// an f32 partial (acc, m, l), and attn_decode_combine merges a sequence's
// partials. Waves share nothing: no barrier. The runs depend on the lengths
// alone, so attn_decode_plan finds them once for all layers of a step:
//   plan [waves] {sequence, first unit in it, its length, units of the run}
//        [S]     {first run, runs}
//   (found by every workgroup for itself they cost each layer ~8 us).
//
// Within a unit all GQ query heads of the group are the columns of one MFMA
// chain: QK^T takes K straight from the cache pages as the A operand (16 B,
// fp8: 8 B per lane), the column-wise online softmax costs two shuffles for
// all heads at once, V goes through a per-wave LDS image that the transpose
// reads of the PV product expect. A wave holds the raw K and V of two units
// in registers: the loads of unit i+2 are issued when unit i has been
// consumed, and fp8 bytes become bf16 (exact, two per instruction) only when
// they are used, so that no conversion waits for a load in flight. (One unit
// per wave and 12 waves per CU spilled and was slower, 108 us for the ragged
// batch below.)
//
// Reading the same pages without any arithmetic reaches 5.3-5.6 TB/s at 1 to
// 2 workgroups per CU, and less at counts between. 28/4 heads x 128, kernel
// and merge, with a workgroup per (sequence, head, part of the grid) before:
//   64 x 1024, bf16            34.4 -> 31.4 us
//   256 of 1..4000, even, bf16   176 us (5.7 TB/s; units all alike and two
//                              workgroups per CU 183)
//   48 x 900..5000, fp8       140.8 -> 33.3 us (its bytes were converted one
//                              by one, in front of the wait for the next)
//
// Cache layout: [num_blocks, num_kv_heads, BLOCK_SIZE, head_dim] bf16 or
// e4m3. q may be a strided row view into the fused QKV projection.
// Fills the runtime-slot contract of scitix/arks natively.
#include "common.h"

#include <cfloat>

namespace arks {

constexpr int KV_BLOCK_SIZE = 16;  // tokens per KV page (matches engine)

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 dec_bf16x4v;
typedef __attribute__((ext_vector_type(2))) __bf16 dec_bf16x2v;
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ f32x4 dec_mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float dec_exp2(float x) {
  return __builtin_amdgcn_exp2f(x);
}

constexpr int DEC_UNIT = 32;      // tokens per unit (2 KV pages)
constexpr int DEC_VT_PAD = 40;    // padded token axis of the P tile

// 8 values of a cache row as they lie there, and as bf16 (e4m3 values are
// bf16 values: the conversion is exact).
template <bool FP8>
struct DecRaw {
  typedef ushort8 type;
};
template <>
struct DecRaw<true> {
  typedef __attribute__((ext_vector_type(2))) uint32_t type;
};

template <bool FP8>
__device__ __forceinline__ ushort8 dec_bf16(const typename DecRaw<FP8>::type& r) {
  if constexpr (!FP8) {
    return r;
  } else {
    union {
      dec_bf16x2v h[4];
      ushort8 u;
    } c;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      c.h[2 * i] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(r[i], 1.f, false);
      c.h[2 * i + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(r[i], 1.f, true);
    }
    return c.u;
  }
}

// First and one-past-last unit of a sequence: tokens below the window are
// left out (their pages may be gone).
__device__ __forceinline__ int dec_first_unit(int len, int window) {
  return window > 0 && len > window ? (len - window) / DEC_UNIT : 0;
}
__device__ __forceinline__ int dec_units(int len, int window) {
  return len <= 0 ? 0
                  : (len + DEC_UNIT - 1) / DEC_UNIT - dec_first_unit(len, window);
}

// Units per run, from the units of all sequences (total) and of the longest
// one. At least 2, what `waves` waves must take, and enough that merging a
// long sequence's partials (about 0.15 of a unit's time each, one after the
// other) does not outlast the runs themselves.
__device__ __forceinline__ int dec_run_length(int total, int longest, int waves) {
  const int merge = (int)ceilf(sqrtf(0.15f * (float)longest));
  return max(max(2, merge), (total + waves - 1) / waves);
}

// A workgroup of 1024 threads finds every wave's run and every sequence's
// runs (the layout is in the header comment).
__global__ __launch_bounds__(1024) void attn_decode_plan_kernel(
    int* __restrict__ plan, const int* __restrict__ lens, const int n,
    const int window, const int waves) {
  constexpr int NW = 1024 / WAVE_SIZE;
  __shared__ int sums[NW], tops[NW], seqs_in[NW], shorter;
  const int tid = threadIdx.x, lane = tid % WAVE_SIZE, wave = tid / WAVE_SIZE;
  const int per = (n + 1023) / 1024;
  const int s0 = min(n, tid * per), s1 = min(n, s0 + per);
  int mine = 0, longest = 0, some = 0;
  for (int s = s0; s < s1; ++s) {
    const int u = dec_units(lens[s], window);
    mine += u;
    some += u > 0;
    longest = max(longest, u);
  }
  int scan = mine, scan_s = some;
#pragma unroll
  for (int off = 1; off < WAVE_SIZE; off <<= 1) {
    const int v = __shfl_up(scan, off, WAVE_SIZE);
    const int vs = __shfl_up(scan_s, off, WAVE_SIZE);
    if (lane >= off) {
      scan += v;
      scan_s += vs;
    }
    longest = max(longest, __shfl_xor(longest, off, WAVE_SIZE));
  }
  if (lane == WAVE_SIZE - 1) {
    sums[wave] = scan;
    seqs_in[wave] = scan_s;
  }
  if (lane == 0) tops[wave] = longest;
  if (tid == 0) shorter = 0;
  __syncthreads();
  int units = scan - mine, seqs_before = scan_s - some, total = 0, held = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    if (w < wave) {
      units += sums[w];
      seqs_before += seqs_in[w];
    }
    total += sums[w];
    held += seqs_in[w];
    longest = max(longest, tops[w]);
  }
  // Equal runs of units, unless some would hold whole sequences: a run waits for
  // a chain of loads (page ids, then rows) at each sequence that it starts, which
  // counts as one unit more then. 28/4 heads x 128, us with the merge, so (equal
  // units): 200 of 20..4000 (even over the logarithm) 60.6 (64.6), fp8 36.1
  // (40.5); 64 of them 24.8 (26.8); 256 of 20..500 23.1 (24.3); 256 of 1..4000
  // 180 (182). Half a unit gives half of it, two no more.
  const int even = dec_run_length(total, longest, waves);
  int less = 0;
  for (int s = s0; s < s1; ++s) {
    const int u = dec_units(lens[s], window);
    less |= u > 0 && u < even;
  }
  if (less) shorter = 1;
  __syncthreads();
  const int front = shorter;
  const int line = total + held * front;
  const int run = shorter ? max(dec_run_length(0, longest, waves),
                                (line + waves - 1) / waves)
                          : even;
  int at = units + seqs_before * front;
  int4* runs = reinterpret_cast<int4*>(plan);
  int2* seqs = reinterpret_cast<int2*>(plan + 4 * waves);
  // unit j of a sequence lies at `at` + front + j. A run (of 2 places at least)
  // holds a unit, and its length is found from the first units of its neighbours.
  for (int s = s0; s < s1; ++s) {
    const int L = lens[s], u = dec_units(L, window), b = at + front;
    if (u == 0) {
      seqs[s] = make_int2(0, 0);
      continue;
    }
    const int w0 = b / run, w1 = (b + u - 1) / run;
    seqs[s] = make_int2(w0, w1 - w0 + 1);
    // (the unit in front of this sequence lies at `at` - 1)
    for (int w = at == 0 || at - 1 < w0 * run ? w0 : w0 + 1; w <= w1; ++w) {
      const int j = max(0, w * run - b);
      runs[w] = make_int4(s, j, L, units + j);
    }
    at = b + u;
    units += u;
  }
  const int used = (line + run - 1) / run;
  __threadfence_block();
  __syncthreads();
  for (int w0 = 0; w0 < waves; w0 += 1024) {
    const int w = w0 + tid;
    const int first = w < used ? runs[w].w : 0;
    const int next = w + 1 < used ? runs[w + 1].w : total;
    __syncthreads();
    if (w < used) runs[w].w = next - first;
    else if (w < waves) runs[w] = make_int4(0, 0, 0, 0);
  }
}

template <int HEAD_DIM, int GQ, bool KV_FP8>
__global__ __launch_bounds__(256, 2) void attn_decode_kernel(
    bf16* __restrict__ out,         // [S, Hq, D]
    float* __restrict__ part_out,   // [waves + S, Hkv, GQ * D + 16]
    const bf16* __restrict__ q,     // rows of length q_stride
    const bf16* __restrict__ k_cache,  // [B, Hkv, 16, D]
    const bf16* __restrict__ v_cache,
    const int* __restrict__ block_tables,  // [S, max_blocks]
    const int* __restrict__ seq_lens,      // [S]
    const int4* __restrict__ runs, const float scale, const int num_kv_heads,
    const int max_blocks, const int64_t q_stride, const int window,
    const int sink, const int waves, const int num_seqs) {
  constexpr int NUM_WAVES = 4;
  constexpr int STEPS = HEAD_DIM / 32;   // QK^T contraction steps
  constexpr int CHUNKS = HEAD_DIM / 16;  // PV output dim chunks
  constexpr int NV = DEC_UNIT * HEAD_DIM / 8 / WAVE_SIZE;
  constexpr int ROW = HEAD_DIM / 8;      // 8-value groups of a cache row
  constexpr int ESZ = KV_FP8 ? 1 : 2;    // bytes of a cache value
  typedef typename DecRaw<KV_FP8>::type raw;

  // V tr16 image [cb = D/16][kb = 8][96] (64 data + 32 pad) and P tile
  constexpr int VT_ELEMS = (HEAD_DIM / 16) * 8 * 96;
  __shared__ __attribute__((aligned(16))) bf16
      smem[NUM_WAVES][VT_ELEMS + 16 * DEC_VT_PAD];
  const int lane = threadIdx.x % WAVE_SIZE;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lq = lane % 16;
  const int la = lane / 16;
  const int kvh = blockIdx.x % num_kv_heads;
  const int w = blockIdx.x / num_kv_heads * NUM_WAVES + wave;
  if (w >= waves) return;
  const int4 d = runs[w];
  int seq = __builtin_amdgcn_readfirstlane(d.x);
  int off = __builtin_amdgcn_readfirstlane(d.y);  // first unit in it
  int L = __builtin_amdgcn_readfirstlane(d.z);
  int left = __builtin_amdgcn_readfirstlane(d.w);
  if (left == 0) return;

  bf16* vt_lds = smem[wave];
  bf16* p_lds = smem[wave] + VT_ELEMS;
  const float scale2 = scale * 1.44269504088896340736f;  // exp2 domain
  const int num_q_heads = num_kv_heads * GQ;
  const int64_t page_elems = (int64_t)num_kv_heads * KV_BLOCK_SIZE * HEAD_DIM;
  const int64_t head_off = (int64_t)kvh * KV_BLOCK_SIZE * HEAD_DIM;
  // byte offsets of this lane's values (unsigned: scalar base + offset)
  const uint32_t k_lane = (lq * HEAD_DIM + 8 * la) * ESZ;
  const uint32_t v_lane = lane * 8 * ESZ;

  while (true) {
    const int units = dec_units(L, window);
    const int npages = (L + KV_BLOCK_SIZE - 1) / KV_BLOCK_SIZE;
    const int c0 = off + dec_first_unit(L, window);
    const int n = min(left, units - off);
    const int* bt = block_tables + (int64_t)seq * max_blocks;

    // Q fragments: B operand [32k x 16 heads] per step; rows g >= GQ zero
    bf16x8 qfrag[STEPS];
    {
      const bool valid = lq < GQ;
      const bf16* qp = q + (int64_t)seq * q_stride +
                       (kvh * GQ + (valid ? lq : 0)) * HEAD_DIM;
#pragma unroll
      for (int st = 0; st < STEPS; ++st) {
        ushort8 x{};
        if (valid) x = *reinterpret_cast<const ushort8*>(qp + st * 32 + 8 * la);
        qfrag[st] = *reinterpret_cast<bf16x8*>(&x);
      }
    }
    float m_run = -FLT_MAX;  // per head lq (replicated over la)
    float l_run = 0.f;
    f32x4 oacc[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) oacc[c] = {0.f, 0.f, 0.f, 0.f};

    raw kr[2][2][STEPS], vr[2][NV];
    // the rows of unit i of a piece whose page ids lie one per lane. V rows
    // are read once, whole lines at a time: non-temporal (a K load takes half
    // a line, and its other half has to stay)
    auto load = [&](int i, int ids, raw (&k)[2][STEPS], raw (&v)[NV]) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int64_t at =
            ((int64_t)__builtin_amdgcn_readlane(ids, 2 * i + sub) * page_elems +
             head_off) * ESZ;
        const char* kp = reinterpret_cast<const char*>(k_cache) + at;
        const char* vp = reinterpret_cast<const char*>(v_cache) + at;
#pragma unroll
        for (int st = 0; st < STEPS; ++st)
          k[sub][st] = *reinterpret_cast<const raw*>(kp + k_lane + st * 32 * ESZ);
        // the 16 rows of a page are one run of 16 * HEAD_DIM values
#pragma unroll
        for (int j = 0; j < NV / 2; ++j)
          v[sub * (NV / 2) + j] = __builtin_nontemporal_load(reinterpret_cast<const raw*>(
              vp + v_lane + j * WAVE_SIZE * 8 * ESZ));
      }
    };

    auto step = [&](int unit, raw (&kx)[2][STEPS], raw (&vx)[NV]) {
      const int tok0 = (c0 + unit) * DEC_UNIT;
      const int t_hi = L - tok0;  // rows below it hold a visible key ..
      const int t_lo = window > 0 ? L - window - tok0 : 0;  // .. from here
      f32x4 sc[2];
      sc[0] = {0.f, 0.f, 0.f, 0.f};
      sc[1] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
          ushort8 kb = dec_bf16<KV_FP8>(kx[sub][st]);
          sc[sub] = dec_mfma(*reinterpret_cast<bf16x8*>(&kb), qfrag[st], sc[sub]);
        }

      // masked column-wise online softmax (head = lq; tokens in lanes)
      float p[8];
      float tile_max = -FLT_MAX;
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = sub * 16 + 4 * la + r;
          const int x = sub * 4 + r;
          p[x] = t < t_hi && t >= t_lo ? sc[sub][r] * scale2 : -FLT_MAX;
          tile_max = fmaxf(tile_max, p[x]);
        }
      tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 16, WAVE_SIZE));
      tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32, WAVE_SIZE));
      const float m_new = fmaxf(m_run, tile_max);
      float alpha = 1.f, psum = 0.f;
      if (m_new > -FLT_MAX) {
        alpha = dec_exp2(m_run - m_new);
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          p[x] = p[x] > -FLT_MAX ? dec_exp2(p[x] - m_new) : 0.f;
          psum += p[x];
        }
      } else {
#pragma unroll
        for (int x = 0; x < 8; ++x) p[x] = 0.f;
      }
      psum += __shfl_xor(psum, 16, WAVE_SIZE);
      psum += __shfl_xor(psum, 32, WAVE_SIZE);
      l_run = l_run * alpha + psum;
      m_run = m_new;
      // rescale O rows (head = 4*la + r in the PV fragment)
      float row_alpha[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        row_alpha[r] = __shfl(alpha, 4 * la + r, WAVE_SIZE);
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) oacc[c][r] *= row_alpha[r];

      // V into the tr16 image; rows without a visible key count as zero
      // (a page's stale rows may hold anything, and 0 * inf is not 0)
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int e = j * WAVE_SIZE + lane;
        const int t = e / ROW, col8 = (e % ROW) * 8;
        ushort8 x = dec_bf16<KV_FP8>(vx[j]);
        if (t >= t_hi || t < t_lo) x = ushort8{};
        *reinterpret_cast<ushort8*>(
            &vt_lds[((col8 >> 4) * 8 + (t >> 2)) * 96 + (t & 3) * 16 +
                    (col8 & 15)]) = x;
      }
      // P to LDS (bf16), then PV over the unit's 32 tokens
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        ushort4v pk;
#pragma unroll
        for (int r = 0; r < 4; ++r) pk[r] = float_to_bf16_bits(p[sub * 4 + r]);
        *reinterpret_cast<ushort4v*>(
            &p_lds[lq * DEC_VT_PAD + sub * 16 + 4 * la]) = pk;
      }
      // lanes of one wave hand data to each other through LDS: wait on the
      // LDS counter only, the loads in flight stay there
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      ushort8 pa = *reinterpret_cast<const ushort8*>(
          &p_lds[lq * DEC_VT_PAD + 8 * la]);
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c) {
        dec_bf16x4v v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (__attribute__((address_space(3))) dec_bf16x4v*)(
                reinterpret_cast<char*>(&vt_lds[(c * 8 + 2 * la) * 96]) +
                lq * 8));
        dec_bf16x4v v2 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (__attribute__((address_space(3))) dec_bf16x4v*)(
                reinterpret_cast<char*>(&vt_lds[(c * 8 + 2 * la + 1) * 96]) +
                lq * 8));
        bf16x8 vb;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vb[e] = v1[e];
          vb[e + 4] = v2[e];
        }
        oacc[c] = dec_mfma(*reinterpret_cast<bf16x8*>(&pa), vb, oacc[c]);
      }
    };

    // pieces of 32 units: the page ids of one are one load, one id per lane,
    // instead of a pointer chase per unit. Pages past the last one repeat it
    // and dropped pages (-1) read page 0: what they hold is masked.
    for (int i0 = 0; i0 < n; i0 += 32) {
      const int m = min(32, n - i0);
      const int ids = max(0, bt[min(2 * (c0 + i0) + lane, npages - 1)]);
      load(0, ids, kr[0], vr[0]);
      if (m > 1) load(1, ids, kr[1], vr[1]);
      // (the markers keep the compiler from merging these loads with the
      // loop's own, behind the wait for the other unit)
      asm volatile("; first units" ::: "memory");
      for (int i = 0; i < m; i += 2) {
        step(i0 + i, kr[0], vr[0]);
        if (i + 2 < m) load(i + 2, ids, kr[0], vr[0]);
        if (i + 1 == m) break;
        step(i0 + i + 1, kr[1], vr[1]);
        if (i + 3 < m) load(i + 3, ids, kr[1], vr[1]);
        asm volatile("; next unit" ::: "memory");
      }
    }

    // heads are rows 4*la + r of the accumulators; m and l lie with head lq
    if (n == units) {  // the whole sequence
      // sink: one more key of score 0 and no value in the denominator
      const float l_all = sink ? l_run + dec_exp2(-m_run) : l_run;
      const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int g = 4 * la + r;
        const float row_inv = __shfl(inv, g, WAVE_SIZE);
        if (g < GQ) {
          bf16* op = out + ((int64_t)seq * num_q_heads + kvh * GQ + g) * HEAD_DIM;
#pragma unroll
          for (int c = 0; c < CHUNKS; ++c)
            op[c * 16 + lq] = float_to_bf16_bits(oacc[c][r] * row_inv);
        }
      }
    } else {
      // (wave, sequence) pairs in line order: w + seq is a slot of its own
      float* pp = part_out + ((int64_t)(w + seq) * num_kv_heads + kvh) *
                                 (GQ * HEAD_DIM + 16);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int g = 4 * la + r;
        if (g < GQ) {
#pragma unroll
          for (int c = 0; c < CHUNKS; ++c)
            pp[g * HEAD_DIM + c * 16 + lq] = oacc[c][r];
        }
      }
      if (la == 0 && lq < GQ) {
        pp[GQ * HEAD_DIM + lq] = m_run;
        pp[GQ * HEAD_DIM + 8 + lq] = l_run;
      }
    }
    left -= n;
    if (left == 0) return;
    off = 0;
    do {  // the next sequence with a key (the bound: a plan of other lengths)
      if (++seq >= num_seqs) return;
      L = __builtin_amdgcn_readfirstlane(seq_lens[seq]);
    } while (L <= 0);
  }
}

// Merge the partials of sequences that more than one run covers: a workgroup
// per (sequence, key/value head), a thread per 4 values of a head. 8
// partials at a time, all of their loads in flight together: the chain is
// plan entry -> loads -> store. (One thread per value walking the partials
// took 16 to 25 us.)
template <int HEAD_DIM>
__global__ __launch_bounds__(256) void attn_decode_combine_kernel(
    bf16* __restrict__ out,              // [S, Hq, D]
    const float* __restrict__ part_out,  // [waves + S, Hkv, GQ * D + 16]
    const int2* __restrict__ seqs, const int gq, const int num_kv_heads,
    const int sink) {
  constexpr int PB = 8;
  const int seq = blockIdx.x, kvh = blockIdx.y, tid = threadIdx.x;
  const int2 d = seqs[seq];
  const int np = d.y;
  if (np == 1 || tid * 4 >= gq * HEAD_DIM) return;  // 1: written by its run
  const int g = tid * 4 / HEAD_DIM;
  bf16* op = out + ((int64_t)seq * num_kv_heads + kvh) * gq * HEAD_DIM + tid * 4;
  const int64_t slot = (int64_t)num_kv_heads * (gq * HEAD_DIM + 16);
  const float* pp = part_out + (d.x + seq) * slot +
                    (int64_t)kvh * (gq * HEAD_DIM + 16);
  const float* pm = pp + gq * HEAD_DIM + g;
  pp += tid * 4;
  float m_run = -FLT_MAX, l_run = 0.f;
  float4v acc = {0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < np; p0 += PB) {
    float m[PB], l[PB];
    float4v a[PB];
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      const int64_t at = min(p0 + j, np - 1) * slot;
      m[j] = pm[at];
      l[j] = pm[at + 8];
      a[j] = *reinterpret_cast<const float4v*>(pp + at);
    }
    float m_new = m_run;
#pragma unroll
    for (int j = 0; j < PB; ++j) m_new = fmaxf(m_new, m[j]);
    const float carry = m_run > -FLT_MAX ? dec_exp2(m_run - m_new) : 0.f;
    l_run *= carry;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] *= carry;
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      if (p0 + j < np && m[j] > -FLT_MAX) {
        const float f = dec_exp2(m[j] - m_new);
        l_run += f * l[j];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += f * a[j][e];
      }
    }
    m_run = m_new;
  }
  if (sink) l_run += dec_exp2(-m_run);
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  ushort4v o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = float_to_bf16_bits(acc[e] * inv);
  *reinterpret_cast<ushort4v*>(op) = o;
}

template <int HEAD_DIM>
void launch_decode_gq(bf16* out, float* part_out, const bf16* q,
                      const bf16* kc, const bf16* vc, const int* bt,
                      const int* sl, const int* plan, float scale, int num_seqs,
                      int num_kv_heads, int gq, int max_blocks, int waves,
                      int64_t q_stride, bool kv_fp8, int window, int sink,
                      hipStream_t stream) {
  const int blocks = num_kv_heads * ((waves + 3) / 4);
  const int4* runs = reinterpret_cast<const int4*>(plan);
#define ARKS_CASE(G)                                                          \
  case G:                                                                     \
    if (kv_fp8) {                                                             \
      hipLaunchKernelGGL((attn_decode_kernel<HEAD_DIM, G, true>),             \
                         dim3(blocks), dim3(256), 0, stream, out, part_out,   \
                         q, kc, vc, bt, sl, runs, scale, num_kv_heads,        \
                         max_blocks, q_stride, window, sink, waves, num_seqs);\
    } else {                                                                  \
      hipLaunchKernelGGL((attn_decode_kernel<HEAD_DIM, G, false>),            \
                         dim3(blocks), dim3(256), 0, stream, out, part_out,   \
                         q, kc, vc, bt, sl, runs, scale, num_kv_heads,        \
                         max_blocks, q_stride, window, sink, waves, num_seqs);\
    }                                                                         \
    break;
  switch (gq) {
    ARKS_CASE(1)
    ARKS_CASE(2)
    ARKS_CASE(3)
    ARKS_CASE(4)
    ARKS_CASE(5)
    ARKS_CASE(6)
    ARKS_CASE(7)
    ARKS_CASE(8)
    default:
      break;  // validated host-side
  }
#undef ARKS_CASE
  hipLaunchKernelGGL((attn_decode_combine_kernel<HEAD_DIM>),
                     dim3(num_seqs, num_kv_heads), dim3(256), 0, stream, out,
                     part_out, reinterpret_cast<const int2*>(plan + 4 * waves),
                     gq, num_kv_heads, sink);
}

}  // namespace arks

using namespace arks;

// plan: 4 * waves + 2 * num_seqs ints (16-byte aligned).
extern "C" void arks_attn_decode_plan(void* plan, const void* seq_lens,
                                      int num_seqs, int window, int waves,
                                      hipStream_t stream) {
  hipLaunchKernelGGL(attn_decode_plan_kernel, dim3(1), dim3(1024), 0, stream,
                     (int*)plan, (const int*)seq_lens, num_seqs, window, waves);
}

// waves: runs per key/value head, as planned; part_out holds
// (waves + num_seqs) * kv heads * (group * head_dim + 16) floats.
extern "C" void arks_attn_decode_paged(void* out, void* part_out, const void* q,
                                       const void* k_cache, const void* v_cache,
                                       const void* block_tables,
                                       const void* seq_lens, const void* plan,
                                       float scale, int num_seqs,
                                       int num_q_heads, int num_kv_heads,
                                       int head_dim, int max_blocks, int waves,
                                       int64_t q_stride, int kv_fp8, int window,
                                       int sink, hipStream_t stream) {
  const int gq = num_q_heads / num_kv_heads;
  if (num_seqs == 0) return;
  if (head_dim == 128) {
    launch_decode_gq<128>((bf16*)out, (float*)part_out, (const bf16*)q,
                          (const bf16*)k_cache, (const bf16*)v_cache,
                          (const int*)block_tables, (const int*)seq_lens,
                          (const int*)plan, scale, num_seqs, num_kv_heads, gq,
                          max_blocks, waves, q_stride, kv_fp8 != 0, window,
                          sink, stream);
  } else if (head_dim == 64) {
    launch_decode_gq<64>((bf16*)out, (float*)part_out, (const bf16*)q,
                         (const bf16*)k_cache, (const bf16*)v_cache,
                         (const int*)block_tables, (const int*)seq_lens,
                         (const int*)plan, scale, num_seqs, num_kv_heads, gq,
                         max_blocks, waves, q_stride, kv_fp8 != 0, window,
                         sink, stream);
  }
}
