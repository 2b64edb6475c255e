// Attention of few query rows against many keys (decoding steps, action chunks against a cached
// prefix) for 16-bit inputs, spread over the chip: the bits of the fused kernel.
//
// The fused kernel (attention_fused.hip) gives one workgroup 128 query rows of one head and the
// whole key range, twice.  With one query row that leaves 127 of 128 rows empty, reads a
// key/value head once per query head of its group, and a batch of 8 x 16 heads keeps only half of
// the compute units busy.  Here the query heads of a group and their query rows are packed into
// the rows of one problem (row = head in group * lq + query row), and a call runs
//   1. split_score_kernel, one workgroup per kSplitKeys keys of a (batch, kv head): S = Q K^T and
//      the reference's transform (round, scale, round, mask), the 16-bit scores s to a workspace
//      and, per row and 32 keys, their maximum;
//   2. split_value_kernel, one workgroup per 4 to 64 rows and 16 to 128 value columns: the row
//      statistics m and l, P = round(exp(s - m) / l) in the input dtype, O = P V over all keys.
//
// A row's bits must not depend on the number of query rows in the call (a prefix in chunks is the
// whole prefix), so every value is the fused kernel's.  S comes from the same MFMA sequence
// (128-byte steps of the head dimension, chunk pairs in order) and transform.  The fused kernel's
// row sum runs over steps of 32 keys, l = l * rescale + part, with the maximum so far: the step
// maxima of kernel 1 give all running maxima at once, the parts (sixteen exponentials added in
// register order, per half-wavefront) and factors are then independent, and only the chain of
// fused multiply-adds is serial.  The sum of P V is one MFMA chain in key order per output, so
// the value kernel is spread over columns and rows, never over keys; one 16x16x32 MFMA gives the
// bits of the two 32x32x16 steps over its 32 keys (gemm_skinny.h).
//
// MI355X, kernels, fused kernel against this: 8 samples, 16 / 4 heads of 128, one query row, 2048
// keys (33.6 MB) 81 -> 18.7 us (scores 6.8, values 11.9); 16 samples, 64 / 8 heads, 4096 keys
// (268 MB) 337 -> 61; 16 rows, 16 samples, 32 / 8 heads, 4096 keys 172 -> 121; one sample, 32 / 8
// heads, one row, 32768 keys 1180 -> 94.  Keys split over workgroups with partial outputs added
// afterwards took 17.3, 65, 136 and 43, but a row of up to 16 query rows then had other bits than
// the same row in a longer call.
//
// Bound: a decoding step streams K and V once (the scores of a few rows are small beside them);
// K goes from memory straight to the MFMA operand registers, V through LDS to the transposing
// read.
#include <algorithm>

#include "attention16.h"
#include "gemm.h"
#include "gemm_skinny.h"

namespace biops {

constexpr int kSplitKeys = 256;      // keys per workgroup of split_score_kernel, 64 per wavefront
// Calls taken (the bits are the same on either path).  Kernel time, MI355X, bf16, head size 128,
// fused kernel against this path:
//   query rows, at 16 samples x 8 kv heads x 4096 keys, where the fused kernel has enough tiles to
//   fill the chip: 1 row 337 -> 61 us (8 heads per kv head), 16 rows 172 -> 121 (4 heads), 340 ->
//   165 (8 heads); more rows were not measured on this form;
//   keys, 1 sample, 4 heads, one row: 700 keys 32.5 -> 12.2.  A second launch costs about 2 us of
//   host time, so calls up to 512 keys, which the host bounds either way, stay on the fused kernel
//   (replayed from a graph, without that cost, 400 keys would gain too).
constexpr int kSplitMaxQuery = 16;   // query rows per head
constexpr int kSplitMinKeys = 512;   // longer key ranges are split
// The fused kernel needs no workspace, so this path must not make a call run out of memory that
// fitted: larger calls stay there (512 pairs of up to 32 rows take 2 GiB at 60000 keys).
constexpr int64_t kSplitMaxWorkspace = int64_t(2) << 30;

struct SplitArgs {
  const void* q; const void* k; const void* v; void* out;
  const void* mask;
  void* s;            // scores in fragment order (score_offset)
  float* smax;        // maximum of [pair][row tile][step of 32 keys][row of 32]
  int64_t sqB, sqH, sqL, skB, skH, skL, svB, svH, svL;
  int64_t mB, mH, mI;
  int32_t hkv, group, lq, lk, d, dv;
  int32_t rows, row_tiles, tiles_per_wg, row_groups;  // rows = group * lq
  int32_t pairs, key_tiles;
  int32_t steps;      // steps of 32 keys, rounded up to whole 64-key blocks
  float scale, kexp;  // kexp: base change of the exponentials (the scale folded in under pow2)
  int32_t pow2;       // scores in units of round(S) (attention_fused.hip, P2)
  int32_t add;        // additive mask
};

template <typename T>
__device__ __forceinline__ ExpBase value_base(const SplitArgs& a, float m) {
  const ExpBase add = attn_exp_base<T, true>(m, a.kexp), plain = attn_exp_base<T, false>(m, a.kexp);
  return ExpBase{plain.m, a.add ? add.k : plain.k, a.add ? add.sh : plain.sh};
}

// Scores of row tile rt (32 rows): one 16-byte piece per lane and 16-key chunk, the registers of
// the fused kernel (lane L: row L % 32, keys 4(L/32) + (0..3) and + 8 of the chunk).
__device__ __forceinline__ int64_t score_offset(const SplitArgs& a, int pair, int rt, int chunk) {
  return (((int64_t)pair * a.row_tiles + rt) * (4 * cdiv(a.lk, 64)) + chunk) * 512;
}

template <typename T>
__device__ __forceinline__ uint32_t split_pack2(float x, float y) {
  if constexpr (std::is_same<T, bf16_t>::value) return f32x2_to_bf16x2_bits(x, y);
  else return (uint32_t)Num<T>::to_bits(x) | ((uint32_t)Num<T>::to_bits(y) << 16);
}

// Workgroup barrier that waits for LDS operations only (__syncthreads also drains the global
// loads in flight).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// MASK: 0 none, 1 boolean (bytes, nonzero = keep), 2 additive (T); contiguous rows, lk % 4 == 0.
template <typename T, int DP, int MASK>
__global__ __launch_bounds__(256) void split_score_kernel(SplitArgs a) {
  constexpr int QF = DP / 16;
  constexpr int E = sizeof(T);
  int x = blockIdx.x;
  const int rg = x % a.row_groups;
  x /= a.row_groups;
  const int kt = x % a.key_tiles;
  const int pair = x / a.key_tiles;
  const int hk = pair % a.hkv;
  const int64_t b = pair / a.hkv;
  const int tid = threadIdx.x;
  const int w = tid >> 6, lane = tid & 63, hf = lane >> 5, l32 = lane & 31;
  const u32x4_t zero4 = {0u, 0u, 0u, 0u};
  const int n0 = kt * kSplitKeys + 64 * w;  // this wavefront's keys
  const bool live = n0 < a.lk;
  const bool whole = n0 + 64 <= a.lk;  // no key limit inside (uniform in the wavefront)

  // K fragments (A operand of S^T = K Q^T): lane holds key n0 + 32 hb + l32, head-dim chunk
  // 2cc + hf; keys past the end repeat the last row (their scores are masked out).
  u32x4_t kf[2][QF];
  if (live) {
    const char* kb = reinterpret_cast<const char*>(a.k) + E * (b * a.skB + hk * a.skH);
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
      const int n = n0 + 32 * hb + l32;
      const char* kr = kb + E * ((int64_t)(n < a.lk ? n : a.lk - 1) * a.skL);
#pragma unroll
      for (int cc = 0; cc < QF; ++cc) {
        const int d0 = 16 * cc + 8 * hf;
        kf[hb][cc] = d0 < a.d ? *reinterpret_cast<const u32x4_t*>(kr + E * d0) : zero4;
      }
    }
  }

  const int rt0 = rg * a.tiles_per_wg;
  const int rt1 = rt0 + a.tiles_per_wg < a.row_tiles ? rt0 + a.tiles_per_wg : a.row_tiles;
  for (int rt = rt0; rt < rt1; ++rt) {
    const int row = 32 * rt + l32;
    const bool row_ok = row < a.rows;
    const int h = hk * a.group + (row_ok ? row / a.lq : 0);
    const int i = row_ok ? row % a.lq : 0;
    if (live) {
      u32x4_t qf[QF];
      const char* qr = reinterpret_cast<const char*>(a.q) + E * (b * a.sqB + h * a.sqH + i * a.sqL);
#pragma unroll
      for (int cc = 0; cc < QF; ++cc) {
        const int d0 = 16 * cc + 8 * hf;
        qf[cc] = (row_ok && d0 < a.d) ? *reinterpret_cast<const u32x4_t*>(qr + E * d0) : zero4;
      }
      const int lim = row_ok ? a.lk : 0;
      f32x16_t acc[2];
#pragma unroll
      for (int hb = 0; hb < 2; ++hb) {
        const int nb = n0 + 32 * hb + 4 * hf;  // acc[hb][r] is key nb + 8(r/4) + r%4
        uint32_t mw[MASK == 2 ? 8 : 4];
        if constexpr (MASK != 0) {
          constexpr int ME = MASK == 1 ? 1 : E;
          const char* mrow = reinterpret_cast<const char*>(a.mask) + ME * (b * a.mB + h * a.mH + i * a.mI);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int n = nb + 8 * j;
            if constexpr (MASK == 1) {
              mw[j] = n < lim ? *reinterpret_cast<const uint32_t*>(mrow + n) : 0u;
            } else {
              const u32x2_t y = n < lim ? *reinterpret_cast<const u32x2_t*>(mrow + E * n) : u32x2_t{0u, 0u};
              mw[2 * j] = y[0];
              mw[2 * j + 1] = y[1];
            }
          }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[hb][r] = 0.f;
#pragma unroll
        for (int cc = 0; cc < QF; ++cc) Mfma<T>::step(acc[hb], kf[hb][cc], qf[cc]);
        float m = -INFINITY;
        auto transform = [&](auto open) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            float s = Num<T>::round(acc[hb][r]);
            if (!a.pow2) s = Num<T>::round(s * a.scale);
            if constexpr (MASK == 1) {
              s = (mw[r >> 2] >> (8 * (r & 3))) & 0xffu ? s : -INFINITY;
            } else if constexpr (MASK == 2) {
              const uint32_t wj = mw[2 * (r >> 2) + ((r & 3) >> 1)];
              s = Num<T>::round(s + Num<T>::from_bits(r & 1 ? wj >> 16 : wj & 0xffffu));
            }
            if constexpr (!decltype(open)::value) s = nb + 8 * (r >> 2) + (r & 3) < a.lk ? s : -INFINITY;
            acc[hb][r] = s;
            m = fmaxf(m, s);
          }
        };
        if (whole) transform(std::true_type{});
        else transform(std::false_type{});
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        if (hf == 0) a.smax[(((int64_t)pair * a.row_tiles + rt) * a.steps + n0 / 32 + hb) * 32 + l32] = m;
      }
      if (row_ok) {
        char* sp = reinterpret_cast<char*>(a.s) + E * (score_offset(a, pair, rt, n0 / 16) + 8 * lane);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const f32x16_t& s = acc[c >> 1];
          const int r = 8 * (c & 1);
          *reinterpret_cast<u32x4_t*>(sp + 1024 * c) =
              u32x4_t{split_pack2<T>(s[r], s[r + 1]), split_pack2<T>(s[r + 2], s[r + 3]),
                      split_pack2<T>(s[r + 4], s[r + 5]), split_pack2<T>(s[r + 6], s[r + 7])};
        }
      }
    }
  }
}

// Keys per stage of the value kernel: 32 KiB of V at most; enough for every thread to have eight
// probabilities to work out (RL rows), up to 512.
constexpr int value_keys(int RL, int NC) {
  const int by_rows = RL <= 4 ? 512 : (RL <= 8 ? 256 : 128);
  return by_rows * NC <= 1024 ? by_rows : 1024 / NC;
}

// Workgroups of one (pair, row block) read the same scores and neighbouring pieces of the same V
// rows: its column blocks are eight workgroups apart, on one XCD.
__device__ __forceinline__ void value_block(int x, int units, int col_blocks, int& unit, int& cb) {
  const int full = units / 8 * 8 * col_blocks;
  if (x < full) {
    const int in = x % (8 * col_blocks);
    unit = x / (8 * col_blocks) * 8 + in % 8;
    cb = in / 8;
  } else {
    const int left = units % 8;
    unit = units / 8 * 8 + (x - full) % left;
    cb = (x - full) / left;
  }
}

// RL packed rows (4, 8 or 16 RT) x 16 NC value columns of one pair over all keys; wavefront w
// computes column tiles w, w + 4, ...
template <typename T, int RL, int NC>
__global__ __launch_bounds__(256) void split_value_kernel(SplitArgs a) {
  constexpr int E = sizeof(T);
  constexpr int RT = RL <= 16 ? 1 : RL / 16, CW = 16 * NC, SK = value_keys(RL, NC);
  constexpr int CT = NC < 4 ? 1 : NC / 4;      // column tiles per wavefront
  constexpr int VCH = CW / 8;                  // 16-byte chunks per V row of the block
  constexpr int VL = SK * VCH / 256;           // V loads per thread and stage
  constexpr int VR = 256 / VCH;                // V rows of one load of the workgroup
  constexpr int PL = RL * SK / 2048 < 1 ? 1 : RL * SK / 2048;  // pieces of P per thread and stage
  constexpr int PT = RL * SK / 8 / PL;         // threads with pieces
  constexpr int PF = VL <= 1 ? 8 : (VL == 2 ? 6 : (VL == 4 ? 4 : 2));  // stages in flight per thread
  constexpr int V_BYTES = SK * CW * E, P_BYTES = SK * RL * E, STAGE = V_BYTES + P_BYTES;
  // Statistics: rounds of SS steps of 32 keys; the running maxima of a row by G threads of PER steps.
  constexpr int SS = RL <= 8 ? 256 : (RL == 16 ? 128 : 64);
  constexpr int G = 256 / RL < 16 ? 256 / RL : 16, PER = SS / G;
  constexpr int STAT_BYTES = 4 * SS * RL * 4;
  constexpr int SMEM = 2 * STAGE > STAT_BYTES ? 2 * STAGE : STAT_BYTES;
  static_assert(VL >= 1 && VL * 256 == SK * VCH && SK % 128 == 0, "whole loads");
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  __shared__ float group_max[G][RL], row_sum[2][RL];
  const int col_blocks = (a.dv + CW - 1) / CW, row_blocks = (a.rows + RL - 1) / RL;
  int unit, cb;
  value_block(blockIdx.x, a.pairs * row_blocks, col_blocks, unit, cb);
  const int r0 = RL * (unit % row_blocks);
  const int pair = unit / row_blocks;
  const int hk = pair % a.hkv;
  const int64_t b = pair / a.hkv;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const u32x4_t zero4 = {0u, 0u, 0u, 0u};
  const int nrows = a.rows - r0 < RL ? a.rows - r0 : RL;
  const int c0 = CW * cb;
  const int stages = (a.lk + SK - 1) / SK, steps = (a.lk + 31) / 32;

  // This thread's row in the statistics and in P (rows past the end repeat the last one: they
  // reach no output); its scores and its V chunk (chunks past dv repeat the block's first).
  const int r = tid & (RL - 1), part = tid / RL;
  const int rr = r0 + (r < nrows ? r : nrows - 1);
  const char* const score = reinterpret_cast<const char*>(a.s) + E * score_offset(a, pair, rr / 32, 0) + 16 * (rr % 32);
  const int vc = tid % VCH, vk = tid / VCH;
  const char* const vbase = reinterpret_cast<const char*>(a.v) + E * (b * a.svB + hk * a.svH + c0 + (c0 + 8 * vc < a.dv ? 8 * vc : 0));
  const char* const vrow0 = vbase + E * (int64_t)vk * a.svL;
  u32x4_t vr[PF][VL], sr[PF][PL];
  // Every stage issues the same loads (stages past the end repeat the last one): the compiler's
  // waits for a stage then leave the later ones in flight.  Keys past the end read the first row.
  auto load = [&](int st, int slot) {
    const int k0 = SK * (st < stages ? st : stages - 1);
#pragma unroll
    for (int p = 0; p < VL; ++p) {
      const char* const v = vrow0 + E * ((int64_t)(k0 + VR * p) * a.svL);
      vr[slot][p] = *reinterpret_cast<const u32x4_t*>(k0 + VR * p + vk < a.lk ? v : vbase);
    }
    // pieces part + (256 / RL) i of the stage: chunk piece / 2, half piece % 2
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      const int piece = part + 256 / RL * i;
      const char* const p = score + 1024 * (int64_t)(k0 / 16) + 512 * piece;
      sr[slot][i] = *reinterpret_cast<const u32x4_t*>(k0 + 16 * (piece >> 1) < 32 * a.steps ? p : score);
    }
  };

  // Row statistics: running maxima and rescale factors, parts, then the chain.  A round's step
  // maxima and its first parts' scores are loaded a round ahead.
  float m = -INFINITY, l = 0.f;  // maximum of the rounds before; this thread's half of the row sum
  {
    float* const run = reinterpret_cast<float*>(smem);  // [step][row] running maximum
    float* const factor = run + SS * RL;                // [step][row]
    float* const parts = factor + SS * RL;              // [step][half][row]
    constexpr int AHEAD = 4;
    // rows of a part item: the valid rows rounded up to a power of two
    const int lr = nrows <= 1 ? 0 : 32 - __builtin_clz(nrows - 1);
    const float* const smax = a.smax + ((int64_t)pair * a.row_tiles + rr / 32) * a.steps * 32 + rr % 32;
    // item i: row i % 2^lr, half, step of the round
    auto item = [&](int i, int& pr, int& hf, int& j) {
      pr = i & ((1 << lr) - 1);
      hf = (i >> lr) & 1;
      j = i >> lr >> 1;
    };
    float v[PER];
    u32x4_t lo[AHEAD], hi[AHEAD];
    auto load_items = [&](int s0, int i0) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        int pr, hf, j;
        item(i0 + 256 * u, pr, hf, j);
        const int row = r0 + (pr < nrows ? pr : 0), step = s0 + j < steps ? s0 + j : 0;
        const char* p = reinterpret_cast<const char*>(a.s) + E * score_offset(a, pair, row / 32, 2 * step) + 16 * (row % 32) + 512 * hf;
        lo[u] = *reinterpret_cast<const u32x4_t*>(p);
        hi[u] = *reinterpret_cast<const u32x4_t*>(p + 1024);
      }
    };
    auto load_round = [&](int s0) {
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int j = s0 + part * PER + u;
        v[u] = smax[(int64_t)(part < G && j < steps ? j : 0) * 32];
      }
      load_items(s0, tid);
    };
    load_round(0);
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      __builtin_amdgcn_sched_barrier(0);  // in stage order: the waits count
      load(j, j);
    }
    __builtin_amdgcn_sched_barrier(0);
    for (int s0 = 0; s0 < steps; s0 += SS) {
      const int n = steps - s0 < SS ? steps - s0 : SS;
      if (part < G) {
        float gm = -INFINITY;
#pragma unroll
        for (int u = 0; u < PER; ++u) {
          v[u] = part * PER + u < n ? v[u] : -INFINITY;
          gm = fmaxf(gm, v[u]);
        }
        group_max[part][r] = gm;
      }
      lds_barrier();
      float before = m, all = m;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float y = group_max[g][r];
        if (g < part) before = fmaxf(before, y);
        all = fmaxf(all, y);
      }
      if (part < G) {
#pragma unroll
        for (int u = 0; u < PER; ++u) {
          const float mn = fmaxf(before, v[u]);
          run[(part * PER + u) * RL + r] = mn;
          factor[(part * PER + u) * RL + r] = attn_rescale(before, value_base<T>(a, mn));
          before = mn;
        }
      }
      m = all;
      lds_barrier();
      const int items = n * 2 << lr;
      for (int i0 = tid; i0 < items; i0 += 256 * AHEAD) {
        if (i0 != tid) load_items(s0, i0);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
          int pr, hf, j;
          item(i0 + 256 * u, pr, hf, j);
          if (i0 + 256 * u >= items || pr >= nrows) continue;
          const ExpBase base = value_base<T>(a, run[j * RL + pr]);
          float sum = 0.f;
#pragma unroll
          for (int e = 0; e < 16; ++e)
            sum += attn_exp(Num<T>::from_bits(((e < 8 ? lo : hi)[u][(e & 7) >> 1] >> (16 * (e & 1))) & 0xffffu), base);
          parts[(2 * j + hf) * RL + pr] = sum;
        }
      }
      if (s0 + SS < steps) load_round(s0 + SS);
      lds_barrier();
      if (tid < 2 * RL) {  // half `part` of row r
        int j = 0;
        for (; j + 8 <= n; j += 8) {
          float f[8], y[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            f[u] = factor[(j + u) * RL + r];
            y[u] = parts[(2 * (j + u) + part) * RL + r];
          }
#pragma unroll
          for (int u = 0; u < 8; ++u) l = __builtin_fmaf(l, f[u], y[u]);
        }
        for (; j < n; ++j) l = __builtin_fmaf(l, factor[j * RL + r], parts[(2 * j + part) * RL + r]);
      }
    }
    if (tid < 2 * RL) row_sum[part][r] = l;
    lds_barrier();
  }
  const float lt = row_sum[0][r] + row_sum[1][r];
  const float inv = m == -INFINITY || lt == 0.f ? 0.f : 1.0f / lt;
  const ExpBase base = value_base<T>(a, m);

  // P V, stage by stage through two LDS buffers, one barrier per stage: a stage's first fragments
  // are read, the next stage's V and P go to the other buffer, then the MFMAs.
  f32x4_t acc[RT][CT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int g = lane >> 4, l16 = lane & 15;
  // Transposing V reads: lane s of a 16-lane group points at row s/4, column 4(s%4) and receives
  // four rows of one column; group g holds the keys of chunk g/2, half g%2 of a step, as P does.
  const int vrow = 16 * (g >> 1) + 4 * (g & 1) + (l16 >> 2);
  const int vcol = 16 * w + 4 * (l16 & 3);
  auto fill = [&](int st, int slot) {
    char* const vb = smem + (st & 1) * STAGE;
    if (SK * (st + 1) > a.lk) {  // keys past the end have no weight, but their V may hold anything
#pragma unroll
      for (int p = 0; p < VL; ++p)
        if (SK * st + VR * p + vk >= a.lk) vr[slot][p] = zero4;
    }
#pragma unroll
    for (int p = 0; p < VL; ++p)
      *reinterpret_cast<u32x4_t*>(vb + lds_off_n<VCH>(VR * p + vk, 8 * vc)) = vr[slot][p];
    if (PT == 256 || tid < PT) {
#pragma unroll
      for (int i = 0; i < PL; ++i) {
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          p[e] = attn_exp(Num<T>::from_bits((sr[slot][i][e >> 1] >> (16 * (e & 1))) & 0xffffu), base) * inv;
        *reinterpret_cast<u32x4_t*>(vb + V_BYTES + ((part + 256 / RL * i) * RL + r) * 16) =
            u32x4_t{split_pack2<T>(p[0], p[1]), split_pack2<T>(p[2], p[3]), split_pack2<T>(p[4], p[5]),
                    split_pack2<T>(p[6], p[7])};
      }
    }
    load(st + PF, slot);
  };
  constexpr int QS = 4, QUADS = SK / 32 / QS;  // steps read together
  struct Frags {
    u32x4_t p[QS][RT], v[QS][CT];
  };
  auto stage = [&](int st, int next_slot) {
    const char* const vb = smem + (st & 1) * STAGE;
    const char* const pb = vb + V_BYTES + (l16 & (RL - 1)) * 16;
    auto read = [&](int q, Frags& f) {
#pragma unroll
      for (int j = 0; j < QS; ++j) {
        const int s = QS * q + j;
#pragma unroll
        for (int t = 0; t < RT; ++t)
          f.p[j][t] = *reinterpret_cast<const u32x4_t*>(pb + ((4 * s + g) * RL + 16 * t) * 16);
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          const u32x2_t lo = lds_read_tr16(vb + lds_off_n<VCH>(32 * s + vrow, vcol + 64 * c));
          const u32x2_t hi = lds_read_tr16(vb + lds_off_n<VCH>(32 * s + vrow + 8, vcol + 64 * c));
          f.v[j][c] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
        }
      }
    };
    auto multiply = [&](auto whole, int q, const Frags& f) {
#pragma unroll
      for (int j = 0; j < QS; ++j) {
        if (!decltype(whole)::value && SK * st + 32 * (QS * q + j) >= a.lk) return;  // as in the fused kernel, no step past the keys
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int t = 0; t < RT; ++t) Mfma16<T>::step(acc[t][c], f.p[j][t], f.v[j][c]);
      }
    };
    Frags f[2];
    if (w < NC) read(0, f[0]);
    fill(st + 1, next_slot);  // past the last stage: read by nobody
    if (w < NC) {
#pragma unroll
      for (int q = 0; q < QUADS; ++q) {
        if (q + 1 < QUADS) read(q + 1, f[(q + 1) & 1]);
        if (SK * (st + 1) <= a.lk) multiply(std::true_type{}, q, f[q & 1]);
        else multiply(std::false_type{}, q, f[q & 1]);
      }
    }
    lds_barrier();
  };
  fill(0, 0);
  lds_barrier();
  for (int st = 0;; st += PF) {
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      if (st + j >= stages) goto done;
      stage(st + j, (j + 1) % PF);
    }
  }
done:

  // Register e of lane L is row 4(L/16) + e, column L % 16 of its 16 x 16 block; out is contiguous
  // [b, kv head, row = head in group * lq + query row, dv].
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int col = c0 + 16 * w + 64 * c + l16;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * t + 4 * g + e;
        if (w < NC && row < nrows && col < a.dv)
          Num<T>::store(reinterpret_cast<T*>(a.out) + ((int64_t)pair * a.rows + r0 + row) * a.dv + col, acc[t][c][e]);
      }
    }
}

struct SplitSizes {
  int64_t smax, total;  // byte offset of the step maxima, and the end
  int64_t rows, row_tiles, key_tiles;
};
static SplitSizes split_sizes(int64_t batch, int64_t hq, int64_t hkv, int64_t lq, int64_t lk) {
  auto al = [](int64_t b) { return (b + 255) & ~int64_t(255); };
  SplitSizes z{};
  z.rows = hq / hkv * lq;
  z.row_tiles = cdiv(z.rows, 32);
  z.key_tiles = cdiv(lk, kSplitKeys);
  const int64_t blocks = batch * hkv * z.row_tiles * cdiv(lk, 64);
  z.smax = al(blocks * 64 * 32 * 2);
  z.total = z.smax + al(blocks * 2 * 32 * 4);
  return z;
}
template <typename T, int MASK>
static int launch_scores(const SplitArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)a.pairs * a.key_tiles * a.row_groups));
  if (a.d <= 64) hipLaunchKernelGGL((split_score_kernel<T, 64, MASK>), grid, dim3(256), 0, s, a);
  else if (a.d <= 128) hipLaunchKernelGGL((split_score_kernel<T, 128, MASK>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((split_score_kernel<T, 256, MASK>), grid, dim3(256), 0, s, a);
  return check_launch("split_score_kernel");
}

template <typename T, int RL, int NC>
static int launch_values_t(const SplitArgs& a, hipStream_t s) {
  const int64_t wgs = (int64_t)a.pairs * cdiv(a.rows, RL) * cdiv(a.dv, 16 * NC);
  hipLaunchKernelGGL((split_value_kernel<T, RL, NC>), dim3((unsigned)wgs), dim3(256), 0, s, a);
  return check_launch("split_value_kernel");
}

// Rows and columns per workgroup.  A workgroup works out the statistics and P of its rows for all
// keys and streams its columns of V, so a launch that leaves the chip idle is cut into small
// blocks (P is then worked out once per column block) and a large one into large blocks (V is
// streamed once per row block).  MI355X, values + scores, us:
//   up to 16 rows, columns 16 / 32 / 64 / 128: 32 pairs (8 x 4 kv heads), 4 rows, 2048 keys 18.7 / 19.0 /
//   21.8 / 29; 64 pairs, 4 rows, 16384 keys 164 / 142 / 156 / 216; 128 pairs, 8 rows, 4096 keys 82 / 64 /
//   61 / 73; 512 pairs, 4 rows, 1024 keys 125 / 80 / 61 / 56: the narrowest of which one workgroup per
//   compute unit is enough;
//   more rows: 4 pairs, 64 rows, 1500 keys: blocks of 16 rows 18.1, of 64 36; 16 pairs, 96 rows, 2048
//   keys 29.7 (16), 34.6 (32), 48 (64); 64 pairs, 128 rows, 1024 keys 42.3 (16), 37.0 (32), 39.3 (64); 128
//   pairs, 128 rows, 4096 keys 258 (16), 199 (32), 165 (64);
//   blocks of 4 and 8 rows have longer stages (value_keys): 8 pairs of 4 rows and 32768 keys 139 -> 94,
//   16 pairs of 4 rows and 3000 keys 18.9 -> 17.3, but 4 pairs of one row and 700 keys 12.2 -> 14.0.
template <typename T, int RL>
static int launch_values_few(const SplitArgs& a, hipStream_t s) {
  const int64_t units = (int64_t)a.pairs * cdiv(a.rows, RL), cus = device_cus();
  if (units * cdiv(a.dv, 16) <= cus) return launch_values_t<T, RL, 1>(a, s);
  if (units * cdiv(a.dv, 32) <= cus) return launch_values_t<T, RL, 2>(a, s);
  if (units * cdiv(a.dv, 64) <= cus) return launch_values_t<T, RL, 4>(a, s);
  return launch_values_t<T, RL, 8>(a, s);
}
template <typename T>
static int launch_values(const SplitArgs& a, hipStream_t s) {
  const int64_t cus = device_cus();
  if (a.rows > 16 && a.pairs * cdiv(a.rows, 16) * cdiv(a.dv, 32) > 2 * cus) {
    if (a.rows > 32 && a.pairs * cdiv(a.rows, 64) * cdiv(a.dv, 128) >= cus) return launch_values_t<T, 64, 8>(a, s);
    return launch_values_t<T, 32, 4>(a, s);
  }
  if (a.lk > 2048 && a.rows <= 4) return launch_values_few<T, 4>(a, s);
  if (a.lk > 2048 && a.rows <= 8) return launch_values_few<T, 8>(a, s);
  return launch_values_few<T, 16>(a, s);
}

template <typename T>
static int launch_split(const SplitArgs& a, int mask_kind, hipStream_t s) {
  const int rc = mask_kind == 0 ? launch_scores<T, 0>(a, s) : (mask_kind == 1 ? launch_scores<T, 1>(a, s) : launch_scores<T, 2>(a, s));
  if (rc != BIOPS_OK) return rc;
  return launch_values<T>(a, s);
}

}  // namespace biops

using namespace biops;

extern "C" int64_t biops_sdpa_split_workspace_size(int dtype, int64_t batch, int64_t hq, int64_t hkv, int64_t lq,
                                                   int64_t lk, int64_t d, int64_t dv, int causal) {
  if (!biops_attention_fused_supported(dtype, d, dv) || causal != BIOPS_CAUSAL_NONE) return -1;
  if (batch <= 0 || hq <= 0 || hkv <= 0 || hq % hkv != 0 || lq <= 0 || lq > kSplitMaxQuery || lk <= kSplitMinKeys) return -1;
  const SplitSizes z = split_sizes(batch, hq, hkv, lq, lk);
  // 32-bit row / key indices, launches of fewer than 2^32 threads (score kernel: at most key_tiles *
  // row_tiles workgroups per pair; value kernel: two of 16 rows per row tile, and 16 column blocks
  // only where they fit the compute units, four beyond)
  const int64_t lim = int64_t(1) << 24;
  if (lk >= (int64_t(1) << 30) || z.rows >= (int64_t(1) << 25) ||
      batch * hkv >= lim / (2 * std::max<int64_t>(z.key_tiles, 4) * z.row_tiles))
    return -1;
  return z.total <= kSplitMaxWorkspace ? z.total : -1;
}

extern "C" int biops_sdpa_split_max_query(void) { return kSplitMaxQuery; }

extern "C" int biops_sdpa_split(int dtype, int64_t batch, int64_t hq, int64_t hkv, int64_t lq, int64_t lk, int64_t d,
                                int64_t dv, const void* q, int64_t sqB, int64_t sqH, int64_t sqL, const void* k,
                                int64_t skB, int64_t skH, int64_t skL, const void* v, int64_t svB, int64_t svH,
                                int64_t svL, const void* mask, int mask_dtype, int64_t mB, int64_t mH, int64_t mI,
                                int64_t mJ, float scale, void* out, void* workspace, int64_t workspace_bytes,
                                void* stream) {
  const int64_t need = biops_sdpa_split_workspace_size(dtype, batch, hq, hkv, lq, lk, d, dv, BIOPS_CAUSAL_NONE);
  if (need < 0) return fail(BIOPS_ERR_ARG, "split attention does not take these sizes");
  if (!q || !k || !v || !out || !workspace) return fail(BIOPS_ERR_ARG, "null pointer");
  if (mask && mask_dtype != BIOPS_BOOL && mask_dtype != dtype)
    return fail(BIOPS_ERR_DTYPE, "mask dtype must be bool or the score dtype");
  if (mask && !biops_attention_fused_mask_ok(mask, mask_dtype, lk, mB, mH, mI, mJ))
    return fail(BIOPS_ERR_LAYOUT, "split attention needs a mask with contiguous, aligned rows and keys % 4 == 0");
  for (const void* p : {q, k, v, static_cast<const void*>(out)})
    if (reinterpret_cast<uintptr_t>(p) & 15) return fail(BIOPS_ERR_LAYOUT, "split attention needs 16-byte aligned tensors");
  for (int64_t st : {sqB, sqH, sqL, skB, skH, skL, svB, svH, svL})
    if (st & 7) return fail(BIOPS_ERR_LAYOUT, "split attention needs 16-byte aligned rows (strides multiples of 8)");
  if (workspace_bytes < need) return fail(BIOPS_ERR_SIZE, "workspace %lld < %lld bytes", (long long)workspace_bytes, (long long)need);
  if (reinterpret_cast<uintptr_t>(workspace) & 255) return fail(BIOPS_ERR_LAYOUT, "workspace must be 256-byte aligned");
  const SplitSizes z = split_sizes(batch, hq, hkv, lq, lk);
  char* ws = reinterpret_cast<char*>(workspace);
  SplitArgs a{};
  a.q = q; a.k = k; a.v = v; a.out = out; a.mask = mask;
  a.s = ws;
  a.smax = reinterpret_cast<float*>(ws + z.smax);
  a.sqB = sqB; a.sqH = sqH; a.sqL = sqL; a.skB = skB; a.skH = skH; a.skL = skL;
  a.svB = svB; a.svH = svH; a.svL = svL;
  a.mB = mB; a.mH = mH; a.mI = mI;
  a.hkv = (int32_t)hkv; a.group = (int32_t)(hq / hkv); a.lq = (int32_t)lq; a.lk = (int32_t)lk;
  a.d = (int32_t)d; a.dv = (int32_t)dv;
  a.rows = (int32_t)z.rows; a.row_tiles = (int32_t)z.row_tiles;
  a.pairs = (int32_t)(batch * hkv); a.key_tiles = (int32_t)z.key_tiles;
  a.steps = (int32_t)(2 * cdiv(lk, 64));
  a.scale = scale;
  a.pow2 = dtype == BIOPS_BF16 && (!mask || mask_dtype == BIOPS_BOOL) ? pow2_scale(scale) : 0;
  a.kexp = a.pow2 ? scale * kLog2e : kLog2e;
  a.add = mask && mask_dtype != BIOPS_BOOL;
  // row tiles per workgroup of the score kernel: as many as leave two workgroups per compute unit
  // (each workgroup reads its keys once for all of its row tiles)
  const int64_t wgs = (int64_t)a.pairs * a.key_tiles * a.row_tiles;
  a.tiles_per_wg = (int32_t)std::max<int64_t>(1, std::min<int64_t>(a.row_tiles, wgs / (2 * device_cus())));
  a.row_groups = (int32_t)cdiv(a.row_tiles, a.tiles_per_wg);
  hipStream_t s = (hipStream_t)stream;
  const int kind = !mask ? 0 : (mask_dtype == BIOPS_BOOL ? 1 : 2);
  return dtype == BIOPS_F16 ? launch_split<f16_t>(a, kind, s) : launch_split<bf16_t>(a, kind, s);
}
