// Fused attention for float32 inputs: no score matrix in memory, one pass over the keys.
//
// The eager composite rounds nothing between its float32 products (batch_invariant_ops.py:
// 1194-1212), so unlike the 16-bit kernels (attention_fused.hip) the probabilities need not be
// normalised before they meet V: a workgroup (four wavefronts, 32 query rows each, of one (batch, head))
// walks the keys once in blocks of 32, in order,
//   S^T = K Q^T (v_mfma_f32_32x32x2_f32, the GEMM's chunk order), s = round(S * scale), masks as in
//   the composite; running maximum m, p = exp(s - m), l = l * c + sum p, O^T = O^T * c + V^T P^T
// with c = exp(m_old - m), and writes O / l at the end (a row without a visible key gives zeros).
// p is float32 throughout; the materialised path differs only in the order of its sums and in
// dividing before instead of after the product.
//
// The scores are computed transposed: lane L holds query row L % 32 and keys 8j + 4(L/32) + i (j, i =
// 0..3).  Register r = 4j + i of both half-wavefronts is then exactly the B operand of the V^T P^T
// step over keys 8j + i and 8j + 4 + i, and the row statistics and the rescaling stay inside a lane.
//
// The keys are cut into chunks of kF32Chunk, each with its own maximum, sum and O^T, and the chunks
// are merged in order (f32_merge): by the workgroup itself, which then keeps the running total in the
// output rows, or, when the launch has too few query tiles to fill the chip, by f32_combine_kernel
// after a launch with one workgroup per chunk; the smallest launches have workgroups of 32 query
// rows that share a chunk's blocks (f32_few_kernel).  All do the same operations in the same order,
// so the choice, which depends on the batch, changes no bit.
//
// Batch invariance: the chunks, the block order, the MFMA chains and the statistics depend on the
// sample's own rows and lengths only.
//
// Bound: the fp32 matrix rate (157 TF/s): 4 x 9 + 16 x 3 MFMAs of 64 cycles per 32 x 32 block at
// head size 72, beside about 230 vector instructions.  MI355X, call times against scores in memory
// (three launches): 8 x 16 heads x 256 x 256, head size 72 (2.4 GFLOP, 18 us at the matrix rate) 66.3 ->
// 39.3 us; causal 2 x 8 / 2 heads x 1000 x 1000, 128: 133 -> 97; 1 x 16 heads, causal, 1024 x 1024, 64: 91 -> 56;
// 4 x 32 / 8 x 1500 x 1500, 128, additive mask: 2780 -> 2010.  Of the 39 us the two products take about 20,
// the block loads and barriers 5, the chunk merge 4, the softmax 4, launch and first loads the rest.
// Chunks of 256 keys saved the merges of large launches but doubled the chain of the small ones.
#include <algorithm>

#include "gemm.h"
#include "rowops.h"

namespace biops {

typedef uint32_t u32_any_t __attribute__((aligned(1)));

constexpr int kF32Rows = 128;  // query rows per workgroup
constexpr int kF32Keys = 32;   // keys per block
constexpr int kF32Chunk = 128; // keys per chunk

struct F32AttnArgs {
  const float* q; const float* k; const float* v; float* out;
  const void* mask;
  int64_t sqB, sqH, sqL, skB, skH, skL, svB, svH, svL;
  int64_t mB, mH, mI, mJ;
  int64_t hq, hkv, group, pairs;
  int32_t lq, lk, d, dv, qtiles;
  float scale;
  int32_t causal;
  int32_t mvec;  // mask rows have unit stride
  int64_t tile0;   // first tile of the launch
  int32_t chunks;  // split launch: chunks of the longest key range
  float* partial;  // split launch: O^T of [chunk][pair][row][dv], then {m, l} of [chunk][pair][row]
  float* stats;
};

// exp(x - m), x <= m, to the accuracy of expf (whose place it takes: the fp32 softmax has expf).  With d =
// x - m: e = round(d log2 e), 2^e * exp2(d log2 e - e), the difference from log2 e in two parts, so its
// error stays near 2^-25 at any d (the exp2 of the rounded product alone is off by |d| 2^-24 and
// flushes below 2^-126).  e is kept at -160 and above, where everything is 0: -inf gives 0, NaN
// comes through the difference.  8 x 16 x 256 x 256, head size 72: 40.9 us with expf, 39.3 so,
// 37.8 with the plain exp2.
__device__ __forceinline__ float f32_exp(float x, float m) {
  constexpr float kLow = 1.925963e-8f;  // log2 e - kLog2e
  const float d = x - m;
  const float e = fmaxf(__builtin_rintf(d * kLog2e), -160.f);
  const float a = __builtin_fmaf(d, kLow, __builtin_fmaf(d, kLog2e, -e));
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(a), (int)e);
}

// Adds a chunk's (mc, lc) to the running (m, l); the running O becomes O * c1 + Oc * c2 (f32_merge_o).
// A chunk whose keys are all masked is added too, with the weight 0 that its keys have: what its
// values hold (NaN, infinities) reaches the row, as in the composite's product.
__device__ __forceinline__ void f32_merge(float& m, float& l, float mc, float lc, float& c1, float& c2) {
  const float mn = fmaxf(m, mc);
  c1 = m == mn ? 1.f : f32_exp(m, mn);
  c2 = mc == mn ? 1.f : f32_exp(mc, mn);
  l = __builtin_fmaf(l, c1, lc * c2);
  m = mn;
}
__device__ __forceinline__ float f32_merge_o(float o, float oc, float c1, float c2, bool first) {
  const float t = oc * c2;
  return first ? t : __builtin_fmaf(o, c1, t);
}
// O / l at the end of a row; 0 where no score compares (all of them -inf or NaN), as the softmax kernels give.
__device__ __forceinline__ f32x4_t f32_final(f32x4_t o, float m, float l) {
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  return m == -INFINITY || l == 0.f ? zero : o * (1.0f / l);
}

// MASK: 0 none, 1 boolean (bytes, nonzero = keep), 2 additive.  DP, DVP: head and value size rounded up
// to 32 elements; QP: chunk pairs (8 elements) of the head size that are multiplied (zeros beyond).
// Two wavefronts per SIMD; the masked 128-wide kernels that merge their chunks themselves would spill
// a third of their registers then (4 x 16 / 4 heads x 700 x 701, boolean: 406 us).
template <int DP, int MASK, bool SPLIT>
constexpr int f32_waves() { return DP > 96 && MASK != 0 && !SPLIT ? 1 : 2; }

template <int DP, int QP, int DVP, int MASK, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(f32_waves<DP, MASK, SPLIT>(), f32_waves<DP, MASK, SPLIT>()))) void f32_attn_kernel(F32AttnArgs a) {
  static_assert(8 * QP <= DP, "chunk pairs");
  constexpr int OF = DVP / 32;
  constexpr int KCH = DP <= 64 ? 16 : 32;     // 16-byte chunk slots of a K / V row in LDS
  constexpr int VCH = DVP <= 64 ? 16 : 32;
  constexpr int K_BYTES = kF32Keys * KCH * 16, V_BYTES = kF32Keys * VCH * 16;
  constexpr int KL = kF32Keys * (DP / 4) / 256, VL = kF32Keys * (DVP / 4) / 256;  // loads per thread
  static_assert(kF32Keys * (DP / 4) % 256 == 0 && kF32Keys * (DVP / 4) % 256 == 0, "whole loads");
  __shared__ __attribute__((aligned(16))) char smem[2 * (K_BYTES + V_BYTES)];

  // longest causal key ranges first, all (batch, head) pairs per level
  const int64_t t = SPLIT ? blockIdx.x / a.chunks : a.tile0 + blockIdx.x;
  const int chunk0 = SPLIT ? (int)(blockIdx.x % a.chunks) : 0;
  const int qt = a.qtiles - 1 - (int)(t / a.pairs);
  const int64_t pair = t % a.pairs;
  const int64_t b = pair / a.hq, h = pair % a.hq, hk = h / a.group;
  const int tid = threadIdx.x;
  const int w = tid >> 6, lane = tid & 63, hf = lane >> 5, l32 = lane & 31;
  const u32x4_t zero4 = {0u, 0u, 0u, 0u};
  const int i0 = qt * kF32Rows;
  const int qrows = a.lq - i0 < kF32Rows ? a.lq - i0 : kF32Rows;
  const int shift = a.causal == BIOPS_CAUSAL_BOTTOM_RIGHT ? a.lk - a.lq : 0;
  auto row_lim = [&](int r) -> int {  // keys n >= row_lim(r) are masked out; grows with the row
    if (a.causal == BIOPS_CAUSAL_NONE) return a.lk;
    const int c = i0 + r + shift + 1;
    return c < 0 ? 0 : (c > a.lk ? a.lk : c);
  };
  const int rloc = 32 * w + l32;
  const bool row_ok = rloc < qrows;
  const int lim = row_ok ? row_lim(rloc) : 0;
  const int kend = row_lim(qrows - 1);
  constexpr int CB = kF32Chunk / kF32Keys;  // blocks per chunk
  const int blk0 = chunk0 * CB;
  const int nall = (kend + kF32Keys - 1) / kF32Keys;
  const int nblk = SPLIT && nall > blk0 + CB ? blk0 + CB : nall;
  if (SPLIT && blk0 >= nblk) return;
  const int wrows = qrows - 32 * w;
  const int wave_lim = wrows > 0 ? row_lim(32 * w + (wrows < 32 ? wrows : 32) - 1) : 0;
  // keys below this are visible to every lane (rows past the tile's end included in none)
  const int wave_open = wrows >= 32 ? row_lim(32 * w) : 0;

  const float* kb = a.k + b * a.skB + hk * a.skH;
  const float* vb = a.v + b * a.svB + hk * a.svH;
  const float* qr = a.q + b * a.sqB + h * a.sqH + (int64_t)(i0 + (row_ok ? rloc : 0)) * a.sqL;
  u32x4_t qf[QP];
#pragma unroll
  for (int c = 0; c < QP; ++c) {
    const int d0 = 8 * c + 4 * hf;
    qf[c] = (row_ok && d0 < a.d) ? *reinterpret_cast<const u32x4_t*>(qr + d0) : zero4;
  }

  // Block loads: chunk s = tid + 256 p is key s / (D / 4), chunk s % (D / 4); keys past the end and
  // chunks past the head size read a valid address and are zeroed when they are stored (a use of
  // the loaded value before the block's products would wait for it there).
  u32x4_t kr[KL], vr[VL];
  uint32_t koff[KL], voff[VL];  // byte offsets inside a block (32-bit: checked by the launcher)
#pragma unroll
  for (int p = 0; p < KL; ++p) {
    const int s = tid + 256 * p, c = 4 * (s % (DP / 4));
    koff[p] = 4u * (uint32_t)(s / (DP / 4) * a.skL + (c < a.d ? c : 0));
  }
#pragma unroll
  for (int p = 0; p < VL; ++p) {
    const int s = tid + 256 * p, c = 4 * (s % (DVP / 4));
    voff[p] = 4u * (uint32_t)(s / (DVP / 4) * a.svL + (c < a.dv ? c : 0));
  }
  auto load = [&](int blk) {
    const int n0 = blk * kF32Keys;
    const char* kp = reinterpret_cast<const char*>(kb + (int64_t)n0 * a.skL);
    const char* vp = reinterpret_cast<const char*>(vb + (int64_t)n0 * a.svL);
#pragma unroll
    for (int p = 0; p < KL; ++p)  // keys past the end: the block's first key
      kr[p] = *reinterpret_cast<const u32x4_t*>(kp + (n0 + (tid + 256 * p) / (DP / 4) < a.lk ? koff[p] : 0u));
#pragma unroll
    for (int p = 0; p < VL; ++p)
      vr[p] = *reinterpret_cast<const u32x4_t*>(vp + (n0 + (tid + 256 * p) / (DVP / 4) < a.lk ? voff[p] : 0u));
  };
  // K chunk c of row r at slot c ^ (r & 15): sixteen rows of one chunk in distinct banks.  V as the
  // GEMM's fp32 N-major stage: rows k and k + 4 in opposite halves of the banks.
  auto k_off = [](int r, int c) { return (r * KCH + (c ^ (r & 15))) * 16; };
  auto store = [&](int blk) {
    char* ks = smem + (blk & 1) * (K_BYTES + V_BYTES);
    const int n0 = blk * kF32Keys;
#pragma unroll
    for (int p = 0; p < KL; ++p) {
      const int s = tid + 256 * p, r = s / (DP / 4), c = s % (DP / 4);
      *reinterpret_cast<u32x4_t*>(ks + k_off(r, c)) = n0 + r < a.lk && 4 * c < a.d ? kr[p] : zero4;
    }
#pragma unroll
    for (int p = 0; p < VL; ++p) {
      const int s = tid + 256 * p, r = s / (DVP / 4), c = 4 * (s % (DVP / 4));
      *reinterpret_cast<u32x4_t*>(ks + K_BYTES + lds_off_n32<VCH>(r, c)) = n0 + r < a.lk && c < a.dv ? vr[p] : zero4;
    }
  };

  const int64_t moff = b * a.mB + h * a.mH + (int64_t)(i0 + rloc) * a.mI;
  float m = -INFINITY, l = 0.f;
  f32x16_t oacc[OF];  // O^T: register r of block e is column 32e + 8(r/4) + 4hf + r%4 of row l32
#pragma unroll
  for (int e = 0; e < OF; ++e)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[e][r] = 0.f;

  auto block = [&](int blk, const char* ks) {
    const int nb = blk * kF32Keys + 4 * hf;  // register r: key nb + 8(r/4) + r%4
    float mv[MASK == 2 ? 16 : 1];
    uint32_t mb[MASK == 1 ? 4 : 1];
    // four keys of a row of unit stride are one load at any alignment; the last keys of a row and
    // strided rows go key by key
    if constexpr (MASK == 1) {
      const uint8_t* mp = reinterpret_cast<const uint8_t*>(a.mask) + moff;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = nb + 8 * j;
        mb[j] = 0;
        if (n < lim) {
          if (a.mvec && n + 4 <= a.lk) {
            mb[j] = *reinterpret_cast<const u32_any_t*>(mp + n);
          } else {
            for (int i = 0; i < 4 && n + i < lim; ++i) mb[j] |= (uint32_t)(mp[(n + i) * a.mJ] != 0) << (8 * i);
          }
        }
      }
    } else if constexpr (MASK == 2) {
      const float* mp = reinterpret_cast<const float*>(a.mask) + moff;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = nb + 8 * j;
        f32x4_t y = {0.f, 0.f, 0.f, 0.f};
        if (n < lim) {
          if (a.mvec && n + 4 <= a.lk) {
            y = __builtin_bit_cast(f32x4_t, load_16(mp + n));
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (n + i < lim) y[i] = mp[(n + i) * a.mJ];
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) mv[4 * j + i] = y[i];
      }
    }
    f32x16_t acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int c = 0; c < QP; ++c)
      Mfma<float>::step(acc, *reinterpret_cast<const u32x4_t*>(ks + k_off(l32, 2 * c + hf)), qf[c]);
    // V values of step r (keys 8(r/4) + 4hf + r%4): read one step ahead of their MFMAs
    const char* vs = ks + K_BYTES;
    float xv[2][OF];
    auto read_v = [&](int r) {
#pragma unroll
      for (int e = 0; e < OF; ++e)
        xv[r & 1][e] = *reinterpret_cast<const float*>(vs + lds_off_n32<VCH>(8 * (r >> 2) + 4 * hf + (r & 3), 32 * e + l32));
    };
    read_v(0);
    float bm = -INFINITY;
    const bool open = blk * kF32Keys + kF32Keys <= wave_open;
    auto transform = [&](auto all) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float s = acc[r] * a.scale;
        if constexpr (MASK == 1) s = (mb[r >> 2] >> (8 * (r & 3))) & 0xffu ? s : -INFINITY;
        if constexpr (MASK == 2) s += mv[r];
        if constexpr (!decltype(all)::value) s = nb + 8 * (r >> 2) + (r & 3) < lim ? s : -INFINITY;
        acc[r] = s;
        bm = fmaxf(bm, s);
      }
    };
    if (open) transform(std::true_type{});
    else transform(std::false_type{});
    bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
    const float mn = fmaxf(m, bm);
    const float base = mn == -INFINITY ? 0.f : mn;
    if (__any(mn > m)) {  // some row's maximum grew: rescale what was summed so far
      const float c = f32_exp(m, base);
      const float cc = mn > m ? c : 1.f;
      l *= cc;
#pragma unroll
      for (int e = 0; e < OF; ++e)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[e][r] *= cc;
      m = mn;
    }
    float part = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[r] = f32_exp(acc[r], base);
      part += acc[r];
    }
    l += part;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if (r < 15) read_v(r + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < OF; ++e)
        oacc[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[r & 1][e], acc[r], oacc[e], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  float* orow = a.out + (pair * a.lq + i0 + rloc) * (int64_t)a.dv;  // out is contiguous
  float mt = -INFINITY, lt = 0.f;  // running maximum and sum over the chunks
  // The end of a chunk: merge it into the output rows, or store it for the combine kernel.
  auto end_chunk = [&](int chunk, bool last) {
    const float lc = l + __shfl_xor(l, 32, 64);
    if constexpr (SPLIT) {
      const int64_t r = (chunk * a.pairs + pair) * a.lq + i0 + rloc;
      if (row_ok) {
        if (hf == 0) *reinterpret_cast<f32x2_t*>(a.stats + 2 * r) = f32x2_t{m, lc};
#pragma unroll
        for (int e = 0; e < OF; ++e)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int col = 32 * e + 8 * j + 4 * hf;
            if (col < a.dv)
              *reinterpret_cast<f32x4_t*>(a.partial + r * a.dv + col) =
                  f32x4_t{oacc[e][4 * j], oacc[e][4 * j + 1], oacc[e][4 * j + 2], oacc[e][4 * j + 3]};
          }
      }
      return;
    }
    // the last chunk's merge divides by the row sum and stores the result
    const bool first = chunk == 0, some = chunk * kF32Chunk < lim;  // rows that end before the chunk have none of it
    if (row_ok && (some || last)) {
      float c1 = 1.f, c2 = 0.f;
      if (some) f32_merge(mt, lt, m, lc, c1, c2);
#pragma unroll
      for (int e = 0; e < OF; ++e) {
        f32x4_t o[4];  // a column block's loads before their first use (columns past dv read column 0)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int col = 32 * e + 8 * j + 4 * hf;
          o[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          if (!first && lim > 0) o[j] = *reinterpret_cast<const f32x4_t*>(orow + (col < a.dv ? col : 0));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int col = 32 * e + 8 * j + 4 * hf;
          if (some) {
#pragma unroll
            for (int i = 0; i < 4; ++i) o[j][i] = f32_merge_o(o[j][i], oacc[e][4 * j + i], c1, c2, first);
          }
          if (col < a.dv) *reinterpret_cast<f32x4_t*>(orow + col) = last ? f32_final(o[j], mt, lt) : o[j];  // dv is a multiple of 4
        }
        __builtin_amdgcn_sched_barrier(0);  // one column block's registers at a time
      }
    }
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int e = 0; e < OF; ++e)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[e][r] = 0.f;
  };

  if (nblk > blk0) {
    load(blk0);
    store(blk0);
    __syncthreads();
  }
  for (int blk = blk0; blk < nblk; ++blk) {
    if (blk + 1 < nblk) load(blk + 1);
    if (blk * kF32Keys < wave_lim) block(blk, smem + (blk & 1) * (K_BYTES + V_BYTES));
    if (blk + 1 < nblk) store(blk + 1);
    if ((blk + 1) % CB == 0 || blk + 1 == nblk) end_chunk(blk / CB, blk + 1 == nblk);
    __syncthreads();
  }
  if (!SPLIT && nblk == 0) end_chunk(0, true);  // no visible key: zeros
}

// Launches of few query rows: a workgroup per 32 rows and chunk, with the bits of f32_attn_kernel.
// There a wavefront walks its chunk's four blocks by itself, a chain of 4 x (4 QP + 16) dependent MFMAs
// (head size 128: 14 us) that a small launch has nothing to overlap with.  Here wavefront w computes
// the scores and probabilities of block w, with the running maximum from the four block maxima, and
// columns 32 w .. 32 w + 31 of O^T over the four blocks: 4 QP + 64 MFMAs in a row.  K, V and Q go from
// memory to the operand registers; only the probabilities pass through LDS.  One chunk: the result
// is written at once.
template <int QP, int OF, int MASK>
__global__ __launch_bounds__(256) void f32_few_kernel(F32AttnArgs a) {
  constexpr int CB = kF32Chunk / kF32Keys;
  static_assert(CB == 4 && OF <= 4, "a wavefront per block and per column block");
  __shared__ float ps[CB][16][64], parts[CB][64], block_max[CB][32];
  const int64_t t = blockIdx.x / a.chunks;
  const int chunk = (int)(blockIdx.x % a.chunks);
  const int qt = (int)((a.lq + 31) / 32 - 1 - t / a.pairs);
  const int64_t pair = t % a.pairs;
  const int64_t b = pair / a.hq, h = pair % a.hq, hk = h / a.group;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, hf = lane >> 5, l32 = lane & 31;
  const u32x4_t zero4 = {0u, 0u, 0u, 0u};
  const int i0 = 32 * qt;
  const int qrows = a.lq - i0 < 32 ? a.lq - i0 : 32;
  const int shift = a.causal == BIOPS_CAUSAL_BOTTOM_RIGHT ? a.lk - a.lq : 0;
  auto row_lim = [&](int r) -> int {
    if (a.causal == BIOPS_CAUSAL_NONE) return a.lk;
    const int c = i0 + r + shift + 1;
    return c < 0 ? 0 : (c > a.lk ? a.lk : c);
  };
  const bool row_ok = l32 < qrows;
  const int lim = row_ok ? row_lim(l32) : 0;
  const int kend = row_lim(qrows - 1);
  const int n0 = kF32Chunk * chunk;
  if (chunk > 0 && n0 >= kend) return;  // no row has keys here

  // V^T of column block w: register 16 j + r is key n0 + 32 j + 8(r/4) + 4 hf + r%4 (keys past the end read
  // row 0 and are zeroed below)
  float xv[CB][16];
  if (w < OF) {
    const float* const vb = a.v + b * a.svB + hk * a.svH + (32 * w + l32 < a.dv ? 32 * w + l32 : 0);
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = n0 + 32 * j + 8 * (r >> 2) + 4 * hf + (r & 3);
        xv[j][r] = a.lk > 0 ? vb[(int64_t)(n < a.lk ? n : 0) * a.svL] : 0.f;
      }
  }
  const int nw = n0 + 32 * w;  // this wavefront's block of keys
  float s[16];
  float bm = -INFINITY;
  if (nw < kend) {
    const float* const qr = a.q + b * a.sqB + h * a.sqH + (int64_t)(i0 + (row_ok ? l32 : 0)) * a.sqL;
    const float* const kr = a.k + b * a.skB + hk * a.skH + (int64_t)(nw + l32 < a.lk ? nw + l32 : 0) * a.skL;
    u32x4_t qf[QP], kf[QP];
#pragma unroll
    for (int c = 0; c < QP; ++c) {
      const int d0 = 8 * c + 4 * hf;
      qf[c] = (row_ok && d0 < a.d) ? *reinterpret_cast<const u32x4_t*>(qr + d0) : zero4;
      kf[c] = d0 < a.d ? *reinterpret_cast<const u32x4_t*>(kr + d0) : zero4;
    }
    // mask of keys nb + 8(r/4) + r%4
    const int nb = nw + 4 * hf;
    const int64_t moff = b * a.mB + h * a.mH + (int64_t)(i0 + l32) * a.mI;
    float mv[MASK != 0 ? 16 : 1];  // MASK 1: 0 drops the key
    if constexpr (MASK != 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = nb + 8 * (r >> 2) + (r & 3);
        mv[r] = 0.f;
        if (n < lim) {
          if constexpr (MASK == 1) mv[r] = reinterpret_cast<const uint8_t*>(a.mask)[moff + n * a.mJ] != 0 ? 1.f : 0.f;
          else mv[r] = reinterpret_cast<const float*>(a.mask)[moff + n * a.mJ];
        }
      }
    }
    f32x16_t acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int c = 0; c < QP; ++c) Mfma<float>::step(acc, kf[c], qf[c]);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float y = acc[r] * a.scale;
      if constexpr (MASK == 1) y = mv[r] != 0.f ? y : -INFINITY;
      if constexpr (MASK == 2) y += mv[r];
      s[r] = nb + 8 * (r >> 2) + (r & 3) < lim ? y : -INFINITY;
      bm = fmaxf(bm, s[r]);
    }
    bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
  }
  if (hf == 0) block_max[w][l32] = bm;
  __syncthreads();
  float m[CB + 1];  // the maximum before block j
  m[0] = -INFINITY;
#pragma unroll
  for (int j = 0; j < CB; ++j) m[j + 1] = fmaxf(m[j], block_max[j][l32]);
  auto base = [&](int j) { return m[j + 1] == -INFINITY ? 0.f : m[j + 1]; };
  if (nw < kend) {
    float own = base(0);
#pragma unroll
    for (int j = 1; j < CB; ++j) own = w == j ? base(j) : own;
    float part = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = f32_exp(s[r], own);
      ps[w][r][lane] = p;
      part += p;
    }
    parts[w][lane] = part;
  }
  __syncthreads();
  float l = 0.f;
  f32x16_t o;
#pragma unroll
  for (int r = 0; r < 16; ++r) o[r] = 0.f;
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    if (n0 + 32 * j >= kend) break;
    {
#pragma clang fp contract(off)  // the sum is rounded after the rescale, as in f32_attn_kernel
      const float cc = m[j + 1] > m[j] ? f32_exp(m[j], base(j)) : 1.f;
      l = l * cc;
      l = l + parts[j][lane];
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] *= cc;
    }
    if (w < OF) {
      float p[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) p[r] = ps[j][r][lane];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float x = n0 + 32 * j + 8 * (r >> 2) + 4 * hf + (r & 3) < a.lk ? xv[j][r] : 0.f;
        o = __builtin_amdgcn_mfma_f32_32x32x2f32(x, p[r], o, 0, 0, 0);
      }
    }
  }
  const float lc = l + __shfl_xor(l, 32, 64);
  if (!row_ok) return;
  const int64_t row = pair * a.lq + i0 + l32;
  float* const dst = a.chunks > 1 ? a.partial + ((int64_t)chunk * a.pairs * a.lq + row) * a.dv : a.out + row * a.dv;
  if (a.chunks > 1 && w == 0 && hf == 0)
    *reinterpret_cast<f32x2_t*>(a.stats + 2 * ((int64_t)chunk * a.pairs * a.lq + row)) = f32x2_t{m[CB], lc};
  if (w < OF) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = 32 * w + 8 * j + 4 * hf;
      const f32x4_t x = {o[4 * j], o[4 * j + 1], o[4 * j + 2], o[4 * j + 3]};
      if (col < a.dv) *reinterpret_cast<f32x4_t*>(dst + col) = a.chunks > 1 ? x : f32_final(x, m[CB], lc);
    }
  }
}

// The chunks of a split launch, four output elements per thread.
__global__ __launch_bounds__(256) void f32_combine_kernel(F32AttnArgs a) {
  const int64_t n = a.pairs * a.lq * (a.dv / 4);
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= n) return;
  const int64_t rows = a.pairs * a.lq;
  const int64_t r = idx / (a.dv / 4);
  const int col = 4 * (int)(idx - r * (a.dv / 4));
  const int i = (int)(r % a.lq);
  int lim = a.lk;
  if (a.causal != BIOPS_CAUSAL_NONE) {
    const int c = i + (a.causal == BIOPS_CAUSAL_BOTTOM_RIGHT ? a.lk - a.lq : 0) + 1;
    lim = c < 0 ? 0 : (c > a.lk ? a.lk : c);
  }
  const int nc = (lim + kF32Chunk - 1) / kF32Chunk;
  float m = -INFINITY, l = 0.f;
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int c = 0; c < nc; ++c) {
    const f32x2_t st = *reinterpret_cast<const f32x2_t*>(a.stats + 2 * (c * rows + r));
    const f32x4_t oc = *reinterpret_cast<const f32x4_t*>(a.partial + (c * rows + r) * a.dv + col);
    float c1, c2;
    f32_merge(m, l, st[0], st[1], c1, c2);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = f32_merge_o(o[e], oc[e], c1, c2, c == 0);
  }
  *reinterpret_cast<f32x4_t*>(a.out + r * a.dv + col) = f32_final(o, m, l);
}

// Workgroups of a launch: fewer than 2^32 threads.  A call of more tiles (millions of samples of one
// query row) takes several launches.
constexpr int64_t kF32MaxGrid = ((int64_t(1) << 32) - 1) / 256;

template <int DP, int QP, int DVP, bool SPLIT>
static int launch_f32_masks(F32AttnArgs a, int mask_kind, hipStream_t s) {
  const int64_t total = a.pairs * a.qtiles * (SPLIT ? a.chunks : 1);  // split: within one launch
  for (a.tile0 = 0; a.tile0 < total; a.tile0 += kF32MaxGrid) {
    const dim3 grid((unsigned)std::min(total - a.tile0, kF32MaxGrid)), block(256);
    if (mask_kind == 0) hipLaunchKernelGGL((f32_attn_kernel<DP, QP, DVP, 0, SPLIT>), grid, block, 0, s, a);
    else if (mask_kind == 1) hipLaunchKernelGGL((f32_attn_kernel<DP, QP, DVP, 1, SPLIT>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((f32_attn_kernel<DP, QP, DVP, 2, SPLIT>), grid, block, 0, s, a);
    const int rc = check_launch("f32_attn_kernel");
    if (rc != BIOPS_OK) return rc;
  }
  return BIOPS_OK;
}
template <int QP, int OF>
static int launch_f32_few(F32AttnArgs a, int mask_kind, hipStream_t s) {
  if (a.chunks == 0) a.chunks = 1;
  const dim3 grid((unsigned)(a.pairs * cdiv(a.lq, 32) * a.chunks)), block(256);
  if (mask_kind == 0) hipLaunchKernelGGL((f32_few_kernel<QP, OF, 0>), grid, block, 0, s, a);
  else if (mask_kind == 1) hipLaunchKernelGGL((f32_few_kernel<QP, OF, 1>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((f32_few_kernel<QP, OF, 2>), grid, block, 0, s, a);
  return check_launch("f32_few_kernel");
}
// Up to two workgroups of 32 rows and 128 keys per compute unit (more of them read K and V too often:
// 16 x 16 heads x 128 x 128, head size 64, 1024 workgroups, 17.6 -> 32.3 us), and not for a single block of
// keys with head sizes up to 96, which has nothing to spread (8 heads x 32 x 32, head size 64, 6.9 against
// 8.1 us).  MI355X, f32_attn_kernel against this, and with scores in memory: 8 heads x 100 x 100, head size
// 128, 26.7 -> 14.9 us (18.9); 200 x 200 28.0 -> 18.5 (22.7); 1 x 256 25.1 -> 16.2 (16.2); 1 head x 65 x 600
// 27.3 -> 18.9 (38.1); 8 heads x 16 x 2048 31.6 -> 23.0 (69.8); 8 x 65 x 65, head size 64, 12.7 -> 10.2 (17.5).
template <int DP>
static bool f32_few(const F32AttnArgs& a) {
  const int64_t chunks = a.partial ? a.chunks : 1;
  return (a.partial || a.lk <= kF32Chunk) && (DP > 96 || a.lk > kF32Keys) &&
         a.pairs * cdiv(a.lq, 32) * chunks <= 2 * (int64_t)device_cus();
}
template <int DP, int QP, int DVP>
static int launch_f32_attn(const F32AttnArgs& a, int mask_kind, hipStream_t s) {
  const bool few = f32_few<DP>(a);
  if (!a.partial) return few ? launch_f32_few<QP, DVP / 32>(a, mask_kind, s) : launch_f32_masks<DP, QP, DVP, false>(a, mask_kind, s);
  const int rc = few ? launch_f32_few<QP, DVP / 32>(a, mask_kind, s) : launch_f32_masks<DP, QP, DVP, true>(a, mask_kind, s);
  if (rc != BIOPS_OK) return rc;
  hipLaunchKernelGGL(f32_combine_kernel, dim3((unsigned)cdiv(a.pairs * a.lq * (a.dv / 4), 256)), dim3(256), 0, s, a);
  return check_launch("f32_combine_kernel");
}

// Chunks of a split launch, 0: the workgroups merge their chunks themselves.  Split while the
// query tiles leave the chip short of two workgroups per compute unit (one for two chunks, where the
// combine launch costs more than it spreads): 4 query tiles against 1200 keys (head size 128, additive
// mask) 205 -> 35 us, 128 tiles of 1000 causal keys 162 -> 103; 8 x 16 heads x 256 x 256, 256 tiles of two
// chunks, 41 against 44 split.
static int64_t f32_split_chunks(int64_t batch, int64_t hq, int64_t lq, int64_t lk, int64_t dv) {
  const int64_t tiles = batch * hq * cdiv(lq, kF32Rows), chunks = cdiv(lk, kF32Chunk);
  if (chunks < 2 || tiles >= (chunks == 2 ? 1 : 2) * (int64_t)device_cus()) return 0;
  if (tiles * chunks > kF32MaxGrid || cdiv(batch * hq * lq * (dv / 4), 256) > kF32MaxGrid) return 0;
  return chunks;
}
static int64_t f32_stats_offset(int64_t chunks, int64_t rows, int64_t dv) {
  return (chunks * rows * dv * 4 + 255) & ~int64_t(255);
}

}  // namespace biops

using namespace biops;

extern "C" int biops_sdpa_f32_supported(int64_t batch, int64_t hq, int64_t lq, int64_t lk, int64_t d, int64_t dv) {
  const int64_t lim = int64_t(1) << 30;  // the sizes of one sample: the path must not depend on the batch
  (void)batch;
  (void)hq;
  return d >= 1 && d <= 128 && dv >= 1 && dv <= 128 && d % 4 == 0 && dv % 4 == 0 && lq < lim && lk < lim;
}

extern "C" int64_t biops_sdpa_f32_workspace_size(int64_t batch, int64_t hq, int64_t lq, int64_t lk, int64_t d, int64_t dv) {
  if (batch < 0 || hq < 0 || lq < 0 || lk < 0 || !biops_sdpa_f32_supported(batch, hq, lq, lk, d, dv)) return -1;
  const int64_t chunks = f32_split_chunks(batch, hq, lq, lk, dv), rows = batch * hq * lq;
  return chunks ? f32_stats_offset(chunks, rows, dv) + chunks * rows * 8 : 0;
}

extern "C" int biops_sdpa_f32(int64_t batch, int64_t hq, int64_t hkv, int64_t lq, int64_t lk, int64_t d, int64_t dv,
                              const void* q, int64_t sqB, int64_t sqH, int64_t sqL, const void* k, int64_t skB,
                              int64_t skH, int64_t skL, const void* v, int64_t svB, int64_t svH, int64_t svL,
                              const void* mask, int mask_dtype, int64_t mB, int64_t mH, int64_t mI, int64_t mJ,
                              int causal, float scale, void* out, void* workspace, int64_t workspace_bytes,
                              void* stream) {
  if (batch < 0 || hq < 0 || hkv <= 0 || lq < 0 || lk < 0) return fail(BIOPS_ERR_ARG, "invalid attention sizes");
  if (!biops_sdpa_f32_supported(batch, hq, lq, lk, d, dv))
    return fail(BIOPS_ERR_SIZE, "fused float32 attention takes head sizes <= 128, multiples of 4");
  if (hq % hkv != 0) return fail(BIOPS_ERR_ARG, "query heads must be a multiple of kv heads");
  if (mask && causal != BIOPS_CAUSAL_NONE) return fail(BIOPS_ERR_ARG, "mask and causal are exclusive");
  if (mask && mask_dtype != BIOPS_BOOL && mask_dtype != BIOPS_F32)
    return fail(BIOPS_ERR_DTYPE, "mask dtype must be bool or the score dtype");
  if (batch == 0 || hq == 0 || lq == 0) return BIOPS_OK;
  if (!q || !out || (lk > 0 && (!k || !v))) return fail(BIOPS_ERR_ARG, "null pointer");
  for (const void* p : {q, k, v, static_cast<const void*>(out)})
    if (reinterpret_cast<uintptr_t>(p) & 15) return fail(BIOPS_ERR_LAYOUT, "fused float32 attention needs 16-byte aligned tensors");
  for (int64_t st : {sqB, sqH, sqL, skB, skH, skL, svB, svH, svL})
    if (st & 3) return fail(BIOPS_ERR_LAYOUT, "fused float32 attention needs 16-byte aligned rows (strides multiples of 4)");
  for (int64_t st : {skL, svL})
    if (st < 0 || 4 * kF32Keys * st >= (int64_t(1) << 32))
      return fail(BIOPS_ERR_LAYOUT, "fused float32 attention row strides too large");
  F32AttnArgs a{};
  a.q = static_cast<const float*>(q); a.k = static_cast<const float*>(k); a.v = static_cast<const float*>(v);
  a.out = static_cast<float*>(out);
  a.mask = mask;
  a.sqB = sqB; a.sqH = sqH; a.sqL = sqL; a.skB = skB; a.skH = skH; a.skL = skL;
  a.svB = svB; a.svH = svH; a.svL = svL;
  a.mB = mB; a.mH = mH; a.mI = mI; a.mJ = mJ;
  a.hq = hq; a.hkv = hkv; a.group = hq / hkv; a.pairs = batch * hq;
  a.lq = (int32_t)lq; a.lk = (int32_t)lk; a.d = (int32_t)d; a.dv = (int32_t)dv;
  a.qtiles = (int32_t)cdiv(lq, kF32Rows);
  a.scale = scale;
  a.causal = causal;
  const int kind = !mask ? 0 : (mask_dtype == BIOPS_BOOL ? 1 : 2);
  a.mvec = mJ == 1;
  const int64_t need = biops_sdpa_f32_workspace_size(batch, hq, lq, lk, d, dv);
  if (workspace_bytes < need)
    return fail(BIOPS_ERR_SIZE, "workspace %lld < %lld bytes", (long long)workspace_bytes, (long long)need);
  if (need > 0) {
    if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255))
      return fail(BIOPS_ERR_LAYOUT, "workspace must be 256-byte aligned");
    a.chunks = (int32_t)cdiv(lk, kF32Chunk);
    a.partial = static_cast<float*>(workspace);
    a.stats = reinterpret_cast<float*>(static_cast<char*>(workspace) + f32_stats_offset(a.chunks, batch * hq * lq, dv));
  }
  hipStream_t s = (hipStream_t)stream;
  if (d <= 64 && dv <= 64) return launch_f32_attn<64, 8, 64>(a, kind, s);
  if (d <= 96 && dv <= 96) {
    if (d <= 72) return launch_f32_attn<96, 9, 96>(a, kind, s);
    if (d <= 80) return launch_f32_attn<96, 10, 96>(a, kind, s);
    return launch_f32_attn<96, 12, 96>(a, kind, s);
  }
  return launch_f32_attn<128, 16, 128>(a, kind, s);
}
