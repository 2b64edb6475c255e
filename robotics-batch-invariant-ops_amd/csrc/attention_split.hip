// Attention of few query rows against many keys (decoding steps, action chunks against a cached
// prefix) for 16-bit inputs: the keys are split over workgroups.
//
// The fused kernel (attention_fused.hip) gives one workgroup 128 query rows of one head and the
// whole key range, twice.  With one query row that leaves 127 of 128 rows empty, reads a
// key/value head once per query head of its group, and a batch of 8 x 16 heads keeps only half of
// the compute units busy.  Here the query heads of a group and their query rows are packed into
// the rows of one problem (row = head in group * lq + query row), in tiles of 32, and a call runs
//   1. split_score_kernel, one workgroup per kSplitKeys keys of a (batch, kv head): S = Q K^T and
//      the reference's transform (round, scale, round, mask), the 16-bit scores s to a workspace
//      and, per row, the maximum m_j and the sum l_j of exp(s - m_j) over the workgroup's keys;
//   2. split_value_kernel, one workgroup per kvalue keys and row tile: m = max m_j,
//      l = sum l_j exp(m_j - m) in key order, P = round(exp(s - m) / l) in the input dtype, the
//      fp32 partial O = P V of its keys;
//   3. split_combine_kernel: the partial O added in key order and rounded once (one value split:
//      kernel 2 writes the output itself).
// The roundings are those of the eager composite (batch_invariant_ops.py:1194-1212), as in the
// fused kernel: S comes from the same MFMA sequence (128-byte steps of the head dimension, chunk
// pairs in order) with the same transform, and P is normalised before it is rounded; only the
// fp32 orders of the row sum and of the P V sum differ.
//
// Batch invariance: the key ranges of the workgroups are fixed multiples (kSplitKeys,
// value_split_keys) that depend on the key count only, and every sum runs in key order.  How many row tiles share a workgroup depends on
// the launch size; it changes no value.
//
// MI355X, 8 samples, 16 / 4 heads of 128, one query row, 2048 keys (33.6 MB): fused kernel 82 us,
// here 18.6 (scores 6.5, values 8.6, combine 3.5); 16 samples, 64 / 8 heads, 4096 keys (268 MB)
// 358 -> 68 us (4.3 TB/s on K, 4.2 TB/s on V).
//
// Bound: a decoding step streams K and V once (the scores of a few rows are small beside them);
// K goes from memory straight to the MFMA operand registers, V through a wavefront's own LDS
// rows to the transposing read, without workgroup barriers in either loop.
#include <algorithm>

#include "gemm.h"
#include "rowops.h"

namespace biops {

constexpr int kSplitKeys = 256;      // keys per workgroup of split_score_kernel, 64 per wavefront
// Calls taken (a rule on the sizes of one sample; the batch size must not enter).  Kernel time,
// MI355X, bf16, head size 128, fused kernel against this path:
//   query rows, at 16 samples x 8 kv heads x 4096 keys, 4 heads per kv head, where the fused
//   kernel has enough tiles to fill the chip: 1 row 358 -> 68 us (8 heads per kv head), 16 rows
//   183 -> 136, 32 rows 188 -> 206; one sample gains at any row count (16 heads, 64 rows, 1500
//   keys: 64 -> 28), but the line has to hold for every batch size;
//   keys, 1 sample, 16 / 4 heads, one row: 200 keys 16.2 -> 10.5, 400 keys 22.8 -> 13.5, 700 keys
//   32.6 -> 13.9.  Two more launches cost about 4 us of host time, so calls up to 512 keys, which
//   the host bounds either way, stay on the fused kernel.
constexpr int kSplitMaxQuery = 16;   // query rows per head
constexpr int kSplitMinKeys = 512;   // longer key ranges are split

struct SplitArgs {
  const void* q; const void* k; const void* v; void* out;
  const void* mask;
  void* s;            // scores in fragment order (score_offset)
  float* stats;       // {m_j, l_j} of [pair][key tile][padded row]
  float* partial;     // [value split][pair][row][dv]
  int64_t sqB, sqH, sqL, skB, skH, skL, svB, svH, svL;
  int64_t mB, mH, mI;
  int32_t hkv, group, lq, lk, d, dv;
  int32_t rows, row_tiles, tiles_per_wg, row_groups;  // rows = group * lq
  int32_t pairs, key_tiles, splits, split_keys;
  float scale;
};

// Scores of row tile rt: one 16-byte piece per lane and 16-key chunk, the A operand fragment of
// the P V MFMA (lane L: row L % 32, keys 4(L/32) + (0..3) and + 8 of the chunk).
__device__ __forceinline__ int64_t score_offset(const SplitArgs& a, int pair, int rt, int chunk) {
  return (((int64_t)pair * a.row_tiles + rt) * (4 * cdiv(a.lk, 64)) + chunk) * 512;
}

template <typename T>
__device__ __forceinline__ uint32_t split_pack2(float x, float y) {
  if constexpr (std::is_same<T, bf16_t>::value) return f32x2_to_bf16x2_bits(x, y);
  else return (uint32_t)Num<T>::to_bits(x) | ((uint32_t)Num<T>::to_bits(y) << 16);
}

// exp(x - m).  The difference is taken before the factor log2 e: keys that carry a mask of the type's
// lowest value leave a finite maximum whose multiple by log2 e is not (a wavefront's 64 keys masked
// that way gave NaN with fma(x, log2 e, -m log2 e)).
__device__ __forceinline__ float split_exp(float x, float m) { return __builtin_amdgcn_exp2f((x - m) * kLog2e); }

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
  __shared__ float part[2][4][32][2];
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
    float m = -INFINITY, l = 0.f;
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
        auto transform = [&](auto open) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            float s = Num<T>::round(Num<T>::round(acc[hb][r]) * a.scale);
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
      }
      m = fmaxf(m, __shfl_xor(m, 32, 64));
      const float base = m == -INFINITY ? 0.f : m;
#pragma unroll
      for (int hb = 0; hb < 2; ++hb)
#pragma unroll
        for (int r = 0; r < 16; ++r) l += split_exp(acc[hb][r], base);
      l += __shfl_xor(l, 32, 64);
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
    // the four wavefronts' statistics, in key order (two buffers: one barrier per row tile)
    float (*const p)[32][2] = part[(rt - rt0) & 1];
    if (hf == 0) {
      p[w][l32][0] = m;
      p[w][l32][1] = l;
    }
    lds_barrier();
    if (tid < 32) {
      float mm = p[0][tid][0];
#pragma unroll
      for (int j = 1; j < 4; ++j) mm = fmaxf(mm, p[j][tid][0]);
      const float base = mm == -INFINITY ? 0.f : mm;
      float ll = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        ll = __builtin_fmaf(p[j][tid][1], split_exp(p[j][tid][0], base), ll);
      float* st = a.stats + 2 * (((int64_t)pair * a.key_tiles + kt) * 32 * a.row_tiles + 32 * rt + tid);
      st[0] = mm;
      st[1] = ll;
    }
  }
}

// RT row tiles of one (pair, value split).  Wavefront w takes the w-th 16-key chunk of every
// 64-key block, all columns; PF blocks of V rows and scores are in flight per wavefront.
template <typename T, int DVP, int RT, int PF>
__global__ __launch_bounds__(256) void split_value_kernel(SplitArgs a) {
  constexpr int E = sizeof(T);
  constexpr int VCH = DVP / 8;       // 16-byte chunks per V row
  constexpr int OF = DVP / 32;       // 32-column output blocks
  constexpr int VL = 16 * VCH / 64;  // V loads per lane and chunk
  constexpr int ROWS = 32 * RT;
  constexpr int SG = 256 / ROWS;     // threads per row in the statistics
  constexpr int SREG = 4;
  constexpr int V_BYTES = 16 * DVP * 2;                       // one wavefront's V rows
  constexpr int OB = OF < 4 ? OF : 4;                         // column blocks summed per round
  constexpr int SMEM = 4 * OB * 4096 > 8 * V_BYTES ? 4 * OB * 4096 : 8 * V_BYTES;
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  __shared__ float sm[SG][ROWS], sl[SG][ROWS];
  __shared__ float base_[ROWS], inv_[ROWS];
  const int rgroups = (a.row_tiles + RT - 1) / RT;
  int x = blockIdx.x;
  const int rg = x % rgroups;
  x /= rgroups;
  const int sp = x % a.splits;
  const int pair = x / a.splits;
  const int hk = pair % a.hkv;
  const int64_t b = pair / a.hkv;
  const int tid = threadIdx.x;
  const int w = tid >> 6, lane = tid & 63, hf = lane >> 5, l32 = lane & 31;
  const u32x4_t zero4 = {0u, 0u, 0u, 0u};
  const int rt0 = rg * RT;
  const int k0 = sp * a.split_keys;
  const int k1 = k0 + a.split_keys < a.lk ? k0 + a.split_keys : a.lk;
  const int nblk = (k1 - k0 + 63) / 64;

  const char* vbase = reinterpret_cast<const char*>(a.v) + E * (b * a.svB + hk * a.svH);
  u32x4_t vr[PF][VL], sr[PF][RT];
  auto load = [&](int blk, int slot) {
    const int kb = k0 + 64 * blk + 16 * w;
    if (kb >= k1) return;
#pragma unroll
    for (int p = 0; p < VL; ++p) {
      const int s = lane + 64 * p, r = s / VCH, c = s % VCH;
      const bool ok = kb + r < k1 && 8 * c < a.dv;
      const u32x4_t y = *reinterpret_cast<const u32x4_t*>(vbase + E * ((int64_t)(ok ? kb + r : kb) * a.svL + (ok ? 8 * c : 0)));
      vr[slot][p] = ok ? y : zero4;
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const int row = 32 * (rt0 + t) + l32;
      const char* p = reinterpret_cast<const char*>(a.s) + E * (score_offset(a, pair, rt0 + t, kb / 16) + 8 * lane);
      sr[slot][t] = row < a.rows ? *reinterpret_cast<const u32x4_t*>(p) : zero4;
    }
  };
#pragma unroll
  for (int j = 0; j < PF; ++j) load(j, j);

  // m and 1/l of the rows: SG threads per row take key tiles g, g + SG, ... (the first SREG of a
  // thread stay in registers between the maximum and the sum), then g in order
  {
    const int r = tid % ROWS, g = tid / ROWS;
    const int row = 32 * rt0 + r;
    const int nt = row < 32 * a.row_tiles ? a.key_tiles : 0;
    const int64_t step = 32 * a.row_tiles;
    const f32x2_t* st = reinterpret_cast<const f32x2_t*>(a.stats) + (int64_t)pair * a.key_tiles * step + row;
    f32x2_t y[SREG];
#pragma unroll
    for (int u = 0; u < SREG; ++u) y[u] = g + SG * u < nt ? st[(g + SG * u) * step] : f32x2_t{-INFINITY, 0.f};
    float m = -INFINITY;
#pragma unroll
    for (int u = 0; u < SREG; ++u) m = fmaxf(m, y[u][0]);
    for (int j = g + SG * SREG; j < nt; j += SG) m = fmaxf(m, st[j * step][0]);
    sm[g][r] = m;
    lds_barrier();
#pragma unroll
    for (int j = 0; j < SG; ++j) m = fmaxf(m, sm[j][r]);
    const float base = m == -INFINITY ? 0.f : m;
    float l = 0.f;
    auto add = [&](const f32x2_t& z) {
      l = __builtin_fmaf(z[1], split_exp(z[0], base), l);
    };
#pragma unroll
    for (int u = 0; u < SREG; ++u) add(y[u]);
    for (int j = g + SG * SREG; j < nt; j += SG) add(st[j * step]);
    sl[g][r] = l;
    lds_barrier();
    if (g == 0) {
      float lt = sl[0][r];
#pragma unroll
      for (int j = 1; j < SG; ++j) lt += sl[j][r];
      const bool dead = m == -INFINITY || lt == 0.f;
      base_[r] = base;
      inv_[r] = dead ? 0.f : 1.0f / lt;
    }
    lds_barrier();
  }
  float base[RT], inv[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    base[t] = base_[32 * t + l32];
    inv[t] = inv_[32 * t + l32];
  }

  f32x16_t oacc[RT][OF];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int e = 0; e < OF; ++e)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[t][e][r] = 0.f;
  // Transposing V reads: lane s of a 16-lane group points at row s/4, column 4(s%4) and receives
  // four rows of one column; rows 4hf + (0..3) and + 8 match the scores' key order.
  const int vrow = 4 * hf + ((lane & 15) >> 2);
  const int vcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  char* const vw = smem + 2 * V_BYTES * w;
  auto block = [&](int blk, int slot, char* vb) {
    if (k0 + 64 * blk + 16 * w >= k1) return;
#pragma unroll
    for (int p = 0; p < VL; ++p) {
      const int s = lane + 64 * p;
      *reinterpret_cast<u32x4_t*>(vb + lds_off_n<VCH>(s / VCH, 8 * (s % VCH))) = vr[slot][p];
    }
    u32x4_t pa[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      float p[8];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        p[e] = split_exp(Num<T>::from_bits((sr[slot][t][e >> 1] >> (16 * (e & 1))) & 0xffffu), base[t]) * inv[t];
      pa[t] = u32x4_t{split_pack2<T>(p[0], p[1]), split_pack2<T>(p[2], p[3]), split_pack2<T>(p[4], p[5]),
                      split_pack2<T>(p[6], p[7])};
    }
    load(blk + PF, slot);
    // the rows were written by other lanes of this wavefront: LDS operations of a wavefront
    // complete in order, the fence keeps the compiler from reordering them
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int e = 0; e < OF; ++e) {
      const u32x2_t lo = lds_read_tr16(vb + lds_off_n<VCH>(vrow, 32 * e + vcol));
      const u32x2_t hi = lds_read_tr16(vb + lds_off_n<VCH>(vrow + 8, 32 * e + vcol));
      const u32x4_t vf = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
      for (int t = 0; t < RT; ++t) Mfma<T>::step(oacc[t][e], pa[t], vf);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  for (int blk = 0; blk < nblk; blk += PF)
#pragma unroll
    for (int j = 0; j < PF; ++j)
      if (blk + j < nblk) block(blk + j, j, vw + V_BYTES * (j & 1));

  // O of the four wavefronts as (w0 + w1) + (w2 + w3): OB column blocks per round through LDS
  // (register r of lane L is row 8(r/4) + 4(L/32) + r%4, column L % 32 of its block).
  // Registers past the tile's last valid row (groups of 8 rows) are left out.
  float* const red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int left = a.rows - 32 * (rt0 + t);
    const int nr = left >= 32 ? 16 : (left <= 0 ? 0 : 4 * ((left + 7) / 8));
#pragma unroll
    for (int e0 = 0; e0 < OF; e0 += OB) {
      lds_barrier();
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        if (4 * r4 < nr) {
#pragma unroll
          for (int e = 0; e < OB; ++e)
#pragma unroll
            for (int r = 4 * r4; r < 4 * r4 + 4; ++r) red[((w * 16 + r) * OB + e) * 64 + lane] = oacc[t][e0 + e][r];
        }
      }
      lds_barrier();
      for (int idx = tid; idx < nr * OB * 64; idx += 256) {  // (r * OB + e) * 64 + lane
        const float o = (red[idx] + red[idx + OB * 1024]) + (red[idx + 2 * OB * 1024] + red[idx + 3 * OB * 1024]);
        const int ln = idx & 63, e = (idx >> 6) % OB, r = idx / (64 * OB);
        const int row = 32 * (rt0 + t) + 8 * (r >> 2) + 4 * (ln >> 5) + (r & 3);
        const int col = 32 * (e0 + e) + (ln & 31);
        if (row < a.rows && col < a.dv) {
          // out is contiguous [b, kv head, row = head in group * lq + query row, dv]
          if (a.splits == 1) Num<T>::store(reinterpret_cast<T*>(a.out) + ((int64_t)pair * a.rows + row) * a.dv + col, o);
          else a.partial[(((int64_t)sp * a.pairs + pair) * a.rows + row) * a.dv + col] = o;
        }
      }
    }
  }
}

// Four output elements per thread: the partial O of the value splits added in key order.
template <typename T>
__global__ __launch_bounds__(256) void split_combine_kernel(const float* partial, T* out, int64_t n4, int splits) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const f32x4_t* p = reinterpret_cast<const f32x4_t*>(partial) + i;
  f32x4_t o = p[0];
#pragma unroll 8
  for (int s = 1; s < splits; ++s) o += p[s * n4];
  *reinterpret_cast<u32x2_t*>(out + 4 * i) = u32x2_t{split_pack2<T>(o[0], o[1]), split_pack2<T>(o[2], o[3])};
}

// Keys per workgroup of split_value_kernel: short ranges for few keys (a decoding step of 8
// samples with 4 kv heads and 2048 keys: 256 workgroups of 256 keys 8.6 us, 128 of 512 keys 11.6),
// longer ones as the partial outputs and the per-workgroup fixed cost grow (4096 keys, 128 kv
// heads: 512 keys 32 us, 256 keys 39).
static int value_split_keys(int64_t lk) { return lk <= 2048 ? 256 : (lk <= 8192 ? 512 : 1024); }

struct SplitSizes {
  int64_t stats, partial, total;  // byte offsets of the statistics and partial sums, and the end
  int64_t rows, row_tiles, key_tiles, splits;
};
static SplitSizes split_sizes(int64_t batch, int64_t hq, int64_t hkv, int64_t lq, int64_t lk, int64_t dv) {
  auto al = [](int64_t b) { return (b + 255) & ~int64_t(255); };
  SplitSizes z{};
  z.rows = hq / hkv * lq;
  z.row_tiles = cdiv(z.rows, 32);
  z.key_tiles = cdiv(lk, kSplitKeys);
  z.splits = cdiv(lk, value_split_keys(lk));
  const int64_t pairs = batch * hkv;
  z.stats = al(pairs * z.row_tiles * cdiv(lk, 64) * 64 * 32 * 2);
  z.partial = z.stats + al(pairs * z.key_tiles * z.row_tiles * 32 * 8);
  z.total = z.partial + (z.splits > 1 ? al(z.splits * pairs * z.rows * dv * 4) : 0);
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

// Row tiles per workgroup and blocks in flight: two tiles share the V rows where their
// accumulators leave two wavefronts per SIMD (not with 256-wide values).
template <typename T, int DVP, int RT, int PF>
static int launch_values_rt(const SplitArgs& a, hipStream_t s) {
  const int64_t wgs = (int64_t)a.pairs * a.splits * cdiv(a.row_tiles, RT);
  hipLaunchKernelGGL((split_value_kernel<T, DVP, RT, PF>), dim3((unsigned)wgs), dim3(256), 0, s, a);
  return check_launch("split_value_kernel");
}

template <typename T>
static int launch_values(const SplitArgs& a, hipStream_t s) {
  if (a.dv > 128) return launch_values_rt<T, 256, 1, 2>(a, s);
  if (a.row_tiles == 1) return a.dv <= 64 ? launch_values_rt<T, 64, 1, 4>(a, s) : launch_values_rt<T, 128, 1, 4>(a, s);
  return a.dv <= 64 ? launch_values_rt<T, 64, 2, 2>(a, s) : launch_values_rt<T, 128, 2, 2>(a, s);
}

template <typename T>
static int launch_split(const SplitArgs& a, int mask_kind, hipStream_t s) {
  int rc = mask_kind == 0 ? launch_scores<T, 0>(a, s) : (mask_kind == 1 ? launch_scores<T, 1>(a, s) : launch_scores<T, 2>(a, s));
  if (rc != BIOPS_OK) return rc;
  rc = launch_values<T>(a, s);
  if (rc != BIOPS_OK || a.splits == 1) return rc;
  const int64_t n4 = (int64_t)a.pairs * a.rows * a.dv / 4;  // dv is a multiple of 8
  hipLaunchKernelGGL(split_combine_kernel<T>, dim3((unsigned)cdiv(n4, 256)), dim3(256), 0, s, a.partial,
                     reinterpret_cast<T*>(a.out), n4, a.splits);
  return check_launch("split_combine_kernel");
}

}  // namespace biops

using namespace biops;

extern "C" int64_t biops_sdpa_split_workspace_size(int dtype, int64_t batch, int64_t hq, int64_t hkv, int64_t lq,
                                                   int64_t lk, int64_t d, int64_t dv, int causal) {
  if (!biops_attention_fused_supported(dtype, d, dv) || causal != BIOPS_CAUSAL_NONE) return -1;
  if (batch <= 0 || hq <= 0 || hkv <= 0 || hq % hkv != 0 || lq <= 0 || lq > kSplitMaxQuery || lk <= kSplitMinKeys) return -1;
  const SplitSizes z = split_sizes(batch, hq, hkv, lq, lk, dv);
  const int64_t lim = int64_t(1) << 31;
  // 32-bit workgroup counts and row / key indices
  if (lk >= lim / 2 || z.rows >= lim / 64 || batch * hkv >= lim / (z.key_tiles * z.row_tiles) ||
      cdiv(batch * hq * lq * dv / 4, 256) >= lim)
    return -1;
  return z.total;
}

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
  const SplitSizes z = split_sizes(batch, hq, hkv, lq, lk, dv);
  char* ws = reinterpret_cast<char*>(workspace);
  SplitArgs a{};
  a.q = q; a.k = k; a.v = v; a.out = out; a.mask = mask;
  a.s = ws;
  a.stats = reinterpret_cast<float*>(ws + z.stats);
  a.partial = reinterpret_cast<float*>(ws + z.partial);
  a.sqB = sqB; a.sqH = sqH; a.sqL = sqL; a.skB = skB; a.skH = skH; a.skL = skL;
  a.svB = svB; a.svH = svH; a.svL = svL;
  a.mB = mB; a.mH = mH; a.mI = mI;
  a.hkv = (int32_t)hkv; a.group = (int32_t)(hq / hkv); a.lq = (int32_t)lq; a.lk = (int32_t)lk;
  a.d = (int32_t)d; a.dv = (int32_t)dv;
  a.rows = (int32_t)z.rows; a.row_tiles = (int32_t)z.row_tiles;
  a.pairs = (int32_t)(batch * hkv); a.key_tiles = (int32_t)z.key_tiles;
  a.splits = (int32_t)z.splits; a.split_keys = value_split_keys(lk);
  a.scale = scale;
  // row tiles per workgroup of the score kernel: as many as leave two workgroups per compute unit
  // (each workgroup reads its keys once for all of its row tiles)
  const int64_t wgs = (int64_t)a.pairs * a.key_tiles * a.row_tiles;
  a.tiles_per_wg = (int32_t)std::max<int64_t>(1, std::min<int64_t>(a.row_tiles, wgs / (2 * device_cus())));
  a.row_groups = (int32_t)cdiv(a.row_tiles, a.tiles_per_wg);
  hipStream_t s = (hipStream_t)stream;
  const int kind = !mask ? 0 : (mask_dtype == BIOPS_BOOL ? 1 : 2);
  return dtype == BIOPS_F16 ? launch_split<f16_t>(a, kind, s) : launch_split<bf16_t>(a, kind, s);
}
