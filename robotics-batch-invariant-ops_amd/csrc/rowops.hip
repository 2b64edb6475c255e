// Softmax / log-softmax and mean / L2-norm reductions.
#include <algorithm>
#include <type_traits>

#include "rowops.h"

namespace biops {

// ------------------------------------------------------------------ softmax ----
struct SoftmaxArgs {
  const void* in;
  void* out;
  int64_t rows, cols, ld_in, ld_out;
};

// Sum and maximum over a workgroup of NW wavefronts (each wavefront's butterfly, then the
// wavefront results in wavefront order); every thread returns the same bits.  `part` holds NW
// floats and may be reused after the next barrier.
template <int NW>
__device__ __forceinline__ float block_sum(float v, float* part) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = part[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) s += part[i];
  return s;
}
template <int NW>
__device__ __forceinline__ float block_max(float v, float* part) {
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = part[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) s = fmaxf(s, part[i]);
  return s;
}

// Rows longer than a wavefront's registers (over 256 chunks): one workgroup of T threads per
// row, thread t holding chunks t, t + T, ... (NC of them, all loads issued before the first
// reduction), so the row is read from memory once.  LOOP: rows past the register file of 1024
// threads, read three times in groups of NC chunks per thread.  Bound by the row's read and
// write; one wavefront per row, as the shorter rows have, leaves most of the chip idle at the row
// counts of a decoding batch.  The same rule for every row count: the tree may depend on the row
// length only.  MI355X, one wavefront per row with element-wise loads of misaligned rows ->
// this: log-softmax [32, 50257] fp32 217 -> 12.5 us a call, softmax [64, 32000] bf16 57 -> 6.4 us,
// [4096, 8192] bf16 44.3 -> 22.8 us (5.9 TB/s of read + write), [1, 131072] fp32 376 -> 38 us.
template <typename Tin, typename Tout, int MODE, int T, int NC, bool LOOP>
__global__ __launch_bounds__(T) void softmax_block_kernel(SoftmaxArgs a) {
  constexpr int VEC = 16 / sizeof(Tin);
  constexpr int NW = T / 64;
  __shared__ float part[2][NW];
  const int64_t r = blockIdx.x;
  const int t = threadIdx.x;
  const Tin* in = reinterpret_cast<const Tin*>(a.in) + r * a.ld_in;
  Tout* out = reinterpret_cast<Tout*>(a.out) + r * a.ld_out;
  const int64_t cols = a.cols, nchunks = cdiv(cols, VEC);
  const int64_t groups = LOOP ? cdiv(nchunks, T * NC) : 1;

  // Chunk of group g held in slot j, and its raw bits; columns past the row end read as -inf.
  auto chunk = [&](int64_t g, int j) { return t + T * (g * NC + j); };
  constexpr uint32_t kNegInf = sizeof(Tin) == 4 ? 0xff800000u : (std::is_same<Tin, bf16_t>::value ? 0xff80ff80u : 0xfc00fc00u);
  u32x4_t raw[NC];
  auto load = [&](int64_t g) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int64_t c0 = chunk(g, j) * VEC;
      raw[j] = u32x4_t{kNegInf, kNegInf, kNegInf, kNegInf};
      if (c0 + VEC <= cols) {
        raw[j] = load_16(in + c0);
      } else if (c0 < cols) {
#pragma unroll
        for (int e = 0; e < VEC - 1; ++e) {
          if (c0 + e < cols) {
            if constexpr (sizeof(Tin) == 4) {
              raw[j][e] = __float_as_uint(in[c0 + e]);
            } else {
              const uint32_t x = reinterpret_cast<const uint16_t*>(in)[c0 + e];
              raw[j][e >> 1] = (e & 1) ? (raw[j][e >> 1] & 0xffffu) | (x << 16) : (raw[j][e >> 1] & 0xffff0000u) | x;
            }
          }
        }
      }
    }
  };
  // Redefines the 16-bit rows' registers, so that the compiler unpacks them again instead of
  // keeping the fp32 values of a whole row across a reduction (it spilled at NC = 16).
  auto keep_raw = [&]() {
    if constexpr (!LOOP && sizeof(Tin) == 2) {
#pragma unroll
      for (int j = 0; j < NC; ++j) asm volatile("" : "+v"(raw[j]));
    }
  };
  // exp of a column past the row end is 0 (NaN only where the whole row gives NaN)
  auto exps = [&](float (&v)[VEC], bool neg_inf, const SoftShift& shift) {
#pragma unroll
    for (int e = 0; e < VEC; ++e)
      v[e] = (MODE != kLogSoftmax && neg_inf) ? 0.f : soft_exp<Tin, Tout>(v[e], shift);
  };

  float mx = -INFINITY;
  for (int64_t g = 0; g < groups; ++g) {
    load(g);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      float v[VEC];
      unpack_chunk<Tin>(raw[j], v);
#pragma unroll
      for (int e = 0; e < VEC; ++e) mx = fmaxf(mx, v[e]);
    }
  }
  mx = block_max<NW>(mx, part[0]);
  keep_raw();
  const bool neg_inf = (mx == -INFINITY);
  const SoftShift shift = soft_shift<Tin>((MODE == kLogSoftmax || !neg_inf) ? mx : 0.f);

  // fp32 softmax of a resident row keeps the exponentials in the row's registers
  constexpr bool kKeepExp = !LOOP && sizeof(Tin) == 4 && MODE == kSoftmax;
  float sum = 0.f;
  for (int64_t g = 0; g < groups; ++g) {
    if constexpr (LOOP) load(g);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      float v[VEC];
      unpack_chunk<Tin>(raw[j], v);
      exps(v, neg_inf, shift);
#pragma unroll
      for (int e = 0; e < VEC; ++e) sum += v[e];
      if constexpr (kKeepExp) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) raw[j][e] = __float_as_uint(v[e]);
      }
    }
  }
  sum = block_sum<NW>(sum, part[1]);
  keep_raw();

  const bool zero = (sum == 0.f);
  const float inv = zero ? 0.f : 1.0f / sum;
  const float lse = MODE == kLogSoftmax ? logf(sum) : 0.f;
  for (int64_t g = 0; g < groups; ++g) {
    if constexpr (LOOP) load(g);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int64_t ci = chunk(g, j);
      if (ci >= nchunks) continue;
      float v[VEC];
      unpack_chunk<Tin>(raw[j], v);
      if constexpr (MODE == kLogSoftmax) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] = v[e] - mx - lse;
      } else {
        if constexpr (!kKeepExp) exps(v, neg_inf, shift);
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] = zero ? 0.f : v[e] * inv;
      }
      store_row_chunk<Tout, VEC, true>(out, cols, ci * VEC, v);
    }
  }
}

// Rows of at most 64*NC chunks (NC = 1, 2, 4 per lane): fit_rows<NC>() rows per wavefront, whose
// loads are all issued before the first reduction, with non-temporal output stores.
// Rows per wavefront R for rows of NC chunks per lane: two rows of one chunk, else one row
// (measured on 512 MiB of bf16 rows: more rows per wavefront left fewer wavefronts in flight).
template <int NC>
constexpr int fit_rows() { return NC == 1 ? 2 : 1; }

template <typename Tin, typename Tout, int MODE, int NC>
__global__ __launch_bounds__(256) void softmax_fit_kernel(SoftmaxArgs a) {
  constexpr int R = fit_rows<NC>();
  const int64_t r = ((int64_t)blockIdx.x * kRowWaves + (threadIdx.x >> 6)) * R;
  if (r >= a.rows) return;
  const int n = a.rows - r < R ? (int)(a.rows - r) : R;
  softmax_rows_fit<Tin, Tout, MODE, R, NC>(reinterpret_cast<const Tin*>(a.in) + r * a.ld_in, a.ld_in,
                                           reinterpret_cast<Tout*>(a.out) + r * a.ld_out, a.ld_out, n,
                                           a.cols);
}

// A launch has fewer than 2^32 threads: rows beyond that go to further launches of the same kernel.
// Calls launch(first row, rows) with at most `per_group` rows per `threads` threads.
template <typename F>
static int launch_row_ranges(int64_t rows, int per_group, int threads, F&& launch) {
  const int64_t most = ((int64_t(1) << 32) - 1) / threads * per_group;
  for (int64_t first = 0; first < rows; first += most) {
    const int rc = launch(first, std::min(rows - first, most));
    if (rc != BIOPS_OK) return rc;
  }
  return BIOPS_OK;
}

template <typename Tin, typename Tout>
static SoftmaxArgs softmax_rows_from(const SoftmaxArgs& a, int64_t first, int64_t rows) {
  SoftmaxArgs b = a;
  b.in = reinterpret_cast<const Tin*>(a.in) + first * a.ld_in;
  b.out = reinterpret_cast<Tout*>(a.out) + first * a.ld_out;
  b.rows = rows;
  return b;
}

template <typename Tin, typename Tout, int NC>
static int launch_softmax_fit(const SoftmaxArgs& a, int is_log, hipStream_t s) {
  constexpr int kRows = kRowWaves * fit_rows<NC>();
  return launch_row_ranges(a.rows, kRows, 256, [&](int64_t first, int64_t rows) {
    const SoftmaxArgs b = softmax_rows_from<Tin, Tout>(a, first, rows);
    const dim3 grid((unsigned)cdiv(rows, kRows));
    if (is_log)
      hipLaunchKernelGGL((softmax_fit_kernel<Tin, Tout, kLogSoftmax, NC>), grid, dim3(256), 0, s, b);
    else
      hipLaunchKernelGGL((softmax_fit_kernel<Tin, Tout, kSoftmax, NC>), grid, dim3(256), 0, s, b);
    return check_launch("softmax_fit_kernel");
  });
}

template <typename Tin, typename Tout, int T, int NC, bool LOOP = false>
static int launch_softmax_block(const SoftmaxArgs& a, int is_log, hipStream_t s) {
  return launch_row_ranges(a.rows, 1, T, [&](int64_t first, int64_t rows) {
    const SoftmaxArgs b = softmax_rows_from<Tin, Tout>(a, first, rows);
    const dim3 grid((unsigned)rows);
    if (is_log)
      hipLaunchKernelGGL((softmax_block_kernel<Tin, Tout, kLogSoftmax, T, NC, LOOP>), grid, dim3(T), 0, s, b);
    else
      hipLaunchKernelGGL((softmax_block_kernel<Tin, Tout, kSoftmax, T, NC, LOOP>), grid, dim3(T), 0, s, b);
    return check_launch("softmax_block_kernel");
  });
}

template <typename Tin, typename Tout>
static int launch_softmax(const SoftmaxArgs& a, int is_log, hipStream_t s) {
  constexpr int VEC = 16 / (int)sizeof(Tin);
  const int64_t nchunks = cdiv(a.cols, VEC);
  if (nchunks <= 64) return launch_softmax_fit<Tin, Tout, 1>(a, is_log, s);
  if (nchunks <= 128) return launch_softmax_fit<Tin, Tout, 2>(a, is_log, s);
  if (nchunks <= 256) return launch_softmax_fit<Tin, Tout, 4>(a, is_log, s);
  if (nchunks <= 1024) return launch_softmax_block<Tin, Tout, 256, 4>(a, is_log, s);
  if (nchunks <= 4096) return launch_softmax_block<Tin, Tout, 1024, 4>(a, is_log, s);
  if (nchunks <= 8192) return launch_softmax_block<Tin, Tout, 1024, 8>(a, is_log, s);
  if (nchunks <= 16384) return launch_softmax_block<Tin, Tout, 1024, 16>(a, is_log, s);
  return launch_softmax_block<Tin, Tout, 1024, 8, true>(a, is_log, s);
}

// ------------------------------------------------------------------ reductions ----
// Contiguous rows (K == 1).  Rows of up to kWaveRowChunks 16-byte chunks: one wavefront per row
// with the tree described in rowops.h (reduce_rows_fit when the row is whole chunks, else
// reduce_rows_wave; same bits).  Longer rows: one workgroup per row, of 256 threads up to
// kBlock256Chunks chunks and of 1024 beyond.  The choice depends on N only.
constexpr int64_t kWaveRowChunks = 512;
constexpr int64_t kBlock256Chunks = 2048;

struct ReduceArgs {
  const void* in;
  void* out;
  int64_t M, N, K, sM, sN, sK;
  int32_t kvec;  // K > 1: k contiguous and every (m, n) row start 16-byte aligned
};

template <int OP>
__device__ __forceinline__ float reduce_add(float acc, float x) {
  // L2: acc + x * x with one rounding (a fused multiply-add), written out so that the compiler's
  // contraction choices (which product to fuse next to a known-zero accumulator) cannot differ
  // between the kernels below
  return OP == BIOPS_REDUCE_L2 ? __builtin_fmaf(x, x, acc) : acc + x;
}
template <int OP>
__device__ __forceinline__ float reduce_final(float s, int64_t n) {
  return OP == BIOPS_REDUCE_L2 ? sqrtf(s) : s / (float)n;
}

template <typename Tin, typename Tout, int OP>
__global__ __launch_bounds__(256) void reduce_rows_wave(ReduceArgs a) {
  constexpr int VEC = 16 / sizeof(Tin);
  const int64_t r = (int64_t)blockIdx.x * kRowWaves + (threadIdx.x >> 6);
  if (r >= a.M) return;
  const int lane = threadIdx.x & 63;
  const Tin* row = reinterpret_cast<const Tin*>(a.in) + r * a.sM;
  const int64_t nchunks = cdiv(a.N, VEC);
  float acc = 0.f;
  for (int64_t ci = lane; ci < nchunks; ci += 64) {
    float v[VEC];
    load_row_chunk<Tin>(row, a.N, ci * VEC, 0.f, v);
#pragma unroll
    for (int e = 0; e < VEC; ++e)
      if (ci * VEC + e < a.N) acc = reduce_add<OP>(acc, v[e]);
  }
  acc = wave_sum(acc);
  if (lane == 0) Num<Tout>::store(reinterpret_cast<Tout*>(a.out) + r, reduce_final<OP>(acc, a.N));
}

// reduce_rows_wave for rows of whole 16-byte chunks, at most 64 NC of them: the NC loads of a
// lane are issued together, then added in the same order as reduce_rows_wave adds them (chunk
// lane, lane + 64, ..., elements in order), so the bits are the same.  Measured on MI355X
// ([8192, 2048] bf16, inputs streamed from HBM): 9.0 -> 7.4 us per call; two, four or eight rows
// per wavefront, or workgroups of 2 to 16 wavefronts, measured no faster.
template <typename Tin, typename Tout, int OP, int NC>
__global__ __launch_bounds__(256) void reduce_rows_fit(ReduceArgs a) {
  constexpr int VEC = 16 / sizeof(Tin);
  const int64_t r = (int64_t)blockIdx.x * kRowWaves + (threadIdx.x >> 6);
  if (r >= a.M) return;
  const int lane = threadIdx.x & 63;
  const Tin* row = reinterpret_cast<const Tin*>(a.in) + r * a.sM;
  const int nchunks = (int)(a.N / VEC);
  u32x4_t raw[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int ci = lane + 64 * j;
    raw[j] = ci < nchunks ? load_16(row + (int64_t)ci * VEC) : u32x4_t{0u, 0u, 0u, 0u};
  }
  float acc = 0.f;
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    if (lane + 64 * j < nchunks) {
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float x;
        if constexpr (sizeof(Tin) == 4) x = __uint_as_float(raw[j][e]);
        else x = Num<Tin>::from_bits((raw[j][e >> 1] >> (16 * (e & 1))) & 0xffffu);
        acc = reduce_add<OP>(acc, x);
      }
    }
  }
  acc = wave_sum(acc);
  if (lane == 0) Num<Tout>::store(reinterpret_cast<Tout*>(a.out) + r, reduce_final<OP>(acc, a.N));
}

// One workgroup of T threads per row: thread t adds chunks t, t + T, ... in order, kBlockUnroll
// loads in flight, then the wavefronts' butterflies in wavefront order.  A row is one compute
// unit's stream, so what bounds a few long rows is the loads that unit keeps in flight (one
// wavefront per row takes 34.4 us for [2, 50000] fp32, a workgroup 7.7; [512, 65536] bf16 53.5 and
// 11.8 us).
constexpr int kBlockUnroll = 4;

template <typename Tin, typename Tout, int OP, int T>
__global__ __launch_bounds__(T) void reduce_rows_block(ReduceArgs a) {
  constexpr int VEC = 16 / sizeof(Tin);
  constexpr int NW = T / 64;
  __shared__ float part[NW];
  const int64_t r = blockIdx.x;
  const int t = threadIdx.x;
  const Tin* row = reinterpret_cast<const Tin*>(a.in) + r * a.sM;
  const int64_t whole = a.N / VEC;  // chunks inside the row
  float acc = 0.f;
  auto add = [&](const u32x4_t& raw) {
    float v[VEC];
    unpack_chunk<Tin>(raw, v);
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc = reduce_add<OP>(acc, v[e]);
  };
  int64_t ci = t;
  for (; ci + (kBlockUnroll - 1) * T < whole; ci += kBlockUnroll * T) {
    u32x4_t raw[kBlockUnroll];
#pragma unroll
    for (int u = 0; u < kBlockUnroll; ++u) raw[u] = load_16(row + (ci + u * T) * VEC);
#pragma unroll
    for (int u = 0; u < kBlockUnroll; ++u) add(raw[u]);
  }
  for (; ci < whole; ci += T) add(load_16(row + ci * VEC));
  if (ci == whole)  // the thread whose turn the partial chunk is
    for (int64_t n = whole * VEC; n < a.N; ++n) acc = reduce_add<OP>(acc, Num<Tin>::load(row + n));
  const float s = block_sum<NW>(acc, part);
  if (t == 0) Num<Tout>::store(reinterpret_cast<Tout*>(a.out) + r, reduce_final<OP>(s, a.N));
}

// Strided reduction (K > 1): a workgroup owns 64*VK consecutive k of one m (VK consecutive k
// per lane: 16 bytes when the k run is contiguous and aligned, else 1); wavefront w adds the
// elements n = w, w+4, w+8, ... of each of its columns in increasing n, and the four partials
// are added as (p0 + p1) + (p2 + p3).  Depends on N only (VK only decides how columns are
// grouped into loads).  The loads of kUnroll consecutive n of a wavefront are issued before
// their additions, which still happen in increasing n.
constexpr int kStridedUnroll = 8;

template <typename Tin, int VK>
__device__ __forceinline__ void load_k_run(const Tin* p, int64_t sK, int valid, float (&v)[VK]) {
  if constexpr (VK > 1) {
    if (valid >= VK) {
      const u32x4_t raw = *reinterpret_cast<const u32x4_t*>(p);
      if constexpr (sizeof(Tin) == 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __uint_as_float(raw[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = Num<Tin>::from_bits((raw[e >> 1] >> (16 * (e & 1))) & 0xffffu);
      }
      return;
    }
  }
#pragma unroll
  for (int e = 0; e < VK; ++e) v[e] = e < valid ? Num<Tin>::load(p + e * sK) : 0.f;
}

template <typename Tin, typename Tout, int OP, int VK>
__global__ __launch_bounds__(256) void reduce_strided(ReduceArgs a) {
  __shared__ float part[4][64 * VK];
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int64_t kblocks = cdiv(a.K, 64 * VK);
  const int64_t m = blockIdx.x / kblocks;
  const int64_t k0 = (blockIdx.x - m * kblocks) * 64 * VK + (int64_t)lane * VK;
  const int valid = k0 < a.K ? (int)(a.K - k0 < VK ? a.K - k0 : VK) : 0;
  float acc[VK];
#pragma unroll
  for (int e = 0; e < VK; ++e) acc[e] = 0.f;
  // Lanes with a whole k run take a branch-free loop (its loads stay in flight together); the
  // lanes of a partial run (last workgroup of a row only) take the element-wise one.
  auto run = [&](auto whole) {
    constexpr bool WHOLE = decltype(whole)::value;
    const int nv = WHOLE ? VK : valid;
    const Tin* base = reinterpret_cast<const Tin*>(a.in) + m * a.sM + k0 * a.sK;
    int64_t n = w;
    for (; n + 4 * (kStridedUnroll - 1) < a.N; n += 4 * kStridedUnroll) {
      float v[kStridedUnroll][VK];
#pragma unroll
      for (int u = 0; u < kStridedUnroll; ++u) load_k_run<Tin, VK>(base + (n + 4 * u) * a.sN, a.sK, nv, v[u]);
#pragma unroll
      for (int u = 0; u < kStridedUnroll; ++u)
#pragma unroll
        for (int e = 0; e < VK; ++e) acc[e] = reduce_add<OP>(acc[e], v[u][e]);
    }
    for (; n < a.N; n += 4) {
      float v[VK];
      load_k_run<Tin, VK>(base + n * a.sN, a.sK, nv, v);
#pragma unroll
      for (int e = 0; e < VK; ++e) acc[e] = reduce_add<OP>(acc[e], v[e]);
    }
  };
  if (valid == VK) run(std::true_type{});
  else if (valid > 0) run(std::false_type{});
#pragma unroll
  for (int e = 0; e < VK; ++e) part[w][lane * VK + e] = acc[e];
  __syncthreads();
  if (w == 0) {
#pragma unroll
    for (int e = 0; e < VK; ++e) {
      if (e < valid) {
        const int i = lane * VK + e;
        const float s = (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]);
        Num<Tout>::store(reinterpret_cast<Tout*>(a.out) + m * a.K + k0 + e, reduce_final<OP>(s, a.N));
      }
    }
  }
}

template <typename Tin, typename Tout, int OP>
static int launch_reduce_rows(const ReduceArgs& a0, hipStream_t s) {
  constexpr int VEC = 16 / (int)sizeof(Tin);
  const int64_t nc = cdiv(cdiv(a0.N, VEC), 64);  // chunks per lane
  const bool wave = nc <= kWaveRowChunks / 64, narrow = nc <= kBlock256Chunks / 64;
  return launch_row_ranges(a0.M, wave ? kRowWaves : 1, narrow ? 256 : 1024, [&](int64_t first, int64_t rows) {
    ReduceArgs a = a0;
    a.in = reinterpret_cast<const Tin*>(a0.in) + first * a0.sM;
    a.out = reinterpret_cast<Tout*>(a0.out) + first;
    a.M = rows;
    const dim3 grid((unsigned)(wave ? cdiv(rows, kRowWaves) : rows));
    if (wave && a.N % VEC == 0) {
      if (nc <= 1) hipLaunchKernelGGL((reduce_rows_fit<Tin, Tout, OP, 1>), grid, dim3(256), 0, s, a);
      else if (nc <= 2) hipLaunchKernelGGL((reduce_rows_fit<Tin, Tout, OP, 2>), grid, dim3(256), 0, s, a);
      else if (nc <= 4) hipLaunchKernelGGL((reduce_rows_fit<Tin, Tout, OP, 4>), grid, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((reduce_rows_fit<Tin, Tout, OP, 8>), grid, dim3(256), 0, s, a);
    } else if (wave) {
      hipLaunchKernelGGL((reduce_rows_wave<Tin, Tout, OP>), grid, dim3(256), 0, s, a);
    } else if (narrow) {
      hipLaunchKernelGGL((reduce_rows_block<Tin, Tout, OP, 256>), grid, dim3(256), 0, s, a);
    } else {
      hipLaunchKernelGGL((reduce_rows_block<Tin, Tout, OP, 1024>), grid, dim3(1024), 0, s, a);
    }
    return check_launch("reduce");
  });
}

template <typename Tin, typename Tout, int OP>
static int launch_reduce(const ReduceArgs& a, hipStream_t s) {
  if (a.K == 1) {
    return launch_reduce_rows<Tin, Tout, OP>(a, s);
  } else if (a.kvec) {
    constexpr int VK = 16 / (int)sizeof(Tin);
    const int64_t blocks = a.M * cdiv(a.K, 64 * VK);
    if (blocks > 0x7fffffffLL) return fail(BIOPS_ERR_ARG, "reduction too large");
    hipLaunchKernelGGL((reduce_strided<Tin, Tout, OP, VK>), dim3((unsigned)blocks), dim3(256), 0, s, a);
  } else {
    const int64_t blocks = a.M * cdiv(a.K, 64);
    if (blocks > 0x7fffffffLL) return fail(BIOPS_ERR_ARG, "reduction too large");
    hipLaunchKernelGGL((reduce_strided<Tin, Tout, OP, 1>), dim3((unsigned)blocks), dim3(256), 0, s, a);
  }
  return check_launch("reduce");
}

template <typename Tin, typename Tout>
static int launch_reduce_op(int op, const ReduceArgs& a, hipStream_t s) {
  if (op == BIOPS_REDUCE_L2) return launch_reduce<Tin, Tout, BIOPS_REDUCE_L2>(a, s);
  return launch_reduce<Tin, Tout, BIOPS_REDUCE_MEAN>(a, s);
}

}  // namespace biops

using namespace biops;

#define BIOPS_DISPATCH_IN_OUT(din, dout, FN, ...)                                              \
  do {                                                                                        \
    switch ((din) * 3 + (dout)) {                                                              \
      case BIOPS_F32 * 3 + BIOPS_F32: return FN<float, float>(__VA_ARGS__);                   \
      case BIOPS_F32 * 3 + BIOPS_F16: return FN<float, f16_t>(__VA_ARGS__);                   \
      case BIOPS_F32 * 3 + BIOPS_BF16: return FN<float, bf16_t>(__VA_ARGS__);                 \
      case BIOPS_F16 * 3 + BIOPS_F32: return FN<f16_t, float>(__VA_ARGS__);                   \
      case BIOPS_F16 * 3 + BIOPS_F16: return FN<f16_t, f16_t>(__VA_ARGS__);                   \
      case BIOPS_F16 * 3 + BIOPS_BF16: return FN<f16_t, bf16_t>(__VA_ARGS__);                 \
      case BIOPS_BF16 * 3 + BIOPS_F32: return FN<bf16_t, float>(__VA_ARGS__);                 \
      case BIOPS_BF16 * 3 + BIOPS_F16: return FN<bf16_t, f16_t>(__VA_ARGS__);                 \
      case BIOPS_BF16 * 3 + BIOPS_BF16: return FN<bf16_t, bf16_t>(__VA_ARGS__);               \
    }                                                                                         \
  } while (0)

extern "C" int biops_softmax(int dtype_in, int dtype_out, int64_t rows, int64_t cols,
                             const void* in, int64_t ld_in, void* out, int64_t ld_out, int is_log,
                             void* stream) {
  if (!is_float_dtype(dtype_in) || !is_float_dtype(dtype_out))
    return fail(BIOPS_ERR_DTYPE, "unsupported softmax dtype %d -> %d", dtype_in, dtype_out);
  if (rows < 0 || cols < 0) return fail(BIOPS_ERR_ARG, "negative size");
  if (rows == 0 || cols == 0) return BIOPS_OK;
  if (!in || !out) return fail(BIOPS_ERR_ARG, "null pointer");
  SoftmaxArgs a{in, out, rows, cols, ld_in, ld_out};
  BIOPS_DISPATCH_IN_OUT(dtype_in, dtype_out, launch_softmax, a, is_log, (hipStream_t)stream);
  return fail(BIOPS_ERR_DTYPE, "unsupported softmax dtype");
}

extern "C" int biops_reduce(int op, int dtype_in, int dtype_out, int64_t M, int64_t N, int64_t K,
                            const void* in, int64_t sM, int64_t sN, int64_t sK, void* out,
                            void* stream) {
  if (op != BIOPS_REDUCE_MEAN && op != BIOPS_REDUCE_L2) return fail(BIOPS_ERR_ARG, "bad op %d", op);
  if (!is_float_dtype(dtype_in) || !is_float_dtype(dtype_out))
    return fail(BIOPS_ERR_DTYPE, "unsupported reduce dtype %d -> %d", dtype_in, dtype_out);
  if (M < 0 || N < 0 || K < 0) return fail(BIOPS_ERR_ARG, "negative size");
  if (M == 0 || K == 0) return BIOPS_OK;
  if (!in || !out) return fail(BIOPS_ERR_ARG, "null pointer");
  if (K == 1 && sN != 1 && N > 1) return fail(BIOPS_ERR_LAYOUT, "rows must be contiguous when K == 1");
  ReduceArgs a{in, out, M, N, K, sM, sN, sK, 0};
  const int elt = dtype_bytes(dtype_in);
  a.kvec = K > 1 && sK == 1 && (reinterpret_cast<uintptr_t>(in) % 16 == 0) && ((sM * elt) % 16 == 0) &&
           ((sN * elt) % 16 == 0);
  if (M > 0x7fffffffLL) return fail(BIOPS_ERR_ARG, "too many rows");
  if (op == BIOPS_REDUCE_L2) {
    BIOPS_DISPATCH_IN_OUT(dtype_in, dtype_out, launch_reduce_op, BIOPS_REDUCE_L2, a, (hipStream_t)stream);
  } else {
    BIOPS_DISPATCH_IN_OUT(dtype_in, dtype_out, launch_reduce_op, BIOPS_REDUCE_MEAN, a, (hipStream_t)stream);
  }
  return fail(BIOPS_ERR_DTYPE, "unsupported reduce dtype");
}
