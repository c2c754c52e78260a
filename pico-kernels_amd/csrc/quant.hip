// Quantization, packing and cast kernels (HBM-bound elementwise / column-group work).
//
// Reference semantics (torch rounding chain) reproduced bit-exactly:
//   gemm_int4.quantize_int4   gemm_int4.py:58-62
//   gemm_int4.pack_int4_n     gemm_int4.py:65-72   (+ the unpack at gemm_int4.py:44-49)
//   quantize.quantize_col     quantize.py:42-60
//   quantize.rtn_layer        quantize.py:63-68
//   gemm_fp8.quantize         gemm_fp8.py:89-95
#include "pk_internal.h"

namespace pk {

constexpr int kThreads = 256;
constexpr int kMaxAbsmaxBlocks = 1024;

static inline dim3 grid_for(int64_t work_items, int per_thread) {
  int64_t b = cdiv(cdiv(work_items, per_thread), kThreads);
  if (b < 1) b = 1;
  if (b > 65535LL * 8) b = 65535LL * 8;
  return dim3((unsigned)b);
}

// ---------------------------------------------------------------------------------------
// absmax. Maxima are taken over |x|'s bit patterns, which order as the values do (NaN above
// infinity, so that a NaN wins as torch's max lets it); max is order-independent, so the result
// is exact and reproducible. Two forms: per-block partial maxima and a second launch that
// folds them (pk_absmax: no workspace to initialise), and one launch whose last workgroup folds
// them and hands the result on (pk_absmax_post).
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t block_max(uint32_t v, uint32_t* red) {
  for (int m = 32; m >= 1; m >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, m, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  v = red[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w) v = max(v, red[w]);
  return v;
}

// The workgroup's maximum as fp32 bits: 16-byte loads, four in flight per thread, over the
// aligned bulk; the rest (and all of a misaligned x) element by element.
template <int DT>
__device__ __forceinline__ uint32_t absmax_block(const void* __restrict__ x, int64_t n, uint32_t* red) {
  constexpr int ES = DT == PK_F32 ? 4 : 2, PER = 16 / ES, U = 4;
  constexpr uint32_t kAbs = DT == PK_F32 ? 0x7fffffffu : 0x7fff7fffu;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t nv = (reinterpret_cast<uintptr_t>(x) & 15) == 0 ? n / PER : 0;
  const pk_u4v* xv = reinterpret_cast<const pk_u4v*>(x);
  pk_u4v m4 = {0u, 0u, 0u, 0u};
  auto take = [&](pk_u4v v) {
    v &= kAbs;
    if constexpr (DT == PK_F32) {
      m4 = __builtin_elementwise_max(m4, v);
    } else {
      typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
      m4 = __builtin_bit_cast(pk_u4v, __builtin_elementwise_max(__builtin_bit_cast(u16x8, m4),
                                                               __builtin_bit_cast(u16x8, v)));
    }
  };
  for (int64_t j = i; j < nv; j += U * stride) {  // past the end the last chunk again
    pk_u4v v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = xv[min(j + u * stride, nv - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u) take(v[u]);
  }
  auto widen = [](uint32_t bits) {  // an element's bits as fp32 bits
    if constexpr (DT == PK_F32) return bits;
    else if constexpr (DT == PK_BF16) return bits << 16;
    else return __builtin_bit_cast(uint32_t, (float)__builtin_bit_cast(pk_half, (uint16_t)bits));
  };
  uint32_t m = 0u;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if constexpr (DT == PK_F32) m = max(m, (uint32_t)m4[w]);
    else m = max(m, max(widen(m4[w] & 0xffffu), widen(m4[w] >> 16)));
  }
  for (int64_t k = nv * PER + i; k < n; k += stride) {
    if constexpr (DT == PK_F32) m = max(m, reinterpret_cast<const uint32_t*>(x)[k] & kAbs);
    else m = max(m, widen(reinterpret_cast<const uint16_t*>(x)[k] & 0x7fffu));
  }
  return block_max(m, red);
}

template <int DT>
__global__ __launch_bounds__(kThreads) void absmax_partial_kernel(const void* __restrict__ x,
                                                                  int64_t n,
                                                                  uint32_t* __restrict__ partial) {
  __shared__ uint32_t red[kThreads / 64];
  const uint32_t m = absmax_block<DT>(x, n, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = m;
}

__global__ __launch_bounds__(kThreads) void absmax_final_kernel(const uint32_t* __restrict__ partial,
                                                                int nparts,
                                                                uint32_t* __restrict__ out) {
  __shared__ uint32_t red[kThreads / 64];
  uint32_t m = 0u;
  for (int i = threadIdx.x; i < nparts; i += blockDim.x) m = max(m, partial[i]);
  m = block_max(m, red);
  if (threadIdx.x == 0) out[0] = m;
}

// One launch: bound by HBM for large x, by two device-scope round trips for small. The partial
// maxima cross XCDs as device-scope stores and loads, acknowledged before the arrival that
// publishes them. out: the result, then one partial per workgroup.
// Measured on MI355X, 1000 x 4096 bf16: 4.8 + 2.9 us and a synchronising copy (two launches) ->
// 7.0 us, read by the host while the cast runs.
template <int DT>
__global__ __launch_bounds__(kThreads) void absmax_post_kernel(const void* __restrict__ x, int64_t n,
                                                               uint32_t* __restrict__ out, Post p) {
  __shared__ uint32_t red[kThreads / 64];
  __shared__ bool last;
  uint32_t m = absmax_block<DT>(x, n, red);
  if (threadIdx.x == 0) {
    __hip_atomic_store(out + 1 + blockIdx.x, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    bool any = false;
    last = post_arrive(p, &any);
  }
  __syncthreads();
  if (!last) return;
  m = 0u;
  for (unsigned i = threadIdx.x; i < gridDim.x; i += kThreads)
    m = max(m, __hip_atomic_load(out + 1 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  m = block_max(m, red);
  if (threadIdx.x == 0) {
    out[0] = m;
    post(p, m);
  }
}

// A thread's four loads make one flight: 16 fp32 or 32 16-bit elements. With 16 of the latter (two
// loads, twice the workgroups to arrive), and the cast's first loads behind its scale, a
// quantize() call on 1000 x 4096 bf16 took 19.9 us, 18.5 so; 333 rows 18.0 -> 17.3.
static int absmax_blocks(int64_t n, int dtype = PK_F32) {
  int64_t b = cdiv(n, (int64_t)kThreads * (dtype == PK_F32 ? 16 : 32));
  if (b < 1) b = 1;
  if (b > kMaxAbsmaxBlocks) b = kMaxAbsmaxBlocks;
  return (int)b;
}

// ---------------------------------------------------------------------------------------
// Per-tensor int4 codes (gemm_int4.py:60-61): q = int8(clamp(round(T(w / s)), -8, 7)).
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void quantize_int4_kernel(const void* __restrict__ w,
                                                                 int dtype, int64_t n,
                                                                 float scale,
                                                                 int8_t* __restrict__ q) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    float v = load_as_f32(w, dtype, i);
    float t = round_to_dtype(v / scale, dtype);  // IEEE fp32 division, then tensor dtype
    float r = clamp_nan(__builtin_rintf(t), -8.0f, 7.0f);
    q[i] = (r == r) ? (int8_t)(int)r : (int8_t)0;
  }
}

// ---------------------------------------------------------------------------------------
// Pack / unpack (gemm_int4.py:65-72, 44-49).
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void pack_int4_kernel(const int8_t* __restrict__ q,
                                                             int64_t rows, int64_t cols,
                                                             int64_t ldq,
                                                             uint8_t* __restrict__ out) {
  const int64_t half = cols / 2, total = rows * half;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    int64_t r = i / half, j = i - r * half;
    const int8_t* row = q + r * ldq;
    uint32_t lo = (uint32_t)(uint8_t)row[2 * j] & 0xfu;
    uint32_t hi = (uint32_t)(uint8_t)row[2 * j + 1] & 0xfu;
    out[i] = (uint8_t)(lo | (hi << 4));
  }
}

__global__ __launch_bounds__(kThreads) void unpack_int4_kernel(const uint8_t* __restrict__ p,
                                                               int64_t rows, int64_t cols,
                                                               int8_t* __restrict__ q) {
  const int64_t half = cols / 2, total = rows * half;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    uint32_t b = p[i];
    int lo = (int)(b & 0xfu), hi = (int)(b >> 4);
    q[2 * i] = (int8_t)(lo >= 8 ? lo - 16 : lo);
    q[2 * i + 1] = (int8_t)(hi >= 8 ? hi - 16 : hi);
  }
}

// ---------------------------------------------------------------------------------------
// Group RTN quantization along K (quantize.py:42-68): per column and group of rows the absmax,
// the scale, then every row's code.
//
// Bound by HBM (the weights in, codes and scales out). A thread owns 8 consecutive columns
// (one word of the packed (K, N/8) layout, one or two 16-byte loads a row) of every RS-th row
// of a group. Groups of at most 128 rows (quantize_group_kernel) are read once: 256 threads
// take 256 columns, a thread's 16 rows stay in registers with all their loads in flight,
// the 8 row sets' maxima meet in LDS, and the codes are made from the registers. Measured on
// MI355X, 4096 x 14336 fp16, group 128: 520 -> 37.7 us, 3.9 TB/s (one thread per 8 columns and group
// before, which read each element by a 2-byte load, twice, in 224 workgroups); 4 or 16 row sets,
// or 64, 128 or 512 columns, in a workgroup run 42-63 us. Longer groups
// (quantize_group_long_kernel; one scale per column is one group of K rows) do not fit the
// registers: 1024 threads take 64 columns, so that few columns still make many workgroups,
// and read the group twice (6144 x 4096 bf16, one scale per column: 31.8 ms -> 87 us).
// ---------------------------------------------------------------------------------------
template <int DT>
struct QgRow {  // 8 columns of one row as loaded
  pk_u4v w[DT == PK_F32 ? 2 : 1];
  __device__ __forceinline__ float at(int c) const {
    if constexpr (DT == PK_F32) return __builtin_bit_cast(float, (uint32_t)w[c >> 2][c & 3]);
    const uint32_t u = w[0][c >> 1];
    const uint16_t h = (uint16_t)((c & 1) ? u >> 16 : u);
    if constexpr (DT == PK_F16) return (float)__builtin_bit_cast(pk_half, h);
    else return bf16_to_f32(h);
  }
};

// Maxima of 8 columns as |v|'s bit patterns, which order as the values do (NaN above infinity, so
// that a NaN wins as torch's max lets it): two 16-bit columns per word, or one fp32 column.
template <int DT>
struct QgMax {
  static constexpr int kWords = DT == PK_F32 ? 8 : 4;
  uint32_t m[kWords];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (auto& x : m) x = 0u;
  }
  __device__ __forceinline__ void take(int i, uint32_t bits) {
    if constexpr (DT == PK_F32) {
      m[i] = max(m[i], bits);
    } else {
      typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
      m[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, m[i]),
                                                                    __builtin_bit_cast(u16x2, bits)));
    }
  }
  __device__ __forceinline__ void take(const QgRow<DT>& r) {
    constexpr uint32_t kAbs = DT == PK_F32 ? 0x7fffffffu : 0x7fff7fffu;
#pragma unroll
    for (int i = 0; i < kWords; ++i) take(i, r.w[i >> 2][i & 3] & kAbs);
  }
  __device__ __forceinline__ float at(int c) const {
    QgRow<DT> r;
#pragma unroll
    for (int i = 0; i < kWords; ++i) r.w[i >> 2][i & 3] = m[i];
    return r.at(c);
  }
};

struct QgParams {
  const void* w;
  int64_t K, N, ldw;
  int qmax, group, half_math;
  uint32_t* qweight;
  void* scales;
  int scale_dtype;
  void* fake;
  int fake_dtype;
  int fake_vec;  // fake's 8 columns of a thread may be stored together
};

// Row k's 8 columns from n0; VEC: rows of whole, 16-byte aligned chunks. Columns past N read 0.
// ONCE: the row is read once (but for the rare row that is emitted again).
template <int DT, bool VEC, bool ONCE>
__device__ __forceinline__ QgRow<DT> qg_load(const QgParams& p, int64_t k, int64_t n0) {
  constexpr int ES = DT == PK_F32 ? 4 : 2;
  QgRow<DT> r;
  const char* src = reinterpret_cast<const char*>(p.w) + (k * p.ldw + n0) * ES;
  if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < ES / 2; ++i)
      r.w[i] = ONCE ? __builtin_nontemporal_load(reinterpret_cast<const pk_u4v*>(src) + i)
                    : reinterpret_cast<const pk_u4v*>(src)[i];
  } else {
    uint32_t u[2 * ES];
#pragma unroll
    for (int i = 0; i < 2 * ES; ++i) u[i] = 0u;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (n0 + c >= p.N) continue;
      if constexpr (DT == PK_F32) u[c] = reinterpret_cast<const uint32_t*>(src)[c];
      else u[c >> 1] |= (uint32_t)reinterpret_cast<const uint16_t*>(src)[c] << (16 * (c & 1));
    }
#pragma unroll
    for (int i = 0; i < ES / 2; ++i) r.w[i] = pk_u4v{u[4 * i], u[4 * i + 1], u[4 * i + 2], u[4 * i + 3]};
  }
  return r;
}

// The group's scales s[c] (stored by the threads with `store`) and what the codes need.
struct QgScale {
  float s[8], inv[8];
  bool divide;  // take the true quotient of every element
};
template <int DT>
__device__ __forceinline__ QgScale qg_scale(const QgParams& p, const QgMax<DT>& m, int mdt,
                                            int64_t g, int64_t n0, bool store) {
  // In fp16/bf16 tensor math the 1e-12 floor is itself rounded to the tensor dtype
  // (it underflows to 0 in fp16).
  const float floor_v = round_to_dtype(1e-12f, mdt);
  QgScale q;
  q.divide = p.half_math != 0;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float amax = m.at(c);
    const float a = amax < floor_v ? floor_v : amax;  // clamp_min, NaN passes through
    q.s[c] = round_to_dtype(a / (float)p.qmax, mdt);
    q.inv[c] = 1.0f / q.s[c];
    q.divide |= !(q.s[c] > 0x1p-100f && q.s[c] < 0x1p100f);  // 1 / s stays a normal number
    if (store && p.scales != nullptr && n0 + c < p.N)
      store_from_f32(p.scales, p.scale_dtype, g * p.N + n0 + c, q.s[c]);
  }
  return q;
}

// One row's codes (and fake-quantized values). The code is rint(fl(v / s)). With t = fl(v * fl(1 / s)),
// |t - fl(v / s)| < |t| 2^-22, so rint(t) is the same unless t is that close to a half-integer;
// only then (and for scales whose reciprocal is not a normal number, and in 16-bit tensor math,
// where the quotient is rounded to the dtype first) the division has to be carried out: returns
// whether this row needs that, for the caller to load it again and emit it with DIVIDE (a rare
// second pass over single rows, so that the division's code stands once and not beside every
// row's). No value is stored before: values may be written over the weights. (Codes are: to leave
// their store out costs the packing 1%, 4096 x 14336 37.7 -> 38.1 us.)
// Without it |v / s| is at most qmax (1 + 2^-23), so no code needs clamping, and none is NaN.
template <int DT, bool FAKE, bool DIVIDE>
__device__ __forceinline__ bool qg_emit(const QgParams& p, const QgRow<DT>& row, const QgScale& q,
                                        int mdt, int64_t k, int64_t n0) {
#pragma clang fp contract(off)  // every product and quotient rounded by itself
  float r[8];
  float near = 0.0f;
  uint32_t word = 0;
  if constexpr (DIVIDE) {
    const float fq = (float)p.qmax;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      r[c] = clamp_nan(__builtin_rintf(round_to_dtype(row.at(c) / q.s[c], mdt)), -fq, fq);
      word |= ((r[c] == r[c]) ? (uint32_t)(int)r[c] & 0xfu : 0u) << (4 * c);
    }
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float t = row.at(c) * q.inv[c];
      r[c] = __builtin_rintf(t);
      near = __builtin_fmaxf(near, __builtin_fmaf(__builtin_fabsf(t), 0x1p-21f, __builtin_fabsf(t - r[c])));
      word |= ((uint32_t)(int)r[c] & 0xfu) << (4 * c);
    }
  }
  const bool redo = !DIVIDE && (q.divide || near > 0.5f);
  if (FAKE && redo) return true;
  if (p.qweight != nullptr) p.qweight[k * (p.N / 8) + (n0 >> 3)] = word;
  if constexpr (FAKE) {
    float f[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) f[c] = round_to_dtype(fp32_value(r[c] * q.s[c]), mdt);
    if (p.fake_dtype == PK_F32) {
      float* o = reinterpret_cast<float*>(p.fake) + k * p.N + n0;
      if (p.fake_vec) {
        *reinterpret_cast<pk_f4*>(o) = pk_f4{f[0], f[1], f[2], f[3]};
        *reinterpret_cast<pk_f4*>(o + 4) = pk_f4{f[4], f[5], f[6], f[7]};
      } else {
#pragma unroll
        for (int c = 0; c < 8; ++c)
          if (n0 + c < p.N) o[c] = f[c];
      }
    } else {
      uint16_t h[8];
      if (p.fake_dtype == PK_F16) {
#pragma unroll
        for (int c = 0; c < 8; ++c) h[c] = __builtin_bit_cast(uint16_t, (pk_half)f[c]);
      } else {
#pragma unroll
        for (int c = 0; c < 8; ++c) h[c] = f32_to_bf16_rne(f[c]);
      }
      uint16_t* o = reinterpret_cast<uint16_t*>(p.fake) + k * p.N + n0;
      if (p.fake_vec) {
        *reinterpret_cast<pk_u4v*>(o) =
            pk_u4v{h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16),
                   h[4] | ((uint32_t)h[5] << 16), h[6] | ((uint32_t)h[7] << 16)};
      } else {
#pragma unroll
        for (int c = 0; c < 8; ++c)
          if (n0 + c < p.N) o[c] = h[c];
      }
    }
  }
  return redo;
}

constexpr int kQgRows = 128;  // rows of a group the register kernel holds
constexpr int kQgSets = 8;    // its row sets
constexpr int kQgLanes = 32;  // threads along a row, 8 columns each
constexpr int kQgThreads = kQgLanes * kQgSets;

template <int DT, bool VEC, bool FAKE>
__global__ __launch_bounds__(kQgThreads) void quantize_group_kernel(QgParams p) {
  constexpr int PER = kQgRows / kQgSets;
  constexpr int W = QgMax<DT>::kWords;
  __shared__ uint32_t red[kQgSets][kQgLanes * W];
  const int t = threadIdx.x, set = t / kQgLanes, cl = t % kQgLanes;
  const int64_t tiles = cdiv(p.N, 8 * kQgLanes), items = tiles * cdiv(p.K, p.group);
  const int mdt = p.half_math ? DT : PK_F32;
  for (int64_t b = blockIdx.x; b < items; b += gridDim.x) {
    const int64_t g = b / tiles, n0 = ((b - g * tiles) * kQgLanes + cl) * 8, k0 = g * p.group;
    const int rows = (int)min((int64_t)p.group, p.K - k0);
    const bool cols = n0 < p.N;
    QgRow<DT> v[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int r = i * kQgSets + set;
      if (cols && r < rows) {
        v[i] = qg_load<DT, VEC, true>(p, k0 + r, n0);
      } else {
#pragma unroll
        for (auto& w : v[i].w) w = pk_u4v{0u, 0u, 0u, 0u};
      }
    }
    QgMax<DT> m;
    m.clear();
#pragma unroll
    for (int i = 0; i < PER; ++i) m.take(v[i]);
#pragma unroll
    for (int i = 0; i < W; ++i) red[set][W * cl + i] = m.m[i];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kQgSets; ++u)
#pragma unroll
      for (int i = 0; i < W; ++i) m.take(i, red[u][W * cl + i]);
    const QgScale q = qg_scale(p, m, mdt, g, n0, set == 0);
    uint32_t redo = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int r = i * kQgSets + set;
      if (cols && r < rows && qg_emit<DT, FAKE, false>(p, v[i], q, mdt, k0 + r, n0)) redo |= 1u << i;
    }
    for (; redo != 0; redo &= redo - 1) {
      const int64_t k = k0 + (__builtin_ctz(redo) * kQgSets + set);
      qg_emit<DT, FAKE, true>(p, qg_load<DT, VEC, false>(p, k, n0), q, mdt, k, n0);
    }
    __syncthreads();  // red is read before the next item writes it
  }
}

constexpr int kQgLongThreads = 1024;
constexpr int kQgLongSets = kQgLongThreads / 8;  // 64 columns per workgroup

template <int DT, bool VEC, bool FAKE>
__global__ __launch_bounds__(kQgLongThreads) void quantize_group_long_kernel(QgParams p) {
  constexpr int W = QgMax<DT>::kWords;
  __shared__ uint32_t red[kQgLongThreads / 64][8 * W];
  const int t = threadIdx.x, set = t >> 3, lane = t & 63;
  const int64_t tiles = cdiv(p.N, 64), items = tiles * cdiv(p.K, p.group);
  const int mdt = p.half_math ? DT : PK_F32;
  constexpr int U = 4;  // rows in flight per thread
  for (int64_t b = blockIdx.x; b < items; b += gridDim.x) {
    const int64_t g = b / tiles, n0 = (b - g * tiles) * 64 + 8 * (t & 7);
    const int64_t k0 = g * p.group, k1 = min(k0 + p.group, p.K);
    const bool cols = n0 < p.N;
    QgMax<DT> m;
    m.clear();
    for (int64_t k = k0 + set; cols && k < k1; k += U * kQgLongSets) {
      QgRow<DT> v[U];
#pragma unroll
      for (int u = 0; u < U; ++u)  // past the group: the last row again
        v[u] = qg_load<DT, VEC, false>(p, min(k + u * kQgLongSets, k1 - 1), n0);
#pragma unroll
      for (int u = 0; u < U; ++u) m.take(v[u]);
    }
#pragma unroll
    for (int i = 0; i < W; ++i) {
      for (int x = 8; x < 64; x <<= 1) m.take(i, (uint32_t)__shfl_xor((int)m.m[i], x, 64));
      if (lane < 8) red[t >> 6][W * lane + i] = m.m[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < W; ++i)
      for (int u = 0; u < kQgLongThreads / 64; ++u) m.take(i, red[u][W * (t & 7) + i]);
    const QgScale q = qg_scale(p, m, mdt, g, n0, set == 0);
    for (int64_t k = k0 + set; cols && k < k1; k += U * kQgLongSets) {
      QgRow<DT> v[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        v[u] = qg_load<DT, VEC, false>(p, min(k + u * kQgLongSets, k1 - 1), n0);
      uint32_t redo = 0;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (k + u * kQgLongSets < k1 &&
            qg_emit<DT, FAKE, false>(p, v[u], q, mdt, k + u * kQgLongSets, n0))
          redo |= 1u << u;
      for (; redo != 0; redo &= redo - 1) {
        const int64_t kr = k + __builtin_ctz(redo) * kQgLongSets;
        qg_emit<DT, FAKE, true>(p, qg_load<DT, VEC, false>(p, kr, n0), q, mdt, kr, n0);
      }
    }
    __syncthreads();  // red is read before the next item writes it
  }
}

// ---------------------------------------------------------------------------------------
// Scaled e4m3 cast (gemm_fp8.py:95): out = e4m3(T(x * scale)), the scale given by value or as
// 448 / max|x| of a maximum still on its way in device memory (the division in fp64, as the
// Python expression's, then narrowed). Bound by HBM: 16 elements per thread, 16-byte loads and
// stores (the rest, and misaligned operands, element by element). Measured on MI355X, 1000 x 4096 bf16: 8.0 ->
// 5.6 us; 4096 x 6144 bf16 33 -> 18.9 us (2-byte loads and branches before).
// ---------------------------------------------------------------------------------------
// OCP FP8 E4M3 ("e4m3fn": no infinities, S.1111.111 is NaN, max finite 448), round to nearest even,
// not saturating: what rounds above 448 (anything above 464, the tie with the missing 480), Inf
// and NaN become NaN (0x7f | sign). From the format's definition, without branches:
//   normal:    (-1)^s * 2^(e-7) * (1 + m/8), e in 1..15 (e = 15, m = 7 reserved for NaN): half an ulp
//              less one plus the kept lowest bit added, then truncated; a carry out of the
//              mantissa raises the exponent
//   subnormal: (-1)^s * 2^-6 * (m/8): whole multiples of 2^-9 (8 of them the smallest normal)
__device__ __forceinline__ uint32_t e4m3_select(float f) {
  const uint32_t u = __builtin_bit_cast(uint32_t, f), a = u & 0x7fffffffu;
  const uint32_t sub = (uint32_t)__builtin_rintf(__builtin_bit_cast(float, a) * 512.0f);
  const uint32_t norm = ((a + 0x7ffffu + ((a >> 20) & 1u)) >> 20) - ((127u - 7u) << 3);
  const uint32_t c = a < 0x3c800000u ? sub : norm;
  return (a > 0x43e80000u ? 0x7fu : c) | ((u >> 24) & 0x80u);
}

template <int DT>
__global__ __launch_bounds__(kThreads) void cast_e4m3_kernel(const void* __restrict__ x, int64_t n,
                                                             float scale,
                                                             const float* __restrict__ absmax,
                                                             uint8_t* __restrict__ out) {
  constexpr int ES = DT == PK_F32 ? 4 : 2;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const bool vec = ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(x)) & 15) == 0;
  const int64_t nv = vec ? n / 16 : 0;
  pk_u4v v[ES];  // a chunk ahead; the first is on its way while the scale is made
  auto load = [&](int64_t j) {
#pragma unroll
    for (int u = 0; u < ES; ++u) v[u] = reinterpret_cast<const pk_u4v*>(x)[j * ES + u];
  };
  if (i < nv) load(i);
  if (absmax != nullptr) scale = (float)(448.0 / (double)absmax[0]);
  for (int64_t j = i; j < nv; j += stride) {
    pk_u4v o;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      uint32_t word = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = 4 * w + e;
        float f;
        if constexpr (DT == PK_F32) {
          f = __builtin_bit_cast(float, (uint32_t)v[k >> 2][k & 3]);
        } else {
          const uint32_t d = v[k >> 3][(k & 7) >> 1];
          const uint16_t h = (uint16_t)((k & 1) ? d >> 16 : d);
          f = DT == PK_F16 ? (float)__builtin_bit_cast(pk_half, h) : bf16_to_f32(h);
        }
        word |= e4m3_select(round_to_dtype(fp32_value(f * scale), DT)) << (8 * e);
      }
      o[w] = word;
    }
    reinterpret_cast<pk_u4v*>(out)[j] = o;
    if (j + stride < nv) load(j + stride);
  }
  for (int64_t k = nv * 16 + i; k < n; k += stride)
    out[k] = (uint8_t)e4m3_select(round_to_dtype(fp32_value(load_as_f32(x, DT, k) * scale), DT));
}

static bool float_dtype(int d) { return d == PK_F32 || d == PK_F16 || d == PK_BF16; }

template <typename F>
static void by_dtype(int dtype, F f) {  // f with the (checked) dtype as a constant
  if (dtype == PK_F32) f(pk_int_c<PK_F32>{});
  else if (dtype == PK_F16) f(pk_int_c<PK_F16>{});
  else f(pk_int_c<PK_BF16>{});
}

static void cast_launch(const void* x, int dtype, int64_t n, float scale, const float* absmax,
                        uint8_t* out, hipStream_t s) {
  by_dtype(dtype, [&](auto D) {
    cast_e4m3_kernel<decltype(D)::value><<<grid_for(n, 16), kThreads, 0, s>>>(x, n, scale, absmax, out);
  });
}

}  // namespace pk

using namespace pk;

extern "C" size_t pk_absmax_workspace_bytes(int64_t n) {
  return (size_t)absmax_blocks(n < 1 ? 1 : n) * sizeof(float);
}

extern "C" int pk_absmax(const void* x, int x_dtype, int64_t n, float* out_dev, void* workspace,
                         size_t workspace_bytes, void* stream) {
  PK_REQUIRE(x != nullptr && out_dev != nullptr, "pk_absmax: null pointer");
  PK_REQUIRE(float_dtype(x_dtype), "pk_absmax: unsupported dtype %d", x_dtype);
  PK_REQUIRE(n >= 1, "pk_absmax: empty input (max of an empty tensor is undefined)");
  int blocks = absmax_blocks(n, x_dtype);
  if (workspace == nullptr || workspace_bytes < (size_t)blocks * sizeof(float)) {
    set_error("pk_absmax: workspace of %zu bytes needed", (size_t)blocks * sizeof(float));
    return PK_EWORKSPACE;
  }
  hipStream_t s = (hipStream_t)stream;
  uint32_t* partial = reinterpret_cast<uint32_t*>(workspace);
  by_dtype(x_dtype, [&](auto D) {
    absmax_partial_kernel<decltype(D)::value><<<blocks, kThreads, 0, s>>>(x, n, partial);
  });
  absmax_final_kernel<<<1, kThreads, 0, s>>>(partial, blocks, reinterpret_cast<uint32_t*>(out_dev));
  PK_LAUNCH_CHECK("pk_absmax");
  return PK_OK;
}

extern "C" int pk_absmax_post(const void* x, int x_dtype, int64_t n, float* out_dev, void* counters,
                              void* mailbox, uint32_t seq, void* stream) {
  PK_REQUIRE(x != nullptr && out_dev != nullptr && counters != nullptr && mailbox != nullptr,
             "pk_absmax_post: null pointer");
  PK_REQUIRE(float_dtype(x_dtype), "pk_absmax_post: unsupported dtype %d", x_dtype);
  PK_REQUIRE(n >= 1, "pk_absmax_post: empty input (max of an empty tensor is undefined)");
  const Post p{static_cast<uint64_t*>(mailbox), static_cast<unsigned*>(counters), seq};
  const unsigned blocks = (unsigned)absmax_blocks(n, x_dtype);
  by_dtype(x_dtype, [&](auto D) {
    absmax_post_kernel<decltype(D)::value><<<blocks, kThreads, 0, (hipStream_t)stream>>>(
        x, n, reinterpret_cast<uint32_t*>(out_dev), p);
  });
  PK_LAUNCH_CHECK("pk_absmax_post");
  return PK_OK;
}

extern "C" int pk_quantize_int4(const void* w, int w_dtype, int64_t n, float scale, int8_t* q,
                                void* stream) {
  PK_REQUIRE(w != nullptr && q != nullptr, "pk_quantize_int4: null pointer");
  PK_REQUIRE(float_dtype(w_dtype), "pk_quantize_int4: unsupported dtype %d", w_dtype);
  if (n <= 0) return PK_OK;
  quantize_int4_kernel<<<grid_for(n, 4), kThreads, 0, (hipStream_t)stream>>>(w, w_dtype, n,
                                                                              scale, q);
  PK_LAUNCH_CHECK("pk_quantize_int4");
  return PK_OK;
}

extern "C" int pk_pack_int4(const int8_t* q, int64_t rows, int64_t cols, int64_t ldq,
                            uint8_t* packed, void* stream) {
  PK_REQUIRE(q != nullptr && packed != nullptr, "pk_pack_int4: null pointer");
  PK_REQUIRE(rows >= 0 && cols >= 0 && cols % 2 == 0, "pk_pack_int4: N must be even");
  PK_REQUIRE(ldq >= cols, "pk_pack_int4: ldq < cols");
  if (rows * cols == 0) return PK_OK;
  pack_int4_kernel<<<grid_for(rows * cols / 2, 4), kThreads, 0, (hipStream_t)stream>>>(
      q, rows, cols, ldq, packed);
  PK_LAUNCH_CHECK("pk_pack_int4");
  return PK_OK;
}

extern "C" int pk_unpack_int4(const uint8_t* packed, int64_t rows, int64_t cols, int8_t* q,
                              void* stream) {
  PK_REQUIRE(q != nullptr && packed != nullptr, "pk_unpack_int4: null pointer");
  PK_REQUIRE(rows >= 0 && cols >= 0 && cols % 2 == 0, "pk_unpack_int4: N must be even");
  if (rows * cols == 0) return PK_OK;
  unpack_int4_kernel<<<grid_for(rows * cols / 2, 4), kThreads, 0, (hipStream_t)stream>>>(
      packed, rows, cols, q);
  PK_LAUNCH_CHECK("pk_unpack_int4");
  return PK_OK;
}

extern "C" int pk_quantize_group(const void* w, int w_dtype, int64_t K, int64_t N, int64_t ldw,
                                 int bits, int group_size, int half_math, uint32_t* qweight,
                                 void* scales, int scale_dtype, void* fake, int fake_dtype,
                                 void* stream) {
  PK_REQUIRE(w != nullptr, "pk_quantize_group: null weight");
  PK_REQUIRE(float_dtype(w_dtype), "pk_quantize_group: unsupported dtype %d", w_dtype);
  PK_REQUIRE(K >= 0 && N >= 0 && ldw >= N, "pk_quantize_group: bad shape");
  PK_REQUIRE(bits >= 2 && bits <= 15, "pk_quantize_group: bits must be in [2, 15]");
  PK_REQUIRE(!half_math || w_dtype != PK_F32, "pk_quantize_group: half_math needs fp16/bf16");
  PK_REQUIRE(qweight == nullptr || (bits == 4 && N % 8 == 0),
             "pk_quantize_group: packed output needs bits == 4 and N % 8 == 0");
  PK_REQUIRE(scales == nullptr || float_dtype(scale_dtype), "pk_quantize_group: scale dtype");
  PK_REQUIRE(fake == nullptr || float_dtype(fake_dtype), "pk_quantize_group: fake dtype");
  if (K == 0 || N == 0) return PK_OK;
  const int group = group_size > 0 ? group_size : (int)K;
  const int qmax = (1 << (bits - 1)) - 1;
  hipStream_t s = (hipStream_t)stream;
  const int64_t groups = cdiv(K, group);
  const int es = w_dtype == PK_F32 ? 4 : 2;
  const bool vec = N % 8 == 0 && (ldw * es) % 16 == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0;
  const bool fake_vec = N % 8 == 0 && (reinterpret_cast<uintptr_t>(fake) & 15) == 0;
  const QgParams p{w, K, N, ldw, qmax, group, half_math, qweight, scales, scale_dtype, fake,
                   fake_dtype, fake_vec};
  const bool longer = group > kQgRows;
  const int64_t items = cdiv(N, longer ? 64 : 8 * kQgLanes) * groups;
  const unsigned grid = (unsigned)(items < (1 << 20) ? items : (1 << 20));  // the kernels loop
  auto go = [&](auto DT, auto V) {
    constexpr int dt = decltype(DT)::value;
    constexpr bool v = decltype(V)::value != 0;
    if (longer && fake) quantize_group_long_kernel<dt, v, true><<<grid, kQgLongThreads, 0, s>>>(p);
    else if (longer) quantize_group_long_kernel<dt, v, false><<<grid, kQgLongThreads, 0, s>>>(p);
    else if (fake) quantize_group_kernel<dt, v, true><<<grid, kQgThreads, 0, s>>>(p);
    else quantize_group_kernel<dt, v, false><<<grid, kQgThreads, 0, s>>>(p);
  };
  auto by_vec = [&](auto DT) {
    if (vec) go(DT, pk_int_c<1>{});
    else go(DT, pk_int_c<0>{});
  };
  by_dtype(w_dtype, by_vec);
  PK_LAUNCH_CHECK("pk_quantize_group");
  return PK_OK;
}

extern "C" int pk_cast_e4m3(const void* x, int x_dtype, int64_t n, float scale, uint8_t* out,
                            void* stream) {
  PK_REQUIRE(x != nullptr && out != nullptr, "pk_cast_e4m3: null pointer");
  PK_REQUIRE(float_dtype(x_dtype), "pk_cast_e4m3: unsupported dtype %d", x_dtype);
  if (n <= 0) return PK_OK;
  cast_launch(x, x_dtype, n, scale, nullptr, out, (hipStream_t)stream);
  PK_LAUNCH_CHECK("pk_cast_e4m3");
  return PK_OK;
}

extern "C" int pk_cast_e4m3_absmax(const void* x, int x_dtype, int64_t n, const float* absmax_dev,
                                   uint8_t* out, void* stream) {
  PK_REQUIRE(x != nullptr && out != nullptr && absmax_dev != nullptr,
             "pk_cast_e4m3_absmax: null pointer");
  PK_REQUIRE(float_dtype(x_dtype), "pk_cast_e4m3_absmax: unsupported dtype %d", x_dtype);
  if (n <= 0) return PK_OK;
  cast_launch(x, x_dtype, n, 0.0f, absmax_dev, out, (hipStream_t)stream);
  PK_LAUNCH_CHECK("pk_cast_e4m3_absmax");
  return PK_OK;
}
