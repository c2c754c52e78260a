// Activation preparation for the W4A16 matmul of per-input-feature quantized weights.
//
// The reference's quantize_model (quantize.py:160-181) writes back, for every linear layer
// W [out, in], wq[:, j] = q[:, j] * s_j with ONE scale per input feature j taken over all
// output rows (quantize_col with group_size=None, quantize.py:52-54, through rtn_layer or
// gptq_layer, quantize.py:63-115). The product x @ wq^T = (x * s) @ q^T, so the packed layer
// keeps the int4 codes q^T (in, out) and folds s into the activations:
//   y[m, k] = fp16(x[m, k] * s[k] * mul)        (x fp32, fp16 or bf16; s fp32, optional)
// after which the W4A16 kernels run in their per-tensor mode with tensor_scale = 1 / mul.
// With s absent this is the input cast (fp32 / bf16 -> fp16) of the packed linear layer.
// One pass over x: 8 consecutive k per thread (K % 8 == 0), 16-byte loads where x's rows are
// aligned for them, a 16-byte fp16 store.
//
// With a mailbox the same pass also tells the host whether a finite x became an infinite y
// (pk_w4a16_prep_checked): a workgroup ORs its elements' answers, the last one posts. Bound by
// latency: at M = 8, K = 14336 the pass moves 0.5 MB. Measured on MI355X, whole
// QuantLinear calls on bf16 activations, against the five torch kernels and the synchronising
// copy that the check took before: 8 x 14336 x 4096 87 -> 20.9 us, 333 x 4096 x 6144 with
// per-input scales 91 -> 43 us.
#include "pk_internal.h"

namespace pk {

constexpr int kPrepThreads = 256;
constexpr int kPrepCheckBlocks = 1024;

template <int XD, bool HAS_S, bool CHECK>
__global__ __launch_bounds__(kPrepThreads) void w4a16_prep_kernel(
    const void* __restrict__ x, int64_t ldx, int vec, const float* __restrict__ s, float mul,
    pk_half* __restrict__ y, int64_t ldy, int K, int chunks, int units, Post pt) {
  constexpr int ES = XD == PK_F32 ? 4 : 2;
  bool bad = false;
  for (int u = blockIdx.x; u < units; u += gridDim.x) {  // a unit: 2048 k of one row
    const int m = u / chunks, k0 = ((u - m * chunks) * kPrepThreads + (int)threadIdx.x) * 8;
    if (k0 >= K) continue;
    float v[8];
    if (vec) {
      pk_u4v raw[ES / 2];
      const char* src = reinterpret_cast<const char*>(x) + ((int64_t)m * ldx + k0) * ES;
#pragma unroll
      for (int i = 0; i < ES / 2; ++i) raw[i] = reinterpret_cast<const pk_u4v*>(src)[i];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if constexpr (XD == PK_F32) {
          v[i] = __builtin_bit_cast(float, (uint32_t)raw[i >> 2][i & 3]);
        } else {
          const uint32_t w = raw[0][i >> 1];
          const uint16_t h = (uint16_t)((i & 1) ? w >> 16 : w);
          v[i] = XD == PK_F16 ? (float)__builtin_bit_cast(pk_half, h) : bf16_to_f32(h);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = load_as_f32(x, XD, (int64_t)m * ldx + k0 + i);
    }
    pk_half8 h;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float t = v[i];
      if constexpr (HAS_S) t = t * s[k0 + i];
      h[i] = (pk_half)fp32_value(t * mul);
      if constexpr (CHECK)
        bad |= __builtin_isinf((float)h[i]) && __builtin_isfinite(v[i]);
    }
    *reinterpret_cast<pk_half8*>(y + (int64_t)m * ldy + k0) = h;
  }
  if constexpr (CHECK) {
    bool any = __syncthreads_or(bad) != 0;
    if (threadIdx.x == 0 && post_arrive(pt, &any)) post(pt, any ? 1u : 0u);
  }
}

static int prep_launch(const char* name, const void* x, int x_dtype, int64_t ldx,
                       const float* in_scale, float mul, void* y, int64_t ldy, int M, int K,
                       Post pt, hipStream_t s) {
  PK_REQUIRE(x != nullptr && y != nullptr, "%s: null pointer", name);
  PK_REQUIRE(M >= 1 && K >= 8 && K % 8 == 0, "%s: M=%d K=%d (K %% 8)", name, M, K);
  PK_REQUIRE(x_dtype == PK_F32 || x_dtype == PK_F16 || x_dtype == PK_BF16,
             "%s: input dtype %d", name, x_dtype);
  PK_REQUIRE(ldx >= K && ldy >= K && ldy % 8 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0,
             "%s: output rows must be 16-byte aligned (ldy=%lld)", name, (long long)ldy);
  const int chunks = (int)cdiv(K / 8, kPrepThreads);
  PK_REQUIRE((int64_t)chunks * M < (1ll << 31), "%s: M=%d too large", name, M);
  const int units = chunks * M;
  const int es = x_dtype == PK_F32 ? 4 : 2;
  const int vec = (ldx * es) % 16 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
  // the checked pass: few enough workgroups that their arrivals at one counter stay short
  const unsigned grid = (unsigned)(pt.box != nullptr && units > kPrepCheckBlocks ? kPrepCheckBlocks : units);
  pk_half* yh = reinterpret_cast<pk_half*>(y);
  auto go = [&](auto DT, auto S, auto C) {
    constexpr int xd = decltype(DT)::value;
    constexpr bool hs = decltype(S)::value != 0, ck = decltype(C)::value != 0;
    w4a16_prep_kernel<xd, hs, ck><<<grid, kPrepThreads, 0, s>>>(x, ldx, vec, in_scale, mul, yh, ldy, K,
                                                                chunks, units, pt);
  };
  auto by_form = [&](auto DT) {
    if (pt.box != nullptr) {
      if (in_scale) go(DT, pk_int_c<1>{}, pk_int_c<1>{});
      else go(DT, pk_int_c<0>{}, pk_int_c<1>{});
    } else {
      if (in_scale) go(DT, pk_int_c<1>{}, pk_int_c<0>{});
      else go(DT, pk_int_c<0>{}, pk_int_c<0>{});
    }
  };
  if (x_dtype == PK_F32) by_form(pk_int_c<PK_F32>{});
  else if (x_dtype == PK_F16) by_form(pk_int_c<PK_F16>{});
  else by_form(pk_int_c<PK_BF16>{});
  PK_LAUNCH_CHECK("w4a16 activation prep");
  return PK_OK;
}

}  // namespace pk

using namespace pk;

extern "C" int pk_w4a16_prep_activations(const void* x, int x_dtype, int64_t ldx,
                                         const float* in_scale, float mul, void* y, int64_t ldy,
                                         int M, int K, void* stream) {
  return prep_launch("pk_w4a16_prep_activations", x, x_dtype, ldx, in_scale, mul, y, ldy, M, K,
                     Post{nullptr, nullptr, 0}, (hipStream_t)stream);
}

extern "C" int pk_w4a16_prep_checked(const void* x, int x_dtype, int64_t ldx, const float* in_scale,
                                     float mul, void* y, int64_t ldy, int M, int K, void* counters,
                                     void* mailbox, uint32_t seq, void* stream) {
  PK_REQUIRE(counters != nullptr && mailbox != nullptr, "pk_w4a16_prep_checked: null pointer");
  return prep_launch("pk_w4a16_prep_checked", x, x_dtype, ldx, in_scale, mul, y, ldy, M, K,
                     Post{static_cast<uint64_t*>(mailbox), static_cast<unsigned*>(counters), seq},
                     (hipStream_t)stream);
}
