// Dense fp16 / bf16 GEMM with a row-major (K, N) B on gfx950 (gemm.triton_gemm, gemm.py:103-128;
// gemm_splitk.triton_gemm_splitk, gemm_splitk.py:26-80): C = A @ B, fp32 accumulate.
//
// Bound by the matrix cores for large shapes. The kernel it replaces there (gemm_v3_f16_kernel's
// dense forms: 64 x 64 per wave, B transposed on its way through registers into LDS) asked LDS
// for 128 bytes per clock at full matrix rate, beside the B tile's ds_writes, byte permutes
// and registers. Here nothing passes through registers on its way in, and a wave's block is
// 128 x 64:
//  * BM x 256 workgroup tiles (BM = 128, or 64 where that takes less time: dense_tr_rows), k-tiles
//    of 32, eight waves. Wave w owns columns 64 (w % 4) .. +63 of all the tile's rows and the k half
//    h = w / 4 of every k-tile: waves w and w + 4 share a SIMD, compute the same block over
//    different k and add their accumulators once, at the end. LDS serves 96 bytes per clock at
//    full matrix rate. v_mfma_f32_32x32x16 with B as the first operand, so that a lane holds four
//    consecutive output columns per register quad.
//  * A and B go global -> LDS by buffer DMA through six stages of 24 KB: one being multiplied, one
//    being read, four on their way, which the DMA's latency needs (three stages of 64-deep
//    k-tiles, two of 48 KB on their way, ran 2048 x 4096 x 4096 in 70 us against 63.6). A rows are
//    64 bytes (32 k), 16-byte chunk c of row r in slot c ^ ((r >> 2) & 3). B rows are the 512 bytes
//    of 256 columns at one k, chunk c of row r in slot c ^ 4 (r % 4 + 4 ((r >> 3) & 1)): the eight
//    k-rows that one transposing read touches lie in eight different 64-byte windows.
//  * B leaves LDS through ds_read_b64_tr_b16: the 16 lanes of a group address a 4 (k) x 16
//    (columns) block, lane q the 8 bytes of columns 4 (q % 4) .. +3 at k-row q / 4, and lane q
//    receives column q's four k values. For a 32 x 32 x 16 step group g holds columns 16 (g % 2) + q
//    at k 8 (g / 2) .. +7: two reads.
//  * Per k-tile one barrier, before which every wave has waited for its own DMA of tile t + 1 and
//    finished with tile t - 1: behind it the DMA of tile t + 5 goes into tile t - 1's stage and tile
//    t + 1's operands are read while tile t's products run.
// Measured on MI355X, fp32 output, bf16 (before in gemm_v3_f16_kernel -> here): 2048 x 4096 x 4096
// 81.6 -> 63.6 us (1081 TFLOP/s), 4096^3 146 -> 120, 8192^3 1140 -> 982, 1024 x 4096 x 4096 63 -> 43,
// 1024 x 1024 x 4096 55 -> 37, 256 x 256 x 1408 23 -> 12; split 4 of 512 x 512 x 8192 34 -> 25.
#include "pk_internal.h"

namespace pk {

struct DenseTrParams {
  const void* a;
  int64_t lda;  // elements
  const void* b;
  int64_t ldb;  // elements
  void* c;
  int c_dtype;
  int64_t ldc;
  int M, K;
  int tiles_m, tiles_n;
  int kt_slice;     // k-tiles per split-K slice
  int64_t c_slice;  // elements between the slices' outputs (fp32 partial planes)
};

typedef short dt_s4 __attribute__((ext_vector_type(4)));
typedef short dt_s8 __attribute__((ext_vector_type(8)));
#define PK_DT_LDS(T, p) ((__attribute__((address_space(3))) T*)(p))

__device__ __forceinline__ void dt_dma16(__amdgpu_buffer_rsrc_t r, char* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, PK_DT_LDS(void, lds), 16, voff, soff, 0, 0);
}
__device__ __forceinline__ dt_s4 dt_read_tr(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(PK_DT_LDS(dt_s4, const_cast<char*>(p)));
}

// XCD-aware tile order: consecutive logical tiles on one XCD, walked 4 tile rows deep.
__device__ __forceinline__ void dt_tile_of(int bid, int tiles_m, int tiles_n, int* tm, int* tn) {
  const int total = tiles_m * tiles_n;
  int logical = bid;
  if (total % 8 == 0) logical = (bid % 8) * (total / 8) + bid / 8;
  constexpr int GROUP_M = 4;
  const int per_group = GROUP_M * tiles_n;
  const int g = logical / per_group;
  const int first_m = g * GROUP_M;
  const int gm = min(tiles_m - first_m, GROUP_M);
  const int in_g = logical - g * per_group;
  *tm = first_m + in_g % gm;
  *tn = in_g / gm;
}

template <bool BF16, int BM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_dense_tr_kernel(DenseTrParams p) {
  constexpr int BN = 256, WN = 64, FM = BM / 32, FN = 2;
  constexpr int B_DMA = 2, VPT = 1 + B_DMA;  // 1 KB instructions per wave and k-tile
  __shared__ __align__(16) char sA0[BM * 64];
  __shared__ __align__(16) char sB0[32 * 512];
  __shared__ __align__(16) char sA1[BM * 64];
  __shared__ __align__(16) char sB1[32 * 512];
  __shared__ __align__(16) char sA2[BM * 64];
  __shared__ __align__(16) char sB2[32 * 512];
  __shared__ __align__(16) char sA3[BM * 64];
  __shared__ __align__(16) char sB3[32 * 512];
  __shared__ __align__(16) char sA4[BM * 64];
  __shared__ __align__(16) char sB4[32 * 512];
  __shared__ __align__(16) char sA5[BM * 64];
  __shared__ __align__(16) char sB5[32 * 512];

  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int h = wave >> 2, wn0 = (wave & 3) * WN;
  int tm, tn;
  dt_tile_of(blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int kt0 = blockIdx.y * p.kt_slice, ktiles = p.kt_slice, last = ktiles - 1;

  const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.a, (uint32_t)((int64_t)p.M * p.lda * 2));
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(p.b, (uint32_t)((int64_t)p.K * p.ldb * 2));
  // A: rows 16 aw .. +15 (with 64 rows waves 4-7 write the bytes of waves 0-3 again, so that every
  // wave issues the same loads)
  const int aw = BM == 128 ? wave : wave & 3, ar = 16 * aw + (lane >> 2);
  const int a_off = (int)((int64_t)min(m0 + ar, p.M - 1) * p.lda * 2) + (((lane & 3) ^ ((ar >> 2) & 3)) << 4);
  int b_off[B_DMA];
#pragma unroll
  for (int i = 0; i < B_DMA; ++i) {  // k-rows 2 (2 w + i), +1
    const int r = 2 * (B_DMA * wave + i) + (lane >> 5);
    b_off[i] = (int)(r * p.ldb * 2) + n0 * 2 + (((lane & 31) ^ (((r & 3) | ((r >> 3) & 1) << 2) << 2)) << 4);
  }
  auto issue = [&](int kt, char* sA, char* sB) {
    const int k0 = (kt0 + kt) * 32;
    dt_dma16(ra, sA + aw * 1024, a_off, k0 * 2);
    const int bk = (int)(k0 * p.ldb * 2);
#pragma unroll
    for (int i = 0; i < B_DMA; ++i) dt_dma16(rb, sB + (B_DMA * wave + i) * 1024, b_off[i], bk);
  };

  const int l32 = lane & 31, lh = lane >> 5, g = lane >> 4, q = lane & 15;
  // A: row l32 (+ 32 i), chunk 2 h + lh
  const int aoff = l32 * 64 + (((2 * h + lh) ^ ((l32 >> 2) & 3)) << 4);
  int boff[FN];  // k-row 16 h + 8 (g / 2) + q / 4 (+ 4 r2)
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int row = 16 * h + 8 * (g >> 1) + (q >> 2);
    const int col = wn0 + 32 * j + 16 * (g & 1) + 4 * (q & 3);
    const int slot = (col >> 3) ^ (((q >> 2) | (g >> 1) << 2) << 2);
    boff[j] = row * 512 + (slot << 4) + 8 * (q & 1);
  }

  pk_f16v acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = (pk_f16v){};
  pk_u4v af[2][FM];
  dt_s4 bf[2][FN][2];
  auto read = [&](const char* sA, const char* sB, int s) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r2 = 0; r2 < 2; ++r2) bf[s][j][r2] = dt_read_tr(sB + boff[j] + r2 * 2048);
#pragma unroll
    for (int i = 0; i < FM; ++i) af[s][i] = *reinterpret_cast<const pk_u4v*>(sA + aoff + 2048 * i);
  };
  auto mfma_step = [&](int s) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const dt_s8 b8 = __builtin_shufflevector(bf[s][j][0], bf[s][j][1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        if constexpr (BF16)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(pk_bf16x8, b8),
                                                              __builtin_bit_cast(pk_bf16x8, af[s][i]), acc[i][j], 0, 0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pk_half8, b8),
                                                             __builtin_bit_cast(pk_half8, af[s][i]), acc[i][j], 0, 0, 0);
      }
    }
  };
  auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
  // one LDS read, and with NV one DMA, per MFMA
  auto pattern = [] {
    constexpr int nv = VPT, nd = FM + 2 * FN, nm = FM * FN;
#pragma unroll
    for (int m = 0; m < nm; ++m) {
      if (m < nv) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      if (m == nm - 1 && nv > nm) __builtin_amdgcn_sched_group_barrier(0x020, nv - nm + 1, 0);
      if (m < nd) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (m == nm - 1 && nd > nm) __builtin_amdgcn_sched_group_barrier(0x100, nd - nm + 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
  };

  auto wait_tiles = [](auto NT) {  // this wave's DMA of all but the last NT tiles issued
    constexpr int n = decltype(NT)::value * VPT;
    __builtin_amdgcn_s_waitcnt((n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14));
  };
  issue(0, sA0, sB0);
  issue(min(1, last), sA1, sB1);
  issue(min(2, last), sA2, sB2);
  issue(min(3, last), sA3, sB3);
  issue(min(4, last), sA4, sB4);
  wait_tiles(pk_int_c<4>{});
  asm volatile("s_barrier" ::: "memory");
  read(sA0, sB0, 0);

  // k-tile t, its operands ready on entry; tile t + 1 in stage n, stage x held t - 1. (After the
  // last tile the reads touch a stage that holds a repeat of the last tile.)
  auto tile = [&](int kt, char* sAn, char* sBn, char* sAx, char* sBx, auto PAR) {
    constexpr int par = decltype(PAR)::value;
    fence();
    wait_tiles(pk_int_c<3>{});
    asm volatile("s_barrier" ::: "memory");
    fence();
    issue(min(kt + 5, last), sAx, sBx);
    mfma_step(par);
    read(sAn, sBn, par ^ 1);
    pattern();
    fence();
  };
  const pk_int_c<0> even{};
  const pk_int_c<1> odd{};
  int kt = 0;
  for (; kt + 6 <= ktiles; kt += 6) {
    tile(kt, sA1, sB1, sA5, sB5, even);
    tile(kt + 1, sA2, sB2, sA0, sB0, odd);
    tile(kt + 2, sA3, sB3, sA1, sB1, even);
    tile(kt + 3, sA4, sB4, sA2, sB2, odd);
    tile(kt + 4, sA5, sB5, sA3, sB3, even);
    tile(kt + 5, sA0, sB0, sA4, sB4, odd);
  }
  const int rem = ktiles - kt;
  if (rem > 0) tile(kt, sA1, sB1, sA5, sB5, even);
  if (rem > 1) tile(kt + 1, sA2, sB2, sA0, sB0, odd);
  if (rem > 2) tile(kt + 2, sA3, sB3, sA1, sB1, even);
  if (rem > 3) tile(kt + 3, sA4, sB4, sA2, sB2, odd);
  if (rem > 4) tile(kt + 4, sA5, sB5, sA3, sB3, even);
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): no DMA into LDS outlives the waves
  mfma_drain();

  // ---- epilogue: the k-half-1 waves park their accumulators in LDS (column wave c in its own
  // 16 KB, four fragments at a time, lane-major), the k-half-0 waves add them, stage slices of
  // rows in the same memory and store whole lines ------------------------------------------
  __syncthreads();
  const int cw = wave & 3;
  char* const region = cw == 0 ? sB0 : cw == 1 ? sB1 : cw == 2 ? sB2 : sB3;
  float* const park = reinterpret_cast<float*>(region);
#pragma unroll
  for (int half = 0; half < FM / 2; ++half) {
    if (h == 1) {
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int r = 0; r < 16; ++r) park[(f * 16 + r) * 64 + lane] = acc[2 * half + f / 2][f % 2][r];
    }
    __syncthreads();
    if (h == 0) {
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[2 * half + f / 2][f % 2][r] += park[(f * 16 + r) * 64 + lane];
    }
    __syncthreads();
  }
  if (h == 1) return;
  char* const out_base = reinterpret_cast<char*>(p.c);
  const int64_t out_off = (int64_t)blockIdx.y * p.c_slice;
  with_dtype(p.c_dtype, [&](auto DT) {
    constexpr int dt = decltype(DT)::value;
    constexpr int E = dt == PK_F32 ? 4 : 2;
    constexpr int RB = WN * E, NCH = RB / 16;  // bytes and 16-byte chunks per staged row
    constexpr int ROWS = 8192 / RB, FPS = ROWS / 32;
#pragma unroll
    for (int i0 = 0; i0 < FM; i0 += FPS) {
#pragma unroll
      for (int ii = 0; ii < FPS; ++ii)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int qq = 0; qq < 4; ++qq) {
            const int r = 32 * ii + l32, byte = (32 * j + 8 * qq + 4 * lh) * E;
            char* dst = region + r * RB + ((((byte >> 4) ^ (r % NCH)) << 4) | (byte & 15));
            const pk_f4 v = {acc[i0 + ii][j][4 * qq], acc[i0 + ii][j][4 * qq + 1],
                             acc[i0 + ii][j][4 * qq + 2], acc[i0 + ii][j][4 * qq + 3]};
            if constexpr (dt == PK_F32) {
              *reinterpret_cast<pk_f4*>(dst) = v;
            } else if constexpr (dt == PK_F16) {
              const pk_half4 hv = {(pk_half)v[0], (pk_half)v[1], (pk_half)v[2], (pk_half)v[3]};
              *reinterpret_cast<pk_u2v*>(dst) = __builtin_bit_cast(pk_u2v, hv);
            } else {
              *reinterpret_cast<pk_u2v*>(dst) =
                  pk_u2v{(uint32_t)f32_to_bf16_rne(v[0]) | ((uint32_t)f32_to_bf16_rne(v[1]) << 16),
                         (uint32_t)f32_to_bf16_rne(v[2]) | ((uint32_t)f32_to_bf16_rne(v[3]) << 16)};
            }
          }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the slice is in LDS
#pragma unroll
      for (int c0 = 0; c0 < ROWS * NCH; c0 += 64) {
        const int idx = c0 + lane, r = idx / NCH, ch = idx % NCH;
        const pk_u4v val = *reinterpret_cast<const pk_u4v*>(region + r * RB + ((ch ^ (r % NCH)) << 4));
        const int gm = m0 + 32 * i0 + r, gn = n0 + wn0 + ch * (16 / E);
        if (gm < p.M) __builtin_nontemporal_store(val, PK_GLOBAL(pk_u4v, out_base + (out_off + (int64_t)gm * p.ldc + gn) * E));
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // the slice is read back before the next one lands
    }
  });
}

bool dense_tr_ok(int M, int N, int K, int split, int64_t lda, const void* b, int64_t ldb,
                 int64_t ldc, int c_dtype, const void* c) {
  const int es = c_dtype == PK_F32 ? 4 : 2;
  if (N % 256 || K % (32 * split) || M < 64) return false;
  // A whole round of workgroups or more with slices of at most 1024 k is left to gemm_v3_f16_kernel
  // (slices of whole 64s). This kernel runs into the card's power limit there: its time depends on
  // what ran before and on the operands (fp16 2048 x 4096 x 512, both kernels in turn: 16.5 against
  // 17.6 us after a long run, 21 to 24 against 18.1 in bursts of 5 to 100, 14.5 against 15.8 on zeros), and
  // bursts take, old / new us: fp16 2048 x 4096 x 384 16.7 / 20.6, 3072 x 4096 x 512 29.2 / 32.5, 4096^2 x 768
  // 42.4 / 46.0, 2048 x 4096 x 1024 26.0 / 28.1; x 1536 34.3 / 30.7, 4096^2 x 1536 65.5 / 59.7. Fewer tiles have no
  // such K: 2048 x 3072 x 512 16.6 / 14.5, 1024 x 4096 x 256 11.8 / 8.5.
  const int64_t tiles = cdiv(M, 128) * (N / 256) * split;
  if (tiles >= 256 && K / split <= 1024 && K / split % 64 == 0) return false;
  if (ldb % 8 || (reinterpret_cast<uintptr_t>(b) & 15)) return false;
  if (split == 1 && ((ldc * es) % 16 || (reinterpret_cast<uintptr_t>(c) & 15))) return false;
  // 32-bit buffer offsets
  return (int64_t)M * lda * 2 < (1ll << 31) && (int64_t)K * ldb * 2 < (1ll << 31);
}

// 64-row tiles where as many rounds of the 256 CUs do (which is one round): 1024 x 4096 x 4096, 128 or
// 256 tiles: 51.7 against 42.7 us. A round of them takes 0.7 to 0.85 of one of 128 rows, so one
// more round is never made good: bf16 3840 x 2048 x 1600, 240 tiles of 128 rows 28.6 us, 480 of 64 rows
// 44; 3072 x 4096 x 2048, 384 or 768 tiles: 62 against 68.
int dense_tr_rows(int M, int N, int split) {
  auto rounds = [&](int rows) { return cdiv(cdiv(M, rows) * (N / 256) * split, 256); };
  return rounds(64) == rounds(128) ? 64 : 128;
}

int dense_tr_launch(bool bf16, const void* a, int64_t lda, const void* b, int64_t ldb, void* c,
                    int c_dtype, int64_t ldc, int M, int N, int K, int split, float* partials,
                    hipStream_t s) {
  DenseTrParams p;
  p.a = a;
  p.lda = lda;
  p.b = b;
  p.ldb = ldb;
  p.c = split > 1 ? (void*)partials : c;
  p.c_dtype = split > 1 ? (int)PK_F32 : c_dtype;
  p.ldc = split > 1 ? N : ldc;
  p.c_slice = split > 1 ? (int64_t)M * N : 0;
  p.M = M;
  p.K = K;
  p.kt_slice = K / split / 32;
  p.tiles_n = N / 256;
  const int bm = dense_tr_rows(M, N, split);
  p.tiles_m = (int)cdiv(M, bm);
  const dim3 grid(p.tiles_m * p.tiles_n, split);
  if (bf16 && bm == 128) gemm_dense_tr_kernel<true, 128><<<grid, 512, 0, s>>>(p);
  else if (bf16) gemm_dense_tr_kernel<true, 64><<<grid, 512, 0, s>>>(p);
  else if (bm == 128) gemm_dense_tr_kernel<false, 128><<<grid, 512, 0, s>>>(p);
  else gemm_dense_tr_kernel<false, 64><<<grid, 512, 0, s>>>(p);
  PK_LAUNCH_CHECK("gemm dense");
  if (split > 1) return splitk_reduce(partials, split, M, N, OutEpi(1.0f), c, c_dtype, ldc, s);
  return PK_OK;
}

}  // namespace pk
