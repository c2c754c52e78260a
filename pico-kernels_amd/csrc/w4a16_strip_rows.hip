// W4A16 matmul for a batch of rows (5 <= M <= 64) on strip-layout weights (w4a16_strips.hip gives
// the layout): C = tensor_scale * A (M, K) fp16 @ dequant(q, S) (+ bias), in one launch.
//
// What it replaces at these rows, the register-dequant kernel on the block layout, splits K over
// workgroups and hands fp32 partials over through L2: its loads, products, LDS sums and
// hand-off follow one another in a single round of workgroups, and more loads in flight (1,
// 2 or 4 k-steps) change nothing. Here a workgroup owns 16 * NS columns over the whole of K, so
// nothing is handed over, and its NW waves take every NW-th 128-row block: the block's weights
// (1 KB contiguous per strip) and activations (256 bytes of each row) go to the wave's own LDS by
// DMA, two blocks ahead, so a wave waits for no other until the end.
//
// A 1 KB block's 16-byte chunk L = 16g + 4rs + cps holds rows 32rs + 8g + e (e = 0..7) of the
// columns 4cps .. 4cps+3: byte 8h + e the columns 4cps + 2h (low nibble) and + 1 (high). The B
// operand of v_mfma_f32_16x16x32_f16 for the 32 rows of row set rs wants in lane 16g + j the 8 rows
// 8g + e of one column: lane j = 4q + cps reads the 8 bytes of chunk (g, rs, cps) at h = q / 2
// and takes nibble q % 2, i.e. column 4cps + q. So every MFMA works on 16 columns and 16 rows of
// activations (the decode kernel's form spends its columns on four row sets of four columns
// each, which serves at most eight rows). Its A operand is the plain one: lane 16g + i loads
// k = 8g + e of activation row i, 16 bytes.
//
// Dequantisation is exact: the bytes are shifted and masked to u = v + 8, a byte permute puts two
// of them under the fp16 exponent of 1024 (0x64), and a packed fp16 add of -1032 leaves v. Group
// sums are scaled in fp32 at each group's end (FOLDS per block), per-tensor sums once.
//
// What bounds it is the activations: every workgroup reads all M * K * 2 bytes, so NS strips
// share one copy. Loaded to registers as the MFMA wants them (16 rows of 64 bytes per
// instruction) they came at 11 bytes per clock and CU (4096 x 4096 M = 32 10.2 us); a DMA of whole
// 256-byte row pieces takes 7.3 us. LDS slot c of row r holds chunk c ^ (r % 16), so that sixteen
// rows read at one chunk touch sixteen bank groups.
//
// Measured on MI355X in graphs over rotating weights, against the register-dequant kernel (M = 8:
// the decode kernel) and the kernels it fell back to where the weights cannot be blocks: M = 8 /
// 16 / 32 / 64 of 4096 x 6144 7.5 / 9.0 / 11.6 / 15.7 -> 6.5 / 6.8 / 9.2 / 13.8 us, 4096 x 4096
// M = 16 / 32 7.2 / 9.7 -> 5.9 / 7.3, 4096 x 14336 M = 8 / 16 / 32 11.5 / 13.1 / 16.8 -> 10.1 / 10.7 /
// 13.5, 8192 x 14336 M = 32 26.8 -> 21.4, 1024 x 2048 M = 32 7.5 -> 3.8; no blocks: 4096 x 14352
// M = 32 20.9 -> 14.2, 6272 x 12304 (49 slices before) 63 -> 19. Not everywhere: where its workgroups
// just miss a round of 256 (8064 x 9216 M = 64 24.0 -> 41.3) or are few (13312 x 1920 M = 31 14.0 -> 16.8)
// the other kernels are the faster ones, and so is the decode kernel up to 8 rows with groups of 32
// (10496 x 6144 14.2 -> 17.3): the callers' rules say which serves a call.
#include "pk_internal.h"

namespace pk {


struct StripRowsParams {
  const pk_half* a;
  int64_t lda;
  const uint8_t* qs;  // strips of kb 1 KB blocks
  const pk_half* ss;  // (N/16, K/G, 16) or null
  int group;
  OutEpi epi;
  void* c;
  int c_dtype;
  int64_t ldc;
  int M, strips, kb, kg;  // kb: 128-row blocks, kg: groups
  int per_xcd;            // workgroups per XCD
};

// 16 bytes per lane, global -> LDS (lane L writes lds + 16 L). A device-only helper: the
// generic-to-LDS pointer cast must not appear in host-visible code (lambdas).
template <int AUX>
__device__ __forceinline__ void sr_dma16(__amdgpu_buffer_rsrc_t r, char* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, AUX);
}
// Waits until at most N of this wave's loads are in flight (in issue order).
template <int N>
__device__ __forceinline__ void sr_wait_loads() {
  static_assert(N < 64, "vmcnt holds at most 63");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}

// MB: 16-row activation blocks; NS: strips per workgroup; FOLDS: group ends per 128-row block (1:
// groups of 128 or more, 2 or 4: of 64 or 32), 0: per-tensor.
template <int MB, int NS, int NW, int FOLDS>
__global__ __launch_bounds__(64 * NW) void w4a16_strip_rows_kernel(StripRowsParams p) {
  __shared__ __align__(16) char stage0[NW * NS * 1024];
  __shared__ __align__(16) char stage1[NW * NS * 1024];
  __shared__ __align__(16) char act0[NW * MB * 4096];  // the waves' sums in the end
  __shared__ __align__(16) char act1[NW * MB * 4096];
  auto red = reinterpret_cast<float (*)[NS][MB * 16][16]>(act0);
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int j = lane & 15, g = lane >> 4, cps = j & 3, q = j >> 2;
  // workgroup b runs on XCD b % 8: neighbouring strips (whole output lines) on one XCD
  const int wg = (blockIdx.x & 7) * p.per_xcd + (blockIdx.x >> 3);
  const int s0 = wg * NS;
  if (s0 >= p.strips) return;
  const int live = min(NS, p.strips - s0);  // the last workgroup's strips past the end repeat its last

  const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.a, (uint32_t)((int64_t)p.M * p.lda * 2));
  int a_off[4 * MB];
#pragma unroll
  for (int i = 0; i < 4 * MB; ++i) {
    const int r = 4 * i + g;
    a_off[i] = (int)(min(r, p.M - 1) * p.lda) * 2 + (j ^ (r & 15)) * 16;
  }
  const __amdgpu_buffer_rsrc_t rq =
      make_rsrc(p.qs + (int64_t)s0 * p.kb * 1024, (uint32_t)live * (uint32_t)p.kb * 1024u);
  const int strip_bytes = p.kb * 1024;
  const __amdgpu_buffer_rsrc_t rsc =
      make_rsrc(FOLDS ? (const void*)(p.ss + (int64_t)s0 * p.kg * 16) : (const void*)p.a,
                FOLDS ? (uint32_t)live * (uint32_t)p.kg * 32u : 0u);

  constexpr int SPB = FOLDS > 1 ? FOLDS : 1;  // scales per block and strip
  uint32_t sc[2][NS][SPB];
  // A stage's loads: the scales, then the DMAs, which nothing but an explicit wait holds LDS reads
  // back for (kDma counts them: the wait for a stage leaves the next one's in flight).
  constexpr int kDma = NS + 4 * MB;
  auto load = [&](int which, char* stage, char* act, int b) {
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FOLDS != 0) {
#pragma unroll
      for (int st = 0; st < NS; ++st)
#pragma unroll
        for (int f = 0; f < SPB; ++f) {
          const int grp = FOLDS > 1 ? b * FOLDS + f : b * 128 / p.group;
          sc[which][st][f] = __builtin_amdgcn_raw_buffer_load_b16(
              rsc, (4 * cps + q) * 2, (min(st, live - 1) * p.kg + grp) * 32, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < NS; ++st)
      sr_dma16<kPkLoadStream>(rq, stage + (wave * NS + st) * 1024, lane * 16,
                              min(st, live - 1) * strip_bytes + b * 1024);
#pragma unroll
    for (int i = 0; i < 4 * MB; ++i)
      sr_dma16<0>(ra, act + wave * MB * 4096 + i * 1024, a_off[i], b * 256);
    __builtin_amdgcn_sched_barrier(0);
  };

  pk_f4 acc[NS][MB];
#pragma unroll
  for (int st = 0; st < NS; ++st)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[st][mb] = pk_f4{0.0f, 0.0f, 0.0f, 0.0f};
  const int shift = 4 * (q & 1);
  const int rd = 256 * g + 16 * cps + 8 * (q >> 1);  // the lane's 8 bytes of row set 0
  const pk_half2 m1032 = {(pk_half)-1032.0f, (pk_half)-1032.0f};

  auto compute = [&](int which, const char* stage, const char* act) {
    pk_u4v x[4][MB];
#pragma unroll
    for (int rs = 0; rs < 4; ++rs)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        x[rs][mb] = *reinterpret_cast<const pk_u4v*>(act + wave * MB * 4096 + (mb * 16 + j) * 256 + (((4 * rs + g) ^ j) << 4));
#pragma unroll
    for (int st = 0; st < NS; ++st) {
      const char* blk = stage + (wave * NS + st) * 1024 + rd;
      pk_u2v w[4];
#pragma unroll
      for (int rs = 0; rs < 4; ++rs) w[rs] = *reinterpret_cast<const pk_u2v*>(blk + 64 * rs);
      pk_f4 d[MB];
#pragma unroll
      for (int rs = 0; rs < 4; ++rs) {
        const uint32_t u0 = (w[rs][0] >> shift) & 0x0f0f0f0fu, u1 = (w[rs][1] >> shift) & 0x0f0f0f0fu;
        pk_u4v b;
        b[0] = __builtin_amdgcn_perm(0x64646464u, u0, 0x04010400u);  // 0x64 over bytes 0 and 1
        b[1] = __builtin_amdgcn_perm(0x64646464u, u0, 0x04030402u);
        b[2] = __builtin_amdgcn_perm(0x64646464u, u1, 0x04010400u);
        b[3] = __builtin_amdgcn_perm(0x64646464u, u1, 0x04030402u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t bi = b[i];
          b[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(pk_half2, bi) + m1032);
        }
        const pk_half8 bv = __builtin_bit_cast(pk_half8, b);
        constexpr int RPF = FOLDS > 1 ? 4 / FOLDS : 4;  // row sets per fold
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          const pk_half8 av = __builtin_bit_cast(pk_half8, x[rs][mb]);
          if constexpr (FOLDS == 0) {
            acc[st][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, acc[st][mb], 0, 0, 0);
          } else {
            d[mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                av, bv, rs % RPF == 0 ? pk_f4{0.0f, 0.0f, 0.0f, 0.0f} : d[mb], 0, 0, 0);
            if (rs % RPF == RPF - 1) {
              uint32_t sb = sc[which][st][FOLDS > 1 ? rs / RPF : 0];
              asm volatile("" : "+v"(sb));  // converted here, not as soon as it is loaded
              const float s = (float)__builtin_bit_cast(pk_half, (uint16_t)sb);
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[st][mb][r] = __builtin_fmaf(d[mb][r], s, acc[st][mb][r]);
            }
          }
        }
      }
    }
  };

  // wave-uniform: blocks wave, wave + NW, ... through two stages
  if (wave < p.kb) load(0, stage0, act0, wave);
  if (wave + NW < p.kb) load(1, stage1, act1, wave + NW);
  for (int b = wave; b < p.kb; b += 2 * NW) {
    const bool two = b + NW < p.kb;
    if (two) sr_wait_loads<kDma>();
    else sr_wait_loads<0>();
    compute(0, stage0, act0);
    const bool more = b + 2 * NW < p.kb;
    if (more) load(0, stage0, act0, b + 2 * NW);
    if (two) {
      if (more) sr_wait_loads<kDma>();
      else sr_wait_loads<0>();
      compute(1, stage1, act1);
      if (b + 3 * NW < p.kb) load(1, stage1, act1, b + 3 * NW);
    }
  }
  if constexpr (FOLDS == 0) mfma_drain();

  // ---- the waves' sums, in wave order -----------------------------------------------------
  __syncthreads();  // act0 has been read
#pragma unroll
  for (int st = 0; st < NS; ++st)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][st][mb * 16 + 4 * g + r][4 * cps + q] = acc[st][mb][r];
  __syncthreads();
  for (int i = t; i < p.M * NS * 16; i += 64 * NW) {
    const int m = i / (NS * 16), col = i % (NS * 16), st = col / 16;
    if (st >= live) continue;
    float v = red[0][st][m][col % 16];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += red[w][st][m][col % 16];
    const int n = s0 * 16 + col;
    store_from_f32(p.c, p.c_dtype, (int64_t)m * p.ldc + n, p.epi(v, n));
  }
}

template <int MB, int NS, int NW>
static void strip_rows_launch_t(const StripRowsParams& p, int folds, hipStream_t s) {
  const dim3 grid(8 * p.per_xcd), block(64 * NW);
  if (folds == 0) w4a16_strip_rows_kernel<MB, NS, NW, 0><<<grid, block, 0, s>>>(p);
  else if (folds == 1) w4a16_strip_rows_kernel<MB, NS, NW, 1><<<grid, block, 0, s>>>(p);
  else if (folds == 2) w4a16_strip_rows_kernel<MB, NS, NW, 2><<<grid, block, 0, s>>>(p);
  else w4a16_strip_rows_kernel<MB, NS, NW, 4><<<grid, block, 0, s>>>(p);
}

// Strips per workgroup: the fewest whose workgroups fit the 256 CUs in one round (measured on
// MI355X at NS = 1 / 2 / 4, M = 16: 4096 x 4096 6.0 / 6.7 / 9.4 us, 4096 x 8192 8.9 / 7.2 / 9.6,
// 4096 x 14336 14.3 / 12.4 / 10.7); above 32 rows two at most (four 16-row blocks of activations
// leave LDS for no more).
static int strip_rows_ns(int M, int N) {
  const int strips = N / 16;
  return strips <= 256 ? 1 : strips <= 512 || M > 32 ? 2 : 4;
}

int strip_rows_launch(const void* a, int64_t lda, const uint8_t* qs, const void* ss, int group,
                      OutEpi epi, void* c, int c_dtype, int64_t ldc, int M, int N, int K,
                      hipStream_t s) {
  StripRowsParams p;
  p.a = reinterpret_cast<const pk_half*>(a);
  p.lda = lda;
  p.qs = qs;
  p.ss = reinterpret_cast<const pk_half*>(ss);
  p.group = ss ? group : K;
  p.epi = epi;
  p.c = c;
  p.c_dtype = c_dtype;
  p.ldc = ldc;
  p.M = M;
  p.strips = N / 16;
  p.kb = K / 128;
  p.kg = ss ? K / group : 1;
  const int ns = strip_rows_ns(M, N);
  p.per_xcd = (int)cdiv(cdiv(p.strips, ns), 8);
  const int folds = ss == nullptr ? 0 : group >= 128 ? 1 : 128 / group;
  if (M <= 16) {
    if (ns == 1) strip_rows_launch_t<1, 1, 8>(p, folds, s);
    else if (ns == 2) strip_rows_launch_t<1, 2, 8>(p, folds, s);
    else strip_rows_launch_t<1, 4, 8>(p, folds, s);
  } else if (M <= 32) {
    if (ns == 1) strip_rows_launch_t<2, 1, 8>(p, folds, s);
    else if (ns == 2) strip_rows_launch_t<2, 2, 8>(p, folds, s);
    else strip_rows_launch_t<2, 4, 6>(p, folds, s);
  } else {
    if (ns == 1) strip_rows_launch_t<4, 1, 4>(p, folds, s);
    else strip_rows_launch_t<4, 2, 4>(p, folds, s);
  }
  PK_LAUNCH_CHECK("w4a16 strip rows");
  return PK_OK;
}

}  // namespace pk
