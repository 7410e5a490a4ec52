// bf16 GEMM on 128 x 128 and 64 x 64 output tiles for gfx950: the products whose 256 x 256 tiles (llattn_gemm.hip)
// are too few for the chip, i.e. a few thousand rows and less -- prompts, micro-batches, the pooled latents.
//
// C[m][n] = sum_k A(m, k) B(n, k) with every operand layout, output and epilogue of llattn_gemm; the k split is inside
// the workgroup, and over workgroups (EPI_PART, the ordered reduction of llattn_gemm.hip behind it) only where a long
// contraction has a few tiles.
//
// Four waves (2 x 2), each 16 MB x 16 NB, share a tile's operands through NST LDS stages of 64 k filled by
// direct-to-LDS loads (as in llattn_gemm.hip), NST - 1 steps ahead; one barrier per step.  KG groups of four waves
// take a contiguous 1/KG of the steps each and their sums are added through LDS in order (deterministic, no partials
// in memory, no second launch).
//
// What bounds it: a CU's share of L2 bandwidth (a 128 x 128 tile needs 64 bytes per clock and CU at the full matrix
// rate, a 64 x 64 tile twice that) and, for tiles few enough that a CU has one, the latency of a step's loads.
// Deeper prefetch, fragments read a sub-step ahead and loads issued between the products gave nothing (a 128 x 128
// step stays at 0.75-0.9 us for a workgroup alone); measured times stand at tile_plan.
#include <algorithm>

#include "llattn_gemm.h"

namespace llattn {
namespace gemm {

namespace {

constexpr int SK = 64;  // k per stage

// Tile operand of O rows / columns x 64 k.  k-contiguous: rows of 128 bytes, chunk c (8 k) of row o at slot
// c ^ pswz<PERM>(o).  m/n-contiguous: 64 k-rows of 2 O bytes, chunk c (8 columns) of k-row k at c ^ 2 (k & 3).
template <bool KC, bool PERM, int O>
struct TileOp {
  static constexpr int BYTES = O * 128, NB = BYTES / 1024 / 4;  // NB: 1 KB DMA blocks per wave
  uint32_t off[NB];
  int kc[NB];
  __device__ __forceinline__ void init(int64_t ld, int o0, int omax, int w4, int lane) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int bi = w4 * NB + i;
      if constexpr (KC) {  // rows past omax are clamped to a valid row (their outputs are never stored)
        const int row = 8 * bi + (lane >> 3), c = (lane & 7) ^ pswz<PERM>(row);
        off[i] = (uint32_t)(((int64_t)min(o0 + row, omax - 1) * ld + 8 * c) * 2);
        kc[i] = 8 * c;
      } else {
        constexpr int PER = O / 8;
        const int q = bi * 64 + lane, k = q / PER, c = (q % PER) ^ (2 * (k & 3));
        off[i] = step_off(((int64_t)k * ld + min(o0 + 8 * c, omax - 8)) * 2);
        kc[i] = 0;
      }
    }
  }
  // block i of this wave; klim = K - k0 of the step: k-contiguous chunks at or past K read zero
  __device__ __forceinline__ void dma(const i32x4& rs, unsigned char* st, int w4, int i, int klim) const {
    dma_block(rs, KC ? kmask(off[i], kc[i], klim) : off[i], st + (w4 * NB + i) * 1024);
  }
  static __device__ __forceinline__ bf16x8 frag(const unsigned char* st, int o16, int r, int g, int h) {
    if constexpr (KC) {
      return frag64<true, PERM>(st, o16, r, g, h);
    } else {
      const int kb = 32 * h + 8 * g, col = o16 + 4 * (r & 3), chunk = col >> 3, inner = (col & 7) << 1;
      bf16x4 hv[2];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int k = kb + 4 * half + (r >> 2);
        const unsigned char* p = st + k * (2 * O) + ((chunk ^ (2 * (k & 3))) << 4) + inner;
        hv[half] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(p));
      }
      return bf16x8{hv[0][0], hv[0][1], hv[0][2], hv[0][3], hv[1][0], hv[1][1], hv[1][2], hv[1][3]};
    }
  }
};

// C[row][col .. col + 4) = v with the epilogue of the 256 x 256 kernels: bias, accumulation or row addends in fp32,
// one rounding, then the activation on the rounded value.
// EPI_PART: the plain sums into the partials of split `split`.
template <int EPI>
__device__ __forceinline__ void finish4(const GemmArgs& a, int split, int row, int col, f32x4 x) {
  if (row >= a.M || col >= a.N) return;
  if constexpr (EPI == EPI_PART) {
    *reinterpret_cast<f32x4*>(a.part + ((int64_t)split * a.M + row) * a.N + col) = x;
    return;
  }
  float v[4] = {x[0], x[1], x[2], x[3]};
  if (a.bias) {
    const float4 b = *reinterpret_cast<const float4*>(a.bias + col);
    v[0] += b.x; v[1] += b.y; v[2] += b.z; v[3] += b.w;
  }
  if constexpr (EPI == EPI_F32) {
    float* p = static_cast<float*>(a.C) + (int64_t)row * a.ldc + col;
    if (a.accumulate) {
      const float4 o = *reinterpret_cast<const float4*>(p);
      v[0] += o.x; v[1] += o.y; v[2] += o.z; v[3] += o.w;
    }
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    const int64_t o = a.ch.T ? (int64_t)heads_off(a.ch, (uint32_t)row, (uint32_t)col) : (int64_t)row * a.ldc + col;
    uint16_t* p = static_cast<uint16_t*>(a.C) + o;
    if (a.accumulate) {
      float c[4];
      load4<uint16_t>(p, c);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += c[e];
    }
    if (a.ra_ptr[0]) rowadd4(a, 0, row, col, v);
    if (a.ra_ptr[1]) rowadd4(a, 1, row, col, v);
    if (a.act) {
      uint16_t* pa = a.aux + (int64_t)row * a.ld_aux + col;
      float h[4];
      if (a.act == LLATTN_ACT_MUL_AUX) load4<uint16_t>(pa, h);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float xb = round_t<uint16_t>(v[e]);
        if (a.act == LLATTN_ACT_GELU) gelu_pair(xb, v[e], h[e]);
        else v[e] = xb * h[e];
      }
      if (a.act == LLATTN_ACT_GELU) store4<uint16_t>(pa, h);
    }
    store4<uint16_t>(p, v);
  }
}

constexpr int stage_bytes(int mb, int nb) { return 32 * (mb + nb) * 128; }

// Workgroup `block` of `blocks` of a product (EPI_PART: of a.n_split times its tiles); smem: KG NST stages.
template <bool AK, bool BKM, int EPI, int MB, int NB, int KG, int NST>
__device__ __forceinline__ void tile_product(const GemmArgs& a, int block, int blocks, unsigned char* smem) {
  constexpr int TM = 32 * MB, TN = 32 * NB;
  typedef TileOp<AK, false, TM> OpA;
  typedef TileOp<BKM, false, TN> OpB;
  constexpr int STAGE = stage_bytes(MB, NB), LOADS = OpA::NB + OpB::NB;  // loads of a wave per step
  static_assert(STAGE == OpA::BYTES + OpB::BYTES, "a stage holds both tiles");
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w4 = wave & 3, kg = wave >> 2;
  const int wm = w4 >> 1, wn = w4 & 1;
  // contiguous tile ranges per XCD, then groups of 8 tile rows
  int t = xcd_remap(block, blocks);
  int split = 0;
  int64_t a_bytes = a.a_bytes, b_bytes = a.b_bytes;
  int K = a.K, steps = a.k_pairs;
  if constexpr (EPI == EPI_PART) {  // k steps [split steps, + steps): the product of a shorter K and operands that end there
    const int tiles = a.tiles_m * a.tiles_n;
    split = t / tiles;
    t -= split * tiles;
    steps = (a.k_pairs + a.n_split - 1) / a.n_split;
    K = min(K, (split + 1) * steps * SK);
    if (!AK) a_bytes = min(a_bytes, ((int64_t)(K - 1) * a.lda + a.M) * 2);
    if (!BKM) b_bytes = min(b_bytes, ((int64_t)(K - 1) * a.ldb + a.N) * 2);
  }
  constexpr int GM = 8;
  const int group = t / (GM * a.tiles_n), first_m = group * GM, gm = min(a.tiles_m - first_m, GM);
  const int m0 = (first_m + (t % (GM * a.tiles_n)) % gm) * TM, n0 = (t % (GM * a.tiles_n)) / gm * TN;
  const bool rs = a.rowsum != nullptr && n0 == 0 && wn == 0;  // wave-uniform
  // every k group runs the same number of steps; those past K read zeros
  const int nk = (steps + KG - 1) / KG, kbeg = (split * steps + kg * nk) * SK;
  unsigned char* sm = smem + kg * NST * STAGE;

  OpA oa;
  OpB ob;
  oa.init(a.lda, m0, a.M, w4, lane);
  ob.init(a.ldb, n0, a.N, w4, lane);
  auto fetch = [&](int kt) {  // step kt (the last one again past the end: never read) into stage kt % NST
    const int k0 = kbeg + min(kt, nk - 1) * SK, klim = K - k0;
    const i32x4 ra = step_rsrc<AK>(a.A, a.lda, a_bytes, k0), rb = step_rsrc<BKM>(a.B, a.ldb, b_bytes, k0);
    unsigned char* st = sm + (kt % NST) * STAGE;
#pragma unroll
    for (int i = 0; i < OpA::NB; ++i) oa.dma(ra, st, w4, i, klim);
#pragma unroll
    for (int i = 0; i < OpB::NB; ++i) ob.dma(rb, st + OpA::BYTES, w4, i, klim);
  };
  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float rsum[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) rsum[i] = 0.f;
#pragma unroll
  for (int s = 0; s < NST - 1; ++s) fetch(s);
  for (int kt = 0; kt < nk; ++kt) {
    // this wave's loads of step kt have landed: loads complete in order and no store is in flight before the
    // epilogue, so a count of the youngest loads is exact
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0((NST - 2) * LOADS));
    __builtin_amdgcn_s_barrier();  // every wave's; and every wave has read step kt - 1, whose stage is free
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    fetch(kt + NST - 1);
    const unsigned char* st = sm + (kt % NST) * STAGE;
    bf16x8 fa[2][MB], fb[2][NB];  // k 0..31 and 32..63
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < NB; ++j) fb[h][j] = OpB::frag(st + OpA::BYTES, wn * 16 * NB + 16 * j, r, g, h);
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[h][i] = OpA::frag(st, wm * 16 * MB + 16 * i, r, g, h);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)  // B first: lane (r, g) accumulates C[m = r][n = 4 g + e]
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[h][j], fa[h][i], acc[i][j], 0, 0, 0);
    if (rs) {
      typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
      const bf16x2 one2 = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            rsum[i] = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{fa[h][i][2 * e], fa[h][i][2 * e + 1]}, one2, rsum[i], false);
    }
  }
  __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));  // no DMA in flight past this point
  // [KG][32 MB] row sums: behind the partial sums of the k groups where the stages leave room; for one k group, which
  // has none, in the stages themselves (five 64 x 64 workgroups then fill a CU's LDS to the byte)
  constexpr bool OWN = KG > 1 && NST * STAGE == MB * NB * 4096;
  __shared__ float own[OWN ? KG * TM : 1];
  float* rsl = OWN ? own : reinterpret_cast<float*>(smem + (KG > 1 ? KG * MB * NB * 4096 : 0));
  if (!OWN && a.rowsum && n0 == 0) __syncthreads();  // every wave's loads have landed and its fragments are read
  if (rs) {  // the four lane groups hold the row's four 8-wide k slices
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      float v = rsum[i];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (g == 0) rsl[kg * TM + wm * 16 * MB + 16 * i + r] = v;
    }
  }
  __syncthreads();
  const int rowb = m0 + wm * 16 * MB + r, colb = n0 + wn * 16 * NB + 4 * g;
  if constexpr (KG == 1) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) finish4<EPI>(a, split, rowb + 16 * i, colb + 16 * j, acc[i][j]);
  } else {
    f32x4* red = reinterpret_cast<f32x4*>(smem);  // [KG][4 waves][MB][NB][64]
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) red[((wave * MB + i) * NB + j) * 64 + lane] = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < MB * NB; ++u) {  // blocks are shared out among the k groups
      if (u % KG != kg) continue;
      f32x4 v = red[(w4 * MB * NB + u) * 64 + lane];
#pragma unroll
      for (int w = 1; w < KG; ++w) v += red[((4 * w + w4) * MB * NB + u) * 64 + lane];
      finish4<EPI>(a, split, rowb + 16 * (u / NB), colb + 16 * (u % NB), v);
    }
  }
  if (a.rowsum && n0 == 0 && threadIdx.x < TM && m0 + (int)threadIdx.x < a.M) {
    float v = rsl[threadIdx.x];
#pragma unroll
    for (int w = 1; w < KG; ++w) v += rsl[w * TM + threadIdx.x];
    float* out = EPI == EPI_PART ? a.part + ((int64_t)a.n_split * a.N + split) * a.M : a.rowsum;
    out[m0 + threadIdx.x] = v;
  }
}

template <bool AK, bool BKM, int EPI, int MB, int NB, int KG, int NST>
__global__ __launch_bounds__(256 * KG) void gemm_tile_kernel(const GemmArgs a) {
  __shared__ __align__(1024) unsigned char smem[KG * NST * stage_bytes(MB, NB)];
  tile_product<AK, BKM, EPI, MB, NB, KG, NST>(a, blockIdx.x, gridDim.x, smem);
}

// Two independent products in one launch: the first n0 workgroups (a multiple of 8, so that both see their XCD) take
// the first one.  An input and a weight gradient of the same dy, or two projections, each fill the chip badly at a
// few thousand rows; together they share its last round and one launch.
template <bool AK0, bool BK0, int EPI0, bool AK1, bool BK1, int EPI1, int MB, int KG>
__global__ __launch_bounds__(256 * KG) void gemm_tile_pair_kernel(const GemmArgs a0, const GemmArgs a1, int n0) {
  __shared__ __align__(1024) unsigned char smem[KG * 2 * stage_bytes(MB, MB)];
  const int b = blockIdx.x, c0 = a0.tiles_m * a0.tiles_n, c1 = a1.tiles_m * a1.tiles_n;
  if (b < n0) {
    if (b < c0) tile_product<AK0, BK0, EPI0, MB, MB, KG, 2>(a0, b, c0, smem);
  } else if (b - n0 < c1) {
    tile_product<AK1, BK1, EPI1, MB, MB, KG, 2>(a1, b - n0, c1, smem);
  }
}

// 128 x 128 tiles run two workgroups per CU with one k group, one with two; 64 x 64 tiles five with one, and with two k
// groups one of four stages each, or two of two stages where there are more tiles than CUs (1024 x 1408 x 4096, 352
// tiles: two rounds of the first 31 us, one of the second 26; 333 x 1408 x 4096, 132 tiles: 17 against 24).
template <bool AK, bool BKM, int EPI>
void launch_epi(const GemmArgs& a, const TilePlan& p, hipStream_t st) {
  const dim3 grid(a.tiles_m * a.tiles_n);
  if constexpr (EPI == EPI_PART) {
    hipLaunchKernelGGL((gemm_tile_kernel<AK, BKM, EPI, 2, 2, 1, 2>), dim3(grid.x * a.n_split), dim3(256), 0, st, a);
  } else if (p.mb == 4 && p.kg == 1) hipLaunchKernelGGL((gemm_tile_kernel<AK, BKM, EPI, 4, 4, 1, 2>), grid, dim3(256), 0, st, a);
  else if (p.mb == 4) hipLaunchKernelGGL((gemm_tile_kernel<AK, BKM, EPI, 4, 4, 2, 2>), grid, dim3(512), 0, st, a);
  else if (p.kg == 1) hipLaunchKernelGGL((gemm_tile_kernel<AK, BKM, EPI, 2, 2, 1, 2>), grid, dim3(256), 0, st, a);
  else if (grid.x > 256) hipLaunchKernelGGL((gemm_tile_kernel<AK, BKM, EPI, 2, 2, 2, 2>), grid, dim3(512), 0, st, a);
  else hipLaunchKernelGGL((gemm_tile_kernel<AK, BKM, EPI, 2, 2, 2, 4>), grid, dim3(512), 0, st, a);
}
template <bool AK, bool BKM>
void launch_dt(const GemmArgs& a, const TilePlan& p, int c_dtype, hipStream_t st) {
  if (a.n_split > 1) launch_epi<AK, BKM, EPI_PART>(a, p, st);
  else if (c_dtype == LLATTN_F32) launch_epi<AK, BKM, EPI_F32>(a, p, st);
  else launch_epi<AK, BKM, EPI_BF16>(a, p, st);
}

}  // namespace

// Time in us of the 256 x 256 kernels with S k splits: 6 us to fill and drain, rounds of (tile, split) workgroups over 256 CUs, 1.2 us per
// 64-k step of a workgroup alone up to 1.75 with every CU at work, and for S > 1 the ordered reduction with its fp32
// partials written and read at 7 TB/s.  (1024 x 4736 x 1408, 76 tiles: 32 us; 8192 x 4096 x 1408, 512: 83;
// 1536 x 1536 x 4011, 36 tiles in 7 splits: 41.)
static double big_us(int64_t M, int64_t N, int steps, int S) {
  const int64_t n = ((M + BM - 1) / BM) * ((N + BN - 1) / BN) * S;
  const double last = (double)(n % 256) / 256.0;
  const double per = (double)(n / 256) * 1.75 + (n % 256 ? 1.2 + 0.55 * last * last : 0.0);
  return 6.0 + (double)((steps + S - 1) / S) * per + (S > 1 ? 7.0 + 8.0 * S * (double)M * (double)N / 7e6 : 0.0);
}

// The tiles that a product takes, fitted to the times of 38 products (16 x 1024 x 1408 to 3000 x 4736 x 1408; all
// layouts) whose operands the launches before had just written, as a step finds them: 2-5 us longer than on operands
// left in L2 by the same product.
//   128 x 128, one k group: rounds of two tiles per CU, 1.27 us per 64-k step (1.02 for a last round of up to two, 0.75
//   for one), 8.5 us once;  two k groups: rounds of one, 5.5 us each and 0.95 per step of a group;
//   64 x 64, one k group: rounds of four tiles per CU, 0.85 us per step (0.5 for a last round of one, 0.52 of two, 0.68
//   of three), 4.5 us once;  two k groups: 0.44 us per step of a group for up to one tile per CU, 0.68 for up to two.
//   (Four k groups: no faster.)
//   64 x 64 split over workgroups: 5.2 us and 0.07 per split with the reduction's launch, the same steps (from memory 2.8 TB/s at most, in
//   pieces of 128 bytes a k row), partials written and read at 4.2 TB/s.
//   (dyᵀ x, 128 x 128 x 16384: 15.6 us in 16 splits against 62 in two k groups and 36 on 256 x 256 tiles in 64 splits;
//   512 x 512 x 16384 27 in 16 splits against 42 there; 1408 x 512 x 8192, 176 tiles, 31 in 4 splits against 36.)
// Only where 256 x 256 tiles leave CUs idle (below 224 of them): from there on
// those tiles' half as large operand traffic wins (4011 x 4992 x 1536: 69 us against 81).  Epilogue and layouts enter
// through the 256 x 256 kernels' split count alone: near the line a product stored split-head or with row addends takes
// these tiles where the plain one is split there, and its sums run in another k order (2950 x 1408 x 4096, x Wᵀ).
// Measured on operands just written, in us: 333 x 4736 x 1408 13.5, 1024 x 1408 x 1408 13.3,
// 1024 x 1408 x 4096 26.8, 1024 x 4096 x 1408 18.7, 4011 x 384 x 1536 (dy W) 14.3, 1536 x 384 x 4011 (dyT x) 18.5;
// with L2-resident operands against the 256 x 256 kernels and the register-staged 64 x 64 tiles that this replaced:
//   333 x 4736 x 1408: 30 -> 12.5;  1024 x 4096 x 1408: 30 -> 17;  1536 x 384 x 4011: 52 -> 18;  32768 x 64 x 1024:
//   24 -> 13.
TilePlan tile_plan(const llattn_gemm_desc* d, double* us) {
  const TilePlan none{0, 0, 0, 1};
  if (d->split_k > 0 || d->M <= 0 || d->N <= 0 || d->K <= 0) return none;
  const int64_t M = d->M, N = d->N;
  if (((M + BM - 1) / BM) * ((N + BN - 1) / BN) >= 224) return none;
  const int steps = (d->K + SK - 1) / SK;
  TilePlan best = none;
  double best_t = 0.97 * big_us(M, N, steps, resolve_split(d));
  const auto take = [&](double t, int mb, int kg, int S = 1) {
    if (t < best_t) {
      best_t = t;
      best = TilePlan{mb, mb, kg, S};
    }
  };
  const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128), t64 = ((M + 63) / 64) * ((N + 63) / 64);
  const auto split = [&](int kg) { return (double)((steps + kg - 1) / kg); };
  const int64_t r128 = t128 % 512, r64 = (t64 % 1024 + 255) / 256;
  take(8.5 + steps * ((double)(t128 / 512) * 1.27 + (r128 == 0 ? 0.0 : r128 <= 256 ? 0.75 : 1.02)), 4, 1);
  if (steps >= 4) take(3.0 + (double)((t128 + 255) / 256) * (5.5 + split(2) * 0.95), 4, 2);
  const double last[] = {0.0, 0.5, 0.52, 0.68, 0.82};
  take(4.5 + steps * ((double)(t64 / 1024) * 0.85 + last[r64]), 2, 1);
  if (steps >= 4 && t64 <= 256) take(3.8 + split(2) * 0.44, 2, 2);
  if (steps >= 4 && t64 > 256 && t64 <= 512) take(5.6 + split(2) * 0.68, 2, 2);
  // a few tiles of a long contraction: 64 x 64 tiles over S ranges of at least two steps, their partials reduced in order.
  // From K = 6144 on: below, the GPU gains at most 10 us (128 x 128 x 4096 16 -> 8), and a step of products this small
  // waits for the host, to which the second launch costs 4 (with it from K = 2048: the 0.55b model over 64 tokens
  // 3310 -> 3460 us, a 256-wide block's training pass over 4096 tokens 308 -> 320).
  const double stream = 2.0 * (double)(M + N) * (double)d->K / 2.8e6;
  for (int S = 2; S <= 32 && steps >= 96; S *= 2) {
    const int64_t per = (steps + S - 1) / S, parts = (steps + per - 1) / per, n = t64 * parts;  // no range is empty
    if (per < 2 || n > 2048) break;
    take(5.2 + 0.07 * (double)parts + std::max(stream, (double)per * ((double)(n / 1024) * 0.85 + last[(n % 1024 + 255) / 256])) +
             8.0 * (double)parts * (double)M * (double)N / 4.2e6, 2, 1, (int)parts);
  }
  if (us) *us = best_t;
  return best;
}

void launch_tile(const GemmArgs& a0, const TilePlan& p, bool a_kmaj, bool b_kmaj, int c_dtype, hipStream_t st) {
  GemmArgs a = a0;
  a.tiles_m = (a.M + 32 * p.mb - 1) / (32 * p.mb);
  a.tiles_n = (a.N + 32 * p.nb - 1) / (32 * p.nb);
  a.n_split = p.splits;
  if (a_kmaj && b_kmaj) launch_dt<true, true>(a, p, c_dtype, st);
  else if (a_kmaj) launch_dt<true, false>(a, p, c_dtype, st);
  else if (!b_kmaj) launch_dt<false, false>(a, p, c_dtype, st);
  else launch_dt<false, true>(a, p, c_dtype, st);
}

namespace {

// Time in us of a product by itself, as tile_plan and resolve_split leave it.
double alone_us(const llattn_gemm_desc* d) {
  double t = 0.0;
  const TilePlan p = tile_plan(d, &t);
  const int64_t tiles = ((d->M + BM - 1) / BM) * (int64_t)((d->N + BN - 1) / BN);
  if (!p.mb) t = tiles >= 224 ? big_us(d->M, d->N, (d->K + SK - 1) / SK, 1) : big_us(d->M, d->N, (d->K + SK - 1) / SK, resolve_split(d));
  return t;
}

template <int MB, int KG>
void launch_pair_as(const GemmArgs& a0, const GemmArgs& a1, bool nt0, bool nt1, int n0, dim3 grid, hipStream_t st) {
  const dim3 block(256 * KG);
  if (nt1)
    hipLaunchKernelGGL((gemm_tile_pair_kernel<true, true, EPI_BF16, true, true, EPI_BF16, MB, KG>), grid, block, 0, st,
                       a0, a1, n0);
  else if (nt0)
    hipLaunchKernelGGL((gemm_tile_pair_kernel<true, true, EPI_BF16, false, false, EPI_F32, MB, KG>), grid, block, 0, st,
                       a0, a1, n0);
  else
    hipLaunchKernelGGL((gemm_tile_pair_kernel<true, false, EPI_BF16, false, false, EPI_F32, MB, KG>), grid, block, 0, st,
                       a0, a1, n0);
}

}  // namespace

// Tiles of two products in one launch, or none where they are better run one by one: the work of all tiles at a full
// chip's rate per (tile, step), or the longest tile at the rate of the tiles that share its CU, and part of a shorter
// one for the ragged end; taken where that saves 5%.  (q|k|v and the latents' keys and values of a 0.55b layer over 333
// tokens: 17 + 8 us in two launches, 18 in one of one k group, 14 of two; the latent projections' two gradients of
// 4 x 8192 tokens with 64-token query blocks 5 + 10 us in two, 11.5 in one.  The gradients of a few thousand tokens'
// large projections stay apart: the weight gradient's long contraction wants its own k split.)
TilePlan pair_plan(const llattn_gemm_desc* d0, const llattn_gemm_desc* d1) {
  const TilePlan none{0, 0, 0, 1};
  for (const llattn_gemm_desc* d : {d0, d1})
    if (d->split_k > 0 || d->M <= 0 || d->N <= 0 || d->K <= 0) return none;
  const bool bf0 = d0->c_dtype == LLATTN_BF16 && !d0->a_trans, nt1 = d1->c_dtype == LLATTN_BF16 && !d1->a_trans && !d1->b_trans;
  const bool tn1 = d1->c_dtype == LLATTN_F32 && d1->a_trans && d1->b_trans;
  if (!bf0 || !(tn1 || (nt1 && !d0->b_trans))) return none;
  const double s0 = (d0->K + SK - 1) / SK, s1 = (d1->K + SK - 1) / SK;
  double best_t = 0.95 * (alone_us(d0) + alone_us(d1));
  TilePlan best = none;
  const auto take = [&](int mb, int kg, double fill, double rate, const auto& alone) {
    const int64_t T = 32 * mb;
    const double t0 = (double)(((d0->M + T - 1) / T) * ((d0->N + T - 1) / T));
    const double t1 = (double)(((d1->M + T - 1) / T) * ((d1->N + T - 1) / T));
    const double most = std::max(s0, s1), least = std::min(s0, s1), step = alone(t0 + t1);
    if (step == 0.0) return;
    const double t = fill + std::max((t0 * s0 + t1 * s1) * rate, step * most) + 0.18 * step * least;
    if (t < best_t) {
      best_t = t;
      best = TilePlan{mb, mb, kg, 1};
    }
  };
  take(4, 1, 8.5, 1.27 / 512.0, [](double n) { return n <= 256 ? 0.75 : 1.02; });
  take(2, 1, 4.5, 0.85 / 1024.0, [](double n) { return n <= 512 ? 0.52 : n <= 768 ? 0.68 : 0.82; });
  if (s0 >= 4 && s1 >= 4) take(2, 2, 5.6, 0.8 / 1024.0, [](double n) { return n <= 512 ? 0.34 : 0.0; });
  return best;
}

void launch_pair(GemmArgs a0, GemmArgs a1, const TilePlan& p, bool b_kmaj0, bool weight1, hipStream_t st) {
  const int T = 32 * p.mb;
  for (GemmArgs* a : {&a0, &a1}) {
    a->tiles_m = (a->M + T - 1) / T;
    a->tiles_n = (a->N + T - 1) / T;
  }
  const int n0 = (a0.tiles_m * a0.tiles_n + 7) / 8 * 8;
  const dim3 grid(n0 + a1.tiles_m * a1.tiles_n);
  if (p.mb == 4) launch_pair_as<4, 1>(a0, a1, b_kmaj0, !weight1, n0, grid, st);
  else if (p.kg == 1) launch_pair_as<2, 1>(a0, a1, b_kmaj0, !weight1, n0, grid, st);
  else launch_pair_as<2, 2>(a0, a1, b_kmaj0, !weight1, n0, grid, st);
}

}  // namespace gemm
}  // namespace llattn
