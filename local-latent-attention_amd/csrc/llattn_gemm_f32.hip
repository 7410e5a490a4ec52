// fp32 projection GEMM for gfx950: C = A Bᵀ (+ bias) (+ C) with fp32 operands and fp32 accumulation on
// v_mfma_f32_16x16x4_f32, the fp32 counterpart of llattn_gemm for the fp32 module (the reference's
// nn.Linear products in fp32, models.py:80-84, 315, 333-353, 395, 462, and their autograd).
//
// Same descriptor and operand layouts as llattn_gemm: A(m, k) is A[m * lda + k] (a_trans = 0) or
// A[k * lda + m] (a_trans = 1); B(n, k) is B[n * ldb + k] (b_trans = 0) or B[k * ldb + n] (b_trans = 1).
//
// What bounds it: the fp32 matrix rate (64 flop per clock and SIMD, a sixteenth of bf16's) where there are tiles
// enough for every CU, and otherwise the latency of a chain of loads and the last round of tiles.  Three kernels:
//
// * gemm_f32_lds_kernel, 64 x 64 or 64 x 32 output tiles: four waves (2 x 2) share the tile's operands through LDS,
//   two stages of 32 k filled by direct-to-LDS loads (whole 128-byte lines), a stage's loads in flight during the
//   previous stage's products.  KG groups of four waves take a contiguous 1/KG of the k steps each, so that a CU
//   with one tile still has KG waves per SIMD.
// * gemm_f32_kernel, 32 x 32 tiles: a wave owns the tile for a range of k and loads its MFMA operands straight into
//   registers (nothing is shared, so LDS would add a round trip); WK waves share a tile.  For products of a few
//   tiles, and for operands that are not 16-byte aligned or whose edges cut a 16-byte piece.
// * gemm_f32_staged_kernel, 64 x 64 tiles staged through registers and LDS: for many tiles of operands that the
//   direct loads do not take (not 16-byte aligned, a 16-byte piece cut by an edge, 4 GiB and more); the register tiles
//   load each element twice as often.
//
// In the first two, the k ranges of a tile are added through LDS in order: deterministic, no atomics, no workspace.
//
// MFMA operands of a 16-k chunk for lane (r, g): rows MB r + i (i < MB) of the wave's 16 MB, k = 4 g + s of product
// s (s < 4).  A k-contiguous operand supplies them as one 16-byte piece per i, an m/n-contiguous one as one piece of
// MB consecutive rows per s.  So lane (r, g) accumulates C[MB (4 g + e) + i][NB r + j] in acc[i][j][e]: NB
// consecutive columns per store.
//
// With a_rowsum, the waves of the first tile column also add their A operands over k (the bias gradient of a
// weight-gradient product dyᵀ x), in a fixed order.
//
// Measured (MI355X; before: 64 x 64 tiles, one 16-k step loaded, stored to LDS and multiplied at a time):
//   4096 x 3072 x 1024, x Wᵀ     201 us, 128 TFLOP/s (the library's fp32 product of 8192 cubed runs at 153)
//   1000 x 4736 x 1408, x Wᵀ     117 us, 113 TFLOP/s; 1000 x 1408 x 4736, dy W: 131 us, 102 TFLOP/s
//   1000 x 1408 x 1408            43 us, 92 TFLOP/s; 4736 x 1408 x 1000, dyᵀ x: 112 us, 118 TFLOP/s
//   the twelve products of a 0.55b block's training pass over 1000 tokens: 1302 us a pass before, 605 now
#include <algorithm>

#include "llattn_abi.h"
#include "llattn_device.h"

namespace llattn {
namespace {

constexpr int FK = 16;  // k per chunk

struct GemmF32Args {
  int M, N, K, tiles_m, tiles_n, accumulate;
  int vec_a, vec_b, vec_c;  // 16-byte aligned with ld a multiple of 4
  const float* A;
  int64_t lda, a_bytes;
  const float* B;
  int64_t ldb, b_bytes;
  float* C;
  int64_t ldc;
  const float* bias;
  float* rowsum;
};

template <int N> struct FVec { typedef float type __attribute__((ext_vector_type(N))); };

// One operand's rows [o0, o0 + 16 MB) for this lane; KC: k-contiguous.
template <bool KC, int MB>
struct Operand {
  typedef typename FVec<MB>::type vec_t;
  const float* p[KC ? MB : 1];  // row MB r + i at k = 4 g; or k = 4 g of the row group MB r
  const float* base;
  int64_t ld;
  int o0, O, K, kq, row;  // kq: 4 g; row: o0 + MB r
  bool vec, cut;

  __device__ __forceinline__ void init(const float* b, int64_t l, int o, int Oo, int Kk, int r, int g, int v) {
    base = b; ld = l; o0 = o; O = Oo; K = Kk; kq = 4 * g; row = o + MB * r; vec = v != 0;
    cut = !KC && o + 16 * MB > Oo && Oo % MB != 0;
    if constexpr (KC) {
#pragma unroll
      for (int i = 0; i < MB; ++i) p[i] = base + (int64_t)min(row + i, O - 1) * ld + kq;
    } else {
      p[0] = base + (int64_t)kq * ld + min(row, (O - 1) / MB * MB);
    }
  }
  // chunk k0 can be loaded by vectors that stay inside the matrix (wave-uniform)
  __device__ __forceinline__ bool whole(int k0) const { return vec && k0 + FK <= K && !(cut && k0 + FK >= K); }
  // f[s][i]: row MB r + i at k = k0 + 4 g + s
  __device__ __forceinline__ void load(float (&f)[4][MB], int k0) const {
    if constexpr (KC) {
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(p[i] + k0);
#pragma unroll
        for (int s = 0; s < 4; ++s) f[s][i] = x[s];
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const vec_t x = *reinterpret_cast<const vec_t*>(p[0] + (int64_t)(k0 + s) * ld);
#pragma unroll
        for (int i = 0; i < MB; ++i) f[s][i] = x[i];
      }
    }
  }
  // the same element by element, zero past the matrix
  __device__ __forceinline__ void load_checked(float (&f)[4][MB], int k0) const {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int k = k0 + kq + s, o = row + i;
        f[s][i] = (k < K && o < O) ? base[KC ? (int64_t)o * ld + k : (int64_t)k * ld + o] : 0.f;
      }
  }
};

// C[m][n .. n + MB) = v (+ bias) (+ C); columns past N are not stored
template <int MB>
__device__ __forceinline__ void store_row(const GemmF32Args& a, int m, int n, typename FVec<MB>::type v) {
  typedef typename FVec<MB>::type vec_t;
  float* c = a.C + (int64_t)m * a.ldc + n;
  if (a.vec_c && n + MB <= a.N) {
    if (a.bias) {
#pragma unroll
      for (int j = 0; j < MB; ++j) v[j] += a.bias[n + j];
    }
    if (a.accumulate) v = *reinterpret_cast<const vec_t*>(c) + v;
    *reinterpret_cast<vec_t*>(c) = v;
  } else {
#pragma unroll
    for (int j = 0; j < MB; ++j)
      if (n + j < a.N) {
        const float x = v[j] + (a.bias ? a.bias[n + j] : 0.f);
        c[j] = a.accumulate ? c[j] + x : x;
      }
  }
}

// Rows past M / N are clamped to a valid row or pair of rows (their outputs are never stored).
template <bool AK, bool BKM, int WK>
__global__ __launch_bounds__(64 * WK) void gemm_f32_kernel(const GemmF32Args a) {
  constexpr int MB = 2;
  typedef typename FVec<MB>::type vec_t;
  constexpr int T = 16 * MB, ROWS = 4 * MB;  // tile; (i, e) rows of MB columns that a lane holds
  __shared__ __align__(16) vec_t red[WK > 1 ? WK : 1][WK > 1 ? ROWS : 1][64];
  __shared__ float rsl[WK][T];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // tile: contiguous ranges per XCD, then groups of 8 tile rows (their operand panels meet in one L2)
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  constexpr int GM = 8;
  const int group = t / (GM * a.tiles_n), first_m = group * GM, gm = min(a.tiles_m - first_m, GM);
  const int m0 = (first_m + (t % (GM * a.tiles_n)) % gm) * T, n0 = (t % (GM * a.tiles_n)) / gm * T;
  const bool rs = a.rowsum != nullptr && n0 == 0;  // workgroup-uniform
  const int chunks = (a.K + FK - 1) / FK, c0 = wave * chunks / WK, c1 = (wave + 1) * chunks / WK;

  Operand<AK, MB> A;
  Operand<BKM, MB> B;
  A.init(a.A, a.lda, m0, a.M, a.K, r, g, a.vec_a);
  B.init(a.B, a.ldb, n0, a.N, a.K, r, g, a.vec_b);
  f32x4 acc[MB][MB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float rsum[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) rsum[i] = 0.f;
  auto products = [&](const float (&fa)[4][MB], const float (&fb)[4][MB]) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[s][i], fb[s][j], acc[i][j], 0, 0, 0);
    if (rs) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < MB; ++i) rsum[i] += fa[s][i];
    }
  };
  // Whole chunks first: two register sets, the next chunk's loads in flight during this one's products.  Every
  // step issues the same loads (past the last whole chunk that one again, unused), so the waits for a set are
  // exact counts: with the loads under a condition the compiler waited for all of them before each set's products.
  float fa0[4][MB], fb0[4][MB];
  int cw = c1;  // chunks [c0, cw) are whole in both operands
  if (!A.vec || !B.vec) cw = c0;
  else if (c1 > c0 && !(A.whole((c1 - 1) * FK) && B.whole((c1 - 1) * FK))) cw = c1 - 1;
  if (c0 < cw) {
    float fa1[4][MB], fb1[4][MB];
    A.load(fa0, c0 * FK);
    B.load(fb0, c0 * FK);
    int c = c0;
    for (; c + 1 < cw; c += 2) {
      A.load(fa1, (c + 1) * FK);
      B.load(fb1, (c + 1) * FK);
      __builtin_amdgcn_sched_barrier(0);
      products(fa0, fb0);
      __builtin_amdgcn_sched_barrier(0);
      const int cn = min(c + 2, cw - 1);
      A.load(fa0, cn * FK);
      B.load(fb0, cn * FK);
      __builtin_amdgcn_sched_barrier(0);
      products(fa1, fb1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (c < cw) products(fa0, fb0);
  }
  for (int c = cw; c < c1; ++c) {
    A.load_checked(fa0, c * FK);
    B.load_checked(fb0, c * FK);
    products(fa0, fb0);
  }

  if (rs) {  // the four lane groups hold k = 4 g + s of every chunk
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      float v = rsum[i];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (g == 0) rsl[wave][MB * r + i] = v;
    }
  }
  auto store = [&](int q, vec_t v) {  // q = 4 i + e
    const int m = m0 + MB * (4 * g + (q & 3)) + (q >> 2);
    if (m < a.M) store_row<MB>(a, m, n0 + MB * r, v);
  };
  auto own = [&](int q) {
    vec_t v;
#pragma unroll
    for (int j = 0; j < MB; ++j) v[j] = acc[q >> 2][j][q & 3];
    return v;
  };
  if constexpr (WK == 1) {
    __syncthreads();  // rsl
#pragma unroll
    for (int q = 0; q < ROWS; ++q) store(q, own(q));
  } else {
#pragma unroll
    for (int q = 0; q < ROWS; ++q) red[wave][q][lane] = own(q);
    __syncthreads();
    constexpr int PER = ROWS / WK;  // each wave adds and stores ROWS / WK of the rows
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int q = wave * PER + u;
      vec_t v = red[0][q][lane];
#pragma unroll
      for (int w = 1; w < WK; ++w) v += red[w][q][lane];
      store(q, v);
    }
  }
  if (rs && threadIdx.x < T && m0 + (int)threadIdx.x < a.M) {
    float v = rsl[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < WK; ++w) v += rsl[w][threadIdx.x];
    a.rowsum[m0 + threadIdx.x] = v;
  }
}

// ---- tiles shared by four waves through LDS -----------------------------------------------------------------
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int SK = 32;  // k per LDS stage

// One wave copies 64 x 16 bytes into the 1 KB LDS block at dst (lane i at dst + 16 i); a lane whose offset lies past
// the descriptor's extent reads zero.  Inline asm: the compiler must not see an LDS write in flight, or it would
// wait for it before every LDS read (the stage read and the stage written are different ones); the main loop waits
// itself before the barrier that publishes a stage.
__device__ __forceinline__ void dma_block(const i32x4& rs, uint32_t off, const unsigned char* dst) {
  const i32x4 srs = {__builtin_amdgcn_readfirstlane(rs[0]), __builtin_amdgcn_readfirstlane(rs[1]),
                     __builtin_amdgcn_readfirstlane(rs[2]), __builtin_amdgcn_readfirstlane(rs[3])};
  const uint32_t sdst = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)dst);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
               :
               : "v"(off), "s"(srs), "s"(sdst)
               : "memory", "m0");
}
constexpr int kWaitAll = 0x0070;        // vmcnt(0) lgkmcnt(0)
constexpr uint32_t kPast = 0xFFFFFFF0u;  // past every extent (operands are below 4 GiB - 16 bytes): reads zero

// An operand's tile of O rows x 32 k per stage.  k-contiguous: rows of 128 bytes, 16-byte chunk c (4 k) of row o at
// slot c ^ ((o >> 2) & 7); m/n-contiguous: 32 k-rows of 4 O bytes.
template <bool KC, int MB>
struct Tile {
  static constexpr int O = 32 * MB, BYTES = O * SK * 4, NB = BYTES / 1024 / 4;  // NB: DMA blocks per wave
  uint32_t off[NB];
  int kc[NB];
  const float* base;
  int64_t ld, bytes;
  __device__ __forceinline__ void init(const float* b, int64_t l, int64_t by, int o0, int omax, int w4, int lane) {
    base = b; ld = l; bytes = by;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int bi = w4 * NB + i;
      if constexpr (KC) {
        const int row = 8 * bi + (lane >> 3), c = (lane & 7) ^ ((row / MB) & 7);
        off[i] = (uint32_t)(((int64_t)min(o0 + row, omax - 1) * ld + 4 * c) * 4);
        kc[i] = 4 * c;
      } else {
        constexpr int PER = O / 4;  // 16-byte pieces of a k-row
        const int q = bi * 64 + lane, k = q / PER, c = q % PER;
        off[i] = (uint32_t)(((int64_t)k * ld + min(o0 + 4 * c, omax - 4)) * 4);
        kc[i] = 0;
      }
    }
  }
  __device__ __forceinline__ i32x4 rsrc(int k0) const {
    const int64_t skip = (KC ? (int64_t)k0 : (int64_t)k0 * ld) * 4;
    const uint64_t addr = reinterpret_cast<uint64_t>(base) + (uint64_t)skip;
    const int64_t ext = bytes > skip ? bytes - skip : 0;
    return i32x4{(int)(uint32_t)addr, (int)((addr >> 32) & 0xffff), (int)(uint32_t)ext, 0x00020000};
  }
  // block i of this wave for a step; klim = K - k0 of the step: chunks that start at or past K read zero
  __device__ __forceinline__ void dma(const i32x4& rs, unsigned char* st, int w4, int i, int klim) const {
    dma_block(rs, (KC && kc[i] >= klim) ? kPast : off[i], st + (w4 * NB + i) * 1024);
  }
  // operands of a 16-k sub-step h: v[i] holds k = 4 g + s (k-contiguous), v[s] the rows MB r + i (m/n-contiguous)
  typedef typename FVec<KC ? 4 : MB>::type frag_t;
  static constexpr int NF = KC ? MB : 4;
  static __device__ __forceinline__ frag_t frag(const unsigned char* st, int o16, int r, int g, int h, int f) {
    if constexpr (KC) {
      const int row = o16 + MB * r + f;
      return *reinterpret_cast<const frag_t*>(st + row * 128 + (((4 * h + g) ^ ((row / MB) & 7)) << 4));
    } else {
      return *reinterpret_cast<const frag_t*>(st + ((16 * h + 4 * g + f) * O + o16 + MB * r) * 4);
    }
  }
  static __device__ __forceinline__ float at(const frag_t (&v)[NF], int s, int i) {
    if constexpr (KC) return v[i][s];
    else return v[s][i];
  }
};

template <bool AK, bool BKM, int MB, int NB, int KG>
__global__ __launch_bounds__(256 * KG) void gemm_f32_lds_kernel(const GemmF32Args a) {
  typedef Tile<AK, MB> TA;
  typedef Tile<BKM, NB> TB;
  typedef typename FVec<NB>::type vec_t;
  constexpr int T = 32 * MB, TN = 32 * NB, ROWS = 4 * MB, STAGE = TA::BYTES + TB::BYTES;
  __shared__ __align__(1024) unsigned char smem[KG * 2 * STAGE];
  __shared__ float rsl[KG][T];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w4 = wave & 3, kg = wave >> 2;
  const int wm = w4 >> 1, wn = w4 & 1;
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  constexpr int GM = 8;
  const int group = t / (GM * a.tiles_n), first_m = group * GM, gm = min(a.tiles_m - first_m, GM);
  const int m0 = (first_m + (t % (GM * a.tiles_n)) % gm) * T, n0 = (t % (GM * a.tiles_n)) / gm * TN;
  const bool rs = a.rowsum != nullptr && n0 == 0 && wn == 0;  // wave-uniform
  // every k group runs the same number of steps; those past K read zeros
  const int steps = (a.K + SK - 1) / SK, nk = (steps + KG - 1) / KG, kbeg = kg * nk * SK;
  unsigned char* sm = smem + kg * 2 * STAGE;

  TA ta;
  TB tb;
  ta.init(a.A, a.lda, a.a_bytes, m0, a.M, w4, lane);
  tb.init(a.B, a.ldb, a.b_bytes, n0, a.N, w4, lane);
  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float rsum[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) rsum[i] = 0.f;
  typename TA::frag_t fa[2][TA::NF];
  typename TB::frag_t fb[2][TB::NF];
  auto read = [&](int set, int stage, int h) {
    const unsigned char* st = sm + stage * STAGE;
#pragma unroll
    for (int f = 0; f < TA::NF; ++f) fa[set][f] = TA::frag(st, wm * 16 * MB, r, g, h, f);
#pragma unroll
    for (int f = 0; f < TB::NF; ++f) fb[set][f] = TB::frag(st + TA::BYTES, wn * 16 * NB, r, g, h, f);
  };
  auto products = [&](int set) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(TA::at(fa[set], s, i), TB::at(fb[set], s, j), acc[i][j], 0, 0, 0);
    if (rs) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < MB; ++i) rsum[i] += TA::at(fa[set], s, i);
    }
  };
  auto fetch = [&](int stage, int kt) {
    const int k0 = kbeg + min(kt, nk - 1) * SK, klim = a.K - k0;
    const i32x4 ra = ta.rsrc(k0), rb = tb.rsrc(k0);
    unsigned char* st = sm + stage * STAGE;
#pragma unroll
    for (int i = 0; i < TA::NB; ++i) ta.dma(ra, st, w4, i, klim);
#pragma unroll
    for (int i = 0; i < TB::NB; ++i) tb.dma(rb, st + TA::BYTES, w4, i, klim);
  };
  fetch(0, 0);
  __builtin_amdgcn_s_waitcnt(kWaitAll);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  fetch(1, 1);
  read(0, 0, 0);
  for (int kt = 0; kt < nk; ++kt) {
    const int s = kt & 1;
    __builtin_amdgcn_sched_barrier(0);
    read(1, s, 1);
    products(0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitAll);  // this wave's DMA of step kt + 1 and its reads of step kt
    __builtin_amdgcn_s_barrier();          // every wave's: step kt + 1 is readable, step kt's stage free
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    read(0, s ^ 1, 0);
    fetch(s, kt + 2);
    products(1);
  }
  __builtin_amdgcn_s_waitcnt(kWaitAll);  // no DMA in flight past this point
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  if (rs) {
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      float v = rsum[i];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (g == 0) rsl[kg][wm * 16 * MB + MB * r + i] = v;
    }
  }
  auto store = [&](int q, vec_t v) {  // q = 4 i + e
    const int m = m0 + wm * 16 * MB + MB * (4 * g + (q & 3)) + (q >> 2), n = n0 + wn * 16 * NB + NB * r;
    if (m < a.M) store_row<NB>(a, m, n, v);
  };
  auto own = [&](int q) {
    vec_t v;
#pragma unroll
    for (int j = 0; j < NB; ++j) v[j] = acc[q >> 2][j][q & 3];
    return v;
  };
  if constexpr (KG == 1) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < ROWS; ++q) store(q, own(q));
  } else {
    vec_t* red = reinterpret_cast<vec_t*>(smem);  // [KG][4 waves][ROWS][64]
#pragma unroll
    for (int q = 0; q < ROWS; ++q) red[(wave * ROWS + q) * 64 + lane] = own(q);
    __syncthreads();
    constexpr int PER = ROWS / KG;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int q = kg * PER + u;
      vec_t v = red[(w4 * ROWS + q) * 64 + lane];
#pragma unroll
      for (int w = 1; w < KG; ++w) v += red[((4 * w + w4) * ROWS + q) * 64 + lane];
      store(q, v);
    }
  }
  if (a.rowsum && n0 == 0 && threadIdx.x < T && m0 + (int)threadIdx.x < a.M) {
    float v = rsl[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < KG; ++w) v += rsl[w][threadIdx.x];
    a.rowsum[m0 + threadIdx.x] = v;
  }
}

// ---- staged tiles: operands that the direct-to-LDS loads do not take ----------------------------------------
constexpr int ST = 64, SP = ST + 4;  // tile, padded LDS row (floats)

// 4 elements of a 64 x 16 operand tile into the k-major LDS tile s[k][o]: thread t takes row o = t / 4 and
// k = 4 (t % 4) .. + 3 of k-contiguous storage, else k = t / 16 and o = 4 (t % 16) .. + 3.  Zero past the matrix.
// (The layout as an argument: as a template parameter of the kernel it took 5% longer.)
__device__ __forceinline__ void stage_tile(const float* __restrict__ p, int64_t ld, bool kc, int o0, int k0, int O, int K,
                                           int t, float (*s)[SP]) {
  float v[4];
  if (kc) {
    const int o = t >> 2, k = 4 * (t & 3), go = o0 + o, gk = k0 + k;
    const float* q = p + (int64_t)go * ld + gk;
    if (go < O && gk + 3 < K && ((uintptr_t)q & 15) == 0) {
      const float4 x = *reinterpret_cast<const float4*>(q);
      v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (go < O && gk + e < K) ? q[e] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s[k + e][o] = v[e];
  } else {
    const int o = 4 * (t & 15), k = t >> 4, go = o0 + o, gk = k0 + k;
    const float* q = p + (int64_t)gk * ld + go;
    if (gk < K && go + 3 < O && ((uintptr_t)q & 15) == 0) {
      const float4 x = *reinterpret_cast<const float4*>(q);
      v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (gk < K && go + e < O) ? q[e] : 0.f;
    }
    *reinterpret_cast<float4*>(&s[k][o]) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

// Four waves of 32 x 32 (2 x 2); a 16-k chunk is staged and multiplied at a time.
__global__ __launch_bounds__(256) void gemm_f32_staged_kernel(const GemmF32Args a, int kc_a, int kc_b) {
  __shared__ __align__(16) float As[FK][SP];
  __shared__ __align__(16) float Bs[FK][SP];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = tid >> 6, wm = wave >> 1, wn = wave & 1;
  const int m0 = (blockIdx.x / a.tiles_n) * ST, n0 = (blockIdx.x % a.tiles_n) * ST;
  const bool rs = a.rowsum != nullptr && n0 == 0;  // workgroup-uniform
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float rsum = 0.f;  // rs: thread t < 64 sums row m0 + t of A over k
  for (int k0 = 0; k0 < a.K; k0 += FK) {
    stage_tile(a.A, a.lda, kc_a, m0, k0, a.M, a.K, tid, As);
    stage_tile(a.B, a.ldb, kc_b, n0, k0, a.N, a.K, tid, Bs);
    __syncthreads();
    if (rs && tid < ST) {
#pragma unroll
      for (int k = 0; k < FK; ++k) rsum += As[k][tid];
    }
#pragma unroll
    for (int kk = 0; kk < FK; kk += 4) {  // lane (r, g) supplies A[m = r][k = g] and B[n = r][k = g]
      float av[2], bv[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) av[i] = As[kk + g][wm * 32 + 16 * i + r];
#pragma unroll
      for (int j = 0; j < 2; ++j) bv[j] = Bs[kk + g][wn * 32 + 16 * j + r];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)  // lane (r, g) holds C[m = 16 i + 4 g + e][n = 16 j + r] of the wave's block
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm * 32 + 16 * i + 4 * g + e, n = n0 + wn * 32 + 16 * j + r;
        if (m >= a.M || n >= a.N) continue;
        float* c = a.C + (int64_t)m * a.ldc + n;
        const float v = acc[i][j][e] + (a.bias ? a.bias[n] : 0.f);
        *c = a.accumulate ? *c + v : v;
      }
  if (rs && tid < ST && m0 + tid < a.M) a.rowsum[m0 + tid] = rsum;
}

// Kernel, tile and k split: the least of a time model in us, fitted to a sweep of 20 products (16 x 64 x 256 to
// 4096 x 3072 x 1024, each layout; within 15% of the best configuration on all of them).
//   LDS tiles: rounds of tiles over 256 CUs at 256 flop per clock and CU and 2.25 GHz, times the share that a round
//   really takes (a CU with one tile has fewer waves to hide a barrier behind; 1000 x 4736 x 1408, 1184 tiles of
//   64 x 64, 5 rounds: 117 us against 100), plus 3 us to fill and drain.
//   32 x 32 register tiles: a chunk of 16 k takes 0.28 us of load latency with one chunk ahead, or 0.45 us per wave
//   that shares the SIMD (twice the operand bytes of a 64 x 64 tile: 1000 x 4736 x 1408 takes 186 us), plus 2 us.
//   Operands that are not 16-byte aligned: the register tiles load by the element, 2.8 times as long.
//   Staged tiles: 1.3 us per chunk of 16 k (1.7 by the element), or 0.40 (0.62) us per tile of a CU where that is more,
//   plus 3 us.  Measured, register against staged tiles, in rows padded to 16 bytes: 1000 x 1409 x 1409 65 against
//   120 us, 20000 x 1025 x 255 167 against 121, 1 200 000 x 1024 x 1024 (4.9 GB) 37.0 against 22.3 ms; by the element:
//   333 x 1409 x 1407 62 against 147, 1000 x 1409 x 1409 177 against 155, 4096 x 3073 x 1025 1020 against 490.
struct F32Plan { int nb, k; };  // LDS tiles of 64 x 32 nb with k groups (0: staged); nb = 0: register tiles with k waves
F32Plan plan_f32(int M, int N, int K, bool lds_ok, bool aligned) {
  F32Plan best{0, 1};
  double best_t = 1e30;
  const auto take = [&](double t, int nb, int k) {
    if (t < best_t) {
      best_t = t;
      best = F32Plan{nb, k};
    }
  };
  const int chunks = (K + FK - 1) / FK;
  for (int wk : {1, 2, 4, 8}) {
    const int64_t tiles = (int64_t)((M + 31) / 32) * ((N + 31) / 32), per_simd = (tiles * wk + 1023) / 1024;
    if (wk > 1 && (chunks < 2 * wk || tiles * wk >= (int64_t(1) << 32) / 64)) break;  // a grid holds 2^32 threads
    take(((chunks + wk - 1) / wk) * std::max(0.28, 0.45 * (double)per_simd) * (aligned ? 1.0 : 2.8) + 2.0, 0, wk);
  }
  const int64_t staged = (int64_t)((M + ST - 1) / ST) * ((N + ST - 1) / ST);
  if (!lds_ok && staged < (int64_t(1) << 24))
    take(chunks * (aligned ? std::max(1.3, 0.40 * (double)staged / 256.0) : std::max(1.7, 0.62 * (double)staged / 256.0)) + 3.0, 2, 0);
  if (!lds_ok) return best;
  struct { int nb, kg; double one, more; } const opt[] = {{2, 1, 1.43, 1.18}, {2, 2, 1.28, 1.22}, {1, 2, 1.45, 1.31}, {1, 4, 1.35, 1.55}};
  for (const auto& o : opt) {
    const int64_t tiles = (int64_t)((M + 63) / 64) * ((N + 32 * o.nb - 1) / (32 * o.nb)), rounds = (tiles + 255) / 256;
    const double tile_us = 2.0 * 64 * 32 * o.nb * (double)((K + SK - 1) / SK * SK) / 256.0 / 2250.0;
    take((double)rounds * tile_us * (rounds == 1 ? o.one : o.more) + 3.0, o.nb, o.kg);
  }
  return best;
}

template <bool AK, bool BKM>
void launch_f32(const GemmF32Args& a, const F32Plan& p, hipStream_t st) {
  const dim3 grid(a.tiles_m * a.tiles_n);
  if (p.nb == 2) {
    if (p.k == 0) hipLaunchKernelGGL(gemm_f32_staged_kernel, grid, dim3(256), 0, st, a, AK, BKM);
    else if (p.k == 1) hipLaunchKernelGGL((gemm_f32_lds_kernel<AK, BKM, 2, 2, 1>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gemm_f32_lds_kernel<AK, BKM, 2, 2, 2>), grid, dim3(512), 0, st, a);
  } else if (p.nb == 1) {
    if (p.k == 2) hipLaunchKernelGGL((gemm_f32_lds_kernel<AK, BKM, 2, 1, 2>), grid, dim3(512), 0, st, a);
    else hipLaunchKernelGGL((gemm_f32_lds_kernel<AK, BKM, 2, 1, 4>), grid, dim3(1024), 0, st, a);
  } else if (p.k == 1) hipLaunchKernelGGL((gemm_f32_kernel<AK, BKM, 1>), grid, dim3(64), 0, st, a);
  else if (p.k == 2) hipLaunchKernelGGL((gemm_f32_kernel<AK, BKM, 2>), grid, dim3(128), 0, st, a);
  else if (p.k == 4) hipLaunchKernelGGL((gemm_f32_kernel<AK, BKM, 4>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((gemm_f32_kernel<AK, BKM, 8>), grid, dim3(512), 0, st, a);
}

}  // namespace
}  // namespace llattn

using namespace llattn;

extern "C" int32_t llattn_gemm_f32(const llattn_gemm_desc* d, void* stream) {
  if (!d) return fail(LLATTN_ERR_SHAPE, "llattn_gemm_f32: null descriptor");
  if (d->M <= 0 || d->N <= 0 || d->K <= 0)
    return fail(LLATTN_ERR_SHAPE, "llattn_gemm_f32: sizes must be positive (M=%d N=%d K=%d)", d->M, d->N, d->K);
  if (d->c_dtype != LLATTN_F32)
    return fail(LLATTN_ERR_DTYPE, "llattn_gemm_f32: fp32 C only (c_dtype %d)", d->c_dtype);
  if (d->split_k > 1 || d->rowadd[0].ptr || d->rowadd[1].ptr || d->act != LLATTN_ACT_NONE || d->c_heads.T != 0)
    return fail(LLATTN_ERR_UNSUPPORTED, "llattn_gemm_f32: no K split, row addends, activation or split-head C");
  if (!d->A || !d->B || !d->C || (uintptr_t)d->A % 4 || (uintptr_t)d->B % 4 || (uintptr_t)d->C % 4 ||
      (d->bias && (uintptr_t)d->bias % 4) || (d->a_rowsum && (uintptr_t)d->a_rowsum % 4))
    return fail(LLATTN_ERR_LAYOUT, "llattn_gemm_f32: operands must be non-null and 4-byte aligned");
  if (d->lda < (d->a_trans ? d->M : d->K) || d->ldb < (d->b_trans ? d->N : d->K) || d->ldc < d->N)
    return fail(LLATTN_ERR_LAYOUT, "llattn_gemm_f32: leading dimensions smaller than the rows they hold");
  const int64_t a_bytes = (d->a_trans ? (int64_t)(d->K - 1) * d->lda + d->M : (int64_t)(d->M - 1) * d->lda + d->K) * 4;
  const int64_t b_bytes = (d->b_trans ? (int64_t)(d->K - 1) * d->ldb + d->N : (int64_t)(d->N - 1) * d->ldb + d->K) * 4;
  const auto vec = [](const void* p, int64_t ld) { return (int)(aligned16(p) && ld % 4 == 0); };
  // the LDS kernel moves 16-byte pieces by 32-bit offsets: none may straddle the end of a contiguous dimension, and
  // the rows of a stage that lie past K must be past the extent, not wrapped around into it (SK ld 4 < 2^32)
  const auto span = [](int32_t trans, int64_t ld) { return !trans || ld < (int64_t(1) << 32) / (4 * SK); };
  const bool lds_ok = vec(d->A, d->lda) && vec(d->B, d->ldb) && (d->a_trans ? d->M : d->K) % 4 == 0 &&
                      (d->b_trans ? d->N : d->K) % 4 == 0 && span(d->a_trans, d->lda) && span(d->b_trans, d->ldb) &&
                      a_bytes <= (int64_t)kPast && b_bytes <= (int64_t)kPast;
  const F32Plan plan = plan_f32(d->M, d->N, d->K, lds_ok, vec(d->A, d->lda) && vec(d->B, d->ldb));
  const int TM = plan.nb ? 64 : 32, TN = plan.nb ? 32 * plan.nb : 32;
  const int64_t tiles = (int64_t)((d->M + TM - 1) / TM) * ((d->N + TN - 1) / TN);
  if (tiles > 0x7fffffff) return fail(LLATTN_ERR_UNSUPPORTED, "llattn_gemm_f32: too many output tiles");
  GemmF32Args a{};
  a.M = d->M; a.N = d->N; a.K = d->K;
  a.tiles_m = (d->M + TM - 1) / TM; a.tiles_n = (d->N + TN - 1) / TN;
  a.accumulate = d->accumulate;
  a.A = static_cast<const float*>(d->A); a.lda = d->lda; a.a_bytes = a_bytes; a.vec_a = vec(d->A, d->lda);
  a.B = static_cast<const float*>(d->B); a.ldb = d->ldb; a.b_bytes = b_bytes; a.vec_b = vec(d->B, d->ldb);
  a.C = static_cast<float*>(d->C); a.ldc = d->ldc; a.vec_c = vec(d->C, d->ldc);
  a.bias = d->bias;
  a.rowsum = d->a_rowsum;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (!d->a_trans && !d->b_trans) launch_f32<true, true>(a, plan, st);
  else if (!d->a_trans) launch_f32<true, false>(a, plan, st);
  else if (d->b_trans) launch_f32<false, false>(a, plan, st);
  else launch_f32<false, true>(a, plan, st);
  return check_launch("llattn_gemm_f32");
}
