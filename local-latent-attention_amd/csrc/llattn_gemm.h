// What the bf16 GEMM kernels share (llattn_gemm.hip: 256 x 256 tiles; llattn_gemm_tile.hip: smaller ones): the
// launch arguments, the epilogue arithmetic, direct-to-LDS loads and the fragment reads of 64-k LDS stages.
#pragma once

#include <type_traits>

#include "llattn_abi.h"
#include "llattn_device.h"
#include "llattn_heads.h"

namespace llattn {
namespace gemm {

constexpr int BM = 256, BN = 256;  // output tile

enum Epi { EPI_BF16 = 0, EPI_F32 = 1, EPI_PART = 2 };

struct GemmArgs {
  int M, N, K, k_pairs, n_split, tiles_m, tiles_n, accumulate;  // k_pairs: 64-wide k steps, ceil(K / 64)
  const uint16_t* A; int64_t lda, a_bytes;
  const uint16_t* B; int64_t ldb, b_bytes;
  void* C; int64_t ldc;
  const float* bias;
  float* part;     // split-K partials [S][M][N], then (rowsum) [S][M]
  float* rowsum;   // fp32 [M] or null: sum_k A(m, k), from a column of ones in place of B's column N or summed beside the products
  // bf16 C only: C[m][n] += ra[(m / T) * n_seg + (m % T) / seg][n] / divisor for each of up to two addends
  const uint16_t* ra_ptr[2];
  int64_t ra_ld[2];
  int ra_T[2], ra_seg[2], ra_nseg[2], ra_div[2];
  // bf16 C only: LLATTN_ACT_GELU writes C = gelu(pre), aux = gelu'(pre); LLATTN_ACT_MUL_AUX scales C by aux
  int act;
  uint16_t* aux;
  int64_t ld_aux;
  HeadsMap ch;  // bf16 C stored split-head (ch.T > 0): the persistent kernel, the smaller tiles and their reduction
};

// Exact GELU u * Phi(u) of the reference FeedForward (reference models.py:57, F.gelu) and its derivative
// Phi(u) + u phi(u), in fp32.  erf comes from Abramowitz & Stegun 7.1.26 (Handbook of Mathematical
// Functions): erf(z) = 1 - t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) exp(-z^2), t = 1 / (1 + p z), z >= 0,
// absolute error below 1.5e-7 (far under the bf16 rounding of the outputs).  With z = |u| / sqrt(2),
// exp(-z^2) = exp(-u^2 / 2) is also the Gaussian density's exponential, so Phi and phi share one exp:
//   q = t P(t) exp(-u^2/2) / 2,  Phi(u) = 1 - q (u >= 0) or q (u < 0),  phi(u) = exp(-u^2/2) / sqrt(2 pi).
struct NormalCdf {
  float cdf, pdf;
};
__device__ __forceinline__ NormalCdf normal_cdf_pdf(float u) {
  constexpr float p = 0.3275911f, a1 = 0.254829592f, a2 = -0.284496736f, a3 = 1.421413741f,
                  a4 = -1.453152027f, a5 = 1.061405429f;
  const float z = fabsf(u) * 0.70710678118654752f;
  const float t = __builtin_amdgcn_rcpf(fmaf(p, z, 1.f));
  const float poly = t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, a5, a4), a3), a2), a1);
  const float e = __builtin_amdgcn_exp2f(-0.5f * 1.4426950408889634f * u * u);  // exp(-u^2 / 2)
  const float q = 0.5f * poly * e;
  return NormalCdf{u >= 0.f ? 1.f - q : q, e * 0.39894228040143268f};
}
// gelu(u) and gelu'(u) of one value
__device__ __forceinline__ void gelu_pair(float u, float& g, float& gp) {
  const NormalCdf n = normal_cdf_pdf(u);
  g = u * n.cdf;
  gp = fmaf(u, n.pdf, n.cdf);
}
// Eight bf16 pre-activations (packed pairs; the activation acts on the bf16-rounded value, as bf16
// autocast does) -> gelu and gelu' as bf16.
__device__ __forceinline__ void gelu_bf16x8(uint4 x, uint4& g, uint4& gp) {
  const uint32_t xs[4] = {x.x, x.y, x.z, x.w};
  uint32_t o[4], d[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float g0, g1, p0, p1;
    gelu_pair(__uint_as_float(xs[e] << 16), g0, p0);
    gelu_pair(__uint_as_float(xs[e] & 0xffff0000u), g1, p1);
    o[e] = pack_bf16x2(g0, g1);
    d[e] = pack_bf16x2(p0, p1);
  }
  g = make_uint4(o[0], o[1], o[2], o[3]);
  gp = make_uint4(d[0], d[1], d[2], d[3]);
}
// bf16 x * s elementwise (eight packed values each)
__device__ __forceinline__ uint4 mul_bf16x8(uint4 x, uint4 s) {
  const uint32_t xs[4] = {x.x, x.y, x.z, x.w}, ss[4] = {s.x, s.y, s.z, s.w};
  uint32_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = pack_bf16x2(__uint_as_float(xs[e] << 16) * __uint_as_float(ss[e] << 16),
                       __uint_as_float(xs[e] & 0xffff0000u) * __uint_as_float(ss[e] & 0xffff0000u));
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// Row of addend q (0, 1) that C row m reads, and its scale (the pooled gradient broadcast to its tokens).
__device__ __forceinline__ const uint16_t* rowadd_row(const GemmArgs& a, int q, int m, float& sc) {
  const int T = a.ra_T[q], t = m % T, s = t / a.ra_seg[q];
  sc = a.ra_div[q] == LLATTN_DIV_COUNT ? 1.f / (float)(min((s + 1) * a.ra_seg[q], T) - s * a.ra_seg[q])
     : a.ra_div[q] == LLATTN_DIV_SEG ? 1.f / (float)a.ra_seg[q] : 1.f;
  return a.ra_ptr[q] + ((int64_t)(m / T) * a.ra_nseg[q] + s) * a.ra_ld[q];
}
__device__ __forceinline__ void add_bf16x4(uint2 u, float sc, float (&v)[4]) {
  v[0] += sc * __uint_as_float(u.x << 16);
  v[1] += sc * __uint_as_float(u.x & 0xffff0000u);
  v[2] += sc * __uint_as_float(u.y << 16);
  v[3] += sc * __uint_as_float(u.y & 0xffff0000u);
}
__device__ __forceinline__ void rowadd4(const GemmArgs& a, int q, int m, int c, float (&v)[4]) {
  float sc;
  const uint16_t* p = rowadd_row(a, q, m, sc);
  add_bf16x4(*reinterpret_cast<const uint2*>(p + c), sc, v);
}

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void gbl_void;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

typedef int i32x4 __attribute__((ext_vector_type(4)));

// LDS byte address of a pointer into shared memory
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

constexpr int kRsrcWord3 = 0x00020000;  // raw buffer, gfx9 family

// One wave copies 64 x 16 bytes from global memory into the 1 KB LDS block at
// `dst` (lane i lands at dst + 16 i) with buffer_load_dwordx4 ... lds: the
// step's base address lives in the scalar buffer descriptor and each lane
// adds its fixed 32-bit offset.  Offsets past the descriptor's extent read 0.
// Written as inline asm so that the compiler does not see an LDS write in
// flight: it would otherwise make every later LDS read wait for all of it
// (vmcnt(0)), although the reads target another stage.  The main loop waits
// for these loads itself (vmcnt) before the barrier that publishes them.
// The descriptor and the LDS address are wave-uniform at every call; readfirstlane states it for the
// cases where the compiler cannot prove it (it then keeps them in SGPRs, as the instruction requires).
__device__ __forceinline__ void dma_block(const i32x4& rs, uint32_t off, const unsigned char* dst) {
  const i32x4 srs = {__builtin_amdgcn_readfirstlane(rs[0]), __builtin_amdgcn_readfirstlane(rs[1]),
                     __builtin_amdgcn_readfirstlane(rs[2]), __builtin_amdgcn_readfirstlane(rs[3])};
  const uint32_t sdst = __builtin_amdgcn_readfirstlane(lds_addr(dst));
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
               :
               : "v"(off), "s"(srs), "s"(sdst)
               : "memory", "m0");
}

// s_waitcnt immediates (gfx9 encoding: vmcnt [3:0]+[15:14], expcnt [6:4], lgkmcnt [11:8]);
// issued through the builtin so that the compiler's own wait insertion sees them.
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0070 | 0x0F00; }       // vmcnt(n)
constexpr int wait_vm_lgkm0(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0070; }        // vmcnt(n) lgkmcnt(0)

// An offset past every operand extent (operands are below 4 GiB - 16 bytes): the lane reads zero.
constexpr uint32_t kOffPastK = 0xFFFFFFF0u;
// A lane's 32-bit offset within a step.  The rows of an m/n-contiguous stage that lie past K must read zero; with wide
// strides (64 ld 2 >= 2^32 bytes) their offsets pass 32 bits, and cut short they would fall inside the operand again.
__device__ __forceinline__ uint32_t step_off(int64_t bytes) { return (uint32_t)min(bytes, (int64_t)kOffPastK); }
// A k-contiguous lane's offset for a step whose K tail starts `klim` elements in, its chunk starting at kc.
__device__ __forceinline__ uint32_t kmask(uint32_t off, int kc, int klim) { return kc < klim ? off : kOffPastK; }

// Buffer descriptor of an operand from step k0 on (`bytes`: storage extent of the operand).
template <bool KMAJ>
__device__ __forceinline__ i32x4 step_rsrc(const uint16_t* base, int64_t ld, int64_t bytes, int k0) {
  const int64_t skip = (KMAJ ? (int64_t)k0 : (int64_t)k0 * ld) * 2;
  const uint64_t addr = reinterpret_cast<uint64_t>(base) + (uint64_t)skip;
  // a step wholly past K can start beyond a small operand's end: extent 0, every lane reads zero
  const int64_t ext = bytes > skip ? bytes - skip : 0;
  return i32x4{(int)(uint32_t)addr, (int)((addr >> 32) & 0xffff), (int)(uint32_t)ext, kRsrcWord3};
}

// 64-k LDS stages (two of 64 KB), shared by gemm_kernel and the persistent kernel.  k-contiguous tiles:
// 256 rows of 128 bytes, 16-byte chunk c of row r at slot c ^ pswz(r) (A fragments read rows o16 + r, eight
// consecutive rows per LDS cycle -> r & 7; permuted B fragments read rows o16 + 8 (r / 4) + r % 4 ->
// (r & 3) | (bit 3 of the row at bit 2); both conflict-free).  mn-contiguous tiles: 64 k-rows of 512 bytes,
// chunk c of k-row k at c ^ 2 (k & 3) (transposing reads, conflict-free).
constexpr int PBK = 64;                  // k per LDS stage
constexpr int PTILE = BM * PBK * 2;      // 32 KB per operand per stage
constexpr int PSTAGE = 2 * PTILE;        // A then B
constexpr int PDMA = PTILE / 1024 / 4;   // 1 KB DMA blocks per wave per operand and step (8)

template <bool PERM>
__device__ __forceinline__ int pswz(int row) {
  return PERM ? ((row & 3) | (((row >> 3) & 1) << 2)) : (row & 7);
}

// Byte offsets (relative to the operand base at the step's first k) of this lane's 16-byte chunk in each
// of the wave's 8 DMA blocks of a 64-k operand tile (rows / columns [o0, o0 + 256)).  k-contiguous: block i
// = rows 8 (8 wave + i) .. + 7, lane -> row + lane / 8, LDS slot lane % 8 receives the row's chunk
// (lane % 8) ^ pswz(row); rows past omax are clamped to a valid row (their outputs are never stored).
// mn-contiguous: block i = k-rows 2 (8 wave + i) + lane / 32, 32 chunks each; columns clamped likewise.
// kc: first k of the lane's chunk (k-contiguous K tail; mn-contiguous rows past K lie beyond the extent).
template <bool KMAJ, bool PERM = false>
__device__ __forceinline__ void tile_offsets64(uint32_t (&off)[PDMA], int (&kc)[PDMA], int64_t ld, int o0, int omax,
                                               int wave, int lane) {
#pragma unroll
  for (int i = 0; i < PDMA; ++i) {
    const int bi = wave * PDMA + i;
    if constexpr (KMAJ) {
      const int row = 8 * bi + (lane >> 3);
      const int c = (lane & 7) ^ pswz<PERM>(row);
      off[i] = (uint32_t)(((int64_t)min(o0 + row, omax - 1) * ld + 8 * c) * 2);
      kc[i] = 8 * c;
    } else {
      const int k = 2 * bi + (lane >> 5);
      const int c = (lane & 31) ^ (2 * (k & 3));
      off[i] = step_off(((int64_t)k * ld + min(o0 + 8 * c, omax - 8)) * 2);
      kc[i] = 0;
    }
  }
}

// 8 k values (32h + 8g .. + 7 of a 64-k stage) of tile row / column o16 + r for lane (r, g).  PERM
// (k-contiguous B only): lane r reads row o16 + 8 (r / 4) + r % 4 instead, so that with o16 = 32p + 4u the
// output columns a lane accumulates for the block pair (u = 0, 1) are 8 consecutive ones.
template <bool KMAJ, bool PERM = false>
__device__ __forceinline__ bf16x8 frag64(const unsigned char* tile, int o16, int r, int g, int h) {
  if constexpr (KMAJ) {
    const int row = PERM ? o16 + 8 * (r >> 2) + (r & 3) : o16 + r;
    return *reinterpret_cast<const bf16x8*>(tile + row * 128 + (((4 * h + g) ^ pswz<PERM>(row)) << 4));
  } else {
    // transposing reads: the 16 lanes of group g supply k-rows kb + j/4, 8 bytes at column o16 + 4(j%4);
    // lane r receives column o16 + r of those four rows
    const int kb = 32 * h + 8 * g;
    const int col = o16 + 4 * (r & 3), chunk = col >> 3, inner = (col & 7) << 1;
    bf16x4 hv[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int k = kb + 4 * half + (r >> 2);
      const unsigned char* p = tile + k * 512 + ((chunk ^ (2 * (k & 3))) << 4) + inner;
      hv[half] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(p));
    }
    return bf16x8{hv[0][0], hv[0][1], hv[0][2], hv[0][3], hv[1][0], hv[1][1], hv[1][2], hv[1][3]};
  }
}

// Number of K splits of a product on 256 x 256 tiles (llattn_gemm.hip).
int resolve_split(const llattn_gemm_desc* d);

// Tile (32 mb x 32 nb), k groups and k splits over workgroups of a product on the smaller tiles; mb = 0: not taken
// (llattn_gemm_tile.hip).
struct TilePlan { int mb, nb, kg, splits; };
TilePlan tile_plan(const llattn_gemm_desc* d, double* us = nullptr);  // us: the time it expects
void launch_tile(const GemmArgs& a, const TilePlan& p, bool a_kmaj, bool b_kmaj, int c_dtype, hipStream_t st);
// Two independent products in one launch: x Wᵀ or dy W into bf16, and then dyᵀ x into fp32 or (after x Wᵀ) another x Wᵀ.
TilePlan pair_plan(const llattn_gemm_desc* d0, const llattn_gemm_desc* d1);
void launch_pair(GemmArgs a0, GemmArgs a1, const TilePlan& p, bool b_kmaj0, bool weight1, hipStream_t st);

}  // namespace gemm
}  // namespace llattn
