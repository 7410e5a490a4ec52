// Whole steps of the attention block, its core and the feed-forward (include/llattn_steps.h): the launches of the
// single entry points in a row.  A training pass of the block is ~25 launches whose kernels take 5-50 us each at a
// few thousand tokens; issued one by one from Python (a call of 15-25 us each: argument structs, workspace queries,
// output tensors) the GPU waited for the host.  One call issues them in about 4 us each.  Measured (MI355X, a pass
// before -> with these calls; in brackets with the kernels for small products since): a 0.55b layer's forward over 333
// tokens 267 -> 100 us (57), its fwd + bwd over 3 x 1337 tokens (0.60b) 905 -> 640 us (574), the op at head dim 128 over
// 2 x 3001 tokens 488 -> 293 us (264 to 305, the host's; 53 us of it gradients laid out as their inputs, which autograd
// then need not copy), the 0.55b model over 1024 tokens 9.4 -> 4.9 ms (3.9).
//
// The sequences are those of the Python path (module.py, ops.py, linear.py, ffn.py: kept for profiling and for
// parameters this path does not take), product by product with the same operands and roundings.  Two products that do
// not depend on each other share a launch where that pays (llattn_gemm_pair); the k order of their sums can then differ
// from the single products', otherwise both paths give the same bits.
//
// Every step is one function run twice: by the size query with a null base, where buffers only count and launches
// only ask for their workspace, and by the call itself.  Scratch is a stack, and an output's buffer holds scratch until
// the output is written: a 0.55b layer's training pass over 32768 tokens peaks at 1402 MB (1595 with everything side by
// side, 1363 product by product), its forward alone at 505 (644, 570).
#include <algorithm>

#include "llattn_abi.h"
#include "llattn_pool.h"
#include "llattn_steps.h"

namespace llattn {
namespace {

constexpr size_t up(size_t n) { return (n + 255) & ~size_t(255); }

// Hands out 256-byte aligned pieces of a buffer as a stack; base null: only counts.  What was given back is handed out
// again: the launches of a step run in order on one stream.
struct Arena {
  char* base;
  size_t used = 0, peak = 0;
  template <typename T = void>
  T* take(size_t bytes) {
    char* p = base ? base + used : nullptr;
    used += up(bytes);
    peak = std::max(peak, used);
    return reinterpret_cast<T*>(p);
  }
};

// Runs launches until one fails (its status is `rc`), with scratch from `a`; dry: nothing runs, a.peak is what it takes.
struct Exec {
  void* stream = nullptr;
  bool dry = true;
  Arena a{nullptr};
  int32_t rc = LLATTN_OK;

  template <typename F>
  void run(F f) {
    if (!dry && rc == LLATTN_OK) rc = f();
  }

  void gemm(const llattn_gemm_desc& d, bool f32) {
    if (f32) {
      run([&] { return llattn_gemm_f32(&d, stream); });
      return;
    }
    const size_t n = llattn_gemm_workspace_size(&d), mark = a.used;
    void* ws = n ? a.take(n) : nullptr;
    run([&] { return llattn_gemm(&d, ws, n, stream); });
    a.used = mark;
  }
  // two products that do not depend on each other
  void gemm(const llattn_gemm_desc& d0, const llattn_gemm_desc& d1, bool f32) {
    if (f32) {
      gemm(d0, true);
      gemm(d1, true);
      return;
    }
    const size_t n = llattn_gemm_pair_workspace_size(&d0, &d1), mark = a.used;
    void* ws = n ? a.take(n) : nullptr;
    run([&] { return llattn_gemm_pair(&d0, &d1, ws, n, stream); });
    a.used = mark;
  }
  // y [M][N] = x [M][K] w [N][K]ᵀ (+ b)
  static llattn_gemm_desc linear(int dt, int M, int N, int K, const void* x, const void* w, const float* b, void* y,
              const llattn_heads_layout* heads = nullptr, int act = LLATTN_ACT_NONE, void* aux = nullptr) {
    llattn_gemm_desc d{};
    d.M = M; d.N = N; d.K = K;
    d.A = x; d.lda = K;
    d.B = w; d.ldb = K;
    d.C = y; d.ldc = N; d.c_dtype = dt;
    d.bias = b;
    if (heads) d.c_heads = *heads;
    d.act = act; d.aux = aux; d.ld_aux = aux ? N : 0;
    return d;
  }
  // dx [M][K] = dy [M][N] w [N][K] (+ row addends; * aux): through w_t where there is one
  static llattn_gemm_desc input_grad(int dt, int M, int N, int K, const void* dy, const void* w, const void* w_t, void* dx,
                  const llattn_heads_layout* heads = nullptr, const llattn_gemm_rowadd* ra = nullptr, int n_ra = 0,
                  void* aux = nullptr) {
    llattn_gemm_desc d{};
    d.M = M; d.N = K; d.K = N;
    d.A = dy; d.lda = N;
    if (w_t) {
      d.B = w_t; d.ldb = N;
    } else {
      d.b_trans = 1;
      d.B = w; d.ldb = K;
    }
    d.C = dx; d.ldc = K; d.c_dtype = dt;
    if (heads) d.c_heads = *heads;
    for (int q = 0; q < n_ra; ++q) d.rowadd[q] = ra[q];
    if (aux) {
      d.act = LLATTN_ACT_MUL_AUX;
      d.aux = aux;
      d.ld_aux = K;
    }
    return d;
  }
  // dw [N][D] = dy [M][N]ᵀ x [M][D] in fp32, db [N] = the column sums of dy
  static llattn_gemm_desc weight_grad(int dt, int M, int N, int D, const void* dy, const void* x, float* dw, float* db) {
    llattn_gemm_desc d{};
    d.M = N; d.N = D; d.K = M;
    d.a_trans = d.b_trans = 1;
    d.A = dy; d.lda = N;
    d.B = x; d.ldb = D;
    d.C = dw; d.ldc = D; d.c_dtype = LLATTN_F32;
    d.a_rowsum = db;
    return d;
  }
  void pool(int dt, const void* x, void* out, int B, int T, int D, int seg, int n, int div) {
    run([&] {
      return llattn_pool_fwd(x, (int64_t)T * D, D, out, (int64_t)n * D, D, B, T, D, seg, n, div, dt, stream);
    });
  }
};

// Weights cast or concatenated in one launch.
struct Casts {
  static constexpr int MAX = 8;
  int n = 0;
  const float* src[MAX];
  void* dst[MAX];
  int64_t count[MAX], ld_t[MAX];
  int32_t dt[MAX], rows[MAX];
  void* dst_t[MAX];
  bool any_t = false;
  void add(const float* s, void* d, int64_t r, int64_t c, int32_t t, void* tr = nullptr, int64_t ld = 0) {
    src[n] = s; dst[n] = d; count[n] = r * c; dt[n] = t;
    dst_t[n] = tr; ld_t[n] = tr ? ld : 0; rows[n] = tr ? (int32_t)r : 0;
    any_t |= tr != nullptr;
    ++n;
  }
  void launch(Exec& e) {
    if (n == 0) return;
    e.run([&] {
      return any_t ? llattn_cast_transposed(n, src, dst, count, dt, dst_t, ld_t, rows, e.stream)
                   : llattn_cast(n, src, dst, count, dt, e.stream);
    });
  }
  // with up to two poolings of x [B][T][D] in the same launch
  int n_pools = 0;
  llattn::PoolArgs pools[llattn::kCastPools];
  void pool(const void* x, void* out, int B, int T, int D, int seg, int segs, int div) {
    pools[n_pools++] = llattn::PoolArgs{x, (int64_t)T * D, D, out, (int64_t)segs * D, D, B, T, D, seg, segs, div, 0};
  }
  void launch_with_pools(Exec& e, int pool_dtype) {
    e.run([&] {
      return llattn::cast_and_pool(n, src, dst, count, dt, any_t ? dst_t : nullptr, ld_t, rows, pools, n_pools,
                                   pool_dtype, e.stream);
    });
  }
};

// bf16 input gradients of this many rows run through a transposed weight (gemm.py: input_grad_persistent), on the
// persistent kernel or, with too few tiles for it, the smaller ones; fewer rows read the weight by transposing LDS loads
bool persistent_grad(int64_t M, int64_t N, int64_t K) { return M >= 4096 && K % 8 == 0 && N % 8 == 0 && N > 64; }

llattn_tensor view(const void* p, int64_t off, int64_t es, int64_t sb, int64_t sn, int64_t sh) {
  return llattn_tensor{p ? const_cast<char*>(static_cast<const char*>(p)) + off * es : nullptr, sb, sn, sh};
}

// ---- core ----------------------------------------------------------------------------------------------------
struct Core {  // kept by the forward
  void *r_w, *r_wt, *lat, *R, *ol;
  float *lse_lat, *lse, *w;
};

struct Dims {
  int dt, B, T, H, Dh, Lh, Ldh, nq, nc;
  int64_t es, D, Ld, M, Mq;
  explicit Dims(const llattn_shape& s)
      : dt(s.dtype), B(s.B), T(s.T), H(s.H), Dh(s.Dh), Lh(s.Lh), Ldh(s.Ldh), nq(s.n_q), nc(s.n_chunks),
        es(elem_size(s.dtype)), D((int64_t)s.H * s.Dh), Ld((int64_t)s.Lh * s.Ldh), M((int64_t)s.B * s.T),
        Mq((int64_t)s.B * s.n_q) {}
  bool macro() const { return nq != T; }
};

// lat_at, R_at: where these lie if not in the arena
Core core_layout(const llattn_block_cfg& c, Arena& a, void* lat_at = nullptr, void* R_at = nullptr) {
  const Dims d(c.shape);
  const bool bf = d.dt == LLATTN_BF16;
  Core k{};
  if (bf) k.r_w = a.take(d.D * d.Ld * 2);
  if (bf && c.saved && persistent_grad(d.Mq, d.D, d.Ld)) k.r_wt = a.take(d.D * d.Ld * 2);
  k.lat = lat_at ? lat_at : a.take(d.Mq * d.Ld * d.es);
  k.R = R_at ? R_at : a.take(d.Mq * d.D * d.es);
  if (c.saved) {
    k.lse_lat = a.take<float>((size_t)d.B * d.Lh * d.nq * 4);
    k.ol = a.take(d.M * d.D * d.es);
    k.lse = a.take<float>(d.M * d.H * 4);
    k.w = a.take<float>(d.M * d.H * 4);
  }
  return k;
}

llattn_tensor remote_view(const llattn_block_cfg& c, const Dims& d, const void* R) {
  if (c.remote_heads) return view(R, 0, d.es, (int64_t)d.H * d.nq * d.Dh, d.Dh, (int64_t)d.nq * d.Dh);
  return view(R, 0, d.es, d.nq * d.D, d.D, d.Dh);
}

void core_fwd(Exec& e, const llattn_block_cfg& c, const llattn_core_views& in, const float* gl, const float* gr,
              const void* r_w, const float* r_b, const Core& k, const llattn_tensor& y) {
  const Dims d(c.shape);
  const llattn_tensor lat = view(k.lat, 0, d.es, d.nq * d.Ld, d.Ld, d.Ldh);
  e.run([&] { return llattn_latent_fwd(&c.shape, &in.gq, &in.gk, &in.gv, &lat, k.lse_lat, e.stream); });
  const llattn_heads_layout rh{d.nq, d.Dh, d.H, 0};
  e.gemm(e.linear(d.dt, (int)d.Mq, (int)d.D, (int)d.Ld, k.lat, r_w, r_b, k.R, c.remote_heads ? &rh : nullptr),
         d.dt == LLATTN_F32);
  const llattn_tensor R = remote_view(c, d, k.R);
  // o_local is the op's own: head-major, a head's rows one contiguous run
  const llattn_tensor ol = view(k.ol, 0, d.es, (int64_t)d.H * d.T * d.Dh, d.Dh, (int64_t)d.T * d.Dh);
  e.run([&] {
    return llattn_local_gate_fwd(&c.shape, &in.q, &in.k, &in.v, &R, gl, gr, &y, k.ol ? &ol : nullptr, k.lse, k.w,
                                 e.stream);
  });
}

void core_bwd(Exec& e, const llattn_block_cfg& c, const llattn_core_views& in, const float* gl,
              const float* gr, const void* r_w, const Core& k, const llattn_tensor& dy, const llattn_core_views& out,
              float* dgl, float* dgr, float* dr_w, float* dr_b) {
  const Dims d(c.shape);
  Arena& a = e.a;
  void* drem = a.take(d.M * d.D * d.es);
  const size_t mark = a.used, n_local = llattn_workspace_size(&c.shape, LLATTN_WS_LOCAL_BWD);
  void* ws_local = a.take(n_local);
  const llattn_tensor R = remote_view(c, d, k.R), dr = view(drem, 0, d.es, d.T * d.D, d.D, d.Dh);
  const llattn_tensor ol = view(k.ol, 0, d.es, (int64_t)d.H * d.T * d.Dh, d.Dh, (int64_t)d.T * d.Dh);
  e.run([&] {
    return llattn_local_gate_bwd(&c.shape, &in.q, &in.k, &in.v, &R, gl, gr, &ol, k.lse, k.w, &dy, &out.q, &out.k,
                                 &out.v, &dr, dgl, dgr, dr_b, ws_local, n_local, e.stream);
  });
  a.used = mark;
  void* dR = drem;
  if (c.shape.q_block > 1 || d.macro()) {
    dR = a.take(d.Mq * d.D * d.es);
    e.pool(d.dt, drem, dR, d.B, d.T, (int)d.D, c.shape.q_block, d.nq, LLATTN_DIV_ONE);
  }
  void* dlat = a.take(d.Mq * d.Ld * d.es);
  const llattn_heads_layout lh{d.nq, d.Ldh, d.Lh, 0};
  e.gemm(e.input_grad(d.dt, (int)d.Mq, (int)d.D, (int)d.Ld, dR, r_w, k.r_wt, dlat, c.lat_heads ? &lh : nullptr),
         e.weight_grad(d.dt, (int)d.Mq, (int)d.D, (int)d.Ld, dR, k.lat, dr_w, nullptr), d.dt == LLATTN_F32);
  const llattn_tensor dl = c.lat_heads ? view(dlat, 0, d.es, d.Ld * d.nq, d.Ldh, (int64_t)d.nq * d.Ldh)
                                       : view(dlat, 0, d.es, d.nq * d.Ld, d.Ld, d.Ldh);
  const size_t n_lat = llattn_workspace_size(&c.shape, LLATTN_WS_LATENT_BWD);
  void* ws_lat = a.take(n_lat);
  e.run([&] {
    return llattn_latent_bwd(&c.shape, &in.gq, &in.gk, &in.gv, k.lse_lat, &dl, &out.gq, &out.gk, &out.gv, ws_lat,
                             n_lat, e.stream);
  });
}

// ---- block ---------------------------------------------------------------------------------------------------
struct Block {  // kept by the forward
  void *w_qkv, *w_qkvt, *w_rq, *w_rkv, *w_out, *w_outt;
  float* b_qkv;
  void *qkvr, *pq, *pooled, *rq, *gkgv, *y;
  Core core;
};

// the query-block means and the latent chunk means are the same values where every segment is full and equal
bool twin_pools(const llattn_block_cfg& c) {
  const llattn_shape& s = c.shape;
  return c.macro && s.q_block == s.chunk && s.n_q == s.n_chunks && (int64_t)s.n_q * s.q_block <= s.T;
}

// out: the output's buffer.  With no backward to follow it holds R until the product that writes it (R has no more
// rows than the output), and y lies over the projection's weights and the latent output, which nothing reads any more
// when the local kernel writes it.
Block block_layout(const llattn_block_cfg& c, Arena& a, void* out) {
  const Dims d(c.shape);
  const int64_t Dm = c.d_model, width = 3 * Dm + (c.macro ? 0 : d.Ld);
  const bool bf = d.dt == LLATTN_BF16;
  Block k{};
  const size_t mark = a.used;
  if (bf || !c.macro) {
    k.w_qkv = a.take(width * Dm * d.es);
    if (c.has_bias) k.b_qkv = a.take<float>(width * 4);
  }
  void* lat = nullptr;
  if (!c.saved) {
    lat = a.take(d.Mq * d.Ld * d.es);
    if (!lat) lat = &a;  // a dry run's counts as placed
    const size_t end = a.used;
    a.used = mark;
    k.y = a.take(d.M * d.D * d.es);
    a.used = std::max(a.used, end);
  }
  if (bf) {
    if (c.saved && persistent_grad(d.M, width, Dm)) k.w_qkvt = a.take(width * Dm * 2);
    if (c.macro) k.w_rq = a.take(d.Ld * Dm * 2);
    k.w_rkv = a.take(2 * d.Ld * Dm * 2);
    k.w_out = a.take(Dm * Dm * 2);
    if (c.saved && persistent_grad(d.M, Dm, Dm)) k.w_outt = a.take(Dm * Dm * 2);
  }
  k.qkvr = a.take(d.M * width * d.es);
  k.pooled = a.take((int64_t)d.B * d.nc * Dm * d.es);
  if (c.macro) {
    k.pq = twin_pools(c) ? k.pooled : a.take(d.Mq * Dm * d.es);
    k.rq = a.take(d.Mq * d.Ld * d.es);
  }
  k.gkgv = a.take((int64_t)d.B * d.nc * 2 * d.Ld * d.es);
  if (c.saved) k.y = a.take(d.M * d.D * d.es);
  k.core = core_layout(c, a, lat, c.saved ? nullptr : out);
  return k;
}

llattn_core_views block_views(const llattn_block_cfg& c, const void* qkvr, bool heads, const void* rq, const void* gkgv) {
  const Dims d(c.shape);
  llattn_core_views v{};
  const int64_t width = 3 * d.D + (c.macro ? 0 : d.Ld);
  llattn_tensor* qkv[3] = {&v.q, &v.k, &v.v};
  for (int i = 0; i < 3; ++i)
    *qkv[i] = heads ? view(qkvr, i * d.D * d.T, d.es, 3 * d.D * d.T, d.Dh, (int64_t)d.T * d.Dh)
                    : view(qkvr, i * d.D, d.es, d.T * width, width, d.Dh);
  if (c.macro) v.gq = view(rq, 0, d.es, d.nq * d.Ld, d.Ld, d.Ldh);
  else if (heads) v.gq = view(qkvr, d.M * 3 * d.D, d.es, d.T * d.Ld, d.Ldh, (int64_t)d.T * d.Ldh);
  else v.gq = view(qkvr, 3 * d.D, d.es, d.T * width, width, d.Ldh);
  v.gk = view(gkgv, 0, d.es, d.nc * 2 * d.Ld, 2 * d.Ld, d.Ldh);
  v.gv = view(gkgv, d.Ld, d.es, d.nc * 2 * d.Ld, 2 * d.Ld, d.Ldh);
  return v;
}

// the weights that the products read: the kept copies, or in fp32 the parameters themselves
struct Weights {
  const void *qkv, *rq, *rkv, *r, *out;
  const float* b_qkv;
};
Weights block_weights(const llattn_block_cfg& c, const llattn_block_params& p, const Block& k) {
  if (c.shape.dtype == LLATTN_BF16) return Weights{k.w_qkv, k.w_rq, k.w_rkv, k.core.r_w, k.w_out, k.b_qkv};
  if (c.macro) return Weights{p.w_qkv, p.w_rq, p.w_rkv, p.w_r, p.w_out, p.b_qkv};
  return Weights{k.w_qkv, nullptr, p.w_rkv, p.w_r, p.w_out, k.b_qkv};
}

void block_fwd(Exec& e, const llattn_block_cfg& c, const llattn_block_params& p, const void* x, const Block& k, void* out) {
  const Dims d(c.shape);
  const llattn_shape& s = c.shape;
  const int64_t Dm = c.d_model, width = 3 * Dm + (c.macro ? 0 : d.Ld);
  const int32_t dt = d.dt;
  Casts casts;
  if (k.w_qkv) {
    casts.add(p.w_qkv, k.w_qkv, 3 * Dm, Dm, dt, k.w_qkvt, width);
    if (!c.macro)
      casts.add(p.w_rq, view(k.w_qkv, 3 * Dm * Dm, d.es, 0, 0, 0).ptr, d.Ld, Dm, dt,
                k.w_qkvt ? view(k.w_qkvt, 3 * Dm, 2, 0, 0, 0).ptr : nullptr, width);
    if (c.has_bias) {
      casts.add(p.b_qkv, k.b_qkv, 3 * Dm, 1, LLATTN_F32);
      if (!c.macro) casts.add(p.b_rq, k.b_qkv ? k.b_qkv + 3 * Dm : nullptr, d.Ld, 1, LLATTN_F32);
    }
  }
  if (dt == LLATTN_BF16) {
    if (c.macro) casts.add(p.w_rq, k.w_rq, d.Ld, Dm, dt);
    casts.add(p.w_rkv, k.w_rkv, 2 * d.Ld, Dm, dt);
    casts.add(p.w_out, k.w_out, Dm, Dm, dt, k.w_outt, Dm);
    casts.add(p.w_r, k.core.r_w, d.D, d.Ld, dt, k.core.r_wt, d.D);
  }
  if (c.macro) {
    if (!twin_pools(c)) casts.pool(x, k.pq, d.B, d.T, (int)Dm, s.q_block, d.nq, LLATTN_DIV_SEG);
    else casts.pool(x, k.pooled, d.B, d.T, (int)Dm, s.chunk, d.nc, LLATTN_DIV_SEG);
  }
  if (!twin_pools(c)) casts.pool(x, k.pooled, d.B, d.T, (int)Dm, s.chunk, d.nc, LLATTN_DIV_COUNT);
  casts.launch_with_pools(e, dt);
  const Weights w = block_weights(c, p, k);
  const llattn_heads_layout hl{d.T, d.Dh, 3 * d.H, c.macro ? 0 : d.Ldh};
  const bool f32 = dt == LLATTN_F32;
  e.gemm(e.linear(dt, (int)d.M, (int)width, (int)Dm, x, w.qkv, w.b_qkv, k.qkvr, c.heads ? &hl : nullptr),
         e.linear(dt, d.B * d.nc, (int)(2 * d.Ld), (int)Dm, k.pooled, w.rkv, p.b_rkv, k.gkgv), f32);
  if (c.macro) e.gemm(e.linear(dt, (int)d.Mq, (int)d.Ld, (int)Dm, k.pq, w.rq, p.b_rq, k.rq), f32);
  const llattn_tensor y = view(k.y, 0, d.es, d.T * d.D, d.D, d.Dh);
  core_fwd(e, c, block_views(c, k.qkvr, c.heads, k.rq, k.gkgv), p.gate_l, p.gate_r, w.r, p.b_r, k.core, y);
  e.gemm(e.linear(dt, (int)d.M, (int)Dm, (int)d.D, k.y, w.out, p.b_out, out), f32);
}

void block_bwd(Exec& e, const llattn_block_cfg& c, const llattn_block_params& p, const void* x,
               const Block& k, const void* dy, void* dx, const llattn_block_grads& g) {
  const Dims d(c.shape);
  const llattn_shape& s = c.shape;
  const int64_t Dm = c.d_model, width = 3 * Dm + (c.macro ? 0 : d.Ld);
  const int dt = d.dt;
  const bool bf = dt == LLATTN_BF16;
  const Weights w = block_weights(c, p, k);
  Arena& a = e.a;
  void* dqkv = a.take(d.M * width * d.es);
  void* drq = c.macro ? a.take(d.Mq * d.Ld * d.es) : nullptr;
  void* dgkgv = a.take((int64_t)d.B * d.nc * 2 * d.Ld * d.es);
  const size_t mark = a.used;
  // the core's output gradient lies in dx, which the last product writes, long after its last reader
  void* dyc = dx ? dx : a.take(d.M * d.D * d.es);
  const llattn_heads_layout yh{d.T, d.Dh, d.H, 0};
  e.gemm(e.input_grad(dt, (int)d.M, (int)Dm, (int)d.D, dy, w.out, k.w_outt, dyc, c.dy_heads ? &yh : nullptr),
         e.weight_grad(dt, (int)d.M, (int)Dm, (int)d.D, dy, k.y, g.w_out, g.b_out), !bf);
  // the gradient in plain rows whatever the storage of qkv: the projection's backward reads it row-major
  const llattn_core_views out = block_views(c, dqkv, false, drq, dgkgv);
  const llattn_tensor dyv = c.dy_heads ? view(dyc, 0, d.es, (int64_t)d.T * d.D, d.Dh, (int64_t)d.T * d.Dh)
                                       : view(dyc, 0, d.es, d.T * d.D, d.D, d.Dh);
  core_bwd(e, c, block_views(c, k.qkvr, c.heads, k.rq, k.gkgv), p.gate_l, p.gate_r, w.r, k.core, dyv, out, g.gate_l,
           g.gate_r, g.w_r, g.b_r);
  a.used = mark;
  const int Mc = d.B * d.nc;
  void* dpooled = dx ? a.take((int64_t)Mc * Dm * d.es) : nullptr;
  // an input gradient (where it is wanted) with the weight gradient of the same dy
  auto grads = [&](const llattn_gemm_desc& di, const llattn_gemm_desc& dw) {
    if (dx) e.gemm(di, dw, !bf);
    else e.gemm(dw, !bf);
  };
  grads(e.input_grad(dt, Mc, (int)(2 * d.Ld), (int)Dm, dgkgv, w.rkv, nullptr, dpooled),
        e.weight_grad(dt, Mc, (int)(2 * d.Ld), (int)Dm, dgkgv, k.pooled, g.w_rkv, g.b_rkv));
  void* dpq = dx && c.macro ? a.take(d.Mq * Dm * d.es) : nullptr;
  if (c.macro)
    grads(e.input_grad(dt, (int)d.Mq, (int)d.Ld, (int)Dm, drq, w.rq, nullptr, dpq),
          e.weight_grad(dt, (int)d.Mq, (int)d.Ld, (int)Dm, drq, k.pq, g.w_rq, g.b_rq));
  // the poolings' gradients join the input gradient: in bf16 in the product's epilogue, query blocks first
  static char there;  // a dry run's addends count as present
  if (e.dry) dpq = dpooled = &there;
  llattn_gemm_rowadd ra[2];
  int n = 0;
  if (c.macro) ra[n++] = llattn_gemm_rowadd{dpq, Dm, d.T, s.q_block, d.nq, LLATTN_DIV_SEG};
  ra[n++] = llattn_gemm_rowadd{dpooled, Dm, d.T, s.chunk, d.nc, LLATTN_DIV_COUNT};
  grads(e.input_grad(dt, (int)d.M, (int)width, (int)Dm, dqkv, w.qkv, k.w_qkvt, dx, nullptr, ra, bf ? n : 0),
        e.weight_grad(dt, (int)d.M, (int)width, (int)Dm, dqkv, x, g.w_qkv, g.b_qkv));
  for (int q = 0; q < n && !bf && dx; ++q)
    e.run([&] {
      return llattn_pool_bwd(ra[q].ptr, (int64_t)ra[q].n_seg * Dm, Dm, dx, d.T * Dm, Dm, d.B, d.T, (int)Dm, ra[q].seg,
                             ra[q].n_seg, ra[q].divisor, 1, dt, e.stream);
    });
}

int32_t check_cfg(const char* what, const llattn_block_cfg* c, bool block) {
  if (!c) return fail(LLATTN_ERR_SHAPE, "%s: null configuration", what);
  if (const int32_t rc = check_shape(&c->shape)) return rc;
  const llattn_shape& s = c->shape;
  const int64_t D = (int64_t)s.H * s.Dh, Ld = (int64_t)s.Lh * s.Ldh;
  const int64_t most = 0x7fffffff;
  if ((int64_t)s.B * s.T > most || (int64_t)s.B * s.n_q > most || 3 * D + Ld > most)
    return fail(LLATTN_ERR_UNSUPPORTED, "%s: more rows or columns than 2^31", what);
  if (block && (c->d_model != D || (!c->macro && (s.n_q != s.T || s.q_block != 1)) || s.gate_per_head))
    return fail(LLATTN_ERR_SHAPE, "%s: d_model %d of %d heads of %d, %d queries over %d tokens (macro %d)", what,
                c->d_model, s.H, s.Dh, s.n_q, s.T, c->macro);
  return LLATTN_OK;
}

int32_t begin(Exec& e, const char* what, size_t need, void* ws, size_t ws_bytes, void* stream) {
  if (need && (!ws || ws_bytes < need || !aligned16(ws)))
    return fail(LLATTN_ERR_WORKSPACE, "%s needs %zu scratch bytes (got %zu)", what, need, ws_bytes);
  e.stream = stream;
  e.dry = false;
  e.a = Arena{static_cast<char*>(ws)};
  return LLATTN_OK;
}

template <typename F>
size_t measure(F f) {
  Exec e;
  f(e);
  return e.a.peak;
}

enum Pass { FWD = 1, BWD = 2, BWD_NO_DX = 3 };  // what a size is asked for (llattn_*_bytes)

size_t block_need(const llattn_block_cfg& c, int pass) {
  return measure([&](Exec& e) {
    Arena none{nullptr};
    const Block k = block_layout(c, none, nullptr);
    // a dry run reads no pointer, but the routes follow from which transposed copies exist
    Block with = k;
    static char there;
    const Dims d(c.shape);
    const bool bf = d.dt == LLATTN_BF16;
    const int64_t width = 3 * (int64_t)c.d_model + (c.macro ? 0 : d.Ld);
    if (bf && c.saved && persistent_grad(d.M, width, c.d_model)) with.w_qkvt = &there;
    if (bf && c.saved && persistent_grad(d.M, c.d_model, c.d_model)) with.w_outt = &there;
    if (bf && c.saved && persistent_grad(d.Mq, d.D, d.Ld)) with.core.r_wt = &there;
    const llattn_block_params p{};
    if (pass == FWD) {
      block_fwd(e, c, p, nullptr, with, nullptr);
    } else {
      llattn_block_grads g{};
      if (c.has_bias) g.b_qkv = g.b_rq = g.b_rkv = g.b_out = reinterpret_cast<float*>(&there);
      block_bwd(e, c, p, nullptr, with, nullptr, pass == BWD ? &there : nullptr, g);
    }
  });
}

size_t core_need(const llattn_block_cfg& c, int pass) {
  return measure([&](Exec& e) {
    Arena none{nullptr};
    Core k = core_layout(c, none);
    static char there;
    const Dims d(c.shape);
    if (d.dt == LLATTN_BF16 && c.saved && persistent_grad(d.Mq, d.D, d.Ld)) k.r_wt = &there;
    const llattn_core_views v{};
    const llattn_tensor t{};
    if (pass == FWD) core_fwd(e, c, v, nullptr, nullptr, nullptr, nullptr, k, t);
    else core_bwd(e, c, v, nullptr, nullptr, nullptr, k, t, v, nullptr, nullptr, nullptr, nullptr);
  });
}

// ---- feed-forward --------------------------------------------------------------------------------------------
struct Ffn {  // kept by the forward
  void *w1, *w1t, *w2, *w2t, *g, *gp;
};
Ffn ffn_layout(const llattn_ffn_cfg& c, Arena& a) {
  const int64_t M = c.rows, d = c.d, f = c.d_ff, o = c.d_out;
  Ffn k{};
  k.w1 = a.take(f * d * 2);
  if (c.saved && persistent_grad(M, f, d)) k.w1t = a.take(f * d * 2);
  k.w2 = a.take(o * f * 2);
  if (c.saved && persistent_grad(M, o, f)) k.w2t = a.take(o * f * 2);
  k.g = a.take(M * f * 2);
  k.gp = a.take(M * f * 2);
  return k;
}
void ffn_fwd(Exec& e, const llattn_ffn_cfg& c, const void* x, const float* w1, const float* b1, const float* w2,
             const float* b2, const Ffn& k, void* y) {
  Casts casts;
  casts.add(w1, k.w1, c.d_ff, c.d, LLATTN_BF16, k.w1t, c.d_ff);
  casts.add(w2, k.w2, c.d_out, c.d_ff, LLATTN_BF16, k.w2t, c.d_out);
  casts.launch(e);
  static char there;
  e.gemm(e.linear(LLATTN_BF16, c.rows, c.d_ff, c.d, x, k.w1, b1, k.g, nullptr, LLATTN_ACT_GELU, e.dry ? &there : k.gp), false);
  e.gemm(e.linear(LLATTN_BF16, c.rows, c.d_out, c.d_ff, k.g, k.w2, b2, y), false);
}
void ffn_bwd(Exec& e, const llattn_ffn_cfg& c, const void* x, const Ffn& k, const void* dy, void* dx,
             float* dw1, float* db1, float* dw2, float* db2) {
  void* dh = e.a.take((int64_t)c.rows * c.d_ff * 2);
  static char there;
  e.gemm(e.input_grad(LLATTN_BF16, c.rows, c.d_out, c.d_ff, dy, k.w2, k.w2t, dh, nullptr, nullptr, 0, e.dry ? &there : k.gp),
         e.weight_grad(LLATTN_BF16, c.rows, c.d_out, c.d_ff, dy, k.g, dw2, db2), false);
  const llattn_gemm_desc dw = e.weight_grad(LLATTN_BF16, c.rows, c.d_ff, c.d, dh, x, dw1, db1);
  if (dx) e.gemm(e.input_grad(LLATTN_BF16, c.rows, c.d_ff, c.d, dh, k.w1, k.w1t, dx), dw, false);
  else e.gemm(dw, false);
}
size_t ffn_need(const llattn_ffn_cfg& c, int pass) {
  return measure([&](Exec& e) {
    Arena none{nullptr};
    Ffn k = ffn_layout(c, none);
    static char there;
    if (c.saved && persistent_grad(c.rows, c.d_ff, c.d)) k.w1t = &there;
    if (c.saved && persistent_grad(c.rows, c.d_out, c.d_ff)) k.w2t = &there;
    float* bias = reinterpret_cast<float*>(&there);
    if (pass == FWD) ffn_fwd(e, c, nullptr, nullptr, nullptr, nullptr, nullptr, k, nullptr);
    else ffn_bwd(e, c, nullptr, k, nullptr, pass == BWD ? &there : nullptr, nullptr, bias, nullptr, bias);
  });
}
int32_t check_ffn(const char* what, const llattn_ffn_cfg* c) {
  if (!c || c->rows <= 0 || c->d <= 0 || c->d_ff <= 0 || c->d_out <= 0)
    return fail(LLATTN_ERR_SHAPE, "%s: sizes must be positive", what);
  return LLATTN_OK;
}

}  // namespace
}  // namespace llattn

using namespace llattn;

extern "C" {

size_t llattn_block_bytes(const llattn_block_cfg* c, int32_t which) {
  if (check_cfg("llattn_block_bytes", c, true)) return 0;
  if (which != 0) return block_need(*c, which);
  Arena a{nullptr};
  static char there;
  block_layout(*c, a, &there);
  return a.used;
}

int32_t llattn_block_fwd(const llattn_block_cfg* c, const llattn_block_params* p, const void* x, void* kept, void* ws,
                         size_t ws_bytes, void* out, void* stream) {
  const char* what = "llattn_block_fwd";
  if (const int32_t rc = check_cfg(what, c, true)) return rc;
  if (!p || !x || !kept || !out || !aligned16(kept)) return fail(LLATTN_ERR_LAYOUT, "%s: null or misaligned buffer", what);
  Exec e;
  if (const int32_t rc = begin(e, what, block_need(*c, FWD), ws, ws_bytes, stream)) return rc;
  Arena ka{static_cast<char*>(kept)};
  block_fwd(e, *c, *p, x, block_layout(*c, ka, out), out);
  return e.rc;
}

int32_t llattn_block_bwd(const llattn_block_cfg* c, const llattn_block_params* p, const void* x, const void* kept,
                         const void* dy, void* dx, const llattn_block_grads* g, void* ws, size_t ws_bytes,
                         void* stream) {
  const char* what = "llattn_block_bwd";
  if (const int32_t rc = check_cfg(what, c, true)) return rc;
  if (!p || !x || !kept || !dy || !g || !c->saved) return fail(LLATTN_ERR_LAYOUT, "%s: null buffer or nothing kept", what);
  Exec e;
  if (const int32_t rc = begin(e, what, block_need(*c, dx ? BWD : BWD_NO_DX), ws, ws_bytes, stream)) return rc;
  Arena ka{static_cast<char*>(const_cast<void*>(kept))};
  block_bwd(e, *c, *p, x, block_layout(*c, ka, nullptr), dy, dx, *g);
  return e.rc;
}

size_t llattn_core_bytes(const llattn_block_cfg* c, int32_t which) {
  if (check_cfg("llattn_core_bytes", c, false)) return 0;
  if (which != 0) return core_need(*c, which);
  Arena a{nullptr};
  core_layout(*c, a);
  return a.used;
}

int32_t llattn_core_fwd(const llattn_block_cfg* c, const llattn_core_views* in, const float* gate_l,
                        const float* gate_r, const float* r_w, const float* r_b, void* kept, void* ws,
                        size_t ws_bytes, const llattn_tensor* y, void* stream) {
  const char* what = "llattn_core_fwd";
  if (const int32_t rc = check_cfg(what, c, false)) return rc;
  if (!in || !r_w || !kept || !y || !aligned16(kept)) return fail(LLATTN_ERR_LAYOUT, "%s: null or misaligned buffer", what);
  Exec e;
  if (const int32_t rc = begin(e, what, core_need(*c, FWD), ws, ws_bytes, stream)) return rc;
  Arena ka{static_cast<char*>(kept)};
  const Core k = core_layout(*c, ka);
  const Dims d(c->shape);
  Casts casts;
  if (k.r_w) casts.add(r_w, k.r_w, d.D, d.Ld, LLATTN_BF16, k.r_wt, d.D);
  casts.launch(e);
  core_fwd(e, *c, *in, gate_l, gate_r, k.r_w ? k.r_w : r_w, r_b, k, *y);
  return e.rc;
}

int32_t llattn_core_bwd(const llattn_block_cfg* c, const llattn_core_views* in, const float* gate_l,
                        const float* gate_r, const float* r_w, const void* kept, const llattn_tensor* dy,
                        const llattn_core_views* dv, float* dgate_l, float* dgate_r, float* dr_w, float* dr_b,
                        void* ws, size_t ws_bytes, void* stream) {
  const char* what = "llattn_core_bwd";
  if (const int32_t rc = check_cfg(what, c, false)) return rc;
  if (!in || !r_w || !kept || !dy || !dv || !c->saved) return fail(LLATTN_ERR_LAYOUT, "%s: null buffer or nothing kept", what);
  Exec e;
  if (const int32_t rc = begin(e, what, core_need(*c, BWD), ws, ws_bytes, stream)) return rc;
  Arena ka{static_cast<char*>(const_cast<void*>(kept))};
  const Core k = core_layout(*c, ka);
  core_bwd(e, *c, *in, gate_l, gate_r, k.r_w ? k.r_w : r_w, k, *dy, *dv, dgate_l, dgate_r, dr_w, dr_b);
  return e.rc;
}

size_t llattn_ffn_bytes(const llattn_ffn_cfg* c, int32_t which) {
  if (check_ffn("llattn_ffn_bytes", c)) return 0;
  if (which != 0) return ffn_need(*c, which);
  Arena a{nullptr};
  ffn_layout(*c, a);
  return a.used;
}

int32_t llattn_ffn_fwd(const llattn_ffn_cfg* c, const void* x, const float* w1, const float* b1, const float* w2,
                       const float* b2, void* kept, void* ws, size_t ws_bytes, void* y, void* stream) {
  const char* what = "llattn_ffn_fwd";
  if (const int32_t rc = check_ffn(what, c)) return rc;
  if (!x || !w1 || !w2 || !kept || !y || !aligned16(kept)) return fail(LLATTN_ERR_LAYOUT, "%s: null or misaligned buffer", what);
  Exec e;
  if (const int32_t rc = begin(e, what, ffn_need(*c, FWD), ws, ws_bytes, stream)) return rc;
  Arena ka{static_cast<char*>(kept)};
  ffn_fwd(e, *c, x, w1, b1, w2, b2, ffn_layout(*c, ka), y);
  return e.rc;
}

int32_t llattn_ffn_bwd(const llattn_ffn_cfg* c, const void* x, const void* kept, const void* dy, void* dx, float* dw1,
                       float* db1, float* dw2, float* db2, void* ws, size_t ws_bytes, void* stream) {
  const char* what = "llattn_ffn_bwd";
  if (const int32_t rc = check_ffn(what, c)) return rc;
  if (!x || !kept || !dy || !dw1 || !dw2 || !c->saved) return fail(LLATTN_ERR_LAYOUT, "%s: null buffer or nothing kept", what);
  Exec e;
  if (const int32_t rc = begin(e, what, ffn_need(*c, dx ? BWD : BWD_NO_DX), ws, ws_bytes, stream)) return rc;
  Arena ka{static_cast<char*>(const_cast<void*>(kept))};
  ffn_bwd(e, *c, x, ffn_layout(*c, ka), dy, dx, dw1, db1, dw2, db2);
  return e.rc;
}

}  // extern "C"
