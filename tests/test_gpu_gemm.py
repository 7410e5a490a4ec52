"""GPU parity of the gfx950 projection GEMM (``llattn_gemm`` through the C ABI) against a float32 torch
product of the same bf16 operands.

Tolerances: bf16 output within 1e-2 of max(1, max|ref|) (one bf16 rounding of the result is 2^-8
relative); fp32 output within 1e-4 of max(1, max|ref|) (fp32 accumulation over up to 32k terms).
"""
from __future__ import annotations

import pytest
import torch

from gpu_helpers import require_cuda

pytestmark = pytest.mark.gpu

BF16_TOL, FP32_TOL = 1e-2, 1e-4


def _err(got, ref):
    return float((got.float() - ref).abs().max()) / max(1.0, float(ref.abs().max()))


def _rand(*shape, gen, dev):
    return torch.randn(*shape, device=dev, generator=gen).to(torch.bfloat16)


@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (300, 264, 128), (97, 40, 192), (1000, 1408, 512),
                                   (32768, 4736, 1408)])
def test_linear_with_bias(M, N, K):
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: linear", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x, w = _rand(M, K, gen=g, dev=dev), _rand(N, K, gen=g, dev=dev)
    b = torch.randn(N, device=dev, generator=g)
    ref = x.float() @ w.float().T + b
    assert _err(gemm.linear(x, w, b), ref) < BF16_TOL


@pytest.mark.parametrize("M,N,K,dt,acc", [(512, 64, 1024, torch.float32, False), (97, 40, 192, torch.float32, False),
                                          (512, 128, 1000, torch.float32, True), (512, 64, 1024, torch.bfloat16, True),
                                          (256, 1024, 1408, torch.bfloat16, False)])
def test_small_product_bias_and_accumulate(M, N, K, dt, acc):
    """Products of few 64 x 64 tiles over a long contraction (the pooled-latent and query-block projections)
    run as K splits plus the ordered reduction; bias and accumulation apply once, for an fp32 output too."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: small product", M, N, K, dt, acc, flush=True)
    g = torch.Generator(device=dev).manual_seed(M + 3 * N + K)
    x, w = _rand(M, K, gen=g, dev=dev), _rand(N, K, gen=g, dev=dev)
    b = torch.randn(N, device=dev, generator=g)
    c0 = torch.randn(M, N, device=dev, generator=g).to(dt)
    out = c0.clone() if acc else torch.empty((M, N), dtype=dt, device=dev)
    gemm.linear(x, w, b, out=out, accumulate=acc)
    ref = x.float() @ w.float().T + b + (c0.float() if acc else 0.0)
    assert _err(out, ref) < BF16_TOL


@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (1, 40, 72), (97, 40, 200), (33, 264, 1000), (4096, 512, 200),
                                   (2000, 136, 8), (194, 208, 88)])
def test_linear_k_tail(M, N, K):
    """Contractions that are not a multiple of the 64-wide k step: the k-contiguous lanes past K read zero
    (a single row included, whose buffer ends inside the last step)."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: linear k tail", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(M * 7 + N + K)
    # operands cut out of wider rows, so the elements past K are real data that must not leak in
    xb, wb = _rand(M, K + 24, gen=g, dev=dev) * 50, _rand(N, K + 24, gen=g, dev=dev) * 50
    x, w = xb[:, :K], wb[:, :K]
    b = torch.randn(N, device=dev, generator=g)
    assert _err(gemm.linear(x, w, b), x.float() @ w.float().T + b) < BF16_TOL


@pytest.mark.parametrize("M,N,K", [(32768, 1024, 64), (8192, 1408, 40), (32768, 256, 8)])
def test_linear_single_k_step(M, N, K):
    """A contraction of at most one 64-wide step on the persistent kernel (config 3's r_out forward, K = Ld =
    64): the pipeline runs it as two steps, the second reading zeros; the split-head store gives the same
    bits."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: linear single k step", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(M + 5 * N + K)
    xb, wb = _rand(M, K + 24, gen=g, dev=dev), _rand(N, K + 24, gen=g, dev=dev)
    x, w = xb[:, :K], wb[:, :K]
    b = torch.randn(N, device=dev, generator=g)
    got = gemm.linear(x, w, b)
    assert _err(got, x.float() @ w.float().T + b) < BF16_TOL
    if N % 64 == 0:
        T = 2048
        heads = gemm.linear(x, w, b, heads=(T, 64, N // 64))
        assert torch.equal(heads, _to_heads(got, T, 64, N // 64))


@pytest.mark.parametrize("M,N,K", [(97, 40, 208), (300, 264, 1000), (3, 512, 72)])
def test_matmul_nn_k_tail(M, N, K):
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: nn k tail", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(5 * M + N + K)
    ab = _rand(M, K + 40, gen=g, dev=dev) * 50
    a, b = ab[:, :K], _rand(K, N, gen=g, dev=dev)
    assert _err(gemm.matmul_nn(a, b), a.float() @ b.float()) < BF16_TOL


@pytest.mark.parametrize("K,M,N,S", [(194, 264, 136, 0), (33, 40, 96, 1), (1001, 1408, 512, 0), (5000, 264, 136, 3),
                                     (122, 16, 8, 2)])
def test_matmul_tn_token_tail(K, M, N, S):
    """Weight gradients over token counts that are not a multiple of 64 (nor of 8): rows past K lie beyond
    the operands' extent and read zero; with split-K the last split is the short one."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: tn token tail", K, M, N, S, flush=True)
    g = torch.Generator(device=dev).manual_seed(K + 3 * M + N)
    a, b = _rand(K, M, gen=g, dev=dev), _rand(K, N, gen=g, dev=dev)
    rs = torch.full((M,), float("nan"), device=dev)
    got = gemm.matmul_tn(a, b, split_k=S, rowsum=rs)
    assert _err(got, a.float().T @ b.float()) < FP32_TOL
    assert _err(rs, a.float().sum(0)) < FP32_TOL


@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (300, 264, 128), (1000, 1408, 512)])
def test_matmul_nn(M, N, K):
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: nn", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(7 * M + N)
    a, b = _rand(M, K, gen=g, dev=dev), _rand(K, N, gen=g, dev=dev)
    assert _err(gemm.matmul_nn(a, b), a.float() @ b.float()) < BF16_TOL


@pytest.mark.parametrize("B,T,N,K,pools", [
    (2, 300, 264, 128, [(64, 0)]),               # latent-style mean, last segment 44 tokens
    (3, 256, 136, 192, [(64, 1), (100, 0)]),     # query-block (zero-padded) mean and a ragged chunk mean
    (16, 2048, 1408, 4736, [(128, 0)]),          # config 2: qkv input gradient with the latent pooling
    (2, 97, 40, 64, [(17, 2)]),                  # plain sums
    (2, 2048, 1408, 4736, [(128, 0), (64, 1)]),  # a split-K shape: the addends join in the ordered reduction
])
def test_matmul_nn_rowadd(B, T, N, K, pools):
    """Input gradient with the pooling backward in its epilogue: a @ b + sum over poolings of rows[b, t // seg] /
    divisor (divisor 0: real tokens in the segment, 1: seg, 2: one), against fp32 torch; bf16 output."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: nn rowadd", B, T, N, K, pools, flush=True)
    g = torch.Generator(device=dev).manual_seed(B * T + N)
    a, b = _rand(B * T, K, gen=g, dev=dev), _rand(K, N, gen=g, dev=dev)
    ref = a.float() @ b.float()
    rowadd = []
    t = torch.arange(T, device=dev)
    for seg, div in pools:
        n_seg = -(-T // seg)
        rows = _rand(B * n_seg, N, gen=g, dev=dev) * 4
        s_id = t // seg
        count = torch.minimum((s_id + 1) * seg, torch.full_like(s_id, T)) - s_id * seg
        scale = {0: 1.0 / count.float(), 1: torch.full((T,), 1.0 / seg, device=dev), 2: torch.ones(T, device=dev)}[div]
        add = rows.float().view(B, n_seg, N)[:, s_id] * scale[None, :, None]
        ref = ref + add.reshape(B * T, N)
        rowadd.append((rows, T, seg, n_seg, div))
    assert _err(gemm.matmul_nn(a, b, rowadd=rowadd), ref) < BF16_TOL


@pytest.mark.parametrize("K,M,N,S", [(64, 256, 264, 1), (1024, 264, 136, 0), (2048, 40, 96, 1), (4096, 264, 136, 3),
                                     (4096, 1000, 520, 1), (32768, 1408, 1408, 0), (32768, 4736, 1408, 0),
                                     # N a multiple of 256 (no spare column): the first tile column's extra
                                     # products against ones; single pass, split-K, a ragged M and token tail
                                     (4096, 1000, 512, 1), (4096, 264, 256, 3), (1001, 520, 768, 2),
                                     (32768, 3200, 1024, 0), (32768, 1024, 1024, 0),
                                     # automatic 2-way splits of 90 tiles, a token tail in the last step, both
                                     # row-sum layouts
                                     (8200, 2304, 2504, 0), (8192, 2304, 2560, 0)])
def test_matmul_tn_rowsum(K, M, N, S):
    """Weight gradient with the bias gradient of the same pass: rowsum = a.sum(0), contracted against a column
    of ones in the spare column N of the last tile, or (N a multiple of 256) against ones in extra products of
    the first tile column; the product itself is unchanged by it."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: tn rowsum", K, M, N, S, flush=True)
    g = torch.Generator(device=dev).manual_seed(3 * K + M + N)
    a, b = _rand(K, M, gen=g, dev=dev), _rand(K, N, gen=g, dev=dev)
    rs = torch.full((M,), float("nan"), device=dev)
    got = gemm.matmul_tn(a, b, split_k=S, rowsum=rs)
    assert _err(got, a.float().T @ b.float()) < FP32_TOL
    assert _err(rs, a.float().sum(0)) < FP32_TOL
    # run to run: bitwise identical (ordered split-K reduction)
    rs2 = torch.empty_like(rs)
    got2 = gemm.matmul_tn(a, b, split_k=S, rowsum=rs2)
    assert torch.equal(rs, rs2) and torch.equal(got, got2)
    assert torch.equal(got, gemm.matmul_tn(a, b, split_k=S))  # the same products with and without the row sums


@pytest.mark.parametrize("K,M,N,S", [(64, 256, 256, 1), (1024, 264, 136, 0), (4096, 1408, 512, 4),
                                     (2048, 40, 96, 2), (4096, 264, 136, 3), (32768, 1408, 1408, 0),
                                     (32768, 4736, 1408, 0), (32768, 1408, 512, 0)])
def test_matmul_tn_fp32_out(K, M, N, S):
    """Weight-gradient products, including split-K (S > 1 or automatic) at the config-2 shapes."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: tn", K, M, N, S, flush=True)
    g = torch.Generator(device=dev).manual_seed(K + M)
    a, b = _rand(K, M, gen=g, dev=dev), _rand(K, N, gen=g, dev=dev)
    got = gemm.matmul_tn(a, b, split_k=S)
    assert got.dtype == torch.float32
    assert _err(got, a.float().T @ b.float()) < FP32_TOL


@pytest.mark.parametrize("M,N", [(1, 8), (97, 40), (1000, 136), (32768, 1408), (32768, 4736)])
def test_colsum(M, N):
    """Bias-gradient column sums, including ragged stripes and row blocks, and their determinism."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: colsum", M, N, flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N)
    big = _rand(M, N + 16, gen=g, dev=dev)
    x = big[:, 8:8 + N]                       # strided view
    got = gemm.colsum(x)
    assert _err(got, x.float().sum(0)) < FP32_TOL
    torch.testing.assert_close(got, gemm.colsum(x), rtol=0, atol=0)


def test_accumulate_and_strided_views():
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: accumulate", flush=True)
    g = torch.Generator(device=dev).manual_seed(3)
    big = _rand(512, 200, gen=g, dev=dev)
    x = big[:, 8:136]                      # row stride 200, 128 columns
    w = _rand(256, 128, gen=g, dev=dev)
    c0 = _rand(512, 256, gen=g, dev=dev)
    out = c0.clone()
    gemm.linear(x, w, out=out, accumulate=True)
    assert _err(out, c0.float() + x.float() @ w.float().T) < BF16_TOL
    acc = torch.randn(256, 128, device=dev, generator=g)
    dy = _rand(1024, 256, gen=g, dev=dev)
    xx = _rand(1024, 128, gen=g, dev=dev)
    ref = acc + dy.float().T @ xx.float()
    gemm.matmul_tn(dy, xx, out=acc, accumulate=True)
    assert _err(acc, ref) < FP32_TOL


def test_deterministic_split_k():
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: split-K determinism", flush=True)
    g = torch.Generator(device=dev).manual_seed(11)
    a, b = _rand(32768, 512, gen=g, dev=dev), _rand(32768, 1408, gen=g, dev=dev)
    torch.testing.assert_close(gemm.matmul_tn(a, b), gemm.matmul_tn(a, b), rtol=0, atol=0)


def test_project_matches_fp32_linear():
    """The bf16 projection autograd function (shared-input layers in one GEMM) vs fp32 F.linear on the same
    bf16-rounded input: output, input gradient, fp32 weight and bias gradients."""
    from llattn_amd.linear import project
    dev = require_cuda()
    print("case: project", flush=True)
    torch.manual_seed(0)
    l1, l2 = torch.nn.Linear(256, 384).to(dev), torch.nn.Linear(256, 64).to(dev)
    x = torch.randn(2, 512, 256, device=dev).to(torch.bfloat16).requires_grad_(True)
    dy = torch.randn(2, 512, 448, device=dev)
    with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
        y = project(x, l1, l2)
    y.backward(dy.to(y.dtype))
    xr = x.detach().float().requires_grad_(True)
    # fp32 leaves holding the bf16-rounded weights, so the reference gradients are not rounded to bf16
    wr = torch.cat([l1.weight, l2.weight]).detach().to(torch.bfloat16).float().requires_grad_(True)
    br = torch.cat([l1.bias, l2.bias]).detach().to(torch.bfloat16).float().requires_grad_(True)
    yr = torch.nn.functional.linear(xr, wr, br)
    yr.backward(dy.to(torch.bfloat16).float())
    assert y.dtype == torch.bfloat16 and l1.weight.grad.dtype == torch.float32
    assert _err(y, yr) < BF16_TOL
    assert _err(x.grad, xr.grad) < BF16_TOL
    assert _err(torch.cat([l1.weight.grad, l2.weight.grad]), wr.grad) < 1e-3
    assert _err(torch.cat([l1.bias.grad, l2.bias.grad]), br.grad) < 1e-3


def test_project_with_pools_matches_fp32():
    """Poolings that ride on the projection: forward values and the input gradient, which sums the
    projection's and both poolings' gradients in place (ragged last segment in the second pooling)."""
    from llattn_amd import _lib as L
    from llattn_amd.linear import project
    dev = require_cuda()
    print("case: project+pools", flush=True)
    torch.manual_seed(1)
    lin = torch.nn.Linear(256, 320).to(dev)
    B, T, K = 2, 512, 256
    x = torch.randn(B, T, K, device=dev).to(torch.bfloat16).requires_grad_(True)
    pools = [(64, 8, L.DIV_COUNT), (100, 6, L.DIV_SEG)]
    with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
        y, p1, p2 = project(x, lin, pools=pools)
    dy = torch.randn_like(y, dtype=torch.float32).to(torch.bfloat16)
    d1 = torch.randn_like(p1, dtype=torch.float32).to(torch.bfloat16)
    d2 = torch.randn_like(p2, dtype=torch.float32).to(torch.bfloat16)
    torch.autograd.backward([y, p1, p2], [dy, d1, d2])

    xr = x.detach().float().requires_grad_(True)
    wr = lin.weight.detach().to(torch.bfloat16).float()
    br = lin.bias.detach().to(torch.bfloat16).float()
    yr = torch.nn.functional.linear(xr, wr, br)
    r1 = xr.view(B, 8, 64, K).mean(2)
    pad = torch.nn.functional.pad(xr, (0, 0, 0, 600 - T))
    r2 = pad.view(B, 6, 100, K).sum(2) / 100
    torch.autograd.backward([yr, r1, r2], [dy.float(), d1.float(), d2.float()])
    assert _err(y, yr) < BF16_TOL
    assert _err(p1, r1) < BF16_TOL and _err(p2, r2) < BF16_TOL
    assert _err(x.grad, xr.grad) < BF16_TOL


@pytest.mark.parametrize("sizes", [[(4224, 1408), (512, 1408)], [(5,), (13,), (1029,)], [(7,)] * 11])
def test_pack_params_matches_torch_casts(sizes):
    """llattn_cast through pack_params: bf16 groups equal torch.cat(...).to(bfloat16) bit for bit (round to
    nearest even), fp32 groups equal the concatenation; lengths that are not multiples of 8 and more than 8
    arrays (two launches) included."""
    from llattn_amd.linear import pack_params
    dev = require_cuda()
    print("case: pack", sizes, flush=True)
    g = torch.Generator(device=dev).manual_seed(len(sizes))
    ts = [torch.randn(*s, device=dev, generator=g) * 3.0 for s in sizes]
    ts[0].view(-1)[:4] = torch.tensor([1.0 + 2 ** -8, 1.0 + 3 * 2 ** -8, -2.5e-39, float("inf")], device=dev)
    half = len(ts) // 2 or 1
    groups = [(ts[:half], torch.bfloat16)] + ([(ts[half:], torch.float32)] if ts[half:] else [])
    outs = pack_params(groups)
    assert torch.equal(outs[0].view(torch.int16), torch.cat(ts[:half]).to(torch.bfloat16).view(torch.int16))
    if ts[half:]:
        assert torch.equal(outs[1], torch.cat(ts[half:]))


@pytest.mark.parametrize("sizes", [
    [(4224, 1408), (512, 1408)],   # config 2's qkv | rq weights: two segments of one W^T
    [(1408, 512)],                 # r_out
    [(8, 72), (200, 72), (64, 72)],  # ragged 64-tiles, an 8-row segment
    [(12, 16)],                    # rows not a multiple of 8: no transposed copy
    [(64, 64)] * 9,                # more than 8 segments: two launches
])
def test_pack_params_transposed_copy(sizes):
    """llattn_cast_transposed through pack_params: the cast and its transposed copy equal torch's
    .to(bfloat16) and .t().contiguous() bit for bit, next to a plain bf16 group and an fp32 group in the same
    launch; with rows that are not multiples of 8 the pair carries None."""
    from llattn_amd.linear import pack_params
    dev = require_cuda()
    print("case: pack transposed", sizes, flush=True)
    g = torch.Generator(device=dev).manual_seed(7 + len(sizes))
    ts = [torch.randn(*s, device=dev, generator=g) * 3.0 for s in sizes]
    ts[0].view(-1)[:4] = torch.tensor([1.0 + 2 ** -8, 1.0 + 3 * 2 ** -8, -2.5e-39, float("inf")], device=dev)
    plain = [torch.randn(37, device=dev, generator=g)]
    bias = [torch.randn(24, device=dev, generator=g)]
    (w, w_t), wp, b = pack_params([(ts, torch.bfloat16, True), (plain, torch.bfloat16), (bias, torch.float32)])
    ref = torch.cat(ts).to(torch.bfloat16)
    assert torch.equal(w.view(torch.int16), ref.view(torch.int16))
    if all(s[0] % 8 == 0 and s[1] % 8 == 0 for s in sizes):
        assert w_t is not None and w_t.is_contiguous()
        assert torch.equal(w_t.view(torch.int16), ref.t().contiguous().view(torch.int16))
    else:
        assert w_t is None
    assert torch.equal(wp.view(torch.int16), plain[0].to(torch.bfloat16).view(torch.int16))
    assert torch.equal(b, bias[0])


def _gelu_and_grad(u):
    uu = u.float().requires_grad_(True)
    g = torch.nn.functional.gelu(uu)
    g.backward(torch.ones_like(g))
    return g.detach(), uu.grad


@pytest.mark.parametrize("M,N,K", [(32768, 4096, 1408), (300, 264, 200), (97, 40, 64)])
def test_linear_gelu_epilogue(M, N, K):
    """LLATTN_ACT_GELU: gelu and gelu' of the bf16-rounded pre-activation from one GEMM, against torch's F.gelu
    and its backward on the bf16-rounded fp32 product (small M takes the split-K reduction)."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: linear gelu", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(M + 2 * N + K)
    x, w = _rand(M, K, gen=g, dev=dev), _rand(N, K, gen=g, dev=dev) * 0.1
    b = torch.randn(N, device=dev, generator=g) * 0.5
    got_g, got_gp = gemm.linear_gelu(x, w, b)
    ref_g, ref_gp = _gelu_and_grad((x.float() @ w.float().T + b).to(torch.bfloat16))
    for got, ref in ((got_g, ref_g), (got_gp, ref_gp)):
        assert got.dtype == torch.bfloat16
        assert _err(got, ref) < BF16_TOL
        # one bf16 rounding of the result, plus the rare pre-activation that rounds to the neighbouring bf16
        assert float((got.float() - ref).abs().mean()) < 2 ** -8 * float(ref.abs().mean())


@pytest.mark.parametrize("M,N,K", [(32768, 4096, 1408), (300, 264, 200), (97, 40, 64)])
def test_matmul_nn_scaled_epilogue(M, N, K):
    """LLATTN_ACT_MUL_AUX: bf16(dy W) * s elementwise, against torch on the bf16-rounded product."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: nn scaled", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(3 * M + N + K)
    a, b = _rand(M, K, gen=g, dev=dev), _rand(K, N, gen=g, dev=dev) * 0.1
    sc = _rand(M, N, gen=g, dev=dev)
    got = gemm.matmul_nn_scaled(a, b, sc)
    ref = (a.float() @ b.float()).to(torch.bfloat16).float() * sc.float()
    assert _err(got, ref) < BF16_TOL


def test_feed_forward_matches_fp32_reference():
    """The LM's FeedForward under bf16 autocast (GELU in the GEMM epilogues) against fp32 w2(gelu(w1 x)) on the
    same bf16-rounded input and weights: output, input gradient, weight and bias gradients."""
    from llattn_amd.ffn import feed_forward
    dev = require_cuda()
    print("case: feed forward", flush=True)
    torch.manual_seed(2)
    w1, w2 = torch.nn.Linear(256, 1024).to(dev), torch.nn.Linear(1024, 256).to(dev)
    x = torch.randn(2, 300, 256, device=dev).to(torch.bfloat16).requires_grad_(True)
    dy = torch.randn(2, 300, 256, device=dev)
    with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
        y = feed_forward(x, w1, w2)
    y.backward(dy.to(y.dtype))
    xr = x.detach().float().requires_grad_(True)
    p = {n: t.detach().to(torch.bfloat16).float().requires_grad_(True)
         for n, t in (("w1", w1.weight), ("b1", w1.bias), ("w2", w2.weight), ("b2", w2.bias))}
    yr = torch.nn.functional.linear(torch.nn.functional.gelu(torch.nn.functional.linear(xr, p["w1"], p["b1"])),
                                    p["w2"], p["b2"])
    yr.backward(dy.to(torch.bfloat16).float())
    assert y.dtype == torch.bfloat16
    assert _err(y, yr) < BF16_TOL
    assert _err(x.grad, xr.grad) < BF16_TOL
    for got, name in ((w1.weight.grad, "w1"), (w1.bias.grad, "b1"), (w2.weight.grad, "w2"), (w2.bias.grad, "b2")):
        assert got.dtype == torch.float32
        assert _err(got, p[name].grad) < 2e-2, name


@pytest.mark.parametrize("R,C", [(1408, 1408), (4736, 1408), (8, 16), (200, 72)])
def test_transpose_bf16(R, C):
    """llattn_transpose is an exact copy: bitwise equal to torch's transpose (ragged 64-tiles included)."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: transpose", R, C, flush=True)
    g = torch.Generator(device=dev).manual_seed(R + C)
    w = _rand(R, C, gen=g, dev=dev)
    assert torch.equal(gemm.transpose(w), w.t().contiguous())


@pytest.mark.parametrize("M,N,K", [(32768, 1408, 1408), (32768, 512, 1408), (4096, 1408, 4096), (300, 264, 128)])
def test_input_grad_through_transposed_weight(M, N, K):
    """dy @ w through the persistent kernel and a transposed weight (large M) or the tiled kernel (small M)."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: input grad", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(M + 3 * N + K)
    dy, w = _rand(M, K, gen=g, dev=dev), _rand(K, N, gen=g, dev=dev)
    assert _err(gemm.input_grad(dy, w), dy.float() @ w.float()) < BF16_TOL


@pytest.mark.parametrize("B,T,N,K,pools,bitwise", [
    (16, 2048, 1408, 4736, [(128, 0)], True),          # config 2: the qkv input gradient with the latent pooling
    (4, 2000, 520, 264, [(64, 0), (100, 1)], True),    # ragged segments, two addends, K with a 64-wide tail
    (2, 4096, 136, 1024, [(512, 2)], False),           # 32 tiles: the tiled kernel splits K here
])
def test_input_grad_rowadd_persistent_equals_tiled(B, T, N, K, pools, bitwise):
    """The input gradient with pooled-gradient row addends through the transposed weight and the persistent
    kernel matches fp32 torch, and gives the same bits as the tiled kernel with transposing fragment reads
    wherever that one does not split K (same k order, same epilogue arithmetic)."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: input grad rowadd persistent", B, T, N, K, pools, flush=True)
    g = torch.Generator(device=dev).manual_seed(B * T + N + K)
    dy, w = _rand(B * T, K, gen=g, dev=dev), _rand(K, N, gen=g, dev=dev)
    ref = dy.float() @ w.float()
    rowadd = []
    t = torch.arange(T, device=dev)
    for seg, div in pools:
        n_seg = -(-T // seg)
        rows = _rand(B * n_seg, N, gen=g, dev=dev) * 4
        s_id = t // seg
        count = torch.minimum((s_id + 1) * seg, torch.full_like(s_id, T)) - s_id * seg
        scale = {0: 1.0 / count.float(), 1: torch.full((T,), 1.0 / seg, device=dev), 2: torch.ones(T, device=dev)}[div]
        ref = ref + (rows.float().view(B, n_seg, N)[:, s_id] * scale[None, :, None]).reshape(B * T, N)
        rowadd.append((rows, T, seg, n_seg, div))
    got = gemm.input_grad(dy, w, rowadd=rowadd)
    if bitwise:
        assert torch.equal(got, gemm.matmul_nn(dy, w, rowadd=rowadd))
    assert _err(got, ref) < BF16_TOL


# ---- split-head operands (llattn_heads_layout): the q|k|v projection output stored as head slabs ----

def _to_heads(x: torch.Tensor, T: int, dh: int, n: int, tdh: int = 0) -> torch.Tensor:
    """Row-major [B T, W] -> the same matrix in split-head storage, as a [B T, W] tensor: the first n dh
    columns as [B][n][T][dh] slabs, then the other columns packed [B T][W - n dh] (tdh = 0) or as
    [B][(W - n dh) / tdh][T][tdh] slabs (torch permute, independent of the kernels' offset arithmetic)."""
    R, W = x.shape
    B, c = R // T, n * dh
    head = x[:, :c].reshape(B, T, n, dh).permute(0, 2, 1, 3).reshape(-1)
    rest = x[:, c:]
    if tdh:
        rest = rest.reshape(B, T, (W - c) // tdh, tdh).permute(0, 2, 1, 3)
    return torch.cat([head, rest.reshape(-1)]).view(R, W)


def _from_heads(s: torch.Tensor, T: int, dh: int, n: int, tdh: int = 0) -> torch.Tensor:
    R, W = s.shape
    B, c = R // T, n * dh
    flat = s.reshape(-1)
    head = flat[:R * c].view(B, n, T, dh).permute(0, 2, 1, 3).reshape(R, c)
    rest = flat[R * c:]
    rest = rest.view(B, (W - c) // tdh, T, tdh).permute(0, 2, 1, 3).reshape(R, W - c) if tdh else rest.view(R, W - c)
    return torch.cat([head, rest], dim=1)


HEADS_CASES = [  # (B, T, dh, n, tail, K, tdh): head columns n dh, plus `tail` columns (packed, or as slabs of tdh
    # columns); K the contraction
    (2, 160, 32, 6, 64, 192, 0),
    (3, 97, 88, 12, 0, 136, 0),      # T not a multiple of 32 or 256: slabs start inside tiles and k steps
    (2, 300, 16, 6, 512, 256, 0),
    (1, 64, 64, 3, 8, 72, 0),
    (16, 2048, 88, 48, 512, 1408, 0),  # config 2's q|k|v|rq with the latent queries packed
    (2, 160, 32, 6, 64, 192, 16),
    (3, 97, 88, 12, 96, 136, 24),    # tail slabs that start inside tiles, heads not a multiple of 16 wide
    (2, 300, 16, 6, 512, 256, 64),
    (16, 2048, 88, 48, 512, 1408, 64),  # config 2: q|k|v|rq of the 0.55b layer
    (16, 2048, 64, 8, 0, 1408, 0),   # config 2: the latent output's gradient as Lh slabs
]


@pytest.mark.parametrize("case", HEADS_CASES)
def test_linear_split_head_output(case):
    """The persistent kernel's stores in split-head order: the same product as the row-major output."""
    from llattn_amd import gemm
    B, T, dh, n, tail, K, tdh = case
    dev = require_cuda()
    print("case: linear split-head C", case, flush=True)
    g = torch.Generator(device=dev).manual_seed(B * T + dh + n + tail + tdh)
    M, N = B * T, n * dh + tail
    x, w = _rand(M, K, gen=g, dev=dev), _rand(N, K, gen=g, dev=dev)
    b = torch.randn(N, device=dev, generator=g)
    got = gemm.linear(x, w, b, heads=(T, dh, n, tdh))
    assert _err(_from_heads(got, T, dh, n, tdh), x.float() @ w.float().T + b) < BF16_TOL
    if M * N >= 1 << 24:  # both on the persistent kernel: only the store order differs
        assert torch.equal(got, _to_heads(gemm.linear(x, w, b), T, dh, n, tdh))


def test_input_grad_split_head_output():
    """The input gradient on the persistent kernel stored as head slabs (the latent output's gradient of
    config 2, [B][Lh][n_q][Ldh]): the same bits as the row-major input gradient (256 output tiles: unsplit on
    the persistent kernel too), permuted; the small-M route refuses a split-head output."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: input_grad split-head", flush=True)
    g = torch.Generator(device=dev).manual_seed(5)
    B, T, Lh, Ldh, D = 16, 2048, 8, 64, 1408
    dy, w = _rand(B * T, D, gen=g, dev=dev), _rand(D, Lh * Ldh, gen=g, dev=dev)
    plain = gemm.input_grad(dy, w)
    got = gemm.input_grad(dy, w, heads=(T, Ldh, Lh))
    assert torch.equal(got, _to_heads(plain, T, Ldh, Lh))
    assert _err(plain, dy.float() @ w.float()) < BF16_TOL
    with pytest.raises(ValueError, match="persistent"):
        gemm.input_grad(dy[:1024], w, heads=(1024, Ldh, Lh))


@pytest.mark.parametrize("M,N,K", [(1, 8, 1), (97, 40, 64), (64, 64, 16), (300, 264, 1000), (33, 130, 37),
                                   (2048, 1408, 256), (256, 1024, 1408)])
def test_gemm_f32_products(M, N, K):
    """The fp32 products of llattn_gemm_f32 against float64 CPU references: x W^T + b, dy W (through a strided
    view of W), dy^T x with the row sums of dy^T (the bias gradient), and accumulation into C; ragged tiles
    and contraction lengths that are not multiples of 4 or 16 included."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: gemm f32", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(M * 7 + N + K)
    x = torch.randn(M, K, device=dev, generator=g)
    w_full = torch.randn(N, K + 8, device=dev, generator=g)
    w = w_full[:, :K]  # leading dimension K + 8
    b = torch.randn(N, device=dev, generator=g)
    ref = (x.double() @ w.double().T + b.double()).float()
    assert _err(gemm.linear_f32(x, w, b), ref) < 1e-5
    dy = torch.randn(M, N, device=dev, generator=g)
    assert _err(gemm.matmul_nn_f32(dy, w), (dy.double() @ w.double()).float()) < 1e-5
    rs = torch.full((N,), float("nan"), device=dev)
    dw = gemm.matmul_tn_f32(dy, x, rowsum=rs)
    assert _err(dw, (dy.double().T @ x.double()).float()) < 1e-5
    assert _err(rs, dy.double().sum(0).float()) < 1e-5
    assert torch.equal(dw, gemm.matmul_tn_f32(dy, x))  # the same products with and without the row sums
    out = torch.randn(M, N, device=dev, generator=g)
    ref_acc = out.double() + x.double() @ w.double().T
    gemm._run_f32(M, N, K, x, False, w, False, out, accumulate=True)
    assert _err(out, ref_acc.float()) < 1e-5



@pytest.mark.parametrize("M,N,K", [
    (1, 1, 1), (3, 5, 7), (31, 33, 17), (32, 32, 16), (65, 130, 257), (128, 1, 48),  # register tiles, every edge
    (40, 24, 600), (33, 2, 4100),                                # split over waves; pieces of 16 bytes cut by N = 2
    (1024, 800, 256), (260, 1028, 100), (2052, 516, 36),          # LDS tiles of 64 x 64, k tails of 4 in 32
    (1000, 512, 1408), (1000, 1412, 520), (1400, 516, 1000),      # two and four k groups, 64 x 32 tiles
    (2049, 1089, 70), (1500, 2000, 65)])                          # at odd strides: staged 64 x 64 tiles
def test_gemm_f32_kernels_and_layouts(M, N, K):
    """The fp32 kernels and every operand layout (A and B k- or m/n-contiguous, aligned and at odd strides and
    offsets) against float64.  The K roundings of partial sums of unit products, each up to 2^-24 of a partial of
    size sqrt(k), add up to about 2^-24 K / 2, where the terms' absolute values sum to 0.64 K: an error of about
    2^-24 of that sum, which (unlike the result) cannot cancel.  Four times that is allowed."""
    from llattn_amd import gemm
    dev = require_cuda()
    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 7 * K)
    tol = 4 * 2.0 ** -24

    def off(got, ref, terms):
        return float((got.double() - ref).norm() / terms.norm())

    def view(rows, cols, pad, start):  # a matrix of the values of its storage from (start, start) on
        full = torch.randn(rows + start, cols + start + pad, device=dev, generator=g)
        return full[start:, start:start + cols]

    for pad, start in ((0, 0), (4, 4), (3, 1)):
        for a_trans in (False, True):
            for b_trans in (False, True):
                print("case: gemm f32 layouts", M, N, K, pad, start, a_trans, b_trans, flush=True)
                a = view(K, M, pad, start) if a_trans else view(M, K, pad, start)
                b = view(K, N, pad, start) if b_trans else view(N, K, pad, start)
                a64, b64 = (a.t() if a_trans else a).double(), (b if b_trans else b.t()).double()
                bias = torch.randn(N, device=dev, generator=g)
                out = torch.full((M, N), float("nan"), device=dev)
                rs = torch.full((M,), float("nan"), device=dev)
                gemm._run_f32(M, N, K, a, a_trans, b, b_trans, out, bias=bias, rowsum=rs)
                assert off(out, a64 @ b64 + bias.double(), a64.abs() @ b64.abs() + bias.double().abs()) < tol
                assert off(rs, a64.sum(1), a64.abs().sum(1)) < tol
                again = torch.full((M, N), float("nan"), device=dev)
                gemm._run_f32(M, N, K, a, a_trans, b, b_trans, again, bias=bias)
                assert torch.equal(out, again)


def test_gemm_f32_wide_strides():
    """Rows past K at a stride whose byte offsets pass 2^32 within a stage of 32 k do not come back as other rows:
    the row sums of A are those of its K rows."""
    from llattn_amd import gemm
    dev = require_cuda()
    M, N, K, ld = 3072, 1024, 20, 50_000_000
    print("case: gemm f32 wide strides", flush=True)
    g = torch.Generator(device=dev).manual_seed(1)
    a = torch.ones((K - 1) * ld + M, device=dev).as_strided((K, M), (ld, 1))
    a.copy_(torch.randn(K, M, device=dev, generator=g))
    b = torch.randn(K, N, device=dev, generator=g)
    out, rs = torch.empty(M, N, device=dev), torch.empty(M, device=dev)
    gemm._run_f32(M, N, K, a, True, b, True, out, rowsum=rs)
    assert _err(out, (a.double().T @ b.double()).float()) < 1e-5
    assert _err(rs, a.double().sum(0).float()) < 1e-5


def test_gemm_f32_grid_of_many_tiles():
    """An output of nine million 32 x 32 tiles (the odd K in rows of 256 keeps it off the direct-to-LDS ones): with
    eight waves each they would pass the 2^32 threads that a grid holds, and the last tiles would stay unwritten."""
    from llattn_amd import gemm
    dev = require_cuda()
    M, N, K = 8_700_000, 1025, 255
    print("case: gemm f32 many tiles", flush=True)
    g = torch.Generator(device=dev).manual_seed(1)
    a, b = torch.randn(M, K + 1, device=dev, generator=g)[:, :K], torch.randn(N, K + 1, device=dev, generator=g)[:, :K]
    out = gemm.linear_f32(a, b)
    for r in (slice(0, 64), slice(M // 2, M // 2 + 64), slice(M - 64, M)):
        ref, mag = a[r].double() @ b.double().T, a[r].double().abs() @ b.double().abs().T
        assert ((out[r] - ref).abs() <= K * 2.0 ** -24 * mag).all()


def test_gemm_wide_strides():
    """The same for the bf16 kernels (64 k rows per stage; 64 x 64 and 128 x 128 tiles, 256 x 256 ones with row sums of
    their own or from a column of ones): NaN everywhere between the operands' rows reaches neither the products nor
    the row sums.  fp32 sums of K = 24 terms: K * 2^-24 of the sum of magnitudes."""
    from llattn_amd import gemm
    dev = require_cuda()
    K, ld = 24, 50_000_000
    base = torch.full(((K - 1) * ld + 16384,), float("nan"), device=dev, dtype=torch.bfloat16)
    g = torch.Generator(device=dev).manual_seed(1)
    for M, N in ((512, 320), (3072, 1024), (3072, 2056), (4096, 4096), (4096, 4104)):
        print("case: gemm wide strides", M, N, flush=True)
        a, b = base.as_strided((K, M), (ld, 1)), base.as_strided((K, N), (ld, 1), 8192)
        for t in (a, b):
            t.copy_(torch.randn(t.shape, device=dev, generator=g))
        A, B = a.double(), b.double()
        rs = torch.empty(M, device=dev)
        out = gemm.matmul_tn(a, b, rowsum=rs)
        assert ((out - A.T @ B).abs() <= K * 2.0 ** -24 * (A.abs().T @ B.abs())).all()
        assert ((rs - A.sum(0)).abs() <= K * 2.0 ** -24 * A.abs().sum(0)).all()
        x = torch.randn(M, K, device=dev, generator=g).bfloat16()
        X = x.double()
        tol = (2.0 ** -8) * (X @ B).abs() + 2 * K * 2.0 ** -24 * (X.abs() @ B.abs())
        assert ((gemm.matmul_nn(x, b) - X @ B).abs() <= tol).all()
        base.as_strided((K, 16384), (ld, 1)).fill_(float("nan"))


@pytest.mark.parametrize("M,K,N", [(4096, 72, 8), (4099, 128, 264), (8200, 256, 1040), (16384, 64, 2048), (4096, 4096, 4096)])
def test_scaled_input_grad_through_the_transpose(M, K, N):
    """``matmul_nn_scaled`` with the transposed copy (the persistent kernel's MUL_AUX epilogue, or its split-K
    counterpart where the tiles are few): within the two bf16 roundings (2 x 2^-9) and the fp32 sum of the float32
    product, and where neither route splits K the same bits as the route through the untransposed operand."""
    from llattn_amd import gemm
    dev = require_cuda()
    print("case: scaled input grad", M, K, N, flush=True)
    g = torch.Generator(device=dev).manual_seed(M + K + N)
    dy = torch.randn(M, K, device=dev, generator=g).bfloat16()
    w = torch.randn(K, N, device=dev, generator=g).bfloat16()
    s = torch.randn(M, N, device=dev, generator=g).bfloat16()
    got = gemm.matmul_nn_scaled(dy, w, s, gemm.transpose(w))
    ref = (dy.float() @ w.float()) * s.float()
    assert float((got.float() - ref).norm() / ref.norm()) < 2 * 2.0 ** -9
    if ((M + 255) // 256) * ((N + 255) // 256) >= 224:
        assert torch.equal(got, gemm.matmul_nn_scaled(dy, w, s))


@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (64, 64, 64), (264, 136, 72), (72, 136, 200), (1000, 520, 328),
                                   (1000, 1416, 328), (1000, 4104, 264), (1000, 4104, 1032), (1024, 4096, 1408),
                                   (1288, 72, 4008),
                                   # split over workgroups: few tiles, a k tail in the last of 2, 16 and 32 ranges
                                   (72, 136, 6152), (24, 64, 8200), (264, 520, 8264), (136, 128, 16392)])
def test_gemm_tiles_layouts_and_epilogues(M, N, K):
    """The smaller tiles (64 x 64 and 128 x 128, one and two k groups, split over workgroups): every operand layout at strides of its own,
    into bf16 and fp32, with bias, accumulation, row addends, the activations, split-head storage and row sums,
    against float64, element by element.  fp32: 2^-20 of the sum of the terms' absolute values (an fp32 sum's typical
    error is 2^-24 of it; the largest of millions of elements is several times that); bf16: 2^-8 of the result more,
    twice a rounding's 2^-9."""
    from llattn_amd import _lib as L
    from llattn_amd import gemm
    dev = require_cuda()
    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 7 * K)

    def rnd(rows, cols, pad=8):
        return torch.randn(rows, cols + pad, device=dev, generator=g).bfloat16()[:, :cols]

    def near(got, ref, terms, roundings):
        off = (got.double() - ref).abs()
        return bool((off <= roundings * 2.0 ** -8 * ref.abs() + 2.0 ** -20 * terms).all())

    bias = torch.randn(N, device=dev, generator=g)
    for a_trans in (False, True):
        for b_trans in (False, True):
            print("case: gemm tiles", M, N, K, a_trans, b_trans, flush=True)
            a = rnd(K, M) if a_trans else rnd(M, K)
            b = rnd(K, N) if b_trans else rnd(N, K)
            a64, b64 = (a.t() if a_trans else a).double(), (b if b_trans else b.t()).double()
            ref, terms = a64 @ b64, a64.abs() @ b64.abs() + 8
            out = torch.full((M, N), float("nan"), device=dev, dtype=torch.bfloat16)
            gemm._run(M, N, K, a, a_trans, b, b_trans, out, bias, False)
            assert near(out, ref + bias.double(), terms, 1)
            plain = torch.empty_like(out)
            gemm._run(M, N, K, a, a_trans, b, b_trans, plain, None, False)
            start = rnd(M, N, 0)
            acc = start.clone()
            gemm._run(M, N, K, a, a_trans, b, b_trans, acc, None, True)
            assert near(acc, ref + start.double(), terms, 1)
            f = torch.full((M, N), float("nan"), device=dev)
            rs = torch.full((M,), float("nan"), device=dev) if b_trans and (N % 256 or a_trans) else None
            gemm._run(M, N, K, a, a_trans, b, b_trans, f, bias, False, rowsum=rs)
            assert near(f, ref + bias.double(), terms, 0)
            if rs is not None:
                assert near(rs, a64.sum(1), a64.abs().sum(1) + 8, 0)
            f2 = f.clone()
            gemm._run(M, N, K, a, a_trans, b, b_trans, f2, None, True)
            assert near(f2, 2 * ref + bias.double(), 2 * terms, 0)
            if a_trans:
                continue
            aux = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
            gl = torch.empty_like(out)
            gemm._run(M, N, K, a, a_trans, b, b_trans, gl, bias, False, act=L.ACT_GELU, aux=aux)
            h = out.double()
            phi = 0.5 * (1 + torch.erf(h / 2 ** 0.5))
            assert near(gl, h * phi, h.abs() + 8, 1)
            assert near(aux, phi + h * torch.exp(-h * h / 2) / (2 * torch.pi) ** 0.5, torch.full_like(h, 8), 1)
            sc = rnd(M, N, 0)
            gemm._run(M, N, K, a, a_trans, b, b_trans, gl, None, False, act=L.ACT_MUL_AUX, aux=sc)
            assert torch.equal(gl, (plain.float() * sc.float()).bfloat16())
            if b_trans:
                seg, T = 24, M // 2
                n = -(-T // seg)
                rows = rnd(2 * n, N, 0)
                add = rows.view(2, n, N).double().repeat_interleave(seg, 1)[:, :T].reshape(M, N) / seg
                gemm._run(M, N, K, a, a_trans, b, b_trans, gl, None, False, rowadd=[(rows, T, seg, n, L.DIV_SEG)])
                assert near(gl, ref + add, terms, 1)
            elif M % 2 == 0:  # two sequences, heads of 8 columns over half the width, the rest in slabs of 8
                heads = N // 16
                st = torch.empty(M * N, device=dev, dtype=torch.bfloat16).view(M, N)
                gemm._run(M, N, K, a, a_trans, b, b_trans, st, None, False, c_heads=(M // 2, 8, heads, 8) if heads else (M // 2, 8, 1, 0))
                flat, cols = st.view(-1), 8 * max(heads, 1)
                got = flat[:M * cols].view(2, -1, M // 2, 8).transpose(1, 2).reshape(M, cols)
                assert torch.equal(got, plain[:, :cols])
                if heads:
                    tail = flat[M * cols:].view(2, -1, M // 2, 8).transpose(1, 2).reshape(M, N - cols)
                    assert torch.equal(tail, plain[:, cols:])


# (layouts, first product (M, N, K), second): two shapes of each tile and k-group plan, in this order: 64 x 64 with one k
# group, with two, 128 x 128
PAIRS = [("fwd", (401, 24, 8), (155, 1112, 8)), ("fwd", (1066, 1960, 296), (265, 1176, 296)),
         ("fwd", (29, 192, 376), (165, 16, 376)), ("fwd", (1088, 288, 800), (318, 696, 800)),
         ("fwd", (2003, 3720, 928), (391, 80, 928)),
         ("w_t", (27, 64, 32), (32, 64, 27)), ("w_t", (706, 2400, 720), (720, 2400, 706)),
         ("w_t", (493, 8, 200), (200, 8, 493)), ("w_t", (619, 880, 448), (448, 880, 619)),
         ("w_t", (1029, 2944, 1080), (1080, 2944, 1029)),
         ("w", (660, 8, 8), (8, 8, 660)), ("w", (710, 2184, 776), (776, 2184, 710)),
         ("w", (309, 16, 472), (472, 16, 309)), ("w", (1327, 872, 224), (224, 872, 1327)),
         ("w", (1203, 2704, 1096), (1096, 2704, 1203)), ("w", (4096, 4096, 64), (64, 4096, 4096))]  # the last: one by one


@pytest.mark.parametrize("kind,s0,s1", PAIRS)
def test_gemm_pair(kind, s0, s1):
    """Two independent products in one launch: two x W^T, or an input gradient (through W^T or W) with the weight
    gradient and its row sums, at ragged sizes and strides of their own, with bias, row addends, an elementwise factor
    and split-head storage, element by element against float64 (bounds as for the smaller tiles above)."""
    import ctypes
    from llattn_amd import _lib as L
    dev = require_cuda()
    g = torch.Generator(device=dev).manual_seed(sum(s0) + 3 * sum(s1))
    ref = ctypes.byref

    def rnd(rows, cols, pad=8):
        return torch.randn(rows, cols + pad, device=dev, generator=g).bfloat16()[:, :cols]

    def near(got, want, terms, roundings):
        return bool(((got.double() - want).abs() <= roundings * 2.0 ** -8 * want.abs() + 2.0 ** -20 * terms).all())

    def product(s, a_trans, b_trans, dtype, bias=None):
        M, N, K = s
        a, b = rnd(K, M) if a_trans else rnd(M, K), rnd(K, N) if b_trans else rnd(N, K)
        out = torch.full((M, N), float("nan"), device=dev, dtype=dtype)
        d = L.LlattnGemmDesc(M, N, K, int(a_trans), int(b_trans), a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0),
                             out.data_ptr(), N, L.dtype_code(dtype), 0, None if bias is None else bias.data_ptr(), 0, None)
        A, B = (a.t() if a_trans else a).double(), (b if b_trans else b.t()).double()
        want, terms = A @ B, A.abs() @ B.abs() + 8
        return d, (a, b), out, want if bias is None else want + bias.double(), terms

    for extra in ("plain", "heads" if kind != "w" else "plain", "scaled", "rowadd" if kind != "fwd" else "plain"):
        print("case: gemm pair", kind, s0, s1, extra, flush=True)
        M, N, K = s0
        bias = torch.randn(N, device=dev, generator=g) if kind == "fwd" else None
        d0, keep0, o0, w0, t0 = product(s0, False, kind == "w", torch.bfloat16, bias)
        b1 = torch.randn(s1[1], device=dev, generator=g) if kind == "fwd" else None
        d1, keep1, o1, w1, t1 = product(s1, kind != "fwd", kind != "fwd", torch.bfloat16 if kind == "fwd" else torch.float32, b1)
        rs = torch.full((s1[0],), float("nan"), device=dev)
        if kind != "fwd":
            d1.a_rowsum = rs.data_ptr()
        roundings = 1
        if extra == "scaled":
            aux = rnd(M, N, 0)
            d0.act, d0.aux, d0.ld_aux = L.ACT_MUL_AUX, aux.data_ptr(), N
            w0, t0, roundings = w0 * aux.double(), t0 * (aux.double().abs() + 1), 2
        elif extra == "heads":
            d0.c_heads = L.LlattnHeadsLayout(M, 8, N // 8, 0)
        elif extra == "rowadd":
            seg = 5
            n = -(-M // seg)
            rows = rnd(n, N, 0)
            d0.rowadd[0] = L.LlattnGemmRowadd(rows.data_ptr(), N, M, seg, n, L.DIV_SEG)
            w0 = w0 + rows.double().repeat_interleave(seg, 0)[:M] / seg
        lib = L.load()
        nws = lib.llattn_gemm_pair_workspace_size(ref(d0), ref(d1))
        ws = torch.empty(max(nws, 16), dtype=torch.uint8, device=dev)
        L.check(lib.llattn_gemm_pair(ref(d0), ref(d1), ws.data_ptr(), nws, L.stream_ptr(dev)), "llattn_gemm_pair")
        if extra == "heads":
            o0 = o0.view(-1).view(N // 8, M, 8).transpose(0, 1).reshape(M, N)
        assert near(o0, w0, t0, roundings), extra
        assert near(o1, w1, t1, 1 if kind == "fwd" else 0), extra
        if kind != "fwd":
            a1 = keep1[0].t().double()
            assert near(rs, a1.sum(1), a1.abs().sum(1) + 8, 0), extra
