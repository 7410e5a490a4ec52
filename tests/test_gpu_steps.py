"""The native steps (one call per direction) against the Python path that issues the same products one by one: the
same bits for every output and gradient, or the same values up to the order of a product's sums where two products
share a launch.  The Python path runs while calls are logged."""
from __future__ import annotations

import contextlib

import pytest
import torch

from gpu_helpers import require_cuda

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _logged():
    from llattn_amd import ops
    ops.EVENT_LOG = []
    try:
        yield ops.EVENT_LOG
    finally:
        ops.EVENT_LOG = None


def _both(fn, entry):
    """fn() by native steps (asserted: ``entry`` is called) and, logged, by the Python path."""
    from llattn_amd import steps
    seen, real = [], steps._call
    steps._call = lambda name, *a: (seen.append(name), real(name, *a))[1]
    try:
        native = fn()
    finally:
        steps._call = real
    assert entry in seen, seen
    with _logged() as log:
        python = fn()
    assert log
    return native, python


def _close(native, python, bf16):
    """Equal up to the order in which a product's fp32 sums are formed.  In fp32 that is 2^-21 of an output's norm; in
    bf16 a sum on a rounding boundary moves an element by one unit, 2^-8 of it at most, here and there, and what is
    computed from it by as much: 2^-9 of the norm."""
    assert len(native) == len(python)
    for i, (a, b) in enumerate(zip(native, python)):
        assert (a is None) == (b is None), i
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape, i
            off, norm = float((a.double() - b.double()).norm()), float(b.double().norm())
            assert off <= (2.0 ** -9 if bf16 else 2.0 ** -21) * norm, (i, off, norm)


def _same(native, python):
    assert len(native) == len(python)
    for i, (a, b) in enumerate(zip(native, python)):
        assert (a is None) == (b is None), i
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), i


BLOCKS = [  # B, T, d_model, heads, latent width, latent heads, window, latents, query block
    (2, 97, 64, 2, 16, 2, 16, 6, 0),      # one small tile, ragged
    (1, 1, 128, 4, 64, 2, 64, 16, 0),     # one token
    (1, 1, 128, 4, 64, 2, 64, 16, 64),    # one token, one query block
    (3, 333, 128, 4, 64, 2, 64, 16, 0),
    (1, 333, 1408, 16, 512, 8, 64, 16, 0),  # two projections in one launch with two k groups
    (2, 640, 256, 4, 32, 2, 128, 10, 64),  # query blocks that are the latent chunks: one pooling
    (2, 650, 256, 4, 32, 2, 300, 10, 48),  # others
    (2, 2100, 256, 4, 128, 2, 64, 16, 0),  # transposed weights (4200 rows), split-head storage
    (16, 1024, 1408, 16, 512, 8, 64, 16, 0),  # gradients stored split-head as well
    (1, 3287, 1536, 16, 384, 8, 64, 16, 0),  # two projections in one launch of 128 x 128 tiles
    (13, 362, 1024, 16, 64, 2, 64, 50, 0),  # an input gradient through its transposed weight beside a weight gradient
]


@pytest.mark.parametrize("cfg", BLOCKS)
@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("bias", [True, False])
def test_block_step_matches_python_path(cfg, bf16, bias):
    from llattn_amd import LocalLatentAttentionTriton
    B, T, D, H, Ld, Lh, W, N, qb = cfg
    if not bf16 and B * T > 5000:
        pytest.skip("the fp32 path has one layout")
    dev = require_cuda()
    print("case: block step", cfg, bf16, bias, flush=True)
    torch.manual_seed(1)
    m = LocalLatentAttentionTriton(D, H, Lh, Ld, N, W, bias=bias, latent_query_block_size=qb).to(dev)
    g = torch.Generator(device=dev).manual_seed(2)
    x = torch.randn(B, T, D, device=dev, generator=g).to(torch.bfloat16 if bf16 else torch.float32)
    dy = torch.randn(B, T, D, device=dev, generator=g).to(x.dtype)

    def cast():
        return torch.autocast("cuda", dtype=torch.bfloat16, enabled=bf16)

    def train(need_dx=True):
        xx = x.clone().requires_grad_(need_dx)
        m.zero_grad(set_to_none=True)
        with cast():
            y = m(xx)
        y.backward(dy)
        return [y.detach(), xx.grad, *(p.grad for p in m.parameters())]

    # fp32: the Python path forms the poolings' input gradients apart and adds them; here they are added in place
    native, python = _both(train, "llattn_block_bwd")
    _close(native, python, bf16)
    _close(*_both(lambda: train(False), "llattn_block_bwd"), bf16)
    _same(train(), native)

    def infer():
        with torch.no_grad(), cast():
            return [m(x)]

    a, b = _both(infer, "llattn_block_fwd")
    _close(a, b, bf16)
    assert torch.equal(a[0], native[0])


def test_block_step_retained_graph_checkpoint_and_streams():
    """Two backward passes of one graph, the block under non-reentrant checkpointing, and a pass on another stream
    give the gradients of a plain pass."""
    from torch.utils.checkpoint import checkpoint
    from llattn_amd import LocalLatentAttentionTriton
    dev = require_cuda()
    torch.manual_seed(3)
    m = LocalLatentAttentionTriton(128, 4, 2, 64, 16, 64).to(dev)
    x = torch.randn(2, 200, 128, device=dev).bfloat16()
    dy = torch.randn_like(x)

    def grads(run):
        xx = x.clone().requires_grad_()
        m.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = run(xx)
        return xx, y

    xx, y = grads(m)
    y.backward(dy, retain_graph=True)
    first = [xx.grad.clone()] + [p.grad.clone() for p in m.parameters()]
    xx.grad = None
    m.zero_grad(set_to_none=True)
    y.backward(dy)
    _same(first, [xx.grad] + [p.grad for p in m.parameters()])
    xx, y = grads(lambda t: checkpoint(m, t, use_reentrant=False))
    y.backward(dy)
    _same(first, [xx.grad] + [p.grad for p in m.parameters()])
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        xx, y = grads(m)
        y.backward(dy)
    torch.cuda.current_stream().wait_stream(s)
    _same(first, [xx.grad] + [p.grad for p in m.parameters()])


def test_block_step_leaves_other_inputs_to_the_python_path():
    """Inputs and parameters that the native step does not take give the results they gave: a strided and a float32
    input under bf16 autocast, a misaligned parameter."""
    from llattn_amd import LocalLatentAttentionTriton, steps
    dev = require_cuda()
    torch.manual_seed(4)
    m = LocalLatentAttentionTriton(128, 4, 2, 64, 16, 64).to(dev)
    x = torch.randn(2, 96, 256, device=dev).bfloat16()
    called, real = [], steps._call
    steps._call = lambda name, *a: (called.append(name), real(name, *a))[1]
    try:
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
            ref = m(x[..., :128].contiguous())
            assert called
            del called[:]
            _close([m(x[..., :128])], [ref], True)
            wide = m(x[..., :128].float().contiguous())  # pooled in float32 before the rounding
            assert float((wide - ref).float().norm() / ref.float().norm()) < 0.02
            odd = torch.empty(m.out.weight.numel() + 1, device=dev)[1:].view_as(m.out.weight).copy_(m.out.weight)
            m.out.weight = torch.nn.Parameter(odd)
            _close([m(x[..., :128].contiguous())], [ref], True)
        assert not called
    finally:
        steps._call = real


@pytest.mark.parametrize("contiguous", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("qb,T,per_head", [(0, 300, False), (48, 500, True), (0, 2100, False)])
def test_op_step_matches_python_path(contiguous, dtype, qb, T, per_head):
    from llattn_amd import LLAttnFunction
    dev = require_cuda()
    print("case: op step", contiguous, dtype, qb, T, per_head, flush=True)
    B, H, Dh, Lh, Ldh, chunk = 2, 3, 40, 2, 64, 50
    g = torch.Generator(device=dev).manual_seed(T)
    nq = -(-T // qb) if qb > 1 else T
    nc = -(-T // chunk)

    def heads(h, n, d):
        t = torch.randn(B, n, h, d, device=dev, generator=g).to(dtype).transpose(1, 2)
        return t.contiguous() if contiguous else t

    ins = [heads(H, T, Dh) for _ in range(3)] + [heads(Lh, nq, Ldh), heads(Lh, nc, Ldh), heads(Lh, nc, Ldh)]
    ins += [torch.randn(H if per_head else 1, Dh, device=dev, generator=g) for _ in range(2)]
    ins += [torch.randn(H * Dh, Lh * Ldh, device=dev, generator=g) * 0.1]
    rb, dO = torch.randn(H * Dh, device=dev, generator=g), heads(H, T, Dh)

    def run():
        leaves = [t.detach().requires_grad_() for t in ins]
        b = rb.detach().requires_grad_()
        y = LLAttnFunction.apply(*leaves, 64, chunk, b, 128, qb)
        y.backward(dO)
        for t in leaves:
            assert t.grad.stride() == t.stride()
        return [y.detach(), *(t.grad for t in leaves), b.grad]

    native, python = _both(run, "llattn_core_bwd")
    _close(native, python, dtype == torch.bfloat16)
    # nothing needs a gradient: a smaller buffer, the same output
    assert torch.equal(LLAttnFunction.apply(*[t.detach() for t in ins], 64, chunk, rb, 128, qb), native[0])


@pytest.mark.parametrize("shape,d_ff,bias", [((3, 7, 64), 128, True), ((2, 600, 128), 256, False),
                                             ((1, 1000, 1408), 4096, True), ((2, 2100, 256), 1024, True)])
def test_ffn_step_matches_python_path(shape, d_ff, bias):
    from llattn_amd.ffn import feed_forward
    dev = require_cuda()
    print("case: ffn step", shape, d_ff, bias, flush=True)
    torch.manual_seed(5)
    w1, w2 = torch.nn.Linear(shape[-1], d_ff, bias=bias).to(dev), torch.nn.Linear(d_ff, shape[-1], bias=bias).to(dev)
    x, dy = (torch.randn(shape, device=dev).bfloat16() for _ in range(2))

    def run(grad=True):
        xx = x.clone().requires_grad_(grad)
        for p in (*w1.parameters(), *w2.parameters()):
            p.grad = None
        with torch.set_grad_enabled(grad), torch.autocast("cuda", dtype=torch.bfloat16):
            y = feed_forward(xx, w1, w2)
        if not grad:
            return [y]
        y.backward(dy)
        return [y.detach(), xx.grad, *(p.grad for p in (*w1.parameters(), *w2.parameters()))]

    _close(*_both(run, "llattn_ffn_bwd"), True)
    _close(*_both(lambda: run(False), "llattn_ffn_fwd"), True)


@pytest.mark.parametrize("seg", [1, 7, 8, 9, 25, 32, 33, 57, 100, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_pool_segment_lengths(seg, dtype):
    """Segments around the eight row groups and their four rows in flight, the last one short.  fp32 sums of `seg`
    terms: seg * 2^-24 of the sum of magnitudes; a bf16 result rounds by at most 2^-8 of itself on top."""
    from llattn_amd import DIV_COUNT, pool
    dev = require_cuda()
    print("case: pool", seg, dtype, flush=True)
    n, B, D = 5, 2, 264
    T = n * seg - seg // 3
    x = torch.randn(B, T, D, device=dev, generator=torch.Generator(device=dev).manual_seed(seg)).to(dtype)
    got = pool(x, seg, n, DIV_COUNT).double().cpu()
    for i in range(n):
        rows = x[:, i * seg:(i + 1) * seg].double().cpu()
        ref, mag = rows.mean(1), rows.abs().mean(1)
        tol = (seg + 2) * 2.0 ** -24 * mag + (2.0 ** -8 * ref.abs() if dtype == torch.bfloat16 else 0)
        assert ((got[:, i] - ref).abs() <= tol).all(), i


@pytest.mark.parametrize("entry", ["block", "ffn"])
def test_forward_only_steps_refuse_tangents_and_vmap(entry):
    """A forward that keeps nothing for a backward is still an autograd function: a forward-mode tangent or a batched
    input raises instead of being dropped."""
    import torch.autograd.forward_ad as fwad
    from llattn_amd import LocalLatentAttentionTriton
    from llattn_amd.ffn import feed_forward
    dev = require_cuda()
    m = LocalLatentAttentionTriton(128, 4, 2, 64, 16, 64).to(dev).requires_grad_(False)
    w1, w2 = (torch.nn.Linear(*s).to(dev).requires_grad_(False) for s in ((128, 256), (256, 128)))
    fn = m if entry == "block" else lambda t: feed_forward(t, w1, w2)
    x = torch.randn(2, 64, 128, device=dev).bfloat16()
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        fn(x)
        with fwad.dual_level(), pytest.raises(RuntimeError):
            fn(fwad.make_dual(x, torch.ones_like(x)))
        with pytest.raises(RuntimeError):
            torch.func.vmap(fn)(x[None])


def test_block_with_frozen_parts_stops_its_backward_early():
    """Only ``out`` trains and the input needs no gradient: the backward forms that projection's gradients alone."""
    from llattn_amd import LocalLatentAttentionTriton, steps
    dev = require_cuda()
    torch.manual_seed(6)
    m = LocalLatentAttentionTriton(128, 4, 2, 64, 16, 64).to(dev)
    x, dy = (torch.randn(2, 96, 128, device=dev).bfloat16() for _ in range(2))

    def grads(frozen):
        m.zero_grad(set_to_none=True)
        for n, p in m.named_parameters():
            p.requires_grad_(not frozen or n.startswith("out."))
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = m(x)
        y.backward(dy)
        return [m.out.weight.grad, m.out.bias.grad]

    called, real = [], steps._call
    steps._call = lambda name, *a: (called.append(name), real(name, *a))[1]
    try:
        ref = grads(False)
        assert "llattn_block_bwd" in called
        del called[:]
        got = grads(True)
    finally:
        steps._call = real
    assert not called
    _close(got, ref, True)


@pytest.mark.parametrize("bf16", [True, False])
def test_block_with_other_projection_widths_and_gates(bf16):
    """Replaced projections: a wider and a narrower ``out`` give the columns that their rows give one by one, another
    width of ``rkv_proj`` is refused, and gates per head act on their own heads."""
    from llattn_amd import LocalLatentAttentionTriton
    dev = require_cuda()
    torch.manual_seed(7)
    D, H = 128, 4
    m = LocalLatentAttentionTriton(D, H, 2, 64, 16, 64).to(dev)
    x = torch.randn(2, 200, D, device=dev).to(torch.bfloat16 if bf16 else torch.float32)
    w, b = torch.randn(2 * D, D, device=dev) * 0.1, torch.randn(2 * D, device=dev)

    def out_linear(rows):
        lin = torch.nn.Linear(D, len(w[rows])).to(dev)
        with torch.no_grad():
            lin.weight.copy_(w[rows])
            lin.bias.copy_(b[rows])
        return lin

    def run(dy):
        m.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=bf16):
            y = m(x)
        y.backward(dy.to(y.dtype))
        return y.detach(), m.out.weight.grad, m.out.bias.grad

    dy = torch.randn(2, 200, 2 * D, device=dev)
    parts = []
    for i in range(2):
        m.out = out_linear(slice(i * D, (i + 1) * D))
        parts.append(run(dy[..., i * D:(i + 1) * D]))
    for rows in (slice(0, 2 * D), slice(0, D // 2)):
        m.out = out_linear(rows)
        got = run(dy[..., rows])
        _close(got, [torch.cat([p[0] for p in parts], -1)[..., rows], torch.cat([p[1] for p in parts])[rows],
                     torch.cat([p[2] for p in parts])[rows]], bf16)

    m.out = torch.nn.Linear(D, D, bias=True).to(dev)
    with torch.no_grad():
        m.out.weight.copy_(torch.eye(D, device=dev))
        m.out.bias.zero_()
    gates = [torch.randn(1, D // H, device=dev) for _ in range(2)]

    def heads(gate):
        m.gate_local.weight, m.gate_remote.weight = torch.nn.Parameter(gate), torch.nn.Parameter(gate.flip(-1))
        m.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=bf16):
            y = m(x)
        y.backward(dy[..., :D].to(y.dtype))
        return y.detach().view(2, 200, H, D // H), m.gate_local.weight.grad

    (y0, g0), (y1, g1) = heads(gates[0]), heads(gates[1])
    y, g = heads(torch.cat([gates[0], gates[1], gates[1], gates[1]]))
    _close([y], [torch.cat([y0[:, :, :1], y1[:, :, 1:]], 2)], bf16)
    same, gs = heads(gates[1].expand(H, -1).contiguous())
    _close([same, gs[1:]], [y1, g[1:]], bf16)
    # the shared gate's gradient is the heads' sum: fp32 sums of B T H = 1600 terms in another order, 1600 * 2^-24 of
    # their magnitudes, which the signed sum is taken to be a tenth of
    assert float((gs.sum(0) - g1[0]).norm()) <= 1e-3 * float(g1.norm())

    m.rkv_proj = torch.nn.Linear(D, 64).to(dev)
    with pytest.raises(ValueError):
        heads(gates[0])


def test_ffn_with_a_short_bias_is_refused():
    from llattn_amd.ffn import feed_forward
    dev = require_cuda()
    w1, w2 = torch.nn.Linear(128, 256).to(dev), torch.nn.Linear(256, 128).to(dev)
    x = torch.randn(2, 64, 128, device=dev).bfloat16()
    for lin in (w1, w2):
        full, lin.bias = lin.bias, torch.nn.Parameter(torch.zeros(64, device=dev))
        with pytest.raises(ValueError), torch.autocast("cuda", dtype=torch.bfloat16):
            feed_forward(x, w1, w2)
        lin.bias = full


def test_op_refuses_other_batches_and_mixed_gates():
    from llattn_amd import LLAttnFunction
    dev = require_cuda()
    B, H, T, Dh, Lh, Ldh, chunk = 2, 4, 64, 32, 2, 32, 16
    q = torch.randn(B, H, T, Dh, device=dev)
    gq, gk = torch.randn(B, Lh, T, Ldh, device=dev), torch.randn(B, Lh, T // chunk, Ldh, device=dev)
    shared, per_head, r_w = (torch.randn(*s, device=dev) for s in ((1, Dh), (H, Dh), (H * Dh, Lh * Ldh)))
    for a in ((gq[:1], shared, shared), (gq, per_head, shared), (gq, shared, per_head)):
        with pytest.raises(ValueError):
            LLAttnFunction.apply(q, q, q, a[0], gk, gk, a[1], a[2], r_w, 16, chunk)


def test_block_step_with_more_poolings_than_one_launch_holds():
    """A million short sequences: the two poolings' workgroups pass 2^32 threads in a row, so that they are launched
    apart from the weight casts.  Sequences do not see each other: the first ones equal a small batch's."""
    from llattn_amd import LocalLatentAttentionTriton
    dev = require_cuda()
    torch.manual_seed(8)
    B, T, D = 1 << 20, 12, 64
    m = LocalLatentAttentionTriton(D, 2, 2, 16, T, 16, latent_query_block_size=2).to(dev)
    assert B * (T + T // 2) * 256 >= 1 << 32
    x = torch.randn(B, T, D, device=dev, dtype=torch.bfloat16)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        (a,), (b,) = _both(lambda: [m(x)], "llattn_block_fwd")
        _close([a[:64], a[-64:]], [m(x[:64]), m(x[-64:])], True)
        _close([a[B // 2:B // 2 + 64]], [b[B // 2:B // 2 + 64]], True)


@pytest.mark.parametrize("qb", [0, 64])
@pytest.mark.parametrize("bf16", [True, False])
def test_block_step_peak_memory(qb, bf16):
    """The native step's peak: a forward alone takes no more than the products one by one; a training pass at most the
    attention output that its one node keeps to the end and the parameter gradients that it allocates together."""
    from llattn_amd import LocalLatentAttentionTriton
    dev = require_cuda()
    torch.manual_seed(9)
    D = 512
    m = LocalLatentAttentionTriton(D, 8, 4, 128, 16, 64, latent_query_block_size=qb).to(dev)
    x = torch.randn(4, 2048, D, device=dev).to(torch.bfloat16 if bf16 else torch.float32)

    def peak(grad):
        for _ in range(2):
            m.zero_grad(set_to_none=True)
            xx = x.detach().requires_grad_(grad)
            torch.cuda.synchronize()
            before = torch.cuda.memory_allocated()
            torch.cuda.reset_peak_memory_stats()
            with torch.set_grad_enabled(grad), torch.autocast("cuda", dtype=torch.bfloat16, enabled=bf16):
                y = m(xx)
            if grad:
                y.backward(x)
            torch.cuda.synchronize()
            got = torch.cuda.max_memory_allocated() - before
            del xx, y
        return got

    for grad in (False, True):
        native = peak(grad)
        with _logged():
            single = peak(grad)
        more = x.numel() * x.element_size() + 4 * sum(p.numel() for p in m.parameters()) if grad else 0
        assert native <= single + more + (1 << 20), (grad, native, single, more)
