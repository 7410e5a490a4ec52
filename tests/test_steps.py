"""CPU tests of the native steps' interface (include/llattn_steps.h): nothing is launched."""
from __future__ import annotations

import ctypes
import re
import shutil
import subprocess

import pytest

from conftest import REPO


def test_steps_header_matches_the_binding(tmp_path):
    from llattn_amd import _lib as L
    text = (REPO / "include" / "llattn_steps.h").read_text()
    names = set(re.findall(r"^(?:int32_t|size_t)\s+(llattn_\w+)\s*\(", text, re.M))
    assert names == set(L.STEP_SIGNATURES) and all(hasattr(L.load(), n) for n in names)
    if shutil.which("gcc") is None:
        pytest.skip("gcc not available")
    structs = {"llattn_block_cfg": L.LlattnBlockCfg, "llattn_block_params": L.LlattnBlockParams,
               "llattn_block_grads": L.LlattnBlockParams, "llattn_core_views": L.LlattnCoreViews,
               "llattn_ffn_cfg": L.LlattnFfnCfg}
    lines = ["#include <stddef.h>", "#include <stdio.h>", '#include "llattn_steps.h"', "int main(void) {"]
    for name, cls in structs.items():
        lines.append(f'  printf("%zu ", sizeof({name}));')
        lines += [f'  printf("%zu ", offsetof({name}, {f}));' for f, _ in cls._fields_]
    src = tmp_path / "layout.c"
    src.write_text("\n".join(lines) + "\n  return 0;\n}\n")
    subprocess.run(["gcc", "-std=c11", f"-I{REPO / 'include'}", str(src), "-o", str(tmp_path / "layout")], check=True)
    got = [int(n) for n in subprocess.run([str(tmp_path / "layout")], check=True, capture_output=True, text=True).stdout.split()]
    want = []
    for cls in structs.values():
        want += [ctypes.sizeof(cls)] + [getattr(cls, f).offset for f, _ in cls._fields_]
    assert got == want


def test_step_sizes_and_refusals():
    from llattn_amd import _lib as L
    from llattn_amd._lib import resolve_layout
    import torch
    lib, ref = L.load(), ctypes.byref
    lay = resolve_layout(2, 100, 128, 4, 64, 2, 64, 256, 16, 0)
    cfg = L.LlattnBlockCfg(lay.shape(torch.bfloat16), 128, 0, 1, 1, 1, 0, 0, 0)
    kept = lib.llattn_block_bytes(ref(cfg), 0)
    # the projection output, the attention outputs and the weight copies at least
    assert kept > 200 * (3 * 128 + 64) * 2 + 4 * 200 * 128 * 2 + (5 * 128 * 128) * 2
    cfg.saved = 0
    assert 0 < lib.llattn_block_bytes(ref(cfg), 0) < kept
    cfg.saved = 1
    buf = ctypes.create_string_buffer(64)
    p = L.LlattnBlockParams()
    small = lib.llattn_block_bwd(ref(cfg), ref(p), buf, buf, buf, None, ref(p), buf, 16, None)
    assert small in (L.ERR_WORKSPACE, L.ERR_LAYOUT)
    cfg.d_model = 136
    assert lib.llattn_block_bytes(ref(cfg), 0) == 0
    assert lib.llattn_block_fwd(ref(cfg), ref(p), buf, buf, None, 0, buf, None) == L.ERR_SHAPE
    assert lib.llattn_block_fwd(None, ref(p), buf, buf, None, 0, buf, None) == L.ERR_SHAPE
    f = L.LlattnFfnCfg(0, 64, 128, 64, 1)
    assert lib.llattn_ffn_bytes(ref(f), 0) == 0 and b"positive" in lib.llattn_last_error()


@pytest.mark.parametrize("name,change", [
    ("none", None), ("wider out", ("out", 128, 256)), ("narrower out", ("out", 128, 64)),
    ("narrower rkv_proj", ("rkv_proj", 128, 64)), ("wider rq_proj", ("rq_proj", 128, 128)),
    ("other r_out", ("r_out", 32, 128)), ("short qkv_proj", ("qkv_proj", 128, 128)), ("gates per head", None),
    ("short bias", None)])
def test_block_step_takes_only_the_layouts_shapes(name, change, monkeypatch):
    """A parameter of another shape than the layout's never reaches the native call, which sees pointers alone."""
    import torch
    from llattn_amd import LocalLatentAttentionTriton, steps
    taken = object()
    monkeypatch.setattr(steps, "Block", type("Taken", (), {"apply": staticmethod(lambda *a: taken)}))
    m = LocalLatentAttentionTriton(128, 4, 2, 64, 16, 64)
    if change is not None:
        setattr(m, change[0], torch.nn.Linear(*change[1:]))
    elif name == "gates per head":
        m.gate_local.weight = torch.nn.Parameter(torch.randn(4, 32))
    elif name == "short bias":
        m.out.bias = torch.nn.Parameter(torch.zeros(64))
    x = torch.randn(2, 96, 128)
    assert m._forward_native(x, m.layout(2, 96)) is (taken if name == "none" else None)


@pytest.mark.parametrize("which,shape", [(None, None), (0, (256, 64)), (1, (128,)), (2, (128, 128)), (3, (64,)), (3, (1, 128))])
def test_ffn_step_takes_only_matching_shapes(which, shape):
    """A weight or a bias of another shape never reaches the native call."""
    import torch
    from llattn_amd import ffn
    ps = [torch.zeros(s) for s in ((256, 128), (256,), (128, 256), (128,))]
    if which is not None:
        ps[which] = torch.zeros(shape)
    cfg = ffn._step_cfg(torch.zeros(3, 7, 128, dtype=torch.bfloat16), ps)
    assert (cfg is None) == (which is not None)
    if cfg is not None:
        assert [cfg.rows, cfg.d, cfg.d_ff, cfg.d_out, cfg.saved] == [21, 128, 256, 128, 0]


def test_gates_of_two_forms_are_refused():
    """Both shared by the heads or both per head: the kernels read them by one rule."""
    import torch
    from llattn_amd import ops
    H, Dh = 4, 32
    shared, per_head = torch.randn(1, Dh), torch.randn(H, Dh)
    for a, b in ((shared, shared), (shared[0], shared), (per_head, per_head), (shared.expand(H, Dh), per_head)):
        gl, gr = ops._gates(a, b, H, Dh)
        assert torch.equal(gl, a) and torch.equal(gr, b) and gl.is_contiguous() and gr.is_contiguous()
    for a, b in ((per_head, shared), (shared, per_head), (per_head[:2], per_head[:2]), (shared[:, :16], shared),
                 (per_head, per_head[:3])):
        with pytest.raises(ValueError, match="gates"):
            ops._gates(a, b, H, Dh)
