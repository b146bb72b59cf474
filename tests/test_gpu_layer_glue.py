"""The small kernels and product layouts around the attention: a layer's windows and score weights
(bit for bit the torch expressions) and the LM-head loss over row counts and vocabularies on both
sides of its layout rules."""
from __future__ import annotations

import ctypes
import os
import subprocess

import pytest
import torch
import torch.nn.functional as F

from dsalt_amd import _lib, ops
from dsalt_amd.kernels import cross_entropy as CE
from dsalt_amd.modules import DSALTAttention

DEV = "cuda"
HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "dsalt_amd.h")


def test_selectors_args_layout_and_validation(tmp_path):
    cls, fields = _lib.SelectorsArgs, [f for f, _ in _lib.SelectorsArgs._fields_]
    src = tmp_path / "l.c"
    src.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "%s"\nint main(void){printf("%%zu",sizeof(dsalt_selectors_args));%s'
                   'return 0;}' % (HEADER, "".join('printf(" %%zu",offsetof(dsalt_selectors_args,%s));' % f for f in fields)))
    subprocess.run(["gcc", "-o", str(tmp_path / "l"), str(src)], check=True)
    got = subprocess.run([str(tmp_path / "l")], capture_output=True, text=True, check=True).stdout.split()
    assert [int(x) for x in got] == [ctypes.sizeof(cls)] + [getattr(cls, f).offset for f in fields]
    lib, fake = _lib.load(), 1 << 20
    for f, v in (("total_len", -1), ("dtype", 3), ("gate", None), ("gate_stride", 0), ("alpha", None), ("w", None)):
        a = cls(4, 2, 1, fake, 1, fake, 1.0, 2.0, fake, fake)
        setattr(a, f, v)
        assert lib.dsalt_layer_selectors(ctypes.byref(a), None) == 1, f


@pytest.mark.parametrize("BT,chunk,want", [(0, 512, 0), (5, 512, 5), (959, 4096, 959), (960, 4096, 960), (961, 4096, 1024),
                                           (4096 + 961, 4096, 4096 + 1024), (4096 + 3, 4096, 4099), (4001, 4001, 4032)])
def test_rows_of_the_last_chunk(BT, chunk, want):
    assert CE._whole_rows(BT, chunk) == want


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n_min,n_max", [(32, 256), (1, 2), (0, 7), (16, 4096), (12.5, 99.25)])
def test_layer_selectors_bit_exact(dt, n_min, n_max):
    g = torch.Generator(device=DEV).manual_seed(0)
    gate = torch.cat([torch.randn(70001, generator=g, device=DEV) * 4, torch.linspace(-120, 120, 5000, device=DEV),
                      torch.tensor([float("inf"), float("-inf"), 0.0, -0.0], device=DEV)]).to(dt)
    aw = (torch.randn(17, generator=g, device=DEV) * 3).to(dt)
    w, alpha = ops.layer_selectors(gate, aw, n_min, n_max)
    ref = (n_min + torch.sigmoid(gate) * (n_max - n_min)).floor().clamp(min=1).to(torch.int32)
    assert torch.equal(w, ref) and torch.equal(alpha, torch.sigmoid(aw).float())
    wide = torch.stack([gate, gate], 1)[:, 1]  # a column of a wider buffer
    assert torch.equal(ops.layer_selectors(wide, aw, n_min, n_max)[0], ref)
    assert ops.layer_selectors(gate[:0], aw, n_min, n_max)[0].numel() == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_layer_without_its_selector_kernel_is_the_same(dt):
    """A subclass that redefines the windows keeps its own expression; with the parent's
    expression both layers give the same bits."""
    class Own(DSALTAttention):
        def _window_continuous(self, x):
            return super()._window_continuous(x)

    torch.manual_seed(1)
    kw = dict(d_model=256, n_heads=4, n_min=8, n_max=90, k_lmk=11, max_seq_len=512, n_kv_heads=2)
    a = DSALTAttention(**kw).to(DEV, dt).eval()
    b = Own(**kw).to(DEV, dt).eval()
    b.load_state_dict(a.state_dict())
    for lens in ([333], [200, 0, 1, 130], [1]):
        x = torch.randn(sum(lens), 256, device=DEV).to(dt)
        cl = [0]
        for n in lens:
            cl.append(cl[-1] + n)
        cu = torch.tensor(cl, dtype=torch.int32, device=DEV)
        with torch.no_grad():
            assert all(torch.equal(u, v) for u, v in zip(a._selectors(x), b._selectors(x)))
            ya, yb = a(x, cu_seqlens=cu, cu_list=cl)[0], b(x, cu_seqlens=cu, cu_list=cl)[0]
        assert ya.shape == x.shape and (ya - yb).abs().max() <= 2e-2 * yb.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [3, 959, 1001, 1024])
@pytest.mark.parametrize("V,bias", [(1003, False), (1003, True), (1000, False), (4096, True)])
@pytest.mark.parametrize("dt,accum", [(torch.bfloat16, None), (torch.bfloat16, torch.float32), (torch.float16, None),
                                      (torch.float32, None)])
def test_lm_loss_layouts(rows, V, bias, dt, accum, monkeypatch):
    """Loss and gradients against plain torch in float32 on the 16-bit logits the loss is defined
    on.  The gradient of a logit is rounded to the type once, the sums once more, a second chunk once
    more: relative 2-norm at most 3 u (u = 2^-8, 2^-11); asked for is 2 u in bfloat16, where every
    rounding at its largest would be needed for more, 4 u in float16 (gradients of 1e-6 reach its
    subnormals), and 1e-5 in float32."""
    g = torch.Generator(device=DEV).manual_seed(rows + V)
    H = 96
    x = torch.randn(rows, H, generator=g, device=DEV).to(dt).requires_grad_(True)
    w = (torch.randn(V, H, generator=g, device=DEV) * 0.1).to(dt).requires_grad_(True)
    b = torch.randn(V, generator=g, device=DEV).to(dt).requires_grad_(True) if bias else None
    t = torch.randint(0, V, (rows,), generator=g, device=DEV)
    t[::7] = -100
    z = x.detach().float() @ w.detach().float().T + (b.detach().float() if bias else 0)
    z = z.to(dt).float()
    n = int((t != -100).sum())
    loss = F.cross_entropy(z, t, ignore_index=-100)
    d = torch.softmax(z, 1)
    keep = t != -100
    d[keep, t[keep]] -= 1
    d[~keep] = 0
    d = (d / n).to(dt).float()
    ref = [d @ w.detach().float(), d.T @ x.detach().float()] + ([d.sum(0)] if bias else [])
    tol = {torch.bfloat16: 2 * 2.0 ** -8, torch.float16: 4 * 2.0 ** -11, torch.float32: 1e-5}[dt]
    for chunk_bytes in (1 << 31, 512 * V * x.element_size()):  # one chunk, and chunks of 512 rows
        monkeypatch.setattr(CE, "_CHUNK_BYTES", chunk_bytes)
        got = CE.LigerFusedLinearCrossEntropyFunction.apply(x, w, t, b, None, -100, 0.0, 0.0, "mean", None, False, accum)[0]
        assert abs(float(got.detach()) - float(loss)) <= 2e-5 * abs(float(loss)) + (0 if dt == torch.float32 else 1e-3)
        grads = torch.autograd.grad(got, [x, w] + ([b] if bias else []))
        for a, r in zip(grads, ref):
            assert a.shape == r.shape and a.is_contiguous()
            assert (a.float() - r).norm() <= tol * r.norm() + 1e-12, (chunk_bytes, a.shape)
        with torch.no_grad():  # no gradients wanted: the loss alone
            alone = CE.LigerFusedLinearCrossEntropyFunction.apply(x.detach(), w.detach(), t, b.detach() if bias else None)[0]
            assert abs(float(alone) - float(loss)) <= 2e-5 * abs(float(loss)) + (0 if dt == torch.float32 else 1e-3)
