"""Ordering of landmark sets (ops.sort_landmarks) and the float32 result / upstream gradient the
attention kernels take themselves: both are exact (whole numbers, and the same roundings as a
conversion in a pass of its own)."""
from __future__ import annotations

import ctypes
import os
import subprocess

import pytest
import torch

from dsalt_amd import _lib, ops
from dsalt_amd.kernels.dsalt_attn import dsalt_attention
from dsalt_amd.kernels.dsalt_train import dsalt_train_attention

DEV = "cuda"
HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "dsalt_amd.h")


def test_sort_args_layout_matches_c(tmp_path):
    cls, fields = _lib.SortArgs, [f for f, _ in _lib.SortArgs._fields_]
    src = tmp_path / "l.c"
    src.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "%s"\nint main(void){printf("%%zu",sizeof(dsalt_sort_args));%s'
                   'return 0;}' % (HEADER, "".join('printf(" %%zu",offsetof(dsalt_sort_args,%s));' % f for f in fields)))
    subprocess.run(["gcc", "-o", str(tmp_path / "l"), str(src)], check=True)
    got = subprocess.run([str(tmp_path / "l")], capture_output=True, text=True, check=True).stdout.split()
    assert [int(x) for x in got] == [ctypes.sizeof(cls)] + [getattr(cls, f).offset for f in fields]


def test_new_entries_reject_bad_arguments():
    lib = _lib.load()
    fake = 1 << 20  # never dereferenced: validation fails before any launch
    a = _lib.SortArgs(4, 8, 4, fake, fake, fake, None, None, 0)
    for f, v in (("k", 2049), ("n_sets", -1), ("idx_bytes", 2), ("idx", None), ("perm", None), ("bias", fake)):
        b = _lib.SortArgs.from_buffer_copy(a)
        setattr(b, f, v)
        assert lib.dsalt_sort_landmarks(ctypes.byref(b), None) == 1, f
    a.bias = a.bias_sorted = fake
    a.bias_bytes = 8
    assert lib.dsalt_sort_landmarks(ctypes.byref(a), None) == 1
    assert lib.dsalt_sort_landmarks(None, None) == 1
    f, b = _lib.FwdArgs(), _lib.BwdArgs()
    f.p.dtype = b.p.dtype = _lib.DTYPE_BF16
    assert lib.dsalt_fwd_f32out(ctypes.byref(f), None, None) == 1 and lib.dsalt_fwd_f32out(None, fake, None) == 1
    assert lib.dsalt_fwd_f32out(ctypes.byref(f), fake + 4, None) == 1
    for st, sh, ptr in ((0, 64, fake), (130, 64, fake), (128, 66, fake), (128, 64, fake + 8), (128, -64, fake)):
        assert lib.dsalt_bwd_f32dout(ctypes.byref(b), ptr, st, sh, None) == 1
    f.p.dtype = b.p.dtype = _lib.DTYPE_F32
    assert lib.dsalt_fwd_f32out(ctypes.byref(f), fake, None) == 2
    assert lib.dsalt_bwd_f32dout(ctypes.byref(b), fake, 128, 64, None) == 2


def _reference(idx, bias):
    """A stable sort by (position, or past every position for an empty slot)."""
    key = torch.where(idx < 0, torch.full_like(idx, 2 ** 31 - 1), idx).to(torch.int64)
    srt, perm = key.sort(dim=-1, stable=True)
    return torch.where(srt == 2 ** 31 - 1, -1, srt).int(), None if bias is None else bias.gather(-1, perm), perm


@pytest.mark.gpu
@pytest.mark.parametrize("K", [1, 2, 63, 256, 257, 2048])
@pytest.mark.parametrize("kind", ["sorted", "shuffled", "repeated", "empty"])
@pytest.mark.parametrize("dt,bdt", [(torch.int64, torch.float32), (torch.int32, torch.bfloat16), (torch.int64, None)])
def test_sort_landmarks(K, kind, dt, bdt):
    g = torch.Generator().manual_seed(K)
    idx = torch.stack([torch.randperm(5000, generator=g)[:K] for _ in range(6)]).view(3, 2, 1, K)
    if kind == "repeated":
        idx = idx % 7
    if kind == "sorted":
        idx = idx.sort(-1).values
        idx[..., K // 2 + 1:] = -1
    elif kind == "empty":
        idx = torch.full_like(idx, -3)
    else:
        idx[torch.rand(idx.shape, generator=g) < 0.2] = -1
    idx = idx.to(dt)
    bias = None if bdt is None else torch.randn(idx.shape, generator=g).to(bdt)
    out, b, perm = ops.sort_landmarks(idx.to(DEV), None if bias is None else bias.to(DEV))
    ro, rb, rp = _reference(idx, bias)
    assert torch.equal(out.cpu(), ro) and torch.equal(perm.cpu(), rp)
    assert (b is None) == (bias is None) and (b is None or torch.equal(b.cpu(), rb))
    # a strided view of a larger tensor is the same sets
    wide = torch.stack([idx, idx + 1], dim=-1).to(DEV)[..., 0]
    assert torch.equal(ops.sort_landmarks(wide)[0].cpu(), ro)


@pytest.mark.gpu
@pytest.mark.parametrize("K,kernel", [(1, True), (512, True), (513, False), (2048, False)])
def test_large_sets_are_not_counted(K, kernel, monkeypatch):
    """Sets past the kernel's size, which it would order in k^2 steps, go to the library sort."""
    called, check = [], _lib.check
    monkeypatch.setattr(_lib, "check", lambda name, rc: (called.append(name), check(name, rc)))
    idx = torch.randint(0, 7, (3, 1, 1, K), generator=torch.Generator().manual_seed(K))
    out, _, perm = ops.sort_landmarks(idx.to(DEV))
    ro, _, rp = _reference(idx, None)
    assert torch.equal(out.cpu(), ro) and torch.equal(perm.cpu(), rp)
    assert called == (["dsalt_sort_landmarks"] if kernel else [])
    monkeypatch.setattr(ops, "_SORT_SLOTS", 2048)  # the kernel itself takes them all
    out, _, perm = ops.sort_landmarks(idx.to(DEV))
    assert called and torch.equal(out.cpu(), ro) and torch.equal(perm.cpu(), rp)


@pytest.mark.gpu
def test_sort_landmarks_under_transforms():
    """Forward-mode tangents, vmap and traces see the torch operations; so does a 0-dim set."""
    from torch.autograd import forward_ad as fw
    from torch.fx.experimental.proxy_tensor import make_fx
    g = torch.Generator().manual_seed(5)
    idx = torch.stack([torch.randperm(500, generator=g)[:9] for _ in range(12)]).view(3, 4, 1, 9).to(DEV)
    idx[0, :, 0, 3] = -1
    bias, tan = (torch.randn(idx.shape, generator=g).to(DEV) for _ in range(2))
    ro, rb, rp = ops.sort_landmarks(idx, bias)
    with fw.dual_level():
        o, b, p = ops.sort_landmarks(idx, fw.make_dual(bias, tan))
        assert torch.equal(o, ro) and torch.equal(fw.unpack_dual(b).tangent, tan.gather(-1, rp))
    _, t = torch.func.jvp(lambda x: ops.sort_landmarks(idx, x)[1], (bias,), (tan,))
    assert torch.equal(t, tan.gather(-1, rp))
    for a, r in zip(torch.vmap(ops.sort_landmarks)(idx, bias), (ro, rb, rp)):
        assert torch.equal(a, r)
    other, obias = idx.flip(-1), bias * 2
    want = ops.sort_landmarks(other, obias)
    for f in (make_fx(ops.sort_landmarks)(idx, bias), torch.jit.trace(ops.sort_landmarks, (idx, bias), check_trace=False)):
        for a, r in zip(f(other, obias), want):
            assert torch.equal(a, r)
    assert int(ops.sort_landmarks(torch.tensor(7, device=DEV))[0]) == 7


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,dt,T", [(4, 4, 64, torch.bfloat16, 1601), (4, 2, 64, torch.float16, 130),
                                        (16, 4, 64, torch.bfloat16, 6500), (4, 2, 128, torch.bfloat16, 777)])
@pytest.mark.parametrize("train", [False, True])
def test_float32_result_and_gradient_in_the_kernels(H, G, D, dt, T, train):
    """The operators' float32 result is the 16-bit output converted, and the gradients of a float32
    upstream gradient are those of its rounded values, bit for bit, whatever its layout."""
    g = torch.Generator(device=DEV).manual_seed(T)
    lens = [T - 30, 0, 30]
    cu_list = [0, lens[0], lens[0], T]
    cu = torch.tensor(cu_list, dtype=torch.int32, device=DEV)
    q, k, v = (torch.randn(T, n, D, generator=g, device=DEV).to(dt).requires_grad_(True) for n in (H, G, G))
    lmk = torch.randint(0, T - 30, (H, 3, 9), generator=g, device=DEV)
    lmk[:, 1] = -1
    lmk[:, 2] %= 30
    w = torch.rand(T, generator=g, device=DEV) * 90 + 1
    lw = torch.randn(lmk.shape, generator=g, device=DEV)
    idx, lws, perm = ops.sort_landmarks(lmk[:, :, None], lw[:, :, None])
    ml = max(lens)
    if train:
        out = dsalt_train_attention(q, k, v, lmk, lw, w, cu, cu_list=cu_list)
        o16, lse = ops.train_forward(q, k, v, w, cu, idx, lws, max_seqlen=ml)
    else:
        wi = w.int()
        out = dsalt_attention(q, k, v, lmk, None, wi, cu, cu_list=cu_list)
        o16, lse = ops.attention_forward(q, k, v, wi, cu, idx, max_seqlen=ml)
    assert out.dtype == torch.float32 and torch.equal(out.detach(), o16.float())
    base = torch.randn(T, H, D, generator=g, device=DEV)
    shapes = {"plain": base, "heads expanded": base[:, :1].expand(T, H, D), "wide rows": torch.cat([base, base], 2)[..., :D],
              "odd rows": torch.cat([base, base], 2)[..., 1:D + 1], "all expanded": base[0, 0, 0].expand(T, H, D),
              "head-major": base.transpose(0, 1).contiguous().transpose(0, 1)}
    for name, do in shapes.items():
        got = torch.autograd.grad(out, (q, k, v), do, retain_graph=True)
        if train:
            ref = ops.train_backward(do.to(dt), q, k, v, o16, lse, w, cu, idx, lws, max_seqlen=ml)[:3]
        else:
            ref = ops.attention_backward(do.to(dt), q, k, v, o16, lse, wi, cu, idx, max_seqlen=ml)[:3]
        for a, b in zip(got, ref):
            assert torch.equal(a, b), name
