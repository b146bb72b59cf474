"""Which windows and score weights the attention layer runs at inference: its own methods' values,
also where a program replaces them, and one evaluation of the window gate a call."""
from __future__ import annotations

import types

import pytest
import torch

from dsalt_amd.modules import DSALTAttention

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _layer(dt=torch.bfloat16, **kw):
    torch.manual_seed(2)
    args = dict(d_model=256, n_heads=4, n_min=8, n_max=90, k_lmk=11, max_seq_len=512, n_kv_heads=2)
    args.update(kw)
    return DSALTAttention(**args).to(DEV, dt).eval()


def _run(m, T=300):
    x = torch.randn(T, 256, generator=torch.Generator(device=DEV).manual_seed(T), device=DEV).to(m.out_proj.weight.dtype)
    with torch.no_grad():
        return m(x, cu_seqlens=torch.tensor([0, T], dtype=torch.int32, device=DEV), cu_list=[0, T])[0]


@pytest.mark.parametrize("where", ["instance", "class", "subclass"])
@pytest.mark.parametrize("name", ["_alpha", "_window_continuous", "_window_sizes"])
def test_replaced_methods_are_called(name, where, monkeypatch):
    calls = []
    body = {"_alpha": lambda self: torch.full((4,), 0.9, device=DEV),
            "_window_continuous": lambda self, x: torch.full((x.shape[0],), 31.5, device=DEV),
            "_window_sizes": lambda self, x, floor: torch.full((x.shape[0],), 17.0, device=DEV)}[name]

    def repl(self, *a, **kw):
        calls.append(name)
        return body(self, *a, **kw)

    m = _layer()
    if where == "instance":
        setattr(m, name, types.MethodType(repl, m))
    elif where == "class":
        monkeypatch.setattr(DSALTAttention, name, repl)
    else:
        m.__class__ = type("Own", (DSALTAttention,), {name: repl})
    w, alpha = m._selectors(torch.randn(300, 256, device=DEV, dtype=torch.bfloat16))
    assert calls and w.dtype == torch.int32 and alpha.dtype == torch.float32
    if name == "_alpha":
        assert torch.equal(alpha, torch.full_like(alpha, 0.9))
    else:
        assert torch.equal(w, torch.full_like(w, 31 if name == "_window_continuous" else 17))
    assert torch.isfinite(_run(m)).all()


@pytest.mark.parametrize("alpha_dt", [torch.bfloat16, torch.float32])
def test_the_window_gate_runs_once(alpha_dt):
    """Also where the types differ (16-bit weights with float32 score weights): its hooks see one call."""
    m = _layer()
    m.alpha_w.data = m.alpha_w.data.to(alpha_dt)
    calls = []
    m.win_gate.register_forward_hook(lambda mod, a, y: calls.append(y))
    x = torch.randn(300, 256, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        w, alpha = m._selectors(x)
        assert len(calls) == 1
        gate = calls[0].squeeze(-1)
        ref = (m.n_min + torch.sigmoid(gate) * (m.n_max - m.n_min)).floor().clamp(min=1).int()
    assert torch.equal(w, ref) and torch.equal(alpha, torch.sigmoid(m.alpha_w.data).float())
    _run(m)
    assert len(calls) == 2


@pytest.mark.parametrize("kw", [dict(select_mode="causal"), dict(stats_scope="batch")])
def test_unknown_modes_are_refused(kw):
    with pytest.raises(KeyError):
        _run(_layer(**kw))
