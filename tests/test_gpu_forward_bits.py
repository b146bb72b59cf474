"""The size rule of the forward chooses among tilings that give the same bits: a call's output does
not depend on how many heads it holds."""
from __future__ import annotations

import pytest
import torch

from dsalt_amd import ops
from tests.test_gpu_tiling_rules import _inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("lens,H,G,D,dt,block,train", [
    ([8200], 16, 16, 64, torch.bfloat16, 0, False),
    ([24600], 16, 16, 64, torch.bfloat16, 0, False),      # 128-row blocks, an odd number of tiles
    ([20001, 6000], 16, 8, 64, torch.float16, 0, False),
    ([24600], 16, 16, 64, torch.bfloat16, 256, False),
    ([65, 400, 64] * 48, 16, 16, 64, torch.bfloat16, 0, False),  # short sequences
    ([65601], 32, 32, 128, torch.bfloat16, 0, False),     # eight waves, an odd number of tiles
    ([8200], 16, 16, 64, torch.bfloat16, 0, True),
    ([24600], 16, 8, 64, torch.float16, 0, True),
])
def test_output_bits_do_not_depend_on_the_number_of_heads(lens, H, G, D, dt, block, train):
    q, k, v, w, cu, idx = _inputs(lens, H, G, D, 70, 300, dt, seed=sum(lens), block=block)
    v = (v.float() * torch.exp(torch.randn(*v.shape[:2], 1, device=DEV))).to(dt)  # heavy-tailed norms
    lw = torch.nn.functional.logsigmoid(torch.randn(idx.shape, device=DEV))

    def run(h0, h1):
        g0, g1 = h0 * G // H, h1 * G // H
        a = [t.contiguous() for t in (q[:, h0:h1], k[:, g0:g1], v[:, g0:g1])]
        i = idx[h0:h1].contiguous()
        if train:
            return ops.train_forward(*a, w.float() + 0.25, cu, i, lw[h0:h1].contiguous(), max_seqlen=max(lens))
        return ops.attention_forward(*a, w, cu, i, max_seqlen=max(lens), block_size=block or 512,
                                     select_mode=ops.SELECT_BLOCK if block else ops.SELECT_GLOBAL)

    whole = run(0, H)
    for h0 in (0, H // 2, H - 2):
        part = run(h0, h0 + 2)
        for a, b in zip(whole, part):
            assert torch.equal(a[:, h0:h0 + 2], b)
