"""Size rules that choose a kernel or a split of the work: both sides of each line, at lengths off
every tile edge, against plain torch in float32 / float64 on the GPU.

Bound of a 16-bit forward: each probability is rounded to the tensor type (relative u = 2^-9 for
bfloat16, 2^-12 for float16) in the product and in its row sum, and the quotient once more, so an
output element is off by at most about 3 u max|v| (float32 sums add orders of magnitude less)."""
from __future__ import annotations

import math

import pytest
import torch

from dsalt_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
UNIT = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}


def _inputs(lens, H, G, D, K, wmax, dt, seed, block=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    T, S, L = sum(lens), len(lens), max(lens)
    q, k, v = (torch.randn(T, n, D, generator=g, device=DEV).to(dt) for n in (H, G, G))
    w = torch.randint(1, wmax + 1, (T,), generator=g, device=DEV, dtype=torch.int32)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    nset = -(-L // block) if block else 1
    idx = torch.full((H, S, nset, K), -1, dtype=torch.int32, device=DEV)
    for s, n in enumerate(lens):
        for b in range(nset):
            m = min(b * block, n) if block else n
            cnt = min(m, max(K - 1 - s, 0))  # the last slots stay empty
            if cnt:
                r = torch.rand(H, m, generator=g, device=DEV).argsort(1)[:, :cnt]
                idx[:, s, b, :cnt] = r.sort(1).values.int()
    return q, k, v, w, cu, idx


def _dense(q, k, v, w, cu, idx, block, heads):
    """Outputs of the given query heads, float32, one (head, sequence) at a time."""
    out = torch.zeros(q.shape[0], len(heads), q.shape[2], device=DEV)
    rep = q.shape[1] // k.shape[1]
    for s in range(cu.numel() - 1):
        a, n = int(cu[s]), int(cu[s + 1] - cu[s])
        i = torch.arange(n, device=DEV)
        lo = (i - w[a:a + n].long() + 1).clamp(min=0)
        band = (i[None] <= i[:, None]) & (i[None] >= lo[:, None])
        for c, h in enumerate(heads):
            mask = band.clone()
            for b in range(idx.shape[2]):
                p = idx[h, s, b]
                p = p[p >= 0].long()
                rows = slice(b * block, (b + 1) * block) if block else slice(0, n)
                mask[rows, p] |= p[None] < lo[rows, None]
            sc = q[a:a + n, h].float() @ k[a:a + n, h // rep].float().T / math.sqrt(q.shape[2])
            out[a:a + n, c] = torch.softmax(sc.masked_fill(~mask, float("-inf")), 1) @ v[a:a + n, h // rep].float()
    return out


@pytest.mark.parametrize("lens,H,G,D,dt,block", [
    ([6143], 16, 4, 64, torch.bfloat16, 0),               # below 1536 tiles of 64 rows
    ([6145], 16, 16, 64, torch.bfloat16, 0),              # above, an odd number of tiles
    ([4097, 1, 2050, 190], 16, 2, 64, torch.float16, 0),  # ragged
    ([6400], 16, 4, 64, torch.bfloat16, 256),             # block sets, whole 128-row blocks in a set
    ([6400], 16, 4, 64, torch.bfloat16, 192),             # sets of 192 rows keep 64-row blocks
    ([8191], 128, 8, 128, torch.bfloat16, 0),             # below 16384 tiles
    ([8321], 128, 8, 128, torch.bfloat16, 0),             # above, an odd number of tiles
    ([5000, 3333], 128, 128, 128, torch.float16, 0),
])
def test_forward_tiling_by_size(lens, H, G, D, dt, block):
    q, k, v, w, cu, idx = _inputs(lens, H, G, D, 9, 150, dt, seed=sum(lens), block=block)
    mode = ops.SELECT_BLOCK if block else ops.SELECT_GLOBAL
    out, lse = ops.attention_forward(q, k, v, w, cu, idx, max_seqlen=max(lens), select_mode=mode, block_size=block or 512)
    assert torch.isfinite(lse).all()
    heads = sorted({0, H // 2 + 1, H - 1})
    ref = _dense(q, k, v, w, cu, idx, block, heads)
    assert (out[:, heads].float() - ref).abs().max() <= 3 * UNIT[dt] * v.float().abs().max()
