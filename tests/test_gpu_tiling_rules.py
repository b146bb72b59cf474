"""Size rules that choose a kernel or a split of the work: both sides of each line, at lengths off
every tile edge, against plain torch in float32 / float64 on the GPU.

Bound of a 16-bit forward (u = 2^-8 for bfloat16, 2^-11 for float16, the largest relative error of a
rounding): each probability is rounded in the product and in its row sum alike, which moves the
quotient by at most u max|v - o| <= 2 u max|v|, and the quotient is rounded once more: 3 u max|v| with
every rounding at its largest and of one sign (float32 sums add orders of magnitude less).  The tests
ask for half of that.  The LSE is the logarithm of the rounded probabilities' sum: at most u off."""
from __future__ import annotations

import math

import pytest
import torch

from dsalt_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
UNIT = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


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
    """Outputs and LSE of the given query heads, float32, one (head, sequence) at a time."""
    out = torch.zeros(q.shape[0], len(heads), q.shape[2], device=DEV)
    lse = torch.zeros(q.shape[0], len(heads), device=DEV)
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
            sc.masked_fill_(~mask, float("-inf"))
            lse[a:a + n, c] = torch.logsumexp(sc, 1)
            out[a:a + n, c] = torch.softmax(sc, 1) @ v[a:a + n, h // rep].float()
    return out, lse


@pytest.mark.parametrize("lens,H,G,D,dt,block", [
    ([8190], 8, 8, 64, torch.bfloat16, 0),                # the blocks make their own row plan
    ([8200], 8, 8, 64, torch.bfloat16, 0),                # past 1024 tiles a launch before them does
    ([6143], 16, 4, 64, torch.bfloat16, 0),               # 64-row blocks of a plan made before
    ([6145], 16, 16, 64, torch.bfloat16, 0),              # an odd number of tiles
    ([4097, 1, 2050, 190], 16, 2, 64, torch.float16, 0),  # ragged
    ([6400], 16, 4, 64, torch.bfloat16, 256),
    ([6400], 16, 4, 64, torch.bfloat16, 192),
    ([12288], 32, 8, 64, torch.bfloat16, 0),              # 6144 tiles: 128-row blocks
    ([12350], 32, 8, 64, torch.float16, 0),               # an odd number of tiles in them
    ([6400, 1, 5950], 32, 4, 64, torch.bfloat16, 256),    # block sets, whole 128-row blocks in a set
    ([12350], 32, 8, 64, torch.bfloat16, 192),            # sets of 192 rows keep 64-row blocks
    ([8191], 128, 8, 128, torch.bfloat16, 0),             # head_dim 128, four waves
    ([8321], 128, 8, 128, torch.bfloat16, 0),             # an odd number of tiles
    ([5000, 3333], 128, 128, 128, torch.float16, 0),
])
def test_forward_tiling_by_size(lens, H, G, D, dt, block):
    q, k, v, w, cu, idx = _inputs(lens, H, G, D, 9, 150, dt, seed=sum(lens), block=block)
    mode = ops.SELECT_BLOCK if block else ops.SELECT_GLOBAL
    out, lse = ops.attention_forward(q, k, v, w, cu, idx, max_seqlen=max(lens), select_mode=mode, block_size=block or 512)
    assert torch.isfinite(lse).all()
    heads = sorted({0, H // 2 + 1, H - 1})
    ref, rlse = _dense(q, k, v, w, cu, idx, block, heads)
    assert (out[:, heads].float() - ref).abs().max() <= 1.5 * UNIT[dt] * v.float().abs().max()
    assert (lse[:, heads] - rlse).abs().max() <= UNIT[dt] + 1e-5


@pytest.mark.parametrize("lens,H", [([8190], 8), ([8200], 8), ([700, 0, 1, 64, 65], 4), ([700, 0, 1, 64, 65], 160),
                                    ([2000] + [5] * 100, 4)])
@pytest.mark.parametrize("D,dt", [(64, torch.bfloat16), (128, torch.float16), (64, torch.float32)])
def test_plan_made_by_the_blocks(lens, H, D, dt):
    """The row plan of the attention's own blocks (small calls) is the selection's, byte for byte,
    tiles past a sequence's end included, and the output that of a plan made before."""
    q, k, v, w, cu, idx = _inputs(lens, H, 2, D, 9, 150, dt, seed=3)
    h, alpha = torch.randn(q.shape[0], 64, device=DEV).to(dt), torch.full((H,), 0.5, device=DEV)
    made, given = (ops.new_plan(q, k, cu, idx, max_seqlen=max(lens)).fill_(0) for _ in range(2))
    ops.select_landmarks(h, v, alpha, w, cu, 4, max_seqlen=max(lens), plan=given)
    a = ops.attention_forward(q, k, v, w, cu, idx, max_seqlen=max(lens), plan=made)
    b = ops.attention_forward(q, k, v, w, cu, idx, max_seqlen=max(lens), plan=given, plan_ready=True)
    n = sum(x * y for x, y in ((64, 1), (16, 4), (1, 4))) * len(lens) * -(-max(lens) // 64)
    assert torch.equal(made, given) and made.numel() >= n
    T = int(cu[-1])
    assert torch.equal(a[0][:T], b[0][:T]) and torch.equal(a[1][:T], b[1][:T])


@pytest.mark.parametrize("lens,H,G,D,K,dt", [
    ([1201, 77, 1, 640], 8, 2, 64, 32, torch.float16),    # four heads of a group side by side; row sums split in four
    ([1201, 77, 1, 640], 8, 4, 64, 128, torch.bfloat16),  # two heads side by side, largest set searched by a wave
    ([700, 65], 16, 2, 64, 129, torch.bfloat16),          # eight heads swept in order, larger sets
    ([2100], 12, 3, 128, 100, torch.bfloat16),            # head_dim 128: swept in order
    ([64, 63], 4, 1, 64, 1, torch.bfloat16),              # a single tile, fewer chunks than a split
    ([3000], 128, 32, 64, 70, torch.bfloat16),            # few chunks: one wave a row
    ([7200], 32, 16, 64, 128, torch.bfloat16),            # eight chunks, 2048 owner rows: one wave a row
    ([7200], 32, 16, 64, 127, torch.bfloat16),            # 2032 owner rows: four waves a row
    ([4097], 128, 32, 64, 20, torch.bfloat16),            # 2080 blocks: the four heads of a group in order
    ([4161], 32, 8, 64, 20, torch.bfloat16),              # 528 blocks, likewise
    ([6145], 32, 8, 64, 20, torch.float16),               # 776 blocks: side by side in their fourth round
    ([70] * 60 + [0, 1, 64, 65], 8, 4, 64, 20, torch.bfloat16),  # many rows of short sequences
    ([30] * 300, 8, 4, 64, 4, torch.bfloat16),            # 1200 blocks of one short sequence: heads in order
    ([9300] + [0, 40] * 60, 8, 8, 64, 6, torch.bfloat16),  # many rows, most of them empty, 10 chunks
    ([520, 333], 4, 1, 64, 9, torch.float32),
])
@pytest.mark.parametrize("train", [False, True])
def test_grouped_gradients_equal_those_of_repeated_heads(lens, H, G, D, K, dt, train):
    """dK / dV of grouped heads against the one-head-per-key/value-head kernels on repeated k and v,
    summed over each group.  Both form the same products per head; the repeated heads' gradients
    are rounded to the tensor type before the sum and the grouped ones after it: at most 2 rep u of the
    largest head's gradient for rep heads a group.  Asked for is (rep + 2) u / 2 (roundings of both signs;
    float32: sums in another order, 1e-5)."""
    q, k, v, w, cu, idx = _inputs(lens, H, G, D, K, 200, dt, seed=K)
    rep = H // G
    for hh in range(0, H, 2):  # half of the heads share their neighbour's set, as value norms make them do
        idx[hh] = idx[(hh + 1) % H]
    if K > 2:  # a repeated position in the first head's sets (ascending still)
        idx[0, :, :, 1] = idx[0, :, :, 0]
    g = torch.Generator(device=DEV).manual_seed(1)
    do = torch.randn(q.shape, generator=g, device=DEV).to(dt)
    ml = max(lens)
    if train:
        wc = w.float() + 0.25
        lw = torch.randn(idx.shape, generator=g, device=DEV)
        run = lambda kk, vv: ops.train_backward(do, q, kk, vv, *ops.train_forward(q, kk, vv, wc, cu, idx, lw, max_seqlen=ml),  # noqa: E731
                                                wc, cu, idx, lw, max_seqlen=ml)
    else:
        run = lambda kk, vv: ops.attention_backward(do, q, kk, vv, *ops.attention_forward(q, kk, vv, w, cu, idx, max_seqlen=ml),  # noqa: E731
                                                    w, cu, idx, max_seqlen=ml)
    got, ref = run(k, v), run(k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1))
    assert torch.equal(got[0], ref[0]) and torch.equal(got[3], ref[3])  # dq, d_bias: per query head
    unit = (rep + 2) / 2 * UNIT[dt] if dt != torch.float32 else 1e-5
    for a, b in ((got[1], ref[1]), (got[2], ref[2])):
        b = b.double()
        s = b.view(b.shape[0], G, rep, D).sum(2)
        assert (a.double() - s).abs().max() <= unit * b.abs().max()
    again = run(k, v)
    for a, b in zip(got, again):
        assert torch.equal(a, b)  # one writer per element, sums in a fixed order


@pytest.mark.parametrize("lens,K", [([2047], 32), ([2048], 600), ([2049], 32), ([1, 0, 30, 2048], 40), ([5, 3], 2048),
                                    ([2048, 2049, 700], 512), ([1500], 1)])
@pytest.mark.parametrize("scope", [ops.STATS_PACKED, ops.STATS_SEQUENCE])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_selection_of_one_part_sets_bit_exact(lens, K, scope, dt):
    """Sequences of up to 2048 tokens are selected by one block a set, longer ones by parts and
    merges: the oracle's indices on both sides."""
    import numpy as np

    from oracle import select as OS
    from tests.helpers import bits, oracle_dtype
    g = torch.Generator().manual_seed(sum(lens) + K)
    T, H, G = sum(lens), 4, 2
    h, v = torch.randn(T, 96, generator=g).to(dt), torch.randn(T, G, 64, generator=g).to(dt)
    v[torch.rand(T, generator=g) < 0.1] = 0  # ties
    w = torch.randint(1, 200, (T,), generator=g, dtype=torch.int32)
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    alpha = torch.tensor([0.0, 0.3, 0.7, 1.0])
    idx = ops.select_landmarks(h.to(DEV), v.to(DEV), alpha.to(DEV), w.to(DEV), cu.to(DEV), K, max_seqlen=max(lens),
                               stats_scope=scope)
    ref = OS.select(bits(h), bits(v), alpha.numpy(), w.numpy(), cu.numpy(), K, oracle_dtype(dt), stats_scope=scope)
    assert np.array_equal(idx.cpu().numpy(), ref)
