"""The forward's size rule as the library reports it, and the autotune's names for what runs (CPU only:
queries, no launches)."""
from __future__ import annotations

import ctypes

import pytest
import torch

from dsalt_amd import _lib, ops
from dsalt_amd.kernels import autotune as AT


def _tile(T, H, D, variant=0, S=1, G=None, K=64, block=0, dt=_lib.DTYPE_BF16):
    p = _lib.Problem(T, S, min(T, -(-T // S) + 5), H, G or H, D, K, 1 if block else 0, block, dt)
    out = [ctypes.c_int32() for _ in range(3)]
    rc = _lib.load().dsalt_fwd_tile(ctypes.byref(p), variant, *map(ctypes.byref, out))
    return tuple(t.value for t in out) if rc == 0 else rc


@pytest.mark.parametrize("args,want", [
    (dict(T=24575, H=16, D=64), (64, 64, 4)),                      # one token under 6144 tiles
    (dict(T=24576, H=16, D=64), (128, 64, 4)),
    (dict(T=24576, H=16, D=64, S=24), (128, 64, 4)),               # 1024 tokens a sequence
    (dict(T=24576, H=16, D=64, S=25), (64, 64, 4)),
    (dict(T=24576, H=16, D=64, block=256), (128, 64, 4)),
    (dict(T=24576, H=16, D=64, block=192), (64, 64, 4)),           # 128 rows would span two sets
    (dict(T=24576, H=16, D=64, block=100), (64, 64, 4)),
    (dict(T=24576, H=16, D=64, K=513), (64, 64, 4)),
    (dict(T=24576, H=16, D=64, dt=_lib.DTYPE_F32), (64, 32, 4)),
    (dict(T=100, H=4, D=128), (64, 32, 4)),
    (dict(T=131071, H=16, D=128), (64, 32, 4)),                    # one token under 32768 tiles
    (dict(T=131072, H=16, D=128), (128, 32, 8)),
    (dict(T=131072, H=16, D=128, block=512), (128, 32, 8)),
    (dict(T=131072, H=16, D=128, block=64), (64, 32, 4)),
    (dict(T=131072, H=16, D=128, S=2), (128, 32, 8)),              # 65536 tokens a sequence
    (dict(T=131072, H=16, D=128, S=3), (64, 32, 4)),
    (dict(T=131072, H=16, D=128, G=8), (64, 32, 4)),               # grouped heads
    (dict(T=65536, H=64, D=128, S=1024), (64, 32, 4)),             # many short sequences
    (dict(T=100, H=4, D=128, dt=_lib.DTYPE_F32), (64, 16, 4)),
])
def test_tile_by_size(args, want):
    assert _tile(**args) == want


@pytest.mark.parametrize("T", [640, 65536])
def test_bits_name_their_tiling_at_any_size(T):
    for D, variant, want in ((64, AT.VARIANT_FWD_BN64, (64, 64, 4)), (64, AT.VARIANT_FWD_BN32, (64, 32, 4)),
                             (64, AT.VARIANT_FWD_RG2, (128, 64, 4)), (64, AT.VARIANT_FWD_RG2 | AT.VARIANT_FWD_BN32, (128, 32, 4)),
                             (128, AT.VARIANT_FWD_BN32, (64, 32, 4)), (128, AT.VARIANT_FWD_BN64, (64, 64, 4)),
                             (128, AT.VARIANT_FWD_RG2, (128, 32, 4)), (128, AT.VARIANT_FWD_8W, (128, 32, 8))):
        assert _tile(T, 32, D, variant) == want, (D, variant)
        assert _tile(T, 32, D, variant | AT.VARIANT_LMK_SHORT) == want
    assert _tile(T, 32, 64, 64) == 1 and _tile(T, 32, 96) == 2  # unknown bit, unsupported head_dim


@pytest.mark.parametrize("T,H,D", [(2048, 4, 64), (32768, 16, 64), (2048, 4, 128), (131072, 16, 128)])
def test_autotune_names_the_tiling_that_runs(T, H, D):
    """Each candidate's blocks are those of the library's query, every forward tiling is listed once, and
    the 64-row blocks are among them whatever the library picks by itself."""
    q = torch.empty(1, dtype=torch.bfloat16).expand(T, H, D)  # shapes only
    cu, idx = torch.tensor([0, T], dtype=torch.int32), torch.empty(H, 1, 1, 64, dtype=torch.int32)
    runner = AT.operator_runner(q, q, q, None, cu, idx, None, max_seqlen=T)
    cands = AT._candidate_configs(D, None, 2, runner.forward_tile)
    assert cands[0]["variant"] == 0
    for c in cands:
        assert (c["BLOCK_M"], c["BLOCK_N"], c["num_warps"]) == _tile(T, H, D, c["variant"]), c
    fwd = [(c["BLOCK_M"], c["BLOCK_N"], c["num_warps"]) for c in cands if not c["variant"] & AT._BWD_BITS]
    assert len(set(fwd)) == len(fwd) and (64, 64 if D == 64 else 32, 4) in fwd
    assert ops.forward_tile(q, q, cu, idx, max_seqlen=T) == fwd[0]
