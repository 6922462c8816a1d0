"""Paged decode over uneven sequences: how a launch is split, merged, and its block mass kept.

Sequences from one token to some hundred blocks in one step, so that the work items of a
sequence number from one to about a hundred (every slot count per merge thread, 1 to 16 and
beyond one batch), across head dims, block sizes (mass kept per tile, and per block where a
block holds many tiles) and element types. Against the float32 oracle: outputs within 2e-3
beyond the two roundings to the model's type that the reference's kernel makes too, and the
scores handed to the pager within 1e-5 (fp32 sums of weights at most 1, scores within 1e-5
relative of the oracle's).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from test_paged_decode_gpu import MIB16, TOL, Pair

pytestmark = pytest.mark.gpu

CONTEXTS = {
    "single": [3100],
    "6 slots": [1500],
    "10 slots": [2300],
    "12 slots": [2800],
    "few": [1, 1700, 40, 900],
    "many": [15, 16, 17, 33, 700, 95, 96, 97, 300, 64, 5, 128, 31, 32, 511, 210, 47, 48, 49, 1000],
}


@pytest.mark.parametrize("contexts", CONTEXTS)
@pytest.mark.parametrize("policy", ["recent_only", "sinks_heavy_hitter"])
@pytest.mark.parametrize("hq,hkv,d,tpb,dtype", [
    (14, 2, 64, 32, torch.float16), (12, 2, 128, 16, torch.bfloat16), (16, 1, 16, 64, torch.float16),
    (8, 1, 256, 32, torch.bfloat16), (4, 2, 256, 64, torch.float16), (6, 3, 32, 48, torch.float16),
    (4, 1, 64, 128, torch.float16), (8, 1, 256, 16, torch.bfloat16),
])
def test_uneven_sequences_match_the_oracle(hq, hkv, d, tpb, dtype, policy, contexts):
    print(f"uneven sequences: {contexts} {policy} {hq}/{hkv} d={d} tpb={tpb} {dtype}", flush=True)
    g = torch.Generator().manual_seed(d + tpb)
    ctx = CONTEXTS[contexts]
    p = Pair(layers=2, hq=hq, hkv=hkv, d=d, tpb=tpb, dtype=dtype, pool_blocks=sum(c // tpb + 4 for c in ctx),
             host_blocks=sum(c // tpb + 8 for c in ctx))
    for i, c in enumerate(ctx):  # every third sequence keeps most of its blocks on the host
        blocks = 2 if i % 3 == 2 else c // tpb + 3
        p.add(ctx=c, capacity=c + 3 * tpb, gen=g, vram_budget=blocks * MIB16, ram_budget=1024 * MIB16,
              recent_window=1, policy=policy)
    for _ in range(2):
        res, ref, _ = p.step(g, rounding_allowance=True)
        for sid in p.sids:
            got, want = res[sid]["block_attention"], ref["placement"][sid]["scores"]
            assert len(got) == len(want)
            if len(want):
                assert float(np.abs(np.array(got) - np.array(want)).max()) < 1e-5


def test_uneven_sequences_with_windows_and_softcap():
    g = torch.Generator().manual_seed(7)
    ctx = CONTEXTS["many"]
    p = Pair(layers=2, hq=8, hkv=2, d=64, tpb=32, dtype=torch.float16, pool_blocks=sum(c // 32 + 4 for c in ctx),
             host_blocks=sum(c // 32 + 8 for c in ctx), softcap=30.0)
    for c in ctx:
        p.add(ctx=c, capacity=c + 96, gen=g, vram_budget=(c // 32 + 3) * MIB16, ram_budget=1024 * MIB16,
              recent_window=1, policy="sinks_heavy_hitter")
    for _ in range(2):
        _, _, err = p.step(g, windows=[100, None], rounding_allowance=True)
        assert err < TOL


def test_more_than_512_slots_at_head_dim_16():
    """The merge's widest form: 1024 threads, 128 groups of slots combined in rounds."""
    g = torch.Generator().manual_seed(16)
    n = 33000  # 2063 blocks of 16 tokens, four per work item
    p = Pair(layers=1, hq=2, hkv=1, d=16, tpb=16, dtype=torch.float16, pool_blocks=n // 16 + 8, host_blocks=n // 16 + 8)
    p.add(ctx=n, capacity=n + 64, gen=g, vram_budget=(n // 16 + 4) * MIB16, ram_budget=1024 * MIB16, recent_window=1,
          policy="sinks_heavy_hitter")
    for _ in range(2):
        res, ref, _ = p.step(g, rounding_allowance=True)
        got, want = res[p.sids[0]]["block_attention"], ref["placement"][p.sids[0]]["scores"]
        assert float(np.abs(np.array(got) - np.array(want)).max()) < 1e-5
