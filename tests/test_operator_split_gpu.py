"""One workgroup per head or several: the operator API around the sizes where a chunk is split.

A chunk that one workgroup holds updates the running state in the attention launch; a longer one
goes through partials and the merge, whose shape follows the number of splits. Chunks on both
sides of the line are folded into one carried state, with masked rows, fully masked rows and
inactive rows, and compared with float64. Tolerances as at the tile edges: 1e-4 for fp32 sums,
plus two roundings to the 16-bit type for what P.V and the output round.
"""
from __future__ import annotations

import pytest
import torch

from pager_hf.streaming_attention import (
    streaming_attention_accumulate_step,
    streaming_attention_finalize,
    streaming_attention_fold_fixed_step,
    streaming_attention_state_init,
    streaming_attention_stats_step,
    streaming_attention_step,
)
from test_operator_tiles_gpu import UNIT, _check, _inputs, _reference

pytestmark = pytest.mark.gpu

# Tokens per chunk: one workgroup (up to 256, or 128 at head dim 256), the sizes next to the line,
# and enough splits for 2, 4, 8 and more partials per merge thread.
CHUNKS = [[64, 65, 128, 129], [256, 257, 1, 480], [1024, 16], [2600, 3], [5001, 255]]


@pytest.mark.parametrize("chunks", CHUNKS, ids=lambda c: "+".join(map(str, c)))
@pytest.mark.parametrize("hq,hkv,d,dtype", [
    (7, 1, 64, torch.float16), (16, 1, 128, torch.bfloat16), (6, 3, 8, torch.float16), (4, 2, 256, torch.bfloat16),
    (4, 2, 256, torch.float32), (4, 2, 128, torch.float32), (5, 1, 32, torch.float32), (4, 4, 16, torch.float16),
])
def test_chunks_on_both_sides_of_the_split(hq, hkv, d, dtype, chunks):
    print(f"operator split: {hq}/{hkv} d={d} {dtype} {chunks}", flush=True)
    n = sum(chunks)
    q, k, v, valid = _inputs((2, hq, hkv, n), d, dtype, d + n)
    valid[1, : n // 3] = 0  # row 1 starts late: its first chunks may hold nothing valid
    m_ref, l_ref, out_ref, w_ref = _reference(q, k, v, valid)
    out_tol = 1e-4 + UNIT[dtype] * (float(v.abs().max()) + float(out_ref.abs().max()))
    q, k, v, valid = (x.cuda() for x in (q, k, v, valid))
    edges = [sum(chunks[:i]) for i in range(len(chunks) + 1)]
    parts = [(k[:, :, a:b].contiguous(), v[:, :, a:b].contiguous(), valid[:, a:b].contiguous())
             for a, b in zip(edges, edges[1:])]
    m, l, acc = streaming_attention_state_init(2, hq, d, q.device)
    m2, l2, acc2 = streaming_attention_state_init(2, hq, d, q.device)
    for kc, vc, ok in parts:
        before = [x.clone() for x in (m, l, acc)]
        streaming_attention_step(q, kc, vc, m, l, acc, valid=ok)
        for r in range(2):
            if not bool(ok[r].any()):  # nothing valid: the row's state is untouched
                assert all(torch.equal(x[r], y[r]) for x, y in zip(before, (m, l, acc)))
        streaming_attention_stats_step(q, kc, m2, l2, valid=ok)
    _check(m, m_ref, 1e-4)
    _check(l, l_ref, 1e-4)
    _check(streaming_attention_finalize(acc, l, dtype), out_ref, out_tol)
    _check(m2, m_ref, 1e-4)
    _check(l2, l_ref, 1e-4)
    mass = torch.zeros(2, hq, sum((c + 31) // 32 for c in chunks), device="cuda")
    first, want = 0, []
    for (kc, vc, ok), a, b in zip(parts, edges, edges[1:]):
        if (b - a) % 32 == 0:
            streaming_attention_accumulate_step(q, kc, vc, m2, l2, acc2, mass, first, 32, valid=ok)
            want.append((first, w_ref[..., a:b].reshape(2, hq, -1, 32).sum(-1)))
            first += (b - a) // 32
        else:
            streaming_attention_fold_fixed_step(q, kc, vc, m2, l2, acc2, valid=ok)
    for at, w in want:
        _check(mass[..., at:at + w.shape[-1]], w, 1e-4)
    _check(streaming_attention_finalize(acc2, l2, dtype), out_ref, out_tol)


@pytest.mark.parametrize("n", [40, 256, 700])
def test_inactive_rows_keep_their_state(n):
    q, k, v, _ = _inputs((3, 6, 2, n), 64, torch.float16, n)
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    active = torch.tensor([1, 0, 1], dtype=torch.int32, device="cuda")
    m, l, acc = streaming_attention_state_init(3, 6, 64, q.device)
    streaming_attention_step(q, k, v, m, l, acc)
    before = [x.clone() for x in (m, l, acc)]
    streaming_attention_step(q, k, v, m, l, acc, active=active)
    assert all(torch.equal(x[1], y[1]) for x, y in zip(before, (m, l, acc)))
    torch.testing.assert_close(l[0], 2 * before[1][0], rtol=1e-5, atol=0)
    torch.testing.assert_close(acc[2], 2 * before[2][2], rtol=1e-5, atol=1e-5)
