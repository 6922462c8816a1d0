"""The operator kernels at the edges of their tiles, for every element type and head dim.

Chunk lengths around the 16-token tile, the 64-token workgroup and several tiles per wave (odd
and even counts, a ragged last tile), inputs whose storage starts one element past an aligned
address, and a mask. Oracle: the same attention in float64 on the CPU.

Tolerances. m and l carry fp32 rounding only: scores are sums of D products (D * 2^-24 relative
to sum |q k|, below 1e-5 absolute here), so 1e-4. acc / l and the outputs of 16-bit inputs add
two roundings to the 16-bit type (each weight before P.V, at most u * max|v|, and the output, at
most u * |out|; u = 2^-11 fp16, 2^-8 bf16); fp32 has neither.
"""
from __future__ import annotations

import math

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

pytestmark = pytest.mark.gpu

UNIT = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8, torch.float32: 0.0}
# (batch, query heads, KV heads, tokens): one tile and its neighbours, the workgroup's edge, and
# batch * KV heads * tiles beyond 2048, where a wave folds two, three and four tiles.
SHAPES = [(1, 7, 1, 1), (2, 4, 2, 15), (1, 16, 1, 16), (3, 2, 2, 17), (1, 5, 1, 64), (2, 6, 3, 65),
          (16, 8, 8, 272), (16, 8, 8, 523), (16, 16, 8, 1003)]


def _off_by_one(t):
    """The same values in storage that starts one element past an aligned address."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
    view = flat[1:].view(t.shape)
    view.copy_(t)
    return view


def _inputs(shape, d, dtype, seed):
    b, hq, hkv, n = shape
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(*s, generator=g).to(dtype) for s in ((b, hq, d), (b, hkv, n, d), (b, hkv, n, d)))
    valid = (torch.rand(b, n, generator=g) > 0.25).to(torch.int32)
    valid[:, -1] = 1
    return q, k, v, valid


def _reference(q, k, v, valid, softcap=None):
    b, hq, d = q.shape
    hkv, n = k.shape[1], k.shape[2]
    s = torch.matmul(q.double().view(b, hkv, -1, d), k.double().transpose(2, 3)) / math.sqrt(d)
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    s = s.masked_fill(valid[:, None, None, :] == 0, -math.inf)
    m = s.amax(-1)
    p = torch.exp(s - m[..., None])
    l = p.sum(-1)
    out = torch.matmul(p, v.double()) / l[..., None]
    return m.view(b, hq), l.view(b, hq), out.view(b, hq, d), (p / l[..., None]).view(b, hq, n)


def _check(got, want, atol):
    torch.testing.assert_close(got.double().cpu(), want, atol=atol, rtol=1e-4)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("d", [8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_one_and_two_passes_at_tile_edges(shape, d, dtype):
    print(f"operator tiles: {shape} d={d} {dtype}", flush=True)
    q, k, v, valid = _inputs(shape, d, dtype, 31 * d + shape[3])
    m_ref, l_ref, out_ref, w_ref = _reference(q, k, v, valid)
    u = UNIT[dtype]
    out_tol = 1e-4 + u * (float(v.abs().max()) + float(out_ref.abs().max()))
    q, k, v = _off_by_one(q), _off_by_one(k), _off_by_one(v)
    valid = valid.cuda()
    b, hq, n = q.shape[0], q.shape[1], k.shape[2]

    m, l, acc = streaming_attention_state_init(b, hq, d, q.device)
    streaming_attention_step(q, k, v, m, l, acc, valid=valid)
    _check(m, m_ref, 1e-4)
    _check(l, l_ref, 1e-4)
    _check(acc / l[..., None], out_ref, out_tol)
    _check(streaming_attention_finalize(acc, l, dtype), out_ref, out_tol)

    # Two passes: statistics, whole blocks with their mass, the tail at the fixed maximum.
    tpb = 32
    whole = n // tpb * tpb
    m2, l2, acc2 = streaming_attention_state_init(b, hq, d, q.device)
    streaming_attention_stats_step(q, k, m2, l2, valid=valid)
    _check(m2, m_ref, 1e-4)
    _check(l2, l_ref, 1e-4)
    mass = torch.zeros(b, hq, whole // tpb + 1, device="cuda")
    if whole:
        streaming_attention_accumulate_step(q, k[:, :, :whole], v[:, :, :whole], m2, l2, acc2, mass, 1, tpb,
                                            valid=valid[:, :whole])
        _check(mass[..., 1:], w_ref[..., :whole].reshape(b, hq, whole // tpb, tpb).sum(-1), 1e-4)
    assert float(mass[..., 0].abs().max()) == 0.0
    if whole < n:
        streaming_attention_fold_fixed_step(q, k[:, :, whole:], v[:, :, whole:], m2, l2, acc2,
                                            valid=valid[:, whole:])
    _check(streaming_attention_finalize(acc2, l2, dtype), out_ref, out_tol)


@pytest.mark.parametrize("dtype,d", [(torch.float32, 64), (torch.float32, 256), (torch.bfloat16, 256),
                                     (torch.float16, 16), (torch.float16, 8)])
def test_masked_values_and_non_finite_scores(dtype, d):
    """A masked position adds nothing whatever its K and V hold; a chunk with nothing valid
    leaves the state as it was; an infinite valid value reaches the output as it does in float64."""
    q, k, v, valid = _inputs((2, 4, 2, 37), d, dtype, 5)
    ref = _reference(q, k, v, valid)
    k, v = k.clone(), v.clone()
    off = (valid == 0)[:, None, :, None].expand_as(k)
    k[off] = math.nan
    v[off] = math.inf
    m, l, acc = streaming_attention_state_init(2, 4, d, torch.device("cuda"))
    streaming_attention_step(q.cuda(), k.cuda(), v.cuda(), m, l, acc, valid=torch.zeros_like(valid).cuda())
    assert torch.isneginf(m).all() and (l == 0).all() and (acc == 0).all()
    streaming_attention_step(q.cuda(), k.cuda(), v.cuda(), m, l, acc, valid=valid.cuda())
    tol = 1e-4 + UNIT[dtype] * 2 * float(_inputs((2, 4, 2, 37), d, dtype, 5)[2].abs().max())
    _check(acc / l[..., None], ref[2], tol)
    v[0, 0, 36, 0] = math.inf  # position 36 is valid
    m, l, acc = streaming_attention_state_init(2, 4, d, torch.device("cuda"))
    streaming_attention_step(q.cuda(), k.cuda(), v.cuda(), m, l, acc, valid=valid.cuda())
    got = acc / l[..., None]
    assert torch.isposinf(got[0, :2, 0]).all()
    assert torch.isfinite(got[0, 2:]).all() and torch.isfinite(got[1]).all() and torch.isfinite(got[0, :2, 1:]).all()


@pytest.mark.parametrize("hq,hkv,d,bound", [(6, 3, 8, 1.85e-7), (4, 2, 16, 2.13e-7), (16, 1, 32, 2.79e-7)])
def test_fp32_sums_at_small_head_dims(hq, hkv, d, bound):
    """The relative error of acc (2-norm, mean over 12 inputs) at 200 tokens, where one wave adds up 64
    of them. Bounds: half way between the tile's products added pairwise (1.65, 1.96 and 2.66e-7
    measured) and one chain of additions per wave (2.06, 2.32 and 2.93e-7); 12 inputs' means
    scatter by about 1%."""
    errors = []
    for seed in range(12):
        q, k, v, valid = _inputs((16, hq, hkv, 200), d, torch.float32, 100 * d + seed)
        valid.fill_(1)
        _, l_ref, out_ref, _ = _reference(q, k, v, valid)
        m, l, acc = streaming_attention_state_init(16, hq, d, torch.device("cuda"))
        streaming_attention_step(q.cuda(), k.cuda(), v.cuda(), m, l, acc)
        want = out_ref * l_ref[..., None]
        errors.append(float((acc.cpu().double() - want).norm() / want.norm()))
    mean = sum(errors) / len(errors)
    print(f"fp32 sums, head dim {d}: {mean:.3e}", flush=True)
    assert mean <= bound


@pytest.mark.parametrize("dtype,bound", [(torch.float16, 1.49e-4), (torch.bfloat16, 1.19e-3)], ids=["fp16", "bf16"])
@pytest.mark.parametrize("hq,hkv,d", [(16, 1, 32), (32, 4, 64), (28, 4, 128)])
def test_16_bit_weights_of_short_chunks(hq, hkv, d, dtype, bound):
    """The relative error of acc (2-norm, mean over 4 inputs) at 200 tokens in one workgroup, four
    tiles per wave: from rounding the weights before P.V, so from the maximum they are taken under.
    Bounds: half way between a maximum per tile, as split over workgroups (1.38 to 1.41e-4 in fp16,
    1.10 to 1.12e-3 in bf16) and one per wave (1.56 to 1.58e-4 and 1.25 to 1.27e-3)."""
    errors = []
    for seed in range(4):
        q, k, v, valid = _inputs((16, hq, hkv, 200), d, dtype, 100 * d + seed)
        valid.fill_(1)
        _, l_ref, out_ref, _ = _reference(q, k, v, valid)
        m, l, acc = streaming_attention_state_init(16, hq, d, torch.device("cuda"))
        streaming_attention_step(q.cuda(), k.cuda(), v.cuda(), m, l, acc)
        want = out_ref * l_ref[..., None]
        errors.append(float((acc.cpu().double() - want).norm() / want.norm()))
    mean = sum(errors) / len(errors)
    print(f"{dtype} weights, head dim {d}: {mean:.3e}", flush=True)
    assert mean <= bound
