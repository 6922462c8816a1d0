"""A whole prompt imported in one call: more (layer, row) pairs than one launch takes, and every
form of the caller's K/V, read back bit for bit."""
from __future__ import annotations

import ctypes

import pytest
import torch

from pager_hf import PagedDecoder

pytestmark = pytest.mark.gpu

MIB16 = 16 * 2**20


@pytest.mark.parametrize("layers,rows,n", [(24, 3, 333), (65, 1, 64), (2, 2, 31), (64, 1, 1)])
@pytest.mark.parametrize("form", ["tensors", "lists", "strided", "one tensor", "more rows"])
def test_prompt_reads_back(layers, rows, n, form):
    print(f"prompt import: {layers} layers, {rows} rows, {n} tokens, {form}", flush=True)
    hkv, d = 2, 16
    g = torch.Generator(device="cuda").manual_seed(layers + n)
    shape = (layers, rows + (form == "more rows"), hkv, n + 5, d)
    ks = torch.randn(*shape, device="cuda", generator=g).half()
    vs = torch.randn(*shape, device="cuda", generator=g).half()
    keys, values = [ks[i] for i in range(layers)], [vs[i] for i in range(layers)]
    if form == "lists":
        keys, values = [list(k) for k in keys], [list(v) for v in values]
    elif form == "strided":
        keys = [k.transpose(1, 2).contiguous().transpose(1, 2) for k in keys]
        values = [v[..., :n, :] for v in values]
        values = [torch.cat([v, v.new_zeros(*v.shape[:2], 5, d)], 2)[:, :, : n + 5] for v in values]
    elif form == "one tensor":
        keys, values = ks, vs
    dec = PagedDecoder(num_layers=layers, num_query_heads=4, num_kv_heads=hkv, head_dim=d, tokens_per_block=32,
                       dtype=torch.float16, device="cuda", pool_blocks=64, host_blocks=128, staging_blocks=16)
    sid = dec.add_session(capacity_tokens=n + 64, rows=rows, vram_budget=2 * MIB16, ram_budget=1 << 40,
                          recent_window=1, policy="recent_only")
    dec.prefill(sid, keys, values, n)
    for layer in range(layers):
        for row in range(rows):
            k, v = dec.pool.export_tokens(sid, row, layer, n)
            assert torch.equal(k, ks[layer, row, :, :n]) and torch.equal(v, vs[layer, row, :, :n]), (layer, row)
    dec.pool.close()


def test_prompt_import_refuses_what_a_single_import_does():
    dec = PagedDecoder(num_layers=2, num_query_heads=4, num_kv_heads=2, head_dim=16, tokens_per_block=32,
                       dtype=torch.float16, device="cuda", pool_blocks=8, host_blocks=16, staging_blocks=16)
    sid = dec.add_session(capacity_tokens=128, rows=2, vram_budget=2 * MIB16, ram_budget=1 << 40)
    dec.pool.set_length(sid, 40)
    good = [torch.zeros(2, 2, 40, 16, device="cuda").half() for _ in range(2)]
    flat = torch.zeros(2 * 2 * 40 * 16 + 1, device="cuda").half()
    off = flat[1:].view(2, 2, 40, 16)
    for keys, error in [([good[0], good[1][:1]], IndexError), ([good[0], good[1][:, :, :39]], ValueError),
                        ([good[0], good[1].float()], TypeError), ([good[0], good[1].cpu()], ValueError),
                        ([good[0], off], ValueError)]:
        with pytest.raises(error):
            dec.pool.import_prompt(sid, 2, keys, keys, 40)
    with pytest.raises(ValueError):
        dec.pool.import_prompt(sid, 2, good, good, 41)
    dec.pool.import_prompt(sid, 2, good, good, 40)
    dec.pool.close()


def test_index_buffer_of_a_failed_import_is_not_reused_before_the_gpu_has_read_it():
    """An import that reports an error after some of its launches went out: the buffer of block
    indices those launches read comes round again (four buffers) only once they have run."""
    hip = ctypes.CDLL("libamdhip64.so")
    layers, n = 65, 40  # two launches
    dec = PagedDecoder(num_layers=layers, num_query_heads=2, num_kv_heads=1, head_dim=16, tokens_per_block=32,
                       dtype=torch.float16, device="cuda", pool_blocks=16, host_blocks=16, staging_blocks=16)
    sids = [dec.add_session(capacity_tokens=128, rows=1, vram_budget=4 * MIB16, ram_budget=1 << 40) for _ in range(2)]
    kv = [torch.zeros(1, 1, n, 16, device="cuda").half() for _ in range(layers)]
    for sid in sids:
        dec.prefill(sid, kv, kv, n)
    torch.cuda.synchronize()
    torch.cuda._sleep(10_000_000)  # about 100 ms ahead of the imports
    done = torch.cuda.Event()
    done.record()
    assert hip.hipSetDevice(9999) != 0  # leaves an error for the import's launch check to find
    with pytest.raises(RuntimeError):
        dec.pool.import_prompt(sids[0], 1, kv, kv, n)
    assert not done.query()
    for _ in range(4):
        dec.pool.import_prompt(sids[1], 1, kv, kv, n)
    assert done.query()
    dec.pool.close()
