"""Prompt import: what the pool hands to the library. The import kernel reads [Hkv, n_src, D] by the
pool's Hkv and D and one n_src for K and V, so a tensor of another shape is refused before a launch."""
from __future__ import annotations

import weakref

import pytest
import torch

from pager_hf.kv_pool import NativeKVPool

LAYERS, ROWS, HKV, D, N = 2, 2, 2, 16, 40


class _Pool(NativeKVPool):
    """The argument handling of a pool without a device: records the library calls."""

    def __init__(self):
        self.num_layers, self.num_kv_heads, self.head_dim = LAYERS, HKV, D
        self.device, self.dtype, self.lib, self.handle = torch.device("cpu"), torch.float16, _Lib(), None
        self.calls = []

    def _stream(self):
        return 0

    def _call(self, what, fn, *args):
        self.calls.append((fn, args))


class _Lib:
    def __getattr__(self, name):
        return name


def _kv(*shape):
    return torch.arange(torch.Size(shape).numel(), dtype=torch.float16).remainder(97).view(shape)


def _import(pool, form, k, v):
    """One (row, layer) or the whole prompt, with k, v [rows, Hkv, n, D] as layer 1's."""
    if form == "single":
        pool.import_tokens(0, 0, 1, k[0], v[0], N)
    else:
        good = _kv(ROWS, HKV, N, D)
        keys, values = [good, k], [good, v]
        if form == "lists":
            keys, values = [list(x) for x in keys], [list(x) for x in values]
        pool.import_prompt(0, ROWS, keys, values, N)


@pytest.mark.parametrize("form", ["single", "tensors", "lists"])
@pytest.mark.parametrize("bad", [(ROWS, HKV, N - 1, D), (ROWS, HKV - 1, N, D), (ROWS, HKV + 1, N, D),
                                 (ROWS, HKV, N, D - 8), (ROWS, HKV, N, 2 * D), (ROWS, HKV, N)])
@pytest.mark.parametrize("side", ["keys", "values", "both"])
def test_other_shapes_are_refused(form, bad, side):
    if side == "both" and bad[2:] == (N - 1, D):
        return  # K and V of one length below n_tokens: refused by the library
    good, other = _kv(ROWS, HKV, N, D), _kv(*bad)
    k, v = (other if side != "values" else good), (other if side != "keys" else good)
    pool = _Pool()
    with pytest.raises(ValueError):
        _import(pool, form, k, v)
    assert not pool.calls


@pytest.mark.parametrize("form", ["single", "tensors", "lists"])
@pytest.mark.parametrize("nk,nv", [(N, N + 3), (N + 3, N), (N + 1, N + 3)])
def test_keys_and_values_of_two_lengths_share_one_stride(form, nk, nv):
    pool = _Pool()
    _import(pool, form, _kv(ROWS, HKV, nk, D), _kv(ROWS, HKV, nv, D))
    fn, args = pool.calls[-1]
    n_src = args[5] if form == "single" else list(args[5])[-1]
    assert n_src == N  # both cut to the prompt's length


@pytest.mark.parametrize("form", ["single", "tensors", "lists"])
def test_one_length_beyond_the_prompt_is_read_in_place(form):
    k, v = _kv(ROWS, HKV, N + 5, D), _kv(ROWS, HKV, N + 5, D)
    pool = _Pool()
    _import(pool, form, k, v)
    fn, args = pool.calls[-1]
    if form == "single":
        assert args[3:6] == (k.data_ptr(), v.data_ptr(), N + 5)
    else:
        assert args[:3] == (0, 0, LAYERS)  # session, first layer, layers
        assert list(args[3])[-1] == k[1].data_ptr() and list(args[4])[-1] == v[1].data_ptr()
        assert list(args[5])[-2:] == [N + 5] * 2


@pytest.mark.parametrize("n,layers,spans", [
    (16384, 8, [(0, 8)]),  # 4 MiB of copies per layer
    (16384, 40, [(0, 16), (16, 16), (32, 8)]),
    (524288, 2, ["row 0", "row 1", "row 0", "row 1"]),  # 128 MiB: a row's K and V at a time
])
def test_copies_of_a_strided_prompt_are_bounded(n, layers, spans):
    strided = _kv(1, n, HKV, D).transpose(1, 2).expand(ROWS, HKV, n, D)
    live, most = [], []

    class Pool(_Pool):
        def _row_kv(self, k, v, n_tokens):
            got = super()._row_kv(k, v, n_tokens)
            live.extend(weakref.ref(t) for t in got)
            return got

        def _call(self, what, fn, *args):
            most.append(sum(t().numel() * 2 for t in live if t() is not None))
            super()._call(what, fn, *args)

    pool = Pool()
    pool.num_layers = layers
    pool.import_prompt(0, ROWS, [strided] * layers, [strided] * layers, n)
    assert max(most) <= 64 << 20
    assert [f"row {a[1]}" if fn == "pgr_kv_import" else a[1:3] for fn, a in pool.calls] == spans
