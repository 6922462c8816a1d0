"""The operator API's two call paths: _pgr_ops for plain tensors, the Python path for the rest.

Every form of argument goes through the public functions twice, as it is and with _pgr_ops
answering None (the general path alone): the results are the same bit for bit (both launch the
same kernels on the same values), and what one refuses the other refuses with the same error.
"""
from __future__ import annotations

import os
import subprocess
import sys

import pytest
import torch

from pager_hf import streaming_attention as S

gpu = pytest.mark.gpu


class _General:
    """_pgr_ops that hands every call to the general path."""

    def __getattr__(self, name):
        return lambda *args: None


class _Counting:
    def __init__(self, ops):
        self.ops, self.taken = ops, 0

    def __getattr__(self, name):
        fn = getattr(self.ops, name)

        def call(*args):
            got = fn(*args)
            self.taken += got is not None
            return got
        return call


class _Sub(torch.Tensor):
    pass


def _passes(q, k, v, valid, active, scale, softcap, dtype):
    """One fold, one two-pass run with mass and tail, and the outputs of both."""
    b, hq, d = q.shape
    m, l, acc = S.streaming_attention_state_init(b, hq, d, k.device)
    S.streaming_attention_step(q, k, v, m, l, acc, valid=valid, active=active, scale=scale, softcap=softcap)
    out = S.streaming_attention_finalize(acc, l, dtype)
    m2, l2, acc2 = S.streaming_attention_state_init(b, hq, d, k.device)
    S.streaming_attention_stats_step(q, k, m2, l2, valid=valid, active=active, scale=scale, softcap=softcap)
    mass = torch.zeros(b, hq, k.shape[2] // 16 + 1, device="cuda")
    S.streaming_attention_accumulate_step(q, k, v, m2, l2, acc2, mass, 0, 16, valid=valid, active=active, scale=scale,
                                          softcap=softcap)
    S.streaming_attention_fold_fixed_step(q, k, v, m2, l2, acc2, valid=valid, scale=scale, softcap=softcap)
    return [m, l, acc, out, m2, l2, acc2, mass]


def _forms():
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(*s, generator=g).half().cuda() for s in ((2, 6, 32), (2, 2, 40, 32), (2, 2, 40, 32)))
    valid = (torch.rand(2, 40, generator=g) > 0.3).to(torch.int32).cuda()
    active = torch.tensor([1, 0], dtype=torch.int32, device="cuda")
    plain = dict(q=q, k=k, v=v, valid=valid, active=active, scale=None, softcap=None, dtype=torch.float16)
    yield "plain", plain, True
    yield "no masks", dict(plain, valid=None, active=None), True
    yield "fp32", dict(plain, q=q.float(), k=k.float(), v=v.float(), dtype=torch.float32), True
    yield "bf16, scale and softcap", dict(plain, q=q.bfloat16(), k=k.bfloat16(), v=v.bfloat16(), scale=0.1,
                                          softcap=20.0, dtype=torch.bfloat16), True
    yield "integer scale and softcap", dict(plain, scale=1, softcap=30), None
    yield "zero softcap", dict(plain, softcap=0.0), True
    yield "bool masks", dict(plain, valid=valid.bool(), active=active.bool()), None
    yield "strided k", dict(plain, k=k.transpose(1, 2).contiguous().transpose(1, 2)), None
    yield "strided q and mask", dict(plain, q=q.repeat(1, 1, 2)[..., :32], valid=valid.repeat(1, 2)[:, ::2]), None
    yield "requires grad", dict(plain, q=q.clone().requires_grad_(), v=v.clone().requires_grad_()), True
    yield "parameter", dict(plain, q=torch.nn.Parameter(q.clone())), None
    yield "subclass", dict(plain, k=k.as_subclass(_Sub)), None
    yield "offset storage", dict(plain, q=torch.cat([q.flatten()[:1], q.flatten()])[1:].view(q.shape)), True


@gpu
def test_every_form_gives_the_general_paths_results(monkeypatch):
    for name, args, taken in _forms():
        print(f"call path: {name}", flush=True)
        count = _Counting(S._ops)
        monkeypatch.setattr(S, "_ops", count)
        with torch.no_grad():
            got = _passes(**args)
        monkeypatch.setattr(S, "_ops", _General())
        with torch.no_grad():
            want = _passes(**args)
        monkeypatch.setattr(S, "_ops", count.ops)
        for a, b in zip(got, want):
            # (an inactive row's output is 0 / 0 on both paths)
            torch.testing.assert_close(a, b, rtol=0, atol=0, equal_nan=True, msg=lambda m: f"{name}: {m}")
        assert taken is None or count.taken == 7, (name, count.taken)  # every call of _passes


@gpu
def test_both_paths_refuse_alike(monkeypatch):
    q, k = torch.zeros(1, 4, 32, device="cuda").half(), torch.zeros(1, 2, 16, 32, device="cuda").half()
    m, l, acc = S.streaming_attention_state_init(1, 4, 32, q.device)
    mass = torch.zeros(1, 4, 1, device="cuda")
    wide = torch.zeros(1, 34, 32, device="cuda").half()
    wm, wl, wacc = S.streaming_attention_state_init(1, 34, 32, q.device)
    odd = torch.zeros(1, 4, 40, device="cuda").half()
    om, ol, oacc = S.streaming_attention_state_init(1, 4, 40, q.device)
    okv = torch.zeros(1, 2, 16, 40, device="cuda").half()
    bad = [
        lambda: S.streaming_attention_step(q, k.float(), k, m, l, acc),
        lambda: S.streaming_attention_step(q, k, k[:, :, :8], m, l, acc),
        lambda: S.streaming_attention_step(q.cpu(), k, k, m, l, acc),
        lambda: S.streaming_attention_step(q, k, k, m.half(), l, acc),
        lambda: S.streaming_attention_step(q, k, k, m, l.t(), acc),
        lambda: S.streaming_attention_step(q, k, k, m, l, acc[..., :16]),
        lambda: S.streaming_attention_step(q, k, k, m, l, acc.transpose(1, 2).contiguous().transpose(1, 2)),
        lambda: S.streaming_attention_step(wide, k, k, wm, wl, wacc),
        lambda: S.streaming_attention_step(odd, okv, okv, om, ol, oacc),
        lambda: S.streaming_attention_step(q, k, k, m, l, acc, valid=torch.ones(1, 15, device="cuda")),
        lambda: S.streaming_attention_step(q, k, k, m, l, acc, scale=-1.0),
        lambda: S.streaming_attention_step(q, k, k, m, l, acc, scale=float("nan")),
        lambda: S.streaming_attention_stats_step(q.double(), k.double(), m, l),
        lambda: S.streaming_attention_accumulate_step(q, k, k, m, l, acc, mass, 1, 16),
        lambda: S.streaming_attention_accumulate_step(q, k, k, m, l, acc, mass, 0, 24),
        lambda: S.streaming_attention_accumulate_step(q, k, k, m, l, acc, mass[0], 0, 16),
        lambda: S.streaming_attention_finalize(acc, l[:, :2], torch.float16),
        lambda: S.streaming_attention_finalize(acc, l, torch.float64),
        lambda: S.streaming_attention_state_init(1, 4, 32, torch.device("cpu")),
    ]
    ops = S._ops
    for i, call in enumerate(bad):
        seen = []
        for path in (ops, _General()):
            monkeypatch.setattr(S, "_ops", path)
            with pytest.raises(Exception) as e:
                call()
            seen.append((e.type, str(e.value)))
        monkeypatch.setattr(S, "_ops", ops)
        assert seen[0] == seen[1], i
    # Empty chunks and batches fold nothing on either path.
    before = (m.clone(), l.clone(), acc.clone())
    S.streaming_attention_step(q, k[:, :, :0], k[:, :, :0], m, l, acc)
    assert all(torch.equal(a, b) for a, b in zip(before, (m, l, acc)))


@gpu
def test_functorch_and_modes_take_the_general_path():
    from torch.utils._python_dispatch import TorchDispatchMode

    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Mode():
        m, l, acc = S.streaming_attention_state_init(1, 2, 16, torch.device("cuda"))
    assert len(seen) == 3 and torch.isneginf(m).all() and not acc.any()
    x = torch.zeros(3, 1, 2, 16, device="cuda").half()
    kv = torch.zeros(1, 2, 16, 16, device="cuda").half()
    taken = []

    def probe(q):
        taken.append(S._ops.step(q, kv, kv, m, l, acc, None, None, None, None))
        return q

    torch.func.vmap(probe)(x)
    assert taken == [None]


_ALLOCATOR_C = """
#include <stddef.h>
#include <sys/types.h>
static int (*dev_malloc)(void**, size_t);
static int (*dev_free)(void*);
long sizes[1024];
int n_sizes;
void set_functions(void* m, void* f) { dev_malloc = m; dev_free = f; }
void* dev_alloc(ssize_t size, int device, void* stream) {
  void* p = 0;
  if (n_sizes < 1024) sizes[n_sizes++] = size;
  return dev_malloc(&p, size) == 0 ? p : 0;
}
void dev_release(void* p, ssize_t size, int device, void* stream) { dev_free(p); }
"""

_ALLOCATOR_PY = """
import ctypes, sys
import torch
so, hip = ctypes.CDLL(sys.argv[1]), ctypes.CDLL("libamdhip64.so")
so.set_functions(ctypes.cast(hip.hipMalloc, ctypes.c_void_p), ctypes.cast(hip.hipFree, ctypes.c_void_p))
torch.cuda.memory.change_current_allocator(
    torch.cuda.memory.CUDAPluggableAllocator(sys.argv[1], "dev_alloc", "dev_release"))
from pager_hf import _native as N
from pager_hf import streaming_attention as S
q, k = torch.randn(1, 4, 64).half().cuda(), torch.randn(1, 2, 3001, 64).half().cuda()
m, l, acc = S.streaming_attention_state_init(1, 4, 64, q.device)
S.streaming_attention_step(q, k, k, m, l, acc)
out = S.streaming_attention_finalize(acc, l, torch.float32)
p = torch.softmax(q.float().view(2, 2, 64) @ k[0].float().transpose(1, 2).contiguous() / 8, -1)
assert torch.allclose(out.view(2, 2, 64), p @ k[0].float(), atol=2e-3)
nbytes = N.lib().pgr_attn_workspace_bytes(1, 4, 2, 3001, 64, N.nat.MODE_FOLD, 16)
sizes = list((ctypes.c_long * 1024).in_dll(so, "sizes"))[: ctypes.c_int.in_dll(so, "n_sizes").value]
assert nbytes in sizes, (nbytes, sizes)
print("workspace from the program's allocator")
"""


@gpu
def test_workspace_comes_from_the_allocator_that_the_program_set(tmp_path):
    """change_current_allocator must run before any GPU allocation, so in a process of its own."""
    src, so = tmp_path / "allocator.c", tmp_path / "allocator.so"
    src.write_text(_ALLOCATOR_C)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    res = subprocess.run([sys.executable, "-c", _ALLOCATOR_PY, str(so)], capture_output=True, text=True, timeout=100,
                         env=dict(os.environ, PYTHONPATH=os.pathsep.join(sys.path)))
    assert res.returncode == 0 and "workspace from" in res.stdout, res.stdout + res.stderr


def test_ordinary_cpu_tensors_are_left_to_the_general_path():
    q, k = torch.zeros(1, 2, 16), torch.zeros(1, 2, 4, 16)
    assert S._ops.step(q, k, k, q[..., 0], q[..., 0], q, None, None, None, None) is None
    assert S._ops.finalize(q, q[..., 0], torch.float32) is None
    assert S._ops.state_init(1, 2, 16, torch.device("cpu")) is None
    with pytest.raises(TypeError):
        S._ops.step(q)
