"""The native host calls (csrc/host_calls.cpp) against the general path in Python: the
same outputs bit for bit and the same layouts over the layouts, dtypes and scalar forms a
call can have, and the same exception where a call is refused.  ``native`` says which of
the forms the native calls serve; the others must reach the general path."""

import pytest
import torch

import mimir_amd
from mimir_amd import _capi
from mimir_amd import prefixlm as P
from mimir_amd.cache import Cache, attention_with_cache
from mimir_amd.workloads import make_case

pytestmark = pytest.mark.gpu


class _Counted:
    """The host calls with the number of calls each served, or none at all (``off``)."""

    def __init__(self, off):
        self.off, self.served, self.real = off, 0, _capi.host()

    def __getattr__(self, name):
        def call(*args):
            res = None if self.off else getattr(self.real, name)(*args)
            self.served += res is not None
            return res

        return call


def both(monkeypatch, fn, native):
    """fn() through the native calls and through the general path; both results (or exceptions)."""
    got = []
    for off in (False, True):
        host = _Counted(off)
        monkeypatch.setattr(_capi, "host", lambda h=host: h)
        try:
            got.append(fn())
        except Exception as e:  # compared below
            got.append(e)
        monkeypatch.undo()
        if not off:
            assert host.served == native, host.served
    a, b = got
    if isinstance(b, Exception):
        assert type(a) is type(b) and str(a) == str(b), (a, b)
        return
    assert not isinstance(a, Exception), a
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride()
        assert torch.equal(x, y)


def _case(device, dtype, d=64):
    return make_case([70, 33, 1], [20, 33, 0], 4, 2, d, seed=3, dtype=dtype, pad_to=120).to(device)


def _layouts(c, form):
    T = c.T
    if form == "contiguous":
        return c.q, c.k, c.v
    if form == "projection":  # strided head slices of one buffer
        x = torch.cat((c.q, c.k, c.v), dim=1)
        return x.split((4, 2, 2), dim=1)
    if form == "heads_first":  # [H, T, D] storage
        return tuple(t.transpose(0, 1).contiguous().transpose(0, 1) for t in (c.q, c.k, c.v))
    if form == "offset":  # rows off a 16-byte boundary
        return tuple(torch.cat((t.flatten(), t.flatten()[:1]))[1:].as_strided(t.shape, t.stride()) for t in (c.q, c.k, c.v))
    if form == "expanded":  # one token for all: the row stride is 0
        return c.q, c.k[:1].expand(T, 2, -1), c.v
    if form == "dim_strided":  # every second column
        return tuple(torch.stack((t, t), dim=-1).flatten(-2)[..., ::2] for t in (c.q, c.k, c.v))
    raise AssertionError(form)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("form,native", [("contiguous", 2), ("projection", 2), ("heads_first", 2), ("offset", 0),
                                         ("expanded", 0), ("dim_strided", 0)])
def test_step(device, monkeypatch, dtype, form, native):
    c = _case(device, dtype)
    q, k, v = (t.detach().requires_grad_(True) for t in _layouts(c, form))

    def step():
        out, lse = mimir_amd.prefixlm_attn_fwd(q, k, v, False, *c.oracle_args(), c.max_seqlen_all)
        return (out, lse, *torch.autograd.grad(out, (q, k, v), c.dout))

    both(monkeypatch, step, native)


@pytest.mark.parametrize("form,native", [("int64 metadata", 0), ("cpu metadata", 0), ("int32 scalar", 0), ("ints", 2),
                                         ("numseqs too large", 0), ("total too large", 0), ("dout strided", 2),
                                         ("dout fp32", 1), ("fp16", 0), ("kv heads", 0), ("causal", 2)])
def test_step_arguments(device, monkeypatch, form, native):
    c = _case(device, torch.bfloat16)
    q, k, v, dout = c.q, c.k, c.v, c.dout
    meta = [c.prefix_lens, c.causal_lens, c.cu_seqlens]
    total, n, longest = c.total_seqlen, c.numseqs, c.max_seqlen_all
    if form == "int64 metadata":
        meta = [m.long() for m in meta]
    elif form == "cpu metadata":
        meta = [m.cpu() for m in meta]
    elif form == "int32 scalar":
        total = total.int()
    elif form == "ints":
        total, n, longest = int(total), int(n), int(longest)
    elif form == "numseqs too large":
        n = torch.tensor(500)
    elif form == "total too large":
        total = torch.tensor(500)
    elif form == "dout strided":
        dout = dout.transpose(0, 1).contiguous().transpose(0, 1)
    elif form == "dout fp32":
        dout = dout.float()
    elif form == "fp16":
        q, k, v, dout = (t.half() for t in (q, k, v, dout))
    elif form == "kv heads":
        q = q[:, :3]
        dout = dout[:, :3]
    q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))

    def step():
        out, lse = mimir_amd.prefixlm_attn_fwd(q, k, v, form == "causal", *meta, total, n, longest)
        if form == "dout fp32":
            return P._bwd_impl(dout, q.detach(), k.detach(), v.detach(), out.detach(), lse, q.new_empty(0),
                               q.new_empty(0, dtype=torch.int32), False, *meta, total, n, longest, 0.125)
        return (out, lse, *torch.autograd.grad(out, (q, k, v), dout))

    both(monkeypatch, step, native)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("rope", [False, True])
def test_layer(device, monkeypatch, dtype, rope):
    c = _case(device, dtype)
    T, d = c.T, 64
    x = torch.randn(T, 12 * d, device=device).to(dtype).requires_grad_(True)
    dy = torch.randn(T, 4 * d, device=device).to(dtype)
    angle = torch.randn(T, d // 2, device=device).repeat(1, 2)
    tables = (angle.cos(), angle.sin()) if rope else None
    names = ("prefix_lens", "causal_lens", "cu_seqlens", "total_seqlen", "numseqs")

    def step():
        y = mimir_amd.gated_attention(x, tables, 4, 2, False, max_seqlen_all=c.max_seqlen_all,
                                      **dict(zip(names, c.oracle_args())))
        return (y, *torch.autograd.grad(y, x, dy))

    both(monkeypatch, step, 4 if rope else 2)


@pytest.mark.parametrize("form,native", [("plain", 1), ("rows", 1), ("int32", 1), ("cpu lengths", 0), ("heads_first", 1),
                                         ("offset", 0), ("mixed indices", 0), ("fp32", 0), ("cache shape", 0)])
def test_cache(device, monkeypatch, form, native):
    gen = torch.Generator().manual_seed(7)
    mk = lambda *s: torch.randn(*s, generator=gen).to(torch.bfloat16).to(device)
    q, k, v = mk(3, 2, 8, 64), mk(3, 2, 2, 64), mk(3, 2, 2, 64)
    keys, values = mk(4, 200, 2, 64), mk(4, 200, 2, 64)
    lens, rows = torch.tensor([0, 100, 198], device=device), None
    if form == "rows":
        rows = torch.tensor([3, 0, 2], device=device)
    elif form == "int32":
        lens = lens.int()
    elif form == "cpu lengths":
        lens = lens.cpu()
    elif form == "heads_first":
        keys, values = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (keys, values))
    elif form == "offset":
        q = torch.cat((q.flatten(), q.flatten()[:1]))[1:].view(q.shape)
    elif form == "mixed indices":
        rows = torch.tensor([3, 0, 2], device=device, dtype=torch.int32)
    elif form == "fp32":
        q = q.float()
    elif form == "cache shape":
        keys = keys[:, :, :1]

    def step():
        cache = Cache(keys.clone(), values.clone())
        out = attention_with_cache(q, k, v, cache, lens, True, rows)
        return out, cache.keys, cache.values

    both(monkeypatch, step, native)


def test_rope(device, monkeypatch):
    x = torch.randn(33, 6, 64, device=device).bfloat16()
    cos, sin = torch.randn(2, 33, 64, device=device)
    both(monkeypatch, lambda: (mimir_amd.rope(x[:, 1:5], cos, sin),), 1)
    both(monkeypatch, lambda: (mimir_amd.rope(x, cos[None], sin[None], inverse=True),), 0)
    both(monkeypatch, lambda: (mimir_amd.rope(x, cos.double(), sin),), 0)

    def in_place():
        y = x.clone()
        part = y[:, 2:]
        assert mimir_amd.rope(part, cos, sin, out=part) is part
        return (y,)

    both(monkeypatch, in_place, 1)
