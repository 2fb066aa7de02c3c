"""Which KV caches the attention kernels may append to themselves: ``cache_rows_distinct``
(csrc/prefixlm_cache_layout.h, built for the host) against a count of the addresses that the
rows of both cache tensors take.  It may call a distinct layout shared (that costs a launch),
never a shared one distinct, and the layouts in ordinary use have to be distinct."""

import ctypes
import itertools
import os
import subprocess
from pathlib import Path

import pytest
import torch

from mimir_amd import _capi

CSRC = Path(__file__).resolve().parents[1] / "mimir_amd" / "csrc"
D = 64


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    out = tmp_path_factory.mktemp("layout") / "layout.so"
    src = f'#include "{CSRC}/prefixlm_cache_layout.h"\n' \
          'extern "C" int distinct(const MimirCacheAttnParams* p) { return mimir::cache_rows_distinct(*p); }\n'
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-shared", "-fPIC", "-x", "c++", "-", "-o", str(out)],
                   input=src, text=True, check=True)
    lib = ctypes.CDLL(str(out))
    lib.distinct.argtypes = [ctypes.POINTER(_capi.CacheAttnParams)]

    def call(keys, values, batch, indices):
        p = _capi.CacheAttnParams()
        p.cache_k, p.cache_v = keys.data_ptr(), values.data_ptr()
        p.ck_stride_batch, p.ck_stride_token, p.ck_stride_head = keys.stride()[:3]
        p.cv_stride_batch, p.cv_stride_token, p.cv_stride_head = values.stride()[:3]
        p.batch, (p.cache_rows, p.cache_len, p.num_kv_heads, p.head_dim) = batch, keys.shape
        p.batch_indices = 1 if indices else None
        return bool(lib.distinct(ctypes.byref(p)))

    return call


def _addresses(t, base):
    """The element offset of every entry of ``t`` from ``base``."""
    off = torch.tensor((t.data_ptr() - base.data_ptr()) // 2)
    for n, s in zip(t.shape, t.stride()):
        off = off[..., None] + torch.arange(n) * s
    return off.flatten()


def _really(keys, values, base, batch, indices):
    n = keys.shape[0] if indices else min(batch, keys.shape[0])
    a = torch.cat((_addresses(keys[:n], base), _addresses(values[:n], base)))
    return a.unique().numel() == a.numel()


def _bf16(*shape):
    return torch.zeros(shape, dtype=torch.bfloat16)


def _ordinary():
    R, L, H = 3, 5, 2
    two = _bf16(2, R, L, H, D)
    yield "one buffer", two[0], two[1], two
    yield "one row", two[0, :1], two[1, :1], two
    x = _bf16(R, L, 2, H, D)
    yield "keys and values by position", x[:, :, 0], x[:, :, 1], x
    x = _bf16(R, L, H, 2, D)
    yield "keys and values by head", x[:, :, :, 0], x[:, :, :, 1], x
    x = _bf16(R, L, H, 2 * D)
    yield "values behind keys", x[..., D:], x[..., :D], x
    x = _bf16(R, 2, H, L, D).transpose(2, 3)
    yield "heads first", x[:, 0], x[:, 1], x
    x = _bf16(L, R, 2, H, D).transpose(0, 1)
    yield "positions first", x[:, :, 0], x[:, :, 1], x
    x = _bf16(R, L, 4, 2, H, D)
    yield "a layer of several", x[:, :, 1, 0], x[:, :, 1, 1], x
    x = _bf16(2, R, L + 3, H + 1, D + 8)
    yield "inside a larger buffer", x[0, :, :L, :H, :D], x[1, :, 1:L + 1, 1:, 8:], x


@pytest.mark.parametrize("name,keys,values,base", list(_ordinary()), ids=lambda x: x.replace(" ", "_") if isinstance(x, str) else "")
def test_ordinary_layouts_are_distinct(rule, name, keys, values, base):
    for batch, indices in ((1, False), (3, False), (2, True)):
        assert _really(keys, values, base, batch, indices)
        assert rule(keys, values, batch, indices)


def _shared():
    R, L, H = 3, 5, 2
    a, b = _bf16(2, 1, L, H, D)
    yield "expanded over the batch", a.expand(R, L, H, D), b.expand(R, L, H, D), 3, False
    yield "expanded, by index", a.expand(R, L, H, D), b.expand(R, L, H, D), 1, True
    a, b = _bf16(2, R, L, 1, D)
    yield "expanded over the heads", a.expand(R, L, H, D), b.expand(R, L, H, D), 3, False
    a, b = _bf16(2, R + L, H, D)
    yield "windows", a.as_strided((R, L, H, D), (H * D, H * D, D, 1)), b.as_strided((R, L, H, D), (H * D, H * D, D, 1)), 2, False
    a = _bf16(R, L, H, D)
    yield "one tensor", a, a, 1, False
    a = _bf16(R, L + 2, H, D)
    yield "values two positions on", a[:, :L], a[:, 2:], 1, False


@pytest.mark.parametrize("name,keys,values,batch,indices", list(_shared()),
                         ids=lambda x: x.replace(" ", "_") if isinstance(x, str) else "")
def test_shared_rows_are_found(rule, name, keys, values, batch, indices):
    assert not rule(keys, values, batch, indices)


def test_a_batch_of_one_reaches_one_row(rule):
    a, b = _bf16(2, 1, 5, 2, D)
    assert rule(a.expand(3, 5, 2, D), b.expand(3, 5, 2, D), 1, False)


def test_never_distinct_where_addresses_repeat(rule):
    """All stride combinations of a small grid, values at several offsets from keys."""
    base = torch.zeros(1 << 13, dtype=torch.bfloat16)
    shape = (2, 3, 2, D)
    strides = [0, 64, 128, 192, 256, 384]
    distinct = 0
    for sb, st, sh in itertools.product(strides, strides[1:], strides):
        keys = base.as_strided(shape, (sb, st, sh, 1))
        for off in (0, 64, 128, 384, 768, 2048):
            values = base.as_strided(shape, (sb, st, sh, 1), off)
            for batch in (1, 2):
                if rule(keys, values, batch, False):
                    distinct += 1
                    assert _really(keys, values, base, batch, False), (sb, st, sh, off, batch)
    assert distinct > 50
