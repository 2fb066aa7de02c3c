"""GPU parity of the KV-cache attention (mimir_amd.cache, inference path of
src/mimir/model/layers.py:134-167) against the oracle's restatement.

Tolerances: output <= 2e-2 max-abs (the bf16 operator bar; the oracle runs in
fp32 on the same bf16 values); the cache writes are exact copies and every other
cache position is left untouched.  Cases cover decode (S = 1, key range split
over workgroups and merged), chunked prefill into a non-empty cache (causal and
bidirectional), GQA, batch_indices, an unsplit launch, and the IndexError of a
write past the cache.
"""

import pytest
import torch

from mimir_amd.cache import Cache, attention_with_cache
from oracle import layer_oracle as LO

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def _run(device, B, S, hq, hkv, d, L, lens, causal, rows=None, cache_rows=None, seed=0, index_dtype=torch.int64):
    gen = torch.Generator().manual_seed(seed)
    cache_rows = cache_rows or B
    q = torch.randn(B, S, hq, d, generator=gen).to(BF16)
    k = torch.randn(B, S, hkv, d, generator=gen).to(BF16)
    v = torch.randn(B, S, hkv, d, generator=gen).to(BF16)
    ck = torch.randn(cache_rows, L, hkv, d, generator=gen).to(BF16)
    cv = torch.randn(cache_rows, L, hkv, d, generator=gen).to(BF16)
    lens_t = torch.tensor(lens, dtype=index_dtype)
    rows_t = None if rows is None else torch.tensor(rows, dtype=index_dtype)
    ck_ref, cv_ref = ck.clone(), cv.clone()
    ref = LO.attention_with_cache(q, k, v, ck_ref, cv_ref, lens_t, causal, rows_t)

    cache = Cache(ck.to(device), cv.to(device))
    out = attention_with_cache(q.to(device), k.to(device), v.to(device), cache, lens_t.to(device), causal,
                               None if rows_t is None else rows_t.to(device))
    torch.cuda.synchronize()
    err = (out.float().cpu() - ref.float()).abs().max().item()
    print(f"[cache] B={B} S={S} hq={hq} hkv={hkv} d={d} L={L} lens={lens} causal={causal} err={err:.3g}", flush=True)
    assert err <= 2e-2
    assert torch.equal(cache.keys.cpu(), ck_ref) and torch.equal(cache.values.cpu(), cv_ref)


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("index_dtype", [torch.int64, torch.int32])
def test_decode_split_keys(device, d, index_dtype):
    _run(device, B=5, S=1, hq=8, hkv=2, d=d, L=1500, lens=[0, 1, 777, 1499, 64], causal=True,
         rows=[3, 0, 6, 1, 4], cache_rows=7, index_dtype=index_dtype)


@pytest.mark.parametrize("S,causal", [(3, True), (4, True), (4, False), (5, True)])
def test_short_chunks_around_the_decode_kernel(device, S, causal):
    """S * G <= 32 query rows per kv head take the decode kernel (each wave its own key tiles,
    merged through LDS), 40 rows the row-tile kernel; causal masks per token."""
    _run(device, B=3, S=S, hq=16, hkv=2, d=128, L=900, lens=[0, 451, 880], causal=causal, seed=20 + S)


@pytest.mark.parametrize("B,S,hq,hkv,d,L,seed", [
    (70, 1, 8, 2, 64, 300, 1),      # one workgroup per pair; more batch rows than a wave has lanes
    (300, 2, 4, 1, 128, 70, 2),
    (2, 32, 2, 2, 128, 200, 3),     # 32 new rows over two tiles, 32 query rows
    (3, 1, 4, 4, 128, 9000, 4),     # equal shares: pairs over many shares
    (70, 1, 4, 1, 64, 3000, 5),     # shares over several pairs, batch rows past the first 64
    (5, 8, 4, 1, 128, 700, 6),      # 32 query rows merged over parts
    (6, 17, 2, 2, 64, 900, 7),      # 17 query rows, several pairs per share
    (40, 3, 10, 2, 128, 300, 8),    # 15 query rows, one workgroup per pair
    (33, 32, 3, 3, 64, 260, 9),
    (3, 1, 24, 24, 64, 1500, 10),   # a run of the line for each of 24 kv heads
    (2, 1, 300, 300, 64, 2100, 11), # more kv heads than there are CUs: one run for each
    (9, 1, 6, 3, 128, 2000, 12),    # 3 kv heads: their runs leave two workgroups out
    (20, 1, 2, 2, 64, 2500, 13),    # head_dim 64: one unit for each run, or none
    (3, 9, 6, 3, 128, 2200, 14),    # 18 query rows: parts merged a few loads at a time, many of them
    (1, 32, 1, 1, 64, 9000, 15),
    (130, 20, 4, 4, 64, 600, 16),   # 20 query rows and a workgroup per pair
])
def test_decode_work_split(device, B, S, hq, hkv, d, L, seed):
    """One workgroup per pair, and the line of key tiles dealt to equal shares: ragged lengths
    (0 keys to the whole cache), shuffled cache rows, new rows across a tile edge."""
    gen = torch.Generator().manual_seed(seed)
    lens = torch.randint(0, L - S + 1, (B,), generator=gen).tolist()
    lens[0], lens[-1] = 0, L - S
    _run(device, B=B, S=S, hq=hq, hkv=hkv, d=d, L=L, lens=lens, causal=True,
         rows=torch.randperm(B, generator=gen).tolist(), seed=seed)


@pytest.mark.parametrize("hq,hkv,d", [(16, 4, 128), (8, 8, 64)])
def test_decode_does_not_depend_on_the_split(device, hq, hkv, d):
    """One row alone (a tile or two per wave) and the same row 64 times over (whole pairs per
    workgroup, or shares of many tiles per wave) round P alike, so they differ by fp32 sums
    alone: 1e-6, which moves about one bf16 result in a thousand by 2^-8 of itself (1e-4 in
    all).  Under maxima that depend on the split, P rounds elsewhere: 1e-3 and more."""
    gen = torch.Generator(device=device).manual_seed(3)
    mk = lambda *s: torch.randn(*s, generator=gen, device=device).to(BF16)
    for L, n in ((1024, 700), (4096, 2500)):
        q, k, v = mk(1, 1, hq, d), mk(1, 1, hkv, d), mk(1, 1, hkv, d)
        keys, values = mk(1, L, hkv, d), mk(1, L, hkv, d)
        one = attention_with_cache(q, k, v, Cache(keys.clone(), values.clone()), torch.tensor([n], device=device), True)
        many = [t.repeat(64, 1, 1, 1) for t in (q, k, v, keys, values)]
        out = attention_with_cache(*many[:3], Cache(*many[3:]), torch.tensor([n] * 64, device=device), True)
        err = (out.float() - one.float()).norm() / (one.float().norm() * 8)
        print(f"[split] hq={hq} d={d} L={L} n={n} err={err:.3g}", flush=True)
        assert err <= 4e-4


def test_decode_reference_of_a_low_tile(device):
    """Key tiles whose scores lie far below (and far above) those of the tiles before them."""
    B, L, d = 2, 512, 128
    gen = torch.Generator().manual_seed(4)
    q = torch.randn(B, 1, 2, d, generator=gen)
    scale = torch.tensor([40.0, 1e-3, 40.0, 0.1] * 4).repeat_interleave(L // 16)[None, :, None, None]
    keys = (q.mean(2, keepdim=True) * scale + torch.randn(B, L, 2, d, generator=gen) * 1e-2).to(BF16)
    values = torch.randn(B, L, 2, d, generator=gen).to(BF16)
    q, k, v = q.to(BF16), keys[:, :1].clone(), values[:, :1].clone()
    lens = torch.tensor([L - 1, 100])
    ref = LO.attention_with_cache(q, k, v, keys.clone(), values.clone(), lens, True)
    out = attention_with_cache(q.to(device), k.to(device), v.to(device), Cache(keys.to(device), values.to(device)),
                               lens.to(device), True)
    torch.cuda.synchronize()
    assert (out.float().cpu() - ref.float()).abs().max().item() <= 2e-2


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("scale", [1e-38, 1e-30])
def test_decode_with_a_tiny_scale(device, d, scale):
    """Every score is 0: the mean of the values, also for a token that a later tile holds no key for."""
    B, S, L, n = 1, 2, 4096, 63  # token 0 ends with tile 1, token 1 is alone in tile 2
    gen = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(B, S, 2, d, generator=gen).to(BF16).to(device) for _ in range(3))
    cache = Cache(*(torch.randn(B, L, 2, d, generator=gen).to(BF16).to(device) for _ in range(2)))
    out = attention_with_cache(q, k, v, cache, torch.tensor([n], device=device), True, softmax_scale=scale)
    ref = torch.stack([cache.values[0, :n + 1 + i].double().mean(0) for i in range(S)])
    # every probability is 1: what is left is the rounding of the output
    assert (out[0].double() - ref).abs().max().item() <= 2.0**-8 * ref.abs().max().item()


def test_decode_rows_sharing_a_cache_row(device):
    """Batch rows on one cache row attend each other's new keys, as after appending all of them
    first: consecutive tokens of a sequence fed as separate batch rows, and one far behind."""
    _run(device, B=5, S=1, hq=8, hkv=2, d=128, L=700, lens=[63, 64, 65, 10, 300], causal=False,
         rows=[1, 1, 1, 1, 0], cache_rows=2, seed=31)
    _run(device, B=3, S=2, hq=4, hkv=2, d=64, L=200, lens=[30, 32, 150], causal=False, rows=[0, 0, 0], cache_rows=1,
         seed=32)  # one workgroup per pair


@pytest.mark.parametrize("d,S,lens", [
    (128, 1, [10, 63, 64, 40]),       # one workgroup per pair
    (128, 2, [700, 2, 704, 702]),     # equal shares
    (64, 8, [100, 92, 1990, 84]),
    (128, 40, [0, 120, 40, 80]),      # prefill, one key split
    (64, 100, [1500, 1300, 1400, 0]), # and several
])
@pytest.mark.parametrize("form", ["expanded", "windows", "one tensor"])
def test_cache_rows_that_share_memory(device, d, S, lens, form):
    """Every batch row sees all new rows that lie among its keys, as after appending all of them
    first: batch rows on the same positions, overlapping windows, one tensor for keys and values."""
    gen = torch.Generator().manual_seed(d + S)
    B, L, hq, hkv = len(lens), max(lens) + S + 5, 4, 2
    q = torch.randn(B, S, hq, d, generator=gen).to(BF16)
    k, v = (torch.randn(B, S, hkv, d, generator=gen).to(BF16) for _ in range(2))
    step = {"expanded": 0, "windows": 3, "one tensor": 2 * L}[form]  # positions from one row to the next
    flat = torch.randn(2, L + (B - 1) * step, hkv, d, generator=gen).to(BF16)

    def view(x):  # [B, L, hkv, d], batch row b at position b * step
        return x.as_strided((B, L, hkv, d), (step * hkv * d, hkv * d, d, 1), x.storage_offset())

    if form == "windows":  # new rows at positions of their own
        lens = [n - 3 * b if n >= 3 * b else n for b, n in enumerate(lens)]
        spans = sorted((n + b * step, n + b * step + S) for b, n in enumerate(lens))
        assert all(e <= s for (_, e), (s, _) in zip(spans, spans[1:])), spans
    kf, vf = (flat[0].clone(), flat[0 if form == "one tensor" else 1].clone())
    if form == "one tensor":
        vf = kf
    for b, n in enumerate(lens):
        kf[b * step + n:b * step + n + S] = k[b]
        vf[b * step + n:b * step + n + S] = v[b]
    dev = flat.to(device)
    cache = Cache(view(dev[0]), view(dev[0 if form == "one tensor" else 1]))
    out = attention_with_cache(q.to(device), k.to(device), v.to(device), cache, torch.tensor(lens, device=device), True)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        for i in range(S):
            ks, vs = (x[b * step:b * step + n + i + 1].float().repeat_interleave(hq // hkv, 1) for x in (kf, vf))
            p = torch.softmax(torch.einsum("hd,khd->hk", q[b, i].float(), ks) / d ** 0.5, dim=1)
            assert (out[b, i].float().cpu() - torch.einsum("hk,khd->hd", p, vs)).abs().max().item() <= 2e-2, (b, i)
    assert torch.equal(dev[0].cpu(), kf) and torch.equal(dev[0 if form == "one tensor" else 1].cpu(), vf)


@pytest.mark.parametrize("B,S,hq,hkv,d,L,rows", [
    (65, 1, 2, 1, 64, 3000, None),        # shares: one batch row past the first 64
    (130, 2, 4, 2, 128, 1300, None),      # three chunks of batch rows
    (512, 1, 2, 1, 64, 1100, "distinct"), # pairs: in a cache this short
    (512, 1, 2, 1, 64, 2100, "distinct"), # as many as a share looks through
    (513, 1, 2, 1, 64, 1100, None),       # a workgroup per pair from here on
    (100, 1, 4, 2, 128, 300, "distinct"), # pairs, appended first
    (200, 1, 4, 1, 64, 1500, "shared"),   # pairs: 200 batch rows on 90 cache rows
    (200, 1, 4, 1, 64, 3000, "shared"),   # shares: batch rows of one cache row in several chunks
    (130, 2, 4, 2, 128, 2600, "shared"),
    (70, 2, 2, 2, 128, 200, "shared"),
])
def test_decode_of_large_batches(device, B, S, hq, hkv, d, L, rows):
    """More batch rows than a wave has lanes: ragged lengths among them 0 and the whole cache,
    chosen cache rows, batch rows that share one (each at positions of its own)."""
    gen = torch.Generator().manual_seed(B)
    lens = torch.randint(0, L - S + 1, (B,), generator=gen).tolist()
    lens[0], lens[-1] = 0, L - S
    if rows is None:
        _run(device, B=B, S=S, hq=hq, hkv=hkv, d=d, L=L, lens=lens, causal=True, seed=B)
    elif rows == "distinct":
        _run(device, B=B, S=S, hq=hq, hkv=hkv, d=d, L=L, lens=lens, causal=True, seed=B, cache_rows=B + 3,
             rows=torch.randperm(B + 3, generator=gen)[:B].tolist())
    else:
        n = 90 if B > 90 else 40
        lens = (torch.randperm(L // S - 1, generator=gen)[:B] * S).tolist()
        _run(device, B=B, S=S, hq=hq, hkv=hkv, d=d, L=L, lens=lens, causal=False, seed=B, cache_rows=n,
             rows=[b % n for b in range(B)])


@pytest.mark.parametrize("B,L", [(3, 200), (3, 2000), (100, 2000), (600, 100)])
def test_decode_batch_rows_without_keys(device, B, L):
    """Batch rows outside the cache get zeros, write nothing and take no part of the work."""
    gen = torch.Generator().manual_seed(B)
    mk = lambda *s: torch.randn(*s, generator=gen).to(BF16)
    q, k, v, keys, values = mk(B, 1, 4, 64), mk(B, 1, 2, 64), mk(B, 1, 2, 64), mk(B, L, 2, 64), mk(B, L, 2, 64)
    rows = torch.randperm(B, generator=gen)
    lens = torch.randint(0, L, (B,), generator=gen)
    gone = torch.arange(B) % 3 == 1
    ck, cv = keys.clone(), values.clone()
    ref = torch.zeros_like(q)
    ref[~gone] = LO.attention_with_cache(q[~gone], k[~gone], v[~gone], ck, cv, lens[~gone], True, rows[~gone])
    rows[gone] = torch.where(torch.arange(int(gone.sum())) % 2 == 0, -1, B)
    cache = Cache(keys.to(device), values.to(device))
    out = attention_with_cache(q.to(device), k.to(device), v.to(device), cache, lens.to(device), True, rows.to(device))
    torch.cuda.synchronize()
    assert torch.count_nonzero(out[gone]) == 0
    assert (out.float().cpu() - ref.float()).abs().max().item() <= 2e-2
    assert torch.equal(cache.keys.cpu(), ck) and torch.equal(cache.values.cpu(), cv)


def test_decode_uneven_rows(device):
    """Rows whose key ranges split into different numbers of parts (1 key to the whole cache)."""
    _run(device, B=8, S=1, hq=16, hkv=4, d=128, L=4096, lens=[0, 63, 64, 65, 1000, 4095, 2048, 129],
         causal=True, seed=5)


@pytest.mark.parametrize("causal", [True, False])
def test_chunked_prefill(device, causal):
    _run(device, B=3, S=100, hq=8, hkv=2, d=128, L=700, lens=[0, 37, 600], causal=causal, seed=1)


def test_prefill_mha_d64(device):
    _run(device, B=2, S=130, hq=4, hkv=4, d=64, L=400, lens=[5, 200], causal=True, seed=2)


@pytest.mark.parametrize("S,hq,hkv,d,lens", [
    (257, 6, 2, 128, [0, 64, 100, 443]),   # 3 heads a group: tokens across row tiles; chunks on and off a tile edge
    (600, 4, 4, 64, [0, 1, 63, 100]),
    (512, 16, 16, 64, [188, 0]),
])
def test_prefill_reads_the_new_rows_in_place(device, S, hq, hkv, d, lens):
    """Enough row tiles that the key range is not split: no append launch, the keys of the chunk
    come from k / v and each workgroup stores its own tokens' rows."""
    B, L = 24, 700
    lens = (lens * B)[:B]
    _run(device, B=B, S=S, hq=hq, hkv=hkv, d=d, L=L, lens=lens, causal=True, seed=S)
    _run(device, B=B, S=S, hq=hq, hkv=hkv, d=d, L=L, lens=lens, causal=False, seed=S + 1)


@pytest.mark.parametrize("B,S,hq,hkv,d,lens", [
    (24, 700, 4, 4, 64, [0, 87]),         # 576 row tiles: more than two to a CU, about equal lengths
    (24, 700, 4, 4, 64, [0, 88]),         # lengths too far apart for the order by rank
    (33, 520, 6, 6, 64, [11, 0, 65]),     # 990: an odd run of CUs cut short
    (13, 300, 32, 8, 128, [100]),         # 1040, grouped heads: 1200 rows in ten row tiles
    (70, 200, 2, 2, 64, [50]),            # more batch rows than lanes
])
def test_prefill_order_of_the_row_tiles(device, B, S, hq, hkv, d, lens):
    """Unsplit chunks on rows of about equal length are dealt by rank, others as they come."""
    lens = (lens * B)[:B]
    for causal, rows in ((True, None), (True, list(range(B))[::-1]), (False, None)):
        _run(device, B=B, S=S, hq=hq, hkv=hkv, d=d, L=max(lens) + S, lens=lens, causal=causal, rows=rows, seed=B)


@pytest.mark.parametrize("S,hq,hkv,d,lens", [
    (33, 4, 4, 128, [0, 31, 1000]),      # one row tile per head, the chunk inside the last key split
    (129, 8, 2, 128, [63, 64, 1367]),    # 516 rows: five row tiles, the last of four rows
    (200, 2, 2, 64, [1296, 5, 127]),     # up to the end of the cache
])
def test_prefill_reads_the_new_rows_in_place_split_keys(device, S, hq, hkv, d, lens):
    """The same with the key range split: the chunk's keys lie in one or several splits."""
    for causal in (True, False):
        _run(device, B=3, S=S, hq=hq, hkv=hkv, d=d, L=1496, lens=lens, causal=causal, seed=S)


@pytest.mark.parametrize("S", [1024, 1025])
def test_prefill_around_the_longest_chunk_appended_in_place(device, S):
    """The longest chunk whose rows the attention kernel appends, and the first that a launch of
    its own does; a q head per kv head, so that a workgroup appends 128 tokens."""
    for causal in (True, False):
        _run(device, B=2, S=S, hq=2, hkv=2, d=128, L=1100, lens=[70, 0], causal=causal, seed=S)


def _prefill(device, B, S, hq, hkv, d, L, lens, rows, cache_rows, causal, strided, seed):
    """A chunk against the oracle, with q / k / v contiguous or slices of one projection (``strided``
    names them), into cache rows ``rows``; batch rows outside the cache (-1, cache_rows) get zeros."""
    gen = torch.Generator().manual_seed(seed)
    mk = lambda *s: torch.randn(*s, generator=gen).to(BF16)
    heads = dict(q=hq, k=hkv, v=hkv)
    fused = mk(B, S, hq + 2 * hkv, d)
    parts = dict(zip("qkv", fused.split((hq, hkv, hkv), dim=2)))
    ck, cv = mk(cache_rows, L, hkv, d), mk(cache_rows, L, hkv, d)
    cache = Cache(ck.to(device), cv.to(device))
    dev = dict(zip("qkv", fused.to(device).split((hq, hkv, hkv), dim=2)))
    args = [dev[n] if n in strided else dev[n].contiguous() for n in "qkv"]
    assert all((a.stride(1) != heads[n] * d) == (n in strided) for n, a in zip("qkv", args))
    rows_t = None if rows is None else torch.tensor(rows)
    out = attention_with_cache(*args, cache, torch.tensor(lens, device=device), causal,
                               None if rows is None else rows_t.to(device))
    torch.cuda.synchronize()
    inside = torch.ones(B, dtype=torch.bool) if rows is None else (rows_t >= 0) & (rows_t < cache_rows)
    ref = torch.zeros(B, S, hq, d, dtype=BF16)
    ref[inside] = LO.attention_with_cache(*(parts[n][inside] for n in "qkv"), ck, cv, torch.tensor(lens)[inside], causal,
                                          None if rows is None else rows_t[inside])
    assert (out.float().cpu() - ref.float()).abs().max().item() <= 2e-2
    assert torch.count_nonzero(out[~inside]) == 0
    assert torch.equal(cache.keys.cpu(), ck) and torch.equal(cache.values.cpu(), cv)


# Sizes with the key range split (few row tiles) and not (24 batch rows).
@pytest.mark.parametrize("B,S,hq,hkv,d,L", [(4, 50, 8, 2, 128, 900), (4, 130, 2, 2, 64, 900), (24, 300, 8, 4, 128, 420),
                                            (24, 600, 4, 4, 64, 700)])
@pytest.mark.parametrize("form", ["shuffled", "outside", "shared"])
def test_prefill_into_chosen_cache_rows(device, B, S, hq, hkv, d, L, form):
    """batch_indices: the new rows are appended by a launch of their own.  Shuffled rows of a larger
    cache; one of them outside it; several batch rows on a cache row, each at positions of its own,
    which then see each other's new rows."""
    gen = torch.Generator().manual_seed(B + S)
    lens = torch.randint(0, L - S + 1, (B,), generator=gen).tolist()
    rows = torch.randperm(B + 3, generator=gen)[:B].tolist()
    n, causal = B + 3, True
    if form == "outside":
        rows[1], rows[-1] = -1, n
    elif form == "shared":
        per = L // S  # batch rows on one cache row
        n, causal = -(-B // per), False
        rows, lens = [b // per for b in range(B)], [b % per * S for b in range(B)]
    _prefill(device, B, S, hq, hkv, d, L, lens, rows, n, causal, "", seed=S)


@pytest.mark.parametrize("B,S,hq,hkv,d,L", [(3, 60, 8, 2, 128, 900), (24, 300, 8, 4, 128, 420), (4, 200, 4, 4, 64, 500)])
@pytest.mark.parametrize("strided", ["v", "k", "kv", "qkv"])
def test_prefill_from_the_projection(device, B, S, hq, hkv, d, L, strided):
    """k or v (or both) as slices of the fused projection, whose token stride is not the cache's:
    appended by a launch of their own also where only one of the strides differs."""
    gen = torch.Generator().manual_seed(S)
    lens = torch.randint(0, L - S + 1, (B,), generator=gen).tolist()
    for causal in (True, False):
        _prefill(device, B, S, hq, hkv, d, L, lens, None, B, causal, strided, seed=S)


def test_prefill_with_the_strides_of_a_wider_cache(device):
    """New rows whose token stride is the cache's although neither is dense: slices of wider buffers."""
    B, S, hq, hkv, d, L = 3, 70, 4, 2, 64, 300
    gen = torch.Generator().manual_seed(8)
    mk = lambda *s: torch.randn(*s, generator=gen).to(BF16)
    q, kw, vw, ckw, cvw = mk(B, S, hq, d), mk(B, S, 5, d), mk(B, S, 5, d), mk(B, L, 5, d), mk(B, L, 5, d)
    ck, cv = ckw[:, :, 1:3], cvw[:, :, 2:4]
    dev = [t.to(device) for t in (q, kw, vw, ckw, cvw)]
    lens = torch.tensor([0, 100, 230])
    out = attention_with_cache(dev[0], dev[1][:, :, :2], dev[2][:, :, 3:], Cache(dev[3][:, :, 1:3], dev[4][:, :, 2:4]),
                               lens.to(device), True)
    torch.cuda.synchronize()
    ref = LO.attention_with_cache(q, kw[:, :, :2], vw[:, :, 3:], ck, cv, lens, True)
    assert (out.float().cpu() - ref.float()).abs().max().item() <= 2e-2
    assert torch.equal(dev[3].cpu(), ckw) and torch.equal(dev[4].cpu(), cvw)


@pytest.mark.parametrize("S", [1, 40])
def test_lengths_outside_the_cache(device, S):
    """Without validation, new rows at positions outside the cache are dropped, and the row attends
    the min(max(length, 0) + S, cache_len) first keys."""
    gen = torch.Generator().manual_seed(S)
    L, d, lens = 100, 64, [-1, -30, 90, 100, 150]
    B = len(lens)
    q, k, v = (torch.randn(B, S, 2, d, generator=gen).to(BF16) for _ in range(3))
    ck, cv = (torch.randn(B, L, 2, d, generator=gen).to(BF16) for _ in range(2))
    cache = Cache(ck.to(device), cv.to(device))
    out = attention_with_cache(q.to(device), k.to(device), v.to(device), cache, torch.tensor(lens, device=device), True)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        for i in range(S):
            if 0 <= n + i < L:
                ck[b, n + i], cv[b, n + i] = k[b, i], v[b, i]
        start = min(max(n, 0), L)
        keys = min(start + S, L)
        for i in range(S):
            end = min(start + i + 1, keys)
            p = torch.softmax(torch.einsum("hd,khd->hk", q[b, i].float(), ck[b, :end].float()) / d ** 0.5, dim=1)
            ref = torch.einsum("hk,khd->hd", p, cv[b, :end].float())
            assert (out[b, i].float().cpu() - ref).abs().max().item() <= 2e-2, (b, i)
    assert torch.equal(cache.keys.cpu(), ck) and torch.equal(cache.values.cpu(), cv)


def test_unsplit_launch(device):
    """Enough row tiles that the key range is not split (one workgroup per row tile)."""
    _run(device, B=4, S=1024, hq=16, hkv=4, d=128, L=1100, lens=[0, 3, 40, 76], causal=True, seed=3)


@pytest.mark.parametrize("validate", [True, False])
def test_validated_lengths(device, validate):
    """With validation the split is sized from the actual lengths; a write past the cache raises."""
    from mimir_amd import set_validate_metadata
    set_validate_metadata(validate)
    try:
        _run(device, B=3, S=1, hq=4, hkv=1, d=128, L=3000, lens=[10, 2000, 700], causal=True, seed=4)
        if validate:
            q = torch.zeros(1, 4, 2, 64, dtype=BF16, device=device)
            k = torch.zeros(1, 4, 2, 64, dtype=BF16, device=device)
            cache = Cache.create(1, 10, 2, 64, dtype=BF16, device=device)
            with pytest.raises(IndexError):
                attention_with_cache(q, k, k, cache, torch.tensor([7], device=device), True)
    finally:
        set_validate_metadata(False)


def test_rows_outside_the_cache_are_skipped(device):
    """Without validation a batch index outside the cache writes nothing and yields zeros."""
    gen = torch.Generator().manual_seed(9)
    q = torch.randn(2, 1, 4, 128, generator=gen).to(BF16).to(device)
    k = torch.randn(2, 1, 2, 128, generator=gen).to(BF16).to(device)
    cache = Cache(torch.randn(2, 64, 2, 128, generator=gen).to(BF16).to(device),
                  torch.randn(2, 64, 2, 128, generator=gen).to(BF16).to(device))
    before = cache.keys.clone()
    out = attention_with_cache(q, k, k, cache, torch.tensor([3, 5], device=device), True,
                               torch.tensor([1, 7], device=device))
    torch.cuda.synchronize()
    assert torch.count_nonzero(out[1]) == 0 and torch.isfinite(out).all()
    assert torch.equal(cache.keys[0], before[0])
    # batch row 0 -> cache row 1, position cache_lengths[0] = 3
    assert torch.equal(cache.keys[1, 3], k[0, 0]) and torch.equal(cache.keys[1, :3], before[1, :3])
    assert torch.equal(cache.keys[1, 4:], before[1, 4:])


def test_repeated_calls_and_graph_replay(device):
    """Back-to-back calls and replays of a captured decode step (no host synchronisation, no
    memset) match the eager result."""
    gen = torch.Generator().manual_seed(11)
    B, hq, hkv, d, L = 4, 8, 2, 128, 2048
    q = torch.randn(B, 1, hq, d, generator=gen).to(BF16).to(device)
    k = torch.randn(B, 1, hkv, d, generator=gen).to(BF16).to(device)
    v = torch.randn(B, 1, hkv, d, generator=gen).to(BF16).to(device)
    cache = Cache(torch.randn(B, L, hkv, d, generator=gen).to(BF16).to(device),
                  torch.randn(B, L, hkv, d, generator=gen).to(BF16).to(device))
    lens = torch.tensor([5, 2000, 700, 1300], device=device)
    first = attention_with_cache(q, k, v, cache, lens, True)
    second = attention_with_cache(q, k, v, cache, lens, True)  # the same append again: same output
    torch.cuda.synchronize()
    assert torch.equal(first, second)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        attention_with_cache(q, k, v, cache, lens, True)  # warm-up on the capture stream
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = attention_with_cache(q, k, v, cache, lens, True)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, first)
        eager = attention_with_cache(q, k, v, cache, lens, True)  # eager work between replays
        torch.cuda.synchronize()
        assert torch.equal(eager, first)
