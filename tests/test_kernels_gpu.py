"""Numerics of every hand-written gfx950 kernel against the plain-PyTorch fp32
reference of the same op (omnia_amd.ops.reference).  GPU only."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from omnia_amd import ops
from omnia_amd.ops import reference as ref

DEV = "cuda"


def _close(a, b, atol, rtol=0.0):
    a, b = a.float(), b.float()
    err = (a - b).abs().max().item()
    tol = atol + rtol * b.abs().max().item()
    assert err <= tol, f"max err {err} > {tol}"


def test_extension_is_native():
    k = ops.kernels()
    assert k.arch == "gfx950"
    assert k.__file__.endswith("_omnia_kernels.so")


@pytest.mark.parametrize("rows,d", [(1, 4096), (37, 4096), (256, 8192), (5, 2048)])
def test_rmsnorm(rows, d):
    torch.manual_seed(0)
    x = torch.randn(rows, d, device=DEV, dtype=torch.bfloat16)
    w = torch.randn(d, device=DEV, dtype=torch.bfloat16)
    y = ops.rmsnorm(x, w, 1e-5)
    _close(y, ref.rmsnorm(x, w, 1e-5), 0.05, 0.01)


def test_fused_add_rmsnorm():
    torch.manual_seed(1)
    x = torch.randn(33, 4096, device=DEV, dtype=torch.bfloat16)
    r = torch.randn(33, 4096, device=DEV, dtype=torch.bfloat16)
    w = torch.randn(4096, device=DEV, dtype=torch.bfloat16)
    ey, er = ref.fused_add_rmsnorm(x, r, w, 1e-5)
    ops.fused_add_rmsnorm(x, r, w, 1e-5)
    _close(r, er, 0.0)
    _close(x, ey, 0.05, 0.01)


def test_silu_mul():
    x = torch.randn(19, 2 * 14336, device=DEV, dtype=torch.bfloat16)
    _close(ops.silu_mul(x), ref.silu_mul(x), 0.02, 0.01)


def test_embedding():
    w = torch.randn(1000, 4096, device=DEV, dtype=torch.bfloat16)
    ids = torch.randint(0, 1000, (57,), device=DEV, dtype=torch.int32)
    _close(ops.embedding(ids, w), w[ids.long()], 0.0)
    # vocab-parallel shard: ids outside [500, 1000) give zero rows
    y = ops.embedding(ids, w[500:].contiguous(), vocab_start=500)
    exp = torch.where((ids >= 500)[:, None], w[ids.long()], torch.zeros_like(w[ids.long()]))
    _close(y, exp, 0.0)


def _make_cache(nb, hkv, bs, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kc = torch.randn(nb, hkv, bs, 128, device=DEV, dtype=torch.bfloat16, generator=g)
    vc = torch.randn(nb, hkv, bs, 128, device=DEV, dtype=torch.bfloat16, generator=g)
    return kc, vc


@pytest.mark.parametrize("bs", [16, 32])
def test_rope_kv(bs):
    T, hq, hkv = 23, 32, 8
    qkv = torch.randn(T, (hq + 2 * hkv) * 128, device=DEV, dtype=torch.bfloat16)
    q = qkv[:, : hq * 128]
    k = qkv[:, hq * 128: (hq + hkv) * 128]
    v = qkv[:, (hq + hkv) * 128:]
    pos = torch.randint(0, 4000, (T,), device=DEV, dtype=torch.int32)
    cs = ref.rope_cos_sin(8192, 128, 500000.0, device=DEV)
    kc, vc = _make_cache(16, hkv, bs)
    kc0, vc0 = kc.clone(), vc.clone()
    slots = torch.randperm(16 * bs, device=DEV)[:T].long()
    eq = ref.apply_rope(q.reshape(T, hq, 128).clone(), pos, cs)
    ek = ref.apply_rope(k.reshape(T, hkv, 128).clone(), pos, cs)
    ev = v.reshape(T, hkv, 128).clone()
    ref.write_kv(kc0, vc0, ek, ev, slots)
    ops.rope_kv(q, k, v, pos, cs, kc, vc, slots, hq, hkv, bs)
    _close(q.reshape(T, hq, 128), eq, 0.02, 0.01)
    _close(kc, kc0, 0.02, 0.01)
    _close(vc, vc0, 0.0)


def _tables(lens, bs, nb_total):
    maxb = max((l + bs - 1) // bs for l in lens)
    perm = torch.randperm(nb_total)
    bt = torch.zeros(len(lens), maxb + 2, dtype=torch.int32)
    p = 0
    for i, l in enumerate(lens):
        nb = (l + bs - 1) // bs
        bt[i, :nb] = perm[p:p + nb].int()
        p += nb
    return bt.to(DEV)


@pytest.mark.parametrize("part", [512, 1024, 2048])
@pytest.mark.parametrize("hq,hkv", [(32, 8), (64, 8), (8, 8), (16, 8)])
@pytest.mark.parametrize("bs", [16, 32, 64])
def test_decode_attention(hq, hkv, bs, part):
    """Groups of 1, 2, 4 and 8 query heads a KV head, every page size, the partition lengths that
    the models choose; contexts of one and of several partitions."""
    torch.manual_seed(3)
    lens = [1, 17, 64, 513, 1500, 3000]
    B = len(lens)
    nb_total = sum((l + bs - 1) // bs for l in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=3)
    bt = _tables(lens, bs, nb_total)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = torch.randn(B, hq, 128, device=DEV, dtype=torch.bfloat16)
    scale = 1 / math.sqrt(128)
    out = ops.decode_attention(q, kc, vc, bt, sl, scale, part_size=part)
    qsl = torch.arange(B + 1, dtype=torch.int32)
    exp = ref.paged_attention(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), qsl, sl.cpu(), scale)
    _close(out.cpu(), exp, 0.02, 0.02)


@pytest.mark.parametrize("splits,split_min", [(2, 64), (4, 64), (8, 32), (64, 64)])
@pytest.mark.parametrize("hq,hkv", [(32, 8), (8, 1)])
def test_decode_attention_length_balanced_split(hq, hkv, splits, split_min):
    """Device-side split (splits > 0): every context cut into up to `splits`
    equal page-aligned partitions (>= split_min keys, <= part_size) and merged
    -- against the fp32 oracle and the fixed-partition kernel."""
    torch.manual_seed(5)
    bs = 32
    lens = [1, 31, 32, 33, 200, 513, 640, 1500, 3000]
    B = len(lens)
    nb_total = sum((l + bs - 1) // bs for l in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=5)
    bt = _tables(lens, bs, nb_total)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = torch.randn(B, hq, 128, device=DEV, dtype=torch.bfloat16)
    scale = 1 / math.sqrt(128)
    out = ops.decode_attention(q, kc, vc, bt, sl, scale, part_size=512, splits=splits,
                               split_min=split_min)
    qsl = torch.arange(B + 1, dtype=torch.int32)
    exp = ref.paged_attention(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), qsl, sl.cpu(), scale)
    _close(out.cpu(), exp, 0.02, 0.02)
    fixed = ops.decode_attention(q, kc, vc, bt, sl, scale, part_size=512)
    _close(out.float().cpu(), fixed.float().cpu(), 0.02, 0.02)


@pytest.mark.parametrize("bs", [16, 32])
@pytest.mark.parametrize("hq,hkv,hp,qt", [(32, 8, 1, 64), (32, 8, 2, 64), (32, 8, 4, 64),
                                          (64, 8, 4, 64), (8, 8, 0, 64), (32, 8, 1, 128),
                                          (8, 8, 1, 128), (32, 8, 0, 32), (64, 8, 0, 32),
                                          (16, 8, 0, 32), (8, 8, 0, 32), (8, 1, 0, 32)])
def test_prefill_attention(bs, hq, hkv, hp, qt):
    torch.manual_seed(4)
    # (new tokens, cached prefix) per sequence: ragged + page-boundary edges
    specs = [(1, 0), (64, 0), (100, 37), (257, 0), (5, 600), (130, 64)]
    lens = [q + c for q, c in specs]
    qlens = [q for q, _ in specs]
    nb_total = sum((l + bs - 1) // bs for l in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=4)
    bt = _tables(lens, bs, nb_total)
    T = sum(qlens)
    q = torch.randn(T, hq, 128, device=DEV, dtype=torch.bfloat16)
    qsl = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32, device=DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    scale = 1 / math.sqrt(128)
    out = ops.prefill_attention(q, kc, vc, bt, qsl, sl, scale, heads_per_wave=hp, q_tile=qt)
    exp = ref.paged_attention(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), qsl.cpu(), sl.cpu(), scale)
    _close(out.cpu(), exp, 0.03, 0.02)


def _attention64(q, kc, vc, bt, qlens, lens, scale):
    """Paged attention in float64."""
    out, r, bs, (hkv, hq) = [], 0, kc.shape[2], (kc.shape[1], q.shape[1])
    for i, (n, ctx) in enumerate(zip(qlens, lens)):
        pages = bt[i, : -(-ctx // bs)].long()
        k, v = (c[pages].transpose(1, 2).reshape(-1, hkv, 128)[:ctx].double()
                .repeat_interleave(hq // hkv, 1) for c in (kc, vc))
        s = (q[r:r + n].double().transpose(0, 1) @ k.permute(1, 2, 0)) * scale
        at = torch.arange(ctx, device=q.device)
        s.masked_fill_(at[None] > (ctx - n + torch.arange(n, device=q.device))[:, None], -math.inf)
        out.append((s.softmax(-1) @ v.transpose(0, 1)).transpose(0, 1))
        r += n
    return torch.cat(out)


@pytest.mark.parametrize("parts", [2, 3, 16])
@pytest.mark.parametrize("hq,hkv,bs", [(32, 8, 16), (16, 8, 32), (8, 8, 64)])
def test_prefill_attention_in_key_partitions(parts, hq, hkv, bs):
    """Partitions that no row of a tile, some rows (the causal edge inside the tile) and all rows
    reach; contexts of one 64-key tile and of fewer tiles than partitions; ragged query tiles."""
    torch.manual_seed(6)
    specs = [(1, 0), (1, 127), (33, 96), (77, 1100), (40, 216), (5, 600)]
    lens, qlens = [q + c for q, c in specs], [q for q, _ in specs]
    nb_total = sum((n + bs - 1) // bs for n in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=6)
    bt = _tables(lens, bs, nb_total)
    q = torch.randn(sum(qlens), hq, 128, device=DEV, dtype=torch.bfloat16)
    qsl = torch.tensor([0, *torch.tensor(qlens).cumsum(0)], dtype=torch.int32, device=DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    tiles = [torch.tensor(t, dtype=torch.int32, device=DEV) for t in ops.prefill_tiles(qlens, 32)]
    one, split = (torch.full_like(q, math.nan) for _ in range(2))
    for out, p in ((one, 1), (split, parts)):
        ops.kernels().prefill_attention(out, q, kc, vc, bt, qsl, sl, *tiles, 128 ** -0.5, 0, 32,
                                        None, None, p)
    exp = _attention64(q, kc, vc, bt, qlens, lens, 128 ** -0.5)
    errs = [(o.double() - exp).norm().item() / exp.norm().item() for o in (one, split)]
    # P is rounded to bf16 in both; the partials are fp32
    assert errs[1] <= 1.05 * errs[0] + 1e-4, errs
    _close(split.cpu(), exp.cpu(), 0.03, 0.02)


@pytest.mark.parametrize("hq,hkv,bs", [(32, 8, 16), (16, 8, 32), (8, 8, 64)])
@pytest.mark.parametrize("parts", [1, 2])
def test_prefill_attention_by_two_groups_of_waves(parts, hq, hkv, bs):
    """Tables of few pages are walked by one group of waves, those of more (here behind the same
    ones, not reached) by two: from one tile of keys to uneven numbers of them."""
    torch.manual_seed(8)
    specs = [(1, 0), (64, 0), (33, 32), (1, 128), (40, 153), (129, 0), (97, 160), (9, 290)]
    lens, qlens = [q + c for q, c in specs], [q for q, _ in specs]
    nb_total = sum((n + bs - 1) // bs for n in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=8)
    bt = _tables(lens, bs, nb_total)[:, : -(-max(lens) // bs)].contiguous()
    assert bt.shape[1] * bs < 360
    wide = torch.zeros(len(lens), 1024 // bs, dtype=torch.int32, device=DEV)
    wide[:, : bt.shape[1]] = bt
    q = torch.randn(sum(qlens), hq, 128, device=DEV, dtype=torch.bfloat16)
    qsl = torch.tensor([0, *torch.tensor(qlens).cumsum(0)], dtype=torch.int32, device=DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    tiles = [torch.tensor(t, dtype=torch.int32, device=DEV) for t in ops.prefill_tiles(qlens, 32)]
    one, two = (torch.full_like(q, math.nan) for _ in range(2))
    for out, table in ((one, bt), (two, wide)):
        ops.kernels().prefill_attention(out, q, kc, vc, table, qsl, sl, *tiles, 128 ** -0.5, 0, 32,
                                        None, None, parts)
    exp = _attention64(q, kc, vc, bt, qlens, lens, 128 ** -0.5)
    errs = [(o.double() - exp).norm().item() / exp.norm().item() for o in (one, two)]
    assert errs[1] <= 1.05 * errs[0] + 1e-4, errs
    _close(two.cpu(), exp.cpu(), 0.03, 0.02)


def test_prefill_attention_of_ranks_that_share_a_device():
    """Where two groups of waves would share a walk over the keys, such ranks keep to one: the bits
    of one group, whose blocks leave half of a CU's registers to the peers' all-reduce."""
    torch.manual_seed(9)
    kc, vc = _make_cache(40, 2, 32, seed=9)
    bt = _tables([500], 32, 40)
    q = torch.randn(200, 8, 128, device=DEV, dtype=torch.bfloat16)
    qsl, sl = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in ([0, 200], [500]))
    tiles = [torch.tensor(t, dtype=torch.int32, device=DEV) for t in ops.prefill_tiles([200], 32)]
    args = (q, kc, vc, bt, qsl, sl, 128 ** -0.5, *tiles)
    parts = ops.prefill_parts(tiles[0].numel(), 8, 2, bt.shape[1] * 32, True)
    one = torch.empty_like(q)
    ops.kernels().prefill_attention(one, *args[:6], *tiles, 128 ** -0.5, 0, 32, None, None, parts,
                                    True)
    assert not torch.equal(ops.prefill_attention(*args), one)
    assert torch.equal(ops.prefill_attention(*args, shared_device=True), one)


@pytest.mark.parametrize("news,past,two", [([100] * 8, 1000, False), ([512] * 4, 512, False),
                                           ([1000] * 2, 0, True), ([100] * 2, 1000, True)])
def test_prompt_attention_of_walks_alike_by_one_group(news, past, two):
    """Two blocks a CU are of two groups only where the walks over the keys differ, one a CU are
    whatever they walk."""
    torch.manual_seed(10)
    hkv, hq = (16, 32) if past == 1000 else (8, 32)
    lens = [n + past for n in news]
    nb_total = sum(-(-n // 32) for n in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, 32, seed=10)
    bt = _tables(lens, 32, nb_total)
    q = torch.randn(sum(news), hq, 128, device=DEV, dtype=torch.bfloat16)
    qsl = torch.tensor([0, *torch.tensor(news).cumsum(0)], dtype=torch.int32, device=DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    tiles = [torch.tensor(t, dtype=torch.int32, device=DEV) for t in ops.prefill_tiles(news, 32)]
    got = []
    for one_group in (False, True):
        got.append(torch.empty_like(q))
        ops.kernels().prefill_attention(got[-1], q, kc, vc, bt, qsl, sl, *tiles, 128 ** -0.5, 0, 32,
                                        None, None, 1, one_group)
    assert torch.equal(*got) != two


def test_prefill_partitions_only_with_few_blocks():
    assert ops.prefill_parts(3, 32, 8, 400) == 1 < ops.prefill_parts(3, 32, 8, 2000)
    assert ops.prefill_parts(65, 32, 8, 100000) == 1  # 520 blocks
    assert ops.prefill_parts(1, 32, 8, 100000) == 16
    with pytest.raises(RuntimeError):  # partials of other tiles do not exist
        q = torch.zeros(1, 8, 128, device=DEV, dtype=torch.bfloat16)
        kc, vc = _make_cache(1, 8, 16)
        i = torch.zeros(1, 1, dtype=torch.int32, device=DEV)
        ops.kernels().prefill_attention(q, q, kc, vc, i, i[0], i[0], i[0], i[0], 1.0, 0, 64, None,
                                        None, 2)


@pytest.mark.parametrize("parts", [2, 5, 63, 64, 65, 130])
def test_decode_attention_merge_of_many_partitions(parts):
    torch.manual_seed(7)
    lens, hq, hkv, bs = [64 * parts, 64 * parts - 63, 64], 8, 2, 16
    nb_total = sum((n + bs - 1) // bs for n in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=7)
    bt = _tables(lens, bs, nb_total)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = torch.randn(3, hq, 128, device=DEV, dtype=torch.bfloat16)
    out = ops.decode_attention(q, kc, vc, bt, sl, 128 ** -0.5, part_size=64)
    exp = _attention64(q, kc, vc, bt, [1, 1, 1], lens, 128 ** -0.5)
    # all sums are fp32: what is left is the result's rounding to bf16
    err = (out.double() - exp).abs()
    assert (err <= exp.abs() * 2.0 ** -8 + 1e-4).all(), err.max()


@pytest.mark.parametrize("hq,hkv,bs", [(4, 4, 16), (8, 4, 64), (32, 8, 16), (16, 2, 32)])
def test_decode_attention_around_whole_key_groups(hq, hkv, bs):
    """Waves with no, one and several 16-key groups, ragged last groups, scores whose maximum
    keeps growing along the keys (the running maximum moves) and falls."""
    torch.manual_seed(8)
    lens = [1, 15, 16, 17, 48, 63, 64, 65, 127, 129, 1000]
    nb_total = sum((n + bs - 1) // bs for n in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=8)
    bt = _tables(lens, bs, nb_total)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = torch.randn(len(lens), hq, 128, device=DEV, dtype=torch.bfloat16)
    q[:, ::2], kc[..., 0] = q[:, ::2].abs(), 0  # dimension 0 carries the slope
    q[..., 0] = torch.where(torch.arange(hq, device=DEV) % 2 == 0, 16.0, -16.0)
    for i, n in enumerate(lens):
        for p in range(-(-n // bs)):
            kc[bt[i, p].long(), :, :, 0] = (torch.arange(bs, device=DEV) + p * bs).bfloat16() / 8
    out = ops.decode_attention(q, kc, vc, bt, sl, 128 ** -0.5, part_size=1024)
    exp = _attention64(q, kc, vc, bt, [1] * len(lens), lens, 128 ** -0.5)
    # scores up to 250 carry an fp32 error of 250 * 2^-23 into the exponent; the rest is the
    # result's rounding to bf16
    err = (out.double() - exp).abs()
    assert (err <= exp.abs() * 2.0 ** -8 + 2e-4 * vc.abs().max()).all(), err.max()


@pytest.mark.parametrize("part", [128, 1024])
@pytest.mark.parametrize("n", [17, 33, 200, 1023])
def test_decode_attention_with_infinite_scores_and_values(n, part):
    """Keys whose scores are -inf weigh nothing, whichever groups of a wave or whole partitions
    they fill; an infinite value of the last key reaches its own dimension only, with its sign."""
    torch.manual_seed(9)
    hq, hkv, bs = 8, 2, 16
    kc, vc = _make_cache(-(-n // bs) + 1, hkv, bs, seed=9)
    bt = _tables([n], bs, -(-n // bs) + 1)
    sl = torch.tensor([n], dtype=torch.int32, device=DEV)
    q = torch.rand(1, hq, 128, device=DEV).bfloat16() + 1
    at = bt[0, :-2].long()
    kc[at[:-1]] = -3e38  # sums of 128 such products overflow fp32
    vc[at[-1], 0, (n - 1) % bs, 5] = math.inf
    vc[at[-1], 1, (n - 1) % bs, 7] = -math.inf
    out = ops.decode_attention(q, kc, vc, bt, sl, 128 ** -0.5, part_size=part).double()
    exp = _attention64(q, kc, vc, bt, [1], [n], 128 ** -0.5)
    assert torch.equal(out.isinf(), exp.isinf()) and exp.isinf().sum() == 8
    assert torch.equal(out[exp.isinf()], exp[exp.isinf()])
    rest = ~exp.isinf()
    # all sums are fp32: what is left is the result's rounding to bf16
    err = (out - exp).abs()[rest]
    assert (err <= exp[rest].abs() * 2.0 ** -8 + 1e-4).all(), err.max()


@pytest.mark.parametrize("shared,splits", [(64, 0), (640, 0), (640, 8)])
def test_decode_attention_on_shared_prefix_pages(shared, splits):
    """Sequences of one prompt prefix read the same pages, whole partitions of them or parts."""
    torch.manual_seed(10)
    lens, hq, hkv, bs = [shared + n for n in (1, 7, 32, 200, 513)], 8, 2, 32
    nb_total = sum(-(-n // bs) for n in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=10)
    bt = _tables(lens, bs, nb_total)
    bt[1:, :shared // bs] = bt[0, :shared // bs]
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = torch.randn(len(lens), hq, 128, device=DEV, dtype=torch.bfloat16)
    out = ops.decode_attention(q, kc, vc, bt, sl, 128 ** -0.5, part_size=512, splits=splits)
    exp = _attention64(q, kc, vc, bt, [1] * len(lens), lens, 128 ** -0.5)
    # all sums are fp32: what is left is the result's rounding to bf16
    err = (out.double() - exp).abs()
    assert (err <= exp.abs() * 2.0 ** -8 + 1e-4).all(), err.max()


@pytest.mark.parametrize("hq,bs,part,splits", [(8, 32, 1024, 0), (16, 16, 512, 0), (8, 64, 512, 3)])
@pytest.mark.parametrize("lens", [[700], [511, 512, 513], [640, 191, 705, 1030, 64] * 4])
def test_decode_attention_past_and_through_the_caches(lens, hq, bs, part, splits):
    """Long and short sequences and partitions, alone and beside others, every third sharing a
    prefix with the next: both walks give the same sums."""
    torch.manual_seed(13)
    hkv, B = 2, len(lens)
    nb_total = sum(-(-n // bs) for n in lens) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=13)
    bt = _tables(lens, bs, nb_total)
    for i in range(0, B - 1, 3):
        k = min(lens[i], lens[i + 1], 256) // bs
        bt[i + 1, :k] = bt[i, :k]
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = torch.randn(B, hq, 128, device=DEV, dtype=torch.bfloat16)
    out = ops.decode_attention(q, kc, vc, bt, sl, 128 ** -0.5, part_size=part, splits=splits)
    exp = _attention64(q, kc, vc, bt, [1] * B, lens, 128 ** -0.5)
    # all sums are fp32: what is left is the result's rounding to bf16
    err = (out.double() - exp).abs()
    assert (err <= exp.abs() * 2.0 ** -8 + 1e-4).all(), err.max()


@pytest.mark.parametrize("B,hkv,hq", [(64, 4, 4), (64, 4, 32), (65, 4, 16), (128, 2, 8), (300, 1, 2)])
@pytest.mark.parametrize("short", [0, 0.25, 0.5])
def test_decode_attention_of_batches_past_the_caches(B, hkv, hq, short):
    """Blocks enough without partitions: where two thirds of the sequences are long, long ones that
    share no page go past the caches, looked for by a wave up to 64 rows and by the block beyond;
    empty rows are none."""
    torch.manual_seed(15)
    bs, g = 32, torch.Generator().manual_seed(B)
    lens = torch.randint(512, 900, (B,), generator=g)
    lens[torch.rand(B, generator=g) < short] = 70
    lens[3::17] = 0
    n = [int(x) for x in lens]
    nb_total = sum(-(-x // bs) for x in n) + 8
    kc, vc = _make_cache(nb_total, hkv, bs, seed=15)
    bt = _tables([max(x, 1) for x in n], bs, nb_total + B)
    bt %= nb_total
    for i in range(0, B - 40, 9):  # 40 rows apart
        k = min(n[i], n[i + 40], 256) // bs
        bt[i + 40, :k] = bt[i, :k]
    sl = lens.int().to(DEV)
    q = torch.randn(B, hq, 128, device=DEV, dtype=torch.bfloat16)
    out = ops.decode_attention(q, kc, vc, bt, sl, 128 ** -0.5, part_size=1024)
    live = (sl > 0).nonzero().view(-1)
    exp = _attention64(q[live], kc, vc, bt[live], [1] * len(live), [x for x in n if x], 128 ** -0.5)
    err = (out[live].double() - exp).abs()
    assert (err <= exp.abs() * 2.0 ** -8 + 1e-4).all(), err.max()


def test_decode_attention_finds_sharers_far_apart():
    """Prompt prefixes shared by sequences 32 rows apart: the sums are right, and the shared pages go
    through the caches as those of neighbours do (past them 1.4 times as long)."""
    torch.manual_seed(14)
    B, hq, hkv, bs, shared, n = 256, 32, 8, 32, 512, 576
    own = -(-n // bs) - shared // bs
    nb = 32 * (shared // bs) + B * own
    kc, vc = (torch.randn(nb, hkv, bs, 128, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    q = torch.randn(B, hq, 128, device=DEV, dtype=torch.bfloat16)
    sl = torch.full((B,), n, dtype=torch.int32, device=DEV)
    rows = torch.arange(B)

    def table(group):
        pre = group[:, None] * (shared // bs) + torch.arange(shared // bs)
        tail = 32 * (shared // bs) + rows[:, None] * own + torch.arange(own)
        return torch.cat([pre, tail], 1).int().to(DEV)

    best, tables = {}, {"apart": table(rows % 32), "all": table(rows * 0)}
    for _ in range(12):
        for name, bt in tables.items():
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(10):
                out = ops.decode_attention(q, kc, vc, bt, sl, 128 ** -0.5, part_size=1024)
            b.record()
            torch.cuda.synchronize()
            best[name] = min(best.get(name, 1e9), a.elapsed_time(b))
            if name == "apart":
                got = out[::37]
    exp = _attention64(q[::37], kc, vc, tables["apart"][::37], [1] * 7, [n] * 7, 128 ** -0.5)
    assert ((got.double() - exp).abs() <= exp.abs() * 2.0 ** -8 + 1e-4).all()
    assert best["apart"] < 1.2 * best["all"], best


def test_sample_greedy_matches_argmax():
    logits = torch.randn(7, 128256, device=DEV)
    temp = torch.zeros(7, device=DEV)
    tok = ops.sample(logits, temp)
    assert torch.equal(tok.long().cpu(), logits.argmax(-1).cpu())
    tok16 = ops.sample(logits.bfloat16(), temp)
    assert torch.equal(tok16.long().cpu(), logits.bfloat16().float().argmax(-1).cpu())


def test_sample_bf16_vector_path_logprob_and_masked():
    """bf16 rows take the fused one-pass max/argmax/partition sweep (16-B
    loads): token, log-prob and -inf (grammar-masked) entries vs fp32 torch."""
    torch.manual_seed(11)
    B, V = 9, 128256
    logits = (torch.randn(B, V, device=DEV) * 4).bfloat16()
    logits[0, :1000] = float("-inf")
    logits[1, 5] = 30.0
    logits[2, 7] = 25.0
    logits[2, 9] = 25.0  # tie -> lowest index, like argmax
    temp = torch.zeros(B, device=DEV)
    lp = torch.empty(B, device=DEV)
    tok = ops.sample(logits, temp, out_logprob=lp).long().cpu()
    f = logits.float().cpu()
    assert torch.equal(tok, f.argmax(-1))
    exp_lp = torch.log_softmax(f, -1)[torch.arange(B), tok]
    assert (lp.cpu() - exp_lp).abs().max() < 1e-3
    # temperature path (same fused sweep feeds its max / partition function)
    temp = torch.full((B,), 0.9, device=DEV)
    seeds = torch.arange(B, dtype=torch.int64, device=DEV)
    tok = ops.sample(logits, temp, seeds=seeds, steps=seeds, out_logprob=lp).long().cpu()
    exp_lp = torch.log_softmax(f / 0.9, -1)[torch.arange(B), tok]
    assert (lp.cpu() - exp_lp).abs().max() < 1e-3
    assert bool(torch.isfinite(f[torch.arange(B), tok]).all())


def test_sample_topk_topp_support():
    torch.manual_seed(5)
    B, V = 6, 32000
    logits = torch.randn(B, V, device=DEV) * 3
    temp = torch.full((B,), 0.8, device=DEV)
    top_k = torch.tensor([0, 1, 5, 50, 0, 20], dtype=torch.int32, device=DEV)
    top_p = torch.tensor([1.0, 1.0, 1.0, 0.9, 0.5, 0.3], device=DEV)
    allowed = ref.sample_mask(logits.cpu(), temp.cpu(), top_k.cpu(), top_p.cpu())
    for step in range(20):
        seeds = torch.full((B,), 1234, dtype=torch.int64, device=DEV)
        steps = torch.full((B,), step, dtype=torch.int64, device=DEV)
        tok = ops.sample(logits, temp, top_k, top_p, seeds=seeds, steps=steps).long().cpu()
        assert allowed[torch.arange(B), tok].all(), (step, tok)
    # top_k = 1 is greedy
    assert int(tok[1]) == int(logits[1].argmax())


def test_sample_distribution_temperature():
    """Gumbel-max draw matches softmax(logits / T) in distribution."""
    V = 8
    logits = torch.tensor([[2.0, 1.0, 0.5, 0.0, -1.0, -2.0, 0.3, 1.5]], device=DEV)
    temp = torch.full((4096,), 0.7, device=DEV)
    big = logits.expand(4096, V).contiguous()
    seeds = torch.arange(4096, dtype=torch.int64, device=DEV)
    tok = ops.sample(big, temp, seeds=seeds, steps=torch.zeros(4096, dtype=torch.int64,
                                                                  device=DEV)).long().cpu()
    freq = torch.bincount(tok, minlength=V).float() / 4096
    exp = torch.softmax(logits[0].cpu() / 0.7, -1)
    assert (freq - exp).abs().max() < 0.03


def test_sample_penalties():
    B, V = 2, 1000
    logits = torch.zeros(B, V, device=DEV)
    logits[:, 10] = 5.0
    logits[:, 20] = 4.0
    counts = torch.zeros(B, V, dtype=torch.int32, device=DEV)
    counts[0, 10] = 3
    temp = torch.zeros(B, device=DEV)
    freq = torch.tensor([1.0, 1.0], device=DEV)
    pres = torch.tensor([0.0, 0.0], device=DEV)
    tok = ops.sample(logits, temp, counts=counts, freq_pen=freq, pres_pen=pres).cpu()
    assert tok.tolist() == [20, 10]
    assert int(counts[0, 20]) == 1 and int(counts[1, 10]) == 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("V", [1000, 128256])
def test_apply_token_mask_matches_reference(dtype, V):
    g = torch.Generator().manual_seed(5)
    B, W = 5, (V + 31) // 32
    logits = torch.randn(B, V, generator=g).to(dtype)
    mask = torch.randint(-2**31, 2**31 - 1, (B, W), generator=g, dtype=torch.int64).to(torch.int32)
    mask[2] = -1  # an unconstrained row stays untouched
    want = ref.apply_token_mask(logits.float().clone(), mask)
    got = ops.apply_token_mask(logits.cuda(), mask.cuda()).float().cpu()
    assert torch.equal(torch.isinf(got), torch.isinf(want))
    fin = torch.isfinite(want)
    assert torch.equal(got[fin], want[fin])
    # masked greedy sampling picks the best ALLOWED token
    tok = ops.sample(ops.apply_token_mask(logits.cuda(), mask.cuda()),
                     torch.zeros(B, device="cuda"))
    assert torch.equal(tok.cpu().long(), want.argmax(-1))
