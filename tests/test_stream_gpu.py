"""Projections of a few rows (``csrc/stream.hip``) and of some tens (``csrc/panel.hip``)
against float64."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

from omnia_amd import ops
from omnia_amd.ops import reference as ref

U = 2.0 ** -8  # half an ulp of a bf16 result, relative


def _mk(M, R, K, seed, lead=()):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(*lead, R, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    return x, w


def _close(got, want, K, rounded=1):
    """fp32 sums of K bf16 products of about 1 / sqrt(K) each, then ``rounded`` bf16 roundings."""
    err = (got.double() - want).abs()
    bound = rounded * U * want.abs() + 4 * K * 2.0 ** -24 * want.abs().clamp(min=1.0)
    assert (err <= bound).all(), float((err - bound).max())


def _weight(w, packed):
    return ops.stream_pack(w) if packed else w


def _normed(x, n=1):
    """Partial sums of squares of the rows, and the rows as a norm kernel leaves them."""
    ss = x.float().pow(2).view(x.shape[0], n, -1).sum(2).contiguous()
    inv = torch.rsqrt(ss.sum(1, keepdim=True) / x.shape[1] + 1e-5)
    return ss, (x.float() * inv).to(torch.bfloat16)


def _close_normed(got, x, w, K, f=lambda h: h):
    """A row's factor is good to an ulp of fp32, which may turn the bf16 rounding of an x here
    and there: half an ulp each, in random directions."""
    want = f(x.double() @ w.double().T)
    err = (got.double() - want).abs()
    bound = 2 * U * want.abs() + 16 * U * (x.double().abs().amax() * w.double().abs().amax()) + 1e-5
    assert (err <= bound).all(), float((err - bound).max())
    assert err.norm() <= 1.2 * U * want.norm()


# one row to a fragment; K of one chunk, fewer chunks than waves, odd numbers of chunks
SIZES = [(1, 16, 64), (15, 48, 192), (16, 4096, 576), (7, 96, 1024), (13, 64, 4160), (16, 512, 640)]


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_plain_norm_and_residual(M, N, K, packed):
    x, w = _mk(M, N, K, M + N + K)
    want = x.double() @ w.double().T
    wk, bias = _weight(w, packed), torch.randn(N, device="cuda")
    _close(ops.stream(0, x, wk, packed=packed, bias=bias), want + bias.double(), K)
    for n in (1, K // 64, K):  # one partial sum a row, some, more than 4 a lane
        ss, xn = _normed(x, n)
        got = ops.stream(0, x, wk, packed=packed, ss=ss, inv_d=1.0 / K, eps=1e-5)
        _close_normed(got, xn, w, K)
    res = torch.randn(M, N, device="cuda").to(torch.bfloat16)
    old = res.clone()
    ss = ops.stream_sums(M, w, "cuda")
    out = ops.stream(2, x, wk, packed=packed, out=res, ss=ss)
    assert out is res
    # the projection in bf16 (a sum at the edge of a rounding may turn it by an ulp), then theirs
    both = want.float().to(torch.bfloat16).double() + old.double()
    err = (res.double() - both).abs()
    assert (err <= U * both.abs() + 2 * U * want.abs() + 1e-6).all()
    assert (err > U * both.abs()).sum() <= 2 + 0.01 * err.numel()
    torch.testing.assert_close(ss.sum(1), res.float().pow(2).sum(1), rtol=1e-5, atol=1e-5)
    # strided rows (columns of a wider matrix), and rows off the 16-byte grid
    wide = torch.randn(M, K + 72, device="cuda").to(torch.bfloat16)
    for off in (8, 3):
        v = wide[:, off:off + K]
        _close(ops.stream(0, v, wk, packed=packed), v.double() @ w.double().T, K)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_gated(M, N, K, gelu, packed):
    x, w = _mk(M, 2 * N, K, M * N)
    wk, b = _weight(w, packed), torch.randn(2 * N, device="cuda")
    h = x.double() @ w.double().T

    def act(v, u):
        return (F.gelu(v, approximate="tanh") if gelu else F.silu(v)) * u

    # v_exp_f32 and v_rcp_f32 are good to a few ulp of fp32: below the bf16 rounding
    hb = h + b.double()
    _close(ops.stream(1, x, wk, packed=packed, bias=b, gelu=gelu), act(*hb.chunk(2, 1)), 4 * K, 1.1)
    ss, xn = _normed(x)
    got = ops.stream(1, x, wk, packed=packed, gelu=gelu, ss=ss, inv_d=1.0 / K, eps=1e-5)
    _close_normed(got, xn, w, K, lambda h: act(*h.chunk(2, 1)))


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("M,hq,hkv,K", [(1, 1, 1, 64), (5, 32, 8, 512), (16, 4, 2, 4096),
                                        (12, 8, 1, 192), (9, 7, 1, 1024)])
def test_qkv(M, hq, hkv, K, packed):
    x, w = _mk(M, (hq + 2 * hkv) * 128, K, M + hq)
    page, nb = 16, 6
    cache = torch.zeros(2, nb, hkv, page, 128, device="cuda", dtype=torch.bfloat16)
    slots = torch.randperm(nb * page, device="cuda")[:M].contiguous()
    if M > 2:
        slots[1] = -1
    pos = torch.randint(0, 500, (M,), device="cuda", dtype=torch.int32)
    cs = ref.rope_cos_sin(512, 128, 10000.0, device="cuda")
    q = ops.stream(3, x, _weight(w, packed), packed=packed, positions=pos, cos_sin=cs,
                   k_cache=cache[0], v_cache=cache[1], slots=slots, hq=hq, hkv=hkv)
    h = (x.double() @ w.double().T).view(M, -1, 128)
    c, s = (t.double()[:, None] for t in cs[pos.long()].chunk(2, 1))
    a, b = h[..., :64], h[..., 64:]
    r = torch.cat([a * c - b * s, b * c + a * s], -1)
    lim = 2 * U * h.abs().amax()  # the projection's rounding, turned, and the result's
    assert (q.view(M, hq, 128).double() - r[:, :hq]).abs().max() <= lim
    want = torch.zeros_like(cache, dtype=torch.float64)
    for m, at in enumerate(slots.tolist()):
        if at >= 0:
            want[0, at // page, :, at % page] = r[m, hq:hq + hkv]
            want[1, at // page, :, at % page] = h[m, hq + hkv:]
    assert (cache.double() - want).abs().max() <= lim


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("glu,gelu", [(None, False), ((1.702, 7.0), False), (None, True)])
@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (5, 8, 2), (32, 8, 2), (3, 33, 1), (7, 4, 4)])
def test_experts_match_the_64_row_kernels(T, E, k, glu, gelu, packed, monkeypatch):
    """Segments of 16 rows, some experts without a row and some with two segments (every row
    to expert 1): the same products as moe.hip's, summed in another order."""
    d, ff = 192, 320
    g = torch.Generator(device="cuda").manual_seed(T + E)
    _, up = _mk(1, ff if gelu else 2 * ff, d, 3, (E,))
    _, down = _mk(1, d, ff, 4, (E,))
    x = torch.randn(T, d, generator=g, device="cuda").to(torch.bfloat16)
    ids = torch.stack([torch.randperm(E, generator=g, device="cuda")[:k] for _ in range(T)]).int()
    if T == 32:
        ids[:, 0], ids[:, 1] = 1, 2
    wts = torch.rand(T, k, generator=g, device="cuda")
    args = (x, up, down, ids.contiguous(), wts, k, E, 0, E, 64, glu, gelu)
    monkeypatch.setattr(ops, "moe_stream_ok", lambda *a: False)
    want = ops._moe_grouped(*args).double()
    monkeypatch.setattr(ops, "moe_stream_ok", lambda *a: True)
    streams = (ops.stream_pack(up), ops.stream_pack(down)) if packed else None
    got = ops._moe_grouped(*args, streams=streams).double()
    # the activations may round apart by an ulp, and so may the results
    assert (got - want).norm() <= 2 * U * want.norm()
    assert ((got - want).abs() <= 4 * U * want.abs().clamp(min=want.pow(2).mean().sqrt())).all()


@pytest.mark.parametrize("T,E,k,lo,hi", [(32, 8, 2, 2, 6), (64, 64, 1, 0, 64), (16, 5, 4, 4, 5),
                                         (33, 8, 2, 0, 8), (6, 65, 2, 0, 65), (1, 4, 1, 0, 4)])
def test_sorted_by_the_kernel_or_before(T, E, k, lo, hi, monkeypatch):
    """Up to 64 assignments and experts the kernel sorts them itself: a shard's experts only, one
    expert with every row, more of either, rows of every lane."""
    g = torch.Generator(device="cuda").manual_seed(T)
    _, up = _mk(1, 256, 128, 3, (hi - lo,))
    _, down = _mk(1, 128, 128, 4, (hi - lo,))
    x = torch.randn(T, 128, generator=g, device="cuda").to(torch.bfloat16)
    ids = torch.stack([torch.randperm(E, generator=g, device="cuda")[:k] for _ in range(T)]).int()
    if E == 5:
        ids[:] = torch.arange(1, 5, device="cuda")
    wts = torch.rand(T, k, generator=g, device="cuda")
    local = ((ids >= lo) & (ids < hi)).view(-1)
    args = (x, up, down, ids.contiguous(), wts, k, E, lo, hi, 64)
    monkeypatch.setattr(ops, "moe_panel_rows", lambda *a: 0)
    res = []
    for few in (False, True):
        monkeypatch.setattr(ops, "moe_stream_ok", lambda *a: few)
        res.append(ops._moe_grouped(*args).double()[local])
    assert (res[0] - res[1]).norm() <= 2 * U * res[0].norm()


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("glu,gelu", [(None, False), ((1.702, 7.0), False), (None, True)])
@pytest.mark.parametrize("bm,T,E,k", [(64, 3, 8, 2), (64, 40, 4, 4), (128, 65, 1, 1),
                                      (128, 129, 3, 1), (128, 300, 9, 2)])
def test_experts_in_panel_segments(bm, T, E, k, glu, gelu, packed, monkeypatch):
    """Segments of 64 and 128 rows: nearly empty, full and one row over (every row of an expert),
    experts without a row, a column tile that is not whole: as the 64-row kernels above."""
    d, ff = 224, 352
    g = torch.Generator(device="cuda").manual_seed(T + E)
    _, up = _mk(1, ff if gelu else 2 * ff, d, 3, (E,))
    _, down = _mk(1, d, ff, 4, (E,))
    up, down = (F.pad(t, (0, -t.shape[2] % 64)).contiguous() for t in (up, down))
    ff = down.shape[2]
    if not gelu:
        up = up.view(E, 2, -1, up.shape[2])
    up = F.pad(up, (0, 0, 0, ff - up.shape[-2])).reshape(E, -1, up.shape[-1]).contiguous()
    down = F.pad(down, (0, 0, 0, up.shape[2] - d)).contiguous()
    x = F.pad(torch.randn(T, d, generator=g, device="cuda"), (0, -d % 64)).to(torch.bfloat16)
    ids = torch.stack([torch.randperm(E, generator=g, device="cuda")[:k] for _ in range(T)]).int()
    if T == 129:
        ids[:] = 1
    wts = torch.rand(T, k, generator=g, device="cuda")
    args = (x, up, down, ids.contiguous(), wts, k, E, 0, E, 64, glu, gelu)
    monkeypatch.setattr(ops, "moe_stream_ok", lambda *a: False)
    monkeypatch.setattr(ops, "moe_panel_rows", lambda *a: 0)
    want = ops._moe_grouped(*args).double()
    monkeypatch.setattr(ops, "moe_panel_rows", lambda *a: bm)
    streams = (ops.stream_pack(up), ops.stream_pack(down)) if packed else None
    got = ops._moe_grouped(*args, streams=streams).double()
    assert (got - want).norm() <= 2 * U * want.norm()
    assert ((got - want).abs() <= 4 * U * want.abs().clamp(min=want.pow(2).mean().sqrt())).all()


def test_segments_by_rows_an_expert():
    """Segments grow with the rows an expert has, the 256-row tile last, and only weights that the
    panel kernel covers take it."""
    up, down = (torch.empty(8, *s, dtype=torch.bfloat16, device="cuda")
                for s in ((256, 2048), (2048, 2048)))
    for packed in (False, True):
        segs = [ops.moe_panel_rows(n, 8, up, down, packed) for n in range(65, 4096, 13)]
        assert segs == sorted(segs) and set(segs) <= {0, 64, 128} and segs[-1] == 128
        assert packed or 64 not in segs
    assert ops.moe_panel_rows(100, 8, up[..., :1024], down[:, :1024], True) == 0
    assert ops.moe_panel_rows(1000, 8, up.float(), down, False) == 0
    # a tile covers what 128-row segments begin with, and few tiles wait for fuller ones
    assert ops.moe_panel_rows(8 * ops.moe_tile_rows(8, 4096) - 1, 8, up, down, False) == 128
    assert ops.moe_tile_rows(8, 2048) > ops.moe_tile_rows(8, 4096) == ops.moe_tile_rows(64, 512)


def test_what_is_refused():
    x, w = _mk(17, 64, 128, 1)
    with pytest.raises(RuntimeError):
        ops.stream(0, x, w)  # rows
    with pytest.raises(RuntimeError):
        ops.stream(0, x[:4, :96].contiguous(), w[:, :96].contiguous())  # whole 64-k chunks
    with pytest.raises(RuntimeError):
        ops.stream(0, x[:4], w[:40].contiguous())  # whole 16-row fragments
    assert not ops.stream_ok(4, w[:40]) and not ops.stream_ok(257, w)
    x, _ = _mk(257, 64, 128, 1)
    with pytest.raises(RuntimeError):
        ops.panel(0, x, w)
    with pytest.raises(RuntimeError):
        ops.panel(0, x[:4], w[:40].contiguous())


def _off_grid(t, at=1):
    """``t`` at an address ``at`` elements past the 16-byte grid."""
    buf = torch.empty(t.numel() + at, dtype=t.dtype, device=t.device)
    return buf[at:].view(t.shape).copy_(t)


@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("M", [1, 16, 40, 200])
def test_weights_the_kernels_do_not_cover_take_the_library(M, strided):
    """Off the 16-byte grid or strided: projections that ran before these kernels still run."""
    from omnia_amd.models.projection import Projections

    class Model(Projections):
        device, dtype, tp, _ws = torch.device("cuda"), torch.bfloat16, 1, {}

    x, w = _mk(M, 64, 128, M)
    v = F.pad(w, (0, 8))[:, :128] if strided else _off_grid(w)
    assert not ops.stream_ok(M, v) and ops.stream_ok(M, w)
    y = Model()._proj("o", x, v, True)
    _close(y, x.double() @ w.double().T, 128)


@pytest.mark.parametrize("key", ["qkv", "o", "gate_up", "down"])
def test_a_layer_with_a_weight_off_the_grid(key):
    """Steps of a few rows run, and give the same, where only a later layer's weight is so."""
    from omnia_amd.models import build_model, resolve

    out = []
    for off in (False, True):
        m = build_model(resolve("tiny-llama"), device="cuda", seed=3)
        assert m.prepack_decode(4) > 0
        if off:
            m.w["layers"][1][key] = _off_grid(m.w["layers"][1][key])
        out.append(_step(m, 4))
    assert torch.equal(*out)


def _step(m, rows, past=40, decode=True, replays=0):
    """Logits of a decode step of ``rows`` sequences, or of a prompt of as many tokens; with
    ``replays`` those of every replay of its captured graph."""
    from omnia_amd.models import allocate_cache
    from omnia_amd.models.llama import ForwardBatch

    def full(n, b=rows):
        return torch.full((b,), n, dtype=torch.int32, device="cuda")

    bs, per, g = 32, -(-(past + 1) // 32), torch.Generator(device="cuda").manual_seed(rows)
    kv = allocate_cache(m, rows * per + 4, bs, "cuda", torch.bfloat16, rows + 1)
    for t in kv.page_tensors():
        t.normal_(generator=g)
    ids = torch.randint(0, m.cfg.vocab_size, (rows,), generator=g, device="cuda").int()
    every = torch.arange(rows, device="cuda")
    if decode:
        bt = (torch.arange(rows * per, device="cuda", dtype=torch.int32) + 1).view(rows, per)
        fb = ForwardBatch(ids, full(past), bt[:, past // bs].long() * bs + past % bs, bt,
                          full(past + 1), every, num_seqs=rows)
    else:
        bt = torch.arange(1, 1 + -(-(past + rows) // bs), device="cuda", dtype=torch.int32)[None]
        at = past + every
        tiles = [torch.tensor(t, dtype=torch.int32, device="cuda")
                 for t in ops.prefill_tiles([rows])]
        fb = ForwardBatch(ids, at.int(), bt[0, at // bs].long() * bs + at % bs, bt,
                          full(past + rows, 1), every, is_decode=False, num_seqs=1,
                          q_start_loc=torch.tensor([0, rows], dtype=torch.int32, device="cuda"),
                          tile_seq=tiles[0], tile_q0=tiles[1])
    if getattr(m, "stateful", False):
        fb.state_slots = torch.arange(1, rows + 1, dtype=torch.int32, device="cuda")
    if not replays:
        return m.forward(fb, kv).float()
    side, out = torch.cuda.Stream(), []
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        m.forward(fb, kv)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        logits = m.forward(fb, kv)
    for _ in range(replays):
        graph.replay()
        out.append(logits.float())
        torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("write", [True, False])
@pytest.mark.parametrize("rows", [3, 40])
@pytest.mark.parametrize("name", ["tiny-llama", "tiny-mixtral", "tiny-sivadra", "tiny-sekazen"])
def test_packed_copies_of_weights_that_change(name, rows, write):
    """Weights written to, or replaced by others (which may take the old ones' addresses), are
    what a step computes with from then on."""
    from omnia_amd.models import build_model, resolve

    def change(v):
        for k in v if isinstance(v, dict) else range(len(v)):
            t = v[k]
            if isinstance(t, (dict, list)):
                change(t)
            elif k in type(m).STREAM_KEYS and isinstance(t, torch.Tensor):
                new = t.flip(-1)
                if write:
                    t.copy_(new)
                else:
                    v[k] = None
                    del t  # the last reference but the model's own
                    v[k] = new.clone()

    out = []
    for pack in (True, False):
        m = build_model(resolve(name), device="cuda", seed=3)
        if pack:
            assert m.prepack_decode(rows) > 0
            before = _step(m, rows)
        change(m.w["layers"])
        out.append(_step(m, rows))
    assert not torch.equal(before, out[1])
    # the copies' products sum in another order than the weights' as they are
    assert (out[0] - out[1]).norm() <= 0.02 * out[1].norm()


@pytest.mark.parametrize("T", [3, 40, 1000])
def test_expert_rows_and_weights_off_the_grid(T):
    """Rows are copied where a kernel reads 16 bytes at a time; weights stay with moe.hip, and so
    do shapes that it refuses."""
    E, d, k = 4, 256, 2
    g = torch.Generator(device="cuda").manual_seed(T)
    _, up = _mk(1, 256, d, 3, (E,))
    _, down = _mk(1, d, 128, 4, (E,))
    x = torch.randn(T, d, generator=g, device="cuda").to(torch.bfloat16)
    router = torch.randn(E, d, generator=g, device="cuda").to(torch.bfloat16)
    want = ops.moe(x, router, up, down, k, E)
    assert torch.equal(ops.moe(_off_grid(x), router, up, down, k, E), want)
    for ws in ((_off_grid(up), down), (up, _off_grid(down))):
        assert not ops.moe_stream_ok(1, E, *ws, False) and not ops.moe_panel_rows(999, E, *ws, False)
        got = ops.moe(x, router, *ws, k, E).double()
        assert (got - want).norm() <= 2 * U * want.double().norm()
    part = up[:, :224].contiguous(), F.pad(down[:, :, :112], (0, 16))
    assert not ops.moe_stream_ok(1, E, *part, True) and not ops.moe_panel_rows(999, E, *part, True)


# rows around the tiles of 64 to 256; columns of fewer units than waves and of a remainder;
# K of one chunk, of slices of unequal length and of fewer chunks than the ring has stages
PANEL = [(1, 16, 64), (17, 48, 128), (63, 272, 576), (64, 2048, 8192), (65, 528, 1024),
         (128, 64, 4160), (129, 4096, 640), (192, 80, 1088), (193, 64, 256), (256, 144, 2048)]



@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("M,N,K", PANEL)
def test_panel_every_split(M, N, K, packed, monkeypatch):
    x, w = _mk(M, N, K, M + N + K)
    want, wk = x.double() @ w.double().T, _weight(w, packed)
    for wn in (4, 8):
        for S in {1, 2, 3, min(16, K // 64)}:
            if S > K // 64:
                continue
            monkeypatch.setattr(ops, "panel_plan", lambda *a: (wn, S))
            got = ops.panel(0, x, wk, packed=packed, slabs=True)
            if S > 1:
                assert got.shape == (S, M, N) and got.dtype == torch.float32
                _close(got.sum(0), want, K, 0)
            else:
                _close(got, want, K)
    monkeypatch.undo()
    wide = torch.randn(M, K + 72, device="cuda").to(torch.bfloat16)
    for off in (8, 3):  # strided rows, and rows off the 16-byte grid
        v = wide[:, off:off + K]
        _close(ops.panel(0, v, wk, packed=packed), v.double() @ w.double().T, K)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("M,N,K", PANEL)
def test_panel_gated(M, N, K, gelu, packed, monkeypatch):
    x, w = _mk(M, 2 * N, K, M * N)
    b = torch.randn(2 * N, device="cuda")
    hb = (x.double() @ w.double().T + b.double()).chunk(2, 1)
    want = (F.gelu(hb[0], approximate="tanh") if gelu else F.silu(hb[0])) * hb[1]
    for wn in (4, 8):
        monkeypatch.setattr(ops, "panel_plan", lambda *a: (wn, 1))
        got = ops.panel(1, x, _weight(w, packed), packed=packed, bias=b, gelu=gelu)
        _close(got, want, 4 * K, 1.1)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("M", [16, 32, 33, 48, 80, 81, 96, 97, 144, 160, 161, 208, 224, 225, 240])
def test_panel_every_height(M, packed, monkeypatch):
    """Blocks of every height, also those whose waves load unlike parts of x, over K from fewer
    chunks than the ring has stages to two rounds of it."""
    for chunks in range(1, 11):
        x, w = _mk(M, 208, 64 * chunks, M + chunks)
        want, wk = x.double() @ w.double().T, _weight(w, packed)
        got = []
        for wn in (2, 4, 8):
            monkeypatch.setattr(ops, "panel_plan", lambda *a: (wn, 1))
            got.append(ops.panel(0, x, wk, packed=packed))
            _close(got[-1], want, 64 * chunks)
            assert torch.equal(got[-1], got[0])


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("M,R,K", [(1, 32, 64), (17, 96, 192), (64, 160, 640), (81, 8192, 128),
                                   (129, 96, 1088), (256, 416, 2048)])
def test_panel_gated_in_blocks_of_two_waves(M, R, K, packed, monkeypatch):
    """The bits of blocks of four waves, blocks without all of their rows included; never slabs."""
    x, w = _mk(M, R, K, M + R + K)
    wk, b = _weight(w, packed), torch.randn(R, device="cuda")
    assert ops.panel_plan(M, R, K, False) == (2, 1)
    got = ops.panel(1, x, wk, packed=packed, bias=b)
    monkeypatch.setattr(ops, "panel_plan", lambda *a: (4, 1))
    assert torch.equal(got, ops.panel(1, x, wk, packed=packed, bias=b))
    g, u = (x.double() @ w.double().T + b.double()).chunk(2, 1)
    _close(got, F.silu(g) * u, 4 * K, 1.1)
    with pytest.raises(RuntimeError):
        ops.kernels().panel_gemm(2, x.new_empty(1, M, R, dtype=torch.float32), x, wk, 2, packed,
                                 None, False)


@pytest.mark.parametrize("gated,R,K", [(False, 32784, 1024), (False, 32768, 1088), (False, 2048, 16448),
                                       (True, 16416, 2112), (True, 16384, 2048)])
def test_panel_of_weights_whose_chunks_are_taken_apart(gated, R, K):
    """Row-major weights of 64 MB and more: of every chunk once, in order where a walk has not 32 of them (gated:
    nor 64), also where their number is odd, has a small power of two or more than 64, in slices too; a row's
    bits are the same whatever the rows beside it and in blocks of other waves."""
    x, w = _mk(200, R, K, R + K)
    whole = ops.panel(int(gated), x, w, slabs=not gated)
    y = whole.sum(0) if whole.dim() == 3 else whole
    want = x.double() @ w.double().T
    if gated:
        g, u = want.chunk(2, 1)
        want = F.silu(g) * u
    _close(y, want, 4 * K, 1.1)
    for M in (1, 33, 100):
        assert torch.equal(ops.panel(int(gated), x[:M], w, slabs=not gated), whole[..., :M, :])
    if whole.dim() == 2:
        out = [torch.empty_like(whole) for _ in range(3)]
        for o, wn in zip(out, (2, 4, 8)):
            ops.kernels().panel_gemm(int(gated), o, x, w, wn, False, None, False)
            assert torch.equal(o, whole)


@pytest.mark.parametrize("gated,R,K,S,apart", [
    (False, 32768, 2048, 1, True), (False, 4096, 14336, 7, True), (False, 8192, 8192, 4, True),
    (True, 16384, 2048, 1, True), (True, 16384, 4096, 1, True),
    (False, 16368, 2048, 1, False), (True, 16352, 2048, 1, False),  # below 64 MB
    (False, 16384, 4096, 1, False), (True, 16384, 2112, 1, False)])
def test_panel_walks_of_32_chunks_are_apart(gated, R, K, S, apart):
    """Large row-major weights in walks of 32 chunks, gated also of 64: every chunk once, in an order that is
    not the packed copy's; others have its bits.  A row's bits are the same whatever the rows beside it and in
    blocks of other waves."""
    x, w = _mk(200, R, K, R + K)
    slabs = S > 1
    whole, packed = (ops.panel(int(gated), x, v, packed=p, slabs=slabs)
                     for v, p in ((w, False), (ops.stream_pack(w), True)))
    assert (whole.shape[0] == S and whole.dim() == 3) == slabs
    want = x.double() @ w.double().T
    if gated:
        g, u = want.chunk(2, 1)
        want = F.silu(g) * u
    for got in (whole, packed):
        _close(got.sum(0) if slabs else got, want, 4 * K, 1.1)
    assert torch.equal(whole, packed) != apart
    for M in (1, 33, 100):
        assert torch.equal(ops.panel(int(gated), x[:M], w, slabs=slabs), whole[..., :M, :])
    for wn in (4, 8) if slabs else (2, 4, 8):
        out = torch.empty_like(whole)
        ops.kernels().panel_gemm(2 if slabs else int(gated), out, x, w, wn, False, None, False)
        assert torch.equal(out, whole)


def test_panel_plans_fit_the_kernel():
    """Whatever the size, a plan is one that the kernel covers, with slices that do not depend on
    the rows."""
    for rows in (16, 240, 4096, 8256, 128256):
        for K in (64, 192, 1024, 14336):
            plans = [ops.panel_plan(M, rows, K, True) for M in (1, 64, 65, 128, 129, 256)]
            assert {wn for wn, _ in plans} <= {4, 8} and len({S for _, S in plans}) == 1
            assert 1 <= plans[0][1] <= min(16, K // 64)
            assert ops.panel_plan(100, rows, K, False)[1] == 1


def test_panel_rows_do_not_depend_on_each_other():
    """The same rows in steps of other sizes give the same bits, slabs included."""
    x, w = _mk(256, 2048, 4096, 9)
    for slabs in (False, True):
        whole = ops.panel(0, x, w, slabs=slabs)
        for M in (1, 20, 64, 100, 130):
            assert torch.equal(ops.panel(0, x[:M], w, slabs=slabs), whole[..., :M, :])


@pytest.mark.parametrize("decode", [True, False])
@pytest.mark.parametrize("pack", [True, False])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 32])
def test_llama_layers_match_the_unfused_path(rows, pack, decode, monkeypatch):
    """Decode steps, captured too, and prompt steps of a small model: the four streamed
    projections a layer (up to 16 rows of packed weights, or of small row-major ones in an eager
    step) and the panel kernel's, against the library's GEMMs with separate norm, RoPE, SwiGLU
    and residual kernels."""
    from omnia_amd.models import build_model, resolve

    m = build_model(resolve("tiny-llama"), device="cuda", seed=4)
    if pack:
        assert m.prepack_decode(32) > 0
    used, real = [], m._use_stream
    monkeypatch.setattr(m, "_use_stream", lambda fb: used.append(real(fb)) or used[-1])
    got = _step(m, rows, decode=decode)
    assert used == [rows <= 16 and (pack or not decode)] and got.shape[0] == rows
    monkeypatch.setattr(ops, "_stream_on", False)
    want = _step(m, rows, decode=decode)
    assert not used[-1]
    # bf16 projections whose sums run in another order, through two layers
    assert (got - want).norm() <= 0.02 * want.norm()
    assert ((got - want).norm(dim=1) <= 0.03 * want.norm(dim=1)).all()
    if decode:
        monkeypatch.setattr(ops, "_stream_on", True)
        for replay in _step(m, rows, replays=3):
            assert torch.equal(replay, got)


def test_gated_tiles_are_taken_where_they_fill_the_chip():
    """Only for more rows than the panel kernel takes, not where one row more leaves most of a
    round empty, and only for weights that the tile covers."""
    for N in (8192, 14336):
        w = torch.empty(2 * N, 128, dtype=torch.bfloat16, device="cuda")
        taken = [M for M in range(1, 2049) if ops.gated_tile_fills(M, w)]
        assert min(taken) > ops.PANEL_MAX_M and 2048 in taken
        for M in taken:  # a round of 256 tiles of 256 x 128, three quarters of it useful
            tiles = -(-M // 256) * (N // 128)
            assert M * N / (-(-tiles // 256) * 256 * 256 * 128) > 0.75
        assert not ops.gated_tile_fills(2048, _off_grid(w))
        assert not ops.gated_tile_fills(2048, F.pad(w, (0, 8))[:, :128])


@pytest.mark.parametrize("M", [511, 512, 513])
def test_gated_projection_on_both_sides_of_the_rule(M):
    """32768 features: two rows of 256 tiles up to 512 rows, half-empty third ones after."""
    from omnia_amd.models.projection import Projections

    class Model(Projections):
        device, dtype, tp, _ws = torch.device("cuda"), torch.bfloat16, 1, {}

    m, N, K = Model(), 32768, 128
    x, w = _mk(M, 2 * N, K, 5)
    assert m._pgemm_ok(M, K, N, False, w) == (M <= 512)
    assert not m._pgemm_ok(M, K, N, False) and not m._pgemm_ok(M, K, N, True, w)
    assert not m._pgemm_ok(M, K, N, False, _off_grid(w))
    g, u = (x.double() @ w.double().t()).split(N, 1)
    _close(ops.pgemm(1, x, w), F.silu(g) * u, K)


@pytest.mark.parametrize("M", [1, 16, 33, 64, 65, 128, 129, 192, 193, 256])
def test_kernels_of_a_projection_by_its_rows(M):
    """Whichever kernel the rows, the size and the layout choose, slabs or not, the product is the
    same; unsliced walks of few blocks and large row-major weights stay with the library."""
    from omnia_amd.models.projection import Parts, Projections

    class Model(Projections):
        device, dtype, tp, _ws = torch.device("cuda"), torch.bfloat16, 1, {}

    for R, K in ((64, 4096), (2048, 192), (8192, 64), (12288, 128), (24576, 64)):
        x, w = _mk(M, R, K, M + R)
        for packed in (False, True):
            m = Model()
            if packed:
                m.w = {"layers": [{"o": w}]}
                assert m.pack_streams() > 0
            for slabs in (False, True):
                y = m._proj("o", x, w, True, slabs)
                assert slabs or not isinstance(y, Parts)
                y = y.t.sum(0) if isinstance(y, Parts) else y
                _close(y, x.double() @ w.double().T, K)
            a = m._few(1, x, w)
            if a is not None:
                g, u = (x.double() @ w.double().T).chunk(2, 1)
                _close(a, F.silu(g) * u, 4 * K, 1.1)
    pay = ops.few_rows_pay
    assert not pay(M, 64, 4096, False, True, False)
    assert pay(M, 57344, 8192, True, False, False) == (M <= 32)
    assert pay(M, 28672, 4096, True, True, False)
    for R, K in ((2048, 2048), (2048, 8192), (4096, 4096)):  # whose slabs hand on fp32 sums
        assert ops.panel_slices(R, K) > 1
        assert pay(M, R, K, False, True, True) and pay(M, R, K, False, False, True)
