"""Prefill GEMM with fused epilogues (ops/csrc/pgemm.hip) against fp32 PyTorch
references of the same ops: plain / row-scaled GEMM, gate_up + SwiGLU, residual
add + row sum of squares, QKV + RoPE + paged KV write.  Ragged M (not a multiple
of the 256-row tile) and K > one iteration are covered; every check has a
negative control (a deliberately wrong reference must FAIL the same tolerance)."""
import pytest
import torch

from omnia_amd import ops
from omnia_amd.ops import reference as ref

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _rand(*shape, std=1.0, gen=None):
    return (torch.randn(*shape, device=DEV, generator=gen) * std).to(torch.bfloat16)


def _close(got, want, tol):
    err = (got.float() - want.float()).abs().max().item()
    scale = want.float().abs().max().item()
    return err <= tol * scale, err / max(scale, 1e-30)


@pytest.fixture(scope="module")
def gen():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    g = torch.Generator(device=DEV)
    g.manual_seed(1234)
    return g


@pytest.mark.parametrize("M,N,K", [(256, 512, 128), (300, 768, 512), (1000, 1024, 1280)])
def test_plain_and_row_scaled(gen, M, N, K):
    x = _rand(M, K, gen=gen)
    w = _rand(N, K, std=0.05, gen=gen)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.pgemm(0, x, w, out=out)
    want = x.float() @ w.float().t()
    ok, e = _close(out, want, 1e-2)
    assert ok, e
    # asymmetric negative control: the transposed-operand product must not match
    bad = x.float() @ w.float().flip(0).t()
    assert not _close(out, bad, 1e-2)[0]
    # row scale from 3 partial sums of squares
    ss = torch.rand(M, 3, device=DEV, generator=gen) * K
    ops.pgemm(0, x, w, out=out, ss_in=ss, inv_d=1.0 / K, eps=1e-5)
    rs = torch.rsqrt(ss.sum(1) / K + 1e-5)
    ok, e = _close(out, want * rs[:, None], 1e-2)
    assert ok, e
    assert not _close(out, want, 1e-2)[0]


@pytest.mark.parametrize("M,F,K", [(256, 256, 256), (517, 384, 640)])
def test_swiglu(gen, M, F, K):
    x = _rand(M, K, gen=gen)
    w = _rand(2 * F, K, std=0.05, gen=gen)
    ss = torch.rand(M, 2, device=DEV, generator=gen) * K
    out = torch.empty(M, F, dtype=torch.bfloat16, device=DEV)
    ops.pgemm(1, x, w, out=out, ss_in=ss, inv_d=1.0 / K, eps=1e-6)
    rs = torch.rsqrt(ss.sum(1) / K + 1e-6)[:, None]
    h = (x.float() @ w.float().t()) * rs
    g, u = h[:, :F], h[:, F:]
    want = torch.nn.functional.silu(g) * u
    ok, e = _close(out, want, 1.5e-2)
    assert ok, e
    swapped = torch.nn.functional.silu(u) * g
    assert not _close(out, swapped, 1.5e-2)[0]


@pytest.mark.parametrize("M,N,K", [(256, 512, 256), (389, 1024, 384)])
def test_residual_sumsq(gen, M, N, K):
    x = _rand(M, K, gen=gen)
    w = _rand(N, K, std=0.05, gen=gen)
    res = _rand(M, N, gen=gen)
    res0 = res.clone()
    ss = torch.full((M, N // 256), -1.0, device=DEV)
    ops.pgemm(2, x, w, out=res, ss_out=ss)
    g = (x.float() @ w.float().t()).to(torch.bfloat16)
    want = (res0.float() + g.float()).to(torch.bfloat16)
    ok, e = _close(res, want, 1e-2)
    assert ok, e
    want_ss = want.float().pow(2).view(M, N // 256, 256).sum(-1)
    ok, e = _close(ss, want_ss, 1e-3)
    assert ok, e
    assert not _close(res, res0, 1e-2)[0]


def test_qkv_rope_kv_write(gen):
    hq, hkv, D, bs = 8, 2, 128, 16
    M, K = 300, 512
    N = (hq + 2 * hkv) * D
    x = _rand(M, K, gen=gen)
    w = _rand(N, K, std=0.05, gen=gen)
    ss = torch.rand(M, 1, device=DEV, generator=gen) * K
    positions = torch.randint(0, 4000, (M,), device=DEV, dtype=torch.int32, generator=gen)
    cos_sin = ref.rope_cos_sin(8192, D, 5e5, {"rope_type": "llama3", "factor": 8.0}, device=DEV)
    nb = 64
    kc = torch.zeros(nb, hkv, bs, D, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    perm = torch.randperm(nb * bs, device=DEV, generator=gen)[:M]
    slots = perm.to(torch.int64)
    slots[5] = -1  # padding row: no KV write
    q = torch.empty(M, hq * D, dtype=torch.bfloat16, device=DEV)
    ops.pgemm(3, x, w, out=q, ss_in=ss, inv_d=1.0 / K, eps=1e-5, positions=positions,
              cos_sin=cos_sin, k_cache=kc, v_cache=vc, slots=slots, hq=hq, hkv=hkv,
              block_size=bs)
    rs = torch.rsqrt(ss.sum(1) / K + 1e-5)[:, None]
    qkv = ((x.float() @ w.float().t()) * rs).to(torch.bfloat16)
    qq = ref.apply_rope(qkv[:, : hq * D].view(M, hq, D), positions, cos_sin)
    kk = ref.apply_rope(qkv[:, hq * D:(hq + hkv) * D].view(M, hkv, D), positions, cos_sin)
    vv = qkv[:, (hq + hkv) * D:].view(M, hkv, D)
    ok, e = _close(q.view(M, hq, D), qq, 2e-2)
    assert ok, e
    unrotated = qkv[:, : hq * D]
    assert not _close(q, unrotated, 2e-2)[0]
    kc_want = torch.zeros_like(kc)
    vc_want = torch.zeros_like(vc)
    keep = slots >= 0
    ref.write_kv(kc_want, vc_want, kk[keep], vv[keep], slots[keep])
    ok, e = _close(kc, kc_want, 2e-2)
    assert ok, e
    ok, e = _close(vc, vc_want, 2e-2)
    assert ok, e


def test_row_sumsq(gen):
    x = _rand(333, 4096, gen=gen)
    ss = torch.empty(333, device=DEV)
    ops.row_sumsq(x, out=ss)
    ok, e = _close(ss, x.float().pow(2).sum(1), 1e-4)
    assert ok, e


def test_rejects_bad_shapes(gen):
    x = _rand(256, 192, gen=gen)  # K not a multiple of 128
    w = _rand(256, 192, gen=gen)
    with pytest.raises(RuntimeError):
        ops.pgemm(0, x, w, out=torch.empty(256, 256, dtype=torch.bfloat16, device=DEV))


@pytest.mark.parametrize("epi,cols", [(0, 128), (0, 256), (1, 128), (1, 256), (2, 256)])
def test_a_rows_bits_are_its_own(gen, epi, cols):
    """A row's result does not depend on how many rows the step has, on where in the step it lies, or
    on the run."""
    K, N = 1024, 512
    x = _rand(777, K, gen=gen)
    w = _rand(2 * N if epi == 1 else N, K, std=0.05, gen=gen)
    ss = torch.rand(777, 2, device=DEV, generator=gen) * K
    res = _rand(777, N, gen=gen)

    def run(a, b):
        if epi == 2:
            o, sso = res[a:b].clone(), torch.zeros(b - a, N // 256, device=DEV)
            ops.pgemm(2, x[a:b], w, out=o, ss_out=sso)
            return o, sso
        return (ops.pgemm(epi, x[a:b], w, ss_in=ss[a:b], inv_d=1.0 / K, eps=1e-5, cols=cols),)

    whole = run(0, 777)
    for a, b in ((0, 777), (0, 1), (255, 258), (300, 777)):
        for got, want in zip(run(a, b), whole):
            assert torch.equal(got, want[a:b])


@pytest.mark.parametrize("M,N,K,S", [(256, 512, 1024, 4), (192, 768, 2048, 8), (77, 256, 512, 2),
                                     (300, 512, 896, 7)])
def test_splitk_slabs(gen, M, N, K, S):
    """EPI 4: fp16 slab s holds x[:, Ks] @ w[:, Ks]^T of K-slice s; decode sizes
    (one m-tile, ragged) and prefill sizes (two m-tiles) against fp32 matmuls."""
    x = _rand(M, K, gen=gen)
    w = _rand(N, K, std=0.05, gen=gen)
    parts = torch.full((S, M, N), float("nan"), dtype=torch.float16, device=DEV)
    ops.pgemm_splitk(x, w, S, parts)
    ks = K // S
    for s in range(S):
        want = x[:, s * ks:(s + 1) * ks].float() @ w[:, s * ks:(s + 1) * ks].float().t()
        ok, e = _close(parts[s], want, 2e-3)
        assert ok, (s, e)
    total = x.float() @ w.float().t()
    ok, e = _close(parts.float().sum(0), total, 5e-3)
    assert ok, e
    # negative control: the slabs in the wrong K order do not match slice 0
    want0 = x[:, :ks].float() @ w[:, :ks].float().t()
    assert not _close(parts[S - 1], want0, 2e-3)[0]


def test_splitk_saturates_fp16(gen):
    """A K-slice partial beyond the fp16 range saturates to +-65504 (finite), so
    the consumer never sees inf / NaN."""
    M, N, K, S = 256, 256, 512, 2
    x = torch.full((M, K), 16.0, dtype=torch.bfloat16, device=DEV)
    w = torch.full((N, K), 16.0, dtype=torch.bfloat16, device=DEV)  # partial = 256*256 = 65536
    w[: N // 2] = -16.0
    parts = torch.empty(S, M, N, dtype=torch.float16, device=DEV)
    ops.pgemm_splitk(x, w, S, parts)
    assert torch.isfinite(parts).all()
    assert (parts[:, :, N // 2:] == 65504).all() and (parts[:, :, : N // 2] == -65504).all()


def test_mid_size_slabs_hold_large_sums():
    """A step of 512 rows, whose projection of 4096 the table cuts in 8: the slabs hold a row's sum
    of 393216, 49152 each."""
    from omnia_amd.models.projection import Parts, Projections

    class Model(Projections):
        device, dtype, tp, _ws = torch.device(DEV), torch.bfloat16, 1, {}

    x = torch.full((512, 4096), 16.0, dtype=torch.bfloat16, device=DEV)
    y = Model()._proj("o", x, torch.full((4096, 4096), 6.0, dtype=torch.bfloat16, device=DEV), False)
    assert isinstance(y, Parts) and (y.t.float().sum(0) == 96 * 4096).all()


def test_slabs_of_the_split_tile_in_fp32():
    """OMNIA_SPLITK_FP32=1 on it too: sums past fp16's range."""
    from omnia_amd.models.projection import Projections

    class Model(Projections):
        device, dtype, tp, _ws = torch.device(DEV), torch.bfloat16, 1, {}
        splitk_half = False

    x = torch.full((512, 4096), 16.0, dtype=torch.bfloat16, device=DEV)
    w = torch.full((4096, 4096), 96.0, dtype=torch.bfloat16, device=DEV)
    y = Model()._proj("o", x, w, False)
    assert y.t.dtype == torch.float32 and (y.t.sum(0) == 1536 * 4096).all()


def test_slices_of_the_narrow_tile_whatever_torchs_default_type(gen):
    """Their slabs are fp32, not of the type that new tensors have by default."""
    from omnia_amd.models.projection import Parts, Projections

    class Model(Projections):
        device, dtype, tp, _ws = torch.device(DEV), torch.bfloat16, 1, {}

    x, w = _rand(300, 8192, gen=gen), _rand(2048, 8192, std=0.05, gen=gen)
    want = x.double() @ w.double().t()
    torch.set_default_dtype(torch.bfloat16)
    try:
        y = Model()._proj("down", x, w, False)
    finally:
        torch.set_default_dtype(torch.float32)
    assert isinstance(y, Parts) and y.t.dtype == torch.float32
    # fp32 sums of K exact products: K roundings of at most 2^-24 of the sum of magnitudes
    bound = 8192 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert ((y.t.double().sum(0) - want).abs() <= bound).all()


def test_splitk_feeds_consumer(gen):
    """pgemm split-K slabs through splitk_swiglu == SwiGLU of the fp32 product."""
    M, F, K, S = 256, 512, 2048, 4
    x = _rand(M, K, gen=gen)
    w = _rand(2 * F, K, std=0.05, gen=gen)
    act = ops.splitk_swiglu(ops.pgemm_splitk(x, w, S))
    h = (x.float() @ w.float().t()).to(torch.bfloat16).float()
    want = torch.nn.functional.silu(h[:, :F]) * h[:, F:]
    ok, e = _close(act, want, 2e-2)
    assert ok, e


def test_splitk_rejects_bad_split(gen):
    x = _rand(256, 1024, gen=gen)
    w = _rand(256, 1024, gen=gen)
    with pytest.raises(RuntimeError):  # K / S = 341.33
        ops.pgemm_splitk(x, w, 3)
    with pytest.raises(RuntimeError):  # K / S = 64: an odd number of K-tiles
        ops.pgemm_splitk(x, w, 16)


@pytest.mark.parametrize("M,N,K,S", [(300, 256, 320, 5), (129, 512, 448, 4), (257, 256, 1152, 5),
                                     (513, 256, 64, 1), (700, 512, 4096, 3)])
@pytest.mark.parametrize("cols", [128, 256])
def test_uneven_slices(gen, M, N, K, S, cols):
    """One K-tile a slice, odd numbers of them and slices of two lengths: each slab is its slice's sum, to
    K roundings of at most 2^-24 of the sum of magnitudes."""
    x, w = _rand(M, K, gen=gen), _rand(N, K, std=0.05, gen=gen)
    parts = torch.empty(S, M, N, device=DEV)
    ops.pgemm_splitk(x, w, S, parts, cols=cols, uneven=True)
    at = [s * (K // 64) // S * 64 for s in range(S + 1)]
    for s, (a, b) in enumerate(zip(at, at[1:])):
        xs, ws = x[:, a:b].double(), w[:, a:b].double().t()
        assert ((parts[s].double() - xs @ ws).abs() <= K * 2.0 ** -24 * (xs.abs() @ ws.abs())).all()
    assert torch.equal(ops.pgemm_splitk(x, w, S, cols=cols, uneven=True), parts.half())
    with pytest.raises(RuntimeError):  # a slice without a K-tile
        ops.pgemm_splitk(x, w, K // 64 + 1, cols=cols, uneven=True) if K < 1024 else \
            ops.pgemm_splitk(x, w, S, cols=cols)


@pytest.mark.parametrize("hq,hkv", [(8, 1), (4, 1), (6, 1)])
def test_qkv_epilogue_tp_shard_heads(gen, hq, hkv):
    """TP shards' QKV: one KV head per rank (Llama-3-70B at TP=8: hq 8, hkv 1 ->
    10 heads = 5 tiles) -- 256-column tiles straddle the q / k / v boundaries;
    the per-head epilogue still routes q, k and v correctly."""
    D, bs, M, K = 128, 16, 300, 512
    N = (hq + 2 * hkv) * D
    x = _rand(M, K, gen=gen)
    w = _rand(N, K, std=0.05, gen=gen)
    positions = torch.randint(0, 4000, (M,), device=DEV, dtype=torch.int32, generator=gen)
    cos_sin = ref.rope_cos_sin(8192, D, 5e5, None, device=DEV)
    nb = 64
    kc = torch.zeros(nb, hkv, bs, D, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    slots = torch.randperm(nb * bs, device=DEV, generator=gen)[:M].to(torch.int64)
    q = torch.empty(M, hq * D, dtype=torch.bfloat16, device=DEV)
    ops.pgemm(3, x, w, out=q, positions=positions, cos_sin=cos_sin, k_cache=kc, v_cache=vc,
              slots=slots, hq=hq, hkv=hkv, block_size=bs)
    qkv = (x.float() @ w.float().t()).to(torch.bfloat16)
    qq = ref.apply_rope(qkv[:, : hq * D].view(M, hq, D), positions, cos_sin)
    kk = ref.apply_rope(qkv[:, hq * D:(hq + hkv) * D].view(M, hkv, D), positions, cos_sin)
    vv = qkv[:, (hq + hkv) * D:].view(M, hkv, D)
    ok, e = _close(q.view(M, hq, D), qq, 2e-2)
    assert ok, e
    kw, vw = torch.zeros_like(kc), torch.zeros_like(vc)
    ref.write_kv(kw, vw, kk, vv, slots)
    assert _close(kc, kw, 2e-2)[0] and _close(vc, vw, 2e-2)[0]
    assert not _close(vc, kw, 2e-2)[0]  # k and v not swapped


@pytest.mark.parametrize("M,N,K", [
    (1, 256, 128), (255, 256, 256), (257, 512, 384),  # a row, a tile less and more than one
    (1100, 768, 640), (2049, 512, 768),  # groups of 4 m-tiles and a rest; the ring's turns
    (2100, 16384, 4224),  # more than 128 MB of weights: groups of 8 m-tiles and a rest
])
def test_tile_and_ring_edges(gen, M, N, K):
    """Ragged rows, short and wrapping rings of K-tiles, both block orders: every element once,
    nothing outside.  fp32 sums of K products rounded to bf16: 2^-8 of a value, and the same
    again for values small beside their products' sum."""
    x = _rand(M, K, gen=gen)
    w = _rand(N, K, std=0.05, gen=gen)
    whole = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.pgemm(0, x, w, out=whole[:M])
    want = x.float() @ w.float().t()
    assert ((whole[:M].float() - want).abs() <= 2 ** -8 * (want.abs() + K ** 0.5 * 0.05)).all()
    assert (whole[M] == 7.0).all()


@pytest.mark.parametrize("M,N,K", [(1, 256, 128), (255, 768, 256), (257, 256, 384),
                                   (513, 512, 1152), (300, 128, 512)])
def test_narrow_tile(gen, M, N, K):
    """The tile of 128 columns walks K as the wide one does: the same bits, of every epilogue and
    from fewer K-tiles than its ring has to three rounds of it."""
    x = _rand(M, K, gen=gen)
    w = _rand(N, K, std=0.05, gen=gen)
    ss = torch.rand(M, 3, device=DEV, generator=gen) * K
    if N % 256 == 0:
        for kw in (dict(epi=0), dict(epi=0, ss_in=ss, inv_d=1.0 / K, eps=1e-5), dict(epi=1),
                   dict(epi=1, ss_in=ss, inv_d=1.0 / K, eps=1e-5), dict(epi=1, gelu=True),
                   dict(epi=1, bias=torch.randn(N, device=DEV, generator=gen))):
            assert torch.equal(ops.pgemm(x=x, w=w, cols=128, **kw),
                               ops.pgemm(x=x, w=w, cols=256, **kw))
    want = x.double() @ w.double().t()
    for S in (1, 2, 3):
        if K % (128 * S):
            continue
        half = ops.pgemm_splitk(x, w, S, cols=128)
        if N % 256 == 0:
            assert torch.equal(half, ops.pgemm_splitk(x, w, S, cols=256))
        for cols in (128, 256) if N % 256 == 0 else (128,):
            parts = torch.empty(S, M, N, device=DEV)
            ops.pgemm_splitk(x, w, S, parts, cols=cols)
            # fp32 sums of K exact products: K roundings of at most 2^-24 of the sum of magnitudes
            bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
            assert ((parts.double().sum(0) - want).abs() <= bound).all()
            assert torch.equal(parts.half(), half)


@pytest.mark.parametrize("M,N,K", [(1, 128, 64), (127, 384, 128), (129, 128, 320), (300, 256, 384),
                                   (641, 640, 1152), (2048, 2048, 2048)])
@pytest.mark.parametrize("cols", [64, 128])
def test_small_tile(gen, M, N, K, cols):
    """Tiles of 128 x 128 and 128 x 64, fewer K-tiles than their ring has and more, groups of four m-tiles and a rest:
    the bits of the wide tile where that has whole columns, nothing outside."""
    x = _rand(M, K, gen=gen)
    w = _rand(N, K, std=0.05, gen=gen)
    whole = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.kernels().pgemm_small(whole[:M], x, w, cols)
    want = x.float() @ w.float().t()
    assert ((whole[:M].float() - want).abs() <= 2 ** -8 * (want.abs() + K ** 0.5 * 0.05)).all()
    assert (whole[M] == 7.0).all()
    if N % 256 == 0 and K % 128 == 0:
        assert torch.equal(whole[:M], ops.pgemm(0, x, w))
    for bad in (w[:, :K // 2], w[1:], torch.empty(N * K + 4, dtype=w.dtype, device=DEV)[4:].view(N, K)):
        with pytest.raises(RuntimeError):
            ops.kernels().pgemm_small(whole[:M], x[:, :bad.shape[1]].contiguous(), bad, cols)


@pytest.mark.parametrize("M,tiles", [(255, 1), (512, 128), (257, 130), (700, 255), (250, 257),
                                     (1000, 384), (900, 388), (2049, 513)])
def test_tiles_cut_in_two(gen, M, tiles):
    """Wide tiles of a last round of 128 or fewer are cut: the bits of the narrow tile, every element
    once, for sizes of less than a round, of one and more, on both sides of half a round."""
    K, mt = 256, -(-M // 256)
    n = -(-tiles // mt)
    x = _rand(M, K, gen=gen)
    w = _rand(512 * n, K, std=0.05, gen=gen)
    ss = torch.rand(M, 3, device=DEV, generator=gen) * K
    for kw in (dict(epi=0, w=w[:256 * n]), dict(epi=0, w=w[:256 * n], ss_in=ss, inv_d=1.0 / K, eps=1e-5),
               dict(epi=1, w=w[:256 * n]), dict(epi=1, w=w[:256 * n], gelu=True),
               dict(epi=1, w=w[:256 * n], bias=torch.randn(256 * n, device=DEV, generator=gen))):
        cols = kw["w"].shape[0] // (1 + kw["epi"])
        out = torch.full((2, M + 1, cols), 7.0, dtype=torch.bfloat16, device=DEV)
        for o, c in zip(out, (128, 256)):
            ops.pgemm(x=x, out=o[:M], cols=c, **kw)
        assert torch.equal(out[0], out[1]) and (out[:, M] == 7.0).all()


def test_a_second_m_tile_of_a_row_costs_less_than_a_full_one(gen):
    """Narrow tiles of two m-tiles share W's way from HBM, also where one of them has next to nothing to
    do: 257 rows of a gated 4096 x 14336 take .79 as long as 512 (1.02, were W read once for each)."""
    ws = [_rand(4096, 14336, std=0.02, gen=gen) for _ in range(5)]

    def us(M):
        x, out = _rand(M, 14336, gen=gen), torch.empty(M, 2048, dtype=torch.bfloat16, device=DEV)
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for i in range(20):
                ops.pgemm(1, x, ws[i % 5], out=out, cols=128)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 50)
        return best

    assert us(257) < 0.9 * us(512)


@pytest.mark.parametrize("M,N,K", [(2049, 3840, 384), (100, 33024, 1152), (1030, 6656, 4224),
                                   (4000, 6400, 640)])
@pytest.mark.parametrize("how", ["plain", "scaled", "silu", "silu scaled", "silu bias", "gelu"])
def test_wide_tiles_left_whole(gen, M, N, K, how):
    """More than 128 wide tiles in the last round are not cut: 135, 129, 130 and 400, over rings that turn
    often.  The bits of the narrow tile, of tiles of 128 rows and of fewer rows, which are cut; against 64
    bits the roundings of K sums, of at most 2^-24 of the sum of magnitudes, and of the result to bf16."""
    tiles = -(-M // 256) * (N // 256)
    assert tiles % 256 > 128  # a whole round, or tiles % 256 of one, stays
    x, w = _rand(M, K, gen=gen), _rand(N, K, std=0.05, gen=gen)
    kw, one = {}, torch.ones(M, 1, device=DEV, dtype=torch.float64)
    if "scaled" in how:
        ss = torch.rand(M, 3, device=DEV, generator=gen) * K
        kw, one = dict(ss_in=ss, inv_d=1.0 / K, eps=1e-5), \
            torch.rsqrt(ss.double().sum(1) / K + 1e-5)[:, None]
    if "bias" in how:
        kw["bias"] = torch.randn(N, device=DEV, generator=gen)
    epi = int(how.startswith(("silu", "gelu")))
    got = ops.pgemm(epi, x, w, cols=256, gelu=how == "gelu", **kw)
    assert torch.equal(got, ops.pgemm(epi, x, w, cols=128, gelu=how == "gelu", **kw))
    few = dict(kw, ss_in=kw["ss_in"][:60]) if "scaled" in how else kw
    assert torch.equal(got[:60], ops.pgemm(epi, x[:60], w, cols=256, gelu=how == "gelu", **few))
    if how == "plain":
        for cols in (64, 128):
            assert torch.equal(got, ops.pgemm_small(x, w, cols))
    parts = []
    for h, b in zip(w.chunk(1 + epi), kw["bias"].chunk(2) if "bias" in how else (0.0, 0.0)):
        mags = x.double().abs() @ h.double().abs().t()
        parts.append(((x.double() @ h.double().t()) * one + b, K * 2.0 ** -24 * mags * one))
    want, bound = parts[0]
    if epi:  # the activations' slopes stay below 1.2
        (g, dg), (u, du) = parts
        f = torch.nn.functional
        want = (f.gelu(g, approximate="tanh") if how == "gelu" else f.silu(g)) * u
        bound = 1.2 * (dg * (u.abs() + du) + g.abs() * du) + 1e-5 * g.abs() * u.abs()
    assert ((got.double() - want).abs() <= bound + 2.0 ** -8 * want.abs()).all()


def test_narrow_tile_refuses(gen):
    x, w = _rand(4, 128, gen=gen), _rand(192, 128, gen=gen)
    for call in (lambda: ops.pgemm(0, x, w, cols=128), lambda: ops.pgemm(0, x, w[:128], cols=64),
                 lambda: ops.pgemm(0, x, w[:128]), lambda: ops.pgemm_splitk(x, w, 1, cols=128)):
        with pytest.raises(RuntimeError):
            call()
