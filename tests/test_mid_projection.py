"""Projections of more rows than the few-row kernels take and fewer than the prefill GEMM asks for:
which way each goes, the product, and the sums that its consumer makes of it."""
import pytest
import torch

from omnia_amd import ops
from omnia_amd.models.projection import Parts, Projections

ROWS = (257, 512, 999, 2001, 2049)
# weight rows, K -> the way of each of ROWS: the table's slices are elsewhere (test_midm_dispatch.py)
WAYS = {(2048, 8192): ("slices", "slices", "slices", "slices", "tile"),  # long K
        (4096, 2048): ("library", "library", "library", "plain", "tile"),  # fills a round at 2001
        (2048, 2048): ("library", "library", "library", "library", "tile")}


class Model(Projections):
    device, dtype, tp, _ws = torch.device("cuda"), torch.bfloat16, 1, {}


def _spied(monkeypatch):
    used = []

    def spy(name):
        f = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, **kw: (used.append(name), f(*a, **kw))[1])

    for name in ("pgemm", "pgemm_splitk", "linear"):
        spy(name)
    return used


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("R,K", WAYS)
def test_way_and_product(R, K, M, dev, monkeypatch):
    g = torch.Generator().manual_seed(M + R)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(dev)
    w = (torch.randn(R, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(dev)
    way = WAYS[R, K][ROWS.index(M)]
    used = _spied(monkeypatch)
    y = Model()._proj("down", x, w, False)
    assert used == {"slices": ["pgemm_splitk"], "library": ["linear"]}.get(way, ["pgemm"])
    assert isinstance(y, Parts) == (way == "slices")
    want = x.double() @ w.double().t()
    p = y.t.double().sum(0) if isinstance(y, Parts) else y.double()
    # fp32 sums, rounded to bf16 where they are not slabs: 2^-8 of a value and of what it is near
    assert ((p - want).abs() <= (2.0 ** -8 if way != "slices" else 1e-4) * (want.abs() + 1)).all()
    if way == "slices":  # their consumer: residual += bf16(sum), and its norm
        res = torch.randn(M, R, generator=g).to(torch.bfloat16).to(dev)
        sums = res.double() + want
        h = ops.splitk_add_rmsnorm(y.t, res, torch.ones(R, dtype=torch.bfloat16, device=dev), 1e-5)
        assert ((res.double() - sums).abs() <= 2.0 ** -7 * (sums.abs() + want.abs() + 0.1)).all()
        rms = (res.double().pow(2).mean(1, keepdim=True) + 1e-5).sqrt()
        assert ((h.double() - res.double() / rms).abs() <= 2.0 ** -6 * (h.double().abs() + 0.1)).all()


@pytest.mark.parametrize("how", ["switch", "decode", "plain rows", "off grid", "strided", "ranks"])
def test_what_stays_with_the_library(how, monkeypatch):
    """Long K of 512 rows, but: OMNIA_MIDM=0, a decode step, a consumer that takes no slabs, weights
    off the 16-byte grid or of other strides, and ranks of a tensor-parallel group."""
    m, used = Model(), _spied(monkeypatch)
    x = torch.zeros(512, 8192, dtype=torch.bfloat16)
    w = torch.zeros(2048, 8192, dtype=torch.bfloat16)
    if how == "switch":
        monkeypatch.setattr(ops, "_midm_on", False)
    if how == "off grid":
        w = torch.zeros(2048 * 8192 + 1, dtype=torch.bfloat16)[1:].view(2048, 8192)
    if how == "strided":
        w = torch.zeros(2048, 8200, dtype=torch.bfloat16)[:, :8192]
    if how == "ranks":
        m.tp = 2
    y = m._proj("down", x, w, how == "decode", how != "plain rows")
    assert used == ["linear"] and y.shape == (512, 2048)


@pytest.mark.parametrize("M,N,K,pays", [
    (256, 8192, 2048, False), (384, 8192, 2048, False), (385, 8192, 2048, True),  # a narrow round
    (512, 8192, 2048, True), (513, 8192, 2048, False), (999, 8192, 2048, True),  # and a wide one
    (512, 14336, 4096, True), (513, 14336, 4096, False), (768, 14336, 4096, True)])
def test_gated_projections_on_both_sides_of_the_rule(M, N, K, pays):
    """A gated tile, wide or narrow, from three quarters of its rounds' work useful."""
    w = torch.empty(2 * N, K, dtype=torch.bfloat16, device="meta")
    assert Model()._pgemm_ok(M, K, N, False, w) == pays
    assert not Model()._pgemm_ok(M, K, N, True, w)


@pytest.mark.parametrize("M,R,K,fills", [
    (1843, 4096, 2048, False), (1844, 4096, 2048, True), (2048, 4096, 2048, True),  # .9 of a round
    (2049, 4096, 2048, False),                                           # nine rows of tiles
    (1024, 8192, 1024, True), (1024, 8192 + 128, 1024, False), (1024, 8192, 1024 + 64, False),
    (1449, 16128, 11392, False), (1014, 23808, 1024, False),             # three narrow rounds
    (1001, 15872, 14208, False), (2048, 8192, 2048, False)])             # one wide one
def test_plain_projections_on_both_sides_of_the_rule(M, R, K, fills):
    w = torch.empty(R, K, dtype=torch.bfloat16, device="meta")
    assert ops.plain_tile_fills(M, w) == fills


@pytest.mark.parametrize("M,R,K,cols", [
    (256, 10240, 512, 0), (257, 10240, 512, 128), (257, 16384, 512, 0),      # 240 and 384 tiles
    (1126, 2048, 2048, 0), (1127, 2048, 2048, 128), (2048, 2048, 2048, 128),  # .55 of a round
    (563, 2048, 2048, 0), (564, 2048, 2048, 64), (1024, 2048, 2048, 64), (1025, 2048, 2048, 0),
    (1536, 2048, 2112, 0), (1537, 2048, 2112, 128),                          # K past 2048: .75
    (665, 2048, 2112, 0), (666, 2048, 2112, 64),                             # and .65
    (2048, 2048, 6144, 128), (2048, 2048, 6208, 0), (2049, 2048, 2048, 0),
    (999, 1664 + 64, 2048, 64), (999, 1664 + 32, 2048, 0), (2000, 2048, 2048 + 32, 0)])
def test_smaller_tiles_on_both_sides_of_the_rule(M, R, K, cols):
    w = torch.empty(R, K, dtype=torch.bfloat16, device="meta")
    assert ops.small_tile_cols(M, w) == cols
    assert not ops.small_tile_cols(M, w[:, ::2])


def test_down_tile_cols():
    """Narrow while the segments to be expected are one round of narrow tiles, half of each expert's
    last one empty; of a shard's experts, their part of the assignments."""
    cols = ops.down_tile_cols
    assert cols(3072, 8, 8, 2048) == 128 and cols(3200, 8, 8, 2048) == 256  # 16 segments of 16
    assert cols(1024, 8, 8, 4096) == 128 and cols(1040, 8, 8, 4096) == 256  # 8 of 32
    assert cols(8192, 8, 1, 2048) == 128
    assert cols(1, 1, 1, 2048 + 128) == 256  # not whole wide tiles: refused either way
