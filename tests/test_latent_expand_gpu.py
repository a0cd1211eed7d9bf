"""Latent attention's decode chain: merge and expansion in one launch against the two kernels they
stand for, and the row preparation past a thread's registers."""
import pytest
import torch

from omnia_amd import ops
from omnia_amd.models.config import LatentAttentionSpec, RotarySpec
from omnia_amd.ops import mixers as mops
from omnia_amd.ops import reference_mixers as ref

pytestmark = pytest.mark.gpu


# rows of a block: 4, 8, 16 of a product's; ends of tiles in rows, columns and latent
@pytest.mark.parametrize("rows,heads", [(1, 16), (7, 20), (67, 16), (150, 16)])
@pytest.mark.parametrize("rank,vdim", [(512, 128), (480, 64), (96, 24)])
@pytest.mark.parametrize("splits", [1, 3, 11, 32])
def test_expand_merges(rows, heads, rank, vdim, splits):
    spec = LatentAttentionSpec(heads=heads, dim=64, rot_dim=32, vdim=vdim, q_rank=64, kv_rank=rank,
                               scale=0.1, rotary=RotarySpec(32, 1e4), window=700)
    assert mops.latent_expands_parts(spec)
    g = torch.Generator().manual_seed(rows + rank)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).bfloat16().cuda()

    pages = rnd(64, 32, spec.padded_cache_width)
    bt = torch.stack([torch.randperm(64, generator=g) for _ in range(rows)]).int().cuda()
    pos = torch.tensor([0, 1, 63, 64, 65, 699, 700, 701, 1500, 2047] * 15)[:rows].int().cuda()
    q, w_uv = rnd(rows, heads * spec.padded_cache_width) * 0.5, rnd(heads, spec.v_pad, spec.latent_pad)
    gate = rnd(rows, heads + 24)[:, 8:8 + heads]  # columns of a wider tensor
    o = mops.latent_decode(q, pages, bt, pos, spec, splits)
    want = mops.latent_expand(o, w_uv, spec, gate)
    o, parts = mops.latent_decode(q, pages, bt, pos, spec, splits, merge=False)
    got = mops.latent_expand(o, w_uv, spec, gate, parts=parts)
    # the same sums; fp32 weights of the parts may round the other way, which moves a latent by a
    # bf16 unit, and the results are rounded to bf16 once more
    assert float((got.float() - want.float()).norm() / want.float().norm()) < 2.0 ** -8


@pytest.mark.parametrize("Q,C,R", [(1300, 1100, 64), (1024, 512, 64), (70, 30, 2), (256, 257, 600)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_prep(Q, C, R, dtype):
    g = torch.Generator().manual_seed(Q)

    def rnd(*shape):
        return torch.randn(*shape, generator=g)

    T, Qp, Cp, Rp = 5, -(-Q // 8) * 8, -(-C // 8) * 8, -(-R // 8) * 8
    Lp = Cp + Rp
    x = rnd(T, Qp + Cp + Rp + 8).to(dtype)
    wq, wc, cos_sin = rnd(Q), rnd(C), rnd(40, R)
    pos, slots = torch.tensor([0, 39, 7, 3, 8]).int(), torch.tensor([3, 0, -1, 17, 30])
    cache = torch.zeros(2, 16, Lp, dtype=dtype)
    want = cache.clone()
    wcq = ref.latent_prep(want, x, wq, wc, pos, slots, cos_sin, Qp, Cp, R, 1e-6)
    got = cache.cuda()
    cq = mops.latent_prep(got, x.cuda(), wq.cuda(), wc.cuda(), pos.cuda(), slots.cuda(),
                          cos_sin.cuda(), Qp, Cp, 1e-6)
    # fp32 sums of up to 1300 squares; bf16 results a unit apart where a sum rounds the other way
    tol = 2e-6 if dtype == torch.float32 else 2.0 ** -8
    for a, b in ((cq, wcq), (got, want)):
        assert float((a.cpu().float() - b.float()).norm() / b.float().norm()) < tol
    assert int((got != 0).any(-1).sum()) == 4
