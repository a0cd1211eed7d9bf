"""Preparation and block records of the delta rule in one launch against the kernels they stand for."""
import pytest
import torch

from omnia_amd import ops

pytestmark = pytest.mark.gpu


def inputs(lens, D, V, KH, H, taps, dtype):
    g = torch.Generator().manual_seed(D + len(lens))
    B, T, C = len(lens), sum(lens), 2 * KH * D + H * V
    width = C + H * V + 2 * H

    def rnd(*shape):
        return torch.randn(*shape, generator=g)

    x = rnd(T, width + (-width % 8) + 8).to(dtype).cuda()[:, :width]
    conv_w, conv = (rnd(C, taps) * 0.5).to(dtype).cuda(), rnd(B + 1, taps - 1, C).to(dtype).cuda()
    a_log, dt_bias = (rnd(H) * 0.5 + 1.0).cuda(), (rnd(H) - 3.0).cuda()
    starts = torch.tensor([0] + lens).cumsum(0).int().cuda()
    # slots in another order than the sequences; one starts anew, one is padding
    slots = torch.arange(B, 0, -1, dtype=torch.int32)
    pos = torch.cat([torch.arange(n) + (0 if i == B - 1 else 5) for i, n in enumerate(lens)]).int()
    if B > 2:
        slots[1] = -1
    return x, conv_w, conv, a_log, dt_bias, starts, pos.cuda(), slots.cuda()


# ends inside, at and past a record and its runs of four, sequences shorter than the taps, none;
# widths under, at and off a wave's 128 channels; strided input rows
@pytest.mark.parametrize("lens", [[1], [16, 4, 21], [2, 0, 47, 3, 64, 1], [333] * 3,
                                  [16] * 32, [1264]])
@pytest.mark.parametrize("D,V,KH,H,taps", [(128, 128, 8, 16, 4), (128, 96, 2, 2, 4), (20, 30, 1, 2, 3),
                                           (64, 128, 2, 4, 2), (126, 6, 1, 1, 4)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_prep_blocks(lens, D, V, KH, H, taps, dtype):
    k, dev = ops.kernels(), "cuda"
    x, conv_w, conv, a_log, dt_bias, starts, pos, slots = inputs(lens, D, V, KH, H, taps, dtype)
    B, T, Dp, Vs = len(lens), sum(lens), -(-D // 4) * 4, -(-V // 4) * 4
    S0 = torch.randn(B + 1, H, D, Vs, device=dev) * 0.1
    res = []
    for one in (False, True):
        qn, kn = (torch.full((T, KH, Dp), float("nan"), device=dev) for _ in range(2))
        vc = torch.empty(T, H * V, dtype=dtype, device=dev)
        decay, beta = (torch.empty(T, H, device=dev) for _ in range(2))
        rec = torch.zeros(k.delta_records(T, B, H), device=dev)
        o, S, c = torch.zeros(T, H, Vs, device=dev), S0.clone(), conv.clone()
        if one:
            assert k.delta_prep_blocks(rec, qn, kn, vc, x, conv_w, c, a_log, dt_bias, starts, pos,
                                       slots, KH, H, D, Dp, V, taps)
            assert torch.equal(c, conv)
            decay = beta = None
        else:
            k.delta_prep(qn, kn, vc, decay, beta, x, conv_w, c, a_log, dt_bias, starts, pos, slots,
                         KH, H, D, Dp, V, taps)
        k.delta_scan(o, S, c, rec, qn, kn, vc, decay, beta, x, starts, pos, slots, KH, H, D, Dp, V,
                     taps)
        res.append((qn, kn, vc, rec, o, S, c))
    for a, b in zip(*res[:2]):
        assert torch.equal(a, b)  # which kernel prepares a step changes no bit


@pytest.mark.parametrize("D,V,KH,H,taps", [(130, 64, 1, 1, 4), (64, 130, 1, 1, 4), (63, 64, 1, 1, 4),
                                           (64, 64, 1, 4, 4), (64, 64, 1, 1, 5), (64, 64, 1, 1, 1),
                                           (64, 64, 8, 16, 4)])
def test_not_covered(D, V, KH, H, taps):
    T = 2000 if KH == 8 else 8
    x, conv_w, conv, a_log, dt_bias, starts, pos, slots = inputs([T], D, V, KH, H, taps,
                                                                 torch.float32)
    k, dev, Dp = ops.kernels(), "cuda", -(-D // 4) * 4
    qn, kn = (torch.empty(T, KH, Dp, device=dev) for _ in range(2))
    assert not k.delta_prep_blocks(torch.empty(k.delta_records(T, 1, H), device=dev), qn, kn,
                                   torch.empty(T, H * V, device=dev), x, conv_w, conv, a_log,
                                   dt_bias, starts, pos, slots, KH, H, D, Dp, V, taps)
