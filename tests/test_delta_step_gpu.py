"""Decode of the delta rule in one launch against the kernels it stands for."""
import pytest
import torch

from omnia_amd import ops

pytestmark = pytest.mark.gpu


# one and two heads a key head; widths under, at and off a wave's 128 channels, states of 4, 8 and 16
# rows a thread; rows that start anew and padded ones (slot -1), strided input rows
@pytest.mark.parametrize("T", [1, 5, 64])
@pytest.mark.parametrize("D,V,KH,H,taps", [(128, 128, 8, 16, 4), (128, 128, 2, 2, 4),
                                           (20, 30, 1, 2, 3), (64, 128, 2, 4, 2), (96, 80, 2, 2, 3),
                                           (126, 6, 1, 1, 4), (128, 124, 1, 2, 4)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_step(T, D, V, KH, H, taps, dtype):
    k, dev = ops.kernels(), "cuda"
    g = torch.Generator().manual_seed(T + D)

    def rnd(*shape):
        return torch.randn(*shape, generator=g)

    C, Dp, Vs = 2 * KH * D + H * V, -(-D // 4) * 4, -(-V // 4) * 4
    Vp, n = -(-V // 8) * 8, T + 2
    width = C + H * V + 2 * H
    x = rnd(T, width + (-width % 8) + 8).to(dtype).to(dev)[:, :width]
    conv_w = (rnd(C, taps) * 0.5).to(dtype).to(dev)
    a_log, dt_bias, norm = (t.to(dev) for t in (rnd(H) * 0.5 + 1.0, rnd(H) - 3.0, rnd(V) + 2.0))
    state, conv = (rnd(n, H, D, Vs) * 0.1).to(dev), rnd(n, taps - 1, C).to(dtype).to(dev)
    slots = torch.randperm(n, generator=g)[:T].int()
    pos = torch.randint(1, 50, (T,), generator=g).int()
    if T > 2:
        slots[1], pos[2] = -1, 0
    slots, pos = slots.to(dev), pos.to(dev)

    s1, c1 = state.clone(), conv.clone()
    qn, kn = (torch.empty(T, KH, Dp, device=dev) for _ in range(2))
    vc = torch.empty(T, H * V, dtype=dtype, device=dev)
    decay, beta = (torch.empty(T, H, device=dev) for _ in range(2))
    want = torch.empty(T, H * Vp, dtype=dtype, device=dev)
    k.delta_prep(qn, kn, vc, decay, beta, x, conv_w, c1, a_log, dt_bias, None, pos, slots, KH, H,
                 D, Dp, V, taps)
    k.delta_step(want, s1, c1, qn, kn, vc, decay, beta, x, norm, pos, slots, KH, H, D, Dp, V, Vp,
                 taps, 1e-6)

    s2, c2, got = state.clone(), conv.clone(), torch.empty_like(want)
    assert k.delta_step_conv(got, s2, c2, x, conv_w, a_log, dt_bias, norm, pos, slots, KH, H, D, V,
                             Vp, taps, 1e-6)
    assert torch.equal(c1, c2)
    # which of them a step takes changes no bit
    assert torch.equal(s1, s2) and torch.equal(want, got)


@pytest.mark.parametrize("T,D,V,KH,H,taps", [
    (1, 130, 64, 1, 1, 4), (1, 64, 130, 1, 1, 4), (1, 63, 64, 1, 1, 4), (1, 64, 64, 1, 3, 4),
    (1, 64, 64, 1, 1, 5), (1, 64, 1028, 1, 1, 4), (1, 20, 30, 1, 4, 3), (64, 128, 124, 1, 4, 4),
    (97, 128, 64, 8, 16, 4), (112, 64, 128, 8, 16, 4)])
def test_sizes_left_to_the_two_kernels(T, D, V, KH, H, taps):
    k, dev = ops.kernels(), "cuda"
    C, Vs, Vp = 2 * KH * D + H * V, -(-V // 4) * 4, -(-V // 8) * 8
    f = lambda *s: torch.zeros(*s, device=dev)  # noqa: E731
    i = torch.zeros(T, dtype=torch.int32, device=dev)
    assert not k.delta_step_conv(f(T, H * Vp), f(T, H, D, Vs), f(T, taps - 1, C),
                                 f(T, C + H * V + 2 * H), f(C, taps), f(H), f(H), f(V), i, i, KH,
                                 H, D, V, Vp, taps, 1e-6)
