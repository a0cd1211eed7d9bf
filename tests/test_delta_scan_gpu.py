"""The blocked delta-rule scan at the edges of its blocks, tiles and waves, against float64."""
import pytest
import torch

from omnia_amd import ops

pytestmark = pytest.mark.gpu


def exact(qn, kn, v, decay, beta, S, starts, H):
    out, S = torch.zeros_like(v), S.clone()
    rep = H // kn.shape[1]
    for s, (a, b) in enumerate(zip(starts, starts[1:])):
        for t in range(a, b):
            k, q = (x[t].repeat_interleave(rep, 0)[:, :, None] for x in (kn, qn))
            S[s] *= decay[t].exp()[:, None, None]
            u = beta[t][:, None] * (v[t] - (S[s] * k).sum(1))
            S[s] += k * u[:, None]
            out[t] = (S[s] * q).sum(1)
    return out, S


# few sequences: one group of 16 columns a block; many: two, of up to 64 key dimensions four.  Widths
# in every padding of the key dimensions, odd value widths, groups of columns that end inside a block
@pytest.mark.parametrize("lens", [[1], [16], [15, 33, 64, 1], [47, 32] + [2] * 120])
@pytest.mark.parametrize("D,V,H,KH", [(128, 128, 4, 2), (20, 29, 2, 1), (32, 16, 2, 2),
                                      (64, 40, 3, 1), (96, 72, 2, 1), (200, 48, 2, 1),
                                      (40, 61, 4, 2), (64, 64, 4, 4), (32, 128, 2, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scan(D, V, H, KH, lens, dtype):
    k = ops.kernels()
    g = torch.Generator().manual_seed(D + len(lens))

    def rnd(*shape):
        return torch.randn(*shape, generator=g)

    B, T, taps = len(lens), sum(lens), 4
    Dp, Vs, C = -(-D // 4) * 4, -(-V // 4) * 4, 2 * KH * D + H * V
    starts = [0]
    for n in lens:
        starts.append(starts[-1] + n)
    qn, kn = torch.zeros(2, T, KH, Dp)
    qn[..., :D] = torch.nn.functional.normalize(rnd(T, KH, D), dim=-1) * D ** -0.5
    kn[..., :D] = torch.nn.functional.normalize(rnd(T, KH, D), dim=-1)
    v = rnd(T, H, V).to(dtype)
    decay, beta = -torch.exp(rnd(T, H) * 0.5 - 2.0), torch.sigmoid(rnd(T, H))
    state = torch.zeros(B + 1, H, D, Vs)
    state[..., :V] = rnd(B + 1, H, D, V) * 0.1
    conv = rnd(B + 1, taps - 1, C).to(dtype)
    x = rnd(T, C + H * V + 2 * H).to(dtype)
    # slots in another order than the sequences; the last sequence starts anew, whatever its slot
    # holds
    slots = torch.arange(B, 0, -1, dtype=torch.int32)
    pos = torch.cat([torch.arange(n) + (0 if i == B - 1 else 5) for i, n in enumerate(lens)]).int()
    S0 = state[slots.long()].double()
    S0[-1] = 0.0
    want, S1 = exact(qn[..., :D].double(), kn[..., :D].double(), v.double(), decay.double(),
                     beta.double(), S0[..., :V], starts, H)
    dev = "cuda"
    o = torch.empty(T, H, Vs, device=dev)
    st, cv = state.to(dev), conv.to(dev)
    rec = torch.empty(k.delta_records(T, B, H), device=dev)
    k.delta_scan(o, st, cv, rec, qn.to(dev), kn.to(dev), v.reshape(T, H * V).to(dev),
                 decay.to(dev), beta.to(dev), x.to(dev),
                 torch.tensor(starts, dtype=torch.int32, device=dev), pos.to(dev), slots.to(dev),
                 KH, H, D, Dp, V, taps)
    st, cv = st.cpu(), cv.cpu()
    # fp32 sums of up to 256 terms: 2^-24 sqrt(256) of the terms' size, and four roundings a token
    for got, ref in ((o[..., :V].cpu().double(), want), (st[slots.long()][..., :V].double(), S1)):
        assert float((got - ref).norm() / ref.norm()) < 2e-6
    assert torch.equal(st[0], state[0])  # nobody's slot
    assert torch.equal(st[..., V:], state[..., V:])  # padding columns stay zero
    for i, n in enumerate(lens):
        old = torch.zeros(taps - 1, C, dtype=dtype) if i == B - 1 else conv[slots[i]]
        full = torch.cat([old, x[starts[i]:starts[i + 1], :C]])
        assert torch.equal(cv[slots[i]], full[-(taps - 1):])


# the shape that a step takes (few sequences: one group of columns, four waves; many: two of two)
# changes no bit of a sequence's outputs and state
@pytest.mark.parametrize("D,V,H,KH", [(24, 40, 6, 3), (24, 64, 8, 4), (64, 64, 16, 8), (96, 80, 8, 8),
                                      (128, 128, 16, 8), (200, 128, 8, 8)])
def test_sequences_beside_change_nothing(D, V, H, KH):
    k, dev = ops.kernels(), "cuda"
    n, taps, C = 77, 4, 2 * KH * D + H * V

    def run(B):
        g = torch.Generator().manual_seed(D)

        def rnd(*shape):
            return torch.randn(*shape, generator=g)

        def all_rows(t):
            return t.to(dev).repeat(B, *[1] * (t.dim() - 1))

        qn = torch.nn.functional.normalize(rnd(n, KH, D), dim=-1) * D ** -0.5
        kn = torch.nn.functional.normalize(rnd(n, KH, D), dim=-1)
        v, decay, beta = rnd(n, H * V), -torch.exp(rnd(n, H) * 0.5 - 2.0), torch.sigmoid(rnd(n, H))
        state, x = rnd(1, H, D, V) * 0.1, rnd(n, C + H * V + 2 * H)
        qn, kn, v, decay, beta, state, x = map(all_rows, (qn, kn, v, decay, beta, state, x))
        state = state.contiguous()
        conv = torch.zeros(B, taps - 1, C, device=dev)
        starts = (torch.arange(B + 1) * n).int().to(dev)
        pos = torch.arange(5, 5 + n).repeat(B).int().to(dev)
        o = torch.empty(n * B, H, V, device=dev)
        rec = torch.empty(k.delta_records(n * B, B, H), device=dev)
        k.delta_scan(o, state, conv, rec, qn, kn, v, decay, beta, x, starts, pos,
                     torch.arange(B, dtype=torch.int32, device=dev), KH, H, D, D, V, taps)
        return o, state

    (o1, s1), (o, s) = run(1), run(40)
    assert torch.equal(o.view(40, n, H, V), o1[None].expand(40, -1, -1, -1))
    assert torch.equal(s, s1.expand_as(s))
