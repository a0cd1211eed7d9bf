"""Experts chosen behind the residual step of a few rows, against the kernel that only routes."""
from types import SimpleNamespace

import pytest
import torch

from omnia_amd import ops
from omnia_amd.ops import mixers as mops

pytestmark = pytest.mark.gpu


# widths where the last threads have no columns and where all have; counts of experts around the
# kernel's two; every kind of choice; a row of NaN
@pytest.mark.parametrize("rows,d", [(1, 1056), (8, 2048), (77, 4096), (512, 2080)])
@pytest.mark.parametrize("E,k,score,renorm,groups,keep,extra", [
    (8, 2, "sigmoid", False, 1, 1, False), (6, 2, "softmax", True, 1, 1, True),
    (1, 1, "sigmoid", True, 1, 1, False), (9, 4, "softmax", False, 3, 2, False),
    (16, 4, "sigmoid", True, 4, 2, True)])
def test_route(rows, d, E, k, score, renorm, groups, keep, extra):
    dev, bf = "cuda", torch.bfloat16
    g = torch.Generator().manual_seed(d + E)

    def rnd(*shape):
        return torch.randn(*shape, generator=g)

    spec = SimpleNamespace(top=k, score=score, renorm=renorm, groups=groups, keep=keep)
    w = {"router": (rnd(E, d) * d ** -0.5).to(bf).to(dev)}
    if extra:
        w |= {"correction": rnd(E).to(dev) * 0.1, "router_b": rnd(E).to(dev)}
    post, pre = (mops.RMSNorm((rnd(d) * 0.1 + 1.0).to(dev), d, 1e-5) for _ in range(2))
    m, x0 = rnd(rows, d).to(bf).to(dev), rnd(rows, d).to(dev)
    if rows > 8:
        x0[3] = float("nan")
    x1, x2 = x0.clone(), x0.clone()
    route = mops.Routing(w, spec)
    h1 = mops.rms_residual(x1, m, post, pre, bf, route=route)
    h2 = mops.rms_residual(x2, m, post, pre, bf)
    assert torch.equal(x1.nan_to_num(), x2.nan_to_num())
    assert torch.equal(h1.nan_to_num(), h2.nan_to_num()) and route.ids is not None
    ids, wts = route.empty(rows, dev)
    ops.kernels().moe_route(ids, wts, h2, w["router"], k, score == "sigmoid", renorm,
                            w.get("correction"), groups, keep, w.get("router_b"))
    # fp32 sums of d products in two orders: some 2^-24 sqrt(d) of logits of about one.  Where the
    # choice lies that close, either is right
    close = (route.wts - wts).abs().amax(1) <= 2e-5
    same = (route.ids == ids).all(1)
    assert bool((same & close)[torch.arange(rows, device=dev) != 3].float().mean() >= 0.99)
    assert int(route.ids.min()) >= 0 and int(route.ids.max()) < E
    assert all(len(set(r)) == k for r in route.ids.tolist())


@pytest.mark.parametrize("rows,d,E", [(513, 2048, 8), (8, 1024, 8), (8, 4128, 8), (8, 2048, 17),
                                      (257, 2016, 9)])
def test_sizes_left_to_the_router(rows, d, E):
    dev, bf = "cuda", torch.bfloat16
    spec = SimpleNamespace(top=1, score="sigmoid", renorm=False, groups=1, keep=1)
    route = mops.Routing({"router": torch.zeros(E, d, dtype=bf, device=dev)}, spec)
    post = mops.RMSNorm(torch.ones(d, device=dev), d, 1e-5)
    x, m = torch.zeros(rows, d, device=dev), torch.ones(rows, d, dtype=bf, device=dev)
    h = mops.rms_residual(x, m, post, None, bf, route=route)
    assert route.ids is None and bool((h == 1).all()) and bool((x - 1).abs().max() < 1e-4)
