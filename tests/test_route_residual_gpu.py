"""Experts chosen behind the residual step of a few rows, against the kernel that only routes."""
from types import SimpleNamespace

import pytest
import torch

from omnia_amd import ops
from omnia_amd.ops import mixers as mops

pytestmark = pytest.mark.gpu


# widths where the last threads have no columns and where all have; counts of experts up to the
# kernel's 16; every kind of choice; a row of NaN
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
    # the sums of both kernels are the same, so that experts do not depend on a step's count of rows
    assert torch.equal(route.ids, ids) and torch.equal(route.wts, wts)
    assert int(route.ids.min()) >= 0 and int(route.ids.max()) < E
    assert all(len(set(r)) == k for r in route.ids.tolist())


@pytest.mark.parametrize("rows,d,E", [(513, 2048, 8), (8, 1024, 8), (8, 4128, 8), (8, 2048, 17)])
def test_sizes_left_to_the_router(rows, d, E):
    dev, bf = "cuda", torch.bfloat16
    spec = SimpleNamespace(top=1, score="sigmoid", renorm=False, groups=1, keep=1)
    route = mops.Routing({"router": torch.zeros(E, d, dtype=bf, device=dev)}, spec)
    post = mops.RMSNorm(torch.ones(d, device=dev), d, 1e-5)
    x, m = torch.zeros(rows, d, device=dev), torch.ones(rows, d, dtype=bf, device=dev)
    h = mops.rms_residual(x, m, post, None, bf, route=route)
    assert route.ids is None and bool((h == 1).all()) and bool((x - 1).abs().max() < 1e-4)


# what a residual step sums (ptype and parts of the kernel): fp32 and fp16 slabs, a row's slots, a plain
# fp32 projection; rows of infinities and NaN choose as the kernel that only routes
@pytest.mark.parametrize("rows,d", [(5, 1056), (33, 2080)])
@pytest.mark.parametrize("E,k", [(8, 2), (7, 3), (16, 4)])
@pytest.mark.parametrize("kind", ["fp32", "fp32 slabs", "fp16 slabs", "slots"])
def test_route_of_parts(rows, d, E, k, kind):
    dev, bf = "cuda", torch.bfloat16
    g = torch.Generator().manual_seed(d + E)

    def rnd(*shape):
        return torch.randn(*shape, generator=g)

    m = {"fp32": lambda: rnd(rows, d), "fp32 slabs": lambda: rnd(3, rows, d),
         "fp16 slabs": lambda: rnd(4, rows, d).half(), "slots": lambda: rnd(rows, 2, d).to(bf)}[kind]()
    m, x0 = m.to(dev), rnd(rows, d).to(dev)
    x0[1, 17], x0[2, d - 1], x0[3, 4] = float("inf"), -float("inf"), float("nan")
    w = {"router": (rnd(E, d) * d ** -0.5).to(bf).to(dev)}
    spec = SimpleNamespace(top=k, score="sigmoid", renorm=False, groups=1, keep=1)
    post = mops.RMSNorm((rnd(d) * 0.1 + 1.0).to(dev), d, 1e-5)
    x1, x2, route = x0.clone(), x0.clone(), mops.Routing(w, spec)
    h1 = mops.rms_residual(x1, m, post, None, bf, slots=kind == "slots", route=route)
    h2 = mops.rms_residual(x2, m, post, None, bf, slots=kind == "slots")
    assert route.ids is not None
    for a, b in ((x1, x2), (h1, h2)):
        assert torch.equal(a.nan_to_num(nan=7.0), b.nan_to_num(nan=7.0))
    ids, wts = route.empty(rows, dev)
    ops.kernels().moe_route(ids, wts, h2, w["router"], k, True, False, None, 1, 1, None)
    assert torch.equal(route.ids, ids)
    assert torch.equal(route.wts.nan_to_num(nan=7.0), wts.nan_to_num(nan=7.0))
