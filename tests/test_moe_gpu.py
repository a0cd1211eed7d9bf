"""MoE kernels (K14) vs the fp32 oracle; Mixtral engine on the GPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from omnia_amd import ops
from omnia_amd.ops import reference as ref


def _weights(E, d, I, g, dev="cuda"):
    wgu = (torch.randn(E, 2 * I, d, generator=g) * 0.05).to(torch.bfloat16)
    wd = (torch.randn(E, d, I, generator=g) * 0.05).to(torch.bfloat16)
    router = (torch.randn(E, d, generator=g) * 0.2).to(torch.bfloat16)
    return router.to(dev), wgu.to(dev), wd.to(dev)


@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (37, 8, 2), (256, 8, 2), (64, 16, 4)])
def test_moe_topk_matches_reference(T, E, k):
    g = torch.Generator().manual_seed(T * E)
    logits = torch.randn(T, E, generator=g)
    ids = torch.empty(T, k, dtype=torch.int32, device="cuda")
    w = torch.empty(T, k, dtype=torch.float32, device="cuda")
    ops.kernels().moe_topk(ids, w, logits.cuda(), k, True)
    rid, rw = ref.moe_route(logits, k)
    assert torch.equal(ids.cpu(), rid)
    torch.testing.assert_close(w.cpu(), rw, atol=1e-5, rtol=1e-5)


def test_moe_topk_nan_and_padding_rows_route_to_valid_distinct_experts():
    """A NaN row (e.g. a padded decode row) or an all -inf row must still yield k
    distinct ids in [0, E) and finite weights: the expert-parallel dispatch turns
    ids into send-buffer slots, so a -1 there would be an out-of-bounds write."""
    E, k = 8, 2
    logits = torch.randn(6, E)
    logits[1] = float("nan")
    logits[2] = float("-inf")
    logits[3, :5] = float("nan")  # partially NaN: the finite experts win
    ids = torch.full((6, k), -7, dtype=torch.int32, device="cuda")
    w = torch.empty(6, k, dtype=torch.float32, device="cuda")
    ops.kernels().moe_topk(ids, w, logits.cuda(), k, True)
    ids, w = ids.cpu(), w.cpu()
    assert ((ids >= 0) & (ids < E)).all() and (ids[:, 0] != ids[:, 1]).all()
    assert torch.isfinite(w).all()
    assert set(ids[3].tolist()) <= {5, 6, 7}
    torch.testing.assert_close(w[1], torch.full((k,), 1.0 / k))
    rid, rw = ref.moe_route(logits[[0, 4, 5]], k)
    assert torch.equal(ids[[0, 4, 5]], rid)


@pytest.mark.parametrize("T,d,I,E,k,e_lo,e_n", [
    (1, 256, 256, 8, 2, 0, 8), (13, 512, 256, 8, 2, 0, 8), (256, 512, 512, 8, 2, 0, 8),
    (100, 256, 256, 8, 2, 4, 4),  # expert-parallel shard: experts 4..7 only
])
def test_moe_grouped_path_matches_reference(T, d, I, E, k, e_lo, e_n):
    g = torch.Generator().manual_seed(T + d)
    router, wgu, wd = _weights(E, d, I, g)
    x = (torch.randn(T, d, generator=g)).to(torch.bfloat16).cuda()
    wgu_l, wd_l = wgu[e_lo:e_lo + e_n].contiguous(), wd[e_lo:e_lo + e_n].contiguous()
    out = ops.moe(x, router, wgu_l, wd_l, k, E, e_lo, graph_safe=True)
    # pin the oracle to the kernel's routing (bf16 router logits, as in ops.moe)
    logits = torch.nn.functional.linear(x, router)
    ids = torch.empty(T, k, dtype=torch.int32, device="cuda")
    w = torch.empty(T, k, dtype=torch.float32, device="cuda")
    ops.kernels().moe_topk(ids, w, logits, k, True)
    rid, rw = ref.moe_route(logits.float().cpu(), k)
    assert torch.equal(ids.cpu(), rid)
    exp = ref.moe(x.cpu(), router.cpu(), wgu_l.cpu(), wd_l.cpu(), k, e_lo, ids=rid, wts=rw,
                  act_dtype=torch.bfloat16)
    torch.testing.assert_close(out.float().cpu(), exp, atol=1e-2, rtol=1e-2)


def test_moe_library_path_matches_grouped(monkeypatch):
    g = torch.Generator().manual_seed(5)
    E, d, I, k, T = 4, 256, 512, 2, 2048
    router, wgu, wd = _weights(E, d, I, g)
    x = torch.randn(T, d, generator=g).to(torch.bfloat16).cuda()
    monkeypatch.setattr(ops, "MOE_TILE256_ROWS", 1 << 30)  # the 64-row grouped kernels
    a = ops.moe(x, router, wgu, wd, k, E, 0, graph_safe=True)
    monkeypatch.setenv("OMNIA_MOE_LIBRARY", "1")
    b = ops.moe(x, router, wgu, wd, k, E, 0, graph_safe=False)  # hipBLASLt per expert
    torch.testing.assert_close(a.float(), b.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("T,d,I,E,k,e_lo,e_n", [
    (2048, 512, 512, 8, 2, 0, 8),    # prefill-sized: 256x256-tile grouped GEMMs
    (2500, 256, 384, 8, 2, 0, 8),    # ragged expert segments, I not a multiple of 256
    (4096, 512, 256, 8, 2, 4, 4),    # expert-parallel shard: experts 4..7 only
    (897, 256, 256, 8, 2, 0, 8),     # from 224 rows an expert, segments not full
    (4097, 512, 128, 64, 2, 0, 64),  # from 128 where the down product has 128 tiles
])
def test_moe_tile256_prefill_matches_reference(T, d, I, E, k, e_lo, e_n):
    """Large batches run the 256-row-segment grouped GEMMs (pgemm.hip EPI 5 / 6)
    without a host sync: against the fp32 oracle pinned to the kernel's routing,
    and against the 64-row grouped kernels (a different tiling of the same sums)."""
    g = torch.Generator().manual_seed(T + I)
    router, wgu, wd = _weights(E, d, I, g)
    x = (torch.randn(T, d, generator=g)).to(torch.bfloat16).cuda()
    wgu_l, wd_l = wgu[e_lo:e_lo + e_n].contiguous(), wd[e_lo:e_lo + e_n].contiguous()
    assert T * k >= ops.moe_tile_rows(e_n, d) * E  # the 256-tile path is the one under test
    out = ops.moe(x, router, wgu_l, wd_l, k, E, e_lo, graph_safe=True)
    logits = torch.nn.functional.linear(x, router)
    rid, rw = ref.moe_route(logits.float().cpu(), k)
    exp = ref.moe(x.cpu(), router.cpu(), wgu_l.cpu(), wd_l.cpu(), k, e_lo, ids=rid, wts=rw,
                  act_dtype=torch.bfloat16)
    torch.testing.assert_close(out.float().cpu(), exp, atol=1e-2, rtol=1e-2)
    saved = ops.MOE_TILE256_ROWS
    try:
        ops.MOE_TILE256_ROWS = 1 << 30
        small = ops.moe(x, router, wgu_l, wd_l, k, E, e_lo, graph_safe=True)
    finally:
        ops.MOE_TILE256_ROWS = saved
    torch.testing.assert_close(out.float(), small.float(), atol=1e-2, rtol=1e-2)
    # negative control: dropping the routing weights must not pass
    assert not torch.allclose(out.float().cpu(), exp * 2, atol=1e-2, rtol=1e-2)


def test_moe_tile256_is_graph_capturable():
    """No host sync: the prefill-sized grouped path captures into a hipGraph and
    replays to the eager result."""
    g = torch.Generator().manual_seed(11)
    E, d, I, k, T = 8, 512, 512, 2, 2048
    router, wgu, wd = _weights(E, d, I, g)
    x = torch.randn(T, d, generator=g).to(torch.bfloat16).cuda()
    want = ops.moe(x, router, wgu, wd, k, E, 0, graph_safe=True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.moe(x, router, wgu, wd, k, E, 0, graph_safe=True)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.moe(x, router, wgu, wd, k, E, 0, graph_safe=True)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_mixtral_engine_graphs_match_eager():
    from omnia_amd.engine.engine import EngineConfig, LLMEngine
    from omnia_amd.engine.sampling_params import SamplingParams

    def run(graphs):
        e = LLMEngine(EngineConfig(model="tiny-mixtral", device="cuda", num_blocks=128,
                                   max_batch=8, max_model_len=1024, use_graphs=graphs))
        p = SamplingParams(temperature=0, max_tokens=10, ignore_eos=True)
        return [s.output for s in e.generate([list(range(3, 90)), list(range(40, 60))], p)]

    assert run(True) == run(False)


def test_moe_decode_layer_bandwidth_report():
    """Mixtral-8x7B-shaped MoE layer at decode batch 256 (prints achieved HBM rate)."""
    g = torch.Generator(device="cuda").manual_seed(0)
    E, d, I, k, T = 8, 4096, 14336, 2, 256
    router = (torch.randn(E, d, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    wgu = (torch.randn(E, 2 * I, d, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    wd = (torch.randn(E, d, I, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    x = torch.randn(T, d, device="cuda", generator=g).to(torch.bfloat16)
    for _ in range(3):
        ops.moe(x, router, wgu, wd, k, E)
    torch.cuda.synchronize()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    n = 10
    for _ in range(n):
        ops.moe(x, router, wgu, wd, k, E)
    e.record()
    torch.cuda.synchronize()
    ms = s.elapsed_time(e) / n
    gb = (wgu.numel() + wd.numel()) * 2 / 1e9
    print(f"\nMoE decode layer T={T}: {ms:.3f} ms, weights {gb:.2f} GB -> {gb / ms:.2f} TB/s")
    assert ms > 0


@pytest.mark.parametrize("T,d,E,k", [(1, 4096, 8, 2), (333, 4096, 8, 2), (4096, 1024, 16, 4),
                                     (64, 512, 64, 6)])
def test_router_topk_fused_matches_linear_then_topk(T, d, E, k):
    """The fused router GEMM + top-k (no logits tensor, no library GEMM) routes
    like bf16 F.linear followed by moe_topk -- up to bf16 rounding ties of the
    logits, which may order near-equal experts differently (<= 0.5 % of rows
    against the library GEMM; 2-6 % against fp32 at E=16-64, k=4-6)."""
    g = torch.Generator().manual_seed(T * E + d)
    x = torch.randn(T, d, generator=g).to(torch.bfloat16).cuda()
    router = (torch.randn(E, d, generator=g) * 0.02).to(torch.bfloat16).cuda()
    ids = torch.empty(T, k, dtype=torch.int32, device="cuda")
    w = torch.empty(T, k, dtype=torch.float32, device="cuda")
    ops.kernels().moe_router_topk(ids, w, x, router, k, True)
    ids2 = torch.empty_like(ids)
    w2 = torch.empty_like(w)
    ops.kernels().moe_topk(ids2, w2, torch.nn.functional.linear(x, router), k, True)
    same = (ids == ids2).all(1)
    assert same.float().mean().item() >= 0.995, same.float().mean().item()
    torch.testing.assert_close(w[same], w2[same], atol=1e-2, rtol=1e-2)
    # against the fp32 oracle: every chosen expert's fp32 logit, in the kernel's
    # order, equals the fp32 top-k value at that rank up to bf16 rounding (the
    # kernel, like the library GEMM, rounds logits to bf16, so near-ties may swap)
    lf = torch.nn.functional.linear(x.float(), router.float()).cpu()
    rid, rw = ref.moe_route(lf, k)
    sel = lf.gather(1, ids.cpu().long())
    top = lf.topk(k, dim=1).values
    tol = 2.0 ** -7 * lf.abs().amax(1, keepdim=True)
    assert ((sel - top).abs() <= tol).all()
    m = (ids.cpu() == rid).all(1)  # rows whose order no near-tie swapped
    assert m.float().mean().item() >= 0.9
    torch.testing.assert_close(w.cpu()[m], rw[m], atol=1e-2, rtol=1e-2)


def _spied(monkeypatch):
    """Names of the expert kernels that run from here on."""
    used, native = [], ops.kernels()

    class Spy:
        def __getattr__(self, name):
            f = getattr(native, name)
            if not name.endswith(("_moe", "moe_gemm")):
                return f
            return lambda *a: (used.append(name), f(*a))[1]

    monkeypatch.setattr(ops, "kernels", Spy)
    return used


@pytest.mark.parametrize("T,kernel", [(1, "stream_moe"), (64, "moe_gemm"), (300, "panel_moe"),
                                      (2000, "pgemm_moe")])
def test_a_shard_counts_its_rows_over_all_experts(T, kernel, monkeypatch):
    """The kernel of a shard's experts follows the rows an expert has, which are those of all
    assignments over all experts: one expert of eight takes the one that eight take."""
    d, E, k = 256, 8, 2
    g = torch.Generator().manual_seed(T)
    router, wgu, wd = _weights(E, d, 256, g)
    x = torch.randn(T, d, generator=g).to(torch.bfloat16).cuda()
    used = _spied(monkeypatch)
    whole = ops.moe(x, router, wgu, wd, k, E).float()
    of_whole, used[:] = set(used), []
    parts = [ops.moe(x, router, wgu[e:e + 1].contiguous(), wd[e:e + 1].contiguous(), k, E, e)
             for e in range(E)]
    assert of_whole == set(used) == {kernel}
    # the shards' sums round to bf16 one by one
    torch.testing.assert_close(sum(p.float() for p in parts), whole, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("T,kernel", [(1, "stream_moe"), (300, "moe_gemm"), (2000, "moe_gemm")])
def test_ranks_that_share_a_device_take_blocks_of_little_lds(T, kernel, monkeypatch):
    """Ranks on one device spin in all-reduce blocks beside this rank's: no tile or panel blocks.
    The model asks for it wherever its ranks share a device."""
    from types import SimpleNamespace

    from omnia_amd.models import mixtral

    d, E, k = 256, 8, 2
    g = torch.Generator().manual_seed(T)
    router, wgu, wd = _weights(E, d, 256, g)
    x = torch.randn(T, d, generator=g).to(torch.bfloat16).cuda()
    want = ops.moe(x, router, wgu, wd, k, E).float()
    used = _spied(monkeypatch)
    monkeypatch.setattr(mixtral.pstate, "ranks_per_device", lambda: 2)
    m = SimpleNamespace(ep_mode="tp", tp=2, e_lo=0, graph_safe=True,
                        cfg=SimpleNamespace(experts_per_token=k, num_experts=E))
    got = mixtral.MixtralModel.mlp(
        m, {"router": router, "experts_gate_up": wgu, "experts_down": wd}, x).float()
    assert set(used) == {kernel}
    torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("E,rows", [
    (20, [1, 127, 128, 129, 255, 256, 257, 300, 383, 384, 385, 512, 513, 0, 2, 0, 130, 640, 3, 250]),
    (9, [300, 300, 300, 300, 300, 300, 300, 300, 300]),  # an expert's last segment: 44 rows
    (4, [90, 120, 7, 128]),                              # light segments alone
    (4, [256, 512, 256, 200]),                           # none
    (100, [40 + 3 * e for e in range(100)]),             # more than a word of segments
    (200, [200 + e for e in range(200)])])               # more than are put in order
def test_segments_of_few_rows(E, rows):
    """Segments of 128 rows or fewer run as half a tile behind the others: the bits of the narrow
    tile, which knows no such segments, in every product."""
    kk, dev, d, I = ops.kernels(), "cuda", 256, 384
    g = torch.Generator().manual_seed(E)
    n = sum(rows)
    ids = torch.arange(E).repeat_interleave(torch.tensor(rows))[torch.randperm(n, generator=g)]
    ids = ids.int().view(n, 1).to(dev)
    x = torch.randn(n, d, generator=g).to(torch.bfloat16).to(dev)
    up = (torch.randn(E, 2 * I, d, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    down = (torch.randn(E, d, I, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    wts = torch.rand(n, generator=g).to(dev)
    mb = kk.moe_max_blocks(n, E, 256)
    order = torch.empty(mb * 256, dtype=torch.int32, device=dev)
    blk = torch.empty(mb, dtype=torch.int32, device=dev)
    nb = torch.empty(1, dtype=torch.int32, device=dev)
    kk.moe_align(order, blk, nb, ids, E, 0, E)
    live = (order < n) & (torch.arange(mb * 256, device=dev) < nb * 256)
    for mode, w, rw in ((0, up, None), (2, up, wts), (3, up[:, :I].contiguous(), None)):
        acts = []
        for cols in (256, 128):
            if w.shape[1] // (1 if mode == 3 else 2) % (cols // (1 if mode == 3 else 2)):
                continue
            act = torch.zeros(mb * 256, w.shape[1] // (1 if mode == 3 else 2), device=dev,
                              dtype=torch.bfloat16)
            kk.pgemm_moe(mode, act, x, w, order, blk, nb, rw, 1, n, 0, 1.702, 7.0, cols)
            acts.append(act[live])
        assert len(acts) == 1 or torch.equal(*acts)
        if mode != 0:
            continue
        y = torch.empty(2, n, d, device=dev, dtype=torch.bfloat16)
        for i, cols in enumerate((256, 128)):
            kk.pgemm_moe(1, y[i], act, down, order, blk, nb, wts, 1, n, 0, 0.0, 0.0, cols)
        assert torch.equal(y[0], y[1])
        for e in set(range(E)) if E <= 20 else {0, E // 2, E - 1}:
            of = ids.view(-1) == e
            a, b = (x[of].float() @ up[e].float().t()).split(I, 1)
            want = (torch.nn.functional.silu(a) * b) @ down[e].float().t() * wts[of, None]
            torch.testing.assert_close(y[0][of].float(), want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("rows", [[300, 5, 700], [0, 1, 256], [5376] * 4, [5632] * 4])
def test_column_tiles_that_walk_k_in_orders_of_their_own(rows):
    """Experts of 4 KB rows, 9 wide column tiles (two octets): tiles wide, narrow, cut in two and of
    half height take the K-tiles in the same order, each once, of less than a round, three and more."""
    kk, dev, E, d, I = ops.kernels(), "cuda", len(rows), 2048, 1152
    n = sum(rows)
    ids = torch.arange(E).repeat_interleave(torch.tensor(rows)).int().view(n, 1).to(dev)
    x = torch.randn(n, d, device=dev).to(torch.bfloat16)
    up = (torch.randn(E, 2 * I, d, device=dev) * 0.02).to(torch.bfloat16)
    wts = torch.rand(n, device=dev)
    mb = kk.moe_max_blocks(n, E, 256)
    order = torch.empty(mb * 256, dtype=torch.int32, device=dev)
    blk = torch.empty(mb, dtype=torch.int32, device=dev)
    nb = torch.empty(1, dtype=torch.int32, device=dev)
    kk.moe_align(order, blk, nb, ids, E, 0, E)
    live = (order < n) & (torch.arange(mb * 256, device=dev) < nb * 256)
    for mode, w, rw in ((0, up, None), (2, up, wts), (3, up[:, :I - 128].contiguous(), None)):
        out = w.shape[1] // (1 if mode == 3 else 2)
        acts = [torch.zeros(mb * 256, out, device=dev, dtype=torch.bfloat16) for _ in range(2)]
        for act, cols in zip(acts, (256, 128)):
            kk.pgemm_moe(mode, act, x, w, order, blk, nb, rw, 1, n, 0, 1.702, 7.0, cols)
        assert torch.equal(*(a[live] for a in acts))
        if mode:
            continue
        for e in (e for e in range(E) if rows[e]):
            of = ids.view(-1) == e
            a, b = (x[of][:64].float() @ up[e].float().t()).split(I, 1)
            got = torch.empty(n, I, device=dev)
            got[order[live].long()] = acts[0][live].float()
            torch.testing.assert_close(got[of][:64], torch.nn.functional.silu(a) * b,
                                       atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("rows", [[1100] * 4, [2300, 0, 2700, 300]])
@pytest.mark.parametrize("K,N", [(384, 2048), (1152, 1792), (4224, 2048)])
def test_experts_wide_tiles_left_whole(rows, K, N):
    """More than 128 wide tiles are not all cut, over rings that turn often: the bits of the narrow tile, and against 64 bits the roundings of K sums, of at most 2^-24 of the sum of
    magnitudes, and of the result to bf16."""
    kk, dev, E, n = ops.kernels(), "cuda", len(rows), sum(rows)
    ids = torch.arange(E).repeat_interleave(torch.tensor(rows)).int().view(n, 1).to(dev)
    x = torch.randn(n, K, device=dev).to(torch.bfloat16)
    up = (torch.randn(E, 2 * N, K, device=dev) * 0.05).to(torch.bfloat16)
    wts = torch.rand(n, device=dev)
    mb = kk.moe_max_blocks(n, E, 256)
    order = torch.empty(mb * 256, dtype=torch.int32, device=dev)
    blk = torch.empty(mb, dtype=torch.int32, device=dev)
    nb = torch.empty(1, dtype=torch.int32, device=dev)
    kk.moe_align(order, blk, nb, ids, E, 0, E)
    live = (order < n) & (torch.arange(mb * 256, device=dev) < nb * 256)
    at = order[live].long()
    rowed = torch.zeros(mb * 256, K, device=dev, dtype=torch.bfloat16)  # down: rows in sorted order
    rowed[live] = x[at]
    for mode in (0, 1, 2, 3):
        w = up if mode in (0, 2) else up[:, :N].contiguous()
        tiles = nb.item() * (N // (128 if mode in (0, 2) else 256))
        assert tiles > 128
        res = []
        for cols in (256, 128):
            act = torch.zeros(n if mode == 1 else mb * 256, N, device=dev, dtype=torch.bfloat16)
            kk.pgemm_moe(mode, act, rowed if mode == 1 else x, w, order, blk, nb,
                         wts if mode in (1, 2) else None, 1, n, 0, 1.702, 7.0, cols)
            if mode != 1:
                got = torch.zeros(n, N, device=dev, dtype=torch.bfloat16)
                got[at] = act[live]
                act = got
            res.append(act)
        assert torch.equal(*res)
        if mode > 1:
            continue
        for e in (e for e in range(E) if rows[e]):
            of = (ids.view(-1) == e).nonzero().view(-1)[::7]
            parts = [(x[of].double() @ h.double().t(),
                      K * 2.0 ** -24 * (x[of].double().abs() @ h.double().abs().t()))
                     for h in w[e].chunk(1 if mode else 2)]
            if mode:
                want, bound = (t * wts[of, None].double() for t in parts[0])
            else:
                (g, dg), (u, du) = parts
                want = torch.nn.functional.silu(g) * u
                bound = 1.2 * (dg * (u.abs() + du) + g.abs() * du) + 1e-5 * g.abs() * u.abs()
            err = (res[0][of].double() - want).abs()
            assert (err <= bound + 2.0 ** -8 * want.abs()).all()


@pytest.mark.parametrize("cols", [256, 128])
def test_an_experts_rows_bits_are_their_own(cols):
    """Experts of 4 KB rows: a row's bits follow neither the rows beside it, in steps of 9 tiles to more
    than three rounds, nor the experts that are there."""
    kk, dev, E, d, I, most = ops.kernels(), "cuda", 4, 2048, 1152, 5632
    x = torch.randn(E, most, d, device=dev).to(torch.bfloat16)
    up = (torch.randn(E, 2 * I, d, device=dev) * 0.02).to(torch.bfloat16)
    wts = torch.rand(E, most, device=dev)

    def run(mode, rows, lo=0, hi=E):
        """{expert: its rows' activations} of the first rows[e] tokens of each expert."""
        n = sum(rows)
        ids = torch.arange(E).repeat_interleave(torch.tensor(rows)).int().view(n, 1).to(dev)
        rw = torch.cat([w[:r] for w, r in zip(wts, rows)]) if mode == 2 else None
        mb = kk.moe_max_blocks(n, E, 256)
        order = torch.empty(mb * 256, dtype=torch.int32, device=dev)
        blk = torch.empty(mb, dtype=torch.int32, device=dev)
        nb = torch.empty(1, dtype=torch.int32, device=dev)
        kk.moe_align(order, blk, nb, ids, E, lo, hi)
        w = up[lo:hi] if mode != 3 else up[lo:hi, :I - 128].contiguous()
        act = torch.zeros(mb * 256, w.shape[1] // (1 if mode == 3 else 2), device=dev,
                          dtype=torch.bfloat16)
        kk.pgemm_moe(mode, act, torch.cat([t[:r] for t, r in zip(x, rows)]), w, order, blk, nb, rw, 1,
                     n, lo, 1.702, 7.0, cols)
        live = (order < n) & (torch.arange(mb * 256, device=dev) < nb * 256)
        got = torch.zeros(n, act.shape[1], device=dev, dtype=act.dtype)
        got[order[live].long()] = act[live]
        return {e: t for e, t in enumerate(got.split(rows)) if lo <= e < hi}

    for mode in (0, 2, 3):
        whole = run(mode, [most] * E)  # 88 segments of 9 (of mode 3: 4) wide column tiles
        for rows, lo, hi in (([300, 5, 700, 1], 0, E), ([0, 0, 1, 0], 0, E), ([3000] * E, 0, E),
                             ([300, 5, 700, 1], 2, 4), ([most] * E, 1, 3)):
            for e, got in run(mode, rows, lo, hi).items():
                assert torch.equal(got, whole[e][:rows[e]]), (mode, rows, lo, e)


def test_segments_of_few_rows_take_no_longer_than_full_ones():
    """Apart from their expert's others, light segments read its weights once more, so many of them
    stay where they are: 8 light segments of 24 against 24 full ones (1.26 times as long apart)."""
    kk, dev, E, d, I = ops.kernels(), "cuda", 8, 4096, 4096
    up = [torch.randn(E, 2 * I, d, device=dev, dtype=torch.bfloat16) * 0.02 for _ in range(2)]
    runs = {}
    for rows in (600, 768):
        n = E * rows
        ids = torch.arange(E, dtype=torch.int32, device=dev).repeat(rows).view(n, 1)
        x = torch.randn(n, d, device=dev).to(torch.bfloat16)
        mb = kk.moe_max_blocks(n, E, 256)
        order = torch.empty(mb * 256, dtype=torch.int32, device=dev)
        blk = torch.empty(mb, dtype=torch.int32, device=dev)
        nb = torch.empty(1, dtype=torch.int32, device=dev)
        kk.moe_align(order, blk, nb, ids, E, 0, E)
        assert nb.item() == 24
        act = torch.empty(mb * 256, I, device=dev, dtype=torch.bfloat16)
        runs[rows] = lambda w, a=(x, order, blk, nb, n, act): kk.pgemm_moe(
            0, a[5], a[0], w, *a[1:4], None, 1, a[4], 0)
    best = {}
    for _ in range(12):
        for rows, run in runs.items():
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for w in up * 3:
                run(w)
            b.record()
            torch.cuda.synchronize()
            best[rows] = min(best.get(rows, 1e9), a.elapsed_time(b))
    assert best[600] < 1.1 * best[768], best
