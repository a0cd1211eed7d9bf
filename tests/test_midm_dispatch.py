"""Mid-size step dispatch (ops.midm_config, ops/tuned/midm_mi355x.json): bucket
mapping, the decode / prefill-tile boundaries, mode-1 (gate_up) unsplit
entries, and the OMNIA_MIDM kill switch -- pure table logic, CPU."""
import json
import os

import pytest
import torch

from omnia_amd import ops
from omnia_amd.models import projection


def test_table_file_is_well_formed():
    p = os.path.join(os.path.dirname(ops.__file__), "tuned", "midm_mi355x.json")
    t = json.load(open(p))
    for k, S in t.items():
        mode, b, N, K = (int(x) for x in k.split(":"))
        assert mode in (0, 1) and b in ops.MIDM_BUCKETS
        assert S >= 1 and K % S == 0 and (K // S) % 128 == 0  # pgemm split-K constraints
        assert mode == 1 or N % 256 == 0


def test_bucket_mapping_and_boundaries():
    cfg = ops.midm_config(600, 4096, 14336, 0)  # down at 600 rows -> the 768 bucket
    assert cfg == (256, ops.PGEMM_SPLIT, 4)
    assert ops.midm_config(512, 4096, 14336, 0)[2] == 8
    assert ops.midm_config(256, 4096, 14336, 0) is None  # decode sizes: the tile table
    assert ops.midm_config(5000, 4096, 14336, 0) is None  # past the last bucket
    assert ops.midm_config(1500, 6144, 4096, 0) is None  # qkv: the library wins there
    assert ops.midm_config(1024, 14336, 4096, 1)[2] == 1  # gate_up: unsplit fused tile
    assert ops.midm_config(700, 1234, 4096, 0) is None  # unknown shape


def test_slices_are_the_tables():
    """No fewer fp16 slabs than the table says: each would saturate at less of the row's sum."""
    p = os.path.join(os.path.dirname(ops.__file__), "tuned", "midm_mi355x.json")
    for k, S in json.load(open(p)).items():
        mode, b, N, K = (int(x) for x in k.split(":"))
        assert ops.midm_config(b, N, K, mode) == (256, ops.PGEMM_SPLIT, S)


def test_more_slices_where_tiles_leave_cus_idle():
    """3 and 5 tiles of 256 rows: slices of uneven length; never fewer than the table's, one round."""
    more = ops.midm_slices
    assert more(600, 4096, 14336, 4) == 5 and more(1100, 4096, 14336, 2) == 3
    assert more(512, 4096, 14336, 8) == 8 and more(1024, 4096, 4096, 4) == 4
    assert more(512, 6144, 4096, 4) == 5 and more(1400, 4096, 4096, 2) == 2
    for M in range(257, 2049, 37):
        for N in (1024, 4096, 6144, 10240):
            for K in (2048, 4096, 14336):
                for S in (2, 4):
                    s = more(M, N, K, S)
                    assert s == S or (S < s <= 16 and -(-M // 256) * (N // 256) * s <= 256)


@pytest.mark.parametrize("how", ["own device", "switch", "shared device", "off grid", "192 rows"])
def test_decode_rows_on_the_prefill_tile_only_where_it_may_run(how, monkeypatch):
    """193 to 256 decode rows: the tile's entry, but the table's tgemm entry with OMNIA_PGEMM=0, beside ranks
    on one device (whose all-reduce blocks spin), for weights off the 16-byte grid and for fewer rows."""
    class Model(projection.Projections):
        device, dtype, tp, use_pgemm = torch.device("cuda"), torch.bfloat16, 2, how != "switch"

    monkeypatch.setattr(projection.pstate, "ranks_per_device", lambda: 2 if how == "shared device" else 1)
    p = os.path.join(os.path.dirname(ops.__file__), "tuned", "decode_tile_mi355x.json")
    tiles = json.load(open(p))
    assert tiles
    M = 192 if how == "192 rows" else 256
    for key, (cols, S) in tiles.items():
        mode, N, K = (int(x) for x in key.split(":"))
        w = torch.empty(N << mode, K, dtype=torch.bfloat16, device="meta") if how != "off grid" else \
            torch.empty(K * (N << mode) + 1, dtype=torch.bfloat16)[1:].view(-1, K)
        cfg, table = Model()._wcfg(M, N, K, mode, True, w), ops.wgemm_config(M, N, K, mode)
        assert table is not None and ops.PGEMM_SPLIT < table[1] < 0
        assert cfg == ((cols, ops.PGEMM_SPLIT, S) if how == "own device" else table)


def test_kill_switch(monkeypatch):
    monkeypatch.setattr(ops, "_midm_on", False)
    assert ops.midm_config(600, 4096, 14336, 0) is None


def test_slices_of_the_narrow_tile_fit_the_kernel():
    """Whole K-tile pairs in every slice, one round of blocks, only between the few-row kernels and
    the prefill rows, and only where it takes a tenth less than the library by their models."""
    taken = 0
    for M in (1, 256, 257, 512, 999, 2001, 2048, 2049, 5000):
        for R in (128, 256, 1000, 1024, 1536, 2048, 4096, 16384):
            for K in (128, 1000, 2048, 4096, 5120, 6144, 8192, 14336, 16384):
                S = ops.tile_slices(M, R, K)
                if S:
                    taken += 1
                    assert 256 < M <= 2048 and R % 128 == 0 and K % (128 * S) == 0
                    assert S > 1 and -(-M // 256) * (R // 128) * S <= 256
                    assert R >= 2048 or K >= 6144  # below, the library is faster
    assert taken and ops.tile_slices(999, 2048, 8192) == 4 and not ops.tile_slices(999, 2048, 2048)


def test_tile_width():
    """Narrow where one round of it does, or three for two wide ones; never for rows that leave no
    whole wide tiles, which the kernel refuses."""
    assert ops.tile_cols(512, 16384) == 128 and ops.tile_cols(999, 16384) == 256
    assert ops.tile_cols(600, 28672) == 128 and ops.tile_cols(16384, 28672) == 256
    assert ops.tile_cols(512, 16384 - 128) == 256
