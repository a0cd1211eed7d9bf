"""Mid-size step dispatch (ops.midm_config, ops/tuned/midm_mi355x.json): bucket
mapping, the decode / prefill-tile boundaries, mode-1 (gate_up) unsplit
entries, and the OMNIA_MIDM kill switch -- pure table logic, CPU."""
import json
import os

from omnia_amd import ops


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
