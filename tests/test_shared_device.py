"""Ranks that share a device: what the model tells the kernels whose blocks would leave no room
beside the peers' spinning all-reduce blocks."""
from types import SimpleNamespace

import pytest
import torch

from omnia_amd import ops
from omnia_amd.models.llama import LlamaModel
from omnia_amd.parallel import state as pstate


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("tp,ranks", [(1, 1), (2, 1), (2, 2)])
def test_prompt_attention_is_told(tp, ranks, mixed, monkeypatch):
    told = []
    monkeypatch.setattr(pstate, "ranks_per_device", lambda: ranks)
    monkeypatch.setattr(ops, "prefill_attention",
                        lambda *a, shared_device=False, **kw: told.append(shared_device))
    monkeypatch.setattr(ops, "decode_attention", lambda *a, **kw: None)
    m = LlamaModel.__new__(LlamaModel)
    m.tp, m.scale, m.hq, m.hkv, m._ws, m.decode_part_size = tp, 1.0, 2, 1, {}, 256
    m.cfg = SimpleNamespace(head_dim=8)
    fb = SimpleNamespace(is_decode=False, num_decode=int(mixed), block_tables=None,
                         q_start_loc=None, seq_lens=None, tile_seq=None, tile_q0=None,
                         dec_block_tables=torch.zeros(1, 1), dec_seq_lens=None)
    kv = SimpleNamespace(k=[None], v=[None], block_size=16)
    m._attend(0, torch.zeros(3, 2, 8), fb, kv)
    assert told == [ranks > 1]
