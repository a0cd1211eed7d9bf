"""Llama-3 family forward on the engine's paged KV cache (TP-aware).

Per layer (T tokens, hidden d):
    fused_add_rmsnorm -> QKV GEMM -> RoPE + paged KV write (HIP) ->
    paged attention (HIP prefill / decode) -> O GEMM [-> TP all-reduce] ->
    fused_add_rmsnorm -> gate_up GEMM + SwiGLU -> down GEMM [-> all-reduce]
GEMMs go through :func:`omnia_amd.ops.linear`: the hand MFMA decode kernel
(``ops/csrc/gemm.hip``, SwiGLU fused in its epilogue) on the shapes where the
MI355X sweep measured it faster, tuned hipBLASLt everywhere else.
Weights are kept in their natural [out, in] layout so ``F.linear`` maps onto a
single hipBLASLt GEMM; column-parallel shards (QKV, gate_up) and row-parallel
shards (O, down) follow Megatron.  The reference has no model code at all
(SURVEY §0.2); this replaces its remote Provider (``internal/runtime/provider.go:95-151``).
"""
from __future__ import annotations

import math
import os
from dataclasses import dataclass

import torch
import torch.nn.functional as F

from .. import ops
from ..ops import reference as ref
from ..parallel import overlap
from ..parallel import state as pstate
from .config import ModelConfig
from .projection import (Parts, Projections, RowPar, packed_copy, shared_device,
                         version)

# decode attention: below this many (sequence, kv head) pairs a step splits every
# live context on the device (``LlamaModel.decode_part``)
DECODE_SPLIT_PAIRS = int(os.environ.get("OMNIA_DECODE_SPLIT_PAIRS", "256"))


@dataclass
class ForwardBatch:
    """Flattened step inputs.  All tensors live on the model device."""

    input_ids: torch.Tensor  # int32 [T]
    positions: torch.Tensor  # int32 [T]
    slots: torch.Tensor  # int64 [T]  flat KV slot of each token
    block_tables: torch.Tensor  # int32 [B, max_blocks]
    seq_lens: torch.Tensor  # int32 [B] total context incl. this step's tokens
    logits_indices: torch.Tensor  # int64 [B] rows of T whose logits are needed
    is_decode: bool = True
    q_start_loc: torch.Tensor | None = None  # int32 [B+1] (prefill)
    tile_seq: torch.Tensor | None = None  # int32 [n_tiles] (prefill)
    tile_q0: torch.Tensor | None = None
    num_seqs: int = 0
    # mixed step: the first ``num_decode`` tokens are decode rows (one token of a
    # running sequence each, attended by the decode kernel over dec_*), the rest
    # are prefill chunks described by q_start_loc / seq_lens / block_tables
    num_decode: int = 0
    dec_block_tables: torch.Tensor | None = None  # int32 [Bd, max_blocks]
    dec_seq_lens: torch.Tensor | None = None  # int32 [Bd]
    # decode rows whose input token is still on the device: tok_slots[ids_src[r]]
    # where ids_src[r] >= 0 (resolved inside the embedding kernel)
    ids_src: torch.Tensor | None = None
    tok_slots: torch.Tensor | None = None
    # context-parallel prefill (parallel/context_parallel.py CPPrefill): this
    # rank's zig-zag shard of one long prompt; K/V go to the CP scratch pages and
    # attention is the ring over the CP group
    cp: object = None
    # models with recurrent layers: state slot of each sequence (decode rows first,
    # then the prefill portions); -1 = padded row
    state_slots: torch.Tensor | None = None  # int32
    # models whose prefill attention works on a dense copy of the visible keys: rows
    # [kv_start[s], kv_start[s+1]) hold positions kv_first[s].. of sequence s
    # (64-aligned ranges, kv_rows in all)
    kv_start: torch.Tensor | None = None  # int32 [B+1]
    kv_first: torch.Tensor | None = None  # int32 [B]
    kv_rows: int = 0


@dataclass
class KVCache:
    k: list  # per layer [NB, Hkv_local, BS, D]
    v: list
    block_size: int
    num_blocks: int

    @staticmethod
    def allocate(cfg: ModelConfig, num_blocks: int, block_size: int, device, tp_size: int = 1,
                 dtype=torch.bfloat16) -> "KVCache":
        hkv = max(1, cfg.num_kv_heads // tp_size)
        buf = torch.empty(cfg.num_layers, 2, num_blocks, hkv, block_size, cfg.head_dim,
                          dtype=dtype, device=device)
        return KVCache(k=[buf[i, 0] for i in range(cfg.num_layers)],
                       v=[buf[i, 1] for i in range(cfg.num_layers)],
                       block_size=block_size, num_blocks=num_blocks)

    def page_tensors(self) -> list:
        """Every per-page tensor (page index first): what a page move copies."""
        return [t for kv in zip(self.k, self.v) for t in kv]

    def state_tensors(self) -> list:
        return []


def _init(shape, std, device, dtype, gen):
    t = torch.empty(shape, dtype=torch.float32, device=device)
    t.normal_(0.0, std, generator=gen)
    return t.to(dtype)


class LlamaModel(Projections):
    def __init__(self, cfg: ModelConfig, device="cpu", dtype=torch.bfloat16, seed: int = 0,
                 weights: dict | None = None, decode_part_size: int = 512):
        self.cfg = cfg
        self.device = torch.device(device)
        self.dtype = dtype
        st = pstate.get_state()
        self.tp, self.tpr = st.tp_size, st.tp_rank
        if cfg.num_heads % self.tp:
            raise ValueError("num_heads not divisible by tp")
        self.hq = cfg.num_heads // self.tp
        self.hkv = max(1, cfg.num_kv_heads // self.tp)
        self.inter = cfg.intermediate_size // self.tp
        self.vocab_local = cfg.vocab_size // self.tp if cfg.vocab_size % self.tp == 0 else None
        if self.vocab_local is None:
            raise ValueError("vocab not divisible by tp")
        self.vocab_start = self.tpr * self.vocab_local
        self.scale = 1.0 / math.sqrt(cfg.head_dim)
        self.seed = seed
        self.decode_part_size = decode_part_size
        self.cos_sin = ref.rope_cos_sin(cfg.max_position, cfg.head_dim, cfg.rope_theta,
                                        cfg.rope_scaling, device=self.device)
        self.w = weights if weights is not None else self._random_weights(seed)
        self.fold_norms()
        self._ws = {}
        ops.dgemm_prepare(self.device)  # split-K workspace, before any graph capture

    # ------------------------------------------------------------ weights
    def _random_weights(self, seed: int) -> dict:
        """Random-init shard of this TP rank (no checkpoint available offline).

        Std 0.02 like HF init; norms at 1.  Initialised directly on the device."""
        cfg, dev, dt = self.cfg, self.device, self.dtype
        g = torch.Generator(device=dev)
        g.manual_seed(seed * 1000 + self.tpr)
        d, D = cfg.hidden_size, cfg.head_dim
        w = {
            "embed": _init((self.vocab_local, d), 0.02, dev, dt, g),
            "final_norm": torch.ones(d, dtype=dt, device=dev),
            "layers": [],
        }
        w["lm_head"] = w["embed"] if cfg.tie_embeddings else _init((self.vocab_local, d), 0.02,
                                                                   dev, dt, g)
        for li in range(cfg.num_layers):
            layer = {
                "in_norm": torch.ones(d, dtype=dt, device=dev),
                "post_norm": torch.ones(d, dtype=dt, device=dev),
                "qkv": _init(((self.hq + 2 * self.hkv) * D, d), 0.02, dev, dt, g),
                "o": _init((d, self.hq * D), 0.02 / math.sqrt(2 * cfg.num_layers), dev, dt, g),
            }
            layer.update(self._random_mlp(g, li))
            w["layers"].append(layer)
        return w

    def _random_mlp(self, g, li: int = 0) -> dict:
        cfg, dev, dt, d = self.cfg, self.device, self.dtype, self.cfg.hidden_size
        return {
            "gate_up": _init((2 * self.inter, d), 0.02, dev, dt, g),
            "down": _init((d, self.inter), 0.02 / math.sqrt(2 * cfg.num_layers), dev, dt, g),
        }

    def weight_bytes(self) -> int:
        n = 0
        seen = set()

        def add(t):
            nonlocal n
            if isinstance(t, torch.Tensor) and t.data_ptr() not in seen:
                seen.add(t.data_ptr())
                n += t.numel() * t.element_size()

        for k, v in self.w.items():
            if k == "layers":
                for layer in v:
                    for t in layer.values():
                        if isinstance(t, list):
                            for x in t:
                                add(x)
                        else:
                            add(t)
            else:
                add(v)
        return n

    # RMSNorm(h) @ W^T == rsqrt(mean(h^2) + eps) * (h @ (W diag(w))^T): the norm
    # weight folds into the consumer's weight rows once at load, after which
    # every norm of the model is weightless.  The prefill path (pgemm.hip) then
    # applies the row scale in the QKV / gate_up epilogue from the row sums of
    # squares its producer (O / down residual epilogue) emits, and the decode /
    # TP / CP paths run their existing norm kernels with a ones weight.
    fold_post_norm = True  # Mixtral's post-attention norm also feeds the router

    def fold_norms(self) -> None:
        for layer in self.w["layers"]:
            pairs = [("in_norm", "qkv")]
            if self.fold_post_norm:
                pairs.append(("post_norm", "gate_up"))
            for nk, wk in pairs:
                nw = layer[nk]
                if bool(torch.all(nw == 1)):
                    continue
                W = layer[wk]
                layer[wk] = (W.float() * nw.float()[None, :]).to(W.dtype)
                layer[nk] = torch.ones_like(nw)

    # tile-packed decode weights (ops.tgemm_pack): a second, stage-contiguous copy
    # of each projection the tuned table sends to tgemm.  Streamed alone, row-major
    # weights (128-B pieces of rows 2*K bytes apart) reach ~4.5 TB/s and packed
    # ones ~6.0 TB/s; inside the full kernel, next to the x re-reads and the
    # MFMAs, the gain is 0-3 % per projection (profiles/r5/decode_gemm/); end to
    # end the closed-loop bench gains +0.8 % tok/s and -2 % TPOT, 3 of 3
    # interleaved pairs (profiles/r6/bench/tgemm_pack/, of all projections; gate_up
    # and down have since gone on to the prefill tile, which reads row-major weights:
    # 256 rows of an 8B model, 577 keys each, 8824 / 8683 us).  Only batches past the
    # few-row kernels (193 to 256 rows) run it.  The copy is built before the KV
    # pool is sized, by default whenever it and the few-row copies fit
    # pack_budget_frac of HBM (70B TP=1 and MoE models: never);
    # OMNIA_TGEMM_PACK=0 turns it off.
    pack_budget_frac = 0.10  # of the device's HBM, copies for the few-row kernels included

    def prepack_decode(self, max_batch: int) -> int:
        """Pack the projections for the few-row kernels and, for the batches up to
        ``max_batch`` that go on to tgemm, for that; returns the bytes packed (0: off /
        over budget)."""
        n = self.pack_streams()
        return n + self._prepack_tiles(max_batch, n)

    def _prepack_tiles(self, max_batch: int, packed: int) -> int:
        self._packed = {}
        env = os.environ.get("OMNIA_TGEMM_PACK", "1")
        if env not in ("1", "force") or self.device.type != "cuda" or self.tp != 1 \
                or self.cfg.is_moe:
            return 0
        want, known = {}, {}
        top = next((b for b in ops.WGEMM_BUCKETS if b >= max_batch), ops.WGEMM_BUCKETS[-1])
        for layer in self.w["layers"]:
            for key, mode in (("qkv", 0), ("o", 0), ("down", 0), ("gate_up", 1)):
                w = layer[key]
                kind = key, w.shape, packed_copy(self, w) is not None
                if kind not in known:  # the entries that some batch runs, which few rows do not
                    N = w.shape[0] // 2 if mode == 1 else w.shape[0]
                    known[kind] = {self._wcfg(M, N, w.shape[1], mode, True, w)
                                   for M in range(1, top + 1)}
                for cfg in known[kind]:
                    if cfg is None or cfg[1] >= 0 or cfg[1] == ops.PGEMM_SPLIT or (-1 - cfg[1]) & 2:
                        continue  # not tgemm, or its 32-k stage form
                    pmode = 1 if mode == 1 and cfg[2] == 1 else 0
                    want[(w.data_ptr(), cfg[0], pmode)] = w
        total = sum(w.numel() * w.element_size() for w in want.values())
        cap = torch.cuda.get_device_properties(self.device).total_memory * self.pack_budget_frac
        if not want or (env != "force" and packed + total > cap):
            return 0
        for (ptr, bn, pmode), w in want.items():
            self._packed[(ptr, bn, pmode)] = w, version(w), ops.tgemm_pack(w, bn, pmode)
        return total

    # ------------------------------------------------------------ forward
    def add_norm(self, x, residual: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
        """residual += x (TP-reduced); returns RMSNorm(residual) * w."""
        eps = self.cfg.rms_eps
        if isinstance(x, RowPar):
            return overlap.rowparallel_add_norm(x.x, x.w, residual, w, eps)
        if isinstance(x, Parts):
            if self.tp == 1:
                return ops.splitk_add_rmsnorm(x.t, residual, w, eps)
            x = ops.splitk_reduce(x.t)
        if self.tp > 1:
            return pstate.tp_all_reduce_add_rmsnorm(x, residual, w, eps)
        ops.fused_add_rmsnorm(x, residual, w, eps)
        return x

    def mlp(self, layer: dict, h: torch.Tensor, is_decode: bool = False):
        M, K = h.shape
        I2 = layer["gate_up"].shape[0]
        if self._pgemm_ok(M, K, I2 // 2, is_decode, layer["gate_up"]):
            # gate_up + SwiGLU in the prefill kernel's epilogue (pgemm EPI 1)
            return self._proj("down", ops.pgemm(1, h, layer["gate_up"]), layer["down"], False)
        cfg = self._wcfg(M, I2 // 2, K, 1, is_decode, layer["gate_up"])
        if cfg is None:
            a = None if M > ops.PANEL_MAX_M else self._few(1, h, layer["gate_up"])
            if a is None:
                a = ops.linear_silu(h, layer["gate_up"])  # SwiGLU fused into decode GEMMs
        elif cfg[1] == ops.PGEMM_SPLIT and cfg[2] == 1:
            a = ops.pgemm(1, h, layer["gate_up"])  # the unsplit fused tile
        else:
            nw, nwaves, S = cfg
            if S == 1 and nwaves != ops.PGEMM_SPLIT:
                a = self._wgemm(1, h, layer["gate_up"], 1, nw, nwaves)
            else:
                a = ops.splitk_swiglu(self._wgemm(
                    2, h, layer["gate_up"], S, nw, nwaves,
                    out=self._parts("gu", S, M, I2, self._slab_dtype(nwaves))))
        return self._proj("down", a, layer["down"], is_decode)

    def attention(self, li: int, h: torch.Tensor, fb: ForwardBatch, kv: KVCache):
        T = h.shape[0]
        D = self.cfg.head_dim
        wqkv = self.w["layers"][li]["qkv"]
        if fb.cp is None and D == 128 and (self.hq + 2 * self.hkv) % 2 == 0 and \
                self._pgemm_ok(T, h.shape[1], wqkv.shape[0], fb.is_decode):
            # QKV + RoPE + paged KV write in the prefill kernel's epilogue (pgemm
            # EPI 3, no row scale: h is already normalised on this path)
            q = ops.pgemm(3, h, wqkv, positions=fb.positions, cos_sin=self.cos_sin,
                          k_cache=kv.k[li], v_cache=kv.v[li], slots=fb.slots, hq=self.hq,
                          hkv=self.hkv, block_size=kv.block_size)
            o = self._attend(li, q.view(T, self.hq, D), fb, kv)
            return self._proj("o", o.view(T, self.hq * D), self.w["layers"][li]["o"], False)
        qkv = self._proj("qkv", h, wqkv, fb.is_decode, slabs=fb.cp is None)
        if fb.cp is not None:
            cp = fb.cp
            q = qkv[:, : self.hq * D]
            ops.rope_kv(q, qkv[:, self.hq * D: (self.hq + self.hkv) * D],
                        qkv[:, (self.hq + self.hkv) * D:], fb.positions, self.cos_sin,
                        cp.scratch[0], cp.scratch[1], fb.slots, self.hq, self.hkv, cp.bs)
            o = cp.attention(kv.k[li], kv.v[li], q.view(T, self.hq, D), self.scale)
            return self._proj("o", o.view(T, self.hq * D), self.w["layers"][li]["o"], False)
        if isinstance(qkv, Parts):
            q = ops.splitk_rope_kv(qkv.t, fb.positions, self.cos_sin, kv.k[li], kv.v[li],
                                   fb.slots, self.hq, self.hkv, kv.block_size)
        else:
            q = qkv[:, : self.hq * D]
            k = qkv[:, self.hq * D: (self.hq + self.hkv) * D]
            v = qkv[:, (self.hq + self.hkv) * D:]
            ops.rope_kv(q, k, v, fb.positions, self.cos_sin, kv.k[li], kv.v[li], fb.slots,
                        self.hq, self.hkv, kv.block_size)
        o = self._attend(li, q.view(T, self.hq, D), fb, kv)
        return self._proj("o", o.view(T, self.hq * D), self.w["layers"][li]["o"], fb.is_decode)

    def _mixed_attention(self, li: int, q3: torch.Tensor, fb: ForwardBatch, kv: KVCache):
        """Mixed step: decode rows (the first ``num_decode``) on the split-K decode
        kernel (K/V read once per GQA group), prefill chunks on the flash prefill
        kernel, one output."""
        T, D = q3.shape[0], self.cfg.head_dim
        Bd = fb.num_decode
        o = torch.empty_like(q3) if q3.is_contiguous() else torch.empty(
            T, self.hq, D, dtype=q3.dtype, device=q3.device)
        mb = fb.dec_block_tables.shape[1]
        part, splits = self.decode_part(Bd, mb * kv.block_size)
        ws = self._decode_ws(1 << max(0, Bd - 1).bit_length(), mb, kv.block_size, q3.device,
                             part, splits)  # pow2 rows: few workspace shapes across mixed steps
        ops.decode_attention(q3[:Bd], kv.k[li], kv.v[li], fb.dec_block_tables,
                             fb.dec_seq_lens, self.scale, part_size=part, workspace=ws,
                             out=o[:Bd], splits=splits)
        if T > Bd:
            ops.prefill_attention(q3[Bd:], kv.k[li], kv.v[li], fb.block_tables,
                                  fb.q_start_loc, fb.seq_lens, self.scale, fb.tile_seq,
                                  fb.tile_q0, out=o[Bd:], shared_device=shared_device(self))
        return o

    def decode_part(self, batch: int, max_ctx: int) -> tuple[int, int]:
        """(partition length, splits) of the split-K decode attention.

        With >= DECODE_SPLIT_PAIRS (sequence, kv head) pairs the pairs alone give every
        CU a block: one partition up to 2048 keys, else partitions of 1024 (fewer starts
        and partials, but ragged ends).  us at 512 / 1024 / 2048 keys, 8 KV heads: 32
        sequences of 1000 31 / 27 / 27, 128 of 1000 106 / 95 / 95, 64 of 2000 104 / 98 / 91,
        40 of 3500 113 / 107 / 116; ragged from 100 to 2000 keys 32 sequences 39 / 38 / 33,
        64 63 / 60 / 62, 128 119 / 117 / 114; 8 of 2000 among 248 of 500 242 / 227 / 214.
        One of 2000 among 63 of 500 is bounded by its own walk: 48 / 52 / 58.

        With fewer pairs (small batches, one KV head per TP rank) every live context is cut
        on the device into up to ``splits`` equal partitions (``ops.decode_attention``), so
        short contexts still spread over the CUs; the captured graph needs no host-known
        length."""
        pairs = batch * self.hkv
        if 0 < pairs < DECODE_SPLIT_PAIRS:
            splits = -(-DECODE_SPLIT_PAIRS // pairs)
            splits = max(1, min(splits, -(-max_ctx // ops.DECODE_SPLIT_MIN)))
            return self.decode_part_size, splits
        part = self.decode_part_size
        while part < (2048 if max_ctx <= 2048 else 1024) and part < max_ctx:
            part *= 2
        return part, 0

    def _attend(self, li: int, q3: torch.Tensor, fb: ForwardBatch, kv: KVCache):
        """Attention of a step's rotated queries over the pages."""
        if fb.is_decode:
            T, mb = q3.shape[0], fb.block_tables.shape[1]
            part, splits = self.decode_part(T, mb * kv.block_size)
            ws = self._decode_ws(T, mb, kv.block_size, q3.device, part, splits)
            return ops.decode_attention(q3, kv.k[li], kv.v[li], fb.block_tables, fb.seq_lens,
                                        self.scale, part_size=part, workspace=ws, splits=splits)
        if fb.num_decode:
            return self._mixed_attention(li, q3, fb, kv)
        return ops.prefill_attention(q3, kv.k[li], kv.v[li], fb.block_tables, fb.q_start_loc,
                                     fb.seq_lens, self.scale, fb.tile_seq, fb.tile_q0,
                                     shared_device=shared_device(self))

    def _decode_ws(self, B, max_blocks, bs, device, part, splits=0):
        key = (B, max_blocks, bs, str(device), part, splits)
        ws = self._ws.get(key)
        if ws is None:
            if device.type != "cuda":
                return None
            ws = ops.decode_workspace(B, self.hq, max_blocks, bs, part, device, splits)
            self._ws[key] = ws
        return ws

    def embed(self, ids: torch.Tensor, src: torch.Tensor | None = None,
              tok_slots: torch.Tensor | None = None) -> torch.Tensor:
        h = ops.embedding(ids, self.w["embed"], self.vocab_start, src=src, tok_slots=tok_slots)
        return pstate.tp_all_reduce(h) if self.tp > 1 else h

    # ------------------------------------------------ fused prefill (pgemm.hip)
    def _use_fused(self, fb: ForwardBatch) -> bool:
        """Prefill chunks -- and mixed steps, whose decode rows ride the same
        GEMMs -- on one GPU run the fused-epilogue prefill layer: QKV+RoPE+KV-write,
        O+residual, gate_up+SwiGLU, down+residual, with the RMSNorms riding the
        epilogues (no standalone norm / SwiGLU / RoPE launch)."""
        if not (self.use_pgemm and self.device.type == "cuda" and not fb.is_decode
                and fb.cp is None and self.tp == 1):
            return False
        T = fb.input_ids.shape[0]
        if T < (self.PGEMM_MIXED_MIN_ROWS if fb.num_decode else self.PGEMM_MIN_ROWS):
            return False
        cfg, d = self.cfg, self.cfg.hidden_size
        return (cfg.head_dim == 128 and d % 256 == 0 and d % 128 == 0
                and (self.hq + 2 * self.hkv) % 2 == 0
                and self.inter % 128 == 0
                and self.fold_post_norm and not self.cfg.is_moe)

    def _fused_residual(self, fb: ForwardBatch, kv: KVCache) -> torch.Tensor:
        """Residual stream after the last layer (un-normalised) of a prefill chunk."""
        cfg = self.cfg
        T, d, D = fb.input_ids.shape[0], cfg.hidden_size, cfg.head_dim
        inv_d, eps = 1.0 / d, cfg.rms_eps
        h = self.embed(fb.input_ids)
        ss = ops.row_sumsq(h).view(T, 1)
        nsl = d // 256
        ss_mid = torch.empty(T, nsl, dtype=torch.float32, device=h.device)
        ss_out = torch.empty(T, nsl, dtype=torch.float32, device=h.device)
        q = torch.empty(T, self.hq * D, dtype=h.dtype, device=h.device)
        act = torch.empty(T, self.inter, dtype=h.dtype, device=h.device)
        for li, layer in enumerate(self.w["layers"]):
            ops.pgemm(3, h, layer["qkv"], out=q, ss_in=ss, inv_d=inv_d, eps=eps,
                      positions=fb.positions, cos_sin=self.cos_sin, k_cache=kv.k[li],
                      v_cache=kv.v[li], slots=fb.slots, hq=self.hq, hkv=self.hkv,
                      block_size=kv.block_size)
            o = self._attend(li, q.view(T, self.hq, D), fb, kv)
            ops.pgemm(2, o.view(T, self.hq * D), layer["o"], out=h, ss_out=ss_mid)
            ops.pgemm(1, h, layer["gate_up"], out=act, ss_in=ss_mid, inv_d=inv_d, eps=eps)
            ops.pgemm(2, act, layer["down"], out=h, ss_out=ss_out)
            ss = ss_out  # the next QKV reads it before the next down overwrites it
        return h

    # ------------------------------------------------ a few rows (stream.hip)
    def _use_stream(self, fb: ForwardBatch) -> bool:
        """Steps of a few rows run a layer as four projections and attention: norms, RoPE and
        KV write, SwiGLU and residual ride in the projections' kernels."""
        cfg = self.cfg
        if fb.cp is not None or not self.fold_post_norm or cfg.head_dim != 128:
            return False
        T, layer = fb.input_ids.shape[0], self.w["layers"][0]
        if T > ops.STREAM_MAX_M:
            return False
        ws = [self._stream_weight(T, layer[k], k == "gate_up")
              for k in ("qkv", "o", "gate_up", "down")]
        if not all(ws):
            return False
        # row-major weights reach that kernel in pieces: separate kernels on the panel take 0.76
        # of a step of 16 rows at 8192 x 28672, 0.92 at 4096 x 14336, 0.86 at 2048 x 8192 and 0.92
        # at 1024 x 4096 (captured), and 1.4 where an eager step of layers of 34 MB waits for its
        # launches
        return all(packed for _, packed in ws) or \
            (not fb.is_decode and sum(w.numel() for w, _ in ws) <= 1 << 25)

    def _stream_residual(self, fb: ForwardBatch, kv: KVCache) -> torch.Tensor:
        """Residual stream after the last layer (un-normalised) of a step of a few rows."""
        cfg = self.cfg
        T = fb.input_ids.shape[0]
        norm = dict(inv_d=1.0 / cfg.hidden_size, eps=cfg.rms_eps)
        h = self.embed(fb.input_ids, fb.ids_src, fb.tok_slots)
        ss = ops.row_sumsq(h).view(T, 1)

        def stream(epi, x, w, **kw):
            # the first layer's are covered; another's may lie off the 16-byte grid
            w, packed = self._stream_weight(T, w, epi == 1) or (
                w.clone(memory_format=torch.contiguous_format), False)
            return ops.stream(epi, x, w, packed=packed, **kw)

        mid, end = (ops.stream_sums(T, self.w["layers"][0][k], h.device) for k in ("o", "down"))
        for li, layer in enumerate(self.w["layers"]):
            q = stream(3, h, layer["qkv"], ss=ss, positions=fb.positions, cos_sin=self.cos_sin,
                       k_cache=kv.k[li], v_cache=kv.v[li], slots=fb.slots, hq=self.hq,
                       hkv=self.hkv, **norm)
            o = self._attend(li, q.view(T, self.hq, cfg.head_dim), fb, kv)
            stream(2, o.view(T, -1), layer["o"], out=h, ss=mid)
            a = stream(1, h, layer["gate_up"], ss=mid, **norm)
            stream(2, a, layer["down"], out=h, ss=end)
            ss = end
        return h

    def _residual(self, fb: ForwardBatch, kv: KVCache) -> torch.Tensor | None:
        """The un-normalised residual of a step on one of the fused layer paths, else None."""
        if self._use_fused(fb):
            return self._fused_residual(fb, kv)
        return self._stream_residual(fb, kv) if self._use_stream(fb) else None

    def hidden_states(self, fb: ForwardBatch, kv: KVCache) -> torch.Tensor:
        r = self._residual(fb, kv)
        if r is not None:
            return ops.rmsnorm(r, self.w["final_norm"], self.cfg.rms_eps)
        return self._hidden_rows(fb, kv)

    def _hidden_rows(self, fb: ForwardBatch, kv: KVCache) -> torch.Tensor:
        """Final-normed rows by the unfused layer path."""
        cfg = self.cfg
        self._min_rows = self.PGEMM_MIXED_MIN_ROWS if fb.num_decode else self.PGEMM_MIN_ROWS
        residual = self.embed(fb.input_ids, fb.ids_src, fb.tok_slots)
        h = ops.rmsnorm(residual, self.w["layers"][0]["in_norm"], cfg.rms_eps)
        m = None
        for li, layer in enumerate(self.w["layers"]):
            if li > 0:
                h = self.add_norm(m, residual, layer["in_norm"])
            a = self.attention(li, h, fb, kv)
            h = self.add_norm(a, residual, layer["post_norm"])
            m = self.mlp(layer, h, fb.is_decode)
        return self.add_norm(m, residual, self.w["final_norm"])

    def logits(self, h: torch.Tensor, gather: bool = True,
               is_decode: bool = False) -> torch.Tensor:
        """LM head.  Under TP the result is this rank's vocab slice unless
        ``gather`` (the distributed sampler, parallel/tp_sampling.py, needs
        only the slice).  Decode batches use the weight-streaming tile kernel
        when the measured table lists an unsplit (bf16-out) config for it."""
        W = self.w["lm_head"]
        cfg = self._wcfg(h.shape[0], W.shape[0], h.shape[1], 0, is_decode, W, False)
        if cfg is not None and cfg[2] == 1:
            lg = ops.wgemm(0, h, W, 1, cfg[0], cfg[1])
        else:
            lg = self._few(0, h, W)
            lg = ops.linear(h, W) if lg is None else lg
        return pstate.tp_all_gather_lastdim(lg) if (self.tp > 1 and gather) else lg

    def forward(self, fb: ForwardBatch, kv: KVCache, gather: bool = True) -> torch.Tensor:
        r = self._residual(fb, kv)
        h = self._hidden_rows(fb, kv) if r is None else r
        # decode rows are their own logits rows (logits_indices is the identity)
        if not (fb.is_decode and fb.logits_indices.shape[0] == h.shape[0]):
            h = h.index_select(0, fb.logits_indices)
        if r is not None:
            h = ops.rmsnorm(h, self.w["final_norm"], self.cfg.rms_eps)
        return self.logits(h, gather, fb.is_decode)
