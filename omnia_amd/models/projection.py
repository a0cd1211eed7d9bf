"""Dispatch of a model's linear projections to the measured GEMM paths.

Every model family mixes this in: decode batches go to the weight-streaming /
tile kernels where the measured tables list a win (their split-K slabs are
reduced by the consumer kernel), prefill to the 256x256 MFMA tile, everything
else (and every fp32 model) to the library GEMM.
"""
from __future__ import annotations

import os

import torch

from .. import ops
from ..parallel import overlap
from ..parallel import state as pstate


class Parts:
    """fp32 split-K partial slabs [S, M, N] of a projection (wgemm.hip MODE 2)."""

    __slots__ = ("t",)

    def __init__(self, t: torch.Tensor):
        self.t = t


class RowPar:
    """A deferred TP row-parallel projection ``x @ w.T`` (prefill): ``add_norm``
    runs it chunked along M with each chunk's all-reduce + residual + RMSNorm
    overlapped on a side stream (``parallel/overlap.py``)."""

    __slots__ = ("x", "w")

    def __init__(self, x: torch.Tensor, w: torch.Tensor):
        self.x, self.w = x, w


def version(t: torch.Tensor) -> int | None:
    """Counts in-place writes (None: inference tensors do not)."""
    return None if t.is_inference() else t._version


def unchanged(w: torch.Tensor, t: torch.Tensor, at: int | None) -> bool:
    """Whether ``w``, at the address of ``t``, is ``t`` as it was at version ``at``."""
    # eager steps wait for this, so what is known is not asked for again
    same = t is w or (t.shape == w.shape and t.dtype == w.dtype and w.is_contiguous())
    return same and (at is None or at == w._version)


def packed_copy(model, w: torch.Tensor) -> torch.Tensor | None:
    """The model's packed copy of a weight (``Projections.pack_streams``), while the weight is
    what was copied."""
    streams = getattr(model, "_streams", None)
    hit = streams.get(w.data_ptr()) if streams else None
    if hit is None:
        return None
    t, at, copy = hit
    return copy if unchanged(w, t, at) else None


def few_weight(model, M: int, w: torch.Tensor, gated: bool, slabs: bool):
    """(weight, packed) to run ``M`` rows of a projection on the few-row kernels where they beat
    the other paths, else None."""
    if not 1 <= M <= ops.PANEL_MAX_M or not ops.streams_on():
        return None
    copy = packed_copy(model, w)  # the kernels cover what has one
    if copy is not None and M <= ops.STREAM_MAX_M:
        return copy, True
    if copy is None and not ops.stream_ok(M, w, gated):
        return None
    R, K = w.shape
    if not ops.few_rows_pay(M, R, K, gated, copy is not None, slabs):
        return None
    return (w, False) if copy is None else (copy, True)


def packed_experts(model, up: torch.Tensor, down: torch.Tensor):
    """Packed copies of a layer's expert weights, or None."""
    t = packed_copy(model, up), packed_copy(model, down)
    return None if t[0] is None or t[1] is None else t


def shared_device(model) -> bool:
    """Whether other ranks, whose all-reduce blocks may spin, run on this one's device."""
    return model.tp > 1 and pstate.ranks_per_device() > 1


class Projections:
    """Needs ``device``, ``dtype``, ``tp`` and ``_ws`` (workspace dict) on the model."""

    use_pgemm = os.environ.get("OMNIA_PGEMM", "1") != "0"
    # prefill chunks take the fused layer from this many rows.  Below it the
    # unsplit 256x256 tile leaves most CUs idle on qkv / o / down; the unfused
    # path runs them split-K on the same tile (ops.midm_config) and is 1.2-2.2x
    # faster per layer at 512-2048 rows (profiles/r6/open/)
    PGEMM_MIN_ROWS = int(os.environ.get("OMNIA_PGEMM_MIN_ROWS", "2049"))
    # mixed steps take the fused layer only from this many rows: at the open-loop
    # trickle (~256 decode rows + a few hundred prompt tokens) pgemm's 256x256
    # tiles leave most CUs idle, and the split decode / library path is 1.5x
    # faster per step (profiles/r5/mixed_open_loop/: p50 TPOT 14.9 vs 22.9 ms).
    # Neither threshold holds projections off the tile where it fills the chip
    # (ops.gated_tile_pays, ops.plain_tile_fills), nor long-K ones off its slices
    # (ops.tile_slices; OMNIA_MIDM=0 does): in mixed steps too that is the faster
    # way (gated: 8 layers of 4096 x 14336, 256 decode rows and 190 / 256 prompt
    # rows 3.29 / 3.38 ms with it, 3.37 / 3.45 without; 16 of 2048 x 8192, 256 and
    # 650 5.85 and 6.08.  Plain and sliced: 16 of 2048 x 8192, 256 and 250 / 650 /
    # 1792 / 3700 3.65 / 4.39 / 6.23 / 10.30, without 3.73 / 4.49 / 6.34 / 10.44)
    PGEMM_MIXED_MIN_ROWS = int(os.environ.get("OMNIA_PGEMM_MIXED_MIN_ROWS", "4096"))

    # ---- a few rows (ops.stream, ops.panel)
    # copies of the projections in the order those kernels stream best, made before the KV
    # pool is sized, while they fit this part of HBM
    stream_budget_frac = 0.06
    STREAM_KEYS = {"qkv", "o", "gate_up", "down", "up", "in", "uq", "experts_gate_up",
                   "experts_down"}

    # address -> (weight, its version, copy): the weight is held, so that no other takes its
    # address, and a copy counts only while the weight is what was copied
    _streams: dict = {}

    def pack_streams(self) -> int:
        """Lay the projection weights out for :func:`ops.stream`; returns the bytes (0: off, or
        over budget).  Weights replaced or written to afterwards run as they are."""
        self._streams = {}
        if self.device.type != "cuda" or self.dtype != torch.bfloat16 or self.tp != 1:
            return 0
        found: dict = {}

        def walk(v):
            for k, t in v.items() if isinstance(v, dict) else enumerate(v):
                if isinstance(t, (dict, list, tuple)):
                    walk(t)
                elif k in self.STREAM_KEYS and isinstance(t, torch.Tensor) and \
                        ops.stream_ok(1, t, gated=t.dim() == 3 or k == "gate_up"):
                    found[t.data_ptr()] = t

        walk(self.w["layers"])
        total = sum(t.numel() * t.element_size() for t in found.values())
        cap = torch.cuda.get_device_properties(self.device).total_memory * self.stream_budget_frac
        if total > cap:
            return 0
        self._streams = {p: (t, version(t), ops.stream_pack(t)) for p, t in found.items()}
        return total

    def _stream_weight(self, M: int, w: torch.Tensor, gated: bool = False):
        """(weight, packed) for a layer of the streaming kernel, or None where it does not cover
        the weight."""
        if self.tp != 1 or not ops.stream_ok(M, w, gated):
            return None
        t = packed_copy(self, w)
        return (w, False) if t is None else (t, True)

    def _few(self, epi: int, x: torch.Tensor, w: torch.Tensor, slabs: bool = False, **kw):
        """A plain (epi 0) or gated (1) projection of up to 256 rows: its rows or, with ``slabs``,
        perhaps its slabs; None for more rows and what the kernels do not cover."""
        if self.tp != 1:
            return None
        t = few_weight(self, x.shape[0], w, epi == 1, slabs)
        return None if t is None else ops.few_rows(epi, x, *t, slabs=slabs, **kw)

    # Projections return either a bf16 tensor (library / gemm.hip path, not yet
    # TP-reduced) or :class:`Parts` (fp32 split-K slabs of the weight-streaming
    # kernel, wgemm.hip), which the NEXT kernel reduces while doing its own work:
    # QKV parts -> splitk_rope_kv (RoPE + paged KV write), O / down parts ->
    # splitk_add_rmsnorm (residual add + RMSNorm), gate_up parts -> splitk_swiglu.
    def _wcfg(self, M: int, N: int, K: int, mode: int, is_decode: bool,
              w: torch.Tensor | None = None, slabs: bool = True):
        """The tables' entry for a projection, None where ``w`` runs on the few-row kernels or the
        library."""
        if self.device.type != "cuda" or self.dtype != torch.bfloat16:
            return None
        if not is_decode:
            # mid-size steps below the prefill tile's row threshold: split-K on
            # the 256x256 tile where the table lists a win (ops.midm_config)
            if self.tp == 1 and self.use_pgemm and M < self._min_rows:
                cfg = ops.midm_config(M, N, K, mode)
                return cfg if cfg is None or mode else \
                    (*cfg[:2], ops.midm_slices(M, N, K, cfg[2]))
            return None  # up to 256 rows among them
        # up to 192 rows the few-row kernels come before the tables.  With the consumer's reads of
        # the slabs, us at 64 / 128 / 192 rows, packed panel (fp32 slabs) and table (fp16 from 65
        # rows on): 6144 x 4096 18 / 22 / 26 and 19 / 20 / 24; 4096 x 4096 14 / 19 / 25 and 18 /
        # 17 / 19; 4096 x 14336 28 / 36 / 41 and 33 / 37 / 38; gated 28672 x 4096 44 / 53 / 56 and
        # (library at 64, 128) 56 / 62 / 62.  Beyond, the tables by more: 256 rows 28 and 25, 28
        # and 21, 49 and 45, 69 and 66
        if M <= 192 and w is not None and self.tp == 1 and \
                few_weight(self, M, w, mode == 1, slabs):
            return None
        # the prefill tile asks of decode steps what it asks of others (False); else the table's tgemm
        if self._pgemm_covers(K, N << mode, False) and \
                (w is None or (w.is_contiguous() and ops._on_grid(w))):
            cfg = ops.decode_tile_config(M, N, K, mode)
            if cfg is not None:
                return cfg
        return ops.wgemm_config(M, N, K, mode)

    # split-K slabs of the tile GEMMs in fp16 (tgemm mode 3, pgemm): half the slab bytes
    # the producer writes and the consumer (splitk.hip) reads; each slab is one
    # K-slice's fp32 sum rounded to 11 bits, finer than the bf16 rounding of the
    # projection output itself.  OMNIA_SPLITK_FP32=1 keeps fp32 slabs.
    splitk_half = os.environ.get("OMNIA_SPLITK_FP32", "0") != "1"

    def _slab_dtype(self, nwaves: int) -> torch.dtype:
        return torch.float16 if (self.splitk_half and nwaves < 0) else torch.float32

    def _wgemm(self, mode: int, x: torch.Tensor, w: torch.Tensor, S: int, nw: int, nwaves: int,
               out: torch.Tensor | None = None) -> torch.Tensor:
        """ops.wgemm, on the tile-packed copy of ``w`` when one exists for this
        tgemm config; split-K slabs in fp16 on the tile GEMM (``out``'s dtype)."""
        if nwaves == ops.PGEMM_SPLIT:
            return ops.pgemm_splitk(x, w, S, out, cols=nw, uneven=True)
        if nwaves < 0 and mode == 2 and out is not None and out.dtype == torch.float16:
            mode = 3
        packed = getattr(self, "_packed", None)
        if packed and nwaves < 0:
            src, at, wp = packed.get((w.data_ptr(), nw, 1 if mode == 1 else 0), (None, 0, None))
            if wp is not None and unchanged(w, src, at):
                return ops.tgemm(mode, x, wp, S, nw, (-1 - nwaves) | 8, out)
        if mode == 3:
            return ops.tgemm(3, x, w, S, nw, -1 - nwaves, out)
        return ops.wgemm(mode, x, w, S, nw, nwaves, out=out)

    def _parts(self, tag, S: int, M: int, N: int,
               dtype: torch.dtype = torch.float32) -> torch.Tensor:
        if M > ops.WGEMM_MAX_M:  # mid-size steps: M varies per step, do not pin one per M
            return torch.empty(S, M, N, dtype=dtype, device=self.device)
        key = ("parts", tag, S, M, N, dtype)
        buf = self._ws.get(key)
        if buf is None:
            buf = torch.empty(S, M, N, dtype=dtype, device=self.device)
            self._ws[key] = buf
        return buf

    def _proj(self, tag, x: torch.Tensor, w: torch.Tensor, is_decode: bool, slabs: bool = True):
        """Plain projection: Parts on the split-K paths (unless ``slabs`` is off), else bf16."""
        M, K = x.shape
        if tag in ("o", "down") and not is_decode and overlap.applies(M, x.device):
            return RowPar(x, w)
        if self._pgemm_ok(M, K, w.shape[0], is_decode):
            return ops.pgemm(0, x, w)
        cfg = self._wcfg(M, w.shape[0], K, 0, is_decode, w) if slabs else None
        if cfg is None:
            # a gate and up that come here take the activation kernel as well: no slabs for it
            y = None if M > ops.PANEL_MAX_M else \
                self._few(0, x, w, slabs and not tag.endswith("gate_up"))
            if y is not None:
                return y if y.dim() == 2 else Parts(y)
            return self._mid(x, w, is_decode, slabs and not tag.endswith("gate_up"))
        nw, nwaves, S = cfg
        return Parts(self._wgemm(2, x, w, S, nw, nwaves,
                                 out=self._parts(tag, S, M, w.shape[0], self._slab_dtype(nwaves))))

    def _mid(self, x: torch.Tensor, w: torch.Tensor, is_decode: bool, slabs: bool):
        """More rows than the few-row kernels take and fewer than ``_pgemm_ok`` asks for: the
        prefill tile where it fills the chip, whole or in slices of K (fp32 :class:`Parts`), smaller
        tiles where those do (:func:`ops.small_tile_cols`), else the library."""
        M, K = x.shape
        if M > ops.PANEL_MAX_M and self.tp == 1 and ops._on_grid(x, w) and \
                self._pgemm_covers(K, w.shape[0], is_decode):
            if ops.plain_tile_fills(M, w):
                return ops.pgemm(0, x, w)
            S = 0
            if slabs and ops.midm_on() and w.is_contiguous():
                S = ops.tile_slices(M, w.shape[0], K)
            if S:
                out = torch.empty(S, M, w.shape[0], dtype=torch.float32, device=x.device)
                return Parts(ops.pgemm_splitk(x, w, S, out, cols=128))
            return ops.linear(x, w, tiles=True)
        return ops.linear(x, w)

    _min_rows = int(os.environ.get("OMNIA_PGEMM_MIN_ROWS", "2049"))  # this forward's threshold (mixed steps: the higher one)

    def _pgemm_ok(self, M: int, K: int, N: int, is_decode: bool,
                  gated: torch.Tensor | None = None) -> bool:
        """A prefill-sized projection the hand 256x256 MFMA kernel covers (the
        unfused paths: TP shards, MoE attention, CP): K whole 128-k iterations,
        N whole column tiles (``gated``: of a gate's and an up's half, N features
        each of this weight), and at least this forward's row threshold, or for a
        gated one tiles that fill the chip."""
        return (self._pgemm_covers(K, N if gated is None else 2 * N, is_decode)
                and N % (256 if gated is None else 128) == 0
                and (M >= self._min_rows or (gated is not None and ops.gated_tile_pays(M, gated))))

    def _pgemm_covers(self, K: int, R: int, is_decode: bool) -> bool:
        # TP ranks rehearsed on ONE device (ipc transport) keep the library GEMMs:
        # a 256x256 tile's 160 KB of LDS cannot share a CU with the peers'
        # spinning all-reduce blocks, so a rank's GEMM can wait out their spin
        # bound (the comm.hip error flag) -- real TP has one rank per GPU
        return (self.use_pgemm and not is_decode and K % 128 == 0 and R % 128 == 0
                and self.device.type == "cuda" and self.dtype == torch.bfloat16
                and not shared_device(self))
