"""Kernel front-end for the in-node engine.

On a GPU tensor every op runs the hand-written gfx950 HIP kernel from
``_omnia_kernels.so`` -- and fails LOUDLY if the extension is missing (a silent
eager fallback would hide a broken build).  On CPU tensors the plain-PyTorch
reference in :mod:`omnia_amd.ops.reference` runs instead (the CPU test-suite and
the mock/CPU engine path).
"""
from __future__ import annotations

import contextlib
import functools
import importlib
import os
import threading

import torch
import torch.nn.functional as F

from . import checks
from . import reference as ref

_lock = threading.Lock()
_ext = None
_ext_err: Exception | None = None


def kernels():
    """Return the loaded extension module, building it in-tree on first use if needed."""
    global _ext, _ext_err
    if _ext is not None:
        return _ext
    with _lock:
        if _ext is not None:
            return _ext
        try:
            _ext = importlib.import_module("omnia_amd.ops._omnia_kernels")
        except ImportError as e:  # pragma: no cover - exercised on fresh checkouts
            if os.environ.get("OMNIA_NO_AUTOBUILD"):
                _ext_err = e
                raise RuntimeError(
                    "omnia_amd HIP extension not built; run `python -m omnia_amd.ops.build`"
                ) from e
            from .build import build

            build(verbose=True)
            _ext = importlib.import_module("omnia_amd.ops._omnia_kernels")
    return _ext


def extension_available() -> bool:
    try:
        kernels()
        return True
    except Exception:
        return False


# --------------------------------------------------------------------- ops
def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float, out: torch.Tensor | None = None):
    if x.is_cuda:
        out = torch.empty_like(x) if out is None else out
        kernels().rmsnorm(out, x, w, eps)
        return out
    r = ref.rmsnorm(x, w, eps)
    if out is not None:
        out.copy_(r)
        return out
    return r


def fused_add_rmsnorm(x: torch.Tensor, residual: torch.Tensor, w: torch.Tensor, eps: float):
    """In place: residual += x; x = rmsnorm(residual) * w.  Returns (x, residual)."""
    if x.is_cuda:
        kernels().fused_add_rmsnorm(x, residual, w, eps)
        return x, residual
    y, r = ref.fused_add_rmsnorm(x, residual, w, eps)
    x.copy_(y)
    residual.copy_(r)
    return x, residual


def rope_kv(q, k, v, positions, cos_sin, k_cache, v_cache, slots, hq, hkv, block_size):
    """Rotate q/k in place (neox) and write k/v rows into the paged cache at `slots`."""
    if q.is_cuda:
        if checks.active(q):
            checks.slots("rope_kv", slots, k_cache)
        kernels().rope_kv(q, k, v, positions, cos_sin, k_cache, v_cache, slots, hq, hkv,
                          block_size)
        return
    T = q.shape[0]
    D = q.shape[1] // hq
    qr = ref.apply_rope(q.view(T, hq, D), positions, cos_sin)
    kr = ref.apply_rope(k.reshape(T, hkv, D), positions, cos_sin)
    q.copy_(qr.view(T, hq * D))
    k.copy_(kr.reshape(T, hkv * D))
    if slots is not None:
        ref.write_kv(k_cache, v_cache, kr, v.reshape(T, hkv, D), slots)


# ------------------------------------------------------- decode GEMM (K3/K8/K9/K10)
DGEMM_MAX_M = 256
_DGEMM_WS_FLOATS = 16 << 20  # 64 MiB of split-K slabs per device
_DGEMM_CNT = 8192
_dgemm_ws: dict = {}
_dgemm_table: dict | None = None
_dgemm_on = os.environ.get("OMNIA_DGEMM", "1") != "0"
_dgemm_force = os.environ.get("OMNIA_DGEMM", "") == "force"


_dgemm_branch = 0  # which of a step's concurrent streams calls (see on_branch)


def _dgemm_key(dev: torch.device, branch: int):
    i = dev.index if dev.index is not None else torch.cuda.current_device()
    return (i, branch) if branch else i


@contextlib.contextmanager
def on_branch(n: int, stream):
    """Run on ``stream`` beside the main one, as branch ``n`` > 0 of a step: kernels with a
    workspace take that branch's (``dgemm_prepare(device, n)``)."""
    global _dgemm_branch
    was, _dgemm_branch = _dgemm_branch, n
    try:
        with torch.cuda.stream(stream):
            yield
    finally:
        _dgemm_branch = was


def dgemm_prepare(device, branch: int = 0) -> None:
    """Allocate the split-K workspace + zeroed tile counters for ``device``, for each of the
    streams that work at the same time its own.

    Call eagerly (model init) so nothing is allocated while a hipGraph captures."""
    dev = torch.device(device)
    if dev.type != "cuda":
        return
    key = _dgemm_key(dev, branch)
    if key not in _dgemm_ws:
        _dgemm_ws[key] = (torch.empty(_DGEMM_WS_FLOATS, dtype=torch.float32, device=dev),
                          torch.zeros(_DGEMM_CNT, dtype=torch.int32, device=dev))


def _dgemm_tuned() -> dict:
    global _dgemm_table
    if _dgemm_table is None:
        import json

        p = os.path.join(os.path.dirname(__file__), "tuned", "dgemm_mi355x.json")
        tab = {}
        if os.path.exists(p):
            with open(p) as f:
                for k, v in json.load(f).items():
                    tab[k] = tuple(v)
        _dgemm_table = tab
    return _dgemm_table


DGEMM_BUCKETS = (8, 32, 64, 128, 256)


def dgemm_bucket(M: int) -> int:
    for b in DGEMM_BUCKETS:
        if M <= b:
            return b
    return 0


def dgemm_config(M: int, N: int, K: int, mode: int, force: bool | None = None
                 ) -> tuple[int, int, int] | None:
    """(wm, wn, splits) for a decode GEMM, or None to use hipBLASLt.

    Dispatch is measured, not assumed: ``ops/tuned/dgemm_mi355x.json`` (written
    by ``scripts/dgemm_sweep.py`` on an MI355X, keyed ``mode:Mbucket:N:K``) lists
    the shapes where the hand kernel beat the tuned hipBLASLt solution; every
    other shape stays on the library.  ``force`` (or ``OMNIA_DGEMM=force``) uses
    the heuristic config for any covered shape (tests, sweeps)."""
    if M < 1 or M > DGEMM_MAX_M or K % 64:
        return None
    wm = 1 if M <= 64 else 2 if M <= 128 else 4
    hit = _dgemm_tuned().get(f"{mode}:{dgemm_bucket(M)}:{N}:{K}")
    if hit is not None:
        return tuple(hit)
    if not (force if force is not None else _dgemm_force):
        return None
    wn = 2
    cols = 64 * wn if mode == 0 else 32 * wn
    if N % cols:
        wn = 1
        cols = 64 if mode == 0 else 32
        if N % cols:
            return None
    tiles = N // cols
    s = 1
    while (tiles * s < 256 and s < 8 and K % (64 * s * 2) == 0
           and N * (s * 2) * 64 * wm * ((M + 64 * wm - 1) // (64 * wm))
           * (1 if mode == 0 else 2) <= _DGEMM_WS_FLOATS):
        s *= 2
    return wm, wn, s


def _dgemm(mode: int, x: torch.Tensor, w: torch.Tensor, out: torch.Tensor | None):
    if not (_dgemm_on and x.is_cuda and x.dim() == 2 and x.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16 and w.is_contiguous()):
        return None
    M, K = x.shape
    N = w.shape[0] if mode == 0 else w.shape[0] // 2
    cfg = dgemm_config(M, N, K, mode)
    if cfg is None:
        return None
    key = _dgemm_key(x.device, _dgemm_branch)
    if key not in _dgemm_ws:
        dgemm_prepare(x.device, _dgemm_branch)
    ws, cnt = _dgemm_ws[key]
    x = x.contiguous()
    out = x.new_empty(M, N) if out is None else out
    wm, wn, s = cfg
    kernels().dgemm(mode, out, x, w, ws, cnt, s, wm, wn)
    return out


# ------------------------------------------ weight-streaming decode GEMM (wgemm.hip)
WGEMM_MAX_M = 256


_wgemm_table: dict | None = None
_wgemm_on = os.environ.get("OMNIA_WGEMM", "1") != "0"
WGEMM_BUCKETS = (16, 32, 64, 128, 192, 256)
PGEMM_SPLIT = -64  # table nwaves code: pgemm's tile, in slices fp16 slabs (or ``out``'s fp32)


def wgemm_config(M: int, N: int, K: int, mode: int) -> tuple[int, int, int] | None:
    """(nw, nwaves, splits) of the weight-streaming kernel for a decode projection
    (nwaves == 0 selects the wide-batch 32x32x16 kernel, wgemm_wide.hip, with nw
    32-column tiles per wave; nwaves < 0 the full-batch tile kernel, tgemm.hip,
    with nw weight rows per block and non-temporal weight loads when -2;
    nwaves == PGEMM_SPLIT the 256x256 split-K tile, pgemm.hip EPI 4, 11),
    or None to keep the library / gemm.hip path.  ``mode`` 0 = plain projection
    (its split-K slabs are reduced by the consumer kernel), 1 = gate_up + SwiGLU.
    Measured dispatch: ``ops/tuned/wgemm_mi355x.json`` (scripts/wgemm_sweep.py +
    scripts/wgemm_table.py) lists only the shapes where it won on an MI355X."""
    global _wgemm_table
    if not _wgemm_on or M < 1 or M > WGEMM_MAX_M:
        return None
    if _wgemm_table is None:
        import json

        p = os.path.join(os.path.dirname(__file__), "tuned", "wgemm_mi355x.json")
        _wgemm_table = {}
        if os.path.exists(p):
            with open(p) as f:
                _wgemm_table = {k: tuple(v) for k, v in json.load(f).items()}
    b = next(x for x in WGEMM_BUCKETS if M <= x)
    cfg = _wgemm_table.get(f"{mode}:{b}:{N}:{K}")
    if cfg is None and b == 192:  # the 192 bucket only lists its own wins
        cfg = _wgemm_table.get(f"{mode}:256:{N}:{K}")
    return cfg


_decode_tiles: dict | None = None


def decode_tile_config(M: int, N: int, K: int, mode: int) -> tuple[int, int, int] | None:
    """(columns, PGEMM_SPLIT, splits) of the prefill tile (``csrc/pgemm.hip``, in slices EPI 4, 11, one of
    a gate_up whole, EPI 1) for decode projections of 193 to 256 rows that it runs in the place of
    :func:`wgemm_config`'s entry, where a model may use it (``ops/tuned/decode_tile_mi355x.json``), or
    None.  us, weights from HBM, tgemm on packed copies / so, at 193, 224 and 256 rows: gated 28672 x 4096
    68.6 / 65.2, 69.8 / 63.8, 71.1 / 64.4; 4096 x 14336 38.6 / 36.8, 38.2 / 37.5, 39.0 / 37.6.  In a model's
    step under the trace, by the run, 66.9 to 69.9 / 63.6 to 68.7 and 37.8 to 39.9 / 38.3 to 38.9; the step is
    1.01 to 1.04 times as fast.  Not 8192 x 28672, with its consumer (row-major) 126 / 126, 129 / 125, 129 /
    129."""
    global _decode_tiles
    if not _wgemm_on or not 192 < M <= WGEMM_MAX_M:
        return None
    if _decode_tiles is None:
        import json

        p = os.path.join(os.path.dirname(__file__), "tuned", "decode_tile_mi355x.json")
        _decode_tiles = {}
        if os.path.exists(p):
            with open(p) as f:
                _decode_tiles = {k: (v[0], PGEMM_SPLIT, v[1]) for k, v in json.load(f).items()}
    return _decode_tiles.get(f"{mode}:{N}:{K}")


MIDM_BUCKETS = (512, 768, 1024, 1536, 2048, 3072, 4096)
_midm_table: dict | None = None
_midm_on = os.environ.get("OMNIA_MIDM", "1") != "0"


def midm_on() -> bool:
    return _midm_on


def midm_config(M: int, N: int, K: int, mode: int) -> tuple[int, int, int] | None:
    """Mid-size projections (M = 257..4096 rows: open-loop mixed steps, which
    the unsplit 256x256 prefill tile under-fills): ``(256, PGEMM_SPLIT, S)``
    when ``ops/tuned/midm_mi355x.json`` lists a split-K win of the 256x256 tile
    (+ its slab consumer) over the library path for this shape's M bucket
    (``scripts/midm_sweep.py``), else None (library GEMM)."""
    global _midm_table
    if not (_wgemm_on and _midm_on) or M <= WGEMM_MAX_M or M > MIDM_BUCKETS[-1]:
        return None
    if _midm_table is None:
        import json

        p = os.path.join(os.path.dirname(__file__), "tuned", "midm_mi355x.json")
        _midm_table = {}
        if os.path.exists(p):
            with open(p) as f:
                _midm_table = {k: int(v) for k, v in json.load(f).items()}
    b = next(x for x in MIDM_BUCKETS if M <= x)
    S = _midm_table.get(f"{mode}:{b}:{N}:{K}")
    return (256, PGEMM_SPLIT, S) if S else None


@functools.lru_cache(maxsize=8192)
def midm_slices(M: int, N: int, K: int, S: int) -> int:
    """Slices of K, uneven ones among them, for ``M`` rows of a weight [N, K] on the wide tile where
    :func:`midm_config` says ``S``: more where rows of its bucket leave CUs without a tile, by what a
    K-tile of 64 and an fp16 slab's write and read take.  us with the consumer, the table's / more: 4096 x 14336
    at 600 rows 87.8 / 78.4, 1100 142 / 119; 4096 x 4096 36.6 / 35.1, 54.8 / 48.8; 6144 x 4096 at 257 / 300 /
    400 / 512 35.4 / 36.0, 35.3 / 33.8, 36.3 / 34.9, 37.2 / 36.9, at 600 / 768 52.1 / 45.0, 50.8 / 45.8; 10240
    x 8192 at 257 / 400 / 512 96 / 78, 90 / 79, 91 / 80.  The same numbers do for fp32 slabs (OMNIA_SPLITK_FP32;
    6144 x 4096 at 400 / 512 / 768 42.6 / 42.0, 44.6 / 44.7, 56.9 / 54.5; 4096 x 4096 at 600 / 1100 42.6 /
    41.6, 58.5 / 54.4; 4096 x 14336 92.7 / 85.4, 148 / 127), where by twice the bytes the first, second and
    fourth of these would not be cut.  Never fewer, as each fp16 slab saturates."""
    tiles, nk = -(-M // 256) * (N // 256), K // 64

    def us(s):
        return -(-nk // s) * 1.35 + s * M * N * 2 * (1 / 3.6e6 + 1 / 7e6)

    best = S
    for s in range(S + 1, 17):
        if tiles * s <= 256 and us(s) < 0.98 * us(best):
            best = s
    return best


def wgemm(mode: int, x: torch.Tensor, w: torch.Tensor, splits: int = 1, nw: int = 2,
          nwaves: int = 4, out: torch.Tensor | None = None) -> torch.Tensor:
    """Decode GEMM with W streamed HBM -> MFMA registers (``csrc/wgemm.hip``).

    mode 0: bf16 ``x @ w.T``; mode 1: bf16 ``silu(x Wg^T) * (x Wu^T)`` with
    ``w = [Wg; Wu]``; mode 2: fp32 split-K partial slabs ``[splits, M, N]`` whose
    sum is ``x @ w.T`` (reduced by the consumer kernel)."""
    if nwaves == PGEMM_SPLIT:  # table code for the prefill tile in slices
        if mode not in (2, 3):
            raise ValueError("the pgemm split-K table entry produces slabs (mode 2/3)")
        return pgemm_splitk(x, w, splits, out, cols=nw)
    if nwaves == 0:  # table code for the wide-batch kernel: nw = 32-col tiles per wave
        return wgemm_wide(mode, x, w, splits, nw, out)
    if nwaves < 0:  # table code for the full-batch tile kernel: nw = weight rows per block,
        # -1 - nwaves = tgemm flags (bit 0 non-temporal W, bit 1 32-k stages)
        return tgemm(mode, x, w, splits, nw, -1 - nwaves, out)
    M, K = x.shape
    N = w.shape[0] // 2 if mode == 1 else w.shape[0]
    if out is None:
        out = (torch.empty(splits, M, N, dtype=torch.float32, device=x.device) if mode == 2
               else x.new_empty(M, N))
    kernels().wgemm(mode, out, x.contiguous(), w, splits, nw, nwaves)
    return out


def wgemm_wide(mode: int, x: torch.Tensor, w: torch.Tensor, splits: int = 1, wt: int = 2,
               out: torch.Tensor | None = None) -> torch.Tensor:
    """Wide-batch (128 < M <= 256) weight-streaming decode GEMM on 32x32x16 MFMA
    (``csrc/wgemm_wide.hip``); same modes and outputs as :func:`wgemm`."""
    M, K = x.shape
    N = w.shape[0] // 2 if mode == 1 else w.shape[0]
    if out is None:
        out = (torch.empty(splits, M, N, dtype=torch.float32, device=x.device) if mode == 2
               else x.new_empty(M, N))
    kernels().wgemm_wide(mode, out, x.contiguous(), w, splits, wt)
    return out


def tgemm(mode: int, x: torch.Tensor, w: torch.Tensor, splits: int = 1, bn: int = 128,
          wnt: int = 0, out: torch.Tensor | None = None) -> torch.Tensor:
    """Tile GEMM (``csrc/tgemm.hip``; mode 3 = mode 2's split-K slabs in fp16):
    decode batches (M <= 256, one block owns all
    rows x ``bn`` weight rows) and prefill chunks (256-row tiles), both operands LDS-DMA staged through an
    NS-deep ring with counted waits.  Same modes / outputs as :func:`wgemm`
    (mode 1 = fused SwiGLU needs ``splits == 1``).  ``wnt`` bit 0: non-temporal
    weight loads; bit 1: 32-k ring stages (twice the stages in flight, BN >= 128)."""
    M, K = x.shape
    N = w.shape[0] // 2 if mode == 1 else w.shape[0]
    if out is None:
        out = (torch.empty(splits, M, N, device=x.device,
                           dtype=torch.float32 if mode == 2 else torch.float16) if mode >= 2
               else x.new_empty(M, N))
    if not x.is_cuda:
        r = x.float() @ w.float().t()
        if mode == 1:
            r = ref.silu_mul(r.to(x.dtype)).float()
        if mode >= 2:
            out.zero_()
            out[0].copy_(r)
        else:
            out.copy_(r.to(out.dtype))
        return out
    kernels().tgemm(mode, out, x.contiguous(), w, splits, bn, wnt)
    return out


def tgemm_pack(w: torch.Tensor, bn: int, mode: int) -> torch.Tensor:
    """``w`` [R, K] re-laid for ``tgemm`` (wnt bit 3): [tile][k-stage][bn rows][64],
    the rows of each tile in the kernel's order (mode 1: every wave's gate rows
    then the matching up rows of W = [Wg; Wu]) and each row's eight 16-B chunks
    pre-permuted by the LDS bank swizzle (stored chunk p = chunk p ^ (row & 7)),
    so one k-stage of a tile is one contiguous run the LDS-DMA reads lane by
    lane.  Returned with the original [R, K] shape (same elements, new order)."""
    R, K = w.shape
    BK = 64
    if K % BK:
        raise ValueError("tgemm_pack: K must be a multiple of 64")
    nk = K // BK
    wtn = bn // (4 if bn >= 256 else 2)
    dev = w.device
    rr = torch.arange(bn, device=dev)
    if mode == 1:
        N = R // 2
        ntiles = N // (bn // 2)
        wv, q = rr // wtn, rr % wtn
        f0 = torch.arange(ntiles, device=dev)[:, None] * (bn // 2) + (wv * (wtn // 2))[None, :]
        rows = torch.where((q < wtn // 2)[None, :], f0 + q[None, :], N + f0 + (q - wtn // 2)[None, :])
    else:
        ntiles = R // bn
        rows = torch.arange(ntiles, device=dev)[:, None] * bn + rr[None, :]
    if ntiles * bn != R:
        raise ValueError("tgemm_pack: rows are not a whole number of tiles")
    t = w[rows.reshape(-1)].view(ntiles, bn, nk, 8, 8)
    perm = torch.arange(8, device=dev)[None, :] ^ (rr[:, None] & 7)  # [bn, 8]
    t = torch.gather(t, 3, perm[None, :, None, :, None].expand(ntiles, bn, nk, 8, 8))
    return t.permute(0, 2, 1, 3, 4).contiguous().view(R, K)


def pgemm(epi: int, x: torch.Tensor, w: torch.Tensor, out: torch.Tensor | None = None,
          ss_in: torch.Tensor | None = None, inv_d: float = 0.0, eps: float = 0.0,
          ss_out: torch.Tensor | None = None, positions=None, cos_sin=None, k_cache=None,
          v_cache=None, slots=None, hq: int = 0, hkv: int = 0, block_size: int = 0,
          bias: torch.Tensor | None = None, gelu: bool = False, cols: int = 0):
    """Prefill GEMM ``x @ w.T`` with a fused epilogue (``csrc/pgemm.hip``).

    ``ss_in`` ([M, n] fp32 partial row sums of squares of ``x``) scales row r by
    ``rsqrt(sum(ss_in[r]) * inv_d + eps)`` -- RMSNorm with the norm weight folded
    into ``w``.  epi 0: out = scaled GEMM; 1: out = silu(g) * u with
    ``w = [Wg; Wu]`` (``bias`` fp32 [2N], unscaled only: ``silu(g + bg) * (u + bu)``;
    ``gelu``, unscaled only: ``gelu_tanh(g) * u``);
    2: ``out`` is the residual, updated in place (out += GEMM)
    with ``ss_out[r, t]`` = sum of squares of its new 256-column slice t;
    3: QKV -> RoPE'd q in ``out`` [M, hq*128], RoPE'd k and v written to the
    paged caches at ``slots``.  ``cols``: weight rows of a tile, 256 or (epi 0, 1) 128, to the
    same bits; of 256, a last round's are cut in two where that fills the chip better.  0: 128 where
    all tiles are one round of that, which the kernel of both has 0.4 us more to find, else 256."""
    M, K = x.shape
    N = w.shape[0] // 2 if epi == 1 else w.shape[0]
    if out is None:
        out = x.new_empty(M, hq * 128 if epi == 3 else N)
    if x.is_cuda:
        if epi == 3 and checks.active(x):
            checks.slots("pgemm qkv", slots, k_cache)
        if not cols and epi <= 1 and tile_cols(M, w.shape[0]) == 128 and \
                _tile_rounds(M, w.shape[0], 128) == 1:
            cols = 128
        kernels().pgemm(epi, out, x.contiguous(), w, ss_in, inv_d, eps, ss_out, positions,
                        cos_sin, k_cache, v_cache, slots, hq, hkv, block_size, bias, gelu, cols)
        return out
    h = x.float() @ w.float().t()
    if bias is not None:
        h = h + bias
    if ss_in is not None and epi != 2:
        h = h * torch.rsqrt(ss_in.float().sum(1) * inv_d + eps)[:, None]
    if epi == 0:
        out.copy_(h.to(out.dtype))
    elif epi == 1:
        a = F.gelu(h[:, :N], approximate="tanh") if gelu else F.silu(h[:, :N])
        out.copy_((a * h[:, N:]).to(out.dtype))
    elif epi == 2:
        new = (out.float() + h.to(out.dtype).float()).to(out.dtype)
        out.copy_(new)
        ss_out.copy_(new.float().pow(2).view(M, -1, 256).sum(-1))
    else:
        D = 128
        qkv = h.to(out.dtype)
        qq = ref.apply_rope(qkv[:, : hq * D].reshape(M, hq, D), positions, cos_sin)
        kk = ref.apply_rope(qkv[:, hq * D:(hq + hkv) * D].reshape(M, hkv, D), positions, cos_sin)
        vv = qkv[:, (hq + hkv) * D:].reshape(M, hkv, D)
        keep = slots >= 0
        ref.write_kv(k_cache, v_cache, kk[keep], vv[keep], slots[keep])
        out.copy_(qq.reshape(M, hq * D))
    return out


def _tile_rounds(M: int, R: int, cols: int) -> int:
    return -(-(-(-M // 256) * (R // cols)) // 256)


@functools.lru_cache(maxsize=8192)
def tile_cols(M: int, R: int) -> int:
    """Columns of a tile for ``M`` rows and ``R`` weight rows, were all alike: 128 where that fills
    the rounds over 256 CUs better, by more than its second read of x.  A round of narrow tiles
    takes 0.57 to 0.6 of a wide one's (us wide / narrow and their rounds: gated 16384 x 2048 at 300
    rows 43.8 / 31.2 (1, 1), 600 45.6 / 54.4 (1, 2), 1536 92.5 / 87.0 (2, 3), 2001 103 / 120 (2,
    4); 28672 x 4096 at 600 165 / 149 (2, 3), 1280 253 / 266 (3, 5); plain 4096 x 2048 at 2001
    42.6 / 30.6 (1, 1))."""
    narrow = R % 256 == 0 and 0.6 * _tile_rounds(M, R, 128) < 0.97 * _tile_rounds(M, R, 256)
    return 128 if narrow else 256


def _tiles_useful(M: int, R: int) -> float:
    """Part of the work of :func:`pgemm`'s rounds that is not padding."""
    cols = tile_cols(M, R)
    return M * R / (256 * 256 * cols * _tile_rounds(M, R, cols))


def _cut_rounds(tiles: int) -> float:
    """Rounds over 256 CUs that wide tiles take where those of the last are cut in two if they fill
    half of it or less."""
    return tiles // 256 + (0.0, 0.6, 1.0)[(tiles % 256 > 0) + (tiles % 256 > 128)]


def gated_tile_fills(M: int, w: torch.Tensor) -> bool:
    """Whether a gated :func:`pgemm` of more rows than the panel kernel takes covers ``w`` = [Wg; Wu]
    and its wide tiles (128 features) are worth their rounds over 256 CUs: from three quarters of
    their work useful, the activation in the epilogue makes up for the rest (useful part, us here / library and
    activation kernel; 8192 features of 2048: 512 rows .50 48 / 42, 768 .75 51.5 / 52.7, 999 .98
    55 / 67, 1536 .75 99 / 99, 2001 .98 108 / 124; 14336 of 4096: 320 .55 93 / 88, 512 .88 99 / 112,
    768 .66 177 / 163, 999 .85 187 / 198)."""
    if M <= PANEL_MAX_M:
        return False
    N = w.shape[0] // 2
    rounds = -(-(-(-M // 256) * (N // 128)) // 256)
    return M * N > 0.75 * 256 * 256 * 128 * rounds and \
        w.is_contiguous() and _on_grid(w)


def gated_tile_pays(M: int, w: torch.Tensor) -> bool:
    """:func:`gated_tile_fills` of the wide tile or, by the same line, of the narrow one where
    :func:`tile_cols` takes that (us, here / library and activation kernel: 8192 features of 2048 at
    300 rows .59 useful 31.2 / 35.1, 512 1.0 32.8 / 40.9); of more than a round of wide tiles, whose
    last ones are cut in two, from .67 of :func:`_cut_rounds` useful (14336 of 4096 at 600 .64 144 / 144,
    800 .68 180 / 187, 1100 .72 229 / 242, 1280 .84 235 / 258, 1700 .81 310 / 348; 8192 of 2048 at
    1100 .67 72 / 84, 1280 .78 74.3 / 86.7)."""
    R = w.shape[0]
    if gated_tile_fills(M, w):
        return True
    if M <= PANEL_MAX_M or R % 256 or not (w.is_contiguous() and _on_grid(w)):
        return False
    tiles = -(-M // 256) * (R // 256)
    return (tile_cols(M, R) == 128 and _tiles_useful(M, R) > 0.75) or \
        (tiles > 256 and M * R > 0.67 * 256 ** 3 * _cut_rounds(tiles))


def plain_tile_fills(M: int, w: torch.Tensor) -> bool:
    """Whether an ungated :func:`pgemm` of more rows than the panel kernel takes covers ``w`` and
    beats the library: one round of narrow tiles with nine tenths of their work useful (useful part,
    us here / library: 4096 x 2048 at 1536 rows .75 28.9 / 29.3, 2001 .98 30.6 / 34.6; 4096 x 4096 at
    1536 .75 52.0 / 51.6, 2001 .98 55 / 60; 4096 x 14336 at 1536 .75 180 / 176, 2001 .98 194 / 204;
    2048 x 2048 at 2001 .49 27.1 / 23.8).  Over 28 such sizes the library takes 1.02 to 1.14 as long;
    over 32 of three narrow rounds .86 to 1.6, most of them less (15360 x 5120 at 1448 rows 216 /
    192), over 18 of one wide round .95 to 1.04."""
    if M <= PANEL_MAX_M or w.dim() != 2:
        return False
    R, K = w.shape
    return K % 128 == 0 and R % 256 == 0 and _tiles_useful(M, R) > 0.9 and \
        tile_cols(M, R) == 128 and _tile_rounds(M, R, 128) == 1 and w.is_contiguous() and _on_grid(w)


def small_tile_cols(M: int, w: torch.Tensor) -> int:
    """Columns (128, 64) of the tile on which :func:`pgemm_small` beats the library for more rows than the
    panel kernel takes, 0: none.  One round of its tiles over 256 CUs, .55 of their work useful, where K is
    long three quarters, of the smaller .65 (useful part, us here / library: 128 columns: 4096 x 2048 at 512
    rows .50 21.0 / 17.0; 2048 x 2048 at 1300 .63 17.7 / 21.7, 2001 .98 19.0 / 21.7; 4608 x 2048 at 508 .56
    18.4 / 21.2; 3072 x 1024 at 999 .73 11.6 / 14.3; 2048 x 512 at 2048 1.0 8.9 / 11.1; 4096 x 4096 at 700
    .68 34.3 / 32.6, 999 .98 38.7 / 40.9; 5888 x 6144 at 512 .72 62.3 / 55.0, 3712 x 6144 at 897 .79 50.0 /
    58.5.  64: 2048 x 2048 at 512 .50 13.1 / 12.5, 700 .68 13.8 / 14.7, 999 .98 14.6 / 17.3; 4096 x 2048 at
    512 1.0 14.7 / 17.1; 1472 x 512 at 1075 .75 6.9 / 10.3; 1600 x 2560 at 726 .55 16.9 / 17.3, 2688 x 2560
    at 550 .70 17.6 / 17.4; 3584 x 4096 at 393 .67 24.5 / 29.2; 2048 x 6144 at 860 .84 39.0 / 42.0).  Over
    160 such sizes the library takes .99 to 1.5 as long.  Models ask for whole 128 of rows and K
    (``Projections._pgemm_covers``), :func:`linear` for any of these."""
    return small_cols(M, *w.shape) if w.dim() == 2 and w.is_contiguous() and _on_grid(w) else 0


def small_cols(M: int, R: int, K: int) -> int:
    """:func:`small_tile_cols` of a contiguous weight [R, K] on the 16-byte grid."""
    if M <= PANEL_MAX_M or K % 64 or K > 6144:
        return 0
    for cols, useful in ((128, 0.55 if K <= 2048 else 0.75), (64, 0.55 if K <= 2048 else 0.65)):
        if R % cols == 0 and -(-M // 128) * (R // cols) <= 256 and M * R > useful * 256 * 128 * cols:
            return cols
    return 0


def pgemm_small(x: torch.Tensor, w: torch.Tensor, cols: int = 128) -> torch.Tensor:
    """``x @ w.T`` on MFMA tiles of 128 x ``cols`` (``csrc/pgemm.hip``): whole ones of ``w``, K of whole 64;
    the bits of :func:`pgemm`."""
    if not x.is_cuda:
        return (x.float() @ w.float().t()).to(x.dtype)
    out = x.new_empty(x.shape[0], w.shape[0])
    kernels().pgemm_small(out, x.contiguous(), w, cols)
    return out


@functools.lru_cache(maxsize=8192)
def tile_slices(M: int, R: int, K: int) -> int:
    """K slices in which :func:`pgemm_splitk`'s narrow tile runs ``M`` rows of a weight [R, K] into
    fp32 slabs, where that and the consumer's reads of them take less than the library and its
    rows; 0 where not.  By what both take (us): a tile 0.67 for 64 of K and 5 besides, slabs written
    at 3.6 TB/s and read at 7, as many slices as 256 CUs take at once; the library 9, 1.9 for 1000
    of K and its products at 1.35 PFLOP/s.  With a margin, since its kernels change with every size
    (us with the consumer, library / here, rows of 2048 x 8192: 257 40.7 / 31.4, 512 41.9 / 35.0,
    768 50.5 / 43.2, 999 62.5 / 48.9, 1536 71.2 / 71.9 not taken, 2001 88.7 / 77.4; 4096 x 8192:
    512 61 / 51, 768 71 / 73 not taken; 2048 x 16384: 999 101 / 73; 2048 x 4096: 257 27.6 / 24.3,
    999 37.4 / 36.2 not taken).  That model of the library is one of 2048 rows of weights and more;
    of fewer it is faster up to K of some 5000 (1280 x 2304 at 308 rows 13.0 / 18.7, 1024 x 4608 at 432
    18.3 / 23.1, 1536 x 5120 at 257 21.9 / 24.3, but 1024 x 6144 at 257 23.4 / 21.4, 8192 at 400 28.1 /
    25.0)."""
    if M <= PANEL_MAX_M or M > 2048 or R % 128 or K % 128 or (R < 2048 and K < 6144):
        return 0
    tiles, best = -(-M // 256) * (R // 128), (0.9 * (9.0 + 1.9e-3 * K + 2 * M * R * K / 1.35e9), 0)
    for S in range(2, 17):
        if tiles * S <= 256 and K % (128 * S) == 0:
            t = 5.0 + 0.67 * K / 64 / S + M * R * (4 * S / 3.6e6 + (4 * S - 2) / 7e6)
            best = min(best, (t, S))
    return best[1]


def pgemm_splitk(x: torch.Tensor, w: torch.Tensor, splits: int, out: torch.Tensor | None = None,
                 cols: int = 0, uneven: bool = False) -> torch.Tensor:
    """Split-K slabs ``[splits, M, N]`` of ``x @ w.T`` on the MFMA tile of 256 rows and ``cols``
    (128, else 256) columns (``csrc/pgemm.hip`` EPI 4, 11).  Each
    slab is one K-slice's fp32 sum, saturated to fp16 unless ``out`` is fp32; the splitk consumers
    reduce them.  Decode projections at M <= 256 (one m-tile; the K split fills the chip).
    ``uneven``: slices of any whole 64 of K, else all alike and of whole 128."""
    M, K = x.shape
    N = w.shape[0]
    if out is None:
        out = torch.empty(splits, M, N, dtype=torch.float16, device=x.device)
    if x.is_cuda:
        kernels().pgemm_splitk(out, x.contiguous(), w, 128 if cols == 128 else 256, uneven)
        return out
    at = [s * (K // 64) // splits * 64 for s in range(splits)] + [K] if uneven else \
        range(0, K + 1, K // splits)
    for s, (a, b) in zip(range(splits), zip(at, at[1:])):
        r = x[:, a:b].float() @ w[:, a:b].float().t()
        out[s].copy_(r if out.dtype == torch.float32 else r.clamp(-65504.0, 65504.0))
    return out


# ------------------------------------------------------ projections of a few rows (stream.hip)
STREAM_MAX_M = 16
_stream_on = os.environ.get("OMNIA_STREAM", "1") != "0"


def streams_on() -> bool:
    return _stream_on


def _on_grid(*ts: torch.Tensor) -> bool:
    """Whether 16-byte loads of these tensors are aligned."""
    return all(t.data_ptr() % 16 == 0 for t in ts)


def stream_ok(M: int, w: torch.Tensor, gated: bool = False) -> bool:
    """Whether :func:`stream` and :func:`panel` cover ``M`` rows of this GPU weight
    (:func:`few_rows` chooses)."""
    if not (_stream_on and 1 <= M <= PANEL_MAX_M and w.is_cuda and w.dtype == torch.bfloat16):
        return False
    R, K = w.shape[-2:]
    return K % 64 == 0 and R % (32 if gated else 16) == 0 and w.is_contiguous() and _on_grid(w)


@functools.lru_cache(maxsize=8192)
def few_rows_pay(M: int, R: int, K: int, gated: bool, packed: bool, slabs: bool) -> bool:
    """Whether ``M`` rows of a weight [R, K] run on :func:`few_rows`' kernels rather than on the
    library's (with the activation kernel, if gated); up to 16 rows of packed ones always do.

    In slices of K (``slabs``) a panel fills the chip, and its sums reach the consumer in fp32,
    where the library rounds them to bf16: steps of 193 to 256 rows through 16 layers of 2048 are
    10 % closer to exact sums (error of the logits 0.0108, 0.0119 on the library).  So it is taken
    even where the slabs' bytes cost a little more at many rows (us with the consumer's reads of
    them, panel / library: 2048 x 2048 at 64 / 192 / 256 rows 6.1 / 11.6, 12.2 / 12.0, 14 / 11.7;
    4096 x 2048 at 193 / 256 15 / 13, 17 / 14; 2048 x 8192 at 256 23 / 27; 8256 x 2048 23 / 27;
    16512 x 4096 at 192 / 256 52 / 55, 64 / 58).
    Unsliced, a block walks all of K and takes longer the more rows it has, so few blocks lose:
    2048 x 8192 at 32 rows 32 / 16; 4096 x 4096 at 64 17 / 15; 3072 x 1024 at 128 / 256 9.5 / 12,
    17 / 12; 4096 x 2048 at 80 / 96 / 128 11.1 / 12.5, 12.7 / 13.4, 15.2 / 14.7; 1664 x 2048 at 96
    12.6 / 11.2; 10304 x 2048 at 160 / 192 / 256 21 / 24, 23.5 / 25.2, 29 / 27; 8192 x 2048 at 160
    18.3 / 17.6; gated of 4096 x 2048 at 96 / 128 / 256 14.3 / 15.7, 17.4 / 17.5, 32 / 16; 4096 x
    1024 at 128 / 160 / 192 11.6 / 14.6, 14.0 / 15.2, 16.6 / 15.6; 14336 x 4096 at 128 / 160 36 /
    38, 42 / 42; 16384 x 2048 at 192 / 256 29 / 30, 36 / 34; 28672 x 4096 at 256 76 / 81. Row-major weights of more than 0.7 GB, which the library reads at 6
    TB/s, only up to 32 rows: 57344 x 8192 at 32 / 64 / 256 rows 158 / 182, 182 / 161, 283 / 233;
    128256 x 4096 at 32 / 64 / 128 167 / 169, 205 / 173, 224 / 193 (65536 x 4096, 0.54 GB, at 64
    105 / 127). Layers 1024 wide stay here by a little more: their eager steps wait for the host,
    which these launches cost less (gated 8192 x 1024 at 160 / 256 14.1 / 16.3, 21 / 19, but a
    step of 16 such layers of 200 rows 1.23 ms / 1.74)."""
    if not packed and M > 32 and R * K > 3.5e8:
        return False
    if slabs and not gated and panel_slices(R, K) > 1:
        return True
    if M <= 64:
        return gated or K <= 2048 or R >= 12288
    if gated and K <= 1024:
        return R >= (4096 if M <= 160 else 8192)
    if M <= 96 and 2048 >= K and R >= 4096:
        return True
    if M <= 128:
        return R >= 8192 or K <= 1024
    if M <= 192:
        return R >= (10240 if K <= 2048 else 16384)
    return gated and R >= 16384  # for fp32 into the activation, at what the library takes


def few_rows(epi: int, x: torch.Tensor, w: torch.Tensor, packed: bool, slabs: bool = False,
             **kw) -> torch.Tensor:
    """A plain (epi 0) or gated (1) projection of up to 256 rows on the better kernel.

    Up to 16 rows of packed weights stream (us at 8 rows, stream / panel: 2048 x 2048 4.5 / 4.7,
    4096 x 4096 7.7 / 8.8, 16384 x 2048 14.9 / 14.4), unless few long rows leave that kernel's
    blocks few (2048 x 8192 10.7 / 8.7).  Row-major weights reach the streaming kernel in
    pieces, the panel kernel in whole lines (14.5 / 9.0; 4096 x 4096 9.5 / 8.8)."""
    R, K = w.shape
    if packed and x.shape[0] <= STREAM_MAX_M and not (slabs and R < 192 * 16 and K >= 4096):
        return stream(epi, x, w, packed=True, **kw)
    return panel(epi, x, w, packed=packed, slabs=slabs, **kw)


@functools.lru_cache(maxsize=4096)
def stream_fragments(M: int, rows: int) -> int:
    """16-row weight fragments of a block (1, 2, 4).  More of them share the block's reads of x,
    which cost about 0.3 of the weights' per 16 rows of x and fragment; fewer spread better
    over 256 CUs as long as there are few blocks (4096 rows, one / two fragments: 7.0 / 7.7 us
    at K = 4096; 6144 rows: 10.2 / 9.6, 384 blocks leaving half the CUs with twice the work)."""
    best, cost = 1, float("inf")
    for nw in (1, 2, 4):
        if rows % (16 * nw):
            break
        rounds = rows / (16 * nw * 256)
        c = (rounds if rounds > 1.6 else -(-rounds // 1)) * nw * (1.0 + 0.3 * M / 16 / nw)
        if c < cost - 1e-9:
            best, cost = nw, c
    return best


def stream_pack(w: torch.Tensor) -> torch.Tensor:
    """``w`` [..., R, K] re-laid for :func:`stream` as [R / 16][K / 64][2][4][16][8] (k step, k
    group, row, k), so that a wave reads one contiguous KB; returned with the shape of ``w``."""
    R, K = w.shape[-2:]
    if R % 16 or K % 64:
        raise ValueError("stream_pack: whole 16-row, 64-column blocks")
    t = w.reshape(-1, R // 16, 16, K // 64, 2, 4, 8).permute(0, 1, 3, 4, 5, 2, 6)
    return t.contiguous().view(w.shape)


def stream_sums(M: int, w: torch.Tensor, device) -> torch.Tensor:
    """The ``ss`` an epi 2 :func:`stream` of ``M`` rows writes."""
    return torch.empty(M, w.shape[0] // (16 * stream_fragments(M, w.shape[0])),
                       dtype=torch.float32, device=device)


def stream(epi: int, x: torch.Tensor, w: torch.Tensor, out: torch.Tensor | None = None,
           packed: bool = False, ss: torch.Tensor | None = None, inv_d: float = 0.0,
           eps: float = 0.0, bias=None, gelu: bool = False, positions=None, cos_sin=None,
           k_cache=None, v_cache=None, slots=None, hq: int = 0, hkv: int = 0) -> torch.Tensor:
    """``x @ w.T`` of up to 16 rows with a fused epilogue (``csrc/stream.hip``), GPU only.

    ``ss`` (fp32 [M, n] partial sums of squares of the rows of ``x``) norms the rows first:
    ``x * rsqrt(sum(ss) * inv_d + eps)`` in bf16, an RMSNorm whose weight is folded into ``w``.
    epi 0: plain (+ ``bias``); 1: ``act(g + b) * (u + b)`` with ``w = [Wg; Wu]``, silu or, with
    ``gelu``, its tanh form; 2: ``out`` is the residual, updated in place, and ``ss``
    (:func:`stream_sums`) receives its rows' sums of squares; 3: QKV, as :func:`pgemm`'s.
    ``packed``: ``w`` is from :func:`stream_pack`."""
    M = x.shape[0]
    N = w.shape[0] // 2 if epi == 1 else w.shape[0]
    if out is None:
        out = x.new_empty(M, hq * 128 if epi == 3 else N)
    if x.stride(1) != 1 or x.stride(0) % 8 or x.stride(0) < x.shape[1] or x.data_ptr() % 16:
        x = x.clone(memory_format=torch.contiguous_format)
    if epi == 3 and checks.active(x):
        checks.slots("stream qkv", slots, k_cache)
    ss_in, ss_out = (None, ss) if epi == 2 else (ss, None)
    kernels().stream_gemm(epi, out, x, w, stream_fragments(M, w.shape[0]), packed, ss_in, inv_d,
                          eps, ss_out, bias, gelu, positions, cos_sin, k_cache, v_cache, slots,
                          hq, hkv)
    return out


# -------------------------------------------------- projections of some tens of rows (panel.hip)
PANEL_MAX_M = 256
PANEL_ROWS = (16, 32, 48, 64, 80, 96, 128, 160, 192, 224, PANEL_MAX_M)  # of a block


def _panel_cost(bm: int, rows: int, K: int, wn: int, S: int) -> float:
    """Modelled us of a panel GEMM of ``bm`` rows: a block takes in its weight rows and x at about
    50 GB/s, the chip the weights at 6 TB/s; slabs are written and read once more."""
    blocks = -(-(rows // 16) // wn) * S
    rounds = blocks / 256 if blocks > 3 * 256 else -(-blocks // 256)
    t = max(rounds * (16 * wn + bm) * (K / S) * 2 / 50e3, rows * K * 2 / 6.0e6)
    return t + (S * bm * rows * 8 / 8e6 if S > 1 else 0.0)


@functools.lru_cache(maxsize=4096)
def panel_slices(rows: int, K: int) -> int:
    """K slices of a panel GEMM whose consumer sums slabs, from the weight's size alone: a row's
    result must not depend on the rows beside it.  Chosen for 96 rows (us at 64 rows and 1 / 2 /
    4 / 8 slices: 4096 x 4096 14.9 / 11.3 / 9.6 / 9.8, 2048 x 8192 - / - / 13.4 / 9.7)."""
    return min((_panel_cost(96, rows, K, wn, S), S) for wn in (4, 8)
               for S in range(1, min(16, K // 64) + 1))[1]


@functools.lru_cache(maxsize=8192)
def panel_plan(M: int, rows: int, K: int, slabs: bool) -> tuple[int, int]:
    """(waves a block, K slices) of a panel GEMM with ``rows`` weight rows.  Unsliced, two waves
    while their blocks are one a CU (us at 32 / 64 / 128 rows, 4 / 2 waves: 6400 x 2048 9.3 / 7.9,
    11.5 / 9.9, 16.9 / 15.4; gated 8192 x 2048 10.5 / 8.9, 13.3 / 11.4, 19.9 / 17.8; but 12352 x
    2048 10.7 / 12.5, 12.9 / 15.0, 18.0 / 21.8).  Where 8 and 4 both wait for the weights, 4 up to
    16 rows (a row-major 128256 x 4096 at 1 row, 8 / 4: 164 / 157; above, packed and gated 28672 x
    4096 at 32: 39.7 / 40.5, at 64 42.1 / 47.6)."""
    if not slabs and rows <= 2 * 16 * 256:
        return 2, 1
    bm = next((b for b in PANEL_ROWS if M <= b), PANEL_MAX_M)
    S = panel_slices(rows, K) if slabs else 1
    waves = (4, 8) if bm == 16 and not slabs else (8, 4)  # the first of equals
    return min(waves, key=lambda wn: _panel_cost(bm, rows, K, wn, S)), S


def panel(epi: int, x: torch.Tensor, w: torch.Tensor, packed: bool = False, bias=None,
          gelu: bool = False, slabs: bool = False) -> torch.Tensor:
    """``x @ w.T`` of up to 256 rows (``csrc/panel.hip``), GPU only.  epi 0: plain, or with
    ``slabs`` perhaps fp32 partial slabs [S, M, N] whose sum it is; 1: ``act(g + b) * (u + b)``
    with ``w = [Wg; Wu]``, silu or, with ``gelu``, its tanh form.  ``packed``: ``w`` is from
    :func:`stream_pack`."""
    M, K = x.shape
    N = w.shape[0] // 2 if epi == 1 else w.shape[0]
    if x.stride(1) != 1 or x.stride(0) % 8 or x.stride(0) < K or x.data_ptr() % 16:
        x = x.clone(memory_format=torch.contiguous_format)
    wn, S = panel_plan(M, w.shape[0], K, slabs and epi == 0)
    if S > 1:
        out, epi = torch.empty(S, M, N, dtype=torch.float32, device=x.device), 2
    else:
        out = x.new_empty(M, N)
    kernels().panel_gemm(epi, out, x, w, wn, packed, bias, gelu)
    return out


def row_sumsq(x: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """fp32 [M] sums of squares of the rows of a bf16 [M, d] matrix."""
    if out is None:
        out = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
    if x.is_cuda:
        kernels().row_sumsq(out, x)
        return out
    out.copy_(x.float().pow(2).sum(1))
    return out


def splitk_add_rmsnorm(parts: torch.Tensor, residual: torch.Tensor, w: torch.Tensor, eps: float,
                       out: torch.Tensor | None = None) -> torch.Tensor:
    """``residual += bf16(sum_s parts[s])`` in place; returns ``RMSNorm(residual) * w``."""
    if parts.is_cuda:
        out = residual.new_empty(residual.shape) if out is None else out
        kernels().splitk_add_rmsnorm(out, parts, residual, w, eps)
        return out
    o, r = ref.fused_add_rmsnorm(parts.sum(0).to(residual.dtype), residual, w, eps)
    residual.copy_(r)
    return o


def splitk_rope_kv(parts, positions, cos_sin, k_cache, v_cache, slots, hq, hkv, block_size,
                   q: torch.Tensor | None = None) -> torch.Tensor:
    """QKV split-K partials -> RoPE'd q ``[T, hq*D]`` (returned); RoPE'd k and v
    written to the paged cache at ``slots``."""
    T = parts.shape[1]
    D = 128
    if parts.is_cuda:
        if checks.active(parts):
            checks.slots("splitk_rope_kv", slots, k_cache)
        q = torch.empty(T, hq * D, dtype=k_cache.dtype, device=parts.device) if q is None else q
        kernels().splitk_rope_kv(q, parts, positions, cos_sin, k_cache, v_cache, slots, hq, hkv,
                                 block_size)
        return q
    qkv = parts.sum(0).to(k_cache.dtype)
    qq = qkv[:, : hq * D].reshape(T, hq, D)
    kk = qkv[:, hq * D:(hq + hkv) * D].reshape(T, hkv, D)
    vv = qkv[:, (hq + hkv) * D:].reshape(T, hkv, D)
    qq = ref.apply_rope(qq, positions, cos_sin)
    kk = ref.apply_rope(kk, positions, cos_sin)
    ref.write_kv(k_cache, v_cache, kk, vv, slots)
    return qq.reshape(T, hq * D)


def splitk_swiglu(parts: torch.Tensor) -> torch.Tensor:
    S, M, N2 = parts.shape
    if parts.is_cuda:
        out = torch.empty(M, N2 // 2, dtype=torch.bfloat16, device=parts.device)
        kernels().splitk_swiglu(out, parts)
        return out
    return ref.silu_mul(parts.sum(0).to(torch.bfloat16))


def splitk_reduce(parts: torch.Tensor) -> torch.Tensor:
    S, M, N = parts.shape
    if parts.is_cuda:
        out = torch.empty(M, N, dtype=torch.bfloat16, device=parts.device)
        kernels().splitk_reduce(out, parts)
        return out
    return parts.sum(0).to(torch.bfloat16)


def linear(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor | None = None,
           tiles: bool = False) -> torch.Tensor:
    """``x @ w.T`` (w in [out, in] layout).  Decode-sized GPU batches (M <= 256)
    run the hand MFMA kernel (gemm.hip); larger batches (prefill) hipBLASLt or, with
    ``tiles`` (no other rank's blocks spin on this device), :func:`pgemm_small` where
    that pays."""
    r = _dgemm(0, x, w, out)
    if r is not None:
        return r
    if tiles and out is None and x.is_cuda and x.dim() == 2 and \
            x.dtype == w.dtype == torch.bfloat16 and _on_grid(x):
        cols = small_tile_cols(x.shape[0], w)
        if cols:
            return pgemm_small(x, w, cols)
    if out is not None:
        return torch.mm(x, w.t(), out=out)
    return F.linear(x, w)


def linear_silu(x: torch.Tensor, w_gu: torch.Tensor) -> torch.Tensor:
    """``silu(x Wg^T) * (x Wu^T)`` with ``w_gu = [Wg; Wu]``: the SwiGLU MLP's first
    half.  Decode batches fuse the activation into the GEMM epilogue."""
    r = _dgemm(1, x, w_gu, None)
    if r is not None:
        return r
    return silu_mul(F.linear(x, w_gu))


def silu_mul(x: torch.Tensor, out: torch.Tensor | None = None):
    inter = x.shape[-1] // 2
    if x.is_cuda:
        out = x.new_empty(*x.shape[:-1], inter) if out is None else out
        kernels().silu_mul(out, x)
        return out
    r = ref.silu_mul(x)
    if out is not None:
        out.copy_(r)
        return out
    return r


def embedding(ids: torch.Tensor, w: torch.Tensor, vocab_start: int = 0,
              out: torch.Tensor | None = None, src: torch.Tensor | None = None,
              tok_slots: torch.Tensor | None = None):
    """Token embedding gather.  ``src`` / ``tok_slots`` (decode): row t's token
    is ``tok_slots[src[t]]`` where ``src[t] >= 0`` (sampled on the device by an
    earlier step), else ``ids[t]`` -- resolved inside the kernel."""
    if ids.is_cuda:
        out = w.new_empty(ids.numel(), w.shape[1]) if out is None else out
        kernels().embedding(out, ids, w, vocab_start, src, tok_slots)
        return out
    if src is not None:
        ids = torch.where(src >= 0, tok_slots.index_select(0, src.clamp(min=0).long()), ids)
    local = (ids >= vocab_start) & (ids < vocab_start + w.shape[0])
    idx = torch.where(local, ids - vocab_start, torch.zeros_like(ids)).long()
    r = w[idx] * local[:, None].to(w.dtype)
    if out is not None:
        out.copy_(r)
        return out
    return r


def decode_workspace(batch: int, hq: int, max_blocks: int, block_size: int, part_size: int,
                     device, splits: int = 0) -> tuple[torch.Tensor, torch.Tensor]:
    max_parts = max((max_blocks * block_size + part_size - 1) // part_size, splits)
    part_o = torch.empty(batch * hq * max_parts * 128, dtype=torch.float32, device=device)
    part_ml = torch.empty(batch * hq * max_parts * 2, dtype=torch.float32, device=device)
    return part_o, part_ml


DECODE_SPLIT_MIN = int(os.environ.get("OMNIA_DECODE_SPLIT_MIN", "64"))


def decode_attention(q, k_cache, v_cache, block_tables, seq_lens, scale, part_size=512,
                     workspace=None, out=None, splits=0, split_min=None):
    """q: [B, Hq, D] one query per sequence at position seq_len-1.

    ``part_size``: partition length (splits = 0), or the longest partition the
    length-balanced split may use (splits > 0: each context is cut on the device
    into up to ``splits`` equal page-aligned partitions of >= ``split_min`` keys)."""
    if q.is_cuda:
        B, hq, _ = q.shape
        split_min = DECODE_SPLIT_MIN if split_min is None else split_min
        if checks.active(q):
            checks.paged("decode_attention", block_tables, seq_lens, k_cache, B)
        if out is None:
            out = torch.empty(B, hq, q.shape[2], dtype=q.dtype, device=q.device)
        if workspace is None:
            workspace = decode_workspace(B, hq, block_tables.shape[1], k_cache.shape[2],
                                         part_size, q.device, splits)
        kernels().decode_attention(out, q, k_cache, v_cache, block_tables, seq_lens,
                                   workspace[0], workspace[1], part_size, scale, splits,
                                   split_min)
        return out
    B = q.shape[0]
    qsl = torch.arange(B + 1, dtype=torch.int32)
    r = ref.paged_attention(q, k_cache, v_cache, block_tables, qsl, seq_lens, scale)
    if out is not None:
        out.copy_(r)
        return out
    return r


PREFILL_Q_TILE = int(os.environ.get("OMNIA_PREFILL_Q_TILE", "32"))  # 32 (32-row waves) | 64 | 128


def prefill_tiles(q_lens: list[int], tile: int | None = None) -> tuple[list[int], list[int]]:
    tile = tile or PREFILL_Q_TILE
    seqs, q0s = [], []
    for s, n in enumerate(q_lens):
        for q0 in range(0, n, tile):
            seqs.append(s)
            q0s.append(q0)
    return seqs, q0s


@functools.lru_cache(maxsize=4096)
def prefill_parts(tiles: int, hq: int, hkv: int, max_keys: int, one_group: bool = False) -> int:
    """Most key partitions of a 32-row query tile, for up to 512 blocks, two a CU (fewer where the
    live length gives a partition less than 128 keys).  A block walks its 64-key tiles one after
    the other, 1.35 us each, or, with two groups of waves where blocks are one a CU, 0.975;
    partitions shorten that walk but write and read fp32 partials, at about 3 TB/s, and cost a
    launch (us at 1 / 2 / 4 / 8 partitions, 32 heads on 8: 77 rows on 4000 keys 64 / 43 / 30 / 27, on
    1100 26 / 22 / 20 / 21, on 400 16 / 17 / 17 / 17; 200 on 2200 40 / 33 / 29 / 33; 512 on 3500 59 /
    53 / 56 / 64, on 512 15.9 / 22 / 25 / 25; 1001 on 4000 77 / 96)."""
    group = hq // hkv
    blocks = tiles * hq // (4 if group % 4 == 0 else 2 if group % 2 == 0 else 1)

    def walk(P):
        t = -(-max_keys // 64) / P
        return min(1.35 * t, 0.975 * t + 1.5) if blocks * P <= 256 and not one_group else 1.35 * t

    best, cost = 1, walk(1)
    for P in range(2, min(16, 512 // max(blocks, 1), max_keys // 128) + 1):
        c = walk(P) + 5.0 + P * tiles * 32 * hq * 1024 / 3e6
        if c < cost:
            best, cost = P, c
    return best


def prefill_attention(q, k_cache, v_cache, block_tables, q_start_loc, seq_lens, scale,
                      tile_seq=None, tile_q0=None, out=None, heads_per_wave: int = 0,
                      q_tile: int | None = None, lse=None, kv_lens=None,
                      shared_device: bool = False):
    """q: [T, Hq, D] new tokens of several sequences (varlen, causal w/ cached prefix).

    ``lse`` (fp32 [T, Hq], optional) receives each row's natural-log sum of
    exp of the scaled scores -- the statistic ring attention merges blocks
    with.  ``kv_lens`` (int32 [B], optional) caps the visible keys of sequence
    ``s`` at ``kv_lens[s]`` on top of the causal bound, so a K/V block that lies
    wholly before the queries is attended in full: ``seq_lens = kv_len + qlen``
    puts the queries after every key.  ``shared_device``: other ranks run on this device, whose
    all-reduce blocks may spin until this rank's next: blocks of two groups of waves hold all of a
    CU's registers, do not fit beside them and could wait out their spin bound."""
    if q.is_cuda:
        if tile_seq is None:
            qsl = q_start_loc.cpu().tolist()
            s, q0 = prefill_tiles([qsl[i + 1] - qsl[i] for i in range(len(qsl) - 1)], q_tile)
            tile_seq = torch.tensor(s, dtype=torch.int32, device=q.device)
            tile_q0 = torch.tensor(q0, dtype=torch.int32, device=q.device)
        out = torch.empty_like(q) if out is None else out
        if checks.active(q):
            checks.paged("prefill_attention", block_tables, seq_lens, k_cache,
                         q_start_loc.numel() - 1)
        q_tile = q_tile or PREFILL_Q_TILE
        parts = 1
        if q_tile == 32 and lse is None and kv_lens is None:
            parts = prefill_parts(tile_seq.numel(), q.shape[1], k_cache.shape[1],
                                  block_tables.shape[1] * k_cache.shape[2], shared_device)
        kernels().prefill_attention(out, q, k_cache, v_cache, block_tables, q_start_loc,
                                    seq_lens, tile_seq, tile_q0, scale, heads_per_wave, q_tile,
                                    lse, kv_lens, parts, shared_device)
        return out
    if lse is not None or kv_lens is not None:
        r, l = ref.paged_attention_lse(q, k_cache, v_cache, block_tables, q_start_loc, seq_lens,
                                       scale, kv_lens)
        if lse is not None:
            lse[: l.shape[0]].copy_(l)
    else:
        r = ref.paged_attention(q, k_cache, v_cache, block_tables, q_start_loc, seq_lens, scale)
    if out is not None:
        out.copy_(r)
        return out
    return r


def sample(logits, temperature, top_k=None, top_p=None, seeds=None, steps=None, counts=None,
           freq_pen=None, pres_pen=None, rep_pen=None, out=None, out_logprob=None,
           tok_slots=None, dst=None):
    """Fused GPU sampler; returns int32 [B] token ids.  With ``tok_slots`` /
    ``dst`` the kernel also writes row r's token to ``tok_slots[dst[r]]`` (the
    sequence's device token slot: no scatter op after it in a decode graph)."""
    if logits.is_cuda:
        B = logits.shape[0]
        out = torch.empty(B, dtype=torch.int32, device=logits.device) if out is None else out
        kernels().sample(out, out_logprob, logits, temperature, top_k, top_p, seeds, steps,
                         counts, freq_pen, pres_pen, rep_pen, tok_slots, dst)
        return out
    x = ref.apply_penalties(logits, counts, freq_pen, pres_pen, rep_pen)
    g = None
    if seeds is not None:
        g = torch.Generator().manual_seed(int(seeds[0]) + int(steps[0] if steps is not None else 0))
    r = ref.sample(x, temperature, top_k, top_p, generator=g)
    if counts is not None:
        counts[torch.arange(r.numel()), r.long()] += 1
    if tok_slots is not None:
        tok_slots.index_copy_(0, dst, r.to(tok_slots.dtype))
    if out is not None:
        out.copy_(r)
        return out
    return r


def apply_token_mask(logits: torch.Tensor, mask: torch.Tensor) -> torch.Tensor:
    """K13: in place, logits[r, v] = -inf where bit v of int32 ``mask[r]`` is clear."""
    if logits.is_cuda:
        kernels().apply_token_mask(logits, mask.to(device=logits.device, dtype=torch.int32)
                                   .contiguous())
        return logits
    return ref.apply_token_mask(logits, mask)


# ------------------------------------------------------------- memory tier (K17 / K18)
def mean_pool_l2(hidden: torch.Tensor, cu_seqlens: torch.Tensor) -> torch.Tensor:
    """[T, D] bf16 hidden states + [B+1] int32 offsets -> [B, D] fp32 unit vectors."""
    if hidden.is_cuda:
        B = cu_seqlens.numel() - 1
        out = torch.empty(B, hidden.shape[1], dtype=torch.float32, device=hidden.device)
        kernels().mean_pool_l2(out, hidden, cu_seqlens.to(device=hidden.device,
                                                          dtype=torch.int32).contiguous())
        return out
    return ref.mean_pool_l2(hidden, cu_seqlens)


def cosine_topk(q: torch.Tensor, m: torch.Tensor, k: int, valid: torch.Tensor | None = None):
    """Exact top-k of q . m over unit vectors.

    q: [NQ, D] (any float dtype, normalised), m: [N, D] bf16 (normalised rows),
    valid: optional uint8 [N] (0 = tombstoned).  Returns (scores fp32 [NQ, k],
    indices int64 [NQ, k]) sorted by descending score, ties by ascending index."""
    nq, N = q.shape[0], m.shape[0]
    k = min(k, N)
    if k == 0:
        return (torch.empty(nq, 0, dtype=torch.float32, device=m.device),
                torch.empty(nq, 0, dtype=torch.long, device=m.device))
    if m.is_cuda:
        kk = kernels()
        D = m.shape[1]
        vals, idxs = [], []
        # the kernel stages up to 64 KiB of queries in LDS: chunk by 8/4/2/1
        max_nq = max(1, min(8, (64 * 1024) // (4 * D)))
        i = 0
        while i < nq:
            n = min(max_nq, nq - i)
            npad = 1 if n == 1 else 2 if n == 2 else 4 if n <= 4 else 8
            qq = torch.zeros(npad, D, dtype=torch.float32, device=m.device)
            qq[:n] = q[i:i + n].to(device=m.device, dtype=torch.float32)
            scores = torch.empty(npad, N, dtype=torch.float32, device=m.device)
            kk.cosine_scores(scores, qq, m, valid)
            oi = torch.empty(npad, k, dtype=torch.int32, device=m.device)
            ov = torch.empty(npad, k, dtype=torch.float32, device=m.device)
            kk.topk(oi, ov, scores, k)
            vals.append(ov[:n])
            idxs.append(oi[:n].long())
            i += n
        return torch.cat(vals), torch.cat(idxs)
    return ref.cosine_topk(q, m, k, valid)


# ------------------------------------------------------------- MoE (K14)
MOE_LIBRARY_ROWS = 1024  # mean rows/expert above which eager calls use hipBLASLt per expert
_rows = os.environ.get("OMNIA_MOE_TILE256_ROWS")
MOE_TILE256_ROWS = int(_rows) if _rows else None  # None: by the tiles of the down product


def moe_tile_rows(experts: int, d: int) -> int:
    """Mean rows an expert from which ``experts`` (a shard's own) run on the 256x256 prefill tile
    (pgemm.hip EPI 5 / 6, 256-row segments); below it smaller segments (:func:`moe_panel_rows`)
    waste less padding.

    A segment costs the tile the same up to 256 rows and the panel kernel one step for each 128,
    so the line lies near 128 rows where the tiles of the down product fill half the chip, and
    where they do not, near 224.  Both products, us, 128-row segments (packed) / tile: 8 experts
    of 4096 x 14336 (128 tiles) at 112 rows 604 / 842, at 128 877 / 846, at 150 1053 / 859; 8 of
    2048 x 4096 (64 tiles) at 128 142 / 198, at 200 168 / 203, at 250 223 / 207; of 2048 x 3072 at
    128 117 / 174, at 200 132 / 178, at 250 177 / 183; ungated of 2048 x 6144 at 140 163 / 252 (the
    64-row kernel 230), at 200 165 / 257, at 260 236 / 258; 3 of 4096 x 7168 at 133 211 / 241, at
    233 225 / 250, at 267 341 / 309."""
    if MOE_TILE256_ROWS is not None:
        return MOE_TILE256_ROWS
    return 128 if experts * (d // 256) >= 128 else 224


def down_tile_cols(n: int, n_experts: int, experts: int, d: int) -> int:
    """Columns of the down product's tile for ``n`` assignments to ``n_experts`` experts, of which
    ``experts`` are here: 128 where the narrow tiles of the segments to be expected, half of an
    expert's last one empty, are one round of 256 CUs (us wide / narrow and narrow tiles, 8 experts
    of 2048 x 4096: 600 tokens of two 84 / 61 (128), 1600 85 / 63 (256), 2001 88 / 112 (272); 8 of
    4096 x 14336: 600 313 / 261 (256), 1001 319 / 432 (320))."""
    segments = n * experts / n_experts / 256 + experts / 2
    return 128 if d % 256 == 0 and segments * (d // 128) <= 256 else 256


def moe_stream_ok(n: int, experts: int, w_up: torch.Tensor, w_down: torch.Tensor,
                  packed: bool) -> bool:
    """Whether ``n`` assignments to ``experts`` experts (all of them, where a shard holds some) run
    on the streaming kernel, in 16-row segments (a fuller expert's weights are read once per
    segment).

    Both products, us at 1 / 4 / 8 / 16 / 32 / 64 tokens of 2 experts in 8, 2048 x 4096: 64-row
    kernel 52 / 90 / 82 / 93 / 93 / 93, packed 25 / 63 / 58 / 72 / 74 / 95; 4096 x 14336: 193 /
    383 / 470 / 472 / 475 / 477 and 111 / 315 / 418 / 419 / 431 / 602.  Row-major weights gain
    only where most experts have no row: 29 for 52 and 133 for 193 at 1 token."""
    return n <= (8 * experts if packed else (experts - 1) // 2) and \
        _moe_few_ok(packed, w_up, w_down)


def _moe_few_ok(packed: bool, *ws: torch.Tensor) -> bool:
    """Whether the streaming and panel kernels cover these expert weights: the shapes that
    moe.hip takes, on the 16-byte grid (``packed``: the copies are)."""
    if not _stream_on:
        return False
    for w in ws:
        if w.shape[1] % 64 or w.shape[2] % 64 or \
                not (packed or (w.is_cuda and w.dtype == torch.bfloat16 and _on_grid(w))):
            return False
    return True


def moe_panel_rows(n: int, experts: int, w_up: torch.Tensor, w_down: torch.Tensor,
                   packed: bool) -> int:
    """Segment rows of the panel kernel for ``n`` assignments to ``experts`` experts (all of them,
    where a shard holds some), 0 where moe.hip's 64-row kernel does better.

    From 64 rows an expert most need two segments of 64, so the weights are read twice;
    segments of 128 read them once (both products, us, 64-row kernel / 128-row segments, as they
    are and packed, at 56 / 64 / 75 / 100 rows: 8 experts of 2048 x 4096 99 / 123 / 148 / 159, 119 /
    120 / 123 / 126 and 106 / 105 / 108 / 113; of 4096 x 14336 567 / 752 / 971 / 1048, 584 / 593 /
    604 / 634 and 538 / 544 / 564 / 600; of 2048 x 3072 78 / 99 / 112 / 117, 99 / 101 / 103 / 107 and
    89 / 90 / 93 / 96).  Fewer rows gain from whole-line reads of packed weights where K is long (8
    to 56 rows, 64-row kernel / 64-row segments: the first 94 / 82 to 99 / 92, the second 495 / 446
    to 567 / 527, the third 75 / 70 to 78 / 80; 32 of 2048 x 1024 90 / 97)."""
    if not _moe_few_ok(packed, w_up, w_down):
        return 0
    if n >= 64 * experts:
        return 128
    return 64 if packed and min(w_up.shape[2], w_down.shape[2]) >= 2048 else 0


def _moe_grouped(x, w_gu, w_down, ids, wts, k, n_experts, e_lo, e_hi, bm, glu=None,
                 gelu: bool = False, streams=None, shared_device: bool = False):
    """Grouped expert FFN over device-sorted assignments, no host sync: Y [T*k, d]
    (row t*k + j = slot j of token t, routing weight applied; other experts' rows
    unwritten).  ``bm`` 256: the 256x256 MFMA prefill tile; 64: moe.hip.  ``glu`` =
    (alpha, limit): clamped GLU experts whose INPUT takes the routing weight; ``gelu``:
    ungated experts (``w_gu`` [E, I, d]).  ``streams``: packed copies (:func:`stream_pack`) of
    both weights, or None; in place of ``bm`` 64, few assignments run :func:`moe_stream_ok`'s
    kernel and others :func:`moe_panel_rows`'s (not with ``shared_device``)."""
    kk = kernels()
    n, experts = ids.numel(), e_hi - e_lo
    few = bm == 64 and moe_stream_ok(n, n_experts, w_gu, w_down, streams is not None)
    panel = 0
    if few:
        bm = 16
    elif bm == 64 and not shared_device:
        panel = moe_panel_rows(n, n_experts, w_gu, w_down, streams is not None)
        bm = panel or bm
    if bm != 64 and not _on_grid(x):  # moe.hip takes rows as they lie
        x = x.clone()
    mb = kk.moe_max_blocks(n, experts, bm)
    # a wave of the streaming kernel sorts 64 assignments by itself, an expert a step
    own = few and n <= 64 and experts <= 64
    sorted_ids = torch.empty(0 if own else mb * bm, dtype=torch.int32, device=x.device)
    blk = torch.empty(0 if own else mb, dtype=torch.int32, device=x.device)
    nblk = torch.empty(1, dtype=torch.int32, device=x.device)
    if not own:
        kk.moe_align(sorted_ids, blk, nblk, ids, n_experts, e_lo, e_hi)
    act = torch.empty(mb * bm, w_down.shape[2], dtype=x.dtype, device=x.device)
    Y = torch.empty(n, x.shape[1], dtype=x.dtype, device=x.device)
    gemm = kk.pgemm_moe if bm == 256 else kk.moe_gemm
    if bm == 256 and down_tile_cols(n, n_experts, experts, w_down.shape[1]) == 128:

        def gemm(mode, out, A, w, so, bl, nb, rw, k, n, e0, alpha=0.0, limit=0.0):
            kk.pgemm_moe(mode, out, A, w, so, bl, nb, rw, k, n, e0, alpha, limit,
                         128 if mode == 1 else 256)

    if few:
        # experts whose weights are read, of a shard's as many as of the rest
        live = max(1, min(n, n_experts) * experts // n_experts)

        def gemm(mode, out, A, w, so, bl, nb, rw, k, n, e0, alpha=0.0, limit=0.0):
            frags = min(2, stream_fragments(min(n, 16), w.shape[1] * live))
            if streams is not None:
                w = streams[mode == 1]
            kk.stream_moe(mode, out, A, w, so, bl, nb, rw, k, n, e0, frags, streams is not None,
                          alpha, limit, ids if own else None)

    elif panel:
        # live ones, about: an expert may well have a third more rows than the mean (ungated of
        # 2048 x 6144 at 102 rows, down product with 4 / 8 waves, routed evenly 59 / 71 us, to
        # half of the experts more often 91 / 71)
        segs = experts * -(-4 * n // (3 * n_experts * panel))

        def gemm(mode, out, A, w, so, bl, nb, rw, k, n, e0, alpha=0.0, limit=0.0):
            wn = max(4, panel_plan(panel, w.shape[1] * segs, w.shape[2], False)[0])
            if streams is not None:
                w = streams[mode == 1]
            kk.panel_moe(mode, out, A, w, so, bl, nb, rw, k, n, e0, wn, streams is not None,
                         alpha, limit)

    if glu is not None:
        gemm(2, act, x, w_gu, sorted_ids, blk, nblk, wts.view(-1), k, n, e_lo, *glu)
        gemm(1, Y, act, w_down, sorted_ids, blk, nblk, None, k, n, e_lo)
        return Y
    gemm(3 if gelu else 0, act, x, w_gu, sorted_ids, blk, nblk, None, k, n, e_lo)
    gemm(1, Y, act, w_down, sorted_ids, blk, nblk, wts.view(-1), k, n, e_lo)
    return Y


def moe_rows(rows: torch.Tensor, eids: torch.Tensor, w_gu: torch.Tensor, w_down: torch.Tensor,
             e_lo: int, n_experts: int) -> torch.Tensor:
    """Expert FFN of each row under its own expert id (the receive side of an
    expert-parallel all-to-all): ``y[r] = down_e(silu(gate_e x) * up_e x)`` with
    ``e = eids[r]`` for local experts ``[e_lo, e_lo + w_gu.shape[0])``; rows whose
    id is outside that range (padding, ``-1``) are left unwritten.  Static shapes
    and no host sync (hipGraph-safe): the grouped MFMA kernels with top-1 routing."""
    R, d = rows.shape
    e_hi = e_lo + w_gu.shape[0]
    if not rows.is_cuda:
        y = rows.new_zeros(R, w_down.shape[1])
        local = (eids.long() - e_lo)
        ok = (local >= 0) & (local < w_gu.shape[0])
        li = local.clamp(0, w_gu.shape[0] - 1)
        h = torch.bmm(w_gu.index_select(0, li).float(), rows.float()[:, :, None])[:, :, 0]
        a = ref.silu_mul(h)
        o = torch.bmm(w_down.index_select(0, li).float(), a[:, :, None])[:, :, 0]
        return torch.where(ok[:, None], o.to(rows.dtype), y)
    kk = kernels()
    ids = eids.to(torch.int32).view(R, 1).contiguous()
    mb = kk.moe_max_blocks(R, e_hi - e_lo)
    sorted_ids = torch.empty(mb * 64, dtype=torch.int32, device=rows.device)
    blk = torch.empty(mb, dtype=torch.int32, device=rows.device)
    nblk = torch.empty(1, dtype=torch.int32, device=rows.device)
    kk.moe_align(sorted_ids, blk, nblk, ids, n_experts, e_lo, e_hi)
    act = torch.empty(mb * 64, w_down.shape[2], dtype=rows.dtype, device=rows.device)
    kk.moe_gemm(0, act, rows, w_gu, sorted_ids, blk, nblk, None, 1, R, e_lo)
    y = torch.empty(R, w_down.shape[1], dtype=rows.dtype, device=rows.device)
    ones = torch.ones(R, dtype=torch.float32, device=rows.device)
    kk.moe_gemm(1, y, act, w_down, sorted_ids, blk, nblk, ones, 1, R, e_lo)
    return y


def moe(x: torch.Tensor, router: torch.Tensor, w_gu: torch.Tensor, w_down: torch.Tensor,
        k: int, n_experts: int, e_lo: int = 0, renorm: bool = True,
        graph_safe: bool = True, streams=None, shared_device: bool = False) -> torch.Tensor:
    """Top-k MoE FFN over the local experts ``[e_lo, e_lo + w_gu.shape[0])``.

    x [T, d] bf16, router [E, d], w_gu [E_loc, 2I, d] (gate ; up), w_down [E_loc, d, I].
    Returns the local experts' weighted contribution [T, d] (all-reduce over the
    EP group to complete it).  ``graph_safe`` keeps every shape static and the
    whole path on device (hipGraph decode); otherwise large batches run each
    expert's GEMMs on hipBLASLt after one host sync on the expert counts.  ``streams``:
    :func:`stream_pack` copies of both expert weights.  ``shared_device``: other ranks run on this
    device, whose all-reduce blocks may spin until this rank's next: a block of the 256-row tile or
    the panel kernel holds most of a CU's LDS, does not fit beside them and could wait out their
    spin bound; the other kernels' blocks fit."""
    e_hi = e_lo + w_gu.shape[0]
    if not x.is_cuda:
        return ref.moe(x, router, w_gu, w_down, k, e_lo, renorm).to(x.dtype)
    kk = kernels()
    T, d = x.shape
    n = T * k
    ids = torch.empty(T, k, dtype=torch.int32, device=x.device)
    wts = torch.empty(T, k, dtype=torch.float32, device=x.device)
    # router GEMM + softmax top-k in one hand kernel (moe.hip): no logits tensor,
    # no library GEMM
    kk.moe_router_topk(ids, wts, x.contiguous(), router, k, renorm)
    out = torch.empty_like(x)
    d, inter = x.shape[1], w_down.shape[2]
    if n >= moe_tile_rows(e_hi - e_lo, d) * n_experts and d % 256 == 0 and \
            inter % 128 == 0 and _on_grid(w_gu, w_down) and not shared_device:
        # prefill-sized: the 256x256 MFMA tile, grouped by 256-row expert segments
        # (pgemm.hip EPI 5 / 6) -- hand kernels, graph-safe, no per-expert library
        # calls and no host sync
        Y = _moe_grouped(x, w_gu, w_down, ids, wts, k, n_experts, e_lo, e_hi, 256)
        kk.moe_combine(out, Y, ids, k, e_lo, e_hi)
        return out
    if not graph_safe and n >= MOE_LIBRARY_ROWS * (e_hi - e_lo) and \
            os.environ.get("OMNIA_MOE_LIBRARY", "0") == "1":
        # opt-in comparison path: per-expert hipBLASLt after one host sync
        flat = ids.view(-1)
        order = torch.argsort(flat, stable=True)
        counts = torch.bincount(flat, minlength=n_experts).tolist()  # host sync (eager only)
        xs = x.index_select(0, (order // k))
        ys = torch.empty(n, d, dtype=x.dtype, device=x.device)
        o = sum(counts[:e_lo])
        for e in range(e_lo, e_hi):
            c = counts[e]
            if c:
                h = F.linear(xs[o:o + c], w_gu[e - e_lo])
                ys[o:o + c] = F.linear(silu_mul(h), w_down[e - e_lo])
            o += c
        Y = torch.empty(n, d, dtype=x.dtype, device=x.device)
        Y.index_copy_(0, order, ys * wts.view(-1).index_select(0, order)[:, None].to(x.dtype))
        kk.moe_combine(out, Y, ids, k, e_lo, e_hi)
        return out
    Y = _moe_grouped(x, w_gu, w_down, ids, wts, k, n_experts, e_lo, e_hi, 64, streams=streams,
                     shared_device=shared_device)
    kk.moe_combine(out, Y, ids, k, e_lo, e_hi)
    return out
