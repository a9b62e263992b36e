"""MI355X-native ops: thin Python wrappers over the HIP kernel library.

Every op has two paths:
  * CUDA (= ROCm/HIP) tensors -> the hand-written gfx950 kernel, always.
    There is no eager fallback on GPU; a missing/failed kernel raises.
  * CPU tensors -> a plain fp32 torch reference (used by CPU-only tests and
    as the numerics oracle for the GPU kernels).
"""
from __future__ import annotations

import functools
import ctypes
import itertools
import math

import torch
from torch.autograd import forward_ad

from . import _lib
from ._lib import AfOpsError, native_loaded
from . import reference as ref


def _on_gpu(*ts: torch.Tensor | None) -> bool:
    return any(t is not None and t.is_cuda for t in ts)


# ---------------------------------------------------------------- rmsnorm
def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-5,
            residual: torch.Tensor | None = None):
    """Fused (residual-add) RMSNorm.

    Returns (out, new_residual) when residual is given (residual updated
    in-place to x+residual), else out.
    """
    if not _on_gpu(x):
        return ref.rmsnorm(x, weight, eps, residual)
    T, H = x.shape
    out = torch.empty_like(x)
    rc = _lib.lib().af_rmsnorm(
        _lib.ptr(out), _lib.ptr(residual), _lib.ptr(x), _lib.ptr(residual),
        _lib.ptr(weight), eps, T, H, _lib.cur_stream())
    _lib.check(rc, "af_rmsnorm")
    return (out, residual) if residual is not None else out


# ---------------------------------------------------------------- rope
def rope_table(max_pos: int, head_dim: int, theta: float = 500000.0,
               device="cpu") -> torch.Tensor:
    """Host-precomputed fp32 [max_pos, head_dim] table: [cos | sin] halves."""
    half = head_dim // 2
    inv = 1.0 / (theta ** (torch.arange(0, half, dtype=torch.float64) / half))
    t = torch.arange(max_pos, dtype=torch.float64)
    freqs = torch.outer(t, inv)
    return torch.cat([freqs.cos(), freqs.sin()], dim=-1).float().to(device)


def rope_cache(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
               positions: torch.Tensor, table: torch.Tensor,
               kcache: torch.Tensor, vcache: torch.Tensor,
               slots: torch.Tensor, scale: tuple | None = None) -> None:
    """Fused in-place RoPE on q/k + paged-cache append of k/v.

    q [T, Hq*D], k/v [T, Hk*D] — rows may be strided (views straight out of
    the fused QKV projection); caches [npages, Hk, page, D].
    scale=(ss [T,8], k_dim, eps): rows multiplied by the RMSNorm scalar
    rsqrt(mean+eps) — used when the QKV GEMM ran un-normalized (blas path of
    the fused decode chain; norm weight folded into the projection).
    """
    _, Hk, page, D = kcache.shape
    T = q.shape[0]
    Hq = q.shape[1] // D
    assert q.stride(1) == 1 and k.stride(1) == 1 and v.stride(1) == 1
    if not _on_gpu(q):
        q3 = q.unflatten(-1, (Hq, D))
        k3 = k.unflatten(-1, (Hk, D))
        v3 = v.unflatten(-1, (Hk, D))
        if scale is not None:
            ss, kd, eps = scale
            rstd = torch.rsqrt(ss.view(T, 8).sum(-1) / kd + eps)
            for t3 in (q3, k3, v3):
                t3.mul_(rstd[:, None, None].to(t3.dtype))
        ref.rope(q3, k3, positions, table)
        ref.reshape_and_cache(k3, v3, kcache, vcache, slots)
        return
    if scale is not None:
        ss, kd, eps = scale
        ss_p, inv_k = _lib.ptr(ss), 1.0 / float(kd)
    else:
        ss_p, inv_k, eps = _lib.ptr(None), 0.0, 0.0
    rc = _lib.lib().af_rope_cache(
        _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), _lib.ptr(positions.int()),
        _lib.ptr(table), _lib.ptr(kcache), _lib.ptr(vcache), _lib.ptr(slots),
        ss_p, inv_k, eps,
        T, Hq, Hk, D, q.stride(0), k.stride(0), v.stride(0), page,
        _lib.cur_stream())
    _lib.check(rc, "af_rope_cache")


# ---------------------------------------------------------------- activation
def silu_and_mul(gate_up: torch.Tensor,
                 scale: tuple | None = None) -> torch.Tensor:
    """gate_up [T, 2I] -> silu(gate*r)*(up*r) [T, I] where r is the optional
    per-row RMSNorm scalar from scale=(ss [T,8], k_dim, eps)."""
    T, I2 = gate_up.shape
    if not _on_gpu(gate_up):
        if scale is not None:
            ss, kd, eps = scale
            rstd = torch.rsqrt(ss.view(T, 8).sum(-1) / kd + eps)
            gate_up = (gate_up.float() * rstd[:, None]).to(gate_up.dtype)
        return ref.silu_and_mul(gate_up)
    if scale is not None:
        ss, kd, eps = scale
        ss_p, inv_k = _lib.ptr(ss), 1.0 / float(kd)
    else:
        ss_p, inv_k, eps = _lib.ptr(None), 0.0, 0.0
    out = torch.empty(T, I2 // 2, dtype=gate_up.dtype, device=gate_up.device)
    rc = _lib.lib().af_silu_mul(_lib.ptr(out), _lib.ptr(gate_up), ss_p, inv_k,
                                eps, T, I2 // 2, _lib.cur_stream())
    _lib.check(rc, "af_silu_mul")
    return out


# ---------------------------------------------------------------- cache
def reshape_and_cache(k: torch.Tensor, v: torch.Tensor, kcache: torch.Tensor,
                      vcache: torch.Tensor, slots: torch.Tensor) -> None:
    """Scatter k/v [T,Hk,D] into paged caches [npages,Hk,page,D] at slots [T]."""
    if not _on_gpu(k):
        return ref.reshape_and_cache(k, v, kcache, vcache, slots)
    T = k.shape[0]
    _, Hk, page, D = kcache.shape
    rc = _lib.lib().af_reshape_and_cache(
        _lib.ptr(k), _lib.ptr(v), _lib.ptr(kcache), _lib.ptr(vcache),
        _lib.ptr(slots), T, Hk, D, page, _lib.cur_stream())
    _lib.check(rc, "af_reshape_and_cache")


def embedding(ids: torch.Tensor, table: torch.Tensor,
              ss: torch.Tensor | None = None,
              cut: "DecodeCut | None" = None) -> torch.Tensor:
    """table[ids]; ss [T, 8] gets the rows' sums of squares, and cut, a decode
    step's (decode_cut with fill=False), is made in the same launch."""
    if not _on_gpu(table):
        out = table[ids.long()]
        if ss is not None:
            ss.zero_()
            ss.view(-1, 8)[:, 0] = out.float().pow(2).sum(-1)
        return out
    T = ids.numel()
    V, H = table.shape
    out = torch.empty(T, H, dtype=table.dtype, device=table.device)
    rc = _lib.lib().af_embedding(_lib.ptr(out), _lib.ptr(table),
                                 _lib.ptr(ids.int()), _lib.ptr(ss), T, H,
                                 *(cut.args() if cut else (None, None, 0, 0)),
                                 _lib.cur_stream())
    _lib.check(rc, "af_embedding")
    return out


# ---------------------------------------------------------------- attention
def attn_decode(q: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
                block_table: torch.Tensor, seq_lens: torch.Tensor,
                scale: float | None = None, nsplit: int = 1,
                scratch: tuple[torch.Tensor, torch.Tensor] | None = None,
                out: torch.Tensor | None = None,
                window: int = 0,
                cut: "DecodeCut | None" = None) -> torch.Tensor:
    """Paged decode attention. q [B, Hq*D] (strided rows ok) -> out [B, Hq*D].
    window > 0: sliding-window (Mistral) — only the last `window` cached
    tokens are attended.

    cut: how the step's sequences are cut (decode_cut).  Without one a sequence
    is summed in nsplit parts of its own, whatever is beside it.  With one,
    lengths unlike enough are cut in equal shares of all tokens: where a sequence
    is cut, and so the order of its fp32 sums and its last bit in bf16, then
    depends on the lengths beside it."""
    _, Hk, page, D = kcache.shape
    B = q.shape[0]
    Hq = q.shape[1] // D
    if scale is None:
        scale = 1.0 / math.sqrt(D)
    if not _on_gpu(q):
        return ref.attn_decode(q.unflatten(-1, (Hq, D)), kcache, vcache,
                               block_table, seq_lens, scale,
                               window=window).flatten(1)
    if out is None:
        out = torch.empty(B, Hq * D, dtype=q.dtype, device=q.device)
    G = Hq // Hk
    po = pml = None
    cap = 0
    if cut is not None:
        _need(cut.B == B and cut.nsplit == nsplit and cut.data.device == q.device,
              f"decode attention: {B} sequences in {nsplit} parts, cut as {cut.B} in "
              f"{cut.nsplit}")
    if nsplit > 1:
        if scratch is None:
            scratch = decode_scratch(B, Hk, nsplit, G, q.device, shares=cut is not None)
        po, pml = scratch
        cap = min(po.numel() // (Hk * G * D), pml.numel() // (Hk * G * 2))
    rc = _lib.lib().af_attn_decode(
        _lib.ptr(out), _lib.ptr(po), _lib.ptr(pml), _lib.ptr(q),
        _lib.ptr(kcache), _lib.ptr(vcache), _lib.ptr(block_table),
        _lib.ptr(seq_lens), _lib.ptr(cut.data if cut else None), scale, B, Hq, Hk, D,
        page, block_table.shape[1], nsplit, cap, q.stride(0), window,
        _lib.cur_stream())
    _lib.check(rc, "af_attn_decode")
    return out


def decode_shares(B: int, Hk: int, G: int, nsplit: int, window: int = 0) -> bool:
    """Whether a decode step's sequences may be cut in equal shares: a lane per
    sequence, and room for all blocks at once, or the dispatch evens them out.
    Beyond four parts a sequence is short, or the step is small.  Long sequences
    behind a window are of one length."""
    return (2 <= nsplit <= 4 and 2 <= B <= 64 and window <= 0
            and B * Hk * nsplit <= 256 * (2 if G == 8 else 3))


def decode_scratch(B: int, Hk: int, nsplit: int, G: int, device, D: int = 128,
                   shares: bool = False):
    """Scratch of attn_decode: room for nsplit parts of every sequence, and with
    shares (decode_shares) for one more each."""
    return tuple(torch.empty(B, Hk, nsplit + shares, G, n, dtype=torch.float32,
                             device=device) for n in (D, 2))


class DecodeCut:
    """How the sequences of one decode step are cut, for attn_decode in each of its
    layers: made from the lengths on the device, once a step."""

    def __init__(self, seq_lens: torch.Tensor, nsplit: int):
        self.seq_lens, self.B, self.nsplit = seq_lens, seq_lens.numel(), nsplit
        self.data = torch.empty(self.B, 4, dtype=torch.int32, device=seq_lens.device)

    def args(self):
        return (_lib.ptr(self.data), _lib.ptr(self.seq_lens), self.B, self.nsplit)


def decode_cut(seq_lens: torch.Tensor, Hk: int, G: int, nsplit: int,
               window: int = 0, fill: bool = True) -> DecodeCut | None:
    """The cut of a step of sequences of seq_lens [B] tokens, None where it would
    stay with nsplit parts of each anyway.  fill=False leaves it to be made by
    `embedding`."""
    if not (seq_lens.is_cuda and seq_lens.dtype is torch.int32
            and seq_lens.is_contiguous()
            and decode_shares(seq_lens.numel(), Hk, G, nsplit, window)):
        return None
    cut = DecodeCut(seq_lens, nsplit)
    if fill:
        rc = _lib.lib().af_decode_cut(*cut.args(), _lib.cur_stream())
        _lib.check(rc, "af_decode_cut")
    return cut


def prefill_split(seq_lens: list[int], G: int, Hk: int, max_keys: int):
    """How a packed prefill step's attention is cut: (few_cols, 128-column
    items, 32-column items, key splits of the latter).  A sequence has G columns
    per row; up to few_cols of them go to the kernel with 32 columns per block.

    Sequences of one wave's columns always do.  A batch that would give the
    128-column kernel fewer than 128 blocks goes there whole (four prompts of
    60 rows behind 3000 tokens, 8 K/V heads: 59 us against 108).  Steps of a few
    rows per sequence, i.e. behind a history, also split the keys until there
    are 256 blocks, at least 256 of the largest possible history each (16 x 5
    rows behind 2400 tokens: 51 us against 58); prompts only up to 64 blocks,
    most have no history and a merge costs a launch."""
    cols = [ln * G for ln in seq_lens if ln > 0]
    few_cols = 32
    if sum(-(-c // 128) for c in cols if c > 32) * Hk < 128:
        few_cols = 1 << 30
    items = sum(-(-c // 128) for c in cols if c > few_cols)
    few = sum(-(-c // 32) for c in cols if c <= few_cols)
    nsplit = 1
    if few:
        blocks = 256 if max(seq_lens) <= 16 else 64
        nsplit = max(1, min(8, blocks // (few * Hk), max_keys // 256))
    return few_cols, items, few, nsplit


def attn_prefill(q: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
                 block_table: torch.Tensor, q_start: torch.Tensor,
                 cu_seqlens: torch.Tensor, seq_lens: list[int],
                 scale: float | None = None, head_dim: int = 128,
                 window: int = 0) -> torch.Tensor:
    """Paged causal prefill attention: chunk rows q [T, Hq*D] (strided ok)
    attend to cached history + chunk through the block table.  q_start[s] is
    the chunk's absolute start position (0 = full-prompt prefill); the chunk
    itself must already be appended to the cache (rope_cache does this)."""
    D = head_dim
    _, Hk, page, _ = kcache.shape
    T = q.shape[0]
    Hq = q.shape[1] // D
    if scale is None:
        scale = 1.0 / math.sqrt(D)
    if not _on_gpu(q):
        return ref.attn_prefill_paged(q.unflatten(-1, (Hq, D)), kcache, vcache,
                                      block_table, q_start, cu_seqlens,
                                      scale, window=window).flatten(1)
    G = Hq // Hk
    few_cols, items, few, nsplit = prefill_split(
        seq_lens, G, Hk, block_table.shape[1] * page)
    out = torch.empty(T, Hq * D, dtype=q.dtype, device=q.device)
    po = pml = None
    if nsplit > 1:
        po = torch.empty(few, Hk, nsplit, 32, D, dtype=torch.float32,
                         device=q.device)
        pml = torch.empty(few, Hk, nsplit, 32, 2, dtype=torch.float32,
                          device=q.device)
    rc = _lib.lib().af_attn_prefill(
        _lib.ptr(out), _lib.ptr(po), _lib.ptr(pml), _lib.ptr(q),
        _lib.ptr(kcache), _lib.ptr(vcache), _lib.ptr(block_table),
        _lib.ptr(q_start), _lib.ptr(cu_seqlens), scale, len(seq_lens), items,
        few, few_cols, nsplit, Hq, Hk, D, q.stride(0), page,
        block_table.shape[1], window, _lib.cur_stream())
    _lib.check(rc, "af_attn_prefill")
    return out


# ---------------------------------------------------------------- gemm
def choose_sk(N: int, K: int) -> int:
    """K-split for the skinny GEMM: fill >=1024 workgroups, >=256 K/split."""
    ntiles = N // 64
    sk = max(1, min(16, 1024 // max(1, ntiles)))
    sk = min(sk, max(1, K // 256))
    return sk


@functools.lru_cache(maxsize=None)
def rows_splits(M: int, N: int, K: int) -> int:
    """K splits of the row GEMM's 64- or 128-column blocks (M > 16): one block
    per CU if that comes out nearly full, else two (64-column blocks only, their
    buffers leave room for that), at least four 64-element pieces each.  128
    columns above 64 rows, and above 32 where that fills the chip with at least
    12 pieces each.  Measured at 64 rows: 4096 x 4096 8.5 us in 4 (8.8 in 8 of
    128 columns), 6144 x 4096 11.2 us in 5 (12.8 in 64 columns), 4096 x 14336
    21.7 us in 8 (23.1 in 4 of 64 columns)."""
    pieces = K // 64
    wide = M > 32 and N % 128 == 0
    blocks = N // 128 if wide else N // 64
    n = max(1, 256 // blocks)
    if wide and M <= 64 and (n * blocks < 192 or pieces < 12 * n):
        wide, blocks = False, N // 64
        n = max(1, 256 // blocks)
    if not wide and n * blocks < 224:
        n = max(1, 512 // blocks)
    n = max(1, min(n, 16, pieces // 4))
    per = -(-pieces // n)
    return -(-pieces // per)          # no empty split


_transform = torch._C._functorch.peek_interpreter_stack
_modes = torch._C._len_torch_dispatch_stack


def watched(*tensors: torch.Tensor, grad: bool = True) -> bool:
    """Whether a product of these must be torch's own: autograd records it
    (grad), or forward mode, a function transform, a tracer or a tensor subclass
    has to see it.  Kernels called by address pass all of them by."""
    grad = grad and torch.is_grad_enabled()
    for t in tensors:
        kind = type(t)
        if (kind is not torch.Tensor and kind is not torch.nn.Parameter
                or grad and t.requires_grad):
            return True
    return (forward_ad._current_level >= 0 or _transform() is not None
            or _modes() > 0 or torch.compiler.is_compiling())


def rows_operands_ok(tensors) -> bool:
    """Operands as the row GEMMs read them: bf16, whole, on 16-byte boundaries."""
    bf16 = torch.bfloat16
    for t in tensors:
        if t.dtype is not bf16 or not t.is_contiguous() or t.data_ptr() & 15:
            return False
    return True


def _rows_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """What the row GEMMs take: bf16 rows and weights of one length on one GPU,
    which lie whole and on 16-byte boundaries, whole 64 x 64 tiles of weights,
    1..128 rows.  The kernels read w by the length of x's rows."""
    xs, ws = x.shape, w.shape
    return (x.is_cuda and len(xs) == 2 == len(ws) and xs[1] == ws[1]
            and 0 < xs[0] <= 128 and ws[0] > 0 and ws[0] % 64 == 0
            and ws[1] > 0 and ws[1] % 64 == 0 and x.device == w.device
            and rows_operands_ok((x, w)))


def rows_pay(M: int, N: int) -> bool:
    """Whether plain products of up to 128 rows go to the row GEMMs: those of 33..128
    rows lose to the library where N fills the chip neither in blocks of 128 columns
    nor in several splits.  Measured, library against rows in us: 14336 x 4096
    25.6 / 21.7 at 32 rows, 26.7 / 30.0 at 48, 33.9 / 36.0 at 128; 16384 x 4096
    34.3 / 24.7, 34.9 / 38.9, 39.0 / 43.3; 28672 x 4096 53.9 / 41.5, 64.0 / 42.1,
    56.7 / 51.7; 128256 x 4096 190 / 151 at one row, 214 / 184 at 64, 238 / 215 at
    128.  Between 12288 and 24576
    these two were measured; the limits are the nearest sizes at which rows win."""
    return M <= 32 or N <= 12288 or N >= 24576


def _need(ok: bool, what: str) -> None:
    if not ok:
        raise AfOpsError(what)


def _whole(t: torch.Tensor | None, x: torch.Tensor, *shape: int) -> bool:
    """t can be written as x's kind of rows of that shape, two at a time."""
    return (t is not None and t.shape == shape and t.dtype is x.dtype
            and t.is_contiguous() and t.data_ptr() & 3 == 0
            and t.device == x.device)


def _row_stats(ss: torch.Tensor | None, x: torch.Tensor) -> bool:
    """ss holds (or takes) eight fp32 sums for each of x's rows."""
    return (ss is not None and ss.dtype == torch.float32
            and ss.device == x.device and ss.is_contiguous()
            and ss.numel() >= 8 * x.shape[0])


def _apart(a: torch.Tensor, b: torch.Tensor) -> bool:
    pa, pb = a.data_ptr(), b.data_ptr()
    return pa + a.nbytes <= pb if pa < pb else pb + b.nbytes <= pa


def linear_rows(x: torch.Tensor, w: torch.Tensor, mode: int = 0,
                residual: torch.Tensor | None = None,
                scale: tuple | None = None,
                ss_out: torch.Tensor | None = None, want_out: bool = True,
                out: torch.Tensor | None = None) -> torch.Tensor | None:
    """Weight-streaming GEMM for up to 128 rows with the step behind it; modes
    and scale=(ss, eps) as in linear_skinny.  scale=(None, eps): the RMSNorm
    scalar is computed from x itself (up to 16 rows).  want_out=False (modes 1
    and 4): only the residual is written.  x and residual must not overlap.
    out: contiguous rows to write to."""
    if not _rows_ok(x, w):
        raise AfOpsError(f"row GEMM: {tuple(x.shape)} {x.dtype} rows against "
                         f"{tuple(w.shape)} {w.dtype} weights")
    M, N = x.shape[0], w.shape[0]
    cols = N // 2 if mode == 2 else N
    if mode in (1, 4):
        _need(_whole(residual, x, M, N) and _apart(residual, x),
              "row GEMM: the residual must be whole rows apart from x")
        _need(mode == 1 or _row_stats(ss_out, x),
              "row GEMM: mode 4 leaves fp32 [M, 8] sums in ss_out")
    else:
        _need(mode in (0, 2) and want_out, f"row GEMM: mode {mode}")
    if out is not None:
        _need(_whole(out, x, M, cols) and _apart(out, x),
              f"row GEMM: out must be whole [{M}, {cols}] rows apart from x")
    if scale is not None:
        _need(mode in (0, 2) and (M <= ROWS_MAX if scale[0] is None
                                  else _row_stats(scale[0], x)),
              "row GEMM: fp32 [M, 8] sums of the rows for the norm")
    return launch_rows(x, w, mode, residual, scale, ss_out, want_out, out)


def launch_rows(x, w, mode=0, residual=None, scale=None, ss_out=None,
                want_out=True, out=None):
    """linear_rows for callers that have checked the operands, or made them."""
    M, K = x.shape
    N = w.shape[0]
    if want_out and out is None:
        out = torch.empty(M, N // 2 if mode == 2 else N, dtype=x.dtype,
                          device=x.device)
    splits, parts = 1, None
    if mode != 2 and (M > ROWS_MAX or mode == 4):
        splits = rows_splits(M, N, K)
        if splits > 1 or mode != 0:
            parts = torch.empty(splits, M, N, dtype=torch.float32,
                                device=x.device)
    norm, ss, eps = 0, None, 0.0
    if scale is not None:
        ss, eps = scale
        norm = 2 if ss is None else 1
    rc = _lib.lib().af_rows_linear(
        _lib.ptr(out), _lib.ptr(residual), _lib.ptr(parts), _lib.ptr(ss_out),
        _lib.ptr(x), _lib.ptr(w), M, N, K, splits, mode, norm, _lib.ptr(ss), eps,
        _lib.cur_stream())
    _lib.check(rc, "af_rows_linear")
    return out


# rows up to which the row GEMM needs no partial sums and no row statistics
ROWS_MAX = 16
# plain products of so few rows that one launch takes
ROWS_GROUP = 4


def launch_rows_group(pairs) -> list:
    """[x @ w^T for x, w in pairs], at most ROWS_GROUP of as many rows, ROWS_MAX at
    most, in one launch; for callers that have checked the operands."""
    outs, desc = [], []
    for x, w in pairs:
        out = torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device)
        outs.append(out)
        desc += (out.data_ptr(), x.data_ptr(), w.data_ptr(), *w.shape)
    rc = _lib.lib().af_rows_group((ctypes.c_int64 * len(desc))(*desc), len(pairs),
                                  pairs[0][0].shape[0], _lib.cur_stream())
    _lib.check(rc, "af_rows_group")
    return outs


def qkv_rope_rows(x: torch.Tensor, w: torch.Tensor, eps: float,
                  ss: torch.Tensor | None, positions: torch.Tensor,
                  table: torch.Tensor, kcache: torch.Tensor,
                  vcache: torch.Tensor, slots: torch.Tensor) -> torch.Tensor:
    """q [M, Hq*128] of up to 128 un-normalised rows: QKV projection (norm weight
    folded into w), RMSNorm scalar (from ss [M, 8] above 16 rows), rotary
    positions, and k / v appended to their pages.  Heads of 128 only."""
    if not _rows_ok(x, w):
        raise AfOpsError(f"QKV rows: {tuple(x.shape)} {x.dtype} rows against "
                         f"{tuple(w.shape)} {w.dtype} weights")
    M, N, (_, Hk, _, D) = x.shape[0], w.shape[0], kcache.shape
    _need(N // D - 2 * Hk > 0 and N % D == 0,
          f"QKV rows: {N} outputs for {Hk} K/V heads of {D}")
    _need(M <= ROWS_MAX or _row_stats(ss, x), "QKV rows: sums of the rows")
    pos = qkv_step(M, D, positions, table, slots)
    return launch_qkv_rows(x, w, eps, ss, pos, table, kcache, vcache, slots)


def qkv_step(M: int, D: int, positions: torch.Tensor, table: torch.Tensor,
             slots: torch.Tensor) -> torch.Tensor:
    """What the QKV rows of all layers of a step share, checked once: int32
    positions of M rows."""
    _need(table.shape[1] == D and table.dtype == torch.float32
          and table.is_contiguous(), f"QKV rows: rotary table for heads of {D}")
    _need(positions.numel() == M and slots.numel() == M
          and slots.dtype == torch.int64 and slots.is_contiguous(),
          f"QKV rows: positions and int64 slots of {M} rows")
    return positions.int().contiguous()


def launch_qkv_rows(x, w, eps, ss, pos, table, kcache, vcache, slots):
    """qkv_rope_rows for callers that have checked the rows and weights, or made
    them, and have pos from qkv_step; the pages are looked at here."""
    M, K = x.shape
    pages = kcache.shape
    _, Hk, page, D = pages
    _need(pages == vcache.shape and kcache.dtype is vcache.dtype is x.dtype
          and kcache.is_contiguous() and vcache.is_contiguous(),
          "QKV rows: pages must be whole and of x's type")
    N = w.shape[0]
    Hq = N // D - 2 * Hk
    q = torch.empty(M, Hq * D, dtype=x.dtype, device=x.device)
    splits, parts = 1, None
    if M > ROWS_MAX:
        splits = rows_splits(M, N, K)
        parts = torch.empty(splits, M, N, dtype=torch.float32, device=x.device)
    rc = _lib.lib().af_rows_qkv(
        _lib.ptr(q), _lib.ptr(parts), _lib.ptr(x), _lib.ptr(w), _lib.ptr(ss), M,
        Hq, Hk, D, K, splits, eps, _lib.ptr(pos), _lib.ptr(table),
        _lib.ptr(kcache), _lib.ptr(vcache), _lib.ptr(slots), page,
        _lib.cur_stream())
    _lib.check(rc, "af_rows_qkv")
    return q


def linear_skinny(x: torch.Tensor, w: torch.Tensor, mode: int = 0,
                  residual: torch.Tensor | None = None,
                  sk: int | None = None,
                  scale: tuple | None = None,
                  ss_out: torch.Tensor | None = None) -> torch.Tensor:
    """Decode-path GEMM (M<=256) via the MFMA weight-streaming kernels: up to 128
    rows linear_rows, more (or an explicit sk) the split-K kernel below.

    mode 0: plain; mode 1: +residual (in-place update); mode 2: fused SwiGLU
    (w holds [gate|up] rows, returns [M, N/2]); mode 4: +residual AND
    per-row sum-of-squares stats into ss_out [M,8].
    scale=(ss, eps) applies the RMSNorm row scalar rsqrt(mean(x^2)+eps) on
    the OUTPUT (valid when the norm weight is folded into w — see
    LlamaForCausalLM.fold_norm_weights); x itself stays unnormalized so the
    weight stream keeps its async global_load_lds pipeline.
    """
    M, K = x.shape
    N = w.shape[0]
    if w.shape[1] != K:
        raise AfOpsError(f"linear_skinny: rows of {K} against {w.shape[1]}")
    _need(mode in (0, 2) or residual is not None and mode in (1, 4)
          and (mode == 1 or ss_out is not None), f"linear_skinny: mode {mode}")
    if sk is None and _rows_ok(x, w) and (
            (scale is None or _row_stats(scale[0], x)) if mode in (0, 2) else
            scale is None and _whole(residual, x, M, N) and _apart(residual, x)
            and (mode == 1 or _row_stats(ss_out, x))):
        return linear_rows(x, w, mode, residual, scale, ss_out)
    if sk is None:
        sk = choose_sk(N, K)
    cols = N // 2 if mode == 2 else N
    out = torch.empty(M, cols, dtype=x.dtype, device=x.device)
    partial = torch.empty(sk, M, N, dtype=torch.float32, device=x.device)
    if scale is not None:
        ss, eps = scale
        ss_p = _lib.ptr(ss)
    else:
        ss_p = _lib.ptr(None)
        eps = 0.0
    rc = _lib.lib().af_gemm_skinny(
        _lib.ptr(out), _lib.ptr(partial), _lib.ptr(residual), _lib.ptr(x),
        _lib.ptr(w), M, N, K, sk, mode, ss_p, eps, _lib.ptr(ss_out),
        _lib.cur_stream())
    _lib.check(rc, "af_gemm_skinny")
    return out


def _wide_ok(x: torch.Tensor, w: torch.Tensor, rows: int = 256) -> bool:
    """What the wide GEMM takes: bf16 rows and weights of one length on one GPU,
    whole and on 16-byte boundaries; 256 rows or more (128 with K split), at least
    256 weight rows in 64s, at least 128 columns in 64s, half of w (the up rows)
    within 4 GB."""
    xs, ws = x.shape, w.shape
    return (x.is_cuda and len(xs) == 2 == len(ws) and xs[1] == ws[1]
            and rows <= xs[0] <= 1 << 24 and ws[0] >= 256 and ws[0] % 64 == 0
            and ws[1] >= 128 and ws[1] % 64 == 0
            and (ws[0] // 2 + 256) * ws[1] * 2 < 1 << 32
            and x.device == w.device and rows_operands_ok((x, w)))


def _launches_here(x: torch.Tensor) -> bool:
    """x is on the current device, on whose stream a kernel is launched; torch's
    products go to the device of their operands.  Nor does autocast choose another
    type for the product."""
    return (x.device.index == torch.cuda.current_device()
            and not torch.is_autocast_enabled("cuda"))


def _wide_out_ok(out: torch.Tensor, x: torch.Tensor, M: int, N: int) -> bool:
    return _whole(out, x, M, N) and _apart(out, x) and out.data_ptr() & 15 == 0


@functools.lru_cache(maxsize=4096)
def _library_behind(M: int, N: int, K: int) -> bool:
    """Whether the library's plain product, by what it reaches with 256 x 256 tiles, takes
    1.16 of the wide GEMM's own estimate.  It gives every block the same number of tiles
    where some 232..256 of them come out even, and then reaches 1.4 PFLOP/s; where only
    fewer blocks do, or none of 128 or more, its rate falls with them (means of 1738
    products: none 0.93, 128 0.95, 160 1.08, 192 1.16, 216 1.25 PFLOP/s).  Of 5,460
    products (25 projections, 256..14000 rows) this names 378 that the rules of _wide_pays
    leave to the library, library over wide 1.16 in the mean, 0.965 at least: 4096 x 4096
    at 10284 rows 351 us / 239, 11000 rows 407 / 283, 8256 x 2048 at 7634 rows 242 / 200,
    6144 x 4096 at 1500 rows 78 / 68.  With a K beyond 5120 or more than six rounds of
    tiles it is wrong by more (0.91, 0.93)."""
    tiles = -(-M // 256) * -(-N // 256)
    if K > 5120 or N > 24576 or not 128 < tiles <= 1536:
        return False
    blocks = next((tiles // r for r in range(-(-tiles // 256), tiles // 128 + 1)
                   if tiles % r == 0), 0)
    if blocks >= 232:
        return False
    for (lo, a), (hi, b) in itertools.pairwise(_LIBRARY_RATE):
        if lo <= blocks <= hi:
            rate = a + (b - a) * (blocks - lo) / (hi - lo)
            break
    ns = _lib.lib().af_gemm_wide_ns(M, N, K)
    return 0 < 1.16 * ns < 2e-6 * M * N * K / rate


#: blocks of the library that come out even, PFLOP/s
_LIBRARY_RATE = ((0, .93), (128, .95), (160, 1.08), (192, 1.16), (216, 1.25), (232, 1.38))


def _wide_pays(M: int, N: int, K: int, silu_fuse: bool) -> bool:
    """Whether the wide GEMM beats the library's, by the tiles that its 256 blocks
    take.  Times are the library's over the wide GEMM's, weights not in cache.

    With SwiGLU behind it, which the library leaves to a pass of its own: where its
    smallest tiles, 128 x 256, occupy 172 blocks (16 projections at 257..1373 rows:
    0.89..0.95 up to 168 tiles, 1.18 in the mean from 172 on, 0.96 at least).  Three
    rows of tiles of a K of 2048..4095 need 200: 16384 x 3072 0.84 at 257 rows, 0.92
    at 381, 1.11 at 412; 18432 x 2048, 216 tiles, 1.13.  Not 449..512 rows that make
    one round of 168..192 tall tiles with a longer K: 22016 x 4096 1.09 at 448 rows,
    0.98 at 512, 1.10 at 513, 24576 x 8192 1.09, 0.91, 0.98, but 20480 x 4096 1.08.

    Plain, by 256 x 256 tiles: the library is ahead in whole rounds (4096 x 4096 at
    8000 rows 0.95) and draws level below one, but falls back where a round is begun.
    How far goes with its own choice of tiles; these limits leave 716 of 1374 sizes
    (23 projections, 263..10284 rows), 1.19 in the mean, 0.96 at least:
    - K >= 2N, up to 216 tiles begun: 1.0..1.9 (4096 x 14336 at 4353 rows 1.74, 7400
      rows 1.61).  Not 64 or 128 behind a first round, which the library cuts evenly
      (8192 x 28672 at 2402 rows 0.89, 4096 x 14336 at 5006 0.96), and above 5120
      columns not 64 behind two rounds (0.94) or anything beyond (0.90).
    - up to 5120 columns, 128 begun: 0.96..1.55; 129..216 0.91..1.4.
    - wider: 63 behind one round (128 0.92 at 12288 x 4096), 128 behind two or four
      (1.34 at 10240 x 8192, 4076 rows), 95 behind three or five (0.93 beyond that),
      three not from a K of 8192 on (8192 x 8192 at 6587 rows 0.93), none behind six
      (0.91) or more.  Above 12288 columns one or two rounds lose (28672 x 4096 at 1100
      rows 0.95) and 63 is the limit for all (22016 x 4096 at 2560 rows, 92 behind
      three, 0.86).
    - K < 2N beyond these limits and below a round: _library_behind."""
    cols = -(-N // 256)
    if silu_fuse:
        tiles = -(-M // 128) * cols
        return (tiles >= (200 if M <= 384 and 2048 <= K < 4096 else 172)
                and not (448 < M <= 512 and 336 <= tiles <= 384 and K >= 4096))
    tiles = -(-M // 256) * cols
    rounds, begun = tiles >> 8, tiles & 255
    if K >= 2 * N:
        if rounds < 1 or begun == 0 or rounds == 1 and begun in (64, 128):
            return False
        return begun <= 216 and (N <= 5120 or rounds == 1
                                 or rounds == 2 and begun != 64)
    if rounds >= 1 and begun and not (
            rounds > 5 or rounds < 3 and N > 12288 or rounds == 3 and K >= 8192):
        if N <= 5120 or rounds in (2, 4) and N <= 12288:
            if begun <= 128:
                return True
        elif begun < (64 if rounds == 1 or N > 12288 else 96):
            return True
    return M >= 256 and _library_behind(M, N, K)


def launch_wide(x, w, silu_fuse=False, out=None, groups=0):
    """The wide GEMM itself, for callers that have asked _wide_ok."""
    (M, K), N = x.shape, w.shape[0]
    if out is None:
        out = torch.empty(M, N // 2 if silu_fuse else N, dtype=x.dtype,
                          device=x.device)
    rc = _lib.lib().af_gemm_wide(
        _lib.ptr(out), _lib.ptr(x), _lib.ptr(w), M, N, K, 2 if silu_fuse else 0,
        groups, _lib.cur_stream())
    _lib.check(rc, "af_gemm_wide")
    return out


def _wide_split_pays(M: int, N: int, K: int) -> bool:
    """Whether the wide GEMM with K in shares beats the library's: few tiles of 256 x
    256 and a long K, so that the parts' way through memory is small beside the weights'.
    21 projections at 129..3000 rows, weights not in cache, library over split: with K
    >= 2N, K > 8192, up to 128 tiles and tiles * K up to 2^21 0.96..2.8, 1.33 in the
    mean (14336 -> 4096 at 192 rows 104 us / 48, 640 rows 113 / 84, 1500 rows 170 /
    155; 28672 -> 8192 at 512 rows 309 / 225); beyond that 0.83..1.06 (14336 -> 4096 at
    2500 rows 238 / 270, 28672 -> 8192 at 640 rows 275 / 292), 8192 -> 2048 0.93..1.12,
    K < 2N mostly below 1 (4096 x 4096 at 512 rows 26 / 30).  The shares, which
    divide K in whole pieces, have to occupy most of the blocks: with the 128 that
    11008 allows at 129 rows 44 us / 52.  Many rows of few columns make the parts the
    larger stream again: 10240 -> 2048 at 1275 rows 79 / 70, at 1458 71 / 75, 2068 rows
    103 / 114 (but 16384 -> 2048 at 1275 rows 1.17 or more)."""
    cols = -(-N // 256)
    tiles = -(-M // 256) * cols
    if not (M > 128 and K >= 2 * N and K > 8192 and K % 64 == 0 and tiles <= 128
            and tiles * K <= 1 << 21 and (8 * M <= 5 * N or K >= 16384)):
        return False
    return -(-M // 128) * cols * _lib.lib().af_gemm_wide_splits(M, N, K) >= 192


def launch_wide_split(x, w, out=None, splits=0, groups=0):
    """The wide GEMM with K in shares (0: as many as cost least), for callers that have
    asked _wide_ok."""
    (M, K), N = x.shape, w.shape[0]
    splits = splits or _lib.lib().af_gemm_wide_splits(M, N, K)
    if out is None:
        out = torch.empty(M, N, dtype=x.dtype, device=x.device)
    parts = torch.empty(splits, M, N, dtype=torch.float32, device=x.device)
    rc = _lib.lib().af_gemm_wide_split(
        _lib.ptr(out), _lib.ptr(parts), _lib.ptr(x), _lib.ptr(w), M, N, K, splits,
        groups, _lib.cur_stream())
    _lib.check(rc, "af_gemm_wide_split")
    return out


def linear(x: torch.Tensor, w: torch.Tensor, silu_fuse: bool = False,
           out: torch.Tensor | None = None) -> torch.Tensor:
    """Linear layer dispatch: hand-written weight-streaming kernels up to 128
    rows, the wide GEMM or hipBLASLt (torch.matmul) for prefill GEMMs.  out
    (without silu_fuse): [M, N] rows of x's type to write to."""
    M, N = x.shape[0], w.shape[0]
    if out is not None and (silu_fuse or out.shape != (M, N)):
        raise AfOpsError(f"linear: out {tuple(out.shape)} for a [{M}, {N}] "
                         "product")
    if (M <= 128 and (silu_fuse or rows_pay(M, N))
            and x.is_cuda and not watched(x, w, grad=not silu_fuse)
            and (out is None or _whole(out, x, M, N) and _apart(out, x))
            and _rows_ok(x, w)):
        return launch_rows(x, w, 2 if silu_fuse else 0, out=out)
    if (M > 128 and x.is_cuda and x.dim() == 2 == w.dim()
            and _wide_pays(M, N, x.shape[1], silu_fuse) and _launches_here(x)
            and not watched(x, w, grad=not silu_fuse)
            and (out is None or _wide_out_ok(out, x, M, N))
            and _wide_ok(x, w)):
        return launch_wide(x, w, silu_fuse, out)
    if (not silu_fuse and x.is_cuda and x.dim() == 2
            and _wide_split_pays(M, N, x.shape[1]) and _launches_here(x)
            and not watched(x, w)
            and (out is None or _wide_out_ok(out, x, M, N))
            and _wide_ok(x, w, 128)):
        try:
            return launch_wide_split(x, w, out)
        except torch.OutOfMemoryError:
            pass              # the library needs no room for parts
    if out is not None:
        return torch.mm(x, w.t(), out=out)
    y = x @ w.t()
    if silu_fuse:
        return silu_and_mul(y)
    return y


# ---------------------------------------------------------------- mixture
MOE_MAX_EXPERTS, MOE_MAX_TOP = 64, 8     # limits of the routing kernels


def moe_route_ok(x: torch.Tensor, router: torch.Tensor, k: int) -> bool:
    """What the routing kernels take: bf16 rows and router rows of one length on
    one GPU, read 16 bytes at a time, and k of at most MOE_MAX_EXPERTS experts."""
    if not x.is_cuda or x.dim() != 2 or router.dim() != 2:
        return False
    (T, H), (E, HR) = x.shape, router.shape
    return (H == HR and T > 0 and H % 8 == 0 and 1 <= E <= MOE_MAX_EXPERTS
            and 1 <= k <= min(E, MOE_MAX_TOP) and x.device == router.device
            and rows_operands_ok((x, router)))


def moe_route(x: torch.Tensor, router: torch.Tensor, k: int):
    """Softmax routing of rows x [T, H] over the experts' router [E, H], the k
    largest renormalised, and the (row, choice) entries sorted by expert:
    (weights [T, k] f32, row [T*k] i32 of every sorted position, sorted position
    [T*k] i32 of every entry, first position of every expert [E+1] i32)."""
    if not moe_route_ok(x, router, k):
        raise AfOpsError(f"routing {tuple(x.shape)} rows over "
                         f"{tuple(router.shape)}, k {k}")
    return launch_moe_route(x, router, k)


def launch_moe_route(x, router, k):
    """moe_route for callers that have asked moe_route_ok."""
    T, H = x.shape
    E = router.shape[0]
    dev = x.device
    n = T * k
    topv = torch.empty(T, k, dtype=torch.float32, device=dev)
    idx = torch.empty(3 * n + E + 1, dtype=torch.int32, device=dev)
    topi, row, pos, offs = idx.split([n, n, n, E + 1])
    rc = _lib.lib().af_moe_route(
        _lib.ptr(topi), _lib.ptr(topv), _lib.ptr(offs), _lib.ptr(row),
        _lib.ptr(pos), _lib.ptr(x), _lib.ptr(router), T, H, E, k,
        _lib.cur_stream())
    _lib.check(rc, "af_moe_route")
    return topv, row, pos, offs


def moe_combine(y: torch.Tensor, pos: torch.Tensor,
                weights: torch.Tensor) -> torch.Tensor:
    """out[t] = sum_j weights[t, j] * y[pos[t*k + j]] over the sorted expert rows."""
    T, k = weights.shape
    H = y.shape[1]
    if not (y.is_cuda and y.shape[0] == T * k and H % 8 == 0
            and rows_operands_ok((y,)) and weights.dtype == torch.float32
            and weights.is_contiguous() and weights.device == y.device
            and pos.numel() == T * k and pos.dtype == torch.int32
            and pos.is_contiguous() and pos.device == y.device):
        raise AfOpsError(f"combining {tuple(y.shape)} rows by "
                         f"{tuple(weights.shape)} weights")
    out = torch.empty(T, H, dtype=y.dtype, device=y.device)
    rc = _lib.lib().af_moe_combine(
        _lib.ptr(out), _lib.ptr(y), _lib.ptr(pos), _lib.ptr(weights), T, H, k,
        _lib.cur_stream())
    _lib.check(rc, "af_moe_combine")
    return out


def moe_gemm_ok(x: torch.Tensor, router: torch.Tensor, gate_up: torch.Tensor,
                down: torch.Tensor) -> bool:
    """What the projections over sorted rows take beside moe_route_ok: bf16 weights
    [E, 2I, H] and [E, H, I] of the router's experts on x's GPU, whole and on 16-byte
    boundaries, H and I in 64s."""
    g, d = gate_up.shape, down.shape
    if len(g) != 3 or len(d) != 3:
        return False
    (E, I2, H), I = g, d[2]
    return (d == (E, H, I) and I2 == 2 * I and x.shape[1] == H
            and router.shape[0] == E and H > 0 and H % 64 == 0 and I > 0
            and I % 64 == 0 and x.device == gate_up.device == down.device
            and rows_operands_ok((x, gate_up, down)))


def moe_gemm_pays(n: int, E: int, H: int, I: int) -> bool:
    """Whether one launch per projection beats the row GEMMs expert by expert behind a
    wait of the host.  Not where the down projection, a block to 128 of its columns and
    every expert in use, leaves half of the CUs idle through a long K: the whole
    feed-forward expert by expert / in one launch, us: 2 of 8 experts of 4096 x 14336 at
    one row 150 / 165, 2 of 4 146 / 165, 4 rows of 4 187 / 195, 6 rows of 8 325 / 304;
    1 of 2 of 8192 x 28672 247 / 344, 32 rows 529 / 555; but 2 of 8 of 4096 x 7168 103 /
    100, one of 8192 x 7168 109 / 106."""
    idle = min(n, E) * -(-H // 128) <= 128
    return not (idle and (I > 8192 and n <= 4 or I > 16384 and n <= 32 * E))


def launch_moe_gemm(x, w, offs, n, row=None, swiglu=False):
    """n sorted rows against their expert's w [E, N, K], for callers that have asked
    moe_gemm_ok: x rows through row [n], or x in sorted order."""
    E, N, K = w.shape
    out = torch.empty(n, N // 2 if swiglu else N, dtype=x.dtype, device=x.device)
    rc = _lib.lib().af_moe_gemm(
        _lib.ptr(out), _lib.ptr(x), _lib.ptr(row), _lib.ptr(w), _lib.ptr(offs), n, E,
        N, K, 2 if swiglu else 0, _lib.cur_stream())
    _lib.check(rc, "af_moe_gemm")
    return out


def wide_experts_pay(x_rows: int, n: int, E: int, N: int, K: int,
                     swiglu: bool) -> bool:
    """Whether n sorted rows go to the wide GEMM rather than to moe_gemm: what it
    takes beside moe_gemm_ok (x and half an expert's weights within 4 GB), and rows
    enough that the matrix cores bound it and not the weight stream.  Measured with 8
    experts of 4096 x 14336, moe_gemm / wide in us: gate/up 445 / 454 at 180 rows per
    expert, 478 / 463 at 200, 589 / 536 at 260, 741 / 598 at 300, 1911 / 1567 at
    1024; down 242 / 265 at 200, 282 / 279 at 250, 429 / 287 at 288, 915 / 804 at
    1024.  With 15 shapes of 2..64 experts and 256..6144 x 512..16384 gate/up is ahead
    from 200 rows on in all (1.0..1.7), down from 250 on in all but the fewest tiles (8
    experts of 2048 x 1024, 64 of 256 blocks, 25 / 21 at 250 and 25 / 21 at 320; 4 of
    4096 x 14336 196 / 228 at 320 rows, 241 / 253 at 500, 377 / 253 at 600)."""
    return (n >= (200 if swiglu else 250) * E and N >= 256 and K >= 128
            and x_rows * K * 2 < 1 << 32 and (N // 2 + 256) * K * 2 < 1 << 32
            and n <= 1 << 24)


def launch_wide_experts(x, w, offs, n, row=None, swiglu=False):
    """launch_moe_gemm's product by the wide GEMM, for callers that have asked
    wide_experts_pay."""
    E, N, K = w.shape
    out = torch.empty(n, N // 2 if swiglu else N, dtype=x.dtype, device=x.device)
    rc = _lib.lib().af_gemm_wide_experts(
        _lib.ptr(out), _lib.ptr(x), _lib.ptr(row), _lib.ptr(w), _lib.ptr(offs),
        x.shape[0], n, E, N, K, 2 if swiglu else 0, _lib.cur_stream())
    _lib.check(rc, "af_gemm_wide_experts")
    return out


def launch_experts(x, w, offs, n, row=None, swiglu=False):
    """n sorted rows against their expert's w by the kernel that suits them, for
    callers that have asked moe_gemm_ok."""
    E, N, K = w.shape
    launch = (launch_wide_experts if wide_experts_pay(x.shape[0], n, E, N, K, swiglu)
              else launch_moe_gemm)
    return launch(x, w, offs, n, row, swiglu)


def gemm_bf16(a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """C[M,N] = a[M,K] @ w[N,K]^T via the hand-written MFMA kernel."""
    if not _on_gpu(a):
        return (a.float() @ w.float().t()).to(a.dtype)
    M, K = a.shape
    N = w.shape[0]
    c = torch.empty(M, N, dtype=a.dtype, device=a.device)
    rc = _lib.lib().af_gemm_bf16(_lib.ptr(c), _lib.ptr(a), _lib.ptr(w),
                                 M, N, K, _lib.cur_stream())
    _lib.check(rc, "af_gemm_bf16")
    return c


def gemm_bf16_ring(a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """Deep-pipelined 256x256 ring-buffered MFMA GEMM (K % 32 == 0):
    4-slot LDS K-chunk ring, counted vmcnt (never drained in-loop),
    setprio around the MFMA cluster (guide §5 8-phase structure)."""
    if not _on_gpu(a):
        return (a.float() @ w.float().t()).to(a.dtype)
    M, K = a.shape
    N = w.shape[0]
    c = torch.empty(M, N, dtype=a.dtype, device=a.device)
    rc = _lib.lib().af_gemm_bf16_ring(_lib.ptr(c), _lib.ptr(a),
                                      _lib.ptr(w), M, N, K,
                                      _lib.cur_stream())
    _lib.check(rc, "af_gemm_bf16_ring")
    return c


def gemm_bf16_q8(a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """Block-quadrant 8-phase deep-pipelined MFMA GEMM (K % 64 == 0,
    K >= 128): 8-slot LDS granule ring, one granule staged per phase two
    K-tiles ahead, counted vmcnt(8), barrier-paired 16-MFMA clusters
    under s_setprio.  1.04-1.15 PF measured (vs 0.83 for gemm.hip)."""
    if not _on_gpu(a):
        return (a.float() @ w.float().t()).to(a.dtype)
    M, K = a.shape
    N = w.shape[0]
    c = torch.empty(M, N, dtype=a.dtype, device=a.device)
    rc = _lib.lib().af_gemm_bf16_q8(_lib.ptr(c), _lib.ptr(a),
                                    _lib.ptr(w), M, N, K,
                                    _lib.cur_stream())
    _lib.check(rc, "af_gemm_bf16_q8")
    return c


def gemm_mxfp8(a8: torch.Tensor, sa: torch.Tensor, w8: torch.Tensor,
               sw: torch.Tensor, M: int | None = None,
               N: int | None = None, K: int | None = None) -> torch.Tensor:
    """C[M,N] bf16 = dequant(a8,sa) @ dequant(w8,sw)^T on the CDNA4
    block-scaled MFMA (MX-fp8: OCP e4m3 + E8M0 per-32-K-block scales,
    quantize with agentfield_amd.quant.quantize_mx).  K % 128 == 0,
    K >= 256."""
    M = M or a8.shape[0]
    K = K or a8.shape[1]
    N = N or w8.shape[0]
    if not _on_gpu(a8):
        from ..quant import dequantize_mx
        return (dequantize_mx(a8, sa) @ dequantize_mx(w8, sw).t()).to(
            torch.bfloat16)
    c = torch.empty(M, N, dtype=torch.bfloat16, device=a8.device)
    rc = _lib.lib().af_gemm_mxfp8(_lib.ptr(c), _lib.ptr(a8), _lib.ptr(sa),
                                  _lib.ptr(w8), _lib.ptr(sw), M, N, K,
                                  _lib.cur_stream())
    _lib.check(rc, "af_gemm_mxfp8")
    return c


# ---------------------------------------------------------------- sampling
class SamplerState:
    """Device-side scratch for graph-capturable sampling."""

    def __init__(self, max_b: int, device, seed: int = 0x5EED):
        self.pv = torch.empty(max_b, 16, dtype=torch.float32, device=device)
        self.pi = torch.empty(max_b, 16, dtype=torch.int32, device=device)
        self.step = torch.zeros(1, dtype=torch.int32, device=device)
        self.seed = seed
        # top-k/top-p scratch (histogram threshold selection), per row split
        self.rmax = torch.empty(max_b, 16, dtype=torch.float32, device=device)
        self.hist_n = torch.empty(max_b, 16, 256, dtype=torch.int32,
                                  device=device)
        self.hist_m = torch.empty(max_b, 16, 256, dtype=torch.float32,
                                  device=device)


def sample(logits: torch.Tensor, temps: torch.Tensor, state: SamplerState,
           out: torch.Tensor | None = None,
           topk: torch.Tensor | None = None,
           topp: torch.Tensor | None = None) -> torch.Tensor:
    """Greedy (temp==0) or Gumbel-max temperature sampling; optional
    top-k/top-p nucleus restriction (sort-free histogram threshold).
    logits [B,V] bf16; topk [B] i32 (0 = off); topp [B] f32 (>=1 = off)."""
    B, V = logits.shape
    if not _on_gpu(logits):
        res = ref.sample_greedy(logits)
        if out is not None:
            out[:B].copy_(res)
            return out
        return res
    if out is None:
        out = torch.empty(B, dtype=torch.int32, device=logits.device)
    if topk is not None or topp is not None:
        if topk is None:
            topk = torch.zeros(B, dtype=torch.int32, device=logits.device)
        if topp is None:
            topp = torch.ones(B, dtype=torch.float32, device=logits.device)
        rc = _lib.lib().af_sample_topkp(
            _lib.ptr(out), _lib.ptr(state.pv), _lib.ptr(state.pi),
            _lib.ptr(state.rmax), _lib.ptr(state.hist_n),
            _lib.ptr(state.hist_m), _lib.ptr(logits), _lib.ptr(temps),
            _lib.ptr(topk), _lib.ptr(topp), _lib.ptr(state.step), state.seed,
            B, V, _lib.cur_stream())
        _lib.check(rc, "af_sample_topkp")
        return out
    rc = _lib.lib().af_sample(
        _lib.ptr(out), _lib.ptr(state.pv), _lib.ptr(state.pi), _lib.ptr(logits),
        _lib.ptr(temps), _lib.ptr(state.step), state.seed, B, V, _lib.cur_stream())
    _lib.check(rc, "af_sample")
    return out


def gather_rows(x: torch.Tensor, idx: torch.Tensor) -> torch.Tensor:
    if not _on_gpu(x):
        return x[idx.long()]
    B = idx.numel()
    H = x.shape[1]
    out = torch.empty(B, H, dtype=x.dtype, device=x.device)
    rc = _lib.lib().af_gather_rows(_lib.ptr(out), _lib.ptr(x), _lib.ptr(idx.int()),
                                   B, H, _lib.cur_stream())
    _lib.check(rc, "af_gather_rows")
    return out


def mfma_mx_probe(a8: torch.Tensor, b8: torch.Tensor, sa: torch.Tensor,
                  sb: torch.Tensor) -> torch.Tensor:
    """Single-wave 16x16x128 MX-fp8 scaled MFMA with the assumed layouts.
    a8 [16,128] u8 (e4m3 bytes), b8 [128,16] u8, sa/sb [16,4] u8 (E8M0
    per 32-element K-block)."""
    d = torch.empty(16, 16, dtype=torch.float32, device=a8.device)
    rc = _lib.lib().af_mfma_mx_probe(_lib.ptr(d), _lib.ptr(a8), _lib.ptr(b8),
                                     _lib.ptr(sa), _lib.ptr(sb),
                                     _lib.cur_stream())
    _lib.check(rc, "af_mfma_mx_probe")
    return d


def mfma_probe(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """Single-wave 16x16x32 MFMA with the assumed layouts (GPU layout test)."""
    d = torch.empty(16, 16, dtype=torch.float32, device=a.device)
    rc = _lib.lib().af_mfma_probe(_lib.ptr(d), _lib.ptr(a), _lib.ptr(b),
                                  _lib.cur_stream())
    _lib.check(rc, "af_mfma_probe")
    return d


# the sequence-mixer op set (masked attention for any head size, decayed
# recurrences with state slots, hybrid-decoder glue) lives in its own module
# and kernel library
from . import seqmix  # noqa: E402,F401
