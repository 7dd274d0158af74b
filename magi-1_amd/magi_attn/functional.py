"""Reference-shaped callables over the C-ABI.

The four functions the reference's DiT module imports from third-party CUDA packages
(inference/model/dit/dit_module.py:27-37) keep their names, argument meaning and return
shapes here, so the module-level code reads the same:

  flex_flash_attn_func   (MagiAttention; dit_module.py:1032-1043, 1111-1122)
  flash_attn_func        (flash-attn;    dit_module.py:1062, 1090-1095)
  flash_attn_varlen_func (flash-attn;    dit_module.py:1124-1133)
  apply_rotary_emb       (flash-attn;    dit_module.py:961, 978)

plus the fused prologue and the cache-aware range attention this library adds.  PyTorch is
used for device memory and the current stream only.
"""
from __future__ import annotations

import ctypes as C
import math
from typing import Optional, Tuple

import torch

from . import _lib as L


def _launch(dev: torch.device, fn, *args) -> int:
    """fn(*args, stream) with `dev` current, on its current stream; raises on a negative code."""
    index = dev.index
    if torch._C._cuda_getDevice() == index:
        code = fn(*args, torch._C._cuda_getCurrentRawStream(index))
    else:
        with torch.cuda.device(dev):
            code = fn(*args, torch._C._cuda_getCurrentRawStream(index))
    if code < 0:
        L.check(code)
    return code


_CUS = {}  # compute units by device index


def _compute_units(device: torch.device) -> int:
    n = _CUS.get(device.index)
    if n is None:
        n = _CUS[device.index] = torch.cuda.get_device_properties(device).multi_processor_count
    return n


class BegunCalls(list):
    """A list for range_attention's `held` whose first call is begun at once (magi_attn_fwd_begin): done, or launched but for what brings its
    pieces together, or held where nothing is in pieces; launch_held() then launches what is left and the second call as one where it can."""

    begin = True  # the next call is the first


def _launch_packed(dev: torch.device, name: str, args: type, *fields) -> None:
    """The same for an entry point that takes an argument struct: its fields behind struct_size, in order."""
    call = L.packed(name, args)
    _launch(dev, call.fn, call.pack(call.size, *fields))


def _ptr(t: Optional[torch.Tensor]) -> int:
    return 0 if t is None else t.data_ptr()


def _fp32(t: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """t as a contiguous fp32 tensor (itself when it is one)."""
    return t if t is None or (t.dtype is torch.float32 and t.is_contiguous()) else t.to(torch.float32).contiguous()


def _check_thd(t: torch.Tensor, name: str) -> None:
    if t.dim() != 3:
        raise ValueError(f"{name} must be [tokens, heads, head_dim], got {tuple(t.shape)}")
    if not t.is_cuda:
        raise ValueError(f"{name} must be a CUDA (ROCm) tensor")
    if t.stride(2) != 1:
        raise ValueError(f"{name}: head_dim must be contiguous")


def _dtype_code(t: torch.Tensor) -> int:
    if t.dtype == torch.bfloat16:
        return L.MAGI_DTYPE_BF16
    if t.dtype == torch.float8_e4m3fn:
        return L.MAGI_DTYPE_FP8_E4M3
    raise TypeError(f"unsupported dtype {t.dtype}: bf16 or float8_e4m3fn")


def range_count(q_ranges: torch.Tensor, k_ranges: torch.Tensor, mode: int) -> int:
    """The number of ranges of a pair of device-side lists, refused where a launch could not read them."""
    if q_ranges.dtype != torch.int32 or k_ranges.dtype != torch.int32:
        raise TypeError("q_ranges / k_ranges must be int32")
    if not (q_ranges.is_cuda and k_ranges.is_cuda):
        raise ValueError("q_ranges / k_ranges must live on the device")
    if mode == L.MAGI_RANGES_PAIRS:
        if q_ranges.shape != k_ranges.shape or q_ranges.dim() != 2 or q_ranges.shape[1] != 2:
            raise ValueError("q_ranges / k_ranges must both be [n, 2]")
        return q_ranges.shape[0]
    if q_ranges.numel() != k_ranges.numel():
        raise ValueError("cu_seqlens_q / cu_seqlens_k must have the same length")
    return q_ranges.numel() - 1


def covered_by_launch(n: int, max_seqlen_q: int, rows: int) -> bool:
    """Rows that no range covers are zeros (lse -inf).  Where the ranges can cover the rows, the attention launch takes care
    of the few that are left; a clearing pass over the whole output only where it would have to write most of it."""
    return 1 <= n <= 64 and max_seqlen_q > 0 and n * max_seqlen_q >= rows


def _bounded_split_bytes(Hq: int, Hkv: int, n: int, max_seqlen_q: int, max_seqlen_k: int) -> int:
    """The scratch memory that a bf16 call with bounded scores makes use of."""
    lib, n = L.lib(), max(n, 0)  # (see magi_attn_tile_rows: whole 128-row workgroups make no use of any)
    size = lib.magi_attn_split_bytes(Hq, Hkv, n, max_seqlen_q, max_seqlen_k, L.MAGI_DTYPE_BF16)
    if size and lib.magi_attn_tile_rows(Hq, Hkv, n, max_seqlen_q, max_seqlen_k, size) == 128 and not lib.magi_attn_pieces_bytes(
            Hq, Hkv, n, max_seqlen_q, max_seqlen_k, 1):
        size = 0
    return size


def range_attention(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    q_ranges: torch.Tensor,
    k_ranges: torch.Tensor,
    max_seqlen_q: int,
    max_seqlen_k: int = 0,
    softmax_scale: Optional[float] = None,
    *,
    ranges_mode: int = L.MAGI_RANGES_PAIRS,
    k2: Optional[torch.Tensor] = None,
    v2: Optional[torch.Tensor] = None,
    k_split: Optional[int] = None,
    q_scale: Optional[torch.Tensor] = None,
    k_scale: Optional[torch.Tensor] = None,
    v_scale: Optional[torch.Tensor] = None,
    k2_scale: Optional[torch.Tensor] = None,
    v2_scale: Optional[torch.Tensor] = None,
    scale_chunk_tokens: int = 0,
    fp8_pow2_prescaled: bool = False,
    fp8_fast_exp2: bool = False,
    q_prescaled: bool = False,
    score_bound: float = 0.0,
    q_tile_rows: int = 0,
    bounded_mfma32: bool = False,
    auto_bound: bool = False,
    checked: bool = False,
    static_scratch: bool = False,
    q_norm: Optional[tuple] = None,
    clear_out: bool = False,
    out: Optional[torch.Tensor] = None,
    return_lse: bool = True,
    zero_init: bool = True,
    split_keys: bool = True,
    share_waves: bool = False,
    held: Optional[list] = None,
) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """out[q_range_i] = softmax(q k^T * scale) v over k[k_range_i]; see magi_attn_fwd.

    k and v may be strided views (e.g. the two halves of an interleaved KV cache); with
    k2 / v2 the key axis is the concatenation [k[:k_split] | k2] without copying.

    k2_scale / v2_scale (fp8, with k2 / v2): the side segment's scale rows in tables of their own, row 0 = the chunk
    that starts at k_split; without them k_scale / v_scale are indexed across k_split as one table.

    fp8_fast_exp2 (with fp8_pow2_prescaled): piecewise-linear exp2 for the probabilities, MAGI_ATTN_FP8_FAST_EXP2.

    q_prescaled (bf16): q already carries softmax_scale * log2(e) (qk_prologue(..., q_premul=that)), so q . k is the
    exp2 exponent: the kernel skips its per-score multiply; softmax_scale is ignored.

    score_bound: promise that |q . k| * softmax_scale * log2(e) <= score_bound for every pair (with q_prescaled the
    factor is already in q); see magi_attn_args.score_bound.  Without q_prescaled the kernel applies the scale while
    it loads q.
    q_tile_rows: force a workgroup shape (0 = the library's choice); see magi_attn_args.q_tile_rows.
    bounded_mfma32 (with q_prescaled and score_bound): the 32x32x16 form of the bounded kernel, MAGI_ATTN_BOUNDED_MFMA32.
    auto_bound (bf16, instead of score_bound): the library measures max|q| and max|k| in two streaming passes and
    picks the bounded-score kernel on the device when their product allows it, MAGI_ATTN_AUTO_BOUND.  Its 16-byte
    workspace is a fresh tensor, or with static_scratch the library's own device array (magi_attn_fwd_static_scratch:
    no allocation at all when `out` is given and return_lse is False; such calls must not overlap on one GPU).
    checked (bf16, instead of score_bound): the bounded-score kernel judges by its row sums whether the scores were
    bounded, and a second launch repeats the blocks of rows where they were not, MAGI_ATTN_CHECKED.  Faster than the online
    softmax where the workgroups fill the chip, and its results are further from the exact ones (see _unbounded_mode).
    split_keys: False keeps the library from sharing the keys of a row among workgroups where that fills the chip better
    (magi_attn_args.split_workspace, up to 137 MB of scratch memory for the call; the fp32 sums are then added in another
    order).  Whether it does follows from the sizes of the launch alone, except that the online softmax runs without where there is no such
    memory to be had (the others raise).  Needs max_seqlen_k.  Without it a bf16 row's bits depend on its own range alone (MAGI_ATTN_ROW_BITS); with
    auto_bound also on which of the two kernels the longest rows of the whole call select.
    share_waves (with split_keys, a score_bound and max_seqlen_k): in launches of a few rows the wavefronts of a workgroup may share the keys of
    a row, MAGI_ATTN_SHARE_WAVES.
    held: the call is appended here instead of launched; launch_held() then launches what is in it, two of them as one where it can.
    q may be [batch, rows, Hq, D] with any batch stride (batch of activations laid out [position, batch, ...]): its rows
    count as batch * rows tokens for the ranges, out is (or comes back as) a tensor of q's shape, by default
    [rows, batch, Hq, D] transposed.  Needs a score_bound (math.inf: the online softmax).
    q_norm: (gamma, beta or None, eps[, norm_kind]): q is the raw projection, normalised per (token, head) row inside
    the kernel (fp32, zero-centred gamma) and scaled by softmax_scale * log2(e); needs score_bound.
    clear_out: rows of a given `out` that no range covers become zeros too.  A batched q's `out` may be [batch, rows, groups,
    Hq / groups, D], as a 4-D one otherwise.
    """
    batched = q.dim() == 4
    _check_thd(q[0] if batched else q, "q")
    _check_thd(k, "k")
    _check_thd(v, "v")
    Tq, Hq, D = (q.shape[0] * q.shape[1],) + tuple(q.shape[2:]) if batched else q.shape
    Hkv = k.shape[1]
    total_k = k.shape[0] if k2 is None else int(k_split) + k2.shape[0]
    if k2 is not None:
        _check_thd(k2, "k2")
        _check_thd(v2, "v2")
        if k2.stride() != k.stride() or v2.stride() != v.stride():
            raise ValueError("k2 / v2 must have the strides of k / v")
        if k_split is None or not (0 <= k_split <= k.shape[0]):
            raise ValueError("k_split must lie inside k")
    n = range_count(q_ranges, k_ranges, ranges_mode)
    q_ranges = q_ranges.contiguous()
    k_ranges = k_ranges.contiguous()
    by_kernel = (out is None or clear_out) and covered_by_launch(n, max_seqlen_q, Tq)
    zero_gaps = by_kernel and (zero_init or return_lse or clear_out)
    if clear_out and out is not None and not by_kernel:
        out.zero_()
    if out is None:
        new = torch.zeros if zero_init and not by_kernel else torch.empty
        out = new((q.shape[1], q.shape[0], Hq, D), dtype=torch.bfloat16, device=q.device).transpose(0, 1) if batched else \
            new((Tq, Hq, D), dtype=torch.bfloat16, device=q.device)
    lse = None
    if return_lse:
        lse = torch.empty((Hq, Tq), dtype=torch.float32, device=q.device) if zero_gaps else \
            torch.full((Hq, Tq), float("-inf"), dtype=torch.float32, device=q.device)
    if q_scale is not None or k_scale is not None or v_scale is not None or k2_scale is not None or v2_scale is not None:
        for name, t in (("q_scale", q_scale), ("k_scale", k_scale), ("v_scale", v_scale), ("k2_scale", k2_scale),
                        ("v2_scale", v2_scale)):
            if t is not None and (t.dtype != torch.float32 or not t.is_contiguous() or t.device != q.device):
                raise ValueError(f"{name} must be a contiguous fp32 tensor on q's device")
    if q.dtype == torch.float8_e4m3fn and scale_chunk_tokens > 0:
        # the kernel indexes the tables by token / scale_chunk_tokens without a bound of its own
        C_ = int(scale_chunk_tokens)
        rows_of = lambda n: (n + C_ - 1) // C_
        first = total_k if (k2 is None or k2_scale is None) else int(k_split)
        need = [("q_scale", q_scale, rows_of(Tq), Hq), ("k_scale", k_scale, rows_of(first), Hkv),
                ("v_scale", v_scale, rows_of(first), Hkv)]
        if k2_scale is not None:
            need += [("k2_scale", k2_scale, rows_of(total_k - int(k_split)), Hkv),
                     ("v2_scale", v2_scale, rows_of(total_k - int(k_split)), Hkv)]
        for name, t, rows, heads in need:
            if t is not None and (t.dim() != 2 or t.shape[0] < rows or t.shape[1] != heads):
                raise ValueError(f"{name} must be [>= {rows} chunks, {heads} heads], got {tuple(t.shape)}")
    q_stride, o_stride = q.stride(), out.stride()
    group_heads = o_stride_g = batch_rows = q_stride_b = o_stride_b = 0
    if batched:
        if len(o_stride) == 5 and out.shape[:2] == q.shape[:2] and out.shape[2] * out.shape[3] == Hq and out.shape[4] == D and o_stride[4] == 1:
            o_stride_g, group_heads, o_stride_t = o_stride[2], out.shape[3], o_stride[1]
        elif out.shape != q.shape or o_stride[3] != 1:
            raise ValueError("out must have the shape of a batched q, with contiguous rows")
        batch_rows, q_stride_b, o_stride_b = q.shape[1], q_stride[0], o_stride[0]
    elif len(o_stride) == 4:  # [Tq, groups, heads per group, D]: two-level head addressing
        if out.shape[0] != Tq or out.shape[1] * out.shape[2] != Hq or out.shape[3] != D or o_stride[3] != 1:
            raise ValueError("a 4-D out must be [Tq, groups, Hq / groups, D] with contiguous rows")
        o_stride_g, group_heads = o_stride[1], out.shape[2]
    if not (batched and group_heads):
        o_stride_t = o_stride[0] if group_heads else o_stride[-3]
    flags = ((L.MAGI_ATTN_FP8_POW2_PRESCALED if fp8_pow2_prescaled else 0) | (L.MAGI_ATTN_Q_PRESCALED if q_prescaled else 0)
             | (L.MAGI_ATTN_FP8_FAST_EXP2 if fp8_fast_exp2 else 0) | (L.MAGI_ATTN_BOUNDED_MFMA32 if bounded_mfma32 else 0)
             | (L.MAGI_ATTN_AUTO_BOUND if auto_bound else 0) | (L.MAGI_ATTN_ZERO_UNCOVERED if zero_gaps else 0)
             | (L.MAGI_ATTN_CHECKED if checked else 0) | (L.MAGI_ATTN_SHARE_WAVES if share_waves and split_keys else 0)
             | (0 if split_keys or q.dtype is not torch.bfloat16 else L.MAGI_ATTN_ROW_BITS))
    workspace = None
    if checked:
        workspace = torch.empty(max(4 * Hq * max(n, 0) * ((int(max_seqlen_q) + 255) // 256), 4), dtype=torch.int32, device=q.device)
    if auto_bound and not static_scratch:
        workspace = torch.empty(4, dtype=torch.float32, device=q.device)  # (alive until the launches are enqueued)
    split, split_bytes, online = None, 0, False
    # (beyond two workgroups of 32 rows for each of 256 CUs magi_attn_waves says no; short keys need no memory in any form)
    if (share_waves and max_seqlen_k >= 512 and Hq * n * max_seqlen_q <= 16384 and split_keys and q.dtype is torch.bfloat16
            and 0.0 < score_bound <= L.MAGI_SCORE_BOUND_MAX and not (q_tile_rows or bounded_mfma32)
            and attention_waves(Hq, Hkv, n, ranges_mode, max_seqlen_q, max_seqlen_k)):
        pass  # (keys shared without memory)
    elif split_keys and not static_scratch and max_seqlen_k >= 512 and (
            checked or auto_bound or 0.0 < score_bound <= L.MAGI_SCORE_BOUND_MAX or q.dtype is torch.float8_e4m3fn):
        if q.dtype is not torch.bfloat16:
            split_bytes = L.lib().magi_attn_split_bytes(Hq, Hkv, max(n, 0), int(max_seqlen_q), int(max_seqlen_k), _dtype_code(q))
        elif checked or q_tile_rows == 256:
            split_bytes = 0 if bounded_mfma32 else L.lib().magi_attn_split_bytes_256(Hq, Hkv, max(n, 0), int(max_seqlen_q), int(max_seqlen_k))
        elif not (q_tile_rows or bounded_mfma32):  # (those make no use of any)
            split_bytes = _bounded_split_bytes(Hq, Hkv, n, int(max_seqlen_q), int(max_seqlen_k))
    elif (split_keys and not static_scratch and max_seqlen_k >= 512 and q.dtype is torch.bfloat16 and not (auto_bound or q_prescaled)
          and q_tile_rows in (0, 128)):
        split_bytes, online = L.lib().magi_attn_pieces_bytes(Hq, Hkv, max(n, 0), int(max_seqlen_q), int(max_seqlen_k), 0), True
    if split_bytes:
        try:
            split = torch.empty(split_bytes, dtype=torch.uint8, device=q.device)
        except torch.OutOfMemoryError:
            if not online:  # (no going on without it: the same call would give other bits then)
                raise
            split_bytes = 0  # (a reference-shaped call, which promises nothing about its scores, needs no memory but its output's)
    gamma = beta = None  # (alive until the launch is enqueued)
    norm_eps, norm_kind = 0.0, 0
    if q_norm is not None:
        gamma, beta = _fp32(q_norm[0]), _fp32(q_norm[1])
        norm_eps = float(q_norm[2])
        norm_kind = int(q_norm[3]) if len(q_norm) > 3 else L.MAGI_NORM_LAYERNORM_1P
    k_stride, v_stride = k.stride(), v.stride()
    call = L.packed("magi_attn_fwd_static_scratch" if static_scratch else "magi_attn_fwd", L.AttnArgs)
    args = call.pack(
        call.size, q.data_ptr(), k.data_ptr(), v.data_ptr(), _ptr(k2), _ptr(v2), out.data_ptr(), _ptr(lse), q_ranges.data_ptr(),
        k_ranges.data_ptr(), _ptr(q_scale), _ptr(k_scale), _ptr(v_scale), q_stride[-3], q_stride[-2], k_stride[0], k_stride[1],
        v_stride[0], v_stride[1], o_stride_t, o_stride[-2], Tq, total_k, total_k if k2 is None else int(k_split), max(n, 0),
        ranges_mode, int(max_seqlen_q), int(max_seqlen_k), Hq, Hkv, D, _dtype_code(q), int(scale_chunk_tokens),
        0.0 if softmax_scale is None else float(softmax_scale), flags, group_heads, o_stride_g,
        min(float(score_bound), 3e38), int(q_tile_rows), _ptr(gamma), _ptr(beta), norm_eps, norm_kind, _ptr(k2_scale),
        _ptr(v2_scale), _ptr(workspace), batch_rows, q_stride_b, o_stride_b, _ptr(split), split_bytes)
    if held is None:
        _launch(q.device, call.fn, args)
        return out, lse
    begin = type(held) is BegunCalls and held.begin
    if begin:
        held.begin = False
    if begin and not static_scratch:
        if _launch(q.device, L.packed("magi_attn_fwd_begin", L.AttnArgs).fn, args):
            held.append((q.device, None, args, (q, k, v, k2, v2, q_ranges, k_ranges, gamma, beta, split, out, lse)))
    else:  # (with everything it reads and writes)
        held.append((q.device, call.fn, args, (q, k, v, k2, v2, q_ranges, k_ranges, q_scale, k_scale, v_scale, k2_scale, v2_scale, gamma, beta, workspace,
                                               split, out, lse)))
    return out, lse


def launch_held(calls: list) -> None:
    """The calls that range_attention(held=calls) left, on the current stream: two that do not depend on each other in one launch where their
    sizes are for it (magi_attn_fwd_two).  Empties the list."""
    begun, rest = bool(calls) and calls[0][1] is None, calls
    # (calls with static scratch memory have an entry point of their own: the ones for two would ask them for a workspace)
    fwd = L.packed("magi_attn_fwd", L.AttnArgs).fn
    pair = ((len(calls) == 2 or (begun and len(calls) > 2)) and calls[0][0] == calls[1][0] and calls[1][1] is fwd
            and (begun or calls[0][1] is fwd))
    if begun or pair:
        _launch(calls[0][0], L.packed_pair("magi_attn_fwd_end" if begun else "magi_attn_fwd_two").fn, calls[0][2], calls[1][2] if pair else None)
        rest = calls[2 if pair else 1:]
    for dev, fn, args, _ in rest:
        _launch(dev, fn, args)
    calls.clear()


def qk_norm_score_bound(q_norm_bound: float, k_norm_bound: float, head_dim: int = 128,
                        softmax_scale: Optional[float] = None) -> float:
    """score_bound for QK-normed attention from the lengths the two norms can produce (each at most
    sqrt(head_dim) max|gamma + 1| + |beta|, which a rotary embedding preserves): Cauchy-Schwarz, in exp2-exponent
    units, plus 1 % for the roundings to bf16."""
    scale = head_dim ** -0.5 if softmax_scale is None else softmax_scale
    return 1.01 * scale * math.log2(math.e) * q_norm_bound * k_norm_bound


def _measuring_a_bound_pays(q, k, n_ranges: int, max_seqlen_q: int, max_seqlen_k: int) -> bool:
    """A bf16 call without a score_bound: are the two passes of MAGI_ATTN_AUTO_BOUND (one over q, one over k) small
    beside what the bounded-score kernel saves?  Decided from sizes the host knows, generously on the side of the
    plain online-softmax launch: the saving is put at 12 % of the attention time, the passes at twice their HBM time
    plus three launches."""
    if q.dtype != torch.bfloat16 or q.dim() != 3 or q.shape[-1] != 128:
        return False
    Tq, Hq, D = q.shape
    keys = max_seqlen_k if max_seqlen_k > 0 else k.shape[0]
    attention_s = 4.0 * D * Hq * min(Tq, max(n_ranges, 0) * max_seqlen_q) * keys / 1.2e15
    passes_s = (Tq * Hq + k.shape[0] * k.shape[1]) * 2 * D / 4e12 + 3e-5
    return 0.12 * attention_s > 2 * passes_s


def _unbounded_mode(q, k, n_ranges: int, max_seqlen_q: int, max_seqlen_k: int, score_bound: float,
                    auto_bound: Optional[bool]) -> dict:
    """How a reference-shaped callable runs: with the bound it was given, as it was told to (auto_bound), else with a
    measured bound where the two passes are small beside the attention, and with the online softmax below that.

    Not range_attention's checked, which would be faster there (93600 rows x 24 heads over 400 keys 515 us against 694 us,
    three chunks of 1536 rows 221 against 295): its probabilities are 2^score and not relative to the row's maximum, whose
    own is then 1 and not rounded, so its results are further from float64 (1 to 12 % at unit scores, 10 to 27 % at twice
    that), and where scores are above 64 throughout it takes 1.6 to 1.9 times as long."""
    if score_bound != 0.0:
        return {"score_bound": score_bound}
    if auto_bound is None:
        auto_bound = _measuring_a_bound_pays(q, k, n_ranges, max_seqlen_q, max_seqlen_k)
    return {"auto_bound": bool(auto_bound)}


def flex_flash_attn_func(q, k, v, q_ranges, k_ranges, max_seqlen_q, max_seqlen_k, softmax_scale=None,
                         deterministic=False, disable_fwd_atomic_reduction=True, score_bound: float = 0.0,
                         auto_bound: Optional[bool] = None, **_unused):
    """(out [Tq,Hq,D], lse [Hq,Tq]) for disjoint q ranges.  The forward has one writer per output
    row, so it is deterministic and needs no atomic reduction whatever the two flags say.

    score_bound (no counterpart in the reference's call, optional): the caller's promise that
    |q . k| * softmax_scale * log2(e) <= score_bound for every pair, with q unscaled as the reference passes it
    (qk_norm_score_bound derives it from the norm parameters).  Up to MAGI_SCORE_BOUND_MAX it selects the kernel
    without a running maximum, which applies the scale while it loads q.

    auto_bound: without a score_bound the library can measure one (range_attention's auto_bound).  None (default):
    it does where the two passes over q and k are small beside the attention itself, which is how the reference's
    own call, unchanged, reaches the bounded-score kernel on its QK-normed q and k.  True / False: measure always / take
    the online-softmax kernel."""
    mode = _unbounded_mode(q, k, q_ranges.shape[0], max_seqlen_q, max_seqlen_k, score_bound, auto_bound)
    return range_attention(q, k, v, q_ranges, k_ranges, max_seqlen_q, max_seqlen_k, softmax_scale, **mode)


def flash_attn_func(q, k, v, dropout_p=0.0, softmax_scale=None, causal=False, deterministic=False,
                    score_bound: float = 0.0, auto_bound: Optional[bool] = None, **_unused):
    """q [B,Sq,Hq,D], k/v [B,Sk,Hkv,D] -> [B,Sq,Hq,D]; non-causal, no dropout (what the reference uses).
    score_bound, auto_bound: as in flex_flash_attn_func."""
    if dropout_p != 0.0 or causal:
        raise NotImplementedError("dropout / causal are not part of the MAGI-1 attention path")
    B, Sq, Hq, D = q.shape
    Sk = k.shape[1]
    q3 = q.reshape(B * Sq, Hq, D)
    k3 = k.reshape(B * Sk, k.shape[2], D)
    v3 = v.reshape(B * Sk, v.shape[2], D)
    cu_q = torch.arange(0, (B + 1) * Sq, Sq, dtype=torch.int32, device=q.device)
    cu_k = torch.arange(0, (B + 1) * Sk, Sk, dtype=torch.int32, device=q.device)
    mode = _unbounded_mode(q3, k3, B, Sq, Sk, score_bound, auto_bound)
    out, _ = range_attention(q3, k3, v3, cu_q, cu_k, Sq, Sk, softmax_scale, ranges_mode=L.MAGI_RANGES_CU,
                             return_lse=False, zero_init=False, **mode)
    return out.view(B, Sq, Hq, D)


def flash_attn_varlen_func(q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, dropout_p=0.0,
                           softmax_scale=None, causal=False, deterministic=False, score_bound: float = 0.0,
                           auto_bound: Optional[bool] = None, **_unused):
    """Packed varlen attention; segment s pairs q[cu_q[s]:cu_q[s+1]] with k[cu_k[s]:cu_k[s+1]].
    A segment without keys yields zero rows.  score_bound, auto_bound: as in flex_flash_attn_func."""
    if dropout_p != 0.0 or causal:
        raise NotImplementedError("dropout / causal are not part of the MAGI-1 attention path")
    mode = _unbounded_mode(q, k, cu_seqlens_q.numel() - 1, max_seqlen_q, max_seqlen_k, score_bound, auto_bound)
    out, _ = range_attention(q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, softmax_scale,
                             ranges_mode=L.MAGI_RANGES_CU, return_lse=False, zero_init=True, **mode)
    return out


def apply_rotary_emb(x, cos, sin, interleaved=False, inplace=False, **_unused):
    """x [B,S,H,D] (fp32 or bf16), cos / sin [S, R/2]: rotate the first R features, non-interleaved."""
    if interleaved:
        raise NotImplementedError("the DiT path uses the non-interleaved convention only")
    if x.dim() != 4:
        raise ValueError("x must be [batch, seqlen, heads, head_dim]")
    if x.dtype not in (torch.float32, torch.bfloat16):
        raise TypeError("x must be fp32 or bf16")
    B, S, H, D = x.shape
    R2 = cos.shape[-1]
    if cos.shape != (S, R2) or sin.shape != (S, R2):
        raise ValueError("cos / sin must be [seqlen, rotary_dim / 2]")
    if inplace and not x.is_contiguous():
        raise ValueError("inplace=True needs a contiguous x (a copy would be rotated instead of x)")
    xc = x.contiguous()
    y = xc if inplace else torch.empty_like(xc)
    cosf, sinf = _fp32(cos), _fp32(sin)
    _launch(x.device, L.lib().magi_apply_rotary, xc.data_ptr(), cosf.data_ptr(), sinf.data_ptr(), y.data_ptr(), B, S, H, D, R2,
            int(x.dtype == torch.bfloat16))
    return y


def qk_prologue(q_raw, k_raw, v_raw, rope, gq, bq, gk, bk, *, Hq: int, Hkv: int, eps: float = 1e-6,
                norm_kind: int = L.MAGI_NORM_LAYERNORM_1P, kv_out: Optional[torch.Tensor] = None,
                n_cache_rows: Optional[int] = None, kv_tail: Optional[torch.Tensor] = None,
                q_out: Optional[torch.Tensor] = None, batch: int = 1, q_premul: float = 1.0):
    """Fused norm + rotary + cast + KV write.  q_raw [S, Hq*D], k_raw / v_raw [S, Hkv*D] bf16 (row
    strided views allowed); rope [S, 2*R2] fp32 (sin | cos) or None.

    q_premul multiplies q after norm and rotary, before the one rounding to bf16 (softmax_scale * log2(e) for
    range_attention(..., q_prescaled=True)).

    kv_out is the destination of the first n_cache_rows tokens (a view of the cache starting
    at the write position, [>= n_cache_rows, Hkv, 2D]); kv_tail takes the rest.  With neither,
    a fresh [S, Hkv, 2D] tensor is written.  Returns (q [S,Hq,D], kv_out, kv_tail)."""
    S = q_raw.shape[0]
    D = 128
    dev = q_raw.device
    if q_out is None:
        q_out = torch.empty((S, Hq, D), dtype=torch.bfloat16, device=dev)
    if kv_out is None and kv_tail is None:
        kv_out = torch.empty((S, Hkv, 2 * D), dtype=torch.bfloat16, device=dev)
        n_cache_rows = S
    if n_cache_rows is None:
        n_cache_rows = S if kv_tail is None else 0
    for name, t in (("q_raw", q_raw), ("k_raw", k_raw), ("v_raw", v_raw)):
        if t.dtype != torch.bfloat16 or t.stride(-1) != 1 or t.dim() != 2:
            raise ValueError(f"{name} must be a 2-D bf16 tensor with contiguous rows")
    for name, t in (("kv_out", kv_out), ("kv_tail", kv_tail)):
        if t is not None and (t.dtype != torch.bfloat16 or t.dim() != 3 or t.shape[1:] != (Hkv, 2 * D)
                              or t.stride(2) != 1 or t.stride(1) != 2 * D):
            raise ValueError(f"{name} must be bf16 [rows, Hkv, 2*D] with contiguous heads")
    if kv_out is not None and kv_out.shape[0] < n_cache_rows:
        raise ValueError("kv_out is shorter than n_cache_rows")
    if kv_tail is not None and kv_tail.shape[0] < S - n_cache_rows:
        raise ValueError("kv_tail is shorter than S - n_cache_rows")
    gq, bq, gk, bk = _fp32(gq), _fp32(bq), _fp32(gk), _fp32(bk)
    R2 = 0
    if rope is not None:
        if rope.dtype != torch.float32 or rope.dim() != 2 or rope.shape[0] * max(batch, 1) != S or not rope.is_contiguous():
            raise ValueError("rope must be a contiguous fp32 [S / batch, 2*R2] tensor")
        R2 = rope.shape[1] // 2
    _launch_packed(dev, "magi_qk_prologue", L.PrologueArgs, q_raw.data_ptr(), k_raw.data_ptr(), v_raw.data_ptr(), _ptr(rope),
                   _ptr(gq), _ptr(bq), _ptr(gk), _ptr(bk), q_out.data_ptr(), _ptr(kv_out), _ptr(kv_tail), q_raw.stride(0),
                   k_raw.stride(0), v_raw.stride(0), 0 if kv_out is None else kv_out.stride(0),
                   0 if kv_tail is None else kv_tail.stride(0), S, int(n_cache_rows), Hq, Hkv, D, R2, int(norm_kind), float(eps),
                   int(batch), float(q_premul), L.MAGI_DTYPE_BF16, 0.0, 0.0)
    return q_out, kv_out, kv_tail


def qk_prologue_fp8(q_raw, k_raw, rope, gq, bq, gk, bk, *, Hq: int, Hkv: int, q_scale: float, k_scale: float,
                    eps: float = 1e-6, norm_kind: int = L.MAGI_NORM_LAYERNORM_1P, k_out: Optional[torch.Tensor] = None,
                    n_cache_rows: Optional[int] = None, k_tail: Optional[torch.Tensor] = None,
                    q_out: Optional[torch.Tensor] = None, batch: int = 1, q_premul: float = 1.0, v_raw: Optional[torch.Tensor] = None,
                    v_row_max: Optional[torch.Tensor] = None):
    """qk_prologue with e4m3 outputs (magi_prologue_args.out_dtype): q [S, Hq, D] = sat_e4m3(q * q_premul / q_scale)
    and K rows [*, Hkv, D] = sat_e4m3(k / k_scale) straight from the norm + rotary pass, with the two constant
    scales of the call (powers of two; see pow2_scale_for).  k_out takes the first n_cache_rows tokens (a view of
    an fp8 cache's K rows at the write position), k_tail the rest; with neither a fresh [S, Hkv, D] tensor.
    V is not part of this pass (quantize_fp8_split takes it from the raw projection); with v_raw [S, Hkv*D] and v_row_max, an int16
    [Hkv, S] tensor, the latter receives the largest magnitude of each row, which quantize_fp8_split takes the scales from.
    Returns (q8, k_out, k_tail)."""
    S = q_raw.shape[0]
    D = 128
    dev = q_raw.device
    f8 = torch.float8_e4m3fn
    if q_out is None:
        q_out = torch.empty((S, Hq, D), dtype=f8, device=dev)
    if q_out.dtype != f8 or tuple(q_out.shape) != (S, Hq, D) or not q_out.is_contiguous():
        raise ValueError("q_out must be a contiguous float8_e4m3fn [S, Hq, 128] tensor")
    if k_out is None and k_tail is None:
        k_out = torch.empty((S, Hkv, D), dtype=f8, device=dev)
        n_cache_rows = S
    if n_cache_rows is None:
        n_cache_rows = S if k_tail is None else 0
    for name, t in (("q_raw", q_raw), ("k_raw", k_raw)):
        if t.dtype != torch.bfloat16 or t.stride(-1) != 1 or t.dim() != 2:
            raise ValueError(f"{name} must be a 2-D bf16 tensor with contiguous rows")
    entry, more, v_at, v_stride = ("magi_qk_prologue", L.PrologueArgs), (), 0, 0
    if v_row_max is not None:
        if v_raw is None or v_raw.dtype != torch.bfloat16 or v_raw.dim() != 2 or v_raw.stride(-1) != 1:
            raise ValueError("v_raw must be a 2-D bf16 tensor with contiguous rows")
        if (v_row_max.dtype != torch.int16 or tuple(v_row_max.shape) != (Hkv, S) or not v_row_max.is_contiguous()
                or tuple(v_raw.shape) != (S, Hkv * D) or v_raw.device != dev or v_row_max.device != dev):
            raise ValueError("v_row_max must be a contiguous int16 [Hkv, S] tensor, v_raw [S, Hkv * 128], on q_raw's device")
        entry, more, v_at, v_stride = ("magi_qk_prologue_row_max", L.PrologueArgs, C.c_void_p), (v_row_max.data_ptr(),), v_raw.data_ptr(), v_raw.stride(0)
    for name, t in (("k_out", k_out), ("k_tail", k_tail)):
        if t is not None and (t.dtype != f8 or t.dim() != 3 or t.shape[1:] != (Hkv, D) or t.stride(2) != 1
                              or t.stride(1) != D):
            raise ValueError(f"{name} must be float8_e4m3fn [rows, Hkv, D] with contiguous heads")
    if k_out is not None and k_out.shape[0] < n_cache_rows:
        raise ValueError("k_out is shorter than n_cache_rows")
    if k_tail is not None and k_tail.shape[0] < S - n_cache_rows:
        raise ValueError("k_tail is shorter than S - n_cache_rows")
    gq, bq, gk, bk = _fp32(gq), _fp32(bq), _fp32(gk), _fp32(bk)
    R2 = 0
    if rope is not None:
        if rope.dtype != torch.float32 or rope.dim() != 2 or rope.shape[0] * max(batch, 1) != S or not rope.is_contiguous():
            raise ValueError("rope must be a contiguous fp32 [S / batch, 2*R2] tensor")
        R2 = rope.shape[1] // 2
    call = L.packed(*entry)
    args = call.pack(call.size, q_raw.data_ptr(), k_raw.data_ptr(), v_at, _ptr(rope), _ptr(gq), _ptr(bq), _ptr(gk),
                     _ptr(bk), q_out.data_ptr(), _ptr(k_out), _ptr(k_tail), q_raw.stride(0), k_raw.stride(0), v_stride,
                     0 if k_out is None else k_out.stride(0), 0 if k_tail is None else k_tail.stride(0), S, int(n_cache_rows), Hq,
                     Hkv, D, R2, int(norm_kind), float(eps), int(batch), float(q_premul), L.MAGI_DTYPE_FP8_E4M3, float(q_scale),
                     float(k_scale))
    _launch(dev, call.fn, args, *more)
    return q_out, k_out, k_tail


def qkv_proj_prologue(x: torch.Tensor, w: torch.Tensor, rope, gq, bq, gk, bk, *, Hq: int, Hkv: int, Hqx: int = 0,
                      eps: float = 1e-6, norm_kind: int = L.MAGI_NORM_LAYERNORM_1P, kv_out: Optional[torch.Tensor] = None,
                      n_cache_rows: Optional[int] = None, kv_tail: Optional[torch.Tensor] = None,
                      q_out: Optional[torch.Tensor] = None, qx_out: Optional[torch.Tensor] = None, batch: int = 1,
                      q_premul: float = 1.0):
    """The four projections and the prologue in one launch (magi_qkv_proj_prologue): x [S, K] bf16 (the normalised
    hidden states), w [(Hq + 2 Hkv + Hqx) * 128, K] bf16 with rows ordered q | k | v | qx heads.  Destinations as in
    qk_prologue; qx_out [S, Hqx, 128] receives the cross-attention q projection unnormalised.
    Returns (q [S, Hq, 128], kv_out, kv_tail, qx_out)."""
    D = 128
    if x.dim() != 2 or w.dim() != 2 or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16:
        raise ValueError("x and w must be 2-D bf16 tensors")
    if x.stride(1) != 1 or w.stride(1) != 1 or x.shape[1] != w.shape[1] or w.shape[0] != (Hq + 2 * Hkv + Hqx) * D:
        raise ValueError("x [S, K] and w [(Hq + 2 Hkv + Hqx) * 128, K] must have contiguous rows of the same length")
    if not x.is_cuda or w.device != x.device:
        raise ValueError("x and w must live on the same device (there is no CPU path)")
    S, K = x.shape
    dev = x.device
    if q_out is None:
        q_out = torch.empty((S, Hq, D), dtype=torch.bfloat16, device=dev)
    if qx_out is None and Hqx:
        qx_out = torch.empty((S, Hqx, D), dtype=torch.bfloat16, device=dev)
    if kv_out is None and kv_tail is None:
        kv_out = torch.empty((S, Hkv, 2 * D), dtype=torch.bfloat16, device=dev)
        n_cache_rows = S
    if n_cache_rows is None:
        n_cache_rows = S if kv_tail is None else 0
    for name, t, H in (("q_out", q_out, Hq), ("qx_out", qx_out, Hqx)):
        if t is not None and (t.dtype != torch.bfloat16 or tuple(t.shape) != (S, H, D) or not t.is_contiguous()):
            raise ValueError(f"{name} must be a contiguous bf16 [S, heads, 128] tensor")
    for name, t in (("kv_out", kv_out), ("kv_tail", kv_tail)):
        if t is not None and (t.dtype != torch.bfloat16 or t.dim() != 3 or t.shape[1:] != (Hkv, 2 * D)
                              or t.stride(2) != 1 or t.stride(1) != 2 * D):
            raise ValueError(f"{name} must be bf16 [rows, Hkv, 2*D] with contiguous heads")
    if kv_out is not None and kv_out.shape[0] < n_cache_rows:
        raise ValueError("kv_out is shorter than n_cache_rows")
    if kv_tail is not None and kv_tail.shape[0] < S - n_cache_rows:
        raise ValueError("kv_tail is shorter than S - n_cache_rows")
    gq, bq, gk, bk = _fp32(gq), _fp32(bq), _fp32(gk), _fp32(bk)
    R2 = 0
    if rope is not None:
        if rope.dtype != torch.float32 or rope.dim() != 2 or rope.shape[0] * max(batch, 1) != S or not rope.is_contiguous():
            raise ValueError("rope must be a contiguous fp32 [S / batch, 2*R2] tensor")
        R2 = rope.shape[1] // 2
    _launch_packed(dev, "magi_qkv_proj_prologue", L.QkvProjArgs, x.data_ptr(), w.data_ptr(), x.stride(0), w.stride(0), S, K, Hq, Hkv,
                   Hqx, D, _ptr(rope), R2, _ptr(gq), _ptr(bq), _ptr(gk), _ptr(bk), int(norm_kind), float(eps), int(batch),
                   float(q_premul), q_out.data_ptr(), _ptr(kv_out), _ptr(kv_tail), 0 if kv_out is None else kv_out.stride(0),
                   0 if kv_tail is None else kv_tail.stride(0), int(n_cache_rows), _ptr(qx_out))
    return q_out, kv_out, kv_tail, qx_out


def _rows(t: torch.Tensor, name: str) -> None:
    if t.dim() != 2 or t.dtype != torch.bfloat16 or t.stride(1) != 1 or not t.is_cuda:
        raise ValueError(f"{name} must be a 2-D bf16 device tensor with contiguous rows")


def launch_small_projections(dev: torch.device, *fields) -> None:
    """magi_small_projections with the fields of its argument struct behind struct_size, in order."""
    _launch_packed(dev, "magi_small_projections", L.SmallProjArgs, *fields)


def launch_small_projections_e4m3(dev: torch.device, q_scale: float, k_scale: float, v_out: int, *fields) -> None:
    """magi_small_projections_e4m3, the fields of the struct as above."""
    call = L.packed("magi_small_projections_e4m3", L.SmallProjArgs, C.c_float, C.c_float, C.c_void_p)
    _launch(dev, call.fn, call.pack(call.size, *fields), q_scale, k_scale, v_out)


def launch_small_layer(dev: torch.device, parts: int, *fields) -> None:
    """magi_small_layer with the fields of its argument struct behind parts, in order."""
    _launch_packed(dev, "magi_small_layer", L.SmallLayerArgs, parts, *fields)


def attention_waves(Hq: int, Hkv: int, n: int, mode: int, max_seqlen_q: int, max_seqlen_k: int) -> int:
    """The wavefronts that share a row's keys where range_attention(share_waves=True) with a bound in force does not take another form; else 0."""
    return L.lib().magi_attn_waves(Hq, Hkv, max(n, 0), mode, int(max_seqlen_q), int(max_seqlen_k))


def split_memory(dev: torch.device, Hq: int, Hkv: int, n: int, mode: int, max_seqlen_q: int, max_seqlen_k: int):
    """(the scratch memory that a bf16 call with bounded scores and MAGI_ATTN_SHARE_WAVES makes use of or None, its address, its bytes)"""
    size = 0
    if max_seqlen_k >= 512 and not attention_waves(Hq, Hkv, n, mode, max_seqlen_q, max_seqlen_k):
        size = _bounded_split_bytes(Hq, Hkv, n, max_seqlen_q, max_seqlen_k)
    if not size:
        return None, 0, 0
    t = torch.empty(size, dtype=torch.uint8, device=dev)
    return t, t.data_ptr(), size


def launch_quantize_fp8_split(dev: torch.device, *fields) -> None:
    """magi_quantize_fp8_split with the fields of its argument struct behind struct_size, in order."""
    _launch_packed(dev, "magi_quantize_fp8_split", L.QuantizeArgs, *fields)


def launch_text_attention(dev: torch.device, q: int, rows: int, Hq: int, kv: int, total_k: int, Hkv: int, cu_q: torch.Tensor, cu_k: torch.Tensor,
                          n: int, max_seqlen_q: int, max_seqlen_k: int, out: int, o_row: int, group_heads: int, o_group: int, clear: bool,
                          bound: float, gamma: int, beta: int, eps: float) -> None:
    """range_attention for a caller that has made its tensors itself and knows them to be sound: raw bf16 q rows by address, normalised
    with gamma, beta and eps (rows and heads contiguous, as K | V interleaved per head at kv), cumulative lengths, scores bounded (0 <
    bound <= MAGI_SCORE_BOUND_MAX).  clear: rows no range covers become zeros (the caller has cleared `out` unless covered_by_launch).
    Shares keys as range_attention does."""
    max_seqlen_q, max_seqlen_k = int(max_seqlen_q), int(max_seqlen_k)
    split, split_at, split_bytes = split_memory(dev, Hq, Hkv, n, L.MAGI_RANGES_CU, max_seqlen_q, max_seqlen_k)
    cu_q, cu_k = cu_q.contiguous(), cu_k.contiguous()
    flags = L.MAGI_ATTN_SHARE_WAVES | (L.MAGI_ATTN_ZERO_UNCOVERED if clear and covered_by_launch(n, max_seqlen_q, rows) else 0)
    kv_row = Hkv * 256
    _launch_packed(
        dev, "magi_attn_fwd", L.AttnArgs, q, kv, kv + 256, 0, 0, out, 0, cu_q.data_ptr(), cu_k.data_ptr(), 0, 0, 0,
        Hq * 128, 128, kv_row, 256, kv_row, 256, o_row, 128, rows, total_k, total_k, max(n, 0), L.MAGI_RANGES_CU, max_seqlen_q, max_seqlen_k, Hq, Hkv,
        128, L.MAGI_DTYPE_BF16, 0, 0.0, flags, group_heads, o_group, bound, 0, gamma, beta, eps, L.MAGI_NORM_LAYERNORM_1P, 0, 0, 0, 0, 0, 0,
        split_at, split_bytes)


def launch_fp8_attention(dev: torch.device, q: int, rows: int, Hq: int, k: int, v: int, k_side: int, v_side: int, k_split: int, total_k: int,
                         Hkv: int, scales: tuple, chunk_tokens: int, q_ranges: torch.Tensor, k_ranges: torch.Tensor, n: int, max_seqlen_q: int,
                         max_seqlen_k: int, out: int, o_row: int, group_heads: int, o_group: int, clear: bool, fast_exp2: bool) -> None:
    """The same for the core attention of e4m3 rows with power-of-two scales, heads and rows contiguous, ranges in pairs: K and V rows at
    k / v, those from k_split on at k_side / v_side (0: none); scales: the tables of q, k, v, and of k and v there (0: none) by address."""
    max_seqlen_q, max_seqlen_k = int(max_seqlen_q), int(max_seqlen_k)
    split, split_bytes = None, 0
    if max_seqlen_k >= 512:
        split_bytes = L.lib().magi_attn_split_bytes(Hq, Hkv, max(n, 0), max_seqlen_q, max_seqlen_k, L.MAGI_DTYPE_FP8_E4M3)
        if split_bytes:
            split = torch.empty(split_bytes, dtype=torch.uint8, device=dev)
    q_ranges, k_ranges = q_ranges.contiguous(), k_ranges.contiguous()
    qs, ks, vs, k2s, v2s = scales
    flags = (L.MAGI_ATTN_FP8_POW2_PRESCALED | (L.MAGI_ATTN_FP8_FAST_EXP2 if fast_exp2 else 0)
             | (L.MAGI_ATTN_ZERO_UNCOVERED if clear and covered_by_launch(n, max_seqlen_q, rows) else 0))
    row = Hkv * 128
    _launch_packed(
        dev, "magi_attn_fwd", L.AttnArgs, q, k, v, k_side, v_side, out, 0, q_ranges.data_ptr(), k_ranges.data_ptr(), qs, ks, vs, Hq * 128, 128, row, 128,
        row, 128, o_row, 128, rows, total_k, k_split, max(n, 0), L.MAGI_RANGES_PAIRS, max_seqlen_q, max_seqlen_k, Hq, Hkv, 128,
        L.MAGI_DTYPE_FP8_E4M3, chunk_tokens, 0.0, flags, group_heads, o_group, 0.0, 0, 0, 0, 0.0, 0, k2s, v2s, 0, 0, 0, 0,
        0 if split is None else split.data_ptr(), split_bytes)


def small_projections(x: Optional[torch.Tensor], w: Optional[torch.Tensor], rope, gq, bq, gk, bk, *, Hq: int, Hkv: int, Hqx: int = 0,
                      ln: Optional[tuple] = None, eps: float = 1e-6, batch: int = 1, q_premul: float = 1.0,
                      kv_out: Optional[torch.Tensor] = None, n_cache_rows: Optional[int] = None,
                      kv_tail: Optional[torch.Tensor] = None, text: Optional[tuple] = None):
    """The projections of a small layer and what comes around them in one launch (magi_small_projections).

    x [S, K] bf16 (None: no such rows): ln = (weight, bias, eps) normalises it first; w [(Hq + 2 Hkv + Hqx) * 128, K] bf16 with rows
    ordered q | k | v | qx heads; rope, norm parameters, q_premul, batch and the K | V destinations as in qk_prologue.  qx leaves raw.
    text = (rows [T, Kt], weight [2 Hkv 128, Kt], gamma, beta): K | V of the text tokens, K normed.
    -> (q [S, Hq, 128], kv_out, kv_tail, qx [S, Hqx, 128], text K | V [T, Hkv, 256]); None for what was not
    asked for."""
    D = 128
    q = qx = text_kv = None
    S = K = R2 = ln_fp32 = 0
    ln_eps = 0.0
    ln_w = ln_b = 0
    dev = None
    if x is not None:
        _rows(x, "x")
        _rows(w, "w")
        S, K = x.shape
        dev = x.device
        if w.shape != ((Hq + 2 * Hkv + Hqx) * D, K) or not w.is_contiguous() or w.device != dev:
            raise ValueError("w must be a contiguous [(Hq + 2 Hkv + Hqx) * 128, K] tensor on x's device")
        if ln is not None:
            lw, lb, ln_eps = ln
            if (lw.shape != (K,) or lb.shape != (K,) or lw.dtype != lb.dtype or lw.dtype not in (torch.bfloat16, torch.float32)
                    or not (lw.is_contiguous() and lb.is_contiguous()) or lw.device != dev or lb.device != dev):
                raise ValueError("ln must be (weight, bias, eps) with contiguous bf16 or fp32 [K] tensors on x's device")
            ln_w, ln_b, ln_fp32 = lw.data_ptr(), lb.data_ptr(), int(lw.dtype is torch.float32)
        if kv_out is None and kv_tail is None:
            kv_out, n_cache_rows = torch.empty((S, Hkv, 2 * D), dtype=torch.bfloat16, device=dev), S
        if n_cache_rows is None:
            n_cache_rows = S if kv_tail is None else 0
        for name, t, rows in (("kv_out", kv_out, n_cache_rows), ("kv_tail", kv_tail, S - n_cache_rows)):
            if t is None:
                if rows:
                    raise ValueError(f"{name} is needed for {rows} rows")
            elif t.dtype != torch.bfloat16 or t.shape[1:] != (Hkv, 2 * D) or t.stride(2) != 1 or t.stride(1) != 2 * D or t.shape[0] < rows:
                raise ValueError(f"{name} must be bf16 [>= {rows}, Hkv, 2*D] with contiguous heads")
        if rope is not None:
            if rope.dtype != torch.float32 or rope.dim() != 2 or rope.shape[0] * max(batch, 1) != S or not rope.is_contiguous():
                raise ValueError("rope must be a contiguous fp32 [S / batch, 2*R2] tensor")
            R2 = rope.shape[1] // 2
        q = torch.empty((S, Hq, D), dtype=torch.bfloat16, device=dev)
        if Hqx:
            qx = torch.empty((S, Hqx, D), dtype=torch.bfloat16, device=dev)
        gq, bq, gk, bk = _fp32(gq), _fp32(bq), _fp32(gk), _fp32(bk)
    T = Kt = 0
    tx = wt = gkx = bkx = None
    if text is not None:
        tx, wt, gkx, bkx = text
        _rows(tx, "text")
        _rows(wt, "the text weight")
        T, Kt = tx.shape
        dev = tx.device
        if wt.shape != (2 * Hkv * D, Kt) or not wt.is_contiguous() or wt.device != dev or (x is not None and x.device != dev):
            raise ValueError("the text weight must be a contiguous [2 Hkv 128, Kt] tensor on the text's device")
        gkx, bkx = _fp32(gkx), _fp32(bkx)
        text_kv = torch.empty((T, Hkv, 2 * D), dtype=torch.bfloat16, device=dev)
    if dev is None:
        raise ValueError("neither x nor text given")
    launch_small_projections(
        dev, _ptr(x), _ptr(w) if x is not None else 0, ln_w, ln_b,
        x.stride(0) if S > 1 else K, S, K, ln_fp32, ln_eps, Hq, Hkv, Hqx, R2, _ptr(rope) if R2 else 0, _ptr(gq), _ptr(bq), _ptr(gk),
        _ptr(bk), eps, batch, q_premul,
        n_cache_rows or 0, _ptr(q), _ptr(kv_out), _ptr(kv_tail),
        0 if kv_out is None else kv_out.stride(0), 0 if kv_tail is None else kv_tail.stride(0), _ptr(qx), _ptr(tx), _ptr(wt),
        (tx.stride(0) if T > 1 else Kt) if tx is not None else 0, T, Kt, _ptr(gkx), _ptr(bkx), _ptr(text_kv))
    return q, kv_out, kv_tail, qx, text_kv


def pow2_scale_for(bound: float) -> float:
    """Smallest power of two s with bound / s <= 448 (the largest e4m3 value): the scale to quantise values of
    magnitude <= bound with.  e4m3 being a floating-point format, a bound that is a few times too large costs
    no precision."""
    if not (bound > 0.0) or bound == float("inf"):
        raise ValueError("bound must be positive and finite")
    m, e = math.frexp(bound / 448.0)  # bound / 448 = m * 2^e, 0.5 <= m < 1
    return math.ldexp(1.0, e - 1 if m == 0.5 else e)


def layer_norm(x: torch.Tensor, weight: Optional[torch.Tensor], bias: Optional[torch.Tensor], eps: float = 1e-5,
               out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """LayerNorm over the last axis of a bf16 tensor with fp32 statistics: the layer input norm of
    CustomLayerNormLinear.forward_ln (dit_module.py:401, 412-413).  weight / bias: bf16 or fp32 [cols] or None.
    Rows may be strided (last axis contiguous, leading axes collapsible to one row stride)."""
    if x.dtype != torch.bfloat16:
        raise TypeError("x must be bf16")
    if not x.is_cuda:
        raise ValueError("x must be a device tensor (there is no CPU path)")
    cols = x.shape[-1]
    x2 = x if x.dim() == 2 else x.reshape(-1, cols)  # a view when the leading axes collapse, else a copy
    if x2.stride(-1) != 1:
        x2 = x2.contiguous()
    y = torch.empty(x.shape, dtype=torch.bfloat16, device=x.device) if out is None else out
    if y.shape != x.shape or y.dtype != torch.bfloat16 or y.device != x.device or not y.is_contiguous():
        raise ValueError("out must be a contiguous bf16 tensor of x's shape on x's device")
    fp32 = None
    for name, p in (("weight", weight), ("bias", bias)):
        if p is None:
            continue
        if p.shape != (cols,) or not p.is_contiguous() or p.device != x.device:
            raise ValueError(f"{name} must be a contiguous [{cols}] tensor on x's device")
        if p.dtype not in (torch.bfloat16, torch.float32):
            raise TypeError(f"{name} must be bf16 or fp32")
        if fp32 is not None and fp32 != (p.dtype == torch.float32):
            raise TypeError("weight and bias must share a dtype")
        fp32 = p.dtype == torch.float32
    rows = x2.shape[0]
    _launch(x.device, L.lib().magi_layer_norm, x2.data_ptr(), x2.stride(0) if rows > 1 else cols, _ptr(weight), _ptr(bias),
            int(bool(fp32)), y.data_ptr(), cols, rows, cols, float(eps))
    return y


def div_clamp_to(x: torch.Tensor, scale: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """e4m3fn(bf16(clamp(x.float() / scale.float(), -448, 448))): the input quantiser of the reference's fp8 linears
    (dit_module.py:364-384), double rounding included.  x: bf16, last axis contiguous (leading axes collapsible to one
    row stride); scale: fp32 with one element or one per element of the last axis.  -> float8_e4m3fn, x's shape."""
    if x.dtype != torch.bfloat16:
        raise TypeError("x must be bf16")
    if not x.is_cuda:
        raise ValueError("x must be a device tensor (there is no CPU path)")
    cols = x.shape[-1]
    x2 = x if x.dim() == 2 else x.reshape(-1, cols)
    if x2.stride(-1) != 1:
        x2 = x2.contiguous()
    sc = scale.detach().to(device=x.device, dtype=torch.float32).reshape(-1).contiguous()
    if sc.numel() not in (1, cols):
        raise ValueError("scale must have one element, or one per element of x's last axis")
    y = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device) if out is None else out
    if y.shape != x.shape or y.dtype != torch.float8_e4m3fn or y.device != x.device or not y.is_contiguous():
        raise ValueError("out must be a contiguous float8_e4m3fn tensor of x's shape on x's device")
    rows = x2.shape[0]
    _launch(x.device, L.lib().magi_div_clamp_to_e4m3, x2.data_ptr(), x2.stride(0) if rows > 1 else cols, sc.data_ptr(), sc.numel(),
            y.data_ptr(), cols, rows, cols)
    return y


def layer_norm_div_clamp(x: torch.Tensor, weight: Optional[torch.Tensor], bias: Optional[torch.Tensor], scales, eps: float = 1e-5,
                         out=None):
    """[div_clamp_to(layer_norm(x, weight, bias, eps), s) for s in scales] in one launch, bit for bit the same, without the
    normalised rows in memory (magi_layer_norm_e4m3).  x: contiguous bf16 [..., cols], cols a multiple of 8 up to 8192;
    scales: 1 to 4 contiguous fp32 [cols] tensors.  -> float8_e4m3fn [len(scales), ..., cols]; or `out`, one contiguous
    float8_e4m3fn tensor of x's shape per scale (tensors of their own can be given back one by one)."""
    if x.dtype != torch.bfloat16:
        raise TypeError("x must be bf16")
    cols = x.shape[-1]
    if not x.is_cuda or not x.is_contiguous():
        raise ValueError("x must be a contiguous device tensor (there is no CPU path)")
    fp32 = None
    for name, p in (("weight", weight), ("bias", bias)):
        if p is None:
            continue
        if p.shape != (cols,) or not p.is_contiguous() or p.device != x.device or p.dtype not in (torch.bfloat16, torch.float32):
            raise ValueError(f"{name} must be a contiguous bf16 or fp32 [{cols}] tensor on x's device")
        if fp32 is not None and fp32 != (p.dtype == torch.float32):
            raise TypeError("weight and bias must share a dtype")
        fp32 = p.dtype == torch.float32
    n = len(scales)
    for s in scales:
        if s.dtype != torch.float32 or s.shape != (cols,) or not s.is_contiguous() or s.device != x.device:
            raise ValueError(f"scales must be contiguous fp32 [{cols}] tensors on x's device")
    y = torch.empty((n,) + x.shape, dtype=torch.float8_e4m3fn, device=x.device) if out is None else out
    if out is not None and (len(out) != n or any(t.shape != x.shape or t.dtype != torch.float8_e4m3fn or t.device != x.device
                                                 or not t.is_contiguous() for t in out)):
        raise ValueError("out must be one contiguous float8_e4m3fn tensor of x's shape per scale, on x's device")
    rows = x.numel() // max(cols, 1)
    sp = (C.c_void_p * n)(*[s.data_ptr() for s in scales])
    yp = (C.c_void_p * n)(*[t.data_ptr() for t in (y.unbind(0) if out is None else out)])
    _launch(x.device, L.lib().magi_layer_norm_e4m3, x.data_ptr(), cols, _ptr(weight), _ptr(bias), int(bool(fp32)), sp, yp, n, rows,
            cols, float(eps))
    return y


def head_norm(x: torch.Tensor, gamma, beta, eps: float = 1e-6, norm_kind: int = L.MAGI_NORM_LAYERNORM_1P):
    """x [S, H, 128] bf16 (strided heads allowed) -> contiguous normalised copy."""
    _check_thd(x, "x")
    if x.dtype != torch.bfloat16:
        raise TypeError("x must be bf16")
    S, H, D = x.shape
    y = torch.empty((S, H, D), dtype=torch.bfloat16, device=x.device)
    g, b = _fp32(gamma), _fp32(beta)
    _launch(x.device, L.lib().magi_head_norm, x.data_ptr(), x.stride(0), x.stride(1), _ptr(g), _ptr(b), y.data_ptr(), S, H, D,
            int(norm_kind), float(eps))
    return y


def quantize_fp8(x: torch.Tensor, chunk_tokens: int, premul: float = 1.0, pow2_scales: bool = False,
                 out: Optional[torch.Tensor] = None, scales_out: Optional[torch.Tensor] = None):
    """x [T, H, 128] bf16 (strided heads allowed) -> (y [T, H, 128] float8_e4m3fn, scales [ceil(T/chunk), H] fp32)
    with x * premul ~= y * scales[t // chunk_tokens, h]: per-(chunk, head) absmax * |premul| / 448 (rounded up to a
    power of two with pow2_scales), saturating OCP e4m3fn.

    out / scales_out: contiguous destinations (e.g. the rows of an fp8 KV cache at the write position and the
    matching rows of its scale table) instead of fresh tensors.

    For the fast attention mode quantise q with premul = softmax_scale * log2(e) and q, k, v with pow2_scales,
    then pass fp8_pow2_prescaled=True to range_attention."""
    _check_thd(x, "x")
    if x.dtype != torch.bfloat16:
        raise TypeError("x must be bf16")
    T, H, D = x.shape
    n_chunks = (T + chunk_tokens - 1) // chunk_tokens
    y = torch.empty((T, H, D), dtype=torch.float8_e4m3fn, device=x.device) if out is None else out
    scales = torch.empty((n_chunks, H), dtype=torch.float32, device=x.device) if scales_out is None else scales_out
    if y.dtype != torch.float8_e4m3fn or tuple(y.shape) != (T, H, D) or not y.is_contiguous() or y.device != x.device:
        raise ValueError("out must be a contiguous float8_e4m3fn [T, H, 128] tensor on x's device")
    if (scales.dtype != torch.float32 or tuple(scales.shape) != (n_chunks, H) or not scales.is_contiguous()
            or scales.device != x.device):
        raise ValueError("scales_out must be a contiguous fp32 [ceil(T / chunk_tokens), H] tensor on x's device")
    _launch(x.device, L.lib().magi_quantize_fp8, x.data_ptr(), x.stride(0), x.stride(1), y.data_ptr(), scales.data_ptr(), T, H, D,
            int(chunk_tokens), float(premul), int(pow2_scales))
    return y, scales


def quantize_fp8_split(x: torch.Tensor, chunk_tokens: int, n_rows_first: int, out: Optional[torch.Tensor],
                       scales_out: Optional[torch.Tensor], out2: Optional[torch.Tensor],
                       scales2_out: Optional[torch.Tensor], premul: float = 1.0, pow2_scales: bool = False,
                       row_max: Optional[torch.Tensor] = None) -> None:
    """quantize_fp8 in ONE launch with two destinations (magi_quantize_fp8_split): tokens below n_rows_first (a
    multiple of chunk_tokens unless it is T) go to out / scales_out, e.g. the rows of an fp8 KV cache at the write
    position and the matching rows of its scale table; the others to out2 / scales2_out, indexed from
    n_rows_first.  Destinations are contiguous and at least as long as their share; a share of zero rows may
    pass None.  row_max: the largest magnitudes of x's rows as qk_prologue_fp8 leaves them (int16 [H, T]), instead of a pass over x for
    them; the same bytes."""
    _check_thd(x, "x")
    if x.dtype != torch.bfloat16:
        raise TypeError("x must be bf16")
    T, H, D = x.shape
    n1 = int(n_rows_first)
    if not (0 <= n1 <= T) or (n1 < T and n1 % chunk_tokens):
        raise ValueError("n_rows_first must lie in [0, T] and, below T, be a multiple of chunk_tokens")
    for name, y, sc, rows in (("out", out, scales_out, n1), ("out2", out2, scales2_out, T - n1)):
        if rows == 0:
            continue
        chunks = (rows + chunk_tokens - 1) // chunk_tokens
        if (y is None or y.dtype != torch.float8_e4m3fn or y.dim() != 3 or y.shape[0] < rows or tuple(y.shape[1:]) != (H, D)
                or not y.is_contiguous() or y.device != x.device):
            raise ValueError(f"{name} must be a contiguous float8_e4m3fn [>= {rows}, H, 128] tensor on x's device")
        if (sc is None or sc.dtype != torch.float32 or sc.dim() != 2 or sc.shape[0] < chunks or sc.shape[1] != H
                or not sc.is_contiguous() or sc.device != x.device):
            raise ValueError(f"the scales of {name} must be a contiguous fp32 [>= {chunks}, H] tensor on x's device")
    fields = (x.data_ptr(), x.stride(0), x.stride(1), T, H, D, int(chunk_tokens), float(premul), int(pow2_scales), _ptr(out),
              _ptr(scales_out), n1, _ptr(out2), _ptr(scales2_out))
    if row_max is None:
        _launch_packed(x.device, "magi_quantize_fp8_split", L.QuantizeArgs, *fields)
        return
    if row_max.dtype != torch.int16 or tuple(row_max.shape) != (H, T) or not row_max.is_contiguous() or row_max.device != x.device:
        raise ValueError("row_max must be a contiguous int16 [H, T] tensor on x's device")
    call = L.packed("magi_quantize_fp8_row_max", L.QuantizeArgs, C.c_void_p)
    _launch(x.device, call.fn, call.pack(call.size, *fields), row_max.data_ptr())
