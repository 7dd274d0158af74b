"""The DiT attention layer over libmagi_attn, with the interface of the reference's
FullyParallelAttention for cp_strategy == "none"
(inference/model/dit/dit_module.py:776-1173).

Method names, argument meaning and returned layouts follow the reference so that
TransformerLayer-level code can call it unchanged:

  forward(hidden_states [S,b,h], key_value_states [Ty,h*ratio], inference_params,
          rotary_pos_emb [S,96], meta_args) -> (core_attn_out [S,b,Hq*D], xattn_out [S,b,Hq*D])

What differs is what happens underneath:
  * get_q / get_k / get_v / get_kv: the upcast, LayerNorm, transpose, rotary, downcast and
    re-layout passes are one fused kernel launch;
  * the KV cache is appended to in place by that same launch and READ in place by the
    attention kernel (strided K / V views of the interleaved cache), so the prefix slice,
    the cat and the contiguous copies of _full_adjust_key_and_value / core_attention vanish;
  * when the cache must not be updated (update_kv_cache False, or the last chunk under
    distill_nearly_clean_chunk) the new KV goes to a side buffer and the kernel walks
    [cache prefix | side buffer] as one key axis.

The linear projections and the input LayerNorm are plain library GEMMs / ops (torch on
rocBLAS / hipBLASLt); they are not part of this library.  forward() runs the four projections
q, k, v, qx as ONE GEMM over a shared weight buffer (CustomLayerNormLinear.forward_qkvx).
"""
from __future__ import annotations

from typing import Callable, Optional, Tuple

import itertools
import math
import operator
import os

import torch

from . import _lib as L
from .cache import Fp8KVCache, OffloadedKVCache
from .functional import (_measuring_a_bound_pays, covered_by_launch, launch_fp8_attention, launch_quantize_fp8_split,
                         launch_small_projections_e4m3, launch_text_attention, range_count, split_memory)
from .functional import BegunCalls, _compute_units, attention_waves, launch_held
from .functional import launch_small_layer as launch_small_projections  # (named by the first of the launches it stands for)
from .functional import (div_clamp_to, head_norm, layer_norm, layer_norm_div_clamp, pow2_scale_for, qk_prologue, qk_prologue_fp8, qkv_proj_prologue,
                         quantize_fp8_split,
                         range_attention, small_projections)
from .params import InferenceParams, ModelMetaArgs, PackedCrossAttnParams


# Epochs of all FusedLayerNorm instances (itertools.count draws are atomic): two modules never share one, and neither do the
# modules of two processes, one of which may have been pickled in the other.
_EPOCHS = itertools.count(int.from_bytes(os.urandom(6), "little"))

PROJ_GROUPS = 8  # head groups of the linear_proj input (hard-coded "hn=8", dit_module.py:1338)


def _halves(kv: torch.Tensor, rows: int) -> Tuple[torch.Tensor, torch.Tensor]:
    """(K, V) views [rows, H, D] of the first rows of an interleaved [tokens, H, 2*D] tensor."""
    st, sh, _ = kv.stride()
    D, off = kv.shape[2] // 2, kv.storage_offset()
    size = (rows, kv.shape[1], D)
    return kv.as_strided(size, (st, sh, 1), off), kv.as_strided(size, (st, sh, 1), off + D)


def attn_linear_proj_input(core_attn_out: torch.Tensor, cross_attn_out: torch.Tensor) -> torch.Tensor:
    """[sq, b, Hq*D] x 2 -> [sq, b, 2*Hq*D] in "(hn n hd)" order: the concat + rearrange that precedes linear_proj
    in attn_linear_proj (dit_module.py:1336-1339), done with torch copies."""
    sq, b, hd = core_attn_out.shape
    both = torch.stack([core_attn_out.reshape(sq, b, PROJ_GROUPS, hd // PROJ_GROUPS),
                        cross_attn_out.reshape(sq, b, PROJ_GROUPS, hd // PROJ_GROUPS)], dim=3)
    return both.reshape(sq, b, 2 * hd)


def _param(m: torch.nn.Module, name: str) -> torch.Tensor:
    """m.<name>: straight from the parameters where it is one (attribute lookup on a module costs several times as much), else
    whatever the attribute gives (parametrised, sharded and wrapped modules)."""
    p = m._parameters.get(name)
    return p if p is not None else getattr(m, name)


class FusedLayerNorm(torch.nn.Module):
    """Parameter holder of a per-head LayerNorm with zero-centred gamma (dit_module.py:323-357).
    The arithmetic runs inside the fused kernels; forward() is the stand-alone form."""

    def __init__(self, hidden_size: int, eps: float = 1e-6, zero_centered_gamma: bool = True,
                 dtype=torch.bfloat16, device=None):
        super().__init__()
        self.eps = eps
        self.zero_centered_gamma = zero_centered_gamma
        self.weight = torch.nn.Parameter(torch.zeros(hidden_size, dtype=dtype, device=device))
        self.bias = torch.nn.Parameter(torch.zeros(hidden_size, dtype=dtype, device=device))

    def gamma_beta_fp32(self) -> Tuple[torch.Tensor, torch.Tensor]:
        """(gamma - 1 form, beta) as the kernels take them.  weight + 1 is formed in the parameter
        dtype first, as the reference does, so a bf16 parameter rounds the same way.  Converted once per set of
        parameter values (no launches on later calls) and kept until a parameter is modified or replaced."""
        # (a write through `.data` does not advance _version: callers that patch parameters that way call
        # invalidate_cached_parameters())
        w, b = _param(self, "weight"), _param(self, "bias")
        state = self.__dict__
        # (the two parameters are held, so that a new one cannot come to lie where the old one was; a parametrised weight,
        # computed anew for every look at it, is no parameter and is converted every time)
        held = state.get("_gb_key", (None, None))
        if (held[0] is not w or held[1] is not b
                or held[2] != (w._version, w.data_ptr(), w.dtype, b._version, b.data_ptr(), b.dtype)):
            own = w is self._parameters.get("weight") and b is self._parameters.get("bias")
            key = (w, b, (w._version, w.data_ptr(), w.dtype, b._version, b.data_ptr(), b.dtype)) if own else (None, None)
            g = w.detach()
            g = ((g + 1).float() - 1.0) if self.zero_centered_gamma else (g.float() - 1.0)
            state["_gb"] = (g.contiguous(), b.detach().float().contiguous())
            state["_gb_key"] = key
            state["_gb_epoch"] = next(_EPOCHS)
        return state["_gb"]

    def parameter_epoch(self) -> int:
        """A number that is drawn anew whenever gamma_beta_fp32() had to convert the parameters, and that no other module
        has: what values derived from the parameters (score bounds, quantisation scales) key their own caches on."""
        self.gamma_beta_fp32()
        return self.__dict__["_gb_epoch"]

    def invalidate_cached_parameters(self) -> None:
        self.__dict__.pop("_gb_key", None)

    def output_norm_bound(self) -> float:
        """Upper bound of the Euclidean norm of any output row: the normalised row has norm <= sqrt(n) (exactly
        sqrt(n) up to eps), so |y| <= sqrt(n) max|gamma + 1| + |beta|.  One host read of the parameters."""
        g, b = self.gamma_beta_fp32()
        n = g.numel()
        return float(math.sqrt(n) * (g + 1.0).abs().max().item() + b.norm().item())

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        g, b = self.gamma_beta_fp32()
        shape = x.shape
        y = head_norm(x.reshape(-1, shape[-2], shape[-1]).to(torch.bfloat16), g, b, self.eps)
        return y.reshape(shape).to(x.dtype)


def qk_score_bound(q_norm: FusedLayerNorm, k_norm: FusedLayerNorm, rotary_half: int = 0) -> float:
    """Upper bound of |q . k| over all rows the two norms can produce, with a rotary embedding of 2 * rotary_half
    features (pairs (i, i + rotary_half); 0 = none) applied to both.

    A normed row is n * (gamma + 1) + beta with |n|^2 <= D.  The rotation acts inside each pair and preserves the
    pair's length, so with groups p = the rotary pairs and the unpaired features one by one,
    G_p = max over the group of |gamma + 1| and B_p = the length of beta inside the group:

        |q . k| <= sum_p (Gq_p |nq_p| + Bq_p) (Gk_p |nk_p| + Bk_p)
                <= D max_p(Gq_p Gk_p) + sqrt(D) (|Gq * Bk| + |Gk * Bq|) + Bq . Bk          (Cauchy-Schwarz)

    which is never above the product of the two rows' lengths (sqrt(D) max|gamma + 1| + |beta|)^2 and is tighter
    when the large gains of the two norms sit on different features.  One host read of the parameters."""
    gq, bq = q_norm.gamma_beta_fp32()
    gk, bk = k_norm.gamma_beta_fp32()
    D = gq.numel()
    r = int(rotary_half)
    if not 0 <= 2 * r <= D:
        raise ValueError("rotary_half must satisfy 0 <= 2 * rotary_half <= head_dim")

    def groups(g, b):
        G, B2 = (g.double() + 1.0).abs(), b.double() ** 2
        if r:
            Gp, Bp = torch.maximum(G[:r], G[r:2 * r]), B2[:r] + B2[r:2 * r]
            G, B2 = torch.cat([Gp, G[2 * r:]]), torch.cat([Bp, B2[2 * r:]])
        return G, B2.sqrt()

    Gq, Bq = groups(gq, bq)
    Gk, Bk = groups(gk, bk)
    bound = (D * (Gq * Gk).max() + math.sqrt(D) * ((Gq * Bk).norm() + (Gk * Bq).norm()) + (Bq * Bk).sum())
    return float(bound.item())


def _transformed() -> bool:
    """Whether what is called is recorded or transformed (torch.compile, jit.trace, dispatch modes, vmap and the other function transforms,
    forward-mode derivatives): row counts of its own and out= are not for those."""
    return (torch.compiler.is_compiling() or torch._C._is_tracing() or torch._C._len_torch_dispatch_stack() > 0
            or torch._C._functorch.maybe_current_level() is not None or torch.autograd.forward_ad._current_level >= 0)


def _rows_ahead(rows: int, cols: int, depth: int, cus: int) -> int:
    """How many rows of a [rows, depth] x [cols, depth]^T product to run in a call of their own, 0: none.

    The library works in tiles of 256 x 256.  Where the column tiles divide the CUs, 256 * cus / tiles rows are one round of
    tiles (2048 rows at 8192 columns); one call over a number of rows in between leaves the last round partly empty or falls
    back to slower tiles.  Cut where that happens: whole rounds first, then the rest.  Measured, one call / cut, over 1 to
    41 rounds and 14 rests each at depth 3072 and 8192 columns (9360 rows 444 / 352 us, 2604 183 / 105, 25268 958 / 836, 54902
    1971 / 1852): the cut takes 1.5 % (41 rounds) to 43 % less time (one or two) as long as the rest leaves a row of
    tiles empty, 0 to 2 % more now and then; with a rest that fills its round, or with more than half a round behind a
    single one, it takes 1 to 4 % more and gains nothing, so these are left alone.  2048 and 4096 deep, and 4096 and 16384
    columns, draw the same lines.  Column counts whose tiles do not divide the CUs (14336: 56 tiles) gain nothing on
    average."""
    tiles = cols // 256
    if cols % 256 or not 0 < tiles <= cus or cus % tiles or depth < 1024:
        return 0
    row_tiles = cus // tiles  # of one round
    rounds, rest = divmod(rows, 256 * row_tiles)
    used = (rest + 255) // 256
    if rounds == 0 or used == 0 or used == row_tiles or (rounds == 1 and 2 * rest > 256 * row_tiles):
        return 0
    return rows - rest


def _linear_in_whole_rounds(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """torch.nn.functional.linear(x, w), the rows cut in two where that suits the library's tiles better (_rows_ahead)."""
    cols, depth = w.shape
    if (depth >= 1024 and cols % 256 == 0 and x.is_cuda and x.is_contiguous() and x.dtype is w.dtype
            and not torch.is_autocast_enabled() and not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad)) and not torch._C._is_tracing()):
        rows = x.numel() // depth
        head = _rows_ahead(rows, cols, depth, _compute_units(x.device))
        if head and not _transformed():
            x2, wt = x.view(rows, depth), w.t()
            y = torch.empty((rows, cols), dtype=x.dtype, device=x.device)
            torch.mm(x2[:head], wt, out=y[:head])
            torch.mm(x2[head:], wt, out=y[head:])
            return y.view(x.shape[:-1] + (cols,))
    return torch.nn.functional.linear(x, w)


def _rows_ahead_e4m3(rows: int, cols: int, depth: int, cus: int) -> int:
    """The same for the library's e4m3 product: the rows that are rounds of 256 x 256 tiles whole to the last one, where at most a seventh as
    many are left.

    Just behind such rounds the library takes smaller tiles for all rows: at 1024 columns and depth 3072 16384 rows are 39 us, 16974 99, cut
    47; at 6144 columns and depth 6144 86400 rows 2231 / 2115.  Measured, one call / cut, over eight weights and 100 row counts: 92 within the
    line take 0.98 to 1.93 times as long in one call, 1.17 on average; with more rows left 0.74 to 1.29, even on average (1024 columns,
    depth 3072: 21600 rows 61 / 65, 28080 67 / 71; behind rounds that end within a row of tiles, 6144 columns: 14155 rows 362 / 469).
    The library's kernels for the two numbers of rows may add in another order: of the fp32 sums of 86400 rows 6144 deep one in 16000 to 100000
    differs by its last bits, next to none rounds to another bf16 (three of nine draws of the 720p layer have 12 to 76 other outputs
    of 1.06e9); the error against float64 is the same to five digits."""
    tiles = cols // 256
    if rows * cols < 65536 * cus or cols % 256 or not 0 < tiles <= cus or depth < 1024:  # (less than one round, ...)
        return 0
    whole = 256 * (cus // math.gcd(cus, tiles))
    head = rows // whole * whole
    return head if 0 < 7 * (rows - head) <= head else 0


_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _plain_weight(w: torch.Tensor, heads: int, K: int, device: torch.device) -> bool:
    """Whether w is as small_projections takes a weight: plain bf16 rows [heads * 128, K], K a multiple of 64, aligned, on the device;
    no subclass of tensors with a product of its own, no autocast that would have the library's product convert it."""
    return (type(w) in _PLAIN and w.shape == (128 * heads, K) and w.dtype is torch.bfloat16 and K % 64 == 0 and w.is_contiguous()
            and w.device == device and w.data_ptr() % 16 == 0 and not torch.is_autocast_enabled())


def _plain_rows(x: torch.Tensor, w: torch.Tensor, heads: int) -> bool:
    """The same of the rows x [rows, K] and their weight w."""
    if type(x) not in _PLAIN or x.dim() != 2 or x.dtype is not torch.bfloat16 or not x.is_cuda:
        return False
    rows, K = x.shape
    st = x.stride()
    return (rows > 0 and st[1] == 1 and K <= st[0] <= 1 << 24 and st[0] % 8 == 0 and x.data_ptr() % 16 == 0
            and _plain_weight(w, heads, K, x.device))


def _projects_in_one_launch(rows: int, heads: int, text_rows: int, text_heads: int, K: int, cus: int) -> bool:
    """Whether a layer's projections run as one launch of small_projections: where its workgroups (32 rows x one head each, 64 rows up
    to K = 768) are one round, or up to four of the taller ones.  In one round the launch takes less time than the norm, the library's
    two products, the prologue and the text's head norm (K = 768, 20 + 4 heads, 24 text rows: 240 rows 11.6 / 22.1 us, 768 rows 17.8 / 25.7), in
    several more (840 rows 29.6 / 26.9, 1344 32.7 / 30.4, 2048 48.1 / 35.7), but the host issues the layer 80 us sooner and such layers wait
    for it: 840 rows over 1260 keys 68 / 150 us in all, 1344 over 2688 76 / 154, 2048 over 6144 118 / 154.
    Replayed from a graph, which waits for no host, the same layers take 70 / 71, 79 / 77, 120 / 108 us.  The choice does not look at whether the
    stream is being captured all the same: an eager pass ahead of the capture would not have brought the library's product up, and
    bringing it up is not permitted in a capture."""
    tile = lambda n: ((rows + n - 1) // n) * heads + ((text_rows + n - 1) // n) * text_heads  # noqa: E731
    return tile(64) <= 4 * cus if K <= 768 else tile(32) <= cus


def _text_in_one_launch(flop: float, rows: int, heads: int, K: int, cus: int) -> bool:
    """Whether the K | V projection of the text rows and the K norm run as one launch of small_projections rather than as the library's
    product and a head norm.  The host takes 8.5 instead of 29 us for it, which counts where the layer is waiting for it: whole layers of
    24 heads, 468 rows over 2340 keys (3.1e10 flop) 151 / 132 us, two chunks of 648 rows with 348 text rows (9e10) 162 / 160, 900 rows over 4500
    keys in fp8 with 300 (8.4e10) 268 / 247; from 7e10 on with fewer than 200 text rows 924 over 4620 in fp8 191 / 198.  In one round of its
    workgroups (32 rows x one of the `heads`): more rows (64 a workgroup then) gain nothing, four chunks of 1170 rows with 674 in
    all 374 / 376.  At K = 6144 the product is the faster one (400 rows 25 / 29 us).
    Up to 2^17 results of a long sum the library cuts K in pieces (64 rows at 16 heads, 128 at 8): another order of the sums, other bits.
    Those layers keep the library's.
    On the device, weights out of memory, norm and product / this launch: K = 768 and 4 heads 10.3 / 7.7 us with 100 rows; K = 3072 and 16 heads
    14.5 / 19.4 with 100, 19.8 / 18.6 with 130, 21.1 / 17.7 with 300, 8 heads 14.1 / 17.6 with 200 and 19.0 / 17.1 with 300: it is the
    host's time that decides up to 2^18 results, in a captured stream too (see _projects_in_one_launch)."""
    return (flop < 7e10 or rows >= 200) and K <= 3072 and (K <= 1024 or rows * heads > 1024) and (rows + 31) // 32 * heads <= cus


def _global_hooks() -> bool:
    """Whether hooks are registered that see every module's call (torch.nn.modules.module.register_module_forward_hook)."""
    return bool(torch.nn.modules.module._has_any_global_hook())


class _Own:
    """The library's functions of these names in a class of modules.  of(m): whether calling them on m runs the library's code as it
    stands here, no other class, no patch of the class and none of the instance replaces one."""

    def __init__(self, cls: type, *names: str):
        self.cls, self.names = cls, names
        self.get = operator.attrgetter(*names) if len(names) > 1 else lambda t, _get=operator.attrgetter(*names): (_get(t),)
        self.functions = self.get(cls)

    def of(self, m: torch.nn.Module) -> bool:
        return isinstance(m, self.cls) and self.get(type(m)) == self.functions and m.__dict__.keys().isdisjoint(self.names)


class PerTensorQuantizedFp8Linear(torch.nn.Module):
    """The reference's fp8 linear layer (dit_module.py:431-456) with its parameter names and shapes, so that its
    checkpoints load: `weight` [1, out, in] float8_e4m3fn, `weight_scale` [1] fp32, `input_scale` [in] fp32.

    forward: x8 = div_clamp_to(x, input_scale) (magi_div_clamp_to_e4m3: the reference's quantiser, bf16 intermediate
    included), then the library's fp8 GEMM with fp32 accumulation, de-quantised by input_scale * weight_scale, bf16
    out (the reference calls flashinfer's bmm_fp8, which reads ONE value behind each scale pointer: with the
    per-channel shape the reference gives input_scale, that is its first element, as here).  The GEMM itself is
    a library routine (hipBLASLt through torch._scaled_mm), like the bf16 projections'."""

    def __init__(self, in_features: int, out_features: int, bias=False, dtype=torch.bfloat16, device=None) -> None:
        super().__init__()
        self.in_features, self.out_features, self.output_dtype = in_features, out_features, dtype
        P_ = torch.nn.Parameter
        self.weight = P_(torch.zeros((1, out_features, in_features), device=device).to(torch.float8_e4m3fn), requires_grad=False)
        self.weight_scale = P_(torch.ones(1, dtype=torch.float32, device=device), requires_grad=False)
        self.input_scale = P_(torch.ones(in_features, dtype=torch.float32, device=device), requires_grad=False)

    @classmethod
    def from_linear(cls, lin: torch.nn.Linear, input_absmax: float) -> "PerTensorQuantizedFp8Linear":
        """Per-tensor quantisation of a bf16 linear layer (for tests and calibration scripts): weight scale from the
        weight's absmax, input scale from the given absmax of the inputs, both so that the maximum maps to 448."""
        w = lin.weight.detach().float()
        q = cls(lin.in_features, lin.out_features, dtype=lin.weight.dtype, device=w.device)
        ws = (w.abs().max() / 448.0).clamp_min(1e-12)
        q.weight.data = (w / ws).clamp(-448, 448).to(torch.float8_e4m3fn)[None]
        q.weight_scale.data = ws.reshape(1).float()
        q.input_scale.data = torch.full((lin.in_features,), float(input_absmax) / 448.0, dtype=torch.float32, device=w.device)
        return q

    def forward(self, input: torch.Tensor) -> torch.Tensor:
        return self.forward_quantized(div_clamp_to(input, self.input_scale))

    def forward_quantized(self, x8: torch.Tensor) -> torch.Tensor:
        """The GEMM alone, on an input that is already div_clamp_to(input, self.input_scale)."""
        x2 = x8 if x8.dim() == 2 else x8.reshape(-1, self.in_features)
        w, scale_a, scale_b = _param(self, "weight"), _param(self, "input_scale").reshape(-1)[:1], _param(self, "weight_scale").reshape(-1)[:1]
        head = 0
        # (a round of 256 CUs: four calls a layer that may wait for the host)
        if x2.shape[0] * self.out_features >= 1 << 24 and x2.is_cuda and not _transformed():
            head = _rows_ahead_e4m3(x2.shape[0], self.out_features, self.in_features, _compute_units(x2.device))
        if head and (type(x2) in _PLAIN and type(w) in _PLAIN and x2.is_contiguous()
                     and not (torch.is_grad_enabled() and any(t.requires_grad for t in (x2, w, scale_a, scale_b)))):
            y = torch.empty((x2.shape[0], self.out_features), dtype=self.output_dtype, device=x2.device)
            for rows in (slice(0, head), slice(head, None)):
                torch._scaled_mm(x2[rows], w[0].t(), scale_a=scale_a, scale_b=scale_b, out_dtype=self.output_dtype, out=y[rows])
        else:
            y = torch._scaled_mm(x2, w[0].t(), scale_a=scale_a, scale_b=scale_b, out_dtype=self.output_dtype)
        return y if x2 is x8 else y.reshape(x8.shape[:-1] + (self.out_features,))


class CustomLayerNormLinear(torch.nn.Module):
    """Input LayerNorm + the four projections q, qx, k, v (dit_module.py:390-425).

    fp8_quant=True builds the four projections as PerTensorQuantizedFp8Linear, as the reference does for every
    layer but the first and the last under EngineConfig.fp8_quant (:405-409): each quantises the normalised input
    with its own input scale and runs the library's fp8 GEMM; there is no shared weight buffer then.

    The four weights keep the reference's parameter names (q.weight, qx.weight, k.weight, v.weight) but live
    side by side in ONE buffer, rows ordered [q | k | v | qx], so forward_qkvx() is a single GEMM over the
    normalised input instead of four (the input, 1 GB at the 720p shape, is read once, and the fused prologue
    takes q / k / v as row-strided views of the one result).  Loading a state dict copies into the shared buffer
    in place; after anything that re-allocates the parameters (.to(), .bfloat16()) the buffer is rebuilt on the
    next call."""

    def __init__(self, input_size: int, output_size_q: int, output_size_kv: int, eps: float = 1e-6,
                 dtype=torch.bfloat16, device=None, fp8_quant: bool = False):
        super().__init__()
        self.fp8_quant = bool(fp8_quant)
        self.layer_norm = torch.nn.LayerNorm(input_size, eps=eps, dtype=dtype, device=device)
        mk = (lambda n: PerTensorQuantizedFp8Linear(input_size, n, dtype=dtype, device=device)) if self.fp8_quant else \
            (lambda n: torch.nn.Linear(input_size, n, bias=False, dtype=dtype, device=device))
        self.q, self.qx, self.k, self.v = mk(output_size_q), mk(output_size_q), mk(output_size_kv), mk(output_size_kv)
        if not self.fp8_quant:
            self._fuse_weights()

    def _projections(self):
        m = self._modules
        return m["q"], m["k"], m["v"], m["qx"]  # row order of the shared buffer

    def _fuse_weights(self) -> torch.Tensor:
        """Move the four weights into one [2*out_q + 2*out_kv, in] buffer and make each parameter a view of it."""
        ws = [m.weight.data for m in self._projections()]
        fused = torch.cat(ws, dim=0)
        row = 0
        for m, w in zip(self._projections(), ws):
            m.weight.data = fused[row:row + w.shape[0]]
            row += w.shape[0]
        return fused

    def _fused_rows(self) -> Tuple[torch.Tensor, int]:
        """(the first parameter of the shared buffer, the rows of all four), 0 rows where they do not share one."""
        base, ptr, rows = None, 0, 0
        for m in self._projections():
            w = _param(m, "weight")
            if base is None:
                base, ptr = w, w.data_ptr()
                row_bytes = w.shape[1] * w.element_size()
            if w.data_ptr() != ptr or w.dtype is not base.dtype or not w.is_contiguous():
                return base, 0
            n = w.shape[0]
            ptr += n * row_bytes
            rows += n
        # back to back, and all of it inside the first one's allocation
        if base.untyped_storage().nbytes() - base.storage_offset() * base.element_size() < rows * row_bytes:
            return base, 0
        return base, rows

    def fused_weight(self) -> torch.Tensor:
        """The [q | k | v | qx] weight as one tensor (rebuilt first if the parameters no longer share a buffer)."""
        base, rows = self._fused_rows()
        if rows == 0:
            return self._fuse_weights()
        return base.data.as_strided((rows, base.shape[1]), (base.shape[1], 1))

    def forward_qkvx(self, hidden_states):
        """One GEMM for all four projections of the (already normalised) input -> views (q, k, v, qx) of one
        [..., 2*out_q + 2*out_kv] result.  (fp8_quant: four quantise + fp8 GEMM pairs, each with its own scales.)"""
        if self.fp8_quant:
            return tuple(m(hidden_states) for m in self._projections())
        return self._split(torch.nn.functional.linear(hidden_states, self.fused_weight()))

    def _split(self, y: torch.Tensor):
        oq, okv = _param(self.q, "weight").shape[0], _param(self.k, "weight").shape[0]
        return y.split((oq, okv, okv, oq), dim=-1)

    def _takes_e4m3(self, m, cols: int) -> bool:
        """Whether the fused norm may hand m its quantised input: m is the fp8 linear itself (another class has its own
        attributes and its own idea of the input), nothing watches or replaces its call, and its input_scale is as
        layer_norm_div_clamp takes it."""
        if type(m) is not PerTensorQuantizedFp8Linear or not _OWN_FP8_LINEAR.of(m):
            return False
        if m._forward_hooks or m._forward_pre_hooks or _global_hooks():
            return False
        s, w = m.input_scale, self.layer_norm.weight
        return s.shape == (cols,) and s.dtype == torch.float32 and s.is_contiguous() and s.device == w.device

    def forward_ln_qkvx_rows(self, hidden_states):
        """forward_qkvx(forward_ln(hidden_states)) as [tokens, out] rows.  With fp8_quant the norm and the four input
        quantisers are one launch that writes the e4m3 inputs of the four GEMMs only (layer_norm_div_clamp)."""
        cols = hidden_states.shape[-1]
        if self.fp8_quant:
            linears = self._projections()
            if cols % 8 == 0 and cols <= 8192 and hidden_states.is_contiguous() and all(self._takes_e4m3(m, cols) for m in linears):
                ln = self.layer_norm
                x2 = hidden_states.view(-1, cols)
                # (a tensor each, given back behind its GEMM: together they would take more memory than the norm's bf16
                # rows and one e4m3 input at a time)
                x8 = [torch.empty_like(x2, dtype=torch.float8_e4m3fn) for _ in linears]
                layer_norm_div_clamp(x2, ln.weight.detach(), ln.bias.detach(), [m.input_scale.detach() for m in linears], ln.eps, out=x8)
                return tuple([m.forward_quantized(x8.pop(0)) for m in linears])
            x = self.forward_ln(hidden_states).view(-1, cols)
            return tuple(m(x) for m in linears)
        return self._split(_linear_in_whole_rounds(self.forward_ln(hidden_states).view(-1, cols), self.fused_weight()))

    def forward_ln(self, hidden_states):
        """LayerNorm of the layer input (dit_module.py:412-413) as one HIP launch; the parameters stay on the
        torch.nn.LayerNorm sub-module under the reference's names."""
        ln = self._modules["layer_norm"]
        return layer_norm(hidden_states, _param(ln, "weight"), _param(ln, "bias"), ln.eps)

    def forward_q(self, hidden_states):
        return self.q(hidden_states)

    def forward_qx(self, hidden_states):
        return self.qx(hidden_states)

    def forward_k(self, hidden_states):
        return self.k(hidden_states)

    def forward_v(self, hidden_states):
        return self.v(hidden_states)


class FullyParallelAttention(torch.nn.Module):
    def __init__(self, hidden_size: int, num_attention_heads: int, num_query_groups: int, kv_channels: int = 128,
                 layer_number: int = 0, layernorm_epsilon: float = 1e-6, apply_layernorm_1p: bool = True,
                 xattn_cond_hidden_ratio: float = 1.0, params_dtype=torch.bfloat16, device=None,
                 attention_dtype: str = "bf16", fp8_fast_exp2: bool = False, fused_projection: bool = False,
                 fp8_quant: bool = False):
        """attention_dtype "fp8" (not in the reference, which has no fp8 attention) runs the self-attention on
        e4m3 operands with per-(video chunk, head) power-of-two scales and keeps the KV cache in that form
        (Fp8KVCache); the cross attention and everything else stay in bf16.
        fp8_fast_exp2: False (default) = the exact exponential, "softmax in fp32"; True opts into the fp8 kernel's
        piecewise-linear exp2 (MAGI_ATTN_FP8_FAST_EXP2: about 15 % faster, probabilities up to 6.2 % off each, the
        output inside a looser accuracy bar; see include/magi_attn.h).
        fp8_quant: the q / qx / k / v projections as PerTensorQuantizedFp8Linear (the reference's fp8_quant layers).
        fused_projection: run the four projections and the prologue as ONE launch (magi_qkv_proj_prologue, the
        hand-written GEMM whose epilogue is the prologue) instead of a library GEMM followed by the prologue kernel;
        bf16 attention at batch 1 only.  Off by default: at the 720p shape the library GEMM + prologue take
        10.9 ms, the fused launch 14.9 ms."""
        super().__init__()
        if kv_channels != 128:
            raise NotImplementedError("head_dim 128 only")
        if attention_dtype not in ("bf16", "fp8"):
            raise ValueError("attention_dtype must be 'bf16' or 'fp8'")
        self.attention_dtype = attention_dtype
        self.fp8_fast_exp2 = bool(fp8_fast_exp2)
        self.fused_projection = bool(fused_projection) and not fp8_quant
        # When the bound that follows from the norm parameters exceeds MAGI_SCORE_BOUND_MAX (it takes the largest gain
        # on both sides for every element), the core attention has the library MEASURE max|q| max|k| on the actual
        # rows (MAGI_ATTN_AUTO_BOUND), which is far smaller for gains that vary across features.  None: where the two
        # passes are small beside the attention; True / False: always / never.
        self.measure_bound_above_limit: Optional[bool] = None
        # forward() has the prologue fold softmax_scale * log2(e) into q ahead of q's one rounding to bf16 and tells
        # the attention kernel so (no per-score multiply there); get_q / get_qkv return q unscaled, as the reference
        self._q_premul = kv_channels ** -0.5 * math.log2(math.e)
        self.layer_number = layer_number
        self.hidden_size_per_attention_head = kv_channels
        self.num_attention_heads = num_attention_heads
        self.num_query_groups_per_partition = num_query_groups
        self.query_projection_size = kv_channels * num_attention_heads
        self.kv_projection_size = kv_channels * num_query_groups
        self.eps = layernorm_epsilon
        self.linear_qkv = CustomLayerNormLinear(hidden_size, self.query_projection_size, self.kv_projection_size,
                                                eps=layernorm_epsilon, dtype=params_dtype, device=device, fp8_quant=fp8_quant)
        self.linear_kv_xattn = torch.nn.Linear(int(hidden_size * xattn_cond_hidden_ratio), 2 * self.kv_projection_size,
                                               bias=False, dtype=params_dtype, device=device)
        mk = lambda dt: FusedLayerNorm(kv_channels, layernorm_epsilon, apply_layernorm_1p, dtype=dt, device=device)
        # the self-attention norms run in fp32 in the reference (promoted after load,
        # inference/model/dit/dit_model.py:628-633); the cross-attention norms stay in bf16
        self.q_layernorm = mk(torch.float32)
        self.k_layernorm = mk(torch.float32)
        self.q_layernorm_xattn = mk(params_dtype)
        self.k_layernorm_xattn = mk(params_dtype)

    # ------------------------------------------------------------------ score bounds
    def score_bounds(self, rotary_half: int = 48) -> Tuple[float, float]:
        """(self attention, cross attention) upper bounds of |q . k| in exp2-exponent units (q carrying
        softmax_scale * log2(e)), from the norm parameters (qk_score_bound: QK-normed rows have a known length, and
        the rotary embedding of 2 * rotary_half features preserves it), plus 1 % for the roundings to bf16.  Within
        MAGI_SCORE_BOUND_MAX the attention kernels then need no running maximum (magi_attn_args.score_bound);
        larger values make them fall back to it.  Computed once per set of parameter values (it reads them on the
        host) and cached until a parameter is modified or replaced (see invalidate_cached_parameters)."""
        m = self._modules
        lns = (m["q_layernorm"], m["k_layernorm"], m["q_layernorm_xattn"], m["k_layernorm_xattn"])
        key = (lns[0].parameter_epoch(), lns[1].parameter_epoch(), lns[2].parameter_epoch(), lns[3].parameter_epoch())
        state = self.__dict__
        if state.get("_bounds_key") != key:
            self._bounds, self._bounds_key = {}, key
        bounds = state["_bounds"]
        r = int(rotary_half)
        if r not in bounds:  # (the cross-attention half does not depend on r)
            cross = next(iter(bounds.values()))[1] if bounds else 1.01 * self._q_premul * qk_score_bound(lns[2], lns[3], 0)
            bounds[r] = (1.01 * self._q_premul * qk_score_bound(lns[0], lns[1], r), cross)
        return bounds[r]

    def invalidate_cached_parameters(self) -> None:
        """Forget everything derived from the norm parameters (their fp32 forms, the score bounds, the e4m3 operand
        scales).  Needed only after a parameter was written through `.data`, which advances no version counter;
        in-place writes (`copy_`, `load_state_dict`) and replaced parameters (`load_state_dict(assign=True)`, `.to()`)
        are noticed by themselves."""
        for ln in (self.q_layernorm, self.k_layernorm, self.q_layernorm_xattn, self.k_layernorm_xattn):
            ln.invalidate_cached_parameters()
        self._bounds_key = self._fp8_scales_key = None

    # ------------------------------------------------------------------ cache
    def _allocate_key_and_value_memory(self, sequence_length: int, batch_size: int, dtype) -> torch.Tensor:
        """[max_seq * max_bs, Hkv, 2D] in HBM (dit_module.py:800-819).  The pinned-host variant is not made here: a
        KVCacheArena(kv_offload=True) attached to the InferenceParams supplies it for all layers."""
        return torch.empty(sequence_length * batch_size, self.num_query_groups_per_partition,
                           2 * self.hidden_size_per_attention_head, dtype=dtype,
                           device=self.linear_qkv.q.weight.device)

    def _cache(self, inference_params: InferenceParams, dtype) -> torch.Tensor:
        d = inference_params.key_value_memory_dict
        if self.layer_number not in d:
            d[self.layer_number] = self._allocate_key_and_value_memory(
                inference_params.max_sequence_length, inference_params.max_batch_size, dtype)
        return d[self.layer_number]

    def _cache_fp8(self, inference_params: InferenceParams, chunk_tokens: int) -> Fp8KVCache:
        d = inference_params.key_value_memory_dict
        if self.layer_number not in d:
            d[self.layer_number] = Fp8KVCache(inference_params.max_sequence_length * inference_params.max_batch_size,
                                              self.num_query_groups_per_partition, chunk_tokens,
                                              self.hidden_size_per_attention_head,
                                              device=self.linear_qkv.q.weight.device)
        cache = d[self.layer_number]
        if not isinstance(cache, Fp8KVCache) or cache.chunk_tokens != chunk_tokens:
            raise ValueError("this layer's cache entry is not an Fp8KVCache with chunk_tokens == clip_token_nums")
        return cache

    def fp8_operand_scales(self) -> Tuple[float, float]:
        """Constant power-of-two scales for the e4m3 forms of q (carrying softmax_scale * log2(e)) and k: no
        element of a QK-normed row can exceed the row's length, which the norm parameters bound
        (FusedLayerNorm.output_norm_bound) and the rotary embedding preserves, so these scales never saturate and
        the prologue can quantise without an absmax pass.  Cached like score_bounds()."""
        lns = (self.q_layernorm, self.k_layernorm)
        key = tuple(ln.parameter_epoch() for ln in lns)
        if getattr(self, "_fp8_scales_key", None) != key:
            nq, nk = (ln.output_norm_bound() for ln in lns)
            self._fp8_scales = (pow2_scale_for(self._q_premul * nq), pow2_scale_for(nk))
            self._fp8_scales_key = key
        return self._fp8_scales

    def _const_scale_table(self, value: float, rows: int, heads: int, device) -> torch.Tensor:
        """[rows, heads] fp32 filled with `value`, kept between calls (a launch only when it has to grow)."""
        tabs = self.__dict__.setdefault("_const_tabs", {})
        key = (value, heads, str(device))
        t = tabs.get(key)
        if t is None or t.shape[0] < rows:
            if len(tabs) > 8:
                tabs.clear()
            t = torch.full((max(rows, 16), heads), value, dtype=torch.float32, device=device)
            tabs[key] = t
        return t[:rows]

    def _side_buffer(self, name: str, shape, dtype, device) -> torch.Tensor:
        """A per-layer buffer for rows that must not be persisted, kept between calls."""
        t = getattr(self, name, None)
        if t is None or t.shape[0] < shape[0] or t.shape[1:] != tuple(shape[1:]) or t.dtype != dtype or t.device != device:
            t = torch.empty(shape, dtype=dtype, device=device)
            setattr(self, name, t)
        return t[:shape[0]]

    def _core_attention_fp8(self, raw, rope: torch.Tensor, inference_params: Optional[InferenceParams],
                            meta_args: ModelMetaArgs, use_cache: bool, out: Optional[torch.Tensor], held: Optional[list] = None) -> torch.Tensor:
        """Self-attention on e4m3 operands, three launches from the raw projections (q_raw, k_raw, v_raw) on: the
        prologue writes q and k as e4m3 with the constant scales of fp8_operand_scales(), k straight into the
        cache rows, and leaves the largest magnitude of each row of v; one quantiser launch takes v's per-(chunk, head) absmax
        scales from those and writes v; the attention.
        Scale chunks are video chunks (clip_token_nums tokens), so the cache rules of the bf16 path
        (dit_module.py:905-931: append at slice_point, keep nothing when update_kv_cache is False, keep all but
        the last chunk under distill_nearly_clean_chunk) carry over chunk by chunk."""
        D = self.hidden_size_per_attention_head
        Hq, Hkv = self.num_attention_heads, self.num_query_groups_per_partition
        Lc = meta_args.clip_token_nums
        p = meta_args.core_attn_params
        q_raw, k_raw, v_raw = raw  # [S, n]
        S = q_raw.shape[0]
        dev = q_raw.device
        n_chunks = (S + Lc - 1) // Lc
        v3 = v_raw.view(S, Hkv, D)
        qs_c, ks_c = self.fp8_operand_scales()
        gq, bq = self.q_layernorm.gamma_beta_fp32()
        gk, bk = self.k_layernorm.gamma_beta_fp32()
        pro = dict(Hq=Hq, Hkv=Hkv, q_scale=qs_c, k_scale=ks_c, eps=self.eps, q_premul=self._q_premul)
        # The largest magnitudes of v's rows, from the prologue to the quantiser.  Not in chunks that a workgroup of the quantiser has in
        # flight as a whole or nearly (400 rows 9.3 -> 7.3 us, 200 rows 7.1 -> 7.5), nor below 256 rows per CU (of all heads), where the two launches
        # gain 2 to 7 us together and layers with e4m3 products wait for the host, which pays 3 (1536 rows x 24 heads 264 / 270).
        row_max = torch.empty((Hkv, S), dtype=torch.int16, device=dev) if min(Lc, S) > 256 and S * Hq >= 256 * _compute_units(dev) else None
        if row_max is not None:
            pro.update(v_raw=v_raw, v_row_max=row_max)
        kw = dict(q_scale=self._const_scale_table(qs_c, n_chunks, Hq, dev), scale_chunk_tokens=Lc,
                  fp8_pow2_prescaled=True, fp8_fast_exp2=self.fp8_fast_exp2, out=out, return_lse=False, held=held)
        f8 = torch.float8_e4m3fn
        if not use_cache:
            q8, k8, _ = qk_prologue_fp8(q_raw, k_raw, rope, gq, bq, gk, bk, **pro)
            v8 = torch.empty((S, Hkv, D), dtype=f8, device=dev)
            vs = torch.empty((n_chunks, Hkv), dtype=torch.float32, device=dev)
            quantize_fp8_split(v3, Lc, S, v8, vs, None, None, pow2_scales=True, row_max=row_max)
            o, _ = range_attention(q8, k8, v8, p.q_range, p.k_range, p.max_seqlen_q, p.max_seqlen_k,
                                   k_scale=self._const_scale_table(ks_c, n_chunks, Hkv, dev), v_scale=vs, **kw)
            return o
        cache = self._cache_fp8(inference_params, Lc)
        start = meta_args.slice_point * Lc
        if inference_params.update_kv_cache:
            n_keep = S - Lc if meta_args.distill_nearly_clean_chunk else S
        else:
            n_keep = 0
        if S % Lc or n_keep < 0:
            raise ValueError("the fp8 path works on whole video chunks")
        if start + n_keep > cache.max_sequence_length:
            raise ValueError("KV cache overflow")
        c0 = start // Lc
        n_side = S - n_keep
        k_side = v_side = vs_side = None
        if n_side:
            k_side = self._side_buffer("_k8_side", (n_side, Hkv, D), f8, dev)
            v_side = self._side_buffer("_v8_side", (n_side, Hkv, D), f8, dev)
            vs_side = self._side_buffer("_v8_side_scale", (n_side // Lc, Hkv), torch.float32, dev)
        if n_keep:
            cache.note_constant_k_scale(ks_c, c0, n_keep // Lc)
        q8, _, _ = qk_prologue_fp8(q_raw, k_raw, rope, gq, bq, gk, bk, k_out=cache.k[start:], n_cache_rows=n_keep,
                                   k_tail=k_side, **pro)
        quantize_fp8_split(v3, Lc, n_keep, cache.v[start:], cache.v_scale[c0:], v_side, vs_side, pow2_scales=True, row_max=row_max)
        split = start + n_keep
        if not n_side:
            o, _ = range_attention(q8, cache.k[:split], cache.v[:split], p.q_range, p.k_range, p.max_seqlen_q,
                                   p.max_seqlen_k, k_scale=cache.k_scale, v_scale=cache.v_scale, **kw)
            return o
        # rows that must not be persisted: side buffers behind the cached prefix, with scale tables of their own
        o, _ = range_attention(q8, cache.k[:split], cache.v[:split], p.q_range, p.k_range, p.max_seqlen_q, p.max_seqlen_k,
                               k2=k_side, v2=v_side, k_split=split, k_scale=cache.k_scale, v_scale=cache.v_scale,
                               k2_scale=self._const_scale_table(ks_c, n_side // Lc, Hkv, dev), v2_scale=vs_side, **kw)
        return o

    # --------------------------------------------------- reference-shaped pieces
    def _prologue_single(self, raw: torch.Tensor, which: str, cos_emb, sin_emb) -> torch.Tensor:
        """raw [sq, b, H*D] -> [(sq b), H, D] through the fused kernel (one of q / k)."""
        sq, b = raw.shape[0], raw.shape[1]
        D = self.hidden_size_per_attention_head
        flat = raw.reshape(sq * b, -1)
        H = flat.shape[1] // D
        rope = torch.cat([sin_emb, cos_emb], dim=-1).float().contiguous()
        ln = self.q_layernorm if which == "q" else self.k_layernorm
        g, be = ln.gamma_beta_fp32()
        if which == "q":
            q, _, _ = qk_prologue(flat, flat[:, :0], flat[:, :0], rope, g, be, None, None, Hq=H, Hkv=0, eps=self.eps,
                                  batch=b)
            return q
        # K alone: run it through the Q slot (same arithmetic, contiguous output)
        k, _, _ = qk_prologue(flat, flat[:, :0], flat[:, :0], rope, g, be, None, None, Hq=H, Hkv=0, eps=self.eps,
                              batch=b)
        return k

    def get_q(self, mixed_qqkv: torch.Tensor, cos_emb: torch.Tensor, sin_emb: torch.Tensor) -> torch.Tensor:
        """[sq, b, h] -> [(sq b), Hq, D]; dit_module.py:953-963."""
        return self._prologue_single(self.linear_qkv.forward_q(mixed_qqkv), "q", cos_emb, sin_emb)

    def get_k(self, mixed_qqkv: torch.Tensor, cos_emb: torch.Tensor, sin_emb: torch.Tensor) -> torch.Tensor:
        """dit_module.py:970-980."""
        return self._prologue_single(self.linear_qkv.forward_k(mixed_qqkv), "k", cos_emb, sin_emb)

    def get_v(self, mixed_qqkv: torch.Tensor) -> torch.Tensor:
        """dit_module.py:987-989."""
        v = self.linear_qkv.forward_v(mixed_qqkv)
        return v.reshape(v.shape[0] * v.shape[1], -1, self.hidden_size_per_attention_head)

    def get_kv(self, mixed_qqkv: torch.Tensor, cos_emb: torch.Tensor, sin_emb: torch.Tensor) -> torch.Tensor:
        """[(sq b), Hkv, 2D] with K | V interleaved per head; dit_module.py:991-996."""
        _, kv = self._fused_qkv(mixed_qqkv, cos_emb, sin_emb, want_q=False)
        return kv

    def get_qkv(self, mixed_qqkv, cos_emb, sin_emb):
        """dit_module.py:998-1003."""
        q, kv = self._fused_qkv(mixed_qqkv, cos_emb, sin_emb, want_q=True)
        D = self.hidden_size_per_attention_head
        return q, kv[..., :D].contiguous(), kv[..., D:].contiguous()

    def _fused_qkv(self, mixed_qqkv, cos_emb, sin_emb, want_q=True, kv_out=None, n_cache_rows=None, kv_tail=None,
                   raw=None, q_premul=1.0, rope=None):
        """raw: (q_raw, k_raw, v_raw) already projected ([sq, b, n] or [sq * b, n] views), else projected here.
        q_premul: factor folded into q ahead of its rounding to bf16 (see qk_prologue).
        rope: the [S, 2*R2] sin | cos table when the caller has it in one piece (else built from the two halves)."""
        sq, b = mixed_qqkv.shape[0], mixed_qqkv.shape[1]
        S = sq * b
        Hq, Hkv = self.num_attention_heads, self.num_query_groups_per_partition
        if raw is not None:
            q_raw, k_raw, v_raw = (t if t.dim() == 2 else t.reshape(S, -1) for t in raw)  # [sq, b, n] row-strided: still a view
        else:
            k_raw = self.linear_qkv.forward_k(mixed_qqkv).reshape(S, -1)
            v_raw = self.linear_qkv.forward_v(mixed_qqkv).reshape(S, -1)
            if want_q:
                q_raw = self.linear_qkv.forward_q(mixed_qqkv).reshape(S, -1)
            else:
                q_raw = k_raw[:, :0]
        if rope is None:
            rope = torch.cat([sin_emb, cos_emb], dim=-1).float().contiguous()
        gq, bq = self._modules["q_layernorm"].gamma_beta_fp32()
        gk, bk = self._modules["k_layernorm"].gamma_beta_fp32()
        q, kv, tail = qk_prologue(q_raw, k_raw, v_raw, rope, gq, bq, gk, bk, Hq=Hq if want_q else 0, Hkv=Hkv,
                                  eps=self.eps, kv_out=kv_out, n_cache_rows=n_cache_rows, kv_tail=kv_tail, batch=b,
                                  q_premul=q_premul)
        return (q if want_q else None), (kv if tail is None else (kv, tail))

    def get_xqkv(self, mixed_qqkv: torch.Tensor, key_value_states: torch.Tensor, qx_raw: Optional[torch.Tensor] = None):
        """Cross-attention q (normed) and k (normed) / v from the text states; dit_module.py:1005-1021.
        qx_raw: the qx projection when the caller already has it (forward_qkvx), else projected here."""
        D = self.hidden_size_per_attention_head
        qx = self.linear_qkv.forward_qx(mixed_qqkv) if qx_raw is None else qx_raw  # [sq, b, Hq*D]
        qx = qx.transpose(0, 1).reshape(qx.shape[0] * qx.shape[1], -1, D)  # "(b sq) hn hd"
        gq, bq = self.q_layernorm_xattn.gamma_beta_fp32()
        qx = head_norm(qx, gq, bq, self.eps)
        kv = torch.nn.functional.linear(key_value_states, self.linear_kv_xattn.weight)  # [Ty, 2*Hkv*D]
        kv = kv.view(key_value_states.shape[0], -1, 2 * D)
        gk, bk = self.k_layernorm_xattn.gamma_beta_fp32()
        kx = head_norm(kv[..., :D], gk, bk, self.eps)  # strided read, contiguous result
        return qx, kx, kv[..., D:]

    def _full_adjust_key_and_value(self, inference_params: InferenceParams, key_and_value: torch.Tensor,
                                   meta_args: ModelMetaArgs) -> torch.Tensor:
        """Appends key_and_value's persistent rows to this layer's cache and returns [cached prefix | key_and_value]
        (dit_module.py:891-931).  With an offloaded cache the prefix comes through the staging buffer and the appended
        rows go back to the host."""
        cache = self._cache(inference_params, key_and_value.dtype)
        start = meta_args.slice_point * meta_args.clip_token_nums * inference_params.max_batch_size
        offloaded = cache if isinstance(cache, OffloadedKVCache) else None
        if offloaded is not None:
            cache = offloaded.stage(start)
        clip = 0
        try:
            prefix = cache[:start]
            if inference_params.update_kv_cache:
                total = key_and_value.size(0)
                clip = (total - meta_args.clip_token_nums * inference_params.max_batch_size
                        if meta_args.distill_nearly_clean_chunk else total)
                if start + clip > cache.shape[0]:
                    clip = 0
                    raise ValueError("KV cache overflow")
                cache[start:start + clip] = key_and_value[:clip]
            return torch.cat([prefix, key_and_value], dim=0)
        finally:
            if offloaded is not None:
                offloaded.release(start, clip)

    def adjust_key_and_value_for_inference(self, key_and_value: torch.Tensor, inference_params: Optional[InferenceParams],
                                           meta_args: ModelMetaArgs):
        """Copying form with the reference's exact semantics (dit_module.py:933-946), for callers
        that hold a materialised key_and_value.  forward() does not use it: it appends in place."""
        D = self.hidden_size_per_attention_head
        if inference_params is None:
            return key_and_value[..., :D], key_and_value[..., D:]
        if meta_args.extract_prefix_video_feature or meta_args.fwd_extra_1st_chunk or meta_args.slice_point > 0:
            key_and_value = self._full_adjust_key_and_value(inference_params, key_and_value, meta_args)
        return key_and_value[..., :D].contiguous(), key_and_value[..., D:].contiguous()

    def core_attention(self, query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, bs: int,
                       meta_args: ModelMetaArgs, out: Optional[torch.Tensor] = None,
                       q_prescaled: bool = False, score_bound: float = 0.0, auto_bound: bool = False,
                       split_keys: bool = False, held: Optional[list] = None) -> torch.Tensor:
        """query [(sq b), Hq, D], key / value [(sk b), Hkv, D] -> [(sq b), Hq, D]; dit_module.py:1023-1066.
        bs > 1 only occurs with one range per batch row (asserted there too).  `out` is a
        destination view, possibly in the grouped layout of range_attention (bs > 1: [sq, bs * groups, heads, D]).  q_prescaled: query carries
        softmax_scale * log2(e); score_bound, auto_bound: see range_attention.  split_keys: whether the keys of a row may
        be shared among workgroups and wavefronts, the sums added in an order that depends on what else the launch holds; without it a
        row's bits are those of full_attention on its range alone (with auto_bound, where the measured bound does not hold).  held (bs 1):
        see range_attention."""
        p = meta_args.core_attn_params
        if bs == 1:
            out, _ = range_attention(query, key, value, p.q_range, p.k_range, p.max_seqlen_q, p.max_seqlen_k,
                                     out=out, return_lse=False, q_prescaled=q_prescaled, score_bound=score_bound,
                                     auto_bound=auto_bound, split_keys=split_keys, share_waves=split_keys, held=held)
            return out
        if meta_args.denoising_range_num > 1:
            raise ValueError("bs > 1 with several denoising ranges is not a layout the pipeline produces")
        # Batch rows attend to themselves over the whole sequence (dit_module.py:1046-1050): with the token axis
        # ordered (position, batch) that is ONE range over positions with bs * Hq heads, since head b * Hq + h of
        # the [(sq), (b Hq), D] view uses kv head (b * Hq + h) / (Hq / Hkv) = b * Hkv + h / (Hq / Hkv).
        sq, sk = query.shape[0] // bs, key.shape[0] // bs
        Hq, Hkv, D = query.shape[1], key.shape[1], query.shape[2]
        if not (query.is_contiguous() and key.stride(0) == Hkv * key.stride(1) and value.stride(0) == Hkv * value.stride(1)):
            raise ValueError("bs > 1 needs the (position, batch, head) axes of q / k / v evenly strided")
        dev = query.device
        ranges = getattr(self, "_one_range", None)
        if ranges is None or ranges[0] != (sq, sk, dev):
            ranges = ((sq, sk, dev), torch.tensor([[0, sq]], dtype=torch.int32, device=dev),
                      torch.tensor([[0, sk]], dtype=torch.int32, device=dev))
            self._one_range = ranges
        o, _ = range_attention(query.view(sq, bs * Hq, D), key.as_strided((sk, bs * Hkv, D), (bs * key.stride(0), key.stride(1), 1)),
                               value.as_strided((sk, bs * Hkv, D), (bs * value.stride(0), value.stride(1), 1)),
                               ranges[1], ranges[2], sq, sk, return_lse=False, q_prescaled=q_prescaled,
                               score_bound=score_bound, split_keys=split_keys, out=out)
        return o if out is not None else o.view(sq * bs, Hq, D)

    def full_attention(self, bs: int, meta_args: ModelMetaArgs, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, i: int,
                       score_bound: float = 0.0) -> torch.Tensor:
        """The rectangle of denoising range i alone: q [rows of range i, Hq, D] against the keys k_range[i] of the
        whole key axis k / v [(sk), Hkv, D] -> [rows, Hq, D]; dit_module.py:1068-1096 (what the reference's
        cp_shuffle_overlap strategy calls chunk by chunk, batch 1 only as there).  The range tensors are sliced on the
        device, so the call does not synchronise."""
        if bs != 1:
            raise ValueError("full_attention is defined for batch 1 (as in the reference)")
        p = meta_args.core_attn_params
        q_range = (p.q_range[i:i + 1] - p.q_range[i, 0]).contiguous()
        out, _ = range_attention(q, k, v, q_range, p.k_range[i:i + 1].contiguous(), p.max_seqlen_q, p.max_seqlen_k,
                                 return_lse=False, score_bound=score_bound, split_keys=False)
        return out

    def cross_attention(self, mixed_qqkv: torch.Tensor, key_value_states: torch.Tensor,
                        cross_attn_params: PackedCrossAttnParams, get_xqkv_func: Callable,
                        out: Optional[torch.Tensor] = None) -> torch.Tensor:
        """-> [sq, b, Hq*D]; dit_module.py:1098-1136.  With `out` (b == 1 only: a destination view, possibly in
        the grouped layout of range_attention) the result is written there (segments without text get zero rows
        from the kernel) and `out` is returned."""
        qx, kx, vx = get_xqkv_func(mixed_qqkv, key_value_states)
        b = mixed_qqkv.shape[1]
        sq = mixed_qqkv.shape[0]
        if out is not None:
            if b != 1:
                raise ValueError("a destination view for the cross attention needs batch 1")
            range_attention(qx, kx, vx, cross_attn_params.cu_seqlens_q, cross_attn_params.cu_seqlens_kv,
                            cross_attn_params.max_seqlen_q, cross_attn_params.max_seqlen_kv,
                            ranges_mode=L.MAGI_RANGES_CU, out=out, return_lse=False)
            return out
        out, _ = range_attention(qx, kx, vx, cross_attn_params.cu_seqlens_q, cross_attn_params.cu_seqlens_kv,
                                 cross_attn_params.max_seqlen_q, cross_attn_params.max_seqlen_kv,
                                 ranges_mode=L.MAGI_RANGES_CU, return_lse=False, zero_init=True)
        out = out.view(b, sq, -1)
        return out.transpose(0, 1).contiguous() if b > 1 else out.view(sq, 1, -1)

    def _cross_attention_fused(self, qx_raw: torch.Tensor, sq: int, b: int, key_value_states: torch.Tensor,
                               cross_attn_params: PackedCrossAttnParams, out: Optional[torch.Tensor],
                               bound: float, own_text: bool = False, held: Optional[list] = None) -> Optional[torch.Tensor]:
        """Cross attention on the RAW qx projection [sq * b, Hq*D].  Batch 1: the attention kernel applies q_layernorm_xattn
        while it loads q (no normalised copy of q in memory) and, the scores of normed q and k being bounded, runs without a
        running maximum; returns None when that path does not apply (then the caller takes get_xqkv + cross_attention).
        Batch > 1: head norm and online softmax, the arithmetic of get_xqkv + cross_attention bit for bit, on the [position,
        batch] rows where they are (no copy to batch-major order and back: 230 MB each way at the 480p unconditional pass).
        own_text: the text's K | V rows come from small_projections where it takes the states (else the library's GEMM and a head norm).
        held (batch 1): see range_attention.
        -> [sq, b, Hq, D] contiguous, or `out` (batch > 1: [sq, b, groups, heads, D])."""
        if b == 1 and not (0.0 < bound <= L.MAGI_SCORE_BOUND_MAX):
            return None
        D = self.hidden_size_per_attention_head
        q = qx_raw.view(sq * b, -1, D)  # row-strided view of the projection
        m = self._modules
        text_kv = None
        if own_text:
            w = _param(m["linear_kv_xattn"], "weight")
            if _plain_rows(key_value_states, w, 2 * self.num_query_groups_per_partition):  # (others have as many heads as the weight)
                gk, bk = m["k_layernorm_xattn"].gamma_beta_fp32()
                text_kv = small_projections(None, None, None, None, None, None, None, Hq=0, Hkv=self.num_query_groups_per_partition,
                                            eps=self.eps, text=(key_value_states, w, gk, bk))[4]
        if text_kv is not None:
            kx, v_ = _halves(text_kv, text_kv.shape[0])
        else:
            kv = torch.nn.functional.linear(key_value_states, _param(m["linear_kv_xattn"], "weight"))
            k_, v_ = _halves(kv.view(key_value_states.shape[0], -1, 2 * D), kv.shape[0])
            gk, bk = m["k_layernorm_xattn"].gamma_beta_fp32()
            kx = head_norm(k_, gk, bk, self.eps)
        gq, bq = m["q_layernorm_xattn"].gamma_beta_fp32()
        if b == 1:
            q_kw = {"score_bound": bound, "q_norm": (gq, bq, self.eps), "share_waves": True, "held": held}
        else:
            q = head_norm(q, gq, bq, self.eps).view(sq, b, -1, D).transpose(0, 1)
            q_kw = {"score_bound": math.inf, "clear_out": True}
            out = out if out is None else out.transpose(0, 1)
        o, _ = range_attention(q, kx, v_, cross_attn_params.cu_seqlens_q, cross_attn_params.cu_seqlens_kv,
                               cross_attn_params.max_seqlen_q, cross_attn_params.max_seqlen_kv,
                               ranges_mode=L.MAGI_RANGES_CU, out=out, return_lse=False, zero_init=True, **q_kw)
        return o if b == 1 else o.transpose(0, 1)  # (of a given `out` too)

    def _project_rows(self, hidden_states: torch.Tensor):
        """-> (q, k, v, qx) of the normalised input as [tokens, out] rows, and that input where it exists: with the library's
        own projections only the rows are formed, others have their forward_ln and forward_qkvx called."""
        m = self._modules["linear_qkv"]
        if _OWN_PROJECTIONS.of(m):
            return m.forward_ln_qkvx_rows(hidden_states), None
        x = m.forward_ln(hidden_states)
        return tuple(t.reshape(-1, t.shape[-1]) for t in m.forward_qkvx(x)), x

    def _tail_rows(self, rows: int, cache: torch.Tensor) -> torch.Tensor:
        """Side buffer for the K | V rows that must not be persisted, kept between calls."""
        tail = getattr(self, "_kv_tail", None)
        if (tail is None or tail.shape[0] < rows or tail.shape[1:] != cache.shape[1:] or tail.dtype != cache.dtype
                or tail.device != cache.device):
            tail = torch.empty(rows, cache.shape[1], cache.shape[2], dtype=cache.dtype, device=cache.device)
            self._kv_tail = tail
        return tail[:rows]

    def _norm_parameters(self):
        """gamma_beta_fp32() of the four head norms.  Where they and score_bounds() are the library's own, forward() has just had the
        parameters converted or checked (score_bounds asks each norm for its parameter_epoch)."""
        m = self._modules
        lns = (m["q_layernorm"], m["k_layernorm"], m["q_layernorm_xattn"], m["k_layernorm_xattn"])
        if (type(self).score_bounds is not _SCORE_BOUNDS or "score_bounds" in self.__dict__ or FusedLayerNorm.gamma_beta_fp32 is not _GAMMA_BETA
                or FusedLayerNorm.parameter_epoch is not _PARAMETER_EPOCH):
            return [ln.gamma_beta_fp32() for ln in lns]
        return [d["_gb"] if type(ln) is FusedLayerNorm and "gamma_beta_fp32" not in (d := ln.__dict__) and "parameter_epoch" not in d
                else ln.gamma_beta_fp32() for ln in lns]

    def _small_layer_weights(self, hidden_states: torch.Tensor, key_value_states: torch.Tensor, rope: torch.Tensor, own: "_Own"):
        """(w, wt, ln, lw, lb): the parameter that the weight of the four projections starts with, the text's weight, the input norm and its parameters, of a small layer
        at batch 1 whose projections are the library's own and whose tensors are as magi_small_projections takes them; else None."""
        S, b, K = hidden_states.shape
        if K > 1024 or b != 1 or key_value_states.dim() != 2 or not hidden_states.is_cuda or self.fused_projection:
            return None
        dev = hidden_states.device
        Hq, Hkv, D, (T, Kt) = self.num_attention_heads, self.num_query_groups_per_partition, 128, key_value_states.shape
        if Kt > 1024 or not _projects_in_one_launch(S, 2 * (Hq + Hkv), T, 2 * Hkv, max(K, Kt), _compute_units(dev)):
            return None
        m = self._modules
        lin = m["linear_qkv"]
        if lin.__dict__.get("fp8_quant", True) or not hidden_states.is_contiguous() or rope.shape[-1] % 16 or rope.shape[-1] > D:
            return None
        if not (_OWN_SMALL_PROJECTIONS.of(lin) and own.of(self)):
            return None
        w, rows = lin._fused_rows()
        if rows == 0:
            w = lin._fuse_weights()
            rows = w.shape[0]
        wt, ln = _param(m["linear_kv_xattn"], "weight"), lin._modules["layer_norm"]
        lw, lb = _param(ln, "weight"), _param(ln, "bias")
        if (hidden_states.dtype is not torch.bfloat16 or type(hidden_states) not in _PLAIN or S == 0 or hidden_states.data_ptr() % 16
                or rows != 2 * (Hq + Hkv) * D or not _plain_weight(w, w.shape[0] // D, K, dev) or not _plain_rows(key_value_states, wt, 2 * Hkv)
                or lw is None or lb is None):
            return None
        if _param(lin._modules["q"], "weight").shape[0] != Hq * D or _param(lin._modules["k"], "weight").shape[0] != Hkv * D:
            return None
        if lw.dtype is not lb.dtype or lw.dtype not in (torch.bfloat16, torch.float32) or not (lw.is_contiguous() and lb.is_contiguous()) or (
                lw.shape[0] != K or lb.shape[0] != K or (lw.data_ptr() | lb.data_ptr()) % 16 or lw.device != dev or key_value_states.device != dev):
            return None
        return w, wt, ln, lw, lb

    def _small_layer_outputs(self, S: int, dev: torch.device, proj_layout: bool, core_n: int, core_most: int, cross_n: int, cross_most: int):
        """-> (tensors, address of core's rows, of cross's, row stride, heads per group, group stride, whether rows that no range covers are
        cleared): one tensor in linear_proj's layout or two, as forward() returns them."""
        Hq, D = self.num_attention_heads, 128
        if proj_layout and Hq % PROJ_GROUPS == 0:
            # (rows that no q range / cu_seqlens segment covers are left as allocated: the pipeline's ranges cover
            # every row, dit_model.py:220-222, 246)
            out = torch.empty(S, 1, 2 * Hq * D, dtype=torch.bfloat16, device=dev)
            per = Hq // PROJ_GROUPS
            return (out,), out.data_ptr(), out.data_ptr() + 2 * per * D, 2 * Hq * D, per, 2 * per * D, False
        core, cross = torch.empty(S, 1, Hq * D, dtype=torch.bfloat16, device=dev), torch.empty(S, 1, Hq * D, dtype=torch.bfloat16, device=dev)
        for t, n, most in ((core, core_n, core_most), (cross, cross_n, cross_most)):
            if not covered_by_launch(n, most, S):
                t.zero_()
        return (core, cross), core.data_ptr(), cross.data_ptr(), Hq * D, 0, 0, True

    def _forward_small(self, hidden_states: torch.Tensor, key_value_states: torch.Tensor, inference_params: Optional[InferenceParams],
                       rope: torch.Tensor, meta_args: ModelMetaArgs, proj_layout: bool, bound_core: float, bound_cross: float):
        """forward() of a small bf16 layer at batch 1 with both score bounds in force, whose projections are the library's own:
        magi_small_projections, core attention and cross attention (in one launch where both are small) with their arguments put together in
        one go.  None, before anything is launched or written, where forward() goes on with the separate launches: other methods, projections or caches, larger
        layers, tensors of other types or layouts.  (The layer's cache and its side buffer may have been allocated by then, as forward() would.)

        Such a layer waits for the host: 240 + 45 rows, 20 + 4 heads, 87 us through the callables, 44 this way (49 with three calls into the library).  There
        each launch brings its own checks, allocations and views with it."""
        use_cache = inference_params is not None and (
            meta_args.extract_prefix_video_feature or meta_args.fwd_extra_1st_chunk or meta_args.slice_point > 0)
        parts = self._small_layer_weights(hidden_states, key_value_states, rope, _OWN_SMALL if use_cache else _OWN_SMALL_UNCACHED)
        if parts is None:
            return None
        w, wt, ln, lw, lb = parts
        (S, _, K), dev, m = hidden_states.shape, hidden_states.device, self._modules
        Hq, Hkv, D, (T, Kt) = self.num_attention_heads, self.num_query_groups_per_partition, 128, key_value_states.shape
        cache = tail = offloaded = None
        start = n_keep = persisted = 0
        if use_cache:
            if inference_params.max_batch_size != 1:
                return None
            cache = self._cache(inference_params, hidden_states.dtype)
            if isinstance(cache, OffloadedKVCache):
                offloaded, cache = cache, cache.arena.stages[0]  # (they are all alike; the one in use comes from stage() below)
            if not isinstance(cache, torch.Tensor) or cache.dtype is not torch.bfloat16 or cache.stride()[1:] != (2 * D, 1) or (
                    cache.shape[1:] != (Hkv, 2 * D) or cache.stride(0) % 8 or cache.data_ptr() % 16 or cache.device != dev):
                return None
            start = meta_args.slice_point * meta_args.clip_token_nums
            if inference_params.update_kv_cache:
                n_keep = S - meta_args.clip_token_nums if meta_args.distill_nearly_clean_chunk else S
            if start < 0 or n_keep < 0 or start + n_keep > cache.shape[0]:
                return None  # (forward() refuses it)
            if n_keep < S:
                tail = self._tail_rows(S - n_keep, cache)
                if tail.stride() != cache.stride():
                    return None
        p, cp = meta_args.core_attn_params, meta_args.cross_attn_params
        if rope.dim() != 2 or rope.shape[0] != S:
            raise ValueError("rope must be a contiguous fp32 [S / batch, 2*R2] tensor")
        core_n = range_count(p.q_range, p.k_range, L.MAGI_RANGES_PAIRS)
        cross_n = range_count(cp.cu_seqlens_q, cp.cu_seqlens_kv, L.MAGI_RANGES_CU)
        (gq, bq), (gk, bk), (gx, bx), (gkx, bkx) = self._norm_parameters()
        # one buffer for q, the raw cross-attention q, the text's K | V rows, and K | V without a cache
        ws = torch.empty(D * (2 * Hq * S + 2 * Hkv * (T + (S if cache is None else 0))), dtype=torch.bfloat16, device=dev)
        q = ws.data_ptr()
        qx = q + 2 * D * Hq * S
        text_kv = qx + 2 * D * Hq * S
        row = 2 * D * Hkv  # elements of a K | V row
        side = 0 if tail is None else tail.data_ptr()
        outs, core_out, cross_out, o_row, groups, o_group, clear = self._small_layer_outputs(S, dev, proj_layout, core_n, p.max_seqlen_q, cross_n,
                                                                                             cp.max_seqlen_q)
        if offloaded is not None:  # kv_offload: the prefix comes through a device staging buffer
            cache = offloaded.stage(start)
        try:
            if cache is None:
                kv, kv_row, new, kept, total = text_kv + 2 * row * T, row, text_kv + 2 * row * T, S, S
            else:
                kv, kv_row, kept, total = cache.data_ptr(), cache.stride(0), n_keep, start + S
                new = kv + 2 * kv_row * start
            core_q, core_k, cross_q, cross_k = int(p.max_seqlen_q), int(p.max_seqlen_k), int(cp.max_seqlen_q), int(cp.max_seqlen_kv)
            zero = L.MAGI_ATTN_ZERO_UNCOVERED if clear else 0
            core_split = split_memory(dev, Hq, Hkv, core_n, L.MAGI_RANGES_PAIRS, core_q, core_k)
            cross_split = split_memory(dev, Hq, Hkv, cross_n, L.MAGI_RANGES_CU, cross_q, cross_k)
            ranges = [t.contiguous() for t in (p.q_range, p.k_range, cp.cu_seqlens_q, cp.cu_seqlens_kv)]
            fields = (
                hidden_states.data_ptr(), w.data_ptr(), lw.data_ptr(), lb.data_ptr(), rope.data_ptr(), gq.data_ptr(), bq.data_ptr(), gk.data_ptr(),
                bk.data_ptr(), key_value_states.data_ptr(), wt.data_ptr(), gkx.data_ptr(), bkx.data_ptr(), gx.data_ptr(), bx.data_ptr(),
                key_value_states.stride(0) if T > 1 else Kt, S, K, int(lw.dtype is torch.float32), T, Kt, Hq, Hkv, rope.shape[1] // 2, ln.eps, self.eps,
                self._q_premul, q, qx, text_kv, kv, new, side, kv_row, kept, start + kept, total, groups, o_row, o_group, ranges[0].data_ptr(),
                ranges[1].data_ptr(), core_n, core_q, core_k, zero if covered_by_launch(core_n, core_q, S) else 0, bound_core, core_out, core_split[1],
                core_split[2], ranges[2].data_ptr(), ranges[3].data_ptr(), cross_n, cross_q, cross_k,
                zero if covered_by_launch(cross_n, cross_q, S) else 0, bound_cross, cross_out, cross_split[1], cross_split[2])
            launch_small_projections(dev, 3 if offloaded is None else 1, *fields)
            persisted = n_keep
        finally:
            if offloaded is not None:  # the persisted rows go back to the host behind the attention launch
                offloaded.release(start, persisted)
        if offloaded is not None:
            launch_small_projections(dev, 2, *fields)
        return outs[0] if len(outs) == 1 else attn_linear_proj_input(*outs) if proj_layout else outs

    def _forward_small_fp8(self, hidden_states: torch.Tensor, key_value_states: torch.Tensor, inference_params: Optional[InferenceParams],
                           rope: torch.Tensor, meta_args: ModelMetaArgs, proj_layout: bool, bound_cross: float):
        """_forward_small for e4m3 attention (the text's scores bounded): magi_small_projections_e4m3, the quantiser of V, core attention,
        cross attention.  None where forward() goes on with the separate launches (among others in the extra forward of a first chunk,
        which runs once a video and not once a step), or refuses the call.  240 + 45 rows, 20 + 4
        heads: 153 us through the callables, 66 this way."""
        use_cache = inference_params is not None and (meta_args.extract_prefix_video_feature or meta_args.slice_point > 0)
        parts = None if meta_args.fwd_extra_1st_chunk else self._small_layer_weights(hidden_states, key_value_states, rope, _OWN_SMALL_FP8)
        if parts is None:
            return None
        w, wt, ln, lw, lb = parts
        (S, _, K), dev, m = hidden_states.shape, hidden_states.device, self._modules
        Hq, Hkv, D, (T, Kt) = self.num_attention_heads, self.num_query_groups_per_partition, 128, key_value_states.shape
        Lc, row = meta_args.clip_token_nums, Hkv * D  # bytes of a K or V row
        start = n_keep = 0
        cache = None
        if use_cache:
            if inference_params.max_batch_size != 1 or Lc <= 0:
                return None
            cache = self._cache_fp8(inference_params, Lc)
            start = meta_args.slice_point * Lc
            if inference_params.update_kv_cache:
                n_keep = S - Lc if meta_args.distill_nearly_clean_chunk else S
            if type(cache) is not Fp8KVCache or S % Lc or start < 0 or n_keep < 0 or start + n_keep > cache.max_sequence_length:
                return None
            chunks = (start + n_keep) // Lc
            for t, dtype, heads, rows in ((cache.k, torch.float8_e4m3fn, (Hkv, D), start + n_keep), (cache.v, torch.float8_e4m3fn, (Hkv, D), start + n_keep),
                                          (cache.k_scale, torch.float32, (Hkv,), chunks), (cache.v_scale, torch.float32, (Hkv,), chunks)):
                if (type(t) is not torch.Tensor or t.dtype is not dtype or t.shape[1:] != heads or t.shape[0] < rows or not t.is_contiguous()
                        or t.device != dev or t.data_ptr() % 16):
                    return None
        if Lc <= 0:
            return None
        p, cp = meta_args.core_attn_params, meta_args.cross_attn_params
        if rope.dim() != 2 or rope.shape[0] != S:
            raise ValueError("rope must be a contiguous fp32 [S / batch, 2*R2] tensor")
        core_n = range_count(p.q_range, p.k_range, L.MAGI_RANGES_PAIRS)
        cross_n = range_count(cp.cu_seqlens_q, cp.cu_seqlens_kv, L.MAGI_RANGES_CU)
        q_scale, k_scale = self.fp8_operand_scales()
        (gq, bq), (gk, bk), (gx, bx), (gkx, bkx) = self._norm_parameters()
        n_side = S - n_keep  # rows that must not be persisted (all of them without a cache), in chunks of their own
        side_chunks = (n_side + Lc - 1) // Lc
        # one buffer: raw cross-attention q, v, the text's K | V rows (bf16), the e4m3 q, K and V rows that are not kept and the latter's scales
        sizes = (2 * D * Hq * S, 2 * row * S, 4 * row * T, D * Hq * S, row * n_side, row * n_side, 4 * side_chunks * Hkv)
        at = list(itertools.accumulate(((n + 255) // 256 * 256 for n in sizes), initial=0))
        ws = torch.empty(at[-1], dtype=torch.uint8, device=dev)
        qx, v_raw, text_kv, q8, k_side, v_side, vs_side = (ws.data_ptr() + o for o in at[:-1])
        tables = self._const_scale_table(q_scale, (S + Lc - 1) // Lc, Hq, dev)
        side_ks = self._const_scale_table(k_scale, max(side_chunks, 1), Hkv, dev)
        outs, core_out, cross_out, o_row, groups, o_group, clear = self._small_layer_outputs(S, dev, proj_layout, core_n, p.max_seqlen_q, cross_n,
                                                                                             cp.max_seqlen_q)
        if cache is None:  # everything in the one buffer
            k_new, v_new, vs_new, kept, k_tail, v_tail, vs_tail = k_side, v_side, vs_side, S, 0, 0, 0
            k_all, v_all, scales, split, total = k_side, v_side, (tables.data_ptr(), side_ks.data_ptr(), vs_side, 0, 0), S, S
        else:
            if n_keep:
                cache.note_constant_k_scale(k_scale, start // Lc, n_keep // Lc)
            k_all, v_all = cache.k.data_ptr(), cache.v.data_ptr()
            k_new, v_new, vs_new, kept = k_all + start * row, v_all + start * row, cache.v_scale.data_ptr() + 4 * Hkv * (start // Lc), n_keep
            k_tail, v_tail, vs_tail = (k_side, v_side, vs_side) if n_side else (0, 0, 0)
            scales = (tables.data_ptr(), cache.k_scale.data_ptr(), cache.v_scale.data_ptr()) + ((side_ks.data_ptr(), vs_side) if n_side else (0, 0))
            split, total = start + n_keep, start + S
        launch_small_projections_e4m3(
            dev, q_scale, k_scale, v_raw, hidden_states.data_ptr(), w.data_ptr(), lw.data_ptr(), lb.data_ptr(), K, S, K, int(lw.dtype is torch.float32),
            ln.eps, Hq, Hkv, Hq, rope.shape[1] // 2, rope.data_ptr(), gq.data_ptr(), bq.data_ptr(), gk.data_ptr(), bk.data_ptr(), self.eps, 1,
            self._q_premul, kept, q8, k_new, k_tail, row, row, qx, key_value_states.data_ptr(), wt.data_ptr(),
            key_value_states.stride(0) if T > 1 else Kt, T, Kt, gkx.data_ptr(), bkx.data_ptr(), text_kv)
        launch_quantize_fp8_split(dev, v_raw, row, D, S, Hkv, D, Lc, 1.0, 1, v_new if kept else 0, vs_new if kept else 0, kept, v_tail, vs_tail)
        launch_fp8_attention(dev, q8, S, Hq, k_all, v_all, k_tail, v_tail, split, total, Hkv, scales, Lc, p.q_range, p.k_range, core_n,
                             p.max_seqlen_q, p.max_seqlen_k, core_out, o_row, groups, o_group, clear, self.fp8_fast_exp2)
        launch_text_attention(dev, qx, S, Hq, text_kv, T, Hkv, cp.cu_seqlens_q, cp.cu_seqlens_kv, cross_n, cp.max_seqlen_q, cp.max_seqlen_kv,
                              cross_out, o_row, groups, o_group, clear, bound_cross, gx.data_ptr(), bx.data_ptr(), self.eps)
        return outs[0] if len(outs) == 1 else attn_linear_proj_input(*outs) if proj_layout else outs

    # ------------------------------------------------------------------ forward
    def forward(self, hidden_states: torch.Tensor, key_value_states: torch.Tensor,
                inference_params: Optional[InferenceParams], rotary_pos_emb: torch.Tensor, meta_args: ModelMetaArgs,
                proj_layout: bool = False):
        """-> (core_attn_out, xattn_out), each [sq, b, Hq*D], as the reference (dit_module.py:1138-1173).

        With proj_layout=True the return value is ONE tensor [sq, b, 2*Hq*D] already in the "(hn n hd)" order
        that linear_proj consumes (what attn_linear_proj builds with concat + rearrange, dit_module.py:1332-1340):
        both attention launches write straight into it (of a batch where both are the library's own methods)."""
        if rotary_pos_emb is None:
            raise ValueError("FullyParallelAttention needs rotary_pos_emb")
        # the incoming table already is the [sin | cos] layout the prologue takes
        rope = rotary_pos_emb if (rotary_pos_emb.dtype == torch.float32 and rotary_pos_emb.is_contiguous()) else \
            rotary_pos_emb.float().contiguous()
        bound_core, bound_cross = self.score_bounds(rotary_pos_emb.shape[-1] // 2)
        core_bound_kw = {"score_bound": bound_core}  # (above the limit: the online-softmax kernel, unless measured)
        measured = False
        if not (0.0 < bound_core <= L.MAGI_SCORE_BOUND_MAX) and self.attention_dtype == "bf16" and hidden_states.shape[1] == 1:
            p_ = meta_args.core_attn_params
            n_q = hidden_states.shape[0]
            measured = self.measure_bound_above_limit
            if measured is None:
                shape_q = torch.empty(n_q, self.num_attention_heads, 128, dtype=torch.bfloat16, device="meta")
                shape_k = torch.empty(max(int(p_.max_seqlen_k), n_q), self.num_query_groups_per_partition, 128,
                                      dtype=torch.bfloat16, device="meta")
                measured = _measuring_a_bound_pays(shape_q, shape_k, p_.q_range.shape[0], p_.max_seqlen_q, p_.max_seqlen_k)
            if measured:
                core_bound_kw = {"auto_bound": True}
        bs = hidden_states.shape[1]
        sq = hidden_states.shape[0]
        D = self.hidden_size_per_attention_head
        # which attention kernels this forward selects (diagnostics; the choice follows from the norm parameters)
        core_bounded, cross_bounded = 0.0 < bound_core <= L.MAGI_SCORE_BOUND_MAX, bs == 1 and 0.0 < bound_cross <= L.MAGI_SCORE_BOUND_MAX
        self.__dict__["last_forward_kernels"] = {
            "core": "fp8" if self.attention_dtype == "fp8" else
            ("measured bound: bounded-score or online softmax, chosen on the device" if measured else _KERNEL_NAMES[core_bounded]),
            "core_score_bound": bound_core, "cross": _KERNEL_NAMES[cross_bounded], "cross_score_bound": bound_cross}
        if core_bounded and cross_bounded and self.attention_dtype == "bf16":
            small = self._forward_small(hidden_states, key_value_states, inference_params, rope, meta_args, proj_layout, bound_core, bound_cross)
            if small is not None:
                return small
        if cross_bounded and self.attention_dtype == "fp8":
            small = self._forward_small_fp8(hidden_states, key_value_states, inference_params, rope, meta_args, proj_layout, bound_cross)
            if small is not None:
                return small
        one_launch = (self.fused_projection and self.attention_dtype == "bf16" and bs == 1
                      and rope.shape[-1] == 96 and hidden_states.shape[-1] % 64 == 0)
        if one_launch:
            # projections + prologue in one launch: nothing raw reaches memory (qx leaves unnormalised, as the
            # cross-attention kernel takes it)
            mixed_qqkv = self.linear_qkv.forward_ln(hidden_states)
            raw = qx_raw = None
        else:
            # all four projections in one GEMM; q / k / v feed the fused prologue as row-strided views of its result
            (q_raw, k_raw, v_raw, qx_raw), mixed_qqkv = self._project_rows(hidden_states)
            raw = (q_raw, k_raw, v_raw)
        own_cross = _OWN_CROSS.of(self)
        if mixed_qqkv is None:  # (the library's own methods use its shape only: every projection is in hand)
            mixed_qqkv = hidden_states if own_cross else self.linear_qkv.forward_ln(hidden_states)

        def project(kv_out=None, n_cache_rows=None, kv_tail=None):
            """-> (q [S, Hq, D] carrying the softmax scale, kv destination(s), qx_raw [sq * b, Hq*D])"""
            if not one_launch:
                q_, kv_ = self._fused_qkv(mixed_qqkv, None, None, kv_out=kv_out, n_cache_rows=n_cache_rows,
                                          kv_tail=kv_tail, raw=raw, q_premul=self._q_premul, rope=rope)
                return q_, kv_, qx_raw
            gq_, bq_ = self.q_layernorm.gamma_beta_fp32()
            gk_, bk_ = self.k_layernorm.gamma_beta_fp32()
            q_, kv_, tail_, qx_ = qkv_proj_prologue(
                mixed_qqkv.view(sq, -1), self.linear_qkv.fused_weight(), rope, gq_, bq_, gk_, bk_,
                Hq=self.num_attention_heads, Hkv=self.num_query_groups_per_partition, Hqx=self.num_attention_heads,
                eps=self.eps, kv_out=kv_out, n_cache_rows=n_cache_rows, kv_tail=kv_tail, q_premul=self._q_premul)
            return q_, (kv_ if tail_ is None else (kv_, tail_)), qx_.view(sq, -1)

        def cross_fused(dst):
            if bs > 1 and not own_cross:  # (a replaced cross attention runs; at batch 1 with a bound in force it never did)
                return None
            flop = 512.0 * sq * Hq * (hidden_states.shape[2] + p.max_seqlen_k)
            text_rows, heads = key_value_states.shape[0], 2 * self.num_query_groups_per_partition
            own_text = (bs == 1 and key_value_states.dim() == 2 and hidden_states.is_cuda
                        and "_cross_attention_fused" not in self.__dict__ and type(self)._cross_attention_fused is _CROSS_FUSED
                        and _text_in_one_launch(flop, text_rows, heads, key_value_states.shape[1], _compute_units(hidden_states.device)))
            more = {"own_text": True} if own_text else {}  # (one put in its place may not know these)
            if held is not None:
                more["held"] = held
            return self._cross_attention_fused(qx_raw, sq, bs, key_value_states, meta_args.cross_attn_params, dst, bound_cross, **more)

        get_xqkv = lambda m, y: self.get_xqkv(m, y, qx_raw=qx_raw.view(sq, bs, -1))
        p = meta_args.core_attn_params
        Hq = self.num_attention_heads
        fused = None
        core_dst = cross_dst = None
        # Core and text attention, which do not depend on each other, go into one launch behind the text's projection where both take a form
        # for it: few rows (waves), or two rounds of 256-row workgroups.  There the text's workgroups run beside the core's last ones: 2 to 4 %
        # of a layer of 3120 to 16200 rows and 24 or 48 heads (1233 -> 1197 us, 2215 -> 2183, 6414 -> 6264, 7670 -> 7426), 0.6 % of
        # 21600 rows x 2 chunks (29.7 -> 29.5 ms).  Between the two the core is issued as soon as it can be: its keys are in pieces that fill
        # the chip anyway, and the device would wait for what the host does for the text (one round and below: 0.90 to 1.04 of the speed);
        # what brings the pieces together then goes beside the text, and a core of whole 256-row items into the text's launch after all: 55 drawn
        # layers of 128 to 512 rows per CU 0.994 to 1.096 times as fast (2112 rows 390 -> 381 us, 2964 403 -> 389; whole 3888 373 -> 340,
        # 4176 505 -> 480), cores of other forms the same; from 44 to 83 rows per CU, which wait for the host, 0.985 to 1.026.
        held = None
        if core_bounded and cross_bounded and self.attention_dtype == "bf16":
            rows_per_cu = sq * Hq / _compute_units(hidden_states.device)  # of all heads
            if 32 < rows_per_cu < 128 or not _OWN_CROSS_FUSED.of(self):
                pass
            elif rows_per_cu <= 32:
                cp, Hkv = meta_args.cross_attn_params, self.num_query_groups_per_partition
                if attention_waves(Hq, Hkv, p.q_range.shape[0], L.MAGI_RANGES_PAIRS, p.max_seqlen_q, p.max_seqlen_k) and attention_waves(
                        Hq, Hkv, cp.cu_seqlens_q.numel() - 1, L.MAGI_RANGES_CU, cp.max_seqlen_q, cp.max_seqlen_kv):
                    held = []
            else:
                held = [] if rows_per_cu >= 512 else BegunCalls()
        elif (cross_bounded and self.attention_dtype == "fp8" and sq * Hq >= 64 * _compute_units(hidden_states.device) and _OWN_CROSS_FUSED.of(self)
              and _OWN_CORE_FP8.of(self)):
            # (e4m3 core: the text beside it in a form of its own, attn_fwd_fp8_text.hip.  28 drawn layers from 122 rows per CU on 1.006 to 1.096
            # times as fast, 86400 rows 1.001; 20 of 64 to 121, of which most wait for the host, 0.994 to 1.035; 18 below 0.997 to 1.004: their
            # core and text do not fill the chip together)
            held = []
        if proj_layout and bs == 1 and Hq % PROJ_GROUPS == 0:
            # (rows that no q range / cu_seqlens segment covers are left as allocated: the pipeline's ranges cover
            # every row, dit_model.py:220-222, 246; bf16, what the launches write, whatever hidden_states is)
            fused = torch.empty(sq, 1, 2 * Hq * D, dtype=torch.bfloat16, device=hidden_states.device)
            grouped = fused.view(sq, PROJ_GROUPS, 2, Hq // PROJ_GROUPS, D)
            core_dst, cross_dst = grouped[:, :, 0], grouped[:, :, 1]
        elif (proj_layout and bs > 1 and Hq % PROJ_GROUPS == 0 and own_cross and _OWN_BATCH.of(self) and self.attention_dtype == "bf16"
              and hidden_states.is_cuda):
            # (batch rows are further groups of heads to the core attention: position, batch, group, core | cross, head.  Without the copy that
            # put the two together: two rows of 13824 tokens, 24 heads, 4.59 -> 4.33 ms; three of 3420, 48 heads, 2.52 -> 2.30)
            fused = torch.empty(sq, bs, 2 * Hq * D, dtype=torch.bfloat16, device=hidden_states.device)
            grouped = fused.view(sq, bs, PROJ_GROUPS, 2, Hq // PROJ_GROUPS, D)
            core_dst, cross_dst = grouped.view(sq, bs * PROJ_GROUPS, 2, Hq // PROJ_GROUPS, D)[:, :, 0], grouped[:, :, :, 1]

        use_cache = inference_params is not None and (
            meta_args.extract_prefix_video_feature or meta_args.fwd_extra_1st_chunk or meta_args.slice_point > 0)
        if self.attention_dtype == "fp8":
            if bs != 1 or (use_cache and inference_params.max_batch_size != 1):
                raise ValueError("the fp8 self-attention runs at batch 1")
            core = self._core_attention_fp8(raw, rope, inference_params, meta_args, use_cache, core_dst, **({} if held is None else {"held": held}))
        elif not use_cache:
            q, kv, qx_raw = project()
            if not _OWN_CORE.of(self):
                held = None
            core = self.core_attention(q, *_halves(kv, kv.shape[0]), bs, meta_args, out=core_dst, q_prescaled=True,
                                       split_keys=True, **core_bound_kw, **({} if held is None else {"held": held}))
        else:
            if bs != 1 or inference_params.max_batch_size != 1:
                raise ValueError("the cached path runs at batch 1 (as the reference pipeline does)")
            cache = self._cache(inference_params, hidden_states.dtype)
            start = meta_args.slice_point * meta_args.clip_token_nums
            S = sq
            offloaded = cache if isinstance(cache, OffloadedKVCache) else None
            if offloaded is not None:  # kv_offload: the prefix comes through a device staging buffer
                held = None
                cache = offloaded.stage(start)
            if inference_params.update_kv_cache:
                n_keep = S - meta_args.clip_token_nums if meta_args.distill_nearly_clean_chunk else S
            else:
                n_keep = 0
            if start + n_keep > cache.shape[0]:
                if offloaded is not None:
                    offloaded.release()
                raise ValueError("KV cache overflow")
            tail = self._tail_rows(S - n_keep, cache) if n_keep < S else None
            persisted = 0
            try:
                q, _, qx_raw = project(kv_out=cache[start:], n_cache_rows=n_keep, kv_tail=tail)
                split = start + n_keep
                kc, vc = _halves(cache, split)
                if tail is None:
                    core, _ = range_attention(q, kc, vc, p.q_range, p.k_range, p.max_seqlen_q, p.max_seqlen_k,
                                              out=core_dst, return_lse=False, q_prescaled=True, share_waves=True, held=held, **core_bound_kw)
                else:
                    k2, v2 = _halves(tail, tail.shape[0])
                    core, _ = range_attention(q, kc, vc, p.q_range, p.k_range, p.max_seqlen_q, p.max_seqlen_k,
                                              k2=k2, v2=v2, k_split=split, out=core_dst,
                                              return_lse=False, q_prescaled=True, share_waves=True, held=held, **core_bound_kw)
                persisted = n_keep
            finally:
                if offloaded is not None:  # the persisted rows go back to the host behind the attention launch
                    offloaded.release(start, persisted)
        if type(held) is BegunCalls and not held:  # (the core is done: nothing for the text to go with)
            held = None
        if fused is not None:
            if cross_fused(cross_dst) is None:
                self.cross_attention(mixed_qqkv, key_value_states, meta_args.cross_attn_params, get_xqkv, out=cross_dst)
            if held is not None:
                launch_held(held)
            return fused
        core_attn_out = core.view(sq, bs, -1)
        xo = cross_fused(None)
        if held is not None:
            launch_held(held)
        if xo is not None:
            xattn_out = xo.reshape(sq, bs, -1)
        else:
            xattn_out = self.cross_attention(mixed_qqkv, key_value_states, meta_args.cross_attn_params, get_xqkv)
        if proj_layout:
            return attn_linear_proj_input(core_attn_out, xattn_out)
        return core_attn_out, xattn_out


_KERNEL_NAMES = ("online softmax, 32 rows per wavefront", "bounded-score, 64 rows per wavefront (32 in small launches)")  # by: a bound is in force
# the methods whose work forward() does in another shape, as long as they are these
_OWN_FP8_LINEAR = _Own(PerTensorQuantizedFp8Linear, "forward")
_OWN_PROJECTIONS = _Own(CustomLayerNormLinear, "forward_ln", "forward_qkvx")
_OWN_SMALL_PROJECTIONS = _Own(CustomLayerNormLinear, "forward_ln", "forward_qkvx", "forward_ln_qkvx_rows", "_split", "fused_weight")
_OWN_CROSS = _Own(FullyParallelAttention, "get_xqkv", "cross_attention")
_CROSS_FUSED = FullyParallelAttention._cross_attention_fused
_OWN_CROSS_FUSED = _Own(FullyParallelAttention, "_cross_attention_fused")
_OWN_CORE = _Own(FullyParallelAttention, "core_attention")
_OWN_CORE_FP8 = _Own(FullyParallelAttention, "_core_attention_fp8")
_OWN_SMALL = _Own(FullyParallelAttention, "_project_rows", "_fused_qkv", "_cross_attention_fused")
_OWN_SMALL_UNCACHED = _Own(FullyParallelAttention, "_project_rows", "_fused_qkv", "_cross_attention_fused", "core_attention")
_OWN_SMALL_FP8 = _Own(FullyParallelAttention, "_project_rows", "_core_attention_fp8", "_cross_attention_fused")
_SCORE_BOUNDS = FullyParallelAttention.score_bounds
_GAMMA_BETA, _PARAMETER_EPOCH = FusedLayerNorm.gamma_beta_fp32, FusedLayerNorm.parameter_epoch
_OWN_BATCH = _Own(FullyParallelAttention, "core_attention", "_cross_attention_fused")
