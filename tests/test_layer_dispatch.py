"""Layers with replaced parts or inputs of another type: what they run beside the library's own methods."""
import pytest
import torch

from magi_attn import module as MOD
from magi_attn import params as P
from magi_attn import ranges as R

D = 128


def _meta(dev, batch, chunks, Lc, text):
    mask = (torch.arange(max(text))[None] < torch.tensor(text)[:, None]).float().view(len(text), 1, 1, -1)
    return P.ModelMetaArgs(
        H=Lc, W=1, cp_pad_size=None, cp_split_sizes=None, slice_point=0, denoising_range_num=chunks, range_num=chunks,
        extract_prefix_video_feature=False, fwd_extra_1st_chunk=False, distill_nearly_clean_chunk=False, clip_token_nums=Lc, enable_cuda_graph=False,
        core_attn_params=P.build_core_attn_params(R.q_ranges_from_chunks(chunks, Lc).to(dev), R.generate_default_kvrange(0, chunks, Lc).to(dev), Lc),
        cross_attn_params=P.build_cross_attn_params(mask.to(dev), Lc, max(text)))


def _layer(dev, hidden=256, Hq=8, Hkv=2, **kw):
    torch.manual_seed(7)
    layer = MOD.FullyParallelAttention(hidden, Hq, Hkv, layer_number=1, device=dev, **kw)
    with torch.no_grad():
        for p in layer.parameters():
            p.copy_(torch.randn_like(p.float()) * (hidden ** -0.5 if p.dim() == 2 else 0.1))
        layer.linear_qkv.layer_norm.weight.add_(1.0)
    return layer


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 2])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_layout_of_the_projection_for_rows_of_another_type(dev, batch, dtype):
    """An input norm that takes other types than bf16: what the attentions write is bf16 whatever the rows that came in are."""
    layer, rows = _layer(dev), 40
    own = layer.linear_qkv.forward_ln
    layer.linear_qkv.forward_ln = lambda h: own(h.bfloat16())
    hs = torch.randn(rows, batch, 256, device=dev).bfloat16()
    y = torch.randn(13 * batch, 256, device=dev).bfloat16()
    meta, rope = _meta(dev, batch, 1, rows, [13] * batch), torch.randn(rows, 96, device=dev)
    with torch.no_grad():
        want = layer(hs, y, None, rope, meta, proj_layout=True)
        got = layer(hs.to(dtype), y, None, rope, meta, proj_layout=True)
        apart = MOD.attn_linear_proj_input(*layer(hs.to(dtype), y, None, rope, meta))
    assert got.dtype is torch.bfloat16 and torch.equal(got, apart) and torch.equal(got, want)


@pytest.mark.parametrize("attention", ["bf16", "fp8"])
@pytest.mark.parametrize("how", ["instance", "subclass", "norm's epoch"])
def test_norm_parameters_where_the_bounds_do_not_look_at_them(attention, how):
    """Bounds of a caller's own, which need not ask the norms for anything: the parameters are converted all the same, and again when
    they change."""
    layer = MOD.FullyParallelAttention(256, 8, 2, attention_dtype=attention)
    lns = [getattr(layer, n) for n in ("q_layernorm", "k_layernorm", "q_layernorm_xattn", "k_layernorm_xattn")]
    own = lambda self, rotary_half=48: (30.0, 30.0)  # noqa: E731
    if how == "instance":
        layer.score_bounds = own.__get__(layer)
    elif how == "subclass":
        layer.__class__ = type("Other", (type(layer),), {"score_bounds": own})
    else:
        for ln in lns:
            ln.parameter_epoch = lambda: 1
    for step in range(3):
        with torch.no_grad():
            for ln in lns:
                ln.weight.fill_(step * 0.5)
                ln.bias.fill_(step * 0.25)
        layer.score_bounds(48)
        for g, b in layer._norm_parameters():
            assert (g == step * 0.5).all() and (b == step * 0.25).all()
