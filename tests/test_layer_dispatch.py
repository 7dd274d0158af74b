"""Layers with replaced parts: what they run beside the library's own methods."""
import pytest
import torch

from magi_attn import module as MOD


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
