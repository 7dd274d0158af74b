"""Layers whose core and text attention share a launch, and whose prologue leaves the row maxima of v: forward() against itself with each of its
launches by itself, bit for bit, outputs and cache rows; and which launches there are."""
import pytest
import torch

import magi_attn as M
from magi_attn import module as MOD
from magi_attn import params as P
from magi_attn import ranges as R
from magi_attn.cache import Fp8KVCache

pytestmark = pytest.mark.gpu
D, Hq, Hkv, HIDDEN = 128, 24, 8, 256


def _case(dev, attention, chunks, Lc, prefix, cache, proj, text):
    torch.manual_seed(Lc + chunks)
    layer = MOD.FullyParallelAttention(HIDDEN, Hq, Hkv, layer_number=1, device=dev, attention_dtype=attention)
    with torch.no_grad():
        for q in layer.parameters():
            q.copy_(torch.randn_like(q.float()) * (HIDDEN ** -0.5 if q.dim() == 2 else 0.1))
        layer.linear_qkv.layer_norm.weight.add_(1.0)
    hs = torch.randn(chunks * Lc, 1, HIDDEN, device=dev).bfloat16()
    y = torch.randn(sum(text), HIDDEN, device=dev).bfloat16()
    mask = (torch.arange(max(text))[None] < torch.tensor(text)[:, None]).float().view(chunks, 1, 1, -1)
    meta = P.ModelMetaArgs(
        H=Lc, W=1, cp_pad_size=None, cp_split_sizes=None, slice_point=prefix, denoising_range_num=chunks, range_num=prefix + chunks,
        extract_prefix_video_feature=False, fwd_extra_1st_chunk=False, distill_nearly_clean_chunk=cache == "distill", clip_token_nums=Lc,
        enable_cuda_graph=False, core_attn_params=P.build_core_attn_params(R.q_ranges_from_chunks(chunks, Lc).to(dev),
                                                                          R.generate_default_kvrange(prefix, chunks, Lc).to(dev), Lc),
        cross_attn_params=P.build_cross_attn_params(mask.to(dev), Lc, max(text)))
    rope = torch.randn(chunks * Lc, 96, device=dev)
    k = torch.nn.functional.layer_norm(torch.randn(prefix * Lc, Hkv, D, device=dev), (D,))
    v = torch.randn(prefix * Lc, Hkv, D, device=dev).bfloat16()

    def run():
        ip, kept = None, []
        if cache != "none":
            ip = P.InferenceParams(1, (prefix + chunks) * Lc)
            ip.update_kv_cache = cache != "side"
            if attention == "fp8":
                store = Fp8KVCache((prefix + chunks) * Lc, Hkv, Lc, device=dev)
                scale = layer.fp8_operand_scales()[1]
                store.k[:prefix * Lc] = (k / scale).clamp(-448, 448).to(torch.float8_e4m3fn)
                store.note_constant_k_scale(scale, 0, prefix)
                M.quantize_fp8(v, Lc, 1.0, True, out=store.v[:prefix * Lc], scales_out=store.v_scale[:prefix])
                kept = [store.k.view(torch.uint8), store.v.view(torch.uint8), store.v_scale, store.k_scale]
            else:
                store = torch.zeros((prefix + chunks) * Lc, Hkv, 2 * D, dtype=torch.bfloat16, device=dev)
                store[:prefix * Lc] = torch.cat([k.bfloat16(), v], -1)
                kept = [store]
            ip.key_value_memory_dict[1] = store
        n0 = M.lib().magi_launch_count()
        with torch.no_grad():
            out = layer(hs, y, ip, rope, meta, proj_layout=proj)
        return (list(out) if isinstance(out, tuple) else [out]) + kept, M.lib().magi_launch_count() - n0

    return run


def _apart(monkeypatch):
    """forward() with nothing held and no row maxima.  (The text's items are whole in a shared launch.)"""
    attention, prologue, quantise = MOD.range_attention, MOD.qk_prologue_fp8, MOD.quantize_fp8_split

    def one(*a, held=None, **kw):
        if kw.get("q_norm") is not None:
            kw["split_keys"] = False
        return attention(*a, **kw)

    monkeypatch.setattr(MOD, "range_attention", one)
    monkeypatch.setattr(MOD, "launch_held", lambda calls: None)
    monkeypatch.setattr(MOD, "qk_prologue_fp8", lambda *a, v_raw=None, v_row_max=None, **kw: prologue(*a, **kw))
    monkeypatch.setattr(MOD, "quantize_fp8_split", lambda *a, row_max=None, **kw: quantise(*a, **kw))


# bf16: a core in pieces, of whole 256-row items, done by its first half (128 to 512 rows per CU of all heads); two rounds of 256-row workgroups and more.
# fp8: from 64 rows per CU on; row maxima from 256 rows per CU and chunks above 256 rows on.  Every kind of cache, both layouts of the outputs, text around
# a tile of 32 and 64 keys, a chunk without text.
@pytest.mark.parametrize("attention,chunks,Lc,prefix,cache,proj,text,how", [
    ("bf16", 1, 2310, 2, "append", False, [97], "begun"), ("bf16", 1, 2310, 2, "side", True, [400], "begun"), ("bf16", 3, 1296, 0, "none", True, [660, 1, 129], "begun"),
    ("bf16", 3, 1392, 2, "distill", False, [732, 70, 31], "begun"), ("bf16", 3, 1392, 2, "side", True, [64, 65, 33], "begun"),
    ("bf16", 4, 384, 4, "append", True, [162, 1, 32, 64], "done"), ("bf16", 4, 384, 4, "distill", False, [5, 0, 800, 64], "done"),
    ("bf16", 4, 1400, 1, "append", False, [31, 32, 0, 400], "held"), ("bf16", 2, 2900, 1, "distill", True, [77, 800], "held"), ("bf16", 1, 5600, 0, "none", False, [129], "held"),
    ("bf16", 4, 1400, 1, "side", True, [1, 2, 3, 4], "held"),
    ("fp8", 2, 640, 1, "append", True, [400, 33], "held"), ("fp8", 12, 240, 1, "distill", False, [24] * 11 + [0], "held"), ("fp8", 3, 1000, 2, "append", False, [65, 0, 300], "held, maxima"),
    ("fp8", 3, 1000, 2, "side", True, [65, 129, 300], "held, maxima"), ("fp8", 3, 1001, 1, "distill", True, [31, 800, 97], "held, maxima"),
    ("fp8", 1, 2801, 0, "none", False, [161], "held, maxima"), ("fp8", 3, 1001, 1, "distill", False, [31, 800, 97], "held, maxima")])
def test_the_bits_of_the_launches_one_by_one(dev, monkeypatch, attention, chunks, Lc, prefix, cache, proj, text, how):
    run = _case(dev, attention, chunks, Lc, prefix, cache, proj, text)
    seen = []
    launch, quantise = MOD.launch_held, MOD.quantize_fp8_split
    monkeypatch.setattr(MOD, "_compute_units", lambda device: 256)
    with monkeypatch.context() as m:
        m.setattr(MOD, "launch_held", lambda calls: (seen.append("begun" if calls[0][1] is None else "held"), seen.append(len(calls)), launch(calls)))
        m.setattr(MOD, "quantize_fp8_split", lambda *a, **kw: (seen.append("maxima") if kw.get("row_max") is not None else None, quantise(*a, **kw))[1])
        got, n = run()
    with monkeypatch.context() as m:
        _apart(m)
        want, n_apart = run()
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        kind = how.split(",")[0]
        assert [s for s in seen if s != "maxima"] == ([] if kind == "done" else [kind, 2]) and ("maxima" in seen) == ("maxima" in how)
        assert n == n_apart - (kind != "done")
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.shape == b.shape and torch.equal(a, b) and (a.dtype is torch.uint8 or bool(torch.isfinite(a).all()))
