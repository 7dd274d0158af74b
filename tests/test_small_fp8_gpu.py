"""Small layers with e4m3 attention: magi_small_projections_e4m3, the quantiser of V and two attention launches, against the separate
launches and against float64."""
import pytest
import torch

import magi_attn as M
from magi_attn import functional as F
from magi_attn import module as MOD
from magi_attn import params as P
from magi_attn import ranges as R
from magi_attn.cache import Fp8KVCache
from magi_attn.module import FullyParallelAttention
from magi_attn.rope import LearnableRotaryEmbeddingCat

pytestmark = pytest.mark.gpu
D = 128


def _case(dev, hidden, heads, frames, rows, cols, dn, sp, cache, proj, text):
    torch.manual_seed(hidden + dn)
    Hq, Hkv = heads
    Lc = frames * rows * cols
    layer = FullyParallelAttention(hidden, Hq, Hkv, layer_number=1, device=dev, attention_dtype="fp8")
    with torch.no_grad():
        for q in layer.parameters():
            q.copy_(torch.randn_like(q.float()) * (hidden ** -0.5 if q.dim() == 2 else 0.1))
        layer.linear_qkv.layer_norm.weight.add_(1.0)
    hs = torch.randn(dn * Lc, 1, hidden, device=dev).bfloat16()
    y = torch.randn(sum(text), hidden, device=dev).bfloat16()
    mask = (torch.arange(max(text))[None] < torch.tensor(text)[:, None]).float().view(dn, 1, 1, -1)
    meta = P.ModelMetaArgs(
        H=rows, W=cols, cp_pad_size=None, cp_split_sizes=None, slice_point=sp, denoising_range_num=dn, range_num=sp + dn,
        extract_prefix_video_feature=False, fwd_extra_1st_chunk=False, distill_nearly_clean_chunk=cache == "distill", clip_token_nums=Lc,
        enable_cuda_graph=False, core_attn_params=P.build_core_attn_params(R.q_ranges_from_chunks(dn, Lc).to(dev),
                                                                          R.generate_default_kvrange(sp, dn, Lc).to(dev), Lc),
        cross_attn_params=P.build_cross_attn_params(mask.to(dev), Lc, max(text)))
    rope = LearnableRotaryEmbeddingCat(D, device=dev).get_embed_for_forward(dn * frames, rows, cols, sp, dn)
    k = torch.nn.functional.layer_norm(torch.randn(sp * Lc, Hkv, D, device=dev), (D,))
    v = torch.randn(sp * Lc, Hkv, D, device=dev).bfloat16()

    def run():
        ip, kept = None, []
        if cache != "none":
            ip = P.InferenceParams(1, (sp + dn) * Lc)
            ip.update_kv_cache = cache != "side"
            store = Fp8KVCache((sp + dn) * Lc, Hkv, Lc, device=dev)
            scale = layer.fp8_operand_scales()[1]
            store.k[:sp * Lc] = (k / scale).clamp(-448, 448).to(torch.float8_e4m3fn)
            store.note_constant_k_scale(scale, 0, sp)
            M.quantize_fp8(v, Lc, 1.0, True, out=store.v[:sp * Lc], scales_out=store.v_scale[:sp])
            ip.key_value_memory_dict[1] = store
            kept = [store.k.view(torch.uint8), store.v.view(torch.uint8), store.v_scale, store.k_scale]
        n0 = M.lib().magi_launch_count()
        with torch.no_grad():
            out = layer(hs, y, ip, rope, meta, proj_layout=proj)
        n = M.lib().magi_launch_count() - n0
        return list(out) if isinstance(out, tuple) else [out], kept, n

    return layer, run


CASES = [(768, (6, 2), (2, 6, 10), 2, 2, "append", False, [24, 13]), (768, (8, 2), (2, 6, 10), 2, 2, "side", True, [3, 800]),
         (256, (6, 2), (1, 5, 9), 3, 1, "distill", False, [8, 0, 1]), (1024, (3, 3), (1, 3, 11), 1, 0, "none", True, [40]),
         (768, (6, 2), (2, 14, 10), 3, 2, "append", False, [300, 9, 77])]


@pytest.mark.parametrize("hidden,heads,grid,dn,sp,cache,proj,text", CASES)
def test_gives_what_the_separate_launches_give(dev, monkeypatch, hidden, heads, grid, dn, sp, cache, proj, text):
    """Both sum the products over K from first to last and round at the same places, so q, k and v are the same up to a neighbouring
    value where a sum lies beside a rounding boundary: one in some thousand bytes of the cache, and the outputs accordingly."""
    layer, run = _case(dev, hidden, heads, *grid, dn, sp, cache, proj, text)
    out, kept, n = run()
    monkeypatch.setattr(MOD, "_projects_in_one_launch", lambda *a: False)
    monkeypatch.setattr(MOD, "_text_in_one_launch", lambda *a: False)
    ref, ref_kept, n_apart = run()
    assert n == 4 and n_apart == n + 2  # (and the library's two products)
    for a, b in zip(kept[:2], ref_kept[:2]):
        assert (a != b).float().mean().item() <= 1e-3
    for a, b in zip(kept[2:], ref_kept[2:]):
        assert torch.equal(a, b)
    for a, b in zip(out, ref):
        x, y = a.double().flatten(), b.double().flatten()
        # (a direction 1.4e-2 away at most, and no scale of its own; measured: no element differs in any of the cases)
        assert a.shape == b.shape and float(x @ y / (x.norm() * y.norm())) >= 0.9999 and float((x - y).norm() / y.norm()) <= 1.5e-2


@pytest.mark.parametrize("S,K,T,kept", [(1, 64, 1, 1), (33, 192, 65, 20), (97, 1024, 0, 0), (1313, 256, 129, 700), (65, 1088, 33, 65)])
def test_e4m3_projections_against_float64(dev, S, K, T, kept):
    Hq, Hkv, Hqx, R2, premul, qs, ks = 3, 2, 1, 48, 0.1275, 2.0 ** -6, 2.0 ** -4
    g = torch.Generator(device=dev).manual_seed(S + K)
    rnd = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
    x, w, wt = rnd(S, K).bfloat16(), (rnd((Hq + 2 * Hkv + Hqx) * D, K) * K ** -0.5).bfloat16(), (rnd(2 * Hkv * D, K) * K ** -0.5).bfloat16()
    text, rope, par = rnd(max(T, 1), K).bfloat16(), rnd(S, 2 * R2), [rnd(D) * 0.2 for _ in range(6)]
    q8, k8, side = (torch.zeros(n, h, D, dtype=torch.float8_e4m3fn, device=dev) for n, h in ((S, Hq), (kept + 1, Hkv), (S - kept + 1, Hkv)))
    v, qx, tkv = (torch.zeros(n, h, d, dtype=torch.bfloat16, device=dev) for n, h, d in ((S, Hkv, D), (S, Hqx, D), (max(T, 1), Hkv, 2 * D)))
    F.launch_small_projections_e4m3(
        x.device, qs, ks, v.data_ptr(), x.data_ptr(), w.data_ptr(), 0, 0, K, S, K, 0, 0.0, Hq, Hkv, Hqx, R2, rope.data_ptr(), *(p.data_ptr() for p in par[:4]),
        1e-6, 1, premul, kept, q8.data_ptr(), k8.data_ptr(), side.data_ptr(), Hkv * D, Hkv * D, qx.data_ptr(), text.data_ptr(), wt.data_ptr(), K, T, K,
        par[4].data_ptr(), par[5].data_ptr(), tkv.data_ptr())
    raw = (x.double() @ w.double().T).bfloat16().double().view(S, -1, D)

    def normed(r, gamma, beta):
        y = torch.nn.functional.layer_norm(r, (D,), eps=1e-6) * (gamma.double() + 1) + beta.double()
        s, c = rope.double()[:, None, :R2], rope.double()[:, None, R2:]
        a, b = y[..., :R2], y[..., R2:2 * R2]
        return torch.cat([a * c - b * s, a * s + b * c, y[..., 2 * R2:]], -1)

    got = [q8.float() * qs, torch.cat([k8[:kept], side[:S - kept]]).float() * ks]
    want = [normed(raw[:, :Hq], par[0], par[1]) * premul, normed(raw[:, Hq:Hq + Hkv], par[2], par[3])]
    for a, b in zip(got, want):
        # e4m3: 2^-4 of the value, 2^-10 of the scale below its normal range; the raw projection's neighbour, 2^-8, where its sum is beside a boundary
        scale = qs if a is got[0] else ks
        assert ((a.double() - b).abs() <= b.abs() * (2.0 ** -4 + 2.0 ** -6) + scale * 2.0 ** -9 + 2.0 ** -7 * b.abs().amax(-1, keepdim=True)).all()
    assert torch.equal(k8[kept].view(torch.uint8), torch.zeros_like(k8[kept].view(torch.uint8)))  # (the row behind the share is not touched)
    assert ((v.double() - raw[:, Hq + Hkv:Hq + 2 * Hkv]).abs() <= raw[:, Hq + Hkv:Hq + 2 * Hkv].abs() * 2.0 ** -7 + 1e-6).all()


def test_refused_calls_stay_refused(dev):
    layer, run = _case(dev, 768, (6, 2), 2, 6, 10, 2, 2, "append", False, [24, 13])
    store = Fp8KVCache(120 * 3, 2, 120, device=dev)  # one chunk short
    hs = torch.zeros(240, 1, 768, dtype=torch.bfloat16, device=dev)
    for cache, error in ((store, "overflow"), (Fp8KVCache(480, 2, 60, device=dev), "chunk_tokens"), (torch.zeros(480, 2, 256, device=dev), "Fp8KVCache")):
        ip = P.InferenceParams(1, 480)
        ip.update_kv_cache = True
        ip.key_value_memory_dict[1] = cache
        meta = P.ModelMetaArgs(
            H=6, W=10, cp_pad_size=None, cp_split_sizes=None, slice_point=2, denoising_range_num=2, range_num=4, extract_prefix_video_feature=False,
            fwd_extra_1st_chunk=False, distill_nearly_clean_chunk=False, clip_token_nums=120, enable_cuda_graph=False,
            core_attn_params=P.build_core_attn_params(R.q_ranges_from_chunks(2, 120).to(dev), R.generate_default_kvrange(2, 2, 120).to(dev), 120),
            cross_attn_params=P.build_cross_attn_params(torch.ones(2, 1, 1, 5, device=dev), 120, 5))
        with pytest.raises(ValueError, match=error), torch.no_grad():
            layer(hs, torch.zeros(10, 768, dtype=torch.bfloat16, device=dev), ip, torch.zeros(240, 96, device=dev), meta)


@pytest.mark.parametrize("how", ["instance", "subclass"])
@pytest.mark.parametrize("on,name", [("layer", "_core_attention_fp8"), ("layer", "_cross_attention_fused"), ("layer", "_project_rows"),
                                     ("linear_qkv", "forward_ln_qkvx_rows"), ("linear_qkv", "forward_ln")])
def test_replaced_methods_are_called(dev, on, name, how):
    """What the separate launches call runs where it is not the library's own."""
    for cache in ("none", "append"):
        layer, run = _case(dev, 256, (6, 2), 1, 5, 9, 2, 0 if cache == "none" else 1, cache, False, [8, 5])
        want, _, n_small = run()
        m, calls = layer if on == "layer" else layer.linear_qkv, []
        own = getattr(type(m), name)
        new = lambda self, *a, **k: calls.append(1) or own(self, *a, **k)  # noqa: E731
        if how == "instance":
            m.__dict__[name] = new.__get__(m)
        else:
            m.__class__ = type("Other", (type(m),), {name: new})
        got, _, n = run()
        assert n_small == 4 and n > n_small and calls
        for a, b in zip(got, want):
            x, y = a.double().flatten(), b.double().flatten()
            assert float(x @ y / (x.norm() * y.norm())) >= 0.9999
