"""The projections of a small layer in one launch (magi_small_projections) against float64, and the layer that takes it.

Expected values: the normalised input in float64 rounded to bf16, the product in float64 rounded to bf16 (the raw projection), norm,
rotary and factor in float64.  The kernel rounds at the same places from fp32 sums, so a value beside a rounding boundary may
land on the neighbouring bf16, as in any product summed in another order: the 2-norm of a difference stays near that of the one
rounding to bf16 that the expected values do without (2^-9 / sqrt(3) = 1.1e-3 uniformly, 1.7e-3 at the low end of a binade), bar
2.5e-3, and no element is further off than 2^-6 of its row's largest."""
import ctypes as C
import dataclasses
import os
import subprocess

import pytest
import torch

import magi_attn as M
from magi_attn import _lib as L
from magi_attn import module as MOD
from magi_attn import params as P
from magi_attn import ranges as R

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
D = 128


def _near(got, want, what):
    got, want = got.double().cpu().reshape(-1, D), want.double().cpu().reshape(-1, D)
    assert torch.isfinite(got).all(), what
    assert (got - want).norm() <= 2.5e-3 * want.norm(), (what, float((got - want).norm() / want.norm()))
    assert ((got - want).abs().amax(1) <= 2.0 ** -6 * want.abs().amax(1) + 1e-12).all(), what


def _head_norm(raw, gamma, beta, eps=1e-6):
    x = raw.view(raw.shape[0], -1, D)
    return torch.nn.functional.layer_norm(x, (D,), eps=eps) * (gamma.double() + 1) + (0 if beta is None else beta.double())


def _rotate(x, rope, batch, R2):
    t = rope.double().repeat_interleave(batch, 0)[:, None]
    s, c = t[..., :R2], t[..., R2:]
    a, b = x[..., :R2], x[..., R2:2 * R2]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., 2 * R2:]], -1)


# K: one stage, fewer stages than the kernel keeps in flight, all remainders of the ring, resident limits; S and T: edges of 32
# and 64 rows; the taller workgroups (more than one round of the 32-row ones, K up to 768); rows that stream (K above 1024)
@pytest.mark.gpu
@pytest.mark.parametrize("S,K,T,Kt,Hq,Hkv,batch,kept,ln,beta,R2", [
    (1, 64, 1, 64, 2, 1, 1, 1, "bf16", True, 48), (31, 128, 33, 192, 6, 2, 1, 0, "fp32", True, 48), (33, 192, 65, 64, 3, 3, 3, 20, "bf16", False, 48),
    (64, 256, 31, 320, 6, 2, 2, 64, None, True, 32), (240, 768, 24, 768, 6, 2, 1, 120, "bf16", True, 48), (97, 1024, 40, 1024, 4, 2, 1, 97, "bf16", True, 0),
    (1313, 256, 129, 256, 6, 2, 1, 700, "bf16", True, 48), (700, 768, 63, 704, 6, 2, 1, 699, "fp32", False, 48), (1281, 64, 0, 0, 6, 2, 1, 1281, "bf16", True, 64),
    (65, 1088, 33, 3072, 2, 2, 1, 1, None, True, 48), (0, 0, 402, 3072, 0, 8, 1, 0, None, True, 0), (0, 0, 1, 1088, 0, 1, 1, 0, None, False, 0),
    (0, 0, 97, 1152, 0, 40, 1, 0, None, True, 0), (150, 1088, 0, 0, 26, 3, 1, 150, None, True, 48), (0, 0, 800, 3072, 0, 8, 1, 0, None, True, 0)])
def test_small_projections_against_float64(dev, S, K, T, Kt, Hq, Hkv, batch, kept, ln, beta, R2):
    g = torch.Generator(device=dev).manual_seed(S + T + K)
    rnd = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
    par = [rnd(D) * 0.2 for _ in range(6)]
    if not beta:
        par[1] = par[3] = par[5] = None
    kw, x, w, rope = {}, None, None, None
    if S:
        heads = 2 * Hq + 2 * Hkv
        x = (rnd(S, K + 8) * 3 + 1).bfloat16()[:, :K]  # (rows further apart than they are long, a mean well away from zero)
        w = (rnd(heads * D, K) * K ** -0.5).bfloat16()
        if ln:
            dt = torch.float32 if ln == "fp32" else torch.bfloat16
            kw["ln"] = ((1 + 0.1 * rnd(K)).to(dt), (0.1 * rnd(K)).to(dt), 1e-5)
        if R2:
            angle = torch.rand(S // batch, R2, device=dev, generator=g) * 60
            rope = torch.cat([angle.sin(), angle.cos()], -1)
        cache, tail = (torch.full((n, Hkv, 2 * D), 7.0, device=dev, dtype=torch.bfloat16) for n in (kept + 2, S - kept + 2))
        kw.update(kv_out=cache if kept else None, kv_tail=tail if kept < S else None, n_cache_rows=kept)
    if T:
        y = (rnd(T, Kt + 16) * 0.5).bfloat16()[:, :Kt]
        wt = (rnd(2 * Hkv * D, Kt) * Kt ** -0.5).bfloat16()
        kw["text"] = (y, wt, par[4], par[5])
    q, _, _, qx, kv_text = M.small_projections(x, w, rope, *par[:4], Hq=Hq, Hkv=Hkv, Hqx=Hq if S else 0, batch=batch, q_premul=0.1275, **kw)
    if S:
        xn = x.double()
        if ln:
            lw, lb, le = kw["ln"]
            xn = torch.nn.functional.layer_norm(xn, (K,), lw.double(), lb.double(), le).bfloat16().double()
        raw = (xn @ w.double().T).bfloat16().double()
        rq, rk, rv, rx = raw.split((Hq * D, Hkv * D, Hkv * D, Hq * D), -1)
        want = [_head_norm(rq, par[0], par[1]), _head_norm(rk, par[2], par[3])]
        if R2:
            want = [_rotate(t, rope, batch, R2) for t in want]
        _near(q, want[0] * 0.1275, "q")
        _near(qx, rx, "qx")
        kv = torch.cat([cache[:kept], tail[:S - kept]])
        _near(kv[..., :D], want[1], "k")
        _near(kv[..., D:], rv, "v")
        assert (cache[kept:] == 7).all() and (tail[S - kept:] == 7).all()  # nothing beyond the rows asked for
    if T:
        raw = (y.double() @ wt.double().T).bfloat16().double().view(T, Hkv, 2 * D)
        _near(kv_text[..., :D], _head_norm(raw[..., :D].reshape(T, -1), par[4], par[5]), "text k")
        _near(kv_text[..., D:], raw[..., D:], "text v")


@pytest.mark.gpu
def test_small_projections_refuses_what_it_does_not_implement(dev):
    b = lambda *s: torch.zeros(*s, device=dev, dtype=torch.bfloat16)  # noqa: E731
    p = torch.zeros(D, device=dev)
    call = lambda K, **kw: M.small_projections(b(4, K), b(3 * D, K), None, p, p, p, p, Hq=1, Hkv=1, **kw)  # noqa: E731
    for K, kw in ((96, {}), (1088, {"ln": (b(1088), b(1088), 1e-6)}), (64, {"ln": (b(64), b(64), 1e-6), "text": (b(2, 1088), b(2 * D, 1088), p, p)})):
        with pytest.raises(M.MagiError):
            call(K, **kw)
    with pytest.raises(ValueError):
        call(64, kv_out=b(3, 1, 2 * D), n_cache_rows=4)
    with pytest.raises(ValueError):
        M.small_projections(None, None, None, p, p, p, p, Hq=1, Hkv=1)


def _layer_case(dev, hidden, frames, rows, cols, dn, sp, cache, proj, text, seed=3):
    from magi_attn.rope import LearnableRotaryEmbeddingCat

    Hq, Hkv, Lc = 8, 2, frames * rows * cols
    torch.manual_seed(seed)
    layer = MOD.FullyParallelAttention(hidden, Hq, Hkv, layer_number=1, device=dev)
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
    prefix = torch.randn(sp * Lc, Hkv, 2 * D, device=dev).bfloat16()

    def run():
        ip = None
        if cache != "none":
            ip = P.InferenceParams(1, (sp + dn) * Lc)
            ip.update_kv_cache = cache != "side"
            kept = torch.zeros((sp + dn) * Lc, Hkv, 2 * D, dtype=torch.bfloat16, device=dev)
            kept[:sp * Lc] = prefix
            ip.key_value_memory_dict[1] = kept
        n0 = M.lib().magi_launch_count()
        with torch.no_grad():
            out = layer(hs, y, ip, rope, meta, proj_layout=proj)
        n = M.lib().magi_launch_count() - n0
        return (list(out) if isinstance(out, tuple) else [out]) + ([] if ip is None else [kept]), n

    return layer, run, (hs, y, meta, rope)


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,grid,dn,sp,cache,proj,text", [
    (768, (2, 6, 10), 2, 2, "append", False, [24, 13]), (768, (2, 6, 10), 2, 2, "side", True, [3, 800]), (256, (1, 5, 9), 3, 1, "distill", False, [8, 0, 1]),
    (1024, (1, 3, 11), 1, 0, "none", True, [40]), (768, (2, 14, 10), 3, 2, "append", False, [300, 9, 77])])
def test_small_layer_gives_what_the_separate_launches_give(dev, monkeypatch, hidden, grid, dn, sp, cache, proj, text):
    """Outputs and cache rows, within what the order of the products' sums does to them (the bar of the fused projection: cosine
    0.9999, 2e-2 of magnitude-one outputs); three launches instead of five of this library's, and no library product."""
    layer, run, _ = _layer_case(dev, hidden, *grid, dn, sp, cache, proj, text)
    got, n_small = run()
    monkeypatch.setattr(MOD, "_projects_in_one_launch", lambda *a: False)
    monkeypatch.setattr(MOD, "_text_in_one_launch", lambda *a: False)
    want, n_apart = run()
    assert n_small == n_apart - 2
    for a, b in zip(got, want):
        x, y = a.double().flatten(), b.double().flatten()
        assert a.shape == b.shape and float(x @ y / (x.norm() * y.norm())) >= 0.9999 and float((x - y).abs().max()) <= 2e-2 * max(1.0, float(y.abs().max()))


# K: one piece for a part of the norm's 64 lanes, for all of them, two pieces; 32 and 64 rows a workgroup; rows that stream
@pytest.mark.gpu
@pytest.mark.parametrize("S,K,T,Kt,Hq,Hkv,ln,beta", [
    (32, 64, 32, 128, 2, 1, "bf16", True), (97, 448, 40, 512, 6, 2, "fp32", True), (240, 768, 45, 768, 6, 2, "bf16", True), (96, 1024, 33, 1024, 4, 4, "bf16", False),
    (1344, 768, 131, 768, 6, 2, "fp32", False), (0, 0, 65, 3072, 0, 8, None, True), (0, 0, 300, 3072, 0, 8, None, False), (0, 0, 800, 1088, 0, 8, None, True)])
def test_bits_are_those_of_the_separate_launches(dev, S, K, T, Kt, Hq, Hkv, ln, beta):
    """Norm, projections, prologue and head norm one after the other give every bit of the one launch, at sizes where the library's
    product does not cut K in pieces; and a row's bits do not depend on where it lies."""
    g = torch.Generator(device=dev).manual_seed(S + T + K)
    rnd = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
    par = [rnd(D) * 0.2 for _ in range(6)]
    if not beta:
        par[1] = par[3] = par[5] = None
    linear, kw, x, w, rope = torch.nn.functional.linear, {}, None, None, None
    if S:
        x, w = (rnd(S, K) * 2 + 0.5).bfloat16(), (rnd(2 * (Hq + Hkv) * D, K) * K ** -0.5).bfloat16()
        dt = torch.float32 if ln == "fp32" else torch.bfloat16
        kw["ln"] = ((1 + 0.1 * rnd(K)).to(dt), (0.1 * rnd(K)).to(dt), 1e-6)
        angle = torch.rand(S, 48, device=dev, generator=g) * 60
        rope = torch.cat([angle.sin(), angle.cos()], -1)
    y, wt = rnd(T, Kt).bfloat16(), (rnd(2 * Hkv * D, Kt) * Kt ** -0.5).bfloat16()
    one = lambda x, rope, y: M.small_projections(x, w, rope, *par[:4], Hq=Hq, Hkv=Hkv, Hqx=Hq, q_premul=0.1275,  # noqa: E731
                                                 text=(y, wt, par[4], par[5]), **kw)
    q, kv, _, qx, text_kv = one(x, rope, y)
    if S:
        rq, rk, rv, rx = linear(M.layer_norm(x, *kw["ln"]), w).split((Hq * D, Hkv * D, Hkv * D, Hq * D), -1)
        want_q, want_kv, _ = M.qk_prologue(rq, rk, rv, rope, *par[:4], Hq=Hq, Hkv=Hkv, q_premul=0.1275)
        assert torch.equal(qx.view(S, -1), rx) and torch.equal(kv, want_kv) and torch.equal(q, want_q)
    raw = linear(y, wt).view(T, Hkv, 2 * D)
    assert torch.equal(text_kv[..., D:], raw[..., D:]) and torch.equal(text_kv[..., :D], M.head_norm(raw[..., :D], par[4], par[5]))
    turned = one(None if x is None else x.flip(0).contiguous(), None if rope is None else rope.flip(0).contiguous(), y.flip(0).contiguous())
    for a, b in zip((q, kv, qx, text_kv), (turned[0], turned[1], turned[3], turned[4])):
        assert a is None or torch.equal(a, b.flip(0))


@pytest.mark.gpu
@pytest.mark.parametrize("ranges", ["a gap behind each", "one of three"])
def test_rows_outside_the_ranges_of_a_small_layer_are_zeros(dev, ranges):
    """By the attention launch where the ranges can cover the rows, by a clearing pass where they cannot."""
    layer, _, (hs, y, meta, rope) = _layer_case(dev, 256, 1, 5, 9, 3, 0, "none", False, [8, 3, 1])
    p = meta.core_attn_params
    if ranges == "one of three":
        q, k, covered = p.q_range[1:2].contiguous(), p.k_range[1:2].contiguous(), torch.arange(135, device=dev) // 45 == 1
    else:
        q, k, covered = p.q_range - torch.tensor([0, 4], dtype=torch.int32, device=dev), p.k_range, torch.arange(135, device=dev) % 45 < 41
    with torch.no_grad():
        whole = layer(hs, y, None, rope, meta)[0]
        layer(hs * 3, y, None, rope, meta)  # (so that freshly allocated outputs hold something)
        part = layer(hs, y, None, rope, dataclasses.replace(meta, core_attn_params=dataclasses.replace(p, q_range=q, k_range=k)))[0]
    assert (part[~covered] == 0).all() and torch.equal(part[covered], whole[covered])


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["patched forward_ln", "hidden rows apart", "text rows backwards", "fp32 text", "autocast", "above the bound", "batch"])
def test_layers_that_the_one_launch_does_not_take(dev, monkeypatch, what):
    """Replaced projections are called; other layouts, types and modes go where they went."""
    layer, run, (hs, y, meta, rope) = _layer_case(dev, 256, 1, 4, 6, 2, 1, "none", False, [8, 5])
    taken = []
    for name in ("small_projections", "launch_small_projections"):
        monkeypatch.setattr(MOD, name, lambda *a, _f=getattr(MOD, name), **k: taken.append(1) or _f(*a, **k))
    call = lambda h, t: layer(h, t, None, rope, meta)  # noqa: E731
    with torch.no_grad():
        want = call(hs, y)
        assert taken
        taken.clear()
        if what == "patched forward_ln":
            calls, own = [], layer.linear_qkv.forward_ln
            layer.linear_qkv.forward_ln = lambda t: calls.append(1) or own(t)
            got = call(hs, y)
            assert calls
        elif what == "hidden rows apart":
            got = call(torch.cat([hs, hs], -1)[..., :256], y)
        elif what == "text rows backwards":  # (columns apart: not rows in one piece)
            got = call(hs, torch.stack([y, y], -1)[..., 0])
        elif what == "fp32 text":
            with pytest.raises(RuntimeError):
                call(hs, y.float())
            return
        elif what == "autocast":
            with torch.autocast("cuda", dtype=torch.bfloat16):
                got = call(hs, y)
        elif what == "above the bound":
            layer.q_layernorm_xattn.weight.fill_(20.0)
            got, want = call(hs, y), None
        else:
            with pytest.raises(ValueError):  # (as ever: a batch is one range)
                layer(torch.cat([hs, hs], 1), y, None, rope, meta)
            return
    text_only = what in ("patched forward_ln", "hidden rows apart")
    assert len(taken) <= (1 if text_only else 0)
    if want is not None:
        for a, b in zip(got, want):
            assert float((a.float() - b.float()).abs().max()) <= 2e-2 * max(1.0, float(b.abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["instance", "subclass"])
@pytest.mark.parametrize("on,name", [("layer", "core_attention"), ("layer", "_fused_qkv"), ("layer", "_cross_attention_fused"),
                                     ("layer", "_project_rows"), ("linear_qkv", "forward_ln_qkvx_rows"), ("linear_qkv", "forward_ln")])
def test_replaced_methods_of_a_small_layer_are_called(dev, on, name, how):
    """Whatever the separate launches call runs in small layers too where it is not the library's own; core_attention without a cache
    only, as ever.  One put in its place may have the arguments of before the text's own launch."""
    for cache in ("none", "append"):
        layer, run, _ = _layer_case(dev, 256, 1, 5, 9, 2, 1, cache, False, [33, 20])
        want, n_small = run()
        m, calls = layer if on == "layer" else layer.linear_qkv, []
        own = getattr(type(m), name)
        new = lambda self, *a, **k: calls.append(k) or own(self, *a, **k)  # noqa: E731
        if name == "_cross_attention_fused":
            new = lambda self, qx, sq, b, kvs, p, dst, bound: calls.append(1) or own(self, qx, sq, b, kvs, p, dst, bound)  # noqa: E731
        if how == "instance":
            m.__dict__[name] = new.__get__(m)
        else:
            m.__class__ = type("Other", (type(m),), {name: new})
        got, n = run()
        assert bool(calls) == (name != "core_attention" or cache == "none")
        assert (n > n_small) == bool(calls)
        assert all(torch.equal(a, b) for a, b in zip(got, want))


class _TwiceTheProduct(torch.Tensor):
    """A weight with a product of its own, as quantised or sharded ones have."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        out = super().__torch_function__(func, types, args, kwargs or {})
        return out.as_subclass(torch.Tensor) * 2 if func is torch.nn.functional.linear else out


@pytest.mark.gpu
@pytest.mark.parametrize("small", [True, False])
def test_text_weight_with_a_product_of_its_own(dev, monkeypatch, small):
    """Is asked for it, not read: the values (not normed) and so the cross attention come out twice as large."""
    layer, run, _ = _layer_case(dev, 256, 1, 5, 9, 2, 1, "none", False, [33, 20])
    if not small:
        monkeypatch.setattr(MOD, "_projects_in_one_launch", lambda *a: False)
    want, _ = run()
    layer.linear_kv_xattn.weight = torch.nn.Parameter(layer.linear_kv_xattn.weight.detach().as_subclass(_TwiceTheProduct), requires_grad=False)
    got, _ = run()
    assert torch.equal(got[0], want[0])
    assert float((got[1].float() - 2 * want[1].float()).abs().max()) <= 2e-2 * float(want[1].abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("slice_point", [-1, 3, 5])
def test_positions_outside_the_cache_are_refused_in_small_layers(dev, monkeypatch, slice_point):
    """Ahead of and behind the cached rows, before anything is launched by address."""
    layer, _, (hs, y, meta, rope) = _layer_case(dev, 256, 1, 5, 9, 2, 1, "append", False, [33, 20])
    monkeypatch.setattr(MOD, "launch_small_projections", lambda *a: pytest.fail("launched"))
    ip = P.InferenceParams(1, 4 * 45)
    ip.key_value_memory_dict[1] = torch.full((4 * 45, 2, 2 * D), 7.0, dtype=torch.bfloat16, device=dev)
    ip.update_kv_cache = True
    with torch.no_grad(), pytest.raises(ValueError):
        layer(hs, y, ip, rope, dataclasses.replace(meta, slice_point=slice_point, extract_prefix_video_feature=True))
    assert (ip.key_value_memory_dict[1] == 7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("heads", [1, 4, 8])
@pytest.mark.parametrize("small", [True, False])
def test_text_weight_with_other_heads_than_the_layer(dev, monkeypatch, small, heads):
    """The text has as many key heads as linear_kv_xattn's weight (the layer has two), in a small layer and where the text alone
    would go in one launch."""
    layer, run, _ = _layer_case(dev, 256, 1, 5, 9, 2, 1, "append", False, [33, 20])
    layer.linear_kv_xattn = torch.nn.Linear(256, 2 * heads * D, bias=False, device=dev, dtype=torch.bfloat16)
    if not small:
        monkeypatch.setattr(MOD, "_projects_in_one_launch", lambda *a: False)
    got, _ = run()
    for name in ("_projects_in_one_launch", "_text_in_one_launch"):
        monkeypatch.setattr(MOD, name, lambda *a: False)
    want, _ = run()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,grid,dn,text", [(768, (2, 6, 10), 2, [24, 13]), (768, (2, 14, 15), 2, [40, 30]), (3072, (1, 9, 12), 1, [300])])
def test_captured_layers_take_the_launches_of_the_eager_pass(dev, monkeypatch, hidden, grid, dn, text):
    """An eager pass brings up what the capture needs, and no more: where it makes no product of the library, the capture makes none
    (the library cannot be brought up in a capture).  Every replay gives the eager bits."""
    layer, run, (hs, y, meta, rope) = _layer_case(dev, hidden, *grid, dn, 1, "none", False, text)
    products, linear = [], torch.nn.functional.linear
    monkeypatch.setattr(torch.nn.functional, "linear", lambda *a: products.append(a[1].shape) or linear(*a))
    want, n = run()
    eager = list(products)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.stream(side):
        layer(hs, y, None, rope, meta)
    torch.cuda.synchronize()
    products.clear()
    n0 = M.lib().magi_launch_count()
    with torch.no_grad(), torch.cuda.graph(graph):
        out = layer(hs, y, None, rope, meta)
    assert M.lib().magi_launch_count() - n0 == n and products == eager and len(eager) == (hidden == 3072)
    kept = hs.clone()
    for i in range(3):
        hs.copy_(kept * (2 if i == 1 else 1))
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, run()[0] if i == 1 else want))


def test_which_layers_take_the_one_launch():
    cus = 256
    one = MOD._projects_in_one_launch
    assert one(240, 20, 48, 4, 768, cus) and one(2048, 20, 1600, 4, 768, cus) and not one(3265, 20, 40, 4, 768, cus)
    assert one(380, 20, 100, 4, 1024, cus) and not one(400, 20, 100, 4, 1024, cus)  # (no taller workgroups there: one round)
    text = MOD._text_in_one_launch
    assert text(6e10, 512, 16, 3072, cus) and not text(6e10, 513, 16, 3072, cus) and text(6e10, 2048, 4, 768, cus)
    assert text(6e10, 65, 16, 3072, cus) and not text(6e10, 64, 16, 3072, cus) and text(6e10, 3, 4, 1024, cus)  # (where the library cuts K)
    assert not text(6e10, 100, 16, 6144, cus) and not text(8e10, 199, 16, 3072, cus) and text(8e10, 200, 16, 3072, cus)


def test_struct_layout_matches_header(tmp_path):
    fields = [f[0] for f in L.SmallProjArgs._fields_]
    src = ['#include <stdio.h>', '#include <stddef.h>', '#include "magi_attn.h"', 'int main(void){', 'printf("%zu\\n", sizeof(magi_small_proj_args));']
    src += ['printf("%%zu\\n", offsetof(magi_small_proj_args, %s));' % f for f in fields] + ['return 0;}']
    c, exe = tmp_path / "layout.c", tmp_path / "layout"
    c.write_text("\n".join(src))
    subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(c), "-o", str(exe)], check=True)
    out = [int(v) for v in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    assert out == [C.sizeof(L.SmallProjArgs)] + [getattr(L.SmallProjArgs, f).offset for f in fields]
