"""The reference's fp8 linear layers in front of the prologue (inference/model/dit/dit_module.py:364-384 div_clamp_to,
:431-456 PerTensorQuantizedFp8Linear; q / qx / k / v of every layer but the first and the last under fp8_quant,
:405-409).

The input quantiser is integer-exact work: bit-identical to the oracle's restatement of div_clamp_to, bf16
intermediate included.  The GEMM behind it is the library's fp8 GEMM (fp32 accumulation of exact e4m3 products), so
the layer is compared with fp32 arithmetic on the de-quantised operands to one rounding of the bf16 result."""
import pytest
import torch

import magi_attn as M
from magi_attn import module as MOD
from oracle import magi_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,per_column", [(1000, 6144, False), (333, 3072, True), (5, 8, False), (4099, 1536, True),
                                                  (1, 520, False)])
def test_div_clamp_to_bit_exact_with_oracle(dev, rows, cols, per_column):
    g = torch.Generator().manual_seed(rows + cols)
    x = (torch.randn(rows, cols, generator=g) * 3.0).bfloat16()
    x[0, :8] = torch.tensor([0.0, -0.0, 1e-30, 1e30, -1e30, 447.0, 449.0, float("nan")]).bfloat16()
    scale = (torch.rand(cols if per_column else 1, generator=g) * 0.02 + 0.003)
    y = M.div_clamp_to(x.to(dev), scale.to(dev))
    ref = O.quantize_e4m3(x, scale, via_bf16=True)
    gb, rb = y.cpu().view(torch.uint8), ref.view(torch.uint8)
    nan = torch.isnan(x.float())
    assert torch.equal(gb[~nan], rb[~nan])
    assert torch.all((gb[nan] & 0x7f) == 0x7f)  # a NaN stays a NaN
    # saturation at +-448 and the double rounding: values that a direct conversion would round the other way exist
    direct = O.quantize_e4m3(x, scale, via_bf16=False).view(torch.uint8)
    assert y.float().abs()[~nan.to(dev)].max() <= 448
    if rows * cols > 100000:
        assert (direct[~nan] != rb[~nan]).any(), "the bf16 intermediate must matter somewhere in a sample this large"


def test_div_clamp_to_strided_rows_leading_axes_and_checks(dev):
    g = torch.Generator().manual_seed(3)
    wide = torch.randn(77, 2 * 512, generator=g).bfloat16()
    sc = torch.tensor([0.01])
    y = M.div_clamp_to(wide.to(dev)[:, 512:], sc.to(dev))
    assert torch.equal(y.cpu().view(torch.uint8), O.quantize_e4m3(wide[:, 512:], sc, via_bf16=True).view(torch.uint8))
    x3 = torch.randn(20, 3, 256, generator=g).bfloat16()
    y3 = M.div_clamp_to(x3.to(dev), sc.to(dev))
    assert y3.shape == x3.shape
    assert torch.equal(y3.cpu().view(torch.uint8), O.quantize_e4m3(x3, sc, via_bf16=True).view(torch.uint8))
    with pytest.raises(TypeError):
        M.div_clamp_to(x3.float().to(dev), sc.to(dev))
    with pytest.raises(ValueError):
        M.div_clamp_to(x3.to(dev), torch.ones(7, device=dev))
    with pytest.raises(M.MagiError):
        M.div_clamp_to(torch.zeros(4, 12, dtype=torch.bfloat16, device=dev), sc.to(dev))  # cols % 8


def test_per_tensor_fp8_linear_matches_dequantised_arithmetic(dev):
    torch.manual_seed(5)
    S, K, N = 640, 1024, 768
    lin = torch.nn.Linear(K, N, bias=False, dtype=torch.bfloat16, device=dev)
    x = (torch.randn(S, 1, K, device=dev) * 1.3).bfloat16()
    q = MOD.PerTensorQuantizedFp8Linear.from_linear(lin, x.float().abs().max().item())
    assert q.weight.shape == (1, N, K) and q.weight.dtype == torch.float8_e4m3fn
    assert q.weight_scale.shape == (1,) and q.input_scale.shape == (K,)
    y = q(x)
    assert y.shape == (S, 1, N) and y.dtype == torch.bfloat16
    x8 = O.quantize_e4m3(x.cpu(), q.input_scale.cpu(), via_bf16=True).float().view(S, K)
    ref = (x8.double() @ q.weight[0].float().cpu().double().t()) * q.input_scale[0].item() * q.weight_scale.item()
    d = (y.view(S, N).double().cpu() - ref).abs()
    assert torch.all(d <= ref.abs() * 2.0 ** -7 + 1e-3)  # one bf16 rounding of an fp32-accumulated sum
    # and it approximates the bf16 layer it was made from to e4m3 precision
    full = torch.nn.functional.linear(x, lin.weight).float().view(S, N).cpu()
    cos = torch.nn.functional.cosine_similarity(y.view(S, N).float().cpu().flatten(), full.flatten(), dim=0).item()
    assert cos >= 0.998, cos


@pytest.mark.parametrize("rows,cols,params,kinds", [
    (1, 8, "bf16", "r"), (17, 520, "fp32", "rs"), (300, 1024, "none", "tttt"), (4100, 3072, "bf16", "rrtt"),
    (515, 6144, "bf16", "rtrs"), (33, 8192, "weight", "sr"), (40, 1536, "bf16", "xrx"), (16 * 256 + 5, 256, "bf16", "trtr")])
def test_norm_and_quantisers_in_one_launch_give_the_same_bytes(dev, rows, cols, params, kinds):
    """layer_norm_div_clamp against layer_norm and one div_clamp_to per scale: every byte the same, for random scales (r),
    scales whose quotients fall on and next to the middle between two bf16 values (t), one scale for all columns (s),
    and scales outside the range the reciprocal serves (x: subnormal, zero, infinite, NaN, huge)."""
    g = torch.Generator(device=dev).manual_seed(rows + cols)
    x = (torch.randn(rows, cols, device=dev, generator=g) * 2 + 0.3).bfloat16()
    if rows > 20:
        x[3, 5] = float("nan")
        x[7] = 0.0
    p_dtype = torch.float32 if params == "fp32" else torch.bfloat16
    w = None if params == "none" else (torch.rand(cols, device=dev, generator=g) + 0.5).to(p_dtype)
    b = None if params in ("none", "weight") else (torch.randn(cols, device=dev, generator=g) * 0.3).to(p_dtype)
    scales = []
    for kind in kinds:
        s = torch.rand(cols, device=dev, generator=g) * 0.02 + 0.003
        if kind == "s":
            s = torch.full((cols,), 6.0 / 448.0, device=dev)
        elif kind == "t":
            step = torch.randint(-3, 4, (cols,), device=dev, generator=g)
            s = (1.0 / ((1 + 2.0 ** -8) * 2.0 ** (step + 5).float())).view(torch.int32).add_(step.int()).view(torch.float32)
        elif kind == "x":
            odd = torch.tensor([1e-40, 0.0, float("inf"), float("nan"), 3e38, 1e-38, -0.01], device=dev)
            s[:cols:5] = odd[torch.arange(len(s[:cols:5]), device=dev) % 7]
        scales.append(s.contiguous())
    if kinds == "trtr":
        scales[2:] = [t.clone() for t in scales[:2]]  # equal pairs are converted once
    n0 = M.lib().magi_launch_count()
    got = M.layer_norm_div_clamp(x, w, b, scales, 1e-6)
    assert M.lib().magi_launch_count() - n0 == 1
    h = M.layer_norm(x, w, b, 1e-6)
    for k, s in enumerate(scales):
        want = M.div_clamp_to(h, s).view(torch.uint8)
        bytes_ = got[k].view(torch.uint8)
        nan = (want & 0x7f) == 0x7f
        assert torch.equal(bytes_[~nan], want[~nan]) and bool(((bytes_[nan] & 0x7f) == 0x7f).all())


def test_rows_of_whole_rounds_ahead_of_the_rest(dev, monkeypatch):
    """forward_quantized cuts the rows behind whole rounds of tiles in two calls of the library and has their bits (256 CUs: 16384 rows are one
    round at 1024 columns); one call where the rest is long, a gradient is asked for or the tensor is another class.  One call for all rows
    may add in another order, in fp32: 1024 terms, 2^-14 of their size at most, and a bf16 step."""
    K, N, rows = 1024, 1024, 16384 + 300
    m = MOD.PerTensorQuantizedFp8Linear(K, N, device=dev)
    m.weight.data = (torch.randn(1, N, K, device=dev) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    m.weight_scale.data.fill_(0.02)
    m.input_scale.data.fill_(0.01)
    x8 = (torch.randn(rows, K, device=dev) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    calls, product = [], torch._scaled_mm
    monkeypatch.setattr(torch, "_scaled_mm", lambda x, *a, **k: calls.append(x.shape[0]) or product(x, *a, **k))
    monkeypatch.setattr(MOD, "_compute_units", lambda device: 256)
    y = m.forward_quantized(x8)
    assert calls == [16384, 300] and y.shape == (rows, N) and y.dtype == torch.bfloat16
    of = lambda t: product(t, m.weight[0].t(), scale_a=m.input_scale[:1], scale_b=m.weight_scale, out_dtype=torch.bfloat16)
    want, whole = torch.cat([of(x8[:16384]), of(x8[16384:])]), of(x8)
    assert torch.equal(y, want)
    assert torch.allclose(y.float(), whole.float(), rtol=2.0 ** -7, atol=2.0 ** -14 * whole.float().abs().max().item())
    calls.clear()
    assert torch.equal(m.forward_quantized(x8.view(2, rows // 2, K)), want.view(2, rows // 2, N)) and calls == [16384, 300]
    calls.clear()
    m.forward_quantized(x8[:16384])
    m.weight_scale.requires_grad_(True)
    m.forward_quantized(x8)
    with torch.no_grad():
        m.forward_quantized(x8)
    assert calls == [16384, rows, 16384, 300]


@pytest.mark.parametrize("how", ["vmap", "jit.trace", "make_fx"])
def test_products_that_are_cut_under_transforms(dev, how):
    """vmap has no batched form of a product with out=, and a recorded one is run with other numbers of rows: one call for all rows there.
    (Of 1024 terms in another order, fp32 sums: 2^-14 of their size at most, and a bf16 step.)"""
    K, N, rows = 1024, 1024, 16384 + 300
    m = MOD.PerTensorQuantizedFp8Linear(K, N, device=dev)
    m.weight.data = (torch.randn(1, N, K, device=dev) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    x8 = (torch.randn(2, rows, K, device=dev) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    w = torch.randn(2048, K, device=dev, dtype=torch.bfloat16)  # (8 columns of tiles: 8192 rows are a round)
    for f, x in ((lambda t: m.forward_quantized(t), x8), (lambda t: MOD._linear_in_whole_rounds(t, w), torch.randn(2, 8192 + 300, K, device=dev, dtype=torch.bfloat16))):
        with torch.no_grad():
            want = torch.stack([f(x[0]), f(x[1])])
            if how == "vmap":
                got = torch.vmap(f)(x)
            else:
                from torch.fx.experimental.proxy_tensor import make_fx
                recorded = torch.jit.trace(f, (x[0],), check_trace=False) if how == "jit.trace" else make_fx(f)(x[0])
                got = torch.stack([recorded(t) for t in x])
                for n in (96, x.shape[1] + 96):
                    more = x.reshape(-1, K)[:n]
                    assert torch.allclose(recorded(more).float(), f(more).float(), rtol=2.0 ** -7, atol=2.0 ** -14 * want.float().abs().max().item())
        assert torch.allclose(got.float(), want.float(), rtol=2.0 ** -7, atol=2.0 ** -14 * want.float().abs().max().item())


def test_products_that_are_cut_under_graph_capture(dev):
    """Replays, with eager work between them, against the eager products: e4m3 and bf16."""
    K, N, rows = 1024, 1024, 16384 + 300
    m = MOD.PerTensorQuantizedFp8Linear(K, N, device=dev)
    m.weight.data = (torch.randn(1, N, K, device=dev) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    w = torch.randn(2048, K, device=dev, dtype=torch.bfloat16)
    draw8 = lambda: (torch.randn(rows, K, device=dev) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    draw16 = lambda: torch.randn(8192 + 300, K, device=dev, dtype=torch.bfloat16)
    x8, x16 = draw8(), draw16()
    both = lambda: (m.forward_quantized(x8), MOD._linear_in_whole_rounds(x16, w))
    with torch.no_grad():
        both()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = both()
        for _ in range(4):
            x8.view(torch.uint8).copy_(draw8().view(torch.uint8))
            x16.copy_(draw16())
            want = both()
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(out, want))


def test_projections_hold_no_more_memory_than_norm_and_quantisers_apart(dev):
    """The e4m3 inputs of the four linears are given back one by one: the most that is held is below the outputs, the norm's
    bf16 rows and one e4m3 input, which is what separate calls hold."""
    rows, K, q, kv = 4096, 1024, 2048, 512
    c = MOD.CustomLayerNormLinear(K, q, kv, device=dev, fp8_quant=True)
    x = torch.randn(rows, 1, K, device=dev).bfloat16()
    with torch.no_grad():
        want = tuple(m(c.forward_ln(x)).view(rows, -1) for m in c._projections())
        c.forward_ln_qkvx_rows(x)  # (the library's workspace is there from here on)
        torch.cuda.synchronize()
        base = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        got = c.forward_ln_qkvx_rows(x)
        peak = torch.cuda.max_memory_allocated() - base
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert peak <= 2 * rows * (2 * q + 2 * kv) + 3 * rows * K, peak


def test_layer_with_fp8_quant_projections(dev):
    """FullyParallelAttention(fp8_quant=True): q / qx / k / v through PerTensorQuantizedFp8Linear.  Against the same
    layer with bf16 projections made of the DE-QUANTISED weights, fed the same inputs: the only difference left is the
    e4m3 rounding of the normalised input (2.7 % per element, averaged over hidden-size products per output), so
    the attention outputs agree to cosine >= 0.999."""
    from magi_attn import params as P
    from magi_attn import ranges as R
    from magi_attn.rope import LearnableRotaryEmbeddingCat

    hidden, Hq, Hkv, D = 256, 8, 2, 128
    fr, H, W, dn = 2, 3, 4, 2
    L = fr * H * W
    S = dn * L
    torch.manual_seed(9)
    ref = MOD.FullyParallelAttention(hidden, Hq, Hkv, layer_number=1, device=dev)
    with torch.no_grad():
        for p in ref.parameters():
            p.copy_(torch.randn_like(p.float()) * (0.1 if p.dim() == 1 else hidden ** -0.5))
        ref.linear_qkv.layer_norm.weight.add_(1.0)
    q8 = MOD.FullyParallelAttention(hidden, Hq, Hkv, layer_number=1, device=dev, fp8_quant=True)
    sd = {k: v for k, v in ref.state_dict().items() if not k.startswith(("linear_qkv.q.", "linear_qkv.qx.", "linear_qkv.k.", "linear_qkv.v."))}
    q8.load_state_dict(sd, strict=False)
    for name in ("q", "qx", "k", "v"):
        lin = getattr(ref.linear_qkv, name)
        fq = MOD.PerTensorQuantizedFp8Linear.from_linear(lin, 6.0)  # normalised hidden states: |x| < 6
        setattr(q8.linear_qkv, name, fq)
        with torch.no_grad():  # the reference layer continues with the de-quantised weights
            lin.weight.copy_((fq.weight[0].float() * fq.weight_scale).to(lin.weight.dtype))
    g = torch.Generator().manual_seed(10)
    hs = torch.randn(S, 1, hidden, generator=g).bfloat16().to(dev)
    lens = torch.tensor([5, 8])
    mask = (torch.arange(8)[None] < lens[:, None]).float().view(dn, 1, 1, 8)
    y = (torch.randn(int(lens.sum()), hidden, generator=g) * 0.5).bfloat16().to(dev)
    kr = R.generate_kv_range_for_uncondition(dn, L)
    meta = P.ModelMetaArgs(H=H, W=W, cp_pad_size=None, cp_split_sizes=None, slice_point=0, denoising_range_num=dn,
                           range_num=dn, extract_prefix_video_feature=False, fwd_extra_1st_chunk=False,
                           distill_nearly_clean_chunk=False, clip_token_nums=L, enable_cuda_graph=False,
                           core_attn_params=P.build_core_attn_params(R.q_ranges_from_chunks(dn, L).to(dev), kr.to(dev), L),
                           cross_attn_params=P.build_cross_attn_params(mask.to(dev), L, 8))
    rope = LearnableRotaryEmbeddingCat(128, device=dev).get_embed_for_forward(dn * fr, H, W, 0, dn)
    with torch.no_grad():
        c0, x0 = ref(hs, y, None, rope, meta)
        c1, x1 = q8(hs, y, None, rope, meta)
    for a, b, nm in ((c1, c0, "core"), (x1, x0, "cross")):
        cos = torch.nn.functional.cosine_similarity(a.float().flatten(), b.float().flatten(), dim=0).item()
        assert torch.isfinite(a).all() and cos >= 0.999, (nm, cos)
