"""GPU tests of launches whose last round of items is shared by several workgroups each (magi_attn_args.split_workspace): the
pieces' fp32 sums, added up, give what one workgroup gives, up to the order of the additions."""
import pytest
import torch

import magi_attn as M
from magi_attn import _lib as L
from oracle import magi_oracle as O

pytestmark = pytest.mark.gpu

PRE = 128 ** -0.5 * 1.4426950408889634


def _inputs(dev, Tq, Tk, Hq, Hkv, seed):
    q, k, v = O.synthetic_qkv(Tq, Tk, Hq, Hkv, 128, seed=seed)
    return q.to(dev), k.to(dev), v.to(dev)


def _same_but_for_the_order(a, b, lse_a, lse_b):
    """fp32 sums of at most 2^13 terms in another order differ by a few 2^-24 of the sum of the terms' sizes (values of about 1,
    outputs of about 0.05): far less than half a bf16 step, so elements differ by one such step at most, or where they
    are near 0 by 1e-5."""
    d = (a.float() - b.float()).abs()
    assert torch.isfinite(a).all() and (d <= b.float().abs() * 2.0 ** -7 + 1e-5).all(), d.max().item()
    fin = torch.isfinite(lse_b)
    assert torch.equal(fin, torch.isfinite(lse_a)) and (lse_a - lse_b)[fin].abs().max().item() <= 1e-5


# (rows per range, ranges, cached ranges, heads, max_seqlen_k): equal pieces, two unequal ones behind whole rounds, odd head counts
# (padding in the grid), ranges with fewer keys than the launch was sized for (down to fewer tiles than pieces), none at all
CASES = [(500, 2, 2, 6, 2, 0), (257, 1, 8, 3, 1, 0), (64, 3, 40, 12, 4, 0), (9000, 1, 0, 24, 8, 0), (700, 2, 8, 24, 8, 0),
         (300, 4, 0, 5, 5, 4000), (1, 1, 4096, 1, 1, 0), (2000, 2, 3, 24, 8, 0)]


@pytest.mark.parametrize("mode", ["bounded", "scaled", "norm", "checked", "auto"])
@pytest.mark.parametrize("rows,n,sp,Hq,Hkv,max_k", CASES)
def test_split_items_give_what_whole_ones_give(dev, rows, n, sp, Hq, Hkv, max_k, mode):
    Tk = (sp + n) * rows
    mk = max_k or Tk
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert cus != 256 or L.lib().magi_attn_split_bytes(Hq, Hkv, n, rows, mk, L.MAGI_DTYPE_BF16) > 0
    q, k, v = _inputs(dev, n * rows + 7, Tk, Hq, Hkv, seed=rows + n)
    qr = torch.tensor([[i * rows, (i + 1) * rows] for i in range(n)], dtype=torch.int32, device=dev)
    kr = torch.tensor([[0, (sp + 1 + i) * rows] for i in range(n)], dtype=torch.int32, device=dev)
    if max_k:
        kr[0] = kr[0, 0]  # no keys
        kr[1, 1] = 3
    kw = {"bounded": {"q_prescaled": True, "score_bound": 40.0}, "scaled": {"score_bound": 40.0}, "checked": {"checked": True},
          "norm": {"score_bound": 40.0, "q_norm": (torch.zeros(128, device=dev), None, 1e-6)}, "auto": {"auto_bound": True}}[mode]
    if mode == "bounded":
        q = (q.float() * PRE).bfloat16()
    n0 = M.lib().magi_launch_count()
    a, la = M.range_attention(q, k, v, qr, kr, rows, mk, **kw)
    n1 = M.lib().magi_launch_count()
    b, lb = M.range_attention(q, k, v, qr, kr, rows, mk, split_keys=False, **kw)
    assert n1 - n0 == M.lib().magi_launch_count() - n1 + (1 if cus == 256 else 0)
    _same_but_for_the_order(a, b, la, lb)
    assert torch.equal(a, M.range_attention(q, k, v, qr, kr, rows, mk, **kw)[0])  # whatever order the pieces end in
    if rows == 500 and mode != "norm":  # (the oracle takes normed q)
        ref = O.range_attention((q.float() / PRE if mode == "bounded" else q).bfloat16().cpu(), k.cpu(), v.cpu(), qr.cpu().numpy(), kr.cpu().numpy())
        assert (a[:n * rows].float().cpu() - ref[:n * rows]).abs().max().item() <= 2e-2


@pytest.mark.parametrize("where", ["everywhere", "first piece", "last piece", "tiny sums", "large values", "side segment"])
def test_split_blocks_outside_the_window_are_computed_again(dev, where):
    rows, Hq, Hkv, Tk = 300, 4, 2, 3000
    q, k, v = _inputs(dev, 2 * rows, Tk, Hq, Hkv, seed=11)
    k2 = v2 = None
    split = Tk
    if where == "everywhere":
        q = (q.float() * 30).bfloat16()
    elif where == "first piece":
        k[2, 1] *= 60
    elif where == "last piece":
        k[-3, 0] *= 60
    elif where == "tiny sums":
        k[:, 0] = (k[:, 0].float() * 0.05 + 8.0).bfloat16()
        q[3, 0] = -8.0
    elif where == "large values":
        v[:, 1] *= 2.0 ** 100
    else:
        split = 1501
        k[split + 5, 1] *= 60
    qr = torch.tensor([[0, rows], [rows, 2 * rows]], dtype=torch.int32, device=dev)
    kr = torch.tensor([[0, Tk], [0, Tk - 1]], dtype=torch.int32, device=dev)
    kw = {}
    kc, vc = k, v
    if split < Tk:
        kc, vc = k[:split].contiguous(), v[:split].contiguous()
        kw = {"k2": k[split:].contiguous(), "v2": v[split:].contiguous(), "k_split": split}
    n0 = M.lib().magi_launch_count()
    a, la = M.range_attention(q, kc, vc, qr, kr, rows, Tk, checked=True, **kw)
    n1 = M.lib().magi_launch_count() - n0
    b, lb = M.range_attention(q, kc, vc, qr, kr, rows, Tk, **kw)
    assert n1 == 3 or torch.cuda.get_device_properties(dev).multi_processor_count != 256
    # probabilities are rounded to bf16 relative to different maxima: 2^-8 each, of sums of values of the column's size
    scale = v.float().abs().amax(dim=(0, 2)).repeat_interleave(Hq // Hkv)[None, :, None]
    assert torch.isfinite(a).all() and ((a.float() - b.float()).abs() <= 2.0 ** -7 * scale).all()
    assert (la - lb).abs().max().item() <= 1e-3


def test_a_workspace_that_is_too_small_leaves_the_items_whole(dev, monkeypatch):
    q, k, v = _inputs(dev, 256, 4096, 2, 1, seed=5)
    qr = torch.tensor([[0, 256]], dtype=torch.int32, device=dev)
    kr = torch.tensor([[0, 4096]], dtype=torch.int32, device=dev)
    call = lambda **kw: M.range_attention(q, k, v, qr, kr, 256, 4096, score_bound=40.0, **kw)[0]
    whole = call(split_keys=False)
    real = L.lib().magi_attn_split_bytes
    monkeypatch.setattr(L.lib(), "magi_attn_split_bytes", lambda *a: max(real(*a) - 1, 16))
    n0 = M.lib().magi_launch_count()
    assert torch.equal(call(), whole) and M.lib().magi_launch_count() - n0 == 1


def test_short_memory_is_an_error_and_not_another_order_of_the_sums(dev, monkeypatch):
    q, k, v = _inputs(dev, 256, 4096, 2, 1, seed=5)
    qr = torch.tensor([[0, 256]], dtype=torch.int32, device=dev)
    kr = torch.tensor([[0, 4096]], dtype=torch.int32, device=dev)
    if not L.lib().magi_attn_split_bytes(2, 1, 1, 256, 4096, L.MAGI_DTYPE_BF16):
        pytest.skip("not split on this card")
    real = torch.empty

    def empty(*size, dtype=None, **kw):
        if dtype is torch.uint8:
            raise torch.OutOfMemoryError("no scratch memory")
        return real(*size, dtype=dtype, **kw)

    monkeypatch.setattr(torch, "empty", empty)
    with pytest.raises(torch.OutOfMemoryError):
        M.range_attention(q, k, v, qr, kr, 256, 4096, score_bound=40.0)
    M.range_attention(q, k, v, qr, kr, 256, 4096, score_bound=40.0, split_keys=False)


def _exact(q, k, v, kr, rows):
    """float64 attention of q (scale and log2(e) folded in) over the operands as given."""
    G = q.shape[1] // k.shape[1]
    out = []
    for i, (b, e) in enumerate(kr):
        kk, vv = (t[b:e].double().repeat_interleave(G, 1).transpose(0, 1) for t in (k, v))
        p = torch.softmax(q[i * rows:(i + 1) * rows].double().transpose(0, 1) @ kk.transpose(1, 2) * 0.6931471805599453, -1)
        out.append((p @ vv).transpose(0, 1))
    return torch.cat(out)


@pytest.mark.parametrize("pow2", [True, False])
@pytest.mark.parametrize("rows,n,sp,Hq,Hkv,chunk,split", [(1300, 1, 12, 80, 8, 1300, None), (1300, 2, 12, 50, 5, 650, 9000),
                                                          (129, 13, 150, 64, 8, 129, None)])
def test_split_items_of_the_fp8_kernel(dev, rows, n, sp, Hq, Hkv, chunk, split, pow2):
    """e4m3 operands with a scale per (chunk, head), cuts inside and at the ends of scale chunks, two key segments: the split launch
    is as near to float64 on the same operands as the whole one (both round the probabilities to e4m3: 2^-4 each at most)."""
    Tk, f8 = (sp + n) * rows, torch.float8_e4m3fn
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert cus != 256 or L.lib().magi_attn_split_bytes(Hq, Hkv, n, rows, Tk, L.MAGI_DTYPE_FP8_E4M3) > 0
    q, k, v = _inputs(dev, n * rows, Tk, Hq, Hkv, seed=rows)
    tab = lambda T, H, x: x * 2.0 ** torch.arange(((T + chunk - 1) // chunk) * H, device=dev).remainder(3).float().view(-1, H)
    qs, ks, vs = tab(n * rows, Hq, 2.0 ** -6), tab(Tk, Hkv, 2.0 ** -5), tab(Tk, Hkv, 2.0 ** -5)
    if not pow2:
        qs, ks, vs = qs * 1.1, ks * 0.9, vs * 1.2
    row = lambda s, T: s.repeat_interleave(chunk, 0)[:T, :, None]
    enc = lambda x, s: (x.float() / row(s, x.shape[0])).clamp(-448, 448).to(f8)
    q8, k8, v8 = enc(q * PRE if pow2 else q, qs), enc(k, ks), enc(v, vs)
    qr = torch.tensor([[i * rows, (i + 1) * rows] for i in range(n)], dtype=torch.int32, device=dev)
    ends = [(0, (sp + 1 + i) * rows - 5 * (i == n - 1)) for i in range(n)]
    kr = torch.tensor(ends, dtype=torch.int32, device=dev)
    kc, vc, kw = k8, v8, {}
    if split:
        kc, vc = k8[:split].contiguous(), v8[:split].contiguous()
        kw = {"k2": k8[split:].contiguous(), "v2": v8[split:].contiguous(), "k_split": split}
    call = lambda s: M.range_attention(q8, kc, vc, qr, kr, rows, Tk, q_scale=qs, k_scale=ks, v_scale=vs, scale_chunk_tokens=chunk,
                                       fp8_pow2_prescaled=pow2, split_keys=s, **kw)
    n0 = M.lib().magi_launch_count()
    a, la = call(True)
    assert M.lib().magi_launch_count() - n0 == (2 if cus == 256 else 1)
    b, lb = call(False)
    assert torch.equal(a, call(True)[0])
    heads = slice(0, Hq, max(1, Hq // 5))  # (float64 on a few heads)
    G = Hq // Hkv
    dq = (q8.float() * row(qs, q8.shape[0]))[:, heads] * (1.0 if pow2 else PRE)
    kv_heads = [h // G for h in range(Hq)][heads]
    dk, dv = ((t.float() * row(s, Tk))[:, kv_heads] for t, s in ((k8, ks), (v8, vs)))
    want = _exact(dq, dk, dv, ends, rows)
    err = lambda x: ((x[:, heads].double() - want).norm() / want.norm()).item()
    assert torch.isfinite(a).all() and err(a) <= 1.05 * err(b) + 1e-3 and err(b) <= 2.0 ** -4, (err(a), err(b))
    assert (la - lb).abs().max().item() <= 2e-2  # the row sums are of rounded probabilities too


def _fp8_call(dev, Tq, Tk, Hq, Hkv, qr, kr, max_q, **kw):
    """range_attention on e4m3 operands with power-of-two scales; -> call(split_keys, out=None), the de-quantised operands"""
    q, k, v = _inputs(dev, Tq, Tk, Hq, Hkv, seed=Tq)
    (q8, qs), (k8, ks), (v8, vs) = M.quantize_fp8(q, 1 << 20, PRE, True), M.quantize_fp8(k, 1 << 20, 1.0, True), M.quantize_fp8(v, 1 << 20, 1.0, True)
    deq = [x.float() * s[:1, :, None] for x, s in ((q8, qs), (k8, ks), (v8, vs))]
    return lambda split, out=None: M.range_attention(q8, k8, v8, qr, kr, max_q, Tk, q_scale=qs, k_scale=ks, v_scale=vs,
                                                     scale_chunk_tokens=1 << 20, fp8_pow2_prescaled=True, split_keys=split, out=out, **kw), deq


@pytest.mark.parametrize("kind", ["bounded", "checked", "again", "fp8"])
def test_rows_outside_the_ranges_of_split_items_are_cleared(dev, kind):
    """Gaps ahead of, between and behind ranges whose items are shared, and all of whose blocks are computed again; the memory of
    out and lse is poisoned."""
    if kind == "fp8":
        Tq, Tk, Hq, Hkv, max_q, spans = 1310, 16900, 80, 8, 1310, [(5, 1301)]
    else:
        Tq, Tk, Hq, Hkv, max_q, spans = 660, 3000, 4, 2, 330, [(20, 320), (345, 645)]
    qr = torch.tensor(spans, dtype=torch.int32, device=dev)
    kr = torch.tensor([[0, Tk]] * len(spans), dtype=torch.int32, device=dev)
    assert len(spans) * max_q >= Tq  # (what has the launch clear the gaps)
    if kind == "fp8":
        call, _ = _fp8_call(dev, Tq, Tk, Hq, Hkv, qr, kr, max_q)
    else:
        q, k, v = _inputs(dev, Tq, Tk, Hq, Hkv, seed=3)
        q = (q.float() * 30).bfloat16() if kind == "again" else q
        kw = {"score_bound": 40.0} if kind == "bounded" else {"checked": True}
        call = lambda split: M.range_attention(q, k, v, qr, kr, max_q, Tk, split_keys=split, **kw)
    res = []
    for split in (True, False):
        for t, n in ((torch.bfloat16, Tq * Hq * 128), (torch.float32, Hq * Tq)):
            poison = torch.full((n,), float("nan"), dtype=t, device=dev)
            del poison
        n0 = M.lib().magi_launch_count()
        res.append(call(split) + (M.lib().magi_launch_count() - n0,))
    (a, la, na), (b, lb, nb) = res
    assert na == nb + 1 or torch.cuda.get_device_properties(dev).multi_processor_count != 256
    done = torch.zeros(Tq, dtype=torch.bool, device=dev)
    for s, e in spans:
        done[s:e] = True
    for o, lse in ((a, la), (b, lb)):
        assert torch.isfinite(o).all() and (o[done].abs().sum(-1) > 0).all() and torch.count_nonzero(o[~done]) == 0
        assert (lse[:, ~done] == float("-inf")).all() and torch.isfinite(lse[:, done]).all()
    if kind in ("bounded", "checked"):
        _same_but_for_the_order(a, b, la, lb)


@pytest.mark.parametrize("kind", ["grouped", "grouped fp8", "batch"])
def test_split_items_write_grouped_and_batched_outputs(dev, kind):
    """The launch that adds the pieces up addresses the rows itself: two-level head strides, [position, batch] rows.  What lies
    between the rows stays."""
    fp8 = kind.endswith("fp8")
    rows, Tk, Hq, Hkv, n = (1300, 16900, 80, 8, 1) if fp8 else (300, 3000, 4, 2, 2)
    qr = torch.tensor([[i * rows, (i + 1) * rows] for i in range(n)], dtype=torch.int32, device=dev)
    kr = torch.tensor([[0, Tk - 9 * i] for i in range(n)], dtype=torch.int32, device=dev)
    if fp8:
        call, _ = _fp8_call(dev, rows, Tk, Hq, Hkv, qr, kr, rows)
    else:
        q, k, v = _inputs(dev, n * rows, Tk, Hq, Hkv, seed=4)
        if kind == "batch":
            q4 = q.view(n, rows, Hq, 128).transpose(0, 1).contiguous().transpose(0, 1)
            assert not q4.is_contiguous()
        call = lambda split, out=None: M.range_attention(q4 if kind == "batch" and split else q, k, v, qr, kr, rows, Tk, score_bound=40.0,
                                                         split_keys=split, out=out)
    n0 = M.lib().magi_launch_count()
    plain, lse = call(False)
    assert M.lib().magi_launch_count() - n0 == 1
    if kind == "batch":
        got, lse_g = call(True)
        assert got.transpose(0, 1).is_contiguous()
        got = got.reshape(plain.shape)
    else:
        both = torch.full((n * rows, 2, 2, Hq // 2, 128), 7.0, dtype=torch.bfloat16, device=dev)
        out, lse_g = call(True, both[:, :, 1])
        assert (both[:, :, 0] == 7.0).all()
        got = out.reshape(plain.shape)
    assert M.lib().magi_launch_count() - n0 == (3 if torch.cuda.get_device_properties(dev).multi_processor_count == 256 else 2)
    if fp8:  # (each rounds its probabilities to e4m3, 2^-4 at most, of columns of values of about 1)
        assert (got.float() - plain.float()).norm() <= 2.0 ** -4 * plain.float().norm() and (lse_g - lse).abs().max().item() <= 2e-2
    else:
        _same_but_for_the_order(got, plain, lse_g, lse)


def test_split_items_of_the_fp8_kernel_with_piecewise_linear_exponentials(dev):
    """MAGI_ATTN_FP8_FAST_EXP2: probabilities are off by -4 to +6.2 % each, by where their exponents lie, whole or in pieces: both
    within that of float64, the pieces no further than the whole rows, row sums within the two ends of each other."""
    rows, Tk, Hq, Hkv = 1300, 16900, 80, 8
    qr, kr = (torch.tensor([[0, n]], dtype=torch.int32, device=dev) for n in (rows, Tk))
    call, (dq, dk, dv) = _fp8_call(dev, rows, Tk, Hq, Hkv, qr, kr, rows, fp8_fast_exp2=True)
    n0 = M.lib().magi_launch_count()
    a, la = call(True)
    assert M.lib().magi_launch_count() - n0 == 2 or torch.cuda.get_device_properties(dev).multi_processor_count != 256
    b, lb = call(False)
    heads = [3, 41, 79]
    want = _exact(dq[:, heads], *(t[:, [h // (Hq // Hkv) for h in heads]] for t in (dk, dv)), [(0, Tk)], rows)
    err = lambda x: ((x[:, heads].double() - want).norm() / want.norm()).item()
    assert torch.isfinite(a).all() and err(a) <= 1.05 * err(b) + 1e-3 and err(b) <= 0.1, (err(a), err(b))
    assert (la - lb).abs().max().item() <= 0.102  # ln(1.062 / 0.96) and the roundings


@pytest.mark.parametrize("n,rows,mk,dtype,split", [
    (4, 1403, 7015, "bf16", False), (4, 1400, 9800, "bf16", True),  # a shortest range of 2 of 5 chunks, of 4 of 7
    (2, 7070, 14140, "bf16", False), (2, 3612, 10836, "bf16", True),  # of 1 of 2, of 2 of 3
    (3, 5781, 23124, "bf16", True), (3, 5781, 23122, "bf16", False),  # of half of the longest, of just less
    (4, 4644, 4644, "bf16", True),  # a batch: every range its own rows
    (4, 200, 12000, "bf16", True), (4, 200, 700, "bf16", False),  # no whole round: lengths do not matter, the time saved does
    (2, 1756, 5268, "bf16", False),  # but for several ranges in more than 5/8 of the slots: 42 of 64,
    (3, 1200, 9536, "bf16", False), (3, 1200, 9537, "bf16", True),  # 45 over 149 and 150 tiles,
    (2, 1383, 4149, "bf16", True), (1, 3500, 5268, "bf16", True),  # 36 of 64, and 42 of one range
    (2, 2131, 4262, "fp8", False), (2, 2131, 4264, "fp8", True),  # six items behind a round, of half of the longest and of more
    (4, 3830, 15320, "fp8", True)])
def test_which_launches_share_the_keys_of_several_ranges(dev, n, rows, mk, dtype, split):
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the sizes are chosen for 256 CUs")
    code = L.MAGI_DTYPE_BF16 if dtype == "bf16" else L.MAGI_DTYPE_FP8_E4M3
    assert (L.lib().magi_attn_split_bytes(24, 8, n, rows, mk, code) > 0) == split
