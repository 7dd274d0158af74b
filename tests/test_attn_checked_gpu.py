"""GPU tests of the bounded-score kernel that checks itself (MAGI_ATTN_CHECKED): on inputs whose scores are bounded it gives
the bits of the call with a stated bound; every 64-row block whose row sums leave the window is computed again with a
running maximum, whatever the reason (scores too large or too small, in the first tile or later, non-finite inputs)."""
import numpy as np
import pytest
import torch

import magi_attn as M
from oracle import magi_oracle as O

pytestmark = pytest.mark.gpu


def _ranges(dev, *arrs):
    return [torch.tensor(np.asarray(a), dtype=torch.int32, device=dev) for a in arrs]


def _close(out, ref):
    d = (out.float().cpu() - ref).abs()
    assert torch.isfinite(out).all() and d.max().item() <= 2e-2, d.max().item()


@pytest.mark.parametrize("L,dn,sp,Hq,Hkv", [(1, 3, 2, 6, 1), (64, 2, 1, 4, 2), (200, 3, 1, 6, 2), (333, 4, 3, 12, 4), (257, 2, 0, 3, 3)])
def test_bounded_inputs_give_the_bits_of_a_stated_bound(dev, L, dn, sp, Hq, Hkv):
    q, k, v = O.synthetic_qkv(dn * L, (sp + dn) * L, Hq, Hkv, 128, seed=L)
    qr, kr = O.q_ranges_for(dn, L), O.default_kvrange(sp, dn, L)
    tq, tk = _ranges(dev, qr, kr)
    qp = (q.float() * (128 ** -0.5 * 1.4426950408889634)).bfloat16().to(dev)
    kd, vd = k.to(dev), v.to(dev)
    n0 = M.lib().magi_launch_count()
    out, lse = M.range_attention(qp, kd, vd, tq, tk, L, checked=True, q_prescaled=True)
    assert M.lib().magi_launch_count() - n0 == 2
    want, lse_w = M.range_attention(qp, kd, vd, tq, tk, L, score_bound=17.0, q_prescaled=True)
    assert torch.equal(out, want) and torch.equal(lse, lse_w)
    # unscaled q: the scale is applied to the fp32 scores, q is not rounded a second time
    out, lse = M.range_attention(q.to(dev), kd, vd, tq, tk, L, checked=True)
    online, lse_o = M.range_attention(q.to(dev), kd, vd, tq, tk, L)
    _close(out, O.range_attention(q, k, v, qr, kr))
    assert (lse - lse_o).abs().max().item() <= 1e-3


@pytest.mark.parametrize("where", ["everywhere", "first tile", "late tile", "one row", "tiny sums", "side segment"])
@pytest.mark.parametrize("L,Tk", [(300, 700), (65, 64), (130, 1000)])
def test_blocks_outside_the_window_are_computed_again(dev, where, L, Tk):
    """Scores far above 64 (and, for tiny sums, all far below -64) in the places named, against the fp32 oracle; blocks
    around them stay right.  lse against the online-softmax kernel's: both sum fp32 probabilities."""
    Hq, Hkv = 4, 2
    g = torch.Generator().manual_seed(L + Tk)
    q = torch.randn(2 * L, Hq, 128, generator=g).bfloat16()
    k = torch.randn(Tk, Hkv, 128, generator=g).bfloat16()
    v = torch.randn(Tk, Hkv, 128, generator=g).bfloat16()
    split = None
    if where == "everywhere":
        q = (q.float() * 12).bfloat16()
    elif where == "first tile":  # the kernel starts with the last tile of the range
        k[-3, 1] *= 40
    elif where == "late tile":
        k[5, 0] *= 40
    elif where == "one row":
        q[L + 1, 2] *= 40
    elif where == "tiny sums":  # one direction shared by all keys, one query against it
        k[:, 0] = (k[:, 0].float() * 0.05 + 8.0).bfloat16()
        q[3, 0] = -8.0
    else:
        split = Tk // 2 + 3
        k[split + 2, 1] *= 40
    qr, kr = [[0, L], [L, 2 * L]], [[0, Tk], [0, Tk - 1]]
    tq, tk = _ranges(dev, qr, kr)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    kw = {} if split is None else dict(k2=kd[split:], v2=vd[split:], k_split=split)
    k1, v1 = (kd, vd) if split is None else (kd[:split], vd[:split])
    out, lse = M.range_attention(qd, k1, v1, tq, tk, L, checked=True, **kw)
    _close(out, O.range_attention(q, k, v, np.array(qr), np.array(kr)))
    online, lse_o = M.range_attention(qd, k1, v1, tq, tk, L, **kw)
    assert (lse - lse_o).abs().max().item() <= 1e-3 + 1e-6 * lse_o.abs().max().item()
    # pre-scaled q, output in groups of heads
    qp = (q.float() * (128 ** -0.5 * 1.4426950408889634)).bfloat16().to(dev)
    buf = torch.zeros(2 * L, 2, 2, 2, 128, dtype=torch.bfloat16, device=dev)
    M.range_attention(qp, k1, v1, tq, tk, L, checked=True, q_prescaled=True, out=buf[:, :, 0], return_lse=False, **kw)
    plain, _ = M.range_attention(qp, k1, v1, tq, tk, L, q_prescaled=True, **kw)
    assert (buf[:, :, 0].reshape(plain.shape).float() - plain.float()).abs().max().item() <= 2e-2  # (the same rounded q)
    assert torch.count_nonzero(buf[:, :, 1]) == 0


def test_non_finite_inputs_stay_where_they_belong(dev):
    L, Hq, Hkv = 200, 4, 2
    q, k, v = O.synthetic_qkv(2 * L, 2 * L, Hq, Hkv, 128, seed=3)
    k[7, 1, 5] = float("nan")
    q[L + 3, 0, 0] = float("inf")
    tq, tk = _ranges(dev, [[0, L], [L, 2 * L]], [[0, L], [L, 2 * L]])
    out, _ = M.range_attention(q.to(dev), k.to(dev), v.to(dev), tq, tk, L, checked=True)
    nan = torch.isnan(out).any(-1).cpu()
    want = torch.zeros_like(nan)
    want[:L, 2:] = True   # every row that sees the key with a NaN
    want[L + 3, 0] = True
    assert torch.equal(nan, want)


@pytest.mark.parametrize("size", [2.0 ** 83, 2.0 ** -83])
def test_values_of_any_size(dev, size):
    """Exponents around 52 or around -52 are within the kernel's, but not times values as large or as small as these: the
    accumulators would overflow or go subnormal.  Relative to the values, against the oracle."""
    L, Hq, Hkv = 150, 4, 2
    q, k, v = O.synthetic_qkv(2 * L, 300, Hq, Hkv, 128, seed=8)
    k[:, 0] = (k[:, 0].float() * 0.05 + 2.0).bfloat16()
    q[:, :2] = (q[:, :2].float() * 0.05 + (1.6 if size > 1 else -1.6)).bfloat16()
    qr, kr = np.array([[0, L], [L, 2 * L]]), np.array([[0, 300], [7, 299]])
    out, _ = M.range_attention(q.to(dev), k.to(dev), (v.float() * size).bfloat16().to(dev), *_ranges(dev, qr, kr), L, checked=True)
    _close(out.float() / size, O.range_attention(q, k, v, qr, kr))


@pytest.mark.parametrize("Tk", [5, 70, 97])
def test_keys_past_the_end_stay_out_at_a_small_softmax_scale(dev, Tk):
    """The masked keys of a ragged tile take no part whatever the scale that the scores are multiplied by."""
    L, Hq, Hkv = 70, 2, 1
    q, k, v = O.synthetic_qkv(L, Tk, Hq, Hkv, 128, seed=Tk)
    tq, tk = _ranges(dev, [[0, L]], [[0, Tk]])
    for scale in (1e-3, 1e-6):
        out, lse = M.range_attention(q.to(dev), k.to(dev), v.to(dev), tq, tk, L, softmax_scale=scale, checked=True)
        online, lse_o = M.range_attention(q.to(dev), k.to(dev), v.to(dev), tq, tk, L, softmax_scale=scale)
        assert (out.float() - online.float()).abs().max().item() <= 2e-2 and (lse - lse_o).abs().max().item() <= 1e-3


def test_many_ranges_empty_ranges_and_gaps(dev):
    """More ranges than one wavefront (and than the workgroup) ranks, some without keys, some rows in no range."""
    for n in (3, 65, 300):
        g = torch.Generator().manual_seed(n)
        lens = torch.randint(0, 70, (n,), generator=g).numpy()
        starts = np.concatenate([[0], np.cumsum(lens + 3)])
        qr = np.stack([starts[:-1], starts[:-1] + lens], 1)
        ks = torch.randint(0, 300, (n,), generator=g).numpy()
        kr = np.stack([ks, ks + np.where(np.arange(n) % 4 == 1, 0, 90)], 1)
        Tq = int(starts[-1]) + 2
        q, k, v = O.synthetic_qkv(Tq, 400, 3, 1, 128, seed=n)
        q[::7] = (q[::7].float() * 12).bfloat16()
        ref = O.range_attention(q, k, v, qr, kr)
        out, _ = M.range_attention(q.to(dev), k.to(dev), v.to(dev), *_ranges(dev, qr, kr), 70, checked=True)
        _close(out, ref)


@pytest.mark.parametrize("gain", [1.0, 2.0, 40.0])
@pytest.mark.parametrize("L,n,cu_k", [(2600, 4, [0, 130, 130, 390, 520]),  # short key ranges, one of them empty
                                      (1536, 3, [0, 1536, 3072, 4608])])
def test_reference_shaped_callables_round_relative_to_the_maximum(dev, L, n, cu_k, gain):
    """varlen, flex and flash calls that promise nothing about the scores give the online softmax's bits in its one launch, also
    where 256-row workgroups would fill the chip.  The probability of a row's largest score is then 1 exactly, which the
    checked kernel rounds: it is further from float64 than these calls may be."""
    Hq, Hkv, D = 24, 8, 128
    q, k, v = (t.to(dev) for t in O.synthetic_qkv(n * L, cu_k[-1], Hq, Hkv, D, seed=9))
    q = (q.float() * gain).bfloat16()
    cq = torch.arange(0, (n + 1) * L, L, dtype=torch.int32, device=dev)
    ck = torch.tensor(cu_k, dtype=torch.int32, device=dev)
    qr, kr = torch.stack([cq[:-1], cq[1:]], 1).contiguous(), torch.stack([ck[:-1], ck[1:]], 1).contiguous()
    online, lse = M.range_attention(q, k, v, qr, kr, L)
    calls = [lambda: M.flash_attn_varlen_func(q, k, v, cq, ck, L, 800), lambda: M.flex_flash_attn_func(q, k, v, qr, kr, L, 800)[0]]
    if len(set(np.diff(cu_k))) == 1:
        calls.append(lambda: M.flash_attn_func(*(t.view(n, -1, t.shape[1], D) for t in (q, k, v))).view(n * L, Hq, D))
    for call in calls:
        n0 = M.lib().magi_launch_count()
        out = call()
        assert M.lib().magi_launch_count() - n0 == 1 and torch.equal(out, online)
    if gain > 2:
        return
    checked, _ = M.range_attention(q, k, v, qr, kr, L, checked=True)
    sel = torch.arange(0, L, 13, device=dev)
    k64, v64 = (t[:cu_k[1]].double().repeat_interleave(Hq // Hkv, 1).transpose(0, 1) for t in (k, v))
    want = (torch.softmax(q[sel].double().transpose(0, 1) @ k64.transpose(1, 2) * D ** -0.5, -1) @ v64).transpose(0, 1)
    err = lambda x: ((x[sel].double() - want).norm() / want.norm()).item()
    assert err(online) < err(checked), (err(online), err(checked))


def test_checked_argument_checks(dev):
    q = torch.zeros(8, 2, 128, dtype=torch.bfloat16, device=dev)
    r = torch.tensor([[0, 8]], dtype=torch.int32, device=dev)
    for kw in ({"score_bound": 10.0}, {"auto_bound": True}, {"q_tile_rows": 128}, {"static_scratch": True}):
        with pytest.raises(M.MagiError):
            M.range_attention(q, q, q, r, r, 8, checked=True, **kw)
