"""Bounded scores in launches of a few rows: the wavefronts of a workgroup share the keys of 32 rows (MAGI_ATTN_SHARE_WAVES); two calls in one
launch (magi_attn_fwd_two), in this form or in 256-row workgroups."""
import pytest
import torch

import magi_attn as M
from magi_attn import _lib as L
from magi_attn import functional as F

pytestmark = pytest.mark.gpu
D, PRE = 128, 128 ** -0.5 * 1.4426950408889634


def _case(dev, Hq, Hkv, q_ranges, k_ranges, Tq, k_split=None, mode="scaled", most_k=None, seed=0):
    """(call(**kw) -> (out, lse), the attention over |v|)"""
    g = torch.Generator(device=dev).manual_seed(seed + Tq)
    Tk = max(max(e for _, e in k_ranges), 1)
    q = torch.nn.functional.layer_norm(torch.randn(Tq, Hq, D, device=dev, generator=g, dtype=torch.bfloat16), (D,))
    kv = torch.randn(Tk, Hkv, 2 * D, device=dev, generator=g, dtype=torch.bfloat16)
    k, v = torch.nn.functional.layer_norm(kv[..., :D], (D,)), kv[..., D:].contiguous()
    qr, kr = (torch.tensor(r, dtype=torch.int32, device=dev) for r in (q_ranges, k_ranges))
    kw = {"score_bound": 20.0}
    if mode == "as it is":
        q, kw["q_prescaled"] = (q.float() * PRE).bfloat16(), True
    elif mode == "normed":
        kw["q_norm"] = tuple(torch.randn(D, device=dev, generator=g) * 0.1 for _ in range(2)) + (1e-6,)
    most_q = max(e - b for b, e in q_ranges)
    most_k = most_k or max(max(e - b for b, e in k_ranges), 1)

    def call(values=v, **o):
        parts = {}
        kk, vv = k, values
        if k_split is not None:
            parts = {"k2": k[k_split:].clone(), "v2": values[k_split:].clone(), "k_split": k_split}
            kk, vv = k[:k_split].clone(), values[:k_split].clone()
        return M.range_attention(q, kk, vv, qr, kr, most_q, most_k, **kw, **parts, **o)

    return call, call(v.abs(), split_keys=False)[0], L.lib().magi_attn_waves(Hq, Hkv, len(q_ranges), 0, most_q, most_k)


# a key, a slab of 32 and one more, a slab for every wavefront of four and one key more, 1024 and 1025 keys (four wavefronts, eight), more than one slab per
# wavefront; rows around 32; ranges without keys, of unequal length, in another order, rows in no range; two key segments, one with a slab in both
@pytest.mark.parametrize("mode", ["as it is", "scaled", "normed"])
@pytest.mark.parametrize("Hq,Hkv,Tq,q_ranges,k_ranges,k_split", [
    (1, 1, 1, [(0, 1)], [(0, 1)], None), (6, 2, 33, [(0, 33)], [(3, 35)], 20), (2, 2, 65, [(0, 32), (32, 65)], [(0, 33), (10, 139)], 64),
    (3, 1, 120, [(64, 120), (0, 60)], [(5, 5), (0, 128)], None), (6, 2, 40, [(0, 31)], [(0, 1024)], 1000), (6, 2, 31, [(0, 31)], [(0, 1025)], None),
    (24, 8, 70, [(0, 35), (35, 70)], [(7, 1290), (0, 257)], 512), (5, 5, 300, [(0, 150), (150, 300)], [(0, 3000), (0, 40)], 77), (24, 8, 420, [(0, 420)], [(0, 700)], None)])
def test_shared_keys_give_what_the_other_forms_give(dev, mode, Hq, Hkv, Tq, q_ranges, k_ranges, k_split):
    """The scores and probabilities are the same to the bit, fp32 sums of n terms in another order: within n 2^-24 of their absolute values'
    sum (`size`: the attention over |v|; n 2^-24 < 2^-12), and a bf16 step."""
    call, size, waves = _case(dev, Hq, Hkv, q_ranges, k_ranges, Tq, k_split, mode)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert waves == (8 if max(e - b for b, e in k_ranges) > 1024 else 4)
    want, lse_want = call(split_keys=False)
    n0 = M.lib().magi_launch_count()
    got, lse = call(share_waves=True)
    assert M.lib().magi_launch_count() - n0 == 1 and torch.isfinite(got).all()
    assert ((got.float() - want.float()).abs() <= size.float() * 2.0 ** -12 + want.float().abs() * 2.0 ** -7).all()
    fin = torch.isfinite(lse_want)
    assert torch.equal(fin, torch.isfinite(lse)) and (lse - lse_want)[fin].abs().max().item() <= 2e-5
    assert torch.equal(call(share_waves=True, split_keys=False)[0], want)  # (a row's bits are asked for)
    if Hq % 2 == 0:  # grouped outputs
        o = torch.full((Tq, 2, 2, Hq // 2, D), 3.0, device=dev, dtype=torch.bfloat16)
        call(share_waves=True, out=o[:, :, 1], clear_out=True)
        assert torch.equal(o[:, :, 1].reshape(Tq, Hq, D), got) and (o[:, :, 0] == 3.0).all()


# one key, a few, a whole slab; rows around a workgroup's 32 and two of them; a range without keys; rows in no range; two key segments
@pytest.mark.parametrize("mode", ["as it is", "scaled", "normed"])
@pytest.mark.parametrize("Hq,Hkv,Tq,q_ranges,k_ranges,k_split", [
    (1, 1, 1, [(0, 1)], [(0, 1)], None), (6, 2, 33, [(0, 33)], [(3, 34)], 20), (24, 8, 70, [(2, 66)], [(0, 32)], None), (6, 2, 65, [(0, 32), (32, 65)], [(7, 7), (0, 9)], 4)])
def test_one_slab_of_keys_has_the_bits_of_the_other_forms(dev, mode, Hq, Hkv, Tq, q_ranges, k_ranges, k_split):
    """By itself such a call takes those; in one launch with another one a wavefront of its workgroup has all of the keys, in the same order."""
    call, _, waves = _case(dev, Hq, Hkv, q_ranges, k_ranges, Tq, k_split, mode)
    want = call(split_keys=False)
    held = []
    one, got, other = call(share_waves=True), call(share_waves=True, held=held), call(share_waves=True, held=held)
    n0 = M.lib().magi_launch_count()
    F.launch_held(held)
    assert not waves or M.lib().magi_launch_count() - n0 == 1
    for o, lse in (one, got, other):
        assert torch.equal(o, want[0]) and torch.equal(lse, want[1])


# both small (four wavefronts; four and eight), one of them or both in other forms; the number of launches
@pytest.mark.parametrize("first,second,launches", [
    ((6, 2, [(0, 120), (120, 240)], [(0, 360), (0, 480)], 240), (6, 2, [(0, 240)], [(0, 30)], 240), 1),
    ((6, 2, [(0, 200)], [(0, 1500)], 200), (24, 8, [(0, 90)], [(0, 333)], 90), 1), ((24, 8, [(0, 90)], [(0, 333)], 90), (6, 2, [(0, 200)], [(0, 1500)], 200), 1),
    ((24, 8, [(0, 900)], [(0, 900)], 900), (6, 2, [(0, 50)], [(0, 70)], 50), 2), ((6, 2, [(0, 50)], [(0, 70)], 50), (24, 8, [(0, 900)], [(0, 900)], 900), 2),
    ((24, 8, [(0, 900)], [(0, 900)], 900), (24, 8, [(0, 800)], [(0, 400)], 800), 2)])
def test_two_calls_have_the_bits_of_each(dev, first, second, launches):
    calls = [_case(dev, *c, mode=mode)[0] for c, mode in ((first, "as it is"), (second, "normed"))]
    want = [call(share_waves=True) for call in calls]
    held = []
    got = [call(share_waves=True, held=held) for call in calls]
    n0 = M.lib().magi_launch_count()
    F.launch_held(held)
    assert not held and (M.lib().magi_launch_count() - n0 == launches or torch.cuda.get_device_properties(dev).multi_processor_count != 256)
    for (a, la), (b, lb) in zip(got, want):
        assert torch.equal(a, b) and torch.equal(la, lb)


# 256 rows to a workgroup in both: whole items; the last round's keys shared in the first (a launch more, for the sums), in the second (two calls);
# ranges without keys, rows in no range, two key segments; q as it is, raw or (no form for two) unscaled; the smaller one ahead; both orders of q's kinds
@pytest.mark.parametrize("first,second,modes,launches", [
    ((24, 8, [(0, 4200)], [(0, 700)], 4200), (24, 8, [(0, 4190)], [(0, 70)], 4190), ("as it is", "normed"), 1),
    ((24, 8, [(0, 4200)], [(0, 700)], 4201, 130), (24, 8, [(5, 4190)], [(3, 70)], 4195), ("normed", "as it is"), 1),
    ((24, 8, [(0, 3000), (3000, 6000)], [(0, 1500), (0, 3000)], 6000), (24, 8, [(0, 3000), (3000, 6001)], [(0, 1), (9, 9)], 6003), ("as it is", "normed"), 2),
    ((4, 1, [(0, 20000)], [(0, 300)], 20000), (24, 8, [(0, 3000), (3000, 6000)], [(0, 1500), (0, 3000)], 6000), ("normed", "as it is"), 3),
    ((24, 8, [(0, 4200)], [(0, 700)], 4200), (24, 8, [(0, 4190)], [(0, 70)], 4190), ("scaled", "normed"), 2),
    ((24, 8, [(0, 4200)], [(0, 700)], 4200), (24, 8, [(0, 4190)], [(0, 70)], 4190), ("as it is", "scaled"), 2),
    ((24, 8, [(0, 4200)], [(0, 700)], 4200), (6, 2, [(0, 300)], [(0, 70)], 300), ("as it is", "normed"), 2)])
def test_two_large_calls_have_the_bits_of_each(dev, first, second, modes, launches):
    calls = [_case(dev, *c, mode=m)[0] for c, m in zip((first, second), modes)]
    want = [call() for call in calls]
    held = []
    got = [call(held=held) for call in calls]
    n0 = M.lib().magi_launch_count()
    F.launch_held(held)
    assert M.lib().magi_launch_count() - n0 == launches or torch.cuda.get_device_properties(dev).multi_processor_count != 256
    for (a, la), (b, lb) in zip(got, want):
        assert torch.equal(a, b) and torch.equal(la, lb)
    del want
    graph, held = torch.cuda.CUDAGraph(), []
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        again = [call(return_lse=False, held=held)[0] for call in calls]
        F.launch_held(held)
    for _ in range(3):
        for t in again:
            t.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, (b, _) in zip(again, got))


def test_a_refused_second_call_raises_and_the_first_has_run(dev):
    call = _case(dev, 6, 2, [(0, 50)], [(0, 70)], 50)[0]
    held = []
    want, (got, _) = call(share_waves=True)[0], call(share_waves=True, held=held)
    call(share_waves=True, held=held)
    bad = list(held[1])
    args = L.AttnArgs.from_buffer_copy(bad[2])
    args.D = 64
    bad[2] = bytes(args)
    with pytest.raises(M.MagiError):
        F.launch_held([held[0], tuple(bad)])
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_captured_pairs_replay(dev):
    calls = [_case(dev, 6, 2, [(0, 100)], [(0, 480)], 100, mode="as it is")[0], _case(dev, 6, 2, [(0, 100)], [(0, 24)], 100, mode="normed")[0]]
    want = [call(share_waves=True, return_lse=False)[0] for call in calls]
    torch.cuda.synchronize()
    graph, held = torch.cuda.CUDAGraph(), []
    with torch.cuda.graph(graph):
        got = [call(share_waves=True, return_lse=False, held=held)[0] for call in calls]
        F.launch_held(held)
    for _ in range(3):
        for t in got:
            t.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
