"""The core attention in two halves, the second beside the text attention: the bits and the number of launches of the calls one by one."""
import pytest
import torch

import magi_attn as M
from magi_attn import _lib as L
from magi_attn.functional import BegunCalls, attention_waves, launch_held, range_attention

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available()
    return torch.device("cuda")


# keys in pieces: less than a round of 256-row workgroups, a round and a part; ranges of two lengths; text around the 32- and 64-key tiles, of
# which one segment has none; 256-row items all whole ("whole": both in one launch; text of 128-row items, in pieces by itself); a core of another
# form (done by its first half); text in a launch of its own (few rows)
@pytest.mark.parametrize("chunks,Lc,prefix,Hq,Hkv,text,pieces", [
    (3, 1296, 0, 24, 8, (660, 1, 129), "whole"), (4, 660, 0, 48, 8, (577, 0, 96, 32), "whole"), (3, 1392, 2, 24, 8, (732, 70, 31), "whole"),
    (1, 1350, 7, 24, 8, (468,), True), (1, 672, 5, 48, 8, (33,), True), (3, 1134, 8, 48, 8, (0, 259, 800), True), (2, 1440, 1, 24, 8, (31, 65), True),
    (1, 9360, 0, 24, 8, (400,), True), (1, 2310, 2, 24, 8, (97,), True), (4, 384, 4, 24, 8, (162, 1, 32, 64), False),
    (4, 336, 3, 48, 8, (72, 5, 0, 96), False), (1, 240, 12, 24, 8, (45,), False)])
def test_the_bits_of_the_calls_one_by_one(dev, chunks, Lc, prefix, Hq, Hkv, text, pieces):
    g = torch.Generator(device=dev).manual_seed(Lc + Hq)
    D, S, K, T = 128, chunks * Lc, (chunks + prefix) * Lc, sum(text)
    rows = lambda *s: torch.nn.functional.layer_norm(torch.randn(*s, D, device=dev, generator=g), (D,)).bfloat16()
    q = (rows(S, Hq).float() * (D ** -0.5 * 1.4426950408889634)).bfloat16()
    cache = torch.randn(K, Hkv, 2 * D, device=dev, generator=g, dtype=torch.bfloat16)
    cache[..., :D] = rows(K, Hkv)
    q_ranges = torch.tensor([[i * Lc, (i + 1) * Lc] for i in range(chunks)], dtype=torch.int32, device=dev)
    k_ranges = torch.tensor([[0, (prefix + i + 1) * Lc] for i in range(chunks)], dtype=torch.int32, device=dev)
    qx = torch.randn(S, 2 * Hq, D, device=dev, generator=g, dtype=torch.bfloat16)[:, Hq:]  # a view of the projection
    kv = torch.randn(T, Hkv, 2 * D, device=dev, generator=g, dtype=torch.bfloat16)
    kv[..., :D] = rows(T, Hkv)
    gamma, beta = torch.randn(D, device=dev, generator=g) * 0.1, torch.randn(D, device=dev, generator=g) * 0.1
    cu_q = torch.arange(0, S + 1, Lc, dtype=torch.int32, device=dev)
    cu_k = torch.tensor((0,) + text, dtype=torch.int32, device=dev).cumsum(0).to(torch.int32)
    waves = attention_waves(Hq, Hkv, chunks, L.MAGI_RANGES_CU, Lc, 800)

    def core(held):
        return range_attention(q, cache[..., :D], cache[..., D:], q_ranges, k_ranges, Lc, K, return_lse=False, q_prescaled=True, score_bound=17.0,
                               share_waves=True, held=held)[0]

    def cross(held, split=True):
        return range_attention(qx, kv[..., :D], kv[..., D:], cu_q, cu_k, Lc, 800, ranges_mode=L.MAGI_RANGES_CU, return_lse=False, score_bound=30.0,
                               q_norm=(gamma, beta, 1e-6), share_waves=True, held=held, split_keys=split)[0]

    n = M.lib().magi_launch_count
    n0 = n()
    want = core(None)
    n1 = n()
    want_x = cross(None, split=not pieces or bool(waves))  # (beside the merge the text's own items are whole)
    assert n1 - n0 == (2 if pieces is True else 1)
    held, n0 = BegunCalls(), n()
    got = core(held)
    assert n() - n0 == int(pieces != "whole") and len(held) == int(bool(pieces))
    got_x = cross(held)
    launch_held(held)
    assert not held and torch.equal(got, want) and torch.equal(got_x, want_x)
    assert bool(torch.isfinite(got.float()).all()) and bool(torch.isfinite(got_x.float()).all())
    if pieces:
        assert n() - n0 == (1 if pieces == "whole" else 2)  # (the core;) its merge, or all of it, and the text
        held = BegunCalls()
        alone = core(held)
        launch_held(held)  # (nothing beside it)
        assert torch.equal(alone, want)


# a second call of 128-row items whose keys are shared; one of the online softmax; one that joins the merge
@pytest.mark.parametrize("rows,keys,raw", [(480, 4000, True), (480, 4000, False), (2112, 400, True)])
def test_one_scratch_buffer_for_both(dev, rows, keys, raw):
    """A caller that keeps one split_workspace per stream: the second call may not leave its pieces there ahead of the first one's merge."""
    g = torch.Generator(device=dev).manual_seed(rows)
    D, Hq, Hkv, S, K = 128, 24, 8, 2112, 14784
    draw = lambda *s: torch.randn(*s, D, device=dev, generator=g, dtype=torch.bfloat16)
    norm = lambda t: torch.nn.functional.layer_norm(t.float(), (D,))
    q, k, v = (norm(draw(S, Hq)) * (D ** -0.5 * 1.4426950408889634)).bfloat16(), norm(draw(K, Hkv)).bfloat16(), draw(K, Hkv)
    qx, kx, vx = draw(rows, Hq), norm(draw(keys, Hkv)).bfloat16(), draw(keys, Hkv)
    ranges = lambda n: torch.tensor([[0, n]], dtype=torch.int32, device=dev)
    more = dict(score_bound=30.0, q_norm=(torch.randn(D, device=dev, generator=g) * 0.1, None, 1e-6)) if raw else {}
    core = lambda held: range_attention(q, k, v, ranges(S), ranges(K), S, K, return_lse=False, q_prescaled=True, score_bound=17.0, held=held)[0]
    cross = lambda held: range_attention(qx, kx, vx, ranges(rows), ranges(keys), rows, keys, return_lse=False, held=held, **more)[0]
    want, want_x = core(None), cross(None)
    held = []
    got, got_x = core(held), cross(held)
    calls = [L.AttnArgs.from_buffer_copy(c[2]) for c in held]
    assert calls[0].split_workspace and (calls[1].split_workspace or rows > 480)
    scratch = torch.empty(max(c.split_workspace_bytes for c in calls), dtype=torch.uint8, device=dev)
    for c in calls:
        c.split_workspace, c.split_workspace_bytes = scratch.data_ptr(), scratch.numel()
    stream = torch.cuda.current_stream().cuda_stream
    lib = L.lib()
    assert lib.magi_attn_fwd_begin(calls[0], stream) == 1 and lib.magi_attn_fwd_end(calls[0], calls[1], stream) == 0
    assert torch.equal(got, want) and torch.equal(got_x, want_x)


@pytest.mark.parametrize("static", ["first", "second", "both"])
@pytest.mark.parametrize("calls", [list, BegunCalls])
def test_held_calls_with_static_scratch_memory(dev, calls, static):
    """They take no workspace, which the entry points for two calls and for two halves would ask a measured bound for."""
    g = torch.Generator(device=dev).manual_seed(5)
    t = torch.randn(4200, 24, 128, device=dev, generator=g, dtype=torch.bfloat16) * 0.25  # (256-row items, which a first half leaves)
    r = torch.tensor([[0, 4200]], dtype=torch.int32, device=dev)

    def call(i, held):
        kw = {"auto_bound": True, "static_scratch": True} if static in ("both", ("first", "second")[i]) else {"score_bound": 60.0, "q_prescaled": True}
        return range_attention(t, t[:, i::3], t[:, i::3], r, r, 4200, 4200, return_lse=False, held=held, **kw)[0]

    want, held = [call(i, None) for i in (0, 1)], calls()
    got = [call(i, held) for i in (0, 1)]
    launch_held(held)
    assert not held and all(torch.equal(a, b) for a, b in zip(got, want))


def test_an_end_without_pieces_is_refused(dev):
    q = torch.randn(64, 4, 128, device=dev, dtype=torch.bfloat16)
    r = torch.tensor([[0, 64]], dtype=torch.int32, device=dev)
    held = []
    range_attention(q, q, q, r, r, 64, 64, held=held, return_lse=False)
    with pytest.raises(M.MagiError):
        launch_held([(held[0][0], None) + held[0][2:]])


@pytest.mark.parametrize("chunks,Lc,prefix,text", [(1, 1350, 2, (468,)), (3, 1296, 0, (660, 1, 129))])  # in pieces; whole items
def test_captured_in_a_graph(dev, chunks, Lc, prefix, text):
    g = torch.Generator(device=dev).manual_seed(Lc)
    Hq, Hkv, D, S, K, T = 24, 8, 128, chunks * Lc, (chunks + prefix) * Lc, sum(text)
    norm = lambda t: torch.nn.functional.layer_norm(t.float(), (D,))
    draw = lambda *s: torch.randn(*s, D, device=dev, generator=g, dtype=torch.bfloat16)
    q, qx, v, vx = draw(S, Hq), draw(S, Hq), draw(K, Hkv), draw(T, Hkv)
    k, kx = norm(draw(K, Hkv)).bfloat16(), norm(draw(T, Hkv)).bfloat16()
    q_ranges = torch.tensor([[i * Lc, (i + 1) * Lc] for i in range(chunks)], dtype=torch.int32, device=dev)
    k_ranges = torch.tensor([[0, (prefix + i + 1) * Lc] for i in range(chunks)], dtype=torch.int32, device=dev)
    gamma = torch.randn(D, device=dev, generator=g) * 0.1
    cu_q = torch.arange(0, S + 1, Lc, dtype=torch.int32, device=dev)
    cu_k = torch.tensor((0,) + text, dtype=torch.int32, device=dev).cumsum(0).to(torch.int32)

    def both():
        held = BegunCalls()
        a, _ = range_attention(q, k, v, q_ranges, k_ranges, Lc, K, return_lse=False, q_prescaled=True, score_bound=17.0, held=held)
        b, _ = range_attention(qx, kx, vx, cu_q, cu_k, Lc, 800, ranges_mode=L.MAGI_RANGES_CU, return_lse=False, score_bound=30.0,
                               q_norm=(gamma, None, 1e-6), held=held)
        launch_held(held)
        return a, b

    fill = lambda: (q.copy_(norm(draw(S, Hq)) * (D ** -0.5 * 1.4426950408889634)), qx.copy_(draw(S, Hq)))
    fill()
    both()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = both()
    for _ in range(3):
        fill()
        want = both()
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(out, want):
            assert torch.equal(x, y)
