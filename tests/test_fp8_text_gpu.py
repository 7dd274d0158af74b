"""Core attention of e4m3 rows and text attention in one launch: the bits of the two launches, and how many there are."""
import pytest
import torch

import magi_attn as M
from magi_attn import _lib as L
from magi_attn.functional import attention_waves, launch_held, range_attention

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available()
    return torch.device("cuda")


# rows and text lengths around the tiles (128 rows; 32 and 64 keys): one key, 31 to 33, 63 to 65, 95 to 97, no text for one segment; ranges in
# pieces (a round of workgroups and a part of one); few heads; a text launch that would be in pieces by itself (beside the core it is not:
# against the call without memory for them, but where the wavefronts of a workgroup share the keys, which stays a launch of its own)
@pytest.mark.parametrize("chunks,Lc,prefix,Hq,Hkv,text", [(1, 1, 0, 8, 1, (1,)), (2, 130, 1, 24, 8, (31, 32)), (3, 127, 0, 6, 2, (33, 0, 63)),
                                                          (2, 640, 1, 24, 8, (64, 65)), (2, 1300, 0, 48, 8, (95, 400)), (1, 4000, 1, 24, 8, (97,)),
                                                          (4, 257, 2, 3, 1, (800, 1, 96, 128)), (2, 5000, 0, 24, 8, (161, 77)),
                                                          (1, 9360, 0, 24, 8, (800,))])
@pytest.mark.parametrize("fast", [False, True])
def test_the_bits_of_the_two_launches(dev, chunks, Lc, prefix, Hq, Hkv, text, fast):
    g = torch.Generator(device=dev).manual_seed(Lc + Hq)
    D, S, K, T = 128, chunks * Lc, (chunks + prefix) * Lc, sum(text)
    rows = lambda *s: torch.nn.functional.layer_norm(torch.randn(*s, D, device=dev, generator=g), (D,)).bfloat16()
    q8, qs = M.quantize_fp8(rows(S, Hq), Lc, D ** -0.5 * 1.4426950408889634, True)
    k8, ks = M.quantize_fp8(rows(K, Hkv), Lc, 1.0, True)
    v8, vs = M.quantize_fp8(torch.randn(K, Hkv, D, device=dev, generator=g, dtype=torch.bfloat16), Lc, 1.0, True)
    q_ranges = torch.tensor([[i * Lc, (i + 1) * Lc] for i in range(chunks)], dtype=torch.int32, device=dev)
    k_ranges = torch.tensor([[0, (prefix + i + 1) * Lc] for i in range(chunks)], dtype=torch.int32, device=dev)
    qx = torch.randn(S, 2 * Hq, D, device=dev, generator=g, dtype=torch.bfloat16)[:, Hq:]  # a view of the projection
    kv = torch.randn(T, Hkv, 2 * D, device=dev, generator=g, dtype=torch.bfloat16)
    kv[..., :D] = rows(T, Hkv)
    gamma, beta = torch.randn(D, device=dev, generator=g) * 0.1, torch.randn(D, device=dev, generator=g) * 0.1
    cu_q = torch.arange(0, S + 1, Lc, dtype=torch.int32, device=dev)
    cu_k = torch.tensor((0,) + text, dtype=torch.int32, device=dev).cumsum(0).to(torch.int32)

    waves = attention_waves(Hq, Hkv, chunks, L.MAGI_RANGES_CU, Lc, 800)

    def calls(held):
        core, _ = range_attention(q8, k8, v8, q_ranges, k_ranges, Lc, K, q_scale=qs, k_scale=ks, v_scale=vs, scale_chunk_tokens=Lc,
                                  fp8_pow2_prescaled=True, fp8_fast_exp2=fast, return_lse=False, held=held)
        cross, _ = range_attention(qx, kv[..., :D], kv[..., D:], cu_q, cu_k, Lc, 800, ranges_mode=L.MAGI_RANGES_CU, return_lse=False,
                                   score_bound=30.0, q_norm=(gamma, beta, 1e-6), share_waves=True, held=held,
                                   split_keys=held is not None or bool(waves))
        return core, cross

    one_by_one = calls(None)
    held = []
    before = M.lib().magi_launch_count()
    together = calls(held)
    assert M.lib().magi_launch_count() == before and len(held) == 2
    launch_held(held)
    assert not held and 1 <= M.lib().magi_launch_count() - before <= 4
    turned = calls(held)
    held.reverse()  # (the text first: two launches)
    launch_held(held)
    for a, b, c in zip(together, one_by_one, turned):
        assert torch.equal(a, b) and torch.equal(c, b) and bool(torch.isfinite(a.float()).all())


def test_a_held_call_by_itself(dev):
    q8 = torch.randn(64, 4, 128, device=dev).to(torch.float8_e4m3fn)
    sc, r = torch.ones(1, 4, device=dev), torch.tensor([[0, 64]], dtype=torch.int32, device=dev)
    kw = dict(q_scale=sc, k_scale=sc, v_scale=sc, scale_chunk_tokens=64, fp8_pow2_prescaled=True, return_lse=False)
    held = []
    a, _ = range_attention(q8, q8, q8, r, r, 64, 64, held=held, **kw)
    launch_held(held)
    assert torch.equal(a, range_attention(q8, q8, q8, r, r, 64, 64, **kw)[0])
