"""The largest magnitudes of v's rows, which the e4m3 prologue leaves for the quantiser: the bytes, scales and launches of the quantiser that
reads v for them, and q and k as the prologue without them writes them."""
import math

import pytest
import torch

import magi_attn as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available()
    return torch.device("cuda")


# one row; edges of the 64 rows of a pass and the 256 of a batch of loads; odd and ragged chunks; several tokens per workgroup (few heads);
# more row groups than the 32 of a workgroup; slices that come out empty (share x rows of a slice past the chunk)
@pytest.mark.parametrize("S,Lc,n1,Hq,Hkv", [(1, 1, 1, 2, 1), (63, 63, 63, 24, 8), (64, 64, 0, 24, 8), (65, 65, 65, 6, 2), (130, 65, 65, 3, 1),
                                            (771, 257, 514, 24, 8), (1000, 300, 1000, 24, 8), (1023, 1023, 0, 48, 8), (4200, 4200, 4200, 6, 1),
                                            (9360, 9360, 9360, 24, 8), (5001, 5001, 5001, 8, 3)])
def test_row_maxima_give_the_bytes_of_the_pass_over_v(dev, S, Lc, n1, Hq, Hkv):
    g = torch.Generator(device=dev).manual_seed(S + Hq)
    D, f8 = 128, torch.float8_e4m3fn
    raw = torch.randn(S, (Hq + 2 * Hkv) * D, device=dev, generator=g, dtype=torch.bfloat16)
    q, k, v = raw.split([Hq * D, Hkv * D, Hkv * D], 1)
    v[0, :D] = 0.0
    v[S // 2, 5] = -7.25e3
    if S > 600:
        v[S - 1, D - 1] = math.inf
        v[S // 3, 0] = math.nan
    rope = torch.randn(S, 96, device=dev, generator=g)
    par = [torch.randn(D, device=dev, generator=g) * 0.1 for _ in range(4)]
    kw = dict(Hq=Hq, Hkv=Hkv, q_scale=0.125, k_scale=0.25, q_premul=0.13)
    row_max = torch.full((Hkv, S), -1, dtype=torch.int16, device=dev)
    q8, k8, _ = M.qk_prologue_fp8(q, k, rope, *par, v_raw=v, v_row_max=row_max, **kw)
    q0, k0, _ = M.qk_prologue_fp8(q, k, rope, *par, **kw)
    byte = lambda t: t.view(torch.uint8)
    assert torch.equal(byte(q8), byte(q0)) and torch.equal(byte(k8), byte(k0))
    want = (v.reshape(S, Hkv, D).contiguous().view(torch.int16).int() & 0x7FFF).amax(-1).t()
    assert torch.equal(row_max.int() & 0xFFFF, want)

    def quantise(**more):
        y = [torch.zeros((n, Hkv, D), dtype=torch.uint8, device=dev).view(f8) for n in (n1, S - n1)]
        sc = [torch.zeros(((n + Lc - 1) // Lc, Hkv), device=dev) for n in (n1, S - n1)]
        before = M.lib().magi_launch_count()
        M.quantize_fp8_split(v.reshape(S, Hkv, D), Lc, n1, y[0], sc[0], y[1], sc[1], pow2_scales=True, **more)
        assert M.lib().magi_launch_count() == before + 1
        return [byte(t) for t in y] + [t.view(torch.int32) for t in sc]

    for a, b in zip(quantise(row_max=row_max), quantise()):
        assert torch.equal(a, b)


def test_row_maxima_of_another_shape_are_refused(dev):
    x = torch.randn(8, 2, 128, device=dev, dtype=torch.bfloat16)
    y, sc = torch.empty(8, 2, 128, dtype=torch.float8_e4m3fn, device=dev), torch.empty(1, 2, device=dev)
    for bad in (torch.zeros(8, 2, dtype=torch.int16, device=dev), torch.zeros(2, 8, device=dev), torch.zeros(2, 8, dtype=torch.int16)):
        with pytest.raises(ValueError):
            M.quantize_fp8_split(x, 8, 8, y, sc, None, None, row_max=bad)
