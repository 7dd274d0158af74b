"""GPU tests of the online softmax on 16x16x32 MFMAs: whole items in more workgroups than run at a time, and items whose keys are
shared by several workgroups (magi_attn_args.split_workspace)."""
import pytest
import torch

import magi_attn as M
from magi_attn import _lib as L
from oracle import magi_oracle as O

pytestmark = pytest.mark.gpu


def _ranges(pairs, dev):
    return torch.tensor(pairs, dtype=torch.int32, device=dev)


def _near(a, b, size, lse_a, lse_b):
    """Probabilities p are rounded to bf16 relative to the running maximum: 2^-9 p each, on either side; the outputs are rounded too.
    So two results differ by at most 2^-8 sum(p |v|) / sum(p) (`size`, the attention over |v|) and one bf16 step."""
    d = (a.float() - b.float()).abs()
    assert torch.isfinite(a).all() and (d <= size.float() * 2.0 ** -8 + b.float().abs() * 2.0 ** -8 + 1e-6).all(), d.max().item()
    fin = torch.isfinite(lse_b)
    assert torch.equal(fin, torch.isfinite(lse_a)) and (lse_a - lse_b)[fin].abs().max().item() <= 2e-5


# (rows per range, ranges, cached ranges, heads, max_seqlen_k): last tiles with wavefronts and rows missing, a last piece of one key,
# odd head counts (padding in the grid), ranges of unequal length (surplus pieces), ranges of no keys and of less than a piece
CASES = [(300, 1, 5, 3, 1, 0), (129, 2, 12, 6, 2, 0), (33, 3, 60, 12, 4, 0), (1, 1, 4097, 1, 1, 0), (300, 4, 0, 5, 5, 4000),
         (500, 2, 4, 24, 8, 0), (700, 3, 3, 3, 1, 0)]


@pytest.mark.parametrize("rows,n,sp,Hq,Hkv,max_k", CASES)
def test_shared_keys_give_what_one_workgroup_gives(dev, rows, n, sp, Hq, Hkv, max_k):
    Tk = (sp + n) * rows
    mk = max_k or Tk
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert cus != 256 or L.lib().magi_attn_pieces_bytes(Hq, Hkv, n, rows, mk, 0) > 0
    q, k, v = (t.to(dev) for t in O.synthetic_qkv(n * rows + 7, Tk, Hq, Hkv, 128, seed=rows + n))
    qr = _ranges([[i * rows, (i + 1) * rows] for i in range(n)], dev)
    kr = _ranges([[0, (sp + 1 + i) * rows] for i in range(n)], dev)
    if max_k:
        kr[0] = kr[0, 0]  # no keys
        kr[1, 1] = 3
    n0 = M.lib().magi_launch_count()
    a, la = M.range_attention(q, k, v, qr, kr, rows, mk)
    n1 = M.lib().magi_launch_count()
    b, lb = M.range_attention(q, k, v, qr, kr, rows, mk, split_keys=False)
    assert n1 - n0 == M.lib().magi_launch_count() - n1 + (1 if cus == 256 else 0)
    size = M.range_attention(q, k, v.abs(), qr, kr, rows, mk, split_keys=False)[0]
    _near(a, b, size, la, lb)
    assert torch.equal(a, M.range_attention(q, k, v, qr, kr, rows, mk)[0])  # whatever order the pieces end in
    ref = O.range_attention(q.cpu(), k.cpu(), v.cpu(), qr.cpu().numpy(), kr.cpu().numpy())
    assert (a[:n * rows].float().cpu() - ref[:n * rows]).abs().max().item() <= 2e-2


@pytest.mark.parametrize("what", ["large scores", "one key above all", "side segment", "grouped out", "strided"])
def test_shared_keys_other_inputs(dev, what):
    rows, Hq, Hkv, Tk = 300, 8, 2, 3000
    q, k, v = (t.to(dev) for t in O.synthetic_qkv(rows, Tk, Hq, Hkv, 128, seed=4))
    qr, kr = _ranges([[0, rows]], dev), _ranges([[0, Tk]], dev)
    kw, tail = {}, {}
    if what == "large scores":
        q = (q.float() * 40).bfloat16()
    elif what == "one key above all":
        k[1700] *= 50  # rows whose other pieces vanish beside one key's
    elif what == "side segment":
        tail = dict(k2=k[1000:].contiguous(), v2=v[1000:].contiguous(), k_split=1000)
    elif what == "strided":
        kv = torch.cat([k, v], 2)
        k, v = kv[..., :128], kv[..., 128:]
    ref = M.range_attention(q, k, v, qr, kr, rows, Tk, split_keys=False)
    size = M.range_attention(q, k, v.abs(), qr, kr, rows, Tk, split_keys=False)[0]
    if what == "grouped out":
        out = torch.empty(2, rows, 4, 128, dtype=torch.bfloat16, device=dev).transpose(0, 1)
        got = M.range_attention(q, k, v, qr, kr, rows, Tk, out=out)
        got = (got[0].reshape(rows, Hq, 128), got[1])
    elif tail:
        got = M.range_attention(q, k[:1000].contiguous(), v[:1000].contiguous(), qr, kr, rows, Tk, **tail)
    else:
        got = M.range_attention(q, k, v, qr, kr, rows, Tk, **kw)
    d = (got[0].float() - ref[0].float()).abs()
    assert (d <= size.float() * 2.0 ** -8 + ref[0].float().abs() * 2.0 ** -8 + 1e-6).all(), d.max().item()
    # (scores up to 2^10: the running maximum's share of lse is rounded to 2^-14)
    assert (got[1] - ref[1]).abs().max().item() <= 2e-4


def test_shared_keys_captured(dev):
    rows, Hq, Hkv, Tk = 200, 6, 2, 4000
    q, k, v = (t.to(dev) for t in O.synthetic_qkv(rows, Tk, Hq, Hkv, 128, seed=9))
    qr, kr = _ranges([[0, rows]], dev), _ranges([[0, Tk]], dev)
    want = M.range_attention(q, k, v, qr, kr, rows, Tk)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = M.range_attention(q, k, v, qr, kr, rows, Tk)
    for _ in range(3):
        got[0].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_more_whole_items_than_run_at_a_time(dev):
    """896 workgroups of every key count around the tile's edges, among them none; rows no range covers; the lse."""
    rows, Hq, Hkv = 200, 64, 8
    keys = [0, 1, 63, 64, 65, 129, 200]
    n, Tk = len(keys), 400
    q, k, v = (t.to(dev) for t in O.synthetic_qkv(n * rows + 5, Tk, Hq, Hkv, 128, seed=2))
    qr = _ranges([[i * rows, (i + 1) * rows] for i in range(n)], dev)
    kr = _ranges([[7 * i, 7 * i + c] for i, c in enumerate(keys)], dev)
    out, lse = M.range_attention(q, k, v, qr, kr, rows, 200)
    ref = O.range_attention(q.cpu(), k.cpu(), v.cpu(), qr.cpu().numpy(), kr.cpu().numpy())
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2
    assert not out[:rows].any() and not out[n * rows:].any()
    for i, c in enumerate(keys):
        s = torch.einsum("qd,kd->qk", q[i * rows:(i + 1) * rows, 9].float().cpu(), k[7 * i:7 * i + c, 1].float().cpu()) * 128 ** -0.5
        want = s.logsumexp(1) if c else torch.full((rows,), float("-inf"))
        assert torch.allclose(lse[9, i * rows:(i + 1) * rows].cpu(), want, atol=2e-5)
    assert torch.isinf(lse[:, n * rows:]).all()


@pytest.mark.parametrize("call", ["flex", "varlen"])
def test_without_memory_for_the_pieces_the_items_stay_whole(dev, monkeypatch, call):
    """The rebound callables need no memory but their output's: where there is none to share the keys with, they run as they do without."""
    rows, Hq, Hkv, Tk = 300, 6, 2, 4000
    q, k, v = (t.to(dev) for t in O.synthetic_qkv(rows, Tk, Hq, Hkv, 128, seed=3))
    qr, kr = _ranges([[0, rows]], dev), _ranges([[0, Tk]], dev)
    want = M.range_attention(q, k, v, qr, kr, rows, Tk, split_keys=False)[0]
    real, refused = torch.empty, []

    def empty(*size, dtype=None, **kw):
        if dtype is torch.uint8:
            refused.append(size)
            raise torch.OutOfMemoryError("no scratch memory")
        return real(*size, dtype=dtype, **kw)

    monkeypatch.setattr(torch, "empty", empty)
    if call == "flex":
        got = M.flex_flash_attn_func(q, k, v, qr, kr, rows, Tk)[0]
    else:
        got = M.flash_attn_varlen_func(q, k, v, qr[0], kr[0], rows, Tk)
    assert torch.equal(got, want) and (refused or torch.cuda.get_device_properties(dev).multi_processor_count != 256)
