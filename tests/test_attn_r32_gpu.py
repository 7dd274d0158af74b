"""GPU tests of launches without a running maximum in 128-row workgroups, three per CU: whole items have the bits of 256-row workgroups,
pieces of the keys add up to them."""
import pytest
import torch

import magi_attn as M
from magi_attn import _lib as L
from oracle import magi_oracle as O

pytestmark = pytest.mark.gpu
PRE = 128 ** -0.5 * 1.4426950408889634


def _case(dev, rows, n, Hq, Hkv, keys, mode, seed=0):
    Tk = max(b for _, b in keys)
    q, k, v = (t.to(dev) for t in O.synthetic_qkv(n * rows + 5, Tk, Hq, Hkv, 128, seed=seed))
    qr = torch.tensor([[i * rows, (i + 1) * rows] for i in range(n)], dtype=torch.int32, device=dev)
    kr = torch.tensor(keys, dtype=torch.int32, device=dev)
    kw = {"as it is": {"q_prescaled": True, "score_bound": 40.0}, "scaled": {"score_bound": 40.0},
          "norm": {"score_bound": 40.0, "q_norm": (torch.linspace(-0.2, 0.2, 128, device=dev), None, 1e-6)}}[mode]
    if mode == "as it is":
        q = (q.float() * PRE).bfloat16()
    return q, k, v, qr, kr, kw


# more than two workgroups per CU and at most three; tiles with wavefronts and rows missing; ranges of one key, of a tile's and half a tile's
# edges, of none; no launch of the other forms
@pytest.mark.parametrize("mode", ["as it is", "scaled", "norm"])
@pytest.mark.parametrize("rows,Hq,Hkv,keys", [
    (200, 48, 8, [(0, 1), (0, 0), (3, 35), (3, 36), (5, 69), (0, 200)]), (129, 64, 8, [(0, 64), (0, 65), (0, 128), (9, 300), (0, 31)]),
    (2700, 24, 8, [(0, 500)])])
def test_whole_items_have_the_bits_of_256_rows(dev, rows, Hq, Hkv, keys, mode):
    n = len(keys)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    items = Hq * n * ((rows + 127) // 128)
    assert cus != 256 or 2 * cus < items <= 3 * cus
    q, k, v, qr, kr, kw = _case(dev, rows, n, Hq, Hkv, keys, mode)
    a, la = M.range_attention(q, k, v, qr, kr, rows, 500, **kw)
    b, lb = M.range_attention(q, k, v, qr, kr, rows, 500, q_tile_rows=256, split_keys=False, **kw)
    assert torch.equal(a, b) and torch.equal(la, lb)


# single and unequal ranges, odd head counts, fewer keys than the launch was sized for (surplus pieces), a last piece of one key
@pytest.mark.parametrize("mode", ["as it is", "scaled", "norm"])
@pytest.mark.parametrize("rows,Hq,Hkv,keys,max_k", [
    (270, 6, 2, [(0, 1601)], 0), (300, 3, 1, [(0, 1200), (0, 1500), (0, 1800)], 0), (129, 5, 5, [(0, 3), (7, 7), (0, 2400)], 3000), (1, 1, 1, [(0, 4097)], 0),
    (432, 24, 8, [(0, 1728)], 0)])
def test_pieces_add_up(dev, rows, Hq, Hkv, keys, max_k, mode):
    n, mk = len(keys), max_k or max(b for _, b in keys)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert cus != 256 or L.lib().magi_attn_pieces_bytes(Hq, Hkv, n, rows, mk, 1) > 0
    q, k, v, qr, kr, kw = _case(dev, rows, n, Hq, Hkv, keys, mode, seed=rows)
    a, la = M.range_attention(q, k, v, qr, kr, rows, mk, **kw)
    b, lb = M.range_attention(q, k, v, qr, kr, rows, mk, split_keys=False, **kw)
    # fp32 sums in another order: far less than half a bf16 step of outputs of about 0.05 (test_attn_split_gpu.py)
    d = (a.float() - b.float()).abs()
    assert torch.isfinite(a).all() and (d <= b.float().abs() * 2.0 ** -7 + 1e-5).all(), d.max().item()
    fin = torch.isfinite(lb)
    assert torch.equal(fin, torch.isfinite(la)) and (la - lb)[fin].abs().max().item() <= 1e-5
    assert torch.equal(a, M.range_attention(q, k, v, qr, kr, rows, mk, **kw)[0])
    if mode == "scaled":
        ref = O.range_attention(q.cpu(), k.cpu(), v.cpu(), qr.cpu().numpy(), kr.cpu().numpy())
        assert (a[:n * rows].float().cpu() - ref[:n * rows]).abs().max().item() <= 2e-2


def test_a_gate_closes_pieces_too(dev):
    """Scores that the measured bound hands to the online softmax: the launch in pieces and its merge leave the output alone."""
    q, k, v, qr, kr, _ = _case(dev, 270, 1, 6, 2, [(0, 1601)], "scaled")
    q = (q.float() * 60).bfloat16()
    a = M.range_attention(q, k, v, qr, kr, 270, 1601, auto_bound=True)
    b = M.range_attention(q, k, v, qr, kr, 270, 1601, split_keys=False)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("batch", [2, 3])
def test_batched_rows_in_groups_of_heads(dev, batch):
    rows, Hq, Hkv, n = 150, 8, 2, 90
    torch.manual_seed(batch)
    q = torch.randn(rows, batch, Hq, 128, device=dev).bfloat16().transpose(0, 1)
    kv = torch.randn(n, Hkv, 256, device=dev).bfloat16()
    cq = torch.tensor([0, rows], dtype=torch.int32, device=dev)  # (the other batch rows are covered by no range)
    ck = torch.tensor([0, n], dtype=torch.int32, device=dev)
    for bound in (60.0, float("inf")):
        kw = dict(ranges_mode=L.MAGI_RANGES_CU, return_lse=False, score_bound=bound)
        want, _ = M.range_attention(q, kv[..., :128], kv[..., 128:], cq, ck, batch * rows, n, **kw)
        store = torch.full((rows, batch, 4, 2, 2, 128), float("nan"), dtype=torch.bfloat16, device=dev)
        out = store[:, :, :, 1].transpose(0, 1)
        got, _ = M.range_attention(q, kv[..., :128], kv[..., 128:], cq, ck, batch * rows, n, out=out, clear_out=True, **kw)
        assert got is out and torch.equal(out.reshape(batch, rows, Hq, 128), want)
        assert torch.isnan(store[:, :, :, 0]).all()


# (the last: 3072 workgroups of 384 rows, which is what such a launch takes from 9 per CU and a stated max_seqlen_k of 4096 on; 1024 in one range)
@pytest.mark.parametrize("rows,Hq,Hkv", [(1536, 24, 8), (130, 256, 32), (3500, 24, 8), (1400, 256, 32)])
def test_rows_have_the_bits_of_their_range_alone(dev, rows, Hq, Hkv):
    """Without shared keys, where all ranges are a launch of more than three workgroups per CU (and one range is not, or is in the larger
    workgroups of many rounds): the online softmax keeps to one order of the keys."""
    torch.manual_seed(rows)
    n = 3
    q = torch.randn(n * rows, Hq, 128, device=dev).bfloat16()
    k, v = (torch.randn(n * rows, Hkv, 128, device=dev).bfloat16() for _ in range(2))
    qr = torch.tensor([[i * rows, (i + 1) * rows] for i in range(n)], dtype=torch.int32, device=dev)
    kr = torch.tensor([[0, (i + 1) * rows] for i in range(n)], dtype=torch.int32, device=dev)
    all_rows, _ = M.range_attention(q, k, v, qr, kr, rows, n * rows, split_keys=False)
    for i in range(n):
        one, _ = M.range_attention(q[i * rows:(i + 1) * rows], k, v, qr[:1], kr[i:i + 1], rows, n * rows, split_keys=False)
        assert torch.equal(one, all_rows[i * rows:(i + 1) * rows]), i
    with pytest.raises(M.MagiError, match="ROW_BITS"):  # (nor with memory for shared keys)
        a = L.AttnArgs(dtype=L.MAGI_DTYPE_BF16, D=128, Hq=1, Hkv=1, total_q=1, total_k=0, n_ranges=1, max_seqlen_q=1, flags=L.MAGI_ATTN_ROW_BITS,
                       q=q.data_ptr(), out=q.data_ptr(), q_ranges=qr.data_ptr(), k_ranges=kr.data_ptr(), split_workspace=q.data_ptr(),
                       split_workspace_bytes=16, **{"%s_stride_%s" % (x, y): 128 for x in "qkvo" for y in "th"})
        L.check(L.lib().magi_attn_fwd(a, None))


@pytest.mark.parametrize("bounded", [False, True])
@pytest.mark.parametrize("stated", [2000, 1920, 5000])
def test_ranges_that_are_not_as_long_as_stated(dev, stated, bounded):
    """max_seqlen_k plans the pieces and no more: the last one of a longer range takes the rest, a shorter one has fewer."""
    rows, n, Hq, Hkv = 200, 4321, 6, 2
    assert L.lib().magi_attn_pieces_bytes(Hq, Hkv, 2, rows, stated, int(bounded)) > 0
    q, k, v = (t.to(dev) for t in O.synthetic_qkv(2 * rows, n, Hq, Hkv, 128, seed=stated))
    qr = torch.tensor([[0, rows], [rows, 2 * rows]], dtype=torch.int32, device=dev)
    kr = torch.tensor([[0, n], [17, 17 + n // 3]], dtype=torch.int32, device=dev)
    kw = dict(score_bound=30.0) if bounded else {}
    got, lse = M.range_attention(q, k, v, qr, kr, rows, stated, **kw)
    want, want_lse = M.range_attention(q, k, v, qr, kr, rows, stated, split_keys=False, **kw)
    size = M.range_attention(q, k, v.abs(), qr, kr, rows, stated, split_keys=False, **kw)[0].float()
    # (bf16 probabilities and results on both sides, as in test_attn_online_split_gpu.py)
    assert ((got.float() - want.float()).abs() <= 2.0 ** -6 * size + 1e-6).all()
    assert (lse - want_lse).abs().max() < 1e-4


@pytest.mark.parametrize("bounded", [False, True])
@pytest.mark.parametrize("stated", [1500, 2 ** 31 - 1])
def test_pieces_of_a_range_far_along_the_key_axis(dev, stated, bounded):
    """Keys 2e9 .. 2e9 + 1500 of an axis whose first segment is never looked at: pieces are counted from the range's first key, those
    behind its end, at positions beyond 2^31 with the largest stated length, leave nothing."""
    rows, n, far, Hq, Hkv = 200, 1500, 2_000_000_000, 6, 2
    size = L.lib().magi_attn_pieces_bytes(Hq, Hkv, 1, rows, stated, int(bounded))
    assert size > 0
    q, k, v = (t.to(dev) for t in O.synthetic_qkv(rows, n, Hq, Hkv, 128, seed=5))
    kw = dict(score_bound=30.0) if bounded else {}
    want, _ = M.range_attention(q, k, v, *(torch.tensor([[0, m]], dtype=torch.int32, device=dev) for m in (rows, n)), rows, stated, **kw)
    out, scratch = torch.empty_like(q), torch.empty(size, dtype=torch.uint8, device=dev)
    qr, kr = torch.tensor([[0, rows]], dtype=torch.int32, device=dev), torch.tensor([[far, far + n]], dtype=torch.int32, device=dev)
    a = L.AttnArgs(dtype=L.MAGI_DTYPE_BF16, D=128, Hq=Hq, Hkv=Hkv, total_q=rows, total_k=far + n, n_ranges=1, max_seqlen_q=rows, max_seqlen_k=stated,
                   q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), k2=k.data_ptr(), v2=v.data_ptr(), k_split=far, out=out.data_ptr(),
                   q_ranges=qr.data_ptr(), k_ranges=kr.data_ptr(), split_workspace=scratch.data_ptr(), split_workspace_bytes=size, **kw,
                   **{"%s_stride_t" % x: (Hkv if x in "kv" else Hq) * 128 for x in "qkvo"}, **{"%s_stride_h" % x: 128 for x in "qkvo"})
    L.check(L.lib().magi_attn_fwd(a, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out, want)


@pytest.mark.parametrize("size", [(24, 8, 1, 432, 1728), (6, 2, 1, 270, 1350), (6, 2, 1, 270, 1601)])
def test_forms_without_pieces_take_no_memory_for_them(dev, monkeypatch, size):
    """Workgroups of 256 rows whatever the sizes take what their last round's items need, the 32x32x16 form and 512 rows nothing."""
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the sizes are chosen for 256 CUs")
    Hq, Hkv, n, rows, mk = size
    lib = L.lib()
    split, pieces = lib.magi_attn_split_bytes_256(*size), lib.magi_attn_pieces_bytes(*size, 1)
    assert max(split, pieces) == lib.magi_attn_split_bytes(*size, L.MAGI_DTYPE_BF16) and split < pieces
    q, k, v, qr, kr, kw = _case(dev, rows, n, Hq, Hkv, [(0, mk)] * n, "as it is")
    real, got = torch.empty, []

    def empty(*a, **o):
        if o.get("dtype") is torch.uint8:
            got.append(a[0])
        return real(*a, **o)

    monkeypatch.setattr(torch, "empty", empty)
    for form, want in (({}, [pieces]), ({"q_tile_rows": 256}, [split] * (split > 0)), ({"q_tile_rows": 512}, []), ({"bounded_mfma32": True}, [])):
        M.range_attention(q, k, v, qr, kr, rows, mk, **kw, **form)
        assert got == want, form
        got.clear()
    M.range_attention(q, k, v, qr, kr, rows, mk, checked=True)
    assert got == [split] * (split > 0)
