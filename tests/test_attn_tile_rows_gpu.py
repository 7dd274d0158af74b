"""The bounded-score kernel in workgroups of 128 rows: which launches take it, and that a row's bits are those of the 256-row workgroups
(which are checked against the oracle by the tests that force them, and whose launches are the ones of the larger tests)."""
import pytest
import torch

import magi_attn as M
from magi_attn import _lib as L

D, PRE = 128, 128 ** -0.5 * 1.4426950408889634


def _rows(g, dev, *shape):
    x = torch.randn(*shape, device=dev, generator=g, dtype=torch.bfloat16)
    return torch.nn.functional.layer_norm(x, (D,))


def _kernels(call):
    """What call() returns, and the names of the attention kernels that ran in it."""
    from torch.profiler import ProfilerActivity, profile

    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        out = call()
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if "attn_fwd_bf16" in e.name]
    if not names:
        pytest.skip("the profiler records no kernels here: nothing says which of them ran")
    return out, names


# rows around 32 (a wavefront), 128 and 256 (a workgroup); keys around half a tile and a tile; one and several ranges, an empty one,
# rows that no range covers, ranges in another order, a key axis in two pieces
@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["as it is", "scaled", "normed"])
@pytest.mark.parametrize("Hq,Hkv,Tq,q_ranges,k_ranges,k_split", [
    (1, 1, 1, [(0, 1)], [(0, 1)], None), (6, 2, 31, [(0, 31)], [(3, 35)], 20), (2, 2, 129, [(0, 33), (33, 129)], [(0, 64), (10, 75)], 64),
    (24, 8, 260, [(130, 257), (0, 128)], [(5, 5), (0, 97)], None), (3, 1, 515, [(0, 257), (260, 510)], [(0, 321), (100, 130)], 200)])
def test_rows_of_the_smaller_workgroups_have_the_same_bits(dev, mode, Hq, Hkv, Tq, q_ranges, k_ranges, k_split):
    g = torch.Generator(device=dev).manual_seed(Tq)
    Tk = max(e for _, e in k_ranges)
    q, kv = _rows(g, dev, Tq, Hq, D), torch.randn(Tk, Hkv, 2 * D, device=dev, generator=g, dtype=torch.bfloat16)
    k, v = torch.nn.functional.layer_norm(kv[..., :D], (D,)), kv[..., D:]
    qr, kr = (torch.tensor(r, dtype=torch.int32, device=dev) for r in (q_ranges, k_ranges))
    kw = {"score_bound": 20.0}
    if mode == "as it is":
        q, kw["q_prescaled"] = (q.float() * PRE).bfloat16(), True
    elif mode == "normed":
        kw["q_norm"] = (torch.randn(D, device=dev, generator=g) * 0.1, torch.randn(D, device=dev, generator=g) * 0.1, 1e-6)
    if k_split is not None:
        k2, v2 = (torch.empty(Tk - k_split, Hkv, 2 * D, device=dev, dtype=torch.bfloat16)[..., :D] for _ in range(2))
        k = torch.empty(Tk, Hkv, 2 * D, device=dev, dtype=torch.bfloat16)[..., :D].copy_(k)
        k2.copy_(k[k_split:])
        v2.copy_(v[k_split:])
        kw.update(k2=k2, v2=v2, k_split=k_split)
        k, v = k[:k_split], v[:k_split]
    most_q, most_k = max(e - b for b, e in q_ranges), max(e - b for b, e in k_ranges)
    call = lambda rows, **o: M.range_attention(q, k, v, qr, kr, most_q, most_k, q_tile_rows=rows, split_keys=False, **kw, **o)  # noqa: E731
    (a, la), ran = _kernels(lambda: call(0))
    (b, lb), ran_256 = _kernels(lambda: call(256))
    assert torch.equal(a, b) and torch.equal(la, lb)
    form = {"as it is": 0, "normed": 1, "scaled": 2}[mode]
    for names, blocks in ((ran, 2), (ran_256, 4)):  # (query blocks of 16 rows per wavefront: the two forms that were compared)
        assert len(names) == 1 and f"attn_fwd_bf16_x16_kernel<{form}, {blocks}>" in names[0], names
    if Hq % 2 == 0:  # grouped outputs
        o = [torch.full((Tq, 2, 2, Hq // 2, D), 3.0, device=dev, dtype=torch.bfloat16) for _ in range(2)]
        call(0, out=o[0][:, :, 1])
        call(256, out=o[1][:, :, 1])
        assert torch.equal(o[0], o[1])
    if len(q_ranges) == 1 and Tq > 1 and k_split is None:  # a batch of [position, batch] rows
        two = torch.stack([q, q], 1).transpose(0, 1)
        qr2, kr2 = torch.cat([qr, qr + Tq]), torch.cat([kr, kr])
        x, _ = M.range_attention(two, k, v, qr2, kr2, most_q, most_k, return_lse=False, split_keys=False, **kw)
        assert torch.equal(x[0], a) and torch.equal(x[1], a)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,prefix,Hq,Hkv,split,smaller", [
    (240, 2, 2, 6, 2, True, True), (2600, 1, 0, 24, 8, True, True), (3800, 1, 0, 24, 8, True, False), (240, 1, 13, 24, 8, True, False),
    (240, 1, 13, 24, 8, False, True), (2600, 1, 4, 24, 8, True, True), (1300, 1, 3, 24, 8, True, False), (1000, 3, 2, 24, 8, True, False)])
def test_which_launches_take_the_smaller_workgroups(dev, rows, n, prefix, Hq, Hkv, split, smaller):
    """By the name of the kernel that runs; no launch behind it that adds pieces up."""
    q, kv = (torch.randn(r, h, 2 * D, device=dev, dtype=torch.bfloat16) * 0.1 for r, h in ((n * rows, Hq), ((n + prefix) * rows, Hkv)))
    qr = torch.tensor([[i * rows, (i + 1) * rows] for i in range(n)], dtype=torch.int32, device=dev)
    kr = torch.tensor([[0, (prefix + i + 1) * rows] for i in range(n)], dtype=torch.int32, device=dev)
    _, names = _kernels(lambda: M.range_attention(q[..., :D], kv[..., :D], kv[..., D:], qr, kr, rows, (n + prefix) * rows, q_prescaled=True,
                                                  score_bound=60.0, split_keys=split, return_lse=False))
    assert any("x16_kernel<0, 2>" in x for x in names) == smaller, names
    assert not (smaller and any("merge" in x for x in names)), names


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,prefix,Hq,Hkv,smaller", [(2600, 1, 4, 24, 8, True), (1300, 1, 3, 24, 8, False)])
def test_launches_of_smaller_workgroups_allocate_no_scratch_memory(dev, monkeypatch, rows, n, prefix, Hq, Hkv, smaller):
    """As the library says which they are; checked launches, in 256-row workgroups always, do."""
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the sizes are chosen for 256 CUs")
    Tk = (n + prefix) * rows
    size = (Hq, Hkv, n, rows, Tk)
    asked = L.lib().magi_attn_split_bytes(*size, L.MAGI_DTYPE_BF16)
    assert asked > 0 and (L.lib().magi_attn_tile_rows(*size, asked) == 128) == smaller and L.lib().magi_attn_tile_rows(*size, 0) == 128
    q, kv = (torch.randn(r, h, 2 * D, device=dev, dtype=torch.bfloat16) * 0.1 for r, h in ((rows, Hq), (Tk, Hkv)))
    qr, kr = (torch.tensor([[0, e]], dtype=torch.int32, device=dev) for e in (rows, Tk))
    call = lambda **kw: M.range_attention(q[..., :D], kv[..., :D], kv[..., D:], qr, kr, rows, Tk, return_lse=False, **kw)[0]  # noqa: E731
    whole, real, got = call(split_keys=False, score_bound=60.0), torch.empty, []

    def empty(*a, **kw):
        if kw.get("dtype") is torch.uint8:
            got.append(a[0])
        return real(*a, **kw)

    monkeypatch.setattr(torch, "empty", empty)
    assert torch.equal(call(score_bound=60.0), whole) == smaller and got == ([] if smaller else [asked])
    call(checked=True)
    assert got[-1] == asked
