"""The launches that two attention calls share, in each of their forms, against the calls one by one: on a stream that is not the default one, from two
threads, with q of a batch, and with infinities and NaN among the keys and values."""
import math
import threading

import pytest
import torch

from magi_attn import _lib as L
from magi_attn.functional import BegunCalls, launch_held, quantize_fp8, range_attention

pytestmark = pytest.mark.gpu
D, PRE = 128, 128 ** -0.5 * 1.4426950408889634
FORMS = ["waves", "pair", "e4m3", "pieces", "whole"]
# form: query and key heads, chunks, rows and (core) prefix chunks of a chunk, text of each chunk
SIZES = {"waves": (6, 2, 2, 120, 2, (24, 33)), "pair": (24, 8, 2, 2800, 0, (70, 129)), "e4m3": (24, 8, 2, 640, 1, (64, 65)),
         "pieces": (24, 8, 1, 2310, 2, (97,)), "whole": (24, 8, 3, 1296, 0, (330, 1, 65))}


class _Calls:
    """The core and the text attention of a layer; odd = (key or value, its place, its value) in both."""

    def __init__(self, dev, form, seed=0, batch=False, odd=None):
        Hq, Hkv, n, Lc, prefix, text = SIZES[form]
        g = torch.Generator(device=dev).manual_seed(seed)
        S, K, T = n * Lc, (n + prefix) * Lc, sum(text)
        rows = lambda *s: torch.nn.functional.layer_norm(torch.randn(*s, D, device=dev, generator=g), (D,)).bfloat16()
        self.form, self.Lc, self.K = form, Lc, K
        self.q, self.k, self.v = (rows(S, Hq).float() * PRE).bfloat16(), rows(K, Hkv), torch.randn(K, Hkv, D, device=dev, generator=g).bfloat16()
        self.qx, self.kx, self.vx = rows(S, Hq), rows(T, Hkv), torch.randn(T, Hkv, D, device=dev, generator=g).bfloat16()
        if odd:
            which, at, value = odd
            for t in ((self.k, self.kx) if which == "k" else (self.v, self.vx)):
                t[at if at >= 0 else t.shape[0] + at, 0, 5] = value
        self.gamma = torch.randn(D, device=dev, generator=g) * 0.1
        pairs = lambda r: torch.tensor(r, dtype=torch.int32, device=dev)
        self.q_ranges, self.k_ranges = pairs([[i * Lc, (i + 1) * Lc] for i in range(n)]), pairs([[0, (prefix + i + 1) * Lc] for i in range(n)])
        self.cu_q = torch.arange(0, S + 1, Lc, dtype=torch.int32, device=dev)
        self.cu_k = pairs([0] + list(text)).cumsum(0).to(torch.int32)
        if batch:  # [position, batch] rows, the batch outermost
            turn = lambda t: t.view(n, Lc, Hq, D).transpose(0, 1).contiguous().transpose(0, 1)
            self.q, self.qx = turn(self.q), turn(self.qx)
        if form == "e4m3":
            self.q, self.qs = quantize_fp8(self.q, Lc, 1.0, True)
            self.k, self.ks = quantize_fp8(self.k, Lc, 1.0, True)
            self.v, self.vs = quantize_fp8(self.v, Lc, 1.0, True)

    def core(self, held=None):
        if self.form == "e4m3":
            return range_attention(self.q, self.k, self.v, self.q_ranges, self.k_ranges, self.Lc, self.K, q_scale=self.qs, k_scale=self.ks, v_scale=self.vs,
                                   scale_chunk_tokens=self.Lc, fp8_pow2_prescaled=True, return_lse=False, held=held)[0]
        return range_attention(self.q, self.k, self.v, self.q_ranges, self.k_ranges, self.Lc, self.K, return_lse=False, q_prescaled=True, score_bound=20.0,
                               share_waves=True, held=held)[0]

    def text(self, held=None, split=True):
        return range_attention(self.qx, self.kx, self.vx, self.cu_q, self.cu_k, self.Lc, 330, ranges_mode=L.MAGI_RANGES_CU, return_lse=False, score_bound=30.0,
                               q_norm=(self.gamma, None, 1e-6), share_waves=split, held=held, split_keys=split)[0]

    def one_by_one(self):
        return self.core(), self.text(split=self.form == "waves")  # (whole items in a shared launch)

    def together(self):
        held = BegunCalls() if self.form in ("pieces", "whole") else []
        out = self.core(held), self.text(held)
        before = L.lib().magi_launch_count()
        launch_held(held)
        self.launches = L.lib().magi_launch_count() - before
        return out


def _same(got, want):
    return all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(got, want))


@pytest.mark.parametrize("form", FORMS)
def test_on_a_stream_of_its_own(dev, form):
    c = _Calls(dev, form)
    want = c.one_by_one()
    stream = torch.cuda.Stream()
    for _ in range(3):
        # work ahead of the call on that stream, which the launches have to wait for: q comes late
        q, fresh = c.q, torch.zeros_like(c.q.view(torch.uint8)).view(c.q.dtype)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            torch.cuda._sleep(2_000_000)
            fresh.view(torch.uint8).copy_(q.view(torch.uint8))
            c.q = fresh
            got = c.together()
        stream.synchronize()
        c.q = q
        assert _same(got, want)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert c.launches == 1


@pytest.mark.parametrize("forms", [("waves", "pair"), ("e4m3", "pieces"), ("whole", "e4m3"), ("pieces", "pieces")])
def test_from_two_threads(dev, forms):
    calls = [_Calls(dev, f, seed=i) for i, f in enumerate(forms)]
    want = [c.one_by_one() for c in calls]
    torch.cuda.synchronize()
    bad, start = [], threading.Barrier(2)

    def work(i):
        try:
            with torch.cuda.device(dev), torch.cuda.stream(torch.cuda.Stream()):
                start.wait(30)
                for _ in range(8):
                    got = calls[i].together()
                    torch.cuda.current_stream().synchronize()
                    if not _same(got, want[i]):
                        bad.append(forms[i])
        except Exception as e:  # noqa: BLE001 (shown by the assertion)
            bad.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not bad and not any(t.is_alive() for t in threads)


@pytest.mark.parametrize("form", ["waves", "pair", "whole"])
def test_q_of_a_batch(dev, form):
    """(e4m3 rows have no batch)"""
    flat, c = _Calls(dev, form), _Calls(dev, form, batch=True)
    want = flat.one_by_one()
    got = c.together()
    assert c.q.dim() == 4 and _same([t.reshape(w.shape) for t, w in zip(got, want)], want)
    assert _same(got, c.one_by_one())


# the first key, one in the middle, the last one, whose copies fill the ragged end of a tile
@pytest.mark.parametrize("at", [0, 40, -1])
@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("which", ["k", "v"])
@pytest.mark.parametrize("form", FORMS)
def test_infinities_and_nan(dev, form, which, value, at):
    """The same rows and features are not finite, whatever shares the launch; the others have the same bits (shared keys: fp32 sums of up to 480
    terms of a few units in another order, and a bf16 step)."""
    c = _Calls(dev, form, odd=(which, at, value))
    got, want = c.together(), c.one_by_one()
    if form == "waves":  # (against the forms that do not share keys: sums in another order where they are finite)
        want = [range_attention(c.q, c.k, c.v, c.q_ranges, c.k_ranges, c.Lc, c.K, return_lse=False, q_prescaled=True, score_bound=20.0, split_keys=False)[0],
                c.text(split=False)]
    for a, b in zip(got, want):
        if form == "waves":
            assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isposinf(a), torch.isposinf(b))
            assert torch.equal(torch.isneginf(a), torch.isneginf(b))
            fin = torch.isfinite(b)
            assert ((a - b)[fin].float().abs() <= 2.0 ** -7 * b[fin].float().abs() + 2.0 ** -9).all()
        else:
            assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a[~torch.isnan(a)], b[~torch.isnan(b)])
