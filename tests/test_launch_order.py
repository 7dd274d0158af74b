"""Two attention calls that share launches where they can: what api.cpp launches, in which order, and whose pieces are in the scratch memory then
(no GPU: linked with host_launches.cpp in place of the kernels)."""
import ctypes as C
import os
import subprocess

import pytest

from magi_attn import _lib as L

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"
SCRATCH, WORKSPACE = 0x7000000, 0x7100000  # (addresses that nobody reads)


@pytest.fixture(scope="module")
def api(tmp_path_factory):
    csrc = os.path.join(ROOT, "magi-1_amd", "csrc")
    so = str(tmp_path_factory.mktemp("host") / "host_launches.so")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-fPIC", "-shared", "-I" + os.path.join(ROOT, "include"), "-I" + csrc,
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument", "-x", "hip",
                    os.path.join(csrc, "api.cpp"), os.path.join(ROOT, "tests", "host_launches.cpp"), "-o", so], check=True)
    lib = C.CDLL(so)
    lib.take_log.restype = C.c_char_p
    lib.magi_last_error.restype = C.c_char_p
    for name in ("magi_attn_fwd_two", "magi_attn_fwd_end"):
        getattr(lib, name).argtypes = [C.POINTER(L.AttnArgs), C.POINTER(L.AttnArgs), C.c_void_p]
    for name in ("magi_attn_fwd", "magi_attn_fwd_begin"):
        getattr(lib, name).argtypes = [C.POINTER(L.AttnArgs), C.c_void_p]
    return lib


def _call(out, rows, keys, kind, n=1, Hq=24, Hkv=8, scratch=SCRATCH, **more):
    """rows of q over keys in each of n ranges; kind: what q and the scores are"""
    e4m3 = kind == "e4m3"
    a = L.AttnArgs(q=0x1000000, k=0x2000000, v=0x3000000, out=out, q_ranges=0x4000000, k_ranges=0x4100000, q_stride_t=Hq * 128, q_stride_h=128,
                   k_stride_t=Hkv * 128, k_stride_h=128, v_stride_t=Hkv * 128, v_stride_h=128, o_stride_t=Hq * 128, o_stride_h=128, total_q=n * rows,
                   total_k=keys, n_ranges=n, max_seqlen_q=rows, max_seqlen_k=keys, Hq=Hq, Hkv=Hkv, D=128, dtype=int(e4m3), split_workspace=scratch,
                   split_workspace_bytes=1 << 40)
    if e4m3:
        a.q_scale = a.k_scale = a.v_scale = 0x5000000
        a.scale_chunk_tokens, a.flags = 64, L.MAGI_ATTN_FP8_POW2_PRESCALED
    elif kind == "as it is":
        a.score_bound, a.flags = 17.0, L.MAGI_ATTN_Q_PRESCALED
    elif kind == "unscaled":
        a.score_bound = 17.0
    elif kind in ("raw", "raw, wavefronts"):
        a.score_bound, a.q_norm_gamma, a.q_norm_eps = 30.0, 0x5100000, 1e-6
        a.flags = L.MAGI_ATTN_SHARE_WAVES if kind != "raw" else 0
    elif kind in ("measured", "checked"):
        a.flags, a.workspace = L.MAGI_ATTN_AUTO_BOUND if kind == "measured" else L.MAGI_ATTN_CHECKED, WORKSPACE
    for name, value in more.items():
        setattr(a, name, value)
    return a


def _launches(api):
    """(launch, [(output, scratch of its pieces, what is done there)], workgroups) of each since the last look"""
    lines = [line.split() for line in api.take_log().decode().splitlines()]
    addr = lambda t: 0 if t == "(nil)" else int(t, 16)
    return [(f[0], [(addr(f[i]), addr(f[i + 1]), f[i + 2]) for i in range(1, len(f) - 1, 3)], int(f[-1])) for f in lines]


def _check_order(launches, first, second):
    """Nothing of the second call ahead of a launch of the first, but for the measurements of a bound; pieces are the call's own when they are
    brought together."""
    whose, seen_second = {}, False
    for name, jobs, _ in launches:
        for out, scratch, does in jobs:
            assert out in (first, second)
            if out == first:
                assert not seen_second, launches
            if does == "w":
                whose[scratch] = out
            elif does == "r":
                assert whose.get(scratch) == out, launches
            elif does == "b":
                whose.pop(scratch, None)
        seen_second |= any(out == second for out, _, _ in jobs) or not jobs
    assert any(out == first for _, jobs, _ in launches for out, _, _ in jobs) and seen_second


SECONDS = [("raw", 480, 4000), ("raw", 2112, 400), ("raw, wavefronts", 96, 400), ("raw", 4200, 3000), ("unscaled", 480, 4000), ("as it is", 480, 4000),
           ("online", 480, 4000), ("measured", 480, 4000), ("checked", 2112, 9000), ("e4m3", 5000, 6000)]


@pytest.mark.parametrize("kind,rows,keys", SECONDS)
@pytest.mark.parametrize("core", [(2112, 14784, 1), (1296, 3888, 3)])  # in pieces; whole items
def test_the_second_half_is_ahead_of_the_second_call(api, core, kind, rows, keys):
    first, second = _call(0x100, core[0], core[1], "as it is", core[2]), _call(0x200, rows, keys, kind)
    _launches(api)
    assert api.magi_attn_fwd_begin(C.byref(first), None) == 1
    assert api.magi_attn_fwd_end(C.byref(first), C.byref(second), None) == 0
    got = _launches(api)
    _check_order(got, 0x100, 0x200)
    # in one launch what the header says, and nothing that is not there
    alone = (kind, rows) not in (("raw", 2112), ("raw", 4200))
    assert (len(got[-1][1]) == 2) != alone
    if alone:  # the launches of the call by itself
        api.magi_attn_fwd(C.byref(second), None)
        mine = _launches(api)
        assert got[-len(mine):] == mine


@pytest.mark.parametrize("kind,rows,keys", SECONDS)
@pytest.mark.parametrize("core", [("as it is", 5400, 7000), ("as it is", 120, 480), ("e4m3", 5400, 9000), ("as it is", 900, 900), ("online", 900, 4000)])
def test_two_calls_are_launched_in_their_order(api, core, kind, rows, keys):
    first, second = _call(0x100, core[1], core[2], core[0]), _call(0x200, rows, keys, kind)
    if core[1] == 120:
        first.flags |= L.MAGI_ATTN_SHARE_WAVES
    _launches(api)
    assert api.magi_attn_fwd_two(C.byref(first), C.byref(second), None) == 0
    _check_order(_launches(api), 0x100, 0x200)


def test_a_refused_second_call_leaves_the_first_done(api):
    for call, first in ((api.magi_attn_fwd_end, _call(0x100, 2112, 14784, "as it is")), (api.magi_attn_fwd_two, _call(0x100, 5400, 7000, "e4m3"))):
        second = _call(0x200, 480, 4000, "online", D=64)
        if call is api.magi_attn_fwd_end:
            assert api.magi_attn_fwd_begin(C.byref(first), None) == 1
        _launches(api)
        assert call(C.byref(first), C.byref(second), None) < 0 and b"head_dim" in api.magi_last_error()
        got = _launches(api)
        assert len(got) == 1 and [out for out, _, _ in got[0][1]] == [0x100]


@pytest.mark.parametrize("kind,rows,keys", [("as it is, wavefronts", 96, 400), ("raw, wavefronts", 96, 400), ("as it is", 480, 4000), ("unscaled", 2112, 14784),
                                            ("online", 2112, 14784), ("measured", 2112, 14784), ("checked", 2112, 14784), ("e4m3", 2112, 14784), ("raw", 0, 400)])
def test_an_end_of_what_was_not_begun_is_refused(api, kind, rows, keys):
    """A form that the first half launches as a whole: the second half launches nothing of it, and nothing beside it."""
    first, second = _call(0x100, rows, keys, kind.split(",")[0]), _call(0x200, 480, 400, "raw")
    if "wavefronts" in kind:
        first.flags |= L.MAGI_ATTN_SHARE_WAVES
    assert api.magi_attn_fwd_begin(C.byref(first), None) == 0
    _launches(api)
    for beside in (None, C.byref(second)):
        assert api.magi_attn_fwd_end(C.byref(first), beside, None) == -22 and b"magi_attn_fwd_end" in api.magi_last_error()
    assert not _launches(api)


@pytest.mark.parametrize("first,entry", [(("as it is", 5400, 7000, 1), "two"), (("e4m3", 5400, 9000, 1), "two"), (("as it is", 1296, 3888, 3), "end"),
                                         (("as it is", 2112, 14784, 1), "end")])
def test_launches_that_fit_apart_only_are_launched_apart(api, first, entry):
    """HIP takes less than 2^32 threads in a launch: 16777215 workgroups of 256.  A long max_seqlen_q, whose tiles lie beyond the rows mostly, is
    just within that by itself (with e4m3 rows and beside pieces in tiles of 128 rows, twice as many), and not with the first call."""
    kind, rows, keys, n = first
    most = 16777215
    calls = [_call(0x100, rows, keys, kind, n), _call(0x200, 4096, 400, "raw")]

    def launches(max_q):
        calls[1].max_seqlen_q = max_q
        if entry == "end":
            assert api.magi_attn_fwd_begin(C.byref(calls[0]), None) == 1
        _launches(api)
        assert getattr(api, "magi_attn_fwd_" + entry)(C.byref(calls[0]), C.byref(calls[1]), None) == 0
        got = _launches(api)
        assert all(w <= most for _, _, w in got) and sum(len(jobs) for _, jobs, _ in got) == 2
        return got

    per_tile = 24  # (workgroups of all heads)
    tile = 128 if kind == "e4m3" or rows == 2112 else 256
    whole = launches(256 * (most // per_tile - 100))
    assert len(whole) == (2 if tile == 128 else 1)
    others = launches(256 * 1024)[0][2] - 1024 * (256 // tile) * per_tile  # of the first call
    edge = (most - others) // per_tile
    got = launches(tile * edge)
    assert len(got) == 1 and got[0][2] == others + edge * per_tile
    assert len(launches(tile * edge + 1)) == 2


@pytest.mark.parametrize("keys", [1, 31, 32, 33])
def test_less_than_a_slab_of_keys_is_shared_beside_another_small_call_only(api, keys):
    waves = lambda out, n, kind: _call(out, 96, n, kind, flags=L.MAGI_ATTN_SHARE_WAVES | (L.MAGI_ATTN_Q_PRESCALED if kind == "as it is" else 0))
    core, text = waves(0x100, keys, "as it is"), waves(0x200, keys, "raw")
    name = lambda: [(f[0], len(f[1])) for f in _launches(api)]
    of_one = [("launch_attn_fwd_bf16_x16" if keys < 32 else "launch_attn_fwd_bf16_waves", 1)]
    both = [("launch_attn_fwd_bf16_waves", 2)]
    name()
    for call in (core, text):
        assert api.magi_attn_fwd(C.byref(call), None) == 0 and name() == of_one
    assert api.magi_attn_fwd_begin(C.byref(core), None) == 0 and name() == of_one
    for a, b in ((core, text), (core, waves(0x200, 400, "raw")), (waves(0x100, 400, "as it is"), text)):
        assert api.magi_attn_fwd_two(C.byref(a), C.byref(b), None) == 0 and name() == both
    large = _call(0x300, 4200, 3000, "as it is")
    for a, b in ((core, large), (large, core)):  # (and no other call in the launch)
        assert api.magi_attn_fwd_two(C.byref(a), C.byref(b), None) == 0 and sorted(name()) == sorted(of_one + [("launch_attn_fwd_bf16_x16", 1)])
