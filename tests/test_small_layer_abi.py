"""magi_small_layer's argument struct against the header, and its refusals (no GPU)."""
import ctypes as C
import os
import subprocess

import magi_attn as M
from magi_attn import _lib as L

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_struct_layout_matches_header(tmp_path):
    fields = [f[0] for f in L.SmallLayerArgs._fields_]
    src = ['#include <stdio.h>', '#include <stddef.h>', '#include "magi_attn.h"', 'int main(void){', 'printf("%zu\\n", sizeof(magi_small_layer_args));']
    src += ['printf("%%zu\\n", offsetof(magi_small_layer_args, %s));' % f for f in fields] + ['return 0;}']
    c, exe = tmp_path / "layout.c", tmp_path / "layout"
    c.write_text("\n".join(src))
    subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(c), "-o", str(exe)], check=True)
    out = [int(v) for v in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    assert out == [C.sizeof(L.SmallLayerArgs)] + [getattr(L.SmallLayerArgs, f).offset for f in fields]


def test_refusals():
    lib, a = M.lib(), L.SmallLayerArgs()
    assert lib.magi_small_layer(None, None) == -22
    a.struct_size = C.sizeof(a) - 8
    assert lib.magi_small_layer(C.byref(a), None) == -22 and b"struct_size" in lib.magi_last_error()
    a.struct_size = C.sizeof(a)
    for parts in (0, 4):
        a.parts = parts
        assert lib.magi_small_layer(C.byref(a), None) == -22 and b"parts" in lib.magi_last_error()
    a.parts, a.S, a.K, a.Hq, a.Hkv = 3, 5, 60, 2, 1  # (what the launches refuse)
    assert lib.magi_small_layer(C.byref(a), None) == -38 and b"multiple of 64" in lib.magi_last_error()
    a.parts = 2
    assert lib.magi_small_layer(C.byref(a), None) == 0  # no ranges: nothing to do
