"""CPU tests of the host side: range generators and rope table of the product against the
oracle and the reference's worked examples, the metadata builders, and the C-ABI library
(loads, exports every declared symbol, rejects bad arguments before touching a GPU)."""
import copy
import ctypes as C
import os
import re

import numpy as np
import pytest
import torch

import magi_attn
from magi_attn import _lib as L
from magi_attn import params as P
from magi_attn import ranges as R
from magi_attn import rope as RP
from oracle import magi_oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_loads_and_exports_every_declared_symbol():
    lib = magi_attn.lib()
    assert lib.magi_version() >= 100
    header = open(os.path.join(ROOT, "include", "magi_attn.h")).read()
    declared = set(re.findall(r"\b(magi_[a-z0-9_]+)\s*\(", header))
    assert declared == set(L.EXPORTS), declared ^ set(L.EXPORTS)
    for name in declared:
        assert hasattr(lib, name), name


def test_measurement_library_exports_what_its_header_declares():
    """libmagi_probe.so (MFMA-only and streaming loops that bench.py reports its ceilings from) is built by the same
    Makefile; nothing in the package loads it.  No compute call without a GPU: argument checks only."""
    path = os.path.join(ROOT, "magi-1_amd", "magi_attn", "libmagi_probe.so")
    assert os.path.exists(path), "build it with `make -C magi-1_amd/csrc`"
    lib = C.CDLL(path)
    header = open(os.path.join(ROOT, "magi-1_amd", "csrc", "probe", "magi_probe.h")).read()
    declared = re.findall(r"\b(magi_probe_\w+)\s*\(", header)
    assert sorted(set(declared)) == ["magi_probe_mfma_only", "magi_probe_stream"]
    for name in declared:
        assert hasattr(lib, name), name
    lib.magi_probe_stream.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p, C.POINTER(C.c_float)]
    lib.magi_probe_stream.restype = C.c_int
    ms = C.c_float(0)
    assert lib.magi_probe_stream(7, None, None, 1024, 1, None, C.byref(ms)) == -22      # unknown kind
    assert lib.magi_probe_stream(0, None, None, 1024, 1, None, C.byref(ms)) == -22      # no buffers
    assert lib.magi_probe_stream(2, None, C.c_void_p(256), 1000, 1, None, C.byref(ms)) == -22  # not a multiple of 16
    for pkg_file in os.listdir(os.path.join(ROOT, "magi-1_amd", "magi_attn")):
        if pkg_file.endswith(".py"):
            assert "magi_probe" not in open(os.path.join(ROOT, "magi-1_amd", "magi_attn", pkg_file)).read(), pkg_file


def test_missing_library_is_an_error_not_a_fallback(tmp_path):
    """The library beside the package is the only compute path: when it is not there the first call raises (checked
    in a child process on a copy of the package without its .so; no environment variable redirects the loader)."""
    import shutil
    import subprocess
    import sys

    pkg = tmp_path / "magi_attn"
    shutil.copytree(os.path.join(ROOT, "magi-1_amd", "magi_attn"), pkg,
                    ignore=shutil.ignore_patterns("*.so", "__pycache__"))
    code = (
        "import sys; sys.path.insert(0, %r)\n"
        "import magi_attn._lib as L\n"
        "assert L.LIB_PATH.startswith(%r), L.LIB_PATH\n"
        "try:\n"
        "    L.lib()\n"
        "except RuntimeError as e:\n"
        "    assert 'no fallback' in str(e), e; print('raised')\n"
    ) % (str(tmp_path), str(pkg))
    env = dict(os.environ, MAGI_ATTN_LIBRARY=os.path.join(ROOT, "magi-1_amd", "magi_attn", "libmagi_attn.so"))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env=env, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "raised", (r.stdout, r.stderr[-2000:])


def test_struct_layouts_match_header(tmp_path):
    """ctypes mirrors vs the C compiler's view of include/magi_attn.h (sizes and field offsets)."""
    import subprocess

    pairs = (("magi_attn_args", L.AttnArgs), ("magi_prologue_args", L.PrologueArgs),
             ("magi_qkv_proj_args", L.QkvProjArgs), ("magi_quantize_args", L.QuantizeArgs))
    src = ['#include <stdio.h>', '#include <stddef.h>', '#include "magi_attn.h"', 'int main(void){']
    for cname, mirror in pairs:
        src += ['printf("%%zu\\n", sizeof(%s));' % cname]
        src += ['printf("%%zu\\n", offsetof(%s, %s));' % (cname, f[0]) for f in mirror._fields_]
    src += ['return 0;}']
    c = tmp_path / "layout.c"
    c.write_text("\n".join(src))
    exe = tmp_path / "layout"
    subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(c), "-o", str(exe)], check=True)
    out = [int(x) for x in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    pos = 0
    for cname, mirror in pairs:
        names = [f[0] for f in mirror._fields_]
        assert names[0] == "struct_size" and getattr(mirror, "struct_size").offset == 0
        assert out[pos] == C.sizeof(mirror), cname
        assert out[pos + 1:pos + 1 + len(names)] == [getattr(mirror, f).offset for f in names], cname
        assert mirror().struct_size == C.sizeof(mirror)  # filled in by the mirror's constructor
        pos += 1 + len(names)
    assert pos == len(out)


def test_a_struct_of_another_size_is_refused():
    """Every argument struct starts with its size as the caller compiled it; a caller built against another
    version of the header (a shorter or longer struct) gets MAGI_EINVAL instead of having fields read that it
    never wrote.  The Python mirrors are bound to one library version and refuse to load another."""
    lib = magi_attn.lib()
    assert lib.magi_version() == L.ABI_VERSION
    for mk, fn in ((L.AttnArgs, lib.magi_attn_fwd), (L.PrologueArgs, lib.magi_qk_prologue),
                   (L.QkvProjArgs, lib.magi_qkv_proj_prologue), (L.QuantizeArgs, lib.magi_quantize_fp8_split)):
        a = mk()
        for wrong in (0, a.struct_size - 8, a.struct_size + 8):
            a.struct_size = wrong
            assert fn(C.byref(a), None) == -22 and b"struct_size" in lib.magi_last_error(), mk.__name__
    assert isinstance(lib.magi_launch_count(), int)


def test_attn_argument_validation_without_gpu():
    lib = magi_attn.lib()
    a = L.AttnArgs()
    a.D, a.Hq, a.Hkv = 64, 4, 2
    assert lib.magi_attn_fwd(C.byref(a), None) == -38  # head_dim not implemented
    assert b"head_dim" in lib.magi_last_error()
    a.D, a.Hq, a.Hkv = 128, 5, 2
    assert lib.magi_attn_fwd(C.byref(a), None) == -22
    a.Hq = 4
    a.dtype = 7
    assert lib.magi_attn_fwd(C.byref(a), None) == -22
    a.dtype = 0
    a.n_ranges = 0
    assert lib.magi_attn_fwd(C.byref(a), None) == 0  # nothing to do
    a.n_ranges, a.total_q, a.max_seqlen_q = 1, 8, 8
    assert lib.magi_attn_fwd(C.byref(a), None) == -22  # NULL q
    assert b"NULL" in lib.magi_last_error()
    a.q = a.out = a.q_ranges = a.k_ranges = 4096
    a.q_stride_t = a.o_stride_t = 512
    a.q_stride_h = a.o_stride_h = 128
    a.k_stride_t, a.k_stride_h, a.v_stride_t, a.v_stride_h = 256, 128, 256, 100
    assert lib.magi_attn_fwd(C.byref(a), None) == -22  # misaligned stride
    a.v_stride_h = 128
    a.k = a.v = 4096
    a.total_k = 8
    a.out_group_heads = 3  # does not divide Hq = 4
    assert lib.magi_attn_fwd(C.byref(a), None) == -22 and b"out_group_heads" in lib.magi_last_error()
    assert lib.magi_attn_fwd(None, None) == -22


def test_prologue_argument_validation_without_gpu():
    lib = magi_attn.lib()
    p = L.PrologueArgs()
    p.D = 64
    assert lib.magi_qk_prologue(C.byref(p), None) == -38
    p.D, p.S = 128, 0
    assert lib.magi_qk_prologue(C.byref(p), None) == 0
    p.S, p.Hq, p.Hkv, p.R2 = 4, 2, 1, 44
    assert lib.magi_qk_prologue(C.byref(p), None) == -22 and b"R2" in lib.magi_last_error()
    p.R2 = 48
    assert lib.magi_qk_prologue(C.byref(p), None) == -22  # NULL buffers
    assert lib.magi_head_norm(None, 0, 0, None, None, None, 4, 2, 128, 0, 1e-6, None) == -22
    # layer norm: validation happens before any device work
    buf = (C.c_char * 64)()
    p16 = (C.addressof(buf) + 15) & ~15
    assert lib.magi_layer_norm(None, 64, None, None, 0, None, 64, 0, 64, 1e-5, None) == 0  # no rows: nothing to do
    assert lib.magi_layer_norm(None, 64, None, None, 0, None, 64, 4, 64, 1e-5, None) == -22
    assert lib.magi_layer_norm(p16, 64, None, None, 0, p16, 64, 4, 60, 1e-5, None) == -38  # cols % 8
    assert lib.magi_layer_norm(p16, 64, None, None, 0, p16, 64, 4, 8200, 1e-5, None) == -38
    assert lib.magi_layer_norm(p16, 32, None, None, 0, p16, 64, 4, 64, 1e-5, None) == -22  # stride < cols
    assert lib.magi_layer_norm(p16 + 2, 64, None, None, 0, p16, 64, 4, 64, 1e-5, None) == -22  # alignment
    assert b"magi_layer_norm" in lib.magi_last_error()
    assert lib.magi_apply_rotary(None, None, None, None, 1, 4, 2, 128, 80, 0, None) == -22


def test_generate_sequences_reference_examples_and_oracle():
    assert R.generate_sequences(8, 4, 2) == ([2, 2, 2, 2, 3, 4, 5, 6, 7], [3, 4, 5, 6, 7, 8, 8, 8, 8],
                                             [0, 0, 0, 0, 0, 0, 1, 2, 3], [1, 2, 3, 4, 4, 4, 4, 4, 4])
    for args in [(8, 8, 0), (8, 4, 0), (8, 1, 0), (12, 4, 3), (5, 7, 1), (1, 1, 0)]:
        assert R.generate_sequences(*args) == O.generate_sequences(*args)


def test_kvrange_generators_match_oracle():
    L_ = 9360
    for sp, dn in [(0, 1), (0, 4), (4, 4), (8, 4), (3, 2)]:
        assert np.array_equal(R.generate_default_kvrange(sp, dn, L_).numpy(), O.default_kvrange(sp, dn, L_))
        steps = [32, 17, 8, 0][:dn]
        a = R.generate_noise2clean_kvrange(sp, dn, L_, [5, 4, 3, 2], 1, steps, 32).numpy()
        assert np.array_equal(a, O.noise2clean_kvrange(sp, dn, L_, [5, 4, 3, 2], 1, steps, 32))
        assert a.dtype == np.int32
        b = R.generate_kvrange_for_denoising_video(sp, dn, L_, [], -1, steps, 32).numpy()
        assert np.array_equal(b, O.default_kvrange(sp, dn, L_))
    assert np.array_equal(R.generate_kvrange_for_prefix_video(5, L_, 1).numpy(), O.prefix_video_kvrange(5, L_, 1))
    assert np.array_equal(R.generate_kvrange_for_prefix_video(5, L_, -1, [5, 4, 3, 2]).numpy(),
                          O.prefix_video_kvrange(5, L_, -1, [5, 4, 3, 2]))
    assert np.array_equal(R.generate_kv_range_for_uncondition(4, L_).numpy(), O.uncondition_kvrange(4, L_))
    assert np.array_equal(R.q_ranges_from_chunks(4, L_).numpy(), O.q_ranges_for(4, L_))
    # batch > 1 offsets every row by b * range_num chunks (video_generate.py:461-463)
    two = R.generate_default_kvrange(1, 2, 10, batch_size=2).tolist()
    assert two == [[0, 20], [0, 30], [30, 50], [30, 60]]
    with pytest.raises(ValueError):
        R.generate_noise2clean_kvrange(0, 2, 10, [5, 4, 3], 1, [0, 0], 32)


def test_rope_module_matches_oracle():
    m = RP.LearnableRotaryEmbeddingCat(128)
    assert torch.equal(m.bands.detach(), O.freq_bands(16))
    for T, H, W, sp, dn in [(6, 4, 6, 2, 3), (2, 16, 16, 0, 1), (4, 8, 13, 5, 2)]:
        a = m.get_embed_for_forward(T, H, W, sp, dn)
        b = O.rope_for_forward(T, H, W, sp, dn)
        assert a.shape == (T * H * W, 96) and torch.equal(a, b)
    assert torch.equal(m.get_embed([3, 4, 6]), O.rope_table(3, 4, 6))
    # the reference's two builder functions by name: (sin, cos) halves of the same table, and their per-axis form
    sin, cos = RP.build_rotary_pos_embed([3, 4, 6], bands=m.bands.detach(), dim=128)
    assert sin.shape == cos.shape == (72, 48) and torch.equal(torch.cat([sin, cos], -1), O.rope_table(3, 4, 6))
    f_sin, f_cos = RP.build_fourier_pos_embed([3, 4, 6], num_bands=16)
    assert f_sin.shape == (3, 4, 6, 3, 16) and torch.equal(f_sin.reshape(72, 48), sin) and torch.equal(f_cos.reshape(72, 48), cos)
    assert torch.equal(f_sin[2, 1, 5, 0], torch.sin(2.0 * RP.freq_bands(16)))            # axis 0 is time: position 2
    with pytest.raises(NotImplementedError):
        RP.build_rotary_pos_embed([3, 4, 6], in_pixels=True)
    assert RP.LearnableRotaryEmbeddingCat(128, in_pixels=False).bands.shape == (16,)


def test_param_builders():
    qr = torch.tensor([[0, 10], [10, 20]], dtype=torch.int32)
    kr = torch.tensor([[20, 50], [10, 60]], dtype=torch.int32)
    p = P.build_core_attn_params(qr, kr, 10)
    assert p.max_seqlen_k == 50 and p.max_seqlen_q == 10 and p.np_k_range.tolist() == kr.tolist()
    mask = torch.zeros(3, 1, 1, 16)
    mask[0, ..., :7] = 1
    mask[2, ..., :3] = 1
    x = P.build_cross_attn_params(mask, 10, 800)
    cq, ck, qr2, kr2 = O.cross_attn_params_from_mask(mask.reshape(3, 16), 10)
    assert torch.equal(x.cu_seqlens_q, cq) and torch.equal(x.cu_seqlens_kv, ck)
    assert torch.equal(x.q_ranges, qr2) and torch.equal(x.kv_ranges, kr2)
    assert x.cu_seqlens_q.dtype == torch.int32 and x.max_seqlen_kv == 800
    ip = P.InferenceParams(1, 100)
    assert ip.key_value_memory_dict == {} and ip.update_kv_cache is False


def test_functional_rejects_cpu_tensors():
    q = torch.zeros(4, 2, 128, dtype=torch.bfloat16)
    r = torch.zeros(1, 2, dtype=torch.int32)
    with pytest.raises(ValueError):
        magi_attn.range_attention(q, q, q, r, r, 4)


def test_kv_cache_arena_views_accounting_and_errors():
    from magi_attn.cache import KVCacheArena
    # the 24B 720p figure of the design notes: 48 layers x 259200 tokens x 8 heads x 256 x 2 B = 51 GB
    assert KVCacheArena.bytes_needed(48, 259200, 8) == 48 * 259200 * 8 * 256 * 2
    arena = KVCacheArena(3, 40, 2, device="cpu")
    ip = P.InferenceParams(1, 40)
    d = arena.attach(ip, layer_numbers=[5, 6, 7])
    assert sorted(d) == [5, 6, 7] and d[6].shape == (40, 2, 256)
    d[6][3, 1, 200] = 2.5  # a view: writes land in the arena, layers do not overlap
    assert arena.layer(1)[3, 1, 200] == 2.5 and arena.buffer.data_ptr() == d[5].data_ptr()
    assert d[7].data_ptr() - d[6].data_ptr() == 40 * 2 * 256 * 2
    with pytest.raises(ValueError):
        arena.attach(P.InferenceParams(1, 41))
    with pytest.raises(ValueError):
        arena.attach(ip, layer_numbers=[1, 1, 2])
    with pytest.raises(MemoryError):
        KVCacheArena(48, 259200, 8, device="cpu", memory_budget_bytes=1 << 30)
    with pytest.raises(ValueError):
        KVCacheArena(1, 8, 1, device="cpu", kv_offload=True)   # the staging buffers need a GPU
    with pytest.raises(ValueError):
        KVCacheArena(1, 8, 1, device="cuda", kv_offload=True, max_batch_size=2)
    with pytest.raises(MemoryError):                              # with kv_offload the budget counts the staging ring
        KVCacheArena(48, 259200, 8, device="cuda", kv_offload=True, memory_budget_bytes=1 << 30)


def test_projection_weights_share_one_buffer():
    """q / k / v / qx keep the reference's parameter names but are rows of one buffer, so one GEMM serves all four;
    the sharing survives load_state_dict and is re-established after a dtype / device move."""
    from magi_attn.module import CustomLayerNormLinear

    torch.manual_seed(0)
    m = CustomLayerNormLinear(64, 48, 16, dtype=torch.float32)
    assert sorted(n for n, _ in m.named_parameters()) == ["k.weight", "layer_norm.bias", "layer_norm.weight", "q.weight",
                                                          "qx.weight", "v.weight"]
    w = m.fused_weight()
    assert w.shape == (128, 64) and w.data_ptr() == m.q.weight.data_ptr()
    x = torch.randn(5, 1, 64)
    q, k, v, qx = m.forward_qkvx(x)
    for got, lin in ((q, m.forward_q), (k, m.forward_k), (v, m.forward_v), (qx, m.forward_qx)):
        assert torch.allclose(got, lin(x), atol=1e-6)
    sd = {n: torch.randn_like(t) for n, t in m.state_dict().items()}
    m.load_state_dict(sd)
    w2 = m.fused_weight()
    assert w2.data_ptr() == w.data_ptr()  # copied in place, still shared
    assert torch.equal(w2, torch.cat([sd["q.weight"], sd["k.weight"], sd["v.weight"], sd["qx.weight"]]))
    m = m.to(torch.bfloat16)  # re-allocates every parameter: the buffer is rebuilt on the next call
    w3 = m.fused_weight()
    assert w3.dtype == torch.bfloat16 and w3.data_ptr() == m.q.weight.data_ptr()
    assert m.k.weight.data_ptr() == w3.data_ptr() + 48 * 64 * 2
    assert torch.equal(w3[80:], sd["qx.weight"].bfloat16())


def test_projection_buffer_is_released_and_wrapped_weights_are_read_through_their_attribute():
    """The shared buffer lives as long as the parameters in it and no longer; a parametrised weight, which is no parameter
    under its name, is read through its attribute; forward_qkvx runs on the CPU and carries gradients and tangents at sizes
    whose rows the device path cuts in two."""
    from torch.multiprocessing.reductions import StorageWeakRef

    from magi_attn.module import CustomLayerNormLinear, FusedLayerNorm

    class Double(torch.nn.Module):
        def forward(self, w):
            return 2 * w

    m = CustomLayerNormLinear(64, 48, 16, dtype=torch.float32)
    buffer = StorageWeakRef(m.fused_weight().untyped_storage())
    m = m.to(torch.bfloat16)
    assert buffer.expired()
    for lin in (m.q, m.v):
        lin.weight.data.normal_()
    torch.nn.utils.parametrize.register_parametrization(m.v, "weight", Double())
    assert torch.equal(m.fused_weight()[64:80], m.v.weight) and torch.equal(m.fused_weight()[:48], m.q.weight)
    n = FusedLayerNorm(16, dtype=torch.float32)
    n.weight.data.fill_(0.5)
    torch.nn.utils.parametrize.register_parametrization(n, "weight", Double())
    assert torch.equal(n.gamma_beta_fp32()[0], torch.ones(16))

    m = CustomLayerNormLinear(1024, 96, 32, dtype=torch.float32)
    x, t = torch.randn(2, 1, 1024, requires_grad=True), torch.randn(2, 1, 1024)
    grad = torch.autograd.grad(m.forward_qkvx(x)[0].sum(), x)[0]
    assert torch.allclose(grad, m.q.weight.sum(0).expand(2, 1, -1), atol=1e-4)
    tangent = torch.func.jvp(lambda x_: m.forward_qkvx(x_)[3], (x.detach(),), (t,))[1]
    assert torch.allclose(tangent, m.forward_qx(t), atol=1e-4)


def test_fp8_kv_cache_shapes_and_layer_option():
    from magi_attn.cache import Fp8KVCache
    from magi_attn.module import FullyParallelAttention

    c = Fp8KVCache(10 * 24, 2, 24)
    assert c.k.shape == c.v.shape == (240, 2, 128) and c.k.dtype == torch.float8_e4m3fn
    assert c.k_scale.shape == c.v_scale.shape == (10, 2) and c.max_sequence_length == 240
    assert Fp8KVCache(25, 1, 24).k_scale.shape == (2, 1)  # a partial last chunk has a scale row too
    with pytest.raises(ValueError):
        Fp8KVCache(0, 2, 24)
    with pytest.raises(ValueError):
        FullyParallelAttention(64, 2, 1, attention_dtype="fp4")
    assert FullyParallelAttention(64, 2, 1, attention_dtype="fp8").attention_dtype == "fp8"


def test_replaced_fp8_projections_are_called_and_not_read(monkeypatch):
    """fp8_quant hands the quantised input only to a PerTensorQuantizedFp8Linear that nothing replaces, patches, watches or
    keeps elsewhere; any other projection is called with the normalised input."""
    from magi_attn import module as MOD

    K = 64
    c = MOD.CustomLayerNormLinear(K, 256, 128, fp8_quant=True)
    assert all(c._takes_e4m3(m, K) for m in c._projections()) and not c._takes_e4m3(c.q, 2 * K)
    c.q.register_forward_hook(lambda m, i, o: None)
    c.k.register_forward_pre_hook(lambda m, i: None)
    c.v.forward = lambda x: x.new_zeros(x.shape[0], 128)
    assert not any(c._takes_e4m3(m, K) for m in (c.q, c.k, c.v)) and c._takes_e4m3(c.qx, K)
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: None)
    try:
        assert not c._takes_e4m3(c.qx, K)
    finally:
        handle.remove()
    for scale in (torch.ones(1), torch.ones(K).half(), torch.ones(2 * K)[::2], torch.ones(K, device="meta")):
        c.qx.input_scale = torch.nn.Parameter(scale, requires_grad=False)
        assert not c._takes_e4m3(c.qx, K)
    c = MOD.CustomLayerNormLinear(K, 256, 128, fp8_quant=True)
    with monkeypatch.context() as patch:
        patch.setattr(MOD.PerTensorQuantizedFp8Linear, "forward", lambda self, x: x)
        assert not c._takes_e4m3(c.q, K)
    assert c._takes_e4m3(c.q, K)
    # classes without input_scale among the four, called in their places
    c = MOD.CustomLayerNormLinear(K, 256, 128, fp8_quant=True)
    calls = []

    class Fixed(torch.nn.Module):
        def __init__(self, name, n):
            super().__init__()
            self.name, self.n = name, n

        def forward(self, x):
            calls.append(self.name)
            return x.new_full((x.shape[0], self.n), ord(self.name[-1]))

    for name, n in (("q", 256), ("k", 128), ("v", 128), ("qx", 256)):
        setattr(c, name, Fixed(name, n))
    monkeypatch.setattr(MOD, "layer_norm", lambda x, w, b, eps: torch.nn.functional.layer_norm(x, (K,), w, b, eps))
    out = c.forward_ln_qkvx_rows(torch.randn(5, 1, K).bfloat16())
    assert sorted(calls) == ["k", "q", "qx", "v"] and [t[0, 0].item() for t in out] == [ord(x) for x in "qkvx"]


@pytest.mark.parametrize("cols,round_rows", [(8192, 2048), (4096, 4096), (16384, 1024), (256, 65536)])
def test_projection_rows_are_cut_only_where_a_round_of_tiles_is_left_partly_empty(cols, round_rows):
    from magi_attn.module import _rows_ahead

    for rounds in (0, 1, 2, 5, 41):
        for rest in (0, 1, 255, 256, 257, round_rows // 2, round_rows // 2 + 1, round_rows - 256, round_rows - 255, round_rows - 1):
            if not 0 <= rest < round_rows:
                continue
            gap = -(-rest // 256) < round_rows // 256  # (a row of tiles of the last round stays empty)
            cut = rounds > 0 and rest > 0 and gap and (rounds > 1 or rest <= round_rows // 2)
            assert _rows_ahead(rounds * round_rows + rest, cols, 3072, 256) == (rounds * round_rows if cut else 0), (rounds, rest)
    for cols_, depth, cus in ((14336, 6144, 256), (8192, 1016, 256), (8200, 3072, 256), (0, 3072, 256), (8192, 3072, 304), (131072, 3072, 256)):
        assert _rows_ahead(9360, cols_, depth, cus) == 0


@pytest.mark.parametrize("begun", [False, True])
@pytest.mark.parametrize("devices", ["0", "00", "01", "000", "010", "0000"])
def test_every_held_call_is_launched_once(monkeypatch, begun, devices):
    from magi_attn import _lib as L
    from magi_attn import functional as F

    done = []
    monkeypatch.setattr(F, "_launch", lambda dev, fn, *args: done.append((dev, fn, args)))
    names, fwd = [f"call {i}" for i in range(len(devices))], L.packed("magi_attn_fwd", L.AttnArgs).fn
    held = [(dev, None if begun and i == 0 else fwd, name, ()) for i, (dev, name) in enumerate(zip(devices, names))]
    F.launch_held(held)
    assert not held and [a for _, _, args in done for a in args if a] == names  # each once, in their order
    together = [args for _, _, args in done if len(args) == 2 and args[1]]
    assert together == ([tuple(names[:2])] if devices[:2] == "00" and (begun or len(devices) == 2) else [])
    for dev, _, args in done:
        assert all(devices[names.index(a)] == dev for a in args if a)


@pytest.mark.parametrize("cols,whole", [(1024, 16384), (3072, 16384), (6144, 8192), (8192, 2048), (256, 65536), (5120, 16384)])
def test_e4m3_rows_are_cut_behind_rounds_that_are_whole_to_the_last_tile(cols, whole):
    from magi_attn.module import _rows_ahead_e4m3

    for n in (0, 1, 2, 7, 9):
        for rest in (0, 1, n * whole // 7, n * whole // 7 + 1, whole - 1):
            if rest >= whole:
                continue
            assert _rows_ahead_e4m3(n * whole + rest, cols, 1024, 256) == (n * whole if 0 < rest and 7 * rest <= n * whole else 0), (n, rest)
    for cols_, depth, cus in ((1024, 1016, 256), (1000, 3072, 256), (0, 3072, 256), (131072, 3072, 256)):
        assert _rows_ahead_e4m3(16974, cols_, depth, cus) == 0


def test_replaced_projection_methods_are_called(monkeypatch):
    """forward() projects through linear_qkv.forward_ln and .forward_qkvx where these are not the library's own: another module
    that offers the two, a subclass, a method patched onto the instance."""
    from magi_attn import module as MOD

    K, widths = 64, (256, 128, 128, 256)
    monkeypatch.setattr(MOD, "layer_norm", lambda x, w, b, eps: torch.nn.functional.layer_norm(x, (K,), w, b, eps))
    layer = MOD.FullyParallelAttention(K, 2, 1)
    x = torch.randn(6, 3, K).bfloat16()
    rows, mixed = layer._project_rows(x)
    assert mixed is None and [t.shape for t in rows] == [(18, n) for n in widths]

    class Sub(MOD.CustomLayerNormLinear):
        def forward_qkvx(self, h):
            return tuple(t * 2 for t in super().forward_qkvx(h))

    class Other(torch.nn.Module):  # (no forward_ln_qkvx_rows)
        def forward_ln(self, h):
            return h + 1

        def forward_qkvx(self, h):
            return tuple(h[..., :1].expand(*h.shape[:-1], n) for n in widths)

    own = layer.linear_qkv
    sub = Sub(K, 256, 128)
    sub.load_state_dict(own.state_dict())
    layer.linear_qkv = sub
    got, mixed = layer._project_rows(x)
    assert torch.equal(mixed, own.forward_ln(x)) and all(torch.equal(a, 2 * b) for a, b in zip(got, rows))
    layer.linear_qkv = Other()
    got, mixed = layer._project_rows(x)
    assert torch.equal(mixed, x + 1) and all(torch.equal(a, (x + 1)[..., :1].reshape(18, 1).expand(18, n)) for a, n in zip(got, widths))
    layer.linear_qkv = own
    own.forward_ln = lambda h: h * 0
    got, mixed = layer._project_rows(x)
    assert not mixed.any() and not any(t.any() for t in got)
    del own.forward_ln
    assert layer._project_rows(x)[1] is None
    # and onto the class
    was = MOD.CustomLayerNormLinear.forward_qkvx
    monkeypatch.setattr(MOD.CustomLayerNormLinear, "forward_qkvx", lambda self, h: tuple(-t for t in was(self, h)))
    got, mixed = layer._project_rows(x)
    assert torch.equal(mixed, own.forward_ln(x)) and all(torch.equal(a, -b) for a, b in zip(got, rows))


def test_a_replaced_norm_module_is_noticed():
    """Score bounds and e4m3 operand scales belong to the norm modules they were derived from, not to how often those had
    converted their parameters."""
    from magi_attn import module as MOD

    def norm(gain):
        ln = MOD.FusedLayerNorm(128, dtype=torch.float32)
        torch.nn.init.constant_(ln.weight, gain - 1.0)
        return ln

    def fresh(gains):
        layer = MOD.FullyParallelAttention(64, 2, 1)
        for name, gain in zip(names, gains):
            setattr(layer, name, norm(gain))
        return layer.score_bounds(), layer.fp8_operand_scales()

    names = ("q_layernorm", "k_layernorm", "q_layernorm_xattn", "k_layernorm_xattn")
    layer = MOD.FullyParallelAttention(64, 2, 1)
    gains = [1.0] * 4
    for i, gain in ((None, 1.0), (0, 21.0), (1, 0.5), (2, 3.0), (3, 7.0), (0, 1.0)):
        if i is not None:
            gains[i] = gain
            setattr(layer, names[i], norm(gain))
        assert (layer.score_bounds(), layer.fp8_operand_scales()) == fresh(gains), (i, gain)
    # two norms exchanged
    layer.q_layernorm, layer.q_layernorm_xattn = layer.q_layernorm_xattn, layer.q_layernorm
    gains[0], gains[2] = gains[2], gains[0]
    assert (layer.score_bounds(), layer.fp8_operand_scales()) == fresh(gains)


def test_a_norm_parameter_at_the_address_of_the_last_one_is_noticed():
    """A parametrised weight is a new tensor at every look, here always at one address and now and then with the id of the
    one before."""
    from magi_attn import module as MOD

    memory = np.zeros(128, np.float32)

    class Twice(torch.nn.Module):
        def forward(self, x):
            np.multiply(x.detach().numpy(), 2.0, out=memory)
            return torch.from_numpy(memory)

    ln = MOD.FusedLayerNorm(128, dtype=torch.float32)
    torch.nn.utils.parametrize.register_parametrization(ln, "weight", Twice())
    with torch.no_grad():
        for i in range(200):
            ln.parametrizations.weight.original.fill_(float(i))
            assert ln.gamma_beta_fp32()[0][0].item() == 2.0 * i
    plain = MOD.FusedLayerNorm(128, dtype=torch.float32)
    first = plain.gamma_beta_fp32()
    assert plain.gamma_beta_fp32() is first  # (converted once)
    twin = copy.deepcopy(plain)
    torch.nn.init.constant_(twin.weight, 3.0)
    assert twin.gamma_beta_fp32()[0][0].item() == 3.0 and plain.gamma_beta_fp32() is first


def test_attention_kernels_keep_their_registers():
    """A register spill inside a tile loop costs a drain of the tile loads per tile (parity stays green while the
    launch runs 1.7x slower), and the allocator decides per instantiation: compile the attention sources for
    gfx950 and check the compiler's own resource report.  The bf16 instantiations must use no scratch memory at
    all; the fp8 kernel is allowed its known 24 bytes (values parked across the loop and reloaded on the ragged-tile
    path and in the epilogue, not in the steady-state loop)."""
    import shutil
    import subprocess

    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    csrc = os.path.join(ROOT, "magi-1_amd", "csrc")
    flags = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-I" + os.path.join(ROOT, "include"), "-I" + csrc,
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument",
             "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c", "-o", os.devnull]
    # The bf16 kernels must not spill at all (the 16x16x32 kernel once parked two accumulators around its first tile:
    # outside the steady-state loop, but a round trip to scratch memory for every workgroup, 12 % more bytes written).
    for src, limit in (("attn_fwd_bf16.hip", 0), ("attn_fwd_fp8.hip", 24), ("attn_fwd_bf16_w64.hip", 0),
                       ("attn_fwd_bf16_x16.hip", 0)):
        r = subprocess.run([hipcc] + flags + [os.path.join(csrc, src)], capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, r.stderr[-2000:]
        names = re.findall(r"Function Name: (\S+)", r.stderr)
        scratch = [int(x) for x in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", r.stderr)]
        vgprs = [int(x) for x in re.findall(r" VGPRs: (\d+)", r.stderr)]
        assert names and len(names) == len(scratch) == len(vgprs), (len(names), len(scratch), len(vgprs))
        seen = 0
        for n, sc, vg in zip(names, scratch, vgprs):
            if "attn_fwd" in n:
                seen += 1
                assert sc <= limit, f"{n}: {sc} bytes of scratch per lane"
                assert vg <= 256
        assert seen >= 2


def test_inference_params_swap_key_value_dict():
    """Batch rows of the (position, batch)-ordered caches are re-ordered in every layer; an empty dict raises, as in
    the reference (inference/common/dataclass.py:72-83)."""
    from magi_attn.params import InferenceParams

    ip = InferenceParams(3, 4)
    with pytest.raises(ValueError):
        ip.swap_key_value_dict([0, 1, 2])
    c = torch.arange(4 * 3 * 2 * 8, dtype=torch.float32).view(12, 2, 8)  # [max_seq * max_bs, Hkv, 2D]
    ip.key_value_memory_dict[0] = c.clone()
    ip.key_value_memory_dict[5] = c.clone() + 1000
    ip.swap_key_value_dict([2, 0, 1])
    want = c.view(4, 3, 2, 8)[:, [2, 0, 1]].reshape(12, 2, 8)
    assert torch.equal(ip.key_value_memory_dict[0], want) and torch.equal(ip.key_value_memory_dict[5], want + 1000)
    with pytest.raises(ValueError):
        ip.swap_key_value_dict([0, 1])


def test_copying_form_of_the_cache_update_matches_the_reference_semantics():
    """FullyParallelAttention.adjust_key_and_value_for_inference, the method with the reference's signature for
    callers that hold a materialised key_and_value (dit_module.py:891-946): pure tensor work, so it runs on the CPU.
    Against the oracle's list-of-rows model through a schedule with appends, reads without update, the distill form
    that drops the last chunk, no inference_params at all, and batch 2."""
    from magi_attn.module import FullyParallelAttention
    from oracle import magi_oracle as O
    Hkv, D, L_ = 2, 128, 5
    for bs in (1, 2):
        layer = FullyParallelAttention(64, 4, Hkv, layer_number=2, device="cpu")
        ip = P.InferenceParams(bs, 6 * L_)
        model = O.KVCacheModel(6 * L_, Hkv, D, max_batch_size=bs)
        g = torch.Generator().manual_seed(bs)
        written = 0
        # (slice_point, chunks, update, distill, fwd_extra_1st_chunk)
        for sp, dn, update, distill, extra in ((0, 2, True, False, True), (2, 2, False, False, False),
                                               (2, 2, True, True, False), (3, 3, True, False, False),
                                               (0, 1, True, False, False)):
            kv = torch.randn(dn * L_ * bs, Hkv, 2 * D, generator=g).bfloat16()
            ip.update_kv_cache = update
            meta = P.ModelMetaArgs(H=1, W=L_, cp_pad_size=None, cp_split_sizes=None, slice_point=sp, denoising_range_num=dn,
                                   range_num=sp + dn, extract_prefix_video_feature=False, fwd_extra_1st_chunk=extra,
                                   distill_nearly_clean_chunk=distill, clip_token_nums=L_, enable_cuda_graph=False,
                                   core_attn_params=None, cross_attn_params=None)
            k, v = layer.adjust_key_and_value_for_inference(kv, ip, meta)
            k_ref, v_ref = model.adjust(kv, has_inference_params=True, update_kv_cache=update, slice_point=sp,
                                        clip_token_nums=L_, fwd_extra_1st_chunk=extra, distill_nearly_clean_chunk=distill)
            assert torch.equal(k, k_ref) and torch.equal(v, v_ref), (bs, sp, dn)
            if update:
                written = max(written, (sp + dn - (1 if distill else 0)) * L_ * bs)
            # (the layer's cache is allocated uninitialised, as the reference's: rows written so far)
            assert torch.equal(ip.key_value_memory_dict[2][:written], model.mem[:written])
        k, v = layer.adjust_key_and_value_for_inference(kv, None, meta)
        assert torch.equal(k, kv[..., :D]) and torch.equal(v, kv[..., D:])


@pytest.mark.parametrize("version,exports", [(104, ()), (L.ABI_VERSION, ("magi_attn_fwd",))])
def test_a_library_of_another_version_or_without_an_entry_point_is_refused(tmp_path, monkeypatch, version, exports):
    """Version 104 had neither MAGI_ATTN_ROW_BITS, which it would ignore, nor the entry points that came with it."""
    import subprocess

    src, so = tmp_path / "old.c", tmp_path / "old.so"
    src.write_text("int magi_version(void) { return %d; }\n" % version + "".join("int %s(void) { return 0; }\n" % n for n in exports))
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    monkeypatch.setattr(L, "_lib", None)
    monkeypatch.setattr(L, "LIB_PATH", str(so))
    with pytest.raises(RuntimeError, match="rebuild the library"):
        L.lib()


@pytest.mark.parametrize("size", [(6, 2, 1, 200), (24, 8, 1, 1300), (24, 8, 4, 288)])
def test_plans_of_the_longest_stated_key_ranges(size):
    """A max_seqlen_k as large as the type: the plan is that of one that differs by less than a tile of 64 keys in 2^25."""
    lib, longest, near = L.lib(), 2 ** 31 - 1, 2 ** 31 - 128
    memory = lib.magi_attn_split_bytes(*size, near, L.MAGI_DTYPE_BF16)
    assert memory > 0 and memory == lib.magi_attn_split_bytes(*size, longest, L.MAGI_DTYPE_BF16)
    assert lib.magi_attn_tile_rows(*size, near, memory) == lib.magi_attn_tile_rows(*size, longest, memory)
    for bounded in (0, 1):
        assert lib.magi_attn_pieces_bytes(*size, near, bounded) == lib.magi_attn_pieces_bytes(*size, longest, bounded)


def test_memory_of_256_row_workgroups_is_part_of_what_a_bounded_call_asks_for():
    for size in ((24, 8, 1, 432, 1728), (6, 2, 1, 270, 1350), (24, 8, 1, 720, 2880), (24, 8, 4, 288, 2016), (0, 1, 1, 1, 1), (3, 2, 1, 1, 1), (6, 2, 0, 1, 1)):
        whole, pieces = L.lib().magi_attn_split_bytes(*size, L.MAGI_DTYPE_BF16), L.lib().magi_attn_pieces_bytes(*size, 1)
        assert max(L.lib().magi_attn_split_bytes_256(*size), pieces) == whole
