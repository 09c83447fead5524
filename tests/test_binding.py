"""The calls that go from Python to the C ABI without ctypes: plain arguments give what the general path gives, and every other
form is left to that path, with nothing done."""
import ctypes
import os
import subprocess
import sys
import sysconfig

import numpy as np
import pytest
import torch

import lmdeploy_amd.turbomind as tm
from lmdeploy_amd._lib import GemmDesc, W4A16Error, binding, lib
from oracle import w4a16_oracle as O


class Wrapped(torch.Tensor):
    pass


def test_other_forms_are_left_to_the_general_path():
    good = [None, None, None, None, None, 128, 1, 128, 128, 0, -1, 0]
    assert binding.gemm_static(*good) == lib.w4a16_gemm_static(*good) == -4  # (null pointers are refused)
    assert binding.gemm(0, *good) == lib.w4a16_gemm(0, *good) == -4
    for at, bad in [(0, torch.zeros(2)), (1, torch.zeros(2).as_subclass(Wrapped)), (2, 5), (5, 1.0), (6, np.int64(1)), (7, 1 << 31),
                    (8, -(1 << 31) - 1), (9, ctypes.c_int(0)), (10, None), (11, ctypes.c_void_p(0)), (11, 1 << 64)]:
        assert binding.gemm_static(*good[:at], bad, *good[at + 1:]) is None, (at, bad)
    assert binding.gemm_static(*good[:-1]) is None and binding.ptr(torch.zeros(2)) is None
    assert binding.ffn(0, *[None] * 8, 128, 128, 1.5, 128, 0) is None and binding.gemm(None, *good) is None
    with pytest.raises(ValueError, match="live on the GPU"):
        tm.gemm_static(torch.zeros(2), None, None, None, 128, 1, 128, 128)
    with pytest.raises(ctypes.ArgumentError):
        tm.gemm_static(None, None, None, None, 128, 1.0, 128, 128, stream=0)
    with pytest.raises(W4A16Error, match="null"):
        tm.gemm_static(None, None, None, None, 128, 1, 128, 128, stream=0)


def test_validation_of_a_layer():
    ptrs = lambda n, skip=-1: (ctypes.c_void_p * n)(*[None if i == skip else 0x2000 for i in range(n)])
    ints = lambda *v: (ctypes.c_int * len(v))(*v)
    call = lambda A=ptrs(4), Q=ptrs(4), w=ptrs(7), n=(256, 128, 128, 256, 512, 512, 256), k=(256, 256, 256, 512), D=128, g=128: \
        lib.w4a16_deploy_layer(A, Q, w, ptrs(7), ptrs(7), ints(*n), ints(*k), D, g, None)
    assert call(g=16) == -1 and call(D=96) == -2 and call(D=3) == -2 and call(D=0) == -2
    assert call(n=(256, 128, 256, 256, 512, 512, 256)) == -2 and call(n=(256, 128, 128, 256, 512, 504, 256)) == -2
    assert call(n=(256, 128, 128, 264, 512, 512, 256)) == -2 and call(n=(256, 128, 128, 256, 516, 516, 256)) == -2
    assert call(k=(256, 200, 256, 512)) == -2 and call(k=(256, -128, 256, 512)) == -4 and call(n=(-256, 128, 128, 256, 512, 512, 256)) == -4
    assert call(A=None) == -4 and call(A=ptrs(4, 2)) == -4 and call(Q=ptrs(4, 3)) == -4 and call(w=ptrs(7, 5)) == -4
    assert call(n=(0,) * 7) == 0 and call(k=(0,) * 4) == 0      # nothing to do


@pytest.mark.parametrize("count", [0, 1, 5])
def test_descriptors(count):
    gemms = [(None, None, None, None, 8 * i, -i, i % 3, None, i % 2 == 0) for i in range(count)]
    arr = (GemmDesc * count)()
    assert binding.describe(arr, gemms) is True and binding.describe(arr, tuple(gemms)) is True
    for i, d in enumerate(arr):
        assert (d.C, d.A, d.X, d.Q, d.R, d.n_out, d.k, d.epilogue, d.depends) == (None,) * 5 + (8 * i, -i, i % 3, int(i % 2 == 0))
    assert binding.describe((GemmDesc * (count + 1))(), gemms) is None  # (a wrong number of them)
    if count:
        for bad in (gemms[-1][:8], list(gemms[-1]), gemms[-1][:4] + (1.0,) + gemms[-1][5:], (torch.zeros(1),) + gemms[-1][1:],
                    gemms[-1][:8] + ("yes",)):
            assert binding.describe(arr, gemms[:-1] + [bad]) is None, bad


def test_a_tree_without_the_extension_imports_and_calls():
    """The library alone is enough: what the extension would take goes through ctypes, and a warning says so."""
    code = """
import sys, warnings
sys.modules["lmdeploy_amd._binding"] = None     # as if it had not been built
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    import lmdeploy_amd.turbomind as tm
assert ["ctypes" in str(w.message) for w in seen if "lmdeploy_amd._binding" in str(w.message)] == [True], seen
import ctypes, torch
for call in (lambda: tm.gemm_static(None, None, None, None, 128, 1, 128, 128, stream=0), lambda: tm.check(tm.lib.w4a16_ffn(*[None] * 9, 128, 128, 1, 128, None))):
    try:
        call()
    except tm.W4A16Error as e:
        assert e.code == -4 and "null" in str(e)
    else:
        raise AssertionError
try:
    tm.gemm_static(torch.zeros(2), None, None, None, 128, 1, 128, 128, stream=0)
except ValueError as e:
    assert "live on the GPU" in str(e)
print("fine")
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("fine"), r.stderr[-2000:]


def test_an_extension_for_another_torch_is_left_alone():
    """It reads tensors by the layout that it was compiled with: of another torch it takes no call."""
    code = """
import sys, types, warnings
other = types.ModuleType("lmdeploy_amd._binding")
other.torch_version, other.bind = "0.0.0", None
sys.modules["lmdeploy_amd._binding"] = other
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    import lmdeploy_amd
    lmdeploy_amd._binding = other
    from lmdeploy_amd import _lib
assert isinstance(_lib.binding, _lib.General) and any("0.0.0" in str(w.message) for w in seen), seen
print("fine")
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("fine"), r.stderr[-2000:]


def test_the_extension_is_named_after_its_interpreter(monkeypatch, tmp_path):
    """Another interpreter does not take it for its own, and one without that name, which it would take, is removed by a build."""
    import lmdeploy_amd.build as build
    suffix = sysconfig.get_config_var("EXT_SUFFIX")
    assert "%d%d" % sys.version_info[:2] in suffix and binding.__file__.endswith(suffix)
    old = tmp_path / "_binding.so"
    old.write_bytes(b"of another interpreter")
    monkeypatch.setattr(build, "BINDING_UNNAMED", str(old))
    monkeypatch.setattr(build, "BINDING_PATH", str(tmp_path / os.path.basename(build.BINDING_PATH)))
    assert build.build_binding(verbose=False) == build.BINDING_PATH
    assert [f.name for f in tmp_path.iterdir()] == ["_binding" + suffix]


@pytest.mark.parametrize("what", ["compiler", "Python's headers", "torch's headers"])
def test_a_build_without_what_the_extension_needs_says_so_and_leaves_none(what, monkeypatch, tmp_path, capsys):
    import lmdeploy_amd.build as build
    old = tmp_path / "_binding.so"
    old.write_bytes(b"of another source")
    monkeypatch.setattr(build, "BINDING_PATH", str(old))
    if what == "compiler":
        monkeypatch.setattr(build.shutil, "which", lambda name: None)
    elif what == "Python's headers":
        monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    else:
        monkeypatch.setattr(torch, "__file__", str(tmp_path / "__init__.py"))
    assert build.build_binding() is None
    assert not old.exists() and "ctypes" in capsys.readouterr().out


@pytest.mark.gpu
def test_both_paths_give_the_same():
    T, K, N, g = 3, 256, 128, 128
    d = O.make_inputs(77, T, K, N, g, residual=True)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).cuda()
    qw, qz, s, X, R = (dev(d[n]) for n in ("qweight", "qzeros", "scales", "X", "R"))
    A, Q = torch.zeros_like(qw), torch.zeros_like(s, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, torch.zeros_like(s), qw, s, qz, N, K, g)
    op = tm.GemmS4F16()
    out = [torch.empty(T, N, dtype=torch.float16, device="cuda") for _ in range(7)]
    other = lambda t: t.as_subclass(Wrapped)
    at = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    op.Run(out[0], A, X, Q, N, T, K, g, 2, -1, residual=R)
    op.Run(out[1], torch.nn.Parameter(A, requires_grad=False), X, Q, N, T, K, g, 2, residual=R)
    op.Run(other(out[2]), A, other(X), Q, N, T, K, g, 2, residual=R)
    op.Run(out[3], A, X, Q, N, ctypes.c_int(T), K, g, 2, residual=R, stream=at)
    tm.gemm_static(out[4], A, X, Q, N, T, K, g, 2, residual=R)
    tm.gemm_static(out[5], A, X, Q, N, T, K, g, 2, residual=other(R))
    op.sequence([[out[6], A, X, Q, N, K, 2, R, False]], T, g)
    torch.cuda.synchronize()
    want = O.gemm_s4_f16(d["X"], d["qweight"], d["qzeros"], d["scales"], g, 2, d["R"])
    assert O.max_abs_rel(out[0].cpu().numpy(), want) <= 1e-2
    for o in out[1:]:
        assert torch.equal(o, out[0])
    A2, Q2 = torch.zeros_like(A), torch.zeros_like(Q)
    tm.convert_s4_k_m8(other(A2), Q2, None, qw, other(s), qz, N, K, g)
    assert torch.equal(A2, A) and torch.equal(Q2, Q)
    plain, mixed = (qw, qz, s), (other(qw), qz, other(s))
    for a, b in zip(tm.deploy_layer(*[plain] * 6, mixed, 128, g), tm.deploy_layer(*[plain] * 7, 128, g)):
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    with pytest.raises(ValueError, match="contiguous"):
        op.Run(out[0], A, X.t(), Q, N, T, K, g)
    with pytest.raises(RuntimeError):  # inside a transform a tensor has no address
        torch.vmap(lambda x: op.Run(out[0], A, x, Q, N, T, K, g))(X.expand(2, T, K).contiguous())


@pytest.mark.gpu
def test_every_call_without_the_extension(monkeypatch):
    from lmdeploy_amd._lib import General
    T, H, F, g = 3, 256, 512, 128
    gen = torch.Generator(device="cuda").manual_seed(5)
    words = lambda *size: torch.randint(-2 ** 31, 2 ** 31, size, dtype=torch.int32, device="cuda", generator=gen)
    awq = lambda k, n: (words(k, n // 8), words(k // g, n // 8), (torch.rand((k // g, n), device="cuda", generator=gen) * 0.01 + 1e-3).half())
    parts = [awq(H, H) for _ in range(4)] + [awq(H, F), awq(H, F), awq(F, H)]
    X, R = torch.randn((2, T, H), device="cuda", generator=gen).half()
    op = tm.GemmS4F16()

    def everything():
        new = lambda n: torch.empty((T, n), dtype=torch.float16, device="cuda")
        (A0, Q0), (A1, Q1), (A2, Q2), (A3, Q3) = made = tm.deploy_layer(*parts, 128, g)
        A, Q = torch.empty_like(A1), torch.empty_like(Q1)
        tm.convert_s4_k_m8(A, Q, None, parts[3][0], parts[3][2], parts[3][1], H, H, g)
        out = [new(3 * H), new(3 * H), new(F), new(H), new(H)]
        op.Run(out[0], A0, X, Q0, 3 * H, T, H, g)
        tm.gemm_static(out[1], A0, X, Q0, 3 * H, T, H, g)
        op.ffn(out[3], out[2], X, A2, Q2, A3, Q3, H, F, T, g, residual=R)
        op.sequence([(out[4], A1, X, Q1, H, H, op.kFusedAdd, R, True)], T, g)
        torch.cuda.synchronize()
        return [t for pair in made for t in pair] + [A, Q] + out

    want = everything()
    absent = General()
    monkeypatch.setattr(tm, "binding", absent)
    for name, of in (("_gemm", "gemm"), ("_gemm_static", "gemm_static"), ("_ffn", "ffn"), ("_describe", "describe"), ("_plain_ptr", "ptr")):
        monkeypatch.setattr(tm, name, getattr(absent, of))
    for a, b in zip(want, everything()):
        assert torch.equal(a, b)
