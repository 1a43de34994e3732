"""The native launchers (csrc/launchers.cpp) against the general ctypes way of the same wrappers:
every form of argument gives the same result, or the same error."""
import math
import subprocess
import sys

import numpy as np
import pytest

from conftest import PKG_DIR, ROOT, rand_bf16


def outcome(fn, *args, **kw):
    try:
        return fn(*args, **kw)
    except Exception as e:  # the type and the message are what is compared
        return type(e), str(e)


def both(pkg, monkeypatch, name, *args, **kw):
    """(outcome as called, outcome of the general way)"""
    pkg.lib()
    native = outcome(getattr(pkg, name), *args, **kw)
    with monkeypatch.context() as m:
        m.setattr(pkg, "_native", None)
        general = outcome(getattr(pkg, name), *args, **kw)
    return native, general


def test_built_for_this_python(pkg):
    pkg.lib()
    assert pkg._native is not None and pkg._native.__file__ == str(pkg.LAUNCHERS_PATH)


@pytest.mark.parametrize("setup", [
    "pkg.LAUNCHERS_PATH = pathlib.Path('/nonexistent/_launchers.so')",
    "pkg.LAUNCHERS_PATH = pathlib.Path(pkg.__file__)",  # no shared object
    "pkg.LAUNCHERS_PATH = pkg.HERE.parent / 'oracle' / 'liboracle.so'",  # no module
    "import torch; torch.__version__ = '0.0.0'"])
def test_the_library_works_without_them(setup):
    """A module that is missing, does not load or was built over another torch: every call goes
    through ctypes."""
    code = ("import pathlib, sys; sys.path.insert(0, 'tests'); from conftest import load_package;"
            f"pkg = load_package(); {setup}; pkg.lib(); assert pkg._native is None\n"
            "try: pkg.gemv_forward(4096, 4096, 4096, 4, 7, stream=0)\n"
            "except pkg.LlmError as e: print(e)")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, check=True)
    assert "cols 7 is not a multiple of 8" in r.stdout


@pytest.mark.parametrize("lacking", ["PY_INC=/nonexistent", "TORCH=/nonexistent", "PYTHON=/nonexistent"])
def test_make_builds_the_library_without_headers_or_torch(lacking):
    def plan(*args):
        return subprocess.run(["make", "-n", "-B", "-C", str(PKG_DIR), *args], capture_output=True,
                              text=True, check=True).stdout
    assert "launchers.cpp" in plan(f"PYTHON={sys.executable}")
    lean = plan(lacking)
    assert "launchers.cpp" not in lean and "libllm_amd.so" in lean


# calls that the library or the wrapper refuses before a launch: no GPU needed
@pytest.mark.parametrize("rows", [0, -1, True - 1, np.int64(0), 0.0, "0", None, 2 ** 32, -2 ** 70])
@pytest.mark.parametrize("eps", [1e-6, 1, np.float64(1e-6), None])
@pytest.mark.parametrize("out", [4096, None, -1, True, 2 ** 64 + 16, 1.5, "cpu tensor"])
def test_refused_calls_are_refused_alike(pkg, monkeypatch, rows, eps, out):
    import torch
    if isinstance(out, str):
        out = torch.zeros(8, dtype=torch.bfloat16)
    native, general = both(pkg, monkeypatch, "rmsnorm_forward", out, 4096, 4096, rows, 8, eps, stream=0)
    assert native == general and native is not None


@pytest.mark.parametrize("args", [(16, 32, 48, 0, 8), (16, 32, 48, 8, 12), (16, 8, 48, 4, 8),
                                  (16, 32, 48, 4, 8, 64)])
def test_library_errors_are_raised(pkg, monkeypatch, args):
    if len(args) == 6:  # in aliases x
        args = (16, 32, 16, 4, 8, 64)
    for stream in (0, True, 0.5, "s"):
        native, general = both(pkg, monkeypatch, "gemv_residual_forward", *args[:5], None, stream)
        assert native == general and native is not None
    assert pkg.lib().llm_last_error() is None


@pytest.mark.gpu
def test_accepted_forms_give_the_same_result(gpu, monkeypatch):
    """Tensors (bf16, raw 16-bit, a Parameter, a subclass), addresses, streams and numbers."""
    import torch
    rng = np.random.default_rng(5)
    rows, dim = 3, 264

    class Sub(torch.Tensor):
        pass

    raw = torch.from_numpy(rand_bf16(rng, (rows, dim)).view(np.int16)).cuda()
    w = torch.from_numpy(rand_bf16(rng, dim).view(np.int16)).cuda().view(torch.bfloat16)
    x = raw.view(torch.bfloat16)
    side = torch.cuda.Stream()
    want = torch.zeros_like(x)
    gpu.rmsnorm_forward(want, x, w, rows, dim, 1e-6)
    torch.cuda.synchronize()
    forms = [x, raw, raw.view(torch.uint16), torch.nn.Parameter(x), x.as_subclass(Sub), x.data_ptr(),
             x[:, :], x.float(), x.half(), x.t(), x.cpu(), None]
    for form in forms:
        for stream in (None, side, side.cuda_stream):
            got = []
            for use_native in (True, False):
                out = torch.zeros_like(x)
                torch.cuda.synchronize()
                with monkeypatch.context() as m:
                    if not use_native:
                        m.setattr(gpu, "_native", None)
                    result = None
                    if form is not None:
                        result = outcome(gpu.rmsnorm_forward, out, form, w, rows, dim, 1e-6, stream)
                torch.cuda.synchronize()
                got.append((result, out))
            assert got[0][0] == got[1][0]
            assert torch.equal(got[0][1].view(torch.int16), got[1][1].view(torch.int16))
            if got[0][0] is None and form is not None:
                assert torch.equal(got[0][1].view(torch.int16), want.view(torch.int16))
    # the current stream of a stream context: the launch is captured, not run
    graph, out = torch.cuda.CUDAGraph(), torch.zeros_like(x)
    with torch.cuda.graph(graph):
        gpu.rmsnorm_forward(out, x, w, rows, dim, 1e-6)
    torch.cuda.synchronize()
    assert not out.any()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))


@pytest.mark.gpu
def test_attention_workspace_is_checked(gpu, monkeypatch):
    import torch
    hq, hkv, D, max_seq = 4, 2, 64, 100
    need = gpu.attention_workspace_floats(hq, D, max_seq)
    q = torch.zeros(hq * D, device="cuda", dtype=torch.bfloat16)
    kv = torch.zeros(max_seq, hkv * D, device="cuda", dtype=torch.bfloat16)
    norm = torch.ones(D, device="cuda", dtype=torch.bfloat16)
    pos = torch.zeros(1, device="cuda", dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    for floats in (need, need - 1):
        att = torch.zeros(floats, device="cuda")
        a = both(gpu, monkeypatch, "attention_forward", q, q.clone(), kv, kv, att, hq, hkv, D, pos,
                 max_seq, scale)
        b = both(gpu, monkeypatch, "qk_norm_rope_attention_forward", q, q.clone(), kv[0], kv[1], norm,
                 norm, kv, kv, att, pos, hq, hkv, D, 1e-6, 1e6, max_seq, scale)
        assert a[0] == a[1] and b[0] == b[1]
        assert (a[0] is None) == (b[0] is None) == (floats == need)
    torch.cuda.synchronize()
