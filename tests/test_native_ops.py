"""The operators' native call path: it gives what the Python text gives, leaves to that text every call with something unusual
about it, and raises what the text raises."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from rocmforge_amd import _lib, _native, ops, quantize as Q

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NAMES = ("gemv", "rms_norm_gemv", "mlp_swiglu", "gemm_f16", "arrange", "gemm_f16_arranged", "dequant")


def test_unusual_arguments_are_left_to_the_python_text():
    w, x = torch.zeros(20, dtype=torch.uint8), torch.zeros(32)
    assert _native.gemv(Q.Q4_0, w, x, 1, 32, None) is None                 # host tensors
    assert _native.gemv(Q.Q4_0, None, x, 1, 32, None) is None
    assert _native.gemv(1.0, w, x, 1, 32, None) is None
    assert _native.gemv(Q.Q4_0, w, x, 1 << 40, 32, None) is None
    assert _native.gemv(Q.Q4_0, w, x, -1, 32, None) is None
    assert _native.gemv(Q.Q4_0, torch.nn.Parameter(w, requires_grad=False), x, 1, 32, None) is None
    assert _native.dequant(Q.Q4_0, w, 32, None) is None and _native.arrange(x) is None
    with pytest.raises(TypeError):
        _native.gemv(Q.Q4_0, w, x)


def test_fake_tensors_are_left_to_the_python_text():
    """Device tensors by every property, but without memory: in their mode, and after it."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        w, x = torch.empty(20, dtype=torch.uint8, device="cuda"), torch.empty(32, device="cuda")
        assert w.is_cuda and _native.gemv(Q.Q4_0, w, x, 1, 32, None) is None
    assert _native.gemv(Q.Q4_0, w, x, 1, 32, None) is None
    assert _native.dequant(Q.Q4_0, w, 32, None) is None


def python(code, *argv, **env):
    return subprocess.run([sys.executable, "-c", code, *argv], cwd=ROOT, env={**os.environ, **env}, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=110)


def test_the_library_is_built_without_torch():
    """C++ and Rust programs need librfq.so alone: its targets ask for neither Python nor torch, and the default target does not fail
    where they are not there."""
    for args in (["lib"], ["all", "PYTHON=false"], ["PYTHON=/no/such/python"]):
        p = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "rocmforge_amd", "csrc"), *args], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        assert p.returncode == 0 and "-shared" in p.stdout and "rfq_api.hip" in p.stdout and "rfq_torch.cpp" not in p.stdout, (args, p.stdout[-2000:])
    p = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "rocmforge_amd", "csrc")], stdout=subprocess.PIPE, text=True)
    assert p.returncode == 0 and "rfq_torch.cpp" in p.stdout


def test_another_torch_than_the_one_built_for_is_refused():
    p = python("import torch; torch.__version__ = '0.0.0'; import rocmforge_amd.ops")
    assert p.returncode != 0 and f"was built for torch {torch.__version__}" in p.stdout and "0.0.0" in p.stdout


def test_operators_without_their_native_calls(tmp_path):
    """The library alone beside the package: the operators import, and every call goes through the text."""
    here = os.path.join(ROOT, "rocmforge_amd")
    package = tmp_path / "rocmforge_amd"
    package.mkdir()
    for name in os.listdir(here):
        if name.endswith(".py") or name == "librfq.so":
            (package / name).symlink_to(os.path.join(here, name))
    p = python("import sys; sys.path.insert(0, sys.argv[1])\n"
               "import torch; from rocmforge_amd import ops, _lib; assert _lib.lib().rfq_version() > 0 and ops.__file__.startswith(sys.argv[1])\n"
               "try: ops.gemv(2, torch.zeros(20, dtype=torch.uint8), torch.zeros(32), 1, 32)\n"
               "except ValueError as e: print('text:', e)\n", str(tmp_path))
    assert p.returncode == 0 and "text: packed weights must be" in p.stdout, p.stdout


def test_one_library_in_the_process(tmp_path):
    """The library beside the package, once, whatever other librfq.so the loader would find first (a C++ program's installation)."""
    subprocess.run(["gcc", "-shared", "-fPIC", "-x", "c", os.devnull, "-o", str(tmp_path / "librfq.so")], check=True)
    p = python("import rocmforge_amd.ops as o; o.lib()\n"
               "print(sorted({l.split()[-1] for l in open('/proc/self/maps') if 'librfq' in l}))", LD_LIBRARY_PATH=str(tmp_path) + ":" + os.environ.get("LD_LIBRARY_PATH", ""))
    assert p.returncode == 0 and str([os.path.join(os.path.realpath(ROOT), "rocmforge_amd", "librfq.so")]) in p.stdout, p.stdout


@pytest.fixture
def text_only(monkeypatch):
    def switch():
        for name in NAMES:
            monkeypatch.setattr(ops._native, name, lambda *a: None)
    return switch


@pytest.mark.gpu
def test_native_calls_equal_the_python_text(cuda, text_only):
    n, k, fmt = 96, 256, Q.Q8_0
    w = torch.from_numpy(Q.make_weights(fmt, n, k, seed=1)).to(cuda)
    sq = torch.from_numpy(Q.make_weights(fmt, k, k, seed=2)).to(cuda)
    rng = np.random.default_rng(3)
    x = torch.from_numpy(rng.standard_normal((3, k)).astype(np.float32)).to(cuda)
    nw = torch.ones(k, device=cuda) * 1.5
    a = x.half()

    def every():
        out, f = torch.empty((3, n), device=cuda), torch.empty(n * k, device=cuda)
        h = torch.empty((3, n), dtype=torch.float16, device=cuda)
        A = ops.ArrangedA(a)
        r = [ops.gemv(fmt, w, x, n, k), ops.gemv(fmt, w, x[0], n, k), ops.gemv(fmt, w, x, n, k, out=out), ops.rms_norm_gemv(fmt, w, x, nw, 1e-5, n, k),
             ops.rms_norm_gemv(fmt, w, x[1], nw, 1e-5, n, k), ops.mlp_swiglu(fmt, sq, sq, fmt, sq, x, nw, 1e-5, k, k),
             ops.mlp_swiglu(fmt, sq, sq, fmt, sq, x[2], None, 1e-5, k, k, scratch=torch.empty(16 * k, dtype=torch.uint8, device=cuda)),
             ops.gemm_f16(fmt, w, a, n, k), ops.gemm_f16(fmt, w, a, n, k, out_dtype=torch.float32, one_plane=True), ops.gemm_f16(fmt, w, a, n, k, out=h),
             ops.gemm_f16_arranged(fmt, w, A, n), ops.gemm_f16_arranged(fmt, w, A, n, out_dtype=torch.float32), ops.dequant(fmt, w, n * k), ops.dequant(fmt, w, n * k, out=f)]
        assert r[2] is out and r[9] is h and r[13] is f and (A.m, A.k) == (3, k)
        return r

    got = every()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):                                           # the current stream is the one that is taken
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            captured = ops.gemv(fmt, w, x[0], n, k)
        g.replay()
        side.synchronize()
    assert torch.equal(captured, got[1])
    text_only()
    for i, (p, q) in enumerate(zip(got, every())):
        assert p.shape == q.shape and p.dtype == q.dtype and torch.equal(p, q), i


@pytest.mark.gpu
def test_native_errors_are_the_python_texts(cuda):
    n, k = 8, 64
    w = torch.from_numpy(Q.make_weights(Q.Q4_0, n, k, seed=1)).to(cuda)
    x = torch.zeros((2, k), device=cuda)
    with pytest.raises(_lib.RfqError):
        ops.gemv(Q.Q4_0, w[:-20], x, n, k)                                   # bytes do not match the shape: the library refuses
    with pytest.raises(_lib.RfqError):
        ops.gemv(99, w, x, n, k)
    with pytest.raises(ValueError):
        ops.gemv(Q.Q4_0, w, x.t().contiguous().t(), n, k)                     # not contiguous
    with pytest.raises(ValueError):
        ops.gemm_f16(Q.Q4_0, w, x.half()[0], n, k)
    with pytest.raises(ValueError):
        ops.mlp_swiglu(Q.Q4_0, w, w[20:], Q.Q4_0, w, x, None, 1e-5, k, n)
    with pytest.raises(KeyError):
        ops.gemm_f16(Q.Q4_0, w, x.half(), n, k, out_dtype=torch.bfloat16)

    class Listener(torch.overrides.TorchFunctionMode):
        seen = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Listener.seen += 1
            return func(*args, **(kwargs or {}))

    with Listener():                                                        # whoever listens to torch functions hears the call
        y = ops.gemv(Q.Q4_0, w, x, n, k)
    assert Listener.seen > 0 and torch.equal(y, ops.gemv(Q.Q4_0, w, x, n, k))
    assert not ops.gemv(Q.Q4_0, w, x.clone().requires_grad_(), n, k).requires_grad


@pytest.mark.gpu
def test_calls_under_transforms_and_modes_end_as_the_python_texts(cuda, text_only):
    """Tensors without storage of their own (vmap, functional transforms), tangents and dispatch modes: the same result, or the same
    error, with the native calls as without them, and a mode hears as much."""
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode
    n, k, fmt = 8, 64, Q.Q4_0
    w = torch.from_numpy(Q.make_weights(fmt, n, k, seed=1)).to(cuda)
    wide = torch.from_numpy(Q.make_weights(fmt, k, k, seed=2)).to(cuda)
    x = torch.randn((3, k), device=cuda)
    calls = {"gemv": lambda v: ops.gemv(fmt, w, v, n, k), "norm": lambda v: ops.rms_norm_gemv(fmt, w, v, torch.ones(k, device=cuda), 1e-5, n, k),
             "mlp": lambda v: ops.mlp_swiglu(fmt, wide, wide, fmt, wide, v, None, 1e-5, k, k), "gemm": lambda v: ops.gemm_f16(fmt, w, v.half(), n, k),
             "arrange": lambda v: ops.ArrangedA(v.half()).buf, "dequant": lambda v: ops.dequant(fmt, w, n * k, out=v.new_empty(n * k))}

    class Heard(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    def dispatch(f):
        with Heard() as mode:
            y = f(x)
        assert mode.names
        return y, tuple(mode.names)

    def dual(f):
        with forward_ad.dual_level():
            y = forward_ad.unpack_dual(f(forward_ad.make_dual(x, torch.ones_like(x))))
            return y.primal, y.tangent is None

    contexts = {"vmap": lambda f: torch.func.vmap(f)(x.reshape(3, 1, k)), "grad": lambda f: torch.func.grad(lambda v: f(v).float().sum())(x),
                "jvp": lambda f: torch.func.jvp(f, (x,), (torch.ones_like(x),)), "dispatch": dispatch, "dual": dual,
                "inference": torch.inference_mode()(lambda f: f(x)), "grad mode": lambda f: f(x.clone().requires_grad_()).requires_grad}

    def outcome(context, f):
        try:
            return context(f)
        except Exception as e:                                              # (whatever torch says there)
            return type(e), str(e).splitlines()[0]

    def same(a, b):
        if isinstance(a, torch.Tensor): return isinstance(b, torch.Tensor) and a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
        if isinstance(a, tuple): return isinstance(b, tuple) and len(a) == len(b) and all(same(p, q) for p, q in zip(a, b))
        return a == b

    got = {(c, f): outcome(contexts[c], calls[f]) for c in contexts for f in calls}
    text_only()
    for (c, f), r in got.items():
        want = outcome(contexts[c], calls[f])
        assert same(r, want), (c, f, r, want)
    assert isinstance(got["dispatch", "gemv"][0], torch.Tensor) and isinstance(got["inference", "mlp"], torch.Tensor)
