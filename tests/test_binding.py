"""The native entry points against the package's Python functions that they take the plain calls off (`__wrapped__`)."""
import copy
import importlib.util
import inspect
import os
import pickle
import subprocess
import sys
import threading
import warnings

import pytest
import torch

from test_gpu_parity import pa  # noqa: F401

import __graft_entry__ as ge

NAMES = ["gemm", "gemm_w8a8", "gemm_mx", "gemv_mxfp4", "gemv_mxfp4_packed", "tquant_int8", "tquant_mx", "tdequant"]


def outcome(f, *args, **kw):
    try:
        return f(*args, **kw)
    except Exception as e:  # noqa: BLE001
        return type(e), str(e)


@pytest.mark.parametrize("name", NAMES)
def test_an_entry_point_looks_like_its_function(name):
    p = ge.load_package()
    f = getattr(p, name)
    assert f is not f.__wrapped__ and inspect.isfunction(f.__wrapped__)
    assert inspect.signature(f) == inspect.signature(f.__wrapped__)
    assert (f.__name__, f.__qualname__, f.__module__, f.__doc__, f.__defaults__) == tuple(
        getattr(f.__wrapped__, a) for a in ("__name__", "__qualname__", "__module__", "__doc__", "__defaults__"))
    assert copy.copy(f) is f and copy.deepcopy(f) is f and pickle.loads(pickle.dumps(f)) is f

    class Holder:
        method, function = f, f.__wrapped__
    assert outcome(Holder().method) == outcome(Holder().function)  # (a class attribute binds to its instances)


@pytest.mark.parametrize("name", NAMES)
def test_refused_calls_raise_what_the_function_raises(name):
    f = getattr(ge.load_package(), name)
    a, v = torch.zeros(4, 64), torch.zeros(4)
    calls = [((), {}), ((a,), {}), ((a, a, 2), {"wrong": 1}), ((a, a, 2), {"a": a}), ((a,) * 30, {}), ((a, a, a, a, 4, 4, 64, 6, 6), {}), ((a, v), {}),
             ((a, 0), {}), ((a, v, v), {}), ((1, 2, 3, 4, 5, 6, 7, 8, 9), {}), ((a, a, 4, 64), {}), ((a, a, a, 4, 64), {}), ((None,) * 4, {}),
             ((a, a, "f32"), {}), ((a, a, 2 ** 70), {})]
    for args, kw in calls:
        assert outcome(f, *args, **kw) == outcome(f.__wrapped__, *args, **kw), (name, args, kw)


def _package_anew():
    spec = importlib.util.spec_from_file_location("package_loaded_anew", os.path.join(ge.PKG_DIR, "__init__.py"), submodule_search_locations=[ge.PKG_DIR])
    module = importlib.util.module_from_spec(spec)
    with warnings.catch_warnings(record=True) as raised:
        warnings.simplefilter("always")
        spec.loader.exec_module(module)
    return module, [w for w in raised if issubclass(w.category, RuntimeWarning)]


@pytest.mark.parametrize("what", ["version", "commit", "python", "none"])
def test_another_torch_or_python_keeps_the_functions(monkeypatch, what):
    import sysconfig
    if what == "version":
        monkeypatch.setattr(torch, "__version__", torch.__version__ + ".post1")
    elif what == "commit":
        monkeypatch.setattr(torch.version, "git_version", "0" * 40)
    elif what == "python":
        suffix = sysconfig.get_config_var("EXT_SUFFIX")
        monkeypatch.setattr(sysconfig, "get_config_var", lambda name: ".other" + suffix)
    module, raised = _package_anew()
    assert [inspect.isfunction(getattr(module, n)) for n in NAMES] == [what != "none"] * len(NAMES)
    assert len(raised) == (what != "none")


def _make(python, *targets):
    return subprocess.run(["make", "-C", ge.PKG_DIR, "-n", "-B", f"PYTHON={python}", *targets], capture_output=True, text=True)


def test_the_build_needs_no_torch():
    """Without a torch (an interpreter without its packages, no interpreter at all) everything but the binding is built; with one the
    binding is named and compiled for the interpreter that was asked for."""
    for python in (sys.executable + " -S", "/no/such/python"):
        steps = _make(python)
        assert steps.returncode == 0 and "entry_points.cpp" not in steps.stdout, steps.stdout[-2000:] + steps.stderr
        for lib in ("libptoamd.so", "libpto_gemm_performance.so", "libpto_gemm_tiled.so", "libpto_mxmatmul_performance.so"):
            assert f"-o lib/{lib}" in steps.stdout, lib
    import sysconfig
    steps = _make(sys.executable)
    assert steps.returncode == 0 and "ptoamd_binding" + sysconfig.get_config_var("EXT_SUFFIX") in steps.stdout
    assert f"{torch.__version__} {torch.version.git_version}" in steps.stdout and sysconfig.get_paths()["include"] in steps.stdout


def _cases(p):
    """name -> calls as (args, keywords); calls that write into an `out` of their own get it from a function."""
    g = torch.Generator(device="cuda").manual_seed(5)

    def rnd(*shape, dtype=torch.bfloat16):
        return torch.randn(shape, generator=g, device="cuda").to(dtype)

    def ints(*shape):
        return torch.randint(-100, 101, shape, generator=g, device="cuda", dtype=torch.int8)
    a, b, wide = rnd(33, 96), rnd(40, 96), rnd(40, 128)
    nd, bias, ws = rnd(96, 40), torch.rand(40, generator=g, device="cuda"), torch.empty(40 * 256, dtype=torch.uint8, device="cuda")
    x8, w8, sa, sb = ints(33, 96), ints(40, 96), torch.rand(33, generator=g, device="cuda"), torch.rand(40, generator=g, device="cuda")
    f32 = rnd(64, 128, dtype=torch.float32)
    ca, ea = p.tquant_mx(rnd(33, 256), p.OCP_MXFP8, want_aux=False)
    cb, eb = p.tquant_mx(rnd(40, 256), p.OCP_MXFP8, want_aux=False)
    xg = rnd(5, 2048)
    w4, s4 = p.tquant_mx(rnd(48, 2048), p.OCP_MXFP4, want_aux=False)
    packed = p.gemv_mxfp4_pack(w4, s4, 48, 2048)
    out = lambda n=40, t=torch.float32, w=40: torch.zeros((33, w), dtype=t, device="cuda")[:, :n]  # noqa: E731
    return {
        "gemm": [((a, b, p.BF16), {}), ((a, b, p.BF16, p.BF16, p.B_DN), {}), ((a, nd, p.BF16, p.F16, p.B_ND), {}), ((a, wide[:, :96], p.BF16), {}),
                 ((a, b, p.BF16), {"bias": bias, "relu": True}), ((a, nd, p.BF16), {"b_layout": p.B_ND, "workspace": ws, "bias": None}),
                 ((a, b, p.BF16), {"out": out}), ((a, b, p.BF16), {"out": lambda: out(40, w=44)}), ((a, b), {"ab_type": p.BF16, "relu": p.RELU}),
                 ((a, b, p.BF16), {"c_in": out}), ((a, b, p.BF16), {"k": 64}), ((a.t(), b, p.BF16), {}), ((a, b[:, ::2], p.BF16), {}),
                 ((a, b, p.BF16, p.I32), {}), ((a, b, p.BF16, 99), {}), ((a[:0], b, p.BF16), {}), ((a, b, p.BF16), {"stream": torch.cuda.current_stream()}),
                 ((a, torch.nn.Parameter(b.float()).to(torch.bfloat16), p.BF16), {}), ((a, torch.nn.Parameter(b), p.BF16), {}), ((a, b, p.BF16), {"relu": 8}),
                 ((a, b, p.BF16), {"bias": bias.cpu()}), ((a, b.cpu(), p.BF16), {}), ((a[0], b, p.BF16), {}), ((a, nd, p.BF16), {"b_layout": p.B_ND, "workspace": ws[:128]})],
        "gemm_w8a8": [((x8, w8, sa, sb), {}), ((x8, w8, sa, sb), {"want_acc": True}), ((x8, w8, sa, sb), {"out": lambda: out(t=torch.bfloat16)}),
                      ((x8, w8.t().contiguous(), sa, sb, p.B_ND), {}), ((x8, w8, sa[:, None], sb), {}), ((x8, w8, sa[::2], sb), {}), ((x8, w8, None, sb), {})],
        "gemm_mx": [((ca, cb, ea, eb, 33, 40, 256, p.E4M3, p.E4M3), {}), ((ca, cb, ea, eb, 33, 40, 256, p.E4M3, p.E4M3, p.BF16), {}),
                    ((ca, cb, ea, eb, 33, 40, 256, p.E4M3, p.E4M3), {"out": out}), ((ca, cb, ea, eb, 33, 40, 256, p.E4M3, p.E4M3), {"bias": bias}),
                    ((ca, cb, ea, eb, 33, 40, 250, p.E4M3, p.E4M3), {}), ((ca, cb, ea, eb, 33, 40, 256, p.E4M3, p.E2M1), {}),
                    ((ca.flatten(), cb, ea, eb, 33, 40, 256, p.E4M3, p.E4M3), {}), ((ca, cb, ea, eb, -1, 40, 256, p.E4M3, p.E4M3), {})],
        "gemv_mxfp4": [((xg, w4, s4, 48, 2048), {}), ((xg, w4, s4, 48, 2048, p.BF16), {}), ((xg[:, :1024], w4, s4, 48, 1024), {}), ((xg, w4, s4, 48, 100), {}),
                       ((xg.repeat(4, 1), w4, s4, 48, 2048), {})],
        "gemv_mxfp4_packed": [((xg, packed, 48, 2048), {}), ((xg, packed, 48, 2048, p.F16), {}), ((xg, packed, 48, 1000), {}), ((xg, packed[1:], 48, 2048), {})],
        "tquant_int8": [((f32, sa[:1].expand(64).contiguous()), {}), ((f32, torch.rand(64, device="cuda", generator=g), torch.rand(64, device="cuda", generator=g)), {}),
                        ((f32, torch.rand(8, 2, device="cuda", generator=g)), {}), ((f32.t(), sa), {})],
        "tquant_mx": [((f32, p.OCP_MXFP8), {}), ((f32, p.OCP_MXFP4, 1, False), {}), ((f32.half(), p.NV_MXFP4), {"axis": 0}), ((f32.bfloat16(), p.NV_MXFP8), {"want_aux": False}),
                      ((f32.double(), p.OCP_MXFP8), {}), ((f32[:, :40].contiguous(), p.OCP_MXFP8), {}), ((f32, 9), {}), ((f32, p.OCP_MXFP8, 2), {})],
        "tdequant": [((x8, sa, sa), {}), ((x8.short(), sa, sa), {}), ((x8.int(), sa, sa), {}), ((x8.float(), sa, sa), {}), ((x8, sa[:, None].repeat(1, 4), sa[:, None].repeat(1, 4)), {}),
                     ((x8, sa.cpu(), sa), {})],
    }


def same(x, y):
    if isinstance(x, torch.Tensor):
        return isinstance(y, torch.Tensor) and x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride() and torch.equal(
            x.contiguous().view(torch.uint8), y.contiguous().view(torch.uint8))
    if isinstance(x, tuple) and x and isinstance(x[0], torch.Tensor):
        return isinstance(y, tuple) and len(x) == len(y) and all(same(p, q) for p, q in zip(x, y))
    return x == y


@pytest.mark.gpu
@pytest.mark.parametrize("name", NAMES)
def test_every_form_gives_what_the_function_gives(pa, name):  # noqa: F811
    f = getattr(pa, name)
    for i, (args, kw) in enumerate(_cases(pa)[name]):
        got, ref = (outcome(g, *args, **{k: v() if callable(v) else v for k, v in kw.items()}) for g in (f, f.__wrapped__))
        assert same(got, ref), (name, i, got, ref)


@pytest.mark.gpu
def test_streams_threads_and_modes(pa):  # noqa: F811
    from torch._subclasses.fake_tensor import FakeTensorMode
    (a, b, t), _ = _cases(pa)["gemm"][0]
    ref = pa.gemm.__wrapped__(a, b, t)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = pa.gemm(a, b, t)
    side.synchronize()
    assert torch.equal(got, ref)
    results = [None] * 4

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                results[i] = pa.gemm(a, b, t)
            torch.cuda.current_stream().synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    torch.cuda.synchronize()
    [x.start() for x in threads], [x.join() for x in threads]
    assert all(torch.equal(r, ref) for r in results)
    with torch.device("cuda"):
        assert torch.equal(pa.gemm(a, b, t), ref)
    with torch.inference_mode():
        assert pa.gemm(a, b, t).is_inference() and torch.equal(pa.gemm(a, b, t), ref)
    grad = pa.gemm(a.clone().requires_grad_(), b, t)
    assert torch.equal(grad, ref) and not grad.requires_grad
    with FakeTensorMode() as mode:
        fa, fb = mode.from_tensor(a), mode.from_tensor(b)
        assert outcome(pa.gemm, fa, fb, t)[0] is outcome(pa.gemm.__wrapped__, fa, fb, t)[0]
    batch = torch.stack([a, a])
    errors = [outcome(lambda f=f: torch.vmap(lambda x: f(x, b, t))(batch))[0] for f in (pa.gemm, pa.gemm.__wrapped__)]
    assert errors[0] is errors[1]


@pytest.mark.gpu
def test_capture_and_replay(pa):  # noqa: F811
    (a, b, t), _ = _cases(pa)["gemm"][0]
    pa.gemm(a, b, t)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = pa.gemm(a, b, t)
    for i in range(3):
        a.mul_(1.5)
        graph.replay()
        assert torch.equal(got, pa.gemm.__wrapped__(a, b, t)), i


@pytest.mark.gpu
def test_compiled_and_traced_callers(pa):  # noqa: F811
    """torch.compile breaks its graph at an entry point and calls it: the eager result.  torch.jit.trace records what it records of
    the Python function (the allocation of the result, which nothing fills when the trace is run)."""
    (a, b, t), _ = _cases(pa)["gemm"][0]
    ref = pa.gemm.__wrapped__(a + 1, b, t) * 2
    torch._dynamo.reset()
    compiled = torch.compile(lambda x: pa.gemm(x + 1, b, t) * 2, backend="eager")
    for _ in range(2):
        assert torch.equal(compiled(a), ref)
    code = [torch.jit.trace(lambda x: f(x + 1, b, t) * 2, (a,), check_trace=False).code for f in (pa.gemm, pa.gemm.__wrapped__)]  # noqa: B023
    assert code[0] == code[1], code
