"""The native host path of the Python binding (csrc/cq_host.cpp) without a GPU: the same source built for CPU tensors, with
entry points that only record the call and fill the output, against QuantLinear's general route (which refuses CPU tensors,
so what it adds to a product is stated here)."""
import ctypes
import importlib.util
import shutil
import subprocess
import sys
from pathlib import Path

import pytest
import torch

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "mixed-precision-cuda-kernel_amd"
K, N = 256, 64
FILL = 3.0  # what the stub entry points write into every output element

_CPU = [("PyInit_cherryq_host(", "PyInit_cherryq_host_cpu("),
        ("vec->is_cuda()", "vec->is_cpu()"), ("x->is_cuda()", "x->is_cpu()"), ("t->is_cuda()", "t->is_cpu()"),
        ("at::kCUDA, device", "at::kCPU"), ("c10::hip::current_device() != device", "device != -1"),
        ("c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream()", "reinterpret_cast<void *>((intptr_t)device)")]


def build_cpu_host(directory):
    spec = importlib.util.spec_from_file_location("cherryq_build", PKG / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    source = (PKG / "csrc" / "cq_host.cpp").read_text()
    for gpu, cpu in _CPU:
        assert gpu in source, gpu
        source = source.replace(gpu, cpu)
    assert "is_cuda" not in source
    (directory / "cq_host_cpu.cpp").write_text(source)
    cmd = build.host_command(directory / "cq_host_cpu.cpp", directory / "cherryq_host_cpu.so")
    subprocess.run([c if c != "-O2" else "-O0" for c in cmd], check=True, capture_output=True, text=True)


def load_cpu_host(directory):
    """The module, bound to stub entry points; its `calls` lists the entry points that ran."""
    spec = importlib.util.spec_from_file_location("cherryq_host_cpu", str(Path(directory) / "cherryq_host_cpu.so"))
    host = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(host)
    vp, i, sz = ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t
    calls = []

    def fill(name, out, batch, n):
        calls.append(name)
        (ctypes.c_uint16 * (batch * n)).from_address(out)[:] = [0x4200] * (batch * n)  # FILL in fp16
        return 0

    matmul = ctypes.CFUNCTYPE(i, vp, vp, vp, vp, vp, vp, i, i, i, i, i, i, vp, sz, vp, sz, vp)
    size4, size5 = ctypes.CFUNCTYPE(sz, i, i, i, i), ctypes.CFUNCTYPE(sz, i, i, i, i, i)
    over_stream = ctypes.CFUNCTYPE(i, i, vp, vp, sz, vp, i, i, i, i, i, vp)
    over_stream_rows = ctypes.CFUNCTYPE(i, i, vp, vp, sz, vp, i, i, i, i, i, vp, sz, vp)
    shape = ctypes.CFUNCTYPE(i, i, i, i, i, i, i)
    fused = [matmul(lambda *a, name=name: fill(name, a[5], a[6], a[8])) for name in ("vecquant4", "vecquant3")]
    f32 = matmul(lambda *a: calls.append("vecquant3_f32") or 0)
    stubs = [*fused, f32, size4(lambda *a: 4096), size4(lambda *a: 512), size4(lambda *a: 512), size5(lambda *a: 256),
             over_stream(lambda *a: fill("matvec_prepacked", a[4], a[5], a[7])),
             over_stream_rows(lambda *a: fill("matmul_prepacked", a[4], a[5], a[7])), shape(lambda *a: 1), shape(lambda *a: 1)]
    host.bind(tuple(ctypes.cast(s, vp).value for s in stubs))
    return host, calls, stubs


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    if shutil.which("g++") is None or not Path("/opt/rocm/include").is_dir():
        pytest.skip("needs g++ and the HIP headers")
    directory = tmp_path_factory.mktemp("host")
    build_cpu_host(directory)
    module, calls, stubs = load_cpu_host(directory)
    module_dir = str(directory)
    yield module, calls, module_dir
    del stubs


def layer(bias=False, stream=False, cls=None):
    from llama.qlinear import QuantLinear
    from llama.quantizer import FullSymQuantizer
    q = (cls or QuantLinear)(4, 128, FullSymQuantizer, 1 / 16, K, N, bias=bias)
    if stream:
        q._stream = torch.zeros(4096, dtype=torch.uint8)
    return q


@pytest.mark.parametrize("stream", [False, True])
@pytest.mark.parametrize("rows", [1, 3])
def test_every_form_of_a_bias_is_added(host, stream, rows):
    from llama.qlinear import QuantLinear
    linear = host[0].linear
    x = torch.ones(rows, K, dtype=torch.float16)
    b = torch.arange(N, dtype=torch.float16)
    plain, want = torch.full((rows, N), FILL, dtype=torch.float16), FILL + b.expand(rows, N)
    assert torch.equal(linear(layer(stream=stream), x), plain)

    def taken_or_left(q):  # None leaves the call to the general route, which reads self.bias
        out = linear(q, x)
        return out is None or torch.equal(out, want)

    q = layer(bias=True, stream=stream)
    q.bias.copy_(b)
    assert torch.equal(linear(q, x), want)                      # a buffer
    q = layer(stream=stream)
    q.bias = b.clone()
    assert torch.equal(linear(q, x), want)                      # set where none was registered
    q = layer(stream=stream)
    q.bias = torch.nn.Parameter(b.clone())
    assert "bias" in q._parameters and taken_or_left(q)         # a parameter where none was registered
    q = layer(bias=True, stream=stream)
    del q.bias
    q.bias = torch.nn.Parameter(b.clone())
    assert "bias" in q._parameters and taken_or_left(q)         # ... and in the place of the buffer

    class Own(QuantLinear):  # computed where it is asked for
        @property
        def bias(self):
            return b

        @bias.setter
        def bias(self, value):
            pass
    assert taken_or_left(layer(stream=stream, cls=Own))

    q = layer(bias=True, stream=stream)
    q.__class__ = type("Shadowed", (QuantLinear,), {"bias": property(lambda self: b)})
    assert "bias" in q._buffers and taken_or_left(q)            # the class's answer comes before the buffer

    class Scaled(torch.nn.Module):
        def forward(self, value):
            return value * 2

    q = layer(stream=stream)
    q.bias = torch.nn.Parameter(b / 2)
    torch.nn.utils.parametrize.register_parametrization(q, "bias", Scaled(), unsafe=True)
    assert torch.equal(q.bias.detach(), b) and taken_or_left(q)


def test_an_accumulate_without_a_truth_value_raises_before_the_launch(host, monkeypatch):
    module, calls, _ = host
    q, s = layer(), layer(stream=True)
    x, out, both = torch.ones(3, K, dtype=torch.float16), torch.zeros(3, N, dtype=torch.float16), torch.ones(2)
    calls.clear()
    reached = []  # a stub that is called with an exception set fails on it before it can record the call
    monkeypatch.setattr(sys, "unraisablehook", reached.append)
    with pytest.raises(RuntimeError):
        module.vecquant(4, x, q.qweight, q.cherry_weight, q.cherry_indices, q.scales, out, 128, both)
    with pytest.raises(RuntimeError):
        module.matvec_prepacked(4, x, s._stream, out, K, q.num_cherries, both)
    assert not calls and not reached and not out.any()


def test_plain(host):
    plain = host[0].plain
    t = torch.zeros(6, 16, dtype=torch.float16)
    assert plain(t, -1, 6, 16) and plain(torch.nn.Parameter(t), -1, 6, 16) and plain(t[2:], -1, 4, 16) and plain(t.view(-1), -1, 96)
    for bad in ((t, 0, 6, 16), (t, -1, 6), (t, -1, 16, 6), (t, -1, 6, 16, 1), (t.t(), -1, 16, 6), (t[:, :8], -1, 6, 8), (None, -1, 6, 16),
                (t.float(), -1, 6, 16), (t.bfloat16(), -1, 6, 16), (t.view(-1)[1:17], -1, 16), (t.to("meta"), -1, 6, 16), (t,)):
        assert plain(*bad) is False, bad
    seen = []
    torch.func.vmap(lambda v: seen.append(plain(v, -1, 16)) or v)(t)
    torch.func.grad(lambda v: seen.append(plain(v, -1, 6, 16)) or v.sum())(t)
    assert seen == [False, False]


_TRANSFORMED = """
import sys
sys.path[:0] = [{tests!r}, {pkg!r}]
import torch
import test_host_binding_cpu as t
host, calls, stubs = t.load_cpu_host({directory!r})
K, N = t.K, t.N
q, s = t.layer(), t.layer(stream=True)
x = torch.ones(3, K, dtype=torch.float16)
out = torch.zeros(3, N, dtype=torch.float16)
entries = dict(
    linear=lambda v: host.linear(q, v), linear_stream=lambda v: host.linear(s, v),
    vecquant=lambda v: host.vecquant(4, v, q.qweight, q.cherry_weight, q.cherry_indices, q.scales, out, 128, False),
    matvec_prepacked=lambda v: host.matvec_prepacked(4, v, s._stream, out, K, q.num_cherries, False))
transforms = dict(grad=lambda f: torch.func.grad(f)(x), vmap=lambda f: torch.func.vmap(f)(x.expand(2, 3, K)),
                  jvp=lambda f: torch.func.jvp(f, (x,), (x,)))
for name, f in entries.items():
    for kind, under in transforms.items():
        print(name, kind, flush=True)
        try:
            under(f)
        except RuntimeError as e:
            assert "data pointer" in str(e) or "storage" in str(e), (name, kind, e)
        else:
            raise AssertionError((name, kind, "no error"))
    assert calls == [], calls
    got = f(x)
    assert torch.equal(out if isinstance(got, int) else got, torch.full_like(out, t.FILL)), name
    assert len(calls) == 1
    calls.clear()
print("done")
"""


def test_tensors_without_memory_raise(host):
    """Under torch.func a call's tensors are wrappers without memory: an error as from data_ptr(), not a crash, nothing
    launched, and the kept buffers of the stream (here made by the first call, inside a transform) are ordinary ones."""
    code = _TRANSFORMED.format(tests=str(ROOT / "tests"), pkg=str(PKG), directory=host[2])
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and "done" in run.stdout, (run.returncode, run.stdout[-500:], run.stderr[-2000:])


def test_kept_buffers_are_made_without_the_pools_lock(tmp_path, monkeypatch):
    """Autograd's threads ask for a kept buffer without the interpreter's lock, other callers with it; an allocation that asks for
    the interpreter (a record of allocations with Python's stacks) does not meet a caller that holds it and waits for the pool."""
    if shutil.which("g++") is None or not Path("/opt/rocm/include").is_dir():
        pytest.skip("needs g++ and the HIP headers")
    asks = """#include <Python.h>
#include <ATen/ATen.h>
static at::Tensor asking_zeros(at::IntArrayRef sizes, const at::TensorOptions &options) {
    const PyGILState_STATE state = PyGILState_Ensure();
    PyRun_SimpleString("allocating()");
    PyGILState_Release(state);
    return at::zeros(sizes, options);
}
namespace {

using at::Tensor;"""
    monkeypatch.setattr(sys.modules[__name__], "_CPU", [*_CPU, ("at::zeros(", "asking_zeros("), ("namespace {\n\nusing at::Tensor;", asks)])
    build_cpu_host(tmp_path)
    script = f"""
import importlib.util, threading, torch
spec = importlib.util.spec_from_file_location("cherryq_host_cpu", {str(tmp_path / "cherryq_host_cpu.so")!r})
host = importlib.util.module_from_spec(spec)
spec.loader.exec_module(host)
threads, results = [], []

def allocating():
    if not threads:
        threads.append(threading.Thread(target=lambda: results.append(host.workspace(-1, 7, 64))))
        threads[0].start()
        threads[0].join()

results.append(host.workspace(-1, 7, 64))
assert len(threads) == 1 and len(results) == 2 and results[0].data_ptr() == results[1].data_ptr() == host.workspace(-1, 7, 64).data_ptr()
grown = host.workspace(-1, 7, results[0].numel() + 1)
assert grown.numel() == 2 * results[0].numel() and not grown.any() and host.workspace(-1, 7, 64).data_ptr() == grown.data_ptr()
print("done")
"""
    r = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "done\n", r.stderr


def test_a_workspace_made_while_a_stream_records_is_not_kept(host):
    """Its zeros are only recorded: another graph, or a call outside, would count from whatever lies there before the first replay."""
    module, recording = host[0], 1
    asks = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p)(lambda stream: recording if stream == 9 else 0)
    module.bind_capturing(ctypes.cast(asks, ctypes.c_void_p).value)
    try:
        one, two = module.workspace(-1, 9, 64), module.workspace(-1, 9, 64)
        assert one.data_ptr() != two.data_ptr() and one.numel() == two.numel() == 64 and not one.any()
        recording = 0
        kept = module.workspace(-1, 9, 64)
        assert kept.data_ptr() not in (one.data_ptr(), two.data_ptr()) and kept.numel() > 64
        recording = 1
        assert module.workspace(-1, 9, 64).data_ptr() == kept.data_ptr()  # a warm stream's is there
        larger = module.workspace(-1, 9, kept.numel() + 1)
        assert larger.numel() == kept.numel() + 1 and module.workspace(-1, 9, 64).data_ptr() == kept.data_ptr()
        scratch = module.scratch(-1, 9, 64)  # holds nothing from call to call
        assert module.scratch(-1, 9, 64).data_ptr() == scratch.data_ptr()
    finally:
        module.bind_capturing(0)


def test_the_library_beside_the_module_is_loaded(tmp_path):
    """... whatever lies on sys.path in front of it or was imported under its name."""
    (tmp_path / "cherryq_host.py").write_text("built_for = linear = None\n")
    code = (f"import sys; sys.path[:0] = [{str(tmp_path)!r}, {str(PKG)!r}]\n"
            "import cherryq_host, quant_cuda\n"
            "assert cherryq_host.linear is None\n"
            f"assert quant_cuda._host.__file__ == {str(PKG / 'cherryq_host.so')!r} and quant_cuda._host.linear")
    subprocess.run([sys.executable, "-c", code], check=True, timeout=300)


def test_another_torch_needs_another_host_library(monkeypatch, tmp_path):
    spec = importlib.util.spec_from_file_location("cherryq_build", PKG / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not build.LIB.exists() or build.needs_build():
        pytest.skip("the libraries are not built from these sources")
    version = torch.__version__
    monkeypatch.setattr(torch, "__version__", version + ".1")
    assert build.needs_build()
    monkeypatch.setattr(torch, "__version__", version[:-1])
    assert build.needs_build()


def test_descriptions_of_plain_modules_only(host):
    """What the whole-prompt call is told of a product's modules, and which modules are left to their own calls."""
    import cherryq_decoder as dec
    from llama.qlinear import QuantLinear
    from llama.quantizer import FullSymQuantizer
    module = host[0]

    def describe(*mods, rows=40, cls=QuantLinear):
        product, held = dec._PrefillProduct(), []
        ok = module.describe(ctypes.addressof(product), rows, -1, cls, held, *mods)
        return (product, held) if ok else None

    mods = [layer(), layer(), layer()]
    for n in (1, 2, 3):
        product, held = describe(*mods[:n])
        assert (product.n_layers, product.w_bits, product.in_features, product.group_size) == (n, 4, K, 128)
        assert product.num_cherries == mods[0].num_cherries and len(held) == 4 * n
        for w, m in zip(product.layers, mods[:n]):
            assert (w.qweight, w.scales, w.cherry_weight, w.cherry_indices, w.out_features) == (
                m.qweight.data_ptr(), m.scales.data_ptr(), m.cherry_weight.data_ptr(), m.cherry_indices.data_ptr(), N)
        assert any(t is mods[0].qweight for t in held)
    assert describe(mods[0], rows=QuantLinear.prefill_rows) is None
    assert describe(mods[0], layer(bias=True)) is None
    assert describe(mods[0], torch.nn.Linear(K, N)) is None and describe(mods[0], None) is None
    assert describe(type("Own", (QuantLinear,), {})(4, 128, FullSymQuantizer, 1 / 16, K, N, bias=False)) is None
    assert describe(QuantLinear(3, 128, FullSymQuantizer, 1 / 16, K, N, bias=False), mods[0]) is None  # not of one kind
    for change in (lambda q: q.register_forward_hook(lambda *a: None), lambda q: q.register_forward_pre_hook(lambda *a: None),
                   lambda q: setattr(q, "forward", lambda x: x), lambda q: setattr(q, "dequantized", True),
                   lambda q: setattr(q, "_released", True), lambda q: setattr(q, "bias", torch.nn.Parameter(torch.zeros(N))),
                   lambda q: setattr(q, "scales", q.scales.float()), lambda q: setattr(q, "qweight", q.qweight[:-1]),
                   lambda q: setattr(q, "cherry_weight", q.cherry_weight.t().contiguous().t())):
        q = layer()
        assert describe(q) is not None
        change(q)
        assert describe(q) is None
    with QuantLinear.dmode(False):
        assert describe(mods[0]) is None


def dense_layer(bits=4, group=128, k=K, n=N, seed=0):
    from llama.qlinear import QuantLinear
    from llama.quantizer import FullSymQuantizer
    gen = torch.Generator().manual_seed(seed)
    q = QuantLinear(bits, group, FullSymQuantizer, 1 / 16, k, n, bias=False)
    q.qweight = torch.randint(0, 256, q.qweight.shape, dtype=torch.uint8, generator=gen)
    q.scales = (torch.rand(q.scales.shape, generator=gen) * 0.02 + 0.001).half()
    q.cherry_weight = torch.randn(q.cherry_weight.shape, generator=gen).half()
    q.cherry_indices = torch.randperm(k, generator=gen)[:q.num_cherries].sort().values.to(torch.int16)
    return q


@pytest.mark.parametrize("rows", [512, 600, 2303])
@pytest.mark.parametrize("bits,group", [(4, 128), (4, 64), (3, 24)])
def test_many_rows_on_the_host(rows, bits, group):
    """From 512 rows there is a dense product for what the fused kernel refuses, tensors on the host among it."""
    q, x = dense_layer(bits, group), torch.randn(rows, K, generator=torch.Generator().manual_seed(1)).half()
    assert torch.equal(q(x), torch.matmul(x, q.unpack().t()))
    with pytest.raises(RuntimeError):
        q(x[:511])


class _DispatchMode(torch.utils._python_dispatch.TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _FunctionMode(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_many_rows_are_taken_where_a_launch_is_sure_to_do(host):
    """From 512 rows the native call asks whether the prompt kernel takes the product, and leaves calls whose operations something
    records, replaces or transforms to torch's."""
    module, calls, _ = host
    answers, asked = [1], []
    stub = ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_int] * 6, ctypes.c_void_p)(lambda *a: asked.append(a[:6]) or answers[0])
    q, x = layer(), torch.ones(600, K, dtype=torch.float16)
    want = torch.full((600, N), FILL, dtype=torch.float16)
    assert module.linear(q, x) is None  # no one to ask
    try:
        module.bind_prompt(ctypes.cast(stub, ctypes.c_void_p).value)
        assert torch.equal(module.linear(q, x), want) and asked == [(4, 600, K, N, q.num_cherries, 128)]
        with _DispatchMode():
            assert module.linear(q, x) is None
        with _FunctionMode():
            assert module.linear(q, x) is None
        left = []
        torch.func.vmap(lambda t: left.append(module.linear(q, t)) or t)(x.expand(2, 600, K))
        torch.jit.trace(lambda t: left.append(module.linear(q, t)) or t * 1, x, check_trace=False)
        assert left == [None, None]
        assert torch.equal(module.linear(q, x), want)
        answers[0] = 0
        assert module.linear(q, x) is None
        assert torch.equal(module.linear(q, x[:511]), want[:511])
    finally:
        module.bind_prompt(0)


def test_traces_of_many_rows_hold_the_product():
    q, gen = dense_layer(), torch.Generator().manual_seed(1)
    x, other = (torch.randn(600, K, generator=gen).half() for _ in range(2))
    traced = torch.jit.trace(q, x)
    assert torch.equal(traced(other), q(other))


def test_descriptions_of_layers_that_the_entry_point_takes(host):
    """... only: the others' own calls may go to a dense product."""
    import cherryq_decoder as dec
    from llama.qlinear import QuantLinear
    from llama.quantizer import FullSymQuantizer
    module = host[0]
    answers, product = [1], dec._PrefillProduct()
    stub = ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_int] * 6, ctypes.c_void_p)(lambda *a: answers[0])

    def described(q, rows=40):
        return module.describe(ctypes.addressof(product), rows, -1, QuantLinear, [], q)

    assert described(layer()) and not described(layer(), 600)
    try:
        module.bind_prompt(ctypes.cast(stub, ctypes.c_void_p).value)
        assert described(layer(), 600)
        answers[0] = 0
        assert not described(layer(), 600)
    finally:
        module.bind_prompt(0)
    for bits, group in ((4, 64), (3, 24)):
        assert not described(QuantLinear(bits, group, FullSymQuantizer, 1 / 16, K, N, bias=False))
    for name, nbytes in (("qweight", 4), ("scales", 8), ("cherry_weight", 2), ("cherry_indices", 2)):
        q = layer()
        t = getattr(q, name)
        flat = torch.zeros(t.numel() + 8, dtype=t.dtype)[nbytes // t.element_size():][:t.numel()]
        setattr(q, name, flat.view(t.shape))
        assert not described(q), name
