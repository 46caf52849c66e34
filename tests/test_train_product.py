"""The training layer in one native call (csrc/cq_host.cpp: train_linear) and its matrix products (csrc/cq_gemm.hip).

Bound of the kernel: fp32 sums of exact 16-bit products, rounded once.  The rounding is half an ulp of the result's type, at most
2^-11 (fp16) or 2^-8 (bf16) of an element, its 2-norm about 0.6 of that; a sum of K terms of random signs adds about sqrt(K) 2^-24 of
the result, 2^-17 at the largest K here.  So 2^-11 / 2^-8 of the 2-norm holds with room."""
import contextlib
import ctypes
import gc
import shutil
import weakref
from pathlib import Path

import pytest
import torch

import llama.cherry_linear as cl

LIMIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


# ---- the native call, built for CPU tensors, with stand-ins for the kernels -----------------------------------
@pytest.fixture(scope="module")
def native(tmp_path_factory):
    """(train_linear, calls): the stand-in for the fake quantisation halves the weight; products come from torch."""
    import test_host_binding_cpu as t
    if shutil.which("g++") is None or not Path("/opt/rocm/include").is_dir():
        pytest.skip("needs g++ and the HIP headers")
    directory = tmp_path_factory.mktemp("train")
    t.build_cpu_host(directory)
    host, _, stubs = t.load_cpu_host(directory)
    vp, i, sz, calls, workspaces = ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t, [], []

    def at(address, rows, cols, dtype):
        return torch.frombuffer((ctypes.c_uint8 * (rows * cols * dtype.itemsize)).from_address(address), dtype=dtype).view(rows, cols)

    def quantise(dtype):
        def f(bits, w, idx, out, k, n, c, g, ste, stream):
            if bits > 4:
                return -1
            calls.append("quantise")
            at(out, n, k, dtype).copy_(at(w, n, k, dtype) / 2)
            return 0
        return ctypes.CFUNCTYPE(i, i, vp, vp, vp, i, i, i, i, i, vp)(f)

    def gemm(bf16, a_by_k, b_by_k, a, b, out, m, n, k, ws, wsz, sc, scz, stream):
        calls.append((a_by_k, b_by_k))
        dtype = torch.bfloat16 if bf16 else torch.float16
        x, y = at(a, k if a_by_k else m, m if a_by_k else k, dtype), at(b, k if b_by_k else n, n if b_by_k else k, dtype)
        assert wsz >= 16 and scz == 64
        workspaces.append((ctypes.string_at(ws, 16), wsz))
        at(out, m, n, dtype).copy_((x.t() if a_by_k else x).float() @ (y if b_by_k else y.t()).float())
        return 0

    size = ctypes.CFUNCTYPE(sz, i, i, i)
    mine = [quantise(d) for d in (torch.float16, torch.bfloat16, torch.float32)]
    mine += [size(lambda *_: 16), size(lambda *_: 64), ctypes.CFUNCTYPE(i, i, i, i, i, i)(lambda *a: 1),
             ctypes.CFUNCTYPE(i, i, i, i, vp, vp, vp, i, i, i, vp, sz, vp, sz, vp)(gemm)]
    host.bind_train(tuple(ctypes.cast(f, vp).value for f in mine))

    def call(x, w, bits=4):
        return host.train_linear(x, w, torch.arange(8, dtype=torch.int32), bits, 8)

    call.host, call.workspaces = host, workspaces
    yield call, calls
    del stubs, mine


def through_torch(x, w):
    return torch.nn.functional.linear(x, (w.detach() / 2 - w).detach() + w)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(8, 16), (2, 3, 16)])
@pytest.mark.parametrize("needs", [(True, True), (True, False), (False, True)])
def test_native_call_and_gradients_equal_torch(native, dtype, shape, needs):
    torch.manual_seed(0)
    x, w, g = torch.randn(shape).to(dtype), torch.randn(24, 16).to(dtype), torch.randn(*shape[:-1], 24).to(dtype)
    results = []
    for f in (native[0], through_torch):
        native[1].clear()
        xs, ws = x.clone().requires_grad_(needs[0]), w.clone().requires_grad_(needs[1])
        y = f(xs, ws)
        y += 1  # a bias, in place
        y.backward(g)
        results.append((y.detach(), xs.grad, ws.grad))
        if f is native[0]:
            own = [] if dtype == torch.float32 else [(0, 0)] + [(0, 1)] * needs[0] + [(1, 1)] * needs[1]
            assert native[1] == ["quantise"] + own
    for a, b in zip(*results):
        assert (a is None) == (b is None)
        if a is not None:  # another order of the sums, rounded once more
            torch.testing.assert_close(a, b, rtol=2 * torch.finfo(dtype).eps, atol=8 * torch.finfo(dtype).eps)


def test_native_call_keeps_what_a_gradient_reads(native):
    x, w = torch.randn(6, 16, requires_grad=True), torch.randn(24, 16)
    h = x * 1
    y = native[0](h, w)
    h.add_(1)  # torch's linear with a frozen weight does not keep its input
    y.sum().backward()
    torch.testing.assert_close(x.grad, w.sum(0).expand_as(x) / 2)
    w.requires_grad_()
    y = native[0](x.detach(), w)
    with torch.no_grad():
        w.add_(1)  # an optimiser's step in front of the gradients: the quantised weight is what was multiplied
    y.sum().backward()
    torch.testing.assert_close(w.grad, x.detach().sum(0).expand_as(w))
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t) or len(kept) - 1, lambda i: kept[i] * 2):
        y = native[0](x, w)
    dx, dw = torch.autograd.grad(y, (x, w), torch.ones_like(y))
    assert len(kept) == 2
    torch.testing.assert_close((dx, dw), ((w.sum(0).expand_as(x)).detach(), 2 * x.sum(0).expand_as(w).detach()))


@pytest.mark.parametrize("twice", [False, True])
def test_gradients_that_nobody_asks_for_are_not_computed(native, twice):
    f, calls = native
    x, w, g = torch.randn(6, 16).half().requires_grad_(), torch.randn(24, 16).half().requires_grad_(), torch.randn(6, 24).half()
    want = torch.autograd.grad(f(x, w), (x, w), g)
    for i, asked in enumerate((x, w)):
        y = f(x, w)
        calls.clear()
        with Counted() if twice else contextlib.nullcontext() as mode:
            dt, = torch.autograd.grad(y, asked, g, create_graph=twice)
        assert (calls == [] and mode.products == 1) if twice else calls == [(i, 1)]
        torch.testing.assert_close(dt.detach(), want[i], rtol=2 ** -9, atol=2 ** -7)
    y = f(x, w)
    y.backward(g, inputs=[x])
    assert calls[-1] == (0, 1) and w.grad is None


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_second_derivatives_equal_torch(native, dtype):
    torch.manual_seed(1)
    x, w, v = torch.randn(4, 16).to(dtype), torch.randn(8, 16).to(dtype), torch.randn(4, 16).to(dtype)
    results = []
    for f in (native[0], through_torch):
        xs, ws = x.clone().requires_grad_(), w.clone().requires_grad_()
        (dx, dw) = torch.autograd.grad((f(xs, ws).float() ** 2).sum(), (xs, ws), create_graph=True)
        results.append(torch.autograd.grad((dx * v).float().sum() + (dw.float() ** 2).mean(), (xs, ws)))
    torch.testing.assert_close(*results, rtol=40 * torch.finfo(dtype).eps, atol=100 * torch.finfo(dtype).eps)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_second_derivatives_reach_the_weight_as_it_was(native, dtype):
    """A computed weight that is changed in place behind the forward pass: the gradient goes where it came from then.  The node keeps
    what its gradients multiply, not the weight."""
    torch.manual_seed(3)
    x, w = torch.randn(4, 16).to(dtype), torch.randn(8, 16).to(dtype)
    results = []
    for f in (native[0], through_torch):
        xs, ws = x.clone().requires_grad_(), w.clone().requires_grad_()
        h = ws * 1
        y = f(xs, h)
        h.mul_(3)
        dx, = torch.autograd.grad((y.float() ** 2).sum(), xs, create_graph=True)
        results.append(torch.autograd.grad(dx.float().sum(), (xs, ws)))
    torch.testing.assert_close(*results, rtol=40 * torch.finfo(dtype).eps, atol=100 * torch.finfo(dtype).eps)
    h = w.clone().requires_grad_() * 1
    y, gone = native[0](x.clone().requires_grad_(), h), weakref.ref(h)
    del h
    gc.collect()
    assert gone() is None and y.grad_fn is not None


def test_calls_that_are_not_plain_are_left_to_the_general_route(native):
    f, calls = native
    x, w = torch.randn(6, 16), torch.randn(24, 16)
    assert f(x, w) is not None and f(x[:, ::2].repeat(1, 2), w) is not None
    calls.clear()

    class Sub(torch.Tensor):
        pass

    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert all(r is None for r in (f(x.double(), w.double()), f(x.half(), w), f(x[:, :8], w), f(x[0], w), f(x, w.t().contiguous().t()), f(x, w, 8),
                                   f(x[:0], w), f(x.as_subclass(Sub), w), f(x.to("meta"), w)))
    with torch.autograd.forward_ad.dual_level():
        assert f(torch.autograd.forward_ad.make_dual(x, x), w) is None
        assert f(x, torch.autograd.forward_ad.make_dual(w, w)) is None
    with Mode():
        assert f(x, w) is None
    with torch.autocast("cpu", torch.bfloat16):
        assert f(x, w) is None
    torch.func.vmap(lambda x: [x, [None for r in [f(x, w)] if r is not None][:1]][0])(x[None])
    assert calls == []


def other_dual(g):
    return torch.autograd.forward_ad.make_dual(g, torch.full_like(g, 0.5))


class Counted(torch.utils._python_dispatch.TorchDispatchMode):
    """The products that a dispatch mode sees."""
    products = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.products += func.overloadpacket in (torch.ops.aten.mm, torch.ops.aten.bmm, torch.ops.aten.addmm)
        return func(*args, **(kwargs or {}))


def gradients_with_a_tangent(f, x, w, g):
    with torch.autograd.forward_ad.dual_level():
        out = torch.autograd.grad(f(x, w), (x, w), other_dual(g))
        return [torch.autograd.forward_ad.unpack_dual(t).tangent for t in out]


def a_later_layer_with_a_tangent(f, x, w, g):
    with torch.autograd.forward_ad.dual_level():
        y = torch.nn.functional.linear(f(x, w), other_dual(w[:, :8].repeat(1, 3).detach()))
        out = torch.autograd.grad((y * y).mean(), (x, w))
        return [torch.autograd.forward_ad.unpack_dual(t).tangent for t in out]


def under_a_mode(f, x, w, g):
    y = f(x, w)
    with Counted() as mode:
        out = torch.autograd.grad(y, (x, w), g)
    return [*out, torch.tensor(float(mode.products))]


def under_autocast(f, x, w, g):
    y, other = f(x, w), torch.float16 if x.dtype == torch.bfloat16 else torch.bfloat16
    with torch.autocast("cpu", other):
        return torch.autograd.grad(y, (x, w), g)


def of_a_wrapper(f, x, w, g):
    from torch.testing._internal.two_tensor import TwoTensor
    out = torch.autograd.grad(f(x, w), (x, w), TwoTensor(g, g * 2))
    return [t for two in out for t in (two.a, two.b)]


def kept(change):
    def call(f, x, w, g):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), change):
            y = f(x, w)
        return torch.autograd.grad(y, (x, w), g)
    return call


# what arrives at the backward of a forward pass that was plain
ARRIVES = {
    "tangent": gradients_with_a_tangent,
    "later tangent": a_later_layer_with_a_tangent,
    "batched": lambda f, x, w, g: torch.autograd.grad(f(x, w), (x, w), torch.stack([g, 2 * g, g * g]), is_grads_batched=True),
    "vmap": lambda f, x, w, g: (lambda y: torch.func.vmap(lambda v: torch.autograd.grad(y, (x, w), v, retain_graph=True))(torch.stack([g, 2 * g])))(f(x, w)),
    "jacobian": lambda f, x, w, g: torch.autograd.functional.jacobian(f, (x, w), vectorize=True),
    "negated": lambda f, x, w, g: torch.autograd.grad(f(x, w), (x, w), torch._neg_view(g)),
    "zeros": lambda f, x, w, g: torch.autograd.grad(f(x, w), (x, w), torch._efficientzerotensor(g.shape, dtype=g.dtype, device=g.device)),
    "mode": under_a_mode,
    "autocast": under_autocast,
    "wrapper": of_a_wrapper,
    "kept negated": kept(torch._neg_view),
    "sparse": lambda f, x, w, g: torch.autograd.grad(f(x, w), (x, w), g.to_sparse()),
    "kept sparse": kept(lambda t: t.to_sparse()),
    "kept elsewhere": kept(lambda t: t.to("meta")),
}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", ARRIVES)
def test_gradients_of_what_is_not_plain_are_left_to_torch(native, case, dtype):
    """A launch sees addresses: what arrives at the backward has to be asked there, whatever the forward's arguments were."""
    torch.manual_seed(2)
    x, w, g = (torch.randn(shape).to(dtype) for shape in ((6, 16), (24, 16), (6, 24)))
    results = []
    for f in (native[0], through_torch):
        native[1].clear()
        results.append(ARRIVES[case](f, x.clone().requires_grad_(), w.clone().requires_grad_(), g))
        assert not {(0, 1), (1, 1)} & set(native[1]), native[1]
    for a, b in zip(*results):
        assert a is not None and a.shape == b.shape and a.device == b.device
        if case != "kept elsewhere":
            torch.testing.assert_close(a, b, rtol=4 * torch.finfo(dtype).eps, atol=32 * torch.finfo(dtype).eps)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_inputs_without_sizes_and_negated_weights_are_left_to_the_general_route(native, dtype):
    """A nested tensor has rows of its own for every sequence, which torch's linear takes and a launch does not."""
    x, w = torch.randn(6, 16).to(dtype), torch.randn(24, 16).to(dtype)
    nested = torch.nested.nested_tensor([torch.randn(2, 16), torch.randn(3, 16)], dtype=dtype)
    native[1].clear()
    for args in ((nested, w), (x, torch._neg_view(w)), (x, torch._efficientzerotensor(w.shape, dtype=dtype, device="cpu")), (x.to_sparse(), w), (torch._neg_view(x), w)):
        assert native[0](*args) is None
    assert native[1] == []


def test_recorded_products_take_tickets_of_their_own(native):
    """A stream under capture: nothing kept is used, the sizes are exactly what the call asks for, and the tickets are zeros."""
    f, _ = native
    stub = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p)(lambda stream: recording)
    f.host.bind_capturing(ctypes.cast(stub, ctypes.c_void_p).value)
    try:
        for recording in (0, 1, 0):
            f.workspaces.clear()
            f(torch.randn(6, 16).half().requires_grad_(), torch.randn(24, 16).half().requires_grad_()).backward(torch.ones(6, 24).half())
            assert len(f.workspaces) == 3 and all(zeros == bytes(16) and (size == 16) == recording for zeros, size in f.workspaces)
    finally:
        f.host.bind_capturing(0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_a_saved_weight_of_another_shape_raises(native, dtype):
    x, w = torch.randn(6, 16).to(dtype).requires_grad_(), torch.randn(24, 16).to(dtype)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t[:2].clone()):
        y = native[0](x, w)
    native[1].clear()
    with pytest.raises(RuntimeError):
        y.backward(torch.ones_like(y))
    assert native[1] == []


def test_replaced_functions_are_called(monkeypatch):
    """What the native call stands for may have been replaced: torch's linear, the class's fake quantisation, an instance's."""
    from types import SimpleNamespace

    import quant_cuda
    lin = cl.QuantLinear(16, 24, w_bits=4, group_size=8, cherryq=True, cherry_fraction=1 / 2).train()
    lin.register_cherry_indices(torch.arange(8))
    on_gpu, taken = SimpleNamespace(is_cuda=True), object()
    monkeypatch.setattr(quant_cuda, "train_linear", lambda *_: taken)
    assert lin._native_linear(None, on_gpu) is taken
    for where, name in ((vars(torch.nn.functional), "linear"), (cl.QuantLinear, "_adjust_weight"), (cl.QuantLinear, "_fused_fake_quant"),
                        (vars(lin), "_adjust_weight"), (vars(lin), "_fused_fake_quant")):
        with monkeypatch.context() as patch:
            (patch.setitem if isinstance(where, dict) else patch.setattr)(where, name, lambda *a, **b: None)
            assert lin._native_linear(None, on_gpu) is None, name
        assert lin._native_linear(None, on_gpu) is taken


def test_sizes_the_kernel_is_not_for():
    import quant_cuda
    for by_k in ((False, False), (False, True), (True, True)):
        assert not quant_cuda.gemm_preferred(*by_k, 0, 256, 256) and not quant_cuda.gemm_preferred(*by_k, 4096, 4100, 4096)
    assert not quant_cuda.gemm_preferred(False, False, 2048, 4096, 4100) and quant_cuda.gemm_preferred(False, False, 2047, 11008, 4096)
    assert not quant_cuda.gemm_preferred(True, True, 4096, 1 << 20, 2048)  # past 2 GiB


@pytest.mark.parametrize("m,n,k", [(2048, 11008, 4096), (4096, 11008, 2048), (11008, 4096, 2048), (8, 8, 8)])
def test_the_form_that_was_not_compared_is_not_preferred(m, n, k):
    import quant_cuda
    assert not quant_cuda.gemm_preferred(True, False, m, n, k)
    for by_k in ((False, False), (False, True), (True, True)):
        assert quant_cuda.gemm_preferred(*by_k, m, n, k) == (k > 8)


def test_limits_of_the_sizes():
    """Offsets are 32 bits: rows of an operand by_k that 63 rows of which do not fit them are refused (in front of anything that reads the
    pointers); sizes that no form takes have no plan, so nothing is computed from numbers of tiles that do not fit 32 bits."""
    import quant_cuda
    lib, fake, unsupported = quant_cuda._lib, 4096, -7
    if torch.cuda.is_available():
        pytest.skip("calls the entry point with addresses that are none: without a GPU only")

    def refused(a_by_k, b_by_k, m, n, k):
        return lib.cherryq_gemm_16(0, a_by_k, b_by_k, fake, fake, fake, m, n, k, None, 0, None, 0, None) == unsupported

    wide = 34087040
    for k in (8, 16, 24):
        assert 2 * wide * k < 0x7FFF0000 and 63 * 2 * wide + 512 >= 1 << 32 > 63 * 2 * (wide - 8) + 512
        assert refused(True, True, wide, 8, k) and refused(True, False, wide, 8, k) and refused(True, True, 8, wide, k) and refused(False, True, 8, wide, k)
        assert not quant_cuda.gemm_preferred(True, True, wide, 8, k)
    for m, n, k in ((2 ** 31 - 1, 2 ** 31 - 8, 8), (2 ** 31 - 1, 8, 8), (1 << 20, 1 << 20, 8), (1 << 21, 1 << 15, 1 << 11), (0, 8, 8), (8, 8, -8)):
        assert lib.cherryq_gemm_workspace_bytes(m, n, k) == lib.cherryq_gemm_scratch_bytes(m, n, k) == 0


def test_kernels_keep_their_distances(tmp_path):
    """The products are written out as inline assembly, around which the compiler keeps no distances (tests/test_mfma_distances.py)."""
    import os
    import re
    import shutil
    import subprocess

    from test_mfma_distances import LIB, OBJDUMP, too_close
    if not os.path.exists(OBJDUMP):
        pytest.skip("needs ROCm's llvm-objdump")
    lib = shutil.copy(LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    found = 0
    for path in tmp_path.iterdir():
        if not path.name.endswith("gfx950") or b"gemm_kernel" not in path.read_bytes():
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", path], check=True, capture_output=True, text=True).stdout
        for symbol, body in re.findall(r"^<(\S*gemm_kernel\S*)>:\n(.*?)(?=^<|\Z)", text, re.S | re.M):
            code = [line.split("//")[0].split(None, 1) for line in body.splitlines() if line.strip() and not line.rstrip().endswith(":")]
            code = [(x[0], [o.strip() for o in x[1].split(",")] if len(x) > 1 else []) for x in code if x]
            assert sum(op.startswith("v_mfma") for op, _ in code) == 64 and not too_close(code), (symbol, too_close(code)[:4])
            found += 1
    assert found == 8


# ---- the kernel --------------------------------------------------------------------------------------
def operands(m, n, k, a_by_k, b_by_k, dtype, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn((k, m) if a_by_k else (m, k), device="cuda", generator=gen).to(dtype)
    b = (torch.randn((n, k) if not b_by_k else (k, n), device="cuda", generator=gen) * 0.02).to(dtype)
    return a, b


def reference(a, b, a_by_k, b_by_k):
    a, b = (t.float().cpu().double() for t in (a, b))
    return (a.t() if a_by_k else a) @ (b if b_by_k else b.t())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("a_by_k,b_by_k", [(False, False), (False, True), (True, True), (True, False)])
# one tile and its edges, a step and its remainders, one step; 2, 4 and 8 workgroups a tile; more rows of tiles than 8; a whole round
# of 256 tiles, with a rest behind it that is split and one that is not
@pytest.mark.parametrize("m,n,k", [(256, 256, 64), (8, 8, 8), (264, 520, 136), (128, 96, 1000), (1000, 3000, 1504), (72, 4104, 4000),
                                   (248, 264, 8192), (2312, 264, 72), (4096, 4352, 1032),
                                   (4096, 4352, 2056)])
def test_gemm_against_64_bits(m, n, k, a_by_k, b_by_k, dtype):
    import quant_cuda
    print("gemm", m, n, k, a_by_k, b_by_k, dtype, flush=True)
    a, b = operands(m, n, k, a_by_k, b_by_k, dtype)
    want = reference(a, b, a_by_k, b_by_k)
    first = quant_cuda.gemm(a, b, a_by_k, b_by_k)
    err = ((first.cpu().double() - want).norm() / want.norm()).item()
    assert err < LIMIT[dtype], err
    for _ in range(3):  # the order of arrival does not show, and the tickets are zero again
        assert torch.equal(quant_cuda.gemm(a, b, a_by_k, b_by_k).view(torch.int16), first.view(torch.int16))


@pytest.mark.gpu
def test_rows_that_are_no_multiple_and_values_past_the_edge():
    """Infinities and NaN of one row and one column stay there; odd numbers of rows in either place."""
    import quant_cuda
    for m, k, a_by_k in ((2047, 264, False), (256, 333, True)):
        a, b = operands(m, 512, k, a_by_k, a_by_k, torch.float16)
        want = quant_cuda.gemm(a, b, a_by_k, a_by_k)
        (a.t() if a_by_k else a)[m - 1, 0], (b.t() if a_by_k else b)[511, 1] = float("inf"), float("nan")
        got = quant_cuda.gemm(a, b, a_by_k, a_by_k)
        assert torch.equal(got[:-1, :-1], want[:-1, :-1]) and not got[-1].isfinite().any() and got[:, -1].isnan().all()


@pytest.mark.gpu
def test_gemm_in_a_graph_and_on_two_streams():
    import quant_cuda
    a, b = operands(2048, 4096, 8192, False, True, torch.bfloat16)
    assert quant_cuda._lib.cherryq_gemm_scratch_bytes(2048, 4096, 8192) > 0
    want, out = quant_cuda.gemm(a, b, False, True), torch.empty(2048, 4096, device="cuda", dtype=torch.bfloat16)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out.copy_(quant_cuda.gemm(a, b, False, True))
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert torch.equal(quant_cuda.gemm(a, b, False, True), want) and torch.equal(out, want)
    streams, results = [torch.cuda.Stream() for _ in range(2)], []
    torch.cuda.synchronize()
    for i in range(6):
        with torch.cuda.stream(streams[i % 2]):
            results.append(quant_cuda.gemm(a, b, False, True))
    torch.cuda.synchronize()
    assert all(torch.equal(r, want) for r in results)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,k,n", [((3, 683), 4096, 4104), ((5, 7), 264, 72)])  # the kernel's products, and torch's
def test_training_pass_equals_the_general_route(dtype, rows, k, n):
    import quant_cuda
    with torch.device("cuda"):
        lin = cl.QuantLinear(k, n, bias=True, w_bits=4, group_size=128, cherryq=True, cherry_fraction=1 / 16).to(dtype).train()
    lin.register_cherry_indices(torch.arange(lin.num_cherries) * 7)
    x = torch.randn(*rows, k, device="cuda").to(dtype).requires_grad_()
    g = torch.randn(*rows, n, device="cuda").to(dtype)
    assert quant_cuda.gemm_preferred(True, True, n, k, rows[0] * rows[1]) == (k == 4096)
    results = []
    for native in (True, False):
        if not native:
            lin._native_linear = lambda *_: None
        x.grad = lin.weight.grad = lin.bias.grad = None
        y = lin(x)
        assert ("TrainLinear" in type(y.grad_fn.next_functions[0][0]).__name__ + y.grad_fn.next_functions[0][0].name()) == native
        y.backward(g)
        results.append([y.detach(), x.grad, lin.weight.grad, lin.bias.grad])
    for a, b in zip(*results):
        assert a.shape == b.shape and ((a.double() - b.double()).norm() / b.double().norm()).item() < 2 * LIMIT.get(dtype, 2.0 ** -18)


@pytest.mark.gpu
def test_training_passes_in_two_graphs():
    """Forward and backward captured twice on one stream, replayed the other way round, with eager passes between and what is kept for
    that stream full of other calls' counts: a graph's tickets are its own."""
    import quant_cuda
    rows, k, n = 2048, 3584, 10752
    print("training passes in two graphs", rows, k, n, flush=True)
    for form in ((False, False, rows, n, k), (False, True, rows, k, n), (True, True, n, k, rows)):
        assert quant_cuda.gemm_preferred(*form) and quant_cuda._lib.cherryq_gemm_workspace_bytes(*form[2:]) > 0
    with torch.device("cuda"):
        lin = cl.QuantLinear(k, n, bias=False, w_bits=4, group_size=128, cherryq=True, cherry_fraction=1 / 16).bfloat16().train()
    lin.register_cherry_indices(torch.arange(lin.num_cherries) * 7)
    inputs = [(torch.randn(rows, k, device="cuda").bfloat16().requires_grad_(), torch.randn(rows, n, device="cuda").bfloat16()) for _ in range(2)]

    def step(x, g):
        y = lin(x)
        return [y.detach(), *torch.autograd.grad(y, (x, lin.weight), g)]

    want, stream = [step(*i) for i in inputs], torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step(*inputs[0])
    torch.cuda.synchronize()
    graphs, outs = [torch.cuda.CUDAGraph() for _ in inputs], []
    for graph, i in zip(graphs, inputs):
        with torch.cuda.graph(graph, stream=stream):
            outs.append(step(*i))
    kept = quant_cuda._host.workspace(0, stream.cuda_stream, 8)
    torch.cuda.synchronize()
    kept.fill_(0x7f)
    for which in (1, 0, 0, 1, 0):
        for t in outs[which]:
            t.zero_()
        graphs[which].replay()
        eager = step(*inputs[which])
        torch.cuda.synchronize()
        for got, again, w in zip(outs[which], eager, want[which]):
            assert torch.equal(got, w) and torch.equal(again, w)
    assert (kept == 0x7f).all()
    kept.zero_()
    torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_a_wait_for_counts_that_never_come_ends(dtype):
    """A workspace that is not zero, against the interface: the last workgroup of each split tile gives its wait up (a quarter of a second
    or so) and its tile is NaN; tiles that are not split are as ever."""
    import quant_cuda
    m, n, k = 4096, 4352, 2056
    lib, lead = quant_cuda._lib, 256
    tiles, nbytes = lib.cherryq_gemm_workspace_bytes(m, n, k) // 8, lib.cherryq_gemm_scratch_bytes(m, n, k)
    print("a wait that ends", m, n, k, tiles, flush=True)
    assert 0 < tiles < m // lead * (n // lead)
    a, b = operands(m, n, k, False, False, dtype)
    want, out = quant_cuda.gemm(a, b), torch.empty(m, n, device="cuda", dtype=dtype)
    counts, scratch = torch.zeros(2 * tiles, dtype=torch.int32, device="cuda"), torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    for planted in (1 << 30, 0):
        counts[1::2] = planted
        assert lib.cherryq_gemm_16(dtype == torch.bfloat16, 0, 0, a.data_ptr(), b.data_ptr(), out.data_ptr(), m, n, k, counts.data_ptr(),
                                   4 * counts.numel(), scratch.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        nan = out.isnan().view(m // lead, lead, n // lead, lead).transpose(1, 2).flatten(2)
        assert torch.equal(nan.any(-1), nan.all(-1)) and int(nan.all(-1).sum()) == (tiles if planted else 0)
        assert torch.equal(out[~out.isnan()], want[~out.isnan()])
        counts.zero_()
