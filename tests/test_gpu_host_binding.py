"""The native host path of the Python binding (csrc/cq_host.cpp) against the general one: same results bit for bit,
and every call that is not what it takes reaches the general route (its result or its error)."""
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(bits, k, n, group=128, bias=False, seed=0):
    import quant_cuda
    from llama.qlinear import QuantLinear
    from llama.quantizer import FullSymQuantizer
    gen = torch.Generator(device="cuda").manual_seed(seed)
    with torch.device("cuda"):
        q = QuantLinear(bits, group, FullSymQuantizer, 1 / 256, k, n, bias=bias)
    idx = torch.randperm(k, device="cuda", generator=gen)[:q.num_cherries]
    w = (torch.randn(n, k, device="cuda", generator=gen) * 0.02).half()
    q.cherry_indices, q.cherry_weight, q.qweight, q.scales = quant_cuda.pack_cherryq(bits, w, idx, group)
    if bias:
        q.bias = torch.randn(n, device="cuda", generator=gen).half()
    return q


@pytest.mark.parametrize("bits,k,n,group,stream", [(4, 4096, 512, 128, True), (3, 2056, 264, 128, False), (3, 1024, 136, 64, False),
                                                   (4, 4096, 1024, 128, False)])
@pytest.mark.parametrize("rows", [1, 2, 5, 16, 17, 40])
def test_forward_equals_the_general_route(bits, k, n, group, stream, rows):
    print("[case] host forward", bits, k, n, group, stream, rows, flush=True)
    sys.stdout.flush()
    import quant_cuda
    q = _layer(bits, k, n, group, bias=rows % 2 == 1)
    if stream:
        assert q.prepack()
    for shape, dtype in (((rows, k), torch.float16), ((1, rows, k), torch.float32), ((rows, k), torch.bfloat16)):
        x = torch.randn(shape, device="cuda").to(dtype)
        native = quant_cuda._host.linear(q, x)
        assert native is not None and native.is_inference()
        want = q._forward(x)
        assert native.dtype == want.dtype == dtype and native.shape == want.shape
        assert torch.equal(native, want) and torch.equal(q(x), want)
    wide = torch.randn(rows, 2 * k, device="cuda").half()
    assert torch.equal(q(wide[:, ::2]), q._forward(wide[:, ::2]))
    if stream:
        assert q.prepack(release_reference=True)
        x = torch.randn(rows, k, device="cuda").half()
        assert torch.equal(q(x), q._forward(x))


def test_calls_that_are_not_taken():
    print("[case] host refusals", flush=True)
    import quant_cuda as qc
    from llama.qlinear import QuantLinear
    q = _layer(4, 1024, 256)
    x = torch.randn(3, 1024, device="cuda").half()
    out = torch.empty(3, 256, dtype=torch.float16, device="cuda")
    good = [4, x, q.qweight, q.cherry_weight, q.cherry_indices, q.scales, out, 128, False]
    assert qc._host.vecquant(*good) == 0
    bad = {1: [x.float(), x.cpu(), x[:, :512], x[:2], None], 2: [q.qweight[:-1], q.qweight.to(torch.int8)], 3: [q.cherry_weight.float()],
           4: [q.cherry_indices.int()], 5: [q.scales[:, :128]], 6: [out[:, :128], out.t()], 7: [64, 128.0], 0: [3]}
    for at, values in bad.items():
        for v in values:
            args = list(good)
            args[at] = v
            assert qc._host.vecquant(*args) is None, (at, v)
    assert qc._host.linear(q, x.cpu()) is None and qc._host.linear(q, x[:, :512]) is None and qc._host.linear(q, x[:0]) is None
    assert qc._host.linear(q, torch.randn(QuantLinear.prefill_rows, 1024, device="cuda").half()) is None
    assert q(x[:0]).shape == (0, 256)
    with pytest.raises(RuntimeError):
        q(x.cpu())
    with QuantLinear.dmode(layerwise_dequantize=False):
        assert qc._host.linear(q, x) is None
        q(x)
    assert qc._host.linear(q, x) is None
    with pytest.raises(RuntimeError):
        q(x)
    with pytest.raises(RuntimeError):
        qc.vecquant4matmul_cherryq(x, q.qweight.byte(), out, out, out, out, 128)


def test_replaced_buffers_and_workspace_growth():
    print("[case] host replaced buffers", flush=True)
    import quant_cuda as qc
    a, b = _layer(4, 1024, 256, seed=1), _layer(4, 1024, 256, seed=2)
    x = torch.randn(2, 1024, device="cuda").half()
    want = b(x)
    a.load_state_dict(b.state_dict())
    assert torch.equal(a(x), want)
    side = torch.cuda.Stream()
    small = qc._host.workspace(0, side.cuda_stream, 100)
    assert small.numel() == 1 << 18 and int(small.sum()) == 0
    assert qc._host.workspace(0, side.cuda_stream, 1 << 18).data_ptr() == small.data_ptr()
    grown = qc._host.workspace(0, side.cuda_stream, (1 << 18) + 1)
    assert grown.numel() == 1 << 19 and int(grown.sum()) == 0


def test_graphs_on_a_stream_without_a_workspace():
    """The first calls on a stream are recorded, in two graphs, and the second one is replayed first: no graph counts from what only
    the other one sets to zero, and nothing that a graph sets to zero is kept for calls outside."""
    print("[case] host graphs on a new stream", flush=True)
    import quant_cuda as qc
    q, stream = _layer(4, 11008, 512), torch.cuda.Stream()
    inputs = [torch.randn(rows, 11008, device="cuda").half() for rows in (1, 16)]
    a = torch.randn(256, 64, device="cuda").half()
    outs = [torch.empty(x.shape[0], 512, device="cuda", dtype=torch.float16) for x in inputs]
    want = []
    for x, out in zip(inputs, outs):
        qc.vecquant4matmul_cherryq(x, q.qweight, q.cherry_weight, q.cherry_indices, q.scales, out.zero_(), 128)
        want.append(out.clone())
    graphs, made = [torch.cuda.CUDAGraph() for _ in inputs], []
    for graph, x, out in zip(graphs, inputs, outs):
        with torch.cuda.graph(graph, stream=stream):
            qc.gemm(a, a)
            out.zero_()
            qc.vecquant4matmul_cherryq(x, q.qweight, q.cherry_weight, q.cherry_indices, q.scales, out, 128)
            made.append(qc._host.workspace(0, stream.cuda_stream, 8))
    kept = qc._host.workspace(0, stream.cuda_stream, 8)
    assert len({t.data_ptr() for t in (*made, kept)}) == 3
    for which in (1, 0, 0, 1):
        outs[which].fill_(7)
        graphs[which].replay()
        torch.cuda.synchronize()
        assert torch.equal(outs[which], want[which])
    assert not kept.any()


@pytest.mark.parametrize("stream", [False, True])
def test_every_form_of_a_bias_is_added(stream):
    print("[case] host bias forms", stream, flush=True)
    from llama.qlinear import QuantLinear

    class Own(QuantLinear):
        bias = property(lambda self: self.own, lambda self, value: None)

    x = torch.randn(3, 1024, device="cuda").half()
    b = torch.randn(256, device="cuda").half()
    plain = _layer(4, 1024, 256)
    want = None
    for form in ("buffer", "attribute", "parameter", "parameter over the buffer", "property"):
        q = _layer(4, 1024, 256, bias=form in ("buffer", "parameter over the buffer"))
        if form == "property":
            q.__class__, q.own = Own, b
        else:
            if form == "parameter over the buffer":
                del q.bias
            q.bias = torch.nn.Parameter(b.clone()) if form.startswith("parameter") else b.clone()
        if stream:
            assert q.prepack() and plain.prepack()
        want = plain(x) + b if want is None else want
        assert torch.equal(q(x), want) and torch.equal(q._forward(x), want), form


def test_function_transforms_raise_and_leave_the_binding_usable():
    print("[case] host under torch.func", flush=True)
    import quant_cuda as qc
    q, s = _layer(4, 1024, 256), _layer(4, 1024, 256)
    assert s.prepack()
    x, out = torch.randn(3, 1024, device="cuda").half(), torch.empty(3, 256, dtype=torch.float16, device="cuda")
    args = (q.qweight, q.cherry_weight, q.cherry_indices, q.scales, out, 128)
    entries = (q, s, lambda v: qc.vecquant4matmul_cherryq(v, *args), lambda v: qc.matmul_cherryq(4, v, *args),
               lambda v: qc.matvec_prepacked_cherryq(4, v, s._stream, out, 1024, q.num_cherries))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # a stream whose kept buffers are made inside the transform
        for f in entries:
            for under in (lambda: torch.func.grad(f)(x), lambda: torch.func.vmap(f)(x.expand(2, 3, 1024))):
                with pytest.raises(RuntimeError):
                    under()
        got = q(x)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, q(x))


def _shifted(t, nbytes):
    """The same values `nbytes` behind an address that is aligned."""
    flat = torch.empty(t.numel() + 16, dtype=t.dtype, device=t.device)[nbytes // t.element_size():][:t.numel()]
    return flat.view(t.shape).copy_(t)


@pytest.mark.parametrize("rows", [512, 600, 2303])
@pytest.mark.parametrize("bits,group,moved", [(4, 64, None), (4, 136, None), (3, 24, None), (3, 32, None), (4, 128, "qweight"), (3, 128, "scales"),
                                              (4, 128, "cherry_weight"), (3, 128, "x"), (4, 128, "wide x")])
def test_many_rows_of_layers_that_the_fused_kernel_refuses(rows, bits, group, moved):
    """From 512 rows there is the dense product: groups that are no multiple of 32 (4 bits: below 128), buffers off 16 bytes.  Weights are
    rounded to fp16 in either path; a result is rounded once (2^-11), the sum of a thousand products far less."""
    print("[case] many rows", bits, group, moved, rows, flush=True)
    from llama.qlinear import QuantLinear
    from llama.quantizer import FullSymQuantizer
    k, n = 1024, 264
    gen = torch.Generator(device="cuda").manual_seed(rows + group)
    q = QuantLinear(bits, group, FullSymQuantizer, 1 / 64, k, n, bias=False).cuda()
    q.qweight = torch.randint(0, 256, q.qweight.shape, dtype=torch.uint8, device="cuda", generator=gen)
    q.scales = (torch.rand(q.scales.shape, device="cuda", generator=gen) * 0.02 + 0.001).half()
    q.cherry_weight = torch.randn(q.cherry_weight.shape, device="cuda", generator=gen).half()
    q.cherry_indices = torch.randperm(k, device="cuda", generator=gen)[:q.num_cherries].sort().values.to(torch.int16)
    x = torch.randn(rows, k, device="cuda", generator=gen).half()
    want = x.double() @ q.unpack().double().t()
    if moved == "x":
        x = _shifted(x, 2)
    elif moved == "wide x":
        x = torch.cat([x, x], 1)[:, :k]
    elif moved is not None:
        t = getattr(q, moved)
        setattr(q, moved, _shifted(t, {"qweight": 4, "scales": 8, "cherry_weight": 2}[moved]))
    assert float((q(x).double() - want).norm() / want.norm()) <= 2.0 ** -11


def test_many_rows_transformed_and_captured():
    """Calls of 512 rows and more under vmap, and captured: a graph shares no kept buffer with the calls between its replays."""
    print("[case] many rows transformed", flush=True)
    import quant_cuda
    from llama.qlinear import QuantLinear
    q = _layer(4, 1024, 256)
    gen = torch.Generator(device="cuda").manual_seed(3)
    x, other = (torch.randn(600, 1024, device="cuda", generator=gen).half() for _ in range(2))
    dense = torch.matmul(other, q.unpack().t()).double()
    assert QuantLinear._dense_rows <= 600 < QuantLinear.prefill_rows
    both = torch.func.vmap(q)(torch.stack([x, other]))
    assert float((both[1].double() - dense).norm() / dense.norm()) <= 2.0 ** -10
    static, graph = x.clone(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = q(static)
        stream = torch.cuda.current_stream().cuda_stream
    # nothing was kept for the stream under capture: asked for now, its first buffer is the smallest there is
    assert quant_cuda._host.scratch(0, stream, 8).numel() == 8
    for inputs in (other, x, other):
        static.copy_(inputs)
        eager = q(inputs)
        graph.replay()
        torch.cuda.synchronize()
        assert float((out.double() - eager.double()).norm() / eager.double().norm()) <= 2.0 ** -10
