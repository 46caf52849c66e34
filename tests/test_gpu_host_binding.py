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
