"""The launches between the linears of a whole-prompt pass, against the same operations in 64 bits."""
import sys
from pathlib import Path

import pytest
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "mixed-precision-cuda-kernel_amd"))

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dec():
    import cherryq_decoder
    return cherryq_decoder


def rel(a, b):
    return float((a.double().cpu() - b).norm() / b.norm())


def stream():
    return torch.cuda.current_stream().cuda_stream


# one key block with and without a remainder, both query tiles (16 queries below 512 tiles of 32, else 32), grouped heads
@pytest.mark.parametrize("tokens,nh,nkv", [(1, 2, 1), (16, 3, 3), (33, 4, 2), (130, 8, 1), (257, 32, 8), (255, 64, 64), (700, 24, 12)])
def test_prefill_attention(dec, tokens, nh, nkv):
    print("[case] prefill attention", tokens, nh, nkv, flush=True)
    lib, ml = dec._lib, tokens + 3
    gen = torch.Generator().manual_seed(tokens)
    q, k, v = (torch.randn(tokens, n * 128, generator=gen).half() for n in (nh, nkv, nkv))
    ang = torch.outer(torch.arange(tokens).double(), 10000.0 ** -(torch.arange(64).double() / 64))
    cos, sin = ang.cos().half(), ang.sin().half()

    def rope(x, n):  # every product and sum rounded to fp16
        x = x.view(tokens, n, 128).transpose(0, 1)
        c, s = torch.cat([cos, cos], -1), torch.cat([sin, sin], -1)
        return x * c + torch.cat([-x[..., 64:], x[..., :64]], -1) * s

    qr, kr, vr = rope(q, nh), rope(k, nkv), v.view(tokens, nkv, 128).transpose(0, 1)
    kd, vd = (t.double().repeat_interleave(nh // nkv, 0) for t in (kr, vr))
    s = qr.double() @ kd.transpose(1, 2) / 128 ** 0.5 + torch.full((tokens, tokens), float("-inf"), dtype=torch.float64).triu(1)
    want = (torch.softmax(s, -1) @ vd).transpose(0, 1).reshape(tokens, -1)

    kc, vc = (torch.zeros(nkv, ml, 128, dtype=torch.float16, device="cuda") for _ in range(2))
    out = torch.empty(tokens, nh * 128, dtype=torch.float16, device="cuda")
    scratch = torch.full((lib.cherryq_prefill_attention_bytes(tokens, nkv),), 255, dtype=torch.uint8, device="cuda")  # NaN
    d = [t.cuda() for t in (q, k, v, cos, sin)]
    args = [t.data_ptr() for t in (*d, kc, vc, out, scratch)]
    assert lib.cherryq_prefill_attention_f16(*args, scratch.numel() - 1, tokens, nh, nkv, 128, ml, stream()) == -4
    assert lib.cherryq_prefill_attention_f16(*args, scratch.numel(), tokens, nh, nkv, 64, ml, stream()) == -7
    assert lib.cherryq_prefill_attention_f16(*args, scratch.numel(), tokens, nh, nkv, 128, tokens - 1, stream()) == -2
    assert lib.cherryq_prefill_attention_f16(*args, scratch.numel(), tokens, nh, nkv, 128, ml, stream()) == 0
    torch.cuda.synchronize()
    assert torch.equal(kc[:, :tokens].cpu(), kr) and torch.equal(vc[:, :tokens].cpu(), vr)
    assert not kc[:, tokens:].any() and not vc[:, tokens:].any()
    # probabilities and results are rounded to fp16, 2^-11 each at most
    assert rel(out, want) < 2 * 2 ** -11


@pytest.mark.parametrize("rows,hidden", [(1, 8), (3, 2056), (17, 4096), (130, 5120), (5, 8192)])
@pytest.mark.parametrize("add", [False, True])
def test_prefill_norm(dec, rows, hidden, add):
    print("[case] prefill norm", rows, hidden, add, flush=True)
    gen = torch.Generator().manual_seed(rows)
    h, d = torch.randn(rows, hidden, generator=gen).half(), torch.randn(rows, hidden, generator=gen).half()
    w = (torch.rand(hidden, generator=gen) + 0.5).half()
    hd, dd, wd = h.cuda(), d.cuda(), w.cuda()
    y = torch.empty_like(hd)
    assert dec._lib.cherryq_prefill_norm_f16(hd.data_ptr(), dd.data_ptr() if add else None, wd.data_ptr(), y.data_ptr(), rows,
                                             hidden, 1e-6, stream()) == 0
    torch.cuda.synchronize()
    hs = h + d if add else h
    want = w.double() * (hs.double() * torch.rsqrt(hs.double().pow(2).mean(-1, keepdim=True) + 1e-6))
    assert torch.equal(hd.cpu(), hs)
    assert rel(y, want) < 2 * 2 ** -11  # two roundings
    assert dec._lib.cherryq_prefill_norm_f16(hd.data_ptr(), None, wd.data_ptr(), y.data_ptr(), rows, 8200, 1e-6, stream()) == -7


@pytest.mark.parametrize("n,shift", [(8, 0), (4096, 0), (4100, 0), (2048, 1)])
def test_silu_mul_widths(dec, n, shift):
    print("[case] silu_mul", n, shift, flush=True)
    g, u = (torch.randn(n + shift).half().cuda()[shift:] for _ in range(2))
    out = torch.zeros(n + shift + 8, dtype=torch.float16, device="cuda")
    o = out[shift:]
    assert dec._lib.cherryq_decode_silu_mul_f16(g.data_ptr(), u.data_ptr(), o.data_ptr(), n, stream()) == 0
    torch.cuda.synchronize()
    want = torch.nn.functional.silu(g.double()).cpu() * u.double().cpu()
    assert rel(o[:n], want) < 2 * 2 ** -11 and not o[n:].any()


# layers of different widths whose tiles share a launch: a remainder of columns, K splits, groups that are no whole unit
@pytest.mark.parametrize("bits,k,ns,rows,group", [(4, 1024, (1024, 256, 256), 17, 128), (4, 4096, (520, 8), 99, 128),
                                                  (3, 4096, (1000, 2056, 504), 40, 64), (4, 2048, (5504, 5504), 511, 256),
                                                  (3, 8192, (8192, 1024, 1024), 128, 128), (4, 1032, (264,), 33, 128)])
def test_matmul_group_matches_the_single_products(dec, bits, k, ns, rows, group):
    print("[case] matmul_group", bits, k, ns, rows, group, flush=True)
    cfg = dec.DecoderConfig(w_bits=bits, group_size=group, cherry_fraction=1 / 64)
    gen = torch.Generator(device="cuda").manual_seed(k + rows)
    mods = [dec.random_packed_linear(cfg, k, n, gen, torch.device("cuda")) for n in ns]
    x = torch.randn(rows, k, device="cuda", generator=gen).half()
    assert dec.matmul_group_supported(mods, rows)
    for _ in range(2):  # the second call finds the workspace as the first one left it
        got = dec.matmul_group(mods, x)
        for m, o in zip(mods, got):
            # the same operands summed in another order, then rounded: half a unit of fp16 each
            assert rel(o, m(x).double().cpu()) < 2 ** -11
            want = x.double().cpu() @ m.unpack().double().cpu().t()
            assert rel(o, want) < 2 ** -11
    mods[0].register_forward_hook(lambda *a: None)
    assert not dec.matmul_group_supported(mods, rows) and not dec.matmul_group_supported(mods[1:] or mods, 16)


# the channels' share decides how a unit's columns are found: staged ahead (up to 128 channels), staged behind the
# channels, channels too many for LDS, and rows whose address allows no wide loads
@pytest.mark.parametrize("k,fraction,shift", [(4096, 1 / 256, 0), (4104, 1 / 32, 0), (4096, 1 / 30, 0), (8192, 1 / 16, 0),
                                              (4096, 1 / 3, 0), (4096, 1 / 256, 2), (2048, 1 / 8, 2), (1032, 0.0, 0)])
@pytest.mark.parametrize("bits,rows", [(4, 17), (3, 99)])
def test_activations_gathered_around_the_channels(dec, bits, rows, k, fraction, shift):
    print("[case] gathered activations", bits, rows, k, fraction, shift, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(k)
    m = dec.random_packed_linear(dec.DecoderConfig(w_bits=bits, cherry_fraction=fraction), k, 264, gen, torch.device("cuda"))
    x = torch.randn(rows * k + shift, device="cuda", generator=gen).half()[shift:].view(rows, k)
    assert x.data_ptr() % 16 == 2 * shift
    got = m(x)
    # one rounding of the result to fp16; weights are the dense ones
    assert rel(got, x.double().cpu() @ m.unpack().double().cpu().t()) < 2 ** -11
