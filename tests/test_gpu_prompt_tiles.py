"""The prompt-sized product at the edges of its tiles, K shares and cherry chunks, against the dequantised weight in 64 bits."""
import pytest
import torch

from prompt_cases import SHAPE_CASES

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qc():
    import quant_cuda
    return quant_cuda


def against_64_bits(qc, bits, k, n, c, group, rows):
    gen = torch.Generator(device="cuda").manual_seed(rows * 7 + k)
    kn = k - c
    q = torch.randint(0, 256, (kn // 8 * bits, n), device="cuda", generator=gen, dtype=torch.uint8)
    scales = (torch.rand((-(-kn // group), n), device="cuda", generator=gen) * 0.02 + 0.001).half()
    cw = (torch.randn((c, n), device="cuda", generator=gen) * 0.2).half()
    idx = torch.randperm(k, device="cuda", generator=gen)[:c].sort().values.to(torch.int16)
    x = torch.randn((rows, k), device="cuda", generator=gen).half()
    before = torch.randn((rows, n), device="cuda", generator=gen).half()
    w = qc.unpack_cherryq(bits, q, cw, idx, scales, k, group).double().t().contiguous()
    ref = x.double() @ w
    # products are exact in fp32, k of them are added up (in any order) and the sum is rounded to fp16
    slack = k * 2.0 ** -24 * (x.double().abs() @ w.abs()) + 2.0 ** -25
    if rows <= 16:  # the weights may go unrounded, then they differ from the dequantised ones by half a unit of theirs
        slack = slack + 2.0 ** -11 * (x.double().abs() @ w.abs())
    for accumulate in (False, True):
        out = before.clone()
        qc.matmul_cherryq(bits, x, q, cw, idx, scales, out, group, accumulate=accumulate)
        want = ref + before.double() if accumulate else ref
        assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -11 + slack * (1 + 2.0 ** -11)).all())


# rows around every tile height; columns off the tiles' 64 and 128; one unit of 128 positions, fewer than K shares, a ragged last
# one; no cherries, a partial step of 32, several chunks of steps; groups of whole units, and not
@pytest.mark.parametrize("rows", [5, 16, 17, 33, 48, 64, 81, 112, 113, 129, 193, 257, 520])
@pytest.mark.parametrize("bits,k,n,c,group", [(4, 128, 72, 0, 128), (3, 136, 64, 8, 32), (4, 520, 1032, 40, 160), (3, 1024, 264, 24, 96),
                                              (4, 1800, 2056, 520, 192), (3, 2560, 520, 296, 256), (4, 4096, 11008, 16, 128)])
def test_rows_around_the_tiles(qc, bits, k, n, c, group, rows):
    print("[case] prompt tiles", bits, k, n, c, group, rows, flush=True)
    against_64_bits(qc, bits, k, n, c, group, rows)


# groups of whole units of 128 positions are another instance than others, which may straddle units
@pytest.mark.parametrize("rows,k,n,c", SHAPE_CASES)
@pytest.mark.parametrize("bits,group", [(4, 128), (4, 160), (3, 128), (3, 96)])
def test_every_tile_shape(qc, bits, group, rows, k, n, c):
    print("[case] prompt shapes", bits, k, n, c, group, rows, flush=True)
    against_64_bits(qc, bits, k, n, c, group, rows)
