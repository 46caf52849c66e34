"""The prompt-sized product at the edges of its tiles, K shares and cherry chunks, against the dequantised weight in 64 bits."""
import pytest
import torch

from prompt_cases import ROUND_CASES, SHAPE_CASES, SPLIT_ROUND_CASES

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


@pytest.mark.parametrize("rows,k,n,c", ROUND_CASES)
@pytest.mark.parametrize("bits,group", [(4, 128), (3, 96)])
def test_more_tiles_than_compute_units(qc, bits, group, rows, k, n, c):
    print("[case] prompt rounds", bits, k, n, c, group, rows, flush=True)
    against_64_bits(qc, bits, k, n, c, group, rows)


@pytest.mark.parametrize("rows,k,n,c", SPLIT_ROUND_CASES)
@pytest.mark.parametrize("bits,group", [(4, 128), (3, 96)])
def test_more_pieces_of_split_tiles_than_compute_units(qc, bits, group, rows, k, n, c):
    print("[case] prompt split rounds", bits, k, n, c, group, rows, flush=True)
    against_64_bits(qc, bits, k, n, c, group, rows)


# pieces of four columns, of eight and of 96 columns, 16 rows, shared K
SCALE_CASES = [(66, 912, 11320, 112), (306, 320, 8456, 40), (423, 344, 4176, 0), (5, 264, 656, 8), (20, 272, 104, 8), (36, 264, 8304, 8)]


@pytest.mark.parametrize("rows,k,n,c", SCALE_CASES)
@pytest.mark.parametrize("bits,group", [(4, 128), (4, 160), (3, 128), (3, 96)])
def test_weights_are_the_dense_ones_at_any_scale(qc, bits, group, rows, k, n, c):
    """Rows that are ones of the identity: the product is the dense weight's value, whose one rounding from code times scale it has, bit for bit.
    Half of the scales lie below 2^-12, where a half of them need not have an fp16 value."""
    print("[case] prompt scales", bits, k, n, c, group, rows, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    kn, shape = k - c, (-(-(k - c) // group), n)
    small, any_ = (torch.randint(1, end, shape, device="cuda", generator=gen, dtype=torch.int16) for end in (0x0c00, 0x6c00))
    scales = torch.where(torch.rand(shape, device="cuda", generator=gen) < 0.5, small, any_).view(torch.float16)
    q = torch.randint(0, 256, (kn // 8 * bits, n), device="cuda", generator=gen, dtype=torch.uint8)
    cw = torch.randn((c, n), device="cuda", generator=gen).half()
    idx = torch.randperm(k, device="cuda", generator=gen)[:c].sort().values.to(torch.int16)
    at = torch.randint(0, k, (rows,), device="cuda", generator=gen)
    x = torch.nn.functional.one_hot(at, k).half()
    out = torch.zeros((rows, n), dtype=torch.float16, device="cuda")
    qc.matmul_cherryq(bits, x, q, cw, idx, scales, out, group)
    assert torch.equal(out, qc.unpack_cherryq(bits, q, cw, idx, scales, k, group).t()[at])


@pytest.mark.parametrize("bits,group", [(4, 128), (4, 160), (3, 128), (3, 96)])
@pytest.mark.parametrize("rows", [24, 100, 300])
def test_an_infinite_scale_is_no_nan(qc, bits, group, rows):
    print("[case] prompt infinite scale", bits, group, rows, flush=True)
    k, n = 1280, 1032
    q = torch.zeros((k // 8 * bits, n), device="cuda", dtype=torch.uint8)  # the lowest code: weights of -c_b s
    scales = torch.ones((-(-k // group), n), device="cuda", dtype=torch.float16)
    scales[1, 3::5] = float("inf")
    cw, idx = torch.zeros((0, n), dtype=torch.float16, device="cuda"), torch.zeros(0, dtype=torch.int16, device="cuda")
    out = torch.zeros((rows, n), dtype=torch.float16, device="cuda")
    qc.matmul_cherryq(bits, torch.ones((rows, k), dtype=torch.float16, device="cuda"), q, cw, idx, scales, out, group)
    want = torch.full((rows, n), -k * (2 ** bits - 1) / 2, device="cuda")
    want[:, 3::5] = float("-inf")
    assert torch.equal(out.float(), want.half().float())
