"""The dense weight (cherryq_unpack_f16) with every fp16 number as a scale (MI355X only).

A weight is RN16((u - c_b) * scale): 4 by 11 significant bits, so the oracle's product in fp32 is exact and
its rounding to fp16 the only one.  The kernel multiplies in fp16; subnormal scales and results, results at the
overflow threshold, zeros of either sign and infinities have to be the same bits, a NaN has to stay one.
"""
import numpy as np
import pytest
import torch

from oracle import cherryq_oracle as orc
from oracle import c_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [4, 3])
@pytest.mark.parametrize("frac", [1 / 32, 1 / 256])
def test_unpack_takes_every_scale(bits, frac):
    assert torch.cuda.is_available(), "this test needs the MI355X"
    import quant_cuda
    k, n, group = 512, 32768, 128
    print("[case] unpack every scale", bits, k, n, frac, flush=True)
    p = orc.synthetic_packed_fast(k, n, bits, group, seed=bits, cherry_fraction=frac)
    rows = p["scales"].shape[0]
    # every 16-bit pattern at least once in two rows of groups, and in another order in the rest
    pattern = np.arange(rows * n, dtype=np.uint32).reshape(rows, n)
    pattern[2:] = (pattern[2:] * 40503) & 0xFFFF
    p["scales"] = np.ascontiguousarray((pattern & 0xFFFF).astype(np.uint16)).view(np.float16)
    t = {name: torch.from_numpy(np.ascontiguousarray(p[name])).cuda()
         for name in ("cherry_indices", "cherry_weight", "qweight", "scales")}
    got = quant_cuda.unpack_cherryq(bits, t["qweight"], t["cherry_weight"], t["cherry_indices"], t["scales"], k, group)
    got = got.cpu().numpy()
    with np.errstate(all="ignore"):
        want = c_oracle.unpack(p, bits, group, k)
    nan = np.isnan(want)
    assert nan.any() and np.isinf(want).any()
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got.view(np.uint16)[~nan], want.view(np.uint16)[~nan])
