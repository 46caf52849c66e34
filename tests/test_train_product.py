"""The training layer's matrix products (csrc/cq_gemm.hip).

Bound of the kernel: fp32 sums of exact 16-bit products, rounded once.  The rounding is half an ulp of the result's type, at most
2^-11 (fp16) or 2^-8 (bf16) of an element, its 2-norm about 0.6 of that; a sum of K terms of random signs adds about sqrt(K) 2^-24 of
the result, 2^-17 at the largest K here.  So 2^-11 / 2^-8 of the 2-norm holds with room."""
import pytest
import torch

LIMIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def test_sizes_the_kernel_is_not_for():
    import quant_cuda
    for by_k in ((False, False), (False, True), (True, True)):
        assert not quant_cuda.gemm_preferred(*by_k, 0, 256, 256) and not quant_cuda.gemm_preferred(*by_k, 4096, 4100, 4096)
    assert not quant_cuda.gemm_preferred(False, False, 2048, 4096, 4100) and quant_cuda.gemm_preferred(False, False, 2047, 11008, 4096)
    assert not quant_cuda.gemm_preferred(True, True, 4096, 1 << 20, 2048)  # past 2 GiB


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
