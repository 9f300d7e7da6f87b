"""The K-split decomposition of the fused prefill GEMM: whole tiles, halves and
quarters in 1 to 8 pieces (test_dispatch_rules.py checks that the shapes here
plan to them), tokens and rows that end inside a tile, a part and a piece of few
steps.  The same bf16 weights and x give every output within the
fp32 summation bound of the exact product (bf16 x bf16 products are exact in
fp32: K terms in any order are off by at most K 2^-24 sum |w x|), repeated calls
the same bits, and nothing past y is written."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_0, Q8_0, Q4_K, Q6_K, BF16 = 2, 8, 12, 14, 30


SHAPES = [
    (65, 130, 2560), (70, 4096, 1024), (100, 6144, 2048), (128, 257, 14336), (129, 1000, 4608),
    (200, 1500, 2048), (256, 4096, 1536), (300, 6144, 1024), (385, 700, 4096), (777, 2000, 5120),
    (250, 16100, 8192), (257, 14300, 5120), (777, 4096, 14336)]


@pytest.mark.parametrize("dtype", [Q4_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("m,rows,cols", SHAPES)
def test_gemm_split_parts(pkg, orc, monkeypatch, dtype, m, rows, cols):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    pkg.init()
    raw = pkg.synth_quantized(dtype, m ^ rows, 0.02, rows, cols)
    w = torch.from_numpy(orc.dequantize(dtype, raw, rows * cols)).cuda().reshape(rows, cols)
    w = w.bfloat16().double()
    gen = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, cols, generator=gen, device="cuda").bfloat16()
    want = x.double() @ w.t()
    bound = cols * 2.0 ** -24 * (x.double().abs() @ w.abs().t())
    d_w = torch.from_numpy(raw).cuda()
    s = torch.cuda.current_stream().cuda_stream
    first = None
    routes = ["fused", "fused"]
    if (dtype, m, rows, cols) == (Q6_K, 777, 4096, 14336):
        routes.append(None)  # the route such a call takes by default
    for route in routes:
        if route:
            monkeypatch.setenv("SWAMP_GEMM_ROUTE", route)
        else:
            monkeypatch.delenv("SWAMP_GEMM_ROUTE")
        print("[gpu case] gemm split", dtype, m, rows, cols, route, flush=True)
        y = torch.full((m + 1, rows), 7.0, dtype=torch.float32, device="cuda")
        pkg.qgemm(dtype, d_w.data_ptr(), raw.size, x.data_ptr(), BF16, y.data_ptr(), m, rows, cols,
                  s)
        assert (y[m] == 7.0).all()
        err = (y[:m].double() - want).abs()
        assert (err <= bound).all(), float((err / bound).max())
        first = y if first is None else first
        assert torch.equal(y, first)
