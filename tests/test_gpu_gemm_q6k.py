"""The fused Q6_K prefill GEMM (more than 64 tokens, rows of whole block pairs)
at the edges of its tiles and its decompositions: one row, ragged rows and
tokens, one pair of blocks per row, K pieces of 4 steps, half tiles, full
rounds.  Every output lies within the fp32 summation bound of the bf16
weights' exact product (bf16 x bf16 products are exact in fp32, so K terms
summed in any order are off by at most K 2^-24 sum |w x|), and so does the
dequantize-once route on the same call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q6_K, BF16 = 14, 30


@pytest.mark.parametrize("m,rows,cols", [
    (65, 1, 512), (65, 257, 1024), (128, 33, 1536), (129, 256, 512), (256, 255, 2560),
    (257, 512, 4096), (777, 300, 14336), (300, 33000, 512), (65, 12000, 1024)])
def test_gemm_q6k_fused_edges(pkg, orc, monkeypatch, m, rows, cols):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    pkg.init()
    rng = np.random.default_rng(m * 7 + rows)
    nb = rows * cols // 256
    raw = rng.integers(0, 256, (nb, 210), dtype=np.uint8)  # every code and scale occurs
    raw[:, 208:] = rng.uniform(1e-4, 2e-3, nb).astype(np.float16).view(np.uint8).reshape(nb, 2)
    raw = raw.reshape(-1)
    w = torch.from_numpy(orc.dequantize(Q6_K, raw, rows * cols)).cuda().reshape(rows, cols)
    w = w.bfloat16().double()
    gen = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, cols, generator=gen, device="cuda").bfloat16()
    want = x.double() @ w.t()
    bound = cols * 2.0 ** -24 * (x.double().abs() @ w.abs().t())
    d_w = torch.from_numpy(raw).cuda()
    s = torch.cuda.current_stream().cuda_stream
    for route in ("fused", "dq"):
        monkeypatch.setenv("SWAMP_GEMM_ROUTE", route)
        print("[gpu case] gemm q6k", route, m, rows, cols, flush=True)
        y = torch.full((m + 1, rows), 7.0, dtype=torch.float32, device="cuda")
        pkg.qgemm(Q6_K, d_w.data_ptr(), raw.size, x.data_ptr(), BF16, y.data_ptr(), m, rows, cols,
                  s)
        assert (y[m] == 7.0).all()
        err = (y[:m].double() - want).abs()
        assert (err <= bound).all(), (route, float((err / bound).max()))
