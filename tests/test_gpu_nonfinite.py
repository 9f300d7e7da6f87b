"""Infinities and NaN in the kernels that form their operands anew: the fused
Q6_K GEMM, the register-x small batch and the SwiGLU product.  What is not finite
in the exact result (products and sums in 64 bits of the weights and activations
as the kernel rounds them) is not finite in y, and nothing else is: no padding
token, row or quad lets a NaN through, and finite outputs stay within the bounds of
their own tests.  Which of infinity and NaN a sum becomes depends on how it is
grouped (the GEMVs sum d (sum q x) - 8 d (sum x) per block, inf - inf for an
infinite x), so that is compared only where products are summed one by one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_0, Q8_0, Q4_K, Q6_K, BF16 = 2, 8, 12, 14, 30
BLOCK = {Q4_0: (32, 18, 0), Q8_0: (32, 34, 0), Q4_K: (256, 144, 0), Q6_K: (256, 210, 208)}
INF, NINF, NAN = 0x7C00, 0xFC00, 0x7E01  # binary16


@pytest.fixture(scope="module")
def torch_dev(pkg):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    pkg.init()
    return torch


def weights(pkg, orc, torch, dtype, rows, cols, scales):
    """Quantized rows with {(row, block): half bits} as block scales."""
    bs, ts, at = BLOCK[dtype]
    raw = pkg.synth_quantized(dtype, rows ^ cols, 0.02, rows, cols).reshape(rows, cols // bs, ts)
    for (row, block), bits in scales.items():
        raw[row, block, at:at + 2] = np.array([bits], np.uint16).view(np.uint8)
    raw = raw.reshape(-1)
    w = torch.from_numpy(orc.dequantize(dtype, raw, rows * cols)).cuda().reshape(rows, cols)
    return raw, torch.from_numpy(raw).cuda(), w


def check(torch, y, want, bound):
    bad = ~torch.isfinite(want)
    assert torch.equal(~torch.isfinite(y), bad)
    err = (y.double() - want).abs()[~bad]
    assert (err <= bound[~bad]).all()


@pytest.mark.parametrize("route", ["fused", "dq"])
@pytest.mark.parametrize("m,rows,cols", [(65, 257, 1024), (300, 512, 4096)])
def test_gemm_q6k(pkg, orc, torch_dev, monkeypatch, route, m, rows, cols):
    torch = torch_dev
    raw, d_w, w = weights(pkg, orc, torch, Q6_K, rows, cols,
                          {(0, 0): INF, (33, 3): NINF, (34, 2): NAN, (rows - 1, cols // 256 - 1): INF})
    w = w.bfloat16().double()
    x = torch.randn(m, cols, device="cuda", generator=torch.Generator("cuda").manual_seed(m))
    x[1, 5], x[m - 1, cols - 1], x[40, 300] = float("inf"), float("-inf"), float("nan")
    x = x.bfloat16()
    want = x.double() @ w.t()
    mag = torch.nan_to_num(x.double().abs(), posinf=0) @ torch.nan_to_num(w.abs(), posinf=0).t()
    monkeypatch.setenv("SWAMP_GEMM_ROUTE", route)
    print("[gpu case] nonfinite gemm q6k", route, m, rows, cols, flush=True)
    y = torch.empty((m, rows), dtype=torch.float32, device="cuda")
    pkg.qgemm(Q6_K, d_w.data_ptr(), raw.size, x.data_ptr(), BF16, y.data_ptr(), m, rows, cols,
              torch.cuda.current_stream().cuda_stream)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    inf = torch.isinf(want)
    assert inf.any() and torch.equal(y[inf].double(), want[inf])
    check(torch, y, want, cols * 2.0 ** -24 * mag)


@pytest.mark.parametrize("dtype", [Q4_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("n,rows,cols", [(5, 1000, 2048), (3, 4096, 1536), (5, 4113, 2048),
                                         (7, 12400, 2048)])
def test_batched_few(pkg, orc, torch_dev, dtype, n, rows, cols):
    torch = torch_dev
    bs = BLOCK[dtype][0]
    raw, d_w, w = weights(pkg, orc, torch, dtype, rows, cols,
                          {(0, 0): INF, (17, 3): NINF, (34, 2): NAN, (rows - 1, cols // bs - 1): INF})
    x = torch.randn(n, cols, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    x[1, 5], x[n - 1, cols - 1] = float("inf"), float("nan")
    want = x.double() @ w.double().t()
    fx, fw = (torch.nan_to_num(t.double().abs(), posinf=0) for t in (x, w))
    bound = (fx @ fw.t()) * (2.0 ** -10 * (1 + 2.0 ** -11) + cols * 2.0 ** -24)
    bound += 2.0 ** -25 * (fx.sum(1)[:, None] + fw.sum(1)[None, :])
    print("[gpu case] nonfinite batched few", dtype, n, rows, cols, flush=True)
    y = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    pkg.qgemv_batched(dtype, d_w.data_ptr(), raw.size, x.data_ptr(), y.data_ptr(), n, rows, cols,
                      False, torch.cuda.current_stream().cuda_stream)
    assert torch.isfinite(want).any()
    check(torch, y, want, bound)


@pytest.mark.parametrize("dtype", [Q4_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("rows,cols", [(300, 2048), (1000, 8192), (2100, 8192), (700, 9216),
                                       (520, 20480)])
@pytest.mark.parametrize("case", ["weights", "inf", "nan"])
def test_swiglu(pkg, orc, torch_dev, dtype, rows, cols, case):
    """gate = -inf is NaN in the reference's silu (-inf / inf), gate = -200 a
    zero, gate = 200 passes up through."""
    torch = torch_dev
    bs = BLOCK[dtype][0]
    last = (rows - 1, cols // bs - 1)
    raw, d_w, w = weights(pkg, orc, torch, dtype, rows, cols,
                          {(0, 0): INF, (17, 3): NAN, last: INF} if case == "weights" else {})
    gen = torch.Generator("cuda").manual_seed(rows)
    g, u = (torch.randn(cols, generator=gen, device="cuda") for _ in range(2))
    g[7], g[cols - 1] = 200.0, -200.0
    if case == "inf":
        g[cols - 3] = float("inf")
    if case == "nan":
        g[1] = float("-inf")
    y = torch.empty(rows, dtype=torch.float32, device="cuda")
    print("[gpu case] nonfinite swiglu", dtype, rows, cols, case, flush=True)
    pkg.qgemv_swiglu(dtype, d_w.data_ptr(), raw.size, g.data_ptr(), u.data_ptr(), y.data_ptr(),
                     rows, cols, False, torch.cuda.current_stream().cuda_stream)
    gd = g.double()
    h = gd / (1 + (-gd).exp()) * u.double()
    want = (w.double() * h).sum(1)
    assert torch.isfinite(want).any() == (case == "weights")
    fw, fh = (torch.nan_to_num(t.double().abs(), posinf=0) for t in (w, h))
    check(torch, y, want, (cols + 16) * 2.0 ** -24 * (fw @ fh) + 2.0 ** -22)
