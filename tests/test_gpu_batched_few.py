"""The register-x small-batch kernel (few tokens, short rows) at its edges: one
row, ragged 16-row tiles, one to eight tiles per workgroup and a last workgroup
with fewer, rows of less than a round of waves and of several passes, 1-16
tokens, y written and accumulated; and the shapes past its line, which take the
staged kernel.  Weights round to fp16 and x to fp16
(2^-11 each, products exact in fp32): an output is within 2^-10 (1 + 2^-11)
sum |w x| of the exact product, plus the fp32 sums' K 2^-24 sum |w x|, plus
fp16's smallest step (2^-25 absolute per weight and per x)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14
SHAPES = [(1, 256), (17, 512), (40, 2048), (1024, 4096), (4096, 3584), (4097, 4096), (8200, 2048),
          (12400, 2048), (20000, 2048), (32768, 2048), (30001, 4096), (33000, 2048)]


@pytest.mark.parametrize("dtype", [Q4_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_batched_few_tokens(pkg, orc, dtype, rows, cols):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    pkg.init()
    if dtype == Q6_K and cols % 512:
        cols *= 2
    raw = pkg.synth_quantized(dtype, rows ^ cols, 0.02, rows, cols)
    w = torch.from_numpy(orc.dequantize(dtype, raw, rows * cols)).cuda().reshape(rows, cols).double()
    d_w = torch.from_numpy(raw).cuda()
    s = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device="cuda").manual_seed(rows)
    for n in (1, 3, 8, 9, 16):
        for acc in (False, True):
            if acc and dtype == Q6_K:
                continue
            print("[gpu case] batched few", dtype, rows, cols, n, acc, flush=True)
            x = torch.randn(n, cols, generator=gen, device="cuda")
            y = torch.full((n + 1, rows), 3.0, dtype=torch.float32, device="cuda")
            pkg.qgemv_batched(dtype, d_w.data_ptr(), raw.size, x.data_ptr(), y.data_ptr(), n, rows,
                              cols, acc, s)
            assert (y[n] == 3.0).all()
            want = x.double() @ w.t() + (3.0 if acc else 0.0)
            mag = x.double().abs() @ w.abs().t()
            bound = mag * (2.0 ** -10 * (1 + 2.0 ** -11) + cols * 2.0 ** -24)
            bound += 2.0 ** -25 * (x.double().abs().sum(1)[:, None] + w.abs().sum(1)[None, :])
            bound += 2.0 ** -22  # the accumulating add
            err = (y[:n].double() - want).abs()
            assert (err <= bound).all(), (n, acc, float((err / bound).max()))
