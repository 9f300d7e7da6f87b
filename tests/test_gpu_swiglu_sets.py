"""The SwiGLU GEMV with two row sets per workgroup, of four waves (rows of 8193
to 16384 weights) where its second set runs out of tiles: one row, an odd number
of tiles, one tile more than a round; and of two waves (rows of 4097 to 8192)
on both sides of the line between its two prologues; written and accumulated.  h = silu(gate) up is formed with hardware exp2 and
reciprocal (about 1 ulp each) and y in fp32, so an output is within
(cols + 16) 2^-24 sum |w h| of the exact sum, and the add rounds once more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14


@pytest.mark.parametrize("dtype", [Q4_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("rows,cols", [(1, 8704), (3, 16384), (513, 9216), (1027, 11264),
                                       (3073, 8704), (4099, 14336), (1, 4608), (2048, 8192),
                                       (2049, 4608), (2051, 7680), (4099, 8192)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_swiglu_two_sets(pkg, orc, dtype, rows, cols, accumulate):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    pkg.init()
    raw = pkg.synth_quantized(dtype, rows ^ cols, 0.02, rows, cols)
    w = torch.from_numpy(orc.dequantize(dtype, raw, rows * cols)).cuda().reshape(rows, cols).double()
    gen = torch.Generator(device="cuda").manual_seed(rows)
    g = 3 * torch.randn(cols, generator=gen, device="cuda")
    u = torch.randn(cols, generator=gen, device="cuda")
    y = torch.full((rows + 1,), 2.0, dtype=torch.float32, device="cuda")
    d_w = torch.from_numpy(raw).cuda()
    print("[gpu case] swiglu sets", dtype, rows, cols, accumulate, flush=True)
    pkg.qgemv_swiglu(dtype, d_w.data_ptr(), raw.size, g.data_ptr(), u.data_ptr(), y.data_ptr(),
                     rows, cols, accumulate, torch.cuda.current_stream().cuda_stream)
    gd = g.double()
    h = gd / (1 + (-gd).exp()) * u.double()
    want = w @ h + (2.0 if accumulate else 0.0)
    bound = (cols + 16) * 2.0 ** -24 * (w.abs() @ h.abs()) + 2.0 ** -22
    assert y[rows] == 2.0
    err = (y[:rows].double() - want).abs()
    assert (err <= bound).all(), float((err / bound).max())
