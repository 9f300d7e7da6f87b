"""The fp32 dequantizer at the edges of its lane-contiguous kernel: a lane
makes 4 weights per step, a wave 2 steps of 256, a workgroup 2048.  Counts
around those multiples, counts that end inside a lane's 4, and an output that
is not 16-byte aligned (element stores) all give the oracle's bits; what lies
past the output is left alone.  Uniformly random block bytes, so every scale
code occurs, NaN and infinities among them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14
BLOCK = {Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}


@pytest.mark.parametrize("dtype", [Q4_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("offset", [0, 1])
def test_dequant_edges(pkg, orc, dtype, offset):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    pkg.init()
    bs, ts = BLOCK[dtype]
    blocks = (5 * 2048 + 512) // bs
    raw = np.random.default_rng(dtype).integers(0, 256, blocks * ts, dtype=np.uint8)
    d_raw = torch.from_numpy(raw).cuda()
    ref = orc.dequantize(dtype, raw, blocks * bs)
    for n in [1, 3, 4, 5, 31, 255, 256, 257, 511, 513, 2047, 2048, 2049, 2051, 4097, 10239, 10242]:
        print("[gpu case] dequant edges", dtype, offset, n, flush=True)
        d_y = torch.full((n + offset + 8,), 7.0, dtype=torch.float32, device="cuda")
        pkg.qdequant(dtype, d_raw.data_ptr(), (n + bs - 1) // bs * ts,
                     d_y.data_ptr() + 4 * offset, n, torch.cuda.current_stream().cuda_stream)
        y = d_y.cpu().numpy()
        assert (y[:offset] == 7.0).all() and (y[offset + n:] == 7.0).all()
        got, want = y[offset:offset + n], ref[:n]
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan)
        assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


@pytest.mark.parametrize("dtype", [Q4_0, Q8_0, Q4_K, Q6_K])
def test_dequant_every_scale_bit_for_bit(pkg, orc, dtype):
    """A block for each of the 65536 halves as its scale: the lane-contiguous
    kernel (16-byte aligned output) and the element-store one give the same bits,
    NaN payloads included, and the oracle's values."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    pkg.init()
    bs, ts = BLOCK[dtype]
    raw = np.random.default_rng(dtype).integers(0, 256, (65536, ts), dtype=np.uint8)
    at = 208 if dtype == Q6_K else 0
    raw[:, at:at + 2] = np.arange(65536, dtype=np.uint16).view(np.uint8).reshape(-1, 2)
    raw, n = raw.reshape(-1), 65536 * bs
    d_raw = torch.from_numpy(raw).cuda()
    out = []
    for offset in (0, 1):
        print("[gpu case] dequant every scale", dtype, offset, flush=True)
        d_y = torch.empty(n + 4, dtype=torch.float32, device="cuda")
        pkg.qdequant(dtype, d_raw.data_ptr(), raw.size, d_y.data_ptr() + 4 * offset, n,
                     torch.cuda.current_stream().cuda_stream)
        out.append(d_y[offset:offset + n].cpu().numpy())
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
    ref = orc.dequantize(dtype, raw, n)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(out[0]), nan)
    assert np.array_equal(out[0][~nan].view(np.uint32), ref[~nan].view(np.uint32))

