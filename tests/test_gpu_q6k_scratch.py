"""Q6_K prefill under graph capture, where nothing is allocated: a reservation
of what a long prompt reports runs the shorter prompts of the same matrix, scratch
that holds the dequantized weights but not the fused kernel's partial sums runs
with the weights dequantized, and no scratch at all runs the fused kernel with
atomic sums -- only calls that the fused kernel does not take are refused.  Each
replay (with eager work and synchronisations in between) is checked: the same
bits as the eager call where the sums have an order, else the fp32 summation
bound of the bf16 weights' exact product (test_gpu_gemm_q6k.py)."""
import pytest

pytestmark = pytest.mark.gpu

Q6_K, BF16 = 14, 30


@pytest.fixture(scope="module")
def torch_dev(pkg):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    pkg.init()
    return torch


def fresh_stream(pkg, torch):
    """A stream of its own, never destroyed: torch hands out a fixed set of
    streams in turn, whose scratch earlier tests may have grown."""
    return torch.cuda.ExternalStream(pkg.gpu_lib().gpu_stream_create())


class Call:
    def __init__(self, pkg, torch, raw, d_w, m, rows, cols):
        gen = torch.Generator(device="cuda").manual_seed(m)
        self.pkg, self.torch, self.raw, self.d_w = pkg, torch, raw, d_w
        self.m, self.rows, self.cols = m, rows, cols
        self.x = torch.randn(m, cols, generator=gen, device="cuda").bfloat16()
        self.y = torch.empty((m, rows), dtype=torch.float32, device="cuda")

    def run(self, s):
        self.pkg.qgemm(Q6_K, self.d_w.data_ptr(), self.raw.size, self.x.data_ptr(), BF16,
                       self.y.data_ptr(), self.m, self.rows, self.cols, s)

    def eager(self):
        self.run(self.torch.cuda.current_stream().cuda_stream)
        self.torch.cuda.synchronize()
        return self.y.clone()


def replays(torch, stream, calls, check):
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        for c in calls:
            c.run(stream.cuda_stream)
    for rep in range(3):
        for c in calls:
            c.y.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for c in calls:
            check(c, rep)


def weights(pkg, torch, rows, cols):
    raw = pkg.synth_quantized(Q6_K, rows ^ cols, 0.02, rows, cols)
    return raw, torch.from_numpy(raw).cuda()


def report(pkg, m, rows, cols):
    return pkg.gpu_lib().swamp_qgemm_workspace(Q6_K, BF16, m, rows, cols)


def test_long_prompt_reservation_runs_short_prompts(pkg, torch_dev):
    """512 tokens fill the GPU without scratch; 64 and 1 need their weights in
    it."""
    torch = torch_dev
    rows, cols = 33024, 512
    raw, d_w = weights(pkg, torch, rows, cols)
    calls = [Call(pkg, torch, raw, d_w, m, rows, cols) for m in (512, 300, 64, 1)]
    stream = fresh_stream(pkg, torch)
    print("[gpu case] q6k reservation of a long prompt", flush=True)
    pkg.workspace_reserve(stream.cuda_stream, report(pkg, 512, rows, cols))
    want = {c.m: c.eager() for c in calls}
    replays(torch, stream, calls, lambda c, rep: _equal(torch, c, want[c.m], rep))


def test_report_of_shapes_that_are_refused(pkg, torch_dev):
    for m, rows, cols in [(0, 4, 512), (4, 0, 512), (4, 4, 0), (-1, 4, 512), (4, 4, 100)]:
        assert report(pkg, m, rows, cols) == 0, (m, rows, cols)


def _equal(torch, c, want, rep):
    assert torch.equal(c.y, want), (c.m, c.rows, c.cols, rep)


def test_scratch_of_the_weights_alone(pkg, torch_dev, monkeypatch):
    """2048 tokens x 1000 x 10240 splits into 8 pieces, more bytes than the
    dequantized weights and their own pieces take."""
    torch = torch_dev
    m, rows, cols = 2048, 1000, 10240
    raw, d_w = weights(pkg, torch, rows, cols)
    c = Call(pkg, torch, raw, d_w, m, rows, cols)
    need = report(pkg, m, rows, cols)
    monkeypatch.setenv("SWAMP_GEMM_ROUTE", "dq")
    once = report(pkg, m, rows, cols)
    want = c.eager()
    monkeypatch.delenv("SWAMP_GEMM_ROUTE")
    assert rows * cols * 2 <= once < need
    stream = fresh_stream(pkg, torch)
    print("[gpu case] q6k scratch of the weights alone", flush=True)
    pkg.workspace_reserve(stream.cuda_stream, once)
    replays(torch, stream, [c], lambda c, rep: _equal(torch, c, want, rep))


@pytest.mark.parametrize("m,rows,cols", [(300, 4096, 2560), (65, 4000, 8704), (777, 1027, 20480),
                                         (129, 257, 2048)])
def test_capture_without_scratch(pkg, orc, torch_dev, monkeypatch, m, rows, cols):
    """Split plans of the fused route, and (the last) a shape whose default is
    the dequantize-once route."""
    torch = torch_dev
    raw, d_w = weights(pkg, torch, rows, cols)
    c = Call(pkg, torch, raw, d_w, m, rows, cols)
    w = torch.from_numpy(orc.dequantize(Q6_K, raw, rows * cols)).cuda().reshape(rows, cols)
    w = w.bfloat16().double()
    want = c.x.double() @ w.t()
    bound = cols * 2.0 ** -24 * (c.x.double().abs() @ w.abs().t())
    print("[gpu case] q6k capture without scratch", m, rows, cols, flush=True)

    def check(c, rep):
        err = (c.y.double() - want).abs()
        assert (err <= bound).all(), (rep, float((err / bound).max()))

    assert report(pkg, m, rows, cols) > 0
    c.eager()
    check(c, "eager")
    replays(torch, fresh_stream(pkg, torch), [c], check)


@pytest.mark.parametrize("m,rows,cols", [(64, 512, 1024), (300, 512, 1280)])
def test_calls_that_need_their_weights_dequantized_are_refused(pkg, torch_dev, m, rows, cols):
    torch = torch_dev
    raw, d_w = weights(pkg, torch, rows, cols)
    c = Call(pkg, torch, raw, d_w, m, rows, cols)
    stream = fresh_stream(pkg, torch)
    rcs = []
    print("[gpu case] q6k refused without scratch", m, rows, cols, flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        c.y.zero_()
        with pytest.raises(pkg.GpuError) as e:
            c.run(stream.cuda_stream)
        rcs.append(e.value.code)
    assert rcs == [pkg.EWORKSPACE]
