"""The rules that choose a kernel by size (csrc/dispatch.hpp), on the CPU."""
import importlib.util
import os
import types

import pytest

from dispatch_rules import CUS, REPO, SPLIT, Q4_0, Q4_K, Q6_K, Q8_0, Rules


@pytest.fixture(scope="session")
def rules(tmp_path_factory):
    return Rules(str(tmp_path_factory.mktemp("rules")))


@pytest.fixture(scope="session")
def bench():
    spec = importlib.util.spec_from_file_location("bench_mod", os.path.join(REPO, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_bench_route_labels_follow_the_rule(rules, bench):
    """bench.py repeats the route rule in Python to name the kernels behind its
    prefill lines: the same answer on both sides of every condition."""
    gpu = types.SimpleNamespace(cuda=types.SimpleNamespace(
        get_device_properties=lambda i: types.SimpleNamespace(multi_processor_count=CUS)))
    seen = set()
    for dt in (Q4_0, Q8_0, Q4_K, Q6_K):
        for m in (1, 64, 65, 128, 129, 256, 257, 512, 513, 777, 1000, 1023, 1024, 1025, 2048, 4096):
            for rows in (1, 256, 1000, 2048, 4096, 4097, 6144, 8192, 14336, 28672, 128256):
                for cols in (512, 768, 1024, 4096, 4352, 8192, 8704, 14336, 19968, 20480):
                    want = rules.dequantize_once(dt, m, rows, cols)
                    label = bench.gemm_route(gpu, dt == Q6_K, m, rows, cols, "bf16")
                    assert label.startswith("dequantize-once") == want, (dt, m, rows, cols, label)
                    seen.add((dt == Q6_K, want))
    assert len(seen) == 4


# (dtype, tokens, rows, weights per row, us staged, us in registers), measured on
# an MI355X over rotating weights
SMALL_BATCH = [
    (Q4_0, 1, 4096, 256, 5.15, 5.29), (Q4_0, 5, 4096, 4096, 7.99, 7.59),
    (Q4_0, 8, 4096, 4096, 8.12, 9.01), (Q4_0, 12, 4096, 2048, 7.13, 7.51),
    (Q4_0, 8, 14336, 2048, 9.64, 9.38), (Q4_0, 5, 14336, 4096, 15.72, 14.06),
    (Q4_0, 3, 5120, 8192, 12.30, 15.14), (Q4_0, 1, 16384, 4096, 13.70, 14.46),
    (Q4_0, 12, 28672, 2048, 15.15, 14.19), (Q4_0, 1, 5120, 28672, 24.97, 38.96),
    (Q4_0, 6, 4096, 2048, 6.76, 6.46), (Q4_0, 9, 2048, 2048, 6.97, 6.77),
    (Q4_0, 12, 14336, 2048, 10.28, 10.25), (Q8_0, 5, 4096, 4096, 9.86, 8.62),
    (Q8_0, 14, 4096, 2048, 8.35, 8.94), (Q8_0, 12, 4096, 2560, 8.77, 9.14),
    (Q8_0, 5, 14336, 4096, 22.37, 19.74), (Q8_0, 14, 14336, 4096, 24.24, 22.49),
    (Q8_0, 4, 5120, 8192, 17.38, 20.60), (Q8_0, 1, 5120, 28672, 38.38, 55.86),
    (Q8_0, 3, 5120, 10240, 20.48, 24.49), (Q8_0, 8, 4096, 2048, 8.16, 7.57),
    (Q8_0, 16, 2560, 2048, 8.16, 9.23), (Q4_K, 3, 4096, 4096, 7.70, 7.14),
    (Q4_K, 5, 4096, 4096, 7.91, 7.45), (Q4_K, 5, 1024, 4096, 7.88, 7.35),
    (Q4_K, 6, 4096, 4096, 7.97, 8.38), (Q4_K, 8, 4096, 4096, 8.10, 10.08),
    (Q4_K, 9, 4096, 3584, 7.94, 9.36), (Q4_K, 10, 4096, 2560, 7.76, 9.02),
    (Q4_K, 12, 4096, 2560, 7.87, 10.23), (Q4_K, 12, 4096, 1280, 8.12, 7.72),
    (Q4_K, 16, 4096, 768, 7.67, 7.08), (Q4_K, 16, 4096, 2048, 7.53, 11.65),
    (Q4_K, 16, 1024, 2048, 6.82, 8.62), (Q4_K, 5, 14336, 4096, 15.73, 14.43),
    (Q4_K, 1, 16384, 4096, 13.60, 14.51), (Q4_K, 4, 5120, 8192, 12.60, 16.14),
    (Q4_K, 2, 5120, 14336, 16.65, 23.44), (Q4_K, 16, 20480, 2048, 12.94, 14.90),
    (Q4_K, 8, 28672, 2048, 14.77, 13.76), (Q4_K, 8, 4096, 2048, 7.13, 7.66),
    (Q4_K, 14, 5120, 2048, 7.71, 8.52), (Q4_K, 11, 4096, 1024, 6.56, 6.99),
    (Q4_K, 14, 512, 1280, 7.25, 6.18), (Q4_K, 13, 512, 1536, 7.68, 6.34),
    (Q4_K, 16, 4096, 1280, 7.75, 8.72),
    (Q6_K, 5, 1024, 4096, 10.36, 8.34),
    (Q6_K, 8, 4096, 4096, 10.49, 9.66), (Q6_K, 16, 4096, 2048, 9.87, 8.86),
    (Q6_K, 4, 5120, 8192, 18.06, 21.80), (Q6_K, 5, 14336, 6144, 27.27, 24.70),
    (Q6_K, 3, 5120, 6144, 13.95, 16.19), (Q6_K, 5, 28672, 4096, 31.03, 29.60)]


@pytest.mark.parametrize("dt,n,rows,cols,staged,registers", SMALL_BATCH)
def test_small_batch_takes_the_faster_kernel(rules, dt, n, rows, cols, staged, registers):
    """3%: what two runs of one side differ by."""
    if rules.in_registers(dt, n, rows, cols):
        assert registers <= 1.03 * staged
    else:
        assert staged <= 1.03 * registers


# (dtype, rows, weights per row, added to y, us both vectors staged, us product staged)
SWIGLU = [
    (Q4_0, 2560, 8192, False, 7.49, 6.90), (Q4_0, 14336, 8192, False, 15.52, 15.26),
    (Q4_K, 4096, 5632, False, 8.64, 7.64), (Q4_K, 8192, 8192, False, 12.13, 11.96),
    (Q8_0, 1536, 8192, False, 7.08, 6.24), (Q8_0, 2048, 8192, False, 7.99, 7.70),
    (Q8_0, 2304, 5632, False, 8.05, 7.63), (Q8_0, 3072, 4608, False, 7.98, 7.61),
    (Q8_0, 2304, 8192, False, 8.43, 8.81), (Q8_0, 2560, 5632, True, 8.62, 8.09),
    (Q8_0, 5120, 5632, False, 9.55, 10.53), (Q8_0, 6144, 8192, False, 13.17, 14.55),
    (Q8_0, 8192, 8192, False, 15.56, 17.02), (Q8_0, 8192, 4096, False, 10.40, 9.56),
    (Q8_0, 14336, 16384, False, 46.47, 43.60), (Q6_K, 1900, 5632, False, 8.43, 7.19),
    (Q6_K, 2560, 8192, True, 10.06, 9.29), (Q6_K, 2560, 5632, True, 9.32, 8.89),
    (Q6_K, 4096, 8192, True, 12.22, 12.91), (Q6_K, 4096, 8192, False, 11.29, 12.83),
    (Q6_K, 8192, 5632, False, 15.08, 15.99), (Q6_K, 8192, 8192, False, 16.54, 17.75),
    (Q6_K, 8192, 8704, False, 31.34, 24.93)]


@pytest.mark.parametrize("dt,rows,cols,add,both,product", SWIGLU)
def test_swiglu_takes_the_faster_prologue(rules, dt, rows, cols, add, both, product):
    if rules.product_staged(dt, rows, cols, add):
        assert product <= 1.03 * both
    else:
        assert both <= 1.03 * product


# (dtype, tokens, rows, weights per row, us of each (parts of a tile, K pieces)
# within 1.3 times the fastest)
PLANS = [
    (Q4_0, 256, 4096, 1024, {(4, 1): 15.4, (4, 2): 19.2}),
    (Q4_0, 640, 10240, 14336, {(1, 2): 206.6, (2, 1): 238.7}),
    (Q4_0, 300, 14336, 14336, {(1, 2): 193.0, (2, 1): 220.7}),
    (Q4_0, 100, 6144, 4096, {(2, 4): 29.5, (2, 5): 29.3, (2, 6): 27.8, (2, 7): 26.9, (2, 8):
     27.2, (4, 2): 30.6, (4, 3): 26.7, (4, 4): 26.2, (4, 5): 24.6}),
    (Q4_0, 512, 6144, 4096, {(1, 3): 56.9, (1, 4): 52.8, (1, 5): 54.0, (2, 1): 58.4, (2, 2):
     46.5, (4, 1): 47.6}),
    (Q8_0, 300, 14336, 5120, {(1, 2): 90.4, (2, 1): 109.9}),
    (Q8_0, 640, 8192, 5120, {(1, 2): 87.3, (2, 1): 107.9}),
    (Q8_0, 300, 6144, 28672, {(1, 4): 205.2, (1, 5): 180.3, (2, 3): 206.2}),
    (Q8_0, 777, 2048, 1024, {(2, 1): 23.1, (4, 1): 19.3, (4, 2): 23.8}),
    (Q8_0, 128, 4096, 4096, {(2, 5): 30.7, (2, 6): 29.7, (2, 7): 28.9, (2, 8): 28.4, (4, 4):
     29.1, (4, 5): 26.9, (4, 6): 25.3, (4, 7): 24.9, (4, 8): 24.5}),
    (Q4_K, 512, 2048, 1024, {(4, 1): 15.6, (4, 2): 19.5}),
    (Q4_K, 150, 6144, 1024, {(2, 1): 20.9, (4, 1): 16.1, (4, 2): 19.1}),
    (Q4_K, 150, 6144, 4096, {(1, 6): 38.2, (1, 8): 35.4, (2, 3): 36.5, (2, 4): 31.4, (4, 2):
     32.8, (4, 3): 29.9}),
    (Q4_K, 2048, 4096, 14336, {(1, 2): 229.8, (2, 1): 247.2}),
    (Q4_K, 65, 1024, 14336, {(2, 7): 36.0, (2, 8): 32.8, (4, 6): 34.5, (4, 7): 30.2, (4, 8):
     27.9}),
    (Q6_K, 300, 6144, 28672, {(1, 4): 235.3, (1, 5): 205.0, (2, 3): 246.3}),
    (Q6_K, 640, 4096, 1024, {(2, 1): 28.8, (2, 2): 34.4}),
    (Q6_K, 777, 4096, 14336, {(1, 3): 164.0, (1, 4): 141.7, (2, 2): 177.5}),
    (Q6_K, 512, 4096, 4096, {(1, 4): 57.3, (1, 6): 55.1, (1, 8): 54.9, (2, 2): 59.6, (2, 3):
     51.9, (2, 4): 46.0})]


@pytest.mark.parametrize("dt,m,rows,cols,us", PLANS)
def test_gemm_plan_is_near_the_fastest(rules, dt, m, rows, cols, us):
    """5%: what two runs of one plan differ by at these sizes (they are bound
    by power, so the clock moves with what ran before)."""
    kind, parts, pieces, _, _ = rules.plan(dt, m, rows, cols)
    assert kind == SPLIT
    assert us.get((parts, pieces), 1e9) <= 1.05 * min(us.values()), (parts, pieces)


# (tokens, rows, weights per row, us fused, us dequantized once), Q6_K
Q6K_ROUTES = [
    (65, 4096, 4096, 25.9, 30.1), (65, 2048, 14336, 53.4, 46.5), (128, 28672, 4096, 74.2, 141.1),
    (256, 4096, 14336, 70.9, 81.8), (256, 1024, 8192, 36.0, 32.5), (300, 3000, 28672, 123.3, 163.5),
    (350, 3584, 6144, 44.7, 52.0), (400, 2048, 2048, 29.2, 25.4), (450, 3584, 10240, 71.2, 78.9),
    (512, 2048, 1024, 26.2, 22.1), (512, 3000, 8192, 64.6, 59.3), (512, 4096, 4096, 46.1, 46.4),
    (512, 28672, 4096, 148.6, 183.4), (512, 128256, 4096, 630.0, 769.2),
    (520, 6144, 14336, 167.9, 265.4), (700, 7168, 10240, 153.0, 190.6),
    (777, 2048, 28672, 150.2, 164.5), (777, 4096, 14336, 143.2, 157.9),
    (1000, 2048, 8192, 70.4, 61.0), (1000, 6144, 4096, 102.2, 74.6),
    (1300, 4096, 8192, 140.6, 117.1), (1300, 6144, 14336, 394.4, 338.7),
    (1700, 1024, 8192, 66.2, 55.9), (1700, 1024, 28672, 149.5, 161.3),
    (2048, 3000, 8192, 145.1, 121.5), (2048, 4096, 8192, 172.7, 152.6)]


@pytest.mark.parametrize("m,rows,cols,fused,once", Q6K_ROUTES)
def test_q6k_gemm_takes_the_faster_route(rules, m, rows, cols, fused, once):
    if rules.dequantize_once(Q6_K, m, rows, cols):
        assert once <= 1.03 * fused
    else:
        assert fused <= 1.03 * once


@pytest.mark.parametrize("dt", [Q4_0, Q8_0, Q4_K, Q6_K])
def test_gemm_split_shapes_reach_every_part_size(rules, dt):
    """What test_gpu_gemm_split.py runs on the GPU covers whole tiles, halves and
    quarters (Q6_K has none) in several K pieces, and a part size unsplit."""
    import test_gpu_gemm_split
    plans = [rules.plan(dt, *shape) for shape in test_gpu_gemm_split.SHAPES]
    assert all(p[0] == SPLIT for p in plans)
    split = {p[1] for p in plans if p[2] > 1}
    assert split == ({1, 2} if dt == Q6_K else {1, 2, 4})
    assert any(p[2] == 1 for p in plans) and any(p[2] == 8 for p in plans)
    assert not rules.dequantize_once(Q6_K, 777, 4096, 14336)

def plain_split_bytes(dt, m, rows, cols):
    """Scratch of the simplest split: whole tiles in as many K pieces as the CUs
    hold or halves in at most 4, by 2.0 and 1.3 us a K step and 6 TB/s for the
    partial sums.  A plan takes no more than this or than the allocation-free
    entry point's scratch leaves beside the bf16 x."""
    steps, tiles = cols // 64, -(-m // 256) * -(-rows // 256)

    def piece(n):
        k = -(-steps // n)
        return -(-k // 4) * 4 if dt in (Q4_K, Q6_K) else k

    def us(step, n):
        return piece(n) * step + ((2 * n + 1) * m * rows * 4 / 6e6 if n > 1 else 0)

    whole = min(CUS // tiles, 8, steps // 8)
    half = max(1, min(CUS // (2 * tiles), 4, steps // 8)) if 4 * tiles <= CUS else 1
    pieces = -(-steps // piece(whole if whole >= 2 and us(2.0, whole) < us(1.3, half) else half))
    return pieces * m * rows * 4 if pieces > 1 else 0


@pytest.mark.parametrize("dt", [Q4_0, Q8_0, Q4_K])
def test_calls_of_the_fixed_scratch_keep_fitting(rules, dt):
    """swamp_qgemv_batched_noalloc refuses a call whose bf16 x and partial sums
    exceed its 32 MiB: every shape that fits with the simplest split fits."""
    limit, pad, near = 32 << 20, lambda b: -(-b // 256) * 256, 0
    for m in [*range(65, 520, 13), *range(520, 2049, 61)]:
        for rows in (130, 1000, 1024, 2048, 2560, 3000, 4096, 5120, 6144, 8192, 11008, 14336,
                     28672):
            if 2 * -(-m // 256) * -(-rows // 256) > CUS:
                continue
            for cols in (512, 1024, 2048, 4096, 5120, 8192, 14336, 28672):
                xb = pad(m * cols * 2)
                before = xb + pad(plain_split_bytes(dt, m, rows, cols))
                now = xb + pad(rules.plan(dt, m, rows, cols)[4])
                assert now <= max(limit, before), (m, rows, cols)
                near += 0.8 * limit < now <= limit
    assert near > 50, near


# (tokens, rows, weights per row, us in K phases, us in K groups)
K_GROUPS = [
    # Q4_0
    (32, 4096, 1024, 7.91, 8.94), (25, 14337, 1024, 8.14, 12.04), (63, 14337, 1024, 12.22, 18.93),
    (64, 4096, 1024, 11.11, 10.87), (16, 2048, 2048, 6.94, 7.95), (50, 16384, 2048, 18.56, 18.51),
    (17, 12288, 1536, 10.23, 10.50), (8, 4096, 6144, 11.69, 10.48), (48, 1024, 4096, 24.73, 11.17),
    # Q8_0
    (17, 6144, 1024, 8.05, 9.37), (32, 14337, 2048, 15.74, 17.55),
    # Q4_K
    (16, 4096, 2048, 7.26, 8.13), (16, 4096, 1536, 8.28, 7.77), (16, 12288, 1536, 8.88, 9.98),
    (16, 4096, 1792, 8.52, 7.80), (32, 12288, 2048, 12.43, 13.27), (32, 4096, 2048, 10.14, 9.70),
    (16, 4096, 4096, 9.99, 8.78),
    # Q6_K
    (25, 6144, 1024, 9.88, 11.64), (32, 4096, 2048, 12.72, 11.91), (32, 4096, 1536, 12.99, 11.62)]


@pytest.mark.parametrize("n,rows,cols,phases,groups", K_GROUPS)
def test_small_batch_splits_k_where_it_is_faster(rules, n, rows, cols, phases, groups):
    if rules.k_groups(n, rows, cols):
        assert groups <= 1.03 * phases
    else:
        assert phases <= 1.03 * groups
