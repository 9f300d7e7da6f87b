"""The rules that choose a kernel by size (csrc/dispatch.hpp), on the CPU."""
import importlib.util
import os
import types

import pytest

from dispatch_rules import CUS, REPO, Q4_0, Q4_K, Q6_K, Q8_0, Rules


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
                for cols in (512, 768, 1024, 4096, 4352, 7680, 8192, 14336, 28672):
                    want = rules.dequantize_once(dt, m, rows, cols)
                    label = bench.gemm_route(gpu, dt == Q6_K, m, rows, cols, "bf16")
                    assert label.startswith("dequantize-once") == want, (dt, m, rows, cols, label)
                    seen.add((dt == Q6_K, want))
    assert len(seen) == 4
