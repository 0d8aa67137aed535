"""bench.py's rates of the same-spin kernels: an achieved rate only where the
kernel does the operations that are counted (FP32); the FP64 tiles, which
leave out part of the dense product, report the dense equivalent."""
import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_only_counted_operations_are_an_achieved_rate():
    spec = importlib.util.spec_from_file_location("bench_for_rates", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    assert bench.gemm_rate("sym_same_f32", 2e12, 20.0) == {"flops": 2e12, "TFLOPs": 100.0}
    for name in ("same_gemm", "sym_same"):
        assert bench.gemm_rate(name, 2e12, 20.0) == {"dense_flops": 2e12, "dense_equiv_TFLOPs": 100.0}
