"""The split of a small film's step in the bench line: kernel times come from a run
with timing, which makes other launches than the run that gives the rate, so the
kernels' share is of that run's own wall time (no GPU)."""

import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_kernel_share_is_of_the_timed_run():
    spec = importlib.util.spec_from_file_location("bench_line", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    st = dict(steps=1000, f_calls=8000)
    timed = dict(steps=1000, f_calls=8000, demag_passes=8000, demag_ms=60.0, llg_ms=20.0, vec_ms=40.0)
    out = bench._line(0.080, st, (0.150, timed), 1e6)
    assert out["steps_per_s"] == 1000 / 0.080 and abs(out["ms_per_step"] - 0.08) < 1e-12
    assert abs(out["timed_run_ms_per_step"] - 0.15) < 1e-12
    assert abs(out["gpu_kernel_frac_of_timed_step"] - 0.12 / 0.15) < 1e-12
    assert "gpu_kernel_frac_of_step" not in out  # 0.12 of 0.08 ms
    assert abs(out["demag_ms_per_launch"] - 60.0 / 8000) < 1e-15
