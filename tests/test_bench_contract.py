"""bench.py's command-line contract, checked without a GPU."""

import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_more_than_one_gpu_is_refused():
    proc = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--gpus", "2"],
                          capture_output=True, text=True, timeout=120)
    assert proc.returncode == 2
    assert "one GPU" in proc.stderr and proc.stdout == ""


def test_help_lists_the_contract_flags():
    proc = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--help"],
                          capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0
    for flag in ("--gpus", "--steps", "--warmup"):
        assert flag in proc.stdout


def test_the_peak_is_that_of_the_kernel_that_ran():
    sys.path.insert(0, str(ROOT))
    import bench
    for plan, peak in (([(5, 1, 8192)], bench.PEAK_BF16X6_MFMA_TFLOPS),
                       ([(1, 4, 700)], bench.PEAK_BF16X6_MFMA_TFLOPS),
                       ([(10, 1, 256)], bench.PEAK_FP32_MFMA_TFLOPS),
                       ([(4, 1, 1792), (4, 3, 256)], bench.PEAK_FP32_MFMA_TFLOPS),
                       ([], bench.PEAK_FP32_MFMA_TFLOPS)):
        assert bench.roofline("mfma", 1.0, split=bench.on_bf16(plan))["peak"] == peak
