"""The LDS addresses the k-loops read operand fragments at, against the LDS layout, on the CPU: the
address functions select k-halves and column blocks by XOR, which holds only where the stage buffers
start on the alignment that their type (StageRing) carries."""
import subprocess
from pathlib import Path

from grouped_gemm_gpu_kernel_amd import build

SRC = Path(__file__).resolve().parent / "cpp" / "lds_fragments.hip"


def test_fragment_addresses_follow_the_layout_at_every_base(tmp_path):
    exe = tmp_path / "lds_fragments"
    compiled = subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--offload-host-only", str(SRC), "-o", str(exe)],
                              capture_output=True, text=True)
    assert compiled.returncode == 0, compiled.stderr[-4000:]
    ran = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert ran.returncode == 0, ran.stdout + ran.stderr


def test_kernels_hold_their_stages_in_the_aligned_type():
    """Both kernels declare their stage buffers as StageRing, whatever else they keep in LDS."""
    text = (build.CSRC_DIR / "gg_kernels.hip").read_text()
    assert text.count("__shared__ StageRing<KernelLds<S>::HALVES> lds;") == 2
    assert "__shared__ __attribute__" not in text
