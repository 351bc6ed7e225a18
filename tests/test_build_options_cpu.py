"""Ring depths the matrix-core kernels can be built with: the index entries of scattered rows are timed for the
default depths, so deeper rings of the kernel of wide tiles have to build without the kernels that read them.  The streaming
kernel has the one depth that its LDS holds."""

import os
import subprocess

import pytest

from async_llm_amd import build

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("source,flags,scattered", [
    ("va_mfma_wide.hip", [], True),
    ("va_mfma_wide.hip", ["-DVA_WIDE_BUFFERS=5"], False),
    ("va_mfma_stream.hip", [], True),
])
def test_ring_depths_build(source, flags, scattered):
    # (the host pass alone: it instantiates the kernels, with their static assertions)
    run = subprocess.run([HIPCC, *build.COMMON_FLAGS, "--offload-arch=gfx950", "--cuda-host-only", *flags, "-S", "-O0",
                          os.path.join(build.CSRC, source), "-o", "-"], capture_output=True, text=True, cwd=build.CSRC)
    assert run.returncode == 0, run.stderr[-2000:]
    assert ("Li256ELb1E" in run.stdout) == scattered
