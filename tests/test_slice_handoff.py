"""The slice GEMM2 of the smallest batches requantises rows into LDS and reads them back from other lanes of
the same wavefront: in the compiled code a wavefront fence lies between the two, so that neither may be
moved across or answered from a lane's own stores."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "mlsys26-flashinfer-moe_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not Path(HIPCC).exists():
        pytest.skip("hipcc is not installed")
    ll = tmp_path_factory.mktemp("ir") / "gemm.ll"
    res = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                          "-packed-fp32-ops", "--offload-device-only", "-S", "-emit-llvm", str(CSRC / "gemm.hip"),
                          "-o", str(ll)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    kernels = re.findall(r"^define .*gemm2_slice_kernel(ILb[01]ELi\d)E.*\{$\n((?:.*\n)*?)^\}$", ll.read_text(), re.M)
    return dict(kernels)


@pytest.mark.parametrize("instance", ["ILb1ELi2", "ILb0ELi1"])   # packed 2 tokens, row-major 1
def test_a_wavefront_fence_lies_between_the_rows_stores_and_loads(kernels, instance):
    lines = kernels[instance].splitlines()
    at = lambda pattern: [i for i, line in enumerate(lines) if re.search(pattern, line)]
    release, acquire = at(r'fence syncscope\("wavefront"\) release'), at(r'fence syncscope\("wavefront"\) acquire')
    stores = at(r"store i32 .*, ptr addrspace\(3\)")        # four requantised bytes
    loads = at(r"load <4 x i32>, ptr addrspace\(3\)")       # half of a fragment
    assert stores and loads
    assert len(release) == len(acquire) == 1
    assert max(stores) < release[0] < acquire[0] < min(loads)
