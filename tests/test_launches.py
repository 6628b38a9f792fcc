"""Which kernels a call launches, recorded without a GPU (tests/launches.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "mlsys26-flashinfer-moe_amd"

# both sides of every size at which a kernel or its instance changes
SIZES = (1, 2, 3, 4, 5, 8, 9, 16, 64, 65, 128, 129, 256, 257, 2048, 2049, 4095, 4096, 16384, 16385)


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    if shutil.which("g++") is None or not Path("/opt/rocm/include/hip").exists():
        pytest.skip("g++ or the HIP headers are not installed")
    exe = tmp_path_factory.mktemp("launches") / "launches"
    res = subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                          f"-I{ROOT / 'include'}", str(ROOT / "tests" / "launches.cpp"), "-o", str(exe), f"-L{PKG}",
                          "-l:libmoe_fp8.so", f"-Wl,-rpath,{PKG}", "-Wl,-rpath,/opt/rocm/lib",
                          "-Wl,--allow-shlib-undefined"], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr

    def run(*calls):
        """[(return code, [events and kernels])] of calls (tokens, packed, profiled, failing launch)."""
        text = "\n".join(" ".join(str(int(x)) for x in c) for c in calls)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, timeout=60, check=True).stdout
        lines = [line.split() for line in out.splitlines()]
        assert len(lines) == len(calls)
        return [(int(f[0]), f[1:]) for f in lines]
    return run


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("T", SIZES)
def test_a_profiled_call_makes_the_launches_of_an_unprofiled_one(launches, T, packed):
    (rc, plain), (rc_profiled, timed) = launches((T, packed, False, 0), (T, packed, True, 0))
    assert rc == rc_profiled == 0 and plain
    assert [x for x in timed if x[0] != "E"] == plain
    marks = [x for x in timed if x[0] == "E"]
    assert marks == ["E0", "E1", "E2", "E3"] and timed[0] == "E0" and timed[-1] == "E3"
    gemm1 = timed[timed.index("E1") + 1:timed.index("E2")]
    assert len(gemm1) == 1 and gemm1[0].startswith(("gemm1_stream_dispatch", "gemm_stream_kernel<1", "gemm_tile_kernel<true"))


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 6, 7, 8, 9, 64])
def test_the_ring_of_gemm1(launches, T, packed):
    """6 slots up to 2 tokens, 4 up to 4 (packed 8), where 4 lose on the row-major weights with 6 experts or
    more; the kernel routes up to 4 tokens."""
    (rc, seq), = launches((T, packed, False, 0))
    slots = 6 if T <= 2 else 4 if T <= (8 if packed else 4) else 0
    p = str(packed).lower()
    gemm1 = f"gemm1_stream_dispatch_deep_kernel<{p},{slots},{str(T <= 4).lower()}>" if slots else f"gemm1_stream_dispatch_kernel<{p}>"
    assert rc == 0 and [x.split("@")[0] for x in seq if x.startswith("gemm1")] == [gemm1]
    assert any(x.startswith("route") for x in seq) == (T > 4)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("T", SIZES)
def test_a_failed_launch_is_reported(launches, T, packed):
    (_, seq), = launches((T, packed, False, 0))
    failed = launches(*[(T, packed, False, n) for n in range(1, len(seq) + 1)])
    assert [rc for rc, _ in failed] == [-6] * len(seq)   # MOE_FP8_ELAUNCH
