"""Downloads (csrc/transfer.cpp) built for the host over a stand-in for the HIP
calls they make (tests/native/transfer_host.cpp): what is shared between handles
and threads, without a GPU."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "scale-dg-kernel-extraction_amd"
ROCM = Path("/opt/rocm")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++") or not (ROCM / "include" / "hip").exists():
        pytest.skip("needs g++ and the HIP headers")
    exe = tmp_path_factory.mktemp("transfer") / "transfer_host"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    f"-I{ROOT}/include", f"-I{PKG}/csrc", "-o", str(exe),
                    str(ROOT / "tests" / "native" / "transfer_host.cpp"),
                    str(PKG / "csrc" / "transfer.cpp"), "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["handles_while_waiting", "download_while_waiting",
                                      "plain_count_ends_with_handles", "sliced_sizes",
                                      "plain_destinations_and_failures"])
def test_scenario(program, scenario):
    r = subprocess.run([str(program), scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
