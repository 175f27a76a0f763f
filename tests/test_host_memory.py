"""Device memory of the projection in range order, under the mock HIP runtime (CPU only):
failing allocations and copies, what a launch reads, and what is held and given back
(tests/host_mock/memory_driver.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests", "host_mock")
CSRC = os.path.join(ROOT, "openbcsim_amd", "csrc")
ROCM_INCLUDE = "/opt/rocm/include"


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir(ROCM_INCLUDE):
        pytest.skip("g++ or the HIP headers are not available")
    out = tmp_path_factory.mktemp("memory_driver")
    flags = ["-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM_INCLUDE}",
             f"-I{os.path.join(ROOT, 'include')}", "-pthread", "-Wno-deprecated-declarations", "-Wno-unused-result"]
    renamed = [f"-D{f}=mock_{f}" for f in ("hipMalloc", "hipMemcpy", "launch_project_tile")]
    sources = {os.path.join(HERE, "mock_hip.cpp"): renamed, os.path.join(HERE, "memory_driver.cpp"): []}
    sources.update({os.path.join(CSRC, f): [] for f in ("sim_host.cpp", "batch_host.cpp", "serve_host.cpp")})
    jobs = [(subprocess.Popen(["g++", *flags, *extra, "-c", src, "-o", str(out / (os.path.basename(src) + ".o"))],
                              stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)) for src, extra in sources.items()]
    for j in jobs:
        log, _ = j.communicate(timeout=600)
        assert j.returncode == 0, log[-4000:]
    exe = str(out / "memory_driver")
    subprocess.run(["g++", "-pthread", "-o", exe, *[str(out / (os.path.basename(s) + ".o")) for s in sources]], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["table_failures", "optional_buffers", "crowds", "origins", "captured_frames",
                                      "server_budget", "tuned_radix", "tuned_shapes_by_origin", "tuned_order", "batch_shapes"])
def test_memory(driver, scenario):
    res = subprocess.run([driver, scenario], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300,
                         env=dict(os.environ, MOCK_DELAY_US="20"))
    print(res.stdout[-3000:])
    assert res.returncode == 0 and f"DONE {scenario}" in res.stdout, res.stdout[-4000:]
