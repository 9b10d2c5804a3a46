"""Error paths of the library's host code, built without its kernels on a HIP
runtime of the test's own (host_hip): no GPU is used.  Every allocation or
launch of a call is made to fail in turn."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests", "host_hip")
SOURCES = ("hs2_kernels.hip", "hs2_lines.hip", "hs2_dense.hip", "hs2_adjoint.hip", "hs2_api.cpp",
           "hs2_noalloc.hip")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = tmp_path_factory.mktemp("host_hip")
    cmds = [["hipcc", "--cuda-host-only", "-x", "hip", "--offload-arch=gfx950", "-O1",
             "-std=c++17", "-fPIC", "-fuse-cuid=none", "-I", os.path.join(ROOT, "include"), "-c",
             os.path.join(ROOT, "heatsim2_amd", "csrc", s), "-o", str(out / (s + ".o"))]
            for s in SOURCES]
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cmds += [["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I",
              os.path.join(rocm, "include"), "-c", os.path.join(HERE, s), "-o",
              str(out / (s + ".o"))] for s in ("host_hip.cpp", "error_paths.cpp")]
    procs = [subprocess.Popen(c) for c in cmds]
    assert [p.wait() for p in procs] == [0] * len(procs)
    exe = str(out / "error_paths")
    subprocess.run(["g++", "-Wl,--allow-multiple-definition"] +
                   [str(out / f) for f in sorted(os.listdir(out)) if f.endswith(".o")] +
                   ["-o", exe], check=True)
    return exe


@pytest.mark.parametrize("what", ["set_compact_host_memory", "set_compact_device_memory",
                                  "set_config_host_memory", "set_config_device_memory",
                                  "batch_lanes", "batch_lanes_graphs", "backward_lanes"])
def test_error_path(program, what):
    run = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout[-2000:] + run.stderr[-2000:]
