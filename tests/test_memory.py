"""The device memory that the library keeps between calls, on a device that exists only in the test, and the rules by which a plan
takes the forms that are made on the device (no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "matxtractt_amd", "csrc")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = str(tmp_path_factory.mktemp("memory") / "memory_driver")
    cmd = ["g++", "-O1", "-g", "-std=c++17", "-pthread", "-fopenmp", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"),
           "-I" + SRC, "-I/opt/rocm/include", os.path.join(ROOT, "tests", "cxx", "memory_driver.cpp"), os.path.join(SRC, "mx_util.cpp"), os.path.join(SRC, "mx_upload.cpp"),
           "-o", exe]
    b = subprocess.run(cmd, capture_output=True, text=True)
    assert b.returncode == 0, b.stderr[-2000:]
    return exe


@pytest.mark.parametrize("check", ["wait_refused", "bound", "age", "scope_full", "scope_share", "one_stream", "host_memory", "copies", "copies_of_threads", "copies_refused"])
def test_memory_kept_between_calls(driver, check):
    """tests/cxx/memory_driver.cpp, one check at a time."""
    r = subprocess.run([driver, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.fixture(scope="module")
def forms(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = str(tmp_path_factory.mktemp("forms") / "forms_driver")
    cmd = ["g++", "-O0", "-std=c++17", "-fopenmp", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"), "-I" + SRC,
           "-I/opt/rocm/include", os.path.join(ROOT, "tests", "cxx", "forms_driver.cpp"), os.path.join(ROOT, "tests", "sanitize", "launch_stubs.cpp")] + \
          [os.path.join(SRC, f) for f in ("mx_util.cpp", "mx_upload.cpp", "mx_partition.cpp", "mx_host_layout.cpp", "mx_plan.cpp", "mx_plan_device.cpp",
                                          "mx_plan_view.cpp", "mx_run.cpp")] + \
          ["-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-o", exe]
    b = subprocess.run(cmd, capture_output=True, text=True)
    assert b.returncode == 0, b.stderr[-2000:]
    return exe


@pytest.mark.parametrize("check", ["no_memory", "window_rule", "keep_rule", "offset_waves", "offset_lists", "csr_blocks", "strides", "window_buckets", "host_look"])
def test_forms_looked_for(forms, check):
    """tests/cxx/forms_driver.cpp, one check at a time."""
    r = subprocess.run([forms, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.fixture(scope="module")
def host_arrays(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = str(tmp_path_factory.mktemp("arrays") / "host_arrays_driver")
    cmd = ["g++", "-O1", "-std=c++17", "-fopenmp", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"), "-I" + SRC,
           "-I/opt/rocm/include", os.path.join(ROOT, "tests", "cxx", "host_arrays_driver.cpp"), os.path.join(ROOT, "tests", "sanitize", "launch_stubs.cpp")] + \
          [os.path.join(SRC, f) for f in ("mx_util.cpp", "mx_upload.cpp", "mx_partition.cpp", "mx_host_layout.cpp", "mx_plan.cpp", "mx_plan_device.cpp",
                                          "mx_plan_view.cpp", "mx_run.cpp")] + \
          ["-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-o", exe]
    b = subprocess.run(cmd, capture_output=True, text=True)
    assert b.returncode == 0, b.stderr[-2000:]
    return exe


@pytest.mark.parametrize("check", ["refused", "memory", "sizes"])
def test_parts_from_host_arrays(host_arrays, check):
    """tests/cxx/host_arrays_driver.cpp, one check at a time."""
    r = subprocess.run([host_arrays, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
