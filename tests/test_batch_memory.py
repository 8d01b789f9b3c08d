"""A batch that could be set up on a frame of its own when there is no device memory for it (CPU: the library runs on
a HIP runtime of host memory that fails one call on request, tests/cpp/batch_without_memory.c)."""
import os
import shutil
import subprocess

import pytest

import fastfft_amd as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
OUT_OF_MEMORY, INVALID_VALUE = 2, 1  # hipError_t


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("gcc") is None:
        pytest.skip("gcc not found")
    exe = str(tmp_path_factory.mktemp("batch") / "batch_without_memory")
    r = subprocess.run(["gcc", "-std=gnu11", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                        f"-I{os.path.join(ROOT, 'include')}", os.path.join(ROOT, "tests", "cpp", "batch_without_memory.c"),
                        "-o", exe, "-ldl"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(what="malloc", k=0, code=0):
        env = dict(os.environ, FASTFFT_TUNING_WRITE="")
        r = subprocess.run([exe, F.library_path(), what, str(k), str(code)], capture_output=True, text=True, timeout=60, env=env)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout.split("\n")

    return run


def test_frame_of_small_templates(program):
    out = program()
    assert out[:2] == ["set_batch 0", "batch 0"] and "frame=512x256" in out[2], out


@pytest.mark.parametrize("k", [1, 2, 3])  # the frame, the plan's workspace, the batch's slots
def test_without_memory_the_batch_runs_per_template(program, k):
    out = program("malloc", k, OUT_OF_MEMORY)
    assert out[:2] == ["set_batch 0", "batch 0"] and "frame=full" in out[2] and "chunk=0" in out[2], out


@pytest.mark.parametrize("what,k", [("malloc", 1), ("malloc", 3), ("memcpy", 1)])
def test_other_failures_are_reported(program, what, k):
    out = program(what, k, INVALID_VALUE)
    assert out[0] == f"set_batch {F.HIP_ERROR}", out
