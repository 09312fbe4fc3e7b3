"""A batch whose workspace cannot be allocated leaves a context that later
batches can use: the runtime's host code on a HIP runtime of host memory
(tests/emulation/runtime_alloc.cpp) whose allocations fail on request."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("emulation") / "runtime_alloc")
    subprocess.run(["/opt/rocm/llvm/bin/clang++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I", "/opt/rocm/include", os.path.join(HERE, "emulation", "runtime_alloc.cpp"), "-o", out,
                    "-lpthread", "-ldl"], check=True)
    return lambda fail: int(subprocess.run([out, str(fail)], check=True, capture_output=True, text=True).stdout)


# the slot pool, then the tables: slots, parameters, results, and the pinned
# parameters, results and slots
@pytest.mark.parametrize("fail", range(7))
def test_context_survives_a_failed_allocation(emu, fail):
    assert emu(fail) == 0


def test_only_these_allocations(emu):
    assert emu(7) == -1
