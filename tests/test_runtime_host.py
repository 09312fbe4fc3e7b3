"""The runtime's host code on a HIP runtime of host memory
(tests/emulation/runtime_host.cpp): allocations that fail on request, and the
graphs and streams of batches in parts."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("emulation") / "runtime_host")
    subprocess.run(["/opt/rocm/llvm/bin/clang++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I", "/opt/rocm/include", os.path.join(HERE, "emulation", "runtime_host.cpp"), "-o", out,
                    "-lpthread", "-ldl"], check=True)
    return lambda arg: subprocess.run([out, str(arg)], check=True, capture_output=True, text=True).stdout


# the slot pool, then the tables: slots, parameters, results, and the pinned
# parameters, results and slots
@pytest.mark.parametrize("fail", range(7))
def test_context_survives_a_failed_allocation(emu, fail):
    assert int(emu(fail)) == 0


def test_only_these_allocations(emu):
    assert int(emu(7)) == -1


def test_parts_are_linear_graphs_on_their_own_streams(emu):
    # no fork or join inside a capture: the branches of a graph run on streams
    # of its own, which share hardware queues with the others'
    assert emu("split").split("\n")[:3] == ["4 0 4 4", "0 0 4 4", "2 0 2 2"]
