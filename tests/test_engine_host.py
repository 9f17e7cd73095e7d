"""What the host engine does when an allocation or a launch fails, on the CPU:
engine.cpp with stand-ins for the HIP runtime and the kernels (engine_stub.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def engine(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("engine") / "engine_stub")
    # launchers that no scenario reaches stay undefined
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "gpu_cc_tb_amd/csrc/host/engine.cpp"),
                    os.path.join(ROOT, "tests/engine_stub.cpp"), "-o", exe, "-no-pie",
                    "-Wl,--unresolved-symbols=ignore-all", "-lpthread"], check=True)

    def run(*args):
        p = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=60)
        assert p.returncode == 0 and p.stdout.strip() == "ok", (args, p.returncode, p.stdout, p.stderr)

    return run


@pytest.mark.parametrize("which", ["map", "bits", "count"])
@pytest.mark.parametrize("scheme", ["gacco", "gputx"])
def test_load_after_failed_allocation(engine, scheme, which):
    """The buffers of the written-row filter are all there after a load that
    returns OK, also when one of them could not be had in the load before."""
    engine("alloc", scheme, ["map", "bits", "count"].index(which))


@pytest.mark.parametrize("when", ["first", "later"])
@pytest.mark.parametrize("scheme", ["tpl_nw", "to", "mvcc", "tictoc", "gacco", "gputx"])
def test_run_after_failed_load(engine, scheme, when):
    """A run after a load that failed finds no transactions, not the new
    counts on buffers that are missing or too small."""
    engine("run", scheme, when)


@pytest.mark.parametrize("scheme", ["tpl_nw", "to"])
def test_run_waits_for_queued_batches(engine, scheme):
    """A plain run whose launch fails returns with no batch still running."""
    engine("launch", scheme)


def test_tpcc_queues_behind_an_error(engine):
    """Each batch's combiner is told where an error shows."""
    engine("tpcc")
