"""Host side of transfers against a runtime of host memory (tests/native/fake_hip.h),
so that failures of the runtime can be had without a GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def _build(tmp_path_factory, name):
    out = str(tmp_path_factory.mktemp("native") / name)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-unused-result",
                    os.path.join(HERE, "native", name + ".cpp"), "-o", out, "-lpthread"], check=True)
    return out


@pytest.fixture(scope="module")
def transfer_check(tmp_path_factory):
    return _build(tmp_path_factory, "transfer_check")


# 1 MB: two chunks; 2: three; 20: 21 chunks, more than the ring has, with threads
@pytest.mark.parametrize("megabytes", [1, 2, 20])
@pytest.mark.parametrize("what,call", [("none", 0), ("record", 0), ("record", 1), ("record", 18), ("sync", 0), ("sync", 2)])
@pytest.mark.parametrize("direction", ["up", "down", "stage"])
def test_transfers_that_fail_leave_nothing_in_flight(transfer_check, direction, what, call, megabytes):
    if direction == "stage":
        megabytes = min(megabytes, 15)  # what the ring holds
    r = subprocess.run([transfer_check, direction, what, str(call), str(megabytes)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout)


@pytest.fixture(scope="module")
def pool_check(tmp_path_factory):
    return _build(tmp_path_factory, "pool_check")


@pytest.mark.parametrize("check", ["give_without_host_memory", "keeps_the_largest", "close_fit", "full_device"])
def test_blocks_kept_by_a_device_handle(pool_check, check):
    r = subprocess.run([pool_check, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


def test_every_device_allocation_can_use_idle_blocks():
    """hipMalloc is called in wr_memory.h alone: an allocation elsewhere would fail
    while a device handle holds idle blocks that it could have had."""
    csrc = os.path.join(os.path.dirname(HERE), "wurstrenderer_amd", "csrc")
    users = {f for f in os.listdir(csrc) if "hipMalloc(" in open(os.path.join(csrc, f)).read()}
    assert users == {"wr_memory.h"}
