"""The planes' transfers (csrc/stage.hip) on the host over a stand-in for the HIP runtime (tests/host/fake_hip.hpp): the
same bytes both ways whatever the caller's memory is and whatever fails."""
import pytest

from helpers import WORLD_SOURCES, host_program, run_host


@pytest.fixture(scope="module")
def stage(tmp_path_factory):
    return host_program(tmp_path_factory.mktemp("stage"), "stage", ["stage.hip", "util.cpp"])


@pytest.mark.parametrize("case", ["pageable", "pinned", "threads", "device"])
def test_transfers(stage, case):
    run_host(stage, case)


def test_a_failed_transfer_leaves_no_device_memory(tmp_path):
    run_host(host_program(tmp_path, "world_transfer", WORLD_SOURCES))
