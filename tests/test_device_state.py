"""What the host code keeps on the device between calls, on the CPU: tests/native/device_state runs the host sources
against a stand-in for the HIP runtime that knows which memory is allocated, what a stream capture forbids and
what a captured graph launches."""

from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

NATIVE = Path(__file__).resolve().parent / "native"


@pytest.fixture(scope="module")
def driver() -> Path:
    res = subprocess.run(["make", "-C", str(NATIVE), "-j8", "_build/device_state"], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout[-3000:] + res.stderr[-3000:]
    return NATIVE / "_build" / "device_state"


SCENARIOS = [
    "graph_of_large_workspace",
    "capture_of_a_walk_after_a_short_run",
    "capture_without_durations_after_a_short_run",
    "capture_of_a_short_run_after_a_walk",
    "short_run_beside_a_capture",
    "capture_of_a_first_run",
    "statistics_in_little_memory",
    "short_run_without_room_for_its_plan",
    "release_of_workspaces",
    "wide_steps_below_a_round",
    "shapes_of_two_samples_per_lane",
    "two_passes_where_they_are_faster",
]


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_device_state(driver: Path, scenario: str) -> None:
    res = subprocess.run([str(driver), scenario], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0 and res.stdout.strip() == "OK", res.stdout + res.stderr
