"""The number of CPUs that the read-back threads may use: affinity mask and control-group quota (no GPU)."""
import ctypes as C
import os

import pytest

from overlap_amd import ovl

PLENTY = len(os.sched_getaffinity(0))


def cpus(root):
    return ovl.lib().ovl_hostcopy_cpus(os.fsencode(str(root)))


@pytest.mark.parametrize("text,want", [
    ("max 100000\n", PLENTY), ("200000 100000\n", 2), ("250000 100000\n", 2), ("50000 100000\n", 1),
    ("100000000 100000\n", PLENTY), ("", PLENTY), ("nonsense\n", PLENTY)])
def test_quota_of_version_2(tmp_path, text, want):
    (tmp_path / "cpu.max").write_text(text)
    assert cpus(tmp_path) == min(want, PLENTY)


@pytest.mark.parametrize("quota,want", [("-1", PLENTY), ("300000", 3), ("1000", 1)])
def test_quota_of_version_1(tmp_path, quota, want):
    (tmp_path / "cpu").mkdir()
    (tmp_path / "cpu" / "cpu.cfs_quota_us").write_text(quota + "\n")
    (tmp_path / "cpu" / "cpu.cfs_period_us").write_text("100000\n")
    assert cpus(tmp_path) == min(want, PLENTY)


def test_no_control_group(tmp_path):
    assert cpus(tmp_path) == PLENTY
    assert 1 <= ovl.lib().ovl_hostcopy_cpus(C.c_char_p(None)) <= PLENTY
