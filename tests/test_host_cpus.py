"""The CPUs that the host passes may use: the quota of control groups, read as the kernel lays it out."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "tpu_compiler_amd", "csrc", "host")


@pytest.fixture(scope="module")
def quota(tmp_path_factory):
    folder = tmp_path_factory.mktemp("cpus")
    (folder / "main.cpp").write_text("""
#include "host_cpus.hpp"
#include <cstdio>
int main(int, char **argv) { printf("%d %d", tpuhip::cpus_of_groups(argv[1], argv[2]), tpuhip::usable_cpus()); }
""")
    subprocess.check_call(["g++", "-std=c++17", "-I" + HOST, str(folder / "main.cpp"), "-o", str(folder / "main")])
    return lambda *args: [int(v) for v in subprocess.check_output([str(folder / "main")] + [str(a) for a in args]).split()]


@pytest.mark.parametrize("groups,files,want", [
    ("0::/\n", {"cpu.max": "max 100000\n"}, 0),
    ("0::/\n", {"cpu.max": "1600000 100000\n"}, 16),
    ("0::/\n", {"cpu.max": "50000 100000\n"}, 1),
    ("0::/\n", {}, 0),
    ("0::/a/b\n", {"a/b/cpu.max": "max 100000\n", "a/cpu.max": "250000 100000\n"}, 2),
    ("0::/a/b\n", {"a/b/cpu.max": "300000 100000\n", "a/cpu.max": "800000 100000\n"}, 3),
    ("4:cpu,cpuacct:/c\n2:memory:/m\n", {"cpu/c/cpu.cfs_quota_us": "400000\n", "cpu/c/cpu.cfs_period_us": "100000\n"}, 4),
    ("4:cpu,cpuacct:/c\n", {"cpu/c/cpu.cfs_quota_us": "-1\n", "cpu/c/cpu.cfs_period_us": "100000\n"}, 0),
    ("3:cpuset:/c\n", {"cpu/c/cpu.cfs_quota_us": "100000\n", "cpu/c/cpu.cfs_period_us": "100000\n"}, 0),
    ("1:cpu:/\n0::/\n", {"cpu/cpu.cfs_quota_us": "700000\n", "cpu/cpu.cfs_period_us": "100000\n", "cpu.max": "600000 100000\n"}, 6),
    ("nothing\n", {}, 0)])
def test_quota_of_control_groups(quota, tmp_path, groups, files, want):
    (tmp_path / "groups").write_text(groups)
    for name, text in files.items():
        at = tmp_path / "fs" / name
        at.parent.mkdir(parents=True, exist_ok=True)
        at.write_text(text)
    got, usable = quota(tmp_path / "groups", tmp_path / "fs")
    assert got == want
    assert 1 <= usable <= len(os.sched_getaffinity(0))
