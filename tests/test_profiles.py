"""The committed kernel profiles and the byte counts bench.py sets against them belong to the kernels
that are there."""
import glob
import os
import re

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def kernels_in_sources():
    names = set()
    for path in glob.glob(os.path.join(ROOT, "pfem_amd", "csrc", "*.hip")):
        with open(path) as f:
            names |= set(re.findall(r"__global__[^;{]*?\b(k_[a-z0-9_]+)\(", f.read()))
    return names


def test_profile_tables_name_present_kernels():
    have = kernels_in_sources()
    assert {"k_kry_v", "k_wc_mom", "k_amg_rr"} <= have
    for path in sorted(glob.glob(os.path.join(ROOT, "profiles", "*.md"))):
        with open(path) as f:
            rows = [line.split("|")[1] for line in f if line.startswith("| `")]
        gone = set(re.findall(r"\bk_[a-z0-9_]+", " ".join(rows))) - have
        assert not gone, (os.path.basename(path), gone)


def test_traffic_belongs_to_the_timed_kernel(tmp_path):
    assert bench.pmc_traffic() > 500_000_000
    other = tmp_path / "other.md"
    other.write_text("kernel: k_kry_v<double, 16>\ntraffic_bytes_per_launch: 541480892\n")
    assert bench.pmc_traffic(str(other)) is None


def test_wc_step_bytes_counts_the_steps_arrays():
    N, E = 1000, 5000
    words, pos, hmin = 2 * 4 * E * 4, 2 * N * 3 * 8, 2 * N * 8
    v = a = vh = 3 * N
    p = rho = p_old = N
    for s in (4, 8):
        assert bench.wc_step_bytes(3, N, E, s) == words + pos + hmin + 2 * s * (v + a + p + rho + vh + p_old)
