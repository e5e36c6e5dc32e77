"""Kernel sources run on the host, lane by lane, between guard pages: shapes whose accesses are checked here and not by
running them on a GPU."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "torch-points-kernels_amd", "csrc")


def _emulated(folder, unit, name):
    for source_name in os.listdir(CSRC):
        if not source_name.endswith(".h") and source_name != unit + ".hip":
            continue
        with open(os.path.join(CSRC, source_name)) as f:
            source = f.read()
        # dynamic LDS is a pointer into the emulated one, the one instruction written by hand an assignment
        source = re.sub(r"extern __shared__ (?:__align__\(16\) )?([a-z0-9 ]+?) ([a-z_]+)\[\];", r"\1* const \2 = reinterpret_cast<\1*>(emulation::lds);", source)
        source = source.replace('asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "s"(uniform_value));', "v = uniform_value;")
        source = re.sub(r"typedef _Float16 (\w+) __attribute__\(\(vector_size\((\d+)\)\)\);", r"typedef emulation::Halves<\2 / 2> \1;", source)
        source = source.replace('"../../include/tpk.h"', '"%s"' % os.path.join(ROOT, "include", "tpk.h"))
        with open(os.path.join(folder, source_name.replace(".hip", ".cpp")), "w") as f:
            f.write(source)
    program = os.path.join(folder, name)
    subprocess.run(["g++", "-std=c++17", "-O2", "-w", "-fpermissive", "-Wno-psabi", "-ffp-contract=off", "-U_FORTIFY_SOURCE", "-fsanitize=bounds",
                    "-fno-sanitize-recover=bounds", "-I" + folder, "-I" + os.path.join(HERE, "emulation"),
                    os.path.join(HERE, "emulation", name + ".cpp"), "-o", program], check=True)
    return program


@pytest.fixture(scope="module")
def ball_query_dense(tmp_path_factory):
    return _emulated(str(tmp_path_factory.mktemp("emulated")), "nn_grid", "ball_query_dense")


@pytest.fixture(scope="module")
def ball_query_packed(tmp_path_factory):
    return _emulated(str(tmp_path_factory.mktemp("emulated")), "ball_table", "ball_query_packed")


# (clouds of 9373 points: windows of 8192 that hold parts of two clouds, the last of 75 points, whose second part is empty; the first
# is the call that test_ball_query_of_the_clouds_own_points leaves to this test)
@pytest.mark.parametrize("clouds,points,queries,nsample,radius,own", [(7, 9373, 9373, 16, 0.05, 1), (7, 9373, 640, 16, 0.05, 0), (2, 8193, 8193, 64, 0.1, 0)])
def test_dense_ball_query_stays_in_bounds(ball_query_dense, clouds, points, queries, nsample, radius, own):
    done = subprocess.run([ball_query_dense] + [str(v) for v in (clouds, points, queries, nsample, radius, own)], capture_output=True,
                          text=True, timeout=300)
    assert done.returncode == 0, done.stdout + done.stderr


# (radius 2: all points of a cloud in a few buckets; 0.02: hardly two in one; 12291 points: the last workgroup counts three; 65537 points: 512 by a
# workgroup, the last one a single point)
@pytest.mark.parametrize("clouds,points,queries,nsample,radius,sort", [(1, 12291, 8192, 16, 2.0, 0), (3, 8200, 8195, 5, 0.3, 0), (1, 9000, 8192, 16, 0.02, 0),
                                                                       (2, 8192, 700, 64, 0.2, 1), (1, 65537, 1100, 16, 0.15, 1)])
def test_packed_ball_query_counts_with_few_atomics(ball_query_packed, clouds, points, queries, nsample, radius, sort):
    """In bounds and right; and however many points a bucket holds, those of a workgroup's 256 to 1024 consecutive ones that lie in it share
    one atomic, in a small array where a bucket holds six of them (atomics on one address wait for each other: an atomic per point took 550 us where a ball held a cloud of 100000)."""
    done = subprocess.run([ball_query_packed] + [str(v) for v in (clouds, points, queries, nsample, radius, sort)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout + done.stderr
    wrong, atomics, buckets, by_group, chunks = (int(v) for v in re.findall(r"(\d+) (?:wrong|atomics|buckets|by group|chunks)", done.stdout))
    assert wrong == 0 and atomics <= by_group + chunks


@pytest.fixture(scope="module")
def chamfer(tmp_path_factory):
    return _emulated(str(tmp_path_factory.mktemp("emulated")), "nn_grid", "chamfer")


# (530 points: a last cell of 18, whose second 32 queries are none; wavefronts that share a cell have half of their queries at most; 1032 points:
# a second tile of products without queries in the last cell of every part; 58 pairs of 18 cells: wavefronts with all queries of a cell)
@pytest.mark.parametrize("clouds,n,m,kind", [shape + (kind,) for shape in [(1, 530, 1032), (2, 1032, 700)]
                                             for kind in ("even", "lattice", "scan", "outliers", "scaled", "twins", "far", "not a number")]
                         + [(58, 514, 513, "outliers"), (58, 514, 513, "twins")])
def test_chamfer_finds_the_nearest(chamfer, clouds, n, m, kind):
    """The search's answers where the matrix products err by as much as its bound assumes and a NaN has the sign that orders above everything."""
    done = subprocess.run([chamfer] + [str(v) for v in (clouds, n, m, kind, 1)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout + done.stderr
