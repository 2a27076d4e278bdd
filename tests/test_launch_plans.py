"""Launch plans that the host forms, over all sizes they serve: what a kernel
assumes of its workgroup and its memory holds for each (no GPU needed; the
library's own plan functions, called from tests/launch_plans.cpp)."""
import os
import subprocess

import pytest

from paratc_amd import capi

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(capi.LIB_PATH), "csrc")


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plans") / "launch_plans")
    lib = os.path.dirname(os.path.abspath(capi.LIB_PATH))
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-I", CSRC,
                    "-I", os.path.join(HERE, "..", "include"), os.path.join(HERE, "launch_plans.cpp"), "-o", exe,
                    "-L", lib, "-lparatc_gpu", "-Wl,-rpath," + lib], check=True)
    out = {}
    for line in subprocess.run([exe], capture_output=True, text=True, check=True).stdout.splitlines():
        kind, *v = line.split()
        out.setdefault(kind, []).append(tuple(int(q) for q in v))
    return out


def test_flow_rate_sum_exchanges_among_lanes_of_the_workgroup(plans):
    """The Crank-Nicolson launch sums the flow-rate partials by lane exchanges:
    each lane's partner is a thread of the workgroup, also where an odd number
    of 32-lane chunks ends in half a wavefront."""
    assert [p[0] for p in plans["cn"]] == list(range(4, 257))
    halves = 0
    for ny, chunks, rows, lanes, width in plans["cn"]:
        threads = chunks * lanes
        assert chunks * rows >= ny and width <= 64
        halves += threads % 64 != 0
        off = width // 2
        while off:
            assert all(t ^ off < threads for t in range(threads)), (ny, threads, off)
            off //= 2
    assert halves == 32  # ny 193-208 and 225-240


def test_crank_nicolson_plan_of_every_height(plans):
    """Every height up to 256 has a plan of one of the four compiled shapes, each
    of which some height takes, within its launch bound and the factor table."""
    cap = {(12, 64): 1024, (8, 64): 1024, (4, 64): 1024, (16, 32): 512}
    assert {(p[2], p[3]) for p in plans["cn"]} == set(cap)
    for ny, chunks, rows, lanes, _ in plans["cn"]:
        assert chunks == -(-ny // rows) and chunks * lanes <= cap[rows, lanes], ny
        assert chunks * rows <= 256 and 2 * chunks <= 64, ny
    # the two sides of each change of shape
    by_ny = {p[0]: (p[2], p[3], p[1]) for p in plans["cn"]}
    assert by_ny[192] == (12, 64, 16) and by_ny[193] == (16, 32, 13) and by_ny[256] == (16, 32, 16)


def test_run_time_x_lines_fit_the_lds_they_ask_for(plans):
    """Every line up to 4096 values has a launch on gfx950, and no accepted
    launch asks for more LDS than the limit or than its kernels' last slot
    needs: n / 8 padding slots, and one slot past the line in the inverse."""
    seen = {}
    for h, limit, ok, g, lines, threads, pad, nbytes in plans["x"]:
        seen.setdefault(limit, set()).add(h)
        if limit == 163840:
            assert ok, h
        if ok:
            assert lines * g <= threads <= 1024 and nbytes <= limit, (h, nbytes)
            line = h + (h >> pad) + 1
            assert nbytes >= 16 * lines * line and nbytes >= 8 * threads, (h, nbytes)
    assert seen[65536] == seen[163840] and {3375, 3675, 4096} <= seen[65536]


def test_rhs_rows_fit_the_lds(plans):
    """The RHS kernel's rows (nine quantities, the workgroup's rows and two
    ghost rows each) fit the device's LDS for every row length and request;
    gfx950's limit takes no row away from a shape."""
    for nx, ny, seg, rows, limit, tx, ty, nbytes in plans["rhs"]:
        assert nbytes <= limit and 1 <= ty <= ny and tx * ty <= 512, (nx, ny, seg, rows, limit, nbytes)
        assert nbytes >= 8 * 9 * (ty + 2) * min(nx, tx), (nx, ny, seg, rows, nbytes)
        if limit == 163840 and rows:
            assert ty == max(1, min(rows, 512 // tx, ny)), (nx, ny, seg, rows)
