"""The library's host code over a stand-in for the HIP runtime (tests/hip_stub.cpp,
tests/host_runtime.py): what it asks of the device, in which order, on which
stream. On the CPU."""

import json
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="session")
def stub():
    import shutil

    include = Path("/opt/rocm/include")
    if not (include / "hip" / "hip_runtime_api.h").exists() or shutil.which("g++") is None:
        pytest.skip("needs g++ and the HIP headers")
    out = HERE / "_build" / "libhip_stub.so"
    out.parent.mkdir(exist_ok=True)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", f"-I{include}", str(HERE / "hip_stub.cpp"), "-o",
                    str(out)], check=True)
    return out


def scene(stub, name):
    r = subprocess.run([sys.executable, str(HERE / "host_runtime.py"), name], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout.splitlines()[-1])


def test_new_trees_start_from_cleared_state_on_their_own_stream(stub):
    """Sort tickets and look-back words are clear when the first pass of a tree (or
    of a ray order) reads them, whatever the memory held and however late a fill
    on the null stream comes; no device write is ordered on the null stream."""
    r = scene(stub, "clears")
    assert r["completed"] == 11 and r["evictions"] >= 2 and r["uploads"] >= 6 and r["passes"] > 20
    assert r["bad"] == []
    assert r["null_writes"] == 0


def test_failed_device_checks_reach_the_caller(stub):
    """The error bits of a build or a walk are read after a scene's upload and when
    the server retires a batch: the call (or the request) fails, and the next one
    does not."""
    from lux_amd import abi

    r = scene(stub, "errors")
    fails = abi.LUX_ERR_DEVICE_CHECK
    for name in ("create", "update", "first_use", "served_upload", "served_render"):
        assert r[name] == fails, name
    for name in ("update_again", "kept", "served_again", "served_after", "open", "destroy"):
        assert r[name] == 0, name
    assert r["polled"] == [0, fails]


def test_scenes_report_the_memory_they_hold(stub):
    """A scene's device bytes, which the server's budget counts, are those of its
    allocations (the light tables are counted at their largest: 1 KiB here)."""
    for resident, deferred, held, tris in scene(stub, "bytes_held")["scenes"]:
        assert held <= resident <= held + 1024, tris
        assert resident <= deferred <= resident + 1024, tris


def test_instances_lost_in_a_failed_update_are_not_queried(stub):
    """Between a TLAS that is rebuilt and records that are not, every ray would
    miss: such a scene refuses queries until its instances are set."""
    tries = scene(stub, "lost_instances")["tries"]
    assert len(tries) > 10 and tries[-1] == [0, 0]
    assert tries[:-1] == [[6, 1]] * (len(tries) - 1)  # out of memory; refused


def test_traversal_copies_are_made_for_their_first_reader(stub):
    """Builds and refits make no copy that nobody has asked for; a captured query
    makes them keep its copy, since it may be replayed after them; captured builds
    and refits make both; scenes always have both."""
    r = scene(stub, "copies")
    #                     build trace any trace overlap overlap refit refit any overlap trace build overlap
    assert r["first"] == ["-", "r", "-", "-", "p", "-", "-", "-", "r", "p", "-", "-", "p"]
    #              graph:refit trace overlap trace refit graph:trace trace refit trace overlap graph:build graph:trace
    assert r["recorded"] == ["rp", "r", "-", "-", "-", "r", "r", "r", "-", "p", "rp", "-"]
    assert r["scene"] == ["rp", "rp"]


def test_trees_of_few_triangles_take_one_lane_a_ray(stub):
    """Below 16 records a ray is not cut in parts; a tree without records has the
    preorder walk's kernel."""
    assert scene(stub, "query_launches") == {
        "1": ["preorder", 0], "2": ["k_trace", 1024], "16": ["k_trace", 1024], "17": ["parts", 16000],
        "300": ["parts", 16000]}


def test_trace_launches_fit_their_walk(stub):
    """64 x 48 paths: 16 lanes a ray where a walk takes parts, so that many threads
    (or the tuned grid of 8 x 256); trees of few triangles, and the preorder walk, on
    the pairs' kernel, plain mode included."""
    two_level, pairs, mesh, parts = "0", "1", "2", "3"
    paths, lanes, tuned = 64 * 48, 64 * 48 * 16, 8 * 256
    assert scene(stub, "trace_launches") == {
        "room plain": [two_level, lanes], "room plain preorder": [two_level, lanes],
        "room wave": [two_level, tuned], "room wave preorder": [two_level, tuned],
        "box plain": [pairs, paths], "box plain preorder": [pairs, paths],
        "box wave": [pairs, tuned], "box wave preorder": [pairs, tuned],
        "sphere plain": [mesh, paths], "sphere plain preorder": [pairs, paths],
        "sphere wave": [parts, tuned], "sphere wave preorder": [pairs, tuned],
    }


def test_a_build_after_a_failed_one_has_all_its_arrays(stub):
    """Out of memory in the middle of a tree's buffers (of the ray order's, of a path
    buffer's): nothing of them stays, and the next call of no greater size does not take
    the rest for allocated."""
    r = scene(stub, "failed_builds")
    assert len(r["tries"]) > 25 and r["tries"][:-1] == [6] * (len(r["tries"]) - 1) and r["tries"][-1] == 0
    assert not any(r["left"])
    assert r["later"] == {"order": 7, "paths": 12}  # (paths: a buffer for one, then the batch)


def test_two_threads_on_one_tree_wait_for_its_copies(stub):
    r = scene(stub, "two_threads")
    assert r["walks"] == 800 and r["late"] == 0


def test_host_queries_wait_for_their_own_results(stub):
    """Whatever stream another thread's call has made the tree's last one."""
    assert scene(stub, "host_queries") == {"calls": 2, "open": [0, 0]}
