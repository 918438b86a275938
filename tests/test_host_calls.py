"""What the library's host code asks of the HIP runtime, on the CPU: each test
runs in a process of its own with tests/host_runtime.cpp in the runtime's
place (no kernel runs, every launch and wait is logged)."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    so = tmp_path_factory.mktemp("rt") / "host_runtime.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", "-o", str(so),
                    os.path.join(HERE, "host_runtime.cpp")], check=True)
    return str(so)


PRELUDE = """
import ctypes, sys, threading
sys.path.insert(0, {root!r})
rt = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
rt.rt_memory_limit.argtypes = [ctypes.c_size_t]
rt.rt_events.argtypes = [ctypes.c_char_p, ctypes.c_size_t]
rt.rt_events.restype = ctypes.c_size_t
def events():
    buf = ctypes.create_string_buffer(rt.rt_events(None, 0) + (1 << 20))
    rt.rt_events(buf, len(buf))
    return [line.split(" ", 1) for line in buf.value.decode().splitlines()]
import numpy as np
import tfm_amd
from tfm_amd import ccp
L = ccp.lib()
"""


def run(runtime, *parts):
    code = PRELUDE.format(root=ROOT, so=runtime) + "\n".join(textwrap.dedent(p) for p in parts) + "\nprint('done')"
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr


CELL_LIST = """
def call(n=64, cps=8):
    u = lambda k: (ctypes.c_uint32 * k)()
    return L.ccp_cell_list_noalloc((ctypes.c_float * (3 * n))(), n, 1.0, cps, u(n), u(n), u(cps ** 3), u(cps ** 3), None)
"""


@pytest.mark.parametrize("cps", [8, 70])
def test_cell_list_calls_do_not_overlap(runtime, cps):
    # The calls of a GPU share one array, and the scan's blocks wait for words
    # of it: one call's launches and its wait come before the next one's first
    # launch, whatever threads they come from.
    run(runtime, CELL_LIST, f"""
    cps = {cps}
    assert call(cps=cps) == 0
    per_call = len(events())
    rt.rt_launch_time(200)
    rcs = []
    ts = [threading.Thread(target=lambda: [rcs.append(call(cps=cps)) for _ in range(5)]) for _ in range(4)]
    for t in ts: t.start()
    for t in ts: t.join()
    assert rcs == [0] * 20
    log = events()
    assert len(log) == 20 * per_call
    for k in range(0, len(log), per_call):
        group = log[k:k + per_call]
        assert len({{t for t, _ in group}}) == 1, log
        assert "k_na_clear" in group[0][1] and group[-1][1] == "wait", log
    """)


def test_cell_list_call_that_fails_waits_for_its_launches(runtime):
    # an error found after the launches: the call ends behind a wait, so that
    # the next one's launches cannot meet them
    run(runtime, CELL_LIST, """
    assert call() == 0
    events()
    rt.rt_fail_last_error(1)
    assert call() == tfm_amd.CCP_ERR_HIP
    log = events()
    assert any("k_na_finish" in e for _, e in log) and log[-1][1] == "wait", log
    assert call() == 0
    """)


SHAPE = """
def fine_cells(n, vf, **kw):
    rco = 1.154701
    r = rco / 2 + rco / 2 * (n / vf) ** (1 / 3)
    s = tfm_amd.Simulation({"number_of_particles": n, "nucleus_radius": f"{r:.6f}", "seed": 1, **kw})
    side, cps = float(s.info.fine_csl), int(s.info.fine_cps)
    s.close()
    return side, cps
"""


@pytest.mark.parametrize("n,vf,half", [
    (1024, 0.2, True), (16384, 0.03, True), (32768, 0.03, False), (65536, 0.1, True), (65536, 0.04, False),
    (131072, 0.1, True), (131072, 0.06, False), (262144, 0.15, True), (262144, 0.08, False), (524288, 0.2, True),
    (524288, 0.1, False), (524289, 0.2, False), (600000, 0.3, False)])
def test_default_cells_of_ccp_field(runtime, n, vf, half):
    # eight lanes over cells of about 1.2 sigma where they were measured to be
    # the faster shape, and at no size above the one that has run
    run(runtime, SHAPE, f"""
    side, cps = fine_cells({n}, {vf})
    assert (1.2 <= side < 1.34) if {half} else side == 2.0, (side, cps)
    assert not {half} or cps ** 3 <= min(32 * {n} + 32768, (2e7 * {n}) ** 0.5)
    assert fine_cells({n}, {vf}, lanes_per_bead=3)[0] == 2.0
    """)


MAPS = """
def sim(n):
    r = 0.577 + 0.577 * (n / 0.2) ** (1 / 3)
    return tfm_amd.Simulation({"number_of_particles": n, "nucleus_radius": f"{r:.6f}", "seed": 1,
                               "contact_bin_size": 1, "contact_cutoff": 1.5})
"""


def test_maps_need_no_memory_beyond_their_own(runtime):
    # the list of a map's nonzero words is a faster way to the host: where the
    # GPU has no memory for it, maps come as they did without it
    run(runtime, MAPS, """
    s = sim(4096)
    rt.rt_memory_limit(0)
    m, _ = s.contact_map()  # the map is on the device already
    assert m.shape == (4096, 4096)
    rt.rt_memory_limit(4 * (1024 * 1025 // 2) + 64)  # the frame's map itself, without its list
    assert s.frame_contact_map().size == 1024 * 1025 // 2
    assert s.contact_map()[0].shape == (4096, 4096)
    rt.rt_memory_limit(2**64 - 1)
    assert s.frame_contact_map().size == 1024 * 1025 // 2
    s.close()
    """)


def test_dense_frame_map_takes_back_the_lists_memory(runtime):
    # a frame's map of too many pixels for its list, with memory for either
    run(runtime, MAPS, """
    s = sim(4096)
    words = 1024 * 1025 // 2
    rt.rt_memory_limit(4 * words + 64)
    rt.rt_fill_copies(1)  # the list's count comes back as 2^32 - 1
    assert s.frame_contact_map().size == words
    assert s.frame_contact_map().size == words
    s.close()
    """)


def test_full_contact_map_is_listed_once(runtime):
    # a summed map with too many nonzero words for its list keeps them until it
    # is cleared: only the first read tries the list
    run(runtime, MAPS, """
    s = sim(4096)
    def listed():
        events()
        assert s.contact_map()[0].shape == (4096, 4096)
        return sum("k_list_words" in e for _, e in events())
    assert [listed(), listed()] == [1, 1]
    rt.rt_fill_copies(1)  # the list's count comes back as 2^32 - 1
    assert [listed(), listed(), listed()] == [1, 0, 0]
    rt.rt_fill_copies(0)
    s.contact_sample()
    assert listed() == 0
    s.contact_reset()
    assert [listed(), listed()] == [1, 1]
    s.close()
    """)
