"""Host paths of the library on a stand-in for the HIP runtime
(fake_hip.cpp): what it allocates, launches and copies, and what it does when
an allocation is refused.  Each test body runs in a process of its own, since
the stand-in has to be loaded before the library."""
import os
import subprocess
import sys

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(TESTS)

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
fake.fake_device_bytes.restype = ctypes.c_size_t
fake.fake_limit_device.argtypes = [ctypes.c_size_t]
for f in (fake.fake_fail_host_alloc, fake.fake_fail_events, fake.fake_fail_new):
    f.argtypes = [ctypes.c_long]
import numpy as np
import glp_amd as G

def log():
    return fake.fake_log().decode().split()

def edgeless(n):
    return G.Graph.from_csr(np.zeros(n + 1, dtype=np.int32), np.zeros(0, dtype=np.int32))

def with_labels(s, n, seed=0):
    # a session showing labels of its own, and those labels
    state = bytearray(s.save())
    lab = np.random.default_rng(seed).integers(0, n, n).astype(np.int32)
    state[-4 * n:] = lab.tobytes()
    s.load(bytes(state))
    return lab
"""


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I" + os.path.join(rocm, "include"),
                    os.path.join(TESTS, "fake_hip.cpp"), "-o", out], check=True)

    def run(body):
        env = dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""))
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, out], capture_output=True, text=True, env=env,
                           timeout=300)
        assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-4000:])
        return r.stdout

    return run


def test_result_copies_without_pinned_memory(fake_hip):
    """Results are copied whether or not pinned slots and their events can be
    had, for sizes with one and with several copying threads."""
    fake_hip("""
for n in (1 << 19, 3 << 19, 1 << 22, (1 << 22) + 5):
    for fail, least in ((fake.fake_fail_host_alloc, 0), (fake.fake_fail_events, 0), (fake.fake_fail_events, 1),
                        (fake.fake_fail_events, 5), (fake.fake_fail_host_alloc, -1)):
        s = G.Session(edgeless(n))
        lab = with_labels(s, n)
        fail(least)
        for _ in range(3):
            assert np.array_equal(s.labels(), lab), (n, least)
        fail(-1)
        assert np.array_equal(s.labels(), lab), (n, least)  # and once there is memory again
        s.free()
""")


def test_result_copies_when_no_thread_state_can_be_allocated(fake_hip):
    """A copy by several threads neither throws nor ends the process when an
    allocation fails inside it, whichever one: it gives the labels."""
    fake_hip("""
n = (1 << 22) + 5
s = G.Session(edgeless(n))
lab = with_labels(s, n)
out = np.empty(n, dtype=np.int32)
copy = G.lib().glp_session_labels
for after in (-1, 0, 1, 2, 3, 4, 5, 6):
    out[:] = -1
    fake.fake_fail_new(after)
    rc = copy(s._h, out.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)))
    fake.fake_fail_new(-1)
    assert rc == 0 and np.array_equal(out, lab), after
""")


def test_result_copies_by_several_threads(fake_hip):
    """Threads that read one session's results at a time, with sizes for one
    and for several copying threads, each get their own."""
    fake_hip("""
import threading
for n in (3 << 19, (1 << 22) + 5):
    s = G.Session(edgeless(n), method=G.LAYERED, gamma=(1, 2))
    rng = np.random.default_rng(n)
    want = {"labels": rng.integers(0, n, n).astype(np.int32), "volume": rng.integers(0, n, n).astype(np.int32)}
    state = bytearray(s.save())
    state[-8 * n:] = want["labels"].tobytes() + want["volume"].tobytes()
    s.load(bytes(state))
    s.labels()
    wrong = []

    def read(what):
        for _ in range(20):
            if not np.array_equal(getattr(s, what)(), want[what]):
                wrong.append(what)

    threads = [threading.Thread(target=read, args=(w,)) for w in ("labels", "volume", "labels", "volume")]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, (n, len(wrong))
""")


def test_copy_slots_stay_with_the_graph(fake_hip):
    """The pinned slots of result copies are made once for all sessions on a
    graph, one after another or alive together, and freed with it."""
    fake_hip("""
for n, slots in (((1 << 22) + 5, 4), (1 << 20, 1)):
    g = edgeless(n)
    log()
    for _ in range(5):
        G.run(g, 1)
    a, b = G.Session(g), G.Session(g, method=G.LAYERED)
    for s in (a, b, a):
        s.labels()
    a.free()
    b.free()
    seen = log()
    assert sum(x.startswith("hipHostMalloc") for x in seen) == slots and "hipHostFree" not in seen
    g.free()
    assert log().count("hipHostFree") == slots
""")


def test_results_are_read_after_the_graph_is_freed(fake_hip):
    """A session's labels can still be copied when its graph has gone; the
    slots go with the last of them."""
    fake_hip("""
n = (1 << 22) + 5
g = edgeless(n)
s = G.Session(g)
lab = with_labels(s, n)
for gone in (False, True):
    if gone:
        log()
        g.free()
        assert "hipHostFree" not in log()
    assert np.array_equal(s.labels(), lab)
s.free()
assert log().count("hipHostFree") == 4
""")


def test_dominant_label_scratch_only_where_it_is_used(fake_hip):
    """Sessions on a large graph hold the dominant label's scratch, and end
    their steps one by one, while gamma is 0; where that memory cannot be had
    they run without it."""
    fake_hip("""
n = 1 << 22
deg = np.full(n, 4, dtype=np.int64)
deg[0] = 5000
off = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
nbr = (np.arange(off[-1], dtype=np.int64) * 7919 % n).astype(np.int32)
g = G.Graph.from_csr(off, nbr)
scratch = n + g.m // 8  # at least

def count(s, steps=3):
    log()
    s.step(steps)
    seen = log()
    return [sum(k in x for x in seen) for k in ("k_dominant_decide", "k_end_stepE", "k_end_stepsE")]

G.Session(g).free()  # the graph's device copy
held = []
for gamma in ((1, 4), (0, 1)):
    before = fake.fake_device_bytes()
    s = G.Session(g, method=G.LAYERED, gamma=gamma)
    held.append(fake.fake_device_bytes() - before)
    if gamma[0]:
        assert count(s) == [0, 0, 1]
        before = fake.fake_device_bytes()
        s.set_gamma(0, 1)
        assert fake.fake_device_bytes() - before >= scratch
        assert count(s) == [3, 3, 0]
        s.set_gamma(1, 4)
        assert count(s) == [0, 0, 1]
        s.set_gamma(1, 2)
        s.set_gamma(0, 1)
        assert fake.fake_device_bytes() - before < 2 * scratch
        s.reset()
        assert count(s) == [2, 3, 0]  # none in the first step
    s.free()
assert held[1] - held[0] >= scratch
for method in (G.CLASSIC, G.LAYERED):
    s = G.Session(g, method=method)
    whole = fake.fake_device_bytes()
    s.free()
    fake.fake_limit_device(whole - fake.fake_device_bytes() - 1)
    s = G.Session(g, method=method)
    assert count(s) == [0, 0, 1]
    s.free()
    fake.fake_limit_device(ctypes.c_size_t(-1).value)
s = G.Session(g, method=G.LAYERED, gamma=(1, 4))
fake.fake_limit_device(0)
s.set_gamma(0, 1)
assert count(s) == [0, 0, 1]
""")


def test_one_launch_keeps_to_the_tuned_shapes(fake_hip):
    """The launch of all tiers runs 32 lanes per half-tier vertex and 512
    threads per block-tier vertex: other shapes asked for by tuning get their
    own launches, and the autotuner times no value that the launch ignores."""
    fake_hip("""
def kernels(**tuned):
    with G.tuning(**tuned):
        s = G.Session(G.Graph.rmat(12, 16, seed=9))
        s.step(1)  # (the first step has launches of its own kind)
        log()
        s.step(1)
        return [x for x in log() if "ClassicHooks" in x]

def has(seen, name):
    return any(name in x for x in seen)

for same in ({}, {"half_lanes": 32}, {"block_threads": 512}, {"half_lanes": 16, "half_max_deg": 0}):
    seen = kernels(**same)
    assert has(seen, "k_tiers") and not has(seen, "k_half") and not has(seen, "k_block"), (same, seen)
seen = kernels(half_lanes=16)
assert not has(seen, "k_tiers") and has(seen, "k_halfINS_12ClassicHooksELb0ELb0ELi1ELi16E"), seen
seen = kernels(block_threads=1024)
assert not has(seen, "k_tiers") and has(seen, "k_blockINS_12ClassicHooksELb0ELb0ELi1024E"), seen

def tuned_runs(graph):  # per timed run of an autotuning: whether its steps were one launch each
    log()
    G.autotune(graph, G.make_params(), steps=2)
    runs = []
    for x in log():
        if "k_reset" in x:
            runs.append(False)
        if "k_tiers" in x:
            runs[-1] = True
    return runs

candidates = 1 + 4 + 2 + 2 + 3 + 4 + 2 + 2 + 2 + 1  # the tuning it begins with, and each key's other values
runs = tuned_runs(G.Graph.rmat(12, 16, seed=9))
assert len(runs) == candidates - 2  # (half_lanes 32 and block_threads 512)
assert runs.count(False) == 3       # (half_lanes 16, block_threads 1024, fused_small 1)
assert len(tuned_runs(G.Graph.rmat(19, 16, seed=9))) == candidates  # too large for one launch
""")


def test_neighbour_order_is_checked_where_it_is_used(fake_hip, tmp_path):
    """Whether a file's neighbour lists ascend is found out for the first
    session whose steps ask, once, without waiting for other work on the
    device; serving such graphs does without."""
    fake_hip("path = %r" % str(tmp_path / "g.bin") + """
np.random.default_rng(3).integers(0, 300, (3000, 2)).astype(np.int32).tofile(path)
g = G.Graph.load_bin(path)
log()
sv = G.Server(1 << 30, max_slots=4)
gid = sv.add_graph(g)
for jid in (sv.submit(g, 2), sv.submit_resident(gid, 2)):
    sv.wait(jid, g.n)
sv.close()
a = G.Session(g, method=G.FREQUENT)
b = G.Session(g, method=G.SEEDED)
c = G.Session(g, gather=True)
assert not any("k_descents" in x for x in log())
sessions = [G.Session(g, method=m) for m in (G.LAYERED, G.CLASSIC, G.SLPA)]
seen = log()
assert sum("k_descents" in x for x in seen) == 1 and "hipFree" not in seen
log()
G.autotune(G.Graph.load_bin(path), G.make_params(), steps=1)
assert sum("k_descents" in x for x in log()) == 1
""")


def test_batch_time_begins_after_the_reset(fake_hip):
    """A reset is queued and not waited for; the time that a batch's run
    reports is that of its steps."""
    fake_hip("""
graphs = [G.Graph.planted(500, 5, 6.0, 2.0, seed=i) for i in range(3)]
b = G.Batch(graphs)
for mode, reset in ((0, False), (1, True), (2, True), (2, True), (0, True)):
    if reset:
        b.reset()
    if mode == 2:
        b.run(0, mode=2)  # (its sessions are made)
        b.reset()
    log()
    b.run(2, mode=mode)
    seen = log()
    step = [i for i, x in enumerate(seen) if "k_tiers" in x or "k_packed" in x or x == "hipGraphLaunch"][0]
    assert seen[:step].count("hipStreamSynchronize") >= (len(graphs) if mode == 2 else 1), (mode, seen)
""")
