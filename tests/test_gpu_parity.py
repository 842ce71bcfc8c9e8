"""GPU parity: the HIP path (libglp.so through its C ABI) against the CPU
oracle, bit-exact at every step."""
import numpy as np
import pytest

import glp_amd as G
import oracle_lib as O

pytestmark = pytest.mark.gpu


def gpu_steps(graph, steps, **kw):
    _, dump, _ = G.run(graph, steps, dump=True, **kw)
    return dump


def hand_graph(edges, n, weights=None):
    off, nbr, w = O.csr_from_edges(n, edges, weights)
    return G.Graph.from_csr(off, nbr, w), off, nbr, w


def assert_steps_equal(got, want):
    for t in range(len(want)):
        bad = np.flatnonzero(got[t] != want[t])
        assert len(bad) == 0, "step %d: %d labels differ, first v=%d gpu=%d oracle=%d" % (
            t + 1, len(bad), bad[0], got[t][bad[0]], want[t][bad[0]])


# ------------------------------------------------------------------ classic ----

def test_classic_closed_forms():
    g, off, nbr, _ = hand_graph([(0, 1), (1, 2), (0, 2), (3, 4), (4, 5), (3, 5), (2, 3)], 7)
    got = gpu_steps(g, 2)
    assert got[0].tolist() == [2, 2, 3, 5, 5, 4, 6]
    assert got[1].tolist() == [3, 3, 2, 5, 5, 5, 6]
    star, *_ = hand_graph([(0, i) for i in range(1, 6)], 6)
    got = gpu_steps(star, 2)
    assert got[0].tolist() == [5, 0, 0, 0, 0, 0] and got[1].tolist() == [0, 5, 5, 5, 5, 5]


def test_classic_planted_65536_twenty_steps():
    g = G.Graph.planted(65536, 64, 12.0, 4.0, seed=1)
    off, nbr, _ = g.csr()
    got = gpu_steps(g, 20)
    assert_steps_equal(got, O.classic(off, nbr, 20))


@pytest.mark.parametrize("scale,ef,sort", [(14, 16, True), (16, 16, True), (15, 8, False)])
def test_classic_rmat_all_tiers(scale, ef, sort):
    g = G.Graph.rmat(scale, ef, seed=scale * 7 + ef, degree_sort=sort)
    off, nbr, _ = g.csr()
    labels, dump, timing = G.run(g, 6, dump=True)
    assert_steps_equal(dump, O.classic(off, nbr, 6))
    if scale == 16:  # max degree ~1e4: packed, wave, block and hub tiers all run
        for tier in ("packed", "wave", "block", "hub"):
            assert timing["tier_vertices"][tier] > 0, tier


def tier_boundary_graph(seed=0):
    """Centres with degrees on every tier and hub-chunk boundary, attached to a
    ring of small communities so neighbour labels repeat and tie."""
    rng = np.random.default_rng(seed)
    degs = [1, 2, 31, 32, 33, 63, 64, 65, 255, 256, 257, 511, 512, 513, 2047, 2048, 2049,
            4095, 4096, 4097, 8191, 8192, 8193, 12289]
    base = len(degs)
    pool = 20000
    n = base + pool
    edges = []
    for i, d in enumerate(degs):
        nb = rng.choice(pool, size=d, replace=False) + base
        edges += [(i, int(x)) for x in nb]
    # background: pool vertices in communities of 50 with sparse ties
    for c in range(pool // 50):
        members = base + c * 50 + np.arange(50)
        for _ in range(120):
            a, b = rng.choice(members, size=2, replace=False)
            edges.append((int(a), int(b)))
    return n, edges


def test_classic_tier_boundaries():
    n, edges = tier_boundary_graph()
    g, off, nbr, _ = hand_graph(edges, n)
    assert_steps_equal(gpu_steps(g, 5), O.classic(off, nbr, 5))


@pytest.mark.parametrize("half,pack,lanes", [(0, 32, 16), (48, 32, 16), (64, 32, 16), (64, 0, 16),
                                             (48, 32, 32), (64, 32, 32), (64, 0, 32)])
def test_half_wave_tier(half, pack, lanes):
    """Degrees in (pack_max_deg, half_max_deg] run 64/lanes per wavefront
    (16 or 32 lanes per vertex); half_max_deg=0 sends them through the
    one-vertex wave path.  pack_max_deg=0 puts degrees 1..64 in the half
    tier.  Classic unweighted and weighted, and layered, must match the
    oracle either way; a planted-partition graph run to convergence takes
    the majority shortcut and the lane merging."""
    with G.tuning(pack_max_deg=pack, half_max_deg=half, half_lanes=lanes):
        gp = G.Graph.planted(6000, 6, 28.0, 8.0, seed=35)
        offp, nbrp, _ = gp.csr()
        _, dumpp, _ = G.run(gp, 12, dump=True)
        assert_steps_equal(dumpp, O.classic(offp, nbrp, 12))
        g = G.Graph.rmat(14, 16, seed=33)
        off, nbr, _ = g.csr()
        _, dump, timing = G.run(g, 6, dump=True)
        assert_steps_equal(dump, O.classic(off, nbr, 6))
        gw = G.Graph.rmat(13, 16, seed=34, wmax=8)
        offw, nbrw, w = gw.csr()
        _, dumpw, _ = G.run(gw, 5, dump=True, weighted=True)
        assert_steps_equal(dumpw, O.classic(offw, nbrw, 5, w=w))
        _, duml, _ = G.run(gw, 4, dump=True, method=G.LAYERED, gamma=(1, 4), weighted=True)
        assert_steps_equal(duml, O.layered(offw, nbrw, 4, 1, 4, w=w)[0])
        n, edges = tier_boundary_graph(seed=3)
        gb, offb, nbrb, _ = hand_graph(edges, n)
        assert_steps_equal(gpu_steps(gb, 4), O.classic(offb, nbrb, 4))


@pytest.mark.parametrize("limit", [0, 8])
def test_hub_partition_and_halving(limit):
    """Tiny thresholds push most vertices through the hub passes; part_limit=8
    forces nearly every hash range to overflow and be halved."""
    with G.tuning(pack_max_deg=8, wave_max_deg=16, block_max_deg=32, hub_chunk=256,
                  part_keys=256, part_limit=limit):
        g = G.Graph.rmat(14, 16, seed=21)
        off, nbr, _ = g.csr()
        labels, dump, timing = G.run(g, 5, dump=True)
    assert timing["tier_vertices"]["hub"] > 1000
    assert_steps_equal(dump, O.classic(off, nbr, 5))


@pytest.mark.parametrize("n", [1500, 5000, 9000, 20000, 41000])
def test_hub_part_batches(n):
    """Every vertex a one-part hub: the part counts lie in each batch length
    of the counting pass (1, 2, 4, 8 and 16 parts per workgroup)."""
    with G.tuning(pack_max_deg=2, half_max_deg=0, wave_max_deg=2, block_max_deg=2, hub_chunk=256, part_keys=256):
        g = G.Graph.planted(n, max(1, n // 500), 10.0, 2.0, seed=5)
        off, nbr, _ = g.csr()
        _, dump, timing = G.run(g, 3, dump=True)
    assert timing["tier_vertices"]["hub"] > 0.95 * n
    assert_steps_equal(dump, O.classic(off, nbr, 3))


@pytest.mark.parametrize("part_keys", [256, 4096])
@pytest.mark.parametrize("chunks", [7, 8, 9, 63, 256, 257, 520])
def test_hub_part_runs(chunks, part_keys):
    """One hub of `chunks` runs per part, short or long ones, walked by all
    waves together or a quarter by each, in one window of 64 runs or more."""
    n = chunks * 256 - 3
    rng = np.random.default_rng(chunks)
    e = np.stack([np.zeros(n, np.int64), np.arange(1, n + 1)], 1)
    e = np.concatenate([e, rng.integers(1, n + 1, (n // 2, 2))])
    with G.tuning(hub_chunk=256, part_keys=part_keys, wave_max_deg=64, block_max_deg=128):
        g, off, nbr, _ = hand_graph([tuple(x) for x in e], n + 1)
        _, dump, timing = G.run(g, 4, dump=True)
    assert timing["tier_vertices"]["hub"] == 1
    assert_steps_equal(dump, O.classic(off, nbr, 4))


def test_hub_weighted_small_tiers():
    with G.tuning(pack_max_deg=4, wave_max_deg=8, block_max_deg=16, hub_chunk=256, part_keys=256):
        g = G.Graph.rmat(13, 16, seed=22, wmax=8)
        off, nbr, w = g.csr()
        got = gpu_steps(g, 4, weighted=True)
    assert_steps_equal(got, O.classic(off, nbr, 4, w=w))


def test_classic_multigraph_and_isolated():
    rng = np.random.default_rng(1)
    n = 3000
    e = rng.integers(0, n // 2, size=(20000, 2))          # upper half isolated
    e = np.concatenate([e, e[:5000]])                      # duplicates
    g, off, nbr, _ = hand_graph([tuple(x) for x in e], n)
    assert_steps_equal(gpu_steps(g, 4), O.classic(off, nbr, 4))


def test_classic_weighted():
    g = G.Graph.rmat(13, 16, seed=5, wmax=8)
    off, nbr, w = g.csr()
    assert_steps_equal(gpu_steps(g, 5, weighted=True), O.classic(off, nbr, 5, w=w))


def test_neighbour_order_invariance():
    g = G.Graph.rmat(13, 16, seed=9)
    off, nbr, _ = g.csr()
    rng = np.random.default_rng(0)
    nbr2 = nbr.copy()
    for v in range(len(off) - 1):
        rng.shuffle(nbr2[off[v]:off[v + 1]])
    g2 = G.Graph.from_csr(off, nbr2)
    assert np.array_equal(gpu_steps(g, 4), gpu_steps(g2, 4))


@pytest.mark.parametrize("kw", [{}, {"gather": True}, {"frontier": True},
                                {"frontier": True, "gather": True}])
def test_empty_and_edgeless(kw):
    g = G.Graph.from_csr(np.zeros(1, np.int32), np.zeros(0, np.int32))
    labels, _ = G.run(g, 3, **kw)
    assert labels.shape == (0,)
    g = G.Graph.from_csr(np.zeros(11, np.int32), np.zeros(0, np.int32))
    labels, _ = G.run(g, 3, **kw)
    assert labels.tolist() == list(range(10))


def test_separate_gather_matches_fused():
    g = G.Graph.rmat(15, 16, seed=3)
    off, nbr, _ = g.csr()
    want = O.classic(off, nbr, 5)
    assert_steps_equal(gpu_steps(g, 5, gather=True), want)


def test_graph_replay_matches_eager_and_changes():
    g = G.Graph.rmat(14, 16, seed=4)
    off, nbr, _ = g.csr()
    want = O.classic(off, nbr, 7)
    with G.Session(g) as s:
        s.step(3)
        s.sync()
        assert np.array_equal(s.labels(), want[2])
        for k in range(4):                      # replays with eager syncs between
            s.step(1, graph=True)
            s.sync()
            assert np.array_equal(s.labels(), want[3 + k])
        ch = s.changes()
    prev = np.vstack([np.arange(len(off) - 1, dtype=np.int32), want[:-1]])
    assert ch.tolist() == [int((want[t] != prev[t]).sum()) for t in range(7)]


@pytest.mark.parametrize("scale,tiny", [(14, False), (15, False), (13, True)])
def test_frontier_equals_dense(scale, tiny):
    """The frontier recomputes only vertices with a changed neighbour once a
    step changes at most n/32 labels; every step must equal the dense run."""
    kw = dict(pack_max_deg=8, wave_max_deg=16, block_max_deg=32, hub_chunk=256,
              part_keys=256) if tiny else {}
    with G.tuning(**kw):
        g = G.Graph.rmat(scale, 16, seed=50 + scale)
        off, nbr, _ = g.csr()
        want = O.classic(off, nbr, 14)
        _, dump, _ = G.run(g, 14, dump=True, frontier=True)
        assert_steps_equal(dump, want)
        with G.Session(g, frontier=True) as s:
            s.step(2)
            s.step(12, graph=True)
            assert np.array_equal(s.labels(), want[-1])
            ch = s.changes()
    prev = np.vstack([np.arange(len(off) - 1, dtype=np.int32), want[:-1]])
    assert ch.tolist() == [int((want[t] != prev[t]).sum()) for t in range(14)]
    assert ch[-1] < (len(off) - 1) // 32   # the frontier was in use at the end


def _push_steps(off, nbr, want, back=1):
    """Steps (1-based) whose frontier gather takes the push form: once adj
    has been gathered `back` times, when the sources whose label in the step
    before differs from their label `back` steps earlier have at most m/8
    in-edges (the gather's own rule; back = 2 is the two-step lookahead)."""
    n, m = len(off) - 1, len(nbr)
    indeg = np.bincount(nbr, minlength=n)
    labs = [np.arange(n, dtype=np.int32)] + list(want)
    return [t for t in range(back + 1, len(labs))
            if int(indeg[labs[t - 1] != labs[t - 1 - back]].sum()) <= m // 8]


@pytest.mark.parametrize("scale,tiny,weighted,frontier", [(14, False, False, 1), (13, True, False, 1),
                                                          (13, False, True, 1), (16, False, False, 1),
                                                          (14, False, False, 2), (13, True, False, 2),
                                                          (13, False, True, 2), (16, False, False, 2)])
def test_frontier_gather_equals_dense(scale, tiny, weighted, frontier):
    """Separate gather with the frontier: after a step whose changed sources
    have few in-edges the gather pushes their labels through the inverse
    index, otherwise it rewrites every edge; every step must equal the
    oracle, also under graph replay and across a checkpoint (which forces a
    full gather).  Sources with more in-edges than one push entry holds
    (256) occur at every scale here; at scale 16 some have thousands.
    frontier=2 adds the two-step lookahead (two adj buffers, changes
    against two steps back)."""
    kw = dict(pack_max_deg=8, wave_max_deg=16, block_max_deg=32, hub_chunk=256,
              part_keys=256) if tiny else {}
    with G.tuning(**kw):
        g = G.Graph.rmat(scale, 16, seed=70 + scale, wmax=8 if weighted else 0)
        off, nbr, w = g.csr()
        want = O.classic(off, nbr, 16, w=w if weighted else None)
        _, dump, _ = G.run(g, 16, dump=True, frontier=frontier, gather=True, weighted=weighted)
        assert_steps_equal(dump, want)
        with G.Session(g, frontier=frontier, gather=True, weighted=weighted) as s:
            s.step(3)
            s.step(8, graph=True)
            assert np.array_equal(s.labels(), want[10])
            state = s.save()
        with G.Session(g, frontier=frontier, gather=True, weighted=weighted) as s2:
            s2.load(state)
            s2.step(5)
            assert np.array_equal(s2.labels(), want[15])
    push = _push_steps(off, nbr, want, back=frontier)
    assert len(push) >= 4 and push[-1] == 16, push   # the push form was in use
    assert int(np.diff(off).max()) > 256


def test_frontier_needs_symmetric_graph():
    """A changed vertex marks its out-neighbours, which are all the vertices
    that read its label only when every edge has its reverse: the frontier
    refuses an asymmetric graph and runs on a symmetric one built from
    caller arrays (checked, not assumed)."""
    g = G.Graph.from_csr([0, 1, 2, 2], [1, 2])   # 0->1->2
    with pytest.raises(G.GLPError):
        G.run(g, 2, frontier=True)
    with pytest.raises(G.GLPError):
        G.run(g, 2, frontier=True, gather=True)
    off, nbr, _ = G.Graph.rmat(12, 8, seed=61).csr()
    gs = G.Graph.from_csr(off, nbr)
    _, dump, _ = G.run(gs, 10, dump=True, frontier=True)
    assert_steps_equal(dump, O.classic(off, nbr, 10))


def test_frontier_rejected_for_layered():
    g = G.Graph.rmat(10, 8, seed=1)
    with pytest.raises(G.GLPError):
        G.run(g, 2, method=G.LAYERED, gamma=(1, 4), frontier=True)


def test_checkpoint_resume():
    g = G.Graph.rmat(13, 16, seed=6)
    off, nbr, _ = g.csr()
    want = O.classic(off, nbr, 6)
    with G.Session(g) as s:
        s.step(3)
        state = s.save()
    with G.Session(g) as s2:
        s2.load(state)
        s2.step(3)
        assert np.array_equal(s2.labels(), want[5])


def test_profile_mode_matches():
    g = G.Graph.rmat(14, 16, seed=8)
    off, nbr, _ = g.csr()
    labels, t = G.run(g, 3, profile=True)
    assert np.array_equal(labels, O.classic(off, nbr, 3)[-1])
    assert t["tier_launches"]["packed"] == 3


@pytest.mark.parametrize("order", ["ascending", "one_swap", "descending", "repeats"])
@pytest.mark.parametrize("weighted", [False, True])
def test_first_step_by_neighbour_order(order, weighted):
    """The step from L0 gathers no labels, and with strictly ascending lists
    needs no tables: every tier of a graph whose lists ascend, one with a
    single pair swapped, one descending and one with repeated neighbours, for
    each method with such a step, eager and replayed, and a restored state of
    step 0 whose labels are not L0."""
    g = G.Graph.rmat(13, 16, seed=5, wmax=8)
    off, nbr, w = g.csr()
    nbr = nbr.copy()
    if order == "one_swap":
        v = int(np.flatnonzero(np.diff(off) > 300)[-1])
        nbr[off[v + 1] - 2:off[v + 1]] = nbr[off[v + 1] - 2:off[v + 1]][::-1].copy()
    elif order == "descending":
        for v in range(len(off) - 1):
            nbr[off[v]:off[v + 1]] = nbr[off[v]:off[v + 1]][::-1].copy()
    elif order == "repeats":
        for v in range(0, len(off) - 1, 3):
            if off[v + 1] - off[v] >= 2:
                nbr[off[v + 1] - 1] = nbr[off[v + 1] - 2]
    ww = w if weighted else None
    with G.tuning(block_max_deg=512, hub_chunk=256, part_keys=256):
        g = G.Graph.from_csr(off, nbr, w)
        want = O.classic(off, nbr, 3, w=ww)
        assert_steps_equal(gpu_steps(g, 3, weighted=weighted), want)
        for gamma in ((0, 1), (1, 4)):
            assert_steps_equal(gpu_steps(g, 3, method=G.LAYERED, gamma=gamma, weighted=weighted),
                               O.layered(off, nbr, 3, gamma[0], gamma[1], w=ww)[0])
        with G.Session(g, method=G.SLPA, slpa_T=3, weighted=weighted) as s:
            s.step(3)
            assert np.array_equal(s.slpa_memory(4), O.slpa(off, nbr, 1, 3, w=ww))
        with G.Session(g, weighted=weighted) as s:
            s.step(3, graph=True)
            assert np.array_equal(s.labels(), want[2])
            s.reset()
            s.step(2, graph=True)
            assert np.array_equal(s.labels(), want[1])
            s.reset()
            state = bytearray(s.save())
            lab = np.random.default_rng(1).integers(0, len(off) - 1, len(off) - 1).astype(np.int32)
            state[-4 * len(lab):] = lab.tobytes()
            s.load(bytes(state))
            s.step(1)
            assert np.array_equal(s.labels(), O.classic_step(off, nbr, lab, ww))


def test_first_step_of_a_loaded_file(tmp_path):
    """A .bin graph's lists are in file order with repeats: the order is
    checked on the device copy."""
    rng = np.random.default_rng(3)
    pairs = rng.integers(0, 300, (3000, 2)).astype(np.int32)
    pairs.tofile(tmp_path / "g.bin")
    chain = np.stack([np.arange(299), np.arange(1, 300)], 1).astype(np.int32)  # ascending lists
    chain.tofile(tmp_path / "c.bin")
    for name in ("g.bin", "c.bin"):
        g = G.Graph.load_bin(str(tmp_path / name))
        off, nbr, _ = g.csr()
        assert_steps_equal(gpu_steps(g, 3), O.classic(off, nbr, 3))


@pytest.mark.parametrize("more", [5, 1021])
def test_dominant_label_of_ragged_vertex_counts(more):
    """Vertices past a full workgroup's share, with degrees on both sides of
    each split of the deciding pass (64, 256 and the hubs' 4,096 edges)."""
    base = G.Graph.rmat(20, 20, seed=12)
    off, nbr, _ = base.csr()
    u = np.repeat(np.arange(base.n, dtype=np.int64), np.diff(off))
    keep = u < nbr
    degs = np.resize([64, 256, 65, 257, 4096, 4097, 3, 0], more)
    rng = np.random.default_rng(more)
    u2 = np.repeat(base.n + np.arange(more), degs)
    v2 = np.concatenate([rng.choice(base.n, d, replace=False) for d in degs])
    e = np.concatenate([np.stack([u[keep], nbr[keep].astype(np.int64)], 1), np.stack([u2, v2], 1)])
    g = G.Graph.from_edges(base.n + more, e)
    assert g.m >= 1 << 24 and np.array_equal(np.diff(g.csr()[0])[base.n:], degs)
    steps = 8
    want = gpu_steps(g, steps, gather=True)
    assert np.bincount(want[steps - 2][g.csr()[1]]).max() > 0.55 * g.m  # the last step has a dominant label
    assert_steps_equal(gpu_steps(g, steps), want)


@pytest.mark.parametrize("sort", [False, True])
def test_dominant_label_settles_the_same_labels(sort):
    """A graph large enough for the dominant label's passes (2^24 edges,
    hubs): the labels and change counts of each step, while labels are
    diverse, converge and have converged, equal those of the separate gather,
    which has no such passes; classic and layered gamma 0, replayed, after a
    restore and across gammas."""
    g = G.Graph.rmat(20, 20, seed=11, degree_sort=sort)
    assert g.m >= 1 << 24
    steps = 8
    want = gpu_steps(g, steps, gather=True)
    _, nbr, _ = g.csr()
    assert np.bincount(want[steps - 2][nbr]).max() > 0.55 * g.m  # the last step has a dominant label
    assert_steps_equal(gpu_steps(g, steps), want)
    assert_steps_equal(gpu_steps(g, steps, method=G.LAYERED, gamma=(0, 1)), want)
    L0 = np.arange(g.n, dtype=np.int32)
    with G.Session(g) as s:
        s.step(steps, graph=True)
        assert np.array_equal(s.labels(), want[-1])
        assert s.changes().tolist() == [int((want[t] != (want[t - 1] if t else L0)).sum()) for t in range(steps)]
        s.reset()
        s.step(5)
        state = s.save()
        s.step(2)
        s.load(state)
        s.step(3)
        assert np.array_equal(s.labels(), want[-1])
    # gamma 0, 1/4, 0: the label chosen before the switch may have moved on
    dumps = []
    for gather in (False, True):
        with G.Session(g, method=G.LAYERED, gamma=(0, 1), gather=gather) as s:
            for gamma, k in (((0, 1), 6), ((1, 4), 2), ((0, 1), 2)):
                s.set_gamma(*gamma)
                s.step(k)
            dumps.append(s.labels())
    assert np.array_equal(dumps[0], dumps[1])


@pytest.mark.parametrize("n,spread", [(1245184, 1), (1245185, 1), (1 << 22, 1), (1 << 22, 3), (41000003, 39)])
def test_dominant_label_look_ups_of_large_vertex_ranges(n, spread):
    """The edges pass looks a neighbour's bit up in LDS (all vertices up to
    1,245,184; else the first ones), in a bit per block of 64 vertices (up to
    39.8 M) or in memory: a graph of 2^20 vertices whose first 1,000 keep
    their ids and whose others lie at the end of n, side by side or `spread`
    apart.  The ids keep their order, so every step's labels are the small
    graph's."""
    g = G.Graph.rmat(20, 20, seed=14)
    off, nbr, _ = g.csr()
    steps = 8
    want = gpu_steps(g, steps, gather=True)
    assert np.bincount(want[steps - 2][nbr]).max() > 0.55 * g.m  # the last step has a dominant label
    ids = n - spread * (g.n - np.arange(g.n, dtype=np.int64))
    ids[:1000] = np.arange(1000)
    deg = np.zeros(n, dtype=np.int64)
    deg[ids] = np.diff(off)
    ids = ids.astype(np.int32)
    large = G.Graph.from_csr(np.concatenate([[0], np.cumsum(deg)]).astype(np.int32), ids[nbr])
    with G.Session(large) as s:
        for t in range(steps):
            s.step(1)
            labels = np.arange(n, dtype=np.int32)
            labels[ids] = ids[want[t]]
            assert np.array_equal(s.labels(), labels), t
        prev = np.vstack([np.arange(g.n, dtype=np.int32)[None], want[:-1]])
        assert s.changes().tolist() == (want != prev).sum(axis=1).tolist()


def test_dominant_label_counts_small_hubs_once():
    """With hubs from 129 edges on, the deciding pass leaves each of them to
    its own workgroup: the change counts are those of the labels."""
    steps = 8
    with G.tuning(pack_max_deg=16, wave_max_deg=64, block_max_deg=128):
        g = G.Graph.rmat(20, 20, seed=13)
        off, nbr, _ = g.csr()
        deg = np.diff(off)
        src = np.repeat(np.arange(g.n), deg)
        want = gpu_steps(g, steps, gather=True)
        hit = 0  # hubs of at most 256 edges that a step's dominant label, on most of their edges, moves to it
        for t in range(1, steps):
            top = np.bincount(want[t - 1][nbr])
            if top.max() > 0.55 * g.m:
                label = top.argmax()
                most = 2 * np.bincount(src[want[t - 1][nbr] == label], minlength=g.n) > deg
                hit += int((most & (want[t - 1] != label) & (deg > 128) & (deg <= 256)).sum())
        assert hit > 0
        with G.Session(g) as s:
            s.step(steps)
            prev = np.vstack([np.arange(g.n, dtype=np.int32)[None], want[:-1]])
            assert s.changes().tolist() == (want != prev).sum(axis=1).tolist()
            assert np.array_equal(s.labels(), want[-1])


@pytest.mark.parametrize("kw", [dict(), dict(weighted=True), dict(method=G.LAYERED, gamma=(1, 4)),
                                dict(method=G.LAYERED, gamma=(1, 2), weighted=True), dict(method=G.USER),
                                dict(method=G.SLPA, slpa_T=4), dict(frontier=1)])
@pytest.mark.parametrize("tuned", [dict(), dict(pack_max_deg=4, half_max_deg=20, wave_max_deg=40, block_max_deg=300,
                                                hub_chunk=256, part_keys=256), dict(half_max_deg=0),
                                   dict(block_max_deg=8192)])
def test_one_launch_equals_a_launch_per_tier(kw, tuned):
    """Small graphs count all tiers in one launch; timing the tiers one by one
    (profile) takes a launch each.  Degrees on both sides of every tier's
    bound, and a weighted R-MAT graph, with several tier layouts."""
    with G.tuning(**tuned):
        n, edges = tier_boundary_graph(seed=7)
        w = np.random.default_rng(1).integers(1, 9, len(edges)).astype(np.uint32)
        graphs = [G.Graph.rmat(12, 16, seed=9, wmax=8), G.Graph.from_edges(n, edges, w)]
        for g in graphs:
            one = gpu_steps(g, 4, **kw)
            assert_steps_equal(one, gpu_steps(g, 4, profile=True, **kw))


@pytest.mark.parametrize("calls", [[1], [31], [32], [33], [70], [20, 0, 13, 1, 64]])
def test_change_counts_over_many_steps(calls):
    """The change counters of a call's steps are summed together, 32 steps at
    a time: counts and labels for calls around that length, eager and
    replayed, and again after a reset."""
    g = G.Graph.planted(3000, 30, 6.0, 3.0, seed=4)
    off, nbr, _ = g.csr()
    total = sum(calls)
    want = O.classic(off, nbr, total)
    prev = np.vstack([np.arange(g.n, dtype=np.int32)[None], want[:-1]])
    counts = (want != prev).sum(axis=1).tolist()
    with G.Session(g) as s:
        for replay in (False, True, False):
            for k in calls:
                s.step(k, graph=replay)
            assert s.changes().tolist() == counts
            assert np.array_equal(s.labels(), want[-1])
            s.reset()
