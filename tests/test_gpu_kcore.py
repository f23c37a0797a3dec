"""GPU: k-core (kcore_algo_t::compute_shell_index, kcore.hpp:80-268) against the oracle.

Integer work: coreness and the per-epoch log (modified vertices, size of the next
active set) must be bit-exact.  The iteration is Jacobi, so neither depends on the
order in which the device visits vertices; relabeling the graph must not change them
either."""
import numpy as np
import pytest

import oracle
from conftest import golden

pytestmark = pytest.mark.gpu


def _check(g, og, out_edges=False):
    from plato_amd.algo import kcore
    res = kcore(g, out_edges=out_edges)
    core, mod, nxt = oracle.kcore(og, out_edges=out_edges)
    assert np.array_equal(res.coreness, core)
    assert np.array_equal(res.modified, mod) and np.array_equal(res.next_active, nxt)
    assert res.epochs == len(mod)
    return res


def test_hand_worked(ctx):
    from plato_amd import Graph
    s = np.array([0, 1, 2, 2], np.uint32)
    d = np.array([1, 2, 0, 3], np.uint32)
    g = Graph.from_edges(ctx, s, d, 4, directed=False)
    assert _check(g, oracle.CSC(4, s, d, symmetrize=True)).coreness.tolist() == [2, 2, 2, 1]
    s = np.array([0, 1, 2, 4, 5], np.uint32)
    d = np.array([2, 2, 3, 3, 4], np.uint32)
    g = Graph.from_edges(ctx, s, d, 6, build_csr=True)
    og = oracle.CSC(6, s, d)
    assert _check(g, og).coreness.tolist() == [0, 0, 2, 1, 1, 0]
    assert _check(g, og, out_edges=True).coreness.tolist() == [1, 1, 1, 0, 1, 1]


def test_reference_fixtures(ctx):
    from plato_amd import Graph
    for name in ("v100_e2150_ua_c3.csv", "v100_e4300_da_c3.csv", "graph_10_9.csv",
                 "complete_binary_tree_10_9.csv", "kcore_test_7_11.csv"):
        s, d = oracle.read_edge_csv(golden(name))
        V = int(max(s.max(), d.max())) + 1
        for directed in (True, False):
            print(f"case: kcore {name} directed={directed}", flush=True)
            g = Graph.from_edges(ctx, s, d, V, directed=directed, build_csr=True)
            og = oracle.CSC(V, s, d, symmetrize=not directed)
            _check(g, og)
            if directed:
                _check(g, og, out_edges=True)
            g.close()


@pytest.mark.parametrize("scale,directed", [(12, True), (14, False), (16, False), (18, False)])
def test_rmat_bit_exact(ctx, scale, directed):
    """RMAT graphs with their duplicates and self-loops; hubs go through the wave-per-vertex
    pass (and, at scale 18, its search above the 1024-bin histogram in the first epochs)."""
    from plato_amd import Graph
    print(f"case: kcore rmat s{scale} directed={directed}", flush=True)
    s, d = oracle.rmat_edges(scale, 16, 7)
    g = Graph.rmat(ctx, scale, 16, seed=7, directed=directed, build_csr=True)
    og = oracle.CSC(1 << scale, s, d, symmetrize=not directed)
    res = _check(g, og)
    if directed:
        _check(g, og, out_edges=True)
    assert res.coreness.max() > 0
    g.close()
    gr = Graph.rmat(ctx, scale, 16, seed=7, directed=directed, relabel=True)
    assert np.array_equal(_check(gr, og).coreness, res.coreness)
    gr.close()


def test_big_vertex_search_above_histogram(ctx):
    """A clique of 1100 vertices (coreness 1099, above the wave pass's 1024 histogram
    bins, so the block pass takes them) plus a tail."""
    from plato_amd import Graph
    n = 1100
    a, b = np.triu_indices(n, 1)
    s = np.concatenate([a, [0, n, n + 1]]).astype(np.uint32)
    d = np.concatenate([b, [n, n + 1, n + 2]]).astype(np.uint32)
    V = n + 3
    g = Graph.from_edges(ctx, s, d, V, directed=False)
    res = _check(g, oracle.CSC(V, s, d, symmetrize=True))
    assert res.coreness[:n].tolist() == [n - 1] * n and res.coreness[n:].tolist() == [1, 1, 1]


def test_giant_hub(ctx):
    """A vertex of 70000 neighbours (above the 65536 at which its adjacency is cut into
    chunks whose histograms add up in global memory), on a wheel whose rim carries random
    chords, so the hub's h-index moves over several epochs; directed and relabeled too."""
    from plato_amd import Graph
    rim = 70000
    rng = np.random.default_rng(8)
    r = np.arange(1, rim + 1, dtype=np.uint32)
    chord_a = rng.integers(1, rim + 1, 3 * rim).astype(np.uint32)
    chord_b = rng.integers(1, rim + 1, 3 * rim).astype(np.uint32)
    s = np.concatenate([np.zeros(rim, np.uint32), r, chord_a])
    d = np.concatenate([r, r % rim + 1, chord_b])
    V = rim + 1
    print(f"case: kcore giant hub V={V} E={len(s)}", flush=True)
    og = oracle.CSC(V, s, d, symmetrize=True)
    assert int(np.diff(og.col_ptr)[0]) > 65536
    res = _check(Graph.from_edges(ctx, s, d, V, directed=False), og)
    assert res.coreness[0] >= 3
    _check(Graph.from_edges(ctx, s, d, V, directed=False, relabel=True), og)
    # directed: the hub's 70000 in-edges come from the rim's reversed edges
    s2, d2 = np.concatenate([s, r]), np.concatenate([d, np.zeros(rim, np.uint32)])
    _check(Graph.from_edges(ctx, s2, d2, V, build_csr=True), oracle.CSC(V, s2, d2))


@pytest.mark.parametrize("n,mult", [(22, 820), (18, 965), (80, 1000)])
@pytest.mark.parametrize("directed", [False, True])
def test_answers_above_the_block_histogram(ctx, n, mult, directed):
    """n vertices joined pairwise by 0.9 to 1.1 * mult parallel edges: h-indices around and
    above the 16384 bins of the block pass (18 * 965 straddles them), which take a second
    round over a value range, in one block per vertex and (n = 80) in chunks."""
    from plato_amd import Graph
    rng = np.random.default_rng(n)
    a, b = np.triu_indices(n, 1)
    m = rng.integers(int(mult * 0.9), int(mult * 1.1), a.size)
    s, d = np.repeat(a, m).astype(np.uint32), np.repeat(b, m).astype(np.uint32)
    if directed:
        s, d = np.concatenate([s, d]), np.concatenate([d, s])
    V = n + 1
    print(f"case: kcore multigraph n={n} mult={mult} directed={directed}", flush=True)
    g = Graph.from_edges(ctx, s, d, V, directed=directed, build_csr=True)
    res = _check(g, oracle.CSC(V, s, d, symmetrize=not directed))
    if n * mult > 15000:
        assert res.coreness.max() > 14000
    g.close()


@pytest.mark.parametrize("length", [64, 65, 1024, 1025, 4096, 4097, 65536, 65537])
@pytest.mark.parametrize("directed", [False, True])
def test_adjacency_length_classes(ctx, length, directed):
    """Eight vertices of exactly `length` neighbours (the last of one pass and the first of the
    next) over a random graph, so their values move over several epochs."""
    from plato_amd import Graph
    rng = np.random.default_rng(length)
    rim, hubs = max(4 * length // 3, 200), 8
    s = np.concatenate([np.full(length, rim + h) for h in range(hubs)] + [rng.integers(0, rim, 6 * rim)])
    d = np.concatenate([rng.choice(rim, length, replace=False) for _ in range(hubs)] + [rng.integers(0, rim, 6 * rim)])
    s, d = s.astype(np.uint32), d.astype(np.uint32)
    if directed:
        s, d = np.concatenate([s, d]), np.concatenate([d, s])
    V = rim + hubs
    og = oracle.CSC(V, s, d, symmetrize=not directed)
    assert int(np.diff(og.col_ptr)[rim]) == length
    print(f"case: kcore length={length} directed={directed}", flush=True)
    g = Graph.from_edges(ctx, s, d, V, directed=directed, relabel=length % 2 == 1)
    _check(g, og)
    g.close()


@pytest.mark.parametrize("length", [60, 64, 1500, 4096, 5000, 40000])
def test_values_that_fall_epoch_after_epoch(ctx, length):
    """Hubs of `length` neighbours over a skewed rim: they drop in several epochs running, so the
    value of a drop comes from the previous epoch's walk in the pass of each adjacency length."""
    from plato_amd import Graph
    rng = np.random.default_rng(length)
    rim, hubs = max(2 * length, 300), 6
    m = 12 * rim
    s = np.concatenate([np.full(length, rim + h) for h in range(hubs)] + [(rim * rng.random(m) ** 3).astype(np.int64)])
    d = np.concatenate([rng.choice(rim, length, replace=False) for _ in range(hubs)]
                       + [(rim * rng.random(m) ** 2).astype(np.int64)])
    s, d = s.astype(np.uint32), d.astype(np.uint32)
    V = rim + hubs
    print(f"case: kcore falling values length={length}", flush=True)
    g = Graph.from_edges(ctx, s, d, V, directed=False)
    _check(g, oracle.CSC(V, s, d, symmetrize=True))
    g.close()


def _lengths(length):
    rng = np.random.default_rng(length)
    rim, hubs = max(4 * length // 3, 200), 8
    s = np.concatenate([np.full(length, rim + h) for h in range(hubs)] + [rng.integers(0, rim, 6 * rim)])
    d = np.concatenate([rng.choice(rim, length, replace=False) for _ in range(hubs)] + [rng.integers(0, rim, 6 * rim)])
    return rim + hubs, s, d


def _falling(length):
    rng = np.random.default_rng(length)
    rim, hubs = max(2 * length, 300), 6
    m = 12 * rim
    s = np.concatenate([np.full(length, rim + h) for h in range(hubs)] + [(rim * rng.random(m) ** 3).astype(np.int64)])
    d = np.concatenate([rng.choice(rim, length, replace=False) for _ in range(hubs)]
                       + [(rim * rng.random(m) ** 2).astype(np.int64)])
    return rim + hubs, s, d


def _multi(n):
    a, b = np.triu_indices(n, 1)
    m = np.random.default_rng(n).integers(870, 1060, a.size)
    return n + 1, np.repeat(a, m), np.repeat(b, m)


def _giant(rim):
    rng = np.random.default_rng(8)
    r = np.arange(1, rim + 1)
    chords = rng.integers(1, rim + 1, (2, 3 * rim))
    return rim + 1, np.concatenate([np.zeros(rim, int), r, chords[0]]), np.concatenate([r, r % rim + 1, chords[1]])


@pytest.mark.parametrize("make,size", [(_lengths, n) for n in (64, 65, 1025, 4096, 4097, 65536, 65537)]
                         + [(_falling, n) for n in (60, 1500, 5000, 40000)] + [(_multi, 18), (_multi, 80), (_giant, 70000)])
def test_byte_marks_with_counts(ctx, make, size):
    """The form that symmetrized graphs of 2^31 entries and more take (counts, and the active
    marks as bytes), on graphs of every adjacency class with values that fall over several
    epochs: coreness and log against the oracle, and the marks in the values beside it."""
    import ctypes as C
    from plato_amd import Graph
    from plato_amd._lib import KcoreStats, check
    V, s, d = make(size)
    s, d = s.astype(np.uint32), d.astype(np.uint32)
    core, mod, nxt = oracle.kcore(oracle.CSC(V, s, d, symmetrize=True))
    for relabel in (False, True):
        print(f"case: kcore byte marks {make.__name__} {size} relabel={relabel}", flush=True)
        g = Graph.from_edges(ctx, s, d, V, directed=False, relabel=relabel)
        for limit in (0, g.nnz, g.nnz + 1, 1 << 63):  # bytes, bytes, values, values (2^31 at most)
            got, m, n, st = np.zeros(V, np.uint32), np.zeros(4096, np.uint64), np.zeros(4096, np.uint64), KcoreStats()
            check(g.lib.pe_kcore_byte_marks(g.h, 0, limit, got.ctypes.data, m.ctypes.data, n.ctypes.data, 4096,
                                            C.byref(st)), ctx.h)
            assert np.array_equal(got, core)
            assert np.array_equal(m[:st.epochs], mod) and np.array_equal(n[:st.epochs], nxt)
        g.close()
