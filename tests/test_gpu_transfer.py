"""GPU: transfers between device vectors and host arrays at the edges of their chunks (small
ones go through the runtime, one slot, the calling thread alone, worker threads, several
rounds of the ring of eight 2 MiB slots), plain, widened and reordered, and on two contexts
at once.  The data must arrive bit for bit."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SLOT = (2 << 20) // 4  # elements of 4 bytes
SIZES = [1, 65536, 65537, SLOT - 1, SLOT, SLOT + 1, 3 * SLOT, 3 * SLOT + 1, 8 * SLOT + 5, 25 * SLOT + 77]


def _round_trip(ctx, n, seed):
    from plato_amd import DenseState
    rng = np.random.default_rng(seed)
    for dt in (np.uint32, np.float32, np.float64):
        a = rng.integers(0, 1 << 30, n).astype(dt)
        v = DenseState(ctx, n, dt)
        v.upload(a)
        assert np.array_equal(v.numpy(), a)
        assert np.array_equal(v.to_f64(), a.astype(np.float64))
        v.close()


@pytest.mark.parametrize("n", SIZES)
def test_round_trip(ctx, n):
    print(f"case: transfer n={n}", flush=True)
    _round_trip(ctx, n, n)


@pytest.mark.parametrize("V", [1, 70001, SLOT, SLOT + 1, 4 * SLOT + 3])
def test_reordered_and_widened(ctx, V):
    """A relabeled graph's out-degrees, its permutation and its ranks after no iteration."""
    from plato_amd import Graph
    from plato_amd.algo import pagerank, pagerank_opts_t
    rng = np.random.default_rng(V)
    s = rng.integers(0, V, 2 * V).astype(np.uint32)
    d = rng.integers(0, V, 2 * V).astype(np.uint32)
    od = np.bincount(s, minlength=V)
    print(f"case: transfer relabeled V={V}", flush=True)
    for relabel in (False, True):
        g = Graph.from_edges(ctx, s, d, V, relabel=relabel)
        assert np.array_equal(g.out_degrees(), od.astype(np.uint32))
        rank_of = g.permutation()
        assert np.array_equal(np.sort(rank_of), np.arange(V, dtype=np.uint32))
        assert relabel == bool(g.info.relabeled)
        got = pagerank(g, pagerank_opts_t(0, 0.85, 0.0)).rank
        want = (1.0 / np.maximum(od, 1).astype(np.float64)).astype(np.float32).astype(np.float64)
        assert np.array_equal(got, want)
        g.close()


def test_two_contexts_in_two_threads(ctx):
    from plato_amd import Context
    errors = []

    def work(seed):
        try:
            with Context(0) as c:
                for n in (SLOT + 1, 9 * SLOT + 3):
                    _round_trip(c, n, seed)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("direction", ["download", "upload"])
def test_waiting_for_queued_work_costs_one_core(ctx, direction):
    """A transfer behind device work that is still running: only the calling thread (and the
    runtime's own) may be busy until the work is done."""
    import time
    from plato_amd import DenseState
    a, b, v = (DenseState(ctx, n, np.float32) for n in (1 << 29, 1 << 29, 1 << 23))
    host = np.arange(v.n, dtype=np.float32)
    v.upload(host)

    def timed(copies):
        for _ in range(copies):
            a.copy_from(b)  # 2 GiB, left running
        t, c = time.perf_counter(), time.process_time()
        if direction == "download":
            assert np.array_equal(v.numpy(), host)
        else:
            v.upload(host)
        return time.perf_counter() - t, time.process_time() - c

    alone, _ = timed(0)
    wall, cpu = timed(300)
    print(f"case: transfer behind work {direction}: {wall * 1e3:.0f} ms ({alone * 1e3:.1f} alone), {cpu * 1e3:.0f} ms of CPU", flush=True)
    assert wall > 0.1 and wall > 5 * alone  # it did wait
    assert cpu < 2.5 * wall
    assert np.array_equal(v.numpy(), host)
    for x in (a, b, v):
        x.close()


# results of up to 16384 words come by mail: its ends in 4- and 8-byte elements, and a count that
# gives each of the kernel's 1024 threads more than one
MAIL_SIZES = [2, 1023, 1024, 1025, 8191, 8192, 8193, 16383, 16384, 16385, 32768, 32769]


@pytest.mark.parametrize("n", MAIL_SIZES)
def test_small_results(ctx, n):
    print(f"case: small transfer n={n}", flush=True)
    _round_trip(ctx, n, n)


@pytest.mark.parametrize("V", MAIL_SIZES)
def test_small_reordered(ctx, V):
    test_reordered_and_widened(ctx, V)
