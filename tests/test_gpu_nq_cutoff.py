"""n-queens at the reference's benchmark settings (evaluation/2-comparison/nq/gtap_nq.cu:10-99:
tasks to row `cutoff`, sequential search below, no taskwait, one counter) gives the
solution counts of the oracle for every cutoff, including cutoffs at or beyond N."""
import pytest

import gtap_amd as G
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def runtime():
    G.gtap_set_config(timeout_ms=30000)
    assert G.gtap_initialize() == 0
    yield
    assert G.gtap_finalize() == 0


@pytest.mark.parametrize("n", [1, 4, 6, 8, 10, 12, 13])
def test_cutoff_counts(n):
    for cutoff in (0, 3, 7, n - 1, n, n + 2):
        if cutoff < 0:
            continue
        print(f"case nq cutoff n={n} cutoff={cutoff}", flush=True)
        v, s = G.nqueens_cutoff(n, cutoff)
        assert v == O.nq(n)[0]


def test_cutoff_nq14_reference_setting():
    print("case nq cutoff n=14 cutoff=7", flush=True)
    v, s = G.nqueens_cutoff(14, 7)
    assert v == 365596


@pytest.mark.parametrize("n", [2, 3, 5, 9, 11])
def test_cutoff_walk_depths(n):
    """The sequential walk from every depth (none of it to all of it: it starts in row
    cutoff + 1), with its last-row count; the worker counts add up to the result."""
    for cutoff in range(n):
        print(f"case nq cutoff walk n={n} cutoff={cutoff}", flush=True)
        v, _ = G.nqueens_cutoff(n, cutoff)
        assert v == O.nq(n)[0]
        assert int(G.worker_stats()[:, 15].sum()) == v


def test_cutoff_largest_board():
    print("case nq cutoff n=16 (diagonal sets of 31 bits)", flush=True)
    assert G.nqueens_cutoff(16, 9)[0] == 14772512
