"""SpMV (examples/spmv/spmv_thread.cu:34-66), the binary-tree workload
(examples/binary_tree/binary_tree_thread.cu:63-120) and the block-mode BFS
(examples/asynchronous_bfs/asynchronous_bfs_block.cu:17-37) on the GPU, bit-exact against
the oracle; a graph read from a file in the reference's CSR format through BFS."""
import numpy as np
import pytest

import gtap_amd as G
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def runtime():
    G.gtap_set_config(timeout_ms=20000)
    assert G.gtap_initialize() == 0
    yield
    assert G.gtap_finalize() == 0


@pytest.mark.parametrize("rows,avg,cutoff", [(1, 3, 16), (17, 5, 16), (1000, 8, 16), (50000, 24, 16),
                                             (50000, 24, 1), (50000, 24, 200), (200000, 300, 16)])
def test_spmv_matches_oracle(rows, avg, cutoff):
    print(f"case spmv rows={rows} avg={avg} cutoff={cutoff}", flush=True)
    rp, ci, va = G.spmv_random(rows, avg, rows + avg)
    x = np.random.default_rng(rows).uniform(-2, 2, rows)
    y, s = G.spmv(rp, ci, va, x, cutoff)
    assert np.array_equal(y, O.spmv(rp, ci, va, x))
    # one task per row plus the range tasks (a binary split of [0, rows) down to <= cutoff rows)
    assert s["tasks_executed"] >= rows


def test_spmv_range_cutoff_beyond_deque_capacity_is_reported():
    # 64 lanes each spawning up to 1000 row tasks in one round need more deque slots than
    # gtap_config.deque_capacity provides beyond the published tasks: a round's children stay
    # private until the round ends, so the launch ends with a queue-overflow error (the
    # reference's GTAP_MAX_TASKS_PER_WARP trap), and the next launch runs normally
    print("case spmv cutoff 1000 (queue overflow reported)", flush=True)
    rp, ci, va = G.spmv_random(50000, 4, 1)
    x = np.ones(50000)
    with pytest.raises(G.GtapError) as e:
        G.spmv(rp, ci, va, x, 1000)
    assert "QUEUE_OVERFLOW" in str(e.value)
    y, _ = G.spmv(rp, ci, va, x, 16)
    assert np.array_equal(y, O.spmv(rp, ci, va, x))


def test_spmv_empty_rows_and_zero_matrix():
    print("case spmv empty rows", flush=True)
    rp = np.array([0, 0, 2, 2, 3, 3], dtype=np.int32)
    ci = np.array([0, 4, 2], dtype=np.int32)
    va = np.array([1.5, -2.0, 3.0])
    x = np.array([2.0, 9.0, 1.0, 9.0, 0.25])
    y, _ = G.spmv(rp, ci, va, x)
    assert y.tolist() == [0.0, 1.5 * 2.0 - 2.0 * 0.25, 0.0, 3.0, 0.0]
    y0, _ = G.spmv(np.zeros(8, dtype=np.int32), np.zeros(0, dtype=np.int32), np.zeros(0), np.ones(7))
    assert np.all(y0 == 0.0)


@pytest.mark.parametrize("lengths", [[0, 1, 7, 8, 9], [15, 16, 17, 31, 32, 33], [63, 64, 65, 127, 128, 129],
                                     [511, 512, 513, 1, 0], [5000], [0], [100, 3] * 40, [300] * 70, [1] * 1000])
@pytest.mark.parametrize("cutoff", [1, 16, 500])
def test_spmv_row_lengths(lengths, cutoff):
    """Rows whose lengths meet the edges of a step (8 entries for each of a row's 1 to 64 lanes),
    few and many in a batch, and the batch sizes of short and long mean rows."""
    print(f"case spmv lengths {lengths[:6]} x {len(lengths)} cutoff={cutoff}", flush=True)
    rng = np.random.default_rng(len(lengths) + cutoff)
    cols = max(max(lengths), 40)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(cols, k, replace=False)) for k in lengths] + [[]]).astype(np.int32)
    va = rng.uniform(-1, 1, ci.size)
    x = rng.uniform(-2, 2, cols)
    x[0] = np.inf  # an entry that no row uses by accident: padding must not be multiplied in
    ci[ci == 0] = 1
    y, _ = G.spmv(rp, ci, va, x, cutoff)
    assert np.array_equal(y, O.spmv(rp, ci, va, x))


def test_spmv_bad_column_is_reported():
    print("case spmv bad column", flush=True)
    rp, ci, va = G.spmv_random(500, 30, 3)
    for bad in (-1, 500, 2**31 - 1):
        c = ci.copy()
        c[len(c) // 2] = bad
        with pytest.raises(G.GtapError) as e:
            G.spmv(rp, c, va, np.ones(500))
        assert "INVALID_ARGUMENT" in str(e.value)
    assert np.array_equal(G.spmv(rp, ci, va, np.ones(500))[0], O.spmv(rp, ci, va, np.ones(500)))


@pytest.mark.parametrize("avg,row,at", [(3, 0, 0), (3, 399, 1), (30, 250, 20), (200, 77, 0), (200, 300, 150), (900, 2, 700)])
def test_spmv_bad_column_report_names_task_and_row(avg, row, at):
    """Rows of 1 to 64 lanes and of several steps; the entry's offset is not the row."""
    print(f"case spmv bad column report avg={avg} row={row} at={at}", flush=True)
    n = 400
    lengths = np.full(n, avg)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    ci = np.tile(np.arange(avg, dtype=np.int32), n)
    ci[rp[row] + at] = 1000
    with pytest.raises(G.GtapError) as e:
        G.spmv(rp, ci, np.ones(ci.size), np.ones(1000), 1000)
    r = e.value.report
    assert e.value.code == 11 and r["valid"] == 1
    assert r["value"] == row and r["limit"] == 1000 and r["tid"] > 0


@pytest.mark.parametrize("height,mem_ops,iters", [(0, 4, 4), (1, 0, 0), (5, 64, 512), (10, 16, 32), (15, 64, 512),
                                                  (12, 0, 1000)])
def test_tree_matches_oracle(height, mem_ops, iters):
    print(f"case tree height={height} mem_ops={mem_ops} iters={iters}", flush=True)
    inp = G.tree_input(1 << 16, height + 1)
    out, s = G.tree(height, mem_ops, iters, inp)
    nodes = (1 << (height + 1)) - 1
    assert out.size == nodes
    assert np.array_equal(out, O.tree(height, mem_ops, iters, inp))
    assert s["tasks_spawned"] == nodes - 1


@pytest.mark.parametrize("height", [0, 2, 3, 6])
@pytest.mark.parametrize("mem_ops,iters", [(1, 1), (3, 63), (31, 64), (32, 65), (33, 0), (255, 7), (256, 8), (257, 129)])
def test_tree_lane_groups(height, mem_ops, iters):
    """A node's reads and steps are divided among 64 / m lanes (m nodes in the round, up to 8
    here): counts around the groups' step of 4 reads a lane and around whole steps."""
    print(f"case tree groups height={height} mem_ops={mem_ops} iters={iters}", flush=True)
    inp = G.tree_input(1 << 12, 7) * 1e6
    out, _ = G.tree(height, mem_ops, iters, inp)
    assert np.array_equal(out, O.tree(height, mem_ops, iters, inp))


@pytest.mark.parametrize("height,mem_ops,iters", [(16, 2, 8), (17, 2, 8), (16, 32, 0), (17, 32, 0), (17, 20, 640)])
def test_tree_batch_sizes(height, mem_ops, iters):
    """One size on each side of the rule that picks 8, 16 or 32 nodes a batch."""
    print(f"case tree batches height={height} mem_ops={mem_ops} iters={iters}", flush=True)
    inp = G.tree_input(1 << 16, height)
    out, s = G.tree(height, mem_ops, iters, inp)
    assert np.array_equal(out, O.tree(height, mem_ops, iters, inp))
    assert s["tasks_executed"] == 3 * (1 << height) - 2


def test_tree_most_steps():
    """One node with the most steps the argument holds: the lanes' walks (64 steps apart) end past
    2^31 - 1."""
    iters = 2**31 - 1
    print(f"case tree height=0 iters={iters}", flush=True)
    inp = G.tree_input(16, 3)
    out, s = G.tree(0, 3, iters, inp)
    assert s["error_code"] == 0 and np.array_equal(out, O.tree(0, 3, iters, inp))


def test_bfs_on_graph_read_from_reference_format(tmp_path):
    print("case bfs from a CSR file", flush=True)
    row, col = G.rmat_csr(14, 8, 5)
    p = str(tmp_path / "graph.bin")
    G.write_csr(p, row, col)
    r2, c2 = G.read_csr(p)
    depth, _ = G.bfs(r2, c2, 0, 4, 64)
    assert np.array_equal(depth, O.bfs(row, col, 0))


@pytest.mark.parametrize("scale,ef", [(8, 4), (14, 8), (18, 16)])
def test_block_bfs_matches_oracle(scale, ef):
    print(f"case block bfs rmat scale={scale} ef={ef}", flush=True)
    row, col = G.rmat_csr(scale, ef, scale)
    depth, s = G.bfs_block(row, col, 0)
    assert np.array_equal(depth, O.bfs(row, col, 0))


def test_block_bfs_chain_and_star():
    print("case block bfs chain and star", flush=True)
    n = 3000
    row = np.concatenate([np.arange(n), [n - 1]]).astype(np.int32)  # chain 0 -> 1 -> ... (the reference's default graph)
    col = np.arange(1, n, dtype=np.int32)
    depth, _ = G.bfs_block(row, col, 0)
    assert depth.tolist() == list(range(n))
    star_row = np.array([0, 5000] + [5000] * 5000, dtype=np.int32)  # vertex 0 -> 1..5000
    star_col = np.arange(1, 5001, dtype=np.int32)
    depth, _ = G.bfs_block(star_row, star_col, 0)
    assert depth[0] == 0 and np.all(depth[1:] == 1)
