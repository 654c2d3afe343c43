"""The deque overflow ring at 4096-slot deques. A lowered program in which one task spawns n
detached children in one round (gtap_amd/lower/examples/burst.gtap.cu) publishes more than
half of its wave's deque at the round's end, so the wave hands its oldest tasks to the
overflow ring and idle waves take them back: every child runs once (the counters it adds to
are exact) and every task moved to the ring is taken again, launch after launch. A star
graph's BFS with 4 wavefront workers, where the deques fill and drain quickly, stays
bit-exact. Where one wave spawns and the others run, ids pass from wave to wave through the id
rings, whose state between launches is read back."""
import ctypes

import numpy as np
import pytest

import gtap_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def few_workers_small_deques():
    gtap_amd.gtap_set_config(timeout_ms=30000, deque_capacity=4096, blocks=1)
    assert gtap_amd.gtap_initialize() == 0
    yield
    assert gtap_amd.gtap_finalize() == 0
    gtap_amd.gtap_set_config()


@pytest.fixture(scope="module")
def burst_module():
    import ctypes
    from gtap_amd import build as gbuild
    return gtap_amd.EntryModule(gbuild.lowered_lib("burst"), "burst"), ctypes


def ring_counts():
    ws = gtap_amd.worker_stats()
    return int(ws[:, gtap_amd.WORKER_RING_SPILLED].sum()), int(ws[:, gtap_amd.WORKER_RING_TAKEN].sum())


def star(leaves):
    """Vertex 0 with an edge to each of `leaves` vertices that have no out-edges."""
    n = leaves + 1
    row = np.full(n + 1, leaves, dtype=np.int32)
    row[0] = 0
    col = np.arange(1, n, dtype=np.int32)
    return row, col


@pytest.mark.parametrize("queues", [1, 4])
@pytest.mark.parametrize("leaves", [1 << 18, 1 << 20])
def test_star_overflows_into_the_ring(queues, leaves):
    print(f"case bfs star leaves={leaves} queues={queues} split 8, deque capacity 4096, 4 workers", flush=True)
    row, col = star(leaves)
    depth, st = gtap_amd.bfs(row, col, 0, num_queues=queues, split=8)
    assert st["error_code"] == 0
    spilled, taken = ring_counts()
    print(f"ring: {spilled} tasks spilled, {taken} taken", flush=True)
    assert taken == spilled
    expect = np.ones(leaves + 1, dtype=np.int32)
    expect[0] = 0
    assert np.array_equal(depth, expect)
    assert np.array_equal(depth, oracle.bfs(row, col, 0))


def test_joined_program_after_ring_use():
    """A fork-join launch on the same rings after the star runs (positions carried over)."""
    print("case fib(25) after ring use", flush=True)
    v, st = gtap_amd.fib(25)
    assert v == oracle.fib(25) and st["error_code"] == 0


@pytest.mark.parametrize("n", [3050, 2000, 1])
def test_burst_spills_into_the_ring(burst_module, n):
    m, ctypes = burst_module
    u64 = ctypes.c_uint64
    total_spilled = 0
    for rep in range(3):
        print(f"case burst n={n} rep={rep} deque capacity 4096", flush=True)
        m.set_symbol("d_count", 0, u64)
        m.set_symbol("d_sum", 0, u64)
        assert m.launch("burst_kernel", [ctypes.c_int], n) == 0
        assert gtap_amd.gtap_get_runtime_error_code() == 0
        assert m.get_symbol("d_count", u64) == n
        assert m.get_symbol("d_sum", u64) == n * (n - 1) // 2
        spilled, taken = ring_counts()
        print(f"ring: {spilled} tasks spilled, {taken} taken", flush=True)
        assert taken == spilled
        total_spilled += spilled
    if n == 3050:
        # 2986 published at the round's end, past the 2048 half: thieves would have to take
        # 939 of them before the wave's own claim for a launch not to spill
        assert total_spilled > 0


class Rings:
    """The id rings as GtapDev (gtap_amd/csrc/device/gtap_dev.hpp) describes them: the descriptor
    comes to a registered module's setup function at gtap_reset."""
    seen = []

    @staticmethod
    @ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_uint64)
    def setup(desc, nbytes):
        Rings.seen.append(ctypes.string_at(desc, nbytes))
        return 0

    def __init__(self):
        self.seen.clear()
        gtap_amd._check(gtap_amd.lib().gtap_register_entry_module(self.setup), "gtap_register_entry_module")
        assert gtap_amd.lib().gtap_reset() == 0
        words = np.frombuffer(self.seen[-1], dtype=np.uint32)
        pointers = words.view(np.uint64)
        self.pool_seq, self.pool_ctl = int(pointers[3]), int(pointers[4])
        stride, self.ncells, self.n = int(words[34]), int(words[37]), int(words[38])
        assert stride == gtap_amd.gtap_get_config()["record_stride"] and self.n == 8

    def state(self):
        """(enqueue positions, dequeue positions, sequence numbers [ring, cell])."""
        ctl = np.empty(self.n * 32, dtype=np.uint64)
        seq = np.empty((self.n, self.ncells), dtype=np.uint32)
        for a, at in ((ctl, self.pool_ctl), (seq, self.pool_seq)):
            gtap_amd._check(gtap_amd.lib().gtap_memcpy_dtoh(a.ctypes.data, at, a.nbytes), "gtap_memcpy_dtoh")
        low = ctl.view(np.uint32).reshape(self.n, 64)
        return low[:, 0].copy(), low[:, 32].copy(), seq

    def all_free(self):
        enq, deq, seq = self.state()
        cell = np.arange(self.ncells, dtype=np.uint32)
        ok = np.array_equal(enq, deq)
        for r in range(self.n):  # cell of position p is free when it reads p, p from the enqueue position on
            ok = ok and np.array_equal(seq[r], enq[r] + ((cell - enq[r]) & np.uint32(self.ncells - 1)))
        return ok


def hub_chain(hubs, leaves):
    """Hub h points to `leaves` leaves of its own and, last, to hub h + 1; every leaf points back to
    hub 0. One wave goes along the hubs and spawns, the others run the leaves."""
    first = hubs + np.arange(hubs) * leaves  # vertex of each hub's first leaf
    col = np.empty((hubs, leaves + 1), dtype=np.int32)
    col[:, :leaves] = first[:, None] + np.arange(leaves)
    col[:, leaves] = np.arange(1, hubs + 1) % hubs
    n = hubs + hubs * leaves
    row = np.concatenate([np.arange(hubs + 1) * (leaves + 1), hubs * (leaves + 1) + 1 + np.arange(hubs * leaves)])
    depth = np.concatenate([np.arange(hubs), np.repeat(np.arange(hubs) + 1, leaves)]).astype(np.int32)
    assert row.size == n + 1
    return row.astype(np.int32), np.concatenate([col.reshape(-1), np.zeros(hubs * leaves, np.int32)]), depth


@pytest.mark.parametrize("bad", [False, True])
def test_ids_left_in_the_rings_are_given_up_by_the_reset(bad):
    """3 waves free more ids than they can park, so chunks go to the rings; what is left there when
    a launch ends, or is ended by an error, is freed by the next reset, and the positions go on."""
    hubs, leaves = 300, 500
    row, col, expect = hub_chain(hubs, leaves)
    rings = Rings()
    assert rings.all_free()
    passed = left = 0
    for rep in range(3):
        print(f"case id rings bad={bad} rep={rep}", flush=True)
        enq0, _, _ = rings.state()
        if bad:
            broken = col.copy()
            broken[row[hubs - 1] + leaves] = expect.size + 7  # the last hub's last edge
            with pytest.raises(gtap_amd.GtapError):
                gtap_amd.bfs(row, broken, 0, num_queues=1, split=4096)
        else:
            depth, st = gtap_amd.bfs(row, col, 0, num_queues=1, split=4096)
            assert st["error_code"] == 0 and np.array_equal(depth, expect)
        enq, deq, _ = rings.state()
        passed += int((enq - enq0).sum())
        left += int((enq - deq).sum())
        assert gtap_amd.lib().gtap_reset() == 0
        assert rings.all_free()
        assert np.array_equal(rings.state()[0], enq)  # the positions go on
        v, st = gtap_amd.fib(20)
        assert v == oracle.fib(20) and st["tasks_executed"] == 3 * oracle.fib(21) - 2
    print(f"id rings: {passed} chunks passed through, {left} left in them at a launch's end", flush=True)
    assert passed > 0 and left > 0
