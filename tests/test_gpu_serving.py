"""Served admission by free task ids (GPU): with a small task-id pool, the reservation ledger
must hold jobs back; every job still gives the oracle's result, the same as in the batched
run (alone == in the mix), and the job table is reused as a ring when it is smaller than the
stream."""
import numpy as np
import pytest

import gtap_amd
import oracle

pytestmark = pytest.mark.gpu

SMALL_POOL = 768 << 20  # 4.2 M task records of 192 bytes


@pytest.fixture(scope="module", autouse=True)
def runtime():
    gtap_amd.gtap_set_config(timeout_ms=60000, pool_bytes=SMALL_POOL)
    assert gtap_amd.gtap_initialize() == 0
    yield
    assert gtap_amd.gtap_finalize() == 0
    gtap_amd.gtap_set_config()


def expected(st):
    out = []
    for k, p, s in zip(st.kind, st.param, st.key_seed):
        if k == 2:
            out.append(oracle.sort_checksum(np.sort(oracle.gen_keys_u32(int(p), int(s)))))
        else:
            out.append(oracle.job_result(int(k), int(p), int(s)))
    return np.array(out, dtype=np.int64)


def test_admission_holds_jobs_back_and_results_stay_exact():
    st = gtap_amd.Stream(seed=31, njobs=600)
    try:
        exp = expected(st)
        print("case served 600 jobs, small pool, all arriving within ~3 ms", flush=True)
        res, lat, tot, stats = st.serve(rate=200_000.0, arrival_seed=5, max_live=1024)
        assert np.array_equal(res, exp)
        assert stats["admission_holds"] > 0, stats
        assert stats["error_code"] == 0
        print("case batched, same jobs", flush=True)
        res_b, _, _ = st.run_batched()
        assert np.array_equal(res_b, exp)
        print("case served with a 256-slot job ring (max_live 64)", flush=True)
        res_r, lat_r, _, stats_r = st.serve(rate=200_000.0, arrival_seed=6, max_live=64)
        assert np.array_equal(res_r, exp)
        assert stats_r["jobs_taken"] == 600
        assert np.all(lat_r > 0)
    finally:
        st.close()


def test_id_rings_carry_over_launches():
    """The id rings keep their positions from launch to launch; what a launch leaves in them is
    given up by the next one's reset. Served, fork-join, block-mode and failing launches in turn on
    one pool stay exact (a doubled id would break results); the rings' own state is read back in
    test_gpu_overflow_star.py."""
    st = gtap_amd.Stream(seed=47, njobs=200)
    try:
        exp = expected(st)
        for k in range(4):
            print(f"case served, launch {k} on the same rings", flush=True)
            res, _, _, stats = st.serve(rate=100_000.0, arrival_seed=k, max_live=256)
            assert np.array_equal(res, exp) and stats["error_code"] == 0
            v, s = gtap_amd.fib(22 + k)
            assert v == oracle.fib(22 + k) and s["tasks_executed"] == 3 * oracle.fib(23 + k) - 2
            keys = oracle.gen_keys_u32(50_001, k)
            assert np.array_equal(gtap_amd.cilksort(keys)[0], np.sort(keys))
            rp, ci, va = gtap_amd.spmv_random(50000, 4, 1)
            with pytest.raises(gtap_amd.GtapError):  # ends early: queue overflow
                gtap_amd.spmv(rp, ci, va, np.ones(50000), 1000)
    finally:
        st.close()


def test_statistics_rows_are_whole():
    """A launch writes every worker's whole statistics row: nothing of an earlier launch shows."""
    print("case statistics rows of thread, block and thread launches in turn", flush=True)
    _, s0 = gtap_amd.nqueens_cutoff(9, 4)
    _, s1 = gtap_amd.cilksort(oracle.gen_keys_u32(40_000, 3))
    ws = gtap_amd.worker_stats()
    assert ws.shape[0] == s1["workers"] and int(ws[:, 0].sum()) == s1["tasks_executed"]
    assert np.all(ws[:, [8, 9, 10, 13, 14, 15]] == 0)
    v, s2 = gtap_amd.fib(15)
    assert v == oracle.fib(15) and s2["tasks_executed"] == 3 * oracle.fib(16) - 2
