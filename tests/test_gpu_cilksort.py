"""Block-cooperative cilksort through the C ABI on the GPU: the sorted keys are bit-exact
against an independent sort (numpy) and the oracle's cilksort restatement."""
import numpy as np
import pytest

import gtap_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def runtime():
    gtap_amd.gtap_set_config(timeout_ms=20000)
    assert gtap_amd.gtap_initialize() == 0
    yield
    assert gtap_amd.gtap_finalize() == 0


@pytest.mark.parametrize("n", [0, 1, 2, 3, 100, 4095, 4096, 4097, 16384, 16385, 65537, 262147, 1000003])
def test_cilksort_sizes(n):
    print(f"case cilksort n={n}", flush=True)
    keys = oracle.gen_keys_u32(n, seed=1000 + n)
    out, st = gtap_amd.cilksort(keys)
    assert np.array_equal(out, np.sort(keys))
    assert st["error_code"] == 0


@pytest.mark.parametrize("leaf,merge_leaf", [(64, 256), (4096, 4096), (1, 3), (4096, 1 << 20)])
def test_cilksort_cutoffs(leaf, merge_leaf):
    print(f"case cilksort leaf={leaf} merge_leaf={merge_leaf}", flush=True)
    rng = np.random.default_rng(leaf * 7 + merge_leaf)
    for keys in (rng.integers(0, 2**32, 200003, dtype=np.uint64).astype(np.uint32),
                 rng.integers(0, 5, 100000).astype(np.uint32),
                 np.arange(70000, dtype=np.uint32)[::-1].copy()):
        out, _ = gtap_amd.cilksort(keys, leaf=leaf, merge_leaf=merge_leaf)
        assert np.array_equal(out, np.sort(keys))
        assert np.array_equal(out, oracle.cilksort_u32(keys, leaf, merge_leaf))


def sort_nodes(n, leaf):
    """Ranges of the sort tree above `leaf` keys, each of which spawns 4 sorts and 3 merges."""
    if n <= leaf:
        return 0
    h = n // 2
    return 1 + sum(sort_nodes(k, leaf) for k in (h // 2, h - h // 2, (n - h) // 2, n - h - (n - h) // 2))


@pytest.mark.parametrize("n", [70_003, 200_003, (2 << 20) + 3])
def test_cilksort_obeys_the_largest_merge(n):
    """A merge_leaf that the caller gives is taken as it is: with one of n no merge is cut, however
    many tiles it has; the default cuts them."""
    print(f"case cilksort merge_leaf of the caller, n={n}", flush=True)
    keys = oracle.gen_keys_u32(n, n)
    out, st = gtap_amd.cilksort(keys, leaf=1024, merge_leaf=n)
    assert np.array_equal(out, np.sort(keys))
    assert st["tasks_spawned"] == 7 * sort_nodes(n, 1024)
    out, st = gtap_amd.cilksort(keys, leaf=1024)
    assert np.array_equal(out, np.sort(keys))
    assert st["tasks_spawned"] > 7 * sort_nodes(n, 1024)


def test_cilksort_benchmark_keys():
    n = 1 << 26
    print(f"case cilksort benchmark n={n}", flush=True)
    keys = gtap_amd.gen_keys(n)  # gen_vector keys, seed 123456789
    out, st = gtap_amd.cilksort(keys)
    assert np.array_equal(out, np.sort(keys))


@pytest.mark.parametrize("n", [7, 256, 2047, 2048, 2049, 4096, 4097, 8191, 8192, 8193, 16384, 32768, 32769, 40_000])
@pytest.mark.parametrize("leaf", [4096, 2048, 3000])
def test_cilksort_leaf_sizes(n, leaf):
    """Leaf sorts of 8, 16 and 32 keys a thread at their limits, keys equal to the padding value,
    runs in both directions and ties."""
    print(f"case cilksort leaf sizes n={n} leaf={leaf}", flush=True)
    rng = np.random.default_rng(n + leaf)
    for keys in (rng.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32),
                 np.full(n, 0xFFFFFFFF, dtype=np.uint32),
                 np.where(rng.random(n) < 0.5, 0xFFFFFFFF, 0).astype(np.uint32),
                 np.arange(n, dtype=np.uint32)[::-1].copy(),
                 rng.integers(0, 3, n).astype(np.uint32)):
        out, _ = gtap_amd.cilksort(keys, leaf=leaf)
        assert np.array_equal(out, np.sort(keys))


@pytest.mark.parametrize("n", [(2 << 20) + 1, (8 << 20), (8 << 20) + 1, (32 << 20) + 5])
def test_cilksort_size_rules(n):
    """One size on each side of the rules that choose the largest merge and the kernel build."""
    print(f"case cilksort size rules n={n}", flush=True)
    keys = np.random.default_rng(n).integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32)
    out, _ = gtap_amd.cilksort(keys)
    assert np.array_equal(out, np.sort(keys))


@pytest.mark.parametrize("n", [256, 2049, 4096, 4097, 8191, 8192, 8193, 16385, 32769, 40_000])
@pytest.mark.parametrize("leaf", [0, 4096, 4095, 2048])
def test_cilksort_obeys_the_leaf(n, leaf):
    """A leaf that the caller gives is taken as it is, 4096 too; the default sorts ranges of up to 8192
    keys whole. (merge_leaf = n: no merge is cut, so the spawns are those of the sort tree.)"""
    print(f"case cilksort leaf of the caller, n={n} leaf={leaf}", flush=True)
    rng = np.random.default_rng(n + leaf)
    for keys in (rng.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32),
                 np.where(rng.random(n) < 0.5, 0xFFFFFFFF, 0).astype(np.uint32),
                 np.arange(n, dtype=np.uint32)[::-1].copy(),
                 rng.integers(0, 3, n).astype(np.uint32)):
        out, st = gtap_amd.cilksort(keys, leaf=leaf, merge_leaf=n)
        assert np.array_equal(out, np.sort(keys))
        assert st["tasks_spawned"] == 7 * sort_nodes(n, leaf or 8192)


def test_cilksort_refuses_larger_leaves():
    print("case cilksort leaf=4097 (refused)", flush=True)
    with pytest.raises(gtap_amd.GtapError):
        gtap_amd.cilksort(np.arange(10, dtype=np.uint32), leaf=4097)
