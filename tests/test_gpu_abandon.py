"""GPU fused scan with abandoned tiles: a 64-vector tile is dropped when its partial sums after a quarter or half of the
sub-spaces already exceed every query's admission bound, the bounds shared between the waves of a block and the blocks
of a slab. Results must stay those of the oracle, bit for bit, for clustered codes (most tiles dropped), uniform codes
(hardly any), exact ties at the bound, distances that overflow to infinity, padded query slots, and repeated searches
of one searcher with changing shapes (the shared bounds return to their initial state).
"""
import numpy as np
import pytest

import veckern_amd as vk
from tests import datagen
from oracle import binding as orc

pytestmark = pytest.mark.gpu

V8, V9 = vk.ScanVariant.FusedWarp, vk.ScanVariant.FusedWarpF16


def assert_same(got_d, got_i, exp, label):
    bad = np.argwhere((got_i != exp["id"]) | (got_d.view(np.uint32) != exp["dist"].view(np.uint32)))
    assert not bad.size, f"{label}: {len(bad)} mismatches, first at {bad[0]}"


def fixture(family, n, d, m, nq):
    if family == "clusters":
        return datagen.pq_fixture(n, d, m, nq, seed=900 + m)
    if family == "uniform":
        return datagen.random_fixture(n, d, m, nq, seed=901 + m)
    if family == "ties":
        return datagen.tie_fixture(n, d, m, nq, seed=902 + m)
    cent, codes, queries = datagen.pq_fixture(n, d, m, nq, seed=903 + m)
    cent[:, 5:60] *= np.float32(1e19)  # squares overflow: infinite distances among finite ones
    return cent, codes, queries


@pytest.mark.parametrize("family", ["clusters", "uniform", "ties", "overflow"])
@pytest.mark.parametrize("d,m", [(64, 16), (64, 32), (96, 48), (128, 64)])
def test_abandoned_tiles_match_oracle(family, d, m):
    n, nq = 140_003, 21  # at 1 to 4 blocks per slab, enough vectors per block for these scans
    cent, codes, queries = fixture(family, n, d, m, nq)
    with vk.PQSearcher(cent, codes, d) as s:
        for q, threads, blocks in [(1, 256, 4), (2, 1024, 2), (4, 512, 1), (4, 256, 3), (8, 1024, 3), (4, 256, 0)]:
            s.set_tuning(vk.Tuning(queries_per_block=q, scan_threads=threads, blocks_per_query=blocks))
            for k, count in [(1, nq), (10, 1), (64, 5), (100, nq)]:
                got_d, got_i, _ = s.search(queries[:count], k, V8)
                assert_same(got_d, got_i, orc.adc_search(cent, d, codes, queries[:count], k),
                            f"v8 Q={q} threads={threads} blocks={blocks} k={k} nq={count}")
            got_d, got_i, _ = s.search(queries, 10, V9)
            assert_same(got_d, got_i, orc.adc_search_f16(cent, d, codes, queries, 10), f"v9 Q={q} threads={threads}")


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 4097])
def test_abandoned_tiles_small_databases(n):
    cent, codes, queries = datagen.random_fixture(n, 64, 16, 5, seed=910 + n)
    with vk.PQSearcher(cent, codes, 64) as s:
        for k in (1, min(n, 100)):
            got_d, got_i, _ = s.search(queries, k, V8)
            assert_same(got_d, got_i, orc.adc_search(cent, 64, codes, queries, k), f"n={n} k={k}")


def test_single_query_over_many_blocks_repeats():
    cent, codes, queries = datagen.pq_fixture(600_000, 64, 16, 4, seed=920)
    exp = orc.adc_search(cent, 64, codes, queries, 10)
    with vk.PQSearcher(cent, codes, 64) as s:
        s.set_tuning(vk.Tuning(queries_per_block=4, blocks_per_query=12))
        for r in range(12):  # each search starts without the bounds of the one before
            q = r % 4
            got_d, got_i, _ = s.search(queries[q:q + 1], 10, V8)
            assert_same(got_d, got_i, exp[q:q + 1], f"repeat {r}")
            got_d, got_i, _ = s.search(queries, 10, V8)
            assert_same(got_d, got_i, exp, f"batch {r}")
