"""GPU fused scan with abandoned tiles: a 64-vector tile is dropped when its partial sums after a quarter or half of the
sub-spaces already exceed every query's admission bound, the bounds shared between the waves of a block and the blocks
of a slab. Results must stay those of the oracle, bit for bit, for clustered codes (most tiles dropped), uniform codes
(hardly any), exact ties at the bound, distances that overflow to infinity, NaN, padded query slots, and repeated
searches of one searcher with changing shapes (the shared bounds return to their initial state).

Left to itself a searcher abandons tiles only where its codes are alike within tiles and a block scans many vectors, so
the families run with abandonment forced as well, and the kernel that ran is asserted.
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
    if family == "clustered ties":  # few distinct vectors, in clusters: whole tiles tie with the K-th best
        rng = np.random.default_rng(904 + m)
        cent = rng.integers(0, 3, size=(m, 256, d // m)).astype(np.float32)
        kinds = rng.integers(0, 256, size=(300, m), dtype=np.uint8)
        queries = rng.integers(0, 3, size=(nq, d)).astype(np.float32)
        return cent, kinds[rng.integers(0, 300, n)], queries
    cent, codes, queries = datagen.pq_fixture(n, d, m, nq, seed=903 + m)
    if family == "nan":
        cent[3, 40:90, 0] = np.nan  # NaN distances among finite ones
        queries[1] = np.nan         # and a query that has no other
        queries[4, 2] = np.inf
        return cent, codes, queries
    cent[:, 5:60] *= np.float32(1e19)  # squares overflow: infinite distances among finite ones
    return cent, codes, queries


def expect_abandoned(s, k, q):
    """The last scan abandoned tiles exactly where an instance exists."""
    kernel = s.last_kernel()
    assert kernel.abandons == (k <= 64 and kernel.tables == 1), kernel
    assert kernel.queries_per_table * kernel.tables <= q


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


@pytest.mark.parametrize("family", ["clusters", "uniform", "ties", "clustered ties", "overflow", "nan"])
@pytest.mark.parametrize("d,m", [(64, 16), (64, 32), (96, 48), (128, 64)])
def test_forced_abandonment_matches_oracle(family, d, m):
    n, nq = 20_003, 21
    cent, codes, queries = fixture(family, n, d, m, nq)
    with np.errstate(all="ignore"), vk.PQSearcher(cent, codes, d) as s:

        def expected(count, k, variant):
            if family == "nan":  # the order of NaN distances is not defined: as the plain scan has it
                s.set_abandon(vk.Abandon.Never)
                dist, ids, _ = s.search(queries[:count], k, variant)
                assert not s.last_kernel().abandons
                s.set_abandon(vk.Abandon.Always)
                exp = np.empty(ids.shape, dtype=vk.NEIGHBOR_DTYPE)
                exp["dist"], exp["id"] = dist, ids
                return exp
            return (orc.adc_search if variant == V8 else orc.adc_search_f16)(cent, d, codes, queries[:count], k)

        s.set_abandon(vk.Abandon.Always)
        for q, threads, blocks in [(1, 256, 4), (2, 1024, 2), (4, 512, 1), (4, 1024, 7), (4, 256, 0), (8, 256, 3)]:
            s.set_tuning(vk.Tuning(queries_per_block=q, scan_threads=threads, blocks_per_query=blocks))
            for variant, k, count in [(V8, 1, nq), (V8, 10, 1), (V8, 16, nq), (V8, 64, 5), (V8, 65, nq), (V9, 10, nq)]:
                got_d, got_i, _ = s.search(queries[:count], k, variant)
                expect_abandoned(s, k, q)
                assert_same(got_d, got_i, expected(count, k, variant),
                            f"{vk.variant_name(variant)} Q={q} threads={threads} blocks={blocks} k={k} nq={count}")


@pytest.mark.parametrize("variant,q,nq", [(V8, 1, 170), (V8, 2, 340), (V8, 4, 1_000), (V9, 8, 1_360)])
def test_queries_far_from_the_data_go_to_the_plain_scan(variant, q, nq):
    # A million vectors per block, where the blocks first vote: all leave when the queries are far from every vector, none
    # does when they are near. The second scan may not cost what abandoning in vain did (Q = 2: 1.59 times the plain scan,
    # fp16 1.44; measured with the vote 1.14 and 1.07).
    cent, codes, near = datagen.pq_fixture(20_011, 64, 16, nq, seed=940)
    codes = np.tile(codes, (50, 1))
    far = np.random.default_rng(941).standard_normal((nq, 64), dtype=np.float32) * 3
    d_far = vk.DeviceArray.from_host(far)
    d_out = vk.DeviceArray(nq * 10 * vk.NEIGHBOR_DTYPE.itemsize)

    def scan_ms():
        return min(s.search_device(d_far.address, nq, 10, variant, d_out.address).scan_ms for _ in range(8))

    try:
        with vk.PQSearcher(cent, codes, 64) as s:
            s.set_tuning(vk.Tuning(queries_per_block=q))
            results, times = {}, {}
            for mode in (vk.Abandon.Never, vk.Abandon.Auto):
                s.set_abandon(mode)
                for name, x in (("far", far), ("near", near), ("mixed", np.concatenate([near[:nq // 2], far[nq // 2:]])),
                                ("far", far)):
                    dist, ids, _ = s.search(x, 10, variant)
                    kernel = s.last_kernel()
                    assert kernel.abandons == kernel.votes == (mode == vk.Abandon.Auto and name != "far"), (name, kernel)
                    if mode == vk.Abandon.Never:
                        results[name] = dist, ids
                    else:
                        assert (ids == results[name][1]).all() and (dist == results[name][0]).all(), name
                times[mode] = scan_ms()
            got = d_out.download(np.empty((nq, 10), dtype=vk.NEIGHBOR_DTYPE))
            assert (got["id"] == results["far"][1]).all()
            assert times[vk.Abandon.Auto] < 1.32 * times[vk.Abandon.Never], times
    finally:
        d_far.free()
        d_out.free()


def test_abandonment_modes():
    cent, codes, queries = datagen.pq_fixture(140_003, 64, 16, 4, seed=930)
    exp = orc.adc_search(cent, 64, codes, queries, 10)
    with vk.PQSearcher(cent, codes, 64) as s:
        with pytest.raises(vk.VkLogicError):
            s.last_kernel()
        with pytest.raises(vk.VkInvalidArgument):
            s.set_abandon(3)
        for blocks, mode, abandons in [(1, vk.Abandon.Auto, True), (16, vk.Abandon.Auto, False),
                                       (16, vk.Abandon.Always, True), (1, vk.Abandon.Never, False)]:
            s.set_abandon(mode)
            s.set_tuning(vk.Tuning(queries_per_block=4, blocks_per_query=blocks))
            got_d, got_i, _ = s.search(queries, 10, V8)
            assert s.last_kernel().abandons == abandons, (blocks, mode)
            assert_same(got_d, got_i, exp, f"blocks={blocks} mode={mode}")
        # One query per table earns the first bounds back from 64k vectors per block, unless it is the only slab.
        s.set_abandon(vk.Abandon.Auto)
        for count, blocks, abandons in [(4, 3, False), (4, 2, True), (1, 3, True), (1, 5, False)]:
            s.set_tuning(vk.Tuning(queries_per_block=1, blocks_per_query=blocks))
            got_d, got_i, _ = s.search(queries[:count], 10, V8)
            assert s.last_kernel().abandons == abandons, (count, blocks)
            assert_same(got_d, got_i, exp[:count], f"Q=1 nq={count} blocks={blocks}")


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 4097])
def test_abandoned_tiles_small_databases(n):
    cent, codes, queries = datagen.random_fixture(n, 64, 16, 5, seed=910 + n)
    with vk.PQSearcher(cent, codes, 64) as s:
        for mode in (vk.Abandon.Auto, vk.Abandon.Always):
            s.set_abandon(mode)
            for k in sorted({1, min(n, 60), min(n, 100)}):
                got_d, got_i, _ = s.search(queries, k, V8)
                assert s.last_kernel().abandons == (mode == vk.Abandon.Always and k <= 64)
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
            assert s.last_kernel().abandons
            got_d, got_i, _ = s.search(queries, 10, V8)
            assert s.last_kernel().abandons
            assert_same(got_d, got_i, exp, f"batch {r}")
