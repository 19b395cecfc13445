"""GPU tests of size- and layout-dependent branches of the strategies, each at
the sizes where it can go wrong, against the oracle (bit-exact for integers)."""
import numpy as np
import pytest

import oracle as O
from eiger_amd import gamax as G
from test_groupby_gpu import STRATEGIES, assert_same, run, sorted_by_key

pytestmark = pytest.mark.gpu
A = G.aggregation_id


@pytest.mark.parametrize("n", [1, 4095, 4097, 70_001])
@pytest.mark.parametrize("dtype,shift,low,minimum", [
    (np.int64, 12, 7, -(1 << 40)), (np.int32, 5, 31, -(1 << 20)), (np.uint64, 40, 0, 1 << 63), (np.uint32, 0, 0, 5),
    (np.int64, 62, 1, 0)])
def test_sort_strategy_keys_sharing_low_bits(n, dtype, shift, low, minimum):
    """Keys whose low bits are all alike (ids handed out in blocks): the sort
    covers only the varying bits of key - min; output ascending."""
    rng = np.random.default_rng(n + shift)
    codes = rng.integers(0, 2 if shift == 62 else 3000, n)
    keys = (np.array([minimum], dtype=dtype) + ((codes.astype(dtype) << dtype(shift)) | dtype(low))).astype(dtype)
    vals = rng.integers(-1000, 1000, n).astype(np.int64)
    reqs = [(0, A.SUM), (-1, A.COUNT_ALL)]
    exp = sorted_by_key(O.groupby(keys, [vals], reqs))
    for fn in (G.sort_groupby, G.sort_groupby_gfur):
        assert_same(run(fn, keys, [vals], reqs), exp)


@pytest.mark.parametrize("ktype", [np.int32, np.int64])
@pytest.mark.parametrize("vtype,kinds", [
    (np.int64, (A.SUM, A.MIN, A.MAX, A.COUNT_ALL)), (np.float32, (A.SUM, A.MIN, A.MAX)), (np.uint32, (A.MAX, A.MIN)),
    (np.int16, (A.SUM, A.MIN)), (np.float64, (A.MAX, A.SUM)), (None, (A.COUNT_ALL,)), (np.int32, (A.ANY, A.COUNT_ALL))])
def test_batch_value_widths_hot_keys_and_full_tables(ktype, vtype, kinds):
    """One batch of every way through the aggregation kernel: whole-query,
    row-range and partition items; 1/4/8-byte and no values; a key most rows
    hold; more groups than the LDS table has slots; the empty-slot key; row
    counts around a step."""
    rng = np.random.default_rng(11)
    info = np.iinfo(ktype)
    shapes = [(1, 1), (63, 5), (4096, 40), (4097, 4097), (40_000, 300), (70_001, 3000), (200_003, 20_000)]
    queries, datas, keep = [], [], []
    for n, d in shapes:
        keys = rng.integers(0, d, n).astype(ktype)
        keys[rng.random(n) < 0.5] = keys[0]          # a hot key
        if n > 10:
            keys[5], keys[6] = info.min, info.max    # INT_MIN encodes to the empty slot word
        vals = None
        if vtype is not None:
            vals = (rng.integers(-500, 500, n) if np.dtype(vtype).kind != "u" else rng.integers(0, 1000, n)).astype(vtype)
            if kinds[0] == A.ANY:
                vals = (keys.astype(np.int64) % 1000).astype(vtype)  # one value per key
        g = len(np.unique(keys))
        outs = [G.make_column(G.to_type_id(ktype), g)]
        for k in kinds:
            outs.append(G.make_column(G.agg_output_data_type(k, G.to_type_id(vtype or np.int64)), g))
        kc = G.make_column_from_host(keys)
        vc = None if vals is None else G.make_column_from_host(vals)
        keep += [kc, vc]
        queries.append(G.batch_query(kc, vc, g, outs[0], outs[1:]))
        datas.append((keys, vals, outs))
    reqs = [(-1 if k == A.COUNT_ALL else 0, k) for k in kinds]
    for tuning in (G.batch_tuning(tile_rows_log2=16, lds_slots_log2=9, lds_max_bound_log2=12, blocks_per_cu=2, radix_bits=10),
                   G.batch_tuning(tile_rows_log2=10, lds_slots_log2=6, lds_max_bound_log2=8, blocks_per_cu=1, radix_bits=0)):
        plan = G.batch_plan(queries, G.to_type_id(ktype), G.to_type_id(vtype or np.int64), reqs, tuning)
        for launch in (plan.run, plan.graph_launch, plan.graph_launch):
            launch()
            ng, st = plan.results()
            assert not st.any()
            for (keys, vals, outs), g in zip(datas, ng):
                exp = sorted_by_key(O.groupby(keys, [] if vals is None else [vals], reqs))
                got = sorted_by_key([o.to_numpy()[:g] for o in outs])
                assert_same(got, exp, 1e-5 if vtype == np.float32 else 1e-9)
        plan.free()


@pytest.mark.parametrize("dtype", [np.int32, np.int64, np.uint16, np.uint32])
@pytest.mark.parametrize("m", [4096, 4097, 6143, 6145, 12_289, 50_000])
def test_dictionary_table_sizes_around_the_lds_limit_and_load(dtype, m):
    """Dictionaries around the last LDS table, around the load at which the
    HBM table doubles, with repeats, absent keys and the type's extremes."""
    info = np.iinfo(dtype)
    rng = np.random.default_rng(m)
    pool = rng.integers(info.min, info.max, m, dtype=dtype, endpoint=True)
    pool[0], pool[1] = info.min, info.max
    pool[m // 2] = pool[m // 3]  # a repeated key: its first position counts
    n = 4 * 2048 + 77
    keys = np.where(rng.random(n) < 0.7, rng.choice(pool, n), rng.integers(info.min, info.max, n, dtype=dtype, endpoint=True)).astype(dtype)
    kc, dc = G.make_column_from_host(keys), G.make_column_from_host(pool)
    got = G.dictionary_encode_with_dict(kc, dc).to_numpy()
    np.testing.assert_array_equal(got, O.dict_encode(keys, pool))


@pytest.mark.parametrize("dtype,m", [
    (np.int32, 314_572), (np.int32, 314_573), (np.int32, 655_360), (np.int32, 655_361),  # 3/5 of 2^19, 5/8 of 2^20 slots
    (np.int64, 262_144), (np.int64, 262_145), (np.int64, 524_289)])  # 2^19, 2^20, 2^21 slots: one, two a step
def test_dictionary_table_sizes_around_the_l2(dtype, m):
    """Large dictionaries on both sides of the lines between table sizes and
    between one and two slots a step; half of the keys are absent."""
    rng = np.random.default_rng(m)
    info = np.iinfo(dtype)
    pool = rng.integers(info.min, info.max, m, dtype=dtype, endpoint=True)
    pool[0], pool[1] = info.min, info.max
    n = 600_011
    keys = np.where(rng.random(n) < 0.5, rng.choice(pool, n), rng.integers(info.min, info.max, n, dtype=dtype, endpoint=True)).astype(dtype)
    kc, dc = G.make_column_from_host(keys), G.make_column_from_host(pool)
    got = G.dictionary_encode_with_dict(kc, dc).to_numpy()
    np.testing.assert_array_equal(got, O.dict_encode(keys, pool))


@pytest.mark.parametrize("bits", [(16, 16), (17, 16), (1, 31), (32,), (33,), (8, 8, 8, 8)])
@pytest.mark.parametrize("algo", ["AUTO_ALGO", "HASH", "SORT", "PARTITION"])
def test_fused_keys_around_32_bits(bits, algo):
    """Key columns whose fields take just under, exactly and just over 32
    bits: the fused key is 4 or 8 bytes wide; the extreme tuples are there."""
    rng = np.random.default_rng(sum(bits))
    n = 9001
    cols = []
    for b in bits:
        c = rng.integers(0, 1 << b, n, dtype=np.int64)
        c[0], c[1] = 0, (1 << b) - 1
        cols.append(c - (1 << (b - 1)))
    if len(cols) == 1:
        cols.append(np.full(n, -7, np.int16))  # a constant column: no bits
    for c in cols:
        c[2:200] = c[200:398]  # some repeated tuples
    vals = rng.integers(-100, 100, n).astype(np.int32)
    kc = [G.make_column_from_host(c) for c in cols]
    t = G.groupby(kc, [G.make_column_from_host(vals)], [(0, A.SUM), (-1, A.COUNT_ALL)],
                  G.groupby_hint(groupby_algo=G.groupby_algo[algo], enable_skf=True))
    got = t.to_numpy()
    exp = {}
    for i, tup in enumerate(zip(*[c.tolist() for c in cols])):
        s, k = exp.get(tup, (0, 0))
        exp[tup] = (s + int(vals[i]), k + 1)
    rows = list(zip(*[g.tolist() for g in got[:len(cols)]]))
    assert len(rows) == len(exp)
    for r, s, k in zip(rows, got[-2].tolist(), got[-1].tolist()):
        assert exp[r] == (s, k)
    if algo == "SORT":
        assert rows == sorted(rows)


@pytest.mark.parametrize("dtype", [np.int32, np.int64, np.uint64])
@pytest.mark.parametrize("d", [1, 16, 1000, 7999, 16_400])
@pytest.mark.parametrize("n", [16 * 4096, 200_003])
def test_hash_tables_of_many_workgroups_merged(dtype, d, n):
    """Grids of 16 and 49 workgroups, whose LDS tables are flushed with atomics
    (few groups, and 16,400, above twice the LDS slots) or stored and merged:
    the keys whose encodings are the empty word, and undersized bounds."""
    rng = np.random.default_rng(d)
    info = np.iinfo(dtype)
    keys = rng.integers(0, d, n).astype(dtype)
    keys[7::1000], keys[8::999] = info.min, info.max
    if dtype == np.uint64:
        keys[9::501] = 1 << 63
    vals = rng.integers(-1000, 1000, n).astype(np.int64)
    f = rng.random(n).astype(np.float32)
    for reqs in ([(0, A.SUM), (-1, A.COUNT_ALL)], [(0, A.MIN), (0, A.MAX), (1, A.SUM), (-1, A.COUNT_ALL), (0, A.SUM)]):
        exp = sorted_by_key(O.groupby(keys, [vals, f], reqs))
        for bound in (len(exp[0]), max(1, len(exp[0]) // 3)):
            got = sorted_by_key(run(G.hash_groupby, keys, [vals, f], reqs, G.groupby_hint(groups_upper_bound=bound)))
            assert_same(got, exp)


@pytest.mark.parametrize("n,bound,d,stored", [
    (61_440, 8000, 500, False), (61_441, 8000, 500, True),      # 15 and 16 blocks
    (65_536, 313, 313, False), (65_536, 314, 314, True),        # 16 tiles: 16 * bound against 5000 + 16
    (1 << 20, 20, 20, False), (1 << 20, 21, 18, True),          # 256 tiles: one a compute unit
    ((1 << 20) + 1, 20, 3, False), ((1 << 20) + 1, 21, 1, True),
    (200_003, 16_272, 16_000, True), (200_003, 16_273, 16_000, False),  # twice the LDS slots of two states
])
def test_hash_tables_stored_or_flushed(n, bound, d, stored):
    """Both sides of the lines between flushing and storing the workgroups'
    tables, by the kernels that ran; generic and specialised kernels."""
    rng = np.random.default_rng(bound)
    keys = rng.integers(0, d, n).astype(np.int32)
    vals = rng.integers(-1000, 1000, n).astype(np.int64)
    reqs = [(0, A.SUM), (-1, A.COUNT_ALL)]
    exp = sorted_by_key(O.groupby(keys, [vals], reqs))
    before = G.jit_stats()
    try:
        for mode in (G.jit_mode.OFF, G.jit_mode.SYNC):
            G.jit_configure(mode, 0)
            G.kernel_timing(True)
            G.kernel_timing_reset()
            l0 = G.jit_stats()["launches"]
            got = sorted_by_key(run(G.hash_groupby, keys, [vals], reqs, G.groupby_hint(groups_upper_bound=bound)))
            assert_same(got, exp)
            assert G.kernel_time("hash_merge")[0] == (1 if stored else 0)
            assert G.jit_stats()["launches"] - l0 == (0 if mode == G.jit_mode.OFF else 1)
    finally:
        G.kernel_timing(False)
        G.kernel_timing_reset()
        G.jit_configure(before["mode"], before["min_rows"])


@pytest.mark.parametrize("n", [1, 1023, 1025, 4096, 4097])
@pytest.mark.parametrize("ktype", [np.int32, np.int64, np.uint8, np.float32])
def test_tiny_inputs_in_one_workgroup(n, ktype):
    """Row counts around one workgroup's rows, one group to a group a row, 1-
    to 8-byte values, few and many states (more than its LDS holds), the keys
    whose encodings are the empty word, a key every row holds."""
    rng = np.random.default_rng(n)
    for d in (1, 7, n):
        keys = rng.integers(0, max(1, min(d, 250)) if ktype == np.uint8 else d, n).astype(ktype)
        if np.dtype(ktype).kind == "i" and n > 3 and d > 1:
            keys[1], keys[2] = np.iinfo(ktype).min, np.iinfo(ktype).max
        vals = [rng.integers(-100, 100, n).astype(t) for t in (np.int64, np.int8, np.int16, np.float64)]
        for reqs in ([(0, A.SUM), (-1, A.COUNT_ALL)], [(1, A.MIN), (2, A.MAX)],
                     [(i, k) for i in range(4) for k in (A.SUM, A.MIN, A.MAX)]):
            exp = sorted_by_key(O.groupby(keys, vals, reqs))
            got = sorted_by_key(run(G.hash_groupby, keys, vals, reqs, G.groupby_hint(groups_upper_bound=max(1, d // 2))))
            assert_same(got, exp, 1e-9)


@pytest.mark.parametrize("bound", [300, 100_000, 390_000, 1_100_000])
def test_partition_counts_around_the_one_launch_unit_list(bound):
    """Bounds that give 2, 64, 256 and 1024 partitions (one launch makes the
    unit list of up to 512), over keys far fewer than the bound with one key
    that most rows hold (its partition is sliced)."""
    n = 1_200_007
    keys = O.gen_keys_uniform(n, 20_011, seed=bound)
    keys[np.random.default_rng(3).random(n) < 0.6] = 77
    vals = O.gen_values(n, O.VAL_UNIFORM_I64, np.int64, seed=4, stream_id=2)
    reqs = [(0, A.SUM), (0, A.MIN), (-1, A.COUNT_ALL)]
    exp = sorted_by_key(O.groupby(keys, [vals], reqs))
    for fn in (G.partition_groupby, G.partition_groupby_gfur):
        assert_same(sorted_by_key(run(fn, keys, [vals], reqs, G.groupby_hint(groups_upper_bound=min(bound, n - 1)))), exp)


@pytest.mark.parametrize("n,bound", [(9_000_011, 500_000), (18_000_011, 800_000), (9_000_011, 300_000)])
@pytest.mark.parametrize("hot", [0.0, 0.0005, 0.005, 0.3])
def test_partitions_a_little_larger_than_the_average(n, bound, hot):
    """512, 1024 and 256 partitions with one from about the average size to
    many times it: whole below 5/4 of the average, sliced above, or all sliced
    (256).  The slices' groups come out once and the spill table is used."""
    rng = np.random.default_rng(bound)
    keys = O.gen_keys_uniform(n, 20_011, seed=bound)
    keys[rng.random(n) < hot] = 77
    vals = O.gen_values(n, O.VAL_UNIFORM_I64, np.int64, seed=4, stream_id=2)
    reqs = [(0, A.SUM), (0, A.MIN), (0, A.MAX), (-1, A.COUNT_ALL), (0, A.ANY)]
    exp = sorted_by_key(O.groupby(keys, [vals], reqs[:4]))
    got = sorted_by_key(run(G.partition_groupby, keys, [vals], reqs, G.groupby_hint(groups_upper_bound=bound)))
    assert_same(got[:5], exp)
    assert (exp[2] <= got[5]).all() and (got[5] <= exp[3]).all()


@pytest.mark.parametrize("states,slots", [(2, 4060), (3, 2912), (12, 800)])
@pytest.mark.parametrize("fill,passes", [(0.5, 1), (0.65, 1), (0.8, 2), (0.87, 2)])
def test_partition_passes_at_a_true_bound(states, slots, fill, passes):
    """256 tables of about `slots` slots as full as the bound says: one digit
    pass up to 2/3 full, above that two passes into more partitions."""
    n, d = 1_500_007, int(256 * slots * fill)
    _check_partitioned(n, d, d, states, passes)


@pytest.mark.parametrize("states,slots", [(2, 4060), (3, 2912), (12, 800)])
@pytest.mark.parametrize("fill", [0.85, 0.95, 1.1])
def test_partition_tables_fuller_than_planned(states, slots, fill):
    """More groups than the bound: the unit tables fill to `fill` of their
    slots, keys whose buckets are full go to the HBM table (and where that
    fills too, the call runs again with a larger one)."""
    _check_partitioned(1_500_007, int(256 * slots * fill), int(256 * slots * 0.6), states, 1)


def _check_partitioned(n, d, bound, states, passes):
    rng = np.random.default_rng(d)
    keys = np.concatenate([rng.permutation(d), rng.integers(0, d, n - d)]).astype(np.int32)
    vals = [rng.integers(-1000, 1000, n).astype(np.int64) for _ in range(4)]
    reqs = ([(-1, A.COUNT_ALL)] + [(c, k) for k in (A.SUM, A.MIN, A.MAX) for c in range(4)])[:states]
    exp = sorted_by_key(O.groupby(keys, vals, reqs))
    try:
        G.kernel_timing(True)
        G.kernel_timing_reset()
        got = sorted_by_key(run(G.partition_groupby, keys, vals, reqs, G.groupby_hint(groups_upper_bound=bound)))
        assert G.kernel_time("radix_scatter")[0] == passes
    finally:
        G.kernel_timing(False)
        G.kernel_timing_reset()
    assert_same(got, exp)


@pytest.mark.parametrize("before,rows,after", [
    (b, r, a) for b in (0, 1, 2048, 126 * 2048 + 5, 128 * 2048 - 1, 128 * 2048)
    for r, a in ((128 * 2048, 0), (128 * 2048 + 1, 1), (258 * 2048 + 3, 130 * 2048))] + [(77, 66 * 128 * 2048, 3)])
def test_sort_groups_longer_than_a_span_of_tiles(before, rows, after):
    """One group of more rows than 128 tiles of 2048, its head in, at and
    around the first tile of a span, with groups before and after it."""
    rng = np.random.default_rng(before + rows + after)
    keys = np.concatenate([np.sort(rng.integers(0, 5, before)), np.full(rows, 7), 9 + np.sort(rng.integers(0, 3, after))])
    keys = keys.astype(np.int32)
    a = rng.integers(-1000, 1000, len(keys)).astype(np.int64)
    one = (keys * 3).astype(np.int32)  # one value per key
    reqs = [(0, A.SUM), (0, A.MIN), (0, A.MAX), (-1, A.COUNT_ALL), (1, A.ANY)]
    exp = sorted_by_key(O.groupby(keys, [a, one], reqs))
    for fn in (G.sort_groupby, G.sort_groupby_gfur):
        assert_same(run(fn, keys, [a, one], reqs), exp)
