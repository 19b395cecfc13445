"""Learned dispatch on the GPU: the HIP feature, forward and gradient kernels
against the fp64 oracle, training that lowers the loss, and the guarantee
that the dispatcher's choice never changes a group-by result."""
import numpy as np
import pytest

import oracle as O
from eiger_amd import gamax as G

pytestmark = pytest.mark.gpu
A = G.aggregation_id


@pytest.mark.parametrize("kt", [np.int32, np.int64])
def test_features_match_oracle(kt):
    rng = np.random.default_rng(3)
    cases = [(1, 1), (100, 7), (4096, 4096), (5000, 3), (200_000, 50_000), (1_000_003, 1 << 24)]
    cols, exp = [], []
    for i, (rows, d) in enumerate(cases):
        if i % 2:
            keys = rng.integers(-d, d, rows).astype(kt)
        else:
            keys = np.sort(rng.integers(0, d, rows)).astype(kt)
        cols.append(G.make_column_from_host(keys))
        exp.append(O.sample_features(keys, group_bound=d if i == 2 else 0, nops=5, value_bytes=12))
    got = G.mlp_features(cols, group_bounds=[0, 0, 4096, 0, 0, 0], nops=5, value_bytes=12)
    # counts are exact; entropy and logs differ only by fp32 rounding order
    np.testing.assert_allclose(got, np.array(exp), rtol=1e-5, atol=1e-6)


def test_forward_matches_fp64_oracle():
    rng = np.random.default_rng(0)
    P = G.mlp_init(7)
    P[1024:1088] = rng.standard_normal(64) * 0.1
    x = rng.random((1000, 16)).astype(np.float32)
    got = G.mlp_forward(P, x)
    exp = O.mlp_forward(P.astype(np.float64), x)
    np.testing.assert_allclose(got, exp, rtol=1e-4, atol=1e-5)


def test_gradient_matches_fp64_oracle():
    """eg_mlp_loss_grad (fp32 HIP backward, 64 samples per workgroup, fixed-order
    reduction) against the analytic fp64 gradient of the oracle, itself pinned
    by finite differences in the CPU tests."""
    rng = np.random.default_rng(1)
    P = G.mlp_init(3)
    P[1024:1088] = rng.standard_normal(64) * 0.1
    n = 777
    x = rng.random((n, 16)).astype(np.float32)
    t = rng.dirichlet([1, 1, 1], n).astype(np.float32)
    c = rng.random(n).astype(np.float32)
    loss, g = G.mlp_loss_grad(P, x, t, c, 0.5)
    eloss, eg = O.mlp_loss_grad(P.astype(np.float64), x, t, c, 0.5)
    assert abs(loss - eloss) <= 1e-5 * abs(eloss)
    scale = np.abs(eg).max()
    np.testing.assert_allclose(g, eg, rtol=1e-3, atol=1e-5 * scale)
    assert np.linalg.norm(g - eg) <= 1e-4 * np.linalg.norm(eg)


def test_training_lowers_the_loss_and_learns_a_rule():
    """A synthetic labelling (best strategy from feature 2 thresholds, card =
    feature 3) is learned by eg_mlp_train."""
    rng = np.random.default_rng(5)
    n = 8192
    x = rng.random((n, 16)).astype(np.float32)
    lab = np.where(x[:, 2] < 0.4, 0, np.where(x[:, 5] < 0.5, 1, 2))
    t = np.eye(3, dtype=np.float32)[lab]
    c = x[:, 3].copy()
    P0 = G.mlp_init(11)
    l0, _ = G.mlp_loss_grad(P0, x, t, c, 1.0)
    P, losses = G.mlp_train(P0, x, t, c, epochs=40, batch=512, lr=3e-3, lam=1.0, seed=2)
    l1, _ = G.mlp_loss_grad(P, x, t, c, 1.0)
    assert l1 < 0.25 * l0 and losses[-1] < losses[0]
    pred = np.argmax(G.mlp_forward(P, x)[:, :3], axis=1)
    assert (pred == lab).mean() > 0.95


def test_dispatch_choice_never_changes_results():
    n = 1 << 20
    keys = O.gen_keys_uniform(n, 70_000, seed=9)
    vals = O.gen_values(n, O.VAL_UNIFORM_I64, np.int64, seed=9, stream_id=2)
    reqs = [(-1, A.COUNT_ALL), (0, A.SUM), (0, A.MAX)]
    exp = O.groupby(keys, [vals], reqs)
    kc, vc = G.make_column_from_host(keys), G.make_column_from_host(vals)
    for bias in range(3):  # a model that always picks HASH, SORT, then PARTITION
        P = np.zeros(G.MLP_PARAMS, np.float32)
        P[5504 + bias] = 5.0
        P[5507] = np.log2(70_000) / 32
        G.mlp_load(P)
        assert G.mlp_loaded()
        algo, card = G.mlp_select(kc, nops=3, value_bytes=8)
        assert algo == [G.groupby_algo.HASH, G.groupby_algo.SORT, G.groupby_algo.PARTITION][bias]
        assert abs(np.log2(card) - np.log2(70_000)) < 0.01
        h = G.groupby_hint()
        t = G.groupby([kc], [vc], reqs, h)
        assert h.groupby_algo == algo
        got = t.to_numpy()
        order = np.argsort(got[0], kind="stable")
        for g, e in zip(got, exp):
            np.testing.assert_array_equal(g[order], e)
        t.free()
    G.mlp_load(None)
    assert not G.mlp_loaded()


def test_batched_selection_equals_single_query_selection():
    rng = np.random.default_rng(21)
    keys = []
    for i, (rows, d) in enumerate([(1000, 10), (50_000, 40_000), (300_000, 1 << 20), (70_000, 3), (0, 1)]):
        k = rng.integers(0, d, rows).astype(np.int32 if i % 2 else np.int64)
        keys.append(G.make_column_from_host(k))
    ra, rn = G.auto_select_groupby_algo_batch(keys)
    for k, a, nd in zip(keys, ra, rn):
        if k.size == 0:
            assert nd == 0 and a == G.groupby_algo.HASH
            continue
        h = G.groupby_hint()
        G.auto_select_groupby_algo([k], h)
        assert h.groupby_algo == a and nd == G.compute_ndv_approx(k)
    P = G.mlp_init(4)
    G.mlp_load(P)
    try:
        live = [k for k in keys if k.size > 0]
        ma, mc = G.mlp_select_batch(live, None, 2, 8)
        for k, a, c in zip(live, ma, mc):
            a1, c1 = G.mlp_select(k, 0, 2, 8)
            assert a1 == a and c1 == c
    finally:
        G.mlp_load(None)


@pytest.mark.parametrize("log_rows,bound,algo,card,singles,exp", [
    # (bound, expected, full estimate): the estimate with headroom, or the caller's bound
    (20, 1 << 18, "PARTITION", 10_000, 0.9, (26_024, 10_000, False)),
    (20, 20_000, "PARTITION", 10_000, 0.9, (20_000, 10_000, False)),
    (24, 1 << 18, "PARTITION", 10_000, 0.2, (26_024, 10_000, False)),     # few singletons: the estimate stands
    (28, 1 << 24, "PARTITION", 1_500_000, 0.2, (3_751_024, 1_500_000, False)),
    (28, 1 << 24, "PARTITION", 2_000_000, 0.2, (1 << 24, 5_001_024, False)),  # perhaps short of a tight bound
    (24, 1 << 18, "PARTITION", 10_000, 0.9, (1 << 18, 26_024, False)),    # 2^24 rows: three digit bits do not pay
    (28, 1 << 18, "PARTITION", 10_000, 0.9, (26_024, 10_000, True)),      # 2^28 rows: they do
    (28, 1 << 18, "PARTITION", 100_000, 0.9, (1 << 18, 251_024, False)),  # no digit bit saved
    (28, 1 << 17, "PARTITION", 25_000, 0.9, (1 << 17, 63_524, False)),    # seven bits to six
    (28, 1 << 22, "PARTITION", 50_000, 0.9, (126_024, 50_000, True)),     # a pass saved
    (28, 1 << 22, "PARTITION", 452_975, 1.0, (1 << 22, 1_133_461, False)),  # the same, of singletons
    (28, 1 << 22, "PARTITION", 415_000, 1.0, (1_038_524, 415_000, True)),   # below a quarter of it
    (28, 1 << 18, "PARTITION", 61_752, 1.0, (1 << 18, 155_404, False)),
    (28, 1 << 24, "PARTITION", 6_000_000, 0.9, (1 << 24, 15_001_024, False)),
    (28, 1 << 26, "PARTITION", 20_000_000, 0.9, (50_001_024, 20_000_000, True)),  # small partitions
    (28, 1 << 18, "HASH", 10_000, 0.9, (26_024, 10_000, True)),
    (28, 0, "PARTITION", 10_000, 0.9, (26_024, 10_000, True)),            # no caller bound
    (24, 0, "PARTITION", 1 << 24, 0.9, (1 << 24, 1 << 24, True)),
])
def test_sizing_of_dispatched_tables(log_rows, bound, algo, card, singles, exp):
    """Five states over rows of 16 bytes: each side of the lines between the
    model's estimate, the caller's bound and the full-column estimate."""
    got = G.dispatch_sizing(G.type_id.INT32, 1 << log_rows, bound, 5, 12, G.groupby_algo[algo], card, singles)
    assert got == exp


@pytest.mark.parametrize("log_rows,nops,ktype,card,bound,exp", [
    # card: what the model estimates; it scores PARTITION best
    (20, 2, np.int32, 2000, 0, "HASH"), (20, 2, np.int32, 2100, 0, "PARTITION"),
    (24, 2, np.int32, 2000, 0, "HASH"), (24, 2, np.int32, 2100, 0, "PARTITION"),
    (20, 10, np.int32, 1900, 0, "HASH"), (24, 10, np.int32, 1980, 0, "PARTITION"),     # 1936 slots
    (20, 16, np.int64, 1150, 0, "HASH"), (20, 16, np.int64, 1260, 0, "PARTITION"),     # ~1200 slots
    # a caller's bound
    (20, 2, np.int32, 2100, 2048, "HASH"), (20, 2, np.int32, 2100, 2049, "PARTITION"),
    (20, 16, np.int32, 2100, 1280, "HASH"), (20, 16, np.int32, 2100, 1281, "PARTITION"),
    (24, 16, np.int32, 2100, 2048, "HASH"), (24, 16, np.int32, 2100, 2049, "PARTITION"),
    ((1 << 17) - 1, 2, np.int32, 5000, 0, "HASH"), (17, 2, np.int32, 5000, 0, "PARTITION"),
])
def test_hash_by_group_count_depends_on_the_states(log_rows, nops, ktype, card, bound, exp):
    """A model that always scores partition best and estimates `card`: few
    enough groups for the LDS table of that many states go to hash."""
    n = log_rows if log_rows > 64 else 1 << log_rows
    k = G.make_column(G.to_type_id(ktype), n)
    P = np.zeros(G.MLP_PARAMS, np.float32)
    P[5504 + 2] = 5.0
    P[5507] = np.log2(card) / 32
    loaded = G.mlp_loaded()
    G.mlp_load(P)
    try:
        algo, _ = G.mlp_select(k, bound, nops=nops, value_bytes=8)
        assert algo == G.groupby_algo[exp]
        assert list(G.mlp_select_batch([k], [bound], nops=nops, value_bytes=8)[0]) == [algo]
    finally:
        G.mlp_load(None)
        if loaded:
            G.load_dispatch_model()
        k.free()


@pytest.mark.parametrize("nops,value_bytes", [(5, 12), (8, 24), (10, 32), (16, 8), (16, 32)])
@pytest.mark.parametrize("d", [600, 4000, 100_000])
def test_group_estimates_of_wide_requests(d, nops, value_bytes):
    """The shipped model's estimate is about the group count (its sizing leaves
    2.5x headroom) also for requests wider than the ones it was trained on."""
    k = G.gen_keys_uniform(1 << 20, d, seed=7)
    loaded = G.mlp_loaded()
    assert G.load_dispatch_model()
    try:
        algo, card = G.mlp_select(k, 0, nops=nops, value_bytes=value_bytes)
        assert d / 2.5 <= card <= 2.5 * d
        a, c = G.mlp_select_batch([k], None, nops=nops, value_bytes=value_bytes)
        assert a[0] == algo and abs(int(c[0]) - card) <= 1 + card // 1000
    finally:
        if not loaded:
            G.mlp_load(None)
        k.free()
