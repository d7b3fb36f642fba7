"""FP64 GPU path vs the CPU oracle: bit-for-bit.

The GPU kernels and the oracle implement the same canonical arithmetic
(rr_math functions, 64-lane canonical sums, Eigen's ColPivHouseholderQR
operation order), so coefficients, 1-R2 and RMSE must be identical bits; the
only allowance is the sign of a NaN produced by a hardware operation (x86 and
AMDGPU default NaNs differ), which is compared as "both NaN".

Tests that set no option run at a new context's: form 1 at four rows a thread
(two up to 512 rows, one up to 256).  Form 0 runs at two where four are asked
for, and raw trees run the form asked for at every stack depth.
"""
import numpy as np
import pytest

import capi
import oracle_lib as O
import treegen

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    both_nan = np.isnan(a) & np.isnan(b)
    eq = a.view(np.uint64) == b.view(np.uint64)
    return bool(np.all(eq | both_nan))


def make_data(seed, n, d, lo=-5.0, hi=5.0):
    rng = np.random.default_rng(seed)
    X = rng.uniform(lo, hi, size=(n, d))
    y = np.sin(X[:, 0]) * 3.0 + X[:, min(1, d - 1)] ** 2 - 0.5 * X[:, 0] + rng.normal(0, 0.01, n)
    return X, y


SPECIAL = np.array([0.0, -0.0, 1.0, -1.0, 0.5, 2.0, np.pi, 1e-300, 5e-324, 1e300, -1e300, np.inf, -np.inf, np.nan,
                    709.78, 709.79, -745.1, -745.2, 1e8, 2.0 ** 28, 2.0 ** 28 + 1, 1e22, 6.38e189, 1e308,
                    3.0 * np.pi / 2, 1e-8, 0.7853981633974483, 710.0, 1e16])


def test_elementwise_ops_bitexact(ctx):
    print("case: elementwise ops over special + random inputs", flush=True)
    rng = np.random.default_rng(7)
    x = np.concatenate([SPECIAL, -SPECIAL, rng.uniform(-10, 10, 3000), rng.uniform(-1e6, 1e6, 500),
                        10.0 ** rng.uniform(-300, 300, 500), rng.normal(0, 1, 1000)])
    y2 = rng.normal(0, 2, x.size)
    X = np.stack([x, y2], axis=1)
    h = ctx.upload(X, np.zeros(x.size))
    od = O.Dataset(X, np.zeros(x.size))
    for pre in ["sin x0", "cos x0", "ln x0", "exp x0", "sqrt x0", "sqr x0", "+ x0 x1", "- x0 x1", "* x0 x1",
                "/ x0 x1", "< x0 x1", "> x0 x1", "== x0 x0", "!= x0 x1", "min x0 x1", "max x0 x1",
                "/ x0 c0x0p+0", "- c0x1.8p+1 x0"]:
        g = ctx.predict(h, pre, x.size)
        o = od.eval(pre)
        assert same_bits(g, o), pre
    ctx.free(h)


# one row; a slot's last row and the first of the next (4 MiB: 524288 rows of
# one feature, 26176 of 20); several slots; rows wider than a slot
@pytest.mark.parametrize("n,d", [(1, 1), (65, 3), (524288, 1), (524289, 1), (26176, 20), (26177, 20), (90001, 20),
                                 (3, 600000)])
def test_predict_rows_bitexact(ctx, n, d):
    print("case: predict_rows n=%d d=%d" % (n, d), flush=True)
    X = np.random.default_rng(n + d).uniform(-4, 4, (n, d))
    pre = "+ * c0x1.8p+1 sin x0 / exp x%d c0x1.4p+1" % (d - 1)
    assert same_bits(ctx.predict_rows(X, pre), O.Dataset(X, np.zeros(n)).eval(pre))


def test_predict_rows_leaves_no_older_kernel_time(ctx):
    """rr_last_kernel_ms after rr_predict_rows is 0, not an older call's time,
    and the other entry points' own again after that."""
    X, y = make_data(6, 3000, 2)
    h = ctx.upload(X, y)
    ctx.fitness(h, capi.build_batch([["sin x0"]]))
    assert ctx.kernel_ms() > 0
    ctx.predict_rows(X, "sin x0")
    assert ctx.kernel_ms() == 0.0
    ctx.predict(h, "sin x0", 3000)
    assert ctx.kernel_ms() > 0
    ctx.free(h)


def test_predict_rows_argument_errors(ctx):
    for X, pre in [(np.zeros((0, 2)), "x0"), (np.zeros((4, 2)), "x2")]:
        with pytest.raises(RuntimeError):
            ctx.predict_rows(X, pre)
    assert same_bits(ctx.predict_rows(np.zeros((4, 0)), "c0x1p+0"), np.ones(4))


def test_dataset_stats_match(ctx):
    X, y = make_data(3, 1000, 3)
    h = ctx.upload(X, y)
    assert ctx.stats(h) == O.Dataset(X, y).stats()
    ctx.free(h)


# one row; whole and ragged chunks; one slot's worth of values (4 MiB) and one
# value more; a column across two slots
@pytest.mark.parametrize("n,d", [(1, 1), (4096, 3), (4097, 3), (262144, 1), (262145, 1), (100001, 11)])
def test_upload_places_columns_and_statistics(ctx, n, d):
    print("case: upload n=%d d=%d" % (n, d), flush=True)
    X, y = make_data(5, n, d)
    h = ctx.upload(X, y)
    assert ctx.stats(h) == O.Dataset(X, y).stats()
    for j in {0, d // 2, d - 1}:
        assert same_bits(ctx.predict(h, "x%d" % j, n), X[:, j])
        v, e = ctx.predict_fp32(h, "x%d" % j, n)
        assert np.array_equal(v, X[:, j].astype(np.float32))
    od = O.Dataset(X, y)   # y, the ones and the norms of bare factors
    tu = od.tune("+ x0 x%d" % (d - 1))
    coefs, fit = ctx.fitness(h, capi.build_batch([tu["factors"]]), mode="ols")
    assert same_bits(coefs[0], tu["coefs"]) and same_bits([fit[0]["e0"], fit[0]["e1"]], tu["fit"][:2])
    ctx.free(h)


@pytest.mark.parametrize("n,d,seed", [(150, 2, 1), (1000, 5, 2), (4099, 10, 3)])
def test_raw_fitness_bitexact(ctx, n, d, seed):
    print("case: raw n=%d d=%d seed=%d" % (n, d, seed), flush=True)
    X, y = make_data(seed, n, d)
    trees = treegen.random_trees(seed, 300, 1, 40, d)
    h = ctx.upload(X, y)
    od = O.Dataset(X, y)
    arrs = capi.build_batch([[t] for t in trees])
    _, fit = ctx.fitness(h, arrs, mode="raw")
    for t, f in zip(trees, fit):
        e0, e1, _ = od.score(t)
        assert same_bits([f["e0"], f["e1"]], [e0, e1]), t
    ctx.free(h)


# 70001 and 135000 rows: 18 and 33 chunks, folded in two and three groups of
# 16 chunks (the last group of one chunk or a few)
@pytest.mark.parametrize("n,d,seed", [(150, 2, 11), (777, 4, 12), (5000, 10, 13), (64, 3, 14), (7, 3, 15),
                                      (70001, 6, 16), (135000, 3, 17)])
def test_ols_bitexact(ctx, n, d, seed):
    print("case: ols n=%d d=%d seed=%d" % (n, d, seed), flush=True)
    X, y = make_data(seed, n, d)
    trees = treegen.random_trees(seed, 250, 3, 40, d)
    trees += ["+ + * c0x1p+1 x0 sin x1 c0x1.8p+1", "+ sin c0x1p+0 x0", "+ x0 x0", "- * x0 c0x1p+1 + x0 x0",
              "+ + x0 sqr x1 * x0 x1", "ln - x0 x0", "+ x0 ln - x0 x0", "sin c0x1p+0"]
    od = O.Dataset(X, y)
    tuned = [od.tune(t) for t in trees]
    arrs = capi.build_batch([tu["factors"] for tu in tuned])
    h = ctx.upload(X, y)
    coefs, fit = ctx.fitness(h, arrs, mode="ols")
    for t, tu, c, f in zip(trees, tuned, coefs, fit):
        assert len(c) == len(tu["coefs"]), t
        assert same_bits(c, tu["coefs"]), (t, c, tu["coefs"])
        assert f["rank"] == tu["rank"], t
        assert same_bits([f["e0"], f["e1"]], [tu["fit"][0], tu["fit"][1]]), (t, f, tu["fit"])
    ctx.free(h)


def _full_tree(rng, levels, d):
    """A full binary tree: its program needs levels - 1 stack slots even in
    the best evaluation order."""
    if levels == 0:
        return "x%d" % rng.integers(d)
    op = rng.choice(["*", "/", "-", "+", "max"]) if levels > 1 else rng.choice(["*", "-", "+"])
    return "%s %s %s" % (op, _full_tree(rng, levels - 1, d), _full_tree(rng, levels - 1, d))


@pytest.mark.parametrize("form,rows", [(1, 1), (1, 4), (0, 1), (0, 2), (0, 4)])
def test_eval_forms_bitexact(ctx, form, rows):
    """Both factor interpreters (fp64_eval_form 0: operand stack in registers,
    transcendentals called; 1: stack in LDS, inlined) at every row count
    besides the default (form 1, 2 rows, which every other test runs): the
    same bits as the oracle, over a ragged last chunk, with programs of stack
    depth up to 4."""
    print("case: eval form %d rows=%d" % (form, rows), flush=True)
    X, y = make_data(61, 9001, 4)
    rng = np.random.default_rng(61)
    trees = treegen.random_trees(61, 200, 3, 40, 4)
    shallow = trees[:]
    deep = ["* sin %s cos %s" % (_full_tree(rng, L, 4), _full_tree(rng, L, 4)) for L in (2, 3, 4, 5) for _ in range(3)]
    od = O.Dataset(X, y)
    h = ctx.upload(X, y)
    ctx.set_option("fp64_eval_rows", rows)
    ctx.set_option("fp64_eval_form", form)
    try:
        for batch in (shallow, shallow + deep):
            tuned = [od.tune(t) for t in batch]
            coefs, fit = ctx.fitness(h, capi.build_batch([tu["factors"] for tu in tuned]), mode="ols")
            for t, tu, c, f in zip(batch, tuned, coefs, fit):
                assert same_bits(c, tu["coefs"]), (t, c, tu["coefs"])
                assert f["rank"] == tu["rank"], t
                assert same_bits([f["e0"], f["e1"]], [tu["fit"][0], tu["fit"][1]]), (t, f, tu["fit"])
    finally:
        ctx.set_option("fp64_eval_rows", 2)
        ctx.set_option("fp64_eval_form", 1)
    ctx.free(h)


def test_ols_chunked_slab_same_bits(ctx):
    """A tiny slab budget forces many launches; results must not change."""
    X, y = make_data(21, 3000, 4)
    trees = treegen.random_trees(21, 120, 3, 30, 4)
    od = O.Dataset(X, y)
    arrs = capi.build_batch([od.tune(t)["factors"] for t in trees])
    h = ctx.upload(X, y)
    c1, f1 = ctx.fitness(h, arrs)
    ctx.set_option("slab_budget_mb", 1)
    c2, f2 = ctx.fitness(h, arrs)
    ctx.set_option("slab_budget_mb", 32768)
    assert all(same_bits(a, b) for a, b in zip(c1, c2))
    assert same_bits(f1["e0"], f2["e0"]) and same_bits(f1["e1"], f2["e1"])
    ctx.free(h)


def test_bad_program_rejected_before_launch(ctx):
    X, y = make_data(1, 100, 2)
    h = ctx.upload(X, y)
    arrs = capi.build_batch([["x5"]])          # variable index out of range
    with pytest.raises(RuntimeError, match="out of range"):
        ctx.fitness(h, arrs, mode="raw")
    arrs = capi.build_batch([["x0"]])
    arrs["code"] = np.array([capi.D["RR_OP_BIN"]], dtype=np.uint32)  # binary op on empty accumulator
    with pytest.raises(RuntimeError):
        ctx.fitness(h, arrs, mode="raw")
    ctx.free(h)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_multi_dataset_batch_same_bits_as_solo(ctx, precision):
    """Candidates of three datasets (different n, d, y) in one rr_fitness_multi
    launch, interleaved, give the same bits as each dataset's own batch."""
    print("case: multi-dataset batch %s" % precision, flush=True)
    shapes = [(1500, 3, 31), (7000, 2, 32), (333, 4, 33)]
    hs, per_ds = [], []
    for n, d, seed in shapes:
        X, y = make_data(seed, n, d)
        od = O.Dataset(X, y)
        trees = treegen.random_trees(seed, 40, 3, 30, d)
        per_ds.append([od.tune(t)["factors"] for t in trees])
        hs.append(ctx.upload(X, y))
    for mode in ["ols", "raw"]:
        lists = per_ds if mode == "ols" else [[[f[0]] for f in fl if f] for fl in per_ds]
        solo = [ctx.fitness(h, capi.build_batch(fl), mode=mode, precision=precision) for h, fl in zip(hs, lists)]
        mixed, owner = [], []
        for i in range(max(len(fl) for fl in lists)):
            for s, fl in enumerate(lists):
                if i < len(fl):
                    mixed.append(fl[i])
                    owner.append((s, i))
        cm, fm = ctx.fitness(None, capi.build_batch(mixed), mode=mode, precision=precision,
                             handles=[hs[s] for s, _ in owner])
        for q, (s, i) in enumerate(owner):
            cs, fs = solo[s]
            assert same_bits([fm[q]["e0"], fm[q]["e1"], fm[q]["err"]], [fs[i]["e0"], fs[i]["e1"], fs[i]["err"]]), \
                (mode, s, i)
            assert fm[q]["flags"] == fs[i]["flags"] and fm[q]["rank"] == fs[i]["rank"]
            if mode == "ols":
                assert same_bits(cm[q], cs[i]), (s, i)
    for h in hs:
        ctx.free(h)


def test_autotune_keeps_fp64_bits(ctx):
    """Whatever schedule the autotuner picks, FP64 results are the same bits
    (the summation order does not depend on rows per thread)."""
    print("case: autotune fp64", flush=True)
    X, y = make_data(41, 20000, 4)
    trees = treegen.random_trees(41, 150, 3, 30, 4)
    od = O.Dataset(X, y)
    arrs = capi.build_batch([od.tune(t)["factors"] for t in trees])
    h = ctx.upload(X, y)
    ctx.set_option("fp64_eval_rows", 1)
    c1, f1 = ctx.fitness(h, arrs)
    ms = ctx.autotune(h, arrs, precision="fp64")
    assert ms > 0 and ctx.get_option("fp64_eval_rows") in (1, 2, 4) and ctx.get_option("fp64_eval_form") in (0, 1)
    c2, f2 = ctx.fitness(h, arrs)
    assert all(same_bits(a, b) for a, b in zip(c1, c2))
    assert same_bits(f1["e0"], f2["e0"]) and same_bits(f1["e1"], f2["e1"])
    ms32 = ctx.autotune(h, arrs, precision="fp32")
    assert ms32 > 0 and ctx.get_option("fp32_chunk_rows") in (2048, 4096, 8192, 16384)
    ctx.set_option("fp64_eval_rows", 2)
    ctx.set_option("fp64_eval_form", 1)
    ctx.set_option("fp32_rows", 2)
    ctx.set_option("fp32_chunk_rows", 4096)
    ctx.set_option("fp32_streams", 0)
    ctx.free(h)


def test_shared_factors_same_bits(ctx):
    """Candidates that repeat the same factors (equal programs, constants at
    different pool indexes), inside one candidate too, over two datasets in one
    launch, with candidates settled by the factor-0 pre-pass (ln x0 first over
    x0 < 0) sharing factors with live ones, and factors only such candidates
    use: every result is the same bits as the candidate scored alone, and the
    coefficients of candidates with finite columns are the oracle's QR
    solution of [factors, 1] against y."""
    print("case: shared factors, two datasets", flush=True)
    pool = ["sin x0", "* x0 c0x1p+1", "sqr + x1 c0x1.8p+1", "cos * x0 x1", "exp * x1 c0x1p-2",
            "* x0 c0x1.0000000000001p+1", "+ x0 c0x0p+0", "+ x0 c-0x0p+0", "/ x1 + sqr x0 c0x1p+0"]
    only_dead = ["sqrt x1", "sqr sin x1"]
    rng = np.random.default_rng(51)
    cands = []
    for i in range(160):
        f = [pool[j] for j in rng.choice(len(pool), size=int(rng.integers(1, 5)), replace=True)]
        if i % 7 == 0:
            f.append("x%d" % (i % 2))
        if i % 5 == 0:
            f = ["ln x0"] + f + [only_dead[i % 2]]
        cands.append(f)
    cands.append(["sin x0", "sin x0"])
    datasets = [make_data(52, 4100, 2), make_data(53, 9000, 2)]
    hs = [ctx.upload(X, y) for X, y in datasets]
    owner = [i % 2 for i in range(len(cands))]
    cm, fm = ctx.fitness(None, capi.build_batch(cands), handles=[hs[s] for s in owner])
    ods = [O.Dataset(X, y) for X, y in datasets]
    for q, (f, s) in enumerate(zip(cands, owner)):
        cs, fs = ctx.fitness(hs[s], capi.build_batch([f]))
        assert same_bits([fm[q]["e0"], fm[q]["e1"]], [fs[0]["e0"], fs[0]["e1"]]), (q, f)
        assert fm[q]["rank"] == fs[0]["rank"] and fm[q]["flags"] == fs[0]["flags"], (q, f)
        assert same_bits(cm[q], cs[0]), (q, f)
        cols = [ods[s].eval(p) for p in f] + [np.ones(datasets[s][1].size)]
        A = np.stack(cols, axis=1)
        if np.all(np.isfinite(A)):
            c, rank = O.qr_solve(A, datasets[s][1])
            assert same_bits(cm[q], c) and fm[q]["rank"] == rank, (q, f)
    assert any(np.isnan(c).all() for c in cm)   # the pre-pass settled some
    for h in hs:
        ctx.free(h)


def _shared_factor_batch(seed, count):
    """Candidates drawn from a small pool of factors (equal programs with
    constants at different pool indexes), some with a constant factor."""
    pool = ["sin x0", "* x0 c0x1p+1", "sqr + x1 c0x1.8p+1", "cos * x0 x1", "exp * x1 c0x1p-2", "sqrt x1",
            "/ x1 + sqr x0 c0x1p+0", "* sin x0 cos x1", "c0x1.8p+1"]
    rng = np.random.default_rng(seed)
    return [[pool[j] for j in rng.choice(len(pool), size=int(rng.integers(1, 6)), replace=False)]
            for _ in range(count)]


def test_shared_factors_across_slab_chunks_same_bits(ctx):
    """Kept columns are shared within a launch chunk only: with a 1 MB slab
    budget (a few candidates per chunk) the results are the same bits as in
    one chunk."""
    print("case: shared factors, many slab chunks", flush=True)
    X, y = make_data(61, 6000, 2)
    arrs = capi.build_batch(_shared_factor_batch(61, 300))
    h = ctx.upload(X, y)
    c1, f1 = ctx.fitness(h, arrs)
    ctx.set_option("slab_budget_mb", 1)
    c2, f2 = ctx.fitness(h, arrs)
    ctx.set_option("slab_budget_mb", 32768)
    ctx.free(h)
    assert all(same_bits(a, b) for a, b in zip(c1, c2))
    assert f1.tobytes() == f2.tobytes()


def test_shared_factors_checked_form_takes_fp64_bits(ctx):
    """RR_FP32_CHECKED plans FP64 launches over subsets of the batch (the
    candidates sent to FP64 up front, then the ones the FP32 form could not
    certify); on a batch that repeats its factors, every result it takes
    from the FP64 form is the plain FP64 form's, bit for bit."""
    print("case: shared factors, checked form", flush=True)
    X, y = make_data(62, 5000, 2)
    arrs = capi.build_batch(_shared_factor_batch(62, 300))
    h = ctx.upload(X, y)
    c64, f64 = ctx.fitness(h, arrs, precision="fp64")
    cc, fc = ctx.fitness(h, arrs, precision="fp32c")
    ctx.free(h)
    n64 = 0
    for i in range(len(fc)):
        if fc[i]["flags"] & 4:
            n64 += 1
            assert fc[i]["e0"].tobytes() == f64[i]["e0"].tobytes(), i
            assert fc[i]["e1"].tobytes() == f64[i]["e1"].tobytes(), i
            assert cc[i].tobytes() == c64[i].tobytes(), i
    assert n64 > 0   # the constant-factor candidates at least


@pytest.mark.parametrize("n", [2, 3, 4, 5, 9, 300, 4097])
def test_sparse_columns_and_tiny_n_bitexact(ctx, n):
    """The QR's last two steps on the edge cases they branch on: columns that
    are zero below row 0 or 1 (an identity reflector, tau = 0, at the step
    before the last), a single row left (n - p == 1), and n at or just above
    the column count."""
    print("case: sparse columns n=%d" % n, flush=True)
    rng = np.random.default_rng(70 + n)
    X = np.zeros((n, 4))
    X[:, 0] = rng.uniform(-3, 3, n)
    X[0, 1] = 2.5                      # zero below row 0
    X[:2, 2] = [1.5, -0.75]            # zero below row 1
    X[:, 3] = rng.uniform(0.5, 2.0, n)
    y = 1.5 * X[:, 0] - 0.5 * X[:, 3] + rng.normal(0, 0.01, n)
    trees = ["x1", "x2", "+ x1 x0", "+ x2 x0", "+ x1 x2", "+ + x0 x1 x2", "+ + x1 x2 x3", "* x1 c0x1p+1",
             "+ x0 x3", "+ + x0 x3 sqr x1", "+ + + x0 x1 x2 x3", "+ sin x1 x0", "+ sqr x2 x1"]
    od = O.Dataset(X, y)
    tuned = [od.tune(t) for t in trees]
    arrs = capi.build_batch([tu["factors"] for tu in tuned])
    h = ctx.upload(X, y)
    coefs, fit = ctx.fitness(h, arrs, mode="ols")
    ctx.free(h)
    for t, tu, c, f in zip(trees, tuned, coefs, fit):
        assert same_bits(c, tu["coefs"]), (t, c, tu["coefs"])
        assert f["rank"] == tu["rank"], t
        assert same_bits([f["e0"], f["e1"]], [tu["fit"][0], tu["fit"][1]]), (t, f, tu["fit"])


def wide_trees(rng, d, count, lo=10, hi=20):
    """Sums of lo..hi-1 distinct terms over d variables: candidates of more
    than ten columns (with the free term), which take the step-synchronous QR."""
    pool = []
    for i in range(d):
        pool += ["x%d" % i, "sin x%d" % i, "cos x%d" % i, "sqr x%d" % i, "exp * c0x1p-2 x%d" % i]
        pool += ["* x%d x%d" % (i, j) for j in range(i + 1, d)]
    trees = []
    for _ in range(count):
        m = int(rng.integers(lo, hi))
        terms = [pool[i] for i in rng.choice(len(pool), m, replace=False)]
        trees.append("+ " * (m - 1) + " ".join(terms))
    return trees


@pytest.mark.parametrize("n", [7, 12, 150, 4096, 4097, 9000])
def test_wide_candidates_bitexact(ctx, n):
    """Candidates of 11 to 20 columns: the whole QR in one launch when every
    candidate's rows fit one chunk (n <= 4096), launches per step beyond;
    n below the column count stops after n steps."""
    print("case: wide candidates n=%d" % n, flush=True)
    rng = np.random.default_rng(90 + n)
    X, y = make_data(90 + n, n, 4)
    trees = wide_trees(rng, 4, 40)
    od = O.Dataset(X, y)
    tuned = [od.tune(t) for t in trees]
    assert all(len(tu["factors"]) >= 10 for tu in tuned)
    arrs = capi.build_batch([tu["factors"] for tu in tuned])
    h = ctx.upload(X, y)
    coefs, fit = ctx.fitness(h, arrs, mode="ols")
    ctx.free(h)
    for t, tu, c, f in zip(trees, tuned, coefs, fit):
        assert same_bits(c, tu["coefs"]), (t, c, tu["coefs"])
        assert f["rank"] == tu["rank"], t
        assert same_bits([f["e0"], f["e1"]], [tu["fit"][0], tu["fit"][1]]), (t, f, tu["fit"])


@pytest.mark.parametrize("sizes", [(150, 3000), (150, 5000)])
def test_wide_candidates_of_several_datasets_bitexact(ctx, sizes):
    """Wide candidates of two datasets interleaved in one launch: each its own
    dataset's rows, the whole QR in one launch when both fit one chunk, per
    step when one does not."""
    print("case: wide candidates of datasets %s" % (sizes,), flush=True)
    hs, tuned, owner = [], [], []
    for s, n in enumerate(sizes):
        rng = np.random.default_rng(190 + n)
        X, y = make_data(190 + n, n, 3)
        od = O.Dataset(X, y)
        tuned.append([od.tune(t) for t in wide_trees(rng, 3, 20, 10, 16)])
        hs.append(ctx.upload(X, y))
    mixed = []
    for i in range(20):
        for s in range(len(sizes)):
            mixed.append(tuned[s][i]["factors"])
            owner.append((s, i))
    assert all(len(f) >= 10 for f in mixed)
    coefs, fit = ctx.fitness(None, capi.build_batch(mixed), mode="ols", handles=[hs[s] for s, _ in owner])
    for h in hs:
        ctx.free(h)
    for q, (s, i) in enumerate(owner):
        tu = tuned[s][i]
        assert same_bits(coefs[q], tu["coefs"]), (s, i)
        assert fit[q]["rank"] == tu["rank"], (s, i)
        assert same_bits([fit[q]["e0"], fit[q]["e1"]], [tu["fit"][0], tu["fit"][1]]), (s, i)


def test_phase_timing_and_early_flag(ctx):
    """Option phase_timing splits the kernel time of a call by phase; the
    phases of the plain FP64 form (one stream) add up to no more than the
    call's kernel time.  Candidates the factor-0 pre-pass settles carry
    RR_F_EARLY and are sentinels; no other candidate carries it."""
    print("case: phase timing", flush=True)
    X, y = make_data(81, 20000, 3)
    trees = treegen.random_trees(81, 200, 3, 30, 3) + ["ln x0", "+ sqrt x1 x2"]
    od = O.Dataset(X, y)
    tuned = [od.tune(t) for t in trees]
    arrs = capi.build_batch([tu["factors"] for tu in tuned])
    h = ctx.upload(X, y)
    ctx.set_option("phase_timing", 1)
    try:
        coefs, fit = ctx.fitness(h, arrs)
        ph = ctx.phase_ms()
        total = ctx.kernel_ms()
        _, fit32 = ctx.fitness(h, arrs, precision="fp32")
        ph32 = ctx.phase_ms()
    finally:
        ctx.set_option("phase_timing", 0)
    ctx.free(h)
    print("phases:", ph, "total", total, "fp32:", ph32, flush=True)
    for k in ("prepass", "eval", "qr", "score", "host_check", "host_plan"):
        assert ph[k] > 0, k
    assert ph["fp32"] == 0 and ph["host_tail"] >= 0
    assert sum(ph[k] for k in ("prepass", "eval", "qr", "score")) <= total * 1.05 + 0.01
    assert ph32["fp32"] > 0 and ph32["prepass"] > 0
    early = (fit["flags"] & capi.D["RR_F_EARLY"]) != 0
    assert early.any() and np.all(fit["flags"][early] & 1)
    assert np.array_equal(early, (fit32["flags"] & capi.D["RR_F_EARLY"]) != 0)
    ln_x0 = len(trees) - 2
    assert early[ln_x0]     # ln of a negative x0 within the first rows
    for t, tu, c, f in zip(trees, tuned, coefs, fit):   # the flag does not change any result
        assert same_bits(c, tu["coefs"]) and same_bits([f["e0"], f["e1"]], [tu["fit"][0], tu["fit"][1]]), t


def test_graph_replays_same_bits(ctx):
    """Option graph: the plain FP64 form's launches go out as an executable
    graph, kept per launch sequence and updated with each call's arguments.
    Calls of different shapes (OLS batches of different sizes, a RAW batch)
    with eager calls between the replays: every replay gives the eager bits,
    and repeated shapes reuse their executable graph."""
    print("case: graph replays", flush=True)
    X, y = make_data(91, 20000, 4)
    od = O.Dataset(X, y)
    h = ctx.upload(X, y)
    tuned_a = [od.tune(t) for t in treegen.random_trees(91, 300, 3, 40, 4)]
    tuned_b = [od.tune(t) for t in treegen.random_trees(92, 80, 3, 20, 4)]
    arr_a = capi.build_batch([tu["factors"] for tu in tuned_a])
    arr_b = capi.build_batch([tu["factors"] for tu in tuned_b])
    raw = capi.build_batch([[t] for t in treegen.random_trees(93, 200, 3, 30, 4)])
    eager = {"a": ctx.fitness(h, arr_a), "b": ctx.fitness(h, arr_b), "raw": ctx.fitness(h, raw, mode="raw")}
    arrays = {"a": arr_a, "b": arr_b, "raw": raw}
    ctx.set_option("graph", 1)
    try:
        made0, upd0 = ctx.get_option("graph_made"), ctx.get_option("graph_updated")
        for step, name in enumerate(["a", "b", "a", "raw", "a", "b", "raw", "a"]):
            mode = "raw" if name == "raw" else "ols"
            c, f = ctx.fitness(h, arrays[name], mode=mode)
            ce, fe = eager[name]
            assert same_bits(f["e0"], fe["e0"]) and same_bits(f["e1"], fe["e1"]), (step, name)
            if mode == "ols":
                assert all(same_bits(p, q) for p, q in zip(c, ce)), (step, name)
            ctx.set_option("graph", 0)                 # eager work between the replays
            c2, f2 = ctx.fitness(h, arrays[name], mode=mode)
            assert same_bits(f2["e0"], fe["e0"]), (step, name)
            ctx.set_option("graph", 1)
        made, upd = ctx.get_option("graph_made") - made0, ctx.get_option("graph_updated") - upd0
        print("graphs made", made, "updated", upd, flush=True)
        assert made >= 1 and upd >= 1 and made + upd == 8
    finally:
        ctx.set_option("graph", 0)
    for tu, c, f in zip(tuned_a, *eager["a"]):            # and the eager bits are the oracle's
        assert same_bits(c, tu["coefs"]) and same_bits([f["e0"], f["e1"]], [tu["fit"][0], tu["fit"][1]])
    ctx.free(h)


def test_pipelined_calls_same_bits(ctx):
    """rr_fitness_submit / rr_fitness_wait: OLS and RAW batches of different
    sizes, two in flight at a time, give rr_fitness_batch's bits; a third
    submit while two are pending is refused; a synchronous call completes the
    pending ones first; with phase timing on, submit runs the call at once."""
    print("case: pipelined calls n=20000 d=4", flush=True)
    X, y = make_data(91, 20000, 4)
    trees = treegen.random_trees(91, 300, 3, 40, 4)
    od = O.Dataset(X, y)
    facs = [od.tune(t)["factors"] for t in trees]
    h = ctx.upload(X, y)
    big = capi.build_batch(facs)
    small = capi.build_batch(facs[::3][:70])
    raw = capi.build_batch([[t] for t in trees[:100]])
    want = {"big": ctx.fitness(h, big), "small": ctx.fitness(h, small), "raw": ctx.fitness(h, raw, mode="raw")}

    def assert_same(got, exp):
        (cg, fg), (cw, fw) = got, exp
        assert len(cg) == len(cw)
        for a, b in zip(cg, cw):
            assert same_bits(a, b)
        assert fg.tobytes() == fw.tobytes()

    seq = [("big", big, "ols"), ("small", small, "ols"), ("raw", raw, "raw"), ("big", big, "ols"),
           ("small", small, "ols")]
    pending = []
    for name, arrs, mode in seq:
        pending.append((ctx.submit(h, arrs, mode), name))
        if len(pending) == 2:
            ctx.wait()
            r, name0 = pending.pop(0)
            assert_same(r(), want[name0])
    ctx.wait()
    r, name0 = pending.pop(0)
    assert_same(r(), want[name0])
    a = ctx.submit(h, small)
    b = ctx.submit(h, big)
    with pytest.raises(RuntimeError, match="two calls are pending"):
        ctx.submit(h, small)
    assert_same(ctx.fitness(h, small), want["small"])   # completes both pending calls first
    assert_same(a(), want["small"])
    assert_same(b(), want["big"])
    ctx.wait()                                           # each submit is still retired by its wait
    ctx.wait()
    with pytest.raises(RuntimeError, match="no pipelined call"):
        ctx.wait()
    ctx.set_option("phase_timing", 1)
    try:
        r = ctx.submit(h, big)
        assert_same(r(), want["big"])                    # written by the submit itself
        ctx.wait()
    finally:
        ctx.set_option("phase_timing", 0)
    ctx.free(h)


def test_repeated_candidates_take_the_same_results(ctx):
    """Candidates whose factor programs are the same (constants compared by
    value) are launched once and the others take the results: every result is
    still the oracle's, synchronously and pipelined; a constant one bit apart
    is a different factor."""
    print("case: repeated candidates n=9000 d=3", flush=True)
    X, y = make_data(77, 9000, 3)
    trees = ["+ sin x0 * x1 x2", "exp * x0 c0x1p-2", "+ + sin x0 * x1 x2 c0x1.8p+1", "+ sin x0 * x1 x2",
             "exp * x0 c0x1.0000000000001p-2", "* c0x1.4p+1 exp * x0 c0x1p-2", "ln x0", "ln x0",
             "+ sqrt x2 x0", "+ x0 sqrt x2", "+ sqrt x2 x0"]
    od = O.Dataset(X, y)
    tuned = [od.tune(t) for t in trees]
    arrs = capi.build_batch([tu["factors"] for tu in tuned])
    h = ctx.upload(X, y)
    got = [ctx.fitness(h, arrs)]
    r = ctx.submit(h, arrs)
    ctx.wait()
    got.append(r())
    for coefs, fit in got:
        for t, tu, c, f in zip(trees, tuned, coefs, fit):
            assert same_bits(c, tu["coefs"]), t
            assert same_bits([f["e0"], f["e1"]], [tu["fit"][0], tu["fit"][1]]), t
        assert fit[0].tobytes() == fit[2].tobytes() == fit[3].tobytes()
        assert fit[1].tobytes() == fit[5].tobytes()
        assert fit[8].tobytes() == fit[10].tobytes()
    assert tuned[4]["factors"] != tuned[1]["factors"]
    ctx.free(h)


# row groups of 64 and 256 around their edges, tables whose columns do and do
# not fit a workgroup's LDS, one column a lane up to 64 and one more
@pytest.mark.parametrize("n", [11, 64, 65, 150, 256, 257, 600, 700])
def test_wide_candidates_of_small_tables_bitexact(ctx, n):
    """The one-workgroup QR of wide candidates on small tables: coefficients
    and rank of the oracle's QR over 10 to 66 columns, with columns that are
    zero below row 0 or 1, repeated, constant, NaN or infinite among them."""
    print("case: wide candidates of small tables n=%d" % n, flush=True)
    rng = np.random.default_rng(290 + n)
    X, y = make_data(290 + n, n, 5)
    X[:, 3] = 0.0
    X[0, 3] = 2.5
    X[:, 4] = 0.0
    X[:2, 4] = [1.5, -0.75]
    pool = ["sin * x%d c0x%dp-1" % (i, m) for i in range(3) for m in range(1, 10)]
    pool += ["exp * x%d c0x%dp-4" % (i, m) for i in range(3) for m in range(1, 10)]
    pool += ["sqr x0", "sqr x1", "* x0 x1", "* x1 x2", "x0", "x1", "x2", "cos x0", "cos x1", "cos x2"]
    special = ["x3", "x4", "+ x0 c0x0p+0", "x0", "c0x1.8p+1", "ln x1", "exp * x2 c0x1p+9"]
    cands = []
    for width in [9, 10, 13, 20, 63, 64, 65]:
        for plain in (True, True, False, False, False):
            f = [pool[i] for i in rng.choice(len(pool), min(width, len(pool)), replace=False)]
            while len(f) < width:
                f.append("sin + x0 c0x%dp+0" % len(f))
            if not plain:
                for s in rng.choice(len(special), 2, replace=False):
                    f[int(rng.integers(1, width))] = special[s]
            cands.append(f)
    od = O.Dataset(X, y)
    h = ctx.upload(X, y)
    coefs, fit = ctx.fitness(h, capi.build_batch(cands), mode="ols")
    alone = [ctx.fitness(h, capi.build_batch([f]), mode="ols") for f in cands]
    ctx.free(h)
    for f, c, ft, (ca, fa) in zip(cands, coefs, fit, alone):
        o, rank = O.qr_solve(np.stack([od.eval(p) for p in f] + [np.ones(n)], axis=1), y)
        assert same_bits(c, o), (len(f), f, c, o)
        assert ft["rank"] == rank, (len(f), f)
        assert same_bits(ca[0], o) and fa[0]["rank"] == rank, (len(f), f)
        assert same_bits([ft["e0"], ft["e1"]], [fa[0]["e0"], fa[0]["e1"]]), (len(f), f)


@pytest.mark.parametrize("form,rows", [(1, 1), (1, 2), (1, 4), (0, 2)])
def test_raw_eval_forms_bitexact(ctx, form, rows):
    """Raw scoring through both interpreters, over a ragged last chunk, with
    programs of stack depth up to 4 (beyond form 1's LDS at 4 rows: form 0)."""
    print("case: raw form %d rows=%d" % (form, rows), flush=True)
    X, y = make_data(62, 9001, 4)
    rng = np.random.default_rng(62)
    trees = treegen.random_trees(62, 60, 1, 40, 4) + [_full_tree(rng, lv, 4) for lv in (2, 3, 4, 5, 6, 7)]
    od = O.Dataset(X, y)
    h = ctx.upload(X, y)
    try:
        ctx.set_option("fp64_eval_rows", rows)
        ctx.set_option("fp64_eval_form", form)
        for batch in (trees[:60], trees):
            _, fit = ctx.fitness(h, capi.build_batch([[t] for t in batch]), mode="raw")
            for t, f in zip(batch, fit):
                e0, e1, _ = od.score(t)
                assert same_bits([f["e0"], f["e1"]], [e0, e1]), t
    finally:
        ctx.set_option("fp64_eval_rows", 2)
        ctx.set_option("fp64_eval_form", 1)
    ctx.free(h)


@pytest.mark.parametrize("sizes", [(1, 64), (150, 150), (4096, 4097), (9000, 33)])
def test_small_raw_batches_bitexact(ctx, sizes):
    """Raw calls of 1 to 60 trees: the smallest go out with their inputs in
    the launch's argument, the others staged; synchronous, pipelined and over
    two datasets, with one chunk of rows and several."""
    print("case: small raw batches n=%s" % (sizes,), flush=True)
    data = [make_data(90 + i, n, 3) for i, n in enumerate(sizes)]
    hs = [ctx.upload(X, y) for X, y in data]
    ods = [O.Dataset(X, y) for X, y in data]
    trees = treegen.random_trees(91, 60, 1, 40, 3)
    want = [[od.score(t)[:2] for t in trees] for od in ods]

    def check(fit, expected):
        for f, (e0, e1) in zip(fit, expected):
            assert same_bits([f["e0"], f["e1"]], [e0, e1])
    for count in (1, 2, 5, 9, 10, 11, 12, 13, 14, 15, 16, 20, 30, 60):
        arrs = capi.build_batch([[t] for t in trees[:count]])
        check(ctx.fitness(hs[0], arrs, mode="raw")[1], want[0])
        which = [i % 2 for i in range(count)]
        _, fit = ctx.fitness(None, arrs, mode="raw", handles=[hs[w] for w in which])
        check(fit, [want[w][i] for i, w in enumerate(which)])
        first = ctx.submit(hs[1], arrs, mode="raw")
        second = ctx.submit(hs[0], capi.build_batch([[t] for t in trees[::-1]]), mode="raw")
        ctx.wait()
        third = ctx.submit(hs[0], arrs, mode="raw")
        check(first()[1], want[1])
        ctx.wait()
        check(second()[1], want[0][::-1])
        ctx.wait()
        check(third()[1], want[0])
    for h in hs:
        ctx.free(h)


@pytest.mark.parametrize("n", [513, 4097])
@pytest.mark.parametrize("levels", [4, 5, 6, 8])
def test_deep_stacks_at_four_rows_bitexact(ctx, n, levels):
    """Programs whose operand stack fits the LDS slots of four rows a thread
    beside programs that take one row at a time."""
    print("case: deep stacks n=%d levels=%d" % (n, levels), flush=True)
    rng = np.random.default_rng(levels)
    X, y = make_data(70 + levels, n, 4)
    trees = ["* sin %s x1" % _full_tree(rng, L, 4) for L in (1, 2, 3, levels, levels)]
    od = O.Dataset(X, y)
    tuned = [od.tune(t) for t in trees]
    keep = ctx.get_option("fp64_eval_rows")
    ctx.set_option("fp64_eval_rows", 4)
    h = ctx.upload(X, y)
    coefs, fit = ctx.fitness(h, capi.build_batch([tu["factors"] for tu in tuned]), mode="ols")
    ctx.set_option("fp64_eval_rows", keep)
    ctx.free(h)
    for t, tu, c, f in zip(trees, tuned, coefs, fit):
        assert same_bits(c, tu["coefs"]), (t, c, tu["coefs"])
        assert same_bits([f["e0"], f["e1"]], [tu["fit"][0], tu["fit"][1]]), (t, f, tu["fit"])


def test_shared_context_is_at_its_defaults(ctx):
    """After the tests above, which set options, the shared context still has
    a new context's options."""
    import conftest
    fresh = capi.Context(0)
    want = {k: fresh.get_option(k) for k in conftest.OPTIONS}
    fresh.close()
    assert {k: ctx.get_option(k) for k in conftest.OPTIONS} == want


@pytest.mark.parametrize("rows", [1, 2, 4])
@pytest.mark.parametrize("n", [150, 600, 4097, 9000])
def test_small_raw_batches_at_every_row_count(ctx, n, rows):
    """Raw calls with their inputs in the launch's argument and staged ones at
    one, two and four rows a thread."""
    print("case: small raw batches n=%d rows=%d" % (n, rows), flush=True)
    X, y = make_data(97, n, 3)
    od = O.Dataset(X, y)
    trees = treegen.random_trees(98, 60, 1, 40, 3)
    want = [od.score(t)[:2] for t in trees]
    h = ctx.upload(X, y)
    ctx.set_option("fp64_eval_rows", rows)
    for count in (1, 5, 60):
        _, fit = ctx.fitness(h, capi.build_batch([[t] for t in trees[:count]]), mode="raw")
        for t, f, w in zip(trees, fit, want):
            assert same_bits([f["e0"], f["e1"]], w), t
    ctx.free(h)


def test_register_stack_form_keeps_to_two_rows(ctx):
    """fp64_eval_form 0 at the default four rows a thread runs at two, which
    its registers hold: the time of two rows asked for (spilled, four rows
    take three to seven times as long)."""
    print("case: register stack form, raw and OLS, n=50021", flush=True)
    X, y = make_data(99, 50021, 4)
    trees = treegen.random_trees(100, 100, 10, 30, 4)
    od = O.Dataset(X[:100], y[:100])
    h = ctx.upload(X, y)
    ctx.set_option("fp64_eval_form", 0)
    for mode, arrs in (("raw", capi.build_batch([[t] for t in trees])),
                       ("ols", capi.build_batch([od.tune(t)["factors"] for t in trees]))):
        best = {}
        for rows in (2, 4):
            ctx.set_option("fp64_eval_rows", rows)
            times = []
            for _ in range(6):
                ctx.fitness(h, arrs, mode=mode)
                times.append(ctx.kernel_ms())
            best[rows] = min(times)
        assert best[4] < 2 * best[2], (mode, best)
    ctx.free(h)


def _comb_batch(progs):
    """Raw trees `op v0 (op v1 (... vk))` in the order written (left operand
    first), which takes a stack slot per operator: few instructions, many
    slots.  progs: (operators, variables) pairs; returns the batch and the
    trees in prefix form."""
    code, starts, trees = [], [0], []
    for ops, xs in progs:
        for x in xs[:-1]:
            code += [(x << 8) | capi.D["RR_OP_LDV"], capi.D["RR_OP_PUSH"]]
        code.append((xs[-1] << 8) | capi.D["RR_OP_LDV"])
        code += [capi.D["RR_OP_BIN"] + 8 * capi.BINARY[op] + capi.D["RR_M_S"] for op in reversed(ops)]
        starts.append(len(code))
        trees.append(" ".join("%s x%d" % p for p in zip(ops, xs)) + (" x%d" % xs[-1]))
    arrs = {"cand_start": np.arange(len(progs) + 1, dtype=np.int32), "prog_start": np.array(starts, dtype=np.int32),
            "code": np.array(code, dtype=np.uint32), "consts": np.zeros(1), "n_consts": 0, "n_cands": len(progs)}
    return arrs, trees


# one to three chunks of rows; row counts that take two and four rows a thread
@pytest.mark.parametrize("form,rows", [(1, 4), (1, 2), (1, 1), (0, 4), (0, 1)])
@pytest.mark.parametrize("n", [512, 513, 4097, 9001])
def test_raw_deep_stacks_bitexact(ctx, n, form, rows):
    """Raw trees of 1 to 8 stack slots (8 is the most a program may take; form
    1's LDS is sized by the call's deepest tree, up to 64 KiB), in calls small
    enough for the launch's argument and staged ones, over two datasets,
    pipelined and without allocation."""
    print("case: raw deep stacks n=%d form=%d rows=%d" % (n, form, rows), flush=True)
    assert capi.D["RR_MAX_STACK"] == 8
    rng = np.random.default_rng(n)
    progs = [([str(o) for o in rng.choice(["+", "-", "*", "max", "min"], slots)],
              [int(x) for x in rng.integers(0, 4, slots + 1)])
             for slots in (3, 8, 1, 4, 7, 2, 5, 6, 8, 3)] * 10
    data = [make_data(95, n, 4), make_data(96, 150, 4)]
    ods = [O.Dataset(X, y) for X, y in data]
    hs = [ctx.upload(X, y) for X, y in data]
    ctx.set_option("fp64_eval_rows", rows)
    ctx.set_option("fp64_eval_form", form)

    def check(fit, trees, which):
        for t, f, w in zip(trees, fit, which):
            e0, e1, _ = ods[w].score(t)
            assert same_bits([f["e0"], f["e1"]], [e0, e1]), (w, t)
    seven = [p for p in progs if len(p[0]) < 8]
    for part in (progs[:1], seven[:8], seven, progs[:2], progs[:10], progs):
        arrs, trees = _comb_batch(part)
        check(ctx.fitness(hs[0], arrs, mode="raw")[1], trees, [0] * len(part))
        check(ctx.fitness_noalloc(hs[0], arrs, mode="raw")[1], trees, [0] * len(part))
        which = [i % 2 for i in range(len(part))]
        check(ctx.fitness(None, arrs, mode="raw", handles=[hs[w] for w in which])[1], trees, which)
        pending = ctx.submit(hs[0], arrs, mode="raw")
        ctx.wait()
        check(pending()[1], trees, [0] * len(part))
    for h in hs:
        ctx.free(h)
