"""predict_proba of host rows in row chunks: how many chunks a call takes,
and that any number of them gives the probabilities of the whole matrix."""
import numpy as np
import pytest

from conftest import make_data

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model():
    from bsscl_gbm import HybridHistGBMNumbaV1_0_1
    X, y = make_data(3000, 20, seed=5, nan_frac=0.1, nan_cols=[0, 3])
    return HybridHistGBMNumbaV1_0_1(n_estimators=12, max_depth=4, random_state=3,
                                    verbose=False).fit(X, y)


# (rows, chunks): up to 16 MB of X go as one; then an eighth of X between 8
# and 64 MB, rounded up to whole 1,024 rows.
@pytest.mark.parametrize("n,chunks", [(1, 1), (1024, 1), (1025, 1), (1500, 1), (10_000, 1),
                                      (65_000, 1), (209_715, 1), (209_716, 2), (300_001, 3),
                                      (1_000_000, 8)])
def test_rows_go_in_as_few_chunks(model, n, chunks):
    from bsscl_gbm import estimator as est_mod
    print(f"[case] {n} x 20 in {chunks} chunks", flush=True)
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 20)).astype(np.float32)
    eng = est_mod._engine(0)
    packed = {"features": model._packed_features, "thresholds": model._packed_thresholds,
              "values": model._packed_values, "left": model._packed_left,
              "right": model._packed_right, "offsets": model._tree_offsets}
    eng.bin_features(1, X, model.bin_edges, model.feature_bin_counts, model._nan_bin_id)
    want = eng.predict_proba(1, n, packed, len(model.trees), model.learning_rate,
                             model.base_score_)
    eng.set_profiling(1)
    try:
        got = model.predict_proba(X)
        launches = eng.stats()["predict_launches"]
    finally:
        eng.set_profiling(0)
    np.testing.assert_array_equal(got, want)
    assert launches == chunks


@pytest.mark.parametrize("case", ["f32", "f64", "bins_300", "class_without_trees", "one_chunk"])
def test_multiclass_chunks_equal_the_whole_matrix(engine, monkeypatch, case):
    """bsscl_predict_proba_mc_rows over many chunks, the last one ragged (its
    score columns lie closer together), equals bsscl_bin_features and
    bsscl_predict_proba_mc bit for bit; matrix slot 1 keeps its codes."""
    from bsscl_gbm import HybridHistGBMNumbaV1_0_1
    from bsscl_gbm import estimator as est_mod
    print(f"[case] multiclass chunks {case}", flush=True)
    rng = np.random.default_rng(9)
    F, K = 7, 5
    X = rng.standard_normal((4000, F)).astype(np.float32)
    y = (X @ rng.standard_normal((F, K)) + rng.gumbel(size=(4000, K))).argmax(1)
    X[rng.random(X.shape) < 0.05] = np.nan
    m = HybridHistGBMNumbaV1_0_1(n_estimators=6, max_depth=5, random_state=3, verbose=False,
                                 n_bins=300 if case == "bins_300" else 255).fit(X, y)
    n = 21_777
    Xp = rng.standard_normal((n, F)) * 1.5
    Xp[rng.random(Xp.shape) < 0.05] = np.nan
    Xp = Xp if case == "f64" else Xp.astype(np.float32)
    packs, counts = list(m._mc_packed), [len(t) for t in m.mc_trees]
    if case == "class_without_trees":
        packs[1], counts[1] = None, 0
    eng = est_mod._engine(0)
    eng.bin_features(1, Xp, m.bin_edges, m.feature_bin_counts, m._nan_bin_id)
    want = eng.predict_proba_mc(1, n, packs, counts, m.learning_rate)
    codes = eng.get_codes(1, n, F)
    if case != "one_chunk":
        monkeypatch.setenv("BSSCL_TEST_PREDICT_CHUNK_ROWS", "4096")  # six chunks
    eng.set_profiling(1)
    try:
        got = eng.predict_proba_mc_rows(Xp, m.bin_edges, m.feature_bin_counts, m._nan_bin_id,
                                        packs, counts, m.learning_rate)
        launches = eng.stats()["predict_launches"]
    finally:
        eng.set_profiling(0)
    np.testing.assert_array_equal(got, want)
    assert launches == (1 if case == "one_chunk" else 6)
    np.testing.assert_array_equal(eng.get_codes(1, n, F), codes)


@pytest.mark.parametrize("piece", [0, 1, 2])
def test_failed_upload_leaves_nothing_behind(model, monkeypatch, piece):
    """A call whose upload fails after some of its pieces, on either copy
    stream, returns the error with its streams idle: the next call, whose
    rows take the same buffers at once, gets its own probabilities."""
    print(f"[case] upload fails after piece {piece}", flush=True)
    rng = np.random.default_rng(3)
    X = rng.standard_normal((300_001, 20)).astype(np.float32)
    want = model.predict_proba(X)
    monkeypatch.setenv("BSSCL_TEST_UPLOAD_FAIL", str(piece))
    with pytest.raises(RuntimeError, match="BSSCL_TEST_UPLOAD_FAIL"):
        model.predict_proba(-X)
    monkeypatch.delenv("BSSCL_TEST_UPLOAD_FAIL")
    np.testing.assert_array_equal(model.predict_proba(X), want)
