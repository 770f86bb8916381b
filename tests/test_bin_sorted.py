"""Binning against ascending edges in LDS (k_bin_sorted) against the oracle's
binning, code by code, at its tile, bin-count and column-chunk edges, and
with values on, next to and beyond the edges; edges that do not ascend take
the general kernel and give the same codes."""
import numpy as np
import pytest

from oracle import model as om

pytestmark = pytest.mark.gpu


def _edges(rng, nb, dtype):
    """nb + 1 ascending edges, float64 values between float32 neighbours
    among them, some equal."""
    e = np.sort(rng.standard_normal(nb + 1)) * rng.choice([1e-40, 1.0, 1e30])
    if dtype == np.float32:  # float32 edges, as a float32 column's fit has them
        e[::2] = e[::2].astype(np.float32)
    if nb > 4:
        e[2] = e[1]
    return np.sort(e)


def _values(rng, n, e, dtype):
    with np.errstate(over="ignore"):
        near = rng.choice(e, n).astype(dtype)
    pick = rng.integers(0, 5, n)
    v = np.where(pick == 0, near, np.nextafter(near, dtype(np.inf)))
    v = np.where(pick == 1, np.nextafter(near, dtype(-np.inf)), v)
    v = np.where(pick == 2, (rng.standard_normal(n) * np.abs(e).max()).astype(dtype), v)
    odd = np.array([np.inf, -np.inf, 0.0, -0.0, np.nan, np.finfo(dtype).max,
                    np.finfo(dtype).tiny / 8], dtype)
    return np.where(rng.random(n) < 0.05, rng.choice(odd, n), v).astype(dtype)


# (rows, bin counts by column in turn, columns, dtype, NaN columns)
CASES = {
    "one_row": (1, [5], 1, np.float32, 0),
    "rows_255": (255, [255], 7, np.float32, 3),
    "rows_257": (257, [256, 1, 2], 9, np.float32, 9),
    "tiers_257": (1000, [257, 40], 31, np.float32, 2),
    "levels_512": (513, [512, 511], 33, np.float32, 1),
    "too_many_bins": (513, [513], 5, np.float32, 1),
    "f64": (777, [255, 300], 17, np.float64, 5),
    "wide": (600, [63, 64, 65], 120, np.float32, 40),
    "many_tiles": (300_001, [128], 12, np.float32, 4),
    "many_tiles_chunks": (140_003, [256], 50, np.float64, 10),
}


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("ascending", [True, False])
def test_bin_sorted_equals_oracle(engine, case, ascending):
    n, counts, F, dtype, n_nan = CASES[case]
    print(f"[case] bin {case}: {n} x {F} {np.dtype(dtype).name}, ascending={ascending}", flush=True)
    rng = np.random.default_rng(n + F)
    nb = np.array([counts[j % len(counts)] for j in range(F)], np.int32)
    E = np.zeros((F, int(nb.max()) + 2))
    X = np.empty((n, F), dtype)
    for j in range(F):
        e = _edges(rng, int(nb[j]), dtype)
        X[:, j] = _values(rng, n, e, dtype)
        E[j, :len(e)], E[j, len(e):] = e, e[-1]
    if not ascending:
        E[0, :2] = E[0, 1::-1]
        E[F - 1, nb[F - 1]] = np.nan
    nan_id = np.full(F, -1, np.int32)
    nan_id[rng.permutation(F)[:n_nan]] = 0
    if n_nan == 0:
        X = np.nan_to_num(X, nan=0.5)
    engine.bin_features(1, X, E, nb, nan_id)
    got = engine.get_codes(1, n, F, u16=True)
    want = om.bin_features(X, E, nb, nan_id, "standard").astype(np.int64)
    # (A value above a NaN feature's last edge has the code nb, which the
    # tiers hold up to 255 each.)
    tiers = max(1 if b <= 256 else (int(b) - 2) // 255 + 1 for b in nb)
    np.testing.assert_array_equal(got, np.minimum(want, 255 * tiers))
