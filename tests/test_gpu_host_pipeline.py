"""Host batches of several pieces and chunks: features are sent piece by piece while later pieces are gathered, chunk by chunk on
two streams. Rows and columns at the edges of pieces and chunks against the oracle. Needs an MI355X."""
import threading

import numpy as np
import pytest

import catboost_amd as cb
from oracle import model_builder as mb
from oracle.oracle import OracleModel

pytestmark = pytest.mark.gpu


def _model(rng, n_float, one_hot=False):
    ffs = [mb.float_feature(i, i) for i in range(n_float)]
    cats = [mb.cat_feature(0, n_float)] if one_hot else []
    trees = []
    for t in range(8):
        splits = [("float", int(f), float(np.float32(b))) for f, b in zip(rng.integers(0, n_float, 4), rng.normal(size=4))]
        splits.append(("float", max(0, n_float - 1 - t % 2), float(np.float32(0.1 * t - 0.4))))  # the last column is read
        if one_hot:
            splits[t % 5] = ("onehot", 0, 1 + t % 3)
        trees.append((splits, rng.normal(size=32)))
    model = mb.build_oblivious(ffs, cats, 1, trees, bias=[0.5])
    m = cb.ModelCalcer()
    m.load_from_dict(model)
    m.enable_gpu_evaluation(0)
    return m, OracleModel(model)


# 200 floats: a unit is 327 rows, a chunk of 64 MB 83 712; 7 floats: units of 9362 rows
@pytest.mark.parametrize("n_float,docs", [(200, 2620), (200, 2621), (200, 327 * 8), (200, 20_931), (200, 83_711), (200, 83_712),
                                          (200, 83_713), (200, 167_425), (7, 9362), (7, 9363), (7, 300_001), (1, 70_001)])
def test_rows_and_columns_at_the_edges_of_pieces_and_chunks(n_float, docs):
    rng = np.random.default_rng(n_float + docs)
    m, oracle = _model(rng, n_float)
    x = rng.standard_normal((docs, n_float), dtype=np.float32)
    expected = oracle.calc(x, threads=8)
    np.testing.assert_array_equal(m.calc_flat(x), expected)
    np.testing.assert_array_equal(m.calc_flat_transposed(np.ascontiguousarray(x.T)), expected)
    np.testing.assert_array_equal(m.calc_flat(x), expected)  # buffers of an earlier call


def test_columns_wider_than_a_piece():
    rng = np.random.default_rng(5)
    m, oracle = _model(rng, 3)
    x = rng.standard_normal((1_200_000, 3), dtype=np.float32)  # a column is more than a unit; two chunks
    np.testing.assert_array_equal(m.calc_flat_transposed(np.ascontiguousarray(x.T)), oracle.calc(x, threads=8))


def test_callers_side_by_side():
    rng = np.random.default_rng(6)
    m, oracle = _model(rng, 100, one_hot=True)
    xs = [rng.standard_normal((n, 101), dtype=np.float32) for n in (200_000, 30_000, 170_001, 90_000, 20_000, 165_000)]
    for x in xs:
        x[:, 100] = rng.integers(0, 5, size=len(x)).astype(np.int32).view(np.float32)
    expected = [oracle.calc(x, threads=8) for x in xs]
    got = [[None] * 2 for _ in xs]

    def work(i):
        for r in range(2):
            got[i][r] = m.calc_flat(xs[i])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(len(xs)):
        for r in range(2):
            np.testing.assert_array_equal(got[i][r], expected[i])
