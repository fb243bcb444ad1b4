"""Register kernels of three dimensions (a pair and an odd one that stands alone in the leaf tables) and of few buckets, at the
edges of their shapes, against the oracle. Needs an MI355X."""
import numpy as np
import pytest

import catboost_amd as cb
from oracle import model_builder as mb
from oracle.oracle import OracleModel

pytestmark = pytest.mark.gpu


def _model(rng, n_float, dim, depth, trees, borders, one_hot):
    """Every feature in use, so that the model has n_float buckets (and one more with one-hot splits)."""
    ffs = [mb.float_feature(i, i) for i in range(n_float)]
    cats = [mb.cat_feature(0, n_float)] if one_hot else []
    out, feature = [], 0
    for t in range(max(trees, (n_float + depth - 1) // depth)):
        splits = []
        for _ in range(depth if t % 3 else 1 + t % depth):
            splits.append(("float", feature % n_float, float(np.float32((feature * 7 % borders) / borders * 3 - 1.5))))
            feature += 1
        if one_hot and t % 4 == 0:
            splits[-1] = ("onehot", 0, 1 + t % 3)
        out.append((splits, rng.normal(size=(1 << len(splits)) * dim)))
    for f in range(n_float):  # what one-hot splits took the place of
        out.append(([("float", f, 0.25)], rng.normal(size=2 * dim)))
    return mb.build_oblivious(ffs, cats, dim, out, scale=1.5, bias=list(rng.normal(size=dim)))


def _case(n_float, dim, depth, borders, one_hot, docs):
    rng = np.random.default_rng(n_float * 100 + dim)
    model = _model(rng, n_float, dim, depth, 45, borders, one_hot)
    x = rng.normal(size=(docs, n_float + one_hot)).astype(np.float32)
    if one_hot:
        x[:, n_float] = rng.integers(0, 5, size=docs).astype(np.int32).view(np.float32)
    m = cb.ModelCalcer()
    m.load_from_dict(model)
    m.enable_gpu_evaluation(0)
    return model, m, x


@pytest.mark.parametrize("n_float,dim,depth,borders,one_hot,kernels", [
    (5, 3, 6, 20, False, "b104_w4_p3"), (104, 3, 6, 20, False, "b104_w4_p3"), (105, 3, 6, 20, False, "b176_w4_p3"),
    (176, 3, 6, 20, False, "b176_w4_p3"), (177, 3, 6, 20, False, "b192_w4_p2"), (30, 3, 4, 100, False, "b104_w4_p3"),
    (40, 3, 6, 20, True, "b104_w4_p3"), (50, 7, 6, 20, False, "b160_w4_p4 b104_w4_p3"), (104, 9, 5, 20, False, "b128_w4_p6 b104_w4_p3"),
    (56, 9, 6, 20, False, "b56_w4_p6 b104_w4_p3"), (105, 9, 6, 20, False, "b128_w4_p6 b176_w4_p3"), (80, 2, 6, 20, False, "b80_w4_p2"),
    (81, 2, 6, 20, False, "b192_w4_p2"), (56, 6, 6, 20, False, "b56_w4_p6"), (57, 5, 6, 20, False, "b128_w4_p6"),
    (79, 2, 3, 100, True, "b80_w4_p2"),
])
def test_shapes_of_few_buckets_and_of_three_dimensions(n_float, dim, depth, borders, one_hot, kernels):
    docs = 1300
    model, m, x = _case(n_float, dim, depth, borders, one_hot, docs)
    evaluate = m.evaluator().describe_kernels(cb.LAYOUT_FLAT_ROWS, 1 << 20)["evaluate"]
    assert all("cbamd_eval_reg_%s_l64" % k in evaluate for k in kernels.split()), evaluate
    oracle = OracleModel(model)
    np.testing.assert_array_equal(m.calc_flat(x), oracle.calc(x))
    n = len(model["tree_sizes"])
    for begin, end in ((0, n - 3), (5, n), (17, 34)):  # launches that hand on and take over raw sums
        np.testing.assert_array_equal(m.calc_flat(x, tree_start=begin, tree_end=end), oracle.calc(x, tree_start=begin, tree_end=end))


@pytest.mark.small_batch
@pytest.mark.parametrize("n_float,dim,docs", [(60, 3, 17_000), (104, 9, 16_900), (70, 2, 33_000), (56, 6, 20_001), (120, 3, 40_000)])
def test_sliced_batches_of_these_shapes(n_float, dim, docs):
    model, m, x = _case(n_float, dim, 6, 20, False, docs)
    assert "slices" in m.evaluator().describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)["evaluate"]
    pick = np.r_[0:300, docs // 2:docs // 2 + 300, docs - 300:docs]
    got = np.reshape(m.calc_flat(x), (docs, dim))[pick]
    np.testing.assert_allclose(got, np.reshape(OracleModel(model).calc(x[pick]), got.shape), rtol=1e-9, atol=1e-12)
