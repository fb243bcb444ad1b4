"""Features with exactly as many borders as the byte-parallel compares of the register and fused kernels hold: 128 in the 7-bit
form (a bin of 128 has bit 7 set by itself) and 64 in the six-bit form, next to one border less and one more. Needs an MI355X."""
import numpy as np
import pytest

import catboost_amd as cb
from oracle import model_builder as mb
from oracle.oracle import OracleModel

pytestmark = pytest.mark.gpu


def _model(rng, borders, n_float, depth, dim, one_hot):
    """Every border of every feature in use; trees of every depth up to `depth`, so that the walk has levels that stand for
    none, whose register (the tree's first) holds the largest bin for many documents."""
    ffs = [mb.float_feature(i, i) for i in range(n_float)]
    cats = [mb.cat_feature(0, n_float)] if one_hot else []
    cands = [np.unique(rng.normal(size=8 * borders).astype(np.float32))[:borders] for _ in range(n_float)]
    assert all(len(c) == borders for c in cands)
    trees = []
    for f in range(n_float):
        order, at = rng.permutation(borders), 0
        while at < borders:
            levels = order[at:at + 1 + len(trees) % depth]
            at += len(levels)
            splits = [("float", f, float(cands[f][i])) for i in levels]
            if one_hot and len(trees) % 5 == 0 and len(splits) < depth:
                splits.append(("onehot", 0, int(rng.integers(1, 4))))
            trees.append((splits, rng.normal(size=(1 << len(splits)) * dim)))
    trees.append(([], rng.normal(size=dim)))
    model = mb.build_oblivious(ffs, cats, dim, trees, scale=0.5, bias=list(rng.normal(size=dim)))
    return model, cands


@pytest.mark.parametrize("fused", ["1", "0"])
@pytest.mark.parametrize("borders,n_float,depth,dim,one_hot", [
    (63, 20, 6, 1, False), (64, 20, 6, 1, False), (65, 20, 6, 1, False), (64, 70, 8, 1, False), (64, 16, 6, 3, False),
    (127, 20, 6, 1, False), (128, 20, 6, 1, False), (129, 20, 6, 1, False), (128, 70, 8, 1, False), (128, 16, 8, 4, False),
    (128, 10, 10, 1, False), (64, 10, 10, 1, False), (128, 12, 6, 1, True), (64, 100, 6, 1, False), (128, 100, 8, 1, False),
])
def test_buckets_of_as_many_values_as_a_form_holds(monkeypatch, borders, n_float, depth, dim, one_hot, fused):
    monkeypatch.setenv("CATBOOST_AMD_FUSED", fused)
    rng = np.random.default_rng(borders * 1000 + n_float + depth)
    model, cands = _model(rng, borders, n_float, depth, dim, one_hot)
    docs = 1500
    x = rng.normal(size=(docs, n_float + one_hot)).astype(np.float32)
    for f in range(n_float):
        x[:500, f] = rng.choice(cands[f], size=500)   # on the borders
        x[500:800, f] = cands[f][-1] + np.float32(1)  # the largest bin
        x[800:900, f] = rng.choice(cands[f][-3:], size=100) + np.float32(1e-4)
    x[900:950, :n_float] = np.inf
    x[950:1000, :n_float] = -np.inf
    x[1000:1050, :n_float] = np.nan
    if one_hot:
        x[:, n_float] = rng.integers(0, 5, size=docs).astype(np.int32).view(np.float32)
    oracle = OracleModel(model)
    m = cb.ModelCalcer()
    m.load_from_dict(model)
    m.enable_gpu_evaluation(0)
    kernels = m.evaluator().describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)
    assert ("fused" in kernels) == (fused == "1" and dim == 1 and depth <= 8 and n_float >= 16 and not one_hot and borders <= 128), kernels
    name = kernels.get("fused") or kernels["evaluate"].split(" ")[0]
    assert name.startswith("cbamd_")
    if not one_hot:
        assert name.endswith("_s") == (borders <= 64) and "_m" not in name, name
    np.testing.assert_array_equal(m.quantize_flat(x), oracle.binarize(x))
    np.testing.assert_array_equal(m.calc_flat(x), oracle.calc(x))
    n = len(model["tree_sizes"])
    np.testing.assert_array_equal(m.calc_flat(x, tree_start=3, tree_end=n - 2), oracle.calc(x, tree_start=3, tree_end=n - 2))
