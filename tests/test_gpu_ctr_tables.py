"""CTR features of one projection share a hash table of bins: entries of one and of several 16-byte pieces, features of
more than 254 borders (several buckets), tables of one projection that know different hashes, batches whose workgroups
share the projections out. Needs an MI355X."""
import numpy as np
import pytest

import catboost_amd as cb
from oracle.oracle import OracleModel
from oracle.cbm_reader import read_cbm

from tests import ctr_models
from tests.cbm_writer import write_cbm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", ["1", "0"])
@pytest.mark.parametrize("copies,wide", [(1, False), (4, False), (13, False), (5, True)])
def test_projections_of_many_buckets(monkeypatch, tile, copies, wide):
    monkeypatch.setenv("CATBOOST_AMD_CTR_TILE", tile)
    model, known = ctr_models.random_ctr_model(21, n_cat=6, n_bases=15, n_trees=30)
    rng = np.random.default_rng(copies)
    features = []
    for c in model["ctr_features"]:
        for k in range(copies):
            lo, hi = float(c["shift"] * c["scale"]), float((1 + c["shift"]) * c["scale"])
            count = 300 if wide and k == 2 else int(rng.integers(1, 20))
            features.append(dict(c, prior_num=np.float32(k / 8.0),
                                 borders=np.unique(rng.uniform(lo, hi, size=count).astype(np.float32))))
    model["ctr_features"], model["ctr_feature_count"] = features, len(features)
    total = (sum(f["borders"].size for f in model["float_features"]) +
             sum(o["values"].size for o in model["one_hot_features"]) + sum(c["borders"].size for c in features))
    model["tree_splits"] = rng.integers(0, total, size=len(model["tree_splits"])).astype(np.int32)
    data = write_cbm(model)
    o, g = OracleModel(read_cbm(data)), cb.ModelCalcer(buffer=data)
    for docs in (1, 257, 5000):
        floats, cats = ctr_models.random_documents(model, known, docs, 3 + docs)
        np.testing.assert_array_equal(g.quantize_hashed(floats, cats), o.binarize(floats, cats, layout="split"))


def test_large_tables_are_built_side_by_side():
    """Tables of 20 000 further hashes each, so that the projections' tables are made by several host threads."""
    model, known = ctr_models.random_ctr_model(22, n_cat=6, n_bases=15, n_trees=30)
    rng = np.random.default_rng(22)
    for table in model["ctr_tables"]:
        index = table["index_hash_raw"].view(np.dtype([("hash", "<u8"), ("row", "<u4")]))
        index = np.sort(index[index["hash"] != np.uint64(ctr_models.MASK64)], order="row")
        rows = table["ctr_blob"].reshape(len(index), -1)
        assert (index["row"] == np.arange(len(index))).all()
        more = rng.integers(0, 2**63, size=20_000, dtype=np.uint64)
        table["index_hash_raw"] = ctr_models.build_index_hash([int(h) for h in np.unique(np.concatenate([index["hash"], more]))])
        order = np.argsort(np.argsort(np.concatenate([index["hash"], more])))
        blob = np.concatenate([rows, rows[rng.integers(0, len(rows), size=len(more))]])
        placed = np.empty_like(blob)
        placed[order] = blob
        table["ctr_blob"] = placed.ravel().copy()
    data = write_cbm(model)
    o, g = OracleModel(read_cbm(data)), cb.ModelCalcer(buffer=data)
    floats, cats = ctr_models.random_documents(model, known, 3000, 5)
    bins = g.quantize_hashed(floats, cats)
    np.testing.assert_array_equal(bins, o.binarize(floats, cats, layout="split"))
    np.testing.assert_allclose(g.calc_hashed(floats, cats), o.calc(floats, cats, layout="split"), rtol=1e-9, atol=1e-12)


def _model_of_large_tables(more_hashes):
    model, known = ctr_models.random_ctr_model(23, n_cat=6, n_bases=15, n_trees=30)
    for table in model["ctr_tables"]:
        rng = np.random.default_rng(23)  # the same hashes in every table of a projection
        index = table["index_hash_raw"].view(np.dtype([("hash", "<u8"), ("row", "<u4")]))
        index = np.sort(index[index["hash"] != np.uint64(ctr_models.MASK64)], order="row")
        rows = table["ctr_blob"].reshape(len(index), -1)
        keys = np.unique(np.concatenate([index["hash"], rng.integers(0, 2**63, size=more_hashes, dtype=np.uint64)]))
        row_of = {int(h): int(r) for h, r in index}
        table["index_hash_raw"] = ctr_models.build_index_hash([int(h) for h in keys])
        table["ctr_blob"] = rows[[row_of.get(int(h), i % len(rows)) for i, h in enumerate(keys)]].ravel().copy()
    return model, known


@pytest.mark.parametrize("more_hashes,roomy", [(3000, True), (60_000, False)])
def test_tables_are_roomy_only_while_they_are_small_together(more_hashes, roomy):
    """Tables a quarter full cost lookups more than they give once all of them together outgrow the L2s."""
    import torch

    model, known = _model_of_large_tables(more_hashes)
    data = write_cbm(model)
    projections = {(tuple(c["base"]["cat_features"]), tuple(c["base"]["float_splits"]), tuple(c["base"]["one_hot_splits"]))
                   for c in model["ctr_features"]}
    entries = 2
    while entries < 2 * more_hashes:
        entries *= 2
    half = len(projections) * entries * 16  # (entries of one piece, and of two where a projection has many features)
    assert (2 * half <= 10 << 20) == roomy and (half > 12 << 20) != roomy
    warm = cb.ModelCalcer(buffer=write_cbm(_model_of_large_tables(10)[0]))
    warm.enable_gpu_evaluation(0)
    warm.evaluator()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    g = cb.ModelCalcer(buffer=data)
    g.enable_gpu_evaluation(0)
    g.evaluator()
    used = before - torch.cuda.mem_get_info()[0]
    if not roomy:
        assert half <= used < 1.9 * half, (used, half)
    o = OracleModel(read_cbm(data))
    floats, cats = ctr_models.random_documents(model, known, 3000, 5)
    np.testing.assert_array_equal(g.quantize_hashed(floats, cats), o.binarize(floats, cats, layout="split"))
