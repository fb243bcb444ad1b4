"""The exchange kernels (wide one-dimensional models, most batches of more than 32768 documents) add a document's trees as the
pair-tile kernel does, from bins or (the fused form) from flat rows: the same bits from all, and the oracle's values within the
usual tolerance."""
import numpy as np
import pytest

import catboost_amd as cb
from oracle import model_builder as mb
from oracle.oracle import OracleModel

from .test_gpu_small_batch import _model_of_buckets

pytestmark = pytest.mark.gpu


def _evaluators(model, monkeypatch):
    out = []
    for fused, exchange in (("1", "1"), ("0", "1"), ("1", "0")):
        monkeypatch.setenv("CATBOOST_AMD_FUSED", fused)
        monkeypatch.setenv("CATBOOST_AMD_EXCHANGE", exchange)
        g = cb.ModelCalcer()
        g.load_from_dict(model)
        g.enable_gpu_evaluation(0)
        out.append(g)
    return out


# buckets: the most that the registers hold, ragged; trees: none, one and many of the sixteen waves' rounds of four, odd ones;
# first: a bucket of more than 63 values takes the model out of the six-bit form
@pytest.mark.parametrize("buckets,cats,trees,depth,first,kernel", [
    (1024, 0, 300, 8, 1, "cbamd_eval_exchange_d8_s"),
    (700, 10, 201, 8, 1, "cbamd_eval_exchange_d8_s"),
    (990, 7, 1285, 7, 100, "cbamd_eval_exchange_d8"),
    (640, 0, 129, 8, 120, "cbamd_eval_exchange_d8"),
    (1000, 0, 250, 6, 1, "cbamd_eval_exchange_d6_s"),
    (650, 16, 333, 5, 100, "cbamd_eval_exchange_d6"),
    (600, 9, 150, 8, 100, "cbamd_eval_exchange_d8"),     # the 256-document tile fits LDS, but not with the row-tile kernel's regions
])
def test_exchange_kernel_gives_the_pair_tile_kernels_bits(buckets, cats, trees, depth, first, kernel, monkeypatch):
    import torch

    rng = np.random.default_rng(buckets + trees)
    model, hashes = _model_of_buckets(rng, buckets, cats, trees, depth, 1, first)
    fused, exchange, pair = _evaluators(model, monkeypatch)
    docs = 98_561                               # a workgroup per CU, and a generation of half as many behind them
    x = rng.normal(size=(docs, buckets)).astype(np.float32)
    borders = np.float32([f["borders"][len(f["borders"]) // 2] if len(f["borders"]) else 0 for f in model["float_features"]])
    for value in (np.nan, np.inf, -np.inf, borders, np.nextafter(borders, np.float32(9))):
        x[:, :buckets - cats] = np.where(rng.random((docs, 1)) < 0.1, value, x[:, :buckets - cats])
    for i in range(cats):
        x[:, buckets - cats + i] = rng.choice(hashes[i], size=docs).view(np.float32)
    flat = torch.from_numpy(x).to("cuda:0")
    results = {}
    for name, g in (("fused", fused), ("exchange", exchange), ("pair", pair)):
        ev = g.evaluator()
        feats = ev.features(cb.LAYOUT_FLAT_ROWS, flat.data_ptr(), flat.shape[1])
        for n in (32768, 32769, 46_081, docs):
            kernels = ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, n)
            if name == "fused" and n > 46_080:          # seven tenths of the CUs have a workgroup
                assert kernels == {"fused": kernel.replace("eval", "fused")}
            else:
                assert kernels["evaluate"] == (kernel if name != "pair" and n > 32768 else "EvalObliviousPairTileKernel")
            out = torch.full((n + 1,), -3.0, dtype=torch.float64, device="cuda:0")
            torch.cuda.synchronize()
            ev.eval_data(feats, n, out.data_ptr())
            assert out[n].item() == -3.0
            results[name, n] = out[:n].clone()
    for n in (32768, 32769, 46_081, docs):
        assert torch.equal(results["exchange", n], results["pair", n]), n
        assert torch.equal(results["fused", n], results["pair", n]), n
    # rows further apart than the model's features, and the last document's row at the end of its memory
    wide = torch.full((docs * (buckets + 5) - 5,), float("nan"), device="cuda:0")
    torch.as_strided(wide, (docs, buckets), (buckets + 5, 1)).copy_(flat)
    out = torch.zeros(docs, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev = fused.evaluator()
    ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, wide.data_ptr(), buckets + 5), docs, out.data_ptr())
    assert torch.equal(out, results["pair", docs])
    sample = rng.choice(docs, size=300, replace=False)
    np.testing.assert_allclose(results["exchange", docs].cpu().numpy()[sample], OracleModel(model).calc(x[sample]), rtol=1e-9, atol=1e-12)
    # a range of the trees takes the pair-tile kernel, the whole model the exchange kernel
    ranged = exchange.calc_flat(x[:33_000], tree_start=1, tree_end=trees)
    np.testing.assert_allclose(ranged[sample[sample < 33_000]],
                               OracleModel(model).calc(x[sample[sample < 33_000]], tree_start=1, tree_end=trees), rtol=1e-9, atol=1e-12)


@pytest.mark.parametrize("share,depth,exchange", [(0.0, 8, True), (0.1, 8, True), (0.35, 8, False), (0.05, 6, True), (0.3, 6, False)])
def test_models_that_look_at_one_bucket_most_keep_the_pair_tile_kernel(share, depth, exchange, monkeypatch):
    """One wave compares all levels of a bucket, so the exchange kernels are slower than the pair-tile kernel when a bucket has too many of
    them. The values are the same bits whatever kernel takes the batch."""
    import torch

    rng = np.random.default_rng(17)
    buckets, trees, docs = 700, 600, 130_000
    at = list(rng.permutation(buckets))
    tree_list = []
    for _ in range(trees):
        columns = [0 if rng.random() < share else int(at.pop() if at else rng.integers(0, buckets)) for _ in range(depth)]
        tree_list.append(([("float", c, float(np.float32(rng.integers(-30, 31) / 20))) for c in columns], rng.normal(size=1 << depth)))
    model = mb.build_oblivious([mb.float_feature(f) for f in range(buckets)], [], 1, tree_list)
    x = rng.normal(size=(docs, buckets)).astype(np.float32)
    flat = torch.from_numpy(x).to("cuda:0")
    results = []
    for g in _evaluators(model, monkeypatch):
        ev = g.evaluator()
        kernels = ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)
        if len(results) < 2 and exchange:
            assert "exchange" in kernels.get("fused", kernels.get("evaluate"))
            assert ("fused" in kernels) == (len(results) == 0)
        else:
            assert kernels["evaluate"] == "EvalObliviousPairTileKernel"
        out = torch.zeros(docs, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, flat.data_ptr(), buckets), docs, out.data_ptr())
        results.append(out)
    assert torch.equal(results[0], results[2]) and torch.equal(results[1], results[2])
    sample = rng.choice(docs, size=200, replace=False)
    np.testing.assert_allclose(results[0].cpu().numpy()[sample], OracleModel(model).calc(x[sample]), rtol=1e-9, atol=1e-12)


@pytest.mark.parametrize("buckets,trees,depth,first,share,kernel", [
    (575, 499, 8, 200, 0.0, "EvalObliviousTileKernel"),       # a bucket of two rows: no exchange kernel
    (575, 500, 8, 200, 0.0, "EvalObliviousPairTileKernel"),
    (620, 149, 6, 200, 0.0, "EvalObliviousTileKernel"),
    (620, 499, 7, 1, 0.0, "cbamd_eval_exchange_d8_s"),
    (620, 300, 8, 1, 0.45, "EvalObliviousTileKernel"),        # too many levels on one bucket for the exchange kernels
    (620, 500, 8, 1, 0.45, "EvalObliviousPairTileKernel"),
    (700, 300, 8, 1, 0.45, "EvalObliviousPairTileKernel"),    # more buckets than the tile holds
])
def test_models_of_few_trees_keep_the_tile_kernel(buckets, trees, depth, first, share, kernel, monkeypatch):
    """Models whose tile of 256 documents fits LDS without the row-tile kernel's regions. Whatever kernel takes the model, the same bits
    at every batch size; ranges of few and of many trees."""
    import torch

    monkeypatch.setenv("CATBOOST_AMD_FUSED", "0")
    rng = np.random.default_rng(trees)
    model, _ = _model_of_buckets(rng, buckets, 0, trees, depth, 1, first)
    if share:
        at = list(rng.permutation(buckets))
        model = mb.build_oblivious([mb.float_feature(f) for f in range(buckets)], [], 1, [
            ([("float", 0 if rng.random() < share else int(at.pop() if at else rng.integers(0, buckets)),
               float(np.float32(rng.integers(-20, 21) / 20))) for _ in range(depth)], rng.normal(size=1 << depth)) for _ in range(trees)])
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    ev = g.evaluator()
    docs = 66_000
    assert ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)["evaluate"] == kernel
    x = rng.normal(size=(docs, buckets)).astype(np.float32)
    flat = torch.from_numpy(x).to("cuda:0")
    feats = ev.features(cb.LAYOUT_FLAT_ROWS, flat.data_ptr(), buckets)
    sample = rng.choice(3000, size=200, replace=False)
    oracle = OracleModel(model)
    whole = torch.zeros(docs, dtype=torch.float64, device="cuda:0")
    out = torch.zeros(docs, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev.eval_data(feats, docs, whole.data_ptr())
    np.testing.assert_allclose(whole.cpu().numpy()[sample], oracle.calc(x[sample]), rtol=1e-9, atol=1e-12)
    for n in (100, 3000, 20_000, 40_000):
        ev.eval_data(feats, n, out.data_ptr())
        assert torch.equal(out[:n], whole[:n]), n
    for tree_range in ((0, trees - 1), (1, trees), (5, 6), (7, 7), (0, trees // 3), (trees // 2, trees)):
        for n in (3000, docs):
            ev.eval_data(feats, n, out.data_ptr(), tree_start=tree_range[0], tree_end=tree_range[1])
            np.testing.assert_allclose(out.cpu().numpy()[sample], oracle.calc(x[sample], tree_start=tree_range[0], tree_end=tree_range[1]),
                                       rtol=1e-9, atol=1e-12)


def test_no_alloc_entry_point_takes_batches_beyond_its_buffer(monkeypatch):
    """eval_data_no_alloc: a wide model of a fused kernel uses no bin buffer, so it is refused at no size, also where eval_data takes
    two launches (few workgroups in the last generation, or no batch at all is faster fused); eager and replayed from a graph."""
    import torch

    model, _ = _model_of_buckets(np.random.default_rng(4), 700, 3, 320, 8, 1, 1)
    fused, _, pair = _evaluators(model, monkeypatch)
    ev = fused.evaluator()
    limit = (32 << 20) // ev.quantized_bytes(256) * 256
    docs = 70_001
    assert limit < 50_000 and "fused" not in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)
    x = torch.from_numpy(np.random.default_rng(5).normal(size=(docs, 700)).astype(np.float32)).to("cuda:0")
    feats = ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), 700)
    expected = torch.zeros(docs, dtype=torch.float64, device="cuda:0")
    out = torch.zeros(docs, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    pair.evaluator().eval_data(feats, docs, expected.data_ptr())
    for n in (limit, limit + 1, docs):
        out.fill_(-1.0)
        torch.cuda.synchronize()
        ev.eval_data_no_alloc(feats, n, out.data_ptr())
        ev.synchronize()
        assert torch.equal(out[:n], expected[:n]) and bool((out[n:] == -1.0).all()), n
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ev.eval_data_no_alloc(feats, docs, out.data_ptr(), stream=torch.cuda.current_stream().cuda_stream)
    for replay in range(3):
        x.copy_(x.flip(0))
        out.fill_(-1.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        pair.evaluator().eval_data(feats, docs, expected.data_ptr())
        assert torch.equal(out, expected), replay
    with pytest.raises(cb.CatBoostError, match="exceeds the fixed bin buffer"):
        ev.eval_data_no_alloc(feats, docs, out.data_ptr(), tree_start=1)      # a range of the trees has no fused kernel


def test_batches_of_more_documents_than_a_launch_can_count():
    """2^29 documents and more: the exchange kernels are not chosen (their launch counts work-items in 32 bits); prediction types whose kernel
    has 64 documents a workgroup refuse what that grid cannot hold."""
    import torch

    model, _ = _model_of_buckets(np.random.default_rng(2), 700, 3, 201, 8, 1, 1)
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    ev = g.evaluator()
    for layout in (cb.LAYOUT_FLAT_ROWS, cb.LAYOUT_FLAT_COLUMNS):
        assert "exchange" in str(ev.describe_kernels(layout, (1 << 29) - 1))
        assert "exchange" not in str(ev.describe_kernels(layout, 1 << 29))
    dims = cb.ModelCalcer()
    dims.build_oblivious([dict(index=0, flat_index=0)], [], 9, [([("float", 0, 0.5)], [0.25] * 18)])
    dims.enable_gpu_evaluation(0)
    raw, result = torch.zeros(9, dtype=torch.float64, device="cuda:0"), torch.zeros(9, dtype=torch.float64, device="cuda:0")
    for kind in (cb.APT_PROBABILITY, cb.APT_CLASS, cb.APT_MULTI_PROBABILITY):
        with pytest.raises(cb.CatBoostError, match="too many documents"):
            dims.evaluator().apply_prediction_type(kind, (1 << 37) + 64, raw.data_ptr(), result.data_ptr())


def test_empty_batches():
    """No documents: every call returns without touching a buffer, null pointers among them."""
    import torch

    model, _ = _model_of_buckets(np.random.default_rng(2), 700, 3, 201, 8, 1, 1)
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    ev = g.evaluator()
    assert "fused" in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, 60_000)
    assert "fused" not in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, 0)
    assert g.calc_flat(np.zeros((0, 700), np.float32)).size == 0
    assert g.calc_flat_transposed(np.zeros((700, 0), np.float32)).size == 0
    assert g.quantize_flat(np.zeros((0, 700), np.float32)).size == 0
    assert g.calc_leaf_indexes_flat(np.zeros((0, 700), np.float32)).size == 0
    guard = torch.full((16,), 7.0, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    for pointer in (guard.data_ptr(), 0):
        for layout in (cb.LAYOUT_FLAT_ROWS, cb.LAYOUT_FLAT_COLUMNS):
            feats = ev.features(layout, pointer, 700)
            ev.eval_data(feats, 0, pointer)
            ev.eval_data_no_alloc(feats, 0, pointer)
            ev.quantize(feats, 0, pointer)
        ev.eval_quantized(pointer, 0, pointer)
    ev.synchronize()
    assert bool((guard == 7.0).all())
