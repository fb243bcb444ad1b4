"""Small batches on the register-resident kernels: slices of the trees on workgroups of their own. Needs an MI355X.

The reference special-cases single documents (c_api.cpp:383-384, cpu/evaluator_impl.cpp:417-460); here a
batch too small to fill the chip is spread by cutting the trees into slices whose raw sums a second kernel
adds in slice order. Bar: 1e-9 relative / 1e-12 absolute against the oracle, the same bits on every call,
and the bit-exact single pass again from the size on where slicing stops.
"""
import numpy as np
import pytest

import catboost_amd as cb
from catboost_amd import synthetic as syn
from oracle import model_builder as mb
from oracle.cbm_reader import read_cbm
from oracle.oracle import OracleModel

pytestmark = [pytest.mark.gpu, pytest.mark.small_batch]


@pytest.mark.parametrize("cfg,trees", [("C2", 1000), ("C1", 200), ("C3", 300), ("C2", 37)])
def test_small_batches_through_tree_slices(cfg, trees):
    import torch

    model, info = syn.build_model(cfg, trees=trees)
    model.set_scale_and_bias(0.25, [0.5 + k for k in range(info["dim"])])
    model.enable_gpu_evaluation(0)
    ev = model.evaluator()
    oracle = OracleModel(read_cbm(model.save_to_buffer()))
    dim = info["dim"]
    x = syn.device_features(info, 530_000)  # more than 256 workgroups of eight 256-document blocks
    host = x.cpu().numpy()
    for docs in (1, 256, 4096, 65_536):
        part = x[:docs].contiguous()
        feats = ev.features(cb.LAYOUT_FLAT_ROWS, part.data_ptr(), part.shape[1])
        a = torch.full((docs * dim,), -1.0, dtype=torch.float64, device="cuda:0")
        b = torch.full((docs * dim,), -2.0, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        ev.eval_data(feats, docs, a.data_ptr())
        ev.eval_data(feats, docs, b.data_ptr())
        torch.cuda.synchronize()
        assert torch.equal(a, b), "two calls differ"
        expected = oracle.calc(host[:docs], threads=8)
        np.testing.assert_allclose(a.cpu().numpy(), expected, rtol=1e-9, atol=1e-12)
        # the host entry point takes the same path
        np.testing.assert_array_equal(model.calc_flat(host[:min(docs, 5000)]), a.cpu().numpy()[:min(docs, 5000) * dim])
    # a batch that fills the chip goes the single pass again: the CPU evaluator's bits (one-dimensional models)
    docs = host.shape[0]
    out = torch.zeros(docs * dim, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), x.shape[1]), docs, out.data_ptr())
    torch.cuda.synchronize()
    expected = oracle.calc(host, threads=8)
    if dim == 1:
        np.testing.assert_array_equal(out.cpu().numpy(), expected)
    else:
        np.testing.assert_allclose(out.cpu().numpy(), expected, rtol=1e-9, atol=1e-12)


def test_small_batch_slicing_switched_off_through_the_api():
    """CbHipSetSmallBatchSlicing / CbHipEvaluatorSetSmallBatchSlicing: with the slices off a small batch is summed in
    one pass in tree order, the CPU evaluator's bits, through the model handle's host calls and the evaluator's
    device calls; switched on again the slices are back."""
    import torch

    model, info = syn.build_model("C2", trees=200)
    model.enable_gpu_evaluation(0)
    oracle = OracleModel(read_cbm(model.save_to_buffer()))
    x = syn.device_features(info, 3000)
    host = x.cpu().numpy()
    expected = oracle.calc(host, threads=8)
    ev = model.evaluator()
    assert "slices" in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, 3000)["evaluate"]
    sliced = model.calc_flat(host)
    np.testing.assert_allclose(sliced, expected, rtol=1e-9, atol=1e-12)
    model.set_small_batch_slicing(False)
    assert "slices" not in str(ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, 3000))   # (this model: the fused kernel at any size)
    np.testing.assert_array_equal(model.calc_flat(host), expected)
    out = torch.zeros(3000, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), x.shape[1]), 3000, out.data_ptr())
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), expected)
    # the setting survives a new evaluator of the handle (a feature layout rebuilds it)
    model.set_feature_layout(None, None, None)
    np.testing.assert_array_equal(model.calc_flat(host), expected)
    ev = model.evaluator()
    ev.set_small_batch_slicing(True)
    assert "slices" in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, 3000)["evaluate"]
    np.testing.assert_array_equal(model.calc_flat(host), sliced)


@pytest.mark.parametrize("seed,n_float,n_cat,trees,depth,dim,many,docs", [
    (1, 7, 2, 1, 6, 1, False, (1, 2)),
    (2, 20, 0, 31, 4, 1, False, (1, 15, 16, 17)),
    (3, 9, 6, 63, 8, 1, True, (5, 640, 641)),        # a slice of two turns and a ragged one; one-hot; more than 254 borders
    (4, 130, 3, 64, 7, 1, False, (33, 1000)),        # two slices; cells of three turns of the tile
    (5, 300, 4, 97, 6, 2, False, (3, 320, 321)),     # two dimensions: documents count twice
    (6, 40, 2, 1100, 5, 3, False, (17, 700)),        # more slices than rows of a workgroup
    (7, 12, 1, 33, 8, 9, False, (16, 400)),          # three passes over the dimensions, the last of one
    (8, 700, 10, 200, 8, 1, False, (1, 64, 1500)),   # wider than the register kernels
])
def test_small_kernels_against_the_oracle(seed, n_float, n_cat, trees, depth, dim, many, docs):
    """One launch from the features to the results: a lane per tree for few documents, sixteen lanes of documents per
    slice of the trees beyond. Every layout, device and host entry points, NaN modes, one-hot splits."""
    import torch

    from tests.test_oracle import _random_flat_data, _random_oblivious

    rng = np.random.default_rng(seed)
    model, cat_values = _random_oblivious(rng, n_float=n_float, n_cat=n_cat, trees=trees, max_depth=depth, dim=dim,
                                          many_borders=many, scale=0.5, bias=rng.normal(size=dim))
    o = OracleModel(model)
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    ev = g.evaluator()
    float_at = [f["flat_index"] for f in model["float_features"]]
    cat_at = [c["flat_index"] for c in model["cat_features"]]
    for n in docs:
        kernel = ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, n)["evaluate"]
        passes = 1 if dim <= 2 else (dim + 3) // 4
        assert kernel.startswith("FewDocumentsKernel" if n * passes <= 640 else "SmallBatchKernel"), kernel
        x = _random_flat_data(rng, model, cat_values, n)
        expected = o.calc(x)
        close = dict(rtol=1e-9, atol=1e-12)
        np.testing.assert_allclose(g.calc_flat(x), expected, **close)
        np.testing.assert_allclose(g.calc_flat_transposed(np.ascontiguousarray(x.T)), expected, **close)
        floats, cats = np.ascontiguousarray(x[:, float_at]), np.ascontiguousarray(x[:, cat_at]).view(np.int32)
        if n_cat:
            np.testing.assert_allclose(g.calc_hashed(floats, cats), expected, **close)
        flat, columns = torch.from_numpy(x).to("cuda:0"), torch.from_numpy(np.ascontiguousarray(x.T)).to("cuda:0")
        f, c = torch.from_numpy(floats).to("cuda:0"), torch.from_numpy(cats).to("cuda:0")
        for feats in (ev.features(cb.LAYOUT_FLAT_ROWS, flat.data_ptr(), flat.shape[1]),
                      ev.features(cb.LAYOUT_FLAT_COLUMNS, columns.data_ptr(), n),
                      ev.features(cb.LAYOUT_SPLIT_ROWS, f.data_ptr(), f.shape[1], c.data_ptr(), c.shape[1])):
            out = torch.full((n * dim + 8,), -3.0, dtype=torch.float64, device="cuda:0")
            torch.cuda.synchronize()
            ev.eval_data(feats, n, out.data_ptr())
            np.testing.assert_allclose(out.cpu().numpy()[:n * dim], expected, **close)
            assert (out.cpu().numpy()[n * dim:] == -3.0).all()
        assert ev.last_kernel_times()[1] > 0.0


def test_kernel_times_beside_running_small_batches():
    """The last call's times are read from its launch's clock stamps while other threads' launches of growing size write
    theirs: each reading is one launch's own."""
    import threading

    model, info = syn.build_model("C1", trees=150)
    model.enable_gpu_evaluation(0)
    ev = model.evaluator()
    host = syn.device_features(info, 8000).cpu().numpy()
    expected = model.calc_flat(host)
    failures, running = [], threading.Event()
    running.set()

    def read_times():
        try:
            while running.is_set():
                assert 0.0 < ev.last_kernel_times()[1] < 1000.0
        except Exception as e:  # noqa: BLE001 (reported below)
            failures.append(repr(e))

    def call(offset):
        try:
            for docs in range(1 + offset, 8000, 601):
                assert np.array_equal(model.calc_flat(host[:docs]), expected[:docs])
        except Exception as e:  # noqa: BLE001
            failures.append(repr(e))

    reader = threading.Thread(target=read_times)
    callers = [threading.Thread(target=call, args=(i,)) for i in range(3)]
    for t in [reader] + callers:
        t.start()
    for t in callers:
        t.join()
    running.clear()
    reader.join()
    assert not failures, failures


def test_a_documents_value_does_not_depend_on_the_small_kernel_that_took_it():
    """The slices of the trees and the order of their sums are those of the register kernels' small batches."""
    import torch

    model, info = syn.build_model("C1", trees=150)
    model.enable_gpu_evaluation(0)
    ev = model.evaluator()
    x = syn.device_features(info, 20_000)
    values = {}
    for docs in (3, 640, 641, 16_384, 20_000):
        part = x[:docs].contiguous()
        out = torch.zeros(docs, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, part.data_ptr(), part.shape[1]), docs, out.data_ptr())
        values[docs] = out.cpu().numpy()
    assert "cbamd_eval_reg" in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, 20_000)["evaluate"]
    for docs, v in values.items():
        np.testing.assert_array_equal(v, values[20_000][:docs])


@pytest.mark.parametrize("seed,n_float,n_cat,trees,depth,dim,many,docs", [
    (1, 40, 0, 150, 6, 1, False, 131_073),    # five slices, the last of 22 trees; 16-tree blocks
    (2, 150, 0, 500, 8, 1, False, 60_001),    # sixteen slices, the last of 20 trees
    (3, 30, 6, 330, 8, 1, True, 100_000),     # bins in mapped registers, one-hot splits
    (4, 60, 0, 200, 7, 6, False, 70_007),     # several dimensions: small tree blocks, many to a slice
    (5, 50, 0, 161, 10, 1, False, 90_001),    # deep trees: byte selectors in scalar registers; a slice of one tree
])
def test_workgroups_that_walk_several_slices(seed, n_float, n_cat, trees, depth, dim, many, docs):
    """A batch of more (document, slice) pairs than the chip holds workgroups has workgroups walk several slices: the
    same bits as batches whose workgroups take one slice each."""
    import torch

    from tests.test_oracle import _random_flat_data, _random_oblivious

    rng = np.random.default_rng(seed)
    model, cat_values = _random_oblivious(rng, n_float=n_float, n_cat=n_cat, trees=trees, max_depth=depth, dim=dim,
                                          many_borders=many, scale=0.5, bias=rng.normal(size=dim))
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    ev = g.evaluator()
    kernels = ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)["evaluate"]
    assert "cbamd_eval_reg" in kernels and "slices" in kernels, kernels
    x = _random_flat_data(rng, model, cat_values, docs)
    flat = torch.from_numpy(x).to("cuda:0")
    out = torch.full((docs * dim + 8,), -3.0, dtype=torch.float64, device="cuda:0")
    parts = torch.zeros(docs * dim, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, flat.data_ptr(), flat.shape[1]), docs, out.data_ptr())
    for begin in range(0, docs, 2048):
        n = min(2048, docs - begin)
        ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, flat[begin:].data_ptr(), flat.shape[1]), n, parts[begin * dim:].data_ptr())
    assert torch.equal(out[:docs * dim], parts)
    assert bool((out[docs * dim:] == -3.0).all())
    sample = rng.choice(docs, size=2000, replace=False)
    np.testing.assert_allclose(out.cpu().numpy()[:docs * dim].reshape(docs, dim)[sample],
                               OracleModel(model).calc(x[sample]).reshape(-1, dim), rtol=1e-9, atol=1e-12)


def test_kernel_times_are_read_without_waiting_for_other_streams():
    """A small-batch call's times come at once while the null stream is busy, and leave a capture alone."""
    import torch

    model, info = syn.build_model("C1", trees=150)
    model.enable_gpu_evaluation(0)
    ev = model.evaluator()
    docs = 2000
    x = syn.device_features(info, docs)
    out = torch.zeros(docs, dtype=torch.float64, device="cuda:0")
    feats = ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), x.shape[1])
    torch.cuda.synchronize()
    ev.eval_data(feats, docs, out.data_ptr())
    expected = ev.last_kernel_times()
    assert expected[0] == 0.0 and 0.0 < expected[1] < 100.0
    busy = torch.cuda.Event()
    torch.cuda._sleep(500_000_000)  # some 0.2 s on the null stream
    busy.record()
    assert ev.last_kernel_times() == expected
    assert not busy.query(), "the times waited for the null stream"
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    ones = torch.ones(16, device="cuda:0")
    with torch.cuda.graph(graph):
        ones += 1.0
        assert ev.last_kernel_times() == expected
    for i in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert bool((ones == 2.0 + i).all())


def _model_of_buckets(rng, buckets, cats, trees, depth, dim, borders_of_first):
    """Every one of `buckets` columns is split on, the last `cats` of them one-hot; trees of different depths."""
    floats = buckets - cats
    hashes = rng.integers(-2**31, 2**31, size=(cats, 5), dtype=np.int64).astype(np.int32)
    columns = list(rng.permutation(buckets)) + [0] * (borders_of_first if borders_of_first > 1 else 0)
    tree_list = []
    for t in range(trees):
        size = depth if len(columns) > 0 or t % 5 else int(rng.integers(0, depth + 1))
        splits = []
        for _ in range(size):
            c = int(columns.pop() if columns else rng.integers(0, buckets))
            splits.append(("float", c, float(np.float32(rng.normal()))) if c < floats
                          else ("onehot", c - floats, int(rng.choice(hashes[c - floats]))))
        tree_list.append((splits, rng.normal(size=dim << size)))
    assert not columns
    model = mb.build_oblivious([mb.float_feature(f) for f in range(floats)], [mb.cat_feature(i, floats + i) for i in range(cats)],
                               dim, tree_list, scale=0.5, bias=rng.normal(size=dim))
    return model, hashes


@pytest.mark.parametrize("buckets,cats,trees,depth,dim,first,switch,kernel", [
    (400, 2, 301, 8, 1, 1, "", "EvalObliviousRowTileKernel"),
    (230, 0, 203, 6, 1, 1, "", "EvalObliviousRowTileKernel"),          # eight waves
    (560, 0, 117, 8, 1, 200, "", "EvalObliviousRowTileKernel"),        # a bucket of more than 127 values
    (330, 0, 150, 8, 3, 1, "", "EvalObliviousRowTileKernel"),
    (260, 3, 90, 6, 10, 1, "", "EvalObliviousRowTileKernel"),
    (300, 3, 170, 8, 1, 200, "ROW_TILE", "EvalObliviousTileKernel"),
    (500, 3, 333, 8, 1, 1, "ROW_TILE", "EvalObliviousTileKernel"),
    (300, 0, 77, 4, 5, 1, "ROW_TILE", "EvalObliviousTileKernel"),
    (700, 10, 201, 8, 1, 1, "", "EvalObliviousPairTileKernel"),        # a last tree without a partner
    (1000, 0, 250, 6, 1, 1, "", "EvalObliviousPairTileKernel"),
    (700, 10, 205, 8, 1, 1, "PAIR_TILE", "EvalObliviousHalfTileKernel"),
    (1150, 0, 303, 8, 1, 1, "", "EvalObliviousQuadTileKernel"),        # three trees behind the last four
    (1150, 5, 250, 6, 1, 1, "", "EvalObliviousQuadTileKernel"),
    (2100, 5, 420, 6, 1, 1, "", "EvalObliviousQuadTileKernel"),        # four waves
    (900, 0, 150, 7, 2, 1, "", "EvalObliviousKernel"),                 # one pass in tree order
])
def test_wide_models_round_alike_at_every_batch_size(buckets, cats, trees, depth, dim, first, switch, kernel, monkeypatch):
    """Models that the register kernels do not take: the small kernels add a document's trees in the order of the kernel
    that takes larger batches, so its value is the same bits whatever came with it."""
    import torch

    if switch:
        monkeypatch.setenv("CATBOOST_AMD_" + switch, "0")
    rng = np.random.default_rng(buckets)
    model, hashes = _model_of_buckets(rng, buckets, cats, trees, depth, dim, first)
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    ev = g.evaluator()
    docs = 17_000
    assert ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)["evaluate"] == kernel
    x = rng.normal(size=(docs, buckets)).astype(np.float32)
    for i in range(cats):
        x[:, buckets - cats + i] = rng.choice(hashes[i], size=docs).view(np.float32)
    flat = torch.from_numpy(x).to("cuda:0")
    feats = ev.features(cb.LAYOUT_FLAT_ROWS, flat.data_ptr(), flat.shape[1])
    expected = torch.zeros(docs * dim, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev.eval_data(feats, docs, expected.data_ptr())
    sample = rng.choice(docs, size=500, replace=False)
    np.testing.assert_allclose(expected.cpu().numpy().reshape(docs, dim)[sample], OracleModel(model).calc(x[sample]).reshape(-1, dim),
                               rtol=1e-9, atol=1e-12)
    small = set()
    for n in (1, 33, 700, 1500, 4001):
        small.add(ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, n)["evaluate"].split("<")[0])
        out = torch.full((n * dim,), -3.0, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        ev.eval_data(feats, n, out.data_ptr())
        assert torch.equal(out, expected[:n * dim]), n
    assert {"FewDocumentsKernel", "SmallBatchKernel"} <= small, small


def test_fewer_trees_than_waves_round_alike(monkeypatch):
    import torch

    monkeypatch.setenv("CATBOOST_AMD_REG_KERNEL", "0")
    rng = np.random.default_rng(5)
    for trees in (1, 2, 3, 5, 7):
        g = cb.ModelCalcer()
        g.load_from_dict(mb.build_oblivious([mb.float_feature(f) for f in range(60)], [], 1, [
            ([("float", int(f), float(np.float32(rng.normal()))) for f in rng.choice(60, size=8, replace=False)],
             rng.normal(size=256)) for _ in range(trees)]))
        g.enable_gpu_evaluation(0)
        ev = g.evaluator()
        assert ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, 17_000)["evaluate"] == "EvalObliviousRowTileKernel"
        x = torch.from_numpy(rng.normal(size=(17_000, 60)).astype(np.float32)).to("cuda:0")
        feats = ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), 60)
        out = torch.zeros(17_000, dtype=torch.float64, device="cuda:0")
        part = torch.zeros(900, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        ev.eval_data(feats, 17_000, out.data_ptr())
        for n in (1, 900):
            ev.eval_data(feats, n, part.data_ptr())
            assert torch.equal(part[:n], out[:n])


@pytest.mark.parametrize("n_float,n_cat,dim,docs", [
    (100, 0, 1, (245, 246, 600, 1474, 1475, 5000)),  # columns: 24 K values of few documents, 144 K of more
    (300, 0, 2, (40, 82, 700)),
    (90, 10, 10, (60, 213, 700, 2500, 5461)),        # three passes: rows beyond 2.5 MB of repeated reads
])
def test_host_batches_read_in_place_and_copied(n_float, n_cat, dim, docs):
    """Small host batches on either side of the sizes from which the features are copied to the device first: the bits
    of the device call, rows, columns and split rows."""
    import torch

    rng = np.random.default_rng(n_float)
    model, hashes = _model_of_buckets(rng, n_float + n_cat, n_cat, 200, 6, dim, 1)
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    ev = g.evaluator()
    for n in docs + docs[:1]:
        x = rng.normal(size=(n, n_float + n_cat)).astype(np.float32)
        for i in range(n_cat):
            x[:, n_float + i] = rng.choice(hashes[i], size=n).view(np.float32)
        assert "slices" in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, n)["evaluate"]
        flat = torch.from_numpy(x).to("cuda:0")
        out = torch.zeros(n * dim, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, flat.data_ptr(), flat.shape[1]), n, out.data_ptr())
        expected = out.cpu().numpy()
        np.testing.assert_allclose(expected, OracleModel(model).calc(x), rtol=1e-9, atol=1e-12)
        np.testing.assert_array_equal(g.calc_flat(x), expected)
        np.testing.assert_array_equal(g.calc_flat_transposed(np.ascontiguousarray(x.T)), expected)
        floats, cats = np.ascontiguousarray(x[:, :n_float]), np.ascontiguousarray(x[:, n_float:]).view(np.int32)
        np.testing.assert_array_equal(g.calc_hashed(floats, cats), expected)


def test_categorical_features_without_float_rows():
    """One-hot features alone: the float rows may be a null pointer, in small batches as in large ones."""
    rng = np.random.default_rng(3)
    model, hashes = _model_of_buckets(rng, 12, 12, 80, 6, 1, 1)
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    oracle = OracleModel(model)
    for n in (1, 700, 17_000):
        cats = np.stack([rng.choice(h, size=n) for h in hashes], axis=1)
        np.testing.assert_allclose(g.calc_hashed(np.zeros((n, 0), np.float32), cats),
                                   oracle.calc(np.zeros((n, 0), np.float32), cats, layout="split"), rtol=1e-9, atol=1e-12)


def test_results_of_a_batch_that_a_slice_cannot_address():
    """262 000 documents of 2080 dimensions: more result bytes than a launch addresses, so the trees are not sliced."""
    import torch

    rng = np.random.default_rng(9)
    dim, docs = 2080, 262_000
    model, _ = _model_of_buckets(rng, 4, 0, 70, 1, dim, 1)
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    ev = g.evaluator()
    assert "slices" in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs - 6000)["evaluate"]
    assert "slices" not in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)["evaluate"]
    x = torch.randn(docs, 4, device="cuda:0")
    out = torch.full((docs * dim + 64,), -3.0, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), 4), docs, out.data_ptr())
    assert bool((out[docs * dim:] == -3.0).all())
    out = out[:docs * dim].reshape(docs, dim)
    sample = np.concatenate([rng.choice(docs, size=100, replace=False), [0, docs - 1]])
    np.testing.assert_allclose(out[torch.from_numpy(sample).to("cuda:0")].cpu().numpy(),
                               OracleModel(model).calc(x.cpu().numpy()[sample]).reshape(-1, dim), rtol=1e-9, atol=1e-12)


@pytest.mark.parametrize("dim,n_float", [(1, 100), (3, 40), (9, 30)])
def test_few_host_documents_whose_workgroups_set_flags(dim, n_float):
    """Host batches of up to sixteen workgroups return when the workgroups' flags are set, larger ones with the launch: rows
    and columns, call after call with other values, other calls in between, kernel times, and callers side by side."""
    import threading

    rng = np.random.default_rng(dim)
    ffs = [mb.float_feature(i, i) for i in range(n_float)]
    trees = []
    for t in range(150):
        splits = [("float", int(f), float(np.float32(b))) for f, b in zip(rng.integers(0, n_float, 6), rng.normal(size=6))]
        trees.append((splits, rng.normal(size=64 * dim)))
    model = mb.build_oblivious(ffs, [], dim, trees, scale=0.5, bias=list(rng.normal(size=dim)))
    m = cb.ModelCalcer()
    m.load_from_dict(model)
    m.enable_gpu_evaluation(0)
    x = rng.normal(size=(400, n_float)).astype(np.float32)
    expected = m.calc_flat(x).reshape(400, dim)  # the launch's event
    np.testing.assert_allclose(expected.ravel(), OracleModel(model).calc(x), rtol=1e-9, atol=1e-12)

    def check(seed):
        own = np.random.default_rng(seed)
        for _ in range(60):
            docs = int(own.integers(1, 19))
            at = int(own.integers(0, 400 - docs))
            rows = x[at:at + docs]
            got = m.calc_flat(rows) if own.integers(0, 2) else m.calc_flat_transposed(np.ascontiguousarray(rows.T))
            np.testing.assert_array_equal(got.reshape(docs, dim), expected[at:at + docs])

    check(0)
    m.calc_flat(x[:1])
    binarize_ms, eval_ms = m.evaluator().last_kernel_times()
    assert binarize_ms == 0.0 and 0.0 < eval_ms < 5.0
    failures = []

    def caller(seed):
        try:
            check(seed)
        except BaseException as e:  # noqa: B902
            failures.append(e)

    threads = [threading.Thread(target=caller, args=(s,)) for s in range(1, 7)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures[0]


@pytest.mark.small_batch
@pytest.mark.parametrize("ticket,wait_us", [(0, "1000000"), (2**32 - 21, "1000000"), (0, "0")])
def test_which_wait_ends_calls_of_few_host_documents(monkeypatch, ticket, wait_us):
    """Up to sixteen workgroups the flags end a call, also where the ticket wraps around; above, and where the flags take
    longer than the wait for them, the launch's event does."""
    monkeypatch.setenv("CATBOOST_AMD_FLAG_TICKET", str(ticket))
    monkeypatch.setenv("CATBOOST_AMD_FLAG_WAIT_US", wait_us)
    rng = np.random.default_rng(ticket % 1000)
    ffs = [mb.float_feature(i, i) for i in range(60)]
    trees = []
    for _ in range(300):
        splits = [("float", int(f), float(np.float32(b))) for f, b in zip(rng.integers(0, 60, 6), rng.normal(size=6))]
        trees.append((splits, rng.normal(size=64)))
    model = mb.build_oblivious(ffs, [], 1, trees, bias=[0.25])
    m = cb.ModelCalcer()
    m.load_from_dict(model)
    m.enable_gpu_evaluation(0)
    x = rng.normal(size=(40, 60)).astype(np.float32)
    expected = m.calc_flat(x)  # the launch's event
    np.testing.assert_allclose(expected, OracleModel(model).calc(x), rtol=1e-9, atol=1e-12)

    def flagged():
        return int(m.evaluator().describe_kernels(cb.LAYOUT_FLAT_ROWS, 1)["flagged"])

    assert flagged() == 0
    m.calc_flat(x[:16])  # (makes the memory, which takes longer than the launch)
    began = flagged()
    for call in range(50):
        docs = 1 + call % 16
        np.testing.assert_array_equal(m.calc_flat(x[call % 24:call % 24 + docs]), expected[call % 24:call % 24 + docs])
    assert flagged() - began == (50 if wait_us != "0" else 0)
    for docs in (17, 40):
        np.testing.assert_array_equal(m.calc_flat(x[:docs]), expected[:docs])
    assert flagged() - began == (50 if wait_us != "0" else 0)


@pytest.mark.parametrize("trees,dim", [(64, 1), (513, 3), (544, 1), (545, 1), (1056, 2), (1057, 1)])
def test_slices_are_added_in_order(trees, dim):
    """The kernel that adds the slices keeps sixteen loads in flight: two slices, a whole turn of sixteen after the first
    and one slice more, the same after two turns. The small batches' kernel adds the same slices in the same order."""
    import torch

    from tests.test_oracle import _random_flat_data, _random_oblivious

    rng = np.random.default_rng(trees)
    model, cat_values = _random_oblivious(rng, n_float=12, n_cat=1, trees=trees, max_depth=4, dim=dim, scale=0.5,
                                          bias=rng.normal(size=dim))
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    ev = g.evaluator()
    docs = 16_641
    assert "CombineSlicesKernel" in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)["evaluate"]
    assert "SmallBatchKernel" in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, 4000)["evaluate"]
    flat = torch.from_numpy(_random_flat_data(rng, model, cat_values, docs)).to("cuda:0")
    out = torch.full((docs * dim + 8,), -3.0, dtype=torch.float64, device="cuda:0")
    part = torch.zeros(4000 * dim, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, flat.data_ptr(), flat.shape[1]), docs, out.data_ptr())
    for begin in (0, docs - 4000):
        ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, flat[begin:].data_ptr(), flat.shape[1]), 4000, part.data_ptr())
        assert torch.equal(part, out[begin * dim:(begin + 4000) * dim])
    assert bool((out[docs * dim:] == -3.0).all())


@pytest.mark.parametrize("trees,dim", [(96, 1), (128, 3), (160, 1), (320, 2), (321, 1)])
def test_few_slices_are_added_in_order(trees, dim):
    """Three loads in flight up to ten slices: a turn that ends in the last slice's again, whole turns, the first number with sixteen."""
    test_slices_are_added_in_order(trees, dim)


@pytest.mark.parametrize("trees,limit", [(500, 16384), (501, 12288), (812, 12288), (813, 10240)])
def test_small_batches_of_models_with_many_levels(trees, limit):
    """Models of more levels leave the small-batch kernel for the binarize and register kernels earlier; both add the same slices."""
    import torch

    model, info = syn.build_model("C2", trees=trees)
    model.enable_gpu_evaluation(0)
    ev = model.evaluator()
    x = syn.device_features(info, limit + 1)
    out = []
    for docs in (limit, limit + 1):
        result = torch.full((docs,), -1.0, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        ev.eval_data(ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), x.shape[1]), docs, result.data_ptr())
        out.append(result)
        assert ("SmallBatch" in ev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs)["evaluate"]) == (docs == limit)
        assert (ev.last_kernel_times()[0] == 0.0) == (docs == limit)
    assert torch.equal(out[0], out[1][:limit])
    np.testing.assert_array_equal(model.calc_flat(x[-700:].cpu().numpy()), out[1][-700:].cpu().numpy())  # SmallBatchKernel, from host memory
