"""Leaf indexes written in whole lines by shares of the trees: group, share and line edges against the oracle. Needs an
MI355X."""
import numpy as np
import pytest

import catboost_amd as cb
from catboost_amd import synthetic as syn
from oracle.cbm_reader import read_cbm
from oracle.oracle import OracleModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg,trees,docs", [
    ("C1", 1, 1), ("C1", 63, 257), ("C1", 64, 256), ("C1", 65, 255), ("C1", 128, 64), ("C1", 200, 1000),  # six levels
    ("C2", 97, 300), ("C2", 160, 513), ("C2", 416, 70), ("C2B", 131, 300),  # eight levels; bins above 127
])
def test_leaf_indexes_at_the_edges_of_groups_shares_and_lines(cfg, trees, docs):
    import torch

    model, info = syn.build_model(cfg, trees=trees)
    model.enable_gpu_evaluation(0)
    ev = model.evaluator()
    x = syn.device_features(info, docs)
    expected = OracleModel(read_cbm(model.save_to_buffer())).leaf_indexes(x.cpu().numpy())
    bins = torch.zeros(ev.quantized_bytes(docs), dtype=torch.uint8, device="cuda:0")
    torch.cuda.synchronize()
    ev.quantize(ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), x.shape[1]), docs, bins.data_ptr())
    for begin, end in {(0, trees), (trees // 3, trees), (0, max(1, trees - 1)), (trees // 2, trees // 2 + 1)}:
        for shift in (0, 1, 31):  # rows that start anywhere in a line; the words around the result stay as they are
            count = docs * (end - begin)
            out = torch.full((shift + count + 40,), -7, dtype=torch.int32, device="cuda:0")
            torch.cuda.synchronize()
            ev.leaf_indexes_quantized(bins.data_ptr(), docs, out.data_ptr() + 4 * shift, begin, end)
            ev.synchronize()
            got = out.cpu().numpy()
            np.testing.assert_array_equal(got[shift:shift + count].reshape(docs, end - begin), expected[:, begin:end])
            assert (got[:shift] == -7).all() and (got[shift + count:] == -7).all()


@pytest.mark.parametrize("cfg", ["C1", "C2", "C2B"])
def test_leaf_indexes_of_bins_at_an_address_that_is_no_multiple_of_sixteen(cfg):
    """A caller's buffer of bins may start at any multiple of four."""
    import torch

    trees, docs = 130, 700
    model, info = syn.build_model(cfg, trees=trees)
    model.enable_gpu_evaluation(0)
    ev = model.evaluator()
    x = syn.device_features(info, docs)
    expected = OracleModel(read_cbm(model.save_to_buffer())).leaf_indexes(x.cpu().numpy())
    size = ev.quantized_bytes(docs)
    bins = torch.zeros(size, dtype=torch.uint8, device="cuda:0")
    torch.cuda.synchronize()
    ev.quantize(ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), x.shape[1]), docs, bins.data_ptr())
    ev.synchronize()
    for shift in (4, 8, 12):
        moved = torch.full((size + 16,), 0xff, dtype=torch.uint8, device="cuda:0")
        moved[shift:shift + size] = bins
        out = torch.full((docs, trees), -7, dtype=torch.int32, device="cuda:0")
        torch.cuda.synchronize()
        ev.leaf_indexes_quantized(moved.data_ptr() + shift, docs, out.data_ptr(), 0, trees)
        ev.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), expected)


@pytest.mark.parametrize("buckets,trees,depth,one_hot,docs", [
    (508, 161, 8, False, 300), (509, 161, 8, False, 300),   # the widest tile beside groups of 64 trees; groups of 32
    (575, 130, 6, False, 515), (576, 97, 8, False, 70), (576, 224, 8, True, 257), (540, 193, 6, False, 256),
    (577, 130, 8, False, 300),                              # no room for a tile
])
def test_leaf_indexes_of_wide_models(buckets, trees, depth, one_hot, docs):
    """Group, share and line edges where the tile leaves room for the smaller groups only."""
    import torch

    from oracle import model_builder as mb

    rng = np.random.default_rng(buckets + trees)
    cats = 8 if one_hot else 0
    floats = buckets - cats
    hashes = rng.integers(-2**31, 2**31, size=(cats, 5), dtype=np.int64).astype(np.int32)
    column = list(rng.permutation(buckets)) + [int(v) for v in rng.integers(0, buckets, size=trees * depth - buckets)]
    tree_list = []
    for t in range(trees):
        splits = []
        for c in column[t * depth:(t + 1) * depth]:
            if c < floats:
                splits.append(("float", int(c), float(np.float32(rng.normal()))))
            else:
                splits.append(("onehot", int(c - floats), int(rng.choice(hashes[c - floats]))))
        tree_list.append((splits, np.zeros(1 << depth)))
    model = mb.build_oblivious([mb.float_feature(f) for f in range(floats)],
                               [mb.cat_feature(i, floats + i) for i in range(cats)], 1, tree_list)
    g = cb.ModelCalcer()
    g.load_from_dict(model)
    g.enable_gpu_evaluation(0)
    assert g.bucket_count == buckets
    ev = g.evaluator()
    x = rng.normal(size=(docs, buckets)).astype(np.float32)
    for i in range(cats):
        x[:, floats + i] = rng.choice(hashes[i], size=docs).view(np.float32)
    expected = OracleModel(model).leaf_indexes(x)
    flat = torch.from_numpy(x).to("cuda:0")
    bins = torch.zeros(ev.quantized_bytes(docs), dtype=torch.uint8, device="cuda:0")
    torch.cuda.synchronize()
    ev.quantize(ev.features(cb.LAYOUT_FLAT_ROWS, flat.data_ptr(), flat.shape[1]), docs, bins.data_ptr())
    for begin, end in {(0, trees), (trees // 3, trees), (0, 32), (1, 66), (trees // 2, trees // 2 + 1)}:
        for shift in (0, 1, 31):
            count = docs * (end - begin)
            out = torch.full((shift + count + 40,), -7, dtype=torch.int32, device="cuda:0")
            torch.cuda.synchronize()
            ev.leaf_indexes_quantized(bins.data_ptr(), docs, out.data_ptr() + 4 * shift, begin, end)
            ev.synchronize()
            got = out.cpu().numpy()
            np.testing.assert_array_equal(got[shift:shift + count].reshape(docs, end - begin), expected[:, begin:end])
            assert (got[:shift] == -7).all() and (got[shift + count:] == -7).all()


@pytest.mark.parametrize("cfg,trees,docs", [("C1", 200, 336_001), ("C2B", 131, 513_000), ("C2", 416, 161_500)])
def test_leaf_indexes_larger_than_the_memory_side_cache(cfg, trees, docs):
    """More than 256 MB of indexes take streaming stores: the same indexes as two calls for halves of the documents."""
    import torch

    model, info = syn.build_model(cfg, trees=trees)
    model.enable_gpu_evaluation(0)
    ev = model.evaluator()
    x = syn.device_features(info, docs)
    half = docs // 512 * 256
    assert docs * trees * 4 > 256 << 20 > (docs - half) * trees * 4
    pitch = ev.quantized_bytes(256)
    bins = torch.zeros(ev.quantized_bytes(docs), dtype=torch.uint8, device="cuda:0")
    out = torch.full((2, docs, trees), -7, dtype=torch.int32, device="cuda:0")
    torch.cuda.synchronize()
    ev.quantize(ev.features(cb.LAYOUT_FLAT_ROWS, x.data_ptr(), x.shape[1]), docs, bins.data_ptr())
    ev.leaf_indexes_quantized(bins.data_ptr(), docs, out[0].data_ptr())
    ev.leaf_indexes_quantized(bins.data_ptr(), half, out[1].data_ptr())
    ev.leaf_indexes_quantized(bins.data_ptr() + half // 256 * pitch, docs - half, out[1, half:].data_ptr())
    ev.synchronize()
    assert torch.equal(out[0], out[1])
    expected = OracleModel(read_cbm(model.save_to_buffer())).leaf_indexes(x[-700:].cpu().numpy())
    np.testing.assert_array_equal(out[0, -700:].cpu().numpy(), expected)
