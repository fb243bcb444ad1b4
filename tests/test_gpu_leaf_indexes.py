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
