"""The fused kernels of column-major documents (binarize + evaluate in one launch) against the two launches and the oracle, at the
edges of units, images, document blocks and shapes. Needs an MI355X."""
import numpy as np
import pytest

import catboost_amd as cb
from oracle import model_builder as mb
from oracle.oracle import OracleModel

pytestmark = pytest.mark.gpu


def _model(rng, n_float, used, borders, depth, trees, nans):
    """A model over `used` of n_float columns, every one of them in use."""
    columns = np.sort(rng.choice(n_float, size=used, replace=False))
    ffs = [mb.float_feature(i, i, has_nans=nans, nan_treatment=2 if nans and i % 3 else 0) for i in range(n_float)]
    cands = {int(f): np.unique(rng.normal(size=6 * borders).astype(np.float32))[:borders] for f in columns}
    order = [int(f) for f in columns] * (1 + trees * depth // used)
    splits, out = iter(order), []
    for t in range(max(trees, (used + depth - 1) // depth)):
        levels = depth if t % 4 else 1 + t % depth
        out.append(([("float", f, float(rng.choice(cands[f]))) for f in (next(splits, order[0]) for _ in range(levels))], None))
    for f in columns[::7]:  # one of the features with every border in use
        out.extend(([("float", int(f), float(b)) for b in cands[int(f)][at:at + depth]], None) for at in range(0, borders, depth))
    for f in columns:
        out.append(([("float", int(f), float(cands[int(f)][0]))], None))
    trees = [(s, rng.normal(size=1 << len(s))) for s, _ in out]
    return mb.build_oblivious(ffs, [], 1, trees, scale=0.75, bias=[0.25]), cands


def _eval(model, x, stride, monkeypatch, fused):
    import torch

    monkeypatch.setenv("CATBOOST_AMD_FUSED", fused)
    m = cb.ModelCalcer()
    m.load_from_dict(model)
    m.enable_gpu_evaluation(0)
    ev = m.evaluator()
    docs, width = x.shape
    columns = torch.full((width * stride,), 7.5, dtype=torch.float32, device="cuda:0")
    columns.view(width, stride)[:, :docs] = torch.from_numpy(np.ascontiguousarray(x.T)).to("cuda:0")
    out = torch.full((docs + 1,), -1.0, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev.eval_data(ev.features(cb.LAYOUT_FLAT_COLUMNS, columns.data_ptr(), stride), docs, out.data_ptr())
    assert out[docs] == -1.0
    return m, ev, out[:docs].cpu().numpy()


@pytest.mark.parametrize("n_float,used,borders,depth,docs,pad,shape", [
    (1, 1, 20, 6, 300, 0, "b64_w8_d6_s"), (15, 15, 63, 6, 257, 1, "b64_w8_d6_s"), (20, 16, 64, 8, 255, 0, "b64_w8_s"),
    (17, 17, 30, 6, 1, 0, "b64_w8_d6_s"), (64, 64, 30, 8, 1000, 3, "b64_w8_s"), (90, 65, 30, 6, 5000, 0, "b80_w8_d6_s"),
    (80, 80, 100, 8, 513, 2, "b80_w8"), (64, 33, 128, 6, 700, 0, "b64_w8_d6"), (97, 97, 30, 6, 2049, 0, "b160_w4_d6_s"),
    (130, 128, 63, 8, 300, 5, "b160_w4_s"), (160, 160, 20, 6, 4096, 0, "b160_w4_d6_s"), (161, 161, 20, 8, 900, 0, "b208_w4_s"),
    (208, 208, 20, 6, 1500, 1, "b208_w4_d6_s"), (200, 150, 127, 6, 600, 0, "b160_w4_d6"), (208, 193, 128, 8, 300, 0, "b208_w4"),
    (96, 90, 20, 6, 300, 0, "b160_w4_d6_s"), (209, 209, 10, 6, 300, 0, ""),
])
def test_fused_columns_equal_the_two_launches(monkeypatch, n_float, used, borders, depth, docs, pad, shape):
    rng = np.random.default_rng(n_float * 1000 + used + borders)
    model, cands = _model(rng, n_float, used, borders, depth, 60, nans=n_float % 2 == 0)
    x = rng.normal(size=(docs, n_float)).astype(np.float32)
    for f, c in cands.items():
        x[::5, f] = rng.choice(c, size=len(x[::5]))  # on the borders
    x[rng.random(x.shape) < 0.03] = np.nan
    x[rng.random(x.shape) < 0.01] = np.inf
    x[rng.random(x.shape) < 0.01] = -np.inf
    m, ev, a = _eval(model, x, docs + pad, monkeypatch, "1")
    assert ev.describe_kernels(cb.LAYOUT_FLAT_COLUMNS, docs).get("fused", "") == (shape and "cbamd_fused_cols_" + shape)
    if shape:
        assert ev.last_kernel_times()[0] == 0.0, "the fused kernel did not run"
    _, tev, b = _eval(model, x, docs + pad, monkeypatch, "0")
    assert "fused" not in tev.describe_kernels(cb.LAYOUT_FLAT_COLUMNS, docs)
    np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(a, OracleModel(model).calc(x))
    np.testing.assert_array_equal(m.calc_flat_transposed(np.ascontiguousarray(x.T)), a)


def test_columns_further_apart_than_32_bits_reach(monkeypatch):
    rng = np.random.default_rng(3)
    model, _ = _model(rng, 40, 40, 20, 6, 30, nans=False)
    x = rng.normal(size=(1000, 40)).astype(np.float32)
    _, ev, a = _eval(model, x, 30_000_001, monkeypatch, "1")  # 4.8 GB from the first column to the last
    assert "fused" in ev.describe_kernels(cb.LAYOUT_FLAT_COLUMNS, 1000)
    np.testing.assert_array_equal(a, OracleModel(model).calc(x))


@pytest.mark.parametrize("docs", [410_003, 1_100_003])
def test_large_batches_of_columns(monkeypatch, docs):
    """More workgroups than CUs, and more than the chip holds at a time."""
    rng = np.random.default_rng(4)
    model, _ = _model(rng, 120, 120, 40, 6, 100, nans=False)
    x = rng.standard_normal((docs, 120), dtype=np.float32)
    _, ev, a = _eval(model, x, docs, monkeypatch, "1")
    assert ev.describe_kernels(cb.LAYOUT_FLAT_COLUMNS, docs)["fused"] == "cbamd_fused_cols_b160_w4_d6_s"
    assert ev.last_kernel_times()[0] == 0.0, "the fused kernel did not run"
    np.testing.assert_array_equal(a, OracleModel(model).calc(x, threads=8))


def test_refused_columns_stay_refused():
    import torch

    rng = np.random.default_rng(5)
    model, _ = _model(rng, 20, 20, 20, 6, 10, nans=False)
    m = cb.ModelCalcer()
    m.load_from_dict(model)
    m.enable_gpu_evaluation(0)
    ev = m.evaluator()
    x = torch.zeros(20 * 300, dtype=torch.float32, device="cuda:0")
    out = torch.zeros(300, dtype=torch.float64, device="cuda:0")
    with pytest.raises(Exception, match="column stride is shorter"):
        ev.eval_data(ev.features(cb.LAYOUT_FLAT_COLUMNS, x.data_ptr(), 299), 300, out.data_ptr())


@pytest.mark.small_batch
@pytest.mark.parametrize("used,trees,docs,fused", [
    (1, 30, 530_000, False), (4, 100, 530_001, False), (11, 30, 600_000, False), (8, 300, 530_000, True), (12, 30, 530_000, True),
    (4, 30, 520_000, True), (16, 30, 530_000, True), (17, 30, 530_000, True),
])
def test_models_of_few_columns(monkeypatch, used, trees, docs, fused):
    """Large column-major batches of models with few buckets and few trees take two launches; both give the sums of one pass."""
    rng = np.random.default_rng(used + trees)
    model, _ = _model(rng, used, used, 6, 6, trees, nans=False)
    x = rng.standard_normal((docs, used), dtype=np.float32)
    x[::7, 0] = np.nan
    _, ev, a = _eval(model, x, docs, monkeypatch, "1")
    assert ("fused" in ev.describe_kernels(cb.LAYOUT_FLAT_COLUMNS, docs)) == fused
    assert (ev.last_kernel_times()[0] == 0.0) == fused
    np.testing.assert_array_equal(a, OracleModel(model).calc(x, threads=8))


@pytest.mark.small_batch
@pytest.mark.parametrize("used,trees,docs,fused", [(20, 1000, 262_144, False), (30, 600, 300_001, False), (20, 1000, 393_215, False), (20, 1000, 393_217, True),
                                                   (20, 100, 262_144, True), (60, 300, 290_000, True), (80, 1200, 270_000, False),
                                                   (150, 1000, 262_144, True)])
def test_medium_batches_of_many_trees(monkeypatch, used, trees, docs, fused):
    """Medium column-major batches of models with many trees are cut into slices, as smaller ones are."""
    import torch

    rng = np.random.default_rng(used + trees)
    model, _ = _model(rng, used, used, 6, 6, trees, nans=False)
    x = rng.standard_normal((docs, used), dtype=np.float32)
    _, ev, a = _eval(model, x, docs, monkeypatch, "1")
    kernels = ev.describe_kernels(cb.LAYOUT_FLAT_COLUMNS, docs)
    assert ("fused" in kernels) == fused and ("slices" in kernels.get("evaluate", "")) != fused
    assert (ev.last_kernel_times()[0] == 0.0) == fused
    pick = np.r_[0:600, docs - 600:docs]
    expected = OracleModel(model).calc(x[pick])
    np.testing.assert_allclose(a[pick], expected, rtol=1e-9, atol=1e-12)
    # without memory for slices: one pass, fused whatever the trees
    columns = torch.from_numpy(np.ascontiguousarray(x.T)).to("cuda:0")
    out = torch.zeros(docs, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    ev.eval_data_no_alloc(ev.features(cb.LAYOUT_FLAT_COLUMNS, columns.data_ptr(), docs), docs, out.data_ptr())
    ev.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy()[pick], expected)
