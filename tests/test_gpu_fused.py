"""The fused kernels (binarize + evaluate in one launch, the bins in registers only) against the two-launch
path and the oracle. Needs an MI355X.

CbHipEvalData and the host entry points take a fused kernel for float-only one-dimensional oblivious
models whose rows are at least sixteen columns wide and whose used columns make at most four units of sixteen
or five (the kernels of 64 and 80 bins registers) or which have more than 96 buckets (the kernel of 208); CATBOOST_AMD_FUSED=0
keeps an evaluator on the two launches. Both add the leaves in tree order in fp64: results must be equal bit for bit, and within
1e-9 relative / 1e-12 absolute of the oracle.
"""
import numpy as np
import pytest

import catboost_amd as cb
from catboost_amd import synthetic as syn
from oracle import model_builder as mb
from oracle.cbm_reader import read_cbm
from oracle.oracle import OracleModel

pytestmark = pytest.mark.gpu


def _evaluators(model_bytes, monkeypatch):
    """(fused, two-launch) evaluators of one model."""
    out = []
    for switch in ("1", "0"):
        monkeypatch.setenv("CATBOOST_AMD_FUSED", switch)
        m = cb.ModelCalcer(buffer=model_bytes)
        m.enable_gpu_evaluation(0)
        out.append((m, m.evaluator()))
    monkeypatch.delenv("CATBOOST_AMD_FUSED")
    return out


def _compare(model_bytes, x, monkeypatch, stride=None):
    import torch

    oracle = OracleModel(read_cbm(model_bytes))
    (fm, fev), (tm, tev) = _evaluators(model_bytes, monkeypatch)
    docs, width = x.shape
    stride = stride or width
    padded = np.full((docs, stride), np.float32(7.5))
    padded[:, :width] = x
    dx = torch.from_numpy(np.ascontiguousarray(padded, np.float32)).to("cuda:0")
    a = torch.full((docs,), -1.0, dtype=torch.float64, device="cuda:0")
    b = torch.full((docs,), -2.0, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    fev.eval_data(fev.features(cb.LAYOUT_FLAT_ROWS, dx.data_ptr(), stride), docs, a.data_ptr())
    tev.eval_data(tev.features(cb.LAYOUT_FLAT_ROWS, dx.data_ptr(), stride), docs, b.data_ptr())
    torch.cuda.synchronize()
    assert fev.last_kernel_times()[0] == 0.0, "the fused kernel did not run"
    assert tev.last_kernel_times()[0] > 0.0
    assert torch.equal(a, b)
    np.testing.assert_allclose(a.cpu().numpy(), oracle.calc(x, threads=8), rtol=1e-9, atol=1e-12)
    # the host entry point takes the same kernel
    np.testing.assert_array_equal(fm.calc_flat(x[:3000]), a.cpu().numpy()[:3000])
    return a


@pytest.mark.parametrize("cfg,trees,docs", [("C2", 50, 1), ("C2", 50, 255), ("C2", 50, 257), ("C2", 64, 5000),
                                             ("C2", 1000, 20000), ("C2", 200, 30011),
                                             ("C1", 200, 5000), ("C1", 37, 1), ("C1", 37, 2049)])
def test_fused_equals_two_launches(cfg, trees, docs, monkeypatch):
    model, info = syn.build_model(cfg, trees=trees)
    x = syn.host_features(info, docs, seed=3)
    _compare(model.save_to_buffer(), x, monkeypatch)
    if docs == 5000:
        _compare(model.save_to_buffer(), x, monkeypatch, stride=x.shape[1] + 5)


def _random_model(rng, columns, used, trees, depth, borders_of, nan_true=()):
    """An oblivious model over `columns` float columns of which `used` are split on; borders_of(f) draws
    the candidate borders of column f."""
    feats = []
    for f in range(columns):
        ff = mb.float_feature(f)
        if f in nan_true:
            ff["has_nans"], ff["nan_treatment"] = True, 2
        feats.append(ff)
    cands = {f: np.unique(np.asarray(borders_of(f), np.float32)) for f in used}
    tree_list = []
    for _ in range(trees):
        splits = []
        for _ in range(depth):
            f = int(rng.choice(used))
            splits.append(("float", f, float(rng.choice(cands[f]))))
        tree_list.append((splits, rng.normal(0, 0.01, size=1 << depth)))
    return mb.build_oblivious(feats, [], 1, tree_list, scale=0.75, bias=[0.125])


def _bytes(model_dict):
    m = cb.ModelCalcer()
    m.load_from_dict(model_dict)
    return m.save_to_buffer()


def test_fused_sparse_columns_clustered_borders_and_nan_as_true(monkeypatch):
    """Columns that no split reads between the used ones, a row whose last unit is moved back, borders so
    close together that a grid cell holds up to fifteen of them (three and four search steps), NaN that
    counts as +inf, values on the borders and infinities."""
    rng = np.random.default_rng(11)
    columns = 203
    used = sorted(set(rng.choice(columns, size=125, replace=False).tolist() + [202]))

    def borders_of(f):
        if f % 3 == 0:  # clustered: a few tight groups far apart
            centers = rng.normal(0, 3, size=4)
            return np.concatenate([c + rng.normal(0, 1e-3, size=rng.integers(3, 12)) for c in centers])
        return rng.normal(0, 1, size=rng.integers(1, 50))

    model = _random_model(rng, columns, used, trees=420, depth=8, borders_of=borders_of, nan_true=set(used[::4]))
    x = rng.normal(0, 2, size=(6000, columns)).astype(np.float32)
    for f in used:
        b = np.asarray(model["float_features"][f]["borders"], np.float32)
        rows = rng.integers(0, x.shape[0], size=200)
        x[rows, f] = rng.choice(b, size=200)
    x[rng.random(x.shape) < 0.05] = np.nan
    x[rng.random(x.shape) < 0.01] = np.inf
    x[rng.random(x.shape) < 0.01] = -np.inf
    _compare(_bytes(model), x, monkeypatch)


def test_fused_shallow_trees_and_mixed_depths(monkeypatch):
    rng = np.random.default_rng(5)
    columns = 130
    feats = [mb.float_feature(f) for f in range(columns)]
    trees = []
    for t in range(160):
        depth = int(rng.integers(0, 9))
        splits = [("float", int(rng.integers(0, columns)), float(np.float32(rng.normal()))) for _ in range(depth)]
        trees.append((splits, rng.normal(0, 0.01, size=1 << depth)))
    model = mb.build_oblivious(feats, [], 1, trees)
    x = rng.normal(size=(3001, columns)).astype(np.float32)
    _compare(_bytes(model), x, monkeypatch)


@pytest.mark.parametrize("columns,used_count,depth,max_borders,shape",
                         [(16, 16, 8, 120, 64), (23, 9, 8, 40, 64), (64, 64, 6, 30, 64), (50, 50, 8, 126, 64),
                          (300, 40, 7, 60, 64), (61, 33, 3, 5, 64), (80, 80, 8, 100, 80), (70, 70, 6, 30, 80),
                          (77, 60, 5, 126, 80)])
def test_fused_small_models(columns, used_count, depth, max_borders, shape, monkeypatch):
    """Models of at most four or five units: the fused kernels of 64 and 80 bins registers, in their seven-bit
    form (a feature with more than 63 borders) and their six-bit form, behind the six-level and the eight-level
    evaluate kernels' tables (the fused kernel then walks six or eight levels), with used columns far apart (300 columns, 40 of them used in three clusters) and a
    last unit that is moved back into the row."""
    rng = np.random.default_rng(columns * 1000 + used_count)
    if columns == 300:
        used = sorted(set(range(3, 17)) | set(range(140, 153)) | set(range(287, 300)))
    else:
        used = sorted(rng.choice(columns, size=used_count, replace=False).tolist())
    model = _random_model(rng, columns, used, trees=150, depth=depth,
                          borders_of=lambda f: rng.normal(0, 1, size=rng.integers(1, max_borders + 1)),
                          nan_true=set(used[::3]))
    x = rng.normal(0, 1.5, size=(4099, columns)).astype(np.float32)
    for f in used:
        b = np.asarray(model["float_features"][f]["borders"], np.float32)
        rows = rng.integers(0, x.shape[0], size=100)
        x[rows, f] = rng.choice(b, size=100)
    x[rng.random(x.shape) < 0.03] = np.nan
    x[rng.random(x.shape) < 0.01] = np.inf
    (fm, fev), _ = _evaluators(_bytes(model), monkeypatch)
    name = fev.describe_kernels(cb.LAYOUT_FLAT_ROWS, x.shape[0]).get("fused", "")
    assert name.startswith("cbamd_fused_b%d_w8" % shape)
    assert ("_d6" in name) == (depth <= 6), "models of depth <= 6 take the form that walks six levels"
    _compare(_bytes(model), x, monkeypatch)
    _compare(_bytes(model), x[:300], monkeypatch, stride=columns + 3)


@pytest.mark.parametrize("max_depth,borders", [(6, 40), (5, 100), (7, 40)])
def test_fused_wide_models_by_depth(max_depth, borders, monkeypatch):
    """The fused kernel of 208 bins registers in its six-level form (models of depth <= 6) and its eight-level
    form, six-bit and seven-bit."""
    rng = np.random.default_rng(max_depth * 100 + borders)
    columns = 170
    used = list(range(columns))
    feats_borders = {f: rng.normal(0, 1, size=rng.integers(1, borders + 1)) for f in used}
    model = _random_model(rng, columns, used, trees=90, depth=max_depth, borders_of=lambda f: feats_borders[f])
    x = rng.normal(0, 1.5, size=(2500, columns)).astype(np.float32)
    x[rng.random(x.shape) < 0.02] = np.nan
    (fm, fev), _ = _evaluators(_bytes(model), monkeypatch)
    name = fev.describe_kernels(cb.LAYOUT_FLAT_ROWS, x.shape[0]).get("fused", "")
    assert name.startswith("cbamd_fused_b208_w4") and ("_d6" in name) == (max_depth <= 6)
    _compare(_bytes(model), x, monkeypatch)


def test_fused_split_rows_layout(monkeypatch):
    """Separate float rows (the Index positions of the model's features, which need not be their flat positions)
    take the fused kernel of their own unit tables."""
    import torch

    rng = np.random.default_rng(21)
    columns = 150
    feats = []
    for f in range(columns):
        ff = mb.float_feature(f, flat_index=2 * f + 1)  # flat positions differ from the float positions
        feats.append(ff)
    trees = []
    for _ in range(64):
        splits = [("float", int(rng.integers(0, columns)), float(np.float32(rng.normal()))) for _ in range(8)]
        trees.append((splits, rng.normal(0, 0.01, size=256)))
    model_bytes = _bytes(mb.build_oblivious(feats, [], 1, trees))
    oracle = OracleModel(read_cbm(model_bytes))
    x = rng.normal(size=(7001, columns)).astype(np.float32)
    x[rng.random(x.shape) < 0.03] = np.nan
    (fm, fev), (tm, tev) = _evaluators(model_bytes, monkeypatch)
    dx = torch.from_numpy(x).to("cuda:0")
    a = torch.zeros(x.shape[0], dtype=torch.float64, device="cuda:0")
    b = torch.zeros_like(a)
    torch.cuda.synchronize()
    fev.eval_data(fev.features(cb.LAYOUT_SPLIT_ROWS, dx.data_ptr(), columns), x.shape[0], a.data_ptr())
    tev.eval_data(tev.features(cb.LAYOUT_SPLIT_ROWS, dx.data_ptr(), columns), x.shape[0], b.data_ptr())
    torch.cuda.synchronize()
    assert fev.last_kernel_times()[0] == 0.0 and tev.last_kernel_times()[0] > 0.0
    assert torch.equal(a, b)
    np.testing.assert_array_equal(a.cpu().numpy(), oracle.calc(x, layout="split", threads=8))
    np.testing.assert_array_equal(fm.calc_hashed(x, np.zeros((x.shape[0], 0), np.int32)), a.cpu().numpy())


@pytest.mark.parametrize("columns,depth,shape", [(24, 8, 64), (24, 6, 64), (12, 7, 64), (150, 8, 208), (150, 6, 208), (130, 7, 208)])
def test_fused_images_with_units_that_the_model_lacks(columns, depth, shape, monkeypatch):
    """Six-bit models of one, two, nine and ten units of sixteen columns: the last image then holds two or three units in a
    row that the model lacks. All documents of a batch that keeps every CU busy against the two launches, bit for bit."""
    import torch

    rng = np.random.default_rng(columns * 10 + depth)
    width = max(columns, 16)
    model = _random_model(rng, width, list(range(columns)), trees=60, depth=depth,
                          borders_of=lambda f: rng.normal(0, 1, size=rng.integers(20, 60)))
    (_, fev), (_, tev) = _evaluators(_bytes(model), monkeypatch)
    docs = 1_000_003 if columns < 100 else 400_009
    name = fev.describe_kernels(cb.LAYOUT_FLAT_ROWS, docs).get("fused", "")
    assert name.startswith("cbamd_fused_b%d_w" % shape) and name.endswith("_s")
    generator = torch.Generator(device="cuda:0")
    generator.manual_seed(columns)
    dx = torch.randn(docs, width, device="cuda:0", generator=generator)
    a = torch.full((docs,), -1.0, dtype=torch.float64, device="cuda:0")
    b = torch.full((docs,), -2.0, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    for _ in range(3):
        fev.eval_data(fev.features(cb.LAYOUT_FLAT_ROWS, dx.data_ptr(), width), docs, a.data_ptr())
        tev.eval_data(tev.features(cb.LAYOUT_FLAT_ROWS, dx.data_ptr(), width), docs, b.data_ptr())
        assert fev.last_kernel_times()[0] == 0.0 and tev.last_kernel_times()[0] > 0.0
        assert torch.equal(a, b)
        a.fill_(-1.0)
        torch.cuda.synchronize()


@pytest.mark.parametrize("columns,trees", [(40, t) for t in (1, 16, 17, 32, 33, 48, 49, 63, 64, 65, 80, 112, 127, 128, 129, 144, 193)] +
                         [(110, t) for t in (63, 64, 65, 96, 128, 129, 193)])
def test_fused_six_level_walks_end_behind_any_sixteenth_tree(columns, trees, monkeypatch):
    """The six-level kernels' buffers hold 64 trees of 64 leaves, and a walk may end after any sixteen of them."""
    rng = np.random.default_rng(trees * 7 + columns)
    model = _bytes(_random_model(rng, columns, list(range(columns)), trees, 6, lambda f: rng.normal(0, 1, size=12)))
    _compare(model, rng.normal(0, 1, size=(1100, columns)).astype(np.float32), monkeypatch)


@pytest.mark.parametrize("columns,used", [(20, list(range(20))), (40, [3, 4, 9, 21, 22, 23, 24, 33, 39]), (17, [16]), (90, list(range(0, 90, 5)))])
@pytest.mark.parametrize("few", [True, False])
def test_fused_grids_at_their_edges(columns, used, few, monkeypatch):
    """Borders far from zero, a few denormal numbers apart, further apart than a float holds, one border, many in one cell; values
    on them and next to them, infinities and NaN; sixteens and fours of columns of which splits look at some or none. Rows and
    columns."""
    import torch

    rng = np.random.default_rng(columns + few)
    count = 15 if few else 70  # the six-bit form and the other one

    def borders_of(f):
        n = rng.integers(1, count)
        return [1e6 + rng.integers(0, 64, size=n) / 16.0, rng.integers(-7, 7, size=n) * 1.5e-45, [-3e38, 0.0, 3e38], [0.25],
                rng.normal(size=n), [-0.0, 1e-30, 1.0], -1e20 - rng.random(n) * 1e15][f % 7]

    model = _random_model(rng, columns, used, trees=300, depth=6, borders_of=borders_of, nan_true=set(used[::3]))
    borders = {f: model["float_features"][f]["borders"] for f in used}
    x = rng.normal(size=(3000, columns)).astype(np.float32)
    for f, b in borders.items():
        if len(b):
            near = np.concatenate([b, np.nextafter(b, np.float32(np.inf)), np.nextafter(b, np.float32(-np.inf))])
            x[100:, f] = rng.choice(near, size=2900)
    x[rng.random(x.shape) < 0.02] = np.nan
    x[rng.random(x.shape) < 0.02] = np.inf
    x[rng.random(x.shape) < 0.02] = -np.inf
    rows = _compare(_bytes(model), x, monkeypatch)
    (_, fev), _ = _evaluators(_bytes(model), monkeypatch)
    dx = torch.from_numpy(np.ascontiguousarray(x.T)).to("cuda:0")
    out = torch.zeros(len(x), dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    fev.eval_data(fev.features(cb.LAYOUT_FLAT_COLUMNS, dx.data_ptr(), len(x)), len(x), out.data_ptr())
    assert fev.last_kernel_times()[0] == 0.0, "the fused kernel did not run"
    assert torch.equal(out, rows)
