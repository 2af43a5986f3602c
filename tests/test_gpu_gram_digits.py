"""t(X) %*% X of byte-code blocks on the integer matrix cores (k_gram_tiles_i8, option tsmm_digits): the edges of its tiles and of its roles
of waves, sums at their largest, long shares of the rows, and the blocks whose values its digits do not suit."""
import numpy as np
import pytest

from parity import assert_matches_truth
from test_gpu_gram_tiles import columns

pytestmark = pytest.mark.gpu


def product(cla, specs, n_rows, n_cols, digits, options=()):
    blk = cla.build_block(n_rows, n_cols, specs)
    for key, value in (("tsmm_digits", digits), *options):
        blk.set_option(key, value)
    out, nnz = blk.tsmm()
    lds = {k["lds"] for k in blk.stats()["kernels"] if k["name"] == "k_gram_tiles"}
    blk.close()
    return out, nnz, lds


@pytest.mark.parametrize("n_cols", [17, 31, 32, 33, 48, 49, 50, 52, 53, 64, 65, 68, 80, 81, 82, 84, 85, 96, 97, 99, 100, 101, 112])
@pytest.mark.parametrize("n_rows,n_vals", [(1, 3), (63, 256), (257, 7), (16449, 256), (40009, 60)])
def test_edges(cla, ora, n_cols, n_rows, n_vals):
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols + n_rows)
    specs = columns(synth, rng, n_rows, n_cols, n_vals, np.uint8, 1)
    out, nnz, _ = product(cla, specs, n_rows, n_cols, 2)
    D = ora.np_decompress(specs, n_rows, n_cols)
    assert np.array_equal(out, out.T)
    assert_matches_truth(out, D.T, D, what=f"{n_rows} x {n_cols}")
    assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("width", [8, 40])
@pytest.mark.parametrize("one_kernel", [0, 1])
def test_wide_groups_constants_and_zeros(cla, ora, width, one_kernel):
    """Few wide groups (cells inside a group come from the code counts), columns that only carry a constant, one of zeros, constants added."""
    from systemds_amd import synth
    rng = np.random.default_rng(width)
    n_rows, n_cols = 9001, 84
    specs = columns(synth, rng, n_rows, n_cols - 4, 30, np.uint8, width)
    specs[1].dict[:, 0] = 0.0
    specs.append(synth.GroupSpec("const", np.array([n_cols - 3, n_cols - 1], np.int32), np.array([[2.5, -1.0]])))
    specs.append(synth.GroupSpec("const", np.array([0, 7], np.int32), np.array([[1.5, 0.25]])))
    out, nnz, _ = product(cla, specs, n_rows, n_cols, 2, [("tsmm_one_kernel", one_kernel)])
    D = ora.np_decompress(specs, n_rows, n_cols)
    assert_matches_truth(out, D.T, D, what="constants")
    assert np.array_equal(out, out.T) and nnz == np.count_nonzero(out)


@pytest.mark.parametrize("n_cols,sign", [(20, 1), (35, -1), (100, 1)])
def test_largest_sums(cla, n_cols, sign):
    """Every digit at its largest magnitude in every row, on shares of the rows so long that the sums are joined on the way: n v v is exact
    to rounding (one of the value, the products left out 2^-55 of it: below 4 units in the last place)."""
    from systemds_amd import synth
    n_rows = 5_200_007
    v = sum(sign * (127 if sign > 0 else -128) * 256.0 ** k for k in range(7)) * 2.0 ** -55 if sign > 0 else -sum(128 * 256.0 ** k for k in range(7)) * 2.0 ** -55
    code = np.zeros(n_rows, np.uint8)
    specs = [synth.GroupSpec("ddc", np.array([c], np.int32), np.array([[v], [v / 2]]), code) for c in range(n_cols)]
    out, _, _ = product(cla, specs, n_rows, n_cols, 2)
    assert np.max(np.abs(out / (n_rows * v * v) - 1.0)) < 4 * 2.0 ** -53


def test_whole_numbers_are_exact(cla):
    from systemds_amd import synth
    rng = np.random.default_rng(3)
    n_rows, n_cols = 300_001, 97
    codes = rng.integers(0, 200, (n_cols, n_rows)).astype(np.uint8)
    dicts = rng.integers(-1000, 1000, (n_cols, 200)).astype(np.float64)
    out, nnz, _ = product(cla, [synth.GroupSpec("ddc", np.array([c], np.int32), dicts[c][:, None], codes[c]) for c in range(n_cols)], n_rows, n_cols, 1)
    D = np.stack([dicts[c][codes[c]] for c in range(n_cols)])
    assert np.array_equal(out, D @ D.T) and nnz == np.count_nonzero(out)


@pytest.mark.parametrize("kind", ["far apart", "rare and large", "infinite", "tiny", "one-hot"])
def test_values_that_digits_do_not_suit(cla, ora, kind):
    """Cells whose terms are far below their columns' largest values keep fp64's accuracy: those blocks stay with the fp64 kernel (one-hot
    columns lose nothing to digits and do not)."""
    from systemds_amd import synth
    rng = np.random.default_rng(4)
    n_rows, n_cols = 20_011, 66
    specs = columns(synth, rng, n_rows, n_cols, 40, np.uint8, 1)
    for s in specs:
        if kind == "far apart":
            s.dict[:20, 0] *= 1e-9
            s.codes[:] = np.where(np.arange(n_rows) % n_cols == s.cols[0], 20 + s.codes % 20, s.codes % 20)  # never two large ones in a row
        elif kind == "rare and large":
            s.dict[39, 0] = 1e12
            s.codes[s.codes == 39] = 0
            s.codes[s.cols[0]] = 39
        elif kind == "tiny":
            s.dict *= 1e-200
        elif kind == "one-hot":
            s.dict[:, 0] = np.arange(40) == 3
    if kind == "infinite":
        specs[5].dict[3, 0] = np.inf
    out, _, lds = product(cla, specs, n_rows, n_cols, 2)
    want, _, fp64 = product(cla, specs, n_rows, n_cols, 0)
    assert (lds == fp64) == (kind != "one-hot")
    if kind == "infinite":
        assert np.array_equal(np.isfinite(out), np.isfinite(want))
        return
    D = ora.np_decompress(specs, n_rows, n_cols)
    if kind == "tiny":
        D, out = D * 1e200, out * 1e200 * 1e200  # (products near 1e-400 are zero either way)
        assert np.array_equal(out, want * 1e200 * 1e200)
        return
    assert_matches_truth(out, D.T, D, what=kind)


def on_digits(cla, specs, n_rows, n_cols, digits, options=(), plain=product):
    """product, of the integer kernel: both forms report as k_gram_tiles, their LDS differs."""
    out, nnz, lds = plain(cla, specs, n_rows, n_cols, digits, options)
    assert len(lds) == 1 and lds != plain(cla, specs, n_rows, n_cols, 0, options)[2]
    return out, nnz, lds


@pytest.mark.parametrize("n_cols", [17, 32, 33, 49, 52, 65, 84, 97, 101, 112])
@pytest.mark.parametrize("n_rows,n_vals", [(63, 256), (257, 7), (16449, 256), (40009, 60)])
def test_edges_on_digits(cla, ora, monkeypatch, n_cols, n_rows, n_vals):
    monkeypatch.setitem(globals(), "product", on_digits)
    test_edges(cla, ora, n_cols, n_rows, n_vals)


@pytest.mark.parametrize("n_cols", [17, 31, 32, 33, 48, 49, 50, 52, 53, 64, 65, 68, 80, 81, 82, 84, 85, 96, 97, 99, 100, 101, 112])
def test_one_row_on_digits(cla, ora, n_cols):
    """Values near their columns' largest: the magnitudes' rule takes the block."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols)
    specs = columns(synth, rng, 1, n_cols, 3, np.uint8, 1)
    for spec in specs:
        spec.dict = rng.uniform(0.3, 1.0, spec.dict.shape) * rng.choice([-1.0, 1.0], spec.dict.shape)
    out, nnz, _ = on_digits(cla, specs, 1, n_cols, 2)
    D = ora.np_decompress(specs, 1, n_cols)
    assert np.array_equal(out, out.T) and nnz == np.count_nonzero(out)
    assert_matches_truth(out, D.T, D, what=f"1 x {n_cols}")


@pytest.mark.parametrize("width", [8, 40])
@pytest.mark.parametrize("one_kernel", [0, 1])
def test_wide_groups_on_digits(cla, ora, monkeypatch, width, one_kernel):
    monkeypatch.setitem(globals(), "product", on_digits)
    test_wide_groups_constants_and_zeros(cla, ora, width, one_kernel)


def test_sums_and_whole_numbers_on_digits(cla, monkeypatch):
    monkeypatch.setitem(globals(), "product", on_digits)
    test_largest_sums(cla, 35, -1)
    test_whole_numbers_are_exact(cla)


def errors(specs, out, n_cols):
    """|error| / sum of the terms' magnitudes per cell, against exact counts of pairs of values in long double."""
    err = []
    for i in range(n_cols):
        for j in range(i, n_cols):
            x, y = (specs[c].dict[:, 0].astype(np.longdouble) for c in (i, j))
            count = np.bincount(specs[i].codes.astype(np.int64) * len(y) + specs[j].codes, minlength=len(x) * len(y)).reshape(len(x), len(y))
            terms = x[:, None] * y[None] * count
            err.append(abs(float(out[i, j] - terms.sum())) / float(abs(terms).sum()))
    return np.array(err)


@pytest.mark.parametrize("kind,n_rows,n_cols,n_vals,digits", [
    ("one tuple", 500, 100, 256, False), ("one tuple", 60_011, 100, 40, False), ("one at 5", 10_007, 100, 256, False), ("one at 10", 10_007, 100, 256, False),
    ("three decades", 500, 100, 256, False), ("normal", 2_000, 100, 256, False), ("normal", 600_007, 50, 40, True), ("uniform", 10_007, 60, 40, True)])
def test_no_less_precise_than_fp64(cla, kind, n_rows, n_cols, n_vals, digits):
    """Unasked a block goes to digits only where their error does not exceed the fp64 kernel's, also where the values' magnitudes alone would let
    it in: one tuple with nearly all rows, whose rounding is added again and again, a rare value that takes the others' digits, short blocks."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + n_cols)
    share = np.cumsum(1 / np.arange(1, n_vals + 1) ** 1.1)
    specs = []
    for c in range(n_cols):
        d = rng.standard_normal(n_vals)
        codes = np.searchsorted(share / share[-1], rng.random(n_rows)).clip(max=n_vals - 1)
        if kind == "one tuple":  # 0.135 and 1.1 / 128 of the largest value
            d = rng.permutation([0.135, 1.1 / 128])[0] * (1 + 0.01 * d)
            d[0] = 1.0
            codes = np.where(rng.random(n_rows) < 0.99, 1, np.where(rng.random(n_rows) < 0.5, 0, codes))
        elif kind.startswith("one at"):
            d[200] = float(kind.split()[-1])
        elif kind == "three decades":
            d *= 10 ** rng.uniform(-3, 0, n_vals)
        elif kind == "uniform":
            codes = rng.integers(0, n_vals, n_rows)
        specs.append(synth.GroupSpec("ddc", np.array([c], np.int32), d[:, None], codes.astype(np.uint8)))
    out, _, lds = product(cla, specs, n_rows, n_cols, 1)
    want, _, fp64 = product(cla, specs, n_rows, n_cols, 0)
    assert (lds != fp64) == digits
    if digits:
        got, ref = (errors(specs, o, n_cols) for o in (out, want))
        assert np.sqrt((got ** 2).mean()) <= np.sqrt((ref ** 2).mean()) and got.max() <= ref.max()
