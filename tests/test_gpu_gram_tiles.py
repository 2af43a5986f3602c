"""t(X) %*% X of all-DDC blocks on k_gram_tiles: the edges of its tiles (rows and columns), its three ways of decoding,
dictionaries beside the tiles and behind them, constants added to the columns."""
import numpy as np
import pytest

from parity import assert_matches_truth

pytestmark = pytest.mark.gpu


def check(cla, ora, specs, n_rows, n_cols, what, options=()):
    blk = cla.build_block(n_rows, n_cols, specs)
    for key, value in options:
        blk.set_option(key, value)
    out, nnz = blk.tsmm()
    names = {k["name"] for k in blk.stats()["kernels"]}
    blk.close()
    assert names - {"k_tsmm_self"} == {"k_gram_tiles"}, names  # (few wide groups: cells inside a group from the code counts)
    D = ora.np_decompress(specs, n_rows, n_cols)
    assert np.array_equal(out, out.T)
    assert_matches_truth(out, D.T, D, what=what)
    assert nnz == np.count_nonzero(out)


def columns(synth, rng, n_rows, n_cols, n_vals, dtype, width):
    order = rng.permutation(n_cols).astype(np.int32)
    return [synth.GroupSpec("ddc", order[c:c + width], rng.standard_normal((n_vals, len(order[c:c + width]))),
                            rng.integers(0, n_vals, n_rows).astype(dtype)) for c in range(0, n_cols, width)]


@pytest.mark.parametrize("n_cols", [13, 16, 17, 20, 24, 25, 33, 40, 48, 52, 64, 65, 68, 72, 73, 80, 81, 88, 96, 97, 100, 112, 113, 120, 127, 128])
@pytest.mark.parametrize("n_rows", [1, 31, 33, 8191, 40009])
def test_byte_codes(cla, ora, n_cols, n_rows):
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols + n_rows)
    check(cla, ora, columns(synth, rng, n_rows, n_cols, 200, np.uint8, 1), n_rows, n_cols, f"{n_rows} x {n_cols}, bytes")


@pytest.mark.parametrize("n_cols", [14, 16, 18, 20, 24, 26, 32, 34, 40, 42, 48, 50, 64, 66, 70, 74, 82, 90, 98, 106, 114, 128])
@pytest.mark.parametrize("n_rows,n_vals", [(1, 300), (65, 4096), (16387, 2500)])
def test_column_pairs(cla, ora, n_cols, n_rows, n_vals):
    """Groups of two columns, two-byte codes: one group per instruction, whole tuples (every number of units that a wave can miss)."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols + n_rows)
    specs = columns(synth, rng, n_rows, n_cols, n_vals, np.uint16, 2)
    check(cla, ora, specs, n_rows, n_cols, f"{n_rows} x {n_cols}, pairs", [("tsmm_route", 2)])  # (few groups: decoded all the same)


@pytest.mark.parametrize("n_cols,width,n_vals", [(66, 1, 300), (99, 3, 1000), (101, 2, 4096), (128, 1, 260)])
def test_two_byte_codes(cla, ora, n_cols, width, n_vals):
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols)
    check(cla, ora, columns(synth, rng, 12345, n_cols, n_vals, np.uint16, width), 12345, n_cols, f"{n_cols} columns, width {width}")


@pytest.mark.parametrize("dtype,width,n_vals", [(np.uint8, 1, 17), (np.uint16, 2, 700)])
def test_constant_columns_and_offsets(cla, ora, dtype, width, n_vals):
    """Columns that only carry a constant, and a constant added to decoded columns: the dictionaries are copied with it."""
    from systemds_amd import synth
    rng = np.random.default_rng(5)
    n_rows, n_cols = 9001, 70
    specs = columns(synth, rng, n_rows, n_cols - 2, n_vals, dtype, width)
    specs.append(synth.GroupSpec("const", np.array([n_cols - 2, n_cols - 1], np.int32), np.array([[2.5, -1.0]])))
    specs.append(synth.GroupSpec("const", np.array([0, 7], np.int32), np.array([[1.5, 0.25]])))
    check(cla, ora, specs, n_rows, n_cols, "constants")


def test_infinities_and_nan_stay_in_their_cells(cla, ora):
    from systemds_amd import synth
    rng = np.random.default_rng(6)
    n_rows, n_cols = 5003, 68
    specs = columns(synth, rng, n_rows, n_cols, 300, np.uint16, 2)
    specs[3].dict[5, 0] = np.inf
    specs[9].dict[7, 1] = np.nan
    blk = cla.build_block(n_rows, n_cols, specs)
    out, _ = blk.tsmm()
    blk.close()
    D = ora.np_decompress(specs, n_rows, n_cols)
    with np.errstate(invalid="ignore"):
        want = D.T @ D
    ok = np.isfinite(want)
    assert np.array_equal(np.isfinite(out), ok)
    assert np.allclose(out[ok], want[ok], rtol=0, atol=1e-11 * n_rows)  # n_rows terms of size about 1, eps 1.1e-16


@pytest.mark.parametrize("n_cols,width,n_vals,dtype,bound", [(20, 1, 7, np.uint8, 1.0e-14), (44, 1, 7, np.uint8, 1.0e-14), (112, 1, 7, np.uint8, 1.7e-14),
                                                          (20, 2, 300, np.uint16, 3.5e-15)])
def test_sums_of_like_terms(cla, n_cols, width, n_vals, dtype, bound):
    """Diagonal cells of few distinct positive values, against the exact sum of counts times products: a chain of additions of like
    terms drifts with its length, so the waves' chains must stay short. The bounds on the rms relative error are about 1.4 times what
    4096 chains leave (112 columns: 2048); half as many leave 1.7 - 2 times as much."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols)
    n_rows = 4_000_000
    p = 1.0 / np.arange(1, n_vals + 1)
    specs, exact = [], np.zeros(n_cols)
    for c in range(0, n_cols, width):
        codes = np.searchsorted(np.cumsum(p / p.sum()), rng.random(n_rows), side="right").clip(max=n_vals - 1).astype(dtype)
        d = rng.random((n_vals, width)) + 0.1
        specs.append(synth.GroupSpec("ddc", np.arange(c, c + width, dtype=np.int32), d, codes))
        n = np.bincount(codes, minlength=n_vals).astype(np.longdouble)
        exact[c:c + width] = (n[:, None] * d.astype(np.longdouble) ** 2).sum(0)
    blk = cla.build_block(n_rows, n_cols, specs)
    out, _ = blk.tsmm()
    names = {k["name"] for k in blk.stats()["kernels"]}
    blk.close()
    assert names - {"k_tsmm_self"} == {"k_gram_tiles"}, names  # (few wide groups: cells inside a group from the code counts)
    rel = np.diag(out) / exact - 1.0
    assert np.sqrt((rel ** 2).mean()) < bound, np.sqrt((rel ** 2).mean())


@pytest.mark.parametrize("n_rows,n_cols,n_vals,kernel", [
    (150_000, 13, 900, "k_gram_tiles"), (150_001, 13, 900, "k_tsmm_decode"), (400_001, 16, 890, "k_tsmm_decode"),  # dictionaries in LDS there
    (400_001, 16, 700, "k_gram_tiles"),                                                                          # ... and here
    (60_000, 16, 3000, "k_gram_tiles"), (60_001, 16, 3000, "k_tsmm_decode"), (250_001, 14, 3000, "k_gram_tiles"),  # in global memory
    (60_001, 13, 61000, "k_tsmm_decode"), (90_001, 17, 50000, "k_gram_tiles"), (150_001, 17, 50000, "k_tsmm_decode"),  # past the L2
    (250_001, 17, 50000, "k_gram_tiles"), (500_001, 17, 50000, "k_tsmm_decode")])
def test_two_byte_codes_where_the_older_kernel_is_faster(cla, n_rows, n_cols, n_vals, kernel):
    """The rule that leaves two-byte blocks to k_tsmm_decode, at its lines; t(X) %*% X against exact integers (dictionaries of
    whole numbers, whose products and sums stay below 2^53)."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + n_cols)
    codes = rng.integers(0, n_vals, (n_cols, n_rows)).astype(np.uint16)
    dicts = rng.integers(-1000, 1000, (n_cols, n_vals)).astype(np.float64)
    blk = cla.build_block(n_rows, n_cols, [synth.GroupSpec("ddc", np.array([c], np.int32), dicts[c][:, None], codes[c]) for c in range(n_cols)])
    out, nnz = blk.tsmm()
    names = [k["name"] for k in blk.stats()["kernels"]]
    blk.close()
    assert names == [kernel], names
    D = np.stack([dicts[c][codes[c]] for c in range(n_cols)])
    assert np.array_equal(out, D @ D.T) and nnz == np.count_nonzero(out)


@pytest.mark.parametrize("n_cols", [17, 24, 33, 48, 52, 65, 72, 81, 97, 112])
@pytest.mark.parametrize("n_rows", [1, 31, 33, 8191, 40009])
def test_byte_codes_in_fp64(cla, ora, n_cols, n_rows):
    """The integer kernel, which reports under the same name, takes some of these unasked."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols + n_rows)
    specs = columns(synth, rng, n_rows, n_cols - 2, 200, np.uint8, 1)
    specs.append(synth.GroupSpec("const", np.array([n_cols - 2, n_cols - 1], np.int32), np.array([[2.5, -1.0]])))
    specs.append(synth.GroupSpec("const", np.array([0, 7], np.int32), np.array([[1.5, 0.25]])))
    check(cla, ora, specs, n_rows, n_cols, f"{n_rows} x {n_cols}, bytes", [("tsmm_digits", 0)])
