"""Y %*% X on k_lmm_direct (a few streamed columns next to run-length columns): every number of rows of Y per pass and of code
and dense columns it is filled up to, row counts at the edges of its steps, run ends at every place of a step."""
import numpy as np
import pytest

from parity import assert_matches_truth

pytestmark = pytest.mark.gpu


def block(synth, rng, n_rows, n_rle, n_short, n_byte, n_sdc, n_dense, mean_run=400):
    order = list(rng.permutation(n_rle + n_short + n_byte + n_sdc + n_dense).astype(np.int32))
    specs = []
    for _ in range(n_rle):
        starts = np.flatnonzero(rng.random(n_rows) < 1.0 / mean_run)
        codes = np.repeat(rng.integers(-1, 32, len(starts) + 1), np.diff(np.concatenate(([0], starts, [n_rows]))))  # -1: rows that no run covers
        ptr, rle = synth.encode_rle(codes, 32)
        specs.append(synth.GroupSpec("rle", np.array([order.pop()], np.int32), rng.standard_normal((32, 1)), ptr=ptr, rle=rle))
    for k in range(n_short + n_byte):
        v, t = (700, np.uint16) if k < n_short else (9, np.uint8)
        specs.append(synth.GroupSpec("ddc", np.array([order.pop()], np.int32), rng.standard_normal((v, 1)), rng.integers(0, v, n_rows).astype(t)))
    for _ in range(n_sdc):
        rows = np.flatnonzero(rng.random(n_rows) < 0.1)
        rows = rows if len(rows) else np.array([0])
        deltas, first, last, n = synth.encode_offsets(rows)
        specs.append(synth.GroupSpec("sdc", np.array([order.pop()], np.int32), rng.standard_normal((16, 1)), rng.integers(0, 16, n).astype(np.uint8),
                                     np.array([1.0]), deltas, first, last, n))
    if n_dense:
        specs.append(synth.GroupSpec("unc", np.sort(np.array(order, np.int32)), dense=rng.standard_normal((n_rows, n_dense))))
    return specs, n_rle + n_short + n_byte + n_sdc + n_dense


def shape_of(specs):
    """Code columns and dense ones of a block whose run-length columns are followed by run."""
    return sum(s.type in ("ddc", "sdc") for s in specs), sum(len(s.cols) for s in specs if s.type == "unc")


def passes(p, n_code, n_dense):
    """Launches of k_lmm_direct for p <= 16 rows of Y: 8 rows each while at most 8 columns are streamed, else 6 (code columns are
    filled up to 4, 8, 10 or 12, dense ones to 2 or 4)."""
    nd = 0 if n_dense == 0 else 2 if n_dense <= 2 else 4
    nc = 4 if n_code <= 4 else 8 if n_code <= 8 else 10 if n_code <= 10 and nd == 2 else 12
    return -(-p // (6 if nc + nd > 8 else 8))


def kernels(p, n_rows, n_code, n_dense):
    """What serves p rows of Y, 16 at a time: several passes only on many rows, else the tile kernel takes the 16 at once."""
    out = []
    for p0 in range(0, p, 16):
        k = passes(min(16, p - p0), n_code, n_dense)
        out += ["k_lmm_direct"] * k if k == 1 or n_rows > 500000 * (k - 1) else ["k_lmm_decode"]
    return out


def check(cla, ora, specs, n_cols, n_rows, p, what, rng, expect=None):
    Y = rng.standard_normal((p, n_rows))
    blk = cla.build_block(n_rows, n_cols, specs)
    out, nnz = blk.lmm(Y)
    ran = [k["name"] for k in blk.stats()["kernels"]]
    tile, _ = blk.set_option("tsmm_direct", 0).lmm(Y)
    only = {k["name"] for k in blk.stats()["kernels"]}
    blk.close()
    assert "k_lmm_direct" not in only, only
    assert ran == (expect if expect else kernels(p, n_rows, *shape_of(specs))) + ["k_take_block"], ran
    D = ora.np_decompress(specs, n_rows, n_cols)
    assert_matches_truth(out, Y, D, what=what)
    assert_matches_truth(tile, Y, D, what=what + ", tile kernel")
    assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("shape", [(8, 8, 0, 2, 2), (2, 2, 0, 1, 1), (0, 3, 2, 0, 0), (5, 4, 3, 1, 0), (1, 0, 1, 2, 4), (8, 6, 4, 2, 0), (3, 5, 1, 2, 3), (2, 8, 0, 0, 0), (1, 3, 1, 0, 2)])
@pytest.mark.parametrize("p", [1, 2, 3, 4, 5, 6, 7, 8, 11, 16, 17])
def test_shapes(cla, ora, shape, p):
    from systemds_amd import synth
    rng = np.random.default_rng(p)
    n_rows = 70003
    specs, n_cols = block(synth, rng, n_rows, *shape)
    check(cla, ora, specs, n_cols, n_rows, p, f"{shape}, {p} rows", rng)


@pytest.mark.parametrize("shape", [(0, 1, 0, 0, 3), (3, 1, 0, 0, 3), (8, 0, 1, 0, 3), (2, 0, 1, 0, 4), (0, 3, 0, 0, 4), (2, 0, 0, 1, 3)])
@pytest.mark.parametrize("n_rows,p", [(129, 1), (1030, 4), (70003, 8), (300001, 3)])
def test_more_dense_columns_than_columns_behind_codes(cla, ora, shape, n_rows, p):
    """One code column next to three dense ones: more dense values than the Gram kernel stages per unit of rows, which is no limit here."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + p)
    specs, n_cols = block(synth, rng, n_rows, *shape)
    check(cla, ora, specs, n_cols, n_rows, p, f"{shape}, {p} rows", rng)


@pytest.mark.parametrize("p,mean_run,kernel", [(6, 8, "k_lmm_decode"), (6, 40, "k_lmm_decode"), (6, 60, "k_lmm_direct"), (1, 8, "k_lmm_decode")])
def test_many_short_runs_take_the_tile_kernel(cla, ora, p, mean_run, kernel):
    """Eight run-length columns of short runs next to too few other bytes for one-code-per-row copies: a run end for every row
    or two is what the tile kernel does better (run ends are counted once per column, so 8 of mean run 48 lie at the rule's edge)."""
    from systemds_amd import synth
    rng = np.random.default_rng(mean_run)
    n_rows = 100003
    specs, n_cols = block(synth, rng, n_rows, 8, 0, 2, 0, 0, mean_run)
    check(cla, ora, specs, n_cols, n_rows, p, f"runs of {mean_run}", rng, [kernel])


@pytest.mark.parametrize("n_rows,p", [(500003, 7), (500003, 11), (1000003, 13), (1000003, 16), (500001, 8)])
@pytest.mark.parametrize("shape", [(2, 4, 0, 4, 1), (1, 2, 1, 1, 2)])
def test_passes_over_many_rows(cla, ora, n_rows, p, shape):
    """More rows of Y than a pass takes, on row counts where the passes are taken (and where they just are not)."""
    from systemds_amd import synth
    rng = np.random.default_rng(p)
    specs, n_cols = block(synth, rng, n_rows, *shape)
    check(cla, ora, specs, n_cols, n_rows, p, f"{shape}, {n_rows} rows, {p} of Y", rng)


@pytest.mark.parametrize("n_rows", [1, 2, 3, 63, 64, 127, 128, 129, 131, 255, 1030, 16383, 16384, 40005])
@pytest.mark.parametrize("p,mean_run", [(3, 400), (6, 70), (8, 30)])
def test_row_edges(cla, ora, n_rows, p, mean_run):
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows)
    specs, n_cols = block(synth, rng, n_rows, 4, 3, 2, 1, 2, mean_run)
    check(cla, ora, specs, n_cols, n_rows, p, f"{n_rows} rows", rng)


@pytest.mark.parametrize("n_rows", [63, 65, 129, 70003])
@pytest.mark.parametrize("p", [1, 6, 8])
def test_infinities_in_the_last_row(cla, ora, n_rows, p):
    """An infinity in the last row of a dense column and an infinite constant under a dictionary column reach their own column as
    they do row by row: the rows that fill up the last step do not multiply them by zero."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + p)
    specs, n_cols = block(synth, rng, n_rows, 2, 2, 1, 1, 2)
    specs[-1].dense[-1, 0], specs[-1].dense[-1, 1] = np.inf, -np.inf
    Y = rng.random((p, n_rows)) + 0.5
    D = ora.np_decompress(specs, n_rows, n_cols)
    blk = cla.build_block(n_rows, n_cols, specs)
    out, nnz = blk.lmm(Y)
    blk.close()
    dense = specs[-1].cols
    assert np.all(out[:, dense[0]] == np.inf) and np.all(out[:, dense[1]] == -np.inf)
    rest = np.setdiff1d(np.arange(n_cols), dense)
    assert_matches_truth(out[:, rest], Y, D[:, rest], what=f"{n_rows} rows")
    assert nnz == np.count_nonzero(out)

    specs, n_cols = block(synth, rng, n_rows, 0, 3, 1, 0, 0)
    specs.append(synth.GroupSpec("const", np.array([specs[0].cols[0]], np.int32), np.array([[np.inf]])))
    D = ora.np_decompress(specs[:-1], n_rows, n_cols)
    blk = cla.build_block(n_rows, n_cols, specs)
    out, _ = blk.lmm(Y)
    blk.close()
    rest = np.setdiff1d(np.arange(n_cols), specs[0].cols)
    assert np.all(out[:, specs[0].cols] == np.inf)
    assert_matches_truth(out[:, rest], Y, D[:, rest], what=f"{n_rows} rows, constant")


@pytest.mark.parametrize("big", [1e14, 1e200, -1e290])
@pytest.mark.parametrize("p,mean_run", [(1, 3000), (4, 400), (6, 90)])
def test_large_values_where_a_run_length_column_is_zero(cla, ora, big, p, mean_run):
    """Y may be of any size on rows that no run covers or whose value is zero: such rows leave no trace in the column's sums
    (each cell within 1e-12 of |Y| %*% |X|, to which they add nothing)."""
    from systemds_amd import synth
    rng = np.random.default_rng(p)
    n_rows = 40005
    specs, n_cols = block(synth, rng, n_rows, 5, 3, 1, 1, 1, mean_run)
    row = np.arange(n_rows)
    specs[0].ptr, specs[0].rle = synth.encode_rle(np.where(row < 5000, -1, 3), 32)         # one run behind rows that none covers
    specs[1].ptr, specs[1].rle = synth.encode_rle(np.where(row // 137 % 2 == 0, 2, 3), 32)  # every other run is of zeros
    specs[1].dict[2] = 0.0
    Y = rng.standard_normal((p, n_rows))
    D = ora.np_decompress(specs, n_rows, n_cols)
    zero = np.flatnonzero((D[:, specs[0].cols[0]] == 0.0) & (D[:, specs[1].cols[0]] == 0.0))
    Y[:, [0, 17, zero[-1]] + list(rng.choice(zero, 5))] = big
    blk = cla.build_block(n_rows, n_cols, specs)
    out, nnz = blk.lmm(Y)
    blk.close()
    for c in range(n_cols):  # (a column at a time: the largest output of one is no scale for another)
        assert_matches_truth(out[:, c:c + 1], Y, D[:, c:c + 1], what=f"column {c}, y of {big}")
    assert nnz == np.count_nonzero(out)
