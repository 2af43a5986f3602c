"""Y %*% X on decoded rows, call after call on one block: the workspace that a call leaves at zero for the next one, whatever the rows of Y
were and whether they held a non-finite value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rows", [3001, 70001])
def test_calls_in_a_row(cla, ora, n_rows):
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows)
    runs = np.repeat(rng.integers(0, 9, n_rows // 50 + 1), 50)[:n_rows]
    ptr, data = synth.encode_rle(runs, 9)
    specs = [synth.GroupSpec("rle", np.array([0], np.int32), rng.standard_normal((9, 1)), ptr=ptr, rle=data),
             synth.GroupSpec("ddc", np.array([1, 3], np.int32), rng.standard_normal((500, 2)), rng.integers(0, 500, n_rows).astype(np.uint16)),
             synth.sdc_group(rng, n_rows, [2], 16, 0.1, 1.0),
             synth.GroupSpec("unc", np.array([4], np.int32), dense=rng.standard_normal((n_rows, 1)))]
    D = ora.np_decompress(specs, n_rows, 5)
    blk = cla.build_block(n_rows, 5, specs)
    for p, bad in ((3, None), (16, np.inf), (3, None), (40, None), (1, np.nan), (2, -np.inf), (40, np.inf), (7, None)):
        Y = rng.standard_normal((p, n_rows))
        if bad is not None:
            Y[p // 2, 11] = bad
        out, nnz = blk.lmm(Y)
        fresh = cla.build_block(n_rows, 5, specs)
        want, want_nnz = fresh.lmm(Y)
        fresh.close()
        finite = np.isfinite(want)
        assert np.array_equal(finite, np.isfinite(out)) and np.array_equal(np.isnan(want), np.isnan(out)) and nnz == want_nnz
        # two orders of fp64 additions: fewer than 300 roundings in either
        scale = np.abs(np.where(np.isfinite(Y), Y, 0.0)) @ np.abs(D)
        assert np.all((np.abs(out - want) <= 600 * 2.0 ** -53 * scale) | ~finite), (p, bad)
    blk.close()


@pytest.mark.parametrize("p,bad_p,at", [(5, 2, 42), (7, 3, 63), (16, 4, 84)])
def test_a_zero_row_behind_a_non_finite_one(cla, p, bad_p, at):
    """Only dictionary and dense columns, whose sums a non-finite Y leaves as they are: the report of one (word `at` of the workspace, a cell
    of a later call's sums) must not outlive its call. A row of zeros in Y gives a row of zeros, not the smallest number there is."""
    from systemds_amd import synth
    rng = np.random.default_rng(p)
    n_rows, n_cols = 4001, 10
    assert at == bad_p * (2 * n_cols + 1) and at < p * n_cols
    specs = [synth.GroupSpec("ddc", np.array([c, c + 1], np.int32), rng.standard_normal((400, 2)), rng.integers(0, 400, n_rows).astype(np.uint16))
             for c in range(0, 8, 2)] + [synth.GroupSpec("unc", np.array([8, 9], np.int32), dense=rng.standard_normal((n_rows, 2)))]
    blk = cla.build_block(n_rows, n_cols, specs)
    Y = rng.standard_normal((p, n_rows))
    Y[at // n_cols] = 0.0
    want, want_nnz = blk.lmm(Y)
    assert "k_take_block" in [k["name"] for k in blk.stats()["kernels"]]
    bad = rng.standard_normal((bad_p, n_rows))
    bad[0, 17] = np.nan
    blk.lmm(bad)
    out, nnz = blk.lmm(Y)
    blk.close()
    assert not out[at // n_cols].any() and nnz == want_nnz == (p - 1) * n_cols, (nnz, out[at // n_cols])
