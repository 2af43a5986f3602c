"""t(X) %*% X of blocks of two to six column pairs with two-byte codes on k_gram_tiles: tile edges, dictionaries of every size, and blocks that
go by pairs of groups (many rows, by option), against the oracle."""
import numpy as np
import pytest

from parity import assert_matches_truth
from test_gpu_gram_tiles import columns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_cols", [4, 6, 8, 10, 12])
@pytest.mark.parametrize("n_rows,n_vals", [(1, 3), (255, 300), (257, 1500), (2049, 5000), (70001, 9000), (140003, 20000)])
@pytest.mark.parametrize("one_kernel", [0, 1])
def test_few_pairs(cla, ora, n_cols, n_rows, n_vals, one_kernel):
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols + n_rows)
    specs = columns(synth, rng, n_rows, n_cols, n_vals, np.uint16, 2)
    if n_rows == 257:  # a constant beside the dictionaries
        specs.append(synth.GroupSpec("const", np.array([1, n_cols - 1], np.int32), np.array([[1.5, -0.25]])))
    blk = cla.build_block(n_rows, n_cols, specs)
    blk.set_option("tsmm_one_kernel", one_kernel)
    out, nnz = blk.tsmm()
    names = [k["name"] for k in blk.stats()["kernels"]]
    again, _ = blk.tsmm()
    blk.set_option("tsmm_route", 1)
    pairs, _ = blk.tsmm()
    blk.close()
    D = ora.np_decompress(specs, n_rows, n_cols)
    assert not any("pair" in n or "decode" in n for n in names), names
    for got in (out, again, pairs):
        assert_matches_truth(got, D.T, D, what=f"{n_rows} x {n_cols} of {n_vals}")
        assert np.array_equal(got, got.T)
    assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("n_rows,by_pairs", [(2_500_000, False), (2_500_001, True)])
def test_many_rows_go_by_pairs_of_groups(cla, ora, n_rows, by_pairs):
    """Two or three groups go by pairs of groups from there on (shorter chains of additions)."""
    from systemds_amd import synth
    rng = np.random.default_rng(1)
    n_cols = 6
    specs = columns(synth, rng, n_rows, n_cols, 300, np.uint16, 2)
    blk = cla.build_block(n_rows, n_cols, specs)
    out, nnz = blk.tsmm()
    names = [k["name"] for k in blk.stats()["kernels"]]
    blk.close()
    assert ("k_gram_tiles" not in names) == by_pairs, names
    D = ora.np_decompress(specs, n_rows, n_cols)
    assert_matches_truth(out, D.T, D, what=str(names))
    assert np.array_equal(out, out.T) and nnz == np.count_nonzero(out)
