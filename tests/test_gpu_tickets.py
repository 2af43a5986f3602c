"""The last block of a call writes its output or counts its non-zeros: products of one block in turn whose numbers of blocks lie on
both sides of every rule (tickets on one line or on eight, sums in one accumulator or in one per XCD, added by the last block or by the
last of each XCD), each finding what the one in front has left."""
import numpy as np
import pytest

from parity import assert_fp64_close, assert_matches_truth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rows", [70, 20011, 150001])
@pytest.mark.parametrize("n_cols", [3, 44, 45, 46, 100])  # (2 x 512 cells of the upper triangle lie between 44 and 45 columns)
def test_products_in_turn(cla, ora, n_rows, n_cols):
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + n_cols)
    specs = [synth.GroupSpec("ddc", np.array([c], np.int32), rng.standard_normal((9, 1)), rng.integers(0, 9, n_rows).astype(np.uint8)) for c in range(n_cols)]
    blk = cla.build_block(n_rows, n_cols, specs)
    D = ora.np_decompress(specs, n_rows, n_cols)
    gram, scale = D.T @ D, ora.abs_matmul(D.T, D)
    v = rng.standard_normal((n_cols, 1))
    for p in (1, 16, 17, 33, 48, 2, 64):  # (16 rows of Y per layer of blocks)
        Y = rng.standard_normal((p, n_rows))
        out, nnz = blk.lmm(Y)
        assert_matches_truth(out, Y, D, what=f"{p} rows of Y")
        assert nnz == np.count_nonzero(out)
        out, nnz = blk.tsmm()
        assert_fp64_close(out, gram, scale, what="gram", n_terms=n_rows)
        assert nnz == np.count_nonzero(out) and np.array_equal(out, out.T)
        out, nnz = blk.mmchain(v)
        assert_matches_truth(out.reshape(-1, 1), D.T, D @ v, what="chain")
        assert nnz == np.count_nonzero(out)
    blk.close()


@pytest.mark.parametrize("n_rows", [5000, 200003])
def test_offset_lists_in_turn(cla, ora, n_rows):
    from test_gpu_sdc_matvec import sdc_block
    rng = np.random.default_rng(n_rows)
    specs, n_cols = sdc_block(3, n_rows, 30, 0.05, 20)
    blk = cla.build_block(n_rows, n_cols, specs)
    D = ora.np_decompress(specs, n_rows, n_cols)
    for p in (1, 3, 16, 2, 40, 1):
        Y = rng.standard_normal((p, n_rows))
        out, nnz = blk.lmm(Y)
        assert_matches_truth(out, Y, D, what=f"{p} rows of Y")
        assert nnz == np.count_nonzero(out)
    blk.close()


@pytest.mark.parametrize("n_cols", [6, 16, 24, 50])  # (one slab of groups, two, three, seven)
@pytest.mark.parametrize("n_rows", [5000, 150001])
def test_column_pairs_in_turn(cla, ora, n_rows, n_cols):
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + n_cols)
    specs = [synth.GroupSpec("ddc", np.array([c, c + 1], np.int32), rng.standard_normal((1000, 2)), rng.integers(0, 1000, n_rows).astype(np.uint16))
             for c in range(0, n_cols, 2)]
    blk = cla.build_block(n_rows, n_cols, specs)
    D = ora.np_decompress(specs, n_rows, n_cols)
    v = rng.standard_normal((n_cols, 1))
    for k in range(4):
        Y = rng.standard_normal((1, n_rows))
        out, nnz = blk.lmm(Y)
        assert_matches_truth(out, Y, D, what="a row of Y")
        assert nnz == np.count_nonzero(out)
        out, nnz = blk.mmchain(v)
        assert_matches_truth(out.reshape(-1, 1), D.T, D @ v, what="chain")
        assert nnz == np.count_nonzero(out)
    blk.close()
