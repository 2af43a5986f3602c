"""Y %*% X with infinities and NaN in Y on the blocks that the kernels on decoded rows serve: a row that a group does not cover stays
out of its sums, as in the bin kernels and the oracle, without the host's look at Y."""
import numpy as np
import pytest

from conftest import mixed_block
from parity import assert_fp64_close
from test_gpu_lmm_direct import block

pytestmark = pytest.mark.gpu


def blocks(kind, n_rows):
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows)
    if kind == "mixed":
        return mixed_block(13, n_rows, with_unc=True, big_dict=False)
    if kind == "mixed, no constants":
        return mixed_block(4, n_rows, with_unc=True, with_const=False, big_dict=False)
    if kind == "constants":  # under a dictionary column, a dense one and a run-length one, and on columns that no other group covers
        specs, n_cols = block(synth, rng, n_rows, 2, 2, 1, 1, 2)
        cols = np.array([next(s for s in specs if s.type == t).cols[0] for t in ("ddc", "unc", "rle")] + [n_cols, n_cols + 1], np.int32)
        return specs + [synth.GroupSpec("const", cols, np.array([[-0.75, 1.5, 2.0, 0.0, -3.0]]))], n_cols + 2
    if kind == "short runs":
        return block(synth, rng, n_rows, 8, 1, 0, 0, 0, mean_run=7)
    if kind == "wide groups":
        specs, n_cols = block(synth, rng, n_rows, 1, 0, 1, 1, 0)
        specs.append(synth.GroupSpec("ddc", np.arange(n_cols, n_cols + 7, dtype=np.int32), rng.standard_normal((300, 7)), rng.integers(0, 300, n_rows).astype(np.uint16)))
        codes = np.repeat(rng.integers(-1, 5, n_rows // 9 + 1), 9)[:n_rows]
        ptr, rle = synth.encode_rle(codes, 5)
        specs.append(synth.GroupSpec("rle", np.arange(n_cols + 7, n_cols + 10, dtype=np.int32), rng.standard_normal((5, 3)), ptr=ptr, rle=rle))
        return specs, n_cols + 10
    return block(synth, rng, n_rows, *{"runs": (8, 4, 2, 1, 2), "streams": (0, 5, 3, 0, 0), "dense": (2, 0, 1, 1, 4)}[kind])


@pytest.mark.parametrize("kind", ["mixed", "mixed, no constants", "runs", "streams", "dense", "constants", "short runs", "wide groups"])
@pytest.mark.parametrize("n_rows,p", [(1, 1), (257, 3), (1025, 17), (40001, 2), (40001, 9), (300007, 70)])
@pytest.mark.parametrize("direct", [1, 0])
def test_non_finite_y(cla, ora, kind, n_rows, p, direct):
    specs, n_cols = blocks(kind, n_rows)
    rng = np.random.default_rng(p)
    Y = rng.standard_normal((p, n_rows))
    clean = Y.copy()
    for i in range(0, p, 2):  # (every other row of Y stays finite)
        for r in rng.integers(0, n_rows, 3):
            Y[i, r] = rng.choice([np.inf, -np.inf, np.nan])
    blk = cla.build_block(n_rows, n_cols, specs).set_option("tsmm_direct", direct)
    first, nnz0 = blk.lmm(clean)
    finite = [k["name"] for k in blk.stats()["kernels"]]
    out, nnz = blk.lmm(Y)
    ran = [k["name"] for k in blk.stats()["kernels"]]
    again, nnz2 = blk.lmm(clean)  # (nothing of the call in front is left)
    bins, _ = blk.set_option("lmm_joint", 0).lmm(Y)
    blk.close()
    assert ran == finite and (n_rows < 1025 or ran[-1] == "k_take_block"), (finite, ran)
    fin = np.isfinite(bins)
    assert np.array_equal(np.isfinite(out), fin) and np.array_equal(out[~fin], bins[~fin], equal_nan=True)
    assert nnz == np.count_nonzero(out) and nnz0 == np.count_nonzero(first) and nnz2 == np.count_nonzero(again)
    D = ora.np_decompress(specs, n_rows, n_cols)
    scale = ora.abs_matmul(np.nan_to_num(Y, nan=0.0, posinf=0.0, neginf=0.0), D)
    assert_fp64_close(out[fin], bins[fin], scale[fin], what=f"{kind}, finite cells", n_terms=n_rows)
    assert_fp64_close(again, first, ora.abs_matmul(clean, D), what=f"{kind}, finite Y", n_terms=n_rows)
    if n_rows < 100000 and p < 10:
        ref, _ = ora.lmm(ora.Groups(specs, n_rows, n_cols), Y, 4)
        assert np.array_equal(out[~fin], ref[~fin], equal_nan=True) and np.array_equal(np.isfinite(ref), fin)
