"""X %*% v and t(y) %*% X of DDC blocks with two-byte codes and large dictionaries (k_rmm_q1_short, k_lmm_q1_short): the
edges of their units and slabs, against exact sums; X %*% v bit for bit against the oracle, which adds in the same order."""
import numpy as np
import pytest

from parity import assert_matches_truth

pytestmark = pytest.mark.gpu


def block(synth, rng, n_rows, n_groups, width, n_vals):
    order = rng.permutation(n_groups * width).astype(np.int32)
    specs = []
    for g in range(n_groups):
        v = n_vals - (g % 3)  # dictionaries of odd sizes: the next one starts at any multiple of 8 bytes
        specs.append(synth.GroupSpec("ddc", order[g * width:(g + 1) * width], rng.standard_normal((v, width)),
                                     rng.integers(0, v, n_rows).astype(np.uint16)))
        specs[-1].codes[-1] = v - 1
    return specs


@pytest.mark.parametrize("n_rows", [1, 3, 257, 70002, 400001, 1100003])
@pytest.mark.parametrize("n_groups,width,n_vals,const", [(1, 2, 4096, False), (2, 1, 4097, True), (7, 2, 4096, True), (13, 1, 3001, False),
                                                        (5, 2, 8192, False), (3, 1, 8192, True), (14, 1, 300, False)])
def test_vector_products(cla, ora, n_rows, n_groups, width, n_vals, const):
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + n_vals)
    n_cols = n_groups * width
    specs = block(synth, rng, n_rows, n_groups, width, n_vals)
    if const:
        specs.append(synth.GroupSpec("const", np.array([n_cols], np.int32), np.array([[1.25]])))
        n_cols += 1
    v, y = rng.standard_normal((n_cols, 1)), rng.standard_normal((1, n_rows))
    blk = cla.build_block(n_rows, n_cols, specs)
    out, nnz = blk.rmm(v)
    assert [k["name"] for k in blk.stats()["kernels"]][-1] == ("k_rmm_q1_short" if n_rows > 400000 else "k_rmm_q1_short_rows")
    left, lnnz = blk.lmm(y)
    ran = {k["name"] for k in blk.stats()["kernels"]}
    blk.close()
    if n_vals * width * 8 < 150 * 1024:
        assert "k_lmm_q1_short" in ran, ran
    ref, rnnz = ora.rmm(ora.Groups(specs, n_rows, n_cols), v, 1)
    assert np.array_equal(out, ref) and nnz == rnnz
    D = ora.np_decompress(specs, n_rows, n_cols)
    assert_matches_truth(left, y, D, what="t(y) %*% X")
    assert lnnz == np.count_nonzero(left)


def test_non_finite_vector(cla, ora):
    """An infinite and a NaN entry of y reach the columns, and only those cells are non-finite that the rows make so."""
    from systemds_amd import synth
    rng = np.random.default_rng(3)
    n_rows = 3000
    specs = block(synth, rng, n_rows, 3, 2, 4096)
    blk = cla.build_block(n_rows, 6, specs)
    y = rng.standard_normal((1, n_rows))
    y[0, n_rows - 1] = np.inf
    D = ora.np_decompress(specs, n_rows, 6)
    out, _ = blk.lmm(y)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(out, np.where(D[-1] > 0, np.inf, -np.inf)[None, :])
    y[0, 5] = np.nan
    assert np.all(np.isnan(blk.lmm(y)[0]))
    blk.close()


@pytest.mark.parametrize("n_rows,n_groups,n_vals,kernel", [
    (300000, 3, 1001, "k_rmm_q1_short_rows"), (300001, 3, 1000, "k_rmm_q1_short_rows"), (300001, 3, 1001, "k_rmm_q1_short"), (400001, 3, 300, "k_rmm_q1_short"),
    (300000, 8, 4097, "k_rmm_q1_short_rows"), (300001, 8, 4097, "k_rmm_rows"), (300001, 7, 4097, "k_rmm_q1_short"), (300001, 8, 4096, "k_rmm_q1_short"),
    (450000, 8, 4097, "k_rmm_rows"), (450001, 8, 4097, "k_rmm_q1_short")])
def test_which_kernel_multiplies_by_a_vector(cla, ora, n_rows, n_groups, n_vals, kernel):
    """X %*% v on both sides of the lines between its kernels, bit for bit against the oracle, and the chain with weights (which
    k_rmm_rows leaves to a kernel of its own) against exact sums."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_vals)
    specs = block(synth, rng, n_rows, n_groups, 1, n_vals)
    v, w = rng.standard_normal((n_groups, 1)), rng.random((n_rows, 1))
    blk = cla.build_block(n_rows, n_groups, specs)
    out, nnz = blk.rmm(v)
    assert kernel in [k["name"] for k in blk.stats()["kernels"]]
    ref, rnnz = ora.rmm(ora.Groups(specs, n_rows, n_groups), v, 1)
    assert np.array_equal(out, ref) and nnz == rnnz
    chain, _ = blk.mmchain(v, w, 1)
    blk.close()
    assert_matches_truth(chain.reshape(1, -1), (w * ref).reshape(1, -1), ora.np_decompress(specs, n_rows, n_groups), what="weighted chain")
