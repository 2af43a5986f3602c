"""The multiply chain of blocks of single-column lists in one kernel (k_chain_sdc): rows and columns at the edges of its quarters and of its
sums, lists longer than what a lane requests ahead, every kind of chain, non-finite operands, and blocks that are not of its shape."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def block(cla, rng, n_rows, n_cols, n_vals, density, gaps=0, default=None):
    from systemds_amd import synth
    at = np.sort(rng.permutation(n_cols + gaps)[:n_cols])
    specs = [synth.sdc_group(rng, n_rows, [int(c)], n_vals, density, default) for c in at]
    return specs, cla.build_block(n_rows, n_cols + gaps, specs)


def chain(blk, v, w, ctype):
    out, nnz = blk.mmchain(v, w if ctype else None, ctype)
    return out.ravel(), nnz, [k["name"] for k in blk.stats()["kernels"]]


@pytest.mark.parametrize("ctype", [0, 1, 2])
@pytest.mark.parametrize("n_rows, n_cols, n_vals, density", [
    (255, 3, 2, 0.5), (256, 1, 1, 0.3), (257, 16, 64, 0.2), (1023, 65, 10, 0.1), (4097, 40, 64, 0.3), (70001, 60, 64, 0.3), (33333, 132, 64, 0.05),
    (600000, 20, 200, 0.02)])
def test_chain_in_one_kernel(cla, ora, n_rows, n_cols, n_vals, density, ctype):
    rng = np.random.default_rng(n_rows + ctype)
    specs, blk = block(cla, rng, n_rows, n_cols, n_vals, density, gaps=ctype)
    n_cols += ctype
    v, w = rng.standard_normal((n_cols, 1)), rng.standard_normal((n_rows, 1))
    for _ in range(2):  # (the second call finds the first one's tickets and workspace)
        out, nnz, names = chain(blk, v, w, ctype)
    blk.close()
    assert names == ["k_chain_sdc"], names
    D = ora.np_decompress(specs, n_rows, n_cols)
    xv = D.astype(np.longdouble) @ v.astype(np.longdouble)
    u = xv * w if ctype == 1 else xv - w if ctype == 2 else xv
    # at most n_cols additions in a row's sum, and in a column's a share of the rows per block and value, then values and blocks: 3000 roundings of either part
    scale = np.abs(D).T @ (np.abs(D) @ np.abs(v) * (np.abs(w) if ctype == 1 else 1.0) + (np.abs(w) if ctype == 2 else 0.0))
    want = D.astype(np.longdouble).T @ u
    assert np.all(np.abs(out.reshape(-1, 1) - want) <= 3000 * 2.0 ** -53 * scale)
    assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("where", ["v", "w"])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_non_finite_operands(cla, where, bad):
    rng = np.random.default_rng(7)
    specs, blk = block(cla, rng, 5000, 30, 20, 0.1)
    specs[3].dict[2, 0] = 0.0
    v, w = rng.standard_normal((30, 1)), rng.standard_normal((5000, 1))
    (v if where == "v" else w)[3] = bad
    out, nnz, names = chain(blk, v, w, 1)
    blk.set_option("chain_fused", 0)
    want, want_nnz, two = chain(blk, v, w, 1)
    blk.close()
    assert names == ["k_chain_sdc"] and "k_chain_sdc" not in two
    finite = np.isfinite(want)
    assert np.array_equal(finite, np.isfinite(out)) and np.array_equal(np.isnan(want), np.isnan(out)) and nnz == want_nnz
    np.testing.assert_allclose(out[finite], want[finite], rtol=1e-12)


@pytest.mark.parametrize("kind", ["default", "table too large", "option", "infinite", "rows too long"])
def test_blocks_of_another_shape(cla, ora, kind):
    rng = np.random.default_rng(8)
    n_cols, density = (140, 0.05) if kind == "table too large" else (60, 0.9) if kind == "rows too long" else (20, 0.1)
    specs, blk = block(cla, rng, 6000, n_cols, 64, density, default=1.5 if kind == "default" else None)
    if kind == "option":
        blk.set_option("sdc_rows", 0)
    if kind == "infinite":
        blk.close()
        specs[2].dict[5, 0] = np.inf
        blk = cla.build_block(6000, n_cols, specs)
    v = rng.standard_normal((n_cols, 1))
    out, nnz, names = chain(blk, v, None, 0)
    blk.close()
    assert "k_chain_sdc" not in names, names
    if kind != "infinite":
        D = ora.np_decompress(specs, 6000, n_cols)
        np.testing.assert_allclose(out, (D.T @ (D @ v)).ravel(), rtol=1e-10, atol=1e-9)
