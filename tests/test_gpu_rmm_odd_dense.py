"""X %*% B on blocks with an odd number of dense columns: the kernel on streams takes a filler column beside them. Edges of its
slices of 128 rows, widths of B around the rule's lines, infinities and NaN in the dense columns; the tile kernel forms the same sums."""
import numpy as np
import pytest

from parity import assert_matches_truth

pytestmark = pytest.mark.gpu


def block(cla, synth, rng, n_rows, unc, runs, odd_values):
    specs, c = [], 0
    for _ in range(runs):
        lens = rng.geometric(1.0 / 900.0, size=n_rows // 300 + 16)
        codes = np.repeat(rng.integers(0, 8, size=lens.size), lens)[:n_rows]
        ptr, data = synth.encode_rle(np.concatenate([codes, np.zeros(n_rows - codes.size, codes.dtype)]), 8)
        specs.append(synth.GroupSpec("rle", np.array([c], np.int32), rng.standard_normal((8, 1)), ptr=ptr, rle=data))
        c += 1
    for n_vals, dt in [(700, np.uint16), (30, np.uint8), (1, np.uint8)]:
        specs.append(synth.GroupSpec("ddc", np.array([c], np.int32), rng.standard_normal((n_vals, 1)), rng.integers(0, n_vals, n_rows).astype(dt)))
        c += 1
    dense = rng.standard_normal((n_rows, unc))
    if odd_values:
        for v in (np.inf, -np.inf, np.nan):
            dense[rng.integers(0, n_rows), rng.integers(0, unc)] = v
    specs.append(synth.GroupSpec("unc", np.arange(c, c + unc, dtype=np.int32), dense=dense))
    return specs, c + unc, cla.build_block(n_rows, c + unc, specs)


@pytest.mark.parametrize("n_rows", [4097, 32767, 32768, 32895, 33025, 300001])
@pytest.mark.parametrize("unc, runs, odd_values", [(1, 0, False), (1, 3, False), (3, 2, True), (5, 0, True)])
@pytest.mark.parametrize("q", [1, 2, 7, 10, 11, 15, 16, 17])
def test_odd_number_of_dense_columns(cla, ora, n_rows, unc, runs, odd_values, q):
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + 10 * unc + q)
    specs, n_cols, blk = block(cla, synth, rng, n_rows, unc, runs, odd_values)
    B = rng.standard_normal((n_cols, q))
    out, nnz = blk.rmm(B)
    names = [k["name"] for k in blk.stats()["kernels"]]
    tiles, _ = blk.set_option("rmm_direct", 0).rmm(B)
    blk.close()
    # (32,768 rows: a slice per CU of 256; 262,144: half of their 16 waves with one each)
    streams = q <= 15 and n_rows >= (32768 if q <= 10 else 262144)
    assert ("k_rmm_direct" in names) == streams and ("k_rmm_decode" in names) != streams, names
    fin = np.isfinite(tiles)
    assert np.array_equal(np.isfinite(out), fin) and np.array_equal(out[~fin], tiles[~fin], equal_nan=True)
    assert nnz == np.count_nonzero(out)
    D = ora.np_decompress(specs, n_rows, n_cols)
    rows = fin.all(axis=1)
    if rows.any():
        assert_matches_truth(out.reshape(n_rows, q)[rows], D[rows], B, what=f"odd dense q={q}")


@pytest.mark.parametrize("q", [11, 12, 15])
def test_more_columns_on_few_rows(cla, ora, q):
    """Nine columns and more take the kernel on streams from a slice per CU on, whatever the number of columns of B up to 15."""
    from systemds_amd import synth
    for n_rows in (32768, 40003):
        rng = np.random.default_rng(n_rows + q)
        specs, n_cols, blk = block(cla, synth, rng, n_rows, 3, 3, False)
        B = rng.standard_normal((n_cols, q))
        out, nnz = blk.rmm(B)
        names = [k["name"] for k in blk.stats()["kernels"]]
        blk.close()
        assert n_cols == 9 and "k_rmm_direct" in names, names
        assert_matches_truth(out, ora.np_decompress(specs, n_rows, n_cols), B, what=f"nine columns, q={q}")
        assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("n_rows", [257, 1003, 40003])
@pytest.mark.parametrize("q", [15, 16])
def test_sixteen_columns_of_b(cla, ora, n_rows, q):
    """An even number of dense columns: as for 15 columns of B next to run-length columns, on the tile kernel without them."""
    from systemds_amd import synth
    for runs in (3, 0):
        rng = np.random.default_rng(n_rows + q)
        specs, n_cols, blk = block(cla, synth, rng, n_rows, 2, runs, False)
        B = rng.standard_normal((n_cols, q))
        out, nnz = blk.rmm(B)
        names = [k["name"] for k in blk.stats()["kernels"]]
        blk.close()
        assert ("k_rmm_direct" in names) == (q == 15 or runs > 0), (runs, names)
        assert_matches_truth(out, ora.np_decompress(specs, n_rows, n_cols), B, what=f"{runs} run-length columns, q={q}")
        assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("n_rows", [1, 31, 33, 129, 40003])
@pytest.mark.parametrize("n_vals", [60, 970, 1010])
@pytest.mark.parametrize("q", [1, 4, 8, 10, 12, 15, 16, 24, 32])
def test_staging_with_and_without_gaps(cla, ora, n_rows, n_vals, q):
    """Rows on their way out of the kernel on streams: pairs of rows apart in LDS where 12 dictionaries leave room for it (with 16 columns of B those
    of 970 values do, those of 1010 do not), behind one another where they do not."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_vals + q)
    specs, n_cols = [], 12
    for c in range(n_cols):
        specs.append(synth.GroupSpec("ddc", np.array([c], np.int32), rng.standard_normal((n_vals, 1)), rng.integers(0, n_vals, n_rows).astype(np.uint16)))
    if n_rows > 1:  # (run-length columns: 16 columns of B on this kernel, too)
        codes = np.where(np.arange(n_rows) < n_rows // 2, 1, 0)
        ptr, data = synth.encode_rle(codes, 2)
        specs.append(synth.GroupSpec("rle", np.array([n_cols], np.int32), rng.standard_normal((2, 1)), ptr=ptr, rle=data))
        n_cols += 1
    B = rng.standard_normal((n_cols, q))
    blk = cla.build_block(n_rows, n_cols, specs)
    out, nnz = blk.rmm(B)
    blk.close()
    D = ora.np_decompress(specs, n_rows, n_cols)
    assert_matches_truth(out, D, B, what=f"{n_vals} values, q={q}")
    assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("unc, row_bytes, q, n_rows, direct", [(11, 92, 15, 2717391, True), (11, 92, 15, 2717392, False), (11, 92, 14, 2717392, True), (12, 100, 16, 2500000, True),
                                                               (12, 100, 16, 2500001, False), (13, 108, 15, 2400000, True)])
def test_streams_beyond_the_cache(cla, ora, unc, row_bytes, q, n_rows, direct):
    """Streams of 250 MB together and a row more, 15 and 16 columns of B: the kernel on streams, the tile kernel (up to 16 columns)."""
    from systemds_amd import synth
    rng = np.random.default_rng(q)
    specs, n_cols, blk = block(cla, synth, rng, n_rows, unc, 1, False)
    assert n_cols == unc + 4 and row_bytes == 8 * unc + 4
    B = rng.standard_normal((n_cols, q))
    out, nnz = blk.rmm(B)
    names = [k["name"] for k in blk.stats()["kernels"]]
    blk.close()
    assert ("k_rmm_direct" in names) == direct and ("k_rmm_decode" in names) != direct, names
    D = ora.np_decompress(specs, n_rows, n_cols)
    # (two fp64 sums of at most 17 terms, each within 17 * 2^-53 of the sum of magnitudes)
    assert np.all(np.abs(out - D @ B) <= 34 * 2.0 ** -53 * (np.abs(D) @ np.abs(B)))
    assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("n_rows, q, direct", [(1003, 17, True), (899999, 17, False), (900000, 17, True), (900001, 19, False), (249999, 24, False), (250000, 24, True),
                                               (250001, 18, True), (499999, 40, False), (500000, 40, True), (500003, 33, False), (20011, 16, True)])
def test_wide_b_beside_dictionaries_that_fill_lds(cla, ora, n_rows, q, direct):
    """Dictionaries that leave the tile kernel no room: more than 16 columns of B on decompressed rows below the lines (but for very
    few rows), on streams above."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + q)
    specs, c = [], 0
    for _ in range(3):
        codes = np.repeat(rng.integers(0, 8, n_rows // 500 + 1), 500)[:n_rows]
        ptr, data = synth.encode_rle(codes, 8)
        specs.append(synth.GroupSpec("rle", np.array([c], np.int32), rng.standard_normal((8, 1)), ptr=ptr, rle=data))
        c += 1
    for _ in range(8):
        specs.append(synth.GroupSpec("ddc", np.array([c], np.int32), rng.standard_normal((1024, 1)), rng.integers(0, 1024, n_rows).astype(np.uint16)))
        c += 1
    specs.append(synth.GroupSpec("unc", np.arange(c, c + 5, dtype=np.int32), dense=rng.standard_normal((n_rows, 5))))
    c += 5
    B = rng.standard_normal((c, q))
    blk = cla.build_block(n_rows, c, specs)
    out, nnz = blk.rmm(B)
    names = [k["name"] for k in blk.stats()["kernels"]]
    blk.close()
    assert ("k_rmm_direct" in names) == direct and ("k_dense_rmm" in names) != direct, names
    D = ora.np_decompress(specs, n_rows, c)
    # (two fp64 sums of at most 17 terms, each within 17 * 2^-53 of the sum of magnitudes)
    assert np.all(np.abs(out - D @ B) <= 34 * 2.0 ** -53 * (np.abs(D) @ np.abs(B)))
    assert nnz == np.count_nonzero(out)
