"""X %*% v of byte-code blocks of few rows (k_rmm_q1_u8_few): bit for bit the oracle's sums, at the edges of its rows per thread, threads
per block, batches of groups and table sizes, and where it hands over to k_rmm_q1_u8."""
import numpy as np
import pytest

from devmem import DevBuf

pytestmark = pytest.mark.gpu


def block_specs(rng, n_rows, n_cols, n_vals):
    from systemds_amd import synth
    return [synth.GroupSpec("ddc", np.array([c], np.int32), rng.standard_normal((n_vals, 1)), rng.integers(0, n_vals, n_rows).astype(np.uint8))
            for c in range(n_cols)]


@pytest.mark.parametrize("n_rows, n_cols, n_vals", [
    (1, 1, 1), (2, 16, 2), (3, 17, 3), (511, 32, 256), (513, 33, 255), (1025, 70, 256), (5000, 97, 100),
    (131071, 3, 5), (131073, 15, 200), (262143, 5, 16), (262145, 31, 37), (524287, 4, 7), (524291, 18, 64), (786431, 8, 9), (786433, 8, 9),
    (1048575, 9, 4), (1048577, 9, 4), (600001, 75, 256), (2000, 80, 256),
    (600001, 96, 208), (600001, 96, 210), (600001, 79, 252), (600001, 79, 254), (4000, 96, 208), (4000, 79, 254)])
def test_bit_for_bit(cla, ora, n_rows, n_cols, n_vals):
    rng = np.random.default_rng(n_rows + n_cols)
    specs = block_specs(rng, n_rows, n_cols, n_vals)
    v, w = rng.standard_normal((n_cols, 1)), rng.standard_normal((n_rows, 1))
    blk = cla.build_block(n_rows, n_cols, specs)
    stride = max((n_vals + 1) // 2 * 2, 2)
    entries = 512 * 38 if n_rows <= 256 * 2048 else 1024 * 20
    # (of 163840 bytes of LDS the kernel has 256 of its own)
    takes = n_rows <= 256 * (3072 if n_cols <= 8 else 4096) and n_cols * stride <= entries and ((n_cols + 1) * stride + n_cols) * 8 <= 160 * 1024 - 256
    for _ in range(3):  # (the counters of consecutive calls take turns)
        out, nnz = blk.rmm(v)
        names = [k["name"] for k in blk.stats()["kernels"]]
        assert names == ["k_rmm_q1_u8_few" if takes else "k_rmm_q1_u8"], names
    ref, rnnz = ora.rmm(ora.Groups(specs, n_rows, n_cols), v, 1)
    assert np.array_equal(out, ref) and nnz == rnnz
    # with the chain's weights: the row sums rounded, then the product or difference rounded
    blk.set_option("chain_fused", 0)
    for ctype in (1, 2):
        chain, _ = blk.mmchain(v, w, ctype)
        want, _ = blk.lmm((ref * w if ctype == 1 else ref - w).reshape(1, -1))
        np.testing.assert_allclose(chain.reshape(-1), want.reshape(-1), rtol=0, atol=1e-12 * np.abs(ref).sum() * max(1.0, np.abs(w).max()) * 10)
    blk.close()


def test_output_at_odd_places(cla, ora):
    """An output that starts 8 bytes behind a multiple of 16."""
    rng = np.random.default_rng(3)
    for n_rows in (777, 200003, 400001):
        specs = block_specs(rng, n_rows, 6, 11)
        v = rng.standard_normal((6, 1))
        ref, _ = ora.rmm(ora.Groups(specs, n_rows, 6), v, 1)
        blk = cla.build_block(n_rows, 6, specs)
        dv, do = DevBuf.from_numpy(v), DevBuf.from_numpy(np.full(n_rows + 2, 7.0))
        blk.rmm_dev(dv.ptr, 1, do.ptr + 8)
        got = do.to_numpy(n_rows + 2)
        blk.close()
        assert got[0] == 7.0 and got[-1] == 7.0 and np.array_equal(got[1:-1], ref.reshape(-1))
