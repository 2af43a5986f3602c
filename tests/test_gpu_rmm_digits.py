"""X %*% B of byte-code blocks on the integer matrix cores (k_rmm_mfma_i8, option rmm_digits): the edges of its tiles, steps and passes, and the
rows and right-hand sides that its digits do not suit, which the fp64 kernel computes."""
import ctypes as C

import numpy as np
import pytest

from devmem import DevBuf, hip
from test_gpu_gram_tiles import columns

pytestmark = pytest.mark.gpu


def product(cla, specs, n_rows, n_cols, B, digits=2):
    blk = cla.build_block(n_rows, n_cols, specs)
    blk.set_option("rmm_digits", digits)
    out, nnz = blk.rmm(B)
    names = [k["name"] for k in blk.stats()["kernels"]]
    again, _ = blk.rmm(B)  # (the marks are the call's)
    blk.close()
    assert np.array_equal(out, again, equal_nan=True)
    return out, nnz, names


def check(out, D, B, rows=slice(None)):
    """Outputs against 80-bit products. Digits lose 6 products of weight 7 a column (each of standard deviation 2^-70 74^2 of the largest possible
    term), which is 1.1e-16 sqrt(K / 100) of it together, and an output's terms come to 2^-2 sqrt(K / 100) of it at least: 4.5e-16 of their
    sum. 8e-15 is 17 times that, and more than 100 rounded additions in fp64 come to."""
    D = D[rows].astype(np.longdouble)
    err = np.abs(out[rows] - D @ B.astype(np.longdouble))
    assert np.all(err <= 8e-15 * (np.abs(D) @ np.abs(B).astype(np.longdouble)))


@pytest.mark.parametrize("n_cols", [64, 65, 68, 69, 80, 95, 96, 97, 100])
@pytest.mark.parametrize("n_rows,n_vals,q", [(1, 3, 64), (31, 256, 33), (257, 7, 9), (511, 256, 128), (33 * 512 + 5, 256, 32), (256 * 257 + 33, 60, 81), (256 * 300, 256, 61)])
def test_edges(cla, ora, n_cols, n_rows, n_vals, q):
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols * q + n_rows)
    specs = columns(synth, rng, n_rows, n_cols, n_vals, np.uint8, 1)
    B = rng.standard_normal((n_cols, q))
    out, nnz, names = product(cla, specs, n_rows, n_cols, B)
    assert "k_rmm_mfma_i8" in names, names
    check(out, ora.np_decompress(specs, n_rows, n_cols), B, np.r_[0:min(n_rows, 1200), max(0, n_rows - 1200):n_rows])
    assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("q", [9, 50, 130])
@pytest.mark.parametrize("digits", [0, 2])
def test_wide_groups_and_constants(cla, ora, q, digits):
    """Constants come with the layout of B, 64 columns of B at a time, not from a kernel of their own; the counter is cleared once."""
    from systemds_amd import synth
    rng = np.random.default_rng(5)
    n_rows, n_cols = 9001, 90
    specs = columns(synth, rng, n_rows, n_cols - 4, 30, np.uint8, 8)
    specs[1].dict[:, 0] = 0.0
    specs.append(synth.GroupSpec("const", np.array([n_cols - 3, n_cols - 1], np.int32), np.array([[2.5, -1.0]])))
    specs.append(synth.GroupSpec("const", np.array([0, 7], np.int32), np.array([[1.5, 0.25]])))
    B = rng.standard_normal((n_cols, q))
    B[:, 3] = 0.0
    out, nnz, names = product(cla, specs, n_rows, n_cols, B, digits)
    assert ("k_rmm_mfma_i8" in names) == (digits == 2) and "k_preagg" not in names
    D = ora.np_decompress(specs, n_rows, n_cols)
    check(out, D, B)
    assert nnz == np.count_nonzero(out) and not out[:, 3].any()


def test_whole_numbers_are_exact(cla):
    """Products below 2^53 together have no digits at weights above 6, whatever their factors' sizes."""
    from systemds_amd import synth
    rng = np.random.default_rng(3)
    n_rows, n_cols, q = 70_001, 99, 40
    codes = rng.integers(0, 200, (n_cols, n_rows)).astype(np.uint8)
    bits = rng.integers(1, 36, n_cols)
    dicts = np.stack([rng.integers(-2 ** int(b), 2 ** int(b) + 1, 200) for b in bits])
    B = np.stack([rng.integers(-2 ** int(45 - b), 2 ** int(45 - b) + 1, q) for b in bits])
    specs = [synth.GroupSpec("ddc", np.array([c], np.int32), dicts[c].astype(np.float64)[:, None], codes[c]) for c in range(n_cols)]
    out, nnz, names = product(cla, specs, n_rows, n_cols, B.astype(np.float64))
    D = np.stack([dicts[c][codes[c]] for c in range(n_cols)], 1)
    assert np.array_equal(out, (D @ B).astype(np.float64)) and nnz == np.count_nonzero(out)


@pytest.mark.parametrize("kind", ["some rows", "most rows", "one-hot", "far apart", "infinite B", "nan B", "tiny B", "huge B", "infinite", "far columns"])
@pytest.mark.parametrize("q", [20, 64])
def test_values_that_digits_do_not_suit(cla, ora, kind, q):
    """Outputs whose terms are far below their columns' largest values keep fp64's accuracy, and what is not finite in B comes out as in fp64."""
    from systemds_amd import synth
    rng = np.random.default_rng(4)
    n_rows, n_cols = 140_011, 66
    specs = columns(synth, rng, n_rows, n_cols, 40, np.uint8, 1)
    B = rng.standard_normal((n_cols, q))
    small = {"some rows": np.arange(n_rows) % 9973 == 17, "most rows": np.arange(n_rows) % 50 < 40}.get(kind)
    for s in specs:
        if small is not None:
            s.dict[:20, 0] *= 1e-9
            s.codes[:] = np.where(small, s.codes % 20, 20 + s.codes % 20)
        elif kind == "one-hot":
            s.dict[:, 0] = np.arange(40) == 3
        elif kind == "far apart":
            s.dict[0, 0] = 1e12
    if kind == "infinite B":
        B[7, 5] = np.inf
    elif kind == "nan B":
        B[7, 5] = np.nan
    elif kind == "tiny B":
        B *= 1e-290
    elif kind == "huge B":
        B *= 1e290
        specs[0].dict *= 1e17
    elif kind == "infinite":
        specs[5].dict[3, 0] = np.inf
    elif kind == "far columns":  # (only the last columns' terms count: the first step's magnitudes are not enough)
        B[:40] *= 1e-12
    out, nnz, names = product(cla, specs, n_rows, n_cols, B)
    want, want_nnz, _ = product(cla, specs, n_rows, n_cols, B, 0)
    assert ("k_rmm_mfma_i8" in names) == (kind != "infinite")
    if kind in ("infinite B", "nan B", "infinite", "tiny B", "huge B"):
        assert np.array_equal(np.isfinite(out), np.isfinite(want)) and np.array_equal(np.isnan(out), np.isnan(want))
        if kind not in ("tiny B", "huge B"):
            assert np.array_equal(out, want, equal_nan=True) and nnz == want_nnz
            return
    assert nnz == np.count_nonzero(out)
    D = ora.np_decompress(specs, n_rows, n_cols)
    rows = np.r_[0:3000] if small is None else np.r_[0:1000, np.flatnonzero(small)[:1000]]
    check(out, D, B, rows)


def test_capture_without_a_plan(cla, ora):
    """A block prepared without the digits' plan can be captured all the same (in fp64: a capture refuses the plan's allocation); eager calls
    between the replays take the digits."""
    from systemds_amd import synth
    rng = np.random.default_rng(11)
    n_rows, n_cols, q = 1500, 80, 32
    specs = columns(synth, rng, n_rows, n_cols, 30, np.uint8, 1)
    D = ora.np_decompress(specs, n_rows, n_cols)
    blk = cla.build_block(n_rows, n_cols, specs)
    h, stream = hip(), C.c_void_p()
    ok = lambda rc: (_ for _ in ()).throw(AssertionError(rc)) if rc else None
    ok(h.hipStreamCreate(C.byref(stream)))
    blk.set_stream(stream.value)
    blk.set_option("rmm_digits", 0)
    blk.prepare(rmm_cols=q)
    blk.set_option("rmm_digits", 2)
    dB, dO = DevBuf.from_numpy(np.zeros((n_cols, q))), DevBuf(n_rows * q * 8)
    graph, run = C.c_void_p(), C.c_void_p()
    ok(h.hipStreamBeginCapture(stream, 0))
    blk.rmm_dev_async(dB.ptr, q, dO.ptr)
    ok(h.hipStreamEndCapture(stream, C.byref(graph)))
    names = [k["name"] for k in blk.stats()["kernels"]]
    assert "k_rmm_mfma" in names and "k_rmm_mfma_i8" not in names, names
    ok(h.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
    for _ in range(3):
        B = rng.standard_normal((n_cols, q))
        ok(h.hipMemcpy(dB.ptr, B.ctypes.data_as(C.c_void_p), B.nbytes, 1))
        dO.zero()
        ok(h.hipDeviceSynchronize())
        ok(h.hipGraphLaunch(run, stream))
        ok(h.hipStreamSynchronize(stream))
        got = dO.to_numpy(n_rows * q).reshape(n_rows, q)
        assert blk.nnz() == np.count_nonzero(got)
        check(got, D, B)
        out, _ = blk.rmm(B)
        assert "k_rmm_mfma_i8" in [k["name"] for k in blk.stats()["kernels"]]
        check(out, D, B)
    ok(h.hipGraphExecDestroy(run))
    ok(h.hipGraphDestroy(graph))
    blk.close()
    ok(h.hipStreamDestroy(stream))


def test_replays_behind_an_option(cla, ora):
    """Captured products on digits, replayed behind options set since (unrelated ones, and those that send the eager calls between the
    replays elsewhere): what they read and write stays with the block."""
    from systemds_amd import synth
    rng = np.random.default_rng(12)
    n_rows, n_cols, q = 21_000, 80, 32
    specs = columns(synth, rng, n_rows, n_cols, 200, np.uint8, 1)
    for s in specs:
        s.dict = rng.uniform(-1, 1, s.dict.shape)
    D = ora.np_decompress(specs, n_rows, n_cols)
    h, stream = hip(), C.c_void_p()
    ok = lambda rc: (_ for _ in ()).throw(AssertionError(rc)) if rc else None
    ok(h.hipStreamCreate(C.byref(stream)))
    blk = cla.build_block(n_rows, n_cols, specs)
    blk.set_stream(stream.value)
    for key in ("rmm_digits", "tsmm_digits"):
        blk.set_option(key, 2)
    blk.prepare(rmm_cols=q, tsmm=True)
    dB, dO, dG = DevBuf.from_numpy(np.zeros((n_cols, q))), DevBuf(n_rows * q * 8), DevBuf(n_cols * n_cols * 8)
    runs = []
    for call in (lambda: blk.rmm_dev_async(dB.ptr, q, dO.ptr), lambda: blk.tsmm_dev_async(dG.ptr)):
        graph, run = C.c_void_p(), C.c_void_p()
        ok(h.hipStreamBeginCapture(stream, 0))
        call()
        ok(h.hipStreamEndCapture(stream, C.byref(graph)))
        ok(h.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
        runs.append((graph, run, {k["name"]: k["lds"] for k in blk.stats()["kernels"]}))
    assert "k_rmm_mfma_i8" in runs[0][2]
    gram = blk.tsmm()[0]
    for options in ((("sdc_rows", 1),), (("rmm_digits", 0), ("tsmm_digits", 0)), (("rmm_digits", 2), ("tsmm_digits", 1))):
        for key, value in options:
            blk.set_option(key, value)
        others = [DevBuf(1 << 20) for _ in range(8)]  # (freed memory would be given out again)
        for o in others:
            o.zero()
        B = rng.standard_normal((n_cols, q))
        eager, _ = blk.rmm(B)
        out, _ = blk.tsmm()
        if options[-1] == ("tsmm_digits", 0):
            assert blk.stats()["kernels"][0]["lds"] != runs[1][2]["k_gram_tiles"]  # (the captured one is the digits' kernel)
        ok(h.hipMemcpy(dB.ptr, B.ctypes.data_as(C.c_void_p), B.nbytes, 1))
        dO.zero()
        dG.zero()
        ok(h.hipDeviceSynchronize())
        for _, run, _ in runs:
            ok(h.hipGraphLaunch(run, stream))
        ok(h.hipStreamSynchronize(stream))
        got = dO.to_numpy(n_rows * q).reshape(n_rows, q)
        check(got, D, B)
        check(eager, D, B)
        assert np.array_equal(dG.to_numpy(n_cols * n_cols).reshape(n_cols, n_cols), gram)  # (the same sums in every call)
        assert np.allclose(out, gram, rtol=0, atol=2 * n_rows ** 2 * 2.0 ** -53)  # (as many roundings of sums below n_rows)
    for graph, run, _ in runs:
        ok(h.hipGraphExecDestroy(run))
        ok(h.hipGraphDestroy(graph))
    blk.close()
    ok(h.hipStreamDestroy(stream))


@pytest.mark.parametrize("kind,digits", [("normal", True), ("uniform", True), ("X t", False), ("B t", False), ("X one at 8", False), ("B one at 20", False), ("X lognormal", False),
                                         ("X mostly zeros", False), ("B three decades", False), ("B one column", False)])
@pytest.mark.parametrize("n_cols", [64, 100])
def test_no_less_precise_than_fp64(cla, ora, kind, digits, n_cols):
    """Unasked, columns of B go to digits only where the error that is to be expected does not exceed the fp64 kernel's."""
    from systemds_amd import synth
    rng = np.random.default_rng(n_cols)
    n_rows, n_vals, q = 3001, 256, 64
    specs = columns(synth, rng, n_rows, n_cols, n_vals, np.uint8, 1)
    B = rng.standard_normal((n_cols, q))
    for s in specs:
        if kind == "uniform":
            s.dict = rng.uniform(-1, 1, s.dict.shape)
        elif kind == "X t":
            s.dict = rng.standard_t(3, s.dict.shape)
        elif kind == "X one at 8":
            s.dict[200] = 8.0
        elif kind == "X lognormal":
            s.dict = np.exp(s.dict)
        elif kind == "X mostly zeros":
            s.dict[rng.random(s.dict.shape) < 0.9] = 0.0
    if kind == "B t":
        B = rng.standard_t(2, B.shape)
    elif kind == "B one at 20":
        B[33] = 20.0
    elif kind == "B three decades":
        B *= 10 ** rng.uniform(-3, 0, B.shape)
    elif kind == "B one column":  # (one of the second half whose values but one are far below that)
        B[:, 40] *= 1e-4
        B[5, 40] = 1.0
    out, nnz, names = product(cla, specs, n_rows, n_cols, B, 1)
    want, want_nnz, _ = product(cla, specs, n_rows, n_cols, B, 0)
    assert nnz == want_nnz == np.count_nonzero(out)
    if not digits:
        assert np.array_equal(out, want)  # (the fp64 kernel's sums have one order)
        return
    assert "k_rmm_mfma_i8" in names
    D = ora.np_decompress(specs, n_rows, n_cols).astype(np.longdouble)
    scale = np.abs(D) @ np.abs(B)
    got, ref = (np.abs(o - D @ B.astype(np.longdouble)) / scale for o in (out, want))
    assert not np.array_equal(out, want) and np.sqrt((got ** 2).mean()) <= np.sqrt((ref ** 2).mean()) and got.max() <= ref.max()


@pytest.mark.parametrize("n_rows,low,digits", [(60_000, 0, True), (60_000, 1, False), (300_001, 0, True), (300_001, 20, True), (300_001, 60, False)])
def test_rows_far_below_the_others(cla, ora, n_rows, low, digits):
    """512 rows with one that digits do not suit go through both kernels: a block with many such rows is not sent to digits at all, nor is a
    short one with any (117 and 586 times 512 rows)."""
    from systemds_amd import synth
    rng = np.random.default_rng(low)
    n_cols, q = 80, 40
    specs = columns(synth, rng, n_rows, n_cols, 200, np.uint8, 1)
    at = np.arange(low) * 512 * (n_rows // 512 // max(low, 1)) + 3
    for s in specs:
        s.dict[:20] *= 1e-9
        s.codes[:] = 20 + s.codes % 180
        s.codes[at] %= 20
    B = rng.standard_normal((n_cols, q))
    out, nnz, names = product(cla, specs, n_rows, n_cols, B, 1)
    assert ("k_rmm_mfma_i8" in names) == digits and nnz == np.count_nonzero(out)
    check(out, ora.np_decompress(specs, n_rows, n_cols), B, np.r_[0:1000, at.astype(int), n_rows - 1000:n_rows])
