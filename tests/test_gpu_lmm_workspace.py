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


def test_captured_calls_and_larger_ones(cla, ora):
    """A call is captured with more rows of Y than the workspace has seen (the tables of an X %*% B have the room); eager calls of many more rows,
    which take a larger workspace, come between the replays of it and of one captured with what there was."""
    import ctypes as C
    from devmem import DevBuf, hip
    from systemds_amd import synth
    rng = np.random.default_rng(8)
    n_rows, n_cols = 5001, 10
    specs = [synth.GroupSpec("ddc", np.array([c, c + 1], np.int32), rng.standard_normal((400, 2)), rng.integers(0, 400, n_rows).astype(np.uint16))
             for c in range(0, 8, 2)] + [synth.GroupSpec("unc", np.array([8, 9], np.int32), dense=rng.standard_normal((n_rows, 2)))]
    D = ora.np_decompress(specs, n_rows, n_cols)

    def check(out, Y):  # (sums of 5001 terms in any order; fewer than 600 roundings on the way of each)
        assert np.all(np.abs(out - Y @ D) <= 600 * 2.0 ** -53 * (np.abs(Y) @ np.abs(D)))

    h, stream = hip(), C.c_void_p()
    ok = lambda rc: (_ for _ in ()).throw(AssertionError(rc)) if rc else None
    ok(h.hipStreamCreate(C.byref(stream)))
    blk = cla.build_block(n_rows, n_cols, specs)
    blk.set_stream(stream.value)
    blk.prepare(rmm_cols=16, lmm_rows=2)
    runs = []
    for p in (2, 5):
        dY, dO = DevBuf.from_numpy(np.zeros((p, n_rows))), DevBuf(p * n_cols * 8)
        graph, run = C.c_void_p(), C.c_void_p()
        ok(h.hipStreamBeginCapture(stream, 0))
        blk.lmm_dev_async(dY.ptr, p, dO.ptr)
        ok(h.hipStreamEndCapture(stream, C.byref(graph)))
        assert "k_take_block" in [k["name"] for k in blk.stats()["kernels"]]
        ok(h.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
        runs.append((p, dY, dO, graph, run))
    for p_eager in (5, 16, 40, 100):
        Y = rng.standard_normal((p_eager, n_rows))
        check(blk.lmm(Y)[0], Y)
        for p, dY, dO, _, run in runs:
            Y = rng.standard_normal((p, n_rows))
            ok(h.hipMemcpy(dY.ptr, Y.ctypes.data_as(C.c_void_p), Y.nbytes, 1))
            ok(h.hipGraphLaunch(run, stream))
            ok(h.hipStreamSynchronize(stream))
            check(dO.to_numpy(p * n_cols).reshape(p, n_cols), Y)
    for _, _, _, graph, run in runs:
        ok(h.hipGraphExecDestroy(run))
        ok(h.hipGraphDestroy(graph))
    blk.close()
    ok(h.hipStreamDestroy(stream))
