"""The multiply chain of blocks of column pairs with two-byte codes in one kernel (k_chain_pairs): numbers of pairs and rows at the edges of its
instantiations and blocks, dictionaries in and out of LDS, non-finite operands, and blocks that are not of its shape."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def block(cla, rng, n_rows, n_cols, n_vals, gaps=0, width=2, bad=None):
    from systemds_amd import synth
    at = rng.permutation(n_cols + gaps)[:n_cols].astype(np.int32)
    specs = []
    for c in range(0, n_cols, width):
        d = rng.standard_normal((n_vals, len(at[c:c + width])))
        d[rng.integers(0, n_vals)] = 0.0
        specs.append(synth.GroupSpec("ddc", at[c:c + width], d, rng.integers(0, n_vals, n_rows).astype(np.uint16)))
    if bad is not None:
        specs[0].dict[0, 0] = bad
    return specs, cla.build_block(n_rows, n_cols + gaps, specs)


def chain(blk, v, w, ctype):
    out, nnz = blk.mmchain(v, w if ctype else None, ctype)
    return out.ravel(), nnz, [k["name"] for k in blk.stats()["kernels"]]


@pytest.mark.parametrize("n_cols", [2, 8, 10, 16, 18, 24, 26, 32, 34, 40, 42, 50])
@pytest.mark.parametrize("n_rows, n_vals, ctype", [(1, 3, 1), (511, 300, 0), (513, 5000, 2), (20001, 300, 1), (140001, 1000, 0)])
def test_chain_in_one_kernel(cla, ora, n_cols, n_rows, n_vals, ctype):
    rng = np.random.default_rng(n_rows + n_cols)
    specs, blk = block(cla, rng, n_rows, n_cols, n_vals, gaps=ctype)
    n_cols += ctype
    v, w = rng.standard_normal((n_cols, 1)), rng.standard_normal((n_rows, 1))
    for _ in range(2):  # (the second call finds the first one's tickets and workspace)
        out, nnz, names = chain(blk, v, w, ctype)
    blk.close()
    assert names == ["k_chain_pairs"], names
    D = ora.np_decompress(specs, n_rows, n_cols)
    xv = D.astype(np.longdouble) @ v.astype(np.longdouble)
    u = xv * w if ctype == 1 else xv - w if ctype == 2 else xv
    # a row's sum and a thread's rows (2 at most here) are short chains, then 64 lanes, 8 waves and the blocks: fewer than 500 roundings of either part
    scale = np.abs(D).T @ (np.abs(D) @ np.abs(v) * (np.abs(w) if ctype == 1 else 1.0) + (np.abs(w) if ctype == 2 else 0.0))
    want = D.astype(np.longdouble).T @ u
    assert np.all(np.abs(out.reshape(-1, 1) - want) <= 500 * 2.0 ** -53 * scale)
    assert nnz == np.count_nonzero(out)


@pytest.mark.parametrize("where", ["v", "w"])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("n_vals", [40, 6000])
def test_non_finite_operands(cla, where, bad, n_vals):
    rng = np.random.default_rng(7)
    specs, blk = block(cla, rng, 5000, 12, n_vals)
    v, w = rng.standard_normal((12, 1)), rng.standard_normal((5000, 1))
    (v if where == "v" else w)[3] = bad
    out, nnz, names = chain(blk, v, w, 1)
    blk.set_option("chain_fused", 0)
    want, want_nnz, two = chain(blk, v, w, 1)
    blk.close()
    assert names == ["k_chain_pairs"] and "k_chain_pairs" not in two
    finite = np.isfinite(want)
    assert np.array_equal(finite, np.isfinite(out)) and np.array_equal(np.isnan(want), np.isnan(out)) and nnz == want_nnz
    np.testing.assert_allclose(out[finite], want[finite], rtol=1e-12)


@pytest.mark.parametrize("kind", ["52 columns", "single columns", "option", "infinite", "many lookups"])
def test_blocks_of_another_shape(cla, ora, kind):
    rng = np.random.default_rng(8)
    n_rows, n_cols, n_vals, width = 6000, 12, 300, 2
    if kind == "52 columns":
        n_cols = 52
    if kind == "single columns":
        width = 1
    if kind == "many lookups":  # (large dictionaries on many rows: the tables of the two products are the faster way)
        n_rows, n_cols, n_vals = 520_000, 50, 4000
    specs, blk = block(cla, rng, n_rows, n_cols, n_vals, width=width, bad=np.inf if kind == "infinite" else None)
    if kind == "option":
        blk.set_option("chain_fused", 0)
    v = rng.standard_normal((n_cols, 1))
    out, nnz, names = chain(blk, v, None, 0)
    blk.close()
    assert "k_chain_pairs" not in names, names
    if kind != "infinite":
        D = ora.np_decompress(specs, n_rows, n_cols)
        np.testing.assert_allclose(out, (D.T @ (D @ v)).ravel(), rtol=1e-9, atol=1e-7)


@pytest.mark.parametrize("kind", ["pairs", "byte codes", "lists"])
def test_replays_behind_a_chain_of_two_products(cla, ora, kind):
    """A captured chain, replayed behind one that runs as two products and needs a larger workspace: its own stays with the block."""
    import ctypes as C
    from devmem import DevBuf, hip
    from systemds_amd import synth
    rng = np.random.default_rng(13)
    n_rows, n_cols = 30_011, 12
    if kind == "pairs":
        specs, blk = block(cla, rng, n_rows, n_cols, 300)
    else:
        specs = [synth.sdc_group(rng, n_rows, [c], 16, 0.05, None) if kind == "lists" else
                 synth.GroupSpec("ddc", np.array([c], np.int32), rng.standard_normal((30, 1)), rng.integers(0, 30, n_rows).astype(np.uint8)) for c in range(n_cols)]
        blk = cla.build_block(n_rows, n_cols, specs)
    D = ora.np_decompress(specs, n_rows, n_cols)
    h, stream = hip(), C.c_void_p()
    ok = lambda rc: (_ for _ in ()).throw(AssertionError(rc)) if rc else None
    ok(h.hipStreamCreate(C.byref(stream)))
    blk.set_stream(stream.value)
    blk.prepare(rmm_cols=1, lmm_rows=1)
    dV, dO = DevBuf.from_numpy(np.zeros(n_cols)), DevBuf(n_cols * 8)
    graph, run = C.c_void_p(), C.c_void_p()
    ok(h.hipStreamBeginCapture(stream, 0))
    blk.mmchain_dev_async(dV.ptr, None, 0, dO.ptr)
    ok(h.hipStreamEndCapture(stream, C.byref(graph)))
    assert len(blk.stats()["kernels"]) == 1
    ok(h.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
    for fused in (0, 1, 0):
        v = rng.standard_normal((n_cols, 1))
        blk.set_option("chain_fused", fused)
        eager, _, names = chain(blk, v, None, 0)
        assert (len(names) == 1) == bool(fused)
        others = [DevBuf(1 << 16) for _ in range(16)]  # (freed memory would be given out again)
        for o in others:
            o.zero()
        ok(h.hipMemcpy(dV.ptr, v.ctypes.data_as(C.c_void_p), v.nbytes, 1))
        dO.zero()
        ok(h.hipDeviceSynchronize())
        ok(h.hipGraphLaunch(run, stream))
        ok(h.hipStreamSynchronize(stream))
        scale = np.abs(D).T @ (np.abs(D) @ np.abs(v))
        want = D.T.astype(np.longdouble) @ (D @ v.astype(np.longdouble))
        for got in (dO.to_numpy(n_cols), eager):  # (3000 roundings as above)
            assert np.all(np.abs(got.reshape(-1, 1) - want) <= 3000 * 2.0 ** -53 * scale)
    ok(h.hipGraphExecDestroy(run))
    ok(h.hipGraphDestroy(graph))
    blk.close()
    ok(h.hipStreamDestroy(stream))
