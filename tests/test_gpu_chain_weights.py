"""The multiply chain's weights and subtracted vector, applied where X %*% v writes its rows: every kernel that does so, over
their row edges, against the exact chain; and bit for bit what the two products and a separate pass give."""
import numpy as np
import pytest

from conftest import mixed_block
from parity import assert_matches_truth

pytestmark = pytest.mark.gpu


def specs_of(synth, kind, rng, n_rows, n_cols):
    if kind == "mixed":
        return mixed_block(3, n_rows, with_unc=False)
    out = []
    for c in range(n_cols):
        col = np.array([c], np.int32)
        if kind == "bytes":
            out.append(synth.GroupSpec("ddc", col, rng.standard_normal((40, 1)), rng.integers(0, 40, n_rows).astype(np.uint8)))
        elif kind == "shorts":
            out.append(synth.GroupSpec("ddc", col, rng.standard_normal((1000, 1)), rng.integers(0, 1000, n_rows).astype(np.uint16)))
        else:
            rows = np.flatnonzero(rng.random(n_rows) < 0.1)
            deltas, first, last, n = synth.encode_offsets(rows)
            out.append(synth.GroupSpec("sdc", col, rng.standard_normal((16, 1)), rng.integers(0, 16, n).astype(np.uint8), None, deltas, first, last, n))
    if kind == "lists_default":
        out.append(synth.GroupSpec("const", np.array([0], np.int32), np.array([[0.5]])))
    return out, n_cols


@pytest.mark.parametrize("kind", ["bytes", "shorts", "lists", "lists_default", "mixed"])
@pytest.mark.parametrize("n_rows", [17, 1024, 40001, 500003])
@pytest.mark.parametrize("ctype", [0, 1, 2])
def test_chain(cla, ora, kind, n_rows, ctype):
    from systemds_amd import synth
    rng = np.random.default_rng(n_rows + ctype)
    specs, n_cols = specs_of(synth, kind, rng, n_rows, 21)
    v, w = rng.standard_normal((n_cols, 1)), rng.standard_normal((n_rows, 1))
    blk = cla.build_block(n_rows, n_cols, specs)
    out, nnz = blk.mmchain(v, w if ctype else None, ctype)
    xv, _ = blk.rmm(v)  # the product itself is as it was
    blk.close()
    D = ora.np_decompress(specs, n_rows, n_cols)
    assert_matches_truth(xv, D, v, what="X %*% v")
    u = xv * w if ctype == 1 else xv - w if ctype == 2 else xv
    assert_matches_truth(out.reshape(-1, 1), D.T, u, what=f"chain {kind} {ctype}")
    assert nnz == np.count_nonzero(out)
