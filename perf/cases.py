"""The multiplies that algorithm scripts run on a compressed matrix, as cases to time.

A case is a matrix (its family of column groups, its size) and one product, called through systemds_amd.capi the way
a program that keeps its matrix in HBM calls it: the block is uploaded and prepared once, a product is one call with
operands and output on the device (`_dev_async`), and only the small case of a JVM that hands over Java arrays goes
through the host-pointer entry point. All matrices are fp64, as in the library.

Families
  ddc      single-column dictionary groups with byte codes (Zipf(1.1) over 2 - 256 values)
  cocoded  pairs of columns sharing a dictionary of 257 - 4096 tuples, two-byte codes (Zipf(1.0))
  sdc      single-column offset lists (2 - 10 % of the rows, 64 values, default 0)
  mixed    run-length, two-byte dictionary, offset-list (default 1) and uncompressed columns side by side
"""
import numpy as np
import torch

from systemds_amd import capi
from systemds_amd.synth import GroupSpec

_stream = None


def listed():
    return [
        # Scoring of a small table, a partition of it or a validation fold: latency and launches.
        {"name": "ddc_matvec_small", "family": "ddc", "op": "matvec", "rows": 100_000, "cols": 20, "vals": 16},
        # The inner step of conjugate-gradient regression from a JVM: t(X) %*% (X %*% p) with Java arrays in and out.
        {"name": "ddc_chain_host", "family": "ddc", "op": "chain_host", "rows": 250_007, "cols": 54, "vals": 200},
        # Scoring of a large table.
        {"name": "ddc_matvec", "family": "ddc", "op": "matvec", "rows": 10_000_000, "cols": 100, "vals": 256},
        # Projection onto 64 components, distances to 64 centroids.
        {"name": "ddc_matmult", "family": "ddc", "op": "matmult", "rows": 10_000_000, "cols": 100, "vals": 256, "q": 64},
        # Gradient of multinomial regression with nine classes, the centroid update of clustering: t(P) %*% X.
        {"name": "ddc_leftmult", "family": "ddc", "op": "leftmult", "rows": 2_000_003, "cols": 100, "vals": 256, "p": 8},
        # Normal equations, covariance of more columns than one decoded Gram matrix holds.
        {"name": "ddc_tsmm", "family": "ddc", "op": "tsmm", "rows": 2_000_003, "cols": 100, "vals": 256},
        # Conjugate-gradient step on a co-coded block.
        {"name": "cocoded_chain", "family": "cocoded", "op": "chain", "rows": 2_500_009, "cols": 50, "vals": 4096, "ctype": 0},
        # Covariance of a large co-coded block.
        {"name": "cocoded_tsmm", "family": "cocoded", "op": "tsmm", "rows": 10_000_000, "cols": 50, "vals": 4096},
        # Weighted conjugate-gradient step (generalised linear models) on sparse one-hot style columns.
        {"name": "sdc_chain", "family": "sdc", "op": "chain", "rows": 10_000_000, "cols": 200, "density": 0.05, "ctype": 1},
        # X %*% B with ten classes on a long table of mixed encodings.
        {"name": "mixed_matmult", "family": "mixed", "op": "matmult", "rows": 50_000_000, "rle": 8, "ddc": 8, "sdc": 2, "unc": 2, "q": 10},
        # The matching gradient t(P) %*% X on one of an ordinary size.
        {"name": "mixed_leftmult", "family": "mixed", "op": "leftmult", "rows": 5_000_011, "rle": 8, "ddc": 8, "sdc": 2, "unc": 2, "p": 6},
        # Its normal equations.
        {"name": "mixed_tsmm", "family": "mixed", "op": "tsmm", "rows": 50_000_000, "rle": 8, "ddc": 8, "sdc": 2, "unc": 2},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    family, op = rng.choice([
        ("ddc", "matvec"), ("ddc", "chain_host"), ("ddc", "chain"), ("ddc", "matmult"), ("ddc", "leftmult"), ("ddc", "tsmm"),
        ("cocoded", "chain"), ("cocoded", "tsmm"), ("sdc", "chain"), ("mixed", "matmult"), ("mixed", "leftmult"), ("mixed", "tsmm")])
    c = {"family": family, "op": op}
    if family == "mixed":
        c.update(rows=_log(rng, 100_000, 40_000_000), rle=rng.randint(2, 8), ddc=rng.randint(2, 8), sdc=rng.randint(1, 2), unc=rng.randint(1, 2))
    elif family == "sdc":
        c.update(rows=_log(rng, 100_000, 10_000_000), cols=_log(rng, 20, 200), density=round(rng.uniform(0.02, 0.1), 3))
    elif family == "cocoded":
        c.update(rows=_log(rng, 20_000, 8_000_000), cols=2 * rng.randint(3, 25), vals=_log(rng, 257, 4096))
    else:
        c.update(rows=_log(rng, 1_000, 8_000_000), cols=_log(rng, 5, 100), vals=_log(rng, 2, 256))
        if op == "chain_host":
            c["rows"] = _log(rng, 1_000, 2_000_000)
    if op == "tsmm" and family == "ddc":
        c["rows"] = _log(rng, 10_000, 2_000_000)
    if op == "chain":
        c["ctype"] = rng.randint(0, 2)
    if op == "matmult":
        c["q"] = rng.randint(2, 64) if family == "ddc" else rng.randint(2, 16)
    if op == "leftmult":
        c["p"] = rng.randint(2, 16)
        c["rows"] = min(c["rows"], 5_000_000)
    return c


# ---- inputs, made on the GPU

def _zipf(gen, n, n_vals, s):
    """n codes below n_vals, Zipf(s) over values in a random order."""
    p = 1.0 / torch.arange(1, n_vals + 1, dtype=torch.float64, device="cuda") ** s
    cdf = torch.cumsum(p / p.sum(), 0)
    at = torch.searchsorted(cdf, torch.rand(n, dtype=torch.float64, device="cuda", generator=gen), right=True).clamp_(max=n_vals - 1)
    return torch.randperm(n_vals, device="cuda", generator=gen)[at]


def _normal(gen, *shape):
    return torch.randn(*shape, dtype=torch.float64, device="cuda", generator=gen)


def _host(t, dtype=None):
    a = t.cpu().numpy()
    return a if dtype is None else a.view(dtype)


def _offset_list(gen, n, col, density, n_vals, default):
    """An SDC / SDCZeros group: byte gaps between the listed rows, a zero byte for every 255 rows on the way."""
    rows = torch.nonzero(torch.rand(n, device="cuda", generator=gen) < density).flatten()
    gaps = rows[1:] - rows[:-1]
    skips = (gaps - 1) // 255
    end = torch.cumsum(skips + 1, 0) - 1
    deltas = torch.zeros(int(end[-1]) + 1 if gaps.numel() else 0, dtype=torch.uint8, device="cuda")
    deltas[end] = (gaps - 255 * skips).to(torch.uint8)
    codes = torch.randint(0, n_vals, (rows.numel(),), device="cuda", generator=gen).to(torch.uint8)
    return GroupSpec("sdc", np.array([col], np.int32), _host(_normal(gen, n_vals, 1)), _host(codes),
                     None if default is None else np.array([default]), _host(deltas), int(rows[0]), int(rows[-1]), rows.numel())


def _run_list(gen, n, col, n_vals, mean_run):
    """An RLE group: per value its (gap, length) pairs, gaps of more than 65535 rows with empty runs on the way."""
    m = int(n / mean_run * 1.3) + 64
    u = torch.rand(m, dtype=torch.float64, device="cuda", generator=gen)
    lens = _host((torch.log(1.0 - u) / np.log(1.0 - 1.0 / mean_run)).long() + 1)
    lens = np.minimum(lens, 65535)
    codes = _host(torch.randint(0, n_vals, (m,), device="cuda", generator=gen))
    ends = np.cumsum(lens)
    if ends[-1] < n:
        raise RuntimeError("too few runs were drawn")
    k = int(np.searchsorted(ends, n)) + 1
    starts, ends, codes = (ends - lens)[:k], np.minimum(ends[:k], n), codes[:k]
    order = np.lexsort((starts, codes))
    starts, ends, codes = starts[order], ends[order], codes[order]
    before = np.concatenate(([0], ends[:-1]))
    before[np.concatenate(([True], codes[1:] != codes[:-1]))] = 0
    gaps = starts - before
    fill = np.maximum(gaps - 1, 0) // 65535
    data = np.zeros((int((fill + 1).sum()), 2), np.uint16)
    data[:, 0] = 65535
    at = np.cumsum(fill + 1) - 1
    data[at, 0] = gaps - 65535 * fill
    data[at, 1] = ends - starts
    ptr = np.zeros(n_vals + 1, np.int32)
    ptr[1:] = 2 * np.cumsum(np.bincount(codes, weights=fill + 1, minlength=n_vals))
    return GroupSpec("rle", np.array([col], np.int32), _host(_normal(gen, n_vals, 1)), ptr=ptr, rle=data.reshape(-1))


def _groups(case, gen):
    """The block's column groups one after the other."""
    n = case["rows"]
    if case["family"] == "ddc":
        for c in range(case["cols"]):
            codes = _zipf(gen, n, case["vals"], 1.1).to(torch.uint8)
            yield GroupSpec("ddc", np.array([c], np.int32), _host(_normal(gen, case["vals"], 1)), _host(codes))
    elif case["family"] == "cocoded":
        for c in range(0, case["cols"], 2):
            codes = _zipf(gen, n, case["vals"], 1.0).to(torch.int16)
            d = torch.rand(case["vals"], 2, dtype=torch.float64, device="cuda", generator=gen) * 2 - 1
            yield GroupSpec("ddc", np.array([c, c + 1], np.int32), _host(d), _host(codes, np.uint16))
    elif case["family"] == "sdc":
        for c in range(case["cols"]):
            yield _offset_list(gen, n, c, case["density"], 64, None)
    else:
        c = 0
        for _ in range(case["rle"]):
            yield _run_list(gen, n, c, 32, 1000.0)
            c += 1
        for _ in range(case["ddc"]):
            codes = torch.randint(0, 1024, (n,), device="cuda", generator=gen).to(torch.int16)
            yield GroupSpec("ddc", np.array([c], np.int32), _host(_normal(gen, 1024, 1)), _host(codes, np.uint16))
            c += 1
        for _ in range(case["sdc"]):
            yield _offset_list(gen, n, c, 0.1, 16, 1.0)
            c += 1
        dense = _host(_normal(gen, n, case["unc"]))
        yield GroupSpec("unc", np.arange(c, c + case["unc"], dtype=np.int32), dense=dense)


def _cols(case):
    return case["cols"] if "cols" in case else case["rle"] + case["ddc"] + case["sdc"] + case["unc"]


def prepare(case, seed):
    """The block on the device with what its product derives from it built (cla_block_prepare), the operands and the output."""
    global _stream
    if _stream is None:
        torch.cuda.init()
        capi.init(torch.cuda.current_device())
        _stream = torch.cuda.Stream()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    n, m, op = case["rows"], _cols(case), case["op"]
    blk = capi.ClaBlock(n, m)
    for g in _groups(case, gen):
        blk.add(g)
    blk.finalize()
    blk.set_stream(_stream.cuda_stream)
    s = {"op": op, "blk": blk}
    if op == "matvec":
        s["B"], s["q"], s["out"] = _normal(gen, m, 1), 1, torch.empty(n, 1, dtype=torch.float64, device="cuda")
        blk.prepare(rmm_cols=1)
    elif op == "matmult":
        s["B"], s["q"], s["out"] = _normal(gen, m, case["q"]), case["q"], torch.empty(n, case["q"], dtype=torch.float64, device="cuda")
        blk.prepare(rmm_cols=case["q"])
    elif op == "leftmult":
        s["Y"], s["p"], s["out"] = _normal(gen, case["p"], n), case["p"], torch.empty(case["p"], m, dtype=torch.float64, device="cuda")
        blk.prepare(lmm_rows=case["p"])
    elif op == "tsmm":
        s["out"] = torch.empty(m, m, dtype=torch.float64, device="cuda")
        blk.prepare(tsmm=True)
    elif op == "chain":
        s["v"], s["out"] = _normal(gen, m), torch.empty(m, dtype=torch.float64, device="cuda")
        s["ctype"] = case["ctype"]
        s["w"] = torch.rand(n, dtype=torch.float64, device="cuda", generator=gen) if case["ctype"] else None
        blk.prepare(rmm_cols=1, lmm_rows=1)
    elif op == "chain_host":
        s["v"] = _host(_normal(gen, m))
        blk.prepare(rmm_cols=1, lmm_rows=1)
    torch.cuda.synchronize()
    return s


def run(state):
    op, blk = state["op"], state["blk"]
    if op in ("matvec", "matmult"):
        blk.rmm_dev_async(state["B"].data_ptr(), state["q"], state["out"].data_ptr())
    elif op == "leftmult":
        blk.lmm_dev_async(state["Y"].data_ptr(), state["p"], state["out"].data_ptr())
    elif op == "tsmm":
        blk.tsmm_dev_async(state["out"].data_ptr())
    elif op == "chain":
        w = state["w"]
        blk.mmchain_dev_async(state["v"].data_ptr(), None if w is None else w.data_ptr(), state["ctype"], state["out"].data_ptr())
    else:
        return blk.mmchain(state["v"])  # (out, number of non-zeros)
    return state["out"]


def work(case):
    """The compressed matrix once, operands and output once. Multiply-adds of the product on the decoded matrix where it
    is a contraction with a wide operand; a product with one vector needs one add per stored code."""
    n, m, op = case["rows"], _cols(case), case["op"]
    if case["family"] == "ddc":
        x, cells = n * m + 8 * m * case["vals"], n * m
    elif case["family"] == "cocoded":
        x, cells = n * m + 8 * m * case["vals"], n * m
    elif case["family"] == "sdc":
        x, cells = 2 * n * m * case["density"], n * m * case["density"]
    else:
        x = n * (2 * case["ddc"] + 2 * 0.1 * case["sdc"] + 8 * case["unc"]) + case["rle"] * n / 1000 * 4
        cells = n * m
    if op == "matvec":
        return {"bytes": x + 8 * (m + n), "flops": cells}
    if op == "matmult":
        return {"bytes": x + 8 * case["q"] * (m + n), "flops": 2 * cells * case["q"]}
    if op == "leftmult":
        return {"bytes": x + 8 * case["p"] * (m + n), "flops": 2 * cells * case["p"]}
    if op == "tsmm":
        return {"bytes": x + 8 * m * m, "flops": cells * (m + 1)}
    # the chain: both products' result depends on a whole row of X at a time, so X can be read once
    return {"bytes": x + 8 * (2 * m + (n if case.get("ctype") else 0)), "flops": 3 * cells}


def tolerance(case):
    # Four times the largest difference between two kernels of the library that form the same fp64 sums in another order
    # (chosen with cla_block_set_option): 2.7e-16 / 2.7e-15 (relative, largest) for X %*% B, 1.7e-15 / 5.2e-15 for Y %*% X and
    # the chain, 5.5e-14 / 1.3e-13 for t(X) %*% X, whose sums have up to 50 million terms.
    if case["op"] in ("matvec", "matmult"):
        return {"rel": 1.2e-15, "max": 1.2e-14}
    if case["op"] == "tsmm":
        return {"rel": 2.2e-13, "max": 6e-13}
    return {"rel": 7e-15, "max": 2.5e-14}
