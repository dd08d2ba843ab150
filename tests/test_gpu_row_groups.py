"""FLAT row groups (k_vector: FLAT "tiles" 2..32 are lanes per row) on the GPU, against the oracle.

Every edge case of csr_cases (empty rows, empty rows at both ends, one row, rows longer than the lanes and
than 256 nnz, duplicate and unsorted columns, rectangular x) and scaled C1, C2 and C4, for every lane count
and every value type, y NaN-prefilled before each call:

* initVec values bit for bit against spmv_serial (fp16: against the once-rounded exact sum): the products
  and partial sums are small integers, exact in any order;
* U[-1,1] values within the tolerance of assert_parity;
* the plan is one launch with no split-row workspace (row_aligned 1, needs_fixup 0, one workgroup per 256
  lanes) and the same y on its first and later calls.
"""
import numpy as np
import pytest

import oracle
import prefree_amd as pf
from csr_cases import edge_cases
from gpu_util import NP, assert_parity, gpu_spmv, kat_exact_possible

pytestmark = pytest.mark.gpu

LANES = [2, 4, 8, 16, 32]


def _cases():
    out = list(edge_cases())
    for cfg, scale in ((1, 0), (2, 200), (4, 300000)):
        rp, col, _ = pf.synth_csr(cfg, seed=3, scale_n=scale, dtypes=())
        out.append((f"C{cfg}", rp, col, len(rp) - 1))
    return out


CASES = _cases()


@pytest.mark.parametrize("dtype", ["f64", "f32", "f16"])
@pytest.mark.parametrize("lanes", LANES)
def test_row_groups_match_oracle(lanes, dtype):
    assert lanes in pf.supported_tiles("flat", dtype)
    for name, rp, col, n in CASES:
        m = len(rp) - 1
        if m == 0:
            continue
        what = f"{name} lanes={lanes} {dtype}"
        print(what, flush=True)
        kv, kx = oracle.initvec(len(col), NP[dtype]), oracle.initvec(n, NP[dtype])
        y, info = gpu_spmv(rp, col, kv, kx, "flat", tile=lanes, dtype=dtype)
        assert (info["tile"], info["row_aligned"], info["needs_fixup"]) == (lanes, 1, 0), what
        assert info["ntiles"] == max(1, -(-m * lanes // 256)), what
        assert_parity(rp, col, kv, kx, y, dtype, exact=kat_exact_possible(rp, dtype), what=what + " kat")
        rng = np.random.default_rng(lanes * 31 + len(col))
        uv = rng.uniform(-1, 1, len(col)).astype(NP[dtype])
        ux = rng.uniform(-1, 1, n).astype(NP[dtype])
        y, _ = gpu_spmv(rp, col, uv, ux, "flat", tile=lanes, dtype=dtype)
        assert_parity(rp, col, uv, ux, y, dtype, what=what + " random")


def test_auto_takes_row_groups_for_small_short_rows():
    """AUTO's rule on real plans: C1 takes 16 lanes, C2 at 512^2 (262,144 rows of 5) takes 2; one row more
    than 2^18 takes row-aligned tiles."""
    for cfg, scale, lanes in ((1, 0, 16), (2, 512, 2)):
        rp, col, v = pf.synth_csr(cfg, seed=1, scale_n=scale)
        x = pf.synth_x(cfg, len(rp) - 1, seed=1)["f64"]
        y, info = gpu_spmv(rp, col, v["f64"], x, "auto")
        assert (info["variant_name"], info["tile"]) == ("flat", lanes), (cfg, info)
        assert_parity(rp, col, v["f64"], x, y, "f64", what=f"C{cfg} auto")
    m = (1 << 18) + 1
    rp = np.arange(m + 1, dtype=np.int32) * 3
    col = (np.arange(3 * m, dtype=np.int64) * 7919 % m).astype(np.int32)
    y, info = gpu_spmv(rp, col, oracle.initvec(len(col)), oracle.initvec(m), "auto")
    assert info["tile"] in (1024, 2048) and info["row_aligned"] == 1, info


def test_row_groups_at_the_rule_bounds():
    """2^18 rows of up to 256 nnz: fp32 values and columns within 256 MB take row groups (half the mean row of
    48: 32 lanes), the same pattern at 128 nnz per row in fp64 (403 MB) takes tiles; both against the oracle."""
    rng = np.random.default_rng(17)
    m = 1 << 18
    for dtype, lam, want_groups in (("f32", 48.0, True), ("f64", 128.0, False)):
        lens = np.minimum(rng.poisson(lam, m), 256)
        rp = np.zeros(m + 1, dtype=np.int64)
        np.cumsum(lens, out=rp[1:])
        rp = rp.astype(np.int32)
        col = rng.integers(0, m, int(rp[-1])).astype(np.int32)
        val = oracle.initvec(len(col), NP[dtype])
        x = oracle.initvec(m, NP[dtype])
        print(f"bounds {dtype} nnz={len(col)}", flush=True)
        y, info = gpu_spmv(rp, col, val, x, "auto", dtype=dtype)
        groups = info["variant_name"] == "flat" and info["tile"] <= 32
        assert groups == want_groups, (dtype, info)
        if want_groups:
            assert info["tile"] == 32, info
        assert_parity(rp, col, val, x, y, dtype, exact=kat_exact_possible(rp, dtype), what=f"bounds {dtype}")


@pytest.mark.parametrize("dtype", ["f64", "f32", "f16"])
@pytest.mark.parametrize("extra,longest,groups", [(0, 64, True), (-1, 64, False), (0, 65, False)])
def test_auto_over_2_18_rows_of_middling_length(extra, longest, groups, dtype):
    """One row more than 2^18, 7 nnz per row on average: row groups at the rule's lower edge and at the longest row
    it takes, tiles one nnz below the one or above the other; ragged rows, empty ones among them, against the oracle."""
    rng = np.random.default_rng(7)
    m = (1 << 18) + 1
    lens = rng.integers(0, 14, m)
    lens[rng.integers(0, m)] = 0
    lens[m - 1] = longest
    short = 7 * m + extra - int(lens.sum())  # the rest of the nnz, over rows that stay under 32
    at = rng.choice(m - 1, abs(short), replace=False)
    if short < 0:
        at = np.flatnonzero(lens[:m - 1] > 0)[:-short]
    lens[at] += 1 if short > 0 else -1
    assert lens.sum() == 7 * m + extra and lens.max() == longest and lens.min() == 0
    rp = np.zeros(m + 1, dtype=np.int64)
    np.cumsum(lens, out=rp[1:])
    rp = rp.astype(np.int32)
    col = rng.integers(0, 60000, int(rp[-1])).astype(np.int32)
    val, x = oracle.initvec(len(col), NP[dtype]), oracle.initvec(60000, NP[dtype])
    y, info = gpu_spmv(rp, col, val, x, "auto", dtype=dtype)
    assert (info["variant_name"], info["tile"] <= 32) == ("flat", groups), info
    assert_parity(rp, col, val, x, y, dtype, exact=kat_exact_possible(rp, dtype), what=f"{extra} {longest} {dtype}")


@pytest.mark.parametrize("dtype", ["f64", "f32", "f16"])
@pytest.mark.parametrize("block", [1, 2])
@pytest.mark.parametrize("pattern,groups", [("9-point", False), ("random", True)])
def test_auto_over_2_18_rows_looks_at_the_columns(pattern, groups, block, dtype):
    """9 columns a row: a stencil keeps its tiles, whole or as the second half of its rows (whose columns lie far from
    its local row numbers); random columns take row groups, but not in fp64 over the 4.2 MB of x of the half (24.2 us
    in row groups, 21.0 in tiles)."""
    groups = groups and not (block == 2 and dtype == "f64")
    side = 513 if block == 1 else 726
    n = side * side
    if pattern == "random":
        rng = np.random.default_rng(8)
        cols = np.sort(rng.integers(0, n, (n, 9)), axis=1)
    else:
        d = np.array([-1, 0, 1])
        cols = np.arange(n)[:, None] + (side * d[:, None] + d[None, :]).ravel()[None, :]
    cols = cols[n - n // block:]
    ok = (cols >= 0) & (cols < n)
    rp = np.zeros(len(cols) + 1, dtype=np.int32)
    rp[1:] = np.cumsum(ok.sum(1))
    col = cols[ok].astype(np.int32)
    assert len(cols) > 1 << 18
    val, x = oracle.initvec(len(col), NP[dtype]), oracle.initvec(n, NP[dtype])
    y, info = gpu_spmv(rp, col, val, x, "auto", dtype=dtype)
    assert (info["variant_name"], info["tile"] <= 32) == ("flat", groups), info
    assert_parity(rp, col, val, x, y, dtype, exact=kat_exact_possible(rp, dtype), what=f"{pattern} {block} {dtype}")


@pytest.mark.parametrize("per,rows,dtype,random_groups,band_groups", [
    (8, 400003, "f64", True, True), (8, 600001, "f64", False, True),     # x of 3.2 and 4.8 MB
    (10, 290001, "f64", True, True), (10, 400003, "f64", False, True),   # 2.3 and 3.2 MB
    (12, 400003, "f64", True, True),
    (8, 600001, "f32", True, True), (8, 900001, "f32", False, True),     # 2.4 and 3.6 MB
    (10, 500001, "f32", True, True), (10, 700001, "f32", False, True),   # 2.0 and 2.8 MB
    (12, 300007, "f32", True, False), (12, 700001, "f32", False, False),
    (16, 500001, "f32", True, True), (10, 700001, "f16", True, True),
])
def test_auto_over_2_18_rows_looks_at_the_size_of_x(per, rows, dtype, random_groups, band_groups):
    """Scattered columns, random over all of x or within 20,000 of their row: row groups up to the rule's x, and over
    it only in a band."""
    rng = np.random.default_rng(9)
    rp = (np.arange(rows + 1) * per).astype(np.int32)
    val, x = oracle.initvec(rows * per, NP[dtype]), oracle.initvec(rows, NP[dtype])
    for w, groups in ((0, random_groups), (20000, band_groups)):
        cols = (np.arange(rows)[:, None] + rng.integers(-w, w + 1, (rows, per))) % rows if w else \
            rng.integers(0, rows, (rows, per))
        col = np.sort(cols, axis=1).astype(np.int32).ravel()
        y, info = gpu_spmv(rp, col, val, x, "auto", dtype=dtype)
        assert (info["variant_name"], info["tile"] <= 32) == ("flat", groups), (w, info)
        assert_parity(rp, col, val, x, y, dtype, exact=kat_exact_possible(rp, dtype), what=f"{per} {rows} {dtype} {w}")
