"""Row groups beside long rows: AUTO's plan for a few long rows among short ones of middling length, against the
oracle, at the edges of its rule and of its kernel (batches of 8192 nnz, rows that start inside a line, long rows
first, last and next to each other)."""
import numpy as np
import pytest
import torch

import oracle
import prefree_amd as pf
from csr_cases import csr_from_lengths
from gpu_util import DEV, NP, assert_parity, dev, gpu_spmv, kat_exact_possible

pytestmark = pytest.mark.gpu

# lengths of the long rows, and where they stand among 3001 short rows of 0-40 nnz (an odd count, so that they
# start anywhere in a line)
LONG = {
    "one": [(1500, 3000)],
    "first_and_last": [(0, 1024), (3000, 1025)],
    "adjacent": [(7, 8191), (8, 8192), (9, 8193)],
    "largest": [(100, 65536), (2000, 257 + 1800)],
    "batch_pairs": [(3, 16384), (4, 16385), (2999, 24576)],
}


def _matrix(name, n=70001, seed=5):
    rng = np.random.default_rng(seed)
    lengths = rng.integers(0, 41, 3001)
    lengths[rng.integers(0, 3001, 60)] = 0
    for at, length in LONG[name]:
        lengths[at] = length
    rp, col = csr_from_lengths([int(v) for v in lengths], n, rng)
    return rp, col, n


@pytest.fixture(autouse=True)
def split_rows_table(tmp_path):
    """Table rows as the shipped table has at these sizes: split-row tiles, or row groups beside long rows."""
    t = tmp_path / "table.txt"
    t.write_text("".join(f"t -1 {rows} {d} flat {tile} 0 0 0 0\n" for d in ("f64", "f32", "f16")
                         for rows in ("dense", "skewed") for tile in (16, 2048)))
    pf.set_tuning_table(str(t))
    yield
    pf.set_tuning_table(None)


@pytest.mark.parametrize("dtype", ["f64", "f32", "f16"])
@pytest.mark.parametrize("name", sorted(LONG))
def test_long_rows_beside_row_groups(name, dtype):
    rp, col, n = _matrix(name)
    kv, kx = oracle.initvec(len(col), NP[dtype]), oracle.initvec(n, NP[dtype])
    y, info = gpu_spmv(rp, col, kv, kx, "auto", dtype=dtype)
    assert (info["variant_name"], info["tile"], info["hybrid"]) == ("flat", 16, 0), info
    nlong = len(LONG[name])
    assert info["dense_rows"] == nlong and info["ntiles"] == info["grid"] == (3001 * 16 + 1023) // 1024 + nlong, info
    assert_parity(rp, col, kv, kx, y, dtype, exact=kat_exact_possible(rp, dtype), what=f"{name}/kat")
    rng = np.random.default_rng(1)
    val = rng.uniform(-1, 1, len(col)).astype(NP[dtype])
    x = rng.uniform(-1, 1, n).astype(NP[dtype])
    y, _ = gpu_spmv(rp, col, val, x, "auto", dtype=dtype)
    assert_parity(rp, col, val, x, y, dtype, what=f"{name}/random")


@pytest.mark.parametrize("what,change", [
    ("a row over 2^16", lambda l: l.__setitem__(5, 65537)),
    ("a short row over 128", lambda l: l.__setitem__(5, 129)),
    ("long rows under 1024 on average", lambda l: l.__setitem__(1500, 900)),
    ("short rows under 12 on average", lambda l: l.__setitem__(slice(2000, None), 0)),
])
def test_rule_refuses(what, change):
    rng = np.random.default_rng(6)
    lengths = rng.integers(4, 24, 3001)
    lengths[1500] = 3000
    change(lengths)
    rp, col = csr_from_lengths([int(v) for v in lengths], 70001, rng)
    val, x = oracle.initvec(len(col)), oracle.initvec(70001)
    y, info = gpu_spmv(rp, col, val, x, "auto")
    assert info["tile"] == 2048, (what, info)
    assert_parity(rp, col, val, x, y, "f64", exact=True, what=what)


@pytest.mark.parametrize("tail,tile", [("", 16), ("u -1 any f64 flat 2048 0 0 0 0\n", 16),
                                       ("u -1 skewed f64 flat 2048 0 0 0 0\n", 2048)])
def test_a_lone_table_row_of_16_lanes_means_row_groups(tmp_path, tail, tile):
    """Rows under 12 nnz, where row groups beside long rows do not pay: a "flat 16" row is passed over only if a later
    row repeats its bound, class and type."""
    t = tmp_path / "lone.txt"
    t.write_text("t -1 skewed f64 flat 16 0 0 0 0\n" + tail)
    pf.set_tuning_table(str(t))
    rng = np.random.default_rng(6)
    lengths = rng.integers(0, 8, 3001)
    lengths[1500] = 3000
    rp, col = csr_from_lengths([int(v) for v in lengths], 70001, rng)
    val, x = oracle.initvec(len(col)), oracle.initvec(70001)
    y, info = gpu_spmv(rp, col, val, x, "auto")
    assert (info["variant_name"], info["tile"]) == ("flat", tile), info
    assert_parity(rp, col, val, x, y, "f64", exact=True, what="lone row")


def test_autotune_tells_the_plan_from_plain_row_groups():
    """Where the plan's own row groups beside long rows win, the result says so; FLAT 16 by name has no long rows."""
    rp, col, n = _matrix("largest")
    m, nnz = len(rp) - 1, len(col)
    d = [dev(a) for a in (rp, col, oracle.initvec(nnz), oracle.initvec(n))]
    y = torch.full((m,), float("nan"), dtype=torch.float64, device=DEV)
    want = oracle.spmv_serial(rp, col, oracle.initvec(nnz), oracle.initvec(n))
    with pf.Plan(d[0], d[1], m, n, nnz) as p:
        assert (p.info.tile, p.info.dense_rows) == (16, len(LONG["largest"]))
        r = p.autotune(*d, y, reps=5)
        assert r["hybrid"] == (1 if p.info.dense_rows else 0) and (r["variant"], r["tile"]) == (p.info.variant, p.info.tile)
        assert np.array_equal(y.cpu().numpy(), want)
    with pf.Plan(d[0], d[1], m, n, nnz, "f64", "flat", 16) as p:
        assert (p.info.tile, p.info.dense_rows, p.info.grid) == (16, 0, (16 * m + 255) // 256)
        p.execute(*d, y)
        assert np.array_equal(y.cpu().numpy(), want)


@pytest.mark.parametrize("kind", ["beside", "scattered"])
@pytest.mark.parametrize("what", ["chunk", "row_aligned", "x_windows"])
def test_tile_settings_take_row_groups_back_to_tiles(kind, what):
    """The settings of FLAT tiles on a plan whose tiles gave way to row groups: the tiles', with their y bit for bit;
    a refused value leaves the plan as it is."""
    if kind == "beside":
        rp, col, n = _matrix("adjacent")
    else:
        n, rng = 270001, np.random.default_rng(4)
        rp = (np.arange(n + 1) * 12).astype(np.int32)
        col = np.sort(rng.integers(0, n, (n, 12)), axis=1).astype(np.int32).ravel()
    m, nnz, rng = len(rp) - 1, len(col), np.random.default_rng(5)
    d = [dev(a) for a in (rp, col, rng.uniform(-1, 1, nnz), rng.uniform(-1, 1, n))]
    ys = [torch.full((m,), float("nan"), dtype=torch.float64, device=DEV) for _ in range(2)]
    with pf.Plan(d[0], d[1], m, n, nnz) as p:
        assert p.info.tile == 16
        p.execute(*d, ys[0])
        refused = [lambda: p.set_chunk_nnz(-1), lambda: p.set_row_aligned(True) if kind == "beside" else p.set_x_windows(True)]
        for f in refused:
            with pytest.raises(pf.PrefreeError):
                f()
        assert p.info.tile == 16
        {"chunk": lambda: p.set_chunk_nnz(8192), "row_aligned": lambda: p.set_row_aligned(False),
         "x_windows": lambda: p.set_x_windows(kind == "beside")}[what]()
        info = p.info
        assert info.tile in (1024, 2048) and info.dense_rows == 0
        assert info.chunk_nnz == 8192 if what == "chunk" else True
        with pf.Plan(d[0], d[1], m, n, nnz, "f64", "flat", info.tile) as q:
            q.set_chunk_nnz(info.chunk_nnz)
            q.set_row_aligned(info.row_aligned)
            q.set_x_windows(info.x_windows)
            for _ in range(2):  # searched, then read from the map
                for plan, y in ((p, ys[0]), (q, ys[1])):
                    y.fill_(float("nan"))
                    plan.execute(*d, y)
                assert torch.equal(ys[0], ys[1])
                p.check()
        assert_parity(rp, col, d[2].cpu().numpy(), d[3].cpu().numpy(), ys[0].cpu().numpy(), "f64", what=f"{kind} {what}")


def test_tile_settings_stay_refused_on_small_row_groups():
    rp, col, v = pf.synth_csr(1, seed=2)
    d = [dev(rp), dev(col)]
    with pf.Plan(d[0], d[1], 4096, 4096, len(col)) as p:
        assert p.info.tile == 16
        for f in (lambda: p.set_chunk_nnz(8192), lambda: p.set_row_aligned(False), lambda: p.set_x_windows(False)):
            with pytest.raises(pf.PrefreeError) as e:
                f()
            assert pf.STATUS[e.value.status] == "PF_ERR_UNSUPPORTED"


def _stencil_with_long_rows(points, side, nlong, length, seed=3):
    """`points` columns a row around it on a side x side x side (27) or side x side grid (16), random ones (0: 27
    a row; -w: 24 a row within w of it, of `side` rows), and nlong rows of `length` random columns among them."""
    rng = np.random.default_rng(seed)
    if points < 0:
        off = np.zeros(0, dtype=np.int64)
    elif points == 27:
        d = np.array([-1, 0, 1])
        off = (side * side * d[:, None, None] + side * d[None, :, None] + d[None, None, :]).ravel()
    else:
        d = np.arange(-1, 3)
        off = (side * d[:, None] + d[None, :]).ravel()
    n = side if points < 0 else side ** 3 if points in (0, 27) else side ** 2
    if points < 0:
        cols = np.sort((np.arange(n)[:, None] + rng.integers(points, 1 - points, (n, 24))) % n, axis=1)
    else:
        cols = np.sort(rng.integers(0, n, (n, 27)), axis=1) if points == 0 else np.arange(n)[:, None] + off[None, :]
    ok = (cols >= 0) & (cols < n)
    at = np.sort(rng.choice(n, nlong, replace=False))
    ok[at] = False
    lens = ok.sum(1)
    pieces, start = [], 0
    short = np.concatenate([[0], np.cumsum(lens)])
    flat = cols[ok]
    for r in at:
        pieces += [flat[short[start]:short[r]], np.sort(rng.choice(n, length, replace=False))]
        start = r
    pieces.append(flat[short[start]:])
    lens[at] = length
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    return rp, np.concatenate(pieces).astype(np.int32), n


@pytest.mark.parametrize("points,side,dtype,groups", [
    (27, 56, "f64", False), (27, 56, "f32", True),    # 57 MB of values and columns, 38 MB
    (27, 63, "f32", False), (27, 63, "f16", True),    # 54 MB, 41 MB
    (0, 56, "f64", True), (0, 63, "f32", True),       # random columns at any size within 2.2 MB of x
    (-150000, 300007, "f64", False), (-150000, 300007, "f32", True), (-15000, 300007, "f64", True),  # 2.4 MB, 1.2 MB
    (16, 150, "f64", False), (16, 150, "f32", False), (16, 150, "f16", True), (16, 480, "f16", False),
])
def test_columns_decide_beside_long_rows(points, side, dtype, groups):
    """Long rows among stencils: tiles over the rule's bytes, and at any size where the rows are short; among random
    columns over a large x: tiles, unless they lie in a band."""
    rp, col, n = _stencil_with_long_rows(points, side, 8, 9000)
    val, x = oracle.initvec(len(col), NP[dtype]), oracle.initvec(n, NP[dtype])
    y, info = gpu_spmv(rp, col, val, x, "auto", dtype=dtype)
    assert (info["variant_name"], info["tile"]) == ("flat", 16 if groups else 2048), info
    assert_parity(rp, col, val, x, y, dtype, exact=kat_exact_possible(rp, dtype), what=f"{points} {side} {dtype}")


def test_special_values_and_graph_replay():
    rp, col, n = _matrix("adjacent")
    rng = np.random.default_rng(2)
    val, x = oracle.initvec(len(col)), oracle.initvec(n)
    for a in (val, x):
        at = rng.choice(len(a), 40, replace=False)
        a[at] = np.resize([np.nan, np.inf, -np.inf], 40)
    want = oracle.spmv_serial(rp, col, val, x)
    d = [dev(a) for a in (rp, col, val, x)]
    y = torch.full((len(rp) - 1,), 7.0, dtype=torch.float64, device=DEV)
    with pf.Plan(d[0], d[1], len(rp) - 1, n, len(col)) as p:
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            p.execute(*d, y, stream=s)
            s.synchronize()
            assert np.array_equal(y.cpu().numpy(), want, equal_nan=True)
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                p.execute(*d, y, stream=s)
        for _ in range(3):
            y.fill_(7.0)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(y.cpu().numpy(), want, equal_nan=True)
            d[2].mul_(1.0)  # eager work between the replays
        p.check()


@pytest.mark.parametrize("what", ["a listed row now short", "another row now long"])
def test_row_ptr_changed_after_planning_is_flagged(what):
    rp, col, n = _matrix("one")
    val, x = oracle.initvec(len(col)), oracle.initvec(n)
    d = [dev(a) for a in (rp, col, val, x)]
    y = torch.full((len(rp) - 1,), float("nan"), dtype=torch.float64, device=DEV)
    other = rp.copy()  # in bounds throughout
    if what == "a listed row now short":
        other[1501:] -= 2900
    else:
        other[1498:1501] = other[1500] + 1000  # row 1497 takes over the rows to 1499 and 1000 nnz of the listed row
    with pf.Plan(d[0], d[1], len(rp) - 1, n, len(col)) as p:
        assert p.info.tile == 16
        p.execute(dev(other), d[1], d[2], d[3], y)
        assert np.array_equal(y.cpu().numpy(), oracle.spmv_serial(other, col, val, x))  # and every row summed
        with pytest.raises(pf.PrefreeError) as e:
            p.check()
        assert pf.STATUS[e.value.status] == "PF_ERR_KERNEL"
