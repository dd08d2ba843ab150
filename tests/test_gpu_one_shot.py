"""pf_spmv, the one-shot product, against the oracle: its plan is made in the library's device scratch where that is
free, else in allocations of its own, and both give the product and the errors of a plan."""
import threading

import numpy as np
import pytest
import torch

import oracle
import prefree_amd as pf
from csr_cases import edge_cases
from gpu_util import DEV, NP, TORCH, assert_parity, dev, kat_exact_possible

pytestmark = pytest.mark.gpu

EDGE = {name: (rp, col, n) for name, rp, col, n in edge_cases()}


def _call(rp, col, val, x, dtype, stream=None):
    y = torch.full((max(len(rp) - 1, 1),), float("nan"), dtype=TORCH[dtype], device=DEV)
    pf.spmv(dev(rp), dev(col), dev(val), dev(x), y, len(rp) - 1, len(x), len(col), dtype, stream=stream)
    return y[:len(rp) - 1].cpu().numpy()


@pytest.mark.parametrize("dtype", ["f64", "f32", "f16"])
@pytest.mark.parametrize("name", sorted(EDGE))
def test_edge_cases(name, dtype):
    rp, col, n = EDGE[name]
    val, x = oracle.initvec(len(col), NP[dtype]), oracle.initvec(n, NP[dtype])
    for _ in range(2):  # the second call finds the first one's workspace in the scratch
        y = _call(rp, col, val, x, dtype)
        assert_parity(rp, col, val, x, y, dtype, exact=kat_exact_possible(rp, dtype), what=name)


def test_errors_are_a_plans():
    rp, col, v = pf.synth_csr(1, seed=2)
    x = pf.synth_x(1, len(rp) - 1, seed=2)["f64"]
    bad = col.copy()
    bad[len(bad) // 2] = len(rp)
    with pytest.raises(pf.PrefreeError) as e:
        _call(rp, bad, v["f64"], x, "f64")
    assert pf.STATUS[e.value.status] == "PF_ERR_CSR"
    y = torch.empty(len(rp) - 1, dtype=torch.float64, device=DEV)
    shifted = torch.zeros(len(col) + 1, dtype=torch.float64, device=DEV)[1:]
    for val, yy, want in ((shifted, y, "PF_ERR_ALIGN"), (None, y, "PF_ERR_INVALID"), (dev(v["f64"]), None, "PF_ERR_INVALID")):
        with pytest.raises(pf.PrefreeError) as e:
            pf.spmv(dev(rp), dev(col), val, dev(x), yy, len(rp) - 1, len(x), len(col))
        assert pf.STATUS[e.value.status] == want


def test_threads_share_the_device():
    """Three host threads at once, each on its own stream: the one that holds the scratch and those that do not."""
    jobs, failures = [], []
    for cfg, scale in ((2, 300), (3, 100000), (5, 20000)):
        rp, col, v = pf.synth_csr(cfg, seed=6, scale_n=scale)
        val, x = oracle.initvec(len(col)), oracle.initvec(len(rp) - 1)
        jobs.append((rp, col, val, x, oracle.spmv_serial(rp, col, val, x), torch.cuda.Stream()))
    torch.cuda.synchronize()

    def worker(k):
        rp, col, val, x, want, s = jobs[k]
        try:
            d = [dev(a) for a in (rp, col, val, x)]
            y = torch.empty(len(rp) - 1, dtype=torch.float64, device=DEV)
            torch.cuda.synchronize()
            for it in range(8):
                pf.spmv(*d, y, len(rp) - 1, len(x), len(col), "f64", "auto", s)
                if not np.array_equal(y.cpu().numpy(), want):
                    failures.append((k, it))
        except Exception as e:
            failures.append((k, repr(e)))

    threads = [threading.Thread(target=worker, args=(k,)) for k in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not any(t.is_alive() for t in threads) and not failures, failures


@pytest.mark.parametrize("dtype", ["f64", "f32", "f16"])
@pytest.mark.parametrize("family,size", [(1, 300007), (3, 800000), (5, 40000)],
                         ids=["scattered", "power-law", "dense-rows"])
def test_y_does_not_depend_on_other_threads(family, size, dtype):
    """Random values, whose sums depend on their order: calls that find another thread in the scratch give the bits of
    a call that has it for itself.  Plans of these matrices take other kernels (row groups, long rows, hybrid)."""
    rp, col, v = pf.synth_csr(family, seed=9, scale_n=size, dtypes=(dtype,))
    m = len(rp) - 1
    d = [dev(a) for a in (rp, col, v[dtype], pf.synth_x(family, m, seed=9, dtypes=(dtype,))[dtype])]
    want = torch.full((m,), float("nan"), dtype=TORCH[dtype], device=DEV)
    pf.spmv(*d, want, m, m, len(col), dtype)
    assert_parity(rp, col, v[dtype], d[3].cpu().numpy(), want.cpu().numpy(), dtype, what=f"{family} {dtype} alone")
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    start, failures = threading.Barrier(len(streams)), []

    def worker(k):
        try:
            y = [torch.full((m,), float("nan"), dtype=TORCH[dtype], device=DEV) for _ in range(6)]
            torch.cuda.synchronize()
            start.wait(timeout=60)
            for out in y:
                pf.spmv(*d, out, m, m, len(col), dtype, "auto", streams[k])
            for it, out in enumerate(y):
                if not torch.equal(out, want):
                    failures.append((k, it, int((out != want).sum())))
        except Exception as e:
            failures.append((k, repr(e)))
            start.abort()

    threads = [threading.Thread(target=worker, args=(k,)) for k in range(len(streams))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not any(t.is_alive() for t in threads) and not failures, failures
