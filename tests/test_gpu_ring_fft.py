"""Ring FFTs at the lengths where the kernel that serves them changes, against
the CPU oracle: rings of at most 32 points (summed directly), the other lengths
of the ring kernels, and the wavefront kernels' lengths 512, 1024 and 2048 with
batches on both sides of the count that selects them.
"""
import sys

import numpy as np
import pytest

import gshtrans_amd as G
import oracle

pytestmark = pytest.mark.gpu
SEED0 = 20261206


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def rel(a, b):
    return float(np.linalg.norm(np.ravel(a - b)) / np.linalg.norm(np.ravel(b)))


@pytest.fixture(scope="module")
def torch():
    import torch as _t
    assert _t.cuda.is_available(), "GPU tests need a device"
    return _t


# Short rings: a field that does not depend on longitude has orders m = 0 only.
# Every other bin is a sum of equal samples times roots of unity that cancel in
# pairs, so with exact symmetric roots (2, 4, 8 or 16 points) it is exactly zero;
# a transform through longer ones leaves their rounding in it.
@pytest.mark.parametrize("L", [1, 2, 4, 8])
@pytest.mark.parametrize("real", [False, True])
def test_short_rings_cancel_exactly(torch, L, real):
    say(f"[short rings] L={L} real={real}")
    rng = np.random.default_rng(SEED0 + L)
    ring = rng.standard_normal((3, L + 1, 1))
    if not real:
        ring = ring + 1j * rng.standard_normal(ring.shape)
    f = torch.from_numpy(np.repeat(ring, 2 * L, axis=2)).cuda()
    c = G.GaussLegendreGrid(L, 0).forward(L, 0, f, real=real).cpu().numpy()
    for l in range(L + 1):
        for m in range(0 if real else -l, l + 1):
            if m != 0:
                assert (c[:, G.coefficient_index(L, 0, l, m, real)] == 0.0).all(), (l, m)


# Sums of at most 32 + 17 terms of relative rounding 1.1e-16 each, in norms that
# no cancellation shrinks: below 1e-14.
@pytest.mark.parametrize("L", range(1, 18))
@pytest.mark.parametrize("n,real", [(0, True), (0, False), (1, True), (-1, False)])
def test_short_rings_against_extended_precision(torch, L, n, real):
    say(f"[short rings] L={L} n={n} real={real}")
    g = G.GaussLegendreGrid(L, 1)
    og = oracle.OracleGrid(L, 1, table=False, long_double=True)
    for batch in (1, 9):
        c = G.random_coefficients(L, n, real=real, seed=SEED0 + L, batch=batch)
        f = g.inverse(L, n, torch.from_numpy(c).cuda(), real=real)
        a = g.forward(L, n, f, real=real).cpu().numpy()
        f = f.cpu().numpy()
        for i in (0, batch - 1):
            ref = og.inverse(L, n, c[i], real=real)
            if np.linalg.norm(ref.astype(complex)) > 0:
                assert rel(f[i], ref) <= 1e-14
            ref = og.forward(L, n, f[i], real=real)
            if np.linalg.norm(ref.astype(complex)) > 0:
                assert rel(a[i], ref) <= 1e-14


# The wavefront kernels (512, 1024 and 2048 points, more than 4 fields): partly
# empty field groups (of 4 or 8 rings), odd counts of real fields (two to a ring),
# truncation below the grid, and lmax = N / 2, whose last bin is stored apart.
# FP64 parity as everywhere: 1e-12 of the oracle's norm.  Split BF16 moves FP32
# bins: 2^-24 each and products of bf16x6, against FP64 1e-5.
@pytest.mark.parametrize("L,lmax,n,real,batch", [
    (256, 130, -2, False, 5), (256, 256, 1, False, 9), (256, 70, 2, True, 5),
    (256, 256, 0, True, 17), (512, 512, 1, True, 7), (512, 301, 0, True, 5),
    (512, 512, -1, False, 11), (512, 200, 0, False, 6), (1024, 1024, 0, True, 5),
    (1024, 700, 1, True, 7), (1024, 1024, 2, False, 6), (1024, 515, 0, False, 5)])
def test_wavefront_batches(torch, L, lmax, n, real, batch):
    say(f"[wavefront] L={L} lmax={lmax} n={n} real={real} batch={batch}")
    g = G.GaussLegendreGrid(L, 2)
    og = oracle.OracleGrid(L, 2, table=False)
    c = G.random_coefficients(lmax, n, real=real, seed=SEED0 + L + batch, grid_lmax=L, batch=batch)
    cd = torch.from_numpy(c).cuda()
    f = g.inverse(lmax, n, cd, real=real)
    a = g.forward(lmax, n, f, real=real)
    fh, ah = f.cpu().numpy(), a.cpu().numpy()
    for i in (0, batch - 1):
        assert rel(fh[i], og.inverse(lmax, n, c[i], real=real)) <= 1e-12
        assert rel(ah[i], og.forward(lmax, n, fh[i], real=real)) <= 1e-12
    fm = g.inverse(lmax, n, cd, real=real, precision="bf16x6")
    am = g.forward(lmax, n, f, real=real, precision="bf16x6")
    for x, y in ((fm, f), (am, a)):
        for i in range(batch):
            assert float((x[i] - y[i]).norm() / y[i].norm()) <= 1e-5


# Both families transform the same bins: a batch of more than 4 fields and its
# fields one by one differ by the FFTs' rounding, log2(2048) = 11 levels of
# 1.1e-16, below 1e-14 of a field's norm (not bit for bit at these lengths).
@pytest.mark.parametrize("L", [256, 512, 1024])
@pytest.mark.parametrize("n,real", [(0, True), (2, False)])
def test_batch_against_single_fields(torch, L, n, real):
    say(f"[wavefront] batch against single L={L} n={n} real={real}")
    g = G.GaussLegendreGrid(L, 2)
    c = torch.from_numpy(G.random_coefficients(L, n, real=real, seed=SEED0, batch=9)).cuda()
    f = g.inverse(L, n, c, real=real)
    a = g.forward(L, n, f, real=real)
    for i in range(9):
        one = g.inverse(L, n, c[i:i + 1], real=real)[0]
        assert float((f[i] - one).norm() / one.norm()) <= 1e-14
        one = g.forward(L, n, f[i:i + 1], real=real)[0]
        assert float((a[i] - one).norm() / one.norm()) <= 1e-14


# Plans: the fields of a group in descending degree, so a pair of real fields in
# one ring has two degrees, one of them N / 2, and groups fall on both sides of 4
# fields.  Against the field alone: the FFT's rounding in FP64, FP32 bins (2^-24,
# a plan may choose FP64 ones) in split BF16.
@pytest.mark.parametrize("L", [256, 512, 1024])
@pytest.mark.parametrize("real", [True, False])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-14), ("bf16x6", 1e-6)])
def test_uneven_plans(torch, L, real, precision, tol):
    lmax = [L, L // 2, L, L - 24, 31, L, (7 * L) // 10] + [L, L - 1, 40] + [L]
    n = [0] * 7 + [1] * 3 + [2]
    say(f"[wavefront] uneven plan L={L} real={real} {precision}")
    g = G.GaussLegendreGrid(L, 2)
    plan = G.BatchPlan(g, lmax, n, real=real, precision=precision)
    c = torch.zeros((len(n), plan.cmax), dtype=torch.complex128, device="cuda")
    for i, (lm, k) in enumerate(zip(lmax, n)):
        c[i, :G.coefficient_size(lm, k, real)] = torch.from_numpy(
            G.random_coefficients(lm, k, real=real, seed=SEED0 + i, grid_lmax=L)).cuda()
    f = plan.inverse(c)
    a = plan.forward(f)
    for i, (lm, k) in enumerate(zip(lmax, n)):
        size = G.coefficient_size(lm, k, real)
        one = g.inverse(lm, k, c[i:i + 1, :size].contiguous(), real=real, precision=precision)[0]
        assert float((f[i] - one).norm() / one.norm()) <= tol, i
        one = g.forward(lm, k, f[i:i + 1], real=real, precision=precision)[0]
        assert float((a[i, :size] - one).norm() / one.norm()) <= tol, i


# Few fields with bins in groups of 16 columns (every mode but FP64), on both
# sides of each count at which the FFT family changes, against FP64: FP32 products
# and bins of 2^-24 over sums of at most 1025 terms, below 1e-5.
@pytest.mark.parametrize("L", [256, 512, 1024])
@pytest.mark.parametrize("n,real", [(0, True), (2, False)])
@pytest.mark.parametrize("precision", ["fp32", "bf16x6"])
def test_few_fields_in_wide_bins(torch, L, n, real, precision):
    say(f"[few fields] L={L} n={n} real={real} {precision}")
    g = G.GaussLegendreGrid(L, 2)
    c = torch.from_numpy(G.random_coefficients(L, n, real=real, seed=SEED0, batch=5)).cuda()
    f = g.inverse(L, n, c, real=real)
    a = g.forward(L, n, f, real=real)
    for batch in (1, 2, 3, 4, 5):
        fm = g.inverse(L, n, c[:batch], real=real, precision=precision)
        am = g.forward(L, n, f[:batch], real=real, precision=precision)
        for x, y in ((fm, f), (am, a)):
            for i in range(batch):
                assert float((x[i] - y[i]).norm() / y[i].norm()) <= 1e-5, (batch, i)


# A plan reports the FFT family that its groups run and the tiles of the launch's
# own rule, also where a tuning file says otherwise, and does not take choices
# that a file holds for an earlier generation of the kernels.
def test_plan_reports_what_it_runs(torch, tmp_path, monkeypatch):
    L, degrees = 512, [512, 500, 400]
    lmax = degrees + [512 - 3 * i for i in range(9)] + [512] * 2
    n = [0] * 3 + [1] * 9 + [2] * 2
    cache = tmp_path / "tune.txt"
    monkeypatch.setenv("GSH_TUNE_CACHE", str(cache))
    g = G.GaussLegendreGrid(L, 2)
    # the line of an earlier generation for the group of 3 (FNV-1a of its degrees)
    h = 1469598103934665603
    for l in degrees:
        h = (h ^ l) * 1099511628211 % 2**64
    key = f"L{L}:k{G.COMPLEX}:p{G.PRECISION['fp64']}:s{G.STORAGE['fp64']}:d0:n0:c3:h{h:x}"
    cache.write_text(f"gsh2:{key} 1 1 0\n")

    def run(path):
        monkeypatch.setenv("GSH_TUNE_CACHE", str(path))
        plan = G.BatchPlan(g, lmax, n)
        c = torch.zeros((len(n), plan.cmax), dtype=torch.complex128, device="cuda")
        plan.forward(plan.inverse(c))
        info = {d["n"]: d for d in plan.info()}
        plan.close()
        return info

    first = run(cache)
    lines = [x.split() for x in cache.read_text().splitlines()[1:]]
    say(f"[plan] {first} {lines}")
    assert any(x[0].endswith(":" + key) for x in lines)  # timed, not taken from the old line
    pinned = tmp_path / "pinned.txt"
    pinned.write_text("\n".join(f"{k} {1 if t == '2' else 2} 1 {p}" for k, t, f, p in lines) + "\n")
    second = run(pinned)
    for info in (first, second):
        for k in (0, 2):  # at most 4 fields
            assert info[k]["fft_inverse"] == info[k]["fft_forward"] == 2
    assert second[1]["fft_inverse"] == second[1]["fft_forward"] == 1
    assert {k: d["synth_tiles"] for k, d in second.items()} == \
        {k: d["synth_tiles"] for k, d in first.items()}
