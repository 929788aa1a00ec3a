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
