"""The paired-order FP64 kernels (gsh_pair.hip) and the ring FFTs of any length
(gsh_fft_ring.hip) at the edges of their tiles, against the CPU oracle.

Bar: relative L2 <= 1e-12, that of the FP64 parity tests (sums of at most a
few hundred terms of rounding 1.1e-16 each).
"""
import sys

import numpy as np
import pytest

import gshtrans_amd as G
import oracle

pytestmark = pytest.mark.gpu
SEED0 = 20261205


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def rel(a, b):
    return float(np.linalg.norm(np.ravel(a - b)) / np.linalg.norm(np.ravel(b)))


@pytest.fixture(scope="module")
def torch():
    import torch as _t
    assert _t.cuda.is_available(), "GPU tests need a device"
    return _t


def check(torch, L, lmax, n, real, batch):
    say(f"[pair] L={L} lmax={lmax} n={n} real={real} batch={batch}")
    g = G.GaussLegendreGrid(L, min(2, L))
    og = oracle.OracleGrid(L, min(2, L), table=False)
    c = G.random_coefficients(lmax, n, real=real, seed=SEED0 + L + batch, grid_lmax=L, batch=batch)
    f = g.inverse(lmax, n, torch.from_numpy(c).cuda(), real=real)
    a = g.forward(lmax, n, f, real=real)
    fh, ah = f.cpu().numpy(), a.cpu().numpy()
    for i in sorted({0, batch // 2, batch - 1}):  # first, middle and last columns
        ref = og.inverse(lmax, n, c[i], real=real)
        assert rel(fh[i], ref) <= 1e-12, i
        assert rel(ah[i], og.forward(lmax, n, fh[i], real=real)) <= 1e-12, i


# Columns: 2 batch (real) or 4 batch (complex) virtual columns, around the
# tile widths 4, 8, 16, 32, 64 and 128; rows around 16, 96, 112, 128 and 144
# (n = 0: half of them); degrees around the chunks of 32 and passes of 128.
@pytest.mark.parametrize("batch", [1, 2, 3, 4, 5, 8, 9, 16, 17, 33])
@pytest.mark.parametrize("n,real", [(0, True), (0, False), (1, True), (-2, False)])
def test_column_tiles(torch, n, real, batch):
    check(torch, 40, 33, n, real, batch)


@pytest.mark.parametrize("L,lmax", [(15, 15), (16, 16), (95, 64), (111, 96), (127, 127), (128, 128),
                                    (143, 129), (144, 144), (255, 250), (287, 160)])
@pytest.mark.parametrize("n,real,batch", [(0, True, 3), (2, False, 1), (-1, False, 20)])
def test_row_and_degree_tiles(torch, L, lmax, n, real, batch):
    check(torch, L, lmax, n, real, batch)


# Ring lengths 2 L at the edges of each transform length: powers of two (64 ..
# 1024 points), and the shortest and longest that Bluestein's convolution of
# 64 .. 4096 points serves.
@pytest.mark.parametrize("L", [17, 18, 31, 32, 33, 63, 64, 65, 128, 129, 255, 256, 257, 511, 512,
                               513])
@pytest.mark.parametrize("real", [False, True])
def test_ring_lengths(torch, L, real):
    check(torch, L, min(L, 40), 0 if real else 1, real, 2)
    check(torch, L, L, 0 if real else -1, real, 1)


@pytest.mark.parametrize("n,real", [(0, True), (0, False), (2, False), (1, True)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_left_out_terms_stay_visible(torch, n, real, bad):
    """Near the poles the high orders' values are negligible and their terms
    are left out; an Inf or NaN among them still makes the field (the
    coefficients) it belongs to non-finite, and no other field of the batch."""
    L = 300
    g = G.GaussLegendreGrid(L, 2)
    c = torch.from_numpy(G.random_coefficients(L, n, real=real, seed=SEED0, batch=3)).cuda()
    f = g.inverse(L, n, c, real=real)
    a = g.forward(L, n, f, real=real)
    say(f"[pair] non-finite n={n} real={real} {bad}")
    c[1, G.coefficient_index(L, n, 150, 149, real)] = bad
    g.inverse(L, n, c, field=f, real=real)
    finite = torch.isfinite(torch.view_as_real(f) if f.is_complex() else f).reshape(3, -1)
    assert finite[0].all() and finite[2].all() and not finite[1].any()
    f = torch.nan_to_num(f, nan=1.0, posinf=1.0, neginf=1.0)
    f[1, 1, 5] = bad  # a sample next to the pole
    g.forward(L, n, f, coeffs=a, real=real)
    finite = torch.isfinite(torch.view_as_real(a)).reshape(3, -1, 2)
    assert finite[0].all() and finite[2].all()
    # (L, L) of a complex field is zeroed
    assert not finite[1, :-1].all(dim=-1).any()


# The split-BF16 kernels leave whole blocks of 128 rows x 64 degrees (synthesis)
# and pairs of 32 rows x 64 degrees (analysis) out, so a larger grid; the sums
# kept against FP64: FP32-accurate products and bins, 2^-24 each, 1e-5 for
# bf16x6 and 2^-16 products, 1e-3 for bf16x3.
@pytest.mark.parametrize("n,real", [(0, True), (0, False), (2, False)])
@pytest.mark.parametrize("precision,tol", [("bf16x6", 1e-5), ("bf16x3", 1e-3)])
@pytest.mark.parametrize("L,lmax", [(1000, 1000), (767, 700)])
def test_left_out_split_blocks(torch, L, lmax, n, real, precision, tol):
    say(f"[pair] split L={L} lmax={lmax} n={n} real={real} {precision}")
    g = G.GaussLegendreGrid(L, 2)
    c = torch.from_numpy(G.random_coefficients(lmax, n, real=real, seed=SEED0, grid_lmax=L,
                                               batch=3)).cuda()
    f = g.inverse(lmax, n, c, real=real)
    a = g.forward(lmax, n, f, real=real)
    fp = g.inverse(lmax, n, c, real=real, precision=precision)
    ap = g.forward(lmax, n, f, real=real, precision=precision)
    for x, y in ((fp, f), (ap, a)):
        assert float((x - y).norm() / y.norm()) <= tol
    c[1, G.coefficient_index(lmax, n, lmax - 100, lmax - 105, real)] = float("nan")
    g.inverse(lmax, n, c, field=fp, real=real, precision=precision)
    finite = torch.isfinite(torch.view_as_real(fp) if fp.is_complex() else fp).reshape(3, -1)
    assert finite[0].all() and finite[2].all() and not finite[1].any()
    for row in (1, -2):  # a sample next to either pole
        h = f.clone()
        h[1, row, 5] = float("inf")
        g.forward(lmax, n, h, coeffs=ap, real=real, precision=precision)
        finite = torch.isfinite(torch.view_as_real(ap)).reshape(3, -1, 2)
        assert finite[0].all() and finite[2].all()
        assert not finite[1, :-1].all(dim=-1).any()


# Degrees after an order's last stored state: the order L - 12 rises from
# negligible seeds to 2^-83 at rows near the pole within its last 13 degrees.
# One field for each such ring, zero elsewhere, so its sums hold nothing larger.
# FP64: 13 recurrence steps of a few roundings each and one ring FFT, far below
# 1e-10.  Split BF16: FP32-accurate products of FP32 bins (6e-8), their smallest
# planes above FP32's underflow for values from 2^-92: 1e-5.
@pytest.mark.parametrize("precision", ["fp64", "bf16x6"])
@pytest.mark.parametrize("n", [0, 2])
def test_last_degrees_of_an_order(torch, n, precision):
    L, m = 256, 244
    g = G.GaussLegendreGrid(L, 2)
    og = oracle.OracleGrid(L, 2, table=False)
    idx = [G.coefficient_index(L, n, l, m, False) for l in range(m, L + 1)]
    c = np.zeros(G.coefficient_size(L, n), dtype=np.complex128)
    c[idx] = 1.0
    ring = og.inverse(L, n, c)
    size = np.abs(ring).max(axis=-1)
    rows = np.flatnonzero((size > 2.0**-92) & (size < 2.0**-83))
    say(f"[pair] last degrees n={n} {precision} rows={rows}")
    assert rows.size
    f = np.zeros((rows.size,) + ring.shape, dtype=np.complex128)
    f[np.arange(rows.size), rows] = ring[rows] / size[rows, None]
    a = g.forward(L, n, torch.from_numpy(f).cuda(), precision=precision).cpu().numpy()
    tol = 1e-10 if precision == "fp64" else 1e-5
    for i, t in enumerate(rows):
        ref = og.forward(L, n, f[i])[idx]
        assert np.linalg.norm(a[i][idx] - ref) <= tol * np.linalg.norm(ref), t


# The analysis allocates its coefficients without a fill: every one is written,
# at odd sizes, truncations and column counts, in every mode.
@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x3", "bf16x6"])
@pytest.mark.parametrize("n,real", [(0, True), (0, False), (2, False), (-1, True)])
def test_every_coefficient_is_written(torch, n, real, precision):
    for L, lmax, batch in ((2, 2, 1), (3, 2, 3), (40, 33, 17), (129, 128, 5), (300, 300, 2),
                           (300, 190, 40)):
        say(f"[pair] written L={L} lmax={lmax} n={n} real={real} B={batch} {precision}")
        g = G.GaussLegendreGrid(L, 2)
        size = G.coefficient_size(lmax, n, real)
        c = torch.from_numpy(G.random_coefficients(lmax, n, real=real, seed=SEED0, grid_lmax=L,
                                                   batch=batch)).cuda()
        f = g.inverse(lmax, n, c, real=real, precision=precision)
        out = torch.full((batch, size), float("nan"), dtype=torch.complex128, device="cuda")
        g.forward(lmax, n, f, coeffs=out, real=real, precision=precision)
        assert torch.isfinite(torch.view_as_real(out)).all()
        assert torch.equal(g.forward(lmax, n, f, real=real, precision=precision), out)
        out.fill_(float("nan"))
        g.forward_product(lmax, n, f, torch.ones_like(f), coeffs=out, real=real,
                          precision=precision)
        assert torch.isfinite(torch.view_as_real(out)).all()


# Values below 2^-120 near the poles count as zero by rows and degrees alone, so
# one high order by itself, whose values are that small at many rows, gives the
# same bits alone, in batches of every tile shape and in plans of uneven degrees.
# Against the oracle: 1e-12 of the field, and at each row 1e-12 of the sum of the
# terms' absolute values (alternating terms cancel at a mirror row) and 2^-120
# for each of at most 301 unit coefficients left out.
@pytest.mark.parametrize("n,real", [(0, True), (0, False), (1, True), (2, False)])
def test_one_high_order_in_any_tile(torch, n, real):
    L = 300
    orders = [100 + 6 * i for i in range(33)]
    g = G.GaussLegendreGrid(L, 2)
    og = oracle.OracleGrid(L, 2, table=False)
    c = np.zeros((len(orders), G.coefficient_size(L, n, real)), dtype=np.complex128)
    for i, m in enumerate(orders):
        c[i, [G.coefficient_index(L, n, l, m, real) for l in range(m, L + 1)]] = 1.0
    cd = torch.from_numpy(c).cuda()
    one = torch.cat([g.inverse(L, n, cd[i:i + 1], real=real) for i in range(len(orders))])
    # samples on the rows near the poles alone, where the order is small
    polar = one.clone()
    size = polar.abs().amax(dim=-1, keepdim=True)
    polar = torch.where((size > 0) & (size < 2.0**-90), polar / size.clamp_min(2.0**-1000), 0 * polar)
    back = torch.cat([g.forward(L, n, polar[i:i + 1], real=real) for i in range(len(orders))])
    for batch in (2, 3, 4, 5, 8, 9, 16, 17, 33):
        say(f"[pair] one order n={n} real={real} batch={batch}")
        for i in range(0, len(orders) - batch + 1, batch):
            f = g.inverse(L, n, cd[i:i + batch], real=real)
            assert torch.equal(f, one[i:i + batch]), batch
            a = g.forward(L, n, polar[i:i + batch], real=real)
            assert torch.equal(a, back[i:i + batch]), batch
    lmax = [L] + [L - 7 * (i % 8) for i in range(1, 33)]
    plan = G.BatchPlan(g, lmax, [n] * 33, real=real)
    co = torch.zeros((33, plan.cmax), dtype=torch.complex128, device="cuda")
    single = []
    for i, lm in enumerate(lmax):
        size = G.coefficient_size(lm, n, real)
        co[i, :size] = cd[i, :size]
        single.append(g.inverse(lm, n, co[i:i + 1, :size].contiguous(), real=real))
    f = plan.inverse(co)
    a = plan.forward(polar)
    for i, lm in enumerate(lmax):
        size = G.coefficient_size(lm, n, real)
        assert torch.equal(f[i], single[i][0]), i
        assert torch.equal(a[i, :size], g.forward(lm, n, polar[i:i + 1], real=real)[0]), i
    f = one.cpu().numpy()
    th = og.nodes()[0]
    for i in (0, 16, 32):
        ref = og.inverse(L, n, c[i], real=real)
        assert rel(f[i], ref) <= 1e-12
        if real:  # its rings are transformed in pairs, which rounds to the larger of two
            continue
        idx = [oracle.gsh_index(L, L, n, l, orders[i]) for l in range(orders[i], L + 1)]
        terms = [np.abs(oracle.wigner_block(L, L, n, t)[idx]).sum() for t in th]
        err = np.abs(f[i] - ref).max(axis=1)
        assert (err <= 301 * 2.0**-120 + 1e-12 * np.array(terms)).all()


# A program warms up at one batch size and captures another into a graph: the
# work list of the new shape is made during the capture, and every replay gives
# the eager result, with eager work between.
@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x6"])
@pytest.mark.parametrize("warm,batch", [(8, 3), (3, 40)])
def test_first_call_at_a_batch_size_can_be_captured(torch, warm, batch, precision):
    L, n, real = 160, 0, True
    say(f"[pair] capture batch {batch} after {warm} {precision}")
    g, eager = G.GaussLegendreGrid(L, 2), G.GaussLegendreGrid(L, 2)

    def coeffs(seed, b, n=n, real=real):
        return torch.from_numpy(G.random_coefficients(L, n, real=real, seed=seed, batch=b)).cuda()

    # complex fields of another upper index size the scratch arrays for either batch
    for b, k, r in ((max(warm, batch), 1, False), (warm, n, real)):
        f = g.inverse(L, k, coeffs(SEED0, b, k, r), real=r, precision=precision)
        g.forward(L, k, f, real=r, precision=precision)
    c = coeffs(SEED0 + 1, batch)
    f = torch.zeros((batch, L + 1, 2 * L), dtype=torch.float64, device="cuda")
    a = torch.zeros_like(c)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g.inverse(L, n, c, field=f, real=real, precision=precision)
        g.forward(L, n, f, coeffs=a, real=real, precision=precision)
    for rep in range(3):
        c.copy_(coeffs(SEED0 + 2 + rep, batch))
        graph.replay()
        torch.cuda.synchronize()
        fe = eager.inverse(L, n, c, real=real, precision=precision)
        assert torch.equal(f, fe), rep
        assert torch.equal(a, eager.forward(L, n, fe, real=real, precision=precision)), rep
        torch.cuda.synchronize()


# Analysis tiles chosen for their padding columns: 48 and 80 columns (17 .. 24 and
# 33 .. 40 real fields) in tiles of 16, 96 of few workgroups in tiles of 32.
@pytest.mark.parametrize("L,n,real,batch", [(256, 1, True, 24), (130, 0, True, 40), (256, 2, False, 20),
                                            (256, 0, False, 24), (300, -1, False, 24)])
def test_lean_analysis_tiles(torch, L, n, real, batch):
    check(torch, L, L, n, real, batch)


# Synthesis tiles of launches with workgroups enough for 32 and 64 columns: rows of
# 19 and 20 tiles of 16 (blocks of 6, 7 and 8 tiles), 32 columns (full, and 80 and 96
# in groups of 32), 64 columns (40 to 64 of them used, one to three groups); FP32 with
# groups of 32, 64 and 128.  A field of a batch has the bits that it has alone.
@pytest.mark.parametrize("L", [288, 303, 304])
@pytest.mark.parametrize("n,real,batch", [(1, True, 16), (1, True, 20), (-2, False, 20), (2, True, 45),
                                          (1, False, 32), (-1, False, 45)])
def test_synthesis_tiles(torch, L, n, real, batch):
    check(torch, L, L, n, real, batch)
    g = G.GaussLegendreGrid(L, 2)
    c = torch.from_numpy(G.random_coefficients(L, n, real=real, seed=SEED0 + L, grid_lmax=L,
                                               batch=batch)).cuda()
    f = g.inverse(L, n, c, real=real)
    s = g.inverse(L, n, c, real=real, precision="fp32")
    for i in (0, batch // 2, batch - 1):
        one = c[i:i + 1].contiguous()
        assert torch.equal(f[i:i + 1], g.inverse(L, n, one, real=real)), i
        assert torch.equal(s[i:i + 1], g.inverse(L, n, one, real=real, precision="fp32")), i
        assert rel(s[i].cpu().numpy(), f[i].cpu().numpy()) <= 3e-6, i


# Analysis tiles past 128 columns: 144 and 160 in groups of 32, 176 and 192 in groups
# of 64, 256 in groups of 128.
@pytest.mark.parametrize("n,real,batch", [(1, True, 72), (-2, False, 40), (0, False, 36), (1, False, 48),
                                          (0, True, 88), (2, False, 64)])
def test_wide_analysis_tiles(torch, n, real, batch):
    check(torch, 260, 260, n, real, batch)


# A prepared upper index has every table that depends on it alone: what a first call
# still allocates is its work lists and, growing with the call, the grid's bins.
@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x6"])
def test_prepare_builds_the_checkpoints(torch, precision):
    L = 512
    g = G.GaussLegendreGrid(L, 1)
    before = torch.cuda.mem_get_info()[0]
    g.prepare(1)
    table = before - torch.cuda.mem_get_info()[0]
    # 16-byte states at L + 1 colatitudes every 16 degrees of the orders m >= 0
    states = sum(max(0, (L - max(m, 1)) // 16) for m in range(L + 1))
    assert table >= 16 * (L + 1) * states
    c = torch.from_numpy(G.random_coefficients(L, 1, seed=SEED0, batch=1)).cuda()
    f = g.inverse(L, 1, c, precision=precision)
    g2 = G.GaussLegendreGrid(L, 1)  # not prepared
    assert torch.equal(f, g2.inverse(L, 1, c, precision=precision))
    assert torch.equal(g.forward(L, 1, f, precision=precision), g2.forward(L, 1, f, precision=precision))


# FP32 synthesis of at most 16 columns in blocks of 16 and 17 row tiles (lMax=1024: 65
# tiles, the last block with the extra one; lMax=900, where the last block is short),
# to the bits of the same fields in a wider batch, whose tiles are others.
@pytest.mark.parametrize("L,lmax,n,real", [(1023, 1023, 0, True), (1000, 1000, 2, False),
                                           (900, 900, -1, True), (1023, 899, 1, False)])
def test_fp32_synthesis_of_tall_blocks(torch, L, lmax, n, real):
    say(f"[tall] L={L} lmax={lmax} n={n} real={real}")
    g = G.GaussLegendreGrid(L, 2)
    few = 8 if real else 4
    c = torch.from_numpy(G.random_coefficients(lmax, n, real=real, seed=SEED0 + L, grid_lmax=L,
                                               batch=few + 1)).cuda()
    wide = g.inverse(lmax, n, c, real=real, precision="fp32")
    assert torch.equal(g.inverse(lmax, n, c[:few].contiguous(), real=real, precision="fp32"), wide[:few])
    assert torch.equal(g.inverse(lmax, n, c[:1].contiguous(), real=real, precision="fp32"), wide[:1])
    exact = g.inverse(lmax, n, c, real=real)
    for i in (0, few):
        assert rel(wide[i].cpu().numpy(), exact[i].cpu().numpy()) <= 3e-6, i


# The checkpoints of orders m < 0 are built by the first call that reads them: FP64
# holds half a table, and what other modes compute does not depend on the order in
# which the two halves came.
@pytest.mark.parametrize("n,mode", [(0, "bf16x6"), (0, "fp32"), (1, "fp32"), (-2, "bf16x3")])
def test_checkpoints_of_negative_orders(torch, n, mode):
    L = 400
    def both(g, precision):
        f = g.inverse(L, n, c, precision=precision)
        return f, g.forward(L, n, f, precision=precision)
    c = torch.from_numpy(G.random_coefficients(L, n, seed=SEED0, batch=2)).cuda()
    states = 16 * (L + 1) * sum(max(0, (L - max(m, abs(n))) // 16) for m in range(L + 1))
    g = G.GaussLegendreGrid(L, 2)
    before = torch.cuda.mem_get_info()[0]
    g.prepare(n)
    # seeds and recurrence coefficients: 20 and 32 bytes for each of (2 L + 1)(L + 1) and
    # about L^2 + 64 (2 L + 1) entries, and allocation granules
    others = 20 * (2 * L + 1) * (L + 1) + 32 * (L * L + 66 * (2 * L + 1)) + (16 << 20)
    assert before - torch.cuda.mem_get_info()[0] <= states + others
    first = both(g, "fp64")
    second = both(g, mode)
    for x, y in zip(both(g, "fp64"), first):
        assert torch.equal(x, y)
    g2 = G.GaussLegendreGrid(L, 2)
    for x, y in zip(both(g2, mode), second):
        assert torch.equal(x, y)
    for x, y in zip(both(g2, "fp64"), first):
        assert torch.equal(x, y)
    og = oracle.OracleGrid(L, 2, table=False)
    tol = {"fp32": 3e-6, "bf16x6": 1e-7, "bf16x3": 3e-5}[mode]
    assert rel(second[0][1].cpu().numpy(), og.inverse(L, n, c[1].cpu().numpy(), real=False)) <= tol


# Grids made, used and closed by several threads at once share the stream that builds
# their tables; the results are those of a grid alone.
def test_grids_of_several_threads(torch):
    import threading
    cases = [(16, 1, False), (33, 0, True), (64, 2, False), (47, -1, True)]
    coeffs = [torch.from_numpy(G.random_coefficients(L, n, real=real, seed=SEED0 + L, batch=2)).cuda()
              for L, n, real in cases]

    def use(k):
        L, n, real = cases[k]
        g = G.GaussLegendreGrid(L, 2)
        f = g.inverse(L, n, coeffs[k], real=real)
        a = g.forward(L, n, f, real=real)
        torch.cuda.synchronize()
        g.close()
        return f, a

    alone = [use(k) for k in range(len(cases))]
    got, errors = {}, []

    def work(k):
        try:
            for rep in range(4):
                got[k, rep] = use((k + rep) % len(cases))
        except Exception as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for (k, rep), (f, a) in got.items():
        assert torch.equal(f, alone[(k + rep) % len(cases)][0]), (k, rep)
        assert torch.equal(a, alone[(k + rep) % len(cases)][1]), (k, rep)
