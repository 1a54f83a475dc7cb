"""GPU tests of the transform from the tridiagonal form (k_vec): the inverse
square root by poles, the tiled resolvent sums and the blocked two-sided
product, at the edges of its 16-wide tiles and pole groups.

Tolerance: the reduction to tridiagonal form and the reference's
eigendecomposition are each backward stable, an error of up to k eps |A| in A,
hence up to k eps kappa / 2 relative to the largest entry of T (kappa the ratio
of the largest eigenvalue of M to (k-1)/rho): max(1e-10, k eps kappa) for the
two together, and twice that for overline_w = T T b / (k-1).
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def _case(k, p, scale, seed):
    rng = np.random.default_rng(seed)
    y = scale * rng.standard_normal((k, p)) * np.exp(-0.1 * np.arange(p))[None, :]
    y -= y.mean(axis=0, keepdims=True)
    return (y, (1.0 / rng.uniform(0.5, 2.0, p) ** 2).astype(np.float32), rng.standard_normal(p),
            rng.uniform(0.1, 1.0, p))


def _kappa(c, rho):
    y, rinv, _, rloc = c
    k = y.shape[0]
    return 1.0 + np.linalg.eigvalsh((y * (rinv * rloc)) @ y.T).max() * rho / (k - 1)


# k: 1 and 2 reflectors, the tile edges (one tile, a tile and one row, whole
# tiles), the three kernel widths; scales give kappa from 1 to ~1e9, 8 to ~45
# poles (one to three groups of 16)
@pytest.mark.parametrize("k", [2, 3, 4, 15, 16, 17, 18, 19, 31, 32, 33, 34, 35, 48, 49, 63, 64,
                               65, 66, 80, 81, 96, 113, 127, 128])
def test_transform_edges(k):
    import orc
    from dida_letkf import engine
    rho = 1.13
    cases = [_case(k, p, s, 1000 * k + i) for i, (p, s) in enumerate(
        [(0, 1.0), (1, 1.0), (40, 0.05), (60, 1.0), (60, 30.0), (60, 1e3), (60, 2e4)])]
    args = [[c[i] for c in cases] for i in range(4)]
    t, w, st = engine.letkf_core_batched(*args, inflation_factor=rho)
    assert (st == 0).all()
    old = os.environ.get("DIDA_QL_MAXITER")
    os.environ["DIDA_QL_MAXITER"] = "30"              # the QL recurrence for every analysis
    try:
        tq, wq, sq = engine.letkf_core_batched(*args, inflation_factor=rho)
    finally:
        os.environ.pop("DIDA_QL_MAXITER")
        if old is not None:
            os.environ["DIDA_QL_MAXITER"] = old
    assert (sq == 0).all()
    for i, c in enumerate(cases):
        kap = _kappa(c, rho) if c[0].shape[1] else 1.0
        tol = max(1e-10, k * np.finfo(float).eps * kap)
        t_o, w_o, _ = orc.letkf_core(*c, inflation_factor=rho)
        for tt, ww in ((t[i], w[i]), (tq[i], wq[i])):
            e_t = np.abs(tt - t_o).max() / np.abs(t_o).max()
            e_w = np.abs(ww - w_o).max() / max(1.0, np.abs(w_o).max())
            print(k, i, "kappa %.2g" % kap, e_t, e_w, flush=True)
            assert e_t < tol and e_w < 2 * tol


@pytest.mark.parametrize("k", [20, 40, 100])
def test_weak_and_indefinite(k):
    """Negative R^-1 makes A indefinite.  Where M stays positive definite (its
    smallest eigenvalue far below (k-1)/rho) the first pass still gives the
    transform; where it does not, the list pass's QL takes the matrix, with the
    NaN of the square root of a negative eigenvalue.  (Against numpy's eigh: the
    oracle forms sqrt(R^-1), which is NaN here.)"""
    from dida_letkf import engine
    rng = np.random.default_rng(k)
    y = rng.standard_normal((k, 5))
    y -= y.mean(axis=0, keepdims=True)
    dep, rloc = rng.standard_normal(5), np.ones(5)
    top = np.linalg.eigvalsh(y @ y.T).max()
    cases, want = [], []
    for f in (0.05, 0.2, 0.7, 0.97, 1.5):             # smallest eigenvalue (1 - f) (k-1)
        cases.append((y, np.full(5, -f * (k - 1) / top, np.float32), dep, rloc))
        want.append(f < 1.0)
    t, w, st = engine.letkf_core_batched(*[[c[i] for c in cases] for i in range(4)])
    for i, (yy, rinv, d, _) in enumerate(cases):
        wy = yy * rinv.astype(np.float64)
        lam, v = np.linalg.eigh(wy @ yy.T)
        lam = lam + (k - 1)
        if want[i]:
            w_o = v @ ((v.T @ (wy @ d)) / lam)
            t_o = (v * np.sqrt((k - 1) / lam)) @ v.T + w_o[:, None]
            # kappa / (1 - f) <= 40 here: rounding, amplified 40 times
            assert st[i] == 0
            assert np.abs(t[i] - t_o).max() < 1e-10 * np.abs(t_o).max()
            assert np.abs(w[i] - w_o).max() < 1e-10 * max(1.0, np.abs(w_o).max())
        else:
            assert np.isnan(t[i]).all()


def _failing_case(kind, k, rng):
    y = rng.standard_normal((k, 5))
    y -= y.mean(axis=0, keepdims=True)
    dep, rloc, rinv = rng.standard_normal(5), np.ones(5), np.full(5, 0.5, np.float32)
    if kind == "indefinite":                         # smallest eigenvalue -(k-1)/2
        rinv[:] = -1.5 * (k - 1) / np.linalg.eigvalsh(y @ y.T).max()
    elif kind == "nan":
        y[rng.integers(k), 2] = np.nan
    return y, rinv, dep, rloc


# more failures than any list of them holds (256 per batch, 128 above k = 64)
@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("k,n", [(20, 900), (64, 450), (100, 150)])
def test_many_failures(k, n, noalloc):
    """Good, indefinite and non-finite analyses in turn, after a call of the
    same shape whose transforms are all finite: a non-finite analysis gives a
    nonzero status and NaN outputs, an indefinite one NaN in trans (the square
    root of a negative eigenvalue) and overline_w = M^-1 b, however many there
    are.  Tolerance: a backward error of k eps |M| each for the tridiagonal form
    and for QL, amplified by the condition of M."""
    from dida_letkf import engine
    if noalloc and k == 100:
        n = 144                                      # what the fixed scratch holds
    rng = np.random.default_rng(7 * k)
    kinds = ["good" if i % 9 == 0 else "indefinite" if i % 2 else "nan" for i in range(n)]
    assert sum(x != "good" for x in kinds) > (256 if k <= 64 else 120)
    clean = [_failing_case("good", k, rng) for _ in kinds]
    t, w, st = engine.letkf_core_batched(*[[c[i] for c in clean] for i in range(4)],
                                         noalloc=noalloc)
    assert (st == 0).all() and np.isfinite(t).all() and np.isfinite(w).all()
    cases = [_failing_case(x, k, rng) for x in kinds]
    t, w, st = engine.letkf_core_batched(*[[c[i] for c in cases] for i in range(4)],
                                         noalloc=noalloc)
    for i, (kind, (y, rinv, dep, _)) in enumerate(zip(kinds, cases)):
        if kind == "nan":
            assert st[i] != 0, i
            assert np.isnan(t[i]).all() and np.isnan(w[i]).all(), i
            continue
        assert st[i] == 0, i
        wy = y * rinv.astype(np.float64)
        lam, v = np.linalg.eigh(wy @ y.T)
        lam = lam + (k - 1)
        tol = 2 * k * np.finfo(float).eps * np.abs(lam).max() / np.abs(lam).min()
        w_o = v @ ((v.T @ (wy @ dep)) / lam)
        assert np.abs(w[i] - w_o).max() <= max(tol, 1e-12) * max(1.0, np.abs(w_o).max()), i
        if kind == "indefinite":
            assert np.isnan(t[i]).all(), i
        else:
            t_o = (v * np.sqrt((k - 1) / lam)) @ v.T + w_o[:, None]
            assert np.abs(t[i] - t_o).max() <= max(tol, 1e-12) * np.abs(t_o).max(), i


@pytest.mark.parametrize("k,f32", [(20, False), (64, True), (100, False)])
def test_many_failures_in_a_cycle(k, f32):
    """Three cycles of one handle: good obs, obs whose Yb are NaN (every analysis
    keeps its background and its transforms are NaN), obs of negative R^-1 (the
    NaN of the square root reaches the state and is not counted as a failure,
    as in the reference)."""
    import copy

    import torch
    from dida_letkf import engine, synth
    inst = synth.generate("c0", seed=k, k=k, nlat=16, nlon=30, n_obs=1500, local_dist=900.0)
    cfg = inst.cfg
    dt = torch.float32 if f32 else torch.float64
    dev = torch.device("cuda:0")
    xb = torch.from_numpy(np.ascontiguousarray(inst.xb)).to(dev).to(dt)
    axb = torch.from_numpy(np.ascontiguousarray(inst.axb)).to(dev)
    xa, axa = torch.zeros_like(xb), torch.zeros_like(axb)
    h = cfg.halo
    inner = (slice(h, h + cfg.nlon), slice(h, h + cfg.nlat))
    with engine.LetkfEngine(cfg, keep_transforms=True) as eng:
        eng.set_grid(inst.grid_lat, inst.grid_lon)
        eng.set_stream(torch.cuda.current_stream().cuda_stream)
        run = eng.analyze_device_f32 if f32 else eng.analyze_device

        def cycle(obs):
            eng.set_obs(obs)
            rc = run(xb.data_ptr(), axb.data_ptr(), xa.data_ptr(), axa.data_ptr())
            torch.cuda.synchronize()
            return rc, eng.get_transforms()

        rc, (t, w, nob) = cycle(inst.obs)
        n = t.shape[0]
        assert rc == 0 and np.isfinite(t).all() and n > 256 and (nob > 0).all()
        bad = copy.deepcopy(inst.obs)
        bad.yb[:, 1] = np.nan
        rc, (t, w, _) = cycle(bad)
        assert rc == n and eng.stats.n_flagged == n
        assert np.isnan(t).all() and np.isnan(w).all()
        assert torch.equal(xa[inner], xb[inner]) and torch.equal(axa[inner], axb[inner])
        bad = copy.deepcopy(inst.obs)
        bad.rinv[:] = -1e3 * np.abs(bad.rinv)
        rc, (t, w, _) = cycle(bad)
        assert rc == 0 and np.isnan(t).all() and np.isfinite(w).all()
        assert torch.isnan(xa[inner]).all() and torch.isnan(axa[inner]).all()


@pytest.mark.parametrize("k", [65, 97, 128])
def test_four_wavefronts_same_bits(k):
    """k > 64: the wavefronts of a matrix agree on its poles whatever runs beside
    it.  Matrices of one to five groups of poles, in two orders: the same bits
    for each."""
    from dida_letkf import engine
    cases = [_case(k, 40, 10.0 ** (i % 5), 50 * k + i) for i in range(60)]
    args = [[c[i] for c in cases] for i in range(4)]
    t, w, st = engine.letkf_core_batched(*args)
    tr, wr, sr = engine.letkf_core_batched(*[a[::-1] for a in args])
    assert (st == 0).all() and (sr == 0).all()
    assert np.array_equal(t, tr[::-1]) and np.array_equal(w, wr[::-1])


@pytest.mark.parametrize("rho", [np.inf, 1e308, 1e-300, 5e-324])
@pytest.mark.parametrize("k,precision", [(20, 0), (64, 1), (100, 0)])
def test_inflation_limits(k, precision, rho):
    """(k-1)/rho = 0 (M = A, positive definite here: p > k rows that are not
    centred), next to 0, huge and infinite (trans and overline_w 0): accepted
    by the entry points, so every kernel ends and the result is the formula's.
    Tolerance: k eps cond(A) for the tridiagonal form and the eigensolver
    each, in FP32 the rounding of Yb and its sums, 1e-7, times that condition."""
    from dida_letkf import engine
    rng = np.random.default_rng(k)
    p = 3 * k
    y = rng.standard_normal((k, p))
    rinv, dep, rloc = np.ones(p, np.float32), rng.standard_normal(p), np.ones(p)
    t, w, st = engine.letkf_core_batched([y], [rinv], [dep], [rloc], inflation_factor=rho,
                                         precision=precision)
    assert st[0] == 0
    lam, v = np.linalg.eigh(y @ y.T)
    eps = np.finfo(float).eps if precision == 0 else 1e-7
    tol = 2 * k * eps * lam.max() / lam.min()
    with np.errstate(over="ignore", divide="ignore"):
        lam = lam + np.float64(k - 1) / np.float64(rho)
    w_o = v @ ((v.T @ (y @ dep)) / lam)
    t_o = (v * np.sqrt((k - 1) / lam)) @ v.T + w_o[:, None]
    assert np.abs(w[0] - w_o).max() <= tol * max(np.abs(w_o).max(), 1e-290)
    assert np.abs(t[0] - t_o).max() <= tol * max(np.abs(t_o).max(), 1e-290)


@pytest.mark.parametrize("k", [4, 33, 70])
@pytest.mark.parametrize("top", [1e13, 1e20, 1e60, 1e110])
def test_wide_spectrum(k, top):
    """Obs that each see one member: M is diagonal, its condition from 1e26 to
    1e220, and trans and overline_w have closed forms.  Every term of the pole
    sum is positive and each diagonal entry of the resolvents exact to a few ulp,
    so the entries hold to 1e-13 of themselves (the sum over up to 862 poles
    restated on the CPU: 5e-15)."""
    from dida_letkf import engine
    amp = np.logspace(0, np.log10(top), k - 1)
    y = np.zeros((k, k - 1))
    y[np.arange(k - 1), np.arange(k - 1)] = amp
    dep = np.linspace(1.0, 2.0, k - 1)
    one = np.ones(k - 1)
    t, w, st = engine.letkf_core_batched([y], [one.astype(np.float32)], [dep], [one])
    assert st[0] == 0
    m = np.append(amp ** 2, 0.0) + (k - 1)
    w_o = np.append(amp * dep, 0.0) / m
    assert np.abs(w[0] / np.where(w_o > 0, w_o, 1.0) - (w_o > 0)).max() < 1e-13
    d_o = np.sqrt((k - 1) / m)
    diag = np.diagonal(t[0]) - w[0]
    # taking overline_w off again costs an ulp of it
    assert (np.abs(diag - d_o) <= 1e-13 * d_o + 4e-16 * w_o).all()
