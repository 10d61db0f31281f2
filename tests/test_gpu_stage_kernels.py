"""The stage kernel at the edges of its phase-sum and eigenvector paths,
against the CPU oracle.  Tolerance: 1e-12 relative, as for every single
kernel (FP64, sums of at most a few hundred products of order one)."""
import dataclasses

import numpy as np
import pytest

from sbewh_amd import model
from sbewh_amd.propagator import SBEContext
from sbewh_amd.scan import Scan
from oracle.oracle_py import Oracle
from tests import cases

pytestmark = pytest.mark.gpu


def small_model(n, ext, seed, copies=1):
    """Gaussian blocks on the box |R_d| <= ext[d]; copies > 1: every band
    `copies`-fold degenerate at every k (h x 1)"""
    rng = np.random.default_rng(seed)
    m = n // copies
    cells = np.array([(a, b, 0) for a in range(-ext[0], ext[0] + 1) for b in range(-ext[1], ext[1] + 1)], np.int32)
    H = np.zeros((len(cells), n, n), complex)
    D = np.zeros((len(cells), 3, n, n), complex)
    one = np.eye(copies)
    for i, c in enumerate(cells.tolist()):
        j = len(cells) - 1 - i
        if j < i:
            continue
        f = np.exp(-np.hypot(*c[:2]))
        h = f * 0.1 * (rng.normal(size=(m, m)) + 1j * rng.normal(size=(m, m)))
        r = f * (rng.normal(size=(2, n, n)) + 1j * rng.normal(size=(2, n, n)))
        if i == j:
            h = h + h.conj().T + np.diag(np.linspace(-0.4, 0.4, m))
            r = r + np.conj(np.swapaxes(r, 1, 2))
        H[i], H[j] = np.kron(h, one), np.kron(h, one).conj().T
        D[i, :2], D[j, :2] = r, np.conj(np.swapaxes(r, 1, 2))
    return model.TBModel(cells, H, D, np.eye(3) * 6.0)


def config(n, ext, Nk, Nf, seed=5, copies=1, **kw):
    pul = model.elliptic_sin2(1.0, 0.4, 3000.0, 4.0)
    kw = {"sweeps": 12, "T2_fs": 1.0, **kw}
    return model.Config("edge", small_model(n, ext, seed, copies), 2, (*Nk, 1), (*Nf, 1), pul, **kw)


def states(o, count, steps):
    """states of the same rho with the vector potential moved by `steps`"""
    x = cases.perturbed_state(o.initial_state(0.0), o.n, o.P, o.num_k, seed=3, amp=0.05)
    out, A = [], 0.3
    for q in range(count):
        s = x.copy()
        A += steps[q]
        s[0], s[1] = A, -0.4 * A
        out.append(s)
    return out


def check_sequence(cfg, steps, ctx=None):
    g, o = ctx or SBEContext(cfg), Oracle(cfg)
    for q, x in enumerate(states(o, len(steps), steps)):
        t = 3.0 + 0.1 * q
        a, b = g.rhs(x, t), o.rhs(x, t)
        err = np.abs(a - b).max() / np.abs(b).max()
        print(f"[gpu] n={cfg.model.num_wann} step {steps[q]:g}: {err:.1e}", flush=True)
        assert err < 1e-12
    o.close()


# (bands, lanes per row, R extents, k-grid, Fourier block): wavefronts whose
# k-points lie in one, two and more rows of the phase sum, a last wavefront
# that is not full, R extents below, at and beyond one memory trip and the
# 16-cell limit, padded bands
@pytest.mark.parametrize("n,lr,ext,Nk,Nf", [
    (8, 1, (1, 0), (6, 1), (3, 1)),
    (8, 1, (1, 1), (6, 9), (3, 3)),
    (8, 1, (1, 2), (5, 10), (5, 5)),
    (8, 1, (2, 7), (5, 15), (5, 15)),
    (8, 1, (1, 8), (3, 18), (3, 18)),
    (5, 1, (1, 3), (4, 8), (4, 8)),
    (8, 2, (1, 2), (5, 15), (5, 5)),
    (8, 4, (1, 4), (5, 9), (5, 9)),
    (7, 4, (1, 1), (6, 3), (3, 3)),
    (16, 2, (1, 3), (3, 8), (3, 8)),
    (16, 4, (1, 4), (3, 9), (3, 9)),
    (16, 4, (1, 8), (3, 18), (3, 18)),
    (11, 4, (1, 0), (6, 1), (3, 1)),
])
def test_phase_rows(n, lr, ext, Nk, Nf, monkeypatch):
    monkeypatch.setenv("SBEWH_STAGE_LR", str(lr))
    check_sequence(config(n, ext, Nk, Nf), [0.0, 0.01])


# the warm start after steps of A from rounding to a jump across the zone
STEPS = [0.0, 0.0, 1e-13, 1e-9, 1e-6, 1e-4, -2e-3, 0.02, -0.1, 0.6, 0.0, 2e-3]


@pytest.mark.parametrize("n,copies", [(9, 1), (11, 1), (16, 1), (16, 2), (12, 4)])
def test_warm_start_steps(n, copies, monkeypatch):
    """16-band kernels: warm starts refined by products, and those left to
    the rotations (large steps, near crossings), also with every band
    degenerate"""
    monkeypatch.setenv("SBEWH_STAGE_LR", "4")
    check_sequence(config(n, (2, 2), (6, 5), (6, 5), copies=copies), STEPS)


@pytest.mark.parametrize("n", [13, 14, 15])
def test_warm_start_steps_padded(n, monkeypatch):
    """the same with the last bands of 16 as padding"""
    monkeypatch.setenv("SBEWH_STAGE_LR", "4")
    check_sequence(config(n, (2, 2), (6, 5), (6, 5)), STEPS)


def test_warm_start_without_sweeps(monkeypatch):
    """no sweep allowed: a warm call keeps the previous eigenvectors in every layout"""
    cfg = config(16, (1, 1), (3, 4), (3, 4), sweeps=0)
    out = []
    for lr in ("2", "4"):
        monkeypatch.setenv("SBEWH_STAGE_LR", lr)
        g, o = SBEContext(cfg), Oracle(dataclasses.replace(cfg, sweeps=12))
        out.append([g.rhs(x, 3.0) for x in states(o, 2, [0.0, 0.05])])
        o.close()
    for a, b in zip(*out):
        assert np.abs(a - b).max() / np.abs(b).max() < 1e-12


def test_warm_start_long_chain(monkeypatch):
    """400 warm starts one after the other leave the decomposition unitary
    and converged (the last call agrees with the oracle as the first does)"""
    monkeypatch.setenv("SBEWH_STAGE_LR", "4")
    cfg = config(16, (2, 2), (6, 5), (6, 5))
    g, o = SBEContext(cfg), Oracle(cfg)
    x = states(o, 1, [0.0])[0]
    for q in range(400):
        x[0] += 0.004 * np.cos(0.1 * q)
        a = g.rhs(x, 3.0)
    b = o.rhs(x, 3.0)
    o.close()
    assert np.abs(a - b).max() / np.abs(b).max() < 1e-12


@pytest.mark.parametrize("sweeps", [1, 2])
@pytest.mark.parametrize("n,lr,rotations", [(8, 2, 1), (6, 2, 4), (16, 4, 2), (11, 4, 2), (14, 4, 2)])
def test_warm_chain_small_sweep_bounds(n, lr, rotations, sweeps, monkeypatch):
    """1500 warm starts under a small sweep bound: the decomposition stays unitary (the
    dephasing term then has no trace) and is as good as the rotations' with that bound"""
    cfg = config(n, (2, 2), (6, 5), (6, 5), sweeps=sweeps)
    o = Oracle(dataclasses.replace(cfg, sweeps=12))
    err = []
    for layout in (rotations, lr):
        monkeypatch.setenv("SBEWH_STAGE_LR", str(layout))
        g = SBEContext(cfg)
        x = states(o, 1, [0.0])[0]
        for q in range(1500):
            x[0] += 0.004 * np.cos(0.1 * q)
            a = g.rhs(x, 3.0)
        g.close()
        b = o.rhs(x, 3.0)
        tr = np.trace(a[8:].reshape(o.num_k, o.P)[:, :n * n].reshape(-1, n, n), axis1=1, axis2=2)
        err.append(np.abs(a - b).max() / np.abs(b).max())
        print(f"[gpu] n={n} lanes {layout} sweeps {sweeps}: trace {np.abs(tr).max():.1e} error {err[-1]:.1e}", flush=True)
        assert np.abs(tr).max() < 1e-12 * np.abs(b).max()
    assert err[1] <= max(1e-12, 2 * err[0])
    o.close()


# the grid leaves the last of the four-k wavefronts with two k-points
@pytest.mark.parametrize("n,copies", [(5, 1), (7, 1), (8, 1), (6, 2), (8, 2), (8, 4)])
def test_warm_start_steps_8_bands(n, copies, monkeypatch):
    monkeypatch.setenv("SBEWH_STAGE_LR", "2")
    check_sequence(config(n, (2, 2), (6, 5), (6, 5), copies=copies), STEPS)


@pytest.mark.parametrize("n,ext,Nk,Nf", [
    (8, (1, 0), (6, 1), (3, 1)), (8, (1, 1), (6, 9), (3, 3)), (8, (2, 7), (5, 15), (5, 15)),
    (8, (1, 8), (3, 18), (3, 18)), (5, (1, 3), (4, 8), (4, 8)), (8, (1, 0), (3, 1), (3, 1))])
def test_phase_rows_8_bands(n, ext, Nk, Nf, monkeypatch):
    monkeypatch.setenv("SBEWH_STAGE_LR", "2")
    check_sequence(config(n, ext, Nk, Nf), [0.0, 0.01])


def test_layout_rule():
    """warm calls of 8 and 16 bands take the layouts refined by products, calls
    that start from the identity the fastest timed one"""
    for n, lr in ((8, 2), (11, 4)):
        cfg = config(n, (1, 1), (3, 4), (3, 4))
        for cold in (False, True):
            g = SBEContext(dataclasses.replace(cfg, cold_jacobi=cold))
            o = Oracle(cfg)
            g.rhs(states(o, 1, [0.0])[0], 3.0)
            o.close()
            t = g.stage_tuning()
            assert t["lanes_per_row"] == lr if not cold else len(t["timed"]) > 1


# 5 to 8 bands take a k-point per wavefront up to 1024 k-points and four above (the
# last wavefront with two on 42 x 25 k)
@pytest.mark.parametrize("n,copies,Nk,Nf", [
    (8, 1, (32, 32), (4, 4)), (5, 1, (41, 25), (1, 5)), (8, 1, (42, 25), (6, 5)), (6, 2, (42, 25), (6, 5)),
    (7, 1, (1, 1), (1, 1))])
def test_k_points_per_wavefront_8_bands(n, copies, Nk, Nf):
    ext = (min(1, (Nf[0] - 1) // 2), min(1, (Nf[1] - 1) // 2))
    check_sequence(config(n, ext, Nk, Nf, copies=copies), STEPS)


@pytest.mark.parametrize("n,Nk,Nf", [(8, (4, 5), (4, 5)), (6, (32, 32), (4, 4)), (8, (42, 25), (6, 5)), (12, (4, 5), (4, 5)),
                                      (9, (4, 5), (4, 5))])
def test_attempt_in_one_launch(n, Nk, Nf):
    """a propagation whose attempts are one launch each replays the oracle's steps"""
    cfg = dataclasses.replace(config(n, (1, 1), Nk, Nf, eps_rel=1e-7, T2_fs=10.0, output_count=5),
                              pulses=model.elliptic_sin2(1.0, 0.4, 3000.0, 0.1))
    g, o = SBEContext(cfg), Oracle(cfg)
    a = o.initial_state(0.0)
    b = a.copy()
    ro = o.integrate(a, cfg.output_count)
    rg = g.integrate(b, cfg.output_count, replay=ro["log"])
    assert np.abs(rg["j"] - ro["j"]).max() < 1e-10 * np.abs(ro["j"]).max()
    assert np.abs(b - a).max() < 1e-10 * np.abs(a).max()
    o.close()
    g.close()


@pytest.mark.parametrize("Nk,Nf", [((4, 5), (4, 5)), ((42, 25), (6, 5))])
def test_no_dephasing_8_bands(Nk, Nf, monkeypatch):
    monkeypatch.setenv("SBEWH_STAGE_LR", "2")
    check_sequence(config(7, (1, 1), Nk, Nf, T2_fs=0.0), [0.0, 0.01])


@pytest.mark.parametrize("Nk", [(30, 30), (42, 30)])   # one and four k-points per wavefront
def test_commutator_rounding_8_bands(Nk, monkeypatch):
    """the matrix instructions' commutator is no further from one in long double than that
    of the kernel at four lanes per row, which sums its two products apart (5 % for the
    spread of the mean over some 60000 entries)"""
    cfg = config(8, (2, 2), Nk, (6, 6), T2_fs=0.0)
    cfg.model.H[len(cfg.model.cells) // 2] += np.diag([-1.0] * 4 + [1.0] * 4)
    rms = []
    for lr in ("4", "2"):
        monkeypatch.setenv("SBEWH_STAGE_LR", lr)
        g = SBEContext(cfg)
        x = cases.perturbed_state(g.initial_state(0.0), 8, g.P, g.num_k, seed=3, amp=0.05)
        H = g.hk_mesh(x[:3].real, g.E(3.0))[:, 1].astype(np.clongdouble)
        rho = g.rho(x).astype(np.clongdouble)
        ref = -1j * (np.einsum("kab,kbc->kac", H, rho) - np.einsum("kab,kbc->kac", rho, H))
        err = np.abs(g.rho(g.rhs(x, 3.0)) - ref)
        rms.append(float(np.sqrt((err ** 2).mean() / (np.abs(ref) ** 2).mean())))
        g.close()
    print(f"[gpu] commutator {Nk}: four lanes {rms[0]:.3e}, matrix instructions {rms[1]:.3e}", flush=True)
    assert rms[1] <= 1.05 * rms[0]


@pytest.mark.parametrize("n", [9, 12])
def test_scan_9_to_12_bands(n):
    """two pulses in a scan against single runs: the same kernels and steps"""
    base = dataclasses.replace(config(n, (1, 1), (4, 5), (4, 5), eps_rel=1e-7, T2_fs=10.0, output_count=4),
                               pulses=model.elliptic_sin2(1.0, 0.4, 3000.0, 0.1))
    half = n // 2   # a gap between the halves
    base.model.H[len(base.model.cells) // 2] += np.diag(np.where(np.arange(n) < half, -2.0, 2.0))
    base = dataclasses.replace(base, occupied_bands=half)
    cfgs = [base, dataclasses.replace(base, Nk=(8, 10, 1))]
    r = Scan(cfgs).run(4)
    for i, cfg in enumerate(cfgs):
        g = SBEContext(cfg)
        x = g.initial_state(g.fermi_level(cfg.occupied_bands))
        s = g.integrate(x, 4)
        assert r["steps"][i] == s["steps"]
        assert np.abs(r["j"][i] - s["j"]).max() <= 1e-12 * np.abs(s["j"]).max()
        g.close()


@pytest.mark.parametrize("n", [9, 13, 16])
def test_from_the_identity_16_bands(n, monkeypatch):
    """decompositions by rotations alone at four lanes per row: single right-hand sides,
    attempts in one launch and batched ones"""
    monkeypatch.setenv("SBEWH_STAGE_LR", "4")
    cfg = dataclasses.replace(config(n, (1, 1), (5, 4), (5, 4), eps_rel=1e-7, T2_fs=10.0, output_count=4, cold_jacobi=True),
                              pulses=model.elliptic_sin2(1.0, 0.4, 3000.0, 0.1))
    half = n // 2   # a gap between the halves
    cfg.model.H[len(cfg.model.cells) // 2] += np.diag(np.where(np.arange(n) < half, -2.0, 2.0))
    cfg = dataclasses.replace(cfg, occupied_bands=half)
    check_sequence(cfg, [0.0, 0.01, 0.6])
    g, o = SBEContext(cfg), Oracle(cfg)
    a = o.initial_state(o.fermi_level(half))
    b, c = a.copy(), a.copy()
    ro = o.integrate(a, 4)
    rg = g.integrate(b, 4, replay=ro["log"])
    assert np.abs(rg["j"] - ro["j"]).max() < 1e-10 * np.abs(ro["j"]).max()
    assert np.abs(b - a).max() < 1e-10 * np.abs(a).max()
    s, r = g.integrate(c, 4), Scan([cfg, dataclasses.replace(cfg, Nk=(10, 8, 1))]).run(4)
    assert r["steps"][0] == s["steps"]
    assert np.abs(r["j"][0] - s["j"]).max() <= 1e-10 * np.abs(s["j"]).max()
    o.close()
    g.close()
