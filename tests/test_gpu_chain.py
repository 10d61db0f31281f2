"""1-D two-band chains (a lane per matrix entry, chain_kernels.hip) against the
CPU oracle: single evaluations to 1e-12 relative, replayed propagations to
1e-10 (the bounds of every other path)."""
import dataclasses

import numpy as np
import pytest

from sbewh_amd import model
from sbewh_amd.propagator import SBEContext
from oracle.oracle_py import Oracle
from tests import cases

pytestmark = pytest.mark.gpu


def chain(reach, nk, nf, seed=1, **kw):
    """chain with hoppings up to `reach` cells"""
    rng = np.random.default_rng(seed)
    cells = np.array([(r, 0, 0) for r in range(-reach, reach + 1)], np.int32)
    H = np.zeros((len(cells), 2, 2), complex)
    D = np.zeros((len(cells), 3, 2, 2), complex)
    for i, r in enumerate(range(-reach, 1)):
        h = 0.03 * np.exp(r / 2) * (rng.normal(size=(2, 2)) + 1j * rng.normal(size=(2, 2)))
        d = np.exp(r / 2) * (rng.normal(size=(2, 2)) + 1j * rng.normal(size=(2, 2)))
        if r == 0:
            h, d = h + h.conj().T + np.diag([-0.06, 0.06]), d + d.conj().T
        H[i], H[-1 - i] = h, h.conj().T
        D[i, 0], D[-1 - i, 0] = d, d.conj().T
    pul = [model.Pulse("sin2", 0.5, 3200.0, 0.3, 0.8)]
    return model.Config("chain", model.TBModel(cells, H, D, np.eye(3) * 5.5), 1, (nk, 1, 1), (nf, 1, 1), pul,
                        **{"T2_fs": 2.0, "sweeps": 8, "output_count": 9, **kw})


def state(o, seed=4):
    x = cases.perturbed_state(o.initial_state(0.0), o.n, o.P, o.num_k, seed=seed, amp=0.05)
    x[1] = 0
    return x


# reaches at and beyond the cells kept in registers (2, 4), beyond 16 cells; k
# counts below, at and beyond a wavefront's 16
@pytest.mark.parametrize("reach,nk,nf", [(1, 3, 3), (2, 5, 5), (3, 16, 8), (4, 18, 9), (5, 24, 12), (8, 72, 18),
                                         (0, 17 * 4, 4)])
@pytest.mark.parametrize("kw", [{}, {"gpu_layout": True, "k_global_shift": (0.31, 0.0, 0.0)}, {"T2_fs": -1.0},
                                {"soothing_width_eV": -1.0}, {"cold_jacobi": True, "sweeps": 1}])
def test_chain_against_oracle(reach, nk, nf, kw):
    cfg = chain(reach, nk, nf, **kw)
    g, o = SBEContext(cfg), Oracle(dataclasses.replace(cfg, gpu_layout=False, sweeps=8))
    x = state(o)
    n, P = o.n, o.P

    def host(v):   # oracle layout -> the context's
        return np.concatenate([v[:8], v[8:].reshape(nk, P)[:, :g.P].reshape(-1)])

    for t in (0.5, -3.0):
        b = host(o.rhs(x, t))
        assert np.abs(g.rhs(host(x), t) - b).max() < 1e-12 * np.abs(b).max()
    assert np.abs(g.observe(host(x)) - o.observe_j(x)).max() < 1e-12 * np.abs(o.observe_j(x)).max()
    xo, xg = x.copy(), host(x)
    ro = o.integrate(xo, cfg.output_count)
    rg = g.integrate(xg, cfg.output_count, replay=ro["log"])
    assert np.abs(rg["j"] - ro["j"]).max() < 1e-10 * np.abs(ro["j"]).max()
    assert np.abs(xg - host(xo)).max() < 1e-10
    assert rg["rhs_calls"] == 6 * len(ro["log"].accepted_dts()) + cfg.output_count - 1
    assert g.stage_tuning()["lanes_per_row"] == 0
    g.close()
    o.close()


def test_chain_decoupled_and_degenerate():
    """no coupling between the bands (no rotation), and equal bands"""
    for split in (0.06, 0.0):
        cfg = chain(2, 10, 5)
        H = cfg.model.H.copy()
        H[:, 0, 1] = H[:, 1, 0] = 0
        H[:, 1, 1] = H[:, 0, 0]
        H[2, 0, 0] -= split
        cfg = dataclasses.replace(cfg, model=dataclasses.replace(cfg.model, H=H))
        g, o = SBEContext(cfg), Oracle(cfg)
        x = state(o)
        b = o.rhs(x, 0.5)
        assert np.abs(g.rhs(x, 0.5) - b).max() < 1e-12 * np.abs(b).max()
        g.close()
        o.close()


def test_chain_own_step_control_and_general_path(monkeypatch):
    """the same steps as the general path's layouts (SBEWH_STAGE_LR forces one)"""
    cfg = chain(4, 32, 16, output_count=17)
    res = []
    for lr in (None, "1", "2"):
        if lr:
            monkeypatch.setenv("SBEWH_STAGE_LR", lr)
        g = SBEContext(cfg)
        x = g.initial_state(0.0)
        r = g.integrate(x, 17)
        res.append((r, x))
        g.close()
    for r, x in res[1:]:
        assert r["steps"] == res[0][0]["steps"] and r["rhs_calls"] == res[0][0]["rhs_calls"]
        assert np.abs(x - res[0][1]).max() < 1e-10


@pytest.mark.parametrize("reach,nk,nf", [(2, 256, 16), (4, 256, 16), (12, 250, 25), (40, 243, 81)])
def test_chain_rounding(reach, nk, nf, monkeypatch):
    """right-hand sides are no further from long double than the general path's (5 % for
    the spread of the mean over 16 states)"""
    cfg = chain(reach, nk, nf, T2_fs=-1.0)
    cfg.model.H[reach] += np.diag([-1.0, 1.0])
    pi = np.longdouble("3.14159265358979323846264338327950288")
    rms = []
    for lr in ("1", None):
        if lr:
            monkeypatch.setenv("SBEWH_STAGE_LR", lr)
        else:
            monkeypatch.delenv("SBEWH_STAGE_LR")
        g = SBEContext(cfg)
        k = g.k_index_map()[:, 0].astype(np.longdouble) / nk
        err = []
        rng = np.random.default_rng(5)
        for A in rng.uniform(-0.5, 0.5, 16):
            x = np.zeros(g.state_size, complex)
            x[0] = A
            rho = cases.random_hermitian(rng, nk, 2, 0.3)
            x[8:].reshape(nk, -1)[:, :4] = rho.reshape(nk, 4)
            a = g.rho(g.rhs(x, 0.3))
            arg = (k + np.longdouble(A) * np.longdouble(5.5) / (2 * pi))[:, None] * cfg.model.cells[:, 0]
            arg = 2 * pi * (arg - np.round(arg))
            op = (cfg.model.H + g.E(0.3)[0] * cfg.model.D[:, 0]).astype(np.clongdouble)
            HE = np.einsum("kr,rab->kab", np.cos(arg) + 1j * np.sin(arg), op)
            ref = -1j * (np.einsum("kab,kbc->kac", HE, rho) - np.einsum("kab,kbc->kac", rho, HE))
            err.append(float(np.sqrt((np.abs(a - ref) ** 2).mean() / (np.abs(ref) ** 2).mean())))
        rms.append(np.mean(err))
        g.close()
    print(f"[gpu] chain reach {reach}: general {rms[0]:.3e}, registers {rms[1]:.3e}", flush=True)
    assert rms[1] <= 1.05 * rms[0]
