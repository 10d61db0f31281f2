"""The attempt's error norm at its edges, on every path that forms one: a NaN
ends the integration with SBE_ERR_STEP, and an entry that is zero throughout
has no error, also without an absolute bound."""
import dataclasses

import numpy as np
import pytest

from sbewh_amd import model
from sbewh_amd._lib import SbeError
from sbewh_amd.propagator import SBEContext
from sbewh_amd.scan import Scan
from tests import cases
from tests.test_gpu_chain import chain
from tests.test_gpu_stage_kernels import config

pytestmark = pytest.mark.gpu

NANS = {"quiet": np.array(np.nan), "all bits": np.frombuffer(b"\xff" * 8, np.float64)}


def grid(n, Nk, **kw):
    return dataclasses.replace(config(n, (1, 1), Nk, (3, 3), **kw), pulses=model.elliptic_sin2(1.0, 0.4, 3000.0, 0.2))


def line(n, device):
    """a 1-D model of n bands"""
    cfg = config(n, (1, 0), (64, 1), (4, 1), output_count=5)
    return dataclasses.replace(cfg, dim=1, Nk=(64, 1, 1), Nf=(4, 1, 1), device_controller=device)


# the chain's own kernel and its general layouts, attempts in one launch, in
# one launch per stage, and on the device's step control
CASES = {
    "chain": (lambda: chain(2, 40, 5), None), "chain general": (lambda: chain(2, 40, 5), "1"),
    "chain device": (lambda: chain(2, 40, 5, device_controller=True), None),
    "chain device, one lane": (lambda: chain(2, 40, 5, device_controller=True), "1"),
    "3 bands device": (lambda: line(3, True), None), "8 bands device": (lambda: line(8, True), None),
    "3 bands": (lambda: grid(3, (6, 9)), "1"),
    "8 bands, one k per wavefront": (lambda: grid(8, (6, 9)), None),
    "8 bands, launch per stage": (lambda: grid(8, (51, 51)), None),
    "8 bands, one lane": (lambda: grid(8, (6, 9)), "1"),
    "8 bands, four lanes": (lambda: grid(8, (6, 9)), "4"),
    "11 bands": (lambda: grid(11, (6, 9)), None),
    "16 bands, two lanes": (lambda: grid(16, (6, 9)), "2"),
    "16 bands, launch per stage": (lambda: grid(16, (24, 24)), None),
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("nan", NANS)
def test_nan_state_is_refused(name, nan, monkeypatch):
    make, lr = CASES[name]
    if lr:
        monkeypatch.setenv("SBEWH_STAGE_LR", lr)
    cfg = make()
    print(f"[gpu] {name}: NaN state ({nan})", flush=True)
    g = SBEContext(cfg)
    x0 = g.initial_state(0.0)
    for where in (g.state_size - g.P, 8):       # the last and the first k-point
        x = x0.copy()
        x.view(np.float64)[2 * where] = NANS[nan].item()
        with pytest.raises(SbeError, match="-3"):
            g.integrate(x, 5, log_capacity=0)
    # the context works on afterwards
    x = x0.copy()
    r = g.integrate(x, 5, log_capacity=0)
    assert r["device_controller"] == cfg.device_controller
    assert r["steps"] > 0 and np.isfinite(x).all()
    g.close()


def test_nan_instance_of_a_scan():
    """the instance with a NaN field stops, the other goes on"""
    good = dataclasses.replace(cases.small_square(Nk=(15, 15, 1), cycles=0.2), output_count=4)
    bad = dataclasses.replace(good, pulses=[dataclasses.replace(p, Emax_V_nm=np.nan) for p in good.pulses])
    alone = Scan([good]).run(4)
    r = Scan([bad, good]).run(4)
    assert r["steps"][0] == -3 and r["steps"][1] == alone["steps"][0]
    assert np.abs(r["j"][1] - alone["j"][0]).max() <= 1e-10 * np.abs(alone["j"][0]).max()


@pytest.mark.parametrize("name", ["chain", "chain general", "chain device, one lane", "3 bands", "8 bands, one k per wavefront",
                                  "11 bands", "16 bands, launch per stage"])
def test_relative_bound_alone(name, monkeypatch):
    """eps_abs 0: the slots that stay zero count for nothing, as under a tiny bound (the same bits: no
    layout found by timing)"""
    make, lr = CASES[name]
    if lr:
        monkeypatch.setenv("SBEWH_STAGE_LR", lr)
    out = []
    for eps_abs in (0.0, 1e-290):
        cfg = dataclasses.replace(make(), eps_abs=eps_abs)
        g = SBEContext(cfg)
        x = g.initial_state(0.0)
        x[:cfg.dim] = [0.2, -0.1][:cfg.dim]
        x[8:] += 0.1    # no entry near zero but the unused slots
        out.append((g.integrate(x, 5, log_capacity=0)["steps"], x))
        g.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
