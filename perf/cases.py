"""Performance cases of the propagation path, over the range it is used in.

Five kinds of work, each through the package's public entry points:

* ``rhs``        the right-hand side on device buffers (``SBEContext.rhs_device``),
                 four evaluations per pass at the stages of a fixed Runge-Kutta
                 step: what a program with an integrator of its own calls
* ``integrate``  a whole ``SBEContext.integrate`` (state on the host, output
                 times, adaptive steps on the device), over the whole pulse or
                 a segment of it
* ``observe``    the full observer at output times (regions, occupations,
                 density matrices) on a device state
* ``scan``       a batched scan of many pulses over one model (``Scan.run``)
* ``surrogate``  one batch through the ensemble of the learned surrogate,
                 forward (``mode`` "forward") or with its gradient ("gradient")

Models are seeded tight-binding models with the statistics of the package's
benchmark configurations (Gaussian blocks decaying with |R|, an onsite split
that keeps a band gap), so every number of bands, R extent and k-grid can be
asked for.  torch is imported before the package: the library then binds to
the HIP runtime torch has loaded, and torch's device memory and streams are
valid in its device-buffer entry points.
"""
import functools
import math

import numpy as np
import torch

from sbewh_amd import model

# Hartree atomic units
FS, ANGSTROM, V_NM, EV, KELVIN = 2.4188843266049513e-2, 5.291772109060855e-1, 514.22067475617267, \
    27.211386245771678, 315775.0248015561
LIGHT = 137.035999177

LATTICE_A = {1: 3.0, 2: 3.0, 3: 4.0}      # lattice constant in angstrom by dimension
DECAY = {1: 1.5, 2: 2.0, 3: 1.5}          # decay length of the blocks in lattice constants
SIGMA_EV = {1: 0.5, 2: 0.8, 3: 0.8}       # block scale in eV
T2_FS, WIDTH_EV, TEMP_K = 10.0, 0.025, 300.0
EPS_ABS, EPS_REL = 1e-12, 1e-8
LAMBDA_NM, FIELD_V_NM = 3000.0, 1.0
DIMS = (6, 256, 256, 256, 40)             # the surrogate's layers
MEMBERS = 5


def listed():
    return [
        # the smallest grid: a 1-D two-band chain (9 cells, 256 k), where launches count
        {"name": "rhs chain", "kind": "rhs", "dim": 1, "bands": 2, "ext": 4, "nf": 16, "rep": 16},
        # the 2-D 8-band benchmark model (169 cells, 150 x 150 k)
        {"name": "rhs square", "kind": "rhs", "dim": 2, "bands": 8, "ext": 6, "nf": 15, "rep": 10},
        # the 3-D 16-band benchmark model (729 cells, 48^3 k): the largest grid
        {"name": "rhs cubic", "kind": "rhs", "dim": 3, "bands": 16, "ext": 4, "nf": 12, "rep": 4},
        # odd sizes: 11 bands, a ragged grid, a shifted zone, the unpadded state layout
        {"name": "rhs ragged", "kind": "rhs", "dim": 2, "bands": 11, "ext": 3, "nf": 9, "rep": 7, "gpu_layout": True,
         "shift": 0.13},
        # the chain's whole pulse with 1024 outputs: a short attempt thousands of times
        {"name": "integrate chain", "kind": "integrate", "dim": 1, "bands": 2, "ext": 4, "nf": 16, "rep": 16,
         "cycles": 8.0, "outputs": 1024},
        # the surrogate's grid (8 bands, 15 x 15 k): a segment with a typical output spacing
        {"name": "integrate square 15", "kind": "integrate", "dim": 2, "bands": 8, "ext": 6, "nf": 15, "rep": 1,
         "attempts": 60, "outputs": 6},
        # the 2-D benchmark grid, a segment around the pulse's peak
        {"name": "integrate square 150", "kind": "integrate", "dim": 2, "bands": 8, "ext": 6, "nf": 15, "rep": 10,
         "attempts": 90, "outputs": 8},
        # 16 bands on 24^3 k, a segment around the pulse's peak
        {"name": "integrate cubic 24", "kind": "integrate", "dim": 3, "bands": 16, "ext": 4, "nf": 12, "rep": 2,
         "attempts": 60, "outputs": 6},
        # full observer, 16 bands on 24^3 k: the zone and a moving region, smeared occupations, density matrices
        {"name": "observe cubic 24", "kind": "observe", "dim": 3, "bands": 16, "ext": 4, "nf": 12, "rep": 2,
         "records": 4, "density": True},
        # many pulses over one model on mixed grids, 8 bands
        {"name": "scan square", "kind": "scan", "dim": 2, "bands": 8, "ext": 6, "nf": 15, "rep": 1, "rep2": 4,
         "pulses": 24, "attempts": 24, "outputs": 4},
        # the surrogate: a large query batch, and a training batch with its gradient
        {"name": "surrogate forward", "kind": "surrogate", "mode": "forward", "rows": 4096},
        {"name": "surrogate gradient", "kind": "surrogate", "mode": "gradient", "rows": 256},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _smooth(lo, hi):
    """5-smooth numbers in [lo, hi]: the Fourier block sizes"""
    out = []
    for n in range(lo, hi + 1):
        r = n
        for p in (2, 3, 5):
            while r % p == 0:
                r //= p
        if r == 1:
            out.append(n)
    return out


def _draw_grid(rng, most):
    """bands, R extent and a k-grid with at most `most` entries k x bands^2"""
    dim = rng.choice((1, 2, 3))
    bands = rng.randint(1, 16)
    ext = rng.randint(1, {1: 7, 2: 6, 3: 4}[dim])
    nf = rng.choice(_smooth(2 * ext + 1, 2 * ext + 8))
    top = max(1.0, (min(most / bands ** 2, 160000)) ** (1 / dim) / nf)
    rep = max(1, int(_log_uniform(rng, 1, top)))
    if rep > 1 and (nf * rep) ** dim * bands ** 2 > most:
        rep -= 1
    return {"dim": dim, "bands": bands, "ext": ext, "nf": nf, "rep": rep}


def draw(rng):
    kind = rng.choice(("rhs", "rhs", "integrate", "integrate", "observe", "scan", "surrogate"))
    if kind == "surrogate":
        return {"kind": kind, "mode": rng.choice(("forward", "gradient")), "rows": int(_log_uniform(rng, 1, 4096))}
    if kind == "rhs":
        c = _draw_grid(rng, 48 ** 3 * 256)
        return dict(c, kind=kind, gpu_layout=rng.random() < 0.3, shift=rng.choice((0.0, round(rng.random(), 3))))
    if kind == "integrate":
        c = _draw_grid(rng, 24 ** 3 * 256)
        return dict(c, kind=kind, attempts=rng.randint(12, 60), outputs=rng.randint(2, 9),
                    gpu_layout=rng.random() < 0.3, device=c["dim"] == 1 and c["bands"] <= 8 and rng.random() < 0.5)
    if kind == "observe":
        c = _draw_grid(rng, 24 ** 3 * 256)
        return dict(c, kind=kind, records=rng.randint(1, 4), density=rng.random() < 0.5)
    c = _draw_grid(rng, 60 * 60 * 64)
    return dict(c, kind=kind, bands=max(2, c["bands"]), rep2=c["rep"] + rng.randint(0, 1), pulses=rng.randint(2, 16),
                attempts=rng.randint(8, 24), outputs=rng.randint(2, 4))


# ---- the model, the pulse and the states of a case ---------------------------
def _cells(case):
    r = range(-case["ext"], case["ext"] + 1)
    z = (0,)
    return np.array([(a, b, c) for a in r for b in (r if case["dim"] > 1 else z)
                     for c in (r if case["dim"] > 2 else z)], np.int32)


def _spread(case):
    """half the width of the bands before the split, from the blocks' variance (hartree)"""
    dim = case["dim"]
    R = np.linalg.norm(_cells(case), axis=1)
    s2 = np.sum((SIGMA_EV[dim] / EV * np.exp(-R / DECAY[dim])) ** 2)
    return 2 * math.sqrt(s2 * case["bands"])


def _step_size(case):
    """about the step the error control takes: the bands span some four times _spread"""
    return 0.1 / (4 * _spread(case))


def _occupied(case):
    return max(1, case["bands"] // 2)


@functools.lru_cache(maxsize=4)
def _model(dim, bands, ext, seed):
    """H(R), r(R) with H(-R) = H(R)^dagger; lower half of the orbitals split from the upper half"""
    case = {"dim": dim, "bands": bands, "ext": ext}
    rng = np.random.default_rng(seed)
    cells = _cells(case)
    n, N = bands, len(cells)
    f = np.exp(-np.linalg.norm(cells, axis=1) / DECAY[dim])
    g = lambda *s: (rng.normal(size=s) + 1j * rng.normal(size=s)) / math.sqrt(2)  # noqa: E731
    H = SIGMA_EV[dim] / EV * f[:, None, None] * g(N, n, n)
    D = 1.0 / ANGSTROM * f[:, None, None, None] * g(N, 3, n, n)
    D[:, dim:] = 0
    half = N // 2      # the cells are in lexicographic order: R at i, -R at N - 1 - i
    H[half + 1:] = np.conj(np.swapaxes(H[:half][::-1], 1, 2))
    D[half + 1:] = np.conj(np.swapaxes(D[:half][::-1], 2, 3))
    H[half] = 0.5 * (H[half] + H[half].conj().T)
    D[half] = 0.5 * (D[half] + np.conj(np.swapaxes(D[half], 1, 2)))
    if n > 1:
        occ = _occupied(case)
        H[half] += np.diag([-0.5] * occ + [0.5] * (n - occ)) * (2.0 if n > 3 else 3.0) * _spread(case)
    lat = np.eye(3) * (LATTICE_A[dim] / ANGSTROM)
    return model.TBModel(cells, H, D, lat)


def _omega():
    return 2 * math.pi * LIGHT / (10 * LAMBDA_NM / ANGSTROM)


def _pulse(case, seed, index=0):
    """(field V/nm, cep, fwhm fs, half window in fwhm): the whole pulse, or a segment around its
    peak that takes about `attempts` step attempts (a step resolves the largest level spacing)"""
    rng = np.random.default_rng((seed, 77, index))
    cycles = case.get("cycles", 8.0)
    fwhm = 0.5 * cycles * 2 * math.pi / _omega()      # a.u.; window +- fwhm
    half = 1.0
    if "attempts" in case:
        step = _step_size(case)
        half = 0.5 * case["attempts"] * step / fwhm
    return FIELD_V_NM * rng.uniform(0.5, 1.2), rng.uniform(0, 2 * math.pi), fwhm * FS, half


def _config(case, seed, index=0, rep=None):
    E0, cep, fwhm, half = _pulse(case, seed, index)
    dim, nf, rep = case["dim"], case["nf"], rep or case["rep"]
    grid = lambda v: tuple(v if d < dim else 1 for d in range(3))  # noqa: E731
    pul = [model.Pulse("sin2", E0, LAMBDA_NM, cep, fwhm, t_start=-half, t_end=half)]
    return model.Config("case", _model(dim, case["bands"], case["ext"], seed), dim, grid(nf * rep), grid(nf), pul,
                        T2_fs=T2_FS, soothing_width_eV=WIDTH_EV, temperature_K=TEMP_K, eps_abs=EPS_ABS,
                        eps_rel=EPS_REL, occupied_bands=_occupied(case), output_count=case.get("outputs", 2),
                        k_global_shift=(case.get("shift", 0.0), 0.0, 0.0),
                        gpu_layout=bool(case.get("gpu_layout")), device_controller=bool(case.get("device")))


def _num_k(case, rep=None):
    return (case["nf"] * (rep or case["rep"])) ** case["dim"]


def _stride(case):
    nn = case["bands"] ** 2
    return nn if case.get("gpu_layout") else 8 * ((nn + 7) // 8)


STAGES = (0.0, 0.5, 0.5, 1.0)    # nodes of the classical fourth-order Runge-Kutta step


def _step(case):
    """(t, h): a step near the pulse's peak"""
    return 3.0, _step_size(case)


def _states(case, seed, count, device):
    """`count` device states as a propagation holds them: lower orbitals filled, coherences of a
    few percent, the vector potential of the stage in the special slots"""
    n, nk, P = case["bands"], _num_k(case), _stride(case)
    gen = torch.Generator(device=device).manual_seed(seed)
    t, h = _step(case)
    E = _field(case, seed, t)
    occ = torch.zeros(n, dtype=torch.float64, device=device)
    occ[:_occupied(case)] = 1.0
    out = []
    base = None
    for q in range(count):
        re = torch.randn(nk, n, n, dtype=torch.float64, device=device, generator=gen)
        im = torch.randn(nk, n, n, dtype=torch.float64, device=device, generator=gen)
        z = torch.complex(re, im) * (0.02 if base is None else 0.001)
        z = 0.5 * (z + z.conj().transpose(1, 2))
        rho = z + torch.diag(occ) if base is None else base + z
        base = rho if base is None else base
        s = torch.zeros(8 + P * nk, dtype=torch.complex128, device=device)
        s[8:].view(nk, P)[:, :n * n] = rho.reshape(nk, n * n)
        for d in range(case["dim"]):
            s[d] = 0.2 - 0.1 * d - STAGES[q % 4] * h * E[d]
        out.append(s)
    return out


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


_stream = None


def _user_stream():
    """the program's own stream: all its calls are enqueued there in order"""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def prepare(case, seed):
    if case["kind"] == "surrogate":
        from sbewh_amd.surrogate import MLPEnsemble
        x, t, w = _surrogate_data(case, seed)
        ens = MLPEnsemble(DIMS, MEMBERS)
        for e in range(MEMBERS):
            ens.set_params(e, w[e])
        return {"case": case, "ens": ens, "x": x, "t": t}
    if case["kind"] == "scan":
        from sbewh_amd.scan import Scan
        reps = [case["rep2"] if i % 2 else case["rep"] for i in range(case["pulses"])]
        return {"case": case, "scan": Scan([_config(case, seed, i, r) for i, r in enumerate(reps)])}
    from sbewh_amd.propagator import WHOLE_ZONE, FullObserver, Region, SBEContext
    ctx = SBEContext(_config(case, seed))
    st = {"case": case, "ctx": ctx}
    if case["kind"] == "integrate":
        st["x0"] = ctx.initial_state(0.0)
        st["x"] = np.empty_like(st["x0"])
    else:
        st["in"] = _states(case, seed, 4 if case["kind"] == "rhs" else case["records"], _device())
        st["stream"] = _user_stream().cuda_stream
        t, h = _step(case)
        st["t"] = [t + STAGES[q % 4] * h for q in range(len(st["in"]))]
    if case["kind"] == "rhs":
        st["out"] = [torch.empty_like(s) for s in st["in"]]
    if case["kind"] == "observe":
        st["obs"] = FullObserver(ctx, (WHOLE_ZONE, Region(_centre(case), 0.3, True)),
                                 smearing_width=_smearing(), density_stride=2 if case["density"] else 0, capacity=8)
    return st


def _centre(case):
    return tuple(0.2 if d < case["dim"] else 0.0 for d in range(3))


def _smearing():
    return 0.1 / EV


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "rhs":
        for x, y, t in zip(state["in"], state["out"], state["t"]):
            state["ctx"].rhs_device(x.data_ptr(), y.data_ptr(), t, state["stream"])
        return state["out"]
    if kind == "integrate":
        np.copyto(state["x"], state["x0"])
        r = state["ctx"].integrate(state["x"], case["outputs"], log_capacity=0)
        return {"t": r["t"], "j": r["j"], "state": state["x"]}
    if kind == "observe":
        from sbewh_amd._lib import check, load
        obs = state["obs"]
        obs.reset()
        for x, t in zip(state["in"], state["t"]):
            check(load().sbe_observer_record_device(obs.h, x.data_ptr(), t, None), state["ctx"].h)
        r = obs.collectExpectationValues()
        del r["tDensIndices"]
        return r
    if kind == "scan":
        r = state["scan"].run(case["outputs"])
        return {"t": r["t"], "j": r["j"]}
    if case["mode"] == "forward":
        return state["ens"].forward(state["x"])
    return state["ens"].gradient(state["x"], state["t"])


# ---- what a pass cannot do without -------------------------------------------
def _rhs_work(case, nk):
    """bytes and operations of one right-hand side: rho read and its derivative written once; the
    commutator and the two basis changes (six complex products), an eigen-decomposition (about
    36 n^3), and the phase sum along one axis"""
    n, W = case["bands"], 2 * case["ext"] + 1
    flops = 48 * n ** 3 + 36 * n ** 3 + 16 * W * n * n
    return {"bytes": 32.0 * n * n * nk, "flops": float(flops * nk)}


def work(case):
    kind = case["kind"]
    if kind == "surrogate":
        rows, P = case["rows"], sum(a * b + b for a, b in zip(DIMS, DIMS[1:]))
        W = sum(a * b for a, b in zip(DIMS, DIMS[1:]))
        back = 2 if case["mode"] == "gradient" else 0
        return {"bytes": float(4 * rows * (DIMS[0] + MEMBERS * DIMS[-1]) + MEMBERS * P * (4 if back else 2)),
                "flops": float(2 * MEMBERS * rows * W * (1 + back))}
    if kind == "rhs":
        w = _rhs_work(case, _num_k(case))
        return {k: 4 * v for k, v in w.items()}
    if kind == "observe":
        n, nk, dim = case["bands"], _num_k(case), case["dim"]
        ops = 8 * n ** 3 * 3 + 36 * n ** 3 + 8 * (1 + 2 * dim) * n * n * (2 * case["ext"] + 2)
        return {"bytes": 16.0 * n * n * nk * case["records"], "flops": float(ops * nk * case["records"])}
    # right-hand sides of an integration: six per attempt and one per output interval
    attempts = case["attempts"] if "attempts" in case else 2200
    rhs = 6 * attempts + case["outputs"]
    nks = [_num_k(case)]
    if kind == "scan":
        nks = [_num_k(case, case["rep2"] if i % 2 else case["rep"]) for i in range(case["pulses"])]
    w = _rhs_work(case, sum(nks))
    return {k: rhs * v for k, v in w.items()}


# ---- the same results from plain numpy ----------------------------------------
def _field(case, seed, t):
    E0, cep, fwhm, half = _pulse(case, seed)
    w, F = _omega(), fwhm / FS
    if t < -F or t > F:
        return np.zeros(3)
    b = math.pi / 2 / F
    c, s = math.cos(b * t), math.sin(b * t)
    return np.array([E0 / V_NM * (math.cos(w * t + cep) * c * c - 2 * b / w * math.sin(w * t + cep) * c * s), 0, 0])


def _k_grid(case):
    """(nk, 3) grid indices of the state's k order: blocks of nf^dim points, the index of a point
    inside its block times the number of blocks per axis, plus the block's own index"""
    dim, nf, rep = case["dim"], case["nf"], case["rep"]
    Nf = [nf if d < dim else 1 for d in range(3)]
    Nr = [rep if d < dim else 1 for d in range(3)]
    blk = np.stack(np.meshgrid(*[np.arange(v) for v in Nr], indexing="ij"), -1).reshape(-1, 1, 3)
    pts = np.stack(np.meshgrid(*[np.arange(v) for v in Nf], indexing="ij"), -1).reshape(1, -1, 3)
    return (pts * np.array(Nr) + blk).reshape(-1, 3)


class _Plain:
    """H(k + A), r(k + A) and dH/dk(k + A) by direct sums over R, and the equations of motion"""

    def __init__(self, case, seed, device="cpu"):
        self.case, self.seed, self.dim, self.n = case, seed, case["dim"], case["bands"]
        m = _model(case["dim"], case["bands"], case["ext"], seed)
        nk = case["nf"] * case["rep"]
        self.k = _k_grid(case) / np.array([nk if d < self.dim else 1 for d in range(3)])
        self.k[:, 0] += case.get("shift", 0.0)
        self.cells, self.lat = m.cells.astype(float), m.lattice
        pos = self.cells @ self.lat
        to = lambda a: torch.from_numpy(np.ascontiguousarray(a.reshape(len(m.cells), -1))).to(device)  # noqa: E731
        self.H = to(m.H)
        self.D = [to(m.D[:, d]) for d in range(self.dim)]
        self.dH = [to(1j * pos[:, d, None, None] * m.H) for d in range(self.dim)]
        self.device = device
        self.F2, self.w = 1 / (T2_FS / FS), WIDTH_EV / EV

    def phases(self, A):
        """exp(i 2 pi (k + A) . R) for every k and cell"""
        k = self.k + self.lat @ np.asarray(A, float) / (2 * math.pi)
        arg = torch.from_numpy(k).to(self.device) @ torch.from_numpy(self.cells.T.copy()).to(self.device)
        arg = arg - arg.round()
        return torch.complex(torch.cos(2 * math.pi * arg), torch.sin(2 * math.pi * arg))

    def mesh(self, ph, X):
        return (ph @ X).cpu().numpy().reshape(-1, self.n, self.n)

    def rhs(self, A, rho, t):
        E = _field(self.case, self.seed, t)
        ph = self.phases(A)
        H0 = self.mesh(ph, self.H)
        HE = H0 + sum(E[d] * self.mesh(ph, self.D[d]) for d in range(self.dim) if E[d] != 0)
        e, V = np.linalg.eigh(H0)
        Vh = np.conj(np.swapaxes(V, 1, 2))
        gam = -self.F2 * -np.expm1(-((e[:, :, None] - e[:, None, :]) / self.w) ** 2)
        out = -1j * (HE @ rho - rho @ HE) + V @ (gam * (Vh @ rho @ V)) @ Vh
        return -E, out

    def current(self, A, rho):
        ph = self.phases(A)
        H0 = self.mesh(ph, self.H)
        T = H0 @ rho - rho @ H0
        j = np.zeros((len(rho), 3))
        for d in range(self.dim):
            D, dH = self.mesh(ph, self.D[d]), self.mesh(ph, self.dH[d])
            j[:, d] = np.real(1j * np.einsum("kab,kba->k", D, T) - np.einsum("kab,kba->k", dH, rho))
        return j

    def ground(self):
        """Fermi-Dirac state of H0(k) at chemical potential 0"""
        e, V = np.linalg.eigh(self.mesh(self.phases(np.zeros(3)), self.H))
        f = 1 / (1 + np.exp(np.minimum(e / (TEMP_K / KELVIN), 700.0)))
        return (V * f[:, None, :]) @ np.conj(np.swapaxes(V, 1, 2))


def _pack(case, A, rho):
    n, P = case["bands"], _stride(case)
    out = np.zeros(8 + P * len(rho), complex)
    out[:3] = A
    out[8:].reshape(len(rho), P)[:, :n * n] = rho.reshape(len(rho), n * n)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "surrogate":
        return _surrogate_exact(case, seed)
    if kind == "scan":
        return None
    n, nk = case["bands"], _num_k(case)
    eig_s = nk * (1.5e-6 + 0.3e-6 * n * n)     # about what numpy's decompositions of one evaluation take
    if kind == "integrate":
        attempts = case["attempts"] if "attempts" in case else 2200
        if (6 * attempts + case["outputs"]) * (eig_s + 2e-4) > 16:
            return None
        return _integrate_exact(case, seed)
    dev = _device()
    p = _Plain(case, seed, dev)
    st = _states(case, seed, 4 if kind == "rhs" else case["records"], dev)
    t0, h = _step(case)
    if kind == "rhs":
        out = [None] * 4
        for q in range(4 if eig_s < 3 else 1):
            A, rho = _unpack(case, st[q])
            out[q] = torch.from_numpy(_pack(case, *p.rhs(A, rho, t0 + STAGES[q] * h)))
        return out
    return _observe_exact(case, seed, p, st, [t0 + STAGES[q % 4] * h for q in range(case["records"])])


def _unpack(case, s):
    n, P, s = case["bands"], _stride(case), s.cpu().numpy()
    return s[:3].real.copy(), np.ascontiguousarray(s[8:].reshape(-1, P)[:, :n * n]).reshape(-1, n, n)


def _observe_exact(case, seed, p, states, times):
    n, dim, smear = case["bands"], case["dim"], _smearing()
    out = {k: [] for k in ("t", "E", "A", "kPointWeightSum", "j", "occupationHam", "occupationWan",
                           "occupationHamMin", "occupationHamMax", "wan")}
    for i, (s, t) in enumerate(zip(states, times)):
        A, rho = _unpack(case, s)
        e, V = np.linalg.eigh(p.mesh(p.phases(A), p.H))
        o = np.real(np.einsum("kab,kac,kcb->kb", np.conj(V), rho, V, optimize=True))
        g = np.exp(-((e[:, :, None] - e[:, None, :]) / smear) ** 2)
        o = (g * o[:, None, :]).sum(2) / g.sum(2)
        w = np.ones((2, len(rho)))
        c = p.k - np.array(_centre(case))      # moving frame: + A - A
        c -= np.round(c)
        w[1] = np.exp(-(c[:, :dim] ** 2).sum(1) * 8 * math.log(2) / 0.3 ** 2)
        ws = w.sum(1)
        avg = lambda q: np.tensordot(w, q, 1) / ws.reshape((2,) + (1,) * (q.ndim - 1))  # noqa: E731
        row = {"t": t, "E": _field(case, seed, t), "A": A, "kPointWeightSum": ws, "j": avg(p.current(A, rho)),
               "occupationHam": avg(o), "occupationWan": avg(np.real(np.einsum("kaa->ka", rho))),
               "occupationHamMin": o.min(0), "occupationHamMax": o.max(0)}
        for k, v in row.items():
            out[k].append(v)
        if case["density"] and i % 2 == 0:
            out["wan"].append(avg(rho))
    r = {k: np.array(v, float) for k, v in out.items() if k != "wan"}
    r["wan"] = np.array(out["wan"], complex) if out["wan"] else np.zeros((0, 2, n, n), complex)
    return r


# Dormand-Prince 5(4): nodes, stage rows, and the difference of the two solutions
_C = (0, 1 / 5, 3 / 10, 4 / 5, 8 / 9, 1, 1)
_B = ((), (1 / 5,), (3 / 40, 9 / 40), (44 / 45, -56 / 15, 32 / 9),
      (19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729),
      (9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656),
      (35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84))
_E = (35 / 384 - 5179 / 57600, 0, 500 / 1113 - 7571 / 16695, 125 / 192 - 393 / 640,
      -2187 / 6784 + 92097 / 339200, 11 / 84 - 187 / 2100, -1 / 40)


def _integrate_exact(case, seed):
    """the controlled steps on the output grid, a fresh first derivative at every output"""
    p = _Plain(case, seed)
    rho0 = p.ground()
    shape, n = rho0.shape, rho0.size
    y = np.concatenate([np.zeros(3, complex), rho0.reshape(-1)])

    def f(t, v):
        dA, dr = p.rhs(v[:3].real, v[3:].reshape(shape), t)
        return np.concatenate([dA.astype(complex), dr.reshape(-1)])

    _, _, fwhm, half = _pulse(case, seed)
    t0, t1 = -half * (fwhm / FS), half * (fwhm / FS)
    count = case["outputs"]
    gap = (t1 - t0) / (count - 1)
    ts, js, dt = [], [], gap
    for i in range(count):
        time = t0 + i * gap
        ts.append(time)
        js.append(p.current(y[:3].real, y[3:].reshape(shape)).mean(0))
        if i == count - 1:      # the grid's last interval runs past the window
            break
        t, end = time, time + gap
        k0 = f(t, y)
        while end - t > 2.3e-16:
            if t + dt - end > 2.3e-16:
                dt = end - t
            k = [k0]
            for q in range(1, 7):
                yq = y + sum(dt * b * kk for b, kk in zip(_B[q], k) if b)
                k.append(f(t + _C[q] * dt, yq))
            e = np.abs(sum(dt * c * kk for c, kk in zip(_E, k) if c))
            err = (e / (EPS_ABS + EPS_REL * (np.abs(y) + dt * np.abs(k[0])))).max()
            if err > 1:
                dt *= max(0.9 * err ** (-1 / 3), 0.2)
                continue
            y, k0, t = yq, k[6], t + dt
            if err < 0.5:
                dt *= 0.9 * max(5.0 ** -5, err) ** (-1 / 5)
    return {"t": np.array(ts), "j": np.array(js), "state": _pack(case, y[:3], y[3:].reshape(shape))}


# ---- the surrogate ------------------------------------------------------------
def _surrogate_data(case, seed):
    """normalised pulse parameters, normalised log-yields, and He-uniform weights per member"""
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, (case["rows"], DIMS[0])).astype(np.float32)
    t = rng.normal(size=(case["rows"], DIMS[-1])).astype(np.float32)
    w = []
    for _ in range(MEMBERS):
        parts = []
        for a, b in zip(DIMS, DIMS[1:]):
            lim = math.sqrt(6 / a) * (0.5 if b == DIMS[-1] else 1.0)
            parts += [rng.uniform(-lim, lim, a * b), rng.normal(size=b) * 0.05]
        w.append(np.concatenate(parts).astype(np.float32))
    return x, t, w


def _surrogate_exact(case, seed):
    x, t, w = _surrogate_data(case, seed)
    x, t = torch.from_numpy(x).double(), torch.from_numpy(t).double()
    ys, losses, grads = [], [], []
    for e in range(MEMBERS):
        p = torch.from_numpy(w[e]).double().requires_grad_(True)
        h, o = x, 0
        for i, (a, b) in enumerate(zip(DIMS, DIMS[1:])):
            W, o = p[o:o + a * b].view(b, a), o + a * b
            h, o = h @ W.T + p[o:o + b], o + b
            if i + 2 < len(DIMS):
                h = torch.nn.functional.silu(h)
        ys.append(h.detach())
        if case["mode"] == "gradient":
            loss = ((h - t) ** 2).mean()
            loss.backward()
            losses.append(loss.detach())
            grads.append(p.grad)
    if case["mode"] == "forward":
        return torch.stack(ys)
    return torch.stack(losses), torch.stack(grads)
